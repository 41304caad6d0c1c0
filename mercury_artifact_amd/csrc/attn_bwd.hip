// Block backward of the ring-attention step for gfx950, recomputing P from the saved LSE.
//
// Replaces the flash-attn call at utils/attn_bwd_dsl.py:83-115 of the reference:
//     P = exp(scale * q k^T - lse),  delta = rowsum(dout * out)
//     dV = P^T dout,  dP = dout v^T,  dS = P * (dP - delta),  dQ = scale * dS k,  dK = scale * dS^T q
//
// Two passes, no atomics (so every run is deterministic):
//   dQ       one workgroup per 256 (128) query rows of one head: Q and dout rows stay in registers, K / V tiles stream
//            through LDS; accumulates dQ
//   dK / dV  one workgroup per 128 keys of one KV head: K and V rows stay in registers, Q / dout tiles of the (grouped)
//            query heads stream through LDS together with their lse2 / delta from the workspace; accumulates dK, dV
// Per query row, delta = sum_d dout * out and lse2 = lse * log2(e) (with -inf, a row that saw no key, turned into +inf so
// that P = exp2(s - lse2) = 0 there) are worked out once and left in the workspace.
// Launches that fill the chip run the passes one after the other (bwd_main): dQ first, with eight wavefronts per
// workgroup, two per SIMD (it has half the accumulators of the other and fits 256 registers), and its prologue does
// delta and lse2.  Smaller ones run both passes side by side in one launch (bwd_joint) behind a small one for delta and
// lse2 (bwd_prepare).  Steps over several chunks have both forms too (bwd_main_chunks, bwd_joint_chunks).
// All of them share one body (bwd_pass).  "Stationary" rows (32 per wavefront) sit in the lane index of every
// MFMA accumulator, "streamed" rows in its registers, exactly as in the forward kernel:
//     T1[c][r] = X_str[c] . X_st[r]      (scores)          T2[c][r] = Y_str[c] . Y_st[r]      (dP)
//     acc^T[d][r] += X_str^T[d][c] dS[c][r]                (dQ or dK)
//     acc2^T[d][r] += Y_str^T[d][c] P[c][r]                (dV, DQ=false only)
// so P and dS feed the second MFMA straight from the accumulator registers.  The streamed tiles are
// copied global -> LDS without registers in between (buffer_load ... lds), row-major with swizzled
// 16-byte chunks, four stages deep; T1 / T2 read them with ds_read_b128 and the transposed operands
// of the second MFMAs are gathered from the same tiles with ds_read_b64_tr_b16, in the key order the
// accumulator registers hold.
#include "mhip_common.hpp"

#include <math.h>

#include <atomic>

namespace mhip {
namespace {

constexpr int kD = 128;
constexpr int kTile = 64;             // streamed rows per main-loop tile
constexpr int kRowsKv = 128;          // stationary key rows per workgroup of the dK / dV pass (4 wavefronts x 32)
constexpr int kRowsQ = 256;           // stationary query rows per workgroup of the dQ pass (8 wavefronts x 32)
constexpr int kStages = 4;
constexpr int kNoTile = 0x7fff0000;   // scalar offset that puts every lane of a copy out of range
constexpr int kNoColumn = 0x7fff0000; // vector offset with the same effect for one lane (the sum of the two is
                                      // below 2^32: no wrap)

// dq_acc += dQ and dq = dQ; or one chunk of a ring: dq_acc = dQ, dq_acc += dQ, dq = dq_acc + dQ
enum { kDqAdd = 0, kDqFirst = 1, kDqMiddle = 2, kDqLast = 3 };

struct BwdParams {
  const uint16_t* q; const uint16_t* k; const uint16_t* v; const uint16_t* dout;
  const uint16_t* out; const float* lse;   // saved output and log-sum-exp of the forward
  float* lse2; float* delta;               // both (B, Hq, Sq) fp32: written by the dQ pass, read by the dK / dV pass
  float* softmax_d;                        // rowsum(dout * out) itself for the caller, or null
  uint16_t* dq; uint16_t* dk; uint16_t* dv; float* dq_acc;     // dq may be null next to dq_acc
  float* dk32; float* dv32;                // the same bf16 values in fp32, (B, Sc, Hkv, D) contiguous, or null; dk / dv
                                           // may be null then
  int dq_mode;                             // what dq_acc is for: kDq*
  bool prepared;                           // delta and lse2 are in the workspace already
  int B, Sq, Sc, Hq, Hkv, group;
  Divisor by_hq, by_hkv, by_group;
  int D;            // head dimension of the tensors, a multiple of 8 up to kD; columns D .. kD-1 are zeros on chip
  int64_t q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh, o_sb, o_ss, o_sh;
  float scale, scale_log2;
};

// The workgroups of a pass: one per stationary tile of a (batch, head).
struct TileMap {
  int splits;          // workgroups that share a stationary tile, each with its part of the streamed tiles: a power of two
  int log_splits;
  float* partial;      // with splits > 1: their sums, [split] x the layout of dQ, or of dK and behind all of it dV, fp32
  int n_tiles;         // stationary tiles per (batch, head), times splits
  int total;
  int per_xcd;         // ceil(total / 8); the pass takes 8 * per_xcd workgroups
  int first;           // the first of them in the launch: a multiple of 8, so that both halves of a joint one keep their XCDs
  int heads_per_xcd;   // (batch, stationary head) pairs per XCD when they divide evenly, else 0
  Divisor by_tiles;
  Divisor by_order;    // causal: by all (batch, stationary head) pairs, or by those of an XCD
};

// Several chunks of a step in one launch: the places of BwdParams that differ from chunk to chunk.
struct Chunks {
  int n;
  Divisor by_heads;    // by B * Hkv
  const uint16_t* k[kMaxGroup]; const uint16_t* v[kMaxGroup];
  uint16_t* dk[kMaxGroup]; uint16_t* dv[kMaxGroup];
  float* dk32[kMaxGroup]; float* dv32[kMaxGroup];
};

// KK = k-steps of 16 head-dim values in T1 / T2: 8 computes on all 128 on-chip columns; 4 and 6 are the instantiations for
// head dimensions up to 64 and up to 96, which leave out the MFMAs, accumulators and fragments of the zero columns.  The
// vector work of a tile is the same, so a T1 / T2 slot carries more of it: 4096 x 4096, H32 takes 426 us instead of 654 at
// D 64 and 616 instead of 709 at D 96, 1237 x 1237, B2 H16/8, D 80 78.1 instead of 88.6, 512 x 512, B4 H5, D 96 16.9
// instead of 18.5; results bit-identical.
//
// WAVES = 8 wavefronts of 32 stationary rows (dQ: two per SIMD) or 4 (one per SIMD).  PREPARED: lse2 and delta of the
// query rows are in the workspace already; otherwise the dQ pass works them out.
//
// A row is 256 bytes on chip, on 64 columns 128: with half the LDS and at most 256 registers two workgroups of four
// wavefronts share a CU there, two wavefronts per SIMD, so that the vector work of one runs beside the MFMAs of the other:
// 4096 x 4096 H32 D 64 475 us to 426, 2048 x 2048 H16 70.3 to 59.9, causal 1500 x 1500 B2 H12 47.1 to 40.4, 8192 x 8192 H4
// 245 to 209.
template <int KK>
constexpr int kRowBytesOf = KK == 4 ? 128 : 256;
template <bool DQ, int KK>
constexpr int kStageBytesOf = 2 * kTile * kRowBytesOf<KK> + (DQ ? 0 : 2 * kTile * 4);
template <bool DQ, int WAVES, int KK>
constexpr int kSmemBytesOf =
    WAVES == 8 ? 3 * kStageBytesOf<DQ, KK> + WAVES * 32 * kRowBytesOf<KK> : kStages * kStageBytesOf<DQ, KK>;

// SPLIT: the workgroups of the pass may share their stationary tile (w.splits).  Of several chunks (dQ only) each takes whole ones.
//
// CHUNKS: several chunks of a step at once.  The dK / dV pass has a workgroup per key tile of every chunk; a workgroup of
// the dQ pass visits the chunks one after the other, as the dK / dV pass visits the query heads of a group, so dQ meets the
// sum carried from launch to launch once per launch instead of once per chunk.
//
// M = rows and columns of an MFMA tile, as in the forward kernel: v_mfma_f32_32x32x16_bf16, or v_mfma_f32_16x16x32_bf16, which
// takes less energy for the same work.  With it a lane holds two stationary rows (R), and an operand from LDS feeds an MFMA of each.
// For the dQ pass of eight wavefronts alone, which runs against the board's power (small_tiles); the dK / dV pass has one
// wavefront per SIMD to issue everything, takes 20 % more cycles with twice as many MFMAs and is no faster (4096 x 4096 H32 440 us / 444).
template <bool DQ, bool CAUSAL, int KK, int WAVES, bool PREPARED, bool SPLIT, bool CHUNKS = false, int M = 32>
__device__ __forceinline__ void bwd_pass(const BwdParams& p, const TileMap& w, const int block, unsigned char* smem,
                                         const Chunks* chunks = nullptr) {
  static_assert(DQ || WAVES == 4, "the dK / dV pass has no room for eight wavefronts in a workgroup");
  static_assert(!CHUNKS || (!(SPLIT && !DQ) && !CAUSAL), "launches of several chunks share the tiles of the dQ pass alone");
  static_assert(PREPARED || WAVES == 8, "the pass that prepares is the one with a launch of its own");
  static_assert(M == 32 || (M == 16 && DQ && WAVES == 8 && KK > 4), "32 x 32 or, in the dQ pass, 16 x 16 MFMA tiles");
  constexpr int R = 32 / M;                     // blocks of M stationary rows of a wavefront
  constexpr int NR = M * M / 64;                // registers of an accumulator tile
  constexpr int MB = 32 / M;                    // blocks of M streamed rows in half a tile
  constexpr int KB = KK * M / 32;               // k-steps of 512 / M head-dim values in T1 / T2
  constexpr int DB = KK * 16 / M;               // blocks of M head-dim values in the accumulators
  typedef typename std::conditional<M == 32, f32x16, f32x4>::type Acc;
  constexpr int kWavesWg = WAVES;
  constexpr int kRowsPerWg = kWavesWg * 32;
  constexpr int kRow = kRowBytesOf<KK>;
  constexpr int kLanes = kRow / 16, kRowsPerCopy = 64 / kLanes;      // a copy instruction: whole rows, 16 bytes per lane
  constexpr int kTileBytes = kTile * kRow;
  constexpr int kCpy = kTileBytes / 1024 / kWavesWg;    // copy instructions per wavefront for one tile
  constexpr int kRowsBytes = kRowsPerWg * kRow;         // one tensor's stationary rows
  // X tile, Y tile, and in the dK / dV pass lse2 and delta of the streamed rows
  constexpr int kStageBytes = kStageBytesOf<DQ, KK>;
  constexpr int kOffY = kTileBytes, kOffLse = 2 * kTileBytes, kOffDelta = kOffLse + kTile * 4;
  // chunk c (16 bytes) of row r of a tile is kept at chunk position c ^ swz(r)
  auto swz = [](int row) { return M == 16 ? lds_row_swizzle_16(row) : kRow == 256 ? lds_row_swizzle(row) : lds_half_row_swizzle(row); };
  // The stationary rows pass through LDS on their way into registers, in one stage each; with eight wavefronts X takes
  // the last stage and 32 KB behind it and Y the two stages before.
  constexpr int kXRows = 3 * kStageBytes, kYRows = WAVES == 8 ? kStageBytes : 2 * kStageBytes;
  static_assert(kYRows + kRowsBytes <= kXRows && kXRows + kRowsBytes <= kSmemBytesOf<DQ, WAVES, KK>, "the rows' places");

  // One round of argument loads instead of one before each first use (load_now in the common header says why).
  {
    const Divisor& by = CAUSAL ? w.by_order : w.by_tiles;
    const Divisor& heads = DQ ? p.by_hq : p.by_hkv;
    asm volatile("" ::"s"(w.per_xcd), "s"(w.total), "s"(by.mul), "s"(by.shift), "s"(by.d), "s"(heads.mul), "s"(heads.shift),
                 "s"(heads.d), "s"(p.by_group.mul), "s"(p.by_group.shift), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dout), "s"(p.lse2),
                 "s"(p.delta), "s"(p.B), "s"(p.Sq), "s"(p.Sc), "s"(p.Hq), "s"(p.group), "s"(p.D), "s"(p.q_sb), "s"(p.q_ss),
                 "s"(p.q_sh), "s"(p.k_sb), "s"(p.k_ss), "s"(p.k_sh), "s"(p.scale_log2));
  }
  // Workgroup i runs on XCD i % 8: every XCD gets a contiguous range of (batch, head) pairs.  Under the
  // causal mask the work of a stationary tile grows (query tiles) or shrinks (key tiles) with its index:
  // such launches run the longest tiles first, across all heads.
  int st_tile, bh, split;
  if (!CAUSAL) {
    const int logical = (block & 7) * w.per_xcd + (block >> 3);
    if (logical >= w.total) return;
    bh = w.by_tiles.quotient(logical, st_tile);
    split = 0;
    if (SPLIT) {
      split = st_tile & (w.splits - 1);
      st_tile >>= w.log_splits;
    }
  } else {
    int rank;                                       // position in longest-first order
    if (w.heads_per_xcd > 0) {
      rank = w.by_order.quotient(block >> 3, bh);
      bh += (block & 7) * w.heads_per_xcd;
    } else {
      if (block >= w.total) return;
      rank = w.by_order.quotient(block, bh);
    }
    split = 0;
    if (SPLIT) {
      split = rank & (w.splits - 1);
      rank >>= w.log_splits;
    }
    st_tile = DQ ? (SPLIT ? w.n_tiles >> w.log_splits : w.n_tiles) - 1 - rank : rank;
  }
  const uint16_t* kp = p.k; const uint16_t* vp = p.v;       // the chunk a dK / dV workgroup belongs to; dQ: the first one
  int chunk = 0;
  if (CHUNKS) {
    if (!DQ) chunk = chunks->by_heads.quotient(bh, bh);
    kp = chunks->k[chunk];
    vp = chunks->v[chunk];
  }
  int hs;                                           // stationary head: a q head (DQ) or a kv head
  const int b = (DQ ? p.by_hq : p.by_hkv).quotient(bh, hs);
  const int r0 = st_tile * kRowsPerWg;
  const int n_st = DQ ? p.Sq : p.Sc;                // stationary / streamed sequence lengths
  const int n_str = DQ ? p.Sc : p.Sq;
  const int shift = p.Sc - p.Sq;                    // causal: key j visible to query i iff j <= i + shift

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int ln = lane % M;
  const int lg = lane / M;
  const int my_r = r0 + wave * 32 + ln;             // this lane's (first) stationary row; the other one is M further

  // ---- stationary operands: B operands of T1 / T2, lane (ln, lg) holds row[512/M ks + 8 lg .. +7]; for dQ the
  // query is the stationary row and its lse2 / delta are per-lane scalars.  All loaded further down, behind
  // the first tile copies, so that one wait covers both latencies. ---------------------------------------
  bf16x8 xf[R][KB], yf[R][KB];
  float lse2_lane[R] = {}, delta_lane[R] = {};

  // ---- streamed tiles ---------------------------------------------------------------------------------
  // DQ: K / V rows of kv head hs / group.  Otherwise: Q / dout rows of the `group` query heads that share
  // kv head hs, one head after the other.
  int heads_str = DQ ? (CHUNKS ? chunks->n : 1) : p.group;            // (DQ: chunks)
  int first_tile = 0, tiles_per_head = (n_str + kTile - 1) / kTile;
  if (CAUSAL) {
    if (DQ) {   // keys beyond the last row's diagonal are hidden
      int lim = r0 + kRowsPerWg + shift;
      lim = lim < n_str ? lim : n_str;
      tiles_per_head = lim > 0 ? (lim + kTile - 1) / kTile : 0;
    } else {    // queries before the first key's diagonal see none of these keys
      const int i0 = r0 - shift;
      first_tile = i0 > 0 ? i0 / kTile : 0;
      if (first_tile > tiles_per_head) first_tile = tiles_per_head;
    }
  }
  const int span = tiles_per_head - first_tile;
  // this workgroup's part of the stream: tiles t0 .. t0 + ntiles - 1 of the pass's sequence
  int t0 = 0, ntiles = span * heads_str;
  int first_chunk = 0;
  if (SPLIT && CHUNKS) {
    const int part = (chunks->n + w.splits - 1) >> w.log_splits;
    first_chunk = split * part < chunks->n ? split * part : chunks->n;
    heads_str = first_chunk + part < chunks->n ? first_chunk + part : chunks->n;
    ntiles = span * (heads_str - first_chunk);
  } else if (SPLIT && w.splits > 1) {
    const int all = ntiles, part = (all + w.splits - 1) >> w.log_splits;
    t0 = split * part < all ? split * part : all;
    ntiles = all - t0 < part ? all - t0 : part;
  }

  const uint16_t* xbase; const uint16_t* ybase; int64_t s_ss, s_sh; uint32_t s_bytes;
  const int64_t kv_at = DQ ? b * p.k_sb + p.by_group.quotient(hs) * p.k_sh : 0;
  if (DQ) {
    xbase = kp + kv_at; ybase = vp + kv_at;
    s_ss = p.k_ss; s_sh = 0;
    s_bytes = (uint32_t)(((int64_t)(p.Sc - 1) * p.k_ss + p.D) * 2);
  } else {
    xbase = p.q + b * p.q_sb; ybase = p.dout + b * p.q_sb;
    s_ss = p.q_ss; s_sh = p.q_sh;
    s_bytes = (uint32_t)(((int64_t)(p.Sq - 1) * p.q_ss + (int64_t)(p.Hq - 1) * p.q_sh + p.D) * 2);
  }
  u32x4 xrs = rsrc_words(xbase, s_bytes);
  u32x4 yrs = rsrc_words(ybase, s_bytes);
  // The address words of chunk i's descriptors in lane i: a scalar load of them inside the main loop would make its waits for
  // one LDS operand waits for all.
  uint32_t k_words[2] = {}, v_words[2] = {};
  if (CHUNKS && DQ) {
    const uint64_t ka = (uint64_t)(chunks->k[lane & (kMaxGroup - 1)] + kv_at), va = (uint64_t)(chunks->v[lane & (kMaxGroup - 1)] + kv_at);
    k_words[0] = (uint32_t)ka; k_words[1] = (uint32_t)(ka >> 32) & 0xffffu;
    v_words[0] = (uint32_t)va; v_words[1] = (uint32_t)(va >> 32) & 0xffffu;
    asm volatile("" : "+v"(k_words[0]), "+v"(k_words[1]), "+v"(v_words[0]), "+v"(v_words[1]));
  }

  // Wavefront w copies rows 16w .. 16w+15 of the X and the Y tile: four instructions of 1 KB each; lane l
  // of instruction u lands at row 16w + 4u + l/16, chunk position l%16, and fetches the chunk that lives
  // there.  Rows past the end of the streamed tensor arrive as zeros when the layout puts them past the
  // descriptor's range, and their P / dS are zeroed by index in any case.  lse2 and delta of the 64
  // streamed rows (DQ=false) are copied by the even / odd wavefronts (twice the same bytes: every
  // wavefront then has the same number of copies in flight, which the vmcnt waits rely on).
  int cvoff[kCpy];
#pragma unroll
  for (int u = 0; u < kCpy; ++u) {
    const int row = kRowsPerCopy * (kCpy * wave + u) + lane / kLanes;
    const int chunk = (lane % kLanes) ^ swz(row);
    // chunks past the head dimension: an offset that is out of the descriptor's range for every tile, so they
    // arrive as zeros and a tile in LDS always has 128 columns
    cvoff[u] = chunk * 8 < p.D ? (int)(row * s_ss * 2) + (chunk << 4) : kNoColumn;
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  constexpr int kCopiesPerTile = DQ ? 2 * kCpy : 2 * kCpy + 1;
  // The copies of a tile go out one instruction at a time (piece 0 .. kCopiesPerTile - 1), in the main loop between
  // MFMAs; copy_setup works out the scalar offsets of the next tile that has not been requested yet.  Which one that is is
  // kept as a pair of running counters (position inside the head's span, head of the group; dQ: position in the chunk,
  // chunk) instead of a division per tile: every scalar instruction of the loop takes an issue slot of
  // the one wavefront a SIMD runs in the dK / dV pass.
  int cp_soff = 0, cp_ld_soff = 0, cp_ld_voff = 0;
  int nx_h = SPLIT && !DQ && span > 0 ? t0 / span : first_chunk, nx_t = 0;
  int nx_r = SPLIT && CHUNKS ? 0 : t0 - nx_h * span;
  int cur_r = nx_r;                                   // position of the tile being worked on
  const uint32_t ld_rows = (uint32_t)p.B * (uint32_t)p.Hq * (uint32_t)p.Sq;     // the host keeps this below 2^30
  const u32x4 ldrs = rsrc_words((wave & 1) ? p.delta : p.lse2, ld_rows * 4u);
  auto copy_setup = [&]() {
    const bool live = SPLIT && !CHUNKS ? nx_t < ntiles : DQ && !CHUNKS ? nx_r < span : nx_h < heads_str;
    const uint32_t hq = DQ ? 0u : (uint32_t)(hs * p.group + (live ? nx_h : 0));
    const uint32_t c0 = (uint32_t)((first_tile + (live ? nx_r : 0)) * kTile);
    // element offsets stay below 2^31 (checked by the host), so 32-bit arithmetic is exact
    cp_soff = live ? (int)((c0 * (uint32_t)s_ss + hq * (uint32_t)s_sh) * 2u) : kNoTile;
    if (!DQ) {
      cp_ld_soff = live ? (int)((((uint32_t)b * (uint32_t)p.Hq + hq) * (uint32_t)p.Sq + c0) * 4u) : kNoTile;
      // rows past the end are another head's: out of range (their scores are hidden, but 0 * infinity is not 0)
      cp_ld_voff = (int)c0 + lane < p.Sq ? lane * 4 : kNoColumn;
    }
    if (CHUNKS && DQ && nx_r == 0 && live) {          // the copies of this chunk start here
      xrs[0] = __builtin_amdgcn_readlane(k_words[0], nx_h);
      xrs[1] = __builtin_amdgcn_readlane(k_words[1], nx_h);
      yrs[0] = __builtin_amdgcn_readlane(v_words[0], nx_h);
      yrs[1] = __builtin_amdgcn_readlane(v_words[1], nx_h);
    }
    ++nx_r;
    if (SPLIT) ++nx_t;
    if ((!DQ || CHUNKS) && nx_r == span) { nx_r = 0; ++nx_h; }
  };
  auto copy_piece = [&](int piece, int stage) {
    const uint32_t dst = lds_base + stage * kStageBytes + wave * (kCpy * 1024);
    if (piece < kCpy) copy16_to_lds(xrs, dst + piece * 1024, cvoff[piece < kCpy ? piece : 0], cp_soff);
    else if (piece < 2 * kCpy) copy16_to_lds(yrs, dst + kOffY + (piece - kCpy) * 1024, cvoff[piece < 2 * kCpy ? piece - kCpy : 0], cp_soff);
    else if (!DQ)
      copy4_to_lds(ldrs, lds_base + stage * kStageBytes + ((wave & 1) ? kOffDelta : kOffLse), cp_ld_voff, cp_ld_soff);
  };
  auto copy_tile = [&](int stage) {                   // the next tile, all at once (prologue)
    copy_setup();
#pragma unroll
    for (int piece = 0; piece < kCopiesPerTile; ++piece) copy_piece(piece, stage);
  };

  // row-major operand reads (A of T1 / T2): lane (ln, lg) reads chunk 64/M kk + lg of row M mb + ln
  int rm_rd[KB];                                      // + mb * M rows
#pragma unroll
  for (int kk = 0; kk < KB; ++kk) rm_rd[kk] = ln * kRow + (((64 / M * kk + lg) ^ swz(ln)) << 4);
  // transposed operand reads (A of the second MFMAs) for head-dim block db and k-step j2 of 512/M streamed rows of a half: the
  // lane's 8 rows are X + {0..3} and, 8 (M = 16: 16) rows on, four more, X = 512/M j2 + 4 lg -- the rows its P / dS
  // registers hold.  One ds_read_b64_tr_b16 per group of 4 rows: within 16 lanes, lane s supplies the
  // address of row X + s/4, head-dim values 4 (s%4) .. +3 of the 16-column strip, and receives column s.
  int tr_rd[KK];                                      // 32: [2 db + second four rows], 16: [db]; + j2 * 512/M rows
  {
    const int s16 = lane & 15, strip = M == 32 ? (lane >> 4) & 1 : 0;
    const int cl = 2 * strip + ((s16 & 3) >> 1);
#pragma unroll
    for (int i = 0; i < KK; ++i) {
      const int db = M == 32 ? i / 2 : i, row = (M == 32 ? 8 * (i & 1) : 0) + 4 * lg + (s16 >> 2);
      tr_rd[i] = row * kRow + (((M / 8 * db + cl) ^ swz(row)) << 4) + (s16 & 1) * 8;
    }
  }
  typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4;
  typedef __attribute__((address_space(3))) const bf16x8* lds_bf16x8;
  const Acc zero = {};
  Acc acc1[DB][R], acc2[DB][R];    // DQ: acc1 = dQ^T.  Otherwise acc1 = dK^T, acc2 = dV^T
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int r = 0; r < R; ++r) acc1[i][r] = acc2[i][r] = zero;

  // Tile t lives in stage t % 4 and is processed as two halves of 32 streamed rows.  Per tile the matrix
  // pipe sees one unbroken sequence of MFMA slots in four phases (half as many slots in each on 64 columns, three quarters on 96):
  //   P0  T1 / T2 of (t, second half)      16 slots, each carrying P / dS of one register of (t, first half)
  //   P1  accumulate (t, first half)       16 slots (8 for dQ)
  //   P2  T1 / T2 of (t+1, first half)     16 slots, each carrying P / dS of one register of (t, second half)
  //   P3  accumulate (t, second half)      16 slots (8 for dQ)
  // The LDS operand of slot s+4 is read in slot s, across phase and tile boundaries, so the pipe never
  // waits for LDS at the start of a phase.  An iteration starts by waiting for this wavefront's copies of
  // tile t+1 (those of tile t+2 stay in flight) and a barrier, after which tile t+1 is complete for every
  // wavefront and nobody reads tile t-1 any more, whose stage then receives tile t+3.  Tiles past the end
  // are copied as zeros (and their T1 / T2 computed, unused) so that the number of copies in flight
  // stays the same.
  // operand reads in flight ahead of the MFMAs (2, 4 and 8 measure the same; 2 keeps eight wavefronts inside 256 registers)
  constexpr int kDepth = WAVES == 8 ? 2 : 4;
  constexpr int kT = 2 * KK;                               // slots of a T1 / T2 phase, an operand from LDS and R MFMAs each
  constexpr int kAcc = DQ ? KK : 2 * KK;                   // slots of an accumulate phase
  // 16 x 16 tiles: P / dS of the second row block are due with the first operand of an accumulate phase, where 32 x 32 tiles
  // need the second k-step's half a phase later.  Its MFMAs run kLag slots behind the first block's, those of the last
  // kLag operands in the T1 / T2 phase that follows; the operands stay in the ring for as long.
  constexpr int kLag = M == 16 ? kDepth : 0, kRing = kDepth + kLag;
  constexpr int kP1 = kT, kP2 = kT + kAcc, kP3 = 2 * kT + kAcc, kSlots = 2 * (kT + kAcc);
  // The 16 steps of the vector pipeline are spread over the slots of a T1 / T2 phase: slot i runs steps vec0(i) .. vec0(i + 1) - 1.
  auto vec0 = [](int i) -> int { return i * 16 / kT; };
  typedef __attribute__((address_space(3))) const f32x4* lds_f32x4;
  typedef __attribute__((address_space(3))) const float* lds_f32;
  // LDS addresses of the operand reads.  rm_a / tr_a hold, per lane, the addresses inside ONE tile's stage and are
  // moved on to the next stage in place, each at a point of the slot sequence where no read of its kind is due
  // (rm_a in the last kDepth slots of P0: the reads of the current tile's T1 / T2 operands are all issued by then and
  // those of the next tile start at slot kP2 - kDepth; tr_a in the last kDepth slots, after the last transposed read).
  // ld_cur / ld_next address lse2 / -delta of the current and the next tile.  Everything else about an address
  // is an immediate offset of the LDS instruction.
  int rm_a[KB], tr_a[KK];
#pragma unroll
  for (int kk = 0; kk < KB; ++kk) rm_a[kk] = rm_rd[kk] + (int)lds_base;
#pragma unroll
  for (int i = 0; i < KK; ++i) tr_a[i] = tr_rd[i] + (int)lds_base;
  int ld_cur = (int)lds_base + lg * 16, ld_next = ld_cur + kStageBytes;
  auto mfma = [](const bf16x8& x, const bf16x8& y, const Acc& c) -> Acc {
    if constexpr (M == 32) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
  };
  // slot i of the T1 / T2 sequence of one half: k-step i / (2 MB), X (T1) on even and Y (T2) on odd slots
  auto read_rm = [&](int half, int i) -> bf16x8 {
    return *(lds_bf16x8)(uintptr_t)(uint32_t)(rm_a[i / (2 * MB)] + (half * 32 + (i >> 1) % MB * M) * kRow + ((i & 1) ? kOffY : 0));
  };
  // T1 / T2 of a half: streamed rows M mb + 8 (j / 4) + 4 lg + j % 4 against stationary rows M r + ln
  struct Scores {
    Acc a[MB][R];
    // the order of the vector work: elements 8 i .. 8 i + 7 make B operand i of the second MFMAs, k-step i (M = 16: row block i)
    __device__ __forceinline__ static constexpr int r_of(int e) { return M == 32 ? 0 : e >> 3; }
    __device__ __forceinline__ static constexpr int mb_of(int e) { return M == 32 ? 0 : (e >> 2) & 1; }
    __device__ __forceinline__ static constexpr int j_of(int e) { return e % NR; }
    __device__ __forceinline__ float get(int e) const { return a[mb_of(e)][r_of(e)][j_of(e)]; }
    __device__ __forceinline__ void set(int e, float x) { a[mb_of(e)][r_of(e)][j_of(e)] = x; }
  };
  // T2 starts from -delta of the half's streamed rows (dQ pass: of this lane's stationary rows), so that what
  // the vector unit receives is dP - delta already
  Acc nd[R];
  auto t_mfma = [&](int i, int r, const bf16x8& a, Scores& n1, Scores& n2) {
    const int kk = i / (2 * MB), mb = (i >> 1) % MB;
    if (i & 1) n2.a[mb][r] = mfma(a, yf[r][kk], kk == 0 ? nd[r] : n2.a[mb][r]);
    else n1.a[mb][r] = mfma(a, xf[r][kk], kk == 0 ? zero : n1.a[mb][r]);
  };
  // slot i of an accumulate phase of a half: head-dim block and k-step, X^T (dS) / Y^T (P) alternating for dK, dV
  auto read_acc = [&](int half, int i) -> bf16x8 {
    const int m = DQ ? i : (i >> 1);
    const int off = half * (32 * kRow) + (m / DB) * (512 / M * kRow) + ((!DQ && (i & 1)) ? kOffY : 0);
    const int first = M == 32 ? tr_a[2 * (m % DB) % KK] : tr_a[m % DB], second = M == 32 ? tr_a[(2 * (m % DB) + 1) % KK] : tr_a[m % DB] + 16 * kRow;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4)(uintptr_t)(uint32_t)(first + off));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4)(uintptr_t)(uint32_t)(second + off));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  bf16x8 pfrag[2] = {}, dsfrag[2] = {};     // P and dS of the half being accumulated as B operands (two k-steps or row blocks)
  bf16x8 ring[kRing] = {};
  Scores ta1, ta2, tb1, tb2;      // T1 / T2 of the two halves in flight: (t, first half), (t, second half)
  f32x4 lv[5];                    // lse2 of 4 streamed rows per entry (dK / dV pass), read one group ahead

  // Hidden elements (rows past the end of the streamed tensor, the causal mask) get a score of -inf,
  // hence P = dS = 0.  Only the last tile of a head and the tiles the diagonal crosses need it.
  auto mask_half = [&](Scores& c1, int cb) {
    bool need_mask = cb + 32 > n_str;
    if (CAUSAL) need_mask = need_mask || (DQ ? (cb + 31 > r0 + shift) : (r0 + kRowsPerWg - 1 > cb + shift));
    if (need_mask) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int j = c1.j_of(e), c = cb + c1.mb_of(e) * M + (j >> 2) * 8 + lg * 4 + (j & 3);     // streamed row of this element
        bool hidden = c >= n_str;
        if (CAUSAL) {
          const int row = my_r + c1.r_of(e) * M;
          hidden = hidden || (DQ ? (c > row + shift) : (row > c + shift));
        }
        if (hidden) c1.set(e, -INFINITY);
      }
    }
  };
  // lse2 of rows 8 g + 4 lg .. + 3 of a half of the current (next: of the following) tile
  auto read_ld = [&](bool next, int half, int g, f32x4& l) {
    l = *(lds_f32x4)(uintptr_t)(uint32_t)((next ? ld_next : ld_cur) + kOffLse + (half * 32 + g * 8) * 4);
  };
  // -delta of rows 8 g + 4 lg .. + 3 (g = 0..3) of a half of the current / following tile, in the order of the
  // accumulator registers of T2 (dK / dV pass), one group per call
  auto read_nd = [&](bool next, int half, int g) {
    const f32x4 d = *(lds_f32x4)(uintptr_t)(uint32_t)((next ? ld_next : ld_cur) + kOffDelta + (half * 32 + g * 8) * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) nd[0][(4 * g + e) % NR] = d[e];
  };
  // P / dS of the half in (c1, c2): 16 accumulator registers, spread over the 16 slots in which the next
  // half's T1 / T2 are issued AND the first slots of the accumulate phase that follows (a wavefront issues
  // one vector instruction every ~5 cycles, so 16 slots of 32 cycles do not hold all of it).  Register e
  // enters at slot first_slot(e); its work is a three-stage pipeline so that no instruction waits for the
  // one issued just before it:
  //   first_slot      argument of the exponential
  //   first_slot + 1  exponential
  //   first_slot + 2  dS = P (dP - delta)     (c2 arrives as dP - delta)
  // Registers 0-7 (k-step or row block 0 of the accumulate phase) are packed before that phase starts, registers 8-15
  // before its second half does (M = 16: before slot kLag of it).
  // With 16 x 16 tiles a stage takes two half slots, one behind each of a slot's two MFMAs: behind both, its instructions
  // leave the matrix unit less to do meanwhile (4.98 M cycles instead of 4.89 M for 4096 x 4096 H32).
  auto first_slot = [](int e) -> int {
    if (M == 16) return e < 8 ? (e * 5) / 2 : 2 * e - 2;     // half slots: 0,2,5,..,17 | 14,16,..,28: packed up to 23 and 34
    if (DQ) return e < 8 ? (e * 3) / 2 : 1 + e;          // 0,1,3,4,6,7,9,10 | 9..16: packed at slots 13 and 19 (acc 16-19, 20-23)
    return e < 8 ? (e * 7) / 4 : 5 + e;                  // 0,1,3,5,7,8,10,12 | 13..20: packed at slots 15 and 23 (acc 16-23, 24-31)
  };
  float earg[16];
  auto vector_slot = [&](int s, Scores& c1, Scores& c2, int half) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int f = first_slot(e);
      if (s == f) {
        const float l = DQ ? lse2_lane[c1.r_of(e)] : lv[e >> 2][e & 3];
        earg[e] = __builtin_fmaf(c1.get(e), p.scale_log2, -l);
        // lse2 of the next four rows, one group ahead
        if (!DQ && (e & 3) == 0 && e < 12) read_ld(false, half, (e >> 2) + 1, lv[(e >> 2) + 1]);
      }
      if (s == f + R) c1.set(e, fast_exp2(earg[e]));
      if (s == f + 2 * R) c2.set(e, c1.get(e) * c2.get(e));
    }
    // M = 32: the eight elements of an operand at once, M = 16: two at a time
#pragma unroll
    for (int e = 0; e < 16; e += 2)
      if (s == first_slot(M == 32 ? e | 7 : e + 1) + 3 * R) {
        u32x4 wp = __builtin_bit_cast(u32x4, pfrag[e >> 3]), wd = __builtin_bit_cast(u32x4, dsfrag[e >> 3]);
        wp[(e >> 1) & 3] = pack_bf16(c1.get(e), c1.get(e + 1));
        wd[(e >> 1) & 3] = pack_bf16(c2.get(e), c2.get(e + 1));
        pfrag[e >> 3] = __builtin_bit_cast(bf16x8, wp);
        dsfrag[e >> 3] = __builtin_bit_cast(bf16x8, wd);
      }
  };
  // the vector work behind MFMA r of slot i of a T1 / T2 phase, and of the accumulate phase that follows (steps 16 ..)
  auto vector_t = [&](int i, int r, Scores& c1, Scores& c2, int half) {
#pragma unroll
    for (int v = vec0(i); v < vec0(i + 1); ++v) vector_slot(M == 32 ? v : 2 * v + r, c1, c2, half);
  };
  auto vector_tail = [&](int i, int r, Scores& c1, Scores& c2, int half) {
#pragma unroll
    for (int v = vec0(i); v < vec0(i + 1); ++v)
      if (v < (DQ ? 4 : 8)) vector_slot(M == 32 ? 16 + v : 2 * (16 + v) + r, c1, c2, half);
  };
  auto acc_one = [&](int i, int r, const bf16x8& a) {
    const int m = DQ ? i : (i >> 1);
    const int db = m % DB, at = M == 32 ? m / DB : r;
    if (DQ || !(i & 1)) acc1[db][r] = mfma(a, dsfrag[at], acc1[db][r]);
    else acc2[db][r] = mfma(a, pfrag[at], acc2[db][r]);
  };
  // MFMA r of slot i of an accumulate phase that starts at slot `phase` of the tile
  auto acc_mfma = [&](int i, int r, int phase) {
    if (r == 0) acc_one(i, 0, ring[(phase + i) % kRing]);
    else if (i >= kLag) acc_one(i - kLag, 1, ring[(phase + i - kLag) % kRing]);
  };
  // and the second row block's last MFMAs, in slot i of the T1 / T2 phase behind it
  auto acc_rest = [&](int i, int phase) {
    if (i < kLag) acc_one(kAcc - kLag + i, R - 1, ring[(phase + kAcc - kLag + i) % kRing]);
  };
  // LDS operand of slot s of the current tile's sequence; s >= kSlots continues into the next tile's P0.  The
  // T1 / T2 operands of slots kP2 .. kP3 - 1 and from kSlots on belong to the next tile: rm_a has moved on by then.
  auto read_slot = [&](int s) -> bf16x8 {
    if (s >= kSlots) return read_rm(1, s - kSlots);
    if (s < kP1) return read_rm(1, s);
    if (s < kP2) return read_acc(0, s - kP1);
    if (s < kP3) return read_rm(0, s - kP2);
    return read_acc(1, s - kP3);
  };
  auto refill = [&](int s) { ring[(s + kDepth) % kRing] = read_slot(s + kDepth); };
  static_assert(kP2 - kDepth >= kT && kAcc >= kDepth, "rm_a moves in the last kDepth slots of P0, tr_a in the last kDepth slots of P3");

  // Stationary rows: read straight into the fragment layout every load instruction would touch 32 rows (24 such loads
  // per wavefront in the dQ pass, one wait for all of them and the tiles).  They are copied to LDS instead, four whole
  // rows per instruction and each wavefront its own 32, swizzled like the streamed tiles: 4 - 6 us less per block (both
  // passes, 256 x 256 H4 27.3 -> 23.3 us, 1024 x 1024 H32 71.0 -> 65.4, 4096 x 4096 H32 768 -> 760).  Rows past the end
  // repeat the last one, columns past the head dimension are cleared in the fragment.
  {
    const uint32_t x_lds = lds_base + kXRows + wave * (32 * kRow), y_lds = lds_base + kYRows + wave * (32 * kRow);
    const uint16_t* xsrc = DQ ? p.q + b * p.q_sb + hs * p.q_sh : kp + b * p.k_sb + hs * p.k_sh;
    const uint16_t* ysrc = DQ ? p.dout + b * p.q_sb + hs * p.q_sh : vp + b * p.k_sb + hs * p.k_sh;
    const int64_t st_ss = DQ ? p.q_ss : p.k_ss;
    auto row_of = [&](int u) {                        // row and column of the lane's 16 bytes in copy u
      const int row = r0 + wave * 32 + kRowsPerCopy * u + lane / kLanes;
      return row < n_st ? row : n_st - 1;
    };
    auto col_of = [&](int u) { return ((lane % kLanes) ^ swz(kRowsPerCopy * u + lane / kLanes)) * 8; };
    constexpr int kCopies = 32 / kRowsPerCopy;
    auto copy_rows = [&](const uint16_t* src, uint32_t dst) {
#pragma unroll
      for (int u = 0; u < kCopies; ++u) {
        const int col = col_of(u);
        copy16_to_lds(src + (int64_t)row_of(u) * st_ss + (col < p.D ? col : 0), dst + u * 1024);
      }
    };
    auto read_rows = [&](uint32_t src, bf16x8 (&f)[R][KB]) {
#pragma unroll
      for (int ks = 0; ks < KB; ++ks)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          f[r][ks] = *(lds_bf16x8)(uintptr_t)(src + rm_rd[ks] + r * M * kRow);
          if (ks * (512 / M) + lg * 8 >= p.D) f[r][ks] = bf16x8{};
        }
    };
    // Pin the fragments (the copies are invisible to the compiler's wait counting).  The dK / dV pass keeps these
    // MFMA operands in accumulation registers: its arithmetic registers are needed for the tiles of T1 / T2 that
    // the vector unit works on.  At two wavefronts per SIMD -- the dQ pass, 64 columns -- no accumulation registers are used
    // at all (a kernel that does gets its 256 registers split 128 / 128).
    auto pin = [&]() {
#pragma unroll
      for (int ks = 0; ks < KB; ++ks)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (DQ || KK == 4) { asm volatile("" : "+v"(xf[r][ks])); asm volatile("" : "+v"(yf[r][ks])); }
          else { asm volatile("" : "+a"(xf[r][ks])); asm volatile("" : "+a"(yf[r][ks])); }
        }
    };
    // what row (lane % 32) of the wavefront has, handed to the lanes that hold the row
    auto to_lanes = [&](float x, float (&y)[R]) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        y[r] = M == 32 ? x : __int_as_float(__builtin_amdgcn_ds_bpermute((r * M + ln) << 2, __float_as_int(x)));
    };
    const int half_row = r0 + wave * 32 + (lane & 31);
    if (!PREPARED) {
      // This pass runs first and prepares what both passes need per query row: delta = rowsum(dout * out), kept
      // negated (the dP products start from it), and lse2 = lse * log2(e) with -inf (a row that saw no key) turned
      // into +inf so that P = exp2(s - lse2) = 0 there.
      if (ntiles > 0) copy_tile(0);
      copy_rows(ysrc, y_lds);
      copy_rows(xsrc, x_lds);
      const uint16_t* osrc = p.out + b * p.o_sb + hs * p.o_sh;
      bf16x8 o8[kCopies];
#pragma unroll
      for (int u = 0; u < kCopies; ++u) {
        const int col = col_of(u);
        o8[u] = bf16x8{};
        if (col < p.D) o8[u] = *reinterpret_cast<const bf16x8*>(osrc + (int64_t)row_of(u) * p.o_ss + col);
      }
      const int row = half_row < n_st ? half_row : n_st - 1;
      const int64_t r = ((int64_t)b * p.Hq + hs) * p.Sq + row;
      const float l = p.lse[r];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // Lane (g, i) of four groups of 16 (64 columns: eight of 8) has columns of row 4 u + g (8 u + g) of out and dout in copy
      // u: the sum over the group is the row's delta, left in all of its lanes; lane i keeps the one of copy i % 8
      // (i % 4), and lane l fetches row l % 32's.
      float mine = 0.f;
#pragma unroll
      for (int u = 0; u < kCopies; ++u) {
        const bf16x8 d8 = *(lds_bf16x8)(uintptr_t)(y_lds + u * 1024 + lane * 16);
        float part = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) part = __builtin_fmaf((float)d8[j], (float)o8[u][j], part);
        part = kLanes == 16 ? row16_sum(part) : row8_sum(part);
        mine = lane % kCopies == u ? part : mine;
      }
      const int holder = (lane & 31) % kRowsPerCopy * kLanes + (lane & 31) / kRowsPerCopy;
      const float delta = __int_as_float(__builtin_amdgcn_ds_bpermute(holder << 2, __float_as_int(mine)));
      read_rows(y_lds, yf);
      read_rows(x_lds, xf);
      pin();
      const float lse2 = (l == -INFINITY) ? INFINITY : l * kLog2e;
      to_lanes(lse2, lse2_lane);
      to_lanes(-delta, delta_lane);
      if (lane < 32 && half_row < n_st) {
        p.delta[r] = -delta;
        p.lse2[r] = lse2;
        if (p.softmax_d) p.softmax_d[r] = delta;     // for callers that want flash-attn's softmax_d back
      }
#pragma unroll
      for (int i = 0; i < R; ++i) asm volatile("" : "+v"(lse2_lane[i]), "+v"(delta_lane[i]));
      __builtin_amdgcn_s_barrier();                  // the rows' places are stages 1 .. 3 from here on
      if (ntiles > 0) { copy_tile(1); copy_tile(2); }
    } else if (ntiles > 0) {
      constexpr bool kEarly = WAVES == 4;            // stage 1 is not part of the rows' places
      const int64_t r = DQ ? ((int64_t)b * p.Hq + hs) * p.Sq + (half_row < n_st ? half_row : n_st - 1) : 0;
      const uint32_t ld_lds = lds_base + kSmemBytesOf<true, 4, KK> + wave * 256;     // 32 rows' lse2, then their delta
      if (DQ && !kEarly) {
        to_lanes(p.lse2[r], lse2_lane);
        to_lanes(p.delta[r], delta_lane);
#pragma unroll
        for (int i = 0; i < R; ++i) asm volatile("" : "+v"(lse2_lane[i]), "+v"(delta_lane[i]));
      }
      copy_tile(0);
      // (through LDS like the rows: loads into registers would be waited for before the first copy or with the last)
      if (DQ && kEarly) copy4_to_lds((lane >= 32 ? p.delta : p.lse2) + r, ld_lds);
      copy_rows(xsrc, x_lds);
      copy_rows(ysrc, y_lds);
      if (kEarly) copy_tile(1);
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kEarly ? kCopiesPerTile : 0) : "memory");
      if (DQ && kEarly) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
          lse2_lane[i] = *(lds_f32)(uintptr_t)(ld_lds + (i * M + ln) * 4);
          delta_lane[i] = *(lds_f32)(uintptr_t)(ld_lds + 128 + (i * M + ln) * 4);
        }
      }
      read_rows(x_lds, xf);
      read_rows(y_lds, yf);
      pin();
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (DQ && kEarly) asm volatile("" : "+v"(lse2_lane[i]), "+v"(delta_lane[i]));
      __builtin_amdgcn_s_barrier();                  // tile 0 is there for everybody, the rows' places are free
      if (!kEarly) copy_tile(1);
      copy_tile(2);
    }
  }
  if (ntiles > 0) {
    if (DQ) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < NR; ++j) nd[r][j] = delta_lane[r];
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) read_nd(false, 0, g);
    }
    // T1 / T2 of the first half of tile 0, nothing to interleave with
#pragma unroll
    for (int i = 0; i < kDepth; ++i) ring[i] = read_rm(0, i);
#pragma unroll
    for (int i = 0; i < kT; ++i) {
#pragma unroll
      for (int r = 0; r < R; ++r) t_mfma(i, r, ring[i % kDepth], ta1, ta2);
      if (i + kDepth < kT) ring[i % kDepth] = read_rm(0, i + kDepth);
    }
#pragma unroll
    for (int i = 0; i < kDepth; ++i) ring[i] = read_rm(1, i);            // slots 0 .. 3 of tile 0 (the places behind: zeros)
    if (!DQ) {
      read_ld(false, 0, 0, lv[0]);
#pragma unroll
      for (int g = 0; g < 4; ++g) read_nd(false, 1, g);        // for T2 of the second half, first thing in the loop
    }
  }
  for (int t = 0; t < ntiles; ++t) {
    const int c0 = (first_tile + cur_r) * kTile;
    if (++cur_r == span) cur_r = 0;
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kCopiesPerTile) : "memory");          // one tile of copies stays in flight
    __builtin_amdgcn_s_barrier();
    copy_setup();
    // byte distance from this tile's stage to the next tile's, and from that one to the one after
    const int step1 = ((t + 1) & 3) == 0 ? -3 * kStageBytes : kStageBytes;
    const int step2 = ((t + 2) & 3) == 0 ? -3 * kStageBytes : kStageBytes;
    static_assert(kSlots % kRing == 0 && kT >= kLag, "the ring position is the slot number modulo its depth");
    mask_half(ta1, c0);
#pragma unroll
    for (int i = 0; i < kT; ++i) {                       // P0, carrying the copies of tile t+3
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r > 0) __builtin_amdgcn_sched_barrier(0);
        t_mfma(i, r, ring[i % kRing], tb1, tb2);
        vector_t(i, r, ta1, ta2, 0);
      }
      acc_rest(i, kP3);                                  // of the tile before (the first tile: zeros)
#pragma unroll
      for (int piece = i; piece < kCopiesPerTile; piece += kT) copy_piece(piece, (t + 3) & 3);
      refill(i);
      if (i >= kT - kDepth) {                            // the last read of this tile's T1 / T2 operands is out: on to the next
#pragma unroll
        for (int a = (i - (kT - kDepth)) * KB / kDepth; a < (i + 1 - (kT - kDepth)) * KB / kDepth; ++a) rm_a[a] += step1;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < kAcc; ++i) {                     // P1
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r > 0) __builtin_amdgcn_sched_barrier(0);
        vector_tail(i, r, ta1, ta2, 0);
        acc_mfma(i, r, kP1);
      }
      if (!DQ && i == kAcc - 2) read_ld(false, 1, 0, lv[0]);
      // -delta for T2 of (t+1, first half), which starts in P2: read once the vector work on this half's dP is
      // through (half of the slots), so that the values can land in the registers T2 accumulates in
      if (!DQ && i >= kAcc / 2 && i < kAcc / 2 + 4) read_nd(true, 0, i - kAcc / 2);
      refill(kP1 + i);
      __builtin_amdgcn_sched_barrier(0);
    }
    mask_half(tb1, c0 + 32);
#pragma unroll
    for (int i = 0; i < kT; ++i) {                       // P2
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r > 0) __builtin_amdgcn_sched_barrier(0);
        t_mfma(i, r, ring[(kP2 + i) % kRing], ta1, ta2);
        vector_t(i, r, tb1, tb2, 1);
      }
      acc_rest(i, kP1);
      refill(kP2 + i);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < kAcc; ++i) {                     // P3
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (r > 0) __builtin_amdgcn_sched_barrier(0);
        vector_tail(i, r, tb1, tb2, 1);
        acc_mfma(i, r, kP3);
      }
      if (!DQ && i == kAcc - 2) read_ld(true, 0, 0, lv[0]);
      if (!DQ && i >= kAcc / 2 && i < kAcc / 2 + 4) read_nd(true, 1, i - kAcc / 2);   // T2 of (t+1, second half): P0 of the next tile
      refill(kP3 + i);
      if (i >= kAcc - kDepth) {                          // the last transposed read of this tile has been issued
#pragma unroll
        for (int a = (i - (kAcc - kDepth)) * KK / kDepth; a < (i + 1 - (kAcc - kDepth)) * KK / kDepth; ++a) tr_a[a] += step1;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    ld_cur = ld_next;
    ld_next += step2;
  }
#pragma unroll
  for (int i = 0; i < kLag; ++i) acc_rest(i, kP3);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zero-filled copies of tiles past the end

  // ---- epilogue: acc^T[d][r] -> rows of the output through LDS --------------------------------------------
  // Nothing overlaps it (the dK / dV pass has a CU to itself), so it waits as rarely as it can: one barrier, after which
  // every wavefront has an area of its own and only the order of its own LDS instructions to rely on.
  __syncthreads();
  auto own_lds_order = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // columns 4 c .. 4 c + 3 of a stationary row: lane (ln, lg) has every c = 64/M u + lg of rows M r + ln
  auto unit = [](const Acc (&acc)[DB][R], int u, int r, float mul) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[4 * u / NR][r][(4 * u + e) % NR] * mul;
    return v;
  };
  constexpr int kUnits = DB * NR / 4;
  auto write_out = [&](const Acc (&acc)[DB][R], float mul, uint16_t* dst, int64_t d_sb, int64_t d_ss,
                       int64_t d_sh, int head) {
    own_lds_order();
    constexpr int kOStride = kRow / 2 + 8;
    unsigned char* os = smem + wave * (32 * kOStride * 2);
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const f32x4 v = unit(acc, u, r, mul);
        *reinterpret_cast<u32x2*>(os + (r * M + ln) * (kOStride * 2) + (64 / M * u + lg) * 8) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      }
    own_lds_order();
    const int chunk = lane & 15;
    uint16_t* op = dst + b * d_sb + head * d_sh + chunk * 8;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int r = (lane >> 4) + 4 * it;
      const int row = r0 + wave * 32 + r;
      if (row < n_st && chunk * 8 < p.D) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(os + r * (kOStride * 2) + chunk * 16);
        *reinterpret_cast<u32x4*>(op + (int64_t)row * d_ss) = w;
      }
    }
  };
  // The same with fp32 rows on the way (512 or 256 bytes, their chunks of 4 columns swizzled by the row).  A lane has 4 or 8
  // columns of a row: a lane's own accumulator columns are 16 bytes of 32 different rows.  `fetch` gives what is there already, all
  // of it on the way before the first store (a load cannot pass a store that may be to the same place, so that one row's after
  // the other cost a round trip each), and `finish` gets the sums and that.  With 4 columns to a lane an instruction covers whole rows
  // without a gap, which the carried dQ of a pass by itself gains from: a step of 8 chunks 4096 x 4096 H32 6838 us to 6790.  Elsewhere
  // half as many rows with twice the work are better: 8 chunks 512 x 512 B4 H5, both passes in one launch, 85.5 us / 87.6 with 4; 8
  // chunks 3131 x 3131 B4 H16 D 80, one launch each, dQ carried 6313 / 6435.
  auto write_out32 = [&](const Acc (&acc)[DB][R], float mul, auto columns, auto&& fetch, auto&& finish) {
    own_lds_order();
    constexpr int kH = decltype(columns)::value / 4, kRow32 = 2 * kRow, kPlaces = kRow32 / 16, kLanes = kPlaces / kH;
    constexpr int kRowsAtOnce = 64 / kLanes, kIts = 32 / kRowsAtOnce;
    unsigned char* os = smem + wave * (32 * kRow32);
    const int place = lane % kLanes * kH, col = place * 4, first_row = r0 + wave * 32 + lane / kLanes;
    f32x4 old[kIts][kH];
#pragma unroll
    for (int it = 0; it < kIts; ++it) {
#pragma unroll
      for (int h = 0; h < kH; ++h) old[it][h] = f32x4{};
      if (first_row + it * kRowsAtOnce < n_st && col < p.D)
#pragma unroll
        for (int h = 0; h < kH; ++h) old[it][h] = fetch(first_row + it * kRowsAtOnce, col + 4 * h);
    }
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int row = r * M + ln;
        *reinterpret_cast<f32x4*>(os + row * kRow32 + (((64 / M * u + lg) ^ (row % kPlaces)) << 4)) = unit(acc, u, r, mul);
      }
    own_lds_order();
#pragma unroll
    for (int it = 0; it < kIts; ++it) {
      const int r = lane / kLanes + kRowsAtOnce * it;
      if (first_row + it * kRowsAtOnce < n_st && col < p.D) {
        f32x4 v[kH];
#pragma unroll
        for (int h = 0; h < kH; ++h) v[h] = *reinterpret_cast<const f32x4*>(os + r * kRow32 + (((place + h) ^ (r % kPlaces)) << 4));
        finish(v, old[it], first_row + it * kRowsAtOnce, col);
      }
    }
  };
  const std::integral_constant<int, 8> eight;
  auto pack4 = [](const f32x4& v) { return u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])}; };
  auto pack8 = [=](const f32x4 (&v)[2]) {
    const u32x2 lo = pack4(v[0]), hi = pack4(v[1]);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  auto nothing = [](int, int) { return f32x4{}; };
  if (SPLIT && w.splits > 1) {
    // fp32 sums for bwd_reduce, (b, row, head, column) like the gradient itself
    const int64_t size = (int64_t)p.B * n_st * (DQ ? p.Hq : p.Hkv) * p.D;
    auto part = [&](float* base) {
      return [=](const f32x4 (&v)[2], const f32x4 (&)[2], int row, int col) {
        f32x4* op = reinterpret_cast<f32x4*>(base + split * size + (((int64_t)b * n_st + row) * (DQ ? p.Hq : p.Hkv) + hs) * p.D + col);
        op[0] = v[0];
        op[1] = v[1];
      };
    };
    write_out32(acc1, p.scale, eight, nothing, part(w.partial));
    if (!DQ) write_out32(acc2, 1.f, eight, nothing, part(w.partial + w.splits * size));
  } else if (DQ) {
    if (p.dq_acc == nullptr) {
      write_out(acc1, p.scale, p.dq, p.dq_sb, p.dq_ss, p.dq_sh, hs);
    } else {
      uint16_t* dq = p.dq ? p.dq + b * p.dq_sb + hs * p.dq_sh : nullptr;
      auto at = [&](int row, int col) { return reinterpret_cast<f32x4*>(p.dq_acc + (((int64_t)b * p.Sq + row) * p.Hq + hs) * p.D + col); };
      constexpr int kH = WAVES == 8 ? 1 : 2;
      auto put16 = [=](int row, int col, const f32x4 (&v)[kH]) {
        uint16_t* to = dq + (int64_t)row * p.dq_ss + col;
        if constexpr (kH == 1) *reinterpret_cast<u32x2*>(to) = pack4(v[0]);
        else *reinterpret_cast<u32x4*>(to) = pack8(v);
      };
      write_out32(acc1, p.scale, std::integral_constant<int, 4 * kH>(),
                  [&](int row, int col) { return p.dq_mode != kDqFirst ? *at(row, col) : f32x4{}; },
                  [&](const f32x4 (&v)[kH], const f32x4 (&old)[kH], int row, int col) {
        if (p.dq_mode == kDqAdd && dq) put16(row, col, v);
        f32x4 sum[kH];
#pragma unroll
        for (int h = 0; h < kH; ++h) sum[h] = p.dq_mode != kDqFirst ? v[h] + old[h] : v[h];
        if (p.dq_mode == kDqLast) return put16(row, col, sum);
#pragma unroll
        for (int h = 0; h < kH; ++h) *at(row, col + 4 * h) = sum[h];
      });
    }
  } else if ((CHUNKS ? chunks->dk32[chunk] : p.dk32) == nullptr) {
    write_out(acc1, p.scale, CHUNKS ? chunks->dk[chunk] : p.dk, p.dk_sb, p.dk_ss, p.dk_sh, hs);
    write_out(acc2, 1.f, CHUNKS ? chunks->dv[chunk] : p.dv, p.dk_sb, p.dk_ss, p.dk_sh, hs);
  } else {
    auto store = [&](float* out32, uint16_t* out16) {
      return [=](const f32x4 (&v)[2], const f32x4 (&)[2], int row, int col) {
        const u32x4 w = pack8(v);
        f32x4* op = reinterpret_cast<f32x4*>(out32 + (((int64_t)b * p.Sc + row) * p.Hkv + hs) * p.D + col);
        op[0] = f32x4{bf16_lo(w[0]), bf16_hi(w[0]), bf16_lo(w[1]), bf16_hi(w[1])};
        op[1] = f32x4{bf16_lo(w[2]), bf16_hi(w[2]), bf16_lo(w[3]), bf16_hi(w[3])};
        if (out16) *reinterpret_cast<u32x4*>(out16 + b * p.dk_sb + (int64_t)row * p.dk_ss + hs * p.dk_sh + col) = w;
      };
    };
    write_out32(acc1, p.scale, eight, nothing, store(CHUNKS ? chunks->dk32[chunk] : p.dk32, CHUNKS ? chunks->dk[chunk] : p.dk));
    write_out32(acc2, 1.f, eight, nothing, store(CHUNKS ? chunks->dv32[chunk] : p.dv32, CHUNKS ? chunks->dv[chunk] : p.dv));
  }
}

template <bool DQ, bool CAUSAL, int KK, bool PREPARED, int M>
__global__ __launch_bounds__(DQ ? 512 : 256, !DQ && KK == 4 ? 2 : 1) void bwd_main(const BwdParams p, const TileMap w) {
  constexpr int kWaves = DQ ? 8 : 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytesOf<DQ, kWaves, KK>];
  bwd_pass<DQ, CAUSAL, KK, kWaves, PREPARED, false, false, M>(p, w, (int)blockIdx.x, smem);
}

// A pass over several chunks of a step: the same chains of tiles as in bwd_joint_chunks, where each pass alone fills the chip.
template <bool DQ, int KK, bool PREPARED, int M>
__global__ __launch_bounds__(DQ ? 512 : 256, !DQ && KK == 4 ? 2 : 1) void bwd_main_chunks(const BwdParams p, const TileMap w, const Chunks chunks) {
  constexpr int kWaves = DQ ? 8 : 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytesOf<DQ, kWaves, KK>];
  bwd_pass<DQ, false, KK, kWaves, PREPARED, false, true, M>(p, w, (int)blockIdx.x, smem, &chunks);
}

// Both passes side by side, for launches that leave CUs idle one after the other.
template <bool CAUSAL, int KK, bool SPLIT>
__global__ __launch_bounds__(256, KK == 4 ? 2 : 1) void bwd_joint(const BwdParams p, const TileMap wq, const TileMap wk) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytesOf<false, 4, KK>];
  static_assert(kSmemBytesOf<true, 4, KK> + 1024 <= kSmemBytesOf<false, 4, KK>, "one array for both, and lse2 and delta of the dQ rows");
  const int i = (int)blockIdx.x - wk.first;
  if (i >= 0 && i < wk.per_xcd * 8) bwd_pass<false, CAUSAL, KK, 4, true, SPLIT>(p, wk, i, smem);
  else bwd_pass<true, CAUSAL, KK, 4, true, SPLIT>(p, wq, (int)blockIdx.x - wq.first, smem);
}

// The same for several chunks of a step.
template <int KK, bool SPLIT>
__global__ __launch_bounds__(256, KK == 4 ? 2 : 1) void bwd_joint_chunks(const BwdParams p, const TileMap wq, const TileMap wk, const Chunks chunks) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[kSmemBytesOf<false, 4, KK>];
  const int i = (int)blockIdx.x - wq.first;
  if (i >= 0 && i < wq.per_xcd * 8) bwd_pass<true, false, KK, 4, true, SPLIT, true>(p, wq, i, smem, &chunks);
  else bwd_pass<false, false, KK, 4, true, false, true>(p, wk, (int)blockIdx.x - wk.first, smem, &chunks);
}

// lse2 and delta for bwd_joint: 16 lanes per query row.
__global__ __launch_bounds__(256) void bwd_prepare(const BwdParams p, int rows) {
  const int i = blockIdx.x * 16 + (threadIdx.x >> 4), col = (threadIdx.x & 15) * 8;
  const int at = i < rows ? i : rows - 1;
  const int h = at % p.Hq, bs = at / p.Hq, srow = bs % p.Sq, b = bs / p.Sq;
  float part = 0.f;
  if (col < p.D) {
    const bf16x8 d8 = *reinterpret_cast<const bf16x8*>(p.dout + b * p.q_sb + (int64_t)srow * p.q_ss + h * p.q_sh + col);
    const bf16x8 o8 = *reinterpret_cast<const bf16x8*>(p.out + b * p.o_sb + (int64_t)srow * p.o_ss + h * p.o_sh + col);
#pragma unroll
    for (int j = 0; j < 8; ++j) part = __builtin_fmaf((float)d8[j], (float)o8[j], part);
  }
  const float delta = row16_sum(part);
  if (i < rows && col == 0) {
    const int64_t r = ((int64_t)b * p.Hq + h) * p.Sq + srow;
    const float l = p.lse[r];
    p.lse2[r] = (l == -INFINITY) ? INFINITY : l * kLog2e;
    p.delta[r] = -delta;
    if (p.softmax_d) p.softmax_d[r] = delta;
  }
}

// The sums of the workgroups that shared a stationary tile, added in the order of their parts, and stored the way the
// pass itself would have: 16 lanes per row, 8 columns each.  Rows of dQ first (if that pass was split), then of dK and dV.
__global__ __launch_bounds__(256) void bwd_reduce(const BwdParams p, const TileMap wq, const TileMap wk, int q_rows, int kv_rows) {
  int row = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int col = (threadIdx.x & 15) * 8;
  if (row >= q_rows + 2 * kv_rows || col >= p.D) return;
  const bool is_q = row < q_rows;
  const bool is_v = row >= q_rows + kv_rows;
  row -= is_q ? 0 : is_v ? q_rows + kv_rows : q_rows;
  const int heads = is_q ? p.Hq : p.Hkv, seq = is_q ? p.Sq : p.Sc, splits = is_q ? wq.splits : wk.splits;
  const int64_t size = (int64_t)p.B * seq * heads * p.D, at = (int64_t)row * p.D + col;
  const float* src = (is_q ? wq.partial : wk.partial) + (is_v ? splits * size : 0) + at;
  f32x4 v[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int i = 0; i < splits; ++i) {
    const f32x4* part = reinterpret_cast<const f32x4*>(src + i * size);
    v[0] += part[0];
    v[1] += part[1];
  }
  auto pack8 = [](const f32x4 (&x)[2]) {
    return u32x4{pack_bf16(x[0][0], x[0][1]), pack_bf16(x[0][2], x[0][3]), pack_bf16(x[1][0], x[1][1]), pack_bf16(x[1][2], x[1][3])};
  };
  const int h = row % heads, srow = row / heads % seq, b = row / heads / seq;
  if (is_q) {
    u32x4* qp = reinterpret_cast<u32x4*>(p.dq + b * p.dq_sb + (int64_t)srow * p.dq_ss + h * p.dq_sh + col);
    if (p.dq_acc == nullptr || (p.dq_mode == kDqAdd && p.dq)) *qp = pack8(v);
    if (p.dq_acc == nullptr) return;
    f32x4* ap = reinterpret_cast<f32x4*>(p.dq_acc + at);
    if (p.dq_mode != kDqFirst) { v[0] += ap[0]; v[1] += ap[1]; }
    if (p.dq_mode != kDqLast) { ap[0] = v[0]; ap[1] = v[1]; }
    else *qp = pack8(v);
  } else {
    const u32x4 x = pack8(v);
    if (p.dk32) {
      f32x4* op = reinterpret_cast<f32x4*>((is_v ? p.dv32 : p.dk32) + at);
      op[0] = f32x4{bf16_lo(x[0]), bf16_hi(x[0]), bf16_lo(x[1]), bf16_hi(x[1])};
      op[1] = f32x4{bf16_lo(x[2]), bf16_hi(x[2]), bf16_lo(x[3]), bf16_hi(x[3])};
    }
    uint16_t* out16 = is_v ? p.dv : p.dk;
    if (out16) *reinterpret_cast<u32x4*>(out16 + b * p.dk_sb + (int64_t)srow * p.dk_ss + h * p.dk_sh + col) = x;
  }
}

}  // namespace
}  // namespace mhip

using namespace mhip;

// Scratch of the entry point that allocates nothing: delta and lse2 of up to kScratchRows (batch, head, row)
// triples, and the sums of split passes.  Every GPU the library runs on holds its own copy until the process ends.
constexpr int64_t kScratchRows = int64_t(1) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchRows * 8 + 32 + (int64_t(32) << 20)];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device.  In host code the array's name is only a handle for
// the runtime: the address a kernel can use comes from hipGetSymbolAddress, once per device.
int scratch_address(void** ptr) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return MHIP_ERUNTIME;
  void* cached = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (cached == nullptr) {
    void* fresh = nullptr;
    if (hipGetSymbolAddress(&fresh, HIP_SYMBOL(scratch)) != hipSuccess || fresh == nullptr) {
      (void)hipGetLastError();
      return MHIP_ERUNTIME;
    }
    g_scratch_ptr[dev].store(fresh, std::memory_order_release);   // every thread would store the same address
    cached = fresh;
  }
  *ptr = cached;
  return MHIP_OK;
}

TileMap tile_map(int heads, int seq, int rows, int splits = 1, float* partial = nullptr) {
  TileMap w;
  w.splits = splits;
  for (w.log_splits = 0; (1 << w.log_splits) < splits; ++w.log_splits) {}
  w.partial = partial;
  w.n_tiles = (seq + rows - 1) / rows * splits;
  w.total = heads * w.n_tiles;
  w.per_xcd = (w.total + 7) / 8;
  w.first = 0;
  w.heads_per_xcd = heads % 8 == 0 ? heads / 8 : 0;
  w.by_tiles = Divisor(w.n_tiles);
  w.by_order = Divisor(w.heads_per_xcd > 0 ? w.heads_per_xcd : heads);
  return w;
}

// The order of the passes in a joint launch: the one with the longer chains of tiles first (tq and tk tiles at most, of three and
// four products each), so that the short ones fill the tail.  Us, where it is the other one than dK / dV for a block, dQ for
// several, whose workgroups came first whatever their chains (before / this):
//     1237 x 8192 B2 H16  590 / 510     700 x 6000 H24 D64  114 / 98.0    1024 x 16384 H16  430 / 421     512 x 8192 H8  77.0 / 75.5
//     2 chunks  7430 x 7430 H8/1  1710 / 1417     12000 x 12000 H4/1  1970 / 1690     2048 x 2048 H32/4 D64  325 / 280
void longest_first(TileMap& wq, TileMap& wk, float tq, float tk) {
  if (4.f * tk >= 3.f * tq) wq.first = wk.per_xcd * 8;
  else wk.first = wq.per_xcd * 8;
}

// Estimated time (us) of n workgroups that visit `most` tiles at most and `mean` on average, one workgroup per CU at a
// time: `fixed` per workgroup and `step` per tile, plus `busy` times the share of the CUs at work (clock and L2).  On 64
// columns two workgroups of four wavefronts share a CU, so the estimate is too high there (causal 1500 x 1500 B2 H12: 50 us,
// where the whole backward takes 41); what plan_block and group_chunks choose by it is measured beside the other choices.
struct Cost { float fixed, step, busy; };
float launch_time(float n, float mean, float most, const Cost& c) {
  const float full = floorf(n / 256.f), part = n / 256.f - full;
  const float share = n < 256.f ? part : 1.f;
  const float longest = c.fixed + most * (c.step + share * c.busy);
  float spread = full * (c.fixed + mean * (c.step + c.busy));
  if (part > 0.f) spread += c.fixed + mean * (c.step + part * c.busy);
  return longest > spread ? longest : spread;
}

// How a block runs.  Both passes go into one launch (joint), behind a small one that prepares delta and lse2, while one
// pass alone leaves CUs idle (its dQ wavefronts run one per SIMD instead of two, which costs 4 % once the chip is full).
// Costs fitted to the measured block times, us (two launches / one):
//     B1 H4   256 x 256     23.0 / 12.3      B4 H5    512 x 512    35.1 / 19.7      B1 H2 4096 x 4096   183 / 89.8
//     B1 H32 1024 x 1024    70.6 / 64.1      B1 H16 2048 x 2048     122 /  109      B1 H32 2048 x 2048  205 / 214
//     B1 H32 4096 x 4096     756 /  786      causal: B1 H8 2048 x 2048  103 / 52.3, B1 H32 4096 x 4096  424 / 439
// In one launch a stationary tile may further be shared by several workgroups (sq of the dQ pass, sk of the dK / dV pass),
// where one workgroup's chain of tiles -- with grouped heads, all query heads of the group -- is what the launch waits for;
// their sums meet in a third launch (one / with it):
//     B1 H8/1 512 x 512      82.6 / 27.6     B1 H8/1 2048 x 2048    310 / 73.6     B1 H8/1 4096 x 4096   636 /  221
//     B1 H2/2 4096 x 4096    85.2 / 69.8     B1 H32/4 2048 x 2048   338 /  220
// On 64 columns, where the costs are those of one workgroup per CU (two launches / one, * the form chosen):
//     B1 H4   256 x 256     17.0 / 10.4*     B4 H5    512 x 512    24.5 / 15.0*     B1 H16 2048 x 2048  74.1 / 61.4*
//     B2 H12 1500 x 1500    71.0 / 66.8*     B1 H32 2048 x 2048   117* / 121        B1 H32 4096 x 4096  442* / 448
//     causal: B2 H12 1500 x 1500  60.7 / 40.8*                                      B1 H32 4096 x 4096  249* / 247
// and one / shared by as many workgroups (sq, sk) as chosen: H8/1 2048 x 2048 226 / 46.0 (1, 8), H32/4 247 / 125 (1, 4), H2/2
// 4096 x 4096 63.1 / 48.0 (2, 2), where 44.2 (4, 4) would be better.
Cost dq_cost(int D) { return D <= 64 ? Cost{6.f, 0.95f, 0.45f} : Cost{7.f, 1.45f, 0.75f}; }       // 96 columns: the costs of
Cost dkv_cost(int D) { return D <= 64 ? Cost{6.f, 0.75f, 0.25f} : Cost{7.f, 1.15f, 0.55f}; }      // 128, of which all save the same 12 %
Cost joint_cost(int D) { return D <= 64 ? Cost{6.f, 0.75f, 0.12f} : Cost{7.f, 1.15f, 0.29f}; }
struct Plan { bool joint; int sq, sk; float time; };       // time: estimated, without preparing delta and lse2
constexpr int64_t kPartialMost = int64_t(32) << 20;     // bytes of sums a block may leave for bwd_reduce
int64_t partial_bytes(int B, int S, int H, int D, int tensors, int splits) {
  return splits > 1 ? (int64_t)B * S * H * D * 4 * tensors * splits : 0;
}
Plan plan_block(int B, int Sq, int Sc, int Hq, int Hkv, int D, bool causal) {
  Plan best = {false, 1, 1, 0.f};
  if (Sq == 0 || Sc == 0 || B == 0) return best;
  const Cost dq8 = dq_cost(D), dkv = dkv_cost(D), both = joint_cost(D);
  constexpr float kPrepare = 5.f, kReduce = 4.f, kBytesPerUs = 4e6f;
  const float tq = (float)((Sc + kTile - 1) / kTile), tk = (float)((Sq + kTile - 1) / kTile) * (Hq / Hkv);
  const float half = causal ? 0.53f : 1.f;          // mean share of the tiles under the diagonal
  const float nq8 = (float)tile_map(B * Hq, Sq, kRowsQ).total, nq4 = (float)tile_map(B * Hq, Sq, kRowsQ / 2).total;
  const float nk = (float)tile_map(B * Hkv, Sc, kRowsKv).total;
  float best_time = launch_time(nq8, half * tq, tq, dq8) + launch_time(nk, half * tk, tk, dkv);
  for (int sq = 1; sq <= 16; sq *= 2)
    for (int sk = 1; sk <= 16; sk *= 2) {
      if ((sq > 1 && tq < 2.f * sq) || (sk > 1 && tk < 2.f * sk)) continue;
      const int64_t bytes = partial_bytes(B, Sq, Hq, D, 1, sq) + partial_bytes(B, Sc, Hkv, D, 2, sk);
      if (bytes > kPartialMost) continue;
      const float n = nq4 * sq + nk * sk, mean = half * (nq4 * tq + nk * tk) / n;
      const float most = tq / sq > tk / sk ? tq / sq : tk / sk;
      const float time = kPrepare + launch_time(n, mean, most, both) + (bytes > 0 ? kReduce + 2.f * (float)bytes / kBytesPerUs : 0.f);
      if (time < best_time) { best_time = time; best = {true, sq, sk, 0.f}; }
    }
  best.time = best_time - (best.joint ? kPrepare : 0.f);
  return best;
}

// Estimated time (us) of one launch of both passes over n chunks, if it may have so many workgroups.
float joint_chunks_time(int B, int Sq, int Sc, int Hq, int Hkv, int D, int n, int most) {
  const int64_t nq = tile_map(B * Hq, Sq, kRowsQ / 2).total, nk = tile_map(B * Hkv, Sc, kRowsKv).total;
  const int64_t workgroups = nq + n * nk;
  if (n > kMaxGroup || workgroups > most) return INFINITY;
  const float tq = (float)((Sc + kTile - 1) / kTile), tk = (float)((Sq + kTile - 1) / kTile) * (Hq / Hkv);
  const Cost c = joint_cost(D);
  const float share = workgroups < 256 ? (float)workgroups / 256.f : 1.f, step = c.step + share * c.busy;
  const float longest = c.fixed + (n * tq > tk ? n * tq : tk) * step;
  const float spread = (nq * (c.fixed + n * tq * step) + n * nk * (c.fixed + tk * step)) / 256.f;
  return longest > spread ? longest : spread;
}
// Where both passes fill the chip one after the other, each has a launch over the chunks (apart): the dQ pass keeps its eight
// wavefronts, and its workgroups' ends and the carried sum come once here too.  Us a step, without / with:
//     8 chunks 4096 x 4096 H32     6453 / 6175      2048 x 2048 H32     1820 / 1641      1024 x 1024 B2 H32    1118 /  931
//     512 x 512 B4 H32              757 /  585      6000 x 600 H32      2016 / 1439      2048 x 2048 H32 D64   1004 /  891
//     4 chunks 1024 x 1024 H64      560 /  474      4096 x 4096 H32/8   3121 / 2986      8192 x 8192 H8        3089 / 3013
// and where the estimate expects more of other forms, what they take / both passes apart:
//     8 chunks 1024 x 1024 H32      459 /  491      2048 x 2048 H16      821 /  874      4 chunks 3000 x 3000 H24 D96  1091 / 1202
//     8 chunks 1536 x 1536 H32      953 /  934      2 chunks 7430 x 7430 H8/1  1417 / 1586
// (the costs are those of 32 x 32 MFMA tiles, with which the dQ pass took 5 % longer)
float apart_chunks_time(int B, int Sq, int Sc, int Hq, int Hkv, int D, int n) {
  if (n > kMaxGroup) return INFINITY;
  const float tq = (float)((Sc + kTile - 1) / kTile), tk = (float)((Sq + kTile - 1) / kTile) * (Hq / Hkv);
  const float nq = (float)tile_map(B * Hq, Sq, kRowsQ).total, nk = (float)tile_map(B * Hkv, Sc, kRowsKv).total;
  return launch_time(nq, n * tq, n * tq, dq_cost(D)) + launch_time(n * nk, tk, tk, dkv_cost(D));
}
// Workgroups of a launch of both passes where those of each pass would leave CUs idle, which
// has more to fill it with the more chunks there are.  Us a step, up to kGroupWorkgroups / this many:
//     8 chunks 1024 x 1024 H32      480 /  455      2048 x 2048 H16   840 /  816     700 x 700 B2 H20    345 /  325
//              1536 x 1536 H32      996 /  975      4096 x 4096 H8   1573 / 1562     6000 x 6000 H5     2172 / 2187 (not taken)
//     4 chunks 3000 x 3000 H24 D96 1121 / 1099      3072 x 3072 H24  1390 / 1365     1500 x 1500 H48 D64  394 /  380
constexpr int kStepWorkgroups = 4096;
// More chunks to a launch than kGroupWorkgroups allow stay out with less than this to gain by the estimate, which expects 0.3 %
// for the one case above that loses 0.7 %.  It is off by 15 % and more elsewhere (2 chunks 7430 x 7430 H8/1: 1355 us expected, 1417
// measured; both passes apart 1832 and 1586), so the line tells the measured cases apart and promises nothing for others.
constexpr float kLongerLaunch = 0.996f;
bool chunks_apart(int B, int Sq, int Sc, int Hq, int Hkv, int D, int n) {
  return apart_chunks_time(B, Sq, Sc, Hq, Hkv, D, n) < joint_chunks_time(B, Sq, Sc, Hq, Hkv, D, n, kStepWorkgroups);
}
// Chunks of a step that go together: the number of which the estimate expects the least time for the step, in launches of both
// passes of up to kStepWorkgroups workgroups or in a launch of each (not `step`: of both passes and up to kGroupWorkgroups
// alone).  Together the chunks fill the chip, and dQ's workgroups load their rows and meet the carried
// sum once per launch instead of once per chunk; against it stands that a dQ workgroup's chain of tiles is as many times as
// long.  Us a step, chunk by chunk / in launches of 2 / 4 / 8:
//     8 chunks 512 x 512 B4 H5      162 /  117 / 95.8 / 89.5      1024 x 1024 H32                557 /  497 /  465 /  448
//     256 x 256 H16                 104 / 67.2 / 56.8 / 52.3      512 x 512 H8/1                 201 /  337 /  174 / 90.2
//     1237 x 1237 B2 H16/8 D80      632 /  605 /  510 /  499
// D 64, * the number chosen:
//     8 chunks 512 x 512 B4 H5      114 / 84.6 / 71.7 / 62.3*     1024 x 1024 H32                299 /  297 / 249* / 240
//     256 x 256 H16                91.7 / 61.8 / 52.9 / 48.6*     512 x 512 H8/1                 154 /  248 /  128 / 65.4*
//     1500 x 1500 B2 H12            558 /  446 / 405* / 392       700 x 700 H12                  136 / 98.6 / 88.0 / 77.9*
int group_chunks(int B, int Sq, int Sc, int Hq, int Hkv, int D, int chunks, bool step) {
  if (B == 0 || Sq == 0 || Sc == 0) return 1;
  int best = 1;
  float best_time = plan_block(B, Sq, Sc, Hq, Hkv, D, false).time * chunks;
  for (int launches = chunks; launches >= 1; --launches) {
    const int n = (chunks + launches - 1) / launches;
    if (n > kMaxGroup) break;
    const float joint = joint_chunks_time(B, Sq, Sc, Hq, Hkv, D, n, step ? kStepWorkgroups : kGroupWorkgroups);
    const float apart = step ? apart_chunks_time(B, Sq, Sc, Hq, Hkv, D, n) : INFINITY;
    const bool longer = joint < apart && joint_chunks_time(B, Sq, Sc, Hq, Hkv, D, n, kGroupWorkgroups) == INFINITY;
    const float time = ((chunks + n - 1) / n) * (apart < joint ? apart : joint);
    if (n > 1 && time < (longer ? kLongerLaunch : 1.f) * best_time) { best_time = time; best = n; }
  }
  return best;
}

// Workgroups that share a query tile of the dQ pass in a launch over n chunks, each with its part of them: the chain of tiles
// over all chunks is what a launch waits for whose other workgroups leave CUs idle or are soon done.  Their sums meet in
// bwd_reduce.  Us a step, one workgroup to a tile / as many as chosen:
//     8 chunks 512 x 512 H4     67.1 / 31.4      200 x 200 H2   39.9 / 20.1      1024 x 1024 H8  141 / 121
//     4 chunks 1024 x 1024 H4   68.3 / 42.7      256 x 256 H4   22.3 / 18.7 (not taken, see below)
//     D 64  8 chunks 1024 x 1024 H8  105 / 71.9  700 x 700 H12  77.1 / 61.4      256 x 256 H16  32.7 / 23.7
// Not where the chip is full of other work (two to a tile): 8 chunks 512 x 512 B4 H5 91.2 / 96.9, or where the keys' workgroups
// take as long: 3 chunks 997 x 997 B2 H4/2 60.5 / 62.5 (a tile of the dQ pass is three products to the other's four; the two
// workgroups of a CU on 64 columns take turns, which costs it as much), 2 chunks 564 x 564 H8 D 80 30.0 / 30.8.
// The third launch costs the host 3.5 us.  A step that the GPU is done with before the host has launched the next one (which takes it
// 20 us and 3.5 for each chunk) is so much longer among others, so there it has to save the GPU twice that: 8 chunks 128 x 128
// H16, one workgroup / four, replayed as a graph 32.0 / 28.0, alone 77 / 73, among others 48 / 51.2.
int chunk_splits(int B, int Sq, int Sc, int Hq, int Hkv, int D, int n) {
  const float nq = (float)tile_map(B * Hq, Sq, kRowsQ / 2).total, nk = (float)n * tile_map(B * Hkv, Sc, kRowsKv).total;
  const float tq = (float)((Sc + kTile - 1) / kTile), tk = (float)((Sq + kTile - 1) / kTile) * (Hq / Hkv);
  const Cost c = joint_cost(D);
  const float turn = D <= 64 ? 1.f : 7.f;      // us between the workgroups of a CU (on 64 columns the other one runs on)
  const float products = D <= 64 ? 1.f : 0.75f;
  const float host = 20.f + 3.5f * n;
  int best = 1;
  float best_time = 0.f;
  for (int s = 1; s <= n; s *= 2) {
    const int64_t bytes = partial_bytes(B, Sq, Hq, D, 1, s);
    if (bytes > kPartialMost) break;
    const float share = nq * s + nk < 256.f ? (nq * s + nk) / 256.f : 1.f, step = c.step + share * c.busy;
    const float chain = c.fixed + (n + s - 1) / s * tq * step * products, keys = c.fixed + tk * step;
    const float longest = chain > keys ? chain : keys, spread = (nq * s * (chain + turn) + nk * (keys + turn)) / 256.f;
    const float time = (longest > spread ? longest : spread) + (s > 1 ? 4.f + 2.f * (float)bytes / 4e6f : 0.f);
    const float less = best == 1 && best_time < host ? 7.f : 0.f;
    if (s == 1 || (time < 0.95f * best_time && time < best_time - less)) { best = s; best_time = time; }
  }
  return best;
}

// Whether the dQ pass of eight wavefronts, with workgroups of `tiles` key tiles each (causal: at most), uses 16 x 16 MFMA tiles: where
// it keeps every CU busy for long enough, its time is the board's power.  The pass alone, us, 32 x 32 / 16 x 16 (workgroups x tiles):
//     D 128  512 x 64  327 / 311    256 x 32  87.7 / 83.8    192 x 64  131 / 133      causal  512 x 64  183 / 174   1024 x 32  209 / 207
//     D 96   512 x 64  255 / 247    256 x 32  65.4 / 63.7                             causal  512 x 64  144 / 141
bool small_tiles(const TileMap& w, bool causal, int64_t tiles) {
  const int64_t rounds = ((int64_t)w.total + 255) / 256;
  return tiles >= 32 && (causal ? w.total >= 512 : (int64_t)w.total * 20 >= rounds * 256 * 17);
}

bool small_dq(int B, int Sq, int Sc, int Hq, int D, bool causal, int chunks) {
  return D > 64 && small_tiles(tile_map(B * Hq, Sq, kRowsQ), causal, (int64_t)chunks * ((Sc + kTile - 1) / kTile));
}

// dQ (and, unless prepared, delta / lse2 for both passes): one workgroup per 256 query rows; has to run before the dK / dV pass
template <bool CAUSAL, int KK, bool PREPARED>
void launch_dq(const BwdParams& p, hipStream_t st) {
  const TileMap w = tile_map(p.B * p.Hq, p.Sq, kRowsQ);
  const dim3 grid(w.per_xcd * 8), block(512);
  if constexpr (KK > 4)
    if (small_dq(p.B, p.Sq, p.Sc, p.Hq, p.D, CAUSAL, 1)) {
      hipLaunchKernelGGL((bwd_main<true, CAUSAL, KK, PREPARED, 16>), grid, block, 0, st, p, w);
      return;
    }
  hipLaunchKernelGGL((bwd_main<true, CAUSAL, KK, PREPARED, 32>), grid, block, 0, st, p, w);
}

template <bool CAUSAL, int KK>
void launch_bwd(const BwdParams& p, const Plan& plan, float* partial, hipStream_t st) {
  if (plan.joint) {
    const int rows = p.B * p.Hq * p.Sq;
    if (!p.prepared) hipLaunchKernelGGL(bwd_prepare, dim3((rows + 15) / 16), dim3(256), 0, st, p, rows);
    TileMap wq = tile_map(p.B * p.Hq, p.Sq, kRowsQ / 2, plan.sq, partial);
    TileMap wk = tile_map(p.B * p.Hkv, p.Sc, kRowsKv, plan.sk, partial + partial_bytes(p.B, p.Sq, p.Hq, p.D, 1, plan.sq) / 4);
    longest_first(wq, wk, (float)((p.Sc + kTile - 1) / kTile) / plan.sq, (float)((p.Sq + kTile - 1) / kTile) * p.group / plan.sk);
    const dim3 grid((wk.per_xcd + wq.per_xcd) * 8), block(256);
    // (a kernel of its own: the bookkeeping of shared tiles costs 0.6 us where there are none)
    if (plan.sq > 1 || plan.sk > 1) hipLaunchKernelGGL((bwd_joint<CAUSAL, KK, true>), grid, block, 0, st, p, wq, wk);
    else hipLaunchKernelGGL((bwd_joint<CAUSAL, KK, false>), grid, block, 0, st, p, wq, wk);
    const int q_rows = plan.sq > 1 ? p.B * p.Sq * p.Hq : 0, kv_rows = plan.sk > 1 ? p.B * p.Sc * p.Hkv : 0;
    if (q_rows + kv_rows > 0)
      hipLaunchKernelGGL(bwd_reduce, dim3((q_rows + 2 * kv_rows + 15) / 16), dim3(256), 0, st, p, wq, wk, q_rows, kv_rows);
    return;
  }
  if (p.Sq > 0) p.prepared ? launch_dq<CAUSAL, KK, true>(p, st) : launch_dq<CAUSAL, KK, false>(p, st);
  // dK, dV: one workgroup per 128 keys of one kv head
  if (p.Sc > 0) {
    const TileMap wk = tile_map(p.B * p.Hkv, p.Sc, kRowsKv);
    hipLaunchKernelGGL((bwd_main<false, CAUSAL, KK, true, 32>), dim3(wk.per_xcd * 8), dim3(256), 0, st, p, wk);
  }
}

template <int KK, bool PREPARED>
void launch_dq_chunks(const BwdParams& p, const Chunks& chunks, hipStream_t st) {
  const TileMap w = tile_map(p.B * p.Hq, p.Sq, kRowsQ);
  const dim3 grid(w.per_xcd * 8), block(512);
  if constexpr (KK > 4)
    if (small_dq(p.B, p.Sq, p.Sc, p.Hq, p.D, false, chunks.n)) {
      hipLaunchKernelGGL((bwd_main_chunks<true, KK, PREPARED, 16>), grid, block, 0, st, p, w, chunks);
      return;
    }
  hipLaunchKernelGGL((bwd_main_chunks<true, KK, PREPARED, 32>), grid, block, 0, st, p, w, chunks);
}

template <int KK>
void launch_chunks(const BwdParams& p, const Chunks& chunks, float* partial, hipStream_t st) {
  if (chunks_apart(p.B, p.Sq, p.Sc, p.Hq, p.Hkv, p.D, chunks.n)) {
    p.prepared ? launch_dq_chunks<KK, true>(p, chunks, st) : launch_dq_chunks<KK, false>(p, chunks, st);
    const TileMap wk = tile_map(chunks.n * p.B * p.Hkv, p.Sc, kRowsKv);
    hipLaunchKernelGGL((bwd_main_chunks<false, KK, true, 32>), dim3(wk.per_xcd * 8), dim3(256), 0, st, p, wk, chunks);
    return;
  }
  const int rows = p.B * p.Hq * p.Sq;
  if (!p.prepared) hipLaunchKernelGGL(bwd_prepare, dim3((rows + 15) / 16), dim3(256), 0, st, p, rows);
  const int splits = chunk_splits(p.B, p.Sq, p.Sc, p.Hq, p.Hkv, p.D, chunks.n);
  TileMap wq = tile_map(p.B * p.Hq, p.Sq, kRowsQ / 2, splits, partial);
  TileMap wk = tile_map(chunks.n * p.B * p.Hkv, p.Sc, kRowsKv);
  longest_first(wq, wk, (float)((chunks.n + splits - 1) / splits) * ((p.Sc + kTile - 1) / kTile), (float)((p.Sq + kTile - 1) / kTile) * p.group);
  const dim3 grid((wk.per_xcd + wq.per_xcd) * 8), block(256);
  if (splits > 1) hipLaunchKernelGGL((bwd_joint_chunks<KK, true>), grid, block, 0, st, p, wq, wk, chunks);
  else hipLaunchKernelGGL((bwd_joint_chunks<KK, false>), grid, block, 0, st, p, wq, wk, chunks);
  if (splits > 1) hipLaunchKernelGGL(bwd_reduce, dim3((rows + 15) / 16), dim3(256), 0, st, p, wq, wk, rows, 0);
}

// -delta, lse2 and delta, (B, Hq, Sq) fp32 each, every one starting on a 16-byte boundary
int64_t row_bytes(int B, int Sq, int Hq) { return ((((int64_t)B * Hq * Sq + 3) & ~int64_t(3)) * 3) * 4; }
}  // namespace

// The same for chunks of every length and for every Hkv and D: plan_block leaves at most kPartialMost bytes of sums whatever
// they are, and a caller may keep one workspace for all chunks its query rows meet (no argument of a call says how large
// it is).
extern "C" int64_t mhip_attn_bwd_workspace_bytes(int B, int Sq, int Sc, int Hq, int Hkv, int D) {
  (void)D;
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0) return 0;
  const int64_t rows = row_bytes(B, Sq, Hq);
  return rows > 0 ? rows + kPartialMost : 0;
}

extern "C" int mhip_attn_bwd_plan(int B, int Sq, int Sc, int Hq, int Hkv, int D, int mask, int* splits) {
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || D > kD || !splits) return MHIP_EINVAL;
  if (mask != MHIP_MASK_NONE && mask != MHIP_MASK_CAUSAL) return MHIP_EINVAL;
  const Plan plan = plan_block(B, Sq, Sc, Hq, Hkv, D, mask == MHIP_MASK_CAUSAL);
  splits[0] = plan.sq;
  splits[1] = plan.sk;
  return plan.joint ? 1 : 2;
}

extern "C" int mhip_attn_bwd_chunks_plan(int n, int B, int Sq, int Sc, int Hq, int Hkv, int D, int mask, int* form) {
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || D > kD || !form) return MHIP_EINVAL;
  if (n < 1 || n > kMaxGroup || (mask != MHIP_MASK_NONE && (mask != MHIP_MASK_CAUSAL || n > 1))) return MHIP_EINVAL;
  const bool causal = mask == MHIP_MASK_CAUSAL, one = n == 1 || B == 0 || Sq == 0 || Sc == 0;
  const Plan plan = plan_block(B, Sq, Sc, Hq, Hkv, D, causal);
  const bool joint = one ? plan.joint : !chunks_apart(B, Sq, Sc, Hq, Hkv, D, n);
  form[0] = one ? plan.sq : joint ? chunk_splits(B, Sq, Sc, Hq, Hkv, D, n) : 1;
  form[1] = !joint && small_dq(B, Sq, Sc, Hq, D, causal, one ? 1 : n) ? 16 : 32;
  return joint ? 1 : 2;
}

namespace {
// own_scratch: take the workspace from `scratch` (resolved after the arguments have been checked).  chunks: several of them,
// the first one's places given as k .. dv32 too; they have been checked.
int bwd_block(const void* dout, const void* q, const void* k, const void* v,
              const void* out, const float* lse,
              void* dq, void* dk, void* dv, float* dq_acc, int dq_mode, float* dk32, float* dv32, bool prepared,
              int B, int Sq, int Sc, int Hq, int Hkv, int D,
              int64_t q_sb, int64_t q_ss, int64_t q_sh,
              int64_t k_sb, int64_t k_ss, int64_t k_sh,
              int64_t dk_sb, int64_t dk_ss, int64_t dk_sh,
              int64_t dq_sb, int64_t dq_ss, int64_t dq_sh,
              int64_t o_sb, int64_t o_ss, int64_t o_sh,
              float softmax_scale, int mask, void* workspace, bool own_scratch, hipStream_t st, const Chunks* chunks = nullptr) {
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0) return MHIP_EINVAL;
  if (!(softmax_scale > 0.f) || !(softmax_scale < INFINITY)) return MHIP_EINVAL;
  if (mask != MHIP_MASK_NONE && mask != MHIP_MASK_CAUSAL) return MHIP_EINVAL;
  if (D < 8 || D > kD || (D & 7) != 0) return MHIP_EHEADDIM;     // below 128 the missing columns are zeros on chip
  if (B == 0) return MHIP_OK;
  if (Sq > 0 && (!dout || !q || !out || !lse || (!workspace && !own_scratch))) return MHIP_EINVAL;
  const bool dq_needed = dq_mode == kDqAdd || dq_mode == kDqLast, acc_needed = dq_mode == kDqFirst || dq_mode == kDqMiddle;
  if (Sq > 0 && ((dq_needed && !dq) || (acc_needed && !dq_acc))) return MHIP_EINVAL;
  if (Sc > 0 && (!k || !v || !dk32 != !dv32 || (!dk32 && (!dk || !dv)) || !dk != !dv)) return MHIP_EINVAL;
  const void* ptrs[] = {dout, q, k, v, out, dq, dk, dv, workspace, dq_acc, dk32, dv32};
  for (const void* ptr : ptrs)
    if (ptr && !aligned16(ptr)) return MHIP_EALIGN;
  const int64_t strides[] = {q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh,
                             o_sb, o_ss, o_sh};
  for (int64_t s : strides)
    if (s < 0 || (s & 7)) return MHIP_EALIGN;
  // streamed tiles are fetched through 32-bit buffer offsets
  const int64_t q_span = ((int64_t)Sq * q_ss + (int64_t)Hq * q_sh) * 2;
  const int64_t k_span = (int64_t)Sc * k_ss * 2;
  if (q_span >= (int64_t(1) << 31) || k_span >= (int64_t(1) << 31)) return MHIP_EUNSUPPORTED;
  if ((int64_t)B * Hq * Sq >= (int64_t(1) << 30)) return MHIP_EUNSUPPORTED;     // lse2 / delta are addressed with 32-bit byte offsets
  // below 128 the lanes of the missing columns carry the offset kNoColumn, which has to be out of range
  if (D < kD && (q_span >= (int64_t(1) << 30) || k_span >= (int64_t(1) << 30))) return MHIP_EUNSUPPORTED;
  if (own_scratch && Sq > 0) {
    if ((int64_t)B * Hq * Sq > kScratchRows) return MHIP_ETOOLARGE;
    const int rc = scratch_address(&workspace);
    if (rc != MHIP_OK) return rc;
  }

  BwdParams p;
  p.q = static_cast<const uint16_t*>(q); p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v); p.dout = static_cast<const uint16_t*>(dout);
  float* delta_buf = static_cast<float*>(workspace);
  const int64_t slot = ((int64_t)B * Hq * Sq + 3) & ~int64_t(3);                // 16-byte aligned
  float* lse2_buf = delta_buf + slot;
  float* softmax_d = own_scratch ? nullptr : lse2_buf + slot;      // the built-in scratch has no room for it
  p.lse2 = lse2_buf; p.delta = delta_buf; p.softmax_d = softmax_d;
  // sums of split passes: behind the three row vectors (in the built-in scratch, which has its own place for them)
  float* partial = own_scratch ? delta_buf + (2 * kScratchRows + 8) : lse2_buf + 2 * slot;
  p.out = static_cast<const uint16_t*>(out); p.lse = lse;
  p.dq = static_cast<uint16_t*>(dq); p.dk = static_cast<uint16_t*>(dk); p.dv = static_cast<uint16_t*>(dv);
  p.dq_acc = dq_acc; p.dq_mode = dq_mode; p.prepared = prepared;
  p.dk32 = dk32; p.dv32 = dv32;
  p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq; p.Hkv = Hkv; p.group = Hq / Hkv;
  p.by_hq = Divisor(Hq); p.by_hkv = Divisor(Hkv); p.by_group = Divisor(Hq / Hkv);
  p.D = D;
  p.q_sb = q_sb; p.q_ss = q_ss; p.q_sh = q_sh;
  p.k_sb = k_sb; p.k_ss = k_ss; p.k_sh = k_sh;
  p.dk_sb = dk_sb; p.dk_ss = dk_ss; p.dk_sh = dk_sh;
  p.dq_sb = dq_sb; p.dq_ss = dq_ss; p.dq_sh = dq_sh;
  p.o_sb = o_sb; p.o_ss = o_ss; p.o_sh = o_sh;
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * kLog2e;
  const bool causal = mask == MHIP_MASK_CAUSAL;

  if (chunks) {
    if (D <= 64) launch_chunks<4>(p, *chunks, partial, st);
    else if (D <= 96) launch_chunks<6>(p, *chunks, partial, st);
    else launch_chunks<8>(p, *chunks, partial, st);
    return launch_status();
  }
  const Plan plan = plan_block(B, Sq, Sc, Hq, Hkv, D, causal);
  if (D <= 64) causal ? launch_bwd<true, 4>(p, plan, partial, st) : launch_bwd<false, 4>(p, plan, partial, st);
  else if (D <= 96) causal ? launch_bwd<true, 6>(p, plan, partial, st) : launch_bwd<false, 6>(p, plan, partial, st);
  else causal ? launch_bwd<true, 8>(p, plan, partial, st) : launch_bwd<false, 8>(p, plan, partial, st);
  return launch_status();
}
}  // namespace

// Resolves, for the current device, whatever the entry points otherwise look up on their first call (the address
// of the built-in scratch): a caller that records its calls (HIP graph capture) makes this call first, outside
// the capture.
extern "C" int mhip_init(void) {
  void* unused = nullptr;
  return scratch_address(&unused);
}

extern "C" int mhip_attn_bwd_block(const void* dout, const void* q, const void* k, const void* v,
                                   const void* out, const float* lse,
                                   void* dq, void* dk, void* dv, float* dq_acc,
                                   int B, int Sq, int Sc, int Hq, int Hkv, int D,
                                   int64_t q_sb, int64_t q_ss, int64_t q_sh,
                                   int64_t k_sb, int64_t k_ss, int64_t k_sh,
                                   int64_t dk_sb, int64_t dk_ss, int64_t dk_sh,
                                   int64_t dq_sb, int64_t dq_ss, int64_t dq_sh,
                                   int64_t o_sb, int64_t o_ss, int64_t o_sh,
                                   float softmax_scale, int mask, int deterministic,
                                   void* workspace, void* stream) {
  (void)deterministic;   // there are no atomics: every run is deterministic
  return bwd_block(dout, q, k, v, out, lse, dq, dk, dv, dq_acc, kDqAdd, nullptr, nullptr, false, B, Sq, Sc, Hq, Hkv, D, q_sb, q_ss, q_sh,
                   k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh, o_sb, o_ss, o_sh, softmax_scale, mask,
                   workspace, false,
                   static_cast<hipStream_t>(stream));
}

extern "C" int mhip_attn_bwd_block_noalloc(const void* dout, const void* q, const void* k, const void* v,
                                           const void* out, const float* lse,
                                           void* dq, void* dk, void* dv, float* dq_acc,
                                           int B, int Sq, int Sc, int Hq, int Hkv, int D,
                                           int64_t q_sb, int64_t q_ss, int64_t q_sh,
                                           int64_t k_sb, int64_t k_ss, int64_t k_sh,
                                           int64_t dk_sb, int64_t dk_ss, int64_t dk_sh,
                                           int64_t dq_sb, int64_t dq_ss, int64_t dq_sh,
                                           int64_t o_sb, int64_t o_ss, int64_t o_sh,
                                           float softmax_scale, int mask, int deterministic, void* stream) {
  (void)deterministic;
  // the dQ pass overwrites the part of the scratch the dK / dV pass reads, so nothing has to be cleared
  return bwd_block(dout, q, k, v, out, lse, dq, dk, dv, dq_acc, kDqAdd, nullptr, nullptr, false, B, Sq, Sc, Hq, Hkv, D, q_sb, q_ss, q_sh,
                   k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh, o_sb, o_ss, o_sh, softmax_scale, mask,
                   nullptr, true,
                   static_cast<hipStream_t>(stream));
}

extern "C" int mhip_attn_bwd_chunk(const void* dout, const void* q, const void* k, const void* v,
                                   const void* out, const float* lse,
                                   void* dq, float* dq_acc, int first, int last, int prepared,
                                   void* dk, void* dv, float* dk32, float* dv32,
                                   int B, int Sq, int Sc, int Hq, int Hkv, int D,
                                   int64_t q_sb, int64_t q_ss, int64_t q_sh,
                                   int64_t k_sb, int64_t k_ss, int64_t k_sh,
                                   int64_t dk_sb, int64_t dk_ss, int64_t dk_sh,
                                   int64_t dq_sb, int64_t dq_ss, int64_t dq_sh,
                                   int64_t o_sb, int64_t o_ss, int64_t o_sh,
                                   float softmax_scale, int mask, void* workspace, void* stream) {
  const bool only = first && last;      // the only chunk: nothing to carry
  if (!first && !dq_acc) return MHIP_EINVAL;
  return bwd_block(dout, q, k, v, out, lse, dq, dk, dv, only ? nullptr : dq_acc,
                   only ? kDqAdd : first ? kDqFirst : last ? kDqLast : kDqMiddle, dk32, dv32, prepared != 0,
                   B, Sq, Sc, Hq, Hkv, D, q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh,
                   o_sb, o_ss, o_sh, softmax_scale, mask, workspace, false, static_cast<hipStream_t>(stream));
}

extern "C" int mhip_attn_bwd_group(int B, int Sq, int Sc, int Hq, int Hkv, int D, int chunks) {
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || D > kD || chunks < 1) return MHIP_EINVAL;
  return group_chunks(B, Sq, Sc, Hq, Hkv, D, chunks, false);
}

extern "C" int mhip_attn_bwd_take(int B, int Sq, int Sc, int Hq, int Hkv, int D, int chunks) {
  if (B < 0 || Sq < 0 || Sc < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || D > kD || chunks < 1) return MHIP_EINVAL;
  return group_chunks(B, Sq, Sc, Hq, Hkv, D, chunks, true);
}

extern "C" int mhip_attn_bwd_chunks(const void* dout, const void* q, const void* const* ks, const void* const* vs, int n,
                                    const void* out, const float* lse,
                                    void* dq, float* dq_acc, int first, int last, int prepared,
                                    void* const* dks, void* const* dvs, float* const* dk32s, float* const* dv32s,
                                    int B, int Sq, int Sc, int Hq, int Hkv, int D,
                                    int64_t q_sb, int64_t q_ss, int64_t q_sh,
                                    int64_t k_sb, int64_t k_ss, int64_t k_sh,
                                    int64_t dk_sb, int64_t dk_ss, int64_t dk_sh,
                                    int64_t dq_sb, int64_t dq_ss, int64_t dq_sh,
                                    int64_t o_sb, int64_t o_ss, int64_t o_sh,
                                    float softmax_scale, void* workspace, void* stream) {
  if (n < 1 || n > kMaxGroup || !ks || !vs || !dks || !dvs || !dk32s || !dv32s) return MHIP_EINVAL;
  if (n == 1 || B == 0 || Sq == 0 || Sc == 0) {
    for (int i = 0; i < n; ++i) {
      const int rc = mhip_attn_bwd_chunk(dout, q, ks[i], vs[i], out, lse, dq, dq_acc, first && i == 0, last && i + 1 == n,
                                         prepared || i > 0, dks[i], dvs[i], dk32s[i], dv32s[i], B, Sq, Sc, Hq, Hkv, D, q_sb, q_ss, q_sh,
                                         k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh, o_sb, o_ss, o_sh, softmax_scale,
                                         MHIP_MASK_NONE, workspace, stream);
      if (rc != MHIP_OK) return rc;
    }
    return MHIP_OK;
  }
  if ((int64_t)n * B * Hkv * (((int64_t)Sc + 127) / 128) >= (int64_t(1) << 30)) return MHIP_EUNSUPPORTED;    // workgroups in 32 bits
  Chunks c;
  c.n = n;
  c.by_heads = Divisor(B * (int64_t)Hkv > 0 ? B * Hkv : 1);
  for (int i = 0; i < kMaxGroup; ++i) {
    const int j = i < n ? i : 0;
    c.k[i] = static_cast<const uint16_t*>(ks[j]); c.v[i] = static_cast<const uint16_t*>(vs[j]);
    c.dk[i] = static_cast<uint16_t*>(dks[j]); c.dv[i] = static_cast<uint16_t*>(dvs[j]);
    c.dk32[i] = dk32s[j]; c.dv32[i] = dv32s[j];
    if (!c.k[i] || !c.v[i] || !c.dk32[i] != !c.dv32[i] || !c.dk[i] != !c.dv[i] || (!c.dk32[i] && !c.dk[i])) return MHIP_EINVAL;
    const void* ptrs[] = {c.k[i], c.v[i], c.dk[i], c.dv[i], c.dk32[i], c.dv32[i]};
    for (const void* ptr : ptrs)
      if (ptr && !aligned16(ptr)) return MHIP_EALIGN;
  }
  const bool only = first && last;
  if (!first && !dq_acc) return MHIP_EINVAL;
  return bwd_block(dout, q, ks[0], vs[0], out, lse, dq, dks[0], dvs[0], only ? nullptr : dq_acc,
                   only ? kDqAdd : first ? kDqFirst : last ? kDqLast : kDqMiddle, dk32s[0], dv32s[0], prepared != 0,
                   B, Sq, Sc, Hq, Hkv, D, q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, dk_sb, dk_ss, dk_sh, dq_sb, dq_ss, dq_sh,
                   o_sb, o_ss, o_sh, softmax_scale, MHIP_MASK_NONE, workspace, false, static_cast<hipStream_t>(stream), &c);
}
