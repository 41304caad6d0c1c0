// Block forward of the ring-attention step for gfx950: one Q shard against one KV chunk,
// out = softmax(scale * q k^T) v and lse = logsumexp(scale * q k^T), bf16 in, fp32 accumulate.
//
// Replaces the flash-attn call at utils/flash_attn_dsl.py:159-176 of the reference.
//
// Work decomposition
//   workgroup  = 256 Q rows of one (batch, q-head): 8 wavefronts x 32 rows, one workgroup per CU,
//                two wavefronts per SIMD
//   main loop  = 64-key tiles of the chunk.  K and V tiles go from global memory straight into LDS
//                (buffer_load ... lds, no registers in between), row-major with the 16-byte chunks of
//                a row XOR-swizzled, four stages each; every wavefront copies 8 rows of each tile
//   S^T = K Q^T  : v_mfma_f32_32x32x16_bf16 with A = K rows (LDS), B = Q (registers, loaded once).
//                  The accumulator layout puts one Q row in each lane (lane % 32) and 32 of the
//                  64 keys of the tile in that lane's registers, so the softmax is lane-local.
//                  (Launches bound by the board's power use v_mfma_f32_16x16x32_bf16: two Q rows in
//                  each lane, 16 keys of each, everything else alike.)
//   O^T = V^T P^T: the same lane that produced P^T[key][q] feeds it back as the B operand; the
//                  key order inside one MFMA k-step is whatever the accumulator registers hold, and
//                  the V^T operand is gathered in exactly that order from the row-major V tile by
//                  ds_read_b64_tr_b16 (four keys of one head-dim column per lane), so P never moves.
//   ping-pong    : every tile is split into a matrix phase (S^T of the next tile + O^T of this one,
//                  32 MFMAs) and a vector phase (softmax of the next tile, tile copies).  Wavefronts
//                  0-3 and 4-7 run half a tile apart, separated by workgroup barriers, so on every
//                  SIMD one wavefront feeds the matrix pipe while the other does exponentials.
//   softmax      : the reference score of a row is fixed by the first tile's row maximum and moves only
//                  when a later tile would overflow: the row SUMS are watched (one compare per tile),
//                  not the maxima, so the common path has no maximum, no cross-lane exchange and no
//                  rescale of O; two of a tile's sixteen pairs of exponentials ride behind the last
//                  MFMAs of the matrix phase (the vector phase was the longer of the two).
#include "mhip_common.hpp"

#include <math.h>

namespace mhip {
namespace {

constexpr int kD = 128;            // head dimension
constexpr int kWaves = 8;
constexpr int kBM = kWaves * 32;   // Q rows per workgroup
constexpr int kBN = 64;            // keys per main-loop tile
constexpr int kTileBytes = kBN * kD * 2;   // 16384: one K or V tile in LDS, 64 rows of 256 bytes
constexpr int kStages = 4;                 // K(t+1) .. K(t+4) and V(t) .. V(t+3) live while tile t is processed
constexpr int kVBase = kStages * kTileBytes;   // K rings of all key groups first, then the V rings
constexpr int kNoTile = 0x7fff0000;    // scalar offset that puts every lane of a copy out of range
constexpr int kOStride = kD + 8;   // epilogue staging of O, bf16 elements per row
constexpr int kNoColumn = 0x7fff0000;  // vector offset that is out of every descriptor's range (spans stay below 2^31,
                                       // and so does the scalar tile offset added to it: no 32-bit wrap)
constexpr int kFragDepth = 4;      // LDS operand reads in flight ahead of the MFMAs (6 and 8 measure the same)

struct FwdParams {
  // what a workgroup needs before its first copy: read by one group of loads (see load_now)
  int per_xcd;       // ceil(total / 8)
  int total;         // blocks * B * Hq * nq_tiles
  int blocks;        // results of the launch: the same q against as many chunks, or runs of them
  int nq_tiles;      // ceil(Sq / rows per workgroup)
  int heads_per_xcd; // (block, batch, head) triples per XCD when they divide evenly, else 0
  int Sq, Sc;
  int D;             // head dimension of the tensors, a multiple of 8 up to kD; columns D .. kD-1 are zeros on chip
  Divisor by_q_tiles, by_hq, by_group;
  Divisor by_order;  // causal: by the (block, batch, head) triples, or by those of an XCD
  const uint16_t* q; const uint16_t* k0; const uint16_t* v0;         // k0, v0: the first block's chunk
  int64_t q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, v_sb, v_ss, v_sh;
  float scale, scale_log2;
  // the rest
  int per, chunks;   // consecutive chunks of a result, chunks of the launch
  Divisor by_heads;  // by B * Hq
  int heads;         // B * Hq
  int B, Hq;
  uint16_t* out; float* lse;
  int64_t o_sb, o_ss, o_sh;
  int64_t o_sn, l_sn;    // from one block's results to the next one's, elements
};
// With the chunks of a launch over several of them.  A launch of one block leaves their 256 bytes out: graphs of such launches,
// us, with / without: 256 x 256 H4 D64 5.86 / 5.83, causal 6.22 / 6.10, 512 x 512 B4 H5 9.32 / 9.27, causal 1024 x 1024 H32
// 16.57 / 16.41, 2048 x 2048 H24 D64 29.37 / 29.22.
struct FwdChunks : FwdParams {
  const uint16_t* k[kMaxGroup]; const uint16_t* v[kMaxGroup];        // the chunk of every block
};

// KK = k-steps of 16 head-dim values in S^T: 8 computes on all 128 on-chip columns; 4 and 6 are the instantiations for
// head dimensions up to 64 and up to 96, which leave out the MFMAs that would only see the zero columns (half and a
// quarter of both products).
//
// KS = key groups of a workgroup.  With one group the eight wavefronts hold 8 x 32 Q rows and all visit every key
// tile.  A launch of few (batch, head, 256-row) items leaves most CUs without a workgroup then, and its time is the
// length of one workgroup's serial chain of tiles.  With KS = 2 (4) the workgroup holds 128 (64) rows instead; wavefront
// w works for row group w % (8 / KS) and key group w / (8 / KS), whose tiles are every KS-th one, and the groups' partial
// (O, sum) of a row meet in LDS at the end.  Twice (four times) as many workgroups, each with half (a quarter) of the
// serial chain; the price is as many times the L2 -> LDS traffic per row.  A key group has rings of two stages instead
// of four, of 64-key tiles (KS = 2) or 32-key tiles (KS = 4): 128 KB of LDS in all three cases.
//
// CHAIN: a workgroup visits p.per chunks one after the other, their tiles as one sequence: the ends of a workgroup's life
// (arguments, Q, first tiles, O out) come once instead of once per chunk, and one result stands for all of them, which the
// fold would otherwise write and read back as many times.
//
// M = rows and columns of an MFMA tile: v_mfma_f32_32x32x16_bf16 or v_mfma_f32_16x16x32_bf16, which does half as much work in
// half the time and takes 12 % less energy for it (a register-only loop on random operands under the power cap: 1727 and
// 1955 TFLOP/s).  Its twice as many instructions cost issue slots that the vector phase of the other wavefront wants, so it
// pays where the clock is what gives: launches that keep every CU busy for long (small_tiles).
template <bool CAUSAL, int KK, int KS, class P, bool CHAIN = false, int M = 32>
__global__ __launch_bounds__(kWaves * 64, 2) void attn_fwd_bf16_d128(const P p) {
  constexpr bool kLone = std::is_same<P, FwdParams>::value;
  static_assert(!CHAIN || !kLone, "a run of chunks needs their addresses");
  static_assert(KK == 8 || KK == 6 || KK == 4, "128, 96 or 64 on-chip head-dim columns");
  static_assert(KS == 1 || KS == 2 || KS == 4, "key groups");
  static_assert(!CHAIN || (KS == 1 && !CAUSAL), "chunks are visited one after the other by workgroups of one key group");
  static_assert(M == 32 || (M == 16 && KS == 1), "32 x 32 or 16 x 16 MFMA tiles");
  constexpr int R = 32 / M;         // row blocks of a wavefront
  constexpr int NR = M * M / 64;    // registers of an accumulator tile
  constexpr int KB = KK * M / 32;   // k-steps of 512 / M head-dim values in S^T
  constexpr int DB = KK * 16 / M;   // blocks of M head-dim values in O^T
  typedef typename std::conditional<M == 32, f32x16, f32x4>::type Acc;
  constexpr int RG = kWaves / KS;   // row groups of 32
  constexpr int kRows = 32 * RG;    // Q rows of the workgroup
  constexpr int BN = KS == 4 ? 32 : kBN;             // keys per tile
  constexpr int MB = BN / M;                         // key blocks per tile
  constexpr int kTile = BN * kD * 2;                 // bytes of a tile
  constexpr int kGroupStages = KS == 1 ? kStages : 2;
  constexpr int kSlotsS = MB * KB;      // matrix-phase slots of S^T, an operand from LDS and R MFMAs each
  constexpr int kSteps = BN * M / 512;  // k-steps of 512 / M keys of O^T
  constexpr int kSlotsO = kSteps * DB;  // and of O^T
  static_assert(KS * kGroupStages * kTile == kStages * kTileBytes, "the K rings take 64 KB, and so do the V rings");
  constexpr int kQBase = 2 * kStages * kTileBytes;   // KS > 1: Q rows, later the O rows on their way out
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kStages * kTileBytes + (KS > 1 ? kRows * kD * 2 : 0)];

  // Workgroup i runs on XCD i % 8.  Give every XCD a contiguous range of the (batch, head, q-tile)
  // order so that the workgroups sharing one K/V head also share one L2.
  // Under the causal mask a Q tile's work grows with its index, so there the order is longest tiles
  // first across all heads (of the XCD when the heads divide evenly over the XCDs, of the launch
  // otherwise): the short tiles fill the tail.
  load_now<CAUSAL>(p, p.scale_log2);
  int qt, bh;
  if (!CAUSAL) {
    const int logical = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
    if (logical >= p.total) return;
    bh = p.by_q_tiles.quotient(logical, qt);
  } else if (p.heads_per_xcd > 0) {
    qt = p.nq_tiles - 1 - p.by_order.quotient(blockIdx.x >> 3, bh);
    bh += (blockIdx.x & 7) * p.heads_per_xcd;
  } else {
    if ((int)blockIdx.x >= p.total) return;
    qt = p.nq_tiles - 1 - p.by_order.quotient(blockIdx.x, bh);
  }
  // Several blocks of a step in one launch are so many times the (batch, head) pairs.  (The
  // first one's addresses come with the arguments above: a lone block does not wait for a second round of loads.)
  const uint16_t* kp = p.k0; const uint16_t* vp = p.v0;
  int blk = 0, chunk = 0;
  if constexpr (!kLone)
    if (p.blocks > 1) {
      blk = p.by_heads.quotient(bh, bh);
      chunk = CHAIN ? blk * p.per : blk;
      kp = p.k[chunk];
      vp = p.v[chunk];
    }
  int hq;
  const int b = p.by_hq.quotient(bh, hq);
  const int hk = p.by_group.quotient(hq);
  const int q0 = qt * kRows;
  // Kept in a register: a scalar load that may be under way where the main loop begins turns its waits for one LDS operand
  // into waits for all of them (2048 x 2048 H24, D 64: 32.5 us instead of 30.9).
  float scale_log2 = p.scale_log2;
  asm volatile("" : "+s"(scale_log2));

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: role branches stay uniform
  const int lane = tid & 63;
  const int ln = lane % M;
  const int lg = lane / M;
  const bool group_b = wave >= 4;                 // second ping-pong group
  const int kg = KS == 1 ? 0 : wave / RG;         // key group
  const int rg = KS == 1 ? wave : wave % RG;      // row group

  // ---- number of key tiles this Q tile has to visit -------------------------------------------
  int kv_end = p.Sc;
  if (CAUSAL) {
    const int lim = q0 + kRows + (p.Sc - p.Sq);   // one past the last key visible to the last row
    kv_end = lim < kv_end ? lim : kv_end;
    if (kv_end < 0) kv_end = 0;
  }
  int ntiles = (kv_end + BN * KS - 1) / (BN * KS);   // of each key group; tiles past the end are hidden whole
  int chunks_left = 0;                               // CHAIN: behind the first one
  if (CHAIN) {
    chunks_left = (p.chunks - chunk < p.per ? p.chunks - chunk : p.per) - 1;
    ntiles *= chunks_left + 1;
  }

  // ---- Q fragment: B operand of S^T = K Q^T, lane (ln, lg) holds Q[row][512/M ks + 8 lg .. +7] of rows M r + ln ---
  const int my_q = q0 + rg * 32 + ln;
  bf16x8 qf[R][KB];  // loaded in the prologue

  // ---- global -> LDS copies of the K and V tiles ---------------------------------------------------
  // A tile is 64 rows of 256 bytes.  Chunk c (16 bytes) of row r lives at chunk position c ^ swz(r):
  // the 32 rows a b128 operand read touches then spread over all banks, and so do the 8 rows x 4 chunks
  // of a transposing read.  Wavefront w copies rows 8w .. 8w+7 of every tile with two instructions of
  // 1 KB; lane l of instruction u lands at row 8w + 4u + l/16, position l%16 (the hardware places the
  // lanes back to back) and therefore fetches chunk (l%16) ^ swz(row).  Rows past the end of the chunk
  // are out of the descriptor's range and arrive as zeros, and so do the chunks past the head dimension
  // when it is below 128: their lanes carry an offset that is out of range for every tile, so a tile in
  // LDS always has 128 columns, the upper ones zero, at no cost in memory traffic.
  auto swz = [](int row) { return lds_row_swizzle(row); };
  u32x4 krs = rsrc_words(kp + b * p.k_sb + hk * p.k_sh, (uint32_t)(((int64_t)(p.Sc - 1) * p.k_ss + p.D) * 2));
  u32x4 vrs = rsrc_words(vp + b * p.v_sb + hk * p.v_sh, (uint32_t)(((int64_t)(p.Sc - 1) * p.v_ss + p.D) * 2));
  constexpr int kCpy = BN / RG / 4;                  // copy instructions per wavefront, tile and tensor (4 rows each)
  int kvoff[kCpy], vvoff[kCpy];
#pragma unroll
  for (int u = 0; u < kCpy; ++u) {
    const int row = 4 * kCpy * rg + 4 * u + (lane >> 4);
    const int chunk = (lane & 15) ^ swz(row);
    const bool real = chunk * 8 < p.D;
    kvoff[u] = real ? (int)(row * p.k_ss * 2) + chunk * 16 : kNoColumn;
    vvoff[u] = real ? (int)(row * p.v_ss * 2) + chunk * 16 : kNoColumn;
  }
  const int k_tile_bytes = (int)(BN * p.k_ss * 2);
  const int v_tile_bytes = (int)(BN * p.v_ss * 2);
  const uint32_t lds_smem = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const uint32_t lds_ring = lds_smem + kg * (kGroupStages * kTile);  // this key group's K ring; its V ring is kVBase on
  const uint32_t lds_base = lds_ring + rg * (kCpy * 1024);
  // tile t of this wavefront's key group; with several groups a tile past the last key is put out of range as a whole
  auto tile_offset = [&](int t, int tile_bytes) {
    if (KS == 1) return t * tile_bytes;
    const int tile = t * KS + kg;
    return tile * BN < p.Sc ? tile * tile_bytes : kNoTile;
  };
  // CHAIN: K and V tiles are requested in order; k_off and v_off are the offsets of the next ones inside their chunks, k_pos
  // and v_pos their numbers (rows may all lie at one place).  (The address of a chunk is loaded inside its branch and waited
  // for there.)
  const int chunk_tiles = (p.Sc + BN - 1) / BN;
  int k_off = 0, v_off = 0, k_pos = 0, v_pos = 0, k_chunk = chunk, v_chunk = chunk;
  const int last_chunk = chunk + chunks_left;
  auto enter = [&](u32x4& rs, const uint16_t* base) {
    asm volatile("" : "+s"(base));
    rs[0] = (uint32_t)(uint64_t)base;
    rs[1] = (uint32_t)((uint64_t)base >> 32) & 0xffffu;
  };
  auto cross_k = [&]() {                             // behind the last K tile of a chunk that is not the last one
    k_off = k_pos = 0;
    ++k_chunk;
    if constexpr (CHAIN) enter(krs, p.k[k_chunk] + b * p.k_sb + hk * p.k_sh);
  };
  auto cross_v = [&]() {
    v_off = v_pos = 0;
    ++v_chunk;
    if constexpr (CHAIN) enter(vrs, p.v[v_chunk] + b * p.v_sb + hk * p.v_sh);
  };
  auto chain_k = [&]() {                             // behind the copy of a K tile of the prologue
    k_off += k_tile_bytes;
    if (++k_pos == chunk_tiles && k_chunk != last_chunk) cross_k();
  };
  auto chain_v = [&]() {
    v_off += v_tile_bytes;
    if (++v_pos == chunk_tiles && v_chunk != last_chunk) cross_v();
  };
  // The main loop counts down to the next end of a chunk in either sequence: one test per tile instead of two with their
  // detours (8 chunks, us: 1237 x 1237 B2 H16/8 D80 in pairs 161 to 152, 2048 x 2048 H16 D64 in fours 147 to 143, 700 x 700 H12
  // D64 in pairs 27.0 to 26.1; on 128 columns, where the clock decides, no change).
  int span = 0, till = 0;
  auto next_end = [&]() {
    const int k_left = k_chunk != last_chunk ? chunk_tiles - k_pos : 0x7fffffff;
    const int v_left = v_chunk != last_chunk ? chunk_tiles - v_pos : 0x7fffffff;
    till = span = k_left < v_left ? k_left : v_left;
  };
  auto chain = [&]() {                               // behind the copies of a K and a V tile
    k_off += k_tile_bytes;
    v_off += v_tile_bytes;
    if (__builtin_expect(--till == 0, 0)) {
      k_pos += span;
      v_pos += span;
      if (k_pos == chunk_tiles && k_chunk != last_chunk) cross_k();
      if (v_pos == chunk_tiles && v_chunk != last_chunk) cross_v();
      next_end();
    }
  };
  auto copy_k = [&](int t, int stage) {
    const int soff = CHAIN ? k_off : tile_offset(t, k_tile_bytes);
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy16_to_lds(krs, lds_base + stage * kTile + u * 1024, kvoff[u], soff);
  };
  auto copy_v = [&](int t, int stage) {
    const int soff = CHAIN ? v_off : tile_offset(t, v_tile_bytes);
#pragma unroll
    for (int u = 0; u < kCpy; ++u)
      copy16_to_lds(vrs, lds_base + kVBase + stage * kTile + u * 1024, vvoff[u], soff);
  };

  // K operand of S^T (A, M keys x 512/M head-dim values): lane (ln, lg) reads chunk 64/M ks + lg of row M mb + ln.
  // k_a and v_a hold the LDS addresses inside the stage that is read next and move on in place, each at a point of the
  // slot sequence where no read of its kind is due; everything else about an address is an immediate offset.
  int k_a[KB];                                        // + mb * M rows
#pragma unroll
  for (int ks = 0; ks < KB; ++ks) k_a[ks] = (int)lds_ring + ln * 256 + (((64 / M * ks + lg) ^ swz(ln)) << 4);
  // V^T operand of O^T (A, M head-dim values x 512/M keys) for head-dim block db and k-step t: the lane's 8 keys are rows
  // X + {0..3} and, 8 (M = 16: 16) rows on, four more, X = 512/M t + 4 lg -- the keys its P registers hold.  One
  // ds_read_b64_tr_b16 per group of 4 rows: within 16 lanes, lane s supplies the address of row X + s/4, head-dim values 4 (s%4) .. +3 of the
  // 16-column strip, and receives column s.
  int v_a[KK];                                        // 32: [2 db + second four rows], 16: [db]; + t * 512/M rows
  {
    const int s16 = lane & 15, strip = M == 32 ? (lane >> 4) & 1 : 0;
    const int cl = 2 * strip + ((s16 & 3) >> 1);
#pragma unroll
    for (int i = 0; i < KK; ++i) {
      const int db = M == 32 ? i / 2 : i, row = (M == 32 ? 8 * (i & 1) : 0) + 4 * lg + (s16 >> 2);
      v_a[i] = (int)lds_ring + kVBase + row * 256 + (((M / 8 * db + cl) ^ swz(row)) << 4) + (s16 & 1) * 8;
    }
  }
  typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4;
  typedef __attribute__((address_space(3))) const bf16x8* lds_bf16x8;
  auto read_k = [&](int mb, int ks) -> bf16x8 { return *(lds_bf16x8)(uintptr_t)(uint32_t)(k_a[ks] + mb * M * 256); };
  auto read_v = [&](int db, int t) -> bf16x8 {
    const int at = t * (512 / M) * 256;
    const int first = M == 32 ? v_a[2 * db % KK] : v_a[db], second = M == 32 ? v_a[(2 * db + 1) % KK] : v_a[db] + 4096;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4)(uintptr_t)(uint32_t)(first + at));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4)(uintptr_t)(uint32_t)(second + at));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // byte distance from the stage of tile t to the stage of tile t + 1
  auto stage_step = [](int t) { return (t + 1) % kGroupStages == 0 ? -(kGroupStages - 1) * kTile : kTile; };
  const int causal_shift = p.Sc - p.Sq;

  // ---- accumulators -----------------------------------------------------------------------------
  const Acc zero = {};
  Acc o_acc[DB][R];          // O^T: head-dim values M db + 8 (j / 4) + 4 lg + j % 4 of rows M r + ln
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int r = 0; r < R; ++r) o_acc[i][r] = zero;
  // m_ref: the raw (unscaled) score the exponentials of this lane's Q row are taken relative to.  It is
  // fixed by the first tile's row maximum and moves only when a later tile would overflow: the row sums are
  // watched, not the maxima, so the common path has no maximum, no cross-lane exchange and no rescale of O.
  float m_ref[R] = {};
  float nmsc[R] = {};        // -m_ref * scale * log2(e)
  float l_run[R] = {};       // this lane's share of the running sums (the other keys: lanes ^ 32, with M = 16 ^ 16 and ^ 48 too)
  auto row_sum = [](float x) { return M == 32 ? pair_sum(x) : quad_sum(x); };
  constexpr float kTrigger = 1048576.f;   // a lane's 32 exponentials of one tile sum to less than this, or
  constexpr float kSlack = 14.f;          // rows whose maximum exceeds the reference by 2^kSlack move it
  constexpr float kMost = 0x1.fffffep127f;
  Acc s[MB][R];              // S^T tile: BN keys x 32 q rows per wave, keys M mb + 8 (j / 4) + 4 lg + j % 4
  u32x4 pw[kSteps][R];       // P^T of the current tile as packed bf16 B operands

  auto mfma = [](const bf16x8& x, const bf16x8& y, const Acc& c) -> Acc {
    if constexpr (M == 32) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
  };
  auto s_mfma = [&](int mb, int ks, const bf16x8& kf) {
#pragma unroll
    for (int r = 0; r < R; ++r) s[mb][r] = mfma(kf, qf[r][ks], ks == 0 ? zero : s[mb][r]);
  };
  auto o_mfma = [&](int db, int t, const bf16x8& vf) {
#pragma unroll
    for (int r = 0; r < R; ++r) o_acc[db][r] = mfma(vf, __builtin_bit_cast(bf16x8, pw[t][r]), o_acc[db][r]);
  };
  auto qk = [&]() {                   // S^T(0); leaves k_a at K(1)
#pragma unroll
    for (int ks = 0; ks < KB; ++ks) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) s_mfma(mb, ks, read_k(mb, ks));
      k_a[ks] += kTile;
    }
  };

  auto pv = [&]() {
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
#pragma unroll
      for (int db = 0; db < DB; ++db) o_mfma(db, t, read_v(db, t));
    }
  };

  // keys past the chunk end and the causal diagonal -> -inf
  int chain_kv0 = 0;                                        // first key of the next tile inside its chunk
  auto sm_mask = [&](int t) {
    const int kv0 = CHAIN ? chain_kv0 : (t * KS + kg) * BN;
    if (CHAIN) chain_kv0 = kv0 + BN < p.Sc ? kv0 + BN : 0;
    bool need_mask = kv0 + BN > p.Sc;
    if (CAUSAL) need_mask = need_mask || (kv0 + BN - 1 > q0 + causal_shift);
    if (need_mask) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int lim = p.Sc - 1;                                 // last visible key of this lane's row
        if (CAUSAL) { const int c = my_q + r * M + causal_shift; lim = c < lim ? c : lim; }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int j = 0; j < NR; ++j) {
            const int at = mb * M + (j >> 2) * 8 + (j & 3);
            if (CHAIN ? at + lg * 4 > lim - kv0 : kv0 + at + lg * 4 > lim) s[mb][r][j] = -INFINITY;
          }
      }
    }
  };
  // Exponentials of the tile in 16 pairs (eight of a 32-key tile): pair 4 (R t + r) + d gives dword d of the packed P^T operand of
  // k-step t and row block r.  s stays intact.
  // The first kEarlyPairs pairs are computed inside the matrix phase, between the O^T MFMAs: measured with
  // cycle counters the vector phase is the longer of the two (1314 against 1265 ticks per 64-key tile), and
  // two pairs moved over make the step 3 % faster (four and more slow the matrix phase down by as much as
  // they shorten the other; on 64 columns, where it has half the MFMAs, six do).  A pair may overwrite the P^T operand of k-step t only after the last MFMA of
  // that k-step has been issued.
  float rs[R] = {};
  auto sm_pair = [&](int idx) {
    const int t = idx / (4 * R), r = (idx >> 2) % R, d = idx & 3, mb = (8 * t + 2 * d) / NR, e = (8 * t + 2 * d) % NR;
    float x0 = fast_exp2(__builtin_fmaf(s[mb][r][e], scale_log2, nmsc[r]));
    float x1 = fast_exp2(__builtin_fmaf(s[mb][r][e + 1], scale_log2, nmsc[r]));
    if (t == 0 && d == 0) rs[r] = x0 + x1; else rs[r] += x0 + x1;
    uint32_t w = pack_bf16(x0, x1);
    asm volatile("" : "+v"(w), "+v"(rs[r]));       // keeps the pair where it is written
    pw[t][r][d] = w;
  };
  auto sm_exps = [&]() {
#pragma unroll
    for (int idx = 0; idx < BN / 4; ++idx) sm_pair(idx);
  };
  // Move the reference of the rows whose scores outgrew it (first tile: set it to the row maximum) and
  // rescale O and the running sum accordingly.
  auto sm_fix = [&](bool first) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float mx = s[0][r][0];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < NR; ++j) mx = fmaxf(mx, s[mb][r][j]);
      mx = M == 32 ? pair_max(mx) : quad_max(mx);
      const float grown = (mx - m_ref[r]) * scale_log2;
      const bool move = first || grown > kSlack;                 // false for NaN
      if (!first) {
        const float alpha = move ? fast_exp2(-grown) : 1.f;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int j = 0; j < NR; ++j) o_acc[db][r][j] *= alpha;
        l_run[r] *= alpha;
      }
      // (with scores of -inf alone it stays at the lowest finite one, so that the first key that counts moves it; the product
      // stays finite too, so that scores of -inf have exponentials of 0)
      if (move) m_ref[r] = first ? fmaxf(mx, -kMost) : mx;
      nmsc[r] = fminf(-m_ref[r] * scale_log2, kMost);
    }
  };
  // slot of the matrix phase after which early pair idx runs: behind the DB slots of O^T that read k-step 0, whose first row
  // block the pairs belong to (of 32 x 32 tiles with six pairs: and those of k-step 1), spread over the rest
  constexpr bool kShortMatrix = KS == 1 && KK < 8;
  constexpr int kEarlyPairs = KS == 1 && KK == 4 ? 6 : 2;
  constexpr int kEarlyGap = kEarlyPairs > 2 || MB * DB < 4 ? 1 : 2;
  auto early_slot = [](int idx) { return kSlotsS + DB + (M == 32 ? kEarlyGap * idx : idx * (kSlotsO - DB) / kEarlyPairs); };
  static_assert(M == 16 || (DB + kEarlyGap * (kEarlyPairs - 1) < kSlotsO && (kEarlyPairs <= 4 || (DB + kEarlyGap * 4 >= 2 * DB && kEarlyPairs <= 8))),
                "the early pairs have to fit behind the O^T slots of their k-steps");
  auto sm_tile = [&]() {
#pragma unroll
    for (int idx = kEarlyPairs; idx < BN / 4; ++idx) sm_pair(idx);
    float sum = rs[0];
    if (R == 2) sum += rs[R - 1];
    if (__builtin_amdgcn_ballot_w64(!(sum < kTrigger)) != 0) {
      sm_fix(false);
      sm_exps();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) l_run[r] += rs[r];
  };

  // Matrix phase of tile t: S^T(t+1) and O^T += V^T(t) P^T(t), kSlotsS + kSlotsO operands (32 on 128 columns and 64 keys) from
  // LDS with R MFMAs each.  The reads run kFragDepth operands ahead through a ring of registers, so the LDS latency is
  // covered by the MFMAs in between.
  auto read_frag = [&](int i) -> bf16x8 {
    if (i < kSlotsS) return read_k(i % MB, i / MB);
    return read_v((i - kSlotsS) % DB, (i - kSlotsS) / DB);
  };
  // The first kFragDepth operands (all of K) are read before the barrier that opens the phase, by
  // first_frags, so the matrix pipe starts without waiting for LDS.
  bf16x8 frag[kFragDepth];
  auto first_frags = [&]() {
#pragma unroll
    for (int i = 0; i < kFragDepth; ++i) frag[i] = read_frag(i);
  };
  static_assert(kSlotsO >= KK / 2 && kFragDepth * 2 >= KK, "slots in which the operand addresses move on");
  auto matrix_phase = [&](int t) {
    const int k_step = stage_step(t + 1), v_step = stage_step(t);
#pragma unroll
    for (int i = 0; i < kSlotsS + kSlotsO; ++i) {
      if (i < kSlotsS) s_mfma(i % MB, i / MB, frag[i % kFragDepth]);
      else o_mfma((i - kSlotsS) % DB, (i - kSlotsS) / DB, frag[i % kFragDepth]);
      if (i + kFragDepth < kSlotsS + kSlotsO) frag[i % kFragDepth] = read_frag(i + kFragDepth);
      // the last K read went out in slot kSlotsS - kFragDepth - 1, the last V read kFragDepth slots before the end
      if (i >= kSlotsS && i < kSlotsS + KK / 2) {
#pragma unroll
        for (int e = 0; e < KB / (KK / 2); ++e) k_a[KB / (KK / 2) * (i - kSlotsS) + e] += k_step;
      }
      if (i >= kSlotsS + kSlotsO - KK / 2) {
        const int at = 2 * (i - (kSlotsS + kSlotsO - KK / 2));
        v_a[at] += v_step;
        v_a[at + 1] += v_step;
      }
      // On fewer than 128 columns the vector phase, which is the same length, would hold up a matrix phase that is half or
      // three quarters as long: there the tile copies go out between the S^T MFMAs (K(t) and V(t-1) are read by then,
      // see the main loop).  With that and the early pairs 2048 x 2048 H24 takes 33.3 instead of 39.6 us at D 64 and 41.9
      // instead of 43.9 at D 96, 4096 x 4096 H32 131.6 / 145.4 and 174.7 / 182.8; on 128 columns it is 1 % slower.
      if (kShortMatrix && i < kSlotsS && i % (kSlotsS / 4) == 1) {
        const int u = i / (kSlotsS / 4);
        if (u < 2) copy16_to_lds(krs, lds_base + (t & 3) * kTile + u * 1024, kvoff[u % kCpy], CHAIN ? k_off : tile_offset(t + 4, k_tile_bytes));
        else copy16_to_lds(vrs, lds_base + kVBase + ((t + 3) & 3) * kTile + (u - 2) * 1024, vvoff[u % kCpy], CHAIN ? v_off : tile_offset(t + 3, v_tile_bytes));
      }
      // S^T(t+1) is complete after its last slot; its softmax starts here, in the shadow of the O^T MFMAs
      if (i == kSlotsS) sm_mask(t + 1);
#pragma unroll
      for (int idx = 0; idx < kEarlyPairs; ++idx)
        if (early_slot(idx) == i) sm_pair(idx);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Q goes through LDS: read straight into its fragment layout, every load instruction of a wavefront touches 32 rows and
  // costs as many cache accesses, and one wait would cover every tile requested so far besides.  With the copies a launch
  // of 256 x 256, H4 takes 9.8 us instead of 10.4 (one key group), 4096 x 4096, H32 227.3 instead of 228.6.
  // Four rows per copy instruction, swizzled like a K tile; rows past the end repeat the last one, columns past the
  // head dimension are cleared in the fragment.
  auto copy_q = [&](int row4, uint32_t lds_addr) {
    const int r = row4 + (lane >> 4);
    const int row = q0 + r < p.Sq ? q0 + r : p.Sq - 1;
    const int chunk = (lane & 15) ^ swz(r);
    copy16_to_lds(p.q + b * p.q_sb + (int64_t)row * p.q_ss + hq * p.q_sh + (chunk * 8 < p.D ? chunk * 8 : 0), lds_addr);
  };
  auto read_q = [&](int lds_addr) {                // address of the first of the wavefront's 32 rows
#pragma unroll
    for (int ks = 0; ks < KB; ++ks)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        qf[r][ks] = *(lds_bf16x8)(uintptr_t)(uint32_t)(k_a[ks] - (int)lds_ring + lds_addr + r * M * 256);
        if (ks * (512 / M) + lg * 8 >= p.D) qf[r][ks] = bf16x8{};
      }
  };

  if constexpr (KS == 1) {
    // ---- prologue: the first tiles into LDS, softmax of tile 0 -------------------------------------------
    // Barriers inside the loop are bare s_barrier instructions: a fence would wait for every copy in flight.
    if (ntiles > 0) {
      // The wavefronts' Q rows pass through the stages of K(2), K(3) and V(2), V(3), whose copies go out once every
      // wavefront has its fragments.  Tiles past the chunk arrive as zeros.
      const uint32_t q_lds = lds_smem + (wave < 4 ? 0 : kVBase) + 2 * kTile + (wave & 3) * 8192;
      copy_k(0, 0);
      if (CHAIN) chain_k();
#pragma unroll
      for (int u = 0; u < 8; ++u) copy_q(32 * wave + 4 * u, q_lds + u * 1024);
      copy_v(0, 0);
      if (CHAIN) chain_v();
      copy_k(1, 1);
      if (CHAIN) chain_k();
      copy_v(1, 1);
      if (CHAIN) chain_v();
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(3 * kCpy) : "memory");     // K(0) and Q
      read_q(q_lds);
      // pinned here: otherwise the first use sits inside the main loop and so does the wait for the reads
#pragma unroll
      for (int ks = 0; ks < KB; ++ks)
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(qf[r][ks]));
      __builtin_amdgcn_s_barrier();
      copy_k(2, 2);
      if (CHAIN) chain_k();
      copy_k(3, 3);
      if (CHAIN) chain_k();
      copy_v(2, 2);
      if (CHAIN) chain_v();
      if (CHAIN) next_end();
      qk();
      sm_mask(0);
      sm_fix(true);
      sm_exps();
#pragma unroll
      for (int r = 0; r < R; ++r) l_run[r] = rs[r];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (ntiles > 1) first_frags();
    }
    // Phase p of the main loop: group A (waves 0-3) runs the matrix phase of tile p/2 on even p and its
    // vector phase on odd p; group B does the same one phase later.  K(t) and V(t) live in stage t % 4 of
    // their rings.  In the vector phase of tile t (on fewer than 128 columns in the matrix phase before it, when the
    // other group is past its matrix phase of tile t-1 too) every wavefront starts its share of the copies of K(t+4)
    // (over K(t), last read in the matrix phase of tile t-1) and V(t+3) (over V(t-1)), and before the
    // barrier that ends the vector phase waits for the copies it started one tile earlier: those are then visible
    // to every wavefront two barriers later, in time for first_frags of K(t+3) and the matrix phase of V(t+2).
    if (group_b) __builtin_amdgcn_s_barrier();
    for (int t = 0; t + 1 < ntiles; ++t) {
      // ---- matrix phase: S^T(t+1) = K(t+1) Q^T and O^T += V^T(t) P^T(t), first part of softmax(t+1) ------
      __builtin_amdgcn_s_setprio(2);
      matrix_phase(t);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_s_barrier();
      // ---- vector phase: softmax(t+1), copies of the tiles ahead ---------------------------------------------
      for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s[0][r]), "+v"(s[MB - 1][r]));   // keeps the exponentials behind the barrier
      sm_tile();
      if (!kShortMatrix) {
        copy_k(t + 4, t & 3);
        copy_v(t + 3, (t + 3) & 3);
      }
      if (CHAIN) chain();
      // K(t+2), for the next matrix phase; a chain also reads them where there is none: without the branch its D 64 loop takes
      // 6 % less (2 chunks of 4096 keys, 8192 rows H32: 579 us to 547) and the others 0.4 %, a lone block's 6 % more
      if (CHAIN || t + 2 < ntiles) first_frags();
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");          // the four copies of one tile ago are done
      __builtin_amdgcn_s_barrier();
    }
    if (ntiles > 0) pv();                             // last tile: nothing left to prefetch or exponentiate
    if (!group_b) __builtin_amdgcn_s_barrier();

    // ---- epilogue -----------------------------------------------------------------------------------
    float inv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float l_tot = row_sum(l_run[r]);
      inv[r] = l_tot > 0.f ? 1.f / l_tot : 0.f;
      if (lg == 0 && my_q + r * M < p.Sq) {
        const float lse = l_tot > 0.f ? __builtin_fmaf(fast_log2(l_tot), kLn2, m_ref[r] * p.scale) : -INFINITY;
        p.lse[blk * p.l_sn + ((int64_t)b * p.Hq + hq) * p.Sq + my_q + r * M] = lse;
      }
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // zero-filled copies of tiles past the end included
    __syncthreads();   // every wave is done with the K/V tiles: reuse LDS to transpose O
    unsigned char* os = smem + wave * (32 * kOStride * 2);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int g = 0; g < NR / 4; ++g) {
          u32x2 w;
          w[0] = pack_bf16(o_acc[db][r][4 * g] * inv[r], o_acc[db][r][4 * g + 1] * inv[r]);
          w[1] = pack_bf16(o_acc[db][r][4 * g + 2] * inv[r], o_acc[db][r][4 * g + 3] * inv[r]);
          *reinterpret_cast<u32x2*>(os + (r * M + ln) * (kOStride * 2) + (db * M + g * 8 + lg * 4) * 2) = w;
        }
    __syncthreads();
    {
      const int chunk = lane & 15;
      uint16_t* op = p.out + blk * p.o_sn + b * p.o_sb + hq * p.o_sh + chunk * 8;
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int r = (lane >> 4) + 4 * it;
        const int row = q0 + wave * 32 + r;
        if (row < p.Sq && chunk * 8 < p.D) {
          const u32x4 w = *reinterpret_cast<const u32x4*>(os + r * (kOStride * 2) + chunk * 16);
          *reinterpret_cast<u32x4*>(op + (int64_t)row * p.o_ss) = w;
        }
      }
    }
  } else {
    // ---- several key groups -----------------------------------------------------------------------------------
    if (ntiles > 0) {
      constexpr int kQCpy = kRows / kWaves / 4;        // every Q row is needed by KS wavefronts
      copy_k(0, 0);
#pragma unroll
      for (int u = 0; u < kQCpy; ++u)
        copy_q(4 * (kQCpy * wave + u), lds_smem + kQBase + (kQCpy * wave + u) * 1024);
      copy_v(0, 0);
      copy_k(1, 1);
      copy_v(1, 1);
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(3 * kCpy) : "memory");     // K(0) and Q
      __builtin_amdgcn_s_barrier();
      read_q(lds_smem + kQBase + rg * (32 * kD * 2));
      qk();
      sm_mask(0);
      sm_fix(true);
      sm_exps();
#pragma unroll
      for (int r = 0; r < R; ++r) l_run[r] = rs[r];
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kCpy) : "memory");         // V(0) and K(1)
      __builtin_amdgcn_s_barrier();
      copy_k(2, 0);
      if (ntiles > 1) first_frags();
    }
    // The same two phases per tile as above, with two stages per ring: K(t+2) and V(t+1), requested in the vector phase
    // before, are waited for behind the matrix phase of tile t, and the barrier there makes them visible to the group
    // and says that K(t+1) and V(t) have been read by all of it, whose stages then take K(t+3) and V(t+2).
    if (group_b) __builtin_amdgcn_s_barrier();
    for (int t = 0; t + 1 < ntiles; ++t) {
      __builtin_amdgcn_s_setprio(2);
      matrix_phase(t);
      __builtin_amdgcn_s_setprio(0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      for (int r = 0; r < R; ++r) asm volatile("" : "+v"(s[0][r]), "+v"(s[MB - 1][r]));
      copy_k(t + 3, (t + 1) & 1);
      copy_v(t + 2, t & 1);
      sm_tile();
      if (t + 2 < ntiles) first_frags();
      __builtin_amdgcn_s_barrier();
    }
    if (ntiles > 0) pv();
    if (!group_b) __builtin_amdgcn_s_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // copies of tiles past the end
    __syncthreads();                                   // nobody reads Q, K or V any more

    // ---- the key groups' partial results meet ------------------------------------------------------------------
    // Each group leaves its reference score and sum per row, scales its O by its weight in the row's result, and hands
    // the head-dim columns it does not finish itself to the group that does (group g: chunks g * kShare .. of 8 columns).
    constexpr int kShare = DB * 4 / KS;                // chunks of 8 columns (4 registers of each lane half) per group
    f32x2* stats = reinterpret_cast<f32x2*>(smem + kQBase);              // [key group][row]
    const float l_own = pair_sum(l_run[0]);
    if (lg == 0) stats[kg * kRows + rg * 32 + ln] = f32x2{m_ref[0], l_own};
    __syncthreads();
    float m_all = -INFINITY;
    f32x2 st[KS];
#pragma unroll
    for (int g = 0; g < KS; ++g) {
      st[g] = stats[g * kRows + rg * 32 + ln];
      if (st[g][1] > 0.f) m_all = fmaxf(m_all, st[g][0]);
    }
    float l_tot = 0.f;
#pragma unroll
    for (int g = 0; g < KS; ++g)       // (a sum of NaN is no smaller than 0 and goes into the row's)
      l_tot += st[g][1] > 0.f ? st[g][1] * fast_exp2((st[g][0] - m_all) * scale_log2) : st[g][1];
    const float weight = l_own > 0.f ? fast_exp2((m_ref[0] - m_all) * scale_log2) / l_tot : 0.f;
    if (kg == 0 && lg == 0 && my_q < p.Sq)
      p.lse[blk * p.l_sn + ((int64_t)b * p.Hq + hq) * p.Sq + my_q] =
          l_tot > 0.f ? __builtin_fmaf(fast_log2(l_tot), kLn2, m_all * p.scale) : -INFINITY;
    // slot (row group, finishing group, giving group): kShare vectors of 64 lanes x 16 bytes
    auto slot = [&](int to, int from) {
      return reinterpret_cast<f32x4*>(smem) + ((rg * KS + to) * KS + from) * (kShare * 64) + lane;
    };
    f32x4 keep[kShare];
#pragma unroll
    for (int to = 0; to < KS; ++to) {
      f32x4* dst = slot(to, kg);
#pragma unroll
      for (int c = 0; c < kShare; ++c) {
        const int unit = to * kShare + c;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = o_acc[unit >> 2][0][(unit & 3) * 4 + e] * weight;
        if (to == kg) keep[c] = v;
        else dst[c * 64] = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int o = 1; o < KS; ++o) {
      const f32x4* src = slot(kg, (kg + o) % KS);
#pragma unroll
      for (int c = 0; c < kShare; ++c) keep[c] += src[c * 64];
    }
    // rows of 256 bytes, chunks swizzled like the K rows
    unsigned char* os = smem + kQBase + rg * (32 * kD * 2);
#pragma unroll
    for (int c = 0; c < kShare; ++c) {
      u32x2 w;
      w[0] = pack_bf16(keep[c][0], keep[c][1]);
      w[1] = pack_bf16(keep[c][2], keep[c][3]);
      *reinterpret_cast<u32x2*>(os + ln * 256 + (((kg * kShare + c) ^ swz(ln)) << 4) + lg * 8) = w;
    }
    __syncthreads();
    {
      constexpr int kRowsPerWave = kRows / kWaves;
      const int chunk = lane & 15;
      uint16_t* op = p.out + blk * p.o_sn + b * p.o_sb + hq * p.o_sh + chunk * 8;
#pragma unroll
      for (int it = 0; it < kRowsPerWave / 4; ++it) {
        const int r = wave * kRowsPerWave + (lane >> 4) + 4 * it;
        if (q0 + r < p.Sq && chunk * 8 < p.D) {
          const u32x4 w = *reinterpret_cast<const u32x4*>(smem + kQBase + r * 256 + ((chunk ^ swz(r)) << 4));
          *reinterpret_cast<u32x4*>(op + (int64_t)(q0 + r) * p.o_ss) = w;
        }
      }
    }
  }
}

// Whether the workgroups of a launch with one key group, of `tiles` key tiles each (causal: at most), use 16 x 16 MFMA tiles:
// those that keep every CU busy, whose time is the board's power, and for long enough that their ends do not count.
// Measured, us, 32 x 32 / 16 x 16 (workgroups x tiles):
//     D 128  512 x 512  1644 / 1554   256 x 256   419 /  399   224 x 512   750 /  711   256 x 32  59.6 / 58.6   512 x 8  42.9 / 43.6
//            160 x 512   595 /  597   288 x 512  1333 / 1344   160 x 20   29.1 / 32.0
//     D 96   512 x 128   338 /  328   256 x 64   90.0 / 87.1   224 x 64   80.1 / 80.1   256 x 32  46.6 / 46.5   160 x 20  24.3 / 27.0
//     D 64   runs of chunks: 8 chunks 4096 x 4096 H32 1018 / 1002, H32/8 1020 / 979, 4 chunks 8192 x 8192 H32 2047 / 1973,
//            8 chunks 2048 x 2048 H32 262 / 249, B2 H32/4 524 / 490        224 x 512   477 /  498
//     causal 4096 x 4096 H32: D 128  122.9 / 117.5   D 96  98.1 / 96.7   D 64  74.6 / 75.5
// (on 96 columns 1.4 % at the one causal size measured was not taken for enough).  Chunk by chunk launches up to 64 columns, whose
// vector work is the larger part, gain and lose by turns and more often lose: D 64 4096 x 4096 H32 139 / 134, H32/8 132 / 134,
// 7900 x 7900 H8 122 / 125, 8192 x 8192 H16/2 258 / 264, 16384 x 8192 B2 H8 516 / 527, 4096 x 16384 H64/8 1013 / 1041, B4 H32/4 6000 x 6000
// 1140 / 1156, H32 1181 / 1183; D 40 4000 x 4500 B4 H16 278 / 284.  All on N(0,1) operands.  The fewer bits the
// operands toggle the less there is to save: 4096 x 4096 H32 of N(0,1) values 218 / 213, of integers from -2 to 2 198 / 192, of zeros,
// which no clock has to give way to, 146 / 175 (D 96 120 / 145).
bool small_tiles(const FwdParams& p, bool causal, int64_t tiles) {
  const int64_t total = (int64_t)p.blocks * p.B * p.Hq * ((p.Sq + kBM - 1) / kBM), rounds = (total + 255) / 256;
  if (p.D <= 64 && p.per == 1) return false;
  if (causal) return p.D > 96 && tiles >= 64 && total >= 512;
  return p.D > 96 ? tiles >= 32 && total * 20 >= rounds * 256 * 17 : tiles >= 64 && total * 20 >= rounds * 256 * 19;
}

template <bool CAUSAL, int KK, int KS, int M = 32>
void launch_one(FwdChunks& p, hipStream_t stream) {
  const int rows = kBM / KS;
  p.nq_tiles = (p.Sq + rows - 1) / rows;
  p.total = p.blocks * p.heads * p.nq_tiles;
  p.per_xcd = (p.total + 7) / 8;
  p.heads_per_xcd = (p.blocks * p.heads) % 8 == 0 ? p.blocks * p.heads / 8 : 0;
  p.by_q_tiles = Divisor(p.nq_tiles);
  p.by_order = Divisor(p.heads_per_xcd > 0 ? p.heads_per_xcd : p.blocks * p.heads);
  const dim3 grid(p.per_xcd * 8), block(kWaves * 64);
  const FwdParams& lone = p;
  if (p.blocks > 1) hipLaunchKernelGGL((attn_fwd_bf16_d128<CAUSAL, KK, KS, FwdChunks, false, M>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((attn_fwd_bf16_d128<CAUSAL, KK, KS, FwdParams, false, M>), grid, block, 0, stream, lone);
}
template <int KK>
void launch_chain(FwdChunks& p, hipStream_t stream) {
  p.nq_tiles = (p.Sq + kBM - 1) / kBM;
  p.total = p.blocks * p.heads * p.nq_tiles;
  p.per_xcd = (p.total + 7) / 8;
  p.heads_per_xcd = 0;
  p.by_q_tiles = Divisor(p.nq_tiles);
  p.by_order = Divisor(1);
  const dim3 grid(p.per_xcd * 8), block(kWaves * 64);
  if (small_tiles(p, false, (int64_t)p.per * ((p.Sc + kBN - 1) / kBN)))
    hipLaunchKernelGGL((attn_fwd_bf16_d128<false, KK, 1, FwdChunks, true, 16>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((attn_fwd_bf16_d128<false, KK, 1, FwdChunks, true>), grid, block, 0, stream, p);
}
template <int KK>
void launch_fwd(FwdChunks& p, bool causal, int groups, hipStream_t stream) {
  if constexpr (KK > 4)
    if (groups == 1 && small_tiles(p, causal, (p.Sc + kBN - 1) / kBN)) {
      if (!causal) return launch_one<false, KK, 1, 16>(p, stream);
      if constexpr (KK == 8) return launch_one<true, KK, 1, 16>(p, stream);
    }
  if (causal) {
    if (groups == 4) launch_one<true, KK, 4>(p, stream);
    else if (groups == 2) launch_one<true, KK, 2>(p, stream);
    else launch_one<true, KK, 1>(p, stream);
  } else {
    if (groups == 4) launch_one<false, KK, 4>(p, stream);
    else if (groups == 2) launch_one<false, KK, 2>(p, stream);
    else launch_one<false, KK, 1>(p, stream);
  }
}

// Key groups per workgroup (1, 2 or 4): the count with the least estimated time.  A launch is rounds of up to 256
// workgroups (one per CU); a workgroup costs `fixed` us (Q in, O out, the groups' meeting) and per tile of a group
// `step` us, plus `busy` us times the share of the CUs at work (clock and L2).  Fitted to launches of 4 .. 2048
// workgroups over 64 .. 4096 keys, which it gives to within 15 %; measured (us, groups 1 / 2 / 4):
//     B1 H4  256 x 256      11.2 /  9.2 /  7.8      B4 H5   512 x 512     16.1 / 12.5 / 10.7
//     B1 H32 1024 x 1024    28.8 / 22.6 / 29.6      B2 H16 1237 x 1237    25.2 / 35.4 / 38.7  (D 80)
//     B1 H1  4096 x 4096    70.3 / 45.6 / 33.8      B1 H20 4096 x 4096     187 /  176 /  200
//     B1 H32 4096 x 4096     228 /  255 /  357      B2 H12 1500 x 1500    24.2 / 18.5 / 24.6  (D 64, causal)
// The split kernel puts whole tiles out of range through 32-bit offsets, which asks for spans below 2^30 bytes.
const LaunchCost* costs(int D) {
  static constexpr LaunchCost kCost128[3] = {{7.0f, 1.10f, 0.80f}, {6.5f, 1.19f, 0.90f}, {5.2f, 0.81f, 0.49f}};
  static constexpr LaunchCost kCost96[3] = {{6.5f, 0.62f, 0.66f}, {6.2f, 1.08f, 0.58f}, {4.9f, 0.76f, 0.30f}};
  static constexpr LaunchCost kCost64[3] = {{6.0f, 0.65f, 0.30f}, {6.0f, 0.98f, 0.27f}, {4.7f, 0.72f, 0.12f}};
  return D <= 64 ? kCost64 : D <= 96 ? kCost96 : kCost128;
}
int key_groups(const FwdParams& p, bool causal, float* time_of_best = nullptr) {
  if ((int64_t)p.Sc * p.k_ss >= (1 << 29) || (int64_t)p.Sc * p.v_ss >= (1 << 29)) return 1;
  const LaunchCost* cost = costs(p.D);
  int best = 1;
  float best_time = 0.f;
  for (int i = 0; i < 3; ++i) {
    const int groups = 1 << i;
    const int rows = kBM / groups, tile = groups == 4 ? 32 : kBN;
    const int64_t q_tiles = (p.Sq + rows - 1) / rows;
    const float n = (float)((int64_t)p.blocks * p.B * p.Hq * q_tiles);
    auto steps = [&](int64_t keys) { return (float)((keys + tile * groups - 1) / (tile * groups)); };
    float time;
    if (!causal) {
      time = rounds_time(n, steps(p.Sc), cost[i]);
    } else {
      // longest tiles first: the longest workgroup, or all of the work spread over the CUs
      const int64_t shift = (int64_t)p.Sc - p.Sq;
      auto seen = [&](int64_t row_end) {
        const int64_t k = row_end + shift < p.Sc ? row_end + shift : p.Sc;
        return k > 0 ? k : 0;
      };
      const float first = steps(seen(rows)), last = steps(seen(q_tiles * rows));
      const float share = n < 256.f ? n / 256.f : 1.f;
      const float longest = cost[i].fixed + last * (cost[i].step + 0.5f * share * cost[i].busy);
      const float spread = n / 256.f * (cost[i].fixed + 0.5f * (first + last) * (cost[i].step + cost[i].busy));
      time = longest > spread ? longest : spread;
    }
    if (i == 0 || time < best_time) { best = groups; best_time = time; }
  }
  if (time_of_best) *time_of_best = best_time;
  return best;
}

}  // namespace

int attn_fwd_bf16_plan(int blocks, int B, int Sq, int Sc, int Hq, int D, int64_t k_ss, int64_t v_ss, int mask) {
  FwdParams p{};
  p.blocks = blocks;
  p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq; p.D = D;
  p.k_ss = k_ss; p.v_ss = v_ss;
  return key_groups(p, mask == MHIP_MASK_CAUSAL);
}

int attn_fwd_bf16_tile(int n, int per, int B, int Sq, int Sc, int Hq, int D, int64_t k_ss, int64_t v_ss, int mask) {
  FwdParams p{};
  p.blocks = (n + per - 1) / per; p.per = per;
  p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq; p.D = D;
  p.k_ss = k_ss; p.v_ss = v_ss;
  const bool causal = mask == MHIP_MASK_CAUSAL;
  return (per > 1 || key_groups(p, causal) == 1) && small_tiles(p, causal, (int64_t)per * ((Sc + kBN - 1) / kBN)) ? 16 : 32;
}

// Chunks of a result (1, or how many a workgroup visits one after the other) of a launch of n chunks: the count with the least
// estimated time, the fold of the results included (which is nothing where there is only one).  Where the blocks would all
// run side by side a run of chunks would only make the longest chain longer.  Whole steps of 8 chunks, us, one / two / four /
// eight chunks to a result: 512 x 512 B4 H5 43.9 / 36.0 / 49.7 / 76.1, 1024 x 1024 H32 148 / 133 / 128 / 154, 2048 x 2048 H32
// 488 / 471 / 464 / 441, 4096 x 4096 H32 1790 / 1772 / 1761 / 1720, 1237 x 1237 B2 H16/8 D80 168 / 167 / 199 / 163, 700 x 700 H12
// D64 36.2 / 29.2 / 45.4 / 75.2, 3000 x 3000 H16 D96 433 / 424 / 455 / 432.
int attn_fwd_bf16_chain(int n, int B, int Sq, int Sc, int Hq, int D) {
  if (n < 2 || Sc == 0) return 1;
  FwdParams p{};
  p.blocks = n; p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq; p.D = D;
  const float wgs = (float)B * Hq * ((Sq + kBM - 1) / kBM);
  if (wgs * n <= 256.f) return 1;
  int best = 1;
  float best_time;
  key_groups(p, false, &best_time);
  best_time += fold_time(n, B, Sq, Hq, D);
  for (int results = n; results >= 1; --results) {
    const int per = (n + results - 1) / results;
    if (per == 1 || (n + per - 1) / per != results) continue;
    // (a chain's tiles take a little longer: as one chunk of twice the keys, 2 x 4096 keys take 1.2 % more on 128 columns, up
    // to 4 % on 64, and its launch has no pauses in which the clock recovers)
    LaunchCost c = costs(D)[0];
    c.step *= D > 96 ? 1.03f : 1.05f;
    c.busy *= D > 96 ? 1.03f : 1.05f;
    const float time = rounds_time(wgs * results, (float)per * ((Sc + kBN - 1) / kBN), c) + fold_time(results, B, Sq, Hq, D);
    if (time < best_time) { best_time = time; best = per; }
  }
  return best;
}

int attn_fwd_bf16(const void* q, const void* const* ks, const void* const* vs, int n, int per, void* out, int64_t o_sn, float* lse,
                  int B, int Sq, int Sc, int Hq, int Hkv, int D,
                  const int64_t* st, float scale, int mask, hipStream_t stream) {
  FwdChunks p;
  p.q = static_cast<const uint16_t*>(q);
  for (int i = 0; i < kMaxGroup; ++i) {
    p.k[i] = i < n ? static_cast<const uint16_t*>(ks[i]) : nullptr;
    p.v[i] = i < n ? static_cast<const uint16_t*>(vs[i]) : nullptr;
  }
  p.k0 = p.k[0]; p.v0 = p.v[0];
  p.per = per; p.chunks = n;
  p.blocks = (n + per - 1) / per; p.heads = B * Hq;
  p.o_sn = o_sn; p.l_sn = (int64_t)B * Hq * Sq;
  p.out = static_cast<uint16_t*>(out);
  p.lse = lse;
  p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq;
  p.by_heads = Divisor(B * Hq); p.by_hq = Divisor(Hq); p.by_group = Divisor(Hq / Hkv);
  p.D = D;
  p.q_sb = st[0]; p.q_ss = st[1]; p.q_sh = st[2];
  p.k_sb = st[3]; p.k_ss = st[4]; p.k_sh = st[5];
  p.v_sb = st[6]; p.v_ss = st[7]; p.v_sh = st[8];
  p.o_sb = st[9]; p.o_ss = st[10]; p.o_sh = st[11];
  p.scale = scale;
  p.scale_log2 = scale * kLog2e;
  const bool causal = mask == MHIP_MASK_CAUSAL;
  if (per > 1) {
    if (causal || Sc == 0 || p.k_ss != p.v_ss) return MHIP_EUNSUPPORTED;
    if (D <= 64) launch_chain<4>(p, stream);
    else if (D <= 96) launch_chain<6>(p, stream);
    else launch_chain<8>(p, stream);
    return launch_status();
  }
  const int groups = key_groups(p, causal);
  if (D <= 64) launch_fwd<4>(p, causal, groups, stream);        // half the on-chip columns, half the MFMAs
  else if (D <= 96) launch_fwd<6>(p, causal, groups, stream);   // three quarters of both
  else launch_fwd<8>(p, causal, groups, stream);
  return launch_status();
}

}  // namespace mhip
