// Block forward on e4m3 (OCP float8) Q/K/V for gfx950: out = softmax(scale * q k^T) v in bf16 and
// lse in fp32, with x ~ descale_x * x_q per tensor.  Both contractions run on the 64-deep fp8 MFMA
// (v_mfma_f32_32x32x64_f8f6f4, twice the rate of the bf16 one), fp32 softmax.  Not in the reference; same
// call boundary as the bf16 kernel (utils/flash_attn_dsl.py:159-176) with three extra descale arguments.
//
// Same decomposition as the bf16 kernel: wavefronts of 32 Q rows, eight per workgroup or, in small launches,
// four; S^T = K Q^T keeps one Q row per lane, P^T feeds the second MFMA from the accumulator registers, K and V tiles are copied
// global -> LDS without registers in between, four stages deep.  Differences:
//   * a main-loop tile is 128 keys (as many bytes as the 64-key bf16 tile), rows of 128 bytes whose eight
//     16-byte chunks are XOR-swizzled;
//   * an MFMA takes 32 bytes per lane and operand: for S^T two 16-byte LDS reads of one K row, for O^T four
//     ds_read_b64_tr_b8 of the row-major V tile (8 keys of one head-dim column each);
//   * the K rows of a 32-key block are assigned to the MFMA rows through a permutation chosen so that a
//     lane's 16 accumulator registers hold 16 CONSECUTIVE keys (16 hf + i): the transposing reads, which
//     deliver 8 consecutive keys, then produce V^T in exactly the key order of the P registers;
//   * the descales fold into the softmax scale (q, k) and the final normalisation (v);
//   * P is multiplied by 2^4 before it is rounded to e4m3 (and the result divided by 2^4), so that small
//     probabilities keep their relative precision; the reference score of a row is its first tile's maximum
//     and moves only when the sum of a group of 16 values of 2^4 P reaches the e4m3 maximum of 448 (the sums
//     are watched, not the maxima: the common path has no maximum, no cross-lane exchange, no rescale of O).
//
// What bounds it: the vector work of the softmax (64 fma, exponentials and adds and 32 conversions per 128 keys and lane,
// about 1470 cycles beside 1024 of MFMA) and, with both units at work, the board's power.  A tile is therefore handled
// as two halves, the MFMAs of the halves before and after threaded through the exponentials of the current one: at 16384 x
// 16384 H32 4.14 M cycles instead of 4.84 M (vector unit 71 % busy instead of 62 %, matrix pipe 51 % instead of 43 %), of
// which the clock gives a part back (1.79 GHz instead of 1.94 on the box of the counters): 2078 us instead of 2212.
#include "mhip_common.hpp"

namespace mhip {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(int)))) int i32x8;
typedef __attribute__((__vector_size__(2 * sizeof(int)))) int i32x2;

constexpr int kD = 128;
constexpr int kBN = 128;              // keys per tile
constexpr int kTileBytes = kBN * kD;  // 16384: one K or V tile in LDS, 128 rows of 128 bytes
constexpr int kStages = 4;
constexpr int kVBase = kStages * kTileBytes;
constexpr int kOStride = kD + 8;
constexpr float kPShift = 4.f;        // P is stored as 2^4 P in e4m3
constexpr float kTrigger = 448.f;     // the e4m3 maximum: a group of 16 exponentials has to sum to less
constexpr int kNoColumn = 0x7fff0000;  // vector offset that is out of every descriptor's range (spans stay below 2^30
                                       // when it is used, and so does the scalar tile offset added to it)

struct Fp8Params {
  // what a workgroup needs before its first copy: read by one group of loads (see load_now)
  int per_xcd, total, blocks, nq_tiles, heads_per_xcd;       // as in the bf16 kernel
  int Sq, Sc;
  int D;             // head dimension of the tensors, a multiple of 16 up to kD; columns D .. kD-1 are zeros on chip
  Divisor by_q_tiles, by_hq, by_group;
  Divisor by_order;  // causal: by the (block, batch, head) triples, or by those of an XCD
  const uint8_t* q; const uint8_t* k0; const uint8_t* v0;            // k0, v0: the first block's chunk
  int64_t q_sb, q_ss, q_sh, k_sb, k_ss, k_sh, v_sb, v_ss, v_sh;
  const float* q_descale; const float* k_descale; const float* v_descale;   // device scalars, NULL = 1
  float scale;       // softmax scale
  // the rest
  int per, chunks;   // as in the bf16 kernel: consecutive chunks of a result, chunks of the launch
  Divisor by_heads;  // by B * Hq
  int heads;         // B * Hq
  int B, Hq;
  uint16_t* out; float* lse;
  int64_t o_sb, o_ss, o_sh;
  int64_t o_sn, l_sn;    // from one block's results to the next one's, elements
};
struct Fp8Chunks : Fp8Params {       // of a launch over several chunks, as in the bf16 kernel
  const uint8_t* k[kMaxGroup]; const uint8_t* v[kMaxGroup];          // the chunk of every block
};

// Chunk c (16 bytes) of row r of a tile lives at chunk position c ^ swz8(r).  Row pairs share a 256-byte
// bank line, so the position inside the line is (r & 1, c ^ swz8(r)): the 32 rows of one 16-byte operand
// read and the 16 rows x 2 chunks of one transposing read both cover the 16 positions exactly twice.
__device__ __forceinline__ constexpr int swz8(int row) { return (((row >> 1) & 3) << 1) | ((row >> 3) & 1); }

// DB = blocks of 32 head-dim values in O^T: 4 computes on all 128 on-chip columns; 2 and 3 are the instantiations for head
// dimensions up to 64 and up to 96, which leave out the MFMAs, operand reads and accumulators of the zero columns (1
// and 2 k-steps of 64 in S^T).  The vector work of a tile stays, and it is the larger part: 4096 x 4096 H32 takes 104.6 us
// at D 64 and 129.8 at D 96 where 128 columns take 139.2; results the same.
//
// WAVES = wavefronts of 32 Q rows in a workgroup: eight, two per SIMD, or four where a launch of eight leaves half of the
// CUs without a workgroup.  A wavefront with a SIMD to itself takes less time for a tile than two that share one
// (four / eight): 2048 x 2048 H16 24.2 / 32.4 us, 4096 x 4096 H2 39.8 / 56.9, causal 1024 x 1024 H32/8 15.5 / 21.3; results
// the same.
//
// CHAIN: a workgroup visits p.per chunks one after the other, as in the bf16 kernel.
template <bool CAUSAL, int DB, int WAVES, class P, bool CHAIN = false>
__global__ __launch_bounds__(WAVES * 64, WAVES / 4) void attn_fwd_fp8_d128(const P p) {
  constexpr bool kLone = std::is_same<P, Fp8Params>::value;
  static_assert(!CHAIN || !kLone, "a run of chunks needs their addresses");
  static_assert(WAVES == 8 || WAVES == 4, "two wavefronts per SIMD or one");
  constexpr int kBM = WAVES * 32;
  constexpr int kCpy = 16 / WAVES;              // copy instructions per wavefront for one 16 KB tile
  static_assert(DB >= 2 && DB <= 4, "64, 96 or 128 on-chip head-dim columns");
  constexpr int KK = (DB + 1) / 2;              // k-steps of 64 head-dim values in S^T
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kStages * kTileBytes];

  // The per-tensor descales are read from device memory here (one scalar load each), so a step whose operands are
  // re-quantised every time needs no device-to-host copy and a captured graph sees the values of the replay.
  const float qd = p.q_descale ? *p.q_descale : 1.f;
  const float kd = p.k_descale ? *p.k_descale : 1.f;
  const float out_mul = p.v_descale ? *p.v_descale : 1.f;
  const float scale_eff = p.scale * qd * kd;      // natural-log scale of the integer-like dot
  const float scale_log2 = scale_eff * kLog2e;

  // Workgroup i runs on XCD i % 8: every XCD gets a contiguous range of (batch, head) pairs, so the
  // workgroups that share a K/V head share an L2.  Causal launches run the longest Q tiles first,
  // across all heads.
  load_now<CAUSAL>(p, p.scale);
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
  const uint8_t* kp = p.k0; const uint8_t* vp = p.v0;
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
  const int q0 = qt * kBM;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int ln = lane & 31;
  const int hf = lane >> 5;

  int kv_end = p.Sc;
  if (CAUSAL) {
    const int lim = q0 + kBM + (p.Sc - p.Sq);
    kv_end = lim < kv_end ? lim : kv_end;
    if (kv_end < 0) kv_end = 0;
  }
  int ntiles = (kv_end + kBN - 1) / kBN;
  int chunks_left = 0;                          // CHAIN: behind the first one
  if (CHAIN) {
    chunks_left = (p.chunks - chunk < p.per ? p.chunks - chunk : p.per) - 1;
    ntiles *= chunks_left + 1;
  }

  // ---- Q fragment: B operand of S^T, lane (ln, hf) holds bytes [64 ks + 32 hf, +32) of its row ------------
  const int my_q = q0 + wave * 32 + ln;
  i32x8 qf[KK];    // loaded after the first tile copies are under way, so that one wait covers both latencies

  // ---- global -> LDS copies: wavefront w copies 8 kCpy rows of every K and V tile, 1 KB per
  // instruction; lane l of instruction u lands at row 8 (kCpy w + u) + l/8, chunk position l%8, and
  // fetches the chunk that lives there.  Rows past the end of the chunk arrive as zeros. ---------------------
  // Chunks past the head dimension (D < 128) carry an offset that is out of range for every tile and arrive as
  // zeros too: a tile in LDS always has 128 columns, at no cost in memory traffic.
  u32x4 krs = rsrc_words(kp + b * p.k_sb + hk * p.k_sh, (uint32_t)((int64_t)(p.Sc - 1) * p.k_ss + p.D));
  u32x4 vrs = rsrc_words(vp + b * p.v_sb + hk * p.v_sh, (uint32_t)((int64_t)(p.Sc - 1) * p.v_ss + p.D));
  int kvoff[kCpy], vvoff[kCpy];
#pragma unroll
  for (int u = 0; u < kCpy; ++u) {
    const int row = 8 * (kCpy * wave + u) + (lane >> 3);
    const int chunk = (lane & 7) ^ swz8(row);
    const bool real = chunk * 16 < p.D;
    kvoff[u] = real ? (int)(row * p.k_ss) + chunk * 16 : kNoColumn;
    vvoff[u] = real ? (int)(row * p.v_ss) + chunk * 16 : kNoColumn;
  }
  const int k_tile_bytes = (int)(kBN * p.k_ss);
  const int v_tile_bytes = (int)(kBN * p.v_ss);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * (kCpy * 1024);
  // CHAIN: K and V tiles are requested in order; k_off and v_off are the offsets of the next ones inside their chunks, k_pos
  // and v_pos their numbers (rows may all lie at one place).  (The address of a chunk is loaded inside its branch and waited
  // for there.)
  const int chunk_tiles = (p.Sc + kBN - 1) / kBN;
  int k_off = 0, v_off = 0, k_pos = 0, v_pos = 0, k_chunk = chunk, v_chunk = chunk;
  const int last_chunk = chunk + chunks_left;
  auto enter = [&](u32x4& rs, const uint8_t* base) {
    asm volatile("" : "+s"(base));
    rs[0] = (uint32_t)(uint64_t)base;
    rs[1] = (uint32_t)((uint64_t)base >> 32) & 0xffffu;
  };
  auto copy_k = [&](int u, int t) {
    copy16_to_lds(krs, lds_base + (t & 3) * kTileBytes + u * 1024, kvoff[u], CHAIN ? k_off : t * k_tile_bytes);
  };
  auto copy_v = [&](int u, int t) {
    copy16_to_lds(vrs, lds_base + kVBase + (t & 3) * kTileBytes + u * 1024, vvoff[u], CHAIN ? v_off : t * v_tile_bytes);
  };
  auto chain_k = [&]() {                        // behind the copies of a K tile
    if (!CHAIN) return;
    k_off += k_tile_bytes;
    if (++k_pos == chunk_tiles && k_chunk != last_chunk) {
      k_off = k_pos = 0;
      ++k_chunk;
      if constexpr (CHAIN) enter(krs, p.k[k_chunk] + b * p.k_sb + hk * p.k_sh);
    }
  };
  auto chain_v = [&]() {
    if (!CHAIN) return;
    v_off += v_tile_bytes;
    if (++v_pos == chunk_tiles && v_chunk != last_chunk) {
      v_off = v_pos = 0;
      ++v_chunk;
      if constexpr (CHAIN) enter(vrs, p.v[v_chunk] + b * p.v_sb + hk * p.v_sh);
    }
  };

  // K operand of S^T: MFMA row m of block mb is key 32 mb + pi(m), pi(8 g + 4 h + e) = 16 h + 4 g + e, so
  // that accumulator register i of lane half hf is key 32 mb + 16 hf + i.  The lane reads chunks
  // 4 ks + 2 hf and 4 ks + 2 hf + 1 of that row.
  const int pi = 16 * ((ln >> 2) & 1) + 4 * (ln >> 3) + (ln & 3);
  // k_a and v_a hold the LDS addresses inside the stage that is read next and move on in place; everything else about an
  // address is an immediate offset.
  const int lds_smem = (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  int k_a[KK][2];                                     // [ks][second 16 bytes]  + mb * 4096
#pragma unroll
  for (int ks = 0; ks < KK; ++ks)
#pragma unroll
    for (int u = 0; u < 2; ++u) k_a[ks][u] = lds_smem + pi * 128 + (((4 * ks + 2 * hf + u) ^ swz8(pi)) << 4);
  // V^T operand of O^T for head-dim block db and k-step ks2 (keys 64 ks2 .. +63): bytes 8 n .. 8 n + 7 of
  // the lane's 32 are keys 64 ks2 + 32 (n / 2) + 16 hf + 8 (n % 2) + 0..7, the keys of its P registers.
  // One ds_read_b64_tr_b8 per n: within 16 lanes, lane s supplies the address of row (first key) + s/2,
  // head-dim bytes 8 (s%2) .. +7 of the 16-column strip, and receives column s.
  int v_a[DB][2];                                     // [db][n % 2]  + ks2 * 8192 + (n / 2) * 4096
  {
    const int s16 = lane & 15, strip = (lane >> 4) & 1;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const int row = 16 * hf + 8 * o + (s16 >> 1);
        v_a[db][o] = lds_smem + kVBase + row * 128 + (((2 * db + strip) ^ swz8(row)) << 4) + (s16 & 1) * 8;
      }
  }
  typedef __attribute__((address_space(3))) i32x2* lds_i32x2;
  typedef __attribute__((address_space(3))) const u32x4* lds_u32x4;
  auto read_k = [&](int mb, int ks) -> i32x8 {
    const u32x4 lo = *(lds_u32x4)(uintptr_t)(uint32_t)(k_a[ks][0] + mb * 4096);
    const u32x4 hi = *(lds_u32x4)(uintptr_t)(uint32_t)(k_a[ks][1] + mb * 4096);
    i32x8 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) { r[e] = (int)lo[e]; r[4 + e] = (int)hi[e]; }
    return r;
  };
  auto read_v = [&](int db, int ks2) -> i32x8 {
    i32x8 r;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const i32x2 t = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (lds_i32x2)(uintptr_t)(uint32_t)(v_a[db][n & 1] + ks2 * 8192 + (n >> 1) * 4096));
      r[2 * n] = t[0]; r[2 * n + 1] = t[1];
    }
    return r;
  };
  const int causal_shift = p.Sc - p.Sq;

  f32x16 o_acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o_acc[i][j] = 0.f;
  // m_ref: the raw score the exponentials of this lane's Q row are taken relative to.  It is set to the first tile's row
  // maximum and moves up only when a later half tile would overflow e4m3: what is watched are the sums of its two groups of
  // 16 exponentials (one compare each), not the maxima.  A group sum below 448 means every 2^4 P in it is below the e4m3
  // maximum; P = 1 for all 16 gives 256.  When a sum reaches 448 the reference moves up to the largest score of the half
  // (O and the running sum are rescaled) and the half's exponentials are redone, after which every 2^4 P is at most 16.  In a
  // run of chunks it also moves, in either direction, where a chunk begins (enter_chunk).
  float m_ref = 0.f, msc = -kPShift, l_run = 0.f;      // l_run sums 2^4 P (this lane's half of the keys)
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 sa[2], sb[2];       // S^T of a tile's first and second half: 64 keys x 32 q rows per wavefront each
  i32x8 pa = {}, pb = {};    // their P^T operands: dwords 0-3 = keys of the half's first 32-key block, dwords 4-7 = second
  auto largest = [&](const f32x16 (&s)[2]) -> float {
    float mx = s[0][0];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int j = 0; j < 16; ++j) mx = fmaxf(mx, s[mb][j]);
    return mx;
  };
  auto set_reference = [&](bool first, float mx) {     // mx: the largest of this lane's scores
    mx = pair_max(mx);
    const bool move = first ? (mx != -INFINITY) : (mx > m_ref);      // false for NaN
    if (!first) {
      const float alpha = move ? fast_exp2((m_ref - mx) * scale_log2) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int j = 0; j < 16; ++j) o_acc[db][j] *= alpha;
    }
    m_ref = move ? mx : m_ref;
    msc = m_ref * scale_log2 - kPShift;            // exponent of 2^4 P
  };
  // 2^4 P of a half into its P^T operand, in eight groups of four scores: step g works out the arguments of group g, adds
  // up and converts group g - 1 and takes the exponentials of group g, so that nothing waits for the instruction
  // before it.  r[] are the sums of the two 32-key blocks (this lane's 16 keys of each).  The scores stay intact, so that
  // the pass can be repeated against a new reference.
  float r[2], x[2][4];
  auto vector_step = [&](int g, const f32x16 (&s)[2], i32x8& pw) {
    if (g < 8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[g & 1][j] = __builtin_fmaf(s[g >> 2][(g & 3) * 4 + j], scale_log2, -msc);
    }
    if (g > 0) {
      const int o = g - 1;
      const float (&e)[4] = x[o & 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) r[o >> 2] = (o & 3) == 0 && j == 0 ? e[0] : r[o >> 2] + e[j];
      // the first conversion writes the low half and the second the high half of the operand register, so
      // what it held before needs no clearing
      int packed = pw[o];
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(e[0], e[1], packed, false);
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(e[2], e[3], packed, true);
      pw[o] = packed;
    }
    if (g < 8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[g & 1][j] = fast_exp2(x[g & 1][j]);
    }
  };
  auto mask_half = [&](f32x16 (&s)[2], int kv0) {
    bool need_mask = kv0 + kBN / 2 > p.Sc;
    if (CAUSAL) need_mask = need_mask || (kv0 + kBN / 2 - 1 > q0 + causal_shift);
    if (need_mask) {
      int lim = p.Sc - 1;
      if (CAUSAL) { const int c = my_q + causal_shift; lim = c < lim ? c : lim; }
      int rest = lim - kv0 - hf * 16;              // CHAIN: one register to compare constants with (32 would count along
      if (CHAIN) asm volatile("" : "+v"(rest));    // with the position in a chunk)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (CHAIN ? mb * 32 + j > rest : kv0 + mb * 32 + hf * 16 + j > lim) s[mb][j] = -INFINITY;
    }
  };
  // after a half's last vector step: move the reference and repeat if a sum reached the trigger (or is inf / NaN)
  auto finish_half = [&](const f32x16 (&s)[2], i32x8& pw) {
    if (__builtin_amdgcn_ballot_w64(!(r[0] < kTrigger) || !(r[1] < kTrigger)) != 0) {
      set_reference(false, largest(s));
#pragma unroll
      for (int g = 0; g <= 8; ++g) vector_step(g, s, pw);
    }
    l_run += r[0] + r[1];
  };

  // Tile t lives in stage t % 4 of the K and the V ring and is processed as two halves of 64 keys.  Every phase of the
  // main loop is one sequence of kSlots MFMAs, S^T of the half after the current one and O^T of the half before it, with
  // the exponentials of the current half between them: the matrix pipe and the vector unit are at work at the same time
  // in every wavefront, whichever way the two wavefronts of a SIMD happen to be aligned.
  //   phase 0 of tile t   S^T(t, second half)    O^T(t-1, second half)   exponentials (t, first half)
  //   phase 1             S^T(t+1, first half)   O^T(t, first half)      exponentials (t, second half)
  // The LDS operand of slot i+2 is read in slot i, across phase and tile boundaries.  An iteration starts by waiting for
  // this wavefront's copies of K(t+1) and V(t) (those of K(t+2) and V(t+1) stay in flight) and a barrier: after it
  // they are complete for every wavefront and nobody reads K(t-1) and V(t-2) any more, whose stages then receive K(t+3)
  // and V(t+2).  Tiles past the end are copied as zeros so that the number of copies in flight stays the same.
  constexpr int kSlotsS = 2 * KK, kSlots = kSlotsS + DB;
  i32x8 ring[2];
  auto read_slot = [&](int half, int i) -> i32x8 {         // half: which phase the slot belongs to
    if (i >= kSlots) { i -= kSlots; half ^= 1; }
    if (i < kSlotsS) return read_k((half ? 0 : 2) + (i & 1), i >> 1);
    return read_v(i - kSlotsS, half ? 0 : 1);
  };
  auto s_mfma = [&](int i, const i32x8& a, f32x16 (&s)[2]) {
    s[i & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, qf[i >> 1], i < 2 ? zero : s[i & 1], 0, 0, 0, 0, 0, 0);
  };
  auto o_mfma = [&](int db, const i32x8& a, const i32x8& pw) {
    o_acc[db] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, pw, o_acc[db], 0, 0, 0, 0, 0, 0);
  };
  int chain_kv0 = 0;                              // CHAIN: first key of the tile inside its chunk
  auto phase = [&](int half, int t, f32x16 (&cur)[2], f32x16 (&next)[2], const i32x8& p_before, i32x8& p_cur) {
    mask_half(cur, (CHAIN ? chain_kv0 : t * kBN) + half * (kBN / 2));
    if (CHAIN && half == 1) chain_kv0 = chain_kv0 + kBN < p.Sc ? chain_kv0 + kBN : 0;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      i32x8& operand = ring[(half * kSlots + i) & 1];
      if (i < kSlotsS) s_mfma(i, operand, next);
      else o_mfma(i - kSlotsS, operand, p_before);
      operand = read_slot(half, i + 2);
      if (half == 0) {
#pragma unroll
        for (int c = i; c < 2 * kCpy; c += kSlots) {
          if (c < kCpy) copy_k(c, t + 3);
          else copy_v(c - kCpy, t + 2);
        }
        // the last K read of this phase was slot kSlotsS - 1's, the last V read slot kSlots - 1's
        if (i == kSlotsS - 2) {
          const int step = ((t + 1) & 3) == 0 ? -3 * kTileBytes : kTileBytes;
#pragma unroll
          for (int ks = 0; ks < KK; ++ks) { k_a[ks][0] += step; k_a[ks][1] += step; }
        }
        if (i == kSlots - 2) {                       // (V(0) stands in for V(-1), whose P is zero)
          const int step = t == 0 ? 0 : (t & 3) == 0 ? -3 * kTileBytes : kTileBytes;
#pragma unroll
          for (int db = 0; db < DB; ++db) { v_a[db][0] += step; v_a[db][1] += step; }
        }
      }
#pragma unroll
      for (int g = i * 8 / kSlots; g < (i + 1) * 8 / kSlots; ++g) vector_step(g, cur, p_cur);
      __builtin_amdgcn_sched_barrier(0);
    }
    vector_step(8, cur, p_cur);
    finish_half(cur, p_cur);
    if (half == 0) {                              // (a branch between the MFMAs would cost 60 registers)
      chain_k();
      chain_v();
    }
  };

  if (ntiles > 0) {
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy_k(u, 0);
    chain_k();
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy_v(u, 0);
    chain_v();
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy_k(u, 1);
    chain_k();
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy_k(u, 2);
    chain_k();
#pragma unroll
    for (int u = 0; u < kCpy; ++u) copy_v(u, 1);
    chain_v();
    const int row = my_q < p.Sq ? my_q : p.Sq - 1;
    const uint8_t* qp = p.q + b * p.q_sb + (int64_t)row * p.q_ss + hq * p.q_sh + hf * 32;
#pragma unroll
    for (int ks = 0; ks < KK; ++ks) {
      const u32x4 none = {0u, 0u, 0u, 0u};                        // columns past the head dimension
      const int col = ks * 64 + hf * 32;
      const u32x4 lo = col < p.D ? *reinterpret_cast<const u32x4*>(qp + ks * 64) : none;
      const u32x4 hi = col + 16 < p.D ? *reinterpret_cast<const u32x4*>(qp + ks * 64 + 16) : none;
#pragma unroll
      for (int e = 0; e < 4; ++e) { qf[ks][e] = (int)lo[e]; qf[ks][4 + e] = (int)hi[e]; }
    }
    // pin the loads here: the copies are invisible to the compiler's wait counting
#pragma unroll
    for (int ks = 0; ks < KK; ++ks) asm volatile("" : "+v"(qf[ks]));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < kSlotsS; ++i) {
      s_mfma(i, read_k(i & 1, i >> 1), sa);
      s_mfma(i, read_k(2 + (i & 1), i >> 1), sb);     // here for the maximum; phase 0 computes it again
    }
    mask_half(sa, 0);
    mask_half(sb, kBN / 2);
    set_reference(true, fmaxf(largest(sa), largest(sb)));
    ring[0] = read_slot(0, 0);
    ring[1] = read_slot(0, 1);
  }
  // CHAIN: where a chunk begins the reference becomes the maximum of its first tile, up or down, as if the chunk had a
  // workgroup of its own: P is rounded relative to it.  The half whose P is still due goes into O first.
  auto enter_chunk = [&]() {
#pragma unroll
    for (int db = 0; db < DB; ++db) o_mfma(db, read_v(db, 1), pb);
    pb = i32x8{};
#pragma unroll
    for (int i = 0; i < kSlotsS; ++i) s_mfma(i, read_k(2 + (i & 1), i >> 1), sb);    // phase 0 computes it again
    mask_half(sa, chain_kv0);
    mask_half(sb, chain_kv0 + kBN / 2);
    const float mx = pair_max(fmaxf(largest(sa), largest(sb)));
    // Down only as far as the row's sum stays below 2^64, over however many chunks, and with it O, of which no element is
    // larger than 448 times the sum.  A chunk that is not followed is 2^40 below what the row has: it adds nothing.
    const float down = fast_exp2((m_ref - mx) * scale_log2);
    const bool move = mx != -INFINITY && pair_sum(l_run) * down < 0x1p64f;      // false for NaN
    const float alpha = move ? down : 1.f;
    l_run *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 16; ++j) o_acc[db][j] *= alpha;
    m_ref = move ? mx : m_ref;
    msc = m_ref * scale_log2 - kPShift;
  };
  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * kCpy) : "memory");
    __builtin_amdgcn_s_barrier();
    if (CHAIN && chain_kv0 == 0 && t > 0) enter_chunk();
    phase(0, t, sa, sb, pb, pa);
    phase(1, t, sb, sa, pa, pb);
  }
  if (ntiles > 0) {
#pragma unroll
    for (int db = 0; db < DB; ++db) o_mfma(db, read_v(db, 1), pb);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the zero-filled copies of tiles past the end

  // ---- epilogue ---------------------------------------------------------------------------------------------
  const float l_tot = pair_sum(l_run);
  const float inv = l_tot > 0.f ? out_mul / l_tot : 0.f;           // the two factors 2^4 cancel
  if (hf == 0 && my_q < p.Sq) {
    const float lse = l_tot > 0.f ? m_ref * scale_eff + (fast_log2(l_tot) - kPShift) * kLn2 : -INFINITY;
    p.lse[blk * p.l_sn + ((int64_t)b * p.Hq + hq) * p.Sq + my_q] = lse;
  }
  __syncthreads();
  unsigned char* os = smem + wave * (32 * kOStride * 2);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u32x2 w;
      w[0] = pack_bf16(o_acc[db][4 * g] * inv, o_acc[db][4 * g + 1] * inv);
      w[1] = pack_bf16(o_acc[db][4 * g + 2] * inv, o_acc[db][4 * g + 3] * inv);
      *reinterpret_cast<u32x2*>(os + ln * (kOStride * 2) + (db * 32 + g * 8 + hf * 4) * 2) = w;
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
}

// A launch of one block takes the short arguments (see FwdChunks of the bf16 kernels; graphs of such launches, us, with the
// chunks' addresses / without: 64 x 64 H1 6.32 / 6.03, 256 x 256 H4 7.15 / 6.93, causal 1024 x 1024 H8 14.5 / 14.0).  Not so
// four wavefronts on 64 columns, whose main loop, the same instructions on other registers, takes longer then (1024 x 1024 H8
// 12.2 / 12.5, 4096 x 4096 H2 34.9 / 36.7).
template <int DB, int WAVES>
void launch_fp8(const Fp8Chunks& p, bool causal, hipStream_t stream) {
  const dim3 grid(p.per_xcd * 8), block(WAVES * 64);
  if constexpr (DB > 2 || WAVES > 4)
    if (p.blocks == 1 && p.per == 1) {
      const Fp8Params& lone = p;
      if (causal) hipLaunchKernelGGL((attn_fwd_fp8_d128<true, DB, WAVES, Fp8Params>), grid, block, 0, stream, lone);
      else hipLaunchKernelGGL((attn_fwd_fp8_d128<false, DB, WAVES, Fp8Params>), grid, block, 0, stream, lone);
      return;
    }
  if (p.per > 1) hipLaunchKernelGGL((attn_fwd_fp8_d128<false, DB, WAVES, Fp8Chunks, true>), grid, block, 0, stream, p);
  else if (causal) hipLaunchKernelGGL((attn_fwd_fp8_d128<true, DB, WAVES, Fp8Chunks>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((attn_fwd_fp8_d128<false, DB, WAVES, Fp8Chunks>), grid, block, 0, stream, p);
}

}  // namespace

// Wavefronts per workgroup.  Four while the launch has at most 256 workgroups of 128 rows: twice the CUs at work.  With
// more, they take turns on the CUs (us, eight / four: 2048 x 2048 H16, 256 of them, 32.4 / 24.2; 2176 x 2176 H16
// 34.2 / 46.5; 2048 x 2048 H32 39.7 / 46.3).  Under the causal mask of a square or tall block the longest workgroups hold
// up the launch until there is twice as much work (2048 x 2048 H20 35.2 / 24.4, H32, 512 workgroups, 36.6 / 30.3, H40
// 38.0 / 42.0; 4096 x 2048 H16 34.6 / 24.6).
int attn_fwd_fp8_plan(int blocks, int B, int Sq, int Sc, int Hq, int mask) {
  return (int64_t)blocks * B * Hq * ((Sq + 127) / 128) > (mask == MHIP_MASK_CAUSAL && Sc <= Sq ? 512 : 256) ? 8 : 4;
}

// Chunks of a result of a launch of n chunks, as for the bf16 kernels.  Costs of workgroups of eight and of four
// wavefronts, fitted to the launches above and 4096 x 4096 H32 at 64, 96 and 128 columns.  Whole steps of 8 chunks, us, one / two /
// four / eight chunks to a result: 1024 x 1024 H32 114 / 94.3 / 89.8 / 92.4, 4096 x 4096 H32 1146 / 1102 / 1094 / 1060.
int attn_fwd_fp8_chain(int n, int B, int Sq, int Sc, int Hq, int D) {
  if (n < 2 || Sc == 0 || (float)n * B * Hq * ((Sq + 255) / 256) <= 256.f) return 1;
  const LaunchCost eight = {6.5f, D <= 64 ? 1.1f : D <= 96 ? 1.45f : 1.55f, D <= 64 ? 0.3f : 0.4f};
  const LaunchCost four = {6.f, D <= 64 ? 0.8f : 1.f, 0.07f};
  auto time = [&](int results, int per) {
    const bool wide = attn_fwd_fp8_plan(results, B, Sq, Sc, Hq, MHIP_MASK_NONE) == 8;
    const float wgs = (float)results * B * Hq * (wide ? (Sq + 255) / 256 : (Sq + 127) / 128);
    return rounds_time(wgs, (float)per * ((Sc + kBN - 1) / kBN), wide ? eight : four) + fold_time(results, B, Sq, Hq, D);
  };
  int best = 1;
  float best_time = time(n, 1);
  for (int results = n; results >= 1; --results) {
    const int per = (n + results - 1) / results;
    if (per == 1 || (n + per - 1) / per != results) continue;
    const float t = time(results, per);
    if (t < best_time) { best_time = t; best = per; }
  }
  return best;
}

int attn_fwd_fp8(const void* q, const void* const* ks, const void* const* vs, int n, int per, void* out, int64_t o_sn, float* lse,
                 int B, int Sq, int Sc, int Hq, int Hkv, int D, const int64_t* st, float scale, int mask,
                 const float* q_descale, const float* k_descale, const float* v_descale, hipStream_t stream) {
  Fp8Chunks p;
  p.q = static_cast<const uint8_t*>(q);
  for (int i = 0; i < kMaxGroup; ++i) {
    p.k[i] = i < n ? static_cast<const uint8_t*>(ks[i]) : nullptr;
    p.v[i] = i < n ? static_cast<const uint8_t*>(vs[i]) : nullptr;
  }
  p.k0 = p.k[0]; p.v0 = p.v[0];
  const int blocks = (n + per - 1) / per;
  p.per = per; p.chunks = n;
  p.blocks = blocks; p.heads = B * Hq;
  p.o_sn = o_sn; p.l_sn = (int64_t)B * Hq * Sq;
  p.out = static_cast<uint16_t*>(out); p.lse = lse;
  p.B = B; p.Sq = Sq; p.Sc = Sc; p.Hq = Hq;
  p.by_heads = Divisor(B * Hq); p.by_hq = Divisor(Hq); p.by_group = Divisor(Hq / Hkv);
  p.D = D;
  p.q_sb = st[0]; p.q_ss = st[1]; p.q_sh = st[2];
  p.k_sb = st[3]; p.k_ss = st[4]; p.k_sh = st[5];
  p.v_sb = st[6]; p.v_ss = st[7]; p.v_sh = st[8];
  p.o_sb = st[9]; p.o_ss = st[10]; p.o_sh = st[11];
  p.scale = scale;
  p.q_descale = q_descale; p.k_descale = k_descale; p.v_descale = v_descale;
  const bool causal = mask == MHIP_MASK_CAUSAL;
  if (per > 1 && (causal || Sc == 0 || p.k_ss != p.v_ss)) return MHIP_EUNSUPPORTED;
  const bool wide = attn_fwd_fp8_plan(blocks, B, Sq, Sc, Hq, mask) == 8;
  const int rows = wide ? 256 : 128;
  p.nq_tiles = (Sq + rows - 1) / rows;
  p.total = blocks * p.heads * p.nq_tiles;
  p.per_xcd = (p.total + 7) / 8;
  p.heads_per_xcd = (blocks * p.heads) % 8 == 0 ? blocks * p.heads / 8 : 0;
  p.by_q_tiles = Divisor(p.nq_tiles);
  p.by_order = Divisor(p.heads_per_xcd > 0 ? p.heads_per_xcd : blocks * p.heads);
  if (D <= 64) wide ? launch_fp8<2, 8>(p, causal, stream) : launch_fp8<2, 4>(p, causal, stream);
  else if (D <= 96) wide ? launch_fp8<3, 8>(p, causal, stream) : launch_fp8<3, 4>(p, causal, stream);
  else wide ? launch_fp8<4, 8>(p, causal, stream) : launch_fp8<4, 4>(p, causal, stream);
  return launch_status();
}

}  // namespace mhip
