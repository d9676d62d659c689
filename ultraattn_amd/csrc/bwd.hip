// Block-sparse flash-attention backward for gfx950 (MI355X): two deterministic kernels that
// recompute P from the rows' LSE, no atomics.
//
//  dkdv_kernel : one workgroup per (key tile, head) walks the CSC column of query tiles.
//                A wavefront owns 32 key rows; K and V fragments stay in registers, the Q and
//                dO tiles stream through LDS.  Products (bf16 MFMA, see Mma):
//                  S [q,key]  = Q K^T          dP[q,key]  = dO V^T
//                  dV^T[d,key] += dO^T P       dK^T[d,key] += Q^T dS
//                In the accumulator layout a lane holds one key column, so S / dP blocks
//                become, after the pointwise step, the B operands of the last two products.
//  dq_kernel   : one workgroup per (query tile, head) walks the CSR row of key tiles.
//                A wavefront owns 32 query rows; Q and dO fragments stay in registers, the K
//                and V tiles stream through LDS:
//                  S^T[key,q] = K Q^T          dP^T[key,q] = V dO^T
//                  dQ^T[d,q] += K^T dS^T
//                Here a lane holds one query column, so lse and delta are per-lane scalars.
//  P = exp2(scale*log2e*S - lse*log2e);  dS = P * (dP - delta);  dQ, dK are scaled by
//  softmax_scale on output.
#include <algorithm>
#include <type_traits>
#include "ua_common.h"

namespace ua {

// One side of the backward: the columns (dK, dV; walks the CSC) or the rows (dQ; walks the CSR).
struct BwdSide {
  const int32_t* ptr; const int32_t* idx; const uint8_t* flag; const int32_t* order;
  bf16* out0; bf16* out1;                  // columns: dk, dv; rows: dq, unused
  Strides3 o0s, o1s;
  // The walk is cut into n_parts parts of part_len tiles; with out_f32 part i leaves an fp32 partial result at
  // out + i * o_part (fp32 elements, contiguous [batch, tokens, heads, 128]) for a later sum.
  int n_parts, part_len, out_f32;
  int64_t o_part;
  BlockMap map;
  Div by_lines;                            // tiles of this side
};
struct BwdParams {
  const bf16* q; const bf16* k; const bf16* v; const bf16* dout;
  const float* lse; const float* delta;
  int batch, n_heads, n_qtiles, n_ktiles, nnz;
  Strides3 qs, ks, vs, ds;
  float scale_log2, scale, neg_inv_scale;
  Div by_heads;
  // Dense rectangle (no list arrays).  The rows walk key tiles [0, n_ktiles) of a query tile, with dense_causal
  // [0, qt + diag_off], the last one causal; the columns walk query tiles [0, n_qtiles) of a key tile, with
  // dense_causal [kt - diag_off, n_qtiles), the first one causal.
  int dense, dense_causal, diag_off;
  int n_col_blocks;                        // bwd_kernel: workgroups of the columns, those of the rows follow
  int cols_reversed;                       // launch order of the columns (see launch_bwd)
  int rows_ahead;                          // the rows' wavefronts go first on a CU (see launch_bwd)
  BwdSide cols, rows;
};

// The kernel's parameters read again from the kernel-argument segment.  What only the epilogue needs is read
// through this, so that it does not occupy scalar registers (or get spilled to vector lanes) during the walk.
typedef const __attribute__((address_space(4))) BwdParams* ParamsLate;
__device__ __forceinline__ ParamsLate params_late() {
  ParamsLate p = (ParamsLate)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}
// What a walk needs is read behind the branch that leads to it: read before, the parameters of both sides at once ask for more
// scalar registers than there are, and up to 61 of them live in vector lanes (causal 32 heads of 2048, backward 131.9 -> 121.6 us with
// the two kinds of walk in kernels of their own).  Of several groups, whose short walks are often the columns', the columns' are in flight before the
// branch.  With both sides' there half lines had ten scalars in vector lanes and a private segment of 20 bytes, which no instruction used but every
// launch paid for (32 heads of 512 18.4 -> 17.7 us, 16 of 1024 30.4 -> 29.8; four groups, 8 heads of causal 1024 18.0 -> 17.7).
template <int kForm, bool kRows>
__device__ __forceinline__ const BwdParams& params_of_walk(const BwdParams& given) { return kForm == 1 || kRows ? *(const BwdParams*)params_late() : given; }
// Brings all parameters into the scalar cache while the first ones are on their way, for walks that read them behind a branch (short
// ones of one group: 171 heads of 128, causal, 15.5 -> 14.9 us, 92 of 128 x 256 15.0 -> 14.3, 32 of 1024 53.2 -> 52.5).
__device__ __forceinline__ void touch_params() {
  constexpr int kLines = 9, kWords = sizeof(BwdParams) / 4;
  static_assert(16 * (kLines - 1) < kWords && kWords <= 16 * kLines, "one word of every 64 bytes");
  const auto* p = (const __attribute__((address_space(4))) int*)__builtin_amdgcn_kernarg_segment_ptr();
  int x[kLines];
#pragma unroll
  for (int i = 0; i < kLines; ++i) x[i] = p[16 * i];
  asm volatile("" :: "s"(x[0]), "s"(x[1]), "s"(x[2]), "s"(x[3]), "s"(x[4]), "s"(x[5]), "s"(x[6]), "s"(x[7]), "s"(x[8]));
}
// 32 output rows of a wave: in the caller's strided bf16 tensor, or in part `part` of the fp32 partials.
template <int kM>
__device__ __forceinline__ void store_result(const __attribute__((address_space(4))) BwdSide* p, bf16* out, int64_t os_b, int64_t os_s,
                                             int64_t os_h, int n_heads, int part, int b, int64_t row0, int h, int64_t seq,
                                             const f32x16 (&acc)[4], float mul, uint32_t lds) {
  if (p->out_f32) {
    float* base = reinterpret_cast<float*>(out) + part * p->o_part;
    store_rows_f32<kM>(base + (((int64_t)b * seq + row0) * n_heads + h) * kHeadDim, (int64_t)n_heads * kHeadDim, acc, both(mul), lds);
  } else {
    store_rows_bf16<kM>(out + b * os_b + row0 * os_s + h * os_h, os_s, acc, both(mul), lds);
  }
}

// The same for one block of 32 columns (several groups).
__device__ __forceinline__ void store_block(const __attribute__((address_space(4))) BwdSide* p, bf16* out, int64_t os_b, int64_t os_s,
                                            int64_t os_h, int n_heads, int part, int b, int64_t row0, int h, int64_t seq, int block,
                                            const f32x16& acc, float mul, uint32_t lds) {
  if (p->out_f32) {
    float* base = reinterpret_cast<float*>(out) + part * p->o_part;
    store_block_f32(base + (((int64_t)b * seq + row0) * n_heads + h) * kHeadDim + 32 * block, (int64_t)n_heads * kHeadDim, acc, mul, lds);
  } else {
    store_block_bf16(out + b * os_b + row0 * os_s + h * os_h + 32 * block, os_s, acc, mul, lds);
  }
}

// ---- dK/dV ------------------------------------------------------------------------------------
// Four wavefronts, wave w owns key rows 32w..32w+31 and keeps their K and V rows as B operands; the
// query side is streamed in half tiles of 64 rows (two blocks of 32) through two LDS stages.  Per block:
//   S = Q K^T - lse/scale,  dP' = dO V^T - delta        16 row fragments, Q and dO read 128 bits at a time
//   P = exp2(scale*log2e*S), dS = P * dP'               in the accumulators' lanes
//   dV^T += dO^T P,  dK^T += Q^T dS                     16 column fragments, Q and dO read through the transposing path
// P and dS never leave the wave.  The accumulators of S and dP' start from the rows' statistics.
//
// Bound: the socket's power (both sides 69 % matrix-pipe busy at 1.87 GHz, causal 32k).  192 of a wave's 256 registers
// hold K, V, dK and dV; two independent workgroups share a CU, so that one's exp2 and barriers hide behind
// the other's MFMAs.  Against one workgroup of eight waves in two roles (S/dV and dP/dK, P handed over
// through LDS): strided 128k, 32 heads 37.8 -> 33.5 ms, causal 32k 15.8 -> 13.7 ms (1.25-1.3 PFLOP/s of the four
// products, both kernels with 32x32x16).
//
// LDS: the V-type layout.  The chunk bits that its XOR leaves alone, the row blocks and the stages are all
// compile-time offsets: four address registers serve the 128-bit reads of both operands and four the transposing ones.
#define UA_LDS __attribute__((address_space(3)))
// A group's LDS: stage s holds the first operand's rows at 2s * kPitch and the second's behind them; then the statistics
// -lse/scale and -delta of either stage and the waves' list entries.
template <int kForm>
struct Stages : Groups<kForm> {
  static constexpr int kM = mma_of(kForm);
  static_assert(kForm == 1 || kM == 32, "sums over groups (add_block, sum_blocks, store_block) take a lane to hold one row");
  static constexpr int kBlockPitch = 8 * Mma<kM>::kPitch;            // 32 rows
  static constexpr int kPitch = Groups<kForm>::kRows / 4 * Mma<kM>::kPitch;
  static constexpr int kStatBytes = 2 * Groups<kForm>::kRows * 4;
  static constexpr int kStat = 4 * kPitch;
  static constexpr int kEntries = kStat + 2 * kStatBytes;
  static constexpr int kBytes = kEntries + (kForm == 1 ? 4 * Walk<false, false>::kBytes : 0);
};
static_assert(3 * Stages<1>::kPitch + Stages<1>::kBlockPitch + 4 * Mma<16>::kPitch + 32 < 65536, "operand offsets fit the instructions' offset field");

__device__ __forceinline__ void keep_in_register(uint32_t& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ float in_scalar(float x) {            // a wave-uniform value in a scalar register
  int bits = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x));
  asm volatile("" : "+s"(bits));
  return __builtin_bit_cast(float, bits);
}
__device__ __forceinline__ bf16x8 lds_abs_b128(uint32_t a) { return *reinterpret_cast<const UA_LDS bf16x8*>(a); }
__device__ __forceinline__ bf16x8 lds_abs_tr_pair(uint32_t a_lo, uint32_t a_hi) {
  const bf16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(reinterpret_cast<UA_LDS bf16x4*>(a_lo));
  const bf16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(reinterpret_cast<UA_LDS bf16x4*>(a_hi));
  return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
}
// Per-lane absolute LDS addresses within the first operand's half tile of stage 0; the second operand, later
// rows and stage 1 are compile-time offsets.
// (The row reads of 32x32x16, whose chunks come in pairs 32 bytes apart that the XOR leaves alone, need four address registers too.)
template <int kM>
struct PairAddr {
  uint32_t nat[4];      // 128-bit row reads
  uint32_t tr[4];       // transposing reads
  __device__ __forceinline__ PairAddr(uint32_t lds_base, int lane) {
    using M = Mma<kM>;
    const int row = M::a_row(lane);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      nat[j] = lds_base + (row >> 2) * M::kPitch + (row & 3) * kRowBytes + (slot_v(row, M::a_chunk(lane, kM == 32 ? 2 * j : j)) << 4);
      tr[j] = lds_base + M::tr_offset(lane, j);
      keep_in_register(nat[j]);
      keep_in_register(tr[j]);
    }
  }
  __device__ __forceinline__ void shift(int bytes) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { nat[j] += bytes; tr[j] += bytes; }
  }
};
// Fragment reads (i of 8) at a compile-time offset: of a block's 32 rows, and of those rows transposed.
template <int kOff, int kM>
__device__ __forceinline__ bf16x8 pair_nat(const PairAddr<kM>& ad, int i) {
  return lds_abs_b128(ad.nat[i >> 1] + (kOff + (kM == 32 ? 32 * (i & 1) : Mma<kM>::a_offset(i, Mma<kM>::kPitch))));
}
template <int kOff, int kM>
__device__ __forceinline__ bf16x8 pair_tr(const PairAddr<kM>& ad, int i) {
  using M = Mma<kM>;
  return lds_abs_tr_pair(ad.tr[M::tr_reg(i)] + (kOff + M::tr_first(i)), ad.tr[M::tr_reg(i)] + (kOff + M::tr_first(i) + M::tr_second()));
}

// The walked pair of operands (Q and dO, or K and V): asynchronous copies of a group's rows into an LDS stage.
// 4 copies per wave and operand; copy j fills group kWaves*j + wave (rows 4*kWaves*j + 4*wave ..), lane l the 16-byte
// slot l%16 of row l/16 of the group, whose logical chunk is the slot XORed with 4 * (l/16).
template <int kForm>
struct PairStream {
  using S = Stages<kForm>;
  static constexpr int kCopies = 8;        // per stage and wave, the operands in turn
  const bf16 *x, *y;
  int xs, ys, xoff, yoff;
  uint32_t lds;
  u32x4 rx, ry;                            // the tile that copies read
  __device__ __forceinline__ PairStream(const bf16* x_, int xs_, const bf16* y_, int ys_, uint32_t lds_base, int wave, int lane)
      : x(x_), y(y_), xs(xs_), ys(ys_) {
    const int row = 4 * wave + (lane >> 4), chunk = (lane & 15) ^ ((lane >> 4) << 2);
    xoff = (row * xs + chunk * 8) * 2;
    yoff = (row * ys + chunk * 8) * 2;
    lds = __builtin_amdgcn_readfirstlane(lds_base + wave * Mma<S::kM>::kPitch);
  }
  // Without `more` the copies that follow read nothing and fill with zeros a stage that no step reads: no branch at each of them.
  __device__ __forceinline__ void tile(int t, bool more) {
    const int64_t row0 = (int64_t)t * kTile;
    rx = make_rsrc_words(x + row0 * xs, more ? (uint32_t)((kTile - 1) * xs + kHeadDim) * 2 : 0);
    ry = make_rsrc_words(y + row0 * ys, more ? (uint32_t)((kTile - 1) * ys + kHeadDim) * 2 : 0);
  }
  // (Opaque in every step: the sums of the copies' LDS addresses would occupy scalar registers all along, and vector lanes.  Half lines have scalars enough.)
  __device__ __forceinline__ void next_step() { if (kForm != kHalves) asm volatile("" : "+s"(lds)); }
  // copy n of kCopies into stage kStage, rows from 64 or 32 * part of the tile on
  template <int kStage>
  __device__ __forceinline__ void copy(int n, int part) const {
    const int j = n >> 1, at = 2 * kStage * S::kPitch + S::kWaves * j * Mma<S::kM>::kPitch, row = part * S::kRows + 4 * S::kWaves * j;
    if (n & 1) dma16_abs(ry, lds + at + S::kPitch, yoff, row * ys * 2);
    else       dma16_abs(rx, lds + at, xoff, row * xs * 2);
  }
};

// One block of 32 query rows for this wave's 32 keys.  kOff = LDS offset of the block's Q rows; dO lies kPitch
// behind, -delta kStatBytes / 2 behind -lse/scale.  `copy(n)`, n = 0 .. kCopies - 1, is called between the first MFMAs.
// With 16x16x32 the first 16 rows' P and dS are made before the second ones' products begin: 8 registers fewer are live, which hold
// a third fragment ahead (all 32 rows at once, two ahead: causal 8192, 32 heads, 1462 us, so 1419; one head, causal 4096, 154 and 123).
// Without the barrier between the two halves the compiler mixes them again and takes 2 % longer.
template <int kOff, int kPitch, int kStatOff, int kStatBytes, int kCopies, class Copy>
__device__ __forceinline__ void dkdv_block(const PairAddr<16>& ad, uint32_t stat_base, const bf16x8 (&kf)[8], const bf16x8 (&vf)[8], f32x16 (&dk)[4],
                                           f32x16 (&dv)[4], float scale_log2, bool mask, Copy copy) {
  using M = Mma<16>;
  f32x4 s[2][2], dp[2][2], lse[2], delta[2];                      // [qb][n], [qb]
  uint32_t stat = stat_base + 16 * (fresh_lane() >> 4);           // this lane group's 4 consecutive row statistics
  keep_in_register(stat);                // (the reads' offsets then are constants: a lone workgroup 2 % faster)
  auto rd_stat = [&](int qb) {
    lse[qb] = *reinterpret_cast<const UA_LDS f32x4*>(stat + (kStatOff + 64 * qb));
    delta[qb] = *reinterpret_cast<const UA_LDS f32x4*>(stat + (kStatOff + kStatBytes / 2 + 64 * qb));
  };
  rd_stat(0);
  __builtin_amdgcn_sched_barrier(0);       // the reads below, mixed with what came before them, spill registers
  // 16 row fragments, Q and dO alternating, of the first and then of the second 16 rows, fetched kAhead reads ahead of their MFMAs
  constexpr int kAhead = 3;
  bf16x8 fr[16];
  auto rd = [&](int i) {
    const int part = 2 * (i >> 1 & 3) + (i >> 3);
    return (i & 1) ? pair_nat<kOff + kPitch>(ad, part) : pair_nat<kOff>(ad, part);
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fr[i] = rd(i);
  __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
  bf16x8 pb[2], dsb[2];
  // transposed fragments i: dO for i even (dV), Q for i odd (dK); columns 16 * (i / 2)
  auto rd_tr = [&](int i) { return (i & 1) ? pair_tr<kOff>(ad, i >> 1) : pair_tr<kOff + kPitch>(ad, i >> 1); };
  constexpr int kTAhead = 2;
  bf16x8 ft[16];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
#pragma unroll
    for (int i = 8 * qb; i < 8 * qb + 8; ++i) {
      if (i + kAhead < 16) fr[i + kAhead] = rd(i + kAhead);
      const int ks = i >> 1 & 3;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        if (i & 1) dp[qb][n] = M::mfma(fr[i], vf[2 * ks + n], ks == 0 ? delta[qb] : dp[qb][n]);
        else       s[qb][n] = M::mfma(fr[i], kf[2 * ks + n], ks == 0 ? lse[qb] : s[qb][n]);
      }
      M::interleave<1>();
      if ((i + 1) * kCopies / 16 != i * kCopies / 16) copy(i * kCopies / 16);
    }
    // element j of block (qb, n): query row 16*qb + 4*(lane/16) + j, key column 16*n + lane%16
    if (mask) {
      const int lane = fresh_lane(), key = lane & 15, row = 4 * (lane >> 4);          // (not one difference: see dq_block)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (row + 16 * qb + j - 16 * n < key) s[qb][n][j] = -INFINITY;
    }
    if (qb == 1) {
#pragma unroll
      for (int i = 0; i < kTAhead; ++i) ft[i] = rd_tr(i);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float pv = fast_exp2(s[qb][n][j] * scale_log2);
        pb[n][4 * qb + j] = (bf16)pv;
        dsb[n][4 * qb + j] = (bf16)(pv * dp[qb][n][j]);
      }
    if (qb == 0) rd_stat(1);
    if (qb == 0) __builtin_amdgcn_sched_barrier(0);
  }
  // (Diagonal tiles, whose blocks come without copies: the mask's branch parts the first fragments' reads from the products before it, and one
  // by one between the MFMAs they would all be waited for.  29 heads of causal 2432 x 128 14.6 -> 13.7 us, 17 of 5504 x 384 22.9 -> 21.7, one
  // of 4096 over its list 119.1 -> 118.0; three fragments ahead the same.)
  if (kCopies == 0) __builtin_amdgcn_sched_group_barrier(0x100, 2 * kTAhead, 0);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (i + kTAhead < 16) ft[i + kTAhead] = rd_tr(i + kTAhead);
    if (i & 1) M::second(dk, i >> 1, ft[i], dsb);
    else       M::second(dv, i >> 1, ft[i], pb);
    M::interleave<2>();
  }
}

// The same with 32x32x16.
template <int kOff, int kPitch, int kStatOff, int kStatBytes, int kCopies, class Copy>
__device__ __forceinline__ void dkdv_block(const PairAddr<32>& ad, uint32_t stat_base, const bf16x8 (&kf)[8], const bf16x8 (&vf)[8], f32x16 (&dk)[4],
                                           f32x16 (&dv)[4], float scale_log2, bool mask, Copy copy) {
  using M = Mma<32>;
  f32x16 s, dp;
  uint32_t stat = stat_base + 16 * (fresh_lane() >> 5);           // this lane half's 4 consecutive row statistics
  keep_in_register(stat);                // (the reads' offsets then are constants: a lone workgroup 2 % faster)
  // element i of a block: query row 8*(i/4) + 4*hi + i%4, key column lane%32
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 a = *reinterpret_cast<const UA_LDS f32x4*>(stat + (kStatOff + 32 * g));
    const f32x4 c = *reinterpret_cast<const UA_LDS f32x4*>(stat + (kStatOff + kStatBytes / 2 + 32 * g));
#pragma unroll
    for (int j = 0; j < 4; ++j) { s[4 * g + j] = a[j]; dp[4 * g + j] = c[j]; }
  }
  __builtin_amdgcn_sched_barrier(0);       // the reads below, mixed with what came before them, spill registers
  {
    // 16 row fragments, Q and dO alternating, fetched kAhead reads ahead of their MFMA
    constexpr int kAhead = 2;
    bf16x8 fr[16];
    auto rd = [&](int i) { return (i & 1) ? pair_nat<kOff + kPitch>(ad, i >> 1) : pair_nat<kOff>(ad, i >> 1); };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fr[i] = rd(i);
    __builtin_amdgcn_sched_group_barrier(0x100, 8 + kAhead, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i + kAhead < 16) fr[i + kAhead] = rd(i + kAhead);
      if (i & 1) dp = M::mfma(fr[i], vf[i >> 1], dp);
      else       s = M::mfma(fr[i], kf[i >> 1], s);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if ((i + 1) * kCopies / 16 != i * kCopies / 16) copy(i * kCopies / 16);
    }
  }
  // transposed fragments i: dO for i even (dV), Q for i odd (dK); d-block (i/2)%4, 16-row step i/8
  auto rd_tr = [&](int i) { return (i & 1) ? pair_tr<kOff>(ad, i >> 1) : pair_tr<kOff + kPitch>(ad, i >> 1); };
  constexpr int kTAhead = 2;
  bf16x8 fr[16];
#pragma unroll
  for (int i = 0; i < kTAhead; ++i) fr[i] = rd_tr(i);
  if (mask) {
    const int lane = fresh_lane(), key_b = lane & 31, hi4 = 4 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (key_b > 8 * (i >> 2) + hi4 + (i & 3)) s[i] = -INFINITY;
  }
  bf16x8 pb[2], dsb[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float pv = fast_exp2(s[i] * scale_log2);
    pb[i >> 3][i & 7] = (bf16)pv;
    dsb[i >> 3][i & 7] = (bf16)(pv * dp[i]);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (i + kTAhead < 16) fr[i + kTAhead] = rd_tr(i + kTAhead);
    if (i & 1) M::second(dk, i >> 1, fr[i], dsb);
    else       M::second(dv, i >> 1, fr[i], pb);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
  }
}

// kForm (here and for dQ; other than 1 for dense rectangles only): how the workgroup's waves share the line, see Groups.  Each group walks
// its share of every tile through stages of its own, and the results are added through LDS.  Where the launch gives a CU one workgroup of
// four waves at most, one wave per SIMD would leave the matrix pipe idle between its dependent steps (2.2 us
// per half tile of dK/dV, 0.9 of them MFMAs); the other groups fill the CU without partial results in memory.
template <int kForm, bool kDense>
__device__ __forceinline__ void dkdv_walk(const BwdParams& given, uint32_t lds_block, int block) {
  const BwdParams& p = params_of_walk<kForm, false>(given);
  using S = Stages<kForm>;
  const int tid = threadIdx.x % (64 * S::kWaves), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = S::kCount == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * S::kWaves));
  const uint32_t lds_base = lds_block + group * S::kBytes;
  int pos, bh;
  map_block<S::kLines == 2>(block, p.cols.map, pos, bh);
  const int sub = pos & (S::kLines - 1);         // which half of the tile's keys
  pos >>= S::kLines - 1;
  const int b = quotient(bh, p.by_heads), h = bh - b * p.n_heads;
  int kt, e0, e1, diag = -1, part = 0;
  if constexpr (kDense) {
    part = quotient(pos, p.cols.by_lines);
    kt = pos - part * p.n_ktiles;                          // column 0 is the longest of a causal rectangle
    if (p.cols_reversed) kt = p.n_ktiles - 1 - kt;
    if (p.dense_causal) diag = kt - p.diag_off;            // query tile on the diagonal (may lie outside)
    const int qbeg = p.dense_causal ? min(max(diag, 0), p.n_qtiles) : 0;
    e0 = min(max(part * p.cols.part_len, qbeg), p.n_qtiles);
    e1 = max(min((part + 1) * p.cols.part_len, p.n_qtiles), e0);
  } else {
    kt = min(max(sload(p.cols.order, p.cols_reversed ? p.n_ktiles - 1 - pos : pos), 0), p.n_ktiles - 1);
    e0 = min(max(sload(p.cols.ptr, kt), 0), p.nnz);
    e1 = min(max(sload(p.cols.ptr, kt + 1), e0), p.nnz);
  }
  const int64_t seq_q = (int64_t)p.n_qtiles * kTile;
  PairStream<kForm> in(p.q + b * p.qs.b + h * p.qs.h, (int)p.qs.s, p.dout + b * p.ds.b + h * p.ds.h, (int)p.ds.s, lds_base, wave, lane);
  // A step is one half of a tile, in order; with more groups half or quarter `group` of a tile.
  using W = Walk<kDense, false>;
  W walk(e0, e1, diag, lds_base + S::kEntries + wave * W::kBytes);
  auto fetch = [&](int e) { walk.fetch(e, p.cols.idx, p.cols.flag, p.n_qtiles); };
  // The rows' statistics of a step: its rows' -lse/softmax_scale (lse = -inf, a row without keys, stays -inf so that P = 0) and
  // -delta, which the accumulators of S and dP' start from.  Every wave brings 32 of them (lanes 32..63 do the same), the first half
  // of the waves lse, the others delta: which of the two, and where, are scalars.  They are loaded two steps before their use, turned and
  // put into LDS a step before it: by then everything loaded has arrived at the end of a step, and nothing waits.  (Half of every wave's lanes
  // bringing lse and half delta took 42 more vector instructions a half tile, and a lone workgroup 5 % more time: causal 4096, one head,
  // dK/dV 122.5 -> 116.0 us; causal 8 heads of 6144, backward 275 -> 263; strided 32k, 16 heads, dK/dV 1643 -> 1634.)
  const float scale_log2 = in_scalar(p.scale_log2);        // (else read from memory at every block)
  const bool of_delta = wave >= S::kWaves / 2;
  const float* const stat_rows = (of_delta ? p.delta : p.lse) + ((int64_t)b * p.n_heads + h) * seq_q + 32 * (wave & (S::kWaves / 2 - 1));
  const float factor = in_scalar(of_delta ? -1.f : p.neg_inv_scale), kept = in_scalar(of_delta ? __builtin_nanf("") : -INFINITY);
  auto load_stat = [&](int entry, int part) {
    const float* const rows = stat_rows + (int64_t)walk.tile(entry) * kTile + part * S::kRows;
    return rows[(uint32_t)(fresh_lane() & 31)];
  };
  auto put_stat = [&](int stage, float x) {
    lds_put(lds_base + S::kStat + stage * S::kStatBytes + 128 * wave + 4 * (fresh_lane() & 31), x == kept ? x : x * factor);
  };
  int ent = 0, ent_next = 0;
  float st0 = 0.f, stat = 0.f;
  auto part_of = [&](int stage) { return S::kSteps * group + (S::kSteps == 2 ? stage : 0); };      // half or quarter of the tile
  if (e0 < e1) {
    fetch(e0);
    ent = walk.at(e0);
    in.tile(walk.tile(ent), true);
#pragma unroll
    for (int n = 0; n < in.kCopies; ++n) in.template copy<0>(n, part_of(0));
    st0 = load_stat(ent, part_of(0));
    stat = S::kSteps == 2 ? load_stat(ent, part_of(1)) : load_stat(walk.at(min(e0 + 1, e1 - 1)), group);
  }

  // K and V rows as B operands
  // (through the stage that the first step fills)
  const int k_block = S::kWaves * sub + wave, krow0 = kt * kTile + k_block * 32;
  bf16x8 kf[8], vf[8];
  if constexpr (kForm == 1) {
    u32x4 kraw[8], vraw[8];
    load_rows(kraw, p.k + b * p.ks.b + (int64_t)krow0 * p.ks.s + h * p.ks.h, p.ks.s);
    load_rows(vraw, p.v + b * p.vs.b + (int64_t)krow0 * p.vs.s + h * p.vs.h, p.vs.s);
    const uint32_t turn = lds_base + 2 * S::kPitch + wave * kWaveRowsBytes;
    rows_to_frags<S::kM>(kf, kraw, turn);
    rows_to_frags<S::kM>(vf, vraw, turn);
  } else {
    const int64_t line0 = (int64_t)kt * kTile + sub * 32 * S::kWaves;
    const uint32_t k_lds = lds_block + 2 * S::kPitch, v_lds = k_lds + S::kBytes;           // stage 1 of groups 0 and 1
    copy_shared_rows<32 * S::kWaves, S::kThreads>(p.k + b * p.ks.b + line0 * p.ks.s + h * p.ks.h, (int)p.ks.s, k_lds);
    copy_shared_rows<32 * S::kWaves, S::kThreads>(p.v + b * p.vs.b + line0 * p.vs.s + h * p.vs.h, (int)p.vs.s, v_lds);
    wait_vmem_all();
    __syncthreads();
    shared_rows_to_frags<S::kM>(kf, k_lds, wave);
    shared_rows_to_frags<S::kM>(vf, v_lds, wave);
  }
  f32x16 dk[4], dv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { Mma<S::kM>::clear(dk[i]); Mma<S::kM>::clear(dv[i]); }

  PairAddr<S::kM> ad(lds_base, lane);
  if (e0 < e1) put_stat(0, st0);
  // The compiler does not see the copies that the walk has in flight.  Were the K and V rows still
  // outstanding for it there, it would wait for them by count inside the loop, i.e. for the copies: they are
  // made to arrive here.
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+v"(kf[ks]), "+v"(vf[ks]));
  wait_vmem_all();
  __syncthreads();

  // One step on stage kStage: the copies of the next step's rows go in flight into the other stage, which everyone has left at the
  // barrier that ended the last step, between the MFMAs: all of them at the step's start kept a wave from its first product for
  // 500 to 1100 of 3900 to 6900 cycles (64 bytes a cycle and CU is what the copies' path takes).
  auto step = [&](int e, auto stage_tag) {
    constexpr int kStage = decltype(stage_tag)::value;
    constexpr bool kFirst = S::kSteps == 2 && kStage == 0;        // the tile's second half follows
    if (S::kSteps == 1 && e >= e1) return;                        // workgroup-uniform
    if (S::kSteps == 1 || kFirst) {
      if (!walk.has(e + 1)) fetch(e + 1);
      ent_next = walk.at(min(e + 1, e1 - 1));
    }
    put_stat(kStage ^ 1, stat);
    stat = S::kSteps == 2 ? load_stat(ent_next, part_of(kStage)) : load_stat(walk.at(min(e + 2, e1 - 1)), group);
    in.next_step();
    if (!kFirst) in.tile(walk.tile(ent_next), e + 1 < e1);
    const bool causal = (ent >> 30) != 0;
    // causal tile: query block nb sees none of the wave's keys when nb < k_block, some when nb == k_block
    constexpr int kBlocks = S::kRows / 32, kCopies = in.kCopies / kBlocks, kOff = 2 * kStage * S::kPitch, kStatOff = kStage * S::kStatBytes;
    const int nb = kBlocks * part_of(kStage), part_next = part_of(kStage ^ 1);
    if (!causal) {
      auto block = [&](auto mb_tag) {
        constexpr int kMb = decltype(mb_tag)::value;
        dkdv_block<kOff + kMb * S::kBlockPitch, S::kPitch, kStatOff + kMb * 128, S::kStatBytes, kCopies>(
            ad, lds_base + S::kStat, kf, vf, dk, dv, scale_log2, false, [&](int n) { in.template copy<kStage ^ 1>(kMb * kCopies + n, part_next); });
      };
      block(std::integral_constant<int, 0>{});
      if constexpr (kBlocks == 2) block(std::integral_constant<int, 1>{});
    }
    // (Not the other side of one branch, where the products do not stay in the same registers: 400 to 700 are spilled.)
    int is_causal = __builtin_amdgcn_readfirstlane((int)causal);
    asm volatile("" : "+s"(is_causal));
    if (is_causal) {
      // Rare: one block after the other from the first that sees some of the wave's keys, after the copies.
#pragma unroll
      for (int n = 0; n < in.kCopies; ++n) in.template copy<kStage ^ 1>(n, part_next);
#pragma unroll 1
      for (int mb = max(k_block - nb, 0); mb < kBlocks; ++mb) {
        ad.shift(mb * S::kBlockPitch);
        dkdv_block<kOff, S::kPitch, kStatOff, S::kStatBytes, 0>(ad, lds_base + S::kStat + mb * 128, kf, vf, dk, dv, scale_log2, nb + mb == k_block,
                                                                [](int) {});
        ad.shift(-mb * S::kBlockPitch);
      }
    }
    if (!kFirst) ent = ent_next;
    wait_vmem_all();
    __syncthreads();     // the next stage has landed and everyone is done with this one
  };
  for (int e = e0; e < e1; e += S::kSteps == 2 ? 1 : 2) {
    step(e, std::integral_constant<int, 0>{});
    step(S::kSteps == 2 ? e : e + 1, std::integral_constant<int, 1>{});
  }
  // everyone is done with the stages
  auto area = [&](int g) { return lds_block + (wave * S::kCount + g) * kAccBytes; };       // of group g of this wave's rows
  if constexpr (S::kCount == 2) {
    // the second group finishes dV, the first dK
    if (group) put_acc(area(1), dk); else put_acc(area(0), dv);
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
      if (group) add_block(area(0), mb, dv[mb]); else add_block(area(1), mb, dk[mb]);
  }
  f32x16 dk_sum, dv_sum;             // four groups: each finishes a block of 32 columns of both
  if constexpr (kForm == 4) {
    constexpr float kOnes[4] = {1.f, 1.f, 1.f, 1.f};
    put_acc(area(group), dk, group);
    __syncthreads();
    sum_blocks(dk_sum, dk, group, area, kOnes);
    __syncthreads();
    put_acc(area(group), dv, group);
    __syncthreads();
    sum_blocks(dv_sum, dv, group, area, kOnes);
  }
  const ParamsLate pl = params_late();
  const int64_t seq_k = (int64_t)pl->n_ktiles * kTile;
  const int64_t krow_out = (int64_t)kt * kTile + k_block * 32;
  if constexpr (kForm == 4) {
    // (this wave alone reads the block of its own area that it turns through)
    const uint32_t turn = area(group) + 4096 * group;
    store_block(&pl->cols, pl->cols.out0, pl->cols.o0s.b, pl->cols.o0s.s, pl->cols.o0s.h, pl->n_heads, part, b, krow_out, h, seq_k, group, dk_sum, pl->scale, turn);
    store_block(&pl->cols, pl->cols.out1, pl->cols.o1s.b, pl->cols.o1s.s, pl->cols.o1s.h, pl->n_heads, part, b, krow_out, h, seq_k, group, dv_sum, 1.f, turn);
  } else {
    const uint32_t turn = kForm == 1 ? lds_base + wave * kWaveRowsBytes : area(group ^ 1);
    if (kForm == 1 || group == 0)
      store_result<S::kM>(&pl->cols, pl->cols.out0, pl->cols.o0s.b, pl->cols.o0s.s, pl->cols.o0s.h, pl->n_heads, part, b, krow_out, h, seq_k, dk, pl->scale, turn);
    if (kForm == 1 || group == 1)
      store_result<S::kM>(&pl->cols, pl->cols.out1, pl->cols.o1s.b, pl->cols.o1s.s, pl->cols.o1s.h, pl->n_heads, part, b, krow_out, h, seq_k, dv, 1.f, turn);
  }
}

// ---- dQ -----------------------------------------------------------------------------------------
// Four wavefronts, wave w owns query rows 32w..32w+31 and keeps their Q and dO rows as B operands; K and V are
// streamed like dK/dV's operands.  Per block of 32 keys: S^T = K Q^T and dP'^T = V dO^T - delta (16 row fragments),
// dS^T in the lanes, dQ^T += K^T dS^T (8 column fragments).  A lane holds one query column, or one of each 16, so -delta is one
// value for all of a column's accumulators: it is kept in registers that dP's first MFMAs take as their addend, which spares moves.
template <int kM, int kOff, int kPitch, int kCopies, class Copy, class Side>
__device__ __forceinline__ void dq_block(const PairAddr<kM>& ad, const bf16x8 (&qf)[8], const bf16x8 (&dof)[8], const typename Mma<kM>::Start& neg_delta,
                                         f32x16 (&dq)[4], float scale_log2, const float (&lse2)[2], bool mask, Copy copy, Side side) {
  using M = Mma<kM>;
  f32x16 s, dp;
  {
    // 16 row fragments, K and V alternating, fetched kAhead reads ahead of their MFMAs
    constexpr int kAhead = 4;
    bf16x8 fr[16];
    auto rd = [&](int i) { return (i & 1) ? pair_nat<kOff + kPitch>(ad, i >> 1) : pair_nat<kOff>(ad, i >> 1); };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fr[i] = rd(i);
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i + kAhead < 16) fr[i + kAhead] = rd(i + kAhead);
      if (i & 1) M::first(dp, i >> 1, fr[i], dof, neg_delta);
      else       M::first(s, i >> 1, fr[i], qf, M::start({0.f, 0.f}));
      M::template interleave<1>();
      if ((i + 1) * kCopies / 16 != i * kCopies / 16) copy(i * kCopies / 16);
    }
  }
  // the first K^T fragments of the dQ product are fetched now, behind the pointwise work
  constexpr int kTAhead = 3;
  bf16x8 tfr[8];
#pragma unroll
  for (int i = 0; i < kTAhead; ++i) tfr[i] = pair_tr<kOff>(ad, i);
  // element i: key quad_row + i % 4 of the block, query column col
  if (mask) {
    // (compared with the column, not its difference with 0: of 16 nested conditions the compiler keeps each in scalar registers)
    const int lane = fresh_lane(), row = M::quad_row(lane, 0), col = M::col(lane, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (row + M::quad_row(0, i >> 2) + (i & 3) - M::col(0, M::quad_n(i >> 2)) > col) s[i] = -INFINITY;
  }
  side();
  bf16x8 dsb[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float pv = fast_exp2(fmaf(s[i], scale_log2, -lse2[M::quad_n(i >> 2)]));
    dsb[M::slot_n(i)][M::slot_j(i)] = (bf16)(pv * dp[i]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i + kTAhead < 8) tfr[i + kTAhead] = pair_tr<kOff>(ad, i + kTAhead);
    M::second(dq, i, tfr[i], dsb);
    M::template interleave<2>();
  }
}

template <int kForm, bool kDense>
__device__ __forceinline__ void dq_walk(const BwdParams& given, uint32_t lds_block, int block) {
  const BwdParams& p = params_of_walk<kForm, true>(given);
  static_assert(kDense || kForm == 1, "lists run with one group");
  if (kForm == 1 && kDense && p.rows_ahead) __builtin_amdgcn_s_setprio(1);
  using S = Stages<kForm>;
  const int tid = threadIdx.x % (64 * S::kWaves), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = S::kCount == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * S::kWaves));
  const uint32_t lds_base = lds_block + group * S::kBytes;
  int pos, bh;
  map_block<S::kLines == 2>(block, p.rows.map, pos, bh);
  const int sub = pos & (S::kLines - 1);         // which half of the tile's queries
  pos >>= S::kLines - 1;
  const int b = quotient(bh, p.by_heads), h = bh - b * p.n_heads;
  const int64_t seq_q = (int64_t)p.n_qtiles * kTile;
  int qt, e0, e1, diag = -1, part = 0;
  if constexpr (kDense) {
    part = quotient(pos, p.rows.by_lines);
    const int line = pos - part * p.n_qtiles;
    qt = p.dense_causal ? p.n_qtiles - 1 - line : line;    // longest rows first
    if (p.dense_causal) diag = qt + p.diag_off;
    const int kend = p.dense_causal ? min(max(diag + 1, 0), p.n_ktiles) : p.n_ktiles;
    e0 = min(part * p.rows.part_len, kend);
    e1 = min(e0 + p.rows.part_len, kend);
  } else {
    qt = min(max(sload(p.rows.order, pos), 0), p.n_qtiles - 1);
    e0 = min(max(sload(p.rows.ptr, qt), 0), p.nnz);
    e1 = min(max(sload(p.rows.ptr, qt + 1), e0), p.nnz);
  }
  PairStream<kForm> in(p.k + b * p.ks.b + h * p.ks.h, (int)p.ks.s, p.v + b * p.vs.b + h * p.vs.h, (int)p.vs.s, lds_base, wave, lane);
  Walk<kDense, true> walk(e0, e1, diag);      // steps as in dK/dV's walk
  auto fetch = [&](int e) { walk.fetch(e, p.rows.idx, p.rows.flag, p.n_ktiles); };
  auto part_of = [&](int stage) { return S::kSteps * group + (S::kSteps == 2 ? stage : 0); };      // half or quarter of the tile
  int ent = 0, ent_next = 0;
  if (e0 < e1) {
    fetch(e0);
    ent = walk.at(e0);
    in.tile(walk.tile(ent), true);
#pragma unroll
    for (int n = 0; n < in.kCopies; ++n) in.template copy<0>(n, part_of(0));
  }

  const int q_block = S::kWaves * sub + wave, qrow0 = qt * kTile + q_block * 32;
  bf16x8 qf[8], dof[8];
  u32x4 qraw[8], doraw[8];
  const uint32_t q_lds = lds_block + 2 * S::kPitch, do_lds = q_lds + S::kBytes;            // stage 1 of groups 0 and 1
  if constexpr (kForm == 1) {
    load_rows(qraw, p.q + b * p.qs.b + (int64_t)qrow0 * p.qs.s + h * p.qs.h, p.qs.s);
    load_rows(doraw, p.dout + b * p.ds.b + (int64_t)qrow0 * p.ds.s + h * p.ds.h, p.ds.s);
  } else {
    const int64_t line0 = (int64_t)qt * kTile + sub * 32 * S::kWaves;
    copy_shared_rows<32 * S::kWaves, S::kThreads>(p.q + b * p.qs.b + line0 * p.qs.s + h * p.qs.h, (int)p.qs.s, q_lds);
    copy_shared_rows<32 * S::kWaves, S::kThreads>(p.dout + b * p.ds.b + line0 * p.ds.s + h * p.ds.h, (int)p.ds.s, do_lds);
  }
  using M = Mma<S::kM>;
  float lse_raw[2], neg_delta[2];          // of the lane's queries
#pragma unroll
  for (int n = 0; n < M::kCols; ++n) {
    const int64_t row = ((int64_t)b * p.n_heads + h) * seq_q + qrow0 + M::col(lane, n);
    lse_raw[n] = p.lse[row];
    neg_delta[n] = -p.delta[row];
  }
  if constexpr (kForm == 1) {
    const uint32_t turn = lds_base + 2 * S::kPitch + wave * kWaveRowsBytes;      // in the stage that the first step fills
    rows_to_frags<S::kM>(qf, qraw, turn);
    rows_to_frags<S::kM>(dof, doraw, turn);
  } else {
    wait_vmem_all();
    __syncthreads();
    shared_rows_to_frags<S::kM>(qf, q_lds, wave);
    shared_rows_to_frags<S::kM>(dof, do_lds, wave);
  }
  float lse2[2];
#pragma unroll
  for (int n = 0; n < M::kCols; ++n) lse2[n] = (lse_raw[n] == -INFINITY) ? INFINITY : lse_raw[n] * kLog2e;
  typename M::Start nd = M::start(neg_delta);
  M::keep(nd);         // registers, not one value moved into an accumulator again and again

  f32x16 dq[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) M::clear(dq[i]);
  const PairAddr<S::kM> ad(lds_base, lane);
  // the rows arrive before the walk (see dkdv_kernel)
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+v"(qf[ks]), "+v"(dof[ks]));

  auto step = [&](int e, auto stage_tag) {
    constexpr int kStage = decltype(stage_tag)::value;
    constexpr bool kFirst = S::kSteps == 2 && kStage == 0;        // the tile's second half follows
    if (S::kSteps == 1 && e >= e1) return;                        // workgroup-uniform
    auto look_ahead = [&]() {                                     // the next tile's entry
      if (S::kSteps == 2 && !kFirst) return;
      if (!walk.has(e + 1)) fetch(e + 1);
      ent_next = walk.at(min(e + 1, e1 - 1));
    };
    // (of a list beside the first block, which one group always sees; a group of several may see none of its blocks)
    if (kDense) look_ahead();
    in.next_step();
    if (!kFirst) in.tile(walk.tile(ent_next), e + 1 < e1);
    wait_vmem_all();
    __syncthreads();            // this stage has landed; everyone is done with the other one, which the copies now fill
    const bool causal = (ent >> 30) != 0;
    // causal tile: key block nb is hidden from the wave's queries when nb > q_block, in part when nb == q_block
    constexpr int kBlocks = S::kRows / 32, kCopies = in.kCopies / kBlocks, kOff = 2 * kStage * S::kPitch;
    const int nb = kBlocks * part_of(kStage), part_next = part_of(kStage ^ 1);
    auto block = [&](auto mb_tag) {
      constexpr int kMb = decltype(mb_tag)::value;
      if (!causal || q_block >= nb + kMb)
        dq_block<S::kM, kOff + kMb * S::kBlockPitch, S::kPitch, kCopies>(ad, qf, dof, nd, dq, p.scale_log2, lse2, causal && q_block == nb + kMb,
                                                               [&](int n) { in.template copy<kStage ^ 1>(kMb * kCopies + n, part_next); },
                                                               [&]() { if (!kDense && kFirst && kMb == 0) look_ahead(); });
    };
    if (causal) {                                  // rare: the copies of the blocks that are left out
      for (int mb = 0; mb < kBlocks; ++mb)
        if (q_block < nb + mb)
#pragma unroll
          for (int n = 0; n < kCopies; ++n) in.template copy<kStage ^ 1>(mb * kCopies + n, part_next);
    }
    block(std::integral_constant<int, 0>{});
    if constexpr (kBlocks == 2) block(std::integral_constant<int, 1>{});
    if (!kFirst) ent = ent_next;
  };
  for (int e = e0; e < e1; e += S::kSteps == 2 ? 1 : 2) {
    step(e, std::integral_constant<int, 0>{});
    step(S::kSteps == 2 ? e : e + 1, std::integral_constant<int, 1>{});
  }
  wait_vmem_all();              // the last step's copies filled with zeros a stage that is used for the results now
  __syncthreads();
  const ParamsLate pl = params_late();
  const int64_t qrow_out = (int64_t)qt * kTile + q_block * 32, seq_out = (int64_t)pl->n_qtiles * kTile;
  auto area = [&](int g) { return lds_block + (wave * S::kCount + g) * kAccBytes; };       // of group g of this wave's rows
  if constexpr (kForm == 4) {
    put_acc(area(group), dq, group);
    __syncthreads();
    constexpr float kOnes[4] = {1.f, 1.f, 1.f, 1.f};
    f32x16 sum;
    sum_blocks(sum, dq, group, area, kOnes);
    store_block(&pl->rows, pl->rows.out0, pl->rows.o0s.b, pl->rows.o0s.s, pl->rows.o0s.h, pl->n_heads, part, b, qrow_out, h, seq_out, group, sum,
                pl->scale, area(group) + 4096 * group);
  } else {
    uint32_t turn = lds_base + wave * kWaveRowsBytes;                // stage 0: everyone left it before the last step
    if constexpr (S::kCount == 2) {
      turn = area(1);
      if (group) put_acc(turn, dq);
      __syncthreads();
      if (group) return;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) add_block(turn, mb, dq[mb]);
    }
    store_result<S::kM>(&pl->rows, pl->rows.out0, pl->rows.o0s.b, pl->rows.o0s.s, pl->rows.o0s.h, pl->n_heads, part, b, qrow_out, h, seq_out, dq, pl->scale,
                 turn);
  }
}

// ---- kernels ------------------------------------------------------------------------------------
__global__ __launch_bounds__(Groups<1>::kThreads, 2) void dkdv_kernel(const BwdParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[Stages<1>::kBytes];
  dkdv_walk<1, false>(p, (uint32_t)(uintptr_t)(UA_LDS unsigned char*)smem, blockIdx.x);
}
__global__ __launch_bounds__(Groups<1>::kThreads, 2) void dq_kernel(const BwdParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[Stages<1>::kBytes];
  dq_walk<1, false>(p, (uint32_t)(uintptr_t)(UA_LDS unsigned char*)smem, blockIdx.x);
}
// Both sides in one launch.
template <int kForm, bool kDense>
__global__ __launch_bounds__(Groups<kForm>::kThreads, 2) void bwd_kernel(const BwdParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[Stages<kForm>::kCount * Stages<kForm>::kBytes];
  const uint32_t lds_base = (uint32_t)(uintptr_t)(UA_LDS unsigned char*)smem;
  touch_params();
  if ((int)blockIdx.x < p.n_col_blocks) dkdv_walk<kForm, kDense>(p, lds_base, blockIdx.x);
  else                                  dq_walk<kForm, kDense>(p, lds_base, blockIdx.x - p.n_col_blocks);
}

static int fill_common(BwdParams& p, const void* q, const void* k, const void* v, const void* dout,
                       const float* lse, const float* delta,
                       int batch, int n_heads, int n_qtiles,
                       int n_ktiles, int nnz, int head_dim, const int64_t* qs, const int64_t* ks,
                       const int64_t* vs, const int64_t* ds, float softmax_scale) {
  if (!q || !k || !v || !dout || !lse || !delta || !qs || !ks || !vs || !ds) return UA_ERR_NULL;
  if (batch <= 0 || n_heads <= 0 || n_qtiles <= 0 || n_ktiles <= 0 || nnz < 0) return UA_ERR_SHAPE;
  if ((int64_t)batch * n_heads * n_qtiles * UA_MAX_PARTS > INT32_MAX / 2 ||
      (int64_t)batch * n_heads * n_ktiles * UA_MAX_PARTS > INT32_MAX / 2) return UA_ERR_SHAPE;
  if (head_dim != kHeadDim || !(softmax_scale > 0.f)) return UA_ERR_UNSUPPORTED;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(dout)) return UA_ERR_ALIGN;
  if (!strides_ok(qs) || !strides_ok(ks) || !strides_ok(vs) || !strides_ok(ds)) return UA_ERR_ALIGN;
  for (const int64_t* st : {qs, ks, vs, ds})
    if (st[1] > (INT32_MAX >> 9)) return UA_ERR_SHAPE;
  p.q = (const bf16*)q; p.k = (const bf16*)k; p.v = (const bf16*)v; p.dout = (const bf16*)dout;
  p.lse = lse; p.delta = delta;
  p.batch = batch; p.n_heads = n_heads; p.n_qtiles = n_qtiles; p.n_ktiles = n_ktiles; p.nnz = nnz;
  p.qs = {qs[0], qs[1], qs[2]}; p.ks = {ks[0], ks[1], ks[2]};
  p.vs = {vs[0], vs[1], vs[2]}; p.ds = {ds[0], ds[1], ds[2]};
  p.scale = softmax_scale; p.scale_log2 = softmax_scale * kLog2e; p.neg_inv_scale = -1.f / softmax_scale;
  p.dense = 0; p.dense_causal = 0; p.diag_off = 0; p.n_col_blocks = 0; p.cols_reversed = 0; p.rows_ahead = 0;
  p.cols = BwdSide{}; p.rows = BwdSide{};
  p.cols.n_parts = p.rows.n_parts = 1;
  return UA_OK;
}

// List arrays and outputs of one side (out1 = NULL on the rows' side).
static int fill_side(BwdSide& s, int nnz, const int32_t* ptr, const int32_t* idx, const uint8_t* flag, const int32_t* order, void* out0,
                     const int64_t* o0s, void* out1, const int64_t* o1s, bool dense) {
  if (nnz > 0 && (!idx || !flag)) return UA_ERR_NULL;          // only an empty list may leave them out
  if (flag && !aligned4(flag)) return UA_ERR_ALIGN;            // (a rule of the interface: whole words, so that a reader may take four at once)
  if (!out0 || !o0s || (o1s && !out1) || (!dense && (!ptr || !order))) return UA_ERR_NULL;
  if (!aligned16(out0) || !strides_ok(o0s) || (o1s && (!aligned16(out1) || !strides_ok(o1s)))) return UA_ERR_ALIGN;
  s.ptr = ptr; s.idx = idx; s.flag = flag; s.order = order;
  s.out0 = (bf16*)out0; s.out1 = (bf16*)out1;
  s.o0s = {o0s[0], o0s[1], o0s[2]};
  if (o1s) s.o1s = {o1s[0], o1s[1], o1s[2]};
  return UA_OK;
}

static int launched() { return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH; }
static unsigned col_blocks(const BwdParams& p) { return (unsigned)(p.batch * p.n_heads * p.n_ktiles * p.cols.n_parts); }
// Where the workgroups of both sides are, for `lines` of them per tile.
static void place(BwdParams& p, int lines) {
  p.by_heads = make_div(p.n_heads);
  p.cols.map = block_map(p.batch * p.n_heads, p.n_ktiles * p.cols.n_parts * lines);
  p.rows.map = block_map(p.batch * p.n_heads, p.n_qtiles * p.rows.n_parts * lines);
  p.cols.by_lines = make_div(p.n_ktiles);
  p.rows.by_lines = make_div(p.n_qtiles);
}
static unsigned row_blocks(const BwdParams& p) { return (unsigned)(p.batch * p.n_heads * p.n_qtiles * p.rows.n_parts); }
// The form (see Groups) for n lines of 128 rows on both sides of a rectangle that is not causal together (parts counted):
//  - four groups while half lines leave a CU one workgroup at most (8 heads of 1024: 34 us with one group, 24 with four; one tile 8.7 and 7.5).
//  - half lines of two groups up to 256 lines: the columns' half lines, which take longer, share the CUs with the rows', and the two
//    workgroups of a CU are in different phases of their steps (32 heads of 512 23.1 us with one group, in halves 19.8; 42 of 384 21.0 and
//    18.9).  Beyond, whole lines of one group fill the device as well and copy half as much (44 heads of 384, 264 lines: 21.1, in halves
//    23.2; 22 of 768 34.3 and 35.7).
// A causal one's form is chosen with its cut, see bwd_plan.  Tile lists run with one group, as in the forward.
static int bwd_form(int64_t n) {
  if (2 * n <= kCus) return 4;
  return 2 * n > kCus && n <= kCus ? kHalves : 1;
}
static int launch_bwd(BwdParams& p, int form, hipStream_t st) {
  const unsigned n = col_blocks(p) + row_blocks(p);
  const int lines = form > 2 ? 2 : 1;
  p.n_col_blocks = (int)col_blocks(p) * lines;
  place(p, lines);
  // Up to two workgroups per CU the whole launch is resident at once, and the second 256 join the first in launch
  // order.  Both sides come longest first (lists roughly); the columns are then taken in reverse, so that the long ones
  // of one side share a CU with the short ones of the other (32 causal heads of 1024: 43.6 -> 41.5 us).
  p.cols_reversed = form == kHalves ? p.dense_causal : form == 1 && (p.dense_causal || !p.dense) && n > kCus && n <= 2 * kCus;
  // Of up to three workgroups per CU the third one starts when a row of the first 512 is through, and the launch ends with rows that began
  // second: the rows' wavefronts go first where a CU has a column's as well (16 heads of 2304: 158 us, without 143; 64 of 640: 56.1, 48.9; 9 x 27
  // tiles, 16 heads cut, 113.5, 111.9).  Not where the columns are the longer ones (32 heads of 1536 x 768: 67.6, 75.6), and
  // beyond 768 lines it goes either way (8 x 8 tiles, 896 lines 104.4 and 106.9, 1200 148.5 and 141.4, 1504 175.4 and 189.2).
  p.rows_ahead = form == 1 && p.dense && !p.dense_causal && n > 2 * kCus && n <= 3 * kCus && p.rows.part_len >= p.cols.part_len;
  switch (form) {
    case 4: hipLaunchKernelGGL((bwd_kernel<4, true>), dim3(2 * n), dim3(512), 0, st, p); break;
    case kHalves: hipLaunchKernelGGL((bwd_kernel<kHalves, true>), dim3(2 * n), dim3(Groups<kHalves>::kThreads), 0, st, p); break;
    default:
      // (both sides in one launch at every length: against a launch for each 1-2 % faster at 4096 lines, above that within
      // 1 % either way, strided mask of 128k, 65536 lines, 57.9 and 58.1 ms, of 64k, 32768 lines, 17.10 and 16.99)
      if (p.dense) hipLaunchKernelGGL((bwd_kernel<1, true>), dim3(n), dim3(256), 0, st, p);
      else         hipLaunchKernelGGL((bwd_kernel<1, false>), dim3(n), dim3(256), 0, st, p);
  }
  return launched();
}

// How many parts the two sides of a dense backward are cut into, at most what the workspace holds, and its form.  A cut gives a
// small rectangle enough workgroups for the device and costs the partials' way through memory and a second launch; which wins is decided
// by an estimate of the time in microseconds.
// The sum of the partials takes 2, 0.7 more for columns, 1.3 for columns and rows, the partials 1 per 4.3 MB and 0.3 at 8 MB, 1.2 from 16 on.
//
// Not causal: fitted to all cuts of 1427 rectangles of 1 to 130 heads and 256 to 24000 tokens, causal ones among them:
//  - a start and end (loading the resident rows, storing the results), longer as half lines fill the device, and the longest walks;
//  - with one group per workgroup a tile takes 3.6 (column) or 2.3 (row), 4.1 or 3.6 where two workgroups share the CU.  The second
//    workgroups of 257 to 512 lines are the last of the rows, beside a column;
//  - beyond 512 the last rows begin when something else is through: a row beside a column if those are few and shorter, else a row or
//    column, or a round of columns; sooner where the rows' wavefronts go first (see launch_bwd);
//  - no less than all tiles and workgroups take on a full device; a cut has to win by 3.5 %.
// (2 heads of 11136: 472 us cut in 2 and 1, 409 whole, 389 in 2 and 2; 1024 x 4096, one head: 34 us uncut, 20.7 cut in 1 and 3; 4 heads of
// 1024 19.9 cut in 2 and 1, 18.1 uncut.)
//
// Causal: lines differ in length and even out beyond one round of workgroups, less the more keys there are before the first query.  Every form is
// estimated with every cut up to 768 lines, fitted to 5300 rectangles of 1 to 64 heads and 128 to 24000 tokens; of those kept apart from
// the fit the plan taken is 1.5 % slower than the best one on average, 3 % of them by more than 10, 18 at most.  (One estimate for
// both kinds and bounds of lines for the forms: 5.4 % on average, and half lines or four groups, whose second round it did not see, up
// to 50 % slower than a cut where all lines are long: one head, 4992 x 19968, 222 us, cut 158; 5 of 1024 x 4096 57 and 44.)
//  - a start and end, and the longest walk, whose tiles take longer the fuller the device is;
//  - beyond one round all tiles and workgroups of a CU, and a share of the rows' mean length and of the longest beyond it at the end.
//
// Both were fitted when one group's walks ran on 32x32x16.  On 16x16x32 they take up to 8 % less on a full device and 1 to 2 % more with one wave a
// SIMD, which the estimates do not see.  Of 500 rectangles of up to 1100 lines, against that instruction: 1.1 % less time on average,
// six take 2 to 3 % more and one 5 (30 heads of causal 1664 x 128, a diagonal tile a walk, 11.2 -> 11.8 us).
struct BwdPlan { int cols, rows, form; };
struct BwdWalk { int parts, n, len; };                                     // parts asked for and made, tiles of each
struct BwdRates {
  int form, slots;                           // workgroups that the device holds
  float start, col, col_full, row, row_full, fullest, work, work_even, each, mean, mean_even, beyond;
};
static constexpr BwdRates kCausalRates[3] = {
  {1, 2 * kCus, 5.52f, 3.344f, 0.288f, 2.055f, 0.132f, 2.f, 2.193f, -0.485f, 1.578f, -0.401f, 1.035f, 0.722f},
  {kHalves, 2 * kCus, 5.46f, 1.785f, 0.187f, 1.128f, 0.077f, 2.f, 1.898f, -0.202f, 1.101f, -0.179f, 0.748f, 0.607f},
  {4, kCus, 6.62f, 1.385f, 0.067f, 0.758f, 0.237f, 1.5f, 1.282f, -0.088f, 2.65f, -0.018f, 0.539f, 0.205f},
};
static float bwd_causal_us(const BwdRates& f, float nbh, int n_qtiles, int n_ktiles, float tiles, const BwdWalk& c, const BwdWalk& r) {
  const float lines = nbh * (n_ktiles * c.n + n_qtiles * r.n), groups = (f.form == 1 ? 1 : 2) * lines, full = groups / kCus;
  const float even = n_ktiles > n_qtiles ? (float)(n_ktiles - n_qtiles) / n_ktiles : 0.f;
  const float col = f.col + f.col_full * fminf(full, f.fullest), row = f.row + f.row_full * fminf(full, f.fullest);
  const float walk = fmaxf(std::min(c.len, n_ktiles) * col, r.len * row);                  // (the longest column has n_ktiles queries at most)
  if (full <= 1.f) return f.start + walk;
  const float mean = tiles / (nbh * n_qtiles * r.n);
  const float work = (f.form == 1 ? 1 : 2) * tiles * (col + row) * (f.work + f.work_even * even) / f.slots + f.each * full +
                     ((f.mean + f.mean_even * even) * mean + f.beyond * (r.len - mean)) * row;
  const float longer = fmaxf(walk, work), ratio = fminf(walk, fmaxf(work, 0.f)) / longer, r2 = ratio * ratio, r4 = r2 * r2, r8 = r4 * r4;
  return f.start + longer * sqrtf(sqrtf(sqrtf(sqrtf(1.f + r8 * r8))));
}
static float bwd_us(int form, float nbh, int n_qtiles, int n_ktiles, const BwdWalk& c, const BwdWalk& r) {
  const float wk = nbh * n_ktiles, wq = nbh * n_qtiles, tiles = wk * n_qtiles, n_col_lines = wk * c.n, lines = n_col_lines + wq * r.n;
  const float col = c.len, row = r.len, kFull = 2 * kCus, least = (tiles * 9.31f + lines * 3.34f) / kFull;         // the work of a CU
  constexpr float kCol = 3.56f, kCol2 = 4.09f, kRow = 2.31f, kRow2 = 3.62f;
  if (form == 4) return 7.06f + 1.95f * (lines / 128) * (lines / 128) + fmaxf(fmaxf(col * 1.23f, row * 0.715f), least);
  if (form == kHalves) {
    const float shared = fminf((lines - 128) * (3.f / 128), 1.f);                    // lines > 128
    return 8.67f + fmaxf(col * (1.64f + 0.094f * shared), row * (1.18f + 0.355f * shared));
  }
  float walks;
  const float a = col * kCol2, b = row * kRow2;
  if (lines <= kFull) {
    walks = lines <= kCus ? fmaxf(col * kCol, row * kRow) : b > a ? a + (row - a / kRow2) * kRow : b + (col - b / kCol2) * kCol;
    if (n_col_lines > kCus) walks = fmaxf(walks, a);
  } else {
    const float over = lines - kFull, first_rows = kFull - n_col_lines;
    float from;                                                              // where the last rows begin
    if (first_rows <= 0)                  from = (0.6f * ceilf(over / kFull) + 0.4f * over / kFull) * (a + 12.2f);
    else if (over <= first_rows && b < a) from = 0.69f * b + 12.2f;
    else                                  from = over <= fmaxf(n_col_lines, first_rows) ? 0.8f * fminf(a, b) + 12.2f : fmaxf(a, b) + 12.2f;
    if (lines <= 3 * kCus && r.len >= c.len) from *= 0.48f;
    walks = fmaxf(fmaxf(a, b), from + b);
  }
  return 6.7f + fmaxf(walks, least);
}
static BwdPlan bwd_plan(int64_t nbh, int n_qtiles, int n_ktiles, bool causal, int max_cols, int max_rows) {
  static constexpr int kParts[] = {1, 2, 3, 4, 5, 6, 8, 12, 16};
  auto sides = [](BwdWalk (&s)[9], int most, int list_len) {
    int n = 0;
    for (int parts : kParts)
      if (parts <= most || parts == 1) {
        const int len = (list_len + parts - 1) / parts;
        s[n++] = {parts, (list_len + len - 1) / len, len};
      }
    return n;
  };
  BwdWalk cols[9], rows[9];
  const int n_cols = sides(cols, max_cols, n_qtiles), n_rows = sides(rows, max_rows, n_ktiles);
  const int n_forms = causal && nbh * (n_ktiles + n_qtiles) <= 3 * kCus ? 3 : 1;
  if (n_cols * n_rows * n_forms == 1) return {1, 1, causal ? 1 : bwd_form(nbh * ((int64_t)n_ktiles + n_qtiles))};
  const float wk = (float)nbh * n_ktiles, wq = (float)nbh * n_qtiles, tiles = visible_share(n_qtiles, n_ktiles, causal) * wk * n_qtiles;
  BwdPlan best = {1, 1, 1};
  float best_us = INFINITY;
  for (int i = 0; i < n_cols; ++i)
    for (int j = 0; j < n_rows; ++j) {
      const BwdWalk &c = cols[i], &r = rows[j];
      const float mb = ((c.n > 1 ? 2.f * c.n * wk : 0.f) + (r.n > 1 ? r.n * wq : 0.f)) * (kTile * kHeadDim * 4 / 1e6f), full = fminf(mb / 8, 2.f);
      const float sum = mb > 0.f ? 1.96f + (c.n > 1 ? 0.7f : 0.f) + (c.n > 1 && r.n > 1 ? 0.58f : 0.f) + mb / 4.34f + 0.31f * full * full : 0.f;
      for (int f = 0; f < n_forms; ++f) {
        const int form = causal ? kCausalRates[f].form : bwd_form(nbh * ((int64_t)n_ktiles * c.n + (int64_t)n_qtiles * r.n));
        float us = causal ? bwd_causal_us(kCausalRates[f], (float)nbh, n_qtiles, n_ktiles, tiles, c, r)
                          : bwd_us(form, (float)nbh, n_qtiles, n_ktiles, c, r) * (mb > 0.f ? 1.035f : 1.f);
        us += sum;
        if (us < 0.995f * best_us) { best_us = us; best = {c.parts, r.parts, form}; }      // more parts for a gain, not for a tie
      }
    }
  return best;
}
int64_t bwd_workspace_used(int batch, int n_heads, int n_qtiles, int n_ktiles, bool causal) {
  const DenseSplit d = dense_split(batch, n_heads, n_qtiles, n_ktiles);
  const BwdPlan n = bwd_plan((int64_t)batch * n_heads, n_qtiles, n_ktiles, causal, d.dkdv_parts, d.dq_parts);
  return (n.cols > 1 ? n.cols * d.dkdv_bytes : 0) + (n.rows > 1 ? n.rows * d.dq_bytes : 0);
}

}  // namespace ua

extern "C" int ua_bsa_bwd_dkdv(const void* q, const void* k, const void* v, const void* dout,
                               const float* lse, const float* delta, void* dk, void* dv,
                               const int32_t* col_ptr, const int32_t* row_idx, const uint8_t* cflag,
                               const int32_t* k_order,
                               int batch, int n_heads, int n_qtiles, int n_ktiles, int nnz, int head_dim,
                               const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                               const int64_t* do_strides, const int64_t* dk_strides, const int64_t* dv_strides,
                               float softmax_scale, void* stream) {
  using namespace ua;
  BwdParams p;
  if (int rc = fill_common(p, q, k, v, dout, lse, delta, batch, n_heads, n_qtiles, n_ktiles, nnz, head_dim, q_strides, k_strides,
                           v_strides, do_strides, softmax_scale)) return rc;
  if (!dv_strides) return UA_ERR_NULL;
  if (int rc = fill_side(p.cols, nnz, col_ptr, row_idx, cflag, k_order, dk, dk_strides, dv, dv_strides, false)) return rc;
  if (int rc = check_device()) return rc;
  place(p, 1);
  hipLaunchKernelGGL(dkdv_kernel, dim3(col_blocks(p)), dim3(256), 0, (hipStream_t)stream, p);
  return launched();
}

extern "C" int ua_bsa_bwd_dq(const void* q, const void* k, const void* v, const void* dout,
                             const float* lse, const float* delta, void* dq,
                             const int32_t* row_ptr, const int32_t* col_idx, const uint8_t* flag,
                             const int32_t* q_order,
                             int batch, int n_heads, int n_qtiles, int n_ktiles, int nnz, int head_dim,
                             const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                             const int64_t* do_strides, const int64_t* dq_strides,
                             float softmax_scale, void* stream) {
  using namespace ua;
  BwdParams p;
  if (int rc = fill_common(p, q, k, v, dout, lse, delta, batch, n_heads, n_qtiles, n_ktiles, nnz, head_dim, q_strides, k_strides,
                           v_strides, do_strides, softmax_scale)) return rc;
  if (int rc = fill_side(p.rows, nnz, row_ptr, col_idx, flag, q_order, dq, dq_strides, nullptr, nullptr, false)) return rc;
  if (int rc = check_device()) return rc;
  place(p, 1);
  hipLaunchKernelGGL(dq_kernel, dim3(row_blocks(p)), dim3(256), 0, (hipStream_t)stream, p);
  return launched();
}

extern "C" int ua_bsa_bwd(const void* q, const void* k, const void* v, const void* dout,
                          const float* lse, const float* delta, void* dq, void* dk, void* dv,
                          const int32_t* row_ptr, const int32_t* col_idx, const uint8_t* flag, const int32_t* q_order,
                          const int32_t* col_ptr, const int32_t* row_idx, const uint8_t* cflag, const int32_t* k_order,
                          int batch, int n_heads, int n_qtiles, int n_ktiles, int nnz, int head_dim,
                          const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                          const int64_t* do_strides, const int64_t* dq_strides, const int64_t* dk_strides,
                          const int64_t* dv_strides, float softmax_scale, void* stream) {
  using namespace ua;
  BwdParams p;
  if (int rc = fill_common(p, q, k, v, dout, lse, delta, batch, n_heads, n_qtiles, n_ktiles, nnz, head_dim, q_strides, k_strides,
                           v_strides, do_strides, softmax_scale)) return rc;
  if (!dv_strides) return UA_ERR_NULL;
  if (int rc = fill_side(p.cols, nnz, col_ptr, row_idx, cflag, k_order, dk, dk_strides, dv, dv_strides, false)) return rc;
  if (int rc = fill_side(p.rows, nnz, row_ptr, col_idx, flag, q_order, dq, dq_strides, nullptr, nullptr, false)) return rc;
  if (int rc = check_device()) return rc;
  return launch_bwd(p, 1, (hipStream_t)stream);
}

extern "C" int ua_dense_bwd(const void* dout, const void* q, const void* k, const void* v,
                            const float* lse, const float* delta, void* dq, void* dk, void* dv,
                            int batch, int n_heads, int seqlen_q, int seqlen_k, int head_dim,
                            const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                            const int64_t* do_strides, const int64_t* dq_strides, const int64_t* dk_strides,
                            const int64_t* dv_strides, float softmax_scale, int causal,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace ua;
  if (seqlen_q <= 0 || seqlen_k <= 0 || seqlen_q % kTile || seqlen_k % kTile) return UA_ERR_SHAPE;
  const int n_qtiles = seqlen_q / kTile, n_ktiles = seqlen_k / kTile;
  if (!dv_strides) return UA_ERR_NULL;
  BwdParams p;
  if (int rc = fill_common(p, q, k, v, dout, lse, delta, batch, n_heads, n_qtiles, n_ktiles, 0, head_dim, q_strides, k_strides,
                           v_strides, do_strides, softmax_scale)) return rc;
  if (int rc = fill_side(p.cols, 0, nullptr, nullptr, nullptr, nullptr, dk, dk_strides, dv, dv_strides, true)) return rc;
  if (int rc = fill_side(p.rows, 0, nullptr, nullptr, nullptr, nullptr, dq, dq_strides, nullptr, nullptr, true)) return rc;
  if (int rc = check_device()) return rc;
  hipStream_t st = (hipStream_t)stream;
  p.dense = 1; p.dense_causal = causal != 0; p.diag_off = n_ktiles - n_qtiles;
  p.cols.part_len = n_qtiles; p.rows.part_len = n_ktiles;
  const DenseSplit d = dense_split(batch, n_heads, n_qtiles, n_ktiles);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  // Cut one side: parts of equal length, fp32 partials in the workspace.
  auto cut = [&](BwdSide& s, int parts, int list_len, int64_t part_bytes) {
    s.part_len = (list_len + parts - 1) / parts;
    s.n_parts = (list_len + s.part_len - 1) / s.part_len;
    s.out_f32 = 1;
    s.o_part = part_bytes / 4;
    s.out0 = reinterpret_cast<bf16*>(ws);
    s.out1 = reinterpret_cast<bf16*>(ws + part_bytes / 2);       // columns: dV behind dK
    ws += parts * part_bytes;
  };
  // (without a workspace lines are walked whole by one group; one that is too small or misaligned only keeps them from being cut)
  BwdPlan n = {1, 1, 1};
  if (workspace) {
    auto plan = [&](int max_cols, int max_rows) { return bwd_plan((int64_t)batch * n_heads, n_qtiles, n_ktiles, p.dense_causal, max_cols, max_rows); };
    n = plan(d.dkdv_parts, d.dq_parts);
    const int64_t need = (n.cols > 1 ? n.cols * d.dkdv_bytes : 0) + (n.rows > 1 ? n.rows * d.dq_bytes : 0);
    if (need > 0 && (workspace_bytes < need || !aligned16(workspace))) n = plan(1, 1);
  }
  if (n.cols > 1) cut(p.cols, n.cols, n_qtiles, d.dkdv_bytes);
  if (n.rows > 1) cut(p.rows, n.rows, n_ktiles, d.dq_bytes);
  if (int rc = launch_bwd(p, n.form, st)) return rc;
  PartialSum sums[3];
  int n_sums = 0;
  auto add_sum = [&](const BwdSide& s, const bf16* first, void* out, const int64_t* os, int seqlen) {
    sums[n_sums++] = {reinterpret_cast<const float*>(first), (bf16*)out, s.o_part, s.n_parts, seqlen, {os[0], os[1], os[2]}};
  };
  if (p.cols.out_f32) {
    add_sum(p.cols, p.cols.out0, dk, dk_strides, seqlen_k);
    add_sum(p.cols, p.cols.out1, dv, dv_strides, seqlen_k);
  }
  if (p.rows.out_f32) add_sum(p.rows, p.rows.out0, dq, dq_strides, seqlen_q);
  return n_sums ? launch_partial_sums(sums, n_sums, batch, n_heads, st) : UA_OK;
}
