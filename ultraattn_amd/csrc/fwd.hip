// Block-sparse flash-attention forward for gfx950 (MI355X).
//
// One workgroup (4 wavefronts) per (query tile of 128 rows, head).  It walks the query tile's
// CSR entries; each 128x128 K/V tile is streamed as two 64-key half tiles through two LDS
// stages (A, B) that are filled by asynchronous global->LDS copies while the other stage is
// being consumed.  Each wavefront owns 32 query rows and computes the TRANSPOSED products
//     S^T[key, q] = K Q^T      (A = K fragment from LDS, B = Q fragment held in registers)
//     O^T[d,  q] += V^T P^T    (A = V^T fragment via transposing LDS reads, B = P^T)
// In the accumulator layout (see Mma) a lane holds one query column, or one of each block of 16, so the online-softmax
// statistics of a query row live in one lane and its mirrors: the row max needs an exchange over those alone, the rescale of
// O^T is lane local, and S^T's accumulator registers are, after exp2 and bf16 packing, exactly the B operand of the second
// product.
#include <algorithm>
#include <type_traits>
#include "ua_common.h"

namespace ua {

struct FwdParams {
  const bf16* q; const bf16* k; const bf16* v; bf16* o; float* lse;
  const int32_t* row_ptr; const int32_t* col_idx; const uint8_t* flag; const int32_t* q_order;
  int batch, n_heads, n_qtiles, n_ktiles, nnz;
  int n_first;           // positions of the launch order that are taken in reverse (see fwd_launch)
  Strides3 qs, ks, vs, os;
  float scale_log2;      // softmax_scale * log2(e)
  BlockMap map;
  Div by_heads, by_cut;  // n_heads; query tiles that are cut (1 if none)
  // Dense rectangle (no list arrays): query tile qt walks key tiles [0, n_ktiles), or with
  // dense_causal [0, qt + diag_off] with the last one causal; longest rows first.  The first n_whole query tiles (all
  // if nothing is cut) are walked whole; the key range of the others is cut into n_parts parts of part_len tiles, and
  // part i leaves its partial (O, LSE), contiguous over those n_qtiles - n_whole tiles, at part_o + i * o_part and
  // part_lse + i * lse_part (elements).  The partial O is fp32 (part_f32) beside whole tiles, so that every row of a result is
  // rounded to bf16 once; where everything is cut it is bf16 or fp32, see fwd_cut.
  int dense, dense_causal, diag_off, n_whole, n_parts, part_len, part_f32;
  void* part_o; float* part_lse;
  int64_t o_part, lse_part;
};

// The kernel's parameters read again from the kernel-argument segment.
typedef const __attribute__((address_space(4))) FwdParams* ParamsLate;
__device__ __forceinline__ ParamsLate params_late() {
  ParamsLate p = (ParamsLate)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// P is computed against the row's current reference max without looking at the new scores'
// max; only when a block's row sum shows that some score exceeded the reference by more than
// ~2^kRaiseLog2 is the reference raised (and O, l rescaled, P recomputed).  O/l stay exact
// because numerator and denominator always share the reference.
constexpr float kRaiseSum = 16777216.f;     // 2^24

struct SoftmaxState {
  float m_run = -INFINITY;   // reference max of the row (log2 domain, scaled)
  float m_use = 0.f;         // m_run, or 0 while the row has not seen a visible key
  float l_run = 0.f;         // this lane's partial row sum
};

// kB blocks of 32 keys for this wave's 32 query rows.  With `mask` (wave-uniform) keys beyond
// the query's own tile-local index are hidden; `key0` = tile-local index of the first key.
// kCopies: `copy(n)`, n = 0 .. 7, is called between the MFMAs of S; `side()` beside the softmax.
template <int kM, int kB, bool kCopies, class Copy, class Side>
__device__ __forceinline__ void key_blocks(const unsigned char* sK, const unsigned char* sV, const bf16x8 (&qf)[8],
                                          f32x16 (&oacc)[4], SoftmaxState (&st)[2], const int (&nat)[Mma<kM>::kRowRegs], const int (&tr)[4], float scale_log2,
                                          int q_block, int key0, bool mask, bool first, Copy copy, Side side) {
  using M = Mma<kM>;
  // ---- S^T = K Q^T : kB blocks of 32 keys x 32 queries -----------------------------------
  // The 8 * kB K fragments are fetched kAhead reads ahead of the MFMAs that consume them, so the
  // LDS latency is covered by the preceding MFMAs instead of being paid before each pair.
  f32x16 s[kB];
  {
    constexpr int kAhead = kM == 16 ? 3 : 4;
    constexpr int kParts = kM == 16 ? 2 : 1;                  // fragments of a block's rows, taken in turn with those of the other blocks
    bf16x8 kfr[8 * kB];
    auto frag = [](int i) { return i / (kParts * kB) * kParts + i % kParts; };
    auto block = [](int i) { return i / kParts % kB; };
    auto rd = [&](int i) {
      return lds_read_b128(sK, nat[M::a_reg(frag(i))] + M::a_offset(frag(i), 4 * kRowBytes) + 32 * kRowBytes * block(i));
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) kfr[i] = rd(i);
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);   // kAhead LDS reads up front
#pragma unroll
    for (int i = 0; i < 8 * kB; ++i) {
      if (i + kAhead < 8 * kB) kfr[i + kAhead] = rd(i + kAhead);
      M::first(s[block(i)], frag(i), kfr[i], qf, M::start({0.f, 0.f}));
      M::template interleave<1>();                              // then the fragment's MFMAs and 1 LDS read, ...
      if (kCopies && (i + 1) % kB == 0) copy(i / kB);
    }
  }
  // element (mb, i) of this lane: key key0 + 32 * mb + quad_row + i % 4, query 32 * q_block + col of the tile
  if (mask) {
    // (compared with the column, not their difference with 0: of 32 nested conditions the compiler keeps each in scalar registers)
    const int lane = fresh_lane(), key = key0 + M::quad_row(lane, 0), query = 32 * q_block + M::col(lane, 0);
#pragma unroll
    for (int mb = 0; mb < kB; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (key + 32 * mb + M::quad_row(0, i >> 2) + (i & 3) - M::col(0, M::quad_n(i >> 2)) > query) s[mb][i] = -INFINITY;
  }
  // the first V^T fragments are fetched now: their latency hides behind the softmax
  constexpr int kVAhead = 3;
  bf16x8 vfr[4];
  auto rd_v = [&](int i) {               // fragment i % 8 of 32 keys
    const int at = tr[M::tr_reg(i & 7)] + M::tr_first(i & 7, M::kPitchV) + 8 * M::kPitchV * (i >> 3);
    const bf16x4 lo = lds_read_tr16_b64(sV, at), hi = lds_read_tr16_b64(sV, at + M::tr_second(M::kPitchV));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
#pragma unroll
  for (int i = 0; i < kVAhead; ++i) vfr[i] = rd_v(i);
  side();
  // ---- online softmax (fp32, log2 domain) ---------------------------------------------------
  float rs[2] = {0.f, 0.f};
  bf16x8 pf[kB][2];
  auto exponentials = [&]() {
    rs[0] = rs[1] = 0.f;
#pragma unroll
    for (int mb = 0; mb < kB; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int n = M::quad_n(i >> 2);
        const float pv = fast_exp2(fmaf(s[mb][i], scale_log2, -st[n].m_use));
        rs[n] += pv;
        pf[mb][M::slot_n(i)][M::slot_j(i)] = (bf16)pv;
      }
  };
  bool raise = first;
  if (!first) {
    exponentials();
    raise = __builtin_amdgcn_ballot_w64(!(rs[0] < kRaiseSum) || (M::kCols == 2 && !(rs[1] < kRaiseSum))) != 0;       // wave-uniform, rare
  }
  if (raise) {
#pragma unroll
    for (int n = 0; n < M::kCols; ++n) {
      SoftmaxState& t = st[n];
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int mb = 0; mb < kB; ++mb)
          if (M::quad_n(i >> 2) == n) mx = fmaxf(mx, s[mb][i]);
      mx = M::column_max(mx) * scale_log2;
      // (Of lists only the rows that need it: a row's result must not depend on the rows that share its wave, of which there are 16 or 32.
      // Dense forwards raise all 32 rows at once and keep the bits that they have always had.)
      const bool needed = kM == 32 || first || M::column_max(rs[n] < kRaiseSum ? 0.f : 1.f) > 0.f;
      const float m_new = needed ? fmaxf(t.m_run, mx) : t.m_run;
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = (m_new == t.m_run) ? 1.f : fast_exp2(t.m_run - m_use);      // m_run = -inf -> 0
      t.m_run = m_new;
      t.m_use = m_use;
      t.l_run *= alpha;
#pragma unroll
      for (int mbd = 0; mbd < 4; ++mbd)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (M::quad_n(i >> 2) == n) oacc[mbd][i] *= alpha;
    }
    exponentials();
  }
#pragma unroll
  for (int n = 0; n < M::kCols; ++n) st[n].l_run += rs[n];
  // ---- O^T += V^T P^T : 128 d x 32 queries, kB steps of 32 keys --------------------------------
#pragma unroll
  for (int i = 0; i < 8 * kB; ++i) {
    if (i + kVAhead < 8 * kB) vfr[(i + kVAhead) & 3] = rd_v(i + kVAhead);
    M::second(oacc, i & 7, vfr[i & 3], pf[i >> 3]);
    M::template interleave<2>();                              // MFMAs and 2 LDS reads of one fragment
  }
}

// kForm (1, 2 or 4; other than 1 for dense rectangles only): how the workgroup's waves share the query tile, see Groups; the groups' results
// are combined through LDS.  A launch that gives a CU one workgroup of four waves at most runs it at
// one wave per SIMD, where a half tile takes 1.2 us of which the matrix pipe is busy 0.4; with more groups the CU is
// as full as with two workgroups, without partial results in memory.
template <int kForm, bool kDense, int kM>
__device__ __forceinline__ void fwd_lines(const FwdParams& p) {
  using M = Mma<kM>;
  static_assert(kForm == 1 || kM == 32, "the groups' exchange takes a lane to hold one row");
  constexpr int kWaves = Groups<kForm>::kWaves, kRows = Groups<kForm>::kRows, kLines = Groups<kForm>::kLines;
  constexpr int kStageBytes = kRows * kRowBytes, kStageV = kRows / 4 * M::kPitchV;
  // two pipeline stages per group, distinct arrays so that reads of one stage need not wait for the
  // copies in flight into the other
  __shared__ __attribute__((aligned(1024))) unsigned char sKA[kForm * kStageBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char sVA[kForm * kStageV];
  __shared__ __attribute__((aligned(1024))) unsigned char sKB[kForm * kStageBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char sVB[kForm * kStageV];
  // With four groups the query rows have room of their own: the first step's copies need not wait for everyone's reads of them
  // (with the step's barrier at its end: two causal tiles 6.4 -> 6.25 us, 8 heads of 1024 12.75 -> 12.5).
  constexpr bool kOwnQ = kForm == 4;
  __shared__ __attribute__((aligned(1024))) unsigned char sQ[kOwnQ ? 32 * kWaves * kRowBytes : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_in_block = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (group a constant for one group: the stages' addresses then are constants too, ten additions fewer per tile)
  const int wave = kForm == 1 ? wave_in_block : wave_in_block % kWaves, group = kForm == 1 ? 0 : wave_in_block / kWaves;
  unsigned char *const kA = sKA + group * kStageBytes, *const vA = sVA + group * kStageV;
  unsigned char *const kB = sKB + group * kStageBytes, *const vB = sVB + group * kStageV;
  int pos, bh;
  map_block(blockIdx.x, p.map, pos, bh);
  const int sub = pos & (kLines - 1);      // which half of the tile's rows
  pos >>= kLines - 1;
  if (pos < p.n_first) pos = p.n_first - 1 - pos;
  const int b = quotient(bh, p.by_heads), h = bh - b * p.n_heads;
  int qt, e0, e1, diag = -1, part = -1;
  if constexpr (kDense) {
    int line = pos;
    if (pos >= p.n_whole) {
      part = quotient(pos - p.n_whole, p.by_cut);
      line = pos - part * p.by_cut.d;
    }
    qt = p.dense_causal ? p.n_qtiles - 1 - line : line;
    if (p.dense_causal) diag = qt + p.diag_off;          // key tile on the diagonal (may lie outside the rectangle)
    const int kend = p.dense_causal ? min(max(diag + 1, 0), p.n_ktiles) : p.n_ktiles;
    e0 = part < 0 ? 0 : min(part * p.part_len, kend);
    e1 = part < 0 ? kend : min(e0 + p.part_len, kend);
  } else {
    qt = min(max(sload(p.q_order, pos), 0), p.n_qtiles - 1);
    // list bounds are clamped to the arrays' extent: an inconsistent row_ptr cannot read beyond them
    e0 = min(max(sload(p.row_ptr, qt), 0), p.nnz);
    e1 = min(max(sload(p.row_ptr, qt + 1), e0), p.nnz);
  }
  const bf16* kbase = p.k + b * p.ks.b + h * p.ks.h;
  const bf16* vbase = p.v + b * p.vs.b + h * p.vs.h;
  const int k_stride = (int)p.ks.s, v_stride = (int)p.vs.s;
  int koff[4], voff[4];
  dma_voffsets<slot_k, kWaves>(koff, k_stride, wave, lane);
  dma_voffsets<slot_v, kWaves>(voff, v_stride, wave, lane);
  const int k_half = kRows * k_stride * 2, v_half = kRows * v_stride * 2;                 // bytes of one stage in memory
  const uint32_t k_extent = (uint32_t)((kTile - 1) * k_stride + kHeadDim) * 2;            // bytes of one tile
  const uint32_t v_extent = (uint32_t)((kTile - 1) * v_stride + kHeadDim) * 2;
  auto lds_at = [](unsigned char* x) { return (uint32_t)(uintptr_t)(lds_byte*)x; };
  // One group copies the next stage between the MFMAs of S (pieces 0..7 in turn; at the step's start, 8 at once held a wave's first
  // product up), several groups all of it at the start: of 64 copies per CU and step, late ones are what the next step waits for
  // (2 x 5 heads, causal 1408 x 2688: 27.9 us, between the MFMAs 28.4 to 30.1).
  u32x4 k_rsrc, v_rsrc;                    // the tile that copies read; without `more` they fill with zeros a stage that no step reads
  auto tile = [&](int t, bool more) {
    k_rsrc = make_rsrc_words(kbase + (int64_t)t * kTile * k_stride, more ? k_extent : 0);
    v_rsrc = make_rsrc_words(vbase + (int64_t)t * kTile * v_stride, more ? v_extent : 0);
  };
  // Where the wave's copies land in a stage; made opaque in every step, as the sums with the stages' addresses would occupy scalar
  // registers all along (and 15 to 24 of those vector lanes).
  int k_wave = wave * 1024, v_wave = wave * M::kPitchV;
  auto copy_piece = [&](int n, unsigned char* k_stage, unsigned char* v_stage, int part) {
    const int j = n >> 1;                  // (the offsets of pieces 16 rows apart differ by that alone: one register each for K and V)
    if (n & 1) dma16_abs(v_rsrc, lds_at(v_stage) + 4 * M::kPitchV * j + v_wave, voff[0], part * v_half + j * 32 * v_stride);
    else       dma16_abs(k_rsrc, lds_at(k_stage) + 4096 * j + k_wave, koff[0], part * k_half + j * 32 * k_stride);
  };
  auto copy_stage = [&](int t, unsigned char* k_stage, unsigned char* v_stage, int part) {
    dma_rows_buf<kWaves, 1024>(k_stage, make_rsrc(kbase + (int64_t)t * kTile * k_stride, k_extent), koff, part * k_half, wave);
    dma_rows_buf<kWaves, M::kPitchV>(v_stage, make_rsrc(vbase + (int64_t)t * kTile * v_stride, v_extent), voff, part * v_half, wave);
  };

  // A step is one half of a tile, in order; with more groups half or quarter `group` of a tile.
  Walk<kDense, true> walk(e0, e1, diag);
  auto fetch = [&](int e) { walk.fetch(e, p.col_idx, p.flag, p.n_ktiles); };
  // the first stage goes in flight before anything else
  int ent = 0, ent_next = 0;
  if (e0 < e1) {
    fetch(e0);
    ent = walk.at(e0);
    if constexpr (kForm == 1) {
      tile(walk.tile(ent), true);
#pragma unroll
      for (int n = 0; n < 8; ++n) copy_piece(n, kA, vA, 0);
    } else {
      copy_stage(walk.tile(ent), kA, vA, group);
    }
  }

  // Q fragments (B operands of S^T)
  // (through the stage that the first step fills)
  const int q_block = kWaves * sub + wave;
  const int qrow0 = qt * kTile + q_block * 32;
  bf16x8 qf[8];
  if constexpr (kForm == 1) {
    u32x4 raw[8];
    load_rows(raw, p.q + b * p.qs.b + (int64_t)qrow0 * p.qs.s + h * p.qs.h, p.qs.s);
    rows_to_frags<kM>(qf, raw, (uint32_t)(uintptr_t)(lds_byte*)((wave < 2 ? kB : vB) + (wave & 1) * kWaveRowsBytes));
  } else {
    const uint32_t q_lds = lds_at(kOwnQ ? sQ : sKB);
    copy_shared_rows<32 * kWaves>(p.q + b * p.qs.b + ((int64_t)qt * kTile + sub * 32 * kWaves) * p.qs.s + h * p.qs.h, (int)p.qs.s, q_lds);
    wait_vmem_all();
    __syncthreads();
    shared_rows_to_frags<kM>(qf, q_lds, wave);
    if (!kOwnQ) __syncthreads();
  }
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+v"(qf[ks]));      // read before the walk

  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) M::clear(oacc[i]);
  SoftmaxState st[2];                      // of the lane's queries
  int nat[M::kRowRegs], tr[4];             // row reads of K, transposing reads of V
#pragma unroll
  for (int i = 0; i < M::kRowRegs; ++i) nat[i] = lds_off_k(M::a_row(lane), M::a_chunk(lane, i));
#pragma unroll
  for (int i = 0; i < 4; ++i) tr[i] = M::tr_offset(lane, i, M::kPitchV);

  bool started = false;
  auto step = [&](int e, auto stage_tag) {
    constexpr int kStage = decltype(stage_tag)::value, kBlocks = kRows / 32;
    constexpr bool kFirst = kForm == 1 && kStage == 0;          // the tile's second half follows
    if (kForm > 1 && e >= e1) return;                           // workgroup-uniform
    auto look_ahead = [&]() {                                     // the next tile's entry
      if (kForm == 1 && !kFirst) return;
      if (!walk.has(e + 1)) fetch(e + 1);
      ent_next = walk.at(min(e + 1, e1 - 1));
    };
    if (kForm > 1) look_ahead();
    if (kForm == 1 && !kFirst) tile(walk.tile(ent_next), e + 1 < e1);
    auto landed = [&]() {        // the next stage has landed; everyone is done with this one
      wait_vmem_all();
      __syncthreads();
    };
    if (kForm == 1) {
      asm volatile("" : "+s"(k_wave), "+s"(v_wave));
      landed();
    }
    unsigned char *const k_other = kStage ? kA : kB, *const v_other = kStage ? vA : vB;
    if (kForm > 1 && e + 1 < e1) copy_stage(walk.tile(ent_next), k_other, v_other, group);
    auto copy = [&](int n) { copy_piece(n, k_other, v_other, kStage ^ 1); };
    // causal tile: blocks of keys beyond the wave's block of queries are hidden, that block itself in part
    const int half = kForm == 1 ? kStage : group;
    const bool causal = (ent >> 30) != 0;
    if (!causal || kBlocks * half <= q_block) {
      key_blocks<kM, kBlocks, kForm == 1>(kStage ? kB : kA, kStage ? vB : vA, qf, oacc, st, nat, tr, p.scale_log2, q_block, kRows * half,
                                        causal && q_block < kBlocks * half + kBlocks, kForm == 1 ? kStage == 0 && e == e0 : !started, copy,
                                        [&]() { if (kFirst) look_ahead(); });
      started = true;
    }
    if (kForm == 1 && kStage == 1) {
      // the copies of a hidden half (not the other side of one branch, where the products do not stay in the same registers)
      int hidden = (ent >> 30) * max(kBlocks * half - q_block, 0);
      asm volatile("" : "+s"(hidden));
      if (hidden)
#pragma unroll
        for (int n = 0; n < 8; ++n) copy(n);
    }
    if (!kFirst) ent = ent_next;
    if (kForm > 1) landed();
  };
  for (int e = e0; e < e1; e += kForm == 1 ? 1 : 2) {
    step(e, std::integral_constant<int, 0>{});
    step(kForm == 1 ? e : e + 1, std::integral_constant<int, 1>{});
  }
  if constexpr (kForm == 1) {
    wait_vmem_all();            // the last step's copies filled with zeros a stage that is used for the results now
    __syncthreads();
  }

  // ---- epilogue: normalise, write O (bf16) and LSE (natural log) -------------------------
  float l_tot[2];
#pragma unroll
  for (int n = 0; n < M::kCols; ++n) l_tot[n] = M::column_sum(st[n].l_run);
  // (Walks on 16x16x32 read what only the end needs from the kernel-argument segment now: it would occupy scalar registers during a long walk.  On
  // 32x32x16 there are enough of them, and the read at the end takes a short walk 0.15 us: 19 heads of causal 2048 x 128 7.40 -> 7.22.)
  const FwdParams& pe = kM == 16 ? *(const FwdParams*)params_late() : p;
  bf16* orow = pe.o + b * pe.os.b + (int64_t)qrow0 * pe.os.s + h * pe.os.h;
  float* lrow = pe.lse + ((int64_t)b * pe.n_heads + h) * ((int64_t)pe.n_qtiles * kTile) + qrow0;
  int64_t o_stride = pe.os.s;
  int64_t part_at = 0;                     // element of the partial O
  if (part >= 0) {
    const int64_t seq = (int64_t)(pe.n_qtiles - pe.n_whole) * kTile, row = qrow0 - (int64_t)pe.n_whole * kTile;
    part_at = part * pe.o_part + ((b * seq + row) * pe.n_heads + h) * kHeadDim;
    orow = static_cast<bf16*>(pe.part_o) + part_at;
    lrow = pe.part_lse + part * pe.lse_part + ((int64_t)b * pe.n_heads + h) * seq + row;
    o_stride = (int64_t)pe.n_heads * kHeadDim;
  }
  if constexpr (kForm == 1) {
    RowPair inv;
#pragma unroll
    for (int n = 0; n < M::kCols; ++n) inv.x[n] = l_tot[n] > 0.f ? 1.f / l_tot[n] : 0.f;
    const uint32_t turn = lds_at((wave < 2 ? kA : vA) + (wave & 1) * kWaveRowsBytes);
    if (part >= 0 && pe.part_f32)   store_rows_f32<kM>(static_cast<float*>(pe.part_o) + part_at, o_stride, oacc, inv, turn);
    else                            store_rows_bf16<kM>(orow, o_stride, oacc, inv, turn);
  } else {
    // the groups exchange their rows' max, sum and O.  Area x of the stages' LDS belongs to group x % kForm of wave x / kForm.
    __shared__ float stat[8][2][64];
    auto area = [&](int x) { return lds_at(x < 2 ? sKA : x < 4 ? sVA : x < 6 ? sKB : sVB) + (x & 1) * kAccBytes; };
    const int own = wave * kForm + group;
    constexpr bool kAll = kForm == 2;        // the first group finishes whole rows; with four groups each a block of 32 columns
    stat[own][0][lane] = st[0].m_run;
    stat[own][1][lane] = l_tot[0];
    if (!kAll || group == 1) put_acc(area(own), oacc, kAll ? -1 : group);
    __syncthreads();
    if (kAll && group == 1) return;
    float m = -INFINITY, w[kForm];
#pragma unroll
    for (int g = 0; g < kForm; ++g) m = fmaxf(m, stat[wave * kForm + g][0][lane]);
    const float ms = m == -INFINITY ? 0.f : m;
    l_tot[0] = 0.f;
#pragma unroll
    for (int g = 0; g < kForm; ++g) {
      w[g] = fast_exp2(stat[wave * kForm + g][0][lane] - ms);
      l_tot[0] += stat[wave * kForm + g][1][lane] * w[g];
    }
    st[0].m_run = m;
    const float inv = l_tot[0] > 0.f ? 1.f / l_tot[0] : 0.f;
    if constexpr (kAll) {
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) add_block(area(own + 1), mb, oacc[mb], w[0], w[1]);
      store_rows_bf16<kM>(orow, o_stride, oacc, both(inv), area(own + 1));
    } else {
      f32x16 o;
      sum_blocks(o, oacc, group, [&](int g) { return area(wave * kForm + g); }, w);
      store_block_bf16(orow + 32 * group, o_stride, o, inv, area(own) + 4096 * group);
    }
  }
  const int out_lane = fresh_lane();
  if (out_lane < 32 && group == 0) {
    const bool second = M::kCols == 2 && out_lane >= 16;
    const float l = l_tot[second ? 1 : 0], m = st[second ? 1 : 0].m_run;
    lrow[out_lane] = l > 0.f ? (m + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
  }
}

// Lists run on 16x16x32 matrix instructions, dense rectangles on 32x32x16.  Either sums a product in another order, so that a few in a hundred
// entries of O round to the other bf16: delta = rowsum(dO * O), which the flash-attention signatures return in fp32 beside dense gradients,
// would move by 1.5e-4, for 2 to 4 % of a long forward.
template <int kForm, bool kDense>
__global__ __launch_bounds__(Groups<kForm>::kThreads, 2) void fwd_kernel(const FwdParams p) { fwd_lines<kForm, kDense, kDense ? 32 : 16>(p); }
// A dense rectangle whose results are to be those of its tile list.
template <int kM>
__global__ __launch_bounds__(Groups<1>::kThreads, 2) void fwd_plain_kernel(const FwdParams p) { fwd_lines<1, true, kM>(p); }

// Tile lists of few lines (see few_lines): the walk of fwd_kernel<1> with eight waves of 16 rows instead of four of 32, two on every
// SIMD, one in its products while the other is in its softmax.  A row meets the same products and sums in the same order, so that
// its result is the same bit for bit.
// Bound: LDS.  Every K and V fragment is read for 16 rows instead of 32, 256 KiB a half tile at the 128 bytes a cycle that LDS
// gives: 0.86 us a half tile, with four waves 0.97.  Where two workgroups share a CU it is slower.
template <int kWaveRows>
__global__ __launch_bounds__(512, 2) void fwd_short_kernel(const FwdParams p) {
  using M = Mma<16>;
  static_assert(kWaveRows == 16 && M::kCols * 16 == 32, "one of the two columns that a lane of fwd_kernel holds");
  constexpr int kHalfRows = 64, kStageK = kHalfRows * kRowBytes, kStageV = kHalfRows / 4 * M::kPitchV, kTurnBytes = kWaveRows * kRowBytes;
  __shared__ __attribute__((aligned(1024))) unsigned char sKA[kStageK];
  __shared__ __attribute__((aligned(1024))) unsigned char sVA[kStageV];
  __shared__ __attribute__((aligned(1024))) unsigned char sKB[kStageK];
  __shared__ __attribute__((aligned(1024))) unsigned char sVB[kStageV];
  const int lane = threadIdx.x & 63, row = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int pos, bh;
  map_block(blockIdx.x, p.map, pos, bh);
  const int b = quotient(bh, p.by_heads), h = bh - b * p.n_heads;
  const int qt = min(max(sload(p.q_order, pos), 0), p.n_qtiles - 1);
  const int e0 = min(max(sload(p.row_ptr, qt), 0), p.nnz), e1 = min(max(sload(p.row_ptr, qt + 1), e0), p.nnz);
  const bf16* const kbase = p.k + b * p.ks.b + h * p.ks.h;
  const bf16* const vbase = p.v + b * p.vs.b + h * p.vs.h;
  const int k_stride = (int)p.ks.s, v_stride = (int)p.vs.s;
  // A stage's four copies: fours of rows `wave` and 8 + `wave` of K and V.
  const int four_row = 4 * wave + (lane >> 4);
  const int koff = (four_row * k_stride + slot_k(four_row, row) * 8) * 2, voff = (four_row * v_stride + slot_v(four_row, row) * 8) * 2;
  const uint32_t k_extent = (uint32_t)((kTile - 1) * k_stride + kHeadDim) * 2, v_extent = (uint32_t)((kTile - 1) * v_stride + kHeadDim) * 2;
  auto lds_at = [](unsigned char* x) { return (uint32_t)(uintptr_t)(lds_byte*)x; };
  u32x4 k_rsrc, v_rsrc;                    // without `more` the copies fill with zeros a stage that no step reads
  auto tile = [&](int t, bool more) {
    k_rsrc = make_rsrc_words(kbase + (int64_t)t * kTile * k_stride, more ? k_extent : 0);
    v_rsrc = make_rsrc_words(vbase + (int64_t)t * kTile * v_stride, more ? v_extent : 0);
  };
  auto copy = [&](int n, unsigned char* k_stage, unsigned char* v_stage, int half) {
    const int j = n >> 1, first = half * kHalfRows + 32 * j;
    if (n & 1) dma16_abs(v_rsrc, lds_at(v_stage) + (8 * j + wave) * M::kPitchV, voff, first * v_stride * 2);
    else       dma16_abs(k_rsrc, lds_at(k_stage) + (8 * j + wave) * 1024, koff, first * k_stride * 2);
  };
  Walk<false, true> walk(e0, e1, -1);
  int ent = 0, ent_next = 0;
  if (e0 < e1) {
    walk.fetch(e0, p.col_idx, p.flag, p.n_ktiles);
    ent = walk.at(e0);
    tile(walk.tile(ent), true);
#pragma unroll
    for (int n = 0; n < 4; ++n) copy(n, sKA, sVA, 0);
  }
  const int qrow0 = qt * kTile + kWaveRows * wave, q_block = wave >> 1;
  // Q rows come in, and O goes out, through LDS, so that memory sees whole rows (1.3 us of a walk of one tile, 7.5 -> 6.2 us)
  // (through the stage that the first step fills)
  const bf16* const qrow = p.q + b * p.qs.b + (int64_t)(qrow0 + (lane >> 4)) * p.qs.s + h * p.qs.h + 8 * row;
  const uint32_t q_turn = lds_at(wave < 4 ? sKB : sVB) + (wave & 3) * kTurnBytes;
  u32x4 raw[4];
  bf16x8 qf[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) raw[i] = *reinterpret_cast<const u32x4*>(qrow + 4 * i * p.qs.s);
#pragma unroll
  for (int i = 0; i < 4; ++i) lds_put(q_turn + row_slot(4 * i + (lane >> 4), row), raw[i]);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) qf[ks] = lds_get<bf16x8>(q_turn + row_slot(row, M::a_chunk(lane, ks)));
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(qf[ks]));      // read before the walk
  f32x4 oacc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) oacc[i] = f32x4{0};
  float m_run = -INFINITY, m_use = 0.f, l_run = 0.f;
  int nat[4], tr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    nat[i] = lds_off_k(M::a_row(lane), M::a_chunk(lane, i));
    tr[i] = M::tr_offset(lane, i, M::kPitchV);
  }
  auto step = [&](int e, auto stage_tag) {
    constexpr int kStage = decltype(stage_tag)::value;
    const unsigned char *const sK = kStage ? sKB : sKA, *const sV = kStage ? sVB : sVA;
    unsigned char *const k_other = kStage ? sKA : sKB, *const v_other = kStage ? sVA : sVB;
    if (kStage == 1) tile(walk.tile(ent_next), e + 1 < e1);
    wait_vmem_all();
    __syncthreads();
    const bool causal = (ent >> 30) != 0, hidden = causal && 2 * kStage > q_block;
    if (hidden) {
#pragma unroll
      for (int n = 0; n < 4; ++n) copy(n, k_other, v_other, kStage ^ 1);
    } else {
      f32x4 s[4];
      constexpr int kAhead = 4;
      bf16x8 kfr[16];
      auto rd = [&](int i) { return lds_read_b128(sK, nat[i >> 2] + 16 * kRowBytes * (i & 3)); };
#pragma unroll
      for (int i = 0; i < kAhead; ++i) kfr[i] = rd(i);
      __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (i + kAhead < 16) kfr[i + kAhead] = rd(i + kAhead);
        s[i & 3] = M::mfma(kfr[i], qf[i >> 2], i < 4 ? f32x4{0} : s[i & 3]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if ((i & 3) == 3) copy(i >> 2, k_other, v_other, kStage ^ 1);
      }
      if (causal && q_block < 2 * kStage + 2) {
        const int key = kHalfRows * kStage + 4 * (fresh_lane() >> 4), query = kWaveRows * wave + (fresh_lane() & 15);
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (key + 16 * (i >> 2) + (i & 3) > query) s[i >> 2][i & 3] = -INFINITY;
      }
      constexpr int kVAhead = 4;
      bf16x8 vfr[16];
      auto rd_v = [&](int i) {
        const int at = tr[(i & 7) >> 1] + M::tr_first(i & 7, M::kPitchV) + 8 * M::kPitchV * (i >> 3);
        const bf16x4 lo = lds_read_tr16_b64(sV, at), hi = lds_read_tr16_b64(sV, at + M::tr_second(M::kPitchV));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      };
#pragma unroll
      for (int i = 0; i < kVAhead; ++i) vfr[i] = rd_v(i);
      // (Here, before the softmax: one by one between the MFMAs, where the compiler puts those of a tile's first half, every one is waited for.
      // One head, causal 4096, 57.8 -> 55.3 us.)
      __builtin_amdgcn_sched_barrier(0);
      if (kStage == 0) {                     // the next tile's entry
        if (!walk.has(e + 1)) walk.fetch(e + 1, p.col_idx, p.flag, p.n_ktiles);
        ent_next = walk.at(min(e + 1, e1 - 1));
      }
      const bool first = kStage == 0 && e == e0;
      float rs = 0.f;
      bf16x8 pf[2];
      auto exponentials = [&]() {
        rs = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float pv = fast_exp2(fmaf(s[i >> 2][i & 3], p.scale_log2, -m_use));
          rs += pv;
          pf[i >> 3][i & 7] = (bf16)pv;
        }
      };
      bool raise = first;
      if (!first) {
        exponentials();
        raise = __builtin_amdgcn_ballot_w64(!(rs < kRaiseSum)) != 0;
      }
      if (raise) {                           // as in key_blocks
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i >> 2][i & 3]);
        mx = M::column_max(mx) * p.scale_log2;
        const bool needed = first || M::column_max(rs < kRaiseSum ? 0.f : 1.f) > 0.f;
        const float m_new = needed ? fmaxf(m_run, mx) : m_run;
        const float m_at = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = (m_new == m_run) ? 1.f : fast_exp2(m_run - m_at);
        m_run = m_new;
        m_use = m_at;
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < 8; ++i) oacc[i] *= alpha;
        exponentials();
      }
      l_run += rs;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (i + kVAhead < 16) vfr[i + kVAhead] = rd_v(i + kVAhead);
        oacc[i & 7] = M::mfma(vfr[i], pf[i >> 3], oacc[i & 7]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
    }
    if (kStage == 1) ent = ent_next;
  };
  for (int e = e0; e < e1; ++e) {
    step(e, std::integral_constant<int, 0>{});
    step(e, std::integral_constant<int, 1>{});
  }
  wait_vmem_all();              // the last step's copies filled with zeros a stage that is used for the results now
  __syncthreads();
  const float l_tot = M::column_sum(l_run), inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  const uint32_t turn = lds_at(wave < 4 ? sKA : sVA) + (wave & 3) * kTurnBytes;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    bf16x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (bf16)(oacc[i][j] * inv);
    lds_put(turn + row_slot(row, 2 * i + (lane >> 5)) + 8 * (lane >> 4 & 1), w);
  }
  bf16* const orow = p.o + b * p.os.b + (int64_t)(qrow0 + (lane >> 4)) * p.os.s + h * p.os.h + 8 * row;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<u32x4*>(orow + 4 * i * p.os.s) = lds_get<u32x4>(turn + row_slot(4 * i + (lane >> 4), row));
  if (lane < 16)
    p.lse[((int64_t)b * p.n_heads + h) * ((int64_t)p.n_qtiles * kTile) + qrow0 + lane] =
        l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * kLn2 : -INFINITY;
}

}  // namespace ua

namespace ua {

static int fwd_common(FwdParams& p, const void* q, const void* k, const void* v, void* o, float* lse,
                      int batch, int n_heads, int n_qtiles, int n_ktiles, int head_dim,
                      const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                      const int64_t* o_strides, float softmax_scale) {
  if (!q || !k || !v || !o || !lse || !q_strides || !k_strides || !v_strides || !o_strides) return UA_ERR_NULL;
  if (batch <= 0 || n_heads <= 0 || n_qtiles <= 0 || n_ktiles <= 0) return UA_ERR_SHAPE;
  if ((int64_t)batch * n_heads * n_qtiles * UA_MAX_PARTS > INT32_MAX) return UA_ERR_SHAPE;
  if (head_dim != kHeadDim || !(softmax_scale > 0.f)) return UA_ERR_UNSUPPORTED;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o)) return UA_ERR_ALIGN;
  if (!strides_ok(q_strides) || !strides_ok(k_strides) || !strides_ok(v_strides) || !strides_ok(o_strides))
    return UA_ERR_ALIGN;
  if (k_strides[1] > (INT32_MAX >> 9) || v_strides[1] > (INT32_MAX >> 9)) return UA_ERR_SHAPE;
  p.q = (const bf16*)q; p.k = (const bf16*)k; p.v = (const bf16*)v; p.o = (bf16*)o; p.lse = lse;
  p.row_ptr = nullptr; p.col_idx = nullptr; p.flag = nullptr; p.q_order = nullptr;
  p.batch = batch; p.n_heads = n_heads; p.n_qtiles = n_qtiles; p.n_ktiles = n_ktiles; p.nnz = 0; p.n_first = 0;
  p.qs = {q_strides[0], q_strides[1], q_strides[2]};
  p.ks = {k_strides[0], k_strides[1], k_strides[2]};
  p.vs = {v_strides[0], v_strides[1], v_strides[2]};
  p.os = {o_strides[0], o_strides[1], o_strides[2]};
  p.scale_log2 = softmax_scale * kLog2e;
  p.dense = 0; p.dense_causal = 0; p.diag_off = 0; p.n_whole = n_qtiles; p.n_parts = 1; p.part_len = n_ktiles;
  p.part_o = nullptr; p.part_lse = nullptr; p.o_part = 0; p.lse_part = 0; p.part_f32 = 0;
  return check_device();
}

// Groups per workgroup for n lines of 128 rows (parts counted) of a dense rectangle:
//  - four, on half lines, while those leave a CU one workgroup at most (8 heads of 1024: 17.2 us with two groups, 13.8
//    with four; 2048: 29.9, 24.3).  Walks of one tile keep one group: four would take 5.5 us instead of 5.7, but a row would have
//    other bits in a launch of up to 128 lines than in a longer one, and delta = rowsum(dO * O) move by 2.6e-3 with them.
//  - two, on whole lines, up to one workgroup per CU and from three tiles on (32 heads of 1024: 25 us with one, 22 with two).
//  - The rows of an uncut causal rectangle differ in length.  Run one after the other, longest first, they are
//    balanced, which workgroups resident side by side from the start do not achieve: four groups up to 256 lines of 16
//    tiles (8 heads of 4096: 57 us with two, 48 with four), two up to 512 lines (16 heads of 4096: 89 us with one, 77 with
//    two).
// Groups sum in another order, so that the last bits of a row depend on how many lines the launch has.  Tile lists, whose
// launches are shards of the rows and heads of one mask, therefore run with one group whatever their size: a row's result is
// the same bit for bit in every launch that holds its list.  Lists of up to 128 lines pay for that (one head, causal 4096: forward
// 35 us with four groups, 55 with one, see few_lines, backward 51 and 119; from 512 lines on little changes).
static int fwd_groups(int64_t n, int64_t walk, int n_parts, bool dense_causal) {
  const bool uneven = dense_causal && n_parts == 1;
  if (walk >= 2 && (2 * n <= kCus || (uneven && n <= kCus && walk >= 16))) return 4;
  return walk >= 3 && n <= (uneven ? 2 * kCus : kCus) ? 2 : 1;
}
// Tile lists of n lines that run with eight waves a workgroup: up to one line a CU, and up to seven on eight CUs where nearly all lines are of
// full length and longer than 16 tiles.  Both kernels give the same bits, so that the line is drawn by time alone: us, four waves and eight
//     lines                      128            208            240            256            320
//     causal, 16 tiles     35.2   30.8    36.3   32.1    36.4   33.2    35.9   32.2    36.8   34.4
//     causal, 64 tiles    123.3  109.5                                 126.6  113.6   126.5  121.2
//     strided, 16 tiles    14.5   12.3    16.7   15.2    17.3   16.2    15.6   14.3    20.0   22.7
//     global+local, 16     35.5   32.6    36.6   34.1    37.2   36.8    36.4   35.2    40.2   49.9
//     full, 4 tiles        12.2   10.7    14.0   12.8    14.9   14.4    13.8   12.7    18.7   22.0
//     full, 16 tiles       35.1   33.0    37.2   35.6    37.6   37.4    37.1   37.0    52.3   66.2
//     full, 64 tiles      125.2  112.7                                 133.3  141.4   190.8  242.7
static bool few_lines(const FwdParams& p, int64_t n) {
  const bool uneven = (int64_t)4 * p.nnz <= (int64_t)3 * p.n_qtiles * p.n_ktiles, brief = p.nnz <= 16 * (int64_t)p.n_qtiles;
  return n <= (uneven || brief ? kCus : kCus / 8 * 7);
}
// `plain`: one group per workgroup, and of a dense rectangle the bits of its tile list.
static int fwd_launch(FwdParams& p, bool plain, hipStream_t st) {
  const unsigned n = (unsigned)(p.batch * p.n_heads * (p.n_whole + (p.n_qtiles - p.n_whole) * p.n_parts));
  // (several groups copy Q through a buffer descriptor, whose offsets have 32 bits)
  const int form = plain || p.qs.s > (INT32_MAX >> 9) ? 1 : fwd_groups(n, p.part_len, p.n_parts, p.dense_causal);
  const int n_cut = p.n_qtiles - p.n_whole;
  p.map = block_map(p.batch * p.n_heads, (p.n_whole + n_cut * p.n_parts) * (form == 4 ? 2 : 1));
  p.by_heads = make_div(p.n_heads);
  p.by_cut = make_div(n_cut ? n_cut : 1);
  switch (form) {
    case 4:
      hipLaunchKernelGGL((fwd_kernel<4, true>), dim3(2 * n), dim3(512), 0, st, p);
      break;
    case 2:
      hipLaunchKernelGGL((fwd_kernel<2, true>), dim3(n), dim3(512), 0, st, p);
      break;
    default:
      // Up to two workgroups per CU the whole launch is resident at once, and those after the first 256 join them in
      // launch order.  Lists come roughly by falling length, so the first ones are taken in reverse: long and
      // short lists then share a CU (strided 8k, 8 heads: the longest sum on a CU 40 -> 37 tiles, causal 96 -> 65).
      if (!p.dense && n > kCus && n <= 2 * kCus) p.n_first = kCus * p.n_qtiles / (int)n;
      if (p.dense && plain)    hipLaunchKernelGGL((fwd_plain_kernel<16>), dim3(n), dim3(256), 0, st, p);
      else if (p.dense)        hipLaunchKernelGGL((fwd_kernel<1, true>), dim3(n), dim3(256), 0, st, p);
      else if (few_lines(p, n)) hipLaunchKernelGGL((fwd_short_kernel<16>), dim3(n), dim3(512), 0, st, p);
      else                     hipLaunchKernelGGL((fwd_kernel<1, false>), dim3(n), dim3(256), 0, st, p);
  }
  return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
}

// How many parts the walks of a dense forward are cut into, at most max_parts (what the workspace holds).  A cut
// gives a small rectangle enough workgroups and costs the partials' way through memory, a merge, and a second rounding of
// every row: the partial O is bf16 (error against fp64 2.33e-3 whole and 2.85e-3 cut at 8 heads of 4480, and
// as much in 11 parts as in two).  Two estimates of the launches' time in microseconds therefore have to agree on a cut:
//  - the first, fitted to 47 shapes of 1 to 32 heads and 128 to 8192 tokens, says which rectangles have enough to gain (5 heads of 8192,
//    200 us whole and 179 cut in two, do not);
//  - the second, fitted to 140 rectangles of 1 to 20 heads and 256 to 16384 tokens, counts what a causal rectangle shows and gives the number
//    of parts, or none: 16 heads, causal 640 x 1920, 21.6 us cut in three, 19.5 whole; 2 x 3 causal 6784 94.9 and 89.8.
// Terms: start, loading Q, storing and the end; a tile, and one where two workgroups share the CU; the merge, and the partials' bytes.
// 1024 x 4096, one head: 34 us uncut, 12 cut in 11.
//
// Causal rectangles of more keys than queries whose whole walks run in a second round (more than 128 lines in four groups, more than 256 in
// two) are cut by an estimate of their own: the second round begins when the shortest rows of the first are through, and all rows
// are long.  Their partial O is fp32, so that every row is rounded once (bf16 partials take 2 to 4 us less).  10 heads of 1664 x 6144 87.8 -> 56.4
// us, 3 of 7296 x 29440 430 -> 282; over 5400 causal rectangles of 129 to 511 lines 8 % less time than whole, three of them
// more than 6 % slower, 9 at most.  (256 lines, the most of four groups, stay whole: what callers are told to bring there is two parts in bf16.)
struct FwdCut {
  int parts;
  bool f32;
};
static FwdCut fwd_cut(int64_t nbh, int n_qtiles, int n_ktiles, bool causal, int max_parts) {
  const float lines = (float)nbh * n_qtiles;
  auto share = [](float groups) { return fminf(fmaxf((groups - kCus) / kCus, 0.f), 1.f); };        // of the workgroups with a neighbour
  auto first = [&](int parts) {
    const int len = (n_ktiles + parts - 1) / parts;
    const float density = causal ? 0.5f : 1.f, groups = lines * parts, merge = parts > 1 ? 2.4f + 0.03f * parts + groups * (kTile * kHeadDim * 2) / 1.5e6f : 0.f;
    switch (fwd_groups(nbh * n_qtiles * parts, len, parts, causal)) {
      case 4: return merge + 5.1f + len * 1.1f;
      case 2: return merge + 4.3f + len * 1.8f;
      default: return merge + 3.8f + fmaxf(len * (2.2f + 1.5f * share(groups * density)), density * lines * n_ktiles * 3.7f / (2 * kCus));
    }
  };
  auto second = [&](int parts) {
    const int len = (n_ktiles + parts - 1) / parts, made = (n_ktiles + len - 1) / len;
    const float density = visible_share(n_qtiles, n_ktiles, causal), groups = lines * made;
    const float merge = made > 1 ? 3.3f + 0.034f * made + groups * (kTile * kHeadDim * 2) / 1.72e6f : 0.f;
    switch (fwd_groups(nbh * n_qtiles * made, len, made, causal)) {
      case 4: return merge + 4.3f + 0.5f * (groups / 128) * (groups / 128) + len * 1.04f;
      case 2: return merge + 4.9f + len * 1.55f;
      default: return merge + 3.35f + fmaxf(len * (2.4f + 1.15f * share(groups * density)), density * lines * n_ktiles * 3.66f / (2 * kCus));
    }
  };
  auto least = [&](auto us_of) {
    int best = 1;
    float best_us = INFINITY;
    for (int parts = 1; parts <= max_parts; ++parts) {
      const float us = us_of(parts);
      if (us < 0.99f * best_us) { best_us = us; best = parts; }          // more parts for a gain, not for a tie
    }
    return best;
  };
  if (const int parts = least(first) > 1 ? least(second) : 1; parts > 1) return {parts, false};
  const int whole = fwd_groups(nbh * n_qtiles, n_ktiles, 1, causal), round = whole == 4 ? kCus / 2 : kCus;
  if (!causal || n_ktiles <= n_qtiles || whole == 1 || lines <= round || (whole == 4 && max_parts <= 2)) return {1, false};
  const float shortest = n_ktiles - n_qtiles * round / lines;                  // row of the first round
  auto rounded_once = [&](int parts) {
    // (a workgroup of the second round starts anew; a cut has to win by 3 %)
    if (parts == 1) return 0.97f * (whole == 4 ? fmaxf(5.f + 1.08f * n_ktiles, 9.f + 2.4f * shortest) : fmaxf(5.f + 1.6f * n_ktiles, 14.f + 3.5f * shortest));
    const int len = (n_ktiles + parts - 1) / parts, made = (n_ktiles + len - 1) / len;
    if (fwd_groups(nbh * n_qtiles * made, len, made, causal) != 1) return INFINITY;          // (several groups leave bf16)
    const float density = visible_share(n_qtiles, n_ktiles, causal), groups = lines * made;
    return 6.65f + groups * (kTile * kHeadDim * 4) / 2.5e6f + fmaxf(len * (2.4f + 1.15f * share(groups * density)), density * lines * n_ktiles * 3.66f / (2 * kCus));
  };
  const int parts = least(rounded_once);
  return {parts, parts > 1};
}

static bool contiguous_bshd(const int64_t* st, int seqlen, int n_heads) {
  return st[2] == kHeadDim && st[1] == (int64_t)n_heads * kHeadDim && st[0] == (int64_t)seqlen * n_heads * kHeadDim;
}

}  // namespace ua

extern "C" int ua_bsa_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                          const int32_t* row_ptr, const int32_t* col_idx, const uint8_t* flag,
                          const int32_t* q_order,
                          int batch, int n_heads, int n_qtiles, int n_ktiles, int nnz, int head_dim,
                          const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                          const int64_t* o_strides, float softmax_scale, void* stream) {
  using namespace ua;
  if (!row_ptr || !q_order) return UA_ERR_NULL;
  if (nnz < 0) return UA_ERR_SHAPE;
  if (nnz > 0 && (!col_idx || !flag)) return UA_ERR_NULL;      // only an empty list may leave them out
  if (flag && !aligned4(flag)) return UA_ERR_ALIGN;            // (a rule of the interface: whole words, so that a reader may take four at once)
  FwdParams p;
  if (int rc = fwd_common(p, q, k, v, o, lse, batch, n_heads, n_qtiles, n_ktiles, head_dim, q_strides, k_strides,
                          v_strides, o_strides, softmax_scale)) return rc;
  p.row_ptr = row_ptr; p.col_idx = col_idx; p.flag = flag; p.q_order = q_order; p.nnz = nnz;
  return fwd_launch(p, true, (hipStream_t)stream);
}

namespace ua {

// The last wave of a large rectangle.  Its lines run two to a CU, 512 at a time; up to 256 lines left over would hold
// the launch open for a whole walk with most of the device idle (2304 x 3456, 32 heads: 576 lines of 27 tiles, 149 us, of
// which 50 for the last 64 lines; cut 129).  The left-over query tiles at the end of every sequence are then cut into parts
// that fill the device, if the estimate of that and of their merge is shorter: the fp32 partials take 1 us per 2.5 MB
// (2560 x 2048, 32 heads, 128 lines over: 91.2 us, cut 89.1; 3072 x 2048, 256 over: 97, cut in two 103, not done).  bf16
// partials took up to 3 us less at the first shape and gave the rows of the last wave a second rounding, an error 20 % larger
// than their neighbours'.  Causal rows balance themselves.
struct Cut {
  int tiles, parts;
  bool f32;                                // partial O
};
static Cut fwd_tail(int64_t nbh, int n_qtiles, int n_ktiles) {
  constexpr int kRound = 2 * kCus;
  const int64_t lines = nbh * n_qtiles, rounds = lines / kRound;
  if (rounds == 0 || lines % kRound == 0 || lines % kRound > kCus) return {0, 1, false};
  const int tail = n_qtiles - (int)(rounds * kRound / nbh);
  const int64_t cut = nbh * tail;
  const int64_t most = n_ktiles / 2 < UA_MAX_PARTS ? n_ktiles / 2 : UA_MAX_PARTS, parts = kRound / cut < most ? kRound / cut : most;
  if (tail >= n_qtiles || parts < 2) return {0, 1, false};
  const float us = 3.7f * cut * n_ktiles / kRound + 4.f + 2.4f + cut * parts * (kTile * kHeadDim * 4) / 2.5e6f;
  return us < 2.2f * n_ktiles ? Cut{tail, (int)parts, true} : Cut{0, 1, false};
}
// One part's share of the workspace for n_tiles cut query tiles.
struct PartBytes {
  int64_t o, lse;
  int64_t total() const { return o + lse; }
};
static PartBytes part_bytes(int batch, int n_heads, int n_tiles, bool f32) {
  const int64_t rows = (int64_t)batch * n_heads * n_tiles * kTile;
  return {align256(rows * kHeadDim * (f32 ? 4 : 2)), align256(rows * 4)};
}
// Query tiles at the end that are cut, and into how many parts.
static Cut dense_cut(int batch, int n_heads, int n_qtiles, int n_ktiles, bool causal) {
  const int64_t nbh = (int64_t)batch * n_heads;
  const int max_parts = dense_split(batch, n_heads, n_qtiles, n_ktiles).fwd_parts;
  if (max_parts == 1) return causal ? Cut{0, 1, false} : fwd_tail(nbh, n_qtiles, n_ktiles);
  const FwdCut cut = n_heads > kMaxHeadsLds ? FwdCut{1, false} : fwd_cut(nbh, n_qtiles, n_ktiles, causal, max_parts);       // (more heads: not merged)
  return {cut.parts > 1 ? n_qtiles : 0, cut.parts, cut.f32};
}

static int64_t fwd_workspace_used(int batch, int n_heads, int n_qtiles, int n_ktiles, bool causal) {
  const Cut cut = dense_cut(batch, n_heads, n_qtiles, n_ktiles, causal);
  return cut.tiles ? cut.parts * part_bytes(batch, n_heads, cut.tiles, cut.f32).total() : 0;
}

}  // namespace ua

extern "C" int64_t ua_dense_workspace_used(int batch, int n_heads, int seqlen_q, int seqlen_k, int causal, int backward) {
  using namespace ua;
  if (batch <= 0 || n_heads <= 0 || seqlen_q <= 0 || seqlen_k <= 0 || seqlen_q % kTile || seqlen_k % kTile) return 0;
  return (backward ? bwd_workspace_used : fwd_workspace_used)(batch, n_heads, seqlen_q / kTile, seqlen_k / kTile, causal != 0);
}

extern "C" int64_t ua_dense_workspace_bytes(int batch, int n_heads, int seqlen_q, int seqlen_k, int backward) {
  using namespace ua;
  if (batch <= 0 || n_heads <= 0 || seqlen_q <= 0 || seqlen_k <= 0 || seqlen_q % kTile || seqlen_k % kTile) return 0;
  const int n_qtiles = seqlen_q / kTile, n_ktiles = seqlen_k / kTile;
  const DenseSplit d = dense_split(batch, n_heads, n_qtiles, n_ktiles);
  if (backward) return d.bwd_total;
  if (d.fwd_parts > 1) return std::max(d.fwd_total, fwd_workspace_used(batch, n_heads, n_qtiles, n_ktiles, true));       // (causal ones may leave fp32)
  const Cut t = fwd_tail((int64_t)batch * n_heads, n_qtiles, n_ktiles);
  return t.tiles ? t.parts * part_bytes(batch, n_heads, t.tiles, true).total() : 0;
}

extern "C" int ua_dense_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                            int batch, int n_heads, int seqlen_q, int seqlen_k, int head_dim,
                            const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                            const int64_t* o_strides, float softmax_scale, int causal,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace ua;
  if (seqlen_q <= 0 || seqlen_k <= 0 || seqlen_q % kTile || seqlen_k % kTile) return UA_ERR_SHAPE;
  const int n_qtiles = seqlen_q / kTile, n_ktiles = seqlen_k / kTile;
  FwdParams p;
  if (int rc = fwd_common(p, q, k, v, o, lse, batch, n_heads, n_qtiles, n_ktiles, head_dim, q_strides, k_strides,
                          v_strides, o_strides, softmax_scale)) return rc;
  p.dense = 1; p.dense_causal = causal != 0; p.diag_off = n_ktiles - n_qtiles;
  hipStream_t st = (hipStream_t)stream;
  if (!workspace) return fwd_launch(p, true, st);
  const Cut cut = dense_cut(batch, n_heads, n_qtiles, n_ktiles, p.dense_causal);
  if (cut.tiles == 0) return fwd_launch(p, false, st);
  // cutting needs the caller's workspace and a contiguous output for the merge
  const PartBytes d = part_bytes(batch, n_heads, cut.tiles, cut.f32);
  const int64_t need = cut.parts * d.total();
  if (!aligned16(workspace) || workspace_bytes < need || !contiguous_bshd(o_strides, seqlen_q, n_heads)) return fwd_launch(p, false, st);
  p.n_whole = n_qtiles - cut.tiles;
  p.part_len = (n_ktiles + cut.parts - 1) / cut.parts;
  p.n_parts = (n_ktiles + p.part_len - 1) / p.part_len;
  p.part_o = workspace;
  p.part_lse = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + p.n_parts * d.o);
  p.o_part = d.o / (cut.f32 ? 4 : 2); p.lse_part = d.lse / 4; p.part_f32 = cut.f32;
  if (int rc = fwd_launch(p, false, st)) return rc;
  if (cut.f32) {
    const int64_t first = (int64_t)p.n_whole * kTile;
    return merge_f32_rows((const float*)p.part_o, p.o_part, p.part_lse, p.lse_part, p.n_parts, p.o + first * n_heads * kHeadDim, lse + first, seqlen_q,
                          batch, cut.tiles * kTile, n_heads, st);
  }
  const void* op[UA_MAX_PARTS];
  const float* lp[UA_MAX_PARTS];
  for (int i = 0; i < p.n_parts; ++i) { op[i] = (const bf16*)p.part_o + i * p.o_part; lp[i] = p.part_lse + i * p.lse_part; }
  return ua_merge(op, lp, p.n_parts, p.o, lse, batch, seqlen_q, n_heads, head_dim, stream);
}
