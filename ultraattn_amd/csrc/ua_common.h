// Shared device/host helpers for the gfx950 attention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/ultraattn.h"

namespace ua {

typedef __bf16 bf16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int kCus = 256;               // compute units of the device
constexpr int kTile = UA_TILE;          // 128 x 128 kernel tile
constexpr int kHeadDim = UA_HEAD_DIM;   // 128
constexpr int kRowBytes = kHeadDim * 2; // one K/V/Q row of bf16 in LDS
constexpr int kTileBytes = kTile * kRowBytes;  // 32 KiB
constexpr int kMaxHeadsLds = 256;       // heads whose statistics the merge, update and delta kernels take
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct Strides3 { int64_t b, s, h; };   // element strides of (batch, token, head)

// LDS address (bytes) of 16-byte chunk `c` (0..15) of row `r` in a [128][128] bf16 tile.
// K-type layout: chunk index XOR (row mod 16): 16 consecutive rows at one logical column
// land in 16 different 16-byte slots, so 128-bit row-fragment reads are conflict free.
__device__ __forceinline__ int lds_off_k(int r, int c) { return r * kRowBytes + ((c ^ (r & 15)) << 4); }
// V-type layout: fours of rows (1 KiB each, one copy of one wave) lie at a pitch of 1 KiB and a bit (Mma::kPitch), and the 64-byte
// group index is XORed with row mod 4, so that 128-bit reads of rows and transposing reads are free of bank conflicts.
__device__ __forceinline__ int slot_v(int r, int c) { return c ^ ((r & 3) << 2); }
__device__ __forceinline__ int slot_k(int r, int c) { return c ^ (r & 15); }

__device__ __forceinline__ bf16x8 lds_read_b128(const unsigned char* smem, int off) {
  return *reinterpret_cast<const bf16x8*>(smem + off);
}
// Transposing LDS read: across each group of 16 lanes, lane i receives element (i) of the
// 16-element row that lanes 4j..4j+3 point at, for j = 0..3 (4 rows x 16 columns -> column i).
__device__ __forceinline__ bf16x4 lds_read_tr16_b64(const unsigned char* smem, int off) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(smem + off));
}

template <int kLanes>                       // 16 or 32: with lane l ^ kLanes
__device__ __forceinline__ void swap_lanes(float x, float& a, float& b) {
  const uint32_t u = __float_as_uint(x);
  const auto r = kLanes == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- the matrix instruction of a walk: v_mfma_f32_16x16x32_bf16 or v_mfma_f32_32x32x16_bf16 -----------------------
// Both work on blocks of 32 x 32: acc[i] of a lane = row quad_row(i / 4) + i % 4, column col(quad_n(i / 4)).  The transposed products of the
// walks turn a block's accumulators, packed to bf16, into the B operand of the next product without leaving the lane.
//
// Register-only loops on random operands, at the socket's power limit: 16x16x32 runs at 2.0 to 2.1 GHz, 32x32x16 at 1.76 to 1.79.  With operands
// that change every time that is 1.90 and 1.79 PFLOP/s, with every A operand used twice in a row, as the walks do with 16x16x32,
// 1.98 and 1.81 (a B operand that two instructions share gives nothing).  The long launches, which that
// limit holds, gain 3 to 5 % in the forward (strided 128k 17.7 -> 17.1 ms) and 7 to 8 % in the backward (causal 32k, 32 heads
// 23.5 -> 21.7, strided 128k 57.8 -> 53.6), at 1.81 and 1.87 instead of 1.60 GHz.  But there are twice as many instructions to
// issue: beside a wave that issues them another one's fma, exp2 and add take 28 cycles instead of 22, and a step of a lone
// workgroup takes 6 % more cycles.  Backward launches of several groups a line that end in 5 to 20 us never meet the limit; with 16x16x32 they
// lose up to 13 %, so they run on 32x32x16 (see mma_of).  So do dense forwards, for their bits (see fwd_kernel).
template <int kM> struct Mma;
template <>
struct Mma<16> {
  static constexpr int kCols = 2, kRowRegs = 4;            // columns a lane holds; address registers of row reads
  // Pitch of the V-type layout's fours.  A transposing read gathers 32 bytes of each row of two fours per half wave: the rows are in
  // different 64-byte groups, the two fours in different halves of one.  A 128-bit read of 16 rows is served 16 lanes
  // at a time, half of the rows from either of two adjacent lane groups, whose chunks differ by one: different slots, too.  (With the fours'
  // starts 0, 32, 16 and 48 bytes into a 64-byte group the backward, 32 heads of 4096, met 68 million conflict cycles.  Now there are none in
  // the walks; what is left, 0.8 million, is 384 a workgroup where its rows turn through LDS at the walk's ends.)
  static constexpr int kPitch = 1056, kPitchV = kPitch;
  static __device__ __forceinline__ int col(int lane, int n) { return 16 * n + (lane & 15); }
  static __device__ __forceinline__ int quad_row(int lane, int q) { return 16 * (q >> 1) + 4 * (lane >> 4); }
  static constexpr __device__ int quad_n(int q) { return q & 1; }
  static __device__ __forceinline__ int quad_chunk(int lane, int q) { return 2 * (q >> 1) + (lane >> 5); }     // of 8 rows
  static __device__ __forceinline__ int quad_half(int lane) { return lane >> 4 & 1; }
  static __device__ __forceinline__ int quad_piece(int lane, int q) { return 4 * (q >> 1) + (lane >> 4); }       // of 4 rows
  // B fragment i (of 8) of 32 rows of 128: row and 16-byte chunk
  static __device__ __forceinline__ int frag_row(int lane, int i) { return 16 * (i & 1) + (lane & 15); }
  static __device__ __forceinline__ int frag_chunk(int lane, int i) { return 4 * (i >> 1) + (lane >> 4); }
  // First product, contracted over the 128: A fragment i (of 8) = 16 rows, a quarter of them.  (row and chunk of address register j; the
  // fragments' register and what lies between them)
  static __device__ __forceinline__ int a_row(int lane) { return lane & 15; }
  static __device__ __forceinline__ int a_chunk(int lane, int j) { return 4 * j + (lane >> 4); }
  static constexpr __device__ int a_reg(int i) { return i >> 1; }
  static constexpr __device__ int a_offset(int i, int four_pitch) { return (i & 1) * 4 * four_pitch; }
  // Second product, contracted over 32 rows: A fragment i = columns 16 * i .. + 15, all rows, read through the transposing path
  // as two halves: lane group g supplies rows 4g .. 4g + 3 and 16 + 4g .., as two blocks of 16 accumulator rows do.
  static __device__ __forceinline__ int tr_offset(int lane, int m, int pitch = kPitch) {
    const int g = lane >> 4, r = (lane & 15) >> 2, c = lane & 3;
    return pitch * g + r * kRowBytes + (slot_v(r, 4 * m + (c >> 1)) << 4) + (c & 1) * 8;
  }
  static constexpr __device__ int tr_reg(int i) { return i >> 1; }
  static constexpr __device__ int tr_first(int i, int = kPitch) { return 32 * (i & 1); }
  static constexpr __device__ int tr_second(int pitch = kPitch) { return 4 * pitch; }
  static constexpr __device__ int slot_n(int i) { return i >> 2 & 1; }                    // where acc[i] goes in the next B operand
  static constexpr __device__ int slot_j(int i) { return 4 * (i >> 3) + (i & 3); }
  static __device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ f32x4 quad(const f32x16& x, int q) { return f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]}; }
  static __device__ __forceinline__ void into(f32x16& x, int q, bf16x8 a, bf16x8 b, f32x4 c) {
    c = mfma(a, b, c);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[4 * q + j] = c[j];
  }
  // Zeros, two registers an instruction: of accumulators that are used four by four the compiler clears one register after the other, 128 of dK
  // and dV, and 0.35 us of every backward over lists (one tile 9.3 -> 8.9 us).
  static __device__ __forceinline__ void clear(f32x16& x) {
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      f32x2 zeros;
      asm volatile("v_mov_b64 %0, 0" : "=v"(zeros));
      x[i] = zeros[0];
      x[i + 1] = zeros[1];
    }
  }
  struct Start { f32x4 of[2]; };           // what a lane's columns start from
  static __device__ __forceinline__ Start start(const float (&x)[2]) { return {{f32x4{x[0], x[0], x[0], x[0]}, f32x4{x[1], x[1], x[1], x[1]}}}; }
  static __device__ __forceinline__ void keep(Start& s) { asm volatile("" : "+v"(s.of[0]), "+v"(s.of[1])); }
  static __device__ __forceinline__ void first(f32x16& acc, int i, bf16x8 a, const bf16x8 (&f)[8], const Start& from) {
#pragma unroll
    for (int n = 0; n < 2; ++n) into(acc, 2 * (i & 1) + n, a, f[2 * (i >> 1) + n], i < 2 ? from.of[n] : quad(acc, 2 * (i & 1) + n));
  }
  static __device__ __forceinline__ void second(f32x16 (&acc)[4], int i, bf16x8 a, const bf16x8 (&f)[2]) {
#pragma unroll
    for (int n = 0; n < 2; ++n) into(acc[i >> 1], 2 * (i & 1) + n, a, f[n], quad(acc[i >> 1], 2 * (i & 1) + n));
  }
  static __device__ __forceinline__ float column_max(float x) {
    float a, b;
    swap_lanes<16>(x, a, b);
    swap_lanes<32>(fmaxf(a, b), a, b);
    return fmaxf(a, b);
  }
  static __device__ __forceinline__ float column_sum(float x) {
    float a, b;
    swap_lanes<16>(x, a, b);
    swap_lanes<32>(a + b, a, b);
    return a + b;
  }
  // The instructions' order: an LDS read after the first of a fragment's two MFMAs, or (`reads` = 2) after either.
  template <int kReads>
  static __device__ __forceinline__ void interleave() {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (kReads == 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
};
template <>
struct Mma<32> {
  static constexpr int kCols = 1, kRowRegs = 8;
  // (The rows of two fours that a half wave gathers are whole 64-byte groups.)  V of the forward, of which no rows are read, lies at 1024.
  static constexpr int kPitch = 1040, kPitchV = 1024;
  static __device__ __forceinline__ int col(int lane, int) { return lane & 31; }
  static __device__ __forceinline__ int quad_row(int lane, int q) { return 8 * q + 4 * (lane >> 5); }
  static constexpr __device__ int quad_n(int) { return 0; }
  static __device__ __forceinline__ int quad_chunk(int, int q) { return q; }
  static __device__ __forceinline__ int quad_half(int lane) { return lane >> 5; }
  static __device__ __forceinline__ int quad_piece(int lane, int q) { return 2 * q + (lane >> 5); }
  static __device__ __forceinline__ int frag_row(int lane, int) { return lane & 31; }
  static __device__ __forceinline__ int frag_chunk(int lane, int i) { return 2 * i + (lane >> 5); }
  // First product: A fragment i = 32 rows, an eighth of the 128.
  static __device__ __forceinline__ int a_row(int lane) { return lane & 31; }
  static __device__ __forceinline__ int a_chunk(int lane, int j) { return 2 * j + (lane >> 5); }
  static constexpr __device__ int a_reg(int i) { return i; }
  static constexpr __device__ int a_offset(int, int) { return 0; }
  // Second product: A fragment i = columns 32 * (i % 4) .. + 31, 16 rows from 16 * (i / 4) on; lane half h supplies rows 4h .. 4h + 3 and 8 + 4h ..
  static __device__ __forceinline__ int tr_offset(int lane, int m, int pitch = kPitch) {
    const int i16 = lane & 15, r = i16 >> 2;
    return pitch * (lane >> 5) + r * kRowBytes + (slot_v(r, 4 * m + 2 * (lane >> 4 & 1) + ((i16 & 3) >> 1)) << 4) + (i16 & 1) * 8;
  }
  static constexpr __device__ int tr_reg(int i) { return i & 3; }
  static constexpr __device__ int tr_first(int i, int pitch = kPitch) { return 4 * pitch * (i >> 2); }
  static constexpr __device__ int tr_second(int pitch = kPitch) { return 2 * pitch; }
  static constexpr __device__ int slot_n(int i) { return i >> 3; }
  static constexpr __device__ int slot_j(int i) { return i & 7; }
  static __device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ void clear(f32x16& x) { x = f32x16{0}; }
  struct Start { f32x16 of; };
  static __device__ __forceinline__ Start start(const float (&x)[2]) {
    Start s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s.of[i] = x[0];
    return s;
  }
  static __device__ __forceinline__ void keep(Start& s) { asm volatile("" : "+v"(s.of)); }
  static __device__ __forceinline__ void first(f32x16& acc, int i, bf16x8 a, const bf16x8 (&f)[8], const Start& from) {
    acc = mfma(a, f[i], i == 0 ? from.of : acc);
  }
  static __device__ __forceinline__ void second(f32x16 (&acc)[4], int i, bf16x8 a, const bf16x8 (&f)[2]) { acc[i & 3] = mfma(a, f[i >> 2], acc[i & 3]); }
  static __device__ __forceinline__ float column_max(float x) {
    float a, b;
    swap_lanes<32>(x, a, b);
    return fmaxf(a, b);
  }
  static __device__ __forceinline__ float column_sum(float x) {
    float a, b;
    swap_lanes<32>(x, a, b);
    return a + b;
  }
  template <int kReads>
  static __device__ __forceinline__ void interleave() {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
  }
};
// Of a form of the backward's walks (see Groups).  The several groups' kernels, whose groups' indices take registers too, spill with 16x16x32 or
// read one fragment ahead: 8 heads of 2048 are 6 % faster all the same, of 1024 1 % and, causal, 3 % slower, 256 x 256 causal 13 %.
constexpr int mma_of(int form) { return form == 1 ? 16 : 32; }

// ---- row tiles of one wave: 32 rows of 256 bytes between memory and the operand / accumulator layouts ---------
// In those layouts a lane owns 8 or 16 bytes of a row, and a load or store straight from them touches 32 rows per
// instruction in pieces of 16 or 32 bytes: at 512 x 512, 32 heads the results' stores alone took 2.0 us of a 10 us
// forward and 3.3 of a 25 us backward.  Through 8 KiB of LDS that is the wave's own, memory sees four whole rows per
// instruction.  16-byte chunk c of row r lies in slot c ^ (r % 16), so that both sides are free of bank conflicts;
// a wave's LDS accesses are in order, no barrier is needed.
typedef __attribute__((address_space(3))) unsigned char lds_byte;
constexpr int kWaveRowsBytes = 32 * kRowBytes;
__device__ __forceinline__ uint32_t row_slot(int r, int c) { return r * kRowBytes + ((c ^ (r & 15)) << 4); }
template <class T> __device__ __forceinline__ T lds_get(uint32_t a) { return *reinterpret_cast<const __attribute__((address_space(3))) T*>(a); }
template <class T> __device__ __forceinline__ void lds_put(uint32_t a, T x) { *reinterpret_cast<__attribute__((address_space(3))) T*>(a) = x; }
// The lane number computed afresh: addresses made from it are not shared between a kernel's prologue and its epilogue, so
// none of them occupies a register during the walk.
__device__ __forceinline__ int fresh_lane() {
  int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
  asm volatile("" : "+v"(lane));
  return lane;
}
// The rows' loads in flight: 8 instructions of four rows each; `rows` = first row, row_stride in elements.
__device__ __forceinline__ void load_rows(u32x4 (&raw)[8], const bf16* rows, int64_t row_stride) {
  const int lane = fresh_lane();
  const bf16* p = rows + (lane >> 4) * row_stride + (lane & 15) * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i) raw[i] = *reinterpret_cast<const u32x4*>(p + 4 * i * row_stride);
}
// B operands of 32 rows.
template <int kM>
__device__ __forceinline__ void rows_to_frags(bf16x8 (&f)[8], const u32x4 (&raw)[8], uint32_t lds) {
  const int lane = fresh_lane();
#pragma unroll
  for (int i = 0; i < 8; ++i) lds_put(lds + row_slot(4 * i + (lane >> 4), lane & 15), raw[i]);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = lds_get<bf16x8>(lds + row_slot(Mma<kM>::frag_row(lane, i), Mma<kM>::frag_chunk(lane, i)));
}
// buffer_load_dwordx4 ... lds with the LDS destination (wave-uniform) in M0; see dma16_buf.
// M0 is declared clobbered; "memory" is left out on purpose so that LDS reads of the other
// stage may be scheduled across the copy (completion is awaited explicitly at the step's end).
__device__ __forceinline__ void dma16_abs(u32x4 rsrc, uint32_t lds_addr, int voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff) : "m0");
}
__device__ __forceinline__ u32x4 make_rsrc_words(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  u32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}

// Rows that all groups of a workgroup hold as B operands: copied once, straight into LDS in the same layout,
// with wave w taking the fours of rows j with j % 4 == w % 4, whose source chunks then are one offset.  Every wave loading
// its own, 128 KiB a workgroup, made the first loads of dK/dV last 3.4 us.
template <int kRows, int kThreads = 512>
__device__ __forceinline__ void copy_shared_rows(const bf16* rows, int row_stride, uint32_t lds) {
  const int lane = fresh_lane(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = 4 * (w & 3) + (lane >> 4);                  // row within 16
  const int voff = (r * row_stride + ((lane & 15) ^ r) * 8) * 2;
  const u32x4 rsrc = make_rsrc_words(rows, (uint32_t)((kRows - 1) * row_stride + kHeadDim) * 2);
#pragma unroll
  for (int i = 0; i < kRows * 256 / (16 * kThreads); ++i) {
    const int sixteen = kThreads / 256 * i + (w >> 2);
    dma16_abs(rsrc, lds + (4 * sixteen + (w & 3)) * 1024, voff, sixteen * 32 * row_stride);
  }
}
template <int kM>
__device__ __forceinline__ void shared_rows_to_frags(bf16x8 (&f)[8], uint32_t lds, int block) {
  const int lane = fresh_lane();
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = lds_get<bf16x8>(lds + row_slot(32 * block + Mma<kM>::frag_row(lane, i), Mma<kM>::frag_chunk(lane, i)));
}
// Accumulators of 32 rows x 128 columns: acc[m] is block m of 32 columns, transposed (a lane's columns of the block are rows here).  A
// lane's factors of its rows:
struct RowPair { float x[2]; };
__device__ __forceinline__ RowPair both(float x) { return {{x, x}}; }
// The rows times `mul` as bf16.
template <int kM>
__device__ __forceinline__ void store_rows_bf16(bf16* rows, int64_t row_stride, const f32x16 (&acc)[4], RowPair mul, uint32_t lds) {
  using M = Mma<kM>;
  const int lane = fresh_lane();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    bf16x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (bf16)(acc[i >> 2][4 * (i & 3) + j] * mul.x[M::quad_n(i & 3)]);
    lds_put(lds + row_slot(M::col(lane, M::quad_n(i & 3)), 4 * (i >> 2) + M::quad_chunk(lane, i & 3)) + 8 * M::quad_half(lane), w);
  }
  bf16* p = rows + (lane >> 4) * row_stride + (lane & 15) * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    *reinterpret_cast<u32x4*>(p + 4 * i * row_stride) = lds_get<u32x4>(lds + row_slot(4 * i + (lane >> 4), lane & 15));
}
// The same as fp32, half a row at a time.
template <int kM>
__device__ __forceinline__ void store_rows_f32(float* rows, int64_t row_stride, const f32x16 (&acc)[4], RowPair mul, uint32_t lds) {
  using M = Mma<kM>;
  const int lane = fresh_lane();
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x16& a = acc[2 * half + (i >> 2)];
      const int q = 4 * (i & 3);
      const float f = mul.x[M::quad_n(i & 3)];
      lds_put(lds + row_slot(M::col(lane, M::quad_n(i & 3)), 8 * (i >> 2) + M::quad_piece(lane, i & 3)), f32x4{a[q] * f, a[q + 1] * f, a[q + 2] * f, a[q + 3] * f});
    }
    float* p = rows + (lane >> 4) * row_stride + 64 * half + (lane & 15) * 4;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      *reinterpret_cast<f32x4*>(p + 4 * i * row_stride) = lds_get<f32x4>(lds + row_slot(4 * i + (lane >> 4), lane & 15));
  }
}

// What follows serves the walks of several groups a line, which run on 32x32x16: a lane holds one of the 32 rows.
// One block of 32 columns of the same rows (a wave's share after a sum over groups): acc[4g + j] = column
// 8 * g + 4 * (lane / 32) + j of row lane % 32, `rows` already at the block; through 2 or 4 KiB of LDS.
__device__ __forceinline__ void store_block_bf16(bf16* rows, int64_t row_stride, const f32x16& acc, float mul, uint32_t lds) {
  const int lane = fresh_lane(), r = lane & 31;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    bf16x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (bf16)(acc[4 * g + j] * mul);
    lds_put(lds + r * 64 + ((g ^ (r >> 2 & 3)) << 4) + 8 * (lane >> 5), w);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 16 * i + (lane >> 2), c = lane & 3;
    *reinterpret_cast<u32x4*>(rows + row * row_stride + 8 * c) = lds_get<u32x4>(lds + row * 64 + ((c ^ (row >> 2 & 3)) << 4));
  }
}
__device__ __forceinline__ void store_block_f32(float* rows, int64_t row_stride, const f32x16& acc, float mul, uint32_t lds) {
  const int lane = fresh_lane(), r = lane & 31;
#pragma unroll
  for (int g = 0; g < 4; ++g)
    lds_put(lds + r * 128 + (((2 * g + (lane >> 5)) ^ (r >> 1 & 7)) << 4),
            f32x4{acc[4 * g] * mul, acc[4 * g + 1] * mul, acc[4 * g + 2] * mul, acc[4 * g + 3] * mul});
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * i + (lane >> 3), c = lane & 7;
    *reinterpret_cast<f32x4*>(rows + row * row_stride + 4 * c) = lds_get<f32x4>(lds + row * 128 + ((c ^ (row >> 1 & 7)) << 4));
  }
}
// A wave's accumulators in LDS for the waves of the other groups: 16-byte pieces, 1 KiB per instruction; block mb of 32
// columns is the 4 KiB at 4096 * mb.  Block `own` (wave-uniform), which the wave finishes itself, is left out.
constexpr int kAccBytes = 64 * 64 * 4;
__device__ __forceinline__ void put_acc(uint32_t lds, const f32x16 (&acc)[4], int own = -1) {
  lds += 16 * fresh_lane();
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    if (mb == own) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_put(lds + 4096 * mb + 1024 * i, f32x4{acc[mb][4 * i], acc[mb][4 * i + 1], acc[mb][4 * i + 2], acc[mb][4 * i + 3]});
  }
}
// acc = acc * wa + (block mb in LDS) * wb
__device__ __forceinline__ void add_block(uint32_t lds, int mb, f32x16& acc, float wa = 1.f, float wb = 1.f) {
  lds += 16 * fresh_lane() + 4096 * mb;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 x = lds_get<f32x4>(lds + 1024 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[4 * i + j] = acc[4 * i + j] * wa + x[j] * wb;
  }
}
// sum = the groups' blocks `own` in order, times w: this wave's from its accumulators, the other groups' from at(g).
// (Its own block through LDS as well was a fourth of what the four groups' end moves there: 8 heads of 1024, forward
// 12.85 -> 12.75 us, backward 19.8 -> 19.4; 32 of 512, forward 10.2 -> 9.9.)
template <class At>
__device__ __forceinline__ void sum_blocks(f32x16& sum, const f32x16 (&acc)[4], int own, At at, const float (&w)[4]) {
  sum = f32x16{0};
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    if (g != own) add_block(at(g), own, sum, 1.f, w[g]);
    if (g == own) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[i] += acc[g][i] * w[g];
    }
  }
}
// How a workgroup's waves share a line, by kForm:
//   1       one group of four waves, the 128 rows of a tile, both halves of every tile of the other side one after the other;
//   2       two groups of four waves on those rows, each takes a half of every tile (forward);
//   4       four groups of two waves on half a tile's rows (64), each takes a quarter of every tile;
//   kHalves two groups of two waves on half a tile's rows, each takes two quarters one after the other (backward).
// Forms 2 and 4 fill a CU with one workgroup, 1 and kHalves with two.
constexpr int kHalves = 3;
template <int kForm>
struct Groups {
  static constexpr int kCount = kForm == kHalves ? 2 : kForm;  // groups
  static constexpr int kLines = kForm > 2 ? 2 : 1;             // lines per tile
  static constexpr int kWaves = 4 / kLines;                    // of a group
  static constexpr int kRows = 64 / kLines;                    // rows per stage
  static constexpr int kSteps = 2 * kLines / kCount;           // of a group per tile
  static constexpr int kThreads = 64 * kWaves * kCount;
};

// The entries e0 .. e1 - 1 of a workgroup's line: tile | causal flag << 30.  Of a list every wave holds 64 of them, in a register
// or, where none is left, in kBytes of LDS of its own: read one by one through the scalar cache they cost the walks two
// dependent loads per tile (strided 128k, 32 heads, with the copies between the MFMAs: forward 18.3 -> 17.9 ms, dQ 25.6 -> 24.5).
// Entry e of a dense rectangle is tile e itself.
template <bool kDense, bool kInRegister>
struct Walk {
  static constexpr int kBytes = kDense || kInRegister ? 0 : 256;
  int e0, e1, diag, window;
  uint32_t lds;
  __device__ __forceinline__ Walk(int e0_, int e1_, int diag_, uint32_t lds_ = 0) : e0(e0_), e1(e1_), diag(diag_), window(0), lds(lds_) {}
  // Brings entries e .. e + 63 (e < e1).
  __device__ __forceinline__ void fetch(int e, const int32_t* idx, const uint8_t* flag, int n_tiles) {
    if constexpr (!kDense) {
      const int lane = fresh_lane(), i = min(e + lane, e1 - 1);
      window = min(max(idx[i], 0), n_tiles - 1) | ((int)(flag[i] != 0) << 30);
      if constexpr (!kInRegister) lds_put(lds + 4 * lane, window);
    }
  }
  // The first of every 64 entries has to be fetched before it is asked for.
  __device__ __forceinline__ bool has(int e) const { return kDense || ((e - e0) & 63) != 0 || e >= e1; }
  __device__ __forceinline__ int at(int e) const {
    if constexpr (kDense) return e | ((int)(e == diag) << 30);
    if constexpr (kInRegister) return __builtin_amdgcn_readlane(window, (e - e0) & 63);
    return __builtin_amdgcn_readfirstlane(lds_get<int>(lds + 4 * ((e - e0) & 63)));
  }
  static __device__ __forceinline__ int tile(int entry) { return entry & 0x3fffffff; }
};

__device__ __forceinline__ void wait_vmem_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Wave-uniform reads of the (read-only) tile-list arrays through the scalar cache.
__device__ __forceinline__ int32_t sload(const int32_t* p, int i) {
  return ((const __attribute__((address_space(4))) int32_t*)p)[i];
}

// Asynchronous global -> LDS copy (buffer_load_dwordx4 ... lds), 16 bytes per lane: the wave's
// 64 lanes fill 1 KiB starting at the wave-uniform LDS address `lds_dst`, lane l at +16*l.  The
// source address is descriptor base + per-lane byte offset `voff` + wave-uniform byte offset
// `soff`, so a tile's address arithmetic stays on the scalar unit; reads beyond the descriptor's
// extent return 0.  Completion is tracked by vmcnt.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
__device__ __forceinline__ void dma16_buf(__amdgpu_buffer_rsrc_t r, unsigned char* lds_dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds_dst, 16, voff, soff, 0, 0);
}
// Per-thread byte offsets for staging 16 * NW rows of 128 bf16 with NW waves: each thread issues 4
// copies; copy i of wave w fills LDS rows 4*(NW*i + w) .. +3; lane l lands in
// that group's row l/16, physical 16-byte slot l%16, so it must fetch the logical chunk that the
// XOR layout `SLOT` maps to that slot.
template <int (*SLOT)(int, int), int NW>
__device__ __forceinline__ void dma_voffsets(int (&off)[4], int row_stride, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * (NW * i + wave) + (lane >> 4);
    off[i] = (r * row_stride + SLOT(r, lane & 15) * 8) * 2;
  }
}
// The fours of rows at a pitch of kPitch bytes.
template <int NW, int kPitch>
__device__ __forceinline__ void dma_rows_buf(unsigned char* lds, __amdgpu_buffer_rsrc_t r, const int (&voff)[4],
                                                  int soff, int wave) {
#pragma unroll
  for (int i = 0; i < 4; ++i) dma16_buf(r, lds + (NW * i + wave) * kPitch, voff[i], soff);
}

// n / d for 0 <= n < 2^31 as one multiplication: mul = ceil(2^shift / d), shift = 31 + ceil(log2 d), is off by less than d, so that
// n * mul is off by less than 2^shift.  (A workgroup's place takes three to five divisions in a row before its first copy; with
// the divisors' reciprocals formed there, 30 dependent instructions each, it came 0.4 us later: 8 heads of 1024, forward 12.54 -> 12.39 us,
// backward 19.3 -> 19.1; one head of 256 6.24 -> 6.18.)
struct Div { int d; uint32_t mul, shift; };
inline Div make_div(uint32_t d) {
  uint32_t log = 0;
  while ((1u << log) < d) ++log;
  return {(int)d, (uint32_t)(((1ull << (31 + log)) + d - 1) / d), 31 + log};
}
__device__ __forceinline__ int quotient(int n, const Div& by) { return (int)(((uint64_t)(uint32_t)n * by.mul) >> by.shift); }

// blockIdx -> (position in the launch order, batch*head).  Consecutive workgroups go to
// consecutive XCDs.  Each XCD gets its own heads (heads_per_xcd = batch*n_heads/8 when
// divisible, else 0 = plain mapping) and works on them kHeadGroup at a time, so that the
// workgroups resident on an XCD belong to few heads and share K/V (or Q/dO) tiles in its L2.
// Within a head group the heads take turns, position by position: adjacent positions of the launch order (rows with the same
// or nearly the same tile lists) start together and walk their lists in step.  Each head taking four positions at a turn was
// 0.5 to 2 % slower where L2 is short (strided mask: 32k, 16 heads, dK/dV 1633 -> 1598 us; 128k, 32 heads, 33.5 -> 33.2 ms; causal
// 8192, 32 heads, backward 1567 -> 1553 us, 4096 434 -> 421) and the same elsewhere; so are one head at a time 2 to 4 % and four 1 to 2 %.
constexpr int kHeadGroup = 2;
struct BlockMap {
  int own_heads, heads_per_xcd, bid_shift, group_shift;      // own_heads: -1 with whole heads per XCD, else 0 (and so the others)
  Div by;                                                    // workgroups of a head group, or (batch, head) pairs
  int n_blocks;                                              // workgroups of this map
};
inline BlockMap block_map(int nbh, int n_pos) {
  if (nbh % 8) return {0, 0, 0, 0, make_div(nbh), nbh * n_pos};
  const int heads = nbh / 8, shift = heads % kHeadGroup == 0 ? 1 : 0;
  return {-1, heads, 3, shift, make_div((uint32_t)n_pos << shift), nbh * n_pos};
}
// kPairs: positions 2i and 2i + 1 are the halves of one line.  Where no XCD owns whole heads, 16 consecutive workgroups take the first
// halves of eight lines and then the second ones, the last of them of as many lines as are left: both halves, which walk the same
// tiles at the same time, are on one XCD.  On two of them every tile comes from beyond L2 twice (backward, 85 heads of 128 x 256: whole
// lines 13.7 us, halves apart 15.6, together 13.7; 33 of 256: 13.2, 12.4 and 11.1; causal 85 of 256 x 128: 10.7, 11.9 and 10.0).
template <bool kPairs = false>
__device__ __forceinline__ void map_block(int bid, const BlockMap& m, int& pos, int& bh) {
  if (kPairs && !m.own_heads) {
    const int first = 8 * (bid >> 4), r = bid & 15, lines = min(m.n_blocks / 2 - first, 8), half = r >= lines;
    const int line = first + r - half * lines, at = quotient(line, m.by);
    pos = 2 * at + half;
    bh = line - at * m.by.d;
    return;
  }
  const int idx = bid >> m.bid_shift, q = quotient(idx, m.by), r = idx - q * m.by.d;
  const int own_bh = (bid & 7) * m.heads_per_xcd + (q << m.group_shift) + (r & ((1 << m.group_shift) - 1));
  // (without branches, so that all parameters are read at once)
  pos = q ^ ((q ^ (r >> m.group_shift)) & m.own_heads);
  bh = r ^ ((r ^ own_bh) & m.own_heads);
}

inline bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
inline bool strides_ok(const int64_t* s) { return s && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 && s[1] > 0; }

int check_device();   // UA_OK when the current device is gfx950

// ---- dense rectangles: how many parts a walk may be cut into ----------------------------------
// A dense rectangle launches one workgroup per (tile line, head); with few lines and heads the
// device (256 CUs, two resident workgroups each) stays empty while every workgroup walks a long
// list.  The walk may then be cut into parts that run as workgroups of their own and leave partial
// results, combined by a second kernel.  No cut when the launch fills the device anyway or the list
// is short; else at most as many parts as make ~2 workgroups per CU, of at least two tiles each, and
// at most UA_MAX_PARTS.  How many are made is for the estimates of fwd_cut and bwd_plan to choose.
constexpr int kDenseFullLaunch = 384, kDenseTargetGroups = 512;
inline int dense_parts(int64_t n_workgroups, int list_len) {
  if (n_workgroups >= kDenseFullLaunch || list_len < 4) return 1;
  int64_t want = (kDenseTargetGroups + n_workgroups - 1) / n_workgroups;
  if (want > UA_MAX_PARTS) want = UA_MAX_PARTS;
  if (want > list_len / 2) want = list_len / 2;
  return want >= 2 ? (int)want : 1;
}
// Share of a rectangle's tiles that is visible; causal ones are aligned at the bottom right.
inline float visible_share(int n_qtiles, int n_ktiles, bool causal) {
  if (!causal) return 1.f;
  const float q = (float)n_qtiles, k = (float)n_ktiles;
  return q >= k ? (k + 1) / (2 * q) : (k - q + 0.5f * (q + 1)) / k;
}
inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }
struct DenseSplit {     // parts and workspace layout of one dense call (bytes, 256-byte aligned blocks)
  int fwd_parts, dq_parts, dkdv_parts;
  int64_t fwd_o_bytes, fwd_lse_bytes;          // per part
  int64_t dq_bytes, dkdv_bytes;                // per part (dkdv: dK then dV)
  int64_t fwd_total, bwd_total;
};
inline DenseSplit dense_split(int batch, int n_heads, int n_qtiles, int n_ktiles) {
  DenseSplit d;
  const int64_t nbh = (int64_t)batch * n_heads;
  d.fwd_parts = d.dq_parts = dense_parts(nbh * n_qtiles, n_ktiles);
  // Columns count twice: dQ's rows are in the same launch, and from 192 columns on the estimate would take cuts that do not pay
  // (4096 causal queries x 2048 keys, 23 heads, 368 columns: 92 us, cut 117; 16384 x 8192, 3 heads, 192 columns: 610, 642; in
  // 22 other shapes of 192 to 368 columns it takes none and the time is the same).
  d.dkdv_parts = dense_parts(nbh * n_ktiles * 2, n_qtiles);
  const int64_t q_elems = nbh * n_qtiles * kTile * kHeadDim, k_elems = nbh * n_ktiles * kTile * kHeadDim;
  d.fwd_o_bytes = align256(q_elems * 2);
  d.fwd_lse_bytes = align256(nbh * n_qtiles * kTile * 4);
  d.dq_bytes = align256(q_elems * 4);
  d.dkdv_bytes = 2 * align256(k_elems * 4);
  d.fwd_total = d.fwd_parts > 1 ? d.fwd_parts * (d.fwd_o_bytes + d.fwd_lse_bytes) : 0;
  d.bwd_total = (d.dq_parts > 1 ? d.dq_parts * d.dq_bytes : 0) + (d.dkdv_parts > 1 ? d.dkdv_parts * d.dkdv_bytes : 0);
  return d;
}
// Bytes of workspace that a dense backward of this shape uses (0: it is not cut).
int64_t bwd_workspace_used(int batch, int n_heads, int n_qtiles, int n_ktiles, bool causal);
// One sum of fp32 partial results (contiguous [batch, seqlen, n_heads, 128], part i at base + i * stride floats)
// into a strided bf16 tensor; up to three of them run in one launch.
struct PartialSum {
  const float* base; bf16* out;
  int64_t stride;
  int n_parts, seqlen;
  Strides3 os;
};
// Merge of fp32 partials, part i at o_parts + i * o_part and lse_parts + i * lse_part (contiguous [batch, seqlen, n_heads, 128] and
// [batch, n_heads, seqlen]), into the first `seqlen` of `out_seq` tokens of o and lse, which may point into larger tensors.
int merge_f32_rows(const float* o_parts, int64_t o_part, const float* lse_parts, int64_t lse_part, int n_parts, bf16* o, float* lse, int out_seq,
                   int batch, int seqlen, int n_heads, hipStream_t st);
int launch_partial_sums(const PartialSum* sums, int n_sums, int batch, int n_heads, hipStream_t st);

}  // namespace ua
