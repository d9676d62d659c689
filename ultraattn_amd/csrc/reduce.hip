// Gradient reductions across partial results: HBM-bandwidth bound streaming kernels.
//
//  grad_accumulate_kernel : one step of a running fp32 sum, acc += partial, with the bf16 rounding
//                           of the sum written in the same pass (the accumulation of
//                           ring_flash_attn/ring_flash_attn.py:110-118: partial gradients are added
//                           into fp32 buffers and cast once).
//  grad_sum_kernel        : out = bf16(scale * sum_p part_p) over n_parts partial gradients, fp32 or
//                           bf16, in one pass; the output may be strided by (batch, token, head).
#include <algorithm>
#include "ua_common.h"

namespace ua {

constexpr int kRedThreads = 256;
constexpr int kRedBlocks = 8192;         // grid cap of the sum: 32 workgroups per CU, grid-stride beyond

__device__ __forceinline__ void unpack8(const u32x4 r, float (&x)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) { x[2 * j] = __uint_as_float(r[j] << 16); x[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u); }
}
__device__ __forceinline__ bf16x8 pack8(const float (&x)[8]) {
  bf16x8 w;
#pragma unroll
  for (int j = 0; j < 8; ++j) w[j] = (bf16)x[j];
  return w;
}

// mode 0: acc += partial, out = bf16(acc) when out != NULL
// mode 1: acc  = float(out) + partial, out = bf16(acc)          (first step of a chain)
// mode 2: out  = bf16(float(out) + partial)                     (no fp32 accumulator)
// kSmall: what fits the 32 MiB of L2 (the sum, read again by the next step, and the partial, just written).  One chunk of 8 elements
// per thread gives every CU work, and nothing streams past the caches: 8 heads x 1024 tokens 3.03 -> 2.55 us, 32 x 512 4.0 -> 3.8.  A
// larger sum takes four per thread, every load issued before the first use, and non-temporal accesses: with plain ones 32 x 2304 alone
// takes 17.7 us, so 21.7, but the kernels around it lose as much (a rectangle of 2304 x 3456, forward and backward, 620 us and 621).
template <int kMode, bool kSmall>
__global__ __launch_bounds__(kRedThreads) void grad_accumulate_kernel(float* acc, const bf16* partial, bf16* out, int64_t n_chunks) {
  constexpr int kVec = kSmall ? 1 : 4;
  auto load = [](const auto* p) { return kSmall ? *p : __builtin_nontemporal_load(p); };
  auto store = [](auto x, auto* p) { if (kSmall) *p = x; else __builtin_nontemporal_store(x, p); };
  const int64_t stride = (int64_t)gridDim.x * kRedThreads * kVec;
  for (int64_t c0 = (int64_t)blockIdx.x * kRedThreads * kVec + threadIdx.x; c0 < n_chunks; c0 += stride) {
    u32x4 py[kVec], po[kVec];
    f32x4 a0[kVec], a1[kVec];
#pragma unroll
    for (int u = 0; u < kVec; ++u) {
      const int64_t c = c0 + u * kRedThreads;
      if (c >= n_chunks) break;
      py[u] = load(reinterpret_cast<const u32x4*>(partial) + c);
      if (kMode == 0) {
        a0[u] = load(reinterpret_cast<const f32x4*>(acc) + 2 * c);
        a1[u] = load(reinterpret_cast<const f32x4*>(acc) + 2 * c + 1);
      } else {
        po[u] = load(reinterpret_cast<const u32x4*>(out) + c);
      }
    }
#pragma unroll
    for (int u = 0; u < kVec; ++u) {
      const int64_t c = c0 + u * kRedThreads;
      if (c >= n_chunks) break;
      float x[8], y[8];
      unpack8(py[u], y);
      if (kMode == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { x[j] = a0[u][j]; x[4 + j] = a1[u][j]; }
      } else {
        unpack8(po[u], x);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] += y[j];
      if (kMode != 2) {
        store(f32x4{x[0], x[1], x[2], x[3]}, reinterpret_cast<f32x4*>(acc) + 2 * c);
        store(f32x4{x[4], x[5], x[6], x[7]}, reinterpret_cast<f32x4*>(acc) + 2 * c + 1);
      }
      if (out) store(pack8(x), reinterpret_cast<bf16x8*>(out) + c);
    }
  }
}

struct SumParams {
  const void* parts[UA_MAX_PARTS];
  bf16* out;
  int n_parts, seqlen, n_heads;
  Strides3 os;
  float scale;
  int64_t n_chunks;        // batch * seqlen * n_heads * 16
};

template <bool kF32>
__global__ __launch_bounds__(kRedThreads) void grad_sum_kernel(const SumParams p) {
  for (int64_t c = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; c < p.n_chunks; c += (int64_t)gridDim.x * kRedThreads) {
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = 0.f;
    for (int i = 0; i < p.n_parts; ++i) {
      if (kF32) {
        const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.parts[i]) + 2 * c);
        const f32x4 b = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.parts[i]) + 2 * c + 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) { x[j] += a[j]; x[4 + j] += b[j]; }
      } else {
        float y[8];
        unpack8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.parts[i]) + c), y);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] += y[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] *= p.scale;
    const int64_t row = c >> 4;
    const int h = (int)(row % p.n_heads);
    const int64_t t = row / p.n_heads;
    const int64_t s = t % p.seqlen, b = t / p.seqlen;
    *reinterpret_cast<bf16x8*>(p.out + b * p.os.b + s * p.os.s + h * p.os.h + (c & 15) * 8) = pack8(x);
  }
}

// The partial results of one split backward, summed in one launch: the workgroups of sum j follow those of sum
// j - 1.  The partials were just written and are read from L2; what bounds it at the sizes that split (a few
// MB) is the latency of one launch and of one round of loads, so all loads of a chunk are issued together.
struct PartialSumsParams {
  PartialSum s[3];
  int first_block[4];
  int batch, n_heads;
  Div by_heads, by_seq[3];
};
__global__ __launch_bounds__(kRedThreads) void partial_sums_kernel(const PartialSumsParams p) {
  const int j = (int)blockIdx.x >= p.first_block[2] ? 2 : ((int)blockIdx.x >= p.first_block[1] ? 1 : 0);
  const PartialSum& s = p.s[j];
  const int64_t c = (int64_t)(blockIdx.x - p.first_block[j]) * kRedThreads + threadIdx.x;
  const int row = (int)(c >> 4);
  if (row >= p.batch * s.seqlen * p.n_heads) return;
  const float* src = s.base + c * 8;
  f32x4 x0{0}, x1{0};
  for (int i0 = 0; i0 < s.n_parts; i0 += 8) {
    f32x4 a[8], b[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < s.n_parts) {
        a[u] = *reinterpret_cast<const f32x4*>(src + (i0 + u) * s.stride);
        b[u] = *reinterpret_cast<const f32x4*>(src + (i0 + u) * s.stride + 4);
      }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u < s.n_parts) { x0 += a[u]; x1 += b[u]; }
  }
  const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
  const int t = quotient(row, p.by_heads), h = row - t * p.n_heads, b = quotient(t, p.by_seq[j]), tok = t - b * s.seqlen;
  *reinterpret_cast<bf16x8*>(s.out + b * s.os.b + tok * s.os.s + h * s.os.h + (c & 15) * 8) = pack8(x);
}

int launch_partial_sums(const PartialSum* sums, int n_sums, int batch, int n_heads, hipStream_t st) {
  PartialSumsParams p{};
  p.batch = batch; p.n_heads = n_heads;
  p.by_heads = make_div(n_heads);
  for (int j = 0; j < 3; ++j) {
    p.first_block[j + 1] = p.first_block[j];
    if (j >= n_sums) continue;
    p.s[j] = sums[j];
    p.by_seq[j] = make_div(sums[j].seqlen);
    p.first_block[j + 1] += (int)(((int64_t)batch * sums[j].seqlen * n_heads * 16 + kRedThreads - 1) / kRedThreads);
  }
  hipLaunchKernelGGL(partial_sums_kernel, dim3(p.first_block[3]), dim3(kRedThreads), 0, st, p);
  return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
}

}  // namespace ua

extern "C" int ua_grad_accumulate(float* acc, const void* partial, void* out, int64_t n, int init_from_out, void* stream) {
  using namespace ua;
  if (!partial || (!acc && !out) || (init_from_out && (!acc || !out))) return UA_ERR_NULL;
  if (n <= 0) return UA_ERR_SHAPE;
  if (n % 8 != 0 || !aligned16(partial) || (acc && !aligned16(acc)) || (out && !aligned16(out))) return UA_ERR_ALIGN;
  if (int rc = check_device()) return rc;
  const int64_t n_chunks = n / 8;
  const bool small = n_chunks * 48 <= (24 << 20);
  const int per_block = (small ? 1 : 4) * kRedThreads, blocks = (int)std::min<int64_t>((n_chunks + per_block - 1) / per_block, 4 * kRedBlocks);
  const int mode = !acc ? 2 : init_from_out ? 1 : 0;
  const auto kernel = mode == 2 ? (small ? grad_accumulate_kernel<2, true> : grad_accumulate_kernel<2, false>)
                    : mode == 1 ? (small ? grad_accumulate_kernel<1, true> : grad_accumulate_kernel<1, false>)
                                : (small ? grad_accumulate_kernel<0, true> : grad_accumulate_kernel<0, false>);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kRedThreads), 0, (hipStream_t)stream, acc, (const bf16*)partial, (bf16*)out, n_chunks);
  return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
}

extern "C" int ua_grad_sum(const void* const* parts, int n_parts, int parts_fp32, void* out,
                           int batch, int seqlen, int n_heads, int head_dim, const int64_t* out_strides,
                           float scale, void* stream) {
  using namespace ua;
  if (!parts || !out || !out_strides) return UA_ERR_NULL;
  if (n_parts < 1 || n_parts > UA_MAX_PARTS || head_dim != kHeadDim) return UA_ERR_UNSUPPORTED;
  if (batch <= 0 || seqlen <= 0 || n_heads <= 0) return UA_ERR_SHAPE;
  if (!aligned16(out) || !strides_ok(out_strides)) return UA_ERR_ALIGN;
  for (int i = 0; i < n_parts; ++i) {
    if (!parts[i]) return UA_ERR_NULL;
    if (!aligned16(parts[i])) return UA_ERR_ALIGN;
  }
  if (int rc = check_device()) return rc;
  SumParams p;
  for (int i = 0; i < UA_MAX_PARTS; ++i) p.parts[i] = i < n_parts ? parts[i] : nullptr;
  p.out = (bf16*)out; p.n_parts = n_parts; p.seqlen = seqlen; p.n_heads = n_heads;
  p.os = {out_strides[0], out_strides[1], out_strides[2]};
  p.scale = scale;
  p.n_chunks = (int64_t)batch * seqlen * n_heads * 16;
  const int blocks = (int)std::min<int64_t>((p.n_chunks + kRedThreads - 1) / kRedThreads, kRedBlocks);
  hipStream_t st = (hipStream_t)stream;
  if (parts_fp32) hipLaunchKernelGGL(grad_sum_kernel<true>, dim3(blocks), dim3(kRedThreads), 0, st, p);
  else            hipLaunchKernelGGL(grad_sum_kernel<false>, dim3(blocks), dim3(kRedThreads), 0, st, p);
  return hipGetLastError() == hipSuccess ? UA_OK : UA_ERR_LAUNCH;
}
