// Rows without a valid key under Flax's array-mask rule: equal weights over
// every key, so the mean of V (and dV = dO / Lk).  The attention kernels leave
// such rows at zero with lse = +inf.  Nearly every call has none: a workgroup
// reads its rows' lse and ends, about 3 us for both directions together, where
// forming the mean of V and selecting by row cost 5 passes over V and the
// output (bf16 B=2 H=8 L=2048 D=64: about 100 us forward and backward).
#include "pjx_common.h"
#include "pjx_internal.h"

namespace pjx {

template <int DT>  // PJX_DTYPE_*
struct Elem;
template <>
struct Elem<PJX_DTYPE_F32> {
  typedef float T;
  __device__ static float load(const T* p) { return *p; }
  __device__ static void store(T* p, float x) { *p = x; }
};
template <>
struct Elem<PJX_DTYPE_BF16> {
  typedef uint16_t T;
  __device__ static float load(const T* p) { return __uint_as_float((uint32_t)*p << 16); }
  __device__ static void store(T* p, float x) { *p = Bf16Fmt::bits(x); }
};
template <>
struct Elem<PJX_DTYPE_F16> {
  typedef uint16_t T;
  __device__ static float load(const T* p) { return (float)__builtin_bit_cast(_Float16, *p); }
  __device__ static void store(T* p, float x) { *p = F16Fmt::bits(x); }
};

constexpr int kEmptyThreads = 256;

struct EmptyArgs {
  const float* lse;  // [B, Hq, Lq]
  const void* src;   // forward: V [B, Lk, Hkv, D]; backward: dO [B, Lq, Hq, D]
  void* dst;         // forward: O [B, Lq, Hq, D]; backward: dV [B, Lk, Hkv, D]
  int B, Lq, Lk, Hq, Hkv, D;
};

__device__ __forceinline__ bool block_any(bool x) { return __syncthreads_or(x ? 1 : 0) != 0; }

// Sum over n rows p, p + stride, ... of D elements, column tid % D of the rows
// tid / D + i * (threads / D); sums[] receives the D totals.
template <int DT, typename Keep>
__device__ void column_sums(const typename Elem<DT>::T* p, size_t stride, int n, int D, float* sums, float* part,
                            Keep keep) {
  const int per = kEmptyThreads / D, c = threadIdx.x % D, g = threadIdx.x / D;
  float s = 0.f;
  if (g < per)
    for (int i = g; i < n; i += per)
      if (keep(i)) s += Elem<DT>::load(p + (size_t)i * stride + c);
  part[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < D) {
    float t = 0.f;
    for (int i = 0; i < per; ++i) t += part[i * D + threadIdx.x];
    sums[threadIdx.x] = t;
  }
  __syncthreads();
}

// One workgroup per (batch, query head).
template <int DT>
__global__ __launch_bounds__(kEmptyThreads) void fill_empty_rows_kernel(EmptyArgs a) {
  typedef typename Elem<DT>::T T;
  __shared__ float sums[kEmptyThreads], part[kEmptyThreads];
  const int b = blockIdx.x / a.Hq, h = blockIdx.x % a.Hq, hkv = h / (a.Hq / a.Hkv);
  const float* lse = a.lse + (size_t)blockIdx.x * a.Lq;
  bool any = false;
  for (int i = threadIdx.x; i < a.Lq; i += kEmptyThreads) any |= __float_as_uint(lse[i]) == kPosInfBits;
  if (!block_any(any)) return;
  const T* v = (const T*)a.src + ((size_t)b * a.Lk * a.Hkv + hkv) * a.D;
  column_sums<DT>(v, (size_t)a.Hkv * a.D, a.Lk, a.D, sums, part, [](int) { return true; });
  const float inv = 1.f / a.Lk;
  T* o = (T*)a.dst + ((size_t)b * a.Lq * a.Hq + h) * a.D;
  for (int i = threadIdx.x / a.D; i < a.Lq; i += kEmptyThreads / a.D) {
    if ((int)threadIdx.x / a.D >= kEmptyThreads / a.D || __float_as_uint(lse[i]) != kPosInfBits) continue;
    Elem<DT>::store(o + (size_t)i * a.Hq * a.D + threadIdx.x % a.D, sums[threadIdx.x % a.D] * inv);
  }
}

// One workgroup per (batch, KV head): dV of every key gains the sum over the
// group's empty rows of dO, divided by the number of keys.
template <int DT>
__global__ __launch_bounds__(kEmptyThreads) void empty_rows_grad_kernel(EmptyArgs a) {
  typedef typename Elem<DT>::T T;
  __shared__ float sums[kEmptyThreads], part[kEmptyThreads], total[kEmptyThreads];
  const int b = blockIdx.x / a.Hkv, hkv = blockIdx.x % a.Hkv, G = a.Hq / a.Hkv;
  const float* lse = a.lse + ((size_t)b * a.Hq + (size_t)hkv * G) * a.Lq;
  bool any = false;
  for (long i = threadIdx.x; i < (long)G * a.Lq; i += kEmptyThreads) any |= __float_as_uint(lse[i]) == kPosInfBits;
  if (!block_any(any)) return;
  total[threadIdx.x] = 0.f;
  for (int g = 0; g < G; ++g) {
    const T* d = (const T*)a.src + ((size_t)b * a.Lq * a.Hq + hkv * G + g) * a.D;
    const float* l = lse + (size_t)g * a.Lq;
    column_sums<DT>(d, (size_t)a.Hq * a.D, a.Lq, a.D, sums, part,
                    [&](int i) { return __float_as_uint(l[i]) == kPosInfBits; });
    if ((int)threadIdx.x < a.D) total[threadIdx.x] += sums[threadIdx.x];
  }
  __syncthreads();
  const float inv = 1.f / a.Lk;
  T* dv = (T*)a.dst + ((size_t)b * a.Lk * a.Hkv + hkv) * a.D;
  const int c = threadIdx.x % a.D;
  for (int i = threadIdx.x / a.D; i < a.Lk; i += kEmptyThreads / a.D) {
    if ((int)threadIdx.x / a.D >= kEmptyThreads / a.D) break;
    T* p = dv + (size_t)i * a.Hkv * a.D + c;
    Elem<DT>::store(p, fmaf(total[c], inv, Elem<DT>::load(p)));
  }
}

// The output and dO as the backward kernels see them: copies with zeros in such
// rows, blockIdx.z 0 and 1.  One pass over memory, 16 bytes a lane (a row of any
// kernel's head dim is whole 16-byte chunks), indexed in 32 bits within a batch
// entry.  A step over 2x2048x8x64 in bf16 with a learned bias: 350 us with torch
// operations (compare, two selects by row) here, 319 with this kernel.
struct ZeroArgs {
  const float* lse;     // [B, Hq, Lq]
  const u32x4* src[2];  // [B, Lq, Hq, per]
  u32x4* dst[2];
  int B, Lq, Hq, per;
};

__global__ __launch_bounds__(kEmptyThreads) void zero_empty_rows_kernel(ZeroArgs a) {
  const uint32_t e = blockIdx.x * (uint32_t)kEmptyThreads + threadIdx.x;
  const uint32_t n = (uint32_t)a.Lq * a.Hq * a.per;
  if (e >= n) return;
  const uint32_t row = e / a.per, t = row / a.Hq, h = row % a.Hq;
  for (int b = blockIdx.y; b < a.B; b += gridDim.y) {
    u32x4 x = a.src[blockIdx.z][(size_t)b * n + e];
    if (__float_as_uint(a.lse[((size_t)b * a.Hq + h) * a.Lq + t]) == kPosInfBits) x = u32x4{0u, 0u, 0u, 0u};
    a.dst[blockIdx.z][(size_t)b * n + e] = x;
  }
}

template <int DT>
static int launch_empty(const EmptyArgs& a, bool grad, hipStream_t s) {
  if (grad)
    launch_kernel<empty_rows_grad_kernel<DT>>(dim3((unsigned)(a.B * a.Hkv)), dim3(kEmptyThreads), 0, s, a);
  else
    launch_kernel<fill_empty_rows_kernel<DT>>(dim3((unsigned)(a.B * a.Hq)), dim3(kEmptyThreads), 0, s, a);
  return check_launch("pjx_empty_rows");
}

}  // namespace pjx

using namespace pjx;

extern "C" int pjx_empty_rows(int dtype, int grad, const float* lse, const void* src, void* dst, int64_t batch,
                              int64_t q_len, int64_t kv_len, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                              void* stream) {
  clear_error();
  if (dtype != PJX_DTYPE_BF16 && dtype != PJX_DTYPE_F16 && dtype != PJX_DTYPE_F32)
    return fail(PJX_ERR_INVALID, "pjx_empty_rows: dtype must be PJX_DTYPE_BF16, PJX_DTYPE_F16 or PJX_DTYPE_F32");
  if (batch < 0 || q_len < 0 || kv_len < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || head_dim <= 0 ||
      head_dim > kEmptyThreads || q_len > (1 << 30) || kv_len > (1 << 30) || batch * q_heads > 0x7fffffffL)
    return fail(PJX_ERR_INVALID, "pjx_empty_rows: sizes out of range");
  if (batch == 0 || q_len == 0 || kv_len == 0) return PJX_OK;
  if (!lse || !src || !dst) return fail(PJX_ERR_INVALID, "pjx_empty_rows: pointers must be non-null");
  const EmptyArgs a = {lse, src, dst, (int)batch, (int)q_len, (int)kv_len, (int)q_heads, (int)kv_heads, (int)head_dim};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == PJX_DTYPE_F32) return launch_empty<PJX_DTYPE_F32>(a, grad != 0, s);
  return dtype == PJX_DTYPE_F16 ? launch_empty<PJX_DTYPE_F16>(a, grad != 0, s)
                                : launch_empty<PJX_DTYPE_BF16>(a, grad != 0, s);
}

extern "C" int pjx_zero_empty_rows(int dtype, const float* lse, const void* o, const void* dout, void* o_rows,
                                   void* dout_rows, int64_t batch, int64_t q_len, int64_t q_heads, int64_t head_dim,
                                   void* stream) {
  clear_error();
  if (dtype != PJX_DTYPE_BF16 && dtype != PJX_DTYPE_F16 && dtype != PJX_DTYPE_F32)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: dtype must be PJX_DTYPE_BF16, PJX_DTYPE_F16 or PJX_DTYPE_F32");
  const int64_t row_bytes = head_dim * (dtype == PJX_DTYPE_F32 ? 4 : 2), per = row_bytes / 16;
  // the chunks of a batch entry, and the last block's threads, count in 32 bits
  if (batch < 0 || batch > 0x7fffffffL || q_len < 0 || q_len > (1 << 30) || q_heads <= 0 || q_heads > (1 << 30) ||
      head_dim <= 0 || head_dim > kEmptyThreads || row_bytes % 16 || q_len * q_heads > (int64_t)0xffff0000 / per)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: sizes out of range, or rows that are no whole 16-byte chunks");
  if (batch == 0 || q_len == 0) return PJX_OK;
  if (!lse || !o || !dout || !o_rows || !dout_rows)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: pointers must be non-null");
  if (((uintptr_t)o | (uintptr_t)dout | (uintptr_t)o_rows | (uintptr_t)dout_rows) % 16)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: tensors must start on 16 bytes");
  const ZeroArgs a = {lse, {(const u32x4*)o, (const u32x4*)dout}, {(u32x4*)o_rows, (u32x4*)dout_rows},
                      (int)batch, (int)q_len, (int)q_heads, (int)per};
  const dim3 grid((unsigned)((q_len * q_heads * per + kEmptyThreads - 1) / kEmptyThreads),
                  (unsigned)std::min<int64_t>(batch, 65535), 2);
  launch_kernel<zero_empty_rows_kernel>(grid, dim3(kEmptyThreads), 0, (hipStream_t)stream, a);
  return check_launch("pjx_zero_empty_rows");
}
