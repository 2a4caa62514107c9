// Rows without a valid key under Flax's array-mask rule: equal weights over
// every key, so the mean of V (and dV = dO / Lk).  The attention kernels leave
// such rows at zero with lse = +inf.
#include "pjx_common.h"
#include "pjx_internal.h"

namespace pjx {

// VE consecutive elements as floats: 16 bytes, or one element where rows are no
// whole 16-byte chunks.
template <int DT, int VE>
struct Elems;
template <>
struct Elems<PJX_DTYPE_F32, 4> {
  typedef float T;
  __device__ static void load(const T* p, float* x) { *(f32x4*)x = *(const f32x4*)p; }
  __device__ static void store(T* p, const float* x) { *(f32x4*)p = *(const f32x4*)x; }
};
template <>
struct Elems<PJX_DTYPE_F32, 1> {
  typedef float T;
  __device__ static void load(const T* p, float* x) { *x = *p; }
  __device__ static void store(T* p, const float* x) { *p = *x; }
};
template <typename F, int VE>
struct HalfElems {
  typedef uint16_t T;
  __device__ static void load(const T* p, float* x) {
    if constexpr (VE == 8) {
      const u32x4 r = *(const u32x4*)p;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[2 * j] = F::lo(r[j]);
        x[2 * j + 1] = F::hi(r[j]);
      }
    } else {
      *x = F::lo(*p);
    }
  }
  __device__ static void store(T* p, const float* x) {
    if constexpr (VE == 8) {
      u32x4 r;
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j] = F::pack2(x[2 * j], x[2 * j + 1]);
      *(u32x4*)p = r;
    } else {
      *p = F::bits(*x);
    }
  }
};
template <int VE>
struct Elems<PJX_DTYPE_BF16, VE> : HalfElems<Bf16Fmt, VE> {};
template <int VE>
struct Elems<PJX_DTYPE_F16, VE> : HalfElems<F16Fmt, VE> {};

constexpr int kEmptyThreads = 512, kEmptyWaves = kEmptyThreads / 64;
constexpr int kMaxEmptyDim = 256;
constexpr int kZeroThreads = 256;

struct EmptyArgs {
  const float* lse;  // [B, Hq, Lq]
  const void* src;   // forward: V [B, Lk, Hkv, D]; backward: dO [B, Lq, Hq, D]
  void* dst;         // forward: O [B, Lq, Hq, D]; backward: dV [B, Lk, Hkv, D]
  int B, Lq, Lk, Hq, Hkv, D;
  int chunk;         // rows of dst per workgroup
  int heads;         // (batch, head) pairs: B * Hq, or B * Hkv for the gradient
};

// A workgroup's columns: 64 bytes of a row in lanes of 16, or 64 single
// elements; the lanes past the row's end idle.
template <int VE>
struct Columns {
  static constexpr int LPR = VE > 1 ? 4 : 64;  // lanes per row
  static constexpr int N = LPR * VE;
  static constexpr int ROWS = kEmptyThreads / LPR;
};

// Adds the lanes' sums of one column over the workgroup, in a fixed order;
// sums[] receives the N totals.
template <int VE>
__device__ __forceinline__ void add_columns(float* acc, float (*part)[Columns<VE>::N], float* sums) {
  using C = Columns<VE>;
#pragma unroll
  for (int m = C::LPR; m < 64; m <<= 1)
#pragma unroll
    for (int e = 0; e < VE; ++e) acc[e] += __shfl_xor(acc[e], m, 64);
  if ((threadIdx.x & 63) < C::LPR)
#pragma unroll
    for (int e = 0; e < VE; ++e) part[threadIdx.x >> 6][(threadIdx.x & 63) * VE + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < C::N) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kEmptyWaves; ++w) t += part[w][threadIdx.x];
    sums[threadIdx.x] = t;
  }
  __syncthreads();
}

// Whether any of n lse values is +inf, as far as this thread looks: all of the
// workgroup's threads together look at each once.
__device__ __forceinline__ bool any_empty(const float* lse, long n) {
  bool any = false;
  long done = 0;
  if ((uintptr_t)lse % 16 == 0) {
    done = n / 4 * 4;
#pragma unroll 8
    for (long i = 4 * threadIdx.x; i < done; i += 4 * kEmptyThreads) {
      const u32x4 x = *(const u32x4*)(lse + i);
      any |= x[0] == kPosInfBits || x[1] == kPosInfBits || x[2] == kPosInfBits || x[3] == kPosInfBits;
    }
  }
  for (long i = done + threadIdx.x; i < n; i += kEmptyThreads) any |= __float_as_uint(lse[i]) == kPosInfBits;
  return any;
}

// Both kernels: one workgroup per (batch and head, chunk of the rows written,
// 64-byte column group), more heads than a launch's work-items count taken in
// strides of the grid.  Without an empty row they end after reading the lse,
// the usual call.  A batch padded on the query side has such rows in every
// call; then each workgroup sums its columns of V (of the empty rows' dO)
// itself, from L2 for all but the first, which needs no workspace and no second
// launch, and the chunks and column groups fill the device.
// us with none / a tenth / all of the rows empty, one workgroup of 256 threads
// and 2-byte loads per (batch, head) before -> now:
//   bf16 B=2 L=2048 H=8 D=64:          fill 2.6 / 110 / 138 -> 2.2 / 5.9 / 8.0
//                                      gradient 2.6 / 125 / 180 -> 2.7 / 7.7 / 9.8
//   bf16 B=1 L=4096 H=32 Hkv=1 D=128:  fill 3.5 / 418 / 791 -> 2.3 / 9.3 / 16.5
//                                      gradient 57 / 8910 / 33306 -> 6.4 / 148 / 478
// (Calls after one another; between a training step's other kernels the first
// shape's 2.2 and 2.7 without an empty row are 3.9 and 4.6.)
template <int DT, int VE>
__global__ __launch_bounds__(kEmptyThreads) void fill_empty_rows_kernel(EmptyArgs a) {
  typedef Elems<DT, VE> E;
  using C = Columns<VE>;
  __shared__ float sums[C::N], part[kEmptyWaves][C::N];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.y * a.chunk, r1 = min(r0 + a.chunk, a.Lq);
  const int c = blockIdx.z * C::N + (tid % C::LPR) * VE;
  const bool in = c < a.D;
  const size_t vs = (size_t)a.Hkv * a.D, os = (size_t)a.Hq * a.D;
  for (uint32_t bh = blockIdx.x; bh < (uint32_t)a.heads; bh += gridDim.x) {
    const int b = bh / a.Hq, h = bh % a.Hq, hkv = h / (a.Hq / a.Hkv);
    const float* lse = a.lse + (size_t)bh * a.Lq;
    if (!__syncthreads_or(any_empty(lse + r0, r1 - r0) ? 1 : 0)) continue;
    const typename E::T* v = (const typename E::T*)a.src + (size_t)b * a.Lk * vs + (size_t)hkv * a.D + c;
    float acc[VE] = {};
    if (in) {
#pragma unroll 8
      for (int i = tid / C::LPR; i < a.Lk; i += C::ROWS) {
        float x[VE];
        E::load(v + i * vs, x);
#pragma unroll
        for (int e = 0; e < VE; ++e) acc[e] += x[e];
      }
    }
    add_columns<VE>(acc, part, sums);
    if (!in) continue;
    const float inv = 1.f / a.Lk;
    float mean[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) mean[e] = sums[(tid % C::LPR) * VE + e] * inv;
    typename E::T* o = (typename E::T*)a.dst + (size_t)b * a.Lq * os + (size_t)h * a.D + c;
    for (int i = r0 + tid / C::LPR; i < r1; i += C::ROWS)
      if (__float_as_uint(lse[i]) == kPosInfBits) E::store(o + i * os, mean);
  }
}

// dV of every key gains the sum over the group's empty rows of dO, divided by
// the number of keys.  A wave looks at 256 rows' lse at a time and lists the
// empty ones in LDS, so only their dO is read.
template <int DT, int VE>
__global__ __launch_bounds__(kEmptyThreads) void empty_rows_grad_kernel(EmptyArgs a) {
  typedef Elems<DT, VE> E;
  using C = Columns<VE>;
  __shared__ float sums[C::N], part[kEmptyWaves][C::N];
  __shared__ int rows[kEmptyWaves][64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int G = a.Hq / a.Hkv;
  const long n = (long)G * a.Lq;  // the group's rows, one after the other in the lse
  const int c = blockIdx.z * C::N + (tid % C::LPR) * VE;
  const bool in = c < a.D;
  const size_t vs = (size_t)a.Hkv * a.D, ds = (size_t)a.Hq * a.D;
  for (uint32_t bh = blockIdx.x; bh < (uint32_t)a.heads; bh += gridDim.x) {
    const int b = bh / a.Hkv, hkv = bh % a.Hkv;
    const float* lse = a.lse + ((size_t)b * a.Hq + (size_t)hkv * G) * a.Lq;
    const typename E::T* d = (const typename E::T*)a.src + (size_t)b * a.Lq * ds + (size_t)hkv * G * a.D + c;
    if (!__syncthreads_or(any_empty(lse, n) ? 1 : 0)) continue;
    float acc[VE] = {};
    const int per_head = (a.Lq + 255) / 256;  // blocks of 256 rows of one head
    for (int t = w; t < G * per_head; t += kEmptyWaves) {
      const int g = t / per_head, i0 = t % per_head * 256;
      bool empty[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + 64 * j + lane;
        empty[j] = i < a.Lq && __float_as_uint(lse[(size_t)g * a.Lq + i]) == kPosInfBits;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint64_t m = __builtin_amdgcn_ballot_w64(empty[j]);
        if (m == 0) continue;
        if (empty[j]) rows[w][__builtin_popcountll(m & ((1ull << lane) - 1))] = i0 + 64 * j + lane;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int count = __builtin_popcountll(m);
#pragma unroll 4
        for (int k = lane / C::LPR; k < count; k += 64 / C::LPR) {
          float x[VE];
          if (in) {
            E::load(d + rows[w][k] * ds + (size_t)g * a.D, x);
#pragma unroll
            for (int e = 0; e < VE; ++e) acc[e] += x[e];
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    add_columns<VE>(acc, part, sums);
    if (!in) continue;
    const float inv = 1.f / a.Lk;
    float total[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) total[e] = sums[(tid % C::LPR) * VE + e];
    typename E::T* dv = (typename E::T*)a.dst + (size_t)b * a.Lk * vs + (size_t)hkv * a.D + c;
    const int r1 = min((int)(blockIdx.y + 1) * a.chunk, a.Lk);
    for (int i = blockIdx.y * a.chunk + tid / C::LPR; i < r1; i += C::ROWS) {
      float x[VE];
      E::load(dv + i * vs, x);
#pragma unroll
      for (int e = 0; e < VE; ++e) x[e] = fmaf(total[e], inv, x[e]);
      E::store(dv + i * vs, x);
    }
  }
}

// The output and dO as the backward kernels see them: copies with zeros in such
// rows, blockIdx.z 0 and 1.  One pass over memory, 16 bytes a lane (a row of any
// kernel's head dim is whole 16-byte chunks), indexed in 32 bits within a batch
// entry.  A step over 2x2048x8x64 in bf16 with a learned bias: 350 us with torch
// operations (compare, two selects by row) here, 319 with this kernel.  The
// copies are made in every backward after a fill, whether or not such a row
// exists: 5.4 us of that step.
struct ZeroArgs {
  const float* lse;     // [B, Hq, Lq]
  const u32x4* src[2];  // [B, Lq, Hq, per]
  u32x4* dst[2];
  int B, Lq, Hq, per;
};

__global__ __launch_bounds__(kZeroThreads) void zero_empty_rows_kernel(ZeroArgs a) {
  const uint32_t e = blockIdx.x * (uint32_t)kZeroThreads + threadIdx.x;
  const uint32_t n = (uint32_t)a.Lq * a.Hq * a.per;
  if (e >= n) return;
  const uint32_t row = e / a.per, t = row / a.Hq, h = row % a.Hq;
  for (int b = blockIdx.y; b < a.B; b += gridDim.y) {
    u32x4 x = a.src[blockIdx.z][(size_t)b * n + e];
    if (__float_as_uint(a.lse[((size_t)b * a.Hq + h) * a.Lq + t]) == kPosInfBits) x = u32x4{0u, 0u, 0u, 0u};
    a.dst[blockIdx.z][(size_t)b * n + e] = x;
  }
}

// Chunks of at least 64 rows, as many as give the device about two workgroups a CU.
template <int DT, int VE>
static int launch_empty(EmptyArgs a, bool grad, hipStream_t s) {
  const int64_t heads = (int64_t)a.B * (grad ? a.Hkv : a.Hq), rows = grad ? a.Lk : a.Lq;
  const int groups = (a.D + Columns<VE>::N - 1) / Columns<VE>::N;
  const int64_t chunks = std::min(std::max<int64_t>(512 / (heads * groups), 1), (rows + 63) / 64);
  a.chunk = (int)((rows + chunks - 1) / chunks);
  a.heads = (int)heads;
  const dim3 grid((unsigned)std::min<int64_t>(heads, 0xffffffffLL / kEmptyThreads),
                  (unsigned)((rows + a.chunk - 1) / a.chunk), groups), block(kEmptyThreads);
  if (grad)
    launch_kernel<empty_rows_grad_kernel<DT, VE>>(grid, block, 0, s, a);
  else
    launch_kernel<fill_empty_rows_kernel<DT, VE>>(grid, block, 0, s, a);
  return check_launch("pjx_empty_rows");
}

template <int DT, int VE>
static int launch_empty_rows(const EmptyArgs& a, bool grad, hipStream_t s) {
  const bool vec = a.D % VE == 0 && ((uintptr_t)a.src | (uintptr_t)a.dst) % 16 == 0;
  return vec ? launch_empty<DT, VE>(a, grad, s) : launch_empty<DT, 1>(a, grad, s);
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
      head_dim > kMaxEmptyDim || q_len > (1 << 30) || kv_len > (1 << 30) || batch * q_heads > 0x7fffffffL)
    return fail(PJX_ERR_INVALID, "pjx_empty_rows: sizes out of range");
  if (batch == 0 || q_len == 0 || kv_len == 0) return PJX_OK;
  if (!lse || !src || !dst) return fail(PJX_ERR_INVALID, "pjx_empty_rows: pointers must be non-null");
  const EmptyArgs a = {lse, src, dst, (int)batch, (int)q_len, (int)kv_len, (int)q_heads, (int)kv_heads, (int)head_dim, 0, 0};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == PJX_DTYPE_F32) return launch_empty_rows<PJX_DTYPE_F32, 4>(a, grad != 0, s);
  return dtype == PJX_DTYPE_F16 ? launch_empty_rows<PJX_DTYPE_F16, 8>(a, grad != 0, s)
                                : launch_empty_rows<PJX_DTYPE_BF16, 8>(a, grad != 0, s);
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
      head_dim <= 0 || head_dim > kMaxEmptyDim || row_bytes % 16 || q_len * q_heads > (int64_t)0xffff0000 / per)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: sizes out of range, or rows that are no whole 16-byte chunks");
  if (batch == 0 || q_len == 0) return PJX_OK;
  if (!lse || !o || !dout || !o_rows || !dout_rows)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: pointers must be non-null");
  if (((uintptr_t)o | (uintptr_t)dout | (uintptr_t)o_rows | (uintptr_t)dout_rows) % 16)
    return fail(PJX_ERR_INVALID, "pjx_zero_empty_rows: tensors must start on 16 bytes");
  const ZeroArgs a = {lse, {(const u32x4*)o, (const u32x4*)dout}, {(u32x4*)o_rows, (u32x4*)dout_rows},
                      (int)batch, (int)q_len, (int)q_heads, (int)per};
  const dim3 grid((unsigned)((q_len * q_heads * per + kZeroThreads - 1) / kZeroThreads),
                  (unsigned)std::min<int64_t>(batch, 65535), 2);
  launch_kernel<zero_empty_rows_kernel>(grid, dim3(kZeroThreads), 0, (hipStream_t)stream, a);
  return check_launch("pjx_zero_empty_rows");
}
