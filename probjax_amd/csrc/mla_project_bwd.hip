// Gradients of the materialised latent's up-projection (mla_project.hip):
//   dcache[m, r] = sum_n dK[m, n] wk[n, r] + dV[m, n] wv[n, r]
//   dwk[n, r]    = sum_m dK[m, n] cache[m, r],  dwv likewise
// over latent rows m = b*S + s and channels n = h*width + d (d < the head's
// dim), the chain rule of K = C W_K^T, V = C W_V^T in probjax's VJP of `mla`
// (kernels/latent_attention.py:571-589).  16-bit inputs and outputs, float32
// sums rounded once (K's and V's parts of dcache are added before rounding).
//
// Both products contract over an index that is not contiguous in one or both
// operands; the transposing LDS reads hand out those operands from tiles as
// they lie in memory, where a library product first wants dK and dV
// transposed in memory.  bf16, B=4 S=2048 H=8 width 64 R=128: two transposes,
// four products and an add, 97 us, became 28 us (dcache 11.8, dW 10.8, the sum
// of its parts 5.3), bound by the latency of the stages (two in LDS); S=4096
// H=16 width 128 R=512: 169 -> 74 us; B=4 S=4096 H=32: 898 -> 456 us.  Faster
// at every size tried, so only unaligned ranks and dims and float32 keep the
// library products.
#include "flash_bwd_kernels.h"

namespace pjx {

struct ProjBwdArgs {
  const uint16_t* cache;  // [M, R]
  const uint16_t* w[2];   // [H, dim, R]
  const uint16_t* d[2];   // dK, dV [M, H * width]
  uint16_t* dcache;       // [M, R]
  uint16_t* dw[2];        // [H, dim, R]
  float* part;            // [splits][2][H * width][R]
  float* cpart;           // [csplits][M][R] if csplits > 1
  int64_t M;
  int H, R, width, dim[2], splits, csplits;
};

// dcache: one workgroup per 64 rows x 64 rank entries x channel split (its
// float32 parts go to cpart if there are several), 4 waves of 32 x 32.
// Stages of 64 channels: dK rows [64][64] and W rows [64 channels][64 rank
// entries] by buffer loads, two stages.  The contraction runs in the slot order
// of the transposing reads (8*(j/4) + 4*half + j%4 within 16), so dK's operand
// is two 8-byte reads.
template <typename E>
__global__ __launch_bounds__(kThreads, 2) void mla_project_dcache_kernel(ProjBwdArgs a) {
  using T = BwdTile<64>;
  __shared__ __attribute__((aligned(1024))) unsigned char s0[2 * T::TILE_B];
  __shared__ __attribute__((aligned(1024))) unsigned char s1[2 * T::TILE_B];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int64_t m0 = (int64_t)blockIdx.x * 64;
  const int r0 = blockIdx.y * 64;
  const int N = a.H * a.width, nchunk = N / 64;  // width is a multiple of 64
  const int mvalid = (int)min<int64_t>(64, a.M - m0);
  // tile rows 16 * w + 8 * j + lane / 8, 16-byte chunk lane % 8
  uint32_t doff[T::NLD], woff[T::NLD];
  int dch[T::NLD];
#pragma unroll
  for (int j = 0; j < T::NLD; ++j) {
    const int r = 16 * w + T::RPI * j + lane / T::NC, c = (lane % T::NC) ^ T::swz(r);
    dch[j] = 8 * c;
    doff[j] = r * (uint32_t)N * 2 + 16 * c;
    woff[j] = r0 + 8 * c < a.R ? r * (uint32_t)a.R * 2 + 16 * c : kPastBuffer;
  }
  auto issue = [&](int t, unsigned char* st) {
    const int which = t >= nchunk, n0 = (which ? t - nchunk : t) * 64;
    const int h = n0 / a.width, d0 = n0 % a.width, dim = a.dim[which];
    const int wrows = min(64, dim - d0);  // the head's channels in this chunk
    const rsrc_t rd = make_rsrc(a.d[which] + m0 * N + n0, (uint32_t)(mvalid - 1) * N * 2 + 128);
    const rsrc_t rw = make_rsrc(a.w[which] + ((size_t)h * dim + (wrows > 0 ? d0 : 0)) * a.R + r0,
                                wrows > 0 ? (uint32_t)(wrows - 1) * a.R * 2 + min(64, a.R - r0) * 2 : 0u);
#pragma unroll
    for (int j = 0; j < T::NLD; ++j) {
      // channels past the head's dim read as zero on both sides (0 * inf is NaN)
      buffer_load_lds16(rd, st + (16 * w + T::RPI * j) * T::ROWB, dch[j] < wrows ? doff[j] : kPastBuffer);
      buffer_load_lds16(rw, st + T::TILE_B + (16 * w + T::RPI * j) * T::ROWB, woff[j]);
    }
  };
  BwdOffsets<64> off;
  off.init(lane);
  const int arow = 32 * (w & 1) + col, db = w >> 1;
  uint32_t alo[4], ahi[4];  // channels 16 * c + 4 * half + [0, 4) and 8 further
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    alo[c] = arow * T::ROWB + 16 * ((2 * c) ^ T::swz(arow)) + 8 * half;
    ahi[c] = arow * T::ROWB + 16 * ((2 * c + 1) ^ T::swz(arow)) + 8 * half;
  }
  f32x16 acc = f32x16{};
  auto compute = [&](const unsigned char* st) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const u32x2 lo = *(const u32x2*)(st + alo[c]), hi = *(const u32x2*)(st + ahi[c]);
      const typename E::v8 bf = read_t<E, 64>(st + T::TILE_B, 16 * c, db ? off.tlo[1] : off.tlo[0], db ? off.thi[1] : off.thi[0]);
      acc = E::mma32(E::as8(u32x4{lo[0], lo[1], hi[0], hi[1]}), bf, acc);
    }
  };
  const int t0 = 2 * (int)((int64_t)nchunk * blockIdx.z / a.csplits);
  const int t1 = 2 * (int)((int64_t)nchunk * (blockIdx.z + 1) / a.csplits);
  if (t0 < t1) issue(t0, s0);
  for (int t = t0; t < t1; t += 2) {  // an even number of stages
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    issue(t + 1, s1);
    compute(s0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + 2 < t1) issue(t + 2, s0);
    compute(s1);
  }
  // register r: row 8*(r/4) + 4*half + r%4, rank entry `col`
  const int rr = r0 + 32 * db + col;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t m = m0 + 32 * (w & 1) + 8 * (r >> 2) + 4 * half + (r & 3);
    if (m < a.M && rr < a.R) {
      if (a.csplits == 1)
        a.dcache[m * a.R + rr] = E::bits(acc[r]);
      else
        a.cpart[((size_t)blockIdx.z * a.M + m) * a.R + rr] = acc[r];
    }
  }
}

// Partial dW of one row split: one workgroup per 128 channels x 128 rank
// entries x split, 4 waves of 64 x 64; stages of 64 latent rows of dK (or dV)
// and the cache, both operands by transposing reads.
template <typename E>
__global__ __launch_bounds__(kThreads, 2) void mla_project_dw_kernel(ProjBwdArgs a) {
  using T = BwdTile<128>;
  __shared__ __attribute__((aligned(1024))) unsigned char s0[2 * T::TILE_B];
  __shared__ __attribute__((aligned(1024))) unsigned char s1[2 * T::TILE_B];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int N = a.H * a.width, nt = (N + 127) / 128;
  const int which = blockIdx.y >= (unsigned)nt;
  const int n0 = (blockIdx.y - which * nt) * 128, r0 = blockIdx.x * 128, split = blockIdx.z;
  const int64_t stages = (a.M + 63) / 64;
  const int64_t t0 = stages * split / a.splits, t1 = stages * (split + 1) / a.splits;
  uint32_t doff[T::NLD], coff[T::NLD];
#pragma unroll
  for (int j = 0; j < T::NLD; ++j) {
    const int r = 16 * w + T::RPI * j + lane / T::NC, c = (lane % T::NC) ^ T::swz(r);
    doff[j] = n0 + 8 * c < N ? r * (uint32_t)N * 2 + 16 * c : kPastBuffer;
    coff[j] = r0 + 8 * c < a.R ? r * (uint32_t)a.R * 2 + 16 * c : kPastBuffer;
  }
  auto issue = [&](int64_t t, unsigned char* st) {
    const int64_t m = t * 64;
    const int rows = (int)min<int64_t>(64, a.M - m);
    const rsrc_t rd = make_rsrc(a.d[which] + m * N + n0, (uint32_t)(rows - 1) * N * 2 + min(128, N - n0) * 2);
    const rsrc_t rc = make_rsrc(a.cache + m * a.R + r0, (uint32_t)(rows - 1) * a.R * 2 + min(128, a.R - r0) * 2);
#pragma unroll
    for (int j = 0; j < T::NLD; ++j) {
      buffer_load_lds16(rd, st + (16 * w + T::RPI * j) * T::ROWB, doff[j]);
      buffer_load_lds16(rc, st + T::TILE_B + (16 * w + T::RPI * j) * T::ROWB, coff[j]);
    }
  };
  BwdOffsets<128> off;
  off.init(lane);
  const int wr = w & 1, wc = w >> 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  uint32_t alo[2], ahi[2], blo[2], bhi[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    alo[i] = wr ? off.tlo[2 + i] : off.tlo[i];
    ahi[i] = wr ? off.thi[2 + i] : off.thi[i];
    blo[i] = wc ? off.tlo[2 + i] : off.tlo[i];
    bhi[i] = wc ? off.thi[2 + i] : off.thi[i];
  }
  auto compute = [&](const unsigned char* st) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      typename E::v8 af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[i] = read_t<E, 128>(st, 16 * c, alo[i], ahi[i]);
        bf[i] = read_t<E, 128>(st + T::TILE_B, 16 * c, blo[i], bhi[i]);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = E::mma32(af[i], bf[j], acc[i][j]);
    }
  };
  if (t0 < t1) issue(t0, s0);
  for (int64_t t = t0; t < t1; t += 2) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + 1 < t1) issue(t + 1, s1);
    compute(s0);
    if (t + 1 >= t1) break;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + 2 < t1) issue(t + 2, s0);
    compute(s1);
  }
  float* out = a.part + ((size_t)split * 2 + which) * N * a.R;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + 64 * wr + 32 * i + 8 * (r >> 2) + 4 * half + (r & 3), rr = r0 + 64 * wc + 32 * j + col;
        if (n < N && rr < a.R) out[(size_t)n * a.R + rr] = acc[i][j][r];
      }
}

// dW = the sum of the splits' parts, in order, for the channels that exist
// (blockIdx.y: dwk, dwv).  R is a multiple of 8.
template <typename E>
__global__ __launch_bounds__(kThreads) void mla_project_dw_sum_kernel(ProjBwdArgs a) {
  const int which = blockIdx.y, dim = a.dim[which], N = a.H * a.width;
  const size_t e = 4 * ((size_t)blockIdx.x * kThreads + threadIdx.x);
  if (e >= (size_t)a.H * dim * a.R) return;
  const int n = (int)(e / a.R), h = n / dim, d = n % dim;
  const float* p = a.part + ((size_t)which * N + h * a.width + d) * a.R + e % a.R;
  f32x4 acc = *(const f32x4*)p;
#pragma unroll 8
  for (int s = 1; s < a.splits; ++s) acc += *(const f32x4*)(p + (size_t)s * 2 * N * a.R);
  *(u32x2*)(a.dw[which] + e) = u32x2{E::pack2(acc[0], acc[1]), E::pack2(acc[2], acc[3])};
}

// dcache = the sum of the channel splits' parts, in order.
template <typename E>
__global__ __launch_bounds__(kThreads) void mla_project_dcache_sum_kernel(ProjBwdArgs a) {
  const size_t n = (size_t)a.M * a.R, e = 4 * ((size_t)blockIdx.x * kThreads + threadIdx.x);
  if (e >= n) return;
  f32x4 acc = *(const f32x4*)(a.cpart + e);
#pragma unroll 8
  for (int s = 1; s < a.csplits; ++s) acc += *(const f32x4*)(a.cpart + s * n + e);
  *(u32x2*)(a.dcache + e) = u32x2{E::pack2(acc[0], acc[1]), E::pack2(acc[2], acc[3])};
}

// Splits of the channels for dcache: one where the tiles give every CU a
// workgroup (256) or the contraction is short; else up to 512 workgroups of at
// least 16 stages (the parts' pass over memory costs what about 8 stages do).
// S=1024 H=128 width 128 R=512, 128 tiles of 512 stages: 345 us unsplit, 153
// in four.
static int proj_bwd_csplits(int64_t M, int64_t N, int64_t R) {
  const int64_t tiles = ((M + 63) / 64) * ((R + 63) / 64), stages = N / 32;
  if (tiles >= 256) return 1;
  return (int)std::max<int64_t>(1, std::min<int64_t>({512 / tiles, stages / 16, 64}));
}

// Splits of the latent rows for dW: about 512 workgroups (two per CU), each
// with at least 4 stages of 64 rows; a function of the sizes.  The sum of the
// parts keeps eight loads in flight (32 splits of 512 x 128 twice: 9.6 -> 5.3 us).
static int proj_bwd_splits(int64_t M, int64_t N, int64_t R) {
  const int64_t tiles = 2 * ((N + 127) / 128) * ((R + 127) / 128), stages = (M + 63) / 64;
  return (int)std::max<int64_t>(1, std::min<int64_t>({(512 + tiles - 1) / tiles, stages / 4, 64}));
}

template <typename E>
static int launch_proj_bwd(const ProjBwdArgs& a, hipStream_t s) {
  const int N = a.H * a.width;
  launch_kernel<mla_project_dcache_kernel<E>>(dim3((unsigned)((a.M + 63) / 64), (a.R + 63) / 64, a.csplits), dim3(kThreads), 0, s, a);
  if (a.csplits > 1)
    launch_kernel<mla_project_dcache_sum_kernel<E>>(dim3((unsigned)(((size_t)a.M * a.R / 4 + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, a);
  launch_kernel<mla_project_dw_kernel<E>>(dim3((a.R + 127) / 128, 2 * ((N + 127) / 128), a.splits), dim3(kThreads), 0, s, a);
  const size_t n = (size_t)a.H * std::max(a.dim[0], a.dim[1]) * a.R;
  launch_kernel<mla_project_dw_sum_kernel<E>>(dim3((unsigned)((n / 4 + kThreads - 1) / kThreads), 2), dim3(kThreads), 0, s, a);
  return check_launch("pjx_mla_project_bwd");
}

}  // namespace pjx

using namespace pjx;

extern "C" size_t pjx_mla_project_bwd_workspace_size(int64_t batch, int64_t kv_len, int64_t heads, int64_t rank,
                                                     int64_t width) {
  if (batch <= 0 || kv_len <= 0 || heads <= 0 || rank <= 0 || width <= 0) return 0;
  const int64_t M = batch * kv_len, N = heads * width;
  const int cs = proj_bwd_csplits(M, N, rank);
  return ((size_t)proj_bwd_splits(M, N, rank) * 2 * N + (cs > 1 ? (size_t)cs * M : 0)) * rank * sizeof(float);
}

extern "C" int pjx_mla_project_bwd(int dtype, const void* cache, const void* wk, const void* wv, const void* dk,
                                   const void* dv, void* dcache, void* dwk, void* dwv, void* workspace,
                                   size_t workspace_bytes, int64_t batch, int64_t kv_len, int64_t heads, int64_t rank,
                                   int64_t qk_dim, int64_t v_dim, int64_t width, void* stream) {
  clear_error();
  if (dtype != PJX_DTYPE_BF16 && dtype != PJX_DTYPE_F16)
    return fail(PJX_ERR_INVALID, "pjx_mla_project_bwd: dtype must be PJX_DTYPE_BF16 or PJX_DTYPE_F16");
  if (batch <= 0 || kv_len <= 0 || heads <= 0 || rank <= 0 || rank % 8)
    return fail(PJX_ERR_INVALID, "pjx_mla_project_bwd: sizes must be positive and rank a multiple of 8");
  if (width <= 0 || width % 64 || qk_dim <= 0 || v_dim <= 0 || qk_dim > width || v_dim > width || qk_dim % 8 || v_dim % 8)
    return fail(PJX_ERR_INVALID,
                "pjx_mla_project_bwd: need qk_dim, v_dim multiples of 8, at most width, a multiple of 64");
  // 64 rows of each operand lie below kPastBuffer, and the grids below 65536
  const int64_t kMax = (int64_t)1 << 20;
  if (heads > kMax || width > kMax || heads * width > kMax || rank > kMax || batch > ((int64_t)1 << 31) ||
      kv_len > ((int64_t)1 << 31) || batch * kv_len > ((int64_t)1 << 34))
    return fail(PJX_ERR_INVALID, "pjx_mla_project_bwd: sizes out of range");
  if (!cache || !wk || !wv || !dk || !dv || !dcache || !dwk || !dwv)
    return fail(PJX_ERR_INVALID, "pjx_mla_project_bwd: null pointer");
  if (!workspace || workspace_bytes < pjx_mla_project_bwd_workspace_size(batch, kv_len, heads, rank, width))
    return fail(PJX_ERR_WORKSPACE,
                "pjx_mla_project_bwd: workspace missing or smaller than pjx_mla_project_bwd_workspace_size()");
  ProjBwdArgs a = {};
  a.cache = (const uint16_t*)cache;
  a.w[0] = (const uint16_t*)wk;
  a.w[1] = (const uint16_t*)wv;
  a.d[0] = (const uint16_t*)dk;
  a.d[1] = (const uint16_t*)dv;
  a.dcache = (uint16_t*)dcache;
  a.dw[0] = (uint16_t*)dwk;
  a.dw[1] = (uint16_t*)dwv;
  a.part = (float*)workspace;
  a.M = batch * kv_len;
  a.H = (int)heads;
  a.R = (int)rank;
  a.width = (int)width;
  a.dim[0] = (int)qk_dim;
  a.dim[1] = (int)v_dim;
  a.splits = proj_bwd_splits(a.M, heads * width, rank);
  a.csplits = proj_bwd_csplits(a.M, heads * width, rank);
  a.cpart = a.part + (size_t)a.splits * 2 * heads * width * rank;
  return dtype == PJX_DTYPE_F16 ? launch_proj_bwd<F16Fmt>(a, (hipStream_t)stream)
                                : launch_proj_bwd<Bf16Fmt>(a, (hipStream_t)stream);
}
