// dL/d(bias) of the 16-bit flash attention at head dims 64 and 128, summed over
// the batches and heads the bias broadcasts to.
#include "flash_bwd_kernels.h"

namespace pjx {

struct DbiasArgs {
  FlashBwdArgs w;       // f.bias and dbias are [bias_batch, bias_heads, Lq, Lk]
  int bias_b, bias_h;   // 1 (sum over it) or B / Hq
};

// One workgroup = 2 QS waves = 32 QS queries x 128 keys of one bias slice, 32 x
// 64 per wave; it recomputes S and dP for every (batch, head) the slice stands
// for and adds P (dP - delta) in registers, so the gradient is written once,
// in whole rows, with no zero fill and no sum of per-batch copies.  Queries on
// the MFMA rows put 32 consecutive keys of a row on the lanes: the bias is read
// and its gradient written in 128-byte pieces, the bias once for all batches.
// Q, dO, K and V of the tile go memory -> LDS by buffer loads, row-major with
// the backward's swizzle.
//
// Bound by the bias and its gradient (8 bytes a score) and by the latency of
// the operand tiles, which the other workgroup of a CU covers.  Before, the dQ
// kernel stored one fp32 copy per (batch, head) in 16-byte pieces of 64 rows
// into a buffer the caller had cleared, and a reduction read the copies.
// bf16, bias [1, 8, 2048, 2048], B = 2, D = 64: dQ kernel 145 + clear 18 + sum
// 78 us before, dQ 66 + this kernel 95 us now (2.8 TB/s); operands straight
// from memory instead of through LDS: 152 us; one 8-wave workgroup per CU
// (QS = 4, what D = 128 has room for): 104 us.

template <typename E, int D, int QS, bool EXT>
__global__ __launch_bounds__(128 * QS, 2) void flash_dbias_kernel(DbiasArgs da) {
  const FlashBwdArgs& ba = da.w;
  const FlashArgs& a = ba.f;
  using T = BwdTile<D>;
  constexpr int ROWB = T::ROWB, TILE_B = T::TILE_B;
  constexpr int NW = 2 * QS, QT = QS / 2, NQ = 32 * QS;  // waves; 64-row tiles of Q; queries
  __shared__ __attribute__((aligned(1024))) unsigned char smem[(2 * QT + 4) * TILE_B];  // Q, dO, K, V tiles
  __shared__ __attribute__((aligned(16))) float rows[2][NQ];                            // lse*log2e, delta
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int nslice = da.bias_b * da.bias_h;
  const int block = a.block0 + blockIdx.x;
  const int slice = block % nslice, tile = block / nslice;
  const int nkt = (a.Lk + 127) / 128;
  const int qt0 = (tile / nkt) * NQ, kt0 = (tile % nkt) * 128;
  const int strip = w % QS, kh = w / QS;
  const int q0 = qt0 + 32 * strip, k0 = kt0 + 64 * kh;  // this wave's scores
  const int sb = slice / da.bias_h, sh = slice % da.bias_h;
  const int q_hi = min(a.Lq, a.q_valid);
  const size_t out0 = (size_t)slice * a.Lq * a.Lk;

  // fragments: rows 32 * strip + col of Q and dO, 64 * kh + col (+ 32) of K and V
  BwdOffsets<D> off;
  off.init(lane);
  const unsigned char* qs = smem + (strip >> 1) * TILE_B + (strip & 1) * 32 * ROWB;
  const unsigned char* ks = smem + (2 * QT + kh) * TILE_B;

  float bv[2][16];
  f32x16 acc[2] = {f32x16{}, f32x16{}};
  bool first = true;  // the first tile: its loads and the bias's are in flight together
  const float inv_scale = 1.f / a.scale;
  // every wave loads 64 / NW rows of each tile
  constexpr int LR = 64 / NW, NLD = LR / T::RPI;
  static_assert(LR % T::RPI == 0, "whole loads per wave");
  const int rdim = a.rdim;
  const uint32_t qstride = (uint32_t)a.Hq * rdim * 2, kstride = (uint32_t)a.Hkv * rdim * 2;
  uint32_t voffq[NLD], voffk[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {
    const int r = LR * w + T::RPI * j + lane / T::NC, c = (lane % T::NC) ^ T::swz(r);
    voffq[j] = row_chunk(r, qstride, c, rdim);
    voffk[j] = row_chunk(r, kstride, c, rdim);
  }
  // 64 rows from row0 of head `head` of a [B, L, heads, D] tensor; zeros from row `end` on: a key past a
  // sequence's end has P = 0, and a non-finite V there would make P dP a NaN
  auto load = [&](const void* t, int b, int L, int end, int heads, int head, int row0, uint32_t stride,
                  const uint32_t* voff, unsigned char* dst) {
    const int n = min(64, end - row0);
    const rsrc_t rs = make_rsrc((const unsigned char*)t + ((size_t)(b * L + (n > 0 ? row0 : 0)) * heads + head) * rdim * 2,
                                n > 0 ? (uint32_t)(n - 1) * stride + rdim * 2 : 0u);
#pragma unroll
    for (int j = 0; j < NLD; ++j) buffer_load_lds16(rs, dst + (LR * w + T::RPI * j) * ROWB, voff[j]);
  };

  const int b_end = da.bias_b == 1 ? a.B : sb + 1, h_end = da.bias_h == 1 ? a.Hq : sh + 1;
  for (int b = da.bias_b == 1 ? 0 : sb; b < b_end; ++b) {
    int kv_end = min(a.Lk, a.kv_valid);
    if (a.kv_lengths) kv_end = min(kv_end, max(a.kv_lengths[b], 0));
    // the whole tile masked (the same for every wave)
    if (qt0 >= q_hi || kt0 >= kv_end) continue;
    int qlo[2] = {0, 0}, qhi[2] = {q_hi - 1, q_hi - 1}, segk[2] = {0, 0};
    if constexpr (EXT) {
      int lo, hi, lo1, hi1;
      key_bounds(a.m, a.causal, b, kv_end, q_hi, kt0, lo, hi);
      key_bounds(a.m, a.causal, b, kv_end, q_hi, min(kt0 + 128, kv_end) - 1, lo1, hi1);
      if (qt0 > hi1 || qt0 + NQ - 1 < lo) continue;  // the bounds never decrease with the key
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int key = k0 + 32 * kb + col;
        key_bounds(a.m, a.causal, b, kv_end, q_hi, key, qlo[kb], qhi[kb]);
        if (a.m.seg_k && key < a.Lk) segk[kb] = a.m.seg_k[(size_t)b * a.Lk + key];
      }
    } else if (a.causal && qt0 + NQ - 1 < kt0) {
      continue;
    }
    for (int h = da.bias_h == 1 ? 0 : sh; h < h_end; ++h) {
      const int hkv = h / (a.Hq / a.Hkv);
      if (!first) __syncthreads();  // the tiles of the head before are consumed
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        load(a.q, b, a.Lq, a.Lq, a.Hq, h, qt0 + 64 * i, qstride, voffq, smem + i * TILE_B);
        load(ba.dout, b, a.Lq, a.Lq, a.Hq, h, qt0 + 64 * i, qstride, voffq, smem + (QT + i) * TILE_B);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        load(a.k, b, a.Lk, kv_end, a.Hkv, hkv, kt0 + 64 * i, kstride, voffk, smem + (2 * QT + i) * TILE_B);
        load(a.v, b, a.Lk, kv_end, a.Hkv, hkv, kt0 + 64 * i, kstride, voffk, smem + (2 * QT + 2 + i) * TILE_B);
      }
      if (first) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int q = q0 + 8 * (r >> 2) + 4 * half + (r & 3), key = k0 + 32 * kb + col;
            bv[kb][r] = q < a.Lq && key < a.Lk ? a.bias[out0 + (size_t)q * a.Lk + key] : 0.f;
          }
      }
      first = false;
      if (tid < 2 * NQ) {
        const int q = min(qt0 + tid % NQ, a.Lq - 1);
        const size_t li = ((size_t)b * a.Hq + h) * a.Lq + q;
        rows[tid / NQ][tid % NQ] = tid < NQ ? ba.lse2[li] : ba.delta[li] * inv_scale;
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (q0 >= q_hi || (!EXT && a.causal && q0 + 31 < k0)) continue;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int kw = k0 + 32 * kb, key = kw + col;
        if (kw >= kv_end) continue;
        f32x16 s = f32x16{}, dp = f32x16{};
#pragma unroll
        for (int st = 0; st < D / 16; ++st) {
          s = E::mma32(E::as8(*(const u32x4*)(qs + off.row[st])), E::as8(*(const u32x4*)(ks + kb * 32 * ROWB + off.row[st])), s);
          dp = E::mma32(E::as8(*(const u32x4*)(qs + QT * TILE_B + off.row[st])),
                        E::as8(*(const u32x4*)(ks + 2 * TILE_B + kb * 32 * ROWB + off.row[st])), dp);
        }
        if constexpr (EXT) {
          const HeadMods hm = head_mods(a.m, h);
          ext_scores_S<false>(a, b, hm, key, qlo[kb], qhi[kb], segk[kb], s, q0, half, nullptr,
                              [&](int r, float x, float) { s[r] = x == -INFINITY ? x : x + bv[kb][r]; });
        } else {
          const bool mask = (a.causal && q0 < kw + 31) || kw + 32 > kv_end || q0 + 32 > q_hi;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            s[r] = fmaf(s[r], a.scale, bv[kb][r]);
            const int q = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (mask && !(key < kv_end && q < q_hi && (!a.causal || q >= key))) s[r] = -INFINITY;
          }
        }
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const f32x4 l4 = *(const f32x4*)(rows[0] + 32 * strip + 8 * gq + 4 * half);
          const f32x4 d4 = *(const f32x4*)(rows[1] + 32 * strip + 8 * gq + 4 * half);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int r = 4 * gq + j;
            const float p = fast_exp2(fmaf(s[r], kLog2e, -l4[j]));
            // a dropped score adds nothing, also where its key's V (of another
            // document, outside the window, after the query) or its row's dO is not finite
            acc[kb][r] = fmaf(p, s[r] == -INFINITY ? 0.f : dp[r] - d4[j], acc[kb][r]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int q = q0 + 8 * (r >> 2) + 4 * half + (r & 3), key = k0 + 32 * kb + col;
      if (q < a.Lq && key < a.Lk) ba.dbias[out0 + (size_t)q * a.Lk + key] = acc[kb][r];
    }
}

template <typename E, int D, int QS>
static int launch_dbias(const DbiasArgs& da, hipStream_t s) {
  const FlashArgs& a = da.w.f;
  const long blocks = (a.Lq + 32L * QS - 1) / (32 * QS) * ((a.Lk + 127L) / 128) * da.bias_b * da.bias_h;
  if (blocks > 0x7fffffffL) return fail(PJX_ERR_INVALID, "pjx_flash_dbias: grid too large");
  auto first = [](DbiasArgs& x) -> int& { return x.w.f.block0; };
  if (a.ext) launch_blocks<flash_dbias_kernel<E, D, QS, true>>(blocks, 128 * QS, s, da, first);
  else launch_blocks<flash_dbias_kernel<E, D, QS, false>>(blocks, 128 * QS, s, da, first);
  return check_launch("pjx_flash_dbias");
}

// Two 4-wave workgroups fit a CU at D = 64; at D = 128 the tiles leave room for one, of 8 waves.
template <typename E>
static int launch_dbias(const DbiasArgs& da, int head_dim, hipStream_t s) {
  return head_dim == 128 ? launch_dbias<E, 128, 4>(da, s) : launch_dbias<E, 64, 2>(da, s);
}

}  // namespace pjx

using namespace pjx;

extern "C" int pjx_flash_dbias(int dtype, const void* q, const void* k, const void* v, const void* dout,
                               const void* workspace, float* dbias, const int32_t* kv_lengths, const float* bias,
                               int64_t bias_batch, int64_t bias_heads, int64_t batch, int64_t q_len, int64_t kv_len,
                               int64_t q_heads, int64_t kv_heads, int64_t head_dim, int64_t row_dim, int64_t q_valid,
                               int64_t kv_valid, int causal, float sm_scale, const pjx_score_mods* mods, void* stream) {
  clear_error();
  if (dtype != PJX_DTYPE_BF16 && dtype != PJX_DTYPE_F16)
    return fail(PJX_ERR_INVALID, "pjx_flash_dbias: dtype must be PJX_DTYPE_BF16 or PJX_DTYPE_F16");
  if (batch <= 0 || q_len <= 0 || kv_len <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads)
    return fail(PJX_ERR_INVALID, "pjx_flash_dbias: sizes must be positive and q_heads a multiple of kv_heads");
  const int rrc = check_row_dim(head_dim, row_dim, q_heads, kv_heads, "pjx_flash_dbias");
  if (rrc != PJX_OK) return rrc;
  if (!q || !k || !v || !dout || !workspace || !dbias || !bias)
    return fail(PJX_ERR_INVALID, "pjx_flash_dbias: pointers must be non-null");
  if (!((bias_batch == 1 || bias_batch == batch) && (bias_heads == 1 || bias_heads == q_heads)))
    return fail(PJX_ERR_INVALID, "pjx_flash_dbias: bias must be [1|B, 1|Hq, Lq, Lk]");
  if (!(sm_scale > 0.f)) return fail(PJX_ERR_INVALID, "pjx_flash_dbias: sm_scale must be > 0");
  if (std::max(batch * q_len * q_heads, batch * kv_len * kv_heads) * head_dim > (int64_t)1 << 40 ||
      q_len > (1 << 30) || kv_len > (1 << 30))
    return fail(PJX_ERR_INVALID, "pjx_flash_dbias: sizes out of range");
  DbiasArgs da;
  FlashBwdArgs& ba = da.w;
  FlashArgs& a = ba.f;
  a.q = q; a.k = k; a.v = v; a.o = nullptr; a.lse = nullptr;
  a.kv_lengths = kv_lengths;
  a.bias = bias;
  a.bias_bstride = a.bias_hstride = 0;
  a.B = (int)batch; a.Lq = (int)q_len; a.Lk = (int)kv_len;
  a.Hq = (int)q_heads; a.Hkv = (int)kv_heads;
  a.q_valid = (int)std::min<int64_t>(std::max<int64_t>(q_valid, 0), q_len);
  a.kv_valid = (int)std::min<int64_t>(std::max<int64_t>(kv_valid, 0), kv_len);
  a.causal = causal ? 1 : 0;
  a.f16 = dtype == PJX_DTYPE_F16;
  a.scale = sm_scale;
  a.n_qtiles = 0;
  a.dv = (int)head_dim;
  a.rdim = (int)row_dim;
  const int rc = lower_score_mods(mods, a, "pjx_flash_dbias");
  if (rc != PJX_OK) return rc;
  ba.dout = dout;
  ba.delta = (float*)const_cast<void*>(workspace);
  ba.lse2 = ba.delta + batch * q_heads * q_len;
  ba.dq = ba.dk = ba.dv = nullptr;
  ba.dbias = dbias;
  ba.part = nullptr;
  ba.nsplit = 1;
  da.bias_b = (int)bias_batch;
  da.bias_h = (int)bias_heads;
  return a.f16 ? launch_dbias<F16Fmt>(da, (int)head_dim, (hipStream_t)stream)
               : launch_dbias<Bf16Fmt>(da, (int)head_dim, (hipStream_t)stream);
}
