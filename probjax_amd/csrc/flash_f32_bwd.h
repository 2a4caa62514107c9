// float32 flash backward at head dims 64 and 128, on the bf16 matrix units
// (f32_planes.h); the math and the split into a dQ and a dK/dV kernel are
// those of flash_bwd_kernels.h, with nothing rounded below float32.
//
// Bound as the float32 forward (flash_f32.hip), by the matrix and the vector
// units in turn.  The workgroup shapes follow the forward's: by the number of
// 128-row tiles (128-key blocks), at most one per CU or more.  us per backward,
// float32 MFMA kernels before -> chosen, other shapes (B, H, L, D causal):
//   (1,4,512,64)   138 -> 1x4 50, 2x4 57       (4,8,1024,64) 272 -> 2x4 125, 4x2 148
//   (4,8,2048,64)  743 -> 4x2 345, 2x4 409     (4,16,2048,64 full) 1870 -> 4x2 1220
//   (4,8,1024,128) 540 -> 2x2 279, 4x1 370     (4,8,2048,128) 1092 -> 4x1 805, 2x2 984
// Relative errors against float64 at (4,8,1024,64): dq, dk 4.8e-7 -> 3.6e-7,
// dv 4.0e-7 -> 3.1e-7.
#pragma once

#include "f32_planes.h"
#include "flash_bwd_kernels.h"

namespace pjx {

// ---------------------------------------------------------------------------
// dQ (and delta, lse*log2e): the decomposition of the float32 forward.  RS * KG
// waves; wave (strip, group) owns 32 query rows of the workgroup's 32 * RS and
// takes key block `group` of every stage of 32 * KG keys.  S^T = K Q^T and
// dP^T = V dO^T put keys on the MFMA rows, so dS^T in registers is the B
// operand of dQ^T += K^T dS^T; the groups' sums are added through LDS.
// BIAS: 0 none, 1 dense bias, 2 dense bias and its gradient.
// ---------------------------------------------------------------------------
template <int D, int RS, int KG, int NBUF, int WPE, int BIAS, int EXT>
__global__ __launch_bounds__(64 * RS * KG, WPE) void flash_bwd_dq_f32_planes_kernel(FlashBwdArgs ba) {
  constexpr bool HB = BIAS != 0, DB = BIAS == 2;
  const FlashArgs& a = ba.f;
  constexpr int SK = 32 * KG, BQ = 32 * RS, NT = 64 * RS * KG;
  using T = PlaneTile<D, SK>;
  constexpr int NCH = SK * T::NC;    // 8-value chunks of K (and of V) per stage
  constexpr int PER = 2 * NCH / NT;  // chunks per thread: K's first, then V's
  static_assert(PER >= 1 && 2 * NCH % NT == 0 && (PER == 1 || PER % 2 == 0), "stage shape");
  static_assert((KG - 1) * RS * 64 * (D / 2) * 4 <= NBUF * 2 * T::BYTES, "the sum fits the stages");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NBUF * 2 * T::BYTES];
  __shared__ int flags[4];  // [t % 2], [2 + t % 2] == t + 1: stage t is beyond_sure, beyond_planes

  const int tid = threadIdx.x, lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip = w8 % RS, gi = w8 / RS;
  const int col = lane & 31, half = lane >> 5;
  BlockGeom g = plane_geom(a, a.block0 + blockIdx.x, BQ, strip);
  if constexpr (EXT > 0) ext_block_range(a, g, 32, BQ);
  const int rdim = a.rdim;
  const uint32_t kv_row = (uint32_t)a.Hkv * rdim * 4;
  const unsigned char* Kb = (const unsigned char*)a.k + ((size_t)g.b * a.Lk * a.Hkv + g.hkv) * rdim * 4;
  const unsigned char* Vb = (const unsigned char*)a.v + ((size_t)g.b * a.Lk * a.Hkv + g.hkv) * rdim * 4;
  const bool row_in = g.qi < a.Lq;
  const bool row_ok = g.qi < g.q_hi;

  const size_t roff = ((size_t)(g.b * a.Lq + (row_in ? g.qi : 0)) * a.Hq + g.h) * rdim;
  const float* qrow = (const float*)a.q + roff;
  const float* drow = (const float*)ba.dout + roff;
  Planes qf[D / 16], df[D / 16];
  float dsum = 0.f;
  bool q_wild, q_sure;
  {
    const float* orow = (const float*)a.o + roff;
    PlaneSpan span;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      float x[8] = {}, y[8] = {}, z[8] = {};
      if (row_in && 16 * s + 8 * half < rdim) {
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          *(f32x4*)(x + j) = *(const f32x4*)(qrow + 16 * s + 8 * half + j);
          *(f32x4*)(y + j) = *(const f32x4*)(drow + 16 * s + 8 * half + j);
          *(f32x4*)(z + j) = *(const f32x4*)(orow + 16 * s + 8 * half + j);
        }
      }
      span.add(x);
      span.add(y);
#pragma unroll
      for (int j = 0; j < 8; ++j) dsum = fmaf(z[j], y[j], dsum);
      qf[s] = planes8(x);
      df[s] = planes8(y);
    }
    q_wild = wave_any(span.beyond_planes());
    q_sure = !wave_any(span.beyond_sure());
  }
  const float delta = xor32_sum(dsum);
  const float dsc = delta * a.scale;  // the workspace holds delta * sm_scale
  q_sure = q_sure && !wave_any(!(fabsf(dsc) < kSureScoreGrad));
  float lse2 = 0.f;
  const size_t lidx = ((size_t)g.b * a.Hq + g.h) * a.Lq + g.qi;
  if (row_in) {
    lse2 = a.lse[lidx] * kLog2e;
    if (half == 0 && gi == 0) {
      ba.delta[lidx] = dsc;
      ba.lse2[lidx] = lse2;
    }
  }
  const float* brow = nullptr;
  if constexpr (HB)
    brow = a.bias + (size_t)g.b * a.bias_bstride + (size_t)g.h * a.bias_hstride + (size_t)(row_in ? g.qi : 0) * a.Lk;
  const bool bias_vec = (a.Lk & 3) == 0;
  const bool natural = HB || EXT == 3 || (EXT == 2 && a.m.alibi != nullptr);
  const float cx = natural ? kLog2e : a.scale * kLog2e;
  ExtRows er;
  if constexpr (EXT > 0) er = ext_rows(a, g);
  if constexpr (EXT == 2) ext_segments(a, g, er, 32, (int*)smem, BQ);
  const float wscale = EXT == 3 ? a.scale * er.hm.hscale : a.scale;  // bounds d(score) of the modifiers
  q_sure = q_sure && !scale_beyond_sure(wscale);

  PlaneOffsets<D> off;
  off.init(lane);
  const uint32_t goff = wave_rows_offset<D>(kv_row, rdim);
  uint32_t loff[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int u = (tid + NT * i) % NCH, r = u / T::NC, c = u % T::NC;
    loff[i] = T::chunk(r, c) + ((tid + NT * i) / NCH) * T::BYTES;
  }

  f32x16 acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) acc[i] = f32x16{};
  const int q_last_w = g.qw + 31;
  const int n_stages = max((g.kv_stop - g.kv_begin + SK - 1) / SK, 0);

  auto is_v = [&](int i) { return PER == 1 ? w8 >= RS * KG / 2 : i >= PER / 2; };
  float reg[PER][8];
  auto load = [&](int t) PJX_INLINE_LAMBDA {
    const int k0 = g.kv_begin + t * SK;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = k0 + (64 * w8 + NT * i) % NCH / T::NC;
      const rsrc_t r = wave_rows<D>(is_v(i) ? Vb : Kb, row, g.kv_stop, kv_row, rdim);
      *(f32x4*)reg[i] = buffer_load_f32x4(r, goff);
      *(f32x4*)(reg[i] + 4) = buffer_load_f32x4(r, goff + 16);
    }
  };
  auto store = [&](int t) PJX_INLINE_LAMBDA {
    unsigned char* st = smem + (NBUF == 2 ? (t & 1) * 2 * T::BYTES : 0);
    PlaneSpan span;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      span.add(reg[i]);
      T::store(st, loff[i], reg[i]);
    }
    if (span.beyond_sure()) {
      flags[t & 1] = t + 1;
      if (span.beyond_planes()) flags[2 + (t & 1)] = t + 1;
    }
  };

  auto compute = [&](int t) PJX_INLINE_LAMBDA {
    const int k0 = g.kv_begin + t * SK + 32 * gi;
    if constexpr (EXT > 0) {
      if (!er.any || k0 > er.hi_last || k0 + 31 < er.lo_first) return;
    } else {
      if (a.causal && k0 > q_last_w) return;
    }
    if (k0 >= g.kv_stop) return;
    SegTile seg = kSegWhole;
    if constexpr (EXT == 2) {
      if (a.m.seg_k) {
        const int kk = k0 + col;
        const bool in = half == 0 && kk < g.kv_end;
        const int id = in ? a.m.seg_k[(size_t)g.b * a.Lk + kk] : 0;
        seg = seg_tile(id, in, er.seg_lo, er.seg_hi);
        if (seg == kSegSkip) return;
      }
    }
    const unsigned char* kt = smem + (NBUF == 2 ? (t & 1) * 2 * T::BYTES : 0);
    const unsigned char* vt = kt + T::BYTES;
    const bool sure = q_sure && __builtin_amdgcn_readfirstlane(flags[t & 1]) != t + 1;
    const bool wild = !sure && (q_wild || __builtin_amdgcn_readfirstlane(flags[2 + (t & 1)]) == t + 1);

    // register r holds key k0 + 8*(r/4) + 4*half + r%4 of query `col`
    f32x16 s[1] = {f32x16{}}, dp[1] = {f32x16{}};
    if (!wild) {
#pragma unroll
      for (int st = 0; st < D / 16; ++st) s[0] = mma_planes(T::rows(kt, 32 * gi, off.row[st]), qf[st], s[0]);
#pragma unroll
      for (int st = 0; st < D / 16; ++st) dp[0] = mma_planes(T::rows(vt, 32 * gi, off.row[st]), df[st], dp[0]);
    } else {
      const bool kin = k0 + col < g.kv_stop;
      const size_t ko = (size_t)(kin ? k0 + col : 0) * kv_row;
      const float* kp = (const float*)(Kb + ko) + half * (D / 2);
      const float* vp = (const float*)(Vb + ko) + half * (D / 2);
      const float* qp = qrow + half * (D / 2);
      const float* dop = drow + half * (D / 2);
#pragma unroll 1
      for (int i = 0; i < D / 2; ++i) {
        const bool in = half * (D / 2) + i < rdim;
        s[0] = mfma32x32x2f32(in && kin ? kp[i] : 0.f, in && row_in ? qp[i] : 0.f, s[0]);
        dp[0] = mfma32x32x2f32(in && kin ? vp[i] : 0.f, in && row_in ? dop[i] : 0.f, dp[0]);
      }
    }
    bool ds_wild = wild;
    if (!sure && !wild) ds_wild = score_grads_beyond_planes(dp[0], delta, wscale);
    f32x16 dbv[1];
    if constexpr (EXT == 3) {
      ext_scores_sT<1, HB>(a, g, er, s, k0, half, brow, row_in, [&](int kb, int r, float x, float gg) {
        const float p = fast_exp2(fmaf(x, cx, -lse2));
        const float u = p * (dp[kb][r] - delta);
        if constexpr (DB) dbv[kb][r] = u;
        s[kb][r] = u * a.scale * gg;
      });
    } else {
      if constexpr (HB) {
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const int kk = k0 + 8 * gq + 4 * half;
          f32x4 bv = {0.f, 0.f, 0.f, 0.f};
          if (row_in) bv = bias_vec ? load_bias4<true>(brow, kk, a.Lk) : load_bias4<false>(brow, kk, a.Lk);
#pragma unroll
          for (int j = 0; j < 4; ++j) s[0][4 * gq + j] = fmaf(s[0][4 * gq + j], a.scale, bv[j]);
        }
      }
      if constexpr (EXT == 2) {
        if (a.m.alibi) ext_slope_sT<1, HB>(a, g, er, s, k0, half);
        if (seg == kSegMixed) ext_seg_mask_sT<1>(a, g, er, s, k0, half);
      }
      if constexpr (EXT == 1 || EXT == 2) ext_mask_sT<1>(g, er, s, k0, half);
      const bool need_mask =
          EXT == 0 && ((k0 + 32 > g.kv_end) || (a.causal && k0 + 31 > g.qw) || (g.qw + 31 >= g.q_hi));
      if (need_mask) {
        const int base = k0 + 4 * half;
        int lim = g.kv_end - 1 - base;
        if (a.causal) lim = min(lim, g.qi - base);
        if (!row_ok) lim = -1;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > lim) s[0][r] = -INFINITY;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = fast_exp2(fmaf(s[0][r], cx, -lse2));
        if constexpr (DB) {
          const float u = p * (dp[0][r] - delta);
          dbv[0][r] = u;
          s[0][r] = u * a.scale;
        } else {
          s[0][r] = p * fmaf(dp[0][r], a.scale, -dsc);  // p (dp - delta) scale
        }
      }
    }
    if constexpr (DB) store_dbias<1>(ba, g, dbv, k0, half, row_in);
    // dQ^T[d][query] += K^T dS^T
    if (!ds_wild) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Planes p = planes_step(s[0], c);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          acc[db] = mma_planes(T::cols(kt, 32 * gi + 16 * c, off.tlo[db], off.thi[db]), p, acc[db]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        const bool kin = key < g.kv_stop;
        const float* kp = (const float*)(Kb + (size_t)(kin ? key : 0) * kv_row) + col;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          acc[db] = mfma32x32x2f32(kin && db * 32 + col < rdim ? kp[db * 32] : 0.f, s[0][r], acc[db]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (tid < 4) flags[tid] = 0;
  if (n_stages > 0) {
    load(0);
    __syncthreads();
    store(0);
  }
  __syncthreads();
  for (int t = 0; t < n_stages; ++t) {
    if (t + 1 < n_stages) load(t + 1);
    compute(t);
    if (NBUF == 1) __syncthreads();
    if (t + 1 < n_stages) store(t + 1);
    __syncthreads();
  }

  if constexpr (KG > 1) {
    // Groups 1 .. KG-1 hand their dQ^T sums to group 0 through LDS.
    constexpr int SLOT = RS * 64;
    f32x4* xo = (f32x4*)smem;  // [group - 1][D/32 * 4][SLOT]
    const int slot = strip * 64 + lane;
    if (gi > 0) {
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          xo[((gi - 1) * (D / 8) + 4 * i + r / 4) * SLOT + slot] =
              f32x4{acc[i][r], acc[i][r + 1], acc[i][r + 2], acc[i][r + 3]};
    }
    __syncthreads();
    if (gi > 0) return;
#pragma unroll
    for (int j = 0; j < KG - 1; ++j)
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const f32x4 o = xo[(j * (D / 8) + 4 * i + r / 4) * SLOT + slot];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][r + e] += o[e];
        }
  }
  if (row_in) {
    float* out = (float*)ba.dq + roff;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq)
        if (db * 32 + 8 * gq < rdim)
          *(f32x4*)(out + db * 32 + 8 * gq + 4 * half) =
            f32x4{acc[db][4 * gq], acc[db][4 * gq + 1], acc[db][4 * gq + 2], acc[db][4 * gq + 3]};
  }
}

// ---------------------------------------------------------------------------
// dK, dV: KS * QG waves; wave (strip, group) owns 32 keys of the workgroup's
// 32 * KS, whose K and V planes stay in LDS (V's in registers with VR), and
// takes query block `group` of every stage of 32 * QG queries of one head.  S = Q K^T and
// dP = dO V^T put queries on the MFMA rows, so P and dS in registers are the
// B operands of dV^T += dO^T P and dK^T += Q^T dS.  The query heads of the
// group stream through the same sums.
// ---------------------------------------------------------------------------
template <int D, int KS, int QG, int WPE, bool VR, bool BIAS, int EXT>
__global__ __launch_bounds__(64 * KS * QG, WPE) void flash_bwd_dkdv_f32_planes_kernel(FlashBwdArgs ba) {
  const FlashArgs& a = ba.f;
  constexpr int SQ = 32 * QG, BK = 32 * KS, NT = 64 * KS * QG;
  using T = PlaneTile<D, SQ>;
  using TK = PlaneTile<D, BK>;
  constexpr int NCH = SQ * T::NC;
  constexpr int PER = 2 * NCH / NT;  // chunks per thread: Q's first, then dO's
  static_assert(PER >= 1 && 2 * NCH % NT == 0 && (PER == 1 || PER % 2 == 0) && NT >= 2 * SQ, "stage shape");
  static_assert((QG - 1) * KS * 64 * (D / 2) * 4 <= 2 * T::BYTES, "one sum fits the stage");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * T::BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char kv[(VR ? 1 : 2) * TK::BYTES];  // K, V planes
  __shared__ __attribute__((aligned(16))) float rows[2 * SQ];  // lse*log2e, delta*sm_scale
  __shared__ int flags[4];  // [t % 2], [2 + t % 2] == t + 1: stage t is beyond_sure, beyond_planes

  const int tid = threadIdx.x, lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip = w8 % KS, gi = w8 / KS;
  const int col = lane & 31, half = lane >> 5;
  const int rdim = a.rdim;
  const int BH = a.B * a.Hkv;
  const int block = a.block0 + blockIdx.x;
  const int bh = block % BH;
  const int k0 = (block / BH) * BK;
  const int b = bh / a.Hkv, hkv = bh % a.Hkv;
  const int G = a.Hq / a.Hkv;
  const int kw = k0 + 32 * strip;
  const int key = kw + col;
  int kv_end = min(a.Lk, a.kv_valid);
  if (a.kv_lengths) kv_end = min(kv_end, max(a.kv_lengths[b], 0));
  const int q_hi = min(a.Lq, a.q_valid);
  int q_begin = a.causal ? (k0 / 32) * 32 : 0;
  int q_end = q_hi;
  int qlo = 0, qhi = q_hi - 1, wq_first = 0, wq_last = q_hi - 1, segk = 0;
  int qhi_first = q_hi - 1, qlo_last = 0;  // rows seen by every key of the wave: [qlo_last, qhi_first]
  int seg_lo = 0, seg_hi = 0;
  if constexpr (EXT > 0) {
    q_end = q_begin = 0;
    if (k0 < kv_end) {
      int a0, a1, b0, b1;
      key_bounds(a.m, a.causal, b, kv_end, q_hi, k0, a0, a1);
      key_bounds(a.m, a.causal, b, kv_end, q_hi, min(k0 + BK, kv_end) - 1, b0, b1);
      q_begin = max(a0, 0);
      q_end = b1 + 1;
    }
    key_bounds(a.m, a.causal, b, kv_end, q_hi, key, qlo, qhi);
    if (kw < kv_end) {
      key_bounds(a.m, a.causal, b, kv_end, q_hi, kw, wq_first, qhi_first);
      key_bounds(a.m, a.causal, b, kv_end, q_hi, min(kw + 32, kv_end) - 1, qlo_last, wq_last);
    }
    if (a.m.seg_k && key < a.Lk) segk = a.m.seg_k[(size_t)b * a.Lk + key];
    if constexpr (EXT == 2) {
      if (a.m.seg_k && k0 < kv_end) {
        seg_range(a.m.seg_k, b, a.Lk, kw, 32, kv_end, seg_lo, seg_hi);
        int lo, hi;
        seg_range(a.m.seg_k, b, a.Lk, k0, BK, kv_end, lo, hi);
        seg_narrow(a.m.seg_q, b, a.Lq, lo, hi, (int*)smem, q_begin, q_end);
      }
    }
  }
  const int n_qt = (k0 < kv_end && q_end > q_begin) ? (q_end - q_begin + SQ - 1) / SQ : 0;
  const int n_stages = G * n_qt;

  // K^T and V^T as B operands: lane holds key `key`, dims 16*s + 8*half + [0,8).
  // Group 0 of each strip splits its rows into LDS.
  const bool kin = key < a.Lk;
  const size_t koff = ((size_t)(b * a.Lk + (kin ? key : 0)) * a.Hkv + hkv) * rdim;
  const float* krow = (const float*)a.k + koff;
  const float* vrow = (const float*)a.v + koff;
  PlaneOffsets<D> off;
  off.init(lane);
  Planes vf[VR ? D / 16 : 1];
  bool k_wild, k_sure;
  {
    PlaneSpan span;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      float x[8] = {}, y[8] = {};
      if (kin && 16 * s + 8 * half < rdim) {
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          *(f32x4*)(x + j) = *(const f32x4*)(krow + 16 * s + 8 * half + j);
          *(f32x4*)(y + j) = *(const f32x4*)(vrow + 16 * s + 8 * half + j);
        }
      }
      span.add(x);
      span.add(y);
      if (gi == 0) {
        TK::store(kv, 32 * strip * TK::ROWB + off.row[s], x);
        if (!VR) TK::store(kv + TK::BYTES, 32 * strip * TK::ROWB + off.row[s], y);
      }
      if (VR) vf[s] = planes8(y);
    }
    k_wild = wave_any(span.beyond_planes());
    k_sure = !wave_any(span.beyond_sure()) && !scale_beyond_sure(a.scale);
  }
  auto kfrag = [&](int st) { return TK::rows(kv, 32 * strip, off.row[st]); };
  auto vfrag = [&](int st) { return VR ? vf[VR ? st : 0] : TK::rows(kv + (VR ? 0 : TK::BYTES), 32 * strip, off.row[st]); };
  const bool natural = BIAS || EXT == 3 || (EXT == 2 && a.m.alibi != nullptr);
  const float cx = natural ? kLog2e : a.scale * kLog2e;
  const uint32_t q_row = (uint32_t)a.Hq * rdim * 4;

  const uint32_t goff = wave_rows_offset<D>(q_row, rdim);
  uint32_t loff[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int u = (tid + NT * i) % NCH, r = u / T::NC, c = u % T::NC;
    loff[i] = T::chunk(r, c) + ((tid + NT * i) / NCH) * T::BYTES;
  }

  f32x16 acck[D / 32], accv[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    acck[i] = f32x16{};
    accv[i] = f32x16{};
  }

  // last query tile first, heads innermost (as the 16-bit kernel)
  auto stage_head = [&](int t) { return hkv * G + t % G; };
  auto stage_q0 = [&](int t) { return q_begin + (n_qt - 1 - t / G) * SQ; };
  auto is_d = [&](int i) { return PER == 1 ? w8 >= KS * QG / 2 : i >= PER / 2; };
  float reg[PER][8], rreg = 0.f;
  auto load = [&](int t) PJX_INLINE_LAMBDA {
    const int h = stage_head(t), q0 = stage_q0(t);
    const size_t ro = ((size_t)b * a.Lq * a.Hq + h) * rdim * 4;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = q0 + (64 * w8 + NT * i) % NCH / T::NC;
      const rsrc_t r = wave_rows<D>((const unsigned char*)(is_d(i) ? ba.dout : a.q) + ro, row, a.Lq, q_row, rdim);
      *(f32x4*)reg[i] = buffer_load_f32x4(r, goff);
      *(f32x4*)(reg[i] + 4) = buffer_load_f32x4(r, goff + 16);
    }
    rreg = 0.f;
    if (tid < 2 * SQ) {
      const int qq = q0 + (tid % SQ);
      const size_t li = ((size_t)b * a.Hq + h) * a.Lq + qq;
      if (qq < a.Lq) rreg = tid < SQ ? ba.lse2[li] : ba.delta[li];
    }
  };
  auto store = [&](int t) PJX_INLINE_LAMBDA {
    PlaneSpan span;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      span.add(reg[i]);
      T::store(smem, loff[i], reg[i]);
    }
    if (span.beyond_sure() | ((tid >= SQ) & !(fabsf(rreg) < kSureScoreGrad))) {
      flags[t & 1] = t + 1;
      if (span.beyond_planes()) flags[2 + (t & 1)] = t + 1;
    }
    if (tid < 2 * SQ) rows[tid] = rreg;
  };

  auto compute = [&](int t) PJX_INLINE_LAMBDA {
    const int h = stage_head(t), q0 = stage_q0(t) + 32 * gi;
    if (q0 >= q_hi || kw >= kv_end) return;
    if constexpr (EXT > 0) {
      if (q0 > wq_last || q0 + 31 < wq_first) return;
    } else {
      if (a.causal && q0 + 31 < kw) return;
    }
    SegTile seg = kSegWhole;
    if constexpr (EXT == 2) {
      if (a.m.seg_k) {
        const int qq = q0 + col;
        const bool in = half == 0 && qq < q_hi;
        const int id = in ? a.m.seg_q[(size_t)b * a.Lq + qq] : 0;
        seg = seg_tile(id, in, seg_lo, seg_hi);
        if (seg == kSegSkip) return;
      }
    }
    const unsigned char* qt = smem;
    const unsigned char* dt = qt + T::BYTES;
    const float* lsm = rows + 32 * gi;
    const float* dlm = lsm + SQ;
    bool sure = k_sure && __builtin_amdgcn_readfirstlane(flags[t & 1]) != t + 1;
    float hscale = 1.f;
    if constexpr (EXT == 3) {
      hscale = head_mods(a.m, h).hscale;
      sure = sure && !scale_beyond_sure(a.scale * hscale);
    }
    const bool wild = !sure && (k_wild || __builtin_amdgcn_readfirstlane(flags[2 + (t & 1)]) == t + 1);
    const float* Qg = (const float*)a.q + ((size_t)b * a.Lq * a.Hq + h) * rdim;
    const float* Dg = (const float*)ba.dout + ((size_t)b * a.Lq * a.Hq + h) * rdim;

    // register r holds query q0 + 8*(r/4) + 4*half + r%4 of key `key`
    f32x16 s = f32x16{}, dp = f32x16{};
    if (!wild) {
#pragma unroll
      for (int st = 0; st < D / 16; ++st) {
        s = mma_planes<true>(T::rows(qt, 32 * gi, off.row[st]), kfrag(st), s);
        dp = mma_planes(T::rows(dt, 32 * gi, off.row[st]), vfrag(st), dp);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      const bool qin = q0 + col < a.Lq;
      const size_t qo = (size_t)(qin ? q0 + col : 0) * a.Hq * rdim + half * (D / 2);
#pragma unroll 1
      for (int i = 0; i < D / 2; ++i) {
        const bool in = half * (D / 2) + i < rdim;
        s = mfma32x32x2f32(in && qin ? Qg[qo + i] : 0.f, in && kin ? krow[half * (D / 2) + i] : 0.f, s);
        dp = mfma32x32x2f32(in && qin ? Dg[qo + i] : 0.f, in && kin ? vrow[half * (D / 2) + i] : 0.f, dp);
      }
    }
    bool ds_wild = wild;
    if (!sure && !wild)  // one row's delta * sm_scale a lane
      ds_wild = score_grads_beyond_planes(dp, dlm[col] / a.scale, a.scale * hscale);
    if constexpr (EXT == 3) {
      const float* bbase = nullptr;
      if constexpr (BIAS) bbase = a.bias + (size_t)b * a.bias_bstride + (size_t)h * a.bias_hstride;
      const HeadMods hm = head_mods(a.m, h);
      ext_scores_S<BIAS>(a, b, hm, key, qlo, qhi, segk, s, q0, half, bbase, [&](int r, float x, float gg) {
        const int qi = 8 * (r >> 2) + 4 * half + (r & 3);
        const float p = fast_exp2(fmaf(x, cx, -lsm[qi]));
        s[r] = p;
        dp[r] = p * fmaf(dp[r], a.scale, -dlm[qi]) * gg;
      });
    } else {
      if constexpr (BIAS) {
        const float* bbase = a.bias + (size_t)b * a.bias_bstride + (size_t)h * a.bias_hstride;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qr = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
          const float bv = (qr < a.Lq && key < a.Lk) ? bbase[(size_t)qr * a.Lk + key] : 0.f;
          s[r] = fmaf(s[r], a.scale, bv);
        }
      }
      if constexpr (EXT == 2) {
        if (a.m.alibi) ext_slope_S<BIAS>(a, a.m.alibi[h], s, key, kw + 31, q0, half);
        if (seg == kSegMixed) ext_seg_mask_S(a, b, segk, s, q0, half);
      }
      if constexpr (EXT == 1 || EXT == 2)
        ext_mask_S(s, q0, half, qlo, qhi, !(kw + 31 < kv_end && q0 >= qlo_last && q0 + 31 <= qhi_first));
      const bool need_mask = EXT == 0 && ((a.causal && q0 < kw + 31) || (kw + 32 > kv_end) || (q0 + 32 > q_hi));
      if (need_mask) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qr = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
          const bool keep = key < kv_end && qr < q_hi && (!a.causal || qr >= key);
          if (!keep) s[r] = -INFINITY;
        }
      }
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const f32x4 l4 = *(const f32x4*)(lsm + 8 * gq + 4 * half), d4 = *(const f32x4*)(dlm + 8 * gq + 4 * half);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 4 * gq + j;
          const float p = fast_exp2(fmaf(s[r], cx, -l4[j]));
          s[r] = p;
          dp[r] = p * fmaf(dp[r], a.scale, -d4[j]);
        }
      }
    }
    // dV^T[d][key] += dO^T P and dK^T[d][key] += Q^T dS
    if (!ds_wild) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Planes p = planes_step(s, c);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          accv[db] = mma_planes(T::cols(dt, 32 * gi + 16 * c, off.tlo[db], off.thi[db]), p, accv[db]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Planes p = planes_step(dp, c);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          acck[db] = mma_planes(T::cols(qt, 32 * gi + 16 * c, off.tlo[db], off.thi[db]), p, acck[db]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qq = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
        const bool qin = qq < a.Lq;
        const size_t qo = (size_t)(qin ? qq : 0) * a.Hq * rdim + col;
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
          const bool in = qin && db * 32 + col < rdim;
          accv[db] = mfma32x32x2f32(in ? Dg[qo + db * 32] : 0.f, s[r], accv[db]);
          acck[db] = mfma32x32x2f32(in ? Qg[qo + db * 32] : 0.f, dp[r], acck[db]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (tid < 4) flags[tid] = 0;
  if (n_stages > 0) {
    load(0);
    __syncthreads();
    store(0);
  }
  __syncthreads();
  for (int t = 0; t < n_stages; ++t) {
    if (t + 1 < n_stages) load(t + 1);
    compute(t);
    __syncthreads();
    if (t + 1 < n_stages) store(t + 1);
    __syncthreads();
  }

  // Groups 1 .. QG-1 hand their sums to group 0 through LDS (dK, then dV) and
  // this lane's key row goes out.
  constexpr int SLOT = KS * 64;
  f32x4* xo = (f32x4*)smem;
  const int slot = strip * 64 + lane;
  auto finish = [&](f32x16* acc, float* out) {
    if constexpr (QG > 1) {
      if (gi > 0) {
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
          for (int r = 0; r < 16; r += 4)
            xo[((gi - 1) * (D / 8) + 4 * i + r / 4) * SLOT + slot] =
                f32x4{acc[i][r], acc[i][r + 1], acc[i][r + 2], acc[i][r + 3]};
      }
      __syncthreads();
      if (gi == 0) {
#pragma unroll
        for (int j = 0; j < QG - 1; ++j)
#pragma unroll
          for (int i = 0; i < D / 32; ++i)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
              const f32x4 o = xo[(j * (D / 8) + 4 * i + r / 4) * SLOT + slot];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][r + e] += o[e];
            }
      }
      __syncthreads();
    }
    if (gi == 0 && kin) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq)
          if (db * 32 + 8 * gq < rdim)
            *(f32x4*)(out + koff + db * 32 + 8 * gq + 4 * half) =
              f32x4{acc[db][4 * gq], acc[db][4 * gq + 1], acc[db][4 * gq + 2], acc[db][4 * gq + 3]};
    }
  };
  finish(acck, (float*)ba.dk);
  finish(accv, (float*)ba.dv);
}

template <int D, int RS, int KG, int NBUF, int WPE, int BIAS, int EXT>
static int launch_dq_planes(FlashBwdArgs a, hipStream_t s) {
  a.f.n_qtiles = (a.f.Lq + 32 * RS - 1) / (32 * RS);
  const long blocks = (long)a.f.n_qtiles * a.f.B * a.f.Hq;
  if (blocks > 0x7fffffffL) return fail(PJX_ERR_INVALID, "pjx_flash_bwd: grid too large");
  launch_blocks<flash_bwd_dq_f32_planes_kernel<D, RS, KG, NBUF, WPE, BIAS, EXT>>(
      blocks, 64 * RS * KG, s, a, [](FlashBwdArgs& x) -> int& { return x.f.block0; });
  return check_launch("pjx_flash_bwd (dq)");
}

template <int D, int KS, int QG, int WPE, bool VR, bool BIAS, int EXT>
static int launch_dkdv_planes(const FlashBwdArgs& a, hipStream_t s) {
  const long blocks = (long)((a.f.Lk + 32 * KS - 1) / (32 * KS)) * a.f.B * a.f.Hkv;
  if (blocks > 0x7fffffffL) return fail(PJX_ERR_INVALID, "pjx_flash_bwd: grid too large");
  launch_blocks<flash_bwd_dkdv_f32_planes_kernel<D, KS, QG, WPE, VR, BIAS, EXT>>(
      blocks, 64 * KS * QG, s, a, [](FlashBwdArgs& x) -> int& { return x.f.block0; });
  return check_launch("pjx_flash_bwd (dk, dv)");
}

// The two halves of run_flash_f32_bwd at one head dim, in a unit each.
int run_dq_f32_64(const FlashBwdArgs& a, hipStream_t s);
int run_dq_f32_128(const FlashBwdArgs& a, hipStream_t s);
int run_dkdv_f32_64(const FlashBwdArgs& a, hipStream_t s);
int run_dkdv_f32_128(const FlashBwdArgs& a, hipStream_t s);

// Calls f(std::integral_constant EXT) for the level a.f.ext.
template <typename F>
static int with_ext(const FlashBwdArgs& a, F f) {
  switch (a.f.ext) {
    case 0: return f(std::integral_constant<int, 0>{});
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    default: return f(std::integral_constant<int, 3>{});
  }
}

}  // namespace pjx
