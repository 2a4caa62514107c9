// float32 flash forward at head dims 64 and 128, on the bf16 matrix units
// (f32_planes.h): every operand is three bf16 planes and every product six
// bf16 MFMAs, with float32 precision.
#include "f32_planes.h"

namespace pjx {

// Whether the rows that one wave loads at once (wave_rows) lie further apart than
// a buffer's 32-bit offsets reach: a few million heads.
static bool rows_far(const FlashArgs& a, int head_dim) {
  return (int64_t)a.Hkv * a.rdim * 4 * (512 / head_dim) > 0xffffffffLL;
}

// ---------------------------------------------------------------------------
// One workgroup = RS * KG waves = 32 * RS query rows of one (batch, head);
// wave (strip, group) owns rows 32 * strip .. and takes key block `group` of
// every stage of 32 * KG keys.  A stage's K and V rows are loaded to
// registers while the stage before is computed, then split once for all waves
// into LDS planes (NBUF stages).  S^T = K Q^T with keys as MFMA rows and
// O^T += V^T P^T with P from registers, as in the 16-bit forward; the groups'
// partial (max, sum, O) are merged through LDS at the end.
//
// Bound by the matrix and the vector units in turn: 48 MFMAs (1536 cycles) and
// about 260 vector operations (splitting K, V and P, the softmax) per 32 x 32
// scores at D = 64, which the two waves of a SIMD overlap little: MFMA busy
// 50%, 183 TFLOP/s over 4 x 16 heads of 2048 full rows, above the float32
// MFMA peak of 157.  Not kept: S_{t+1} formed under stage t's softmax inside a
// wave (needs more than 256 registers, 1.3-1.8x slower), three waves per SIMD
// (spills, 1.4x slower), fixed wave priorities (1-2%).
// FAR: rows_far, loads by 64-bit addresses (as a branch here they cost the small
// causal call of (1, 4, 512, 64) 4%).
// ---------------------------------------------------------------------------
template <int D, int RS, int KG, int NBUF, int WPE, bool BIAS, int EXT, bool FAR = false>
__global__ __launch_bounds__(64 * RS * KG, WPE) void flash_fwd_f32_planes_kernel(FlashArgs a) {
  constexpr int SK = 32 * KG, BQ = 32 * RS, NT = 64 * RS * KG;
  using T = PlaneTile<D, SK>;
  constexpr int NCH = SK * T::NC;     // 8-value chunks of K (and of V) per stage
  constexpr int PER = 2 * NCH / NT;   // chunks per thread: K's first, then V's
  static_assert(PER >= 1 && 2 * NCH % NT == 0 && (PER == 1 || PER % 2 == 0), "stage shape");
  static_assert((KG - 1) * RS * 64 * (D / 2 + 2) * 4 <= NBUF * 2 * T::BYTES, "the merge fits the stages");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NBUF * 2 * T::BYTES];
  __shared__ int flags[2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip = w8 % RS, gi = w8 / RS;
  const int col = lane & 31, half = lane >> 5;
  BlockGeom g = plane_geom(a, a.block0 + blockIdx.x, BQ, strip);
  if constexpr (EXT > 0) ext_block_range(a, g, 32, BQ);
  const int rdim = a.rdim;
  const typename std::conditional<FAR, size_t, uint32_t>::type kv_row = (size_t)a.Hkv * rdim * 4;
  const unsigned char* Kb = (const unsigned char*)a.k + ((size_t)g.b * a.Lk * a.Hkv + g.hkv) * rdim * 4;
  const unsigned char* Vb = (const unsigned char*)a.v + ((size_t)g.b * a.Lk * a.Hkv + g.hkv) * rdim * 4;
  const bool row_in = g.qi < a.Lq;
  const bool row_ok = g.qi < g.q_hi;

  // Q^T as the B operand: lane holds query `col`, dims 16*s + 8*half + [0,8).
  const float* qrow = (const float*)a.q + ((size_t)(g.b * a.Lq + (row_in ? g.qi : 0)) * a.Hq + g.h) * rdim;
  Planes qf[D / 16];
  bool q_wild;  // a value beyond the planes' range in the wave's rows
  {
    PlaneSpan span;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (row_in && 16 * s + 8 * half < rdim) {
        *(f32x4*)x = *(const f32x4*)(qrow + 16 * s + 8 * half);
        *(f32x4*)(x + 4) = *(const f32x4*)(qrow + 16 * s + 8 * half + 4);
      }
      span.add(x);
      qf[s] = planes8(x);
    }
    q_wild = wave_any(span.beyond_planes());
  }
  const float* brow = nullptr;
  if constexpr (BIAS)
    brow = a.bias + (size_t)g.b * a.bias_bstride + (size_t)g.h * a.bias_hstride + (size_t)(row_in ? g.qi : 0) * a.Lk;
  const bool bias_vec = (a.Lk & 3) == 0;
  const bool natural = BIAS || EXT == 3 || (EXT == 2 && a.m.alibi != nullptr);
  const float cx = natural ? kLog2e : a.scale * kLog2e;
  ExtRows er;
  if constexpr (EXT > 0) er = ext_rows(a, g);
  if constexpr (EXT == 2) ext_segments(a, g, er, 32, (int*)smem, BQ);

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
  float m_run = kMaxInit, l_run = 0.f;
  float thr = -INFINITY;  // rescale when a raw row max exceeds (m_run + kRescaleLog2) / cx
  const int q_last_w = g.qw + 31;
  const int n_stages = max((g.kv_stop - g.kv_begin + SK - 1) / SK, 0);

  // chunk i is V's (PER == 1: the second half of the waves')
  auto is_v = [&](int i) { return PER == 1 ? w8 >= RS * KG / 2 : i >= PER / 2; };
  float reg[PER][8];
  auto load = [&](int t) PJX_INLINE_LAMBDA {
    const int k0 = g.kv_begin + t * SK;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = k0 + (64 * w8 + NT * i) % NCH / T::NC;
      if constexpr (FAR) {
        const int r = row + lane / T::NC, c = lane % T::NC;
        f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
        if (r < g.kv_stop && 8 * c < rdim) {
          const f32x4* p = (const f32x4*)((is_v(i) ? Vb : Kb) + r * kv_row + 32 * c);
          x = p[0];
          y = p[1];
        }
        *(f32x4*)reg[i] = x;
        *(f32x4*)(reg[i] + 4) = y;
        continue;
      }
      const rsrc_t r = wave_rows<D>(is_v(i) ? Vb : Kb, row, g.kv_stop, kv_row, rdim);
      *(f32x4*)reg[i] = buffer_load_f32x4(r, goff);
      *(f32x4*)(reg[i] + 4) = buffer_load_f32x4(r, goff + 16);
    }
  };
  // flags[t % 2] == t + 1: stage t holds a value beyond the planes' range
  auto store = [&](int t) PJX_INLINE_LAMBDA {
    unsigned char* st = smem + (NBUF == 2 ? (t & 1) * 2 * T::BYTES : 0);
    PlaneSpan span;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      span.add(reg[i]);
      T::store(st, loff[i], reg[i]);
    }
    if (span.beyond_planes()) flags[t & 1] = t + 1;
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
    const bool wild = q_wild || __builtin_amdgcn_readfirstlane(flags[t & 1]) == t + 1;

    // S^T[key][query]: register r holds key k0 + 8*(r/4) + 4*half + r%4.
    f32x16 s[1] = {f32x16{}};
    if (!wild) {
#pragma unroll
      for (int st = 0; st < D / 16; ++st) s[0] = mma_planes(T::rows(kt, 32 * gi, off.row[st]), qf[st], s[0]);
    } else {
      const bool kin = k0 + col < g.kv_stop;
      const float* kp = (const float*)(Kb + (size_t)(kin ? k0 + col : 0) * kv_row) + half * (D / 2);
      const float* qp = qrow + half * (D / 2);
#pragma unroll 1
      for (int i = 0; i < D / 2; ++i) {
        const bool in = half * (D / 2) + i < rdim;
        s[0] = mfma32x32x2f32(in && kin ? kp[i] : 0.f, in && row_in ? qp[i] : 0.f, s[0]);
      }
    }
    if constexpr (EXT == 3) {
      ext_scores_sT<1, BIAS>(a, g, er, s, k0, half, brow, row_in, [&](int kb, int r, float x, float) { s[kb][r] = x; });
    } else if constexpr (BIAS) {
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
      if (a.m.alibi) ext_slope_sT<1, BIAS>(a, g, er, s, k0, half);
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
    float mx = fmaxf(s[0][0], s[0][1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) mx = fmaxf(fmaxf(mx, s[0][r]), s[0][r + 1]);
    mx = xor32_max(mx);
    if (wave_any(mx > thr)) {
      const float m_new = fmaxf(m_run, mx * cx);
      const float corr = fast_exp2(m_run - m_new);
      m_run = m_new;
      thr = (m_run + kRescaleLog2) / cx;
      l_run *= corr;
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= corr;
    }
    float rs0 = 0.f, rs1 = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      s[0][r] = fast_exp2(fmaf(s[0][r], cx, -m_run));
      s[0][r + 1] = fast_exp2(fmaf(s[0][r + 1], cx, -m_run));
      rs0 += s[0][r];
      rs1 += s[0][r + 1];
    }
    l_run += rs0 + rs1;
    if (!wild) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Planes p = planes_step(s[0], c);
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          acc[db] = mma_planes(T::cols(vt, 32 * gi + 16 * c, off.tlo[db], off.thi[db]), p, acc[db]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * half + (r & 3);
        const bool vin = key < g.kv_stop;
        const float* vp = (const float*)(Vb + (size_t)(vin ? key : 0) * kv_row) + col;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
          acc[db] = mfma32x32x2f32(vin && db * 32 + col < rdim ? vp[db * 32] : 0.f, s[0][r], acc[db]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (tid < 2) flags[tid] = 0;
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
    // Groups 1 .. KG-1 hand (max, sum, O) to group 0 through LDS, lane by lane
    // in the same register layout.
    constexpr int SLOT = RS * 64;  // lanes per group
    f32x4* xo = (f32x4*)smem;      // [group - 1][D/32 * 4][SLOT]
    float* xml = (float*)(smem + (KG - 1) * (D / 8) * SLOT * 16);
    const int slot = strip * 64 + lane;
    if (gi > 0) {
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          xo[((gi - 1) * (D / 8) + 4 * i + r / 4) * SLOT + slot] =
              f32x4{acc[i][r], acc[i][r + 1], acc[i][r + 2], acc[i][r + 3]};
      xml[2 * ((gi - 1) * SLOT + slot)] = m_run;
      xml[2 * ((gi - 1) * SLOT + slot) + 1] = l_run;
    }
    __syncthreads();
    if (gi > 0) return;
    float M = m_run;
#pragma unroll
    for (int j = 0; j < KG - 1; ++j) M = fmaxf(M, xml[2 * (j * SLOT + slot)]);
    const float f0 = fast_exp2(m_run - M);
    l_run *= f0;
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][r] *= f0;
#pragma unroll
    for (int j = 0; j < KG - 1; ++j) {
      const float f = fast_exp2(xml[2 * (j * SLOT + slot)] - M);
      l_run = fmaf(xml[2 * (j * SLOT + slot) + 1], f, l_run);
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const f32x4 o = xo[(j * (D / 8) + 4 * i + r / 4) * SLOT + slot];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][r + e] = fmaf(o[e], f, acc[i][r + e]);
        }
    }
    m_run = M;
  }

  const float l_tot = xor32_sum(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (row_in) {
    float* orow = (float*)a.o + ((size_t)(g.b * a.Lq + g.qi) * a.Hq + g.h) * rdim;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq)
        if (db * 32 + 8 * gq < rdim)
          *(f32x4*)(orow + db * 32 + 8 * gq + 4 * half) =
            f32x4{acc[db][4 * gq] * inv, acc[db][4 * gq + 1] * inv, acc[db][4 * gq + 2] * inv, acc[db][4 * gq + 3] * inv};
    if (a.lse && half == 0)
      a.lse[((size_t)g.b * a.Hq + g.h) * a.Lq + g.qi] =
          l_tot > 0.f ? (m_run + __log2f(l_tot)) * kLn2 : INFINITY;
  }
}

template <int D, int RS, int KG, int NBUF, int WPE, bool BIAS, int EXT, bool FAR = false>
static int launch_planes(FlashArgs a, hipStream_t s) {
  a.n_qtiles = (a.Lq + 32 * RS - 1) / (32 * RS);
  const long blocks = (long)a.n_qtiles * a.B * a.Hq;
  if (blocks > 0x7fffffffL) return fail(PJX_ERR_INVALID, "pjx_flash_fwd: grid too large");
  launch_blocks<flash_fwd_f32_planes_kernel<D, RS, KG, NBUF, WPE, BIAS, EXT, FAR>>(
      blocks, 64 * RS * KG, s, a, [](FlashArgs& x) -> int& { return x.block0; });
  return check_launch("pjx_flash_fwd");
}

// Rows and key groups of a workgroup by the size of the grid (256 CUs).  Few
// rows: 32-row workgroups whose 4 waves share the keys.  Up to one 128-row tile
// per CU: 64 rows and 4 key groups, so that a causal grid has twice the
// workgroups and the heavy ones, first, leave room for the light ones.  Above:
// 128 rows and 2 key groups, which split each K / V row for twice the queries
// (extended masks keep the 64-row form).  At D = 128 a wave's Q planes and sums
// take a SIMD's registers alone, and one key group is enough above a tile per CU.
// us per call, float32 MFMA kernels before -> [chosen], others (B, H, L, D causal):
//   (1,4,512,64)  19.0 -> 1x4 [16.8], 2x4 18.8, 4x1 32.5
//   (4,8,1024,64) 82.7 -> 1x4 68.3, 2x4 [43.1], 4x2 48.5, 4x1 60.5
//   (4,8,2048,64) 212 -> 2x4 135, 4x2 [110], 4x1 129
//   (4,8,1024,128) 163 -> 2x2 [85], 4x1 110;  (4,8,2048,128) 411 -> 2x2 295, 4x1 [235]
// Relative error against float64 there: 3.3e-7 -> 2.0e-7 at (4,8,1024,64).
template <int D, bool BIAS, int EXT>
static int launch_f32(const FlashArgs& a, hipStream_t s) {
  const long bh = (long)a.B * a.Hq;
  const bool few = (a.Lq + 127L) / 128 * bh <= 256;
  if constexpr (D == 64) {
    if constexpr (EXT == 0) {
      if ((a.Lq + 31L) / 32 * bh <= 256) return launch_planes<64, 1, 4, 1, 1, BIAS, EXT>(a, s);
      if (!few) return launch_planes<64, 4, 2, 1, 2, BIAS, EXT>(a, s);
    }
    return launch_planes<64, 2, 4, 1, 2, BIAS, EXT>(a, s);
  } else {
    if constexpr (EXT == 0) {
      if (!few) return launch_planes<128, 4, 1, 2, 1, BIAS, EXT>(a, s);
    }
    return launch_planes<128, 2, 2, 1, 1, BIAS, EXT>(a, s);
  }
}

template <int D, bool BIAS>
static int launch_f32_ext(const FlashArgs& a, hipStream_t s) {
  // the general level covers the others
  if (rows_far(a, D)) return launch_planes<D, 2, D == 64 ? 4 : 2, 1, D == 64 ? 2 : 1, BIAS, 3, true>(a, s);
  switch (a.ext) {
    case 0: return launch_f32<D, BIAS, 0>(a, s);
    case 1: return launch_f32<D, BIAS, 1>(a, s);
    case 2: return launch_f32<D, BIAS, 2>(a, s);
    default: return launch_f32<D, BIAS, 3>(a, s);
  }
}

int launch_flash_f32(const FlashArgs& a, int head_dim, hipStream_t s) {
  const bool hb = a.bias != nullptr;
  if (head_dim == 128) return hb ? launch_f32_ext<128, true>(a, s) : launch_f32_ext<128, false>(a, s);
  return hb ? launch_f32_ext<64, true>(a, s) : launch_f32_ext<64, false>(a, s);
}

}  // namespace pjx
