// float32 products on the bf16 matrix units, without losing float32 precision.
//
// A float32 value is the sum of three bf16 values (three times 8 significant
// bits, rounded to nearest at each step, cover its 24): x = h + m + l exactly,
// as long as l does not fall below bf16's range.  A product of two such sums
// has nine terms; the six of order h*h, h*m, m*h, m*m, h*l, l*h are formed as
// bf16 MFMAs with fp32 accumulation, and the three left out (m*l, l*m, l*l)
// are below 2^-25 of the product, half an ulp of float32.  Six
// v_mfma_f32_32x32x16_bf16 of 32 cycles contract 16 indices where
// v_mfma_f32_32x32x2f32 takes 8 of 64 cycles: 192 against 512 cycles.
//
// Range: where h*h overflows, h*m and m*h (2^-9 of it, of either sign) may
// overflow to the other infinity, and an infinite plane times another operand's
// zero plane is NaN; a float32 product gives its one infinity.  Up to kPlaneMax
// no product of two operands, nor the sum of any row of them, overflows.  Tiles
// with a larger value are flagged where they are split and take the float32
// MFMAs from memory instead, so that infinities and large values give what they
// give there.  At the other end l falls below bf16's range, where its spacing is
// 2^-133: of 8 consecutive values whose largest is at least kPlaneMin none is
// off by more than 2^-34 of that one.  8 values below it that are not all zeros
// are flagged like large ones.
// The backward splits an intermediate too, dS = P w with w = scale (dP - delta),
// and w may lie beyond the range of ordinary operands' planes: V of standard
// deviation 2^-118 gave dq and dk a relative error of 1.1e-3, and an overflowing
// dS, whose planes are an infinity and NaNs, NaN for an infinity.  Between
// kSureMin and kSureMax (scale within 2^10 of 1) no operands can do so: dS K and
// dS Q stay below 2^110 a term, and dP's own float32 rounding is above the 2^-134
// that a plane may lose.  Tiles with other operands look at dP and delta, and
// where a lane's largest, times scale, is above kPlaneMax or below kScoreGradMin
// the products of P and dS take the float32 MFMAs.  Backward of (B, H, L, D), us
// without this and with it: (4, 8, 1024, 64) 124 -> 125, (4, 8, 1024, 128) 277
// -> 279, (4, 8, 2048, 128) 786 -> 805.
#pragma once

#include "flash_common.h"

// A stage's loads and stores share registers: called out of line they would go
// through scratch memory (forward of (1, 4, 512, 64) 16.9 -> 31.4 us).
#define PJX_INLINE_LAMBDA __attribute__((always_inline))

namespace pjx {

constexpr float kPlaneMax = 0x1p60f, kPlaneMin = 0x1p-100f;
constexpr float kSureMax = 0x1p30f, kSureMin = 0x1p-40f, kSureScale = 0x1p10f, kScoreGradMin = 0x1p-90f;
constexpr float kSureScoreGrad = 0x1p77f;  // of delta * scale

// Eight consecutive values as three bf16 operands.
struct Planes {
  bf16x8 h, m, l;
};

__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack_bf16x2(a, b);
  a -= Bf16Fmt::lo(h);
  b -= Bf16Fmt::hi(h);
  m = pack_bf16x2(a, b);
  a -= Bf16Fmt::lo(m);
  b -= Bf16Fmt::hi(m);
  l = pack_bf16x2(a, b);
}

__device__ __forceinline__ void split8(const float* x, u32x4& h, u32x4& m, u32x4& l) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t a, b, c;
    split2(x[2 * j], x[2 * j + 1], a, b, c);
    h[j] = a;
    m[j] = b;
    l[j] = c;
  }
}

__device__ __forceinline__ Planes planes8(const float* x) {
  u32x4 h, m, l;
  split8(x, h, m, l);
  return {Bf16Fmt::as8(h), Bf16Fmt::as8(m), Bf16Fmt::as8(l)};
}

// Registers 8c .. 8c+7 of a 32x32 C block as the B operand of k-step c.
__device__ __forceinline__ Planes planes_step(const f32x16& x, int c) {
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = x[8 * c + j];
  return planes8(v);
}

// The range of the chunks of 8 consecutive values seen so far: the largest
// chunk's and the smallest non-zero one's largest magnitude, as bits (`lo` less
// one, so that a chunk of zeros is none): three operations a chunk, compared
// once a stage.
struct PlaneSpan {
  uint32_t hi = 0u, lo = ~0u;
  __device__ __forceinline__ void add(const float* x) {
    float m = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(x[j]));
    hi = max(hi, __float_as_uint(m));
    lo = min(lo, __float_as_uint(m) - 1u);
  }
  __device__ __forceinline__ bool beyond(float least, float most) const {
    return (hi > __float_as_uint(most)) | (lo < __float_as_uint(least) - 1u);
  }
  // beyond the planes' range; dS formed from them may be
  __device__ __forceinline__ bool beyond_planes() const { return beyond(kPlaneMin, kPlaneMax); }
  __device__ __forceinline__ bool beyond_sure() const { return beyond(kSureMin, kSureMax); }
};

__device__ __forceinline__ bool scale_beyond_sure(float scale) {
  return !(fabsf(scale) <= kSureScale && fabsf(scale) >= 1.f / kSureScale);
}

// Whether the dS of any lane of the wave is: its 16 dP and delta, times scale.
__device__ __forceinline__ bool score_grads_beyond_planes(const f32x16& dp, float delta, float scale) {
  float m = fabsf(delta);
#pragma unroll
  for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(dp[r]));
  m *= fabsf(scale);
  return wave_any(m > kPlaneMax || (m > 0.f && m < kScoreGradMin));
}

// c += a b over 16 indices, smallest terms first.  With SWAP the terms come in the
// order of b a, so that scores formed as Q K^T are the bits of those formed as
// K Q^T: P in the dK/dV kernel then has the forward's rounding, not another of
// its own (relative error of dv against float64 at scores of a few hundred,
// L = 1024, D = 64: 1.0e-5 without, float32 MFMAs 9.3e-6).
template <bool SWAP = false>
__device__ __forceinline__ f32x16 mma_planes(const Planes& a, const Planes& b, f32x16 c) {
  c = SWAP ? Bf16Fmt::mma32(a.h, b.l, c) : Bf16Fmt::mma32(a.l, b.h, c);
  c = SWAP ? Bf16Fmt::mma32(a.l, b.h, c) : Bf16Fmt::mma32(a.h, b.l, c);
  c = Bf16Fmt::mma32(a.m, b.m, c);
  c = SWAP ? Bf16Fmt::mma32(a.h, b.m, c) : Bf16Fmt::mma32(a.m, b.h, c);
  c = SWAP ? Bf16Fmt::mma32(a.m, b.h, c) : Bf16Fmt::mma32(a.h, b.m, c);
  return Bf16Fmt::mma32(a.h, b.h, c);
}

// 16 bytes at byte offset `off` of a buffer; zeros past its end.
__device__ __forceinline__ f32x4 buffer_load_f32x4(rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// A tile of ROWS float32 rows of D values held in LDS as three bf16 planes of
// row-major rows, 16-byte chunks XOR-swizzled per row (the swizzle of the
// 16-bit backward tiles: both the 16-byte reads of a row block and the
// transposing reads are free of bank conflicts).
template <int D, int ROWS>
struct PlaneTile {
  static constexpr int ROWB = D * 2;
  static constexpr int NC = D / 8;  // 16-byte chunks per row and plane
  static constexpr int PLANE_B = ROWS * ROWB;
  static constexpr int BYTES = 3 * PLANE_B;
  __device__ static int swz(int r) {
    return D >= 128 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
  }
  __device__ static void store(unsigned char* tile, uint32_t off, const float* x) {
    u32x4 h, m, l;
    split8(x, h, m, l);
    *(u32x4*)(tile + off) = h;
    *(u32x4*)(tile + off + PLANE_B) = m;
    *(u32x4*)(tile + off + 2 * PLANE_B) = l;
  }
  __device__ static uint32_t chunk(int row, int c) { return row * ROWB + 16 * (c ^ swz(row)); }
  // A operand X[row][dim] of a 32-row block: `off` = chunk(col, 2 * step + half)
  __device__ static Planes rows(const unsigned char* tile, int row0, uint32_t off) {
    const unsigned char* p = tile + row0 * ROWB + off;
    return {Bf16Fmt::as8(*(const u32x4*)p), Bf16Fmt::as8(*(const u32x4*)(p + PLANE_B)),
            Bf16Fmt::as8(*(const u32x4*)(p + 2 * PLANE_B))};
  }
  // A operand X^T (32 dims, 16 rows from row0 in slot order 8*(j/4) + 4*half + j%4)
  __device__ static bf16x8 cols1(const unsigned char* p, uint32_t lo, uint32_t hi) {
    const u32x2 a = lds_read_tr16(p + lo), b = lds_read_tr16(p + hi);
    return Bf16Fmt::as8(u32x4{a[0], a[1], b[0], b[1]});
  }
  __device__ static Planes cols(const unsigned char* tile, int row0, uint32_t lo, uint32_t hi) {
    const unsigned char* p = tile + row0 * ROWB;
    return {cols1(p, lo, hi), cols1(p + PLANE_B, lo, hi), cols1(p + 2 * PLANE_B, lo, hi)};
  }
};

// The rows one wave loads with one instruction, 64 / (D/8) of them from row
// `row` (the same in every lane) of a tensor with `row_bytes` between rows, as
// a buffer: lane offsets stay below 8 rows whatever the tensor's size, and
// rows at or past `end` read as zeros.
template <int D>
__device__ __forceinline__ rsrc_t wave_rows(const unsigned char* base, int row, int end, uint32_t row_bytes, int rdim) {
  const int n = min(end - row, 512 / D);
  return make_rsrc(base + (size_t)(n > 0 ? row : 0) * row_bytes, n > 0 ? (uint32_t)(n - 1) * row_bytes + rdim * 4 : 0u);
}
template <int D>
__device__ __forceinline__ uint32_t wave_rows_offset(uint32_t row_bytes, int rdim) {
  const int lane = threadIdx.x & 63, c = lane % (D / 8);
  return 8 * c < rdim ? (lane / (D / 8)) * row_bytes + 32 * c : kPastBuffer;
}

// Geometry of a workgroup of `rows` query rows whose wave owns rows 32*strip ..
// (a.n_qtiles counts tiles of `rows`; heaviest causal tile first, batch*head
// fastest, as block_geom).
__device__ __forceinline__ BlockGeom plane_geom(const FlashArgs& a, int idx, int rows, int strip) {
  BlockGeom g;
  const int BH = a.B * a.Hq;
  const int bh = idx % BH;
  g.b = bh / a.Hq;
  g.h = bh % a.Hq;
  g.hkv = g.h / (a.Hq / a.Hkv);
  g.q0 = (a.n_qtiles - 1 - idx / BH) * rows;
  g.qw = g.q0 + 32 * strip;
  g.qi = g.qw + (threadIdx.x & 31);
  g.q_hi = min(a.Lq, a.q_valid);
  int kv_end = min(a.Lk, a.kv_valid);
  if (a.kv_lengths) kv_end = min(kv_end, max(a.kv_lengths[g.b], 0));
  g.kv_end = kv_end;
  int stop = kv_end;
  if (g.q0 >= g.q_hi) {
    stop = 0;
  } else if (a.causal) {
    stop = min(stop, min(g.q0 + rows, g.q_hi));
  }
  g.kv_stop = stop;
  g.kv_begin = 0;
  return g;
}

// Per-lane offsets of a tile's two read patterns.
template <int D>
struct PlaneOffsets {
  using T = PlaneTile<D, 32>;
  uint32_t row[D / 16], tlo[D / 32], thi[D / 32];
  __device__ void init(int lane) {
    const int col = lane & 31, half = lane >> 5;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) row[s] = T::chunk(col, 2 * s + half);
    const int s16 = lane & 15, grp = lane >> 4;
    const int r = 4 * half + s16 / 4;
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      const int c = 4 * db + 2 * (grp & 1) + ((s16 & 3) >> 1);
      tlo[db] = T::chunk(r, c) + 8 * (s16 & 1);
      thi[db] = T::chunk(r + 8, c) + 8 * (s16 & 1);
    }
  }
};

}  // namespace pjx
