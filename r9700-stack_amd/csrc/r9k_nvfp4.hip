// r9k_nvfp4.hip -- load-time NVFP4 -> MXFP4 conversion with MSE-searched block exponents, on gfx950.
//
// Per 32-element block of a row (reference: r9700_vllm/quant/nvfp4.py:39-90):
//   1. exact dequant  x_i = (E2M1[c_i] * float(s16[i / 16])) / row_div      (fp32 multiply, then fp32 division)
//   2. amax = max(max_i |x_i|, 2^-126);  e0 = ceil(log2(amax / 6)) clamped to [-126, 127]
//   3. for d in (0, -1):  e = clamp(e0 + d, -127, 127);  c_i = nearest E2M1 of x_i / 2^e with ties to the smaller
//      magnitude (torch.bucketize(right=False) on the thresholds 0.25 .. 5.0; > 5 saturates to 6), sign bit set
//      for x_i / 2^e < 0 (so -0.0 encodes as 0, a negative value rounding to zero as 8);
//      err = sum_i (E2M1[c_i] * 2^e - x_i)^2;   the d = -1 candidate wins only if its err is strictly lower
//   4. e8m0 byte = e + 127; codes packed two a byte, element 2i in the low nibble.
// Two places where the reference's torch arithmetic is implementation-defined are computed exactly here:
//   * e0 is the smallest integer e with amax <= 6 * 2^e (frexp), where the reference takes ceil of an fp32 log2;
//     the two differ only when amax / 6 lies within ~2^-20 (relative) above a power of two, which no block with
//     <= 23 significant bits of mantissa above bit 1 reaches -- never for NVFP4-derived values (<= 6 bits);
//   * err is summed in fp64 in ascending i (each term exact in fp64 for fp32 inputs), where torch sums fp32 in an
//     unspecified order; they can only disagree when the two candidates' errors tie within fp32 rounding.
// One thread converts one block: it reads 16 bytes of codes and 2 scale bytes and writes 16 + 1 bytes, so a wave
// streams 1 KB of codes contiguously.
#include "r9k_common.h"

#include <algorithm>

namespace {

using namespace r9k;

// The 8 E2M1 codes of one dword (low nibble first) as fp32 values, exact.
__device__ __forceinline__ void e2m1_decode8(uint32_t w, float (&v)[8]) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0);
  const f2 b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1);
  const f2 c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2);
  const f2 d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
  v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1]; v[4] = c[0]; v[5] = c[1]; v[6] = d[0]; v[7] = d[1];
}

// smallest integer e with a <= 6 * 2^e, for a normal positive fp32 a; past the clamp (128) for +inf, as the
// reference's ceil(log2(inf / 6)) is
__device__ __forceinline__ int exp_no_clip(float a) {
  if (a > 0x1.fffffep127f) return 128;
  int p;
  const float m = frexpf(a, &p);          // a = m * 2^p, m in [0.5, 1)
  return p - 3 + (m > 0.75f ? 1 : 0);     // 6 * 2^e = 0.75 * 2^(e + 3)
}

// The 8 codes of x[0..8) / 2^e, packed low nibble first: for each v = x / 2^e the nearest E2M1 code with ties to the
// smaller magnitude (the reference's bucketize on 0.25 .. 5.0, > 5 saturating to 6), sign bit for v < 0.
// V_CVT_SCALEF32_PK_FP4_F32 (scale 1) converts two values into a byte (four conversions chain the dword); it rounds to
// nearest even and saturates (measured on gfx950 against this rule over 1M values), so it differs exactly at the ties
// whose lower neighbour is odd (|v| = 0.75, 1.75, 3.5, where it takes the even code above) and at -0.0 / NaN (sign or
// code kept; the rule gives 0). One mask subtracts 1 from every tied nibble (its magnitude is >= 2: no borrow), another
// clears every -0.0 / NaN nibble.
__device__ __forceinline__ uint32_t e2m1_encode8(const float* x, int e) {
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = ldexpf(x[j], -e);
  uint32_t w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, v[0], v[1], 1.0f, 0);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[2], v[3], 1.0f, 1);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[4], v[5], 1.0f, 2);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[6], v[7], 1.0f, 3);
  uint32_t tie = 0u, zero = 0u;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const uint32_t b = __float_as_uint(v[j]), t = b & 0x7fffffffu;
    const uint32_t tb = (uint32_t)(t == 0x3f400000u) | (uint32_t)(t == 0x3fe00000u) | (uint32_t)(t == 0x40600000u);
    const uint32_t zb = (uint32_t)(b == 0x80000000u) | (uint32_t)(t > 0x7f800000u);
    tie |= tb << (4 * j);
    zero |= (zb * 0xfu) << (4 * j);
  }
  return (w - tie) & ~zero;
}

// fp32 sum of the squared errors of codes cw at exponent e against the block, each term an fma in ascending order.
// It is within 34 * 2^-24 (relative) of the exact sum whenever it is finite and no term underflows past 2^-100.
__device__ __forceinline__ float block_err32(const float (&x)[32], const uint32_t (&cw)[4], int e) {
  float err = 0.f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    float v[8];
    e2m1_decode8(cw[q], v);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float dv = ldexpf(v[j], e) - x[8 * q + j];
      err = fmaf(dv, dv, err);
    }
  }
  return err;
}

// The reference's comparison sum: fp64 terms added in ascending i (each term's difference exact in fp64).
__device__ __forceinline__ double block_err64(const float (&x)[32], const uint32_t (&cw)[4], int e) {
  double err = 0.0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    float v[8];
    e2m1_decode8(cw[q], v);                              // the codes' values (exact), back at the block scale
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const double dv = (double)ldexpf(v[j], e) - (double)x[8 * q + j];
      err += dv * dv;
    }
  }
  return err;
}

// MSE-searched MXFP4 encode of one 32-element fp32 block: packed codes (4 dwords) and the e8m0 byte. The e0 - 1
// candidate wins when its fp64 error sum (block_err64) is strictly lower. The fp32 sums decide first: each is within
// DELTA (relative) of the exact error and the fp64 sums within ~2^-47, so when the fp32 sums are apart by more than
// that margin the fp64 comparison agrees with them; ties, near-ties and sums outside fp32's safe range fall back to
// the fp64 sums, so the byte and the codes are the same as from the fp64 comparison alone.
__device__ __forceinline__ uint32_t search_block(const float (&x)[32], uint32_t (&best_w)[4]) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(x[i]));
  amax = fmaxf(amax, 0x1p-126f);
  int e0 = exp_no_clip(amax);
  e0 = e0 < -126 ? -126 : (e0 > 127 ? 127 : e0);
  const int e1 = e0 - 1;                                  // >= -127: no clamp needed
  uint32_t c0[4], c1[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    c0[q] = e2m1_encode8(x + 8 * q, e0);
    c1[q] = e2m1_encode8(x + 8 * q, e1);
  }
  const float a = block_err32(x, c0, e0), b = block_err32(x, c1, e1);
  constexpr float DELTA = 1e-5f;                          // > 34 * 2^-24 plus the rounding of these products
  bool take1;
  if (a >= 0x1p-100f && b >= 0x1p-100f && a <= 0x1p120f && b <= 0x1p120f &&
      (b * (1.f + DELTA) < a * (1.f - DELTA) || b * (1.f - DELTA) > a * (1.f + DELTA))) {
    take1 = b < a;
  } else {
    take1 = block_err64(x, c1, e1) < block_err64(x, c0, e0);
  }
#pragma unroll
  for (int q = 0; q < 4; q++) best_w[q] = take1 ? c1[q] : c0[q];
  return (uint32_t)((take1 ? e1 : e0) + 127);
}

// The exact rule on one NVFP4 block, element by element: x = (E2M1[c] * s) / rd, both candidates' fp64 sums in ascending
// order. The path of the few blocks search_nvfp4_block leaves; it recomputes the values per candidate, so that the
// kernel's registers (and waves a SIMD) stay those of the common path.
__device__ __forceinline__ uint32_t search_nvfp4_block_exact(const uint4 pk, uint32_t sc, float rd,
                                                             uint32_t (&bw)[4]) {
  // dword q's values; the loops below stay rolled and select by q, so no value is kept from one pass to the next
  auto values = [&](int q, float (&x)[8]) {
    const float s = e4m3_to_f32(q < 2 ? sc & 0xffu : sc >> 8);
    e2m1_decode8(q == 0 ? pk.x : (q == 1 ? pk.y : (q == 2 ? pk.z : pk.w)), x);
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = (x[j] * s) / rd;
  };
  float x[8], amax = 0.f;
#pragma unroll 1
  for (int q = 0; q < 4; q++) {
    values(q, x);
#pragma unroll
    for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(x[j]));
  }
  amax = fmaxf(amax, 0x1p-126f);
  int e0 = exp_no_clip(amax);
  e0 = e0 < -126 ? -126 : (e0 > 127 ? 127 : e0);
  double best = 0.0;
  uint32_t eb = 0u;
#pragma unroll 1
  for (int d = 0; d < 2; d++) {
    uint32_t c[4] = {0u, 0u, 0u, 0u};
    double err = 0.0;
#pragma unroll 1
    for (int q = 0; q < 4; q++) {
      values(q, x);
      const uint32_t cw = e2m1_encode8(x, e0 - d);
#pragma unroll
      for (int i = 0; i < 4; i++) c[i] = i == q ? cw : c[i];
      float v[8];
      e2m1_decode8(cw, v);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const double dv = (double)ldexpf(v[j], e0 - d) - (double)x[j];
        err += dv * dv;
      }
    }
    if (d == 0 || err < best) {
      best = err;
      eb = (uint32_t)(e0 - d + 127);
#pragma unroll
      for (int i = 0; i < 4; i++) bw[i] = c[i];
    }
  }
  return eb;
}

// ---- the search on an NVFP4 block by its magnitudes
// A group's 16 values are (+-) the 7 nonzero E2M1 magnitudes times one quotient, so a candidate's codes and errors are
// functions of (group, magnitude): at exponent e0 the scaled values are V = {.5 r1, r1, r3, 2 r1, 2 r3, 4 r1, 4 r3}
// (r1 = q1 2^-e0, r3 = q3 2^-e0, with the IEEE quotients q1 = s / rd and q3 = 1.5 s / rd; scaling a correctly rounded
// quotient by a power of two is exact while it stays normal, so these are the element-wise values), and at
// e0 - 1, twice those: the same list two entries further, so 9 encodes serve both candidates of a group where the
// element-wise search does 32. The 16 codes then go through an 8-byte table (v_perm_b32 looks up four at a time), and
// the error sums weigh each magnitude's square by its count (population counts over the code bits). Bound: VALU, ~490
// instructions a block against ~1540 element by element; 17408 x 5120 in one launch 109 -> 53 us (1.85 TB/s of its
// 97.5 MB), 70 us where many blocks' candidates tie exactly (divisor 1: they take the exact search).
struct GroupTab {
  uint32_t lo[2], hi[2];                                   // candidate d: table bytes of magnitudes 0-3 and 4-7
  float err[2];                                            // scaled error sums (at e0 and at e0 - 1)
};

// Counts of the 7 nonzero magnitudes (n[1..7]) among the 16 codes of a group.
__device__ __forceinline__ void mag_counts(uint32_t w0, uint32_t w1, int (&n)[8]) {
  constexpr uint32_t M = 0x11111111u;
  const uint32_t b0 = (w0 & M) | ((w1 & M) << 1), b1 = ((w0 >> 1) & M) | (w1 & (M << 1)),
                 b2 = ((w0 >> 2) & M) | ((w1 >> 1) & (M << 1));
  const uint32_t b21 = b2 & b1;
  const int c7 = __popc(b21 & b0), c21 = __popc(b21), c20 = __popc(b2 & b0), c10 = __popc(b1 & b0);
  n[7] = c7;
  n[6] = c21 - c7;
  n[5] = c20 - c7;
  n[3] = c10 - c7;
  n[4] = __popc(b2) - c21 - n[5];
  n[2] = __popc(b1) - c21 - n[3];
  n[1] = __popc(b0) - c20 - n[3];
}

// The largest value among the codes counted in n.
__device__ __forceinline__ float group_max(const int (&n)[8], float q1, float q3) {
  float m = n[1] ? 0.5f * q1 : 0.f;
  m = n[2] ? q1 : m;
  m = n[3] ? q3 : m;
  m = n[4] ? 2.f * q1 : m;
  m = n[5] ? 2.f * q3 : m;
  m = n[6] ? 4.f * q1 : m;
  return n[7] ? 4.f * q3 : m;
}

__device__ __forceinline__ void group_table(const int (&n)[8], float q1, float q3, int e0, GroupTab& t) {
  const float r1 = ldexpf(q1, -e0), r3 = ldexpf(q3, -e0);
  const float v[9] = {0.5f * r1, r1, r3, 2.f * r1, 2.f * r3, 4.f * r1, 4.f * r3, 8.f * r1, 8.f * r3};
  // codes of the 9 values, one a byte (e2m1_encode8's rule: nearest, a tie whose lower neighbour is odd one step down)
  uint32_t p[3] = {0u, 0u, 0u}, tie[3] = {0u, 0u, 0u};
#define R9K_ENC(I)                                                                                                  \
  {                                                                                                                 \
    p[(I) >> 2] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(p[(I) >> 2], v[I], 0.f, 1.0f, (I) & 3);                  \
    const bool tb = v[I] == 0.75f || v[I] == 1.75f || v[I] == 3.5f;                                                 \
    tie[(I) >> 2] |= tb ? 1u << (8 * ((I) & 3)) : 0u;                                                               \
  }
  R9K_ENC(0) R9K_ENC(1) R9K_ENC(2) R9K_ENC(3) R9K_ENC(4) R9K_ENC(5) R9K_ENC(6) R9K_ENC(7) R9K_ENC(8)
#undef R9K_ENC
#pragma unroll
  for (int i = 0; i < 3; i++) p[i] -= tie[i];
  float sq[9];                                             // squared scaled errors
#define R9K_ERR(I)                                                                                 \
  {                                                                                                \
    const float d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(p[(I) >> 2], 1.0f, (I) & 3)[0] - v[I]; \
    sq[I] = d * d;                                                                                 \
  }
  R9K_ERR(0) R9K_ERR(1) R9K_ERR(2) R9K_ERR(3) R9K_ERR(4) R9K_ERR(5) R9K_ERR(6) R9K_ERR(7) R9K_ERR(8)
#undef R9K_ERR
  float a = 0.f, b = 0.f;
  constexpr int I1[8] = {0, 1, 3, 4, 5, 6, 7, 8};          // magnitude m at e0 - 1: entry I1[m]; at e0: entry m - 1
#pragma unroll
  for (int m = 1; m < 8; m++) {
    const float c = (float)n[m];
    a = fmaf(c, sq[m - 1], a);
    b = fmaf(c, sq[I1[m]], b);
  }
  t.err[0] = a;
  t.err[1] = b;
  // bit 3 of a table byte lets the code's sign through: clear for magnitude 0, and for all of a group whose scale is 0
  // (its values are +-0, which encode as 0)
  const uint32_t f = q1 > 0.f ? 0x08080808u : 0u;
  t.lo[0] = (p[0] << 8) | (f << 8);                                            // 0, C0, C1, C2
  t.hi[0] = __builtin_amdgcn_perm(p[1], p[0], 0x06050403u) | f;                // C3, C4, C5, C6
  t.lo[1] = (__builtin_amdgcn_perm(p[1], p[0], 0x0403010cu) & 0xffffff00u) | (f << 8);   // 0, C1, C3, C4
  t.hi[1] = __builtin_amdgcn_perm(p[2], p[1], 0x04030201u) | f;                // C5, C6, C7, C8
}

// The 8 codes of w through a group's table for one candidate.
__device__ __forceinline__ uint32_t map_codes(uint32_t w, uint32_t lo, uint32_t hi) {
  const uint32_t even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
  const uint32_t re = __builtin_amdgcn_perm(hi, lo, even & 0x07070707u) & (even | 0x07070707u);
  const uint32_t ro = __builtin_amdgcn_perm(hi, lo, odd & 0x07070707u) & (odd | 0x07070707u);
  return re | (ro << 4);
}

// One NVFP4 block by its magnitudes; false when it needs the element-wise search: a group whose quotients could
// leave the normal range, a negative or NaN scale or divisor, or error sums too close (or too small) for fp32 to order. The scaled sums are those
// of block_err32 times 2^(-2 e): S1 / 4 against S0 is the same comparison, and each carries fewer roundings (7 terms a
// group, each one subtraction, one square and one fma) than the 34 * 2^-24 that search_block's margin covers.
__device__ __forceinline__ bool search_nvfp4_block(const uint4 pk, uint32_t sc, float rd, uint32_t (&bw)[4],
                                                   uint32_t& eb) {
  const float s0 = e4m3_to_f32(sc & 0xffu), s1 = e4m3_to_f32(sc >> 8);
  const float q1[2] = {s0 / rd, s1 / rd}, q3[2] = {(1.5f * s0) / rd, (1.5f * s1) / rd};
  bool ok = (sc & 0x8080u) == 0u && rd > 0.f && rd <= 3.0e38f;
#pragma unroll
  for (int g = 0; g < 2; g++) ok = ok && (q1[g] >= 0x1p-125f || q1[g] == 0.f) && q3[g] <= 0x1p125f;
  int n[2][8];
  mag_counts(pk.x, pk.y, n[0]);
  mag_counts(pk.z, pk.w, n[1]);
  const float amax = fmaxf(fmaxf(group_max(n[0], q1[0], q3[0]), group_max(n[1], q1[1], q3[1])), 0x1p-126f);
  int e0 = exp_no_clip(amax);
  e0 = e0 < -126 ? -126 : (e0 > 127 ? 127 : e0);
  GroupTab t[2];
  group_table(n[0], q1[0], q3[0], e0, t[0]);
  group_table(n[1], q1[1], q3[1], e0, t[1]);
  const float a = t[0].err[0] + t[1].err[0], b = 0.25f * (t[0].err[1] + t[1].err[1]);
  constexpr float DELTA = 1e-5f;
  // a sum of exactly 0 is an exact 0 (values from 2^-38 up differ from a code by 0 or by 2^-62 and more, whose square
  // does not underflow), so it decides by itself: common, with power-of-two ratios of scale and divisor
  const bool zero = a == 0.f || b == 0.f;
#pragma unroll
  for (int g = 0; g < 2; g++) ok = ok && (q1[g] == 0.f || ldexpf(q1[g], -e0) >= 0x1p-37f);
  ok = ok && (zero || (a >= 0x1p-90f && b >= 0x1p-90f && a <= 0x1p120f && b <= 0x1p120f &&
                       (b * (1.f + DELTA) < a * (1.f - DELTA) || b * (1.f - DELTA) > a * (1.f + DELTA))));
  if (!ok) return false;
  const bool take1 = b < a;
  eb = (uint32_t)(e0 + 127 - (take1 ? 1 : 0));
  const uint32_t w[4] = {pk.x, pk.y, pk.z, pk.w};
#pragma unroll
  for (int g = 0; g < 2; g++) {
    const uint32_t lo = take1 ? t[g].lo[1] : t[g].lo[0], hi = take1 ? t[g].hi[1] : t[g].hi[0];
    bw[2 * g] = map_codes(w[2 * g], lo, hi);
    bw[2 * g + 1] = map_codes(w[2 * g + 1], lo, hi);
  }
  return true;
}

__global__ void __launch_bounds__(256) nvfp4_to_mxfp4_kernel(const uint8_t* __restrict__ packed,
                                                             const uint8_t* __restrict__ s16,
                                                             const float* __restrict__ row_div,
                                                             uint8_t* __restrict__ out_p, uint8_t* __restrict__ out_e,
                                                             uint32_t nblk, DivMagic bpr) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblk) return;
  const uint4 pk = *reinterpret_cast<const uint4*>(packed + (size_t)b * 16);
  const uint32_t sc = *reinterpret_cast<const uint16_t*>(s16 + (size_t)b * 2);
  const float rd = row_div[div_by(b, bpr)];
  uint32_t bw[4], eb;
  if (!search_nvfp4_block(pk, sc, rd, bw, eb)) eb = search_nvfp4_block_exact(pk, sc, rd, bw);
  *reinterpret_cast<uint4*>(out_p + (size_t)b * 16) = make_uint4(bw[0], bw[1], bw[2], bw[3]);
  out_e[b] = (uint8_t)eb;
}

// (E2M1[c] * s) / rd for the 16 codes of one group, with IEEE division semantics, from two divisions: every E2M1
// magnitude is 2^j or 1.5 * 2^j, and scaling a correctly rounded quotient by 2^j is exact while it stays normal, so
// RN(1.5^b * 2^j * s / rd) = 2^j * RN(1.5^b * s / rd). Groups whose quotients could leave the normal range (or a
// non-finite / non-positive divisor) divide per element.
__device__ __forceinline__ void dequant_group(const uint32_t w0, const uint32_t w1, float s, float rd, float* x) {
  const float q1 = s / rd, q3 = (1.5f * s) / rd;
  const float aq1 = fabsf(q1), aq3 = fabsf(q3);
  const bool fast = (aq1 >= 0x1p-125f || aq1 == 0.f) && aq3 <= 0x1p125f && rd > 0.f && rd <= 3.0e38f;
  float v[16];
  e2m1_decode8(w0, *reinterpret_cast<float(*)[8]>(v));
  e2m1_decode8(w1, *reinterpret_cast<float(*)[8]>(v + 8));
  if (fast) {
    // V = E2M1[c] = +-2^j (mantissa bit clear) or +-1.5 * 2^j (set): x = (V with its mantissa cleared) * (q1 or q3)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const uint32_t vb = __float_as_uint(v[i]);
      x[i] = __uint_as_float(vb & 0xff800000u) * ((vb & 0x00400000u) ? q3 : q1);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = (v[i] * s) / rd;
  }
}

// The conversion of weights too small to fill the chip, element by element (search_block on the block's values): there
// a launch takes as long as its longest wave, and a wave with one block for search_nvfp4_block_exact takes that serial
// path's ~10 us. Blocks, this kernel -> the other, us: 8192 (512 x 512) 6.9 -> 12.0, 65536 (1024 x 2048) 7.0 -> 13-17,
// 2^19 (4096 x 4096) 20.4-23.0 -> 19.2-21.3 (22.6 -> 27.6 at divisor 1, whose candidates often tie), 2.8M (17408 x 5120)
// 85-93 -> 47-62. Same codes and bytes.
constexpr long SMALL_BLOCKS = 1L << 19;

__global__ void __launch_bounds__(256) nvfp4_to_mxfp4_small_kernel(const uint8_t* __restrict__ packed,
                                                                   const uint8_t* __restrict__ s16,
                                                                   const float* __restrict__ row_div,
                                                                   uint8_t* __restrict__ out_p,
                                                                   uint8_t* __restrict__ out_e, uint32_t nblk,
                                                                   DivMagic bpr) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblk) return;
  const uint4 pk = *reinterpret_cast<const uint4*>(packed + (size_t)b * 16);
  const uint32_t sc = *reinterpret_cast<const uint16_t*>(s16 + (size_t)b * 2);
  const float rd = row_div[div_by(b, bpr)];
  const float s0 = e4m3_to_f32(sc & 0xffu), s1 = e4m3_to_f32(sc >> 8);
  float x[32];
  dequant_group(pk.x, pk.y, s0, rd, x);
  dequant_group(pk.z, pk.w, s1, rd, x + 16);
  uint32_t bw[4];
  const uint32_t eb = search_block(x, bw);
  *reinterpret_cast<uint4*>(out_p + (size_t)b * 16) = make_uint4(bw[0], bw[1], bw[2], bw[3]);
  out_e[b] = (uint8_t)eb;
}

// fp32 weights [N, K] (row stride ld floats) -> MXFP4 by the same search (quantize_mxfp4_search on any weight).
__global__ void __launch_bounds__(256) mxfp4_search_kernel(const float* __restrict__ w, long ld,
                                                           uint8_t* __restrict__ out_p, uint8_t* __restrict__ out_e,
                                                           long nblk, int bpr) {
  const long b = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblk) return;
  const long row = b / bpr, col = (b - row * bpr) * 32;
  const float4* src = reinterpret_cast<const float4*>(w + row * ld + col);
  float x[32];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 v = src[i];
    x[4 * i] = v.x; x[4 * i + 1] = v.y; x[4 * i + 2] = v.z; x[4 * i + 3] = v.w;
  }
  uint32_t bw[4];
  const uint32_t eb = search_block(x, bw);
  *reinterpret_cast<uint4*>(out_p + b * 16) = make_uint4(bw[0], bw[1], bw[2], bw[3]);
  out_e[b] = (uint8_t)eb;
}

}  // namespace

// New entry point (no reference C symbol: the reference converts with torch, r9700_vllm/quant/nvfp4.py:78-90).
// packed [N, K/2] u8, s16 [N, K/16] e4m3 bytes, row_div [N] fp32 -> out_packed [N, K/2] u8, out_e8m0 [N, K/32] u8,
// all contiguous, 16-byte aligned codes. 0 / -2 K % 32 / -3 bad pointer / -6 launch error.
extern "C" int r9k_nvfp4_to_mxfp4(long packed, long s16, long row_div, long out_packed, long out_e8m0, int N, int K,
                                  long stream) {
  if (N <= 0) return 0;
  if (K <= 0 || K % 32) return -2;
  if (!packed || !s16 || !row_div || !out_packed || !out_e8m0 || (packed & 15) || (out_packed & 15) || (s16 & 1))
    return -3;
  const int bpr = K / 32;
  // rows in launches of less than 2^31 blocks (32-bit indices in the kernel)
  const long step = std::max(1L, 0x7fffff00L / bpr);
  for (long r0 = 0; r0 < N; r0 += step) {
    const long n = std::min(step, N - r0) * bpr, b0 = r0 * bpr;
    hipLaunchKernelGGL(n <= SMALL_BLOCKS ? nvfp4_to_mxfp4_small_kernel : nvfp4_to_mxfp4_kernel,
                       dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)packed + b0 * 16, (const uint8_t*)s16 + b0 * 2, (const float*)row_div + r0,
                       (uint8_t*)out_packed + b0 * 16, (uint8_t*)out_e8m0 + b0, (uint32_t)n, div_magic((uint32_t)bpr));
    if (hipGetLastError() != hipSuccess) return -6;
  }
  return 0;
}

// fp32 [N, K] (row stride ld floats, 16-byte aligned rows) -> out_packed [N, K/2] u8, out_e8m0 [N, K/32] u8 with the
// same MSE search (reference: r9700_vllm/quant/nvfp4.py:54-75 on an arbitrary fp32 weight). 0 / -2 / -3 / -6.
extern "C" int r9k_quantize_mxfp4_search(long w, long out_packed, long out_e8m0, int N, int K, long stream) {
  if (N <= 0) return 0;
  if (K <= 0 || K % 32) return -2;
  if (!w || !out_packed || !out_e8m0 || (w & 15) || (out_packed & 15)) return -3;
  const int bpr = K / 32;
  const long nblk = (long)N * bpr;
  const long grid = (nblk + 255) / 256;
  if (grid > 0x7fffffffL) return -3;
  hipLaunchKernelGGL(mxfp4_search_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, (const float*)w,
                     (long)K, (uint8_t*)out_packed, (uint8_t*)out_e8m0, nblk, bpr);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}
