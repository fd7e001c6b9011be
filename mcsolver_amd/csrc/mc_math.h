// Deterministic FP32 primitives shared by every MI355X kernel of the engine.
//
// Every function here is a fixed sequence of IEEE-754 single-precision
// operations (explicit fmaf, correctly rounded sqrt/div, no contraction: the
// library is compiled with -ffp-contract=off), so its result does not depend
// on how the compiler schedules it.  That is what lets a CPU checker that
// performs the same sequence reproduce the GPU sweep bit for bit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcg {

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon et al., SC'11): counter-based, 4x32-bit output per
// (counter, key).  Multipliers and Weyl increments are the paper's.
// ---------------------------------------------------------------------------
struct u32x4 {
  uint32_t x, y, z, w;
};

// a ^ b ^ c: one v_bitop3_b32 on the device (the compiler splits the three-way
// xor into two instructions by itself; a draw has 20 of them)
__host__ __device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0x96);
#else
  return a ^ b ^ c;
#endif
}

__host__ __device__ __forceinline__ u32x4 philox4x32_10(u32x4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    c = u32x4{xor3((uint32_t)(p1 >> 32), c.y, k0), (uint32_t)p1, xor3((uint32_t)(p0 >> 32), c.w, k1), (uint32_t)p0};
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// Philox counter tags: which random decision a draw belongs to.
enum : uint32_t {
  TAG_METRO = 0,   // single-site Metropolis update (site, sweep)
  TAG_MAJORITY = 1,// block-spin majority tie break (site, frame)
  TAG_WOLFF = 2,   // Wolff seed + direction + cluster accept (cluster)
  TAG_BOND = 3,    // Wolff bond activation (link, cluster)
  TAG_PT = 4,      // parallel-tempering pair (pair, sweep)
};

// uniform in [0,1) on the 2^-24 grid, exact in float
__host__ __device__ __forceinline__ float u24(uint32_t v) { return (float)(v >> 8) * 0x1p-24f; }

// exp(x) for x <= 0.  Cody-Waite reduction x = k ln2 + r, |r| <= ln2/2, then
// the degree-7 Taylor polynomial of e^r (truncation < 1e-8 relative) and an
// exact scaling by 2^k.  Returns 0 below -80 (e^-80 < 2^-115).
__host__ __device__ __forceinline__ float exp_neg(float x) {
  if (x < -80.0f) return 0.0f;
  const float k = floorf(fmaf(x, 1.44269504088896341f, 0.5f));
  float r = fmaf(k, -0.693145751953125f, x);
  r = fmaf(k, -1.42860682030941723e-6f, r);
  float p = 1.98412698412698413e-4f;
  p = fmaf(p, r, 1.38888888888888889e-3f);
  p = fmaf(p, r, 8.33333333333333333e-3f);
  p = fmaf(p, r, 4.16666666666666667e-2f);
  p = fmaf(p, r, 1.66666666666666667e-1f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  const int ki = (int)k;
  const float scale = __builtin_bit_cast(float, (uint32_t)(ki + 127) << 23);
  return p * scale;
}

// u24(v) < exp(x), for x <= 0: both sides scaled by 2^24, which is exact (the
// draw becomes its integer, the scale 2^k becomes 2^(k+24)).  The same
// operations on r as exp_neg; x < -80 (or NaN) rejects.
__host__ __device__ __forceinline__ bool below_exp(uint32_t v, float x) {
  const float k = floorf(fmaf(x, 1.44269504088896341f, 0.5f));
  float r = fmaf(k, -0.693145751953125f, x);
  r = fmaf(k, -1.42860682030941723e-6f, r);
  float p = 1.98412698412698413e-4f;
  p = fmaf(p, r, 1.38888888888888889e-3f);
  p = fmaf(p, r, 8.33333333333333333e-3f);
  p = fmaf(p, r, 4.16666666666666667e-2f);
  p = fmaf(p, r, 1.66666666666666667e-1f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  const int ki = (int)k;
  const float scale24 = __builtin_bit_cast(float, (uint32_t)(ki + (127 + 24)) << 23);
  return (x >= -80.0f) & ((float)(v >> 8) < p * scale24);
}

// rho = sqrt(1 - rz^2) for a draw's rz = 2 u24 - 1, correctly rounded: on the
// device one Newton step from v_rsq_f32, 6 instructions instead of the 16 of
// the general correctly rounded sqrtf; compared with it over all 2^24 values
// of rz on gfx950: no difference.  1 - rz^2 is 0 or at least 2^-24, so the
// clamp only keeps rsq finite at 0 (then s = 0 and rho = 0).
__host__ __device__ __forceinline__ float unit_rho(float rz) {
  const float x = fmaf(-rz, rz, 1.0f);
#if defined(__HIP_DEVICE_COMPILE__)
  const float y = __builtin_amdgcn_rsqf(fmaxf(x, 0x1p-100f));
  const float s = x * y, e = fmaf(-s, s, x);
  return fmaf(e, 0.5f * y, s);
#else
  return sqrtf(fmaxf(x, 0.0f));
#endif
}

// (cos phi, sin phi) for phi = 2*pi*(v / 2^32): octant from the top three
// bits, a 24-bit fraction inside it, Taylor polynomials of sin and cos on
// [0, pi/4] and exact octant symmetries.  An odd octant folds the fraction f
// to 1 - f; the bits 29..5 of v as a signed number are f in an even octant
// and f - 1 in an odd one (units of 2^-24), so the angle is that number's
// magnitude, and its sign drops out where the octant's signs are set.
__host__ __device__ __forceinline__ void sincos_turn(uint32_t v, float* c, float* s) {
  const int32_t m = (int32_t)(v << 2) >> 7;
  const float a = (float)m * (0.785398163397448310f * 0x1p-24f);
  const float a2 = a * a;
  float ps = 2.75573192239858907e-6f;
  ps = fmaf(ps, a2, -1.98412698412698413e-4f);
  ps = fmaf(ps, a2, 8.33333333333333333e-3f);
  ps = fmaf(ps, a2, -1.66666666666666667e-1f);
  const float sn = fmaf(a, a2 * ps, a);
  float pc = -2.75573192239858907e-7f;
  pc = fmaf(pc, a2, 2.48015873015873016e-5f);
  pc = fmaf(pc, a2, -1.38888888888888889e-3f);
  pc = fmaf(pc, a2, 4.16666666666666667e-2f);
  pc = fmaf(pc, a2, -0.5f);
  const float cs = fmaf(pc, a2, 1.0f);
  // Octants 1,2,5,6 swap (cos, sin); cos < 0 in 2..5, sin < 0 in 4..7.
  const bool swp = (int32_t)((v + 0x20000000u) << 1) < 0;
  const uint32_t x = __builtin_bit_cast(uint32_t, swp ? sn : cs);
  const uint32_t y = __builtin_bit_cast(uint32_t, swp ? cs : sn);
  const uint32_t t = v + 0x40000000u;
  *c = __builtin_bit_cast(float, (x & 0x7FFFFFFFu) | (t & 0x80000000u));
  *s = __builtin_bit_cast(float, (y & 0x7FFFFFFFu) | (v & 0x80000000u));
}

// Renormalisation factor to bring a vector of squared length nn back to
// length |S|, given inv_s2 = 1/S^2 (FP32, correctly rounded): one Newton
// step for 1/sqrt(nn/S^2) from 1, f = 1.5 - 0.5 * nn/S^2.  The reflection
// move keeps nn within ~1e-7 (FP32) or ~1e-3 (FP16 storage) of S^2, so the
// renormalised length is exact to O(delta^2).
__host__ __device__ __forceinline__ float renorm_factor(float nn, float inv_s2) {
  return fmaf(-0.5f, nn * inv_s2, 1.5f);
}

}  // namespace mcg
