// Counter-based noise shared bit-for-bit by the CPU and gfx950: Philox4x32-10
// (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as 1, 2, 3",
// SC'11) and a Box-Muller transform built only from IEEE +,-,*,/, sqrt and
// explicit fma, so both sides return the same doubles.
//
// The reference leaves noise to the user: SDE::noise(&mut self, dt, &mut dw)
// (src/sde/sde.rs:67) fills dW, and the steps consume it at
// src/methods/erk/fixed/stochastic.rs:118-119 and src/methods/milstein.rs:134-135.
// The device SDE families use this generator as their noise() implementation:
//   dW[path][step][i] = sqrt(h_step) * Z(seed, path, step, i)
// keyed by the 0-based step index, so a path's noise does not depend on which
// batch, lane or launch integrates it.
#pragma once

#include "de_common.h"
#include "de_noise_tables.h"

namespace de {

DE_TABLE double kNoiseLogTable[128 * 2] = DE_NOISE_LOG_TABLE;

struct u32x4 {
  uint32_t v[4];
};

DE_HD void mulhilo32(uint32_t a, uint32_t b, uint32_t* hi, uint32_t* lo) {
  uint64_t p = (uint64_t)a * (uint64_t)b;
  *hi = (uint32_t)(p >> 32);
  *lo = (uint32_t)p;
}

// Philox4x32 with 10 rounds.  ctr = (c0,c1,c2,c3), key = (k0,k1).
DE_HD u32x4 philox4x32_10(u32x4 ctr, uint32_t k0, uint32_t k1) {
  const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
  const uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
  for (int round = 0; round < 10; ++round) {
    if (round > 0) {
      k0 += W0;
      k1 += W1;
    }
    uint32_t hi0, lo0, hi1, lo1;
    mulhilo32(M0, ctr.v[0], &hi0, &lo0);
    mulhilo32(M1, ctr.v[2], &hi1, &lo1);
    u32x4 n;
    n.v[0] = hi1 ^ ctr.v[1] ^ k0;
    n.v[1] = lo1;
    n.v[2] = hi0 ^ ctr.v[3] ^ k1;
    n.v[3] = lo0;
    ctr = n;
  }
  return ctr;
}

// a ^ b ^ c, one instruction on gfx950 (a truth-table operation on three words).
DE_HD uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
#else
  return a ^ b ^ c;
#endif
}

// The Philox4x32-10 blocks (j, step, path), j < NB, of one path: the words of
// the first three rounds that do not depend on the step are formed once per
// path, and the one first-round product that depends on the step but not on j
// once per step.  What is left per step is 1 product for all blocks and 15 per
// block instead of 20 per block, each with one three-input exclusive or.
template <int NB>
struct PhiloxPath {
  uint32_t n0;         // round 1: word 0 without the step
  uint32_t p1k[NB];    // round 2: word 1 ^ round 3's key 0
  uint32_t c0h[NB];    // round 3: high half of the first product ^ key 1
  uint32_t c0l[NB];    // round 3: word 3 ^ round 4's key 1

  DE_HD static constexpr uint32_t key0(uint32_t k, int round) {
    return k + (uint32_t)round * 0x9E3779B9u;
  }
  DE_HD static constexpr uint32_t key1(uint32_t k, int round) {
    return k + (uint32_t)round * 0xBB67AE85u;
  }
  static constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u;

  DE_HD void start(uint64_t path, uint32_t k0, uint32_t k1) {
    uint32_t hi, lo;
    mulhilo32(kM1, (uint32_t)path, &hi, &lo);
    n0 = hi ^ k0;
    const uint32_t n1 = lo;
    for (int j = 0; j < NB; ++j) {
      const uint64_t m0j = (uint64_t)kM0 * (uint32_t)j;
      const uint32_t n2 = (uint32_t)(m0j >> 32) ^ (uint32_t)(path >> 32) ^ k1;
      mulhilo32(kM1, n2, &hi, &lo);
      const uint32_t p0 = hi ^ n1 ^ key0(k0, 1);
      p1k[j] = lo ^ key0(k0, 2);
      mulhilo32(kM0, p0, &hi, &lo);
      c0h[j] = hi ^ key1(k1, 2);
      c0l[j] = lo ^ key1(k1, 3);
    }
  }
  // The step's shared product.
  DE_HD void step(uint32_t call, uint32_t* hi, uint32_t* lo) const {
    mulhilo32(kM0, n0 ^ call, hi, lo);
  }
  DE_HD u32x4 block(int j, uint32_t step_hi, uint32_t step_lo, uint32_t k0, uint32_t k1) const {
    uint32_t hi0, lo0, hi1, lo1;
    const uint32_t m0j = (uint32_t)((uint64_t)kM0 * (uint32_t)j);
    mulhilo32(kM1, step_hi ^ (m0j ^ key1(k1, 1)), &hi1, &lo1);
    uint32_t c0 = hi1 ^ p1k[j], c1 = lo1, c2 = c0h[j] ^ step_lo, c3;
    // Round 4, whose key 1 is in c0l already.
    mulhilo32(kM0, c0, &hi0, &lo0);
    mulhilo32(kM1, c2, &hi1, &lo1);
    c0 = xor3(hi1, c1, key0(k0, 3));
    c1 = lo1;
    c2 = hi0 ^ c0l[j];
    c3 = lo0;
#pragma unroll
    for (int round = 4; round < 10; ++round) {
      mulhilo32(kM0, c0, &hi0, &lo0);
      mulhilo32(kM1, c2, &hi1, &lo1);
      c0 = xor3(hi1, c1, key0(k0, round));
      c1 = lo1;
      c2 = xor3(hi0, c3, key1(k1, round));
      c3 = lo0;
    }
    return u32x4{{c0, c1, c2, c3}};
  }
};

// x with its sign flipped where bit 31 of `bit` is set.
DE_HD double flip_sign(double x, uint32_t bit) {
  const uint64_t u = as_u64(x);
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t hi = __builtin_amdgcn_bitop3_b32((uint32_t)(u >> 32), bit, 0x80000000u, 0x78);
#else
  const uint32_t hi = (uint32_t)(u >> 32) ^ (bit & 0x80000000u);
#endif
  return as_f64(((uint64_t)hi << 32) | (uint32_t)u);
}

// fma(a, b, c) as one three-operand instruction on the device.  With c a
// polynomial coefficient that stays live across loop iterations the compiler
// otherwise picks the accumulate form (dst = a * b + dst) and copies c into
// dst first; the operation and its rounding are the same either way.
DE_HD double fma3(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
#else
  return fma(a, b, c);
#endif
}

// 53-bit uniform from two words: m * 2^-53 with m = ((hi << 32) | lo) >> 11,
// formed as hi * 2^-32 + (lo >> 11) * 2^-53: both terms and their sum (53
// significant bits) are exact, so this is the value of the 64-bit formula.
DE_HD double uniform_co(uint32_t hi, uint32_t lo) {  // [0, 1)
  return fma((double)(lo >> 11), 0x1p-53, (double)hi * 0x1p-32);
}

// (m + 1) * 2^-53; (lo >> 11) + 1 <= 2^21 carries into the hi term exactly.
DE_HD double uniform_oc(uint32_t hi, uint32_t lo) {  // (0, 1]
  return fma((double)((lo >> 11) + 1u), 0x1p-53, (double)hi * 0x1p-32);
}

// Natural log for x in [2^-53, 1], about 1 ulp; deterministic, used by the
// Box-Muller radius only (its argument, a 53-bit uniform in (0, 1], is never
// below 2^-53, so x is a normal double).
DE_HD double noise_log(double x) {
  // x = 2^k z: with tmp = bits(x) - OFF (OFF's low word is zero, so only the
  // high words take part), i = bits 45..51 of tmp, k = its top 12 bits
  // (signed), and z = x with k taken out of the exponent.
  const uint64_t ix = as_u64(x);
  const uint32_t xhi = (uint32_t)(ix >> 32);
  const uint32_t thi = xhi - (uint32_t)(DE_NOISE_OFF >> 32);
  const int i = (int)((thi >> 13) & 127u);
  const int32_t k = (int32_t)thi >> 20;
  const double z = as_f64(((uint64_t)(xhi - (thi & 0xfff00000u)) << 32) | (uint32_t)ix);
  double invc = kNoiseLogTable[2 * i + 0];
  double lc = kNoiseLogTable[2 * i + 1];
  double r = fma(z, invc, -1.0);
  const double c[8] = DE_NOISE_LOG_POLY;
  double q = c[7];
  q = fma(r, q, c[6]);
  q = fma(r, q, c[5]);
  q = fma(r, q, c[4]);
  q = fma(r, q, c[3]);
  q = fma(r, q, c[2]);
  q = fma(r, q, c[1]);
  q = fma(r, q, c[0]);
  double r2 = r * r;
  double p = fma(r2 * r, q, -0.5 * r2);
  double kd = (double)k;
  return (kd * DE_NOISE_LN2_HI + lc) + (r + (p + kd * DE_NOISE_LN2_LO));
}

// sin and cos of theta for |theta| <= pi/4 (Taylor to theta^17 / theta^16;
// coefficients generated by gen_noise_tables.py).
DE_HD void noise_sincos_small(double th, double* s, double* c) {
  const double sp[8] = DE_NOISE_SIN_POLY;
  const double cp[8] = DE_NOISE_COS_POLY;
  double t2 = th * th;
  double ps = sp[0];
  double pc = cp[0];
  for (int n = 1; n < 8; ++n) {
    ps = fma3(t2, ps, sp[n]);
    pc = fma3(t2, pc, cp[n]);
  }
  *s = fma(th * t2, ps, th);
  *c = fma(t2, pc, 1.0);
}

// sqrt(x) for x = 0 or 2^-60 <= x < 2^1000: the correctly rounded square root
// that the device compiler expands sqrt into (reciprocal square root seed, two
// Newton-Raphson corrections and two residual corrections), without its
// rescaling of tiny arguments (a multiplication by 2^0 here) and its infinity
// check; the host computes sqrt itself.  Same operations in the same order,
// so the same bits.
DE_HD double noise_sqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rsq(x);
  double y = x * r;
  double hh = r * 0.5;
  const double e = fma(-hh, y, 0.5);
  y = fma(y, e, y);
  hh = fma(hh, e, hh);
  double d = fma(-y, y, x);
  y = fma(d, hh, y);
  d = fma(-y, y, x);
  y = fma(d, hh, y);
  return x == 0.0 ? x : y;
#else
  return sqrt(x);
#endif
}

// Two independent standard normals from one Philox block (Box-Muller).
// Angle 2*pi*u2 is reduced in quarter turns, which is exact.
DE_HD void box_muller(u32x4 w, double* z0, double* z1) {
  DE_NO_CONTRACT
  double u1 = uniform_oc(w.v[0], w.v[1]);
  double rad = noise_sqrt(-2.0 * noise_log(u1));   // 0 or >= 2^-52
  // q4 = 4 u2 with u2 = uniform_co(w.v[2], w.v[3]), exact like u2.
  const double q4 = fma((double)(w.v[3] >> 11), 0x1p-51, (double)w.v[2] * 0x1p-30);
  // The nearest integer of q4 (ties to even, exact operations): the sum's low
  // word is that integer, so the quarter needs no conversion.
  const double qs = q4 + 0x1.8p52;
  const double qd = qs - 0x1.8p52;
  const uint32_t q = (uint32_t)as_u64(qs);
  double f = q4 - qd;                            // [-0.5, 0.5], exact
  double th = f * DE_NOISE_HALF_PI;
  double s, c;
  noise_sincos_small(th, &s, &c);
  // Quarter q: (cos, sin) = (c, s), (-s, c), (-c, -s), (s, -c): swapped for
  // odd q, the signs from bit 1 of q + 1 and of q.
  const double a = (q & 1u) ? s : c;
  const double b = (q & 1u) ? c : s;
  *z0 = rad * flip_sign(a, (q + 1u) << 30);
  *z1 = rad * flip_sign(b, q << 30);
}

// Standard normal for (seed, path, step, component).  Components 2j and 2j+1
// share Philox counter (j, step, path_lo, path_hi).
DE_HD double noise_normal(uint64_t seed, uint64_t path, uint32_t step,
                          uint32_t comp) {
  u32x4 ctr = {{comp >> 1, step, (uint32_t)path, (uint32_t)(path >> 32)}};
  u32x4 w = philox4x32_10(ctr, (uint32_t)seed, (uint32_t)(seed >> 32));
  double z0, z1;
  box_muller(w, &z0, &z1);
  return (comp & 1) ? z1 : z0;
}

// Input-generation streams use a separate counter domain (bit 31 of c1 set) so
// they never collide with per-step noise counters.
DE_HD u32x4 input_block(uint64_t seed, uint64_t item, uint32_t stream,
                        uint32_t j) {
  u32x4 ctr = {{j, 0x80000000u | stream, (uint32_t)item, (uint32_t)(item >> 32)}};
  return philox4x32_10(ctr, (uint32_t)seed, (uint32_t)(seed >> 32));
}

DE_HD double input_uniform(uint64_t seed, uint64_t item, uint32_t stream,
                           uint32_t j) {
  u32x4 w = input_block(seed, item, stream, j);
  return uniform_co(w.v[0], w.v[1]);
}

DE_HD void input_normal_pair(uint64_t seed, uint64_t item, uint32_t stream,
                             uint32_t j, double* z0, double* z1) {
  box_muller(input_block(seed, item, stream, j), z0, z1);
}

}  // namespace de
