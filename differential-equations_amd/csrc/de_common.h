// Shared host/device helpers for the ensemble Runge-Kutta integrator.
//
// This header is compiled three ways: by hipcc for gfx950 device code, by hipcc
// for the host side of the library, and by g++ for CPU-side consumers.  Every
// floating-point expression in the integrator must produce the same bits in all
// three, so:
//   * all translation units are built with -ffp-contract=off (no implicit FMA);
//   * explicit fma() is used only where an exactly rounded fused operation is
//     intended (double-double arithmetic), never as an optimisation;
//   * max/min use fmax/fmin (IEEE maxNum/minNum: a NaN operand yields the other
//     operand), which is the semantics of Rust's f64::max/f64::min that the
//     reference solver uses (src/methods/erk/dormandprince/ordinary.rs:157).
#pragma once

#include <stdint.h>
#include <math.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DE_HD __host__ __device__ inline
#define DE_DEV __device__ inline
// Run once per trajectory (init, result write-back), inside branches a wave
// takes only when one of its lanes starts or ends a trajectory.  Forced
// inline: as calls they would pass the lane state through scratch memory,
// and the partial-wave scratch writes would multiply the kernel's HBM traffic.
#define DE_COLD __host__ __device__ inline __attribute__((always_inline))
#else
#define DE_HD inline
#define DE_DEV inline
#define DE_COLD inline
#endif

#if defined(__HIP_DEVICE_COMPILE__)
#define DE_TABLE __device__ __constant__ static const
#else
#define DE_TABLE static const
#endif

// Code whose every product and sum must be rounded on its own (error-free
// transformations, operation sequences fixed for bit parity), also in
// translation units compiled with FMA contraction.
#if defined(__clang__)
#define DE_NO_CONTRACT _Pragma("clang fp contract(off)")
#define DE_FORCE_INLINE __attribute__((always_inline))
#else
#define DE_NO_CONTRACT
#define DE_FORCE_INLINE
#endif

namespace de {

// f64::EPSILON * 10, the end-of-interval threshold of the solve drivers
// (src/ode/solve_ivp.rs:198,263; src/sde/solve_ivp.rs:217,273).
static constexpr double kTenEps = 2.220446049250313080847e-16 * 10.0;

// Quiet NaN: dense-output points that a solve does not produce.
static constexpr uint64_t kNaNBits = 0x7ff8000000000000ULL;

DE_HD uint64_t as_u64(double x) {
  union { double d; uint64_t u; } v;
  v.d = x;
  return v.u;
}

DE_HD double as_f64(uint64_t u) {
  union { double d; uint64_t u; } v;
  v.u = u;
  return v.d;
}

// Rust f64::signum: 1.0 for +0 and positive values, -1.0 for -0 and negative
// values, NaN for NaN.
DE_HD double signum(double x) { return x != x ? x : copysign(1.0, x); }

// A pointer known to hold global memory, as such.  The lanes' kernels read their
// pointers from an argument block in memory, where the compiler only knows generic
// ones: their accesses would be flat, which count among the scalar loads' waits, so
// that the next attempt's settings would wait for the last output's store.
// The caller has to know it: a local array, a member of a lane or LDS as the argument
// is undefined (a generic address of those is no global one), also where inlining
// happens to hide it.  Functions that also get a lane's own copy of a record read it
// plainly.  A host build that defines DE_ON_GLOBAL_PTR(p) sees every argument
// (tests/cpp/global_ptr_check.cpp).
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
DE_DEV __attribute__((address_space(1))) T* global_ptr(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}
#else
#if !defined(DE_ON_GLOBAL_PTR)
#define DE_ON_GLOBAL_PTR(p) ((void)0)
#endif
template <class T>
DE_HD T* global_ptr(T* p) {
  DE_ON_GLOBAL_PTR(p);
  return p;
}
#endif

// Starts the code after x's computation on a multiple of 8 bytes (one s_nop at most).
// A double precision instruction is 8 bytes long and is fetched slower where it lies
// across such a line; a 4-byte one (a move, a compare) shifts all that follow it.  In
// DOP853's step the run through the stages is long enough to pay: 619 of its 754
// long instructions lay across a line, 118 do now (3 000 Lorenz trajectories: 1.18 to
// 1.07 ms, one wave per SIMD; 1 048 576: 33.5 to 31.6, the time from before the outputs
// became global stores, which had moved the run by four bytes).  DOPRI5's (4.17 against
// 4.21 ms at 1 024 trajectories) and the spring groups' steps (8.87 against 9.52 ms)
// lose more to the break in their order than they gain.
#if defined(__HIP_DEVICE_COMPILE__)
DE_DEV void align_code(double& x) { asm(".p2align 3" : "+v"(x)); }
#else
DE_HD void align_code(double&) {}
#endif

// constrain_step_size (src/utils.rs:22-33): clamp |h| to [h_min, h_max] keeping
// the sign of h (written with selects; a NaN h is returned unchanged).  signum(h)
// times a bound is the bound with its sign flipped where h's is set.
DE_HD double constrain_step_size(double h, double h_min, double h_max) {
  const uint64_t sign = as_u64(h) & 0x8000000000000000ULL;
  const double a = fabs(h);
  return a < h_min ? as_f64(as_u64(h_min) ^ sign) : (a > h_max ? as_f64(as_u64(h_max) ^ sign) : h);
}

// The stiffness test's decision h * sqrt(num / den) > 6.1, with den > 0, as
// the reference evaluates it (dormandprince/ordinary.rs:172-174: a division,
// a square root and a product, each rounded), but usually without them.  For
// h, num and den in [2^-300, 2^300] the products h^2 num and RN(6.1)^2 den
// are within a relative 3 * 2^-53 of their exact values, and the rounded
// expression within a relative 2.5 * 2^-53 of h sqrt(num / den); so when the
// two products differ by more than a relative 1e-12 their order is the
// decision.  Otherwise, and outside that range (h <= 0 included), the
// reference's own sequence decides.
DE_HD bool stiff_exceeds(double h, double num, double den) {
  constexpr double kLo = 0x1p-300, kHi = 0x1p300;
  constexpr double c = 6.1;
  constexpr double c2 = c * c;  // rounded once; inside the 3 * 2^-53 above
  const bool in_range = h > kLo && h < kHi && num > kLo && num < kHi && den > kLo && den < kHi;
  if (in_range) {
    const double lhs = (h * h) * num;
    const double rhs = c2 * den;
    if (lhs < rhs * (1.0 - 1e-12)) return false;
    if (lhs > rhs * (1.0 + 1e-12)) return true;
  }
  return h * sqrt(num / den) > c;
}

// Per-trajectory status codes.  0..4 mirror Status::Complete and the Error
// variants a solve can end with (src/error.rs:13-41), 5 Status::Interrupted
// (an event solout's Terminate), 6 a solout's unwrap of a failed
// interpolation (the reference panics); kRunning is internal.
enum Status : int32_t {
  kComplete = 0,
  kMaxSteps = 1,
  kStepSize = 2,
  kStiffness = 3,
  kBadInput = 4,
  kInterrupted = 5,
  kOutOfBounds = 6,
  kRunning = -1,
};

// validate_step_size_parameters (src/utils.rs:60-157): 0 when the parameters
// are valid, else the number of the first failed check in the reference's
// order (each an Err(Error::BadInput) with its own message):
//   1 tf == t0              2 sign(h0) != sign(tf - t0)   3 h_min < 0
//   4 h_max < 0             5 h_min > h_max                6 |h0| < h_min
//   7 |h0| > h_max          8 |h0| > |tf - t0|             9 h0 == 0
DE_HD int validate_step_size_check(double h0, double h_min, double h_max, double t0,
                                   double tf) {
  if (tf == t0) return 1;
  double sign = signum(tf - t0);
  if (signum(h0) != sign) return 2;
  if (h_min < 0.0) return 3;
  if (h_max < 0.0) return 4;
  if (h_min > h_max) return 5;
  if (fabs(h0) < h_min) return 6;
  if (fabs(h0) > h_max) return 7;
  if (fabs(h0) > fabs(tf - t0)) return 8;
  if (h0 == 0.0) return 9;
  return 0;
}

DE_HD bool validate_step_size(double h0, double h_min, double h_max, double t0,
                              double tf) {
  return validate_step_size_check(h0, h_min, h_max, t0, tf) == 0;
}

}  // namespace de
