// Size classes of the spring chains' group kernels and which of them one launch uses
// (host code, built by g++ for the tests as well).
#pragma once

#include <stdint.h>

namespace de {
namespace parity {

// Size classes: systems of at most kCaps[k] masses.
constexpr int kCaps[] = {4, 8, 16, 32, 64, 128, 256};
constexpr int kNumCaps = 7;

// DOPRI5's size classes: the powers of two and, with three masses per lane, the
// sizes between them: systems of log-uniform size then fill 85% of their lanes'
// masses on average (72% with powers of two alone).
constexpr int kDopri5Caps[] = {4, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256};
constexpr int kMaxClasses = sizeof(kDopri5Caps) / sizeof(kDopri5Caps[0]);
static_assert(kNumCaps <= kMaxClasses, "per-class arrays");

struct ClassSet {
  const int* caps;
  int n;
};
inline ClassSet class_set(bool dopri5) {
  return dopri5 ? ClassSet{kDopri5Caps, kMaxClasses} : ClassSet{kCaps, kNumCaps};
}
inline int class_index(const ClassSet& cs, int masses) {
  int k = 0;
  while (k < cs.n && cs.caps[k] < masses) ++k;
  return k;
}

// The classes of one launch.  Every class is a kernel; those beyond the four hardware
// queues a process gets wait for one another, and the longest solve bounds each.  So
// an ensemble whose sizes span more than four classes may use fewer, wider ones:
//   few   64 lanes per system, one kernel per number of masses per lane;
//   mid   (DOPRI5) five classes of 16 to 256 masses;
//   all   every class.
// A system keeps its sums' tree (three masses per lane or a power of two) in each
// of them, so its result does not depend on the ensemble it is in.
enum Merge { kMergeAll = 0, kMergeMid = 1, kMergeFew = 2 };
constexpr int kQueues = 4;

// The class that `cap`'s systems are solved in.
inline int merged_cap(Merge m, int cap) {
  const bool three = cap % 3 == 0;
  if (m == kMergeFew) return three ? 192 : (cap <= 64 ? 64 : cap);
  if (m == kMergeMid)
    return three ? (cap <= 48 ? 48 : 192) : (cap <= 16 ? 16 : (cap <= 64 ? 64 : 256));
  return cap;
}

// What a launch of the systems count[k] in class k costs with the classes of `m`, in
// wavefronts of one mass per lane:
//   the wavefronts' work: the masses that the launched lanes hold, padding included;
//   2750 (DOPRI5; 1625 for the other methods) for each kernel up to three, the queues
//   beside the one that the caller's stream has, 1250 (1000) up to five and 750 (1000)
//   for each further one: it waits for another but overlaps with the rest.
// Both parts grow with the steps of a solve, so neither spans nor tolerances enter.
// The constants fit 10 size distributions of 256 to 65 536 systems with DOPRI5 and 5 of
// 512 to 32 768 with RK4, DOP853, RKF45 and RKV989E, each timed with every set in
// processes with no, two and three other streams (which hardware queue a stream gets
// depends on them): the set of least cost takes 1.1% and 0.7% more than the fastest one
// on average, 14% and 13% at most.
inline int64_t launch_cost(bool dopri5, Merge m, const int64_t* count) {
  const ClassSet cs = class_set(dopri5);
  int64_t masses = 0;
  bool used[kMaxClasses] = {};
  int kernels = 0;
  for (int k = 0; k < cs.n; ++k) {
    if (count[k] == 0) continue;
    const int cap = merged_cap(m, cs.caps[k]);
    masses += count[k] * cap;
    bool& u = used[class_index(cs, cap)];
    kernels += u ? 0 : 1;
    u = true;
  }
  const auto up_to = [kernels](int n) { return kernels < n ? kernels : n; };
  const int beside = up_to(kQueues - 1), next = up_to(5) - beside;
  return masses / 64 + (dopri5 ? 2750 : 1625) * beside + (dopri5 ? 1250 : 1000) * next +
         (dopri5 ? 750 : 1000) * (kernels - beside - next);
}

// The set of classes of least cost; every class where they are no more than the
// queues.  Few / mid / all in ms, means over those processes, * chosen.  DOPRI5 at
// rtol 1e-6 over t in [0, 10]:
//   4 to 256 masses, log-uniform       2048 systems *1.01 / 1.29 / 1.69, 8192 1.94 /
//                                      *1.78 / 2.00, 32768 6.49 / 4.78 / *4.10
//   4 to 8 masses, 1% larger           8192 1.82 / *1.34 / 1.56, 32768 4.50 / 2.16 /
//                                      *2.04, 65536 8.09 / 3.30 / *2.77
//   4 masses, one of 8, 16, 24 and 32  1024 *0.52 / 0.65 / 0.77, 6144 1.08 / *0.75 /
//                                      0.77, 16384 2.16 / 1.07 / *0.88
//   129 to 256 masses, five smaller    2048 *1.15 / 1.27 / 1.28, 16384 *4.87 / 5.05 / 5.03
// RK4 (h 0.02) over t in [0, 4], few / all:
//   4 to 256 masses, log-uniform       2048 *0.48 / 0.57, 16384 1.48 / *1.20
//   geometric of mean 12 masses        1024 *0.27 / 0.43, 12288 0.81 / *0.55
inline Merge merge_of(bool dopri5, const int64_t* count) {
  const ClassSet cs = class_set(dopri5);
  int classes = 0;
  for (int k = 0; k < cs.n; ++k) classes += count[k] > 0 ? 1 : 0;
  Merge best = kMergeAll;
  if (classes <= kQueues) return best;
  int64_t cost = launch_cost(dopri5, best, count);
  for (Merge m : {kMergeMid, kMergeFew}) {
    if (m == kMergeMid && !dopri5) continue;
    const int64_t c = launch_cost(dopri5, m, count);
    if (c < cost) {
      cost = c;
      best = m;
    }
  }
  return best;
}

// DOPRI5's shape for a caller's number of lanes per system (a power of two up to 64) in
// the class of `cap` masses: that many lanes where 1, 2 or 4 masses per lane fill the
// class, or where 3 hold it in a class of three masses per lane; otherwise the class's
// shape of most masses per lane.  Lanes beyond a class of three masses per lane add
// zeros, so the sums keep their tree.
struct LaneShape {
  int g, c;
};
inline LaneShape group_shape(int cap, int lanes) {
  const bool power = lanes >= 1 && lanes <= 64 && (lanes & (lanes - 1)) == 0;
  if (cap % 3 == 0) return {power && lanes * 3 >= cap ? lanes : cap / 3, 3};
  for (int c = 1; c <= 4; c *= 2)
    if (power && lanes * c == cap) return {lanes, c};
  return {cap / 4, 4};
}

}  // namespace parity
}  // namespace de
