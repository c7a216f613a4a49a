// Spring-chain (ragged, uneven-size) ensemble launchers.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/de_api.h"
#include "de_lane.h"
#include "de_spring_classes.h"
#include "de_spring_solvers.h"

namespace de {
namespace parity {

typedef void (*GroupKernel)(SpringArgs);

// The group kernels of a method other than DOPRI5 (final state and t_eval
// output), one shape per size class.
struct ClassKernel {
  int g;  // lanes per system
  GroupKernel k;
};
// Translation unit `part`'s kernels of a method (kNumCaps entries), or null.
#define DE_SPRING_PARTS(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6)
#define DE_SPRING_PART_DECL(n) const ClassKernel* spring_method_part##n(int method);
DE_SPRING_PARTS(DE_SPRING_PART_DECL)
#undef DE_SPRING_PART_DECL

// Launch a spring-chain ensemble.  `b` holds device pointers; host_sizes is a
// host copy of b->sizes (the launcher buckets systems by size).  Returns 0 on
// success, 1 if unsupported, -1 on HIP error, -4 on allocation failure.
int launch_spring(const de_ode_batch* b, const int32_t* host_sizes, const OdeArgs& a, int sched,
                  hipStream_t s);
int64_t spring_workspace_bytes(const de_ode_batch* b);
// The shape (G, C, block) that the systems of the size class with cap masses were last
// solved with: 0, or -1 if none has been solved with a shape of the library's choice.
int spring_tuned(int cap, int* g, int* c, int* block);

}  // namespace parity
}  // namespace de
