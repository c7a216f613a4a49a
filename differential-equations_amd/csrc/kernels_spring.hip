// Spring-chain ensembles: uneven system sizes (2N in [8, 512]).
//
// Mappings (selected by de_ode_batch.mapping):
//   DE_MAP_LANE   one thread per system, vectors in an HBM workspace (plain
//                 launch; bit-identical to the CPU restatement).
//   DE_MAP_GROUP  G lanes per system with C masses per lane in registers.
//                 DOPRI5 to rounding (its norm is summed over the lanes); the
//                 other methods keep the one-lane solvers' bits and have one
//                 shape per size class (kernels_spring_group.hip).
//   DE_MAP_AUTO   as DE_MAP_GROUP without a group_size.  Systems are bucketed into
//                 size classes, some of which a launch may merge
//                 (de_spring_classes.h); for each class of DOPRI5 an autotuner
//                 times the shapes (G, C) with G*C equal to the class cap on a
//                 sample of the class and keeps the fastest.  Classes run
//                 concurrently on their own streams, each as a persistent kernel
//                 whose groups take the next system of the class from a work
//                 counter when they finish one.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <vector>

#include "de_launch.h"
#include "de_spring.h"
#include "de_spring_solvers.h"

namespace de {
namespace parity {

constexpr int kSpringBlock = 256;

template <class Solver>
__global__ __launch_bounds__(kSpringBlock) void spring_lane_kernel(SpringArgs A) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.o.n) return;
  Solver s;
  if (!s.init(&A, i)) return;
  while (!s.advance()) {
  }
}

// The one-lane solver of each method: its kernel and its workspace doubles
// per state component.
struct LaneSolver {
  void (*kernel)(SpringArgs);
  int vectors;
};
template <class Solver>
static LaneSolver lane_solver_of() {
  return {spring_lane_kernel<Solver>, Solver::kVectors};
}
static LaneSolver lane_solver(int method) {
  switch (method) {
    case DE_METHOD_DOP853: return lane_solver_of<VecDop853>();
    case DE_METHOD_RK4: return lane_solver_of<VecFixed<4>>();
    case DE_METHOD_EULER: return lane_solver_of<VecFixed<1>>();
    case DE_METHOD_RKF45: return lane_solver_of<VecErk<erk_tab::Rkf45>>();
    case DE_METHOD_CASH_KARP: return lane_solver_of<VecErk<erk_tab::CashKarp>>();
    case DE_METHOD_RKV655E: return lane_solver_of<VecErk<erk_tab::Rkv655e>>();
    case DE_METHOD_RKV656E: return lane_solver_of<VecErk<erk_tab::Rkv656e>>();
    case DE_METHOD_RKV766E: return lane_solver_of<VecErk<erk_tab::Rkv766e>>();
    case DE_METHOD_RKV767E: return lane_solver_of<VecErk<erk_tab::Rkv767e>>();
    case DE_METHOD_RKV877E: return lane_solver_of<VecErk<erk_tab::Rkv877e>>();
    case DE_METHOD_RKV878E: return lane_solver_of<VecErk<erk_tab::Rkv878e>>();
    case DE_METHOD_RKV988E: return lane_solver_of<VecErk<erk_tab::Rkv988e>>();
    case DE_METHOD_RKV989E: return lane_solver_of<VecErk<erk_tab::Rkv989e>>();
    default: return lane_solver_of<VecDopri5>();
  }
}

// Occupancy hints: the rarely taken double-double pow fallback raises the
// peak register count past a wave-slot boundary; the hints trade that for a
// few spills outside the step block.
template <int G, int C, bool OUT>
__global__ __launch_bounds__(kSpringBlock) __attribute__((amdgpu_waves_per_eu(C == 1 ? 3 : 2))) void
spring_group_kernel(SpringArgs A) {
  spring_group_loop<GroupDopri5<G, C, OUT>>(A);
}

__global__ void spring_zero_counters(unsigned long long* c, int n) {
  if ((int)threadIdx.x < n) c[threadIdx.x] = 0ull;
}

// The systems of each class: start[k] .. start[k + 1] of the list, by the classes of the
// sizes.  Made on the device, so that the call need not wait for an upload.  A block
// takes its systems' places in every class with one atomic, so that a class's systems
// stand in index order but for the order of the blocks (the solves read and write their
// systems' memory in the list's order: 65 536 systems 8.75 ms, 8.88 with one atomic per
// wavefront); results do not depend on the order.
constexpr int kListBlock = 1024;
struct ListArgs {
  int64_t start[kMaxClasses + 1];
  int classes;
  uint8_t class_of_size[257];
};
__global__ __launch_bounds__(kListBlock) void spring_list_kernel(
    ListArgs a, const int32_t* __restrict__ sizes, int64_t n, unsigned long long* lengths,
    int32_t* __restrict__ list) {
  __shared__ int32_t before[kListBlock / 64][kMaxClasses];  // in the block's earlier wavefronts
  __shared__ unsigned long long first[kMaxClasses];
  const int64_t i = (int64_t)blockIdx.x * kListBlock + threadIdx.x;
  const int32_t m = i < n ? sizes[i] : 0;
  const int mine = m >= 1 && m <= 256 ? a.class_of_size[m] : -1;
  const int wave = threadIdx.x / 64;
  int below = 0;
  for (int k = 0; k < a.classes; ++k) {
    const unsigned long long mask = __ballot(mine == k);
    if (mine == k) below = __popcll(mask & __lanemask_lt());
    if (__lane_id() == 0) before[wave][k] = __popcll(mask);
  }
  __syncthreads();
  if ((int)threadIdx.x < a.classes) {
    int32_t sum = 0;
    for (int w = 0; w < kListBlock / 64; ++w) {
      const int32_t c = before[w][threadIdx.x];
      before[w][threadIdx.x] = sum;
      sum += c;
    }
    first[threadIdx.x] =
        sum ? atomicAdd(&lengths[threadIdx.x], (unsigned long long)sum) : 0ull;
  }
  __syncthreads();
  if (mine < 0) return;
  const int64_t pos = a.start[mine] + (int64_t)first[mine] + before[wave][mine] + below;
  if (pos < a.start[mine + 1]) list[pos] = (int32_t)i;
}

struct Config {
  int g, c;
  GroupKernel k;   // final state and t_eval output
  GroupKernel kx;  // with the point outputs and event solouts
};

#define DE_CFG(G, C) {G, C, spring_group_kernel<G, C, false>, spring_group_kernel<G, C, true>}
static const Config kConfigs[] = {
    DE_CFG(4, 1),  DE_CFG(8, 1),  DE_CFG(16, 1), DE_CFG(32, 1), DE_CFG(64, 1),
    DE_CFG(2, 2),  DE_CFG(4, 2),  DE_CFG(8, 2),  DE_CFG(16, 2), DE_CFG(32, 2), DE_CFG(64, 2),
    DE_CFG(8, 3),  DE_CFG(16, 3), DE_CFG(32, 3), DE_CFG(64, 3),
    DE_CFG(1, 4),  DE_CFG(2, 4),  DE_CFG(4, 4),  DE_CFG(8, 4),  DE_CFG(16, 4), DE_CFG(32, 4),
    DE_CFG(64, 4),
};
#undef DE_CFG
static const int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);

// The shapes the autotuner times: at least four lanes per system, and four masses
// per lane only in the classes that need them.  (On the 64k-system ensemble, 2 000
// to 10 000 systems per class: two lanes of two masses 0.73 against 0.63 ms for
// four lanes of one; four masses per lane 0.79 to 1.28 against 0.65 to 0.98 ms up
// to 64 masses, 1.16 against 1.22 ms at 128.)  Blocks of one wavefront leave their
// slot as soon as its groups have drained.
constexpr int kTunedBlock = 64;
static bool tuned_shape(const Config& cf, int cap) {
  return cf.g * cf.c == cap && cf.g >= 4 && (cf.c < 4 || cap >= 128);
}

struct Choice {
  int cfg = -1;
  int block = kSpringBlock;
};

// A class's kernel in one launch.
struct Shape {
  GroupKernel kernel;
  int g, block;
};

// Process-wide state: autotune decisions per size class, streams, workspace.
static std::mutex g_mu;
// DOPRI5's shapes of the library's choice by class cap: the autotuner's, for ensembles
// that use every class and for those that use five, and the one that each class's
// systems were last solved with.  Which shape is picked does not change a system's
// result.
static std::map<int, Choice> g_tuned[2];
static std::map<int, Choice> g_solved;
static hipStream_t g_streams[kMaxClasses] = {};
static hipEvent_t g_fork = nullptr, g_join[kMaxClasses] = {};
static int g_num_cu = 0;

static int ensure_runtime() {
  if (g_fork) return 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  if (hipDeviceGetAttribute(&g_num_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return -1;
  for (int k = 0; k < kMaxClasses; ++k) {
    if (hipStreamCreateWithFlags(&g_streams[k], hipStreamNonBlocking) != hipSuccess) return -1;
    if (hipEventCreateWithFlags(&g_join[k], hipEventDisableTiming) != hipSuccess) return -1;
  }
  if (hipEventCreateWithFlags(&g_fork, hipEventDisableTiming) != hipSuccess) return -1;
  return 0;
}

static int blocks_per_cu(GroupKernel k, int block) {
  int b = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k, block, 0) != hipSuccess || b < 1)
    b = 1;
  return b;
}

// The group kernel of a launch: with the point outputs and event solouts
// compiled in only when the launch asks for one of them.
static GroupKernel class_kernel(const SpringArgs& base, const Config& cf) {
  return base.o.pts_mode != kPointsNone || base.o.ev.solout != kSoloutDefault ? cf.kx : cf.k;
}

static Shape shape_of(const SpringArgs& base, const Choice& ch) {
  return {class_kernel(base, kConfigs[ch.cfg]), kConfigs[ch.cfg].g, ch.block};
}

// The kernels of a method other than DOPRI5.
static const ClassKernel* method_kernels(int method) {
#define DE_SPRING_PART_TRY(n) \
  if (const ClassKernel* k = spring_method_part##n(method)) return k;
  DE_SPRING_PARTS(DE_SPRING_PART_TRY)
#undef DE_SPRING_PART_TRY
  return nullptr;
}

// The class's counter has been zeroed.
static int launch_class(const SpringArgs& base, const int32_t* d_list, int64_t len,
                        int64_t work_share_blocks, const Shape& sh, unsigned long long* counter,
                        hipStream_t s) {
  SpringArgs A = base;
  A.list = d_list;
  A.list_len = len;
  A.o.counter = counter;
  int64_t groups_per_block = sh.block / sh.g;
  int64_t need = (len + groups_per_block - 1) / groups_per_block;
  int64_t grid = work_share_blocks < need ? work_share_blocks : need;
  if (grid < 1) grid = 1;
  hipLaunchKernelGGL(sh.kernel, dim3((unsigned)grid), dim3(sh.block), 0, s, A);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

static int config_of(const LaneShape& sh) {
  for (int ci = 0; ci < kNumConfigs; ++ci)
    if (kConfigs[ci].g == sh.g && kConfigs[ci].c == sh.c) return ci;
  return -1;
}

// The shape of 64 lanes for `cap` masses.
static Choice wave_per_system(int cap) {
  Choice ch;
  ch.block = kTunedBlock;
  ch.cfg = config_of({64, cap / 64});
  return ch;
}

// Time every candidate for the size class of `cap` masses on (up to) 8192 systems.
static Choice autotune(const SpringArgs& base, int cap, const int32_t* d_list, int64_t len,
                       unsigned long long* counter, hipStream_t s) {
  Choice best;
  best.block = kTunedBlock;
  int candidates = 0;
  for (int ci = 0; ci < kNumConfigs; ++ci)
    if (tuned_shape(kConfigs[ci], cap)) {
      best.cfg = ci;
      candidates += 1;
    }
  if (candidates <= 1) return best;
  // Solves of other streams still run: their classes would lengthen some of the times.
  for (hipStream_t other : g_streams)
    if (hipStreamSynchronize(other) != hipSuccess) return best;
  best.cfg = -1;
  float best_ms = 1e30f;
  const int64_t sample = len < 8192 ? len : 8192;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return best;
  for (int ci = 0; ci < kNumConfigs; ++ci) {
    if (!tuned_shape(kConfigs[ci], cap)) continue;
    Choice ch;
    ch.cfg = ci;
    ch.block = kTunedBlock;
    const int64_t full =
        (int64_t)g_num_cu * blocks_per_cu(class_kernel(base, kConfigs[ci]), ch.block);
    (void)hipEventRecord(e0, s);
    hipLaunchKernelGGL(spring_zero_counters, dim3(1), dim3(64), 0, s, counter, 1);
    if (launch_class(base, d_list, sample, full, shape_of(base, ch), counter, s) != 0) continue;
    (void)hipEventRecord(e1, s);
    if (hipEventSynchronize(e1) != hipSuccess) continue;
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (ms < best_ms) {
      best_ms = ms;
      best = ch;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return best;
}

// One thread per system: when the caller asks for it, and for the point
// outputs and event solouts of the methods beside DOPRI5 (their group kernels
// carry the final state and the t_eval output: with an event's root search
// inlined around a 16-stage interpolant they do not compile in minutes).
static bool lane_mapping(const de_ode_batch* b) {
  return b->mapping == DE_MAP_LANE ||
         (b->method != DE_METHOD_DOPRI5 &&
          (b->points != DE_POINTS_NONE || b->event_solout != DE_SOLOUT_DEFAULT));
}

// Start of each system's point states in points_y (n + 1 values): the slot
// counts times the state lengths, summed over the systems before it.
// Returns 0, 2 for offsets that decrease or are negative, -1 on a HIP error.
static int point_state_offsets(const OdeArgs& a, const int32_t* host_sizes, int64_t n,
                               std::vector<int64_t>& ypos, hipStream_t s) {
  std::vector<int64_t> off((size_t)n + 1);
  if (hipMemcpyAsync(off.data(), a.pts_offset, sizeof(int64_t) * (n + 1),
                     hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return -1;
  ypos.assign((size_t)n + 1, 0);
  for (int64_t i = 0; i < n; ++i) {
    const int64_t slots = off[i + 1] - off[i];
    if (off[i] < 0 || slots < 0) return 2;
    ypos[i + 1] = ypos[i] + slots * 2 * (int64_t)host_sizes[i];
  }
  return 0;
}

// The device memory of a group launch: see launch_spring.
static size_t group_block_bytes(int64_t n, bool pts) {
  return sizeof(unsigned long long) * (2 * kMaxClasses + 1) +
         (pts ? sizeof(int64_t) * (size_t)(n + 1) : 0) + sizeof(int32_t) * (size_t)n;
}

int64_t spring_workspace_bytes(const de_ode_batch* b) {
  if (!b) return 0;
  if (lane_mapping(b)) {
    // The one-lane solver's state-length vectors per system (offsets are
    // device memory here, so the bound uses 512 doubles per system), one more
    // for an event solout and, with a point output, n + 1 state offsets into
    // points_y.
    const int vectors =
        lane_solver(b->method).vectors + (b->event_solout != DE_SOLOUT_DEFAULT ? 1 : 0);
    return (int64_t)vectors * 512 * 8 * b->n +
           (b->points != DE_POINTS_NONE ? 8 * (b->n + 1) : 0);
  }
  return (int64_t)group_block_bytes(b->n, b->points != DE_POINTS_NONE);
}

int launch_spring(const de_ode_batch* b, const int32_t* host_sizes, const OdeArgs& a,
                  int sched, hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (ensure_runtime() != 0) return -1;
  const int64_t n = b->n;
  SpringArgs base;
  base.o = a;
  base.sizes = b->sizes;
  base.state_offset = b->state_offset;
  base.param_offset = b->param_offset;
  base.work = nullptr;
  base.pts_ypos = nullptr;
  base.ev_work = nullptr;
  base.ystate = nullptr;
  base.list = nullptr;
  base.list_len = 0;
  // Host-side size scan: validity, total state length, classes.
  const bool dopri5 = b->method == DE_METHOD_DOPRI5;
  const ClassSet cs = class_set(dopri5);
  int64_t state_len = 0;
  std::vector<int64_t> count(cs.n, 0);
  uint8_t class_of_size[257];
  for (int m = 0; m <= 256; ++m) class_of_size[m] = (uint8_t)class_index(cs, m);
  const bool comp_event =
      b->event_solout != DE_SOLOUT_DEFAULT && a.ev.fn == kEventComponent;
  for (int64_t i = 0; i < n; ++i) {
    const int32_t m = host_sizes[i];
    if (m < 1 || m > 256) return 1;
    if (comp_event && b->event_component >= 2 * m) return 3;
    count[class_of_size[m]] += 1;
    state_len += 2 * (int64_t)m;
  }
  const bool pts = b->points != DE_POINTS_NONE;
  std::vector<int64_t> ypos;
  if (pts) {
    const int r = point_state_offsets(a, host_sizes, n, ypos, s);
    if (r != 0) return r;
  }
  if (lane_mapping(b)) {
    const LaneSolver ls = lane_solver(b->method);
    const bool events = b->event_solout != DE_SOLOUT_DEFAULT;
    const int64_t vec_len = ((int64_t)ls.vectors + (events ? 1 : 0)) * state_len;
    const int64_t need = vec_len + (pts ? n + 1 : 0);
    // The vectors come from the library's workspace pool (within its budget)
    // and return to it, stream-ordered, after the launch.
    double* work = nullptr;
    if (workspace_alloc((void**)&work, sizeof(double) * need, s) != hipSuccess) return -4;
    base.work = work;
    if (events) base.ev_work = work + (int64_t)ls.vectors * state_len;
    if (pts) {
      int64_t* d_ypos = (int64_t*)(work + vec_len);
      if (hipMemcpyAsync(d_ypos, ypos.data(), sizeof(int64_t) * (n + 1), hipMemcpyHostToDevice,
                         s) != hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess) {
        (void)hipFreeAsync(work, s);
        return -1;
      }
      base.pts_ypos = d_ypos;
    }
    int64_t grid = (n + kSpringBlock - 1) / kSpringBlock;
    hipLaunchKernelGGL(ls.kernel, dim3((unsigned)grid), dim3(kSpringBlock), 0, s, base);
    const hipError_t e = hipGetLastError();
    return hipFreeAsync(work, s) == hipSuccess && e == hipSuccess ? 0 : -1;
  }
  // Group mapping: the launch's classes, and their lists to upload (one buffer,
  // classes back to back).
  const bool fixed_group = b->mapping == DE_MAP_GROUP && b->group_size > 0;
  const Merge merge = fixed_group ? kMergeAll : merge_of(dopri5, count.data());
  std::vector<int> merged(cs.n);
  std::vector<int64_t> own = count;
  count.assign(cs.n, 0);
  for (int k = 0; k < cs.n; ++k) {
    merged[k] = class_index(cs, merged_cap(merge, cs.caps[k]));
    count[merged[k]] += own[k];
  }
  ListArgs lists;
  lists.classes = cs.n;
  int64_t* start = lists.start;
  start[0] = 0;
  for (int k = 0; k < cs.n; ++k) start[k + 1] = start[k] + count[k];
  for (int m = 0; m <= 256; ++m) lists.class_of_size[m] = (uint8_t)merged[class_index(cs, m)];
  // One block for this launch (other launches may run at the same time, on other
  // streams): the classes' work counters and list lengths, the autotuner's counter, the
  // point states' offsets and the lists.
  char* block = nullptr;
  if (workspace_alloc((void**)&block, group_block_bytes(n, pts), s) != hipSuccess) return -4;
  unsigned long long* counters = (unsigned long long*)block;
  unsigned long long* lengths = counters + kMaxClasses;
  unsigned long long* tune_counter = lengths + kMaxClasses;
  int64_t* d_ypos = (int64_t*)(tune_counter + 1);
  int32_t* d_list = (int32_t*)(d_ypos + (pts ? n + 1 : 0));
  if (pts) {
    if (hipMemcpyAsync(d_ypos, ypos.data(), sizeof(int64_t) * (n + 1), hipMemcpyHostToDevice,
                       s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
      (void)hipFreeAsync(block, s);
      return -1;
    }
    base.pts_ypos = d_ypos;
  }
  hipLaunchKernelGGL(spring_zero_counters, dim3(1), dim3(64), 0, s, counters, 2 * kMaxClasses);
  hipLaunchKernelGGL(spring_list_kernel, dim3((unsigned)((n + kListBlock - 1) / kListBlock)),
                     dim3(kListBlock), 0, s, lists, b->sizes, n, lengths, d_list);
  bool ok = hipGetLastError() == hipSuccess;
  // Choose a configuration per class.
  const ClassKernel* fixed = method_kernels(b->method);
  std::vector<Shape> shape(cs.n);
  for (int k = 0; k < cs.n; ++k) {
    if (count[k] == 0) continue;
    if (fixed) {
      shape[k] = {fixed[k].k, fixed[k].g, kGroupBlock};
      continue;
    }
    Choice ch;
    if (fixed_group) {
      ch.cfg = config_of(group_shape(cs.caps[k], b->group_size));
    } else {
      if (merge == kMergeFew) {
        ch = wave_per_system(cs.caps[k]);
      } else {
        Choice& known = g_tuned[merge][cs.caps[k]];
        if (known.cfg < 0)
          known = autotune(base, cs.caps[k], d_list + start[k], count[k], tune_counter, s);
        ch = known;
      }
      for (int o = 0; o < cs.n; ++o)
        if (merged[o] == k && own[o] > 0) g_solved[cs.caps[o]] = ch;
    }
    if (ch.cfg < 0) {
      (void)hipFreeAsync(block, s);
      return -1;
    }
    shape[k] = shape_of(base, ch);
  }
  // Launch classes concurrently: every class, smallest first; merged classes, that of up
  // to 16 masses first, then the others largest first.  Every class kernel gets a
  // full-device grid (capped by its number of systems): the kernels are persistent and
  // exit when their class is drained, so blocks of the classes launched later are
  // dispatched as those of earlier ones retire, and the dispatcher balances the classes.
  // The small classes hold few waves whose long step sequences set their time (latency,
  // not throughput): started first, they run beside the large classes (65 536 systems of
  // 4 to 256 masses, 8.9 against 9.1 ms with only those up to 16 masses before the
  // rest; 16 384 with 1% above 8 masses 1.44 against 1.65).  One wavefront per system
  // has no such classes (8192 of 4 to 256 masses with RK4 1.76 ms largest first, 2.09
  // smallest first).  (A fixed share per class left the
  // GPU idle whenever classes waited behind others for one of the few
  // hardware queues a process gets; ordering each class's systems by size was
  // slower, 14.9 ms: it scatters the group's memory accesses.)
  std::vector<int> launch_order;
  const int ascending = merge == kMergeAll ? 256 : 16;
  for (int k = 0; k < cs.n && cs.caps[k] <= ascending; ++k) launch_order.push_back(k);
  for (int k = cs.n - 1; k >= 0 && cs.caps[k] > ascending; --k) launch_order.push_back(k);
  ok = ok && hipEventRecord(g_fork, s) == hipSuccess;
  for (int q = 0; q < cs.n && ok; ++q) {
    const int k = launch_order[q];
    if (count[k] == 0) continue;
    const Shape& sh = shape[k];
    int64_t share = (int64_t)g_num_cu * blocks_per_cu(sh.kernel, sh.block);
    ok = hipStreamWaitEvent(g_streams[k], g_fork, 0) == hipSuccess &&
         launch_class(base, d_list + start[k], count[k], share, sh, counters + k,
                      g_streams[k]) == 0 &&
         hipEventRecord(g_join[k], g_streams[k]) == hipSuccess;
  }
  // The caller's stream waits once every class is launched: it shares a hardware queue
  // with some of the class streams, and a class launched behind one of its waits would
  // start when another class ends (16 384 chains of 4 to 256 masses with the middle
  // classes: 2.7 to 3.5 ms, by the queue that the caller's stream has, against 2.5 to
  // 2.6).
  for (int k : launch_order)
    if (ok && count[k] > 0) ok = hipStreamWaitEvent(s, g_join[k], 0) == hipSuccess;
  // The call returns without waiting, as every solve on device memory: the block goes
  // back to the pool after the classes (stream order).  If a launch failed, the stream
  // may not wait for all that were made before it.
  if (!ok) (void)hipDeviceSynchronize();
  ok = hipFreeAsync(block, s) == hipSuccess && ok;
  return ok ? 0 : -1;
}

// Introspection: the shape (G, C, block) that the systems of the size class of `cap`
// masses were last solved with, or -1 if none has been solved with a shape of the
// library's choice.
int spring_tuned(int cap, int* g, int* c, int* block) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_solved.find(cap);
  if (it == g_solved.end() || it->second.cfg < 0) return -1;
  *g = kConfigs[it->second.cfg].g;
  *c = kConfigs[it->second.cfg].c;
  *block = it->second.block;
  return 0;
}

}  // namespace parity
}  // namespace de
