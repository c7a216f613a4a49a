// Group kernels of the spring chains for the methods beside DOPRI5
// (de_spring_group.h), one to three methods per translation unit
// (DE_SPRING_PART).
#include <hip/hip_runtime.h>

#include "de_launch.h"
#include "de_spring.h"
#include "de_spring_group.h"

#ifndef DE_SPRING_PART
#error "define DE_SPRING_PART"
#endif
#define DE_PASTE2(a, b) a##b
#define DE_PASTE(a, b) DE_PASTE2(a, b)

namespace de {
namespace parity {

// One lane per mass up to 64 masses, then two and four masses per lane.
// VEC: state vectors a step keeps in registers (stages, states, combinations).
#define DE_CLASS(SOLVER, VEC, G, C) \
  {G, spring_method_kernel<SOLVER(G, C), group_waves(VEC, C)>}
#define DE_CLASSES(SOLVER, VEC)                                                          \
  {DE_CLASS(SOLVER, VEC, 4, 1),  DE_CLASS(SOLVER, VEC, 8, 1),  DE_CLASS(SOLVER, VEC, 16, 1), \
   DE_CLASS(SOLVER, VEC, 32, 1), DE_CLASS(SOLVER, VEC, 64, 1), DE_CLASS(SOLVER, VEC, 64, 2), \
   DE_CLASS(SOLVER, VEC, 64, 4)}

#define DE_RK4(G, C) GroupFixed<4, G, C>
#define DE_EULER(G, C) GroupFixed<1, G, C>
#define DE_DOP853(G, C) GroupDop853<G, C>
#define DE_ERK_SOLVER(TAB) DE_PASTE(DE_ERK_, TAB)
#define DE_ERK_Rkf45(G, C) GroupErk<erk_tab::Rkf45, G, C>
#define DE_ERK_CashKarp(G, C) GroupErk<erk_tab::CashKarp, G, C>
#define DE_ERK_Rkv655e(G, C) GroupErk<erk_tab::Rkv655e, G, C>
#define DE_ERK_Rkv656e(G, C) GroupErk<erk_tab::Rkv656e, G, C>
#define DE_ERK_Rkv766e(G, C) GroupErk<erk_tab::Rkv766e, G, C>
#define DE_ERK_Rkv767e(G, C) GroupErk<erk_tab::Rkv767e, G, C>
#define DE_ERK_Rkv877e(G, C) GroupErk<erk_tab::Rkv877e, G, C>
#define DE_ERK_Rkv878e(G, C) GroupErk<erk_tab::Rkv878e, G, C>
#define DE_ERK_Rkv988e(G, C) GroupErk<erk_tab::Rkv988e, G, C>
#define DE_ERK_Rkv989e(G, C) GroupErk<erk_tab::Rkv989e, G, C>
#define DE_ERK_CASE(METHOD, TAB)                                                         \
  case METHOD: {                                                                         \
    static const ClassKernel k[] = DE_CLASSES(DE_ERK_SOLVER(TAB), erk_tab::TAB::S + 5);  \
    return k;                                                                            \
  }

const ClassKernel* DE_PASTE(spring_method_part, DE_SPRING_PART)(int method) {
  switch (method) {
#if DE_SPRING_PART == 0
    case kMethodRk4: {
      static const ClassKernel k[] = DE_CLASSES(DE_RK4, 8);
      return k;
    }
    case kMethodEuler: {
      static const ClassKernel k[] = DE_CLASSES(DE_EULER, 6);
      return k;
    }
    case kMethodDop853: {
      static const ClassKernel k[] = DE_CLASSES(DE_DOP853, 17);
      return k;
    }
#elif DE_SPRING_PART == 1
    DE_ERK_CASE(kMethodRkf45, Rkf45)
    DE_ERK_CASE(kMethodCashKarp, CashKarp)
#elif DE_SPRING_PART == 2
    DE_ERK_CASE(kMethodRkv655e, Rkv655e)
    DE_ERK_CASE(kMethodRkv656e, Rkv656e)
#elif DE_SPRING_PART == 3
    DE_ERK_CASE(kMethodRkv766e, Rkv766e)
    DE_ERK_CASE(kMethodRkv767e, Rkv767e)
#elif DE_SPRING_PART == 4
    DE_ERK_CASE(kMethodRkv877e, Rkv877e)
    DE_ERK_CASE(kMethodRkv878e, Rkv878e)
#elif DE_SPRING_PART == 5
    DE_ERK_CASE(kMethodRkv988e, Rkv988e)
#elif DE_SPRING_PART == 6
    DE_ERK_CASE(kMethodRkv989e, Rkv989e)
#endif
    default: return nullptr;
  }
}

}  // namespace parity
}  // namespace de
