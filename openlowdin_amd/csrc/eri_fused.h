// One launch for the J/K work of all quartet classes of a small build.
//
// A molecule of a few dozen functions has a few quartets to a few thousand
// per class: each class launch lasts as long as one lane's serial chain
// (20-100 us) and leaves the GPU empty, and the GPU runs at most four
// launches at a time (its hardware queues), so 21 launches cost several
// chains one after another plus their own issue.  Here every class's tasks
// are workgroups of one launch: the classes run side by side and the build
// waits for one chain.  The price is the register budget of the largest
// class (one wavefront per SIMD), so builds that fill the GPU keep the class
// launches.
#pragma once
#include "eri_coop.h"

namespace lowdin {

template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void fused_class(const FusedArgs& f, int seg, const Task& t, unsigned int* counts,
                                            double* lds, double* bpd, unsigned int* wg) {
  constexpr int L = LA + LB + LC + LD;
  JKArgs a{};
  a.mols = f.mols;
  a.boys = f.boys;
  a.cbra = LA * (LA + 1) / 2 + LB;
  a.cket = LC * (LC + 1) / 2 + LD;
  a.same_class = LA == LC && LB == LD;
  a.block = 64;
  a.eps = f.eps;
  if constexpr (L >= kCoopL) {
    a.lds_n = 0;
    jk_coop_body<LA, LB, LC, LD>(a, t, counts, lds, wg);
  } else {
    a.lds_n = f.lds_n;
    a.lmax = f.lmax[seg];
    jk_strip_body<LA, LB, LC, LD, false, false>(a, t, counts, lds, bpd, nullptr, wg);
  }
}

// Doubles of dynamic LDS a class needs at strip width n.
template <int LA, int LB, int LC, int LD>
constexpr int fused_doubles(int n) {
  if constexpr (LA + LB + LC + LD >= kCoopL)
    return coop_wave_doubles<LA, LB, LC, LD>();
  else
    return (ncart(LA) + ncart(LB)) * n;
}

}  // namespace lowdin
