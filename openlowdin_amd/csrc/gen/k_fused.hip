// Generated by gen_eri.py -- do not edit.
// The J/K work of every quartet class as one launch (small builds).
#include "../eri_fused.h"

namespace lowdin {
#include "eri_0000.inc"
LOWDIN_ERI_CLASS(0, 0, 0, 0)
#include "eri_1000.inc"
LOWDIN_ERI_CLASS(1, 0, 0, 0)
#include "eri_1010.inc"
LOWDIN_ERI_CLASS(1, 0, 1, 0)
#include "eri_1100.inc"
LOWDIN_ERI_CLASS(1, 1, 0, 0)
#include "eri_1110.inc"
LOWDIN_ERI_CLASS(1, 1, 1, 0)
#include "eri_1111.inc"
LOWDIN_ERI_CLASS(1, 1, 1, 1)
#include "eri_2000.inc"
LOWDIN_ERI_CLASS(2, 0, 0, 0)
#include "eri_2010.inc"
LOWDIN_ERI_CLASS(2, 0, 1, 0)
#include "eri_2011.inc"
LOWDIN_ERI_CLASS(2, 0, 1, 1)
#include "eri_2020.inc"
LOWDIN_ERI_CLASS(2, 0, 2, 0)
#include "eri_2100.inc"
LOWDIN_ERI_CLASS(2, 1, 0, 0)
#include "eri_2110.inc"
LOWDIN_ERI_CLASS(2, 1, 1, 0)
#include "eri_2111.inc"
LOWDIN_ERI_CLASS(2, 1, 1, 1)
#include "c_2111.inc"
#include "eri_2120.inc"
LOWDIN_ERI_CLASS(2, 1, 2, 0)
#include "c_2120.inc"
#include "eri_2121.inc"
LOWDIN_ERI_CLASS(2, 1, 2, 1)
#include "c_2121.inc"
#include "eri_2200.inc"
LOWDIN_ERI_CLASS(2, 2, 0, 0)
#include "eri_2210.inc"
LOWDIN_ERI_CLASS(2, 2, 1, 0)
#include "c_2210.inc"
#include "eri_2211.inc"
LOWDIN_ERI_CLASS(2, 2, 1, 1)
#include "c_2211.inc"
#include "eri_2220.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 0)
#include "c_2220.inc"
#include "eri_2221.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 1)
#include "c_2221.inc"
#include "eri_2222.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 2)
#include "c_2222.inc"
__global__ __launch_bounds__(64) void jk_fused_kernel(FusedArgs f) {
  extern __shared__ double lds[];
  __shared__ double bpd[kMaxStripPrims * kPrimPairStride];
  __shared__ unsigned int wg[3];
  const int b = blockIdx.x;
  int seg = 0;
  while (seg + 1 < f.nseg && b >= f.first[seg + 1]) ++seg;
  const Task t = f.tasks[b];
  unsigned int* counts = f.counts ? f.counts + 3 * (size_t)b : nullptr;
  switch (f.cls[seg]) {
    case 0: fused_class<0, 0, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 1000: fused_class<1, 0, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 1010: fused_class<1, 0, 1, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 1100: fused_class<1, 1, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 1110: fused_class<1, 1, 1, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 1111: fused_class<1, 1, 1, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2000: fused_class<2, 0, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2010: fused_class<2, 0, 1, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2011: fused_class<2, 0, 1, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2020: fused_class<2, 0, 2, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2100: fused_class<2, 1, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2110: fused_class<2, 1, 1, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2111: fused_class<2, 1, 1, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2120: fused_class<2, 1, 2, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2121: fused_class<2, 1, 2, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2200: fused_class<2, 2, 0, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2210: fused_class<2, 2, 1, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2211: fused_class<2, 2, 1, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2220: fused_class<2, 2, 2, 0>(f, seg, t, counts, lds, bpd, wg); break;
    case 2221: fused_class<2, 2, 2, 1>(f, seg, t, counts, lds, bpd, wg); break;
    case 2222: fused_class<2, 2, 2, 2>(f, seg, t, counts, lds, bpd, wg); break;
  }
}

size_t jk_fused_lds(int nmax) {
  int d = 0;
  d = std::max(d, fused_doubles<0, 0, 0, 0>(nmax));
  d = std::max(d, fused_doubles<1, 0, 0, 0>(nmax));
  d = std::max(d, fused_doubles<1, 0, 1, 0>(nmax));
  d = std::max(d, fused_doubles<1, 1, 0, 0>(nmax));
  d = std::max(d, fused_doubles<1, 1, 1, 0>(nmax));
  d = std::max(d, fused_doubles<1, 1, 1, 1>(nmax));
  d = std::max(d, fused_doubles<2, 0, 0, 0>(nmax));
  d = std::max(d, fused_doubles<2, 0, 1, 0>(nmax));
  d = std::max(d, fused_doubles<2, 0, 1, 1>(nmax));
  d = std::max(d, fused_doubles<2, 0, 2, 0>(nmax));
  d = std::max(d, fused_doubles<2, 1, 0, 0>(nmax));
  d = std::max(d, fused_doubles<2, 1, 1, 0>(nmax));
  d = std::max(d, fused_doubles<2, 1, 1, 1>(nmax));
  d = std::max(d, fused_doubles<2, 1, 2, 0>(nmax));
  d = std::max(d, fused_doubles<2, 1, 2, 1>(nmax));
  d = std::max(d, fused_doubles<2, 2, 0, 0>(nmax));
  d = std::max(d, fused_doubles<2, 2, 1, 0>(nmax));
  d = std::max(d, fused_doubles<2, 2, 1, 1>(nmax));
  d = std::max(d, fused_doubles<2, 2, 2, 0>(nmax));
  d = std::max(d, fused_doubles<2, 2, 2, 1>(nmax));
  d = std::max(d, fused_doubles<2, 2, 2, 2>(nmax));
  return (size_t)d * sizeof(double);
}

void launch_jk_fused(const FusedArgs& f, hipStream_t s) {
  if (f.nseg <= 0 || f.first[f.nseg] <= 0) return;
  hipLaunchKernelGGL(jk_fused_kernel, dim3(f.first[f.nseg]), dim3(64), jk_fused_lds(f.lds_n), s, f);
}
}  // namespace lowdin
