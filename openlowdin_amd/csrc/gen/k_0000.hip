// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (00|00): fused ERI + J/K, coupling, Schwarz.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_0000.inc"
LOWDIN_ERI_CLASS(0, 0, 0, 0)

void launch_jk_0000(const JKArgs& args, hipStream_t s) { launch_jk_t<0, 0, 0, 0>(args, s); }
void launch_jks_0000(const JKArgs& args, hipStream_t s) { launch_jk_strip_t<0, 0, 0, 0>(args, s); }
void launch_cp_0000(const CouplingArgs& args, hipStream_t s) { launch_cp_t<0, 0, 0, 0>(args, s); }
void launch_schwarz_00(PairInfo* pairs, int npairs, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) { launch_schwarz_t<0, 0>(pairs, npairs, ls, prim, boys, norma, s); }
}  // namespace lowdin
