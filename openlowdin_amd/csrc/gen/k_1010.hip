// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (10|10): fused ERI + J/K, coupling, Schwarz.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_1010.inc"
LOWDIN_ERI_CLASS(1, 0, 1, 0)

void launch_jk_1010(const JKArgs& args, hipStream_t s) { launch_jk_t<1, 0, 1, 0>(args, s); }
void launch_jks_1010(const JKArgs& args, hipStream_t s) { launch_jk_strip_t<1, 0, 1, 0>(args, s); }
void launch_cp_1010(const CouplingArgs& args, hipStream_t s) { launch_cp_t<1, 0, 1, 0>(args, s); }
void launch_schwarz_10(PairInfo* pairs, int npairs, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) { launch_schwarz_t<1, 0>(pairs, npairs, ls, prim, boys, norma, s); }
}  // namespace lowdin
