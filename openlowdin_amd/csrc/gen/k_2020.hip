// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (20|20): fused ERI + J/K, coupling, Schwarz.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_2020.inc"
LOWDIN_ERI_CLASS(2, 0, 2, 0)

void launch_jk_2020(const JKArgs& args, hipStream_t s) { launch_jk_t<2, 0, 2, 0>(args, s); }
void launch_jks_2020(const JKArgs& args, hipStream_t s) { launch_jk_strip_t<2, 0, 2, 0>(args, s); }
void launch_cp_2020(const CouplingArgs& args, hipStream_t s) { launch_cp_t<2, 0, 2, 0>(args, s); }
void launch_schwarz_20(PairInfo* pairs, int npairs, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) { launch_schwarz_t<2, 0>(pairs, npairs, ls, prim, boys, norma, s); }
}  // namespace lowdin
