// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (11|11): fused ERI + J/K, coupling, Schwarz.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_1111.inc"
LOWDIN_ERI_CLASS(1, 1, 1, 1)

void launch_jk_1111(const JKArgs& args, hipStream_t s) { launch_jk_t<1, 1, 1, 1>(args, s); }
void launch_jks_1111(const JKArgs& args, hipStream_t s) { launch_jk_strip_t<1, 1, 1, 1>(args, s); }
void launch_cp_1111(const CouplingArgs& args, hipStream_t s) { launch_cp_t<1, 1, 1, 1>(args, s); }
void launch_schwarz_11(PairInfo* pairs, int npairs, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) { launch_schwarz_t<1, 1>(pairs, npairs, ls, prim, boys, norma, s); }
}  // namespace lowdin
