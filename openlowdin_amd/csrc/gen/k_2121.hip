// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|21): fused ERI + J/K, coupling, Schwarz, wave-cooperative J/K and coupling.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_2121.inc"
LOWDIN_ERI_CLASS(2, 1, 2, 1)
#include "c_2121.inc"

void launch_schwarz_21(PairInfo* pairs, int npairs, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) { launch_schwarz_t<2, 1>(pairs, npairs, ls, prim, boys, norma, s); }
bool launch_jkc_2121(const JKArgs& args, hipStream_t s) { return launch_jk_coop_t<2, 1, 2, 1>(args, s); }
bool launch_cpc_2121(const CouplingArgs& args, hipStream_t s) { return launch_cp_coop_t<2, 1, 2, 1>(args, s); }
void coop_attr_2121() { coop_attr_t<2, 1, 2, 1>(); }
}  // namespace lowdin
