// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|20): fused ERI + J/K, coupling, wave-cooperative J/K and coupling.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_2220.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 0)
#include "c_2220.inc"

bool launch_jkc_2220(const JKArgs& args, hipStream_t s) { return launch_jk_coop_t<2, 2, 2, 0>(args, s); }
bool launch_cpc_2220(const CouplingArgs& args, hipStream_t s) { return launch_cp_coop_t<2, 2, 2, 0>(args, s); }
void coop_attr_2220() { coop_attr_t<2, 2, 2, 0>(); }
}  // namespace lowdin
