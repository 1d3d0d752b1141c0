// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|21): fused ERI + J/K, coupling, wave-cooperative J/K and coupling.
#include "../eri_coop.h"

namespace lowdin {
#include "eri_2221.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 1)
#include "c_2221.inc"

bool launch_jkc_2221(const JKArgs& args, hipStream_t s) { return launch_jk_coop_t<2, 2, 2, 1>(args, s); }
bool launch_cpc_2221(const CouplingArgs& args, hipStream_t s) { return launch_cp_coop_t<2, 2, 2, 1>(args, s); }
void coop_attr_2221() { coop_attr_t<2, 2, 2, 1>(); }
}  // namespace lowdin
