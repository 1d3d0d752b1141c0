// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|21): G12 (Gaussian-geminal) Fock build and coupling.
#include "../eri_g12.h"

namespace lowdin {
#include "eri_2221.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 1)
LOWDIN_G12_CLASS(2, 2, 2, 1)
#include "c_2221.inc"

void launch_gjk_2221(const G12Args& args, hipStream_t s) { launch_g12_t<2, 2, 2, 1>(args, s); }
void launch_gcp_2221(const G12CouplingArgs& args, hipStream_t s) { launch_g12cp_t<2, 2, 2, 1>(args, s); }
}  // namespace lowdin
