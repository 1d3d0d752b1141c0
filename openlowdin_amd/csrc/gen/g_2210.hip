// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|10): G12 (Gaussian-geminal) Fock build and coupling.
#include "../eri_g12.h"

namespace lowdin {
#include "eri_2210.inc"
LOWDIN_ERI_CLASS(2, 2, 1, 0)
LOWDIN_G12_CLASS(2, 2, 1, 0)
#include "c_2210.inc"

void launch_gjk_2210(const G12Args& args, hipStream_t s) { launch_g12_t<2, 2, 1, 0>(args, s); }
void launch_gcp_2210(const G12CouplingArgs& args, hipStream_t s) { launch_g12cp_t<2, 2, 1, 0>(args, s); }
}  // namespace lowdin
