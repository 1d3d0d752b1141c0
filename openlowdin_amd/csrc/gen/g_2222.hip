// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|22): G12 (Gaussian-geminal) Fock build and coupling.
#include "../eri_g12.h"

namespace lowdin {
#include "eri_2222.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 2)
LOWDIN_G12_CLASS(2, 2, 2, 2)
#include "c_2222.inc"

void launch_gjk_2222(const G12Args& args, hipStream_t s) { launch_g12_t<2, 2, 2, 2>(args, s); }
void launch_gcp_2222(const G12CouplingArgs& args, hipStream_t s) { launch_g12cp_t<2, 2, 2, 2>(args, s); }
}  // namespace lowdin
