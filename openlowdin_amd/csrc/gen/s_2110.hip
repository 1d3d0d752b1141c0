// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|10): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2110.inc"
LOWDIN_ERI_CLASS(2, 1, 1, 0)

void launch_st_2110(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 1, 1, 0>(args, s); }
void launch_cst_2110(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 1, 1, 0>(args, s); }
void store_attr_2110() { store_attr_t<2, 1, 1, 0>(); }
}  // namespace lowdin
