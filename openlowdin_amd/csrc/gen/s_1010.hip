// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (10|10): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_1010.inc"
LOWDIN_ERI_CLASS(1, 0, 1, 0)

void launch_st_1010(const StoreArgs& args, hipStream_t s) { launch_store_t<1, 0, 1, 0>(args, s); }
void launch_cst_1010(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<1, 0, 1, 0>(args, s); }
void store_attr_1010() { store_attr_t<1, 0, 1, 0>(); }
}  // namespace lowdin
