// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|20): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2120.inc"
LOWDIN_ERI_CLASS(2, 1, 2, 0)
#include "c_2120.inc"

void launch_st_2120(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 1, 2, 0>(args, s); }
void launch_cst_2120(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 1, 2, 0>(args, s); }
void store_attr_2120() { store_attr_t<2, 1, 2, 0>(); }
}  // namespace lowdin
