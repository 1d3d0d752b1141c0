// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|10): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2210.inc"
LOWDIN_ERI_CLASS(2, 2, 1, 0)
#include "c_2210.inc"

void launch_st_2210(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 2, 1, 0>(args, s); }
void launch_cst_2210(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 2, 1, 0>(args, s); }
void store_attr_2210() { store_attr_t<2, 2, 1, 0>(); }
}  // namespace lowdin
