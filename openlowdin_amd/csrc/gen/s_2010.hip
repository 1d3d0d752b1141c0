// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (20|10): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2010.inc"
LOWDIN_ERI_CLASS(2, 0, 1, 0)

void launch_st_2010(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 0, 1, 0>(args, s); }
void launch_cst_2010(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 0, 1, 0>(args, s); }
void store_attr_2010() { store_attr_t<2, 0, 1, 0>(); }
}  // namespace lowdin
