// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (20|11): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2011.inc"
LOWDIN_ERI_CLASS(2, 0, 1, 1)

void launch_st_2011(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 0, 1, 1>(args, s); }
void launch_cst_2011(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 0, 1, 1>(args, s); }
void store_attr_2011() { store_attr_t<2, 0, 1, 1>(); }
}  // namespace lowdin
