// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|11): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2111.inc"
LOWDIN_ERI_CLASS(2, 1, 1, 1)
#include "c_2111.inc"

void launch_st_2111(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 1, 1, 1>(args, s); }
void launch_cst_2111(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 1, 1, 1>(args, s); }
void store_attr_2111() { store_attr_t<2, 1, 1, 1>(); }
}  // namespace lowdin
