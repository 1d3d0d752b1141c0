// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (11|11): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_1111.inc"
LOWDIN_ERI_CLASS(1, 1, 1, 1)

void launch_st_1111(const StoreArgs& args, hipStream_t s) { launch_store_t<1, 1, 1, 1>(args, s); }
void launch_cst_1111(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<1, 1, 1, 1>(args, s); }
void store_attr_1111() { store_attr_t<1, 1, 1, 1>(); }
}  // namespace lowdin
