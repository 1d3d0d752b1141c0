// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|21): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2121.inc"
LOWDIN_ERI_CLASS(2, 1, 2, 1)
#include "c_2121.inc"

void launch_st_2121(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 1, 2, 1>(args, s); }
void launch_cst_2121(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 1, 2, 1>(args, s); }
void store_attr_2121() { store_attr_t<2, 1, 2, 1>(); }
}  // namespace lowdin
