// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|11): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2211.inc"
LOWDIN_ERI_CLASS(2, 2, 1, 1)
#include "c_2211.inc"

void launch_st_2211(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 2, 1, 1>(args, s); }
void launch_cst_2211(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 2, 1, 1>(args, s); }
void store_attr_2211() { store_attr_t<2, 2, 1, 1>(); }
}  // namespace lowdin
