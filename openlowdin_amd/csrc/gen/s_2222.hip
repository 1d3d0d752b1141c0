// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|22): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2222.inc"
LOWDIN_ERI_CLASS(2, 2, 2, 2)
#include "c_2222.inc"

void launch_st_2222(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 2, 2, 2>(args, s); }
void launch_cst_2222(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 2, 2, 2>(args, s); }
void store_attr_2222() { store_attr_t<2, 2, 2, 2>(); }
}  // namespace lowdin
