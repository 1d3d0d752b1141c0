// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (10|00): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_1000.inc"
LOWDIN_ERI_CLASS(1, 0, 0, 0)

void launch_st_1000(const StoreArgs& args, hipStream_t s) { launch_store_t<1, 0, 0, 0>(args, s); }
void launch_cst_1000(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<1, 0, 0, 0>(args, s); }
void store_attr_1000() { store_attr_t<1, 0, 0, 0>(); }
}  // namespace lowdin
