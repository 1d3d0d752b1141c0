// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (21|00): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2100.inc"
LOWDIN_ERI_CLASS(2, 1, 0, 0)

void launch_st_2100(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 1, 0, 0>(args, s); }
void launch_cst_2100(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 1, 0, 0>(args, s); }
void store_attr_2100() { store_attr_t<2, 1, 0, 0>(); }
}  // namespace lowdin
