// Generated by gen_eri.py -- do not edit.
// Kernels of quartet class (22|00): integral store and first-quarter transform.
#include "../eri_store.h"

namespace lowdin {
#include "eri_2200.inc"
LOWDIN_ERI_CLASS(2, 2, 0, 0)

void launch_st_2200(const StoreArgs& args, hipStream_t s) { launch_store_t<2, 2, 0, 0>(args, s); }
void launch_cst_2200(const CouplingStoreArgs& args, hipStream_t s) { launch_cstore_t<2, 2, 0, 0>(args, s); }
void store_attr_2200() { store_attr_t<2, 2, 0, 0>(); }
}  // namespace lowdin
