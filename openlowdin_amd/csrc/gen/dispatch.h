// Generated by gen_eri.py -- do not edit.
#pragma once
#include "../lowdin_kernels.h"
namespace lowdin {
void launch_jk_0000(const JKArgs&, hipStream_t);
void launch_jks_0000(const JKArgs&, hipStream_t);
void launch_cp_0000(const CouplingArgs&, hipStream_t);
void launch_st_0000(const StoreArgs&, hipStream_t);
void launch_cst_0000(const CouplingStoreArgs&, hipStream_t);
void store_attr_0000();
void launch_gjk_0000(const G12Args&, hipStream_t);
void launch_gcp_0000(const G12CouplingArgs&, hipStream_t);
void launch_jk_1000(const JKArgs&, hipStream_t);
void launch_jks_1000(const JKArgs&, hipStream_t);
void launch_cp_1000(const CouplingArgs&, hipStream_t);
void launch_st_1000(const StoreArgs&, hipStream_t);
void launch_cst_1000(const CouplingStoreArgs&, hipStream_t);
void store_attr_1000();
void launch_gjk_1000(const G12Args&, hipStream_t);
void launch_gcp_1000(const G12CouplingArgs&, hipStream_t);
void launch_jk_1010(const JKArgs&, hipStream_t);
void launch_jks_1010(const JKArgs&, hipStream_t);
void launch_cp_1010(const CouplingArgs&, hipStream_t);
void launch_st_1010(const StoreArgs&, hipStream_t);
void launch_cst_1010(const CouplingStoreArgs&, hipStream_t);
void store_attr_1010();
void launch_gjk_1010(const G12Args&, hipStream_t);
void launch_gcp_1010(const G12CouplingArgs&, hipStream_t);
void launch_jk_1100(const JKArgs&, hipStream_t);
void launch_jks_1100(const JKArgs&, hipStream_t);
void launch_cp_1100(const CouplingArgs&, hipStream_t);
void launch_st_1100(const StoreArgs&, hipStream_t);
void launch_cst_1100(const CouplingStoreArgs&, hipStream_t);
void store_attr_1100();
void launch_gjk_1100(const G12Args&, hipStream_t);
void launch_gcp_1100(const G12CouplingArgs&, hipStream_t);
void launch_jk_1110(const JKArgs&, hipStream_t);
void launch_jks_1110(const JKArgs&, hipStream_t);
void launch_cp_1110(const CouplingArgs&, hipStream_t);
void launch_st_1110(const StoreArgs&, hipStream_t);
void launch_cst_1110(const CouplingStoreArgs&, hipStream_t);
void store_attr_1110();
void launch_gjk_1110(const G12Args&, hipStream_t);
void launch_gcp_1110(const G12CouplingArgs&, hipStream_t);
void launch_jk_1111(const JKArgs&, hipStream_t);
void launch_jks_1111(const JKArgs&, hipStream_t);
void launch_cp_1111(const CouplingArgs&, hipStream_t);
void launch_st_1111(const StoreArgs&, hipStream_t);
void launch_cst_1111(const CouplingStoreArgs&, hipStream_t);
void store_attr_1111();
void launch_gjk_1111(const G12Args&, hipStream_t);
void launch_gcp_1111(const G12CouplingArgs&, hipStream_t);
void launch_jk_2000(const JKArgs&, hipStream_t);
void launch_jks_2000(const JKArgs&, hipStream_t);
void launch_cp_2000(const CouplingArgs&, hipStream_t);
void launch_st_2000(const StoreArgs&, hipStream_t);
void launch_cst_2000(const CouplingStoreArgs&, hipStream_t);
void store_attr_2000();
void launch_gjk_2000(const G12Args&, hipStream_t);
void launch_gcp_2000(const G12CouplingArgs&, hipStream_t);
void launch_jk_2010(const JKArgs&, hipStream_t);
void launch_jks_2010(const JKArgs&, hipStream_t);
void launch_cp_2010(const CouplingArgs&, hipStream_t);
void launch_st_2010(const StoreArgs&, hipStream_t);
void launch_cst_2010(const CouplingStoreArgs&, hipStream_t);
void store_attr_2010();
void launch_gjk_2010(const G12Args&, hipStream_t);
void launch_gcp_2010(const G12CouplingArgs&, hipStream_t);
void launch_jk_2011(const JKArgs&, hipStream_t);
void launch_jks_2011(const JKArgs&, hipStream_t);
void launch_cp_2011(const CouplingArgs&, hipStream_t);
void launch_st_2011(const StoreArgs&, hipStream_t);
void launch_cst_2011(const CouplingStoreArgs&, hipStream_t);
void store_attr_2011();
void launch_gjk_2011(const G12Args&, hipStream_t);
void launch_gcp_2011(const G12CouplingArgs&, hipStream_t);
void launch_jk_2020(const JKArgs&, hipStream_t);
void launch_jks_2020(const JKArgs&, hipStream_t);
void launch_cp_2020(const CouplingArgs&, hipStream_t);
void launch_st_2020(const StoreArgs&, hipStream_t);
void launch_cst_2020(const CouplingStoreArgs&, hipStream_t);
void store_attr_2020();
void launch_gjk_2020(const G12Args&, hipStream_t);
void launch_gcp_2020(const G12CouplingArgs&, hipStream_t);
void launch_jk_2100(const JKArgs&, hipStream_t);
void launch_jks_2100(const JKArgs&, hipStream_t);
void launch_cp_2100(const CouplingArgs&, hipStream_t);
void launch_st_2100(const StoreArgs&, hipStream_t);
void launch_cst_2100(const CouplingStoreArgs&, hipStream_t);
void store_attr_2100();
void launch_gjk_2100(const G12Args&, hipStream_t);
void launch_gcp_2100(const G12CouplingArgs&, hipStream_t);
void launch_jk_2110(const JKArgs&, hipStream_t);
void launch_jks_2110(const JKArgs&, hipStream_t);
void launch_cp_2110(const CouplingArgs&, hipStream_t);
void launch_st_2110(const StoreArgs&, hipStream_t);
void launch_cst_2110(const CouplingStoreArgs&, hipStream_t);
void store_attr_2110();
void launch_gjk_2110(const G12Args&, hipStream_t);
void launch_gcp_2110(const G12CouplingArgs&, hipStream_t);
void launch_jk_2111(const JKArgs&, hipStream_t);
void launch_jks_2111(const JKArgs&, hipStream_t);
void launch_cp_2111(const CouplingArgs&, hipStream_t);
void launch_st_2111(const StoreArgs&, hipStream_t);
void launch_cst_2111(const CouplingStoreArgs&, hipStream_t);
void store_attr_2111();
void launch_gjk_2111(const G12Args&, hipStream_t);
void launch_gcp_2111(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2111(const JKArgs&, hipStream_t);
bool launch_cpc_2111(const CouplingArgs&, hipStream_t);
void coop_attr_2111();
void launch_jk_2120(const JKArgs&, hipStream_t);
void launch_jks_2120(const JKArgs&, hipStream_t);
void launch_cp_2120(const CouplingArgs&, hipStream_t);
void launch_st_2120(const StoreArgs&, hipStream_t);
void launch_cst_2120(const CouplingStoreArgs&, hipStream_t);
void store_attr_2120();
void launch_gjk_2120(const G12Args&, hipStream_t);
void launch_gcp_2120(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2120(const JKArgs&, hipStream_t);
bool launch_cpc_2120(const CouplingArgs&, hipStream_t);
void coop_attr_2120();
void launch_st_2121(const StoreArgs&, hipStream_t);
void launch_cst_2121(const CouplingStoreArgs&, hipStream_t);
void store_attr_2121();
void launch_gjk_2121(const G12Args&, hipStream_t);
void launch_gcp_2121(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2121(const JKArgs&, hipStream_t);
bool launch_cpc_2121(const CouplingArgs&, hipStream_t);
void coop_attr_2121();
void launch_jk_2200(const JKArgs&, hipStream_t);
void launch_jks_2200(const JKArgs&, hipStream_t);
void launch_cp_2200(const CouplingArgs&, hipStream_t);
void launch_st_2200(const StoreArgs&, hipStream_t);
void launch_cst_2200(const CouplingStoreArgs&, hipStream_t);
void store_attr_2200();
void launch_gjk_2200(const G12Args&, hipStream_t);
void launch_gcp_2200(const G12CouplingArgs&, hipStream_t);
void launch_jk_2210(const JKArgs&, hipStream_t);
void launch_jks_2210(const JKArgs&, hipStream_t);
void launch_cp_2210(const CouplingArgs&, hipStream_t);
void launch_st_2210(const StoreArgs&, hipStream_t);
void launch_cst_2210(const CouplingStoreArgs&, hipStream_t);
void store_attr_2210();
void launch_gjk_2210(const G12Args&, hipStream_t);
void launch_gcp_2210(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2210(const JKArgs&, hipStream_t);
bool launch_cpc_2210(const CouplingArgs&, hipStream_t);
void coop_attr_2210();
void launch_st_2211(const StoreArgs&, hipStream_t);
void launch_cst_2211(const CouplingStoreArgs&, hipStream_t);
void store_attr_2211();
void launch_gjk_2211(const G12Args&, hipStream_t);
void launch_gcp_2211(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2211(const JKArgs&, hipStream_t);
bool launch_cpc_2211(const CouplingArgs&, hipStream_t);
void coop_attr_2211();
void launch_st_2220(const StoreArgs&, hipStream_t);
void launch_cst_2220(const CouplingStoreArgs&, hipStream_t);
void store_attr_2220();
void launch_gjk_2220(const G12Args&, hipStream_t);
void launch_gcp_2220(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2220(const JKArgs&, hipStream_t);
bool launch_cpc_2220(const CouplingArgs&, hipStream_t);
void coop_attr_2220();
void launch_st_2221(const StoreArgs&, hipStream_t);
void launch_cst_2221(const CouplingStoreArgs&, hipStream_t);
void store_attr_2221();
void launch_gjk_2221(const G12Args&, hipStream_t);
void launch_gcp_2221(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2221(const JKArgs&, hipStream_t);
bool launch_cpc_2221(const CouplingArgs&, hipStream_t);
void coop_attr_2221();
void launch_st_2222(const StoreArgs&, hipStream_t);
void launch_cst_2222(const CouplingStoreArgs&, hipStream_t);
void store_attr_2222();
void launch_gjk_2222(const G12Args&, hipStream_t);
void launch_gcp_2222(const G12CouplingArgs&, hipStream_t);
bool launch_jkc_2222(const JKArgs&, hipStream_t);
bool launch_cpc_2222(const CouplingArgs&, hipStream_t);
void coop_attr_2222();
void launch_schwarz_00(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
void launch_schwarz_10(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
void launch_schwarz_11(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
void launch_schwarz_20(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
void launch_schwarz_21(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
void launch_schwarz_22(PairInfo*, int, int, const double*, const double*, const double*, hipStream_t);
inline bool dispatch_jk(int la, int lb, int lc, int ld, const JKArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_jk_0000(a, s); return true;
    case 1000: launch_jk_1000(a, s); return true;
    case 1010: launch_jk_1010(a, s); return true;
    case 1100: launch_jk_1100(a, s); return true;
    case 1110: launch_jk_1110(a, s); return true;
    case 1111: launch_jk_1111(a, s); return true;
    case 2000: launch_jk_2000(a, s); return true;
    case 2010: launch_jk_2010(a, s); return true;
    case 2011: launch_jk_2011(a, s); return true;
    case 2020: launch_jk_2020(a, s); return true;
    case 2100: launch_jk_2100(a, s); return true;
    case 2110: launch_jk_2110(a, s); return true;
    case 2111: launch_jk_2111(a, s); return true;
    case 2120: launch_jk_2120(a, s); return true;
    case 2200: launch_jk_2200(a, s); return true;
    case 2210: launch_jk_2210(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_jk_strip(int la, int lb, int lc, int ld, const JKArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_jks_0000(a, s); return true;
    case 1000: launch_jks_1000(a, s); return true;
    case 1010: launch_jks_1010(a, s); return true;
    case 1100: launch_jks_1100(a, s); return true;
    case 1110: launch_jks_1110(a, s); return true;
    case 1111: launch_jks_1111(a, s); return true;
    case 2000: launch_jks_2000(a, s); return true;
    case 2010: launch_jks_2010(a, s); return true;
    case 2011: launch_jks_2011(a, s); return true;
    case 2020: launch_jks_2020(a, s); return true;
    case 2100: launch_jks_2100(a, s); return true;
    case 2110: launch_jks_2110(a, s); return true;
    case 2111: launch_jks_2111(a, s); return true;
    case 2120: launch_jks_2120(a, s); return true;
    case 2200: launch_jks_2200(a, s); return true;
    case 2210: launch_jks_2210(a, s); return true;
    default: return false;
  }
}
// wave-cooperative J/K kernel; false when the class has none or the launch
// does not fit in LDS
inline bool dispatch_jk_coop(int la, int lb, int lc, int ld, const JKArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 2111: return launch_jkc_2111(a, s);
    case 2120: return launch_jkc_2120(a, s);
    case 2121: return launch_jkc_2121(a, s);
    case 2210: return launch_jkc_2210(a, s);
    case 2211: return launch_jkc_2211(a, s);
    case 2220: return launch_jkc_2220(a, s);
    case 2221: return launch_jkc_2221(a, s);
    case 2222: return launch_jkc_2222(a, s);
    default: return false;
  }
}
inline bool has_jk_coop(int la, int lb, int lc, int ld) { return la + lb + lc + ld >= 5; }
// raise the dynamic LDS limit of the kernels that may use more (once per process)
inline void coop_attr_all() {
  store_attr_0000();
  store_attr_1000();
  store_attr_1010();
  store_attr_1100();
  store_attr_1110();
  store_attr_1111();
  store_attr_2000();
  store_attr_2010();
  store_attr_2011();
  store_attr_2020();
  store_attr_2100();
  store_attr_2110();
  store_attr_2111();
  coop_attr_2111();
  store_attr_2120();
  coop_attr_2120();
  store_attr_2121();
  coop_attr_2121();
  store_attr_2200();
  store_attr_2210();
  coop_attr_2210();
  store_attr_2211();
  coop_attr_2211();
  store_attr_2220();
  coop_attr_2220();
  store_attr_2221();
  coop_attr_2221();
  store_attr_2222();
  coop_attr_2222();
}
// wave-cooperative coupling kernel; false when the class has none
inline bool dispatch_cp_coop(int la, int lb, int lc, int ld, const CouplingArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 2111: return launch_cpc_2111(a, s);
    case 2120: return launch_cpc_2120(a, s);
    case 2121: return launch_cpc_2121(a, s);
    case 2210: return launch_cpc_2210(a, s);
    case 2211: return launch_cpc_2211(a, s);
    case 2220: return launch_cpc_2220(a, s);
    case 2221: return launch_cpc_2221(a, s);
    case 2222: return launch_cpc_2222(a, s);
    default: return false;
  }
}
inline bool dispatch_cp(int la, int lb, int lc, int ld, const CouplingArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_cp_0000(a, s); return true;
    case 1000: launch_cp_1000(a, s); return true;
    case 1010: launch_cp_1010(a, s); return true;
    case 1100: launch_cp_1100(a, s); return true;
    case 1110: launch_cp_1110(a, s); return true;
    case 1111: launch_cp_1111(a, s); return true;
    case 2000: launch_cp_2000(a, s); return true;
    case 2010: launch_cp_2010(a, s); return true;
    case 2011: launch_cp_2011(a, s); return true;
    case 2020: launch_cp_2020(a, s); return true;
    case 2100: launch_cp_2100(a, s); return true;
    case 2110: launch_cp_2110(a, s); return true;
    case 2111: launch_cp_2111(a, s); return true;
    case 2120: launch_cp_2120(a, s); return true;
    case 2200: launch_cp_2200(a, s); return true;
    case 2210: launch_cp_2210(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_store(int la, int lb, int lc, int ld, const StoreArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_st_0000(a, s); return true;
    case 1000: launch_st_1000(a, s); return true;
    case 1010: launch_st_1010(a, s); return true;
    case 1100: launch_st_1100(a, s); return true;
    case 1110: launch_st_1110(a, s); return true;
    case 1111: launch_st_1111(a, s); return true;
    case 2000: launch_st_2000(a, s); return true;
    case 2010: launch_st_2010(a, s); return true;
    case 2011: launch_st_2011(a, s); return true;
    case 2020: launch_st_2020(a, s); return true;
    case 2100: launch_st_2100(a, s); return true;
    case 2110: launch_st_2110(a, s); return true;
    case 2111: launch_st_2111(a, s); return true;
    case 2120: launch_st_2120(a, s); return true;
    case 2121: launch_st_2121(a, s); return true;
    case 2200: launch_st_2200(a, s); return true;
    case 2210: launch_st_2210(a, s); return true;
    case 2211: launch_st_2211(a, s); return true;
    case 2220: launch_st_2220(a, s); return true;
    case 2221: launch_st_2221(a, s); return true;
    case 2222: launch_st_2222(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_cstore(int la, int lb, int lc, int ld, const CouplingStoreArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_cst_0000(a, s); return true;
    case 1000: launch_cst_1000(a, s); return true;
    case 1010: launch_cst_1010(a, s); return true;
    case 1100: launch_cst_1100(a, s); return true;
    case 1110: launch_cst_1110(a, s); return true;
    case 1111: launch_cst_1111(a, s); return true;
    case 2000: launch_cst_2000(a, s); return true;
    case 2010: launch_cst_2010(a, s); return true;
    case 2011: launch_cst_2011(a, s); return true;
    case 2020: launch_cst_2020(a, s); return true;
    case 2100: launch_cst_2100(a, s); return true;
    case 2110: launch_cst_2110(a, s); return true;
    case 2111: launch_cst_2111(a, s); return true;
    case 2120: launch_cst_2120(a, s); return true;
    case 2121: launch_cst_2121(a, s); return true;
    case 2200: launch_cst_2200(a, s); return true;
    case 2210: launch_cst_2210(a, s); return true;
    case 2211: launch_cst_2211(a, s); return true;
    case 2220: launch_cst_2220(a, s); return true;
    case 2221: launch_cst_2221(a, s); return true;
    case 2222: launch_cst_2222(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_g12(int la, int lb, int lc, int ld, const G12Args& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_gjk_0000(a, s); return true;
    case 1000: launch_gjk_1000(a, s); return true;
    case 1010: launch_gjk_1010(a, s); return true;
    case 1100: launch_gjk_1100(a, s); return true;
    case 1110: launch_gjk_1110(a, s); return true;
    case 1111: launch_gjk_1111(a, s); return true;
    case 2000: launch_gjk_2000(a, s); return true;
    case 2010: launch_gjk_2010(a, s); return true;
    case 2011: launch_gjk_2011(a, s); return true;
    case 2020: launch_gjk_2020(a, s); return true;
    case 2100: launch_gjk_2100(a, s); return true;
    case 2110: launch_gjk_2110(a, s); return true;
    case 2111: launch_gjk_2111(a, s); return true;
    case 2120: launch_gjk_2120(a, s); return true;
    case 2121: launch_gjk_2121(a, s); return true;
    case 2200: launch_gjk_2200(a, s); return true;
    case 2210: launch_gjk_2210(a, s); return true;
    case 2211: launch_gjk_2211(a, s); return true;
    case 2220: launch_gjk_2220(a, s); return true;
    case 2221: launch_gjk_2221(a, s); return true;
    case 2222: launch_gjk_2222(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_g12cp(int la, int lb, int lc, int ld, const G12CouplingArgs& a, hipStream_t s) {
  switch (la * 1000 + lb * 100 + lc * 10 + ld) {
    case 0: launch_gcp_0000(a, s); return true;
    case 1000: launch_gcp_1000(a, s); return true;
    case 1010: launch_gcp_1010(a, s); return true;
    case 1100: launch_gcp_1100(a, s); return true;
    case 1110: launch_gcp_1110(a, s); return true;
    case 1111: launch_gcp_1111(a, s); return true;
    case 2000: launch_gcp_2000(a, s); return true;
    case 2010: launch_gcp_2010(a, s); return true;
    case 2011: launch_gcp_2011(a, s); return true;
    case 2020: launch_gcp_2020(a, s); return true;
    case 2100: launch_gcp_2100(a, s); return true;
    case 2110: launch_gcp_2110(a, s); return true;
    case 2111: launch_gcp_2111(a, s); return true;
    case 2120: launch_gcp_2120(a, s); return true;
    case 2121: launch_gcp_2121(a, s); return true;
    case 2200: launch_gcp_2200(a, s); return true;
    case 2210: launch_gcp_2210(a, s); return true;
    case 2211: launch_gcp_2211(a, s); return true;
    case 2220: launch_gcp_2220(a, s); return true;
    case 2221: launch_gcp_2221(a, s); return true;
    case 2222: launch_gcp_2222(a, s); return true;
    default: return false;
  }
}
inline bool dispatch_schwarz(int la, int lb, PairInfo* p, int np, int ls, const double* prim, const double* boys, const double* norma, hipStream_t s) {
  switch (la * 10 + lb) {
    case 0: launch_schwarz_00(p, np, ls, prim, boys, norma, s); return true;
    case 10: launch_schwarz_10(p, np, ls, prim, boys, norma, s); return true;
    case 11: launch_schwarz_11(p, np, ls, prim, boys, norma, s); return true;
    case 20: launch_schwarz_20(p, np, ls, prim, boys, norma, s); return true;
    case 21: launch_schwarz_21(p, np, ls, prim, boys, norma, s); return true;
    case 22: launch_schwarz_22(p, np, ls, prim, boys, norma, s); return true;
    default: return false;
  }
}
}  // namespace lowdin
