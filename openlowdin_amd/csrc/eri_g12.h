// Templates of the Gaussian-geminal (G12) kernels: the intra-species Fock
// build and the inter-species coupling with the operator
// sum_k c_k exp(-g_k r12^2) in place of 1/r12.
//
// Reference behaviour reproduced (openLOWDIN src/ints/Libint2Iface.cpp):
//   compute_g12_direct (2193-2365): the Fock build's quartet loops over the
//     pair list without a density screen (2263-2281), degeneracy
//     (2291-2294), the six J/K updates with the 0.5*factor exchange weight
//     (2324-2329), G = 0.25 (G + G^T) (2363);
//   compute_g12inter_direct (2367-2550): every pair s1 <= s2 of both
//     species, |raw| < 1e-10 dropped, the coupling build's element sets and
//     off-diagonal doubling (2495-2519).
// Primitive integrals: one-dimensional Gaussian moments (gen_eri.py,
// G12Gen) per geminal term, then the same HGP HRR as the Coulomb kernels.
#pragma once
#include "eri_coop.h"

namespace lowdin {

template <int LA, int LB, int LC, int LD>
struct G12Class;
#define LOWDIN_G12_CLASS(a, b, c, d)                                                                 \
  template <>                                                                                        \
  struct G12Class<a, b, c, d> {                                                                      \
    template <typename R>                                                                            \
    __device__ static __forceinline__ void vrr(R XAx, R XAy, R XAz, R XCx, R XCy, R XCz, R s11,      \
                                               R s12, R s22, R pref, R* acc) {                       \
      g12vrr_##a##b##c##d<R>(XAx, XAy, XAz, XCx, XCy, XCz, s11, s12, s22, pref, acc);                \
    }                                                                                                \
  };

// Contracted raw G12 quartet (canonical orientation) for one lane.  Per
// primitive quartet and geminal term g (weight c), with D = pq + g(p+q):
//   [00|00] = c K_ab K_cd (pq sqrt(pi) / 2) D^(-3/2) exp(-pq g |PQ|^2 / D)
// (the pair records' K carry sqrt(2) pi^(5/4) / p), then the moment
// recursion of G12Gen into [e0|f0] and one HRR.
//
// 2^ls neighbouring lanes share the quartet: first the primitive quartets go
// round them, then, where there are fewer of those than lanes, the geminal
// terms; the partial [e0|f0] are summed before the HRR.  A contracted (ss|ss)
// of 6-31G** is 1296 primitive quartets of (with 26 terms) 33696
// exponentials, one after another 7.6 ms of a 15 ms build of (H2O)2 (90 us
// shared).
template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void g12_quartet(gcptr<double> bprim, int nbp, gcptr<double> kprim, int nkp,
                                            const double* gem, int nterm, int sub, int ls, double ABx, double ABy,
                                            double ABz, double CDx, double CDy, double CDz, double* out) {
  using C = EriClass<LA, LB, LC, LD>;
  using G = G12Class<LA, LB, LC, LD>;
  double acc[C::nacc];
#pragma unroll
  for (int k = 0; k < C::nacc; ++k) acc[k] = 0.0;
  const double half_sqrt_pi = 0.88622692545275801365;
  const int nq = nbp * nkp;
  int lp = 0;   // 2^lp lanes over the primitive quartets, the rest over the terms
  while (lp < ls && (1 << lp) < nq) ++lp;
  const int i0 = sub & ((1 << lp) - 1), k0 = sub >> lp, kstep = 1 << (ls - lp);
  for (int i = i0; i < nq; i += 1 << lp) {
    const int kp = i / nbp, ip = i - kp * nbp;
    const gcptr<double> kq = kprim + kp * kPrimPairStride;
    const gcptr<double> bp = bprim + ip * kPrimPairStride;
    const double q = kq[0];
    const double Qx = kq[2], Qy = kq[3], Qz = kq[4];
    const double QCx = kq[5], QCy = kq[6], QCz = kq[7];
    const double p = bp[0];
    const double PQx = bp[2] - Qx, PQy = bp[3] - Qy, PQz = bp[4] - Qz;
    const double R2 = PQx * PQx + PQy * PQy + PQz * PQz;
    const double pq = p * q, spq = p + q;
    const double base = bp[8] * kq[8] * pq * half_sqrt_pi;
    const double PAx = bp[5], PAy = bp[6], PAz = bp[7];
    for (int k = k0; k < nterm; k += kstep) {
      const double c = gem[2 * k], g = gem[2 * k + 1];
      const double r = rsqrt_nr(pq + g * spq);   // D^(-1/2)
      const double iD = r * r;
      const double pref = c * base * iD * r * exp(-pq * g * R2 * iD);
      const double gqD = g * q * iD, gpD = g * p * iD;
      G::template vrr<double>(PAx - gqD * PQx, PAy - gqD * PQy, PAz - gqD * PQz, QCx + gpD * PQx, QCy + gpD * PQy,
                              QCz + gpD * PQz, 0.5 * (q + g) * iD, 0.5 * g * iD, 0.5 * (p + g) * iD, pref, acc);
    }
  }
  if (ls > 0) group_sum<C::nacc>(acc, 1 << ls);
  C::template hrr<double>(acc, ABx, ABy, ABz, CDx, CDy, CDz, out);
}

// The geminal's (weight, exponent) pairs in LDS: the lanes of a group read
// different terms.
__device__ __forceinline__ void stage_geminal(const G12Params& gem, double* lds) {
  for (int k = threadIdx.x; k < gem.n; k += blockDim.x) {
    lds[2 * k] = gem.c[k];
    lds[2 * k + 1] = gem.g[k];
  }
  __syncthreads();
}

// A wavefront: one bra pair and up to 64 kets, 2^ls lanes each; the J/K
// updates of the Coulomb wavefront kernel: the bra pair's J block reduced
// across the wavefront, the other five blocks as FP64 atomics.
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void g12_jk_kernel(G12Args a) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  __shared__ double gem[2 * kMaxGeminal];
  stage_geminal(a.gem, gem);
  const int wid = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (wid >= a.ntasks) return;
  const Task t = a.tasks[wid];
  const int lane = threadIdx.x & 63;
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const int ls = split_units((long)P.nprim * a.ket[t.j0].nprim * a.gem.n, a.lmax);
  const int j = t.j0 + (lane >> ls), sub = lane & ((1 << ls) - 1);
  const bool active = j < t.j1;
  const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + (active ? j : t.j0));
  const gcptr<double> nrm = (gcptr<double>)a.norma;
  const gptr<double> G = (gptr<double>)a.Graw;
  double jab[NA * NB];
#pragma unroll
  for (int k = 0; k < NA * NB; ++k) jab[k] = 0.0;
  if (active) {
    double out[NA * NB * NC * ND];
    g12_quartet<LA, LB, LC, LD>((gcptr<double>)a.prim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                (gcptr<double>)a.prim + (size_t)K.poff * kPrimPairStride, K.nprim, gem, a.gem.n, sub,
                                ls, P.ABx, P.ABy, P.ABz, K.ABx, K.ABy, K.ABz, out);
    const double deg = (P.sa != P.sb ? 2.0 : 1.0) * (K.sa != K.sb ? 2.0 : 1.0) *
                       ((a.same_class && j == t.bra) ? 1.0 : 2.0);
    if (sub == 0) {   // the first lane of a group applies the quartet's updates
      jk_quartet_update<LA, LB, LC, LD>(out, P, K, a.n, (gcptr<double>)a.D, nrm, G, deg, a.half_factor, jab);
#pragma unroll
      for (int k = 0; k < NA * NB; ++k) jab[k] *= deg;
    }
  }
  const uint64_t amask = __ballot(active);
#pragma unroll
  for (int ia = 0; ia < NA; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib) {
      const double s = wave_sum(jab[ia * NB + ib]);
      if (lane == 0 && amask)
        global_add(G + (size_t)(P.bfa + ia) * a.n + P.bfb + ib, s * nrm[P.bfa + ia] * nrm[P.bfb + ib]);
    }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void g12_coupling_kernel(G12CouplingArgs ga) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  const CouplingArgs& a = ga.cp;
  __shared__ double gem[2 * kMaxGeminal];
  stage_geminal(ga.gem, gem);
  const int wid = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (wid >= a.ntasks) return;
  const Task t = a.tasks[wid];
  const int lane = threadIdx.x & 63;
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const int ls = split_units((long)P.nprim * a.ket[t.j0].nprim * ga.gem.n, ga.lmax);
  const int j = t.j0 + (lane >> ls), sub = lane & ((1 << ls) - 1);
  if (j >= t.j1) return;
  const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
  double out[NA * NB * NC * ND];
  g12_quartet<LA, LB, LC, LD>((gcptr<double>)a.bprim + (size_t)P.poff * kPrimPairStride, P.nprim,
                              (gcptr<double>)a.kprim + (size_t)K.poff * kPrimPairStride, K.nprim, gem, ga.gem.n, sub,
                              ls, P.ABx, P.ABy, P.ABz, K.ABx, K.ABy, K.ABz, out);
  if (sub != 0) return;
  coupling_scatter<LA, LB, LC, LD>(a, P, K, out);
}

// ------------------------------------------- wave-cooperative quartets
// From total L = kCoopL up one wavefront evaluates one quartet: a lane's
// [e0|f0] accumulators (256 to 961) would live in scratch.  The terms of the
// quartet (primitive quartet x geminal term) go in batches of 21: lane 3u + d
// runs axis d's moment recursion of term u into a table in LDS, then every
// lane adds the products of its own [e0|f0] elements over the batch's terms,
// at most 16 accumulators in registers; the HRR and the contractions are
// those of the Coulomb kernels.  (H2O)2 6-31G**, 26 terms, us by lanes that
// share quartets (one lane each) / by wavefronts: (dd|dd) 1337 (2958) / 52,
// (dd|dp) 700 (2732) / 29, (dd|pp) 331 (2403) / 44, (dp|dp) 328 (1875) / 42.
constexpr int kG12Batch = 21;

template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int g12_coop_doubles() {
  return coop_wave_doubles<LA, LB, LC, LD>() + 3 * kG12Batch * (LA + LB + 1) * (LC + LD + 1);
}

// Exponents of component k of the shells l = l0, l0 + 1, ... listed one after
// another (xx, xy, xz, yy, yz, zz order).
__device__ __forceinline__ void cart_exponents(int l0, int k, int* e) {
  int l = l0;
  while (k >= ncart(l)) k -= ncart(l++);
  int r = 0;   // l - lx
  while (k > r) k -= ++r;
  e[0] = l - r;
  e[1] = r - k;
  e[2] = k;
}

template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void g12_coop_quartet(double* R, const uint2* pg, gcptr<double> bprim, int nbp,
                                                 gcptr<double> kprim, int nkp, const double* gem, int nterm,
                                                 const PairInfo& P, const PairInfo& K, int lane) {
  constexpr int NE = LA + LB + 1, NF = LC + LD + 1, S = NE * NF;
  constexpr int NACC = EriClass<LA, LB, LC, LD>::nacc, NT = (NACC + 63) / 64;
  constexpr int nf = []() constexpr {
    int n = 0;
    for (int l = LC; l <= LC + LD; ++l) n += ncart(l);
    return n;
  }();
  double* tab = R + coop_wave_doubles<LA, LB, LC, LD>();
  // table offsets of this lane's elements: axis x | y << 8 | z << 16
  unsigned at[NT];
  double acc[NT];
#pragma unroll
  for (int r = 0; r < NT; ++r) {
    const int el = lane + 64 * r < NACC ? lane + 64 * r : 0;
    int e[3], f[3];
    cart_exponents(LA, el / nf, e);
    cart_exponents(LC, el % nf, f);
    at[r] = (unsigned)(e[0] * NF + f[0]) | (unsigned)(e[1] * NF + f[1]) << 8 | (unsigned)(e[2] * NF + f[2]) << 16;
    acc[r] = 0.0;
  }
  const double half_sqrt_pi = 0.88622692545275801365;
  const int units = nbp * nkp * nterm;
  for (int u0 = 0; u0 < units; u0 += kG12Batch) {
    const int nu = min(kG12Batch, units - u0);
    const int u = lane / 3, d = lane - 3 * u;
    if (u < nu) {
      const int i = (u0 + u) / nterm, k = u0 + u - i * nterm;
      const int kp = i / nbp, ip = i - kp * nbp;
      const gcptr<double> kq = kprim + kp * kPrimPairStride;
      const gcptr<double> bp = bprim + ip * kPrimPairStride;
      const double q = kq[0], p = bp[0];
      const double PQx = bp[2] - kq[2], PQy = bp[3] - kq[3], PQz = bp[4] - kq[4];
      const double PQ = d == 0 ? PQx : (d == 1 ? PQy : PQz);
      const double c = gem[2 * k], g = gem[2 * k + 1];
      const double pq = p * q;
      const double rt = rsqrt_nr(pq + g * (p + q));   // D^(-1/2)
      const double iD = rt * rt;
      const double XA = bp[5 + d] - g * q * iD * PQ, XC = kq[5 + d] + g * p * iD * PQ;
      const double s11 = 0.5 * (q + g) * iD, s12 = 0.5 * g * iD, s22 = 0.5 * (p + g) * iD;
      double v = 1.0;
      if (d == 0)
        v = c * (bp[8] * kq[8] * pq * half_sqrt_pi) * iD * rt * exp(-pq * g * (PQx * PQx + PQy * PQy + PQz * PQz) * iD);
      double I[NE][NF];
      I[0][0] = v;
#pragma unroll
      for (int x = 1; x < NE; ++x)
        I[x][0] = XA * I[x - 1][0] + (x > 1 ? (double)(x - 1) * s11 * I[x > 1 ? x - 2 : 0][0] : 0.0);
#pragma unroll
      for (int y = 1; y < NF; ++y)
#pragma unroll
        for (int x = 0; x < NE; ++x)
          I[x][y] = XC * I[x][y - 1] + (x > 0 ? (double)x * s12 * I[x > 0 ? x - 1 : 0][y - 1] : 0.0) +
                    (y > 1 ? (double)(y - 1) * s22 * I[x][y > 1 ? y - 2 : 0] : 0.0);
      double* o = tab + (size_t)lane * S;
#pragma unroll
      for (int x = 0; x < NE; ++x)
#pragma unroll
        for (int y = 0; y < NF; ++y) o[x * NF + y] = I[x][y];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int w = 0; w < nu; ++w) {
      const double* o = tab + (size_t)(3 * w) * S;
#pragma unroll
      for (int r = 0; r < NT; ++r)
        acc[r] += o[at[r] & 255u] * o[S + ((at[r] >> 8) & 255u)] * o[2 * S + (at[r] >> 16)];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int r = 0; r < NT; ++r)
    if (lane + 64 * r < NACC) R[kCoopAcc + lane + 64 * r] = acc[r];
  coop_hrr<LA, LB, LC, LD>(R, pg, P, K, lane);
}

// One wavefront per workgroup: a bra pair and its task's kets in turn.
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(64) void g12_jk_coop_kernel(G12Args a) {
  using Pg = CoopProgram<LA, LB, LC, LD>;
  constexpr int NA = ncart(LA), NB = ncart(LB), NAB = NA * NB;
  extern __shared__ double R[];
  __shared__ double gem[2 * kMaxGeminal];
  stage_geminal(a.gem, gem);
  const int lane = threadIdx.x;
  const Task t = a.tasks[blockIdx.x];
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const gcptr<double> nrm = (gcptr<double>)a.norma;
  const gptr<double> G = (gptr<double>)a.Graw;
  const gcptr<double> D = (gcptr<double>)a.D;
  if (lane < 2) R[kCoopZero + lane] = 0.0;
  if (lane < NAB) {
    const int fa = P.bfa + lane / NB, fb = P.bfb + lane % NB;
    R[Pg::kRegion + lane] = D[(size_t)fa * a.n + fb] * nrm[fa] * nrm[fb];
  }
  const CoopJk u{a.n, D, nrm, G, nullptr, nullptr, 0, a.half_factor, nullptr, nullptr, 0};
  double jab = 0.0;
  for (int j = t.j0; j < t.j1; ++j) {
    const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
    g12_coop_quartet<LA, LB, LC, LD>(R, Pg::prog() + lane, (gcptr<double>)a.prim + (size_t)P.poff * kPrimPairStride,
                                     P.nprim, (gcptr<double>)a.prim + (size_t)K.poff * kPrimPairStride, K.nprim, gem,
                                     a.gem.n, P, K, lane);
    const double deg = (P.sa != P.sb ? 2.0 : 1.0) * (K.sa != K.sb ? 2.0 : 1.0) *
                       ((a.same_class && j == t.bra) ? 1.0 : 2.0);
    coop_jk_update<false, LA, LB, LC, LD>(R, u, P, K, j, deg, lane, jab);
  }
  if (lane < NAB) {
    const int fa = P.bfa + lane / NB, fb = P.bfb + lane % NB;
    global_add(G + (size_t)fa * a.n + fb, jab * nrm[fa] * nrm[fb]);
  }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(64) void g12_coupling_coop_kernel(G12CouplingArgs ga) {
  const CouplingArgs& a = ga.cp;
  extern __shared__ double R[];
  __shared__ double gem[2 * kMaxGeminal];
  stage_geminal(ga.gem, gem);
  const int lane = threadIdx.x;
  const Task t = a.tasks[blockIdx.x];
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  if (lane < 2) R[kCoopZero + lane] = 0.0;
  coop_coupling_weights<LA, LB, LC, LD>(R, a, P, lane);
  for (int j = t.j0; j < t.j1; ++j) {
    const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
    g12_coop_quartet<LA, LB, LC, LD>(R, CoopProgram<LA, LB, LC, LD>::prog() + lane,
                                     (gcptr<double>)a.bprim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                     (gcptr<double>)a.kprim + (size_t)K.poff * kPrimPairStride, K.nprim, gem, ga.gem.n,
                                     P, K, lane);
    coop_coupling_update<LA, LB, LC, LD>(R, a, P, K, lane);
  }
}

template <int LA, int LB, int LC, int LD>
static void launch_g12_t(const G12Args& a, hipStream_t s) {
  if (a.ntasks <= 0) return;
  if constexpr (LA + LB + LC + LD >= kCoopL) {
    constexpr size_t lds = sizeof(double) * g12_coop_doubles<LA, LB, LC, LD>();
    hipLaunchKernelGGL((g12_jk_coop_kernel<LA, LB, LC, LD>), dim3((unsigned)a.ntasks), dim3(64), lds, s, a);
  } else {
    hipLaunchKernelGGL((g12_jk_kernel<LA, LB, LC, LD>), dim3((unsigned)((a.ntasks + 3) / 4)), dim3(256), 0, s, a);
  }
}

template <int LA, int LB, int LC, int LD>
static void launch_g12cp_t(const G12CouplingArgs& a, hipStream_t s) {
  if (a.cp.ntasks <= 0) return;
  if constexpr (LA + LB + LC + LD >= kCoopL) {
    constexpr size_t lds = sizeof(double) * g12_coop_doubles<LA, LB, LC, LD>();
    hipLaunchKernelGGL((g12_coupling_coop_kernel<LA, LB, LC, LD>), dim3((unsigned)a.cp.ntasks), dim3(64), lds, s, a);
  } else {
    hipLaunchKernelGGL((g12_coupling_kernel<LA, LB, LC, LD>), dim3((unsigned)((a.cp.ntasks + 3) / 4)), dim3(256), 0,
                       s, a);
  }
}

}  // namespace lowdin
