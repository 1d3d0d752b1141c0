// Templates of the integral-store and first-quarter-transform kernels: the
// MEMORY and integral-transformation variants of the two-particle path.
// They share the generated quartet evaluation (Obara-Saika VRR + HGP HRR)
// and the work decomposition of the Fock-build kernels: a wavefront owns one
// bra shell pair and up to 64 ket shell pairs, 2^ls lanes each; from total
// L = kCoopL up a wavefront evaluates one quartet (eri_coop.h).
//
// Reference behaviour reproduced (openLOWDIN src/ints/Libint2Iface.cpp):
//   compute_2body_directAll (2552-2742): the Fock build's quartet set and
//     screen (2629-2669), integrals with |raw| > 1e-10 normalised by norma
//     and written to all eight index images (2698-2717);
//   compute_2body_directIT (620-921): GG[j][k][l] += C(p,i) (ij|kl) over
//     the distinct index permutations, accumulated into k <= l (803-851),
//     then the k > l triangle mirrored (864-874);
//   compute_coupling_directAll (2744-2908): every pair s1 <= s2 of both
//     species, no screen, elements bf1 <= bf2 / obf1 <= obf2 with
//     |raw| >= 1e-10 and their four images (2864-2880);
//   compute_coupling_directIT (1296-1622): the same quartets transformed
//     on the index of the calling species (1455-1545), mirrored (1562-1572).
#pragma once
#include <algorithm>

#include "eri_coop.h"

namespace lowdin {

// Elements of one block have the same eight index images where the shells of
// a pair are the same, or bra and ket are the same pair: (a b) and (b a), (c d)
// and (d c), (ab|cd) and (cd|ab).  Their recursions round differently, and
// lanes that share a block store it side by side, so only the last kept one of
// them is stored: all images of an integral hold the same bits, whatever the
// timing.  True where a later element than (ia ib|ic id) is stored for it.
template <int NA, int NB, int NC, int ND>
__device__ __forceinline__ bool stored_later(const double* w, int ia, int ib, int ic, int id, bool bdiag, bool kdiag,
                                             bool same, double drop) {
  const int e = ((ia * NB + ib) * NC + ic) * ND + id;
  bool later = false;
#pragma unroll
  for (int t = 1; t < 8; ++t) {
    const bool k = t & 1, b = t & 2, s = t & 4;   // swap c and d, a and b, bra and ket
    if ((k && NC != ND) || (b && NA != NB) || (s && (NA != NC || NB != ND))) continue;
    const int x = b ? ib : ia, y = b ? ia : ib, z = k ? id : ic, u = k ? ic : id;
    const int f = s ? ((z * NB + u) * NC + x) * ND + y : ((x * NB + y) * NC + z) * ND + u;
    if (f > e) later = later || ((!k || kdiag) && (!b || bdiag) && (!s || same) && fabs(w[f]) > drop);
  }
  return later;
}

// The eight index images of one kept integral of an intra-species quartet.
__device__ __forceinline__ void store_images(double* A, size_t n, size_t i, size_t j, size_t k, size_t l, double v) {
  const size_t n2 = n * n, n3 = n2 * n;
  A[i * n3 + j * n2 + k * n + l] = v;
  A[j * n3 + i * n2 + k * n + l] = v;
  A[i * n3 + j * n2 + l * n + k] = v;
  A[j * n3 + i * n2 + l * n + k] = v;
  A[k * n3 + l * n2 + i * n + j] = v;
  A[k * n3 + l * n2 + j * n + i] = v;
  A[l * n3 + k * n2 + i * n + j] = v;
  A[l * n3 + k * n2 + j * n + i] = v;
}

// ------------------------------------------------------ intra-species store
// The lanes that share a quartet also share the stores of its block.
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void store_kernel(StoreArgs a) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  const int wid = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (wid >= a.ntasks) return;
  const Task t = a.tasks[wid];
  const int lane = threadIdx.x & 63;
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const int ls = split_shift(P.nprim, a.ket[t.j0].nprim, a.lmax);
  const int j = t.j0 + (lane >> ls), sub = lane & ((1 << ls) - 1);
  if (j >= t.j1) return;
  const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
  if (a.screen && quartet_dnorm((gcptr<double>)a.Dn, a.nshell, P, K) * P.Q * K.Q < a.eps) return;
  double out[NA * NB * NC * ND];
  contracted_quartet<LA, LB, LC, LD>((gcptr<double>)a.prim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                     (gcptr<double>)a.prim + (size_t)K.poff * kPrimPairStride, K.nprim, a.boys,
                                     P.ABx, P.ABy, P.ABz, K.ABx, K.ABy, K.ABz, out, sub, 1 << ls);
  const gcptr<double> nrm = (gcptr<double>)a.norma;
  double na[NA], nb[NB], nc[NC], nd[ND];
#pragma unroll
  for (int i = 0; i < NA; ++i) na[i] = nrm[P.bfa + i];
#pragma unroll
  for (int i = 0; i < NB; ++i) nb[i] = nrm[P.bfb + i];
#pragma unroll
  for (int i = 0; i < NC; ++i) nc[i] = nrm[K.bfa + i];
#pragma unroll
  for (int i = 0; i < ND; ++i) nd[i] = nrm[K.bfb + i];
  // only (c d) and (d c) can coincide: one comparison for half of the elements,
  // by itself (in stored_later's form the spilling (dp|pp) takes 250-270 us of a
  // (H2O)3 store instead of 205)
  constexpr bool kKetOnly = NA != NB && NC == ND;
  const bool bdiag = P.sa == P.sb, kdiag = K.sa == K.sb, same = a.same_class && j == t.bra;
  int turn = 0;
#pragma unroll
  for (int ia = 0; ia < NA; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib)
#pragma unroll
      for (int ic = 0; ic < NC; ++ic)
#pragma unroll
        for (int id = 0; id < ND; ++id) {
          const double v = out[((ia * NB + ib) * NC + ic) * ND + id];
          bool mine = (turn++ & ((1 << ls) - 1)) == sub;
          if constexpr (kKetOnly) {
            if (ic < id) mine = mine && !(kdiag && fabs(out[((ia * NB + ib) * NC + id) * ND + ic]) > a.drop);
          } else {
            mine = mine && !stored_later<NA, NB, NC, ND>(out, ia, ib, ic, id, bdiag, kdiag, same, a.drop);
          }
          if (mine && fabs(v) > a.drop)
            store_images(a.out, a.n, P.bfa + ia, P.bfb + ib, K.bfa + ic, K.bfb + id,
                         v * na[ia] * nb[ib] * nc[ic] * nd[id]);
        }
}

// ---------------------------------------------------- first-quarter transform
// GG[x][k][l] += sum_i c[i] (i x|k l).  While it accumulates, slab x of the
// result holds its (k, l) values packed by shell pair in its first part:
// element e of pair q of a class at jpoff[class] + e * (pairs of the class) +
// q (unpack_slabs then spreads them over both triangles).  A workgroup owns
// one bra pair (a b) and a run of kets, so
//   (ab|cd), (ba|cd): slabs b and a, pair (c d): neighbouring lanes add to
//     neighbouring doubles;
//   (cd|ab), (dc|ab): slabs d and c, pair (a b): summed over the kets in LDS,
//     NA NB rows of n, and flushed once per workgroup.  Where the rows do not
//     all fit (n above 568 for (dd|), 1136 for (dp|)) the launch is repeated
//     for the next ones; the first pass does the slabs of a and b.
// Scattered over GG, one lane per quartet, these atomics bounded the
// transform: C8H18 cc-pVDZ (n = 210) 11.2 ms; packed 3.3 ms (9.6 ms of kernels
// over four streams, (ds|pp), (ps|ss), (dd|ps) and (pp|pp) longest).
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void it_strip_kernel(StoreArgs a) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  extern __shared__ double strip[];   // rows row0 .. row0 + rows - 1 of n
  const int tid = threadIdx.x, n = a.n;
  const Task t = a.tasks[blockIdx.x];
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const gcptr<double> prim = (gcptr<double>)a.prim;
  const gcptr<double> nrm = (gcptr<double>)a.norma;
  const gcptr<double> c = (gcptr<double>)a.c;
  const gptr<double> GG = (gptr<double>)a.out;
  const size_t n2 = (size_t)n * n;
  for (int k = tid; k < a.rows * n; k += blockDim.x) strip[k] = 0.0;
  __syncthreads();
  double na[NA], nb[NB], ca[NA], cb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    na[i] = nrm[P.bfa + i];
    ca[i] = c[P.bfa + i];
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    nb[i] = nrm[P.bfb + i];
    cb[i] = c[P.bfb + i];
  }
  const bool sab = P.sa != P.sb;
  int nround = 0;
  for (int jr = t.j0; jr < t.j1; jr += nround) {
    const int ls = split_shift(P.nprim, a.ket[jr].nprim, a.lmax);
    nround = (int)blockDim.x >> ls;
    const int j = jr + (tid >> ls), sub = tid & ((1 << ls) - 1);
    if (j >= t.j1) continue;
    const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
    if (a.screen && quartet_dnorm((gcptr<double>)a.Dn, a.nshell, P, K) * P.Q * K.Q < a.eps) continue;
    double out[NA * NB * NC * ND];
    contracted_quartet<LA, LB, LC, LD>(prim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                       prim + (size_t)K.poff * kPrimPairStride, K.nprim, a.boys, P.ABx, P.ABy, P.ABz, K.ABx, K.ABy, K.ABz, out, sub, 1 << ls);
    if (sub != 0) continue;
    double nc[NC], nd[ND], cc[NC], cd[ND];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      nc[i] = nrm[K.bfa + i];
      cc[i] = c[K.bfa + i];
    }
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      nd[i] = nrm[K.bfb + i];
      cd[i] = c[K.bfb + i];
    }
    // drop (|raw| > drop kept) and normalise
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
      for (int ib = 0; ib < NB; ++ib)
#pragma unroll
        for (int ic = 0; ic < NC; ++ic)
#pragma unroll
          for (int id = 0; id < ND; ++id) {
            double& v = out[((ia * NB + ib) * NC + ic) * ND + id];
            v = fabs(v) > a.drop ? v * na[ia] * nb[ib] * nc[ic] * nd[id] : 0.0;
          }
    const bool scd = K.sa != K.sb;
    const bool spk = !(a.same_class && j == t.bra);
    // (ab|cd) and (ba|cd); within a pair of one shell the block holds both
    // orders and its k <= l elements feed the slot
#pragma unroll
    for (int ic = 0; ic < NC; ++ic)
#pragma unroll
      for (int id = 0; id < ND; ++id) {
        if (a.row0 != 0 || (!scd && ic > id)) continue;
        const size_t slot = (size_t)a.kpk + (size_t)(ic * ND + id) * a.nket + j;
#pragma unroll
        for (int ib = 0; ib < NB; ++ib) {
          double s = 0.0;
#pragma unroll
          for (int ia = 0; ia < NA; ++ia) s += ca[ia] * out[((ia * NB + ib) * NC + ic) * ND + id];
          if (s != 0.0) global_add(GG + (size_t)(P.bfb + ib) * n2 + slot, s);
        }
        if (sab) {
#pragma unroll
          for (int ia = 0; ia < NA; ++ia) {
            double s = 0.0;
#pragma unroll
            for (int ib = 0; ib < NB; ++ib) s += cb[ib] * out[((ia * NB + ib) * NC + ic) * ND + id];
            if (s != 0.0) global_add(GG + (size_t)(P.bfa + ia) * n2 + slot, s);
          }
        }
      }
    if (!spk) continue;
    // (cd|ab) and (dc|ab)
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
      for (int ib = 0; ib < NB; ++ib) {
        const int r = ia * NB + ib - a.row0;
        if ((!sab && ia > ib) || r < 0 || r >= a.rows) continue;
        double* row = strip + r * n;
#pragma unroll
        for (int id = 0; id < ND; ++id) {
          double s = 0.0;
#pragma unroll
          for (int ic = 0; ic < NC; ++ic) s += cc[ic] * out[((ia * NB + ib) * NC + ic) * ND + id];
          if (s != 0.0) atomicAdd(&row[K.bfb + id], s);
        }
        if (scd) {
#pragma unroll
          for (int ic = 0; ic < NC; ++ic) {
            double s = 0.0;
#pragma unroll
            for (int id = 0; id < ND; ++id) s += cd[id] * out[((ia * NB + ib) * NC + ic) * ND + id];
            if (s != 0.0) atomicAdd(&row[K.bfa + ic], s);
          }
        }
      }
  }
  __syncthreads();
  for (int e = 0; e < a.rows; ++e)
    for (int x = tid; x < n; x += blockDim.x) {
      const double v = strip[e * n + x];
      if (v != 0.0) global_add(GG + (size_t)x * n2 + a.bpk + (size_t)(a.row0 + e) * a.nbra + t.bra, v);
    }
}

// ------------------------------------- one wavefront per quartet (high L)
// One lane per quartet kept these classes' blocks in scratch: (H2O)3 6-31G**
// (dd|dd) 1060 -> 33 us, (dd|dp) 901 -> 31, the store 4.0 -> 0.55 ms.  Store
// (MODE 0) or transform (MODE 1, packed slabs as above, every update a global
// atomic: these classes have few quartets): the lanes share the elements of the
// (ab|cd) block in LDS.
template <int LA, int LB, int LC, int LD, int MODE>
__global__ __launch_bounds__(64) void store_coop_kernel(StoreArgs a) {
  using Pg = CoopProgram<LA, LB, LC, LD>;
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  extern __shared__ double R[];
  const int lane = threadIdx.x;
  const Task t = a.tasks[blockIdx.x];
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const gcptr<double> prim = (gcptr<double>)a.prim;
  const gcptr<double> nrm = (gcptr<double>)a.norma;
  const gcptr<double> c = (gcptr<double>)a.c;
  const gptr<double> GG = (gptr<double>)a.out;
  const size_t n2 = (size_t)a.n * a.n;
  if (lane < 2) R[kCoopZero + lane] = 0.0;
  for (int j = t.j0; j < t.j1; ++j) {
    const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
    if (a.screen && quartet_dnorm((gcptr<double>)a.Dn, a.nshell, P, K) * P.Q * K.Q < a.eps) continue;
    coop_quartet<LA, LB, LC, LD>(R, Pg::prog() + lane, prim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                 prim + (size_t)K.poff * kPrimPairStride, K.nprim, a.boys, P, K, lane);
    double* out = R + Pg::kOut;
    const bool sab = P.sa != P.sb, scd = K.sa != K.sb;
    const bool spk = !(a.same_class && j == t.bra);
    for (int e = lane; e < NA * NB * NC * ND; e += 64) {
      const int id = e % ND, ic = e / ND % NC, ib = e / (ND * NC) % NB, ia = e / (ND * NC * NB);
      const double v = out[e];
      const double w = fabs(v) > a.drop ? v * nrm[P.bfa + ia] * nrm[P.bfb + ib] * nrm[K.bfa + ic] * nrm[K.bfb + id] : 0.0;
      if constexpr (MODE == 0) {
        if (w != 0.0 && !stored_later<NA, NB, NC, ND>(out, ia, ib, ic, id, !sab, !scd, !spk, a.drop))
          store_images(a.out, a.n, P.bfa + ia, P.bfb + ib, K.bfa + ic, K.bfb + id, w);
      } else {
        out[e] = w;
      }
    }
    if constexpr (MODE == 1) {
      for (int e = lane; e < NC * ND * (NA + NB); e += 64) {   // (ab|cd), (ba|cd)
        const int x = e / (NC * ND), id = e % ND, ic = e / ND % NC;
        if (!scd && ic > id) continue;
        double s = 0.0;
        if (x < NB) {
          for (int ia = 0; ia < NA; ++ia) s += c[P.bfa + ia] * out[((ia * NB + x) * NC + ic) * ND + id];
        } else if (sab) {
          for (int ib = 0; ib < NB; ++ib) s += c[P.bfb + ib] * out[(((x - NB) * NB + ib) * NC + ic) * ND + id];
        }
        if (s != 0.0)
          global_add(GG + (size_t)(x < NB ? P.bfb + x : P.bfa + x - NB) * n2 + a.kpk +
                         (size_t)(ic * ND + id) * a.nket + j,
                     s);
      }
      for (int e = lane; spk && e < NA * NB * (NC + ND); e += 64) {   // (cd|ab), (dc|ab)
        const int x = e / (NA * NB), ab = e % (NA * NB);
        if (!sab && ab / NB > ab % NB) continue;
        double s = 0.0;
        if (x < ND) {
          for (int ic = 0; ic < NC; ++ic) s += c[K.bfa + ic] * out[(ab * NC + ic) * ND + x];
        } else if (scd) {
          for (int id = 0; id < ND; ++id) s += c[K.bfb + id] * out[(ab * NC + x - ND) * ND + id];
        }
        if (s != 0.0)
          global_add(GG + (size_t)(x < ND ? K.bfb + x : K.bfa + x - ND) * n2 + a.bpk + (size_t)ab * a.nbra + t.bra, s);
      }
    }
  }
}

// ------------------------------------------------- inter-species store / IT
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void coupling_store_kernel(CouplingStoreArgs a) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  const int wid = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (wid >= a.ntasks) return;
  const Task t = a.tasks[wid];
  const int lane = threadIdx.x & 63;
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const int ls = split_shift(P.nprim, a.ket[t.j0].nprim, a.lmax);
  const int j = t.j0 + (lane >> ls), sub = lane & ((1 << ls) - 1);
  if (j >= t.j1) return;
  const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
  double out[NA * NB * NC * ND];
  contracted_quartet<LA, LB, LC, LD>((gcptr<double>)a.bprim + (size_t)P.poff * kPrimPairStride, P.nprim,
                                     (gcptr<double>)a.kprim + (size_t)K.poff * kPrimPairStride, K.nprim, a.boys,
                                     P.ABx, P.ABy, P.ABz, K.ABx, K.ABy, K.ABz, out, sub, 1 << ls);
  if (sub != 0) return;
  double na[NA], nb[NB], nc[NC], nd[ND];
#pragma unroll
  for (int i = 0; i < NA; ++i) na[i] = a.nbra_norma[P.bfa + i];
#pragma unroll
  for (int i = 0; i < NB; ++i) nb[i] = a.nbra_norma[P.bfb + i];
#pragma unroll
  for (int i = 0; i < NC; ++i) nc[i] = a.nket_norma[K.bfa + i];
#pragma unroll
  for (int i = 0; i < ND; ++i) nd[i] = a.nket_norma[K.bfb + i];
  // drop (|raw| < drop dropped) and normalise
#pragma unroll
  for (int ia = 0; ia < NA; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib)
#pragma unroll
      for (int ic = 0; ic < NC; ++ic)
#pragma unroll
        for (int id = 0; id < ND; ++id) {
          const int e = ((ia * NB + ib) * NC + ic) * ND + id;
          const double v = out[e];
          out[e] = fabs(v) < a.drop ? 0.0 : v * na[ia] * nb[ib] * nc[ic] * nd[id];
        }
  const bool bdiag = P.sa == P.sb, kdiag = K.sa == K.sb;
  if (a.mode == 0) {
    double* A = a.out;
    const size_t s1 = a.sx1, s2 = a.sx2, s3 = a.sy1;
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
      for (int ib = 0; ib < NB; ++ib)
#pragma unroll
        for (int ic = 0; ic < NC; ++ic)
#pragma unroll
          for (int id = 0; id < ND; ++id) {
            const int fa = P.bfa + ia, fb = P.bfb + ib, fc = K.bfa + ic, fd = K.bfb + id;
            if ((bdiag && fa > fb) || (kdiag && fc > fd)) continue;
            const double v = out[((ia * NB + ib) * NC + ic) * ND + id];
            if (v == 0.0) continue;
            const size_t x1 = a.bra_is_x ? fa : fc, x2 = a.bra_is_x ? fb : fd;
            const size_t y1 = a.bra_is_x ? fc : fa, y2 = a.bra_is_x ? fd : fb;
            A[x1 * s1 + x2 * s2 + y1 * s3 + y2] = v;
            A[x2 * s1 + x1 * s2 + y1 * s3 + y2] = v;
            A[x1 * s1 + x2 * s2 + y2 * s3 + y1] = v;
            A[x2 * s1 + x1 * s2 + y2 * s3 + y1] = v;
          }
    return;
  }
  const gptr<double> GG = (gptr<double>)a.out;
  const gcptr<double> c = (gcptr<double>)a.c;
  const size_t no = (size_t)a.n_o, no2 = no * no;
  if (a.bra_is_t) {
    // transformed pair (a b), other pair (c d)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib)
#pragma unroll
      for (int ic = 0; ic < NC; ++ic)
#pragma unroll
        for (int id = 0; id < ND; ++id) {
          const int fc = K.bfa + ic, fd = K.bfb + id;
          if (kdiag && fc > fd) continue;
          double s = 0.0;
#pragma unroll
          for (int ia = 0; ia < NA; ++ia) s += c[P.bfa + ia] * out[((ia * NB + ib) * NC + ic) * ND + id];
          if (s != 0.0)
            global_add(GG + (size_t)(P.bfb + ib) * no2 + (size_t)min(fc, fd) * no + max(fc, fd), s);
        }
    if (!bdiag) {
#pragma unroll
      for (int ia = 0; ia < NA; ++ia)
#pragma unroll
        for (int ic = 0; ic < NC; ++ic)
#pragma unroll
          for (int id = 0; id < ND; ++id) {
            const int fc = K.bfa + ic, fd = K.bfb + id;
            if (kdiag && fc > fd) continue;
            double s = 0.0;
#pragma unroll
            for (int ib = 0; ib < NB; ++ib) s += c[P.bfb + ib] * out[((ia * NB + ib) * NC + ic) * ND + id];
            if (s != 0.0)
              global_add(GG + (size_t)(P.bfa + ia) * no2 + (size_t)min(fc, fd) * no + max(fc, fd), s);
          }
    }
  } else {
    // transformed pair (c d), other pair (a b)
#pragma unroll
    for (int id = 0; id < ND; ++id)
#pragma unroll
      for (int ia = 0; ia < NA; ++ia)
#pragma unroll
        for (int ib = 0; ib < NB; ++ib) {
          const int fa = P.bfa + ia, fb = P.bfb + ib;
          if (bdiag && fa > fb) continue;
          double s = 0.0;
#pragma unroll
          for (int ic = 0; ic < NC; ++ic) s += c[K.bfa + ic] * out[((ia * NB + ib) * NC + ic) * ND + id];
          if (s != 0.0)
            global_add(GG + (size_t)(K.bfb + id) * no2 + (size_t)min(fa, fb) * no + max(fa, fb), s);
        }
    if (!kdiag) {
#pragma unroll
      for (int ic = 0; ic < NC; ++ic)
#pragma unroll
        for (int ia = 0; ia < NA; ++ia)
#pragma unroll
          for (int ib = 0; ib < NB; ++ib) {
            const int fa = P.bfa + ia, fb = P.bfb + ib;
            if (bdiag && fa > fb) continue;
            double s = 0.0;
#pragma unroll
            for (int id = 0; id < ND; ++id) s += c[K.bfb + id] * out[((ia * NB + ib) * NC + ic) * ND + id];
            if (s != 0.0)
              global_add(GG + (size_t)(K.bfa + ic) * no2 + (size_t)min(fa, fb) * no + max(fa, fb), s);
          }
    }
  }
}

// The same with one wavefront per quartet (high L).
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(64) void coupling_store_coop_kernel(CouplingStoreArgs a) {
  using Pg = CoopProgram<LA, LB, LC, LD>;
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  extern __shared__ double R[];
  const int lane = threadIdx.x;
  const Task t = a.tasks[blockIdx.x];
  const PairInfo P = load_pair((gcptr<PairInfo>)a.bra + t.bra);
  const gcptr<double> nb = (gcptr<double>)a.nbra_norma, nk = (gcptr<double>)a.nket_norma;
  const gcptr<double> c = (gcptr<double>)a.c;
  const gptr<double> GG = (gptr<double>)a.out;
  const size_t no = (size_t)a.n_o, no2 = no * no;
  if (lane < 2) R[kCoopZero + lane] = 0.0;
  for (int j = t.j0; j < t.j1; ++j) {
    const PairInfo K = load_pair((gcptr<PairInfo>)a.ket + j);
    coop_quartet<LA, LB, LC, LD>(R, Pg::prog() + lane, (gcptr<double>)a.bprim + (size_t)P.poff * kPrimPairStride,
                                 P.nprim, (gcptr<double>)a.kprim + (size_t)K.poff * kPrimPairStride, K.nprim, a.boys, P,
                                 K, lane);
    double* out = R + Pg::kOut;
    const bool bdiag = P.sa == P.sb, kdiag = K.sa == K.sb;
    for (int e = lane; e < NA * NB * NC * ND; e += 64) {
      const int id = e % ND, ic = e / ND % NC, ib = e / (ND * NC) % NB, ia = e / (ND * NC * NB);
      const double v = out[e];
      const double w = fabs(v) < a.drop ? 0.0 : v * nb[P.bfa + ia] * nb[P.bfb + ib] * nk[K.bfa + ic] * nk[K.bfb + id];
      out[e] = w;
      if (a.mode != 0 || w == 0.0 || (bdiag && ia > ib) || (kdiag && ic > id)) continue;
      const int fa = P.bfa + ia, fb = P.bfb + ib, fc = K.bfa + ic, fd = K.bfb + id;
      const size_t x1 = a.bra_is_x ? fa : fc, x2 = a.bra_is_x ? fb : fd;
      const size_t y1 = a.bra_is_x ? fc : fa, y2 = a.bra_is_x ? fd : fb;
      a.out[x1 * a.sx1 + x2 * a.sx2 + y1 * a.sy1 + y2] = w;
      a.out[x2 * a.sx1 + x1 * a.sx2 + y1 * a.sy1 + y2] = w;
      a.out[x1 * a.sx1 + x2 * a.sx2 + y2 * a.sy1 + y1] = w;
      a.out[x2 * a.sx1 + x1 * a.sx2 + y2 * a.sy1 + y1] = w;
    }
    if (a.mode == 0) continue;
    // transformed pair (a b) over the slots of (c d), or the other way round
    const int nx = a.bra_is_t ? NB : ND, ny = a.bra_is_t ? NA : NC, nz = a.bra_is_t ? NC * ND : NA * NB;
    const bool tdiag = a.bra_is_t ? bdiag : kdiag, odiag = a.bra_is_t ? kdiag : bdiag;
    const int nzr = a.bra_is_t ? ND : NB;   // columns of the other pair's block
    const PairInfo& T = a.bra_is_t ? P : K;
    const PairInfo& O = a.bra_is_t ? K : P;
    for (int e = lane; e < nz * (nx + ny); e += 64) {
      const int x = e / nz, z = e % nz, z1 = z / nzr, z2 = z % nzr;
      if (odiag && z1 > z2) continue;
      double s = 0.0;
      if (x < nx) {
        for (int y = 0; y < ny; ++y)
          s += c[T.bfa + y] * (a.bra_is_t ? out[(y * NB + x) * NC * ND + z] : out[z * NC * ND + y * ND + x]);
      } else if (!tdiag) {
        for (int y = 0; y < nx; ++y)
          s += c[T.bfb + y] * (a.bra_is_t ? out[((x - nx) * NB + y) * NC * ND + z] : out[z * NC * ND + (x - nx) * ND + y]);
      }
      const int f1 = O.bfa + z1, f2 = O.bfb + z2;
      if (s != 0.0)
        global_add(GG + (size_t)(x < nx ? T.bfb + x : T.bfa + x - nx) * no2 + (size_t)min(f1, f2) * no + max(f1, f2), s);
    }
  }
}

template <int LA, int LB, int LC, int LD>
static void launch_store_t(const StoreArgs& a, hipStream_t s) {
  if (a.ntasks <= 0) return;
  if constexpr (LA + LB + LC + LD >= kCoopL) {
    constexpr size_t lds = sizeof(double) * coop_wave_doubles<LA, LB, LC, LD>();
    if (a.mode == 0)
      hipLaunchKernelGGL((store_coop_kernel<LA, LB, LC, LD, 0>), dim3((unsigned)a.ntasks), dim3(64), lds, s, a);
    else
      hipLaunchKernelGGL((store_coop_kernel<LA, LB, LC, LD, 1>), dim3((unsigned)a.ntasks), dim3(64), lds, s, a);
  } else if (a.mode == 0) {
    hipLaunchKernelGGL((store_kernel<LA, LB, LC, LD>), dim3((unsigned)((a.ntasks + 3) / 4)), dim3(256), 0, s, a);
  } else {
    constexpr int all = ncart(LA) * ncart(LB);
    StoreArgs g = a;
    const int fit = std::max(1, (int)(kCoopLdsMax / (sizeof(double) * a.n)));
    for (g.row0 = 0; g.row0 < all; g.row0 += g.rows) {
      g.rows = std::min(fit, all - g.row0);
      hipLaunchKernelGGL((it_strip_kernel<LA, LB, LC, LD>), dim3((unsigned)a.ntasks), dim3((unsigned)a.block),
                         sizeof(double) * g.rows * a.n, s, g);
    }
  }
}

// Raise the dynamic LDS limit of the transform kernel of a class.
template <int LA, int LB, int LC, int LD>
static void store_attr_t() {
  if constexpr (LA + LB + LC + LD < kCoopL)
    (void)hipFuncSetAttribute((const void*)it_strip_kernel<LA, LB, LC, LD>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kCoopLdsMax);
}

template <int LA, int LB, int LC, int LD>
static void launch_cstore_t(const CouplingStoreArgs& a, hipStream_t s) {
  if (a.ntasks <= 0) return;
  if constexpr (LA + LB + LC + LD >= kCoopL) {
    constexpr size_t lds = sizeof(double) * coop_wave_doubles<LA, LB, LC, LD>();
    hipLaunchKernelGGL((coupling_store_coop_kernel<LA, LB, LC, LD>), dim3((unsigned)a.ntasks), dim3(64), lds, s, a);
  } else {
    hipLaunchKernelGGL((coupling_store_kernel<LA, LB, LC, LD>), dim3((unsigned)((a.ntasks + 3) / 4)), dim3(256), 0, s,
                       a);
  }
}

}  // namespace lowdin
