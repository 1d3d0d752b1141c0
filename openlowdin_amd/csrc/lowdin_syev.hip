// Symmetric eigenproblems that fit in one compute unit, one workgroup per
// matrix with everything in LDS: Householder tridiagonalisation, Q from its
// reflectors, implicit-shift QL with the rotations applied to Q.
//
// The orthogonalised Fock matrix of an iteration is small (two water
// molecules in 6-31G**: 50), and a library call takes some hundred dependent
// launches over it.  Measured, library / here: n = 25 0.64 / 0.17, 50 1.29 /
// 0.55, 64 1.70 / 0.88 ms; 72 matrices at once take as long as one.  Past 64
// a row no longer fits a lane and the library changes its method: with two
// rows per lane 75 1.16 / 1.32, 100 1.63 / 2.14 ms.  (Parallel Jacobi over the
// same LDS: 50 0.49, 75 1.13 ms, with twice to four times the loss of
// orthogonality.)  Each stage is bound by latency, not by arithmetic:
//   * tridiagonalisation: every wavefront holds the reflector and the matrix
//     product in registers and owns every 8th column, so that a step needs
//     two barriers; scalars are found by all wavefronts alike;
//   * Q: 16 lanes hold a column in registers through all reflectors, without
//     a barrier;
//   * QL, the longest: one lane chases the bulge of the next sweep (a chain of
//     some 14 dependent operations for each of the n^2 rotations, 0.14 us)
//     while a second wavefront applies the last sweep's, one row per lane;
//   * one step of refinement against the matrix itself, five products on the
//     matrix unit (10 us at n = 64): rotations alone leave residuals up to twice
//     the library's.  Worst of 6 matrices of 4 kinds each at n = 64, library /
//     rotations / refined: |AV - VW| / |A| 2.0e-15 / 2.7e-15 / 1.0e-15,
//     |V^T V - 1| 1.4e-14 / 1.8e-14 / 0.5e-14.
#include <hip/hip_runtime.h>

#include <cmath>

#include "lowdin_kernels.h"

namespace lowdin {
namespace {

constexpr int kSyevMax = 64;              // one row per lane
constexpr int kSyevThreads = 512, kSyevWaves = kSyevThreads / 64;
constexpr int kSyevPasses = 16 * kSyevMax / kSyevThreads;   // columns of Q per 16 lanes
constexpr int kSyevIterations = 60;       // QL sweeps per eigenvalue

struct SyevArgs {
  double* a;       // n x n column-major, upper triangle read; eigenvectors on return
  double* w;       // eigenvalues, ascending
  int* info;       // 0, or 1: not converged or not finite
  size_t stride_a, stride_w;
  int n;
};

template <int kCtrl>
__device__ __forceinline__ double dpp(double x) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, kCtrl, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), kCtrl, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ double lane_value(double x, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Sum over 16 neighbouring lanes, and over the wavefront; the same in all.
__device__ __forceinline__ double row_sum(double x) {
  x += dpp<0xB1>(x);    // lanes 1 apart
  x += dpp<0x4E>(x);    // 2
  x += dpp<0x141>(x);   // halves of 8
  x += dpp<0x140>(x);   // of 16
  return x;
}
__device__ __forceinline__ double wave_total(double x) {
  x = row_sum(x);
  return (lane_value(x, 0) + lane_value(x, 16)) + (lane_value(x, 32) + lane_value(x, 48));
}

// 1 / sqrt(x) from the hardware estimate and one cubic step (x normal).
__device__ __forceinline__ double rsqrt_cubic(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double h = fma(-x * y, y, 1.0);
  return fma(y * h, fma(0.375, h, 0.5), y);
}

// 16 x 16 tile (I, J) of c + X Y of n x n matrices on the matrix unit, x(i, k)
// and y(k, j) their elements: a lane's four are rows 16 I + lane / 16 + 4 r,
// column 16 J + lane % 16.
typedef double double4v __attribute__((ext_vector_type(4)));

template <typename X, typename Y>
__device__ __forceinline__ double4v tile_product(double4v c, int n, int I, int J, int lane, X x, Y y) {
  const int i = 16 * I + (lane & 15), j = 16 * J + (lane & 15);
  for (int k0 = 0; k0 < n; k0 += 16) {   // the same for all lanes
    double a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + 4 * u + (lane >> 4);
      a[u] = i < n && k < n ? x(i, k) : 0.0;
      b[u] = k < n && j < n ? y(k, j) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], c, 0, 0, 0);
  }
  return c;
}

template <typename F>
__device__ __forceinline__ void tile_each(int n, int I, int J, int lane, F f) {
  const int j = 16 * J + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 16 * I + (lane >> 4) + 4 * r;
    if (i < n && j < n) f(i, j, r);
  }
}

// Tile t of those on and above the diagonal, by columns.
__device__ __forceinline__ int2 upper_tile(int t) {
  int J = 0;
  while ((J + 1) * (J + 2) / 2 <= t) ++J;
  return make_int2(t - J * (J + 1) / 2, J);
}

__global__ __launch_bounds__(kSyevThreads) void syev_kernel(SyevArgs g) {
  extern __shared__ double lds[];
  const int n = g.n, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ld = n | 1;                     // odd: columns side by side use different banks
  double* A = lds;                          // A[c ld + i]: row i of column c
  double* B = A + n * ld;                   // second matrix of the last step
  double* part = B;                         // kSyevWaves x n partial products
  double* d = B + max(n * ld, kSyevWaves * n);
  double* e = d + n;
  double* tau = e + n;
  double* rot = tau + n;                    // two sweeps of (c, s)
  double* red = rot + 4 * n;
  int* hdr = (int*)(red + kSyevWaves);      // two of (first, last, state)
  double* G = g.a + (size_t)blockIdx.x * g.stride_a;
  double* W = g.w + (size_t)blockIdx.x * g.stride_w;

  // both triangles from the upper one, scaled by a power of two to at most one
  double mx = 0.0;
  for (int k = tid; k < n * n; k += kSyevThreads) {
    const int c = k / n, i = k % n;
    const double v = G[(size_t)max(i, c) * n + min(i, c)];
    A[c * ld + i] = v;
    mx = fabs(v) < INFINITY ? fmax(mx, fabs(v)) : INFINITY;
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if (lane == 0) red[w] = mx;
  __syncthreads();
  mx = 0.0;
  for (int k = 0; k < kSyevWaves; ++k) mx = fmax(mx, red[k]);
  if (!(mx < INFINITY)) {   // not finite: left as it is and reported
    if (tid == 0) g.info[blockIdx.x] = 1;
    return;
  }
  int ex = 0;
  if (mx > 0.0) (void)frexp(mx, &ex);
  for (int k = tid; k < n * ld; k += kSyevThreads) A[k] = ldexp(A[k], -ex);
  __syncthreads();

  // Step j: reflector H = 1 - tau v v^T (v[j+1] = 1) of column j below the
  // diagonal, A22 -= v u^T + u v^T.
  for (int j = 0; j < n - 2; ++j) {
    const bool below = lane > j && lane < n;
    double v = below ? A[j * ld + lane] : 0.0;
    const double x0 = lane_value(v, j + 1);
    const double s2 = wave_total(lane > j + 1 ? v * v : 0.0);
    if (s2 < 1e-290) {   // nothing to eliminate (to 1e-145 of the largest element)
      if (tid == 0) {
        d[j] = A[j * ld + j];
        e[j] = x0;
        tau[j] = 0.0;
      }
      continue;
    }
    const double nrm = sqrt(fma(x0, x0, s2));
    const double beta = x0 > 0.0 ? -nrm : nrm;
    const double t = (beta - x0) / beta, inv = 1.0 / (x0 - beta);
    v = lane == j + 1 ? 1.0 : v * inv;
    double y = 0.0;
    const int c0 = j + 1 + ((w - j - 1) & (kSyevWaves - 1));   // first own column
    for (int c = c0; c < n; c += kSyevWaves)
      if (lane < n) y = fma(A[c * ld + lane], lane_value(v, c), y);
    if (lane < n) part[w * n + lane] = y;
    __syncthreads();
    y = 0.0;
    if (below) {
#pragma unroll
      for (int k = 0; k < kSyevWaves; ++k) y += part[k * n + lane];
    }
    y = t * fma(-0.5 * t * wave_total(y * v), v, y);
    if (w == 0) {
      if (below) A[j * ld + lane] = v;
      if (lane == 0) {
        d[j] = A[j * ld + j];
        e[j] = beta;
        tau[j] = t;
      }
    }
    for (int c = c0; c < n; c += kSyevWaves) {
      const double vc = lane_value(v, c), yc = lane_value(y, c);
      // products rounded one by one: both triangles get the same bits
      if (below) A[c * ld + lane] -= __dadd_rn(__dmul_rn(v, yc), __dmul_rn(y, vc));
    }
    __syncthreads();
  }
  if (tid == 0) {
    for (int j = n > 2 ? n - 2 : 0; j < n; ++j) d[j] = A[j * ld + j];
    if (n > 1) e[n - 2] = A[(n - 2) * ld + n - 1];
  }
  __syncthreads();

  // Q = H_0 H_1 ...: columns tid / 16 + kCols b, rows tid % 16 + 16 k
  {
    constexpr int kCols = kSyevThreads / 16;
    const int col = tid >> 4, sub = tid & 15;
    double q[kSyevPasses][4];
#pragma unroll
    for (int b = 0; b < kSyevPasses; ++b)
#pragma unroll
      for (int k = 0; k < 4; ++k) q[b][k] = sub + 16 * k == col + kCols * b ? 1.0 : 0.0;
    for (int j = n - 3; j >= 0; --j) {
      const double t = tau[j];
      if (t == 0.0) continue;   // that column holds no reflector
      double v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = sub + 16 * k;
        v[k] = i > j && i < n ? A[j * ld + i] : 0.0;
      }
#pragma unroll
      for (int b = 0; b < kSyevPasses; ++b) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) s = fma(v[k], q[b][k], s);
        s = -t * row_sum(s);
#pragma unroll
        for (int k = 0; k < 4; ++k) q[b][k] = fma(s, v[k], q[b][k]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < kSyevPasses; ++b)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int c = col + kCols * b, i = sub + 16 * k;
        if (c < n && i < n) A[c * ld + i] = q[b][k];
      }
  }
  __syncthreads();

  // QL: state 0 (rotations lo..hi-1 of a sweep to apply), 1 done, 2 failed
  int l = 0, iter = 0;
  for (int sweep = 0;; ++sweep) {
    const int par = sweep & 1;
    double* cs = rot + 2 * n * par;
    int* hd = hdr + 3 * par;
    if (w == 0) {
      const double dr = lane < n ? d[lane] : 0.0, er = lane < n - 1 ? e[lane] : 0.0;
      // [l, hi]: first block without a negligible e
      const double dn = lane < n - 1 ? d[lane + 1] : 0.0;
      const unsigned long long small =
          __ballot(lane >= n - 1 || fabs(er) <= fmax(2.220446049250313e-16 * (fabs(dr) + fabs(dn)), 1e-18));
      int hi = l;
      for (; l < n - 1; ++l, iter = 0) {
        const unsigned long long from = small >> l << l;
        hi = from ? min((int)__builtin_ctzll(from), n - 1) : n - 1;
        if (hi > l) break;
      }
      const int state = l >= n - 1 ? 1 : ++iter > kSyevIterations ? 2 : 0;
      if (lane == 0) {
        hd[0] = l;
        hd[1] = hi;
        hd[2] = state;
      }
      if (state == 0) {
        const double e_hi = lane_value(er, hi);   // negligible, or past the end
        const double dl = lane_value(dr, l), el = lane_value(er, l), delta = 0.5 * (lane_value(dr, l + 1) - dl);
        const double root = sqrt(fma(delta, delta, el * el));
        const double sigma = dl - el * el / (delta + (delta < 0.0 ? -root : root));
        double a = lane_value(dr, hi), b = lane_value(dr, hi - 1), gk = lane_value(er, hi - 1), x = a - sigma, z = gk;
        if (lane == 0) {
          // d and e are read from the other lanes' registers: a load would
          // wait for the stores before it
          for (int k = hi - 1; k >= l; --k) {
            const int k1 = k > l ? k - 1 : l;   // after the last rotation not used
            const double bn = lane_value(dr, k1), en = lane_value(er, k1);
            const double r2 = fma(x, x, z * z);
            const bool turn = r2 > 1e-280;
            const double y = turn ? rsqrt_cubic(r2) : 1.0;
            const double c = turn ? x * y : 1.0, s = z * y;
            e[k + 1] = r2 * y;   // of k = hi - 1: put back below
            const double h = fma(s, b - a, (c + c) * gk);
            d[k + 1] = fma(s, h, a);
            cs[2 * k] = c;
            cs[2 * k + 1] = s;
            x = fma(c, h, -gk);
            z = s * en;
            a = fma(-s, h, b);
            b = bn;
            gk = c * en;
          }
          d[l] = a;
          e[l] = x;
          e[hi] = e_hi;
        }
      }
    }
    __syncthreads();
    const int lo = hd[0], hi = hd[1], state = hd[2];
    if (state != 0) {
      if (tid == 0) g.info[blockIdx.x] = state - 1;
      break;
    }
    const int r = tid - 64;
    if (r >= 0 && r < n) {
      double f = A[hi * ld + r];
      int k = hi - 1;
      for (; k >= lo + 3; k -= 4) {
        double c[4], s[4], zk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          c[u] = cs[2 * (k - u)];
          s[u] = cs[2 * (k - u) + 1];
          zk[u] = A[(k - u) * ld + r];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          A[(k - u + 1) * ld + r] = fma(c[u], f, s[u] * zk[u]);
          f = fma(c[u], zk[u], -s[u] * f);
        }
      }
      for (; k >= lo; --k) {
        const double c = cs[2 * k], s = cs[2 * k + 1], zk = A[k * ld + r];
        A[(k + 1) * ld + r] = fma(c, f, s * zk);
        f = fma(c, zk, -s * f);
      }
      A[lo * ld + r] = f;
    }
  }

  // One step of refinement: with S = V^T A V and R = 1 - V^T V of the vectors
  // found, w = S_ii / (1 - R_ii) and V += V E, E_ij = R_ij / 2 + X_ij, X_ij =
  // (S_ij + (w_i + w_j) R_ij / 2) / (w_j - w_i) = -X_ji where that is small
  // enough for its square to vanish, else 0 (levels as close as that rotate
  // into each other by rounding alone).
  const int nt = (n + 15) >> 4;             // tiles of 16 x 16
  __syncthreads();
  for (int k = tid; k < n * n; k += kSyevThreads) {
    const int c = k / n, i = k % n;
    B[c * ld + i] = ldexp(G[(size_t)max(i, c) * n + min(i, c)], -ex);
  }
  __syncthreads();
  double4v acc[2];
  for (int u = 0, t = w; t < nt * nt; ++u, t += kSyevWaves)
    acc[u] = tile_product(double4v{}, n, t / nt, t % nt, lane, [&](int i, int k) { return B[k * ld + i]; },
                          [&](int k, int j) { return A[j * ld + k]; });
  __syncthreads();
  for (int u = 0, t = w; t < nt * nt; ++u, t += kSyevWaves)
    tile_each(n, t / nt, t % nt, lane, [&](int i, int j, int r) { B[j * ld + i] = acc[u][r]; });   // A V
  __syncthreads();
  double4v S[2], N[2];                      // V^T A V, V^T V: tiles I <= J
  for (int u = 0, t = w; t < nt * (nt + 1) / 2; ++u, t += kSyevWaves) {
    const int2 b = upper_tile(t);
    const auto row = [&](int i, int k) { return A[i * ld + k]; };
    S[u] = tile_product(double4v{}, n, b.x, b.y, lane, row, [&](int k, int j) { return B[j * ld + k]; });
    N[u] = tile_product(double4v{}, n, b.x, b.y, lane, row, [&](int k, int j) { return A[j * ld + k]; });
    tile_each(n, b.x, b.y, lane, [&](int i, int j, int r) {
      if (i == j) d[i] = S[u][r] / N[u][r];
    });
  }
  __syncthreads();
  for (int u = 0, t = w; t < nt * (nt + 1) / 2; ++u, t += kSyevWaves) {
    const int2 b = upper_tile(t);
    tile_each(n, b.x, b.y, lane, [&](int i, int j, int r) {
      if (i > j) return;
      const double half = 0.5 * (i == j ? 1.0 - N[u][r] : -N[u][r]);
      const double num = fma(d[i] + d[j], half, S[u][r]), gap = d[j] - d[i];
      const double x = i != j && fabs(num) < 1e-9 * fabs(gap) ? num / gap : 0.0;
      B[j * ld + i] = half + x;
      if (i != j) B[i * ld + j] = half - x;
    });
  }
  __syncthreads();
  for (int u = 0, t = w; t < nt * nt; ++u, t += kSyevWaves) {
    double4v v{};
    tile_each(n, t / nt, t % nt, lane, [&](int i, int j, int r) { v[r] = A[j * ld + i]; });
    acc[u] = tile_product(v, n, t / nt, t % nt, lane, [&](int i, int k) { return A[k * ld + i]; },
                          [&](int k, int j) { return B[j * ld + k]; });
  }
  __syncthreads();
  for (int u = 0, t = w; t < nt * nt; ++u, t += kSyevWaves)
    tile_each(n, t / nt, t % nt, lane, [&](int i, int j, int r) { A[j * ld + i] = acc[u][r]; });

  // ascending order (equal values keep theirs)
  int* rank = (int*)rot;
  __syncthreads();
  for (int i = tid; i < n; i += kSyevThreads) {
    const double wi = d[i];
    int k = 0;
    for (int j = 0; j < n; ++j) k += d[j] < wi || (d[j] == wi && j < i);
    rank[i] = k;
    W[k] = ldexp(wi, ex);
  }
  __syncthreads();
  for (int k = tid; k < n * n; k += kSyevThreads) {
    const int c = k / n, i = k % n;
    G[(size_t)rank[c] * n + i] = A[c * ld + i];
  }
}

size_t syev_lds(int n) {
  const int nld = n * (n | 1), second = nld > kSyevWaves * n ? nld : kSyevWaves * n;
  return sizeof(double) * (size_t)(nld + second + 7 * n + kSyevWaves) + 8 * sizeof(int);
}

}  // namespace

bool launch_syev(double* a, int n, size_t stride_a, double* w, size_t stride_w, int* info, int count, hipStream_t s) {
  if (n < 1 || n > kSyevMax) return false;
  if (count <= 0) return true;
  // above 64 KB from n = 62
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)syev_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)syev_lds(kSyevMax));
  (void)attr;
  const SyevArgs g{a, w, info, stride_a, stride_w, n};
  hipLaunchKernelGGL(syev_kernel, dim3(count), dim3(kSyevThreads), syev_lds(n), s, g);
  return true;
}

}  // namespace lowdin
