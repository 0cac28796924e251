// One-electron integrals on the GPU: overlap S, kinetic T, nuclear attraction V, and the
// Cartesian multipoles up to third order (replaces AOIntegrals::computeAOOneE / OneEDriver,
// src/aointegrals/aointegrals_builders.cpp:27-132,337-467).  McMurchie-Davidson: Hermite expansion coefficients by their closed form
//   E^{ij}_t = sum_{k<=i,l<=j} C(i,k) C(j,l) PA^{i-k} PB^{j-l} n!/(t! m!) (1/4p)^m (1/2p)^t,
//   n = k + l, m = (n - t)/2,
// S_1D(i,j) = E^{ij}_0 sqrt(pi/p),
// T_1D(i,j) = -1/2 [ j(j-1) S(i,j-2) - 2b(2j+1) S(i,j) + 4b^2 S(i,j+2) ],
// V = -(2 pi / p) sum_C Z_C sum_tuv E_t E_u E_v R_tuv(p, P - C).
// S, T and V: one lane per shell pair, the nuclei and primitives over the wavefronts of its
// workgroup, every element of the row-major ncart x ncart matrices stored once.  Multipoles: one
// thread per (shell pair, primitive of a), partial blocks added atomically to zeroed matrices.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "gdirect_kernels.h"
#include "onee.h"

namespace {

__host__ __device__ constexpr int comp_row(int k) {
  int i = 0;
  while ((i + 1) * (i + 2) / 2 <= k) ++i;
  return i;
}
__host__ __device__ constexpr int comp_x(int l, int k) { return l - comp_row(k); }
__host__ __device__ constexpr int comp_y(int l, int k) { return comp_row(k) - (k - comp_row(k) * (comp_row(k) + 1) / 2); }
__host__ __device__ constexpr int comp_z(int l, int k) { return l - comp_x(l, k) - comp_y(l, k); }
// n! for n <= 12 from a table (indices are compile-time constants once the loops unroll, so the
// coefficients fold; a recursive definition would leave run-time calls)
__host__ __device__ constexpr double cfact(int n) {
  constexpr double f[13] = {1.0, 1.0, 2.0, 6.0, 24.0, 120.0, 720.0, 5040.0, 40320.0, 362880.0,
                            3628800.0, 39916800.0, 479001600.0};
  return f[n < 0 ? 0 : (n > 12 ? 12 : n)];
}
__host__ __device__ constexpr double cbinom(int n, int k) { return cfact(n) / (cfact(k) * cfact(n - k)); }

// position of (t, u, v), t + u + v = s, among all Hermite triples with t + u + v <= L:
// the triples of lower sums first, then by descending t and ascending v
__host__ __device__ constexpr int hidx(int t, int u, int v) {
  const int s = t + u + v;
  return s * (s + 1) * (s + 2) / 6 + (s - t) * (s - t + 1) / 2 + v;
}

__device__ __forceinline__ double ipow(double x, int n) {
  double r = 1.0;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (k < n) r *= x;
  return r;
}

// E^{ij}_t for one Cartesian direction (without the exp(-mu AB^2) factor).
__device__ __forceinline__ double hermE(int i, int j, int t, double PA, double PB, double o2p) {
  double s = 0.0;
#pragma unroll
  for (int k = 0; k <= 6; ++k) {
    if (k > i) break;
#pragma unroll
    for (int l = 0; l <= 6; ++l) {
      if (l > j) break;
      const int n = k + l;
      if (n < t || ((n - t) & 1)) continue;
      const int m = (n - t) / 2;
      const double c = cbinom(i, k) * cbinom(j, l) * cfact(n) / (cfact(t) * cfact(m));
      s += c * ipow(PA, i - k) * ipow(PB, j - l) * ipow(0.5 * o2p, m) * ipow(o2p, t);
    }
  }
  return s;
}

// f(0), .., f(N - 1) with compile-time indices
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// E^{ij}_t, i <= LA, j <= LB, of one direction by the recursion over i, then j (every index a
// compile-time constant: the table lives in registers, unused entries are never computed).
template <int LA, int LB>
struct HermE {
  double v[LA + 1][LB + 1][LA + LB + 1];
  __device__ __forceinline__ HermE(double PA, double PB, double o2p) {
    static_for<LA + 1>([&](auto I) {
      static_for<LB + 1>([&](auto J) {
        constexpr int i = I.value, j = J.value;
        if constexpr (i + j == 0) {
          v[0][0][0] = 1.0;
        } else {
          constexpr int si = i > 0 ? i - 1 : i, sj = i > 0 ? j : j - 1, n = i + j;
          const double X = i > 0 ? PA : PB;
          static_for<n + 1>([&](auto T) {
            constexpr int t = T.value;
            double r = 0.0;
            if constexpr (t < n) r = X * v[si][sj][t];
            if constexpr (t > 0) r += o2p * v[si][sj][t - 1];
            if constexpr (t + 1 < n) r += (t + 1) * v[si][sj][t + 1];
            v[i][j][t] = r;
          });
        }
      });
    });
  }
};

// A workgroup takes 64 shell pairs (one per lane) and spreads the nuclei, and the primitives of
// contracted classes, over its wavefronts: NW = PS x (NW / PS) of them, wavefront w taking the
// primitive pairs = w mod PS and the nuclei = w / PS mod NW / PS (S and T: the primitive pairs
// = w mod NW).  The wavefronts' partial blocks meet in LDS and every element is stored once.
// What bounds it is the latency of the (nucleus, primitive pair) evaluations in series per
// wavefront; a thread per (pair, two nuclei) that redid the pair's Hermite coefficients (from
// their closed form, with component loops the compiler left rolled: run-time indices in scratch)
// and added its partial block to HBM atomically took 1.29 ms for (H2O)16/cc-pVDZ.
template <int LA, int LB>
struct OneEShape {
  static constexpr int L = LA + LB;
  static constexpr int NW = L <= 1 ? 16 : 8;
  static constexpr int PS = L <= 1 ? 4 : L == 2 ? 2 : 1;
};

template <int LA, int LB>
__global__ void __launch_bounds__((64 * OneEShape<LA, LB>::NW)) onee_kernel(
    const PairInfo* __restrict__ pairs, int p_begin, int p_end, const OneEShellData sd, const double* __restrict__ Zc,
    const double* __restrict__ xyz, int natom, const double* __restrict__ boys, int ncart, double* __restrict__ S,
    double* __restrict__ T, double* __restrict__ V) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2, NAB = NA * NB, L = LA + LB;
  constexpr int NW = OneEShape<LA, LB>::NW, PS = OneEShape<LA, LB>::PS, CS = NW / PS;
  __shared__ double boys_lds[BOYS_ROWS * BOYS_LDS_W];
  __shared__ double red[NAB * 64];
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  for (int k = threadIdx.x; k < NAB * 64; k += 64 * NW) red[k] = 0.0;
  stage_boys(boys, L, boys_lds);
  const int base = p_begin + (int)blockIdx.x * 64;
  const bool in = base + lane < p_end;
  const PairInfo pi = pairs[in ? base + lane : base];
  const int a = pi.a, b = pi.b;
  const double A[3] = {sd.origin[3 * a], sd.origin[3 * a + 1], sd.origin[3 * a + 2]};
  const double B[3] = {sd.origin[3 * b], sd.origin[3 * b + 1], sd.origin[3 * b + 2]};
  const double AB[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]};
  const double AB2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
  const int pa0 = sd.prim_off[a], pb0 = sd.prim_off[b], npb = sd.prim_off[b + 1] - pb0;
  const int np = in ? (sd.prim_off[a + 1] - pa0) * npb : 0;
  // adds the wavefronts' blocks up and stores them (and their transposes); red is clear again after
  auto store = [&](const double (&x)[NAB], double* M) {
#pragma unroll
    for (int k = 0; k < NAB; ++k) atomicAdd(&red[k * 64 + lane], x[k]);
    __syncthreads();
    for (int k = threadIdx.x; k < NAB * 64; k += 64 * NW) {
      const int q = base + (k & 63);
      if (q < p_end) {
        const PairInfo o = pairs[q];
        const int ab = k >> 6;
        const long r = o.a0 + ab / NB, c = o.b0 + ab % NB;
        M[r * ncart + c] = red[k];
        if (o.a != o.b) M[c * ncart + r] = red[k];
      }
      red[k] = 0.0;
    }
    __syncthreads();
  };
  // ---- nuclear attraction: nuclei of the pair's molecule when several share the context
  {
    int at0 = 0, at1 = natom;
    if (sd.mol_atom0) {
      const int m = sd.shell_mol[a];
      at0 = sd.mol_atom0[m];
      at1 = sd.mol_atom0[m + 1];
    }
    double v[NAB];
#pragma unroll
    for (int k = 0; k < NAB; ++k) v[k] = 0.0;
    for (int k = wid % PS; k < np; k += PS) {
      const int ip = pa0 + k / npb, jp = pb0 + k % npb;
      const double al = sd.alpha[ip], be = sd.alpha[jp];
      const double p = al + be, rp = 1.0 / p;
      const double K = exp(-al * be * rp * AB2) * sd.coef[ip] * sd.coef[jp];
      const double fa = be * rp, fb = -al * rp;   // P - A = fa AB, P - B = fb AB
      const double Px = A[0] + fa * AB[0], Py = A[1] + fa * AB[1], Pz = A[2] + fa * AB[2];
      // Rsum_tuv = sum_C Z_C R_tuv(p, P - C), t + u + w <= L, in the compact index hidx
      constexpr int NH = (L + 1) * (L + 2) * (L + 3) / 6;
      double Rs[NH];
#pragma unroll
      for (int h = 0; h < NH; ++h) Rs[h] = 0.0;
      for (int c = at0 + wid / PS; c < at1; c += CS) {
        // C - P: the sign of (-2p)^n goes into the recursion
        const double D[3] = {xyz[3 * c] - Px, xyz[3 * c + 1] - Py, xyz[3 * c + 2] - Pz};
        double Rb[L + 1];
        boys_scaled<L>(1.0, 2.0 * p, D[0] * D[0] + D[1] * D[1] + D[2] * D[2], Zc[c], boys_lds, Rb);
        // level n of the recursion holds R^n_tuv, t + u + w <= L - n; level 0 is the result
        double R[L + 1][NH];
        static_for<L + 1>([&](auto N) {
          constexpr int n = L - N.value;
          R[n][0] = Rb[n];
          static_for<NH>([&](auto H) {
            constexpr int h = H.value;
            constexpr int s = h < 1 ? 0 : h < 4 ? 1 : h < 10 ? 2 : h < 20 ? 3 : 4;
            if constexpr (h > 0 && s <= L - n) {
              constexpr int o = h - s * (s + 1) * (s + 2) / 6;   // within its sum: by s - t, then w
              constexpr int st = o < 1 ? 0 : o < 3 ? 1 : o < 6 ? 2 : o < 10 ? 3 : 4;
              constexpr int t = s - st, w = o - st * (st + 1) / 2, u = st - w;
              constexpr int d = t > 0 ? 0 : u > 0 ? 1 : 2;
              constexpr int m = t > 0 ? t : u > 0 ? u : w;   // the index that is lowered
              constexpr int h1 = hidx(t - (d == 0), u - (d == 1), w - (d == 2));
              double r = D[d] * R[n + 1][h1];
              if constexpr (m > 1)
                r -= (m - 1) * R[n + 1][hidx(t - 2 * (d == 0), u - 2 * (d == 1), w - 2 * (d == 2))];
              R[n][h] = r;
            }
          });
        });
#pragma unroll
        for (int h = 0; h < NH; ++h) Rs[h] += R[0][h];
      }
      const double o2p = 0.5 * rp, pref = -2.0 * 3.14159265358979323846 * rp * K;
      const HermE<LA, LB> ex(fa * AB[0], fb * AB[0], o2p), ey(fa * AB[1], fb * AB[1], o2p), ez(fa * AB[2], fb * AB[2], o2p);
      static_for<NAB>([&](auto I) {
        constexpr int ia = I.value / NB, ib = I.value % NB;
        constexpr int ax = comp_x(LA, ia), ay = comp_y(LA, ia), az = comp_z(LA, ia);
        constexpr int bx = comp_x(LB, ib), by = comp_y(LB, ib), bz = comp_z(LB, ib);
        double acc = 0.0;
        static_for<ax + bx + 1>([&](auto TT) {
          double au = 0.0;
          static_for<ay + by + 1>([&](auto U) {
            double aw = 0.0;
            static_for<az + bz + 1>([&](auto W) {
              aw += ez.v[az][bz][W.value] * Rs[hidx(TT.value, U.value, W.value)];
            });
            au += ey.v[ay][by][U.value] * aw;
          });
          acc += ex.v[ax][bx][TT.value] * au;
        });
        v[I.value] += pref * acc;
      });
    }
    store(v, V);
  }
  // ---- overlap and kinetic energy
  double s[NAB], t[NAB];
#pragma unroll
  for (int k = 0; k < NAB; ++k) { s[k] = 0.0; t[k] = 0.0; }
  for (int k = wid; k < np; k += NW) {
    const int ip = pa0 + k / npb, jp = pb0 + k % npb;
    const double al = sd.alpha[ip], be = sd.alpha[jp];
    const double p = al + be, rp = 1.0 / p, o2p = 0.5 * rp;
    const double sq = sqrt(3.14159265358979323846 * rp);
    const double K = exp(-al * be * rp * AB2) * sd.coef[ip] * sd.coef[jp] * (sq * sq * sq);
    const double fa = be * rp, fb = -al * rp;
    const HermE<LA, LB + 2> ex(fa * AB[0], fb * AB[0], o2p), ey(fa * AB[1], fb * AB[1], o2p), ez(fa * AB[2], fb * AB[2], o2p);
    auto kin = [&](const HermE<LA, LB + 2>& e, auto I, auto J) {
      constexpr int i = decltype(I)::value, j = decltype(J)::value;
      double d2 = 4.0 * be * be * e.v[i][j + 2][0] - 2.0 * be * (2 * j + 1) * e.v[i][j][0];
      if constexpr (j >= 2) d2 += (double)(j * (j - 1)) * e.v[i][j - 2][0];
      return -0.5 * d2;
    };
    static_for<NAB>([&](auto I) {
      constexpr int ia = I.value / NB, ib = I.value % NB;
      constexpr int ax = comp_x(LA, ia), ay = comp_y(LA, ia), az = comp_z(LA, ia);
      constexpr int bx = comp_x(LB, ib), by = comp_y(LB, ib), bz = comp_z(LB, ib);
      const double sx = ex.v[ax][bx][0], sy = ey.v[ay][by][0], sz = ez.v[az][bz][0];
      using std::integral_constant;
      s[I.value] += K * (sx * sy * sz);
      t[I.value] += K * (kin(ex, integral_constant<int, ax>{}, integral_constant<int, bx>{}) * sy * sz +
                         sx * kin(ey, integral_constant<int, ay>{}, integral_constant<int, by>{}) * sz +
                         sx * sy * kin(ez, integral_constant<int, az>{}, integral_constant<int, bz>{}));
    });
  }
  store(s, S);
  store(t, T);
}

// Cartesian multipole x_C^EX y_C^EY z_C^EZ about C: per direction
//   <i| x_C^e |j> = sum_k C(e,k) (B - C)^(e-k) <i| j + k>     (x - C = (x - B) + (B - C)),
// the overlaps with raised angular momentum on b from the Hermite coefficients E^{i,j+k}_0.
template <int E>
__device__ __forceinline__ double moment_1d(int i, int j, double PA, double PB, double o2p, double BC) {
  double s = 0.0;
#pragma unroll
  for (int k = 0; k <= E; ++k) s += cbinom(E, k) * ipow(BC, E - k) * hermE(i, j + k, 0, PA, PB, o2p);
  return s;
}

template <int LA, int LB, int EX, int EY, int EZ>
__global__ void __launch_bounds__(WG) multipole_kernel(const PairInfo* __restrict__ pairs, int p_begin, int p_end,
                                                       const OneEShellData sd, double Cx, double Cy, double Cz,
                                                       int ncart, double* __restrict__ M) {
  constexpr int NA = (LA + 1) * (LA + 2) / 2, NB = (LB + 1) * (LB + 2) / 2;
  const int P = p_begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (P >= p_end) return;
  const PairInfo pi = pairs[P];
  const int a = pi.a, b = pi.b;
  const int ip = sd.prim_off[a] + (int)blockIdx.y;   // slice: one primitive of a
  if (ip >= sd.prim_off[a + 1]) return;
  const double A[3] = {sd.origin[3 * a], sd.origin[3 * a + 1], sd.origin[3 * a + 2]};
  const double B[3] = {sd.origin[3 * b], sd.origin[3 * b + 1], sd.origin[3 * b + 2]};
  const double AB2 = (A[0] - B[0]) * (A[0] - B[0]) + (A[1] - B[1]) * (A[1] - B[1]) + (A[2] - B[2]) * (A[2] - B[2]);
  const double BCx = B[0] - Cx, BCy = B[1] - Cy, BCz = B[2] - Cz;
  double m[NA][NB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) m[i][j] = 0.0;
  for (int jp = sd.prim_off[b]; jp < sd.prim_off[b + 1]; ++jp) {
    const double al = sd.alpha[ip], be = sd.alpha[jp];
    const double p = al + be, o2p = 0.5 / p;
    const double sq = sqrt(3.14159265358979323846 / p);
    const double K = exp(-al * be / p * AB2) * sd.coef[ip] * sd.coef[jp] * sq * sq * sq;
    const double PA0 = be / p * (B[0] - A[0]), PA1 = be / p * (B[1] - A[1]), PA2 = be / p * (B[2] - A[2]);
    const double PB0 = al / p * (A[0] - B[0]), PB1 = al / p * (A[1] - B[1]), PB2 = al / p * (A[2] - B[2]);
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
      for (int ib = 0; ib < NB; ++ib) {
        const int ax = comp_x(LA, ia), ay = comp_y(LA, ia), az = comp_z(LA, ia);
        const int bx = comp_x(LB, ib), by = comp_y(LB, ib), bz = comp_z(LB, ib);
        m[ia][ib] += K * moment_1d<EX>(ax, bx, PA0, PB0, o2p, BCx) * moment_1d<EY>(ay, by, PA1, PB1, o2p, BCy) *
                     moment_1d<EZ>(az, bz, PA2, PB2, o2p, BCz);
      }
  }
#pragma unroll
  for (int ia = 0; ia < NA; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib) {
      const long r = pi.a0 + ia, cidx = pi.b0 + ib;
      atomicAdd(&M[r * ncart + cidx], m[ia][ib]);
      if (a != b) atomicAdd(&M[cidx * ncart + r], m[ia][ib]);
    }
}

template <int LA, int LB>
void launch_multipole_class(const PairInfo* pairs, int p_begin, int p_end, const OneEShellData& sd, int max_prim,
                            const double* C, int order, int ncart, double* M, hipStream_t stream) {
  const int n = p_end - p_begin;
  const dim3 grid((n + WG - 1) / WG, std::max(1, max_prim));
  const long nc2 = (long)ncart * ncart;
  int k = 0;
#define CQ_MP(EX, EY, EZ)                                                                                   \
  hipLaunchKernelGGL((multipole_kernel<LA, LB, EX, EY, EZ>), grid, dim3(WG), 0, stream, pairs, p_begin, p_end, \
                     sd, C[0], C[1], C[2], ncart, M + (k++) * nc2)
  if (order >= 1) { CQ_MP(1, 0, 0); CQ_MP(0, 1, 0); CQ_MP(0, 0, 1); }
  if (order >= 2) { CQ_MP(2, 0, 0); CQ_MP(1, 1, 0); CQ_MP(1, 0, 1); CQ_MP(0, 2, 0); CQ_MP(0, 1, 1); CQ_MP(0, 0, 2); }
  if (order >= 3) {
    CQ_MP(3, 0, 0); CQ_MP(2, 1, 0); CQ_MP(2, 0, 1); CQ_MP(1, 2, 0); CQ_MP(1, 1, 1);
    CQ_MP(1, 0, 2); CQ_MP(0, 3, 0); CQ_MP(0, 2, 1); CQ_MP(0, 1, 2); CQ_MP(0, 0, 3);
  }
#undef CQ_MP
}

}  // namespace

void launch_multipole(int pair_class, const PairInfo* pairs, int p_begin, int p_end, const OneEShellData& sd,
                      int max_prim, const double* C, int order, int ncart, double* M, hipStream_t stream) {
  if (p_end <= p_begin) return;
  switch (pair_class) {
    case 0: launch_multipole_class<0, 0>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    case 1: launch_multipole_class<1, 0>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    case 2: launch_multipole_class<1, 1>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    case 3: launch_multipole_class<2, 0>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    case 4: launch_multipole_class<2, 1>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    case 5: launch_multipole_class<2, 2>(pairs, p_begin, p_end, sd, max_prim, C, order, ncart, M, stream); break;
    default: break;
  }
}

void launch_onee(int pair_class, const PairInfo* pairs, int p_begin, int p_end, const OneEShellData& sd,
                 const double* Z, const double* xyz, int natom, const double* boys, int ncart, double* S, double* T,
                 double* V, hipStream_t stream) {
  const int n = p_end - p_begin;
  if (n <= 0) return;
#define CQ_ONEE(LA, LB)                                                                                  \
  hipLaunchKernelGGL((onee_kernel<LA, LB>), dim3((n + 63) / 64), dim3(64 * OneEShape<LA, LB>::NW), 0, stream, pairs, \
                     p_begin, p_end, sd, Z, xyz, natom, boys, ncart, S, T, V)
  switch (pair_class) {
    case 0: CQ_ONEE(0, 0); break;
    case 1: CQ_ONEE(1, 0); break;
    case 2: CQ_ONEE(1, 1); break;
    case 3: CQ_ONEE(2, 0); break;
    case 4: CQ_ONEE(2, 1); break;
    case 5: CQ_ONEE(2, 2); break;
    default: break;
  }
}
