// Device-side types and helpers shared by the generated per-class ERI cores and the
// G[D] kernels.  gfx950 only (64-wide wavefronts, FP64 VALU, FP64 global atomics).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

// Boys-function table: F_m(T_i) on T_i = i * BOYS_STEP, i = 0..BOYS_NGRID-1, for
// m = 0..BOYS_MTAB-1, plus exp(-T_i) in the last column.  Each kernel stages a scaled slice
// (9 doubles per grid point) into LDS, with one more row for the asymptotic range (stage_boys).
// The step is just below 0.1 and short in binary (13107 / 2^17), so that i * step is exact.
#define BOYS_STEP (13107.0 / 131072.0)
#define BOYS_INV_STEP (131072.0 / 13107.0)
#define BOYS_TMAX 36.0
#define BOYS_NGRID 361
#define BOYS_MTAB 24
#define BOYS_ROWS (BOYS_NGRID + 1)
#define BOYS_LDS_W 9

// One primitive pair of a shell pair (a, b):
//   p = alpha_a + alpha_b, K = sqrt(2 pi^(5/2)) exp(-alpha_a alpha_b / p |AB|^2) c_a c_b / p
//   (a primitive quartet's prefactor 2 pi^(5/2) K_ab K_cd / (p q sqrt(p + q)) is then
//   K_ab K_cd / sqrt(p + q), split evenly over its two pairs),
//   P = (alpha_a A + alpha_b B) / p, PA = P - A, PB = P - B, o2p = 1 / (2p).
struct alignas(16) PrimPair {
  double p;
  double K;
  double P[3];
  double PA[3];
  double PB[3];
  double o2p;
};

// Per shell pair, in kernel orientation (l_a >= l_b).
struct alignas(16) PairInfo {
  int a, b;        // shells in kernel orientation
  int s1, s2;      // canonical shells (s1 >= s2), as the reference loop visits them
  int p0, p1;      // primitive-pair range in the PrimPair array
  int a0, b0;      // first Cartesian function of a and b
  int loff;        // first Cartesian function of the pair's molecule (0 for one molecule)
  int ar, br;      // first LDS row of a and b: their place among the functions of the
                   // molecule's shells whose angular momentum is la or lb (the pair's class)
  int joff;        // first element of the pair's na x nb block in the pair-ordered Coulomb list
};

struct QuartetArgs {
  const PrimPair* __restrict__ prim;
  int bra_p0, bra_p1, ket_p0, ket_p1;
  int a0, b0, c0, d0;
  double deg;
  bool ket_uniform;          // every lane of the wavefront holds the same ket pair
  bool bra_swap, ket_swap;   // pair held reversed relative to its canonical (s1 >= s2) order
  int ar, br, cr, dr;        // LDS rows of the swept pair's shells (PairInfo::ar, br)
  int jb, jk;                // PairInfo::joff of the bra and of the ket
};

// One density slot per kernel launch (a call with several densities runs one pass per slot).
#define MAX_SLOTS 1
struct JKArgs {
  int ncart;
  int lds_n;                     // rows of an LDS accumulator column (or row): the largest
                                 // molecule's functions of the swept pair class's shells
  const int* rowfn;              // Cartesian function of LDS row r: rowfn[loff + r]
  int pblk, ublk;                // primitive block sizes: lane side, uniform side
  // Density in the Cartesian basis, three copies, so that the digestion reads it along its lanes
  // (with lanes across rows each lane touches a cache line of its own: 8.4 GB of L2 reads per
  // (ss|ps) launch on (H2O)16/cc-pVDZ).  The uniform pair's functions pick rows (a scalar base),
  // the lanes' functions the columns.
  const double* D[MAX_SLOTS];    // row-major ncart x ncart
  const double* Dt[MAX_SLOTS];   // its transpose
  const double* Dp[MAX_SLOTS];   // blocks X(s2,s1) of the shell pairs in pair order (PairInfo::joff)
  // Accumulators.  An FP64 atomic whose wavefront hits 64 consecutive doubles runs at 163 G/s
  // for the whole chip, at scattered or strided addresses at 23 G/s (measured on 160000
  // doubles), so the LDS flushes address memory along their lanes: J in pair order, the K
  // columns of the ket-keyed kernels transposed.
  double* GJ[MAX_SLOTS];         // forward Coulomb updates, pair order (PairInfo::joff)
  double* GJ2[MAX_SLOTS];        // Coulomb updates from the transposed density (matrix, added transposed)
  double* GK[MAX_SLOTS];         // forward exchange updates (matrix)
  double* GK2[MAX_SLOTS];        // exchange updates held transposed: the ket-keyed kernels' K columns
                                 // and the updates from the transposed density (matrix)
  int do_j[MAX_SLOTS];
  int do_k[MAX_SLOTS];
  const int* nonsym;             // device flags: density slot is not symmetric
};

// Element `off` bytes behind a wavefront-uniform row: one scalar base and a 32-bit lane offset
// (an int index would cost a 64-bit address per lane and load)
__device__ __forceinline__ double row_at(const double* __restrict__ row, unsigned off) {
  return *(const double*)((const char*)row + off);
}

// a * b + c rounded once, in the integral type of a kernel (FP64, or FP32 for the mixed
// window's kernels)
__device__ __forceinline__ double fmar(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmar(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// 1/sqrt(x) for x > 0: hardware estimate y0 (about 2^-23 relative), then one third-order
// correction y = y0 (1 + e/2 + 3e^2/8), e = 1 - x y0^2 (the binomial series of (1 - e)^-1/2;
// truncation 2.5 d^3 for a starting error d, far below rounding): five operations where two
// Newton steps take eight, the same accuracy (max 1.4e-16 relative in a CPU emulation with
// |d| <= 2^-22).
__device__ __forceinline__ double rsqrt_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);
  const double c = __builtin_fma(e, 0.375, 0.5);
  return __builtin_fma(y * e, c, y);
}

// Scaled Boys values of a primitive quartet with exponents p, q, s = p + q and centre distance r
// (or, with s = 1 and pq2 = 2 p, of a charge distribution and a point charge).  One rsqrt serves
// the prefactor, the exponent and the asymptotic range:
//   T = p q r^2 / s < 36:  x = s,          b2 = 2 p q / s = 2 alpha,  T2 = r^2 b2 = 2 T
//   T >= 36:               x = 2 p q r^2,  b2 = 1 / r^2
// with rs = 1/sqrt(x), b2 = 2 p q rs^2; then for both
//   (2 alpha)^n F_n(T) / sqrt(s) = rs b2^n G_n,
// G_n = F_n(T) below 36 and sqrt(pi/2) (2n-1)!! above (F_n's asymptotic form; the dropped e^-T
// term is below 2.4e-16), which is the table's last row: nothing is selected behind the table.
// Selecting the argument instead of evaluating both ranges takes the second rsqrt and the
// selects out of the primitive loop: (ss|ps) 68 -> 57 VALU instructions per primitive quartet.
struct BoysArg {
  double rs, b2, T2;
  bool big;
};
__device__ __forceinline__ BoysArg boys_arg(double s, double pq2, double r2) {
  BoysArg a;
  const double xb = pq2 * r2;
  a.big = xb >= 2.0 * BOYS_TMAX * s;
  a.rs = rsqrt_f64(a.big ? xb : s);
  a.b2 = pq2 * (a.rs * a.rs);
  a.T2 = r2 * a.b2;
  return a;
}

// G_0..G_L of a (below 36: F_0..F_L).  Table row i (i * 2 step nearest to T2, or the asymptotic
// row), 8-term Taylor expansion in d = T2_i - T2 (|dT| <= 0.05, truncation below 1e-15 relative):
// the staged coefficients carry 1 / (2^k k!), one FMA per term.  L = 1: F_0 by 9 terms and
// F_1 = -dF_0/dT as the same pass's derivative (d counts in 2T, hence twice it).  L >= 2: F_L, then
// F_m = (2T F_{m+1} + e^-T) / (2m+1) downward with e^-T = e^-T_i e^dT (8 terms); the asymptotic
// row holds G_L with e^-T = 0, and T2 = 1 makes the same recursion G_m = G_{m+1} / (2m+1) (set
// to exactly 1: r^2 b2 would carry its rounding through L steps).  Errors against long double
// over random primitive quartets equal those of evaluating both ranges (3.7e-16 for F_0 of
// L = 0, 8.7e-16 of L = 8).
template <int L>
__device__ __forceinline__ void boys_table(const BoysArg& a, const double* __restrict__ lds, double* G) {
  constexpr double step2 = 2.0 * BOYS_STEP, shift = 6755399441055744.0;   // 1.5 * 2^52
  // L <= 1: the asymptotic row's own T2, so that d = 0; L >= 2: 1, and the row index on its own
  // (the row's higher coefficients are zero)
  const double Tt = a.big ? (L <= 1 ? BOYS_NGRID * step2 : 1.0) : a.T2;
  const double t = __builtin_fma(Tt, 0.5 * BOYS_INV_STEP, shift);   // nearest integer in the low bits
  const unsigned i = L >= 2 && a.big ? BOYS_NGRID : (unsigned)__double2loint(t);
  const double d = __builtin_fma(t - shift, step2, -Tt);
  const double* f = lds + __umul24(i, BOYS_LDS_W);
  if constexpr (L == 0) {
    double p = f[7];
#pragma unroll
    for (int k = 6; k >= 0; --k) p = __builtin_fma(p, d, f[k]);
    G[0] = p;
  } else if constexpr (L == 1) {
    // (the first step of the derivative's recurrence, dp = 0 d + f[8], taken out)
    double dp = f[8], p = __builtin_fma(f[8], d, f[7]);
#pragma unroll
    for (int k = 6; k >= 0; --k) {
      dp = __builtin_fma(dp, d, p);
      p = __builtin_fma(p, d, f[k]);
    }
    G[0] = p;
    G[1] = 2.0 * dp;
  } else {
    double p = f[7];
#pragma unroll
    for (int k = 6; k >= 0; --k) p = __builtin_fma(p, d, f[k]);
    constexpr double c[9] = {1.0, 1.0 / 2, 1.0 / 8, 1.0 / 48, 1.0 / 384, 1.0 / 3840, 1.0 / 46080, 1.0 / 645120,
                             1.0 / 10321920};   // 1 / (2^k k!)
    double e = c[8];
#pragma unroll
    for (int k = 7; k >= 0; --k) e = __builtin_fma(e, d, c[k]);
    e *= f[8];
    G[L] = p;
#pragma unroll
    for (int m = L - 1; m >= 0; --m) G[m] = __builtin_fma(Tt, G[m + 1], e) * (1.0 / (2 * m + 1));
  }
}

// Rb_n = (2 alpha)^n F_n(T) K / sqrt(s), n = 0..L (arguments as in boys_arg).
template <int L>
__device__ __forceinline__ void boys_scaled(double s, double pq2, double r2, double K, const double* __restrict__ lds,
                                            double* Rb) {
  const BoysArg a = boys_arg(s, pq2, r2);
  double G[L + 1];
  boys_table<L>(a, lds, G);
  double pw = K * a.rs;
#pragma unroll
  for (int n = 0; n <= L; ++n) {
    Rb[n] = G[n] * pw;
    pw *= a.b2;
  }
}
// The FP32 integrals' form: F_n in double, rounded, and the prefactors' powers in float (the
// asymptotic range on its own: folding it into the prefactor would round differently).
template <int L>
__device__ __forceinline__ void boys_scaled(double s, double pq2, double r2, double K, const double* __restrict__ lds,
                                            float* Rb) {
  BoysArg a;
  a.rs = rsqrt_f64(s);
  a.b2 = pq2 * (a.rs * a.rs);
  a.T2 = fmin(r2 * a.b2, 2.0 * BOYS_TMAX);
  a.big = false;
  const bool big = r2 * a.b2 >= 2.0 * BOYS_TMAX;
  double F[L + 1];
  boys_table<L>(a, lds, F);
  const double T = big ? 0.5 * (r2 * a.b2) : BOYS_TMAX;
  const double rs = rsqrt_f64(T);
  double fa = 0.88622692545275801365 * rs;   // sqrt(pi)/2 T^-1/2
  const double hr = 0.5 * rs * rs;           // F_{m+1} = F_m (2m+1) / (2T)
  float pw = (float)(K * a.rs);
#pragma unroll
  for (int n = 0; n <= L; ++n) {
    Rb[n] = (float)(big ? fa : F[n]) * pw;
    pw *= (float)a.b2;
    fa = fa * (double)(2 * n + 1) * hr;
  }
}

// Stage the Boys slice for total angular momentum L into LDS (whole workgroup): per grid point
// F_{L+c} / (2^c c!), c = 0..7, and e^{-T_i}; for L = 1 F_c / (2^c c!), c = 0..8.  The last row
// is the asymptotic range's: G_L (L = 1: G_0 and half of G_1) and zeros.
__device__ __forceinline__ void stage_boys(const double* __restrict__ tab, int L, double* lds) {
  constexpr double ifact[9] = {1.0, 1.0 / 2, 1.0 / 8, 1.0 / 48, 1.0 / 384, 1.0 / 3840, 1.0 / 46080, 1.0 / 645120,
                               1.0 / 10321920};
  for (int k = threadIdx.x; k < BOYS_NGRID * BOYS_LDS_W; k += blockDim.x) {
    const int i = k / BOYS_LDS_W, c = k - i * BOYS_LDS_W;
    lds[k] = L == 1 || c < 8 ? tab[i * (BOYS_MTAB + 1) + (L == 1 ? 0 : L) + c] * ifact[c]
                             : tab[i * (BOYS_MTAB + 1) + BOYS_MTAB];
  }
  if (threadIdx.x < BOYS_LDS_W) {
    double g = 1.25331413731550025121;   // sqrt(pi / 2)
    if (L >= 2)
      for (int n = 1; n <= L; ++n) g *= 2 * n - 1;
    lds[BOYS_NGRID * BOYS_LDS_W + threadIdx.x] = threadIdx.x == 0 ? g : L == 1 && threadIdx.x == 1 ? 0.5 * g : 0.0;
  }
  __syncthreads();
}

// Work unit of the segment kernels: `count` tasks of one ket pair starting at `off` in the
// class pair's task list.
struct Segment {
  int off, count, ket, blk;   // ket: the uniform pair; blk: its primitive-block code
};

// Primitive blocks.  A pair with many primitive pairs is split into blocks so that one heavily
// contracted quartet becomes several shorter lane tasks (the digestion is linear in the
// integrals, so partial sums digest independently): blocks of JKArgs::pblk on the per-lane side
// of a task list, blocks of JKArgs::ublk on the wavefront-uniform side (each uniform block is a
// separate work item with an LDS flush of its own).  Task entries and segments carry a block
// code in bits 24..31 of the pair index: 0 = the whole primitive range, k >= 1 = primitives
// [p0 + (k-1) B, min(p1, p0 + k B)).  PRIM_BLOCK and UNI_BLOCK are the sizes of the launches per
// class pair (and PRIM_BLOCK of the Schwarz quartets).
#define PRIM_BLOCK 8
#define UNI_BLOCK 32
#define PAIR_MASK 0xFFFFFFu
__host__ __device__ __forceinline__ unsigned pair_of(unsigned code) { return code & PAIR_MASK; }
__host__ __device__ __forceinline__ unsigned block_of(unsigned code) { return code >> 24; }
__host__ __device__ __forceinline__ void prim_range(const PairInfo& P, unsigned blk, int size, int& p0, int& p1) {
  if (blk == 0) {
    p0 = P.p0;
    p1 = P.p1;
  } else {
    p0 = P.p0 + (int)(blk - 1) * size;
    p1 = P.p1 < p0 + size ? P.p1 : p0 + size;
  }
}

// Sums over the wavefront's lanes of up to four values, added to the LDS words p[0 .. n - 1].
// The FP64 matrix unit, idle otherwise, does the first factor of four: v_mfma_f64_4x4x4 with
// A = 1 (lane = 16 k + 4 b + j holds B[k][j] of block b and D[i = lane / 16][j]) sums a value over
// k into every lane; lanes 16 i .. 16 i + 15 keep value i's, two DPP steps sum over j and four
// lanes per value (b) add to its word.  (Ones in row i only would merge the four values without
// the selects, but 0 x inf would carry an infinity of one value into the other three.)
// 4 matrix + 12 vector instructions and one LDS atomic for four values, where a shuffle tree
// takes 48 LDS and 24 vector instructions.
template <int N>
__device__ __forceinline__ void wave_sum_lds(double* p, const double (&v)[N]) {
  static_assert(N >= 1 && N <= 4, "up to four values");
  const int lane = (int)(threadIdx.x & 63);
  double d = 0.0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const double di = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, v[i], 0.0, 0, 0, 0);
    d = i == 0 || (lane >> 4) == i ? di : d;
  }
  auto quad = [](double x, auto ctrl) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), decltype(ctrl)::value, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), decltype(ctrl)::value, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
  };
  d += quad(d, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  d += quad(d, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  if ((lane & 3) == 0 && (N == 4 || lane < 16 * N)) atomicAdd(p + (lane >> 4), d);
}

// Atomic add of a value whose target is the same on every lane when `uniform` (wavefront-
// uniform flag): the 64 values are summed across lanes first and one lane issues the atomic.
__device__ __forceinline__ void wave_add(double* p, double v, bool uniform) {
  if (uniform) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) atomicAdd(p, v);
  } else {
    atomicAdd(p, v);
  }
}
