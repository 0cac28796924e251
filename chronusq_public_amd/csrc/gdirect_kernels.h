// Kernel wrappers shared by the generated per-class translation units and the host code.
#pragma once
#include "gdirect_device.h"
#include "_gen/eri_counts.inc"

#define WG 256

// ---------------------------------------------------------------------------------------
// Uniform groups and their task regions
// ---------------------------------------------------------------------------------------
// A group is up to MAX_GROUP shell pairs of one class, one molecule and one primitive-block
// count that share their first shell (kernel orientation): kets (c, d_0) .. (c, d_{n-1}) of a
// ket-keyed class pair, bras (a, b_0) .. of a bra-keyed one.  Its pairs are
// uorder[first .. first + n).  The screening kernel sweeps the other class once for the whole
// group; every swept pair that survives against at least one member joins the group's union
// (in sweep order, at most the class pair's union bound per task region).  One task region
// (a run of uint2 entries in the class pair's task list) holds
//   [0]            {n, U}                      members, union size
//   [1 + m]        {count_m, offset_m}         member m's quartet list (offsets from the region)
//   [offset_m + t] {swept pair | block << 24, slot}   one entry per primitive block of every
//                  swept pair whose quartet with member m survives (slot: its union index)
// so the quartets keep every lane busy (the members' lists run as one dense list), while the J
// of a swept pair collects in its LDS slot across the members and primitive blocks and leaves
// the work item once.
#define MAX_GROUP 16
struct GroupRec {
  int first;       // into uorder
  int n;           // members
  int ublk;        // primitive blocks of the uniform side (equal for every member)
  int nslot;       // segment slots reserved for the group's first task region (ublk)
  int task_base;   // the group's task entries, from the start of its batch's task list
  int seg_base;    // the group's segment slots, from the start of its batch's segment list
  int pad0, pad1;
};
// Every group owns a fixed part of its batch's task list, sized by the plan's worst case, and
// ublk reserved segment slots for its first task region, so the screening places its output
// without atomics; further task regions of a group (a union over the bound) take slots of the
// batch's overflow pool (one atomic each).  A group without survivors writes its reserved
// slots with count 0; the kernels skip them.

// ---------------------------------------------------------------------------------------
// ERI kernel wrappers, instantiated once per class pair by the generated units
// ---------------------------------------------------------------------------------------

// Quartet of one lane's bra (pair B, task code bra_code) with the wavefront-uniform ket pair
// kk and its primitive block kblk (both from readfirstlane, so the ket data is loaded through
// the scalar path); lanes that do not own a task of this ket get an empty bra range and
// degeneracy 0.
__device__ __forceinline__ void make_quartet_uniform_ket(const PairInfo& B, unsigned bra_code, unsigned kk,
                                                         unsigned kblk, bool mine,
                                                         const PairInfo* __restrict__ pairs,
                                                         const PrimPair* __restrict__ prims, const JKArgs& jk,
                                                         QuartetArgs& q) {
  const PairInfo K = pairs[kk];
  int bp0, bp1, kp0, kp1;
  prim_range(B, block_of(bra_code), jk.pblk, bp0, bp1);
  prim_range(K, kblk, jk.ublk, kp0, kp1);
  q.prim = prims;
  q.bra_p0 = bp0;
  q.bra_p1 = mine ? bp1 : bp0;
  q.ket_p0 = kp0;
  q.ket_p1 = kp1;
  q.a0 = B.a0; q.b0 = B.b0; q.c0 = K.a0; q.d0 = K.b0;
  const double deg = (B.a == B.b ? 1.0 : 2.0) * (K.a == K.b ? 1.0 : 2.0) * (pair_of(bra_code) == kk ? 1.0 : 2.0);
  q.deg = mine ? deg : 0.0;
  q.ket_uniform = true;
  q.bra_swap = B.a != B.s1;
  q.ket_swap = K.a != K.s1;
  q.ar = B.ar; q.br = B.br;   // LDS rows of the swept bra's shells
  q.cr = 0; q.dr = 0;
  q.jb = B.joff; q.jk = K.joff;
}

// Quartet of the wavefront-uniform bra pair bb and its primitive block bblk (from
// readfirstlane) with one lane's ket (pair K, task code ket_code); lanes that do not own a task
// get an empty ket range and degeneracy 0.
__device__ __forceinline__ void make_quartet_uniform_bra(const PairInfo& K, unsigned ket_code, unsigned bb,
                                                         unsigned bblk, bool mine,
                                                         const PairInfo* __restrict__ pairs,
                                                         const PrimPair* __restrict__ prims, const JKArgs& jk,
                                                         QuartetArgs& q) {
  const PairInfo B = pairs[bb];
  int bp0, bp1, kp0, kp1;
  prim_range(B, bblk, jk.ublk, bp0, bp1);
  prim_range(K, block_of(ket_code), jk.pblk, kp0, kp1);
  q.prim = prims;
  q.bra_p0 = bp0;
  q.bra_p1 = bp1;
  q.ket_p0 = kp0;
  q.ket_p1 = mine ? kp1 : kp0;
  q.a0 = B.a0; q.b0 = B.b0; q.c0 = K.a0; q.d0 = K.b0;
  const double deg = (B.a == B.b ? 1.0 : 2.0) * (K.a == K.b ? 1.0 : 2.0) * (bb == pair_of(ket_code) ? 1.0 : 2.0);
  q.deg = mine ? deg : 0.0;
  q.ket_uniform = false;
  q.bra_swap = B.a != B.s1;
  q.ket_swap = K.a != K.s1;
  q.ar = 0; q.br = 0;
  q.cr = K.ar; q.dr = K.br;   // LDS rows of the swept ket's shells
  q.jb = B.joff; q.jk = K.joff;
}

// Work items come from up to eight queues, one per XCD (workgroups are dispatched round robin over
// the XCDs): queue x hands out items x, x + nq, x + 2 nq, ... to the class pair's workgroups blk
// with blk % nq == x, so the counters do not contend across the chip and every queue has a
// consumer (nq <= nblk, the class pair's workgroups).
#define WORK_QUEUES 8
__device__ __forceinline__ int take_item(unsigned* __restrict__ work, unsigned blk, unsigned nblk) {
  const unsigned nq = nblk < WORK_QUEUES ? nblk : WORK_QUEUES;
  const unsigned x = blk % nq;
  return (int)(x + nq * atomicAdd(&work[x], 1u));
}

// A workgroup's current item: its segment and group (wavefront-uniform), and the members' shells,
// task lists and running block counts in LDS.
struct ItemLds {
  int next;                      // the item after this one, taken while this one runs
  int unit;                      // next unit to hand out
  int sh[MAX_GROUP];             // first function of each member's own (second) shell
  int joff[MAX_GROUP];           // its Coulomb block
  int moff[MAX_GROUP], mcnt[MAX_GROUP];
  int mblk[MAX_GROUP];           // 64-entry blocks of the members up to and including this one
};

// Stages the members of the item's group (first wavefront; the caller synchronises).
__device__ __forceinline__ void stage_members(ItemLds& it, const GroupRec& gr, const uint2* __restrict__ reg,
                                              const PairInfo* __restrict__ pairs, const int* __restrict__ uorder) {
  if (threadIdx.x < 64) {
    const int m = (int)threadIdx.x;
    int nb = 0;
    if (m < gr.n) {
      const uint2 hm = reg[1 + m];
      const PairInfo& P = pairs[uorder[gr.first + m]];
      it.sh[m] = P.b0;
      it.joff[m] = P.joff;
      it.moff[m] = (int)hm.y;
      it.mcnt[m] = (int)hm.x;
      nb = ((int)hm.x + 63) >> 6;
    }
#pragma unroll
    for (int o = 1; o < MAX_GROUP; o <<= 1) {
      const int y = __shfl_up(nb, o);
      if (m >= o) nb += y;
    }
    if (m < gr.n) it.mblk[m] = nb;
  }
}

// Hands the calling wavefront the next unit of the item (beyond the wavefronts' first ones).
__device__ __forceinline__ int next_unit(ItemLds& it) {
  int u = 0;
  if ((threadIdx.x & 63) == 0) u = atomicAdd(&it.unit, 1);
  return __builtin_amdgcn_readfirstlane(u);
}

// Unit u of the item: chunk, member (wavefront-uniform) and 64-entry block of its list; units are
// chunk-major, nbt blocks per chunk.
__device__ __forceinline__ void locate_unit(const ItemLds& it, int n, int nbt, int cpi, int u, int& chunk, int& member,
                                            int& block) {
  chunk = 0;
  if (cpi > 1) {   // (few chunks per item: a short scalar loop instead of a division)
    while (u >= nbt) { u -= nbt; ++chunk; }
  }
  const int lane = (int)(threadIdx.x & 63);
  const int upto = lane < n ? it.mblk[lane] : 0x7fffffff;
  member = __popcll(__ballot(upto <= u));
  block = u - (member > 0 ? it.mblk[member - 1] : 0);
  member = __builtin_amdgcn_readfirstlane(member);
  block = __builtin_amdgcn_readfirstlane(block);
}

// Group kernels.  Work items are (task region, group of cpi chunks) pairs from an atomic queue
// (cpi divides the class pair's chunk count); each workgroup spreads the item's (chunk, member,
// block of 64 of that member's entries) units over its wavefronts -- the member wavefront-
// uniform, one quartet per lane -- then flushes its LDS accumulators to HBM once.  The next item is
// taken from its queue before the units start, so that the round trip of the counter's atomic
// runs beside them:
//  * ket-keyed (DIG 0 or 1): K columns of the shared c shell and of every member's d shell (DIG 1;
//    with DIG 0 K goes to HBM atomics directly), J(c, d_m) of every member, and J of every union
//    bra;
//  * bra-keyed (DIG 2): K rows of the shared a shell and of every member's b shell, J(a, b_m) of
//    every member, and J of every union ket.
// Dynamic LDS: [(NU0 + mmax NU1) LN K columns or rows (not DIG 0)][mmax NU0 NU1 J of the members]
//              [ub NS J slots][ub ints: PairInfo::joff of each slot's swept pair],
// NU0 x NU1 the uniform pair's block (c, d or a, b), NS the size of the swept pair's.
// The flush's lanes walk consecutive LDS words, i.e. consecutive Cartesian functions of one K
// column or row (functions are ordered by angular momentum within a molecule, so a swept class's
// functions are one or two runs) and consecutive elements of the pair-ordered J list: whole
// cache lines per atomic instruction ((H2O)16/cc-pVDZ, (ss|ps): 7.7 M atomics per launch, at
// 23 G/s scattered 0.33 of its 0.57 ms).
// C: the class pair (sizes, chunk count, total angular momentum and the quartet function).  Blocks
// blk of nblk work on it (a whole grid, or a part of a merged launch's).
template <class C, int WGS, int DIG, typename R>
__device__ __forceinline__ void group_body(
    const uint2* __restrict__ tasks, const Segment* __restrict__ segs, int nres, const unsigned* __restrict__ ovf,
    unsigned* __restrict__ work, const PairInfo* __restrict__ pairs, const PrimPair* __restrict__ prims,
    const double* __restrict__ boys, const JKArgs& jk, const GroupRec* __restrict__ groups,
    const int* __restrict__ uorder, int mmax, int ub, int cpi, unsigned blk, unsigned nblk, double* boys_lds,
    ItemLds& s_it, double* dyn_lds) {
  constexpr bool BRA = DIG == 2;   // uniform bra
  constexpr int NU0 = BRA ? C::NA : C::NC, NU1 = BRA ? C::NB : C::ND, NU = NU0 * NU1;
  constexpr int NS = BRA ? C::NC * C::ND : C::NA * C::NB;
  const int nit = C::NCH / cpi;   // items per task region: groups of cpi chunks
  const long nitems = ((long)nres + *ovf) * nit;
  if (nitems == 0) return;
  if (threadIdx.x == 0) s_it.next = take_item(work, blk, nblk);
  __syncthreads();
  int item = __builtin_amdgcn_readfirstlane(s_it.next);
  if (item >= nitems) return;
  const int LN = jk.lds_n;
  const int nacc = DIG == 0 ? 0 : (NU0 + mmax * NU1) * LN;
  double* accK = dyn_lds;
  double* accU = dyn_lds + nacc;
  double* jsl = accU + mmax * NU;
  int* spair = (int*)(jsl + ub * NS);
  for (int k = threadIdx.x; k < nacc + mmax * NU + ub * NS; k += WGS) dyn_lds[k] = 0.0;
  stage_boys(boys, C::L, boys_lds);   // (synchronises: LDS is zeroed, every thread has the item)
  const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  while (item < nitems) {
    int nxt = 0;
    if (threadIdx.x == WGS - 1) nxt = take_item(work, blk, nblk);
    const Segment sg = segs[nit == 1 ? item : item / nit];
    const int ch0 = nit == 1 ? 0 : (item % nit) * cpi;
    const bool filled = sg.count != 0;   // else a slot its group did not fill
    const GroupRec gr = groups[sg.ket];
    const int n = gr.n;
    const uint2* reg = tasks + sg.off;
    int U = 0;
    if (threadIdx.x == 0) s_it.unit = WGS / 64;
    if (filled) {
      U = (int)reg[0].y;
      stage_members(s_it, gr, reg, pairs, uorder);
    }
    __syncthreads();
    if (filled) {
      // units (chunk, member, 64-entry block of the member's list), chunk-major, handed to the
      // workgroup's wavefronts as they come free (a member's list runs from heavily contracted to
      // single primitives): the member is wavefront-uniform
      const int nbt = __builtin_amdgcn_readfirstlane(s_it.mblk[n - 1]);
      for (int u = wid; u < nbt * cpi; u = next_unit(s_it)) {
        int dch, mu, eb;
        locate_unit(s_it, n, nbt, cpi, u, dch, mu, eb);
        const int b0 = eb << 6, t = b0 + lane;
        const bool active = t < s_it.mcnt[mu];
        const uint2 e = reg[s_it.moff[mu] + (active ? t : b0)];
        const PairInfo S = pairs[pair_of(e.x)];
        if (active) spair[e.y] = S.joff;
        const unsigned up = __builtin_amdgcn_readfirstlane((unsigned)uorder[gr.first + mu]);
        QuartetArgs q;
        if constexpr (BRA) make_quartet_uniform_bra(S, e.x, up, (unsigned)sg.blk, active, pairs, prims, jk, q);
        else make_quartet_uniform_ket(S, e.x, up, (unsigned)sg.blk, active, pairs, prims, jk, q);
        C::template jk<DIG, R>(q, jk, boys_lds, ch0 + dch, accK, accK + (NU0 + mu * NU1) * LN, accU + mu * NU,
                               jsl + (long)e.y * NS);
      }
    }
    if (threadIdx.x == WGS - 1) s_it.next = nxt;
    __syncthreads();
    item = __builtin_amdgcn_readfirstlane(s_it.next);
    if (!filled) continue;
    if constexpr (DIG != 0) {   // one K column or row per wavefront and step
      const PairInfo U0 = pairs[uorder[gr.first]];
      double* const G = BRA ? jk.GK[0] : jk.GK2[0];
      for (int c = wid; c < NU0 + n * NU1; c += WGS / 64) {
        const int m = (c - NU0) / NU1;
        const int fn = c < NU0 ? U0.a0 + c : __builtin_amdgcn_readfirstlane(s_it.sh[m]) + (c - NU0 - m * NU1);
        double* g = G + (long)fn * jk.ncart;
        double* acc = accK + c * LN;
        for (int k = lane; k < LN; k += 64) {
          const double v = acc[k];
          if (v != 0.0) {
            atomicAdd(g + jk.rowfn[U0.loff + k], v);
            acc[k] = 0.0;
          }
        }
      }
    }
    for (int k = threadIdx.x; k < n * NU; k += WGS) {
      const double v = accU[k];
      if (v != 0.0) {
        const int m = k / NU;
        atomicAdd(&jk.GJ[0][s_it.joff[m] + k - m * NU], v);
        accU[k] = 0.0;
      }
    }
    for (int k = threadIdx.x; k < U * NS; k += WGS) {
      const double v = jsl[k];
      if (v != 0.0) {
        const int u = k / NS;
        atomicAdd(&jk.GJ[0][spair[u] + k - u * NS], v);
        jsl[k] = 0.0;
      }
    }
    __syncthreads();   // the accumulators are clear and s_it may change
  }
}

#define GROUP_KERNEL_PARAMS                                                                     \
  const uint2 *__restrict__ tasks, const Segment *__restrict__ segs, int nres,                  \
      const unsigned *__restrict__ ovf, unsigned *__restrict__ work,                            \
      const PairInfo *__restrict__ pairs, const PrimPair *__restrict__ prims,                   \
      const double *__restrict__ boys, JKArgs jk, const GroupRec *__restrict__ groups,          \
      const int *__restrict__ uorder, int mmax, int ub, int cpi
#define DEFINE_CLASS_KERNELS(NAME)                                                              \
  template <int WGS, int DIG, typename R>                                                       \
  __global__ void __launch_bounds__(WGS, DIG == 1 ? Cls_##NAME::WAVES : 1) eri_grp_##NAME(GROUP_KERNEL_PARAMS) { \
    __shared__ double boys_lds[BOYS_ROWS * BOYS_LDS_W];                                         \
    __shared__ ItemLds s_it;                                                                    \
    extern __shared__ double dyn_lds[];                                                         \
    group_body<Cls_##NAME, WGS, DIG, R>(tasks, segs, nres, ovf, work, pairs, prims, boys, jk, groups, uorder, mmax, \
                                        ub, cpi, blockIdx.x, gridDim.x, boys_lds, s_it, dyn_lds); \
  }
#define DEFINE_CLASS_BLOCK(NAME)                                                                \
  /* Block kernel: task t adds its (primitive-block) contribution to the contracted Cartesian \
     block of output slot slot[t] (t when slot is null), zeroed by the caller. */              \
  __global__ void __launch_bounds__(WG, Cls_##NAME::WAVES < 2 ? 1 : 2) eri_block_##NAME(        \
      const uint2* __restrict__ tasks, long count, const PairInfo* __restrict__ pairs,          \
      const PrimPair* __restrict__ prims, const double* __restrict__ boys, double* out,          \
      int blk, const int* __restrict__ slot) {                                                  \
    __shared__ double boys_lds[BOYS_ROWS * BOYS_LDS_W];                                         \
    if ((long)blockIdx.x * WG >= count) return;                                                 \
    stage_boys(boys, Cls_##NAME::L, boys_lds);                                                  \
    for (long base = (long)blockIdx.x * WG; base < count; base += (long)gridDim.x * WG) {       \
      const long wbase = base + (threadIdx.x & ~63);                                            \
      if (wbase >= count) break;                                                                \
      const long t = base + threadIdx.x;                                                        \
      const bool active = t < count;                                                            \
      const uint2 tk = tasks[active ? t : wbase];                                               \
      const PairInfo B = pairs[pair_of(tk.x)];                                                  \
      const PairInfo K = pairs[pair_of(tk.y)];                                                  \
      QuartetArgs q;                                                                            \
      q.prim = prims;                                                                           \
      prim_range(B, block_of(tk.x), PRIM_BLOCK, q.bra_p0, q.bra_p1);                            \
      prim_range(K, block_of(tk.y), PRIM_BLOCK, q.ket_p0, q.ket_p1);                            \
      if (active) quartet_block_##NAME(q, out + (slot ? (long)slot[t] : t) * (long)blk, boys_lds); \
    }                                                                                           \
  }

// Bra-keyed group kernel (DIG 2), for class pairs whose bra class has few pairs: the uniform
// members are bras (a, b_m) sharing shell a, the lanes hold the kets that survive against them.
#define DEFINE_CLASS_SEGB(NAME)                                                                 \
  template <typename R>                                                                         \
  __global__ void __launch_bounds__(WG, Cls_##NAME::WAVES) eri_grpb_##NAME(GROUP_KERNEL_PARAMS) { \
    __shared__ double boys_lds[BOYS_ROWS * BOYS_LDS_W];                                         \
    __shared__ ItemLds s_it;                                                                    \
    extern __shared__ double dyn_lds[];                                                         \
    group_body<Cls_##NAME, WG, 2, R>(tasks, segs, nres, ovf, work, pairs, prims, boys, jk, groups, uorder, mmax, ub, \
                                     cpi, blockIdx.x, gridDim.x, boys_lds, s_it, dyn_lds);      \
  }

// ---------------------------------------------------------------------------------------
// Merged launches
// ---------------------------------------------------------------------------------------
// A launch per class pair costs its own start and tail 21 times over, and at most four run at once
// (one per hardware queue): H2O/6-31G* 690 us, most of it launches and the longest lane tasks in
// series, 243 us merged.  A merged launch runs all class pairs of one tier (similar register
// counts) side by side, one range of blocks per class pair, and one grid row (y) per density slot.
struct MergedEntry {
  int k;                         // class pair
  int blk0, nblk;                // its blocks
  int nres, mmax, ub, cpi, lds_n, rowfn;
  long long task_off, seg_off;
};
struct MergedArgs {
  MergedEntry e[CQ_NUM_CLASS_PAIRS];
  int n;
  unsigned jmask, kmask;         // density slots with a Coulomb / an exchange contraction
  long long slot_words;          // workspace words from one slot to the next
};
#define MERGED_KERNEL_PARAMS                                                                    \
  MergedArgs ma, const uint2 *__restrict__ tasks, const Segment *__restrict__ segs,             \
      const unsigned *__restrict__ ovf, unsigned *__restrict__ work,                            \
      const PairInfo *__restrict__ pairs, const PrimPair *__restrict__ prims,                   \
      const double *__restrict__ boys, JKArgs jk0, const GroupRec *__restrict__ groups,         \
      const int *__restrict__ uorder

// The block's entry, and the accumulators and density of its slot.
__device__ __forceinline__ const MergedEntry& merged_entry(const MergedArgs& ma, const JKArgs& jk0, JKArgs& jk) {
  int i = 0;
  while ((int)blockIdx.x >= ma.e[i].blk0 + ma.e[i].nblk) ++i;
  const MergedEntry& e = ma.e[i];
  const int s = (int)blockIdx.y;
  const long long off = s * ma.slot_words;
  jk = jk0;
  jk.D[0] += off; jk.Dt[0] += off; jk.Dp[0] += off;
  jk.GJ[0] += off; jk.GJ2[0] += off; jk.GK[0] += off; jk.GK2[0] += off;
  jk.nonsym += s;
  jk.do_j[0] = (int)(ma.jmask >> s) & 1;
  jk.do_k[0] = (int)(ma.kmask >> s) & 1;
  jk.lds_n = e.lds_n;
  jk.rowfn += e.rowfn;
  return e;
}

typedef void (*BlockKernel)(const uint2*, long, const PairInfo*, const PrimPair*, const double*, double*, int,
                            const int*);
typedef void (*GroupKernel)(const uint2*, const Segment*, int, const unsigned*, unsigned*, const PairInfo*,
                            const PrimPair*, const double*, JKArgs, const GroupRec*, const int*, int, int, int);

typedef void (*MergedKernel)(MergedArgs, const uint2*, const Segment*, const unsigned*, unsigned*, const PairInfo*,
                             const PrimPair*, const double*, JKArgs, const GroupRec*, const int*);

// Bra and ket class, chunks, name and sizes of a class pair in one orientation.
struct ClassShape {
  int bi, ki, nchunk;
  const char* name;
  int nc, nd, na, nb;
};

struct ClassKernels : ClassShape {
  int i, j, L;
  BlockKernel block;
  // grp[precision][variant]: precision 0 FP64 / 1 FP32 integrals; variant 0 ket-keyed with HBM K
  // atomics, 1 ket-keyed with LDS K columns, 2 bra-keyed with LDS K rows (null where the class
  // pair has no bra-keyed form)
  GroupKernel grp[2][3];
  int seg_wg;         // workgroup size of the ket-keyed kernels
  int tier, merged;   // merged launch the class pair belongs to, its form there (1 ket-keyed, 2 bra-keyed)
  ClassShape mrg;     // its orientation there
};
