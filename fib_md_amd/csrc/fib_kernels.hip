// fib_kernels.hip -- gfx950 kernels of the FIB_MD force-and-integrate path.
//
// Pipeline per neighbor rebuild (replaces si_nlist, si.f90:87-276), three to
// seven launches:
//   k_sort_small  the sort of instances of up to 8,192 atoms and cells, each by
//                 one workgroup; of larger ones:
//   k_bin         cell of every atom with the reference's FP64 arithmetic
//                 (nlist.f90:29), atomic histogram per cell bucket
//   k_scan_*      exclusive scan of the bucket histogram in two passes
//   k_scatter     counting-sort scatter; k_fixup restores a deterministic
//                 order inside each bucket (old sorted position)
//   k_reorder     gathers every per-atom array into cell order and resets
//                 what a build resets
//   k_nbuild      one wavefront per cell: the 27-cell halo filtered by the box
//                 around the cell's atoms, the reference pair predicate
//                 (si.f90:156-170) lane-parallel, survivors compacted with
//                 ballots; beside it the copy back of the in-place sort
// Per force evaluation (replaces si_force, si.f90:384-552):
//   k_legs        one thread per atom: SW pair and Moliere forces in registers
//                 and which pairs are three-body legs; from the rows right
//                 after a build, from the near lists it then keeps later on
//   k_tri         one lane per leg, legs staged in LDS: the vertex terms
//                 centred on the leg's atom, force on the leg's neighbour into
//                 G, where the neighbour keeps its force on the atom (RA), and
//                 the reaction on the centre
//     extra_pass  in the same launch: vertex terms of the stale build-time
//                 triplet graph
//   k_force3      one thread per atom: own terms + the G entries its neighbours
//                 wrote for it; the velocity update of either integrator
// Per step (replaces the inline Verlet of onestep, timeint.f90:165-236):
//   k_pos         thermostat scaling, position update, side freeze, rebox and
//                 the sputter-layer rules in one pass
//   k_md_pos      the MD-step mode's integrator: shells, half kick, drift,
//                 pins, removal, displacements
//   k_md_decide   which instances rebuild, and what removed atoms carry out
//   k_md_ctl      the next dt
//
// Reductions (energy, virial, thermostat sums, max KE) use per-block partials,
// which a wavefront per 256 blocks sums in a fixed order, so every result is
// deterministic.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "fib_device.h"
#include "fib_kernels.h"

namespace fibk {

// Kernels of the list build take `gate`: null, or gate[0] = "some instance
// rebuilds" and gate[1 + k] = "instance k rebuilds".  With gate[0] zero they
// return at once (block-uniform), so a build can be enqueued -- or captured
// in a graph -- and skipped on the device; atoms, cells and lists of an
// instance whose own flag is zero are left untouched.  k_md_decide writes
// every flag at the start of each MD step, before any kernel reads them.
#define GATE_OR_RETURN(gate) \
  do {                       \
    if ((gate) && !(gate)[0]) return; \
  } while (0)
// MD-step mode: once a list build of a step overflowed its width, `halt` is
// set and every later kernel of the step (and of the steps after it, when
// they were already enqueued or captured) returns at once, so the host can
// grow the lists and finish the step from the state the overflow left.
#define HALT_OR_RETURN(halt) \
  do {                       \
    if ((halt) && *(halt)) return; \
  } while (0)
__device__ __forceinline__ bool gated_out(const int *gate, int inst) {
  return gate && !gate[1 + inst];
}
// Under a gate, the blocks of FIB_BLOCK atoms of instances that are not
// rebuilt are skipped whole, before any per-atom load: every such block lies
// inside one instance (binst), and the grid-stride loops that use this are
// launched with FIB_BLOCK threads and advance by whole blocks, so all lanes
// of a block take the same branch.
__device__ __forceinline__ bool block_gated_out(const int *gate, const int *__restrict__ binst,
                                                int p) {
  if (!gate) return false;
  const int b = __builtin_amdgcn_readfirstlane(p / FIB_BLOCK);
  return !gate[1 + binst[b]];
}

// Element loops of the list-build kernels run grid-stride over a capped grid
// (GRID_CAP workgroups): a build skipped by its gate then costs a small launch
// instead of one workgroup per 256 atoms.
#define GRID_CAP 2048
#define GRID_STRIDE(p, n) \
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < (n); p += gridDim.x * blockDim.x)

// ---------------------------------------------------------------------------
// helpers
#define OFF_W 32        // bytes per atom of the stencil-offset table (27 used)
// states of an atom's near list (see near_mark_moved): its number of entries,
// at most NEAR_CAP, or one of
#define NEAR_CAP 16
#define NEAR_J 0x7ffffffu
#define NEAR_MOVED 253  // moved more than delta / 2 and told its partners
#define NEAR_FULL 254   // no near list
#define NEAR_FRESH 255  // just built: the next pass makes the near list
__device__ __forceinline__ uint64_t wbits(const double4 &x) {
  return (uint64_t)__double_as_longlong(x.w);
}
__device__ __forceinline__ uint32_t meta_of(const double4 &x) { return (uint32_t)wbits(x); }
__device__ __forceinline__ int32_t orig_of(const double4 &x) { return (int32_t)(wbits(x) >> 32); }
__device__ __forceinline__ int type_of(uint32_t m) { return (int)(m & META_TYPE_MASK); }
__device__ __forceinline__ int inst_of(uint32_t m) { return (int)(m >> META_INST_SHIFT); }

// Workgroups are dispatched round-robin over the 8 XCDs; remap so each XCD
// walks a contiguous range of atoms and neighbour gathers stay in its L2.
__device__ __forceinline__ int xcd_remap(int w, int nb) {
  const int nx = 8;
  int q = nb / nx, r = nb % nx;
  int x = w % nx, loc = w / nx;
  return (x < r) ? x * (q + 1) + loc : r * (q + 1) + (x - r) * q + loc;
}
// The same with every XCD taking a run of 2^xs blocks in turn, for passes
// whose work differs from instance to instance (the pair pass does twice the
// work where the lists are new): an instance is then spread over all XCDs.
// One of four replicas rebuilt: k_legs 205 us with contiguous eighths of the
// batch, where two XCDs had all of it; see xcd_shift for the run's length.
__device__ __forceinline__ int xcd_remap(int w, int nb, int xs) {
  const int full = nb >> (xs + 3) << (xs + 3);
  if (w >= full) return full + xcd_remap(w - full, nb - full);
  return (w >> (xs + 3) << (xs + 3)) + ((w & 7) << xs) + ((w >> 3) & ((1 << xs) - 1));
}

// LDS hand-off between the lanes of one wavefront (no workgroup barrier:
// the wavefronts of a workgroup may work independently).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Reference cell index of one coordinate (nlist.f90:29), no contraction.
__device__ __forceinline__ int ref_cell(double x, double ilb, double lb, double h) {
#pragma clang fp contract(off)
  double t = x * ilb;
  double f = floor(t);
  double w = x - f * lb;
  double q = w / h;
  return (int)q + 1;
}

// Reference minimum-image squared distance (si.f90:156-157), no contraction.
__device__ __forceinline__ double ref_r2(const double4 &a, const double4 &b, const DInst &in) {
#pragma clang fp contract(off)
  double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
  double x0 = d0 - round(d0 * in.ilb[0]) * in.lb[0];
  double x1 = d1 - round(d1 * in.ilb[1]) * in.lb[1];
  double x2 = d2 - round(d2 * in.ilb[2]) * in.lb[2];
  return x0 * x0 + x1 * x1 + x2 * x2;
}
// The raw differences a - b of ref_r2, and its sum of squares when every
// NINT shift is zero (|d| < L/4 makes |d/L| < 1/2): then d - 0*L = d and the
// result equals ref_r2 bit for bit.
__device__ __forceinline__ void ref_diff(const double4 &a, const double4 &b, double &d0,
                                         double &d1, double &d2) {
  d0 = a.x - b.x; d1 = a.y - b.y; d2 = a.z - b.z;
}
__device__ __forceinline__ double ref_sq(double d0, double d1, double d2) {
#pragma clang fp contract(off)
  return d0 * d0 + d1 * d1 + d2 * d2;
}

// Minimum-image difference a - b (force kernels: contraction allowed).
__device__ __forceinline__ void min_image(const double4 &a, const double4 &b, const DInst &in,
                                          double &x0, double &x1, double &x2) {
  double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
  x0 = d0 - round(d0 * in.ilb[0]) * in.lb[0];
  x1 = d1 - round(d1 * in.ilb[1]) * in.lb[1];
  x2 = d2 - round(d2 * in.ilb[2]) * in.lb[2];
}

__device__ __forceinline__ int find_inst_by_cell(const DInst *I, int ninst, int gcell) {
  int lo = 0, hi = ninst - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (I[mid].cell_real_off <= gcell) lo = mid; else hi = mid - 1;
  }
  return lo;
}
__device__ __forceinline__ int find_inst_by_bucket(const DInst *I, int ninst, int b) {
  int lo = 0, hi = ninst - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (I[mid].bucket_off <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Streaming accesses: arrays that a force pass reads or writes once per step
// (its own rows, counts and per-atom results), loaded and stored
// non-temporally so that they do not push the gathered neighbour positions
// out of L2.  FIB_NT_LD (loads) and FIB_NT_ST (stores) hold one bit per
// pass: 1 k_legs, 2 k_tri, 4 k_force3, 8 k_md_pos (velocities, forces,
// build positions, displacements) and 16 (stores only) k_nbuild's rows.
// k_legs reads each list row as four or five 16-byte loads in turn, and
// non-temporal loads fetch the row again for each of them (k_legs 0.70 ->
// 1.04 ms on the 8.2 M-atom dose batch), so its loads stay cached; so do
// k_force3's reads of its own G entries, which the partners' lookups read
// again.  On that batch, streaming the force passes' other accesses makes
// the step 1.5 % faster (mixed), k_md_pos's a further 1.5 % (k_md_pos
// itself 13 %), and k_nbuild's row stores make the next k_md_pos faster too.
#ifndef FIB_NT_LD
#define FIB_NT_LD 14
#endif
#ifndef FIB_NT_ST
#define FIB_NT_ST 31
#endif
template <class V>
struct NtVec { typedef V type; };
template <>
struct NtVec<int4> { typedef int __attribute__((ext_vector_type(4))) type; };
template <>
struct NtVec<float4> { typedef float __attribute__((ext_vector_type(4))) type; };
template <>
struct NtVec<double4> { typedef double __attribute__((ext_vector_type(4))) type; };
template <bool NT, class V>
__device__ __forceinline__ V ld_nt(const V *p) {
  if constexpr (NT) {
    typedef typename NtVec<V>::type N;
    static_assert(sizeof(N) == sizeof(V), "vector size");
    const N t = __builtin_nontemporal_load(reinterpret_cast<const N *>(p));
    V v;
    __builtin_memcpy(&v, &t, sizeof(V));
    return v;
  } else {
    return *p;
  }
}
template <bool NT, class V>
__device__ __forceinline__ void st_nt(V *p, const V &v) {
  if constexpr (NT) {
    typedef typename NtVec<V>::type N;
    static_assert(sizeof(N) == sizeof(V), "vector size");
    N t;
    __builtin_memcpy(&t, &v, sizeof(V));
    __builtin_nontemporal_store(t, reinterpret_cast<N *>(p));
  } else {
    *p = v;
  }
}

// p[byte offset]: one 32-bit offset beside a scalar base, not a 64-bit
// address per lane
template <typename V>
__device__ __forceinline__ V ld_off(const V *p, uint32_t byte) {
  return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(p) + byte);
}
// ---------------------------------------------------------------------------
// Reductions of NV doubles per slot.  Slot operations: RED_SUM, RED_MAX, and
// the exact top two of a set of values over three slots (RED_TOP2 at slot k:
// the largest; k + 1 RED_TOP2_CNT: how many values equal it; k + 2
// RED_TOP2_SND: the largest value below it, -1e300 when there is none).
// Every operation is associative and commutative and the combining order is
// fixed, so results are deterministic.
enum { RED_SUM = 0, RED_MAX = 1, RED_TOP2 = 2, RED_TOP2_CNT = 3, RED_TOP2_SND = 4 };

__device__ __forceinline__ double red_identity(int op) {
  return (op == RED_SUM || op == RED_TOP2_CNT) ? 0.0 : -1.0e300;
}

__device__ __forceinline__ void top2_merge(double &m, double &c, double &s, double m2, double c2,
                                           double s2) {
  const double M = fmax(m, m2);
  const double cn = (m == M ? c : 0.0) + (m2 == M ? c2 : 0.0);
  const double sn = fmax(m < M ? m : s, m2 < M ? m2 : s2);
  m = M;
  c = cn;
  s = sn;
}

// x <- x (op) y, slot by slot (a top-two triple at once).
template <int NV, typename OP>
__device__ __forceinline__ void red_merge(double (&x)[NV], const double (&y)[NV], const OP &op) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (op[k] == RED_TOP2) {
      if (k + 2 < NV) top2_merge(x[k], x[k + 1], x[k + 2], y[k], y[k + 1], y[k + 2]);
    } else if (op[k] == RED_SUM) {
      x[k] += y[k];
    } else if (op[k] == RED_MAX) {
      x[k] = fmax(x[k], y[k]);
    }
  }
}

// Block reduction into per-block partials, layout partials[k * pstride +
// block]; k_finalize combines them per instance.
template <int NV, int BS>
__device__ void block_partials(double (&v)[NV], const int (&op)[NV], int lblock, int pstride,
                               double *__restrict__ partials) {
  __shared__ double red[BS / FIB_WAVE][NV];
  const int lane = threadIdx.x % FIB_WAVE, wid = threadIdx.x / FIB_WAVE;
  for (int o = FIB_WAVE / 2; o > 0; o >>= 1) {
    double y[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) y[k] = __shfl_xor(v[k], o);
    red_merge<NV>(v, y, op);
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) red[wid][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double x[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) x[k] = red[0][k];
    for (int w = 1; w < BS / FIB_WAVE; ++w) {
      double y[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) y[k] = red[w][k];
      red_merge<NV>(x, y, op);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) partials[(size_t)k * pstride + lblock] = x[k];
  }
}

// Per instance, combine the partials of its blocks in a fixed order that
// depends on the instance alone: one wavefront per chunk of FIN_CH blocks
// (lane l takes blocks l, l + 64, ..., then a butterfly), and, when the
// instance has more than one, one wavefront over its chunks the same way.
// All NV slots at once, so the loads of every slot are in flight together,
// except the ten of the energies and the virial, of three producers: a
// wavefront per slot.  A wavefront per chunk instead of a workgroup of 1024
// threads per 1024 blocks: 14 -> 5 us a reduction, at 4 k as at 2 M atoms; up
// to FIN_ONE chunks combined where they are reduced, and the ten slots side by
// side: 101 k atoms (two chunks, ten slots) 18.7 -> 12.8 us.
#define FIN_CH FIB_FIN_CH
// red_merge with the operations of a RedSpec: k_md_pos' six slots start with a
// top-two triple, every other reduction is sums and maxima.
template <int NV>
__device__ __forceinline__ void fin_merge(double (&x)[NV], const double (&y)[NV],
                                          const RedSpec &rs) {
  constexpr int K0 = NV == 6 ? 3 : 0;
  if constexpr (NV == 6) top2_merge(x[0], x[1], x[2], y[0], y[1], y[2]);
#pragma unroll
  for (int k = K0; k < NV; ++k) x[k] = rs.op[k] == RED_MAX ? fmax(x[k], y[k]) : x[k] + y[k];
}
__device__ __forceinline__ int fin_chunks(const DInst &in, int bs) {
  return (in.natm_pad / bs + FIN_CH - 1) / FIN_CH;
}
template <int NV>
__device__ __forceinline__ void fin_wave(double (&x)[NV], const RedSpec &rs) {
  for (int o = FIB_WAVE / 2; o > 0; o >>= 1) {
    double y[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) y[k] = __shfl_xor(x[k], o);
    fin_merge<NV>(x, y, rs);
  }
}
// chunk c of instance `in` from the producers' partials
template <int NV>
__device__ __forceinline__ void fin_chunk(double (&x)[NV], const DInst &in, int c,
                                          const double *__restrict__ partials, int pstride,
                                          const RedSpec &rs) {
  const int blk0 = in.atom_off / rs.bs, nblk = in.natm_pad / rs.bs;
  const int lane = threadIdx.x % FIB_WAVE;
#pragma unroll
  for (int k = 0; k < NV; ++k) x[k] = red_identity(rs.op[k]);
#pragma unroll
  for (int m = 0; m < FIN_CH / FIB_WAVE; ++m) {
    const int b = c * FIN_CH + m * FIB_WAVE + lane;
    if (b < nblk) {
      double y[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) y[k] = partials[(size_t)k * pstride + blk0 + b];
      fin_merge<NV>(x, y, rs);
    }
  }
  fin_wave<NV>(x, rs);
}
// slot k of it, a sum over the regions of k_legs, k_tri (rs.sub partials, one
// or four, for one of the others', see tri_partials, or 0: one or four of four
// places, by the instance) and extra_pass
__device__ __forceinline__ double fin_chunk_slot(int k, const DInst &in, int c,
                                                 const double *__restrict__ partials, int pstride,
                                                 const RedSpec &rs) {
  const int blk0 = in.atom_off / rs.bs, nblk = in.natm_pad / rs.bs;
  const double *const p = partials + (size_t)k * pstride;
  const size_t reg = (size_t)FIB_NRED * pstride;
  const bool four = rs.sub == 4 || (rs.sub == 0 && in.natm_pad <= FIB_TRI_SMALL);
  double x = 0;
#pragma unroll
  for (int m = 0; m < FIN_CH / FIB_WAVE; ++m) {
    const int b = c * FIN_CH + m * FIB_WAVE + (int)(threadIdx.x % FIB_WAVE);
    if (b < nblk) {
      const size_t at = (size_t)(blk0 + b);
      x += p[at];
      const double *const t = p + reg + at * (rs.sub == 1 ? 1 : 4);
      x += four ? (t[0] + t[1]) + (t[2] + t[3]) : t[0];
      x += p[2 * reg + at];
    }
  }
  for (int o = FIB_WAVE / 2; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
// the chunks of an instance
template <int NV>
__device__ __forceinline__ void fin_combine(double (&x)[NV], int inst, int nci, int nch,
                                            const double *__restrict__ tmp, const RedSpec &rs) {
#pragma unroll
  for (int k = 0; k < NV; ++k) x[k] = red_identity(rs.op[k]);
  for (int c = threadIdx.x % FIB_WAVE; c < nci; c += FIB_WAVE) {
    double y[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) y[k] = tmp[((size_t)inst * nch + c) * NV + k];
    fin_merge<NV>(x, y, rs);
  }
  fin_wave<NV>(x, rs);
}
template <int NV>
__device__ __forceinline__ void fin_store(const double (&x)[NV], const RedSpec &rs, DCtl &ctl) {
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (rs.dst[k] >= 0) reinterpret_cast<double *>(&ctl)[rs.dst[k]] = x[k];
}
// one wavefront of any workgroup: the rest of the reduction of instance
// `inst` into its control record, with how = FIN_ALL from the partials (the
// instance has one chunk), FIN_COMBINE from the chunks k_finalize left in
// tmp, FIN_DONE nothing
enum { FIN_DONE = 0, FIN_COMBINE = 1, FIN_ALL = 2 };
template <int NV>
__device__ __forceinline__ void fin_finish(int how, int inst, const DInst &in,
                                           const double *__restrict__ partials, int pstride,
                                           const double *__restrict__ tmp, int nch,
                                           const RedSpec &rs, DCtl &ctl) {
  if (how == FIN_DONE) return;
  double x[NV];
  if (how == FIN_ALL) {
    fin_chunk<NV>(x, in, 0, partials, pstride, rs);
  } else {
    const int nci = fin_chunks(in, rs.bs);
    if (nci <= 1) return;  // k_finalize stored it
    fin_combine<NV>(x, inst, nci, nch, tmp, rs);
  }
  if (threadIdx.x % FIB_WAVE == 0) fin_store<NV>(x, rs, ctl);
}
// Workgroup (k, y): chunks [y * per, (y + 1) * per) of instance k, a wavefront
// each (NV == 10: one per slot of each).  Instances of up to FIN_ONE chunks are
// reduced by one workgroup, which also combines them; of larger ones
// k_finalize2, or the next kernel, combines the chunks.
#define FIN_ONE 8
#define FIN_WAVES 16
template <int NV>
__global__ __launch_bounds__(FIN_WAVES *FIB_WAVE) void k_finalize(
    const DInst *__restrict__ I, const double *__restrict__ partials, int pstride, RedSpec rs,
    int per, DCtl *__restrict__ ctl, double *__restrict__ tmp, const int *__restrict__ halt) {
  HALT_OR_RETURN(halt);
  constexpr int SL = NV == 10 ? NV : 1;  // wavefronts per chunk
  __shared__ double s_x[FIN_ONE * NV];
  const int inst = blockIdx.x, c0 = blockIdx.y * per, nch = gridDim.y * per;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FIB_WAVE);
  const DInst &in = I[inst];
  const int nci = fin_chunks(in, rs.bs), n = min(nci - c0, per);
  // past the chunks of this instance (the grid has those of the largest):
  // s_x stays unwritten, and the record is another workgroup's
  if (n <= 0) return;
  for (int q = wid; q < n * SL; q += blockDim.x / FIB_WAVE) {
    if constexpr (NV == 10) {
      const double x = fin_chunk_slot(q % SL, in, c0 + q / SL, partials, pstride, rs);
      if (threadIdx.x % FIB_WAVE == 0) s_x[q] = x;
    } else {
      double x[NV];
      fin_chunk<NV>(x, in, c0 + q, partials, pstride, rs);
      if (threadIdx.x % FIB_WAVE == 0) {
        if (nci == 1) fin_store<NV>(x, rs, ctl[inst]);  // nothing to combine
#pragma unroll
        for (int k = 0; k < NV; ++k) s_x[q * NV + k] = x[k];
      }
    }
  }
  if (SL == 1 && nci == 1) return;
  __syncthreads();
  if (nci <= per) {
    if (wid != 0) return;
    double x[NV];
    fin_combine<NV>(x, 0, nci, 0, s_x, rs);
    if (threadIdx.x == 0) fin_store<NV>(x, rs, ctl[inst]);
  } else {
    for (int q = threadIdx.x; q < n * NV; q += blockDim.x)
      tmp[((size_t)inst * nch + c0) * NV + q] = s_x[q];
  }
}
template <int NV>
__global__ __launch_bounds__(FIB_WAVE) void k_finalize2(const DInst *__restrict__ I, int nch,
                                                        RedSpec rs, DCtl *__restrict__ ctl,
                                                        const double *__restrict__ tmp,
                                                        const int *__restrict__ halt) {
  HALT_OR_RETURN(halt);
  const int inst = blockIdx.x;
  fin_finish<NV>(FIN_COMBINE, inst, I[inst], nullptr, 0, tmp, nch, rs, ctl[inst]);
}

// ---------------------------------------------------------------------------
// binning.  Atoms arrive mostly in cell order (the previous sort), so the
// lanes of a wavefront form runs of equal buckets: each run takes its ranks
// with one atomic add of its length.  Ranks only need to be distinct; k_fixup
// orders every bucket by previous position.
// Bucket of an atom within its instance (not a padding slot): its cell, or the
// last two buckets for atoms outside every list and removed ones.
__device__ __forceinline__ int bucket_of(const double4 &x, const DInst &in, DCtl &ctl) {
  if (meta_of(x) & META_DEAD) return in.nbucket - 1;
  if (!(isfinite(x.x) && isfinite(x.y) && isfinite(x.z))) {
    atomicOr(&ctl.nonfinite, 1);
    return in.nbucket - 1;
  }
  const int c0 = ref_cell(x.x, in.ilb[0], in.lb[0], in.h[0]);
  const int c1 = ref_cell(x.y, in.ilb[1], in.lb[1], in.h[1]);
  const int c2 = ref_cell(x.z, in.ilb[2], in.lb[2], in.h[2]);
  // Cell N+1 with N > 2 is overwritten by the periodic halo copy of
  // chainlist (nlist.f90:53-64): such atoms drop out of every list.
  const bool drop = (c0 == in.nc[0] + 1 && in.nc[0] > 2) ||
                    (c1 == in.nc[1] + 1 && in.nc[1] > 2) ||
                    (c2 == in.nc[2] + 1 && in.nc[2] > 2) || c0 < 1 || c1 < 1 || c2 < 1 ||
                    c0 > in.nc[0] + 1 || c1 > in.nc[1] + 1 || c2 > in.nc[2] + 1;
  if (drop) return in.nbucket - 2;
  return ((c2 - 1) * in.next[1] + (c1 - 1)) * in.next[0] + (c0 - 1);
}
// whether that bucket is a cell of the grid, whose atoms k_nbuild gives a row
__device__ __forceinline__ bool bucket_is_cell(int local, const DInst &in) {
  if (local >= in.nbucket - 2) return false;
  return local % in.next[0] < in.nc[0] && (local / in.next[0]) % in.next[1] < in.nc[1] &&
         local / (in.next[0] * in.next[1]) < in.nc[2];
}

__global__ void k_bin(const double4 *__restrict__ X, int NA, const DInst *__restrict__ I,
                      int *__restrict__ bkey, int *__restrict__ brank, int *__restrict__ bcnt,
                      DCtl *__restrict__ ctl, const int *__restrict__ binst,
                      const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  const int lane = threadIdx.x % FIB_WAVE;
  const uint64_t le = (lane == FIB_WAVE - 1) ? ~0ull : ((2ull << lane) - 1ull);  // lanes <= me
  // NA and the grid stride are multiples of the wavefront: the lanes of a
  // wavefront run the loop together
  GRID_STRIDE(p, NA) {
    // atoms of instances that are not rebuilt keep no key (k_scatter skips
    // the same blocks)
    if (block_gated_out(gate, binst, p)) continue;
    const double4 x = X[p];
    const uint32_t m = meta_of(x);
    int b = -1;
    if (!(m & META_PAD)) {
      const DInst &in = I[inst_of(m)];
      b = in.bucket_off + bucket_of(x, in, ctl[inst_of(m)]);
    }
    // runs of equal buckets among the lanes; skipped lanes (-1) join none
    const int prev = __shfl_up(b, 1);
    const bool start = lane == 0 || prev != b || b < 0;
    const uint64_t starts = __ballot(start);
    const int lead = 63 - __clzll(starts & le);
    int base = 0;
    if (start && b >= 0) {
      const uint64_t later = starts & ~le;
      const int end = later ? __ffsll((unsigned long long)later) - 1 : FIB_WAVE;
      base = atomicAdd(&bcnt[b], end - lane);
    }
    base = __shfl(base, lead);
    bkey[p] = b;
    if (b >= 0) brank[p] = base + (lane - lead);
  }
}

// Export of the reference cell ids in original atom order.
__global__ void k_cellid(const double4 *__restrict__ X, int NA, const DInst *__restrict__ I,
                         int inst, int32_t *__restrict__ out) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= NA) return;
  double4 x = X[p];
  uint32_t m = meta_of(x);
  if ((m & META_PAD) || inst_of(m) != inst) return;
  const DInst &in = I[inst];
  int o = orig_of(x);
  out[o] = ref_cell(x.x, in.ilb[0], in.lb[0], in.h[0]);
  out[in.natm + o] = ref_cell(x.y, in.ilb[1], in.lb[1], in.h[1]);
  out[2 * in.natm + o] = ref_cell(x.z, in.ilb[2], in.lb[2], in.h[2]);
}

// ---------------------------------------------------------------------------
// exclusive scan (2 phases), chunk = 256 threads x 8 elements
#define SCAN_T 256
#define SCAN_E 8
#define SCAN_CH (SCAN_T * SCAN_E)

__device__ __forceinline__ int block_scan_excl(int v, int &total) {
  __shared__ int ws[SCAN_T / FIB_WAVE];
  const int lane = threadIdx.x % FIB_WAVE, wid = threadIdx.x / FIB_WAVE;
  int x = v;
  for (int o = 1; o < FIB_WAVE; o <<= 1) {
    int y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == FIB_WAVE - 1) ws[wid] = x;
  __syncthreads();
  int off = 0, tot = 0;
  for (int w = 0; w < SCAN_T / FIB_WAVE; ++w) {
    if (w < wid) off += ws[w];
    tot += ws[w];
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

__global__ void k_scan_reduce(const int *__restrict__ in, int n, int *__restrict__ bsum,
                              const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  int base = blockIdx.x * SCAN_CH;
  int s = 0;
  for (int e = 0; e < SCAN_E; ++e) {
    int idx = base + e * SCAN_T + threadIdx.x;
    if (idx < n) s += in[idx];
  }
  int tot;
  block_scan_excl(s, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// out[b] = exclusive prefix over all buckets, out[n] = total: every block
// adds up the totals of the blocks before it, or (SCANNED) finds them added
// up, where there are too many (see scan_top).  A bucket's atoms start at
// out[b] - out[first bucket of its instance] + atom_off, whatever other
// instances hold, so an instance can be sorted while the others stay in
// place (bucket_base).
template <bool SCANNED>
__global__ void k_scan_down(const int *__restrict__ in, int n, const int *__restrict__ bsum,
                            int *__restrict__ out, const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  int carry;
  if (SCANNED) {
    carry = bsum[blockIdx.x];
  } else {
    int before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += SCAN_T) before += bsum[k];
    block_scan_excl(before, carry);
  }
  const int base = blockIdx.x * SCAN_CH + threadIdx.x * SCAN_E;
  int vals[SCAN_E];
  int s = 0;
  for (int e = 0; e < SCAN_E; ++e) {
    const int idx = base + e;
    vals[e] = idx < n ? in[idx] : 0;
    s += vals[e];
  }
  int tot;
  int ex = block_scan_excl(s, tot) + carry;
  for (int e = 0; e < SCAN_E; ++e) {
    const int idx = base + e;
    if (idx <= n) out[idx] = ex;
    ex += vals[e];
  }
}
// Sorted position = cstart[b] + bucket_base for the buckets b of `in`.
__device__ __forceinline__ int bucket_base(const int *__restrict__ cstart, const DInst &in) {
  return in.atom_off - cstart[in.bucket_off];
}

// (and the histogram cleared for the next build: its counts are the
// differences of cstart from here on)
__global__ void k_scatter(const int *__restrict__ bkey, const int *__restrict__ brank, int NA,
                          const DInst *__restrict__ I, const int *__restrict__ cstart,
                          int *__restrict__ perm, int *__restrict__ bcnt, int nb,
                          const int *__restrict__ binst, const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  GRID_STRIDE(b, nb) bcnt[b] = 0;
  GRID_STRIDE(p, NA) {
    if (block_gated_out(gate, binst, p)) continue;
    const DInst &in = I[__builtin_amdgcn_readfirstlane(binst[p / FIB_BLOCK])];
    const int b = bkey[p];
    if (b >= 0) perm[cstart[b] + bucket_base(cstart, in) + brank[p]] = p;
  }
}

// Deterministic order inside a bucket: ascending previous position.
template <typename T>
__device__ __forceinline__ void sort_ascending(T *a, int n) {
  for (int i = 1; i < n; ++i) {
    const T v = a[i];
    int j = i - 1;
    while (j >= 0 && a[j] > v) { a[j + 1] = a[j]; --j; }
    a[j + 1] = v;
  }
}
__global__ void k_fixup(const int *__restrict__ cstart, int nb, const DInst *__restrict__ I,
                        int ninst, int *__restrict__ perm, const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  GRID_STRIDE(b, nb) {
    const int n = cstart[b + 1] - cstart[b];
    if (n < 2) continue;
    const DInst &in = I[find_inst_by_bucket(I, ninst, b)];
    sort_ascending(perm + cstart[b] + bucket_base(cstart, in), n);
  }
}

// The whole sort of a small instance (at most SORT_N atoms and buckets) by
// one workgroup in LDS: binning, histogram, scan, scatter and the order
// inside the buckets: one launch of 9 us (4 k atoms) for the general sort's
// five of about 5 us, and one instead of five when the build is gated off.
#define SORT_T 1024
#define SORT_N FIB_SORT_N
__global__ __launch_bounds__(SORT_T) void k_sort_small(
    const double4 *__restrict__ X, const DInst *__restrict__ I, int *__restrict__ bkey,
    int *__restrict__ cstart, int *__restrict__ perm, DCtl *__restrict__ ctl,
    const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  const int inst = blockIdx.x, t = threadIdx.x;
  if (gated_out(gate, inst)) return;
  constexpr int E = SORT_N / SORT_T;
  __shared__ int cnt[SORT_N + 1];
  __shared__ uint16_t lp[SORT_N];
  __shared__ int ws[SORT_T / FIB_WAVE];
  const DInst &in = I[inst];
  const int n = in.natm_pad, nb = in.nbucket;
  for (int b = t; b <= nb; b += SORT_T) cnt[b] = 0;
  __syncthreads();
  int key[E], rank[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = e * SORT_T + t;
    key[e] = -1;
    if (q < n) {
      const double4 x = X[in.atom_off + q];
      if (!(meta_of(x) & META_PAD)) {
        key[e] = bucket_of(x, in, ctl[inst]);
        rank[e] = atomicAdd(&cnt[key[e]], 1);
      }
      bkey[in.atom_off + q] = key[e] < 0 ? -1 : in.bucket_off + key[e];
    }
  }
  __syncthreads();
  // exclusive scan of the counts, E consecutive buckets per thread
  int v[E], s = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int b = t * E + e;
    v[e] = b < nb ? cnt[b] : 0;
    s += v[e];
  }
  const int lane = t % FIB_WAVE, wid = t / FIB_WAVE;
  int inc = s;
  for (int o = 1; o < FIB_WAVE; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (lane >= o) inc += y;
  }
  if (lane == FIB_WAVE - 1) ws[wid] = inc;
  __syncthreads();
  int ex = inc - s;
  for (int w = 0; w < wid; ++w) ex += ws[w];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int b = t * E + e;
    if (b < nb) {
      cnt[b] = ex;
      cstart[in.bucket_off + b] = in.atom_off + ex;
      ex += v[e];
      if (b == nb - 1) cnt[nb] = ex;
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (key[e] >= 0) lp[cnt[key[e]] + rank[e]] = (uint16_t)(e * SORT_T + t);
  __syncthreads();
  for (int b = t; b < nb; b += SORT_T) sort_ascending(lp + cnt[b], cnt[b + 1] - cnt[b]);
  __syncthreads();
  const int total = cnt[nb];
  for (int q = t; q < total; q += SORT_T) perm[in.atom_off + q] = in.atom_off + (int)lp[q];
}

// Every per-atom array into the new order, and what a build resets: the
// positions of the build (Xb), displacements, near lists, the lists of atoms
// outside every cell (k_nbuild writes the others), and the instance's record.
__global__ void k_reorder(int NA, const int *__restrict__ perm, const int *__restrict__ bkey,
                          const DInst *__restrict__ I, const double4 *__restrict__ X0,
                          double4 *__restrict__ X1, const double *__restrict__ V0,
                          double *__restrict__ V1, const double *__restrict__ F0,
                          double *__restrict__ F1, const double *__restrict__ Xi0,
                          double *__restrict__ Xi1, int *__restrict__ inv,
                          double4 *__restrict__ Xb, float *__restrict__ disp,
                          uint8_t *__restrict__ nst, int *__restrict__ cnt_sw,
                          int *__restrict__ cnt_ion, uint8_t *__restrict__ off_sw,
                          DCtl *__restrict__ ctl, const int *__restrict__ binst,
                          const int *__restrict__ gate) {
  GATE_OR_RETURN(gate);
  GRID_STRIDE(p, NA) {
    if (block_gated_out(gate, binst, p)) continue;
    const int inst = __builtin_amdgcn_readfirstlane(binst[p / FIB_BLOCK]);
    const DInst &in = I[inst];
    if (p == in.atom_off) {
      DCtl &c = ctl[inst];
      c.maxdisp = 0.0;
      c.maxdisp2 = 0.0;
      c.nmaxdisp = 0.0;
      c.maxcnt_sw = 0.0;
      c.maxcnt_ion = 0.0;
      c.near_off = 0;
      c.extra_any = 0;
      c.builds += 1.0;
    }
    if (meta_of(X0[p]) & META_PAD) {
      if (nst) nst[p] = 0;
      continue;
    }
    const int s = perm[p];
    const double4 x = X0[s];
    X1[p] = x;
    for (int c = 0; c < 3; ++c) {
      const size_t a = (size_t)c * NA;
      V1[a + p] = V0[a + s];
      if (F0) F1[a + p] = F0[a + s];
      Xi1[a + p] = Xi0[a + s];
    }
    inv[in.atom_off + orig_of(x)] = p;
    Xb[p] = x;
    disp[p] = 0.0f;
    if (nst) nst[p] = NEAR_FRESH;
    if (!bucket_is_cell(bkey[s] - in.bucket_off, in)) {
      cnt_sw[p] = 0;
      cnt_ion[p] = 0;
      // no row: offsets past any row (see k_force3)
      uint4 *o = reinterpret_cast<uint4 *>(off_sw + (size_t)p * OFF_W);
      o[0] = make_uint4(~0u, ~0u, ~0u, ~0u);
      o[1] = make_uint4(~0u, ~0u, ~0u, ~0u);
    }
  }
}

// In-place variant of the sort: the reordered arrays copied back, so they
// stay where a captured step expects them.  k_nbuild reads the reordered
// positions, so extra workgroups of its launch do this beside the build.
struct CopyBack {
  int blocks;  // workgroups of FIB_BLOCK threads (0: none)
  const double4 *X1;
  double4 *X0;
  const double *V1, *Xi1;
  double *V0, *Xi0;
  const int *binst;
  int NA;
};
__device__ __forceinline__ void copy_back(const CopyBack &cb, int block,
                                          const int *__restrict__ gate) {
  for (int p = block * FIB_BLOCK + threadIdx.x; p < cb.NA; p += cb.blocks * FIB_BLOCK) {
    if (block_gated_out(gate, cb.binst, p)) continue;
    cb.X0[p] = cb.X1[p];
    for (int c = 0; c < 3; ++c) {
      const size_t a = (size_t)c * cb.NA + p;
      cb.V0[a] = cb.V1[a];
      cb.Xi0[a] = cb.Xi1[a];
    }
  }
}

// ---------------------------------------------------------------------------
// neighbour build: one 64-lane block per real cell
#define NB_CHUNK 128
#define NB_XS 4      // log2 of the workgroups that an XCD takes in a row
#define NB_CAND 192   // candidates that a cell's fast build takes
#define NB_ACC 384  // candidates whose acceptance masks are kept for the ranks
#ifndef NB_WAVES
#define NB_WAVES 4  // independent wavefronts per k_nbuild workgroup
#endif
// A row entry of rk_sw holds (stencil cell << 8 | rank) as the build wrote
// it, or, once a force pass has worked it out, RK_SLOT | the slot of the
// row's atom in the neighbour's row (values >= the list width, at most 127,
// mark a neighbour without a row or with the atom past its end).
#define RK_SLOT 0x8000
#define NB_JBITS 27  // atom index bits beside the stencil cell in a staged w (fib_create keeps NA below)

// Stencil bookkeeping for the force gather.  The list row of an atom is the
// concatenation, in the fixed order s = 0..26 of the 27-cell stencil, of the
// accepted atoms of each stencil cell in cell order.  For every atom the
// build stores off[s] = row position where stencil cell s starts (255 for an
// atom without a row), and for every row entry (i -> j) the stencil index s
// of j's cell and the rank of i among the atoms of i's cell that j accepts.
// Stencil offsets are symmetric (cell 26 - s seen from j) and so is the pair
// predicate, so the position of i in j's row is off_j[26 - s] + rank -- no
// search of j's row is needed.  The rank is counted from the acceptance
// masks of the cell's earlier atoms: j accepts a exactly when a accepted j.
//
// Neighbour cell index along one axis (d in {-1, 0, 1}): N > 2 wraps
// periodically ((c + d + N) mod N with one add or subtract); N <= 2 does not
// wrap and index N is the phantom layer holding atoms whose cell id came out
// as N+1; a stencil cell outside [0, N] does not exist.
__device__ __forceinline__ int stencil_axis(int c, int d, int n, bool &ok) {
  int v = c + d;
  if (n > 2) {
    v = v < 0 ? v + n : (v >= n ? v - n : v);
  } else if (v < 0 || v > n) {
    ok = false;
  }
  return v;
}

// v of another lane (uniform), through scalar registers
__device__ __forceinline__ float bcast(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double bcast(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ int mbcnt(uint64_t m) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// One cell whose halo fits two candidates per lane (all but very dense ones).
// The build is bound by vector instructions, so the work that does not
// depend on the atom is done once per cell:
//  - the periodic shift k L of every candidate, from its difference to the
//    cell's first atom (the reference's NINT gives the same k for every atom
//    of the cell when no difference comes near half a box: checked);
//  - candidates farther than the cutoff from the box around the cell's atoms
//    are dropped (FP32 with a margin; of ~105 about 60 stay), the others
//    compacted in order, so most cells test one candidate per lane.
// The candidates then stay in registers, the atom's position comes through
// scalar registers, and the reference's predicate is evaluated as ref_r2
// does, without contraction.  False (nothing written) when a difference is
// too close to half a box, as in boxes of few cells.
// 2.1 M atoms (whole build): 720 -> 523 vector instructions a cell, 871 ->
// 651 us (four waves per SIMD; asked for five or six it spills and takes
// longer than before).
template <int NT>
__device__ __forceinline__ bool nbuild_cell_fast(
    const double4 *__restrict__ X, const DInst &in, int i0, int ni, int rs, int rc, int my_lo,
    int total, const uint64_t (&lm)[NT], double rv2, double rv2lj, int Wsw, int Wion,
    int &most_sw, int &most_ion, int *__restrict__ cnt_sw, int *__restrict__ nbr_sw, int *__restrict__ cnt_ion,
    int *__restrict__ nbr_ion, uint16_t *__restrict__ rk_sw, uint8_t *__restrict__ off_sw,
    double4 *s_x, int *s_j) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x % FIB_WAVE;
  constexpr bool NBNT = (FIB_NT_ST & 16) != 0;
  constexpr uint32_t JM = (1u << NB_JBITS) - 1u;
  // each stencil lane writes its own run of candidates, stencil cell above
  for (int q = 0; __ballot(q < rc) != 0ull; ++q)
    if (q < rc) s_j[my_lo + q] = (int)((uint32_t)lane << NB_JBITS | (uint32_t)(rs + q));
  wave_lds_sync();
  const double4 own = X[i0 + min(lane, ni - 1)];
  const int town = type_of(meta_of(own));
  const double c[3] = {bcast(own.x, 0), bcast(own.y, 0), bcast(own.z, 0)};
  const float own0[3] = {(float)(own.x - c[0]), (float)(own.y - c[1]), (float)(own.z - c[2])};
  float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  for (int ii = 1; ii < ni; ++ii) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float r = bcast(own0[a], ii);
      lo[a] = fminf(lo[a], r);
      hi[a] = fmaxf(hi[a], r);
    }
  }
  // candidates kept, and (lane s) those of them before stencil cell s
  int nk = 0, klo = 0;
  bool ions = false, wraps = false;
  if constexpr (NT == 2) {
    // differences to the cell's first atom
    const bool two = total > FIB_WAVE;
    uint32_t up[2];
    double4 x[2];
    double e0[2][3];
    bool have[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      have[t] = t * FIB_WAVE + lane < total;
      up[t] = have[t] ? (uint32_t)s_j[t * FIB_WAVE + lane] : ~0u;
      if (t == 0 || two) x[t] = X[have[t] ? (int)(up[t] & JM) : i0];
    }
    int far[3] = {0, 0, 0};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (t == 1 && !two) x[1] = x[0];
      e0[t][0] = c[0] - x[t].x;
      e0[t][1] = c[1] - x[t].y;
      e0[t][2] = c[2] - x[t].z;
#pragma unroll
      for (int a = 0; a < 3; ++a) far[a] = max(far[a], __double2hiint(e0[t][a]) & 0x7fffffff);
    }
    // all of them below 0.12 of the box (by the upper words): then every
    // difference from an atom of the cell is below 0.24 and no shift is wanted
    bool any = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) any = any || far[a] >= __double2hiint(0.12 * in.lb[a]);
    wraps = __ballot(any) != 0ull;
    uint32_t code[2] = {0x150u, 0x150u};
    if (wraps) {
      bool bad = false;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bool mine = (up[t] >> NB_JBITS) == 13u;
        code[t] = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double k = rint(e0[t][a] * in.ilb[a]);
          const double e = e0[t][a] - k * in.lb[a];
          e0[t][a] = e;
          // shifts 0 and +-1 are coded 1, 2, 0
          code[t] |= (uint32_t)((int)k + 1) << (4 + 2 * a);
          bad = bad || (have[t] && (fabs(k) > 1.0 || fabs(e) > 0.49 * in.lb[a] - 1.001 * in.h[a] ||
                                    (mine && (k != 0.0 || fabs(e) > 1.001 * in.h[a]))));
        }
      }
      if (__ballot(bad) != 0ull) return false;
    }
    float d2[2];
    bool ion = town == 3;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float sum = 0.0f;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float r = (float)-e0[t][a];
        const float d = fmaxf(fmaxf(lo[a] - r, r - hi[a]), 0.0f);
        sum += d * d;
      }
      const uint32_t ty = meta_of(x[t]) & META_TYPE_MASK;
      ion = ion || ty == 3u;
      x[t].w = __longlong_as_double((long long)((uint64_t)up[t] << 32 | (uint64_t)(code[t] | ty)));
      d2[t] = have[t] ? sum : 3.0e38f;
    }
    // without a Ga atom around, only pairs within the SW list radius are wanted
    ions = __ballot(ion) != 0ull;
    const float r2max = (float)(ions ? fmax(rv2, rv2lj) : rv2) * 1.0001f;
    const uint64_t k0 = __ballot(d2[0] <= r2max), k1 = __ballot(d2[1] <= r2max);
    const int n0 = __popcll(k0);
    nk = n0 + __popcll(k1);
    if (d2[0] <= r2max) s_x[mbcnt(k0)] = x[0];
    if (d2[1] <= r2max) s_x[n0 + mbcnt(k1)] = x[1];
    klo = __popcll(k0 & lm[0]) + __popcll(k1 & lm[1]);
  } else {
    // a batch at a time: the registers do not hold three at once
    const bool last = total > (NT - 1) * FIB_WAVE;  // the last NT-th is wanted
    uint32_t up[NT];
    double4 x[NT];
    bool ion = town == 3;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bool have = t * FIB_WAVE + lane < total;
      up[t] = have ? (uint32_t)s_j[t * FIB_WAVE + lane] : ~0u;
      if (t < NT - 1 || last) x[t] = X[have ? (int)(up[t] & JM) : i0];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (t == NT - 1 && !last) x[t] = x[0];
      ion = ion || type_of(meta_of(x[t])) == 3;
    }
    // without a Ga atom around, only pairs within the SW list radius are wanted
    ions = __ballot(ion) != 0ull;
    const float r2max = (float)(ions ? fmax(rv2, rv2lj) : rv2) * 1.0001f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bool have = t * FIB_WAVE + lane < total;
      // differences to the cell's first atom
      double e0[3] = {c[0] - x[t].x, c[1] - x[t].y, c[2] - x[t].z};
      // all of them below 0.12 of the box (by the upper words): then every
      // difference from an atom of the cell is below 0.24 and no shift is wanted
      bool any = false;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        any = any || (__double2hiint(e0[a]) & 0x7fffffff) >= __double2hiint(0.12 * in.lb[a]);
      uint32_t code = 0x150u;
      if (__ballot(any) != 0ull) {
        wraps = true;
        const bool mine = (up[t] >> NB_JBITS) == 13u;
        bool bad = false;
        code = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double k = rint(e0[a] * in.ilb[a]);
          const double e = e0[a] - k * in.lb[a];
          e0[a] = e;
          // shifts 0 and +-1 are coded 1, 2, 0
          code |= (uint32_t)((int)k + 1) << (4 + 2 * a);
          bad = bad || (have && (fabs(k) > 1.0 || fabs(e) > 0.49 * in.lb[a] - 1.001 * in.h[a] ||
                                 (mine && (k != 0.0 || fabs(e) > 1.001 * in.h[a]))));
        }
        if (__ballot(bad) != 0ull) return false;
      }
      float d2 = 0.0f;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float r = (float)-e0[a];
        const float d = fmaxf(fmaxf(lo[a] - r, r - hi[a]), 0.0f);
        d2 += d * d;
      }
      const bool keep = have && d2 <= r2max;
      const uint64_t km = __ballot(keep);
      const int n = __popcll(km);
      if (NT > 2 && nk + n > NB_CHUNK) return false;
      x[t].w = __longlong_as_double(
          (long long)((uint64_t)up[t] << 32 | (uint64_t)(code | (meta_of(x[t]) & META_TYPE_MASK))));
      if (keep) s_x[nk + mbcnt(km)] = x[t];
      nk += n;
      klo += __popcll(km & lm[t]);
    }
  }
  wave_lds_sync();
  auto rows = [&](auto sets) {
    constexpr int NS = decltype(sets)::value;
    double y[NS][3];
    uint32_t u[NS], low[NS];
    uint64_t before_m[NS];
    int acc[NS];  // atoms of the cell so far that the candidate accepted
#pragma unroll
    for (int t = 0; t < NS; ++t) {
      const double4 v = s_x[t * FIB_WAVE + lane];  // (past nk: unused)
      y[t][0] = v.x; y[t][1] = v.y; y[t][2] = v.z;
      u[t] = (uint32_t)(wbits(v) >> 32);
      low[t] = (uint32_t)wbits(v);
      acc[t] = 0;
      const int cut = min(max(klo - t * FIB_WAVE, 0), FIB_WAVE);
      before_m[t] = cut >= FIB_WAVE ? ~0ull : ((1ull << cut) - 1ull);
    }
    for (int ii = 0; ii < ni; ++ii) {
      const int i = i0 + ii;
      int *const rowj = nbr_sw + (size_t)i * Wsw;
      uint16_t *const rowk = rk_sw + (size_t)i * Wsw;
      const double xi[3] = {bcast(own.x, ii), bcast(own.y, ii), bcast(own.z, ii)};
      int nsw = 0, nion = 0, before = 0;
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        const int j = (int)(u[t] & JM);
        double d[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) d[a] = xi[a] - y[t][a];
        if (wraps) {
#pragma unroll
          for (int a = 0; a < 3; ++a)
            d[a] = d[a] - (double)((int)(low[t] >> (4 + 2 * a) & 3u) - 1) * in.lb[a];
        }
        const double r2 = ref_sq(d[0], d[1], d[2]);
        const bool cand = t * FIB_WAVE + lane < nk && j != i;
        bool sw = cand && r2 < rv2;
        if (ions) {
          const int ti = __builtin_amdgcn_readlane(town, ii);
          const bool swp = max(ti, (int)(low[t] & META_TYPE_MASK)) < 3;
          const bool io = cand && !swp && r2 < rv2lj;
          sw = sw && swp;
          const uint64_t mio = __ballot(io);
          const int pos = nion + mbcnt(mio);
          if (io && pos < Wion) st_nt<NBNT>(nbr_ion + (size_t)i * Wion + pos, j);
          nion += __popcll(mio);
        }
        const uint64_t msw = __ballot(sw);
        const int pos = nsw + mbcnt(msw);
        if (sw && pos < Wsw) {
          st_nt<NBNT>(rowj + pos, j);
          st_nt<NBNT>(rowk + pos, (uint16_t)((u[t] >> NB_JBITS) << 8 | (uint32_t)acc[t]));
        }
        acc[t] += sw ? 1 : 0;
        before += __popcll(msw & before_m[t]);
        nsw += __popcll(msw);
      }
      if (lane < 27) st_nt<NBNT>(off_sw + (size_t)i * OFF_W + lane, (uint8_t)min(before, 254));
      if (lane == 0) {
        st_nt<NBNT>(cnt_sw + i, nsw);
        st_nt<NBNT>(cnt_ion + i, nion);
      }
      most_sw = max(most_sw, nsw);
      most_ion = max(most_ion, nion);
    }
  };
  if (nk <= FIB_WAVE) rows(std::integral_constant<int, 1>{});
  else rows(std::integral_constant<int, 2>{});
  return true;
}

// One cell (cx, cy, cz) of instance `in`, built by one wave.
template <bool WIDE>
__device__ __forceinline__ void nbuild_cell(
    const double4 *__restrict__ X, const DInst &in, int cx, int cy, int cz, int sd0, int sd1,
    int sd2, const int *__restrict__ cstart, int base, double rv2, double rv2lj, int Wsw, int Wion,
    int &most_sw, int &most_ion, int *__restrict__ cnt_sw, int *__restrict__ nbr_sw,
    int *__restrict__ cnt_ion, int *__restrict__ nbr_ion, uint16_t *__restrict__ rk_sw,
    uint8_t *__restrict__ off_sw, double4 *s_x, int *s_j, uint8_t *s_st, int *s_rs, int *s_off,
    uint32_t *s_acc) {
  const int lane = threadIdx.x % FIB_WAVE;
  constexpr bool NBNT = (FIB_NT_ST & 16) != 0;
  // the previous cell of this wave is done with the shared arrays
  wave_lds_sync();
  const int bi = in.bucket_off + (cz * in.next[1] + cy) * in.next[0] + cx;
  const int c0 = cstart[bi], ni = cstart[bi + 1] - c0, i0 = c0 + base;
  if (ni == 0) return;

  // lane s < 27 owns stencil cell s = (sd0, sd1, sd2) + 1 in base 3
  int rs = 0, rc = 0;
  if (lane < 27) {
    bool ok = true;
    const int e0 = stencil_axis(cx, sd0, in.nc[0], ok);
    const int e1 = stencil_axis(cy, sd1, in.nc[1], ok);
    const int e2 = stencil_axis(cz, sd2, in.nc[2], ok);
    if (ok) {
      const int b = in.bucket_off + (e2 * in.next[1] + e1) * in.next[0] + e0;
      rs = cstart[b];
      rc = cstart[b + 1] - rs;
      rs += base;
    }
  }
  // inclusive scan of rc over lanes 0..31 (the stencil lanes)
  int sc = rc;
  for (int o = 1; o < 32; o <<= 1) {
    int y = __shfl_up(sc, o);
    if (lane >= o) sc += y;
  }
  const int total = __builtin_amdgcn_readfirstlane(__shfl(sc, 26));
  // stencil cell s covers candidates [my_lo, my_lo + rc)
  const int my_lo = sc - rc;
  // the candidates of a 64-batch starting at b that lie before stencil cell
  // s, as a lane mask (lane s); the one-chunk cell has batches 0 and 64 only
  auto before_mask = [&](int b) -> uint64_t {
    const int cut = min(max(my_lo - b, 0), 64);
    return cut >= 64 ? ~0ull : ((1ull << cut) - 1ull);
  };
  if (total <= NB_CHUNK && ni <= 32) {
    const uint64_t lm[2] = {before_mask(0), before_mask(FIB_WAVE)};
    if (nbuild_cell_fast<2>(X, in, i0, ni, rs, rc, my_lo, total, lm, rv2, rv2lj, Wsw, Wion,
                            most_sw, most_ion, cnt_sw, nbr_sw, cnt_ion, nbr_ion, rk_sw, off_sw,
                            s_x, s_j))
      return;
  } else if (WIDE && total <= NB_CAND && ni <= 32) {
    const uint64_t lm[3] = {before_mask(0), before_mask(FIB_WAVE), before_mask(2 * FIB_WAVE)};
    if (nbuild_cell_fast<3>(X, in, i0, ni, rs, rc, my_lo, total, lm, rv2, rv2lj, Wsw, Wion,
                            most_sw, most_ion, cnt_sw, nbr_sw, cnt_ion, nbr_ion, rk_sw, off_sw,
                            s_x, s_j))
      return;
  }
  const bool masks = total <= NB_ACC && ni <= 32;
  if (masks)
    for (int g = lane; g < total; g += FIB_WAVE) s_acc[g] = 0;
  const bool one_chunk = total <= NB_CHUNK;
  const uint64_t lm0 = before_mask(0), lm1 = before_mask(FIB_WAVE);
  if (one_chunk) {
    // each stencil lane writes its own run of candidates
    for (int q = 0; __ballot(q < rc) != 0ull; ++q)
      if (q < rc) {
        s_j[my_lo + q] = rs + q;
        s_st[my_lo + q] = (uint8_t)lane;
      }
  } else {
    if (lane < 27) { s_rs[lane] = rs; s_off[lane + 1] = sc; }
    if (lane == 0) s_off[0] = 0;
  }
  wave_lds_sync();

  const double4 *Xc = X;
  // the cell's own atoms are stencil range 13: read them from the staged
  // chunk when it holds them (always, unless the halo is very dense)
  const int own0 = __builtin_amdgcn_readfirstlane(__shfl(my_lo, 13));
  const bool own_staged = one_chunk;
  const double qb0 = 0.25 * in.lb[0], qb1 = 0.25 * in.lb[1], qb2 = 0.25 * in.lb[2];
  for (int ii = 0; ii < ni; ++ii) {
    const int i = i0 + ii;
    int *const rowj = nbr_sw + (size_t)i * Wsw;
    uint16_t *const rowk = rk_sw + (size_t)i * Wsw;
    int *const rowi = nbr_ion + (size_t)i * Wion;
    int nsw = 0, nion = 0;
    int before = 0;  // lane s: accepted candidates before stencil cell s
    double4 xi;
    int ti = 0;
    for (int base = 0; base < total; base += NB_CHUNK) {
      const int n = min(NB_CHUNK, total - base);
      // (re)stage the chunk; a single chunk is loaded once per cell
      if (ii == 0 || !one_chunk) {
        if (!one_chunk) {
          wave_lds_sync();
          for (int q = lane; q < n; q += FIB_WAVE) {
            const int g = base + q;
            // stencil range holding g: binary search over the 28 offsets
            int lo = 0, hi = 26;
            while (lo < hi) {
              const int mid = (lo + hi + 1) >> 1;
              if (s_off[mid] <= g) lo = mid; else hi = mid - 1;
            }
            s_j[q] = s_rs[lo] + (g - s_off[lo]);
            s_st[q] = (uint8_t)lo;
          }
          wave_lds_sync();
        }
        // the staged copy carries the candidate's index and stencil cell in
        // the upper word of w (the original index, which the build does not
        // use): one 32-byte read per candidate in the batches below
        for (int q = lane; q < n; q += FIB_WAVE) {
          const int j = s_j[q];
          double4 x = Xc[j];
          const uint64_t up = ((uint64_t)s_st[q] << NB_JBITS) | (uint64_t)j;
          x.w = __longlong_as_double((long long)((up << 32) | (uint64_t)meta_of(x)));
          s_x[q] = x;
        }
        wave_lds_sync();
      }
      if (base == 0) {
        xi = own_staged ? s_x[own0 + ii] : Xc[i];
        ti = type_of(meta_of(xi));
      }
      for (int q0 = 0; q0 < n; q0 += FIB_WAVE) {
        const int q = q0 + lane;  // < NB_CHUNK: the stage arrays are read unguarded
        const int g = base + q;
        const double4 xj = s_x[q];
        const uint32_t up = (uint32_t)(wbits(xj) >> 32);
        const int j = (int)(up & ((1u << NB_JBITS) - 1u));
        const int st = (int)(up >> NB_JBITS);
        const bool cand = q < n && j != i;
        double d0, d1, d2;
        ref_diff(xi, xj, d0, d1, d2);
        const bool far = cand && !(fabs(d0) < qb0 && fabs(d1) < qb1 && fabs(d2) < qb2);
        // With every difference of the batch under a quarter box, the
        // reference's NINT shifts are all zero: r^2 is the plain sum
        // (bit-identical); otherwise the full minimum image
        double r2;
        if (__ballot(far) == 0ull) r2 = ref_sq(d0, d1, d2);
        else r2 = ref_r2(xi, xj, in);
        const bool swp = max(ti, type_of(meta_of(xj))) < 3;
        const bool sw = cand && swp && r2 < rv2;
        const bool io = cand && !swp && r2 < rv2lj;
        uint64_t msw = __ballot(sw), mio = __ballot(io);
        if (sw) {
          // rank of i among the atoms of its cell that j lists (in cell order)
          int rank = 0;
          if (masks) {
            const uint32_t acc = s_acc[g];
            rank = __popc(acc & ((ii == 0) ? 0u : (~0u >> (32 - ii))));
            s_acc[g] = acc | (1u << ii);
          } else {
            for (int a = 0; a < ii; ++a) {
              const int ia = i0 + a;
              if (ia == j) continue;
              const double4 xa = Xc[ia];
              if (type_of(meta_of(xa)) < 3 && ref_r2(xj, xa, in) < rv2) ++rank;
            }
          }
          const int pos = nsw + (int)__builtin_amdgcn_mbcnt_hi(
                                    (uint32_t)(msw >> 32),
                                    __builtin_amdgcn_mbcnt_lo((uint32_t)msw, 0u));
          if (pos < Wsw) {
            st_nt<NBNT>(rowj + pos, j);
            st_nt<NBNT>(rowk + pos, (uint16_t)((st << 8) | (rank & 0xff)));
          }
        }
        if (mio) {
          if (io) {
            const int pos = nion + (int)__builtin_amdgcn_mbcnt_hi(
                                       (uint32_t)(mio >> 32),
                                       __builtin_amdgcn_mbcnt_lo((uint32_t)mio, 0u));
            if (pos < Wion) st_nt<NBNT>(rowi + pos, j);
          }
        }
        // stencil cell s starts at candidate my_lo: count the accepted ones
        // of this batch of 64 candidates that lie before it
        {
          const int b = base + q0;
          const uint64_t lm = b == 0 ? lm0 : (b == FIB_WAVE ? lm1 : before_mask(b));
          before += __popcll(msw & lm);
        }
        nsw += __popcll(msw);
        nion += __popcll(mio);
      }
    }
    if (lane < 27) st_nt<NBNT>(off_sw + (size_t)i * OFF_W + lane, (uint8_t)min(before, 254));
    if (lane == 0) {
      st_nt<NBNT>(cnt_sw + i, nsw);
      st_nt<NBNT>(cnt_ion + i, nion);
    }
    most_sw = max(most_sw, nsw);
    most_ion = max(most_ion, nion);
  }
}

// Instance k and its first cell number in the build's numbering of cells:
// all real cells in instance order, or under a gate the real cells of the
// gated instances only (prefix cplan, gated-out instances have width 0).
__device__ __forceinline__ int locate_cell(const DInst *__restrict__ I, int ninst,
                                           const int *__restrict__ cplan, int c, int &first) {
  int lo = 0, hi = ninst - 1;
  if (cplan) {
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (cplan[mid] <= c) lo = mid; else hi = mid - 1;
    }
    first = cplan[lo];
  } else {
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (I[mid].cell_real_off <= c) lo = mid; else hi = mid - 1;
    }
    first = I[lo].cell_real_off;
  }
  return lo;
}

// Each wavefront builds NBC consecutive cells; a workgroup holds
// NB_WAVES independent wavefronts (their own LDS, wave-level sync only), so
// that the workgroup-per-CU limit does not cap the resident waves.  The cells
// to build are all real cells, or under a gate the cells of the gated
// instances, numbered by the prefix that k_md_decide writes after the gates;
// the grid covers all real cells and the workgroups past the gated ones leave
// at once (gated-out instances cost a launch of empty workgroups, no more).
// The busy workgroups are remapped so that each XCD builds runs of consecutive
// cells, whose halos then stay in its L2; short ones (2^NB_XS workgroups),
// because a slab's vacuum is empty cells: with an eighth of the box for each
// XCD, one of them builds a 40 x 40 x 12 slab under 540 A of vacuum alone
// (398 us, in runs of 16 workgroups 109; 2.1 M atoms without vacuum 728 and
// 742).  A wave decodes its first cell
// once and steps through the rest in x-fastest order.  A list longer than
// its width is cut; the longest goes to the instance's record, and in MD-step
// mode (under a gate) the rest of the step halts until the host has grown
// the lists and rebuilt them.
// SPARSE: most cells are empty, and a wavefront looks first whether all of its
// cells are (1,000 atoms in 89 million cells 11.4 -> 4.9 ms; a crystal has no
// such runs, and its builds took 1 % longer).
template <int NBC, bool WIDE, bool SPARSE>
__global__ __launch_bounds__(NB_WAVES * FIB_WAVE) __attribute__((amdgpu_waves_per_eu(4)))
void k_nbuild(
    const double4 *__restrict__ X, const DInst *__restrict__ I, int ninst, int total_cells,
    const int *__restrict__ cstart, double rv2, double rv2lj, int Wsw, int Wion,
    int *__restrict__ cnt_sw, int *__restrict__ nbr_sw, int *__restrict__ cnt_ion,
    int *__restrict__ nbr_ion, uint16_t *__restrict__ rk_sw, uint8_t *__restrict__ off_sw,
    DCtl *__restrict__ ctl, const int *__restrict__ gate, int *__restrict__ halt,
    const CopyBack cb) {
  GATE_OR_RETURN(gate);
  static_assert(NB_WAVES * FIB_WAVE == FIB_BLOCK, "copy_back's blocks");
  __shared__ double4 s_x[NB_WAVES][NB_CHUNK];
  __shared__ int s_j[NB_WAVES][WIDE ? NB_CAND : NB_CHUNK];
  __shared__ uint8_t s_st[NB_WAVES][NB_CHUNK];
  __shared__ int s_rs[NB_WAVES][27], s_off[NB_WAVES][28];
  __shared__ uint32_t s_acc[NB_WAVES][NB_ACC];
  if ((int)blockIdx.x < cb.blocks) {
    copy_back(cb, blockIdx.x, gate);
    return;
  }
  const int block = blockIdx.x - cb.blocks;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / FIB_WAVE);  // wave-uniform
  const int *cplan = gate ? gate + 1 + ninst : nullptr;
  const int ncell = gate ? cplan[ninst] : total_cells;
  constexpr int CPB = NB_WAVES * NBC;  // cells per workgroup
  const int nbusy = (ncell + CPB - 1) / CPB;
  if (block >= nbusy) return;
  const int c0 = xcd_remap(block, nbusy, NB_XS) * CPB + w * NBC;
  const int c1 = min(ncell, c0 + NBC);
  const int lane = threadIdx.x % FIB_WAVE;
  const int sd0 = lane % 3 - 1, sd1 = (lane / 3) % 3 - 1, sd2 = lane / 9 - 1;
  int cend = c0, k = 0, cx = 0, cy = 0, cz = 0, base = 0;
  for (int c = c0; c < c1; ++c) {
    if (c >= cend) {
      // first cell, or the first of the next instance
      int first;
      k = locate_cell(I, ninst, cplan, c, first);
      const DInst &in = I[k];
      const int loc = c - first;
      cx = loc % in.nc[0];
      cy = (loc / in.nc[0]) % in.nc[1];
      cz = loc / (in.nc[0] * in.nc[1]);
      cend = first + in.nc[0] * in.nc[1] * in.nc[2];
      if (SPARSE && in.next[0] == in.nc[0] && in.next[1] == in.nc[1]) {
        // the cells that this wavefront has of the instance are consecutive
        // buckets: none of them holds an atom
        const int last = min(c1, cend) - 1, b = in.bucket_off - first;
        if (cstart[b + c] == cstart[b + last + 1]) {
          c = last;
          continue;
        }
      }
      base = bucket_base(cstart, in);
    }
    const DInst &in = I[k];
    int most_sw = 0, most_ion = 0;
    nbuild_cell<WIDE>(X, in, cx, cy, cz, sd0, sd1, sd2, cstart, base, rv2, rv2lj, Wsw, Wion, most_sw,
                most_ion, cnt_sw, nbr_sw, cnt_ion, nbr_ion, rk_sw, off_sw, s_x[w], s_j[w],
                s_st[w], s_rs[w], s_off[w], s_acc[w]);
    if ((most_sw > Wsw || most_ion > Wion) && lane == 0) {
      // (positive doubles order as their bits)
      atomicMax(reinterpret_cast<unsigned long long *>(&ctl[k].maxcnt_sw),
                (unsigned long long)__double_as_longlong((double)most_sw));
      atomicMax(reinterpret_cast<unsigned long long *>(&ctl[k].maxcnt_ion),
                (unsigned long long)__double_as_longlong((double)most_ion));
      if (gate) {
        ctl[k].overflow = 1;
        if (halt) *halt = 1;
      }
    }
    if (++cx == in.nc[0]) {
      cx = 0;
      if (++cy == in.nc[1]) { cy = 0; ++cz; }
    }
  }
}

// Slot of the n-th set bit of m (n is small).
__device__ __forceinline__ int nth_bit(uint64_t m, int n) {
  for (int r = 0; r < n; ++r) m &= m - 1;
  return __ffsll((unsigned long long)m) - 1;
}

// ---------------------------------------------------------------------------
// Force evaluation in three passes, no atomics.
//
// k_legs (one thread per atom): the atom's buffered SW list, or its near list,
// is scanned once.  Pairs inside the pair-force range add the SW pair force
// (and the ion list the Moliere pairs) to the atom in registers.  Pairs inside
// the three-body range are the atom's "legs": a bit each in its leg mask, by
// list slot.  n counts an atom's legs in list-slot order; per-leg arrays are
// slot-major by it ([n * NA + i]).
//
// k_tri (one lane per leg): every vertex term centred on atom i,
// h(a, i, b) = leps E(r_a) E(r_b) (cos + 1/3)^2, is a pair of i's legs.  The
// lane owning leg a sums the force on a's atom over all partners b into
// G[n(a)][i] (w, where energies are wanted: a's third of the energy), and the
// legs of an atom sum to the reaction on it.  A wavefront takes the legs of 64
// atoms in turn (a prefix sum over the atoms' leg counts in LDS maps lanes to
// legs), so atoms with many legs do not stall the others.
//
// k_force3 (one thread per atom): F_i = own pair/Moliere force + the reaction
// on the centre + the G entries its neighbours wrote for it.  Neighbour c's entry for i is the leg of c in the list slot r that
// holds i; its compact index is the popcount of c's leg mask below r.  r
// follows from the stencil offsets the list build stores (see k_nbuild); k_tri
// works the index out per leg and leaves it in RA, so k_force3 makes one
// lookup per leg.  This turns the reference's scatter F(i) += fi, F(j) += fj,
// F(k) += fk (si.f90:544-546) into a gather.  MODE 1 applies the velocity
// update of onestep (timeint.f90:231-236), MODE 2 the MD-step second half kick.
template <bool MIXED>
struct Prec;
template <>
struct Prec<false> {
  typedef double T;
  typedef double4 T4;
};
template <>
struct Prec<true> {
  typedef float T;
  typedef float4 T4;
};

// Entry of G: the force a centre's terms put on one of its legs and, where
// energies are wanted, a share of them.
template <typename T>
struct Vec3 {
  T x, y, z;
};
template <bool MIXED, bool EN>
struct GRec {
  typedef Vec3<typename Prec<MIXED>::T> type;
};
template <bool MIXED>
struct GRec<MIXED, true> {
  typedef typename Prec<MIXED>::T4 type;
};

template <typename T>
struct Leg {
  T e0, e1, e2;  // unit vector from the neighbour to the centre
  T rinv;        // 1/r (FP64: m^-1; mixed: sigma_Si^-1)
  T E;           // exp(gamma/(r/sigma - a))
  T g;           // d ln E / dr (same length unit as rinv)
  T l0, l1, l2;  // mixed: low parts of e0, e1, e2 (see low_part); FP64: 0
};

// sqrt(a) and 1/sqrt(a) of a positive a (a squared distance, far from the
// ends of the exponent range): the hardware's estimate (24 bits), one
// Goldschmidt step and two residual corrections of the root, one Newton step
// of its reciprocal -- 13 operations instead of the 28 of sqrt() and a
// division, with the same results: bit for bit in 3.4e7 squares of r between
// 1e-12 and 1e-8 m and of r/sigma between 0.02 and 3.  (Both are NaN for a = 0.)
__device__ __forceinline__ void sqrt_rsqrt(double a, double &s, double &si) {
  const double y = __builtin_amdgcn_rsq(a);
  double g = a * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, a), h, g);
  s = __builtin_fma(__builtin_fma(-g, g, a), h, g);
  const double y1 = h + h;
  si = __builtin_fma(y1, __builtin_fma(-s, y1, 1.0), y1);
}
// 1/x (x far from the ends of the exponent range): estimate and two Newton
// steps; the division's bits in 3.4e7 values between -1.9 and -0.0018
__device__ __forceinline__ double fast_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
}

// Low part of an FP32 unit-vector component h = fl(x) of the FP64 value x:
// x - h rounded to a multiple of ulp(h)/1024 and at most 511 of them (a
// signed 10-bit number), as FP32.  With the low parts the vertex pass forms
// cos + 1/3 from (nearly) the FP64 unit vectors, where it cancels near the
// tetrahedral angle.  For h = m 2^e with m in [0.5, 1), ulp(h) = 2^(e - 24);
// adding and taking away 1.5 2^(e + 18) rounds to multiples of 2^(e - 34).
__device__ __forceinline__ float low_part(double x, float h) {
  const int e = __builtin_amdgcn_frexp_expf(h);
  const double big = __builtin_amdgcn_ldexp(1.5, e + 18);
  const float most = __builtin_amdgcn_ldexpf(511.0f, e - 34);
  return __builtin_amdgcn_fmed3f((float)(((x - (double)h) + big) - big), -most, most);
}
// a + b - s exactly, for s = fl(a + b) (TwoSum)
__device__ __forceinline__ float two_sum_err(float a, float b, float s) {
  const float bb = s - a;
  return (a - (s - bb)) + (b - bb);
}

// cos and D = cos + 1/3 of a vertex term with legs a and b, the same bits
// for (a, b) and (b, a).
__device__ __forceinline__ void cos_d(const Leg<double> &a, const Leg<double> &b, double &cs,
                                      double &D) {
  cs = a.e0 * b.e0 + a.e1 * b.e1 + a.e2 * b.e2;
  D = cs + 1.0 / 3.0;
}
// Mixed: from the FP32 unit vectors and their low parts, with the products'
// rounding errors (FMA) and the sums' (TwoSum) carried along, each rounded
// to FP32 once; the rest of the term is FP32.  (The products and sums stay
// unfused: an FMA formed from a product and the following sum would break
// the TwoSum error terms.)
__device__ __forceinline__ void cos_d(const Leg<float> &a, const Leg<float> &b, float &cs,
                                      float &D) {
#pragma clang fp contract(off)
  const float p0 = a.e0 * b.e0, p1 = a.e1 * b.e1, p2 = a.e2 * b.e2;
  const float rp = (__builtin_fmaf(a.e0, b.e0, -p0) + __builtin_fmaf(a.e1, b.e1, -p1)) +
                   __builtin_fmaf(a.e2, b.e2, -p2);
  const float x = ((a.e0 * b.l0 + a.l0 * b.e0) + (a.e1 * b.l1 + a.l1 * b.e1)) +
                  (a.e2 * b.l2 + a.l2 * b.e2);
  const float s1 = p0 + p1, s2 = s1 + p2;
  const float lo = (two_sum_err(p0, p1, s1) + two_sum_err(s1, p2, s2)) + (rp + x);
  cs = s2 + lo;
  // 1/3 = THIRD_HI + THIRD_LO
  const float THIRD_HI = 0.333333343267440796f, THIRD_LO = -9.93410748e-09f;
  const float s3 = s2 + THIRD_HI;
  D = s3 + (two_sum_err(s2, THIRD_HI, s3) + (lo + THIRD_LO));
}
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// Force on leg a of one vertex term (centre c, legs a and b), and h.
// h = leps E(ra) E(rb) D^2, D = cos + 1/3, with d cos/dx_a = -(e_b - cos e_a)/r_a and
// d r_a/dx_a = -e_a, so F_a = -dh/dx_a = h g_a e_a + 2 leps Ea Eb D (e_b - cos e_a)/r_a.
template <typename T>
__device__ __forceinline__ void vterm(T leps, const Leg<T> &a, const Leg<T> &b, T cs, T D, T *Fa,
                                      T &hh) {
  const T Eab = leps * a.E * b.E;
  hh = Eab * D * D;
  const T c1 = hh * a.g;
  const T c2 = T(2) * Eab * D * a.rinv;
  // (fused by hand: the rounding does not depend on the compiler's choice)
  Fa[0] = fma_t(fma_t(-cs, a.e0, b.e0), c2, c1 * a.e0);
  Fa[1] = fma_t(fma_t(-cs, a.e1, b.e1), c2, c1 * a.e1);
  Fa[2] = fma_t(fma_t(-cs, a.e2, b.e2), c2, c1 * a.e2);
}

// Minimum image with v_rndne (ties to even).  Neighbour pairs are far from
// the half-box tie, so this equals the reference's NINT image there.
__device__ __forceinline__ void min_image_fast(const double4 &a, const double4 &b,
                                               const DInst &in, double &x0, double &x1,
                                               double &x2) {
  const double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
  x0 = d0 - rint(d0 * in.ilb[0]) * in.lb[0];
  x1 = d1 - rint(d1 * in.ilb[1]) * in.lb[1];
  x2 = d2 - rint(d2 * in.ilb[2]) * in.lb[2];
}

// v[n] of a 4-entry register table by selects (a dynamic index would put
// the table in scratch memory).
template <typename T>
__device__ __forceinline__ T pick4(const T (&v)[4], int n) {
  return n == 0 ? v[0] : n == 1 ? v[1] : n == 2 ? v[2] : v[3];
}

// The leg of difference d = x_centre - x_neighbour (unit vector from the
// neighbour to the centre, 1/r, E, g), with k_legs' arithmetic: FP64 as the
// reference (si.f90:491-509), or the FP32 terms of the mixed mode.  Legs are
// not stored between passes: k_legs decides which pairs are legs (its leg
// mask), and the passes that need the values recompute them here from the
// positions.
template <bool MIXED>
__device__ __forceinline__ void leg_values(double d0, double d1, double d2, double isg,
                                           float rhof, const FConst &fc,
                                           Leg<typename Prec<MIXED>::T> &L) {
  L.l0 = L.l1 = L.l2 = 0;
  if constexpr (!MIXED) {
    double r, rinv;
    sqrt_rsqrt(d0 * d0 + d1 * d1 + d2 * d2, r, rinv);
    const double inv_ra = fast_rcp(r * isg - fc.al);
    L.e0 = d0 * rinv; L.e1 = d1 * rinv; L.e2 = d2 * rinv;
    L.rinv = rinv;
    L.E = exp(fc.gamma * inv_ra);
    L.g = -fc.gamma * inv_ra * inv_ra * isg;
  } else {
    // every leg value from FP64 geometry, rounded to FP32 once: the FP32
    // vertex terms cannot recover accuracy their inputs do not carry
    const double s0 = d0 * isg, s1 = d1 * isg, s2 = d2 * isg;
    double rs, rinv;
    sqrt_rsqrt(s0 * s0 + s1 * s1 + s2 * s2, rs, rinv);
    const double inv_ra = fast_rcp(rs - fc.al);
    const double rho = rhof;
    double x0, x1, x2;
    {
#pragma clang fp contract(off)
      x0 = s0 * rinv; x1 = s1 * rinv; x2 = s2 * rinv;
    }
    L.e0 = (float)x0; L.e1 = (float)x1; L.e2 = (float)x2;
    L.l0 = low_part(x0, L.e0); L.l1 = low_part(x1, L.e1); L.l2 = low_part(x2, L.e2);
    L.rinv = (float)(rinv * rho);
    L.E = expf((float)(fc.gamma * inv_ra));
    L.g = (float)(-fc.gamma * inv_ra * inv_ra * rho);
  }
}
template <bool MIXED>
__device__ __forceinline__ void make_leg(const double4 &xc, const double4 &xn, const DInst &in,
                                         const FConst &fc, int tc, int tn,
                                         Leg<typename Prec<MIXED>::T> &L) {
  double d0, d1, d2;
  min_image_fast(xc, xn, in, d0, d1, d2);
  const int a = tc == 2 ? 1 : 0, b = tn == 2 ? 1 : 0;
  leg_values<MIXED>(d0, d1, d2, fc.isig[a][b], fc.rho[a][b], fc, L);
}

// Register sum of one force vector's terms a * (x, y, z): FP64, or FP32 with
// a compensation term (mixed; TwoSum with the product in its place, unrounded).
template <bool MIXED>
struct FAcc;
template <>
struct FAcc<false> {
  double x = 0, y = 0, z = 0;
  __device__ void add(double a, double p, double q, double r) {
    x = fma_t(a, p, x); y = fma_t(a, q, y); z = fma_t(a, r, z);
  }
  __device__ void get(double s, double &a, double &b, double &c) const {
    a = x * s; b = y * s; c = z * s;
  }
};
template <>
struct FAcc<true> {
  float x = 0, y = 0, z = 0, cx = 0, cy = 0, cz = 0;
  __device__ __forceinline__ static void sum(float &s, float &c, float a, float p) {
#pragma clang fp contract(off)
    const float t = fma_t(a, p, s);
    const float bp = t - s;
    c += (s - (t - bp)) + fma_t(a, p, -bp);
    s = t;
  }
  __device__ void add(float a, float p, float q, float r) {
    sum(x, cx, a, p); sum(y, cy, a, q); sum(z, cz, a, r);
  }
  __device__ void get(double s, double &a, double &b, double &c) const {
    a = ((double)x + (double)cx) * s;
    b = ((double)y + (double)cy) * s;
    c = ((double)z + (double)cz) * s;
  }
};

#define LEGS_BATCH 4  // k_legs: list slots whose positions are loaded together
#define NEAR_BATCH 4  // and entries of a near list

// Near lists.  Half of a row's entries lie so far beyond the cutoff that they
// cannot come into range while no atom has moved much, and the pair pass is
// bound by its gathers of the partners' positions (about 50 cycles for each
// 16 bytes a lane).  The first pass after a build keeps the entries that were
// within cutoff + delta at the build (FConst::near2, delta = a tenth of the
// skin) in near[n * NA + i] = slot << 27 | partner, their count in nst.  It
// runs at the positions of the build, or, when a program builds the lists and
// then steps, after a move: the entries within cutoff + delta + twice the
// largest displacement hold all of them.  While neither the atom nor any partner of its row has moved
// more than delta / 2 since the build, a pair left out is out of range, and
// the pass runs over the near list alone.  An atom that moves farther
// (k_md_pos, k_pos) takes itself and its partners off their near lists until
// the next build.  Rows with more than NEAR_CAP near entries, or one past
// slot 31, have no near list.  4 x 512 k thermal Si atoms under 2 keV ions,
// mixed, per step: 181 us over whole rows before, 122 us over the near lists
// and 207 us in the pass that makes them; 194 -> 144 us over 40 steps with 16
// replica rebuilds (FP64, 2 x 512 k: 138 -> 111 us).
__device__ __forceinline__ void near_mark_moved(int i, int Wsw, const int *__restrict__ cnt_sw,
                                                const int *__restrict__ nbr_sw,
                                                uint8_t *__restrict__ nst) {
  if (nst[i] == NEAR_MOVED) return;
  const int n = min(cnt_sw[i], Wsw);
  const int *row = nbr_sw + (size_t)i * Wsw;
  for (int k = 0; k < n; ++k) {
    const int j = row[k];
    if (nst[j] != NEAR_MOVED) nst[j] = NEAR_FULL;
  }
  nst[i] = NEAR_MOVED;
}

// r^2 / sigma^2, rounded as the pair and leg values are
template <bool MIXED>
__device__ __forceinline__ double scaled_r2(double d0, double d1, double d2, double isg) {
  if constexpr (MIXED) {
    const double s0 = d0 * isg, s1 = d1 * isg, s2 = d2 * isg;
    return s0 * s0 + s1 * s1 + s2 * s2;
  } else {
    return (d0 * d0 + d1 * d1 + d2 * d2) * (isg * isg);
  }
}

// d <- d - rint(d / L) L (min_image_fast's form) for the lanes' values of one
// axis, left out when every |d| is below half a box (by the upper words, so
// up to 1e-6 less): rint is zero then.
template <int N>
__device__ __forceinline__ void wrap_axis(double (&d)[N], double ilb, double lb) {
  const int half = __double2hiint(lb) - (1 << 20);
  int far = 0;
#pragma unroll
  for (int v = 0; v < N; ++v) far = max(far, __double2hiint(d[v]) & 0x7fffffff);
  if (__ballot(far >= half) != 0ull) {
#pragma unroll
    for (int v = 0; v < N; ++v) d[v] -= rint(d[v] * ilb) * lb;
  }
}

template <bool MIXED, bool EN, bool VIR>
__global__ __launch_bounds__(FIB_BLOCK) void k_legs(
    const double4 *__restrict__ X, const DInst *__restrict__ I, const FConst fc,
    const TabEntry *__restrict__ tab, int NA, int Wsw, int Wion, const int *__restrict__ cnt_sw,
    const int *__restrict__ nbr_sw, const int *__restrict__ cnt_ion,
    const int *__restrict__ nbr_ion, uint64_t *__restrict__ amask,
    double *__restrict__ Fpart, double *__restrict__ upart, uint32_t *__restrict__ near,
    uint8_t *__restrict__ nst, const DCtl *__restrict__ ctl, const int *__restrict__ binst,
    int pstride, double *__restrict__ partials, const int *__restrict__ halt, int xs) {
  typedef typename Prec<MIXED>::T T;
  constexpr bool NT = (FIB_NT_LD & 1) != 0, NTS = (FIB_NT_ST & 1) != 0;
  const int lb = xcd_remap(blockIdx.x, gridDim.x, xs);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  // what the pass needs first, asked for at once (a load takes about a
  // microsecond in a small batch, whose data other XCDs have just written);
  // near entries past the list's end are not used
  const int kin = binst[lb];
  const double4 xi = X[i];
  const uint32_t st = near ? nst[i] : NEAR_FULL;
  uint32_t en[NEAR_BATCH];
#pragma unroll
  for (int v = 0; v < NEAR_BATCH; ++v)
    en[v] = near ? ld_nt<NT>(near + (size_t)v * NA + i) : 0u;
  const int nion = cnt_ion[i];
  HALT_OR_RETURN(halt);
  const uint32_t mi = meta_of(xi);
  // every block lies inside one instance: scalar loads of the instance record
  const DInst &in = I[kin];
  const bool live = !(mi & (META_PAD | META_DEAD));
  const int ti = type_of(mi);
  const bool sw_atom = live && ti < 3;
  const int tr = (ti == 2) ? 1 : 0;
  const double isgA = fc.isig[tr][0], isgB = fc.isig[tr][1];
  const double esgA = fc.epssig[tr][0], esgB = fc.epssig[tr][1];
  const double epsA = fc.eps[tr][0], epsB = fc.eps[tr][1];
  const double isgS = fc.isig[0][0];
  const double fscale = MIXED ? fc.eps[0][0] * isgS : 1.0;
  const double lscale = MIXED ? 1.0 / isgS : 1.0;
  // mixed: SW pair force factor eps_ij/sigma_ij in units of eps_Si/sigma_Si
  // and the pair's length unit over sigma_Si, divided on the host
  const float fsA = fc.fsw[tr][0], fsB = fc.fsw[tr][1];
  const float rhoA = fc.rho[tr][0], rhoB = fc.rho[tr][1];
  const double gate2 = MIXED ? fc.cut_sw2 : fc.r2gate;
  const double leg2 = MIXED ? fc.mixed_xleg * fc.mixed_xleg : fc.cut_sw * fc.cut_sw;
  const double iumax = MIXED ? 0.0 : 1.0 / fc.umax;
  const size_t row = (size_t)i * Wsw;
  __shared__ __attribute__((aligned(16))) uint32_t hold[FIB_BLOCK / FIB_WAVE][NEAR_CAP][FIB_WAVE];
  const int lane = threadIdx.x % FIB_WAVE;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FIB_WAVE);

  FAcc<MIXED> f;
  double ui = 0, etot = 0;
  T W[9];
#pragma unroll
  for (int w = 0; w < 9; ++w) W[w] = 0;
  auto addW = [&](T d0, T d1, T d2, T f0, T f1, T f2) {
    W[0] += d0 * f0; W[1] += d0 * f1; W[2] += d0 * f2;
    W[3] += d1 * f0; W[4] += d1 * f1; W[5] += d1 * f2;
    W[6] += d2 * f0; W[7] += d2 * f1; W[8] += d2 * f2;
  };

  // one SW pair in range: pair force and energy
  auto pair = [&](double d0, double d1, double d2, bool jA) {
    const double isg = jA ? isgA : isgB;
    if constexpr (!MIXED) {
      double r, rinv;
      sqrt_rsqrt(d0 * d0 + d1 * d1 + d2 * d2, r, rinv);
      const double rs = fmax(r * isg, 0.0);  // (coincident atoms: r and 1/r are NaN)
      // reference pair force: 3-point Lagrange on the derivative table
      // (si.f90:416-424, 554-573); rs / umax as its product with 1/umax,
      // corrected by the remainder
      const double q0 = rs * iumax;
      const double q = __builtin_fma(__builtin_fma(-q0, fc.umax, rs), iumax, q0);
      const int t1 = (int)(q * fc.tabn1) + 1;
      if (t1 < fc.izero) {
        const TabEntry te = tab[t1];
        const double e1 = rs - te.u0, e2 = rs - te.u1, e3 = rs - te.u2;
        const double df = 0.5 * e2 * e3 * te.t0 - e1 * e3 * te.t1 + 0.5 * e1 * e2 * te.t2;
        const double fs = -df * (jA ? esgA : esgB) * rinv;
        f.add(fs, d0, d1, d2);
        if (VIR) addW(d0, d1, d2, 0.5 * fs * d0, 0.5 * fs * d1, 0.5 * fs * d2);
      }
      if (EN && rs < fc.cut_sw) {
        const double inv_ra = 1.0 / (rs - fc.al);
        const double rs2 = rs * rs;
        const double ul =
            0.5 * (jA ? epsA : epsB) * fc.A * (fc.B / (rs2 * rs2) - 1.0) * exp(inv_ra);
        ui += ul;
        etot += ul;
      }
    } else {
      // Pair geometry in FP64 (pair units: sigma_ij), the pair force factor
      // rounded to FP32 once.  Near the bond length the two parts of dphi/dr
      // cancel to a small remainder, and formed in FP32 their rounding was
      // the largest error of the mixed forces; the exponential and the
      // force vector stay FP32.
      const double s0 = d0 * isg, s1 = d1 * isg, s2 = d2 * isg;
      double rs, rinv;
      sqrt_rsqrt(s0 * s0 + s1 * s1 + s2 * s2, rs, rinv);
      if (rs >= fc.cut_sw) return;  // (coincident atoms: rs is NaN, and the force too)
      const double inv_ra = fast_rcp(rs - fc.al);
      const double ex = (double)expf((float)inv_ra);
      const double ir2 = rinv * rinv;
      const double ir4 = ir2 * ir2;
      // phi2(r) = A (B r^-4 - 1) e^{1/(r-a)};  force on i = -dphi/dr e
      const double br = -4.0 * fc.B * ir4 * rinv - (fc.B * ir4 - 1.0) * inv_ra * inv_ra;
      const float fs = (float)(-fc.A * ex * br * rinv * (double)(jA ? fsA : fsB));
      const float r0 = (float)s0, r1 = (float)s1, r2 = (float)s2;
      f.add(fs, r0, r1, r2);
      if (VIR) {
        const float q = 1.0f / (jA ? rhoA : rhoB);  // 1 for Si-Si
        const float h0 = fs * r0, h1 = fs * r1, h2 = fs * r2;
        addW(r0 * q, r1 * q, r2 * q, 0.5f * h0, 0.5f * h1, 0.5f * h2);
      }
      if (EN) {
        const double ul = rs == rs
                              ? 0.5 * (jA ? epsA : epsB) * (fc.A * (fc.B * ir4 - 1.0) * ex)
                              : (double)INFINITY;
        ui += ul;
        etot += ul;
      }
    }
  };

  uint64_t am = 0;
  // A pair below gate2 is in range; one below leg2 is a leg (beyond, E =
  // exp(gamma/(r-a)) is zero in FP64 and below e^-30 in the mixed mode: each
  // of its terms is below 1e-9 eps/sigma).
  if (near && !ctl[kin].near_off && __ballot(st > NEAR_CAP) == 0ull) {
    const int n = sw_atom ? (int)st : 0;
    // NEAR_BATCH entries at a time: their positions load together, and the
    // next entries while these arrive
#pragma unroll
    for (int v = 0; v < NEAR_BATCH; ++v) en[v] = v < n ? en[v] : (uint32_t)i;
    for (int q = 0; q < n; q += NEAR_BATCH) {
      double4 xq[NEAR_BATCH];
      uint32_t slot[NEAR_BATCH];
#pragma unroll
      for (int v = 0; v < NEAR_BATCH; ++v) {
        xq[v] = ld_off(X, (en[v] & NEAR_J) * 32u);
        slot[v] = en[v] >> 27;
      }
#pragma unroll
      for (int v = 0; v < NEAR_BATCH; ++v)
        en[v] = q + NEAR_BATCH + v < n ? ld_nt<NT>(near + (size_t)(q + NEAR_BATCH + v) * NA + i)
                                       : (uint32_t)i;
      double d[3][NEAR_BATCH];
#pragma unroll
      for (int v = 0; v < NEAR_BATCH; ++v) {
        d[0][v] = xi.x - xq[v].x;
        d[1][v] = xi.y - xq[v].y;
        d[2][v] = xi.z - xq[v].z;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) wrap_axis<NEAR_BATCH>(d[c], in.ilb[c], in.lb[c]);
#pragma unroll
      for (int v = 0; v < NEAR_BATCH; ++v) {
        const uint32_t mj = meta_of(xq[v]);
        const bool jA = type_of(mj) != 2;
        const double rr = scaled_r2<MIXED>(d[0][v], d[1][v], d[2][v], jA ? isgA : isgB);
        if (q + v < n && !(mj & META_DEAD) && rr < gate2) {
          pair(d[0][v], d[1][v], d[2][v], jA);
          if (rr < leg2) am |= 1ull << slot[v];
        }
      }
    }
  } else {
    const int cs = sw_atom ? min(ld_nt<NT>(cnt_sw + i), Wsw) : 0;
    const int4 *r4 = reinterpret_cast<const int4 *>(nbr_sw + row);
    // LEGS_BATCH slots at a time: their indices, then their positions; the
    // next indices are loaded while the positions arrive (every index read
    // lies below cs <= Wsw, inside the row)
    constexpr int LB = LEGS_BATCH, NQ = LB / 4;
    int4 rn[NQ];
    int nn = 0;  // near entries, also those past the list's end
    double near2 = fc.near2;
    if (near && __ballot(st == NEAR_FRESH) != 0ull && ctl[kin].maxdisp > 0.0) {
      const double c = fc.near_c + 2.0 * ctl[kin].maxdisp * fc.near_isg;
      near2 = c * c;
    }
#pragma unroll
    for (int u = 0; u < NQ; ++u) rn[u] = (4 * u < cs) ? ld_nt<NT>(r4 + u) : make_int4(i, i, i, i);
    for (int k0 = 0; __ballot(k0 < cs) != 0ull; k0 += LB) {
      int jq[LB];
#pragma unroll
      for (int u = 0; u < NQ; ++u) {
        const int b = k0 + 4 * u;
        jq[4 * u] = (b < cs) ? rn[u].x : i;
        jq[4 * u + 1] = (b + 1 < cs) ? rn[u].y : i;
        jq[4 * u + 2] = (b + 2 < cs) ? rn[u].z : i;
        jq[4 * u + 3] = (b + 3 < cs) ? rn[u].w : i;
      }
      double4 xq[LB];
#pragma unroll
      for (int v = 0; v < LB; ++v) xq[v] = ld_off(X, (uint32_t)jq[v] * 32u);
#pragma unroll
      for (int u = 0; u < NQ; ++u)
        if (k0 + LB + 4 * u < cs) rn[u] = ld_nt<NT>(r4 + ((k0 + LB) >> 2) + u);
      double d[3][LB];
#pragma unroll
      for (int v = 0; v < LB; ++v) {
        d[0][v] = xi.x - xq[v].x;
        d[1][v] = xi.y - xq[v].y;
        d[2][v] = xi.z - xq[v].z;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) wrap_axis<LB>(d[c], in.ilb[c], in.lb[c]);
#pragma unroll
      for (int v = 0; v < LB; ++v) {
        const uint32_t mj = meta_of(xq[v]);
        const bool jA = type_of(mj) != 2;
        const double rr = scaled_r2<MIXED>(d[0][v], d[1][v], d[2][v], jA ? isgA : isgB);
        // an atom removed since the build is out of the simulation (MD-step mode)
        const bool ok = k0 + v < cs && !(mj & META_DEAD);
        if (ok && rr < near2) {
          if (nn < NEAR_CAP) hold[wid][nn][lane] = (uint32_t)(k0 + v) << 27 | (uint32_t)jq[v];
          nn += k0 + v < 32 ? 1 : NEAR_CAP + 1;
          if (rr < gate2) pair(d[0][v], d[1][v], d[2][v], jA);
          if (rr < leg2) am |= 1ull << (k0 + v);
        }
      }
    }
    // the near lists leave plane by plane, so that the stores coalesce
    if (near && st == NEAR_FRESH) {
      nst[i] = (uint8_t)(nn <= NEAR_CAP ? nn : NEAR_FULL);
      for (int q = 0; q < min(nn, NEAR_CAP); ++q)
        st_nt<NTS>(near + (size_t)q * NA + i, hold[wid][q][lane]);
    }
  }
  st_nt<NTS>(amask + i, am);

  // ---- Moliere pairs (si.f90:426-446): both atoms must be fired ----------
  // One pair of atom a (species ta) with list entry j, where it is in range:
  // the force as v[0] (v[1], v[2], v[3]), the difference v[4..6] in the
  // virial's length unit, and the atom's half of the energy.
  auto moliere = [&](const double4 &xa, int ta, int j, T (&v)[7], double &ul) -> bool {
    const double4 xj = X[j];
    const uint32_t mj = meta_of(xj);
    const int tj = type_of(mj);
    if (tj == 3 && orig_of(xj) >= in.nsg + in.impact) return false;
    if (mj & META_DEAD) return false;
    double d0, d1, d2;
    min_image_fast(xa, xj, in, d0, d1, d2);
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    if (!(r2 < fc.rlj2)) return false;
    const double r = sqrt(r2);
    const double aa = fc.aamol[ta - 1][tj - 1];
    const double zz = fc.ie0 * fc.zmol[ta - 1] * fc.zmol[tj - 1] * fc.ec * fc.ec;
    if (!MIXED || r < fc.mixed_r64) {
      const double x = r / aa;
      const double e1 = exp(-fc.molb[0] * x), e2 = exp(-fc.molb[1] * x),
                   e3 = exp(-fc.molb[2] * x);
      const double sa = fc.molc[0] * e1 + fc.molc[1] * e2 + fc.molc[2] * e3;
      const double sb = (fc.molc[0] * fc.molb[0] * e1 + fc.molc[1] * fc.molb[1] * e2 +
                         fc.molc[2] * fc.molb[2] * e3) / aa;
      const double fcm = zz / r * (sa / r + sb);
      const double rinv = 1.0 / r;
      v[0] = T(1);
      v[1] = (T)(fcm * d0 * rinv / fscale);
      v[2] = (T)(fcm * d1 * rinv / fscale);
      v[3] = (T)(fcm * d2 * rinv / fscale);
      if (EN) ul = 0.5 * zz / r * sa;
    } else {
      // FP32 with lengths in units of aa; F = (zz/aa^2) (1/x)(sa/x + sb) d/(aa x)
      const float x = (float)(r / aa);
      const float e1 = __expf(-(float)fc.molb[0] * x), e2 = __expf(-(float)fc.molb[1] * x),
                  e3 = __expf(-(float)fc.molb[2] * x);
      const float c0 = (float)fc.molc[0], c1 = (float)fc.molc[1], c2 = (float)fc.molc[2];
      const float sa = c0 * e1 + c1 * e2 + c2 * e3;
      const float sb = c0 * (float)fc.molb[0] * e1 + c1 * (float)fc.molb[1] * e2 +
                       c2 * (float)fc.molb[2] * e3;
      const float ix = __builtin_amdgcn_rcpf(x);
      const float fr = ix * (sa * ix + sb) * ix;
      v[0] = (T)(float)(zz / (aa * aa) / fscale);
      v[1] = (T)(fr * (float)(d0 / aa));
      v[2] = (T)(fr * (float)(d1 / aa));
      v[3] = (T)(fr * (float)(d2 / aa));
      if (EN) ul = 0.5 * zz / aa * (double)(sa * ix);
    }
    if (VIR) {
      v[4] = (T)(d0 / lscale);
      v[5] = (T)(d1 / lscale);
      v[6] = (T)(d2 / lscale);
    }
    return true;
  };
  // The wavefront's pairs stand in a row, atom by atom, and its lanes take one
  // each; their results wait in LDS and every atom adds its own in list order.
  // (A Ga atom lists some forty partners, and its lane used to work them off
  // alone, two dependent loads and a few hundred instructions each, while the
  // rest of the pass had long ended: k_legs of 64 x 4 k atoms, mixed, 59.3 ->
  // 32.6 us; of one 4 k slab, FP64, 37.8 -> 18.)
  const bool fired = !(ti == 3 && orig_of(xi) >= in.nsg + in.impact);
  const int ci = live && fired ? min(nion, Wion) : 0;
  const uint64_t rows = __ballot(ci > 0);
  if (rows != 0ull) {
    T *const sv = reinterpret_cast<T *>(&hold[wid][0][0]);  // [7][64], then the energies
    double *const su = reinterpret_cast<double *>(sv + 7 * FIB_WAVE);
    static_assert(sizeof(hold[0]) >= FIB_WAVE * (7 * sizeof(T) + sizeof(double)), "hold");
    int np = 1;  // pairs in the row
    for (int p0 = 0; p0 < np; p0 += FIB_WAVE) {
      const int p = p0 + lane;
      // whose pair p is, which of its list, and where this atom's pairs start
      int own = lane, k = 0, first = 0;
      np = 0;
      for (uint64_t m = rows; m != 0ull; m &= m - 1) {
        const int o = __ffsll((unsigned long long)m) - 1;
        if (p >= np) {
          own = o;
          k = p - np;
        }
        if (lane == o) first = np;
        np += __builtin_amdgcn_readlane(ci, o);
      }
      double4 xo;
      xo.x = __shfl(xi.x, own);
      xo.y = __shfl(xi.y, own);
      xo.z = __shfl(xi.z, own);
      xo.w = 0.0;
      const int to = __shfl(ti, own);
      T v[7];
      double ul = 0;
      const bool hit =
          p < np &&
          moliere(xo, to, nbr_ion[(size_t)(i - lane + own) * Wion + k], v, ul);
      // (a pair out of range adds zeros: the sums are the same, and their
      // values come from LDS several at a time)
      wave_lds_sync();
      if (p < np) {
#pragma unroll
        for (int c = 0; c < (VIR ? 7 : 4); ++c) sv[c * FIB_WAVE + lane] = hit ? v[c] : T(0);
        if (EN) su[lane] = hit ? ul : 0.0;
      }
      wave_lds_sync();
      const int q1 = min(first + ci - p0, FIB_WAVE);
#pragma unroll 4
      for (int q = max(first - p0, 0); q < q1; ++q) {
#pragma unroll
        for (int c = 0; c < (VIR ? 7 : 4); ++c) v[c] = sv[c * FIB_WAVE + q];
        f.add(v[0], v[1], v[2], v[3]);
        if (VIR)
          addW(v[4], v[5], v[6], T(0.5) * (v[0] * v[1]), T(0.5) * (v[0] * v[2]),
               T(0.5) * (v[0] * v[3]));
        if (EN) {
          ui += su[q];
          etot += su[q];
        }
      }
      wave_lds_sync();
    }
  }

  double fx, fy, fz;
  f.get(fscale, fx, fy, fz);
  st_nt<NTS>(Fpart + i, fx);
  st_nt<NTS>(Fpart + (size_t)NA + i, fy);
  st_nt<NTS>(Fpart + 2 * (size_t)NA + i, fz);
  if (EN) upart[i] = ui;
  if (EN || VIR) {
    double v[10];
    v[0] = etot;
    const double ws = MIXED ? fscale * lscale : 1.0;
#pragma unroll
    for (int w = 0; w < 9; ++w) v[1 + w] = (double)W[w] * ws;
    const int op[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    block_partials<10, FIB_BLOCK>(v, op, lb, pstride, partials);
  }
}


// ---------------------------------------------------------------------------
// Vertex terms of the build-time graph that the centre's own list misses.
//
// The reference stores its triplets once per list build (si.f90:191-232):
// every connected triple of the buffered graph.  Between builds the vertex
// term centred on c with legs a and b is evaluated whenever both legs are in
// range *now* (si.f90:491-509), so after atoms have moved more than the list
// skin a term can exist whose leg c-a is not a listed pair, the triple being
// connected through the pairs c-b and b-a instead.  k_legs/k_tri only pair
// legs from c's own list; this pass adds the rest, exactly and without
// atomics: the term (a, c, b) is found by the bridge atom b, which lists both
// a and c.  b keeps its own share and writes the forces on a and c into
// EX[slot][b] by its list slots of a and c; a and c gather them like G.
// Nothing can be missing unless two atoms moved together by more than the
// skin, so the pass exits at once while maxdisp + maxdisp2 <= skin.  Further
// workgroups of k_tri's launch do it, whose results it does not need: a launch
// of its own cost 4.7 us even with nothing to do (fib_step of 1.9 k atoms 47
// -> 43 us a step, of 154 k 85 -> 82).
template <bool MIXED, bool EN, bool VIR>
__device__ __forceinline__ void extra_pass(
    int lb,
    const double4 *__restrict__ X, const DInst *__restrict__ I, const FConst fc, int NA, int Wsw,
    const int *__restrict__ cnt_sw, const int *__restrict__ nbr_sw,
    const uint64_t *__restrict__ amask,
    const float *__restrict__ disp, DCtl *__restrict__ ctl, typename Prec<MIXED>::T4 *__restrict__ EX,
    typename Prec<MIXED>::T4 *__restrict__ EXself, uint64_t *__restrict__ exmask, int pstride,
    double *__restrict__ partials, const uint8_t *__restrict__ nst) {
  typedef typename Prec<MIXED>::T T;
  typedef typename Prec<MIXED>::T4 T4;
  const int b = lb * FIB_BLOCK + threadIdx.x;
  const double4 xb = X[b];
  const uint32_t mb = meta_of(xb);
  const int kin = __builtin_amdgcn_readfirstlane(inst_of(mb));
  const DInst &in = I[kin];
  const double isgS = fc.isig[0][0];
  const double fscale = MIXED ? fc.eps[0][0] * isgS : 1.0;
  const double escale = MIXED ? fc.eps[0][0] : 1.0;
  const double lscale = MIXED ? 1.0 / isgS : 1.0;
  double v[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  const int op[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  // block-uniform: one instance per block
  const bool active = ctl[kin].maxdisp + ctl[kin].maxdisp2 > fc.skin;
  if (!active) {
    // nothing to add: clear the instance's flag so the gather skips EX
    if (threadIdx.x == 0 && lb * FIB_BLOCK == in.atom_off) ctl[kin].extra_any = 0;
    if (EN || VIR) block_partials<10, FIB_BLOCK>(v, op, lb, pstride, partials);
    return;
  }
  const bool live = !(mb & (META_PAD | META_DEAD));
  const int tb = type_of(mb);
  const double lu = MIXED ? 1.0 / fc.eps[0][0] : 1.0;
  const T lp[4] = {(T)(fc.leps[0][0][0] * lu), (T)(fc.leps[0][0][1] * lu),
                   (T)(fc.leps[0][1][1] * lu), (T)(fc.leps[1][1][1] * lu)};
  const float skin = (float)fc.skin;
  uint64_t em = 0;
  double fb0 = 0, fb1 = 0, fb2 = 0;
  T ub = 0, et = 0;
  T W[9];
#pragma unroll
  for (int w = 0; w < 9; ++w) W[w] = 0;
  // An atom with a near list has no partner that moved more than delta / 2
  // (see near_mark_moved), so no two of its partners moved by the skin.  The
  // others look at their partners' displacements first: in most wavefronts
  // no atom has one of more than half the skin.  (Without the two checks the
  // pass took 37 to 49 us for 5.8 k atoms of a fib_step call, a serial chain
  // of gathers per pair.)
  const bool moved = !nst || ctl[kin].near_off || nst[b] > NEAR_CAP;
  if (live && tb < 3 && moved) {
    const int cs = min(cnt_sw[b], Wsw);
    const int *rowb = nbr_sw + (size_t)b * Wsw;
    const uint64_t amb = amask[b];
    // of the two, one moved more than half the skin
    uint64_t far = 0;
    for (int k0 = 0; k0 < cs; k0 += 4) {
      float dk[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) dk[v] = k0 + v < cs ? disp[rowb[k0 + v]] : 0.0f;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (dk[v] > 0.4999f * skin) far |= 1ull << (k0 + v);
    }
    const int na = far ? __popcll(amb) : 0;
    for (int n = 0; n < na; ++n) {
      const int kc = nth_bit(amb, n);  // b's list slot of c
      const int c = rowb[kc];
      const float dc = disp[c];
      const bool cfar = (far >> kc) & 1ull;
      const double4 xc = X[c];
      const int tc = type_of(meta_of(xc));
      Leg<T> Lbc;  // b's leg to c: unit vector from c to b
      make_leg<MIXED>(xb, xc, in, fc, tb, tc, Lbc);
      const int *rowc = nbr_sw + (size_t)c * Wsw;
      const int cc = min(cnt_sw[c], Wsw);
      for (int k = 0; k < cs; ++k) {
        if (!cfar && !((far >> k) & 1ull)) continue;
        const int a = rowb[k];
        if (a == c || !(disp[a] + dc > skin)) continue;
        const double4 xa = X[a];
        const int ta = type_of(meta_of(xa));
        // leg c -> a: d = x_c - x_a (unit vector from a to the centre c)
        double d0, d1, d2;
        min_image_fast(xc, xa, in, d0, d1, d2);
        const double isg = fc.isig[(tc == 2) ? 1 : 0][(ta == 2) ? 1 : 0];
        const double s0 = MIXED ? d0 * isg : d0, s1 = MIXED ? d1 * isg : d1,
                     s2 = MIXED ? d2 * isg : d2;
        const double rr = s0 * s0 + s1 * s1 + s2 * s2;
        if (MIXED && !(rr < fc.cut_sw2)) continue;
        const double r = sqrt(rr);
        if (!((MIXED ? r : r * isg) < (MIXED ? fc.mixed_xleg : fc.cut_sw))) continue;
        bool listed = false;
        for (int q = 0; q < cc; ++q) listed |= (rowc[q] == a);
        if (listed) continue;
        Leg<T> Lca;
        leg_values<MIXED>(d0, d1, d2, isg, fc.rho[(tc == 2) ? 1 : 0][(ta == 2) ? 1 : 0], fc, Lca);
        // leg c -> b is b's leg to c, reversed
        Leg<T> Lcb = Lbc;
        Lcb.e0 = -Lbc.e0; Lcb.e1 = -Lbc.e1; Lcb.e2 = -Lbc.e2;
        Lcb.l0 = -Lbc.l0; Lcb.l1 = -Lbc.l1; Lcb.l2 = -Lbc.l2;
        const int nge = (tc == 2) + (ta == 2) + (tb == 2);
        T Fa[3], Fb[3], hh, cosv, D;
        cos_d(Lca, Lcb, cosv, D);
        // vterm gives the force on its first leg: once per end
        vterm<T>(pick4(lp, nge), Lca, Lcb, cosv, D, Fa, hh);
        vterm<T>(pick4(lp, nge), Lcb, Lca, cosv, D, Fb, hh);
        const T Fc0 = -(Fa[0] + Fb[0]), Fc1 = -(Fa[1] + Fb[1]), Fc2 = -(Fa[2] + Fb[2]);
        fb0 += (double)Fb[0]; fb1 += (double)Fb[1]; fb2 += (double)Fb[2];
        const T third = hh * T(1.0 / 3.0);
        // forces on a (slot k) and c (slot kc) for them to gather
        const uint64_t bits[2] = {1ull << k, 1ull << kc};
        const int slots[2] = {k, kc};
        const T fx[2] = {Fa[0], Fc0}, fy[2] = {Fa[1], Fc1}, fz[2] = {Fa[2], Fc2};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const size_t at = (size_t)slots[e] * NA + b;
          T4 g;
          if (em & bits[e]) {
            g = EX[at];
          } else {
            g.x = g.y = g.z = g.w = T(0);
          }
          g.x += fx[e]; g.y += fy[e]; g.z += fz[e]; g.w += third;
          EX[at] = g;
          em |= bits[e];
        }
        ub += third;
        et += hh;
        if (VIR) {
          // relative to the centre: r_a = x_a - x_c = -e_ca / rinv_ca, same for b
          const T ra = -T(1) / Lca.rinv, rb = -T(1) / Lcb.rinv;
          const T a0 = ra * Lca.e0, a1 = ra * Lca.e1, a2 = ra * Lca.e2;
          const T b0 = rb * Lcb.e0, b1 = rb * Lcb.e1, b2 = rb * Lcb.e2;
          W[0] += a0 * Fa[0] + b0 * Fb[0]; W[1] += a0 * Fa[1] + b0 * Fb[1];
          W[2] += a0 * Fa[2] + b0 * Fb[2]; W[3] += a1 * Fa[0] + b1 * Fb[0];
          W[4] += a1 * Fa[1] + b1 * Fb[1]; W[5] += a1 * Fa[2] + b1 * Fb[2];
          W[6] += a2 * Fa[0] + b2 * Fb[0]; W[7] += a2 * Fa[1] + b2 * Fb[1];
          W[8] += a2 * Fa[2] + b2 * Fb[2];
        }
      }
    }
  }
  exmask[b] = em;
  {
    T4 g;
    g.x = (T)fb0; g.y = (T)fb1; g.z = (T)fb2; g.w = ub;
    EXself[b] = g;
  }
  if (em) {
    // rare: only after atoms outran the list skin (global atomic, vector memory)
    __hip_atomic_fetch_or(&ctl[kin].extra_any, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (EN || VIR) {
    v[0] = (double)et * escale;
    const double ws = MIXED ? fscale * lscale : 1.0;
#pragma unroll
    for (int w = 0; w < 9; ++w) v[1 + w] = (double)W[w] * ws;
    block_partials<10, FIB_BLOCK>(v, op, lb, pstride, partials);
  }
}

// What k_tri's further workgroups need for it (blocks of FIB_BLOCK atoms; 0:
// none).
struct ExtraArgs {
  int blocks;
  const int *cnt_sw;
  const float *disp;
  DCtl *ctl;
  void *EX, *EXself;
  uint64_t *exmask;
  const uint8_t *nst;
};

// Lane-per-leg three-body pass.  Block = 4 independent wavefronts, each
// owning 64 consecutive atoms, whose legs (the pairs of their leg masks) it
// takes in passes of whole atoms with at most 64 legs: one lane computes one
// leg from the positions, and the legs of a pass share their values through
// a small LDS stage; no leg record goes through HBM.  The pass is bound by
// vector instructions (0.75 to 0.85 of a CU's issue cycles), so it is laid
// out to need few of them:
//  - every lane works on a leg, in the stage as in the terms;
//  - mixed: the compensated cos + 1/3, two thirds of a vertex term's
//    instructions and the same for both of its legs, is formed once per
//    unordered pair.  Leg a of an atom's n takes the partners a + 1 ..
//    a + n/2 around the ring of legs (of an even ring's opposite pairs, the
//    first half takes them) and hands cos and D to both legs through LDS;
//    then each leg sums its terms in leg order.  Atoms with more than
//    TRI_QROWS legs have it formed per term instead.
//  - the Ge selections are left out of passes without a Ge atom.
// Results wait in LDS and leave plane by plane for up to NS/2 legs at once,
// so that the stores coalesce.
// 4 x 512 k thermal Si atoms, per step: mixed 4,903 vector instructions per
// wavefront and 300 us with one term per (leg, partner), 3,090 and 213 us
// so; FP64 245 -> 173 us (2 x 512 k).  With the virial, its terms of a run
// of 256 legs used to wait in 24 (FP64: 48) KiB of LDS, which left two blocks
// to a CU; they now turn to their lanes through shuffles, and three fit: 2.1 M
// atoms, mixed, with energies, just built: 588 -> 477 us.  (Each centre summing
// its own legs' terms would not depend on the split; in FP64 it took 570 to 640
// us for the shuffles' 480 there, and 18 for 15.5 of 4 k atoms.)
#ifndef TRI_BATCH
#define TRI_BATCH 4  // 4: the next pass's positions load during this one; 2: only its row entries
#endif
#ifndef TRI_NS_MIXED
#define TRI_NS_MIXED 256  // legs per write-out (mixed)
#endif
#ifndef TRI_NS_FP64
#define TRI_NS_FP64 256  // legs per write-out (FP64)
#endif
#define TRI_QROWS 8   // most legs of an atom whose pairs share cos + 1/3 (mixed)
#define TRI_TAB 384   // legs whose owner and list slot are tabled at once
#define TRI_TAB_VIR 256
// Batches of up to TRI_SMALL atoms have 16 atoms per wavefront instead of 64:
// 4 k atoms are 64 wavefronts of 64 for 1,024 SIMDs, and the passes of one
// wavefront follow each other.  A large batch fills the chip either way and
// pays for 16 with emptier last passes.  us of an MD step's pass over a thermal
// crystal, 64 and 16 atoms:
//            4,096   64,000   130,000  238,080 atoms
//   mixed  20, 12.5  22, 18   25, 30   34, 48
//   FP64   25, 13    30, 25   35, 38   59, 61
// and with energies 23, 14; 27, 21; 32, 35; 43, 58 (mixed) and 28, 14; 34, 29;
// 42, 45; 70, 73 (FP64): the lines between cross at 98 k to 109 k atoms.
#define TRI_SMALL FIB_TRI_SMALL
// and of up to TRI_TINY eight, about 34 legs, one pass.  16 and 8 atoms:
//            4,096    16,128   32,768   64,000 atoms
//   mixed  12.5, 9.9  13, 11   14, 13   18, 20
//   FP64   13, 11     14, 13   16, 17   25, 25
#define TRI_TINY 16384
template <bool MIXED>
struct TriStage {
  static constexpr int N = MIXED ? TRI_NS_MIXED : TRI_NS_FP64;
};
// The partial sums of k_tri, one per workgroup (of 256 or 64 atoms), from each
// lane's sums (the energy, of its own atom; the virial, see there): neighbouring
// atoms first, and pairs of wavefronts here as of workgroups in fin_chunk_slot,
// so that an instance gives the energy's bits whether a wavefront has 64 atoms
// or 16.
template <int LANES>  // that hold sums: the atoms', or all where the virial's are
__device__ __forceinline__ void tri_partials(double (&v)[10], int at, int pstride,
                                             double *__restrict__ partials) {
  constexpr int NW = FIB_BLOCK / FIB_WAVE;
  static_assert(NW == 4, "two levels");
  const int lane = threadIdx.x % FIB_WAVE, wid = threadIdx.x / FIB_WAVE;
  for (int o = 1; o < LANES; o <<= 1) {
#pragma unroll
    for (int k = 0; k < 10; ++k) v[k] += __shfl_xor(v[k], o);
  }
  __shared__ double red[NW][10];
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 10; ++k) red[wid][k] = v[k];
  __syncthreads();
  if (threadIdx.x < 10) {
    const int k = threadIdx.x;
    partials[(size_t)k * pstride + at] = (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
  }
}

template <bool MIXED, bool EN, bool VIR, int NS, int TB, int APW, bool XT>
__global__ __launch_bounds__(FIB_BLOCK) void k_tri(
    const double4 *__restrict__ X, const DInst *__restrict__ I, const FConst fc, int NA,
    int Wsw, const int *__restrict__ nbr_sw, uint16_t *__restrict__ rk_sw,
    const uint8_t *__restrict__ off_sw, const uint64_t *__restrict__ amask,
    typename GRec<MIXED, EN>::type *__restrict__ G, uint32_t *__restrict__ RA,
    double *__restrict__ Gown, double *__restrict__ Gown_u, int pstride,
    double *__restrict__ partials, const int *__restrict__ binst, const int *__restrict__ halt,
    int xs, const ExtraArgs xa) {
  typedef typename Prec<MIXED>::T T;
  typedef typename Prec<MIXED>::T4 T4;
  typedef typename GRec<MIXED, EN>::type GV;
  constexpr int NW = FIB_BLOCK / FIB_WAVE, QR = TRI_QROWS, FL = NS / 2;
  constexpr bool NT = (FIB_NT_LD & 2) != 0, NTS = (FIB_NT_ST & 2) != 0;
  constexpr bool U = EN || VIR;  // the terms' energies are wanted
  __shared__ T4 sE[NW][FIB_WAVE];  // e0, e1, e2 and E, negated when the leg's atom is Ge (E > 0)
  __shared__ float4 sL[NW][MIXED ? FIB_WAVE : 1];       // l0, l1, l2
  __shared__ float2 sQ[NW][MIXED ? QR * FIB_WAVE : 1];  // [partner][leg]: cos, D
  __shared__ T4 sG[NW][FL];
  __shared__ uint32_t sR[NW][FL];
  constexpr int TAB = VIR ? TRI_TAB_VIR : TRI_TAB;
  __shared__ uint16_t tab[NW][TAB];  // owner lane | list slot << 6
  const int nb = XT ? (int)gridDim.x - xa.blocks : (int)gridDim.x;
  if constexpr (XT) {
    if ((int)blockIdx.x >= nb) {
      HALT_OR_RETURN(halt);
      extra_pass<MIXED, EN, VIR>(xcd_remap(blockIdx.x - nb, xa.blocks), X, I, fc, NA, Wsw,
                                 xa.cnt_sw, nbr_sw, amask, xa.disp, xa.ctl, (T4 *)xa.EX,
                                 (T4 *)xa.EXself, xa.exmask, pstride,
                                 partials + (size_t)FIB_NRED * pstride, xa.nst);
      return;
    }
  }
  const int lb = xcd_remap(blockIdx.x, nb, xs);
  const int lane = threadIdx.x % FIB_WAVE;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / FIB_WAVE);
  const int i0 = (lb * NW + wid) * APW;
  const double escale = MIXED ? fc.eps[0][0] : 1.0;
  const double fscale = MIXED ? fc.eps[0][0] * fc.isig[0][0] : 1.0;
  const double lscale = MIXED ? 1.0 / fc.isig[0][0] : 1.0;
  // lambda*eps by number of Ge atoms in the term (symmetric in the three
  // species, prms.f90:464-471), in J or eps_Si
  const double lu = MIXED ? 1.0 / fc.eps[0][0] : 1.0;
  const T lp[4] = {(T)(fc.leps[0][0][0] * lu), (T)(fc.leps[0][0][1] * lu),
                   (T)(fc.leps[0][1][1] * lu), (T)(fc.leps[1][1][1] * lu)};

  // this lane's atom as a centre; every block lies inside one instance (what
  // is needed first is asked for at once, see k_legs)
  const int kin = binst[i0 / FIB_BLOCK];
  const int ic = i0 + (APW < FIB_WAVE ? min(lane, APW - 1) : lane);
  const double4 xc = X[ic];
  const uint64_t amv = amask[ic];
  HALT_OR_RETURN(halt);
  const uint64_t amc = lane < APW ? amv : 0ull;
  const int tci = type_of(meta_of(xc));
  const DInst &in = I[kin];
  if constexpr (VIR && !MIXED)  // (the other launch has this instance: see force_ab)
    if ((in.natm_pad <= TRI_SMALL) != (APW < FIB_WAVE)) return;
  // legs of the wave's atoms: this atom's are [exc, inc)
  const int nl = __popcll(amc);
  int inc = nl;
  for (int o = 1; o < FIB_WAVE; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (lane >= o) inc += y;
  }
  const int exc = inc - nl;

  double uc = 0;
  T W[9];
#pragma unroll
  for (int w = 0; w < 9; ++w) W[w] = 0;

  // results of the legs [fs, ...) of the atoms [f0, f1) wait in sG and sR;
  // each atom's own sum of them, the reaction on the centre, goes with them
  int f0 = 0, fs = 0;
  auto write_out = [&](int f1) {
    wave_lds_sync();
    const bool mine = lane >= f0 && lane < f1;
    double g0 = 0, g1 = 0, g2 = 0, gu = 0;
    for (int a = 0; __ballot(mine && a < nl) != 0ull; ++a) {
      if (mine && a < nl) {
        const size_t at = (size_t)a * NA + ic;
        const int q = exc + a - fs;
        const T4 g = sG[wid][q];
        GV gv;
        gv.x = g.x; gv.y = g.y; gv.z = g.z;
        if constexpr (EN) {
          gv.w = g.w * T(1.0 / 3.0);
          gu += 0.5 * (double)gv.w;
        }
        if (U) uc += (double)g.w;
        G[at] = gv;
        st_nt<NTS>(RA + at, sR[wid][q]);
        g0 -= (double)g.x; g1 -= (double)g.y; g2 -= (double)g.z;
      }
    }
    if (mine) {
      st_nt<NTS>(Gown + ic, g0);
      st_nt<NTS>(Gown + (size_t)NA + ic, g1);
      st_nt<NTS>(Gown + 2 * (size_t)NA + ic, g2);
      if (EN) st_nt<NTS>(Gown_u + ic, gu);
    }
    wave_lds_sync();
  };

  for (int r0 = 0; r0 < APW;) {
    // atoms [r0, r1) whose legs fit the table (an atom has at most Wsw <= 64
    // legs, so every run takes at least one atom, as does every pass)
    const int rs = __builtin_amdgcn_readlane(exc, r0);
    const int r1 = r0 + __popcll(__ballot(lane >= r0 && lane < APW && inc - rs <= TAB));
    wave_lds_sync();
    if (lane >= r0 && lane < r1) {
      uint64_t m = amc;
      for (int a = 0; a < nl; ++a) {
        tab[wid][exc - rs + a] = (uint16_t)(lane | ((__ffsll((unsigned long long)m) - 1) << 6));
        m &= m - 1;
      }
    }
    wave_lds_sync();
    // pass of the atoms [p0, p1), legs [ps, ps + n): this lane's leg, its row
    // entry, and the partner's position, leg mask and row start
    struct Pass {
      int p0, p1, ps, n;
      int o, k, j, rq;
      double4 x;
      uint64_t aq;
      int oq;
    };
    auto entries = [&](Pass &P, int p0) {
      P.p0 = p0;
      P.ps = __builtin_amdgcn_readlane(exc, p0);
      P.p1 = p0 + __popcll(__ballot(lane >= p0 && lane < r1 && inc - P.ps <= FIB_WAVE));
      P.n = __builtin_amdgcn_readlane(inc, P.p1 - 1) - P.ps;
      P.o = p0; P.k = 0; P.j = i0; P.rq = 0xffff;
      if (lane < P.n) {
        const int e = tab[wid][P.ps - rs + lane];
        P.o = e & 63;
        P.k = e >> 6;
        const uint32_t at = (uint32_t)(i0 + P.o) * (uint32_t)Wsw + (uint32_t)P.k;
        P.j = ld_nt<NT>(nbr_sw + at);
        P.rq = (int)ld_nt<NT>(rk_sw + at);
      }
    };
    // Where the partner j keeps the force of its own terms on the owner:
    // G[n * NA + j], n = j's leg index of the owner.  The slot r of the
    // owner in j's row follows from the stencil offsets (see k_nbuild), n
    // from j's leg mask (legs are symmetric); 255 offsets (r >= Wsw) mark a
    // j without a row.  The first time a pair is a leg after a build, r is
    // worked out from j's offsets and kept in the row entry (RK_SLOT set);
    // later steps read it there, without the gather of j's offsets.
    auto partners = [&](Pass &P) {
      P.x = ld_off(X, (uint32_t)P.j * 32u);
      P.aq = ld_off(amask, (uint32_t)P.j * 8u);
      P.oq = (P.rq & RK_SLOT) ? 0 : off_sw[(size_t)P.j * OFF_W + 26 - (P.rq >> 8)];
    };
    Pass P, Q;
    entries(P, r0);
    partners(P);
    while (true) {
      const bool more = P.p1 < r1;
      if (more) entries(Q, P.p1);
      const bool act = lane < P.n;
      // the owner's position, species and legs, from the owner's lane
      double4 xo;
      xo.x = __shfl(xc.x, P.o);
      xo.y = __shfl(xc.y, P.o);
      xo.z = __shfl(xc.z, P.o);
      xo.w = 0.0;
      const int to = __shfl(tci, P.o);
      const int c0 = __shfl(exc, P.o) - P.ps;  // the owner's first leg in the pass
      const int no = __shfl(nl, P.o);          // (every lane takes part)
      const int na = act ? no : 0;
      const int a = lane - c0;
      const int tn = type_of(meta_of(P.x));
      Leg<T> La;
      make_leg<MIXED>(xo, P.x, in, fc, to, tn, La);
      {
        T4 x;
        x.x = La.e0; x.y = La.e1; x.z = La.e2; x.w = tn == 2 ? -La.E : La.E;
        sE[wid][lane] = x;
        if constexpr (MIXED) sL[wid][lane] = make_float4(La.l0, La.l1, La.l2, 0.0f);
      }
      uint32_t ra = ~0u;
      {
        const int r = (P.rq & RK_SLOT) ? (P.rq & ~RK_SLOT) : min(P.oq + (P.rq & 0xff), 127);
        if (act && !(P.rq & RK_SLOT))
          rk_sw[(size_t)(i0 + P.o) * Wsw + P.k] = (uint16_t)(RK_SLOT | r);
        if (r < Wsw)
          ra = (uint32_t)__popcll(P.aq & ((1ull << r) - 1ull)) * (uint32_t)NA + (uint32_t)P.j;
      }
      if (P.ps + P.n - fs > FL) {
        write_out(P.p0);
        f0 = P.p0;
        fs = P.ps;
      }
      if (TB >= 4 && more) partners(Q);
      wave_lds_sync();
      auto low_of = [&](int q, Leg<T> &L) {
        if constexpr (MIXED) {
          const float4 l = sL[wid][q];
          L.l0 = l.x; L.l1 = l.y; L.l2 = l.z;
        }
      };
      // cos and D of every pair of the pass in sQ, or (not SHARED) per term;
      // without a Ge atom in the pass (not GE) lambda eps is that of Si
      const bool shared = MIXED && __ballot(na > QR) == 0ull;
      const bool ge = __ballot(to == 2 || tn == 2) != 0ull;
      T Ga0 = 0, Ga1 = 0, Ga2 = 0, Gu = 0;
      if (shared) {
        const int half = na >> 1, last = half - ((na & 1) == 0 && a >= half ? 1 : 0);
        int b = a;
        for (int t = 1; t <= last; ++t) {
          b = b + 1 == na ? 0 : b + 1;
          Leg<T> Lb;
          const T4 x = sE[wid][c0 + b];
          Lb.e0 = x.x; Lb.e1 = x.y; Lb.e2 = x.z;
          low_of(c0 + b, Lb);
          T cs, D;
          cos_d(La, Lb, cs, D);
          const float2 v = make_float2((float)cs, (float)D);
          sQ[wid][b * FIB_WAVE + lane] = v;
          sQ[wid][a * FIB_WAVE + c0 + b] = v;
        }
        wave_lds_sync();
      }
      auto terms = [&](auto GE_, auto SHARED_) {
        constexpr bool GE = decltype(GE_)::value, SHARED = decltype(SHARED_)::value;
        const int ga = GE ? (to == 2 ? 1 : 0) + (tn == 2 ? 1 : 0) : 0;
        for (int b = a == 0 ? 1 : 0; b < na; b += b + 1 == a ? 2 : 1) {
          Leg<T> Lb;
          const T4 x = sE[wid][c0 + b];
          Lb.e0 = x.x; Lb.e1 = x.y; Lb.e2 = x.z; Lb.E = GE ? fabs(x.w) : x.w;
          T cs, D, Fa[3], hh;
          if constexpr (SHARED) {
            const float2 v = sQ[wid][b * FIB_WAVE + lane];
            cs = (T)v.x;
            D = (T)v.y;
          } else {
            low_of(c0 + b, Lb);
            cos_d(La, Lb, cs, D);
          }
          vterm<T>(GE ? pick4(lp, ga + (x.w < T(0) ? 1 : 0)) : lp[0], La, Lb, cs, D, Fa, hh);
          Ga0 += Fa[0]; Ga1 += Fa[1]; Ga2 += Fa[2];
          if (U) Gu += hh;
        }
      };
      using Yes = std::integral_constant<bool, true>;
      using No = std::integral_constant<bool, false>;
      if constexpr (MIXED) {
        if (shared) {
          if (ge) terms(Yes{}, Yes{}); else terms(No{}, Yes{});
        } else {
          terms(Yes{}, No{});
        }
      } else {
        if (ge) terms(Yes{}, No{}); else terms(No{}, No{});
      }
      if (act) {
        T4 gv;
        gv.x = Ga0; gv.y = Ga1; gv.z = Ga2; gv.w = Gu;
        sG[wid][P.ps - fs + lane] = gv;
        sR[wid][P.ps - fs + lane] = ra;
      }
      if (VIR) {
        // r_a = x_a - x_i = -e_a / rinv_a.  Lane q % 64 sums for leg q of a
        // run (the FP32 sums of the mixed mode then do not depend on how a
        // run is cut into passes): the pass's values turn by its start.
        const T rl = -T(1) / La.rinv;
        T v[6] = {rl * La.e0, rl * La.e1, rl * La.e2, Ga0, Ga1, Ga2};
        const int src = (lane - (P.ps - rs)) & (FIB_WAVE - 1);
#pragma unroll
        for (int c = 0; c < 6; ++c) v[c] = __shfl(v[c], src);
        if (src < P.n) {
#pragma unroll
          for (int c = 0; c < 9; ++c) W[c] = fma_t(v[c / 3], v[3 + c % 3], W[c]);
        }
      }
      wave_lds_sync();
      if (!more) break;
      P = Q;
      if (TB < 4) partners(P);
    }
    r0 = r1;
  }
  write_out(APW);
  if constexpr (EN || VIR) {
    double v[10];
    // every unordered term was summed twice, as (a, b) and (b, a)
    v[0] = uc * 0.5 * escale;
    const double ws = MIXED ? fscale * lscale : 1.0;
#pragma unroll
    for (int w = 0; w < 9; ++w) v[1 + w] = (double)W[w] * ws;
    tri_partials<VIR ? FIB_WAVE : APW>(v, VIR && !MIXED && APW == FIB_WAVE ? lb * NW : lb, pstride, partials);
  }
}

// ---------------------------------------------------------------------------
// MD-step mode: velocity Verlet with a per-instance adaptive timestep
// dt = min(dt_max, dx_max / |v|max), all step control on the device, so one
// step is a fixed sequence of launches that can be captured in a graph:
//   k_md_pos     Berendsen shells, half kick, drift, pinned atoms, removal
//                above the surface, displacement since the list build and
//                the exact two largest per instance;
//                k_md_decide sets the rebuild gate (two largest displacements
//                add up to more than the skin)
//   gated build  bin / sort in place / k_nbuild (skipped on the
//                device when the gate is 0)
//   forces       k_legs, k_tri, extra_pass, k_force3 MODE 2 (second half kick,
//                |v|max, shell sums)
//   k_md_ctl     time += dt, next dt, next shell factor
__device__ __forceinline__ bool in_shell(double x, double y, double z, const DInst &in, double w) {
  return x < w || x > in.lb[0] - w || y < w || y > in.lb[1] - w || z < in.bot_z + w;
}

__global__ __launch_bounds__(FIB_BLOCK) void k_md_pos(double4 *__restrict__ X,
                                                      const DInst *__restrict__ I, int NA,
                                                      double *__restrict__ V,
                                                      const double *__restrict__ F,
                                                      const double *__restrict__ Xi, StepArgs sa,
                                                      int pstride, double *__restrict__ partials,
                                                      const DCtl *__restrict__ ctl,
                                                      const double4 *__restrict__ Xb,
                                                      float *__restrict__ disp,
                                                      int Wsw, const int *__restrict__ cnt_sw,
                                                      const int *__restrict__ nbr_sw,
                                                      uint8_t *__restrict__ nst,
                                                      int *__restrict__ leave,
                                                      const int *__restrict__ binst,
                                                      const int *__restrict__ halt, int xs) {
  constexpr bool NT = (FIB_NT_LD & 8) != 0, NTS = (FIB_NT_ST & 8) != 0;
  const int lb = xcd_remap(blockIdx.x, gridDim.x, xs);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  // every load asked for at once (see k_legs)
  const int kin = binst[lb];
  double4 x = X[i];
  const double4 xb = ld_nt<NT>(Xb + i);
  double v[3], f[3];
  for (int c = 0; c < 3; ++c) {
    v[c] = ld_nt<NT>(V + (size_t)c * NA + i);
    f[c] = ld_nt<NT>(F + (size_t)c * NA + i);
  }
  HALT_OR_RETURN(halt);
  uint32_t mi = meta_of(x);
  const DInst &in = I[kin];
  const bool live = !(mi & (META_PAD | META_DEAD));
  const double dt = ctl[kin].cfg_dt, lam = ctl[kin].cfg_lambda;
  // the two largest displacements since the build (largest, how many share
  // it, largest below it), energy taken by the shells, energy of removed
  // atoms, atoms off their near lists by their own movement; an atom out of
  // the simulation counts as displaced by 0
  double red[6] = {0.0, 1.0, -1.0e300, 0.0, 0.0, 0.0};
  if (live) {
    const int t = type_of(mi);
    const double m = sa.mass[t - 1];
    double xx[3] = {x.x, x.y, x.z};
    if (sa.shell_w > 0.0 && t < 3 && !(mi & META_FROZEN) &&
        in_shell(xx[0], xx[1], xx[2], in, sa.shell_w)) {
      red[3] = 0.5 * m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]) * (1.0 - lam * lam);
      for (int c = 0; c < 3; ++c) v[c] *= lam;
    }
    for (int c = 0; c < 3; ++c) {
      v[c] += 0.5 * f[c] * dt / m;
      xx[c] += v[c] * dt;
    }
    if (mi & META_FROZEN) {
      for (int c = 0; c < 3; ++c) {
        xx[c] = Xi[(size_t)c * NA + i];
        v[c] = 0.0;
      }
    }
    for (int c = 0; c < 3; ++c) xx[c] = fmod(xx[c] + 2. * in.lb[c], in.lb[c]);
    if (xx[2] - in.surf_z > sa.remove_dz && xx[2] < in.lb[2] - sa.remove_dz) {
      // sputtered (or backscattered): out of the simulation from now on,
      // with its kinetic energy here; its interaction energy with the atoms
      // that stay (an atom of a sputtered cluster is still bound) is booked
      // by k_md_decide from the removal list
      mi |= META_DEAD | META_LEAVING;
      red[4] = 0.5 * m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
      for (int c = 0; c < 3; ++c) v[c] = 0.0;
      x.w = __longlong_as_double((long long)((wbits(x) & ~0xffffffffull) | mi));
      const int slot = atomicAdd(&leave[0], 1);
      if (slot < FIB_LEAVE_CAP) leave[1 + slot] = i;
    }
    x.x = xx[0]; x.y = xx[1]; x.z = xx[2];
    X[i] = x;
    for (int c = 0; c < 3; ++c) st_nt<NTS>(V + (size_t)c * NA + i, v[c]);
    double e0, e1, e2;
    min_image_fast(x, xb, in, e0, e1, e2);
    const float dd = (float)sqrt(e0 * e0 + e1 * e1 + e2 * e2);
    st_nt<NTS>(disp + i, dd);
    red[0] = (double)dd;
    if (dd > sa.near_d && t < 3) {
      red[5] = 1.0;
      if (!ctl[kin].near_off) near_mark_moved(i, Wsw, cnt_sw, nbr_sw, nst);
    }
  } else {
    st_nt<NTS>(disp + i, 0.0f);
  }
  const int op[6] = {RED_TOP2, RED_TOP2_CNT, RED_TOP2_SND, RED_SUM, RED_SUM, RED_SUM};
  block_partials<6, FIB_BLOCK>(red, op, lb, pstride, partials);
}

// Interaction energy (FP64, J) of atom i with the atoms that stay in the
// simulation: every SW pair and three-body term and every Moliere pair it
// takes part in (si.f90:278-368 forms), each term divided by the number of
// its atoms that leave in the current step, so that a term is booked once.
// The lists are those of the last build, which hold every pair in range.
// Used for atoms removed in a step and for ions where they are fired.
__device__ double interaction_energy(int i, const double4 *__restrict__ X,
                                 const DInst *__restrict__ I, const FConst &fc, int Wsw,
                                 int Wion, const int *__restrict__ cnt_sw,
                                 const int *__restrict__ nbr_sw, const int *__restrict__ cnt_ion,
                                 const int *__restrict__ nbr_ion) {
  // the parameters in scalars: indexing the parameter block by species (or
  // taking its address in a lambda) would copy it to scratch memory
  const double isg00 = fc.isig[0][0], isg01 = fc.isig[0][1], isg11 = fc.isig[1][1];
  const double eps00 = fc.eps[0][0], eps01 = fc.eps[0][1], eps11 = fc.eps[1][1];
  const double lp0 = fc.leps[0][0][0], lp1 = fc.leps[0][0][1], lp2 = fc.leps[0][1][1],
               lp3 = fc.leps[1][1][1];
  const double swA = fc.A, swB = fc.B, al = fc.al, gam = fc.gamma, cut = fc.cut_sw;
  const double z1 = fc.zmol[0], z2 = fc.zmol[1], z3 = fc.zmol[2];
  const double a13 = fc.aamol[0][2], a23 = fc.aamol[1][2], a33 = fc.aamol[2][2];
  const double c0 = fc.molc[0], c1 = fc.molc[1], c2 = fc.molc[2];
  const double b0 = fc.molb[0], b1 = fc.molb[1], b2 = fc.molb[2];
  const double ie0 = fc.ie0, ec = fc.ec, rlj2 = fc.rlj2;
  auto gone = [](uint32_t m) { return (m & META_DEAD) && !(m & META_LEAVING); };
  auto leaves = [](uint32_t m) { return (m & META_LEAVING) ? 1 : 0; };
  auto isg = [=](int ta, int tb) {
    const int g = (ta == 2) + (tb == 2);
    return g == 0 ? isg00 : g == 1 ? isg01 : isg11;
  };
  auto legE = [=](int ta, int tb, double r) {  // exp(gamma / (r/sigma_ab - a)), 0 out of range
    const double rs = r * isg(ta, tb);
    return rs < cut ? exp(gam / (rs - al)) : 0.0;
  };
  auto leps = [=](int ta, int tb, int tc) {  // by the number of Ge atoms of the term
    const int g = (ta == 2) + (tb == 2) + (tc == 2);
    return g == 0 ? lp0 : g == 1 ? lp1 : g == 2 ? lp2 : lp3;
  };
  const double4 xi = X[i];
  const uint32_t mi = meta_of(xi);
  const DInst &in = I[inst_of(mi)];
  const int ti = type_of(mi);
  double e = 0.0;
  if (ti < 3) {
    const int ci = min(cnt_sw[i], Wsw);
    const int *ri = nbr_sw + (size_t)i * Wsw;
    for (int a = 0; a < ci; ++a) {
      const int j = ri[a];
      const double4 xj = X[j];
      const uint32_t mj = meta_of(xj);
      if (gone(mj)) continue;
      const int tj = type_of(mj);
      double d0, d1, d2;  // x_i - x_j
      min_image_fast(xi, xj, in, d0, d1, d2);
      const double rij = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
      const double rs = rij * isg(ti, tj);
      if (!(rs < cut)) continue;
      const double rs2 = rs * rs;
      const int g = (ti == 2) + (tj == 2);
      const double eij = g == 0 ? eps00 : g == 1 ? eps01 : eps11;
      const double phi = eij * swA * (swB / (rs2 * rs2) - 1.0) * exp(1.0 / (rs - al));
      e += phi / (1 + leaves(mj));
      const double Eij = legE(ti, tj, rij);
      // terms centred on j with legs to i and to another k of j's list
      const int cj = min(cnt_sw[j], Wsw);
      const int *rj = nbr_sw + (size_t)j * Wsw;
      for (int b = 0; b < cj; ++b) {
        const int k = rj[b];
        if (k == i) continue;
        const double4 xk = X[k];
        const uint32_t mk = meta_of(xk);
        if (gone(mk)) continue;
        const int tk = type_of(mk);
        double f0, f1, f2;  // x_k - x_j
        min_image_fast(xk, xj, in, f0, f1, f2);
        const double rjk = sqrt(f0 * f0 + f1 * f1 + f2 * f2);
        const double Ejk = legE(tj, tk, rjk);
        if (Ejk == 0.0) continue;
        const double cs = (d0 * f0 + d1 * f1 + d2 * f2) / (rij * rjk);
        const double D = cs + 1.0 / 3.0;
        e += leps(ti, tj, tk) * Eij * Ejk * D * D / (1 + leaves(mj) + leaves(mk));
      }
      // terms centred on i with legs to j and to a later k of i's list
      for (int b = a + 1; b < ci; ++b) {
        const int k = ri[b];
        const double4 xk = X[k];
        const uint32_t mk = meta_of(xk);
        if (gone(mk)) continue;
        const int tk = type_of(mk);
        double f0, f1, f2;  // x_i - x_k
        min_image_fast(xi, xk, in, f0, f1, f2);
        const double rik = sqrt(f0 * f0 + f1 * f1 + f2 * f2);
        const double Eik = legE(ti, tk, rik);
        if (Eik == 0.0) continue;
        const double cs = (d0 * f0 + d1 * f1 + d2 * f2) / (rij * rik);
        const double D = cs + 1.0 / 3.0;
        e += leps(ti, tj, tk) * Eij * Eik * D * D / (1 + leaves(mj) + leaves(mk));
      }
    }
  }
  // Moliere pairs (si.f90:426-446): both atoms fired, r < 2.5 sigma; one of
  // the two is Ga (the ion list holds no Si-Si or Si-Ge pair)
  const bool ifired = !(ti == 3 && orig_of(xi) >= in.nsg + in.impact);
  const int cn = min(cnt_ion[i], Wion);
  const int *rn = nbr_ion + (size_t)i * Wion;
  for (int a = 0; ifired && a < cn; ++a) {
    const int j = rn[a];
    const double4 xj = X[j];
    const uint32_t mj = meta_of(xj);
    if (gone(mj)) continue;
    const int tj = type_of(mj);
    if (tj == 3 && orig_of(xj) >= in.nsg + in.impact) continue;
    double d0, d1, d2;
    min_image_fast(xi, xj, in, d0, d1, d2);
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    if (!(r2 < rlj2)) continue;
    const double r = sqrt(r2);
    const int other = ti == 3 ? tj : ti;  // the partner of the Ga atom
    const double aa = other == 1 ? a13 : other == 2 ? a23 : a33;
    const double zi = ti == 1 ? z1 : ti == 2 ? z2 : z3, zj = tj == 1 ? z1 : tj == 2 ? z2 : z3;
    const double zz = ie0 * zi * zj * ec * ec;
    const double x = r / aa;
    const double sa = c0 * exp(-b0 * x) + c1 * exp(-b1 * x) + c2 * exp(-b2 * x);
    e += zz / r * sa / (1 + leaves(mj));
  }
  return e;
}

// Rebuild gates of the step: each instance whose two largest displacements
// since the build add up to more than the skin (only then can a pair the
// build left out have come within the cutoff), and whether there is any.
#define DECIDE_T 256  // threads of k_md_decide (a small block keeps the removal path in registers)
static_assert(FIB_LEAVE_CAP == DECIDE_T, "one thread per listed removal");
__global__ __launch_bounds__(DECIDE_T) void k_md_decide(
    int ninst, const DInst *__restrict__ I, DCtl *__restrict__ ctl, double skin,
    int *__restrict__ gate, int *__restrict__ leave, double4 *__restrict__ X, const FConst fc,
    int Wsw, int Wion, const int *__restrict__ cnt_sw, const int *__restrict__ nbr_sw,
    const int *__restrict__ cnt_ion, const int *__restrict__ nbr_ion, int how, const RedSpec rs,
    const double *__restrict__ partials, int pstride, const double *__restrict__ tmp, int nch,
    const int *__restrict__ halt) {
  // halted: no build in this step either (the host restores the flag)
  if (halt && *halt) {
    if (threadIdx.x == 0) gate[0] = 0;
    return;
  }
  __shared__ int s_w[DECIDE_T / FIB_WAVE];
  __shared__ int s_any;
  __shared__ int s_list[FIB_LEAVE_CAP];
  __shared__ double s_e[FIB_LEAVE_CAP];
  const int t = threadIdx.x, lane = t % FIB_WAVE;
  const int wv = __builtin_amdgcn_readfirstlane(t / FIB_WAVE);
  // the rest of k_md_pos' reductions, an instance per wavefront
  if (how != FIN_DONE) {
    for (int k = wv; k < ninst; k += DECIDE_T / FIB_WAVE)
      fin_finish<6>(how, k, I[k], partials, pstride, tmp, nch, rs, ctl[k]);
    __syncthreads();
  }
  // atoms removed in this step: their interaction energy with the atoms that
  // stay goes to the energy carried out, summed in atom order (the list is
  // filled in arbitrary order and sorted here), so the ledger is the same
  // for an instance alone or in any batch
  const int nleave = leave[0];
  if (nleave > 0) {
    const int n = min(nleave, FIB_LEAVE_CAP);
    s_list[t] = t < n ? leave[1 + t] : 0x7fffffff;
    __syncthreads();
    for (int k = 2; k <= FIB_LEAVE_CAP; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        const int u = t ^ j;
        if (u > t) {
          const int a = s_list[t], b = s_list[u];
          if ((a > b) == ((t & k) == 0)) { s_list[t] = b; s_list[u] = a; }
        }
        __syncthreads();
      }
    if (t < n)
      s_e[t] = interaction_energy(s_list[t], X, I, fc, Wsw, Wion, cnt_sw, nbr_sw, cnt_ion,
                                  nbr_ion);
    __syncthreads();
    if (t == 0) {
      for (int q = 0; q < n; ++q) ctl[inst_of(meta_of(X[s_list[q]]))].e_out_step += s_e[q];
      if (nleave > FIB_LEAVE_CAP) ctl[0].leave_overflow = 1;
      leave[0] = 0;
    }
    __syncthreads();
    if (t < n) {
      double4 &x = X[s_list[t]];
      x.w = __longlong_as_double((long long)(wbits(x) & ~(uint64_t)META_LEAVING));
    }
  }
  // one workgroup; behind the gates, the prefix over instances of the real
  // cells of the gated ones (the cell numbering of a gated k_nbuild)
  int *cplan = gate + 1 + ninst;
  if (t == 0) s_any = 0;
  __syncthreads();
  int carry = 0;
  for (int k0 = 0; k0 < ninst; k0 += DECIDE_T) {
    const int k = k0 + t;
    int g = 0, w = 0;
    if (k < ninst) {
      const DCtl &c = ctl[k];
      const double m2 = c.nmaxdisp >= 2.0 ? c.maxdisp : fmax(c.maxdisp2, 0.0);
      g = (c.maxdisp + m2 > skin) ? 1 : 0;
      ctl[k].maxdisp2 = m2;  // the effective second maximum, for extra_pass
      // with many atoms off their near lists, telling their partners costs
      // more than the lists that are left give
      if (c.movers * 16.0 > (double)I[k].natm) ctl[k].near_off = 1;
      gate[1 + k] = g;
      if (g) w = I[k].nc[0] * I[k].nc[1] * I[k].nc[2];
    }
    // inclusive scan of w: in the wave, then over the waves' totals
    int sc = w;
    for (int o = 1; o < FIB_WAVE; o <<= 1) {
      const int y = __shfl_up(sc, o);
      if (lane >= o) sc += y;
    }
    if (lane == FIB_WAVE - 1) s_w[wv] = sc;
    if (__ballot(g) != 0ull && lane == 0) s_any = 1;
    __syncthreads();
    int before = carry;
    for (int v = 0; v < wv; ++v) before += s_w[v];
    if (k < ninst) cplan[k] = before + sc - w;
    for (int v = 0; v < DECIDE_T / FIB_WAVE; ++v) carry += s_w[v];
    __syncthreads();  // s_w is rewritten by the next chunk
  }
  if (t == 0) {
    cplan[ninst] = carry;
    gate[0] = s_any;
  }
}

// A fired ion brings its interaction energy with the atoms near its start
// point in with its kinetic energy (k_set_atom books the latter); q is its
// unsorted index atom_off + orig, evaluated after the lists were rebuilt.
__global__ void k_fire_energy(int q, const int *__restrict__ inv, const double4 *__restrict__ X,
                              const DInst *__restrict__ I, const FConst fc, int Wsw, int Wion,
                              const int *__restrict__ cnt_sw, const int *__restrict__ nbr_sw,
                              const int *__restrict__ cnt_ion, const int *__restrict__ nbr_ion,
                              DCtl *__restrict__ ctl) {
  if (threadIdx.x != 0) return;
  const int p = inv[q];
  const double e = interaction_energy(p, X, I, fc, Wsw, Wion, cnt_sw, nbr_sw, cnt_ion, nbr_ion);
  ctl[inst_of(meta_of(X[p]))].e_in += e;
}

// After the step's second half kick: advance time, choose the next dt and
// the next Berendsen factor of the shells.
// One wavefront per instance, which first finishes k_force3's reductions.
__global__ __launch_bounds__(FIB_WAVE) void k_md_ctl(const DInst *__restrict__ I,
                                                     DCtl *__restrict__ ctl, StepArgs sa, int how,
                                                     const RedSpec rs,
                                                     const double *__restrict__ partials,
                                                     int pstride, const double *__restrict__ tmp,
                                                     int nch, const int *__restrict__ halt) {
  HALT_OR_RETURN(halt);
  const int k = blockIdx.x;
  DCtl &c = ctl[k];
  fin_finish<4>(how, k, I[k], partials, pstride, tmp, nch, rs, c);
  if (threadIdx.x != 0) return;
  c.cfg_time += c.cfg_dt;
  c.cfg_steps += 1.0;
  c.cfg_dt_min = fmin(c.cfg_dt_min, c.cfg_dt);
  c.e_bath += c.e_bath_step;
  c.e_out += c.e_out_step;
  const double dt = c.vmax > 0.0 ? fmin(sa.dt_max, sa.dx_max / c.vmax) : sa.dt_max;
  c.cfg_dt = dt;
  double lam = 1.0;
  if (sa.shell_w > 0.0 && c.n_shell > 0.0 && c.ke_shell > 0.0) {
    const double ts = c.ke_shell / (3.0 * c.n_shell * sa.kB);
    lam = sqrt(1.0 + dt / sa.tau * (sa.ttar / ts - 1.0));
  }
  c.cfg_lambda = lam;
}

// dt from the current |v|max (DCtl::vmax, from k_sums); reset also zeroes the
// clock and the shell factor.
__global__ void k_md_init(int ninst, DCtl *__restrict__ ctl, StepArgs sa, int reset) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ninst) return;
  DCtl &c = ctl[k];
  c.cfg_dt = c.vmax > 0.0 ? fmin(sa.dt_max, sa.dx_max / c.vmax) : sa.dt_max;
  if (reset) {
    c.cfg_time = 0.0;
    c.cfg_steps = 0.0;
    c.cfg_lambda = 1.0;
    c.cfg_dt_min = 1.0e300;
    c.e_bath = c.e_out = c.e_in = 0.0;
    c.leave_overflow = 0;
  }
}

// Cascade outputs: removed SW atoms (sputter yield), removed ions, displaced
// SW atoms (farther than disp_r from their initial site Xi), height of the
// instance's most recently fired ion.
__global__ __launch_bounds__(FIB_BLOCK) void k_md_report(const double4 *__restrict__ X,
                                                         const DInst *__restrict__ I, int NA,
                                                         const double *__restrict__ Xi,
                                                         StepArgs sa, int pstride,
                                                         double *__restrict__ partials) {
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  const double4 x = X[i];
  const uint32_t mi = meta_of(x);
  const int kin = __builtin_amdgcn_readfirstlane(inst_of(mi));
  const DInst &in = I[kin];
  double v[4] = {0.0, 0.0, 0.0, -1.0e300};
  if (!(mi & META_PAD)) {
    const int t = type_of(mi);
    if (mi & META_DEAD) {
      if (t < 3) v[0] = 1.0; else v[1] = 1.0;
    } else if (t < 3) {
      double e0, e1, e2;
      double4 xi;
      xi.x = Xi[i]; xi.y = Xi[(size_t)NA + i]; xi.z = Xi[2 * (size_t)NA + i]; xi.w = 0.0;
      min_image_fast(x, xi, in, e0, e1, e2);
      if (e0 * e0 + e1 * e1 + e2 * e2 > sa.disp_r * sa.disp_r) v[2] = 1.0;
    }
    if (t == 3 && orig_of(x) == in.nsg + in.impact - 1) v[3] = (mi & META_DEAD) ? 1.0e300 : x.z;
  }
  const int op[4] = {0, 0, 0, 1};
  block_partials<4, FIB_BLOCK>(v, op, lb, pstride, partials);
}

// ---------------------------------------------------------------------------
// force pass 3: own terms + the G entries neighbours wrote for this atom;
// MODE 0 = store forces, MODE 1 = reference velocity update
// (timeint.f90:231-236) + thermostat sums; MODE 2 = MD-step mode.
// Bound by the gather of the partners' entries (and, in small batches, by
// the chain of dependent loads): two batches of F3_BATCH legs, the partners'
// places first, then their entries, all of a batch in flight at once.  The
// reaction on the centre comes summed from k_tri, which holds the terms in
// LDS, instead of from its own G entries read again, and G has three
// components where no energies are wanted: 24 B per atom and 4.2 entries of
// 12 B (mixed) or 24 B for 8.4 of 16 or 32.  k_force3 and, for the sums,
// k_tri: 4 x 512 k atoms, mixed, 118 -> 102 us and 206 -> 211; 2 x 512 k,
// FP64, 109 -> 86 and 174 -> 180; 64 x 4 k, mixed, 24 -> 21.5 and 39.5 ->
// 41.4.
#define F3_BATCH 4
template <bool MIXED, bool EN, int MODE>
__global__ __launch_bounds__(FIB_BLOCK) void k_force3(
    const double4 *__restrict__ X, const DInst *__restrict__ I, int NA, int Wsw,
    const int *__restrict__ nbr_sw, const uint16_t *__restrict__ rk_sw,
    const uint8_t *__restrict__ off_sw, const typename GRec<MIXED, EN>::type *__restrict__ G,
    const uint32_t *__restrict__ RA, const double *__restrict__ Gown,
    const double *__restrict__ Gown_u,
    const uint64_t *__restrict__ amask, const int *__restrict__ cnt_sw,
    const double *__restrict__ Fpart, const double *__restrict__ upart, double fscale,
    double escale, double *__restrict__ Fout, double *__restrict__ uout, double *__restrict__ V,
    StepArgs sa, int pstride, double *__restrict__ partials, const DCtl *__restrict__ ctl,
    const typename Prec<MIXED>::T4 *__restrict__ EX,
    const typename Prec<MIXED>::T4 *__restrict__ EXself, const uint64_t *__restrict__ exmask,
    const int *__restrict__ binst, const int *__restrict__ halt, int xs) {
  typedef typename Prec<MIXED>::T4 T4;
  typedef typename GRec<MIXED, EN>::type GV;
  constexpr bool NT = (FIB_NT_LD & 4) != 0, NTS = (FIB_NT_ST & 4) != 0;
  const int lb = xcd_remap(blockIdx.x, gridDim.x, xs);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  // what the pass needs first, asked for at once (see k_legs); entries of
  // legs the atom does not have are not used
  const int kin = binst[lb];
  const double4 xi = X[i];
  const uint64_t am = ld_nt<NT>(amask + i);
  const double fp[3] = {ld_nt<NT>(Fpart + i), ld_nt<NT>(Fpart + (size_t)NA + i),
                        ld_nt<NT>(Fpart + 2 * (size_t)NA + i)};
  const double go[3] = {ld_nt<NT>(Gown + i), ld_nt<NT>(Gown + (size_t)NA + i),
                        ld_nt<NT>(Gown + 2 * (size_t)NA + i)};
  uint32_t ra[F3_BATCH];
#pragma unroll
  for (int u = 0; u < F3_BATCH; ++u) ra[u] = ld_nt<NT>(RA + (size_t)u * NA + i);
  double vold[3] = {0, 0, 0};
  if (MODE == 2)
    for (int c = 0; c < 3; ++c) vold[c] = ld_nt<NT>(V + (size_t)c * NA + i);
  HALT_OR_RETURN(halt);
  const uint32_t mi = meta_of(xi);
  const DInst &in = I[kin];
  const bool live = !(mi & (META_PAD | META_DEAD));
  double f0 = 0, f1 = 0, f2 = 0, u = 0;
  if (live) {
    f0 = fp[0];
    f1 = fp[1];
    f2 = fp[2];
    if (EN) u = upart[i];
    const size_t row = (size_t)i * Wsw;
    // the reaction on the centre, and the forces that the partners' terms put
    // on this atom, from the places k_tri noted for its legs
    double g0 = go[0], g1 = go[1], g2 = go[2], gu = EN ? Gown_u[i] : 0.0;
    const int na = __popcll(am);
    auto partner = [&](uint32_t at, GV &g) {
      if (at != ~0u) {
        g = G[at];
      } else {
        g.x = g.y = g.z = 0;
        if constexpr (EN) g.w = 0;
      }
    };
    auto plus = [&](const GV &g) {
      g0 += (double)g.x; g1 += (double)g.y; g2 += (double)g.z;
      if constexpr (EN) gu += (double)g.w;
    };
    GV theirs[F3_BATCH], theirs2[F3_BATCH];
    uint32_t ra2[F3_BATCH];
#pragma unroll
    for (int u = 0; u < F3_BATCH; ++u) {
      partner(u < na ? ra[u] : ~0u, theirs[u]);
      ra2[u] = F3_BATCH + u < na ? ld_nt<NT>(RA + (size_t)(F3_BATCH + u) * NA + i) : ~0u;
    }
#pragma unroll
    for (int u = 0; u < F3_BATCH; ++u) partner(ra2[u], theirs2[u]);
#pragma unroll
    for (int u = 0; u < F3_BATCH; ++u)
      if (u < na) plus(theirs[u]);
#pragma unroll
    for (int u = 0; u < F3_BATCH; ++u)
      if (F3_BATCH + u < na) plus(theirs2[u]);
    for (int n = 2 * F3_BATCH; n < na; ++n) {
      GV g;
      partner(ld_nt<NT>(RA + (size_t)n * NA + i), g);
      plus(g);
    }
    // vertex terms outside the centre's list (extra_pass), when there are any
    if (ctl[kin].extra_any) {
      const T4 gs = EXself[i];
      g0 += (double)gs.x; g1 += (double)gs.y; g2 += (double)gs.z;
      if (EN) gu += (double)gs.w;
      const int cs = min(cnt_sw[i], Wsw);
      for (int k = 0; k < cs; ++k) {
        const int j = nbr_sw[row + k];
        const uint64_t mj = exmask[j];
        if (!mj) continue;
        const int sr = rk_sw[row + k];
        const int r = (sr & RK_SLOT) ? (sr & ~RK_SLOT)
                                     : off_sw[(size_t)j * OFF_W + 26 - (sr >> 8)] + (sr & 0xff);
        if (r < Wsw && ((mj >> r) & 1ull)) {
          const T4 g = EX[(size_t)r * NA + j];
          g0 += (double)g.x; g1 += (double)g.y; g2 += (double)g.z;
          if (EN) gu += (double)g.w;
        }
      }
    }
    f0 += g0 * fscale; f1 += g1 * fscale; f2 += g2 * fscale;
    if (EN) u += gu * escale;
  }
  if (MODE == 0) {
    if (live) {
      Fout[i] = f0; Fout[(size_t)NA + i] = f1; Fout[2 * (size_t)NA + i] = f2;
      if (EN) uout[i] = u;
    }
    return;
  }
  if (MODE == 2) {
    // MD-step mode: second half kick with the instance's dt; F = F'
    // reductions: |v|max, kinetic energy, shell sum m v^2 and count
    double v[4] = {0, 0, 0, 0};
    if (live) {
      const int t = type_of(mi);
      const double m = sa.mass[t - 1];
      const double dt = ctl[kin].cfg_dt;
      const bool pinned = (mi & META_FROZEN) != 0;
      const double fn[3] = {f0, f1, f2};
      double vv[3];
      for (int c = 0; c < 3; ++c) {
        const size_t a = (size_t)c * NA + i;
        vv[c] = pinned ? 0.0 : vold[c] + 0.5 * fn[c] * dt / m;
        st_nt<NTS>(V + a, vv[c]);
        st_nt<NTS>(Fout + a, fn[c]);
      }
      const double v2 = vv[0] * vv[0] + vv[1] * vv[1] + vv[2] * vv[2];
      v[0] = sqrt(v2);
      v[1] = 0.5 * m * v2;
      if (sa.shell_w > 0.0 && t < 3 && !pinned && in_shell(xi.x, xi.y, xi.z, in, sa.shell_w)) {
        v[2] = m * v2;
        v[3] = 1.0;
      }
    }
    const int op[4] = {1, 0, 0, 0};
    block_partials<4, FIB_BLOCK>(v, op, lb, pstride, partials);
    return;
  }
  // MODE 1: V += 0.5*(F+Fp)*Ts/m ; F = Fp ; thermostat / temperature sums
  double v[5] = {0, 0, 0, 0, 0};
  if (live) {
#pragma clang fp contract(off)
    const int t = type_of(mi);
    const double m = sa.mass[t - 1];
    double vv[3];
    const double fn[3] = {f0, f1, f2};
    for (int c = 0; c < 3; ++c) {
      const size_t a = (size_t)c * NA + i;
      vv[c] = V[a] + 0.5 * (Fout[a] + fn[c]) * sa.ts / m;
      V[a] = vv[c];
      Fout[a] = fn[c];
    }
    if (t < 3) {
      const double m2 = m * (vv[0] * vv[0] + vv[1] * vv[1] + vv[2] * vv[2]);
      v[0] = m2;  // global temperature sum (temp.f90:196-198)
      const double nm = 1.0e-9;
      const bool xs = (xi.x < sa.sidewidth * nm) || (xi.x > (in.lb[0] - sa.sidewidth * nm));
      const bool ys = (xi.y < sa.sidewidth * nm) || (xi.y > (in.lb[1] - sa.sidewidth * nm));
      const bool zc = (xi.z < sa.outz[0] * in.lb[2] / 10.0) || (xi.z > sa.outz[3] * in.lb[2] / 10.0);
      if (xs || (ys && zc)) { v[1] = m2; v[2] = 1.0; }
    }
    v[3] = 0.5 * m * (vv[0] * vv[0] + vv[1] * vv[1] + vv[2] * vv[2]);
    v[4] = sqrt(vv[0] * vv[0] + vv[1] * vv[1] + vv[2] * vv[2]);
  }
  const int op[5] = {0, 0, 0, 0, 1};
  block_partials<5, FIB_BLOCK>(v, op, lb, pstride, partials);
}


// ---------------------------------------------------------------------------
// onestep head (timeint.f90:165-203): Berendsen scaling (adjusttemp
// temp.f90:160-179 or controlsidetemp :32-67), X += V*Ts + 0.5*F*Ts^2/m,
// freezsidesN (tools.f90:38-51), rebox (:26-36), frzsptrdatms (temp.f90:99-127).
// Reductions: sum m v^2 of the rescaled V (equilibration temperature) and
// max 0.5 m v^2/ec (calc_atm's test, timeint.f90:284-293).
__global__ __launch_bounds__(FIB_BLOCK) void k_pos(double4 *__restrict__ X,
                                                   const DInst *__restrict__ I, int NA,
                                                   double *__restrict__ V, double *__restrict__ F,
                                                   const double *__restrict__ Xi, StepArgs sa,
                                                   int pstride, double *__restrict__ partials,
                                                   DCtl *__restrict__ ctl,
                                                   const double4 *__restrict__ Xb,
                                                   float *__restrict__ disp, int Wsw,
                                                   const int *__restrict__ cnt_sw,
                                                   const int *__restrict__ nbr_sw,
                                                   uint8_t *__restrict__ nst) {
#pragma clang fp contract(off)
  const int nb = gridDim.x;
  const int lb = xcd_remap(blockIdx.x, nb);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  double4 x = X[i];
  const uint32_t mi = meta_of(x);
  // every block lies inside one instance: make the index wave-uniform so the
  // instance record is read with scalar loads
  const int kin = __builtin_amdgcn_readfirstlane(inst_of(mi));
  const DInst &in = I[kin];
  const bool live = !(mi & (META_PAD | META_DEAD));
  // slots: thermostat sum, max KE, max displacement, and the displacement
  // again as the second maximum (extra_pass tests maxdisp + maxdisp2)
  double red[4] = {0.0, -1.0, 0.0, 0.0};
  if (live) {
    const int t = type_of(mi);
    const double m = sa.mass[t - 1];
    double v[3], f[3], xx[3] = {x.x, x.y, x.z};
    for (int c = 0; c < 3; ++c) {
      v[c] = V[(size_t)c * NA + i];
      f[c] = F[(size_t)c * NA + i];
    }
    if (sa.mode == 0) {
      if (t < 3) {
        const double s = sqrt(1. + sa.ts / sa.tau * (sa.ttar / sa.temp - 1.));
        for (int c = 0; c < 3; ++c) v[c] = s * v[c];
        red[0] = m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
      }
    } else if (sa.mode == 1) {
      const DCtl &c0 = ctl[kin];
      if (t < 3 && c0.side_cnt > 0.0) {
        const double nm = 1.0e-9;
        const bool xs = (xx[0] < sa.sidewidth * nm) || (xx[0] > (in.lb[0] - sa.sidewidth * nm));
        const bool ys = (xx[1] < sa.sidewidth * nm) || (xx[1] > (in.lb[1] - sa.sidewidth * nm));
        const bool zc = (xx[2] < sa.outz[0] * in.lb[2] / 10.0) ||
                        (xx[2] > sa.outz[3] * in.lb[2] / 10.0);
        if (xs || (ys && zc)) {
          const double tside = c0.side_sum / 3. / c0.side_cnt / sa.kB;
          const double s = sqrt(1. + sa.ts / sa.tau * (sa.ttar / tside - 1.));
          for (int c = 0; c < 3; ++c) v[c] = s * v[c];
        }
      }
    }
    for (int c = 0; c < 3; ++c) xx[c] = xx[c] + v[c] * sa.ts + 0.5 * f[c] * sa.ts * sa.ts / m;
    if (mi & META_FROZEN) {
      for (int c = 0; c < 3; ++c) {
        xx[c] = Xi[(size_t)c * NA + i];
        v[c] = 0.;
      }
    }
    for (int c = 0; c < 3; ++c) xx[c] = fmod(xx[c] + 2. * in.lb[c], in.lb[c]);
    if (sa.frz) {
      const double T = in.lb[2];
      const double z = xx[2];
      const double buffer = 0.3;
      bool zero = false;
      if ((z > sa.outz[0] * T / 10.0) && (z < sa.outz[1] * T / 10.0)) {
        xx[2] = sa.atomz[0] * T / 10.0; zero = true;
      } else if ((z > sa.outz[2] * T / 10.0) && (z < sa.outz[3] * T / 10.0)) {
        xx[2] = sa.atomz[1] * T / 10.0; zero = true;
      } else if ((z > (sa.atomz[0] - buffer) * T / 10.0) && (z < (sa.atomz[0] + buffer) * T / 10.0)) {
        zero = true;
      } else if ((z > (sa.atomz[1] - buffer) * T / 10.0) && (z < (sa.atomz[1] + buffer) * T / 10.0)) {
        zero = true;
      } else if ((z > (sa.ionz - buffer) * T / 10.0) && (z < (sa.ionz + buffer) * T / 10.0)) {
        zero = true;
      }
      if (zero)
        for (int c = 0; c < 3; ++c) { v[c] = 0.0; f[c] = 0.0; }
    }
    red[1] = 0.5 * m * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]) / sa.ec;
    x.x = xx[0]; x.y = xx[1]; x.z = xx[2];
    X[i] = x;
    {
      // displacement since the list build (minimum image across the rebox)
      double e0, e1, e2;
      min_image_fast(x, Xb[i], in, e0, e1, e2);
      const double dd = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
      disp[i] = (float)dd;
      red[2] = dd;
      red[3] = dd;
      if ((float)dd > sa.near_d && t < 3) near_mark_moved(i, Wsw, cnt_sw, nbr_sw, nst);
    }
    for (int c = 0; c < 3; ++c) {
      V[(size_t)c * NA + i] = v[c];
      F[(size_t)c * NA + i] = f[c];
    }
  }
  const int op[4] = {0, 1, 1, 1};
  block_partials<4, FIB_BLOCK>(red, op, lb, pstride, partials);
}

// Thermostat / temperature sums of the current state (same as k_force_b's
// MODE 1 reduction without the velocity update).
__global__ __launch_bounds__(FIB_BLOCK) void k_sums(const double4 *__restrict__ X,
                                                    const DInst *__restrict__ I, int NA,
                                                    const double *__restrict__ V, StepArgs sa,
                                                    int pstride, double *__restrict__ partials,
                                                    DCtl *__restrict__ ctl) {
  const int nb = gridDim.x;
  const int lb = xcd_remap(blockIdx.x, nb);
  const int i = lb * FIB_BLOCK + threadIdx.x;
  const double4 xi = X[i];
  const uint32_t mi = meta_of(xi);
  // every block lies inside one instance: make the index wave-uniform so the
  // instance record is read with scalar loads
  const int kin = __builtin_amdgcn_readfirstlane(inst_of(mi));
  const DInst &in = I[kin];
  const bool live = !(mi & (META_PAD | META_DEAD));
  double v[5] = {0, 0, 0, 0, 0};
  if (live) {
    const int t = type_of(mi);
    const double m = sa.mass[t - 1];
    const double a = V[i], b = V[(size_t)NA + i], c = V[2 * (size_t)NA + i];
    const double vv = a * a + b * b + c * c;
    if (t < 3) {
      const double m2 = m * vv;
      v[0] = m2;
      const double nm = 1.0e-9;
      const bool xs = (xi.x < sa.sidewidth * nm) || (xi.x > (in.lb[0] - sa.sidewidth * nm));
      const bool ys = (xi.y < sa.sidewidth * nm) || (xi.y > (in.lb[1] - sa.sidewidth * nm));
      const bool zc = (xi.z < sa.outz[0] * in.lb[2] / 10.0) || (xi.z > sa.outz[3] * in.lb[2] / 10.0);
      if (xs || (ys && zc)) { v[1] = m2; v[2] = 1.0; }
    }
    v[3] = 0.5 * m * vv;
    v[4] = sqrt(vv);
  }
  const int op[5] = {0, 0, 0, 0, 1};
  block_partials<5, FIB_BLOCK>(v, op, lb, pstride, partials);
}

// ---------------------------------------------------------------------------
// host <-> device layout conversion
__global__ void k_import(int inst, DInst in, int NA, const double *__restrict__ hx,
                         const double *__restrict__ hv, const int32_t *__restrict__ at,
                         const int32_t *__restrict__ xs, const double *__restrict__ hxi,
                         double4 *__restrict__ X0, double4 *__restrict__ X1,
                         double *__restrict__ V0, double *__restrict__ V1,
                         double *__restrict__ F0, double *__restrict__ F1,
                         double *__restrict__ Xi0, double *__restrict__ Xi1,
                         int *__restrict__ inv) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= in.natm_pad) return;
  const int p = in.atom_off + o;
  double4 x;
  uint64_t w;
  double v[3] = {0, 0, 0}, xi[3] = {0, 0, 0};
  if (o < in.natm) {
    x.x = hx[o]; x.y = hx[in.natm + o]; x.z = hx[2 * in.natm + o];
    uint32_t m = (uint32_t)at[o] & META_TYPE_MASK;
    if (xs && xs[o] > 0) m |= META_FROZEN;
    m |= (uint32_t)inst << META_INST_SHIFT;
    w = ((uint64_t)(uint32_t)o << 32) | m;
    for (int c = 0; c < 3; ++c) {
      v[c] = hv ? hv[(size_t)c * in.natm + o] : 0.0;
      xi[c] = hxi ? hxi[(size_t)c * in.natm + o] : (c == 0 ? x.x : (c == 1 ? x.y : x.z));
    }
  } else {
    x.x = x.y = x.z = 0.0;
    w = ((uint64_t)(uint32_t)o << 32) | META_PAD | ((uint32_t)inst << META_INST_SHIFT);
  }
  x.w = __longlong_as_double((long long)w);
  X0[p] = x; X1[p] = x;
  for (int c = 0; c < 3; ++c) {
    const size_t a = (size_t)c * NA + p;
    V0[a] = v[c]; V1[a] = v[c];
    F0[a] = 0.0; F1[a] = 0.0;
    Xi0[a] = xi[c]; Xi1[a] = xi[c];
  }
  inv[p] = p;
}

// One launch for all that a call hands back (three to five kernels of 3 us
// and their gaps before, for 4 k atoms).
__global__ void k_export(DInst in, int NA, const double4 *__restrict__ X, const ExportArgs ex) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0) {
    constexpr int NWORD = sizeof(DCtl) / sizeof(uint32_t);
    if (ex.ctl_out)
      for (int k = threadIdx.x; k < NWORD; k += blockDim.x)
        reinterpret_cast<uint32_t *>(ex.ctl_out)[k] =
            reinterpret_cast<const uint32_t *>(ex.ctl)[k];
    if (ex.utot && threadIdx.x == 0) *ex.utot = ex.ctl->utot;
  }
  if (o >= in.natm_pad) return;
  const int p = in.atom_off + o;
  const double4 x = X[p];
  if (meta_of(x) & META_PAD) return;
  const size_t g = orig_of(x), n = in.natm;
  if (ex.x) {
    ex.x[g] = x.x;
    ex.x[n + g] = x.y;
    ex.x[2 * n + g] = x.z;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
    if (ex.vec[q])
      for (int c = 0; c < 3; ++c) ex.vec[q][c * n + g] = ex.src[q][(size_t)c * NA + p];
  if (ex.scal) ex.scal[g] = ex.scal_src[p];
}

// Places atom p (a fired ion) and books its change of kinetic energy as
// energy brought into its instance.
__global__ void k_set_atom(int NA, double4 *__restrict__ X, double *__restrict__ V, int p,
                           double x0, double x1, double x2, double v0, double v1, double v2,
                           StepArgs sa, DCtl *__restrict__ ctl) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double4 x = X[p];
  const uint32_t m = meta_of(x);
  const double w0 = V[p], w1 = V[(size_t)NA + p], w2 = V[2 * (size_t)NA + p];
  ctl[inst_of(m)].e_in += 0.5 * sa.mass[type_of(m) - 1] *
                          ((v0 * v0 + v1 * v1 + v2 * v2) - (w0 * w0 + w1 * w1 + w2 * w2));
  x.x = x0; x.y = x1; x.z = x2;
  X[p] = x;
  V[p] = v0; V[(size_t)NA + p] = v1; V[2 * (size_t)NA + p] = v2;
}

// ---------------------------------------------------------------------------
// launchers
static inline int nblk(long n, int b) { return (int)((n + b - 1) / b); }
// grid of a GRID_STRIDE kernel over n elements
static inline int gcap(long n) { return std::max(1, std::min(nblk(n, FIB_BLOCK), GRID_CAP)); }

// Blocks (as a power of two) that an XCD takes in turn: an eighth of the
// largest instance, so that each instance meets every XCD, and at least 32
// (8 k atoms, about a layer of cells of a 512 k slab), so that most of a
// block's neighbours are read by the same XCD.
static int xcd_shift(const DevBufs &d) {
  int s = 5;
  while ((8 << s) < d.max_pad / FIB_BLOCK) ++s;
  return s;
}

// Cells per wavefront of the list build: a wavefront builds its cells one
// after the other, each with two or three dependent loads, so a small batch
// takes few per wavefront and a large one eight, which share the decoding of
// their position.  us of a build of a crystal by 1, 2, 4 and 8 cells:
//     1,000 cells  14   19   27   46      63,960 cells 109  103  102  108
//     8,000        25   24   31   49     140,608       227  204  196  201
//    17,576        39   40   46   54     257,920       392  352  335  335
//    34,816        67   63   66   81     571,787       882  772  719  701
// A gated build has the cells of a few of the batch's instances, hence the
// line between 2 and 4 above that of whole builds: MD of 64 x 4 k atoms
// (121,600 cells) 48 ms by 1 or 2 cells, 50 by 4, 53 by 8; of 12 uneven slabs
// (254,772 cells) 61.5, 59.0, 59.0 and 60.5.
int nb_cells_auto(int total_cells) {
  return total_cells < 32768 ? 1 : total_cells < 131072 ? 2 : total_cells < 262144 ? 4 : 8;
}

// Whether the list build expects cells with 129 to 192 candidates, which its
// WIDE variant takes on the fast path too: those of boxes whose sides are not
// close to a multiple of the cutoff, or of long lists.  Silicon has 0.46 atoms
// per sigma^3 (27 cells of rc^3 hold 96 candidates for lists of 1.1 cutoffs,
// 110 for 1.15), and the counts vary by about a tenth.  5 and 5.04 atoms per
// cell (1,000 and 1,728 atoms): 29 -> 14 us; 4.1 and 4.4 (4,096 and 5,832):
// 13.3 -> 13.7 and 13.9 -> 14.4; 2.1 M atoms, 3.6 per cell: 730 -> 780, so
// the variant is left out where it is not wanted.
static bool wide_cells(const DevBufs &d, const FConst &fc) {
  const double is = std::min(fc.isig[0][0], fc.isig[1][1]);
  return 27.0 * 0.46 * d.max_cell * is * is * is > 120.0;
}

// Times the launches issued in its scope under one key.
struct KScope {
  const KTimer *t;
  int id, key;
  KScope(const DevBufs &d, int k) : t(d.kt), id(-1), key(k) {
    if (t && t->begin) id = t->begin(t->ctx, k);
  }
  ~KScope() {
    if (id >= 0) t->end(t->ctx, id, key);
  }
};

// chunks of the largest instance
static int fin_nch(const DevBufs &d, int bs) { return (d.max_pad / bs + FIN_CH - 1) / FIN_CH; }

static RedSpec red_spec(int nv, int bs, const int *op, const int *dst, int sub = 1) {
  RedSpec rs;
  rs.nv = nv;
  rs.bs = bs;
  rs.sub = sub;
  for (int k = 0; k < FIB_NRED; ++k) {
    rs.op[k] = k < nv ? op[k] : 0;
    rs.dst[k] = k < nv ? dst[k] : -1;
  }
  return rs;
}

// Chunks per workgroup of k_finalize: all of an instance, or one.
static int fin_per(const DevBufs &d, int bs) { return fin_nch(d, bs) <= FIN_ONE ? FIN_ONE : 1; }

// Reduces every instance, or the chunks of instances of more than FIN_ONE
// (fin_per is 1: tmp is left to combine).
template <int NV>
static void fin_launch(const DevBufs &d, const RedSpec &rs, hipStream_t s) {
  const int nch = fin_nch(d, rs.bs), per = fin_per(d, rs.bs);
  const int waves = std::min(FIN_WAVES, std::min(nch, per) * (NV == 10 ? NV : 1));
  hipLaunchKernelGGL(k_finalize<NV>, dim3(d.ninst, per == 1 ? nch : 1), dim3(waves * FIB_WAVE), 0,
                     s, d.I, d.partials, d.pstride, rs, per, d.ctl, d.fin_tmp, d.halt);
}

static void finalize(const DevBufs &d, int nv, int bs, const int *op, const int *dst,
                     hipStream_t s, int sub = 1) {
  const RedSpec rs = red_spec(nv, bs, op, dst, sub);
  KScope ks_(d, KT_REDUCE);
#define FIN_CASE(N)                                                                          \
  case N:                                                                                    \
    fin_launch<N>(d, rs, s);                                                                 \
    if (fin_per(d, bs) == 1)                                                                 \
      hipLaunchKernelGGL(k_finalize2<N>, dim3(d.ninst), dim3(FIB_WAVE), 0, s, d.I,           \
                         fin_nch(d, bs), rs, d.ctl, d.fin_tmp, d.halt);                      \
    break;
  switch (nv) {
    FIN_CASE(4)
    FIN_CASE(5)
    FIN_CASE(10)
  }
#undef FIN_CASE
}

static void finalize_thermo(const DevBufs &d, hipStream_t s) {
  const int op[5] = {0, 0, 0, 0, 1};
  const int dst[5] = {DCTL_IDX(glob_sum), DCTL_IDX(side_sum), DCTL_IDX(side_cnt),
                      DCTL_IDX(ke_sum), DCTL_IDX(vmax)};
  finalize(d, 5, FIB_BLOCK, op, dst, s);
}

// Sort of every instance small enough for one workgroup (k_sort_small).
static bool small_sort(const DevBufs &d) {
  return d.max_pad <= SORT_N && d.max_bucket <= SORT_N;
}

// Whether the totals of the scan's nb blocks are scanned by launches of their
// own: the blocks' sums over the totals before them grow with nb squared.
// k_scan_down of 2,747 blocks (5.6 million buckets) 27 us without them, about
// what it takes to read and write the buckets; of 43,500 574 us, 324 (and two
// launches of 5) with them; of 348,500 14.8 ms, 2.5.
static bool scan_top(int nb) { return nb > 8192; }
size_t bsum_len(int nbucket) {
  const size_t nb = (size_t)nblk((long)nbucket + 1, SCAN_CH);
  return nb + (scan_top((int)nb) ? nb + 1 + (size_t)nblk((long)nb + 1, SCAN_CH) : 0);
}

void launch_build(const DevBufs &d, const FConst &fc, hipStream_t s, bool inplace) {
  const int c = d.cur, n = 1 - d.cur;
  if (small_sort(d)) {
    KScope ks_(d, KT_SORT);
    hipLaunchKernelGGL(k_sort_small, dim3(d.ninst), dim3(SORT_T), 0, s, d.X[c], d.I, d.bkey,
                       d.cstart, d.perm, d.ctl, d.gate);
  } else {
    {
      KScope ks_(d, KT_BIN);
      hipLaunchKernelGGL(k_bin, dim3(gcap(d.NA)), dim3(FIB_BLOCK), 0, s, d.X[c], d.NA, d.I,
                         d.bkey, d.brank, d.bcnt, d.ctl, d.binst, d.gate);
    }
    KScope ks_(d, KT_SORT);
    // (the scan writes one entry past the buckets)
    const int nb = nblk(d.nbucket + 1, SCAN_CH);
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_T), 0, s, d.bcnt, d.nbucket, d.bsum,
                       d.gate);
    if (scan_top(nb)) {
      int *const top = d.bsum + nb, *const sum = top + nb + 1;
      const int nt = nblk(nb + 1, SCAN_CH);
      hipLaunchKernelGGL(k_scan_reduce, dim3(nt), dim3(SCAN_T), 0, s, d.bsum, nb, sum, d.gate);
      hipLaunchKernelGGL(k_scan_down<false>, dim3(nt), dim3(SCAN_T), 0, s, d.bsum, nb, sum, top,
                         d.gate);
      hipLaunchKernelGGL(k_scan_down<true>, dim3(nb), dim3(SCAN_T), 0, s, d.bcnt, d.nbucket, top,
                         d.cstart, d.gate);
    } else {
      hipLaunchKernelGGL(k_scan_down<false>, dim3(nb), dim3(SCAN_T), 0, s, d.bcnt, d.nbucket,
                         d.bsum, d.cstart, d.gate);
    }
    hipLaunchKernelGGL(k_scatter, dim3(gcap(std::max(d.NA, d.nbucket))), dim3(FIB_BLOCK), 0, s, d.bkey, d.brank, d.NA,
                       d.I, d.cstart, d.perm, d.bcnt, d.nbucket, d.binst, d.gate);
    hipLaunchKernelGGL(k_fixup, dim3(gcap(d.nbucket)), dim3(FIB_BLOCK), 0, s, d.cstart, d.nbucket,
                       d.I, d.ninst, d.perm, d.gate);
  }
  // the in-place sort of MD-step mode leaves the forces behind: every caller
  // (an MD step's build, the fire-time build) computes them anew before
  // anything reads them
  double *const F0 = inplace ? nullptr : d.F[c];
  {
    KScope ks_(d, KT_SORT);
    hipLaunchKernelGGL(k_reorder, dim3(gcap(d.NA)), dim3(FIB_BLOCK), 0, s, d.NA, d.perm, d.bkey,
                       d.I, d.X[c], d.X[n], d.V[c], d.V[n], F0, d.F[n], d.Xi[c], d.Xi[n], d.inv,
                       d.Xb, d.disp, d.nst, d.cnt_sw, d.cnt_ion, d.off_sw, d.ctl, d.binst, d.gate);
  }
  launch_nbuild(d, fc, s, n, inplace);
}

void launch_nbuild(const DevBufs &d, const FConst &fc, hipStream_t s, int from, bool back) {
  CopyBack cb{};
  if (back) {
    const int c = d.cur, n = 1 - d.cur;
    cb = CopyBack{gcap(d.NA), d.X[n], d.X[c], d.V[n], d.Xi[n], d.V[c], d.Xi[c], d.binst, d.NA};
  }
  KScope ks_(d, KT_NBUILD);
  const int nbc = d.nb_cells ? d.nb_cells : nb_cells_auto(d.total_cells);
  const bool wide = wide_cells(d, fc);
  const bool sparse = nbc == 8 && d.NA < d.total_cells;
#define NB_LAUNCH(C)                                                                           \
  auto *f = wide ? k_nbuild<C, true, false> : k_nbuild<C, false, false>;                       \
  if (sparse) f = wide ? k_nbuild<8, true, true> : k_nbuild<8, false, true>;                   \
  hipLaunchKernelGGL(f, dim3(cb.blocks + nblk(d.total_cells, C * NB_WAVES)),                   \
                     dim3(NB_WAVES * FIB_WAVE), 0, s, d.X[from], d.I, d.ninst, d.total_cells,  \
                     d.cstart, fc.rv2, fc.rv2lj, d.Wsw, d.Wion, d.cnt_sw, d.nbr_sw, d.cnt_ion, \
                     d.nbr_ion, d.rk_sw, d.off_sw, d.ctl, d.gate, d.halt, cb)
  switch (nbc) {
    case 1: { NB_LAUNCH(1); break; }
    case 2: { NB_LAUNCH(2); break; }
    case 4: { NB_LAUNCH(4); break; }
    case 16: { NB_LAUNCH(16); break; }
    default: { NB_LAUNCH(8); break; }
  }
#undef NB_LAUNCH
}

void launch_cellid(const DevBufs &d, int inst, int32_t *dout, hipStream_t s) {
  {
    KScope ks_(d, KT_IO);
    hipLaunchKernelGGL(k_cellid, dim3(nblk(d.NA, FIB_BLOCK)), dim3(FIB_BLOCK), 0, s, d.X[d.cur],
                       d.NA, d.I, inst, dout);
  }
}

template <bool MIXED, bool EN, bool VIR>
static void force_ab(const DevBufs &d, const FConst &fc, hipStream_t s, bool extra) {
  {
    KScope ks_(d, KT_LEGS);
    hipLaunchKernelGGL((k_legs<MIXED, EN, VIR>), dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK), 0, s,
                       d.X[d.cur], d.I, fc, d.tab, d.NA, d.Wsw, d.Wion, d.cnt_sw, d.nbr_sw,
                       d.cnt_ion, d.nbr_ion, d.amask, d.Fpart, d.upart, d.near,
                       d.nst, d.ctl, d.binst, d.pstride, d.partials, d.halt, xcd_shift(d));
  }
  const bool small = !VIR && d.NA <= TRI_SMALL &&
                     (EN || ((!d.tri_ns || d.tri_ns == TriStage<MIXED>::N) &&
                             (!d.tri_tb || d.tri_tb == TRI_BATCH)));
  {
    KScope ks_(d, KT_TRI);
    // the MD step's variant (no energy, no virial) in every tile; the others
    // in the default tile
    const int ns = (EN || VIR || !d.tri_ns) ? TriStage<MIXED>::N : d.tri_ns;
    const int tb = (EN || VIR || !d.tri_tb) ? TRI_BATCH : d.tri_tb;
    // extra_pass runs whenever its partials are reduced (energy, virial) or
    // stale-list terms can exist; the MD step's gate rules the latter out
    const bool xt = EN || VIR || extra;
    ExtraArgs xa{xt ? d.NA / FIB_BLOCK : 0, d.cnt_sw, d.disp, d.ctl, d.EX, d.EXself,
                       d.exmask, d.nst};
#define TRI_LAUNCH(NS_, TB_, APW_)                                                            \
  do {                                                                                        \
    auto *f = k_tri<MIXED, EN, VIR, NS_, TB_, APW_, true>;                                    \
    if constexpr (!EN && !VIR)                                                                \
      if (!xt) f = k_tri<MIXED, EN, VIR, NS_, TB_, APW_, false>;                              \
    hipLaunchKernelGGL(                                                                       \
        f, dim3(d.NA / (FIB_BLOCK / FIB_WAVE * APW_) + xa.blocks), dim3(FIB_BLOCK), 0, s,     \
        d.X[d.cur], d.I, fc, d.NA, d.Wsw, d.nbr_sw, d.rk_sw, d.off_sw, d.amask,               \
        (typename GRec<MIXED, EN>::type *)d.G, d.RA, d.F[1 - d.cur], d.V[1 - d.cur],          \
        d.pstride, d.partials + (size_t)FIB_NRED * d.pstride, d.binst, d.halt,                \
        xcd_shift(d) + (APW_ == 8 ? 3 : APW_ == 16 ? 2 : 0), xa);                             \
  } while (0)
    // (the virial is summed over runs of a wavefront's legs, so its bits depend
    // on the split: in the mixed mode, FP32 sums, the runs stay those of 64
    // atoms; in FP64 each instance has the split of its own size, whatever the
    // batch's is, in one launch for each of the two that the batch holds)
    if constexpr (VIR && !MIXED) {
      const bool both = d.min_pad <= TRI_SMALL && d.max_pad > TRI_SMALL;
      if (d.max_pad > TRI_SMALL) TRI_LAUNCH(TriStage<MIXED>::N, TRI_BATCH, FIB_WAVE);
      if (both) xa.blocks = 0;
      if (d.min_pad <= TRI_SMALL) TRI_LAUNCH(128, TRI_BATCH, 16);
    } else if (small) {
      // (energies: 16 atoms per wavefront at least, see tri_partials)
      if constexpr (!EN && !VIR) {
        if (d.NA <= TRI_TINY) TRI_LAUNCH(128, TRI_BATCH, 8);
        else TRI_LAUNCH(128, TRI_BATCH, 16);
      } else {
        TRI_LAUNCH(128, TRI_BATCH, 16);
      }
    } else if constexpr (EN || VIR) {
      TRI_LAUNCH(TriStage<MIXED>::N, TRI_BATCH, FIB_WAVE);
    } else {
      if (ns == TriStage<MIXED>::N && tb == TRI_BATCH)
        TRI_LAUNCH(TriStage<MIXED>::N, TRI_BATCH, FIB_WAVE);
      else if (ns == 128 && tb == 2) TRI_LAUNCH(128, 2, FIB_WAVE);
      else if (ns == 128 && tb == 4) TRI_LAUNCH(128, 4, FIB_WAVE);
      else if (ns == 256 && tb == 2) TRI_LAUNCH(256, 2, FIB_WAVE);
      else TRI_LAUNCH(256, 4, FIB_WAVE);
    }
#undef TRI_LAUNCH
  }
  if (EN || VIR) {
    int op[10], dst[10];
    for (int k = 0; k < 10; ++k) { op[k] = 0; dst[k] = DCTL_IDX(utot) + k; }
    finalize(d, 10, FIB_BLOCK, op, dst, s, VIR && !MIXED ? 0 : small ? 4 : 1);
  }
}

template <bool MIXED, bool EN, int MODE>
static void force_c(const DevBufs &d, const FConst &fc, const StepArgs &sa, double *Fo,
                    hipStream_t s) {
  typedef typename Prec<MIXED>::T4 T4;
  const double fscale = MIXED ? fc.eps[0][0] * fc.isig[0][0] : 1.0;
  const double escale = MIXED ? fc.eps[0][0] : 1.0;
  {
    KScope ks_(d, KT_GATHER);
    hipLaunchKernelGGL((k_force3<MIXED, EN, MODE>), dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK),
                       0, s, d.X[d.cur], d.I, d.NA, d.Wsw, d.nbr_sw, d.rk_sw, d.off_sw,
                       (const typename GRec<MIXED, EN>::type *)d.G, d.RA, d.F[1 - d.cur],
                       d.V[1 - d.cur], d.amask, d.cnt_sw, d.Fpart,
                       d.upart, fscale, escale, Fo,
                       d.uout, d.V[d.cur], sa, d.pstride, d.partials, d.ctl, (const T4 *)d.EX,
                       (const T4 *)d.EXself, d.exmask, d.binst, d.halt, xcd_shift(d));
  }
  if (MODE == 1) finalize_thermo(d, s);
  // (MODE 2: launch_md_ctl reduces)
}

void launch_force_a(const DevBufs &d, const FConst &fc, bool mixed, bool energy, bool virial,
                    hipStream_t s, bool extra) {
  if (mixed) {
    if (energy) { if (virial) force_ab<true, true, true>(d, fc, s, extra); else force_ab<true, true, false>(d, fc, s, extra); }
    else { if (virial) force_ab<true, false, true>(d, fc, s, extra); else force_ab<true, false, false>(d, fc, s, extra); }
  } else {
    if (energy) { if (virial) force_ab<false, true, true>(d, fc, s, extra); else force_ab<false, true, false>(d, fc, s, extra); }
    else { if (virial) force_ab<false, false, true>(d, fc, s, extra); else force_ab<false, false, false>(d, fc, s, extra); }
  }
}

template <bool MIXED>
static void force_c_mode(const DevBufs &d, const FConst &fc, bool energy, int mode,
                         const StepArgs &sa, double *Fout, hipStream_t s) {
  if (mode == 1) force_c<MIXED, false, 1>(d, fc, sa, Fout, s);
  else if (mode == 2) force_c<MIXED, false, 2>(d, fc, sa, Fout, s);
  else if (energy) force_c<MIXED, true, 0>(d, fc, sa, Fout, s);
  else force_c<MIXED, false, 0>(d, fc, sa, Fout, s);
}

void launch_force_b(const DevBufs &d, const FConst &fc, bool mixed, bool energy, int mode,
                    const StepArgs &sa, double *Fout, hipStream_t s) {
  if (mixed) force_c_mode<true>(d, fc, energy, mode, sa, Fout, s);
  else force_c_mode<false>(d, fc, energy, mode, sa, Fout, s);
}

void launch_pos(const DevBufs &d, const StepArgs &sa, hipStream_t s) {
  {
    KScope ks_(d, KT_POS);
    hipLaunchKernelGGL(k_pos, dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK), 0, s, d.X[d.cur], d.I, d.NA,
                       d.V[d.cur], d.F[d.cur], d.Xi[d.cur], sa, d.pstride, d.partials, d.ctl,
                       d.Xb, d.disp, d.Wsw, d.cnt_sw, d.nbr_sw, d.nst);
  }
  const int op[4] = {0, 1, 1, 1};
  const int dst[4] = {DCTL_IDX(eq_sum), DCTL_IDX(kemax), DCTL_IDX(maxdisp), DCTL_IDX(maxdisp2)};
  finalize(d, 4, FIB_BLOCK, op, dst, s);
}

void launch_md_pos(const DevBufs &d, const FConst &fc, const StepArgs &sa, int *gate,
                   hipStream_t s) {
  int *leave = gate + 2 + 2 * d.ninst;
  {
    KScope ks_(d, KT_POS);
    hipLaunchKernelGGL(k_md_pos, dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK), 0, s, d.X[d.cur], d.I,
                       d.NA, d.V[d.cur], d.F[d.cur], d.Xi[d.cur], sa, d.pstride, d.partials,
                       d.ctl, d.Xb, d.disp, d.Wsw, d.cnt_sw, d.nbr_sw, d.nst, leave,
                       d.binst, d.halt, xcd_shift(d));
  }
  const int op[6] = {RED_TOP2, RED_TOP2_CNT, RED_TOP2_SND, RED_SUM, RED_SUM, RED_SUM};
  const int dst[6] = {DCTL_IDX(maxdisp), DCTL_IDX(nmaxdisp), DCTL_IDX(maxdisp2),
                      DCTL_IDX(e_bath_step), DCTL_IDX(e_out_step), DCTL_IDX(movers)};
  const RedSpec rs = red_spec(6, FIB_BLOCK, op, dst);
  const int nch = fin_nch(d, FIB_BLOCK);
  // a few small instances: k_md_decide's four wavefronts reduce them, two
  // each; otherwise a wavefront per chunk does, and k_md_decide combines
  const int how = nch == 1 && d.ninst <= 8 ? FIN_ALL
                  : fin_per(d, FIB_BLOCK) > 1 ? FIN_DONE
                                              : FIN_COMBINE;
  KScope ks_(d, KT_REDUCE);
  if (how != FIN_ALL) fin_launch<6>(d, rs, s);
  hipLaunchKernelGGL(k_md_decide, dim3(1), dim3(DECIDE_T), 0, s, d.ninst, d.I, d.ctl, sa.skin,
                     gate, leave, d.X[d.cur], fc, d.Wsw, d.Wion, d.cnt_sw, d.nbr_sw, d.cnt_ion,
                     d.nbr_ion, how, rs, d.partials, d.pstride, d.fin_tmp, nch, d.halt);
}

void launch_fire_energy(const DevBufs &d, const FConst &fc, int q, hipStream_t s) {
  hipLaunchKernelGGL(k_fire_energy, dim3(1), dim3(FIB_WAVE), 0, s, q, d.inv, d.X[d.cur], d.I, fc,
                     d.Wsw, d.Wion, d.cnt_sw, d.nbr_sw, d.cnt_ion, d.nbr_ion, d.ctl);
}

void launch_md_ctl(const DevBufs &d, const StepArgs &sa, hipStream_t s) {
  const int op[4] = {RED_MAX, RED_SUM, RED_SUM, RED_SUM};
  const int dst[4] = {DCTL_IDX(vmax), DCTL_IDX(ke_sum), DCTL_IDX(ke_shell), DCTL_IDX(n_shell)};
  const RedSpec rs = red_spec(4, FIB_BLOCK, op, dst);
  const int nch = fin_nch(d, FIB_BLOCK);
  KScope ks_(d, KT_REDUCE);
  if (nch > 1) fin_launch<4>(d, rs, s);
  hipLaunchKernelGGL(k_md_ctl, dim3(d.ninst), dim3(FIB_WAVE), 0, s, d.I, d.ctl, sa,
                     nch == 1 ? FIN_ALL : fin_per(d, FIB_BLOCK) > 1 ? FIN_DONE : FIN_COMBINE, rs, d.partials, d.pstride, d.fin_tmp, nch,
                     d.halt);
}

void launch_md_init(const DevBufs &d, const StepArgs &sa, bool reset, hipStream_t s) {
  hipLaunchKernelGGL(k_md_init, dim3(nblk(d.ninst, FIB_BLOCK)), dim3(FIB_BLOCK), 0, s, d.ninst,
                     d.ctl, sa, reset ? 1 : 0);
}

void launch_md_report(const DevBufs &d, const StepArgs &sa, hipStream_t s) {
  {
    KScope ks_(d, KT_REDUCE);
    hipLaunchKernelGGL(k_md_report, dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK), 0, s, d.X[d.cur],
                       d.I, d.NA, d.Xi[d.cur], sa, d.pstride, d.partials);
  }
  const int op[4] = {0, 0, 0, 1};
  const int dst[4] = {DCTL_IDX(n_removed), DCTL_IDX(n_ga_removed), DCTL_IDX(n_displaced),
                      DCTL_IDX(ion_z)};
  finalize(d, 4, FIB_BLOCK, op, dst, s);
}

// Rows of an ELL list copied into a wider layout (the list grew).
template <typename T>
__global__ void k_copy_rows(int NA, int wold, const T *__restrict__ src, int wnew,
                            T *__restrict__ dst) {
  GRID_STRIDE(p, NA) {
    for (int k = 0; k < wold; ++k) dst[(size_t)p * wnew + k] = src[(size_t)p * wold + k];
  }
}

void launch_copy_rows(int NA, int wold, const int *src, int wnew, int *dst, hipStream_t s) {
  hipLaunchKernelGGL(k_copy_rows<int>, dim3(gcap(NA)), dim3(FIB_BLOCK), 0, s, NA, wold, src,
                     wnew, dst);
}
void launch_copy_rows(int NA, int wold, const uint16_t *src, int wnew, uint16_t *dst,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_copy_rows<uint16_t>, dim3(gcap(NA)), dim3(FIB_BLOCK), 0, s, NA, wold, src,
                     wnew, dst);
}

// After a removal-list overflow: no atom stays marked as leaving.
__global__ void k_clear_leaving(int NA, double4 *__restrict__ X) {
  GRID_STRIDE(p, NA) {
    const double4 x = X[p];
    if (meta_of(x) & META_LEAVING) {
      double4 y = x;
      y.w = __longlong_as_double((long long)(wbits(x) & ~(uint64_t)META_LEAVING));
      X[p] = y;
    }
  }
}

// Clears the list-overflow flags and the halt flag (after the lists grew),
// or the removal-list overflow flags.
__global__ void k_clear_overflow(int ninst, DCtl *__restrict__ ctl, int *__restrict__ halt,
                                 int lists) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < ninst) {
    if (lists) {
      ctl[k].overflow = 0;
      ctl[k].maxcnt_sw = ctl[k].maxcnt_ion = 0.0;
    } else {
      ctl[k].leave_overflow = 0;
    }
  }
  if (k == 0 && lists && halt) *halt = 0;
}

void launch_clear_overflow(const DevBufs &d, hipStream_t s, bool lists) {
  hipLaunchKernelGGL(k_clear_overflow, dim3(nblk(d.ninst, FIB_BLOCK)), dim3(FIB_BLOCK), 0, s,
                     d.ninst, d.ctl, d.halt, lists ? 1 : 0);
}

// Start state of a handle-free evaluation, written by kernels: the instance
// record (by value) and zeroed bookkeeping.
__global__ void k_put_inst(DInst in, DInst *__restrict__ I) {
  if (blockIdx.x == 0 && threadIdx.x == 0) I[0] = in;
}
__global__ void k_fill_zero(uint32_t *__restrict__ p, size_t nwords) {
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < nwords;
       k += (size_t)gridDim.x * blockDim.x)
    p[k] = 0u;
}

void launch_put_inst(const DevBufs &d, const DInst &in, hipStream_t s) {
  hipLaunchKernelGGL(k_put_inst, dim3(1), dim3(FIB_WAVE), 0, s, in, d.I);
}
void launch_fill_zero(void *p, size_t bytes, hipStream_t s) {
  const size_t nw = bytes / 4;  // every array of the arena is a multiple of 4 bytes
  hipLaunchKernelGGL(k_fill_zero, dim3(gcap((long)std::min<size_t>(nw, 1u << 30))),
                     dim3(FIB_BLOCK), 0, s, static_cast<uint32_t *>(p), nw);
}

void launch_clear_leaving(const DevBufs &d, hipStream_t s) {
  hipLaunchKernelGGL(k_clear_leaving, dim3(gcap(d.NA)), dim3(FIB_BLOCK), 0, s, d.NA, d.X[d.cur]);
}

void launch_sums(const DevBufs &d, const StepArgs &sa, hipStream_t s) {
  {
    KScope ks_(d, KT_REDUCE);
    hipLaunchKernelGGL(k_sums, dim3(d.NA / FIB_BLOCK), dim3(FIB_BLOCK), 0, s, d.X[d.cur], d.I, d.NA,
                       d.V[d.cur], sa, d.pstride, d.partials, d.ctl);
  }
  finalize_thermo(d, s);
}

void launch_import(const DevBufs &d, int inst, const DInst &in, const double *X,
                   const double *V, const int32_t *atype, const int32_t *xsides,
                   const double *Xi, hipStream_t s) {
  {
    KScope ks_(d, KT_IO);
    hipLaunchKernelGGL(k_import, dim3(nblk(in.natm_pad, FIB_BLOCK)), dim3(FIB_BLOCK), 0, s, inst, in,
                       d.NA, X, V, atype, xsides, Xi, d.X[0], d.X[1], d.V[0], d.V[1], d.F[0],
                       d.F[1], d.Xi[0], d.Xi[1], d.inv);
  }
}

void launch_export(const DevBufs &d, const DInst &in, const ExportArgs &ex, hipStream_t s) {
  {
    KScope ks_(d, KT_IO);
    hipLaunchKernelGGL(k_export, dim3(nblk(in.natm_pad, FIB_BLOCK)), dim3(FIB_BLOCK), 0, s, in,
                       d.NA, d.X[d.cur], ex);
  }
}

void launch_set_atom(const DevBufs &d, int p, const double x[3], const double v[3],
                     const StepArgs &sa, hipStream_t s) {
  {
    KScope ks_(d, KT_IO);
    hipLaunchKernelGGL(k_set_atom, dim3(1), dim3(FIB_WAVE), 0, s, d.NA, d.X[d.cur], d.V[d.cur], p,
                       x[0], x[1], x[2], v[0], v[1], v[2], sa, d.ctl);
  }
}

}  // namespace fibk
