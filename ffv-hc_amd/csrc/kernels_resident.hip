// Solvers whose blocks stay on the chip: one launch runs a whole solve of up to one 16^3 block per
// compute unit (BiCGSTAB: FFVILS.h:793-974, CG: 661-791, RBGS / Jacobi: 492-594), each workgroup
// keeping its block's vectors in registers and LDS from the first iteration to the last.  Jacobi
// BiCGSTAB, CG, Jacobi and FP32 RBGS also run with two blocks per compute unit (PAIR), at half the
// registers and LDS a block: vectors read once an iteration then stay in memory, which L2 serves.
//
// What bounds a small grid is not bytes but chains: with one launch per stage (kernels_bicg.hip,
// kernels_cg.hip, kernels_core.hip) an iteration is five to seven launches of 7-15 us each at 16-128
// workgroups, every one of them launch -> slot -> block -> case state -> loads -> reduction -> store.
// Here a stage ends in a meeting of the case's workgroups instead of a launch, and a stage's inputs
// are already in registers; only ghost layers and block sums cross memory.
//
// A meeting.  Each workgroup writes up to three block sums into words of its own, and reads every
// workgroup's words until all are there; a word holds a signalling NaN (which no arithmetic
// produces) while it is unset, so the value is its own flag and nothing is counted atomically (a
// single counter costs about 130 ns an arrival).  Where only ghosts change hands, a workgroup waits
// for its neighbours' turn numbers alone.  Ghost values, words and turn numbers are written and read
// as relaxed atomics of device scope, which go past the caches that are not shared between XCDs; a
// workgroup publishes after its wavefronts have waited for their ghost stores, so who has seen its
// turn sees its ghosts.  Three sets of words take turns: who passes meeting m knows that everyone
// has finished reading the words of m - 1 and unsets its own there, and they are written again for
// m + 2, after the waits of m + 1.
//
// The launch is cooperative, so the workgroups of a solve are on the chip together.  A wait ends
// after kWaitTicks all the same (a device shared with something that holds it that long): the
// workgroups leave, the case is marked (parity -1) and the caller solves with one launch per stage.
//
// The arithmetic, each sum's order included, is that of the launch-per-stage kernels: the same bits.
//
// Measured, one iteration with one launch per stage -> resident: two-level BiCGSTAB 55 -> 30 us at 128
// blocks (two preconditioners 2 x 8, meetings 13), Jacobi BiCGSTAB 46 -> 20 us at 128 and 68 ->
// 28 us at 256 blocks, PCG 26 -> 10 us at 60, RBGS 14 -> 8.6 us and Jacobi 13.4 -> 7.9 us at 128.  A
// meeting of everyone takes 2.4 us with 16 workgroups and 3.4-4 with 128, one of neighbours 1.4-2.
// PAIR, a solve: Jacobi BiCGSTAB 48.5 -> 25.7 ms at 288 and 59.7 -> 32.7 ms at 512 blocks, PCG 35.4 -> 20.9
// and 53.2 -> 28.1 ms, 100 Jacobi sweeps 1.81 -> 1.43 and 2.16 -> 1.83 ms.  With x, r0 and the diagonal in
// registers as in the other form the compiler spilled 56-193 of 128 registers (CG 1.1x); what every lane
// has in scalar registers (scalar()) took 26-46 spills out of each kernel.
#include "kcommon.h"
#include "kernels.h"

namespace ffvhc {

constexpr int RS_NT = 512;                // two threads per (i, j) column, 8 cells each
constexpr int RS_NK = NB * NF / RS_NT;    // cells per thread
constexpr unsigned long long kUnset = 0x7FF0DEADBEEF0001ull;
constexpr unsigned long long kWaitTicks = 400000000ull;  // 4 s of the 100 MHz clock
static_assert(RS_NK == 8 && RS_MAX % 256 == 0, "layout of the reductions below");
// words of one kind a lane reads in a meeting, with one or two workgroups a compute unit (PAIR)
template <bool PAIR>
constexpr int kWords = (PAIR ? RS_MAX2 : RS_MAX) / 64;

template <class T>
__device__ inline T load_device(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline void store_device(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
struct PutDevice {
  template <class T>
  __device__ void operator()(T* p, T v) const {
    store_device(p, v);
  }
};

// a value that every lane has, in scalar registers (a struct of 8-byte and 4-byte members too)
template <class V>
__device__ inline V scalar(V v) {
  static_assert(sizeof(V) % 4 == 0);
  uint32_t w[sizeof(V) / 4];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (size_t q = 0; q < sizeof(V) / 4; q++) w[q] = __builtin_amdgcn_readfirstlane(w[q]);
  __builtin_memcpy(&v, w, sizeof(V));
  return v;
}

// Scratch of the meetings in LDS: partial sums by wavefront, results, the mark of a wait that ended
struct MeetLds {
  double red[3][RS_NT / 64];
  double sum[3];
  int failed;
};

struct Meeting {
  unsigned long long* words;  // [3 sets][3 words][RS_COPIES][nslots], then a turn number per slot
  size_t nslots;
  int begin, n, slot;  // the case's slots and this workgroup's
  unsigned epoch = 0, turn = 0;

  __device__ unsigned long long* word(unsigned e, int k, int copy) const {
    return words + (((size_t)(e % 3) * 3 + k) * RS_COPIES + copy) * nslots;
  }

  // All workgroups of the case.  NP words, word k the NW wavefront sums red[k][..] (word 2: NW2 of them)
  // added in wavefront order; word k goes to use(k, e), called by wavefront k with the words e[m] of
  // blocks lane + 64 m (0 past n).  Each workgroup writes its words RS_COPIES times and reads one copy,
  // so that few poll the same cache line (128 workgroups, one copy: 4.2 us a meeting).  False: a wait
  // ended without everyone (uniform over the workgroup).
  template <int NP, int EN, int NW = 4, int NW2 = NW, class Use>
  __device__ bool all(MeetLds& M, const Use& use) {
    const int t = thread_here(), lane = t & 63;
    // this wavefront's stores have arrived: ghosts, and the words it unset in the last meeting
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t < NP * RS_COPIES) {
      const int k = t / RS_COPIES;
      double v = 0.0;
      for (int q = 0; q < (k == 2 ? NW2 : NW); q++) v += M.red[k][q];
      store_device(word(epoch, k, t % RS_COPIES) + slot, (unsigned long long)__double_as_longlong(v));
    }
    const int k = t >> 6;
    if (k < NP) {
      const unsigned long long* const w = word(epoch, k, blockIdx.x % RS_COPIES) + begin;
      unsigned long long b[EN];
#pragma unroll
      for (int m = 0; m < EN; m++) b[m] = lane + 64 * m < n ? kUnset : 0ull;
      const unsigned long long t0 = wall_clock64();
      bool there = false;
      while (!there) {
        bool here = true;
#pragma unroll
        for (int m = 0; m < EN; m++)
          if (b[m] == kUnset) b[m] = load_device(w + lane + 64 * m);
#pragma unroll
        for (int m = 0; m < EN; m++) here = here && b[m] != kUnset;
        there = __all(here);
        if (!there && wall_clock64() - t0 > kWaitTicks) break;
      }
      if (there) {
        double e[EN];
#pragma unroll
        for (int m = 0; m < EN; m++) e[m] = __longlong_as_double((long long)b[m]);
        use(k, e);
        if (t < 3 * RS_COPIES && epoch > 0)
          store_device(word(epoch - 1, t / RS_COPIES, t % RS_COPIES) + slot, kUnset);
      } else {
        M.failed = 1;
      }
    }
    epoch++;
    __syncthreads();
    return M.failed == 0;
  }

  // The workgroups this one exchanges ghosts with (`count` <= 64 slots in `list`): on return their
  // ghost stores of this turn are visible.  Between two turns that use the same halo lies an all().
  __device__ bool neighbours(MeetLds& M, const int* list, int count) {
    const int t = thread_here();
    unsigned long long* const turns = words + (size_t)9 * RS_COPIES * nslots;
    turn++;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's ghost stores have arrived
    __syncthreads();
    if (t < 64) {
      if (t == 0) store_device(turns + slot, (unsigned long long)turn);
      const unsigned long long t0 = wall_clock64();
      bool there = t >= count;
      while (!__all(there)) {
        if (!there) there = load_device(turns + list[t]) >= turn;
        if (wall_clock64() - t0 > kWaitTicks) {
          M.failed = 1;
          break;
        }
      }
    }
    __syncthreads();
    return M.failed == 0;
  }
};

// the sum over the case in the order of the per-case finalisation (case_sum)
template <int EN>
__device__ inline double case_order(const double (&e)[EN]) {
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    double v = 0.0;
#pragma unroll
    for (int m = w; m < EN; m += 4) v += e[m];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    s += v;
  }
  return s;
}
// ... and in that of the coarse application's alpha (one wavefront, lane-strided)
template <int EN>
__device__ inline double lane_order(const double (&e)[EN]) {
  double v = 0.0;
#pragma unroll
  for (int m = 0; m < EN; m++) v += e[m];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ __launch_bounds__(256) void unset_words_kernel(const int* __restrict__ active, int nact,
                                                          unsigned long long* __restrict__ words, size_t nslots) {
  const int i = blockIdx.x * 256 + threadIdx.x, row = i / nact;
  if (row < RS_WORDS) words[(size_t)row * nslots + active[i % nact]] = row < RS_WORDS - 1 ? kUnset : 0ull;
}

// A wavefront sum into red[k][w] (lane 0)
template <int M>
__device__ inline void wave_sums(double (&v)[M], MeetLds& L, int w) {
#pragma unroll
  for (int k = 0; k < M; k++) {
    for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
    if ((threadIdx.x & 63) == 0) L.red[k][w] = v[k];
  }
}

// M sums over the block in the order of a 256-thread kernel (a thread per column, its 16 planes in
// order, then the wavefronts): the lower half column's sums continue in the upper one.  add(v) adds
// the thread's 8 cells in order; leaves the four wavefront sums in L.red[k][0..3].
template <int M, class Add>
__device__ inline void column_sums(double (*chain)[NF], MeetLds& L, const Add& add) {
  const int t = thread_here(), col = t & (NF - 1);
  double v[M];
#pragma unroll
  for (int k = 0; k < M; k++) v[k] = 0.0;
  if (t < NF) {
    add(v);
#pragma unroll
    for (int k = 0; k < M; k++) chain[k][col] = v[k];
  }
  __syncthreads();
  if (t >= NF) {
#pragma unroll
    for (int k = 0; k < M; k++) v[k] = chain[k][col];
    add(v);
    wave_sums<M>(v, L, (t - NF) >> 6);
  }
}

// The block's operand in LDS: its cells with a plane below and above (zpad), and the ghosts of the
// four side faces in halo order
template <class T>
struct Operand {
  T zpad[NC + 2 * NF];
  T side[4 * NF];

  // the ghosts of slot `slot` from the halo array h
  __device__ void load_ghosts(const T* h, int slot) {
    const int t = thread_here();
    T g[NH / RS_NT];
#pragma unroll
    for (int q = 0; q < NH / RS_NT; q++) g[q] = load_device(h + (size_t)slot * NH + t + RS_NT * q);
#pragma unroll
    for (int q = 0; q < NH / RS_NT; q++) {
      const int w = t + RS_NT * q;
      if (w < 4 * NF)
        side[w] = g[q];
      else
        zpad[w < 5 * NF ? w - 4 * NF : NC + w - 4 * NF] = g[q];
    }
  }
  // the six neighbours of cell (tx, ty, k), whose index in zpad is li
  struct Nb {
    T w, e, s, n, b, t;
  };
  __device__ Nb around(int tx, int ty, int k, int li) const {
    Nb v;
    v.w = tx > 0 ? zpad[li - 1] : side[halo_index(0, ty, k)];
    v.e = tx < NB - 1 ? zpad[li + 1] : side[halo_index(1, ty, k)];
    v.s = ty > 0 ? zpad[li - NB] : side[halo_index(2, tx, k)];
    v.n = ty < NB - 1 ? zpad[li + NB] : side[halo_index(3, tx, k)];
    v.b = zpad[li - NF];
    v.t = zpad[li + NF];
    return v;
  }
};

// y = A v over the thread's 8 cells in calc_ax order (bils.f90:195-202).  The bands come from the
// half column's two class rows (its end cell, k = 0 below and NB - 1 above, and the others), read
// along with the ghosts rather than held between the stages; a cell marked in ex (a body cuts it, or
// no rows were made) reads its own.
template <class TM>
struct HalfRows {
  TM in[7], end[7];
  __device__ void load(const ClassRows<TM>& R, int slot, int tx, int ty, bool lower) {
    if (!R.uni) return;
    const TM* tr = class_column(R.tab, slot, tx, ty);
#pragma unroll
    for (int q = 0; q < 7; q++) {
      in[q] = tr[9 * 8 + q];
      end[q] = tr[(lower ? 0 : 18 * 8) + q];
    }
  }
};

template <class T, class TM>
__device__ inline T row_times(const Operand<T>& Z, const TM* w, int tx, int ty, int k) {
  const int li = tx + NB * ty + NF * (k + 1);
  const auto v = Z.around(tx, ty, k, li);
  return (T)w[1] * v.w + (T)w[2] * v.e + (T)w[3] * v.s + (T)w[4] * v.n + (T)w[5] * v.b + (T)w[6] * v.t +
         (T)w[0] * Z.zpad[li];
}

template <class T, class TM>
__device__ inline void half_matvec(const Operand<T>& Z, const HalfRows<TM>& W, const Coef7<TM>& A, unsigned ex,
                                   size_t g0, int tx, int ty, int kb, T (&y)[RS_NK]) {
#pragma unroll
  for (int kk = 0; kk < RS_NK; kk++) {
    TM w[7];
#pragma unroll
    for (int q = 0; q < 7; q++)
      w[q] = kk == 0 ? pick(kb != 0, W.in[q], W.end[q])
                     : kk == RS_NK - 1 ? pick(kb != 0, W.end[q], W.in[q]) : W.in[q];
    y[kk] = row_times<T, TM>(Z, w, tx, ty, kb + kk);
    if (kk & 1) __builtin_amdgcn_sched_barrier(0);  // two cells' operands at a time: registers
  }
  // the marked cells, one at a time (a loop: unrolled, their 56 addresses would fill the registers)
#pragma unroll 1
  for (unsigned m = ex; m; m &= m - 1) {
    const int kk = __builtin_ctz(m);
    TM w[7];
#pragma unroll
    for (int q = 0; q < 7; q++) w[q] = A.p[q][g0 + NF * kk];
    const T v = row_times<T, TM>(Z, w, tx, ty, kb + kk);
#pragma unroll
    for (int k = 0; k < RS_NK; k++) y[k] = k == kk ? v : y[k];
  }
}

// What push_halo reads of the block table, kept in LDS: one trip to memory for a whole solve
struct FaceLds {
  int type[6], bct[6], nbr[6][4], sub[6];
  double xc[6];
  __device__ void load(const DevBlock& B, const DevCase& C, int bcg) {
    const int t = threadIdx.x;
    if (t < 6) {
      type[t] = B.ftype[t];
      sub[t] = B.sub[t];
      bct[t] = C.bct[bcg][t];
      xc[t] = bct[t] == BCT_NEUMANN ? C.bcv[bcg][t] * B.dx : C.bcv[bcg][t];
    }
    if (t < 24) nbr[t >> 2][t & 3] = B.nbr[t >> 2][t & 3];
  }
};

// This block's slot and its neighbours', and for each face quarter where its neighbour is in the list
// (0 for an outer face); formed by one thread
struct NearLds {
  int slot[25], at[24], n;
  __device__ void load(const DevBlock& B, int own) {
    int k = 1;
    slot[0] = own;
    for (int f = 0; f < 6; f++)
      for (int s = 0; s < 4; s++) {
        const bool has = B.ftype[f] == FACE_FINER || (B.ftype[f] != FACE_OUTER && s == 0);
        at[4 * f + s] = has ? k : 0;
        if (has) slot[k++] = B.nbr[f][s];
      }
    n = k;
  }
};

// push_halo by 512 threads, the two faces of an axis at once (256 threads each), device-visible
template <class T, class Acc>
__device__ inline void push_faces(const FaceLds& F, int slot, const Acc& L, const T* hin, T* h) {
  const int t = thread_here(), p = t & (NF - 1);
#pragma unroll
  for (int ax = 0; ax < 3; ax++) {
    const int f = 2 * ax + (t >> 8);
    const int ft = __builtin_amdgcn_readfirstlane(F.type[f]);
    if (ft == FACE_SAME) {
      int i, j, k;
      face_cell(f, p & 15, p >> 4, 0, i, j, k);
      store_device(h + (size_t)F.nbr[f][0] * NH + (f ^ 1) * NF + p, (T)L(i, j, k));
    } else if (ft == FACE_OUTER) {
      const int type = F.bct[f];
      if (type < 0) continue;
      const bool pp = !(f & 1) && F.type[f ^ 1] == FACE_OUTER && F.bct[f ^ 1] == BCT_PERIODIC;
      int i, j, k;
      face_cell(f, p & 15, p >> 4, 0, i, j, k);
      const T xa = L(i, j, k);
      face_cell(f ^ 1, p & 15, p >> 4, 0, i, j, k);
      const T xf = L(i, j, k);
      const size_t at = (size_t)slot * NH + f * NF + p;
      // only a periodic minus face without its partner keeps its old value (outer_value)
      const T old = type == BCT_PERIODIC && !(f & 1) && !pp ? load_device(hin + at) : (T)0;
      store_device(h + at, outer_value<T>(f, type, (T)F.xc[f], xa, xf, old, pp));
    } else if (ft == FACE_COARSER) {
      int oa, ob;
      sub_origins_ab(f, F.sub[f], oa, ob);
      if (p < NF / 4) {
        const int ca = (p & 7) + 8 * oa, cb = (p >> 3) + 8 * ob;
        store_device(h + (size_t)F.nbr[f][0] * NH + halo_index(f ^ 1, ca, cb), f2c_mean<T>(f ^ 1, ca, cb, L, false));
      }
    } else {
#pragma unroll 1
      for (int sub = 0; sub < 4; sub++)
        store_device(h + (size_t)F.nbr[f][sub] * NH + halo_index(f ^ 1, p & 15, p >> 4),
                     c2f_trilinear<T>(f ^ 1, sub, p & 15, p >> 4, L));
    }
  }
}

// ------------------------------------------------------------------------------------------
// BiCGSTAB after its initialisation (r, r0, b.b and rho are there).  TWO false: the reference's
// Jacobi preconditioner on the FP64 matrix.  TWO true: the multiplicative two-level preconditioner
// (bi_precond_gsk_kernel, coarse_apply_mul_kernel) on the FP32 matrix; every workgroup forms the
// coarse corrections of its own and its neighbours' blocks itself, from the block sums that the
// meetings carry along.
//   per iteration: P meet Q meet S meet T meet XR meet
// ------------------------------------------------------------------------------------------
// PAIR (two workgroups a compute unit, Jacobi): 128 registers a thread and 80 KB of LDS.  x and r0 stay
// in memory (32 KB a block, from L2), q_ goes to LDS, p_ is formed again where it is added to x, and the
// columns' partial sums take the place of the ghosts that the matvec has read.
template <bool TWO, bool PAIR>
__global__ __launch_bounds__(RS_NT, PAIR ? 4 : 2) void resident_bicg_kernel(ResidentBicg a) {
  static_assert(!(TWO && PAIR));
  using TM = std::conditional_t<TWO, float, double>;
  constexpr int EN = kWords<PAIR>;
  __shared__ Operand<double> Z;
  // x and r0: read once or twice an iteration, so LDS holds them
  __shared__ double xs[PAIR ? 1 : NC], r0s[PAIR ? 1 : NC], qs[PAIR ? NC : 1];
  __shared__ double chains[PAIR ? 1 : 3][NF];
  double(*const chain)[NF] = PAIR ? reinterpret_cast<double(*)[NF]>(Z.side) : chains;
  static_assert(4 * NF >= 3 * NF);
  __shared__ MeetLds L;
  // TWO: block sums of r, q_, p over the case, the coarse right-hand side, and the corrections of
  // this block (0) and of the blocks its ghosts come from (near.at[4 face + quarter])
  __shared__ double br[TWO ? RS_MAX : 1], bq[TWO ? RS_MAX : 1], bp[TWO ? RS_MAX : 1], cv[TWO ? RS_MAX : 1];
  __shared__ FaceLds faces;
  __shared__ double ev[25];
  __shared__ NearLds near;
  const int slot = a.active[blockIdx.x];
  const DevBlock& B = a.blk[slot];
  const int c = B.case_id;
  SolveState S = scalar(a.st[c]);
  if (S.done) return;
  const DevCase& C = a.cs[c];
  const int t = threadIdx.x, tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK, lane = t & 63;
  const bool lower = kb == 0;
  const size_t g0 = (size_t)slot * NC + tx + NB * ty + NF * kb;
  const int l0 = tx + NB * ty + NF * (kb + 1);  // the thread's first cell in Z.zpad
  const int nn = C.nblk;
  Meeting meet{a.words, a.nslots, C.slot_begin, nn, slot};
  if (t == 0) L.failed = 0;
  faces.load(B, C, BC_NULL);
  const double omega = S.omega;
  int ix = 0, iy = 0, iz = 0;  // where this thread's ghost corrections are in ev
  if (t == 0) near.load(B, slot);
  if constexpr (TWO) {
    __syncthreads();
    auto where = [&](int f, int i, int j) {  // outer face: the block's own
      int u0 = 0, u1 = 0;
      if (B.ftype[f] == FACE_FINER) face_ab_to_o(f, i, j, u0, u1);
      return near.at[4 * f + (u0 >= NB / 2 ? 1 : 0) + (u1 >= NB / 2 ? 2 : 0)];
    };
    ix = where(tx == 0 ? 0 : 1, ty, kb);
    iy = where(ty == 0 ? 2 : 3, tx, kb);
    iz = where(lower ? 4 : 5, tx, ty);
    for (int b = t; b < nn; b += RS_NT) {
      br[b] = a.ce[2 * a.nslots + C.slot_begin + b];
      bq[b] = S.iter ? a.ce[3 * a.nslots + C.slot_begin + b] : 0.0;
      bp[b] = S.iter ? a.ce[4 * a.nslots + C.slot_begin + b] : 0.0;
    }
  }
  ClassRows<TM> R;
  Coef7<TM> A;
  if constexpr (TWO) {
    R = a.R32;
    A = a.A32;
  } else {
    R = a.R64;
    A = a.A64;
  }
  const unsigned ex = R.uni ? R.ex[(size_t)slot * 512 + t] : 0xffu;  // cells with bands of their own
  uint4 rin = {}, rend = {};  // TWO: the preconditioner records of the half column's two classes
  if (TWO && R.uni) {
    const uint4* tr = a.trec + (size_t)slot * 27 + stencil_class1(tx) + 3 * stencil_class1(ty);
    rin = tr[9];
    rend = tr[lower ? 0 : 18];
  }
  double r[RS_NK], p[RS_NK], q[RS_NK], pp[RS_NK], tt[RS_NK];
#pragma unroll
  for (int k = 0; k < RS_NK; k++) {
    r[k] = a.V.r[g0 + NF * k];
    p[k] = S.iter ? a.V.p[g0 + NF * k] : 0.0;
    q[k] = S.iter ? a.V.q[g0 + NF * k] : 0.0;
    if constexpr (PAIR) {
      qs[l0 - NF + NF * k] = q[k];
    } else {
      r0s[l0 - NF + NF * k] = a.V.r0[g0 + NF * k];
      xs[l0 - NF + NF * k] = a.x[g0 + NF * k];
    }
  }
  __syncthreads();

  // TWO: corrections ev = A_c^-1 cv of the blocks in `near`, one wavefront a row.  A case of at most
  // RS_MAX blocks has one float4 of a row per lane; coarse_load, before the meeting whose words the
  // right-hand side waits for, has them on their way.
  constexpr int CR = (25 + RS_NT / 64 - 1) / (RS_NT / 64);
  static_assert(RS_MAX <= 256, "one float4 of a row per lane");
  float4 crow[CR];
  auto coarse_load = [&]() {
    if constexpr (TWO) {
      const int u = thread_here(), np = coarse_pitch(nn);
#pragma unroll
      for (int i = 0; i < CR; i++) {
        const int e = (u >> 6) + i * (RS_NT / 64);
        if (e < near.n && 4 * (u & 63) < np)
          crow[i] = reinterpret_cast<const float4*>(a.cinv + a.coff[c] +
                                                    (size_t)(near.slot[e] - C.slot_begin) * np)[u & 63];
      }
    }
  };
  auto coarse = [&]() {
    if constexpr (TWO) {
      const int u = thread_here(), ln = u & 63;
#pragma unroll
      for (int i = 0; i < CR; i++) {
        const int e = (u >> 6) + i * (RS_NT / 64);
        if (e < near.n) {
          double v = 0.0;  // coarse_row_dot's order (a lane past the row adds nothing)
          if (4 * ln < coarse_pitch(nn)) {
            v += (double)crow[i].x * cv[4 * ln];
            v += (double)crow[i].y * cv[4 * ln + 1];
            v += (double)crow[i].z * cv[4 * ln + 2];
            v += (double)crow[i].w * cv[4 * ln + 3];
          }
          for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
          if (ln == 0) ev[e] = v;
        }
      }
      __syncthreads();
    }
  };
  auto coarse_rhs = [&](auto rhs) {
    if constexpr (TWO) {
      for (int b = t; b < coarse_pitch(nn); b += RS_NT) cv[b] = b < nn ? rhs(b) : 0.0;
      __syncthreads();
    }
  };

  // !TWO: to(k, omega v / Ap) for the thread's cells
  auto jacobi = [&](const double (&v)[RS_NK], const auto& to) __attribute__((always_inline)) {
    const int t = thread_here(), tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK;
    const bool lower = kb == 0;
    const TM* tr = class_column(R.tab, slot, tx, ty);
    const double din = R.uni ? (double)tr[9 * 8] : 0.0, dend = R.uni ? (double)tr[lower ? 0 : 18 * 8] : 0.0;
#pragma unroll
    for (int k = 0; k < RS_NK; k++) {
      double d = k == 0 ? (lower ? dend : din) : k == RS_NK - 1 ? (lower ? din : dend) : din;
      if ((ex >> k) & 1u) d = A.p[0][(size_t)slot * NC + tx + NB * ty + NF * (kb + k)];
      to(k, omega * (v[k] / d));
    }
  };
  // z = M v into Z.zpad (bi_precond_kernel / bi_precond_gsk_kernel), its ghosts pushed to h
  auto precond = [&](const double (&v)[RS_NK], double* h) __attribute__((always_inline)) {
    const int t = thread_here(), tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK;
    const bool lower = kb == 0;
    const size_t g0 = (size_t)slot * NC + tx + NB * ty + NF * kb;
    const int l0 = tx + NB * ty + NF * (kb + 1);
    double* const z = Z.zpad + NF;
    if constexpr (!TWO) {
      jacobi(v, [&](int k, double z) { Z.zpad[l0 + NF * k] = z; });
    } else {
      const double eo = ev[0], ex_ = ev[ix], ey = ev[iy], ez = ev[iz];
      const int par = (tx + ty) & 1;
      double ur[RS_NK / 2], ub[RS_NK / 2];
      uint32_t wr[RS_NK / 2][3], wb[RS_NK / 2][3];
      const uint32_t mx = (tx == 0 ? 0xffff0000u : ~0u) & (tx == NB - 1 ? 0x0000ffffu : ~0u);
      const uint32_t my = (ty == 0 ? 0xffff0000u : ~0u) & (ty == NB - 1 ? 0x0000ffffu : ~0u);
      Z.zpad[t < NF ? t : NC + t] = 0.0;
#pragma unroll
      for (int k = 0; k < RS_NK; k++) {
        uint4 rc = k == 0 ? pick(lower, rend, rin) : k == RS_NK - 1 ? pick(lower, rin, rend) : rin;
        if ((ex >> k) & 1u) rc = a.rec[g0 + NF * k];
        const int ka = kb + k, m = k >> 1;
        double uk = v[k] * (double)__uint_as_float(rc.x);
        uk -= eo + half_lo(rc.y) * (tx > 0 ? eo : ex_) + half_hi(rc.y) * (tx < NB - 1 ? eo : ex_) +
              half_lo(rc.z) * (ty > 0 ? eo : ey) + half_hi(rc.z) * (ty < NB - 1 ? eo : ey) +
              half_lo(rc.w) * (ka > 0 ? eo : ez) + half_hi(rc.w) * (ka < NB - 1 ? eo : ez);
        const uint32_t mz = (ka == 0 ? 0xffff0000u : ~0u) & (ka == NB - 1 ? 0x0000ffffu : ~0u);
        if ((k & 1) == par) {
          ur[m] = uk;
          wr[m][0] = rc.y & mx;
          wr[m][1] = rc.z & my;
          wr[m][2] = rc.w & mz;
        } else {
          ub[m] = uk;
          wb[m][0] = rc.y & mx;
          wb[m][1] = rc.z & my;
          wb[m][2] = rc.w & mz;
        }
      }
      // The sweeps.  The thread's 8 values stay in registers: a cell's own old value and its k
      // neighbours are the thread's (but one across the half column's end), so of seven LDS reads a cell
      // four are left, all issued before the first sum: a half sweep is a chain of LDS latency, sums and
      // a barrier (four sweeps 5.1 us; with seven reads in turn 6.0).
      double zr[RS_NK / 2], zb[RS_NK / 2];
      double* const z0 = z + tx + NB * ty + NF * kb;
#pragma unroll
      for (int m = 0; m < RS_NK / 2; m++) {
        zr[m] = omega * ur[m];
        zb[m] = 0.0;
        z0[NF * (2 * m + par)] = zr[m];
        z0[NF * (2 * m + 1 - par)] = 0.0;
      }
      __syncthreads();
      auto half = [&](auto red_tag, bool from_zero) __attribute__((always_inline)) {
        constexpr bool RED = decltype(red_tag)::value;
        const int cp = RED ? par : 1 - par;
        double(&mine)[RS_NK / 2] = RED ? zr : zb;
        const double(&other)[RS_NK / 2] = RED ? zb : zr;
        const double past = z0[cp ? NF * RS_NK : -NF];  // the k neighbour across the half column's end
        double side[RS_NK / 2][4];
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) {
          const double* const zc = z0 + NF * (2 * m + cp);
          side[m][0] = zc[-1];
          side[m][1] = zc[1];
          side[m][2] = zc[-NB];
          side[m][3] = zc[NB];
        }
        double column[RS_NK / 2 + 2];  // the other colour's values, `past` at either end (one of the two is used)
        column[0] = past;
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) column[m + 1] = other[m];
        column[RS_NK / 2 + 1] = past;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) {
          uint32_t w[3];
#pragma unroll
          for (int b = 0; b < 3; b++) w[b] = RED ? wr[m][b] : wb[m][b];
          // keep the couplings packed (see bi_precond_gsk_kernel)
          asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]));
          const double below = pick(cp != 0, column[m + 1], column[m]);
          const double above = pick(cp != 0, column[m + 2], column[m + 1]);
          double sum = half_lo(w[0]) * side[m][0];
          sum = __builtin_fma(half_hi(w[0]), side[m][1], sum);
          sum = __builtin_fma(half_lo(w[1]), side[m][2], sum);
          sum = __builtin_fma(half_hi(w[1]), side[m][3], sum);
          sum = __builtin_fma(half_lo(w[2]), below, sum);
          sum = __builtin_fma(half_hi(w[2]), above, sum);
          const double zn = (RED ? ur[m] : ub[m]) - sum;
          mine[m] = from_zero ? omega * zn : __builtin_fma(omega, zn - mine[m], mine[m]);
          z0[NF * (2 * m + cp)] = mine[m];
        }
        __syncthreads();
      };
      half(std::false_type{}, true);
#pragma unroll 1
      for (int sweep = 1; sweep < a.sweeps; sweep++) {
        half(std::true_type{}, false);
        half(std::false_type{}, false);
      }
#pragma unroll
      for (int m = 0; m < RS_NK / 2; m++) {
        z0[NF * (2 * m + par)] = zr[m] + eo;
        z0[NF * (2 * m + 1 - par)] = zb[m] + eo;
      }
    }
    __syncthreads();
    push_faces<double>(faces, slot, [&](int i, int j, int k) { return z[i + NB * (j + NB * k)]; }, h, h);
  };
  // y = A z with the ghosts the others pushed
  auto matvec = [&](const double* h, double (&y)[RS_NK]) __attribute__((always_inline)) {
    const int u = thread_here(), ux = u & 15, uy = (u >> 4) & 15, uk = (u >> 8) * RS_NK;
    HalfRows<TM> W;
    W.load(R, slot, ux, uy, uk == 0);
    Z.load_ghosts(h, slot);
    __syncthreads();
    half_matvec<double, TM>(Z, W, A, ex, (size_t)slot * NC + ux + NB * uy + NF * uk, ux, uy, uk, y);
  };
  auto keep = [&](double* to) {  // a word of every block into LDS
    return [=](const double (&e)[EN]) {
      const int lane = thread_here() & 63;
#pragma unroll
      for (int m = 0; m < EN; m++)
        if (lane + 64 * m < nn) to[lane + 64 * m] = e[m];
    };
  };

  auto shadow = [&]() -> const double* {
    if constexpr (PAIR) return a.V.r0 + (size_t)slot * NC;
    return r0s;
  };
  FinXr f = {};
  double alpha = S.alpha, beta = S.beta, gamma = S.gamma, rho = S.rr1, rho_n = rho;
  int n = S.iter;
  const int stop = n + a.turns;
  bool ok = true;
  coarse_load();
  while (true) {
    n++;
    const bool first = n == 1;
    const double ng = -gamma;
    // P
    coarse_rhs([&](int b) { return first ? br[b] : br[b] + beta * (bp[b] + ng * bq[b]); });
    coarse();
    double vs = 0.0;
#pragma unroll
    for (int k = 0; k < RS_NK; k++) {
      const double qk = PAIR ? qs[l0 - NF + NF * k] : q[k];
      p[k] = first ? r[k] : r[k] + beta * (p[k] + ng * qk);
      vs += p[k];
    }
    precond(p, a.V.hpp);
    if constexpr (!PAIR)
#pragma unroll
      for (int k = 0; k < RS_NK; k++) pp[k] = Z.zpad[l0 + NF * k];
    if constexpr (TWO) {
      for (int o = 32; o > 0; o >>= 1) vs += __shfl_xor(vs, o, 64);
      if ((thread_here() & 63) == 0) L.red[2][thread_here() >> 6] = vs;  // goes out with q_'s sums
    }
    ok = meet.neighbours(L, near.slot, near.n);
    if (!ok) break;
    // Q
    matvec(a.V.hpp, q);
    if constexpr (PAIR) __syncthreads();  // the ghosts have been read
    column_sums<2>(chain, L, [&](double* v) {
      const int u = thread_here();  // the thread's cells are u + 256 k in xs and r0s, from the half's base on
      const double* const r0 = shadow() + (u & (NF - 1)) + (u >> 8) * RS_NK * NF;
#pragma unroll
      for (int k = 0; k < RS_NK; k++) {
        v[0] += q[k] * r0[NF * k];
        v[1] += q[k];
      }
    });
    if constexpr (PAIR)
#pragma unroll
      for (int k = 0; k < RS_NK; k++) qs[l0 - NF + NF * k] = q[k];
    coarse_load();
    ok = meet.template all<TWO ? 3 : 1, EN, 4, RS_NT / 64>(L, [&](int k, const double (&e)[EN]) {
      if (k == 1)
        keep(bq)(e);
      else if (k == 2)
        keep(bp)(e);
      else {
        const double s = TWO ? lane_order(e) : case_order(e);
        if (lane == 0) L.sum[0] = s;
      }
    });
    if (!ok) break;
    alpha = scalar(rho / L.sum[0]);
    const double na = -alpha;
    // S (r becomes s)
    coarse_rhs([&](int b) { return na * bq[b] + br[b]; });
    coarse();
#pragma unroll
    for (int k = 0; k < RS_NK; k++) r[k] = na * (PAIR ? qs[l0 - NF + NF * k] : q[k]) + r[k];
    precond(r, a.V.hss);
    ok = meet.neighbours(L, near.slot, near.n);
    if (!ok) break;
    // T
    matvec(a.V.hss, tt);
    if constexpr (PAIR) __syncthreads();
    column_sums<2>(chain, L, [&](double* v) {
#pragma unroll
      for (int k = 0; k < RS_NK; k++) {
        v[0] += tt[k] * r[k];
        v[1] += tt[k] * tt[k];
      }
    });
    ok = meet.template all<2, EN>(L, [&](int k, const double (&e)[EN]) {
      const double s = case_order(e);
      if (lane == 0) L.sum[k] = s;
    });
    if (!ok) break;
    gamma = scalar(L.sum[0] / L.sum[1]);
    const double mg = -gamma;
    // XR
    {
      const int u = thread_here(), own = (u & (NF - 1)) + (u >> 8) * RS_NK * NF;
      double* const xb = PAIR ? a.x + (size_t)slot * NC : xs;
      auto add = [&](int k, double pk) {
        double& x = xb[own + NF * k];
        x = alpha * pk + gamma * Z.zpad[NF + own + NF * k] + x;  // s_ is still there
      };
      if constexpr (PAIR)
        jacobi(p, add);
      else
#pragma unroll
        for (int k = 0; k < RS_NK; k++) add(k, pp[k]);
#pragma unroll
      for (int k = 0; k < RS_NK; k++) r[k] = mg * tt[k] + r[k];
    }
    column_sums<3>(chain, L, [&](double* v) {
      const int u = thread_here();
      const double* const r0 = shadow() + (u & (NF - 1)) + (u >> 8) * RS_NK * NF;
#pragma unroll
      for (int k = 0; k < RS_NK; k++) {
        v[2] += r[k];
        v[0] += r[k] * r[k];
        v[1] += r[k] * r0[NF * k];
      }
    });
    coarse_load();
    ok = meet.template all<TWO ? 3 : 2, EN>(L, [&](int k, const double (&e)[EN]) {
      if (k == 2)
        keep(br)(e);
      else {
        const double s = case_order(e);
        if (lane == 0) L.sum[k] = s;
      }
    });
    if (!ok) break;
    S.alpha = alpha;
    S.gamma = gamma;
    rho_n = rho;
    f = scalar(fin_bi_xr_eval(S, L.sum[0], L.sum[1], n, rho_n));
    rho = f.rr1;
    beta = f.beta;
    if (f.done || n >= stop) break;
  }
  if (!ok) {
    if (t == 0) store_device(&a.st[c].parity, -1);
    return;
  }
#pragma unroll
  for (int k = 0; k < RS_NK; k++) {
    if constexpr (!PAIR) a.x[g0 + NF * k] = xs[l0 - NF + NF * k];
    if (!f.done) {  // to be continued by the next launch
      a.V.r[g0 + NF * k] = r[k];
      a.V.p[g0 + NF * k] = p[k];
      a.V.q[g0 + NF * k] = PAIR ? qs[l0 - NF + NF * k] : q[k];
    }
  }
  if (TWO && t == 0 && !f.done) {
    a.ce[2 * a.nslots + slot] = br[slot - C.slot_begin];
    a.ce[3 * a.nslots + slot] = bq[slot - C.slot_begin];
    a.ce[4 * a.nslots + slot] = bp[slot - C.slot_begin];
  }
  if (t == 0 && slot == C.slot_begin) {
    SolveState& G = a.st[c];
    G.alpha = alpha;
    G.gamma = gamma;
    fin_bi_xr_store(G, f, n, rho_n);
  }
}

// ------------------------------------------------------------------------------------------
// Jacobi-PCG after its initialisation (r, b.b and r.z are there): P neighbours Q meet XR meet
// ------------------------------------------------------------------------------------------
// PAIR: x stays in memory, z and Ap are formed where they are used.
template <class T, bool PAIR>
__global__ __launch_bounds__(RS_NT, PAIR ? 4 : 2) void resident_cg_kernel(ResidentCg<T> a) {
  constexpr int EN = kWords<PAIR>;
  __shared__ Operand<T> Z;
  __shared__ double chain[2][NF];
  __shared__ MeetLds L;
  __shared__ FaceLds faces;
  __shared__ NearLds near;
  const int slot = a.active[blockIdx.x];
  const DevBlock& B = a.blk[slot];
  const int c = B.case_id;
  SolveState S = scalar(a.st[c]);
  if (S.done) return;
  const DevCase& C = a.cs[c];
  const int t = threadIdx.x, tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK, lane = t & 63;
  const size_t g0 = (size_t)slot * NC + tx + NB * ty + NF * kb;
  Meeting meet{a.words, a.nslots, C.slot_begin, C.nblk, slot};
  if (t == 0) {
    L.failed = 0;
    near.load(B, slot);
  }
  faces.load(B, C, BC_NULL);
  const T omega = (T)S.omega;
  const unsigned ex = a.R.uni ? a.R.ex[(size_t)slot * 512 + t] : 0xffu;
  T x[RS_NK], r[RS_NK], p[RS_NK], z[RS_NK], d[RS_NK];  // d: Ap
  // to(k, Ap) for the thread's cells
  auto diagonal = [&](const auto& to) __attribute__((always_inline)) {
    const int t = thread_here(), tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK;
    const bool lower = kb == 0;
    const T* tr = class_column(a.R.tab, slot, tx, ty);
    const T din = a.R.uni ? tr[9 * 8] : (T)0, dend = a.R.uni ? tr[lower ? 0 : 18 * 8] : (T)0;
#pragma unroll
    for (int k = 0; k < RS_NK; k++) {
      T v = k == 0 ? pick(lower, dend, din) : k == RS_NK - 1 ? pick(lower, din, dend) : din;
      if ((ex >> k) & 1u) v = a.A.p[0][(size_t)slot * NC + tx + NB * ty + NF * (kb + k)];
      to(k, v);
    }
  };
#pragma unroll
  for (int k = 0; k < RS_NK; k++) {
    if constexpr (!PAIR) x[k] = a.x[g0 + NF * k];
    r[k] = a.r[g0 + NF * k];
    p[k] = S.iter ? a.p[g0 + NF * k] : (T)0;
  }
  if constexpr (!PAIR)
    diagonal([&](int k, T v) {
      d[k] = v;
      z[k] = omega * (r[k] / v);
    });
  __syncthreads();
  const int stop = S.iter + a.turns;
  bool ok = true;
  for (int n = S.iter + 1;; n++) {
    // P
    const T beta = (T)S.beta;
    {
      const int u = thread_here(), own = (u & (NF - 1)) + NF * ((u >> 8) * RS_NK + 1);
      auto step = [&](int k, T zk) {
        p[k] = n == 1 ? zk : zk + beta * p[k];
        Z.zpad[own + NF * k] = p[k];
      };
      if constexpr (PAIR)
        diagonal([&](int k, T v) { step(k, omega * (r[k] / v)); });
      else
#pragma unroll
        for (int k = 0; k < RS_NK; k++) step(k, z[k]);
    }
    __syncthreads();
    push_faces<T>(faces, slot, [&](int i, int j, int k) { return Z.zpad[NF + i + NB * (j + NB * k)]; }, a.hp, a.hp);
    ok = meet.neighbours(L, near.slot, near.n);
    if (!ok) break;
    // Q
    T q[RS_NK];
    {
      const int u = thread_here(), ux = u & 15, uy = (u >> 4) & 15, uk = (u >> 8) * RS_NK;
      HalfRows<T> W;
      W.load(a.R, slot, ux, uy, uk == 0);
      Z.load_ghosts(a.hp, slot);
      __syncthreads();
      half_matvec<T, T>(Z, W, a.A, ex, (size_t)slot * NC + ux + NB * uy + NF * uk, ux, uy, uk, q);
    }
    column_sums<1>(chain, L, [&](double* v) {
#pragma unroll
      for (int k = 0; k < RS_NK; k++) v[0] += (double)q[k] * (double)p[k];
    });
    ok = meet.template all<1, EN>(L, [&](int, const double (&e)[EN]) {
      const double s = case_order(e);
      if (lane == 0) L.sum[0] = s;
    });
    if (!ok) break;
    S.alpha = scalar(S.rr1 / L.sum[0]);
    const T alpha = (T)S.alpha, nalpha = -alpha;
    // XR
#pragma unroll
    for (int k = 0; k < RS_NK; k++) {
      if constexpr (!PAIR) x[k] = x[k] + alpha * p[k];
      r[k] = r[k] + nalpha * q[k];
      if constexpr (!PAIR) z[k] = omega * (r[k] / d[k]);
    }
    if constexpr (PAIR) {
      const int u = thread_here();
      T* const xb = a.x + (size_t)slot * NC + (u & (NF - 1)) + (u >> 8) * RS_NK * NF;
#pragma unroll
      for (int k = 0; k < RS_NK; k++) xb[NF * k] = xb[NF * k] + alpha * p[k];
      diagonal([&](int k, T v) { z[k] = omega * (r[k] / v); });
    }
    column_sums<2>(chain, L, [&](double* v) {
#pragma unroll
      for (int k = 0; k < RS_NK; k++) {
        v[0] += (double)r[k] * (double)r[k];
        v[1] += (double)r[k] * (double)z[k];
      }
    });
    ok = meet.template all<2, EN>(L, [&](int k, const double (&e)[EN]) {
      const double s = case_order(e);
      if (lane == 0) L.sum[k] = s;
    });
    if (!ok) break;
    S.iter = n;
    cg_end(S, L.sum[0], L.sum[1], n);
    S = scalar(S);
    if (S.done || n >= stop) break;
  }
  if (!ok) {
    if (t == 0) store_device(&a.st[c].parity, -1);
    return;
  }
#pragma unroll
  for (int k = 0; k < RS_NK; k++) {
    if constexpr (!PAIR) a.x[g0 + NF * k] = x[k];
    if (!S.done) {  // to be continued by the next launch
      a.r[g0 + NF * k] = r[k];
      a.p[g0 + NF * k] = p[k];
    }
  }
  if (t == 0 && slot == C.slot_begin) a.st[c] = S;
}

// ------------------------------------------------------------------------------------------
// RBGS (MODE 0) and Jacobi (MODE 1): iteration n sweeps x^{n-1} to x^n, pushes its ghosts into the
// other halo buffer and meets over the residual of x^{n-1} (rbgs_iter_kernel).  The result, x and
// its ghosts, goes to buffer 0.  PAIR: b stays in memory and the bands are read again each iteration.
// ------------------------------------------------------------------------------------------
template <class T, int MODE, bool PAIR>
__global__ __launch_bounds__(RS_NT, PAIR ? 4 : 2) void resident_relax_kernel(ResidentRelax<T> a) {
  constexpr int EN = kWords<PAIR>;
  __shared__ Operand<T> Z;
  __shared__ MeetLds L;
  __shared__ FaceLds faces;
  __shared__ NearLds near;
  const int slot = a.active[blockIdx.x];
  const DevBlock& B = a.blk[slot];
  const int c = B.case_id;
  SolveState S = scalar(a.st[c]);
  if (S.done) return;
  const DevCase& C = a.cs[c];
  const int t = threadIdx.x, tx = t & 15, ty = (t >> 4) & 15, kb = (t >> 8) * RS_NK, lane = t & 63;
  const bool lower = kb == 0;
  const size_t g0 = (size_t)slot * NC + tx + NB * ty + NF * kb;
  Meeting meet{a.words, a.nslots, C.slot_begin, C.nblk, slot};
  if (t == 0) {
    L.failed = 0;
    near.load(B, slot);
  }
  faces.load(B, C, a.bcg);
  const T omega = (T)S.omega;
  const unsigned ex = a.R.uni ? a.R.ex[(size_t)slot * 512 + t] : 0xffu;
  T x[RS_NK], bv[RS_NK], dv[RS_NK];
  HalfRows<T> W;
  if constexpr (!PAIR) W.load(a.R, slot, tx, ty, lower);
#pragma unroll
  for (int k = 0; k < RS_NK; k++) {
    x[k] = a.x[g0 + NF * k];
    if constexpr (!PAIR) {
      bv[k] = a.b[g0 + NF * k];
      dv[k] = k == 0 ? pick(lower, W.end[0], W.in[0]) : k == RS_NK - 1 ? pick(lower, W.in[0], W.end[0]) : W.in[0];
      if ((ex >> k) & 1u) dv[k] = a.A.p[0][g0 + NF * k];
    }
    Z.zpad[tx + NB * ty + NF * (kb + k + 1)] = x[k];
  }
  __syncthreads();
  const int stop = S.iter + a.turns;
  int cur = 0;
  bool ok = true;
  T xn[RS_NK];
  for (int n = S.iter + 1;; n++) {
    const int u = thread_here(), ux = u & 15, uy = (u >> 4) & 15, uk = (u >> 8) * RS_NK;
    const size_t g = (size_t)slot * NC + ux + NB * uy + NF * uk;
    if constexpr (PAIR) W.load(a.R, slot, ux, uy, uk == 0);
    auto b = [&](int kk) -> T {
      if constexpr (PAIR) return a.b[g + NF * kk];
      return bv[kk];
    };
    auto d = [&](int kk) -> T {  // Ap
      if constexpr (!PAIR) return dv[kk];
      const T v = kk == 0 ? pick(uk != 0, W.in[0], W.end[0])
                          : kk == RS_NK - 1 ? pick(uk != 0, W.end[0], W.in[0]) : W.in[0];
      if ((ex >> kk) & 1u) return a.A.p[0][g + NF * kk];
      return v;
    };
    // b less the six neighbour products of cell kk with the bands w
    auto off_sum = [&](T bk, const T* w, int kk) -> T {
      const auto v = Z.around(ux, uy, uk + kk, ux + NB * uy + NF * (uk + kk + 1));
      return bk - w[1] * v.w - w[2] * v.e - w[3] * v.s - w[4] * v.n - w[5] * v.b - w[6] * v.t;
    };
    auto own_bands = [&](T* w, int kk) {
#pragma unroll
      for (int q = 1; q < 7; q++) w[q] = a.A.p[q][g + NF * kk];
    };
    Z.load_ghosts(a.h[cur], slot);
    __syncthreads();
    T rs[RS_NK];
#pragma unroll
    for (int kk = 0; kk < RS_NK; kk++) {
      T w[7];
#pragma unroll
      for (int q = 1; q < 7; q++)
        w[q] = kk == 0 ? pick(uk != 0, W.in[q], W.end[q])
                       : kk == RS_NK - 1 ? pick(uk != 0, W.end[q], W.in[q]) : W.in[q];
      rs[kk] = off_sum(b(kk), w, kk);
      if (kk & 1) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll 1
    for (unsigned m = ex; m; m &= m - 1) {
      const int kk = __builtin_ctz(m);
      T w[7];
      own_bands(w, kk);
      const T bk = a.b[g + NF * kk];
      const T v = off_sum(bk, w, kk);
#pragma unroll
      for (int k = 0; k < RS_NK; k++) rs[k] = k == kk ? v : rs[k];
    }
    double sums[2] = {0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < RS_NK; kk++) {
      const T r = rs[kk] - d(kk) * x[kk];
      sums[0] += (double)r * (double)r;
      if (n == 1) sums[1] += (double)b(kk) * (double)b(kk);
    }
    wave_sums<2>(sums, L, u >> 6);
    if (n <= S.countMax) {
      const int own = (u & (NF - 1)) + NF * (uk + 1);
      if constexpr (MODE == 1) {
#pragma unroll
        for (int kk = 0; kk < RS_NK; kk++) xn[kk] = x[kk] - omega * (x[kk] - rs[kk] / d(kk));
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < RS_NK; kk++) Z.zpad[own + NF * kk] = xn[kk];
      } else {
        // per pair of cells one is red, chosen by the column's parity
        const int par = (ux + uy) & 1;
        T xr[RS_NK / 2];
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) {
          const T xp = pick(par != 0, x[2 * m + 1], x[2 * m]);
          xr[m] = xp - omega * (xp - pick(par != 0, rs[2 * m + 1], rs[2 * m]) / pick(par != 0, d(2 * m + 1), d(2 * m)));
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) Z.zpad[own + NF * (2 * m + par)] = xr[m];
        __syncthreads();
        T sb[RS_NK / 2];  // black: off-diagonal sums from the new red values
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) {
          const bool e = m == 0 ? (par && !uk) : m == RS_NK / 2 - 1 ? (!par && uk) : false;
          T w[7];
#pragma unroll
          for (int q = 1; q < 7; q++) w[q] = pick(e, W.end[q], W.in[q]);
          sb[m] = off_sum(pick(par != 0, b(2 * m), b(2 * m + 1)), w, 2 * m + 1 - par);
        }
#pragma unroll 1
        for (unsigned mm = ex & (par ? 0x55u : 0xaau); mm; mm &= mm - 1) {
          const int kk = __builtin_ctz(mm);
          T w[7];
          own_bands(w, kk);
          const T bk = a.b[g + NF * kk];
          const T v = off_sum(bk, w, kk);
#pragma unroll
          for (int m = 0; m < RS_NK / 2; m++) sb[m] = m == kk >> 1 ? v : sb[m];
        }
#pragma unroll
        for (int m = 0; m < RS_NK / 2; m++) {
          const T xb = pick(par != 0, x[2 * m], x[2 * m + 1]);
          const T v = xb - omega * (xb - sb[m] / pick(par != 0, d(2 * m), d(2 * m + 1)));
          xn[2 * m] = pick(par != 0, v, xr[m]);
          xn[2 * m + 1] = pick(par != 0, xr[m], v);
          Z.zpad[own + NF * (2 * m + 1 - par)] = v;
        }
      }
      __syncthreads();
      push_faces<T>(faces, slot, [&](int i, int j, int k) { return Z.zpad[NF + i + NB * (j + NB * k)]; }, a.h[cur],
                    a.h[cur ^ 1]);
    }
    ok = meet.template all<2, EN, RS_NT / 64>(L, [&](int k, const double (&e)[EN]) {
      const double s = case_order(e);
      if (lane == 0) L.sum[k] = s;
    });
    if (!ok) break;
    // as FIN_RBGS
    S.iter = n;
    if (n == 1) {
      S.bb = L.sum[1];
      if (S.countMax < 1) S.done = 1;
    } else {
      converged(S, L.sum[0], n - 1);
    }
    S = scalar(S);
    if (S.done) break;  // x^{n-1} and the ghosts it was read with are the result
#pragma unroll
    for (int k = 0; k < RS_NK; k++) x[k] = xn[k];
    cur ^= 1;
    if (n >= stop) {  // to be continued by the next launch
      Z.load_ghosts(a.h[cur], slot);
      __syncthreads();
      break;
    }
  }
  if (!ok) {
    if (t == 0) store_device(&a.st[c].parity, -1);
    return;
  }
#pragma unroll
  for (int k = 0; k < RS_NK; k++) a.x[g0 + NF * k] = x[k];
#pragma unroll
  for (int q = 0; q < NH / RS_NT; q++) {
    const int w = t + RS_NT * q;
    a.h[0][(size_t)slot * NH + w] = w < 4 * NF ? Z.side[w] : Z.zpad[w < 5 * NF ? w - 4 * NF : NC + w - 4 * NF];
  }
  if (t == 0 && slot == C.slot_begin) a.st[c] = S;
}

// One workgroup per block of the active cases; kernels[0] with one workgroup a compute unit, for up to
// RS_MAX blocks, kernels[1] with two, for up to RS_MAX2 (limit[0], limit[1]: how many the device holds, -1
// not asked yet).  False: they do not fit on the device together, there is no such kernel, or the launch is
// refused; nothing was launched.
template <class Args>
bool launch_resident(const void* const (&kernels)[2], hipStream_t sm, int nact, int* limits, Args& args) {
  if (nact < 1 || nact > RS_MAX2) return false;
  const int pair = nact > RS_MAX;
  const void* const kernel = kernels[pair];
  if (!kernel) return false;
  int* const limit = limits + pair;
  if (*limit < 0) {
    int per = 0, dev = 0, cus = 0, coop = 0;
    *limit = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, RS_NT, 0) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    *limit = per * cus;
  }
  if (nact > *limit) return false;
  void* list[] = {&args};
  if (hipLaunchCooperativeKernel(kernel, dim3(nact), dim3(RS_NT), list, 0, sm) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}

bool launch_resident_bicg(hipStream_t sm, int nact, bool two, int* limits, ResidentBicg& args) {
  const void* const k[2] = {
      two ? (const void*)resident_bicg_kernel<true, false> : (const void*)resident_bicg_kernel<false, false>,
      two ? nullptr : (const void*)resident_bicg_kernel<false, true>};
  return launch_resident(k, sm, nact, limits, args);
}

template <class T>
bool launch_resident_cg(hipStream_t sm, int nact, int* limits, ResidentCg<T>& args) {
  const void* const k[2] = {(const void*)resident_cg_kernel<T, false>, (const void*)resident_cg_kernel<T, true>};
  return launch_resident(k, sm, nact, limits, args);
}
template <class T>
bool launch_resident_relax(hipStream_t sm, int nact, int mode, int* limits, ResidentRelax<T>& args) {
  const void* pair = (const void*)resident_relax_kernel<T, 1, true>;
  if (mode == 0) {  // FP64: its 36 spilled registers leave 0.95-1.15x of one launch per stage
    pair = nullptr;
    if constexpr (sizeof(T) == 4) pair = (const void*)resident_relax_kernel<T, 0, true>;
  }
  const void* one = (const void*)resident_relax_kernel<T, 1, false>;
  if (mode == 0) one = (const void*)resident_relax_kernel<T, 0, false>;
  const void* const k[2] = {one, pair};
  return launch_resident(k, sm, nact, limits, args);
}
template bool launch_resident_cg<double>(hipStream_t, int, int*, ResidentCg<double>&);
template bool launch_resident_cg<float>(hipStream_t, int, int*, ResidentCg<float>&);
template bool launch_resident_relax<double>(hipStream_t, int, int, int*, ResidentRelax<double>&);
template bool launch_resident_relax<float>(hipStream_t, int, int, int*, ResidentRelax<float>&);

void launch_unset_words(hipStream_t sm, const int* active, int nact, unsigned long long* words, size_t nslots) {
  if (nact)
    hipLaunchKernelGGL(unset_words_kernel, dim3((RS_WORDS * nact + 255) / 256), dim3(256), 0, sm, active, nact, words,
                       nslots);
}

}  // namespace ffvhc
