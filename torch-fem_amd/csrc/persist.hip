// Preconditioned CG of a small system in one kernel.
//
// An iteration of the general path (solver.hip) is two to four launches of 3
// to 6 us each, whatever little they compute: on systems of a few thousand to
// some tens of thousands of unknowns these launches, and the seven launches
// and two host round trips of every refinement, are the solve's time. Here
// one block per CU stays on the chip for the whole solve, refinements
// included. A block owns a contiguous range of nodes and keeps in its 160 KB
// of LDS: its rows of K (FP32 or FP64; streamed from L2 instead when they do
// not fit), its entries of x, r, u, p, s and of the preconditioner, the list
// of the distinct nodes its rows couple to (its halo), and a 16-bit halo
// index per neighbour block.
//
// Per iteration a block gathers the u of its halo once (every entry is then
// used from LDS, about 6 times on a hexahedral mesh), forms w = K u, updates
// p and s, and takes part in two exchanges, eta = p.s and (r.u, r.r):
//   * a block publishes its partial sums as words that carry 32 bits of
//     payload and a 32-bit epoch, and every block polls the words of all
//     blocks and adds them in block order. A sum and a grid barrier are thus
//     one store and one load, about 2.6 us.
//     Each block publishes to 8 copies of its words and polls one of them: 256
//     blocks polling the same lines took 3.6 us per exchange, not 2.7;
//   * (r.u, r.r) are published with u and collected only after the next
//     product, which waits for the blocks that own halo nodes alone;
//   * u goes through device-scope (L2-bypassing) stores and loads; a wave
//     waits for its stores before it publishes, so whoever has seen the epoch
//     sees the u. No fence is needed, and none is paid for: an agent-scope
//     fence per block measured 6 to 16 us on 128 to 256 blocks.
// All blocks form the same sums in the same order, so they take the same
// decisions; results do not vary from run to run, unless a wait is given up (see
// below).
//
// Every wait is bounded (50 ms): if some block has not been scheduled by then
// (another process holds CUs), it sets the abort word and leaves, and with it
// every block that waits for it. x is still a valid guess, some blocks having
// folded a correction into it and others not, and the caller solves on the
// general path, as do the thread's solves on the device for the next 4 s (another
// process on the GPU tends to stay; a solver handle may live for one solve). Whether a solve counts is decided
// by the abort word, read once the kernel has ended, not by block 0: at the
// last exchange of a solve block 0 may have seen every block that another gave
// up on, and at b = 0 the block that left has not cleared its part of x.
//
// Of the 6.4 us of an iteration on a 14^3 Hexa1 cube (84 blocks) about 2.6 are
// the wait for eta, 0.7 and 0.8 those for the neighbours' u and for (r.u, r.r),
// 1.2 the gather and the product, 1.3 the updates. persist_solve compares it
// with the general path.
#include "solver_common.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <mutex>
#include <type_traits>

namespace tfm {
namespace {

constexpr int PT = 1024;                     // threads per block
constexpr unsigned P_STATIC_LDS = 2048;      // room for the static LDS (checked below)
constexpr unsigned P_LDS = 160 * 1024 - P_STATIC_LDS;
constexpr long long P_WAIT_TICKS = 5000000;  // 50 ms of the 100 MHz clock

struct PersistArgs {
  int64_t n_nod;
  int npb;  // nodes per block
  const int32_t *adj_ptr, *adj;
  const int64_t *val_ptr;
  const int64_t *rowptr;
  const int32_t *col;
  const void *val;
  const double *val64, *dblk;
  int pc;
  const double *b;
  double *x;
  void *ug, *pg;
  unsigned long long *slots;
  PersistResult *res;
  double rtol, delta, final_rtol;
  int max_iter, extended;
  int quit;  // the point where the last block gives up (0: none), see `quits`
};

template <typename T> __device__ __forceinline__ T dev_load(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void dev_store(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__host__ __device__ constexpr unsigned up16(unsigned v) { return (v + 15u) & ~15u; }

// LDS bytes before the halo list, for npb nodes.
template <typename T, int ND> __host__ __device__ constexpr unsigned fixed_lds(unsigned npb) {
  return up16(4u * (3u * npb + 2u)) +
         up16((unsigned)sizeof(T) * npb * (6u * ND + (unsigned)pc_size<ND>()));
}

// Shared state of the exchanges of one block.
struct Exchange {
  double red[3 * (PT / 64)];  // wave sums
  double part[3 * 4];         // sums over the blocks polled by one wave
  int nb[PERSIST_MAX_BLOCKS];  // blocks that own halo nodes
  int n_nb;
  int dead;
};

// Slots of one exchange: word w of value k of block b, in each of 8 copies.
// A block publishes to every copy (lanes of one store) and polls copy
// blockIdx % 8 only, so that a line is polled by an eighth of the blocks.
__device__ __forceinline__ unsigned long long *slot(const PersistArgs &A, unsigned epoch, int copy,
                                                    int word) {
  return A.slots + (((size_t)(epoch & 1u) * PERSIST_COPIES + copy) * 6 + word) * PERSIST_MAX_BLOCKS;
}

// Adds v[k] over the block's threads and publishes the sums as exchange
// `epoch`. Stores to device-scope data made before it are visible to whoever
// has seen the epoch in one of this block's words.
template <int NV>
__device__ __forceinline__ void publish(double (&v)[NV], Exchange &X, unsigned epoch,
                                        const PersistArgs &A) {
  constexpr int NW = PT / 64;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = lanes_sum<64>(v[k]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores have arrived
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) X.red[wave * NV + k] = v[k];
  __syncthreads();
  if (wave == 0) {
    double t[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) t[k] = lanes_sum<NW>(lane < NW ? X.red[lane * NV + k] : 0.0);
    // every group of NW lanes beyond the first has summed zeros: broadcast
#pragma unroll
    for (int k = 0; k < NV; ++k) t[k] = __shfl(t[k], 0, 64);
    const int copy = lane % PERSIST_COPIES, word = lane / PERSIST_COPIES;
    unsigned half = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (word == 2 * k) half = (unsigned)__double2loint(t[k]);
      if (word == 2 * k + 1) half = (unsigned)__double2hiint(t[k]);
    }
    if (word < 2 * NV)
      dev_store(slot(A, epoch, copy, word) + blockIdx.x, ((unsigned long long)epoch << 32) | half);
  }
}

// Polls `n` words until each carries the epoch; false after P_WAIT_TICKS or
// once some block has given up.
template <int N>
__device__ __forceinline__ bool poll(const unsigned long long *at, unsigned epoch,
                                     unsigned long long (&w)[N], const PersistArgs &A) {
  unsigned long long *abort = &A.res->abort;
  const long long t0 = wall_clock64();
  for (int spin = 0;; ++spin) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < N; ++k) w[k] = dev_load(at + k * PERSIST_MAX_BLOCKS);
#pragma unroll
    for (int k = 0; k < N; ++k) ok &= (unsigned)(w[k] >> 32) == epoch;
    if (ok) return true;
    if (spin % 32 == 31 && (dev_load(abort) != 0 || wall_clock64() - t0 > P_WAIT_TICKS)) {
      dev_store(abort, 1ull);
      return false;
    }
  }
}

// Waits until the blocks that own halo nodes have published `epoch`.
__device__ __forceinline__ bool wait_neighbours(Exchange &X, unsigned epoch,
                                                const PersistArgs &A) {
  if ((int)threadIdx.x < X.n_nb) {
    unsigned long long w[1];
    if (!poll<1>(slot(A, epoch, blockIdx.x % PERSIST_COPIES, 0) + X.nb[threadIdx.x], epoch, w, A))
      X.dead = 1;
  }
  __syncthreads();
  return X.dead == 0;
}

// The sums over all blocks of exchange `epoch`, the same bits in every block;
// a grid barrier as well. False if some block did not arrive.
template <int NV>
__device__ __forceinline__ bool collect(double (&v)[NV], Exchange &X, unsigned epoch,
                                        const PersistArgs &A) {
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, G = gridDim.x;
  if (wave * 64 < G) {
    double t[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) t[k] = 0.0;
    if (tid < G) {
      unsigned long long w[2 * NV];
      if (!poll<2 * NV>(slot(A, epoch, blockIdx.x % PERSIST_COPIES, 0) + tid, epoch, w, A))
        X.dead = 1;
#pragma unroll
      for (int k = 0; k < NV; ++k)
        t[k] = __hiloint2double((int)(unsigned)w[2 * k + 1], (int)(unsigned)w[2 * k]);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) t[k] = lanes_sum<64>(t[k]);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < NV; ++k) X.part[wave * NV + k] = t[k];
  }
  __syncthreads();
  const int nw = (G + 63) / 64;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double t = X.part[k];
    for (int q = 1; q < nw; ++q) t += X.part[q * NV + k];
    v[k] = t;
  }
  return X.dead == 0;
}

template <int NV>
__device__ __forceinline__ bool exchange(double (&v)[NV], Exchange &X, unsigned &epoch,
                                         const PersistArgs &A) {
  ++epoch;
  publish<NV>(v, X, epoch, A);
  return collect<NV>(v, X, epoch, A);
}

// QUIT: the last block gives up at point A.quit. (With that test in the kernels of
// QUIT = false too, an iteration of three DOFs took 2% longer.)
template <typename T, int ND, int TL, bool CSR, bool QUIT = false>
__global__ void __launch_bounds__(PT) k_pcg_persist(PersistArgs A) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ Exchange X;
  __shared__ int s_lo, s_hi, s_scan[PT / 64], s_H;
  static_assert(sizeof(X) + sizeof(s_scan) + 3 * sizeof(int) + 3 * 16 <= P_STATIC_LDS,
                "static LDS (with its padding) beyond the room left for it");
  constexpr bool FP64 = std::is_same<T, double>::value;
  constexpr bool DIFF = !FP64;  // FP32 values of one rhs are in difference form
  constexpr int PC = pc_size<ND>(), ND2 = ND * ND;
  const int tid = threadIdx.x, lane = tid % TL, team = tid / TL;
  constexpr int TEAMS = PT / TL;
  const int64_t n0 = min((int64_t)blockIdx.x * A.npb, A.n_nod);
  const int64_t n1 = min(n0 + A.npb, A.n_nod);
  const int nloc = (int)(n1 - n0);

  // ------------------------------------------------------------- LDS layout
  int *loc_a = reinterpret_cast<int *>(lds);  // first entry of each own node
  int *loc_v = loc_a + A.npb + 1;             // first value
  int *loc_s = loc_v + A.npb + 1;             // halo index of the node itself
  T *xv = reinterpret_cast<T *>(lds + up16(4u * (3u * A.npb + 2u)));
  T *rv = xv + A.npb * ND, *uv = rv + A.npb * ND, *pv = uv + A.npb * ND, *sv = pv + A.npb * ND;
  T *wv = sv + A.npb * ND, *mi = wv + A.npb * ND;
  const unsigned off_list = fixed_lds<T, ND>((unsigned)A.npb);

  const int64_t a_beg = CSR ? A.rowptr[n0] : (int64_t)A.adj_ptr[n0];
  const int64_t v_beg = CSR ? a_beg : A.val_ptr[n0];
  const int nent = (int)((CSR ? A.rowptr[n1] : (int64_t)A.adj_ptr[n1]) - a_beg);
  const int64_t nval = (CSR ? A.rowptr[n1] : A.val_ptr[n1]) - v_beg;
  const int32_t *cols = (CSR ? A.col : A.adj) + a_beg;
  for (int i = tid; i <= nloc; i += PT) {
    loc_a[i] = (int)((CSR ? A.rowptr[n0 + i] : (int64_t)A.adj_ptr[n0 + i]) - a_beg);
    loc_v[i] = (int)((CSR ? A.rowptr[n0 + i] : A.val_ptr[n0 + i]) - v_beg);
  }

  // -------------------------------------------- halo: the distinct columns
  // a bitmap over the window of columns [lo, hi], its prefix counts, then
  // the compact list and each entry's index in it
  if (tid == 0) {
    s_lo = 0x7fffffff;
    s_hi = -1;
    X.dead = 0;
    X.n_nb = 0;
  }
  __syncthreads();
  {
    int lo = 0x7fffffff, hi = -1;
    for (int k = tid; k < nent; k += PT) {
      const int c = cols[k];
      lo = min(lo, c);
      hi = max(hi, c);
    }
    if (hi >= 0) {
      atomicMin(&s_lo, lo);
      atomicMax(&s_hi, hi);
    }
  }
  __syncthreads();
  const int lo = s_lo;
  const unsigned window = s_hi >= 0 ? (unsigned)(s_hi - lo) + 1u : 0u;
  const unsigned nwords = (window + 31u) / 32u;
  bool fit = (unsigned long long)nwords * 8ull <= (unsigned long long)(P_LDS - off_list);
  const unsigned off_map = fit ? (P_LDS - nwords * 8u) & ~7u : P_LDS;
  fit = fit && off_map >= off_list;
  unsigned *map = reinterpret_cast<unsigned *>(lds + off_map), *pre = map + nwords;
  int H = 0;
  if (fit) {  // uniform in the block
    for (unsigned q = tid; q < nwords; q += PT) map[q] = 0u;
    __syncthreads();
    for (int k = tid; k < nent; k += PT) {
      const unsigned c = (unsigned)(cols[k] - lo);
      atomicOr(&map[c >> 5], 1u << (c & 31u));
    }
    __syncthreads();
    const unsigned chunk = (nwords + PT - 1) / PT, q0 = tid * chunk;
    int cnt = 0;
    for (unsigned q = q0; q < q0 + chunk && q < nwords; ++q) cnt += __popc(map[q]);
    int incl = cnt;  // inclusive scan over the wave, then over the waves
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (tid % 64 >= d) incl += o;
    }
    if (tid % 64 == 63) s_scan[tid / 64] = incl;
    __syncthreads();
    int run = incl - cnt;
    for (int w = 0; w < tid / 64; ++w) run += s_scan[w];
    for (unsigned q = q0; q < q0 + chunk && q < nwords; ++q) {
      pre[q] = (unsigned)run;
      run += __popc(map[q]);
    }
    if (tid == PT - 1) s_H = run;
    __syncthreads();
    H = s_H;
  }
  const unsigned long long off_halo = up16(off_list + 4u * (unsigned)H);
  const unsigned long long off_lidx = off_halo + 8ull * (unsigned)H * ND;
  const unsigned long long off_val = (off_lidx + 2ull * (unsigned)nent + 15ull) & ~15ull;
  fit = fit && H <= 65535 && off_val <= off_map;
  const bool resident = fit && off_val + sizeof(T) * (unsigned long long)nval <= P_LDS;
  int *list = reinterpret_cast<int *>(lds + off_list);
  double *halo64 = reinterpret_cast<double *>(lds + off_halo);
  T *halo = reinterpret_cast<T *>(halo64);
  uint16_t *lidx = reinterpret_cast<uint16_t *>(lds + off_lidx);
  if (fit) {
    for (unsigned q = tid; q < nwords; q += PT) {
      unsigned w = map[q];
      int at = (int)pre[q];
      while (w) {
        const int bit = __ffs(w) - 1;
        list[at++] = lo + (int)(q * 32u) + bit;
        w &= w - 1u;
      }
    }
    auto find = [&](int col) -> int {
      const unsigned c = (unsigned)(col - lo);
      return (int)pre[c >> 5] + __popc(map[c >> 5] & ((1u << (c & 31u)) - 1u));
    };
    for (int k = tid; k < nent; k += PT) lidx[k] = (uint16_t)find(cols[k]);
    // the blocks that own them (each flag is set by any number of threads)
    for (int q = tid; q < PERSIST_MAX_BLOCKS; q += PT) X.nb[q] = 0;
    __syncthreads();
    for (int h = tid; h < H; h += PT) X.nb[list[h] / A.npb] = 1;
    __syncthreads();
    if (tid < 64) {  // compact the flags in place, 64 at a time
      int at = 0;
      for (int q0 = 0; q0 < PERSIST_MAX_BLOCKS; q0 += 64) {
        const bool on = X.nb[q0 + tid] != 0;
        const unsigned long long m = __ballot(on);
        if (on) X.nb[at + __popcll(m & ((1ull << tid) - 1ull))] = q0 + tid;
        at += __popcll(m);
      }
      if (tid == 0) X.n_nb = at;
    }
    if constexpr (DIFF)
      for (int i = tid; i < nloc; i += PT)
        loc_s[i] = loc_a[i + 1] > loc_a[i] ? find((int)(n0 + i)) : -1;
  }
  __syncthreads();
  const T *gval = reinterpret_cast<const T *>(A.val) + v_beg;
  T *lval = reinterpret_cast<T *>(lds + (resident ? off_val : 0));
  if (resident) {
    // element by element: the block's values start at any element of the array
    for (int64_t q = tid; q < nval; q += PT) lval[q] = gval[q];
  }
  for (int i = tid; i < nloc; i += PT) {
    if constexpr (CSR) {
      double d = 0.0;
      for (int k = loc_a[i]; k < loc_a[i + 1]; ++k)
        if (cols[k] == n0 + i) d += (double)gval[k];
      mi[i] = (T)(d != 0.0 ? 1.0 / d : 1.0);
    } else {
      invert_block<T, ND>(A.dblk + (n0 + i) * ND2, A.pc, mi + i * PC);
    }
    for (int a = 0; a < ND; ++a) xv[i * ND + a] = pv[i * ND + a] = sv[i * ND + a] = T(0);
  }

  unsigned epoch = 0;
  int status = PERSIST_OK, iters = 0, nseg = 0;
  double relres = 0.0;
  auto finish = [&]() {
    if (blockIdx.x == 0 && tid == 0) {
      A.res->status = status;
      A.res->iters = iters;
      A.res->segments = nseg;
      A.res->relres = relres;
    }
  };
  {
    double v[1] = {tid == 0 && !fit ? 1.0 : 0.0};
    if (!exchange<1>(v, X, epoch, A)) {
      status = PERSIST_ABORTED;
      finish();
      return;
    }
    if (v[0] != 0.0) {
      status = PERSIST_NOFIT;
      finish();
      return;
    }
  }

  // ---------------------------------------------------------------- pieces
  T *ug = reinterpret_cast<T *>(A.ug), *pg = reinterpret_cast<T *>(A.pg);
  // the halo's entries of a global vector into LDS
  auto gather = [&](auto *dst, const auto *src) {
    for (int t = tid; t < H * ND; t += PT) {
      const int h = t / ND, a = t - h * ND;
      dst[t] = dev_load(src + (int64_t)list[h] * ND + a);
    }
    __syncthreads();
  };
  // own row i of K times the gathered T vector; `own` holds the block's own
  // entries (rows of no element couple to themselves only)
  auto row = [&](const T *vals, const T *own, int i, double (&acc)[ND]) {
#pragma unroll
    for (int a = 0; a < ND; ++a) acc[a] = 0.0;
    const int e0 = loc_a[i], deg = loc_a[i + 1] - e0, L = ND * deg;
    const T *vn = vals + loc_v[i];
    if (deg > 0) {
      Vec<T, ND> xs{};
      int self = -1;
      if constexpr (DIFF) {
        self = loc_s[i];
        xs = ldv<T, ND>(halo + self * ND);
      }
      for (int p = lane; p < deg; p += TL) {
        const int c = lidx[e0 + p];
        Vec<T, ND> rw[ND];
#pragma unroll
        for (int a = 0; a < ND; ++a) rw[a] = ldv<T, ND>(vn + a * L + p * ND);
        const Vec<T, ND> hv = ldv<T, ND>(halo + c * ND);
        T d[ND];
#pragma unroll
        for (int q = 0; q < ND; ++q) {
          if constexpr (DIFF) d[q] = c == self ? hv.v[q] : hv.v[q] - xs.v[q];
          else d[q] = hv.v[q];
        }
#pragma unroll
        for (int a = 0; a < ND; ++a)
#pragma unroll
          for (int q = 0; q < ND; ++q) acc[a] += (double)rw[a].v[q] * (double)d[q];
      }
    } else if (!CSR && lane < ND) {
#pragma unroll
      for (int a = 0; a < ND; ++a)
        if (a == lane) acc[a] = (double)vn[a] * (double)own[i * ND + a];
    }
#pragma unroll
    for (int a = 0; a < ND; ++a) acc[a] = lanes_sum<TL>(acc[a]);
  };
  auto pick = [&](const double (&acc)[ND]) -> double {
    double w = acc[0];
#pragma unroll
    for (int a = 1; a < ND; ++a)
      if (a == lane) w = acc[a];
    return w;
  };
  // K times the gathered vector for the own rows
  auto product = [&](const T *vals, const T *own, T *out) {
    for (int i = team; i < nloc; i += TEAMS) {
      double acc[ND];
      row(vals, own, i, acc);
      if (lane < ND) out[i * ND + lane] = (T)pick(acc);
    }
  };
  // FP64 residual b - K x of the own rows into r (as T); v = (r.r, b.b)
  auto residual = [&](const double *vals, double (&v)[2]) {
    for (int i = team; i < nloc; i += TEAMS) {
      const int e0 = loc_a[i], deg = loc_a[i + 1] - e0, L = ND * deg;
      const double *vn = vals + loc_v[i];
      double hi[ND], low[ND];
#pragma unroll
      for (int a = 0; a < ND; ++a) hi[a] = low[a] = 0.0;
      if (deg > 0) {
        for (int p = lane; p < deg; p += TL) {
          Vec<double, ND> rw[ND];
#pragma unroll
          for (int a = 0; a < ND; ++a) rw[a] = ldv<double, ND>(vn + a * L + p * ND);
          const Vec<double, ND> hv = ldv<double, ND>(halo64 + (int)lidx[e0 + p] * ND);
#pragma unroll
          for (int a = 0; a < ND; ++a)
#pragma unroll
            for (int q = 0; q < ND; ++q) {
              if (A.extended) {
                const double ph = rw[a].v[q] * hv.v[q];
                dd_add(hi[a], low[a], ph, fma(rw[a].v[q], hv.v[q], -ph));
              } else {
                hi[a] += rw[a].v[q] * hv.v[q];
              }
            }
        }
      } else if (!CSR && lane < ND) {
#pragma unroll
        for (int a = 0; a < ND; ++a)
          if (a == lane) {
            const double xo = dev_load(A.x + (n0 + i) * ND + a);
            hi[a] = vn[a] * xo;
            low[a] = A.extended ? fma(vn[a], xo, -hi[a]) : 0.0;
          }
      }
      if (A.extended) {
#pragma unroll
        for (int off = 1; off < TL; off <<= 1)
#pragma unroll
          for (int a = 0; a < ND; ++a) {
            const double oh = __shfl_xor(hi[a], off, TL), ol = __shfl_xor(low[a], off, TL);
            dd_add(hi[a], low[a], oh, ol);
          }
      } else {
#pragma unroll
        for (int a = 0; a < ND; ++a) hi[a] = lanes_sum<TL>(hi[a]);
      }
      if (lane < ND) {
        const int64_t g = (n0 + i) * ND + lane;
        const double bi = A.b[g];
        double r = bi, rl = 0.0;
        if (A.extended) {
          dd_add(r, rl, -pick(hi), -pick(low));
          r += rl;
        } else {
          r = bi - pick(hi);
        }
        rv[i * ND + lane] = (T)r;
        v[0] += r * r;
        v[1] += bi * bi;
      }
    }
  };
  // u = M r of own node i, in LDS and for the other blocks
  auto precondition = [&](int i, const T (&r)[ND], T (&z)[ND]) {
#pragma unroll
    for (int a = 0; a < ND; ++a) {
      T t = T(0);
#pragma unroll
      for (int c = 0; c < ND; ++c) t += mi[i * PC + pc_index<ND>(a, c)] * r[c];
      z[a] = t;
      uv[i * ND + a] = t;
      dev_store(ug + (n0 + i) * ND + a, t);
    }
  };

  // A wait given up on request, as after P_WAIT_TICKS: the last block's for the
  // k-th residual (point 2 k - 1), or the one before it folds its k-th correction
  // into x (point 2 k).
  auto quits = [&](int point) -> bool {
    if (!QUIT || point != A.quit || blockIdx.x != gridDim.x - 1) return false;
    if (tid == 0) dev_store(&A.res->abort, 1ull);
    return true;
  };

  // ------------------------------------------------------------- the solve
  double bnorm = 0.0, rnow = 0.0, rprev = 0.0;
  double g = 0.0, den = 0.0;  // r.u of this iteration and of the last one run
  int it = 0, stall = 0, segf = 0;
  bool first = true;
  for (;;) {
    // true residual at the current x; the target of the next segment
    gather(halo64, (const double *)A.x);
    double v2[2] = {0.0, 0.0};
    if (FP64 && resident) residual(reinterpret_cast<const double *>(lval), v2);
    else residual(A.val64 + v_beg, v2);
    publish<2>(v2, X, ++epoch, A);
    if (quits(2 * nseg + 1) || !collect<2>(v2, X, epoch, A)) {
      status = PERSIST_ABORTED;
      break;
    }
    double rr2 = v2[0];
    if (!isfinite(rr2)) {
      status = PERSIST_NONFINITE;
      break;
    }
    if (first) bnorm = sqrt(v2[1]);
    if (first && v2[1] == 0.0) {  // b = 0: x = 0 whatever the initial guess
      for (int i = tid; i < nloc * ND; i += PT) A.x[n0 * ND + i] = 0.0;
      rr2 = 0.0;
    }
    const double rn = sqrt(rr2);
    rprev = first ? rn : rnow;
    rnow = rn;
    relres = bnorm > 0.0 ? rn / bnorm : rn;
    if (rn <= A.rtol * bnorm) break;
    const bool stuck = !first && rnow > 0.9 * rprev;
    stall = stuck ? stall + 1 : 0;
    if (stall >= 8) {
      status = PERSIST_STAGNATED;
      break;
    }
    if (it >= A.max_iter) {
      status = PERSIST_MAXITER;
      break;
    }
    const double target = (FP64 ? 0.7 * A.rtol : A.final_rtol) * bnorm;
    const double seg = FP64 || A.delta * rn <= A.rtol * bnorm ? target : A.delta * rn;
    const double tol2 = seg * seg;
    // segment start: u = M r; a mixed solve that made progress keeps its
    // direction (p' = p - (r.p / r.u) u, s = K p'), others restart
    double v3[3] = {0.0, 0.0, 0.0};
    for (int i = tid; i < nloc; i += PT) {
      T r[ND], z[ND];
#pragma unroll
      for (int a = 0; a < ND; ++a) r[a] = rv[i * ND + a];
      precondition(i, r, z);
#pragma unroll
      for (int a = 0; a < ND; ++a) {
        v3[0] += (double)r[a] * (double)z[a];
        v3[1] += (double)r[a] * (double)r[a];
        v3[2] += (double)r[a] * (double)pv[i * ND + a];
      }
    }
    if (!exchange<3>(v3, X, epoch, A)) {
      status = PERSIST_ABORTED;
      break;
    }
    g = v3[0];
    double rr = v3[1];
    bool keep = !FP64 && !first && !stuck && it > segf;
    const double c = keep && g != 0.0 ? v3[2] / g : 0.0;
    if (!keep || !(c == c) || !(den == den) || den == 0.0 || g == 0.0) keep = false;
    if (keep) {
      for (int i = tid; i < nloc * ND; i += PT) {
        const T pn = pv[i] - (T)c * uv[i];
        pv[i] = pn;
        dev_store(pg + n0 * ND + i, pn);
      }
      double vb[1] = {0.0};
      if (!exchange<1>(vb, X, epoch, A)) {
        status = PERSIST_ABORTED;
        break;
      }
      gather(halo, (const T *)pg);
      if (resident) product(lval, pv, sv);
      else product(gval, pv, sv);
    } else {
      den = 0.0;
      for (int i = tid; i < nloc * ND; i += PT) pv[i] = sv[i] = T(0);
    }
    first = false;
    segf = it;
    __syncthreads();
    // iterations of the segment. The sums of (r.u, r.r) are published with the
    // new u and collected only after the next product, which needs no more
    // than the neighbours' u: one of the two grid-wide waits of an iteration
    // is hidden behind it (at the price of one product at the segment's end).
    bool stop = false, pending = false;
    for (;;) {
      if (pending && !wait_neighbours(X, epoch, A)) {
        status = PERSIST_ABORTED;
        stop = true;
        break;
      }
      if (!pending && (rr <= tol2 || !(rr == rr) || it >= A.max_iter)) break;
      gather(halo, (const T *)ug);
      if (resident) product(lval, uv, wv);
      else product(gval, uv, wv);
      if (pending) {
        double vg[2];
        if (!collect<2>(vg, X, epoch, A)) {
          status = PERSIST_ABORTED;
          stop = true;
          break;
        }
        g = vg[0];
        rr = vg[1];
        if (rr <= tol2 || !(rr == rr) || it >= A.max_iter) break;
      } else {
        __syncthreads();
      }
      const T beta = (T)(den != 0.0 ? g / den : 0.0);
      double v1[1] = {0.0};
      for (int i = tid; i < nloc * ND; i += PT) {
        const T pn = uv[i] + beta * pv[i];
        const T sn = wv[i] + beta * sv[i];
        pv[i] = pn;
        sv[i] = sn;
        v1[0] += (double)pn * (double)sn;
      }
      if (!exchange<1>(v1, X, epoch, A)) {
        status = PERSIST_ABORTED;
        stop = true;
        break;
      }
      if (!(v1[0] > 0.0)) {
        status = PERSIST_NOT_PD;
        stop = true;
        break;
      }
      const T alpha = (T)(g / v1[0]);
      den = g;
      ++it;
      double vg[2] = {0.0, 0.0};
      for (int i = tid; i < nloc; i += PT) {
        T r[ND], z[ND];
#pragma unroll
        for (int a = 0; a < ND; ++a) {
          const int e = i * ND + a;
          xv[e] += alpha * pv[e];
          r[a] = rv[e] - alpha * sv[e];
          rv[e] = r[a];
        }
        precondition(i, r, z);
#pragma unroll
        for (int a = 0; a < ND; ++a) {
          vg[0] += (double)r[a] * (double)z[a];
          vg[1] += (double)r[a] * (double)r[a];
        }
      }
      publish<2>(vg, X, ++epoch, A);
      pending = true;
    }
    iters += it - segf;
    if (stop) break;
    if (!(rr <= tol2 || !(rr == rr))) {
      status = PERSIST_MAXITER;
      break;
    }
    if (quits(2 * nseg + 2)) {
      status = PERSIST_ABORTED;
      break;
    }
    // fold the correction into x
    ++nseg;
    for (int i = tid; i < nloc * ND; i += PT) {
      dev_store(A.x + n0 * ND + i, dev_load(A.x + n0 * ND + i) + (double)xv[i]);
      xv[i] = T(0);
    }
    double vb[1] = {0.0};
    if (!exchange<1>(vb, X, epoch, A)) {
      status = PERSIST_ABORTED;
      break;
    }
  }
  finish();
}

__global__ void k_clear_slots(unsigned long long *slots, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) slots[i] = 0ull;
}

template <typename T, int ND, int TL, bool CSR, bool QUIT = false>
int launch(hipStream_t s, unsigned grid, const PersistArgs &A) {
  const void *fn = reinterpret_cast<const void *>(&k_pcg_persist<T, ND, TL, CSR, QUIT>);
  TFM_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)P_LDS));
  hipLaunchKernelGGL((k_pcg_persist<T, ND, TL, CSR, QUIT>), dim3(grid), dim3(PT), P_LDS, s, A);
  TFM_CHECK_LAUNCH();
  return TFM_OK;
}

template <typename T, int ND>
int launch_team(hipStream_t s, unsigned grid, double deg, const PersistArgs &A) {
  if (A.quit > 0) return launch<T, ND, 8, false, true>(s, grid, A);
  if (deg > 32.0) return launch<T, ND, 32, false>(s, grid, A);
  if (deg > 16.0) return launch<T, ND, 16, false>(s, grid, A);
  return launch<T, ND, 8, false>(s, grid, A);
}

// One persistent solve per device at a time in this process: two of them on
// different streams could each hold part of the CUs and wait for the rest. A
// solve waits its turn rather than taking the general path, whose sums have
// another order: its results then do not depend on what other threads do.
std::mutex g_turn[64];

// Until when the calling thread's solves on a device take the general path,
// because one of them has given up a wait.
thread_local std::chrono::steady_clock::time_point g_rest[64];

}  // namespace

int persist_solve(hipStream_t s, const PersistJob &J, PersistResult *res, bool *ran) {
  *ran = false;
  if (env_int("TFM_PCG_PERSIST", 1) == 0) return TFM_OK;
  const bool csr = J.m == nullptr;
  const int nd = csr ? 1 : J.m->ndof;
  const int64_t n_nod = csr ? J.n : J.m->n_nod;
  if (n_nod < 1 || J.val64 == nullptr || nd < 1 || nd > 3) return TFM_OK;
  const int dev = J.device;
  int cus = 0, lds = 0;
  TFM_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  TFM_CHECK_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  if (dev < 0 || dev >= 64 || lds < 160 * 1024) return TFM_OK;
  if (std::chrono::steady_clock::now() < g_rest[dev]) return TFM_OK;
  const int max_blocks = std::min(cus, PERSIST_MAX_BLOCKS);
  const unsigned size = J.fp64 ? 8u : 4u;
  // the entry count of a CSR matrix is on the device: 7 per row, as of a 7-point
  // matrix, stands in for it. Denser rows run into the kernel's own LDS check
  // before they reach the limit below (2 bytes per entry are kept there). Against
  // the general path, solves of matrices with 5 to 363 entries per row (stencils,
  // random, permuted) took 0.40 to 0.82 of the time, those that do not fit 1.01
  // to 1.02.
  const double nnz = csr ? 7.0 * n_nod : (double)J.m->nnz;
  const double deg = nnz / ((double)n_nod * nd * nd);
  // values per CU: up to about 120 KB they stay in LDS, beyond they stream
  // from L2 and the Infinity Cache. Against the general path, per iteration:
  // FP32 Hexa1 14^3 6.9 us (15.6), 30^3 9.3 (17.0), 42^3 23.8 (25.9), 48^3
  // (420 KB) 31.3 (32.0), Hexa2 28^3 (780 KB) 46.1 (43.9); FP64, whose general
  // path takes four launches, Hexa1 24^3 7.6 (20.9), 34^3 19.8 (30.9), 44^3
  // (695 KB) 36.0 (47.7); FP64 Quad1 400 x 200 8.2 (22.9); Tetra1 heat 70^3
  // 13.8 (26.2)
  const int kb = env_int("TFM_PCG_PERSIST_KB", J.fp64 ? 720 : 420);
  if (nnz * size > (double)max_blocks * kb * 1024.0) return TFM_OK;
  // small systems: as many nodes per block as give every thread a neighbour
  // block. Fewer blocks make the exchanges shorter, more nodes the product
  // longer; swept 16 to 128 nodes: 6.4 us per iteration at 64 (32: 6.4, 128:
  // 8.0) on Hexa1 14^3, 6.5 at 16 (64: 8.9) on Hexa2 6^3, 5.1 at 128 (32: 6.2)
  // on a 121 x 59 Quad1 plate, 6.2 at 96 (16: 7.6) on Tetra1 12^3
  const int per = std::max(16, (int)(PT / std::max(deg, 1.0)));
  int grid = (int)std::min<int64_t>(max_blocks, (n_nod + per - 1) / per);
  const int npb = (int)((n_nod + grid - 1) / grid);
  grid = (int)((n_nod + npb - 1) / npb);
  const unsigned fixed = nd == 1   ? (J.fp64 ? fixed_lds<double, 1>(npb) : fixed_lds<float, 1>(npb))
                         : nd == 2 ? (J.fp64 ? fixed_lds<double, 2>(npb) : fixed_lds<float, 2>(npb))
                                   : (J.fp64 ? fixed_lds<double, 3>(npb) : fixed_lds<float, 3>(npb));
  if (fixed > P_LDS / 2) return TFM_OK;
  auto *slots = reinterpret_cast<unsigned long long *>(J.scratch);
  PersistArgs A{};
  A.n_nod = n_nod;
  A.npb = npb;
  if (!csr) {
    A.adj_ptr = J.m->adj_ptr;
    A.adj = J.m->adj;
    A.val_ptr = J.m->val_ptr;
  }
  A.rowptr = J.rowptr;
  A.col = J.col;
  A.val = J.val;
  A.val64 = J.val64;
  A.dblk = J.dblk;
  A.pc = J.pc;
  A.b = J.b;
  A.x = J.x;
  A.ug = J.u;
  A.pg = J.p;
  A.slots = slots;
  A.res = reinterpret_cast<PersistResult *>(slots + PERSIST_SLOTS);
  A.rtol = J.rtol;
  A.delta = J.delta;
  A.final_rtol = J.final_rtol;
  A.max_iter = J.max_iter;
  A.extended = J.extended;
  A.quit = env_int("TFM_PCG_PERSIST_QUIT", 0);
  constexpr int words = PERSIST_SCRATCH_BYTES / sizeof(unsigned long long);
  hipLaunchKernelGGL(k_clear_slots, dim3((words + 255) / 256), dim3(256), 0, s, slots, words);
  TFM_CHECK_LAUNCH();
  // what the stream still holds is awaited before the turn, not within it: a
  // turn then lasts as long as its kernel, which waits for nobody else's work
  TFM_CHECK_HIP(hipStreamSynchronize(s));
  std::lock_guard<std::mutex> turn(g_turn[dev]);
  int rc = TFM_OK;
  if (csr && A.quit > 0) rc = launch<double, 1, 8, true, true>(s, grid, A);
  else if (csr) rc = launch<double, 1, 8, true>(s, grid, A);
  else if (J.fp64)
    rc = nd == 1   ? launch_team<double, 1>(s, grid, deg, A)
         : nd == 2 ? launch_team<double, 2>(s, grid, deg, A)
                   : launch_team<double, 3>(s, grid, deg, A);
  else
    rc = nd == 1   ? launch_team<float, 1>(s, grid, deg, A)
         : nd == 2 ? launch_team<float, 2>(s, grid, deg, A)
                   : launch_team<float, 3>(s, grid, deg, A);
  if (rc != TFM_OK) return rc;
  TFM_CHECK_HIP(hipMemcpyAsync(J.h_res, A.res, sizeof(PersistResult), hipMemcpyDeviceToHost, s));
  TFM_CHECK_HIP(hipStreamSynchronize(s));
  *res = *J.h_res;
  if (res->abort) {
    res->status = PERSIST_ABORTED;
    g_rest[dev] = std::chrono::steady_clock::now() +
                  std::chrono::milliseconds(env_int("TFM_PCG_PERSIST_REST_MS", 4000));
  }
  *ran = res->status != PERSIST_NOFIT && res->status != PERSIST_ABORTED;
  return TFM_OK;
}

}  // namespace tfm
