// Pieces shared by the Krylov sources: vector loads, packed nodal
// preconditioner blocks, double-double sums, cross-lane sums, and the
// interface of the persistent small-system solver.
#pragma once

#include "tfm_common.h"

namespace tfm {

// K contiguous values loaded as one unit (one global_load_dwordxN per lane
// where the width allows; the compiler otherwise splits rows unevenly).
template <typename T, int K> struct Vec {
  T v[K];
};

template <typename T, int K>
__device__ __forceinline__ Vec<T, K> ldv(const T *p) {
  Vec<T, K> r;
  __builtin_memcpy(&r, p, sizeof(r));
  return r;
}

template <typename T, int K>
__device__ __forceinline__ void stv(T *p, const Vec<T, K> &v) {
  __builtin_memcpy(p, &v, sizeof(v));
}

// Packed upper triangle of a nodal preconditioner block, row by row.
template <int ND> constexpr int pc_size() { return ND * (ND + 1) / 2; }

template <int ND>
__host__ __device__ constexpr int pc_index(int a, int b) {
  return a <= b ? a * ND - a * (a - 1) / 2 + (b - a) : b * ND - b * (b - 1) / 2 + (a - b);
}

// Inverse of a nodal diagonal block (block Jacobi) or of its diagonal
// (Jacobi), packed (pc_index); a zero pivot keeps the identity.
template <typename T, int ND>
__device__ __forceinline__ void invert_block(const double *dblk, int pc, T *out) {
  double A[ND][ND], R[ND][ND];
  for (int a = 0; a < ND; ++a)
    for (int b = 0; b < ND; ++b) {
      A[a][b] = dblk[a * ND + b];
      R[a][b] = a == b ? 1.0 : 0.0;
    }
  if (pc == TFM_PC_JACOBI || ND == 1) {
    for (int a = 0; a < ND; ++a)
      for (int b = 0; b < ND; ++b) R[a][b] = (a == b && A[a][a] != 0.0) ? 1.0 / A[a][a] : (a == b);
  } else {
    // Gauss-Jordan with partial pivoting on the small SPD block
    for (int c = 0; c < ND; ++c) {
      int piv = c;
      for (int r = c + 1; r < ND; ++r)
        if (fabs(A[r][c]) > fabs(A[piv][c])) piv = r;
      if (A[piv][c] == 0.0) continue;
      if (piv != c)
        for (int k = 0; k < ND; ++k) {
          double t = A[c][k]; A[c][k] = A[piv][k]; A[piv][k] = t;
          t = R[c][k]; R[c][k] = R[piv][k]; R[piv][k] = t;
        }
      const double inv = 1.0 / A[c][c];
      for (int k = 0; k < ND; ++k) { A[c][k] *= inv; R[c][k] *= inv; }
      for (int r = 0; r < ND; ++r)
        if (r != c) {
          const double f = A[r][c];
          for (int k = 0; k < ND; ++k) { A[r][k] -= f * A[c][k]; R[r][k] -= f * R[c][k]; }
        }
    }
  }
  // the two triangles of the inverse agree up to rounding; their mean keeps
  // the preconditioner exactly symmetric
  for (int a = 0; a < ND; ++a)
    for (int b = a; b < ND; ++b) out[pc_index<ND>(a, b)] = (T)(0.5 * (R[a][b] + R[b][a]));
}

// (hi, lo) += (a, b2) in double-double
__device__ __forceinline__ void dd_add(double &hi, double &lo, double a, double b2) {
  const double s = hi + a;
  const double v = s - hi;
  const double e = (hi - (s - v)) + (a - v) + lo + b2;
  hi = s + e;
  lo = e - (hi - s);
}

// v of the lane that differs in bit log2(OFF) of the lane number. Within 16
// lanes by DPP, across them by the row swaps of gfx950: a few cycles instead
// of an LDS permutation's hundred. (The DPP mirrors reach lane^7 and lane^15;
// in a butterfly those lanes hold the same partial sum as lane^4 and lane^8.)
template <int OFF> __device__ __forceinline__ double butterfly_partner_sum(double v) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16 || OFF == 32, "offset");
  const int lo = __double2loint(v), hi = __double2hiint(v);
  if constexpr (OFF <= 8) {
    constexpr int CTRL = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x140;
    const int l2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true);
    const int h2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(h2, l2);
  } else {
    // swap(x, x) leaves the even halves in one result and the odd in the other
    if constexpr (OFF == 16) {
      const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
      return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    } else {
      const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
      return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    }
  }
}

// Sum over aligned groups of N lanes (a power of two), in every lane of the
// group, in a fixed order. Every lane of the group must be active.
template <int N> __device__ __forceinline__ double lanes_sum(double v) {
  if constexpr (N >= 2) v = butterfly_partner_sum<1>(v);
  if constexpr (N >= 4) v = butterfly_partner_sum<2>(v);
  if constexpr (N >= 8) v = butterfly_partner_sum<4>(v);
  if constexpr (N >= 16) v = butterfly_partner_sum<8>(v);
  if constexpr (N >= 32) v = butterfly_partner_sum<16>(v);
  if constexpr (N >= 64) v = butterfly_partner_sum<32>(v);
  return v;
}

// ------------------------------------------------ persistent small solver
enum {
  PERSIST_OK = 0,
  PERSIST_MAXITER = 1,
  PERSIST_NOT_PD = 2,
  PERSIST_STAGNATED = 3,
  PERSIST_NONFINITE = 4,
  PERSIST_NOFIT = 5,  // the block-local index sets do not fit: nothing was done
  PERSIST_ABORTED = 6 // a block did not arrive in time: x holds a valid guess
};

// abort is set by any block that gives up a wait, the others by block 0.
struct PersistResult {
  unsigned long long abort;
  int status, iters, segments, pad;
  double relres;
};

constexpr int PERSIST_MAX_BLOCKS = 256;
constexpr int PERSIST_COPIES = 8;
// exchange slots: [parity][copy][value][2 words][block]
constexpr int PERSIST_SLOTS = 2 * PERSIST_COPIES * 3 * 2 * PERSIST_MAX_BLOCKS;
// device scratch of one solve: the slots and the result
constexpr size_t PERSIST_SCRATCH_BYTES =
    sizeof(unsigned long long) * PERSIST_SLOTS + sizeof(PersistResult);

struct PersistJob {
  // rows: the node blocks of a mesh, or a general CSR matrix (m == nullptr)
  const tfm_mesh_t *m = nullptr;
  int64_t n = 0;   // rows of the CSR matrix
  int device = 0;  // of the stream and the buffers
  const int64_t *rowptr = nullptr;
  const int32_t *col = nullptr;
  bool fp64 = true;
  const void *val = nullptr;      // FP32 (difference form) or FP64 values
  const double *val64 = nullptr;  // FP64 values (refinement residuals)
  const double *dblk = nullptr;   // nodal diagonal blocks (meshes)
  int pc = TFM_PC_BLOCK_JACOBI;
  const double *b = nullptr;
  double *x = nullptr;
  void *u = nullptr, *p = nullptr;  // exchange vectors of n values
  void *scratch = nullptr;          // PERSIST_SCRATCH_BYTES on the device
  PersistResult *h_res = nullptr;   // pinned
  double rtol = 0.0, delta = 0.5, final_rtol = 0.0;
  int max_iter = 0;
  bool extended = false;
};

// Runs the solve in one kernel when the system suits it; *ran tells whether
// `res` holds an outcome (otherwise nothing happened, or x is a new guess,
// and the caller takes the general path).
int persist_solve(hipStream_t s, const PersistJob &job, PersistResult *res, bool *ran);

}  // namespace tfm
