// Element integration, deterministic assembly, internal forces and parameter
// sensitivities for gfx950. All floating-point work is FP64; the FP32 matrix
// copy for the mixed-precision solver is rounded from the FP64 sums.
#include "tfm_common.h"

#include <type_traits>

namespace tfm {

// Shape-function tables, evaluated at compile time (see tfm_common.h).
__constant__ ShapeTable<Quad1> c_quad1 = make_table<Quad1>();
__constant__ ShapeTable<Tetra1> c_tetra1 = make_table<Tetra1>();
__constant__ ShapeTable<Hexa1> c_hexa1 = make_table<Hexa1>();
__constant__ ShapeTable<Hexa2> c_hexa2 = make_table<Hexa2>();

template <> __device__ const ShapeTable<Quad1> &shape_table<Quad1>() { return c_quad1; }
template <> __device__ const ShapeTable<Tetra1> &shape_table<Tetra1>() { return c_tetra1; }
template <> __device__ const ShapeTable<Hexa1> &shape_table<Hexa1>() { return c_hexa1; }
template <> __device__ const ShapeTable<Hexa2> &shape_table<Hexa2>() { return c_hexa2; }

constexpr int odd(int n) { return n | 1; }  // row strides that spread over the LDS banks

// Material parameter i of element e in the layout of `kind`.
template <int MAT, int DIM>
__device__ __forceinline__ double mat_param(const tfm_material_t &mat, int64_t e, int i) {
  if constexpr (MAT == TFM_MAT_ISO) return i == 0 ? mat.p0[e] : mat.p1[e];
  else return mat.p0[e * mat_nparam(MAT, DIM) + i];
}

__device__ __forceinline__ double mat_scale(const tfm_material_t &mat, int64_t e) {
  return mat.scale ? mat.scale[e] : 1.0;
}

// Jacobian of element geometry X[NPE][DIM] at Gauss point g (base.py:307-313).
template <class E>
__device__ __forceinline__ double geometry(const double (*X)[E::DIM], int g,
                                           double (&Ji)[E::DIM][E::DIM]) {
  const auto &T = shape_table<E>();
  double J[E::DIM][E::DIM];
  for (int i = 0; i < E::DIM; ++i)
    for (int k = 0; k < E::DIM; ++k) {
      double acc = 0.0;
      for (int N = 0; N < E::NPE; ++N) acc += T.dN[g][i][N] * X[N][k];
      J[i][k] = acc;
    }
  return inv_jac<E::DIM>(J, Ji);
}

// B[:, N] = J^{-1} dN/dxi[:, N]
template <class E>
__device__ __forceinline__ void bcol(const double (&Ji)[E::DIM][E::DIM], int g, int N,
                                     double *b) {
  const auto &T = shape_table<E>();
  for (int i = 0; i < E::DIM; ++i) {
    double acc = 0.0;
    for (int k = 0; k < E::DIM; ++k) acc += Ji[i][k] * T.dN[g][k][N];
    b[i] = acc;
  }
}

// ========================================================= pattern expansion
// A wave per node, four to a block. Bound by writing rows and cols: 573 MB of
// 53x47x58 Hexa1 in 160 us (284 with a block of 256 per node, every thread of
// which searched the diagonal).
template <int ND>
__global__ void __launch_bounds__(256) k_pattern_rows(tfm_mesh_t m, int64_t *rows, int64_t *cols,
                                                      int64_t *rowptr, int32_t *diag_map) {
  const int64_t n = xcd_block() * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (n >= m.n_nod) return;
  const int a0 = m.adj_ptr[n];
  const int deg = m.adj_ptr[n + 1] - a0;
  const int64_t v0 = m.val_ptr[n];
  const int L = ND * deg;
  if (lane < ND && rowptr) {
    rowptr[n * ND + lane] = v0 + (deg > 0 ? lane * L : lane);
    if (n == m.n_nod - 1 && lane == ND - 1) rowptr[m.n_nod * ND] = m.nnz;
  }
  if (diag_map) {
    if (deg == 0) {
      if (lane < ND) diag_map[n * ND + lane] = (int32_t)(v0 + lane);
    } else {
      for (int p = lane; p < deg; p += 64)
        if (m.adj[a0 + p] == n)
          for (int a = 0; a < ND; ++a)
            diag_map[n * ND + a] = (int32_t)(v0 + a * L + p * ND + a);
    }
  }
  if (!rows && !cols) return;
  const int total = deg > 0 ? ND * L : ND;
  for (int q = lane; q < total; q += 64) {
    int a = q;
    int64_t col = n * ND + q;
    if (deg > 0) {
      int rem = q;  // q = a L + rem
      a = 0;
      for (int k = 1; k < ND; ++k)
        if (rem >= L) {
          rem -= L;
          ++a;
        }
      const int p = rem / ND;
      col = (int64_t)m.adj[a0 + p] * ND + (rem - p * ND);
    }
    if (rows) rows[v0 + q] = n * ND + a;
    if (cols) cols[v0 + q] = col;
  }
}

// k_map[e, i*nd+a, j*nd+b] = slot of (row n_i*nd+a, col n_j*nd+b) (base.py:94-104).
// The row starts of the nodes of EB elements and their slots in LDS; the map
// leaves in consecutive words, its bound: 333 MB of 53x47x58 Hexa1 in 122 us (242
// with all of it looked up per entry; 223 with divisions by run-time widths).
template <int NPE, int ND>
__global__ void __launch_bounds__(256) k_pattern_kmap(tfm_mesh_t m, int32_t *k_map) {
  constexpr int EB = NPE <= 8 ? 4 : 1, W = NPE * ND, W2 = W * W, NP2 = NPE * NPE;
  __shared__ int start[EB * NPE], len[EB * NPE], pos[EB * NP2];
  const int64_t e0 = xcd_block() * EB;
  const int ne = (int)(m.n_elem - e0 < EB ? m.n_elem - e0 : EB);
  for (int t = threadIdx.x; t < ne * NPE; t += 256) {
    const int64_t n = m.elements[e0 * NPE + t];
    start[t] = (int)m.val_ptr[n];
    len[t] = ND * (m.adj_ptr[n + 1] - m.adj_ptr[n]);
  }
  for (int t = threadIdx.x; t < ne * NP2; t += 256) pos[t] = m.epos[e0 * NP2 + t];
  __syncthreads();
  for (int t = threadIdx.x; t < ne * W2; t += 256) {
    const int k = t / W2, q = t - k * W2, r = q / W, c = q - r * W;
    const int i = r / ND, a = r - i * ND, j = c / ND, b = c - j * ND;
    k_map[e0 * W2 + t] = start[k * NPE + i] + a * len[k * NPE + i] + pos[k * NP2 + i * NPE + j] * ND + b;
  }
}

// The same for any number of element nodes: a block per element.
__global__ void __launch_bounds__(256) k_pattern_kmap_any(tfm_mesh_t m, int32_t *k_map) {
  const int64_t e = xcd_block();
  const int npe = m.npe, nd = m.ndof, W = npe * nd;
  for (int t = threadIdx.x; t < W * W; t += 256) {
    const int r = t / W, c = t - r * W;
    const int i = r / nd, a = r - i * nd, j = c / nd, b = c - j * nd;
    const int64_t n = m.elements[e * npe + i];
    const int len = nd * (m.adj_ptr[n + 1] - m.adj_ptr[n]);
    const int pos = m.epos[(e * npe + i) * npe + j];
    k_map[e * W * W + t] = (int32_t)(m.val_ptr[n] + a * len + pos * nd + b);
  }
}

template <int ND>
static int pattern_expand(hipStream_t s, const tfm_mesh_t &m, int64_t *rows, int64_t *cols,
                          int64_t *rowptr, int32_t *k_map, int32_t *diag_map) {
  if (rows || cols || rowptr || diag_map) {
    hipLaunchKernelGGL(k_pattern_rows<ND>, dim3((unsigned)((m.n_nod + 3) / 4)), dim3(256), 0, s, m,
                       rows, cols, rowptr, diag_map);
    TFM_CHECK_LAUNCH();
  }
  if (k_map && m.n_elem > 0) {
    const unsigned by4 = (unsigned)((m.n_elem + 3) / 4), by1 = (unsigned)m.n_elem;
    switch (m.npe) {
      case 4: hipLaunchKernelGGL((k_pattern_kmap<4, ND>), dim3(by4), dim3(256), 0, s, m, k_map); break;
      case 8: hipLaunchKernelGGL((k_pattern_kmap<8, ND>), dim3(by4), dim3(256), 0, s, m, k_map); break;
      case 20: hipLaunchKernelGGL((k_pattern_kmap<20, ND>), dim3(by1), dim3(256), 0, s, m, k_map); break;
      default: hipLaunchKernelGGL(k_pattern_kmap_any, dim3(by1), dim3(256), 0, s, m, k_map);
    }
    TFM_CHECK_LAUNCH();
  }
  return TFM_OK;
}

int launch_pattern_expand(hipStream_t s, const tfm_mesh_t &m, int64_t *rows, int64_t *cols,
                          int64_t *rowptr, int32_t *k_map, int32_t *diag_map) {
  switch (m.ndof) {
    case 1: return pattern_expand<1>(s, m, rows, cols, rowptr, k_map, diag_map);
    case 2: return pattern_expand<2>(s, m, rows, cols, rowptr, k_map, diag_map);
    case 3: return pattern_expand<3>(s, m, rows, cols, rowptr, k_map, diag_map);
    default: TFM_REQUIRE(false, "ndof must be 1, 2 or 3");
  }
}

// ========================================================= element matrices
// Elements per block and threads: a thread for every (I, J) node pair, at
// least 256 threads where several elements fit (448 = 7 waves for the 400
// pairs of a Hexa2).
template <class E> constexpr int matrix_elems() {
  return E::NPE >= 16 ? 1 : 256 / (E::NPE * E::NPE);
}
template <class E> constexpr int matrix_threads() {
  return (matrix_elems<E>() * E::NPE * E::NPE + 63) / 64 * 64;
}

// k_e = sum_g w detJ s B^T C B. A thread per (element, point) forms J^{-1}, a
// thread per (element, point, node) the columns of B and w detJ s B, and a
// thread per (element, I, J) the geometric moments
//   M_IJ[a][c] = sum_g w detJ s (dN_I/dx)_a (dN_J/dx)_c,
// on which the material acts once: the tangent is the same at every point.
// The blocks gather into whole matrices in LDS and leave in consecutive words.
// Bound by writing k: Hexa1 43x37x40 84 us (293 MB, 3.5 TB/s), 166 us with the
// columns of B and the material formed per pair and point and k written in
// pieces of 24 bytes; anisotropic Hexa2 13x15x11 35 us (128).
template <class E, int NDOF, int MAT>
__global__ void __launch_bounds__(matrix_threads<E>())
    k_element_matrices(tfm_mesh_t m, tfm_material_t mat, double *kout, int32_t *bad) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM, NP = mat_nparam(MAT, D);
  constexpr int W = NPE * NDOF, W2 = W * W, EB = matrix_elems<E>(), TB = matrix_threads<E>();
  constexpr int R = NPE * D, ROWS = EB * NGP;
  constexpr int NBUF = 2 * ROWS * R > EB * W2 ? 2 * ROWS * R : EB * W2;
  __shared__ double buf[NBUF];  // B and w detJ s B, then the matrices
  __shared__ double Xs[EB][odd(R)], tbl[NGP][odd(R)];
  __shared__ double Gm[ROWS][odd(D * D + 1)];
  __shared__ double MP[EB][NP];
  double *Bs = buf, *Bw = buf + ROWS * R;
  const int tid = threadIdx.x;
  const int64_t e0 = xcd_block() * EB;
  const int ne = (int)(m.n_elem - e0 < EB ? m.n_elem - e0 : EB);
  const auto &T = shape_table<E>();
  for (int q = tid; q < NGP * R; q += TB) tbl[q / R][q % R] = (&T.dN[0][0][0])[q];
  for (int t = tid; t < ne * NPE; t += TB) {
    const int64_t n = m.elements[e0 * NPE + t];
    for (int d = 0; d < D; ++d) Xs[t / NPE][(t % NPE) * D + d] = m.nodes[n * D + d];
  }
  for (int t = tid; t < ne * NP; t += TB) MP[t / NP][t % NP] = mat_param<MAT, D>(mat, e0 + t / NP, t % NP);
  __syncthreads();
  for (int t = tid; t < ne * NGP; t += TB) {
    const int el = t / NGP, g = t % NGP;
    double J[D][D], Ji[D][D];
    for (int i = 0; i < D; ++i)
      for (int k = 0; k < D; ++k) J[i][k] = 0.0;
#pragma unroll 4
    for (int N = 0; N < NPE; ++N)
      for (int i = 0; i < D; ++i)
        for (int k = 0; k < D; ++k) J[i][k] += tbl[g][i * NPE + N] * Xs[el][N * D + k];
    const double det = inv_jac<D>(J, Ji);
    if (!(det > 0.0)) *bad = 1;
    for (int i = 0; i < D; ++i)
      for (int k = 0; k < D; ++k) Gm[t][i * D + k] = Ji[i][k];
    Gm[t][D * D] = T.w[g] * det * mat_scale(mat, e0 + el);
  }
  __syncthreads();
  for (int t = tid; t < ne * NGP * NPE; t += TB) {
    const int row = t / NPE, N = t - row * NPE, g = row % NGP;
    const double wd = Gm[row][D * D];
    for (int i = 0; i < D; ++i) {
      double v = 0.0;
      for (int k = 0; k < D; ++k) v += Gm[row][i * D + k] * tbl[g][k * NPE + N];
      Bs[row * R + N * D + i] = v;
      Bw[row * R + N * D + i] = v * wd;
    }
  }
  __syncthreads();
  const int el = tid / (NPE * NPE), I = tid / NPE % NPE, Jn = tid % NPE;
  const bool act = el < ne;
  double blk[NDOF * NDOF];
  if (act) {
    double M[D * D];
    for (int q = 0; q < D * D; ++q) M[q] = 0.0;
#pragma unroll 4
    for (int g = 0; g < NGP; ++g) {
      const double *bi = Bs + (el * NGP + g) * R + I * D, *bj = Bw + (el * NGP + g) * R + Jn * D;
      for (int a = 0; a < D; ++a)
        for (int c = 0; c < D; ++c) M[a * D + c] += bi[a] * bj[c];
    }
    const double *mp = MP[el];
    if constexpr (MAT == TFM_MAT_ISO) {
      double tr = 0.0;
      for (int a = 0; a < D; ++a) tr += M[a * D + a];
      for (int a = 0; a < D; ++a)
        for (int c = 0; c < D; ++c)
          blk[a * NDOF + c] = mp[0] * M[a * D + c] + mp[1] * M[c * D + a] + (a == c ? mp[1] * tr : 0.0);
    } else if constexpr (MAT == TFM_MAT_GENERAL) {
      for (int i = 0; i < D; ++i)
        for (int k = 0; k < D; ++k) {
          double v = 0.0;
          for (int a = 0; a < D; ++a)
            for (int c = 0; c < D; ++c) v += mp[((i * D + a) * D + k) * D + c] * M[a * D + c];
          blk[i * NDOF + k] = v;
        }
    } else if constexpr (MAT == TFM_MAT_HEAT_ISO) {
      double tr = 0.0;
      for (int a = 0; a < D; ++a) tr += M[a * D + a];
      blk[0] = mp[0] * tr;
    } else {
      double v = 0.0;
      for (int q = 0; q < D * D; ++q) v += mp[q] * M[q];
      blk[0] = v;
    }
  }
  __syncthreads();
  if (act)
    for (int a = 0; a < NDOF; ++a)
      for (int b = 0; b < NDOF; ++b)
        buf[el * W2 + (I * NDOF + a) * W + Jn * NDOF + b] = blk[a * NDOF + b];
  __syncthreads();
  double *o = kout + e0 * W2;
  for (int t = tid; t < ne * W2; t += TB) o[t] = buf[t];
}

// Element matrices from a tangent given per Gauss point, C[g][e][i][J][k][L]
// (a finite-strain material's dP/dF): k = sum_g w detJ B^T C_g B times the
// optional volume scale. The element's eight (or fewer) tangents are staged
// in LDS next to its J^{-1} and w*detJ.
template <class E>
__global__ void __launch_bounds__(64) k_element_matrices_gp(tfm_mesh_t m, const double *cgp,
                                                            const double *scale, double *kout,
                                                            int32_t *bad) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM, NC = D * D * D * D;
  constexpr int W = NPE * D, ND2 = D * D;
  __shared__ double X[NPE][D];
  __shared__ double Gm[NGP][D * D + 1];
  __shared__ double Cg[NGP][NC];
  const int64_t e = xcd_block();
  const int tid = threadIdx.x;
  for (int t = tid; t < NPE * D; t += 64) {
    const int j = t / D, d = t - j * D;
    X[j][d] = m.nodes[(int64_t)m.elements[e * NPE + j] * D + d];
  }
  for (int t = tid; t < NGP * NC; t += 64) {
    const int g = t / NC, c = t - g * NC;
    Cg[g][c] = cgp[((int64_t)g * m.n_elem + e) * NC + c];
  }
  __syncthreads();
  const double sc = scale ? scale[e] : 1.0;
  for (int g = tid; g < NGP; g += 64) {
    double Ji[D][D];
    const double det = geometry<E>(X, g, Ji);
    if (!(det > 0.0)) *bad = 1;
    for (int i = 0; i < D; ++i)
      for (int k = 0; k < D; ++k) Gm[g][i * D + k] = Ji[i][k];
    Gm[g][D * D] = shape_table<E>().w[g] * det * sc;
  }
  __syncthreads();
  for (int t = tid; t < NPE * NPE; t += 64) {
    const int I = t / NPE, J = t - I * NPE;
    double blk[ND2];
    for (int q = 0; q < ND2; ++q) blk[q] = 0.0;
    for (int g = 0; g < NGP; ++g) {
      double Ji[D][D];
      for (int i = 0; i < D; ++i)
        for (int k = 0; k < D; ++k) Ji[i][k] = Gm[g][i * D + k];
      double bI[D], bJ[D], c[ND2];
      bcol<E>(Ji, g, I, bI);
      bcol<E>(Ji, g, J, bJ);
      coupling_block<D, D, TFM_MAT_GENERAL>(bI, bJ, Cg[g], Gm[g][D * D], c);
      for (int q = 0; q < ND2; ++q) blk[q] += c[q];
    }
    for (int a = 0; a < D; ++a)
      for (int b = 0; b < D; ++b)
        kout[e * W * W + (int64_t)(I * D + a) * W + J * D + b] = blk[a * D + b];
  }
}

// ================================================================ assembly
// One 64-lane block per node n assembles the node's ndof CSR rows: the
// incident elements are visited in ascending order in chunks of KCH; each
// (element, column node) pair forms its ndof x ndof block from the staged
// geometry, and the row entries add the blocks in element order. Every CSR
// value is written exactly once, so no float atomics are needed and the
// result is bitwise reproducible. The Dirichlet epilogue of
// FEM.assemble_matrix (base.py:413-419) is applied on the way out.
template <class E> constexpr int assemble_chunk() { return E::NPE >= 16 ? 4 : 64 / E::NPE; }

template <class E, int NDOF, int MAT>
__global__ void __launch_bounds__(64) k_assemble_rows(tfm_mesh_t m, tfm_material_t mat,
                                                      const uint8_t *con, double *v64,
                                                      float *v32, double *dblk, int32_t *bad,
                                                      int diff32) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM, NP = mat_nparam(MAT, D);
  constexpr int ND2 = NDOF * NDOF, KCH = assemble_chunk<E>();
  __shared__ double X[KCH][NPE][D];
  __shared__ double Gm[KCH][NGP][D * D + 1];
  __shared__ double MP[KCH][NP];
  __shared__ double S[KCH * NPE][ND2];
  __shared__ int Eid[KCH], Iloc[KCH];
  __shared__ int pself;
  extern __shared__ double dyn[];
  double *acc = dyn;                                              // [ND2 * maxdeg]
  signed char *slot = reinterpret_cast<signed char *>(acc + ND2 * m.max_deg);  // [KCH * maxdeg]

  const int64_t n = xcd_block();
  const int tid = threadIdx.x;
  const int a0 = m.adj_ptr[n];
  const int deg = m.adj_ptr[n + 1] - a0;
  const int64_t vb = m.val_ptr[n];
  if (deg == 0) {  // orphan node: only its diagonal is stored (base.py:89-90)
    if (tid < NDOF) {
      const int64_t r = n * NDOF + tid;
      const double v = con[r] ? 1.0 : 0.0;
      if (v64) v64[vb + tid] = v;
      if (v32) v32[vb + tid] = (float)v;
    }
    for (int t = tid; t < ND2; t += 64) {
      const int a = t / NDOF, b = t - a * NDOF;
      dblk[n * ND2 + t] = (a == b && con[n * NDOF + a]) ? 1.0 : 0.0;
    }
    return;
  }
  const int inc0 = m.ne_ptr[n];
  const int ninc = m.ne_ptr[n + 1] - inc0;
  const int L = NDOF * deg;
  for (int q = tid; q < ND2 * deg; q += 64) acc[q] = 0.0;

  for (int c0 = 0; c0 < ninc; c0 += KCH) {
    const int kc = min(KCH, ninc - c0);
    __syncthreads();
    if (tid < kc) {
      Eid[tid] = m.ne_elem[inc0 + c0 + tid];
      Iloc[tid] = m.ne_loc[inc0 + c0 + tid];
    }
    for (int t = tid; t < KCH * deg; t += 64) slot[t] = -1;
    __syncthreads();
    if (c0 == 0 && tid == 0) {
      const int64_t e0 = Eid[0];
      pself = m.epos[(e0 * NPE + Iloc[0]) * NPE + Iloc[0]];
    }
    for (int t = tid; t < kc * NPE * D; t += 64) {
      const int k = t / (NPE * D), r = t - k * NPE * D, j = r / D, d = r - j * D;
      X[k][j][d] = m.nodes[(int64_t)m.elements[(int64_t)Eid[k] * NPE + j] * D + d];
    }
    for (int t = tid; t < kc * NP; t += 64) {
      const int k = t / NP, i = t - k * NP;
      MP[k][i] = mat_param<MAT, D>(mat, Eid[k], i);
    }
    for (int t = tid; t < kc * NPE; t += 64) {
      const int k = t / NPE, j = t - k * NPE;
      const int64_t e = Eid[k];
      slot[k * deg + m.epos[(e * NPE + Iloc[k]) * NPE + j]] = (signed char)j;
    }
    __syncthreads();
    for (int t = tid; t < kc * NGP; t += 64) {
      const int k = t / NGP, g = t - k * NGP;
      double Ji[D][D];
      const double det = geometry<E>(X[k], g, Ji);
      if (!(det > 0.0)) *bad = 1;
      for (int i = 0; i < D; ++i)
        for (int kk = 0; kk < D; ++kk) Gm[k][g][i * D + kk] = Ji[i][kk];
      Gm[k][g][D * D] = shape_table<E>().w[g] * det * mat_scale(mat, Eid[k]);
    }
    __syncthreads();
    for (int t = tid; t < kc * NPE; t += 64) {
      const int k = t / NPE, j = t - k * NPE, i = Iloc[k];
      double blk[ND2];
      for (int q = 0; q < ND2; ++q) blk[q] = 0.0;
      for (int g = 0; g < NGP; ++g) {
        double Ji[D][D];
        for (int a = 0; a < D; ++a)
          for (int b = 0; b < D; ++b) Ji[a][b] = Gm[k][g][a * D + b];
        double bi[D], bj[D], c[ND2];
        bcol<E>(Ji, g, i, bi);
        bcol<E>(Ji, g, j, bj);
        coupling_block<D, NDOF, MAT>(bi, bj, MP[k], Gm[k][g][D * D], c);
        for (int q = 0; q < ND2; ++q) blk[q] += c[q];
      }
      for (int q = 0; q < ND2; ++q) S[t][q] = blk[q];
    }
    __syncthreads();
    for (int q = tid; q < ND2 * deg; q += 64) {
      const int a = q / L, rem = q - a * L, p = rem / NDOF, b = rem - p * NDOF;
      double v = acc[q];
      for (int k = 0; k < kc; ++k) {
        const int j = slot[k * deg + p];
        if (j >= 0) v += S[k * NPE + j][a * NDOF + b];
      }
      acc[q] = v;
    }
  }
  __syncthreads();
  for (int q = tid; q < ND2 * deg; q += 64) {
    const int a = q / L, rem = q - a * L, p = rem / NDOF, b = rem - p * NDOF;
    const int64_t row = n * NDOF + a;
    const int64_t col = (int64_t)m.adj[a0 + p] * NDOF + b;
    double v = acc[q];
    if (con[row] || con[col]) v = (row == col) ? 1.0 : 0.0;
    acc[q] = v;
    if (v64) v64[vb + q] = v;
    if (v32 && (p != pself || !diff32)) v32[vb + q] = (float)v;
    if (p == pself) dblk[n * ND2 + a * NDOF + b] = v;
  }
  // FP32 difference form: the diagonal block holds the row sums of the
  // final FP64 values, added in ascending slot order
  if (v32 && diff32) {
    __syncthreads();
    if (tid < ND2) {
      const int a = tid / NDOF, b = tid - a * NDOF;
      double r = 0.0;
      for (int p = 0; p < deg; ++p) r += acc[a * L + p * NDOF + b];
      v32[vb + a * L + pself * NDOF + b] = (float)r;
    }
  }
}

// What the rows of a tile of NW nodes need: first values, adjacency, the slot
// of the node itself and the Dirichlet bits of its DOFs.
template <int NW> struct Tile {
  int64_t vb[NW + 1];
  int a0[NW], deg[NW], self[NW], crow[NW];
};

template <int NDOF, int NW>
__device__ __forceinline__ void tile_load(const tfm_mesh_t &m, int64_t n0, const uint8_t *con,
                                          Tile<NW> &tile) {
  const int lane = threadIdx.x;
  if (lane < NW) {
    const int64_t nn = n0 + lane;
    const bool ok = nn < m.n_nod;
    tile.a0[lane] = ok ? m.adj_ptr[nn] : 0;
    tile.deg[lane] = ok ? m.adj_ptr[nn + 1] - m.adj_ptr[nn] : 0;
    tile.vb[lane] = m.val_ptr[ok ? nn : m.n_nod];
    tile.self[lane] = -1;
    int cr = 0;
    for (int a = 0; a < NDOF; ++a) cr |= ok && con[nn * NDOF + a] ? 1 << a : 0;
    tile.crow[lane] = cr;
    if (lane == NW - 1) tile.vb[NW] = m.val_ptr[nn + 1 < m.n_nod ? nn + 1 : m.n_nod];
  }
}

// The tile's accumulated rows, with the Dirichlet rows and columns replaced by
// the identity, to the value arrays.
template <int NDOF, int NW>
__device__ __forceinline__ void tile_epilogue(const tfm_mesh_t &m, int64_t n0, double *acc,
                                              int stride, const unsigned char *cmask,
                                              const Tile<NW> &tile, double *v64, float *v32,
                                              double *dblk, int diff32) {
  constexpr int ND2 = NDOF * NDOF;
  const int lane = threadIdx.x;
  // the tile's rows are contiguous in the value arrays: [tile.vb[0], tile.vb[NW])
  const int64_t vb0 = tile.vb[0];
  const int total = (int)(tile.vb[NW] - vb0);
  int wq = 0, beg = 0, end = (int)(tile.vb[1] - vb0);  // lane's node and its value range
  for (int q = lane; q < total; q += 64) {
    while (end <= q) {
      ++wq;
      beg = end;
      end = (int)(tile.vb[wq + 1] - vb0);
    }
    const int64_t nn = n0 + wq;
    const int deg = tile.deg[wq];
    const int ql = q - beg;
    if (deg == 0) {  // orphan node: only its diagonal is stored (base.py:89-90)
      const double v = (tile.crow[wq] >> ql) & 1 ? 1.0 : 0.0;
      if (v64) v64[vb0 + q] = v;
      if (v32) v32[vb0 + q] = (float)v;
      continue;
    }
    const int L = NDOF * deg;
    int a = 0, rem = ql;  // ql = a L + rem
    for (int k = 1; k < NDOF; ++k)
      if (rem >= L) {
        rem -= L;
        ++a;
      }
    const int p = rem / NDOF, b = rem - p * NDOF;
    const int self = tile.self[wq];
    double *A = acc + wq * stride;
    double v = A[ql];
    if (((tile.crow[wq] >> a) & 1) || ((cmask[wq * m.max_deg + p] >> b) & 1))
      v = (p == self && a == b) ? 1.0 : 0.0;  // row == col
    A[ql] = v;
    if (v64) v64[vb0 + q] = v;
    if (v32 && (p != self || !diff32)) v32[vb0 + q] = (float)v;
    if (p == self) dblk[nn * ND2 + a * NDOF + b] = v;
  }
  for (int q = lane; q < NW * ND2; q += 64) {  // orphan diagonal blocks
    const int ww = q / ND2, ab = q - ww * ND2, a = ab / NDOF, b = ab - a * NDOF;
    const int64_t nn = n0 + ww;
    if (nn < m.n_nod && tile.deg[ww] == 0)
      dblk[nn * ND2 + ab] = (a == b && ((tile.crow[ww] >> a) & 1)) ? 1.0 : 0.0;
  }
  // FP32 difference form: the diagonal block holds the row sums of the
  // final FP64 values, added in ascending slot order
  if (v32 && diff32) {
    __syncthreads();
    for (int q = lane; q < NW * ND2; q += 64) {
      const int ww = q / ND2, ab = q - ww * ND2, a = ab / NDOF, b = ab - a * NDOF;
      const int deg = tile.deg[ww];
      if (n0 + ww >= m.n_nod || deg == 0) continue;
      const int L = NDOF * deg;
      const double *A = acc + ww * stride;
      double r = 0.0;
      for (int p = 0; p < deg; ++p) r += A[a * L + p * NDOF + b];
      v32[tile.vb[ww] + a * L + tile.self[ww] * NDOF + b] = (float)r;
    }
  }
}

// Node-tiled assembly. A 64-lane block assembles the rows of NW consecutive
// nodes. A node owns NPE * IP lanes: IP of its incident elements are taken at
// once (incidence t = r IP + ip in round r), each by NPE lanes, lane j for the
// element's column node j. Per incidence, lane g < NGP evaluates the Jacobian
// at Gauss point g once and shares J^{-1} and the scaled row gradient
// w_g det J_g s_e dN_i/dx through LDS; lane j then forms the geometric moments
//   M_ij[a][c] = sum_g w_g det J_g s_e (dN_i/dx)_a (dN_j/dx)_c
// and the material block once (isotropic elasticity: lam M + G M^T + G tr(M) I;
// heat: kappa : M), the per-point form of coupling_block summed over the
// points. The blocks of a round are added into per-node row accumulators in
// LDS one incidence group after the other (ascending t, a fixed order, so the
// sums are bitwise reproducible), and the tile's rows, contiguous in the value
// arrays, leave in one coalesced pass with the Dirichlet epilogue of
// k_assemble_rows. The element data of RB rounds are loaded together: a batch
// costs three dependent global round trips.
// IP and RB per element type, from timings on the 64^3 Hexa1, 80^3 Tetra1 and
// 32^3 Hexa2 cubes (IP 1-4 and RB 1-4 swept; occupancy is bound by VGPRs and
// LDS together)
template <class E> struct NodeTile;
template <> struct NodeTile<Quad1> { static constexpr int IP = 4, RB = 1; };
template <> struct NodeTile<Tetra1> { static constexpr int IP = 2, RB = 1; };
template <> struct NodeTile<Hexa1> { static constexpr int IP = 2, RB = 2; };
template <> struct NodeTile<Hexa2> { static constexpr int IP = 1, RB = 4; };
// the general (anisotropic) stiffness has 81 parameters per element, too many
// to hold per lane: it keeps the one-node-per-block kernel
template <int MAT> constexpr bool node_tiled() { return MAT != TFM_MAT_GENERAL; }
template <class E> constexpr int tile_nodes() { return 64 / (E::NPE * NodeTile<E>::IP); }

template <class E, int NDOF, int MAT>
__global__ void __launch_bounds__(64) k_assemble_nodes(tfm_mesh_t m, tfm_material_t mat,
                                                       const uint8_t *con, double *v64,
                                                       float *v32, double *dblk, int32_t *bad,
                                                       int diff32) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM, NP = mat_nparam(MAT, D);
  constexpr int IP = NodeTile<E>::IP, RB = NodeTile<E>::RB;
  constexpr int ND2 = NDOF * NDOF, LPN = NPE * IP, NW = tile_nodes<E>(), NG = NW * IP;
  constexpr int GW = D * D + D;  // per point: J^{-1}, then the scaled row gradient
  constexpr int CQ = 4;          // Dirichlet-bit chunk: 64 CQ columns
  static_assert(NW >= 1 && NGP <= NPE, "a tile holds whole nodes, one point per lane");
  static_assert(MAT != TFM_MAT_GENERAL, "the general stiffness keeps k_assemble_rows");
  extern __shared__ double acc[];  // [NW][ND2 * max_deg] row accumulators, then
                                   // [NW][max_deg] Dirichlet bits of the columns
  // row strides padded by two doubles: the 8-byte banks of rows that lanes
  // read at the same time then differ (no bank conflicts between groups)
  constexpr int TS = D * NPE + 2, XS = NPE * D + 2, GS = NGP * GW + 2;
  __shared__ double tbl[NGP][TS];  // dN[g][a][N] at [g][a * NPE + N]
  __shared__ double tw[NGP];
  __shared__ double Xs[NG][XS];   // [group][N * D + c]
  __shared__ double Gm[NG][GS];   // [group][g * GW + ...]
  __shared__ Tile<NW> tile;

  const int lane = threadIdx.x;
  const int w = lane / LPN, ip = (lane / NPE) % IP, j = lane % NPE, grp = w * IP + ip;
  const int64_t n0 = xcd_block() * (int64_t)NW;
  const int64_t n = n0 + w;
  const bool valid = lane < NW * LPN && n < m.n_nod;
  const int stride = ND2 * m.max_deg;
  unsigned char *cmask = reinterpret_cast<unsigned char *>(acc + NW * stride);
  int inc0 = 0, ninc = 0;
  if (valid) {
    inc0 = m.ne_ptr[n];
    ninc = m.ne_ptr[n + 1] - inc0;
  }
  tile_load<NDOF, NW>(m, n0, con, tile);
  const auto &T = shape_table<E>();
  for (int q = lane; q < NGP * D * NPE; q += 64) tbl[q / (D * NPE)][q % (D * NPE)] = (&T.dN[0][0][0])[q];
  for (int q = lane; q < NGP; q += 64) tw[q] = T.w[q];
  for (int q = lane; q < NW * stride; q += 64) acc[q] = 0.0;
  __syncthreads();

  // Dirichlet bits of every column node of the tile's rows (two dependent
  // loads each), in chunks of 64 CQ columns; the first chunk rides along with
  // the element loads of the first batch, and the epilogue reads LDS only
  const int nq = NW * m.max_deg;
  auto cm_adj = [&](int q0, int (&nbr)[CQ]) {
#pragma unroll
    for (int c = 0; c < CQ; ++c) {
      const int q = q0 + c * 64 + lane;
      nbr[c] = -1;
      if (q < nq) {
        const int ww = q / m.max_deg, p = q - ww * m.max_deg;
        if (p < tile.deg[ww]) nbr[c] = m.adj[tile.a0[ww] + p];
      }
    }
  };
  auto cm_con = [&](int q0, const int (&nbr)[CQ]) {
#pragma unroll
    for (int c = 0; c < CQ; ++c) {
      const int q = q0 + c * 64 + lane;
      int bits = 0;
      if (nbr[c] >= 0)
        for (int b = 0; b < NDOF; ++b) bits |= con[(int64_t)nbr[c] * NDOF + b] ? 1 << b : 0;
      if (q < nq) cmask[q] = (unsigned char)bits;
    }
  };

  const int rounds = (m.max_inc + IP - 1) / IP;
  for (int r0 = 0; r0 < rounds; r0 += RB) {
    // the batch's element data: incidences, then connectivity, slots and
    // parameters, then coordinates
    int e[RB], il[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int t = (r0 + b) * IP + ip;
      e[b] = -1;
      il[b] = 0;
      if (valid && t < ninc) {
        e[b] = m.ne_elem[inc0 + t];
        il[b] = m.ne_loc[inc0 + t];
      }
    }
    int nbr[CQ];
    if (r0 == 0) cm_adj(0, nbr);
    int64_t id[RB];
    int P[RB];  // slot of the lane's column node in the row node's adjacency
    double mp[RB][NP], se[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      id[b] = 0;
      P[b] = 0;
      se[b] = 0.0;
      for (int q = 0; q < NP; ++q) mp[b][q] = 0.0;
      if (e[b] >= 0) {
        const int64_t eb = e[b];
        id[b] = m.elements[eb * NPE + j];
        P[b] = m.epos[(eb * NPE + il[b]) * NPE + j];
        for (int q = 0; q < NP; ++q) mp[b][q] = mat_param<MAT, D>(mat, eb, q);
        se[b] = mat_scale(mat, eb);
      }
    }
    if (r0 == 0) cm_con(0, nbr);
    double X[RB][D];
#pragma unroll
    for (int b = 0; b < RB; ++b)
      for (int d = 0; d < D; ++d) X[b][d] = e[b] >= 0 ? m.nodes[id[b] * D + d] : 0.0;

#pragma unroll
    for (int b = 0; b < RB; ++b) {
      if (r0 + b >= rounds) break;
      const bool act = e[b] >= 0;
      const int i = il[b];
      if (act) {
        for (int d = 0; d < D; ++d) Xs[grp][j * D + d] = X[b][d];
        if (r0 + b == 0 && ip == 0 && j == i) tile.self[w] = P[b];
      }
      __syncthreads();
      if (act && j < NGP) {  // lane g = j: the geometry of point g
        const int g = j;
        double J[D][D];
        for (int a = 0; a < D; ++a)
          for (int c = 0; c < D; ++c) J[a][c] = 0.0;
        for (int N = 0; N < NPE; ++N)
          for (int a = 0; a < D; ++a)
            for (int c = 0; c < D; ++c) J[a][c] += tbl[g][a * NPE + N] * Xs[grp][N * D + c];
        double Ji[D][D];
        const double det = inv_jac<D>(J, Ji);
        if (!(det > 0.0)) *bad = 1;
        const double wd = tw[g] * det * se[b];
        double *G = &Gm[grp][g * GW];
        for (int a = 0; a < D; ++a) {
          double v = 0.0;
          for (int c = 0; c < D; ++c) {
            G[a * D + c] = Ji[a][c];
            v += Ji[a][c] * tbl[g][c * NPE + i];
          }
          G[D * D + a] = v * wd;
        }
      }
      __syncthreads();
      double blk[ND2];
      if (act) {
        double M[D * D];
        for (int q = 0; q < D * D; ++q) M[q] = 0.0;
        for (int g = 0; g < NGP; ++g) {
          const double *G = &Gm[grp][g * GW];
          double bj[D];
          for (int a = 0; a < D; ++a) {
            double v = 0.0;
            for (int c = 0; c < D; ++c) v += G[a * D + c] * tbl[g][c * NPE + j];
            bj[a] = v;
          }
          if constexpr (MAT == TFM_MAT_HEAT_ISO) {
            for (int a = 0; a < D; ++a) M[0] += G[D * D + a] * bj[a];
          } else {
            for (int a = 0; a < D; ++a)
              for (int c = 0; c < D; ++c) M[a * D + c] += G[D * D + a] * bj[c];
          }
        }
        if constexpr (MAT == TFM_MAT_ISO) {
          double tr = 0.0;
          for (int a = 0; a < D; ++a) tr += M[a * D + a];
          for (int a = 0; a < D; ++a)
            for (int c = 0; c < D; ++c)
              blk[a * NDOF + c] = mp[b][0] * M[a * D + c] + mp[b][1] * M[c * D + a] +
                                  (a == c ? mp[b][1] * tr : 0.0);
        } else if constexpr (MAT == TFM_MAT_HEAT_ISO) {
          blk[0] = mp[b][0] * M[0];
        } else {
          double v = 0.0;
          for (int q = 0; q < D * D; ++q) v += mp[b][q] * M[q];
          blk[0] = v;
        }
      }
      // add the blocks in ascending incidence order: group ip at step ip
      for (int st = 0; st < IP; ++st) {
        if (act && ip == st) {
          double *A = acc + w * stride;
          const int L = NDOF * tile.deg[w];
          for (int a = 0; a < NDOF; ++a)
            for (int c = 0; c < NDOF; ++c) A[a * L + P[b] * NDOF + c] += blk[a * NDOF + c];
        }
        __syncthreads();
      }
    }
  }
  for (int q0 = rounds > 0 ? 64 * CQ : 0; q0 < nq; q0 += 64 * CQ) {
    int nbr[CQ];
    cm_adj(q0, nbr);
    cm_con(q0, nbr);
  }
  __syncthreads();
  tile_epilogue<NDOF, NW>(m, n0, acc, stride, cmask, tile, v64, v32, dblk, diff32);
}

// ============================================================ point teams
// Kernels below give each element one lane per Gauss point, 64 / NGP elements
// to a wave (and a block). The nodal data and the shape-function derivatives
// lie in LDS, so a lane forms the Jacobian and the nodal sums at its point by
// itself: one lane per node instead needs a butterfly over the team for every
// component of J and of grad u at every point, 864 LDS permutations per wave
// of eight Hexa1 elements where this takes about 170 LDS reads.
template <class E> constexpr int point_elems() { return 64 / E::NGP; }

// dN/dxi of every point into LDS: tbl[g][k * NPE + N].
template <class E>
__device__ __forceinline__ void stage_table(double (&tbl)[E::NGP][odd(E::DIM * E::NPE)]) {
  constexpr int R = E::DIM * E::NPE;
  const auto &T = shape_table<E>();
  for (int q = threadIdx.x; q < E::NGP * R; q += blockDim.x) tbl[q / R][q % R] = (&T.dN[0][0][0])[q];
}

// Nodal values v[n][C] of the elements [e0, e0 + ne) into rows of LDS.
template <class E, int C, int S>
__device__ __forceinline__ void stage_nodal(const tfm_mesh_t &m, int64_t e0, int ne,
                                            const double *v, double (*rows)[S]) {
  for (int t = threadIdx.x; t < ne * E::NPE; t += blockDim.x) {
    const int k = t / E::NPE, j = t - k * E::NPE;
    const int64_t n = m.elements[e0 * E::NPE + t];
    for (int c = 0; c < C; ++c) rows[k][j * C + c] = v[n * C + c];
  }
}

// Sums over the nodes of v[N][a] dN_N/dxi_k at one point.
template <class E, int C>
__device__ __forceinline__ void point_sums(const double *row, const double *t,
                                           double (&out)[C][E::DIM]) {
  constexpr int NPE = E::NPE, D = E::DIM;
  for (int a = 0; a < C; ++a)
    for (int k = 0; k < D; ++k) out[a][k] = 0.0;
#pragma unroll 4
  for (int N = 0; N < NPE; ++N)
    for (int a = 0; a < C; ++a)
      for (int k = 0; k < D; ++k) out[a][k] += row[N * C + a] * t[k * NPE + N];
}

// J^{-1} and det J at one point.
template <class E>
__device__ __forceinline__ double point_geometry(const double *X, const double *t,
                                                 double (&Ji)[E::DIM][E::DIM]) {
  constexpr int D = E::DIM;
  double S[D][D], J[D][D];
  point_sums<E, D>(X, t, S);
  for (int i = 0; i < D; ++i)
    for (int k = 0; k < D; ++k) J[i][k] = S[k][i];
  return inv_jac<D>(J, Ji);
}

// H[a][i] = sum_N u[N][a] B[i][N] at one point (base.py:1052).
template <class E, int NDOF>
__device__ __forceinline__ void point_grad(const double *u, const double *t,
                                           const double (&Ji)[E::DIM][E::DIM],
                                           double (&H)[NDOF * E::DIM]) {
  constexpr int D = E::DIM;
  double S[NDOF][D];
  point_sums<E, NDOF>(u, t, S);
  for (int a = 0; a < NDOF; ++a)
    for (int i = 0; i < D; ++i) {
      double acc = 0.0;
      for (int k = 0; k < D; ++k) acc += Ji[i][k] * S[a][k];
      H[a * D + i] = acc;
    }
}

// Material parameters of a lane's element: the few of an isotropic or heat
// layout in registers; the 81 (16) of a general stiffness in LDS where a team
// shares them, and read in place where every lane has an element of its own
// (64 of them would leave two waves per CU).
template <class E, int MAT> struct PointParams {
  static constexpr int NP = mat_nparam(MAT, E::DIM);
  static constexpr bool REG = NP <= 9, LDS = !REG && E::NGP > 1;
  static constexpr int ROWS = LDS ? point_elems<E>() : 1, STRIDE = LDS ? odd(NP) : 1;
  double v[REG ? NP : 1];
  const double *at;
  __device__ __forceinline__ static void stage(const tfm_material_t &mat, int64_t e0, int ne,
                                               double (&rows)[ROWS][STRIDE]) {
    if constexpr (LDS)
      for (int t = threadIdx.x; t < ne * NP; t += blockDim.x) rows[t / NP][t % NP] = mat.p0[e0 * NP + t];
  }
  __device__ __forceinline__ PointParams(const tfm_material_t &mat, int64_t e0, int el,
                                         const double (&rows)[ROWS][STRIDE]) {
    if constexpr (REG) {
      for (int q = 0; q < NP; ++q) v[q] = mat_param<MAT, E::DIM>(mat, e0 + el, q);
    } else {
      at = LDS ? rows[LDS ? el : 0] : mat.p0 + (e0 + el) * NP;
    }
  }
  __device__ __forceinline__ const double *get() const {
    if constexpr (REG) return v;
    else return at;
  }
};

// Internal element forces fe[e][j][a] = sum_g w detJ s sum_i B[i][j] q[a][i]
// with q = flux_prev + flux(grad u) (base.py:1050-1083 / 1250-1268); also
// the Gauss-point means of grad u and q, and both per point. Lane (e, g) forms
// q at its point and T[a][k] = w detJ s sum_i q[a][i] Jinv[i][k]; lane (e, j)
// then adds T[a][k] dN_j/dxi_k over the points. Per-point values pass through
// LDS, so that 64 lanes move the NQ * 64 / NGP consecutive values of a point.
// Bound by the per-point arrays in memory where they are asked for, otherwise
// by LDS reads. With one lane per node instead: Hexa1 43x37x40 with per-point
// arrays (121 MB) 143 us, now 47; Hexa2 21x19x23 means only 87 us, now 14;
// Tetra1 heat 63^3 98 us, now 58.
template <class E, int NDOF, int MAT>
__global__ void __launch_bounds__(64) k_internal_force(tfm_mesh_t m, tfm_material_t mat,
                                                       const double *u, const double *qprev,
                                                       double *fe, double *grad_mean,
                                                       double *flux_mean, double *grad_gp,
                                                       double *flux_gp) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM;
  constexpr int EPB = point_elems<E>(), NQ = NDOF * D, SQ = EPB * NQ;
  __shared__ double tbl[NGP][odd(D * NPE)];
  __shared__ double Xs[EPB][odd(NPE * D)], Us[EPB][odd(NPE * NDOF)];
  using Params = PointParams<E, MAT>;
  __shared__ double MP[Params::ROWS][Params::STRIDE];
  __shared__ double st[64][odd(NQ)];  // per-point values of lane e * NGP + g
  const int lane = threadIdx.x, el = lane / NGP, g = lane % NGP;
  const int64_t e0 = xcd_block() * EPB;
  const int ne = (int)(m.n_elem - e0 < EPB ? m.n_elem - e0 : EPB);
  stage_table<E>(tbl);
  stage_nodal<E, D>(m, e0, ne, m.nodes, Xs);
  stage_nodal<E, NDOF>(m, e0, ne, u, Us);
  Params::stage(mat, e0, ne, MP);
  if (qprev)
    for (int t = lane; t < NGP * SQ; t += 64) {
      const int gg = t / SQ, r = t - gg * SQ, k = r / NQ;
      if (k < ne) st[k * NGP + gg][r - k * NQ] = qprev[((int64_t)gg * m.n_elem + e0) * NQ + r];
    }
  __syncthreads();
  double H[NQ], Q[NQ], T[NQ];
  for (int q = 0; q < NQ; ++q) H[q] = Q[q] = T[q] = 0.0;
  if (el < ne) {
    double Ji[D][D];
    const double det = point_geometry<E>(Xs[el], tbl[g], Ji);
    point_grad<E, NDOF>(Us[el], tbl[g], Ji, H);
    flux_from_grad<D, NDOF, MAT>(H, Params(mat, e0, el, MP).get(), Q);
    if (qprev)
      for (int q = 0; q < NQ; ++q) Q[q] += st[lane][q];
    const double wd = shape_table<E>().w[g] * det * mat_scale(mat, e0 + el);
    for (int a = 0; a < NDOF; ++a)
      for (int k = 0; k < D; ++k) {
        double acc = 0.0;
        for (int i = 0; i < D; ++i) acc += Q[a * D + i] * Ji[i][k];
        T[a * D + k] = wd * acc;
      }
  }
  // a per-point tensor and its mean over the points
  auto emit = [&](const double (&v)[NQ], double *gp, double *mean) {
    __syncthreads();
    for (int q = 0; q < NQ; ++q) st[lane][q] = v[q];
    __syncthreads();
    if (gp)
      for (int t = lane; t < NGP * SQ; t += 64) {
        const int gg = t / SQ, r = t - gg * SQ, k = r / NQ;
        if (k < ne) gp[((int64_t)gg * m.n_elem + e0) * NQ + r] = st[k * NGP + gg][r - k * NQ];
      }
    if (mean)
      for (int t = lane; t < ne * NQ; t += 64) {
        const int k = t / NQ, q = t - k * NQ;
        double acc = 0.0;
        for (int gg = 0; gg < NGP; ++gg) acc += st[k * NGP + gg][q];
        mean[e0 * NQ + t] = acc / NGP;
      }
  };
  if (grad_gp || grad_mean) emit(H, grad_gp, grad_mean);
  if (flux_gp || flux_mean) emit(Q, flux_gp, flux_mean);
  __syncthreads();
  for (int q = 0; q < NQ; ++q) st[lane][q] = T[q];
  __syncthreads();
  for (int t = lane; t < ne * NPE; t += 64) {
    const int k = t / NPE, j = t - k * NPE;
    double f[NDOF];
    for (int a = 0; a < NDOF; ++a) f[a] = 0.0;
#pragma unroll 4
    for (int gg = 0; gg < NGP; ++gg)
      for (int kk = 0; kk < D; ++kk) {
        const double b = tbl[gg][kk * NPE + j];
        for (int a = 0; a < NDOF; ++a) f[a] += st[k * NGP + gg][a * D + kk] * b;
      }
    for (int a = 0; a < NDOF; ++a) fe[(e0 * NPE + t) * NDOF + a] = f[a];
  }
}

// F[n*nd+a] = sum over incident elements (ascending) of fe[e][loc][a]: the
// scatter of FEM.assemble_rhs (base.py:439-445) as an ordered gather.
template <int NDOF>
__global__ void k_gather_nodes(tfm_mesh_t m, const double *fe, double *F) {
  const int64_t t = xcd_block() * blockDim.x + threadIdx.x;
  if (t >= m.n_nod * NDOF) return;
  const int64_t n = t / NDOF;
  const int a = (int)(t - n * NDOF);
  double acc = 0.0;
  int k = m.ne_ptr[n];
  const int k_end = m.ne_ptr[n + 1];
  auto at = [&](int i) -> int64_t {
    return ((int64_t)m.ne_elem[i] * m.npe + m.ne_loc[i]) * NDOF + a;
  };
  // four incident elements per round: their index and value loads are in
  // flight together, and the sum keeps the ascending element order
  for (; k + 3 < k_end; k += 4) {
    const int64_t i0 = at(k), i1 = at(k + 1), i2 = at(k + 2), i3 = at(k + 3);
    const double v0 = fe[i0], v1 = fe[i1], v2 = fe[i2], v3 = fe[i3];
    acc += v0;
    acc += v1;
    acc += v2;
    acc += v3;
  }
  for (; k < k_end; ++k) acc += fe[at(k)];
  F[t] = acc;
}

// Assembly from given element matrices kin [E, W, W]: LPN lanes per node, NW =
// 64 / LPN consecutive nodes per block. The NDOF rows that an element gives a
// node are NDOF * W consecutive values of kin; the lanes load those of U
// elements together and add them into the node's rows in LDS one element after
// the other (ascending, a fixed order, one writer per entry), so every value of
// kin is read once, in whole lines. The tile leaves as in k_assemble_nodes.
// Bound by reading kin: Hexa1 43x37x40 135 us (420 MB in and out, 3.1 TB/s), 297
// us with a gather of every entry from its elements; Hexa2 13x15x11 35 us (99).
// Two or eight elements at once took 135 and 148 us.
// lanes per node: the fewest that hold its values of an element in three rounds
// (72 of Hexa1: 32 lanes and 135 us on 43x37x40; 64 lanes with two rounds, of
// which the second is nearly empty, 145 us)
constexpr int assemble_lanes(int npe, int nd) {
  int l = 4;
  while (l < 64 && l * 3 < npe * nd * nd) l *= 2;
  return l;
}

template <int NPE, int NDOF>
__global__ void __launch_bounds__(64) k_assemble_elements(tfm_mesh_t m, const double *kin,
                                                          const uint8_t *con, double *v64,
                                                          float *v32, double *dblk, int diff32) {
  constexpr int W = NPE * NDOF, ND2 = NDOF * NDOF, NV = NDOF * W;
  constexpr int LPN = assemble_lanes(NPE, NDOF), NW = 64 / LPN;
  constexpr int IR = (NV + LPN - 1) / LPN, U = 4;  // values per lane and element, elements
  extern __shared__ double acc[];  // rows [NW][ND2 * max_deg], Dirichlet bits [NW][max_deg]
  __shared__ Tile<NW> tile;
  const int lane = threadIdx.x, w = lane / LPN, l = lane % LPN;
  const int64_t n0 = xcd_block() * (int64_t)NW;
  const int64_t n = n0 + w;
  const int stride = ND2 * m.max_deg;
  unsigned char *cmask = reinterpret_cast<unsigned char *>(acc + NW * stride);
  int inc0 = 0, ninc = 0;
  if (n < m.n_nod) {
    inc0 = m.ne_ptr[n];
    ninc = m.ne_ptr[n + 1] - inc0;
    if (ninc == 0) inc0 = 0;  // an index that can be read
  }
  int most = ninc;  // over the tile
#pragma unroll
  for (int off = LPN; off < 64; off <<= 1) most = max(most, __shfl_xor(most, off, 64));
  tile_load<NDOF, NW>(m, n0, con, tile);
  for (int q = lane; q < NW * stride; q += 64) acc[q] = 0.0;
  __syncthreads();
  const int deg = tile.deg[w], L = NDOF * deg;
  for (int p = l; p < deg; p += LPN) {
    const int64_t c = m.adj[tile.a0[w] + p];
    int bits = 0;
    for (int b = 0; b < NDOF; ++b) bits |= con[c * NDOF + b] ? 1 << b : 0;
    cmask[w * m.max_deg + p] = (unsigned char)bits;
  }
  for (int t0 = 0; t0 < most; t0 += U) {
    // (no branches around the loads: past the last element, or value, the
    // last one is read again and not added)
    int64_t e[U];
    int il[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = inc0 + max(min(t0 + u, ninc - 1), 0);
      e[u] = m.ne_elem[k];
      il[u] = m.ne_loc[k];
    }
    double v[U][IR];
    int at[U][IR];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < IR; ++r) {
        const int q = min(l + r * LPN, NV - 1), j = q % W / NDOF;
        v[u][r] = kin[e[u] * (W * W) + il[u] * NV + q];
        at[u][r] = m.epos[(e[u] * NPE + il[u]) * NPE + j];
        if (t0 + u == 0 && ninc > 0 && j == il[u]) tile.self[w] = at[u][r];
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < IR; ++r) {
        const int q = l + r * LPN, a = q / W, col = q - a * W;
        at[u][r] = t0 + u < ninc && q < NV ? a * L + at[u][r] * NDOF + col % NDOF : -1;
      }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int r = 0; r < IR; ++r)
        if (at[u][r] >= 0) acc[w * stride + at[u][r]] += v[u][r];
      __syncthreads();
    }
  }
  __syncthreads();
  tile_epilogue<NDOF, NW>(m, n0, acc, stride, cmask, tile, v64, v32, dblk, diff32);
}

// The same for any number of element nodes, and for degrees whose rows do not fit
// LDS: a block per node, which gathers every entry from the node's elements.
template <int NDOF>
__global__ void __launch_bounds__(64) k_assemble_elements_any(tfm_mesh_t m, const double *kin,
                                                              const uint8_t *con, double *v64,
                                                              float *v32, double *dblk,
                                                              int diff32) {
  constexpr int ND2 = NDOF * NDOF;
  extern __shared__ signed char slot_dyn[];  // [max_inc * max_deg]
  const int64_t n = xcd_block();
  const int tid = threadIdx.x;
  const int npe = m.npe, W = npe * NDOF;
  const int a0 = m.adj_ptr[n];
  const int deg = m.adj_ptr[n + 1] - a0;
  const int64_t vb = m.val_ptr[n];
  if (deg == 0) {
    if (tid < NDOF) {
      const double v = con[n * NDOF + tid] ? 1.0 : 0.0;
      if (v64) v64[vb + tid] = v;
      if (v32) v32[vb + tid] = (float)v;
    }
    for (int t = tid; t < ND2; t += 64) {
      const int a = t / NDOF, b = t - a * NDOF;
      dblk[n * ND2 + t] = (a == b && con[n * NDOF + a]) ? 1.0 : 0.0;
    }
    return;
  }
  const int inc0 = m.ne_ptr[n], ninc = m.ne_ptr[n + 1] - inc0;
  for (int t = tid; t < ninc * deg; t += 64) slot_dyn[t] = -1;
  __syncthreads();
  for (int t = tid; t < ninc * npe; t += 64) {
    const int k = t / npe, j = t - k * npe;
    const int64_t e = m.ne_elem[inc0 + k];
    slot_dyn[k * deg + m.epos[(e * npe + m.ne_loc[inc0 + k]) * npe + j]] = (signed char)j;
  }
  __syncthreads();
  int pself = 0;
  for (int p = 0; p < deg; ++p)
    if (m.adj[a0 + p] == n) pself = p;
  const int L = NDOF * deg;
  // entry (a, p, b) of the node's rows with the Dirichlet epilogue applied
  auto entry = [&](int a, int p, int b) -> double {
    double v = 0.0;
    for (int k = 0; k < ninc; ++k) {
      const int j = slot_dyn[k * deg + p];
      if (j >= 0) {
        const int64_t e = m.ne_elem[inc0 + k];
        const int i = m.ne_loc[inc0 + k];
        v += kin[e * W * W + (int64_t)(i * NDOF + a) * W + j * NDOF + b];
      }
    }
    const int64_t row = n * NDOF + a;
    const int64_t col = (int64_t)m.adj[a0 + p] * NDOF + b;
    if (con[row] || con[col]) v = (row == col) ? 1.0 : 0.0;
    return v;
  };
  for (int q = tid; q < ND2 * deg; q += 64) {
    const int a = q / L, rem = q - a * L, p = rem / NDOF, b = rem - p * NDOF;
    const double v = entry(a, p, b);
    if (v64) v64[vb + q] = v;
    if (v32 && (p != pself || !diff32)) v32[vb + q] = (float)v;
    if (p == pself) dblk[n * ND2 + a * NDOF + b] = v;
  }
  // FP32 difference form: the diagonal block holds the FP64 row sums
  if (v32 && diff32 && tid < ND2) {
    const int a = tid / NDOF, b = tid - a * NDOF;
    double r = 0.0;
    for (int p = 0; p < deg; ++p) r += entry(a, p, b);
    v32[vb + a * L + pself * NDOF + b] = (float)r;
  }
}

// Elements per block of the sensitivities: fewer where a lane would have an
// element of its own and the layout is general. The outputs (82 values of an
// anisotropic Tetra1) are the work then, and 64 elements' of them one after the
// other leave a small mesh to a few waves and five waves to a CU. Anisotropic
// Tetra1, 16 right-hand sides: 750 elements 207 us with 64 to a block, 61 with 8
// and 84 with 16 (a lane per node 72); 93,750 elements 647, 481 and 380 (561); the
// line between 8 and 16 lies at a block of 16 for every CU, four times over.
template <class E, int MAT> constexpr bool sens_outputs() {
  return E::NGP == 1 && (MAT == TFM_MAT_GENERAL || MAT == TFM_MAT_HEAT_GENERAL);
}

// Sensitivities of lam^T K(p) u per element (see tfm_sensitivity in tfm.h):
// a lane per Gauss point, whose geometry serves every right-hand side.
// Hexa2 21x19x23 with 12 right-hand sides: 1385 us with a lane per node and
// the geometry formed for each, now 80; Hexa1 47x41x52 with one 186 us, now 28.
template <class E, int NDOF, int MAT, int EPB>
__global__ void __launch_bounds__(64) k_sensitivity(tfm_mesh_t m, tfm_material_t mat,
                                                    const double *u, const double *lam,
                                                    int nrhs, double sign, double *out) {
  constexpr int NPE = E::NPE, NGP = E::NGP, D = E::DIM, NP = mat_nparam(MAT, D);
  constexpr int NQ = NDOF * D;
  constexpr bool ISO = (MAT == TFM_MAT_ISO || MAT == TFM_MAT_HEAT_ISO);
  constexpr int NI = MAT == TFM_MAT_ISO ? 2 : 1, NO = (ISO ? NI : NP) + 1;
  __shared__ double tbl[NGP][odd(D * NPE)];
  __shared__ double Xs[EPB][odd(NPE * D)];
  __shared__ double Us[EPB][odd(NPE * NDOF)], Ls[EPB][odd(NPE * NDOF)];
  using Params = PointParams<E, MAT>;
  __shared__ double MP[Params::ROWS][Params::STRIDE];
  // general layouts: w detJ s grad(lam), sym(grad u) or grad u, and the energy
  __shared__ double st[ISO ? 1 : EPB * NGP][odd(2 * NQ + 1)];
  const int lane = threadIdx.x, el = lane / NGP, g = lane % NGP;
  const int64_t e0 = xcd_block() * EPB;
  const int ne = (int)(m.n_elem - e0 < EPB ? m.n_elem - e0 : EPB);
  const bool live = el < ne;
  stage_table<E>(tbl);
  stage_nodal<E, D>(m, e0, ne, m.nodes, Xs);
  Params::stage(mat, e0, ne, MP);
  __syncthreads();
  const double sc = live ? mat_scale(mat, e0 + el) : 0.0;
  const Params mp(mat, e0, live ? el : 0, MP);
  double Ji[D][D], wd = 0.0;
  for (int i = 0; i < D; ++i)
    for (int k = 0; k < D; ++k) Ji[i][k] = 0.0;
  if (live) wd = shape_table<E>().w[g] * point_geometry<E>(Xs[el], tbl[g], Ji);
  const int64_t ndofs = m.n_nod * NDOF;
  for (int r = 0; r < nrhs; ++r) {
    __syncthreads();
    stage_nodal<E, NDOF>(m, e0, ne, u + r * ndofs, Us);
    stage_nodal<E, NDOF>(m, e0, ne, lam + r * ndofs, Ls);
    __syncthreads();
    double *o = out + ((int64_t)r * m.n_elem + e0) * NO;
    double acc[3] = {0.0, 0.0, 0.0};
    double Hu[NQ], Hl[NQ];
    if (live) {
      double Q[NQ];
      point_grad<E, NDOF>(Us[el], tbl[g], Ji, Hu);
      point_grad<E, NDOF>(Ls[el], tbl[g], Ji, Hl);
      // d/dscale: sum_g w detJ Hl : flux(Hu)
      flux_from_grad<D, NDOF, MAT>(Hu, mp.get(), Q);
      double en = 0.0;
      for (int q = 0; q < NQ; ++q) en += Hl[q] * Q[q];
      acc[2] = wd * en;
      if constexpr (MAT == TFM_MAT_ISO) {
        double tl = 0.0, tu = 0.0, dd = 0.0;
        for (int i = 0; i < D; ++i) {
          tl += Hl[i * D + i];
          tu += Hu[i * D + i];
        }
        for (int i = 0; i < D; ++i)
          for (int k = 0; k < D; ++k) dd += Hl[i * D + k] * (Hu[i * D + k] + Hu[k * D + i]);
        acc[0] = wd * sc * tl * tu;
        acc[1] = wd * sc * dd;
      } else if constexpr (MAT == TFM_MAT_HEAT_ISO) {
        double dd = 0.0;
        for (int i = 0; i < D; ++i) dd += Hl[i] * Hu[i];
        acc[0] = wd * sc * dd;
      }
    }
    if constexpr (ISO) {
#pragma unroll
      for (int off = 1; off < NGP; off <<= 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[c] += __shfl_xor(acc[c], off, 64);
      if (live && g == 0) {
        for (int c = 0; c < NI; ++c) o[el * NO + c] = sign * acc[c];
        o[el * NO + NI] = sign * acc[2];
      }
    } else {
      // general: d/dC[i,J,k,L] = Hl[i][J] eps_u[k][L]; heat: d/dKAPPA[i,j] =
      // dT_l/dx_i dT_u/dx_j. Mechanics pairs Hl with the strain sym(Hu): the
      // residual depends on C only through C : sym(grad u)
      // (elasticity.py:121-123)
      if (live) {
        for (int x = 0; x < NQ; ++x) {
          st[lane][x] = wd * sc * Hl[x];
          double h = Hu[x];
          if constexpr (MAT == TFM_MAT_GENERAL) h = 0.5 * (Hu[x] + Hu[(x % D) * D + x / D]);
          st[lane][NQ + x] = h;
        }
        st[lane][2 * NQ] = acc[2];
      }
      __syncthreads();
      for (int t = lane; t < ne * NO; t += 64) {
        const int k = t / NO, c = t - k * NO;
        double v = 0.0;
        for (int gg = 0; gg < NGP; ++gg) {
          const double *S = st[k * NGP + gg];
          v += c < NP ? S[c / NQ] * S[NQ + c % NQ] : S[2 * NQ];
        }
        o[t] = sign * v;
      }
    }
  }
}

// ================================================================ dispatch
#define TFM_DISPATCH(ETYPE, ...)                                                                \
  switch (ETYPE) {                                                                             \
    case TFM_QUAD1: { using ET = Quad1; __VA_ARGS__; break; }                                  \
    case TFM_TETRA1: { using ET = Tetra1; __VA_ARGS__; break; }                                \
    case TFM_HEXA1: { using ET = Hexa1; __VA_ARGS__; break; }                                  \
    case TFM_HEXA2: { using ET = Hexa2; __VA_ARGS__; break; }                                  \
    default: TFM_REQUIRE(false, "unsupported element type");                                    \
  }

static int check_mesh_mat(const tfm_mesh_t &m, const tfm_material_t &mat) {
  const bool heat = (mat.kind == TFM_MAT_HEAT_ISO || mat.kind == TFM_MAT_HEAT_GENERAL);
  TFM_REQUIRE(mat.kind >= TFM_MAT_ISO && mat.kind <= TFM_MAT_HEAT_GENERAL, "unknown material kind");
  TFM_REQUIRE(heat ? m.ndof == 1 : m.ndof == m.dim,
              "material kind does not match the DOFs per node");
  TFM_REQUIRE(mat.p0 && (mat.kind != TFM_MAT_ISO || mat.p1), "material parameters missing");
  int dim = 0, npe = 0;
  switch (m.etype) {
    case TFM_QUAD1: dim = 2; npe = 4; break;
    case TFM_TETRA1: dim = 3; npe = 4; break;
    case TFM_HEXA1: dim = 3; npe = 8; break;
    case TFM_HEXA2: dim = 3; npe = 20; break;
    default: TFM_REQUIRE(false, "unsupported element type");
  }
  TFM_REQUIRE(m.dim == dim && m.npe == npe, "mesh dim/npe do not match the element type");
  return TFM_OK;
}

// Runs BODY with compile-time ET, ND (DOFs per node) and MK (material kind).
#define TFM_DISPATCH_ALL(m, mat, ...)                                                           \
  do {                                                                                         \
    int _rc = check_mesh_mat(m, mat);                                                          \
    if (_rc != TFM_OK) return _rc;                                                             \
    const bool _heat = (mat.kind == TFM_MAT_HEAT_ISO || mat.kind == TFM_MAT_HEAT_GENERAL);    \
    TFM_DISPATCH(m.etype, {                                                                    \
      if (_heat) {                                                                             \
        constexpr int ND = 1;                                                                  \
        if (mat.kind == TFM_MAT_HEAT_ISO) { constexpr int MK = TFM_MAT_HEAT_ISO; __VA_ARGS__; } \
        else { constexpr int MK = TFM_MAT_HEAT_GENERAL; __VA_ARGS__; }                         \
      } else {                                                                                 \
        constexpr int ND = ET::DIM;                                                            \
        if (mat.kind == TFM_MAT_ISO) { constexpr int MK = TFM_MAT_ISO; __VA_ARGS__; }          \
        else { constexpr int MK = TFM_MAT_GENERAL; __VA_ARGS__; }                              \
      }                                                                                        \
    });                                                                                        \
  } while (0)

int launch_element_matrices(hipStream_t s, const tfm_mesh_t &m, const tfm_material_t &mat,
                            double *k, int32_t *bad) {
  if (m.n_elem == 0) return TFM_OK;
  TFM_DISPATCH_ALL(m, mat, {
    constexpr int EB = matrix_elems<ET>();
    hipLaunchKernelGGL((k_element_matrices<ET, ND, MK>), dim3((unsigned)((m.n_elem + EB - 1) / EB)),
                       dim3(matrix_threads<ET>()), 0, s, m, mat, k, bad);
    TFM_CHECK_LAUNCH();
  });
  return TFM_OK;
}

int launch_assemble(hipStream_t s, const tfm_mesh_t &m, const tfm_material_t &mat,
                    const uint8_t *con, double *v64, float *v32, double *dblk, int32_t *bad,
                    bool diff32) {
  if (m.n_nod == 0) return TFM_OK;
  const int rows_only = env_int("TFM_ASSEMBLE_ROWS", 0);
  TFM_DISPATCH_ALL(m, mat, {
    constexpr int NW = tile_nodes<ET>();
    const size_t tile_shm = (sizeof(double) * ND * ND + 1) * NW * (size_t)m.max_deg;
    if (node_tiled<MK>() && !rows_only && tile_shm <= 48 * 1024) {
      constexpr int MT = node_tiled<MK>() ? MK : TFM_MAT_ISO;
      const int64_t nb = (m.n_nod + NW - 1) / NW;
      hipLaunchKernelGGL((k_assemble_nodes<ET, ND, MT>), dim3((unsigned)nb), dim3(64), tile_shm,
                         s, m, mat, con, v64, v32, dblk, bad, (int)diff32);
      TFM_CHECK_LAUNCH();
      return TFM_OK;
    }
    // one node per block: the general stiffness, node degrees whose tile would
    // not fit in LDS, or TFM_ASSEMBLE_ROWS=1
    constexpr int KCH = assemble_chunk<ET>();
    const size_t shm = sizeof(double) * ND * ND * (size_t)m.max_deg + (size_t)KCH * m.max_deg;
    TFM_REQUIRE(shm <= 48 * 1024, "node degree too large for the assembly kernel");
    hipLaunchKernelGGL((k_assemble_rows<ET, ND, MK>), dim3((unsigned)m.n_nod), dim3(64), shm, s,
                       m, mat, con, v64, v32, dblk, bad, (int)diff32);
    TFM_CHECK_LAUNCH();
  });
  return TFM_OK;
}

int launch_internal_force(hipStream_t s, const tfm_mesh_t &m, const tfm_material_t &mat,
                          const double *u, const double *flux_prev, double *f,
                          double *grad_mean, double *flux_mean, double *grad_gp,
                          double *flux_gp, double *work) {
  TFM_DISPATCH_ALL(m, mat, {
    constexpr int EPB = point_elems<ET>();
    if (m.n_elem > 0) {
      const unsigned nb = (unsigned)((m.n_elem + EPB - 1) / EPB);
      hipLaunchKernelGGL((k_internal_force<ET, ND, MK>), dim3(nb), dim3(64), 0, s, m, mat, u,
                         flux_prev, work, grad_mean, flux_mean, grad_gp, flux_gp);
      TFM_CHECK_LAUNCH();
    }
    if (f) {
      const int64_t nt = m.n_nod * ND;
      hipLaunchKernelGGL((k_gather_nodes<ND>), dim3((unsigned)((nt + 255) / 256)), dim3(256), 0,
                         s, m, work, f);
      TFM_CHECK_LAUNCH();
    }
  });
  return TFM_OK;
}

int launch_element_matrices_gp(hipStream_t s, const tfm_mesh_t &m, const double *cgp,
                               const double *scale, double *k, int32_t *bad) {
  if (m.n_elem == 0) return TFM_OK;
  TFM_REQUIRE(m.ndof == m.dim, "a per-point tangent needs a mechanics mesh");
  TFM_DISPATCH(m.etype, {
    hipLaunchKernelGGL((k_element_matrices_gp<ET>), dim3((unsigned)m.n_elem), dim3(64), 0, s, m,
                       cgp, scale, k, bad);
    TFM_CHECK_LAUNCH();
  });
  return TFM_OK;
}

int launch_assemble_elements(hipStream_t s, const tfm_mesh_t &m, const double *k,
                             const uint8_t *con, double *v64, float *v32, double *dblk,
                             bool diff32) {
  if (m.n_nod == 0) return TFM_OK;
  const size_t slots = (size_t)m.max_inc * m.max_deg;
  TFM_REQUIRE(slots <= 48 * 1024, "node degree too large for the assembly kernel");
  TFM_REQUIRE(m.npe <= 127, "too many element nodes for the assembly kernel");
  auto any = [&](auto kernel) -> int {
    hipLaunchKernelGGL(kernel, dim3((unsigned)m.n_nod), dim3(64), slots, s, m, k, con, v64, v32,
                       dblk, (int)diff32);
    TFM_CHECK_LAUNCH();
    return TFM_OK;
  };
  auto go = [&](auto kernel, int nw, auto general, int nd) -> int {
    // per neighbour and node of the tile a block of values and a byte. A pattern
    // whose max_deg follows from its max_inc needs at most 112 KB under the bound
    // above (Tetra1, three DOFs, four nodes: 292 bytes times 384); a caller may
    // state a larger max_deg.
    const size_t shm = (sizeof(double) * nd * nd + 1) * nw * (size_t)m.max_deg;
    if (shm > 128 * 1024) return any(general);
    if (shm > 60 * 1024)
      TFM_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
    hipLaunchKernelGGL(kernel, dim3((unsigned)((m.n_nod + nw - 1) / nw)), dim3(64), shm, s, m, k,
                       con, v64, v32, dblk, (int)diff32);
    TFM_CHECK_LAUNCH();
    return TFM_OK;
  };
  auto by_npe = [&](auto ndof) -> int {
    constexpr int ND = decltype(ndof)::value;
    auto general = &k_assemble_elements_any<ND>;
    switch (m.npe) {
      case 4: return go(&k_assemble_elements<4, ND>, 64 / assemble_lanes(4, ND), general, ND);
      case 8: return go(&k_assemble_elements<8, ND>, 64 / assemble_lanes(8, ND), general, ND);
      case 20: return go(&k_assemble_elements<20, ND>, 64 / assemble_lanes(20, ND), general, ND);
      default: return any(general);
    }
  };
  switch (m.ndof) {
    case 1: return by_npe(std::integral_constant<int, 1>{});
    case 2: return by_npe(std::integral_constant<int, 2>{});
    case 3: return by_npe(std::integral_constant<int, 3>{});
    default: TFM_REQUIRE(false, "ndof must be 1, 2 or 3");
  }
}

int launch_gather(hipStream_t s, const tfm_mesh_t &m, const double *fe, double *F) {
  const int64_t nt = m.n_nod * m.ndof;
  if (nt == 0) return TFM_OK;
  const unsigned g = (unsigned)((nt + 255) / 256);
  switch (m.ndof) {
    case 1: hipLaunchKernelGGL(k_gather_nodes<1>, dim3(g), dim3(256), 0, s, m, fe, F); break;
    case 2: hipLaunchKernelGGL(k_gather_nodes<2>, dim3(g), dim3(256), 0, s, m, fe, F); break;
    case 3: hipLaunchKernelGGL(k_gather_nodes<3>, dim3(g), dim3(256), 0, s, m, fe, F); break;
    default: TFM_REQUIRE(false, "ndof must be 1, 2 or 3");
  }
  TFM_CHECK_LAUNCH();
  return TFM_OK;
}

int launch_sensitivity(hipStream_t s, const tfm_mesh_t &m, const tfm_material_t &mat,
                       const double *u, const double *lam, int nrhs, double sign, double *out) {
  if (m.n_elem == 0 || nrhs == 0) return TFM_OK;
  TFM_DISPATCH_ALL(m, mat, {
    auto go = [&](auto elems) {
      constexpr int EPB = decltype(elems)::value;
      const unsigned nb = (unsigned)((m.n_elem + EPB - 1) / EPB);
      hipLaunchKernelGGL((k_sensitivity<ET, ND, MK, EPB>), dim3(nb), dim3(64), 0, s, m, mat, u,
                         lam, nrhs, sign, out);
    };
    if constexpr (sens_outputs<ET, MK>()) {
      if (m.n_elem <= 4 * 256 * 16) go(std::integral_constant<int, 8>{});
      else go(std::integral_constant<int, 16>{});
    } else {
      go(std::integral_constant<int, point_elems<ET>()>{});
    }
    TFM_CHECK_LAUNCH();
  });
  return TFM_OK;
}

}  // namespace tfm
