// Implicit path of the BES solver core on MI355X (gfx950).
//
// One backward-Euler pseudo-time step (SolverImplicit.cpp:293-345):
//   k_timestep + k_gradlim          (explicit.hip)
//   k_face_jacobian   first-order flux Jacobians dF/dU_L, dF/dU_R per face by
//                     dual numbers with the reference's Eigen AD rules
//                     (FluxJacobianWrapper.tpp:32-82), one thread per (face,
//                     side), its nv derivatives sharing the values
//   k_assemble        row-owned assembly: second-order fluxes give the right-
//                     hand side b = -dt/V sum +-F*A; the block row gets
//                     I + sum nV x (dt/V*A*J) in the reference's accumulation
//                     order (SolverImplicit.cpp:358-507, CoefficientMatrix.cpp:
//                     166-204, the nV-fold repeat included).  No atomics.
//   GMRES(m)          right-preconditioned, classical Gram-Schmidt with DGKS
//                     re-orthogonalisation, deterministic two-pass reductions;
//                     replaces the reference's AMGCL solve (CoefficientMatrix.cpp:
//                     210-325) with relative tolerance semantics (||r|| <= tol*||b||)
//   preconditioners   block Jacobi, or block ILU(0) in a multicolour order
//                     (colours of the cell adjacency graph: every colour is
//                     one parallel sweep of the triangular solves)
//   k_update          U += x, the implicit update (SolverImplicit.cpp:509-528)
// Matrix layout ("ELL-BSR"): slot 0 = diagonal block, slot 1+m = the block of
// the neighbour through local face m; entries stored [slot][e][N] so a wave
// reads 64 consecutive rows of one entry in one coalesced load.  Matrix and
// Krylov vectors are FP64, or FP32 for the mixed-precision inner solve.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/bes_hip.h"
#include "context.hpp"
#include "flux.hpp"
#include "implicit.hpp"
#include "kernels_common.hpp"

namespace bes {

int launch_timestep(bes_ctx *c, const double *U, double cfl, int local, const double *cfl_b = nullptr);
int launch_face_flux(bes_ctx *c);
struct StageAux;   // explicit.hip
bool split_pass(const bes_ctx *c);
int launch_gradlim(bes_ctx *c, const double *U, double *Gout, double *Pout, const StageAux *aux = nullptr);
int launch_residual(bes_ctx *c, const double *U0, double *Ud, double alpha, int local, double *Rout,
                    unsigned long long *linf_bits);
int state_to_host(bes_ctx *c, const double *dsoa, int ncomp, double *host);
int state_to_device(bes_ctx *c, const double *host, int ncomp, double *dsoa);
int vector_to_host(bes_ctx *c, const double *dvec, double *host);
namespace lp {
int lp_build(bes_ctx *c, Impl *im);
int lp_release(Impl *im);
}  // namespace lp

// ---------------------------------------------------------------------------
// Jacobians
// ---------------------------------------------------------------------------
struct FinfI {
  double p[6];
};

// padded length of one Jacobian block record: nv*nv entries rounded up to 16 bytes
template <typename TJ, int NB>
struct JRec {
  static constexpr int P = (NB * (int)sizeof(TJ) + 15) / 16 * 16 / (int)sizeof(TJ);
};

// Both blocks of a face, a thread per side (and condition).  Bound by FP64
// arithmetic: the values' divisions and square roots, which a thread per input
// column repeated for each of the 2 nv columns, and then the derivatives, whose
// registers leave one wave per SIMD in 3D (346; capped at 256 it spills: 2042 us).
// 4M faces FP64 1820 -> 1294 us, 64k faces x 16 conditions FP32 444 -> 258, 60k
// triangle faces 26 -> 14; two columns to a thread 1536 and 328.
template <int ND, typename TJ>
__global__ __launch_bounds__(256) void k_face_jacobian(const double *__restrict__ U, int N, FaceDev fd,
                                                       GasConst gc, const double *__restrict__ finf,
                                                       TJ *__restrict__ JF, int lgB) {
  constexpr int NV = ND + 2, NB = NV * NV, JP = JRec<TJ, NB>::P;
  using D = DualN<NV>;
  // groups of 64 lanes x 2 sides: the lanes of a wave take 64/B consecutive faces
  // x B conditions and all nv derivatives to one side, which share the values'
  // arithmetic; a face's two blocks sit side by side in one record [2][JP] (JL,
  // then JR, row-major), entry e of condition b at (rec + e)*B + b
  const int B = 1 << lgB;
  const int t = xcd_block() * blockDim.x + threadIdx.x;
  const bool right = __builtin_amdgcn_readfirstlane((t >> 6) & 1);
  const int l = t & 63;
  const int f = (t >> 7) * (64 >> lgB) + (l >> lgB), b = l & (B - 1);
  if (f >= fd.F) return;
  const int o = fd.fo[f], j = fd.fn[f];
  if (j < 0 && right) return;   // boundary faces: left Jacobian only
  double nn[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) nn[d] = fd.fnrm[(size_t)d * fd.F + f];
  D F[NV];
  double xl[NV], xr[NV + 1];
#pragma unroll
  for (int v = 0; v < NV; v++) xl[v] = U[((size_t)v * N + o) * B + b];
  if (j >= 0) {
#pragma unroll
    for (int v = 0; v < NV; v++) xr[v] = U[((size_t)v * N + j) * B + b];
  }
  D u[NV];   // the state differentiated by: its value's derivatives are the unit vectors
#pragma unroll
  for (int v = 0; v < NV; v++)
    u[v] = D::make(right ? xr[v] : xl[v], [&](int k) { return k == v ? 1.0 : 0.0; });
  if (j >= 0) {
    if (right) roe_flux<ND, double, D>(gc, xl, u, nn, F);
    else roe_flux<ND, D, double>(gc, u, xr, nn, F);
  } else if (j == -1) {
    slip_flux<ND, D>(gc, u, nn, F);
  } else {
    D ui[NV + 1];
#pragma unroll
    for (int v = 0; v < NV + 1; v++) ui[v] = D(finf[b * (NV + 1) + v]);
    freestream_flux<ND, D>(gc, u, ui, nn, F);
  }
  TJ *rec = JF + ((size_t)f * 2 + right) * JP * B;
  if (lgB == 0) {   // 16-byte stores of the record
    constexpr int W = 16 / (int)sizeof(TJ);
    TJ out[JP];
#pragma unroll
    for (int e = 0; e < JP; e++) out[e] = e < NB ? (TJ)F[e < NB ? e / NV : 0].d[e < NB ? e % NV : 0] : (TJ)0;
#pragma unroll
    for (int q = 0; q < JP / W; q++) {
      uint4 w;
      __builtin_memcpy(&w, out + q * W, 16);
      reinterpret_cast<uint4 *>(rec)[q] = w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < NB; e++) rec[(size_t)e * B + b] = (TJ)F[e / NV].d[e % NV];
  }
}

// one padded block record (16-byte aligned, JP entries) into registers as doubles
template <typename TJ, int NB>
__device__ __forceinline__ void load_rec(const TJ *__restrict__ rec, double *out) {
  constexpr int JP = JRec<TJ, NB>::P, W = 16 / (int)sizeof(TJ);
  TJ tmp[JP];
#pragma unroll
  for (int q = 0; q < JP / W; q++) {
    const uint4 u = reinterpret_cast<const uint4 *>(rec)[q];
    __builtin_memcpy(tmp + q * W, &u, 16);
  }
#pragma unroll
  for (int e = 0; e < NB; e++) out[e] = (double)tmp[e];
}

// ---------------------------------------------------------------------------
// assembly: right-hand side from second-order fluxes, blocks from JF
// ---------------------------------------------------------------------------
template <int ND, typename TM>
__global__ __launch_bounds__(256) void k_assemble(
    const double *__restrict__ FF, int fs, const double *__restrict__ dt, const double *__restrict__ dtg, DevMesh dm,
    FaceDev fd, const TM *__restrict__ JF, int repeat, double *__restrict__ b, TM *__restrict__ A,
    unsigned long long *__restrict__ linf_b, unsigned long long *__restrict__ linf_r, int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV, JP = JRec<TM, NB>::P;
  const int N = dm.N, B = 1 << lgB;
  const int t = cell_index();
  const int i = t >> lgB, bq = t & (B - 1);
  double bi[NV], ri[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) { bi[v] = 0.0; ri[v] = 0.0; }
  if (i < N) {
    const double mdt = (dtg ? dtg[bq] : dt[(size_t)i * B + bq]) / dm.vol[i];
    const uint32_t info = dm.info[i];
    // right-hand side (SolverImplicit.cpp:441-473) from the second-order face
    // fluxes of k_face_flux, faces in reference order
#pragma unroll
    for (int q = 0; q < K; q++) {
      const int m = (info >> (2 * q)) & 3;
      const bool own = (info >> (8 + m)) & 1;
      const int fdv = dm.cfd[(size_t)m * N + i];
      const double Af = dm.af[(size_t)m * N + i];
      const double mul = mdt * Af;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const double F = FF[((size_t)fdv * fs + v) * B + bq];
        if (own) { bi[v] -= mul * F; ri[v] += F * Af; }
        else { bi[v] += mdt * Af * F; ri[v] -= F * Af; }
      }
    }
#pragma unroll
    for (int v = 0; v < NV; v++) b[((size_t)i * NV + v) * B + bq] = bi[v];
    // blocks: identity, then per face (reference order) the repeated adds.
    // own row: diag += mul*JL, off(i,nbr) = mul*JR; neighbour row:
    // diag += (-m)*JR, off(i,owner) = (-m)*JL.  The diagonal sums in the
    // reference's face order; each off-diagonal block depends on its own face
    // only, so those are written in a second loop in slot order, where every
    // lane of a wave stores into the same slot's planes (whole cache lines;
    // in face order the lanes' slots differ and lines leave L2 part-written).
    double D[NB];
#pragma unroll
    for (int e = 0; e < NB; e++) D[e] = 0.0;
#pragma unroll
    for (int a = 0; a < NV; a++) D[a * NV + a] += 1.0;
    for (int q = 0; q < K; q++) {
      const int m = (info >> (2 * q)) & 3;
      const bool own = (info >> (8 + m)) & 1;
      const int f = fd.cf[(size_t)m * N + i];
      const double Af = dm.af[(size_t)m * N + i];
      const double mul = own ? mdt * Af : -(mdt * Af);
      double J[NB];
      const TM *Jd = JF + ((size_t)f * 2 + (own ? 0 : 1)) * JP * B;
      if (B == 1) load_rec<TM, NB>(Jd, J);
      else {
#pragma unroll
        for (int e = 0; e < NB; e++) J[e] = (double)Jd[(size_t)e * B + bq];
      }
#pragma unroll
      for (int e = 0; e < NB; e++) {
        const double x = mul * J[e];
        for (int r = 0; r < repeat; r++) D[e] += x;
      }
    }
#pragma unroll
    for (int m = 0; m < K; m++) {
      const bool own = (info >> (8 + m)) & 1;
      const int j = dm.nbr[(size_t)m * N + i];
      const int f = fd.cf[(size_t)m * N + i];
      const double Af = dm.af[(size_t)m * N + i];
      const double mul = own ? mdt * Af : -(mdt * Af);
      double J[NB];
      TM *Ao = A + (size_t)(1 + m) * NB * N * B;
      if (j >= 0) {
        const TM *Jo = JF + ((size_t)f * 2 + (own ? 1 : 0)) * JP * B;
        if (B == 1) load_rec<TM, NB>(Jo, J);
        else {
#pragma unroll
          for (int e = 0; e < NB; e++) J[e] = (double)Jo[(size_t)e * B + bq];
        }
#pragma unroll
        for (int e = 0; e < NB; e++) {
          const double x = mul * J[e];
          double s = 0.0;
          for (int r = 0; r < repeat; r++) s += x;
          Ao[((size_t)e * N + i) * B + bq] = (TM)s;
        }
      } else {
#pragma unroll
        for (int e = 0; e < NB; e++) Ao[((size_t)e * N + i) * B + bq] = (TM)0;
      }
    }
#pragma unroll
    for (int e = 0; e < NB; e++) A[((size_t)e * N + i) * B + bq] = (TM)D[e];
  }
  if (linf_b) {   // per condition: [v][B]
#pragma unroll
    for (int v = 0; v < NV; v++) {
      double a = block_max_cond(::fabs(bi[v]), B);
      if ((int)threadIdx.x < B)
        atomicMax(&linf_slot(linf_b, 16 * B)[v * B + threadIdx.x], (unsigned long long)__double_as_longlong(a));
      double c = block_max_cond(::fabs(ri[v]), B);
      if ((int)threadIdx.x < B)
        atomicMax(&linf_slot(linf_r, 16 * B)[v * B + threadIdx.x], (unsigned long long)__double_as_longlong(c));
    }
  }
}

// block Jacobi: LU slot 0 <- inverse of the diagonal block
template <int ND, typename TM>
__global__ __launch_bounds__(256) void k_bj_setup(const TM *__restrict__ A, TM *__restrict__ LU, int N, int lgB) {
  constexpr int NV = ND + 2, NB = NV * NV;
  const int B = 1 << lgB, t = cell_index();
  const int i = t >> lgB, b = t & (B - 1);
  if (i >= N) return;
  double D[NB], Inv[NB];
  load_block_b<TM, NB>(A, 0, N, i, B, b, D);
  block_inverse<NV>(D, Inv);
  store_block_b<TM, NB>(LU, 0, N, i, B, b, Inv);
}

// colour-major copy of the matrix: Ac[se][cpos[i]] = A[se][i], se = slot*nv^2 + e.
// One thread per (cell, condition) copies all nse planes: its reads are
// coalesced, and since the cells of each row group of a colour keep their
// order, the lanes' stores land in a few runs of consecutive positions.  On
// the 2M wing it fetches the matrix once and writes 1.28x it; gathering in
// position order instead read a few entries of each line and fetched 5.7x.
template <typename TM>
__global__ __launch_bounds__(256) void k_ilu_scatter(const TM *__restrict__ A, const int *__restrict__ cpos, int N,
                                                     int nse, TM *__restrict__ Ac, int lgB) {
  const size_t B = (size_t)1 << lgB;
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (size_t)N * B) return;
  const size_t i = q >> lgB, b = q & (B - 1), p = (size_t)cpos[i];
#pragma unroll 5
  for (int se = 0; se < nse; se++) Ac[((size_t)se * N + p) * B + b] = A[((size_t)se * N + i) * B + b];
}

// y = A x with matrix and vectors in colour order (neighbour positions cnp), B conditions
template <int ND, typename TM, typename TV>
__global__ __launch_bounds__(256) void k_spmv_pos(const TM *__restrict__ A, const int *__restrict__ cnp, int N,
                                                  const TV *__restrict__ x, TV *__restrict__ y, int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV;
  const int B = 1 << lgB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int p = t >> lgB, b = t & (B - 1);
  if (p >= N) return;
  // block entries from the row's first entry with the uniform stride es (a
  // full index per entry costs a 64-bit register pair per load in flight)
  const size_t es = (size_t)N * B;
  const TM *Ar = A + (size_t)p * B + b;
  double acc[NV], xv[NV];
#pragma unroll
  for (int c = 0; c < NV; c++) xv[c] = (double)x[((size_t)p * NV + c) * B + b];
#pragma unroll
  for (int r = 0; r < NV; r++) {
    double s = 0;
#pragma unroll
    for (int c = 0; c < NV; c++) s += (double)Ar[(r * NV + c) * es] * xv[c];
    acc[r] = s;
  }
#pragma unroll
  for (int m = 0; m < K; m++) {
    const int q = cnp[(size_t)m * N + p];
    if (q < 0) continue;
#pragma unroll
    for (int c = 0; c < NV; c++) xv[c] = (double)x[((size_t)q * NV + c) * B + b];
    const TM *Ao = Ar + (size_t)(1 + m) * NB * es;
#pragma unroll
    for (int r = 0; r < NV; r++) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < NV; c++) s += (double)Ao[(r * NV + c) * es] * xv[c];
      acc[r] += s;
    }
  }
#pragma unroll
  for (int r = 0; r < NV; r++) y[((size_t)p * NV + r) * B + b] = (TV)acc[r];
}

// y = A x as k_spmv / k_spmv_pos with a thread per (block of a row, cell,
// condition): wave w of a block takes slot w (0 the diagonal, w the neighbour
// w - 1; 1 + K = NV of them) of the block's 64 units u = cell*B + condition, then
// component w of their sums, the products added in slot order.  An absent
// neighbour adds -0.0, which changes nothing.
// Bound by memory latency where a thread per cell is too few waves (its four
// gathers follow one another) and by the last-level cache above: per product 31k
// tetrahedra FP64 11.7 -> 7.0 us, 83k 20.4 -> 16, 249k 61.6 -> 55.1 (FP32 32.6 ->
// 28.7), 590k 138 -> 127; 12.8k triangles 7.1 -> 4.3, 490k 60.9 -> 54.2.  (A
// thread per row of the block repeats the gathers in every row: 18.6, 81.5, 190.)
template <int ND, typename TM, typename TV>
__device__ __forceinline__ void block_product(const TM *__restrict__ Am, size_t es, const TV *__restrict__ xs, int lgB,
                                              double s[ND + 2]) {
  constexpr int NV = ND + 2;
  TV xv[NV];
  TM av[NV][NV];
#pragma unroll
  for (int c = 0; c < NV; c++) xv[c] = xs[(size_t)c << lgB];
#pragma unroll
  for (int r = 0; r < NV; r++)
#pragma unroll
    for (int c = 0; c < NV; c++) av[r][c] = Am[(size_t)(r * NV + c) * es];
#pragma unroll
  for (int r = 0; r < NV; r++) {
    double t = 0;
#pragma unroll
    for (int c = 0; c < NV; c++) t += to_d(av[r][c]) * (double)xv[c];
    s[r] = t;
  }
}

template <int ND, typename TM, typename TV>
__global__ __launch_bounds__(64 * (ND + 2)) void k_spmv_slots(const TM *__restrict__ A, const int *__restrict__ nbr,
                                                              int N, const TV *__restrict__ x, TV *__restrict__ y,
                                                              int lgB) {
  constexpr int NV = ND + 2, NB = NV * NV;
  __shared__ double sh[NV][NV][64];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & 63;
  const int u = blockIdx.x * 64 + t;
  const int p = u >> lgB, b = u & ((1 << lgB) - 1);
  const size_t es = (size_t)N << lgB;
  double s[NV];
#pragma unroll
  for (int r = 0; r < NV; r++) s[r] = -0.0;
  if (p < N) {
    const int q = w == 0 ? p : nbr[(size_t)(w - 1) * N + p];
    if (q >= 0)
      block_product<ND, TM, TV>(A + (size_t)w * NB * es + u, es, x + (((size_t)q * NV) << lgB) + b, lgB, s);
  }
#pragma unroll
  for (int r = 0; r < NV; r++) sh[w][r][t] = s[r];
  __syncthreads();
  if (p >= N) return;
  double acc = sh[0][w][t];
#pragma unroll
  for (int m = 1; m < NV; m++) acc += sh[m][w][t];
  y[(((size_t)p * NV + w) << lgB) + b] = (TV)acc;
}

// rows between cell order and colour order (each row nv*B contiguous values):
// to_colour: dst[p] = src[crow[p]], else dst[crow[p]] = src[p]
template <typename T>
__global__ void k_perm_rows(const T *__restrict__ src, const int *__restrict__ crow, int N, int rw, int to_colour,
                            T *__restrict__ dst) {
  const size_t tot = (size_t)N * rw;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < tot; q += (size_t)gridDim.x * blockDim.x) {
    const size_t p = q / rw, c = q - p * rw;
    const size_t i = (size_t)crow[p];
    if (to_colour) dst[q] = src[i * rw + c];
    else dst[i * rw + c] = src[q];
  }
}

// block ILU(0) of the rows at positions p0 .. p0+nrows-1 (one colour); rows of
// earlier colours are final.  Elimination order: colour, then cell index (not
// position, so the factors do not depend on how rows are laid out in a colour).
// A row's thread first copies its blocks from the colour-order matrix Ac into
// LU (only that thread ever touches the row), eliminates, and leaves slot 0 =
// inv(U_ii), lower slots L_ik, upper slots U_ij.  Finished rows are also kept
// row-major by position (Dr: inv(U_pp); Ur: upper blocks by slot), so a later
// row reads a neighbour's block as one contiguous record.
template <int ND, typename TM>
__global__ __launch_bounds__(256) void k_ilu_factor_color(const TM *__restrict__ Ac, TM *__restrict__ LU, int N,
                                                          const int *__restrict__ cnb, const int *__restrict__ cnp,
                                                          const unsigned char *__restrict__ clow,
                                                          const int *__restrict__ color, const int *__restrict__ crow,
                                                          TM *__restrict__ Dr, TM *__restrict__ Ur, int p0, int nrows,
                                                          int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV;
  const int B = 1 << lgB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nrows << lgB)) return;
  const int p = p0 + (t >> lgB), b = t & (B - 1);
  const int i = crow[p];
  const unsigned lowm = clow[p];
  int nb[K], np_[K];
#pragma unroll
  for (int m = 0; m < K; m++) {
    nb[m] = cnb[(size_t)m * N + p];
    np_[m] = cnp[(size_t)m * N + p];
  }
  // the row's own blocks into the factor storage (boundary slots stay zero),
  // a block at a time (unrolled over the slots, the compiler would hold all
  // 125 entries in registers between the loads and the stores)
#pragma unroll 1
  for (int sl = 0; sl <= K; sl++) {
    if (sl > 0 && nb[sl - 1] < 0) continue;
#pragma unroll
    for (int e = 0; e < NB; e++) {
      const size_t q = (((size_t)sl * NB + e) * N + p) * B + b;
      LU[q] = Ac[q];
    }
  }
  // lower neighbours in elimination order (colour, then cell index)
  int ord[K], okey[K];
  int nl = 0;
#pragma unroll
  for (int m = 0; m < K; m++)
    if ((lowm >> m) & 1) {
      okey[nl] = color[nb[m]];
      ord[nl++] = m;
    }
  for (int a = 1; a < nl; a++)
    for (int bq = a; bq > 0; bq--) {
      const int x = ord[bq - 1], y = ord[bq];
      const int kx = okey[bq - 1], ky = okey[bq];
      if (kx > ky || (kx == ky && nb[x] > nb[y])) {
        ord[bq - 1] = y; ord[bq] = x;
        okey[bq - 1] = ky; okey[bq] = kx;
      }
    }
  double Aii[NB];
  load_block_b<TM, NB>(LU, 0, N, p, B, b, Aii);
  const size_t es = (size_t)N * B;   // stride between a block's entries
  // Each product below sums over pp in the same order as a whole-block
  // product would; they are arranged so that few values are live at once (one
  // row of A_ik, one column of U_kj), which keeps the kernel at two waves per
  // SIMD instead of one.
  for (int q = 0; q < nl; q++) {
    const int m = ord[q];
    const int pk = np_[m];
    double Lik[NB];
    {
      // row k is final: inv(U_kk), from the row-major copy (one contiguous block)
      double Uinv[NB];
#pragma unroll
      for (int e = 0; e < NB; e++) Uinv[e] = (double)Dr[((size_t)pk * NB + e) * B + b];
      // (entries addressed from a per-row base with a uniform stride: computing
      // each entry's full index costs a 64-bit register pair per load in flight)
      const TM *aik = LU + ((size_t)(1 + m) * NB * N + p) * B + b;
#pragma unroll
      for (int r = 0; r < NV; r++) {
        double ar[NV];   // row r of A_ik
#pragma unroll
        for (int pp = 0; pp < NV; pp++) ar[pp] = (double)aik[(r * NV + pp) * es];
#pragma unroll
        for (int c = 0; c < NV; c++) {
          double s = 0;
#pragma unroll
          for (int pp = 0; pp < NV; pp++) s += ar[pp] * Uinv[pp * NV + c];
          Lik[r * NV + c] = s;
        }
      }
    }
    store_block_b<TM, NB>(LU, 1 + m, N, p, B, b, Lik);
    // A_ij -= L_ik U_kj for j in row k's upper part that are in row i's pattern
    // (one j at a time: unrolled, the U_kj loads of all j would be in flight)
    const unsigned lowk = clow[pk];
#pragma unroll 1
    for (int mk = 0; mk < K; mk++) {
      const int jk = cnb[(size_t)mk * N + pk];
      if (jk < 0 || ((lowk >> mk) & 1)) continue;   // not upper in row k
      int target = -1;   // -2 = diagonal of row i
      if (jk == i) target = -2;
      else {
#pragma unroll
        for (int mm = 0; mm < K; mm++) if (nb[mm] == jk) target = mm;
      }
      if (target == -1) continue;
      const TM *urec = Ur + ((size_t)pk * K + mk) * NB * B + b;
#pragma unroll
      for (int c = 0; c < NV; c++) {
        double uc[NV];   // column c of U_kj
#pragma unroll
        for (int pp = 0; pp < NV; pp++) uc[pp] = (double)urec[(size_t)(pp * NV + c) * B];
#pragma unroll
        for (int r = 0; r < NV; r++) {
          double s = 0;
#pragma unroll
          for (int pp = 0; pp < NV; pp++) s += Lik[r * NV + pp] * uc[pp];
          if (target == -2) {
            Aii[r * NV + c] -= s;
          } else {
            TM *aij = LU + ((size_t)(1 + target) * NB * N + p) * B + b + (r * NV + c) * es;
            *aij = (TM)((double)*aij - s);
          }
        }
      }
    }
  }
  double Inv[NB];
  block_inverse<NV>(Aii, Inv);
  store_block_b<TM, NB>(LU, 0, N, p, B, b, Inv);
#pragma unroll
  for (int e = 0; e < NB; e++) Dr[((size_t)p * NB + e) * B + b] = (TM)Inv[e];
  // upper blocks, final from here on, row-major for the rows of later colours
  // (a block at a time, as the copy above)
#pragma unroll 1
  for (int m = 0; m < K; m++) {
    if (nb[m] < 0 || ((lowm >> m) & 1)) continue;
#pragma unroll
    for (int e = 0; e < NB; e++)
      Ur[(((size_t)p * K + m) * NB + e) * B + b] = LU[(((size_t)(1 + m) * NB + e) * N + p) * B + b];
  }
}

// forward sweep of one colour (vectors in colour order): y_p = r_p - sum_(k lower) L_pk y_k.
// Rows of colour 0 have no lower neighbours, so y = r there and is never stored:
// positions below y0end read r. With FUSE (the last colour, which has no upper
// neighbours) the backward step x_p = inv(U_pp) y_p follows at once, y_p rounded
// to TV as a store and reload would round it.
template <int ND, typename TM, typename TV, bool FUSE>
__global__ __launch_bounds__(256) void k_ilu_lower(const TM *__restrict__ LU, int N, const int *__restrict__ cnp,
                                                   const unsigned char *__restrict__ clow, int p0, int nrows,
                                                   const TV *__restrict__ r, TV *__restrict__ y, int y0end,
                                                   TV *__restrict__ x, int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV;
  const int B = 1 << lgB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nrows << lgB)) return;
  const int p = p0 + (t >> lgB), b = t & (B - 1);
  const unsigned lowm = clow[p];
  const size_t es = (size_t)N * B;   // stride between a block's entries
  const TM *Lr = LU + (size_t)p * B + b;
  double acc[NV];
#pragma unroll
  for (int c = 0; c < NV; c++) acc[c] = (double)r[((size_t)p * NV + c) * B + b];
#pragma unroll
  for (int m = 0; m < K; m++) {
    if (!((lowm >> m) & 1)) continue;
    const int q = cnp[(size_t)m * N + p];
    const TV *src = q < y0end ? r : y;
    double yk[NV];
#pragma unroll
    for (int c = 0; c < NV; c++) yk[c] = (double)src[((size_t)q * NV + c) * B + b];
    const TM *L = Lr + (size_t)(1 + m) * NB * es;
#pragma unroll
    for (int a = 0; a < NV; a++) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < NV; c++) s += (double)L[(a * NV + c) * es] * yk[c];
      acc[a] -= s;
    }
  }
  if constexpr (FUSE) {
#pragma unroll
    for (int c = 0; c < NV; c++) acc[c] = (double)(TV)acc[c];
#pragma unroll
    for (int a = 0; a < NV; a++) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < NV; c++) s += (double)Lr[(a * NV + c) * es] * acc[c];
      x[((size_t)p * NV + a) * B + b] = (TV)s;
    }
  } else {
#pragma unroll
    for (int c = 0; c < NV; c++) y[((size_t)p * NV + c) * B + b] = (TV)acc[c];
  }
}

// backward sweep of one colour (vectors in colour order): x_p = inv(U_pp) (y_p - sum_(j upper) U_pj x_j);
// y_p is r_p below y0end (colour 0)
template <int ND, typename TM, typename TV>
__global__ __launch_bounds__(256) void k_ilu_upper(const TM *__restrict__ LU, int N, const int *__restrict__ cnp,
                                                   const unsigned char *__restrict__ clow, int p0, int nrows,
                                                   const TV *__restrict__ y, TV *__restrict__ x,
                                                   const TV *__restrict__ r, int y0end, int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV;
  const int B = 1 << lgB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nrows << lgB)) return;
  const int p = p0 + (t >> lgB), b = t & (B - 1);
  const unsigned lowm = clow[p];
  const TV *own = p < y0end ? r : y;
  const size_t es = (size_t)N * B;   // stride between a block's entries
  const TM *Lr = LU + (size_t)p * B + b;
  double acc[NV];
#pragma unroll
  for (int c = 0; c < NV; c++) acc[c] = (double)own[((size_t)p * NV + c) * B + b];
#pragma unroll
  for (int m = 0; m < K; m++) {
    const int q = cnp[(size_t)m * N + p];
    if (q < 0 || ((lowm >> m) & 1)) continue;
    double xj[NV];
#pragma unroll
    for (int c = 0; c < NV; c++) xj[c] = (double)x[((size_t)q * NV + c) * B + b];
    const TM *Uo = Lr + (size_t)(1 + m) * NB * es;
#pragma unroll
    for (int a = 0; a < NV; a++) {
      double s = 0;
#pragma unroll
      for (int c = 0; c < NV; c++) s += (double)Uo[(a * NV + c) * es] * xj[c];
      acc[a] -= s;
    }
  }
#pragma unroll
  for (int a = 0; a < NV; a++) {
    double s = 0;
#pragma unroll
    for (int c = 0; c < NV; c++) s += (double)Lr[(a * NV + c) * es] * acc[c];
    x[((size_t)p * NV + a) * B + b] = (TV)s;
  }
}

// The sweeps as k_ilu_lower / k_ilu_upper with a thread per (neighbour, row p,
// condition): wave m of a block takes neighbour m of the block's 64 units (the
// last wave has none), then component m of their rows, the products subtracted in
// the order of the neighbours; one not in the sweep subtracts 0.0, which changes
// nothing.  INV: the product with inv(U_pp), whose factor is rounded to TV first
// in the forward sweep.
// Bound as k_spmv_slots; a colour is a third of the mesh, so it pays further up:
// backward, a colour of 29k tetrahedra FP64 8.9 -> 5.3 us, 80k 12.8 -> 8.8, 240k
// 29.2 -> 26.1; forward 9.0 -> 6.6, 22.3 -> 19.7, 43.8 -> 45.8; 15k triangles
// forward 6.3 -> 4.0, backward 5.8 -> 4.1.
template <int ND, typename TM, typename TV, bool UPPER, bool INV>
__global__ __launch_bounds__(64 * (ND + 2)) void k_ilu_slots(const TM *__restrict__ LU, int N,
                                                             const int *__restrict__ cnp,
                                                             const unsigned char *__restrict__ clow, int p0, int nrows,
                                                             const TV *__restrict__ r, const TV *y, int y0end,
                                                             const TV *x, TV *out, int lgB) {
  constexpr int NV = ND + 2, K = ND + 1, NB = NV * NV;
  __shared__ double sh[K][NV][64];
  __shared__ double sa[INV ? NV : 1][64];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & 63;
  const int u = blockIdx.x * 64 + t;
  const bool ok = u < (nrows << lgB);
  const int p = p0 + (u >> lgB), b = u & ((1 << lgB) - 1);
  const size_t es = (size_t)N << lgB, at = (((size_t)p * NV + w) << lgB) + b;
  const TM *Lr = LU + ((size_t)p << lgB) + b;
  TV own = 0;
  TM d[INV ? NV : 1];
  if (ok) {
    own = (UPPER && p >= y0end ? y : r)[at];
    if constexpr (INV)
#pragma unroll
      for (int c = 0; c < NV; c++) d[c] = Lr[(size_t)(w * NV + c) * es];
  }
  if (w < K) {
    double s[NV];
#pragma unroll
    for (int c = 0; c < NV; c++) s[c] = 0.0;
    if (ok) {
      const int q = cnp[(size_t)w * N + p];
      const bool low = (clow[p] >> w) & 1;
      if (UPPER ? q >= 0 && !low : low) {
        const TV *src = UPPER ? x : (q < y0end ? r : y);
        block_product<ND, TM, TV>(Lr + (size_t)(1 + w) * NB * es, es, src + (((size_t)q * NV) << lgB) + b, lgB, s);
      }
    }
#pragma unroll
    for (int c = 0; c < NV; c++) sh[w][c][t] = s[c];
  }
  __syncthreads();
  double acc = (double)own;
#pragma unroll
  for (int m = 0; m < K; m++) acc -= sh[m][w][t];
  if constexpr (INV) {
    sa[w][t] = UPPER ? acc : (double)(TV)acc;
    __syncthreads();
    if (!ok) return;
    double s = 0;
#pragma unroll
    for (int c = 0; c < NV; c++) s += (double)d[c] * sa[c][t];
    out[at] = (TV)s;
  } else {
    if (ok) out[at] = (TV)acc;
  }
}

// ---------------------------------------------------------------------------
// Krylov kernels (vectors [N][nv][B], type TV)
// ---------------------------------------------------------------------------
// z = inv(D_i) r_i (block Jacobi)
template <int ND, typename TM, typename TV>
__global__ __launch_bounds__(256) void k_bj_apply(const TM *__restrict__ LU, int N, const TV *__restrict__ r,
                                                  TV *__restrict__ z, int lgB) {
  constexpr int NV = ND + 2;
  const int B = 1 << lgB, t = cell_index();
  const int i = t >> lgB, b = t & (B - 1);
  if (i >= N) return;
  double ri[NV];
#pragma unroll
  for (int c = 0; c < NV; c++) ri[c] = (double)r[((size_t)i * NV + c) * B + b];
#pragma unroll
  for (int a = 0; a < NV; a++) {
    double s = 0;
#pragma unroll
    for (int c = 0; c < NV; c++) s += (double)LU[((size_t)(a * NV + c) * N + i) * B + b] * ri[c];
    z[((size_t)i * NV + a) * B + b] = (TV)s;
  }
}

// 16-byte packets of Krylov vectors (4 floats or 2 doubles); vectors start on
// 64-element boundaries (Impl::vstride), so packet loads are aligned
template <typename T>
struct Pk {
  static constexpr int W = 16 / sizeof(T);
  T v[16 / sizeof(T)];
};
template <typename T>
__device__ __forceinline__ Pk<T> ldp(const T *p) {
  Pk<T> r;
  const uint4 u = *reinterpret_cast<const uint4 *>(p);
  __builtin_memcpy(r.v, &u, 16);
  return r;
}
template <typename T>
__device__ __forceinline__ void stp(T *p, const Pk<T> &r) {
  uint4 u;
  __builtin_memcpy(&u, r.v, 16);
  *reinterpret_cast<uint4 *>(p) = u;
}

__device__ __forceinline__ void block_store_sums(const double *acc, int nq, double *part) {
  __shared__ double sh[9][4];
  for (int q = 0; q < nq; q++) {
    const double s = wave_sum(acc[q]);
    if ((threadIdx.x & 63) == 0) sh[q][threadIdx.x >> 6] = s;
  }
  __syncthreads();
  if ((int)threadIdx.x < nq) {
    const int q = threadIdx.x;
    part[(size_t)q * gridDim.x + blockIdx.x] = sh[q][0] + sh[q][1] + sh[q][2] + sh[q][3];
  }
}

// Deterministic reductions over a batch of B conditions (vectors [n1][B],
// condition fastest).  Every condition's n1 elements are summed in one fixed
// tree whatever B is, so a condition's dot products, norms and hence its whole
// Krylov solve are the same bits in a batch as alone: lane l of L (L depends
// on n1 only) adds, in order, the elements of the groups g = l, l + L, l + 2L,
// ..., group g being elements 4g .. 4g + 3 (zeros past n1); the L lane sums of
// a condition are then added by sum_lanes in a fixed two-level tree.  Thread
// l*B + b is lane l of condition b, so the loads of a wave are contiguous for
// any B, and one 16-byte packet (FP32) or two (FP64) per vector when B = 1.
constexpr int kLaneGroup = 4;

template <typename TV>
__device__ __forceinline__ void ld_group(const TV *__restrict__ v, size_t e, size_t n1, int lgB, int b,
                                         double x[kLaneGroup]) {
  if (lgB == 0 && e + kLaneGroup <= n1) {
    if (sizeof(TV) == 8) {
      const double2 a = *reinterpret_cast<const double2 *>(v + e);
      const double2 c = *reinterpret_cast<const double2 *>(v + e + 2);
      x[0] = a.x; x[1] = a.y; x[2] = c.x; x[3] = c.y;
    } else {
      const float4 a = *reinterpret_cast<const float4 *>(v + e);
      x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    }
  } else {
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++) x[h] = e + h < n1 ? (double)v[((e + h) << lgB) + b] : 0.0;
  }
}

template <typename TV>
__device__ __forceinline__ void st_group(TV *__restrict__ v, size_t e, size_t n1, int lgB, int b,
                                         const TV r[kLaneGroup]) {
  if (lgB == 0 && e + kLaneGroup <= n1) {
    if (sizeof(TV) == 8) {
      *reinterpret_cast<double2 *>(v + e) = make_double2((double)r[0], (double)r[1]);
      *reinterpret_cast<double2 *>(v + e + 2) = make_double2((double)r[2], (double)r[3]);
    } else {
      *reinterpret_cast<float4 *>(v + e) = make_float4((float)r[0], (float)r[1], (float)r[2], (float)r[3]);
    }
  } else {
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++)
      if (e + h < n1) v[((e + h) << lgB) + b] = r[h];
  }
}

// Rows of the reduced values in the dots buffer (B conditions each): the dot
// products of the first Gram-Schmidt pass from row 0 and of the second from row
// kDots2, product q at 9*(q/8) + q%8 with ||w||^2 at row 8 of each; ||w||^2
// after the update the step ends with, and after its first pass; on the host,
// whether the second pass was taken (1.0 or 0.0).
constexpr int kDots2 = 48, kDotNorm = 40, kDotNorm1 = 41, kDotSecond = 42, kDotRows = 96;
__host__ __device__ constexpr int dot_row(int q) { return 9 * (q / 8) + q % 8; }

// DGKS: condition b takes a second pass when the first left less than eta of
// ||w||.  The kernels of that pass look this up themselves (Gate), so the host
// queues them without waiting for the norms; with no condition in need every
// block returns at once.
struct Gate {
  double eta = 0.0;              // 0: not a second pass
  const double *dots = nullptr;
  __device__ __forceinline__ bool second(int b, int B) const {
    return sqrt(dots[kDotNorm1 * B + b]) < eta * sqrt(dots[8 * B + b]);
  }
  // every thread of the block must call it
  __device__ __forceinline__ bool closed(int B) const {
    return eta > 0.0 && !__syncthreads_or((int)threadIdx.x < B && second(threadIdx.x, B));
  }
};

// Level 1 of the lane sums adds lanes x*1024 + t + 256k, k = 0..3 in order, for
// each t < 256, then the 64 values of each wave by the shuffle tree: four
// partial sums per group of 1024 lanes, which level 2 adds in order.  One
// condition's kernels give a block of 256 threads the lanes of one partial sum:
// block 4x + v, thread 64k + t takes lane x*1024 + 256k + 64v + t, so the block
// reduces them itself (grid: at least 4 blocks; lanes past L count zero).
__device__ __forceinline__ int lane_of(int blk, int t) {
  return (blk >> 2) * 1024 + (t >> 6) * 256 + (blk & 3) * 64 + (t & 63);
}
// thread t's sum of a block's lane values in LDS ([k][64])
__device__ __forceinline__ double lanes4(const double *sm, int t) {
  double s = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) s += sm[k * 64 + t];
  return s;
}

// the lane group at element e for VB neighbouring conditions b .. b+VB-1
// (x[h][k], zeros past n1), loaded without a branch so that the loads of
// several vectors and groups are in flight together: addresses past n1 are
// clamped (B > 1) or lie in the vector's padding (B = 1)
template <typename TV, int VB>
__device__ __forceinline__ void ld_lanes(const TV *__restrict__ v, size_t e, size_t n1, int lgB, int b,
                                         double x[kLaneGroup][VB]) {
  if constexpr (VB == 1) {
    if (lgB == 0) {
      TV r[kLaneGroup];
      if constexpr (sizeof(TV) == 8) {
        const double2 p = *reinterpret_cast<const double2 *>(v + e), q = *reinterpret_cast<const double2 *>(v + e + 2);
        r[0] = p.x; r[1] = p.y; r[2] = q.x; r[3] = q.y;
      } else {
        const float4 p = *reinterpret_cast<const float4 *>(v + e);
        r[0] = p.x; r[1] = p.y; r[2] = p.z; r[3] = p.w;
      }
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++) x[h][0] = e + h < n1 ? (double)r[h] : 0.0;
    } else {
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++) {
        const size_t at = e + h < n1 ? e + h : n1 - 1;
        const double t = (double)v[(at << lgB) + b];
        x[h][0] = e + h < n1 ? t : 0.0;
      }
    }
  } else {
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++) {
      const size_t at = e + h < n1 ? e + h : n1 - 1;
      double t[4];
      const TV *src = v + (at << lgB) + b;
      if constexpr (sizeof(TV) == 8) {
        const double2 p = *reinterpret_cast<const double2 *>(src), q = *reinterpret_cast<const double2 *>(src + 2);
        t[0] = p.x; t[1] = p.y; t[2] = q.x; t[3] = q.y;
      } else {
        const float4 p = *reinterpret_cast<const float4 *>(src);
        t[0] = p.x; t[1] = p.y; t[2] = p.z; t[3] = p.w;
      }
#pragma unroll
      for (int k = 0; k < VB; k++) x[h][k] = e + h < n1 ? t[k] : 0.0;
    }
  }
}

// Dot products <V_q, w>, q < cnt, and ||w||^2 (row cnt) per lane, all chunks
// of Q vectors in one launch (blockIdx.y; w is read once per chunk).  A thread
// is one lane of VB neighbouring conditions (quad_of).  One condition: the block's lanes (lane_of) are summed here
// as level 1 of the lane sums does, out is S2[row][G][4]; a batch stores the
// lane sums S[row*B + b][L].
// Bound by HBM on the 2M wing; on small meshes by the number of waves (L is
// 4096 for 40k triangles: 64 waves), hence Q: with fewer vectors a thread there
// are more blocks and the same vectors are in flight at once.  40k triangles,
// FP64: 11 us a step, where chunks of 8 took 19 us and two sum launches each;
// 83k tetrahedra 15 against 28 us a chunk; unchanged on the 2M wing.
template <typename TV, int VB, int Q>
__global__ __launch_bounds__(256) void k_mdot(const TV *__restrict__ V, size_t stride, int cnt,
                                               const TV *__restrict__ w, size_t n1, int lgB, int L,
                                               double *__restrict__ out, Gate gate) {
  const int B = 1 << lgB, lgU = VB == 1 ? lgB : lgB - 2;
  if (gate.closed(B)) return;
  const size_t u = lgB == 0 ? (size_t)lane_of(blockIdx.x, threadIdx.x) : (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t l = u >> lgU;
  const int b = (int)(u & (((size_t)1 << lgU) - 1)) * VB;
  const int i0 = blockIdx.y * Q;
  const TV *v[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) v[q] = V + (size_t)(i0 + q < cnt ? i0 + q : (cnt > 0 ? cnt - 1 : 0)) * stride;
  double acc[Q + 1][VB];
#pragma unroll
  for (int q = 0; q <= Q; q++)
#pragma unroll
    for (int k = 0; k < VB; k++) acc[q][k] = 0;
  if (l < (size_t)L) {
#pragma unroll Q == 1 ? 4 : (Q <= 3 ? 2 : 1)
    for (size_t e = kLaneGroup * l; e < n1; e += (size_t)kLaneGroup * L) {
      double wx[kLaneGroup][VB], vx[Q][kLaneGroup][VB];
      ld_lanes<TV, VB>(w, e, n1, lgB, b, wx);
#pragma unroll
      for (int q = 0; q < Q; q++) ld_lanes<TV, VB>(v[q], e, n1, lgB, b, vx[q]);
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
          for (int k = 0; k < VB; k++) acc[q][k] += vx[q][h][k] * wx[h][k];
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
        for (int k = 0; k < VB; k++) acc[Q][k] += wx[h][k] * wx[h][k];
    }
  }
  const int nq = min(Q, cnt - i0);
  if (lgB == 0) {
    if constexpr (VB == 1) {
      __shared__ double sm[4][256];
      const int g = threadIdx.x >> 6, t = threadIdx.x & 63;
#pragma unroll
      for (int r0 = 0; r0 <= Q; r0 += 4) {   // four rows at a time, a wave each
        if (r0) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (r0 + r <= Q) sm[r][threadIdx.x] = acc[r0 + r <= Q ? r0 + r : 0][0];
        __syncthreads();
        const int q = r0 + g;   // Q: the norm, from the first chunk only
        const int row = q < Q ? (q < nq ? i0 + q : -1) : (q == Q && blockIdx.y == 0 ? cnt : -1);
        if (row < 0) continue;
        const double s = wave_sum(lanes4(sm[g], t));
        if (t == 0) out[(size_t)row * gridDim.x + blockIdx.x] = s;
      }
    }
    return;
  }
  if (l >= (size_t)L) return;
#pragma unroll
  for (int q = 0; q <= Q; q++) {
    const int row = q < Q ? (q < nq ? i0 + q : -1) : (blockIdx.y == 0 ? cnt : -1);
    if (row < 0) continue;
#pragma unroll
    for (int k = 0; k < VB; k++) out[((size_t)row * B + b + k) * L + l] = acc[q][k];
  }
}

// level 1 of the lane sums of row qb, groups x, from stored lane sums
__global__ __launch_bounds__(256) void k_sum_lanes1(const double *__restrict__ S, int L, double *__restrict__ S2) {
  const int x = blockIdx.x, qb = blockIdx.y, G = gridDim.x;
  double s = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int l = x * 1024 + k * 256 + (int)threadIdx.x;
    if (l < L) s += S[(size_t)qb * L + l];
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) S2[((size_t)qb * G + x) * 4 + (threadIdx.x >> 6)] = s;
}

// group x's four level-1 sums of a row
__device__ __forceinline__ double group_sum(const double *__restrict__ row, int x) {
  const double *p = row + (size_t)x * 4;
  return p[0] + p[1] + p[2] + p[3];
}

// where the sum of row qb = q*B + b goes: the dots layout when qnorm >= 0
// (row qnorm is ||w||^2), else row q
__device__ __forceinline__ size_t sum_at(int qb, int qnorm, int lgB) {
  const int q = qb >> lgB, qo = qnorm < 0 ? q : (q == qnorm ? 8 : dot_row(q));
  return ((size_t)qo << lgB) + (qb & ((1 << lgB) - 1));
}

// level 2: row qb = sum of its G level-1 sums, thread t adding t, t + 256, ...
// in order, then a fixed tree.  A closed gate passes the value at keep on.
__global__ __launch_bounds__(256) void k_sum_lanes(const double *__restrict__ S2, int G, double *__restrict__ out,
                                                   int qnorm, int lgB, Gate gate, const double *__restrict__ keep) {
  const int qb = blockIdx.x;
  if (gate.closed(1 << lgB)) {
    if (keep && threadIdx.x == 0) out[sum_at(qb, qnorm, lgB)] = keep[qb];
    return;
  }
  double s = 0;
  for (int l = threadIdx.x; l < G; l += 256) s += group_sum(S2 + (size_t)qb * G * 4, l);
  __shared__ double sh[4];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[sum_at(qb, qnorm, lgB)] = sh[0] + sh[1] + sh[2] + sh[3];
}

// both levels in one launch, a block per row, for G <= kRowGroups groups (the
// sums are those of the two launches)
constexpr int kRowGroups = 16;
__global__ __launch_bounds__(1024) void k_sum_rows(const double *__restrict__ S, int L, double *__restrict__ out,
                                                   int qnorm, int lgB, Gate gate, const double *__restrict__ keep) {
  const int qb = blockIdx.x, G = (L + 1023) / 1024;
  if (gate.closed(1 << lgB)) {
    if (keep && threadIdx.x == 0) out[sum_at(qb, qnorm, lgB)] = keep[qb];
    return;
  }
  __shared__ double sh[kRowGroups][4];
  const int t = threadIdx.x & 255;
#pragma unroll
  for (int x0 = 0; x0 < kRowGroups; x0 += 4) {
    if (x0 >= G) break;
    const int x = x0 + (threadIdx.x >> 8);
    double s = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int l = x * 1024 + k * 256 + t;
      if (l < L) s += S[(size_t)qb * L + l];
    }
    s = wave_sum(s);
    if ((t & 63) == 0) sh[x][t >> 6] = s;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const double s = wave_sum((int)threadIdx.x < G ? group_sum(sh[0], threadIdx.x) : 0.0);
  if (threadIdx.x == 0) out[sum_at(qb, qnorm, lgB)] = s;
}

// h of a Gram-Schmidt pass into hs[cnt][B].  With S2 (one condition, G <= 64)
// every block does level 2 of the lane sums and block 0 writes it to dots;
// without it h comes from dots.  In a second pass the conditions that need none
// use h = 0.  A barrier must follow.
__device__ __forceinline__ void orth_h(const double *__restrict__ S2, int G, double *dots, int cnt, int B,
                                       const Gate &gate, double *hs) {
  if (S2) {
    const int lane = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q <= cnt; q += 4) {
      const double s = wave_sum(lane < G ? group_sum(S2 + (size_t)q * G * 4, lane) : 0.0);
      if (lane == 0) {
        if (q < cnt) hs[q] = s;
        if (blockIdx.x == 0) dots[q == cnt ? 8 : dot_row(q)] = s;
      }
    }
  } else {
    for (int q = threadIdx.x; q < cnt * B; q += blockDim.x) {
      const int qq = q / B, b = q - qq * B;
      const double h = dots[(size_t)dot_row(qq) * B + b];
      hs[q] = gate.eta > 0.0 && !gate.second(b, B) ? 0.0 : h;
    }
  }
}

// wx -= sum_q h_q V_q for one lane group of VB conditions, NU vectors' loads in
// flight at once
template <typename TV, int VB, int NU>
__device__ __forceinline__ void orth_group(const TV *__restrict__ V, size_t stride, int cnt, const double *hs,
                                           size_t e, size_t n1, int lgB, int b, double wx[kLaneGroup][VB]) {
  auto sub = [&](auto nu, int q) {
    constexpr int M = decltype(nu)::value;
    double vx[M][kLaneGroup][VB];
#pragma unroll
    for (int i = 0; i < M; i++) ld_lanes<TV, VB>(V + (size_t)(q + i) * stride, e, n1, lgB, b, vx[i]);
#pragma unroll
    for (int i = 0; i < M; i++)
#pragma unroll
      for (int k = 0; k < VB; k++) {
        const double hq = hs[((q + i) << lgB) + b + k];
#pragma unroll
        for (int h = 0; h < kLaneGroup; h++) wx[h][k] -= hq * vx[i][h][k];
      }
  };
  int q = 0;
  for (; q + NU <= cnt; q += NU) sub(std::integral_constant<int, NU>{}, q);
  if constexpr (NU > 4)
    if (q + 4 <= cnt) { sub(std::integral_constant<int, 4>{}, q); q += 4; }
  if constexpr (NU > 2)
    if (q + 2 <= cnt) { sub(std::integral_constant<int, 2>{}, q); q += 2; }
  if (q < cnt) sub(std::integral_constant<int, 1>{}, q);
}

// the updated group stored, its squares (of the stored values) in r2
template <typename TV, int VB>
__device__ __forceinline__ void st_lanes(TV *__restrict__ w, size_t e, size_t n1, int lgB, int b,
                                         const double wx[kLaneGroup][VB], double r2[kLaneGroup][VB]) {
  TV r[kLaneGroup][VB];
#pragma unroll
  for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
    for (int k = 0; k < VB; k++) {
      r[h][k] = (TV)wx[h][k];
      r2[h][k] = (double)r[h][k] * (double)r[h][k];
    }
  if constexpr (VB == 1) {
    TV t[kLaneGroup];
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++) t[h] = r[h][0];
    st_group(w, e, n1, lgB, b, t);
  } else {
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++)
      if (e + h < n1) {
        TV *dst = w + ((e + h) << lgB) + b;
        if constexpr (sizeof(TV) == 8) {
          reinterpret_cast<double2 *>(dst)[0] = make_double2(r[h][0], r[h][1]);
          reinterpret_cast<double2 *>(dst)[1] = make_double2(r[h][2], r[h][3]);
        } else {
          *reinterpret_cast<float4 *>(dst) = make_float4(r[h][0], r[h][1], r[h][2], r[h][3]);
        }
      }
  }
}

// w -= sum_q h_q V_q per condition and ||w||^2: one condition's level-1 sums
// S2n[G][4], a batch's lane sums S[b][L].  A block is 256 lanes (VB conditions)
// times SL slots; slot s takes the lane's groups s, s + SL, ..., and with SL > 1
// their squares go through LDS, where the lane's first thread adds them in order.
// Bound by HBM on the 2M wing (232 us, 5.2 TB/s), where SL = 1; with 2^16 lanes
// one slot is one wave per SIMD, which waits for memory: 486k tetrahedra, FP32,
// 54 us a call with one, 34 (4.6 TB/s) with four.
template <typename TV, int VB, int SL>
__global__ __launch_bounds__(256 * SL) void k_orth_lanes(const TV *__restrict__ V, size_t stride, int cnt,
                                                         const double *__restrict__ S2, int G, double *dots,
                                                         TV *__restrict__ w, size_t n1, int lgB, int L,
                                                         double *__restrict__ S, Gate gate) {
  const int B = 1 << lgB, lgU = VB == 1 ? lgB : lgB - 2;
  if (gate.closed(B)) return;
  extern __shared__ double hs[];   // [cnt][B]
  __shared__ double sq[SL > 1 ? kLaneGroup * VB : 1][256 * SL];
  orth_h(S2, G, dots, cnt, B, gate, hs);
  __syncthreads();
  const int t = threadIdx.x & 255, sl = threadIdx.x >> 8;
  const size_t u = lgB == 0 ? (size_t)lane_of(blockIdx.x, t) : (size_t)blockIdx.x * 256 + t;
  const size_t l = u >> lgU;
  const int b = (int)(u & (((size_t)1 << lgU) - 1)) * VB;
  const bool lane_ok = l < (size_t)L;
  double nrm[VB];
#pragma unroll
  for (int k = 0; k < VB; k++) nrm[k] = 0;
  for (size_t g0 = 0; g0 * L * kLaneGroup < n1; g0 += SL) {
    const size_t e = kLaneGroup * (l + (size_t)L * (g0 + sl));
    double r2[kLaneGroup][VB];
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
      for (int k = 0; k < VB; k++) r2[h][k] = 0;
    if (lane_ok && e < n1) {
      double wx[kLaneGroup][VB];
      ld_lanes<TV, VB>(w, e, n1, lgB, b, wx);
      orth_group<TV, VB, VB == 1 ? 4 : 2>(V, stride, cnt, hs, e, n1, lgB, b, wx);
      st_lanes<TV, VB>(w, e, n1, lgB, b, wx, r2);
    }
    if constexpr (SL == 1) {
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
        for (int k = 0; k < VB; k++) nrm[k] += r2[h][k];
    } else {
      if (g0) __syncthreads();
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
        for (int k = 0; k < VB; k++) sq[h * VB + k][threadIdx.x] = r2[h][k];
      __syncthreads();
      if (sl == 0)
#pragma unroll
        for (int i = 0; i < SL; i++)
#pragma unroll
          for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
            for (int k = 0; k < VB; k++) nrm[k] += sq[h * VB + k][i * 256 + t];
    }
  }
  if (lgB == 0) {
    if constexpr (VB == 1) {
      __shared__ double sm[256];
      if (sl == 0) sm[t] = nrm[0];
      __syncthreads();
      if (threadIdx.x < 64) {
        const double s = wave_sum(lanes4(sm, threadIdx.x));
        if (threadIdx.x == 0) S[blockIdx.x] = s;
      }
    }
  } else if (sl == 0 && lane_ok) {
#pragma unroll
    for (int k = 0; k < VB; k++) S[(size_t)(b + k) * L + l] = nrm[k];
  }
}

// The same for few lanes, a thread per lane group: the kOrthSlots groups of a
// lane sit in one block, their squares go through LDS and are added in the
// lane's order; lane sums into S[b][L].  With a thread per lane small meshes
// ran on a few waves, each waiting for memory once per four vectors and group
// (40k triangles, 64 waves: 21 us a call, now 10; 83k tetrahedra 35, now 14).
constexpr int kOrthSlots = 16;
template <typename TV, int VB>
__global__ __launch_bounds__(256) void k_orth_slots(const TV *__restrict__ V, size_t stride, int cnt,
                                                    const double *__restrict__ S2, int G, double *dots,
                                                    TV *__restrict__ w, size_t n1, int lgB, int L,
                                                    double *__restrict__ S, Gate gate) {
  const int B = 1 << lgB, lgU = VB == 1 ? lgB : lgB - 2;
  if (gate.closed(B)) return;
  extern __shared__ double hs[];   // [cnt][B]
  __shared__ double sq[VB][kLaneGroup][256];
  orth_h(S2, G, dots, cnt, B, gate, hs);
  __syncthreads();
  const int p = threadIdx.x & 15, sl = threadIdx.x >> 4;
  const size_t u = (size_t)blockIdx.x * 16 + p, l = u >> lgU;
  const int b = (int)(u & (((size_t)1 << lgU) - 1)) * VB;
  const bool lane_ok = l < (size_t)L;
  double nrm = 0;
  for (size_t g0 = 0; g0 * L * kLaneGroup < n1; g0 += kOrthSlots) {
    const size_t e = kLaneGroup * (l + (size_t)L * (g0 + sl));
    double r2[kLaneGroup][VB];
#pragma unroll
    for (int h = 0; h < kLaneGroup; h++)
#pragma unroll
      for (int k = 0; k < VB; k++) r2[h][k] = 0;
    if (lane_ok && e < n1) {
      double wx[kLaneGroup][VB];
      ld_lanes<TV, VB>(w, e, n1, lgB, b, wx);
      orth_group<TV, VB, VB == 1 ? 8 : 2>(V, stride, cnt, hs, e, n1, lgB, b, wx);
      st_lanes<TV, VB>(w, e, n1, lgB, b, wx, r2);
    }
    if (g0) __syncthreads();
#pragma unroll
    for (int k = 0; k < VB; k++)
#pragma unroll
      for (int h = 0; h < kLaneGroup; h++) sq[k][h][threadIdx.x] = r2[h][k];
    __syncthreads();
    if ((int)threadIdx.x < 16 * VB)   // thread (k, lane p): the lane's squares in order
      for (int i = 0; i < kOrthSlots; i++)
#pragma unroll
        for (int h = 0; h < kLaneGroup; h++) nrm += sq[threadIdx.x >> 4][h][i * 16 + p];
  }
  if ((int)threadIdx.x < 16 * VB && lane_ok) S[(size_t)(b + (threadIdx.x >> 4)) * L + l] = nrm;
}

// r = b - y (b FP64) and ||r||^2 per lane into S[b*L + l]
template <typename TV>
__global__ __launch_bounds__(256) void k_resid(const double *__restrict__ bv, const TV *__restrict__ y,
                                               TV *__restrict__ r, size_t n1, int lgB, int L, double *__restrict__ S) {
  const int B = 1 << lgB;
  const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ((size_t)L << lgB)) return;
  const size_t l = g >> lgB;
  const int b = (int)(g & (B - 1));
  double nrm = 0;
  for (size_t e = kLaneGroup * l; e < n1; e += (size_t)kLaneGroup * L) {
    double bx[kLaneGroup], yx[kLaneGroup];
    ld_group(bv, e, n1, lgB, b, bx);
    ld_group(y, e, n1, lgB, b, yx);
    TV rr[kLaneGroup];
#pragma unroll
    for (int k = 0; k < kLaneGroup; k++) {
      const double v = bx[k] - yx[k];
      rr[k] = (TV)v;
      nrm += v * v;
    }
    st_group(r, e, n1, lgB, b, rr);
  }
  S[(size_t)b * L + l] = nrm;
}

// Element-wise vector kernels.  A thread works on groups of 4 consecutive
// elements (one 16-byte packet in FP32, two in FP64; every vector starts on a
// 64-element boundary) in a grid-stride loop; the grid's thread count is a
// multiple of 64, so element t of every group a thread touches belongs to the
// same condition, (4*tid + t) mod B, and per-condition factors are read once.
template <typename T>
__device__ __forceinline__ void ld4(const T *p, double x[4]) {
  if (sizeof(T) == 8) {
    const double2 a = *reinterpret_cast<const double2 *>(p);
    const double2 c = *reinterpret_cast<const double2 *>(p + 2);
    x[0] = a.x; x[1] = a.y; x[2] = c.x; x[3] = c.y;
  } else {
    const float4 a = *reinterpret_cast<const float4 *>(p);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
  }
}
template <typename T>
__device__ __forceinline__ void st4(T *p, const double x[4]) {
  if (sizeof(T) == 8) {
    *reinterpret_cast<double2 *>(p) = make_double2(x[0], x[1]);
    *reinterpret_cast<double2 *>(p + 2) = make_double2(x[2], x[3]);
  } else {
    *reinterpret_cast<float4 *>(p) = make_float4((float)x[0], (float)x[1], (float)x[2], (float)x[3]);
  }
}

// w = w / sqrt(||w||^2) per condition when that is > 0, the norm (row kDotNorm
// of dots) read on the device, so the launch need not wait for the host.  Block 0
// hands the host the first ndots values of dots (a copy of its own took 2.7 us
// a step and its gap), with the gate's decision in row kDotSecond, so that the
// host adds a second pass's products exactly where the kernels used them.
// (Summing the lane norms here too, by every block, took 8.6 us where the sum and
// this take 7.3: 40k triangles.)
template <typename TV>
__global__ __launch_bounds__(256) void k_scale_norm(TV *__restrict__ w, const double *__restrict__ dots,
                                                    double *__restrict__ hdots, int ndots, size_t n, int lgB,
                                                    Gate gate) {
  const size_t B = (size_t)1 << lgB, tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x,
               nt = (size_t)gridDim.x * blockDim.x, ng = n / 4;
  const double *n2 = dots + kDotNorm * B;
  if (blockIdx.x == 0)
    for (int q = threadIdx.x; q < ndots; q += blockDim.x)
      hdots[q] = q >> lgB != kDotSecond ? dots[q] : (gate.second(q & ((int)B - 1), (int)B) ? 1.0 : 0.0);
  double a[4];
  bool on[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    if (t > 0 && lgB == 0) {   // one condition: one reciprocal
      a[t] = a[0];
      on[t] = on[0];
      continue;
    }
    const double s2 = n2[(4 * tid + t) & (B - 1)];
    on[t] = s2 > 0;
    a[t] = on[t] ? 1.0 / sqrt(s2) : 1.0;
  }
  for (size_t g = tid; g < ng; g += nt) {
    double x[4];
    ld4(w + 4 * g, x);
#pragma unroll
    for (int t = 0; t < 4; t++) x[t] = on[t] ? (double)(TV)(a[t] * x[t]) : x[t];
    st4(w + 4 * g, x);
  }
  for (size_t e = 4 * ng + tid; e < n; e += nt) {
    const double s2 = n2[e & (B - 1)];
    if (s2 > 0) w[e] = (TV)((1.0 / sqrt(s2)) * (double)w[e]);
  }
}

// y = a_b x (scale/copy with conversion), a per condition; y may be x
template <typename TA, typename TB>
__global__ void k_scale_b(const TA *x, CoefB a, TB *y, size_t n, int lgB) {
  const size_t B = (size_t)1 << lgB, tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x,
               nt = (size_t)gridDim.x * blockDim.x, ng = n / 4;
  double c[4];
#pragma unroll
  for (int t = 0; t < 4; t++) c[t] = a.c[(4 * tid + t) & (B - 1)];
  for (size_t g = tid; g < ng; g += nt) {
    double v[4];
    ld4(x + 4 * g, v);
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = c[t] * v[t];
    st4(y + 4 * g, v);
  }
  for (size_t e = 4 * ng + tid; e < n; e += nt) y[e] = (TB)(a.c[e & (B - 1)] * (double)x[e]);
}

// out[q] = sum over blocks of part[q][.], fixed order (deterministic)
__global__ void k_reduce_parts(const double *__restrict__ part, int nblk, int nq, double *__restrict__ out) {
  const int q = blockIdx.x;
  if (q >= nq) return;
  double s = 0;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += part[(size_t)q * nblk + b];
  __shared__ double sh[4];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[q] = sh[0] + sh[1] + sh[2] + sh[3];
}

// y = a*x (scale/copy with conversion)
template <typename TA, typename TB>
__global__ void k_scale(const TA *__restrict__ x, double a, TB *__restrict__ y, size_t n) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x,
               ng = n / 4;
  for (size_t g = tid; g < ng; g += nt) {
    double v[4];
    ld4(x + 4 * g, v);
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = a * v[t];
    st4(y + 4 * g, v);
  }
  for (size_t e = 4 * ng + tid; e < n; e += nt) y[e] = (TB)(a * (double)x[e]);
}

// u = sum_q c[q][b] V[q] per condition
template <typename TV>
__global__ void k_combine(const TV *__restrict__ V, size_t stride, int cnt, const double *__restrict__ c,
                          TV *__restrict__ u, size_t n, int lgB) {
  const size_t B = (size_t)1 << lgB, tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x,
               nt = (size_t)gridDim.x * blockDim.x, ng = n / 4;
  int bt[4];
#pragma unroll
  for (int t = 0; t < 4; t++) bt[t] = (int)((4 * tid + t) & (B - 1));
  for (size_t g = tid; g < ng; g += nt) {
    double s[4] = {0, 0, 0, 0};
    for (int q = 0; q < cnt; q++) {
      double v[4];
      ld4(V + (size_t)q * stride + 4 * g, v);
#pragma unroll
      for (int t = 0; t < 4; t++) s[t] += c[q * B + bt[t]] * v[t];
    }
    st4(u + 4 * g, s);
  }
  for (size_t e = 4 * ng + tid; e < n; e += nt) {
    const size_t b = e & (B - 1);
    double s = 0;
    for (int q = 0; q < cnt; q++) s += c[q * B + b] * (double)V[(size_t)q * stride + e];
    u[e] = (TV)s;
  }
}

// x (FP64) += z
template <typename TV>
__global__ void k_axpy_x(double *__restrict__ x, const TV *__restrict__ z, size_t n) {
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x,
               ng = n / 4;
  for (size_t g = tid; g < ng; g += nt) {
    double xv[4], zv[4];
    ld4(x + 4 * g, xv);
    ld4(z + 4 * g, zv);
#pragma unroll
    for (int t = 0; t < 4; t++) xv[t] += zv[t];
    st4(x + 4 * g, xv);
  }
  for (size_t e = 4 * ng + tid; e < n; e += nt) x[e] += (double)z[e];
}

// implicit update U[v][i][b] += x[i][v][b] for the conditions still advancing
template <int ND>
__global__ __launch_bounds__(256) void k_update(double *__restrict__ U, const double *__restrict__ x, int N, int lgB,
                                                CoefB active) {
  constexpr int NV = ND + 2;
  const int B = 1 << lgB, t = cell_index();
  const int i = t >> lgB, b = t & (B - 1);
  if (i >= N || active.c[b] == 0.0) return;
#pragma unroll
  for (int v = 0; v < NV; v++) U[((size_t)v * N + i) * B + b] += x[((size_t)i * NV + v) * B + b];
}

// bits[q] = max over the Linf copies (copy 0 in place)
__global__ void k_linf_reduce_i(unsigned long long *bits, int nq) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nq) {
    const unsigned long long m = linf_slots_max(bits, nq, q);
    bits[q] = m;
  }
}

__global__ void k_fill_u64_i(unsigned long long *p, int n, unsigned long long v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// BiCGStab vector kernels (AMGCL's bicgstab.hpp, right preconditioning); each
// writes per-block partial sums of the dot products its caller needs next
// ---------------------------------------------------------------------------
// p = r + (-beta*omega) v + beta p   (axpbypcz(1, r, -beta*omega, v, beta, p))
template <typename TV>
__global__ void k_bicg_p(const TV *__restrict__ r, const TV *__restrict__ v, TV *__restrict__ p, double bo,
                         double beta, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
    p[e] = (TV)((double)r[e] + bo * (double)v[e] + beta * (double)p[e]);
}
// dots of a with up to two vectors: (a, u), (a, w); per-block partials [2][grid]
template <typename TV>
__global__ __launch_bounds__(256) void k_dot2(const TV *__restrict__ a, const TV *__restrict__ u,
                                              const TV *__restrict__ w, size_t n, double *__restrict__ part) {
  double acc[2] = {0, 0};
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const double ae = (double)a[e];
    acc[0] += ae * (double)u[e];
    if (w) acc[1] += ae * (double)w[e];
  }
  block_store_sums(acc, 2, part);
}
// x += c T (x FP64); o = i + (-c) y; partials (o, o) and (o, h) (h may be null)
template <typename TV>
__global__ __launch_bounds__(256) void k_bicg_step(double *__restrict__ x, const TV *__restrict__ T, double cf,
                                                   const TV *__restrict__ in, const TV *__restrict__ y,
                                                   TV *__restrict__ o, const TV *__restrict__ h, size_t n,
                                                   double *__restrict__ part) {
  double acc[2] = {0, 0};
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    x[e] += cf * (double)T[e];
    const TV oe = (TV)((double)in[e] + (-cf) * (double)y[e]);
    o[e] = oe;
    acc[0] += (double)oe * (double)oe;
    if (h) acc[1] += (double)oe * (double)h[e];
  }
  block_store_sums(acc, 2, part);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static Impl *impl_of(bes_ctx *c) { return (Impl *)c->impl; }

// Multicolour order of the block ILU(0) (rows of one colour are never
// coupled, so each colour is one parallel sweep).  The colours come from a
// greedy pass over the cells in an order set by mode: 0 device (Morton) order,
// 1 the mesh file's cell order, 2 along the freestream velocity (increasing
// centroid . u_inf).  The order changes the factors (the elimination order is
// colour, then cell index) and so the Krylov iteration counts, not the method.
static int build_colouring(bes_ctx *c, Impl *im, int mode) {
  const Geometry &g = c->geo;
  const int N = c->N, k = c->k, nd = c->nd;
  std::vector<int> visit(N);
  for (int q = 0; q < N; q++) visit[q] = mode == 1 ? (int)c->iperm[q] : q;
  if (mode == 2) {
    std::vector<double> key(N);
    for (int i = 0; i < N; i++) {
      const int64_t e = c->perm[i];
      double t = 0;
      for (int d = 0; d < nd; d++) t += g.centroid[e * nd + d] * c->finf[1 + d];
      key[i] = t;
    }
    std::stable_sort(visit.begin(), visit.end(), [&](int a, int b) { return key[a] < key[b]; });
  }
  std::vector<int> color(N, -1);
  int ncol = 0;
  for (int q = 0; q < N; q++) {
    const int i = visit[q];
    const int64_t e = c->perm[i];
    unsigned used = 0;
    for (int m = 0; m < k; m++) {
      const int64_t j = g.cadj[e * k + m];
      if (j >= 0 && color[c->iperm[j]] >= 0) used |= 1u << color[c->iperm[j]];
    }
    int col = 0;
    while (used & (1u << col)) col++;
    color[i] = col;
    ncol = std::max(ncol, col + 1);
  }
  // Within a colour, rows are grouped by which of their slots are lower (an
  // earlier colour) and which are boundary faces, Morton order inside a group:
  // the sweeps and the factorisation branch per slot on that mask, so waves of
  // one mask load only the blocks they use. Rows of one colour are never
  // coupled and the factorisation orders a row's eliminations by colour and
  // cell index, so this order changes neither the factors nor any row's
  // arithmetic in the sweeps.
  std::vector<unsigned char> ckey(N, 0);
  for (int i = 0; i < N; i++) {
    const int64_t e = c->perm[i];
    for (int m = 0; m < k; m++) {
      const int64_t j = g.cadj[e * k + m];
      if (j < 0) ckey[i] |= (unsigned char)(1u << (4 + m));
      else if (color[c->iperm[j]] < color[i]) ckey[i] |= (unsigned char)(1u << m);
    }
  }
  std::vector<int> crow;
  crow.reserve(N);
  im->color_start.assign(ncol + 1, 0);
  for (int col = 0; col < ncol; col++) {
    im->color_start[col] = (int)crow.size();
    for (int i = 0; i < N; i++) if (color[i] == col) crow.push_back(i);
    std::stable_sort(crow.begin() + im->color_start[col], crow.end(),
                     [&](int a, int b) { return ckey[a] < ckey[b]; });
  }
  im->color_start[ncol] = (int)crow.size();
  im->ncolor = ncol;
  std::vector<int> cpos(N), cnb((size_t)k * N, -1), cnp((size_t)k * N, -1);
  std::vector<unsigned char> clow(N, 0);
  for (int q = 0; q < N; q++) cpos[crow[q]] = q;
  for (int q = 0; q < N; q++) {
    const int64_t e = c->perm[crow[q]];
    for (int m = 0; m < k; m++) {
      const int64_t j = g.cadj[e * k + m];
      if (j < 0) continue;
      const int jd = (int)c->iperm[j];
      cnb[(size_t)m * N + q] = jd;
      cnp[(size_t)m * N + q] = cpos[jd];
      if (cpos[jd] < q) clow[q] |= (unsigned char)(1u << m);
    }
  }
  auto up = [&](auto **p, const auto &h) -> int {
    using T = typename std::decay<decltype(h)>::type::value_type;
    if (*p) BES_HIP(hipFree(*p));
    *p = nullptr;
    BES_HIP(hipMalloc((void **)p, std::max<size_t>(h.size(), 1) * sizeof(T)));
    BES_HIP(hipMemcpy(*p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return BES_OK;
  };
  int s;
  if ((s = up(&im->color, color)) || (s = up(&im->crow, crow)) || (s = up(&im->cpos, cpos)) ||
      (s = up(&im->cnb, cnb)) || (s = up(&im->cnp, cnp)) || (s = up(&im->clow, clow)))
    return s;
  im->coloring = mode;
  im->factored = false;
  return BES_OK;
}

static int impl_alloc(bes_ctx *c, Impl *im) {
  const Geometry &g = c->geo;
  const int N = c->N, k = c->k, nd = c->nd, nv = c->nv, NB = nv * nv;
  const int F = (int)g.nface;
  // faces in device order (sorted by owner cell, as the flux pass) with device
  // cell ids: a cell's Jacobian blocks sit next to its neighbours' in JF
  std::vector<int> fo(F), fn(F), cf((size_t)k * N), mrev((size_t)k * N, -1);
  std::vector<double> fnrm((size_t)nd * F);
  std::vector<int> ref2dev(F);
  for (int q = 0; q < F; q++) ref2dev[c->fref[q]] = q;
  for (int q = 0; q < F; q++) {
    const int64_t f = c->fref[q];
    fo[q] = (int)c->iperm[g.owner[f]];
    if (g.nbr[f] >= 0) fn[q] = (int)c->iperm[g.nbr[f]];
    else fn[q] = (g.btype[f] == kSlipWall) ? -1 : -2;
    for (int d = 0; d < nd; d++) fnrm[(size_t)d * F + q] = g.n[f * nd + d];
  }
  for (int i = 0; i < N; i++) {
    const int64_t e = c->perm[i];
    for (int m = 0; m < k; m++) {
      const int64_t f = g.cface[e * k + m];
      cf[(size_t)m * N + i] = ref2dev[f];
      const int64_t j = g.cadj[e * k + m];
      if (j >= 0)
        for (int mm = 0; mm < k; mm++)
          if (g.cface[j * k + mm] == f) mrev[(size_t)m * N + i] = mm;
    }
  }
  im->fd.F = F;
  im->ninternal = 0;
  for (int f = 0; f < F; f++) if (g.nbr[f] >= 0) im->ninternal++;
  auto up = [&](auto **p, const auto &h) -> int {
    using T = typename std::decay<decltype(h)>::type::value_type;
    BES_HIP(hipMalloc((void **)p, std::max<size_t>(h.size(), 1) * sizeof(T)));
    BES_HIP(hipMemcpy(*p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return BES_OK;
  };
  int s;
  if ((s = up(&im->fd.fo, fo)) || (s = up(&im->fd.fn, fn)) || (s = up(&im->fd.fnrm, fnrm)) ||
      (s = up(&im->fd.cf, cf)) || (s = up(&im->fd.mrev, mrev)) || (s = build_colouring(c, im, im->coloring)))
    return s;
  const size_t nvec = (size_t)N * nv;
  const size_t es = im->prec == 32 ? sizeof(float) : sizeof(double);
  const size_t mat = (size_t)(k + 1) * NB * N;
  // face Jacobian records [F][2][JP] in the matrix precision (FP32 in the mixed forms)
  const size_t jrec = im->prec == 32 ? (size_t)(nd == 2 ? JRec<float, 16>::P : JRec<float, 25>::P)
                                     : (size_t)(nd == 2 ? JRec<double, 16>::P : JRec<double, 25>::P);
  const size_t Bs = (size_t)c->B;   // conditions of the batch, the fastest index of every array below
  BES_HIP(hipMalloc((void **)&im->JF, (size_t)F * 2 * jrec * es * Bs));
  BES_HIP(hipMemset(im->JF, 0, (size_t)F * 2 * jrec * es * Bs));
  BES_HIP(hipMalloc((void **)&im->b, nvec * Bs * sizeof(double)));
  BES_HIP(hipMalloc((void **)&im->x, nvec * Bs * sizeof(double)));
  BES_HIP(hipMalloc(&im->A, mat * es * Bs));
  BES_HIP(hipMalloc(&im->LU, mat * es * Bs));
  BES_HIP(hipMalloc(&im->Ac, mat * es * Bs));
  BES_HIP(hipMalloc((void **)&im->bc, nvec * Bs * sizeof(double)));
  BES_HIP(hipMalloc((void **)&im->xc, nvec * Bs * sizeof(double)));
  im->vstride = (nvec * Bs + 63) / 64 * 64;   // 16-byte aligned packet loads on every vector
  // lanes of the deterministic reductions: a power of two set by the size of
  // one condition's vector only (each lane adds 16 to 64 elements; 2^18 lanes,
  // a thread each, for the 2M-cell wing)
  im->lanes = 256;
  while (im->lanes < (1 << 20) && (size_t)im->lanes * 64 < nvec) im->lanes *= 2;
  // GMRES(m) keeps m + 1 basis vectors; BiCGStab's seven vectors use the same storage
  BES_HIP(hipMalloc(&im->V, (size_t)std::max(im->restart + 1, 7) * im->vstride * es));
  BES_HIP(hipMalloc(&im->Z, 3 * im->vstride * es));
  BES_HIP(hipMalloc((void **)&im->part, 32 * kRedBlocks * sizeof(double)));
  // lane sums: one condition keeps only a norm's, the dot products are summed
  // to S2 in their kernel; a batch keeps those of every product of a step
  const size_t nrow = (size_t)im->restart + 2;
  BES_HIP(hipMalloc((void **)&im->S, (c->B == 1 ? 1 : nrow * Bs) * im->lanes * sizeof(double)));
  BES_HIP(hipMalloc((void **)&im->S2, nrow * Bs * ((im->lanes + 1023) / 1024) * 4 * sizeof(double)));
  BES_HIP(hipMalloc((void **)&im->dots, kDotRows * Bs * sizeof(double)));
  BES_HIP(hipHostMalloc((void **)&im->hdots, kDotRows * Bs * sizeof(double), hipHostMallocDefault));
  BES_HIP(hipEventCreateWithFlags(&im->ev_dots, hipEventDisableTiming));
  BES_HIP(hipMalloc((void **)&im->bits, (size_t)kLinfSlots * 16 * Bs * sizeof(unsigned long long)));
  return BES_OK;
}

static void impl_release(Impl *im) {
  lp::lp_release(im);
  amg_release(im);
  void *ptrs[] = {im->fd.fo, im->fd.fn, im->fd.fnrm, im->fd.cf, im->fd.mrev, im->color, im->crow, im->JF, im->S, im->S2,
                  im->b, im->x, im->A, im->LU, im->LM, im->LMh, im->V, im->Z, im->part, im->dots, im->bits, im->Ac,
                  im->bc, im->xc,
                  im->cpos, im->cnb, im->cnp, im->clow, im->Dr, im->Ur};
  for (void *p : ptrs)
    if (p) hipFree(p);
  if (im->hdots) hipHostFree(im->hdots);
  if (im->ev_dots) hipEventDestroy(im->ev_dots);
  delete im;
}

template <typename TM>
static int launch_assemble(bes_ctx *c, Impl *im) {
  const int bs = tuned_bs(c, kProfAssemble), bsj = tuned_bs(c, kProfJacobian), B = c->B, lgB = c->lgB,
            nb = grid_for(c->N * B, bs);
  const double *dtg = c->dt_local ? nullptr : c->dtg;
  const double nbl = (double)c->nv * c->nv;
  {
    // per face: both states, normal, ids; writes one or two nv x nv blocks
    ProfScope ps(c, kProfJacobian, (double)im->fd.F * (16.0 * c->nv * B + 8.0 * c->nd + 8.0) +
                                       (double)(im->fd.F + im->ninternal) * nbl * sizeof(TM) * B);
    const int groups = (im->fd.F + (64 >> lgB) - 1) / (64 >> lgB);   // groups of 64 lanes
    const int nt = groups * 64 * 2;
    if (c->nd == 2)
      hipLaunchKernelGGL((k_face_jacobian<2, TM>), dim3(grid_for(nt, bsj)), dim3(bsj), 0, c->stream, c->U0, c->N,
                         im->fd, c->gc, c->dfinf, (TM *)im->JF, lgB);
    else
      hipLaunchKernelGGL((k_face_jacobian<3, TM>), dim3(grid_for(nt, bsj)), dim3(bsj), 0, c->stream, c->U0, c->N,
                         im->fd, c->gc, c->dfinf, (TM *)im->JF, lgB);
    BES_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_fill_u64_i, dim3((kLinfSlots * 16 * B + 63) / 64), dim3(64), 0, c->stream, im->bits,
                     kLinfSlots * 16 * B, 0ull);
  int s = launch_face_flux(c);
  if (s) return s;
  // per cell: dt, volume, face records, the cell's face fluxes and both
  // Jacobian blocks of each face; writes b and k+1 matrix blocks
  // (dt, volume, face order word; per face: face id twice, area, neighbour;
  // b written), the face fluxes, every face Jacobian block once, the k+1
  // blocks of every row written
  ProfScope ps(c, kProfAssemble,
               (double)c->N * (12.0 + 8.0 * B + c->k * 20.0 + 8.0 * c->nv * B) +
                   (double)c->dm.F * 8.0 * c->fs * B + (double)(im->fd.F + im->ninternal) * nbl * sizeof(TM) * B +
                   (double)c->N * (c->k + 1) * nbl * sizeof(TM) * B);
  if (c->nd == 2)
    hipLaunchKernelGGL((k_assemble<2, TM>), dim3(nb), dim3(bs), 0, c->stream, c->FF, c->fs, c->dt, dtg, c->dm, im->fd,
                       (const TM *)im->JF, im->repeat_nv, im->b, (TM *)im->A, im->bits, im->bits + 8 * B, lgB);
  else
    hipLaunchKernelGGL((k_assemble<3, TM>), dim3(nb), dim3(bs), 0, c->stream, c->FF, c->fs, c->dt, dtg, c->dm, im->fd,
                       (const TM *)im->JF, im->repeat_nv, im->b, (TM *)im->A, im->bits, im->bits + 8 * B, lgB);
  BES_HIP(hipGetLastError());
  return BES_OK;
}

template <typename TM>
static int factor(bes_ctx *c, Impl *im) {
  if (im->precond == 4) return amg_build(c, im);   // times itself
  // a lagged learned operator: kept for lp_rebuild - 1 solves after its build
  // (GMRES still applies the current matrix)
  if (im->precond == 3 && im->lp_current && im->lp_since + 1 < im->lp_rebuild) {
    im->lp_since++;
    return BES_OK;
  }
  const int bs = tuned_bs(c, kProfFactor), N = c->N, nv = c->nv, B = c->B, lgB = c->lgB;
  const double used = (double)(N + 2 * im->ninternal) * nv * nv * sizeof(TM) * B;   // stored blocks
  // ILU(0): the matrix read and its colour-order copy written, that copy read
  // and the factors written, the row-major pivot inverses and upper blocks
  // written and read once each
  const double rowmaj = (double)(N + im->ninternal) * nv * nv * sizeof(TM) * B;
  ProfScope ps(c, kProfFactor, im->precond == 1 ? 2.0 * N * nv * nv * sizeof(TM) * B : 4.0 * used + 2.0 * rowmaj);
  if (im->precond == 3) {
    const int s = lp::lp_build(c, im);
    if (s) return s;
    im->lp_since = 0;
    im->lp_current = true;
    im->lp_builds++;
    return BES_OK;
  }
  if (im->precond == 1) {
    if (c->nd == 2) hipLaunchKernelGGL((k_bj_setup<2, TM>), dim3(grid_for(N * B, bs)), dim3(bs), 0, c->stream, (const TM *)im->A, (TM *)im->LU, N, lgB);
    else hipLaunchKernelGGL((k_bj_setup<3, TM>), dim3(grid_for(N * B, bs)), dim3(bs), 0, c->stream, (const TM *)im->A, (TM *)im->LU, N, lgB);
  } else if (im->precond == 2) {
    if (!im->Dr) BES_HIP(hipMalloc(&im->Dr, (size_t)N * nv * nv * B * sizeof(TM)));
    if (!im->Ur) BES_HIP(hipMalloc(&im->Ur, (size_t)N * c->k * nv * nv * B * sizeof(TM)));
    hipLaunchKernelGGL((k_ilu_scatter<TM>), dim3(grid_for(N * B, 256)), dim3(256), 0, c->stream, (const TM *)im->A,
                       im->cpos, N, (c->k + 1) * nv * nv, (TM *)im->Ac, lgB);
    for (int col = 0; col < im->ncolor; col++) {
      const int r0 = im->color_start[col], nr = im->color_start[col + 1] - r0;
      if (nr == 0) continue;
      if (c->nd == 2)
        hipLaunchKernelGGL((k_ilu_factor_color<2, TM>), dim3(grid_for(nr * B, bs)), dim3(bs), 0, c->stream,
                           (const TM *)im->Ac, (TM *)im->LU, N, im->cnb, im->cnp, im->clow, im->color, im->crow,
                           (TM *)im->Dr, (TM *)im->Ur, r0, nr, lgB);
      else
        hipLaunchKernelGGL((k_ilu_factor_color<3, TM>), dim3(grid_for(nr * B, bs)), dim3(bs), 0, c->stream,
                           (const TM *)im->Ac, (TM *)im->LU, N, im->cnb, im->cnp, im->clow, im->color, im->crow,
                           (TM *)im->Dr, (TM *)im->Ur, r0, nr, lgB);
    }
  }
  BES_HIP(hipGetLastError());
  return BES_OK;
}

// A thread per block (k_spmv_slots, k_ilu_slots) or per cell and condition.  One
// condition gathers its neighbours' values 40 bytes apart and a colour of a small
// mesh is a few waves, so the split pays while a launch does not fill the chip
// with loads: at 590k cells a product still takes 8 % less (FP32 6), at 2M both
// take the same time and the line lies between.  A batch fills it earlier and its
// gathers are contiguous: FP64 gains 5 % and FP32 nothing at 250k cell-conditions;
// at 500k FP64 gains 2 % and FP32 loses up to 3 %.
static bool slot_split(const bes_ctx *c) { return (size_t)c->N * c->B <= (c->B == 1 ? 1u << 20 : 1u << 18); }

// y = A x, matrix and vectors in cell order
template <typename TM, typename TV>
static void spmv_cells(bes_ctx *c, const TM *A, const TV *x, TV *y, int bs) {
  auto go = [&](auto ndc) {
    constexpr int ND = decltype(ndc)::value;
    if (slot_split(c))
      hipLaunchKernelGGL((k_spmv_slots<ND, TM, TV>), dim3(grid_for(c->N * c->B, 64)), dim3(64 * (ND + 2)), 0, c->stream, A,
                         c->dm.nbr, c->N, x, y, c->lgB);
    else
      hipLaunchKernelGGL((k_spmv<ND, TM, TV>), dim3(grid_for(c->N * c->B, bs)), dim3(bs), 0, c->stream, A, c->dm, x, y,
                         c->lgB);
  };
  if (c->nd == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 3>{});
}

// z = M^-1 r (B conditions at once for the block Jacobi and ILU(0) forms)
template <typename TM, typename TV>
static int precond_apply(bes_ctx *c, Impl *im, const TV *r, TV *z, TV *tmp) {
  if (im->precond == 4) return amg_apply<TV>(c, im, r, z, tmp);
  const int bs = tuned_bs(c, kProfPrecond), N = c->N, B = c->B, lgB = c->lgB;
  const size_t n = (size_t)N * c->nv * B;
  const double vb = (double)n * sizeof(TV), blocks = (double)(N + 2 * im->ninternal) * c->nv * c->nv * B;
  // ILU: every stored block once over both sweeps, r, z, y written and read for
  // the colours between the first and the last, neighbour ids and colours;
  // Jacobi: diagonal inverse, r, z
  const int nc = im->ncolor;
  const double ymid = nc > 1 ? (double)(im->color_start[nc - 1] - im->color_start[1]) / std::max(N, 1) : 0.0;
  ProfScope ps(c, kProfPrecond,
               im->precond == 2 ? blocks * sizeof(TM) + (2.0 + 2.0 * ymid) * vb + 2.0 * N * (4.0 * c->k + 4.0)
               : im->precond == 3 ? blocks * (im->prec == 32 ? 2.0 : (double)sizeof(TM)) + 2.0 * vb + 4.0 * N * c->k
               : (im->precond == 1 ? (double)N * c->nv * c->nv * B * sizeof(TM) + 2.0 * vb : 2.0 * vb));
  if (im->precond == 0) {
    hipLaunchKernelGGL((k_scale<TV, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, r, 1.0, z, n);
  } else if (im->precond == 3 && im->prec == 32) {   // learned operator, FP16 copy: one block SpMV
    spmv_cells(c, (const __half *)im->LMh, r, z, bs);
  } else if (im->precond == 3) {   // learned operator: one block SpMV
    spmv_cells(c, (const TM *)im->LM, r, z, bs);
  } else if (im->precond == 1) {
    if (c->nd == 2) hipLaunchKernelGGL((k_bj_apply<2, TM, TV>), dim3(grid_for(N * B, bs)), dim3(bs), 0, c->stream, (const TM *)im->LU, N, r, z, lgB);
    else hipLaunchKernelGGL((k_bj_apply<3, TM, TV>), dim3(grid_for(N * B, bs)), dim3(bs), 0, c->stream, (const TM *)im->LU, N, r, z, lgB);
  } else {
    // colour 0 needs no forward sweep (y = r); the last colour's backward step
    // is fused into its forward sweep
    const int y0end = nc > 0 ? im->color_start[1] : 0;
    const TM *LU = (const TM *)im->LU;
    const bool slots = slot_split(c);
    auto sweeps = [&](auto ndc) {
      constexpr int ND = decltype(ndc)::value;
      auto lower = [&](auto fuse, int r0, int nr) {
        constexpr bool FUSE = decltype(fuse)::value;
        TV *x = FUSE ? z : nullptr;
        if (slots)
          hipLaunchKernelGGL((k_ilu_slots<ND, TM, TV, false, FUSE>), dim3(grid_for(nr * B, 64)), dim3(64 * (ND + 2)), 0,
                             c->stream, LU, N, im->cnp, im->clow, r0, nr, r, tmp, y0end, (const TV *)nullptr,
                             FUSE ? z : tmp, lgB);
        else
          hipLaunchKernelGGL((k_ilu_lower<ND, TM, TV, FUSE>), dim3(grid_for(nr * B, bs)), dim3(bs), 0, c->stream, LU, N,
                             im->cnp, im->clow, r0, nr, r, tmp, y0end, x, lgB);
      };
      for (int col = 1; col < nc; col++) {
        const int r0 = im->color_start[col], nr = im->color_start[col + 1] - r0;
        if (nr == 0) continue;
        if (col == nc - 1) lower(std::true_type{}, r0, nr);
        else lower(std::false_type{}, r0, nr);
      }
      for (int col = nc > 1 ? nc - 2 : nc - 1; col >= 0; col--) {
        const int r0 = im->color_start[col], nr = im->color_start[col + 1] - r0;
        if (nr == 0) continue;
        if (slots)
          hipLaunchKernelGGL((k_ilu_slots<ND, TM, TV, true, true>), dim3(grid_for(nr * B, 64)), dim3(64 * (ND + 2)), 0,
                             c->stream, LU, N, im->cnp, im->clow, r0, nr, r, tmp, y0end, z, z, lgB);
        else
          hipLaunchKernelGGL((k_ilu_upper<ND, TM, TV>), dim3(grid_for(nr * B, bs)), dim3(bs), 0, c->stream, LU, N,
                             im->cnp, im->clow, r0, nr, tmp, z, r, y0end, lgB);
      }
    };
    if (c->nd == 2) sweeps(std::integral_constant<int, 2>{});
    else sweeps(std::integral_constant<int, 3>{});
  }
  BES_HIP(hipGetLastError());
  return BES_OK;
}

template <typename TM, typename TV>
static int spmv(bes_ctx *c, Impl *im, const TV *x, TV *y) {
  const int bs = tuned_bs(c, kProfSpmv), B = c->B, lgB = c->lgB;
  // stored blocks, x and y once, neighbour ids
  ProfScope ps(c, kProfSpmv, (double)(c->N + 2 * im->ninternal) * c->nv * c->nv * sizeof(TM) * B +
                                 2.0 * c->N * c->nv * sizeof(TV) * B + 4.0 * c->N * c->k);
  if (im->precond != 2) {
    spmv_cells(c, (const TM *)im->A, x, y, bs);
  } else {   // ILU(0) solves run in colour order
    auto go = [&](auto ndc) {
      constexpr int ND = decltype(ndc)::value;
      const TM *A = (const TM *)im->Ac;
      if (slot_split(c))
        hipLaunchKernelGGL((k_spmv_slots<ND, TM, TV>), dim3(grid_for(c->N * B, 64)), dim3(64 * (ND + 2)), 0, c->stream,
                           A, im->cnp, c->N, x, y, lgB);
      else
        hipLaunchKernelGGL((k_spmv_pos<ND, TM, TV>), dim3(grid_for(c->N * B, bs)), dim3(bs), 0, c->stream, A, im->cnp,
                           c->N, x, y, lgB);
    };
    if (c->nd == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 3>{});
  }
  BES_HIP(hipGetLastError());
  return BES_OK;
}

// the lane sums S of nqb rows (q*B + b) into out (see sum_at): one launch for
// up to kRowGroups groups of 1024 lanes, else two levels
static void sum_lanes(bes_ctx *c, Impl *im, int nqb, double *out, int qnorm, Gate gate = Gate(),
                      const double *keep = nullptr) {
  const int L = im->lanes, G = (L + 1023) / 1024;
  if (G <= kRowGroups) {
    hipLaunchKernelGGL(k_sum_rows, dim3(nqb), dim3(1024), 0, c->stream, im->S, L, out, qnorm, c->lgB, gate, keep);
  } else {
    hipLaunchKernelGGL(k_sum_lanes1, dim3(G, nqb), dim3(256), 0, c->stream, im->S, L, im->S2);
    hipLaunchKernelGGL(k_sum_lanes, dim3(nqb), dim3(256), 0, c->stream, im->S2, G, out, qnorm, c->lgB, gate, keep);
  }
}

// Four conditions a thread in the dot products and the thread-per-lane update,
// where their values are one 16-byte load.  FP64 takes two, 32 bytes a thread
// apart, on a quarter of the threads: solves of 250k tetrahedra x 4 took 7.58 ms
// so and 6.79 with a condition a thread (with DGKS 9.32 and 7.82), 486k x 8 28.7
// and 27.8, 120k x 16 13.05 and 12.82, 31k x 64 10.22 and 10.16.  FP32: 250k x 4
// 4.01 and 3.97, 31k x 16 1.69 and 1.78, 83k x 32 8.05 and 8.24.
template <typename TV>
static bool quad_of(int lgB) { return sizeof(TV) == 4 && lgB >= 2; }

// dots h_q = V_q^T w (q < cnt) and ||w||^2 of every condition, reduced to row
// at of the dots buffer (the deterministic lane reductions).  With S2 given, one
// condition's last level may be left to the update kernels: *S2 is then its
// level-1 sums (null: the dots are done).
template <typename TV>
static int multidot(bes_ctx *c, Impl *im, const TV *V, size_t stride, int cnt, const TV *w, int at = 0,
                    Gate gate = Gate(), const double **S2 = nullptr) {
  const int B = c->B, lgB = c->lgB, L = im->lanes, G = (L + 1023) / 1024;
  const size_t n1 = (size_t)c->N * c->nv;
  if (S2) *S2 = nullptr;
  if (cnt > im->restart + 1) { set_error("too many basis vectors"); return BES_ERR_ARG; }
  const bool quad = quad_of<TV>(lgB);
  // vectors per thread: as many as leave about four waves on every SIMD
  const size_t units = (size_t)L * (quad ? B / 4 : B);
  int qmax = quad ? 2 : 8;
  while (qmax > 1 && units * ((cnt + qmax - 1) / qmax) < 262144) qmax /= 2;
  const int ny = std::max(1, (cnt + qmax - 1) / qmax), Q = std::max(1, (cnt + ny - 1) / ny);
  ProfScope ps(c, kProfKrylov, (double)(cnt + ny) * n1 * B * sizeof(TV));
  double *out = B == 1 ? im->S2 : im->S;
  const int bs = 256;
  const dim3 grid(B == 1 ? 4 * G : (unsigned)((units + bs - 1) / bs), ny);
  auto go = [&](auto vb, auto q) {
    hipLaunchKernelGGL((k_mdot<TV, decltype(vb)::value, decltype(q)::value>), grid, dim3(bs), 0, c->stream, V, stride,
                       cnt, w, n1, lgB, L, out, gate);
  };
  using std::integral_constant;
  if (quad) {
    if constexpr (sizeof(TV) == 4) {
      if (Q == 1) go(integral_constant<int, 4>{}, integral_constant<int, 1>{});
      else go(integral_constant<int, 4>{}, integral_constant<int, 2>{});
    }
  } else {
    const integral_constant<int, 1> one;
    switch (Q) {
      case 1: go(one, integral_constant<int, 1>{}); break;
      case 2: go(one, integral_constant<int, 2>{}); break;
      case 3: go(one, integral_constant<int, 3>{}); break;
      case 4: go(one, integral_constant<int, 4>{}); break;
      case 5: go(one, integral_constant<int, 5>{}); break;
      case 6: go(one, integral_constant<int, 6>{}); break;
      case 7: go(one, integral_constant<int, 7>{}); break;
      default: go(one, integral_constant<int, 8>{}); break;
    }
  }
  double *d = im->dots + (size_t)at * B;
  if (B > 1) sum_lanes(c, im, (cnt + 1) * B, d, cnt, gate);
  else if (S2 && G <= 64) *S2 = im->S2;
  else hipLaunchKernelGGL(k_sum_lanes, dim3(cnt + 1), dim3(256), 0, c->stream, im->S2, G, d, cnt, 0, gate, nullptr);
  BES_HIP(hipGetLastError());
  return BES_OK;
}

// Up to this many lanes (times conditions, over four where a batch has as many)
// the update runs a thread per lane group: past it a thread per lane gives at least a wave for
// every other SIMD, and the sixteenfold blocks with their barrier cost more (486k
// tetrahedra, 2^16 lanes, FP32: 79 us against 34; the 2M wing 371 against 232).
constexpr size_t kSlotUnits = 16384;

// one Gram-Schmidt pass of w against V_0 .. V_(cnt-1): dots into row at, w
// updated, its ||w||^2 into row nat (a closed gate copies row kDotNorm1 there)
template <typename TV>
static int orthogonalise(bes_ctx *c, Impl *im, const TV *V, size_t stride, int cnt, TV *w, int at, int nat,
                         Gate gate = Gate()) {
  const int B = c->B, lgB = c->lgB, L = im->lanes, G = (L + 1023) / 1024;
  const size_t n1 = (size_t)c->N * c->nv;
  const double *S2 = nullptr;
  int s = multidot<TV>(c, im, V, stride, cnt, w, at, gate, &S2);
  if (s) return s;
  ProfScope ps(c, kProfKrylov, (double)(cnt + 2) * n1 * B * sizeof(TV));
  double *d = im->dots + (size_t)at * B;
  const size_t units = (size_t)L * (lgB >= 2 ? B / 4 : B), lds = (size_t)cnt * B * sizeof(double);
  double *out = im->dots + (size_t)nat * B;
  const double *keep = im->dots + (size_t)kDotNorm1 * B;
  if (units <= kSlotUnits) {
    const dim3 grid((unsigned)((units + 15) / 16));
    if (lgB >= 2)
      hipLaunchKernelGGL((k_orth_slots<TV, 4>), grid, dim3(256), lds, c->stream, V, stride, cnt, S2, G, d, w, n1, lgB,
                         L, im->S, gate);
    else
      hipLaunchKernelGGL((k_orth_slots<TV, 1>), grid, dim3(256), lds, c->stream, V, stride, cnt, S2, G, d, w, n1, lgB,
                         L, im->S, gate);
    sum_lanes(c, im, B, out, -1, gate, keep);
  } else if (B == 1) {   // level 1 in the kernel (S2 may still be read: the sums go to S)
    auto go = [&](auto sl) {
      constexpr int SL = decltype(sl)::value;
      hipLaunchKernelGGL((k_orth_lanes<TV, 1, SL>), dim3(4 * G), dim3(256 * SL), lds, c->stream, V, stride, cnt, S2, G,
                         d, w, n1, lgB, L, im->S, gate);
    };
    if (L <= 65536) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 1>{});
    hipLaunchKernelGGL(k_sum_lanes, dim3(1), dim3(256), 0, c->stream, im->S, G, out, -1, 0, gate, keep);
  } else {
    auto go = [&](auto vb) {
      constexpr int VB = decltype(vb)::value;
      const size_t nt = (size_t)L * (B / VB);
      hipLaunchKernelGGL((k_orth_lanes<TV, VB, 1>), dim3((unsigned)((nt + 255) / 256)), dim3(256), lds, c->stream, V,
                         stride, cnt, S2, G, d, w, n1, lgB, L, im->S, gate);
    };
    if constexpr (sizeof(TV) == 4) {
      if (quad_of<TV>(lgB)) go(std::integral_constant<int, 4>{});
      else go(std::integral_constant<int, 1>{});
    } else {
      go(std::integral_constant<int, 1>{});
    }
    sum_lanes(c, im, B, out, -1, gate, keep);
  }
  BES_HIP(hipGetLastError());
  return BES_OK;
}

// one lane-reduced norm per condition (S slot 0) into dots[at*B + b]
static int sum_norms(bes_ctx *c, Impl *im, int at) {
  sum_lanes(c, im, c->B, im->dots + (size_t)at * c->B, -1);
  BES_HIP(hipGetLastError());
  return BES_OK;
}

static int fetch_dots(bes_ctx *c, Impl *im, size_t ndbl) {
  BES_HIP(hipMemcpyAsync(im->hdots, im->dots, ndbl * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  BES_HIP(hipStreamSynchronize(c->stream));
  return BES_OK;
}

// Whether a step queues the next one's preconditioner and product before the host
// has read h and ||w||: it saves the device the host's turn (10 to 20 us a step)
// and costs one application and product at the end of a cycle, discarded.
// Without DGKS every step does.  With it (queue / wait, ms, DGKS 0.7): 83k
// tetrahedra FP64 7 iterations 1.04 / 1.05, 46 iterations 6.39 / 6.68; 31k x 8
// FP32 4 iterations 0.81 / 0.78, 19 iterations 3.29 / 3.36; 250k x 4 FP64 6
// iterations 5.33 / 4.91, 23 iterations 23.6 / 23.3; 2M FP64 17 iterations 31.8 /
// 30.9.  An AMG cycle costs more than it hides: 83k 9 iterations 1.80 / 1.76, 486k 12
// iterations 5.07 / 4.86.
static bool queue_ahead(const bes_ctx *c, const Impl *im) {
  return im->reorth_eta <= 0 || (im->precond != 4 && (size_t)c->N * c->B <= (1u << 17));
}

// GMRES(m), right-preconditioned, for the B conditions of the batch at once
// (one launch per kernel for all of them).  Each condition keeps its own
// Arnoldi process, Givens rotations, iteration count and stopping point: a
// condition whose estimate meets its target, whose basis breaks down or that
// reaches maxiter stops at that step of the cycle (its x uses exactly those
// steps), the cycle goes on while any condition is active, and every cycle
// restarts from the true residual of each condition still unconverged.  All
// reductions are the lane reductions above, so a condition's iterates are the
// same bits in a batch as alone.  Classical Gram-Schmidt; with eta > 0 a DGKS
// second pass for the conditions whose w kept less than eta of its norm.
template <typename TM, typename TV>
static int gmres(bes_ctx *c, Impl *im, int *iters_out, double *relres_out) {
  const int m = im->restart, B = c->B, lgB = c->lgB;
  const size_t n1 = (size_t)c->N * c->nv, n = n1 * B, vs = im->vstride;
  const int L = im->lanes, nbl = grid_for(L * B, 256);
  TV *V = (TV *)im->V;
  TV *Z = (TV *)im->Z, *Z1 = Z + vs, *Z2 = Z + 2 * vs;
  // ILU(0) solves run in colour order: b in, x out are permuted once per solve
  const bool colour = im->precond == 2;
  const double *bb = im->b;
  double *xx = colour ? im->xc : im->x;
  if (colour) {
    hipLaunchKernelGGL(k_perm_rows<double>, dim3(1024), dim3(256), 0, c->stream, bb, im->crow, c->N, c->nv * B, 1,
                       im->bc);
    bb = im->bc;
  }
  hipMemsetAsync(xx, 0, n * sizeof(double), c->stream);
  const double *hd = im->hdots;
  const double eta = im->reorth_eta;
  auto hdot = [&](int row, int q, int b) { return hd[(size_t)(row + dot_row(q)) * B + b]; };
  const bool ahead = queue_ahead(c, im);
  const int scale_blocks = (int)std::min<size_t>(kRedBlocks, (n / 4 + 255) / 256 + 1);
  // ||b|| per condition
  hipLaunchKernelGGL((k_scale<double, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, bb, 1.0, Z, n);
  int s;
  if ((s = multidot<TV>(c, im, Z, vs, 0, Z)) || (s = fetch_dots(c, im, (size_t)9 * B))) return s;
  std::vector<double> bnorm(B), target(B), rnorm(B);
  std::vector<char> finished(B, 0), active(B, 0), est_done(B, 0);
  std::vector<int> total(B, 0), jb(B, 0);
  for (int b = 0; b < B; b++) {
    bnorm[b] = std::sqrt(hd[(size_t)8 * B + b]);
    target[b] = im->rtol * bnorm[b];
    rnorm[b] = bnorm[b];
    finished[b] = bnorm[b] == 0 || (!im->skip_b.empty() && im->skip_b[b]);
  }
  std::vector<double> H((size_t)B * (m + 1) * m), cs((size_t)B * m), sn((size_t)B * m), g((size_t)B * (m + 1)),
      yv((size_t)B * m), hcol(m + 1), coef((size_t)m * B);
  CoefB scl;
  bool first = true;
  auto any_open = [&]() {
    for (int b = 0; b < B; b++) if (!finished[b] && total[b] < im->maxiter) return true;
    return false;
  };
  while (any_open()) {
    // r = b - A x (x = 0 on the first cycle, as the reference starts every
    // solve).  Every later cycle starts from the true residual of the current
    // x, and a condition is done only when that is at its target: the Givens
    // estimate of the cycle before can fall below the true residual (rounding
    // in the basis, FP32 Krylov vectors), as AMGCL's FGMRES also rechecks
    // (fgmres.hpp:158-163)
    if (first) {
      for (int b = 0; b < B; b++) scl.c[b] = finished[b] ? 0.0 : 1.0 / bnorm[b];
      hipLaunchKernelGGL((k_scale_b<double, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, bb, scl, V, n, lgB);
    } else {
      hipLaunchKernelGGL((k_scale<double, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, xx, 1.0, Z2, n);
      if ((s = spmv<TM, TV>(c, im, Z2, Z1))) return s;
      hipLaunchKernelGGL((k_resid<TV>), dim3(nbl), dim3(256), 0, c->stream, bb, Z1, Z, n1, lgB, L, im->S);
      if ((s = sum_norms(c, im, 0)) || (s = fetch_dots(c, im, (size_t)B))) return s;
      for (int b = 0; b < B; b++) {
        if (finished[b]) continue;
        rnorm[b] = std::sqrt(hd[b]);
        if (rnorm[b] <= target[b]) finished[b] = 1;
        else if (est_done[b]) im->extra_restarts++;   // the estimate said done, the true residual did not
      }
      if (!any_open()) break;
      for (int b = 0; b < B; b++) scl.c[b] = (!finished[b] && total[b] < im->maxiter) ? 1.0 / rnorm[b] : 0.0;
      hipLaunchKernelGGL((k_scale_b<TV, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, Z, scl, V, n, lgB);
    }
    first = false;
    int nact = 0;
    for (int b = 0; b < B; b++) {
      active[b] = !finished[b] && total[b] < im->maxiter;
      est_done[b] = 0;
      jb[b] = 0;
      nact += active[b];
      std::fill(g.begin() + (size_t)b * (m + 1), g.begin() + (size_t)(b + 1) * (m + 1), 0.0);
      g[(size_t)b * (m + 1)] = rnorm[b];
    }
    bool queued = false;
    for (int j = 0; j < m && nact > 0; j++) {
      TV *vj = V + (size_t)j * vs, *w = V + (size_t)(j + 1) * vs;
      if (!queued) {
        if ((s = precond_apply<TM, TV>(c, im, vj, Z, Z1))) return s;
        if ((s = spmv<TM, TV>(c, im, Z, w))) return s;
      }
      queued = false;
      // classical Gram-Schmidt: the dots, the update, with eta > 0 the second
      // pass (its kernels look up which conditions need it) and the
      // normalisation are queued back to back and the host waits once, for h
      // and ||w||
      size_t ev2 = 0, ev2_end = 0;   // profile records of the second pass
      Gate gate;
      if (eta > 0) {
        if ((s = orthogonalise<TV>(c, im, V, vs, j + 1, w, 0, kDotNorm1))) return s;
        gate.eta = eta;
        gate.dots = im->dots;
        ev2 = c->ev_pending.size();
        if ((s = orthogonalise<TV>(c, im, V, vs, j + 1, w, kDots2, kDotNorm, gate))) return s;
        ev2_end = c->ev_pending.size();
      } else if ((s = orthogonalise<TV>(c, im, V, vs, j + 1, w, 0, kDotNorm))) {
        return s;
      }
      hipLaunchKernelGGL((k_scale_norm<TV>), dim3(scale_blocks), dim3(256), 0, c->stream, w, im->dots,
                         im->hdots, (eta > 0 ? kDotRows : kDotNorm + 1) * B, n, lgB, gate);
      BES_HIP(hipGetLastError());
      BES_HIP(hipEventRecord(im->ev_dots, c->stream));
      // the next step's preconditioner and product need only the normalised w:
      // queued before waiting (queue_ahead), they run while the host reads h and
      // ||w|| (their results are discarded for conditions this step ends)
      bool more = false;
      for (int b = 0; b < B; b++) if (active[b] && total[b] + 1 < im->maxiter) more = true;
      if (ahead && j + 1 < m && more) {
        if ((s = precond_apply<TM, TV>(c, im, w, Z, Z1))) return s;
        if ((s = spmv<TM, TV>(c, im, Z, V + (size_t)(j + 2) * vs))) return s;
        queued = true;
      }
      BES_HIP(hipEventSynchronize(im->ev_dots));
      auto second = [&](int b) { return eta > 0 && hd[(size_t)kDotSecond * B + b] != 0.0; };
      bool any = false;
      for (int b = 0; b < B; b++) any = any || second(b);
      if (!any)   // its kernels returned at once
        for (size_t e = ev2; e < ev2_end; e++) c->ev_pending[e].bytes = 0.0;
      for (int b = 0; b < B; b++) {
        if (!active[b]) continue;
        const double hn = std::sqrt(hd[(size_t)kDotNorm * B + b]);
        const bool re = second(b);
        for (int q = 0; q <= j; q++) hcol[q] = re ? hdot(0, q, b) + hdot(kDots2, q, b) : hdot(0, q, b);
        if (re) im->reorths++;
        hcol[j + 1] = hn;
        double *csb = &cs[(size_t)b * m], *snb = &sn[(size_t)b * m], *gb = &g[(size_t)b * (m + 1)];
        for (int q = 0; q < j; q++) {   // Givens rotations
          const double t = csb[q] * hcol[q] + snb[q] * hcol[q + 1];
          hcol[q + 1] = -snb[q] * hcol[q] + csb[q] * hcol[q + 1];
          hcol[q] = t;
        }
        const double den = std::hypot(hcol[j], hcol[j + 1]);
        csb[j] = den > 0 ? hcol[j] / den : 1.0;
        snb[j] = den > 0 ? hcol[j + 1] / den : 0.0;
        hcol[j] = den;
        hcol[j + 1] = 0;
        gb[j + 1] = -snb[j] * gb[j];
        gb[j] = csb[j] * gb[j];
        for (int q = 0; q <= j; q++) H[((size_t)b * (m + 1) + q) * m + j] = hcol[q];
        total[b]++;
        rnorm[b] = std::fabs(gb[j + 1]);
        jb[b] = j + 1;
        if (rnorm[b] <= target[b] || hn == 0) { est_done[b] = 1; active[b] = 0; nact--; }
        else if (total[b] >= im->maxiter) { active[b] = 0; nact--; }
      }
    }
    // solve H y = g (upper triangular j_b x j_b) per condition; x += M (V y)
    int jmax = 0;
    for (int b = 0; b < B; b++) jmax = std::max(jmax, jb[b]);
    if (jmax == 0) continue;
    std::fill(coef.begin(), coef.end(), 0.0);
    for (int b = 0; b < B; b++) {
      const int j = jb[b];
      const double *gb = &g[(size_t)b * (m + 1)];
      double *yb = &yv[(size_t)b * m];
      for (int q = j - 1; q >= 0; q--) {
        double t = gb[q];
        for (int p = q + 1; p < j; p++) t -= H[((size_t)b * (m + 1) + q) * m + p] * yb[p];
        yb[q] = t / H[((size_t)b * (m + 1) + q) * m + q];
      }
      for (int q = 0; q < j; q++) coef[(size_t)q * B + b] = yb[q];
    }
    BES_HIP(hipMemcpyAsync(im->dots, coef.data(), sizeof(double) * (size_t)jmax * B, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL((k_combine<TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, V, vs, jmax, im->dots, Z2, n, lgB);
    if ((s = precond_apply<TM, TV>(c, im, Z2, Z, Z1))) return s;
    hipLaunchKernelGGL((k_axpy_x<TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, xx, Z, n);
    BES_HIP(hipGetLastError());
  }
  // true residual of the returned solution, per condition
  hipLaunchKernelGGL((k_scale<double, TV>), dim3(kRedBlocks), dim3(256), 0, c->stream, xx, 1.0, Z2, n);
  if ((s = spmv<TM, TV>(c, im, Z2, Z1))) return s;
  hipLaunchKernelGGL((k_resid<TV>), dim3(nbl), dim3(256), 0, c->stream, bb, Z1, Z, n1, lgB, L, im->S);
  if ((s = sum_norms(c, im, 0)) || (s = fetch_dots(c, im, (size_t)B))) return s;
  if (colour)
    hipLaunchKernelGGL(k_perm_rows<double>, dim3(1024), dim3(256), 0, c->stream, im->xc, im->crow, c->N, c->nv * B, 0,
                       im->x);
  im->iters_b.assign(total.begin(), total.end());
  im->relres_b.assign(B, 0.0);
  int itmax = 0;
  double rrmax = 0;
  for (int b = 0; b < B; b++) {
    im->relres_b[b] = bnorm[b] > 0 ? std::sqrt(hd[b]) / bnorm[b] : 0.0;
    if (!im->skip_b.empty() && im->skip_b[b]) im->relres_b[b] = 0.0;
    itmax = std::max(itmax, total[b]);
    rrmax = std::max(rrmax, im->relres_b[b]);
  }
  *iters_out = itmax;
  *relres_out = rrmax;
  return BES_OK;
}

// reduce nq per-block partial sums (written by a kRedBlocks-block kernel) and read them on the host
static int fetch_sums(bes_ctx *c, Impl *im, int nq, double *out) {
  hipLaunchKernelGGL(k_reduce_parts, dim3(nq), dim3(256), 0, c->stream, im->part, kRedBlocks, nq, im->dots);
  BES_HIP(hipGetLastError());
  BES_HIP(hipMemcpyAsync(im->hdots, im->dots, nq * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  BES_HIP(hipStreamSynchronize(c->stream));
  for (int q = 0; q < nq; q++) out[q] = im->hdots[q];
  return BES_OK;
}

// BiCGStab with right preconditioning, as AMGCL's solver (bicgstab.hpp:
// operator()): x = 0, r = rh = b; per iteration rho = (r, rh), p, T = M p,
// v = A T, alpha = rho / (rh, v), x += alpha T, s = r - alpha v; if ||s|| is
// above the target: T = M s, t = A T, omega = (t, s) / (t, t), x += omega T,
// r = s - omega t.  Stops when the recursive residual norm is at the target or
// after maxiter iterations; returns the true relative residual.
template <typename TM, typename TV>
static int bicgstab(bes_ctx *c, Impl *im, int *iters_out, double *relres_out) {
  const size_t n = (size_t)c->N * c->nv, vs = im->vstride;
  TV *V = (TV *)im->V;
  TV *r = V, *rh = V + vs, *p = V + 2 * vs, *v = V + 3 * vs, *sv = V + 4 * vs, *t = V + 5 * vs, *T = V + 6 * vs;
  TV *Z = (TV *)im->Z, *Z1 = Z + vs, *Z2 = Z + 2 * vs;
  const bool colour = im->precond == 2;
  const double *bb = im->b;
  double *xx = colour ? im->xc : im->x;
  const dim3 G(kRedBlocks), B(256);
  if (colour) {
    hipLaunchKernelGGL(k_perm_rows<double>, dim3(1024), B, 0, c->stream, bb, im->crow, c->N, c->nv, 1, im->bc);
    bb = im->bc;
  }
  hipMemsetAsync(xx, 0, n * sizeof(double), c->stream);
  hipLaunchKernelGGL((k_scale<double, TV>), G, B, 0, c->stream, bb, 1.0, r, n);
  hipLaunchKernelGGL((k_scale<double, TV>), G, B, 0, c->stream, bb, 1.0, rh, n);
  double d[2];
  int st;
  hipLaunchKernelGGL((k_dot2<TV>), G, B, 0, c->stream, r, r, (const TV *)nullptr, n, im->part);
  if ((st = fetch_sums(c, im, 1, d))) return st;
  const double bnorm = std::sqrt(d[0]);
  *iters_out = 0;
  *relres_out = 0;
  if (bnorm == 0) {
    if (colour) hipMemsetAsync(im->x, 0, n * sizeof(double), c->stream);
    return BES_OK;
  }
  const double target = im->rtol * bnorm;
  double res = bnorm, rho1 = d[0], rho2 = 0, alpha = 0, omega = 0;   // (r, rh) = ||b||^2 at the start
  int iter = 0;
  for (bool first = true; res > target && iter < im->maxiter; ++iter) {
    rho2 = rho1;
    if (iter > 0) rho1 = d[1];   // (r, rh) of the r the last iteration ended with
    if (first) {
      hipLaunchKernelGGL((k_scale<TV, TV>), G, B, 0, c->stream, r, 1.0, p, n);
      first = false;
    } else {
      if (rho2 == 0 || omega == 0) { set_error("BiCGStab breakdown (zero rho or omega)"); break; }
      const double beta = (rho1 * alpha) / (rho2 * omega);
      hipLaunchKernelGGL((k_bicg_p<TV>), G, B, 0, c->stream, r, v, p, -beta * omega, beta, n);
    }
    if ((st = precond_apply<TM, TV>(c, im, p, T, Z1))) return st;
    if ((st = spmv<TM, TV>(c, im, T, v))) return st;
    hipLaunchKernelGGL((k_dot2<TV>), G, B, 0, c->stream, rh, v, (const TV *)nullptr, n, im->part);
    if ((st = fetch_sums(c, im, 1, d))) return st;
    if (d[0] == 0) { set_error("BiCGStab breakdown ((rh, v) = 0)"); break; }
    alpha = rho1 / d[0];
    hipLaunchKernelGGL((k_bicg_step<TV>), G, B, 0, c->stream, xx, T, alpha, r, v, sv, (const TV *)nullptr, n,
                       im->part);
    if ((st = fetch_sums(c, im, 1, d))) return st;
    res = std::sqrt(d[0]);
    if (res > target) {
      if ((st = precond_apply<TM, TV>(c, im, sv, T, Z1))) return st;
      if ((st = spmv<TM, TV>(c, im, T, t))) return st;
      hipLaunchKernelGGL((k_dot2<TV>), G, B, 0, c->stream, t, sv, t, n, im->part);
      if ((st = fetch_sums(c, im, 2, d))) return st;
      omega = d[1] > 0 ? d[0] / d[1] : 0.0;
      if (omega == 0) { set_error("BiCGStab breakdown (omega = 0)"); ++iter; break; }
      hipLaunchKernelGGL((k_bicg_step<TV>), G, B, 0, c->stream, xx, T, omega, sv, t, r, rh, n, im->part);
      if ((st = fetch_sums(c, im, 2, d))) return st;
      res = std::sqrt(d[0]);
    }
  }
  // true residual of the returned solution
  hipLaunchKernelGGL((k_scale<double, TV>), G, B, 0, c->stream, xx, 1.0, Z2, n);
  if ((st = spmv<TM, TV>(c, im, Z2, Z1))) return st;
  hipLaunchKernelGGL((k_resid<TV>), dim3(grid_for(im->lanes, 256)), B, 0, c->stream, bb, Z1, Z, n, 0, im->lanes,
                     im->S);
  if ((st = sum_norms(c, im, 0)) || (st = fetch_dots(c, im, 1))) return st;
  d[0] = im->hdots[0];
  if (colour)
    hipLaunchKernelGGL(k_perm_rows<double>, dim3(1024), B, 0, c->stream, im->xc, im->crow, c->N, c->nv, 0, im->x);
  BES_HIP(hipGetLastError());
  *iters_out = iter;
  *relres_out = std::sqrt(d[0]) / bnorm;
  return BES_OK;
}

// average device time of fn() over reps launches on the context's stream (one untimed first)
template <typename Fn>
static int time_us(bes_ctx *c, int reps, Fn fn, double *us) {
  hipEvent_t a, b;
  BES_HIP(hipEventCreate(&a));
  BES_HIP(hipEventCreate(&b));
  int s = fn();
  if (!s) {
    hipEventRecord(a, c->stream);
    for (int r = 0; r < reps && !s; r++) s = fn();
    hipEventRecord(b, c->stream);
    hipEventSynchronize(b);
    float ms = 0;
    hipEventElapsedTime(&ms, a, b);
    *us = 1e3 * ms / reps;
  }
  hipEventDestroy(a);
  hipEventDestroy(b);
  return s;
}

}  // namespace bes

using namespace bes;

extern "C" {

void bes_implicit_free(bes_ctx *c) {
  if (c && c->impl) {
    impl_release((Impl *)c->impl);
    c->impl = nullptr;
  }
}

int bes_implicit_setup(bes_ctx *c, int precision, int precond, int restart, int maxiter, double rtol) {
  if (!c || (precision != 64 && precision != 32) || precond < 0 || precond > 4 || restart < 1 || restart > 30 ||
      maxiter < 1 || !(rtol > 0)) {
    set_error("invalid implicit setup argument (precision 64/32, precond 0-4, restart 1-30)");
    return BES_ERR_ARG;
  }
  if (c->B != 1 && precond > 2) {
    set_error("a batch of conditions runs with precond 0-2 (none, block Jacobi, ILU(0)); the learned operator and "
              "the AMG take one condition");
    return BES_ERR_ARG;
  }
  bes_implicit_free(c);
  Impl *im = new Impl();
  im->prec = precision;
  im->precond = precond;
  im->restart = restart;
  im->maxiter = maxiter;
  im->rtol = rtol;
  c->impl = im;
  int s = impl_alloc(c, im);
  if (s) { bes_implicit_free(c); return s; }
  return BES_OK;
}

int bes_implicit_set_reorth(bes_ctx *c, double eta) {
  if (!c || !c->impl || !(eta >= 0.0) || eta > 1.0) { set_error("call bes_implicit_setup first / eta in [0,1]"); return BES_ERR_ARG; }
  impl_of(c)->reorth_eta = eta;
  return BES_OK;
}

int bes_implicit_stats(bes_ctx *c, long *reorths, int *lp_fallbacks, long *extra_restarts) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  if (reorths) *reorths = impl_of(c)->reorths;
  if (lp_fallbacks) *lp_fallbacks = impl_of(c)->lp_fallbacks;
  if (extra_restarts) *extra_restarts = impl_of(c)->extra_restarts;
  return BES_OK;
}

int bes_implicit_set_coloring(bes_ctx *c, int mode) {
  if (!c || !c->impl || mode < 0 || mode > 2) { set_error("call bes_implicit_setup first / coloring 0-2"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  if (im->coloring == mode) return BES_OK;
  BES_HIP(hipStreamSynchronize(c->stream));
  return build_colouring(c, im, mode);
}

int bes_implicit_ncolors(bes_ctx *c) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return -BES_ERR_ARG; }
  return impl_of(c)->ncolor;
}

int bes_implicit_set_solver(bes_ctx *c, int solver) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  if (solver != BES_SOLVER_GMRES && solver != BES_SOLVER_BICGSTAB) {
    set_error("LINEAR_SOLVER: only GMRES (FGMRES) and BICGSTAB are available; LGMRES is not");
    return BES_ERR_ARG;
  }
  if (solver == BES_SOLVER_BICGSTAB && c->B != 1) {
    set_error("LINEAR_SOLVER: BICGSTAB takes one condition; a batch runs GMRES");
    return BES_ERR_ARG;
  }
  impl_of(c)->solver = solver;
  return BES_OK;
}

int bes_implicit_set_precond(bes_ctx *c, int precond) {
  if (!c || !c->impl || precond < 0 || precond > 4) { set_error("call bes_implicit_setup first / precond 0-4"); return BES_ERR_ARG; }
  if (c->B != 1 && precond > 2) { set_error("a batch of conditions runs with precond 0-2"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  im->precond = precond;
  im->factored = false;
  return BES_OK;
}

// time step, gradient, limiter, Jacobians and system of every condition; cfl_b
// (per condition) may be null; linf outputs [B][nv]
static int assemble(bes_ctx *c, Impl *im, double cfl, const double *cfl_b, int local, int repeat_nv, double *linf_b,
                    double *linf_r) {
  im->repeat_nv = repeat_nv ? c->nv : 1;
  const int B = c->B;
  int s;
  hipLaunchKernelGGL(k_fill_u64_i, dim3(1), dim3(64), 0, c->stream, c->err, 1, ~0ull);
  if ((s = launch_timestep(c, c->U0, cfl, local, cfl_b))) return s;
  c->dt_local = local != 0;
  if ((s = launch_gradlim(c, c->U0, nullptr, nullptr))) return s;
  if (im->prec == 64) s = launch_assemble<double>(c, im);
  else s = launch_assemble<float>(c, im);
  if (s) return s;
  hipLaunchKernelGGL(k_linf_reduce_i, dim3(grid_for(16 * B, 64)), dim3(64), 0, c->stream, im->bits, 16 * B);
  std::vector<unsigned long long> bb((size_t)16 * B);
  BES_HIP(hipMemcpyAsync(bb.data(), im->bits, bb.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                         c->stream));
  BES_HIP(hipStreamSynchronize(c->stream));
  for (int b = 0; b < B; b++)
    for (int v = 0; v < c->nv; v++) {   // bits [v][B] of b, then [v][B] of sum F*A
      if (linf_b) std::memcpy(&linf_b[(size_t)b * c->nv + v], &bb[(size_t)v * B + b], 8);
      if (linf_r) std::memcpy(&linf_r[(size_t)b * c->nv + v], &bb[(size_t)(8 + v) * B + b], 8);
    }
  im->assembled = true;
  im->factored = false;
  unsigned long long e = 0;
  BES_HIP(hipMemcpy(&e, c->err, sizeof(e), hipMemcpyDeviceToHost));
  if (e != ~0ull) {
    c->last_err_face = e < c->fref.size() ? (long)c->fref[e] : -1;   // device face -> reference id
    set_error("non-finite flux at face " + std::to_string(c->last_err_face));
    return BES_ERR_NAN;
  }
  return BES_OK;
}

int bes_implicit_assemble(bes_ctx *c, double cfl, int local, int repeat_nv, double *linf_b, double *linf_r) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  return assemble(c, impl_of(c), cfl, nullptr, local, repeat_nv, linf_b, linf_r);
}

// reference CoefficientMatrix layout: scalar CSR rows (cell, var) in reference
// cell order, each row = own block row then neighbour block rows in local face
// order (CoefficientMatrix.cpp:127-160).  rowptr [ncell*nv+1], col/val [nnz].
int bes_implicit_get_system(bes_ctx *c, long *rowptr, long *col, double *val, double *rhs) {
  if (!c || !c->impl || !impl_of(c)->assembled) { set_error("system not assembled"); return BES_ERR_ARG; }
  if (c->B != 1) { set_error("the CSR system is available for one condition (batch size 1)"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  const int N = c->N, nv = c->nv, k = c->k, NB = nv * nv;
  const size_t mat = (size_t)(k + 1) * NB * N;
  std::vector<double> A(mat);
  if (im->prec == 64) {
    BES_HIP(hipMemcpy(A.data(), im->A, mat * sizeof(double), hipMemcpyDeviceToHost));
  } else {
    std::vector<float> Af(mat);
    BES_HIP(hipMemcpy(Af.data(), im->A, mat * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t q = 0; q < mat; q++) A[q] = Af[q];
  }
  const Geometry &g = c->geo;
  long nz = 0, row = 0;
  for (int64_t e = 0; e < N; e++) {
    const int i = (int)c->iperm[e];
    for (int a = 0; a < nv; a++) {
      if (rowptr) rowptr[row] = nz;
      for (int bq = 0; bq < nv; bq++) {
        if (col) col[nz] = e * nv + bq;
        if (val) val[nz] = A[((size_t)0 * NB + a * nv + bq) * N + i];
        nz++;
      }
      for (int m = 0; m < k; m++) {
        const int64_t j = g.cadj[e * k + m];
        if (j < 0) continue;
        for (int bq = 0; bq < nv; bq++) {
          if (col) col[nz] = j * nv + bq;
          if (val) val[nz] = A[((size_t)(1 + m) * NB + a * nv + bq) * N + i];
          nz++;
        }
      }
      row++;
    }
  }
  if (rowptr) rowptr[row] = nz;
  if (rhs) {
    std::vector<double> b((size_t)N * nv);
    BES_HIP(hipMemcpy(b.data(), im->b, b.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int64_t e = 0; e < N; e++)
      for (int v = 0; v < nv; v++) rhs[e * nv + v] = b[(size_t)c->iperm[e] * nv + v];
  }
  return BES_OK;
}

// load a system assembled on the host in the reference CSR layout (the
// CoefficientMatrix::addToBlock / addToVal path, CoefficientMatrix.cpp:166-204)
int bes_implicit_set_system(bes_ctx *c, const double *val, const double *rhs) {
  if (!c || !c->impl || !val || !rhs) { set_error("call bes_implicit_setup first / null argument"); return BES_ERR_ARG; }
  if (c->B != 1) { set_error("a CSR system is loaded for one condition (batch size 1)"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  const int N = c->N, nv = c->nv, k = c->k, NB = nv * nv;
  const size_t mat = (size_t)(k + 1) * NB * N;
  std::vector<double> A(mat, 0.0), b((size_t)N * nv);
  const Geometry &g = c->geo;
  long nz = 0;
  for (int64_t e = 0; e < N; e++) {
    const int i = (int)c->iperm[e];
    for (int a = 0; a < nv; a++) {
      for (int bq = 0; bq < nv; bq++) A[((size_t)a * nv + bq) * N + i] = val[nz++];
      for (int m = 0; m < k; m++) {
        if (g.cadj[e * k + m] < 0) continue;
        for (int bq = 0; bq < nv; bq++) A[((size_t)(1 + m) * NB + a * nv + bq) * N + i] = val[nz++];
      }
    }
    for (int v = 0; v < nv; v++) b[(size_t)i * nv + v] = rhs[e * nv + v];
  }
  if (im->prec == 64) {
    BES_HIP(hipMemcpy(im->A, A.data(), mat * sizeof(double), hipMemcpyHostToDevice));
  } else {
    std::vector<float> Af(A.begin(), A.end());
    BES_HIP(hipMemcpy(im->A, Af.data(), mat * sizeof(float), hipMemcpyHostToDevice));
  }
  BES_HIP(hipMemcpy(im->b, b.data(), b.size() * sizeof(double), hipMemcpyHostToDevice));
  im->assembled = true;
  im->factored = false;
  return BES_OK;
}

long bes_implicit_nnz(bes_ctx *c) {
  if (!c) return -1;
  long nz = 0;
  for (int64_t e = 0; e < c->N; e++) {
    nz++;
    for (int m = 0; m < c->k; m++) if (c->geo.cadj[e * c->k + m] >= 0) nz++;
  }
  return nz * c->nv * c->nv;
}

static int solve_once(bes_ctx *c, Impl *im, int *it, double *rr) {
  int s;
  if (im->prec == 64) {
    if (!im->factored && (s = factor<double>(c, im))) return s;
    im->factored = true;
    return im->solver == 1 ? bicgstab<double, double>(c, im, it, rr) : gmres<double, double>(c, im, it, rr);
  }
  if (!im->factored && (s = factor<float>(c, im))) return s;
  im->factored = true;
  return im->solver == 1 ? bicgstab<float, float>(c, im, it, rr) : gmres<float, float>(c, im, it, rr);
}

int bes_linear_solve(bes_ctx *c, int *iters, double *relres) {
  if (!c || !c->impl || !impl_of(c)->assembled) { set_error("system not assembled"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  if (im->precond == 3 && !im->lp) { set_error("learned preconditioner not initialised (bes_lp_init)"); return BES_ERR_ARG; }
  int s;
  if (im->precond == 3 && im->lp_online_steps > 0) {   // online training on the system just assembled
    std::vector<double> lh(im->lp_online_steps);
    if ((s = bes_lp_train(c, im->lp_online_steps, im->lp_online_lr, im->lp_online_nprobe, im->lp_online_nrich,
                          im->lp_online_seed, lh.data())))
      return s;
    im->lp_online_seed += (unsigned long long)im->lp_online_steps;
    im->lp_online_loss = lh.back();
  }
  int it = 0;
  double rr = 0;
  if ((s = solve_once(c, im, &it, &rr))) return s;
  if (im->precond == 3 && !(rr <= im->rtol * 1.0001) && !(rr == 0)) {
    // the learned operator stalled: solve again with multicolour ILU(0)
    int it2 = 0;
    im->precond = 2;
    im->factored = false;
    s = solve_once(c, im, &it2, &rr);
    im->precond = 3;
    im->factored = false;
    im->lp_current = false;   // rebuild the operator for the next solve
    im->lp_fallbacks++;
    it += it2;
    if (s) return s;
  }
  if ((s = prof_collect(c))) return s;
  im->last_iters = it;
  im->last_relres = rr;
  if (iters) *iters = it;
  if (relres) *relres = rr;
  if (!(rr <= im->rtol * 1.0001) && !(rr == 0)) {
    set_error("linear solver stopped at relative residual " + std::to_string(rr));
    return BES_ERR_SOLVE;
  }
  return BES_OK;
}

int bes_get_linear_solution(bes_ctx *c, double *x) {
  if (!c || !c->impl || !x) { set_error("no solution"); return BES_ERR_ARG; }
  return vector_to_host(c, impl_of(c)->x, x);
}

int bes_amg_apply(bes_ctx *c, const double *r, double *z) {
  if (!c || !c->impl || !r || !z) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  if (c->B != 1) { set_error("the AMG takes one condition"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  if (im->precond != 4 || !im->assembled) { set_error("AMG apply needs precond 4 and an assembled system"); return BES_ERR_ARG; }
  int s;
  if (!im->factored) {
    if ((s = im->prec == 64 ? factor<double>(c, im) : factor<float>(c, im))) return s;
    im->factored = true;
  }
  const int N = c->N, nv = c->nv;
  const size_t n = (size_t)N * nv, vs = im->vstride;
  std::vector<double> h(n);
  for (int64_t e = 0; e < N; e++)
    for (int v = 0; v < nv; v++) h[(size_t)c->iperm[e] * nv + v] = r[e * nv + v];
  if (im->prec == 64) {
    double *Z = (double *)im->Z;
    BES_HIP(hipMemcpyAsync(Z, h.data(), n * sizeof(double), hipMemcpyHostToDevice, c->stream));
    if ((s = amg_apply<double>(c, im, Z, Z + vs, Z + 2 * vs))) return s;
    BES_HIP(hipMemcpyAsync(h.data(), Z + vs, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  } else {
    float *Z = (float *)im->Z;
    std::vector<float> hf(h.begin(), h.end());
    BES_HIP(hipMemcpyAsync(Z, hf.data(), n * sizeof(float), hipMemcpyHostToDevice, c->stream));
    if ((s = amg_apply<float>(c, im, Z, Z + vs, Z + 2 * vs))) return s;
    BES_HIP(hipMemcpyAsync(hf.data(), Z + vs, n * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    BES_HIP(hipStreamSynchronize(c->stream));
    std::copy(hf.begin(), hf.end(), h.begin());
  }
  BES_HIP(hipStreamSynchronize(c->stream));
  for (int64_t e = 0; e < N; e++)
    for (int v = 0; v < nv; v++) z[e * nv + v] = h[(size_t)c->iperm[e] * nv + v];
  return BES_OK;
}

// U += x for the conditions whose active flag is set (all when active is null)
static int update(bes_ctx *c, Impl *im, const std::vector<char> *active) {
  const int bs = tuned_bs(c, kProfUpdate), B = c->B;
  CoefB act;
  for (int b = 0; b < B; b++) act.c[b] = (!active || (*active)[b]) ? 1.0 : 0.0;
  {
    ProfScope ps(c, kProfUpdate, 24.0 * c->N * c->nv * B);
    if (c->nd == 2)
      hipLaunchKernelGGL(k_update<2>, dim3(grid_for(c->N * B, bs)), dim3(bs), 0, c->stream, c->U0, im->x, c->N, c->lgB,
                         act);
    else
      hipLaunchKernelGGL(k_update<3>, dim3(grid_for(c->N * B, bs)), dim3(bs), 0, c->stream, c->U0, im->x, c->N, c->lgB,
                         act);
  }
  BES_HIP(hipGetLastError());
  BES_HIP(hipStreamSynchronize(c->stream));
  return prof_collect(c);
}

int bes_implicit_update(bes_ctx *c) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  return update(c, impl_of(c), nullptr);
}

// SolverImplicit::solve loop (SolverImplicit.cpp:552-600) with the adaptive
// Courant number of SolverImplicit.cpp:530-550, for every condition of the
// batch at once: each keeps its own Courant number, residual history and stop;
// a condition that has reached its drop is frozen (no solve, no update) while
// the others go on.  hist [nsteps][B][2*nv+3]: Linf(b) per var, Linf(sum F*A)
// per var, CFL used, Krylov iterations, relres (NaN rows for frozen conditions).
static int run_steps(bes_ctx *c, Impl *im, int nsteps, double *hist, int *steps_done) {
  const int nv = c->nv, B = c->B, hw = 2 * nv + 3;
  Impl::Run &R = im->run;
  std::vector<double> lb((size_t)B * nv), lr((size_t)B * nv);
  std::vector<char> go(B);
  int done = 0;
  for (int it = 0; it < nsteps && !R.reached; it++) {
    for (int b = 0; b < B; b++) go[b] = !R.done[b];
    im->skip_b.assign(R.done.begin(), R.done.end());
    int s = assemble(c, im, 0.0, R.cfl.data(), R.local, R.repeat_nv, lb.data(), lr.data());
    if (s) { im->skip_b.clear(); if (steps_done) *steps_done = done; return s; }
    int iters = 0;
    double rr = 0;
    s = bes_linear_solve(c, &iters, &rr);
    im->skip_b.clear();
    if (s && s != BES_ERR_SOLVE) { if (steps_done) *steps_done = done; return s; }
    if ((s = update(c, im, &go))) { if (steps_done) *steps_done = done; return s; }
    done = it + 1;
    bool all = true;
    for (int b = 0; b < B; b++) {
      const double *lbb = &lb[(size_t)b * nv], *lrb = &lr[(size_t)b * nv];
      if (hist) {
        double *h = hist + ((size_t)it * B + b) * hw;
        if (!go[b]) {
          for (int q = 0; q < hw; q++) h[q] = std::nan("");
        } else {
          for (int v = 0; v < nv; v++) { h[v] = lbb[v]; h[nv + v] = lrb[v]; }
          h[2 * nv] = R.cfl[b];
          h[2 * nv + 1] = B == 1 ? iters : im->iters_b[b];
          h[2 * nv + 2] = B == 1 ? rr : im->relres_b[b];
        }
      }
      if (go[b]) {
        R.steps[b]++;
        if (R.r0[b] < 0) R.r0[b] = lrb[0];
        // limiter freeze: from the step whose density residual first reaches
        // the freeze drop on, the condition keeps the limiter of that step's
        // gradient pass (stored by it in phi_frz)
        if (c->lim_freeze_drop > 0 && b < (int)c->lim_frozen.size() && !c->lim_frozen[b] && R.r0[b] > 0 &&
            lrb[0] <= c->lim_freeze_drop * R.r0[b]) {
          c->lim_frozen[b] = 1;
          c->lim_epoch++;
        }
        // adaptive Courant number (density monitor of the implicit residual)
        if (R.cfl_max > R.cfl_min) {
          double &lo = R.lb_old[(size_t)b * nv];
          const int ei = (lo > lbb[0]) ? 1 : 0;
          double cf = R.cfl[b] * std::pow(lo / lbb[0], R.ex[ei]);
          cf = std::max(R.cfl_min, cf);
          R.cfl[b] = std::min(R.cfl_max, cf);
        }
        std::copy(lbb, lbb + nv, R.lb_old.begin() + (size_t)b * nv);
        if (R.stop_drop > 0 && R.r0[b] > 0 && lrb[0] <= R.stop_drop * R.r0[b]) R.done[b] = 1;
      }
      all = all && R.done[b];
    }
    R.reached = all;
  }
  if (steps_done) *steps_done = done;
  return BES_OK;
}

int bes_implicit_run(bes_ctx *c, int nsteps, double cfl_min, double cfl_max, const double *exponents, int local,
                     int repeat_nv, double stop_drop, double *hist, int *steps_done) {
  if (!c || !c->impl || nsteps < 0 || !exponents) { set_error("invalid argument"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  Impl::Run &R = im->run;
  R = Impl::Run();
  R.active = true;
  R.cfl_min = cfl_min;
  R.cfl.assign(c->B, cfl_min);
  R.r0.assign(c->B, -1.0);
  R.done.assign(c->B, 0);
  R.steps.assign(c->B, 0);
  R.cfl_max = cfl_max;
  R.ex[0] = exponents[0];
  R.ex[1] = exponents[1];
  R.local = local;
  R.repeat_nv = repeat_nv;
  R.stop_drop = stop_drop;
  R.lb_old.assign((size_t)c->B * c->nv, 0.0);
  return run_steps(c, im, nsteps, hist, steps_done);
}

int bes_autotune(bes_ctx *c, int flags, int *chosen, double *best_us, int *coloring) {
  if (!c || flags < 0 || flags > 7) { set_error("invalid autotune request (flags 0-7)"); return BES_ERR_ARG; }
  Impl *im = (Impl *)c->impl;
  if ((flags & 6) && !(im && im->assembled)) { set_error("implicit autotuning needs an assembled system"); return BES_ERR_ARG; }
  if ((flags & 6) && (im->precond == 3 || im->precond == 4)) {
    set_error("implicit autotuning covers precond 0-2");
    return BES_ERR_ARG;
  }
  BES_HIP(hipStreamSynchronize(c->stream));
  const bool prof = c->prof;
  c->prof = false;
  if (c->graph) { hipGraphExecDestroy(c->graph); c->graph = nullptr; }   // launches captured with old sizes
  const int cand[3] = {64, 128, 256};
  double best[bes_ctx::kProfKinds];
  for (int k = 0; k < bes_ctx::kProfKinds; k++) best[k] = 0;
  int s = BES_OK;
  // fixed: the launch does not take the kind's block size at the context's size
  // (it is timed, the size kept)
  auto tune = [&](int kind, auto fn, bool fixed = false) -> int {
    if (fixed) return time_us(c, 5, fn, &best[kind]);
    double bt = 1e300;
    int bb = 256;
    for (int bs : cand) {
      c->tune_bs[kind] = bs;
      double us = 0;
      int st = time_us(c, 5, fn, &us);
      if (st) return st;
      if (us < bt) { bt = us; bb = bs; }
    }
    c->tune_bs[kind] = bb;
    best[kind] = bt;
    return BES_OK;
  };
  if (!s && (flags & 2)) {   // implicit kernels on the assembled system (re-assembled, re-factored: same values)
    const bool p64 = im->prec == 64;
    auto asmb = [&]() { return p64 ? launch_assemble<double>(c, im) : launch_assemble<float>(c, im); };
    auto fact = [&]() { return p64 ? factor<double>(c, im) : factor<float>(c, im); };
    s = tune(kProfJacobian, asmb);
    if (!s) s = tune(kProfAssemble, asmb);
    if (!s) s = tune(kProfFactor, fact);
    if (!s) {
      const size_t vs = im->vstride;
      const bool slots = slot_split(c), sweeps = im->precond == 2 && slots;
      if (p64) {
        double *V = (double *)im->V, *Z = (double *)im->Z;
        s = tune(kProfSpmv, [&]() { return spmv<double, double>(c, im, V, V + vs); }, slots);
        if (!s) s = tune(kProfPrecond, [&]() { return precond_apply<double, double>(c, im, V, Z, Z + vs); }, sweeps);
      } else {
        float *V = (float *)im->V, *Z = (float *)im->Z;
        s = tune(kProfSpmv, [&]() { return spmv<float, float>(c, im, V, V + vs); }, slots);
        if (!s) s = tune(kProfPrecond, [&]() { return precond_apply<float, float>(c, im, V, Z, Z + vs); }, sweeps);
      }
    }
    im->factored = false;
  }
  if (!s && (flags & 4) && im->precond == 2) {   // ILU(0) colouring: the fastest solve of this system
    double bt = 1e300;
    int bm = im->coloring;
    for (int mode = 0; mode <= 2 && !s; mode++) {
      if ((s = build_colouring(c, im, mode))) break;
      int it = 0;
      double rr = 0;
      auto t0 = std::chrono::steady_clock::now();
      s = solve_once(c, im, &it, &rr);
      BES_HIP(hipStreamSynchronize(c->stream));
      const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
      if (us < bt) { bt = us; bm = mode; }
    }
    if (!s) s = build_colouring(c, im, bm);
    if (coloring) *coloring = bm;
  }
  if (!s && (flags & 1)) {   // explicit kernels on the current state, last: the time step it leaves is at CFL 1
    // (U0 is read, never written; the next assembly or explicit step recomputes dt)
    s = tune(kProfGradlim, [&]() { return launch_gradlim(c, c->U0, nullptr, nullptr); }, split_pass(c));
    if (!s) s = tune(kProfTimestep, [&]() { return launch_timestep(c, c->U0, 1.0, 1); });
    if (!s) s = tune(kProfFaceFlux, [&]() { return launch_face_flux(c); });
    if (!s)
      s = tune(kProfResidual, [&]() { return launch_residual(c, nullptr, nullptr, 0.0, 1, nullptr, nullptr); },
               split_pass(c));
  }
  if (!s) BES_HIP(hipStreamSynchronize(c->stream));
  c->prof = prof;
  if (chosen)
    for (int k = 0; k < bes_ctx::kProfKinds; k++) chosen[k] = tuned_bs(c, k);
  if (best_us)
    for (int k = 0; k < bes_ctx::kProfKinds; k++) best_us[k] = best[k];
  return s;
}

int bes_implicit_batch_state(bes_ctx *c, int *steps, int *reached, double *cfl, int *iters, double *relres) {
  if (!c || !c->impl) { set_error("call bes_implicit_setup first"); return BES_ERR_ARG; }
  Impl *im = impl_of(c);
  const Impl::Run &R = im->run;
  for (int b = 0; b < c->B; b++) {
    if (steps) steps[b] = R.active ? R.steps[b] : 0;
    if (reached) reached[b] = R.active ? R.done[b] : 0;
    if (cfl) cfl[b] = R.active ? R.cfl[b] : 0.0;
    if (iters) iters[b] = b < (int)im->iters_b.size() ? im->iters_b[b] : 0;
    if (relres) relres[b] = b < (int)im->relres_b.size() ? im->relres_b[b] : 0.0;
  }
  return BES_OK;
}

int bes_implicit_continue(bes_ctx *c, int nsteps, double *hist, int *steps_done, int *reached) {
  if (!c || !c->impl || nsteps < 0 || !impl_of(c)->run.active) {
    set_error("no pseudo-time loop to continue (bes_implicit_run first)");
    return BES_ERR_ARG;
  }
  Impl *im = impl_of(c);
  int s = run_steps(c, im, nsteps, hist, steps_done);
  if (reached) *reached = im->run.reached ? 1 : 0;
  return s;
}

}  // extern "C"
