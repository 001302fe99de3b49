// ecsim_field.hip — the implicit ECSIM field equation on the device, over the
// J and M that the deposit leaves resident (one NODE_STRIDE row per node).
//
// The unknown is dE = (E^{n+theta} - E^n) E_conv at the corner nodes of a
// single-level mesh.  Per node n and component iVar (GetStencil_Legacy,
// src/pic/pic_field_solver_ecsim.cpp:740-1228; UpdateMatrixElement
// :6004-6016):
//   (A x)[n][iVar] = sum over iVarIndex, then over the 27 neighbour slots s of
//                    (K[iVar][iVarIndex][s] + M_n[9s + 3iVar + iVarIndex] 4 pi dt theta)
//                    x[nbr(n, s)][iVarIndex]
// with K = identity - coeff^2 Laplacian + coeff coeff grad-div (the
// 27-point stencils the reference composes from edge averages, :7185-7300,
// coeff = c dt theta / dx); neighbours outside the domain or on its boundary
// are dropped (:1032), and a corner on the domain boundary is a row of the
// identity with a zero right-hand side (:782-799).  The right-hand side is
// UpdateRhs_Legacy (:6040-6137): the neighbours' E^n times the opposite
// Laplacian / grad-div coefficients, the mass term times -4 pi dt theta, the
// node's J times -4 pi dt theta and the 16 cell-centred B terms of curl B
// (:1234-1375).  The coefficient tables are built on the host in the
// reference's loop order and every sum runs in the reference's order, so the
// operator, the right-hand side and the B update are bit-exact with the
// oracle's restatement.
//
// The system is solved by restarted GMRES (modified Gram-Schmidt, zero
// initial guess as SetInitialGuess :6296-6301, stop at ||r|| <= tol ||b||):
// vectors, the Krylov basis and the Hessenberg matrix with its rotations stay
// on the device, inner products are fixed-order two-stage reductions (the
// same bits on every run), and the host looks at the state every few steps.
// ProcessFinalSolution (:6311-6318), UpdateE (:5909-5960) and UpdateB
// (:5160-5270) complete a time step.  The reference's solver is SWMF's
// linear_solver_wrapper("GMRES") (srcInterface/LinearSystemCornerNode.h:3282),
// not part of the tree: its iteration count is not reproduced, its converged
// solution is (to the tolerance).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <array>
#include <vector>

#include "amps_common.h"

using namespace amps;

namespace {

constexpr double PI_REF = 3.14159265358979323846;  // Pi of src/general/constants.h
constexpr int RED_BLOCKS = 1024;
constexpr int RED_THREADS = 256;

// curl-B entries of UpdateRhs_Legacy per row component iVar: (coefficient
// axis, sign, ci, cj, ck) of the cell node + (ci, cj, ck); the first 8 take
// B component (iVar + 2) % 3, the next 8 (iVar + 4) % 3 (:1234-1375, groups
// of 4 in the reference's ii-outer / jj-inner order)
__constant__ int c_curlb[3][16][5] = {
    {{1, 1, -1, 0, -1}, {1, 1, -1, 0, 0}, {1, 1, 0, 0, -1}, {1, 1, 0, 0, 0}, {1, -1, -1, -1, -1},
     {1, -1, -1, -1, 0}, {1, -1, 0, -1, -1}, {1, -1, 0, -1, 0}, {2, -1, -1, -1, 0}, {2, -1, -1, 0, 0},
     {2, -1, 0, -1, 0}, {2, -1, 0, 0, 0}, {2, 1, -1, -1, -1}, {2, 1, -1, 0, -1}, {2, 1, 0, -1, -1},
     {2, 1, 0, 0, -1}},
    {{2, 1, -1, -1, 0}, {2, 1, -1, 0, 0}, {2, 1, 0, -1, 0}, {2, 1, 0, 0, 0}, {2, -1, -1, -1, -1},
     {2, -1, -1, 0, -1}, {2, -1, 0, -1, -1}, {2, -1, 0, 0, -1}, {0, -1, 0, -1, -1}, {0, -1, 0, 0, -1},
     {0, -1, 0, -1, 0}, {0, -1, 0, 0, 0}, {0, 1, -1, -1, -1}, {0, 1, -1, 0, -1}, {0, 1, -1, -1, 0},
     {0, 1, -1, 0, 0}},
    {{0, 1, 0, -1, -1}, {0, 1, 0, 0, -1}, {0, 1, 0, -1, 0}, {0, 1, 0, 0, 0}, {0, -1, -1, -1, -1},
     {0, -1, -1, 0, -1}, {0, -1, -1, -1, 0}, {0, -1, -1, 0, 0}, {1, -1, -1, 0, -1}, {1, -1, 0, 0, -1},
     {1, -1, -1, 0, 0}, {1, -1, 0, 0, 0}, {1, 1, -1, -1, -1}, {1, 1, 0, -1, -1}, {1, 1, -1, -1, 0},
     {1, 1, 0, -1, 0}}};

struct Coefs {
  double K[3][3][27];  // operator constants [iVar][iVarIndex][slot]
  double R[3][3][27];  // E^n coefficients of the right-hand side
  double coeff[3];     // c dt theta / dx
};

int slot_of(int di, int dj, int dk) {
  auto a = [](int d) { return d == 0 ? 0 : (d == -1 ? 1 : 2); };
  return a(di) + 3 * a(dj) + 9 * a(dk);
}

// The Laplacian and grad-div stencils as the reference composes them; every
// entry is a dyadic fraction, so the merge order does not change a bit.
using St = std::map<std::array<int, 3>, double>;
void st_add(St& st, const St& o, int di, int dj, int dk, double f) {
  for (const auto& e : o) st[{e.first[0] + di, e.first[1] + dj, e.first[2] + dk}] += f * e.second;
}

void stencils(St lap[3], St gd[3][3]) {
  auto edge = [](std::vector<int> ir, std::vector<int> jr, std::vector<int> kr) {
    St s;
    for (int i : ir)
      for (int j : jr)
        for (int k : kr) s[{i, j, k}] = 0.25;
    return s;
  };
  const St xe0 = edge({0}, {-1, 0}, {-1, 0}), xe4 = edge({-1, 0}, {0}, {-1, 0}), xe8 = edge({-1, 0}, {-1, 0}, {0});
  St f0;
  st_add(f0, xe0, 1, 0, 0, 1.0);
  st_add(f0, xe0, 0, 0, 0, -2.0);
  st_add(f0, xe0, -1, 0, 0, 1.0);
  St dxx;
  for (int i = 0; i < 2; i++)
    for (int j = 0; j < 2; j++) st_add(dxx, f0, 0, i, j, 0.25);
  St dyy, dzz;
  for (const auto& e : dxx) {
    dyy[{e.first[1], e.first[0], e.first[2]}] = e.second;
    dzz[{e.first[2], e.first[1], e.first[0]}] = e.second;
  }
  St dy0 = xe4, dz0 = xe8;
  st_add(dy0, xe4, 0, -1, 0, -1.0);
  st_add(dz0, xe8, 0, 0, -1, -1.0);
  St dxy, dxz, dyz;
  for (int l = 0; l < 2; l++)
    for (int m = 0; m < 2; m++) {
      st_add(dxy, dy0, 1, l, m, 0.25);
      st_add(dxy, dy0, 0, l, m, -0.25);
      st_add(dxz, dz0, 1, l, m, 0.25);
      st_add(dxz, dz0, 0, l, m, -0.25);
      st_add(dyz, dz0, l, 1, m, 0.25);
      st_add(dyz, dz0, l, 0, m, -0.25);
    }
  lap[0] = dxx, lap[1] = dyy, lap[2] = dzz;
  gd[0][0] = dxx, gd[0][1] = dxy, gd[0][2] = dxz;
  gd[1][0] = dxy, gd[1][1] = dyy, gd[1][2] = dyz;
  gd[2][0] = dxz, gd[2][1] = dyz, gd[2][2] = dzz;
}

// the row tables in the reference's accumulation order (GetStencil_Legacy
// :873-910 for the matrix, :1152-1185 for the right-hand side)
Coefs coefficients(const double dx[3], const amps_ecsim_params& p) {
  Coefs C{};
  double coeffSqr[3];
  for (int d = 0; d < 3; d++) {
    const double dxd = dx[d] * p.length_conv;
    C.coeff[d] = p.cDt / dxd * p.theta;
    coeffSqr[d] = C.coeff[d] * C.coeff[d];
  }
  St lap[3], gd[3][3];
  stencils(lap, gd);
  for (int iVar = 0; iVar < 3; iVar++) {
    for (int idim = 0; idim < 3; idim++)
      for (const auto& e : lap[idim]) {
        const int s = slot_of(e.first[0], e.first[1], e.first[2]);
        C.K[iVar][iVar][s] -= e.second * coeffSqr[idim];
        C.R[iVar][iVar][s] += e.second * coeffSqr[idim];
      }
    C.K[iVar][iVar][0] += 1;
    for (int iv = 0; iv < 3; iv++)
      for (const auto& e : gd[iVar][iv]) {
        const int s = slot_of(e.first[0], e.first[1], e.first[2]);
        C.K[iVar][iv][s] += (1 - 0.0) * e.second * C.coeff[iVar] * C.coeff[iv];
        C.R[iVar][iv][s] -= (1 - 0.0) * e.second * C.coeff[iVar] * C.coeff[iv];
      }
  }
  return C;
}

// ---------------------------------------------------------------------------
// kernels: one thread per (node, component) row
// ---------------------------------------------------------------------------
// Eight nodes per workgroup, two per wavefront (as the mass term of
// ecsim.hip): lane s (0..26) of each half reads slot s of its node's M row (72
// contiguous bytes, consecutive lanes) and its neighbour's x, and writes the
// 9 products (K + M 4 pi dt theta) x of the slot to LDS; then 24 lanes, one
// per (node, component) row, add the row's 81 products in the row's element
// order (iVarIndex outer, slot inner), skipping the dropped neighbours.
__global__ __launch_bounds__(256) void k_ecsim_op(int64_t nn, const double* __restrict__ rows,
                                                  const int* __restrict__ nbr, const uint8_t* __restrict__ bnd,
                                                  const Coefs* __restrict__ C, double fpdt,
                                                  const double* __restrict__ x, double* __restrict__ y) {
  __shared__ double term[8][3][3][27];
  __shared__ uint64_t present[4];
  const int64_t per = gridDim.x >> 3;
  const int64_t chunk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (chunk * 8 >= nn) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int half = lane >> 5, s = lane & 31;
  const int ln = wave * 2 + half;
  const int64_t n = chunk * 8 + ln;
  const bool act = n < nn && s < 27;
  bool keep = false;
  if (act) {
    const int j = nbr[n * 27 + s];
    keep = j >= 0 && !bnd[j];
    if (keep) {
      const double* m = rows + n * NODE_STRIDE + 3 + 9 * s;
      const double* xj = x + 3 * (int64_t)j;
      const double xv[3] = {xj[0], xj[1], xj[2]};
#pragma unroll
      for (int iVar = 0; iVar < 3; iVar++)
#pragma unroll
        for (int iv = 0; iv < 3; iv++) {
          const double val = C->K[iVar][iv][s] + m[3 * iVar + iv] * fpdt;
          term[ln][iVar][iv][s] = val * xv[iv];
        }
    }
  }
  const uint64_t pm = __ballot(keep);
  if (lane == 0) present[wave] = pm;
  __syncthreads();
  if (threadIdx.x < 24) {
    const int r = threadIdx.x / 3, iVar = threadIdx.x - 3 * r;
    const int64_t nr = chunk * 8 + r;
    if (nr < nn) {
      double out;
      if (bnd[nr]) {
        out = x[3 * nr + iVar];
      } else {
        const uint64_t p = present[r >> 1] >> (32 * (r & 1));
        double acc = 0.0;
        for (int iv = 0; iv < 3; iv++)
          for (int q = 0; q < 27; q++)
            if ((p >> q) & 1) acc = acc + term[r][iVar][iv][q];
        out = acc;
      }
      y[3 * nr + iVar] = out;
    }
  }
}

// Eight nodes per workgroup, two per wavefront, as the operator above: the
// lane of slot s forms its slot's stencil and mass term for the three rows,
// other lanes the 16 curl-B terms of a row, all parked in LDS; then 24 lanes,
// one per row, add them in the reference's order.  Bound by HBM (the M row,
// 1,944 B a node): 1.30 ms at 2.15 M nodes, 1.52 with a lane walking its row.
__global__ __launch_bounds__(256) void k_ecsim_rhs(int64_t nn, const double* __restrict__ rows,
                                                   const int* __restrict__ nbr, const uint8_t* __restrict__ bnd,
                                                   const int* __restrict__ cells8, const Coefs* __restrict__ C,
                                                   double dtTotal, double theta, double E_conv, double B_conv,
                                                   const double* __restrict__ En, const double* __restrict__ Bc,
                                                   double* __restrict__ out) {
  __shared__ double term[8][3][2 * 27 + 17];  // stencil, mass and curl-B terms of a row, padded
  const int64_t per = gridDim.x >> 3;
  const int64_t chunk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (chunk * 8 >= nn) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int s = lane & 31;
  const int ln = wave * 2 + (lane >> 5);
  const int64_t n = chunk * 8 + ln;
  const double fpdt = 4 * PI_REF * dtTotal * theta;
  if (n < nn && s < 27 && !bnd[n]) {
    const double* e = En + 3 * (int64_t)nbr[n * 27 + s];
    const double* M = rows + n * NODE_STRIDE + 3 + 9 * s;
    const double e0 = e[0], e1 = e[1], e2 = e[2];
#pragma unroll
    for (int iVar = 0; iVar < 3; iVar++) {
      const double* m = M + 3 * iVar;
      term[ln][iVar][s] = (e0 * C->R[iVar][0][s] + e1 * C->R[iVar][1][s] + e2 * C->R[iVar][2][s]) * E_conv;
      term[ln][iVar][27 + s] = (e0 * m[0] + e1 * m[1] + e2 * m[2]) * (-fpdt) * E_conv;
    }
  }
  for (int i = threadIdx.x; i < 8 * 3 * 16; i += 256) {
    const int ln2 = i / 48, iVar = (i / 16) % 3, t = i & 15;
    const int64_t n2 = chunk * 8 + ln2;
    if (n2 < nn && !bnd[n2]) {
      const int* e = c_curlb[iVar][t];
      const int comp = t < 8 ? (iVar + 2) % 3 : (iVar + 4) % 3;
      const int cell = cells8[n2 * 8 + (e[2] + 1) + 2 * (e[3] + 1) + 4 * (e[4] + 1)];
      const double c4 = 0.25 * C->coeff[e[0]];
      term[ln2][iVar][54 + t] = Bc[3 * (int64_t)cell + comp] * (e[1] > 0 ? c4 : -c4) * B_conv;
    }
  }
  __syncthreads();
  if (threadIdx.x < 24) {
    const int r = threadIdx.x / 3, iVar = threadIdx.x - 3 * r;
    const int64_t nr = chunk * 8 + r;
    if (nr < nn) {
      double res = 0.0;
      if (!bnd[nr]) {
        const double* t = term[r][iVar];
        for (int q = 0; q < 54; q++) res += t[q];
        res += rows[nr * NODE_STRIDE + iVar] * (-4 * PI_REF * dtTotal * theta);
        for (int q = 54; q < 70; q++) res += t[q];
      }
      out[3 * nr + iVar] = res;
    }
  }
}

// E^{n+theta} = dE / E_conv + E^n; E^{n+1} = (E^{n+theta} - (1 - theta) E^n) / theta
__global__ __launch_bounds__(256) void k_ecsim_update_e(int64_t n3, const double* __restrict__ En,
                                                        const double* __restrict__ dE, double theta, double E_conv,
                                                        double* __restrict__ Eth, double* __restrict__ E1) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n3) return;
  const double th = dE[i] / E_conv + En[i];
  Eth[i] = th;
  E1[i] = (th - (1.0 - theta) * En[i]) / theta;
}

// UpdateB for every cell: one thread per cell, the 2x2 face averages of the
// corner E^{n+theta} (coefficients coeff4 = c dt / dx / 4, no theta)
__global__ __launch_bounds__(256) void k_ecsim_update_b(int64_t ncell, const int* __restrict__ noc,
                                                        const double* __restrict__ Eth,
                                                        const double* __restrict__ Bc, double c40, double c41,
                                                        double c42, double E_conv, double B_conv,
                                                        double* __restrict__ Bout) {
  const int64_t cid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (cid >= ncell) return;
  const int64_t b = cid / NCELL;
  const int lc = (int)(cid - b * NCELL);
  const int i = lc % NC, j = (lc / NC) % NC, k = lc / (NC * NC);
  double Ex[2][2][2], Ey[2][2][2], Ez[2][2][2];
  for (int kk = 0; kk < 2; kk++)
    for (int jj = 0; jj < 2; jj++)
      for (int ii = 0; ii < 2; ii++) {
        const int64_t nd = noc[b * NCORNER + (i + ii) + NN * ((j + jj) + NN * (k + kk))];
        Ex[ii][jj][kk] = Eth[3 * nd] * E_conv;
        Ey[ii][jj][kk] = Eth[3 * nd + 1] * E_conv;
        Ez[ii][jj][kk] = Eth[3 * nd + 2] * E_conv;
      }
  double t0 = 0.0, t1 = 0.0, t2 = 0.0;
  for (int p = 0; p < 2; p++)
    for (int q = 0; q < 2; q++) t0 += -c41 * (Ez[p][1][q] - Ez[p][0][q]) + c42 * (Ey[p][q][1] - Ey[p][q][0]);
  for (int p = 0; p < 2; p++)
    for (int q = 0; q < 2; q++) t1 += -c42 * (Ex[p][q][1] - Ex[p][q][0]) + c40 * (Ez[1][p][q] - Ez[0][p][q]);
  for (int p = 0; p < 2; p++)
    for (int q = 0; q < 2; q++) t2 += -c40 * (Ey[1][p][q] - Ey[0][p][q]) + c41 * (Ex[p][1][q] - Ex[p][0][q]);
  Bout[3 * cid] = Bc[3 * cid] + t0 / B_conv;
  Bout[3 * cid + 1] = Bc[3 * cid + 1] + t1 / B_conv;
  Bout[3 * cid + 2] = Bc[3 * cid + 2] + t2 / B_conv;
}

// ---------------------------------------------------------------------------
// The solver's operator: symmetric storage, one plane per matrix entry
// ---------------------------------------------------------------------------
// On a single-level mesh the nodes are the points of an N^3 lattice in x, y, z
// order, and the block of row n at slot s equals, bit for bit, the block of
// row n + offset(s) at the opposite slot: both sum the same products of the
// shared cells in the same order, K is even in the offset.  So 14 of the 27
// blocks (offset 0 and those "ahead" in lattice order) carry the matrix; they
// are packed once per solve as planes A[14][9][np] of K + 4 pi dt theta M,
// which consecutive lanes read as consecutive doubles, for a neighbour's
// block as for their own.  The operator is bound by HBM: 1,008 B per node
// instead of the 1,944 B of the node rows; blocks behind come out of the
// caches (one lattice plane of rows is 17 MB at 129^3).  At 2.15 M nodes an
// application takes 0.51 ms against 1.07 from the node rows; packing takes
// 1.7 ms, a solve has some 20 applications.
constexpr int SYM = 14;
__constant__ int c_ahead[SYM] = {0, 2, 6, 7, 8, 18, 19, 20, 21, 22, 23, 24, 25, 26};
// slots ahead are those with (dz, dy, dx) > 0 in that order
__host__ __device__ constexpr int off1(int a) { return a == 0 ? 0 : (a == 1 ? -1 : 1); }
__host__ __device__ constexpr int opposite(int s) {
  const int o[3] = {0, 2, 1};
  return o[s % 3] + 3 * o[(s / 3) % 3] + 9 * o[s / 9];
}
__host__ __device__ constexpr int ahead_index(int s) {
  return s == 0 ? 0 : s == 2 ? 1 : (s >= 6 && s <= 8) ? s - 4 : s >= 18 ? s - 13 : -1;
}

// 32 nodes per workgroup through LDS: row runs in, 32-node plane runs out
__global__ __launch_bounds__(256) void k_sym_pack(int64_t nn, int64_t np, const double* __restrict__ rows,
                                                  const Coefs* __restrict__ C, double fpdt, double* __restrict__ A) {
  __shared__ double T[SYM * 9][33];
  const int64_t n0 = (int64_t)blockIdx.x * 32;
#pragma unroll 8
  for (int i = threadIdx.x; i < 32 * SYM * 9; i += 256) {
    const int t = i / (SYM * 9), e = i - t * (SYM * 9);
    const int k = e / 9, c = e - 9 * k;
    if (n0 + t < nn) {
      const int s = c_ahead[k];
      T[e][t] = C->K[c / 3][c % 3][s] + rows[(n0 + t) * NODE_STRIDE + 3 + 9 * s + c] * fpdt;
    }
  }
  __syncthreads();
#pragma unroll 8
  for (int i = threadIdx.x; i < 32 * SYM * 9; i += 256) {
    const int e = i >> 5, t = i & 31;
    if (n0 + t < nn) A[(int64_t)e * np + n0 + t] = T[e][t];
  }
}

// Solver state on the device; scale[j] = 1 / ||W_j||, the basis vector is
// V_j = scale[j] W_j.
struct GmresState {
  double bnorm, res, last;
  int done, k, it, pad;
};

// y = A x on vectors [3][nn].  Each thread a node (rows 3) or one component
// of it (blockIdx.y, rows 1: three times the threads where the nodes alone
// leave the chip idle); neighbours on the boundary are dropped (MASK: their
// x need not be zero).
template <int ROWS, bool MASK>
__global__ __launch_bounds__(256) void k_sym_op(int64_t nn, int64_t np, int N, const double* __restrict__ A,
                                                const double* __restrict__ x, double* __restrict__ y,
                                                const GmresState* __restrict__ st) {
#pragma clang fp contract(fast)
  if (st && st->done) return;
  const int64_t per = gridDim.x >> 3;
  const int64_t n = ((int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3)) * 256 + threadIdx.x;
  if (n >= nn) return;
  const int r0 = ROWS == 3 ? 0 : blockIdx.y;
  const int ix = (int)(n % N), iy = (int)((n / N) % N), iz = (int)(n / ((int64_t)N * N));
  if (ix == 0 || iy == 0 || iz == 0 || ix == N - 1 || iy == N - 1 || iz == N - 1) {
#pragma unroll
    for (int r = 0; r < ROWS; r++) y[(r0 + r) * nn + n] = x[(r0 + r) * nn + n];
    return;
  }
  double acc[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; r++) acc[r] = 0.0;
#pragma unroll
  for (int q = 0; q < 27; q++) {
    const int dx = off1(q % 3), dy = off1((q / 3) % 3), dz = off1(q / 9);
    const int64_t j = n + dx + (int64_t)N * (dy + (int64_t)N * dz);
    bool keep = true;
    if (MASK)
      keep = !((dx < 0 && ix == 1) || (dx > 0 && ix == N - 2) || (dy < 0 && iy == 1) || (dy > 0 && iy == N - 2) ||
               (dz < 0 && iz == 1) || (dz > 0 && iz == N - 2));
    const bool own = ahead_index(q) >= 0;
    const double* a = A + (int64_t)(own ? ahead_index(q) : ahead_index(opposite(q))) * 9 * np + (own ? n : j);
#pragma unroll
    for (int iv = 0; iv < 3; iv++) {
      double xv = x[iv * nn + j];
      if (MASK && !keep) xv = 0.0;
#pragma unroll
      for (int r = 0; r < ROWS; r++) acc[r] += a[(int64_t)(3 * (r0 + r) + iv) * np] * xv;
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; r++) y[(r0 + r) * nn + n] = acc[r];
}

// ---------------------------------------------------------------------------
// GMRES steps: fixed-order two-stage reductions, no host round trip
// ---------------------------------------------------------------------------
// An Arnoldi step is one pass over the basis for all inner products, W_j . y
// and W_j . W_k (y = A W_k), and one for the new vector and its norm.  The
// coefficients are those of modified Gram-Schmidt, from the triangular system
// (I + L) h = r with L the strictly lower part of V^T V: the same vectors to
// rounding, where one product and one update after another read the basis
// two and a half times as often and took two launches a vector.  Bound by
// HBM at large meshes (2.15 M nodes, 17 steps: 10.5 ms of products and
// updates before, 3.9 now), by launches at small ones (650 a solve before,
// 120 now, at 35,937 nodes).
constexpr int GS_W = 8;  // basis vectors of a workgroup's inner products

// the workgroup's sums of v[NV], in v of thread 0
template <int NV>
__device__ __forceinline__ void block_sums(double* v) {
  __shared__ double s[RED_THREADS / 64][NV];
#pragma unroll
  for (int i = 0; i < NV; i++)
    for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_down(v[i], o);
  if ((threadIdx.x & 63) == 0)
    for (int i = 0; i < NV; i++) s[threadIdx.x >> 6][i] = v[i];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = 0; i < NV; i++) {
      v[i] = s[0][i];
      for (int w = 1; w < RED_THREADS / 64; w++) v[i] += s[w][i];
    }
}

// one wavefront's fixed-order sum of n values
__device__ __forceinline__ double wave_total(const double* __restrict__ p, int n) {
  double v = 0.0;
  for (int i = threadIdx.x & 63; i < n; i += 64) v += p[i];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
  return __shfl(v, 0);
}

// b [nn][3] -> planes [3][nn] in bs and W_0, partial sums of b^2
__global__ __launch_bounds__(RED_THREADS) void k_gs_begin(int64_t nn, const double* __restrict__ b,
                                                          double* __restrict__ bs, double* __restrict__ W0,
                                                          double* __restrict__ x, double* __restrict__ part) {
  double v = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x; i < 3 * nn; i += (int64_t)gridDim.x * RED_THREADS) {
    const int64_t c = i / nn;
    const double t = b[3 * (i - c * nn) + c];
    bs[i] = t;
    W0[i] = t;
    x[i] = 0.0;
    v += t * t;
  }
  block_sums<1>(&v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// W_0 = b - y (W0 null: not stored), partial sums of its square
__global__ __launch_bounds__(RED_THREADS) void k_gs_resid(int64_t n, const double* __restrict__ bs,
                                                          const double* __restrict__ y, double* __restrict__ W0,
                                                          double* __restrict__ part) {
  double v = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_THREADS) {
    const double t = bs[i] - y[i];
    if (W0) W0[i] = t;
    v += t * t;
  }
  block_sums<1>(&v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// The norm of a cycle's first residual.  what 0: of b (the first cycle), 1:
// of a later cycle's, 2: of the final solution (into last).  done only where
// the tolerance is met (b = 0 meets it): a not-a-number never does, so the
// steps go on and carry it into x.
__global__ __launch_bounds__(64) void k_gs_norm(const double* __restrict__ part, int nb, int what, double tol,
                                                GmresState* st, double* __restrict__ scale, double* __restrict__ gv) {
  const double t = sqrt(wave_total(part, nb));
  if (threadIdx.x != 0) return;
  if (what == 2) {
    st->last = t;
    return;
  }
  if (what == 0) st->bnorm = t, st->it = 0;
  st->res = t;
  st->k = 0;
  st->done = t <= tol * st->bnorm;
  scale[0] = t > 0.0 ? 1.0 / t : 0.0;
  gv[0] = t;
}

// partial sums of W_j . y and W_j . W_k for the GS_W vectors of blockIdx.y
__global__ __launch_bounds__(RED_THREADS) void k_gs_dots(int64_t n, int k, const double* __restrict__ W,
                                                         const double* __restrict__ y, double* __restrict__ part,
                                                         const GmresState* __restrict__ st) {
#pragma clang fp contract(fast)
  if (st->done) return;
  const int j0 = blockIdx.y * GS_W, nj = min(GS_W, k + 1 - j0);
  const double* Wk = W + (int64_t)k * n;
  const double* Wj = W + (int64_t)j0 * n;
  double v[2 * GS_W];
#pragma unroll
  for (int i = 0; i < 2 * GS_W; i++) v[i] = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_THREADS) {
    const double a = y[i], b = Wk[i];
    double t[GS_W];
#pragma unroll
    for (int j = 0; j < GS_W; j++) t[j] = j < nj ? Wj[j * n + i] : 0.0;
#pragma unroll
    for (int j = 0; j < GS_W; j++) {
      v[2 * j] += t[j] * a;
      v[2 * j + 1] += t[j] * b;
    }
  }
  block_sums<2 * GS_W>(v);
  if (threadIdx.x == 0)
    for (int j = 0; j < 2 * nj; j++) part[(int64_t)(2 * j0 + j) * gridDim.x + blockIdx.x] = v[j];
}

// The Gram-Schmidt coefficients of step k: h into H's column k, h_j scale_j
// and scale_k into coef.  L: [ld][ld], row j holds V_j . V_i, i < j.
__global__ __launch_bounds__(1024) void k_gs_coef(int k, int ld, const double* __restrict__ part, int nb,
                                                 const double* __restrict__ scale, double* __restrict__ L,
                                                 double* __restrict__ H, double* __restrict__ coef,
                                                 const GmresState* __restrict__ st) {
  if (st->done) return;
  extern __shared__ double r[];  // [k + 1]
  const double sk = scale[k];
  for (int c = threadIdx.x >> 6; c < 2 * (k + 1); c += 16) {
    const double t = wave_total(part + (int64_t)c * nb, nb) * scale[c >> 1] * sk;
    if ((threadIdx.x & 63) == 0) {
      if (c & 1) {
        if ((c >> 1) < k) L[(int64_t)k * ld + (c >> 1)] = t;
      } else {
        r[c >> 1] = t;
      }
    }
  }
  __syncthreads();
  for (int i = 0; i < k; i++) {
    const double hi = r[i];
    for (int j = i + 1 + threadIdx.x; j <= k; j += 1024) r[j] -= L[(int64_t)j * ld + i] * hi;
    __syncthreads();
  }
  for (int j = threadIdx.x; j <= k; j += 1024) {
    H[(int64_t)k * ld + j] = r[j];
    coef[j] = r[j] * scale[j];
  }
  if (threadIdx.x == 0) coef[k + 1] = sk;
}

// W_{k+1} = scale_k y - sum_j coef_j W_j, partial sums of its square
__global__ __launch_bounds__(RED_THREADS) void k_gs_update(int64_t n, int k, const double* __restrict__ y, double* W,
                                                           const double* __restrict__ coef, double* __restrict__ part,
                                                           const GmresState* __restrict__ st) {
#pragma clang fp contract(fast)
  if (st->done) return;
  extern __shared__ double c[];  // [k + 2]
  for (int j = threadIdx.x; j < k + 2; j += RED_THREADS) c[j] = coef[j];
  __syncthreads();
  double* out = W + (int64_t)(k + 1) * n;
  double v = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)RED_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_THREADS) {
    double t = c[k + 1] * y[i];
    int j = 0;
    for (; j + 4 <= k + 1; j += 4) {
      const double a0 = W[(int64_t)j * n + i], a1 = W[(int64_t)(j + 1) * n + i], a2 = W[(int64_t)(j + 2) * n + i],
                   a3 = W[(int64_t)(j + 3) * n + i];
      t -= c[j] * a0;
      t -= c[j + 1] * a1;
      t -= c[j + 2] * a2;
      t -= c[j + 3] * a3;
    }
    for (; j <= k; j++) t -= c[j] * W[(int64_t)j * n + i];
    out[i] = t;
    v += t * t;
  }
  block_sums<1>(&v);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

// The new vector's norm, the Givens rotations of H's column k and the
// residual they leave; ends the cycle at the tolerance.
__global__ __launch_bounds__(256) void k_gs_givens(int k, int ld, const double* __restrict__ part, int nb, double tol,
                                                   double* __restrict__ H, double* __restrict__ rot,
                                                   double* __restrict__ gv, double* __restrict__ scale,
                                                   GmresState* st) {
  if (st->done) return;
  extern __shared__ double sh[];  // column [k + 2], then cosines and sines [2 k]
  double* col = sh;
  double* cs = sh + k + 2;
  for (int j = threadIdx.x; j <= k; j += 256) col[j] = H[(int64_t)k * ld + j];
  for (int j = threadIdx.x; j < 2 * k; j += 256) cs[j] = rot[j];
  const double hn = sqrt(wave_total(part, nb));
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int j = 0; j < k; j++) {
      const double c = cs[2 * j], s = cs[2 * j + 1];
      const double t = c * col[j] + s * col[j + 1];
      col[j + 1] = -s * col[j] + c * col[j + 1];
      col[j] = t;
    }
    const double hk = col[k], rr = hypot(hk, hn);
    const double c = rr > 0 ? hk / rr : 1.0, s = rr > 0 ? hn / rr : 0.0;
    rot[2 * k] = c;
    rot[2 * k + 1] = s;
    col[k] = rr;
    const double g = gv[k];
    gv[k + 1] = -s * g;
    gv[k] = c * g;
    scale[k + 1] = hn > 0.0 ? 1.0 / hn : 0.0;
    st->res = fabs(s * g);
    st->k = k + 1;
    st->it++;
    if (st->res <= tol * st->bnorm || hn == 0.0) st->done = 1;
  }
  __syncthreads();
  for (int j = threadIdx.x; j <= k; j += 256) H[(int64_t)k * ld + j] = col[j];
}

// x += sum_j c[j] W_j; aos: also as [nn][3]
__global__ __launch_bounds__(256) void k_update_x(int64_t nn, int k, const double* __restrict__ c,
                                                  const double* __restrict__ W, double* __restrict__ x,
                                                  double* __restrict__ aos) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, n = 3 * nn;
  if (i >= n) return;
  double v = x[i];
  for (int j = 0; j < k; j++) v += c[j] * W[(int64_t)j * n + i];
  x[i] = v;
  const int64_t d = i / nn;
  aos[3 * (i - d * nn) + d] = v;
}

// The boundary flag and the 8 surrounding cells of every node (single-level
// mesh: the nodes are the points of an N^3 lattice in x, y, z order).  A
// boundary row reads no cell; a missing one is named as cell 0 there.
__global__ __launch_bounds__(256) void k_ecsim_tables(int64_t nn, int N, MeshView m, uint8_t* __restrict__ bnd,
                                                      int* __restrict__ cells8) {
  const int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (n >= nn) return;
  const int g[3] = {(int)(n % N), (int)((n / N) % N), (int)(n / ((int64_t)N * N))};
  bool b = false;
  for (int d = 0; d < 3; d++) b = b || g[d] == 0 || g[d] == N - 1;
  bnd[n] = b ? 1 : 0;
  for (int q = 0; q < 8; q++) {
    const int c[3] = {g[0] - 1 + (q & 1), g[1] - 1 + ((q >> 1) & 1), g[2] - 1 + (q >> 2)};
    int cell = 0;
    if (c[0] >= 0 && c[1] >= 0 && c[2] >= 0 && c[0] < N - 1 && c[1] < N - 1 && c[2] < N - 1) {
      const int blk = m.leaf_of[((c[2] / NC) * m.nf + c[1] / NC) * m.nf + c[0] / NC];
      cell = blk * NCELL + c[0] % NC + NC * (c[1] % NC + NC * (c[2] % NC));
    }
    cells8[n * 8 + q] = cell;
  }
}

dim3 grid_of(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

// ---------------------------------------------------------------------------
// host: tables, checks, work space
// ---------------------------------------------------------------------------
int check_ready(amps_ctx* c, const amps_ecsim_params* p, const char* who) {
  if (!c || !p) return fail(AMPS_E_ARG, std::string(who) + ": null argument");
  if (!c->has_mesh || !c->d_nodeout)
    return fail(AMPS_E_STATE, std::string(who) + ": run amps_gpu_update_j_mass_matrix first (J and M)");
  if (!single_level(c))
    return fail(AMPS_E_STATE, std::string(who) + ": the ECSIM field equation needs a single-level mesh "
                                                 "(the reference solver runs on one resolution level)");
  if (!(p->theta > 0.0) || !(p->E_conv != 0.0) || !(p->B_conv != 0.0) || !(p->length_conv > 0.0))
    return fail(AMPS_E_ARG, std::string(who) + ": theta, E_conv, B_conv and length_conv must be nonzero");
  if (c->nnodes > ((int64_t)1 << 27)) return fail(AMPS_E_RANGE, std::string(who) + ": more than 2^27 nodes");
  return 0;
}

int build_tables(amps_ctx* c) {
  if (int r = build_nbr(c)) return r;
  if (c->d_ecsim_bnd) return 0;
  const int64_t nn = c->nnodes;
  const int N = (NC << c->h_level[0]) + 1;
  if ((int64_t)N * N * N != nn) return fail(AMPS_E_STATE, "ecsim: the nodes are not a cubic lattice");
  HIP_TRY(hipMalloc(&c->d_ecsim_noc, sizeof(int) * std::max<size_t>(1, c->h_node_of_corner.size())));
  HIP_TRY(hipMalloc(&c->d_ecsim_cells8, sizeof(int) * std::max<size_t>(8, (size_t)nn * 8)));
  HIP_TRY(hipMalloc(&c->d_ecsim_bnd, std::max<size_t>(1, (size_t)nn)));
  HIP_TRY(hipMemcpyAsync(c->d_ecsim_noc, c->h_node_of_corner.data(), sizeof(int) * c->h_node_of_corner.size(),
                         hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_ecsim_tables, grid_of(nn), dim3(256), 0, c->stream, nn, N, c->mv, c->d_ecsim_bnd,
                     c->d_ecsim_cells8);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

int ensure_work(amps_ctx* c, size_t len) {
  if (c->ecsim_work_len >= len) return 0;
  (void)hipFree(c->d_ecsim_work);
  c->d_ecsim_work = nullptr;
  c->ecsim_work_len = 0;
  HIP_TRY(hipMalloc(&c->d_ecsim_work, sizeof(double) * len));
  c->ecsim_work_len = len;
  return 0;
}

void cell_size(const amps_ctx* c, double dx[3]) {
  for (int d = 0; d < 3; d++) dx[d] = (c->h_xmax[(size_t)d] - c->h_xmin[(size_t)d]) / NC;
}

// a device copy of the row tables (the tail of the work space)
int upload_coefs(amps_ctx* c, const amps_ecsim_params* p, Coefs* dC) {
  double dx[3];
  cell_size(c, dx);
  const Coefs C = coefficients(dx, *p);
  HIP_TRY(hipMemcpyAsync(dC, &C, sizeof(Coefs), hipMemcpyHostToDevice, c->stream));
  return 0;
}

// layout of the work space (doubles): En, Bc or rhs, x, y/w, dE, Eth, E1, Bout,
// the coefficient tables; for a solve (restart > 0) also b, x and y as planes,
// reduction partials, the small dense arrays, then the Krylov basis
struct Work {
  double *En, *Bc, *rhs, *x, *w, *Eth, *E1, *Bout;
  Coefs* C;
  double *bs, *xs, *ys, *part, *scale, *gv, *rot, *coef, *yv, *L, *H, *V;
  GmresState* st;
};
size_t part_len(int restart) { return (size_t)RED_BLOCKS * 2 * ((size_t)restart + 1); }
size_t work_len(int64_t nn, int64_t ncell, int restart) {
  const size_t n3 = 3 * (size_t)nn, c3 = 3 * (size_t)ncell, ld = (size_t)restart + 2;
  const size_t coef = (sizeof(Coefs) + 7) / 8;
  size_t len = n3 * 6 + c3 * 2 + coef;
  if (restart > 0)
    len += n3 * 3 + part_len(restart) + 6 * ld + 2 * ld * ld + (sizeof(GmresState) + 7) / 8 + n3 * ((size_t)restart + 1);
  return len;
}
Work carve(amps_ctx* c, int restart) {
  const size_t n3 = 3 * (size_t)c->nnodes, c3 = 3 * (size_t)c->mv.nb * NCELL, ld = (size_t)restart + 2;
  double* p = c->d_ecsim_work;
  Work w{};
  w.En = p, p += n3;
  w.rhs = p, p += n3;
  w.x = p, p += n3;
  w.w = p, p += n3;
  w.Eth = p, p += n3;
  w.E1 = p, p += n3;
  w.Bc = p, p += c3;
  w.Bout = p, p += c3;
  w.C = reinterpret_cast<Coefs*>(p), p += (sizeof(Coefs) + 7) / 8;
  if (restart > 0) {
    w.bs = p, p += n3;
    w.xs = p, p += n3;
    w.ys = p, p += n3;
    w.part = p, p += part_len(restart);
    w.scale = p, p += ld;
    w.gv = p, p += ld;
    w.rot = p, p += 2 * ld;
    w.coef = p, p += ld;
    w.yv = p, p += ld;
    w.L = p, p += ld * ld;
    w.H = p, p += ld * ld;
    w.st = reinterpret_cast<GmresState*>(p), p += (sizeof(GmresState) + 7) / 8;
    w.V = p;
  }
  return w;
}

void launch_op(amps_ctx* c, const Work& W, double fpdt, const double* x, double* y) {
  const int64_t nn = c->nnodes;
  // 8 nodes per workgroup, the workgroup count rounded up to 8 (XCD chunks)
  const dim3 grid((unsigned)((((nn + 7) / 8) + 7) / 8 * 8));
  hipLaunchKernelGGL(k_ecsim_op, grid, dim3(256), 0, c->stream, nn, c->d_nodeout, c->d_ecsim_nbr, c->d_ecsim_bnd,
                     W.C, fpdt, x, y);
}

// The packed operator of this solve, y = A x on planes.
struct SymOp {
  const double* A;
  int64_t np;
  int N;
  bool mask;
};
void launch_sym(amps_ctx* c, const SymOp& o, const double* x, double* y, const GmresState* st) {
  const int64_t nn = c->nnodes;
  const unsigned g = (unsigned)(((nn + 255) / 256 + 7) / 8 * 8);
  // below 2^18 nodes a thread per node leaves most of the 256 CUs idle
  if (nn >= ((int64_t)1 << 18)) {
    if (o.mask) hipLaunchKernelGGL((k_sym_op<3, true>), dim3(g), dim3(256), 0, c->stream, nn, o.np, o.N, o.A, x, y, st);
    else hipLaunchKernelGGL((k_sym_op<3, false>), dim3(g), dim3(256), 0, c->stream, nn, o.np, o.N, o.A, x, y, st);
  } else {
    if (o.mask) hipLaunchKernelGGL((k_sym_op<1, true>), dim3(g, 3), dim3(256), 0, c->stream, nn, o.np, o.N, o.A, x, y, st);
    else hipLaunchKernelGGL((k_sym_op<1, false>), dim3(g, 3), dim3(256), 0, c->stream, nn, o.np, o.N, o.A, x, y, st);
  }
}

int pack_operator(amps_ctx* c, const Work& W, double fpdt, bool mask, SymOp* o) {
  const int64_t nn = c->nnodes, np = (nn + 31) / 32 * 32;
  o->np = np;
  o->N = (NC << c->h_level[0]) + 1;
  o->mask = mask;
  if ((int64_t)o->N * o->N * o->N != nn) return fail(AMPS_E_STATE, "ecsim: the nodes are not a cubic lattice");
  if (!c->d_ecsim_sym) HIP_TRY(hipMalloc(&c->d_ecsim_sym, sizeof(double) * SYM * 9 * np));
  o->A = c->d_ecsim_sym;
  hipLaunchKernelGGL(k_sym_pack, dim3((unsigned)(np / 32)), dim3(256), 0, c->stream, nn, np, c->d_nodeout, W.C, fpdt,
                     c->d_ecsim_sym);
  HIP_TRY(hipGetLastError());
  return 0;
}

// Restarted GMRES on the device: W.rhs -> W.x.  The Arnoldi steps are
// enqueued GS_BATCH at a time, each kernel returning at once when the cycle
// has ended; the host looks at the state after a batch.  mask: the rows of
// boundary nodes may have a nonzero right-hand side.
constexpr int GS_BATCH = 8;
int gmres(amps_ctx* c, const Work& W, double fpdt, double tol, int max_iter, int restart, bool mask, int* iters,
          double* relres) {
  const int64_t nn = c->nnodes, n = 3 * nn;
  const int ld = restart + 2;
  // enough workgroups for the chip, few enough partials to sum
  const int nb = (int)std::min<int64_t>(RED_BLOCKS, (n + 2 * RED_THREADS - 1) / (2 * RED_THREADS));
  const dim3 red(RED_THREADS);
  *iters = 0;
  *relres = 0.0;
  SymOp op;
  if (int r = pack_operator(c, W, fpdt, mask, &op)) return r;
  GmresState h;
  auto look = [&]() -> int {
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(&h, W.st, sizeof(h), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return 0;
  };
  std::vector<double> H, gv((size_t)ld), sc((size_t)ld), y;
  int it = 0;
  bool first = true;
  for (;;) {
    if (first) {  // x = 0: the residual is b
      hipLaunchKernelGGL(k_gs_begin, dim3(nb), red, 0, c->stream, nn, W.rhs, W.bs, W.V, W.xs, W.part);
    } else {
      launch_sym(c, op, W.xs, W.ys, nullptr);
      hipLaunchKernelGGL(k_gs_resid, dim3(nb), red, 0, c->stream, n, W.bs, W.ys, W.V, W.part);
    }
    hipLaunchKernelGGL(k_gs_norm, dim3(1), dim3(64), 0, c->stream, W.part, nb, first ? 0 : 1, tol, W.st, W.scale,
                       W.gv);
    first = false;
    const int steps = std::min(restart, max_iter - it);
    for (int k = 0; k < steps;) {
      for (int e = std::min(steps, k + GS_BATCH); k < e; k++) {
        launch_sym(c, op, W.V + (int64_t)k * n, W.ys, W.st);
        hipLaunchKernelGGL(k_gs_dots, dim3(nb, (k + GS_W) / GS_W), red, 0, c->stream, n, k, W.V, W.ys, W.part, W.st);
        hipLaunchKernelGGL(k_gs_coef, dim3(1), dim3(1024), sizeof(double) * (k + 1), c->stream, k, ld, W.part, nb,
                           W.scale, W.L, W.H, W.coef, W.st);
        hipLaunchKernelGGL(k_gs_update, dim3(nb), red, sizeof(double) * (k + 2), c->stream, n, k, W.ys, W.V, W.coef,
                           W.part, W.st);
        hipLaunchKernelGGL(k_gs_givens, dim3(1), dim3(256), sizeof(double) * (3 * k + 2), c->stream, k, ld, W.part, nb,
                           tol, W.H, W.rot, W.gv, W.scale, W.st);
      }
      if (int r = look()) return r;
      if (h.done) break;
    }
    if (steps <= 0)
      if (int r = look()) return r;
    it = h.it;
    const int k = h.k;
    if (h.bnorm == 0.0) {  // b = 0: x = 0
      hipLaunchKernelGGL(k_update_x, grid_of(n), dim3(256), 0, c->stream, nn, 0, W.yv, W.V, W.xs, W.x);
      HIP_TRY(hipGetLastError());
      return 0;
    }
    // y = H^{-1} g over the k columns, then x += V y
    if (k > 0) {
      H.resize((size_t)k * ld);
      y.assign((size_t)k, 0.0);
      HIP_TRY(hipMemcpyAsync(H.data(), W.H, sizeof(double) * H.size(), hipMemcpyDeviceToHost, c->stream));
      HIP_TRY(hipMemcpyAsync(gv.data(), W.gv, sizeof(double) * (k + 1), hipMemcpyDeviceToHost, c->stream));
      HIP_TRY(hipMemcpyAsync(sc.data(), W.scale, sizeof(double) * (k + 1), hipMemcpyDeviceToHost, c->stream));
      HIP_TRY(hipStreamSynchronize(c->stream));
      for (int j = k - 1; j >= 0; j--) {
        double s = gv[(size_t)j];
        for (int l = j + 1; l < k; l++) s -= H[(size_t)l * ld + j] * y[(size_t)l];
        y[(size_t)j] = s / H[(size_t)j * ld + j];
      }
      for (int j = 0; j < k; j++) y[(size_t)j] *= sc[(size_t)j];
      HIP_TRY(hipMemcpyAsync(W.yv, y.data(), sizeof(double) * k, hipMemcpyHostToDevice, c->stream));
    }
    hipLaunchKernelGGL(k_update_x, grid_of(n), dim3(256), 0, c->stream, nn, k, W.yv, W.V, W.xs, W.x);
    if (h.res <= tol * h.bnorm || k == 0 || it >= max_iter) break;
  }
  // the true residual of the returned solution
  launch_sym(c, op, W.xs, W.ys, nullptr);
  hipLaunchKernelGGL(k_gs_resid, dim3(nb), red, 0, c->stream, n, W.bs, W.ys, (double*)nullptr, W.part);
  hipLaunchKernelGGL(k_gs_norm, dim3(1), dim3(64), 0, c->stream, W.part, nb, 2, tol, W.st, W.scale, W.gv);
  if (int r = look()) return r;
  *iters = it;
  *relres = h.last / h.bnorm;
  return 0;
}

int prepare(amps_ctx* c, const amps_ecsim_params* p, int restart, Work* W, const char* who) {
  if (int r = check_ready(c, p, who)) return r;
  (void)hipSetDevice(c->device);
  if (int r = build_tables(c)) return r;
  if (int r = ensure_work(c, work_len(c->nnodes, (int64_t)c->mv.nb * NCELL, restart))) return r;
  *W = carve(c, restart);
  return upload_coefs(c, p, W->C);
}

double fpdt_of(const amps_ecsim_params* p) { return 4 * PI_REF * p->dt * p->theta; }

}  // namespace

namespace amps {
void ecsim_field_free(amps_ctx* c) {
  (void)hipFree(c->d_ecsim_bnd);
  (void)hipFree(c->d_ecsim_cells8);
  (void)hipFree(c->d_ecsim_noc);
  (void)hipFree(c->d_ecsim_work);
  (void)hipFree(c->d_ecsim_sym);
  c->d_ecsim_sym = nullptr;
  c->d_ecsim_bnd = nullptr;
  c->d_ecsim_cells8 = nullptr;
  c->d_ecsim_noc = nullptr;
  c->d_ecsim_work = nullptr;
  c->ecsim_work_len = 0;
}
}  // namespace amps

extern "C" int amps_gpu_ecsim_operator(amps_ctx* c, const amps_ecsim_params* p, const double* x, double* y,
                                       int32_t reps) {
  if (!x || !y) return fail(AMPS_E_ARG, "amps_gpu_ecsim_operator: null array");
  if (reps < 1 || reps > 1000) return fail(AMPS_E_RANGE, "amps_gpu_ecsim_operator: reps must be in 1..1000");
  Work W;
  if (int r = prepare(c, p, 0, &W, "amps_gpu_ecsim_operator")) return r;
  const size_t n3 = 3 * (size_t)c->nnodes;
  if (int r = copy_to_device(c, W.x, x, sizeof(double) * n3)) return r;
  for (int i = 0; i < reps; i++) {
    tbegin(c);
    launch_op(c, W, fpdt_of(p), W.x, W.w);
    tend(c, AMPS_K_ECSIM);
  }
  HIP_TRY(hipGetLastError());
  if (int r = copy_to_host(c, y, W.w, sizeof(double) * n3)) return r;
  return AMPS_OK;
}

extern "C" int amps_gpu_ecsim_rhs(amps_ctx* c, const amps_ecsim_params* p, const double* E_n, const double* B_c,
                                  double* rhs) {
  if (!E_n || !B_c || !rhs) return fail(AMPS_E_ARG, "amps_gpu_ecsim_rhs: null array");
  Work W;
  if (int r = prepare(c, p, 0, &W, "amps_gpu_ecsim_rhs")) return r;
  const int64_t nn = c->nnodes;
  const size_t n3 = 3 * (size_t)nn, c3 = 3 * (size_t)c->mv.nb * NCELL;
  if (int r = copy_to_device(c, W.En, E_n, sizeof(double) * n3)) return r;
  if (int r = copy_to_device(c, W.Bc, B_c, sizeof(double) * c3)) return r;
  hipLaunchKernelGGL(k_ecsim_rhs, dim3((unsigned)((((nn + 7) / 8) + 7) / 8 * 8)), dim3(256), 0, c->stream, nn, c->d_nodeout, c->d_ecsim_nbr,
                     c->d_ecsim_bnd, c->d_ecsim_cells8, W.C, p->dt, p->theta, p->E_conv, p->B_conv, W.En, W.Bc,
                     W.rhs);
  HIP_TRY(hipGetLastError());
  if (int r = copy_to_host(c, rhs, W.rhs, sizeof(double) * n3)) return r;
  return AMPS_OK;
}

extern "C" int amps_gpu_ecsim_solve(amps_ctx* c, const amps_ecsim_params* p, const double* rhs, double tol,
                                    int32_t max_iter, int32_t restart, double* dE, int32_t* iters,
                                    double* rel_residual) {
  if (!rhs || !dE || !iters || !rel_residual) return fail(AMPS_E_ARG, "amps_gpu_ecsim_solve: null argument");
  if (!(tol > 0.0) || max_iter < 1 || restart < 1 || restart > 400)
    return fail(AMPS_E_ARG, "amps_gpu_ecsim_solve: tol > 0, max_iter >= 1 and restart in 1..400 are required");
  Work W;
  if (int r = prepare(c, p, restart, &W, "amps_gpu_ecsim_solve")) return r;
  const size_t n3 = 3 * (size_t)c->nnodes;
  if (int r = copy_to_device(c, W.rhs, rhs, sizeof(double) * n3)) return r;
  int it = 0;
  double rr = 0.0;
  if (int r = gmres(c, W, fpdt_of(p), tol, max_iter, restart, true, &it, &rr)) return r;
  if (int r = copy_to_host(c, dE, W.x, sizeof(double) * n3)) return r;
  *iters = it;
  *rel_residual = rr;
  return AMPS_OK;
}

extern "C" int amps_gpu_ecsim_update_b(amps_ctx* c, const amps_ecsim_params* p, const double* E_theta,
                                       const double* B_c, double* B_out) {
  if (!E_theta || !B_c || !B_out) return fail(AMPS_E_ARG, "amps_gpu_ecsim_update_b: null array");
  Work W;
  if (int r = prepare(c, p, 0, &W, "amps_gpu_ecsim_update_b")) return r;
  const size_t n3 = 3 * (size_t)c->nnodes;
  const int64_t ncell = (int64_t)c->mv.nb * NCELL;
  if (int r = copy_to_device(c, W.Eth, E_theta, sizeof(double) * n3)) return r;
  if (int r = copy_to_device(c, W.Bc, B_c, sizeof(double) * 3 * ncell)) return r;
  double dx[3];
  cell_size(c, dx);
  double c4[3];
  for (int d = 0; d < 3; d++) c4[d] = 0.25 * (p->cDt / (dx[d] * p->length_conv));
  hipLaunchKernelGGL(k_ecsim_update_b, grid_of(ncell), dim3(256), 0, c->stream, ncell, c->d_ecsim_noc, W.Eth,
                     W.Bc, c4[0], c4[1], c4[2], p->E_conv, p->B_conv, W.Bout);
  HIP_TRY(hipGetLastError());
  if (int r = copy_to_host(c, B_out, W.Bout, sizeof(double) * 3 * ncell)) return r;
  return AMPS_OK;
}

extern "C" int amps_gpu_ecsim_time_step(amps_ctx* c, const amps_ecsim_params* p, double* E, double* E_theta,
                                        double* B_c, double tol, int32_t max_iter, int32_t restart, int32_t* iters,
                                        double* rel_residual) {
  if (!E || !B_c || !iters || !rel_residual) return fail(AMPS_E_ARG, "amps_gpu_ecsim_time_step: null argument");
  if (!(tol > 0.0) || max_iter < 1 || restart < 1 || restart > 400)
    return fail(AMPS_E_ARG, "amps_gpu_ecsim_time_step: tol > 0, max_iter >= 1 and restart in 1..400 are required");
  Work W;
  if (int r = prepare(c, p, restart, &W, "amps_gpu_ecsim_time_step")) return r;
  const int64_t nn = c->nnodes;
  const size_t n3 = 3 * (size_t)nn;
  const int64_t ncell = (int64_t)c->mv.nb * NCELL;
  if (int r = copy_to_device(c, W.En, E, sizeof(double) * n3)) return r;
  if (int r = copy_to_device(c, W.Bc, B_c, sizeof(double) * 3 * ncell)) return r;
  // right-hand side, GMRES, E^{n+theta} and E^{n+1}, B^{n+1}
  hipLaunchKernelGGL(k_ecsim_rhs, dim3((unsigned)((((nn + 7) / 8) + 7) / 8 * 8)), dim3(256), 0, c->stream, nn, c->d_nodeout, c->d_ecsim_nbr,
                     c->d_ecsim_bnd, c->d_ecsim_cells8, W.C, p->dt, p->theta, p->E_conv, p->B_conv, W.En, W.Bc,
                     W.rhs);
  int it = 0;
  double rr = 0.0;
  if (int r = gmres(c, W, fpdt_of(p), tol, max_iter, restart, false, &it, &rr)) return r;
  hipLaunchKernelGGL(k_ecsim_update_e, grid_of((int64_t)n3), dim3(256), 0, c->stream, (int64_t)n3, W.En, W.x,
                     p->theta, p->E_conv, W.Eth, W.E1);
  double dx[3];
  cell_size(c, dx);
  double c4[3];
  for (int d = 0; d < 3; d++) c4[d] = 0.25 * (p->cDt / (dx[d] * p->length_conv));
  hipLaunchKernelGGL(k_ecsim_update_b, grid_of(ncell), dim3(256), 0, c->stream, ncell, c->d_ecsim_noc, W.Eth,
                     W.Bc, c4[0], c4[1], c4[2], p->E_conv, p->B_conv, W.Bout);
  HIP_TRY(hipGetLastError());
  if (int r = copy_to_host(c, E, W.E1, sizeof(double) * n3)) return r;
  if (E_theta)
    if (int r = copy_to_host(c, E_theta, W.Eth, sizeof(double) * n3)) return r;
  if (int r = copy_to_host(c, B_c, W.Bout, sizeof(double) * 3 * ncell)) return r;
  *iters = it;
  *rel_residual = rr;
  return AMPS_OK;
}
