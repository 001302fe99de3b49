// deposit_mfma.hip — ECSIM deposit cell pass on the FP64 matrix cores.
//
// The mass-matrix part of ProcessCell (pic_field_solver_ecsim.cpp:2241-2342)
// is, per cell, a sum over the cell's particles of rank-one updates.  In the
// moment form each particle contributes
//     M[t][k] += (mx[tx] my[ty]) * (mz[tz] MC alpha[k])
// with mx = ((1-fx)^2, fx(1-fx), fx^2) (and my, mz alike), t = tx + 3ty + 9tz
// and MC = q (q dt / 2m) / V: a 9 x 27 product over the particles.  The
// current is
//     J[c][d] += (wx[bx] q alphaV[d]) * (wy[by] wz[bz])
// a 6 x 4 product.  Both fit one 16 x 32 tile of A (16 x np) times B (np x 32):
//     A rows 0-8:  mx[tx] my[ty]               B cols 0-26:  mz[tz] MC alpha[k]
//     A rows 9-14: wx[bx] q alphaV[d]          B cols 27-30: wy[by] wz[bz]
// so a cell is two v_mfma_f64_16x16x4f64 per 4 particles, accumulated in
// registers, with the parts of the 16 x 32 result outside these blocks unused.
//
// One workgroup per 4x4x4 sub-tile of a block; wavefront w takes the 16
// cells of z-layer w (8 or 4 cells a wavefront, and fewer layers a workgroup, on
// meshes of few blocks).  Its cells' particles are consecutive runs of the
// key-sorted arrays; the wavefront walks their concatenation, each cell's run
// rounded up to whole steps of 4 (but for SPARSE populations), 64 places at a
// time: each lane turns one particle into its operand record (corner stencil,
// B from the sub-tile's corners staged in LDS, alpha, alpha v) in LDS, then the
// wavefront issues the MFMA steps cell by cell and writes a finished cell's
// 267 values (J[8][3] / V, then M[27][9]) to its partial-sum record.  The
// particles of the next two chunks, and the source indices of the one after,
// are loaded while the current one is accumulated.
//
// What bounds it: what a wavefront issues, record by record and product by
// product, with two of them to a SIMD (80 KB of LDS a workgroup) that overlap
// in part: with counters (15.3 M particles, before) MFMA 38 % and other
// vector instructions 31 % of the cycles, LDS 47 % busy, no unit saturated.
// Fewer instructions a wavefront pay: the inner loop is
// kept to the products and five address increments per four steps, with two
// steps to an LDS read; 2^27 particles on 7,456 blocks 6.37 -> 5.88 ms, 15.3 M
// in FP32 0.69 -> 0.62.  More wavefronts have not: three per SIMD (records written in
// halves of 32 particles, 47 KB) took 8.6 ms, since the halves double the record stores.
//
// PAIRED: eight wavefronts, two per SIMD (w and w + 4, in layers two apart), run
// in opposite phases locked by workgroup barriers: while one builds the
// records of its next chunk (VALU), the other issues the matrix products of
// its current one (MFMA), so the two units overlap instead of taking turns.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "amps_common.h"
#include "center_device.h"
#include "pic_device.h"

using namespace amps;

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// Records are kept field-major, rec[f * FS + particle]: the record stores
// (lane = particle) are contiguous, and with FS = 66 the MFMA operand reads
// (16 fields x 2 particles per 32-lane pass) fall on distinct banks.
constexpr int NFLD = 32;
constexpr int FS = 66;
constexpr int F_A = 0;      // A operand rows 0-14
constexpr int F_ONE = 15;   // 1: A row 15 and the factor of the wy wz columns
constexpr int F_MA = 16;    // MC alpha[k], k = 0..8
constexpr int F_MZ = 25;    // mz[tz], tz = 0..2
constexpr int F_WYZ = 28;   // wy[by] wz[bz] at by + 2bz
constexpr int CS = CELL_STRIDE_MOMENT;  // cell record stride: 267 values + padding

// LDS ordering between the lanes of one wavefront: the DS instructions of a
// wavefront execute in issue order, so a compiler barrier that keeps LDS
// accesses on their side is all that is needed.
__device__ __forceinline__ void wave_lds_sync() { asm volatile("" ::: "memory"); }

// a value every lane of the wavefront holds, kept in a scalar register
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// InterpolationCoefficientTable corner index of offset bits (bx, by, bz)
__device__ __forceinline__ int corner_of(int bx, int by, int bz) { return 4 * bz + (by ? (bx ? 2 : 3) : bx); }

template <bool PAIRED>
constexpr int waves_of() { return PAIRED ? 8 : 4; }

// How the cells are split: 2^lw cells per wavefront; with `extra` workgroups
// (four per list entry) in front of the others, the crowded sub-tiles take
// one workgroup per layer and 4 cells per wavefront.
struct Split {
  int lw, extra;
  const int* count;  // crowded sub-tiles of the layout
  const int* list;
  const uint8_t* crowded;  // per sub-tile
};

// VF32: FP32 velocities (widened when the record is built, not at the load:
// a conversion there would wait for the prefetched data)
// SPARSE: cells of few particles (mean below SPARSE_MEAN).  There the rounding
// to whole steps of 4 costs places, and with them chunks, and the loop's
// start, which loads four steps, costs more than its pace gains: the cells' runs
// stay as they are, one or two steps are issued without the loop and the
// last 1-3 particles as a step of their own, and no chunk past the last is
// looked for.  The pass at 1, 2, 4 and 8
// particles per cell, us: 7,456 blocks 2,338, 2,470, 2,706 and 3,082 against
// 2,459, 2,590, 2,787 and 3,116 in whole steps; 64 blocks, 1, 4 and 8: 22.5,
// 26.0 and 31.5 against 26.5, 28.7 and 32.7.  At 35 a cell whole steps are ahead (7,456
// blocks 5.94 ms against 6.03 with the short runs out of the loop, 6.4 with ragged
// ones).
constexpr int SPARSE_MEAN = 10;

template <bool BC, bool PAIRED, bool FUSED, bool VF32, bool SPARSE>
__global__ __launch_bounds__(64 * waves_of<PAIRED>()) void k_deposit_cell_mfma(MeshView m, Species sp, double dtTotal,
                                                                 const double* __restrict__ B,
                                                                 const int* __restrict__ offset,
                                                                 int64_t cap,
                                                                 const double* __restrict__ x,
                                                                 const double* __restrict__ v,
                                                                 int /*vf32*/,
                                                                 const uint8_t* __restrict__ spec,
                                                                 double* __restrict__ cellpart,
                                                                 const double* __restrict__ Bc,
                                                                 const int* __restrict__ src, Split sp4) {
  constexpr int MW = waves_of<PAIRED>();
  constexpr int MCW = PAIRED ? 8 : 16;  // most cells per wavefront
  __shared__ double sB[125 * 3];
  // 16 doubles of padding: the operand loads run up to four steps (16
  // particles) past a segment's last particle, and are not used there
  __shared__ double rec[MW][NFLD * FS + 16];
  __shared__ double sconst[MAX_SPEC + 1][3];  // chargeQ, QdT_over_2m, matrixConst; the last: an empty place
  __shared__ int sfirst[MW][MCW], scum[MW][MCW + 1];
  __shared__ __align__(16) double sstage[MW][CS + 2];  // a finished cell's record, written out in full lines, and a spare place
  __shared__ int smaxchunks;
  // 2^lw cells per wavefront, 2^(4 - lw) wavefronts per layer, 2^lz layers per
  // workgroup (logarithms: a division by a run-time value is some 30 instructions)
  constexpr int LMW = PAIRED ? 3 : 2;
  int lw = PAIRED ? 3 : BC ? 4 : sp4.lw, lz = LMW - 4 + lw;
  int b, st, sz;
  bool skip = false;
  if (!PAIRED && !BC && (int)blockIdx.x < sp4.extra) {
    // a layer of a crowded sub-tile
    if ((int)(blockIdx.x >> 2) >= sp4.count[0]) return;
    const int tile = sp4.list[blockIdx.x >> 2];
    lw = 2, lz = 0;
    b = tile >> 3, st = tile & 7;
    sz = (st >> 2) * 4 + (blockIdx.x & 3);
  } else {
    // the workgroups of a block on one XCD
    const int extra = PAIRED || BC ? 0 : sp4.extra;
    const int bi = blockIdx.x - extra, ng = gridDim.x - extra;
    const int tile = (bi % N_XCD) * (ng / N_XCD) + bi / N_XCD;
    if (extra) skip = sp4.crowded[tile];  // tested below, when the other loads are on their way
    b = tile >> (5 - lz), st = tile & ((32 >> lz) - 1);
    sz = (st >> 2) << lz;
  }
  const int ncw = 1 << lw;
  const int sx = (st & 1) * 4, sy = ((st >> 1) & 1) * 4;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // wavefront w: layer zl, rows row0.. of it (cell c: x = c % 4, y = row0 + c / 4)
  const int zl = uniform(w >> (4 - lw)), zc = sz + zl;
  const int row0 = uniform((w & ((16 >> lw) - 1)) << (lw - 2));
  const int keybase = b * NCELL;
  if constexpr (!BC) {
    const double* Bb = B + (size_t)b * NCORNER * 3;
    for (int i = threadIdx.x; i < 75 * ((1 << lz) + 1); i += blockDim.x) {
      const int cidx = i / 3, d = i % 3;
      const int a0 = cidx % 5, a1 = (cidx / 5) % 5, a2 = cidx / 25;
      sB[i] = Bb[3 * ((sx + a0) + NN * ((sy + a1) + NN * (sz + a2))) + d];
    }
  }
  BlockGeom g;
  load_block_geom(m, b, g);
  double CellVolume = 1;
  for (int d = 0; d < 3; d++) CellVolume *= (g.xmax[d] - g.xmin[d]) / NC * 1.0;
  double inv_dxs[3];
#pragma unroll
  for (int d = 0; d < 3; d++) inv_dxs[d] = 1.0 / g.dxs[d];
  if (threadIdx.x < sp.n) {
    // per-species factors of ProcessCell, same operations in the same order
    const int s = threadIdx.x;
    double chargeQ = sp.charge[s], mass = sp.mass[s];
    chargeQ *= sp.weight[s];
    mass *= sp.weight[s];
    const double QdT_over_m = chargeQ * dtTotal / mass;
    const double QdT_over_2m = 0.5 * QdT_over_m;
    sconst[s][0] = chargeQ;
    sconst[s][1] = QdT_over_2m;
    sconst[s][2] = chargeQ * QdT_over_2m / CellVolume;
  }
  if (threadIdx.x < 3) sconst[MAX_SPEC][threadIdx.x] = 0.0;
  auto cellkey = [&](int c) { return keybase + (sx + (c & 3)) + NC * ((sy + row0 + (c >> 2)) + NC * zc); };
  // this wavefront's cells: first particle, running counts, each rounded up to
  // whole steps of 4 particles (not SPARSE)
  int cntk = 0;
  {
    // counts of lanes' cells, then an inclusive scan across the lanes
    const int ck = cellkey(lane < ncw ? lane : 0);
    const int o0 = offset[ck];
    cntk = lane < ncw ? offset[ck + 1] - o0 : 0;
    const int cnt = SPARSE ? cntk : (cntk + 3) & ~3;
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < MCW; d <<= 1) {
      const int t = __shfl_up(incl, d, 64);
      if (lane >= d) incl += t;
    }
    if (lane < ncw) {
      sfirst[w][lane] = o0;
      scum[w][lane] = incl - cnt;
    }
    if (lane == ncw - 1) scum[w][ncw] = incl;
  }
  if (threadIdx.x == 0) smaxchunks = 0;
  if (skip) return;  // the whole workgroup: its layers are in the list
  __syncthreads();
  const int* cum = scum[w];
  const int total = uniform(cum[ncw]);
  double* R0 = rec[w];

  // operand selectors of this lane: A row ia = j and B columns j, 16 + j of particle slot lane / 16
  const int j = lane & 15, slot = lane >> 4;
  const int f0a = F_MZ + j / 9, f0b = F_MA + j % 9;
  int f1a, f1b;
  {
    // A row 15 and B column 31 hold ones; the results they touch are not kept
    const int col = 16 + j;
    if (col < 27) {
      f1a = F_MZ + col / 9, f1b = F_MA + col % 9;
    } else if (col < 31) {
      f1a = F_WYZ + (col - 27), f1b = F_ONE;
    } else {
      f1a = F_ONE, f1b = F_ONE;
    }
  }
  const int oa = (F_A + j) * FS, o0a = f0a * FS, o0b = f0b * FS, o1a = f1a * FS, o1b = f1b * FS;
  // destinations of the 8 accumulator values; CS: unused.  v_mfma_f64_16x16x4f64
  // holds A[i][k] in lane i + 16k, B[k][j] in lane j + 16k and D[i][j] in
  // lane 16 (i % 4) + j, accumulator register i / 4.
  double* S = sstage[w];
  int oidx[8];
#pragma unroll
  for (int T = 0; T < 2; T++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = slot + 4 * r, col = 16 * T + j;
      int o = CS;  // not kept
      if (i < 9 && col < 27) {
        o = 24 + 9 * (i + 9 * (col / 9)) + col % 9;
      } else if (i >= 9 && i < 15 && col >= 27 && col < 31) {
        const int bx = (i - 9) / 3, d = (i - 9) % 3, by = (col - 27) & 1, bz = (col - 27) >> 1;
        o = 3 * corner_of(bx, by, bz) + d;
      }
      oidx[4 * T + r] = o;
    }
  }
  const double invV = 1.0 / CellVolume;
  if (lane < CS - CELL_VALS_MOMENT) S[CELL_VALS_MOMENT + lane] = 0.0;

  // each lane's particles of the next two chunks, loaded ahead
  struct Pre {
    double x[3], v[3];
    float vf[3];
    int s, c;
  };
  // lane k < ncw: where cell k starts in the concatenation, and the offset
  // from a position in the concatenation to the particle's index
  const int cumk = lane < ncw ? cum[lane] : 0;
  const int dk = lane < ncw ? sfirst[w][lane] - cum[lane] : 0;
  const int endk = cumk + cntk;  // and where its particles end
  // where the particle at position pbase + lane is (called by the whole
  // wavefront): a position's cell is the last one that starts at or before it.
  // FUSED: the particles are still where the last compaction found them,
  // particle p of the new order at src[p]; that load is a chunk ahead of the
  // ones that need it, so that no wavefront waits for it.
  struct Idx {
    int q, c;  // q < 0: an empty place, up to three at the end of a cell
  };
  auto index = [&](int pbase, Idx& ix) {
    const int pos = pbase + lane;
    int c = __popcll(__ballot(lane >= 1 && lane < ncw && cumk <= pbase));
    uint64_t starts = __ballot(lane >= 1 && lane < ncw && cumk > pbase && cumk <= pbase + 63);
    while (starts) {
      const int k = __builtin_ctzll(starts);
      starts &= starts - 1;
      c += (pos >= __builtin_amdgcn_readlane(cumk, k)) ? 1 : 0;
    }
    const int p = pos + __shfl(dk, c, 64);
    ix.c = c;
    ix.q = -1;
    if (pos < __shfl(endk, c, 64)) ix.q = FUSED ? src[p] : p;
  };
  auto fetch = [&](const Idx& ix, Pre& n) {
    const int q = ix.q;
    n.c = ix.c;
    // an empty place: no charge, so that its record adds zeros
    n.s = MAX_SPEC;
#pragma unroll
    for (int d = 0; d < 3; d++) n.x[d] = g.xmin[d], n.v[d] = 0.0, n.vf[d] = 0.f;
    if (q >= 0) {
      n.x[0] = x[q], n.x[1] = x[cap + q], n.x[2] = x[2 * cap + q];
      if constexpr (VF32) {
        const float* vf = (const float*)v;
        n.vf[0] = vf[q], n.vf[1] = vf[cap + q], n.vf[2] = vf[2 * cap + q];
      } else {
        n.v[0] = v[q], n.v[1] = v[cap + q], n.v[2] = v[2 * cap + q];
      }
      n.s = spec[q];
    }
  };
  Pre n1 = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.f, 0.f, 0.f}, 0, 0}, n2 = n1;

  // the two 16 x 16 halves of the cell's 16 x 32 tile
  dbl4 C0 = {0.0, 0.0, 0.0, 0.0}, C1 = C0;
  int cur = 0;  // the cell being accumulated (uniform)
  auto flush = [&](int c) {
    const int key = cellkey(c);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      S[oidx[r]] = C0[r];
      S[oidx[4 + r]] = C1[r];
    }
    C0 = dbl4{0.0, 0.0, 0.0, 0.0};
    C1 = C0;
    wave_lds_sync();
    // 2176 bytes from a 128-byte boundary: every store covers whole lines
    double2* dst = (double2*)(cellpart + (size_t)key * CS);
#pragma unroll
    for (int i = 0; i < CS / 2; i += 64)
      if (i + lane < CS / 2) dst[i + lane] = ((const double2*)S)[i + lane];
    wave_lds_sync();
  };
  // cells with no particles before the first particle
  while (cur < ncw && uniform(cum[cur + 1]) == 0) flush(cur++);

  Idx ix = {0, 0}, ix2 = {0, 0};
  index(0, ix);
  index(64, ix2);
  fetch(ix, n1);
  fetch(ix2, n2);
  index(128, ix);
  // the records of the chunk starting at particle base (VALU) from its
  // particles in nb; the particles two chunks ahead are then loaded into nb
  // (chunks alternate between n1 and n2)
  auto build = [&](int base, Pre& nb) {
    const int pos = base + lane;
    if (pos < total) {
      // the record: the reference's expressions, contracted to FMA where
      // the compiler finds them (this pass is the tolerance-bound one)
#pragma clang fp contract(fast)
      const double xI[3] = {nb.x[0], nb.x[1], nb.x[2]};
      const double vI[3] = {VF32 ? (double)nb.vf[0] : nb.v[0], VF32 ? (double)nb.vf[1] : nb.v[1],
                            VF32 ? (double)nb.vf[2] : nb.v[2]};
      const int s = nb.s;
      const int nc = nb.c;
      const int iX[3] = {sx + (nc & 3), sy + row0 + (nc >> 2), zc};
      double Lf[6], xn[3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        double xd = xI[d];
        if (fabs(xd - g.xmax[d]) < 1e-10 * g.dxs[d]) xd = g.xmax[d] - 1e-10 * g.dxs[d];
        xn[d] = xd;
        const double t = (xd - g.xmin[d]) * inv_dxs[d] - iX[d];
        const double f = fmin(fmax(t, 0.0), 1.0);
        Lf[2 * d] = 1.0 - f;
        Lf[2 * d + 1] = f;
      }
      double Bv[3] = {0.0, 0.0, 0.0};
      if constexpr (BC) {
        // centre-based B, pic_field_solver_ecsim.cpp:2097-2129; not for an empty
        // place, which lies in the block's first cell: a not-a-number there is
        // not this cell's
        if (s != MAX_SPEC) center_B(m, Bc, xn, b, Bv);
      } else {
        // the corner weights sum to 1 (InitStencil's normalization changes
        // them by rounding only)
        double lxy[4];
#pragma unroll
        for (int l = 0; l < 4; l++) lxy[l] = Lf[l >> 1] * Lf[2 + (l & 1)];
        // the cell's lower corner in the staged corners; corner l
        // at a fixed offset from it
        const double* sBc = sB + 3 * ((nc & 3) + 5 * (row0 + (nc >> 2)) + 25 * zl);
#pragma unroll
        for (int l = 0; l < 8; l++) {
          const double wl = lxy[l >> 1] * Lf[4 + (l & 1)];
          const int c = (l >> 2) + 5 * ((l >> 1) & 1) + 25 * (l & 1);
#pragma unroll
          for (int d = 0; d < 3; d++) Bv[d] += wl * sBc[3 * c + d];
        }
      }
      // alpha = c0 (I + P x + BB) with P = -QdT_over_2m B and BB = P P^T,
      // kept as its numerators a[]; c0 goes into the two factors that use it
      // (MC alpha, and q alpha v, which also takes the 1 / V of J)
      double qb[3];
#pragma unroll
      for (int ii = 0; ii < 3; ii++) qb[ii] = sconst[s][1] * Bv[ii];
      const double c0 = 1.0 / (1.0 + (qb[0] * qb[0] + qb[1] * qb[1] + qb[2] * qb[2]));
      double alpha[9];
      alpha[0] = 1.0 + qb[0] * qb[0];
      alpha[1] = qb[2] + qb[0] * qb[1];
      alpha[2] = -qb[1] + qb[0] * qb[2];
      alpha[3] = -qb[2] + qb[1] * qb[0];
      alpha[4] = 1.0 + qb[1] * qb[1];
      alpha[5] = qb[0] + qb[1] * qb[2];
      alpha[6] = qb[1] + qb[2] * qb[0];
      alpha[7] = -qb[0] + qb[2] * qb[1];
      alpha[8] = 1.0 + qb[2] * qb[2];
      const double MC = sconst[s][2] * c0, qc = sconst[s][0] * c0 * invV;
      double qv[3];
#pragma unroll
      for (int i = 0; i < 3; i++) {
        double vr = 0.0;
#pragma unroll
        for (int jj = 0; jj < 3; jj++) vr += alpha[3 * i + jj] * vI[jj];
        qv[i] = qc * vr;
      }
      double mo[3][3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        mo[d][0] = Lf[2 * d] * Lf[2 * d];
        mo[d][1] = Lf[2 * d] * Lf[2 * d + 1];
        mo[d][2] = Lf[2 * d + 1] * Lf[2 * d + 1];
      }
      double* R = R0 + lane;
#define FLD(f) R[(f) * FS]
#pragma unroll
      for (int ty = 0; ty < 3; ty++)
#pragma unroll
        for (int tx = 0; tx < 3; tx++) FLD(F_A + tx + 3 * ty) = mo[0][tx] * mo[1][ty];
#pragma unroll
      for (int bx = 0; bx < 2; bx++)
#pragma unroll
        for (int d = 0; d < 3; d++) FLD(F_A + 9 + 3 * bx + d) = Lf[bx] * qv[d];
      FLD(F_ONE) = 1.0;
#pragma unroll
      for (int k = 0; k < 9; k++) FLD(F_MA + k) = MC * alpha[k];
#pragma unroll
      for (int tz = 0; tz < 3; tz++) FLD(F_MZ + tz) = mo[2][tz];
#pragma unroll
      for (int bz = 0; bz < 2; bz++)
#pragma unroll
        for (int by = 0; by < 2; by++) FLD(F_WYZ + by + 2 * bz) = Lf[2 + by] * Lf[4 + bz];
#undef FLD
    }
    if (!SPARSE || base + 128 < total) {
      fetch(ix, nb);  // in flight while two chunks are accumulated
      index(base + 192, ix);
    }
  };
  // the matrix products of that chunk, cell by cell, and the finished cells' records
  auto accumulate = [&](int base) {
    const int cend = (base + 64 < total) ? base + 64 : total;
    int q = base;
    while (q < cend) {
      const int ce = uniform(cum[cur + 1]);
      const int se = ce < cend ? ce : cend;
      // steps of 4 particles
      const int nfull = (se - q) >> 2;
      const double* R = R0 + (q - base + slot);
      if (SPARSE && nfull > 0 && nfull <= 2) {
        const double a0 = R[oa], a1 = R[oa + 4];
        const double b00 = R[o0a] * R[o0b], b01 = R[o0a + 4] * R[o0b + 4];
        const double b10 = R[o1a] * R[o1b], b11 = R[o1a + 4] * R[o1b + 4];
        C0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b00, C0, 0, 0, 0);
        C1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b10, C1, 0, 0, 0);
        if (nfull == 2) {
          C0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b01, C0, 0, 0, 0);
          C1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b11, C1, 0, 0, 0);
        }
      } else if (nfull > 0) {
        // the raw operands of four steps in flight ahead of the products (the
        // LDS latency under load exceeds one step's two MFMAs), two steps to
        // a ds_read2_b64; the factors are multiplied just before use.  The five
        // running LDS addresses are opaque to the compiler, which otherwise adds
        // a common offset to each of them again for every pair of steps, vector
        // instructions in a wavefront's way to its next product.
        struct Ops {
          double a[2], x0[2], y0[2], x1[2], y1[2];
        };
        typedef const __attribute__((address_space(3))) double* lds_t;
        unsigned pA = (unsigned)(size_t)(lds_t)(R + oa), pX0 = (unsigned)(size_t)(lds_t)(R + o0a),
                 pY0 = (unsigned)(size_t)(lds_t)(R + o0b), pX1 = (unsigned)(size_t)(lds_t)(R + o1a),
                 pY1 = (unsigned)(size_t)(lds_t)(R + o1b);
        auto ld = [&](int k, Ops& o) {
#pragma unroll
          for (int i = 0; i < 2; i++) {
            o.a[i] = ((lds_t)(size_t)pA)[k + 4 * i];
            o.x0[i] = ((lds_t)(size_t)pX0)[k + 4 * i];
            o.y0[i] = ((lds_t)(size_t)pY0)[k + 4 * i];
            o.x1[i] = ((lds_t)(size_t)pX1)[k + 4 * i];
            o.y1[i] = ((lds_t)(size_t)pY1)[k + 4 * i];
          }
        };
        auto step = [&](const Ops& o, int i) {
          const double b0 = o.x0[i] * o.y0[i], b1 = o.x1[i] * o.y1[i];
          C0 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[i], b0, C0, 0, 0, 0);
          C1 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[i], b1, C1, 0, 0, 0);
        };
        // two operand sets, each reloaded right after its products (the loads
        // of the four steps past the last one read records past the segment,
        // inside rec[], and are not used)
        Ops pa, pb;
        ld(0, pa);
        ld(8, pb);
        __builtin_amdgcn_sched_barrier(0);
        int t = nfull;
        for (; t >= 4; t -= 4) {
          // the scheduling barriers keep each reload where it is issued
          step(pa, 0);
          step(pa, 1);
          pA += 128, pX0 += 128, pY0 += 128, pX1 += 128, pY1 += 128;
          asm volatile("" : "+v"(pA), "+v"(pX0), "+v"(pY0), "+v"(pX1), "+v"(pY1));
          ld(0, pa);
          __builtin_amdgcn_sched_barrier(0);
          step(pb, 0);
          step(pb, 1);
          ld(8, pb);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (t >= 1) step(pa, 0);
        if (t >= 2) step(pa, 1);
        if (t >= 3) step(pb, 0);
      }
      if (SPARSE && q + 4 * nfull < se) {
        // the cell's last 1-3 particles in this chunk: the other slots add zero
        const double* Rt = R + 4 * nfull;
        double a = 0.0, b0 = 0.0, b1 = 0.0;
        if (q + 4 * nfull + slot < se) {
          a = Rt[oa];
          b0 = Rt[o0a] * Rt[o0b];
          b1 = Rt[o1a] * Rt[o1b];
        }
        C0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b0, C0, 0, 0, 0);
        C1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b1, C1, 0, 0, 0);
      }
      q = se;
      if (q == ce) {
        flush(cur++);
        while (cur < ncw && uniform(cum[cur + 1]) == q) flush(cur++);  // empty cells
      }
    }
  };
  if constexpr (!PAIRED) {
    for (int base = 0; base < total; base += 128) {
      build(base, n1);
      wave_lds_sync();
      accumulate(base);
      wave_lds_sync();  // the records are read before the next chunk overwrites them
      if (base + 64 < total) {
        build(base + 64, n2);
        wave_lds_sync();
        accumulate(base + 64);
        wave_lds_sync();
      }
    }
  } else {
    // phase p: waves 0-3 build chunk p/2 at even p and accumulate it at odd
    // p; waves 4-7 (the other wavefront of each SIMD) one phase later
    const int nch = (total + 63) / 64;
    if (lane == 0) atomicMax(&smaxchunks, nch);
    __syncthreads();
    const int grp = w >> 2;
    const int nphase = 2 * smaxchunks + 1;
    for (int ph = 0; ph < nphase; ph++) {
      const int k = ph - grp;
      if (k >= 0 && (k >> 1) < nch) {
        if ((k & 1) == 0) {
          if ((k >> 1) & 1)
            build(64 * (k >> 1), n2);
          else
            build(64 * (k >> 1), n1);
        } else
          accumulate(64 * (k >> 1));
      }
      __syncthreads();
    }
  }
}

template <bool BC, bool PAIRED, bool FUSED, bool VF32, bool SPARSE>
void launch(amps_ctx* c, double dt, const Split& sp4) {
  const int k = c->cur;
  // FUSED: the particles are read from the previous buffer through the
  // migration's source indices
  const int r = FUSED ? 1 - k : k;
  const unsigned grid = (unsigned)(c->mv.nb * (PAIRED || BC ? 8 : 8 << (4 - sp4.lw)) + sp4.extra);
  hipLaunchKernelGGL((k_deposit_cell_mfma<BC, PAIRED, FUSED, VF32, SPARSE>), dim3(grid), dim3(64 * waves_of<PAIRED>()), 0,
                     c->stream, c->mv, c->sp, dt, c->d_B, c->d_offset, c->cap, c->d_x[r], c->d_v[r],
                     c->precision == AMPS_FP32 ? 1 : 0, c->d_spec[r], c->d_cellpart, c->d_Bc, c->d_tmpsrc, sp4);
}

template <bool BC, bool PAIRED, bool FUSED>
void launch_v(amps_ctx* c, double dt, bool vf32) {
  Split s = {4, 0, nullptr, nullptr, nullptr};
  if constexpr (!PAIRED && !BC) {
    // fewer cells per wavefront where 16 would not give the chip its 8
    // wavefronts per CU (two workgroups): 8 blocks take 21, 13.6 and 10.5 us
    // with 16, 8 and 4; at 64 blocks (one round of wavefronts) 16 is ahead,
    // 40.9, 42.7 and 46.5 us, and on 7,456 blocks 5.88, 6.11 and 6.84 ms: each
    // wavefront pays once for its first loads
    const int64_t waves = (int64_t)c->mv.nb * 32, resident = (int64_t)c->n_cu * 8;
    s.lw = waves >= resident ? 4 : 2 * waves >= resident ? 3 : 2;
    if (s.lw == 4) {
      const Crowd cr = crowd_view(c);
      // fewer than half of them hold twice the mean
      s.extra = 4 * (int)std::min<int64_t>(std::min(cr.slots, cr.ntiles / 2), c->n / CROWD_MIN);
      s.count = cr.count, s.list = cr.list, s.crowded = cr.flag;
    }
  }
  // by the host's count, which deletions since then can only have lowered
  const bool sparse = !PAIRED && c->n < (int64_t)SPARSE_MEAN * c->mv.nb * NCELL;
  if (sparse)
    vf32 ? launch<BC, PAIRED, FUSED, true, !PAIRED>(c, dt, s) : launch<BC, PAIRED, FUSED, false, !PAIRED>(c, dt, s);
  else
    vf32 ? launch<BC, PAIRED, FUSED, true, false>(c, dt, s) : launch<BC, PAIRED, FUSED, false, false>(c, dt, s);
}

}  // namespace

namespace amps {
int launch_deposit_cell_mfma(amps_ctx* c, double dt) {
  const bool paired = c->dep_paired != 0;
  const bool vf32 = c->precision == AMPS_FP32;
  if (c->pending_gather) {
    // the records of the last compaction are still where it found them: the
    // pass reads them there (set only with the single-phase pass)
    if (paired) return fail(AMPS_E_STATE, "deposit: records left by a step's migration need the single-phase cell pass");
    c->b_center ? launch_v<true, false, true>(c, dt, vf32) : launch_v<false, false, true>(c, dt, vf32);
    return 0;
  }
  if (c->b_center)
    paired ? launch_v<true, true, false>(c, dt, vf32) : launch_v<true, false, false>(c, dt, vf32);
  else
    paired ? launch_v<false, true, false>(c, dt, vf32) : launch_v<false, false, false>(c, dt, vf32);
  return 0;
}
}  // namespace amps
