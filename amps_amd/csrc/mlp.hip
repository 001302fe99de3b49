// mlp.hip — the cutoff surrogate network on BF16 MFMA (gfx950).
//
// Network 6 -> 128 -> 128 -> 1 with GELU, BF16 weights and activations, FP32
// accumulation (v_mfma_f32_16x16x32_bf16; x16 where the depth is 16 or less).
// Inference: a resident grid, every wavefront on its own 16 samples at a time,
// W2 in LDS.  Training: one workgroup per 32 samples, wave w owning hidden
// units 16w..16w+15, forward, loss and backward fused in one kernel that
// writes a per-workgroup gradient partial; a second kernel reduces the
// partials in a fixed order, applies Adam to the
// FP32 master weights, refreshes the BF16 copies (W2 is kept in both
// orientations so every MFMA operand is a contiguous 128-bit load) and
// advances the step count and batch offset, kept in two device-memory slots
// that consecutive steps use in turn.  Two training steps are captured in one
// hipGraph.
//
// Parameter layout: W1[128][6] | b1[128] | W2[128][128] | b2[128] | w3[128] | b3
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "amps_common.h"

using namespace amps;

namespace {

constexpr int DIN = 6, HID = 128;
constexpr int TB = 64;  // batches are multiples of this
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + HID * DIN, OFF_W2 = OFF_B1 + HID, OFF_B2 = OFF_W2 + HID * HID,
              OFF_W3 = OFF_B2 + HID, OFF_B3 = OFF_W3 + HID, NPARAM = OFF_B3 + 1;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16p __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// two values to BF16, rounded to nearest even (v_cvt_pk_bf16_f32); a in the low half
__device__ __forceinline__ unsigned f2bf2(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16p));
}
__device__ __forceinline__ unsigned short f2bf(float f) { return (unsigned short)f2bf2(f, 0.f); }
__device__ __forceinline__ float bf_lo(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

// Phi(z) = (1 + erf(z / sqrt 2)) / 2 and E = exp(-z^2 / 2), which the
// derivative of GELU uses too.  Below |z| = 1.25, 1/2 + z S(z^2); above,
// the tail q = E t P(t) with t = 1 / (1 + 0.3 |z|), for z > 0 as 1 - q (the
// form of Hastings' rational approximations to erfc).  S and P were fitted
// for this, to the least largest error in Phi and in q / E: 5e-11 and 1.6e-7
// of q, below FP32 rounding, and the tail keeps its relative precision, which
// 1 + erf loses: over |z| <= 12 the largest errors are 7.3e-8 in Phi and 3.8e-7
// in GELU, where erff's were 7.5e-8 and 4.5e-7.  GELU is what bounds inference
// (2^28 of them for 2^20 samples): both branches are some 25 vector
// instructions without a jump, where erff's two were 45 with one.
__device__ __forceinline__ float phi(float z, float& E) {
#pragma clang fp contract(fast)
  const float a = fabsf(z), u = z * z;
  E = __builtin_amdgcn_exp2f(u * -0.72134752044448170f);
  float S = 4.659529819e-07f;
  S = S * u - 9.006645299e-06f;
  S = S * u + 1.149300540e-04f;
  S = S * u - 1.187012792e-03f;
  S = S * u + 9.973455175e-03f;
  S = S * u - 6.649036553e-02f;
  S = S * u + 3.989422798e-01f;
  const float inner = z * S + 0.5f;
  const float t = __builtin_amdgcn_rcpf(a * 0.3f + 1.0f);
  float P = -4.206679138e-02f;
  P = P * t + 5.168405842e-02f;
  P = P * t + 5.813878488e-02f;
  P = P * t + 8.168559249e-02f;
  P = P * t + 1.112835230e-01f;
  P = P * t + 1.192786159e-01f;
  P = P * t + 1.197082510e-01f;
  const float q = (P * t) * E;
  const float outer = z < 0.0f ? q : 1.0f - q;
  return a < 1.25f ? inner : outer;
}
__device__ __forceinline__ bf16x4 ld4(const unsigned short* p) { return *(const bf16x4*)p; }
__device__ __forceinline__ bf16x8 ld8(const unsigned short* p) { return *(const bf16x8*)p; }
__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma8(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <int ROR>
__device__ __forceinline__ float row_ror(float x) {  // within the 16 lanes sharing lane/16
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x120 + ROR, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum16(float x) {  // over lanes sharing lane/16
  x += row_ror<1>(x);
  x += row_ror<2>(x);
  x += row_ror<4>(x);
  x += row_ror<8>(x);
  return x;
}
__device__ __forceinline__ float sum_rows(float x) {  // over the 4 row groups (lane/16)
  x += __shfl_xor(x, 16);
  x += __shfl_xor(x, 32);
  return x;
}

struct MlpView {
  const float* theta;             // FP32 master parameters
  const unsigned short* W1b;      // [128][16] bf16, k >= 6 zero
  const unsigned short* W2b;      // [128][128] bf16 (n, k)
  const unsigned short* W2Tb;     // [128][128] bf16 (k, n)
};

// Inference.  With the hidden units as the rows of every product (D = W H^T), a
// lane holds four consecutive units of one sample, so a layer's activations
// go to LDS as one 8-byte write per tile and come back as the next
// product's 16-byte operand, and the output sum needs two lane exchanges.
// The grid is resident: a workgroup copies W2 into LDS once, in operand order
// (32 KB, conflict-free 16-byte reads), and its wavefronts then take 16 samples
// at a time with no barrier between them.  Bound by the vector work of 256 GELUs
// a sample: 2^20 samples take 0.25 ms, 0.55 with a workgroup per 64 samples that
// read W2 from L2, wrote both orientations and called erff.  FWD_WGS per CU: 50 KB
// of LDS each.
constexpr int HP = HID + 8;  // row stride of [sample][HID] tiles: 16 B reads on distinct banks
constexpr int FWD_WGS = 3;

__global__ __launch_bounds__(256) void k_mlp_forward(MlpView mv, const float* __restrict__ X, int64_t n,
                                                      float* __restrict__ y) {
  __shared__ __align__(16) unsigned short sW2[HID * HID];
  __shared__ __align__(16) unsigned short sH[4][16 * HP];
  __shared__ __align__(16) float sb1[HID], sb2[HID], sw3[HID];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, rl = l & 15, g = l >> 4;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int f = w + 4 * i;  // operand f: rows 16 (f / 4) .., depth 32 (f % 4) ..
    *(bf16x8*)(sW2 + (f * 64 + l) * 8) = ld8(mv.W2b + (16 * (f >> 2) + rl) * HID + 32 * (f & 3) + 8 * g);
  }
  if (threadIdx.x < HID) {
    sb1[threadIdx.x] = mv.theta[OFF_B1 + threadIdx.x];
    sb2[threadIdx.x] = mv.theta[OFF_B2 + threadIdx.x];
    sw3[threadIdx.x] = mv.theta[OFF_W3 + threadIdx.x];
  }
  const float b3 = mv.theta[OFF_B3];
  bf16x4 w1[8];
#pragma unroll
  for (int t = 0; t < 8; t++) w1[t] = ld4(mv.W1b + (16 * t + rl) * 16 + 4 * g);
  __syncthreads();
  unsigned short* H = sH[w];
  const int64_t ntiles = (n + 15) / 16;
  // this lane's inputs of a tile: X[row][4 g .. 4 g + 3] of its sample, columns past the sixth zero
  auto load = [&](int64_t tile, f32x2& xa, f32x2& xb) {
    const int64_t r = 16 * tile + rl;
    xa = f32x2{0.f, 0.f}, xb = xa;
    if (r < n && g < 2) {
      const float* px = X + r * DIN + 4 * g;
      xa = *(const f32x2*)px;
      if (g == 0) xb = *(const f32x2*)(px + 2);
    }
  };
  int64_t tile = (int64_t)blockIdx.x * 4 + w;
  f32x2 xa, xb;
  if (tile < ntiles) load(tile, xa, xb);
  for (; tile < ntiles; tile += (int64_t)gridDim.x * 4) {
    const uint2 xp = {f2bf2(xa[0], xa[1]), f2bf2(xb[0], xb[1])};
    const bf16x4 bx = __builtin_bit_cast(bf16x4, xp);
    load(tile + (int64_t)gridDim.x * 4, xa, xb);  // rows past n read as zero
    float E;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const f32x4 z = mfma(w1[t], bx, *(const f32x4*)(sb1 + 16 * t + 4 * g));
      const uint2 h = {f2bf2(z[0] * phi(z[0], E), z[1] * phi(z[1], E)),
                       f2bf2(z[2] * phi(z[2], E), z[3] * phi(z[3], E))};
      *(uint2*)(H + rl * HP + 16 * t + 4 * g) = h;
    }
    // the LDS operations of one wavefront execute in issue order: a compiler
    // barrier is all the ordering needed
    asm volatile("" ::: "memory");
    bf16x8 h1[4];
#pragma unroll
    for (int k = 0; k < 4; k++) h1[k] = ld8(H + rl * HP + 32 * k + 8 * g);
    float ys = 0.f;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      f32x4 z = *(const f32x4*)(sb2 + 16 * t + 4 * g);
#pragma unroll
      for (int k = 0; k < 4; k++) z = mfma8(ld8(sW2 + ((4 * t + k) * 64 + l) * 8), h1[k], z);
      const f32x4 w3 = *(const f32x4*)(sw3 + 16 * t + 4 * g);
      const unsigned h01 = f2bf2(z[0] * phi(z[0], E), z[1] * phi(z[1], E));
      const unsigned h23 = f2bf2(z[2] * phi(z[2], E), z[3] * phi(z[3], E));
      ys += bf_lo(h01) * w3[0];
      ys += bf_hi(h01) * w3[1];
      ys += bf_lo(h23) * w3[2];
      ys += bf_hi(h23) * w3[3];
    }
    asm volatile("" ::: "memory");
    ys = sum_rows(ys);
    const int64_t r = 16 * tile + rl;
    if (g == 0 && r < n) y[r] = ys + b3;
  }
}

// Fused forward + MSE loss + backward for TS = 32 rows of the batch starting
// at rows [*batch_off, ...) of the data (wrapping at n), spread over the
// columns: wavefront w owns hidden units 16w .. 16w + 15 of both layers, so
// that the chain of dependent products is short.  A step is bound by that chain
// and by the gradient partials (70 KB a workgroup, written here and read
// back by the update): 32 rows a workgroup, two wavefronts per SIMD, halve the
// partials of 16 rows, and fill one product of depth 32.  The W2 part of a
// partial is kept in the order of the accumulators (a lane's four values next to
// each other), one 16-byte store per tile.  A batch of 4,096: 11.6 us, and 4.4 the
// update (20.5 and 6.7 with 16 rows, 4-byte stores and a 64-bit modulo per
// row; 64 rows would leave 64 workgroups of 7 us of vector work).  LDS rows are padded (HP, TP) off the
// bank period; every MFMA operand is an aligned 8- or 16-byte read.
constexpr int TS = 32;               // samples per training workgroup
constexpr int TTHREADS = 512;
constexpr int TP = TS + 8;           // row stride of [HID][TS] and [16][TS] tiles
// a partial: W2 as [tile n][tile k][lane][4], then W1, b1 (as in theta), b2, w3, b3
constexpr int GOFF_W1 = HID * HID, GOFF_B1 = GOFF_W1 + HID * DIN, GOFF_B2 = GOFF_B1 + HID, GOFF_W3 = GOFF_B2 + HID,
              GOFF_B3 = GOFF_W3 + HID, GSTRIDE = (GOFF_B3 + 1 + 63) / 64 * 64;

// the parameter at place jp of a partial, -1 for padding
__device__ __forceinline__ int param_of(int jp) {
  if (jp < GOFF_W1) {
    const int v = jp & 3, l = (jp >> 2) & 63, kt = (jp >> 8) & 7, nt = jp >> 11;
    return OFF_W2 + (16 * nt + 4 * (l >> 4) + v) * HID + 16 * kt + (l & 15);
  }
  if (jp < GOFF_B2) return OFF_W1 + jp - GOFF_W1;
  return jp <= GOFF_B3 ? OFF_B2 + jp - GOFF_B2 : -1;
}

__global__ __launch_bounds__(TTHREADS) void k_mlp_train(MlpView mv, const float* __restrict__ X,
                                                    const float* __restrict__ T, int64_t n, int batch,
                                                    const int64_t* __restrict__ batch_off,
                                                    float* __restrict__ gpart,
                                                    float* __restrict__ lpart) {
  __shared__ __align__(16) unsigned short Xb[TS * 16], XTb[16 * TP];
  __shared__ __align__(16) unsigned short H1b[TS * HP], H1Tb[HID * TP];
  __shared__ __align__(16) unsigned short D2b[TS * HP], D2Tb[HID * TP], D1Tb[HID * TP];
  __shared__ __align__(16) float ypart[8][TS], sT[TS];
  const int64_t base = (batch_off ? *batch_off : 0) + (int64_t)blockIdx.x * TS;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, rl = l & 15, g = l >> 4, kq = 4 * g;
  const int nn = 16 * w + rl;  // this lane's hidden unit
  // everything this lane reads from the weights and targets, loaded up front
  // so that the load latency is paid once, not once per phase
  const bf16x4 bw1 = ld4(mv.W1b + nn * 16 + kq);
  bf16x8 bw2[4], bw2t[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    bw2[k] = ld8(mv.W2b + nn * HID + 32 * k + 8 * g);
    bw2t[k] = ld8(mv.W2Tb + nn * HID + 32 * k + 8 * g);
  }
  const float b1 = mv.theta[OFF_B1 + nn], b2 = mv.theta[OFF_B2 + nn], w3 = mv.theta[OFF_W3 + nn];
  const float b3 = mv.theta[OFF_B3];
  {
    // batches wrap: past the end only in the last one before that
    const int m = threadIdx.x >> 4, k = threadIdx.x & 15;
    int64_t r = base + m;
    if (r >= n) r %= n;
    const unsigned short h = f2bf((k < DIN) ? X[r * DIN + k] : 0.0f);
    Xb[m * 16 + k] = h;
    XTb[k * TP + m] = h;
    if (k == DIN) sT[m] = T[r];
  }
  __syncthreads();
  float* gp = gpart + (int64_t)blockIdx.x * GSTRIDE;
  // layer 1; the D layout: sample 16 t + kq + v, unit nn.  Of a pre-activation z
  // the backward needs GELU's derivative Phi(z) + z exp(-z^2 / 2) / sqrt(2 pi)
  float d1[2][4];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const f32x4 z = mfma(ld4(Xb + (16 * t + rl) * 16 + kq), bw1, f32x4{b1, b1, b1, b1});
    float h[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      float E;
      const float ph = phi(z[v], E);
      h[v] = z[v] * ph;
      d1[t][v] = ph + z[v] * E * 0.39894228040143268f;
    }
    const uint2 hb = {f2bf2(h[0], h[1]), f2bf2(h[2], h[3])};
    *(uint2*)(H1Tb + nn * TP + 16 * t + kq) = hb;
#pragma unroll
    for (int v = 0; v < 4; v++)
      H1b[(16 * t + kq + v) * HP + nn] = (unsigned short)((v < 2 ? hb.x : hb.y) >> (16 * (v & 1)));
  }
  __syncthreads();
  // layer 2 for the same units, and the output layer's partial sums
  float d2[2][4], h2[2][4];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    f32x4 z = {b2, b2, b2, b2};
#pragma unroll
    for (int k = 0; k < 4; k++) z = mfma8(ld8(H1b + (16 * t + rl) * HP + 32 * k + 8 * g), bw2[k], z);
    float h[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      float E;
      const float ph = phi(z[v], E);
      h[v] = z[v] * ph;
      d2[t][v] = ph + z[v] * E * 0.39894228040143268f;
    }
    const unsigned h01 = f2bf2(h[0], h[1]), h23 = f2bf2(h[2], h[3]);
    h2[t][0] = bf_lo(h01), h2[t][1] = bf_hi(h01), h2[t][2] = bf_lo(h23), h2[t][3] = bf_hi(h23);
    f32x4 ys;
#pragma unroll
    for (int v = 0; v < 4; v++) ys[v] = sum16(h2[t][v] * w3);
    if (rl == 0) *(f32x4*)(&ypart[w][16 * t + kq]) = ys;
  }
  __syncthreads();
  // the loss gradient of this lane's rows (every wave computes the same)
  float dy[2][4];
  float lsum = 0.f;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    f32x4 ys = *(const f32x4*)(&ypart[0][16 * t + kq]);
#pragma unroll
    for (int q = 1; q < 8; q++) ys += *(const f32x4*)(&ypart[q][16 * t + kq]);
    const f32x4 tv = *(const f32x4*)(sT + 16 * t + kq);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const float res = (ys[v] + b3) - tv[v];
      dy[t][v] = 2.0f * res / (float)batch;
      lsum += res * res;
    }
  }
  // dZ2 = dy w3 gelu'(z2) on this wave's units; their b2 and w3 gradients
  {
    float sb = 0.f, sw = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      float d[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        d[v] = dy[t][v] * w3 * d2[t][v];
        sb += d[v];
        sw += dy[t][v] * h2[t][v];
      }
      const uint2 db = {f2bf2(d[0], d[1]), f2bf2(d[2], d[3])};
      *(uint2*)(D2Tb + nn * TP + 16 * t + kq) = db;
#pragma unroll
      for (int v = 0; v < 4; v++)
        D2b[(16 * t + kq + v) * HP + nn] = (unsigned short)((v < 2 ? db.x : db.y) >> (16 * (v & 1)));
    }
    sb = sum_rows(sb);
    sw = sum_rows(sw);
    if (l < 16) {
      gp[GOFF_B2 + nn] = sb;
      gp[GOFF_W3 + nn] = sw;
    }
  }
  if (w == 0) {
    float ds = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) ds += dy[t][v];
    float ls = lsum;
    ds = sum_rows(ds);
    ls = sum_rows(ls);
    if (l == 0) {
      gp[GOFF_B3] = ds;
      lpart[blockIdx.x] = ls;
    }
  }
  __syncthreads();
  // dH1 = dZ2 W2 and dZ1 = dH1 gelu'(z1) for this wave's units (of layer 1)
  {
    float sb = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; k++) acc = mfma8(ld8(D2b + (16 * t + rl) * HP + 32 * k + 8 * g), bw2t[k], acc);
      float d[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        d[v] = acc[v] * d1[t][v];
        sb += d[v];
      }
      const uint2 db = {f2bf2(d[0], d[1]), f2bf2(d[2], d[3])};
      *(uint2*)(D1Tb + nn * TP + 16 * t + kq) = db;
    }
    sb = sum_rows(sb);
    if (l < 16) gp[GOFF_B1 + nn] = sb;
  }
  // dW2[n][k] = sum_m dZ2[m][n] H1[m][k] for this wave's rows n, one product per tile
  {
    const bf16x8 a = ld8(D2Tb + nn * TP + 8 * g);
#pragma unroll
    for (int jt = 0; jt < 8; jt++) {
      const f32x4 acc = mfma8(a, ld8(H1Tb + (16 * jt + rl) * TP + 8 * g), f32x4{0.f, 0.f, 0.f, 0.f});
      *(f32x4*)(gp + ((w * 8 + jt) * 64 + l) * 4) = acc;
    }
  }
  // dW1[n][j] = sum_m dZ1[m][n] X[m][j]: the wave's own rows of D1Tb (the
  // LDS operations of one wavefront execute in issue order, so a compiler
  // barrier is all the ordering needed)
  asm volatile("" ::: "memory");
  {
    const f32x4 acc = mfma8(ld8(D1Tb + nn * TP + 8 * g), ld8(XTb + rl * TP + 8 * g), f32x4{0.f, 0.f, 0.f, 0.f});
    if (rl < DIN) {
#pragma unroll
      for (int v = 0; v < 4; v++) gp[GOFF_W1 + (16 * w + kq + v) * DIN + rl] = acc[v];
    }
  }
}

// Sum the workgroup partials in a fixed order, Adam on the FP32 master copy,
// BF16 refresh.  A workgroup takes 64 consecutive parameters: wavefront w of
// its 16 sums rows [w r, (w + 1) r) of the partials (r = nwg / 16 rounded
// up) for the 64 parameters, one coalesced 256-byte row per load, and the
// sixteen sums are added in order.  The moments, the step's factors and the
// partials are loaded and worked out together, ahead of the barrier.  The step count and batch offset are
// read from ctr_in and the advanced ones written to ctr_out by the first
// workgroup: two slots used in turn by consecutive steps, so no workgroup
// reads what another is writing.
constexpr int ADAM_PARAMS = 64, ADAM_WAVES = 16;

__global__ __launch_bounds__(64 * ADAM_WAVES) void k_mlp_adam(const float* __restrict__ gpart, int nwg, float* theta,
                                                   float* m, float* v, float* grad_out,
                                                   const int64_t* __restrict__ ctr_in, int64_t* ctr_out,
                                                   int64_t batch, int64_t nrows, float lr, int apply,
                                                   unsigned short* W1b, unsigned short* W2b, unsigned short* W2Tb) {
  __shared__ float part[ADAM_WAVES][ADAM_PARAMS];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int jp = blockIdx.x * ADAM_PARAMS + l;  // place in the partials
  const int j = param_of(jp);
  const int64_t step = ctr_in[0] + 1;
  const int rows = (nwg + ADAM_WAVES - 1) / ADAM_WAVES, k0 = w * rows, k1 = min(nwg, k0 + rows);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float m0 = 0.f, v0 = 0.f, th0 = 0.f, c1 = 1.f, c2 = 1.f;
  if (w == 0 && j >= 0 && apply) m0 = m[j], v0 = v[j], th0 = theta[j];
  float gsum = 0.f;
  if (j >= 0) {
#pragma unroll 8
    for (int k = k0; k < k1; k++) gsum += gpart[(int64_t)k * GSTRIDE + jp];
  }
  if (w == 0 && apply) {
    c1 = 1.f - powf(b1, (float)step);
    c2 = 1.f - powf(b2, (float)step);
  }
  part[w][l] = gsum;
  __syncthreads();
  if (w == 0 && j >= 0) {
    float gt = part[0][l];
#pragma unroll
    for (int q = 1; q < ADAM_WAVES; q++) gt += part[q][l];
    if (grad_out) grad_out[j] = gt;
    if (apply) {
      const float mj = b1 * m0 + (1.f - b1) * gt;
      const float vj = b2 * v0 + (1.f - b2) * gt * gt;
      m[j] = mj;
      v[j] = vj;
      const float mh = mj / c1;
      const float vh = vj / c2;
      const float th = th0 - lr * mh / (sqrtf(vh) + eps);
      theta[j] = th;
      const unsigned short hb = f2bf(th);
      if (j < OFF_B1) {
        W1b[(j / DIN) * 16 + (j % DIN)] = hb;
      } else if (j >= OFF_W2 && j < OFF_B2) {
        const int q = j - OFF_W2, nn = q / HID, kk = q % HID;
        W2b[nn * HID + kk] = hb;
        W2Tb[kk * HID + nn] = hb;
      }
    }
  }
  if (apply && blockIdx.x == 0 && threadIdx.x == 0) {
    ctr_out[0] = step;
    ctr_out[1] = (ctr_in[1] + batch) % nrows;
  }
}

__global__ __launch_bounds__(256) void k_mlp_refresh_bf16(const float* theta, unsigned short* W1b,
                                                           unsigned short* W2b, unsigned short* W2Tb) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < HID * 16) {
    const int nn = j / 16, kk = j % 16;
    W1b[j] = (kk < DIN) ? f2bf(theta[OFF_W1 + nn * DIN + kk]) : (unsigned short)0;
  }
  if (j < HID * HID) {
    const int nn = j / HID, kk = j % HID;
    const unsigned short h = f2bf(theta[OFF_W2 + j]);
    W2b[j] = h;
    W2Tb[kk * HID + nn] = h;
  }
}

}  // namespace

// =====================================================================
// host side
// =====================================================================
struct MlpState {
  float* theta = nullptr;
  float* m = nullptr;
  float* v = nullptr;
  unsigned short *W1b = nullptr, *W2b = nullptr, *W2Tb = nullptr;
  float *X = nullptr, *T = nullptr;
  int64_t n = 0, cap = 0;
  float* gpart = nullptr;
  float* lpart = nullptr;
  int64_t gpart_wg = 0;
  // two slots of (Adam step count, batch offset), read and written in turn by
  // consecutive steps; slot 0 is the current one between calls
  int64_t* step_dev = nullptr;
  float* grad = nullptr;
  float* qX = nullptr;
  float* qy = nullptr;
  int64_t qcap = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int graph_batch = 0;
  float graph_lr = 0.f;
};

namespace amps {
void mlp_free(amps_ctx* c) {
  MlpState* s = (MlpState*)c->mlp_state;
  if (!s) return;
  if (s->gexec) (void)hipGraphExecDestroy(s->gexec);
  if (s->graph) (void)hipGraphDestroy(s->graph);
  for (void* p : {(void*)s->theta, (void*)s->m, (void*)s->v, (void*)s->W1b, (void*)s->W2b,
                  (void*)s->W2Tb, (void*)s->X, (void*)s->T, (void*)s->gpart, (void*)s->lpart,
                  (void*)s->step_dev, (void*)s->grad, (void*)s->qX, (void*)s->qy})
    (void)hipFree(p);
  delete s;
  c->mlp_state = nullptr;
}
}  // namespace amps

static MlpView view(MlpState* s) { return MlpView{s->theta, s->W1b, s->W2b, s->W2Tb}; }

// The captured training step holds the data and partial buffers' addresses
// and the row count: it is dropped whenever one of them changes.
static void drop_graph(MlpState* s) {
  if (s->gexec) (void)hipGraphExecDestroy(s->gexec);
  if (s->graph) (void)hipGraphDestroy(s->graph);
  s->gexec = nullptr;
  s->graph = nullptr;
}

static int ensure_gpart(amps_ctx* c, MlpState* s, int64_t nwg) {
  if (nwg <= s->gpart_wg) return 0;
  drop_graph(s);
  (void)hipFree(s->gpart);
  (void)hipFree(s->lpart);
  s->gpart = nullptr;
  s->lpart = nullptr;
  HIP_TRY(hipMalloc(&s->gpart, sizeof(float) * GSTRIDE * nwg));
  HIP_TRY(hipMalloc(&s->lpart, sizeof(float) * nwg));
  s->gpart_wg = nwg;
  (void)c;
  return 0;
}

extern "C" int amps_gpu_mlp_init(amps_ctx* c, const float* theta) {
  if (!c || !theta) return fail(AMPS_E_ARG, "mlp_init: null argument");
  (void)hipSetDevice(c->device);
  MlpState* s = (MlpState*)c->mlp_state;
  if (!s) {
    s = new MlpState();
    c->mlp_state = s;
    HIP_TRY(hipMalloc(&s->theta, sizeof(float) * NPARAM));
    HIP_TRY(hipMalloc(&s->m, sizeof(float) * NPARAM));
    HIP_TRY(hipMalloc(&s->v, sizeof(float) * NPARAM));
    HIP_TRY(hipMalloc(&s->grad, sizeof(float) * NPARAM));
    HIP_TRY(hipMalloc(&s->W1b, 2 * HID * 16));
    HIP_TRY(hipMalloc(&s->W2b, 2 * HID * HID));
    HIP_TRY(hipMalloc(&s->W2Tb, 2 * HID * HID));
    HIP_TRY(hipMalloc(&s->step_dev, sizeof(int64_t) * 4));
  }
  HIP_TRY(hipMemcpyAsync(s->theta, theta, sizeof(float) * NPARAM, hipMemcpyHostToDevice, c->stream));
  HIP_TRY(hipMemsetAsync(s->m, 0, sizeof(float) * NPARAM, c->stream));
  HIP_TRY(hipMemsetAsync(s->v, 0, sizeof(float) * NPARAM, c->stream));
  HIP_TRY(hipMemsetAsync(s->step_dev, 0, sizeof(int64_t) * 4, c->stream));
  hipLaunchKernelGGL(k_mlp_refresh_bf16, dim3((HID * HID + 255) / 256), dim3(256), 0, c->stream, s->theta,
                     s->W1b, s->W2b, s->W2Tb);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  return AMPS_OK;
}

static MlpState* mstate(amps_ctx* c) { return c ? (MlpState*)c->mlp_state : nullptr; }

extern "C" int amps_gpu_mlp_get_params(amps_ctx* c, float* theta, int64_t* step) {
  MlpState* s = mstate(c);
  if (!s) return fail(AMPS_E_STATE, "mlp: call amps_gpu_mlp_init first");
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (theta) HIP_TRY(hipMemcpy(theta, s->theta, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  if (step) HIP_TRY(hipMemcpy(step, s->step_dev, sizeof(int64_t), hipMemcpyDeviceToHost));
  return AMPS_OK;
}

extern "C" int amps_gpu_mlp_set_data(amps_ctx* c, int64_t n, const float* X, const float* T) {
  MlpState* s = mstate(c);
  if (!s) return fail(AMPS_E_STATE, "mlp: call amps_gpu_mlp_init first");
  if (n <= 0 || !X || !T) return fail(AMPS_E_ARG, "mlp_set_data: empty data");
  (void)hipSetDevice(c->device);
  HIP_TRY(hipStreamSynchronize(c->stream));
  drop_graph(s);
  if (n > s->cap) {
    (void)hipFree(s->X);
    (void)hipFree(s->T);
    s->X = nullptr;
    s->T = nullptr;
    HIP_TRY(hipMalloc(&s->X, sizeof(float) * DIN * n));
    HIP_TRY(hipMalloc(&s->T, sizeof(float) * n));
    s->cap = n;
  }
  HIP_TRY(hipMemcpyAsync(s->X, X, sizeof(float) * DIN * n, hipMemcpyHostToDevice, c->stream));
  HIP_TRY(hipMemcpyAsync(s->T, T, sizeof(float) * n, hipMemcpyHostToDevice, c->stream));
  const int64_t zero = 0;
  HIP_TRY(hipMemcpyAsync(s->step_dev + 1, &zero, sizeof(int64_t), hipMemcpyHostToDevice, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  s->n = n;
  return AMPS_OK;
}

constexpr int ADAM_BLOCKS = (GSTRIDE + ADAM_PARAMS - 1) / ADAM_PARAMS;

// one Adam step reading the counters of slot `from` and writing the other
static void enqueue_step(amps_ctx* c, MlpState* s, int batch, float lr, int from) {
  const int nwg = batch / TS;
  const int64_t* in = s->step_dev + 2 * from;
  int64_t* out = s->step_dev + 2 * (1 - from);
  hipLaunchKernelGGL(k_mlp_train, dim3(nwg), dim3(TTHREADS), 0, c->stream, view(s), s->X, s->T, s->n,
                     batch, in + 1, s->gpart, s->lpart);
  hipLaunchKernelGGL(k_mlp_adam, dim3(ADAM_BLOCKS), dim3(64 * ADAM_WAVES), 0, c->stream, s->gpart, nwg, s->theta,
                     s->m, s->v, (float*)nullptr, in, out, (int64_t)batch, s->n, lr, 1, s->W1b, s->W2b, s->W2Tb);
}

// Gradient of the mean-squared error over the first n rows of the resident
// data (n a multiple of 64), optionally followed by one Adam step.
extern "C" int amps_gpu_mlp_grad(amps_ctx* c, int64_t n, float* grad_out, float* loss_out) {
  MlpState* s = mstate(c);
  if (!s || s->n == 0) return fail(AMPS_E_STATE, "mlp_grad: init and set_data first");
  if (n <= 0 || n % TB || n > s->n || n > (1 << 24)) return fail(AMPS_E_ARG, "mlp_grad: n must be a positive multiple of 64 <= data size");
  (void)hipSetDevice(c->device);
  const int nwg = (int)(n / TS);
  if (int r = ensure_gpart(c, s, nwg)) return r;
  int64_t zero = 0;
  HIP_TRY(hipMemcpyAsync(s->step_dev + 1, &zero, sizeof(int64_t), hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_mlp_train, dim3(nwg), dim3(TTHREADS), 0, c->stream, view(s), s->X, s->T, s->n, (int)n,
                     s->step_dev + 1, s->gpart, s->lpart);
  hipLaunchKernelGGL(k_mlp_adam, dim3(ADAM_BLOCKS), dim3(64 * ADAM_WAVES), 0, c->stream, s->gpart, nwg, s->theta,
                     s->m, s->v, s->grad, s->step_dev, s->step_dev + 2, (int64_t)0, s->n, 0.f, 0, s->W1b, s->W2b,
                     s->W2Tb);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (grad_out) HIP_TRY(hipMemcpy(grad_out, s->grad, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
  if (loss_out) {
    std::vector<float> lp((size_t)nwg);
    HIP_TRY(hipMemcpy(lp.data(), s->lpart, sizeof(float) * nwg, hipMemcpyDeviceToHost));
    double L = 0;
    for (float x : lp) L += x;
    *loss_out = (float)(L / (double)n);
  }
  return AMPS_OK;
}

// nsteps Adam steps on consecutive batches of the resident data (wrapping),
// replayed from one captured hipGraph.  loss_out[nsteps] (may be NULL)
// receives each step's batch loss.
extern "C" int amps_gpu_mlp_train(amps_ctx* c, int64_t nsteps, int32_t batch, double lr, float* loss_out) {
  MlpState* s = mstate(c);
  if (!s || s->n == 0) return fail(AMPS_E_STATE, "mlp_train: init and set_data first");
  if (batch <= 0 || batch % TB || batch > (1 << 20)) return fail(AMPS_E_ARG, "mlp_train: batch must be a positive multiple of 64");
  if (nsteps < 0) return fail(AMPS_E_ARG, "mlp_train: nsteps < 0");
  (void)hipSetDevice(c->device);
  const int nwg = batch / TS;
  if (int r = ensure_gpart(c, s, nwg)) return r;
  if (!s->gexec || s->graph_batch != batch || s->graph_lr != (float)lr) {
    drop_graph(s);
    // two steps, slot 0 -> 1 -> 0: a replay leaves the counters in slot 0
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    enqueue_step(c, s, batch, (float)lr, 0);
    enqueue_step(c, s, batch, (float)lr, 1);
    HIP_TRY(hipStreamEndCapture(c->stream, &s->graph));
    HIP_TRY(hipGraphInstantiate(&s->gexec, s->graph, nullptr, nullptr, 0));
    s->graph_batch = batch;
    s->graph_lr = (float)lr;
  }
  std::vector<float> lp;
  tbegin(c);
  if (loss_out) {
    // one step at a time, each batch loss read back
    lp.resize((size_t)nwg);
    for (int64_t i = 0; i < nsteps; i++) {
      enqueue_step(c, s, batch, (float)lr, (int)(i & 1));
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipMemcpyAsync(lp.data(), s->lpart, sizeof(float) * nwg, hipMemcpyDeviceToHost, c->stream));
      HIP_TRY(hipStreamSynchronize(c->stream));
      double Ls = 0;
      for (float x : lp) Ls += x;
      loss_out[i] = (float)(Ls / batch);
    }
  } else {
    for (int64_t i = 0; i + 1 < nsteps; i += 2) HIP_TRY(hipGraphLaunch(s->gexec, c->stream));
    if (nsteps & 1) {
      enqueue_step(c, s, batch, (float)lr, 0);
      HIP_TRY(hipGetLastError());
    }
  }
  if (nsteps & 1)  // the counters back in slot 0
    HIP_TRY(hipMemcpyAsync(s->step_dev, s->step_dev + 2, sizeof(int64_t) * 2, hipMemcpyDeviceToDevice, c->stream));
  tend(c, AMPS_K_MLP);
  HIP_TRY(hipStreamSynchronize(c->stream));
  return AMPS_OK;
}

// enough workgroups for a wavefront per tile, at most a resident grid
static unsigned forward_wgs(const amps_ctx* c, int64_t n) {
  const int64_t tiles = (n + 15) / 16, all = (int64_t)FWD_WGS * c->n_cu;
  return (unsigned)std::min((tiles + 3) / 4, all);
}

extern "C" int amps_gpu_mlp_predict(amps_ctx* c, int64_t n, const float* X, float* y) {
  MlpState* s = mstate(c);
  if (!s) return fail(AMPS_E_STATE, "mlp: call amps_gpu_mlp_init first");
  if (n < 0 || (n > 0 && (!X || !y))) return fail(AMPS_E_ARG, "mlp_predict: bad arguments");
  if (n == 0) return AMPS_OK;
  (void)hipSetDevice(c->device);
  if (n > s->qcap) {
    (void)hipFree(s->qX);
    (void)hipFree(s->qy);
    s->qX = nullptr;
    s->qy = nullptr;
    HIP_TRY(hipMalloc(&s->qX, sizeof(float) * DIN * n));
    HIP_TRY(hipMalloc(&s->qy, sizeof(float) * n));
    s->qcap = n;
  }
  if (int r = copy_to_device(c, s->qX, X, sizeof(float) * DIN * n)) return r;
  tbegin(c);
  hipLaunchKernelGGL(k_mlp_forward, dim3(forward_wgs(c, n)), dim3(256), 0, c->stream, view(s), s->qX, n, s->qy);
  HIP_TRY(hipGetLastError());
  tend(c, AMPS_K_MLP);
  return copy_to_host(c, y, s->qy, sizeof(float) * n);
}
