// mlp.hpp -- learned initial pressure for cons2prim: a 3 -> 64 -> 64 -> 1 MLP.
//
// Inputs (log D, |S|/D, tau/D) of a conserved state enter through fixed maps
// (log D, log1p(|S|/D), log of the non-kinetic part of tau/D; see features())
// and a per-feature affine normalisation;
// the output is the normalised log(p/D), so log p = log D + y/out_scale +
// out_mean (the map p/D <-> (|S|/D, tau/D) is scale free).  Hidden layers use
// ReLU.  Parameters are one float array (layout below); inference runs the
// 64x64 hidden layer as BF16 MFMA (v_mfma_f32_32x32x16_bf16, FP32 accumulate)
// over the 64 cells of a wavefront, training runs FP32 forward/backward.
#pragma once

namespace gh {
namespace mlp {

constexpr int H = 64;
// parameter layout (floats)
constexpr int OW1 = 0;                 // W1[64][3]
constexpr int OB1 = OW1 + H * 3;       // b1[64]
constexpr int OW2 = OB1 + H;           // W2[64 out][64 in]
constexpr int OB2 = OW2 + H * H;       // b2[64]
constexpr int OW3 = OB2 + H;           // w3[64]
constexpr int OB3 = OW3 + H;           // b3
constexpr int ONORM = OB3 + 1;         // in_mean[3], in_scale[3], out_mean, out_scale
constexpr int NPARAM = ONORM + 8;
constexpr int NTRAIN = ONORM;          // trained entries (the normalisation is fixed)

// features of a conserved state (D, |S|, tau), normalised: log D, log1p(q)
// and log e with q = |S|/D, t = tau/D and e = t + 1 - sqrt(1 + q^2), the part
// of tau/D that is not bulk kinetic energy.  For a cold gas e ~ (k - 1)(p/rho)/W
// with k = G/(G-1) and W the Lorentz factor, so log e carries log p where t and
// q alone hold it only in digits an FP32 input cannot keep.  e is formed in
// FP64 and floored at the rounding level of t.
GH_HD void features(const float* w, double D, double S, double tau, float* x) {
  double Dp = D > 1e-300 ? D : 1e-300;
  double q = S / Dp, t = tau / Dp;
  double e = t + 1. - sqrt(1. + q * q);
  double fl = 1e-16 * (1. + fabs(t));
  if (!(e > fl)) e = fl;
  double f0 = log(Dp), f1 = log1p(q), f2 = log(e);
  x[0] = (float)((f0 - w[ONORM + 0]) * w[ONORM + 3]);
  x[1] = (float)((f1 - w[ONORM + 1]) * w[ONORM + 4]);
  x[2] = (float)((f2 - w[ONORM + 2]) * w[ONORM + 5]);
}

// network output -> pressure guess
GH_HD double pressure_of(const float* w, double D, float y) {
  double lpd = (double)y / w[ONORM + 7] + w[ONORM + 6];
  return D * exp(lpd);
}

// FP32 forward of one sample; keeps the hidden activations for backprop
GH_HD float forward_f32(const float* w, const float* x, float* h1, float* h2) {
  for (int o = 0; o < H; ++o) {
    float a = w[OB1 + o];
    for (int k = 0; k < 3; ++k) a += w[OW1 + o * 3 + k] * x[k];
    h1[o] = a > 0.f ? a : 0.f;
  }
  for (int o = 0; o < H; ++o) {
    float a = w[OB2 + o];
    for (int k = 0; k < H; ++k) a += w[OW2 + o * H + k] * h1[k];
    h2[o] = a > 0.f ? a : 0.f;
  }
  float y = w[OB3];
  for (int k = 0; k < H; ++k) y += w[OW3 + k] * h2[k];
  return y;
}

}  // namespace mlp
}  // namespace gh

#ifndef GH_EMU
namespace gh {
namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Lane layout of v_mfma_f32_32x32x16_bf16 (checked on the device by
// tests/test_mlp.py::test_mfma_lane_layout):
//   A 32x16: lane l holds A[l%32][8*(l/32) + e], e = 0..7
//   B 16x32: lane l holds B[8*(l/32) + e][l%32]
//   D 32x32: lane l, register r holds D[8*(r/4) + 4*(l/32) + r%4][l%32]
__device__ __forceinline__ int d_row(int l, int r) { return 8 * (r / 4) + 4 * (l / 32) + (r % 4); }

// B operands of the hidden layer, pre-arranged per lane: for k-block kb (0..3)
// and n-block nb (0..1), lane l holds W2[nb*32 + l%32][kb*16 + 8*(l/32) + e]
// (B[k][n] = W2[n][k]).  Index: ((kb*2 + nb)*64 + l)*8 + e.
__host__ inline void pack_w2(const float* w, __bf16* out) {
  for (int kb = 0; kb < 4; ++kb)
    for (int nb = 0; nb < 2; ++nb)
      for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e) {
          int n = nb * 32 + l % 32, k = kb * 16 + 8 * (l / 32) + e;
          out[((kb * 2 + nb) * 64 + l) * 8 + e] = (__bf16)w[OW2 + n * H + k];
        }
}

// Forward of the 64 cells of a wavefront (one per lane, features x).  Must be
// reached by all 64 lanes together (uniform control flow): lanes without a
// cell pass any finite features and ignore the result.  l1(o): unit o of the
// first layer as (b1, W1[o][0..2]); w2: the packed operand of pack_w2 at an index;
// l2(q), l3(q): b2 and w3 of units 4q .. 4q + 3.
// The hidden layer is formed transposed, D = W2 H1^T with the cells along the
// columns: a lane then computes just the first-layer units its B operands
// need (those of cells l%32 and 32 + l%32) and holds 16 units of a cell's
// column, so the output layer is summed inside the lane but for one exchange
// of lane halves per four values.  With the cells along the rows it took 160
// exchanges and an H1 tile in LDS whose rows all began in one bank: 2^20
// cells took 78 us that way.  The sum over units is the balanced tree
// over bits 4, 3, 2, 1, 0 of the unit (blocks 0 and 32 added first).
template <class L1, class W2, class L2, class L3>
__device__ float forward_wave(const float* x, L1&& l1, W2&& w2, L2&& l2, L3&& l3, float b3) {
  int l = threadIdx.x & 63, hf = l >> 5;
  float xo[3], y = 0.f;                             // features of the cell the other half's lane holds
  for (int k = 0; k < 3; ++k) xo[k] = __shfl_xor(x[k], 32, 64);
#pragma unroll 1
  for (int sb = 0; sb < 2; ++sb) {                 // cells 32 sb + l%32, one block at a time: 32 accumulators, not 64
    int at = hf;                                   // opaque: keeps the weights of both blocks' loads in the loop
    asm volatile("" : "+v"(at));
    float xc[3];
    for (int k = 0; k < 3; ++k) xc[k] = sb == hf ? x[k] : xo[k];
    floatx16 acc[2] = {floatx16{}, floatx16{}};    // units 32 nb ..
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      bf16x8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float4 u = l1(kb * 16 + 8 * at + e);
        float a = u.x + u.y * xc[0] + u.z * xc[1] + u.w * xc[2];
        h[e] = (__bf16)fmaxf(a, 0.f);
      }
      for (int nb = 0; nb < 2; ++nb)
        acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w2((kb * 2 + nb) * 64 + l), h, acc[nb], 0, 0, 0);
    }
    float part[16];                                // unit 8 (r/4) + 4 hf + r%4
    for (int r = 0; r < 16; ++r) part[r] = 0.f;
    for (int nb = 0; nb < 2; ++nb)
      for (int q = 0; q < 4; ++q) {
        float4 b = l2(nb * 8 + 2 * q + at), u = l3(nb * 8 + 2 * q + at);
        float b2[4] = {b.x, b.y, b.z, b.w}, w3[4] = {u.x, u.y, u.z, u.w};
        for (int r = 0; r < 4; ++r) {
          float v = acc[nb][4 * q + r] + b2[r];
          part[4 * q + r] += w3[r] * fmaxf(v, 0.f);
        }
      }
    for (int r = 0; r < 8; ++r) part[r] += part[r + 8];
    for (int r = 0; r < 4; ++r) part[r] += part[r + 4];
    for (int r = 0; r < 4; ++r) part[r] += __shfl_xor(part[r], 32, 64);
    float ys = (part[0] + part[2]) + (part[1] + part[3]);
    if (sb == hf) y = ys;
  }
  return y + b3;
}

}  // namespace mlp
}  // namespace gh
#endif
