// Learned band-CG preconditioner: a 4 -> 64 -> 64 -> 64 -> 1 SiLU network
// with bfloat16 weights and FP32 accumulation that maps per-(band, plane
// wave) features to a preconditioner scale, trained on the device.
//
// There is no reference counterpart (the reference's band CG uses the TPA
// preconditioner only, src/eigensolver/uspp_preconditioner.rs:148-180);
// the network's output o modulates that same polynomial:
//   f = [kin_g / E_b, log E_b, V_mean, V_std],  s = t(kin_g / E_b) e^o / E_b,
// with E_b the band's kinetic energy and V the bound local potential, so an
// untrained (zero-output) network is the per-band TPA preconditioner.
// Training pairs come per band (residual r and correction e over the band's
// plane waves). The loss is the band-mean misalignment of the
// preconditioned residual with the correction,
//   L = (1/n_bands) sum_b [1 - (sum_g s_g a_g)^2 / (sum_g s_g^2 c_g sum_g |e_g|^2)],
//   a = -Re(conj(r) e), c = |r|^2,
// which is scale-free per band as band CG's line search is (one
// preconditioned step along s r leaves an error of relative size L_b);
// minimised by Adam on FP32 master weights, the forward pass always with
// the bfloat16-rounded weights.
//
// Kernels: k_mlp_pass<0> (forward over band-aligned 16-sample tiles, per-tile
// sums), k_mlp_band_sums, k_mlp_pass<1> (forward + backward with
// the band coefficients, per-block gradient partials), k_mlp_reduce
// (fixed-order sums), k_mlp_adam, k_mlp_table (one thread per (band, plane
// wave) inference), and the training-pair builder.
#include <algorithm>
#include <cmath>
#include <vector>

#include "blas1.hpp"
#include "impl.hpp"
#include "linalg.hpp"
#include "ops.hpp"

struct chs_mlp {
  chs::DevBuf theta, m, v, grad, wbf, part, tsum, bcoef;
  int t = 0;
};

namespace chs {

constexpr int kH = 64, kIn = 4;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH,
              oW3 = oB2 + kH, oB3 = oW3 + kH * kH, oW4 = oB3 + kH, oB4 = oW4 + kH,
              kNP = oB4 + 1;  // 8705
static_assert(kNP == CHS_MLP_PARAMS, "parameter count");
constexpr int kWP = kH + 1;    // padded row stride of W2, W3 in LDS (k_mlp_table)

__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned int u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float((unsigned int)b << 16); }
__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float tpa_t(float x) {
  const float x2 = x * x, num = 27.0f + 18.0f * x + 12.0f * x2 + 8.0f * x2 * x;
  return num / (num + 16.0f * x2 * x2);
}

// bfloat16 weights -> FP32 in LDS: W1 [64][4], W2 / W3 [64][65] (row = output)
struct MlpLds {
  float w1[kH * kIn], b1[kH], w2[kH * kWP], b2[kH], w3[kH * kWP], b3[kH], w4[kH], b4;
};
__device__ void load_weights(MlpLds& L, const unsigned short* __restrict__ wbf) {
  for (int t = threadIdx.x; t < kNP; t += blockDim.x) {
    const float v = bf2f(wbf[t]);
    if (t < oB1) L.w1[t] = v;
    else if (t < oW2) L.b1[t - oB1] = v;
    else if (t < oB2) { const int q = t - oW2; L.w2[(q / kH) * kWP + q % kH] = v; }
    else if (t < oW3) L.b2[t - oB2] = v;
    else if (t < oB3) { const int q = t - oW3; L.w3[(q / kH) * kWP + q % kH] = v; }
    else if (t < oW4) L.b3[t - oB3] = v;
    else if (t < oB4) L.w4[t - oW4] = v;
    else L.b4 = v;
  }
}

__global__ void k_mlp_to_bf16(const float* __restrict__ theta, unsigned short* __restrict__ wbf) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kNP) wbf[t] = f2bf(theta[t]);
}

// Sample j of a batch: i = (off + j * stride) mod n.
__device__ __forceinline__ long long batch_index(long long j, long long off, long long stride,
                                                 long long n) {
  return (long long)(((unsigned long long)off + (unsigned long long)j * (unsigned long long)stride) %
                     (unsigned long long)n);
}

// ---------------------------------------------------------------------------
// Forward (+ backward) over band-aligned 16-sample tiles, one wavefront per
// tile and no workgroup barrier inside the tile loop. Every 64 x 64 product
// is FP32 matrix-core work (v_mfma_f32_16x16x4_f32: lane l = 16 q + i supplies
// A[i][q] and B[q][i], and holds D[4 q + v][i]):
//  - activations: lane (q, i) holds sample i's units 16 m + 4 q + v (m, v < 4).
//    With the K order (m, v) -> unit 16 m + 4 q + v that is exactly the next
//    layer's B operand, so a layer hands its result on in registers; the
//    weights are laid out in LDS as those A fragments (one conflict-free
//    ds_read_b128 per four k-steps), in both orientations for PASS 1;
//  - weight gradients contract over the 16 samples: D and the layer's input
//    pass through the wavefront's LDS tile [sample][unit] to get samples into
//    K; a wavefront accumulates its tiles in registers (144 for W3, W2 and
//    [W1 | b1]).
// The 192 activations of a sample are evaluated once per pass. Bound: the
// FP32 matrix rate (16.9 kflop per sample in PASS 0, 51 in PASS 1) and the
// exponentials, which run on the vector unit between the products. Measured
// at 1.53e6 samples: PASS 0 3.77 -> 0.41 ms, PASS 1 7.85 -> 1.10 ms; the former
// kernel ran on the vector unit with each activation evaluated by 8 or 16
// threads inside the product loops, and five barriers per product.
// ---------------------------------------------------------------------------
using f32x4 = __attribute__((ext_vector_type(4))) float;
constexpr int kTS = 16;         // samples per tile
constexpr int kTP = 80;         // floats per row of the transposition tile
constexpr int kMlpWaves = 4;    // wavefronts per workgroup
constexpr int kMlpBlocks0 = 1024, kMlpBlocks1 = 256;  // 4 (PASS 0) or 1 wavefront per SIMD

// h = silu(z), ds = silu'(z) from one sigmoid: 1 / (1 + e^-z) as the hardware
// reciprocal with one Newton step, and z / (1 + e^-z) from it with a residual
// step (both round as the division does; without the second step the loss and
// gradient errors double). Below z = -69, where both are under 1e-28, z is taken
// as -69, so that the sum stays finite and the steps have no inf * 0 (the maximum
// hands a NaN on).
__device__ __forceinline__ void silu2(float z, float& h, float& ds) {
  z = __builtin_elementwise_maximum(z, -69.0f);
  const float d = 1.0f + expf(-z);
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  h = z * r;
  h = fmaf(fmaf(-d, h, z), r, h);
  ds = fmaf(h, 1.0f - r, r);
}

// Fragment of a 64 x 64 matrix M for the A operand: entry (mo, mi, lane, v) =
// M[16 mo + i][16 mi + 4 q + v], M = W (forward) or W^T (backward).
__device__ __forceinline__ void load_fragments(float* __restrict__ f,
                                               const unsigned short* __restrict__ w, bool transpose) {
  for (int t = threadIdx.x; t < kH * kH; t += blockDim.x) {
    const int v = t & 3, lane = (t >> 2) & 63, mi = (t >> 8) & 3, mo = t >> 10;
    const int r = 16 * mo + (lane & 15), c = 16 * mi + 4 * (lane >> 4) + v;
    f[t] = bf2f(transpose ? w[c * kH + r] : w[r * kH + c]);
  }
}

// out = M h (+ bias): 64 independent-accumulator MFMAs.
__device__ __forceinline__ void mlp_product(const f32x4* __restrict__ frag, int lane,
                                            const float (&h)[4][4], f32x4 (&acc)[4]) {
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    f32x4 a[4];
#pragma unroll
    for (int mo = 0; mo < 4; ++mo) a[mo] = frag[(mo * 4 + mi) * 64 + lane];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int mo = 0; mo < 4; ++mo)
        acc[mo] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mo][v], h[mi][v], acc[mo], 0, 0, 0);
  }
}

// Per-wavefront orderings of its own LDS tile.
__device__ __forceinline__ void mlp_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Batch: nbb whole bands; batch band j is band (off + j stride) mod NB of
// the pair arrays (band length Lb); tile tt = (j, q0) covers samples q0 ..
// q0 + 15 of band j. PASS 0 writes per-tile sums {sum s a, sum s^2 c,
// sum |e|^2} to tsum; PASS 1 back-propagates dL/do = g1 (g2 s c - a) s with
// the band coefficients bcoef[j] = {g1, g2} and leaves the block's gradient
// partial in part[blockIdx.x][kNP].
template <int PASS>
__global__ void __launch_bounds__(64 * kMlpWaves)
__attribute__((amdgpu_waves_per_eu(PASS == 0 ? 4 : 1)))
k_mlp_pass(const unsigned short* __restrict__ wbf, const float* __restrict__ feat,
           const float* __restrict__ rr, const float* __restrict__ ee, const float* __restrict__ ww,
           long long NB, int Lb, int nbb, long long off, long long stride,
           double* __restrict__ tsum, const double* __restrict__ bcoef, float* __restrict__ part) {
  constexpr int FW = kH * kH;
  // weight fragments (after the tile loop of PASS 1: the block's gradient sum)
  __shared__ __attribute__((aligned(16))) float frag[PASS ? 4 * FW : 2 * FW];
  __shared__ __attribute__((aligned(16))) float bias[3][kH];
  __shared__ __attribute__((aligned(16))) float w4s[kH];
  __shared__ __attribute__((aligned(16))) float tile_mem[PASS ? kMlpWaves * 2 * kTS * kTP : 1];
  static_assert(4 * FW >= kNP, "the gradient sum reuses the fragments");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, i = lane & 15;
  load_fragments(frag, wbf + oW2, false);
  load_fragments(frag + FW, wbf + oW3, false);
  if (PASS) {
    load_fragments(frag + 2 * FW, wbf + oW2, true);
    load_fragments(frag + 3 * FW, wbf + oW3, true);
  }
  if (threadIdx.x < kH) {
    bias[0][threadIdx.x] = bf2f(wbf[oB1 + threadIdx.x]);
    bias[1][threadIdx.x] = bf2f(wbf[oB2 + threadIdx.x]);
    bias[2][threadIdx.x] = bf2f(wbf[oB3 + threadIdx.x]);
    w4s[threadIdx.x] = bf2f(wbf[oW4 + threadIdx.x]);
  }
  const float b4 = bf2f(wbf[oB4]);
  float w1a[4];  // layer 1's A operand: W1[16 m + i][q]
#pragma unroll
  for (int m = 0; m < 4; ++m) w1a[m] = bf2f(wbf[oW1 + (16 * m + i) * kIn + q]);
  __syncthreads();
  const f32x4* f2 = reinterpret_cast<const f32x4*>(frag);
  const f32x4* f3 = f2 + FW / 4;
  const f32x4* t2 = f2 + 2 * (FW / 4);
  const f32x4* t3 = f2 + 3 * (FW / 4);
  auto bias4 = [&](const float* b, int m) {
    return *reinterpret_cast<const f32x4*>(b + 16 * m + 4 * q);
  };
  // PASS 1 accumulators: G[j][i] tiles of W3 and W2; [W1 | b1] in columns 0-4
  f32x4 g3[4][4], g2[4][4], g1[4];
  float gw4[4][4], gb3[4][4], gb2[4][4], gb4 = 0.0f;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    g1[m] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      g3[m][p] = g2[m][p] = f32x4{0, 0, 0, 0};
      gw4[m][p] = gb3[m][p] = gb2[m][p] = 0.0f;
    }
  }
  const int tpb = (Lb + kTS - 1) / kTS;
  const long long tiles = (long long)nbb * tpb;
  float* dt = tile_mem + (PASS ? w * 2 * kTS * kTP : 0);  // D as [sample][unit]
  float* ht = dt + (PASS ? kTS * kTP : 0);                // the layer's input likewise
  auto to_tile = [&](float* t, const float (&x)[4][4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      *reinterpret_cast<f32x4*>(t + i * kTP + 16 * m + 4 * q) =
          f32x4{x[m][0], x[m][1], x[m][2], x[m][3]};
  };
  // G[mt][nt] += D H^T over the tile's 16 samples
  auto wgrad = [&](f32x4 (&g)[4][4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float a[4], b[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        a[m] = dt[(4 * t + q) * kTP + 16 * m + i];
        b[m] = ht[(4 * t + q) * kTP + 16 * m + i];
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int p = 0; p < 4; ++p)
          g[m][p] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], b[p], g[m][p], 0, 0, 0);
    }
  };
  for (long long tile = (long long)blockIdx.x * kMlpWaves + w; tile < tiles;
       tile += (long long)gridDim.x * kMlpWaves) {
    // keeps the fragments in LDS: hoisted out of the loop they would take 128
    // registers per matrix pair and spill
    asm volatile("" ::: "memory");
    const int jb = (int)(tile / tpb), q0 = (int)(tile - (long long)jb * tpb) * kTS;
    const long long base = batch_index(jb, off, stride, NB) * Lb;  // first pair of the band
    const bool in = q0 + i < Lb;
    const long long sidx = base + q0 + i;
    const float fq = in ? feat[sidx * kIn + q] : 0.0f;  // feature q of sample i
    float h1[4][4], h2[4][4], h3[4][4], d1[4][4], d2[4][4], d3[4][4];
    auto activate = [&](const f32x4 (&z)[4], float (&h)[4][4], float (&d)[4][4]) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) silu2(z[m][v], h[m][v], d[m][v]);
    };
    f32x4 z[4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
      z[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1a[m], fq, bias4(bias[0], m), 0, 0, 0);
    activate(z, h1, d1);
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] = bias4(bias[1], m);
    mlp_product(f2, lane, h1, z);
    activate(z, h2, d2);
#pragma unroll
    for (int m = 0; m < 4; ++m) z[m] = bias4(bias[2], m);
    mlp_product(f3, lane, h2, z);
    activate(z, h3, d3);
    // output: each lane its 16 units, then the four lanes of the sample
    float o = 0.0f;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 w4v = bias4(w4s, m);
#pragma unroll
      for (int v = 0; v < 4; ++v) o = fmaf(w4v[v], h3[m][v], o);
    }
    o += __shfl_xor(o, 16);
    o += __shfl_xor(o, 32);
    o += b4;
    const float x = __shfl(fq, i), leb = __shfl(fq, 16 + i);
    float dO = 0.0f;
    double sa = 0.0, sc = 0.0, se = 0.0;
    if (in && ww[sidx] > 0.0f) {
      const float s = tpa_t(x) * expf(o) / expf(leb);
      const float r0 = rr[2 * sidx], r1 = rr[2 * sidx + 1];
      const float e0 = ee[2 * sidx], e1 = ee[2 * sidx + 1];
      const float a = -(r0 * e0 + r1 * e1), c = r0 * r0 + r1 * r1;
      if (PASS == 0) {
        sa = (double)s * a;
        sc = (double)s * s * c;
        se = (double)e0 * e0 + (double)e1 * e1;
      } else {
        const float c1 = (float)bcoef[2 * jb], c2 = (float)bcoef[2 * jb + 1];
        dO = c1 * (c2 * s * c - a) * s;
      }
    }
    if (PASS == 0) {
#pragma unroll
      for (int k = 8; k > 0; k >>= 1) {  // the 16 samples (every q holds them)
        sa += __shfl_xor(sa, k);
        sc += __shfl_xor(sc, k);
        se += __shfl_xor(se, k);
      }
      if (lane == 0) {
        tsum[3 * tile] = sa;
        tsum[3 * tile + 1] = sc;
        tsum[3 * tile + 2] = se;
      }
      continue;
    }
    gb4 += dO;
    // dZ3 = dO w4 silu'(Z3), then back through W3 and W2
    float dz[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 w4v = bias4(w4s, m);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        gw4[m][v] = fmaf(dO, h3[m][v], gw4[m][v]);
        dz[m][v] = dO * w4v[v] * d3[m][v];
        gb3[m][v] += dz[m][v];
      }
    }
    auto back = [&](const f32x4* fr, const float (&d)[4][4]) {
      f32x4 acc[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m] = f32x4{0, 0, 0, 0};
      mlp_product(fr, lane, dz, acc);
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) dz[m][v] = acc[m][v] * d[m][v];
    };
    to_tile(dt, dz);
    to_tile(ht, h2);
    mlp_wave_sync();
    wgrad(g3);
    back(t3, d2);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) gb2[m][v] += dz[m][v];
    mlp_wave_sync();  // the tile's reads precede its next contents
    to_tile(dt, dz);
    to_tile(ht, h1);
    mlp_wave_sync();
    wgrad(g2);
    back(t2, d1);
    mlp_wave_sync();
    to_tile(dt, dz);
    ht[i * kTP + q] = fq;
    mlp_wave_sync();
    // [W1 | b1]: features in columns 0-3, ones in column 4
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float fv = ht[(4 * t + q) * kTP + (i & 3)];
      const float b = i < kIn ? fv : (i == kIn ? 1.0f : 0.0f);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        g1[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(dt[(4 * t + q) * kTP + 16 * m + i], b, g1[m],
                                                     0, 0, 0);
    }
    mlp_wave_sync();
  }
  if (PASS == 0) return;
  // sums over the 16 samples of the per-lane vectors
#pragma unroll
  for (int k = 1; k < 16; k <<= 1) {
    gb4 += __shfl_xor(gb4, k);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        gw4[m][v] += __shfl_xor(gw4[m][v], k);
        gb3[m][v] += __shfl_xor(gb3[m][v], k);
        gb2[m][v] += __shfl_xor(gb2[m][v], k);
      }
  }
  // the wavefronts add their sums in order into LDS, in the parameter layout
  for (int ww2 = 0; ww2 < kMlpWaves; ++ww2) {
    __syncthreads();
    if (w == ww2) {
      auto put = [&](int p, float val) { frag[p] = ww2 == 0 ? val : frag[p] + val; };
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int j = 16 * m + 4 * q + v;
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            put(oW3 + j * kH + 16 * p + i, g3[m][p][v]);
            put(oW2 + j * kH + 16 * p + i, g2[m][p][v]);
          }
          if (i < kIn) put(oW1 + j * kIn + i, g1[m][v]);
          if (i == kIn) put(oB1 + j, g1[m][v]);
          if (i == 0) {
            put(oB2 + j, gb2[m][v]);
            put(oB3 + j, gb3[m][v]);
            put(oW4 + j, gw4[m][v]);
          }
        }
      if (lane == 0) put(oB4, gb4);
    }
  }
  __syncthreads();
  float* pb = part + (size_t)blockIdx.x * kNP;
  for (int p = threadIdx.x; p < kNP; p += blockDim.x) pb[p] = frag[p];
}

// Per batch band, one wavefront: A, B, E from its tiles (lanes over strided
// tiles, fixed-order shuffle sum); L_b = 1 - A^2/(B E) for used bands (B, E >
// 0), 0 otherwise; bcoef = {2A/(B E) / nbb, A/B}; lossv[j] = L_b / nbb.
__global__ void __launch_bounds__(64) k_mlp_band_sums(const double* __restrict__ tsum, int nbb,
                                                      int tpb, double* __restrict__ bcoef,
                                                      double* __restrict__ lossv) {
  for (int j = blockIdx.x; j < nbb; j += gridDim.x) {
    double A = 0, B = 0, E = 0;
    for (int t = threadIdx.x; t < tpb; t += 64) {
      const double* p = tsum + 3 * ((size_t)j * tpb + t);
      A += p[0];
      B += p[1];
      E += p[2];
    }
    for (int k = 32; k > 0; k >>= 1) {
      A += __shfl_xor(A, k);
      B += __shfl_xor(B, k);
      E += __shfl_xor(E, k);
    }
    if (threadIdx.x != 0) continue;
    const bool used = B > 0.0 && E > 0.0;
    bcoef[2 * j] = used ? 2.0 * A / (B * E) / nbb : 0.0;
    bcoef[2 * j + 1] = used ? A / B : 0.0;
    lossv[j] = used ? (1.0 - A * A / (B * E)) / nbb : 0.0;
  }
}

// Gradient from the block partials, 16 parameters per workgroup with 16
// threads over the blocks of each (a serial sum per parameter took 0.13 ms);
// the last workgroup adds up the loss. FP64 sums in a fixed order.
__global__ void __launch_bounds__(256) k_mlp_reduce(const float* __restrict__ part, int nblk,
                                                    const double* __restrict__ lossv, int nl,
                                                    float* __restrict__ grad,
                                                    double* __restrict__ loss) {
  __shared__ double sh[16][17];
  const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
  const int p = blockIdx.x * 16 + c;
  double s = 0.0;
  if (p < kNP)
    for (int b = r; b < nblk; b += 16) s += part[(size_t)b * kNP + p];
  sh[r][c] = s;
  __syncthreads();
  if (threadIdx.x < 16 && p < kNP) {
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += sh[k][c];
    grad[p] = (float)t;
  }
  if (blockIdx.x == gridDim.x - 1) {
    __syncthreads();
    double l = 0.0;
    for (int b = threadIdx.x; b < nl; b += 256) l += lossv[b];
    for (int k = 32; k > 0; k >>= 1) l += __shfl_xor(l, k);
    if ((threadIdx.x & 63) == 0) sh[0][threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) *loss = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
  }
}

__global__ void k_mlp_adam(float* __restrict__ theta, float* __restrict__ m, float* __restrict__ v,
                           const float* __restrict__ g, float lr, float bc1, float bc2,
                           unsigned short* __restrict__ wbf) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kNP) return;
  const float gp = g[p];
  const float mp = 0.9f * m[p] + 0.1f * gp;
  const float vp = 0.999f * v[p] + 0.001f * gp * gp;
  m[p] = mp;
  v[p] = vp;
  const float th = theta[p] - lr * (mp / bc1) / (sqrtf(vp / bc2) + 1e-8f);
  theta[p] = th;
  wbf[p] = f2bf(th);
}

// E_b = sum_g kin_g |psi_bg|^2 / sum_g |psi_bg|^2, one block per band.
__global__ void __launch_bounds__(256) k_band_ekin(const z64* __restrict__ psi,
                                                   const double* __restrict__ kin, int n_pw,
                                                   double* __restrict__ ekin) {
  __shared__ double sh[8];
  const z64* pb = psi + (size_t)blockIdx.x * n_pw;
  double a = 0.0, b = 0.0;
  for (int g = threadIdx.x; g < n_pw; g += blockDim.x) {
    const double w = norm2(pb[g]);
    a += kin[g] * w;
    b += w;
  }
  const double sa = block_sum(a, sh);
  const double sb = block_sum(b, sh);
  if (threadIdx.x == 0) ekin[blockIdx.x] = sb > 0.0 ? sa / sb : 0.0;
}

// mean and standard deviation of the bound local potential (one block)
__global__ void __launch_bounds__(256) k_grid_stats(const double* __restrict__ v, size_t n3,
                                                    double* __restrict__ out) {
  __shared__ double sh[8];
  double a = 0.0, b = 0.0;
  for (size_t i = threadIdx.x; i < n3; i += blockDim.x) {
    a += v[i];
    b += v[i] * v[i];
  }
  const double sa = block_sum(a, sh);
  const double sb = block_sum(b, sh);
  if (threadIdx.x == 0) {
    const double mean = sa / (double)n3;
    out[0] = mean;
    out[1] = sqrt(fmax(sb / (double)n3 - mean * mean, 0.0));
  }
}

// One thread per (band, plane wave): scale table for band CG.
__global__ void __launch_bounds__(256) k_mlp_table(const unsigned short* __restrict__ wbf,
                                                   const double* __restrict__ kin,
                                                   const double* __restrict__ ekin,
                                                   const double* __restrict__ vstat, int n_pw,
                                                   float* __restrict__ table) {
  __shared__ MlpLds L;
  load_weights(L, wbf);
  __syncthreads();
  const int b = blockIdx.y;
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_pw) return;
  const float eb = (float)ekin[b];
  const float f[4] = {(float)(kin[g] / ekin[b]), logf(eb), (float)vstat[0], (float)vstat[1]};
  float h1[kH], h2[kH];
#pragma unroll
  for (int j = 0; j < kH; ++j) {
    float a = L.b1[j];
#pragma unroll
    for (int i = 0; i < kIn; ++i) a = fmaf(L.w1[j * kIn + i], f[i], a);
    h1[j] = silu(a);
  }
#pragma unroll 4
  for (int j = 0; j < kH; ++j) {
    float a = L.b2[j];
#pragma unroll
    for (int i = 0; i < kH; ++i) a = fmaf(L.w2[j * kWP + i], h1[i], a);
    h2[j] = silu(a);
  }
  float o = L.b4;
#pragma unroll 4
  for (int j = 0; j < kH; ++j) {
    float a = L.b3[j];
#pragma unroll
    for (int i = 0; i < kH; ++i) a = fmaf(L.w3[j * kWP + i], h2[i], a);
    o = fmaf(L.w4[j], silu(a), o);
  }
  table[(size_t)b * n_pw + g] = tpa_t(f[0]) * expf(o) / eb;
}

// ---- training pairs -------------------------------------------------------
// Per band b of a block psi (not yet converged) and the converged block
// psi_ref: psi^ = psi / sqrt(<psi|S|psi>), r = (H - eps S) psi^ with
// eps = <psi^|H|psi^>, e = phase-aligned psi_ref_b - psi^ with its
// psi^ component removed. dots[b] slots: 0 <psi|S psi>, 1 <psi|H psi>,
// 2 <psi_ref|S psi>, 3 <S psi^ | e>, 4 |e|^2.
__global__ void __launch_bounds__(256) k_pair_dots(const z64* __restrict__ x, const z64* __restrict__ y,
                                                   int n_pw, z64* __restrict__ out, int slot) {
  __shared__ double sh[8];
  const z64* xb = x + (size_t)blockIdx.x * n_pw;
  const z64* yb = y + (size_t)blockIdx.x * n_pw;
  double re = 0, im = 0;
  for (int g = threadIdx.x; g < n_pw; g += blockDim.x) {
    const z64 c = cmulc(xb[g], yb[g]);
    re += c.x;
    im += c.y;
  }
  const double a = block_sum(re, sh);
  const double b = block_sum(im, sh);
  if (threadIdx.x == 0) out[(size_t)blockIdx.x * 8 + slot] = mk(a, b);
}

// r = (hp - eps sp) / sqrt(n) ; e = t - psi^ with t (in e) the normalised
// projection of psi^ on the reference eigenspace of the band
__global__ void k_pair_build(const z64* __restrict__ psi, const z64* __restrict__ hp,
                             const z64* __restrict__ sp, int n_pw, const z64* __restrict__ dots,
                             z64* __restrict__ r, z64* __restrict__ e) {
  const int b = blockIdx.y, g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_pw) return;
  const z64* d = dots + (size_t)b * 8;
  const double nn = d[0].x, inv = 1.0 / sqrt(nn), eps = d[1].x / nn;
  const size_t i = (size_t)b * n_pw + g;
  const z64 p = psi[i], h = hp[i], s = sp[i];
  r[i] = mk((h.x - eps * s.x) * inv, (h.y - eps * s.y) * inv);
  e[i] = e[i] - mk(p.x * inv, p.y * inv);
}

// e -= psi^ <S psi^|e>, then the f32 pair arrays and features
__global__ void k_pair_emit(const z64* __restrict__ psi, const z64* __restrict__ r,
                            const z64* __restrict__ e, const double* __restrict__ kin,
                            const double* __restrict__ ekin, const double* __restrict__ vstat,
                            const double* __restrict__ wband, int n_pw,
                            const z64* __restrict__ dots, float* __restrict__ feat,
                            float* __restrict__ rf, float* __restrict__ ef, float* __restrict__ wf) {
  const int b = blockIdx.y, g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_pw) return;
  const z64* d = dots + (size_t)b * 8;
  // psi^ <S psi^|e> = psi <S psi|e> / <psi|S psi>
  const double inv2 = 1.0 / d[0].x;
  const z64 proj = d[3];
  const size_t i = (size_t)b * n_pw + g;
  const z64 p = psi[i];
  const z64 ev = e[i] - mk(inv2 * (p.x * proj.x - p.y * proj.y), inv2 * (p.x * proj.y + p.y * proj.x));
  const z64 rv = r[i];
  rf[2 * i] = (float)rv.x;
  rf[2 * i + 1] = (float)rv.y;
  ef[2 * i] = (float)ev.x;
  ef[2 * i + 1] = (float)ev.y;
  wf[i] = (float)wband[b];
  feat[4 * i] = (float)(kin[g] / ekin[b]);
  feat[4 * i + 1] = (float)log(ekin[b]);
  feat[4 * i + 2] = (float)vstat[0];
  feat[4 * i + 3] = (float)vstat[1];
}

__global__ void k_sub_scaled(const z64* __restrict__ e, const z64* __restrict__ psi, int n_pw,
                             const z64* __restrict__ dots, z64* __restrict__ out) {
  const int b = blockIdx.y, g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n_pw) return;
  const z64* d = dots + (size_t)b * 8;
  const double inv2 = 1.0 / d[0].x;
  const z64 proj = d[3];
  const size_t i = (size_t)b * n_pw + g;
  const z64 p = psi[i];
  out[i] = e[i] - mk(inv2 * (p.x * proj.x - p.y * proj.y), inv2 * (p.x * proj.y + p.y * proj.x));
}

static int mlp_stats(chs_context* ctx, const z64* psi, int n_b, double** ekin, double** vstat) {
  Hamiltonian& H = ctx->impl->ham;
  auto* im = ctx->impl;
  CHS_TRY(ensure(ctx, im->small, 64 * sizeof(double)));
  CHS_TRY(ensure(ctx, im->mlp_ws, (size_t)n_b * sizeof(double) * 2 + 256));
  *ekin = (double*)im->mlp_ws.p;
  *vstat = (double*)im->small.p + 40;
  hipLaunchKernelGGL(k_band_ekin, dim3(n_b), dim3(256), 0, ctx->stream, psi, H.kin, H.n_pw, *ekin);
  const size_t n3 = (size_t)H.n_grid * H.n_grid * H.n_grid;
  hipLaunchKernelGGL(k_grid_stats, dim3(1), dim3(256), 0, ctx->stream, H.veff, n3, *vstat);
  CHS_LAUNCH_CHECK(ctx);
  return CHS_OK;
}

static int mlp_batch(chs_context* ctx, chs_mlp* m, const float* feat, const float* r,
                     const float* e, const float* w, long long NB, int Lb, int nbb, long long off,
                     long long stride, double* d_loss) {
  const int tpb = (Lb + kTS - 1) / kTS;
  const long long tiles = (long long)nbb * tpb;
  CHS_TRY(ensure(ctx, m->part, (size_t)kMlpBlocks1 * kNP * sizeof(float)));
  CHS_TRY(ensure(ctx, m->tsum, (size_t)tiles * 3 * sizeof(double)));
  CHS_TRY(ensure(ctx, m->bcoef, (size_t)nbb * 3 * sizeof(double)));
  double* bcoef = (double*)m->bcoef.p;
  double* lossv = bcoef + 2 * (size_t)nbb;
  const long long want = (tiles + kMlpWaves - 1) / kMlpWaves;
  const int nblk0 = (int)std::min<long long>(kMlpBlocks0, want);
  const int nblk1 = (int)std::min<long long>(kMlpBlocks1, want);
  const unsigned short* wbf = (const unsigned short*)m->wbf.p;
  hipLaunchKernelGGL(k_mlp_pass<0>, dim3(nblk0), dim3(64 * kMlpWaves), 0, ctx->stream, wbf, feat, r,
                     e, w, NB, Lb, nbb, off, stride, (double*)m->tsum.p, (const double*)nullptr,
                     (float*)nullptr);
  hipLaunchKernelGGL(k_mlp_band_sums, dim3(std::min(nbb, 1 << 20)), dim3(64), 0, ctx->stream,
                     (const double*)m->tsum.p, nbb, tpb, bcoef, lossv);
  hipLaunchKernelGGL(k_mlp_pass<1>, dim3(nblk1), dim3(64 * kMlpWaves), 0, ctx->stream, wbf, feat, r,
                     e, w, NB, Lb, nbb, off, stride, (double*)nullptr, (const double*)bcoef,
                     (float*)m->part.p);
  hipLaunchKernelGGL(k_mlp_reduce, dim3(ceil_div(kNP, 16)), dim3(256), 0, ctx->stream,
                     (const float*)m->part.p, nblk1, (const double*)lossv, nbb, (float*)m->grad.p,
                     d_loss);
  CHS_LAUNCH_CHECK(ctx);
  return CHS_OK;
}

static long long coprime_stride(long long n) {
  long long s = 1000003;
  auto gcd = [](long long a, long long b) {
    while (b) {
      const long long t = a % b;
      a = b;
      b = t;
    }
    return a;
  };
  while (gcd(s, n) != 1) s += 2;
  return s % n == 0 ? 1 : s % n;
}

}  // namespace chs

using namespace chs;

extern "C" {

int chs_mlp_create(chs_context* ctx, uint64_t seed, chs_mlp** out) {
  if (!ctx || !out) return CHS_ERR_INVALID_ARG;
  *out = nullptr;
  // Glorot-uniform W1..W3 from the 48-bit LCG; biases, w4, b4 zero
  std::vector<float> th(kNP, 0.0f);
  uint64_t s = seed & 0xFFFFFFFFFFFFull;
  auto uni = [&s]() {
    s = (s * 25214903917ull + 11ull) & 0xFFFFFFFFFFFFull;
    return (double)s / 281474976710656.0;
  };
  const struct { int off, fo, fi; } layers[3] = {{oW1, kH, kIn}, {oW2, kH, kH}, {oW3, kH, kH}};
  for (const auto& l : layers) {
    const double lim = std::sqrt(6.0 / (l.fo + l.fi));
    for (int k = 0; k < l.fo * l.fi; ++k) th[l.off + k] = (float)((2.0 * uni() - 1.0) * lim);
  }
  auto* m = new chs_mlp;
  int rc = chs_mlp_set_params(ctx, m, th.data());
  if (rc != CHS_OK) {
    chs_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return CHS_OK;
}

int chs_mlp_destroy(chs_mlp* m) {
  if (!m) return CHS_ERR_INVALID_ARG;
  for (DevBuf* b : {&m->theta, &m->m, &m->v, &m->grad, &m->wbf, &m->part, &m->tsum, &m->bcoef})
    release(*b);
  delete m;
  return CHS_OK;
}

int chs_mlp_set_params(chs_context* ctx, chs_mlp* m, const float* theta) {
  if (!ctx || !m || !theta) return CHS_ERR_INVALID_ARG;
  for (DevBuf* b : {&m->theta, &m->m, &m->v, &m->grad})
    CHS_TRY(ensure(ctx, *b, kNP * sizeof(float)));
  CHS_TRY(ensure(ctx, m->wbf, kNP * sizeof(unsigned short)));
  CHS_HIP(ctx, hipMemcpyAsync(m->theta.p, theta, kNP * sizeof(float), hipMemcpyHostToDevice,
                              ctx->stream));
  ctx->h2d += kNP * sizeof(float);
  CHS_HIP(ctx, hipMemsetAsync(m->m.p, 0, kNP * sizeof(float), ctx->stream));
  CHS_HIP(ctx, hipMemsetAsync(m->v.p, 0, kNP * sizeof(float), ctx->stream));
  hipLaunchKernelGGL(k_mlp_to_bf16, dim3(ceil_div(kNP, 256)), dim3(256), 0, ctx->stream,
                     (const float*)m->theta.p, (unsigned short*)m->wbf.p);
  CHS_LAUNCH_CHECK(ctx);
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  ctx->h2d += kNP * sizeof(float);
  m->t = 0;
  return CHS_OK;
}

int chs_mlp_get_params(chs_context* ctx, chs_mlp* m, float* theta) {
  if (!ctx || !m || !theta || !m->theta.p) return CHS_ERR_INVALID_ARG;
  CHS_HIP(ctx, hipMemcpyAsync(theta, m->theta.p, kNP * sizeof(float), hipMemcpyDeviceToHost,
                              ctx->stream));
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  ctx->d2h += kNP * sizeof(float);
  return CHS_OK;
}

int chs_mlp_loss_grad(chs_context* ctx, chs_mlp* m, const float* d_feat, const float* d_r,
                      const float* d_e, const float* d_w, int64_t n, int band_len, double* loss,
                      float* grad) {
  if (!ctx || !m || !d_feat || !d_r || !d_e || !d_w || n <= 0 || band_len <= 0 ||
      n % band_len != 0)
    return CHS_ERR_INVALID_ARG;
  const long long NB = n / band_len;
  if (NB > (1 << 30)) return CHS_ERR_INVALID_ARG;
  CHS_TRY(ensure(ctx, ctx->impl->small, 64 * sizeof(double)));
  double* dl = (double*)ctx->impl->small.p + 32;
  CHS_TRY(mlp_batch(ctx, m, d_feat, d_r, d_e, d_w, NB, band_len, (int)NB, 0, 1, dl));
  double h = 0.0;
  CHS_HIP(ctx, hipMemcpyAsync(&h, dl, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  ctx->d2h += sizeof(double);
  if (grad) {
    CHS_HIP(ctx, hipMemcpyAsync(grad, m->grad.p, kNP * sizeof(float), hipMemcpyDeviceToHost,
                                ctx->stream));
    ctx->d2h += kNP * sizeof(float);
  }
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (loss) *loss = h;
  return CHS_OK;
}

int chs_mlp_train(chs_context* ctx, chs_mlp* m, const float* d_feat, const float* d_r,
                  const float* d_e, const float* d_w, int64_t n, int band_len, int steps,
                  int batch_bands, float lr, double* loss_trace) {
  if (!ctx || !m || !d_feat || !d_r || !d_e || !d_w || n <= 0 || band_len <= 0 ||
      n % band_len != 0 || steps < 0 || batch_bands <= 0 || !(lr > 0))
    return CHS_ERR_INVALID_ARG;
  const long long NB = n / band_len;
  const int nbb = (int)std::min<long long>(batch_bands, NB);
  const long long stride = coprime_stride(NB);
  CHS_TRY(ensure(ctx, ctx->impl->mlp_ws, (size_t)std::max(steps, 1) * sizeof(double) + 256));
  double* dtrace = (double*)ctx->impl->mlp_ws.p;
  for (int s = 0; s < steps; ++s) {
    const long long off = (long long)(((unsigned long long)s * (unsigned long long)nbb) %
                                      (unsigned long long)NB) * stride % NB;
    CHS_TRY(mlp_batch(ctx, m, d_feat, d_r, d_e, d_w, NB, band_len, nbb, off, stride, dtrace + s));
    m->t += 1;
    const float bc1 = 1.0f - std::pow(0.9f, (float)m->t), bc2 = 1.0f - std::pow(0.999f, (float)m->t);
    hipLaunchKernelGGL(k_mlp_adam, dim3(ceil_div(kNP, 256)), dim3(256), 0, ctx->stream,
                       (float*)m->theta.p, (float*)m->m.p, (float*)m->v.p, (const float*)m->grad.p,
                       lr, bc1, bc2, (unsigned short*)m->wbf.p);
    CHS_LAUNCH_CHECK(ctx);
  }
  if (loss_trace && steps > 0) {
    CHS_HIP(ctx, hipMemcpyAsync(loss_trace, dtrace, steps * sizeof(double), hipMemcpyDeviceToHost,
                                ctx->stream));
    ctx->d2h += steps * sizeof(double);
  }
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return CHS_OK;
}

int chs_mlp_scale_table(chs_context* ctx, chs_mlp* m, const double* d_psi, int n_b,
                        float* d_table) {
  if (!ctx || !m || !d_psi || n_b <= 0 || !d_table) return CHS_ERR_INVALID_ARG;
  Hamiltonian& H = ctx->impl->ham;
  if (!H.bound) return set_error(ctx, CHS_ERR_INVALID_ARG, "no Hamiltonian bound");
  double *ekin, *vstat;
  CHS_TRY(mlp_stats(ctx, (const z64*)d_psi, n_b, &ekin, &vstat));
  hipLaunchKernelGGL(k_mlp_table, dim3(ceil_div(H.n_pw, 256), n_b), dim3(256), 0, ctx->stream,
                     (const unsigned short*)m->wbf.p, H.kin, ekin, vstat, H.n_pw, d_table);
  CHS_LAUNCH_CHECK(ctx);
  return CHS_OK;
}

int chs_mlp_pairs(chs_context* ctx, const double* d_psi, const double* d_psi_ref,
                  const double* eps_ref, int n_b, double gap_min, float* d_feat, float* d_r,
                  float* d_e, float* d_w, int* n_used) {
  if (!ctx || !d_psi || !d_psi_ref || !eps_ref || n_b <= 0 || !d_feat || !d_r || !d_e || !d_w)
    return CHS_ERR_INVALID_ARG;
  Hamiltonian& H = ctx->impl->ham;
  if (!H.bound) return set_error(ctx, CHS_ERR_INVALID_ARG, "no Hamiltonian bound");
  auto* im = ctx->impl;
  const int n_pw = H.n_pw;
  const size_t ne = (size_t)n_b * n_pw, nn2 = (size_t)n_b * n_b;
  CHS_TRY(ensure(ctx, im->ws4, ne * sizeof(z64)));
  CHS_TRY(ensure(ctx, im->ws5, ne * sizeof(z64)));
  CHS_TRY(ensure(ctx, im->ws3, 2 * ne * sizeof(z64)));
  z64* HP = (z64*)im->ws4.p;
  z64* SP = (z64*)im->ws5.p;
  z64* R = (z64*)im->ws3.p;
  z64* E = R + ne;
  const z64* psi = (const z64*)d_psi;
  const z64* ref = (const z64*)d_psi_ref;
  CHS_TRY(apply_h_impl(ctx, CHS_C128, psi, n_b, HP, SP));
  // sized before mlp_stats takes pointers into it
  const size_t dots_off = (((size_t)n_b * 2 * sizeof(double) + 255) / 256) * 256;
  const size_t ov_off = dots_off + (((size_t)n_b * 8 * sizeof(z64) + 255) / 256) * 256;
  CHS_TRY(ensure(ctx, im->mlp_ws, ov_off + nn2 * sizeof(z64) + 256));
  double *ekin, *vstat;
  CHS_TRY(mlp_stats(ctx, psi, n_b, &ekin, &vstat));
  z64* dots = (z64*)((char*)im->mlp_ws.p + dots_off);
  z64* OV = (z64*)((char*)im->mlp_ws.p + ov_off);
  double* wband = ekin + n_b;
  const dim3 eg(ceil_div(n_pw, 256), n_b);
  const z64 one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  hipLaunchKernelGGL(k_pair_dots, dim3(n_b), dim3(256), 0, ctx->stream, psi, SP, n_pw, dots, 0);
  hipLaunchKernelGGL(k_pair_dots, dim3(n_b), dim3(256), 0, ctx->stream, psi, HP, n_pw, dots, 1);
  CHS_LAUNCH_CHECK(ctx);
  // OV[j][b] = <psi*_j | S | psi_b>
  CHS_TRY(zgemm(ctx, 'C', 'N', n_b, n_b, n_pw, one, ref, n_pw, SP, n_pw, zero, OV, n_b));
  std::vector<z64> hov(nn2), hd((size_t)n_b * 8);
  CHS_HIP(ctx, hipMemcpyAsync(hov.data(), OV, nn2 * sizeof(z64), hipMemcpyDeviceToHost,
                              ctx->stream));
  CHS_HIP(ctx, hipMemcpyAsync(hd.data(), dots, hd.size() * sizeof(z64), hipMemcpyDeviceToHost,
                              ctx->stream));
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  ctx->d2h += (nn2 + hd.size()) * sizeof(z64);
  // reference eigenspaces: runs of eigenvalues closer than gap_min; the run
  // touching the top of the block may be incomplete and is not used
  std::vector<int> g0(n_b), g1(n_b);
  for (int b = 0; b < n_b;) {
    int e = b + 1;
    while (e < n_b && eps_ref[e] - eps_ref[e - 1] <= gap_min) ++e;
    for (int j = b; j < e; ++j) {
      g0[j] = b;
      g1[j] = e;
    }
    b = e;
  }
  // t_b = P* psi^_b / |P* psi^_b|: masked, normalised overlap columns
  std::vector<double> wb(n_b, 0.0);
  std::vector<char> ok(n_b, 0);
  for (int b = 0; b < n_b; ++b) {
    double p2 = 0.0;
    for (int j = g0[b]; j < g1[b]; ++j) p2 += norm2(hov[(size_t)j + (size_t)b * n_b]);
    const double nn = hd[(size_t)b * 8].x;
    ok[b] = g1[b] < n_b && nn > 0.0 && p2 / nn > 0.81;
    const double sc = p2 > 0.0 ? 1.0 / std::sqrt(p2) : 0.0;
    for (int j = 0; j < n_b; ++j) {
      z64& o = hov[(size_t)j + (size_t)b * n_b];
      o = (j >= g0[b] && j < g1[b]) ? mk(o.x * sc, o.y * sc) : mk(0.0, 0.0);
    }
  }
  CHS_HIP(ctx, hipMemcpyAsync(OV, hov.data(), nn2 * sizeof(z64), hipMemcpyHostToDevice,
                              ctx->stream));
  ctx->h2d += nn2 * sizeof(z64);
  CHS_TRY(zgemm(ctx, 'N', 'N', n_pw, n_b, n_b, one, ref, n_pw, OV, n_b, zero, E, n_pw));
  hipLaunchKernelGGL(k_pair_build, eg, dim3(256), 0, ctx->stream, psi, HP, SP, n_pw, dots, R, E);
  hipLaunchKernelGGL(k_pair_dots, dim3(n_b), dim3(256), 0, ctx->stream, SP, E, n_pw, dots, 3);
  // |e|^2 after the projection, for the band weights
  hipLaunchKernelGGL(k_sub_scaled, eg, dim3(256), 0, ctx->stream, E, psi, n_pw, dots, HP);
  hipLaunchKernelGGL(k_pair_dots, dim3(n_b), dim3(256), 0, ctx->stream, HP, HP, n_pw, dots, 4);
  CHS_LAUNCH_CHECK(ctx);
  CHS_HIP(ctx, hipMemcpyAsync(hd.data(), dots, hd.size() * sizeof(z64), hipMemcpyDeviceToHost,
                              ctx->stream));
  ctx->d2h += hd.size() * sizeof(z64);
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  int used = 0;
  for (int b = 0; b < n_b; ++b) {
    const double e2 = hd[(size_t)b * 8 + 4].x;
    if (ok[b] && e2 > 1e-24) {
      wb[b] = 1.0 / e2;
      ++used;
    }
  }
  for (double& w : wb) w = used ? w / used : 0.0;
  CHS_HIP(ctx, hipMemcpyAsync(wband, wb.data(), n_b * sizeof(double), hipMemcpyHostToDevice,
                              ctx->stream));
  ctx->h2d += n_b * sizeof(double);
  hipLaunchKernelGGL(k_pair_emit, eg, dim3(256), 0, ctx->stream, psi, R, E, H.kin, ekin, vstat,
                     wband, n_pw, dots, d_feat, d_r, d_e, d_w);
  CHS_LAUNCH_CHECK(ctx);
  CHS_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (n_used) *n_used = used;
  return CHS_OK;
}

}  // extern "C"
