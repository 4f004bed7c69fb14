// Complex GEMM C = alpha op(A) op(B) + beta C (column-major, op in {N, T, C})
// in FP64 (ZGEMM, BlasHandle::gemm_c64, src/device/blas.rs:24-61) and FP32
// with FP32 accumulation (the projector products of the c64 filter).
//
// Block tile 64 x 64 with 256 threads (4 x 4 complex outputs per thread),
// K tiles of 16 staged in LDS. When the output tiles alone cannot fill the
// device (the tall-skinny Gram products Y^H X with K = n_pw), K is split
// across blocks; each slice writes its partial tile and k_gemm_reduce sums
// the slices in a fixed order (deterministic).
#include <algorithm>
#include <utility>

#include "impl.hpp"
#include "linalg.hpp"

namespace chs {

constexpr int GBM = 64, GBN = 64, GBK = 16;

template <typename T, int OP>
__device__ __forceinline__ cplx<T> load_op(const cplx<T>* __restrict__ A, int lda, int r, int c) {
  if (OP == 0) return A[(size_t)r + (size_t)c * lda];
  cplx<T> v = A[(size_t)c + (size_t)r * lda];
  return OP == 2 ? conj(v) : v;
}

template <typename T, int OPA, int OPB>
__global__ void __launch_bounds__(256) k_gemm(int m, int n, int k, cplx<T> alpha,
                                              const cplx<T>* __restrict__ A, int lda,
                                              const cplx<T>* __restrict__ B, int ldb, cplx<T> beta,
                                              cplx<T>* __restrict__ C, int ldc, int klen,
                                              cplx<T>* __restrict__ part) {
  __shared__ cplx<T> As[GBK][GBM + 1];
  __shared__ cplx<T> Bs[GBK][GBN + 1];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m0 = blockIdx.x * GBM, n0 = blockIdx.y * GBN;
  const int kb = blockIdx.z * klen, ke = min(k, kb + klen);
  T ar[4][4], ai[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) ar[i][j] = ai[i][j] = (T)0;
  for (int k0 = kb; k0 < ke; k0 += GBK) {
    for (int t = threadIdx.x; t < GBM * GBK; t += 256) {
      int r, kk;
      if (OPA == 0) { r = t % GBM; kk = t / GBM; } else { kk = t % GBK; r = t / GBK; }
      const int gr = m0 + r, gk = k0 + kk;
      As[kk][r] = (gr < m && gk < ke) ? load_op<T, OPA>(A, lda, gr, gk) : mk((T)0, (T)0);
    }
    for (int t = threadIdx.x; t < GBK * GBN; t += 256) {
      int c, kk;
      if (OPB == 0) { kk = t % GBK; c = t / GBK; } else { c = t % GBN; kk = t / GBN; }
      const int gc = n0 + c, gk = k0 + kk;
      Bs[kk][c] = (gc < n && gk < ke) ? load_op<T, OPB>(B, ldb, gk, gc) : mk((T)0, (T)0);
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GBK; ++kk) {
      cplx<T> a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][tx + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][ty + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ar[i][j] = fma(a[i].x, b[j].x, ar[i][j]);
          ar[i][j] = fma(-a[i].y, b[j].y, ar[i][j]);
          ai[i][j] = fma(a[i].x, b[j].y, ai[i][j]);
          ai[i][j] = fma(a[i].y, b[j].x, ai[i][j]);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = m0 + tx + 16 * i, c = n0 + ty + 16 * j;
      if (r < m && c < n) {
        const cplx<T> acc = mk(ar[i][j], ai[i][j]);
        if (part) {
          part[(size_t)blockIdx.z * m * n + (size_t)r + (size_t)c * m] = acc;
        } else {
          cplx<T> v = alpha * acc;
          if (beta.x != (T)0 || beta.y != (T)0) v = v + beta * C[(size_t)r + (size_t)c * ldc];
          C[(size_t)r + (size_t)c * ldc] = v;
        }
      }
    }
}

// ---------------------------------------------------------------------------
// Matrix-core variant: LDS-staged block tiles (below), register prefetch of
// the next K stage during the MFMAs; the complex product is three real
// 16x16x4 MFMAs per k-step (the 3M form: P1 += ar br, P2 += ai bi,
// P3 += (ar + ai)(br + bi); re = P1 - P2, im = P3 - P1 - P2).
// Operand layout of both v_mfma_f64_16x16x4f64 and v_mfma_f32_16x16x4f32:
// lane l supplies
// A[l % 16][k0 + l / 16] and B[k0 + l / 16][l % 16]. Result layout: lane l
// holds column l % 16, rows 4 (l / 16) + v (f32) or l / 16 + 4 v (f64).
// ---------------------------------------------------------------------------
template <typename T> struct Mfma;
template <> struct Mfma<double> {
  using acc_t = __attribute__((ext_vector_type(4))) double;
  __device__ __forceinline__ static acc_t mac(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <> struct Mfma<float> {
  using acc_t = __attribute__((ext_vector_type(4))) float;
  __device__ __forceinline__ static acc_t mac(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ __forceinline__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// Block tiles of the matrix-core kernel; 4 wavefronts as 2 x 2, each owning
// WTM x WTN MFMA tiles of 16 x 16. Small: 64 x 64 (both precisions); large:
// 128 x 128 x 16 (complex64) or 128 x 64 x 8 (complex128). The autotuner
// picks per GEMM shape.
// WAVES: wavefronts per SIMD the register allocation must leave room for
// (the small tiles keep at least two resident, so one wave's LDS waits and
// barriers do not idle the matrix core).
template <typename T, int V> struct MfmaTile;
template <typename T> struct MfmaTile<T, 1> {
  static constexpr int BM = 64, BN = 64, BK = 16, WTM = 2, WTN = 2;
  static constexpr int WAVES = sizeof(T) == 8 ? 2 : 4;
};
template <> struct MfmaTile<float, 2> {
  static constexpr int BM = 128, BN = 128, BK = 16, WTM = 4, WTN = 4;
  static constexpr int WAVES = 1;
};
// 64 x 64 with a 32-deep K stage: half the barriers per matrix-core product
// and twice the loads in flight per stage, for the long-K products (its
// 16 staged elements per thread need the registers of one wavefront per
// SIMD fewer than the 16-deep tile to stay out of scratch)
template <typename T> struct MfmaTile<T, 3> {
  static constexpr int BM = 64, BN = 64, BK = 32, WTM = 2, WTN = 2;
  static constexpr int WAVES = sizeof(T) == 8 ? 1 : 2;
};
// complex64 tiles with fewer padded rows or columns (gemm_variant says when they
// are tried): 96 x 64 for heights like 864 = 9 x 96, 96 x 32 for widths like
// 160 = 5 x 32. 864 x 512 x 80,725 (beta^H O) 1.90 -> 1.78 ms, 41,000 x 397 x 864
// 0.847 -> 0.825 ms, 23,847 x 160 x 256 84 -> 72 us.
template <> struct MfmaTile<float, 4> {
  static constexpr int BM = 96, BN = 64, BK = 16, WTM = 3, WTN = 2;
  static constexpr int WAVES = 3;
};
template <> struct MfmaTile<float, 5> {
  static constexpr int BM = 96, BN = 32, BK = 16, WTM = 3, WTN = 1;
  static constexpr int WAVES = 4;
};
template <> struct MfmaTile<double, 2> {
  static constexpr int BM = 128, BN = 64, BK = 8, WTM = 4, WTN = 2;
  static constexpr int WAVES = 1;
};

// XCD-aware block order: workgroups are dealt to the eight XCDs round-robin
// by launch index, so physical block p runs on XCD p % 8. Logical block
// L = (p % 8) * (P / 8) + p / 8 gives every XCD a contiguous range of
// logical blocks, ordered (k-slice, then tiles) so that the tiles sharing a
// k-slice sit in one L2. Within a slice the tiles that share the larger
// operand are consecutive (nfast: column tile fastest, so the column tiles
// of one row tile of A run together and A streams from HBM about once;
// otherwise row tile fastest, for a B wider than A is tall).
__device__ __forceinline__ bool gemm_block(int mt, int nt, int kz, int nfast, int* bm, int* bn,
                                           int* bz) {
  const int P = gridDim.x, p = blockIdx.x;
  const int L = (p & 7) * (P >> 3) + (p >> 3);
  if (L >= mt * nt * kz) return false;
  if (nfast) {
    *bn = L % nt;
    *bm = (L / nt) % mt;
  } else {
    *bm = L % mt;
    *bn = (L / mt) % nt;
  }
  *bz = L / (mt * nt);
  return true;
}

// CL: each thread keeps one 32-bit byte offset per staged element from a
// uniform base, set once (rows and columns past the matrix edge clamped to
// the last one: they only feed output elements that are never stored); the
// bases advance by one K stage per stage, so a full stage's loads need no
// address arithmetic or bounds tests, and only a slice's last, partial stage
// tests k against its end. Usable while every offset fits in 32 bits
// (cl_offsets_fit). Otherwise each element's load sits behind its bounds
// test. Which is faster depends on the shape (the autotuner decides).
template <typename T, int OPA, int OPB, int V, bool CL>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(MfmaTile<T, V>::WAVES))) k_gemm_mfma(int m, int n, int k, cplx<T> alpha,
                                                   const cplx<T>* __restrict__ A, int lda,
                                                   const cplx<T>* __restrict__ B, int ldb,
                                                   cplx<T> beta, cplx<T>* __restrict__ C, int ldc,
                                                   int klen, int ksplit, int nfast, int tri,
                                                   cplx<T>* __restrict__ part) {
  using M = Mfma<T>;
  using acc_t = typename M::acc_t;
  using TL = MfmaTile<T, V>;
  constexpr int BM = TL::BM, BN = TL::BN, BK = TL::BK;
  constexpr int WTM = TL::WTM, WTN = TL::WTN;
  int bm, bn, bz;
  if (!gemm_block((m + BM - 1) / BM, (n + BN - 1) / BN, ksplit, nfast, &bm, &bn, &bz)) return;
  if (tri && bm * BM >= (bn + 1) * BN) return;  // Hermitian product: tiles below the diagonal
  // Workgroups that share a CU (every 256th or so) get two wave priorities, so
  // that their product phases do not run in step and leave the matrix cores
  // idle together. Complex64, without and with: 80,725 x 512 x 864 1.825 and
  // 1.785 ms, 63,077 x 360 x 864 1.094 and 1.073, 80,725 x 512 x 512 1.122 and
  // 1.088; short sums lose by it (17,071 x 192 x 256 69.7 and 72.0 us), as do
  // the 96-row tiles, three wavefronts per SIMD
  if constexpr (sizeof(T) == 4 && V == 1 && CL)
    if (klen >= 512 && ((blockIdx.x >> 8) & 1)) __builtin_amdgcn_s_setprio(2);
  constexpr int NA = BM * BK / 256, NB = BN * BK / 256;  // staged elements per thread
  // one padding element per row: the K-major (transposing) stores of T / C
  // operands then hit distinct banks across each phase of lanes, while the
  // MFMA operand reads stay contiguous along the row
  __shared__ cplx<T> As[BK][BM + 1];
  __shared__ cplx<T> Bs[BK][BN + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm0 = (w >> 1) * (16 * WTM), wn0 = (w & 1) * (16 * WTN);
  const int li = lane & 15, lk = lane >> 4;
  const int m0 = bm * BM, n0 = bn * BN;
  const int kb = bz * klen, ke = min(k, kb + klen);
  // three real products per complex one (Re = P1 - P2, Im = P3 - P1 - P2
  // with P1 = sum ar br, P2 = sum ai bi, P3 = sum (ar + ai)(br + bi)).
  // CL stages an op-C operand unconjugated and folds the conjugation into
  // the products: with s_a, s_b = -1 for a conjugated operand (else 1) and
  // P3 = sum (ar + s_a ai)(br + s_b bi), Re = P1 - s_a s_b P2 and
  // Im = P3 - P1 - s_a s_b P2.
  constexpr int SA = CL && OPA == 2 ? -1 : 1, SB = CL && OPB == 2 ? -1 : 1;
  constexpr int OPA_LD = CL && OPA == 2 ? 1 : OPA, OPB_LD = CL && OPB == 2 ? 1 : OPB;
  acc_t p1[WTM][WTN], p2[WTM][WTN], p3[WTM][WTN];
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j) {
      p1[i][j] = acc_t{0, 0, 0, 0};
      p2[i][j] = acc_t{0, 0, 0, 0};
      p3[i][j] = acc_t{0, 0, 0, 0};
    }
  cplx<T> ra[NA], rb[NB];
  auto a_pos = [](int e, int& r, int& kk) {
    if (OPA == 0) { r = e % BM; kk = e / BM; } else { kk = e % BK; r = e / BK; }
  };
  auto b_pos = [](int e, int& c, int& kk) {
    if (OPB == 0) { kk = e % BK; c = e / BK; } else { c = e % BN; kk = e / BN; }
  };
  // CL: per-element byte offsets from the operands' stage bases (32-bit: the
  // host takes the bounds-tested kernel when they would not fit), the bases
  // advanced by one K stage after each stage's loads
  uint32_t oa[CL ? NA : 1], ob[CL ? NB : 1];
  const char* base_a = reinterpret_cast<const char*>(A + (OPA == 0 ? (size_t)kb * lda : kb));
  const char* base_b = reinterpret_cast<const char*>(B + (OPB == 0 ? kb : (size_t)kb * ldb));
  const size_t sa = (OPA == 0 ? (size_t)BK * lda : (size_t)BK) * sizeof(cplx<T>);
  const size_t sb = (OPB == 0 ? (size_t)BK : (size_t)BK * ldb) * sizeof(cplx<T>);
  if constexpr (CL) {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      int r, kk;
      a_pos(threadIdx.x + 256 * j, r, kk);
      const size_t gr = (size_t)min(m0 + r, m - 1);
      oa[j] = (uint32_t)((OPA == 0 ? gr + (size_t)kk * lda : kk + gr * lda) * sizeof(cplx<T>));
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      int c, kk;
      b_pos(threadIdx.x + 256 * j, c, kk);
      const size_t gc = (size_t)min(n0 + c, n - 1);
      ob[j] = (uint32_t)((OPB == 0 ? kk + gc * ldb : gc + (size_t)kk * ldb) * sizeof(cplx<T>));
    }
  }
  // Bounds-tested loads of stage k0 (the non-CL kernel, and the CL kernel's
  // partial last stage of a slice: k >= ke zero, rows and columns past the
  // edge clamped as the offsets are)
  auto load_tested = [&](int k0) {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      int r, kk;
      a_pos(threadIdx.x + 256 * j, r, kk);
      const int gr = CL ? min(m0 + r, m - 1) : m0 + r, gk = k0 + kk;
      ra[j] = (gr < m && gk < ke) ? load_op<T, OPA_LD>(A, lda, gr, gk) : mk((T)0, (T)0);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      int c, kk;
      b_pos(threadIdx.x + 256 * j, c, kk);
      const int gc = CL ? min(n0 + c, n - 1) : n0 + c, gk = k0 + kk;
      rb[j] = (gc < n && gk < ke) ? load_op<T, OPB_LD>(B, ldb, gk, gc) : mk((T)0, (T)0);
    }
  };
  // CL, full stages: one plain load per element at its offset, the values
  // untouched until the LDS store of the next stage, so they are waited for
  // only after this stage's matrix-core products
  auto load_plain = [&]() {
#pragma unroll
    for (int j = 0; j < NA; ++j) ra[j] = *reinterpret_cast<const cplx<T>*>(base_a + oa[j]);
#pragma unroll
    for (int j = 0; j < NB; ++j) rb[j] = *reinterpret_cast<const cplx<T>*>(base_b + ob[j]);
    base_a += sa;
    base_b += sb;
  };
  auto store = [&]() {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      int r, kk;
      a_pos(threadIdx.x + 256 * j, r, kk);
      As[kk][r] = ra[j];
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      int c, kk;
      b_pos(threadIdx.x + 256 * j, c, kk);
      Bs[kk][c] = rb[j];
    }
  };
  auto products = [&]() {
#pragma unroll
    for (int s = 0; s < BK / 4; ++s) {
      const int kk = 4 * s + lk;
      cplx<T> a[WTM], b[WTN];
#pragma unroll
      for (int i = 0; i < WTM; ++i) a[i] = As[kk][wm0 + 16 * i + li];
#pragma unroll
      for (int j = 0; j < WTN; ++j) b[j] = Bs[kk][wn0 + 16 * j + li];
      // independent accumulators back to back: each product class over all
      // tiles before the next
#pragma unroll
      for (int i = 0; i < WTM; ++i)
#pragma unroll
        for (int j = 0; j < WTN; ++j) p1[i][j] = M::mac(a[i].x, b[j].x, p1[i][j]);
#pragma unroll
      for (int i = 0; i < WTM; ++i)
#pragma unroll
        for (int j = 0; j < WTN; ++j) p2[i][j] = M::mac(a[i].y, b[j].y, p2[i][j]);
#pragma unroll
      for (int i = 0; i < WTM; ++i)
#pragma unroll
        for (int j = 0; j < WTN; ++j)
          p3[i][j] = M::mac(a[i].x + (T)SA * a[i].y, b[j].x + (T)SB * b[j].y, p3[i][j]);
    }
  };
  if constexpr (CL) {
    // full stages with the next one's loads in flight, then the partial one
    const int kf = kb + max(0, (ke - kb) / BK) * BK;
    if (kb < kf) load_plain();
    for (int k0 = kb; k0 < kf; k0 += BK) {
      store();
      __syncthreads();
      if (k0 + BK < kf) load_plain();
      products();
      __syncthreads();
    }
    if (kf < ke) {
      load_tested(kf);
      store();
      __syncthreads();
      products();
    }
  } else {
    if (kb < ke) load_tested(kb);
    for (int k0 = kb; k0 < ke; k0 += BK) {
      store();
      __syncthreads();
      if (k0 + BK < ke) load_tested(k0 + BK);  // next stage in flight during the MFMAs
      products();
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = m0 + wm0 + 16 * i + M::row(lane, v);
        const int c = n0 + wn0 + 16 * j + li;
        if (r < m && c < n) {
          const T r1 = (T)p1[i][j][v], r2 = (T)p2[i][j][v];
          const T r2s = SA * SB < 0 ? -r2 : r2;
          const cplx<T> acc = mk(r1 - r2s, (T)p3[i][j][v] - r1 - r2s);
          if (part) {
            part[(size_t)bz * m * n + (size_t)r + (size_t)c * m] = acc;
          } else {
            cplx<T> val = alpha * acc;
            if (beta.x != (T)0 || beta.y != (T)0) val = val + beta * C[(size_t)r + (size_t)c * ldc];
            C[(size_t)r + (size_t)c * ldc] = val;
          }
        }
      }
}

// ---------------------------------------------------------------------------
// Small products (V = 6): 32 x 32 output tiles whose K range is split over the
// four wavefronts of a workgroup, operands loaded straight from L2 into MFMA
// registers (no LDS stage, no barrier in the K loop), the four partial tiles
// summed in order through LDS. For products whose 64 x 64 tiles leave most of
// the chip idle and whose time is the K loop's latency: the coefficient-space
// products of the filter. Complex64: 512 x 160 x 256 in 7.5 us (64 x 64 tiles:
// 26 us for 256 x 160 x 256), 256 x 160 x 23,847 in 69 us (75), 32 x 20 x 2,945
// in 6.5 us (22). Lane (lk, li) supplies k = k0 + 2 lk + u in step u of an
// 8-deep chunk, so a lane's two loads of a K-contiguous operand share 16 bytes.
// ---------------------------------------------------------------------------
constexpr int kSM = 32;  // output tile edge

template <typename T, int OPA>
__global__ void __launch_bounds__(256) k_gemm_small(int m, int n, int k, cplx<T> alpha,
                                                    const cplx<T>* __restrict__ A, int lda,
                                                    const cplx<T>* __restrict__ B, int ldb,
                                                    cplx<T> beta, cplx<T>* __restrict__ C, int ldc,
                                                    int klen, cplx<T>* __restrict__ part) {
  using M = Mfma<T>;
  using acc_t = typename M::acc_t;
  constexpr int SA = OPA == 2 ? -1 : 1;  // conjugation folded into the products (k_gemm_mfma)
  __shared__ cplx<T> red[4][4][4][64];   // [wavefront][tile][v][lane]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int m0 = blockIdx.x * kSM, n0 = blockIdx.y * kSM;
  const int kb = blockIdx.z * klen, ke = min(k, kb + klen);
  const int kw = ((klen + 3) / 4 + 7) / 8 * 8;  // K per wavefront, whole chunks
  const int k0 = min(ke, kb + w * kw), k1 = min(ke, k0 + kw);
  // rows and columns past the edge are clamped: they feed outputs never stored
  const cplx<T>*pa[2], *pb[2];
  const size_t ka = OPA == 0 ? (size_t)lda : 1;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = min(m0 + 16 * i + li, m - 1), c = min(n0 + 16 * i + li, n - 1);
    pa[i] = A + (OPA == 0 ? (size_t)r : (size_t)r * lda);
    pb[i] = B + (size_t)c * ldb;
  }
  acc_t p1[2][2], p2[2][2], p3[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) p1[i][j] = p2[i][j] = p3[i][j] = acc_t{0, 0, 0, 0};
  auto products = [&](const cplx<T> (&a)[2], const cplx<T> (&b)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) p1[i][j] = M::mac(a[i].x, b[j].x, p1[i][j]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) p2[i][j] = M::mac(a[i].y, b[j].y, p2[i][j]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        p3[i][j] = M::mac(a[i].x + (T)SA * a[i].y, b[j].x + b[j].y, p3[i][j]);
  };
  int kk = k0;
#pragma unroll 2
  for (; kk + 8 <= k1; kk += 8) {
    cplx<T> a[2][2], b[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const size_t q = (size_t)(kk + 2 * lk + u);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[u][i] = pa[i][q * ka];
        b[u][i] = pb[i][q];
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) products(a[u], b[u]);
  }
  if (kk < k1) {  // partial chunk: k past the end reads the last one and counts as zero
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int q = kk + 2 * lk + u;
      const bool in = q < k1;
      const size_t qc = (size_t)min(q, k1 - 1);
      cplx<T> a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = in ? pa[i][qc * ka] : mk((T)0, (T)0);
        b[i] = in ? pb[i][qc] : mk((T)0, (T)0);
      }
      products(a, b);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T r1 = (T)p1[i][j][v], r2 = (T)p2[i][j][v], r2s = SA < 0 ? -r2 : r2;
        red[w][2 * i + j][v][lane] = mk(r1 - r2s, (T)p3[i][j][v] - r1 - r2s);
      }
  __syncthreads();
  // wavefront w stores tile w
  const int i = w >> 1, j = w & 1;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const cplx<T> acc = (red[0][w][v][lane] + red[1][w][v][lane]) +
                        (red[2][w][v][lane] + red[3][w][v][lane]);
    const int r = m0 + 16 * i + M::row(lane, v), c = n0 + 16 * j + li;
    if (r < m && c < n) {
      if (part) {
        part[(size_t)blockIdx.z * m * n + (size_t)r + (size_t)c * m] = acc;
      } else {
        cplx<T> val = alpha * acc;
        if (beta.x != (T)0 || beta.y != (T)0) val = val + beta * C[(size_t)r + (size_t)c * ldc];
        C[(size_t)r + (size_t)c * ldc] = val;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// n = 1 (matrix-vector) in the memory-bound form: y = alpha op(A) x + beta y.
// Both forms cut K into slices (blockIdx.y) so that a few thousand
// wavefronts stream A, with four independent loads in flight per lane;
// with more than one slice each writes a partial vector and k_gemv_fin adds
// them in slice order (deterministic).
// op N: one thread per row, A read down its columns (coalesced across rows);
// op T / C: one wavefront per output element, a reduction along the column.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void cmac(cplx<T> a, cplx<T> b, T& re, T& im) {
  re = fma(a.x, b.x, re);
  re = fma(-a.y, b.y, re);
  im = fma(a.x, b.y, im);
  im = fma(a.y, b.x, im);
}

template <typename T>
__device__ __forceinline__ void gemv_out(cplx<T> acc, cplx<T> alpha, cplx<T> beta,
                                         cplx<T>* __restrict__ y, cplx<T>* __restrict__ part,
                                         int m, int i) {
  if (part) {
    part[(size_t)blockIdx.y * m + i] = acc;
  } else {
    cplx<T> v = alpha * acc;
    if (beta.x != (T)0 || beta.y != (T)0) v = v + beta * y[i];
    y[i] = v;
  }
}

// TA: the matrix's element type (complex64 under complex128 vectors and
// accumulation is the mixed form: half the matrix bytes).
template <typename T, typename TA = T>
__device__ __forceinline__ cplx<T> widen_el(cplx<TA> a) {
  return mk((T)a.x, (T)a.y);
}

template <typename T, typename TA = T>
__global__ void __launch_bounds__(256) k_gemv_n(int m, int k, int klen, cplx<T> alpha,
                                                const cplx<TA>* __restrict__ A, int lda,
                                                const cplx<T>* __restrict__ x, cplx<T> beta,
                                                cplx<T>* __restrict__ y,
                                                cplx<T>* __restrict__ part) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const int kb = blockIdx.y * klen, ke = min(k, kb + klen);
  T re[4] = {0, 0, 0, 0}, im[4] = {0, 0, 0, 0};
  int kk = kb;
  for (; kk + 4 <= ke; kk += 4) {
    cplx<T> a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = widen_el<T>(A[(size_t)i + (size_t)(kk + u) * lda]);
#pragma unroll
    for (int u = 0; u < 4; ++u) cmac(a[u], x[kk + u], re[u], im[u]);
  }
  for (; kk < ke; ++kk) cmac(widen_el<T>(A[(size_t)i + (size_t)kk * lda]), x[kk], re[0], im[0]);
  gemv_out(mk((re[0] + re[1]) + (re[2] + re[3]), (im[0] + im[1]) + (im[2] + im[3])), alpha, beta,
           y, part, m, i);
}

template <typename T, int OPA, typename TA = T>
__global__ void __launch_bounds__(256) k_gemv_t(int m, int k, int klen, cplx<T> alpha,
                                                const cplx<TA>* __restrict__ A, int lda,
                                                const cplx<T>* __restrict__ x, cplx<T> beta,
                                                cplx<T>* __restrict__ y,
                                                cplx<T>* __restrict__ part) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= m) return;
  const int kb = blockIdx.y * klen, ke = min(k, kb + klen);
  const cplx<TA>* col = A + (size_t)i * lda;
  T re[4] = {0, 0, 0, 0}, im[4] = {0, 0, 0, 0};
  int kk = kb + lane;
  for (; kk + 192 < ke; kk += 256) {
    cplx<T> a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = widen_el<T>(col[kk + 64 * u]);
      b[u] = x[kk + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (OPA == 2) a[u].y = -a[u].y;
      cmac(a[u], b[u], re[u], im[u]);
    }
  }
  for (; kk < ke; kk += 64) {
    cplx<T> a = widen_el<T>(col[kk]);
    if (OPA == 2) a.y = -a.y;
    cmac(a, x[kk], re[0], im[0]);
  }
  T sr = (re[0] + re[1]) + (re[2] + re[3]), si = (im[0] + im[1]) + (im[2] + im[3]);
  for (int off = 32; off > 0; off >>= 1) {
    sr += __shfl_down(sr, off);
    si += __shfl_down(si, off);
  }
  if (lane == 0) gemv_out(mk(sr, si), alpha, beta, y, part, m, i);
}

template <typename T>
__global__ void k_gemv_fin(int m, int ns, const cplx<T>* __restrict__ part, cplx<T> alpha,
                           cplx<T> beta, cplx<T>* __restrict__ y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  cplx<T> s = part[i];
  for (int z = 1; z < ns; ++z) s = s + part[(size_t)z * m + i];
  cplx<T> v = alpha * s;
  if (beta.x != (T)0 || beta.y != (T)0) v = v + beta * y[i];
  y[i] = v;
}

// K slices of a matrix-vector product with `waves` wavefronts per slice:
// about 4096 wavefronts in all, slices of at least `min_len` elements.
static void gemv_plan(int k, int waves, int min_len, int* ns, int* klen) {
  int s = std::max(1, std::min((4096 + waves - 1) / waves, k / min_len));
  int kl = (k + s - 1) / s;
  *klen = std::max(1, kl);
  *ns = (k + *klen - 1) / *klen;
}

template <typename T, typename TA = T>
static int gemv_launch(chs_context* ctx, int oa, int m, int k, cplx<T> alpha, const cplx<TA>* A,
                       int lda, const cplx<T>* x, cplx<T> beta, cplx<T>* y) {
  int ns, klen;
  if (oa == 0)
    // short rows keep one slice and need no second launch; longer ones want the
    // slices no shorter either (ten-step Lanczos bound of 23,847 plane waves and
    // 256 projectors: 1.22 ms with slices of 64, 1.24 with 32 or 16; 9,315 and
    // 256: 0.78, 0.76, 0.80)
    gemv_plan(k, (int)ceil_div(m, 64), 64, &ns, &klen);
  else
    gemv_plan(k, m, 512, &ns, &klen);
  cplx<T>* part = nullptr;
  if (ns > 1) {
    CHS_TRY(ensure(ctx, ctx->impl->gemv_ws, (size_t)ns * m * sizeof(cplx<T>)));
    part = (cplx<T>*)ctx->impl->gemv_ws.p;
  }
  if (oa == 0)
    hipLaunchKernelGGL((k_gemv_n<T, TA>), dim3(ceil_div(m, 256), ns), dim3(256), 0, ctx->stream, m,
                       k, klen, alpha, A, lda, x, beta, y, part);
  else if (oa == 1)
    hipLaunchKernelGGL((k_gemv_t<T, 1, TA>), dim3(ceil_div(m, 4), ns), dim3(256), 0, ctx->stream, m,
                       k, klen, alpha, A, lda, x, beta, y, part);
  else
    hipLaunchKernelGGL((k_gemv_t<T, 2, TA>), dim3(ceil_div(m, 4), ns), dim3(256), 0, ctx->stream, m,
                       k, klen, alpha, A, lda, x, beta, y, part);
  CHS_LAUNCH_CHECK(ctx);
  if (ns > 1) {
    hipLaunchKernelGGL((k_gemv_fin<T>), dim3(ceil_div(m, 256)), dim3(256), 0, ctx->stream, m, ns,
                       (const cplx<T>*)part, alpha, beta, y);
    CHS_LAUNCH_CHECK(ctx);
  }
  return CHS_OK;
}

template <typename T>
__global__ void k_gemm_reduce(int m, int n, int nz, const cplx<T>* __restrict__ part,
                              cplx<T> alpha, cplx<T> beta, cplx<T>* __restrict__ C, int ldc) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)m * n) return;
  const size_t mn = (size_t)m * n;
  cplx<T> s = mk((T)0, (T)0);
  int z = 0;
  for (; z + 8 <= nz; z += 8) {  // eight loads in flight, added in slice order
    cplx<T> t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = part[(size_t)(z + u) * mn + idx];
#pragma unroll
    for (int u = 0; u < 8; ++u) s = s + t[u];
  }
  for (; z < nz; ++z) s = s + part[(size_t)z * mn + idx];
  const int r = (int)(idx % m), c = (int)(idx / m);
  cplx<T> v = alpha * s;
  if (beta.x != (T)0 || beta.y != (T)0) v = v + beta * C[(size_t)r + (size_t)c * ldc];
  C[(size_t)r + (size_t)c * ldc] = v;
}

int gemm_opcode(char op) {
  switch (op) {
    case 'N': case 'n': return 0;
    case 'T': case 't': return 1;
    case 'C': case 'c': return 2;
    default: return -1;
  }
}

// Split-K plan of a tile shape: when the output tiles alone cannot fill the
// device, K is cut into slices of whole K tiles until about `target`
// workgroups are in flight (more resident waves per CU hide the operand
// latency of the long-K products better; the autotuner picks the target).
// (8192 and 16384 were measured too: never faster on the 216-atom shapes)
static constexpr int kNumSplitTargets = 4;
static constexpr int kSplitTargets[kNumSplitTargets] = {512, 1024, 2048, 4096};

template <typename T>
static void tile_dims(int variant, int* bm, int* bn, int* bk) {
  *bm = GBM; *bn = GBN; *bk = GBK;
  if (variant == 6) *bm = *bn = *bk = kSM;
  if (variant == 7 || variant == 8) {
    using T4 = MfmaTile<float, 4>;
    using T5 = MfmaTile<float, 5>;
    *bm = variant == 7 ? T4::BM : T5::BM;
    *bn = variant == 7 ? T4::BN : T5::BN;
    *bk = variant == 7 ? T4::BK : T5::BK;
  }
  if (variant == 1 || variant == 3) {
    *bm = MfmaTile<T, 1>::BM; *bn = MfmaTile<T, 1>::BN; *bk = MfmaTile<T, 1>::BK;
  } else if (variant == 5) {
    *bm = MfmaTile<T, 3>::BM; *bn = MfmaTile<T, 3>::BN; *bk = MfmaTile<T, 3>::BK;
  } else if (variant == 2 || variant == 4) {
    *bm = MfmaTile<T, 2>::BM; *bn = MfmaTile<T, 2>::BN; *bk = MfmaTile<T, 2>::BK;
  }
}

// tri: only the tiles that reach the diagonal or above are computed
// min_len: shortest slice (the small kernel's wavefronts quarter it again)
static void split_plan(int m, int n, int k, int bm, int bn, int bk, int target, int* ksplit,
                       int* klen, bool tri = false, int min_len = 256) {
  int tiles = (int)(ceil_div(m, bm) * ceil_div(n, bn));
  if (tri) {
    tiles = 0;
    for (int i = 0; i < (int)ceil_div(m, bm); ++i)
      for (int j = 0; j < (int)ceil_div(n, bn); ++j) tiles += i * bm < (j + 1) * bn;
  }
  int ks = 1;
  // at most `target` workgroups: whole rounds of resident workgroups, no
  // nearly empty last round
  if (tiles < target && k > 4 * bk)
    ks = std::max(1, std::min(target / tiles, (k + min_len - 1) / min_len));
  int kl = (k + ks - 1) / ks;
  kl = ((kl + bk - 1) / bk) * bk;
  if (kl == 0) kl = bk;
  *klen = kl;
  *ksplit = std::max(1, (k + kl - 1) / kl);
}

// Split of variant v at a target (gemm_launch and the tuner agree on it).
template <typename T>
static void variant_plan(int v, int m, int n, int k, int target, bool tri, int* ksplit, int* klen) {
  int bm, bn, bk;
  tile_dims<T>(v, &bm, &bn, &bk);
  split_plan(m, n, k, bm, bn, bk, target, ksplit, klen, tri && v != 0, v == 6 ? 128 : 256);
}

// Largest byte offset of a CL kernel's operand element from its stage base
// (rows and columns clamped to the matrix, k within one stage) below 2^32.
template <typename T>
static bool cl_offsets_fit(int oa, int ob, int m, int n, int lda, int ldb, int bk) {
  const double sz = (double)sizeof(cplx<T>);
  const double a = oa == 0 ? (m - 1) + (double)(bk - 1) * lda : (bk - 1) + (double)(m - 1) * lda;
  const double b = ob == 0 ? (bk - 1) + (double)(n - 1) * ldb : (n - 1) + (double)(bk - 1) * ldb;
  return a * sz < 4294967296.0 && b * sz < 4294967296.0;
}

template <typename T>
static int gemm_launch(chs_context* ctx, int choice, int oa, int ob, int m, int n, int k,
                       cplx<T> alpha, const cplx<T>* A, int lda, const cplx<T>* B, int ldb,
                       cplx<T> beta, cplx<T>* C, int ldc, DevBuf& ws, int tri = 0) {
  int variant = choice & 15;
  const int target = kSplitTargets[(choice >> 4) % kNumSplitTargets];
  // the offset-addressed kernels (3, 4, 5) only while their offsets fit 32 bits;
  // otherwise the bounds-tested kernel of the same tile
  if (variant > 8) variant = 0;  // no such kernel (CHS_GEMM_CHOICE, a hand-written cache line)
  if (variant == 6 && (oa == 1 || ob != 0 || tri)) variant = 3;
  if (variant >= 7 && (sizeof(T) == 8 || oa == 1 || ob != 0 || tri)) variant = 3;
  if (variant >= 3 && variant != 6) {
    int bm0, bn0, bk0;
    tile_dims<T>(variant, &bm0, &bn0, &bk0);
    if (!cl_offsets_fit<T>(oa, ob, m, n, lda, ldb, bk0)) variant = variant == 4 ? 2 : 1;
  }
  int bm, bn, bk;
  tile_dims<T>(variant, &bm, &bn, &bk);
  int ksplit, klen;
  variant_plan<T>(variant, m, n, k, target, tri, &ksplit, &klen);
  cplx<T>* part = nullptr;
  if (ksplit > 1) {
    CHS_TRY(ensure(ctx, ws, (size_t)ksplit * m * n * sizeof(cplx<T>)));
    part = (cplx<T>*)ws.p;
  }
  const unsigned nblk = ceil_div(m, bm) * ceil_div(n, bn) * (unsigned)ksplit;
  const int nfast = m > n ? 1 : 0;  // tiles sharing the larger operand run together
  const dim3 g1(((nblk + 7) / 8) * 8);  // multiple of 8 for the XCD-aware order
  const dim3 g3(ceil_div(m, bm), ceil_div(n, bn), ksplit);
  if (variant == 6) {
    if (oa == 0)
      hipLaunchKernelGGL((k_gemm_small<T, 0>), g3, dim3(256), 0, ctx->stream, m, n, k, alpha, A,
                         lda, B, ldb, beta, C, ldc, klen, part);
    else
      hipLaunchKernelGGL((k_gemm_small<T, 2>), g3, dim3(256), 0, ctx->stream, m, n, k, alpha, A,
                         lda, B, ldb, beta, C, ldc, klen, part);
  } else if (variant >= 7) {
    if constexpr (sizeof(T) == 4) {
#define CHS_GEMM_96(OA, V)                                                                       \
  hipLaunchKernelGGL((k_gemm_mfma<T, OA, 0, V, true>), g1, dim3(256), 0, ctx->stream, m, n, k,   \
                     alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part)
      if (variant == 7 && oa == 0)
        CHS_GEMM_96(0, 4);
      else if (variant == 7)
        CHS_GEMM_96(2, 4);
      else if (oa == 0)
        CHS_GEMM_96(0, 5);
      else
        CHS_GEMM_96(2, 5);
#undef CHS_GEMM_96
    }
  } else {
#define CHS_GEMM_CASE(OA, OB)                                                                    \
  if (oa == OA && ob == OB) {                                                                    \
    if (variant == 1)                                                                            \
      hipLaunchKernelGGL((k_gemm_mfma<T, OA, OB, 1, false>), g1, dim3(256), 0, ctx->stream, m,   \
                         n, k, alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part);  \
    else if (variant == 2)                                                                       \
      hipLaunchKernelGGL((k_gemm_mfma<T, OA, OB, 2, false>), g1, dim3(256), 0, ctx->stream, m,   \
                         n, k, alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part);  \
    else if (variant == 3)                                                                       \
      hipLaunchKernelGGL((k_gemm_mfma<T, OA, OB, 1, true>), g1, dim3(256), 0, ctx->stream, m,    \
                         n, k, alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part);  \
    else if (variant == 4)                                                                       \
      hipLaunchKernelGGL((k_gemm_mfma<T, OA, OB, 2, true>), g1, dim3(256), 0, ctx->stream, m,    \
                         n, k, alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part);  \
    else if (variant == 5)                                                                       \
      hipLaunchKernelGGL((k_gemm_mfma<T, OA, OB, 3, true>), g1, dim3(256), 0, ctx->stream, m,    \
                         n, k, alpha, A, lda, B, ldb, beta, C, ldc, klen, ksplit, nfast, tri, part);  \
    else                                                                                         \
      hipLaunchKernelGGL((k_gemm<T, OA, OB>), g3, dim3(256), 0, ctx->stream, m, n, k, alpha, A,  \
                         lda, B, ldb, beta, C, ldc, klen, part);                                 \
  }
  CHS_GEMM_CASE(0, 0) CHS_GEMM_CASE(0, 1) CHS_GEMM_CASE(0, 2)
  CHS_GEMM_CASE(1, 0) CHS_GEMM_CASE(1, 1) CHS_GEMM_CASE(1, 2)
  CHS_GEMM_CASE(2, 0) CHS_GEMM_CASE(2, 1) CHS_GEMM_CASE(2, 2)
#undef CHS_GEMM_CASE
  }
  CHS_LAUNCH_CHECK(ctx);
  if (ksplit > 1) {
    hipLaunchKernelGGL((k_gemm_reduce<T>), dim3(ceil_div((size_t)m * n, 256)), dim3(256), 0,
                       ctx->stream, m, n, ksplit, part, alpha, beta, C, ldc);
    CHS_LAUNCH_CHECK(ctx);
  }
  return CHS_OK;
}

// longest K slice of a complex64 product: beta^H O of the 216-atom cell in 7
// slices of 11,536 (1.77 ms) put the filter's error at 4.7e-7 of the result, in
// 28 of 2,896 (1.80 ms) at 3.7e-7
constexpr int kMaxChain = 3072;

// most 32 x 32 tiles the small-product kernel is tried with: four workgroups per
// CU (with more, 64 x 64 tiles fill the chip and share operands through LDS: at
// 3,730 tiles of the 64-atom O + beta C both take 86 us)
constexpr int kSmallTiles = 1024;
// and the most products (864 x 512 x 80,725 = 3.6e10 takes 2.4 times the 64 x 64
// tiles' time; 256 x 160 x 23,847 = 9.8e8 is 20% faster)
constexpr double kSmallWork = 4e9;

// Split-K target of a complex128 product, by its shape alone. The order of its
// sums, hence the last bits of H_sub and S_sub, sets the signs of Rayleigh-Ritz's
// eigenvectors (inverse iteration keeps the sign of a rounding error), so it must
// not follow the tuner's timings: candidates 1% apart (864 x 512 x 80,725: 18
// slices 3.42 ms, 36 slices 3.44 ms) were picked differently from one context to
// the next. The smallest target that gives enough slices, as long as they stay
// longer than a least length; `ms` below is without and with that target's split.
//  - All tiles: 17 slices whose workgroups fill the target to 97% (864 x 360 x
//    63,077: 12 slices 2.11 ms, 24 2.07; 864 x 440 x 60,245: 20 slices fill 96%,
//    2.32, 41 fill 98%, 2.29), no shorter than 800 (256 x 400 x 23,847: 36 slices
//    of 672 0.305 ms, 18 of 1,328 0.295).
//  - Upper tiles only: 48 slices in a multiple of 8 or 70, since the tiles below
//    the diagonal are launched too and end at once, and with a broken number of
//    slices an XCD gets more of the others (512 x 512 x 80,725: 28 slices 1.70 ms,
//    56 1.57; 302 x 302 x 74,509: 68 slices 0.598, 134 0.550), no shorter than 272
//    (300 x 300 x 13,133: 52 slices of 256 0.141 ms, 33 of 400 0.112).
// Of 180 shapes of the 64- and 216-atom cells all but nine take the split that was
// timed fastest or one within 1.5% of it, those one within 5%.
static int fixed_split_target(int m, int n, int k, bool tri) {
  int bm, bn, bk, ks, kl, ti = 0;
  tile_dims<double>(3, &bm, &bn, &bk);
  const double tiles = (double)ceil_div(m, bm) * ceil_div(n, bn);
  for (int t = 0; t < kNumSplitTargets; ++t) {
    variant_plan<double>(3, m, n, k, kSplitTargets[t], tri, &ks, &kl);
    if (t > 0 && kl < (tri ? 272 : 800)) break;
    ti = t;
    if (tri ? ks >= 70 || (ks >= 48 && ks % 8 == 0)
            : ks >= 17 && tiles * ks >= 0.97 * kSplitTargets[t])
      break;
  }
  return ti;
}

// Kernel choice for a GEMM shape: variant (low 4 bits: 0 vector-FMA 64 x 64,
// 1 MFMA 64 x 64, 2 MFMA 128-wide, 3 and 4 the same with clamped loads, 5
// MFMA 64 x 64 x 32 with clamped loads, 6 the small-product kernel, 7 and 8
// complex64 MFMA 96 x 64 and 96 x 32) and split-K target (bits 4-5, index into
// kSplitTargets). The small-product kernel
// is a candidate for op(A) in {N, C}, B not transposed and up to kSmallTiles
// tiles and kSmallWork products, in complex64 and, where the caller asks (`small`), in complex128.
// Every other complex128 product has the split of fixed_split_target, and only
// the MFMA kernels that cut K into the same slices (and so add in the same order)
// are candidates. Chosen once per (precision, ops, m, n, k) by timing every
// distinct launch into a scratch output (HIP events, context stream);
// outside a stream capture only, otherwise the MFMA 64 x 64 default.
template <typename T>
static int gemm_variant(chs_context* ctx, int oa, int ob, int m, int n, int k, const cplx<T>* A,
                        int lda, const cplx<T>* B, int ldb, int* choice, int tri = 0,
                        bool small = false) {
  auto* im = ctx->impl;
  if (!im->use_mfma) {
    *choice = 0;
    return CHS_OK;
  }
  if (im->gemm_choice >= 0) {
    *choice = im->gemm_choice;
    return CHS_OK;
  }
  const GemmKey key{(int)sizeof(T), oa, ob + 16 * tri + (small && sizeof(T) == 8 ? 32 : 0), m, n, k};
  auto it = im->gemm_tune.find(key);
  if (it != im->gemm_tune.end()) {
    *choice = it->second;
    return CHS_OK;
  }
  const bool fixed = sizeof(T) == 8 && !small;
  const int fixed_ti = fixed ? fixed_split_target(m, n, k, tri != 0) : 0;
  *choice = 1 | (fixed_ti << 4);
  int fixed_ks = 0, fixed_kl = 0;
  if (fixed) variant_plan<T>(1, m, n, k, kSplitTargets[fixed_ti], tri, &fixed_ks, &fixed_kl);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  CHS_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
  if (cs != hipStreamCaptureStatusNone || !im->gemm_autotune) return CHS_OK;
  CHS_TRY(ensure(ctx, im->gemm_tune_c, (size_t)m * n * sizeof(cplx<T>)));
  cplx<T>* Ct = (cplx<T>*)im->gemm_tune_c.p;
  const cplx<T> one = mk((T)1, (T)0), zero = mk((T)0, (T)0);
  double best = 1e300;
  // the vector-FMA kernel never wins a large product: not timed there
  const bool big = (double)m * n * k > 1e9;
  const bool sm = (small || sizeof(T) == 4) && oa != 1 && ob == 0 && !tri &&
                  (int)(ceil_div(m, kSM) * ceil_div(n, kSM)) <= kSmallTiles &&
                  (double)m * n * k <= kSmallWork;
  const bool c64nn = sizeof(T) == 4 && oa != 1 && ob == 0 && !tri;
  auto padded = [](int x, int tile) { return (x + tile - 1) / tile * tile; };
  for (int v = big || fixed ? 1 : 0; v < 9; ++v) {
    if (v == 6 && !sm) continue;
    // 96-row tiles where they pad the rows no more than 64-row ones, 32-column
    // tiles where they pad the columns less
    if (v == 7 && !(c64nn && big && padded(m, 96) <= padded(m, 64))) continue;
    if (v == 8 && !(c64nn && padded(n, 32) < padded(n, 64))) continue;
    int prev_split = -1;
    for (int ti = 0; ti < kNumSplitTargets; ++ti) {
      int ks, kl;
      variant_plan<T>(v, m, n, k, kSplitTargets[ti], tri, &ks, &kl);
      if (fixed && (ti != fixed_ti || ks != fixed_ks || (ks > 1 && kl != fixed_kl))) continue;
      // complex64 sums run at most kMaxChain products before the slices are
      // added, unless no target cuts K that far
      if (sizeof(T) == 4 && kl > kMaxChain && ti + 1 < kNumSplitTargets) continue;
      if (ks == prev_split) continue;  // same launch as a smaller target
      prev_split = ks;
      const int c = v | (ti << 4);
      CHS_TRY(gemm_launch<T>(ctx, c, oa, ob, m, n, k, one, A, lda, B, ldb, zero, Ct, m,
                             im->gemm_tune_ws, tri));  // warm-up, workspace growth
      // best of three launches: candidates a few percent apart must not be
      // ranked by one launch's noise
      float t = 1e30f;
      for (int rep = 0; rep < 3; ++rep) {
        CHS_HIP(ctx, hipEventRecord(im->ev0, ctx->stream));
        CHS_TRY(gemm_launch<T>(ctx, c, oa, ob, m, n, k, one, A, lda, B, ldb, zero, Ct, m,
                               im->gemm_tune_ws, tri));
        CHS_HIP(ctx, hipEventRecord(im->ev1, ctx->stream));
        CHS_HIP(ctx, hipEventSynchronize(im->ev1));
        float tr = 0;
        CHS_HIP(ctx, hipEventElapsedTime(&tr, im->ev0, im->ev1));
        t = std::min(t, tr);
        if (t > 1.25 * best) break;  // far behind: not timed again
      }
      if (t < best) {
        best = t;
        *choice = c;
      }
    }
  }
  im->gemm_tune[key] = *choice;
  tune_cache_store(ctx, "gemm " + std::to_string(key.tsize) + " " + std::to_string(key.oa) + " " +
                            std::to_string(key.ob) + " " + std::to_string(m) + " " +
                            std::to_string(n) + " " + std::to_string(k) + " " +
                            std::to_string(*choice));
  return CHS_OK;
}

template <typename T>
static int gemm_t(chs_context* ctx, char opa, char opb, int m, int n, int k, cplx<T> alpha,
                  const cplx<T>* A, int lda, const cplx<T>* B, int ldb, cplx<T> beta, cplx<T>* C,
                  int ldc, bool small = false) {
  const int oa = gemm_opcode(opa), ob = gemm_opcode(opb);
  if (oa < 0 || ob < 0 || m < 0 || n < 0 || k < 0) return CHS_ERR_INVALID_ARG;
  if (m == 0 || n == 0) return CHS_OK;
  if (n == 1 && ob == 0 && k > 0)  // matrix-vector
    return gemv_launch<T>(ctx, oa, m, k, alpha, A, lda, B, beta, C);
  int choice = 1;
  CHS_TRY(gemm_variant<T>(ctx, oa, ob, m, n, k, A, lda, B, ldb, &choice, 0, small));
  return gemm_launch<T>(ctx, choice, oa, ob, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                        ctx->impl->gemm_ws);
}

int zgemm(chs_context* ctx, char opa, char opb, int m, int n, int k, z64 alpha, const z64* A,
          int lda, const z64* B, int ldb, z64 beta, z64* C, int ldc) {
  return gemm_t<double>(ctx, opa, opb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

int zgemm_small(chs_context* ctx, char opa, char opb, int m, int n, int k, z64 alpha, const z64* A,
                int lda, const z64* B, int ldb, z64 beta, z64* C, int ldc) {
  return gemm_t<double>(ctx, opa, opb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, true);
}

// C[i][j] = conj(C[j][i]) for i > j
__global__ void k_mirror_lower(z64* __restrict__ C, int n, int ldc) {
  const int i = blockIdx.x * 16 + (threadIdx.x & 15), j = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (i < n && j < i) C[(size_t)i + (size_t)j * ldc] = conj(C[(size_t)j + (size_t)i * ldc]);
}

int zgemm_herm(chs_context* ctx, int n, int k, const z64* A, int lda, const z64* B, int ldb, z64* C,
               int ldc) {
  const z64 one = mk(1.0, 0.0), zero = mk(0.0, 0.0);
  if (n < 128 || k <= 0 || !ctx->impl->use_mfma)
    return gemm_t<double>(ctx, 'C', 'N', n, n, k, one, A, lda, B, ldb, zero, C, ldc);
  int choice = 1;
  CHS_TRY(gemm_variant<double>(ctx, 2, 0, n, n, k, A, lda, B, ldb, &choice, 1));
  CHS_TRY(gemm_launch<double>(ctx, choice, 2, 0, n, n, k, one, A, lda, B, ldb, zero, C, ldc,
                              ctx->impl->gemm_ws, 1));
  hipLaunchKernelGGL(k_mirror_lower, dim3(ceil_div(n, 16), ceil_div(n, 16)), dim3(256), 0,
                     ctx->stream, C, n, ldc);
  CHS_LAUNCH_CHECK(ctx);
  return CHS_OK;
}

int cgemm(chs_context* ctx, char opa, char opb, int m, int n, int k, c32 alpha, const c32* A,
          int lda, const c32* B, int ldb, c32 beta, c32* C, int ldc) {
  return gemm_t<float>(ctx, opa, opb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

int zgemv_c32(chs_context* ctx, char opa, int m, int k, z64 alpha, const c32* A, int lda,
              const z64* x, z64 beta, z64* y) {
  const int oa = gemm_opcode(opa);
  if (oa < 0 || m < 0 || k < 1) return CHS_ERR_INVALID_ARG;
  if (m == 0) return CHS_OK;
  return gemv_launch<double, float>(ctx, oa, m, k, alpha, A, lda, x, beta, y);
}

}  // namespace chs

using namespace chs;

extern "C" int chs_zgemm(chs_context* ctx, char opa, char opb, int m, int n, int k,
                         const double alpha[2], const double* d_a, int lda, const double* d_b,
                         int ldb, const double beta[2], double* d_c, int ldc) {
  if (!ctx || !alpha || !beta || (m > 0 && n > 0 && (!d_c || (k > 0 && (!d_a || !d_b)))))
    return CHS_ERR_INVALID_ARG;
  const int oa = gemm_opcode(opa), ob = gemm_opcode(opb);
  if (oa < 0 || ob < 0 || m < 0 || n < 0 || k < 0) return CHS_ERR_INVALID_ARG;
  if (ldc < std::max(1, m) || lda < std::max(1, oa == 0 ? m : k) ||
      ldb < std::max(1, ob == 0 ? k : n))
    return set_error(ctx, CHS_ERR_INVALID_ARG, "zgemm: leading dimension too small");
  return zgemm(ctx, opa, opb, m, n, k, mk(alpha[0], alpha[1]), (const z64*)d_a, lda,
               (const z64*)d_b, ldb, mk(beta[0], beta[1]), (z64*)d_c, ldc);
}

// Synthetic operands for timing (values in [-0.005, 0.005)).
__global__ void k_gemm_fill(float* __restrict__ a, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    uint32_t h = (uint32_t)i * 2654435761u;
    h ^= h >> 15;
    a[i] = ((float)(h & 0xFFFF) / 65536.0f - 0.5f) * 1e-2f;
  }
}

extern "C" int chs_cgemm(chs_context* ctx, char opa, char opb, int m, int n, int k,
                         const float alpha[2], const float* d_a, int lda, const float* d_b, int ldb,
                         const float beta[2], float* d_c, int ldc) {
  if (!ctx || !alpha || !beta || (m > 0 && n > 0 && (!d_c || (k > 0 && (!d_a || !d_b)))))
    return CHS_ERR_INVALID_ARG;
  const int oa = gemm_opcode(opa), ob = gemm_opcode(opb);
  if (oa < 0 || ob < 0 || m < 0 || n < 0 || k < 0) return CHS_ERR_INVALID_ARG;
  if (ldc < std::max(1, m) || lda < std::max(1, oa == 0 ? m : k) ||
      ldb < std::max(1, ob == 0 ? k : n))
    return set_error(ctx, CHS_ERR_INVALID_ARG, "cgemm: leading dimension too small");
  return cgemm(ctx, opa, opb, m, n, k, mk(alpha[0], alpha[1]), (const c32*)d_a, lda,
               (const c32*)d_b, ldb, mk(beta[0], beta[1]), (c32*)d_c, ldc);
}

// Mean duration (HIP events on the context stream) of `reps` complex GEMMs
// C = A B (op(A) m x k, op(B) k x n) on synthetic operands.
extern "C" int chs_profile_gemm(chs_context* ctx, int precision, char opa, char opb, int m, int n,
                                int k, int reps, double* ms) {
  if (!ctx || !ms || m <= 0 || n <= 0 || k <= 0 || reps <= 0 ||
      (precision != CHS_C128 && precision != CHS_C64))
    return CHS_ERR_INVALID_ARG;
  const int oa = gemm_opcode(opa), ob = gemm_opcode(opb);
  if (oa < 0 || ob < 0) return CHS_ERR_INVALID_ARG;
  auto* im = ctx->impl;
  const size_t cs = precision == CHS_C128 ? 16 : 8;
  const size_t na = (size_t)m * k, nb = (size_t)k * n, nc = (size_t)m * n;
  CHS_TRY(ensure(ctx, im->ws1, na * cs));
  CHS_TRY(ensure(ctx, im->ws2, nb * cs));
  CHS_TRY(ensure(ctx, im->ws3, nc * cs));
  for (auto pr : {std::make_pair(im->ws1.p, na), std::make_pair(im->ws2.p, nb)}) {
    const size_t nf = pr.second * cs / sizeof(float);
    hipLaunchKernelGGL(k_gemm_fill, dim3(ceil_div(nf, 256)), dim3(256), 0, ctx->stream,
                       (float*)pr.first, nf);
  }
  CHS_LAUNCH_CHECK(ctx);
  const int lda = oa == 0 ? m : k, ldb = ob == 0 ? k : n;
  auto run = [&]() -> int {
    if (precision == CHS_C128)
      return zgemm(ctx, opa, opb, m, n, k, mk(1.0, 0.0), (const z64*)im->ws1.p, lda,
                   (const z64*)im->ws2.p, ldb, mk(0.0, 0.0), (z64*)im->ws3.p, m);
    return cgemm(ctx, opa, opb, m, n, k, mk(1.0f, 0.0f), (const c32*)im->ws1.p, lda,
                 (const c32*)im->ws2.p, ldb, mk(0.0f, 0.0f), (c32*)im->ws3.p, m);
  };
  CHS_TRY(run());  // warm-up (workspace growth happens here)
  CHS_HIP(ctx, hipEventRecord(im->ev0, ctx->stream));
  for (int r = 0; r < reps; ++r) CHS_TRY(run());
  CHS_HIP(ctx, hipEventRecord(im->ev1, ctx->stream));
  CHS_HIP(ctx, hipEventSynchronize(im->ev1));
  float t = 0;
  CHS_HIP(ctx, hipEventElapsedTime(&t, im->ev0, im->ev1));
  *ms = t / reps;
  return CHS_OK;
}
