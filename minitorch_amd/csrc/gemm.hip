// Strided-batched fp32 GEMM on gfx950 MFMA (v_mfma_f32_16x16x4_f32).
//
// Replaces the reference's Tensor.__matmul__ (tensor.py:207-223) forward and
// both backward products (dA = dC @ B^T, dB = A^T @ dC, via strides: a
// transpose is a stride swap, never a copy) and the Linear layer's x @ W + b
// (layers.py:31-37, bias fused into the epilogue).
//
//   C[b] = alpha * A[b] @ B[b] + beta * C[b] + bias      (bias indexed by n)
//
// Every operand is (rows, cols) with a row stride, a column stride and a batch
// stride (batch stride 0 broadcasts).  One of A's strides and one of B's must
// be 1 (the loader vectorises along it); the wrapper copies otherwise.
//
// Tiling: 256 threads = 4 waves in a 2x2 grid; block tile BM x BN x 16, each
// wave (BM/2) x (BN/2) built from 16x16 MFMA tiles.  The next k-tile is
// prefetched into registers while the current one is multiplied out of LDS.
// Large-K, small-MN products (weight gradients: K = B*T) are split over K:
// each split writes an fp32 partial tile into the caller's workspace and a
// second kernel sums the partials in a fixed order (deterministic), applying
// alpha, beta and bias.
#include "mtx_common.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace mtx {
namespace {

constexpr int kGT = 256;  // threads per GEMM workgroup
#ifndef MTX_GEMM_BK
#define MTX_GEMM_BK 16
#endif
constexpr int BK = MTX_GEMM_BK;  // k-tile depth of the tiled kernel
// split-K planning of long-K products: aim at about MTX_SPLIT_TARGET
// workgroups, each with at least MTX_SPLIT_MINK of K (C2 weight gradients,
// K = 16384, summed over the four shapes of a layer: target 256 5.23 ms,
// 512 4.21, 768 3.98, 1024 4.04-4.08 per step)
#ifndef MTX_SPLIT_TARGET
#define MTX_SPLIT_TARGET 768
#endif
#ifndef MTX_SPLIT_MINK
#define MTX_SPLIT_MINK 256
#endif

struct GemmArgs {
  const float* a; int64_t sam, sak, sab;
  const float* b; int64_t sbk, sbn, sbb;
  float* c; int64_t scm, scn, scb;
  const float* bias;
  float* ws;          // split-K partials: [split][batch][M][N] contiguous
  int M, N, K, batch;
  int ksplit, kchunk; // K range of split s: [s*kchunk, min(K, (s+1)*kchunk))
  float alpha, beta;
  // A and B give 16-byte-aligned vectors along their unit-stride dimension
  // at every multiple of 4 (base, other strides and batch strides: set by
  // the host; enables the interior-tile loads)
  int vec_ok;
  // decode-step epilogue (skinny kernel only): act 1 = GELU (tanh form) on
  // the C columns; product columns [nc, N) go to the KV caches instead of C:
  // the first half to kc, the second to vc, at row lengths[m] - 1 of
  // sequence m (row stride cst, sequence stride csb, T rows)
  int act, nc;
  float* kc;
  float* vc;
  int64_t csb, cst;
  int cT;
  const int* lengths;
  // tiled-kernel activation epilogue (mtx_gemm_act_f32): act 1 = GELU, with
  // the pre-activation value also stored to aux when aux != null; act 2 =
  // multiply by GELU'(aux) (aux = the pre-activation read back); act 4 = add
  // aux (a residual stream)
  float* aux;
  int64_t sxm, sxn, sxb;
  // weight-gradient variant (mtx_gemm_wgrad_f32, batch 1): colsum[n] =
  // sum over k of B[k][n] (the bias gradient), added to colsum when
  // colsum_acc; with split K the per-split sums go to the workspace after the
  // C partials, [split][N], and the reduce adds them in split order
  float* colsum;
  int colsum_acc;
  // skinny kernel: write the partial product to ws even when K is not split
  // (the split-K entry points of one range, K <= 16)
  int to_ws;
  // tiled split kernel (set by the host): the two-piece form may be tried; C's
  // (or the partials') and aux's rows have unit stride and do not overlap
  int fast, rows_vec;
};

// the value stored at C[m][n] of batch b from the product's value v
__device__ __forceinline__ float epilogue(const GemmArgs& g, float v, int bidx, int m, int n) {
  if (g.act == 1) {
    if (g.aux) g.aux[(int64_t)bidx * g.sxb + (int64_t)m * g.sxm + (int64_t)n * g.sxn] = v;
    return gelu_tanh_fast(v);
  }
  if (g.act == 2) return v * gelu_grad_fast(g.aux[(int64_t)bidx * g.sxb + (int64_t)m * g.sxm + (int64_t)n * g.sxn]);
  if (g.act == 4) return v + g.aux[(int64_t)bidx * g.sxb + (int64_t)m * g.sxm + (int64_t)n * g.sxn];
  return v;
}

template <int BM, int BN, bool AK, bool BN1>
struct Tiles {
  // per-thread register staging of one k-tile
  static constexpr int A_VEC = BM * BK / 4 / kGT;  // float4 per thread
  static constexpr int B_VEC = BN * BK / 4 / kGT;
};

// Load one k-tile of A (BM x BK) into registers.
// AK: A is contiguous along k (sak == 1); else contiguous along m (sam == 1).
template <int BM, bool AK>
__device__ __forceinline__ void load_a(const GemmArgs& g, const float* __restrict__ A, int m0, int k0,
                                       int kend, f32x4 (&r)[BM * BK / 4 / kGT], int tid) {
  constexpr int NV = BM * BK / 4 / kGT;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * kGT;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (AK) {
      const int m = m0 + idx / (BK / 4), k = k0 + (idx % (BK / 4)) * 4;
      if (m < g.M) {
        const float* p = A + (int64_t)m * g.sam + k;
        if (k + 3 < kend && ((((uintptr_t)p) & 15u) == 0)) {
          v = *reinterpret_cast<const f32x4*>(p);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (k + j < kend) v[j] = p[j];
        }
      }
    } else {
      const int k = k0 + idx / (BM / 4), m = m0 + (idx % (BM / 4)) * 4;
      if (k < kend) {
        const float* p = A + (int64_t)k * g.sak + m;
        if (m + 3 < g.M && ((((uintptr_t)p) & 15u) == 0)) {
          v = *reinterpret_cast<const f32x4*>(p);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (m + j < g.M) v[j] = p[j];
        }
      }
    }
    r[i] = v;
  }
}

// LDS tiles are k-major, [BK][BM] (A) and [BK][BN] (B), unpadded; within row
// k the 16-float column blocks are XOR-permuted by tswz(k).  A wave's
// fragment read takes 16 consecutive columns from each of 4 consecutive
// rows, and the transposing scalar stores write 16 columns x 4 rows 4 apart:
// with the permutation both touch 64 distinct banks (a padded row of BM + 4
// floats gave the reads 4-way conflicts).  Needs BM, BN >= 64.
__device__ __forceinline__ int tswz(int k) { return ((k + (k >> 2)) & 3) << 4; }

template <int BM, bool AK>
__device__ __forceinline__ void store_a(float* __restrict__ As, const f32x4 (&r)[BM * BK / 4 / kGT], int tid) {
  constexpr int NV = BM * BK / 4 / kGT;
  static_assert(BM >= 64, "the LDS permutation spans 64 columns");
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * kGT;
    if constexpr (AK) {
      const int m = idx / (BK / 4), k = (idx % (BK / 4)) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) As[(k + j) * BM + (m ^ tswz(k + j))] = r[i][j];
    } else {
      const int k = idx / (BM / 4), m = (idx % (BM / 4)) * 4;
      *reinterpret_cast<f32x4*>(As + k * BM + (m ^ tswz(k))) = r[i];
    }
  }
}

// B tile (BK x BN).  BN1: B contiguous along n (sbn == 1); else along k.
template <int BN, bool BN1>
__device__ __forceinline__ void load_b(const GemmArgs& g, const float* __restrict__ Bp, int n0, int k0,
                                       int kend, f32x4 (&r)[BN * BK / 4 / kGT], int tid) {
  constexpr int NV = BN * BK / 4 / kGT;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * kGT;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (BN1) {
      const int k = k0 + idx / (BN / 4), n = n0 + (idx % (BN / 4)) * 4;
      if (k < kend) {
        const float* p = Bp + (int64_t)k * g.sbk + n;
        if (n + 3 < g.N && ((((uintptr_t)p) & 15u) == 0)) {
          v = *reinterpret_cast<const f32x4*>(p);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (n + j < g.N) v[j] = p[j];
        }
      }
    } else {
      const int n = n0 + idx / (BK / 4), k = k0 + (idx % (BK / 4)) * 4;
      if (n < g.N) {
        const float* p = Bp + (int64_t)n * g.sbn + k;
        if (k + 3 < kend && ((((uintptr_t)p) & 15u) == 0)) {
          v = *reinterpret_cast<const f32x4*>(p);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (k + j < kend) v[j] = p[j];
        }
      }
    }
    r[i] = v;
  }
}

template <int BN, bool BN1>
__device__ __forceinline__ void store_b(float* __restrict__ Bs, const f32x4 (&r)[BN * BK / 4 / kGT], int tid) {
  constexpr int NV = BN * BK / 4 / kGT;
  static_assert(BN >= 64, "the LDS permutation spans 64 columns");
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = tid + i * kGT;
    if constexpr (BN1) {
      const int k = idx / (BN / 4), n = (idx % (BN / 4)) * 4;
      *reinterpret_cast<f32x4*>(Bs + k * BN + (n ^ tswz(k))) = r[i];
    } else {
      const int n = idx / (BK / 4), k = (idx % (BK / 4)) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) Bs[(k + j) * BN + (n ^ tswz(k + j))] = r[i][j];
    }
  }
}

template <int BM, int BN, bool AK, bool BN1, int ACT>
__global__ __launch_bounds__(kGT) void gemm_f32_kernel(const GemmArgs g) {
  constexpr int WM = BM / 2, WN = BN / 2;  // wave tile
  constexpr int TM = WM / 16, TN = WN / 16;
  __shared__ __attribute__((aligned(16))) float As[BK * BM];
  __shared__ __attribute__((aligned(16))) float Bs[BK * BN];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int n16 = lane & 15, grp = lane >> 4;
  const int wm = (wid >> 1) * WM, wn = (wid & 1) * WN;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int zb = blockIdx.z;
  const int bidx = zb % g.batch, split = zb / g.batch;
  const int kbeg = split * g.kchunk;
  const int kend = min(g.K, kbeg + g.kchunk);

  const float* __restrict__ A = g.a + (int64_t)bidx * g.sab;
  const float* __restrict__ Bp = g.b + (int64_t)bidx * g.sbb;

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero4();
  // ACT 3: column sums of B from the values each lane feeds the MFMAs (lane
  // (grp, n16) sees B[k][wn + 16j + n16] for every k = grp mod 4)
  float csum[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) csum[j] = 0.f;
  // only the waves whose sums are stored (below) add them (wave-uniform)
  const bool cs_wave = blockIdx.y == 0 && __builtin_amdgcn_readfirstlane(wm) == 0;

  constexpr int AV = BM * BK / 4 / kGT, BV = BN * BK / 4 / kGT;
  f32x4 ra[AV], rb[BV];
  // Interior tiles (every row and column in range, 16-byte aligned vectors
  // checked on the host) load whole k tiles without per-element checks,
  // from per-thread offsets computed once; other tiles and the last partial
  // k tile take the checked loaders.
  const bool interior = g.vec_ok && m0 + BM <= g.M && n0 + BN <= g.N;
  int64_t aoff[AV], boff[BV];
#pragma unroll
  for (int i = 0; i < AV; ++i) {
    const int idx = tid + i * kGT;
    aoff[i] = AK ? (int64_t)(m0 + idx / (BK / 4)) * g.sam + (idx % (BK / 4)) * 4
                 : (int64_t)(idx / (BM / 4)) * g.sak + m0 + (idx % (BM / 4)) * 4;
  }
#pragma unroll
  for (int i = 0; i < BV; ++i) {
    const int idx = tid + i * kGT;
    boff[i] = BN1 ? (int64_t)(idx / (BN / 4)) * g.sbk + n0 + (idx % (BN / 4)) * 4
                  : (int64_t)(n0 + idx / (BK / 4)) * g.sbn + (idx % (BK / 4)) * 4;
  }
  const int64_t ak = AK ? 1 : g.sak, bk = BN1 ? g.sbk : 1;  // k stride of the offsets
  auto fetch = [&](int k0) {
    if (interior && k0 + BK <= kend) {
#pragma unroll
      for (int i = 0; i < AV; ++i) ra[i] = *reinterpret_cast<const f32x4*>(A + aoff[i] + (int64_t)k0 * ak);
#pragma unroll
      for (int i = 0; i < BV; ++i) rb[i] = *reinterpret_cast<const f32x4*>(Bp + boff[i] + (int64_t)k0 * bk);
    } else {
      load_a<BM, AK>(g, A, m0, k0, kend, ra, tid);
      load_b<BN, BN1>(g, Bp, n0, k0, kend, rb, tid);
    }
  };
  if (kbeg < kend) fetch(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    __syncthreads();
    store_a<BM, AK>(As, ra, tid);
    store_b<BN, BN1>(Bs, rb, tid);
    __syncthreads();
    if (k0 + BK < kend) fetch(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      float af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = As[(kk + grp) * BM + ((wm + 16 * i + n16) ^ tswz(kk + grp))];
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = Bs[(kk + grp) * BN + ((wn + 16 * j + n16) ^ tswz(kk + grp))];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j], acc[i][j], 0, 0, 0);
      if constexpr (ACT == 3) {
        if (cs_wave) {
#pragma unroll
          for (int j = 0; j < TN; ++j) csum[j] += bf[j];
        }
      }
    }
  }

  // ACT 3: the first row of tiles (its waves 0 and 1, which together cover
  // the BN columns) adds the four lane groups' sums and stores them
  if constexpr (ACT == 3) {
    if (cs_wave) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        float v = csum[j];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        const int n = n0 + wn + 16 * j + n16;
        if (grp == 0 && n < g.N) {
          if (g.ksplit > 1) {
            g.ws[(int64_t)g.ksplit * g.M * g.N + (int64_t)split * g.N + n] = v;
          } else {
            g.colsum[n] = g.colsum_acc ? g.colsum[n] + v : v;
          }
        }
      }
    }
  }

  // epilogue.  acc[i][j][r] = C[wm+16i+4grp+r][wn+16j+n16]
  if (g.ksplit > 1) {
    float* __restrict__ W = g.ws + ((int64_t)split * g.batch + bidx) * (int64_t)g.M * g.N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + 16 * j + n16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm + 16 * i + 4 * grp + r;
          if (m < g.M && n < g.N) W[(int64_t)m * g.N + n] = acc[i][j][r];
        }
      }
    return;
  }
  float* __restrict__ Cp = g.c + (int64_t)bidx * g.scb;
  // the activation is a template parameter, so the plain GEMMs keep their
  // register budget; the GELU-backward reads one tile row's pre-activations
  // (16 values) ahead of their use
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    float xa[TN][4];
    if constexpr (ACT == 2) {
      const float* __restrict__ X = g.aux + (int64_t)bidx * g.sxb;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = min(n0 + wn + 16 * j + n16, g.N - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = min(m0 + wm + 16 * i + 4 * grp + r, g.M - 1);
          xa[j][r] = X[(int64_t)m * g.sxm + (int64_t)n * g.sxn];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + 16 * j + n16;
      if (n >= g.N) continue;
      const float bv = g.bias ? g.bias[n] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * grp + r;
        if (m < g.M) {
          float* p = Cp + (int64_t)m * g.scm + (int64_t)n * g.scn;
          float v = g.alpha * acc[i][j][r] + bv;
          if (g.beta != 0.f) v += g.beta * *p;
          if constexpr (ACT == 1) {
            if (g.aux) g.aux[(int64_t)bidx * g.sxb + (int64_t)m * g.sxm + (int64_t)n * g.sxn] = v;
            v = gelu_tanh_fast(v);
          } else if constexpr (ACT == 2) {
            v *= gelu_grad_fast(xa[j][r]);
          } else if constexpr (ACT == 4) {
            v += g.aux[(int64_t)bidx * g.sxb + (int64_t)m * g.sxm + (int64_t)n * g.sxn];
          }
          *p = v;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// fp32 products on the bf16 matrix cores (the default for tiles of 128 x 128).
//
// Every fp32 operand value x is split into three bf16 pieces while its tile
// is staged into LDS: x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1)
// (each conversion rounds to nearest even; each difference is exact in fp32),
// so x = x0 + x1 + x2 + r with |r| <= 2^-24 |x|: the pieces carry x's 24-bit
// significand.  A product x*y is accumulated as the six piece products of
// weight >= 2^-16 (x2y0, x1y1, x0y2, x1y0, x0y1, x0y0, smallest first); the
// three dropped ones (x1y2, x2y1, x2y2) weigh at most ~2^-23 |xy| together.
// Each piece product is exact in fp32 and the matrix core adds it into the
// fp32 accumulator, so a dot product's error is the fp32 accumulation error
// (as with fp32 multiply-adds) plus at most ~2^-22 sum|x_k y_k|.  Six
// v_mfma_f32_32x32x16_bf16 (6 x 32 cycles) do the work of sixteen
// v_mfma_f32_16x16x4_f32 (16 x 32 cycles): 2.7x the fp32 matrix rate.
// Non-finite inputs give NaN (x - x0 is Inf - Inf).
//
// Two fp16 pieces do the same in three products where the values' range
// allows (h2 below), and this form stays as what those tiles fall back to and
// for short products.
//
// An operand contiguous along k is staged as [piece][row][k] (rows of 16
// bf16, the two 16-byte chunks swapped on rows 8..15 mod 16) and read with
// ds_read_b128; an operand contiguous along its rows (m or n) as
// [piece][k][row] (rows of R + pad bf16, a stride of 16 or 48 banks mod 64)
// and read with gfx950's transposing ds_read_b64_tr_b16, so staging never
// transposes in registers.  Both layouts are free of LDS bank conflicts.
// MFMA 32x32x16 operands: lane l holds row l%32 and k = 8(l/32) + 0..7;
// accumulator element e of lane l is C[8(e/4) + 4(l/32) + e%4][l%32].
// ---------------------------------------------------------------------------
namespace x3 {
constexpr int BK = 16;  // k-tile depth (one MFMA k step)
// k-contiguous rows hold two 16-byte chunks, swapped on rows 8..15 mod 16:
// a fragment read's 16 rows then cover 16 distinct 16-byte bank groups and
// a staging store's 8 rows x 4 quarters 32 distinct 8-byte ones
__device__ __forceinline__ int kswz(int row) { return ((row >> 3) & 1) * 8; }
}  // namespace x3

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// One operand's R x 16 tile (rows = m for A, n for B).  KC: contiguous along
// k in global memory (rows strided by srow); else contiguous along the rows
// (k strided by sk).  The tile is R*4 float4 vectors; slot i of a thread is
// vector idx = tid + 256 i: KC: row idx/4, k 4(idx%4)..+3; else: k idx/(R/4),
// rows 4(idx%(R/4))..+3.  Where 256 does not divide R*4 the threads past the
// end repeat the vector 128 before (the same values to the same place).
template <bool KC, int R>
struct X3Stage {
  static constexpr int NV = (R * 4 + kGT - 1) / kGT;  // float4 per thread
  static constexpr int NVEC = R * 4;
  static_assert(NVEC % kGT == 0 || NVEC % kGT == 128, "tile rows");
  // k-plane row stride (bf16): 16 or 48 banks mod 64
  static constexpr int LDR = (R / 2) % 64 == 16 || (R / 2) % 64 == 48 ? R : R + 32;
  static_assert((LDR / 2) % 64 == 16 || (LDR / 2) % 64 == 48, "bank stride");
  static constexpr int PS = KC ? R * x3::BK : x3::BK * LDR;  // plane size (bf16)
  const float* __restrict__ base;  // the operand at (row r0, k 0)
  int64_t srow, sk;
  int rows, r0;
  int lput[NV];  // LDS offsets (bf16) of this thread's vectors

  __device__ __forceinline__ int vec(int i, int tid) const {
    const int idx = tid + i * kGT;
    return idx < NVEC ? idx : idx - 128;
  }
  __device__ __forceinline__ void init(const float* b, int64_t s_row, int64_t s_k, int nrows, int row0, int tid) {
    srow = s_row;
    sk = s_k;
    rows = nrows;
    r0 = row0;
    base = b + (int64_t)r0 * srow;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = vec(i, tid);
      if constexpr (KC) {
        lput[i] = (idx / 4) * x3::BK + ((4 * (idx % 4)) ^ x3::kswz(idx / 4));
      } else {
        lput[i] = (idx / (R / 4)) * LDR + 4 * (idx % (R / 4));
      }
    }
  }
  // rows past `rows` and k past kend read as zero; unaligned vectors by element
  __device__ __forceinline__ void fetch_checked(f32x4 (&r)[NV], int k0, int kend, int tid) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = vec(i, tid);
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if constexpr (KC) {
        const int row = idx / 4, k = k0 + 4 * (idx % 4);
        if (r0 + row < rows) {
          const float* p = base + (int64_t)row * srow + k;
          if (k + 3 < kend && (((uintptr_t)p) & 15u) == 0) {
            v = *reinterpret_cast<const f32x4*>(p);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (k + j < kend) v[j] = p[j];
          }
        }
      } else {
        const int k = k0 + idx / (R / 4), row = 4 * (idx % (R / 4));
        if (k < kend) {
          const float* p = base + (int64_t)k * sk + row;
          if (r0 + row + 3 < rows && (((uintptr_t)p) & 15u) == 0) {
            v = *reinterpret_cast<const f32x4*>(p);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (r0 + row + j < rows) v[j] = p[j];
          }
        }
      }
      r[i] = v;
    }
  }
  __device__ __forceinline__ void put(__bf16* __restrict__ lds, const f32x4 (&r)[NV]) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      uint2 h, m, l;
      split3(r[i], h, m, l);
      *reinterpret_cast<uint2*>(lds + lput[i]) = h;
      *reinterpret_cast<uint2*>(lds + PS + lput[i]) = m;
      *reinterpret_cast<uint2*>(lds + 2 * PS + lput[i]) = l;
    }
  }
  // piece p's MFMA operand for tile rows rb .. rb+31: lane l gets row
  // rb + l%32 and k = 8(l/32) + 0..7
  __device__ __forceinline__ static bf16x8 frag(const __bf16* __restrict__ lds, int p, int rb, int lane) {
    if constexpr (KC) {
      const int row = rb + (lane & 31);
      return *reinterpret_cast<const bf16x8*>(lds + p * PS + row * x3::BK + ((8 * (lane >> 5)) ^ x3::kswz(row)));
    } else {
      // transposing read: in each 16-lane group G, lane j = 4i + q addresses
      // k row 8(G/2) + i (+4 for the second half) at rows rb + 16(G%2) + 4q;
      // lane j then receives row rb + 16(G%2) + j at those four k
      const int G = lane >> 4, j = lane & 15;
      const __bf16* p0 = lds + p * PS + (8 * (G >> 1) + (j >> 2)) * LDR + rb + 16 * (G & 1) + 4 * (j & 3);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p0 + 4 * LDR));
      const uint2 ul = __builtin_bit_cast(uint2, lo), uh = __builtin_bit_cast(uint2, hi);
      return __builtin_bit_cast(bf16x8, make_uint4(ul.x, ul.y, uh.x, uh.y));
    }
  }
  // ACT 3 column sums: this thread's share of the staged B values, by
  // column (KC: the 4 k of slot i belong to column idx/4; else slot i holds
  // columns 4(idx%(R/4))..+3, the same for every slot; R = 128)
  __device__ __forceinline__ static void colsum_add(float (&cs)[4], const f32x4 (&r)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if constexpr (KC) {
        cs[i] += (r[i][0] + r[i][1]) + (r[i][2] + r[i][3]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) cs[j] += r[i][j];
      }
    }
  }
};

// ---------------------------------------------------------------------------
// fp32 products from two fp16 pieces of every value, three products each.
//
// A row of A (a column of B) is scaled by a power of two s, then every value
// x is split while its tile is staged into LDS: h = fp16(s x) and
// l = fp16(2^14 (s x - h)), both rounded to nearest, so that s x = h +
// 2^-14 l with an error of at most 2^-23 |s x|, or 2^-39 where that is more.
// C is (sum ah bh + 2^-14 sum (al bh + ah bl)) / (sa sb): the cross terms
// have accumulators of their own, and the dropped al bl weighs at most
// 2^-24 |ab|.  Three v_mfma_f32_32x32x16_f16 do the work of the three-piece
// split's six bf16 ones, and the main accumulator is rounded once per k step
// instead of six times, which is most of a long product's error: against
// float64 the products of the 384-wide model's training step are off by
// 0.5-0.6 of what the three-piece form gave (K = 384: 6.2e-8 against 1.1e-7
// relative; K = 1536: 2.6e-7 against 6.0e-7).
//
// The scale comes from 32 of the row's values, spread evenly over its k range
// (the beginning alone says too little: in the gradient of a packed q/k/v
// projection a first token's row starts with the query's, which is 0 up to
// rounding).  Their largest goes to [2^-4, 2^-3), so the error above is 2^-35
// of it for small values, and other values may be 2^17 times larger before l
// overflows (65504).  A row without a nonzero sample gets the largest scale,
// which any value above 2^-99 overflows; a largest sample outside 2^-60 ..
// 2^60 or not finite gives a scale of Inf.  An overflow leaves Inf or NaN in
// the accumulators of its whole row or column, so one look at them after the
// k loop finds it, and the workgroup then computes its tile again from three
// bf16 pieces (X3Stage), whose range is fp32's.
//
// Tiling: 256 threads = 4 waves; a wave owns MI x NI MFMA tiles of 32 x 32
// and the waves form a WM x WN grid, so the block tile is 32 MI WM x 32 NI
// WN, and 32 deep.  Pipeline: two LDS buffers and one barrier per k step.
// While the products of step t run out of one buffer, the wave splits the
// values of step t + 1 (in registers since the step before) into the other
// buffer and requests those of step t + 2 into the registers as they come
// free: each MFMA occupies the matrix pipe for 32 cycles and the issue port
// for 4, and the split's vector instructions are placed into the gaps
// (sched_group_barrier).
//
// Two workgroups fit a CU, and a launch has no more than fill the chip: each
// takes its tiles one after another, and the pipeline runs on across them
// (the last two steps of a tile request and stage the next one's first two,
// scaled by samples that were read during the epilogue before).  With a
// workgroup per tile every tile began with three exposed round trips to
// memory (samples, first and second step), all 512 resident ones at the same
// time: 16384 x 1536 products took 57-64 us plus 4.1-4.6 us per 32 of K.
// ---------------------------------------------------------------------------
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

namespace h2 {
constexpr int BK = 32;  // k-tile depth: a row's 32 floats are one 128-byte line
// From K = 256 on the error is no larger than the three-piece form's (of a
// shorter product the split's own 6e-8 is most)
constexpr int MINK = 256;

// the scale times 2^14 of a row whose largest |sample| has these bits, and the reciprocal of the scale itself
__device__ __forceinline__ float scale2(uint32_t amax) {
  const int e = (int)(amax >> 23);
  if (amax == 0) return __uint_as_float(254u << 23);
  if (e < 127 - 60 || e > 127 + 60) return __uint_as_float(0x7f800000u);
  return __uint_as_float((uint32_t)(127 + 127 + 14 - 4 - e) << 23);
}
__device__ __forceinline__ float unscale(uint32_t amax) {
  const int e = (int)(amax >> 23);
  if (amax == 0) return __uint_as_float(14u << 23);
  return __uint_as_float((uint32_t)(e + 4) << 23);
}
// x2 = 2^14 s x of four values -> h and l, four fp16 each: two mixed-precision
// multiply-adds a value (zero is a 0 that the compiler cannot see, and the
// pairs are opaque to it: it would otherwise convert every h twice)
__device__ __forceinline__ uint32_t pair_h(float x, float y, float zero) {
  f16x2 h = {(_Float16)__builtin_fmaf(x, 0x1p-14f, zero), (_Float16)__builtin_fmaf(y, 0x1p-14f, zero)};
  uint32_t u = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(u));
  return u;
}
__device__ __forceinline__ uint32_t pair_l(uint32_t hu, float x, float y) {
  const f16x2 h = __builtin_bit_cast(f16x2, hu);
  f16x2 l = {(_Float16)__builtin_fmaf((float)h[0], -16384.f, x), (_Float16)__builtin_fmaf((float)h[1], -16384.f, y)};
  return __builtin_bit_cast(uint32_t, l);
}
__device__ __forceinline__ void split(f32x4 x2, float zero, uint2& h, uint2& l) {
  h.x = pair_h(x2[0], x2[1], zero);
  h.y = pair_h(x2[2], x2[3], zero);
  l.x = pair_l(h.x, x2[0], x2[1]);
  l.y = pair_l(h.y, x2[2], x2[3]);
}
}  // namespace h2

// One operand's R x 32 tile (rows = m for A, n for B), R = 64 (KC), 96 or
// 128.  KC: contiguous along k in global memory (rows strided by srow); else
// contiguous along the rows (k strided by sk).  Slot i of a thread is the
// float4 vector idx = tid + 256 i: KC: row idx/8, k 4(idx%8)..+3; else: k
// idx/(R/4), rows 4(idx%(R/4))..+3.
// LDS planes.  KC: [row][32 k], rows of 64 bytes, the four 16-byte chunks
// permuted by (row/4)%4, so the 16 rows of a fragment read's quarter cover
// all 64 banks.  Else [k][R rows]: the transposing read takes 32 bytes of
// four consecutive k rows per 16 lanes; R = 96 (48 banks a row) spreads them
// by itself, R = 128 permutes the four 64-byte blocks of a row by k%4.
template <bool KC, int R>
struct H2Stage {
  static_assert(R == 96 || R == 128 || (KC && R == 64), "tile rows");
  static constexpr int NV = R * h2::BK / 4 / kGT;              // float4 per thread
  static constexpr int NQ = 2;                                 // sample vectors per thread
  static constexpr int PS = R * h2::BK;                        // plane size (fp16)
  static constexpr int NSC = KC ? NV : R == 128 ? 4 : 4 * NV;  // scales a thread needs
  static constexpr bool kEach = !KC && R == 96;                // slots do not lie a constant apart
  int64_t kstep;      // bytes per k
  uint32_t sstep;     // bytes per row (KC) or k (else)
  uint32_t voff[NV];  // this thread's byte offsets in a k-tile
  int lput[kEach ? NV : 1];
  float sc[NSC];
  // a tile's place: the operand at (its first row, its first k), and the
  // bytes from there to the operand's end; uniform
  struct Src {
    const char* base;
    int64_t left;
  };

  __device__ __forceinline__ void init(int64_t srow, int64_t sk, int tid) {
    kstep = sk * 4;
    sstep = (uint32_t)((KC ? srow : sk) * 4);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * kGT;
      voff[i] = KC ? (uint32_t)(idx / 8) * sstep + 16 * (idx % 8)
                   : (uint32_t)(idx / (R / 4)) * sstep + 16 * (idx % (R / 4));
      if constexpr (kEach) lput[i] = idx * 4;
    }
    if constexpr (KC) {
      const int row = tid / 8, c = (tid % 8) / 2;
      lput[0] = row * h2::BK + 8 * (c ^ ((row >> 2) & 3)) + 4 * (tid & 1);
    } else if constexpr (R == 128) {
      const int k = tid / 32, c = 4 * (tid % 32);
      lput[0] = k * R + (c ^ (32 * (k & 3)));
    }
  }
  __device__ __forceinline__ Src at(const float* b, int64_t srow, int64_t sk, int rows, int K, int r0, int k0) const {
    return {reinterpret_cast<const char*>(b + (int64_t)r0 * srow + (int64_t)k0 * sk),
            ((int64_t)(rows - 1 - r0) * srow + (int64_t)(K - 1 - k0) * sk + 1) * 4};
  }
  __device__ __forceinline__ int put_at(int i) const {
    if constexpr (KC) return lput[0] + i * 32 * h2::BK;       // 32 rows on: the same permutation
    else if constexpr (R == 128) return lput[0] + i * 8 * R;  // 8 k on
    else return lput[i];
  }
  // The k-tile k values from s on, through a buffer resource based at its
  // first value and ending at the operand's last: no per-lane address
  // arithmetic, and rows past the operand's end read as zeros.  (A vector
  // reaching past a row's last value takes what follows it in memory, which
  // the caller allows for rows only: their products land in rows or columns
  // of C that are not stored.)
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t tile(const Src& s, int k) const {
    const int64_t off = (int64_t)k * kstep, left = s.left - off;
    const int hi = (int)(left >> 32);
    const uint32_t bytes = hi < 0 ? 0u : hi > 0 ? 0xfffffff0u : (uint32_t)left;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(s.base + off), (short)0, (int)bytes, 0x00020000);
  }
  __device__ __forceinline__ f32x4 fetch(__amdgpu_buffer_rsrc_t rs, int i) const {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)voff[i], 0, 0));
  }
  // the same by element where a vector may reach past the last row or k
  __device__ __forceinline__ f32x4 fetch_checked(const Src& s, int k0, int n, int nrows, int i, int tid) const {
    const int idx = tid + i * kGT;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    const int row = KC ? idx / 8 : 4 * (idx % (R / 4)), k = k0 + (KC ? 4 * (idx % 8) : idx / (R / 4));
    const float* p = reinterpret_cast<const float*>(s.base + (int64_t)(KC ? row : k) * sstep) + (KC ? k : row);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (row + (KC ? 0 : j) < nrows && k + (KC ? j : 0) < n) v[j] = p[j];
    return v;
  }
  // 16 values of each row, spread evenly over the tile's n k (n >= 256): KC:
  // four vectors, at 0, 1/3, 2/3 and the end; else 16 k rows.  Thread vector
  // i is idx = tid + 256 i (repeating those 128 before where that is past the
  // tile's R*4): KC: row idx/4, place idx%4; else place idx/(R/4).
  __device__ __forceinline__ static int qvec(int i, int tid) {
    const int idx = tid + i * kGT;
    return idx < R * 4 ? idx : idx - (R == 64 ? 256 : 128);
  }
  __device__ __forceinline__ void sample(f32x4 (&q)[NQ], const Src& s, int n, int tid) const {
    const __amdgpu_buffer_rsrc_t rs = tile(s, 0);
    const uint32_t far = KC ? (uint32_t)((n - 4) / 3) * 4u : (uint32_t)((n - 1) / 15) * sstep;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int idx = qvec(i, tid);
      const uint32_t off = KC ? (uint32_t)(idx / 4) * sstep + (uint32_t)(idx % 4) * far
                              : (uint32_t)(idx / (R / 4)) * far + 16 * (idx % (R / 4));
      q[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
    }
  }
  // amax[row] = the largest of each row's samples (as bits); it is zero before
  __device__ __forceinline__ static void row_max(const f32x4 (&q)[NQ], uint32_t* amax, int tid) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int idx = qvec(i, tid);
      if constexpr (KC) {
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) m = max(m, __float_as_uint(q[i][j]) & 0x7fffffffu);
        m = max(m, (uint32_t)__shfl_xor((int)m, 1));
        m = max(m, (uint32_t)__shfl_xor((int)m, 2));
        if ((tid & 3) == 0) amax[idx / 4] = m;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          atomicMax(&amax[4 * (idx % (R / 4)) + j], __float_as_uint(q[i][j]) & 0x7fffffffu);
      }
    }
  }
  __device__ __forceinline__ void scales(const uint32_t* amax, int tid) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * kGT;
      if constexpr (KC) {
        sc[i] = h2::scale2(amax[idx / 8]);
      } else if (R != 128 || i == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[4 * i + j] = h2::scale2(amax[4 * (idx % (R / 4)) + j]);
      }
    }
  }
  __device__ __forceinline__ void put(_Float16* __restrict__ lds, f32x4 r, float zero, int i) const {
    f32x4 x2;
#pragma unroll
    for (int j = 0; j < 4; ++j) x2[j] = r[j] * sc[KC ? i : R == 128 ? j : 4 * i + j];
    uint2 h, l;
    h2::split(x2, zero, h, l);
    *reinterpret_cast<uint2*>(lds + put_at(i)) = h;
    *reinterpret_cast<uint2*>(lds + PS + put_at(i)) = l;
  }
  // piece p's MFMA operand for k 16 sub .. +15 of tile rows rb .. rb+31: lane
  // l gets row rb + l%32 and k = 16 sub + 8(l/32) + 0..7
  __device__ __forceinline__ static f16x8 frag(const _Float16* __restrict__ lds, int p, int sub, int rb, int lane) {
    if constexpr (KC) {
      const int row = rb + (lane & 31);
      return *reinterpret_cast<const f16x8*>(lds + p * PS + row * h2::BK +
                                             8 * ((2 * sub + (lane >> 5)) ^ ((row >> 2) & 3)));
    } else {
      // transposing read, as X3Stage::frag
      const int G = lane >> 4, j = lane & 15;
      const int k = 16 * sub + 8 * (G >> 1) + (j >> 2);
      int c = rb + 16 * (G & 1) + 4 * (j & 3);
      if constexpr (R == 128) c ^= 32 * (k & 3);
      const _Float16* p0 = lds + p * PS + k * R + c;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p0 + 4 * R));
      const uint2 ul = __builtin_bit_cast(uint2, lo), uh = __builtin_bit_cast(uint2, hi);
      return __builtin_bit_cast(f16x8, make_uint4(ul.x, ul.y, uh.x, uh.y));
    }
  }
};

// a thread or lane number whose uses are computed where they stand: code that
// runs once a tile or less otherwise keeps its addresses in registers across
// the k loop, which needs them all
__device__ __forceinline__ int here(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <int MI, int NI, int WM, int WN, bool AK, bool BN1, int ACT>
__global__ __launch_bounds__(kGT, 2) void gemm_x3_kernel(const GemmArgs g) {
  static_assert(WM * WN == 4, "four waves");
  constexpr int BM = 32 * MI * WM, BN = 32 * NI * WN;
  using SA = H2Stage<AK, BM>;
  using SB = H2Stage<!BN1, BN>;  // B^T: rows = n, contiguous along k iff !BN1
  using XA = X3Stage<AK, BM>;
  using XB = X3Stage<!BN1, BN>;
  constexpr int kBuf = 2 * (SA::PS + SB::PS);  // one stage's planes (fp16)
  constexpr int kX3 = 3 * (XA::PS + XB::PS) * 2;
  constexpr int kTiles = 2 * kBuf * 2 > kX3 ? 2 * kBuf * 2 : kX3;
  __shared__ __attribute__((aligned(16))) char smem[kTiles];
  __shared__ float red[ACT == 3 ? 8 * BN : 1];  // column sums
  // rows' and columns' largest sample of the tiles: one in its epilogue, one
  // being staged, one being sampled, one being cleared
  __shared__ __attribute__((aligned(16))) uint32_t amax[4][BM + BN];
  __shared__ int again;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wid / WN) * 32 * MI, wn = (wid % WN) * 32 * NI;

  // Workgroups are dealt round-robin over the 8 XCDs in dispatch order; each
  // XCD's take a contiguous run of row-major tiles, one after another, so the
  // column tiles that share an A row panel read it through the same L2
  const int gx = (g.N + BN - 1) / BN, gy = (g.M + BM - 1) / BM;
  int tile, tend;
  const int wgs = ((int)gridDim.x - (int)(blockIdx.x & 7) + 7) >> 3;  // this XCD's workgroups
  {
    const int nt = gx * gy * g.batch * g.ksplit;
    const int xcd = blockIdx.x & 7, per = nt >> 3, more = nt & 7;
    tile = xcd * per + min(xcd, more);
    tend = tile + per + (xcd < more ? 1 : 0);
    tile += blockIdx.x >> 3;
  }
  struct Place {
    int m0, n0, bidx, split, kbeg, n;
  };
  auto place = [&](int t) {
    Place p;
    p.n0 = t % gx * BN;
    p.m0 = t / gx % gy * BM;
    const int z = t / (gx * gy);
    p.bidx = z % g.batch;
    p.split = z / g.batch;
    p.kbeg = p.split * g.kchunk;
    p.n = min(g.K, p.kbeg + g.kchunk) - p.kbeg;
    return p;
  };
  if (tile >= tend) return;

  SA sa;
  SB sb;
  sa.init(g.sam, g.sak, tid);
  sb.init(g.sbn, g.sbk, tid);
  auto src_a = [&](const Place& p) {
    return sa.at(g.a + (int64_t)p.bidx * g.sab, g.sam, g.sak, g.M, g.K, p.m0, p.kbeg);
  };
  auto src_b = [&](const Place& p) {
    return sb.at(g.b + (int64_t)p.bidx * g.sbb, g.sbn, g.sbk, g.N, g.K, p.n0, p.kbeg);
  };

  f32x16 acc[MI][NI], accx[MI][NI];
  f32x4 ra[SA::NV], rb[SB::NV];
  // ACT 3: column sums of B from the values each thread stages
  float cs[SB::NV][4];
  float zero = 0.f;
  asm("" : "+s"(zero));
  int par = 0;  // the buffer that holds the step to multiply
  auto buf = [&](int b) { return reinterpret_cast<_Float16*>(smem) + b * kBuf; };

  auto colsum = [&] {
    if constexpr (ACT == 3) {
#pragma unroll
      for (int i = 0; i < SB::NV; ++i) {
        if constexpr (!BN1) cs[i][0] += (rb[i][0] + rb[i][1]) + (rb[i][2] + rb[i][3]);
        else
#pragma unroll
          for (int j = 0; j < 4; ++j) cs[0][j] += rb[i][j];
      }
    }
  };
  // the products of one step, MFMA by MFMA: half a step (sub) at a time the
  // four fragments' three products.  fa, fb: [sub][piece][tile].
  constexpr int kT = MI * NI, kM = 6 * kT;
  f16x8 fa[2][2][MI], fb[2][2][NI];
  auto read_frags = [&](const _Float16* cur, int sub, int p) {
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[sub][p][i] = SA::frag(cur, p, sub, wm + 32 * i, lane);
#pragma unroll
    for (int j = 0; j < NI; ++j) fb[sub][p][j] = SB::frag(cur + 2 * SA::PS, p, sub, wn + 32 * j, lane);
  };
  auto product = [&](int q) {
    const int sub = q / (3 * kT), kind = q / kT % 3, i = q % kT / NI, j = q % NI;
    if (kind == 0) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[sub][0][i], fb[sub][0][j], acc[i][j], 0, 0, 0);
    else if (kind == 1)
      accx[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[sub][1][i], fb[sub][0][j], accx[i][j], 0, 0, 0);
    else accx[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[sub][0][i], fb[sub][1][j], accx[i][j], 0, 0, 0);
  };
  // One step: its products in as many groups as there are vectors to stage
  // (kS); beside each group's products one vector of the next step is split
  // and stored, and its register refilled with the step after's (refill).
  constexpr int kS = SA::NV + SB::NV;
  auto step = [&](auto refill, __amdgpu_buffer_rsrc_t ta, __amdgpu_buffer_rsrc_t tb) {
    const _Float16* cur = buf(par);
    _Float16* nxt = buf(par ^ 1);
    read_frags(cur, 0, 0);
    read_frags(cur, 0, 1);
    colsum();
#pragma unroll
    for (int c = 0; c < kS; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      // the second half's fragments, as the first half's come free
      if (c == kS / 2 - 2) read_frags(cur, 1, 0);
      if (c == kS / 2 - 1) read_frags(cur, 1, 1);
#pragma unroll
      for (int q = c * kM / kS; q < (c + 1) * kM / kS; ++q) product(q);
      if (c < SA::NV) {
        sa.put(nxt, ra[c], zero, c);
        if constexpr (decltype(refill)::value) ra[c] = sa.fetch(ta, c);
      } else {
        sb.put(nxt + 2 * SA::PS, rb[c - SA::NV], zero, c - SA::NV);
        if constexpr (decltype(refill)::value) rb[c - SA::NV] = sb.fetch(tb, c - SA::NV);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (c == kS / 2 - 2 || c == kS / 2 - 1) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
      }
    }
    par ^= 1;
    __syncthreads();
  };

  Place cur = place(tile);
  bool primed = false;  // this tile's first step is staged, its second one in registers
  if (tid == 0) again = 0;
  for (int i = tid; i < 4 * (BM + BN); i += kGT) amax[0][i] = 0;
  if (g.fast) {
    f32x4 qa[2][SA::NQ], qb[2][SB::NQ];
    const bool more = tile + wgs < tend;
    const Place p1 = place(more ? tile + wgs : tile);
    sa.sample(qa[0], src_a(cur), cur.n, tid);
    sb.sample(qb[0], src_b(cur), cur.n, tid);
    sa.sample(qa[1], src_a(p1), p1.n, tid);
    sb.sample(qb[1], src_b(p1), p1.n, tid);
    __syncthreads();
    SA::row_max(qa[0], amax[0], tid);
    SB::row_max(qb[0], amax[0] + BM, tid);
    SA::row_max(qa[1], amax[1], tid);
    SB::row_max(qb[1], amax[1] + BM, tid);
    __syncthreads();
  }

  for (int seq = 0;; ++seq) {
    const bool more = tile + wgs < tend;
    const Place next = place(more ? tile + wgs : tile);
    bool scaled = false;  // acc, accx hold the two-piece sums
    float cso[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = accx[i][j][e] = 0.f;

    if (g.fast) {
      const typename SA::Src a0 = src_a(cur);
      const typename SB::Src b0 = src_b(cur);
      const int steps = (cur.n + h2::BK - 1) / h2::BK;
      // The k steps that the unchecked loads take: whole ones, and (where the
      // rows of an operand contiguous along them do not end on a vector) not
      // the operand's last, whose last vectors reach past its end.
      int whole = cur.n / h2::BK;
      if (((!AK && (g.M & 3)) || (BN1 && (g.N & 3))) && cur.kbeg + cur.n == g.K && whole == steps) --whole;
      for (int i = tid; i < BM + BN; i += kGT) amax[(seq + 2) & 3][i] = 0;
      if (!primed) {
        sa.scales(amax[seq & 3], tid);
        sb.scales(amax[seq & 3] + BM, tid);
        // (n >= 256: the first two steps are whole)
        auto ta = sa.tile(a0, 0);
        auto tb = sb.tile(b0, 0);
#pragma unroll
        for (int i = 0; i < SA::NV; ++i) ra[i] = sa.fetch(ta, i);
#pragma unroll
        for (int i = 0; i < SB::NV; ++i) rb[i] = sb.fetch(tb, i);
        if constexpr (ACT == 3) {
#pragma unroll
          for (int i = 0; i < SB::NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) cs[i][j] = 0.f;
        }
        colsum();
        ta = sa.tile(a0, h2::BK);
        tb = sb.tile(b0, h2::BK);
#pragma unroll
        for (int i = 0; i < SA::NV; ++i) {
          sa.put(buf(par), ra[i], zero, i);
          ra[i] = sa.fetch(ta, i);
        }
#pragma unroll
        for (int i = 0; i < SB::NV; ++i) {
          sb.put(buf(par) + 2 * SA::PS, rb[i], zero, i);
          rb[i] = sb.fetch(tb, i);
        }
        __syncthreads();
      }
      int t = 0;
      for (; t + 2 < whole; ++t)
        step(std::true_type{}, sa.tile(a0, (t + 2) * h2::BK), sb.tile(b0, (t + 2) * h2::BK));
      if (t + 2 < steps) {  // at most one step that is not whole
        step(std::false_type{}, sa.tile(a0, 0), sb.tile(b0, 0));
        ++t;
        const int tv = here(tid);
#pragma unroll
        for (int i = 0; i < SA::NV; ++i) ra[i] = sa.fetch_checked(a0, (t + 1) * h2::BK, cur.n, g.M - cur.m0, i, tv);
#pragma unroll
        for (int i = 0; i < SB::NV; ++i) rb[i] = sb.fetch_checked(b0, (t + 1) * h2::BK, cur.n, g.N - cur.n0, i, tv);
      }
      // the last two steps: request, then stage, the next tile's first two
      typename SA::Src a1 = src_a(next);
      typename SB::Src b1 = src_b(next);
      if (!more) a1.left = b1.left = 0;  // reads as zeros
      step(std::true_type{}, sa.tile(a1, 0), sb.tile(b1, 0));
      if constexpr (ACT == 3) {  // from here on the sums are the next tile's
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          cso[j] = BN1 ? cs[0][j] : cs[j % SB::NV][0];
          (BN1 ? cs[0][j] : cs[j % SB::NV][0]) = 0.f;
        }
      }
      sa.scales(amax[(seq + 1) & 3], tid);
      sb.scales(amax[(seq + 1) & 3] + BM, tid);
      step(std::true_type{}, sa.tile(a1, more ? h2::BK : 0), sb.tile(b1, more ? h2::BK : 0));
      primed = more;
      // Inf or NaN in a row or column of the tile: every row of the wave's
      // tile in its first column, every column in its first row
      float z = 0.f;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) z += 0.f * acc[i][0][e] + 0.f * accx[i][0][e];
#pragma unroll
      for (int j = 1; j < NI; ++j) z += 0.f * acc[0][j][0] + 0.f * accx[0][j][0];
      if (!(z == 0.f)) again = seq + 1;  // any lane
      __syncthreads();
      scaled = again != seq + 1;
    }

    if (!scaled) {
      primed = false;  // the buffers are used otherwise
      const int tv = here(tid), lv = tv & 63;
      XA xa;
      XB xb;
      xa.init(g.a + (int64_t)cur.bidx * g.sab, g.sam, g.sak, g.M, cur.m0, tv);
      xb.init(g.b + (int64_t)cur.bidx * g.sbb, g.sbn, g.sbk, g.N, cur.n0, tv);
      __bf16* As = reinterpret_cast<__bf16*>(smem);
      __bf16* Bs = As + 3 * XA::PS;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
      const bool sums = ACT == 3 && !g.fast;  // else they are there already
      const int kbeg = cur.kbeg, kend = cur.kbeg + cur.n;
      f32x4 pa[XA::NV], pb[XB::NV];
      xa.fetch_checked(pa, kbeg, kend, tv);
      xb.fetch_checked(pb, kbeg, kend, tv);
      for (int k0 = kbeg; k0 < kend; k0 += x3::BK) {
        __syncthreads();
        xa.put(As, pa);
        xb.put(Bs, pb);
        if constexpr (ACT == 3) {
          if (sums) XB::colsum_add(cso, pb);
        }
        __syncthreads();
        if (k0 + x3::BK < kend) {
          xa.fetch_checked(pa, k0 + x3::BK, kend, tv);
          xb.fetch_checked(pb, k0 + x3::BK, kend, tv);
        }
        bf16x8 a[3][MI], b[3][NI];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int i = 0; i < MI; ++i) a[p][i] = XA::frag(As, p, wm + 32 * i, lv);
#pragma unroll
          for (int j = 0; j < NI; ++j) b[p][j] = XB::frag(Bs, p, wn + 32 * j, lv);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            f32x16 c = acc[i][j];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2][i], b[0][j], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][i], b[1][j], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[2][j], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][i], b[0][j], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[1][j], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[0][j], c, 0, 0, 0);
            acc[i][j] = c;
          }
      }
      __syncthreads();
    }

    // the samples of the tile after the next, on their way during the epilogue
    const bool more2 = g.fast && tile + 2 * wgs < tend;
    const int tq = here(tid);
    f32x4 qa[SA::NQ], qb[SB::NQ];
    if (more2) {
      const Place p2 = place(tile + 2 * wgs);
      sa.sample(qa, src_a(p2), p2.n, tq);
      sb.sample(qb, src_b(p2), p2.n, tq);
    }

    if constexpr (ACT == 3) {
      // the first row of tiles reduces the per-thread column sums through
      // LDS: KC: 8 (three pieces: 4) threads per column, else 8 threads per 4
      // columns; contributors are added in a fixed order
      static_assert(BN == 128, "column sums");
      if (cur.m0 == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (BN1) {
            red[(tid / 32) * BN + 4 * (tid % 32) + i] = cso[i];
          } else {
            const int idx = tid + i * kGT;
            if (g.fast) red[(idx % 8) * BN + idx / 8] = cso[i];
            else if (i < XB::NV) red[(idx % 4) * BN + idx / 4] = cso[i];
          }
        }
        __syncthreads();
        if (tid < BN) {
          const int nc = BN1 || g.fast ? 8 : 4;
          float v = 0.f;
          for (int c = 0; c < nc; ++c) v += red[c * BN + tid];
          const int n = cur.n0 + tid;
          if (n < g.N) {
            if (g.ksplit > 1) g.ws[(int64_t)g.ksplit * g.M * g.N + (int64_t)cur.split * g.N + n] = v;
            else g.colsum[n] = g.colsum_acc ? g.colsum[n] + v : v;
          }
        }
        __syncthreads();
      }
    }

    // Epilogue, from the accumulators: acc[i][j][e] = wave tile element
    // (32i + 8(e/4) + 4(lane/32) + e%4, 32j + lane%32), so an element e of all
    // lanes is two rows' 32 columns, a whole 128-byte line each.  A row pair
    // is stored (and its aux and old values read) through a resource that
    // begins at its first row and ends with the output: rows past it are
    // dropped, a column past it has an offset that is.
    const int lv = here(lane), lr = lv & 31, lh = lv >> 5;
    const bool to_ws = g.ksplit > 1;
    const bool rd_c = !to_ws && g.beta != 0.f;
    const bool use_x = !to_ws && (ACT == 2 || ACT == 4 || (ACT == 1 && g.aux != nullptr));
    const uint32_t* am = amax[seq & 3];
    const int n1 = cur.n0 + wn;  // the wave's first column
    float unB[NI], bv[NI];       // of this lane's columns
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      unB[j] = scaled ? h2::unscale(am[BM + wn + 32 * j + lr]) : 1.f;
      bv[j] = !to_ws && g.bias && n1 + 32 * j + lr < g.N ? g.bias[n1 + 32 * j + lr] : 0.f;
    }
    // the product's values of row group (i, q): [u][j]
    auto values = [&](int i, int q, float (&v)[4][NI]) {
      const uint4 a4 = *reinterpret_cast<const uint4*>(am + wm + 32 * i + 8 * q + 4 * lh);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float unA = h2::unscale(u == 0 ? a4.x : u == 1 ? a4.y : u == 2 ? a4.z : a4.w);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          float x = acc[i][j][4 * q + u];
          if (scaled) x = __builtin_fmaf(accx[i][j][4 * q + u], 0x1p-14f, x) * unA * unB[j];
          v[u][j] = to_ws ? x : g.alpha * x + bv[j];
        }
      }
    };
    // the output (or this split's partials), its row stride, and the aux rows
    float* Out = to_ws ? g.ws + ((int64_t)cur.split * g.batch + cur.bidx) * (int64_t)g.M * g.N
                       : g.c + (int64_t)cur.bidx * g.scb;
    const int64_t so = to_ws ? g.N : g.scm;
    float* X = g.aux + (int64_t)cur.bidx * g.sxb;
    if (g.rows_vec) {
      uint32_t oo[NI], xo[NI];
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const bool ok = n1 + 32 * j + lr < g.N;
        oo[j] = ok ? (uint32_t)(4 * lh * so + 32 * j + lr) * 4u : 0xfffffff0u;
        xo[j] = ok ? (uint32_t)(4 * lh * g.sxm + 32 * j + lr) * 4u : 0xfffffff0u;
      }
      // the wave's rows of an array: a resource at row r (rows are asked for in
      // steps, the address and the bytes left move by uniform additions)
      struct Rows {
        const char* p;
        int64_t left, step;
        __device__ __forceinline__ __amdgpu_buffer_rsrc_t at(int r) const {
          const int64_t l = left - r * step;
          const int hi = (int)(l >> 32);
          const uint32_t bytes = hi < 0 ? 0u : hi > 0 ? 0xffffff00u : (uint32_t)l;
          return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p + r * step), (short)0, (int)bytes, 0x00020000);
        }
      };
      const int mw = cur.m0 + wm;
      auto rows = [&](const float* p, int64_t stride) {
        return Rows{reinterpret_cast<const char*>(p + (int64_t)mw * stride + n1),
                    n1 < g.N ? ((int64_t)(g.M - 1 - mw) * stride + (g.N - n1)) * 4 : -1, stride * 4};
      };
      const Rows ro = rows(Out, so), rx = rows(X, g.sxm);
      // aux values are requested kAhead row groups before their use
      constexpr int kAhead = NI > 2 ? 2 : 4;
      float xv[kAhead][4][NI];
      auto aux = [&](int iq) {
        if constexpr (ACT == 2 || ACT == 4) {
          if (use_x) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const auto r = rx.at(8 * iq + u);
#pragma unroll
              for (int j = 0; j < NI; ++j)
                xv[iq % kAhead][u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)xo[j], 0, 0));
            }
          }
        }
      };
#pragma unroll
      for (int iq = 0; iq < kAhead; ++iq) aux(iq);
#pragma unroll
      for (int iq = 0; iq < 4 * MI; ++iq) {
        __builtin_amdgcn_sched_barrier(0);
        float old[4][NI], v[4][NI];
        if (rd_c) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const auto r = ro.at(8 * iq + u);
#pragma unroll
            for (int j = 0; j < NI; ++j)
              old[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)oo[j], 0, 0));
          }
        }
        values(iq / 4, iq % 4, v);
        if (rd_c) {
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < NI; ++j) v[u][j] += g.beta * old[u][j];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if constexpr (ACT == 1) {
            if (use_x) {
              const auto r = rx.at(8 * iq + u);
#pragma unroll
              for (int j = 0; j < NI; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[u][j]), r, (int)xo[j], 0, 0);
            }
          }
          const auto r = ro.at(8 * iq + u);
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            float w = v[u][j];
            if constexpr (ACT == 1) w = to_ws ? w : gelu_tanh_fast(w);
            if constexpr (ACT == 2) w = use_x ? w * gelu_grad_fast(xv[iq % kAhead][u][j]) : w;
            if constexpr (ACT == 4) w = use_x ? w + xv[iq % kAhead][u][j] : w;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(w), r, (int)oo[j], 0, 0);
          }
        }
        if (iq + kAhead < 4 * MI) aux(iq + kAhead);
      }
    } else {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[4][NI];
          values(i, q, v);
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < NI; ++j) {
              const int m = cur.m0 + wm + 32 * i + 8 * q + 4 * lh + u, n = n1 + 32 * j + lr;
              if (m >= g.M || n >= g.N) continue;
              float* p = Out + (int64_t)m * so + (int64_t)n * (to_ws ? 1 : g.scn);
              float* xp = X + (int64_t)m * g.sxm + (int64_t)n * g.sxn;
              float w = v[u][j];
              if (rd_c) w += g.beta * *p;
              if constexpr (ACT == 1) {
                if (use_x) *xp = w;
                w = to_ws ? w : gelu_tanh_fast(w);
              }
              if constexpr (ACT == 2) w = use_x ? w * gelu_grad_fast(*xp) : w;
              if constexpr (ACT == 4) w = use_x ? w + *xp : w;
              *p = w;
            }
        }
    }

    if (more2) {
      SA::row_max(qa, amax[(seq + 2) & 3], tq);
      SB::row_max(qb, amax[(seq + 2) & 3] + BM, tq);
    }
    if (!more) break;
    tile += wgs;
    cur = next;
    if (!g.fast || !primed) __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Skinny products: M <= 64 rows (a decode step's sequences), K <= 4096 (in
// up to 8 ranges of 512, one workgroup each, when longer than 512).
// One workgroup of 16 waves owns 16 output columns for every row; the waves
// split K into 16-wide slices dealt round-robin, and their partial tiles are
// summed through LDS in wave order (deterministic, one launch, no split-K
// workspace).  Within a slice the lane of group grp supplies, to the four
// MFMA steps s = 0..3, k = 4*grp + s for both A and B (the same k on both
// sides, so each MFMA contracts over four distinct k and the four steps
// cover the slice); A's four values are then one 16-byte load when A is
// contiguous along k.  Each wave loads kSkG slices before multiplying them
// (one when A needs scalar loads).
// ---------------------------------------------------------------------------
#ifndef MTX_SKINNY_WAVES
#define MTX_SKINNY_WAVES 16
#endif
#ifndef MTX_SKINNY_INFLIGHT
#define MTX_SKINNY_INFLIGHT 1
#endif
constexpr int kSkW = MTX_SKINNY_WAVES;     // waves per workgroup
constexpr int kSkT = kSkW * 64;            // threads per workgroup
constexpr int kSkG = MTX_SKINNY_INFLIGHT;  // slices in flight per wave
// every workgroup reads all of its K range of A (M x K) through its CU, so a
// longer K is split over workgroups of at most kSkMaxK each (grid.z), whose
// partial tiles gemm_splitk_reduce sums in split order (measured at M = 64:
// K = 384 one launch 5.9 us against 8.9 us for tiled split-K + reduce;
// K = 1536 unsplit 16 us)
constexpr int kSkMaxM = 64, kSkMaxK = 512, kSkMaxSplit = 8;

// four values at k..k+3 along a dimension of stride sk; V: the host has
// checked that the operand is contiguous along k, 16-byte aligned at every
// k multiple of 4, and K % 4 == 0, so a k group is either whole or past K
template <bool V>
__device__ __forceinline__ f32x4 load4_k(const float* __restrict__ p, int64_t sk, int k, int K, bool ok) {
  f32x4 x = zero4();
  if constexpr (V) {
    if (ok && k < K) x = *reinterpret_cast<const f32x4*>(p);
  } else {
    if (ok) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j < K) x[j] = p[(int64_t)j * sk];
    }
  }
  return x;
}

template <bool AV, bool BV>
__global__ __launch_bounds__(kSkT) void gemm_skinny_kernel(const GemmArgs g) {
  __shared__ float red[kSkW][kSkMaxM * 16];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int n16 = lane & 15, grp = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int bidx = blockIdx.y;
  const int split = blockIdx.z;
  const int n = n0 + n16;
  const bool nok = n < g.N;
  // this workgroup's 16-wide k slices (kchunk is a multiple of 16)
  const int sbeg = split * (g.kchunk / 16);
  const int nsl = min((g.K + 15) / 16, sbeg + g.kchunk / 16);
  // lane bases: row 16i + n16 of A (i = 0..3 by a row offset of 16 rows),
  // column n of B, both at k = 4 * grp
  const float* __restrict__ Ab = g.a + (int64_t)bidx * g.sab + (int64_t)n16 * g.sam + (int64_t)(4 * grp) * g.sak;
  const float* __restrict__ Bb = g.b + (int64_t)bidx * g.sbb + (int64_t)n * g.sbn + (int64_t)(4 * grp) * g.sbk;
  const int64_t a16 = 16 * g.sam;
  // slices in flight: A with four scalar loads per group needs the registers
  constexpr int G = AV ? kSkG : 1;

  f32x4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = zero4();
  for (int s0 = sbeg + wid; s0 < nsl; s0 += G * kSkW) {
    f32x4 af[G][4], bf[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int kb = (s0 + j * kSkW) * 16;  // past K after the last slice: zeros
      if (G > 1 && s0 + j * kSkW >= nsl) {       // past this split's range
        af[j][0] = af[j][1] = af[j][2] = af[j][3] = bf[j] = zero4();
        continue;
      }
      const int k = kb + 4 * grp;
      const float* pa = Ab + (int64_t)kb * g.sak;
#pragma unroll
      for (int i = 0; i < 4; ++i) af[j][i] = load4_k<AV>(pa + i * a16, g.sak, k, g.K, 16 * i + n16 < g.M);
      bf[j] = load4_k<BV>(Bb + (int64_t)kb * g.sbk, g.sbk, k, g.K, nok);
    }
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[j][i][s], bf[j][s], acc[i], 0, 0, 0);
  }
  // acc[i][r] = partial C[16i + 4grp + r][n16]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wid][(16 * i + 4 * grp + r) * 16 + n16] = acc[i][r];
  __syncthreads();
#pragma unroll
  for (int e = tid; e < kSkMaxM * 16; e += kSkT) {
    const int row = e >> 4, col = n0 + (e & 15);
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kSkW; ++w) v += red[w][e];
    if (row < g.M && col < g.N && (g.ksplit > 1 || g.to_ws)) {
      g.ws[((int64_t)split * g.batch + bidx) * g.M * g.N + (int64_t)row * g.N + col] = v;
    } else if (row < g.M && col < g.N) {
      float o = g.alpha * v + (g.bias ? g.bias[col] : 0.f);
      if (col < g.nc) {
        float* p = g.c + (int64_t)bidx * g.scb + (int64_t)row * g.scm + (int64_t)col * g.scn;
        if (g.beta != 0.f) o += g.beta * *p;
        if (g.act == 1) o = gelu_tanh(o);
        *p = o;
      } else {
        const int half = (g.N - g.nc) >> 1;
        const int j = col - g.nc;
        float* cache = j < half ? g.kc : g.vc;
        const int jj = j < half ? j : j - half;
        const int t = g.lengths[row] - 1;
        if (t >= 0 && t < g.cT) cache[(int64_t)row * g.csb + (int64_t)t * g.cst + jj] = o;
      }
    }
  }
}

// operand contiguous along k with every 4-aligned k group 16-byte aligned
bool k_vec(const float* p, int64_t s_row, int64_t s_k, int64_t s_batch, int K) {
  return s_k == 1 && K % 4 == 0 && (((uintptr_t)p) & 15u) == 0 && s_row % 4 == 0 && s_batch % 4 == 0;
}

bool use_skinny(int M, int K) { return M <= kSkMaxM && K <= kSkMaxK; }
// K splits of the skinny kernel for an M x K activation, 0 when it does not apply
int skinny_splits(int M, int K) {
  if (M > kSkMaxM || K > kSkMaxK * kSkMaxSplit) return 0;
  return cdiv(K, kSkMaxK);
}

// Column sums of B (batch 1) for the weight-gradient entry point when its
// product takes the skinny kernel (M <= 64): 16 columns x 16 k lanes per
// workgroup, the lanes' sums added in lane order.
__global__ __launch_bounds__(256) void gemm_colsum_kernel(const GemmArgs g) {
  __shared__ float part[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int n = blockIdx.x * 16 + tx;
  float s = 0.f;
  if (n < g.N) {
    const float* __restrict__ col = g.b + (int64_t)n * g.sbn;
#pragma unroll 8
    for (int k = ty; k < g.K; k += 16) s += col[(int64_t)k * g.sbk];
  }
  part[ty][tx] = s;
  __syncthreads();
  if (ty == 0 && n < g.N) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += part[k][tx];
    g.colsum[n] = g.colsum_acc ? g.colsum[n] + t : t;
  }
}

// Sum the split-K partials in split order; apply alpha, beta, bias.
__global__ __launch_bounds__(256) void gemm_splitk_reduce(const GemmArgs g) {
  const int64_t MN = (int64_t)g.M * g.N;
  const int64_t total = MN * g.batch;
  // indices past the C elements are the weight-gradient variant's column
  // sums (batch 1), on threads of their own
  const int64_t extra = g.colsum ? g.N : 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total + extra;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (i >= total) {
      const int64_t n = i - total;
      float s = 0.f;
#pragma unroll 8
      for (int sp = 0; sp < g.ksplit; ++sp) s += g.ws[(int64_t)g.ksplit * MN + (int64_t)sp * g.N + n];
      g.colsum[n] = g.colsum_acc ? g.colsum[n] + s : s;
      continue;
    }
    const int bidx = (int)(i / MN);
    const int64_t e = i % MN;
    const int m = (int)(e / g.N), n = (int)(e % g.N);
    float s = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < g.ksplit; ++sp) s += g.ws[((int64_t)sp * g.batch + bidx) * MN + e];
    float* p = g.c + (int64_t)bidx * g.scb + (int64_t)m * g.scm + (int64_t)n * g.scn;
    float v = g.alpha * s + (g.bias ? g.bias[n] : 0.f);
    if (g.beta != 0.f) v += g.beta * *p;
    *p = epilogue(g, v, bidx, m, n);
  }
}

// The same, four columns a thread, where C's rows (and aux's) are whole
// aligned vectors: HBM bound, one 32-bit division per vector instead of two
// 64-bit ones per value (8 partials of 512 x 2048: 19.1 -> 9.2 us).  The sums
// have gemm_splitk_reduce's order.
__global__ __launch_bounds__(256) void gemm_splitk_reduce4(const GemmArgs g) {
  const uint32_t MN = (uint32_t)g.M * (uint32_t)g.N, nv = MN / 4;
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const int bidx = blockIdx.y;
  if (i >= nv) {  // column sums (batch 1), on threads of their own
    const uint32_t n = i - nv;
    if (!g.colsum || n >= (uint32_t)g.N) return;
    float s = 0.f;
#pragma unroll 8
    for (int sp = 0; sp < g.ksplit; ++sp) s += g.ws[(int64_t)g.ksplit * MN + (int64_t)sp * g.N + n];
    g.colsum[n] = g.colsum_acc ? g.colsum[n] + s : s;
    return;
  }
  const uint32_t e = 4 * i, m = e / (uint32_t)g.N, n = e - m * (uint32_t)g.N;
  const float* __restrict__ w = g.ws + (int64_t)bidx * MN + e;
  const int64_t step = (int64_t)g.batch * MN;
  f32x4 s = zero4();
#pragma unroll 8
  for (int sp = 0; sp < g.ksplit; ++sp) s += *reinterpret_cast<const f32x4*>(w + sp * step);
  float* p = g.c + (int64_t)bidx * g.scb + (int64_t)m * g.scm + n;
  f32x4 v, old = zero4();
  if (g.beta != 0.f) old = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float x = g.alpha * s[u] + (g.bias ? g.bias[n + u] : 0.f);
    if (g.beta != 0.f) x += g.beta * old[u];
    v[u] = epilogue(g, x, bidx, (int)m, (int)n + u);
  }
  *reinterpret_cast<f32x4*>(p) = v;
}

int launch_splitk_reduce(const GemmArgs& g, hipStream_t st) {
  const int64_t MN = (int64_t)g.M * g.N;
  const bool vec = g.N % 4 == 0 && MN < ((int64_t)1 << 30) && g.batch < 65536 && g.scn == 1 && g.scm % 4 == 0 &&
                   g.scb % 4 == 0 && (((uintptr_t)g.c) & 15u) == 0 && (((uintptr_t)g.ws) & 15u) == 0;
  if (vec) {
    const int64_t threads = MN / 4 + (g.colsum ? g.N : 0);
    hipLaunchKernelGGL(gemm_splitk_reduce4, dim3((unsigned)((threads + 255) / 256), g.batch), dim3(256), 0, st, g);
  } else {
    const int64_t total = MN * g.batch + (g.colsum ? g.N : 0);
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(gemm_splitk_reduce, dim3(blocks), dim3(256), 0, st, g);
  }
  MTX_LAUNCHED();
  return MTX_OK;
}

// The split-K reduce of a skinny product followed by LayerNorm of the result
// rows (a decode step's "x += h @ W + b, then ln(x)" in one launch): one
// wave per row.  Per element the arithmetic of gemm_splitk_reduce (partials
// added in split order, then alpha, bias, beta * C), then the row
// statistics of layernorm_fwd_kernel on the values just stored, so C and y
// equal the two-launch sequence's.  Every load of the row is issued before
// the first store (a store in between would order each element's loads
// after it), with the split count KS fixed at compile time.
template <int VPL, int KS>
__global__ __launch_bounds__(64) void splitk_reduce_ln_kernel(const GemmArgs g, const float* __restrict__ gamma,
                                                              const float* __restrict__ beta_ln, float eps,
                                                              float* __restrict__ y, int64_t ldy) {
  const int m = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t MN = (int64_t)g.M * g.N;
  float v[VPL], r[VPL], bb[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int n = lane + 64 * i;
    const bool ok = n < g.N;
    const int64_t e = ok ? (int64_t)m * g.N + n : 0;
    float part[KS];
#pragma unroll
    for (int sp = 0; sp < KS; ++sp) part[sp] = g.ws[(int64_t)sp * MN + e];
    float s = 0.f;
#pragma unroll
    for (int sp = 0; sp < KS; ++sp) s += part[sp];
    v[i] = s;
    r[i] = ok && g.beta != 0.f ? g.c[(int64_t)m * g.scm + (int64_t)n * g.scn] : 0.f;
    bb[i] = ok && g.bias ? g.bias[n] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int n = lane + 64 * i;
    float t = g.alpha * v[i] + bb[i];
    if (g.beta != 0.f) t += g.beta * r[i];
    v[i] = n < g.N ? t : 0.f;
    if (n < g.N) g.c[(int64_t)m * g.scm + (int64_t)n * g.scn] = t;
  }
  float mean, sd;
  ln_stats<VPL>(v, lane, g.N, eps, mean, sd);
  const Divisor by_sd(sd);
  float* yr = y + (int64_t)m * ldy;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int n = lane + 64 * i;
    if (n < g.N) yr[n] = ln_apply(v[i], by_sd, gamma[n], beta_ln[n]);
  }
}

template <int VPL>
void launch_reduce_ln(const GemmArgs& g, const float* gamma, const float* beta_ln, float eps, float* y,
                      int64_t ldy, hipStream_t st) {
  const dim3 grid(g.M), block(64);
#define RLN(KS) hipLaunchKernelGGL((splitk_reduce_ln_kernel<VPL, KS>), grid, block, 0, st, g, gamma, beta_ln, eps, y, ldy)
  switch (g.ksplit) {
    case 1: RLN(1); break;
    case 2: RLN(2); break;
    case 3: RLN(3); break;
    case 4: RLN(4); break;
    case 5: RLN(5); break;
    case 6: RLN(6); break;
    case 7: RLN(7); break;
    default: RLN(8); break;
  }
#undef RLN
}

struct Plan {
  int bm, bn, ksplit, kchunk;  // tile rows and columns, K split
};

// Pick the tile and the K split for a problem so that the launch has enough
// workgroups to fill 256 CUs, splitting K only when it is long.
Plan plan_gemm(int M, int N, int K, int batch, size_t ws_bytes) {
  Plan p{128, 128, 1, K};
  auto tiles = [&](int bm, int bn) { return (int64_t)cdiv(M, bm) * cdiv(N, bn) * batch; };
  // Long-K products with both sides >= 128 (weight gradients, K = B*T) keep
  // 128x128 tiles and split K further: with 64x64 tiles every tile row and
  // column re-reads its operand panel from beyond L2, twice the traffic.
  const bool longk = K >= 4096 && M >= 128 && N >= 128;
  // 128x128 tiles only when they fill whole rounds of the 256 CUs: a last,
  // partly filled round of these long-running tiles costs more than the
  // smaller tiles' extra operand traffic (16384 x 1152, K = 384: 179 us with
  // 1152 = 4.5 x 256 tiles of 128x128)
  const int64_t t128 = tiles(128, 128);
  if (!longk && (t128 < 512 || t128 % 256 != 0)) { p.bm = 64; p.bn = 64; }
  const int64_t t = tiles(p.bm, p.bn);
  if (t < 256 && K >= 1024) {
    // up to 64 splits for K >= 4096 (partials: want x M x N floats)
    int want = (int)std::min<int64_t>(K >= 4096 ? 64 : 16, (MTX_SPLIT_TARGET + t - 1) / t);
    // each split keeps >= MTX_SPLIT_MINK of K
    want = std::min(want, std::max(1, K / MTX_SPLIT_MINK));
    const size_t need = (size_t)want * batch * (size_t)(M + 1) * N * sizeof(float);
    if (want > 1 && need <= ws_bytes) {
      p.ksplit = want;
      p.kchunk = cdiv(cdiv(K, want), BK) * BK;
      p.ksplit = cdiv(K, p.kchunk);
    }
  } else if (t < 64 && K >= 128) {
    // skinny products (decode steps: M = sequences): too few output tiles to
    // cover the CUs, so split K into chunks of >= 64
    int want = (int)std::min<int64_t>(16, (256 + t - 1) / t);
    want = std::min(want, K / 64);
    const size_t need = (size_t)want * batch * (size_t)M * N * sizeof(float);
    if (want > 1 && need <= ws_bytes) {
      p.ksplit = want;
      p.kchunk = cdiv(cdiv(K, want), BK) * BK;
      p.ksplit = cdiv(K, p.kchunk);
    }
  }
  return p;
}

template <int BM, int BN, int ACT>
void launch_tile_act(const GemmArgs& g, bool ak, bool bn1, hipStream_t st) {
  dim3 grid(cdiv(g.N, BN), cdiv(g.M, BM), g.batch * g.ksplit);
  if (ak && bn1) hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, true, true, ACT>), grid, dim3(kGT), 0, st, g);
  else if (ak) hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, true, false, ACT>), grid, dim3(kGT), 0, st, g);
  else if (bn1) hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, false, true, ACT>), grid, dim3(kGT), 0, st, g);
  else hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, false, false, ACT>), grid, dim3(kGT), 0, st, g);
}

// the activation epilogue applies only when the tile kernel writes C itself
// (unsplit K); with split K the reduce kernel applies it
template <int BM, int BN>
int launch_tile(const GemmArgs& g, bool ak, bool bn1, hipStream_t st) {
  const int act = g.ksplit > 1 ? 0 : g.act;
  if (g.colsum) launch_tile_act<BM, BN, 3>(g, ak, bn1, st);
  else if (act == 1) launch_tile_act<BM, BN, 1>(g, ak, bn1, st);
  else if (act == 2) launch_tile_act<BM, BN, 2>(g, ak, bn1, st);
  else if (act == 4) launch_tile_act<BM, BN, 4>(g, ak, bn1, st);
  else launch_tile_act<BM, BN, 0>(g, ak, bn1, st);
  MTX_LAUNCHED();
  return MTX_OK;
}

// Which kernel computes fp32 products of at least 128 x 128 (mtx_gemm_set_mode):
// MTX_GEMM_BF16X3 (default) the split kernel on the 16-bit matrix cores (two
// fp16 or three bf16 pieces), MTX_GEMM_FP32 the fp32 MFMA tile kernel.  Smaller products, and
// the decode step's skinny ones, always take the fp32 kernels.
std::atomic<int> g_gemm_mode{MTX_GEMM_BF16X3};

// Products below 2^27 multiply-adds (the C0 model's 512-row ones: a handful
// of 128 x 128 tiles, latency bound) stay on the fp32 kernel's 64 x 64
// tiles: on the split kernel the C0 training step took 0.445 ms against
// 0.379 ms.
// Nor do products with fewer than 64 tiles of 128 x 128 and a K too short to
// split (< 1024): at K = 384 the fp32 kernel's 64 x 64 tiles and the split
// kernel took 19.8 and 20 us for 1000 x 384 (24 tiles), 24.5 and 21.9 for
// 2944 x 384 (69), 22.9 and 19.6 for 1000 x 1152 (72), 26.7 and 25.1 for
// 1000 x 1536 + GELU (96); 8008 x 512 x 512 (252) 48.4 and 36.4.
bool use_x3(int M, int N, int K, int batch) {
  if (g_gemm_mode.load(std::memory_order_relaxed) != MTX_GEMM_BF16X3 || M < 128 || N < 128 ||
      (int64_t)M * N * K * batch < ((int64_t)1 << 27))
    return false;
  const int64_t tiles = (int64_t)cdiv(M, 128) * cdiv(N, 128) * batch;
  return tiles >= 64 || K >= 1024;
}

// Two workgroups of the split kernel fit a CU.
constexpr int kX3Wgs = 512;
constexpr double kX3W96 = 0.8;  // a 128 x 96 tile's time against a 128 x 128 one's

// Time of `tiles` tiles of weight w on kX3Wgs resident workgroups, in tile
// times of two workgroups sharing a CU: whole rounds, and a last one in which
// a workgroup that has its CU for itself is done sooner.
double x3_rounds(int64_t tiles, double w) {
  const int64_t rem = tiles % kX3Wgs;
  return w * ((double)(tiles / kX3Wgs) + (rem == 0 ? 0.0 : rem <= kX3Wgs / 2 ? 0.65 : 1.0));
}

// Tiles of 128 x 128 or, where A is contiguous along k (forward and dX
// products), 128 x 96: whichever ends sooner.  N = 384 is three columns of
// 128 (M = 16384: 384 tiles, a round three quarters full) or four of 96
// (512, one full round): K = 384 + residual 42.0 -> 38.5 us, K = 1536 91 ->
// 83, its dX 84 -> 76.
// K is split only when the 128 x 128 tiles leave the CUs idle (weight
// gradients, K = B*T): into as many ranges as keep one round of kX3Wgs
// workgroups, each with >= h2::MINK of K.
Plan plan_x3(int M, int N, int K, int batch, size_t ws_bytes, bool ak, bool colsum) {
  Plan p{128, 128, 1, K};
  const int64_t t = (int64_t)cdiv(M, 128) * cdiv(N, 128) * batch;
  if (t < 256 && K >= 1024) {
    for (int want = (int)std::min<int64_t>(K / h2::MINK, kX3Wgs / t); want > 1; --want) {
      const int chunk = cdiv(cdiv(K, want), h2::BK) * h2::BK, ks = cdiv(K, chunk);
      const size_t need = (size_t)ks * batch * (size_t)(M + 1) * N * sizeof(float);
      if (ks > 1 && K - (ks - 1) * chunk >= h2::MINK && need <= ws_bytes) {
        p.ksplit = ks;
        p.kchunk = chunk;
        break;
      }
    }
  } else if (ak && !colsum) {
    const int64_t t96 = (int64_t)cdiv(M, 128) * cdiv(N, 96) * batch;
    if (x3_rounds(t96, kX3W96) < x3_rounds(t, 1.0)) p.bn = 96;
  }
  return p;
}

// Whether the two-piece form may be tried: h2::MINK of K and more in every
// range, and 32-bit offsets reach a tile's rows and its samples' k rows.
bool two_pieces(const GemmArgs& g) {
  const int64_t lim = (int64_t)1 << 29;
  auto ok = [&](int64_t s_row, int64_t s_k) {
    return s_row >= 0 && s_k >= 0 && (s_k == 1 ? 128 * s_row + g.kchunk : g.kchunk * s_k + 128) < lim;
  };
  const int last = g.K - (g.ksplit - 1) * g.kchunk;
  return std::min(g.kchunk, last) >= h2::MINK && ok(g.sam, g.sak) && ok(g.sbn, g.sbk);
}

template <int ACT>
void launch_x3_act(const GemmArgs& g, int bn, bool ak, bool bn1, hipStream_t st) {
  const int64_t tiles = (int64_t)cdiv(g.N, bn) * cdiv(g.M, 128) * g.batch * g.ksplit;
  const dim3 grid((unsigned)std::min<int64_t>(tiles, kX3Wgs)), block(kGT);
  if constexpr (ACT != 3) {
    if (bn == 96) {  // four waves of 32 x 96
      if (bn1) hipLaunchKernelGGL((gemm_x3_kernel<1, 3, 4, 1, true, true, ACT>), grid, block, 0, st, g);
      else hipLaunchKernelGGL((gemm_x3_kernel<1, 3, 4, 1, true, false, ACT>), grid, block, 0, st, g);
      return;
    }
  }
  if (ak && bn1) hipLaunchKernelGGL((gemm_x3_kernel<2, 2, 2, 2, true, true, ACT>), grid, block, 0, st, g);
  else if (ak) hipLaunchKernelGGL((gemm_x3_kernel<2, 2, 2, 2, true, false, ACT>), grid, block, 0, st, g);
  else if (bn1) hipLaunchKernelGGL((gemm_x3_kernel<2, 2, 2, 2, false, true, ACT>), grid, block, 0, st, g);
  else hipLaunchKernelGGL((gemm_x3_kernel<2, 2, 2, 2, false, false, ACT>), grid, block, 0, st, g);
}

// as launch_tile: with split K the reduce kernel applies the activation
int launch_x3(const GemmArgs& g, int bn, bool ak, bool bn1, hipStream_t st) {
  const int act = g.ksplit > 1 ? 0 : g.act;
  if (g.colsum) launch_x3_act<3>(g, bn, ak, bn1, st);
  else if (act == 1) launch_x3_act<1>(g, bn, ak, bn1, st);
  else if (act == 2) launch_x3_act<2>(g, bn, ak, bn1, st);
  else if (act == 4) launch_x3_act<4>(g, bn, ak, bn1, st);
  else launch_x3_act<0>(g, bn, ak, bn1, st);
  MTX_LAUNCHED();
  return MTX_OK;
}

}  // namespace
}  // namespace mtx

using namespace mtx;

extern "C" size_t mtx_gemm_workspace_bytes(int M, int N, int K, int batch) {
  if (M < 1 || N < 1 || K < 1 || batch < 1) return 0;
  // The skinny kernel serves plain products with M <= 64; the same shape with
  // an activation epilogue (mtx_gemm_act_f32) or column sums goes to the tile
  // kernel, so the size covers both plans.
  const int sp = skinny_splits(M, K);
  const size_t skinny = sp > 1 ? (size_t)sp * batch * (size_t)M * N * sizeof(float) : 0;
  Plan p = plan_gemm(M, N, K, batch, (size_t)-1);
  // split partials [split][batch][M][N], then the weight-gradient variant's
  // column sums [split][N]
  const size_t tiled = p.ksplit > 1 ? (size_t)p.ksplit * batch * (size_t)(M + 1) * N * sizeof(float) : 0;
  // the split kernel's plan (either mode may be set when the product runs)
  Plan q = plan_x3(M, N, K, batch, (size_t)-1, false, false);
  const size_t split3 = q.ksplit > 1 ? (size_t)q.ksplit * batch * (size_t)(M + 1) * N * sizeof(float) : 0;
  return std::max({skinny, tiled, split3});
}

extern "C" int mtx_gemm_set_mode(int mode) {
  MTX_CHECK_ARG(mode == MTX_GEMM_FP32 || mode == MTX_GEMM_BF16X3,
                "gemm mode %d must be MTX_GEMM_FP32 (0) or MTX_GEMM_BF16X3 (1)", mode);
  g_gemm_mode.store(mode);
  return MTX_OK;
}

extern "C" int mtx_gemm_get_mode(void) { return g_gemm_mode.load(); }

namespace {
int gemm_impl(int M, int N, int K, int batch, float alpha, const float* a, int64_t sa_m, int64_t sa_k,
              int64_t sa_b, const float* b, int64_t sb_k, int64_t sb_n, int64_t sb_b, float beta, float* c,
              int64_t sc_m, int64_t sc_n, int64_t sc_b, const float* bias, int act, float* aux, int64_t sx_m,
              int64_t sx_n, int64_t sx_b, void* workspace, size_t workspace_bytes, void* stream,
              float* colsum = nullptr, int colsum_acc = 0) {
  MTX_CHECK_SHAPE(M >= 0 && N >= 0 && K >= 0 && batch >= 0, "negative GEMM size");
  if (M == 0 || N == 0 || batch == 0) return MTX_OK;
  MTX_CHECK_ARG(c != nullptr, "gemm: null C");
  MTX_CHECK_ARG(K == 0 || (a != nullptr && b != nullptr), "gemm: null A or B");
  // (an empty K leaves A and B unread, whatever their strides)
  MTX_CHECK_ARG(K == 0 || sa_k == 1 || sa_m == 1, "gemm: A needs a unit stride along m or k");
  MTX_CHECK_ARG(K == 0 || sb_n == 1 || sb_k == 1, "gemm: B needs a unit stride along k or n");
  MTX_CHECK_ARG(sc_m >= 0 && sc_n >= 0 && sa_b >= 0 && sb_b >= 0 && sc_b >= 0, "gemm: negative stride");
  MTX_CHECK_SHAPE((int64_t)batch * cdiv(M, 64) < 65535 * 64, "gemm: too many tiles");
  GemmArgs g{a, sa_m, sa_k, sa_b, b, sb_k, sb_n, sb_b, c, sc_m, sc_n, sc_b, bias,
             static_cast<float*>(workspace), M, N, K, batch, 1, K, alpha, beta};
  g.nc = N;
  g.aux = aux;
  g.sxm = sx_m;
  g.sxn = sx_n;
  g.sxb = sx_b;
  g.colsum = colsum;
  g.colsum_acc = colsum_acc;
  {
    const bool a_ok = (((uintptr_t)a) & 15u) == 0 && (sa_k == 1 ? sa_m % 4 == 0 : sa_k % 4 == 0) && sa_b % 4 == 0;
    const bool b_ok = (((uintptr_t)b) & 15u) == 0 && (sb_n == 1 ? sb_k % 4 == 0 : sb_n % 4 == 0) && sb_b % 4 == 0;
    g.vec_ok = a_ok && b_ok;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  // the activation epilogue runs in the tiled kernel and the split-K reduce
  // (the skinny kernel's act field is the decode step's own)
  g.act = act;
  if (K == 0) {  // C = act(beta*C + bias)
    g.ksplit = 1;
    g.kchunk = 0;
    return launch_tile<64, 64>(g, true, true, st);
  }
  if (int sp = act ? 0 : skinny_splits(M, K)) {
    MTX_CHECK_SHAPE(batch < 65536, "gemm: batch too large");
    if (colsum) {  // the skinny kernel and its reduce leave the sums to their own kernel
      hipLaunchKernelGGL(gemm_colsum_kernel, dim3(cdiv(N, 16)), dim3(256), 0, st, g);
      MTX_LAUNCHED();
      g.colsum = nullptr;
    }
    // without room for the partials, one workgroup covers all of K
    if (sp > 1 && (!workspace || workspace_bytes < (size_t)sp * batch * (size_t)M * N * sizeof(float))) sp = 1;
    g.ksplit = sp;
    g.kchunk = sp > 1 ? kSkMaxK : cdiv(K, 16) * 16;
    const bool av = k_vec(a, sa_m, sa_k, sa_b, K), bv = k_vec(b, sb_n, sb_k, sb_b, K);
    const dim3 grid(cdiv(N, 16), batch, sp);
    if (av && bv) hipLaunchKernelGGL((gemm_skinny_kernel<true, true>), grid, dim3(kSkT), 0, st, g);
    else if (av) hipLaunchKernelGGL((gemm_skinny_kernel<true, false>), grid, dim3(kSkT), 0, st, g);
    else if (bv) hipLaunchKernelGGL((gemm_skinny_kernel<false, true>), grid, dim3(kSkT), 0, st, g);
    else hipLaunchKernelGGL((gemm_skinny_kernel<false, false>), grid, dim3(kSkT), 0, st, g);
    MTX_LAUNCHED();
    return sp > 1 ? launch_splitk_reduce(g, st) : MTX_OK;
  }
  const bool ak = sa_k == 1, bn1 = sb_n == 1;
  const bool split3 = use_x3(M, N, K, batch);
  Plan p = split3 ? plan_x3(M, N, K, batch, workspace ? workspace_bytes : 0, ak, colsum != nullptr)
                  : plan_gemm(M, N, K, batch, workspace ? workspace_bytes : 0);
  g.ksplit = p.ksplit;
  g.kchunk = p.kchunk;
  g.fast = split3 && two_pieces(g);
  {
    const int64_t far = (int64_t)1 << 25;
    const bool x_ok = !act || !aux || (sx_n == 1 && sx_m >= N && sx_m < far);
    g.rows_vec = p.ksplit > 1 ? N < far : sc_n == 1 && sc_m >= N && sc_m < far && x_ok;
  }
  int rc = split3 ? launch_x3(g, p.bn, ak, bn1, st)
                  : (p.bm == 128) ? launch_tile<128, 128>(g, ak, bn1, st) : launch_tile<64, 64>(g, ak, bn1, st);
  if (rc) return rc;
  return p.ksplit > 1 ? launch_splitk_reduce(g, st) : MTX_OK;
}
}  // namespace

extern "C" int mtx_gemm_f32(int M, int N, int K, int batch,
                            float alpha, const float* a, int64_t sa_m, int64_t sa_k, int64_t sa_b,
                            const float* b, int64_t sb_k, int64_t sb_n, int64_t sb_b,
                            float beta, float* c, int64_t sc_m, int64_t sc_n, int64_t sc_b,
                            const float* bias, void* workspace, size_t workspace_bytes,
                            void* stream) {
  return gemm_impl(M, N, K, batch, alpha, a, sa_m, sa_k, sa_b, b, sb_k, sb_n, sb_b, beta, c, sc_m, sc_n, sc_b,
                   bias, 0, nullptr, 0, 0, 0, workspace, workspace_bytes, stream);
}

// workgroups a mtx_gemm_ln_f32 product aims at (by splitting K)
constexpr int kLnWgs = 144;

// The split-K product of mtx_gemm_ln_f32 / mtx_gemm_partials_f32: K cut into
// 2..8 ranges of whole 16-wide slices, as many as bring the launch to about
// kLnWgs workgroups (a projection to N = 384 has only 24 column tiles;
// measured at C4: 96 workgroups 0.327, 144 0.315, 192 0.313-0.317 ms per
// token step against 0.340 with mtx_gemm_f32's ranges); range s's partial
// product A[:, range] @ B[range, :] goes to g.ws + s*M*N.  Sets g.ksplit and
// g.kchunk.
void launch_ln_partials(GemmArgs& g, hipStream_t st) {
  const int want = std::min(kSkMaxSplit, std::max({2, skinny_splits(g.M, g.K), cdiv(kLnWgs, cdiv(g.N, 16))}));
  g.kchunk = cdiv(cdiv(g.K, want), 16) * 16;
  g.ksplit = cdiv(g.K, g.kchunk);
  g.nc = g.N;
  g.to_ws = 1;
  const bool av = k_vec(g.a, g.sam, g.sak, 0, g.K), bv = k_vec(g.b, g.sbn, g.sbk, 0, g.K);
  const dim3 grid(cdiv(g.N, 16), 1, g.ksplit);
  if (av && bv) hipLaunchKernelGGL((gemm_skinny_kernel<true, true>), grid, dim3(kSkT), 0, st, g);
  else if (av) hipLaunchKernelGGL((gemm_skinny_kernel<true, false>), grid, dim3(kSkT), 0, st, g);
  else if (bv) hipLaunchKernelGGL((gemm_skinny_kernel<false, true>), grid, dim3(kSkT), 0, st, g);
  else hipLaunchKernelGGL((gemm_skinny_kernel<false, false>), grid, dim3(kSkT), 0, st, g);
}

extern "C" size_t mtx_gemm_ln_workspace_bytes(int M, int N, int K) {
  if (M < 1 || N < 1 || K < 1 || skinny_splits(M, K) == 0) return 0;
  return (size_t)kSkMaxSplit * M * N * sizeof(float);
}

extern "C" int mtx_gemm_ln_f32(int M, int N, int K, float alpha, const float* a, int64_t sa_m, int64_t sa_k,
                               const float* b, int64_t sb_k, int64_t sb_n, float beta, float* c, int64_t sc_m,
                               const float* bias, const float* ln_gamma, const float* ln_beta, float eps, float* y,
                               int64_t ldy, void* workspace, size_t workspace_bytes, void* stream) {
  MTX_CHECK_SHAPE(M >= 1 && N >= 1 && K >= 1, "gemm_ln: sizes must be >= 1");
  MTX_CHECK_SHAPE(M <= kSkMaxM && K <= kSkMaxK * kSkMaxSplit && N <= 64 * 32,
                  "gemm_ln: needs M <= %d, K <= %d and N <= 2048 (got M=%d, N=%d, K=%d)", kSkMaxM,
                  kSkMaxK * kSkMaxSplit, M, N, K);
  MTX_CHECK_ARG(a && b && c && ln_gamma && ln_beta && y, "gemm_ln: null pointer");
  MTX_CHECK_ARG(sa_k == 1 || sa_m == 1, "gemm_ln: A needs a unit stride along m or k");
  MTX_CHECK_ARG(sb_n == 1 || sb_k == 1, "gemm_ln: B needs a unit stride along k or n");
  MTX_CHECK_ARG(sc_m >= N && ldy >= N, "gemm_ln: C and y rows must hold N values");
  MTX_CHECK_ARG((y >= c + (int64_t)(M - 1) * sc_m + N) || (c >= y + (int64_t)(M - 1) * ldy + N),
                "gemm_ln: y must not overlap C");
  const size_t need = mtx_gemm_ln_workspace_bytes(M, N, K);
  MTX_CHECK_ARG(workspace && workspace_bytes >= need, "gemm_ln: workspace too small (%zu < %zu)", workspace_bytes,
                need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  GemmArgs g{a, sa_m, sa_k, 0, b, sb_k, sb_n, 0, c, sc_m, 1, 0, bias,
             static_cast<float*>(workspace), M, N, K, 1, 0, 0, alpha, beta};
  launch_ln_partials(g, st);
  MTX_LAUNCHED();
  const int vpl = cdiv(N, 64);
  if (vpl <= 1) launch_reduce_ln<1>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 2) launch_reduce_ln<2>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 4) launch_reduce_ln<4>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 6) launch_reduce_ln<6>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 8) launch_reduce_ln<8>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 12) launch_reduce_ln<12>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else if (vpl <= 16) launch_reduce_ln<16>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  else launch_reduce_ln<32>(g, ln_gamma, ln_beta, eps, y, ldy, st);
  MTX_LAUNCHED();
  return MTX_OK;
}

extern "C" int mtx_gemm_partials_f32(int M, int N, int K, const float* a, int64_t sa_m, int64_t sa_k,
                                     const float* b, int64_t sb_k, int64_t sb_n, void* workspace,
                                     size_t workspace_bytes, int* nsplit, void* stream) {
  MTX_CHECK_SHAPE(M >= 1 && N >= 1 && K >= 1, "gemm_partials: sizes must be >= 1");
  MTX_CHECK_SHAPE(M <= kSkMaxM && K <= kSkMaxK * kSkMaxSplit && N <= 64 * 32,
                  "gemm_partials: needs M <= %d, K <= %d and N <= 2048 (got M=%d, N=%d, K=%d)", kSkMaxM,
                  kSkMaxK * kSkMaxSplit, M, N, K);
  MTX_CHECK_ARG(a && b && nsplit, "gemm_partials: null pointer");
  MTX_CHECK_ARG(sa_k == 1 || sa_m == 1, "gemm_partials: A needs a unit stride along m or k");
  MTX_CHECK_ARG(sb_n == 1 || sb_k == 1, "gemm_partials: B needs a unit stride along k or n");
  const size_t need = mtx_gemm_ln_workspace_bytes(M, N, K);
  MTX_CHECK_ARG(workspace && workspace_bytes >= need, "gemm_partials: workspace too small (%zu < %zu)",
                workspace_bytes, need);
  GemmArgs g{a, sa_m, sa_k, 0, b, sb_k, sb_n, 0, nullptr, N, 1, 0, nullptr,
             static_cast<float*>(workspace), M, N, K, 1, 0, 0, 1.f, 0.f};
  launch_ln_partials(g, static_cast<hipStream_t>(stream));
  MTX_LAUNCHED();
  *nsplit = g.ksplit;
  return MTX_OK;
}

extern "C" int mtx_gemm_act_f32(int M, int N, int K, int batch,
                                float alpha, const float* a, int64_t sa_m, int64_t sa_k, int64_t sa_b,
                                const float* b, int64_t sb_k, int64_t sb_n, int64_t sb_b,
                                float beta, float* c, int64_t sc_m, int64_t sc_n, int64_t sc_b,
                                const float* bias, int act, float* aux, int64_t sx_m, int64_t sx_n,
                                int64_t sx_b, void* workspace, size_t workspace_bytes, void* stream) {
  MTX_CHECK_ARG(act == 0 || act == 1 || act == 2 || act == 4,
                "gemm_act: act=%d must be 0 (none), 1 (GELU), 2 (GELU backward) or 4 (add aux)", act);
  MTX_CHECK_ARG(act != 2 || aux != nullptr, "gemm_act: act 2 needs the pre-activation aux");
  MTX_CHECK_ARG(act != 4 || (aux != nullptr && aux != c), "gemm_act: act 4 needs a residual aux other than C");
  MTX_CHECK_ARG(sx_m >= 0 && sx_n >= 0 && sx_b >= 0, "gemm_act: negative aux stride");
  return gemm_impl(M, N, K, batch, alpha, a, sa_m, sa_k, sa_b, b, sb_k, sb_n, sb_b, beta, c, sc_m, sc_n, sc_b,
                   bias, act, act ? aux : nullptr, sx_m, sx_n, sx_b, workspace, workspace_bytes, stream);
}

extern "C" int mtx_gemm_wgrad_f32(int M, int N, int K, const float* a, int64_t sa_m, int64_t sa_k,
                                  const float* b, int64_t sb_k, int64_t sb_n, float beta, float* c, int64_t sc_m,
                                  int64_t sc_n, float* dbias, int dbias_accumulate, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  MTX_CHECK_ARG(dbias != nullptr, "gemm_wgrad: null dbias (use mtx_gemm_f32 without a bias gradient)");
  MTX_CHECK_SHAPE(M >= 1 && N >= 1 && K >= 0, "gemm_wgrad: sizes must be M, N >= 1, K >= 0");
  return gemm_impl(M, N, K, 1, 1.f, a, sa_m, sa_k, 0, b, sb_k, sb_n, 0, beta, c, sc_m, sc_n, 0, nullptr, 0,
                   nullptr, 0, 0, 0, workspace, workspace_bytes, stream, dbias, dbias_accumulate ? 1 : 0);
}

extern "C" int mtx_gemm_step_f32(int M, int N, int K, const float* a, int64_t lda, const float* b, int64_t ldb,
                                 float beta, float* c, int64_t ldc, const float* bias, int act, int ncols_c,
                                 float* kcache, float* vcache, int64_t cache_stride_b, int64_t cache_stride_t,
                                 int T, const int* lengths, void* stream) {
  MTX_CHECK_SHAPE(M >= 1 && N >= 1 && K >= 1, "gemm_step: sizes must be >= 1");
  MTX_CHECK_SHAPE(use_skinny(M, K), "gemm_step: needs M <= %d and K <= %d (got M=%d, K=%d)", kSkMaxM, kSkMaxK,
                  M, K);
  MTX_CHECK_ARG(a && b && (ncols_c == 0 || c), "gemm_step: null operand");
  MTX_CHECK_ARG(act == 0 || act == 1, "gemm_step: act must be 0 (none) or 1 (gelu)");
  MTX_CHECK_ARG(ncols_c >= 0 && ncols_c <= N, "gemm_step: ncols_c %d not in [0, N=%d]", ncols_c, N);
  MTX_CHECK_ARG(lda >= K && ldb >= N && (ncols_c == 0 || ldc >= ncols_c), "gemm_step: row strides too small");
  if (ncols_c < N) {
    MTX_CHECK_ARG((N - ncols_c) % 2 == 0, "gemm_step: the cache columns must split evenly into k and v");
    MTX_CHECK_ARG(kcache && vcache && lengths, "gemm_step: null cache or lengths");
    MTX_CHECK_ARG(T >= 1 && cache_stride_t >= (N - ncols_c) / 2 && cache_stride_b >= (int64_t)T * cache_stride_t,
                  "gemm_step: cache strides do not hold (B, T, C) rows");
  }
  GemmArgs g{a, lda, 1, 0, b, ldb, 1, 0, c, ldc, 1, 0, bias, nullptr, M, N, K, 1, 1, cdiv(K, 16) * 16, 1.f, beta};
  g.act = act;
  g.nc = ncols_c;
  g.kc = kcache;
  g.vc = vcache;
  g.csb = cache_stride_b;
  g.cst = cache_stride_t;
  g.cT = T;
  g.lengths = lengths;
  const bool av = k_vec(a, lda, 1, 0, K);
  const dim3 grid(cdiv(N, 16), 1);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (av) hipLaunchKernelGGL((gemm_skinny_kernel<true, false>), grid, dim3(kSkT), 0, st, g);
  else hipLaunchKernelGGL((gemm_skinny_kernel<false, false>), grid, dim3(kSkT), 0, st, g);
  MTX_LAUNCHED();
  return MTX_OK;
}
