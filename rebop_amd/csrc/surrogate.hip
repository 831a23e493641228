// surrogate.hip -- kernels of the learned surrogate of the SSA.
//
// A multilayer perceptron maps (log rate constants, initial counts, t) of a
// Michaelis-Menten network to a K-component mixture per species (negative
// binomials, and binomials on the species' bound).  Its dense layers run on
// the matrix cores: BF16 operands, FP32
// accumulation (v_mfma_f32_16x16x32_bf16).  The loss head (mixture negative
// log-likelihood of the SSA samples and its gradient) runs in FP64.  Adam
// keeps FP32 master weights and writes the BF16 copy the GEMMs read.
//
// MFMA operand layout used below (16x16x32, wave64): lane l supplies
//   A[row = l % 16][k = 8 (l / 16) .. +8]   (8 bf16, k contiguous)
//   B[k = 8 (l / 16) .. +8][col = l % 16]
// and receives D[row = 4 (l / 16) + q][col = l % 16], q = 0..3.
// The GEMM test checks the product against a CPU reference.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "../../include/rebop_surrogate.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace sg {

// ---------------------------------------------------------------------------
// C = op(A) op(B), M x N x K, FP32 out.  !TA: A[m][k] (lda); TA: A stored
// [k][m].  !TB: B[k][n] (ldb); TB: B stored [n][k].  Tiles TM x TN x 32 (TM,
// TN = 64 or 128), four waves in 2 x 2, each (TM/2) x (TN/2) of 16 x 16 MFMA
// tiles: a 128 x 128 tile issues 16 MFMAs per wave per 8 fragment loads.
// M, N multiples of the tile, K of 32.  With gridDim.z > 1 (split K), block z
// covers k in [z*K/gz, (z+1)*K/gz) and adds its partial product into C
// (zeroed beforehand) atomically.  FUSED (gridDim.z == 1): instead of C, the
// epilogue writes act(C + bias) as BF16 to epi.H and/or FP32 to epi.F -- the
// arithmetic of bias_act_kernel on the same FP32 values, so the same bits,
// without the FP32 product's round trip through memory.
struct Epilogue {
  const float *bias;
  int relu;
  __bf16 *H;
  int ldh;
  float *F;
  int ldf;
  bool wide;          // (gemm_nt_kernel) H and F may be written four columns at a time
  const __bf16 *mask; // (EPI_MASK) M x N activations, lead dimension ldh
  float *colsum;      // (EPI_MASK) [M / 64][ldc]: the column sums of each 64 rows
  int ldc;
};
enum { EPI_PLAIN, EPI_BIAS, EPI_MASK };

template <bool TA, bool TB, int TM, int TN, bool FUSED>
__global__ void __launch_bounds__(256) gemm_kernel(int M, int N, int K, const __bf16 *__restrict__ A,
                                                   int lda, const __bf16 *__restrict__ B, int ldb,
                                                   float *__restrict__ C, int ldc, Epilogue epi) {
  constexpr int FM = TM / 32, FN = TN / 32; // 16-row fragments per wave
  __shared__ __attribute__((aligned(16))) __bf16 As[TM][40]; // [m][k], rows padded to 80 B
  __shared__ __attribute__((aligned(16))) __bf16 Bs[TN][40]; // [n][k]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
  floatx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int ksplit = K / (int)gridDim.z; // a multiple of 32 (checked by the host)
  const int kbeg = (int)blockIdx.z * ksplit, kend = kbeg + ksplit;
  for (int k0 = kbeg; k0 < kend; k0 += 32) {
#pragma unroll
    for (int p = 0; p < TM / 64; ++p) {
      const int idx = tid + 256 * p;
      if (!TA) {
        const int r = idx >> 2, c = (idx & 3) * 8;
        *(bf16x8 *)&As[r][c] = *(const bf16x8 *)&A[(size_t)(m0 + r) * lda + k0 + c];
      } else {
        const int kk = idx / (TM / 8), c = (idx % (TM / 8)) * 8;
        const bf16x8 v = *(const bf16x8 *)&A[(size_t)(k0 + kk) * lda + m0 + c];
#pragma unroll
        for (int q = 0; q < 8; ++q) As[c + q][kk] = v[q];
      }
    }
#pragma unroll
    for (int p = 0; p < TN / 64; ++p) {
      const int idx = tid + 256 * p;
      if (TB) {
        const int r = idx >> 2, c = (idx & 3) * 8;
        *(bf16x8 *)&Bs[r][c] = *(const bf16x8 *)&B[(size_t)(n0 + r) * ldb + k0 + c];
      } else {
        const int kk = idx / (TN / 8), c = (idx % (TN / 8)) * 8;
        const bf16x8 v = *(const bf16x8 *)&B[(size_t)(k0 + kk) * ldb + n0 + c];
#pragma unroll
        for (int q = 0; q < 8; ++q) Bs[c + q][kk] = v[q];
      }
    }
    __syncthreads();
    bf16x8 a[FM], b[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) a[i] = *(const bf16x8 *)&As[wm + i * 16 + (lane & 15)][(lane >> 4) * 8];
#pragma unroll
    for (int j = 0; j < FN; ++j) b[j] = *(const bf16x8 *)&Bs[wn + j * 16 + (lane & 15)][(lane >> 4) * 8];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = m0 + wm + i * 16 + (lane >> 4) * 4 + q;
        const int col = n0 + wn + j * 16 + (lane & 15);
        if (FUSED) {
          float v = acc[i][j][q] + epi.bias[col];
          if (epi.relu) v = v > 0.f ? v : 0.f;
          if (epi.H) epi.H[(size_t)row * epi.ldh + col] = (__bf16)v;
          if (epi.F) epi.F[(size_t)row * epi.ldf + col] = v;
        } else if (gridDim.z == 1) {
          C[(size_t)row * ldc + col] = acc[i][j][q];
        } else {
          atomicAdd(&C[(size_t)row * ldc + col], acc[i][j][q]);
        }
      }
}

// v + (v of the lane CTRL pairs this one with), a DPP rotation of a row of 16
template <int CTRL>
__device__ __forceinline__ float dpp_addf(float v) {
  int w;
  __builtin_memcpy(&w, &v, 4);
  w = __builtin_amdgcn_mov_dpp(w, CTRL, 0xF, 0xF, false);
  float o;
  __builtin_memcpy(&o, &w, 4);
  return v + o;
}
__device__ __forceinline__ float row_sumf(float v) { // over a row of 16 lanes, on every lane
  v = dpp_addf<0x128>(v); // row_ror:8
  v = dpp_addf<0x124>(v);
  v = dpp_addf<0x122>(v);
  return dpp_addf<0x121>(v);
}

// The tile of this workgroup.  Consecutive workgroups go to different XCDs;
// taken in linear order the eight tiles of one block of rows would be read
// through eight L2 caches.  XCD x gets the x-th eighth of the tiles instead,
// so it reads its own rows of A (the rows it wrote in the layer before) and
// all of B.
__device__ __forceinline__ void xcd_tile(int &bx, int &by) {
  const int gx = (int)gridDim.x, total = gx * (int)gridDim.y;
  bx = (int)blockIdx.x;
  by = (int)blockIdx.y;
  if (total % 8 == 0) {
    const int lin = bx + gx * by, t = (lin & 7) * (total >> 3) + (lin >> 3);
    bx = t % gx;
    by = t / gx;
  }
}

// The same product for A [M][K] and B stored [N][K] (both k-contiguous, as
// the forward pass and the backward's dX use them).  Bound by the latency of
// its loads: a slice's MFMAs take a fraction of the time its loads need to
// arrive, so two 64-wide slices are under way in registers while a third is
// multiplied out of one of two LDS buffers, with one barrier per slice.  The
// MFMA of the fused epilogues takes B's rows as its first operand, so that a
// lane's four outputs are four consecutive columns of one row, written at
// once.  Same products and summation order per output as
// gemm_kernel<false, true>.
// EPI_BIAS: act(C + bias) as in gemm_kernel.  EPI_MASK: the ReLU derivative
// from the stored activation, epi.H = bf16(mask > 0 ? C : 0), and epi.colsum
// the FP32 sums of its columns (the bias gradient's parts).
// 4096 x 512 x 512: 8.4 us with bias and ReLU (one 32-wide slice ahead:
// 10.0 us), 8.7 us with mask and column sums (8.8 us for the product, 7.5 us
// for the mask and 20 us for the sums as passes of their own).
template <int TM, int TN, int EPI>
__global__ void __launch_bounds__(256) gemm_nt_kernel(int M, int N, int K, const __bf16 *__restrict__ A,
                                                      int lda, const __bf16 *__restrict__ B, int ldb,
                                                      float *__restrict__ C, int ldc, Epilogue epi) {
  constexpr int FM = TM / 32, FN = TN / 32, PA = TM / 32, PB = TN / 32, BK = 64;
  constexpr int LD = BK + 8; // 144 B: sixteen rows start in different banks
  __shared__ __attribute__((aligned(16))) __bf16 As[2][TM][LD];
  __shared__ __attribute__((aligned(16))) __bf16 Bs[2][TN][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int bx, by;
  xcd_tile(bx, by);
  const int m0 = by * TM, n0 = bx * TN;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
  floatx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int ksplit = K / (int)gridDim.z; // a multiple of 32 (checked by the host)
  const int kbeg = (int)blockIdx.z * ksplit, kend = kbeg + ksplit;
  const int nk = (ksplit + BK - 1) / BK;
  // thread tid moves the 8-element chunks tid + 256 p: row (chunk >> 3), k
  // (chunk & 7) * 8; past kend (half a slice) it stores zeros
  const int lr = tid >> 3, lc = (tid & 7) * 8;
  bf16x8 ra[2][PA], rb[2][PB];
  auto gload = [&](auto set, int it) {
    constexpr int q = decltype(set)::value;
    const int k = kbeg + it * BK + lc;
    const bool in = k < kend;
#pragma unroll
    for (int p = 0; p < PA; ++p)
      ra[q][p] = in ? *(const bf16x8 *)&A[(size_t)(m0 + lr + 32 * p) * lda + k] : bf16x8{};
#pragma unroll
    for (int p = 0; p < PB; ++p)
      rb[q][p] = in ? *(const bf16x8 *)&B[(size_t)(n0 + lr + 32 * p) * ldb + k] : bf16x8{};
  };
  auto lstore = [&](auto set) { // register set q goes to LDS buffer q
    constexpr int q = decltype(set)::value;
#pragma unroll
    for (int p = 0; p < PA; ++p) *(bf16x8 *)&As[q][lr + 32 * p][lc] = ra[q][p];
#pragma unroll
    for (int p = 0; p < PB; ++p) *(bf16x8 *)&Bs[q][lr + 32 * p][lc] = rb[q][p];
  };
  typedef std::integral_constant<int, 0> set0;
  typedef std::integral_constant<int, 1> set1;
  auto step = [&](auto set, auto other, int it) {
    constexpr int q = decltype(set)::value;
    if (it + 2 < nk) gload(set, it + 2);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 32) {
      bf16x8 a[FM], b[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = *(const bf16x8 *)&As[q][wm + i * 16 + (lane & 15)][kk + (lane >> 4) * 8];
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = *(const bf16x8 *)&Bs[q][wn + j * 16 + (lane & 15)][kk + (lane >> 4) * 8];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = EPI == EPI_PLAIN ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0)
                                       : __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    }
    if (it + 1 < nk) lstore(other); // that buffer's reads ended at the last barrier
    __syncthreads();
  };
  gload(set0{}, 0);
  if (nk > 1) gload(set1{}, 1);
  lstore(set0{});
  __syncthreads();
  for (int it = 0; it < nk; it += 2) {
    step(set0{}, set1{}, it);
    if (it + 1 < nk) step(set1{}, set0{}, it + 1);
  }

  floatx4 cs[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) cs[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (EPI == EPI_PLAIN) {
        const int row = m0 + wm + i * 16 + (lane >> 4) * 4, col = n0 + wn + j * 16 + (lane & 15);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float *o = &C[(size_t)(row + q) * ldc + col];
          if (gridDim.z == 1) *o = acc[i][j][q];
          else atomicAdd(o, acc[i][j][q]);
        }
      } else {
        const int row = m0 + wm + i * 16 + (lane & 15), col = n0 + wn + j * 16 + (lane >> 4) * 4;
        floatx4 v = acc[i][j];
        __bf16 h[4];
        if constexpr (EPI == EPI_MASK) {
          __bf16 mk[4];
          __builtin_memcpy(mk, __builtin_assume_aligned(&epi.mask[(size_t)row * epi.ldh + col], 8), sizeof mk);
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = (float)mk[q] > 0.f ? v[q] : 0.f;
          cs[j] += v;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v[q] += epi.bias[col + q];
            if (epi.relu) v[q] = v[q] > 0.f ? v[q] : 0.f;
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] = (__bf16)v[q];
        __bf16 *oh = epi.H + (size_t)row * epi.ldh + col;
        float *of = epi.F + (size_t)row * epi.ldf + col;
        if (EPI == EPI_MASK || epi.wide) {
          if (epi.H) __builtin_memcpy(__builtin_assume_aligned(oh, 8), h, sizeof h);
          if (EPI == EPI_BIAS && epi.F) *(floatx4 *)of = v;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (epi.H) oh[q] = h[q];
            if (epi.F) of[q] = v[q];
          }
        }
      }
    }
  if constexpr (EPI == EPI_MASK) {
    float(*red)[TN] = (float(*)[TN])As; // the last reads of As are behind a barrier
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float t = row_sumf(cs[j][q]);
        if ((lane & 15) == 0) red[wave >> 1][wn + j * 16 + (lane >> 4) * 4 + q] = t;
      }
    __syncthreads();
    // a wave covers TM / 2 rows
    if (tid < TN) {
      float *o = epi.colsum + (size_t)by * (TM / 64) * epi.ldc + n0 + tid;
      if constexpr (TM == 64) {
        *o = red[0][tid] + red[1][tid];
      } else {
        o[0] = red[0][tid];
        o[epi.ldc] = red[1][tid];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The weight gradients of every layer in one launch: dW_l = H_l^T dZ_l, H_l
// [B][m_l] and dZ_l [B][n_l] both with the contraction index b outermost.
// A workgroup takes a 64 x 64 tile of one layer and a range of the batch
// (split z), 64 rows at a time: a thread reads 8 columns of 4
// rows, transposes them with byte permutes, and writes 4 consecutive b of
// each column to LDS, from where the MFMA fragments are read.  The rows after
// the current ones are on their way in registers meanwhile.  A layer at a
// time would leave the chip a quarter full; all of them give 216 tiles (five
// layers, width 512).  Splits write their sums to part[z], which
// grad_reduce_kernel adds in order: no atomics, and the same bits every run.
// Bound by the latency of its loads and LDS accesses (the waves wait 45 % of
// their time; LDS instructions and their extra cycles take 15 % of the CU
// cycles).  Five layers of width 512, batch 4096: 23.7 us (a launch
// and a clear per layer with scattered LDS stores: 113 us; rows padded by four
// elements instead of the chunk permutation: 29.5 us).
constexpr int WG_MAXL = 8;
struct WgradNet {
  const __bf16 *H[WG_MAXL], *dZ[WG_MAXL];
  int n[WG_MAXL]; // multiples of 64, as the widths of H
  int ldh[WG_MAXL];
  int tile0[WG_MAXL];       // first tile of layer l
  size_t out[WG_MAXL];      // where dW_l starts, in floats
  int layers;
};

__global__ void __launch_bounds__(256) wgrad_kernel(int units, int splits, WgradNet net, float *__restrict__ part,
                                                    size_t stride) {
  // Rows of nine 16-byte chunks; chunk k of column c is stored at k ^ 2 (c / 16
  // % 4), so that the 32 lanes of a store, four b of columns 8 apart, meet
  // every bank once, as do 16 rows of a fragment.
  constexpr int LD = 72;
  __shared__ __attribute__((aligned(16))) __bf16 T[2][2][64][LD]; // [buffer][H, dZ][column][b]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the splits are a power of two and the fastest index, so consecutive
  // workgroups, which go to different XCDs, share a tile and an XCD keeps to
  // one range of the batch: a layer's operands over it fit its L2
  const int tile = (int)blockIdx.x / splits, z = (int)blockIdx.x % splits;
  const __bf16 *H = net.H[0], *Z = net.dZ[0];
  int n = net.n[0], ldh = net.ldh[0], t0 = 0;
  size_t out = net.out[0];
#pragma unroll
  for (int l = 1; l < WG_MAXL; ++l)
    if (l < net.layers && tile >= net.tile0[l]) {
      H = net.H[l];
      Z = net.dZ[l];
      n = net.n[l];
      ldh = net.ldh[l];
      t0 = net.tile0[l];
      out = net.out[l];
    }
  const int t = tile - t0, tn = n / 64, m0 = t / tn * 64, n0 = t % tn * 64;
  const int ubeg = (int)((int64_t)units * z / splits);
  const int uend = (int)((int64_t)units * (z + 1) / splits);
  const int side = tid >> 7, cg = tid & 7, kq = (tid & 127) >> 3;
  const size_t ld = side ? (size_t)n : (size_t)ldh;
  const __bf16 *src = (side ? Z + n0 : H + m0) + (size_t)(4 * kq) * ld + 8 * cg;
  uint32_t r[4][4];
  auto gload = [&](int u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 v = *(const uint4 *)(src + ((size_t)u * 64 + i) * ld);
      r[i][0] = v.x;
      r[i][1] = v.y;
      r[i][2] = v.z;
      r[i][3] = v.w;
    }
  };
  auto lstore = [&](int buf) {
    const int at = 4 * kq ^ 16 * (cg >> 1);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint2 lo, hi; // columns 2 w and 2 w + 1, rows 0..3
      lo.x = __builtin_amdgcn_perm(r[1][w], r[0][w], 0x05040100u);
      lo.y = __builtin_amdgcn_perm(r[3][w], r[2][w], 0x05040100u);
      hi.x = __builtin_amdgcn_perm(r[1][w], r[0][w], 0x07060302u);
      hi.y = __builtin_amdgcn_perm(r[3][w], r[2][w], 0x07060302u);
      *(uint2 *)&T[buf][side][8 * cg + 2 * w][at] = lo;
      *(uint2 *)&T[buf][side][8 * cg + 2 * w + 1][at] = hi;
    }
  };
  auto frag = [&](int buf, int s, int c, int k) { // 8 consecutive b of column c
    return *(const bf16x8 *)&T[buf][s][c][k ^ 16 * (c >> 4 & 3)];
  };
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  floatx4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  gload(ubeg);
  lstore(0);
  __syncthreads();
  int buf = 0;
  for (int u = ubeg; u < uend; ++u) {
    if (u + 1 < uend) gload(u + 1);
#pragma unroll
    for (int kk = 0; kk < 64; kk += 32) {
      bf16x8 h[2], z[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) h[i] = frag(buf, 0, wm + i * 16 + (lane & 15), kk + (lane >> 4) * 8);
#pragma unroll
      for (int j = 0; j < 2; ++j) z[j] = frag(buf, 1, wn + j * 16 + (lane & 15), kk + (lane >> 4) * 8);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(z[j], h[i], acc[i][j], 0, 0, 0);
    }
    if (u + 1 < uend) lstore(buf ^ 1); // that buffer's reads ended at the last barrier
    __syncthreads();
    buf ^= 1;
  }
  float *o = part + stride * z + out;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = m0 + wm + i * 16 + (lane & 15), col = n0 + wn + j * 16 + (lane >> 4) * 4;
      *(floatx4 *)&o[(size_t)row * n + col] = acc[i][j];
    }
}

// The head's gradient as the backward pass reads it: dZ = bf16(g) and the
// column sums of each 64 rows, 64 x 64 per workgroup.
__global__ void __launch_bounds__(256) head_grad_kernel(int N, const float *__restrict__ g, int ldg,
                                                        __bf16 *__restrict__ dZ, float *__restrict__ colsum,
                                                        int ldc) {
  __shared__ float red[16][64];
  const int c4 = (threadIdx.x & 15) * 4, rg = threadIdx.x >> 4;
  const int n = blockIdx.x * 64 + c4;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const size_t row = (size_t)blockIdx.y * 64 + rg + 16 * i;
    __bf16 h[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v = g[row * ldg + n + q];
      s[q] += v;
      h[q] = (__bf16)v;
    }
    __builtin_memcpy(&dZ[row * N + n], h, sizeof h);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) red[rg][c4 + q] = s[q];
  __syncthreads();
  if (threadIdx.x < 64) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[i][threadIdx.x];
    colsum[(size_t)blockIdx.y * ldc + blockIdx.x * 64 + threadIdx.x] = t;
  }
}

// grads[0, weights) = the sum of the splits' parts (splits > 1: else they are
// in place), 1024 floats per workgroup; then the bias gradients, 64 per
// workgroup, from the column sums [rows][nbias] of every layer side by side.
__global__ void __launch_bounds__(256) grad_reduce_kernel(int splits, size_t weights, size_t stride,
                                                          const float *__restrict__ part, int nbias,
                                                          int rows, const float *__restrict__ colsum,
                                                          float *__restrict__ grads) {
  const unsigned wblk = splits > 1 ? (unsigned)(weights / 1024) : 0u;
  if (blockIdx.x < wblk) {
    const size_t i = (size_t)blockIdx.x * 1024 + threadIdx.x * 4;
    floatx4 v = *(const floatx4 *)&part[i];
    for (int z = 1; z < splits; ++z) v += *(const floatx4 *)&part[stride * z + i];
    *(floatx4 *)&grads[i] = v;
    return;
  }
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int n = (int)(blockIdx.x - wblk) * 64 + c;
  float s = 0.f;
  if (n < nbias)
#pragma unroll 8
    for (int m = g; m < rows; m += 4) s += colsum[(size_t)m * nbias + n];
  red[g][c] = s;
  __syncthreads();
  if (g == 0 && n < nbias) grads[weights + n] = red[0][c] + red[1][c] + red[2][c] + red[3][c];
}

__global__ void zero_kernel(int M, int N, float *__restrict__ C, int ldc) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (size_t)M * N) C[(i / N) * ldc + i % N] = 0.f;
}

// H = bf16(act(C + bias)), act = ReLU or identity; optionally the FP32 result too.
__global__ void bias_act_kernel(int M, int N, const float *__restrict__ C, int ldc,
                                const float *__restrict__ bias, int relu, __bf16 *__restrict__ H,
                                int ldh, float *__restrict__ F, int ldf) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)M * N) return;
  const int m = (int)(idx / N), n = (int)(idx % N);
  float v = C[(size_t)m * ldc + n] + bias[n];
  if (relu) v = v > 0.f ? v : 0.f;
  if (H) H[(size_t)m * ldh + n] = (__bf16)v;
  if (F) F[(size_t)m * ldf + n] = v;
}

// dZ = dH * (H > 0): the ReLU derivative from the stored activation; FP32 in
// place (for the bias gradient) and BF16 (for the next GEMMs).
__global__ void relu_grad_kernel(int M, int N, float *__restrict__ dH, int ldd,
                                 const __bf16 *__restrict__ H, int ldh, __bf16 *__restrict__ dZ,
                                 int ldz) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)M * N) return;
  const int m = (int)(idx / N), n = (int)(idx % N);
  const float h = (float)H[(size_t)m * ldh + n];
  const float g = h > 0.f ? dH[(size_t)m * ldd + n] : 0.f;
  dH[(size_t)m * ldd + n] = g;
  dZ[(size_t)m * ldz + n] = (__bf16)g;
}

// y[c][r] = bf16(x[r][c]) for an R x C matrix
__global__ void transpose_bf16_kernel(int R, int C, const float *__restrict__ x, __bf16 *__restrict__ y) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)R * C) return;
  const int r = (int)(i / C), c = (int)(i % C);
  y[(size_t)c * R + r] = (__bf16)x[i];
}

// Wp[k / 32][n][k % 32] = bf16(W[k][n]) for W [K][N] (K a multiple of 32)
__global__ void pack_kslices_kernel(int K, int N, const float *__restrict__ W, __bf16 *__restrict__ Wp) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)K * N) return;
  const int kk = (int)(i % 32), n = (int)((i / 32) % N), k = (int)(i / (32 * (size_t)N)) * 32 + kk;
  Wp[i] = (__bf16)W[(size_t)k * N + n];
}

__global__ void cast_bf16_kernel(size_t n, const float *__restrict__ x, __bf16 *__restrict__ y) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (__bf16)x[i];
}

// out[n] = sum_m X[m][n]: one thread per column, rows strided (coalesced).
// Column sums over a 2-D grid: block (x, y) sums columns 64x .. 64x+63 over
// rows 256y .. 256y+255 (four row groups of 64 in parallel, combined in LDS)
// and adds its partial sums into out (zeroed first) atomically.
__global__ void __launch_bounds__(256) colsum_kernel(int M, int N, const float *__restrict__ X,
                                                     int ldx, float *__restrict__ out) {
  __shared__ float part[4][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int n = blockIdx.x * 64 + c;
  const int m0 = blockIdx.y * 256 + g * 64;
  float s = 0.f;
  if (n < N)
    for (int m = m0; m < m0 + 64 && m < M; ++m) s += X[(size_t)m * ldx + n];
  part[g][c] = s;
  __syncthreads();
  if (g == 0 && n < N) atomicAdd(&out[n], part[0][c] + part[1][c] + part[2][c] + part[3][c]);
}

__global__ void fill_kernel(int n, float *__restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.f;
}

// Adam with FP32 master weights; writes the BF16 copy read by the GEMMs.
__global__ void adam_kernel(size_t n, float *__restrict__ w, const float *__restrict__ g,
                            float *__restrict__ m, float *__restrict__ v, __bf16 *__restrict__ wb,
                            float lr, float b1, float b2, float eps, float bc1, float bc2) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  w[i] = wi;
  if (wb) wb[i] = (__bf16)wi;
}

// Inputs of item b: (point p, sample i) -> the REBOP_SG_FEATURES features,
// scaled to about [-1, 1]: log10 of the rate constants, E0, S0, t, their
// logs, and the logs of the kinetics' dimensionless groups (kcat t, kf E0 t,
// kf S0 t, K_M / S0 with K_M = (kb + kcat) / kf, kb / kcat, E0 / S0,
// kcat E0 t / S0); e0, s0 = the counts that bound the species (E0 for E and
// ES, S0 for S and P; exact in FP32).
// The item's inputs: rate constants, the bounding counts and the sample time.
struct ItemInputs {
  double kf, kb, kc, e0, s0, t;
};

__device__ __forceinline__ ItemInputs item_inputs(uint32_t p, uint32_t i, const double *__restrict__ rates,
                                                  const int64_t *__restrict__ x0, double tmax, int nb_steps) {
#pragma clang fp contract(off)
  ItemInputs v;
  v.kf = rates[3 * p + 0];
  v.kb = rates[3 * p + 1];
  v.kc = rates[3 * p + 2];
  v.e0 = (double)x0[4 * p + 0];
  v.s0 = (double)x0[4 * p + 1];
  v.t = tmax * (double)i / (double)nb_steps;
  return v;
}

// Log j of the seven the features use: log10 of kf, kb, kc, E0, S0, t and
// kb + kc.
__device__ __forceinline__ double item_log(const ItemInputs &v, int j) {
#pragma clang fp contract(off)
  switch (j) {
  case 0: return log10(v.kf);
  case 1: return log10(v.kb);
  case 2: return log10(v.kc);
  case 3: return log10(v.e0);
  case 4: return log10(v.s0);
  case 5: return log10(v.t);
  default: return log10(v.kb + v.kc);
  }
}

// Feature j (before the FP32 cast) from the inputs and their logs lg[0..6].
__device__ __forceinline__ double item_feature(const ItemInputs &v, const double *lg, double tmax, int j) {
#pragma clang fp contract(off)
  const double lf = lg[0], lb = lg[1], lc = lg[2], le = lg[3], ls = lg[4], lt = lg[5];
  switch (j) {
  case 0: return (lf + 1.0) * 0.5;
  case 1: return (lb + 1.0) * 0.5;
  case 2: return (lc + 1.0) * 0.5;
  case 3: return (v.e0 - 105.0) / 95.0;
  case 4: return (v.s0 - 525.0) / 475.0;
  case 5: return 2.0 * v.t / tmax - 1.0;
  case 6: return (le - 1.65) / 0.65;
  case 7: return (ls - 2.35) / 0.65;
  case 8: return (lt - 0.95) / 0.75;
  case 9: return (lc + lt) / 3.0;
  case 10: return (lf + le + lt - 1.6) / 3.4;
  case 11: return (lf + ls + lt - 2.3) / 3.4;
  case 12: return ((lg[6] - lf) - ls + 2.05) / 4.65; // K_M = (kb + kcat) / kf
  case 13: return (lb - lc) / 4.0;
  case 14: return (le - ls + 0.7) / 1.3;
  default: return (lc + le + lt - ls + 0.75) / 4.05;
  }
}

// X[b][0..ldx) = item b's features, then zeros; bound[b][s] (nullable) = the
// count that bounds species s (E = E0 - ES, S <= S0, ES <= E0, P <= S0).
// Four threads per item: thread q computes logs 2q and 2q + 1 (of seven),
// which the four share through LDS, and features 4q .. 4q+3.  A thread per
// item took seven logarithms in a row on 16 workgroups and wrote its row two
// bytes at a time (4096 items: 13.1 us, now 4.8 us).  wide: rows of X may be
// written eight bytes at a time.
__global__ void __launch_bounds__(256) features_kernel(int B, const uint32_t *__restrict__ item_point,
                                                       const uint32_t *__restrict__ item_sample,
                                                       const double *__restrict__ rates,
                                                       const int64_t *__restrict__ x0, double tmax, int nb_steps,
                                                       __bf16 *__restrict__ X, int ldx, float *__restrict__ bound,
                                                       bool wide) {
  static_assert(REBOP_SG_FEATURES == 16, "four threads x four features per item");
  __shared__ double lg[64][9]; // rows 72 B apart
  const int row = threadIdx.x >> 2, q = threadIdx.x & 3;
  const int b = blockIdx.x * 64 + row;
  ItemInputs v{1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
  if (b < B) v = item_inputs(item_point[b], item_sample[b], rates, x0, tmax, nb_steps);
  lg[row][2 * q] = item_log(v, 2 * q);
  if (q < 3) lg[row][2 * q + 1] = item_log(v, 2 * q + 1);
  __syncthreads();
  if (b >= B) return;
  __bf16 h[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) h[j] = (__bf16)(float)item_feature(v, lg[row], tmax, 4 * q + j);
  __bf16 *x = X + (size_t)b * ldx;
  if (wide) {
    const __bf16 z[4] = {};
    __builtin_memcpy(__builtin_assume_aligned(x + 4 * q, 8), h, sizeof h);
    for (int c = REBOP_SG_FEATURES + 4 * q; c < ldx; c += 16)
      __builtin_memcpy(__builtin_assume_aligned(x + c, 8), z, sizeof z);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[4 * q + j] = h[j];
    for (int c = REBOP_SG_FEATURES + q; c < ldx; c += 4) x[c] = (__bf16)0.f;
  }
  if (bound) bound[4 * (size_t)b + q] = (float)(q & 1 ? v.s0 : v.e0);
}

// head[b][s*3K + K + c] += ln bound[b][s] for the negative-binomial
// components c < K/2: their log means (the binomial components' logits stay).
__global__ void head_offsets_kernel(int B, int S, int K, float *__restrict__ head, int ldh,
                                    const float *__restrict__ bound) {
  const int half = K / 2;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= B * S * half) return;
  const int b = idx / (S * half), s = (idx / half) % S, c = idx % half;
  head[(size_t)b * ldh + (size_t)s * 3 * K + K + c] += logf(bound[(size_t)b * S + s]);
}

// ---------------------------------------------------------------------------
// Inference through the whole network in one launch.  A workgroup of eight
// waves takes 128 items, whose activations stay in LDS (128 rows of up to 512
// BF16, stored in MFMA fragment order: see hs_offset) from the input layer
// to the last hidden layer: HBM sees the inputs and the head only.  Wave w computes
// all 128 rows and columns (N / 8) w .. +N/8 of each layer, so each weight
// fragment is fetched once per workgroup.  The weights come straight from
// global memory (every workgroup reads the same ones, so they stay in L2) in
// the k-slice-major layout Wp[k / 32][n][k % 32] (rebop_sg_pack_kslices_bf16):
// a wave's fragment of one 32-wide slice is 1 KB of consecutive bytes.  The
// MFMA takes the weights as A and the activations as B, so a lane's four
// outputs are four consecutive columns of one row (one 8-byte LDS store per
// fragment).  Per output, the arithmetic is gemm_nt_kernel's: the same
// 16x16x32 MFMAs over k slices 0, 32, 64, ... (a product of two BF16 values
// is exact in FP32, so which operand is A does not matter), then + bias,
// ReLU and the BF16 cast -- the bits of the layer-by-layer forward pass.
// FEAT: the input layer is item_feature of items m0.. (columns >=
// REBOP_SG_FEATURES zero) and the last layer adds head_offsets_kernel's
// ln bound terms, so one launch turns (point, sample) items into mixture
// parameters; otherwise X [M][ldx] is the input.
constexpr int MLP_BM = 128, MLP_MAXW = 512, MLP_MAXL = 8;
constexpr int MLP_HEAD_LD = 128 * 4 + 16; // bytes per row of a staged 128-column head

// Byte offset of activation (m, n) in LDS.  Fragment order: the 16 x 32
// block of rows 16 (m / 16).. and columns 32 (n / 32).. is 1 KB, in which
// lane l's B operand (row l % 16, columns 8 (l / 16) .. +8 of the block)
// is 16 consecutive bytes at 16 l -- so a wave's fragment read is 1 KB of
// consecutive bytes, free of bank conflicts.  Row blocks are 16 KB apart
// (512 columns).
__device__ __forceinline__ uint32_t hs_offset(int m, int n) {
  return (uint32_t)(((m >> 4) * (MLP_MAXW / 32) + (n >> 5)) * 1024 + ((m & 15) + 16 * ((n & 31) >> 3)) * 16 +
                    (n & 7) * 2);
}

struct MlpNet {
  const __bf16 *Wp[MLP_MAXL]; // layer l: [dims[l] / 32][dims[l+1]][32]
  const float *bias[MLP_MAXL];
  int dims[MLP_MAXL + 1]; // dims[0] multiple of 64 up to 512, the others 128, 256 or 512
  int depth;
};

struct MlpItems {
  const uint32_t *item_point, *item_sample;
  const double *rates;
  const int64_t *x0;
  double tmax;
  int nb_steps;
};

// Layer l's table entries, selected without indexing the argument block (a
// runtime index would copy it to scratch memory).
__device__ __forceinline__ int net_dim(const MlpNet &net, int l) {
  int v = net.dims[0];
#pragma unroll
  for (int j = 1; j <= MLP_MAXL; ++j)
    if (j == l) v = net.dims[j];
  return v;
}
__device__ __forceinline__ const __bf16 *net_weights(const MlpNet &net, int l) {
  const __bf16 *v = net.Wp[0];
#pragma unroll
  for (int j = 1; j < MLP_MAXL; ++j)
    if (j == l) v = net.Wp[j];
  return v;
}
__device__ __forceinline__ const float *net_bias(const MlpNet &net, int l) {
  const float *v = net.bias[0];
#pragma unroll
  for (int j = 1; j < MLP_MAXL; ++j)
    if (j == l) v = net.bias[j];
  return v;
}

// NB: 16-column fragments per wave (N = 128 NB); KT: the input width when it
// is known at compile time (the k loop is then unrolled whole, which spares
// the loop header's wait for every outstanding load and the loads past the
// last slice), else 0.
template <int NB, int KT>
__device__ __forceinline__ void mlp_layer(const __bf16 *__restrict__ Wp, const float *__restrict__ bias,
                                          int Kr, bool last, char *Hs, const float (*lnb)[4],
                                          int m0, int M, float *__restrict__ out, int ldo) {
  constexpr int N = 128 * NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int K = KT ? KT : Kr, n0 = wave * 16 * NB;
  // fragment c of the slice at k: Wp[k N + lane_off + 512 c .. +8]
  const uint32_t lane_off = (uint32_t)(n0 + (lane & 15)) * 32u + (uint32_t)(lane >> 4) * 8u;
  auto wload = [&](bf16x8 &dst, int c, int k) {
    // a wave-uniform base (scalar registers) plus the lane's fixed offset,
    // so the unrolled loop needs no vector register per address
    const __bf16 *base = Wp + ((size_t)k * N + (size_t)c * 512);
    dst = *(const bf16x8 *)(base + lane_off);
  };
  // Row fragment r at k: byte offset hb[r / 4] + (16 (r % 4) + k / 32) 1024
  // in Hs.  Rows 64.. get a base register of their own (kept opaque to the
  // compiler) so that every offset fits a DS instruction's 16-bit immediate:
  // one address register for the unrolled loop instead of one per load.
  const uint32_t hb0 = (uint32_t)lane * 16u;
  uint32_t hb1 = hb0 + 4u * 16u * 1024u;
  asm volatile("" : "+v"(hb1));
  auto hload = [&](bf16x8 &dst, int r, int k) {
    const uint32_t off = (r < 4 ? hb0 : hb1) + (uint32_t)((r & 3) * 16 + (k >> 5)) * 1024u;
    dst = *(const bf16x8 *)(Hs + off);
  };
  floatx4 acc[NB][8];
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[c][r] = floatx4{0.f, 0.f, 0.f, 0.f};
  // Software pipeline, fixed with scheduling barriers (left alone, the
  // compiler sinks each load to just before its use): row fragment r of the
  // next slice loads as soon as the MFMAs of this slice have read slot r, and
  // weight fragments load after the first row block of a slice into a set of
  // registers of their own: for the slice after next when the k loop is
  // unrolled (three sets), for the next slice otherwise (two sets).
  bf16x8 h[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) hload(h[r], r, 0);
  if constexpr (KT != 0) {
    constexpr int NS = KT / 32;
    bf16x8 w[3][NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      wload(w[0][c], c, 0);
      if (NS > 1) wload(w[1][c], c, 32);
    }
#pragma unroll
    for (int sl = 0; sl < NS; ++sl) {
      // no loads past the last slice (compile-time conditions: nothing is
      // left in flight for the barrier at the end of the layer to wait for)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
#pragma unroll
        for (int c = 0; c < NB; ++c)
          acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[sl % 3][c], h[r], acc[c][r], 0, 0, 0);
        if (sl + 1 < NS) hload(h[r], r, (sl + 1) * 32);
        if (r == 0 && sl + 2 < NS) {
#pragma unroll
          for (int c = 0; c < NB; ++c) wload(w[(sl + 2) % 3][c], c, (sl + 2) * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    bf16x8 wa[NB], wb[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) wload(wa[c], c, 0);
    auto slice = [&](const bf16x8(&w)[NB], bf16x8(&wn)[NB], int kn) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
#pragma unroll
        for (int c = 0; c < NB; ++c) acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c], h[r], acc[c][r], 0, 0, 0);
        hload(h[r], r, kn);
        if (r == 0) {
#pragma unroll
          for (int c = 0; c < NB; ++c) wload(wn[c], c, kn);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for (int k0 = 0; k0 < K; k0 += 64) { // K is a multiple of 64
      slice(wa, wb, k0 + 32);
      // the last slice's loads fetch that slice again (no branch in the loop)
      slice(wb, wa, k0 + 64 < K ? k0 + 64 : k0 + 32);
    }
  }
  __syncthreads(); // every wave has read this layer's input
  // The epilogue's indices derive from an opaque copy of the lane id: left
  // alone, the compiler computes them for every layer variant up front and
  // keeps them in scratch memory across the k loops (spill traffic in HBM).
  int le = lane;
  asm volatile("" : "+v"(le));
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int n = n0 + c * 16 + (le >> 4) * 4;
    const floatx4 b = *(const floatx4 *)&bias[n];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int m = r * 16 + (le & 15);
      floatx4 v;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = acc[c][r][q] + b[q];
      if (!last) {
        __bf16 hv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) hv[q] = (__bf16)(v[q] > 0.f ? v[q] : 0.f);
        __builtin_memcpy(Hs + hs_offset(m, n), hv, sizeof hv);
      } else {
        if (lnb) {
          // head_offsets_kernel: + ln bound[s] on the negative-binomial log
          // means, columns s*3K + K + c for c < K/2
          constexpr int KC = REBOP_SG_COMPONENTS;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int s = (n + q) / (3 * KC), j = (n + q) % (3 * KC);
            if (s < 4 && j >= KC && j < KC + KC / 2) v[q] += lnb[m][s];
          }
        }
        if constexpr (NB == 1) {
          // a head of 128 columns goes through LDS (free now) so that the
          // stores below write whole rows
          *(floatx4 *)(Hs + m * MLP_HEAD_LD + n * 4) = v;
        } else if (m0 + m < M) {
          __builtin_nontemporal_store(v, (floatx4 *)&out[(size_t)(m0 + m) * ldo + n]);
        }
      }
    }
  }
  __syncthreads(); // the layer's output is whole before the next layer reads it
  if (NB == 1 && last) {
    // 128 rows x 512 B: a wave instruction stores two whole rows (full
    // cache lines, streaming: the head is not read again, and
    // write-allocated lines would push the weights out of L2)
    int te = tid;
    asm volatile("" : "+v"(te));
#pragma unroll
    for (int i = 0; i < MLP_BM * 32 / 512; ++i) {
      const int idx = te + 512 * i, m = idx >> 5, c4 = idx & 31;
      if (m0 + m < M)
        __builtin_nontemporal_store(*(const floatx4 *)(Hs + m * MLP_HEAD_LD + c4 * 16),
                                    (floatx4 *)&out[(size_t)(m0 + m) * ldo + c4 * 4]);
    }
  }
}

template <bool FEAT>
__global__ void __launch_bounds__(512) mlp_infer_kernel(int M, const __bf16 *__restrict__ X, int ldx,
                                                        MlpItems items, MlpNet net,
                                                        float *__restrict__ out, int ldo) {
  __shared__ __attribute__((aligned(16))) char Hs[MLP_BM * MLP_MAXW * 2];
  __shared__ float lnb[FEAT ? MLP_BM : 1][4];
  __shared__ double lg[FEAT ? MLP_BM : 1][8]; // the items' logs, shared by their four threads
  __shared__ __attribute__((aligned(16))) float Bs[MLP_MAXL * MLP_MAXW]; // every layer's bias
  const int tid = threadIdx.x, m0 = blockIdx.x * MLP_BM, K0 = net.dims[0];
  // every layer's bias: loaded into registers here, stored to LDS after the
  // inputs, so its latency overlaps theirs
  float bv[MLP_MAXL];
#pragma unroll
  for (int l = 0; l < MLP_MAXL; ++l)
    bv[l] = l < net.depth && tid < net.dims[l + 1] ? net.bias[l][tid] : 0.f;
  if (FEAT) {
    // four threads per item: thread q computes logs 2q, 2q+1 (of seven),
    // which the item's threads share through LDS, then features 4q .. 4q+3
    // (the arithmetic of item_feature, so the bits of features_kernel)
    static_assert(REBOP_SG_FEATURES == 16 && MLP_BM * 4 == 512, "four threads x four features per item");
    const int item = tid >> 2, q = tid & 3;
    ItemInputs v{1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
    if (m0 + item < M)
      v = item_inputs(items.item_point[m0 + item], items.item_sample[m0 + item], items.rates, items.x0,
                      items.tmax, items.nb_steps);
    lg[item][2 * q] = item_log(v, 2 * q);
    if (q < 3) lg[item][2 * q + 1] = item_log(v, 2 * q + 1);
    __syncthreads();
    double l7[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) l7[j] = lg[item][j];
    __bf16 h4[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float f = m0 + item < M ? (float)item_feature(v, l7, items.tmax, 4 * q + j) : 0.f;
      h4[j] = (__bf16)f;
    }
    __builtin_memcpy(Hs + hs_offset(item, 4 * q), h4, sizeof h4);
    const __bf16 z4[4] = {};
    for (int c = REBOP_SG_FEATURES + 4 * q; c < K0; c += 16) __builtin_memcpy(Hs + hs_offset(item, c), z4, sizeof z4);
    if (q == 0) {
      const float le = logf((float)v.e0), ls = logf((float)v.s0);
      lnb[item][0] = le;
      lnb[item][1] = ls;
      lnb[item][2] = le;
      lnb[item][3] = ls;
    }
  } else {
    // rows m0.. of X, 8 columns per thread and pass; rows past M read as zero
    const int per_row = K0 / 8;
    for (int idx = tid; idx < MLP_BM * per_row; idx += 512) {
      const int r = idx / per_row, c = (idx % per_row) * 8;
      bf16x8 v = {};
      if (m0 + r < M) v = *(const bf16x8 *)&X[(size_t)(m0 + r) * ldx + c];
      *(bf16x8 *)(Hs + hs_offset(r, c)) = v;
    }
  }
#pragma unroll
  for (int l = 0, o = 0; l < MLP_MAXL; o += net.dims[l + 1], ++l)
    if (l < net.depth && tid < net.dims[l + 1]) Bs[o + tid] = bv[l];
  __syncthreads();
  const float(*lp)[4] = FEAT ? lnb : nullptr;
  for (int l = 0, o = 0; l < net.depth; o += net_dim(net, l + 1), ++l) {
    const __bf16 *W = net_weights(net, l);
    const float *bias = Bs + o;
    const int K = net_dim(net, l), N = net_dim(net, l + 1);
    const bool last = l == net.depth - 1;
    // the surrogate's shapes, fully unrolled
    if (K == 512 && N == 512) {
      mlp_layer<4, 512>(W, bias, K, last, Hs, lp, m0, M, out, ldo);
      continue;
    }
    if (K == 64 && N == 512) {
      mlp_layer<4, 64>(W, bias, K, last, Hs, lp, m0, M, out, ldo);
      continue;
    }
    if (K == 512 && N == 128) {
      mlp_layer<1, 512>(W, bias, K, last, Hs, lp, m0, M, out, ldo);
      continue;
    }
    switch (N) {
    case 128: mlp_layer<1, 0>(W, bias, K, last, Hs, lp, m0, M, out, ldo); break;
    case 256: mlp_layer<2, 0>(W, bias, K, last, Hs, lp, m0, M, out, ldo); break;
    default: mlp_layer<4, 0>(W, bias, K, last, Hs, lp, m0, M, out, ldo); break;
    }
  }
}

// ---- special functions (FP64): recurrence to z >= 10, then the asymptotic
// series of ln Gamma (Stirling) and of the digamma function, with the
// Bernoulli-number coefficients B_2n / (2n (2n-1)) and B_2n / (2n).

// 1 / z for normal z away from the ends of the range: the hardware's
// approximation and two Newton-Raphson steps, the last of which rounds
// correctly (equal to the division for all of 7.9e8 values over e^-7 .. e^24).
__device__ __forceinline__ double rcp_pos(double z) {
  double y = __builtin_amdgcn_rcp(z);
  y = __builtin_fma(y, __builtin_fma(-z, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-z, y, 1.0), y);
}

// ln x, within an ulp, for positive normal x: x = 2^k m, m in [sqrt(1/2),
// sqrt(2)), f = m - 1, s = f / (2 + f) and ln m = 2 atanh s = f - s (f - P),
// P = sum 2 s^2n / (2n + 1), whose terms past n = 10 are below 2^-60 of it;
// the arrangement, with ln 2 in two parts, is that of the public-domain
// fdlibm.  A third of the instructions of the library's logarithm, which
// carries a double pair: 0.97 against 0.52 ulp at most (0.2591 against 0.2500
// on average in [0.5, 1.5], 0.2506 against 0.2501 above 10), a difference that
// the sums below do not show (lgamma_digamma_pos).
__device__ __forceinline__ double ln_pos(double x) {
  double m = __builtin_amdgcn_frexp_mant(x);
  int k = __builtin_amdgcn_frexp_exp(x);
  const bool low = m < 0.70710678118654752440;
  m = low ? m + m : m;
  k -= low ? 1 : 0;
  const double f = m - 1.0, s = f * rcp_pos(2.0 + f), w = s * s;
  double p = 2.0 / 21.0;
#pragma unroll
  for (int n = 9; n >= 1; --n) p = __builtin_fma(p, w, 2.0 / (2 * n + 1));
  const double kd = (double)k;
  // k ln2_hi is exact (ln2_hi has 32 bits)
  return __builtin_fma(kd, 0x1.62e42feep-1, f - (s * (f - p * w) - kd * 0x1.a39ef35793c76p-33));
}

// ln Gamma(z) and, with PSI, digamma(z) of one z > 0: they share the
// logarithm and the reciprocal.  With p(z) = z (z+1) ... (z+n-1),
// ln Gamma(z) = ln Gamma(z + n) - ln p(z) and psi(z) = psi(z + n) -
// p'(z) / p(z): one division for the whole shift (at most 10 factors below
// 10: no overflow), and neither it nor ln p where no lane needs a shift.
// Six terms of the series: the first one left out is at most 6.4e-16 of
// ln Gamma and 8.3e-16 of psi (z = 10).  Largest and mean error over z in
// e^-6 .. e^12 with counts 0 .. 1000 added, in units of 2^-53 max(1, |value|):
// ln Gamma 74.1 and 4.53, psi 21.7 and 1.47; with the library's logarithm
// 70.7 and 4.51, 21.7 and 1.45; with it, five terms and the shift of psi as a
// sum of reciprocals, 217 and 28.5, 191 and 18.7.  The library's logarithm
// costs the loss 3.5 us of 62 (4096 items).
template <bool PSI>
__device__ __forceinline__ double lgamma_digamma_pos(double z, double *psi) {
  double prod = 1.0, dprod = 0.0;
  const bool shifted = z < 10.0;
  while (z < 10.0) {
    if (PSI) dprod = __builtin_fma(dprod, z, prod);
    prod *= z;
    z += 1.0;
  }
  double shift = 0.0, dshift = 0.0;
  if (shifted) {
    if (prod > 0.0) {
      shift = ln_pos(prod);
      if (PSI) dshift = dprod * rcp_pos(prod);
    } else { // z <= 0
      shift = log(prod);
      if (PSI) dshift = dprod / prod;
    }
  }
  const double iz = rcp_pos(z), iz2 = iz * iz, lz = ln_pos(z);
  const double series =
      iz * (1.0 / 12.0 -
            iz2 * (1.0 / 360.0 -
                   iz2 * (1.0 / 1260.0 - iz2 * (1.0 / 1680.0 - iz2 * (1.0 / 1188.0 - iz2 * (691.0 / 360360.0))))));
  if (PSI) {
    const double dseries =
        iz2 * (1.0 / 12.0 -
               iz2 * (1.0 / 120.0 -
                      iz2 * (1.0 / 252.0 - iz2 * (1.0 / 240.0 - iz2 * (1.0 / 132.0 - iz2 * (691.0 / 32760.0))))));
    *psi = lz - 0.5 * iz - dseries - dshift;
  }
  return (z - 0.5) * lz - z + 0.91893853320467274178 + series - shift;
}
__device__ __forceinline__ double lgamma_pos(double z) { return lgamma_digamma_pos<false>(z, nullptr); }

// v + (v of the lane CTRL pairs this one with), a DPP rotation of a row of 16
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  int w[2];
  __builtin_memcpy(w, &v, 8);
  w[0] = __builtin_amdgcn_mov_dpp(w[0], CTRL, 0xF, 0xF, false);
  w[1] = __builtin_amdgcn_mov_dpp(w[1], CTRL, 0xF, 0xF, false);
  double o;
  __builtin_memcpy(&o, w, 8);
  return v + o;
}
__device__ __forceinline__ double row_sum(double v) { // over a row of 16 lanes, on every lane
  v = dpp_add<0x128>(v); // row_ror:8
  v = dpp_add<0x124>(v);
  v = dpp_add<0x122>(v);
  return dpp_add<0x121>(v);
}
// Two sums over pairs of lanes in one: the result is a + (a of the other half
// of the wave) in lanes 0..31 and the same of b in lanes 32..63.
__device__ __forceinline__ double fold32(double a, double b) {
  uint32_t x[2], y[2];
  __builtin_memcpy(x, &a, 8);
  __builtin_memcpy(y, &b, 8);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false);
    x[i] = r[0];
    y[i] = r[1];
  }
  __builtin_memcpy(&a, x, 8);
  __builtin_memcpy(&b, y, 8);
  return a + b;
}
// The same within each half: a's sum in rows 0 and 2, b's in rows 1 and 3.
__device__ __forceinline__ double fold16(double a, double b) {
  uint32_t x[2], y[2];
  __builtin_memcpy(x, &a, 8);
  __builtin_memcpy(y, &b, 8);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
    x[i] = r[0];
    y[i] = r[1];
  }
  __builtin_memcpy(&a, x, 8);
  __builtin_memcpy(&b, y, 8);
  return a + b;
}

// What a mixture component's terms need besides the sample, in FP64.
struct NllComp {
  double lpi, pi;    // log softmax of the logits, and the softmax
  double r, mu;      // negative binomial: dispersion and mean; binomial: mu = p
  double lgr, psir;  // ln Gamma(r), digamma(r)
  double c0, cx;     // ll = ... + c0 + x cx (negative binomial)
  double spn, spp;   // softplus(-theta), softplus(theta) (binomial)
  double irm;        // 1 / (r + mu)
  uint32_t clamped;  // bit 0: log mean (or theta), bit 1: log dispersion
};

// Negative log-likelihood of the SSA samples under the predicted mixtures,
// and its gradient w.r.t. the head outputs.  A workgroup of four waves per
// item, one species per wave and one sample per lane (64 samples).  Head
// layout per species s (K components):
// [s*3K + c] mixture logit, [s*3K + K + c] log mean, [s*3K + 2K + c] log
// dispersion.  With bounds, components c < K/2 are negative binomials of the
// count x with log means relative to ln bound, and components c >= K/2 are
// binomial(bound, p) with logit p in the log-mean slot (a bounded count can
// vary less than its mean, which no negative binomial does; their dispersion
// slot is unused).  samples: the SSA output
// [nb+1][S][P * J], item (p, i) reads samples[(i*S + s) * P*J + p*J + j].
// grad = d(mean NLL over items and samples)/d head (FP32, [B][ldh]);
// loss_sum += total NLL (FP64).
//
// Bound by FP64 instructions and the latency of their chains (VALU issue on
// 0.65 of the CU cycles, 54 % of it FP64 arithmetic).  What does not depend on the sample is computed once
// per (species, component), one lane each, and read back from LDS; per sample
// and negative binomial the ln Gamma and digamma share their logarithm,
// reciprocal and shift; the responsibilities come from the exponentials of
// the log-sum-exp; and the 64-lane sums of the 20 (unbounded: 24) gradient
// terms halve the number of values per step instead of reducing each alone.
// Four waves per SIMD (128 VGPRs, 28 bytes of spill) measured 62 us at 4096
// items x 4 species x 64 samples, three 64 us, five 62 us (92 us unbounded),
// the components unrolled at two 75 us; one wave per item with every term on
// every lane 235 us, and at 64 items 9 us against 69 us.
template <int K, bool BOUND>
__global__ void __launch_bounds__(256, 4) nb_mixture_nll_kernel(
    int B, int S, int J, const float *__restrict__ head, int ldh,
    const uint32_t *__restrict__ item_point, const uint32_t *__restrict__ item_sample,
    const int64_t *__restrict__ samples, uint64_t n_traj_total, float *__restrict__ grad,
    double *__restrict__ loss_sum, double scale, const float *__restrict__ bound) {
  constexpr int NBC = BOUND ? K / 2 : K; // negative-binomial components
  __shared__ NllComp comp[4][K];
  __shared__ double nbt[NBC][2][256]; // per sample: log weighted likelihood, its dispersion derivative
  __shared__ double lcn[4]; // ln Gamma(bound + 1)
  __shared__ double part[4];
  const int b = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, j = tid & 63;
  const uint32_t p = item_point[b], i = item_sample[b];
  const bool active = j < J;
  double lane_loss = 0.0;
  for (int s0 = 0; s0 < S; s0 += 4) {
    const int s = s0 + wave;
    const double xs = active && s < S
                          ? (double)samples[((size_t)i * S + s) * n_traj_total + (size_t)p * J + j]
                          : 0.0;
    const double bnd = BOUND && s < S ? (double)bound[(size_t)b * S + s] : 0.0;
    // the sample-independent terms: wave 0 the components' special functions,
    // wave 1 the softmax, wave 2 the bounds'
    if (tid < 4 * K && s0 + tid / K < S) {
      const int cs = tid / K, c = tid % K;
      const float *hc = head + (size_t)b * ldh + (size_t)(s0 + cs) * 3 * K;
      NllComp &o = comp[cs][c];
      if (BOUND && c >= K / 2) {
        // binomial(bound, p), p = sigmoid(theta): ln p = -softplus(-theta)
        const double th = fmin(fmax((double)hc[K + c], -30.0), 30.0);
        o.spn = th < 0.0 ? log1p(exp(th)) - th : log1p(exp(-th));
        o.spp = o.spn + th;
        o.mu = exp(-o.spn);
        o.clamped = (double)hc[K + c] != th ? 1u : 0u;
      } else {
        const double off = BOUND ? log((double)bound[(size_t)b * S + s0 + cs]) : 0.0;
        const double lm = (double)hc[K + c] + off, ld = (double)hc[2 * K + c];
        const double lmu = fmin(fmax(lm, -8.0), 9.0), lr = fmin(fmax(ld, -6.0), 12.0);
        const double mu = exp(lmu), r = exp(lr), lrm = log(r + mu);
        double psi;
        o.lgr = lgamma_digamma_pos<true>(r, &psi);
        o.psir = psi;
        o.mu = mu;
        o.r = r;
        o.c0 = r * (lr - lrm);
        o.cx = lmu - lrm;
        o.spn = lr - lrm;
        o.irm = 1.0 / (r + mu);
        o.clamped = (lm != lmu ? 1u : 0u) | (ld != lr ? 2u : 0u);
      }
    } else if (tid >= 64 && tid < 64 + 4 * K && s0 + (tid - 64) / K < S) {
      const int cs = (tid - 64) / K, c = (tid - 64) % K;
      const float *hc = head + (size_t)b * ldh + (size_t)(s0 + cs) * 3 * K;
      double lmax = -1e300, zs = 0.0;
#pragma unroll
      for (int q = 0; q < K; ++q) lmax = fmax(lmax, (double)hc[q]);
#pragma unroll
      for (int q = 0; q < K; ++q) zs += exp((double)hc[q] - lmax);
      comp[cs][c].lpi = (double)hc[c] - (lmax + log(zs));
      comp[cs][c].pi = exp(comp[cs][c].lpi);
    } else if (BOUND && tid >= 128 && tid < 132 && s0 + tid - 128 < S) {
      lcn[tid - 128] = lgamma_pos((double)bound[(size_t)b * S + s0 + tid - 128] + 1.0);
    }
    __syncthreads();
    if (s < S) { // the same for the whole wave
      const NllComp *cp = comp[wave];
      const double lgx1 = lgamma_pos(xs + 1.0);
      // ln C(bound, x) for the binomial components of a bounded species
      const double lcb = BOUND ? lcn[wave] - lgx1 - lgamma_pos(fmax(bnd - xs, 0.0) + 1.0) : 0.0;
      // one copy of the special functions' code, its results through LDS: the
      // registers of an unrolled loop would leave two waves per SIMD
#pragma unroll 1
      for (int c = 0; c < NBC; ++c) {
        double psi;
        const double lg = lgamma_digamma_pos<true>(xs + cp[c].r, &psi);
        nbt[c][0][tid] = cp[c].lpi + (lg - cp[c].lgr - lgx1 + cp[c].c0 + xs * cp[c].cx);
        nbt[c][1][tid] = psi - cp[c].psir + cp[c].spn;
      }
      double lterm[K];
      double best = -1e300;
#pragma unroll
      for (int c = 0; c < K; ++c) {
        lterm[c] = c < NBC ? nbt[c < NBC ? c : 0][0][tid]
                           : cp[c].lpi + (lcb - xs * cp[c].spn - (bnd - xs) * cp[c].spp);
        best = fmax(best, lterm[c]);
      }
      double se = 0.0;
#pragma unroll
      for (int c = 0; c < K; ++c) {
        lterm[c] = exp(lterm[c] - best);
        se += lterm[c];
      }
      if (active) lane_loss -= best + log(se);
      const double ise = active ? 1.0 / se : 0.0;
      // sums over the samples: [0, K) responsibilities, [K, 2K) log means (less
      // a factor that is the component's), then the log dispersions
      constexpr int NV = 2 * K + NBC;
      static_assert(NV % 4 == 0, "folded in two halvings");
      double v[NV];
#pragma unroll
      for (int c = 0; c < K; ++c) {
        const double gam = active ? lterm[c] * ise : 0.0;
        v[c] = gam;
        if (c >= NBC) {
          v[K + c] = -gam * (xs - bnd * cp[c].mu); // d/dtheta of -ln binomial
        } else {
          const double d = (cp[c].mu - xs) * cp[c].irm;
          v[K + c] = gam * d;
          v[2 * K + (c < NBC ? c : 0)] = -gam * (nbt[c < NBC ? c : 0][1][tid] + d);
        }
      }
      // fold32 keeps the values below NV/2 in lanes 0..31 and the others in
      // 32..63, fold16 halves again, and each row adds up what it is left with
#pragma unroll
      for (int n = 0; n < NV / 2; ++n) v[n] = fold32(v[n], v[n + NV / 2]);
#pragma unroll
      for (int n = 0; n < NV / 4; ++n) v[n] = row_sum(fold16(v[n], v[n + NV / 4]));
      // row w holds the sums w NV/4 .. +NV/4 on all its lanes
      float *g = grad + (size_t)b * ldh + (size_t)s * 3 * K;
      double mine = 0.0;
#pragma unroll
      for (int n = 0; n < NV / 4; ++n)
        if ((j & 15) == n) mine = v[n];
      if ((j & 15) < NV / 4) {
        const int n = (j >> 4) * (NV / 4) + (j & 15);
        const int c = n % K;
        if (n < K) {
          g[n] = (float)(((double)J * cp[c].pi - mine) * scale);
        } else if (n < 2 * K) {
          const double f = c >= NBC ? mine : mine * cp[c].r;
          g[n] = (float)((cp[c].clamped & 1u) ? 0.0 : f * scale);
        } else {
          g[n] = (float)((cp[c].clamped & 2u) ? 0.0 : mine * cp[c].r * scale);
        }
      }
      if (BOUND && j < K - NBC) g[2 * K + NBC + j] = 0.f; // the binomials' unused slot
    }
    if (s0 + 4 < S) __syncthreads(); // the components are read before the next species'
  }
  lane_loss = row_sum(lane_loss);
  lane_loss = fold16(lane_loss, lane_loss);
  lane_loss = fold32(lane_loss, lane_loss);
  if (j == 0) part[wave] = lane_loss;
  __syncthreads();
  if (tid == 0) atomicAdd(loss_sum, part[0] + part[1] + part[2] + part[3]);
}

} // namespace sg

// ---------------------------------------------------------------------------
// C ABI

namespace {
hipError_t g_err = hipSuccess;
int ret(hipError_t e) {
  g_err = e;
  return e == hipSuccess ? 0 : 4;
}
unsigned nblk(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

// The layer table of the fused forward pass; 3 if the shapes are outside
// what mlp_infer_kernel handles.
int mlp_net(int depth, const int *dims, const void *const *Wp, const float *const *bias,
            sg::MlpNet &net) {
  if (depth < 1 || depth > sg::MLP_MAXL || !dims || !Wp || !bias) return 3;
  if (dims[0] <= 0 || dims[0] % 64 || dims[0] > sg::MLP_MAXW) return 3;
  net.depth = depth;
  net.dims[0] = dims[0];
  for (int l = 0; l < depth; ++l) {
    const int n = dims[l + 1];
    if (n != 128 && n != 256 && n != 512) return 3;
    if (!Wp[l] || !bias[l] || (uintptr_t)Wp[l] % 16 || (uintptr_t)bias[l] % 16) return 3;
    net.dims[l + 1] = n;
    net.Wp[l] = (const __bf16 *)Wp[l];
    net.bias[l] = bias[l];
  }
  return 0;
}

// 128 x 128 tiles when there are enough of them to fill the chip
bool big_tiles(int M, int N) { return M % 128 == 0 && N % 128 == 0 && (M / 128) * (N / 128) >= 512; }

// k-contiguous operands: the pipelined kernel
template <int EPI>
void launch_nt(bool big, dim3 grid, hipStream_t s, int M, int N, int K, const __bf16 *a, int lda,
               const __bf16 *b, int ldb, float *C, int ldc, const sg::Epilogue &epi) {
  if (big)
    hipLaunchKernelGGL((sg::gemm_nt_kernel<128, 128, EPI>), grid, dim3(256), 0, s, M, N, K, a, lda, b, ldb, C,
                       ldc, epi);
  else
    hipLaunchKernelGGL((sg::gemm_nt_kernel<64, 64, EPI>), grid, dim3(256), 0, s, M, N, K, a, lda, b, ldb, C,
                       ldc, epi);
}

template <bool TA, bool TB>
void launch_gemm(bool big, dim3 grid, hipStream_t s, int M, int N, int K, const __bf16 *a, int lda,
                 const __bf16 *b, int ldb, float *C, int ldc, const sg::Epilogue *epi = nullptr) {
  if constexpr (!TA && TB) {
    if (epi) launch_nt<sg::EPI_BIAS>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc, *epi);
    else launch_nt<sg::EPI_PLAIN>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc, sg::Epilogue{});
    return;
  } else {
    const sg::Epilogue e = epi ? *epi : sg::Epilogue{};
    if (epi && big)
      hipLaunchKernelGGL((sg::gemm_kernel<TA, TB, 128, 128, true>), grid, dim3(256), 0, s, M, N, K, a, lda, b,
                         ldb, C, ldc, e);
    else if (epi)
      hipLaunchKernelGGL((sg::gemm_kernel<TA, TB, 64, 64, true>), grid, dim3(256), 0, s, M, N, K, a, lda, b, ldb,
                         C, ldc, e);
    else if (big)
      hipLaunchKernelGGL((sg::gemm_kernel<TA, TB, 128, 128, false>), grid, dim3(256), 0, s, M, N, K, a, lda, b,
                         ldb, C, ldc, e);
    else
      hipLaunchKernelGGL((sg::gemm_kernel<TA, TB, 64, 64, false>), grid, dim3(256), 0, s, M, N, K, a, lda, b,
                         ldb, C, ldc, e);
  }
}

sg::Epilogue bias_epilogue(const float *bias, int relu, void *H, int ldh, float *F, int ldf) {
  sg::Epilogue e{};
  e.bias = bias;
  e.relu = relu;
  e.H = (__bf16 *)H;
  e.ldh = ldh;
  e.F = F;
  e.ldf = ldf;
  e.wide = (!H || ((uintptr_t)H % 8 == 0 && ldh % 4 == 0)) && (!F || ((uintptr_t)F % 16 == 0 && ldf % 4 == 0));
  return e;
}

// The shapes of a layer stack's training passes, and how the backward pass
// lays out its workspace: dZ of every layer (BF16), the column sums
// [batch / 64][sum of widths], and with splits > 1 their weight gradients.
struct TrainPlan {
  size_t weights = 0, dz = 0, colsum = 0, part = 0; // floats; BF16 elements; floats; floats
  int nbias = 0, splits = 1, units = 0;
  size_t bytes() const { return 2 * dz + 4 * colsum + 4 * part; }
};
bool train_plan(int B, int depth, const int *dims, TrainPlan &p) {
  if (B <= 0 || B % 64 || depth < 1 || !dims) return false;
  size_t tiles = 0;
  for (int l = 0; l <= depth; ++l) {
    if (dims[l] <= 0 || dims[l] % 64) return false;
    if (l == 0) continue;
    p.weights += (size_t)dims[l - 1] * dims[l];
    tiles += (size_t)(dims[l - 1] / 64) * (dims[l] / 64);
    p.nbias += dims[l];
  }
  p.units = B / 64;
  // a power of two: about 1024 workgroups (four to a CU) of at least 128 rows each
  while (p.splits < 32 && 2 * p.splits <= p.units / 2 && 2 * p.splits * tiles <= 1024) p.splits *= 2;
  p.dz = (size_t)B * p.nbias;
  p.colsum = (size_t)p.units * p.nbias;
  p.part = p.splits > 1 ? p.weights * (size_t)p.splits : 0;
  return true;
}

} // namespace

extern "C" {

const char *rebop_sg_last_error(void) { return hipGetErrorString(g_err); }

int rebop_sg_gemm_bf16(int ta, int tb, int M, int N, int K, const void *A, int lda, const void *B,
                       int ldb, float *C, int ldc, void *stream) {
  if (M % 64 || N % 64 || K % 32 || M <= 0 || N <= 0 || K <= 0) return 3;
  const bool big = big_tiles(M, N);
  const int tile = big ? 128 : 64;
  // split K when the output has too few tiles to fill the chip
  int splits = 1;
  while (!big && (M / 64) * (N / 64) * splits < 512 && K % (64 * splits) == 0 &&
         K / (32 * splits) >= 8)
    splits *= 2;
  const dim3 grid(N / tile, M / tile, splits);
  const __bf16 *a = (const __bf16 *)A, *b = (const __bf16 *)B;
  hipStream_t s = (hipStream_t)stream;
  if (splits > 1)
    hipLaunchKernelGGL(sg::zero_kernel, dim3(nblk((size_t)M * N, 256)), dim3(256), 0, s, M, N, C, ldc);
  if (!ta && !tb) launch_gemm<false, false>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc);
  else if (!ta && tb) launch_gemm<false, true>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc);
  else if (ta && !tb) launch_gemm<true, false>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc);
  else launch_gemm<true, true>(big, grid, s, M, N, K, a, lda, b, ldb, C, ldc);
  return ret(hipGetLastError());
}

int rebop_sg_gemm_bias_act_bf16(int tb, int M, int N, int K, const void *A, int lda, const void *B,
                                int ldb, const float *bias, int relu, void *H, int ldh, float *F,
                                int ldf, void *stream) {
  if (M % 64 || N % 64 || K % 32 || M <= 0 || N <= 0 || K <= 0) return 3;
  if (!bias || (!H && !F)) return 3;
  const bool big = big_tiles(M, N);
  const int tile = big ? 128 : 64;
  const dim3 grid(N / tile, M / tile, 1); // no split K: the epilogue needs the whole sum
  const sg::Epilogue epi = bias_epilogue(bias, relu, H, ldh, F, ldf);
  if (tb)
    launch_gemm<false, true>(big, grid, (hipStream_t)stream, M, N, K, (const __bf16 *)A, lda,
                             (const __bf16 *)B, ldb, nullptr, 0, &epi);
  else
    launch_gemm<false, false>(big, grid, (hipStream_t)stream, M, N, K, (const __bf16 *)A, lda,
                              (const __bf16 *)B, ldb, nullptr, 0, &epi);
  return ret(hipGetLastError());
}

int rebop_sg_mlp_train_forward(int B, const void *X, int ldx, int depth, const int *dims,
                               const void *const *Wt, const float *const *bias, void *const *H,
                               float *head, void *stream) {
  TrainPlan p;
  if (!train_plan(B, depth, dims, p) || !X || !Wt || !bias || !head || (depth > 1 && !H) || ldx < dims[0] || ldx % 8)
    return 3;
  for (int l = 0; l < depth; ++l)
    if (!Wt[l] || !bias[l] || (l < depth - 1 && !H[l])) return 3;
  const void *in = X;
  for (int l = 0; l < depth; ++l) {
    const bool last = l == depth - 1;
    const int rc = rebop_sg_gemm_bias_act_bf16(1, B, dims[l + 1], dims[l], in, l == 0 ? ldx : dims[l], Wt[l],
                                               dims[l], bias[l], !last, last ? nullptr : H[l], dims[l + 1],
                                               last ? head : nullptr, dims[l + 1], stream);
    if (rc) return rc;
    if (!last) in = H[l];
  }
  return 0;
}

size_t rebop_sg_mlp_backward_workspace(int B, int depth, const int *dims) {
  TrainPlan p;
  return train_plan(B, depth, dims, p) ? p.bytes() : 0;
}

int rebop_sg_mlp_backward(int B, int depth, const int *dims, const float *dhead, int ldd, const void *X, int ldx,
                          const void *const *H, const void *const *Wb, void *workspace, float *grads,
                          void *stream) {
  TrainPlan p;
  if (!train_plan(B, depth, dims, p) || !dhead || !X || !Wb || !workspace || !grads || (depth > 1 && !H) ||
      ldd < dims[depth] || ldx < dims[0] || ldx % 8 || (uintptr_t)workspace % 16 ||
      (uintptr_t)grads % 16)
    return 3;
  for (int l = 1; l < depth; ++l)
    if (!H[l - 1] || !Wb[l] || (uintptr_t)H[l - 1] % 16 || (uintptr_t)Wb[l] % 16) return 3;
  hipStream_t s = (hipStream_t)stream;
  float *part = (float *)workspace, *colsum = part + p.part;
  __bf16 *dz = (__bf16 *)(colsum + p.colsum); // p.part and p.colsum are multiples of 64
  // dZ from the last layer to the first, each with its column sums; a layer's
  // dZ lies behind those of the layers before it
  int col = p.nbias;
  const __bf16 *next = nullptr; // dZ of layer l + 1
  for (int l = depth - 1; l >= 0; --l) {
    const int n = dims[l + 1];
    col -= n;
    __bf16 *out = dz + (size_t)B * col;
    if (l == depth - 1) {
      hipLaunchKernelGGL(sg::head_grad_kernel, dim3(n / 64, B / 64), dim3(256), 0, s, n, dhead, ldd, out,
                         colsum + col, p.nbias);
    } else {
      sg::Epilogue e{};
      e.H = out;
      e.ldh = n;
      e.mask = (const __bf16 *)H[l];
      e.colsum = colsum + col;
      e.ldc = p.nbias;
      const bool big = big_tiles(B, n);
      const int tile = big ? 128 : 64, k = dims[l + 2];
      launch_nt<sg::EPI_MASK>(big, dim3(n / tile, B / tile), s, B, n, k, next, k, (const __bf16 *)Wb[l + 1], k,
                              nullptr, 0, e);
    }
    next = out;
  }
  // every layer's weight gradient
  float *wout = p.splits > 1 ? part : grads;
  size_t at = 0;
  col = 0;
  for (int l0 = 0; l0 < depth; l0 += sg::WG_MAXL) {
    sg::WgradNet net{};
    int tiles = 0;
    for (int l = l0; l < depth && l < l0 + sg::WG_MAXL; ++l) {
      const int i = l - l0;
      net.H[i] = (const __bf16 *)(l == 0 ? X : H[l - 1]);
      net.ldh[i] = l == 0 ? ldx : dims[l];
      net.dZ[i] = dz + (size_t)B * col;
      net.n[i] = dims[l + 1];
      net.tile0[i] = tiles;
      net.out[i] = at;
      net.layers = i + 1;
      tiles += (dims[l] / 64) * (dims[l + 1] / 64);
      at += (size_t)dims[l] * dims[l + 1];
      col += dims[l + 1];
    }
    hipLaunchKernelGGL(sg::wgrad_kernel, dim3(tiles * p.splits), dim3(256), 0, s, p.units, p.splits, net, wout,
                       p.weights);
  }
  const unsigned blocks = (p.splits > 1 ? (unsigned)(p.weights / 1024) : 0u) + nblk((size_t)p.nbias, 64);
  hipLaunchKernelGGL(sg::grad_reduce_kernel, dim3(blocks), dim3(256), 0, s, p.splits, p.weights, p.weights, part,
                     p.nbias, p.units, colsum, grads);
  return ret(hipGetLastError());
}

int rebop_sg_bias_act(int M, int N, const float *C, int ldc, const float *bias, int relu, void *H,
                      int ldh, float *F, int ldf, void *stream) {
  hipLaunchKernelGGL(sg::bias_act_kernel, dim3(nblk((size_t)M * N, 256)), dim3(256), 0,
                     (hipStream_t)stream, M, N, C, ldc, bias, relu, (__bf16 *)H, ldh, F, ldf);
  return ret(hipGetLastError());
}

int rebop_sg_relu_grad(int M, int N, float *dH, int ldd, const void *H, int ldh, void *dZ, int ldz,
                       void *stream) {
  hipLaunchKernelGGL(sg::relu_grad_kernel, dim3(nblk((size_t)M * N, 256)), dim3(256), 0,
                     (hipStream_t)stream, M, N, dH, ldd, (const __bf16 *)H, ldh, (__bf16 *)dZ, ldz);
  return ret(hipGetLastError());
}

int rebop_sg_transpose_bf16(int rows, int cols, const float *x, void *y, void *stream) {
  if (rows <= 0 || cols <= 0) return 3;
  hipLaunchKernelGGL(sg::transpose_bf16_kernel, dim3(nblk((size_t)rows * cols, 256)), dim3(256), 0,
                     (hipStream_t)stream, rows, cols, x, (__bf16 *)y);
  return ret(hipGetLastError());
}

int rebop_sg_cast_bf16(size_t n, const float *x, void *y, void *stream) {
  hipLaunchKernelGGL(sg::cast_bf16_kernel, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream,
                     n, x, (__bf16 *)y);
  return ret(hipGetLastError());
}

int rebop_sg_colsum(int M, int N, const float *X, int ldx, float *out, void *stream) {
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(sg::fill_kernel, dim3(nblk((size_t)N, 256)), dim3(256), 0, st, N, out);
  hipLaunchKernelGGL(sg::colsum_kernel, dim3(nblk((size_t)N, 64), nblk((size_t)M, 256)), dim3(256),
                     0, st, M, N, X, ldx, out);
  return ret(hipGetLastError());
}

int rebop_sg_adam(size_t n, float *w, const float *g, float *m, float *v, void *wb, float lr,
                  float b1, float b2, float eps, float bc1, float bc2, void *stream) {
  hipLaunchKernelGGL(sg::adam_kernel, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, n, w,
                     g, m, v, (__bf16 *)wb, lr, b1, b2, eps, bc1, bc2);
  return ret(hipGetLastError());
}

int rebop_sg_features(int B, const uint32_t *item_point, const uint32_t *item_sample,
                      const double *rates, const int64_t *x0, double tmax, int nb_steps, void *X,
                      int ldx, float *bound, void *stream) {
  if (ldx < REBOP_SG_FEATURES) return 3;
  const bool wide = (uintptr_t)X % 8 == 0 && ldx % 4 == 0;
  hipLaunchKernelGGL(sg::features_kernel, dim3(nblk((size_t)B, 64)), dim3(256), 0, (hipStream_t)stream, B,
                     item_point, item_sample, rates, x0, tmax, nb_steps, (__bf16 *)X, ldx, bound, wide);
  return ret(hipGetLastError());
}

int rebop_sg_head_offsets(int B, int S, int K, float *head, int ldh, const float *bound,
                          void *stream) {
  if (ldh < S * 3 * K) return 3;
  hipLaunchKernelGGL(sg::head_offsets_kernel, dim3(nblk((size_t)B * S * K, 256)), dim3(256), 0,
                     (hipStream_t)stream, B, S, K, head, ldh, bound);
  return ret(hipGetLastError());
}

int rebop_sg_pack_kslices_bf16(int K, int N, const float *W, void *Wp, void *stream) {
  if (K <= 0 || N <= 0 || K % 32 || !W || !Wp) return 3;
  hipLaunchKernelGGL(sg::pack_kslices_kernel, dim3(nblk((size_t)K * N, 256)), dim3(256), 0,
                     (hipStream_t)stream, K, N, W, (__bf16 *)Wp);
  return ret(hipGetLastError());
}

int rebop_sg_mlp_forward_bf16(int M, const void *X, int ldx, int depth, const int *dims,
                              const void *const *Wp, const float *const *bias, float *out, int ldo,
                              void *stream) {
  sg::MlpNet net{};
  if (mlp_net(depth, dims, Wp, bias, net) || M <= 0 || !X || !out || (uintptr_t)X % 16 ||
      (uintptr_t)out % 16 || ldx < dims[0] || ldx % 8 || ldo < dims[depth] || ldo % 4)
    return 3;
  const sg::MlpItems none{nullptr, nullptr, nullptr, nullptr, 0.0, 1};
  hipLaunchKernelGGL(sg::mlp_infer_kernel<false>, dim3(nblk((size_t)M, sg::MLP_BM)), dim3(512), 0,
                     (hipStream_t)stream, M, (const __bf16 *)X, ldx, none, net, out, ldo);
  return ret(hipGetLastError());
}

int rebop_sg_infer(int B, const uint32_t *item_point, const uint32_t *item_sample,
                   const double *rates, const int64_t *x0, double tmax, int nb_steps, int depth,
                   const int *dims, const void *const *Wp, const float *const *bias, float *head,
                   int ldh, void *stream) {
  sg::MlpNet net{};
  if (mlp_net(depth, dims, Wp, bias, net) || B <= 0 || !item_point || !item_sample || !rates ||
      !x0 || !head || (uintptr_t)head % 16 || dims[0] < REBOP_SG_FEATURES ||
      dims[depth] < 4 * 3 * REBOP_SG_COMPONENTS || ldh < dims[depth] || ldh % 4 || nb_steps <= 0)
    return 3;
  const sg::MlpItems items{item_point, item_sample, rates, x0, tmax, nb_steps};
  hipLaunchKernelGGL(sg::mlp_infer_kernel<true>, dim3(nblk((size_t)B, sg::MLP_BM)), dim3(512), 0,
                     (hipStream_t)stream, B, nullptr, 0, items, net, head, ldh);
  return ret(hipGetLastError());
}

int rebop_sg_nb_mixture_nll(int B, int S, int K, int J, const float *head, int ldh,
                            const uint32_t *item_point, const uint32_t *item_sample,
                            const int64_t *samples, uint64_t n_traj_total, float *grad,
                            double *loss_sum, double scale, const float *bound, void *stream) {
  if (K != REBOP_SG_COMPONENTS || J > 64 || J <= 0) return 3;
  if (bound)
    hipLaunchKernelGGL((sg::nb_mixture_nll_kernel<REBOP_SG_COMPONENTS, true>), dim3(B), dim3(256), 0,
                       (hipStream_t)stream, B, S, J, head, ldh, item_point, item_sample, samples,
                       n_traj_total, grad, loss_sum, scale, bound);
  else
    hipLaunchKernelGGL((sg::nb_mixture_nll_kernel<REBOP_SG_COMPONENTS, false>), dim3(B), dim3(256), 0,
                       (hipStream_t)stream, B, S, J, head, ldh, item_point, item_sample, samples,
                       n_traj_total, grad, loss_sum, scale, bound);
  return ret(hipGetLastError());
}

} // extern "C"
