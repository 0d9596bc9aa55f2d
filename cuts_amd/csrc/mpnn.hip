// Message-passing network that predicts partial-match table sizes.
// No reference counterpart: cuTS orders queries only with the greedy score
// of src/graph.cpp:62-93 and never looks at how large its trie levels get
// (the sizes live in `lengths`, src/host_funcs.cu:95,153, and are dropped).
//
// Model (one sample = a query graph with <= 16 vertices, a prefix set S of
// its vertices, and per-vertex input features that include data-graph
// statistics):
//   h0 = x                                                   (24 features)
//   h_{l+1}[v] = ReLU(b_l + Ws_l^T h_l[v] + Wn_l^T sum_{u in N(v)} h_l[u]),  l = 0,1,2 (hidden 64)
//   c = [ sum_{v in S} h3[v] ; mean_v h3[v] ]                 (128)
//   y = bo + wo . ReLU(br + Wr^T c)
// and is trained on y ~ log(1 + |T(S)|) / 10 with a mean squared error.
//
// gfx950 mapping: one wave64 per sample; a layer is two 16 x IN x 64 products
// (16 = the padded query vertices), on the FP32 matrix cores
// (v_mfma_f32_16x16x4_f32: FP32 operands and accumulation).  Weights are
// BF16 (kept twice: input-major for the backward products and transposed for
// the forward ones, so that a lane's four consecutive inputs of a product
// are one 8-byte load), widened in registers, with an FP32 master copy
// updated by Adam.  Weight gradients stay in accumulators: a block's four
// waves run four samples forward and backward, then each wave adds all four
// samples' outer products for its own 16 columns of every gradient matrix;
// one row of partial sums per block is written at the end and reduced over
// blocks (no atomics).  Per sample the network is 0.3 MFLOP in a chain of
// dependent products, so a launch is bound by that chain's latency at one to
// two waves per SIMD, and a call by the copy of its samples to the GPU.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "mpnn.hpp"

namespace cuts {
namespace {

constexpr int H = kMpnnHidden, FIN = kMpnnFeats, MAXN = kMpnnNodes;

// parameter offsets (floats) in the flat vector; matrices are input-major
// W[i][j] = W[i*out + j]
constexpr int O_WS0 = 0;
constexpr int O_WN0 = O_WS0 + FIN * H;
constexpr int O_B0 = O_WN0 + FIN * H;
constexpr int O_WS1 = O_B0 + H;
constexpr int O_WN1 = O_WS1 + H * H;
constexpr int O_B1 = O_WN1 + H * H;
constexpr int O_WS2 = O_B1 + H;
constexpr int O_WN2 = O_WS2 + H * H;
constexpr int O_B2 = O_WN2 + H * H;
constexpr int O_WR = O_B2 + H;
constexpr int O_BR = O_WR + 2 * H * H;
constexpr int O_WO = O_BR + H;
constexpr int O_BO = O_WO + H;
constexpr int NPARAM = O_BO + 1;
static_assert(NPARAM == kMpnnParams, "parameter layout");

__device__ __forceinline__ float bf(const uint16_t* w, int i) { return __uint_as_float((uint32_t)w[i] << 16); }

// round-to-nearest-even float -> bf16 (finite inputs)
__device__ __forceinline__ uint16_t to_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

typedef float f4 __attribute__((ext_vector_type(4)));

// Words of an LDS activation row: 64 hidden units (or 24 features) and a pad
// of 4, so that the 16 rows of a product's operand start in different banks.
constexpr int LR = H + 4, LF = FIN + 4;

// The wave's own LDS writes before its later reads of other lanes' words (a
// wave's LDS accesses execute in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float lo16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi16(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ uint32_t lane_of(uint32_t x, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, lane);
}

// acc[nt] += X (16 x IN, LDS rows of `ldx` words) times B (IN x 16 columns
// nt*16 ..), B given as its transpose: row c = column c of B, IN BF16 inputs
// in rows of `ldb`.  Lane (i = lane % 16, g = lane / 16) holds X[i][k] and
// B[k][i] for the inputs k = c*16 + g*4 + t (24 = 16 + 8: then k = 16 + g*2 +
// t): one 16-byte and one 8-byte load for four products.
template <int IN, int NT>
__device__ __forceinline__ void mfma_rows(f4 (&acc)[NT], const float* X, int ldx, const uint16_t* B, int ldb) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int c = 0; c < IN / 16; ++c) {
    const f4 x = *(const f4*)(X + i * ldx + c * 16 + g * 4);
    uint2 b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[nt] = *(const uint2*)(B + (nt * 16 + i) * ldb + c * 16 + g * 4);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0], lo16(b[nt].x), acc[nt], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[1], hi16(b[nt].x), acc[nt], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[2], lo16(b[nt].y), acc[nt], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[3], hi16(b[nt].y), acc[nt], 0, 0, 0);
  }
  if constexpr (IN % 16 == 8) {
    const int k = IN - 8 + g * 2;
    const float2 x = *(const float2*)(X + i * ldx + k);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint32_t b = *(const uint32_t*)(B + (nt * 16 + i) * ldb + k);
      acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, lo16(b), acc[nt], 0, 0, 0);
      acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, hi16(b), acc[nt], 0, 0, 0);
    }
  }
}

// A product's accumulators to 16 LDS rows: lane (j, g) holds rows 4g .. 4g+3
// of column nt*16 + j.
__device__ __forceinline__ void store_acc(const f4 (&acc)[4], float* Y, int ldy) {
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int r = 0; r < 4; ++r) Y[(4 * g + r) * ldy + nt * 16 + j] = acc[nt][r];
}

// Y[v] = sum of X[u] over the neighbours u of v (adjv: lane v holds vertex
// v's neighbour mask), rows k.. zero; lane j owns column j < cols.
__device__ __forceinline__ void neighbour_sums(const float* X, float* Y, int ld, int cols, int k, uint32_t adjv) {
  const int j = threadIdx.x & 63;
  for (int v = 0; v < MAXN; ++v) {
    float s = 0.f;
    if (v < k)
      for (uint32_t m = lane_of(adjv, v); m; m &= m - 1) {
        const int u = __builtin_ctz(m);
        if (j < cols) s += X[u * ld + j];
      }
    if (j < cols) Y[v * ld + j] = s;
  }
}

// One layer's products and bias, ReLU, rows k.. zero, into Y (LDS rows of LR).
template <int IN>
__device__ __forceinline__ void layer(const float* X, const float* A, int ldx, const uint16_t* Ws, const uint16_t* Wn,
                                      int ldw, const uint16_t* bias, int k, float* Y) {
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
  f4 acc[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const float b = bf(bias, nt * 16 + j);
    acc[nt] = f4{b, b, b, b};
  }
  mfma_rows<IN, 4>(acc, X, ldx, Ws, ldw);
  mfma_rows<IN, 4>(acc, A, ldx, Wn, ldw);
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[nt][r] = 4 * g + r < k ? fmaxf(acc[nt][r], 0.f) : 0.f;
  wave_sync();  // Y may be X
  store_acc(acc, Y, LR);
  wave_sync();
}

// Features of one sample to LDS rows of ld words, rows k.. zero.
__device__ __forceinline__ void load_features(const float* __restrict__ x, int k, float* X, int ld) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int e = 0; e < MAXN * FIN; e += 64) {
    const int q = e + lane;
    X[(q / FIN) * ld + q % FIN] = q < k * FIN ? x[q] : 0.f;
  }
}

// Column sums of the last layer's rows: over the set, and the mean over all k.
__device__ __forceinline__ void pool(const float* X, int k, uint32_t smask, float& ss, float& sa) {
  const int j = threadIdx.x & 63;
  ss = sa = 0.f;
  for (int v = 0; v < k; ++v) {
    const float h = X[v * LR + j];
    sa += h;
    if (smask >> v & 1) ss += h;
  }
  sa = sa / (float)k;
}

__device__ __forceinline__ float wave_total(float y) {
  for (int o = 32; o > 0; o >>= 1) y += __shfl_xor(y, o);
  return y;
}

// LDS words (BF16) of one transposed matrix with IN inputs, rows padded by 4
constexpr int lds_mat(int in) { return H * (in + 4); }

}  // namespace

// One wave per sample, FW waves per block around one LDS copy of the
// transposed weights (58 KB; the padded rows keep the 16 columns of a
// product in different banks).
constexpr int FW = 8;
__global__ __launch_bounds__(FW * 64) void k_mpnn_forward(const uint16_t* __restrict__ W,
                                                          const uint16_t* __restrict__ WT, uint32_t n,
                                                          const float* __restrict__ X,
                                                          const uint32_t* __restrict__ ROW,
                                                          const uint16_t* __restrict__ ADJ,
                                                          const uint32_t* __restrict__ META, float* __restrict__ Y) {
  __shared__ __align__(16) uint16_t w[2 * lds_mat(FIN) + 4 * lds_mat(H) + lds_mat(2 * H)];
  __shared__ __align__(16) float buf[FW][2 * MAXN * LR];
  auto stage = [&](uint16_t* dst, int off, int in) {
    const int pairs = in / 2;
    for (int e = threadIdx.x; e < H * pairs; e += FW * 64) {
      const int o = e / pairs, q = e % pairs;
      // matrices of the flat vector start at even words
      *(uint32_t*)(dst + o * (in + 4) + 2 * q) = *(const uint32_t*)(WT + off + o * in + 2 * q);
    }
  };
  uint16_t *ws0 = w, *wn0 = ws0 + lds_mat(FIN), *ws1 = wn0 + lds_mat(FIN), *wn1 = ws1 + lds_mat(H),
           *ws2 = wn1 + lds_mat(H), *wn2 = ws2 + lds_mat(H), *wr = wn2 + lds_mat(H);
  stage(ws0, O_WS0, FIN);
  stage(wn0, O_WN0, FIN);
  stage(ws1, O_WS1, H);
  stage(wn1, O_WN1, H);
  stage(ws2, O_WS2, H);
  stage(wn2, O_WN2, H);
  stage(wr, O_WR, 2 * H);
  __syncthreads();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = threadIdx.x & 63;
  float* h = buf[wave];
  float* a = h + MAXN * LR;
  const float br = bf(W, O_BR + j), wo = bf(W, O_WO + j), bo = bf(W, O_BO);
  for (uint32_t s = blockIdx.x * FW + wave; s < n; s += gridDim.x * FW) {
    const uint32_t meta = META[s];
    const int k = meta & 0xFF;
    const uint32_t smask = meta >> 16;
    const uint32_t adjv = j < MAXN ? ADJ[(uint64_t)s * MAXN + j] : 0u;
    load_features(X + (uint64_t)ROW[s] * FIN, k, h, LR);
    wave_sync();
    neighbour_sums(h, a, LR, FIN, k, adjv);
    wave_sync();
    layer<FIN>(h, a, LR, ws0, wn0, FIN + 4, W + O_B0, k, h);
    neighbour_sums(h, a, LR, H, k, adjv);
    wave_sync();
    layer<H>(h, a, LR, ws1, wn1, H + 4, W + O_B1, k, h);
    neighbour_sums(h, a, LR, H, k, adjv);
    wave_sync();
    layer<H>(h, a, LR, ws2, wn2, H + 4, W + O_B2, k, h);
    float ss, sa;
    pool(h, k, smask, ss, sa);
    a[j] = ss;
    a[H + j] = sa;
    wave_sync();
    float z = br;
    for (int i = 0; i < 2 * H; i += 4) {
      const uint2 q = *(const uint2*)(wr + j * (2 * H + 4) + i);
      const f4 c = *(const f4*)(a + i);
      z += lo16(q.x) * c[0];
      z += hi16(q.x) * c[1];
      z += lo16(q.y) * c[2];
      z += hi16(q.y) * c[3];
    }
    const float y = wave_total(fmaxf(z, 0.f) * wo) + bo;
    if (j == 0) Y[s] = y;
    wave_sync();  // the next sample overwrites a and h
  }
}

namespace {

// Forward state of one sample that its gradients need, and the gradients of
// the layers' pre-activations (dz[2] starts as the last layer's output).
struct Sample {
  float h0[MAXN * LF], a0[MAXN * LF];
  float h[2][MAXN * LR], a[2][MAXN * LR];
  float dz[3][MAXN * LR];
  float t[MAXN * LR];
  float c[2 * H], dzr[H];
};

// acc[mt] += (rows mt*16 .. of X^T) times (columns of D): the outer products
// of the 16 vertices' inputs X (LDS rows of ldx words) with their
// pre-activation gradients d[t] (this lane's column of D for the vertices
// g*4 + t).
template <int MT>
__device__ __forceinline__ void outer(f4 (&acc)[MT], const float* X, int ldx, int cols, const float (&d)[4]) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float x[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = mt * 16 + i < cols ? X[(g * 4 + t) * ldx + mt * 16 + i] : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], d[t], acc[mt], 0, 0, 0);
  }
}

// A gradient matrix's tiles (all inputs x this wave's 16 columns) to the
// block's partial row.
template <int MT>
__device__ __forceinline__ void put(const f4 (&acc)[MT], float* G, int rows) {
  const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4, wave = (threadIdx.x >> 6) & 3;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = mt * 16 + 4 * g + r;
      if (row < rows) G[row * H + wave * 16 + j] = acc[mt][r];
    }
}

}  // namespace

// Forward + backward, four samples at a time per block (one per wave; waves
// without one add zeros); the block's gradient sum goes to
// part[blockIdx.x][NPARAM], its squared error to loss[blockIdx.x].  Loss =
// mean over the n samples of (y - t)^2.  The forward state of four samples
// fills the CU's LDS (157 KB), so a block has the CU to itself; the weights
// come from L2.
constexpr int BW = 4;
__global__ __launch_bounds__(BW * 64) void k_mpnn_backward(const uint16_t* __restrict__ W,
                                                           const uint16_t* __restrict__ WT, uint32_t n,
                                                           const float* __restrict__ X,
                                                           const uint32_t* __restrict__ ROW,
                                                           const uint16_t* __restrict__ ADJ,
                                                           const uint32_t* __restrict__ META,
                                                           const float* __restrict__ T, float* __restrict__ part,
                                                           float* __restrict__ loss) {
  __shared__ __align__(16) Sample S[BW];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, j = lane, col = (int)wave * 16 + (lane & 15), g = lane >> 4;
  Sample& A = S[wave];
  const float inv_n = 1.f / (float)n;
  // gradient tiles of this wave's 16 columns, and its bias columns
  f4 gs0[2] = {}, gn0[2] = {}, gs1[4] = {}, gn1[4] = {}, gs2[4] = {}, gn2[4] = {}, gr[8] = {};
  float gb[3] = {0.f, 0.f, 0.f}, gwo = 0.f, gbr = 0.f, gbo = 0.f, lsum = 0.f;
  for (uint32_t s0 = blockIdx.x * BW; s0 < n; s0 += gridDim.x * BW) {
    const uint32_t s = s0 + wave;
    if (s < n) {
      const uint32_t meta = META[s];
      const int k = meta & 0xFF;
      const uint32_t smask = meta >> 16;
      const uint32_t adjv = j < MAXN ? ADJ[(uint64_t)s * MAXN + j] : 0u;
      load_features(X + (uint64_t)ROW[s] * FIN, k, A.h0, LF);
      wave_sync();
      neighbour_sums(A.h0, A.a0, LF, FIN, k, adjv);
      wave_sync();
      layer<FIN>(A.h0, A.a0, LF, WT + O_WS0, WT + O_WN0, FIN, W + O_B0, k, A.h[0]);
      neighbour_sums(A.h[0], A.a[0], LR, H, k, adjv);
      wave_sync();
      layer<H>(A.h[0], A.a[0], LR, WT + O_WS1, WT + O_WN1, H, W + O_B1, k, A.h[1]);
      neighbour_sums(A.h[1], A.a[1], LR, H, k, adjv);
      wave_sync();
      layer<H>(A.h[1], A.a[1], LR, WT + O_WS2, WT + O_WN2, H, W + O_B2, k, A.dz[2]);
      float ss, sa;
      pool(A.dz[2], k, smask, ss, sa);
      A.c[j] = ss;
      A.c[H + j] = sa;
      wave_sync();
      // z_j = br_j + sum_i Wr[i][j] c_i: the input-major copy, one coalesced row per i
      float z = bf(W, O_BR + j);
#pragma unroll 8
      for (int i = 0; i < 2 * H; ++i) z += bf(W, O_WR + i * H + j) * A.c[i];
      const float wo = bf(W, O_WO + j), rj = fmaxf(z, 0.f);
      const float e = wave_total(rj * wo) + bf(W, O_BO) - T[s];
      lsum += e * e;
      const float dy = 2.f * e * inv_n;
      gwo += dy * rj;
      gbo += dy;
      const float dzrj = z > 0.f ? dy * wo : 0.f;
      gbr += dzrj;
      A.dzr[j] = dzrj;
      wave_sync();
      // dc_i = sum_o Wr[i][o] dzr[o]: the transposed copy, one coalesced row per o
      float dcS = 0.f, dcA = 0.f;
#pragma unroll 8
      for (int o = 0; o < H; ++o) {
        dcS += bf(WT, O_WR + o * 2 * H + j) * A.dzr[o];
        dcA += bf(WT, O_WR + o * 2 * H + H + j) * A.dzr[o];
      }
      dcA = dcA / (float)k;
      for (int v = 0; v < k; ++v) {
        const float d = ((smask >> v & 1) ? dcS : 0.f) + dcA;
        A.dz[2][v * LR + j] = A.dz[2][v * LR + j] > 0.f ? d : 0.f;
      }
      wave_sync();
      // inputs' gradients, layer 2 then 1: dz . Ws^T and the neighbours' dz . Wn^T
#pragma unroll
      for (int l = 2; l >= 1; --l) {
        f4 ds[4] = {}, dn[4] = {};
        mfma_rows<H, 4>(ds, A.dz[l], LR, W + (l == 2 ? O_WS2 : O_WS1), H);
        mfma_rows<H, 4>(dn, A.dz[l], LR, W + (l == 2 ? O_WN2 : O_WN1), H);
        store_acc(ds, A.dz[l - 1], LR);
        store_acc(dn, A.t, LR);
        wave_sync();
        for (int v = 0; v < MAXN; ++v) {
          float d = 0.f;
          if (v < k && A.h[l - 1][v * LR + j] > 0.f) {
            d = A.dz[l - 1][v * LR + j];
            for (uint32_t m = lane_of(adjv, v); m; m &= m - 1) d += A.t[__builtin_ctz(m) * LR + j];
          }
          A.dz[l - 1][v * LR + j] = d;
        }
        wave_sync();
      }
    } else {
      for (int q = lane; q < (int)(sizeof(Sample) / 4); q += 64) ((float*)&A)[q] = 0.f;
    }
    __syncthreads();
    // every wave adds the four samples' outer products for its 16 columns
#pragma unroll 1
    for (int b = 0; b < BW; ++b) {
      const Sample& B = S[b];
      float d[3][4];
#pragma unroll
      for (int l = 0; l < 3; ++l)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          d[l][t] = B.dz[l][(g * 4 + t) * LR + col];
          gb[l] += d[l][t];
        }
      outer<2>(gs0, B.h0, LF, FIN, d[0]);
      outer<2>(gn0, B.a0, LF, FIN, d[0]);
      outer<4>(gs1, B.h[0], LR, H, d[1]);
      outer<4>(gn1, B.a[0], LR, H, d[1]);
      outer<4>(gs2, B.h[1], LR, H, d[2]);
      outer<4>(gn2, B.a[1], LR, H, d[2]);
    }
    // the readout's: the four samples are the product's four inputs
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
      gr[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[g].c[mt * 16 + (lane & 15)], S[g].dzr[col], gr[mt], 0, 0, 0);
    __syncthreads();
  }
  float* G = part + (uint64_t)blockIdx.x * NPARAM;  // this block's gradient sum
  put<2>(gs0, G + O_WS0, FIN);
  put<2>(gn0, G + O_WN0, FIN);
  put<4>(gs1, G + O_WS1, H);
  put<4>(gn1, G + O_WN1, H);
  put<4>(gs2, G + O_WS2, H);
  put<4>(gn2, G + O_WN2, H);
  put<8>(gr, G + O_WR, 2 * H);
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    float b = gb[l];
    b += __shfl_xor(b, 16);
    b += __shfl_xor(b, 32);
    if (g == 0) G[(l == 0 ? O_B0 : l == 1 ? O_B1 : O_B2) + col] = b;
  }
  // per-sample columns, summed over the waves
  float* x = (float*)&S[0];
  x[wave * H + j] = gwo;
  x[(BW + wave) * H + j] = gbr;
  if (lane == 0) {
    x[2 * BW * H + wave] = gbo;
    x[2 * BW * H + BW + wave] = lsum;
  }
  __syncthreads();
  if (wave == 0) {
    float o = 0.f, r = 0.f, bo = 0.f, ls = 0.f;
    for (int b = 0; b < BW; ++b) {
      o += x[b * H + j];
      r += x[(BW + b) * H + j];
      bo += x[2 * BW * H + b];
      ls += x[2 * BW * H + BW + b];
    }
    G[O_WO + j] = o;
    G[O_BR + j] = r;
    if (j == 0) {
      G[O_BO] = bo;
      loss[blockIdx.x] = ls * inv_n;
    }
  }
}

// grad[i] = sum of the blocks' partial rows: RS threads per parameter, each
// every RS-th row, so that a launch has enough loads in flight.
constexpr int RS = 16;
__global__ __launch_bounds__(64 * RS) void k_mpnn_reduce(const float* __restrict__ part, uint32_t nb,
                                                         float* __restrict__ grad) {
  __shared__ float s[RS][64];
  const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
  float t = 0.f;
  if (i < (uint32_t)NPARAM)
    for (uint32_t b = q; b < nb; b += RS) t += part[(uint64_t)b * NPARAM + i];
  s[q][threadIdx.x & 63] = t;
  __syncthreads();
  if (q == 0 && i < (uint32_t)NPARAM) {
    for (int r = 1; r < RS; ++r) t += s[r][threadIdx.x];
    grad[i] = t;
  }
}

// Adam step on the FP32 master copy (Kingma & Ba, 2015), then the two BF16
// copies.  t is the 1-based step number.
__global__ __launch_bounds__(256) void k_mpnn_adam(float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                                                   const float* __restrict__ g, float lr, float b1, float b2, float eps,
                                                   float c1, float c2) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint32_t)NPARAM) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 copies: W (input-major, as stored) and WT (each matrix transposed).
__global__ __launch_bounds__(256) void k_mpnn_pack(const float* __restrict__ p, uint16_t* __restrict__ W,
                                                   uint16_t* __restrict__ WT) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint32_t)NPARAM) return;
  const uint16_t b = to_bf16(p[i]);
  W[i] = b;
  // find the matrix containing i and its shape (rows = inputs, cols = outputs)
  int base = -1, rows = 0, cols = H;
  if (i < (uint32_t)O_WN0) { base = O_WS0; rows = FIN; }
  else if (i < (uint32_t)O_B0) { base = O_WN0; rows = FIN; }
  else if (i >= (uint32_t)O_WS1 && i < (uint32_t)O_WN1) { base = O_WS1; rows = H; }
  else if (i >= (uint32_t)O_WN1 && i < (uint32_t)O_B1) { base = O_WN1; rows = H; }
  else if (i >= (uint32_t)O_WS2 && i < (uint32_t)O_WN2) { base = O_WS2; rows = H; }
  else if (i >= (uint32_t)O_WN2 && i < (uint32_t)O_B2) { base = O_WN2; rows = H; }
  else if (i >= (uint32_t)O_WR && i < (uint32_t)O_BR) { base = O_WR; rows = 2 * H; }
  if (base < 0) {
    WT[i] = b;
    return;
  }
  const uint32_t off = i - base, r = off / cols, c = off % cols;  // W[r][c]
  WT[base + c * rows + r] = b;
}

// ------------------------------------------------------------------ host
template <typename T>
static T* malloc_dev(uint64_t n) {
  return (T*)mpnn_malloc(n * sizeof(T));
}

void mpnn_init(Context& c, Mpnn& n, const float* params) {
  HIPCHECK(hipSetDevice(c.device));
  n.ctx = &c;
  n.p = malloc_dev<float>(NPARAM);
  n.m = malloc_dev<float>(NPARAM);
  n.v = malloc_dev<float>(NPARAM);
  n.g = malloc_dev<float>(NPARAM);
  n.w = malloc_dev<uint16_t>(NPARAM);
  n.wt = malloc_dev<uint16_t>(NPARAM);
  n.nblocks = (uint32_t)c.cus;
  n.part = malloc_dev<float>((uint64_t)n.nblocks * NPARAM);
  n.loss = malloc_dev<float>(n.nblocks);
  HIPCHECK(hipMemset(n.m, 0, NPARAM * 4));
  HIPCHECK(hipMemset(n.v, 0, NPARAM * 4));
  mpnn_set(n, params);
}

void mpnn_set(Mpnn& n, const float* params) {
  HIPCHECK(hipSetDevice(n.ctx->device));
  HIPCHECK(hipMemcpy(n.p, params, NPARAM * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mpnn_pack, dim3((NPARAM + 255) / 256), dim3(256), 0, n.ctx->stream, n.p, n.w, n.wt);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(n.ctx->stream));
  n.step = 0;
  HIPCHECK(hipMemset(n.m, 0, NPARAM * 4));
  HIPCHECK(hipMemset(n.v, 0, NPARAM * 4));
}

void mpnn_get(Mpnn& n, float* params) {
  HIPCHECK(hipSetDevice(n.ctx->device));
  HIPCHECK(hipMemcpy(params, n.p, NPARAM * 4, hipMemcpyDeviceToHost));
}

// What a call's copies to the GPU read (the samples' first rows; the staging
// area is the network's own), until the stream has drained.
struct Upload {
  hipStream_t s;
  std::vector<uint32_t> row;
  Upload(hipStream_t stream, uint32_t n) : s(stream), row(n) {}
  Upload(Upload&&) = default;
  ~Upload() { (void)hipStreamSynchronize(s); }
};

// Samples to the GPU.  From 1,024 samples on, their live rows go through pinned
// memory in chunks, each packed by the host's threads while the one before is
// on its way: 12,000 padded samples are 18 MB, and their copy from pageable
// memory took 0.5 ms of a call (825 -> 469 us).  The staging area
// belongs to the network, of at most 64 MiB; a call with more rows than that
// copies the padded samples as they are.
static Upload upload(Mpnn& n, uint32_t cnt, const float* x, const uint16_t* adj, const uint32_t* meta, const float* t) {
  constexpr uint64_t kMost = 64ull << 20;
  mpnn_reserve(n, cnt);
  hipStream_t s = n.ctx->stream;
  Upload u(s, cnt);
  HIPCHECK(hipMemcpyAsync(n.adj, adj, (uint64_t)cnt * MAXN * 2, hipMemcpyHostToDevice, s));
  HIPCHECK(hipMemcpyAsync(n.meta, meta, (uint64_t)cnt * 4, hipMemcpyHostToDevice, s));
  if (t) HIPCHECK(hipMemcpyAsync(n.t, t, (uint64_t)cnt * 4, hipMemcpyHostToDevice, s));
  uint64_t rows = 0;
  for (uint32_t i = 0; i < cnt; ++i) {
    u.row[i] = (uint32_t)rows;
    rows += meta[i] & 0xFF;
  }
  const uint64_t bytes = rows * FIN * 4;
  bool staged = cnt >= 1024 && bytes <= kMost;
  if (staged && n.staged < bytes) {
    if (n.stage) (void)hipHostFree(n.stage);
    n.stage = nullptr;
    n.staged = 4ull << 20;
    while (n.staged < bytes) n.staged *= 2;
    if (hipHostMalloc(&n.stage, n.staged, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      n.stage = nullptr;
      n.staged = 0;
      staged = false;
    }
  }
  if (staged) {
    const uint32_t chunk = std::max<uint32_t>(512, (cnt + 7) / 8);
    for (uint32_t f = 0; f < cnt; f += chunk) {
      const uint32_t l = std::min(cnt, f + chunk);
      const uint64_t r0 = u.row[f], r1 = l < cnt ? u.row[l] : rows;
      pack_rows(x, meta, u.row.data(), f, l, n.stage + r0 * FIN);
      HIPCHECK(hipMemcpyAsync(n.x + r0 * FIN, n.stage + r0 * FIN, (r1 - r0) * FIN * 4, hipMemcpyHostToDevice, s));
    }
  } else {
    for (uint32_t i = 0; i < cnt; ++i) u.row[i] = i * MAXN;
    HIPCHECK(hipMemcpyAsync(n.x, x, (uint64_t)cnt * MAXN * FIN * 4, hipMemcpyHostToDevice, s));
  }
  HIPCHECK(hipMemcpyAsync(n.row, u.row.data(), (uint64_t)cnt * 4, hipMemcpyHostToDevice, s));
  return u;
}

static void check_meta(uint32_t cnt, const uint32_t* meta) {
  for (uint32_t i = 0; i < cnt; ++i) {
    const uint32_t k = meta[i] & 0xFF;
    if (k < 1 || k > (uint32_t)MAXN) throw Error(-1, "mpnn: sample with k outside 1..16");
  }
}

void mpnn_forward(Mpnn& n, uint32_t cnt, const float* x, const uint16_t* adj, const uint32_t* meta, float* y) {
  HIPCHECK(hipSetDevice(n.ctx->device));
  if (!cnt) return;
  check_meta(cnt, meta);
  const Upload held = upload(n, cnt, x, adj, meta, nullptr);
  const uint32_t grid = std::min<uint32_t>((cnt + FW - 1) / FW, (uint32_t)n.ctx->cus);
  hipLaunchKernelGGL(k_mpnn_forward, dim3(grid), dim3(FW * 64), 0, n.ctx->stream, n.w, n.wt, cnt, n.x, n.row, n.adj,
                     n.meta, n.y);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipMemcpyAsync(y, n.y, (uint64_t)cnt * 4, hipMemcpyDeviceToHost, n.ctx->stream));
  HIPCHECK(hipStreamSynchronize(n.ctx->stream));
}

double mpnn_gradient(Mpnn& n, uint32_t cnt, const float* x, const uint16_t* adj, const uint32_t* meta,
                     const float* t, float* grad_out) {
  HIPCHECK(hipSetDevice(n.ctx->device));
  if (!cnt) throw Error(-1, "mpnn: empty batch");
  check_meta(cnt, meta);
  const Upload held = upload(n, cnt, x, adj, meta, t);
  const uint32_t nb = std::min<uint32_t>(n.nblocks, (cnt + BW - 1) / BW);
  hipLaunchKernelGGL(k_mpnn_backward, dim3(nb), dim3(BW * 64), 0, n.ctx->stream, n.w, n.wt, cnt, n.x, n.row, n.adj,
                     n.meta, n.t, n.part, n.loss);
  HIPCHECK(hipGetLastError());
  hipLaunchKernelGGL(k_mpnn_reduce, dim3((NPARAM + 63) / 64), dim3(64 * RS), 0, n.ctx->stream, n.part, nb, n.g);
  HIPCHECK(hipGetLastError());
  std::vector<float> l(nb);
  HIPCHECK(hipMemcpyAsync(l.data(), n.loss, nb * 4, hipMemcpyDeviceToHost, n.ctx->stream));
  if (grad_out) HIPCHECK(hipMemcpyAsync(grad_out, n.g, NPARAM * 4, hipMemcpyDeviceToHost, n.ctx->stream));
  HIPCHECK(hipStreamSynchronize(n.ctx->stream));
  double s = 0;
  for (float v : l) s += v;
  return s;
}

double mpnn_train_step(Mpnn& n, uint32_t cnt, const float* x, const uint16_t* adj, const uint32_t* meta,
                       const float* t, float lr) {
  const double loss = mpnn_gradient(n, cnt, x, adj, meta, t, nullptr);
  n.step++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)n.step), c2 = 1.f - std::pow(b2, (float)n.step);
  hipLaunchKernelGGL(k_mpnn_adam, dim3((NPARAM + 255) / 256), dim3(256), 0, n.ctx->stream, n.p, n.m, n.v, n.g, lr, b1,
                     b2, 1e-8f, c1, c2);
  hipLaunchKernelGGL(k_mpnn_pack, dim3((NPARAM + 255) / 256), dim3(256), 0, n.ctx->stream, n.p, n.w, n.wt);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(n.ctx->stream));
  return loss;
}

}  // namespace cuts
