// Learned subgrid closure (no reference counterpart): an FP32 MLP
// (n_in -> H -> H -> n_out, GELU) trained and evaluated by the project's own kernels, the
// fine -> coarse L2 projection that builds its training data, and the glue that turns a
// coarse model's state into MLP inputs and the MLP outputs into a tendency correction.
//
// Networks whose hidden layers are at most 256 wide (and whose row tile fits 64 KiB of LDS) run
// on two FP32 matrix-core kernels: k_mlp_rows takes 16 rows of the batch through the whole
// network, forward and, for training, backward, with the activations in LDS and the weights
// read from L2; k_mlp_weight_grad forms all weight and bias gradients (A^T D over the batch) in
// one launch, split over the rows, and k_sum_splits adds the splits in a fixed order, so
// training is deterministic.  Larger networks take layer-by-layer GEMMs: C[M,N] = op(A) op(B)
// with 64x64 output tiles staged through LDS (16-wide k slabs), 256 work-items computing 4x4
// outputs each, the reductions over the batch split and summed in the same way.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "closure.hpp"
#include "mlp_rows.hpp"
#include "../../include/self_amd.h"

using namespace selfamd;

namespace {

constexpr int TM = 64, TN = 64, TK = 16;

// C = op(A) * op(B) (+ bias[col]); op(A) is M x K, op(B) is K x N; lda/ldb are the row
// strides of the stored A/B.  EPI: 0 none, 1 bias, 2 bias + GELU (Z written to Zout too).
// Rows [kBegin, kEnd) of the reduction only (split-K); output to C + split*M*N when split.
template <bool TA, bool TB, int EPI>
__global__ void __launch_bounds__(256) k_gemm(const float *__restrict__ A, const float *__restrict__ B,
                                              float *__restrict__ C, float *__restrict__ Zout,
                                              const float *__restrict__ bias, int M, int N, int K, int lda, int ldb,
                                              int kChunk) {
  __shared__ float sA[TK][TM + 4];
  __shared__ float sB[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int row0 = blockIdx.y * TM, col0 = blockIdx.x * TN;
  const int kBegin = blockIdx.z * kChunk, kEnd = min(K, kBegin + kChunk);
  float acc[4][4] = {{0}};
  for (int k0 = kBegin; k0 < kEnd; k0 += TK) {
    for (int t = threadIdx.x; t < TK * TM; t += 256) {
      // consecutive work-items read consecutive addresses of the stored A
      const int kk = TA ? t / TM : t % TK, r = TA ? t % TM : t / TK;
      const int gr = row0 + r, gk = k0 + kk;
      float v = 0.f;
      if (gr < M && gk < kEnd) v = TA ? A[(size_t)gk * lda + gr] : A[(size_t)gr * lda + gk];
      sA[kk][r] = v;
    }
    for (int t = threadIdx.x; t < TK * TN; t += 256) {
      const int kk = TB ? t % TK : t / TN, c = TB ? t / TK : t % TN;
      const int gc = col0 + c, gk = k0 + kk;
      float v = 0.f;
      if (gc < N && gk < kEnd) v = TB ? B[(size_t)gc * ldb + gk] : B[(size_t)gk * ldb + gc];
      sB[kk][c] = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; kk++) {
      float a[4], b[4];
#pragma unroll
      for (int q = 0; q < 4; q++) { a[q] = sA[kk][ty * 4 + q]; b[q] = sB[kk][tx * 4 + q]; }
#pragma unroll
      for (int p = 0; p < 4; p++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[p][q] = fmaf(a[p], b[q], acc[p][q]);
    }
    __syncthreads();
  }
  float *Cs = C + (size_t)blockIdx.z * M * N;
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const int r = row0 + ty * 4 + p;
    if (r >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int c = col0 + tx * 4 + q;
      if (c >= N) continue;
      float v = acc[p][q];
      if (EPI >= 1) v += bias[c];
      if (EPI == 2) {
        Zout[(size_t)r * N + c] = v;
        v = gelu_f(v);
      }
      Cs[(size_t)r * N + c] = v;
    }
  }
}

// out[i] = sum_s parts[s*n + i] (fixed order), added to out[i] when accumulate is set
__global__ void k_sum_splits(const float *__restrict__ parts, float *__restrict__ out, int n, int splits,
                             int accumulate) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float s = 0.f;
  #pragma unroll 8
    for (int k = 0; k < splits; k++) s += parts[(size_t)k * n + i];
    out[i] = accumulate ? out[i] + s : s;
  }
}

__global__ void k_fill(float *__restrict__ p, float v, size_t n) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) p[t] = v;
}

// dY = 2 (Y - T) / n and the per-block partial loss sums
__global__ void k_mse(const float *__restrict__ Y, const float *__restrict__ T, float *__restrict__ dY,
                      float *__restrict__ partial, size_t n) {
  __shared__ float red[256];
  float s = 0.f;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    const float r = Y[t] - T[t];
    dY[t] = 2.f * r / (float)n;
    s += r * r;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// D = G .* gelu'(Z)
__global__ void k_gelu_back(float *__restrict__ D, const float *__restrict__ Z, size_t n) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
    D[t] = D[t] * gelu_grad_f(Z[t]);
}

// Adam (Kingma & Ba 2015) with bias correction
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                       size_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    const float gt = g[t];
    const float mt = b1 * m[t] + (1.f - b1) * gt;
    const float vt = b2 * v[t] + (1.f - b2) * gt * gt;
    m[t] = mt;
    v[t] = vt;
    p[t] = p[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
  }
}

}  // namespace

struct selfamd_mlp {
  int nIn = 0, nH = 0, nOut = 0, maxB = 0;
  size_t nParams = 0;
  float *memory = nullptr;  // all arrays below
  float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;  // packed W1 b1 W2 b2 W3 b3
  float *Z1 = nullptr, *H1 = nullptr, *Z2 = nullptr, *H2 = nullptr, *Y = nullptr, *dY = nullptr;
  float *D2 = nullptr, *D1 = nullptr, *parts = nullptr, *lossParts = nullptr;
  float *ones = nullptr;  // maxB ones: bias gradients are ones^T D through the split GEMM (layer-by-layer path)
  int splitsMax = 64;
  bool rows = false;  // the network runs on the row kernels (Z1, Z2 and ones are not allocated then)
  float *W1() { return params; }
  float *b1() { return params + (size_t)nIn * nH; }
  float *W2() { return b1() + nH; }
  float *b2() { return W2() + (size_t)nH * nH; }
  float *W3() { return b2() + nH; }
  float *b3() { return W3() + (size_t)nH * nOut; }
  size_t off_b1() const { return (size_t)nIn * nH; }
  size_t off_W2() const { return off_b1() + nH; }
  size_t off_b2() const { return off_W2() + (size_t)nH * nH; }
  size_t off_W3() const { return off_b2() + nH; }
  size_t off_b3() const { return off_W3() + (size_t)nH * nOut; }
};

namespace {

template <bool TA, bool TB, int EPI>
hipError_t gemm(const float *A, const float *B, float *C, float *Z, const float *bias, int M, int N, int K, int lda,
                int ldb, int splits, hipStream_t st) {
  const int kChunk = ((K + splits - 1) / splits + TK - 1) / TK * TK;
  dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM, splits);
  hipLaunchKernelGGL((k_gemm<TA, TB, EPI>), grid, 256, 0, st, A, B, C, Z, bias, M, N, K, lda, ldb, kChunk);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------
// Row kernels: 16 rows of the batch through the whole network on the FP32 matrix cores
// ------------------------------------------------------------------------------
constexpr int kRowMaxHidden = 256, kRowMaxOut = 256, kRowLds = 56 * 1024;  // 64 KiB with the static arrays
constexpr int kRowMaxRows = kRowTile * ((1 << 23) - 1);                    // blocks of 512, below 2^32 work-items

// kRowsForward: Y = net(X).  kRowsLoss: forward, dY = 2 (Y - T) / count, backward.
// kRowsBackward: forward, backward from the cotangent T.  kRowsClosure: features of the state,
// forward, FP64 correction and its mass integral.  kRowsClosureVjp: features of the state (also to
// Xout) and the output cotangent of the correction's cotangent lam (also to dY), forward, backward,
// and the state cotangent added to mu.
enum RowsMode { kRowsForward, kRowsLoss, kRowsBackward, kRowsClosure, kRowsClosureVjp };

struct RowsArgs {
  int nIn, nH, nO, B;
  int ldX, ldH, ldO;  // LDS row strides
  const float *W1, *b1, *W2, *b2, *W3, *b3;
  const float *X, *T;
  float *Y, *H1, *H2, *D1, *D2, *dY, *dX, *lossParts;
  float count;
  const double *S, *geom, *qW;
  const float *inMean, *inScale, *outMean, *outScale;
  double *corr, *massParts;
  int P, nVar, massVar;
  // kRowsClosureVjp: lamParts[nLamParts] add up to the sum of lam's mass variable over the mesh
  const double *lam, *lamParts;
  int nLamParts;
  double invArea;
  float *Xout;
  double *mu;
};

inline size_t rows_lds(int nIn, int nH, int nO) {
  return sizeof(float) * kRowTile * ((size_t)rows_ld(nIn) + 2 * rows_ld(nH) + rows_ld(nO));
}
inline bool rows_fit(int nIn, int nH, int nO, int maxB) {
  if (maxB > kRowMaxRows) return false;
  return nH <= kRowMaxHidden && nO <= kRowMaxOut && rows_lds(nIn, nH, nO) <= kRowLds;
}

// One 16 x 16 tile of rows(LDS) * weights: `b` holds the tile's first 64 reduction indices on
// entry, and the next 64 are loaded while the current ones are multiplied; during the last ones
// the first 64 indices of whatever this wavefront multiplies next are loaded into `next`, which
// stay in flight through the epilogue and the barrier.
template <bool TRANS, bool VEC, class Prefetch>
__device__ __forceinline__ f32x4 rows_tile(const float *rows, int ld, const RowsOperand &o, int n, int lane,
                                           float (&b)[16], Prefetch prefetch) {
  const float *mine = rows + (lane & 15) * ld + 4 * (lane >> 4);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int k0 = 0;
  for (; k0 + 64 < o.K; k0 += 64) {
    float t[16];
    rows_load<TRANS, VEC>(o, n, lane >> 4, k0 + 64, t);
    acc = rows_mul(mine + k0, b, acc);
#pragma unroll
    for (int q = 0; q < 16; q++) b[q] = t[q];
  }
  prefetch();
  return rows_mul(mine + k0, b, acc);
}

// What bounds it: latency.  The configured closure (51 -> 128 -> 128 -> 48) on 4096 rows is 0.24
// GFLOP, 1.6 us at the matrix cores' FP32 rate; a block has its 16 rows' layers in a chain of
// barriers, and 4096 rows are one block per CU.  So a wavefront keeps the weights of its columns
// in registers one piece ahead, across the layers, and one launch does the whole network: TILES
// 16-column tiles of the hidden layers per wavefront (1 up to 128 hidden units, 2 up to 256).
// Element (row, column) of a tile: lane group g holds rows 4 g .. 4 g + 3 of column lane % 16, the
// same in the forward and backward passes, so gelu'(z) stays in registers.
// Measured at that size, per launch: closure evaluation 9.5 us (32.8 us with 32 rows per block,
// FMA lanes and the weights loaded inside the reduction loop), forward + loss + backward
// 16.7 us and all weight gradients 7.9 us (with k_sum_splits, 4 us, about 29 us per training
// step where layer-by-layer GEMMs took 26 launches and 390 us).
template <int MODE, int TILES, bool VEC>
__global__ void __launch_bounds__(kRowThreads) k_mlp_rows(const RowsArgs a) {
  extern __shared__ __align__(16) float rowsLds[];
  __shared__ double sRed[kRowTile];
  // closure: output scale and mean, element J, and w_i w_j per node of the mass variable (0 for the
  // other outputs)
  __shared__ float sScale[MODE == kRowsClosure ? kRowMaxOut : 1], sMean[MODE == kRowsClosure ? kRowMaxOut : 1];
  __shared__ double sWeight[MODE == kRowsClosure ? kRowMaxOut : 1], sJ[MODE == kRowsClosure ? kRowTile : 1];
  float *sX = rowsLds, *sH1 = sX + kRowTile * a.ldX, *sH2 = sH1 + kRowTile * a.ldH, *sO = sH2 + kRowTile * a.ldH;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar branches on it
  const int row0 = blockIdx.x * kRowTile;
  constexpr bool VJP = MODE == kRowsClosureVjp, STATE = MODE == kRowsClosure || VJP;  // rows of a model's state
  constexpr bool GIVEN = MODE == kRowsBackward || VJP;                               // a given output cotangent
  constexpr bool BACK = MODE == kRowsLoss || GIVEN;
  const RowsOperand w1{a.W1, a.nH, a.nIn, a.nH}, w2{a.W2, a.nH, a.nH, a.nH}, w3{a.W3, a.nO, a.nH, a.nO};
  const RowsOperand t3{a.W3, a.nO, a.nO, a.nH}, t2{a.W2, a.nH, a.nH, a.nH}, t1{a.W1, a.nH, a.nH, a.nIn};
  const int n0 = wave * 16 + r;  // this lane's column of the wavefront's first tile of a layer
  float b[2][16];                // the weights in flight; a layer's first piece is in b[0]
  rows_load<false, VEC>(w1, n0, g, 0, b[0]);
  float bias1[TILES], bias2[TILES];
#pragma unroll
  for (int t = 0; t < TILES; t++) {
    const int n = min(n0 + 128 * t, a.nH - 1);
    bias1[t] = a.b1[n];
    bias2[t] = a.b2[n];
  }
  const float bias3 = a.b3[min(n0, a.nO - 1)];
  const int H16 = pad16(a.nH), O16 = pad16(a.nO);
  // input rows and the zero columns of the other operands: 32 work-items per row
  {
    const int row = tid >> 5, c = tid & 31, KX = pad64(a.nIn), KH = pad64(a.nH), KO = pad64(a.nO);
    const bool ok = row0 + row < a.B;
    const size_t e = (size_t)(ok ? row0 + row : 0);
    if constexpr (MODE == kRowsClosure) {
      for (int k = tid; k < a.nO; k += kRowThreads) {
        sScale[k] = a.outScale[k];
        sMean[k] = a.outMean[k];
        const int node = k - a.massVar * a.P * a.P;
        sWeight[k] = node >= 0 && node < a.P * a.P ? a.qW[node % a.P] * a.qW[node / a.P] : 0.0;
      }
      if (c == 0) sJ[row] = ok ? a.geom[e * kGeomStride + 4] : 0.0;
    }
    // two values at a time, loaded before either is used: the launch starts with these loads'
    // round trips to memory (positions past the row read one in it)
    const int nS = a.nVar * a.P * a.P;
    for (int k = c; k < KX; k += 64) {
      double raw[2];
      float mu[2], sd[2], x[2];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int kk = min(k + 32 * j, a.nIn - 1);
        if constexpr (STATE) {
          const double *gr = a.geom + e * kGeomStride;
          raw[j] = *(kk < nS ? a.S + e * nS + kk : kk == nS ? gr + 4 : kk == nS + 1 ? gr : gr + 3);
          mu[j] = a.inMean[kk];
          sd[j] = a.inScale[kk];
        } else {
          x[j] = a.X[e * a.nIn + kk];
        }
      }
#pragma unroll
      for (int j = 0; j < 2; j++) {
        if constexpr (STATE) x[j] = (float)((raw[j] - (double)mu[j]) / (double)sd[j]);
        sX[row * a.ldX + k + 32 * j] = ok && k + 32 * j < a.nIn ? x[j] : 0.f;
        if constexpr (VJP)
          if (ok && k + 32 * j < a.nIn) a.Xout[e * a.nIn + k + 32 * j] = x[j];
      }
    }
    if constexpr (VJP) {
      // every wavefront adds the partial sums itself, in flight beside its other loads
      double total = 0.0;
      for (int k = lane; k < a.nLamParts; k += 256) {
        double t[4];
#pragma unroll
        for (int j = 0; j < 4; j++) t[j] = a.lamParts[min(k + 64 * j, a.nLamParts - 1)];
#pragma unroll
        for (int j = 0; j < 4; j++) total += k + 64 * j < a.nLamParts ? t[j] : 0.0;
      }
      for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off, 64);
      // Forward: corr_k = y_k outScale_k + outMean_k, and for the mass variable corr' = corr - invArea
      // sum_n omega_n corr_n (omega = w_i w_j J); so dY_k = outScale_k (lam_k - omega_k invArea
      // sum_n lam_n) on the mass variable, outScale_k lam_k elsewhere.
      const double J = a.geom[e * kGeomStride + 4];
      for (int k = c; k < O16; k += 32) {
        const int kk = min(k, a.nO - 1), node = kk - a.massVar * a.P * a.P;
        double l = a.lam[e * a.nO + kk];
        if (node >= 0 && node < a.P * a.P) l -= a.qW[node % a.P] * a.qW[node / a.P] * J * a.invArea * total;
        const float d = (float)(l * (double)a.outScale[kk]);
        const bool in = ok && k < a.nO;
        sO[row * a.ldO + k] = in ? d : 0.f;
        if (in) a.dY[e * a.nO + k] = d;
      }
    }
    for (int k = H16 + c; k < KH; k += 32) sH1[row * a.ldH + k] = sH2[row * a.ldH + k] = 0.f;
    for (int k = O16 + c; k < KO; k += 32) sO[row * a.ldO + k] = 0.f;
  }
  __syncthreads();

  float gp1[TILES][4], gp2[TILES][4];
  // the tiles of one hidden-width layer of this wavefront, b[0] holding the first one's first
  // piece: epilogue(t, n, acc) takes each tile; `after` loads the next layer's first piece
  auto layer = [&](auto trans, const float *in, int ld, const RowsOperand &o, auto epilogue, auto after) {
    constexpr bool TR = decltype(trans)::value;
    if (wave * 16 >= H16) {
      after(b[0]);
      return;
    }
    const bool two = TILES > 1 && (wave + kRowWaves) * 16 < H16;
    if (!two) {
      const f32x4 acc = rows_tile<TR, VEC>(in, ld, o, n0, lane, b[0], [&] { after(b[1]); });
      epilogue(std::integral_constant<int, 0>{}, n0, acc);
    } else {
      const f32x4 acc = rows_tile<TR, VEC>(in, ld, o, n0, lane, b[0], [&] { rows_load<TR, VEC>(o, n0 + 128, g, 0, b[1]); });
      epilogue(std::integral_constant<int, 0>{}, n0, acc);
      float cur[16];
#pragma unroll
      for (int q = 0; q < 16; q++) cur[q] = b[1][q];
      const f32x4 acc1 = rows_tile<TR, VEC>(in, ld, o, n0 + 128, lane, cur, [&] { after(b[1]); });
      epilogue(std::integral_constant<int, TILES - 1>{}, n0 + 128, acc1);
    }
#pragma unroll
    for (int q = 0; q < 16; q++) b[0][q] = b[1][q];
  };
  // out = gelu(in W + bias), gelu' kept, the activations also to memory for the weight gradients
  auto hidden = [&](const float *in, int ld, const RowsOperand &o, const float (&bias)[TILES], float *out, float *mem,
                    float (&gp)[TILES][4], auto after) {
    layer(std::false_type{}, in, ld, o, [&](auto t, int n, f32x4 acc) {
      const bool ok = n < a.nH;
      const float bn = bias[decltype(t)::value];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float z = acc[i] + bn;
        float h, d;
        gelu_pair(z, h, d);
        out[(4 * g + i) * a.ldH + n] = h = ok ? h : 0.f;
        if constexpr (BACK) {
          gp[decltype(t)::value][i] = d;
          if (ok && row0 + 4 * g + i < a.B) mem[(size_t)(row0 + 4 * g + i) * a.nH + n] = h;
        }
      }
    }, after);
  };
  hidden(sX, a.ldX, w1, bias1, sH1, a.H1, gp1, [&](float (&x)[16]) { rows_load<false, VEC>(w2, n0, g, 0, x); });
  __syncthreads();
  hidden(sH1, a.ldH, w2, bias2, sH2, a.H2, gp2, [&](float (&x)[16]) {
    if constexpr (GIVEN) rows_load<true, VEC>(t3, n0, g, 0, x);
    else rows_load<false, VEC>(w3, n0, g, 0, x);
  });
  if constexpr (!GIVEN) __syncthreads();

  // output layer
  float loss = 0.f;
  if constexpr (MODE == kRowsBackward) {
    // the cotangent is given: the output itself is not needed
    const int row = tid >> 5;
    const bool ok = row0 + row < a.B;
    for (int k = tid & 31; k < O16; k += 32)
      sO[row * a.ldO + k] = ok && k < a.nO ? a.T[(size_t)(row0 + row) * a.nO + k] : 0.f;
  } else if constexpr (!VJP) {
    for (int ct = wave; ct * 16 < O16; ct += kRowWaves) {
      const int n = ct * 16 + r;
      const bool nok = n < a.nO;
      float tv[4];
      if constexpr (MODE == kRowsLoss) {
#pragma unroll
        for (int i = 0; i < 4; i++) tv[i] = a.T[(size_t)min(row0 + 4 * g + i, a.B - 1) * a.nO + (nok ? n : 0)];
      }
      if (ct != wave) rows_load<false, VEC>(w3, n, g, 0, b[0]);
      const f32x4 acc = rows_tile<false, VEC>(sH2, a.ldH, w3, n, lane, b[0], [] {});
      const float bn = ct == wave ? bias3 : a.b3[nok ? n : 0];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = row0 + 4 * g + i;
        const bool ok = nok && row < a.B;
        float y = nok ? acc[i] + bn : 0.f;
        if constexpr (MODE == kRowsForward) {
          if (ok) a.Y[(size_t)row * a.nO + n] = y;
        } else {
          if constexpr (MODE == kRowsLoss) {
            const float d = ok ? y - tv[i] : 0.f;
            loss += d * d;
            y = 2.f * d / a.count;
            if (ok) a.dY[(size_t)row * a.nO + n] = y;
          }
          sO[(4 * g + i) * a.ldO + n] = y;
        }
      }
    }
    if constexpr (MODE == kRowsLoss) rows_load<true, VEC>(t3, n0, g, 0, b[0]);
  }
  if constexpr (MODE == kRowsForward) return;
  if constexpr (MODE == kRowsClosure) {
    __syncthreads();
    const int row = tid >> 5;
    const size_t e = (size_t)row0 + row;
    double m = 0.0;
    for (int k = tid & 31; k < a.nO; k += 32) {
      const double c = (double)sO[row * a.ldO + k] * (double)sScale[k] + (double)sMean[k];
      if (e < (size_t)a.B) a.corr[e * a.nO + k] = c;
      m += sWeight[k] * c;
    }
    for (int off = 16; off > 0; off >>= 1) m += __shfl_xor(m, off, 32);
    if ((tid & 31) == 0) sRed[row] = sJ[row] * m;
    __syncthreads();
    if (wave == 0) {
      double s = sRed[lane & 15];
      for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 16);
      if (tid == 0) a.massParts[blockIdx.x] = s;
    }
  }
  if constexpr (BACK) {
    // D2 = (dY W3^T) gelu'(z2), D1 = (D2 W2^T) gelu'(z1), dX = D1 W1^T
    if constexpr (MODE == kRowsLoss) {
      for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
      if (lane == 0) sRed[wave] = loss;
    }
    __syncthreads();
    if constexpr (MODE == kRowsLoss) {
      if (tid == 0) {
        double s = 0.0;
        for (int k = 0; k < kRowWaves; k++) s += sRed[k];
        a.lossParts[blockIdx.x] = (float)s;
      }
    }
    auto back = [&](const float *in, int ld, const RowsOperand &o, float *out, float *mem, const float (&gp)[TILES][4],
                    auto after) {
      layer(std::true_type{}, in, ld, o, [&](auto t, int n, f32x4 acc) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float d = n < a.nH ? acc[i] * gp[decltype(t)::value][i] : 0.f;
          out[(4 * g + i) * a.ldH + n] = d;
          if (n < a.nH && row0 + 4 * g + i < a.B) mem[(size_t)(row0 + 4 * g + i) * a.nH + n] = d;
        }
      }, after);
    };
    back(sO, a.ldO, t3, sH2, a.D2, gp2, [&](float (&x)[16]) { rows_load<true, VEC>(t2, n0, g, 0, x); });
    __syncthreads();
    back(sH2, a.ldH, t2, sH1, a.D1, gp1, [&](float (&x)[16]) {
      if constexpr (GIVEN) rows_load<true, VEC>(t1, n0, g, 0, x);
    });
    if (MODE == kRowsLoss || (!VJP && !a.dX)) return;
    __syncthreads();
    // the metric inputs, past the nodal ones, do not depend on the state
    const int nX = VJP ? a.nO : a.nIn;
    for (int ct = wave; ct * 16 < nX; ct += kRowWaves) {
      const int n = ct * 16 + r;
      double m[4], sd = 1.0;
      if constexpr (VJP) {
        const int nn = min(n, nX - 1);
        sd = (double)a.inScale[nn];
#pragma unroll
        for (int i = 0; i < 4; i++) m[i] = a.mu[(size_t)min(row0 + 4 * g + i, a.B - 1) * nX + nn];
      }
      if (ct != wave) rows_load<true, VEC>(t1, n, g, 0, b[0]);
      const f32x4 acc = rows_tile<true, VEC>(sH1, a.ldH, t1, n, lane, b[0], [] {});
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (n < nX && row0 + 4 * g + i < a.B) {
          if constexpr (VJP) a.mu[(size_t)(row0 + 4 * g + i) * nX + n] = m[i] + (double)acc[i] / sd;
          else a.dX[(size_t)(row0 + 4 * g + i) * nX + n] = acc[i];
        }
    }
  }
}

// All weight and bias gradients of one split of the rows: gW = A^T D and gb = column sums of D for
// (A, D) = (X, D1), (H1, D2), (H2, dY), packed like the parameters at parts + split * nParams.  A
// wavefront forms a 32 x 32 tile of one gW, reading both operands straight from L2 (16
// consecutive floats per row and lane group); the tiles of the first 32 rows of a gW also sum D.
struct GradArgs {
  const float *A[3], *D[3];
  int M[3], N[3];
  size_t off[3];      // of the weights in the packed gradients; the bias follows them
  int tilesN[3], first[4];  // column tiles of each product; its first tile, and the total
  float *parts;
  size_t nParams;
  int B, rowsPerSplit;
};
__global__ void __launch_bounds__(256) k_mlp_weight_grad(const GradArgs a) {
  const int tile = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (tile >= a.first[3]) return;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int p = tile >= a.first[2] ? 2 : tile >= a.first[1] ? 1 : 0;
  const float *__restrict__ A = a.A[p], *__restrict__ D = a.D[p];
  const int M = a.M[p], N = a.N[p], local = tile - a.first[p];
  const int tm = local / a.tilesN[p], m0 = tm * 32, n0 = (local - tm * a.tilesN[p]) * 32;
  const int k0 = blockIdx.x * a.rowsPerSplit, k1 = min(a.B, k0 + a.rowsPerSplit);
  // columns past M and N read the last one; what they give is not stored
  const bool nok[2] = {n0 + r < N, n0 + 16 + r < N};
  const unsigned mi[2] = {(unsigned)min(m0 + r, M - 1), (unsigned)min(m0 + 16 + r, M - 1)};
  const unsigned ni[2] = {(unsigned)min(n0 + r, N - 1), (unsigned)min(n0 + 16 + r, N - 1)};
  // this split's rows; rows past its end read its last one
  const float *As = A + (size_t)k0 * M, *Ds = D + (size_t)k0 * N;
  const unsigned rows = k1 - k0;
  f32x4 acc[2][2] = {};
  float bias[2] = {0.f, 0.f};
  constexpr int U = 16;
  auto load = [&](int k, float (&av)[U][2], float (&dv)[U][2]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned row = min((unsigned)(k - k0 + 4 * u + g), rows - 1);
#pragma unroll
      for (int q = 0; q < 2; q++) {
        av[u][q] = load_at<float>(As, row * M + mi[q]);
        dv[u][q] = load_at<float>(Ds, row * N + ni[q]);
      }
    }
  };
  auto multiply = [&](int k, bool tail, float (&av)[U][2], float (&dv)[U][2]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (tail && k + 4 * u + g >= k1) dv[u][q] = av[u][q] = 0.f;
        bias[q] += dv[u][q];
      }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int q = 0; q < 2; q++) acc[s][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u][s], dv[u][q], acc[s][q], 0, 0, 0);
  };
  // 64 rows at a time, the next 64 in flight while the current ones are multiplied
  float av[U][2], dv[U][2];
  load(k0, av, dv);
  int k = k0;
  for (; k + 4 * U < k1; k += 4 * U) {
    float an[U][2], dn[U][2];
    load(k + 4 * U, an, dn);
    multiply(k, false, av, dv);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < 2; q++) { av[u][q] = an[u][q]; dv[u][q] = dn[u][q]; }
  }
  multiply(k, true, av, dv);
  float *out = a.parts + (size_t)blockIdx.x * a.nParams + a.off[p];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int m = m0 + 16 * s + 4 * g + i;
        if (m < M && nok[q]) out[(size_t)m * N + ni[q]] = acc[s][q][i];
      }
  if (tm == 0) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      float s = bias[q];
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (g == 0 && nok[q]) out[(size_t)M * N + ni[q]] = s;
    }
  }
}

RowsArgs rows_args(selfamd_mlp *m, const float *X, int B) {
  RowsArgs a{};
  a.nIn = m->nIn; a.nH = m->nH; a.nO = m->nOut; a.B = B;
  a.ldX = rows_ld(a.nIn); a.ldH = rows_ld(a.nH); a.ldO = rows_ld(a.nO);
  a.W1 = m->W1(); a.b1 = m->b1(); a.W2 = m->W2(); a.b2 = m->b2(); a.W3 = m->W3(); a.b3 = m->b3();
  a.X = X;
  a.H1 = m->H1; a.H2 = m->H2; a.D1 = m->D1; a.D2 = m->D2;
  return a;
}

template <int MODE>
hipError_t launch_rows(const RowsArgs &a, hipStream_t st) {
  const unsigned blocks = (unsigned)((a.B + kRowTile - 1) / kRowTile);
  const size_t lds = rows_lds(a.nIn, a.nH, a.nO);
  // the transposed weights of the backward pass are read 16 bytes at a time where every row of
  // W1, W2 and W3 is 16-byte aligned
  constexpr bool back = MODE == kRowsLoss || MODE == kRowsBackward || MODE == kRowsClosureVjp;
  const bool vec = back && a.nH % 4 == 0 && a.nO % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(a.W1) | reinterpret_cast<uintptr_t>(a.W2) |
                     reinterpret_cast<uintptr_t>(a.W3)) & 15) == 0;
  const bool one = a.nH <= 16 * kRowWaves;
  if (one && !vec) hipLaunchKernelGGL((k_mlp_rows<MODE, 1, false>), blocks, kRowThreads, lds, st, a);
  else if (!vec) hipLaunchKernelGGL((k_mlp_rows<MODE, 2, false>), blocks, kRowThreads, lds, st, a);
  else if constexpr (back) {
    if (one) hipLaunchKernelGGL((k_mlp_rows<MODE, 1, true>), blocks, kRowThreads, lds, st, a);
    else hipLaunchKernelGGL((k_mlp_rows<MODE, 2, true>), blocks, kRowThreads, lds, st, a);
  }
  return hipGetLastError();
}

// Parameter gradients from the activations and cotangents that k_mlp_rows left in memory.  At
// most 64 splits of at least 128 rows: all of a split's loads are then in flight at once, and
// with 64 rows the sum over twice the splits costs more than it saves (9.5 + 4.7 us against
// 7.9 + 3.6 us at 4096 rows).
hipError_t weight_grads_rows(selfamd_mlp *m, const float *X, const float *dY, int B, int accumulate, hipStream_t st) {
  GradArgs a{};
  const float *A[3] = {X, m->H1, m->H2}, *D[3] = {m->D1, m->D2, dY};
  const int M[3] = {m->nIn, m->nH, m->nH}, N[3] = {m->nH, m->nH, m->nOut};
  const size_t off[3] = {0, m->off_W2(), m->off_W3()};
  for (int p = 0; p < 3; p++) {
    a.A[p] = A[p]; a.D[p] = D[p]; a.M[p] = M[p]; a.N[p] = N[p]; a.off[p] = off[p];
    a.tilesN[p] = (N[p] + 31) / 32;
    a.first[p + 1] = a.first[p] + a.tilesN[p] * ((M[p] + 31) / 32);
  }
  a.parts = m->parts; a.nParams = m->nParams; a.B = B;
  const int perSplit = (B + m->splitsMax - 1) / m->splitsMax;
  a.rowsPerSplit = std::max(128, (perSplit + 31) / 32 * 32);
  const int splits = (B + a.rowsPerSplit - 1) / a.rowsPerSplit, n = (int)m->nParams;
  hipLaunchKernelGGL(k_mlp_weight_grad, dim3(splits, (a.first[3] + 3) / 4), 256, 0, st, a);
  hipError_t e = hipGetLastError();
  if (e) return e;
  hipLaunchKernelGGL(k_sum_splits, (n + 255) / 256, 256, 0, st, m->parts, m->grads, n, splits, accumulate);
  return hipGetLastError();
}

// Whether the forward pass of a row network goes layer by layer.  A block of the row kernel has 512
// work-items and 64 reduction indices a piece for its 16 rows, however narrow the network, and pays by
// the launches it saves; on many rows a narrow network's layers are the cheaper ones.  Layers and the row
// kernel, us (in, hidden, out): 1, 1, 1 on 16,384 rows 15 and 10, on 32,768 14 and 18, on 131,072 22 and
// 62; 16, 16, 16 on 32,768 24 and 19, on 65,536 30 and 35, on 400,000 128 and 189; 40, 48, 40 on 400,000
// 259 and 224.  The line follows where they cross over hidden widths 1 to 48 and inputs 1 to 120.
inline bool narrow_by_layers(int nIn, int nH, int B) {
  return nH <= 40 && B >= 24576 + 1280 * nH + 256 * std::min(nIn, 1024);
}
// Y = net(X); Y may lie over X.
hipError_t forward_impl(selfamd_mlp *m, const float *X, float *Y, int B, hipStream_t st) {
  hipError_t e;
  if (m->rows && !narrow_by_layers(m->nIn, m->nH, B)) {
    // a block writes its rows of Y while others still read theirs of X
    const size_t nY = sizeof(float) * (size_t)B * m->nOut;
    const bool over = ranges_overlap(Y, nY, X, sizeof(float) * (size_t)B * m->nIn);
    RowsArgs a = rows_args(m, X, B);
    a.Y = over ? m->Y : Y;
    if ((e = launch_rows<kRowsForward>(a, st)) || !over) return e;
    return hipMemcpyAsync(Y, m->Y, nY, hipMemcpyDeviceToDevice, st);
  }
  float *Z1 = m->rows ? m->D1 : m->Z1, *Z2 = m->rows ? m->D2 : m->Z2;  // no backward pass reads a row network's
  if ((e = gemm<false, false, 2>(X, m->W1(), m->H1, Z1, m->b1(), B, m->nH, m->nIn, m->nIn, m->nH, 1, st))) return e;
  if ((e = gemm<false, false, 2>(m->H1, m->W2(), m->H2, Z2, m->b2(), B, m->nH, m->nH, m->nH, m->nH, 1, st))) return e;
  return gemm<false, false, 1>(m->H2, m->W3(), Y, nullptr, m->b3(), B, m->nOut, m->nH, m->nH, m->nOut, 1, st);
}

// weight gradient gW[in, out] (+)= A^T D over B rows, split over blocks then summed in order
hipError_t weight_grad(selfamd_mlp *m, const float *A, const float *D, float *gW, int B, int nin, int nout,
                       hipStream_t st, int accumulate = 0) {
  int splits = (B + 255) / 256;
  if (splits > m->splitsMax) splits = m->splitsMax;
  if (splits < 1) splits = 1;
  hipError_t e = gemm<true, false, 0>(A, D, m->parts, nullptr, nullptr, nin, nout, B, nin, nout, splits, st);
  if (e) return e;
  const int n = nin * nout;
  hipLaunchKernelGGL(k_sum_splits, (n + 255) / 256, 256, 0, st, m->parts, gW, n, splits, accumulate);
  return hipGetLastError();
}

// Layer-by-layer backward pass from the output cotangent dY (overwritten) through the
// activations that the last forward_impl of the same rows left in Z1, H1, Z2, H2: parameter
// gradients written to (or, with accumulate, added to) m->grads, and the input cotangent
// dX = D1 W1^T when dX is given.
hipError_t backward_layers(selfamd_mlp *m, const float *X, float *dY, int B, int accumulate, float *dX,
                         hipStream_t st) {
  const int H = m->nH, nO = m->nOut;
  float *g = m->grads;
  hipError_t e;
  // layer 3
  if ((e = weight_grad(m, m->H2, dY, g + m->off_W3(), B, H, nO, st, accumulate))) return e;
  if ((e = weight_grad(m, m->ones, dY, g + m->off_b3(), B, 1, nO, st, accumulate))) return e;
  if ((e = gemm<false, true, 0>(dY, m->W3(), m->D2, nullptr, nullptr, B, H, nO, nO, nO, 1, st))) return e;
  hipLaunchKernelGGL(k_gelu_back, (int)std::min<size_t>(((size_t)B * H + 255) / 256, 4096), 256, 0, st, m->D2, m->Z2,
                     (size_t)B * H);
  // layer 2
  if ((e = weight_grad(m, m->H1, m->D2, g + m->off_W2(), B, H, H, st, accumulate))) return e;
  if ((e = weight_grad(m, m->ones, m->D2, g + m->off_b2(), B, 1, H, st, accumulate))) return e;
  if ((e = gemm<false, true, 0>(m->D2, m->W2(), m->D1, nullptr, nullptr, B, H, H, H, H, 1, st))) return e;
  hipLaunchKernelGGL(k_gelu_back, (int)std::min<size_t>(((size_t)B * H + 255) / 256, 4096), 256, 0, st, m->D1, m->Z1,
                     (size_t)B * H);
  // layer 1
  if ((e = weight_grad(m, X, m->D1, g, B, m->nIn, H, st, accumulate))) return e;
  if ((e = weight_grad(m, m->ones, m->D1, g + m->off_b1(), B, 1, H, st, accumulate))) return e;
  if (dX && (e = gemm<false, true, 0>(m->D1, m->W1(), dX, nullptr, nullptr, B, m->nIn, H, H, H, 1, st))) return e;
  return hipGetLastError();
}

// Forward pass of X and backward pass from the output cotangent dY: parameter gradients written
// to (or, with accumulate, added to) m->grads, and the input cotangent when dX is given; dX may lie
// over X or dY.
hipError_t backward_impl(selfamd_mlp *m, const float *X, const float *dY, int B, int accumulate, float *dX,
                         hipStream_t st) {
  hipError_t e;
  if (m->rows) {
    // The weight gradients read X and dY after k_mlp_rows: where dX lies over one of them it is
    // formed last, as a product of its own.
    const size_t nX = sizeof(float) * (size_t)B * m->nIn, nY = sizeof(float) * (size_t)B * m->nOut;
    const bool last = dX && (ranges_overlap(dX, nX, X, nX) || ranges_overlap(dX, nX, dY, nY));
    RowsArgs a = rows_args(m, X, B);
    a.T = dY; a.dX = last ? nullptr : dX;
    if ((e = launch_rows<kRowsBackward>(a, st))) return e;
    if ((e = weight_grads_rows(m, X, dY, B, accumulate, st)) || !last) return e;
    return gemm<false, true, 0>(m->D1, m->W1(), dX, nullptr, nullptr, B, m->nIn, m->nH, m->nH, m->nH, 1, st);
  }
  if ((e = forward_impl(m, X, m->Y, B, st))) return e;
  if ((e = hipMemcpyAsync(m->dY, dY, sizeof(float) * (size_t)B * m->nOut, hipMemcpyDeviceToDevice, st))) return e;
  return backward_layers(m, X, m->dY, B, accumulate, dX, st);
}

}  // namespace

extern "C" {

int selfamd_mlp_create(selfamd_mlp **out, int nIn, int nHidden, int nOut, int maxBatch) {
  SELFAMD_REQUIRE(out && nIn > 0 && nHidden > 0 && nOut > 0 && maxBatch > 0, "mlp_create: bad sizes");
  *out = nullptr;
  selfamd_mlp *m = new selfamd_mlp();
  m->nIn = nIn; m->nH = nHidden; m->nOut = nOut; m->maxB = maxBatch;
  m->nParams = (size_t)nIn * nHidden + nHidden + (size_t)nHidden * nHidden + nHidden + (size_t)nHidden * nOut + nOut;
  const size_t B = maxBatch, H = nHidden;
  m->rows = rows_fit(nIn, nHidden, nOut, maxBatch);
  // One allocation for all arrays (a call each takes longer than the kernels of a training step),
  // each 256-byte aligned; the partial gradients are of at most 64 splits of at least 128 rows.
  const size_t lossBlocks = std::max<size_t>(1024, (B + kRowTile - 1) / kRowTile);
  const size_t splits = std::min<size_t>(m->splitsMax, (B + 127) / 128), general = m->rows ? 0 : B;
  const struct { float **at; size_t n; } arrays[] = {
      {&m->params, m->nParams}, {&m->m1, m->nParams}, {&m->m2, m->nParams}, {&m->grads, m->nParams},
      {&m->H1, B * H}, {&m->H2, B * H}, {&m->Y, B * nOut}, {&m->dY, B * nOut}, {&m->D2, B * H}, {&m->D1, B * H},
      {&m->parts, m->nParams * splits}, {&m->lossParts, lossBlocks},
      {&m->Z1, general * H}, {&m->Z2, general * H}, {&m->ones, general}};
  auto padded = [](size_t n) { return (n + 63) & ~(size_t)63; };
  size_t total = 0;
  for (const auto &a : arrays) total += padded(a.n);
  bool ok = hipMalloc(&m->memory, 4 * total) == hipSuccess;
  if (ok) {
    float *p = m->memory;
    for (const auto &a : arrays) {
      *a.at = a.n ? p : nullptr;
      p += padded(a.n);
    }
    ok = hipMemset(m->params, 0, 4 * 3 * padded(m->nParams)) == hipSuccess;  // params, m1, m2
  }
  if (ok) {
    if (m->ones)
      hipLaunchKernelGGL(k_fill, (unsigned)std::min<size_t>((B + 255) / 256, 4096), 256, 0, nullptr, m->ones, 1.0f, B);
    ok = hipGetLastError() == hipSuccess && hipDeviceSynchronize() == hipSuccess;
  }
  if (!ok) {
    set_error("mlp_create: device allocation failed");
    selfamd_mlp_destroy(m);
    return kHipError;
  }
  *out = m;
  return kOk;
}

int selfamd_mlp_destroy(selfamd_mlp *m) {
  if (!m) return kOk;
  if (m->memory) (void)hipFree(m->memory);
  delete m;
  return kOk;
}

int selfamd_mlp_num_params(selfamd_mlp *m, size_t *n) {
  SELFAMD_REQUIRE(m && n, "mlp_num_params: null argument");
  *n = m->nParams;
  return kOk;
}

// packed host layout: W1[nIn][H] b1[H] W2[H][H] b2[H] W3[H][nOut] b3[nOut] (row-major W[in][out])
int selfamd_mlp_set_params(selfamd_mlp *m, const float *host) {
  SELFAMD_REQUIRE(m && host, "mlp_set_params: null argument");
  SELFAMD_HIP(hipMemcpy(m->params, host, 4 * m->nParams, hipMemcpyHostToDevice));
  SELFAMD_HIP(hipMemset(m->m1, 0, 4 * m->nParams));
  SELFAMD_HIP(hipMemset(m->m2, 0, 4 * m->nParams));
  SELFAMD_HIP(hipStreamSynchronize(nullptr));  // the models' streams do not wait for the null stream
  return kOk;
}

int selfamd_mlp_get_params(selfamd_mlp *m, float *host) {
  SELFAMD_REQUIRE(m && host, "mlp_get_params: null argument");
  SELFAMD_HIP(hipMemcpy(host, m->params, 4 * m->nParams, hipMemcpyDeviceToHost));
  return kOk;
}

int selfamd_mlp_get_grads(selfamd_mlp *m, float *host) {
  SELFAMD_REQUIRE(m && host, "mlp_get_grads: null argument");
  SELFAMD_HIP(hipMemcpy(host, m->grads, 4 * m->nParams, hipMemcpyDeviceToHost));
  return kOk;
}

int selfamd_mlp_forward(selfamd_mlp *m, const float *X, float *Y, int B, void *stream) {
  SELFAMD_REQUIRE(m && X && Y && B >= 1 && B <= m->maxB, "mlp_forward: bad arguments (B=%d, max %d)", B, m ? m->maxB : 0);
  SELFAMD_HIP(forward_impl(m, X, Y, B, reinterpret_cast<hipStream_t>(stream)));
  return kOk;
}

// Forward + backward of the mean-squared error against T; gradients stay on the device
// (selfamd_mlp_get_grads) and *loss is the FP32 loss (synchronises the stream).
int selfamd_mlp_loss_grad(selfamd_mlp *m, const float *X, const float *T, int B, float *loss, void *stream) {
  SELFAMD_REQUIRE(m && X && T && B >= 1 && B <= m->maxB, "mlp_loss_grad: bad arguments");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const size_t n = (size_t)B * m->nOut;
  int blocks;
  if (m->rows) {
    RowsArgs a = rows_args(m, X, B);
    a.T = T; a.dY = m->dY; a.lossParts = m->lossParts; a.count = (float)n;
    blocks = (B + kRowTile - 1) / kRowTile;
    SELFAMD_HIP(launch_rows<kRowsLoss>(a, st));
    SELFAMD_HIP(weight_grads_rows(m, X, m->dY, B, 0, st));
  } else {
    SELFAMD_HIP(forward_impl(m, X, m->Y, B, st));
    blocks = (int)std::min<size_t>((n + 255) / 256, 1024);
    hipLaunchKernelGGL(k_mse, blocks, 256, 0, st, m->Y, T, m->dY, m->lossParts, n);
    SELFAMD_HIP(hipGetLastError());
    SELFAMD_HIP(backward_layers(m, X, m->dY, B, 0, nullptr, st));
  }
  if (loss) {
    std::vector<float> parts(blocks);
    SELFAMD_HIP(hipMemcpyAsync(parts.data(), m->lossParts, 4 * blocks, hipMemcpyDeviceToHost, st));
    SELFAMD_HIP(hipStreamSynchronize(st));
    double s = 0.0;
    for (float p : parts) s += p;
    *loss = (float)(s / (double)n);
  }
  return kOk;
}

int selfamd_mlp_backward(selfamd_mlp *m, const float *X, const float *dY, int B, int accumulate, float *dX,
                         void *stream) {
  SELFAMD_REQUIRE(m && X && dY && B >= 1 && B <= m->maxB, "mlp_backward: bad arguments (B=%d, max %d)", B,
                  m ? m->maxB : 0);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (m->rows) {  // the kernels read dY where it is; the layers read a copy
    const size_t bytes = sizeof(float) * (size_t)B * m->nOut;
    int device = 0;
    SELFAMD_HIP(hipGetDevice(&device));
    const Source from = source_of(dY, bytes, sizeof(float), device);
    SELFAMD_REQUIRE(from != Source::kShort, "mlp_backward: dY holds less than %d rows of %d", B, m->nOut);
    if (from == Source::kCopy) {
      SELFAMD_HIP(hipMemcpyAsync(m->dY, dY, bytes, hipMemcpyDeviceToDevice, st));
      dY = m->dY;
    }
  }
  SELFAMD_HIP(backward_impl(m, X, dY, B, accumulate, dX, st));
  return kOk;
}

int selfamd_mlp_zero_grads(selfamd_mlp *m, void *stream) {
  SELFAMD_REQUIRE(m, "mlp_zero_grads: null argument");
  hipLaunchKernelGGL(k_fill, (int)std::min<size_t>((m->nParams + 255) / 256, 4096), 256, 0,
                     reinterpret_cast<hipStream_t>(stream), m->grads, 0.0f, m->nParams);
  SELFAMD_HIP(hipGetLastError());
  return kOk;
}

int selfamd_mlp_adam_step(selfamd_mlp *m, float lr, int step, void *stream) {
  SELFAMD_REQUIRE(m && step >= 1, "mlp_adam_step: bad arguments");
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, (int)std::min<size_t>((m->nParams + 255) / 256, 4096), 256, 0,
                     reinterpret_cast<hipStream_t>(stream), m->params, m->grads, m->m1, m->m2, m->nParams, lr, b1, b2,
                     1e-8f, c1, c2);
  SELFAMD_HIP(hipGetLastError());
  return kOk;
}

}  // extern "C"

// ------------------------------------------------------------------------------
// Fine -> coarse L2 projection on structured meshes
// ------------------------------------------------------------------------------
// A coarse element (degree Nc) covers r x r fine elements (degree Nf).  Sub-element a of the
// coarse xi-interval spans [-1 + 2a/r, -1 + 2(a+1)/r], so xi_c = -1 + (2a + 1 + xi_f)/r.  The
// L2 projection onto the coarse Gauss-Lagrange basis, with the coarse mass matrix diagonal
// (exact: Gauss with Nc+1 points integrates l_i l_j of degree 2 Nc), is
//   u_c(i,j) = sum_{a,b,p,q} Px[a][i][p] Px[b][j][q] u_f(p,q; a,b),
//   Px[a][i][p] = w_p^f l_i^c(xi_c(a,p)) / (r w_i^c),
// exact whenever the fine quadrature integrates l_i^c times the fine polynomial (degree
// Nc + Nf <= 2 Nf + 1), and mass-conserving: sum_ij w_i w_j u_c = r^-2 sum_ab sum_pq w_p w_q u_f.
namespace {

// One block per coarse element.  The fine rows of elements are read as the contiguous runs they
// are (r nVar Pf^2 doubles per sub-row b), `rowsB` sub-rows at a time, into LDS; then
// row[b][v][q][i] = sum_a,p Px[a][i][p] u, and u_c += sum_b,q Px[b][j][q] row.  Bound by reading
// the fine state: 104 MB (256^2 N = 7, three variables) in 24 us (4.3 TB/s: a block's loads and
// sums do not overlap, five blocks per CU do), where one work-item per coarse value, each reading
// r^2 Pf^2 doubles with its neighbours 64 bytes or whole elements away, took 276 us.  LDS rows of Pf
// doubles are padded by one: four of five rows would share banks at Pf = 8.
constexpr int kProjectArgs = 448, kProjectLds = 6144, kProjectChunk = 3072;  // doubles
constexpr size_t kProjectBlocks = size_t(1) << 24;  // of 256: a grid's work-items stay below 2^32
constexpr size_t kProjectFew = 4000, kProjectProducts = 1300;
struct ProjectArgs {
  const double *fine;
  double *coarse;
  int Pf, Pc, nxc, r, nVar, rowsB;
  unsigned invPf, invRun;      // k / Pf = (k invPf) >> 20 and k / run = high word of k invRun, k < kProjectLds
  double px[kProjectArgs];     // Px[a][i][p]
};
static_assert(sizeof(ProjectArgs) <= 4096, "kernel arguments exceed the 4 KiB kernarg segment");

// PC = Pc with the sums of one LDS row for all i in one work-item (the factors are uniform and
// come in scalar registers), where one sum per work-item reads every u Pc times; PC = 0: one sum
// per work-item, for other degrees.  PF = Pf, so that the LDS reads of a row's sum are in flight at
// once: with a loop over Pf (PF = 0, other degrees) every term waits for its own, 37 us.
template <int PC, int PF>
__global__ void __launch_bounds__(256) k_project(const ProjectArgs a) {
  extern __shared__ double projectLds[];
  const int tid = threadIdx.x, Pf = PF > 0 ? PF : a.Pf, Pc = PC > 0 ? PC : a.Pc, r = a.r, nVar = a.nVar, nPx = r * Pc * Pf, ld = Pf + 1;
  const int run = r * nVar * Pf * Pf, rows = r * nVar * Pf, nOut = nVar * Pc * Pc, perB = nVar * Pf * Pc;
  double *sPx = projectLds, *sU = sPx + nPx, *sRow = sU + a.rowsB * rows * ld, *sOut = sRow + a.rowsB * perB;
  const int I = blockIdx.x % a.nxc, J = blockIdx.x / a.nxc;
  const size_t nxf = (size_t)a.nxc * r;
  for (int k = tid; k < nPx; k += 256) sPx[k] = a.px[k];
  for (int k = tid; k < nOut; k += 256) sOut[k] = 0.0;
  for (int b0 = 0; b0 < r; b0 += a.rowsB) {
    const int nb = min(a.rowsB, r - b0);
    // the whole chunk (up to 3,072 doubles) in flight at once: with one sub-row after another a
    // block waits for memory rowsB times (43 us)
    const double *src = a.fine + (size_t)nVar * Pf * Pf * ((size_t)I * r + nxf * ((size_t)J * r + b0));
    const size_t subRow = (size_t)nVar * Pf * Pf * nxf;
    const int total = nb * run;
    for (int k0 = tid; k0 < total; k0 += kProjectChunk) {
      constexpr int M = kProjectChunk / 256;
      double v[M];
#pragma unroll
      for (int m = 0; m < M; m++) {
        const unsigned k = min(k0 + 256 * m, total - 1), b = __umulhi(k, a.invRun);
        v[m] = src[b * subRow + (k - b * run)];
      }
#pragma unroll
      for (int m = 0; m < M; m++) {
        const unsigned k = k0 + 256 * m;
        if ((int)k < total) sU[k + (k * a.invPf >> 20)] = v[m];  // one pad per row of Pf
      }
    }
    __syncthreads();
    if constexpr (PC > 0) {
      for (int t = tid; t < nb * nVar * Pf; t += 256) {
        const int vq = t % (nVar * Pf), b = t / (nVar * Pf);
        double row[PC] = {};
        for (int aa = 0; aa < r; aa++) {
          const double *u = sU + (b * rows + aa * nVar * Pf + vq) * ld, *px = a.px + aa * PC * Pf;
#pragma unroll
          for (int p = 0; p < Pf; p++) {
            const double x = u[p];
#pragma unroll
            for (int i = 0; i < PC; i++) row[i] += px[i * Pf + p] * x;
          }
        }
#pragma unroll
        for (int i = 0; i < PC; i++) sRow[t * PC + i] = row[i];
      }
    } else for (int t = tid; t < nb * perB; t += 256) {
      const int i = t % Pc, vq = t / Pc % (nVar * Pf), b = t / perB;
      double row = 0.0;
      for (int aa = 0; aa < r; aa++) {
        const double *u = sU + (b * rows + aa * nVar * Pf + vq) * ld, *px = sPx + (aa * Pc + i) * Pf;
        for (int p = 0; p < Pf; p++) row += px[p] * u[p];
      }
      sRow[t] = row;
    }
    __syncthreads();
    for (int t = tid; t < nOut; t += 256) {
      const int i = t % Pc, j = t / Pc % Pc, v = t / (Pc * Pc);
      double acc = sOut[t];
      for (int b = 0; b < nb; b++)
#pragma unroll
        for (int q = 0; q < Pf; q++) acc += sPx[((b0 + b) * Pc + j) * Pf + q] * sRow[b * perB + (v * Pf + q) * Pc + i];
      sOut[t] = acc;
    }
    __syncthreads();
  }
  for (int t = tid; t < nOut; t += 256) a.coarse[(size_t)blockIdx.x * nOut + t] = sOut[t];
}

// The same, one work-item per coarse value, for coarsening factors and degrees whose factors or
// runs are too long for the kernel arguments or LDS of k_project, for meshes beyond its grid, and for
// large meshes of small elements.
__global__ void k_project_values(const double *__restrict__ Sf, double *__restrict__ Sc, const double *__restrict__ Px,
                                 int Nf, int Nc, int nxc, int nyc, int r, int nVar) {
  const int Pf = Nf + 1, Pc = Nc + 1;
  const size_t total = (size_t)Pc * Pc * nVar * nxc * nyc;
  const int nxf = nxc * r;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const int i = t % Pc, j = (t / Pc) % Pc, v = (t / ((size_t)Pc * Pc)) % nVar;
    const size_t E = t / ((size_t)Pc * Pc * nVar);
    const int I = E % nxc, J = E / nxc;
    double acc = 0.0;
    for (int b = 0; b < r; b++)
      for (int q = 0; q < Pf; q++) {
        const double wy = Px[((size_t)b * Pc + j) * Pf + q];
        double row = 0.0;
        for (int a = 0; a < r; a++) {
          const size_t ef = (size_t)(I * r + a) + (size_t)nxf * (J * r + b);
          const double *u = Sf + ((size_t)v + (size_t)nVar * ef) * Pf * Pf + (size_t)Pf * q;
          const double *px = Px + ((size_t)a * Pc + i) * Pf;
          for (int p = 0; p < Pf; p++) row += px[p] * u[p];
        }
        acc += wy * row;
      }
    Sc[t] = acc;
  }
}

// features: X[e][k] = (S_k - mean_k) / scale_k, rounded to FP32
__global__ void k_closure_features(const double *__restrict__ S, const double *__restrict__ geom,
                                   const float *__restrict__ mu, const float *__restrict__ sd, float *__restrict__ X,
                                   int NN, int nVar, int nEl) {
  const int nIn = nVar * NN + 3;
  const size_t total = (size_t)nIn * nEl;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
    const int k = t % nIn;
    const size_t e = t / nIn;
    double raw;
    if (k < nVar * NN) {
      raw = S[e * (size_t)nVar * NN + k];
    } else {
      const double *g = geom + e * kGeomStride;
      raw = k == nVar * NN ? g[4] : (k == nVar * NN + 1 ? g[0] : g[3]);
    }
    X[t] = (float)((raw - (double)mu[k]) / (double)sd[k]);
  }
}

// correction: corr = Y * outScale + outMean (FP64), one wavefront per element; lane = node.
// elemMass[e] = J_e sum_ij w_i w_j corr_mass(i,j), reduced across the wavefront in a fixed order.
__global__ void __launch_bounds__(256) k_closure_correct(const float *__restrict__ Y, const float *__restrict__ muOut,
                                                         const float *__restrict__ sdOut, const double *__restrict__ geom,
                                                         const double *__restrict__ qW, double *__restrict__ corr,
                                                         double *__restrict__ elemMass, int N, int nVar, int massVar,
                                                         int nEl) {
  const int P = N + 1, NN = P * P;
  const int lane = threadIdx.x & 63;
  const size_t e = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= (size_t)nEl) return;  // whole wavefront leaves together
  double m = 0.0;
  if (lane < NN) {
    const int i = lane % P, j = lane / P;
    for (int v = 0; v < nVar; v++) {
      const int k = v * NN + lane;
      const double c = (double)Y[e * (size_t)nVar * NN + k] * (double)sdOut[k] + (double)muOut[k];
      corr[e * (size_t)nVar * NN + k] = c;
      if (v == massVar) m = qW[i] * qW[j] * c;
    }
  }
  for (int off = 32; off > 0; off >>= 1) m += __shfl_xor(m, off, 64);
  if (lane == 0) elemMass[e] = geom[e * kGeomStride + 4] * m;
}

// shift = (sum_e elemMass[e]) / area, summed in a fixed order by one block
__global__ void __launch_bounds__(256) k_closure_shift(const double *__restrict__ elemMass, double *__restrict__ shift,
                                                       double invArea, int nEl) {
  __shared__ double red[256];
  double s = 0.0;
  for (int e = threadIdx.x; e < nEl; e += 256) s += elemMass[e];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) shift[0] = red[0] * invArea;
}

constexpr int kShiftParts = 512;

// Gauss nodes and weights of degree N, computed once: the reference's Newton sweep runs all of
// its 500 iterations for every negative node, about 0.1 ms per degree.
struct GaussRule {
  double x[kMaxN + 1], w[kMaxN + 1];
  bool ok;
};
const GaussRule *gauss_rule(int N) {
  static GaussRule rules[kMaxN + 1];
  static std::once_flag once[kMaxN + 1];
  GaussRule &g = rules[N];
  std::call_once(once[N], [&g, N] {
    double t[kMaxN + 1], bw[kMaxN + 1], m[3][(kMaxN + 1) * (kMaxN + 1)], bM[2 * (kMaxN + 1)];
    g.ok = selfamd_lagrange_init(N, SELFAMD_GAUSS, N, SELFAMD_GAUSS, g.x, t, bw, g.w, m[0], m[1], m[2], bM) == kOk;
  });
  return g.ok ? &g : nullptr;
}

double lagrange_basis(const double *x, int n, int i, double s) {
  double l = 1.0;
  for (int k = 0; k <= n; k++)
    if (k != i) l *= (s - x[k]) / (x[i] - x[k]);
  return l;
}

}  // namespace

namespace selfamd {

hipError_t mlp_forward(selfamd_mlp *m, const float *X, float *Y, int B, hipStream_t st) {
  return forward_impl(m, X, Y, B, st);
}

MlpWeights mlp_weights(const selfamd_mlp *mlp) {
  selfamd_mlp *m = const_cast<selfamd_mlp *>(mlp);
  return {m->rows, m->nH, m->W1(), m->b1(), m->W2(), m->b2(), m->W3(), m->b3()};
}

int mlp_shape(const selfamd_mlp *m, int *nIn, int *nOut, int *maxB) {
  *nIn = m->nIn;
  *nOut = m->nOut;
  *maxB = m->maxB;
  return kOk;
}

hipError_t closure_features(const double *S, const double *geom, const float *inMean, const float *inScale, float *X,
                            int N, int nVar, int nEl, hipStream_t st) {
  const int NN = (N + 1) * (N + 1);
  const size_t total = (size_t)(nVar * NN + 3) * nEl;
  hipLaunchKernelGGL(k_closure_features, (unsigned)std::min<size_t>((total + 255) / 256, 65535), 256, 0, st, S, geom,
                     inMean, inScale, X, NN, nVar, nEl);
  return hipGetLastError();
}

hipError_t closure_evaluate(ClosureBuffers &c, const double *S, const double *geom, const double *qW, int N,
                            int nVar, int massVar, int nEl, hipStream_t st) {
  hipError_t e;
  int nMass = nEl;  // partial mass integrals: one per element, or one per row tile
  if (c.mlp->rows) {
    RowsArgs a = rows_args(c.mlp, nullptr, nEl);
    a.S = S; a.geom = geom; a.qW = qW;
    a.inMean = c.inMean; a.inScale = c.inScale; a.outMean = c.outMean; a.outScale = c.outScale;
    a.corr = c.corr; a.massParts = c.elemMass;
    a.P = N + 1; a.nVar = nVar; a.massVar = massVar;
    nMass = (nEl + kRowTile - 1) / kRowTile;
    if ((e = launch_rows<kRowsClosure>(a, st)) != hipSuccess) return e;
  } else {
    if ((e = closure_features(S, geom, c.inMean, c.inScale, c.X, N, nVar, nEl, st)) != hipSuccess) return e;
    if ((e = forward_impl(c.mlp, c.X, c.Y, nEl, st)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_closure_correct, (nEl + 3) / 4, 256, 0, st, c.Y, c.outMean, c.outScale, geom, qW, c.corr,
                       c.elemMass, N, nVar, massVar, nEl);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  // A few hundred partial integrals are added by the stage kernel itself; its wavefronts each
  // read all of them, so more are reduced to their sum here first (one block, about 4.5 us).
  c.shiftParts = c.elemMass; c.nShift = nMass; c.shiftScale = c.invArea;
  if (nMass > kShiftParts) {
    hipLaunchKernelGGL(k_closure_shift, 1, 256, 0, st, c.elemMass, c.shift, c.invArea, nMass);
    c.shiftParts = c.shift; c.nShift = 1; c.shiftScale = 1.0;
  }
  return hipGetLastError();
}

namespace {
constexpr int kVjpBlock = 256;

// per-block sums of lam over the mass variable's nodes (fixed order), then the total
__global__ void __launch_bounds__(kVjpBlock) k_vjp_mass_partial(const double *__restrict__ lam, double *__restrict__ part,
                                                               int NN, int nVar, int massVar, size_t nNodes) {
  __shared__ double red[kVjpBlock];
  const size_t n = blockIdx.x * (size_t)kVjpBlock + threadIdx.x;
  double v = 0.0;
  if (n < nNodes) {
    const size_t e = n / NN;
    v = lam[(e * nVar + massVar) * NN + n % NN];
  }
  red[threadIdx.x] = v;
  __syncthreads();
  for (int w = kVjpBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(kVjpBlock) k_vjp_sum(double *__restrict__ part, int n) {
  __shared__ double red[kVjpBlock];
  double v = 0.0;
  for (int k = threadIdx.x; k < n; k += kVjpBlock) v += part[k];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int w = kVjpBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[n] = red[0];
}

// Output cotangent.  Forward: corr_k = y_k sdOut_k + muOut_k, and for the mass variable
// corr' = corr - invArea sum_n omega_n corr_n (omega = w_i w_j J); so
// dY_k = sdOut_k (lam_k - omega_k invArea sum_n lam_n) on the mass variable, sdOut_k lam_k elsewhere.
__global__ void k_vjp_dY(const double *__restrict__ lam, const double *__restrict__ total, const float *__restrict__ sdOut,
                         const double *__restrict__ geom, const double *__restrict__ qW, float *__restrict__ dY, int N,
                         int nVar, int massVar, double invArea, size_t n) {
  const int P = N + 1, NN = P * P, nOut = nVar * NN;
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(t % nOut);
    const size_t e = t / nOut;
    double l = lam[t];
    if (k / NN == massVar) {
      const int node = k % NN;
      l -= qW[node % P] * qW[node / P] * geom[e * kGeomStride + 4] * invArea * total[0];
    }
    dY[t] = (float)(l * (double)sdOut[k]);
  }
}

// mu += dX / inScale over the nodal-state inputs (the metric inputs do not depend on the state)
__global__ void k_vjp_mu(const float *__restrict__ dX, const float *__restrict__ sdIn, double *__restrict__ mu, int nIn,
                         int nOut, size_t n) {
  for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    const int k = (int)(t % nOut);
    const size_t e = t / nOut;
    mu[t] += (double)dX[e * nIn + k] / (double)sdIn[k];
  }
}
}  // namespace

size_t closure_vjp_partials(int N, int nEl) {
  const size_t nNodes = (size_t)(N + 1) * (N + 1) * nEl;
  return (nNodes + kVjpBlock - 1) / kVjpBlock + 1;
}

hipError_t closure_vjp(const ClosureBuffers &c, const double *S, const double *geom, const double *qW,
                       const double *lam, double *mu, int N, int nVar, int massVar, int nEl, hipStream_t st) {
  hipError_t e;
  const int NN = (N + 1) * (N + 1);
  const size_t nNodes = (size_t)NN * nEl, nb = (nNodes + kVjpBlock - 1) / kVjpBlock;
  hipLaunchKernelGGL(k_vjp_mass_partial, (unsigned)nb, kVjpBlock, 0, st, lam, c.vjpPartial, NN, nVar, massVar, nNodes);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  // As for the mean correction, a few hundred partial sums are added where they are used.
  const bool sum = !c.mlp->rows || nb > (size_t)kShiftParts;
  if (sum) {
    hipLaunchKernelGGL(k_vjp_sum, 1, kVjpBlock, 0, st, c.vjpPartial, (int)nb);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (c.mlp->rows) {
    // One launch for features, output cotangent, network and state cotangent.  64 x 64 elements of
    // N = 3, 51 -> 128 -> 128 -> 48: 17.6 us where the network's launch took 15.3 and four more
    // 12 us and a launch each; the adjoint of a stage with its reads 139 -> 125 us.
    RowsArgs a = rows_args(c.mlp, nullptr, nEl);
    a.S = S; a.geom = geom; a.qW = qW; a.lam = lam; a.mu = mu;
    a.inMean = c.inMean; a.inScale = c.inScale; a.outScale = c.outScale;
    a.P = N + 1; a.nVar = nVar; a.massVar = massVar; a.invArea = c.invArea;
    a.lamParts = c.vjpPartial + (sum ? nb : 0); a.nLamParts = sum ? 1 : (int)nb;
    a.Xout = c.X; a.dY = c.dY;
    if ((e = launch_rows<kRowsClosureVjp>(a, st)) != hipSuccess) return e;
    return weight_grads_rows(c.mlp, c.X, c.dY, nEl, 1, st);
  }
  if ((e = closure_features(S, geom, c.inMean, c.inScale, c.X, N, nVar, nEl, st)) != hipSuccess) return e;
  const size_t n = (size_t)c.nOut * nEl;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65535);
  hipLaunchKernelGGL(k_vjp_dY, blocks, 256, 0, st, lam, c.vjpPartial + nb, c.outScale, geom, qW, c.dY, N, nVar, massVar,
                     c.invArea, n);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = backward_impl(c.mlp, c.X, c.dY, nEl, 1, c.dX, st)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_vjp_mu, blocks, 256, 0, st, c.dX, c.inScale, mu, c.nIn, c.nOut, n);
  return hipGetLastError();
}

}  // namespace selfamd

extern "C" {

int selfamd_project_l2_structured_2d(const double *fine, double *coarse, int Nf, int Nc, int nxc, int nyc, int r,
                                     int nVar, void *stream) {
  SELFAMD_REQUIRE(fine && coarse, "project_l2_structured_2d: null array");
  SELFAMD_REQUIRE(Nf >= 1 && Nf <= kMaxN && Nc >= 1 && Nc <= kMaxN && nxc >= 1 && nyc >= 1 && r >= 1 && nVar >= 1,
                  "project_l2_structured_2d: bad sizes (Nf=%d Nc=%d nxc=%d nyc=%d r=%d nVar=%d)", Nf, Nc, nxc, nyc, r,
                  nVar);
  SELFAMD_REQUIRE(Nc <= 2 * Nf + 1, "project_l2_structured_2d: fine quadrature too coarse for Nc=%d", Nc);
  const GaussRule *fineRule = gauss_rule(Nf), *coarseRule = gauss_rule(Nc);
  SELFAMD_REQUIRE(fineRule && coarseRule, "project_l2_structured_2d: no quadrature for Nf=%d Nc=%d", Nf, Nc);
  const double *xf = fineRule->x, *wf = fineRule->w, *xc = coarseRule->x, *wc = coarseRule->w;
  const int Pf = Nf + 1, Pc = Nc + 1;
  const size_t nPx = (size_t)r * Pc * Pf, run = (size_t)r * nVar * Pf * Pf;
  auto entry = [&](int a, int i, int p) {
    const double xi = -1.0 + (2.0 * a + 1.0 + xf[p]) / r;
    return wf[p] * lagrange_basis(xc, Nc, i, xi) / (r * wc[i]);
  };
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const size_t elements = (size_t)nxc * nyc;
  // A block per coarse element takes 1.45 ns from some thousand elements on, whatever is in it, and a
  // product of a coarse value and a fine one 1.1e-3 ns by the value-by-value kernel, half of that at
  // Pf = 2.  By values and by blocks: 547^2 elements, r = 2, Pf = Pc = 3, one variable (324 products
  // each) 116 and 417 us; 252^2, r = 2, Pf = Pc = 4, three variables (3,072) 197 and 125 us.
  const size_t products = (size_t)Pc * Pc * nVar * r * r * Pf * Pf;
  const size_t cheap = Pf == 2 ? 2 : 1;
  const bool blocksPay = elements <= kProjectFew / cheap || products >= kProjectProducts * cheap;
  if (nPx <= (size_t)kProjectArgs && run <= (size_t)kProjectLds && elements < kProjectBlocks && blocksPay) {
    ProjectArgs g;
    g.fine = fine; g.coarse = coarse; g.Pf = Pf; g.Pc = Pc; g.nxc = nxc; g.r = r; g.nVar = nVar;
    g.rowsB = std::max(1, std::min(r, kProjectChunk / (int)run));
    g.invPf = ((1u << 20) + Pf - 1) / Pf;
    g.invRun = (unsigned)(((1ull << 32) + run - 1) / run);
    for (int a = 0; a < r; a++)
      for (int i = 0; i < Pc; i++)
        for (int p = 0; p < Pf; p++) g.px[(a * Pc + i) * Pf + p] = entry(a, i, p);
    const size_t lds = nPx + (size_t)g.rowsB * r * nVar * Pf * (Pf + 1) + (size_t)g.rowsB * nVar * Pf * Pc + (size_t)nVar * Pc * Pc;
    if (sizeof(double) * lds <= 64 * 1024) {
      auto run_as = [&](auto kernel) { hipLaunchKernelGGL(kernel, (unsigned)elements, 256, sizeof(double) * lds, st, g); };
#define CASE_F(PC, PF) case PF: run_as(k_project<PC, PF>); break;
#define CASE(PC)                                                                                        \
  case PC:                                                                                              \
    switch (Pf) {                                                                                       \
      CASE_F(PC, 3) CASE_F(PC, 4) CASE_F(PC, 5) CASE_F(PC, 6) CASE_F(PC, 7) CASE_F(PC, 8)               \
      default: run_as(k_project<PC, 0>);                                                                \
    }                                                                                                   \
    break;
      switch (Pc) {
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6)
        default: run_as(k_project<0, 0>);
      }
#undef CASE
#undef CASE_F
      SELFAMD_HIP(hipGetLastError());
      SELFAMD_HIP(hipStreamSynchronize(st));
      return kOk;
    }
  }
  std::vector<double> px(nPx);
  for (int a = 0; a < r; a++)
    for (int i = 0; i < Pc; i++)
      for (int p = 0; p < Pf; p++) px[((size_t)a * Pc + i) * Pf + p] = entry(a, i, p);
  double *dPx = nullptr;
  SELFAMD_HIP(hipMalloc(&dPx, sizeof(double) * px.size()));
  hipError_t e = hipMemcpyAsync(dPx, px.data(), sizeof(double) * px.size(), hipMemcpyHostToDevice, st);
  const size_t total = (size_t)Pc * Pc * nVar * nxc * nyc;
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_project_values, (unsigned)std::min<size_t>((total + 255) / 256, 65535), 256, 0, st, fine, coarse,
                       dPx, Nf, Nc, nxc, nyc, r, nVar);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(dPx);
  SELFAMD_HIP(e);
  return kOk;
}

}  // extern "C"
