// Device functions that the kernels evaluating the closure's network share (closure.hip, the
// resident launch of dg2d_fused.hip): the activation, and 16 rows times a layer's weights on the
// FP32 matrix cores.
#pragma once
#include "selfamd_common.hpp"

namespace selfamd {

// h = gelu(z) = z Phi(z) and d = gelu'(z) = Phi(z) + z phi(z), without branches (a call of erff
// runs both of its branches over a wavefront).  With x = z / sqrt 2: Phi = (1 + erf x) / 2 below
// |x| = 1, erf x = x + x Q(x^2); beyond, from erfc |x| = exp(-x^2) t P(t), t = 1 / (1 + 0.4 |x|)
// (the form of Hastings, Approximations for Digital Computers, 1955), with the exponential that
// phi needs too.  Q and P (degree 6) are least-squares fits, weighted towards the smallest
// maximum: relative errors 1.6e-9 of erf and 2.4e-8 of erfc.  In FP32 against 64 bits over
// |z| <= 8: h within 9.8e-8 (|z| + 0.1), rms 3.5e-8 for normal z; d within 1.4e-7, rms 2.6e-8 (the
// formulas with a correctly rounded erff: 9.9e-8, 3.7e-8, 1.3e-7, 2.6e-8).
__device__ __forceinline__ void gelu_pair(float z, float &h, float &d) {
#pragma clang fp contract(on)  // the same rounding in every kernel
  const float x = z * 0.70710678118654752f, x2 = x * x, ax = fabsf(x);
  float q = 7.72090352e-05f;
  q = fmaf(q, x2, -0.000797249028f);
  q = fmaf(q, x2, 0.00518434215f);
  q = fmaf(q, x2, -0.0268518832f);
  q = fmaf(q, x2, 0.11283543f);
  q = fmaf(q, x2, -0.37612623f);
  q = fmaf(q, x2, 0.128379166f);
  const float lo = fmaf(0.5f, fmaf(x, q, x), 0.5f);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.4f, ax, 1.f));
  float p = -0.117370792f;
  p = fmaf(p, t, 0.246633857f);
  p = fmaf(p, t, 0.00491613708f);
  p = fmaf(p, t, 0.214964211f);
  p = fmaf(p, t, 0.198186055f);
  p = fmaf(p, t, 0.226788446f);
  p = fmaf(p, t, 0.225620806f);
  const float e = expf(-0.5f * z * z), half = 0.5f * (p * t) * e;
  const float phi = ax < 1.f ? lo : (z >= 0.f ? 1.f - half : half);
  h = z * phi;
  d = fmaf(z * e, 0.39894228040143268f, phi);
}
__device__ __forceinline__ float gelu_f(float z) {
  float h, d;
  gelu_pair(z, h, d);
  return h;
}
__device__ __forceinline__ float gelu_grad_f(float z) {
  float h, d;
  gelu_pair(z, h, d);
  return d;
}

constexpr int kRowTile = 16, kRowThreads = 512, kRowWaves = kRowThreads / 64;
using f32x4 = __attribute__((ext_vector_type(4))) float;

// Columns of an operand in LDS: a multiple of 64 (zero beyond the data), rows an odd multiple of
// 4 floats apart, so that the 16 rows of a 16-byte read do not conflict in the banks.
inline __host__ __device__ constexpr int pad16(int n) { return (n + 15) & ~15; }
inline __host__ __device__ constexpr int pad64(int n) { return (n + 63) & ~63; }
inline __host__ __device__ constexpr int rows_ld(int n) { return pad64(n) + 4; }

// element `at` of a uniform base (scalar base, 32-bit vector offset: operands are below 4 GiB)
template <class T>
__device__ __forceinline__ T load_at(const float *base, unsigned at) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + 4u * at);
}
// The weight operand of one layer: weight (k, n), k < K, n < Nc, at W[k ldw + n], or with TRANS at
// W[n ldw + k].  VEC: 16-byte reads along k (K a multiple of 4, rows 16-byte aligned).
struct RowsOperand {
  const float *W;
  int ldw, K, Nc;
};
// 64 reduction indices of this lane's column n, as the matrix instruction takes them: in
// instruction 4 t + q, index k0 + 16 t + 4 g + q (lane group g = lane / 16).  The row operand is
// read with the same index order, so both come in pieces of four consecutive indices.  Indices
// past K and columns past Nc read a weight in range instead, without a select that would wait
// for the load: past K the rows are zero in LDS, past Nc the column is discarded.
template <bool TRANS, bool VEC>
__device__ __forceinline__ void rows_load(const RowsOperand &o, int n, int g, int k0, float (&b)[16]) {
  const unsigned nn = min(n, o.Nc - 1), k = k0 + 4 * g;
  // 32-bit element offsets from the uniform base: one addition and one minimum per load
  const unsigned at = TRANS ? nn * o.ldw + k : k * o.ldw + nn, step = TRANS ? 1 : o.ldw;
  const unsigned last = TRANS ? nn * o.ldw + o.K - 1 : (o.K - 1) * o.ldw + nn;
  if constexpr (TRANS && VEC) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const f32x4 v = load_at<f32x4>(o.W, min(at + 16 * t, last - 3));
#pragma unroll
      for (int q = 0; q < 4; q++) b[4 * t + q] = v[q];
    }
  } else {
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) b[4 * t + q] = load_at<float>(o.W, min(at + (16 * t + q) * step, last));
  }
}
__device__ __forceinline__ f32x4 rows_mul(const float *rows, const float (&b)[16], f32x4 acc) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const f32x4 a = *reinterpret_cast<const f32x4 *>(rows + 16 * t);
#pragma unroll
    for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[4 * t + q], acc, 0, 0, 0);
  }
  return acc;
}
}  // namespace selfamd
