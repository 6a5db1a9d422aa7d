// Row kernels of the chunked readout + cross-entropy loss.
//
// Reference: src/dabsn/runtime/loss.py:52-137 (ChunkedLinearCrossEntropy): per chunk of rows
// the readout GEMM gives logits [rows, V] in the hidden dtype; the loss upcasts them to fp32
// and forms logsumexp, the target logit and the masked NLL (forward), or
// (softmax - onehot(target)) * valid * scale (backward). The GEMMs stay on hipBLASLt; these
// kernels do each row's upcast, reductions and gradient in one pass over the logits (one
// workgroup per row; the forward keeps a running max and exp-sum per thread), instead of
// an fp32 copy plus logsumexp, gather, softmax and scatter kernels. Targets outside
// [0, V) other than ignore_index raise the error word and count as ignored.
#include <algorithm>

#include "../../include/dabsn_hip.h"
#include "capi.hpp"
#include "common.hpp"

namespace dabsn {
namespace loss {

constexpr int NTH = 256;
constexpr uint32_t kErrTarget = 1u;

__device__ __forceinline__ float block_reduce(float v, float* sh, bool is_max) {
  v = is_max ? wave_max(v) : wave_sum(v);
  __syncthreads();  // sh is reused by consecutive reductions
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = sh[0];
#pragma unroll
  for (int w = 1; w < NTH / 64; ++w) r = is_max ? fmaxf(r, sh[w]) : r + sh[w];
  return r;
}

// Fold one value (or the max of a vector with its exp-sum relative to that max) into a
// running (max, sum of exp(x - max)).
__device__ __forceinline__ void fold(float& m, float& s, float vm, float vs) {
  const float nm = fmaxf(m, vm);
  s = (m == -INFINITY ? 0.0f : s * __expf(m - nm)) + (vm == -INFINITY ? 0.0f : vs * __expf(vm - nm));
  m = nm;
}

// Row max m and sum of exp(x - m) in fp32 in one pass: each thread keeps a running
// (max, sum), rescaled once per VEC-element vector; the block combines the pairs.
template <typename E, int VEC>
__device__ __forceinline__ void row_stats(const E* x, int V, float* sh, float& m, float& s) {
  const int nv = V / VEC;
  m = -INFINITY;
  s = 0.0f;
  for (int c = threadIdx.x; c < nv; c += NTH) {
    float v[VEC];
    ldv<E, VEC>(x + static_cast<size_t>(c) * VEC, v);
    float vm = v[0];
#pragma unroll
    for (int e = 1; e < VEC; ++e) vm = fmaxf(vm, v[e]);
    float vs = 0.0f;
#pragma unroll
    for (int e = 0; e < VEC; ++e) vs += __expf(v[e] - vm);
    fold(m, s, vm, vs);
  }
  for (int c = nv * VEC + threadIdx.x; c < V; c += NTH) fold(m, s, ld(x, c), 1.0f);
  // Block combine: the block max, then every thread's sum rescaled to it.
  const float M = block_reduce(m, sh, true);
  s = block_reduce(m == -INFINITY ? 0.0f : s * __expf(m - M), sh, false);
  m = M;
}

__device__ __forceinline__ bool target_ok(int64_t t, int V, int64_t ignore, uint32_t* err) {
  if (t == ignore) return false;
  if (t < 0 || t >= V) {
    if (threadIdx.x == 0) atomicOr(err, kErrTarget);
    return false;
  }
  return true;
}

template <typename E, int VEC>
__global__ void __launch_bounds__(NTH) ce_fwd_kernel(int V, int64_t ldl, const E* __restrict__ logits,
                                                     const int64_t* __restrict__ targets,
                                                     int64_t ignore, float* __restrict__ lse,
                                                     float* __restrict__ nll, uint32_t* err) {
  __shared__ float sh[NTH / 64];
  const int row = blockIdx.x;
  const E* x = logits + static_cast<size_t>(row) * ldl;
  float m, s;
  row_stats<E, VEC>(x, V, sh, m, s);
  if (threadIdx.x != 0) return;
  const float l = m + logf(s);
  lse[row] = l;
  const int64_t t = targets[row];
  nll[row] = target_ok(t, V, ignore, err) ? l - ld(x, static_cast<size_t>(t)) : 0.0f;
}

// d[row, c] = (exp(x - lse) - [c == target]) * valid * scale[0], fp32, row stride V.
template <typename E, int VEC>
__global__ void __launch_bounds__(NTH) ce_bwd_kernel(int V, int64_t ldl, const E* __restrict__ logits,
                                                     const int64_t* __restrict__ targets,
                                                     int64_t ignore, const float* __restrict__ lse,
                                                     const float* __restrict__ scale,
                                                     float* __restrict__ d, uint32_t* err) {
  const int row = blockIdx.x;
  const E* x = logits + static_cast<size_t>(row) * ldl;
  float* o = d + static_cast<size_t>(row) * V;
  const int64_t t = targets[row];
  const bool valid = target_ok(t, V, ignore, err);
  const float sc = valid ? scale[0] : 0.0f;
  const float l = lse[row];
  const int nv = V / VEC;
  for (int c = threadIdx.x; c < nv; c += NTH) {
    float v[VEC];
    ldv<E, VEC>(x + static_cast<size_t>(c) * VEC, v);
    float r[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const int col = c * VEC + e;
      r[e] = (__expf(v[e] - l) - (col == t ? 1.0f : 0.0f)) * sc;
    }
    if constexpr (VEC % 4 == 0) {
#pragma unroll
      for (int e = 0; e < VEC; e += 4)
        *reinterpret_cast<f32x4*>(o + c * VEC + e) = (f32x4){r[e], r[e + 1], r[e + 2], r[e + 3]};
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[c * VEC + e] = r[e];
    }
  }
  for (int c = nv * VEC + threadIdx.x; c < V; c += NTH)
    o[c] = (__expf(ld(x, c) - l) - (c == t ? 1.0f : 0.0f)) * sc;
}

// The bf16 readout's gradient rows as three bf16 planes d = d0 + d1 + d2, each the value's
// next 8 significant bits (truncated, so every remainder is exact and the three hold all 24
// bits of a gradient of at least 2^-110; of a smaller one what lies below bf16's smallest
// subnormal, 2^-133, is cut). The readout's weight and hidden rows are bf16 values, so the
// gradient products run as bf16 matrix products of the planes with fp32 accumulation: the
// products of the fp32 matrix product, exact, at 16 times its rate: 8,192 rows of 2,048 against
// 32,000 words, forward and backward, 34.6 -> 10.6 ms, and the products' error against 64 bits
// before their rounding to bf16 falls (1.7e-6 -> 7e-7 for the hidden rows). Non-finite values keep
// their kind in the first plane, the others are zero.
__device__ __forceinline__ void split3(float v, bf16 (&o)[3]) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  if ((u & 0x7f800000u) == 0x7f800000u) {
    o[0] = (u & 0x007fffffu) ? static_cast<bf16>(0x7fc0) : static_cast<bf16>(u >> 16);
    o[1] = o[2] = 0;
    return;
  }
  o[0] = static_cast<bf16>(u >> 16);
  const float r1 = v - __builtin_bit_cast(float, u & 0xffff0000u);
  const uint32_t u1 = __builtin_bit_cast(uint32_t, r1);
  o[1] = static_cast<bf16>(u1 >> 16);
  const float r2 = r1 - __builtin_bit_cast(float, u1 & 0xffff0000u);
  o[2] = static_cast<bf16>(__builtin_bit_cast(uint32_t, r2) >> 16);
}

// Bound by memory: 2 bytes read and 6 written per element (31 us for 524 rows of 32,000, the
// average of a kernel trace: 4.3 TB/s; the fp32 gradient took 21.8 us plus 41 us for its
// column sums). A block owns kSplitRows rows of a strip of columns: a row's target, logsumexp
// and validity are uniform, and each thread carries its columns' sums over the rows (the
// bias gradient's partials, one row of `part` per block row), which the fp32 gradient took
// another pass over memory for.
constexpr int kSplitRows = 16;
template <int VEC>
__global__ void __launch_bounds__(NTH) ce_split_kernel(
    int rows, int V, int64_t ldl, const bf16* __restrict__ logits,
    const int64_t* __restrict__ targets, int64_t ignore, const float* __restrict__ lse,
    const float* __restrict__ scale, bf16* __restrict__ planes, int64_t plane, int64_t ldp,
    float* __restrict__ part, uint32_t* err) {
  const int strips = (V + NTH * VEC - 1) / (NTH * VEC);
  const int strip = blockIdx.x % strips, blk = blockIdx.x / strips;
  const int64_t c0l = (static_cast<int64_t>(strip) * NTH + threadIdx.x) * VEC;
  const bool live = c0l < V;  // VEC > 1 only where V is a multiple of it
  const int c0 = live ? static_cast<int>(c0l) : 0;
  const int r0 = blk * kSplitRows, r1 = min(rows, r0 + kSplitRows);
  const float sc = scale[0];
  float sum[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) sum[e] = 0.0f;
#pragma unroll 4
  for (int r = r0; r < r1; ++r) {
    const int64_t t = targets[r];
    const bool in = t >= 0 && t < V;
    if (t != ignore && !in && strip == 0 && threadIdx.x == 0) atomicOr(err, kErrTarget);
    const float s = (t != ignore && in) ? sc : 0.0f;
    const float l = lse[r];
    if (!live) continue;
    float v[VEC];
    ldv<bf16, VEC>(logits + static_cast<size_t>(r) * ldl + c0, v);
    bf16 o[3][VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float d = (__expf(v[e] - l) - (c0 + e == t ? 1.0f : 0.0f)) * s;
      sum[e] += d;
      bf16 q[3];
      split3(d, q);
      o[0][e] = q[0];
      o[1][e] = q[1];
      o[2][e] = q[2];
    }
    bf16* dst = planes + static_cast<size_t>(r) * ldp + c0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if constexpr (VEC == 8) {
        *reinterpret_cast<u32x4*>(dst + k * plane) = *reinterpret_cast<const u32x4*>(o[k]);
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) dst[k * plane + e] = o[k][e];
      }
    }
  }
  if (part && live) {
    float* q = part + static_cast<size_t>(blk) * V + c0;
#pragma unroll
    for (int e = 0; e < VEC; ++e) q[e] = sum[e];
  }
}

// out[i] = bf16(p0[i] + p1[i] + p2[i]) (the planes' products, smallest first), n elements each.
__global__ void __launch_bounds__(NTH) ce_join_kernel(int64_t n, const float* __restrict__ p,
                                                      bf16* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * NTH + threadIdx.x;
  if (i < n) out[i] = f2bf((p[i + 2 * n] + p[i + n]) + p[i]);
}

// gbias[c] = (add ? gbias[c] : 0) + the sum of column c of part [nparts][V], rows in order.
__global__ void __launch_bounds__(NTH) ce_bias_kernel(int nparts, int V,
                                                      const float* __restrict__ part, int add,
                                                      float* __restrict__ gbias) {
  const int c = blockIdx.x * NTH + threadIdx.x;
  if (c >= V) return;
  float s = add ? gbias[c] : 0.0f;
#pragma unroll 8
  for (int r = 0; r < nparts; ++r) s += part[static_cast<size_t>(r) * V + c];
  gbias[c] = s;
}

static int checks(int dtype, int64_t rows, int64_t V, int64_t ldl) {
  DABSN_REQUIRE(dtype == kF32 || dtype == kBF16, "cross entropy: bad dtype %d", dtype);
  DABSN_REQUIRE(rows >= 0 && rows < (1ll << 31) && V > 0 && V < (1ll << 31) && ldl >= V,
                "cross entropy: bad shape (rows=%lld, V=%lld, ld=%lld)", (long long)rows,
                (long long)V, (long long)ldl);
  return DABSN_OK;
}

// 8-element vector loads need every row to start 16-byte aligned (bf16: ld a multiple of
// 8; fp32: of 4, the 8-vector being two 16-byte loads); the rest of a row is read singly.
static bool vec_rows(const void* p, int64_t ldl, size_t esize) {
  return (reinterpret_cast<uintptr_t>(p) % 16 == 0) && ((ldl * esize) % 16 == 0);
}

}  // namespace loss
}  // namespace dabsn

using namespace dabsn;
using namespace dabsn::loss;

extern "C" {

int dabsn_hip_ce_fwd(int dtype, int64_t rows, int64_t V, const void* logits, int64_t ldl,
                     const int64_t* targets, int64_t ignore_index, float* lse, float* nll,
                     uint32_t* err, hipStream_t stream) {
  int rc = checks(dtype, rows, V, ldl);
  if (rc != DABSN_OK) return rc;
  if (rows == 0) return DABSN_OK;
  DABSN_REQUIRE(logits && targets && lse && nll && err, "cross entropy: null pointer");
  const size_t es = dtype == kBF16 ? 2 : 4;
  const bool vec = vec_rows(logits, ldl, es);
  const dim3 grid(static_cast<unsigned>(rows));
#define DABSN_LAUNCH(E, VEC)                                                               \
  hipLaunchKernelGGL((ce_fwd_kernel<E, VEC>), grid, dim3(NTH), 0, stream, (int)V, ldl,      \
                     static_cast<const E*>(logits), targets, ignore_index, lse, nll, err)
  if (dtype == kBF16) {
    if (vec) DABSN_LAUNCH(bf16, 8); else DABSN_LAUNCH(bf16, 1);
  } else {
    if (vec) DABSN_LAUNCH(float, 8); else DABSN_LAUNCH(float, 1);
  }
#undef DABSN_LAUNCH
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

int dabsn_hip_ce_bwd(int dtype, int64_t rows, int64_t V, const void* logits, int64_t ldl,
                     const int64_t* targets, int64_t ignore_index, const float* lse,
                     const float* scale, float* dlogits, uint32_t* err, hipStream_t stream) {
  int rc = checks(dtype, rows, V, ldl);
  if (rc != DABSN_OK) return rc;
  if (rows == 0) return DABSN_OK;
  DABSN_REQUIRE(logits && targets && lse && scale && dlogits && err,
                "cross entropy backward: null pointer");
  const size_t es = dtype == kBF16 ? 2 : 4;
  // The 8-wide path also stores 16-byte fp32 vectors into rows of V floats.
  const bool vec = vec_rows(logits, ldl, es) && V % 8 == 0 &&
                   reinterpret_cast<uintptr_t>(dlogits) % 16 == 0;
  const dim3 grid(static_cast<unsigned>(rows));
#define DABSN_LAUNCH(E, VEC)                                                               \
  hipLaunchKernelGGL((ce_bwd_kernel<E, VEC>), grid, dim3(NTH), 0, stream, (int)V, ldl,      \
                     static_cast<const E*>(logits), targets, ignore_index, lse, scale, dlogits, \
                     err)
  if (dtype == kBF16) {
    if (vec) DABSN_LAUNCH(bf16, 8); else DABSN_LAUNCH(bf16, 1);
  } else {
    if (vec) DABSN_LAUNCH(float, 8); else DABSN_LAUNCH(float, 1);
  }
#undef DABSN_LAUNCH
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

int64_t dabsn_hip_ce_split_parts(int64_t rows) { return (rows + kSplitRows - 1) / kSplitRows; }

int dabsn_hip_ce_split(int64_t rows, int64_t V, const void* logits, int64_t ldl,
                       const int64_t* targets, int64_t ignore_index, const float* lse,
                       const float* scale, void* planes, int64_t plane, int64_t ldp, float* part,
                       uint32_t* err, hipStream_t stream) {
  int rc = checks(kBF16, rows, V, ldl);
  if (rc != DABSN_OK) return rc;
  if (rows == 0) return DABSN_OK;
  DABSN_REQUIRE(logits && targets && lse && scale && planes && err,
                "cross entropy split: null pointer");
  DABSN_REQUIRE(ldp >= V && plane >= rows * ldp, "cross entropy split: bad plane (ld=%lld of %lld)",
                (long long)ldp, (long long)plane);
  const bool vec = vec_rows(logits, ldl, 2) && vec_rows(planes, ldp, 2) && V % 8 == 0 &&
                   plane % 8 == 0;
  const int cols = NTH * (vec ? 8 : 1);
  const int64_t blocks = (V + cols - 1) / cols * dabsn_hip_ce_split_parts(rows);
  DABSN_REQUIRE(blocks < (1ll << 31), "cross entropy split: %lld x %lld logits in one call",
                (long long)rows, (long long)V);
  const dim3 grid(static_cast<unsigned>(blocks));
#define DABSN_LAUNCH(VEC)                                                                    \
  hipLaunchKernelGGL((ce_split_kernel<VEC>), grid, dim3(NTH), 0, stream, (int)rows, (int)V, ldl, \
                     static_cast<const bf16*>(logits), targets, ignore_index, lse, scale,      \
                     static_cast<bf16*>(planes), plane, ldp, part, err)
  if (vec) DABSN_LAUNCH(8); else DABSN_LAUNCH(1);
#undef DABSN_LAUNCH
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

int dabsn_hip_ce_join(int64_t n, const float* planes, void* out, hipStream_t stream) {
  DABSN_REQUIRE(n >= 0 && n < (1ll << 38) && (n == 0 || (planes && out)),
                "cross entropy join: bad arguments");
  if (n == 0) return DABSN_OK;
  hipLaunchKernelGGL(ce_join_kernel, dim3(static_cast<unsigned>((n + NTH - 1) / NTH)), dim3(NTH), 0,
                     stream, n, planes, static_cast<bf16*>(out));
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

int dabsn_hip_ce_bias(int64_t nparts, int64_t V, const float* part, int add, float* gbias,
                      hipStream_t stream) {
  DABSN_REQUIRE(nparts >= 0 && nparts < (1ll << 31) && V > 0 && V < (1ll << 31) && gbias &&
                    (part || nparts == 0),
                "cross entropy bias: bad arguments");
  hipLaunchKernelGGL(ce_bias_kernel, dim3(static_cast<unsigned>((V + NTH - 1) / NTH)), dim3(NTH), 0,
                     stream, (int)nparts, (int)V, part, add, gbias);
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

}  // extern "C"
