// Permanent associative delta scan (dabsn::permanent_delta_scan).
//
// Reference: src/dabsn/kernels/permanent.py:39-51 (definition), 70-119 (analytic reverse),
// CPU kernels cpu_runtime.cpp:1075-1188. Per batch row b a fast-weight state
// S [H_v, H_k] starts at zero and, for t = 0 .. T-1,
//   r_t = S k_t                      (output)
//   S  += beta_t (v_t - r_t) k_t^T   (rank-1 delta update)
// Up to H = 512 the scan runs in chunks of 16 steps as matrix products (namespace chunked
// below); wider states walk step by step, and so does the entry without a workspace:
// each value row of S evolves on its own given k_t and beta_t, so the forward gives one
// wave to one (b, row): its 64 lanes hold the row's H columns (H / 64 each, in registers),
// r_t[row] is a wave reduction, the update is elementwise. fp32 state and arithmetic.
//
// Backward (adjoint A = dL/dS_{t+1}, per row a): walking t = T-1 .. 0,
//   Ak = a . k_t,  e = v_t[row] - r_t[row]
//   dv_t[row] = beta_t Ak,  dbeta_t += Ak e  (sum over rows)
//   dk_t += g_t[row] s_t + beta_t e a - beta_t Ak s_t  (sum over rows, s_t = state before t)
//   a = a + g_t[row] k_t - beta_t Ak k_t
// Workgroups of R waves own R rows; each first recomputes its rows' states, keeping r_t and
// every kCkpt-th state s_t (plus the final s_T), then runs the adjoint. The adjoint rebuilds
// s_t from s_{t+1} by undoing the row's update, s_t = s_{t+1} - beta_t (v_t - r_t) k_t, with
// the same e_t the forward used (r_t is taped), and restarts from a kept state at every
// checkpoint, so rounding drift spans at most kCkpt - 1 steps. The reference's reverse
// pass keeps every s_t instead (B H T H floats). The sums over rows are deterministic: the
// R rows of a workgroup are summed through LDS into a per-block partial, and reduce
// kernels add the blocks (dk) and rows (dbeta) in index order.
#include <algorithm>

#include "../../include/dabsn_hip.h"
#include "capi.hpp"
#include "common.hpp"

namespace dabsn {
namespace permanent {

constexpr int kRowsPerBlock = 8;  // backward: waves (value rows) per workgroup
constexpr int kFwdRows = 4;       // forward: waves per workgroup
constexpr int kCkpt = 8;          // backward: steps between kept states

// Kept states of the backward: s_t at index t / kCkpt for t % kCkpt == 0, t < T, and the
// final state s_T at index ceil(T / kCkpt).
__host__ __device__ inline int64_t ckpt_slots(int64_t T) { return (T + kCkpt - 1) / kCkpt + 1; }

// Lane's columns c = lane + 64 j, j < CPL; columns past H read and hold zero.
template <int CPL>
__device__ __forceinline__ void load_cols(const float* row, int lane, int H, float (&x)[CPL]) {
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const int c = lane + 64 * j;
    x[j] = c < H ? row[c] : 0.0f;
  }
}

template <int CPL>
__device__ __forceinline__ float dot_cols(const float (&a)[CPL], const float (&b)[CPL]) {
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < CPL; ++j) s = fmaf(a[j], b[j], s);
  return wave_sum(s);
}

template <int CPL>
__global__ void __launch_bounds__(kFwdRows * 64) perm_fwd_kernel(int T, int H,
                                                                 const float* __restrict__ k,
                                                                 const float* __restrict__ v,
                                                                 const float* __restrict__ beta,
                                                                 float* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kFwdRows + (threadIdx.x >> 6);
  const int b = blockIdx.y;
  if (row >= H) return;  // whole waves; no barriers below
  float s[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) s[j] = 0.0f;
  const size_t base = static_cast<size_t>(b) * T * H;
  float kn[CPL];
  if (T > 0) load_cols<CPL>(k + base, lane, H, kn);
  for (int t = 0; t < T; ++t) {
    float kt[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) kt[j] = kn[j];
    if (t + 1 < T) load_cols<CPL>(k + base + static_cast<size_t>(t + 1) * H, lane, H, kn);
    const size_t o = base + static_cast<size_t>(t) * H + row;
    const float r = dot_cols<CPL>(s, kt);
    if (lane == 0) out[o] = r;
    const float e = beta[static_cast<size_t>(b) * T + t] * (v[o] - r);
#pragma unroll
    for (int j = 0; j < CPL; ++j) s[j] = fmaf(e, kt[j], s[j]);
  }
}

// Workspace of the backward: kept states [B][H][ckpt_slots(T)][H], r tape [B][T][H], per-block dk
// partials [B][T][nrb][H], per-row dbeta partials [B][T][H] (fp32, 256-byte aligned).
struct BwdLayout {
  size_t tape, rtape, pdk, pbeta, end;
};

static size_t align_up(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

static BwdLayout bwd_layout(int64_t B, int64_t T, int64_t H) {
  const size_t nrb = static_cast<size_t>((H + kRowsPerBlock - 1) / kRowsPerBlock);
  BwdLayout l{};
  size_t o = 0;
  l.tape = o; o = align_up(o + static_cast<size_t>(B) * H * ckpt_slots(T) * H * 4);
  l.rtape = o; o = align_up(o + static_cast<size_t>(B) * T * H * 4);
  l.pdk = o; o = align_up(o + static_cast<size_t>(B) * T * nrb * H * 4);
  l.pbeta = o; o = align_up(o + static_cast<size_t>(B) * T * H * 4);
  l.end = o;
  return l;
}

template <int CPL>
__global__ void __launch_bounds__(kRowsPerBlock * 64) perm_bwd_kernel(
    int T, int H, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ beta, const float* __restrict__ g, float* __restrict__ dv,
    float* __restrict__ tape, float* __restrict__ rtape, float* __restrict__ pdk,
    float* __restrict__ pbeta) {
  extern __shared__ float red[];  // [kRowsPerBlock][H]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rb = blockIdx.x, b = blockIdx.y;
  const int nrb = gridDim.x;
  const int row = rb * kRowsPerBlock + w;
  const bool live = row < H;  // waves past H take part in the barriers with zeros
  const size_t base = static_cast<size_t>(b) * T * H;
  const int64_t nck = ckpt_slots(T);
  float* my_tape = tape + (static_cast<size_t>(b) * H + (live ? row : 0)) * nck * H;

  // Forward recompute: r_t of this row, and the kept states.
  float s[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) s[j] = 0.0f;
  for (int t = 0; t < T; ++t) {
    float kt[CPL];
    load_cols<CPL>(k + base + static_cast<size_t>(t) * H, lane, H, kt);
    if (live && t % kCkpt == 0) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const int c = lane + 64 * j;
        if (c < H) my_tape[static_cast<size_t>(t / kCkpt) * H + c] = s[j];
      }
    }
    const size_t o = base + static_cast<size_t>(t) * H + (live ? row : 0);
    const float r = dot_cols<CPL>(s, kt);
    if (live && lane == 0) rtape[o] = r;
    const float e = live ? beta[static_cast<size_t>(b) * T + t] * (v[o] - r) : 0.0f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) s[j] = fmaf(e, kt[j], s[j]);
  }
  if (live) {
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int c = lane + 64 * j;
      if (c < H) my_tape[static_cast<size_t>(nck - 1) * H + c] = s[j];
    }
  }

  // Adjoint. s_t is the kept state at checkpoint steps (exact, s_0 = 0 among them), else
  // rebuilt from sn = s_{t+1}: the kept final state at t = T - 1, otherwise the previous
  // iteration's s_t.
  float a[CPL], sn[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    a[j] = 0.0f;
    sn[j] = 0.0f;
  }
  if (live && T % kCkpt != 1) load_cols<CPL>(my_tape + static_cast<size_t>(nck - 1) * H, lane, H, sn);
  for (int t = T - 1; t >= 0; --t) {
    float kt[CPL], st[CPL];
    load_cols<CPL>(k + base + static_cast<size_t>(t) * H, lane, H, kt);
    const size_t o = base + static_cast<size_t>(t) * H + (live ? row : 0);
    const float bt = beta[static_cast<size_t>(b) * T + t];
    const float gr = live ? g[o] : 0.0f;
    const float e = live ? v[o] - rtape[o] : 0.0f;
    if (t % kCkpt == 0) {
      if (live) {
        load_cols<CPL>(my_tape + static_cast<size_t>(t / kCkpt) * H, lane, H, st);
      } else {
#pragma unroll
        for (int j = 0; j < CPL; ++j) st[j] = 0.0f;
      }
    } else {
      const float eb = bt * e;  // the forward's beta_t (v_t - r_t), bit for bit
#pragma unroll
      for (int j = 0; j < CPL; ++j) st[j] = fmaf(-eb, kt[j], sn[j]);
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) sn[j] = st[j];
    const float ak = dot_cols<CPL>(a, kt);
    if (live && lane == 0) {
      dv[o] = bt * ak;
      pbeta[o] = ak * e;
    }
    // This row's share of dk_t, summed over the workgroup's rows through LDS.
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      const int c = lane + 64 * j;
      if (c < H) red[w * H + c] = gr * st[j] + bt * a[j] * e - bt * st[j] * ak;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < H; c += kRowsPerBlock * 64) {
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < kRowsPerBlock; ++r) sum += red[r * H + c];
      pdk[((base / H + t) * nrb + rb) * H + c] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CPL; ++j) a[j] = fmaf(gr - bt * ak, kt[j], a[j]);
  }
}

// dk[b, t, c] = sum over row blocks of pdk (block order); dbeta[b, t] = sum over rows of
// pbeta (row order). One thread per output element.
__global__ void __launch_bounds__(256) perm_reduce_kernel(int64_t BT, int H, int nrb,
                                                          const float* __restrict__ pdk,
                                                          const float* __restrict__ pbeta,
                                                          float* __restrict__ dk,
                                                          float* __restrict__ dbeta) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < BT * H) {
    const int64_t bt = i / H;
    const int c = static_cast<int>(i % H);
    float sum = 0.0f;
    for (int r = 0; r < nrb; ++r) sum += pdk[(bt * nrb + r) * H + c];
    dk[i] = sum;
  }
  if (i < BT) {
    float sum = 0.0f;
    for (int r = 0; r < H; ++r) sum += pbeta[i * H + r];
    dbeta[i] = sum;
  }
}

// ---------------------------------------------------------------------------
// Chunked scan (H <= 512). Over a chunk of C = 16 steps entered with state S0, with
// G[t][j] = k_t . k_j and e_t = beta_t (v_t - r_t),
//   S_t = S0 + sum_{j<t} e_j k_j^T,   r_t = S0 k_t + sum_{j<t} G[t][j] e_j,
// so a chunk is two matrix products, P = K S0^T and S += E^T K, around a 16-step triangular
// solve per value row: matrix instructions instead of a wave reduction per step. The adjoint
// has the same form backwards, with d_t = g_t - beta_t u_t (u_t = A_{t+1} k_t):
//   u_t = A_end k_t + sum_{j>t} G[t][j] d_j,   A_0 = A_end + D^T K,
//   dk_t = S0^T d_t + A_end^T e_t + sum_j N[t][j] k_j,  N[t][j] = d_max(t,j) . e_min(t,j)
// (dots over value rows, N[t][t] = 0). All in fp32 (v_mfma_f32_16x16x4_f32), as the walk per
// step below, whose order of summation it replaces.
//
// A workgroup owns 16 value rows of one batch row; its 4 waves split the H columns. S^T (or
// A^T) lives in the accumulators as [column][row] tiles: with the k index of the products
// permuted (k-step i takes column 4 (lane / 16) + i) the accumulators are at once the operand
// of P, so the state never moves. The K chunk is staged in LDS one chunk ahead.
//
// Bound by the chunk's serial chain: the products (8 NT MFMAs of 32 cycles a wave, 22 NT + 8
// backward), two barriers and the solve, about 1.6 us a chunk forward and 3.5 us backward at
// H = 256. B = 16, T = 1024, H = 256, step by step -> in chunks: forward 576 -> 98 us with G,
// backward 2410 -> 393 us; error against 64 bits 5.1e-7 -> 4.5e-7 at worst there, and over
// H = 32..512, T = 60..1024 between 0.6 and 1.3 times the walk's, all below 5e-7.
namespace chunked {

constexpr int C = 16;     // steps per chunk
constexpr int RB = 16;    // value rows per workgroup
constexpr int NTH = 256;  // 4 waves
constexpr int ES = 20;    // row stride of the [16][16] LDS tiles (16-byte rows, spread banks)

// Columns per wave: 16 NT; the workgroup covers HP = 64 NT >= H columns (zeros past H).
// LDS row stride: 16-byte aligned, = 20 mod 64 words, so the 16 rows of a 16-byte read and
// the 4 rows of a 4-byte one start on different banks.
template <int NT>
struct Geo {
  static constexpr int HP = 64 * NT, LS = HP + ES;
};

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// A value that is the same in every lane, as a scalar (a resource must be one).
__device__ __forceinline__ uint32_t uniform(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

// Lane J of every 16-lane row, to all lanes of the row (DPP row_newbcast).
template <int J>
__device__ __forceinline__ float row_bcast(float x) {
  const int v = __builtin_bit_cast(int, x);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(v, v, 0x150 + J, 0xF, 0xF, true));
}

// acc += sum over steps of row[j] e_j in solve order, e_j = lane j's f(acc): forward over
// j = 0..15 for the lanes t > j, or backward for those with t < j. A lane that does not depend
// on step j keeps its value by a select, not by a zero coefficient: a non-finite later step
// must not reach an earlier one. After the walk every lane holds its own step's final value.
template <bool REV, typename F>
__device__ __forceinline__ void solve16(const float (&row)[C], int t, float& acc, F f) {
#define DABSN_STEP(J)                                              \
  {                                                                \
    const float x = fmaf(row[J], row_bcast<J>(f(acc)), acc);       \
    acc = (REV ? t < J : t > J) ? x : acc;                         \
  }
  if constexpr (!REV) {
    DABSN_STEP(0) DABSN_STEP(1) DABSN_STEP(2) DABSN_STEP(3) DABSN_STEP(4) DABSN_STEP(5)
    DABSN_STEP(6) DABSN_STEP(7) DABSN_STEP(8) DABSN_STEP(9) DABSN_STEP(10) DABSN_STEP(11)
    DABSN_STEP(12) DABSN_STEP(13) DABSN_STEP(14)
  } else {
    DABSN_STEP(15) DABSN_STEP(14) DABSN_STEP(13) DABSN_STEP(12) DABSN_STEP(11) DABSN_STEP(10)
    DABSN_STEP(9) DABSN_STEP(8) DABSN_STEP(7) DABSN_STEP(6) DABSN_STEP(5) DABSN_STEP(4)
    DABSN_STEP(3) DABSN_STEP(2) DABSN_STEP(1)
  }
#undef DABSN_STEP
}

// 4 consecutive elements of row t of k [T][H] from column c. The loads are unconditional, at
// clamped addresses (a load under a branch is waited for where the branch ends); mask_k4 puts
// the zeros past T and H where the values are used. VEC: H is a multiple of 4 and k 16-byte
// aligned.
template <bool VEC>
__device__ __forceinline__ f32x4 load_k4(const float* __restrict__ k, int T, int H, int t, int c) {
  const float* p = k + static_cast<size_t>(min(t, T - 1)) * H;
  if constexpr (VEC) {
    return *reinterpret_cast<const f32x4*>(p + (c < H ? c : 0));
  } else {
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = p[min(c + i, H - 1)];
    return v;
  }
}
__device__ __forceinline__ f32x4 mask_k4(f32x4 v, int T, int H, int t, int c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = t < T && c + i < H ? v[i] : 0.0f;
  return v;
}

// One chunk's G (steps t0 ..) by one wave: lane's entries [4 (lane / 16) + i][lane % 16]. With the
// k index permuted as above the same registers are both operands.
template <bool VEC>
__device__ __forceinline__ f32x4 gram_tile(const float* __restrict__ kb, int T, int H, int t0, int lane) {
  const int t = t0 + (lane & 15);
  f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
  for (int c = 4 * (lane >> 4); c < H + 4 * (lane >> 4); c += 32) {
    const f32x4 x = mask_k4(load_k4<VEC>(kb, T, H, t, c), T, H, t, c);
    const f32x4 y = mask_k4(load_k4<VEC>(kb, T, H, t, c + 16), T, H, t, c + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a0 = mma(x[i], x[i], a0);
      a1 = mma(y[i], y[i], a1);
    }
  }
  return a0 + a1;
}

// G [B][chunks][16][16] of every chunk: one wave per chunk. Short scans of short keys have every
// workgroup form its own in LDS instead (the same bits), which takes a launch and an allocation
// out of each direction. us forward / backward on the device, with the kernel -> in LDS: B=1 T=16
// H=32 6.0 / 12.8 -> 3.6 / 7.2 (the walk per step 5.2 / 25.5), B=16 T=64 H=256 12.5 / 39.2 -> 11.0
// / 33.5, B=64 T=128 H=64 11.3 / 31.6 -> 10.0 / 27.5; but, every row block forming the same G,
// B=64 T=128 H=256 40.8 / 182 -> 52.3 / 179, B=64 T=64 H=512 69.8 / 398 -> 96.5 / 465 and, past
// the 2,048 row blocks that hide it in their launch, B=256 T=64 H=256 70.8 / 368 -> 90.5 / 382.
constexpr int kShort = 8;
static bool brief(int64_t B, int64_t T, int64_t H) {
  return ((T <= kShort * C && H <= 128) || (T <= kShort / 2 * C && H <= 256)) && B * H <= 2048 * RB;
}
template <bool VEC>
__global__ void __launch_bounds__(NTH) gram_kernel(int T, int H, int nchunk, int64_t total,
                                                   const float* __restrict__ k,
                                                   float* __restrict__ gram) {
  const int64_t id = static_cast<int64_t>(blockIdx.x) * (NTH / 64) + (threadIdx.x >> 6);
  if (id >= total) return;  // whole waves
  const int lane = threadIdx.x & 63;
  const f32x4 g = gram_tile<VEC>(k + static_cast<size_t>(id / nchunk) * T * H, T, H,
                                 static_cast<int>(id % nchunk) * C, lane);
#pragma unroll
  for (int i = 0; i < 4; ++i) gram[id * (C * C) + (4 * (lane >> 4) + i) * C + (lane & 15)] = g[i];
}

// G of a short scan in LDS (SHORT), or row t of it in the workspace.
template <int NT, bool SHORT>
struct Gram {
  float g[!SHORT ? 1 : NT <= 2 ? kShort : kShort / 2][C][C];
  template <bool VEC>
  __device__ __forceinline__ void fill(const float* __restrict__ kb, int T, int H, int nchunk) {
    if constexpr (SHORT) {
      const int lane = threadIdx.x & 63;
      for (int n = threadIdx.x >> 6; n < nchunk; n += NTH / 64) {
        const f32x4 v = gram_tile<VEC>(kb, T, H, n * C, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) g[n][4 * (lane >> 4) + i][lane & 15] = v[i];
      }
      __syncthreads();
    }
  }
};

// A chunk's K rows in registers (one chunk ahead) and in LDS.
template <int NT, bool VEC>
struct Stage {
  f32x4 r[NT];
  __device__ __forceinline__ void load(const float* __restrict__ kb, int T, int H, int t0) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int q = threadIdx.x + i * NTH;
      r[i] = load_k4<VEC>(kb, T, H, t0 + q / (Geo<NT>::HP / 4), q % (Geo<NT>::HP / 4) * 4);
    }
  }
  __device__ __forceinline__ void store(float (*kl)[Geo<NT>::LS], int T, int H, int t0) const {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int q = threadIdx.x + i * NTH;
      const int t = q / (Geo<NT>::HP / 4), c = q % (Geo<NT>::HP / 4) * 4;
      *reinterpret_cast<f32x4*>(&kl[t][c]) = mask_k4(r[i], T, H, t0 + t, c);
    }
  }
};

// This wave's share of K X^T (X^T in `x` as [column][row] tiles), as its [row][t] partial.
template <int NT>
__device__ __forceinline__ void partial(const float (*kl)[Geo<NT>::LS], const f32x4 (&x)[NT],
                                        int lane, int c0, float (*out)[ES]) {
  f32x4 acc[4];  // four chains: shorter sums, and no product waits for the one before it
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const f32x4 kv = *reinterpret_cast<const f32x4*>(&kl[lane & 15][c0 + 16 * n + 4 * (lane >> 4)]);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = mma(kv[i], x[n][i], acc[i]);
  }
  *reinterpret_cast<f32x4*>(&out[lane & 15][4 * (lane >> 4)]) =
      (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

// What a lane of the solve reads of one chunk: lane = 16 (row % 4) + t of wave row / 4. Loaded
// at clamped addresses, zeroed past T and the rows where it is used.
struct StepIn {
  float x, beta, f;  // v (forward) or g and v - r (backward)
  f32x4 g[4];        // row t of G
  template <int NT, bool SHORT>
  __device__ __forceinline__ void load_row(const Gram<NT, SHORT>& gr, const float* __restrict__ gb, int n,
                                           int t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (SHORT)
        g[i] = *reinterpret_cast<const f32x4*>(&gr.g[n][t][4 * i]);
      else
        g[i] = *reinterpret_cast<const f32x4*>(gb + (static_cast<size_t>(n) * C + t) * C + 4 * i);
    }
  }
  // Row t for the solve. The entry it has no use for (15 forward, 0 backward) is kept alive to
  // here: a loaded register that nothing reads is reused, and waited for, right after its load.
  __device__ __forceinline__ void row(float (&r)[C]) const {
#pragma unroll
    for (int j = 0; j < C; ++j) r[j] = g[j / 4][j % 4];
    asm volatile("" : : "v"(r[0]), "v"(r[C - 1]));
  }
  __device__ __forceinline__ void mask(bool in_t, bool in_row) {
    beta = in_t ? beta : 0.0f;
    x = in_t && in_row ? x : 0.0f;
    f = in_t && in_row ? f : 0.0f;
  }
};

template <int NT>
struct FwdLds {
  float kl[2][C][Geo<NT>::LS];
  float pb[4][RB][ES];
  float eb[C][ES];
};

// Forward. TAPE: writes v - r and every chunk's entering state for the backward, else r. `gram`:
// the batch row's G (unless SHORT).
template <int NT, bool VEC, bool TAPE, bool SHORT>
__device__ __forceinline__ void fwd_body(FwdLds<NT>& m_, const Gram<NT, SHORT>& gr, int T, int H,
                                         int nchunk, const float* __restrict__ k, const float* __restrict__ v,
                                         const float* __restrict__ beta,
                                         const float* __restrict__ gb, float* out, float* states) {
  using Ge = Geo<NT>;
  auto& kl = m_.kl;
  auto& pb = m_.pb;
  auto& eb = m_.eb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rb = blockIdx.x, b = blockIdx.y;
  const int c0 = wave * 16 * NT;
  const int t = lane & 15, lr = 4 * wave + (lane >> 4), row = rb * RB + lr;
  const size_t base = static_cast<size_t>(b) * T * H;
  const float* kb = k + base;
  f32x4 s[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) s[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto step_in = [&](int n) {
    StepIn q;
    const int tt = min(n * C + t, T - 1);
    q.x = v[base + static_cast<size_t>(tt) * H + min(row, H - 1)];
    q.beta = beta[static_cast<size_t>(b) * T + tt];
    q.f = 0.0f;
    q.load_row(gr, gb, n, t);
    return q;
  };
  Stage<NT, VEC> st;
  st.load(kb, T, H, 0);
  st.store(kl[0], T, H, 0);
  st.load(kb, T, H, C);
  StepIn in = step_in(0);
  __syncthreads();
  for (int n = 0; n < nchunk; ++n) {
    const int cur = n & 1;
    const StepIn nx = step_in(n + 1 < nchunk ? n + 1 : n);
    if constexpr (TAPE) {
      float* sp = states + ((static_cast<size_t>(b) * gridDim.x + rb) * nchunk + n) * (RB * Ge::HP);
#pragma unroll
      for (int i = 0; i < NT; ++i)
        *reinterpret_cast<f32x4*>(sp + (lane & 15) * Ge::HP + c0 + 16 * i + 4 * (lane >> 4)) = s[i];
    }
    partial<NT>(kl[cur], s, lane, c0, pb[wave]);
    __syncthreads();
    in.mask(n * C + t < T, row < H);
    float r = ((pb[0][lr][t] + pb[1][lr][t]) + pb[2][lr][t]) + pb[3][lr][t];
    float grow[C];
    in.row(grow);
    solve16<false>(grow, t, r, [&](float a) { return in.beta * (in.x - a); });
    const float f = in.x - r;
    eb[t][lr] = in.beta * f;
    if (n * C + t < T && row < H)
      out[base + static_cast<size_t>(n * C + t) * H + row] = TAPE ? f : r;
    st.store(kl[cur ^ 1], T, H, (n + 1) * C);
    st.load(kb, T, H, (n + 2) * C);
    __syncthreads();
    // S^T += K^T E: k-step i takes step 4 (lane / 16) + i.
    float ev[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ev[i] = eb[4 * (lane >> 4) + i][lane & 15];
    float kv[4][NT];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int m = 0; m < NT; ++m)
        kv[i][m] = kl[cur][4 * (lane >> 4) + i][c0 + 16 * m + (lane & 15)];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int m = 0; m < NT; ++m) s[m] = mma(kv[i][m], ev[i], s[m]);
    }
    in = nx;
  }
}

template <int NT, bool VEC, bool SHORT>
__global__ void __launch_bounds__(NTH, 1) fwd_kernel(int T, int H, int nchunk,
                                                     const float* __restrict__ k,
                                                     const float* __restrict__ v,
                                                     const float* __restrict__ beta,
                                                     const float* __restrict__ gram,
                                                     float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) FwdLds<NT> m;
  __shared__ __attribute__((aligned(16))) Gram<NT, SHORT> gr;
  gr.template fill<VEC>(k + static_cast<size_t>(blockIdx.y) * T * H, T, H, nchunk);
  fwd_body<NT, VEC, false, SHORT>(m, gr, T, H, nchunk, k, v, beta,
                           gram + static_cast<size_t>(blockIdx.y) * nchunk * C * C, out, nullptr);
}

// Backward: the forward again for v - r and the entering states, which only this workgroup
// reads, then the chunks from the last. dk goes out as one partial per row block
// ([B][T][nrb][H]), dbeta as one value per row block ([B][T][nrb]); reduce_kernel adds them in
// order.
template <int NT, bool VEC, bool SHORT>
__global__ void __launch_bounds__(NTH, 1) bwd_kernel(int T, int H, int nchunk,
                                                     const float* __restrict__ k,
                                                     const float* __restrict__ v,
                                                     const float* __restrict__ beta,
                                                     const float* __restrict__ g,
                                                     const float* __restrict__ gram,
                                                     float* ftape, float* states,
                                                     float* __restrict__ dv,
                                                     float* __restrict__ pdk,
                                                     float* __restrict__ pbeta) {
  using Ge = Geo<NT>;
  __shared__ __attribute__((aligned(16))) FwdLds<NT> m_;
  __shared__ __attribute__((aligned(16))) Gram<NT, SHORT> gr;
  __shared__ __attribute__((aligned(16))) float at[RB][Ge::LS];  // A_end as [row][column]
  __shared__ __attribute__((aligned(16))) float db[C][ES];
  __shared__ float bb[C][ES];
  auto& kl = m_.kl;
  auto& pb = m_.pb;
  auto& eb = m_.eb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rb = blockIdx.x, b = blockIdx.y, nrb = gridDim.x;
  const int c0 = wave * 16 * NT, hi = 4 * (lane >> 4), lo = lane & 15;
  const int t = lo, lr = 4 * wave + (lane >> 4), row = rb * RB + lr;
  const size_t base = static_cast<size_t>(b) * T * H;
  const float* kb = k + base;
  const float* gb = gram + static_cast<size_t>(b) * nchunk * C * C;
  gr.template fill<VEC>(kb, T, H, nchunk);
  fwd_body<NT, VEC, true, SHORT>(m_, gr, T, H, nchunk, k, v, beta, gb, ftape, states);
  __syncthreads();  // the tape and the states are read by other threads than wrote them
  f32x4 a[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) a[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto step_in = [&](int n) {
    StepIn q;
    const int tt = min(n * C + t, T - 1);
    const size_t o = base + static_cast<size_t>(tt) * H + min(row, H - 1);
    q.x = g[o];
    q.f = ftape[o];
    q.beta = beta[static_cast<size_t>(b) * T + tt];
    q.load_row(gr, gb, n, t);
    return q;
  };
  Stage<NT, VEC> st;
  st.load(kb, T, H, (nchunk - 1) * C);
  st.store(kl[(nchunk - 1) & 1], T, H, (nchunk - 1) * C);
  st.load(kb, T, H, max(nchunk - 2, 0) * C);
  // The entering state as the operand of D S0 (k-step i takes row 4 (lane / 16) + i), loaded a
  // chunk ahead like everything else: a load waits for the partials' stores before it.
  float s0[NT][4];
  auto load_s0 = [&](int n) {
    const float* sp = states + ((static_cast<size_t>(b) * nrb + rb) * nchunk + n) * (RB * Ge::HP);
#pragma unroll
    for (int m = 0; m < NT; ++m) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s0[m][i] = sp[(hi + i) * Ge::HP + c0 + 16 * m + lo];
    }
  };
  load_s0(nchunk - 1);
  StepIn in = step_in(nchunk - 1);
  __syncthreads();
  for (int n = nchunk - 1; n >= 0; --n) {
    const int cur = n & 1;
    const StepIn nx = step_in(n > 0 ? n - 1 : 0);
#pragma unroll
    for (int m = 0; m < NT; ++m) *reinterpret_cast<f32x4*>(&at[lo][c0 + 16 * m + hi]) = a[m];
    partial<NT>(kl[cur], a, lane, c0, pb[wave]);
    __syncthreads();
    in.mask(n * C + t < T, row < H);
    float u = ((pb[0][lr][t] + pb[1][lr][t]) + pb[2][lr][t]) + pb[3][lr][t];
    float grow[C];
    in.row(grow);
    solve16<true>(grow, t, u, [&](float x) { return in.x - in.beta * x; });
    db[t][lr] = in.x - in.beta * u;
    eb[t][lr] = in.beta * in.f;
    bb[t][lr] = u * in.f;
    if (n * C + t < T && row < H) dv[base + static_cast<size_t>(n * C + t) * H + row] = in.beta * u;
    st.store(kl[cur ^ 1], T, H, max(n - 1, 0) * C);
    st.load(kb, T, H, max(n - 2, 0) * C);
    __syncthreads();
    if (threadIdx.x < C && n * C + static_cast<int>(threadIdx.x) < T) {
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < RB; ++r) sum += bb[threadIdx.x][r];
      pbeta[(static_cast<size_t>(b) * T + n * C + threadIdx.x) * nrb + rb] = sum;
    }
    const f32x4 dop = *reinterpret_cast<const f32x4*>(&db[lo][hi]);
    const f32x4 eop = *reinterpret_cast<const f32x4*>(&eb[lo][hi]);
    f32x4 m1 = {0.f, 0.f, 0.f, 0.f}, m2 = m1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m1 = mma(dop[i], eop[i], m1);  // [hi + i][lo] = d_(hi+i) . e_lo
      m2 = mma(eop[i], dop[i], m2);  // [hi + i][lo] = e_(hi+i) . d_lo
    }
    float nop[4], dval[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = hi + i;
      nop[i] = j > lo ? m1[i] : j < lo ? m2[i] : 0.0f;
      dval[i] = db[j][lo];
    }
    f32x4 dkp[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      const int c = c0 + 16 * m + lo;
      float kv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) kv[i] = kl[cur][hi + i][c];
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x, z = x;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x = mma(dop[i], s0[m][i], x);
        y = mma(eop[i], at[hi + i][c], y);
        z = mma(nop[i], kv[i], z);
        a[m] = mma(kv[i], dval[i], a[m]);
      }
      dkp[m] = (x + y) + z;
    }
    load_s0(max(n - 1, 0));
    // Rows past T lie past the resource and columns past H get an offset past it, so the
    // stores need no branches.
    const uint64_t pa = reinterpret_cast<uint64_t>(
        pdk + ((static_cast<size_t>(b) * T + n * C) * nrb + rb) * H);
    const uint64_t pu = static_cast<uint64_t>(uniform(static_cast<uint32_t>(pa))) |
                        static_cast<uint64_t>(uniform(static_cast<uint32_t>(pa >> 32))) << 32;
    const __amdgpu_buffer_rsrc_t pr =
        make_rsrc(reinterpret_cast<const void*>(pu),
                  uniform(static_cast<uint32_t>(((min(C, T - n * C) - 1) * nrb + 1) * H * 4)));
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      const int c = c0 + 16 * m + lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = dkp[m][i];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), pr,
                                              c < H ? ((hi + i) * nrb * H + c) * 4 : 0x7fffffff, 0, 0);
      }
    }
    in = nx;
  }
}

// dk and dbeta from the row blocks' partials, in block order.
__global__ void __launch_bounds__(NTH) reduce_kernel(int64_t BT, int H, int nrb,
                                                     const float* __restrict__ pdk,
                                                     const float* __restrict__ pbeta,
                                                     float* __restrict__ dk,
                                                     float* __restrict__ dbeta) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * NTH + threadIdx.x;
  if (i < BT * H) {
    const float* p = pdk + (i / H * nrb) * H + i % H;
    float sum = 0.0f;
#pragma unroll 8
    for (int r = 0; r < nrb; ++r) sum += p[static_cast<size_t>(r) * H];
    dk[i] = sum;
  }
  if (i < BT) {
    float sum = 0.0f;
    for (int r = 0; r < nrb; ++r) sum += pbeta[i * nrb + r];
    dbeta[i] = sum;
  }
}

// Workspace: G, then (backward) v - r [B][T][H], the entering states, the partials.
struct Layout {
  size_t gram, ftape, states, pdk, pbeta, end;
};
static int tiles_for(int64_t H) {
  for (int n : {1, 2, 4, 8})
    if (H <= 64 * n) return n;
  return 0;
}
static Layout layout(int64_t B, int64_t T, int64_t H, bool backward) {
  const size_t nchunk = static_cast<size_t>((T + C - 1) / C), nrb = static_cast<size_t>((H + RB - 1) / RB);
  const size_t bt = static_cast<size_t>(B) * T;
  auto up = [](size_t x) { return (x + 255) & ~static_cast<size_t>(255); };
  Layout l{};
  size_t o = brief(B, T, H) ? 0 : up(static_cast<size_t>(B) * nchunk * C * C * 4);
  if (backward) {
    l.ftape = o; o = up(o + bt * H * 4);
    l.states = o; o = up(o + static_cast<size_t>(B) * nrb * nchunk * RB * 64 * tiles_for(H) * 4);
    l.pdk = o; o = up(o + bt * nrb * H * 4);
    l.pbeta = o; o = up(o + bt * nrb * 4);
  }
  l.end = o;
  return l;
}

// Forward (out = r), or backward (g given).
template <int NT, bool VEC, bool SHORT>
static void launch(int64_t B, int64_t T, int64_t H, const float* k, const float* v,
                   const float* beta, const float* g, float* out, float* dk, float* dv,
                   float* dbeta, uint8_t* ws, hipStream_t stream) {
  const Layout l = layout(B, T, H, g != nullptr);
  const int nchunk = static_cast<int>((T + C - 1) / C), nrb = static_cast<int>((H + RB - 1) / RB);
  float* gram = reinterpret_cast<float*>(ws + l.gram);
  if constexpr (!SHORT) {
    const int64_t total = B * nchunk;
    hipLaunchKernelGGL((gram_kernel<VEC>), dim3(static_cast<unsigned>((total + 3) / 4)), dim3(NTH), 0,
                       stream, (int)T, (int)H, nchunk, total, k, gram);
  }
  const dim3 grid(static_cast<unsigned>(nrb), static_cast<unsigned>(B));
  if (!g) {
    hipLaunchKernelGGL((fwd_kernel<NT, VEC, SHORT>), grid, dim3(NTH), 0, stream, (int)T, (int)H, nchunk,
                       k, v, beta, gram, out);
    return;
  }
  float* ftape = reinterpret_cast<float*>(ws + l.ftape);
  float* states = reinterpret_cast<float*>(ws + l.states);
  float* pdk = reinterpret_cast<float*>(ws + l.pdk);
  float* pbeta = reinterpret_cast<float*>(ws + l.pbeta);
  hipLaunchKernelGGL((bwd_kernel<NT, VEC, SHORT>), grid, dim3(NTH), 0, stream, (int)T, (int)H, nchunk, k,
                     v, beta, g, gram, ftape, states, dv, pdk, pbeta);
  const int64_t BT = B * T;
  hipLaunchKernelGGL(reduce_kernel, dim3(static_cast<unsigned>((BT * H + NTH - 1) / NTH)), dim3(NTH),
                     0, stream, BT, (int)H, nrb, pdk, pbeta, dk, dbeta);
}

static int run(int64_t B, int64_t T, int64_t H, const float* k, const float* v, const float* beta,
               const float* g, float* out, float* dk, float* dv, float* dbeta, uint8_t* ws,
               hipStream_t stream) {
  const bool vec = H % 4 == 0 && (reinterpret_cast<uintptr_t>(k) & 15u) == 0;
  const bool in_lds = brief(B, T, H);
  switch (tiles_for(H)) {
#define DABSN_RUN(N, SHORT)                                                                   \
  if (vec)                                                                                    \
    launch<N, true, SHORT>(B, T, H, k, v, beta, g, out, dk, dv, dbeta, ws, stream);           \
  else                                                                                        \
    launch<N, false, SHORT>(B, T, H, k, v, beta, g, out, dk, dv, dbeta, ws, stream)
#define DABSN_CASE(N)      \
  case N:                  \
    if (in_lds) {          \
      DABSN_RUN(N, true);  \
    } else {               \
      DABSN_RUN(N, false); \
    }                      \
    break;
    DABSN_CASE(1) DABSN_CASE(2) DABSN_CASE(4)
#undef DABSN_CASE
    case 8:
      DABSN_RUN(8, false);
      break;
#undef DABSN_RUN
  }
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

}  // namespace chunked

static int cpl_for(int64_t H) {
  for (int c : {1, 2, 4, 8, 16, 32})
    if (H <= 64 * c) return c;
  return 0;
}

static int checks(int64_t B, int64_t T, int64_t H, const void* k, const void* v,
                  const void* beta) {
  DABSN_REQUIRE(B > 0 && T >= 0 && H > 0, "permanent scan: bad shape");
  DABSN_REQUIRE(B < 65536 && T < (1 << 30), "permanent scan: dimension too large");
  DABSN_REQUIRE(cpl_for(H) != 0, "permanent scan: H=%lld > 2048 is not supported", (long long)H);
  DABSN_REQUIRE(k && v && beta, "permanent scan: null pointer");
  return DABSN_OK;
}

}  // namespace permanent
}  // namespace dabsn

using namespace dabsn;
using namespace dabsn::permanent;

extern "C" {

size_t dabsn_hip_permanent_scan_fwd_workspace_bytes(int64_t B, int64_t T, int64_t H) {
  if (B <= 0 || T <= 0 || H <= 0 || chunked::tiles_for(H) == 0) return 0;
  return chunked::layout(B, T, H, false).end;
}

int dabsn_hip_permanent_scan_fwd_ws(int64_t B, int64_t T, int64_t H, const float* key,
                                    const float* value, const float* beta, float* out,
                                    void* workspace, size_t workspace_bytes, hipStream_t stream) {
  int rc = checks(B, T, H, key, value, beta);
  if (rc != DABSN_OK) return rc;
  if (chunked::tiles_for(H) == 0)
    return dabsn_hip_permanent_scan_fwd(B, T, H, key, value, beta, out, stream);
  DABSN_REQUIRE(out, "permanent scan: null output");
  if (T == 0) return DABSN_OK;
  const size_t need = chunked::layout(B, T, H, false).end;  // none for short scans
  DABSN_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), "permanent scan: workspace %zu < %zu",
                workspace_bytes, need);
  return chunked::run(B, T, H, key, value, beta, nullptr, out, nullptr, nullptr, nullptr,
                      static_cast<uint8_t*>(workspace), stream);
}

int dabsn_hip_permanent_scan_fwd(int64_t B, int64_t T, int64_t H, const float* key,
                                 const float* value, const float* beta, float* out,
                                 hipStream_t stream) {
  int rc = checks(B, T, H, key, value, beta);
  if (rc != DABSN_OK) return rc;
  DABSN_REQUIRE(out, "permanent scan: null output");
  if (T == 0) return DABSN_OK;
  const dim3 grid(static_cast<unsigned>((H + kFwdRows - 1) / kFwdRows), static_cast<unsigned>(B));
  const dim3 block(kFwdRows * 64);
  switch (cpl_for(H)) {
#define DABSN_CASE(C)                                                                        \
  case C:                                                                                    \
    hipLaunchKernelGGL(perm_fwd_kernel<C>, grid, block, 0, stream, (int)T, (int)H, key, value, \
                       beta, out);                                                           \
    break;
    DABSN_CASE(1) DABSN_CASE(2) DABSN_CASE(4) DABSN_CASE(8) DABSN_CASE(16) DABSN_CASE(32)
#undef DABSN_CASE
  }
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

size_t dabsn_hip_permanent_scan_workspace_bytes(int64_t B, int64_t T, int64_t H) {
  if (B <= 0 || T <= 0 || H <= 0) return 0;
  if (chunked::tiles_for(H) != 0) return chunked::layout(B, T, H, true).end;
  return bwd_layout(B, T, H).end;
}

int dabsn_hip_permanent_scan_bwd(int64_t B, int64_t T, int64_t H, const float* key,
                                 const float* value, const float* beta, const float* grad_out,
                                 float* dkey, float* dvalue, float* dbeta, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
  int rc = checks(B, T, H, key, value, beta);
  if (rc != DABSN_OK) return rc;
  DABSN_REQUIRE(grad_out && dkey && dvalue && dbeta, "permanent scan backward: null pointer");
  if (T == 0) return DABSN_OK;
  if (chunked::tiles_for(H) != 0) {
    const size_t need = chunked::layout(B, T, H, true).end;
    DABSN_REQUIRE(workspace && workspace_bytes >= need,
                  "permanent scan backward: workspace %zu < %zu", workspace_bytes, need);
    return chunked::run(B, T, H, key, value, beta, grad_out, nullptr, dkey, dvalue, dbeta,
                        static_cast<uint8_t*>(workspace), stream);
  }
  const BwdLayout l = bwd_layout(B, T, H);
  DABSN_REQUIRE(workspace && workspace_bytes >= l.end,
                "permanent scan backward: workspace %zu < %zu", workspace_bytes, l.end);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  float* tape = reinterpret_cast<float*>(ws + l.tape);
  float* rtape = reinterpret_cast<float*>(ws + l.rtape);
  float* pdk = reinterpret_cast<float*>(ws + l.pdk);
  float* pbeta = reinterpret_cast<float*>(ws + l.pbeta);
  const int nrb = static_cast<int>((H + kRowsPerBlock - 1) / kRowsPerBlock);
  const dim3 grid(static_cast<unsigned>(nrb), static_cast<unsigned>(B));
  const dim3 block(kRowsPerBlock * 64);
  const size_t lds = static_cast<size_t>(kRowsPerBlock) * H * 4;
  switch (cpl_for(H)) {
#define DABSN_CASE(C)                                                                       \
  case C:                                                                                   \
    hipLaunchKernelGGL(perm_bwd_kernel<C>, grid, block, lds, stream, (int)T, (int)H, key,   \
                       value, beta, grad_out, dvalue, tape, rtape, pdk, pbeta);             \
    break;
    DABSN_CASE(16) DABSN_CASE(32)
#undef DABSN_CASE
  }
  DABSN_HIP_CHECK(hipGetLastError());
  const int64_t BT = B * T;
  hipLaunchKernelGGL(perm_reduce_kernel, dim3(static_cast<unsigned>((BT * H + 255) / 256)),
                     dim3(256), 0, stream, BT, (int)H, nrb, pdk, pbeta, dkey, dbeta);
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

}  // extern "C"
