// Diagonal linear recurrences: the registered dabsn::linear_recurrence pair and the
// fused recurrent long-memory scan.
//
// Reference: src/dabsn/kernels/long.py:24-98 (linear recurrence and its analytic
// reverse), long.py:492-579 (long memory as three recurrences plus glue), loop form in
// src/dabsn/read.py:625-636; CPU kernels cpu_runtime.cpp:92-143.
//
// linear_recurrence: one thread owns one (batch row, unit) channel and walks T;
// consecutive threads own consecutive units, so each time step is one coalesced row
// access, with a block of time steps loaded ahead of the dependent arithmetic.
//
// Long memory, parallel over time as well as channels. Per channel the forward is three
// chained recurrences: E_t = er E + (1-er) w (constant coefficient), R_t = rd R +
// (1-rd)(1 - pe_t) with pe_t = tanh|w_t - E_{t-1}| (constant coefficient, input known once
// E is), and L_t = eff_t L + (1 - eff_t) sal_t w_t (coefficient eff_t known once R is).
// T is cut into chunks of CK steps. A workgroup owns 64 channels of one batch row (16 where
// channels are few); each of its waves holds one chunk's inputs in registers (four chunks of 16
// channels), and the workgroup walks T in blocks of as many chunks as its waves hold. For each recurrence in turn every wave computes its chunk's end value from a zero
// start (and the product of eff_t for L), one barrier shares the ends through LDS, and every
// wave folds the chunks before its own into its true start. So the inputs are read once and
// tanh is evaluated once per step, between one read and one write of memory (the earlier form
// ran a kernel per recurrence: four reads of w, three tanh). The chunk starts are the
// checkpoint, [B][nseg][3][H] fp32, kept for the backward, which replays each chunk's forward
// from it with the same step function (the same bits) and then carries the three adjoints
// backward the same way: gL, then gR, then gE.
//
// Bound by memory and, nearly as much, by the vector ALU (a step is about 56 instructions
// forward and 91 backward): see the figures at the launchers.
#include <algorithm>
#include <type_traits>

#include "../../include/dabsn_hip.h"
#include "capi.hpp"
#include "common.hpp"

namespace dabsn {
namespace longmem {

constexpr int NT = 64;      // threads per block (one wave: spreads channels over CUs)
constexpr int TB = 8;       // time steps loaded ahead
constexpr int CK = DABSN_LONG_CKPT;

template <typename E>
__global__ void __launch_bounds__(NT) linrec_fwd_kernel(int B, int T, int H, const E* a,
                                                        const E* g, const E* y0, E* y) {
  const int64_t ch = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (ch >= static_cast<int64_t>(B) * H) return;
  const int64_t b = ch / H, h = ch % H;
  float carry = ld(y0, ch);
  const size_t base = static_cast<size_t>(b) * T * H + h;
  for (int t0 = 0; t0 < T; t0 += TB) {
    float av[TB], gv[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      // Clamped, unconditional loads: all TB requests are issued before the first use
      // (values past T are never used).
      const size_t o = base + static_cast<size_t>(min(t0 + i, T - 1)) * H;
      av[i] = ld(a, o);
      gv[i] = ld(g, o);
    }
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      const int t = t0 + i;
      if (t < T) {
        carry = av[i] * carry + gv[i];
        st(y, base + static_cast<size_t>(t) * H, carry);
      }
    }
  }
}

// Reverse pass: c_t = gy_t + a_{t+1} c_{t+1}; dg_t = c_t; da_t = c_t y_{t-1};
// dy0 = a_0 c_0. y_{t-1} comes from an fp32 forward replay stored in `yprev`.
template <typename E>
__global__ void __launch_bounds__(NT) linrec_bwd_kernel(int B, int T, int H, const E* a,
                                                        const E* g, const E* y0, const E* gy,
                                                        E* da, E* dg, E* dy0, float* yprev) {
  const int64_t ch = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (ch >= static_cast<int64_t>(B) * H) return;
  const int64_t b = ch / H, h = ch % H;
  const size_t base = static_cast<size_t>(b) * T * H + h;
  float carry = ld(y0, ch);
  for (int t = 0; t < T; ++t) {
    const size_t o = base + static_cast<size_t>(t) * H;
    yprev[o] = carry;
    carry = ld(a, o) * carry + ld(g, o);
  }
  float c = 0.0f;
  for (int t = T - 1; t >= 0; --t) {
    const size_t o = base + static_cast<size_t>(t) * H;
    const float a_next = (t + 1 < T) ? ld(a, o + H) : 0.0f;
    c = ld(gy, o) + a_next * c;
    st(dg, o, c);
    st(da, o, c * yprev[o]);
  }
  st(dy0, ch, T > 0 ? ld(a, base) * c : 0.0f);
}

struct Coef {
  float er, rd, ret, rs;
};

__device__ __forceinline__ Coef load_coef(const float* const* logits) {
  Coef c;
  c.er = sigmoidf_(logits[0][0]);
  c.rd = sigmoidf_(logits[1][0]);
  c.ret = sigmoidf_(logits[2][0]);
  c.rs = sigmoidf_(logits[3][0]);
  return c;
}

struct Logits {
  const float* p[4];
};

// tanh(y) for y >= 0 without a branch (the library's takes one per range, both in a wave whose
// lanes disagree, and the unrolled steps around it cannot be interleaved). The range is split
// as in the Cephes library's tanhf. Below 0.625 the odd polynomial y + y^3 q(y^2), q fitted to
// (tanh y - y) / y^3 by minimax least squares (relative error 4.4e-9, and 8.5e-9 with the
// coefficients rounded to fp32); above, 1 - 2 / (exp(2y) + 1). At most 2 ulp, on average 2.4e-8
// relative. NaN stays NaN, infinity gives 1.
__device__ __forceinline__ float tanh_abs(float y) {
  const float z = y * y;
  float q = fmaf(-0.0057049826718866825f, z, 0.02063908241689205f);
  q = fmaf(q, z, -0.05373971536755562f);
  q = fmaf(q, z, 0.13331441581249237f);
  q = fmaf(q, z, -0.3333328068256378f);
  const float small = fmaf(y * z, q, y);
  const float e = __builtin_amdgcn_exp2f(y * 2.8853900817779268f);  // exp(2y)
  const float large = fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);
  return y < 0.625f ? small : large;
}

// The pieces of one step of the three recurrences (long.py:492-579) from the states entering
// it: pe = tanh|w - E|, then E, R, the retention eff and L advance. Every pass that walks the
// recurrence (forward, and the backward's replays) calls these, so the states a replay
// produces are bit-identical to the forward's. L advances as eff L + y, y = (1 - eff) x: not as
// x + eff (L - x), two instructions shorter, whose difference rounds at the size of x, which
// is well above that of its mean L.
__device__ __forceinline__ float step_E(const Coef& k, float Ev, float wt) {
  return fmaf(k.er, Ev, (1.0f - k.er) * wt);
}
__device__ __forceinline__ float step_R(const Coef& k, float R, float pe) {
  return fmaf(k.rd, R, (1.0f - k.rd) * (1.0f - pe));
}
__device__ __forceinline__ float retention(const Coef& k, float R) {
  return fmaf((1.0f - k.ret) * k.rs, R, k.ret);
}
// er^n for n <= CK by repeated multiplication (fixed order).
__device__ __forceinline__ float powi(float x, int n) {
  float r = 1.0f;
  for (int i = 0; i < n; ++i) r *= x;
  return r;
}

// A wave holds G chunks of 64 / G channels of one batch row; a workgroup of NW waves walks T in
// blocks of NW G chunks.
constexpr int LANES = 64;

// Folds the chunk ends `loc` (from a zero start, [chunk][channel]) of a block of `live` chunks
// into the state x entering the block: returns the state entering chunk `idx`, x becomes the
// state leaving the block. A chunk multiplies its entering state by prod[chunk], or by `power`
// (coef^steps, one value for all). REV: the chunks in reverse (adjoints).
template <int NC, int LC, bool REV>
__device__ __forceinline__ float enter(float& x, const float (*loc)[LC], const float (*prod)[LC],
                                       float power, int idx, int lc, int live) {
  float mine = x;
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int j = REV ? NC - 1 - q : q;
    mine = j == idx ? x : mine;
    if (j < live) x = fmaf(prod ? prod[j][lc] : power, x, loc[j][lc]);
  }
  return mine;
}

// Hides a value's history from the compiler, which otherwise keeps what one walk derives from it
// (conversions, products with a constant) in registers for the next walk: 32 values each time.
template <typename V>
__device__ __forceinline__ void opaque(V& v) {
  asm volatile("" : "+v"(v));
}

// The rows of one chunk of a [.., T, H] tensor as a wave reads and writes them: row i of the
// chunk, this lane's channel. As buffer accesses the row is a scalar offset and the lane a
// 32-bit one that stays put, so no address takes vector registers or instructions. Lanes past H
// get an offset past any chunk (reads give zero, writes are dropped), and so do the rows past
// `rows`. `first`: the lane's first row (its chunk's, where a wave holds several). Offsets are
// 32 bits: rows of 2^24 elements and more use plain pointers.
template <typename E, bool BIG>
struct Rows {
  __amdgpu_buffer_rsrc_t r;
  uint32_t voff, row;
  __device__ __forceinline__ Rows(E* p, int H, int h, int rows, int first = 0)
      : row(static_cast<uint32_t>(H) * sizeof(E)) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint64_t u = static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(a))) & 0xffffffffu;
    const uint64_t v = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32)));
    r = make_rsrc(reinterpret_cast<const void*>(u | v << 32), rows * row);
    voff = h < H && first < rows ? static_cast<uint32_t>(h) * sizeof(E) + first * row : 0x80000000u;
  }
  __device__ __forceinline__ E load(int i) const {
    if constexpr (sizeof(E) == 2) {
      return __builtin_amdgcn_raw_buffer_load_b16(r, voff, i * row, 0);
    } else {
      const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(r, voff, i * row, 0);
      return __builtin_bit_cast(E, w);
    }
  }
  __device__ __forceinline__ void store(int i, E v) const {
    if constexpr (sizeof(E) == 2)
      __builtin_amdgcn_raw_buffer_store_b16(v, r, voff, i * row, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, i * row, 0);
  }
};
template <typename E>
struct Rows<E, true> {
  E* p;
  size_t row;
  bool ok;
  __device__ __forceinline__ Rows(E* q, int H, int h, int rows, int = 0)
      : p(q + min(h, H - 1)), row(static_cast<size_t>(H)), ok(rows > 0 && h < H) {}
  __device__ __forceinline__ E load(int i) const { return p[i * row]; }
  __device__ __forceinline__ void store(int i, E v) const {
    if (ok) p[i * row] = v;
  }
};

// Every 8th step, nothing moves across: steps interleave within a group, without all 32 of a
// chunk in flight (and in registers) at once.
__device__ __forceinline__ void fence(int i) {
  if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
}

// A wave of NW workgroup waves as a scalar, so the addresses of its chunk are scalar too.
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
}

// Occupancy: the forward holds 2 values per step (at most 128 registers, 16 waves per CU).
template <typename E, int NW, int G, bool BIG>
__global__ void __launch_bounds__(NW* LANES, 4)
    long_fwd_kernel(int T, int H, int64_t ldx, const E* __restrict__ w, const E* __restrict__ p,
                    Logits lg, const float* __restrict__ L0, const float* __restrict__ E0,
                    const float* __restrict__ R0, E* __restrict__ out, float* __restrict__ LF,
                    float* __restrict__ EF, float* __restrict__ RF, float* __restrict__ ckpt) {
  constexpr int NC = NW * G, LC = LANES / G;
  __shared__ float se[NC][LC], sr[NC][LC], sl[NC][LC], sp[NC][LC];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int lc = lane % LC, sub = lane / LC, idx = wave * G + sub;
  const int h = blockIdx.x * LC + lc, b = blockIdx.y;
  const bool ok = h < H;
  const int hc = ok ? h : H - 1;
  const Coef k = load_coef(lg.p);
  const float er_full = powi(k.er, CK), rd_full = powi(k.rd, CK);
  const size_t ch = static_cast<size_t>(b) * H + hc;
  float Lc = L0[ch], Ec = E0[ch], Rc = R0[ch];
  E* wb = const_cast<E*>(w) + static_cast<size_t>(b) * ldx;
  E* pb = const_cast<E*>(p) + static_cast<size_t>(b) * ldx;
  E* ob = out + static_cast<size_t>(b) * T * H;
  const int nseg = (T + CK - 1) / CK, nfull = T / CK, tail = T % CK;
  auto keep = [&](int seg, float l, float e, float r) {
    float* c = ckpt + (static_cast<size_t>(b) * nseg + seg) * 3 * H;
    c[h] = l;
    (c + H)[h] = e;
    (c + 2 * static_cast<size_t>(H))[h] = r;
  };
  for (int k0 = 0; k0 < nfull; k0 += NC) {  // blocks of full chunks
    const int live = min(NC, nfull - k0), seg = k0 + idx;
    const bool mine = idx < live;
    const int wlive = min(max(live - wave * G, 0), G);  // chunks of this wave
    const size_t base = static_cast<size_t>(wlive > 0 ? k0 + wave * G : 0) * CK * H;
    const Rows<E, BIG> wr(wb + base, H, h, wlive * CK, sub * CK),
        pr(pb + base, H, h, wlive * CK, sub * CK), orow(ob + base, H, h, wlive * CK, sub * CK);
    E wv[CK], pv[CK];
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      wv[i] = wr.load(i);
      pv[i] = pr.load(i);
    }
    __builtin_amdgcn_sched_barrier(0);
    float e = 0.0f;
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      e = step_E(k, e, to_f(wv[i]));
      fence(i);
    }
#pragma unroll
    for (int i = 0; i < CK; ++i) opaque(wv[i]);
    se[idx][lc] = e;
    __syncthreads();
    const float Es = enter<NC, LC, false>(Ec, se, nullptr, er_full, idx, lc, live);
    float pe[CK], x[CK];
    float r = 0.0f;
    e = Es;
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      const float wt = to_f(wv[i]);
      pe[i] = tanh_abs(fabsf(wt - e));
      x[i] = (to_f(pv[i]) * pe[i]) * wt;
      e = step_E(k, e, wt);
      r = step_R(k, r, pe[i]);
      opaque(x[i]);
      opaque(pe[i]);
      fence(i);
    }
    sr[idx][lc] = r;
    __syncthreads();
    const float Rs = enter<NC, LC, false>(Rc, sr, nullptr, rd_full, idx, lc, live);
    float l = 0.0f, prod = 1.0f;
    r = Rs;
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      r = step_R(k, r, pe[i]);
      pe[i] = retention(k, r);  // from here on: eff of the step, and y
      x[i] = (1.0f - pe[i]) * x[i];
      l = fmaf(pe[i], l, x[i]);
      prod *= pe[i];
      opaque(x[i]);
      fence(i);
    }
    sl[idx][lc] = l;
    sp[idx][lc] = prod;
    __syncthreads();
    l = enter<NC, LC, false>(Lc, sl, sp, 0.0f, idx, lc, live);
    if (ckpt && ok && mine) keep(seg, l, Es, Rs);
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      l = fmaf(pe[i], l, x[i]);
      orow.store(i, from_f<E>(l));
    }
  }
  if (tail && wave == 0) {  // the last, shorter chunk: one wave walks it
    if (ckpt && ok && sub == 0) keep(nfull, Lc, Ec, Rc);
    const size_t base = static_cast<size_t>(nfull) * CK * H;
    const Rows<E, BIG> wr(wb + base, H, h, tail, sub * CK), pr(pb + base, H, h, tail, sub * CK),
        orow(ob + base, H, h, tail, sub * CK);  // past the rows where sub > 0
    for (int i0 = 0; i0 < tail; i0 += TB) {
      E wv[TB], pv[TB];
#pragma unroll
      for (int i = 0; i < TB; ++i) {  // at clamped rows, all in flight at once
        wv[i] = wr.load(min(i0 + i, tail - 1));
        pv[i] = pr.load(min(i0 + i, tail - 1));
      }
#pragma unroll
      for (int i = 0; i < TB; ++i)
        if (i0 + i < tail) {
          const float wt = to_f(wv[i]), pe = tanh_abs(fabsf(wt - Ec));
          Ec = step_E(k, Ec, wt);
          Rc = step_R(k, Rc, pe);
          const float eff = retention(k, Rc);
          Lc = fmaf(eff, Lc, (1.0f - eff) * ((to_f(pv[i]) * pe) * wt));
          orow.store(i0 + i, from_f<E>(Lc));
        }
    }
  }
  if (idx == 0 && ok) {
    LF[ch] = Lc;
    EF[ch] = Ec;
    RF[ch] = Rc;
  }
}

// A few steps (streaming decode, T <= kSingle): one thread per channel walks them from the
// given initial state. The checkpoint (if given) of the one chunk is the initial state.
constexpr int kSingle = 4;
template <typename E>
__global__ void __launch_bounds__(NT) long_fwd_single(int B, int T, int H, int64_t ldx,
                                                      const E* w, const E* p, Logits lg,
                                                      const float* L0, const float* E0,
                                                      const float* R0, E* out, float* LF,
                                                      float* EF, float* RF, float* ckpt) {
  const int64_t ch = static_cast<int64_t>(blockIdx.x) * NT + threadIdx.x;
  if (ch >= static_cast<int64_t>(B) * H) return;
  const Coef k = load_coef(lg.p);
  const int b = static_cast<int>(ch / H), h = static_cast<int>(ch % H);
  const size_t base = static_cast<size_t>(b) * T * H + h;
  const size_t ibase = static_cast<size_t>(b) * ldx + h;
  float L = L0[ch], Ev = E0[ch], R = R0[ch];
  if (ckpt) {
    float* cp = ckpt + static_cast<size_t>(b) * 3 * H + h;
    cp[0] = L;
    cp[H] = Ev;
    cp[2 * H] = R;
  }
  for (int t = 0; t < T; ++t) {
    const size_t o = base + static_cast<size_t>(t) * H, io = ibase + static_cast<size_t>(t) * H;
    const float wt = ld(w, io), pt = ld(p, io);
    const float pe = tanh_abs(fabsf(wt - Ev));
    Ev = step_E(k, Ev, wt);
    R = step_R(k, R, pe);
    const float eff = retention(k, R);
    L = fmaf(eff, L, (1.0f - eff) * ((pt * pe) * wt));
    st(out, o, L);
  }
  LF[ch] = L;
  EF[ch] = Ev;
  RF[ch] = R;
}

// Backward. Walking time in reverse with g_t the output's gradient and x_t = sal_t w_t:
//   gL_t  = g_t + eff_{t+1} gL_{t+1}             (total adjoint of L_t)
//   deff  = gL_t (L_{t-1} - x_t),  dsal = gL_t (1 - eff_t) w_t
//   dR_t  = rd dR_{t+1} + deff (1-ret) rs
//   dpe   = dsal p_t - (1-rd) dR_t,  darg = dpe (1 - pe^2) sign(w_t - E_{t-1})
//   dE_t  = er dE_{t+1} - darg_{t+1}
//   gw_t  = gL_t (1 - eff_t) sal_t + darg + (1-er) dE_t,   gp_t = dsal pe
// three chained recurrences again, with the coefficients eff_t, rd and er. Writes gw, gp (batch
// rows ldo apart) and one partial of the four logit gradients per workgroup (fixed order).
// ACC: gw += the gradient rounded to E, the sum formed in fp32 and rounded once (an add of
// the rounded gradient into an existing gradient buffer).
// The wave keeps 7 values per step (w and p of bf16 in one register): at most 256 registers,
// 8 waves per CU; the 4-wave workgroups of fp32 and of the 16-channel split (one per CU) may use
// twice as many, and spill nothing (B=1, T=4096, H=64 bf16: 89 -> 80 us).
template <typename E>
struct Pair {  // w and p of one step
  E w, p;
  __device__ __forceinline__ void set(E a, E b) {
    w = a;
    p = b;
  }
  __device__ __forceinline__ float fw() const { return to_f(w); }
  __device__ __forceinline__ float fp() const { return to_f(p); }
  __device__ __forceinline__ void opaque_() {
    opaque(w);
    opaque(p);
  }
};
template <>
struct Pair<bf16> {
  uint32_t v;
  __device__ __forceinline__ void set(bf16 a, bf16 b) { v = static_cast<uint32_t>(a) << 16 | b; }
  __device__ __forceinline__ float fw() const { return __builtin_bit_cast(float, v & 0xffff0000u); }
  __device__ __forceinline__ float fp() const { return __builtin_bit_cast(float, v << 16); }
  __device__ __forceinline__ void opaque_() { opaque(v); }
};

// The upstream gradient of one step and (KEEP) the value its write gradient is added to.
template <typename E, bool KEEP>
struct Grads {
  E g;
  __device__ __forceinline__ float up() const { return to_f(g); }
  __device__ __forceinline__ void opaque_() { opaque(g); }
};
template <typename E>
struct Grads<E, true> {
  Pair<E> v;
  __device__ __forceinline__ float up() const { return v.fp(); }
  __device__ __forceinline__ void opaque_() { v.opaque_(); }
};

template <typename E, bool ACC, int NW, int G, bool BIG>
__global__ void __launch_bounds__(NW* LANES, is_bf16<E>::value && G == 1 ? 2 : 1)
    long_bwd_kernel(int T, int H, int64_t ldx, int64_t ldw, int64_t ldo, const E* __restrict__ w,
                    const E* __restrict__ p, Logits lg, const float* __restrict__ ckpt,
                    const E* __restrict__ gout, const float* __restrict__ gLF,
                    const float* __restrict__ gRF, const float* __restrict__ gEF,
                    E* __restrict__ gw, E* __restrict__ gp, float* __restrict__ gL0,
                    float* __restrict__ gR0, float* __restrict__ gE0, float* __restrict__ part) {
  constexpr int NC = NW * G, LC = LANES / G;
  __shared__ float sl[NC][LC], sp[NC][LC], sr[NC][LC], se[NC][LC];
  __shared__ float red[4][NW];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int lc = lane % LC, sub = lane / LC, idx = wave * G + sub;
  const int h = blockIdx.x * LC + lc, b = blockIdx.y;
  const bool ok = h < H;
  const int hc = ok ? h : H - 1;
  const Coef k = load_coef(lg.p);
  const float er_full = powi(k.er, CK), rd_full = powi(k.rd, CK);
  const float kap = (1.0f - k.ret) * k.rs;
  const size_t ch = static_cast<size_t>(b) * H + hc;
  float gLc = gLF ? gLF[ch] : 0.0f, gRc = gRF ? gRF[ch] : 0.0f, gEc = gEF ? gEF[ch] : 0.0f;
  E* wb = const_cast<E*>(w) + static_cast<size_t>(b) * ldx;
  E* pb = const_cast<E*>(p) + static_cast<size_t>(b) * ldx;
  E* gb = const_cast<E*>(gout) + static_cast<size_t>(b) * T * H;
  E* gwb = gw + static_cast<size_t>(b) * ldw;
  E* gpb = gp + static_cast<size_t>(b) * ldo;
  const int nseg = (T + CK - 1) / CK, nfull = T / CK, tail = T % CK;
  float t_er = 0.f, t_rd = 0.f, t_ret = 0.f, t_rs = 0.f;
  auto block = [&](auto full, int k0, int live) {  // as the forward's
    const int seg = k0 + idx;
    const bool mine = idx < live;
    const int wlive = min(max(live - wave * G, 0), G);          // chunks of this wave,
    const int len = wlive == 0 ? 0 : full ? CK * wlive : tail;  // and their steps
    const float er_pow = full ? er_full : powi(k.er, tail);
    const float rd_pow = full ? rd_full : powi(k.rd, tail);
    const size_t base = static_cast<size_t>(wlive > 0 ? k0 + wave * G : 0) * CK * H;
    const int first = sub * CK;
    const Rows<E, BIG> wr(wb + base, H, h, len, first), pr(pb + base, H, h, len, first),
        grow(gb + base, H, h, len, first), gwr(gwb + base, H, h, len, first),
        gpr(gpb + base, H, h, len, first);
    constexpr bool KEEP = ACC && !(is_bf16<E>::value && G == 1);
    Pair<E> wp[CK];
    Grads<E, KEEP> gr[CK];
#pragma unroll
    for (int i = 0; i < CK; ++i) {
      const int j = full && !BIG ? i : min(i, max(len - 1, 0));
      wp[i].set(wr.load(j), pr.load(j));
      if constexpr (KEEP)
        gr[i].v.set(gwr.load(j), grow.load(j));
      else
        gr[i].g = grow.load(j);
    }
    __builtin_amdgcn_sched_barrier(0);
    const float* c = ckpt + (static_cast<size_t>(b) * nseg + (mine ? seg : 0)) * 3 * H;
    float L = c[hc], Ev = (c + H)[hc];
    const float Rs = (c + 2 * static_cast<size_t>(H))[hc];
    // Replay: per step the difference, pe, a = L - x and R after the step; and, walking back,
    // the chunk's gL from zero with its product of eff.
    float diff[CK], pe[CK], a[CK], R[CK], g[CK];
    float l = 0.0f, prod = 1.0f;
    auto forget = [&] {
#pragma unroll
      for (int i = 0; i < CK; ++i) {
        wp[i].opaque_();
        opaque(R[i]);
        gr[i].opaque_();
      }
    };
    float r = Rs;
#pragma unroll
      for (int i = 0; i < CK; ++i)
        if (full || i < tail) {
          const float wt = wp[i].fw();
          diff[i] = wt - Ev;
          pe[i] = tanh_abs(fabsf(diff[i]));
          Ev = step_E(k, Ev, wt);
          r = step_R(k, r, pe[i]);
          R[i] = r;
          const float x = (wp[i].fp() * pe[i]) * wt, eff = retention(k, r);
          a[i] = L - x;
          L = fmaf(eff, L, (1.0f - eff) * x);
          opaque(diff[i]);
          opaque(pe[i]);
          opaque(a[i]);
          opaque(R[i]);
          wp[i].opaque_();
          fence(i);
        }
#pragma unroll
    for (int i = CK - 1; i >= 0; --i)
        if (full || i < tail) {
          const float eff = retention(k, R[i]);
          l = eff * (l + gr[i].up());
          prod *= eff;
          fence(i);
        }
    forget();
    sl[idx][lc] = l;
    sp[idx][lc] = prod;
    __syncthreads();
    l = enter<NC, LC, true>(gLc, sl, sp, 0.0f, idx, lc, live);
    // gL of every step (in g), deff (in a), the chunk's gR from zero.
    r = 0.0f;
#pragma unroll
    for (int i = CK - 1; i >= 0; --i)
        if (full || i < tail) {
          g[i] = l + gr[i].up();
          l = g[i] * retention(k, R[i]);
          a[i] = g[i] * a[i];
          r = fmaf(a[i], kap, r) * k.rd;
          opaque(g[i]);
          opaque(a[i]);
          fence(i);
        }
    forget();
    sr[idx][lc] = r;
    __syncthreads();
    r = enter<NC, LC, true>(gRc, sr, nullptr, rd_pow, idx, lc, live);
    // gp; darg (in pe) and the rest of gw (in g); the chunk's gE from zero.
    float e = 0.0f, d_er = 0.f, d_rd = 0.f, d_ret = 0.f, d_rs = 0.f;
#pragma unroll
    for (int i = CK - 1; i >= 0; --i)
        if (full || i < tail) {
          const float wt = wp[i].fw(), pt = wp[i].fp(), pi = pe[i];
          const float gx = g[i] * (1.0f - retention(k, R[i]));  // gradient of x
          const float dsal = gx * wt;
          const float dR = fmaf(a[i], kap, r);
          r = dR * k.rd;
          const float dpe = fmaf(dsal, pt, -(dR * (1.0f - k.rd)));
          const float m = dpe * fmaf(-pi, pi, 1.0f);
          const float darg = diff[i] == 0.0f ? 0.0f : copysignf(1.0f, diff[i]) * m;
          d_rd = fmaf(dR, (i > 0 ? R[i - 1] : Rs) - (1.0f - pi), d_rd);
          d_ret = fmaf(a[i], fmaf(-k.rs, R[i], 1.0f), d_ret);
          d_rs = fmaf(a[i], R[i], d_rs);
          e = fmaf(k.er, e, -darg);
          g[i] = fmaf(gx, pt * pi, darg);
          pe[i] = darg;
          opaque(g[i]);
          opaque(pe[i]);
          gpr.store(i, from_f<E>(dsal * pi));
          if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        }
    // ACC: the values added to. With registers to spare (KEEP) they came with the inputs; else in
    // groups of 8 rows, a group ahead of the stores of the one before it (all 32 at once spill).
    constexpr int SG = 8;
    constexpr bool LATE = ACC && !KEEP;
    E sv[2][SG];
    auto load_into = [&](int g0, E(&dst)[SG]) {
      if constexpr (LATE) {
#pragma unroll
        for (int i = 0; i < SG; ++i)
          dst[i] = gwr.load(full && !BIG ? g0 + i : min(g0 + i, max(len - 1, 0)));
      }
    };
    load_into(CK - SG, sv[0]);
    se[idx][lc] = e;
    __syncthreads();
    e = enter<NC, LC, true>(gEc, se, nullptr, er_pow, idx, lc, live);
#pragma unroll
    for (int q = 0; q < CK / SG; ++q) {
      const int g0 = CK - SG * (q + 1);
      if (LATE && g0 > 0) load_into(g0 - SG, sv[(q + 1) & 1]);
      if constexpr (LATE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = g0 + SG - 1; i >= g0; --i)
        if (full || i < tail) {
          float v = fmaf(1.0f - k.er, e, g[i]);
          if constexpr (KEEP) v = gr[i].v.fw() + round_to<E>(v);
          if constexpr (LATE) v = to_f(sv[q & 1][i - g0]) + round_to<E>(v);
          d_er = fmaf(-e, diff[i], d_er);
          e = fmaf(k.er, e, -pe[i]);
          gwr.store(i, from_f<E>(v));
        }
      if constexpr (LATE) __builtin_amdgcn_sched_barrier(0);
    }
    t_er += mine ? d_er : 0.0f;
    t_rd += mine ? d_rd : 0.0f;
    t_ret += mine ? d_ret : 0.0f;
    t_rs += mine ? d_rs : 0.0f;
  };
  if (tail) block(std::false_type{}, nfull, 1);
  for (int k0 = nfull > 0 ? (nfull - 1) / NC * NC : -1; k0 >= 0; k0 -= NC)
    block(std::true_type{}, k0, min(NC, nfull - k0));
  if (idx == 0 && ok) {
    gL0[ch] = gLc;
    gR0[ch] = gRc;
    gE0[ch] = gEc;
  }
  // d logit = d coef * sigmoid'(logit), reduced per workgroup in a fixed order.
  const float d[4] = {t_er * k.er * (1.0f - k.er), t_rd * k.rd * (1.0f - k.rd),
                      t_ret * k.ret * (1.0f - k.ret),
                      t_rs * (1.0f - k.ret) * k.rs * (1.0f - k.rs)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float sum = wave_sum(ok ? d[i] : 0.0f);
    if (lane == 0) red[i][wave] = sum;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    float sum = 0.0f;
    for (int i = 0; i < NW; ++i) sum += red[threadIdx.x][i];
    part[(static_cast<size_t>(b) * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = sum;
  }
}

// gw[b][i] += g[b][i], the sum formed in fp32 and rounded once (see the backward's launcher).
template <typename E>
__global__ void __launch_bounds__(256) long_add_kernel(int64_t n, int64_t ldw, const E* __restrict__ g,
                                                       E* __restrict__ gw) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  E* o = gw + blockIdx.y * ldw + i;
  *o = from_f<E>(to_f(*o) + to_f(g[blockIdx.y * n + i]));
}

static int grid_for(int64_t B, int64_t H) { return static_cast<int>((B * H + NT - 1) / NT); }

}  // namespace longmem
}  // namespace dabsn

using namespace dabsn;
using namespace dabsn::longmem;

#define DABSN_SHAPE_CHECK(B, T, H)                                                             \
  DABSN_REQUIRE((B) > 0 && (T) >= 0 && (H) > 0 && (B) * (T) * (H) < (1ll << 46) &&          \
                    (B) * (H) < (1ll << 31) && (T) < (1ll << 30),                            \
                "bad shape B=%lld T=%lld H=%lld", (long long)(B), (long long)(T), (long long)(H))

constexpr int kBigRow = 1 << 24;  // see Rows

constexpr int64_t kMaxChunks = 65536;  // longer sequences are refused: checked up to 2^17 steps

// Batch rows lie in gridDim.y, which holds 65,535: larger batches (of few, narrow channels) run
// as launches of that many rows each.
constexpr int64_t kSlab = 65535;
template <typename P>
static P* row_ptr(P* p, int64_t b0, int64_t stride) {
  return p ? p + b0 * stride : p;
}

// Chunks per wave. A workgroup of 64 channels walks T serially, so few channels leave most CUs
// idle: up to kFew such workgroups a wave takes 4 chunks of 16 channels instead, 4 times the
// workgroups and a quarter of the blocks (at accesses of 32 bytes, which so few channels can
// afford). Backward, bf16: B=1, T=4096, H=64 takes 184 us with 64 channels and 80 with 16 (the
// earlier kernels, parallel over all chunks of T: 74; forward 140 against 68); B=8, T=2573, H=400
// (56 workgroups) 134 and 86 (114); B=32, T=3200, H=256 (128 workgroups) 174 and 187 (215).
constexpr int64_t kFew = 64;
static int wave_chunks(int64_t B, int64_t T, int64_t H) {
  return B * ((H + LANES - 1) / LANES) <= kFew && T >= 4 * CK ? 4 : 1;
}
static int channel_tiles(int64_t B, int64_t T, int64_t H) {
  const int lc = LANES / wave_chunks(B, T, H);
  return static_cast<int>((H + lc - 1) / lc);
}

// Waves per workgroup: as many as there are chunks, up to 8 in the forward (two workgroups per
// CU, one's arithmetic over the other's loads) and 4 in the backward (the same at its 256
// registers; one workgroup of 8 waves took 512 us for the shape below). In the bf16 backward 8
// where every CU has at most one workgroup anyway: B=32, T=3200, H=256 229 -> 175 us.
// B=16, T=4096, H=2048 bf16: 637 -> 230 us (805 MB: 3.5 TB/s).
template <typename E>
static int long_fwd_impl(int B, int T, int H, int64_t ldx, const E* w, const E* p, Logits lg,
                         const float* L0, const float* E0, const float* R0, E* out, float* LF,
                         float* EF, float* RF, float* keep, hipStream_t stream) {
  if (T > 0 && T <= kSingle) {
    hipLaunchKernelGGL((long_fwd_single<E>), dim3(grid_for(B, H)), dim3(NT), 0, stream, B, T, H, ldx,
                       w, p, lg, L0, E0, R0, out, LF, EF, RF, keep);
    DABSN_HIP_CHECK(hipGetLastError());
    return DABSN_OK;
  }
  const int nseg = (T + CK - 1) / CK;
  const bool split = wave_chunks(B, T, H) == 4;
  const int64_t n = static_cast<int64_t>(T) * H;
  for (int64_t b0 = 0; b0 < B; b0 += kSlab) {
    const dim3 grid(channel_tiles(B, T, H), static_cast<unsigned>(std::min(kSlab, B - b0)));
    const int64_t r = b0 * H;
#define DABSN_LONG(NW, G, BIG)                                                               \
  hipLaunchKernelGGL((long_fwd_kernel<E, NW, G, BIG>), grid, dim3(NW * LANES), 0, stream, T, H, ldx, \
                     w + b0 * ldx, p + b0 * ldx, lg, L0 + r, E0 + r, R0 + r, out + b0 * n, LF + r,  \
                     EF + r, RF + r, row_ptr(keep, b0, 3ll * nseg * H))
    if (H >= kBigRow)
      DABSN_LONG(4, 1, true);
    else if (split && nseg <= 16)
      DABSN_LONG(4, 4, false);
    else if (split)
      DABSN_LONG(8, 4, false);
    else if (nseg <= 1)
      DABSN_LONG(1, 1, false);
    else if (nseg <= 2)
      DABSN_LONG(2, 1, false);
    else if (nseg <= 4)
      DABSN_LONG(4, 1, false);
    else
      DABSN_LONG(8, 1, false);
#undef DABSN_LONG
  }
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

// B=16, T=4096, H=2048 bf16: 891 -> 425 us (1.39 GB: 3.3 TB/s); accumulating, on half of the CUs
// and T=768, 307 -> 177.
//
// ACC with 16-channel tiles: a 128-byte line of gw then belongs to several workgroups, on several
// XCDs, and reading lines that another XCD writes stalls each block (B=1, T=4096, H=64 bf16: 235
// us against 80 without ACC). So the split scan writes its gradient to the workspace `ws`, whole,
// and another kernel adds it.
template <typename E, bool ACC>
static int long_bwd_impl(int B, int T, int H, int64_t ldx, const E* w, const E* p, Logits lg,
                         const float* ckpt, const E* gout, const float* gLF, const float* gEF,
                         const float* gRF, E* gw, int64_t ldw, E* gp, int64_t ldo, float* gL0,
                         float* gE0, float* gR0, float* part, E* ws, hipStream_t stream) {
  const bool split = wave_chunks(B, T, H) == 4;
  const int64_t n = static_cast<int64_t>(T) * H;
  if constexpr (ACC) {
    if (split && ws) {
      const int rc = long_bwd_impl<E, false>(B, T, H, ldx, w, p, lg, ckpt, gout, gLF, gEF, gRF, ws, n,
                                             gp, ldo, gL0, gE0, gR0, part, nullptr, stream);
      if (rc != DABSN_OK) return rc;
      hipLaunchKernelGGL(long_add_kernel<E>, dim3(static_cast<unsigned>((n + 255) / 256), B), dim3(256),
                         0, stream, n, ldw, ws, gw);
      DABSN_HIP_CHECK(hipGetLastError());
      return DABSN_OK;
    }
  }
  const int nseg = (T + CK - 1) / CK, tiles = channel_tiles(B, T, H);
  for (int64_t b0 = 0; b0 < B; b0 += kSlab) {
    const dim3 grid(tiles, static_cast<unsigned>(std::min(kSlab, B - b0)));
    const int64_t r = b0 * H;
#define DABSN_LONG(NW, G, BIG)                                                                  \
  hipLaunchKernelGGL((long_bwd_kernel<E, ACC, NW, G, BIG>), grid, dim3(NW * LANES), 0, stream, T, H, \
                     ldx, ldw, ldo, w + b0 * ldx, p + b0 * ldx, lg, row_ptr(ckpt, b0, 3ll * nseg * H), \
                     row_ptr(gout, b0, n), row_ptr(gLF, b0, H), row_ptr(gRF, b0, H),                  \
                     row_ptr(gEF, b0, H), row_ptr(gw, b0, ldw), row_ptr(gp, b0, ldo), gL0 + r, gR0 + r, \
                     gE0 + r, part + 4 * b0 * tiles)
    if (H >= kBigRow)
      DABSN_LONG(4, 1, true);
    else if (split)
      DABSN_LONG(4, 4, false);
    else if (nseg <= 1)
      DABSN_LONG(1, 1, false);
    else if (nseg <= 2)
      DABSN_LONG(2, 1, false);
    else if (nseg <= 4 || static_cast<int64_t>(tiles) * B > 256 || !is_bf16<E>::value)
      DABSN_LONG(4, 1, false);
    else if constexpr (is_bf16<E>::value)
      DABSN_LONG(8, 1, false);
#undef DABSN_LONG
  }
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

extern "C" {

int dabsn_hip_linrec_fwd(int dtype, int64_t B, int64_t T, int64_t H, const void* a, const void* g,
                         const void* y0, void* y, hipStream_t stream) {
  DABSN_SHAPE_CHECK(B, T, H);
  DABSN_REQUIRE(a && g && y0 && (y || T == 0), "linrec: null pointer");
  if (T == 0) return DABSN_OK;
  const int grid = grid_for(B, H);
  if (dtype == kBF16)
    hipLaunchKernelGGL(linrec_fwd_kernel<bf16>, dim3(grid), dim3(NT), 0, stream, (int)B, (int)T,
                       (int)H, (const bf16*)a, (const bf16*)g, (const bf16*)y0, (bf16*)y);
  else if (dtype == kF32)
    hipLaunchKernelGGL(linrec_fwd_kernel<float>, dim3(grid), dim3(NT), 0, stream, (int)B, (int)T,
                       (int)H, (const float*)a, (const float*)g, (const float*)y0, (float*)y);
  else
    DABSN_REQUIRE(false, "linrec: bad dtype %d", dtype);
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

size_t dabsn_hip_linrec_workspace_bytes(int dtype, int64_t B, int64_t T, int64_t H) {
  (void)dtype;
  return static_cast<size_t>(B) * T * H * sizeof(float);
}

int dabsn_hip_linrec_bwd(int dtype, int64_t B, int64_t T, int64_t H, const void* a, const void* g,
                         const void* y0, const void* gy, void* da, void* dg, void* dy0,
                         void* workspace, size_t workspace_bytes, hipStream_t stream) {
  DABSN_SHAPE_CHECK(B, T, H);
  DABSN_REQUIRE(a && g && y0 && gy && da && dg && dy0, "linrec backward: null pointer");
  DABSN_REQUIRE(workspace_bytes >= dabsn_hip_linrec_workspace_bytes(dtype, B, T, H),
                "linrec backward: workspace too small");
  const int grid = grid_for(B, H);
  if (dtype == kBF16)
    hipLaunchKernelGGL(linrec_bwd_kernel<bf16>, dim3(grid), dim3(NT), 0, stream, (int)B, (int)T,
                       (int)H, (const bf16*)a, (const bf16*)g, (const bf16*)y0, (const bf16*)gy,
                       (bf16*)da, (bf16*)dg, (bf16*)dy0, (float*)workspace);
  else if (dtype == kF32)
    hipLaunchKernelGGL(linrec_bwd_kernel<float>, dim3(grid), dim3(NT), 0, stream, (int)B, (int)T,
                       (int)H, (const float*)a, (const float*)g, (const float*)y0,
                       (const float*)gy, (float*)da, (float*)dg, (float*)dy0, (float*)workspace);
  else
    DABSN_REQUIRE(false, "linrec backward: bad dtype %d", dtype);
  DABSN_HIP_CHECK(hipGetLastError());
  return DABSN_OK;
}

// Only the accumulating backward (bit 2 of `backward`) of few channels keeps anything outside its
// registers and LDS: the gradient it adds.
size_t dabsn_hip_long_workspace_bytes(int64_t B, int64_t T, int64_t H, int backward) {
  if (!(backward & 2) || B <= 0 || T <= 0 || H <= 0 || wave_chunks(B, T, H) != 4) return 0;
  return static_cast<size_t>(B) * T * H * sizeof(float);
}

// Batch stride of [B, T, H] operands: ldx elements (0: T H, the contiguous layout); at least
// T H, so a time window of longer [B, T', H] tapes can be passed in place; -1 if invalid.
static int64_t batch_stride(int64_t B, int64_t T, int64_t H, int64_t ldx) {
  if (ldx == 0) return T * H;
  if (ldx < T * H || (B - 1) * ldx + T * H >= (1ll << 46)) return -1;
  return ldx;
}

int dabsn_hip_long_fwd(int dtype, int64_t B, int64_t T, int64_t H, int64_t ldx, const void* w,
                       const void* p, const float* const* logits, const float* L0,
                       const float* E0, const float* R0, void* out, float* LF, float* EF,
                       float* RF, float* ckpt, void* workspace, size_t workspace_bytes,
                       hipStream_t stream) {
  DABSN_SHAPE_CHECK(B, T, H);
  const int64_t lx = batch_stride(B, T, H, ldx);
  DABSN_REQUIRE(lx >= 0, "long scan: bad input batch stride %lld for T=%lld H=%lld",
                (long long)ldx, (long long)T, (long long)H);
  DABSN_REQUIRE(w && p && logits && L0 && E0 && R0 && (out || T == 0) && LF && EF && RF,
                "long scan: null pointer");
  (void)workspace;
  (void)workspace_bytes;
  for (int i = 0; i < 4; ++i) DABSN_REQUIRE(logits[i], "long scan: null logit %d", i);
  DABSN_REQUIRE((T + CK - 1) / CK < kMaxChunks, "long scan: T too long");
  Logits lg{{logits[0], logits[1], logits[2], logits[3]}};
  if (dtype == kBF16)
    return long_fwd_impl<bf16>((int)B, (int)T, (int)H, lx, (const bf16*)w, (const bf16*)p, lg,
                               L0, E0, R0, (bf16*)out, LF, EF, RF, ckpt, stream);
  if (dtype == kF32)
    return long_fwd_impl<float>((int)B, (int)T, (int)H, lx, (const float*)w, (const float*)p, lg,
                                L0, E0, R0, (float*)out, LF, EF, RF, ckpt, stream);
  DABSN_REQUIRE(false, "long scan: bad dtype %d", dtype);
  return DABSN_OK;
}

int64_t dabsn_hip_long_partials(int64_t B, int64_t T, int64_t H) { return B * channel_tiles(B, T, H); }

int dabsn_hip_long_bwd(int dtype, int64_t B, int64_t T, int64_t H, int64_t ldx, const void* w,
                       const void* p, const float* const* logits, const float* ckpt,
                       const void* gout, const float* gLF, const float* gEF, const float* gRF,
                       void* gw, void* gp, int64_t ldo, int gw_accumulate, float* gL0,
                       float* gE0, float* gR0, float* part_logit, void* workspace,
                       size_t workspace_bytes, hipStream_t stream) {
  DABSN_SHAPE_CHECK(B, T, H);
  const int64_t lx = batch_stride(B, T, H, ldx), lo = batch_stride(B, T, H, ldo);
  DABSN_REQUIRE(lx >= 0 && lo >= 0,
                "long scan backward: bad batch stride (inputs %lld, outputs %lld) for T=%lld "
                "H=%lld", (long long)ldx, (long long)ldo, (long long)T, (long long)H);
  DABSN_REQUIRE(w && p && logits && (ckpt || T == 0) && (gout || T == 0) && gL0 && gE0 && gR0 &&
                    part_logit && ((gw && gp) || T == 0),
                "long scan backward: null pointer");
  for (int i = 0; i < 4; ++i) DABSN_REQUIRE(logits[i], "long scan backward: null logit %d", i);
  DABSN_REQUIRE((T + CK - 1) / CK < kMaxChunks, "long scan backward: T too long");
  Logits lg{{logits[0], logits[1], logits[2], logits[3]}};
#define DABSN_LONG_BWD(E, ACC)                                                                 \
  return long_bwd_impl<E, ACC>((int)B, (int)T, (int)H, lx, (const E*)w, (const E*)p, lg, ckpt,   \
                               (const E*)gout, gLF, gEF, gRF, (E*)gw, lo, (E*)gp, lo, gL0, gE0, \
                               gR0, part_logit, workspace && workspace_bytes >= B * T * H * sizeof(E) \
                               ? static_cast<E*>(workspace) : nullptr, stream)
  if (dtype == kBF16) {
    if (gw_accumulate) DABSN_LONG_BWD(bf16, true);
    DABSN_LONG_BWD(bf16, false);
  }
  if (dtype == kF32) {
    if (gw_accumulate) DABSN_LONG_BWD(float, true);
    DABSN_LONG_BWD(float, false);
  }
#undef DABSN_LONG_BWD
  DABSN_REQUIRE(false, "long scan backward: bad dtype %d", dtype);
  return DABSN_OK;
}

}  // extern "C"
