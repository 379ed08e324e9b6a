// The reference's own selective scan (mamformer/layers/mamba2.py:70-130) for gfx950: a decay rate per state
// column and a step size per channel,
//     h_t[c, n] = exp(A_n dt_t[c]) h_{t-1}[c, n] + dt_t[c] x_t[c] B_t[n],   y_t[c] = sum_n C_t[n] h_t[c, n] + D_c x_t[c]
// with A_n = -exp(clamp(A_log_n, -5, 5)), formed here or by the caller.  The decay differs per (channel, state), so the
// recurrence has no matrix-unit factorisation (the per-head SSD form does): every (token, channel, state) costs
// one exponential and a few fused multiply-adds, and the kernels are bound by that VALU work.
//
// rf_scan_kernel, one workgroup per (batch, block of channels), walking the whole sequence:
//   LPC = 32 lanes per channel (16 for N = 16), each owning N / 32 consecutive states, so the sum over states
//   that forms y runs on the DPP crossbar (quad permutes, the row mirrors, then the row-15 broadcast that adds
//   the two rows of a channel); a wave holds 2 channels, a workgroup of 4 waves 8.  Blocks of TB tokens of B, C
//   (fp32), dt, x and the gate are staged in LDS (two stages; the next block's rows are loaded into registers
//   while the current block computes, and each token's LDS values are read two tokens ahead), y is collected per
//   block in LDS and stored as rows of the workgroup's channels.  A wave has its SIMD to itself, so what it waits
//   for nobody fills: with the reads one token ahead and softplus on one wave of four, b1 L2048 d_inner 2048 N 128
//   took 231 us, now 171.
// rf_hs_kernel (h_states, the per-token mean of the state over all channels, mamba2.py:114-116):
//   lane = channel (256 channels per workgroup), a workgroup per (batch, channel block, group of 4 states), so
//   that the sum over channels is a reduce-scatter inside the wave (v_permlane32_swap, v_permlane16_swap, then the
//   DPP row sums) plus a sum over the 4 waves; the per-block sums go to a workspace and rf_hs_reduce_kernel adds
//   them in a fixed order (deterministic).
#include <algorithm>

#include "common.h"
#include "launch.h"
#include "ssd_shared.h"

namespace mh {

namespace {

constexpr int RF_NT = 256;           // threads per workgroup (both kernels)
constexpr int HS_CPB = 256;          // channels per workgroup of h_states
constexpr int HS_NS = 4;             // states per thread of h_states
constexpr int HS_TB = 16;            // tokens per block of h_states
constexpr float LOG2E = 1.4426950408889634f;

// Lanes per channel of the scan, states per lane, channels per workgroup, tokens per LDS block.
template <int N> constexpr int rf_lpc() { return N >= 32 ? 32 : 16; }
template <int N> constexpr int rf_ns() { return N / rf_lpc<N>(); }
template <int N> constexpr int rf_cpb() { return 4 * (64 / rf_lpc<N>()); }
template <int N> constexpr int rf_tb() { return N <= 128 ? 32 : 16; }
constexpr int RF_RK = 16;            // tokens per piece of the backward (the checkpoint spacing)
constexpr int RF_HK = 8;             // tokens whose states and decays the gradient kernel holds in registers at once
constexpr int RF_CH = 64;            // channels per workgroup of the gradient kernel

// The decay rate of state n: A as given, or -exp(clamp(A_log, -5, 5)) (mamba2.py:87-88; a NaN stays one).
__device__ __forceinline__ float rf_rate(const RfParams& p, int n) {
  const float a = p.A[n];
  if (!p.A_log) return a;
  return -expf(a < -5.f ? -5.f : a > 5.f ? 5.f : a);
}

// Per-lane token prologue: dt <- clamp(softplus?(dt + bias), dt_min, dt_max).
__device__ __forceinline__ float rf_dt(const RfParams& p, float raw, float bias) {
  float d = raw + bias;
  if (p.dt_softplus) d = softplus_f(d);
  if (p.has_dt_limit) d = fminf(fmaxf(d, p.dt_min), p.dt_max);
  return d;
}

// Sum over each 16-lane row, in every lane of the row: quad permutes, then the half-row and row mirrors.
__device__ __forceinline__ float row_sum16(float v) {
  v += dppf<0xB1>(v);      // quad_perm 1,0,3,2
  v += dppf<0x4E>(v);      // quad_perm 2,3,0,1
  v += dppf<0x141>(v);     // row_half_mirror
  v += dppf<0x140>(v);     // row_mirror
  return v;
}

// Lane-crossing moves within 16-lane rows (DPP): the value of lane l ^ 8, ^ 4, ^ 2, ^ 1 of the same row.
__device__ __forceinline__ float xor8(float v) { return dppf<0x128>(v); }       // row_ror:8
__device__ __forceinline__ float xor4(float v) {
  // lanes 4-7 and 12-15 (banks 1, 3) read lane l - 4, lanes 0-3 and 8-11 (banks 0, 2) lane l + 4
  const int a = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xa, false);   // row_shr:4
  return __int_as_float(__builtin_amdgcn_update_dpp(a, __float_as_int(v), 0x104, 0xf, 0x5, false));   // row_shl:4
}
__device__ __forceinline__ float xor2(float v) { return dppf<0x4E>(v); }        // quad_perm 2,3,0,1
__device__ __forceinline__ float xor1(float v) { return dppf<0xB1>(v); }        // quad_perm 1,0,3,2

// One step of the reduce-scatter below: the lanes with lane bit M set keep the upper half of their first K
// values and hand the lower half to the partner l ^ M, which keeps its lower half.
template <int M, int K, int NV>
__device__ __forceinline__ void rf_rs_step(float (&v)[NV], int l) {
  const bool up = (l & M) != 0;
#pragma unroll
  for (int k = 0; k < K / 2; ++k) {
    const float keep = up ? v[k + K / 2] : v[k], send = up ? v[k] : v[k + K / 2];
    float r;
    if constexpr (M == 8) r = xor8(send);
    else if constexpr (M == 4) r = xor4(send);
    else if constexpr (M == 2) r = xor2(send);
    else r = xor1(send);
    v[k] = keep + r;
  }
}

// Sums of v[t] (t < 32) over the 32 lanes of a channel (lanes 32 c .. 32 c + 31, two 16-lane rows), lane g of
// the channel ending with the sum for t = g: one exchange-and-add per value pair and step, 31 for 32 tokens,
// where a separate row sum per token took five dependent DPP additions.
__device__ __forceinline__ float rf_reduce_scatter32(float (&v)[32], int l) {
  // lane bit 16: v_permlane16_swap trades the odd rows of its first operand with the even rows of its second,
  // so row 0 of the channel ends with v[k] of both rows and row 1 with v[k + 16] of both
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[k]), __float_as_uint(v[k + 16]), false, false);
    v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  rf_rs_step<8, 16>(v, l);
  rf_rs_step<4, 8>(v, l);
  rf_rs_step<2, 4>(v, l);
  rf_rs_step<1, 2>(v, l);
  return v[0];
}

// 64 values over all 64 lanes of the wave: lane l ends with the sum of v[l] (v_permlane32_swap first).
__device__ __forceinline__ float rf_reduce_scatter64(float (&v)[64], int l) {
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[k]), __float_as_uint(v[k + 32]), false, false);
    v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[k]), __float_as_uint(v[k + 16]), false, false);
    v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  rf_rs_step<8, 16>(v, l);
  rf_rs_step<4, 8>(v, l);
  rf_rs_step<2, 4>(v, l);
  rf_rs_step<1, 2>(v, l);
  return v[0];
}

// 8 consecutive elements of a row: load, convert to fp32, pack from fp32, store.
template <typename T> struct Row8;
template <> struct Row8<bf16> {
  uint4 v;
  __device__ __forceinline__ void load(const bf16* p) { v = *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ void set(const float* s) {
    bf16x8 b;
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = (bf16)s[j];
    v = __builtin_bit_cast(uint4, b);
  }
  __device__ __forceinline__ void store(bf16* d) const { *reinterpret_cast<uint4*>(d) = v; }
  __device__ __forceinline__ void store_f32(float* d) const {
    const bf16x8 b = __builtin_bit_cast(bf16x8, v);
    reinterpret_cast<float4*>(d)[0] = float4{(float)b[0], (float)b[1], (float)b[2], (float)b[3]};
    reinterpret_cast<float4*>(d)[1] = float4{(float)b[4], (float)b[5], (float)b[6], (float)b[7]};
  }
};
template <> struct Row8<float> {
  f32x4 a, b;                  // (vector types that stay in registers: a struct of float4 went to scratch)
  __device__ __forceinline__ void load(const float* p) {
    a = reinterpret_cast<const f32x4*>(p)[0];
    b = reinterpret_cast<const f32x4*>(p)[1];
  }
  __device__ __forceinline__ void set(const float* s) {
    a = f32x4{s[0], s[1], s[2], s[3]};
    b = f32x4{s[4], s[5], s[6], s[7]};
  }
  __device__ __forceinline__ void store(float* d) const {
    reinterpret_cast<f32x4*>(d)[0] = a;
    reinterpret_cast<f32x4*>(d)[1] = b;
  }
  __device__ __forceinline__ void store_f32(float* d) const { store(d); }
};

template <int N, int TB, int CPB>
struct __align__(16) RfStage {
  // 16-byte aligned rows, so that a lane's 4 states of B and C are one 16-byte LDS read at an immediate offset
  __align__(16) float B[TB][N];
  __align__(16) float C[TB][N];
  float dt[TB][CPB];        // processed dt (0 past the sequence)
  float x[TB][CPB];         // x (0 past the sequence)
  float z[TB][CPB];         // gate (GATE only)
};
template <int N, int TB, int CPB>
struct RfSmem {
  RfStage<N, TB, CPB> st[2];
  float y[2][TB][CPB];
};

// The rows of one token block held in registers between its load and its LDS store: thread i owns the 8-element
// pieces i, i + 256, .. of B and of C (TB rows of N), and the elements i, i + 256, .. of dt, x and z (one element per
// thread rather than 4 of a quarter of them: the softplus of dt then runs on every wave, not on one while three wait).
template <typename T, int N, int TB, int CPB>
struct RfRegs {
  static constexpr int NP = TB * N / 8;                     // 8-element pieces of B (and of C) per block
  static constexpr int PB = (NP + RF_NT - 1) / RF_NT;      // per thread
  static constexpr int NQ = TB * CPB;                      // elements of dt (x, z) per block
  static constexpr int PQ = (NQ + RF_NT - 1) / RF_NT;      // per thread
  static_assert(RF_NT % CPB == 0, "a thread's elements are of one channel");
  Row8<T> b[PB], c[PB];
  float dt[PQ];                // raw dt; processed (bias, softplus, clamp, 0 past the end) by rf_store
  T xv[PQ], zv[PQ];            // raw x and gate
};

// Workgroup -> (batch, channel block): runs of 4 consecutive blocks go to the same XCD (workgroups are dealt to
// the 8 XCDs round-robin), so the x, y and z lines they share are read or written through one L2.
__device__ __forceinline__ void rf_block(int nblk, int nper, int& b, int& cb) {
  const int i = blockIdx.x;
  int j = i;
  if ((nblk & 31) == 0) j = 4 * ((i & 7) + 8 * (i >> 5)) + ((i >> 3) & 3);
  b = j / nper;
  cb = j % nper;
}

// Workgroup index of the channel-major walks (rf_hs_kernel: (batch, channel block, state group), state group
// fastest), remapped so that each XCD runs a contiguous range of them: the state groups of a channel block then read
// its rows of dt and x through one L2 (workgroups are dealt to the 8 XCDs
// round-robin; dealt as they come, each row was fetched by all eight).
__device__ __forceinline__ int rf_xcd_block() {
  const int i = blockIdx.x, n = gridDim.x;
  if (n % 8 != 0) return i;
  return (i & 7) * (n >> 3) + (i >> 3);
}

// Loads only (every one unconditional at a clamped row), so that they stay in flight while the current block
// computes: the values are converted, masked and stored to LDS by rf_store a block later.
// ANYC: C's rows are read element by element (the backward's dhs in its place is aligned to its elements only).
template <typename T, int N, int TB, int CPB, bool GATE, bool ANYC = false>
__device__ __forceinline__ void rf_load(const RfParams& p, RfRegs<T, N, TB, CPB>& r, int b, int c0, int t0) {
  using R = RfRegs<T, N, TB, CPB>;
  const int tid = threadIdx.x;
  const int last = p.seqlen - 1;
  const T* Bp = reinterpret_cast<const T*>(p.B) + (int64_t)b * p.B_sb;
  const T* Cp = reinterpret_cast<const T*>(p.C) + (int64_t)b * p.C_sb;
#pragma unroll
  for (int q = 0; q < R::PB; ++q) {
    const int e = min(tid + q * RF_NT, R::NP - 1);        // piece: row e / (N / 8), columns 8 (e % (N / 8))
    const int row = min(t0 + e / (N / 8), last), col = 8 * (e % (N / 8));
    r.b[q].load(Bp + (int64_t)row * p.B_sl + col);
    const T* cp = Cp + (int64_t)row * p.C_sl + col;
    if constexpr (ANYC) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = to_f32(cp[j]);
      r.c[q].set(v);
    } else {
      r.c[q].load(cp);
    }
  }
#pragma unroll
  for (int q = 0; q < R::PQ; ++q) {
    const int e = min(tid + q * RF_NT, R::NQ - 1);        // element: row e / CPB, channel e % CPB
    const int rr = min(t0 + e / CPB, last), col = c0 + e % CPB;
    r.dt[q] = p.dt[(int64_t)b * p.dt_sb + (int64_t)rr * p.dt_sl + col];
    r.xv[q] = (reinterpret_cast<const T*>(p.x) + (int64_t)b * p.x_sb)[(int64_t)rr * p.x_sl + col];
    if constexpr (GATE) r.zv[q] = (reinterpret_cast<const T*>(p.z) + (int64_t)b * p.z_sb)[(int64_t)rr * p.z_sl + col];
  }
}

// The block at t0 into LDS: B and C as fp32; dt processed with the thread's channel's bias, dt and x 0
// past the end of the sequence.
template <typename T, int N, int TB, int CPB, bool GATE>
__device__ __forceinline__ void rf_store(const RfParams& p, const RfRegs<T, N, TB, CPB>& r, RfStage<N, TB, CPB>& s,
                                         int t0, float bias) {
  using R = RfRegs<T, N, TB, CPB>;
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < R::PB; ++q) {
    const int e = tid + q * RF_NT;
    if (R::NP % RF_NT != 0 && e >= R::NP) break;
    r.b[q].store_f32(&s.B[e / (N / 8)][8 * (e % (N / 8))]);
    r.c[q].store_f32(&s.C[e / (N / 8)][8 * (e % (N / 8))]);
  }
#pragma unroll
  for (int q = 0; q < R::PQ; ++q) {
    const int e = tid + q * RF_NT;
    if (R::NQ % RF_NT != 0 && e >= R::NQ) break;
    const int row = e / CPB, col = e % CPB;
    const float in = t0 + row < p.seqlen ? 1.f : 0.f;
    s.dt[row][col] = rf_dt(p, r.dt[q], bias) * in;
    s.x[row][col] = to_f32(r.xv[q]) * in;
    if constexpr (GATE) s.z[row][col] = to_f32(r.zv[q]);
  }
}

// One token's operands, read from LDS ahead of their use (one token or two).
template <int NS>
struct RfTok {
  float dt, x, b[NS], c[NS];
};
template <int N, int TB, int CPB, int NS>
__device__ __forceinline__ void rf_tok(const RfStage<N, TB, CPB>& s, int t, int cl, int n0, RfTok<NS>& o) {
  o.dt = s.dt[t][cl];
  o.x = s.x[t][cl];
  if constexpr (NS % 4 == 0) {
#pragma unroll
    for (int q = 0; q < NS; q += 4) {
      const float4 b4 = *reinterpret_cast<const float4*>(&s.B[t][n0 + q]);
      const float4 c4 = *reinterpret_cast<const float4*>(&s.C[t][n0 + q]);
      o.b[q] = b4.x; o.b[q + 1] = b4.y; o.b[q + 2] = b4.z; o.b[q + 3] = b4.w;
      o.c[q] = c4.x; o.c[q + 1] = c4.y; o.c[q + 2] = c4.z; o.c[q + 3] = c4.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      o.b[q] = s.B[t][n0 + q];
      o.c[q] = s.C[t][n0 + q];
    }
  }
}

// CKPT: the checkpoint pass of the backward, which writes the state entering every piece of RF_RK tokens (p.ckpt) and
// no y.
template <typename T, int N, bool GATE, bool CKPT>
__device__ __forceinline__ void rf_scan_walk(const RfParams& p, RfSmem<N, rf_tb<N>(), rf_cpb<N>()>& sm) {
  constexpr int TB = rf_tb<N>(), LPC = rf_lpc<N>(), NS = rf_ns<N>(), CPB = rf_cpb<N>();
  const int nper = p.d_inner / CPB;
  int b, cb;
  rf_block(p.batch * nper, nper, b, cb);
  const int c0 = cb * CPB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int cl = (64 / LPC) * w + lane / LPC, g = lane % LPC;   // channel within the workgroup, its state group
  const int c = c0 + cl;
  const int n0 = g * NS;
  // the lane that ends up with the channel's y: after the row sums (and, for two rows, the row-15 broadcast
  // into the channel's second row) every lane of the last row holds it; take the row's last lane
  const bool ylane = g == LPC - 1;
  float k2[NS], h[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    k2[s] = rf_rate(p, n0 + s) * LOG2E;                           // exp(A dt) = 2^(A log2(e) dt)
    h[s] = p.init_state ? p.init_state[((int64_t)b * p.d_inner + c) * N + n0 + s] : 0.f;
  }
  const float Dc = p.D ? (p.D_per_channel ? p.D[c] : p.D[c / p.headdim]) : 0.f;
  const int nblk = (p.seqlen + TB - 1) / TB;
  RfRegs<T, N, TB, CPB> r;
  const float bias = p.dt_bias ? p.dt_bias[c0 + tid % CPB] : 0.f;   // of this thread's elements' channel
  if (nblk > 0) {
    rf_load<T, N, TB, CPB, GATE>(p, r, b, c0, 0);
    rf_store<T, N, TB, CPB, GATE>(p, r, sm.st[0], 0, bias);
  }
  if (nblk > 1) rf_load<T, N, TB, CPB, GATE>(p, r, b, c0, TB);
  __syncthreads();
  T* yb = reinterpret_cast<T*>(p.y) + (int64_t)b * p.y_sb + c0;
  for (int k = 0; k < nblk; ++k) {
    const RfStage<N, TB, CPB>& s = sm.st[k & 1];
    float (*ys)[CPB] = sm.y[k & 1];
    if constexpr (TB == LPC && LPC == 32) {
      // the block's 32 tokens unrolled: every token's y is left as one partial per lane, and a reduce-scatter
      // over the channel's 32 lanes after the block hands lane g the sum for token g (CKPT: no y; the state
      // entering every piece is stored)
      float yacc[32];
      // operands two tokens ahead of their use, held there by the scheduling barriers: left to itself the compiler
      // read a token's operands and waited for them, with one wave per SIMD nothing else to run
      RfTok<NS> q0, q1;
      rf_tok<N, TB, CPB, NS>(s, 0, cl, n0, q0);
      rf_tok<N, TB, CPB, NS>(s, 1, cl, n0, q1);
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        RfTok<NS> o = q0;
        q0 = q1;
        if (t + 2 < TB) rf_tok<N, TB, CPB, NS>(s, t + 2, cl, n0, q1);
        if constexpr (CKPT) {
          constexpr int RK = RF_RK;                        // divides TB: a piece starts where t % RK == 0
          const int tt = k * TB + t;
          if (t % RK == 0 && tt < p.seqlen) {
            const int nsb = (p.seqlen + RK - 1) / RK;
            float* o = p.ckpt + (((int64_t)b * nsb + tt / RK) * p.d_inner + c) * N + n0;
#pragma unroll
            for (int s2 = 0; s2 < NS; ++s2) o[s2] = h[s2];
          }
        }
        const float u = o.dt * o.x;
        float yp = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < NS; ++s2) {
          const float a = __builtin_amdgcn_exp2f(o.dt * k2[s2]);
          h[s2] = fmaf(a, h[s2], u * o.b[s2]);
          yp = fmaf(o.c[s2], h[s2], yp);
        }
        yacc[t] = yp;
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (!CKPT) {
        float yv = rf_reduce_scatter32(yacc, lane);
        yv += Dc * s.x[g][cl];
        if constexpr (GATE) yv *= silu_f(s.z[g][cl]);
        ys[g][cl] = yv;
      }
    } else {
    RfTok<NS> cur, nxt;
    rf_tok<N, TB, CPB, NS>(s, 0, cl, n0, cur);
#pragma unroll 2
    for (int t = 0; t < TB; ++t) {
      if (t + 1 < TB) rf_tok<N, TB, CPB, NS>(s, t + 1, cl, n0, nxt);
      if constexpr (CKPT) {
        constexpr int RK = RF_RK;                          // divides TB: a piece starts where t % RK == 0
        const int tt = k * TB + t;
        if (t % RK == 0 && tt < p.seqlen) {
          const int nsb = (p.seqlen + RK - 1) / RK;
          float* o = p.ckpt + (((int64_t)b * nsb + tt / RK) * p.d_inner + c) * N + n0;
#pragma unroll
          for (int s2 = 0; s2 < NS; ++s2) o[s2] = h[s2];
        }
      }
      const float u = cur.dt * cur.x;
      float yp = 0.f;
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        const float a = __builtin_amdgcn_exp2f(cur.dt * k2[s2]);
        h[s2] = fmaf(a, h[s2], u * cur.b[s2]);
        yp = fmaf(cur.c[s2], h[s2], yp);
      }
      if constexpr (!CKPT) {
        yp = row_sum16(yp);
        if constexpr (LPC == 32) yp += dppf<0x142, 0xa>(yp);   // row_bcast:15 -> rows 1, 3: both rows of a channel
        if (ylane) {
          float yv = yp + Dc * cur.x;
          if constexpr (GATE) yv *= silu_f(s.z[t][cl]);
          ys[t][cl] = yv;
        }
      }
      cur = nxt;
    }
    }
    if (k + 1 < nblk) rf_store<T, N, TB, CPB, GATE>(p, r, sm.st[(k + 1) & 1], (k + 1) * TB, bias);
    if (k + 2 < nblk) rf_load<T, N, TB, CPB, GATE>(p, r, b, c0, (k + 2) * TB);
    lds_barrier();                       // (not __syncthreads, which would wait for the loads just issued)
    // y rows of this block: CPB channels = CPB / 8 pieces of 8 per token
    if (!CKPT && tid < TB * (CPB / 8)) {
      const int t = tid / (CPB / 8), piece = tid % (CPB / 8);
      const int row = k * TB + t;
      if (row < p.seqlen) {
        Row8<T> o;
        o.set(&ys[t][8 * piece]);
        o.store(yb + (int64_t)row * p.y_sl + 8 * piece);
      }
    }
  }
  if (!CKPT && p.final_state) {
    float* fo = p.final_state + ((int64_t)b * p.d_inner + c) * N + n0;
#pragma unroll
    for (int q = 0; q < NS; ++q) fo[q] = h[q];
  }
}

template <typename T, int N, bool GATE>
__global__ __launch_bounds__(RF_NT) void rf_scan_kernel(RfParams p) {
  __shared__ RfSmem<N, rf_tb<N>(), rf_cpb<N>()> sm;
  rf_scan_walk<T, N, GATE, false>(p, sm);
}

// h_states: sums over the workgroup's 256 channels of every state of group gs (4 states), per token, into
// part[(b * ncb + cblk) * L + t][N]; channels past d_inner stay zero.
template <typename T, int N>
__global__ __launch_bounds__(RF_NT) void rf_hs_kernel(RfParams p) {
  __shared__ float red[4][HS_TB][HS_NS];
  __shared__ float4 sB[2][HS_TB];                          // the group's 4 states of B per token
  const int ncb = (p.d_inner + HS_CPB - 1) / HS_CPB, ngs = N / HS_NS;
  const int i = rf_xcd_block();
  const int gs = i % ngs, cblk = (i / ngs) % ncb, b = i / (ngs * ncb);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = cblk * HS_CPB + tid;
  const bool on = c < p.d_inner;
  const int cc = on ? c : p.d_inner - 1;
  const int n0 = gs * HS_NS;
  float k2[HS_NS], h[HS_NS];
#pragma unroll
  for (int s = 0; s < HS_NS; ++s) {
    k2[s] = rf_rate(p, n0 + s) * LOG2E;
    h[s] = (on && p.init_state) ? p.init_state[((int64_t)b * p.d_inner + c) * N + n0 + s] : 0.f;
  }
  const float bias = p.dt_bias ? p.dt_bias[cc] : 0.f;
  const T* xp = reinterpret_cast<const T*>(p.x) + (int64_t)b * p.x_sb + cc;
  const float* dtp = p.dt + (int64_t)b * p.dt_sb + cc;
  const T* Bp = reinterpret_cast<const T*>(p.B) + (int64_t)b * p.B_sb + n0;
  float* part = p.hs_part + ((int64_t)b * ncb + cblk) * p.seqlen * N + n0;
  // the next block's dt, x (every thread) and B (threads < HS_TB) in registers while the current one computes
  float dn[HS_TB], xn[HS_TB];
  float4 bn = {0.f, 0.f, 0.f, 0.f};
  auto load = [&](int t0) {
#pragma unroll
    for (int j = 0; j < HS_TB; ++j) {
      const int t = min(t0 + j, p.seqlen - 1);
      dn[j] = dtp[(int64_t)t * p.dt_sl];
      xn[j] = to_f32(xp[(int64_t)t * p.x_sl]);
    }
    if (tid < HS_TB) {
      const T* bp = Bp + (int64_t)min(t0 + tid, p.seqlen - 1) * p.B_sl;
      bn = float4{to_f32(bp[0]), to_f32(bp[1]), to_f32(bp[2]), to_f32(bp[3])};
    }
  };
  const int nblk = (p.seqlen + HS_TB - 1) / HS_TB;
  if (nblk > 0) {
    load(0);
    if (tid < HS_TB) sB[0][tid] = bn;
    __syncthreads();
  }
  static_assert(HS_TB * HS_NS == 64, "one value of the block per lane after the reduce-scatter");
  for (int k = 0; k < nblk; ++k) {
    // the block's steps first (no branch per token: dt and u are 0 for a channel past d_inner or a token past
    // the sequence, whose raw values are finite clamped reads)
    float dtv[HS_TB], uu[HS_TB];
#pragma unroll
    for (int j = 0; j < HS_TB; ++j) {
      const float in = (on && k * HS_TB + j < p.seqlen) ? 1.f : 0.f;
      dtv[j] = rf_dt(p, dn[j], bias) * in;
      uu[j] = dtv[j] * xn[j];
    }
    if (k + 1 < nblk) load((k + 1) * HS_TB);
    // every token's 4 states stay one value per lane (v[4 j + s]); one reduce-scatter over the wave's 64
    // channels after the block leaves lane l the sum for token l / 4, state l % 4 (per-token sums took
    // three swaps and a DPP row sum each)
    float v[64];
#pragma unroll
    for (int j = 0; j < HS_TB; ++j) {
      const float4 b4 = sB[k & 1][j];
      const float bv[HS_NS] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
      for (int s = 0; s < HS_NS; ++s) {
        h[s] = fmaf(__builtin_amdgcn_exp2f(dtv[j] * k2[s]), h[s], uu[j] * bv[s]);
        v[HS_NS * j + s] = h[s];
      }
    }
    red[w][lane / HS_NS][lane % HS_NS] = rf_reduce_scatter64(v, lane);
    if (k + 1 < nblk && tid < HS_TB) sB[(k + 1) & 1][tid] = bn;
    __syncthreads();
    if (tid < HS_TB * HS_NS) {
      const int j = tid / HS_NS, s = tid % HS_NS;
      const int t = k * HS_TB + j;
      if (t < p.seqlen) part[(int64_t)t * N + s] = red[0][j][s] + red[1][j][s] + red[2][j][s] + red[3][j][s];
    }
    __syncthreads();
  }
}

// hs[b, t, n] = (sum over channel blocks of part) / d_inner, blocks added in order.
template <typename T>
__global__ __launch_bounds__(256) void rf_hs_reduce_kernel(RfParams p) {
  const int ncb = (p.d_inner + HS_CPB - 1) / HS_CPB;
  const int64_t per = (int64_t)p.seqlen * p.dstate;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.batch * per) return;
  const int64_t b = i / per, r = i % per;
  float s = 0.f;
  for (int k = 0; k < ncb; ++k) s += p.hs_part[(b * ncb + k) * per + r];
  reinterpret_cast<T*>(p.hs)[i] = from_f32<T>(s / (float)p.d_inner);
}

template <typename T, int N>
hipError_t launch_rf_t(const RfParams& p, hipStream_t st) {
  const int nblk = p.batch * (p.d_inner / rf_cpb<N>());
  if (nblk > 0 && (p.seqlen > 0 || p.final_state)) {
    // (an empty sequence only writes the final state: the initial state, or zero)
    if (p.z && p.seqlen > 0) hipLaunchKernelGGL((rf_scan_kernel<T, N, true>), dim3(nblk), dim3(RF_NT), 0, st, p);
    else hipLaunchKernelGGL((rf_scan_kernel<T, N, false>), dim3(nblk), dim3(RF_NT), 0, st, p);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !p.hs || p.seqlen == 0) return e;
  const int ncb = (p.d_inner + HS_CPB - 1) / HS_CPB;
  hipLaunchKernelGGL((rf_hs_kernel<T, N>), dim3(p.batch * ncb * (N / HS_NS)), dim3(RF_NT), 0, st, p);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t tot = (int64_t)p.batch * p.seqlen * N;
  hipLaunchKernelGGL((rf_hs_reduce_kernel<T>), dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rf_n(const RfParams& p, hipStream_t st) {
  switch (p.dstate) {
    case 16: return launch_rf_t<T, 16>(p, st);
    case 32: return launch_rf_t<T, 32>(p, st);
    case 64: return launch_rf_t<T, 64>(p, st);
    case 128: return launch_rf_t<T, 128>(p, st);
    case 256: return launch_rf_t<T, 256>(p, st);
    default: return hipErrorInvalidValue;
  }
}

// ---------------------------------------------------------------- backward
// With lam_t[c, n] the adjoint of h_t[c, n] (lam after the last token = d_final),
//     lam_t = dy_t[c] C_t[n] + dhs_t[n] / d_inner + a_{t+1} lam_{t+1},      a_t = exp(A_n dt_t[c]),
//     dx_t[c]  = dt_t[c] sum_n lam_t B_t[n] + D_c dy_t[c],
//     ddt_t[c] = (sum_n lam_t A_n a_t h_{t-1} + x_t[c] sum_n lam_t B_t[n]) * d dt / d raw,
//     dB_t[n]  = sum_c lam_t dt_t[c] x_t[c],      dC_t[n] = sum_c dy_t[c] h_t[c, n],
//     dA_n     = sum_{t, c} lam_t a_t dt_t[c] h_{t-1},   d h0 = a_0 lam_0,   dD_c = sum_t dy_t[c] x_t[c].
// Every (c, n) pair follows its own recurrences given the per-token inputs.
//   rf_sweep_kernel: the state entering every piece of RF_RK tokens (a forward walk) and the adjoint a_{t+1} lam_{t+1}
//     handed into every piece from its right (a backward walk, which ends with d h0), both directions in one grid: each
//     is a serial walk that leaves its SIMD waiting on its own for half the time.
//   rf_grad_kernel: every piece of every channel block by itself.  A wave holds the states of LC channels (4 states a
//     lane); a piece's states and decays are recomputed forward into registers 8 tokens at a time, the adjoint runs
//     back through them, and both kinds of sums are formed there: over n (dx, ddt) by a reduce-scatter over the
//     channel's lanes per 8 tokens, over c (dB, dC, dA) in registers over the channels the wave takes one after the
//     other, then over the workgroup.
//   rf_bwd_reduce_kernel / rf_bwd_param_kernel: the channel blocks' and pieces' partials added in a fixed order
//     (deterministic).
// Two kernels that each walked the whole sequence backward, one per kind of sum, formed every exponential twice more
// and left half the issue slots empty: b1 L2048 d_inner 2048 N 128, 1420 us for the three passes where these take
// 650 (226 for the sweep, 424 for the gradients), and 20 for the sums of the partials.

// d dt / d raw for dt = clamp(softplus?(raw + bias), dt_min, dt_max) (the clamp passes the gradient inside its
// closed range, as torch.clamp does).
__device__ __forceinline__ float rf_dt_chain(const RfParams& p, float raw, float bias) {
  const float u = raw + bias;
  float g = 1.f, v = u;
  if (p.dt_softplus) {
    if (u <= 20.f) g = 1.f / (1.f + __expf(-u));
    v = softplus_f(u);
  }
  if (p.has_dt_limit && !(v >= p.dt_min && v <= p.dt_max)) g = 0.f;
  return g;
}

// The adjoint walk through the span, last block first, in the scan's layout.  p carries dy in x's place, C in B's and
// dhs in C's (rf_sweep_kernel); dymul is 0 where dy is missing (a finite stand-in is read); HASG: dhs is given, times
// gmul.
template <typename T, int N, bool HASG>
__device__ __forceinline__ void rf_adj_walk(const RfParams& p, RfSmem<N, rf_tb<N>(), rf_cpb<N>()>& sm, float dymul,
                                            float gmul) {
  constexpr int TB = rf_tb<N>(), LPC = rf_lpc<N>(), NS = rf_ns<N>(), CPB = rf_cpb<N>(), RK = RF_RK;
  const int nper = p.d_inner / CPB;
  int b, cb;
  rf_block(p.batch * nper, nper, b, cb);
  const int c0 = cb * CPB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int cl = (64 / LPC) * w + lane / LPC, g = lane % LPC;
  const int c = c0 + cl, n0 = g * NS, L = p.seqlen;
  const int first = p.span0 * RK / TB, nblk = (min(L, (p.span0 + p.span) * RK) + TB - 1) / TB;   // the span's blocks
  const int64_t state = ((int64_t)b * p.d_inner + c) * N + n0;
  const float* from = (p.span0 + p.span) * RK < L ? p.carry : p.d_final;
  float k2[NS], lamc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    k2[s] = rf_rate(p, n0 + s) * LOG2E;
    lamc[s] = from ? from[state + s] : 0.f;
  }
  RfRegs<T, N, TB, CPB> r;
  const float bias = p.dt_bias ? p.dt_bias[c0 + tid % CPB] : 0.f;
  rf_load<T, N, TB, CPB, false, HASG>(p, r, b, c0, (nblk - 1) * TB);
  rf_store<T, N, TB, CPB, false>(p, r, sm.st[(nblk - 1) & 1], (nblk - 1) * TB, bias);
  if (nblk > first + 1) rf_load<T, N, TB, CPB, false, HASG>(p, r, b, c0, (nblk - 2) * TB);
  __syncthreads();
  float* ck = p.lam_ckpt + ((int64_t)b * p.span * p.d_inner + c) * N + n0;
  for (int k = nblk - 1; k >= first; --k) {
    const RfStage<N, TB, CPB>& s = sm.st[k & 1];
#pragma unroll 16
    for (int t = TB - 1; t >= 0; --t) {
      const int tt = k * TB + t;                           // (past the end: dt = 0, dy = 0, no dhs)
      if (t % RK == RK - 1 && tt - (RK - 1) < L) {
        float* o = ck + (int64_t)(tt / RK - p.span0) * p.d_inner * N;
#pragma unroll
        for (int s2 = 0; s2 < NS; ++s2) o[s2] = lamc[s2];
      }
      RfTok<NS> o;
      rf_tok<N, TB, CPB, NS>(s, t, cl, n0, o);
      const float dy = o.x * dymul, gm = tt < L ? gmul : 0.f;
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        float lam = fmaf(dy, o.b[s2], lamc[s2]);
        if constexpr (HASG) lam = fmaf(gm, o.c[s2], lam);
        lamc[s2] = __builtin_amdgcn_exp2f(o.dt * k2[s2]) * lam;
      }
    }
    if (k > first) rf_store<T, N, TB, CPB, false>(p, r, sm.st[(k - 1) & 1], (k - 1) * TB, bias);
    if (k > first + 1) rf_load<T, N, TB, CPB, false, HASG>(p, r, b, c0, (k - 2) * TB);
    lds_barrier();
  }
  float* to = first > 0 ? p.carry : p.dh0;               // (each lane its own, read above)
  if (to) {
#pragma unroll
    for (int s = 0; s < NS; ++s) to[state + s] = lamc[s];
  }
}

template <typename T, int N, bool HASG>
__global__ __launch_bounds__(RF_NT) void rf_sweep_kernel(RfParams p) {
  __shared__ RfSmem<N, rf_tb<N>(), rf_cpb<N>()> sm;
  if (blockIdx.y + p.sweep0 == 0) {
    rf_scan_walk<T, N, false, true>(p, sm);
    return;
  }
  const float dymul = p.dy ? 1.f : 0.f, gmul = HASG ? 1.f / (float)p.d_inner : 0.f;
  if (p.dy) {
    p.x = p.dy; p.x_sl = p.d_inner; p.x_sb = (int64_t)p.seqlen * p.d_inner;
  }
  p.B = p.C; p.B_sb = p.C_sb; p.B_sl = p.C_sl;
  if constexpr (HASG) {
    p.C = p.dhs; p.C_sl = N; p.C_sb = (int64_t)p.seqlen * N;
  }
  rf_adj_walk<T, N, HASG>(p, sm, dymul, gmul);
}

// Lanes and channels of the gradient kernel's waves: 4 states a lane.
template <int N> constexpr int rfg_ln() { return N / 4; }
template <int N> constexpr int rfg_lc() { return 64 / rfg_ln<N>(); }

template <int N, bool HASG>
struct __align__(16) RfGradSmem {
  float4 sv[RF_RK + 1][RF_CH];         // dt, dt x, dy, x per (token, channel) (0 past the ends); then dx, ddt; the last
  float chain[RF_RK + 1][RF_CH];       // row is nobody's (lanes that finish no token).  chain: d dt / d raw
  float D[RF_CH];
  __align__(16) float B[RF_RK][N], C[RF_RK][N], G[HASG ? RF_RK : 1][N];   // G = dhs / d_inner
  float4 lam[RF_CH][N / 4];            // the adjoint between the piece's halves
  float4 red[2][RF_HK][N / 4];         // dB, dC of a half over the workgroup; at the end each wave's dA
};

// Exchange-and-add over lane bit M: the lanes with the bit set end with the upper half of the K values summed over
// the pair, the others with the lower half.
template <int M, int K, int NV>
__device__ __forceinline__ void rf_halve(float (&v)[NV], int l) {
  if constexpr (M == 32 || M == 16) {
#pragma unroll
    for (int k = 0; k < K / 2; ++k) {
      if constexpr (M == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[k]), __float_as_uint(v[k + K / 2]), false, false);
        v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[k]), __float_as_uint(v[k + K / 2]), false, false);
        v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      }
    }
  } else {
    rf_rs_step<M, K>(v, l);
  }
}
// The value of lane l ^ M.
template <int M>
__device__ __forceinline__ float rf_xor(float v) {
  if constexpr (M == 8) return xor8(v);
  else if constexpr (M == 4) return xor4(v);
  else if constexpr (M == 2) return xor2(v);
  else return xor1(v);
}
// 16 values summed over LN lanes (the low bits of l): lane g of them ends with v[k] the sum of value g K + k,
// K = 16 / LN (at least 1: lanes g and g ^ 1, .. share one where LN > 16).
template <int LN>
__device__ __forceinline__ void rf_sum16(float (&v)[16], int l) {
  if constexpr (LN == 64) {
    rf_halve<32, 16>(v, l); rf_halve<16, 8>(v, l); rf_halve<8, 4>(v, l); rf_halve<4, 2>(v, l);
    v[0] += rf_xor<2>(v[0]);
    v[0] += rf_xor<1>(v[0]);
  } else if constexpr (LN == 32) {
    rf_halve<16, 16>(v, l); rf_halve<8, 8>(v, l); rf_halve<4, 4>(v, l); rf_halve<2, 2>(v, l);
    v[0] += rf_xor<1>(v[0]);
  } else if constexpr (LN == 16) {
    rf_halve<8, 16>(v, l); rf_halve<4, 8>(v, l); rf_halve<2, 4>(v, l); rf_halve<1, 2>(v, l);
  } else if constexpr (LN == 8) {
    rf_halve<4, 16>(v, l); rf_halve<2, 8>(v, l); rf_halve<1, 4>(v, l);
  } else {
    rf_halve<2, 16>(v, l); rf_halve<1, 8>(v, l);
  }
}

// grid batch x pieces x channel blocks (a piece's blocks read the same B and C rows).  The piece's later half first, for
// all of the workgroup's channels, then the earlier one (its adjoint waits in LDS): the sums over the channels then hold 64 registers at a time, and with the
// states and decays of 8 tokens the kernel fits two waves per SIMD (both halves' sums at once spilled 58 registers).
template <typename T, int N, bool HASG>
__global__ __launch_bounds__(RF_NT, 2) void rf_grad_kernel(RfParams p) {
  constexpr int LN = rfg_ln<N>(), LC = rfg_lc<N>(), RK = RF_RK, HK = RF_HK, CH = RF_CH;
  constexpr int NSTEP = CH / (4 * LC);
  __shared__ RfGradSmem<N, HASG> sm;
  const int L = p.seqlen, di = p.d_inner;
  const int nsb = (L + RK - 1) / RK, ncb = (di + CH - 1) / CH;
  const int bj = blockIdx.x / ncb, cb = blockIdx.x - bj * ncb;
  const int b = bj / p.span, j = p.span0 + bj - b * p.span;   // bj: the (row, piece of the span)
  const int t0 = j * RK, c0 = cb * CH;
  const int tid = threadIdx.x, l = tid & 63, w = wave_id(), gl = l % LN;
  const int n0 = 4 * gl;

  // ---- the piece's inputs: every load unconditional at a clamped address, masked by factors afterwards
  {
    const T* xb = reinterpret_cast<const T*>(p.x) + (int64_t)b * p.x_sb;
    const T* dyb = p.dy ? reinterpret_cast<const T*>(p.dy) + (int64_t)b * L * di : xb;
    const int64_t dysl = p.dy ? di : p.x_sl;
    const float dymul = p.dy ? 1.f : 0.f;
    const float* dtb = p.dt + (int64_t)b * p.dt_sb;
#pragma unroll
    for (int k = 0; k < RK * CH / RF_NT; ++k) {
      const int e = tid + RF_NT * k, t = e / CH, q = e % CH, tt = min(t0 + t, L - 1), c = min(c0 + q, di - 1);
      const float in = (t0 + t < L && c0 + q < di) ? 1.f : 0.f;
      const float raw = dtb[(int64_t)tt * p.dt_sl + c], bias = p.dt_bias ? p.dt_bias[c] : 0.f;
      const float x = to_f32(xb[(int64_t)tt * p.x_sl + c]) * in, dy = to_f32(dyb[(int64_t)tt * dysl + c]) * (in * dymul);
      const float dt = rf_dt(p, raw, bias) * in;
      sm.sv[t][q] = float4{dt, dt * x, dy, x};
      sm.chain[t][q] = rf_dt_chain(p, raw, bias) * in;
    }
    if (tid < CH) {
      const int c = c0 + tid;
      sm.D[tid] = p.D && c < di ? (p.D_per_channel ? p.D[c] : p.D[c / p.headdim]) : 0.f;
    }
    const T* Bp = reinterpret_cast<const T*>(p.B) + (int64_t)b * p.B_sb;
    const T* Cp = reinterpret_cast<const T*>(p.C) + (int64_t)b * p.C_sb;
#pragma unroll
    for (int k = 0; k < RK * N / RF_NT; ++k) {
      const int e = tid + RF_NT * k, t = e / N, n = e % N, tt = min(t0 + t, L - 1);
      const float in = t0 + t < L ? 1.f : 0.f;
      sm.B[t][n] = to_f32(Bp[(int64_t)tt * p.B_sl + n]) * in;
      sm.C[t][n] = to_f32(Cp[(int64_t)tt * p.C_sl + n]) * in;
      if constexpr (HASG)
        sm.G[t][n] = to_f32((reinterpret_cast<const T*>(p.dhs) + (int64_t)b * L * N)[(int64_t)tt * N + n]) * (in / (float)di);
    }
  }
  static_assert(RK * CH % RF_NT == 0 && RK * N % RF_NT == 0, "whole passes of the staging");
  float k2[4], As[4], dA[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    As[i] = rf_rate(p, n0 + i);
    k2[i] = As[i] * LOG2E;
    dA[i] = 0.f;
  }
  __syncthreads();
  const int64_t prow = ((int64_t)b * nsb + j) * di, srow = (int64_t)bj * di;   // rows by the sequence's, the span's pieces
  if (tid < CH && c0 + tid < di) {
    float dD = 0.f;
#pragma unroll
    for (int t = 0; t < RK; ++t) dD = fmaf(sm.sv[t][tid].z, sm.sv[t][tid].w, dD);
    p.dD_part[srow + c0 + tid] = dD;
  }
  __syncthreads();                                         // dx takes the place of dt below

  auto chan = [&](int s) { return (4 * s + w) * LC + l / LN; };      // channel within the block
  auto ckpt = [&](const float* base, int64_t row, int q) {
    return *reinterpret_cast<const float4*>(base + (row + min(c0 + q, di - 1)) * N + n0);
  };
  auto half = [&](auto OFFc) {
    constexpr int OFF = decltype(OFFc)::value;             // the half's first token
    float acc[2 * HK * 4];                                 // dB then dC: [token][state] sums over this lane's channels
#pragma unroll
    for (int i = 0; i < 2 * HK * 4; ++i) acc[i] = 0.f;
    float4 hn = ckpt(p.ckpt, prow, chan(0)), ln;
    if constexpr (OFF > 0) ln = ckpt(p.lam_ckpt, srow, chan(0));
    int s = 0;
#pragma unroll 1
    do {                                                   // (no branch inside: a second copy of the sums at every join)
      const int q = chan(s);
      const float on = c0 + q < di ? 1.f : 0.f;            // (a channel past d_inner repeats the last one's states)
      if constexpr (OFF == 0) ln = sm.lam[q][gl];          // (this wave's own)
      float h[4] = {hn.x * on, hn.y * on, hn.z * on, hn.w * on};
      float lamc[4] = {ln.x * on, ln.y * on, ln.z * on, ln.w * on};
      const int qn = chan(min(s + 1, NSTEP - 1));
      hn = ckpt(p.ckpt, prow, qn);
      if constexpr (OFF > 0) ln = ckpt(p.lam_ckpt, srow, qn);
      const float Dc = sm.D[q];
      // the B and C rows are the same every step: laundered here, so that they are read from LDS again instead of
      // held in 128 registers for the whole loop
      int nl = n0;
      asm volatile("" : "+v"(nl));
      // Each token's operands are read one token ahead; the scheduling barriers keep the compiler from reading more
      // of them at once than the registers hold.
      struct Tok { float4 v, B; };
      auto tok = [&](int t) { return Tok{sm.sv[t][q], *reinterpret_cast<const float4*>(&sm.B[t][nl])}; };
      Tok cur = tok(0);
      float hp[HK][4], av[HK][4];
#pragma unroll
      for (int t = 0; t < OFF + HK; ++t) {                 // from the half's first token on states and decays are kept
        const Tok nxt = tok(t + 1 < OFF + HK ? t + 1 : t);
        const float bb[4] = {cur.B.x, cur.B.y, cur.B.z, cur.B.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a = __builtin_amdgcn_exp2f(cur.v.x * k2[i]);
          if (t >= OFF) {
            hp[t >= OFF ? t - OFF : 0][i] = h[i];
            av[t >= OFF ? t - OFF : 0][i] = a;
          }
          h[i] = fmaf(a, h[i], cur.v.y * bb[i]);
        }
        cur = nxt;
        __builtin_amdgcn_sched_barrier(0);
      }
      float vv[2 * HK];                                    // du, qq of token t at 2 t, 2 t + 1
      auto row = [&](const float (*m)[N], int t) { return *reinterpret_cast<const float4*>(&m[t][nl]); };
      float4 C4 = row(sm.C, OFF + HK - 1), G4 = {0.f, 0.f, 0.f, 0.f};
      if constexpr (HASG) G4 = row(sm.G, OFF + HK - 1);
#pragma unroll
      for (int t = HK - 1; t >= 0; --t) {
        const int tn = OFF + (t > 0 ? t - 1 : 0);
        const Tok nxt = tok(tn);
        const float4 Cn = row(sm.C, tn);
        float4 Gn = G4;
        if constexpr (HASG) Gn = row(sm.G, tn);
        const float4 v = cur.v;
        const float bb[4] = {cur.B.x, cur.B.y, cur.B.z, cur.B.w}, cc[4] = {C4.x, C4.y, C4.z, C4.w};
        const float gg[4] = {G4.x * on, G4.y * on, G4.z * on, G4.w * on};
        float du = 0.f, qq = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float lam = fmaf(v.z, cc[i], lamc[i]);
          if constexpr (HASG) lam += gg[i];
          du = fmaf(lam, bb[i], du);
          acc[4 * t + i] = fmaf(lam, v.y, acc[4 * t + i]);
          acc[4 * (HK + t) + i] = fmaf(v.z, t + 1 < HK ? hp[t + 1 < HK ? t + 1 : 0][i] : h[i], acc[4 * (HK + t) + i]);
          lamc[i] = av[t][i] * lam;
          const float pz = lamc[i] * hp[t][i];             // lam a h_{t-1}
          qq = fmaf(pz, As[i], qq);
          dA[i] = fmaf(pz, v.x, dA[i]);
        }
        vv[2 * t] = du;
        vv[2 * t + 1] = qq;
        cur = nxt;
        C4 = Cn;
        G4 = Gn;
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (OFF > 0) sm.lam[q][gl] = float4{lamc[0], lamc[1], lamc[2], lamc[3]};
      rf_sum16<LN>(vv, l);
      // the lane that finishes a token: it holds (or its partner hands it) du and qq
      auto finish = [&](int t, float du, float qq) {
        const float4 v = sm.sv[t][q];
        sm.sv[t][q].x = fmaf(v.x, du, Dc * v.z);
        sm.sv[t][q].y = fmaf(v.w, du, qq) * sm.chain[t][q];
      };
      if constexpr (LN >= 16) {
        constexpr int P = LN / 16;                         // lanes sharing a value
        const float other = rf_xor<P>(vv[0]);
        finish(gl % (2 * P) == 0 ? OFF + gl / (2 * P) : RK, vv[0], other);
      } else {
        constexpr int K = 16 / LN;
#pragma unroll
        for (int k = 0; k < K; k += 2) finish(OFF + (gl * K + k) / 2, vv[k], vv[k + 1]);
      }
    } while (++s < NSTEP);

    // ---- sums over the channels: over the wave's LC channel groups, then over the 4 waves in order
    constexpr int V = 2 * HK * 4 / LC;                     // values per lane afterwards, from index (l / LN) V
    if constexpr (LC >= 2) rf_halve<32, 64>(acc, l);
    if constexpr (LC >= 4) rf_halve<16, 32>(acc, l);
    if constexpr (LC >= 8) rf_halve<8, 16>(acc, l);
    if constexpr (LC >= 16) rf_halve<4, 8>(acc, l);
    float4* red = &sm.red[0][0][0];
    const int base = (l / LN) * (V / 4);                   // in 4-state rows: which * HK + token
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
      if (w == k) {
#pragma unroll
        for (int r = 0; r < V / 4; ++r) {
          float4 a = {acc[4 * r], acc[4 * r + 1], acc[4 * r + 2], acc[4 * r + 3]};
          float4* d = red + (base + r) * (N / 4) + gl;
          if (k) {
            const float4 o = *d;
            a = float4{o.x + a.x, o.y + a.y, o.z + a.z, o.w + a.w};
          }
          *d = a;
        }
      }
      __syncthreads();
    }
    const float* rf = reinterpret_cast<const float*>(red);
    const int s0 = p.span0 * RK, Ls = min(L - s0, p.span * RK);   // the span's tokens
    for (int e = tid; e < 2 * HK * N; e += RF_NT) {
      const int t = t0 + OFF + (e / N) % HK, n = e % N;
      if (t < L) (e < HK * N ? p.dB_part : p.dC_part)[(((int64_t)b * ncb + cb) * Ls + t - s0) * N + n] = rf[e];
    }
    __syncthreads();                                       // red is written again
  };
  half(std::integral_constant<int, HK>{});
  half(std::integral_constant<int, 0>{});

  float* dAw = reinterpret_cast<float*>(&sm.red[0][0][0]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (LC >= 2) dA[i] = sum_halves(dA[i]);
    if constexpr (LC >= 4) dA[i] += __shfl_xor(dA[i], 16, 64);
    if constexpr (LC >= 8) dA[i] += xor8(dA[i]);
    if constexpr (LC >= 16) dA[i] += xor4(dA[i]);
    if (l < LN) dAw[w * N + n0 + i] = dA[i];
  }
  __syncthreads();
  if (tid < N)
    p.dA_part[((int64_t)bj * ncb + cb) * N + tid] = dAw[tid] + dAw[N + tid] + dAw[2 * N + tid] + dAw[3 * N + tid];
  if (tid < CH && c0 + tid < di) {
    float db = 0.f;
#pragma unroll
    for (int t = 0; t < RK; ++t) db += sm.sv[t][tid].y;
    p.dbias_part[srow + c0 + tid] = db;
  }
#pragma unroll
  for (int k = 0; k < RK * CH / RF_NT; ++k) {
    const int e = tid + RF_NT * k, t = e / CH, q = e % CH;
    if (t0 + t < L && c0 + q < di) {
      const int64_t o = ((int64_t)b * L + t0 + t) * di + c0 + q;
      const float4 v = sm.sv[t][q];
      reinterpret_cast<T*>(p.dx)[o] = from_f32<T>(v.x);
      p.ddt[o] = v.y;
    }
  }
}

// dB, dC (b, L, N), the span's tokens = the channel blocks' partials added in order.
template <typename T>
__global__ __launch_bounds__(256) void rf_bwd_reduce_kernel(RfParams p, int ncb) {
  const int s0 = p.span0 * RF_RK;
  const int64_t per = (int64_t)min(p.seqlen - s0, p.span * RF_RK) * p.dstate / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.batch * per) return;
  const int64_t b = i / per, r = i % per;
  const f32x4* pb = reinterpret_cast<const f32x4*>(p.dB_part);
  const f32x4* pc = reinterpret_cast<const f32x4*>(p.dC_part);
  f32x4 sb = {0.f, 0.f, 0.f, 0.f}, sc = sb;
#pragma unroll 8
  for (int k = 0; k < ncb; ++k) {
    sb += pb[(b * ncb + k) * per + r];
    sc += pc[(b * ncb + k) * per + r];
  }
  const int64_t o = (b * p.seqlen + s0) * p.dstate + 4 * r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    reinterpret_cast<T*>(p.dB)[o + j] = from_f32<T>(sb[j]);
    reinterpret_cast<T*>(p.dC)[o + j] = from_f32<T>(sc[j]);
  }
}

// Sum over rows r of part[r][i] for column i of `cols`, by the 64 threads of a column (rows t, t + 64, .. in order, then
// the 64 sums in order): a workgroup of 1024 takes 16 columns (with 16 threads a column, 4096 rows took 32 us, now 8).
__device__ __forceinline__ float rf_column_sum(const float* part, int64_t rows, int64_t cols, int i, bool on,
                                               float (&red)[64][17]) {
  const int t = threadIdx.x >> 4, q = threadIdx.x & 15;
  float s = 0.f;
  if (on)
#pragma unroll 8
    for (int64_t r = t; r < rows; r += 64) s += part[r * cols + i];
  __syncthreads();
  red[t][q] = s;
  __syncthreads();
  float a = 0.f;
#pragma unroll
  for (int k = 0; k < 64; ++k) a += red[k][q];
  return a;
}

// dA (N): partials per (batch, piece, channel block); dD per channel and d dt_bias (d_inner): per (batch, piece), of the
// span, onto those of the spans before (to the right).  One workgroup per 16 columns, dA's first; with D per head the
// channel sums go to dD_sum and rf_bwd_head_kernel adds a head's channels.
__global__ __launch_bounds__(1024) void rf_bwd_param_kernel(RfParams p, int ncb, int na) {
  __shared__ float red[64][17];
  const int di = p.d_inner, N = p.dstate, q = threadIdx.x & 15;
  const int64_t rows = (int64_t)p.batch * p.span;
  if ((int)blockIdx.x < na) {
    const int i = blockIdx.x * 16 + q;
    float a = rf_column_sum(p.dA_part, rows * ncb, N, i, i < N, red);
    if (threadIdx.x < 16 && i < N) {
      if (!p.first) a += p.dA[i];
      const float r = p.A[i];                              // A_log's gradient: through exp, inside the clamp
      p.dA[i] = !p.last || !p.A_log ? a : r >= -5.f && r <= 5.f ? a * rf_rate(p, i) : 0.f;
    }
    return;
  }
  const int i = (blockIdx.x - na) * 16 + q;
  const float d = rf_column_sum(p.dD_part, rows, di, i, i < di, red);
  const float s = rf_column_sum(p.dbias_part, rows, di, i, i < di, red);
  if (threadIdx.x < 16 && i < di) {
    if (p.d_dt_bias) p.d_dt_bias[i] = p.first ? s : p.d_dt_bias[i] + s;
    float* o = p.D_per_channel ? p.dD : p.dD_sum;
    if (p.dD) o[i] = p.first ? d : o[i] + d;
  }
}

__global__ __launch_bounds__(256) void rf_bwd_head_kernel(RfParams p) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.d_inner / p.headdim) return;
  float sd = 0.f;
  for (int q = 0; q < p.headdim; ++q) sd += p.dD_sum[i * p.headdim + q];
  p.dD[i] = sd;
}

// Empty sequence: every sum is zero and d h0 is d_final.
__global__ __launch_bounds__(256) void rf_bwd_empty_kernel(RfParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int di = p.d_inner;
  if (i < p.dstate) p.dA[i] = 0.f;
  if (p.d_dt_bias && i < di) p.d_dt_bias[i] = 0.f;
  if (p.dD && i < (p.D_per_channel ? di : di / p.headdim)) p.dD[i] = 0.f;
  if (p.dh0 && i < (int64_t)p.batch * di * p.dstate) p.dh0[i] = p.d_final ? p.d_final[i] : 0.f;
}

template <typename T, int N>
hipError_t launch_rf_bwd_t(const RfParams& p, hipStream_t st) {
  if (p.seqlen == 0) {
    const int64_t n = std::max<int64_t>(p.dh0 ? (int64_t)p.batch * p.d_inner * N : 0, std::max(p.d_inner, N));
    hipLaunchKernelGGL(rf_bwd_empty_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p);
    return hipGetLastError();
  }
  const unsigned walks = (unsigned)(p.batch * (p.d_inner / rf_cpb<N>()));
  const bool whole = p.span == (p.seqlen + RF_RK - 1) / RF_RK;
  if (!whole && p.span0 + p.span >= (p.seqlen + RF_RK - 1) / RF_RK) {   // the first span of these rows: their states
    hipLaunchKernelGGL((rf_sweep_kernel<T, N, false>), dim3(walks, 1), dim3(RF_NT), 0, st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  RfParams q = p;
  q.sweep0 = whole ? 0 : 1;
  const dim3 sgrid(walks, whole ? 2 : 1);
  if (p.dhs) hipLaunchKernelGGL((rf_sweep_kernel<T, N, true>), sgrid, dim3(RF_NT), 0, st, q);
  else hipLaunchKernelGGL((rf_sweep_kernel<T, N, false>), sgrid, dim3(RF_NT), 0, st, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int ncb = (p.d_inner + RF_CH - 1) / RF_CH;
  const dim3 grid((unsigned)((int64_t)p.batch * p.span * ncb));
  if (p.dhs) hipLaunchKernelGGL((rf_grad_kernel<T, N, true>), grid, dim3(RF_NT), 0, st, p);
  else hipLaunchKernelGGL((rf_grad_kernel<T, N, false>), grid, dim3(RF_NT), 0, st, p);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t tot = (int64_t)p.batch * std::min(p.seqlen - p.span0 * RF_RK, p.span * RF_RK) * N / 4;
  hipLaunchKernelGGL((rf_bwd_reduce_kernel<T>), dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, st, p, ncb);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int na = (N + 15) / 16;
  hipLaunchKernelGGL(rf_bwd_param_kernel, dim3((unsigned)(na + (p.d_inner + 15) / 16)), dim3(1024), 0, st, p, ncb, na);
  e = hipGetLastError();
  if (e != hipSuccess || !p.dD || p.D_per_channel || !p.last) return e;
  hipLaunchKernelGGL(rf_bwd_head_kernel, dim3((unsigned)((p.d_inner / p.headdim + 255) / 256)), dim3(256), 0, st, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rf_bwd_n(const RfParams& p, hipStream_t st) {
  switch (p.dstate) {
    case 16: return launch_rf_bwd_t<T, 16>(p, st);
    case 32: return launch_rf_bwd_t<T, 32>(p, st);
    case 64: return launch_rf_bwd_t<T, 64>(p, st);
    case 128: return launch_rf_bwd_t<T, 128>(p, st);
    case 256: return launch_rf_bwd_t<T, 256>(p, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool ssd_rf_supported(int dstate) {
  return dstate == 16 || dstate == 32 || dstate == 64 || dstate == 128 || dstate == 256;
}

size_t ssd_rf_workspace_bytes(int batch, int seqlen, int d_inner, int dstate, bool h_states) {
  if (!h_states) return 0;
  const size_t ncb = (size_t)(d_inner + HS_CPB - 1) / HS_CPB;
  return align256((size_t)batch * ncb * seqlen * dstate * 4);
}

hipError_t launch_ssd_rf(const RfParams& p, hipStream_t st) {
  if (p.dtype == DT_BF16) return launch_rf_n<bf16>(p, st);
  return launch_rf_n<float>(p, st);
}

// Backward workspace, all fp32 (the parts of RfParams).  Whole, the adjoints are as many as the states and the partials half
// of that: 2.6 times the states' bytes, where a walk backward through the states needs little besides them (b1 L16384
// d_inner 4096 N128: 5.7 GB, states 2.1).  Beyond RF_WHOLE_BYTES the call therefore takes a span of the pieces after
// another, or where there are too few pieces some batch rows after others, so that all of it fits RF_WHOLE_BYTES or 9/8
// of the states, whichever is more.  Spans first: every row's walks still run side by side.  Forward and backward, whole
// and in spans or rows: that size 12.60 and 12.72 ms, b1 L65536 d_inner 2048 N64 14.6 and 16.6, b512 L256 25.0 and 24.3.
constexpr size_t RF_WHOLE_BYTES = (size_t)2 << 30;
struct RfBwdPlan {
  int rows, span;                                          // batch rows and pieces at a time
  size_t ck, lam, carry, part, da, dd, ds;

  RfBwdPlan(int batch, int seqlen, int d_inner, int dstate) {
    const int nsb = (seqlen + RF_RK - 1) / RF_RK;
    if (sizes(batch, nsb, seqlen, d_inner, dstate) <= RF_WHOLE_BYTES) return;
    const size_t most = std::max(RF_WHOLE_BYTES, ck / 8 * 9);
    const int step = dstate <= 128 ? 32 / RF_RK : 1;       // a walk's blocks (rf_tb) are whole
    int least = nsb;
    for (int n = 2; n <= 32 && n <= nsb; ++n) {
      const int sp = ((nsb + n - 1) / n + step - 1) / step * step;
      if (sp >= nsb) continue;
      least = sp;
      if (sizes(batch, sp, seqlen, d_inner, dstate) <= most) return;
    }
    for (int n = 2; n <= batch && n <= 4; ++n)
      if (sizes((batch + n - 1) / n, nsb, seqlen, d_inner, dstate) <= most) return;
    sizes(batch, least, seqlen, d_inner, dstate);          // (a short sequence of one row or two: as near as its blocks allow)
  }

  size_t sizes(int r, int s, int seqlen, int d_inner, int dstate) {
    rows = r;
    span = s;
    const size_t b = r, sp = s, di = d_inner, N = dstate, nsb = ((size_t)seqlen + RF_RK - 1) / RF_RK;
    const size_t ncb = (di + RF_CH - 1) / RF_CH, tokens = std::min<size_t>(seqlen, sp * RF_RK);
    ck = align256(b * nsb * di * N * 4);
    lam = align256(b * sp * di * N * 4);
    carry = sp < nsb ? align256(b * di * N * 4) : 0;
    part = align256(b * ncb * tokens * N * 4);
    da = align256(b * sp * ncb * N * 4);
    dd = align256(b * sp * di * 4);
    ds = align256(di * 4);
    return bytes();
  }
  size_t bytes() const { return ck + lam + carry + 2 * part + da + 2 * dd + ds; }
};

size_t ssd_rf_bwd_workspace_bytes(int batch, int seqlen, int d_inner, int dstate) {
  return RfBwdPlan(batch, seqlen, d_inner, dstate).bytes();
}

hipError_t launch_ssd_rf_bwd(const RfParams& p, void* workspace, hipStream_t st) {
  const RfBwdPlan s(p.batch, p.seqlen, p.d_inner, p.dstate);
  RfParams q = p;
  char* w = reinterpret_cast<char*>(workspace);
  auto take = [&](size_t n) { char* r = w; w += n; return reinterpret_cast<float*>(r); };
  q.ckpt = take(s.ck);
  q.lam_ckpt = take(s.lam);
  q.carry = take(s.carry);
  q.dB_part = take(s.part);
  q.dC_part = take(s.part);
  q.dA_part = take(s.da);
  q.dD_part = take(s.dd);
  q.dbias_part = take(s.dd);
  q.dD_sum = take(s.ds);
  auto launch = [&](const RfParams& r) { return r.dtype == DT_BF16 ? launch_rf_bwd_n<bf16>(r, st) : launch_rf_bwd_n<float>(r, st); };
  q.first = q.last = 1;
  if (p.seqlen == 0) return launch(q);

  const int nsb = (p.seqlen + RF_RK - 1) / RF_RK;
  const int64_t es = p.dtype == DT_BF16 ? 2 : 4, di = p.d_inner, N = p.dstate;
  auto at = [](auto* base, int64_t bytes) {                // null stays null
    using P = decltype(base);
    return base ? reinterpret_cast<P>(reinterpret_cast<uintptr_t>(base) + bytes) : base;
  };
  for (int64_t b0 = 0; b0 < p.batch; b0 += s.rows) {
    RfParams r = q;
    r.batch = (int)std::min<int64_t>(s.rows, p.batch - b0);
    r.x = at(p.x, b0 * p.x_sb * es);
    r.dt = at(p.dt, b0 * p.dt_sb * 4);
    r.B = at(p.B, b0 * p.B_sb * es);
    r.C = at(p.C, b0 * p.C_sb * es);
    r.init_state = at(p.init_state, b0 * di * N * 4);
    r.dy = at(p.dy, b0 * p.seqlen * di * es);
    r.dhs = at(p.dhs, b0 * p.seqlen * N * es);
    r.d_final = at(p.d_final, b0 * di * N * 4);
    r.dx = at(p.dx, b0 * p.seqlen * di * es);
    r.ddt = at(p.ddt, b0 * p.seqlen * di * 4);
    r.dB = at(p.dB, b0 * p.seqlen * N * es);
    r.dC = at(p.dC, b0 * p.seqlen * N * es);
    r.dh0 = at(p.dh0, b0 * di * N * 4);
    for (int j = (nsb - 1) / s.span * s.span; j >= 0; j -= s.span) {   // the last span first: adjoints run backward
      r.span0 = j;
      r.span = std::min(s.span, nsb - j);
      r.first = b0 == 0 && j + s.span >= nsb;
      r.last = b0 + s.rows >= p.batch && j == 0;
      const hipError_t e = launch(r);
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

}  // namespace mh
