// One token through a whole Mamba-2 layer from its cache (Mamba2Block.forward's incremental path,
// mamformer/layers/mamba2.py:272-296, 337-364), bf16, for a batch of up to 64 sequences.
//
// The layer's projections at this size read every weight once for a handful of rows, so they are bound by the weights'
// bytes and, as six library calls with the element-wise pieces between them, by the launches: 242 us a call at d_model
// 2048 and 8 sequences, of which the GPU worked 75.  Four launches here, 37 us a call (26 of GPU time: in_proj 9.3 for
// its 16.8 MB of weights, the two other products 5.4 each, the state update 5.9):
//   1. in_proj, whose epilogue runs the causal conv and SiLU of the x half on the row it has just formed and writes
//      the rolled conv_state;
//   2. the dt (low rank), B and C projections of x_act, as one product over three weight matrices;
//   3. the state update with the gate (ssu_kernel), which forms dt from its low-rank row itself;
//   4. out_proj.
// Intermediate rows (x_act, z, the low-rank dt, B, C, y) are rounded to bf16 where the library calls rounded them.
//
// step_gemm_kernel: Y[m][n] = sum_k X[m][k] W[n][k].  A workgroup owns 16 rows of W (the MFMA's A operand) for all m
// (its B operand, 16 sequences a tile, MT tiles), its 8 waves every 8th 32-wide k-step; a lane reads 16 consecutive
// bytes of a row of W, so the workgroup's loads, all independent, cover whole rows.  The waves' partial tiles are
// summed through LDS in wave order.
#include "common.h"
#include "launch.h"

namespace mh {

namespace {

constexpr int SG_WAVES = 8;

typedef bf16x8 frag8;

__device__ __forceinline__ f32x4 mma16(frag8 a, frag8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// CONV: segment 0 is in_proj; rows below p.d_inner are x (conv, SiLU, conv_state), the others z.
template <int MT, bool CONV>
__global__ __launch_bounds__(64 * SG_WAVES) void step_gemm_kernel(StepGemm p) {
  __shared__ f32x4 red[SG_WAVES][MT][64];
  const int w = wave_id(), l = lane_id(), q = l >> 4, l16 = l & 15;
  int tile = blockIdx.x, sg = 0;
  while (sg + 1 < p.nseg && tile >= p.tiles[sg]) tile -= p.tiles[sg++];
  const StepSeg s = p.seg[sg];
  const int n0 = 16 * tile;
  const bf16* wp = reinterpret_cast<const bf16*>(s.W) + (int64_t)min(n0 + l16, s.rows - 1) * p.K + 8 * q;
  const bf16* xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    xp[i] = reinterpret_cast<const bf16*>(p.X) + (int64_t)min(16 * i + l16, p.batch - 1) * p.x_stride + 8 * q;
  // the conv's operands of the waves that run the epilogue (wave i: sequence 16 i + l % 16, rows n0 + 4 q ..), loaded
  // before the product's: their latency hides behind it (the epilogue alone took 4 us of 10)
  bf16 cv[CONV ? 7 : 1][4], cwv[CONV ? 8 : 1][4];
  const int me = min(16 * w + l16, p.batch - 1), ne = n0 + 4 * q;
  const bool conv_wave = CONV && w < MT && n0 < p.d_inner;
  if constexpr (CONV) {
    if (conv_wave) {
      const bf16* cs = reinterpret_cast<const bf16*>(p.conv_state) + (int64_t)me * p.cs_sb + ne;
      const bf16* cw = reinterpret_cast<const bf16*>(p.conv_w) + (int64_t)ne * p.width;
#pragma unroll
      for (int r = 0; r < 7; ++r)
        if (r < p.cs_len) {
#pragma unroll
          for (int j = 0; j < 4; ++j) cv[r][j] = cs[(int64_t)r * p.cs_sl + j];
        }
#pragma unroll
      for (int r = 0; r < 8; ++r)                        // weight r from the last: row r = x, 1 = the newest cached row
        if (r < p.width) {
#pragma unroll
          for (int j = 0; j < 4; ++j) cwv[r][j] = cw[j * p.width + p.width - 1 - r];
        }
    }
  }
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = MT == 1 ? 8 : MT == 2 ? 4 : 2;       // k-steps whose loads fly together
  const int nst = p.K / 32;
  int st = w;
  for (; st + (U - 1) * SG_WAVES < nst; st += U * SG_WAVES) {
    frag8 a[U], x[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 32 * (st + u * SG_WAVES);
      a[u] = *reinterpret_cast<const frag8*>(wp + k);
#pragma unroll
      for (int i = 0; i < MT; ++i) x[u][i] = *reinterpret_cast<const frag8*>(xp[i] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = mma16(a[u], x[u][i], acc[i]);
  }
  for (; st < nst; st += SG_WAVES) {
    const frag8 a = *reinterpret_cast<const frag8*>(wp + 32 * st);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = mma16(a, *reinterpret_cast<const frag8*>(xp[i] + 32 * st), acc[i]);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) red[w][i][l] = acc[i];
  __syncthreads();

  // lane l of tile i: rows n0 + 4 (l / 16) .. + 3 of sequence 16 i + l % 16
  const int i = threadIdx.x >> 6;
  if (i >= MT) return;
  f32x4 y = red[0][i][l];
#pragma unroll
  for (int j = 1; j < SG_WAVES; ++j) y += red[j][i][l];
  const int m = 16 * i + l16, n = n0 + 4 * q;
  if (m >= p.batch) return;
  const bf16* bias = reinterpret_cast<const bf16*>(s.bias);
  bf16 o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (bf16)(y[j] + (bias && n + j < s.rows ? (float)bias[n + j] : 0.f));
  if constexpr (CONV) {
    const int di = p.d_inner;                            // a multiple of 16: a tile is all x or all z
    if (n >= di) {
      bf16* zr = reinterpret_cast<bf16*>(p.z) + (int64_t)m * di + n - di;
#pragma unroll
      for (int j = 0; j < 4; ++j) zr[j] = o[j];
      return;
    }
    const int S = p.cs_len;                              // cached rows: S <= width - 1
    const bf16* cb = reinterpret_cast<const bf16*>(p.conv_b);
    const int So = min(S + 1, p.width - 1);              // rows of the new conv_state: the last So of (cached, x)
    bf16* co = reinterpret_cast<bf16*>(p.conv_out) + (int64_t)m * So * di + n;
    bf16* xa = reinterpret_cast<bf16*>(p.x_act) + (int64_t)m * di + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float acc = cb ? (float)cb[n + j] : 0.f;
#pragma unroll
      for (int r = 0; r < 7; ++r)                        // cached row r is x of token r - S
        if (r < S) {
          float wr = 0.f;
#pragma unroll
          for (int k = 1; k < 8; ++k) wr = S - r == k ? (float)cwv[k][j] : wr;
          acc += wr * (float)cv[r][j];
          const int ro = r - (S + 1 - So);
          if (ro >= 0) co[(int64_t)ro * di + j] = cv[r][j];
        }
      acc += (float)cwv[0][j] * (float)o[j];
      co[(int64_t)(So - 1) * di + j] = o[j];
      xa[j] = (bf16)silu_f(acc);
    }
  } else {
    bf16* yr = reinterpret_cast<bf16*>(s.out) + (int64_t)m * s.rows + n;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < s.rows) yr[j] = o[j];
  }
}

template <bool CONV>
hipError_t launch_step_gemm(const StepGemm& p, hipStream_t st) {
  unsigned tiles = 0;
  for (int i = 0; i < p.nseg; ++i) tiles += (unsigned)p.tiles[i];
  if (p.batch <= 16) hipLaunchKernelGGL((step_gemm_kernel<1, CONV>), dim3(tiles), dim3(64 * SG_WAVES), 0, st, p);
  else if (p.batch <= 32) hipLaunchKernelGGL((step_gemm_kernel<2, CONV>), dim3(tiles), dim3(64 * SG_WAVES), 0, st, p);
  else hipLaunchKernelGGL((step_gemm_kernel<4, CONV>), dim3(tiles), dim3(64 * SG_WAVES), 0, st, p);
  return hipGetLastError();
}

size_t up256(size_t n) { return (n + 255) / 256 * 256; }

}  // namespace

size_t layer_step_workspace_bytes(const LayerStepParams& p) {
  const size_t b = p.batch, di = p.d_inner, gn = (size_t)p.ngroups * p.dstate;
  return 3 * up256(2 * b * di) + up256(2 * b * p.dt_rank) + 2 * up256(2 * b * gn);
}

hipError_t launch_layer_step(const LayerStepParams& p, void* workspace, hipStream_t st) {
  const size_t b = p.batch, di = p.d_inner, gn = (size_t)p.ngroups * p.dstate;
  char* w = reinterpret_cast<char*>(workspace);
  auto take = [&](size_t n) { char* r = w; w += up256(2 * n); return (void*)r; };
  void *x_act = take(b * di), *z = take(b * di), *y = take(b * di), *dtl = take(b * p.dt_rank), *Bm = take(b * gn),
       *Cm = take(b * gn);
  StepGemm g = {};
  g.batch = p.batch;
  auto seg = [&](int i, const void* W, const void* bias, size_t rows, void* out) {
    g.seg[i].W = W; g.seg[i].bias = bias; g.seg[i].rows = (int)rows; g.seg[i].out = out;
    g.tiles[i] = (int)((rows + 15) / 16);
    g.nseg = i + 1;
  };
  g.K = p.d_model; g.X = p.u; g.x_stride = p.u_sb;
  seg(0, p.in_w, p.in_b, 2 * di, nullptr);
  g.d_inner = p.d_inner; g.width = p.width; g.cs_len = p.cs_len;
  g.conv_w = p.conv_w; g.conv_b = p.conv_b; g.conv_state = p.conv_state; g.cs_sb = p.cs_sb; g.cs_sl = p.cs_sl;
  g.conv_out = p.conv_out; g.x_act = x_act; g.z = z;
  hipError_t e = launch_step_gemm<true>(g, st);
  if (e != hipSuccess) return e;

  g.K = p.d_inner; g.X = x_act; g.x_stride = p.d_inner;
  seg(0, p.dt_w0, p.dt_b0, p.dt_rank, dtl);
  seg(1, p.B_w, p.B_b, gn, Bm);
  seg(2, p.C_w, p.C_b, gn, Cm);
  e = launch_step_gemm<false>(g, st);
  if (e != hipSuccess) return e;

  SsuParams s = {};
  s.batch = p.batch; s.nheads = p.nheads; s.headdim = p.headdim; s.dstate = p.dstate; s.ngroups = p.ngroups;
  s.dtype = DT_BF16; s.dt_softplus = 1;
  s.state_in = p.state_in; s.state_out = p.state_out;
  s.x = x_act; s.x_stride_b = p.d_inner;
  s.A = p.A_log;
  s.B = Bm; s.B_stride_b = (int64_t)gn;
  s.C = Cm; s.C_stride_b = (int64_t)gn;
  s.D = p.D; s.dt_bias = p.dt_bias;
  s.y = y; s.y_stride_b = p.d_inner;
  s.z = z; s.z_stride_b = p.d_inner;
  s.dt_low = dtl; s.dt_w = p.dt_w1; s.dt_wb = p.dt_b1; s.dt_rank = p.dt_rank;
  e = launch_ssu(s, st);
  if (e != hipSuccess) return e;

  g.K = p.d_inner; g.X = y; g.x_stride = p.d_inner;
  seg(0, p.out_w, p.out_b, p.d_model, p.out);
  return launch_step_gemm<false>(g, st);
}

}  // namespace mh
