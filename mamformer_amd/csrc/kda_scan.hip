// KDA linear-attention chunked scans for gfx950: the decay-gated operator
// (kda_gated_kernel) and the reference's normalised phi-kernel scan
// (kda_ref_kernel, further below).
//
//   S_t = diag(exp(g_t)) S_{t-1} + k_t^T v_t          (S: dk x dv, fp32)
//   o_t = (q1_t - lam q2_t) S_t                          (inclusive of token t)
// The differential form is linear in q, so q_e = q1 - lam q2 is formed once.
// With g = 0 this is the un-normalised causal linear attention whose
// normalised phi(x)=elu(x)+1 form is the reference's LinearDiffAttention scan
// (mamformer/layers/kda_diff.py:357-478, mamformer/kernels/triton_ssd.py:121-181).
//
// Per window of tokens (a 64-token tile, or a piece of one), with G the
// in-tile inclusive cumsum of g (per channel k), base / end its values just
// before / at the window's last token and m near the midpoint of its range:
//     A^T[s][t] = sum_k (k_s e^{m-G_s})[k] (q_e,t e^{G_t-m})[k]   (s <= t)   MFMA, K = dk
//     o^T[v][t] = sum_s v^T[v][s] A^T[s][t]                                    MFMA
//               + sum_k (S[k][v] e^{m-base}) (q_e,t e^{G_t-m})[k]              MFMA (state read-out)
//     S[k][v]  <- e^{end-m} (e^{m-base} S[k][v] + sum_s (k_s e^{m-G_s})[k] v_s[v])   MFMA
// Windows are cut so that the spread of G within one never exceeds KRANGE,
// which keeps every factor finite.
#include "common.h"
#include "launch.h"
#include "tiles.h"

namespace mh {

namespace {

constexpr int SEGK = 64;          // tokens per segment (max)
constexpr int DK = 128;
constexpr int DVH = 64;           // v columns per workgroup
constexpr float LOG2E = 1.44269504088896340736f;
// Max spread of G per channel within a window.  Its factors then lie within e^{+-KRANGE / 2} and the one between two
// windows' states (e^{m - base} times e^{end - m} of the window before) within e^{+-KRANGE}, all normal fp32 numbers; bf16
// has the same exponents, so a wide window rounds as a narrow one does (error of o 3.0e-3 to 3.4e-3 at 50 and at 80).
constexpr float KRANGE = 80.f;

// ----------------------------------------------------------------- gated mode
// One workgroup of 8 waves per (b, h, V-half) walks the sequence in 64-token
// tiles, as a pipeline of two roles.  Waves 4..7 prepare: they hold the next
// tile's rows in registers, form the in-tile cumsum of g and write Qt, Kt and V
// of tile n + 1 to LDS.  Waves 0..3 multiply: wave w owns v-tile vt = w & 1 and
// k-half kh = w >> 1, keeps the state tiles S[kh][vt], forms the read-out of tile
// n over its k-half and the state update; waves 1..3 also form the three masked
// A^T tiles.  The k-halves' partials are exchanged through LDS and wave (vt, kh)
// finishes token tile tt = kh.  A tile is one factorisation window, with m the
// midpoint of five of its G (its first token's and those at the end of each 16
// tokens: the range's own for gates of one sign), unless some G lies further than
// KRANGE / 2 from m; it is then cut into shorter windows, which both roles walk
// together.
//
// One workgroup per CU (the grid is 2 B H), so what a tile costs is its chain of
// barriers and LDS round trips, and with every wave in the same phase the
// exponentials and conversions (VALU) never ran beside the products (MFMA, LDS):
// 4.5 us a tile in that form.  Here one wave of each role shares each SIMD and a
// step has two barriers: scaling of tile n + 1 beside the products of tile n,
// then the cumsum of tile n + 2 beside the output of tile n.  The factor between
// two windows' states is applied once, where the read-out needs it; the
// token-contracted operands are read transposed by the LDS.
constexpr int KW = 8;                 // waves per workgroup

struct KdaGatedTile {
  static constexpr int PK = DK + 24, PV = DVH + 32;   // pitches of KdaRefSmem (transposing and row reads spread over the banks)
  bf16 Qt[SEG * PK];                  // q_e e^{G - m}, zero rows outside the window
  bf16 Kt[SEG * PK];                  // k e^{m - G}, zero rows outside the window
  bf16 V[SEG * PV];                   // v[:, V-half]
};
struct KdaGatedSmem {
  alignas(16) KdaGatedTile t[2];      // by the tile's parity; a cut tile's G lies in the other one's Qt and Kt
  Frag<bf16> A[3][2][64];             // masked A^T tiles (s0,t0), (s0,t1), (s1,t1) as B-operand fragments
  AccPark red[2][2];                  // read-out partials for the wave of the other k-half: vt, tt
  bf16 O[4][32 * 32];                 // o blocks staged for coalesced stores (XHalf rows 0..31)
  alignas(16) float wtot[4][DK];      // sums of g over each preparing wave's 16 tokens
  alignas(16) float g1[DK];           // g of the tile's first token
  alignas(16) float mm[4][DK];        // window midpoint m (tiles that are cut), a copy per preparing wave
  alignas(16) float em[2][DK];        // by the tile's parity: e^{m - base + pl}
  alignas(16) float pl[2][DK];        // by the tile's parity: end - m of the window before the tile
  int wend, cut[2];                   // cut: by the tile's parity
};
static_assert(sizeof(bf16) * 2 * SEG * KdaGatedTile::PK >= sizeof(float) * SEG * DK, "G fits beside a tile");

// A preparing thread's rows: 8 tokens x 4 channels of q1, q2, k and g, two 16-byte chunks of v.
struct KdaStage {
  bf16x4 q1[8], q2[8], k[8];
  uint4 v[2];
  f32x4 g[8];
};

// 8 consecutive elements of a row, and the 4 + 4 (8 apart) that match an accumulator's row order, as fragments.
__device__ __forceinline__ Frag<bf16> rows8(const bf16* p) {
  Frag<bf16> f;
  f.v = *reinterpret_cast<const bf16x8*>(p);
  return f;
}
__device__ __forceinline__ Frag<bf16> kset8(const bf16* p) {
  const bf16x4 lo = *reinterpret_cast<const bf16x4*>(p), hi = *reinterpret_cast<const bf16x4*>(p + 8);
  Frag<bf16> f;
  f.v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return f;
}

}  // namespace

// SPLIT: the workgroup walks segment blockIdx.y from the earlier segments' sums; without it the whole sequence (a
// template, as the run-time bounds and the entering sums made the unsplit walk 0.7% slower).
template <bool SPLIT>
__global__ __launch_bounds__(64 * KW) void kda_gated_kernel(KdaParams p) {
  __shared__ KdaGatedSmem sm;
  using TL = KdaGatedTile;
  using XO = XHalf<bf16>;
  const int nbh = p.batch * p.nheads;
  int bh, vh;
  const int L = blockIdx.x;
  if ((nbh & 7) == 0) {               // keep both V-halves of a (b, h) on one XCD (ids congruent mod 8)
    bh = (L & 7) | ((L >> 4) << 3);
    vh = (L >> 3) & 1;
  } else {
    bh = L >> 1;
    vh = L & 1;
  }
  const int h = bh % p.nheads;
  const int w = wave_id(), l = lane_id(), half = l >> 5, l32 = l & 31;
  const int S = p.seqlen;
  const int64_t rowbase = (int64_t)bh * S;          // token row index base in (B,H,S,*) tensors
  const int seg = SPLIT ? blockIdx.y : 0;           // this workgroup's segment: tokens [p0, p1)
  const int p0 = SPLIT ? seg * p.seg_chunks * SEG : 0, p1 = SPLIT ? min(S, p0 + p.seg_chunks * SEG) : S;
  const int nt = (p1 - p0 + SEG - 1) / SEG;
  const int v0 = vh * DVH;
  auto is_cut = [&](int n) { return __builtin_amdgcn_readfirstlane(sm.cut[n & 1]) != 0; };
  // Both roles run the same barriers: one after the first cumsum, then per step n (products of tile n) two for each
  // window of a cut tile but the last, one for that, and two.

  if (w >= 4) {
    // ------------------------------------------------------------ preparing waves
    const bool has_q2 = p.q2 != nullptr, has_g = p.g != nullptr, plain = has_g && has_q2;
    const float lam = p.lam_h ? p.lam_h[h] : p.lam;
    const int pt = threadIdx.x & 255, pw = w - 4;
    const int r0 = 8 * (pt >> 5), c4 = 4 * (pt & 31);   // tokens r0 .., channels c4 ..
    int to = r0 * TL::PK + c4;                           // its place in an operand tile; laundered, so that the rows lie
    asm volatile("" : "+v"(to));                         // at immediate offsets and no address a row is held
    const bf16* q1g = reinterpret_cast<const bf16*>(p.q1) + rowbase * DK;
    const bf16* q2g = reinterpret_cast<const bf16*>(p.q2) + rowbase * DK;
    const bf16* kg = reinterpret_cast<const bf16*>(p.k) + rowbase * DK;
    const bf16* vg = reinterpret_cast<const bf16*>(p.v) + rowbase * 128 + v0;
    const float* gg = p.g + rowbase * DK;
    KdaStage stg;
    // Plain loads (a direct-to-LDS load in flight would make every later LDS access wait for it) from a uniform base
    // and a 32-bit lane offset; rows past the sequence read its last one, a tile past it that row alone.
    auto base_of = [&](int n) { return min(p0 + n * SEG, S - 1); };
    auto off_of = [&](int pos, int i) { return (uint32_t)(min(r0 + i, S - 1 - pos) * DK + c4); };
    auto load_g = [&](auto FULLc, int n) {
      const int pos = base_of(n);
      if (decltype(FULLc)::value || has_g) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stg.g[i] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(gg + (int64_t)pos * DK) + 4 * off_of(pos, i));
      }
    };
    auto load_v = [&](int n) {
      const int pos = base_of(n);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        stg.v[i] = *reinterpret_cast<const uint4*>(
            reinterpret_cast<const char*>(vg + (int64_t)pos * 128) +
            (uint32_t)(min((pt >> 3) + 32 * i, S - 1 - pos) * 256 + 16 * (pt & 7)));
    };
    auto load_row = [&](auto FULLc, int pos, int i) {
      const uint32_t o = 2 * off_of(pos, i);
      stg.q1[i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const char*>(q1g + (int64_t)pos * DK) + o);
      if (decltype(FULLc)::value || has_q2)
        stg.q2[i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const char*>(q2g + (int64_t)pos * DK) + o);
      stg.k[i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const char*>(kg + (int64_t)pos * DK) + o);
    };
    f32x4 G[8], low;                                     // sums of g over this thread's tokens, before them
    // in-tile inclusive cumsum of g, g = 0 past the end (G stays flat); then the next tile's g
    auto cumsum = [&](auto FULLc, int n) {
      constexpr bool FULL = decltype(FULLc)::value;
      const int len = min(SEG, S - (p0 + n * SEG));
      f32x4 run = {0.f, 0.f, 0.f, 0.f}, both;            // both: the wave's 16 tokens
      if (FULL && len == SEG) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          run += stg.g[i];
          G[i] = run;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if ((FULL || has_g) && r0 + i < len) run += stg.g[i];
          G[i] = run;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float first = from_half(run[j], 0);        // every lane active: the swap reads both halves
        low[j] = half ? first : 0.f;
        both[j] = sum_halves(run[j]);
      }
      if (half == 0) {
        *reinterpret_cast<f32x4*>(&sm.wtot[pw][c4]) = both;
        if (pw == 0) *reinterpret_cast<f32x4*>(&sm.g1[c4]) = G[0];
      }
      load_g(FULLc, n + 1);
    };
    // Qt = q_e e^{G - m}, Kt = k e^{m - G}, zero rows past the end, of tile n as one window from base 0.  Every factor is
    // then within e^{+-KRANGE / 2}, or the tile is cut.  m is a midpoint of sampled G and not half of end, for gates that
    // rise and fall within a tile and for drops in its first token, which half of end would cut (b4 H32 S8192 with such
    // gates 1113 us, 404 whole), and for a NaN, which minima and maxima drop: the tokens before it stay as they are.  The
    // samples cost 0.8% of the kernel's time.  Each row's registers take the next tile's row.
    auto scale = [&](auto FULLc, int n) {
      constexpr bool FULL = decltype(FULLc)::value;
      const int par = n & 1, len = min(SEG, S - (p0 + n * SEG)), next = base_of(n + 1);
      TL& T = sm.t[par];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<uint4*>(&T.V[((pt >> 3) + 32 * i) * TL::PV + 8 * (pt & 7)]) = stg.v[i];
      f32x4 end = {0.f, 0.f, 0.f, 0.f}, mn = *reinterpret_cast<const f32x4*>(&sm.g1[c4]), mx = mn;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j && j == pw) {
          low += end;
          asm volatile("" : "+v"(low));                  // a scalar branch, not four selects
        }
        end += *reinterpret_cast<const f32x4*>(&sm.wtot[j][c4]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          mn[k] = fminf(mn[k], end[k]);
          mx[k] = fmaxf(mx[k], end[k]);
        }
      }
      const f32x4 m = 0.5f * (mn + mx), c = (low - m) * LOG2E;
      float top = 0.f;                                   // the largest |G - m|, in units of ln 2
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        bf16x4 qo, ko;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float d = __builtin_fmaf(G[i][j], LOG2E, c[j]);
          const float qe = FULL || has_q2 ? __builtin_fmaf(-lam, (float)stg.q2[i][j], (float)stg.q1[i][j])
                                          : (float)stg.q1[i][j];
          top = fmaxf(top, fabsf(d));
          qo[j] = (bf16)(qe * __builtin_amdgcn_exp2f(d));
          ko[j] = (bf16)((float)stg.k[i][j] * __builtin_amdgcn_exp2f(-d));
        }
        uint2 qw = __builtin_bit_cast(uint2, qo), kw = __builtin_bit_cast(uint2, ko);
        if (!FULL && r0 + i >= len) qw = kw = uint2{0, 0};
        *reinterpret_cast<uint2*>(T.Qt + to + i * TL::PK) = qw;
        *reinterpret_cast<uint2*>(T.Kt + to + i * TL::PK) = kw;
        load_row(FULLc, next, i);
        __builtin_amdgcn_sched_barrier(0);               // a row at a time: interleaved, the rows spill
      }
      load_v(n + 1);
      if (pw == 0 && half == 0) {
        const f32x4 pv = *reinterpret_cast<const f32x4*>(&sm.pl[par][c4]);
        f32x4 e;
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = __expf(m[j] + pv[j]);
        *reinterpret_cast<f32x4*>(&sm.em[par][c4]) = e;
        *reinterpret_cast<f32x4*>(&sm.pl[par ^ 1][c4]) = end - m;
      }
      if (top > 0.5f * KRANGE * LOG2E) sm.cut[par] = 1;  // benign race: every writer stores 1
    };
    // A tile that is cut, between its X and Y: its G to LDS, in the operands of the tile before it (read by nobody after
    // X), and its rows again, in the registers that took the next tile's by now.
    auto park = [&](int n) {
      float* Gs = reinterpret_cast<float*>(sm.t[(n & 1) ^ 1].Qt);
#pragma unroll
      for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(&Gs[(r0 + i) * DK + c4]) = G[i] + low;
      int pos = base_of(n);
      asm volatile("" : "+s"(pos));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        load_row(std::false_type{}, pos, i);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The windows of a cut tile: each the longest from a on whose per-channel spread of G stays within KRANGE (at least
    // one token).  Every wave finds its end for itself, two channels a lane, while the window before is multiplied, so a
    // window takes two barriers; the rows wait in registers until the last window is formed, and the next tile's rows
    // are on their way again behind its products.  With the ends found by two waves between barriers of their own, g
    // summed from memory and the rows read again for each window, b4 H32 S8192 took 7038 us at a decay of 3.1 a token
    // (four windows a tile), the kernel without roles 3709, this 1677 (three windows); one drop of 80 in every eighth
    // tile 896, 908 and 530; 1.1 a token, cut at a spread of 50 and whole at 80, 5312, 2506 and 403.
    auto windows = [&](int n) {
      const int par = n & 1, len = min(SEG, S - (p0 + n * SEG));
      TL& T = sm.t[par];
      const float* Gs = reinterpret_cast<const float*>(sm.t[par ^ 1].Qt);
      int pt = threadIdx.x & 255;                        // formed here: nothing of this path is held by the others
      asm volatile("" : "+v"(pt));
      const int r0 = 8 * (pt >> 5), c4 = 4 * (pt & 31), c2 = 2 * (pt & 63);
      int go = r0 * DK + c4;                             // (one address, rows at immediate offsets)
      asm volatile("" : "+v"(go));
      const float* gr = Gs + go;
      typedef float f32x2_t __attribute__((ext_vector_type(2)));
      auto g2 = [&](int t) { return *reinterpret_cast<const f32x2_t*>(&Gs[t * DK + c2]); };
      f32x2_t m, e, pv = *reinterpret_cast<const f32x2_t*>(&sm.pl[par][c2]);   // pv: end - m of the window before
      int b;
      auto next = [&](int a) {                           // the window from a: b, m, e = e^{m - base + pv}, pv
        constexpr int U = 8;                             // tokens whose spread is looked at together
        f32x2_t mn = {INFINITY, INFINITY}, mx = {-INFINITY, -INFINITY}, v[U], nv[U];
        auto fetch = [&](f32x2_t (&x)[U], int t) {
#pragma unroll
          for (int u = 0; u < U; ++u) x[u] = g2(min(t + u, len - 1));
        };
        auto widen = [&](f32x2_t& lo, f32x2_t& hi, f32x2_t x) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            lo[j] = fminf(lo[j], x[j]);
            hi[j] = fmaxf(hi[j], x[j]);
          }
        };
        auto over = [&](f32x2_t lo, f32x2_t hi) { return __ballot(fmaxf(hi[0] - lo[0], hi[1] - lo[1]) > KRANGE) != 0; };
        b = len;
        fetch(v, a);
        for (int t = a; t < len; t += U) {
          fetch(nv, t + U);
          f32x2_t lo = mn, hi = mx;
#pragma unroll
          for (int u = 0; u < U; ++u) widen(lo, hi, v[u]);
          if (over(lo, hi)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              lo = mn;
              hi = mx;
              widen(lo, hi, v[u]);
              if (over(lo, hi)) {
                b = max(min(t + u, len), a + 1);
                break;
              }
              mn = lo;
              mx = hi;
            }
            break;
          }
          mn = lo;
          mx = hi;
#pragma unroll
          for (int u = 0; u < U; ++u) v[u] = nv[u];
        }
        const f32x2_t end = g2(b - 1);
        f32x2_t base = {0.f, 0.f};
        if (a) base = g2(a - 1);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          m[j] = 0.5f * (mn[j] + mx[j]);
          e[j] = __expf(m[j] - base[j] + pv[j]);
          pv[j] = end[j] - m[j];
        }
      };
      next(0);
      for (int a = 0; a < len;) {
        const int bw = b;
        *reinterpret_cast<f32x2_t*>(&sm.mm[pw][c2]) = m;  // each wave its own copy, read by it alone
        if (pw == 0) {
          *reinterpret_cast<f32x2_t*>(&sm.em[par][c2]) = e;
          if (pt == 0) sm.wend = bw;
        }
        const f32x4 m4 = *reinterpret_cast<const f32x4*>(&sm.mm[pw][c4]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = r0 + i;
          bf16x4 qo = {}, ko = {};
          if (r >= a && r < bw) {
            const f32x4 g4 = *reinterpret_cast<const f32x4*>(gr + i * DK);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float d = g4[j] - m4[j];
              const float qe = has_q2 ? (float)stg.q1[i][j] - lam * (float)stg.q2[i][j] : (float)stg.q1[i][j];
              qo[j] = (bf16)(qe * __expf(d));
              ko[j] = (bf16)((float)stg.k[i][j] * __expf(-d));
            }
          }
          *reinterpret_cast<bf16x4*>(T.Qt + to + i * TL::PK) = qo;
          *reinterpret_cast<bf16x4*>(T.Kt + to + i * TL::PK) = ko;
          __builtin_amdgcn_sched_barrier(0);
        }
        if (bw == len) {
          int pos = base_of(n + 1);
          asm volatile("" : "+s"(pos));                  // addresses formed here, not held through the windows
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            load_row(std::false_type{}, pos, i);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (bw == len && pw == 0) *reinterpret_cast<f32x2_t*>(&sm.pl[par ^ 1][c2]) = pv;
        lds_barrier();                                   // W1: the window's operands
        if (bw < len) {
          next(bw);
          lds_barrier();                                 // W2: they have been read
        }
        a = bw;
      }
    };

    if (pt == 0) sm.cut[0] = sm.cut[1] = 0;
    if (pt < DK) sm.pl[0][pt] = 0.f;
    using Any = std::false_type;
    using Full = std::true_type;
    load_g(Any{}, 0);
    load_v(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) load_row(Any{}, p0, i);
    cumsum(Any{}, 0);
    lds_barrier();
    for (int n = -1; n < nt; ++n) {
      // Steps whose tile n + 1 is whole (a tile n + 2 follows) and whose tile n is not cut, in a loop without other loads
      // than those of a cut tile's rows, which are as many as they replace: every wait for a row's registers then counts
      // the younger loads.  All loads have landed on entry.
      if (plain) {
        wait_vmem();
        for (; n + 2 < nt && !(n >= 0 && is_cut(n)); ++n) {
          scale(Full{}, n + 1);
          lds_barrier();                                 // X
          const int flag = sm.cut[(n + 1) & 1];          // (read ahead of the store: its latency is this step's)
          if (n >= 0 && pt == 0) sm.cut[n & 1] = 0;
          if (__builtin_expect(__builtin_amdgcn_readfirstlane(flag) != 0, 0)) park(n + 1);
          cumsum(Full{}, n + 2);
          lds_barrier();                                 // Y
        }
      }
      if (n >= 0 && is_cut(n)) windows(n);
      if (n + 1 < nt) scale(Any{}, n + 1);
      lds_barrier();                                     // X: tile n + 1 is ready; tile n's partials and A^T tiles
      if (n >= 0 && pt == 0) sm.cut[n & 1] = 0;          // read before X; set again for tile n + 2 after Y
      if (n + 1 < nt && is_cut(n + 1)) park(n + 1);
      if (n + 2 < nt) cumsum(Any{}, n + 2);
      lds_barrier();                                     // Y
    }
    return;
  }

  // -------------------------------------------------------------- multiplying waves
  const int vt = w & 1, kh = w >> 1;
  bf16* og = reinterpret_cast<bf16*>(p.o);
  // state tiles of k-tile 2 kh + i, v-tile vt of this V-half
  f32x16 St[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    St[i] = zero16();
    if (p.init_state) {
      const float* s0 = p.init_state + (int64_t)bh * DK * 128;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * (2 * kh + i) + acc_row(half, r);
        St[i][r] = s0[kr * 128 + v0 + 32 * vt + l32];
      }
    }
  }
  // the state entering the segment: S <- e^{log-decay of segment j} S + (segment j's own sum), j in order
  for (int j = 0; j < seg; ++j) {
    const float* rec = p.seg_sum + ((int64_t)j * nbh + bh) * KDA_REC;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float sv[16], ev[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * (2 * kh + i) + acc_row(half, r);
        sv[r] = rec[kr * 128 + v0 + 32 * vt + l32];
        ev[r] = rec[128 * 128 + kr];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) St[i][r] = St[i][r] * __expf(ev[r]) + sv[r];
    }
  }

  Frag<bf16> vf[4];
  f32x16 o;                                              // token tile tt = kh of the read-out
  // o^T[v][t] = sum_k (S[k][v] e^{m_k - base_k}) Qt[t][k] over this wave's k-half, and
  // St[k][v] <- S[k][v] e^{m_k - base_k} + sum_s Kt[s][k] v_s[v], with S = e^{pl} St of the window before
  auto products = [&](int par) {
    const TL& T = sm.t[par];
    if (w) {
      const int it = w - 1;
      const int st = (it == 2) ? 1 : 0, ttA = (it == 0) ? 0 : 1;
      f32x16 acc = zero16();
#pragma unroll
      for (int c = 0; c < DK / 16; ++c)
        acc = mma(rows8(T.Kt + (32 * st + l32) * TL::PK + 8 * half + 16 * c),
                  rows8(T.Qt + (32 * ttA + l32) * TL::PK + 8 * half + 16 * c), acc);
      if (st == ttA) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(half, r) > l32) acc[r] = 0.f;
      }
      sm.A[it][0][l] = acc_to_frag<bf16>(acc, 0);
      sm.A[it][1][l] = acc_to_frag<bf16>(acc, 1);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) vf[c] = col_frag_tr(T.V, TL::PV, 32 * vt, 16 * c);
    f32x16 ot[2];
    ot[0] = ot[1] = zero16();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int kt = 2 * kh + i;
      f32x16 sv = St[i];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 e4 = *reinterpret_cast<const f32x4*>(&sm.em[par][32 * kt + 8 * q + 4 * half]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sv[4 * q + j] *= e4[j];
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Frag<bf16> sa = acc_to_frag<bf16>(sv, c);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          ot[tt] = mma(sa, kset8(T.Qt + (32 * tt + l32) * TL::PK + 4 * half + 32 * kt + 16 * c), ot[tt]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) sv = mma(col_frag_tr(T.Kt, TL::PK, 32 * kt, 16 * c), vf[c], sv);
      St[i] = sv;
    }
    if (kh == 0) {
      park_acc(sm.red[vt][1], ot[1], l);
      o = ot[0];
    } else {
      park_acc(sm.red[vt][0], ot[0], l);
      o = ot[1];
    }
  };
  // intra-window term and the other k-half's partial, then output rows [a, b) of tile pos, staged for 16-byte stores
  auto output = [&](int pos, int a, int b) {
    if (kh == 0) {
      o = mma(vf[0], sm.A[0][0][l], o);
      o = mma(vf[1], sm.A[0][1][l], o);
    } else {
      o = mma(vf[0], sm.A[1][0][l], o);
      o = mma(vf[1], sm.A[1][1][l], o);
      o = mma(vf[2], sm.A[2][0][l], o);
      o = mma(vf[3], sm.A[2][1][l], o);
    }
    const f32x16 other = unpark_acc(sm.red[vt][kh], l);
    bf16* ob = sm.O[w];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c0 = 8 * q + 4 * half;                   // 4 consecutive v columns inside one 16-byte chunk
      bf16x4 yv;
#pragma unroll
      for (int j = 0; j < 4; ++j) yv[j] = (bf16)(o[4 * q + j] + other[4 * q + j]);
      *reinterpret_cast<bf16x4*>(ob + XO::chunk(l32, c0 >> 3) + (c0 & 7)) = yv;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int e = l + 64 * i;
      const int r = e >> 2, c = e & 3;                   // row t of the block, 16-byte chunk
      const uint4 val = *reinterpret_cast<const uint4*>(ob + XO::chunk(r, c));
      const int t = 32 * kh + r;
      if (t >= a && t < b)
        *reinterpret_cast<uint4*>(og + (rowbase + pos + t) * 128 + v0 + 32 * vt + 8 * c) = val;
    }
  };

  lds_barrier();
  for (int n = -1; n < nt; ++n) {
    const int pos = p0 + n * SEG, len = min(SEG, S - pos);
    int a = 0;                                           // the rows from here on are left for the output below
    if (n >= 0 && is_cut(n)) {
      for (;;) {
        lds_barrier();                                   // W1
        const int b = __builtin_amdgcn_readfirstlane(sm.wend);
        if (b >= len) break;
        products(n & 1);
        lds_barrier();                                   // W2
        output(pos, a, b);
        a = b;
      }
    }
    if (n >= 0) products(n & 1);
    lds_barrier();                                       // X
    if (n >= 0) output(pos, a, len);
    lds_barrier();                                       // Y
  }

  if (p.final_state && p1 == S) {
    float* sf_out = p.final_state + (int64_t)bh * DK * 128;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * (2 * kh + i) + acc_row(half, r);
        sf_out[kr * 128 + v0 + 32 * vt + l32] = St[i][r] * __expf(sm.pl[nt & 1][kr]);
      }
  }
}

// Empty sequence: final state (and z) = initial (or zero), written by a plain kernel (no copy or memset
// node, so a captured launch behaves the same).
__global__ __launch_bounds__(256) void kda_empty_kernel(const float* __restrict__ s0, float* __restrict__ sf, size_t ns,
                                                       const float* __restrict__ z0, float* __restrict__ zf, size_t nz) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (sf && i < ns) sf[i] = s0 ? s0[i] : 0.f;
  if (zf && i < nz) zf[i] = z0 ? z0[i] : 0.f;
}

// ---------------------------------------------------------------------------
// Reference mode: the reference's normalised linear-attention scan
// (LinearDiffAttention._linear_attention_scan, kda_diff.py:357-478, and the
// Triton kernel it dispatches to, triton_ssd.py:121-181):
//     phi(x) = elu(x) + 1 on the first kernel_dim channels (0 beyond, kda_diff.py:67-89)
//     S_t = S_{t-1} + phi(k_t)^T v_t,   z_t = z_{t-1} + phi(k_t)            (inclusive of t)
//     o_i,t = phi(q_i,t) S_t / (phi(q_i,t) z_t + 1e-8)                     (i = 1, 2)
// Outputs: the pair (o1, o2); or, with o2 == NULL and two queries, the fused
// differential combination (o1 - lam o2) / (1 - lam + 1e-8) (kda_diff.py:534-538);
// or, with q2 == NULL, the single-query o1 (triton_ssd.py:184-257).
// Same segment walk and wave split as the gated kernel with g = 0; the
// normaliser is the row sum of the masked phi(q) phi(k)^T tile plus
// phi(q) . z_prev, with z (fp32) kept in LDS.
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ float phi1(float x) { return x > 0.f ? x + 1.f : __expf(x); }

template <int NQ>
struct KdaRefSmem {
  static constexpr int PK = DK + 24;     // bf16 row pitch (76 words: transposing and row reads spread over the banks)
  static constexpr int PV = DVH + 32;    // 48 words: the transposing reads of V spread over the banks
  bf16 Q[NQ][SEGK * PK];                 // phi(q_i)
  bf16 Kt[SEGK * PK];                    // phi(k), zero rows beyond the segment
  bf16 V[SEGK * PV];                     // v[:, V-half], zero rows beyond the segment
  alignas(16) float z[DK];               // running sum of phi(k) before this segment
  float zq[NQ][SEGK];                    // phi(q_i,t) . z
  float nrm[NQ][3][32];                  // row sums of the masked A tiles
  AccPark red[2][NQ][2];                 // k-half 1 read-out partials: vt, query, t-tile
  Frag<bf16> A[3 * NQ][2][64];           // masked A^T tiles as B-operand fragments (bf16 high part)
  Frag<bf16> Alo[3 * NQ][2][64];         // ... and the bf16 rounding remainder (A = A + Alo to ~2^-17)
  AccPark xb[NQ == 2 ? 2 : 1][2];        // fused differential output: query 2's normalised rows (vt, tt)
};

// Threads of a reference-mode workgroup: 4 waves per query stream (v-tile x k-half each).
template <int NQ>
constexpr int kda_ref_threads = 256 * NQ;

// Register-staged raw rows of one segment: per thread 16-byte chunks of k and of each query (element
// e = tid + NT i: token e >> 4, channels 8 (e & 15) ..) and of v (token e >> 3, columns 8 (e & 7) ..).
template <int NQ>
struct KdaRefStage {
  static constexpr int KC = 4 / NQ, VC = 2 / NQ;
  bf16x8 k[KC], q[NQ][KC];
  uint4 v[VC];
};

template <int NQ>
__device__ __forceinline__ void kda_ref_load(KdaRefStage<NQ>& g, const bf16* const (&qp)[2], const bf16* kk,
                                             const bf16* vv, int64_t rowbase, int pos, int len, int v0, int tid) {
  constexpr int NT = kda_ref_threads<NQ>;
#pragma unroll
  for (int i = 0; i < KdaRefStage<NQ>::KC; ++i) {
    const int e = tid + NT * i;
    const int t = e >> 4, k0 = (e & 15) * 8;
    const int64_t r = (rowbase + pos + min(t, len - 1)) * DK + k0;
    g.k[i] = *reinterpret_cast<const bf16x8*>(kk + r);
#pragma unroll
    for (int j = 0; j < NQ; ++j) g.q[j][i] = *reinterpret_cast<const bf16x8*>(qp[j] + r);
  }
#pragma unroll
  for (int i = 0; i < KdaRefStage<NQ>::VC; ++i) {
    const int e = tid + NT * i;
    const int t = e >> 3, c0 = (e & 7) * 8;
    g.v[i] = t < len ? *reinterpret_cast<const uint4*>(vv + (rowbase + pos + t) * 128 + v0 + c0)
                     : make_uint4(0, 0, 0, 0);
  }
}

}  // namespace

// 4 NQ waves: wave w has v-tile vt = w & 1, k-half kh = (w >> 1) & 1 and query stream qw = w >> 2; the two query
// streams' waves keep their own copy of the state tiles.
template <int NQ>
__global__ __launch_bounds__(256 * NQ) void kda_ref_kernel(KdaParams p) {
  __shared__ KdaRefSmem<NQ> sm;
  using SM = KdaRefSmem<NQ>;
  using TM = bf16;
  constexpr int NT = kda_ref_threads<NQ>, NW = NT / 64;
  constexpr int KC = KdaRefStage<NQ>::KC, VC = KdaRefStage<NQ>::VC;
  const int nbh = p.batch * p.nheads;
  int bh, vh;
  const int L = blockIdx.x;
  if ((nbh & 7) == 0) {               // keep both V-halves of a (b, h) on one XCD (ids congruent mod 8)
    bh = (L & 7) | ((L >> 4) << 3);
    vh = (L >> 3) & 1;
  } else {
    bh = L >> 1;
    vh = L & 1;
  }
  const int h = bh % p.nheads;
  const int w = wave_id(), l = lane_id(), half = l >> 5, l32 = l & 31;
  const int vt = w & 1, kh = (w >> 1) & 1, qw = w >> 2;
  const int tid = threadIdx.x;
  const int S = p.seqlen;
  const int kd = p.kernel_dim;
  const bool fuse_diff = (NQ == 2) && (p.o2 == nullptr);
  const float lam = kda_lambda(p.lam_h, p.lam, p.lam_raw, h);
  const float inv_1ml = 1.f / (1.f - lam + 1e-8f);
  const int64_t rowbase = (int64_t)bh * S;
  const int seg = blockIdx.y;                       // this workgroup's segment: tokens [p0, p1)
  const int p0 = seg * p.seg_chunks * SEGK, p1 = min(S, p0 + p.seg_chunks * SEGK);
  const bf16* const qp[2] = {reinterpret_cast<const bf16*>(p.q1), reinterpret_cast<const bf16*>(p.q2)};
  const bf16* kk = reinterpret_cast<const bf16*>(p.k);
  const bf16* vv = reinterpret_cast<const bf16*>(p.v);
  bf16* op[2] = {reinterpret_cast<bf16*>(p.o), reinterpret_cast<bf16*>(p.o2)};
  const int v0 = vh * DVH;

  f32x16 St[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    St[i] = zero16();
    if (p.init_state) {
      const float* s0 = p.init_state + (int64_t)bh * DK * 128;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * (2 * kh + i) + acc_row(half, r);
        St[i][r] = s0[kr * 128 + v0 + 32 * vt + l32];
      }
    }
  }
  // the state and normaliser entering the segment: plus the earlier segments' sums, in order
  for (int j = 0; j < seg; ++j) {
    const float* rec = p.seg_sum + ((int64_t)j * nbh + bh) * KDA_REC;
    float sv[2][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) sv[i][r] = rec[(32 * (2 * kh + i) + acc_row(half, r)) * 128 + v0 + 32 * vt + l32];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) St[i][r] += sv[i][r];
  }
  if (tid < DK) {
    float z = p.init_z ? p.init_z[(int64_t)bh * DK + tid] : 0.f;
    for (int j = 0; j < seg; ++j) z += p.seg_sum[((int64_t)j * nbh + bh) * KDA_REC + 128 * 128 + tid];
    sm.z[tid] = z;
  }

  static_assert(SEGK * (DK / 8) == KC * NT && SEGK * (DVH / 8) == VC * NT, "staging covers a segment");
  KdaRefStage<NQ> stg;
  if (p0 < p1) kda_ref_load<NQ>(stg, qp, kk, vv, rowbase, p0, min(SEGK, S - p0), v0, tid);
  for (int pos = p0; pos < p1; pos += SEGK) {
    const int len = min(SEGK, S - pos);
    // ---- phase B: phi(q_i), phi(k), v tiles from the staged rows; then stage the next segment's rows
    auto stage = [&](auto MASKc) {     // MASK: zero tokens past the segment end and channels past kernel_dim
      constexpr bool MASK = decltype(MASKc)::value;
#pragma unroll
      for (int ie = 0; ie < KC; ++ie) {
        const int e = tid + NT * ie;
        const int t = e >> 4, k0 = (e & 15) * 8;
        const bool in = t < len;
        const bf16x8 kv8 = stg.k[ie];
        bf16x8 ko;
#pragma unroll
        for (int j = 0; j < 8; ++j) {   // computed unconditionally, then selected: no branch per element
          const float f = phi1((float)kv8[j]);
          ko[j] = (bf16)((!MASK || (in && k0 + j < kd)) ? f : 0.f);
        }
        *reinterpret_cast<bf16x8*>(&sm.Kt[t * SM::PK + k0]) = ko;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
          const bf16x8 qv8 = stg.q[i][ie];
          bf16x8 qo;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float f = phi1((float)qv8[j]);
            qo[j] = (bf16)((!MASK || (in && k0 + j < kd)) ? f : 0.f);
          }
          *reinterpret_cast<bf16x8*>(&sm.Q[i][t * SM::PK + k0]) = qo;
        }
      }
    };
    if (len == SEGK && kd >= DK) stage(std::false_type{});
    else stage(std::true_type{});
#pragma unroll
    for (int ie = 0; ie < VC; ++ie) {
      const int e = tid + NT * ie;
      const int t = e >> 3, c0 = (e & 7) * 8;
      *reinterpret_cast<uint4*>(&sm.V[t * SM::PV + c0]) = stg.v[ie];
    }
    if (pos + SEGK < p1) kda_ref_load<NQ>(stg, qp, kk, vv, rowbase, pos + SEGK, min(SEGK, S - pos - SEGK), v0, tid);
    __syncthreads();

    // ---- phase B2: phi(q_i,t) . z_prev  (4 adjacent lanes per (query, token), 32 channels each: one item
    // per thread)
    {
      const int it = tid;
      const int i = it / (SEGK * 4), t = (it >> 2) % SEGK, qq = it & 3;
      const bf16* row = &sm.Q[i][t * SM::PK + 32 * qq];
      float acc = 0.f;
#pragma unroll
      for (int c = 0; c < 32; c += 8) {
        const bf16x8 q8 = *reinterpret_cast<const bf16x8*>(row + c);
        const f32x4 z0 = *reinterpret_cast<const f32x4*>(&sm.z[32 * qq + c]);
        const f32x4 z1 = *reinterpret_cast<const f32x4*>(&sm.z[32 * qq + c + 4]);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += (float)q8[j] * (j < 4 ? z0[j] : z1[j - 4]);
      }
      acc = sum_quad(acc);
      if (qq == 0) sm.zq[i][t] = acc;
    }

    // ---- phase C: masked A^T tiles (query, s-tile, t-tile) and their row sums
    for (int ti = w; ti < 3 * NQ; ti += NW) {
      const int qi = ti / 3, tile = ti - 3 * qi;
      const int st = (tile == 2) ? 1 : 0, tt = (tile == 0) ? 0 : 1;
      f32x16 acc = zero16();
#pragma unroll
      for (int c = 0; c < DK / 16; ++c) {
        Frag<TM> a, bb;
        a.v = *reinterpret_cast<const bf16x8*>(&sm.Kt[(32 * st + l32) * SM::PK + 16 * c + 8 * half]);
        bb.v = *reinterpret_cast<const bf16x8*>(&sm.Q[qi][(32 * tt + l32) * SM::PK + 16 * c + 8 * half]);
        acc = mma(a, bb, acc);
      }
      const int tl = 32 * tt + l32;
      float rs = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int s_ = 32 * st + acc_row(half, r);
        if (!(s_ <= tl && s_ < len)) acc[r] = 0.f;
        rs += acc[r];
      }
      rs = sum_halves(rs);
      if (half == 0) sm.nrm[qi][tile][l32] = rs;
      // The normaliser uses the fp32 row sums, so the weights that multiply v must carry
      // more than bf16 precision or their rounding (independent per entry) does not cancel
      // against it; the differential combination can amplify that by 1/(1 - lam) <= 100.
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        Frag<TM> hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = acc[8 * c + j];
          hi.v[j] = (bf16)x;
          lo.v[j] = (bf16)(x - (float)hi.v[j]);
        }
        sm.A[ti][c][l] = hi;
        sm.Alo[ti][c][l] = lo;
      }
    }
    __syncthreads();

    // ---- z update (z_prev was consumed by phase B2 before the barrier)
    // by the k-half 0 waves, whose read-out phase below has half the intra-segment MFMAs of the k-half 1 waves;
    // one lane per channel, in token order
    if (tid < DK) {
      float zs = 0.f;
#pragma unroll 8
      for (int t = 0; t < SEGK; ++t) zs += (float)sm.Kt[t * SM::PK + tid];
      sm.z[tid] += zs;
    }

    // ---- phase D: per wave (v-tile vt, k-half kh)
    Frag<TM> vf[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) vf[c] = col_frag_tr(sm.V, SM::PV, 32 * vt, 16 * c);

    // read-out of this wave's query stream qw: o[tt] for both t-tiles over this wave's k-half
    f32x16 o[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      f32x16 acc = zero16();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int kt = 2 * kh + i;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const Frag<TM> sa = acc_to_frag<TM>(St[i], c);
          Frag<TM> qb;
          const bf16* row = &sm.Q[qw][(32 * tt + l32) * SM::PK + 32 * kt + 16 * c];
          const bf16x4 lo = *reinterpret_cast<const bf16x4*>(row + 4 * half);
          const bf16x4 hi = *reinterpret_cast<const bf16x4*>(row + 8 + 4 * half);
#pragma unroll
          for (int j = 0; j < 4; ++j) { qb.v[j] = lo[j]; qb.v[4 + j] = hi[j]; }
          acc = mma(sa, qb, acc);
        }
      }
      o[tt] = acc;
    }
    // wave kh finishes token tile tt = kh: it adds the intra-segment term of that tile and hands its
    // read-out partial of the other tile to the partner wave (same vt and query, other k-half)
    if (kh == 0) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        o[0] = mma(vf[c], sm.A[3 * qw + 0][c][l], o[0]);
        o[0] = mma(vf[c], sm.Alo[3 * qw + 0][c][l], o[0]);
      }
      park_acc(sm.red[vt][qw][1], o[1], l);
    } else {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        o[1] = mma(vf[c], sm.A[3 * qw + 1][c][l], o[1]);
        o[1] = mma(vf[c], sm.Alo[3 * qw + 1][c][l], o[1]);
        o[1] = mma(vf[2 + c], sm.A[3 * qw + 2][c][l], o[1]);
        o[1] = mma(vf[2 + c], sm.Alo[3 * qw + 2][c][l], o[1]);
      }
      park_acc(sm.red[vt][qw][0], o[0], l);
    }
    // state update (no decay): S[k][v] += sum_s phi(k_s)[k] v_s[v]
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int kt = 2 * kh + i;
      f32x16 acc = St[i];
#pragma unroll
      for (int c = 0; c < 4; ++c) acc = mma(col_frag_tr(sm.Kt, SM::PK, 32 * kt, 16 * c), vf[c], acc);
      St[i] = acc;
    }
    __syncthreads();
    // normalised rows of token tile tt = kh for query qw
    float res[16];
    const int tl = 32 * kh + l32;
    const bool valid = tl < len;
    auto finish = [&](auto TTc) {
      constexpr int tt = decltype(TTc)::value;
      if (valid) {
        const float nr = sm.zq[qw][tl] + (tt == 0 ? sm.nrm[qw][0][l32] : sm.nrm[qw][1][l32] + sm.nrm[qw][2][l32]);
        const float inv = 1.f / (nr + 1e-8f);
        const f32x16 other = unpark_acc(sm.red[vt][qw][tt], l);
#pragma unroll
        for (int r = 0; r < 16; ++r) res[r] = (o[tt][r] + other[r]) * inv;
      }
    };
    if (kh == 0) finish(std::integral_constant<int, 0>{});
    else finish(std::integral_constant<int, 1>{});
    if (!fuse_diff) {
      if (valid) {
        bf16* orow = op[qw] + (rowbase + pos + tl) * 128 + v0 + 32 * vt;
#pragma unroll
        for (int r = 0; r < 16; ++r) orow[acc_row(half, r)] = (bf16)res[r];
      }
      __syncthreads();
    } else {
      // the differential combination (o1 - lam o2) / (1 - lam + 1e-8): query 2's waves hand their rows over
      if (qw == 1 && valid) park_acc(sm.xb[vt][kh], res, l);
      __syncthreads();
      if (qw == 0 && valid) {
        bf16* orow = op[0] + (rowbase + pos + tl) * 128 + v0 + 32 * vt;
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const f32x4 r2 = sm.xb[vt][kh].p[r >> 2][l];
#pragma unroll
          for (int j = 0; j < 4; ++j) orow[acc_row(half, r + j)] = (bf16)((res[r + j] - lam * r2[j]) * inv_1ml);
        }
      }
    }
  }

  if (p.final_state && qw == 0 && p1 == S) {
    float* sf_out = p.final_state + (int64_t)bh * DK * 128;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kr = 32 * (2 * kh + i) + acc_row(half, r);
        sf_out[kr * 128 + v0 + 32 * vt + l32] = St[i][r];
      }
  }
  if (p.final_z && vh == 0 && tid < DK && p1 == S) p.final_z[(int64_t)bh * DK + tid] = sm.z[tid];
}

// ---------------------------------------------------------------------------
// Sequence split.  A scan of B H heads is 2 B H workgroups of one per CU (LDS), so fewer than 128 heads leave CUs
// idle for the whole serial walk.  The sequence of each (b, h) is then cut into segments of whole chunks that walk
// side by side; kda_sum_kernel first forms each segment's own contribution to the state, and a segment starts from
// the sum of the earlier ones (gated: S <- e^{sum g} S + S_j).  The sums cost one product per chunk where the walk
// has the staging of the queries, the masked tiles, the read-out and the output besides.
// ---------------------------------------------------------------------------
namespace {

enum { SUM_GATED = 0, SUM_PHI = 1, SUM_CENTERED = 2 };

template <int MODE>
struct KdaSumSmem {
  static constexpr int NB = MODE == SUM_GATED ? 1 : 2;    // buffers
  static constexpr int PK = DK + 24, PV = DVH + 32;       // pitches of KdaRefSmem
  bf16 K[NB][SEGK * PK];        // phi(k), phi'(k) or e^{G_end - G_s} k_s
  bf16 V[NB][SEGK * PV];
  alignas(16) float W[MODE == SUM_GATED ? SEGK : 1][DK];   // e^{G_end - G_s}
  float qtot[4][DK], eg[DK];    // gated: token-quarter sums of g, e^{sum of the chunk}
  float k1[2][SEGK];            // centered: sum_k phi'(k_s)
  float red[3][8][DK];          // per-wave partials of the vector sums
};

// grid (2 nbh, nseg - 1): segment blockIdx.y of (b, h, V-half).  8 waves, one 32x32 state tile each (k-tile w & 3,
// v-tile w >> 2).  Every segment but the last is whole chunks, so no row is masked.
template <int MODE>
__global__ __launch_bounds__(512) void kda_sum_kernel(KdaParams p) {
  using SM = KdaSumSmem<MODE>;
  __shared__ SM sm;
  const int nbh = p.batch * p.nheads;
  int bh, vh;
  const int L = blockIdx.x;
  if ((nbh & 7) == 0) {               // both V-halves of a (b, h) on one XCD, as the scan kernels
    bh = (L & 7) | ((L >> 4) << 3);
    vh = (L >> 3) & 1;
  } else {
    bh = L >> 1;
    vh = L & 1;
  }
  const int w = wave_id(), l = lane_id(), half = l >> 5, l32 = l & 31, tid = threadIdx.x;
  const int kt = w & 3, vt = w >> 2;
  const int seg = blockIdx.y;
  const int64_t row0 = (int64_t)bh * p.seqlen + (int64_t)seg * p.seg_chunks * SEGK;
  const int nch = p.seg_chunks, kd = p.kernel_dim;
  const int c8 = tid & 15, kr = tid >> 4;                // k rows kr, kr + 32, columns 8 c8 ..
  const int v8 = tid & 7, vr = tid >> 3;                 // v row vr, columns 8 v8 .. of the half
  const int kc = tid & (DK - 1), qq = tid >> 7;          // gated: channel, token quarter
  const bf16* kp = reinterpret_cast<const bf16*>(p.k) + (row0 + kr) * DK + 8 * c8;
  const bf16* vp = reinterpret_cast<const bf16*>(p.v) + (row0 + vr) * 128 + vh * DVH + 8 * v8;
  const float* gp = MODE == SUM_GATED && p.g ? p.g + (row0 + 16 * qq) * DK + kc : nullptr;

  bf16x8 ks[2], vs;
  float gs[16];
  auto load = [&](int c) {
    const int64_t o = (int64_t)c * SEGK * DK;
    ks[0] = *reinterpret_cast<const bf16x8*>(kp + o);
    ks[1] = *reinterpret_cast<const bf16x8*>(kp + o + 32 * DK);
    vs = *reinterpret_cast<const bf16x8*>(vp + o);
    if constexpr (MODE == SUM_GATED) {
      if (gp) {
#pragma unroll
        for (int i = 0; i < 16; ++i) gs[i] = gp[o + i * DK];
      }
    }
  };
  if constexpr (MODE == SUM_GATED) {
#pragma unroll
    for (int i = 0; i < 16; ++i) gs[i] = 0.f;
  }
  load(0);
  f32x16 acc = zero16();
  float z8[8], s8[8], t8[8];          // sums of phi(k) (this thread's channels), of v and K1 v (its columns)
#pragma unroll
  for (int j = 0; j < 8; ++j) z8[j] = s8[j] = t8[j] = 0.f;
  float gtot = 0.f;

  for (int c = 0; c < nch; ++c) {
    const int b = MODE == SUM_GATED ? 0 : c & 1;
    bf16x8 vcur = vs;
    if constexpr (MODE == SUM_GATED) {
      float suf[16], run = 0.f;                          // sum of the later tokens' g within the quarter
#pragma unroll
      for (int i = 15; i >= 0; --i) {
        suf[i] = run;
        run += gs[i];
      }
      sm.qtot[qq][kc] = run;
      lds_barrier();                                     // also: the previous chunk's tiles are read
      float off = 0.f, tot = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float t = sm.qtot[q][kc];
        if (q > qq) off += t;
        tot += t;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) sm.W[16 * qq + i][kc] = __expf(suf[i] + off);
      if (qq == 0) {
        sm.eg[kc] = __expf(tot);
        gtot += tot;
      }
      lds_barrier();                                     // W
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const f32x4 w0 = *reinterpret_cast<const f32x4*>(&sm.W[kr + 32 * u][8 * c8]);
        const f32x4 w1 = *reinterpret_cast<const f32x4*>(&sm.W[kr + 32 * u][8 * c8 + 4]);
        bf16x8 ko;
#pragma unroll
        for (int j = 0; j < 8; ++j) ko[j] = (bf16)((float)ks[u][j] * (j < 4 ? w0[j] : w1[j - 4]));
        *reinterpret_cast<bf16x8*>(&sm.K[b][(kr + 32 * u) * SM::PK + 8 * c8]) = ko;
      }
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bf16x8 ko;
        float ksum = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = (float)ks[u][j];
          const float e = __expf(x);
          float f = MODE == SUM_CENTERED ? (x > 0.f ? x : e - 1.f) : (x > 0.f ? x + 1.f : e);
          f = 8 * c8 + j < kd ? f : 0.f;
          ko[j] = (bf16)f;
          z8[j] += (float)ko[j];
          ksum += f;
        }
        *reinterpret_cast<bf16x8*>(&sm.K[b][(kr + 32 * u) * SM::PK + 8 * c8]) = ko;
        if constexpr (MODE == SUM_CENTERED) {
          // the token's 16 chunks are one 16-lane row: prefix sums on the DPP crossbar, the total in its last lane
          ksum += dppf<0x111>(ksum);
          ksum += dppf<0x112>(ksum);
          ksum += dppf<0x114>(ksum);
          ksum += dppf<0x118>(ksum);
          if (c8 == 15) sm.k1[b][kr + 32 * u] = ksum;
        }
      }
    }
    *reinterpret_cast<bf16x8*>(&sm.V[b][vr * SM::PV + 8 * v8]) = vcur;
    if (c + 1 < nch) load(c + 1);
    lds_barrier();                                       // the chunk's tiles
    if constexpr (MODE == SUM_CENTERED) {
      const float k1 = sm.k1[b][vr];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = (float)vcur[j];
        s8[j] += v;
        t8[j] += k1 * v;
      }
    }
    if constexpr (MODE == SUM_GATED) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 e4 = *reinterpret_cast<const f32x4*>(&sm.eg[32 * kt + 8 * q + 4 * half]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[4 * q + j] *= e4[j];
      }
    }
#pragma unroll
    for (int s = 0; s < SEGK / 16; ++s)
      acc = mma(col_frag_tr(sm.K[b], SM::PK, 32 * kt, 16 * s), col_frag_tr(sm.V[b], SM::PV, 32 * vt, 16 * s), acc);
  }

  constexpr int REC = MODE == SUM_CENTERED ? KDA_BWD_REC : KDA_REC;
  float* rec = p.seg_sum + ((int64_t)seg * nbh + bh) * REC;
#pragma unroll
  for (int r = 0; r < 16; ++r) rec[(32 * kt + acc_row(half, r)) * 128 + vh * DVH + 32 * vt + l32] = acc[r];
  if constexpr (MODE == SUM_GATED) {
    if (vh == 0 && qq == 0) rec[128 * 128 + kc] = gtot;
  } else {
    // the vector sums: over a wave's token rows by shuffles, over the waves through LDS in wave order
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      z8[j] += __shfl_xor(z8[j], 16, 64);
      z8[j] = sum_halves(z8[j]);
      if constexpr (MODE == SUM_CENTERED) {
        s8[j] += __shfl_xor(s8[j], 8, 64);
        s8[j] += __shfl_xor(s8[j], 16, 64);
        s8[j] = sum_halves(s8[j]);
        t8[j] += __shfl_xor(t8[j], 8, 64);
        t8[j] += __shfl_xor(t8[j], 16, 64);
        t8[j] = sum_halves(t8[j]);
      }
      if (l < 16) sm.red[0][w][8 * c8 + j] = z8[j];
      if (MODE == SUM_CENTERED && l < 8) {
        sm.red[1][w][8 * v8 + j] = s8[j];
        sm.red[2][w][8 * v8 + j] = t8[j];
      }
    }
    lds_barrier();
    auto total = [&](int m, int i) {
      float a = 0.f;
#pragma unroll
      for (int q = 0; q < 8; ++q) a += sm.red[m][q][i];
      return a;
    };
    if (vh == 0 && tid < DK) rec[128 * 128 + tid] = total(0, tid);
    if (MODE == SUM_CENTERED && tid >= 128 && tid < 128 + 2 * DVH) {
      const int m = 1 + (tid - 128) / DVH, i = tid & (DVH - 1);
      rec[128 * 128 + 128 * m + vh * DVH + i] = total(m, i);
    }
  }
}

}  // namespace

void kda_split(int64_t units, int nch, int most, KdaSplitCost cost, int& nseg, int& seg_chunks) {
  // In chunk times of the walk (reference mode about 5 us, gated 2.6), fitted at 16 to 192 workgroups and 200 to 8192
  // tokens: a round of 256 workgroups takes its segments' chunks plus two (the first loads, the entering sums, the
  // drain); the sums, two workgroups per CU, `sums` of that, or `alone` with one; the second launch `launch`.  Reference mode: B1 H16 S1500
  // 8 segments 29 us, unsplit 114; B1 H16 S200 4 segments 13.5, unsplit 21.9; B2 H32 S4096 4 segments 212, unsplit
  // 324; B2 H48 S2048, unsplit by this rule: 157, 8 segments 184.  Gated: B1 H8 S8192 16 segments 56, unsplit 283;
  // B1 H16 S300 5 segments 15.1, unsplit 17.1; by this rule unsplit: B4 H24 S8192 333, 4 segments 476; B2 H32 S1000
  // 42.4, 4 segments 49.2.
  float best = 1e30f;
  nseg = 1;
  seg_chunks = nch;
  for (int s = 1; s <= most && s <= nch; ++s) {
    const int per = (nch + s - 1) / s;
    if ((nch + per - 1) / per != s) continue;            // the same segments as a smaller s
    float t = (float)((units * s + 255) / 256) * (per + 2);
    const int64_t n = units * (s - 1);
    if (s > 1) t += (n <= 256 ? cost.alone : cost.sums * (float)((n + 511) / 512)) * (per + 2) + cost.launch;
    if (t < best) {
      best = t;
      nseg = s;
      seg_chunks = per;
    }
  }
}

size_t kda_plan_segments(KdaParams& p) {
  const int nch = (p.seqlen + SEGK - 1) / SEGK;
  const int64_t nbh = (int64_t)p.batch * p.nheads;
  p.nseg = 1;
  p.seg_chunks = nch;
  if (nch == 0 || kda_precise_path(p)) return 0;
  kda_split(2 * nbh, nch, 16, p.mode == 0 ? KDA_COST_GATED : KDA_COST_REF, p.nseg, p.seg_chunks);
  return p.nseg > 1 ? (size_t)(p.nseg - 1) * nbh * KDA_REC * sizeof(float) : 0;
}

hipError_t launch_kda_centered_sums(const KdaParams& p, hipStream_t st) {
  hipLaunchKernelGGL(kda_sum_kernel<SUM_CENTERED>, dim3((unsigned)(2 * p.batch * p.nheads), (unsigned)(p.nseg - 1)),
                     dim3(512), 0, st, p);
  return hipGetLastError();
}

hipError_t launch_kda(const KdaParams& p_, hipStream_t st) {
  KdaParams p = p_;
  const int nbh = p.batch * p.nheads;
  if (p.seqlen == 0) {
    const size_t ns = p.final_state ? (size_t)nbh * p.dk * p.dv : 0, nz = p.final_z ? (size_t)nbh * p.dk : 0;
    const size_t n = ns > nz ? ns : nz;
    if (n) hipLaunchKernelGGL(kda_empty_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p.init_state,
                              p.final_state, ns, p.init_z, p.final_z, nz);
    return hipGetLastError();
  }
  if (kda_precise_path(p)) return launch_kda_precise(p, st);
  if (!p.seg_sum || p.nseg <= 1) {
    p.nseg = 1;
    p.seg_chunks = (p.seqlen + SEGK - 1) / SEGK;
  } else {
    const dim3 sgrid((unsigned)(2 * nbh), (unsigned)(p.nseg - 1));
    if (p.mode == 0) hipLaunchKernelGGL(kda_sum_kernel<SUM_GATED>, sgrid, dim3(512), 0, st, p);
    else hipLaunchKernelGGL(kda_sum_kernel<SUM_PHI>, sgrid, dim3(512), 0, st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const dim3 grid((unsigned)(2 * nbh), (unsigned)p.nseg);
  if (p.mode == 0) {
    if (p.nseg > 1) hipLaunchKernelGGL(kda_gated_kernel<true>, grid, dim3(64 * KW), 0, st, p);
    else hipLaunchKernelGGL(kda_gated_kernel<false>, grid, dim3(64 * KW), 0, st, p);
  } else if (p.q2) {
    hipLaunchKernelGGL(kda_ref_kernel<2>, grid, dim3(kda_ref_threads<2>), 0, st, p);
  } else {
    hipLaunchKernelGGL(kda_ref_kernel<1>, grid, dim3(kda_ref_threads<1>), 0, st, p);
  }
  return hipGetLastError();
}

}  // namespace mh
