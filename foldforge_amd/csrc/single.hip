// Single-track kernels: attention with pair bias and the wide (non-128) SwiGLU transition.
//
// Shapes: tokens m = b * n + i (M = batch * n rows), single width cs (a multiple of 64),
// heads x dh with dh a multiple of 8 and at most 32. The pair input z is [batch, n, n, 128].
//
// Attention with pair bias (legacy/transformer.py:93-137 of the reference):
//   x = LN_single(s); q = (x W_q^T + b_q), k = x W_k^T, v = x W_v^T, g = sigmoid(x W_g^T + gb)
//   bias[h, i, j] = LN_pair(z[i, j]) . W_b[h]   (the pair norm has no offset)
//   o = softmax_j(q_i . k_j / sqrt(dh) + bias[h, i, j]) over valid keys j, 0 for an empty row
//   out = s + (g * o) W_out^T
// is run as: row_gemm<kEpiApb, kXLn> (LayerNorm prologue; q, k, v^T, gate) and apb_pair_bias (few
// tokens: one launch, apb_project_bias) -> apb_attention (gate applied) -> row_gemm<kEpiResid>.
// The wide transition is row_gemm<kEpiSwiglu, kXLn> -> row_gemm<kEpiResid>.
// The same file holds row_stream, the streaming LayerNorm-fed token-row GEMM that the
// generic pair widths (template stacks, Chai-1's pair 256) run their projections on.
//
// Logits are carried in log2 units: q is scaled by log2(e) / sqrt(dh) and the pair-bias
// weights by log2(e), so the softmax uses exp2. Masked keys (and the padding keys past n)
// get the finite logit kMaskedLogit: their weight is exactly 0 once any valid key is seen.
#include <algorithm>
#include <type_traits>

#include "ffk_device.h"
#include "ffk_kernels.h"

namespace ffk {

namespace {

constexpr float kMaskedLogit = -1e30f;

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (bf16)0.f;
  return r;
}

// Position of key `key` inside the v^T rows: index bits 2 and 3 exchanged, so that the 8
// consecutive positions a lane loads are the 8 keys its P^T operand holds.
__device__ __forceinline__ int vkey_pos(int key) {
  return (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1);
}

// ---------------------------------------------------------------------------- row GEMM
// D[o][m] = sum_k W[o][k] X[m][k] over 32 rows of X per workgroup: A = W rows (fp32 parameters,
// converted in registers), B = X rows. The workgroup's 8 waves cover NO output tiles of 32
// with KS waves each (NO * KS = 8): the KS waves of a tile split k in groups of 64 (part p
// takes groups p, p + KS, ...), keep two groups of global loads in flight, and add their
// partial tiles through LDS; part 0 runs the epilogue. For MFMA step t of a group, lane half g
// supplies k = 32 g + 8 t .. + 7 of both operands (the order of the sums, and with it every output
// bit, is part of the kernel). Weight rows and fp32 x rows are loaded 64 bytes of each half of 8 rows at
// a time, two steps' worth, and turned into operands in a wave-private LDS tile: loaded in operand
// order (a row per lane), an instruction touches 64 cache lines. q / k / v / gate of 201 tokens x
// 384: 15.4 -> 13.3 us; squeeze (k 1536) and expand of 97 tokens 14.8 -> 10.0 and 17.2 -> 13.9;
// transition of 2000 rows x 384 87 -> 73. Three groups in flight (96 VGPRs) ran one workgroup per
// CU and 2-5% slower than two. Bound by its dependent chain at these sizes: launch, LayerNorm,
// one L2 latency per pair of groups, reduction, epilogue.
// Precision: activations enter as fp32 and are split into bf16 hi + lo (two MFMAs); the weights
// are rounded to bf16, or with w_split also split into hi + lo (a third MFMA, lo x hi: the
// products then carry about fp32 accuracy, the lo x lo term below it dropped). The single-track
// ops set w_split: their GEMMs are small and latency-bound, and a bf16 rounding of a weight is
// the same perturbation at every application of the block, so it moves the trunk's trajectory
// rather than averaging out.
// X sources: kXLn = LayerNorm of bf16 rows (ln_x [M][K], statistics and affine in fp32, the
// normalised tile staged in LDS once per workgroup as hi / lo rows); kXF32 = fp32 rows
// streamed from x32 [M][K].
// Epilogue: lane (li, g) holds token m0 + li and outputs o = 32 ot + 8 v + 4 g + e
// (acc[4 v + e]).

constexpr int kGemmWaves = 8;
constexpr int kTurnTile = 2 * 32 * 32;  // a wave's LDS tile: 32 rows x (2 halves x 16 k), hi then lo
__device__ __forceinline__ int turn_off(int r, int p) { return r * 32 + 8 * (p ^ ((r >> 2) & 3)); }

size_t row_gemm_lds(int xsrc, int K) {
  const size_t tiles = (size_t)kGemmWaves * (xsrc == kXLn ? 1 : 2) * kTurnTile * sizeof(bf16);
  return tiles + (xsrc == kXLn ? (size_t)2 * 32 * (K + 8) * sizeof(bf16) : 0);
}

// The input row of logical row m under the row map a.tmap (see kMap* in ffk_kernels.h).
// The last workgroup's rows past M (the grid covers M rounded up to 32) read row M - 1: they
// are never stored, and an unclamped transposed map would read past the end of the input.
__device__ inline int64_t mapped_row(const RowGemmArgs& a, int64_t m) {
  m = min(m, a.M - 1);
  if (a.tmap == kMapPairT) {
    const int64_t nn = (int64_t)a.n * a.n;
    const int64_t b = m / nn, rem = m - b * nn;
    const int r = (int)(rem / a.n), j = (int)(rem - (int64_t)r * a.n);
    return (b * a.n + j) * a.n + r;
  }
  if (a.tmap == kMapPadKeys || a.tmap == kMapPadKeysT) {
    const int64_t bn = m / a.np;
    const int j = min((int)(m - bn * a.np), a.n - 1);
    if (a.tmap == kMapPadKeys) return bn * a.n + j;
    const int64_t b = bn / a.n;
    return (b * a.n + j) * a.n + (bn - b * a.n);
  }
  if (a.tmap == kMapGridOut || a.tmap == kMapGridIn) {
    const int64_t bi = m / a.gk, b = bi / a.n;
    const int i = (int)(bi - b * a.n), k = min((int)(m - bi * a.gk), a.n - 1);
    return a.tmap == kMapGridOut ? (b * a.n + i) * a.n + k : (b * a.n + k) * a.n + i;
  }
  return m;
}

// kEpiOpm: the MSA row read by logical row m = (b n + j) sp + s (rows past the depth repeat
// the last one; their projection is zeroed).
__device__ inline int64_t opm_msa_row(const RowGemmArgs& a, int64_t m) {
  m = min(m, a.M - 1);
  const int64_t bj = m / a.sp;
  const int s = min((int)(m - bj * a.sp), a.depth - 1);
  const int64_t b = bj / a.n;
  const int j = (int)(bj - b * a.n);
  return (b * a.depth + s) * a.n + j;
}

// kEpiApb's width of one projection (q, k, v and, with apb_no_gate == 0, the gate).
__device__ __forceinline__ int apb_width(const RowGemmArgs& a) { return a.O / (a.apb_no_gate ? 3 : 4); }

// The weight row (fp32, K values) multiplied by row li of output tile ot, and the tile's
// segment and first channel as the epilogue reads them (packed tiles: see kEpiTrimul and
// kEpiSwiglu below).
// (row_stream's kEpiApb with flash_rows > 0: an epilogue of its own.)
constexpr int kEpiApbFlash = 100;
template <int EPI>
__device__ inline const float* tile_weight_row(const RowGemmArgs& a, int ot, int li, int& seg, int& cbase) {
  const float* wr;
  seg = 0;
  cbase = 0;
  if (EPI == kEpiApb || EPI == kEpiApbFlash) {
    const int cs = apb_width(a);
    seg = (ot * 32) / cs;
    cbase = ot * 32 - seg * cs;
    const float* base = seg == 0 ? a.w0 : seg == 1 ? a.w1 : seg == 2 ? a.w2 : a.w3;
    wr = base + (int64_t)(cbase + li) * a.K;
  } else if (EPI == kEpiPwa || EPI == kEpiOpm) {
    const int hd = a.O / 2;
    seg = (ot * 32) / hd;
    cbase = ot * 32 - seg * hd;
    wr = (seg == 0 ? a.w0 : a.w1) + (int64_t)(cbase + li) * a.K;
  } else if (EPI == kEpiTrimul) {
    // packed tile: rows 0-15 are projection rows cbase .. cbase + 15 of one side, rows 16-31 the
    // matching gate rows
    const int tps = a.O / 64;  // tiles per side: hid / 16
    seg = ot / tps;
    cbase = (ot - seg * tps) * 16;
    const float* base = li < 16 ? (seg == 0 ? a.w0 : a.w1) : (seg == 0 ? a.w2 : a.w3);
    wr = base + (int64_t)(cbase + (li & 15)) * a.K;
  } else if (EPI == kEpiSwiglu) {
    // packed tile: rows 0-15 are expand_a rows 16 ot .., rows 16-31 the expand_b rows alike
    wr = (li < 16 ? a.w0 : a.w1) + (int64_t)(ot * 16 + (li & 15)) * a.K;
  } else {
    wr = a.w0 + (int64_t)(ot * 32 + li) * a.K;
  }
  return wr;
}

// The per-row value an epilogue reads from memory, once per row rather than per output tile:
// kEpiTrimul's pair mask factor m_i m_k (symmetric, so the same for the transposed read).
template <int EPI>
__device__ __forceinline__ float row_pre(const RowGemmArgs& a, const int64_t m) {
  if (EPI == kEpiTrimul) {
    const int64_t bi = m / a.gk, b = bi / a.n;
    const int i = (int)(bi - b * a.n), k = (int)(m - bi * a.gk);
    return k < a.n && a.mask[b * a.n + i] && a.mask[b * a.n + k] ? 1.f : 0.f;
  }
  return 0.f;
}

// Epilogue of output tile ot for logical row m (< M): lane half g holds outputs
// 32 ot + 8 v + 4 g + e in acc[4 v + e]. lb: the per-output biases (q_bias / gate_b of kEpiApb,
// bias_out of kEpiResid) staged in LDS by output index, or NULL to read them from the arguments.
// The loads an epilogue needs are all issued before its first store. ypre: the yin values of
// kEpiGateResid, loaded by the caller (NULL: loaded here). rpre: the residual values of kEpiResid
// and kEpiGateResid, loaded by the caller (NULL: loaded here); both as the two 16-byte pieces
// (acc_pieces) of the lane.
template <int EPI>
__device__ __forceinline__ void row_epilogue(const RowGemmArgs& a, const f32x16& acc, const int64_t m, const int ot,
                                    const int seg, const int cbase, const int g, const float* lb,
                                    const float pre, const bf16x8* rpre = nullptr,
                                    const bf16x8* ypre = nullptr) {
  // the bias of output o (global index gi of src when not staged)
  auto obias = [&](int o, const float* src, int gi) { return lb ? lb[o] : (src ? src[gi] : 0.f); };
  if (EPI == kEpiApb) {
    const int cs = apb_width(a);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = cbase + 8 * v + 4 * g;
      const int o0 = 32 * ot + 8 * v + 4 * g;
      float y0 = acc[4 * v], y1 = acc[4 * v + 1], y2 = acc[4 * v + 2], y3 = acc[4 * v + 3];
      if (seg == 0) {
        y0 += obias(o0, a.q_bias, c);
        y1 += obias(o0 + 1, a.q_bias, c + 1);
        y2 += obias(o0 + 2, a.q_bias, c + 2);
        y3 += obias(o0 + 3, a.q_bias, c + 3);
        y0 *= a.q_scale;
        y1 *= a.q_scale;
        y2 *= a.q_scale;
        y3 *= a.q_scale;
        store4(a.q + m * cs + c, y0, y1, y2, y3);
      } else if (seg == 1) {
        store4(a.k + m * cs + c, y0, y1, y2, y3);
      } else if (seg == 2) {
        const int64_t b = m / a.n;
        const int key = (int)(m - b * a.n);
        const int pos = vkey_pos(key);
        const float ys[4] = {y0, y1, y2, y3};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int hh = (c + e) / a.dh, d = (c + e) - hh * a.dh;
          a.vt[((b * a.heads + hh) * a.dh + d) * a.np + pos] = (bf16)ys[e];
        }
      } else {
        const float nb = -kLog2e;
        y0 += obias(o0, a.gate_b, c);
        y1 += obias(o0 + 1, a.gate_b, c + 1);
        y2 += obias(o0 + 2, a.gate_b, c + 2);
        y3 += obias(o0 + 3, a.gate_b, c + 3);
        y0 = sigmoid_scaled((y0 + a.gate_bias) * nb);
        y1 = sigmoid_scaled((y1 + a.gate_bias) * nb);
        y2 = sigmoid_scaled((y2 + a.gate_bias) * nb);
        y3 = sigmoid_scaled((y3 + a.gate_bias) * nb);
        store4(a.gate + m * cs + c, y0, y1, y2, y3);
      }
    }
  } else if (EPI == kEpiPwa) {
    const int hd = a.O / 2;
    const int64_t bs = m / a.n;  // b S + s
    const int j = (int)(m - bs * a.n);
    const int64_t b = bs / a.depth, srow = bs - b * a.depth;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = cbase + 8 * v + 4 * g;  // 4 channels of one head (dh % 4 == 0)
      float y[4] = {acc[4 * v], acc[4 * v + 1], acc[4 * v + 2], acc[4 * v + 3]};
      if (seg == 0) {
        const int hh = c / a.dh, d0 = c - hh * a.dh;
        bf16* dst = a.vt + (((b * a.heads + hh) * a.depth + srow) * a.dh + d0) * a.np + j;
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(int64_t)e * a.np] = (bf16)y[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = sigmoid_scaled(-kLog2e * y[e]);
        store4(a.gate + m * hd + c, y[0], y[1], y[2], y[3]);
      }
    }
  } else if (EPI == kEpiOpm) {
    const int64_t bj = m / a.sp;
    const int s = (int)(m - bj * a.sp);
    const int64_t b = bj / a.n;
    const int j = (int)(bj - b * a.n);
    const float keep = s < a.depth && a.rows_mask[(b * a.depth + s) * a.n + j] ? 1.f : 0.f;
    const float* bias = seg == 0 ? a.bias0 : a.bias1;
    const int hd = a.O / 2;  // channels a side (32; Chai-1's grouped form 64)
    bf16* dst = (seg == 0 ? a.lt : a.rt) + bj * hd * a.sp + s;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = cbase + 8 * v + 4 * g + e;
        dst[(int64_t)c * a.sp] = (bf16)((acc[4 * v + e] + (bias ? bias[c] : 0.f)) * keep);
      }
    if (seg == 0 && cbase == 0 && g == 0) a.mt[bj * a.sp + s] = (bf16)keep;
  } else if (EPI == kEpiTrimul) {
    const int hid = a.O / 4;
    const int64_t gg = (int64_t)a.npm * a.npm;
    const int64_t bi = m / a.gk, b = bi / a.n;
    const int64_t rem = (bi - b * a.n) * a.npm + (m - bi * a.gk);
    const float keep = pre;  // the pair mask factor (row_pre)
    bf16* plane = (seg == 0 ? a.pa : a.pb) + b * hid * gg + rem;
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = cbase + 8 * v + 4 * g + e;
        const float proj = acc[4 * v + e] * keep;  // masked before the gate, as the reference
        const bf16 y = (bf16)(proj * sigmoid_scaled(-kLog2e * acc[8 + 4 * v + e]));
        plane[(int64_t)c * gg] = y;
      }
  } else if (EPI == kEpiStoreY) {
    float y[2][8];
    acc_pieces(acc, y);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (bf16)y[k][e];
      *reinterpret_cast<bf16x8*>(a.hy + m * a.O + ot * 32 + 8 * (2 * k + g)) = o;
    }
  } else if (EPI == kEpiGateResid) {
    bf16x8 yv[2], rv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = ot * 32 + 8 * (2 * k + g);
      yv[k] = ypre ? ypre[k] : *reinterpret_cast<const bf16x8*>(a.yin + m * a.O + c);
      if (a.residual) rv[k] = rpre ? rpre[k] : *reinterpret_cast<const bf16x8*>(a.res + m * a.O + c);
    }
    float y[2][8];
    acc_pieces(acc, y);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float t = (float)yv[k][e] * sigmoid_scaled(-kLog2e * y[k][e]);
        if (a.residual) t += (float)rv[k][e];
        o[e] = (bf16)t;
      }
      *reinterpret_cast<bf16x8*>(a.out + m * a.O + ot * 32 + 8 * (2 * k + g)) = o;
    }
  } else if (EPI == kEpiLinear) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = ot * 32 + 8 * v + 4 * g;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = acc[4 * v + e] + (a.bias_out ? a.bias_out[c + e] : 0.f);
        if (a.act == kActSigmoid)
          t = sigmoid_scaled(-kLog2e * t);
        else if (a.act == kActSilu)
          t = t * sigmoid_scaled(-kLog2e * t);
        else if (a.act == kActRelu)
          t = fmaxf(t, 0.f);
        y[e] = t;
      }
      if (a.y_f32) {
        const f32x4 yv = {y[0], y[1], y[2], y[3]};
        *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + m * a.O + c) = yv;
      } else {
        store4(static_cast<bf16*>(a.y) + m * a.O + c, y[0], y[1], y[2], y[3]);
      }
    }
  } else if (EPI == kEpiSwiglu) {
    const int hid = a.O / 2;
    f32x4 y[2];
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float av = acc[4 * v + e], bv = acc[8 + 4 * v + e];
        y[v][e] = av * sigmoid_scaled(-kLog2e * av) * bv;
      }
    if (a.h16) {
      // hidden 8 v + 4 g + 0..3 in y[v]: one exchange gives half g the 8 channels 8 g .. 8 g + 7
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[0][e]), __float_as_uint(y[1][e]),
                                                         false, false);
        o[e] = (bf16)__uint_as_float(sw[0]);
        o[4 + e] = (bf16)__uint_as_float(sw[1]);
      }
      *reinterpret_cast<bf16x8*>(a.h16 + m * hid + ot * 16 + 8 * g) = o;
    } else {
#pragma unroll
      for (int v = 0; v < 2; ++v)
        *reinterpret_cast<f32x4*>(a.h32 + m * hid + ot * 16 + 8 * v + 4 * g) = y[v];
    }
  } else {
    bf16x8 rv[2];
    if (a.residual) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
        rv[k] = rpre ? rpre[k] : *reinterpret_cast<const bf16x8*>(a.res + m * a.O + ot * 32 + 8 * (2 * k + g));
    }
    float y[2][8];
    acc_pieces(acc, y);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = ot * 32 + 8 * (2 * k + g);
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float t = y[k][e] + obias(c + e, a.bias_out, c + e);
        if (a.residual) t += (float)rv[k][e];
        o[e] = (bf16)t;
      }
      *reinterpret_cast<bf16x8*>(a.out + m * a.O + c) = o;
    }
  }
}

template <int EPI, int XSRC, int NO, int kAhead>
__device__ __forceinline__ void row_gemm_body(const RowGemmArgs& a, const int bx, const int by) {
  constexpr int KS = kGemmWaves / NO;
  constexpr int kTurns = XSRC == kXLn ? 1 : 2;  // tiles per wave: weights, fp32 x rows
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // [kGemmWaves][kTurns][kTurnTile]; behind the products a wave's first tile takes its partial sums
  bf16* turns = reinterpret_cast<bf16*>(smem);
  static_assert(64 * 16 * sizeof(float) <= kTurnTile * sizeof(bf16), "partial sums exceed the turn tile");
  bf16* xs_hi = turns + kGemmWaves * kTurns * kTurnTile;
  const int xstride = a.K + 8;  // [32][K + 8]: rows 16 bytes apart modulo 256, conflict-free
  bf16* xs_lo = xs_hi + 32 * xstride;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int osub = wave / KS, part = wave % KS;
  const int ot = by * NO + osub;
  const bool active = ot * 32 < a.O;
  const int64_t m0 = (int64_t)bx * 32;
  const int G = a.K / 64, ng = active && part < G ? (G - part + KS - 1) / KS : 0;

  // this lane's loads: column kc = 4 (lane % 8) of the tile, i.e. k 32 (kc / 16) + 16 h + kc % 16 of the
  // group in its half h, of rows 8 u + lane / 8, u = 0 .. 3 (packed tiles take rows 16-31 from a
  // second matrix: a pointer per 16 rows)
  int seg, cbase;
  const int kc = 4 * (lane & 7), kq = 32 * (kc >> 4) + (kc & 15), row8 = lane >> 3;
  const float* wr[2];
  const float* xr4[4];
#pragma unroll
  for (int u = 0; u < 2; ++u) wr[u] = tile_weight_row<EPI>(a, ot, 16 * u + row8, seg, cbase) + kq;
  if (XSRC == kXF32) {
#pragma unroll
    for (int u = 0; u < 4; ++u) xr4[u] = a.x32 + mapped_row(a, m0 + 8 * u + row8) * a.K + kq;
  }
  bf16* wt = turns + wave * kTurns * kTurnTile;
  bf16* xt = wt + kTurnTile;

  f32x16 acc = zero16();
  f32x4 wv[kAhead][8], xv4[kAhead][XSRC == kXF32 ? 8 : 1];
  auto fetch = [&](int i, f32x4* w, f32x4* x) __attribute__((always_inline)) {
    const int k = 64 * (part + KS * i);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int h = q >> 2, u = q & 3;
      w[q] = *reinterpret_cast<const f32x4*>(wr[u >> 1] + (int64_t)(8 * (u & 1)) * a.K + k + 16 * h);
      if (XSRC == kXF32) x[q] = *reinterpret_cast<const f32x4*>(xr4[u] + k + 16 * h);
    }
  };
  // rows 8 u + lane / 8 of steps 2 h and 2 h + 1 into a tile, hi and (lo_on) lo
  auto turn = [&](const f32x4* v, bf16* tile, bool lo_on) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi[e] = (bf16)v[u][e];
        lo[e] = (bf16)(v[u][e] - (float)hi[e]);
      }
      const int at = turn_off(8 * u + row8, kc >> 3) + (kc & 4);
      *reinterpret_cast<bf16x4*>(tile + at) = hi;
      if (lo_on) *reinterpret_cast<bf16x4*>(tile + 32 * 32 + at) = lo;
    }
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
    if (s < ng) fetch(s, wv[s], xv4[s]);

  if (XSRC == kXLn) {
    // thread t normalises row t / 16, chunks (t % 16) + 16 i of 8 channels, held in registers;
    // the 16 threads of a row are consecutive lanes, joined by DPP sums
    constexpr int kMaxChunks = kLnGemmMaxK / 128;
    const int r = tid >> 4, pc = tid & 15;
    const int nc = a.K / 8;
    const bf16* xr = a.ln_x + (EPI == kEpiOpm ? opm_msa_row(a, m0 + r) : mapped_row(a, m0 + r)) * a.K;
    bf16x8 xv[kMaxChunks];
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i)
      if (pc + 16 * i < nc) xv[i] = ld8(xr + 8 * (pc + 16 * i));
    float s1 = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i)
      if (pc + 16 * i < nc)
#pragma unroll
        for (int e = 0; e < 8; ++e) s1 += (float)xv[i][e];
    const float mean = a.ln_plain ? 0.f : sum16(s1) / (float)a.K;
    float s2 = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i)
      if (pc + 16 * i < nc)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = (float)xv[i][e] - mean;
          s2 += d * d;
        }
    const float eps = a.eps_dev ? *a.eps_dev : a.eps;
    const float rstd = a.ln_plain ? 1.f : __builtin_amdgcn_rsqf(sum16(s2) / (float)a.K + eps);
    const f32x4 one4 = {1.f, 1.f, 1.f, 1.f}, zero4 = {0.f, 0.f, 0.f, 0.f};
    const bool has_w = a.ln_w != nullptr && !a.ln_plain, has_b = a.ln_b != nullptr && !a.ln_plain;
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i) {
      if (pc + 16 * i < nc) {
        const int c = 8 * (pc + 16 * i);
        const f32x4 w0 = has_w ? *reinterpret_cast<const f32x4*>(a.ln_w + c) : one4;
        const f32x4 w1 = has_w ? *reinterpret_cast<const f32x4*>(a.ln_w + c + 4) : one4;
        const f32x4 b0 = has_b ? *reinterpret_cast<const f32x4*>(a.ln_b + c) : zero4;
        const f32x4 b1 = has_b ? *reinterpret_cast<const f32x4*>(a.ln_b + c + 4) : zero4;
        f32x4 y0, y1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y0[e] = ((float)xv[i][e] - mean) * rstd * w0[e] + b0[e];
          y1[e] = ((float)xv[i][4 + e] - mean) * rstd * w1[e] + b1[e];
        }
        bf16x8 hi, lo;
        split8(y0, y1, hi, lo);
        *reinterpret_cast<bf16x8*>(xs_hi + r * xstride + c) = hi;
        *reinterpret_cast<bf16x8*>(xs_lo + r * xstride + c) = lo;
      }
    }
    __syncthreads();
  }

  // (LDS operations of a wave complete in order: a tile is rewritten behind its reads)
  auto consume = [&](int i, const f32x4* w, const f32x4* x) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      turn(w + 4 * h, wt, a.w_split != 0);
      if (XSRC == kXF32) turn(x + 4 * h, xt, true);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int at = turn_off(li, 2 * g + t);
        bf16x8 xhi, xlo;
        if (XSRC == kXLn) {
          const int k = 64 * (part + KS * i) + 32 * g + 16 * h + 8 * t;
          xhi = ld8(xs_hi + li * xstride + k);
          xlo = ld8(xs_lo + li * xstride + k);
        } else {
          xhi = ld8(xt + at);
          xlo = ld8(xt + 32 * 32 + at);
        }
        const bf16x8 whi = ld8(wt + at);
        acc = mfma32(whi, xlo, acc);
        acc = mfma32(whi, xhi, acc);
        if (a.w_split) acc = mfma32(ld8(wt + 32 * 32 + at), xhi, acc);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
#pragma unroll 1
  for (int i = 0; i < ng; i += kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (i + s < ng) {
        consume(i + s, wv[s], xv4[s]);
        if (i + s + kAhead < ng) fetch(i + s + kAhead, wv[s], xv4[s]);
      }
  }
  if (KS > 1) {
    if (part > 0) {
      float* mine = reinterpret_cast<float*>(wt) + lane * 16;
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[r] = acc[r];
    }
    __syncthreads();
    if (part != 0) return;
#pragma unroll
    for (int w = 1; w < KS; ++w) {
      const float* theirs = reinterpret_cast<const float*>(turns + (wave + w) * kTurns * kTurnTile) + lane * 16;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += theirs[r];
    }
  }

  const int64_t m = m0 + li;
  if (!active || m >= a.M) return;
  row_epilogue<EPI>(a, acc, m, ot, seg, cbase, g, nullptr, row_pre<EPI>(a, m));
}

// kAhead: groups in flight, 2, or 1 where no wave has a second one (up to KS groups): 128 VGPRs then, and
// two workgroups per CU (147 to 158 with two). Many rows need that: LayerNorm + linear of 100000 x 64 -> 128
// 50.3 -> 33.9 us, 256 -> 64 70.6 -> 45.3; the grouped outer product of 192 channels, 512 x 200 tokens, 286 -> 221.
template <int EPI, int XSRC, int NO, int kAhead>
__global__ __launch_bounds__(64 * kGemmWaves, kAhead == 1 ? 4 : 2) void row_gemm(RowGemmArgs a) {
  row_gemm_body<EPI, XSRC, NO, kAhead>(a, blockIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------- streaming row GEMM
// The products and epilogues of row_gemm for rows of K = 64 to 512 channels, as a persistent
// kernel: each workgroup converts the weights to bf16 once (LDS, in output-tile order, rows
// K + 8 elements apart so that the operand reads of 16 rows hit distinct banks), then every
// wave walks whole 32-row tiles on its own, with no barrier in the loop. With gridDim.y > 1 the
// output tiles are split into that many equal parts, one per grid row (wide outputs: each
// workgroup then holds a part of the weights and more workgroups fit on a CU). The next tile's input
// rows are loaded while the current one is normalised, multiplied for all O / 32 output tiles
// and stored by the epilogue of each output tile. Rows of up to 128 channels enter the MFMAs as
// bf16 hi + lo (as row_gemm); LayerNorm-fed rows of 256 as the rounded bf16 normalisation (as
// the reference's bf16 LayerNorm output), and 512-channel (plain bf16) rows are held in one
// register buffer, loaded after the last product of the previous tile.
// What the generic path writes key- or row-contiguous (v^T, the contraction's channel planes, the
// outer product's sides) is multiplied turned, D[row][output], so a lane holds one channel's
// consecutive rows and stores 16-byte pieces without a transpose. Bound by the vector ALU
// (LayerNorm, hi / lo split, epilogue) and the stores together; index arithmetic is kept in
// scalar registers (TileRun), which was most of the vector work: pair 256 x 384 tokens, q / k /
// v / gate 183 -> 158 us and trimul planes 147 -> 126; pair 64 x 4 templates 105 -> 88 and
// 84 -> 75 us; MSA 512 x 256 value / gate 22 -> 19 us.
// Lane (li, g) holds row li's channels (K / 2) g .. (K / 2) g + K / 2 - 1; MFMA step s takes
// channels (K / 2) g + 8 s .. + 7 of both operands.
// Waves per workgroup: 4, and 8 (two per SIMD, sharing a weight image of up to 154 KiB, one
// workgroup per CU) for rows of 256 channels or more.
__host__ __device__ constexpr int stream_waves(int K) { return K >= 256 ? 8 : 4; }

// LDS of one workgroup holding the weight rows of Op of the O outputs.
size_t row_stream_lds(int K, int O, int Op) {
  return (size_t)Op * (K + 8) * sizeof(bf16) + (size_t)(2 * K + O) * sizeof(float);
}

// Output tiles that must stay in one part: kEpiTrimul's projection and gate tiles.
__host__ __device__ constexpr int stream_unit(int epi) { return epi == kEpiTrimul ? 2 : 1; }

// Where a 32-row tile starts: logical row (b R + r) L + rem. A wave's walk advances the digits by
// the grid stride with adds and carries (an integer division by a runtime value is 20 to 100
// vector instructions, and a tile has few enough products for that to be most of its time).
struct TileRun {
  uint32_t rem, r, b;
};
template <int EPI>
__device__ __forceinline__ void run_radix(const RowGemmArgs& a, uint32_t& L, uint32_t& R) {
  L = EPI == kEpiTrimul ? a.gk
      : EPI == kEpiOpm  ? a.sp
      : EPI == kEpiPwa || EPI == kEpiApbFlash ? a.np
                                              : a.n;
  R = EPI == kEpiPwa ? a.depth : a.n;
  L = L ? L : 1;  // (the epilogues without a row map leave n unset)
  R = R ? R : 1;
}
__device__ __forceinline__ TileRun run_at(int64_t m, uint32_t L, uint32_t R) {
  TileRun t;
  if ((m >> 32) == 0) {
    const uint32_t x = (uint32_t)m, q = x / L;
    t.rem = x - q * L;
    t.b = q / R;
    t.r = q - t.b * R;
  } else {
    const int64_t q = m / L;
    t.rem = (uint32_t)(m - q * L);
    t.b = (uint32_t)(q / R);
    t.r = (uint32_t)(q - (int64_t)t.b * R);
  }
  return t;
}
__device__ __forceinline__ TileRun run_add(TileRun t, const TileRun& step, uint32_t L, uint32_t R) {
  t.rem += step.rem;
  uint32_t carry = t.rem >= L ? 1u : 0u;
  t.rem -= carry ? L : 0u;
  t.r += step.r + carry;
  carry = t.r >= R ? 1u : 0u;
  t.r -= carry ? R : 0u;
  t.b += step.b + carry;
  return t;
}

// The input row of the tile's row li (rows past M, n or the depth read the last one).
template <int EPI>
__device__ __forceinline__ int64_t run_row(const RowGemmArgs& a, const TileRun& t, int64_t m0, int li) {
  const int n = a.n;
  if (EPI == kEpiOpm) {
    const int s = min((int)t.rem + li, a.depth - 1);
    return (int64_t)t.b * a.depth * n + t.r + (int64_t)s * n;
  }
  if (EPI == kEpiTrimul) {
    const int i = (int)t.r, k = min((int)t.rem + li, n - 1);
    return a.tmap == kMapGridOut ? ((int64_t)t.b * n + i) * n + k
                                 : (int64_t)t.b * n * n + i + (int64_t)k * n;
  }
  if (EPI == kEpiPwa || EPI == kEpiApbFlash) {
    const int j = min((int)t.rem + li, n - 1);
    if (EPI == kEpiPwa || a.tmap == kMapPadKeys)
      return ((int64_t)t.b * (EPI == kEpiPwa ? a.depth : n) + t.r) * n + j;
    return (int64_t)t.b * n * n + t.r + (int64_t)j * n;
  }
  const int64_t left = a.M - 1 - m0;
  const int l = left < li ? (int)left : li;
  if ((EPI == kEpiApb || EPI == kEpiResid) && a.tmap == kMapPairT) {
    uint32_t j = t.rem + l, r = t.r, b = t.b;
    if (n >= 32) {  // at most one row of the pair ends inside the tile
      const bool c = j >= (uint32_t)n;
      j -= c ? (uint32_t)n : 0u;
      r += c ? 1u : 0u;
      const bool c2 = r >= (uint32_t)n;
      r = c2 ? 0u : r;
      b += c2 ? 1u : 0u;
    } else {
      r += j / n;
      j %= n;
      b += r / n;
      r %= n;
    }
    return ((int64_t)b * n + j) * n + r;
  }
  return m0 + l;
}

// Waves per SIMD the registers are held to at K = 64: 128 registers for four workgroups per CU
// where little or nothing spills (unbounded, q / k / v of the template stacks took 137 + 16 and
// three workgroups: 88 -> 75 us), else 168 for three.
__host__ __device__ constexpr int stream_simd_waves(int epi, int K) {
  return K != 64 ? 2 : epi == kEpiTrimul || epi == kEpiOpm || epi == kEpiResid ? 3 : 4;
}

template <int EPI, int XSRC, int K>
__global__ __launch_bounds__(64 * stream_waves(K), stream_simd_waves(EPI, K)) void row_stream(RowGemmArgs a) {
  constexpr int kStreamWaves = stream_waves(K);
  constexpr int KS = K / 16;  // MFMA steps
  constexpr int KH = K / 2;   // channels per lane
  constexpr int WS = K + 8;   // LDS row stride of the weight image (elements)
  constexpr bool BF = XSRC != kXF32;                // bf16 input rows
  constexpr int NX = BF ? KS : 2 * KS;              // 16-byte input pieces per lane
  constexpr bool LO = XSRC != kXBf16 && K <= 128;   // activations as bf16 hi + lo
  // the gate / residual epilogue of wide rows loads every output tile's operands (up to 128
  // VGPRs) at the start of a row tile instead of a second input buffer
  constexpr bool GR = EPI == kEpiGateResid && K >= 256;
  constexpr bool DB = NX <= 16 && !GR;              // two input buffers (64 VGPRs each at most)
  constexpr bool kRuns = EPI == kEpiApb || EPI == kEpiApbFlash || EPI == kEpiTrimul || EPI == kEpiOpm || EPI == kEpiPwa ||
                         EPI == kEpiResid;
  using XT = typename std::conditional<BF, bf16x8, f32x4>::type;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int64_t tiles = (a.M + 31) / 32;
  if ((int64_t)blockIdx.x * kStreamWaves >= tiles) return;
  const int nt = a.O / 32 / (int)gridDim.y;  // output tiles of this workgroup's part
  const int ot0 = (int)blockIdx.y * nt;
  bf16* wl = reinterpret_cast<bf16*>(smem);  // [nt][32][WS]: output tiles ot0 ..
  float* lnp = reinterpret_cast<float*>(smem + (size_t)nt * 32 * WS * sizeof(bf16));  // weight, offset
  float* lb = lnp + 2 * K;  // per-output biases (row_epilogue)
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // kEpiTrimul: tiles 2 p and 2 p + 1 are 32 projection rows of one side and their gate rows
  auto trimul_pair = [&](int p, int& side, int& c0) {
    const int pps = a.O / 128;
    side = p >= pps ? 1 : 0;
    c0 = (p - side * pps) * 32;
  };
  for (int idx = tid; idx < nt * 32 * (K / 8); idx += 64 * kStreamWaves) {
    const int row = idx / (K / 8), ch = 8 * (idx % (K / 8));
    const int ot = ot0 + (row >> 5);
    const float* wr;
    if (EPI == kEpiTrimul) {
      int side, c0;
      trimul_pair(ot >> 1, side, c0);
      wr = ((ot & 1) ? (side ? a.w3 : a.w2) : (side ? a.w1 : a.w0)) + (int64_t)(c0 + (row & 31)) * K;
    } else {
      int seg, cbase;
      wr = tile_weight_row<EPI>(a, ot, row & 31, seg, cbase);
    }
    *reinterpret_cast<bf16x8*>(wl + row * WS + ch) = cvt8(wr + ch);
  }
  for (int o = tid; o < a.O; o += 64 * kStreamWaves) {
    float v = 0.f;
    if (EPI == kEpiApb || EPI == kEpiApbFlash) {
      const int cs = apb_width(a), seg = o / cs, c = o - seg * cs;
      if (seg == 0 && a.q_bias) v = a.q_bias[c];
      if (seg == 3 && a.gate_b) v = a.gate_b[c];
    } else if (EPI == kEpiResid && a.bias_out) {
      v = a.bias_out[o];
    } else if (EPI == kEpiOpm) {
      const int hd = a.O / 2;
      const float* bias = o < hd ? a.bias0 : a.bias1;
      if (bias) v = bias[o < hd ? o : o - hd];
    }
    lb[o] = v;
  }
  if (XSRC == kXLn) {
    const bool plain = a.ln_plain != 0;
    for (int c = tid; c < K; c += 64 * kStreamWaves) {
      lnp[c] = a.ln_w && !plain ? a.ln_w[c] : 1.f;
      lnp[K + c] = a.ln_b && !plain ? a.ln_b[c] : 0.f;
    }
  }
  __syncthreads();

  const int64_t stride = (int64_t)gridDim.x * kStreamWaves;
  int64_t t = (int64_t)blockIdx.x * kStreamWaves + wave;
  if (t >= tiles) return;
  const float eps = XSRC == kXLn && a.eps_dev ? *a.eps_dev : a.eps;
  uint32_t L = 1, R = 1;
  TileRun cur{}, step{};
  if constexpr (kRuns) {
    // (rows read as they are have no digits: the two divisions took 0.2 to 0.8 us of a small call)
    if ((EPI != kEpiApb && EPI != kEpiResid) || a.tmap == kMapPairT) {
      run_radix<EPI>(a, L, R);
      cur = run_at(t * 32, L, R);
      step = run_at(stride * 32, L, R);
    }
  }
  const int apb_cs = EPI == kEpiApbFlash ? apb_width(a) : 1;
  const int dsh = EPI == kEpiApbFlash ? __builtin_ctz(a.dh) : 0;  // head widths 16, 32 or 64

  // the input rows of a tile, and the mask bytes of its rows (kEpiTrimul: of positions k and i;
  // kEpiOpm: of the MSA entry), which the epilogue needs a tile later
  auto fetch = [&](XT* x, uint32_t& keep, const TileRun& tr, int64_t m0) __attribute__((always_inline)) {
    const int64_t row = run_row<EPI>(a, tr, m0, li);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      if (BF)
        x[i] = *reinterpret_cast<const XT*>(a.ln_x + row * K + KH * g + 8 * i);
      else
        x[i] = *reinterpret_cast<const XT*>(a.x32 + row * K + KH * g + 4 * i);
    }
    keep = 0;
    if (EPI == kEpiTrimul) {
      const uint8_t* mb = a.mask + (int64_t)tr.b * a.n;
      const int i = (int)tr.r, k = min((int)tr.rem + li, a.n - 1);
      keep = (uint32_t)mb[k] | ((uint32_t)mb[i] << 8);
    } else if (EPI == kEpiOpm) {
      keep = a.rows_mask[row];
    }
  };
  auto process = [&](XT* x, uint32_t keep, const TileRun& tr, int64_t tile) __attribute__((always_inline)) {
    const int64_t m = tile * 32 + li;
    // rows kept by the mask, bit = row of the tile
    uint32_t bits = ~0u;
    if constexpr (EPI == kEpiTrimul) {
      const bool on = (int)tr.rem + li < a.n && (keep & 0xff) && (keep >> 8);
      bits = (uint32_t)__ballot(on);
      if (bits == 0) {
        // every pair of the tile is masked or padding: zeros, without the products
        const int64_t gg = (int64_t)a.npm * a.npm;
        const int64_t base = ((int64_t)tr.b * (a.O / 4) * a.npm + tr.r) * a.npm + tr.rem;
        const bf16x8 o = zero8();
        for (int u = ot0 / 2; u < (ot0 + nt) / 2; ++u) {
          int side, c0;
          trimul_pair(u, side, c0);
          bf16* dst = (side ? a.pb : a.pa) + base + (int64_t)(c0 + (lane >> 2)) * gg + 8 * (lane & 3);
          *reinterpret_cast<bf16x8*>(dst) = o;
          *reinterpret_cast<bf16x8*>(dst + 16 * gg) = o;
        }
        return;
      }
    }
    if constexpr (EPI == kEpiOpm) {
      bits = (uint32_t)__ballot((int)tr.rem + li < a.depth && keep);
      if (ot0 == 0 && g == 0)
        a.mt[((int64_t)tr.b * a.n + tr.r) * a.sp + tr.rem + li] = (bf16)((bits >> li) & 1 ? 1.f : 0.f);
    }
    const uint32_t bits_g = bits >> (4 * g);
    // GR: the epilogue operands of the first GRS output tiles, loaded first: their wait then
    // comes after the normalisation and the first products, not right behind the previous
    // tile's stores (vmcnt counts stores too). Tiles GRS .. 7 reuse the slots of tiles 0, 1,
    // loaded once those are consumed (all 8 at once would exceed the register file).
    constexpr int GRS = 6;
    bf16x8 gy[GR ? GRS : 1][2], gr[GR ? GRS : 1][2];
    const int64_t mg = m < a.M ? m : a.M - 1;
    auto gr_load = [&](int u, bf16x8 (&yv)[2], bf16x8 (&rv)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int64_t at = mg * a.O + (ot0 + u) * 32 + 8 * (2 * k + g);
        yv[k] = *reinterpret_cast<const bf16x8*>(a.yin + at);
        if (a.residual) rv[k] = *reinterpret_cast<const bf16x8*>(a.res + at);
      }
    };
    if constexpr (GR) {
#pragma unroll
      for (int u = 0; u < GRS; ++u)
        if (u < nt) gr_load(u, gy[u], gr[u]);
    }
    // the MFMA operands: hi + lo of the activations (LO), else the rows of x themselves
    // (kXLn: normalised in place)
    bf16x8 xh[LO ? KS : 1], xl[LO ? KS : 1];
    if (XSRC == kXBf16) {
    } else if (XSRC == kXLn) {
      float s1 = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) s1 += (float)x[s][e];
      const bool plain = a.ln_plain != 0;
      const float mean = plain ? 0.f : pair_sum(s1) * (1.f / K);
      // (K = 256: each pass converts the bf16 rows again; 128 converted values per lane held
      // from one pass to the next would not fit in registers)
      if constexpr (!LO)
#pragma unroll
        for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(x[s]));
      float s2 = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = (float)x[s][e] - mean;
          s2 += d * d;
        }
      const float rstd = plain ? 1.f : __builtin_amdgcn_rsqf(pair_sum(s2) * (1.f / K) + eps);
      if constexpr (!LO)
#pragma unroll
        for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(x[s]));
      const float mr = -mean * rstd;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        // read per tile: held across the loop, the affine would take K registers (K = 256: the
        // offset also waits for the previous step's values, so that the scheduler cannot issue
        // every step's affine reads at once)
        int c = KH * g + 8 * s;
        if constexpr (!LO) {
          if (s > 0)
            asm volatile("" : "+v"(c) : "v"(x[s - 1]));
          else
            asm volatile("" : "+v"(c));
        } else {
          asm volatile("" : "+v"(c));
        }
        const f32x4 w0 = *reinterpret_cast<const f32x4*>(lnp + c);
        const f32x4 w1 = *reinterpret_cast<const f32x4*>(lnp + c + 4);
        const f32x4 b0 = *reinterpret_cast<const f32x4*>(lnp + K + c);
        const f32x4 b1 = *reinterpret_cast<const f32x4*>(lnp + K + c + 4);
        f32x4 y0, y1;
        if constexpr (LO) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y0[e] = ((float)x[s][e] - mean) * rstd * w0[e] + b0[e];
            y1[e] = ((float)x[s][4 + e] - mean) * rstd * w1[e] + b1[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            y0[e] = fmaf(fmaf((float)x[s][e], rstd, mr), w0[e], b0[e]);
            y1[e] = fmaf(fmaf((float)x[s][4 + e], rstd, mr), w1[e], b1[e]);
          }
        }
        if constexpr (LO) {
          split8(y0, y1, xh[s], xl[s]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[s][e] = (bf16)y0[e];
            x[s][4 + e] = (bf16)y1[e];
          }
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) split8(x[2 * s], x[2 * s + 1], xh[s], xl[s]);
    }
    // one output tile: D[output][row], or turned, D[row][output]
    auto product = [&](int u, bool turned) __attribute__((always_inline)) {
      const bf16* wt = wl + (u * 32 + li) * WS + KH * g;
      f32x16 acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bf16x8 w = *reinterpret_cast<const bf16x8*>(wt + 8 * s);
        if constexpr (LO) {
          acc = turned ? mfma32(xl[s], w, acc) : mfma32(w, xl[s], acc);
          acc = turned ? mfma32(xh[s], w, acc) : mfma32(w, xh[s], acc);
        } else if constexpr (BF) {
          acc = turned ? mfma32(x[s], w, acc) : mfma32(w, x[s], acc);
        }
      }
      return acc;
    };
    // 16 rows of 32 channels as 16-byte pieces of 8 rows: channel li's pieces 2 k + g
    auto store_rows = [&](bf16* dst, const f32x16& y) __attribute__((always_inline)) {
      float p[2][8];
      acc_pieces(y, p);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (bf16)p[k][e];
        *reinterpret_cast<bf16x8*>(dst + 16 * k + 8 * g) = o;
      }
    };
    auto out_tile = [&](int ot, const bf16x8* rpre, const bf16x8* ypre = nullptr) __attribute__((always_inline)) {
      const f32x16 acc = product(ot - ot0, false);
      int seg = 0, cbase = 0;
      if (EPI == kEpiApb) (void)tile_weight_row<EPI>(a, ot, li, seg, cbase);
      if (m < a.M) row_epilogue<EPI>(a, acc, m, ot, seg, cbase, g, lb, 0.f, rpre, ypre);
    };
    if constexpr (EPI == kEpiTrimul) {
      // channel planes: lane li holds channel c0 + li, its registers the tile's positions
      const int64_t gg = (int64_t)a.npm * a.npm;
      const int64_t at = ((int64_t)tr.b * (a.O / 4) * a.npm + tr.r) * a.npm + tr.rem + li * gg;
#pragma unroll 1
      for (int u = 0; u < nt; u += 2) {
        f32x16 y = product(u, true);
        const f32x16 gate = product(u + 1, true);
        if (bits != ~0u) {
#pragma unroll
          for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e) y[4 * v + e] = keep_bit(y[4 * v + e], bits_g, v, e);
        }
        // (masked before the gate, as the reference)
#pragma unroll
        for (int r = 0; r < 16; ++r) y[r] *= sigmoid_scaled(-kLog2e * gate[r]);
        int side, c0;
        trimul_pair((ot0 + u) >> 1, side, c0);
        store_rows((side ? a.pb : a.pa) + c0 * gg + at, y);
      }
    } else if constexpr (EPI == kEpiOpm) {
      // MSA rows contiguous per channel: lane li holds channel c0 + li
      const int hd = a.O / 2;  // channels a side (32; Chai-1's grouped form 64)
      const int64_t at = (((int64_t)tr.b * a.n + tr.r) * hd + li) * a.sp + tr.rem;
#pragma unroll 1
      for (int ot = ot0; ot < ot0 + nt; ++ot) {
        f32x16 y = product(ot - ot0, true);
        const float bias = lb[ot * 32 + li];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * v + e] = keep_bit(y[4 * v + e] + bias, bits_g, v, e);
        const int side = ot * 32 >= hd ? 1 : 0;
        store_rows((side ? a.rt : a.lt) + at + (int64_t)(ot * 32 - side * hd) * a.sp, y);
      }
    } else if constexpr (EPI == kEpiPwa) {
      // value tiles: v^T keys contiguous per channel; gate tiles: token rows
      const int hd = a.O / 2;
      const int64_t bs = (int64_t)tr.b * a.depth + tr.r;
      const uint32_t inv = ((1u << 24) + a.dh - 1) / a.dh;  // c / dh = (c inv) >> 24 for c, dh <= 768
      const int j = (int)tr.rem + li;
#pragma unroll 1
      for (int ot = ot0; ot < ot0 + nt; ++ot) {
        if (ot * 32 < hd) {
          const f32x16 y = product(ot - ot0, true);
          const int c = ot * 32 + li, hh = (int)(((uint32_t)c * inv) >> 24), d = c - hh * a.dh;
          if (a.v_frag) {
            // row (s % S) dh + d of the head's S MSA rows, S = 32 / dh: 16-byte pieces of 8 keys
            const int sh = 5 - __builtin_ctz(a.dh), sb = (a.depth + (1 << sh) - 1) >> sh;
            bf16* dst = a.vt +
                        ((((int64_t)tr.b * a.heads + hh) * sb + (tr.r >> sh)) * (a.np >> 4) + (tr.rem >> 4)) * 512 +
                        (32 * g + (int)(tr.r & ((1u << sh) - 1)) * a.dh + d) * 8;
            float p[2][8];
            acc_pieces(y, p);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              bf16x8 o;
#pragma unroll
              for (int e = 0; e < 8; ++e) o[e] = (bf16)p[k][e];
              *reinterpret_cast<bf16x8*>(dst + 512 * k) = o;
            }
            continue;
          }
          store_rows(a.vt + ((((int64_t)tr.b * a.heads + hh) * a.depth + tr.r) * a.dh + d) * a.np + tr.rem, y);
        } else {
          const f32x16 acc = product(ot - ot0, false);
          float y[2][8];
          acc_pieces(acc, y);
          if (j < a.n) {
            bf16* dst = a.gate + (bs * a.n + tr.rem) * hd + li * hd + (ot * 32 - hd);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              bf16x8 o;
#pragma unroll
              for (int e = 0; e < 8; ++e) o[e] = (bf16)sigmoid_scaled(-kLog2e * y[k][e]);
              *reinterpret_cast<bf16x8*>(dst + 16 * k + 8 * g) = o;
            }
          }
        }
      }
    } else if constexpr (EPI == kEpiApbFlash) {
      // the flash core's layouts: everything but the lane's row and piece is uniform
      const int j = (int)tr.rem + li;
#pragma unroll 1
      for (int ot = ot0; ot < ot0 + nt; ++ot) {
        const int o0 = ot * 32;
        const int seg = (o0 >= apb_cs ? 1 : 0) + (o0 >= 2 * apb_cs ? 1 : 0) + (o0 >= 3 * apb_cs ? 1 : 0);
        const int cbase = o0 - seg * apb_cs;
        const int64_t head = (int64_t)a.flash_rows * a.np * a.dh;  // elements of one (b, h)
        if (seg == 2) {
          // v^T, turned: lane li is channel cbase + li and its registers 8 h .. 8 h + 7 are 8
          // consecutive key slots of the core's order, 16 h + 8 g ..
          const f32x16 acc = product(ot - ot0, true);
          const int hh = cbase >> dsh, c = (cbase & (a.dh - 1)) + li;
          bf16* dst = a.vt + ((int64_t)tr.b * a.heads + hh) * head + ((int64_t)tr.r * a.np + tr.rem) * a.dh +
                      (c >> dsh) * head + (c & (a.dh - 1)) * 32 + 8 * g;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (bf16)acc[8 * h + e];
            *reinterpret_cast<bf16x8*>(dst + 16 * h) = o;
          }
          continue;
        }
        const f32x16 acc = product(ot - ot0, false);
        float y[2][8];
        acc_pieces(acc, y);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int c = cbase + 16 * k;  // this lane: channels c + 8 g ..
          bf16x8 o;
          if (seg == 3) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              o[e] = (bf16)sigmoid_scaled((y[k][e] + lb[o0 + 16 * k + 8 * g + e] + a.gate_bias) * -kLog2e);
            if (j < a.n)
              *reinterpret_cast<bf16x8*>(a.gate + (((int64_t)tr.b * a.n + tr.r) * a.n + tr.rem) * apb_cs + c +
                                         li * apb_cs + 8 * g) = o;
            continue;
          }
          if (seg == 0) {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (bf16)((y[k][e] + lb[o0 + 16 * k + 8 * g + e]) * a.q_scale);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (bf16)y[k][e];
          }
          *reinterpret_cast<bf16x8*>((seg == 0 ? a.q : a.k) + ((int64_t)tr.b * a.heads + (c >> dsh)) * head +
                                     ((int64_t)tr.r * a.np + tr.rem) * a.dh + (c & (a.dh - 1)) + li * a.dh +
                                     8 * g) = o;
        }
      }
    } else if (EPI == kEpiResid && a.residual && nt <= 4) {
      // the residual of every output tile is loaded before the tile's first store: a wait
      // for a load issued after stores would wait for those stores too (vmcnt counts both)
      bf16x8 rv[4][2];
      const int64_t mm = m < a.M ? m : a.M - 1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (u < nt)
#pragma unroll
          for (int k = 0; k < 2; ++k)
            rv[u][k] = *reinterpret_cast<const bf16x8*>(a.res + mm * a.O + (ot0 + u) * 32 + 8 * (2 * k + g));
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (u < nt) out_tile(ot0 + u, rv[u]);
    } else if constexpr (GR) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (u < nt) {
          out_tile(ot0 + u, gr[u % GRS], gy[u % GRS]);
          if (u + GRS < 8 && u + GRS < nt) gr_load(u + GRS, gy[u % GRS], gr[u % GRS]);
        }
    } else if (K >= 256 && ((EPI == kEpiResid && a.residual) || EPI == kEpiGateResid)) {
      // the epilogue operands of each output tile (yin, the residual) are loaded one tile
      // ahead, before the previous tile's stores, into two register sets used in turn (rows
      // of 256 channels or more: shorter rows keep the registers for more waves per SIMD)
      const int64_t mm = m < a.M ? m : a.M - 1;
      const int last = ot0 + nt - 1;
      auto epi_load = [&](int ot, bf16x8 (&rv)[2], bf16x8 (&yv)[2]) __attribute__((always_inline)) {
        ot = ot < last ? ot : last;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int64_t at = mm * a.O + ot * 32 + 8 * (2 * k + g);
          if (EPI == kEpiGateResid) yv[k] = *reinterpret_cast<const bf16x8*>(a.yin + at);
          if (a.residual) rv[k] = *reinterpret_cast<const bf16x8*>(a.res + at);
        }
      };
      bf16x8 ra[2], rb[2], ya[2], yb[2];
      epi_load(ot0, ra, ya);
#pragma unroll 1
      for (int ot = ot0; ot <= last; ot += 2) {
        epi_load(ot + 1, rb, yb);
        out_tile(ot, ra, ya);
        if (ot == last) break;
        epi_load(ot + 2, ra, ya);
        out_tile(ot + 1, rb, yb);
      }
    } else {
#pragma unroll 1
      for (int ot = ot0; ot < ot0 + nt; ++ot) out_tile(ot, nullptr);
    }
  };

  // the tile after t, or t again past the last one (its rows are loaded and dropped)
  auto next = [&](const TileRun& tr) __attribute__((always_inline)) {
    return kRuns && t + stride < tiles ? run_add(tr, step, L, R) : tr;
  };
  auto next_m = [&]() __attribute__((always_inline)) { return (t + stride < tiles ? t + stride : t) * 32; };
  uint32_t k0, k1;
  if constexpr (DB) {
    // two register buffers used in turn: the next tile's rows load while the current one is
    // processed
    XT x0[NX], x1[NX];
    fetch(x0, k0, cur, t * 32);
    while (true) {
      TileRun nx = next(cur);
      fetch(x1, k1, nx, next_m());
      process(x0, k0, cur, t);
      t += stride;
      if (t >= tiles) break;
      cur = nx;
      nx = next(cur);
      fetch(x0, k0, nx, next_m());
      process(x1, k1, cur, t);
      t += stride;
      if (t >= tiles) break;
      cur = nx;
    }
  } else {
    XT x0[NX];
    fetch(x0, k0, cur, t * 32);
    while (true) {
      process(x0, k0, cur, t);
      const TileRun nx = next(cur);
      t += stride;
      if (t >= tiles) break;
      cur = nx;
      fetch(x0, k0, cur, t * 32);
    }
  }
}

// ---------------------------------------------------------------------------- pair bias
// bias[b, h, i, j] = rstd_ij * (z_ij . W'_h - mean_ij * sum_c W'_h[c]) with
// W'_h[c] = log2(e) * gamma[c] * W_b[h][c]; this equals LN_pair(z_ij) . W_b[h] * log2(e) for
// the offset-free pair norm. z is exact in bf16 and W' is carried as a bf16 pair
// hi + lo (two MFMA passes), so the bias keeps fp32 accuracy: its error does not grow with
// the logit size (large pair logits would otherwise shift the softmax weights).
// One wave handles a tile of 32 consecutive keys j of one (b, i): lane (li, g) loads its
// row's channels 16 t + 8 g .. 16 t + 8 g + 7 for t < C / 16, so each load instruction reads
// 32 contiguous bytes per row (lanes l and l ^ 32 together), the statistics come from those
// registers (two passes, halves joined across lane l ^ 32), and the heads x keys block is
// one 32 x 32 MFMA tile (A = W' rows, B = the z rows; channels 16 t .. 16 t + 15 feed step t).
// W waves per workgroup, workgroup bx of gx.
template <int C, int W>
__device__ __forceinline__ void pair_bias_body(const PairBiasArgs& a, const int bx, const int gx) {
  constexpr int kU = C / 16;  // 8-channel chunks per lane (each lane half holds C / 2)
  __shared__ float wsum_s[W][32];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int n = a.n;
  const int njt = a.np / 32;
  const int64_t stride = (int64_t)gx * W;

  // Tiles are fetched one ahead (two register buffers used alternately); a fetch past the
  // last tile re-reads the last tile, so every load stays inside z.
  auto fetch = [&](bf16x8* zf, int64_t tile) {
    const int64_t tt = tile < a.tiles ? tile : a.tiles - 1;
    const int64_t bi = tt / njt;
    const int j0 = (int)(tt - bi * njt) * 32;
    const int key = min(j0 + li, n - 1);
    int64_t row = bi * n + key;  // pair position (query i, key): z[b, i, key]
    if (a.transposed) {          // z[b, key, i]
      const int64_t b = bi / n;
      row = (b * n + key) * n + (bi - b * n);
    }
    const bf16* zr = a.z + row * C + 8 * g;
#pragma unroll
    for (int u = 0; u < kU; ++u) zf[u] = ld8(zr + 16 * u);
  };
  int64_t t = (int64_t)bx * W + wave;
  bf16x8 z0[kU], z1[kU];
  fetch(z0, t);

  bf16x8 wf[kU], wl[kU];
  float rs = 0.f;
  const float* wrow = a.w_bias + min(li, a.heads - 1) * C + 8 * g;
  const float* lrow = a.ln_w + 8 * g;
  const float keep = li < a.heads ? kLog2e : 0.f;
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(wrow + 16 * u);
    const f32x4 w1 = *reinterpret_cast<const f32x4*>(wrow + 16 * u + 4);
    const f32x4 l0 = *reinterpret_cast<const f32x4*>(lrow + 16 * u);
    const f32x4 l1 = *reinterpret_cast<const f32x4*>(lrow + 16 * u + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = keep * (e < 4 ? l0[e] * w0[e] : l1[e - 4] * w1[e - 4]);
      wf[u][e] = (bf16)v;
      wl[u][e] = (bf16)(v - (float)wf[u][e]);
      rs += v;
    }
  }
  rs = pair_sum(rs);
  if (g == 0) wsum_s[wave][li] = rs;
  __syncthreads();

  auto process = [&](const bf16x8* zf, int64_t tile) {
    float s1 = 0.f;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) s1 += (float)zf[u][e];
    const float mean = pair_sum(s1) * (1.f / C);
    float s2 = 0.f;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = (float)zf[u][e] - mean;
        s2 += d * d;
      }
    const float rstd = __builtin_amdgcn_rsqf(pair_sum(s2) * (1.f / C) + a.eps);
    f32x16 acc = zero16();
#pragma unroll
    for (int u = 0; u < kU; ++u) acc = mfma32(wl[u], zf[u], acc);
#pragma unroll
    for (int u = 0; u < kU; ++u) acc = mfma32(wf[u], zf[u], acc);

    const int64_t bi = tile / njt;
    const int key = (int)(tile - bi * njt) * 32 + li;
    const int64_t b = bi / n;
    const int64_t i = bi - b * n;
    const bool valid = key < n && a.mask[b * n + key] != 0;
    float* out = a.bias + (b * a.heads * n + i) * a.np + key;
    // blocked: entry (query i, key) of head h at bias_index(b heads + h, ...), a whole number
    // of head strides (np^2) apart
    if (a.blocked) out = a.bias + bias_index(b * a.heads, a.np / 32, i, key);
    const int64_t hstride = a.blocked ? (int64_t)a.np * a.np : (int64_t)n * a.np;
    const float masked = a.blocked ? -INFINITY : kMaskedLogit;
    const int64_t xe = b * a.extra_sb + i * a.extra_si + key;  // head 0's extra logit
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int h = acc_row(r, g);
      if (h < a.heads) {
        float y = rstd * (acc[r] - mean * wsum_s[wave][h]);
        if (a.extra && valid) {
          const int64_t at = xe + h * a.extra_sh;
          y += kLog2e * (a.extra_bf16 ? (float)static_cast<const bf16*>(a.extra)[at]
                                      : static_cast<const float*>(a.extra)[at]);
        }
        out[h * hstride] = valid ? y : masked;
      }
    }
  };
  while (t < a.tiles) {
    fetch(z1, t + stride);
    process(z0, t);
    t += stride;
    if (t >= a.tiles) break;
    fetch(z0, t + stride);
    process(z1, t);
    t += stride;
  }
}

template <int C>
__global__ __launch_bounds__(256) void apb_pair_bias(PairBiasArgs a) {
  pair_bias_body<C, 4>(a, blockIdx.x, gridDim.x);
}

// The single track's projections and its pair bias, which do not depend on each other, in one
// launch: workgroups below gx * gy run the GEMM, the rest the bias. Where the GEMM leaves CUs free,
// either kernel alone is one chain of latencies; together they take the longer one. 201 tokens of 384
// channels: 13.3 + 10.1 -> 15.6 us. launch_apb_project_bias has the rule.
template <int NO>
__global__ __launch_bounds__(512) void apb_project_bias(RowGemmArgs a, PairBiasArgs p, int gx, int gy) {
  const int id = blockIdx.x, gemm = gx * gy;
  if (id < gemm)
    row_gemm_body<kEpiApb, kXLn, NO, 2>(a, id % gx, id / gx);
  else
    pair_bias_body<128, kGemmWaves>(p, id - gemm, gridDim.x - gemm);
}

// The same bias at pair width 128 with the z rows staged through LDS: each wave owns two 8 KB
// tile buffers that its own LDS DMA fills (each transfer is 4 whole rows, 1 KB contiguous for
// the un-transposed orientation, swizzled by off128), one tile ahead of the one it processes, so
// the rows arrive as full lines instead of 32-byte pieces of 32 rows per load; a wave's buffers
// are its own, so the loop has no barrier. Persistent: every wave walks tiles t0, t0 + stride, ...
// (stride = 4 gridDim.x). The waits count this wave's vector-memory operations, which on gfx950
// include its stores: waiting for tile k's rows also waits for the stores of tile k - 1, issued
// one tile earlier.
__global__ __launch_bounds__(256, 2) void apb_pair_bias_lds(PairBiasArgs a) {
  constexpr int C = 128, kU = C / 16;
  __shared__ float wsum_s[4][32];
  __shared__ __attribute__((aligned(16))) bf16 zt[4][2][32 * C];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int n = a.n;
  const int njt = a.np / 32;
  const int64_t stride = (int64_t)gridDim.x * 4;
  const uint32_t zt_lds = lds_addr(&zt[wave][0][0]);

  // Rows j0 .. j0 + 31 of tile `tile` (keys past n repeat key n - 1: finite, masked) into
  // buffer buf; a tile index past the end re-reads the last tile. Piece p = rows 4 p .. 4 p + 3:
  // lane L fills slot L & 15 of row 4 p + L / 16 with the row's chunk (L & 15) ^ (row & 15).
  auto tile_dma = [&](int64_t tile, int buf) {
    const int64_t tt = tile < a.tiles ? tile : a.tiles - 1;
    const int64_t bi = tt / njt;
    const int j0 = (int)(tt - bi * njt) * 32;
    const int64_t b = bi / n, i = bi - b * n;
    const bf16* base = a.transposed ? a.z + (b * n * n + i) * C : a.z + bi * n * C;
    const uint32_t rstride = a.transposed ? (uint32_t)n * C * 2 : (uint32_t)C * 2;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int r = 4 * p + (lane >> 4);
      const int key = min(j0 + r, n - 1);
      dma16_stream(base, (uint32_t)key * rstride + 16 * ((lane & 15) ^ (r & 15)),
                   zt_lds + (uint32_t)(buf * 32 * C * 2 + 1024 * p));
    }
  };
  int64_t t = (int64_t)blockIdx.x * 4 + wave;
  if (t < a.tiles) tile_dma(t, 0);

  bf16x8 wf[kU], wl[kU];
  float rs = 0.f;
  const float* wrow = a.w_bias + min(li, a.heads - 1) * C + 8 * g;
  const float* lrow = a.ln_w + 8 * g;
  const float keep = li < a.heads ? kLog2e : 0.f;
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(wrow + 16 * u);
    const f32x4 w1 = *reinterpret_cast<const f32x4*>(wrow + 16 * u + 4);
    const f32x4 l0 = *reinterpret_cast<const f32x4*>(lrow + 16 * u);
    const f32x4 l1 = *reinterpret_cast<const f32x4*>(lrow + 16 * u + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = keep * (e < 4 ? l0[e] * w0[e] : l1[e - 4] * w1[e - 4]);
      wf[u][e] = (bf16)v;
      wl[u][e] = (bf16)(v - (float)wf[u][e]);
      rs += v;
    }
  }
  rs = pair_sum(rs);
  if (g == 0) wsum_s[wave][li] = rs;
  __syncthreads();
  if (t >= a.tiles) return;  // no transfer of this wave is in flight

  for (int k = 0;; ++k) {
    const bool more = t + stride < a.tiles;
    if (more) {
      tile_dma(t + stride, (k + 1) & 1);
      wait_vm_lds<8>();  // tile k's rows (and everything before them) landed
    } else {
      wait_vm_lds<0>();
    }
    bf16x8 zf[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) zf[u] = ld8(&zt[wave][k & 1][off128(li, 2 * u + g)]);

    float s1 = 0.f;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) s1 += (float)zf[u][e];
    const float mean = pair_sum(s1) * (1.f / C);
    float s2 = 0.f;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = (float)zf[u][e] - mean;
        s2 += d * d;
      }
    const float rstd = __builtin_amdgcn_rsqf(pair_sum(s2) * (1.f / C) + a.eps);
    f32x16 acc = zero16();
#pragma unroll
    for (int u = 0; u < kU; ++u) acc = mfma32(wl[u], zf[u], acc);
#pragma unroll
    for (int u = 0; u < kU; ++u) acc = mfma32(wf[u], zf[u], acc);

    const int64_t bi = t / njt;
    const int key = (int)(t - bi * njt) * 32 + li;
    const int64_t b = bi / n;
    const int64_t i = bi - b * n;
    const bool valid = key < n && a.mask[b * n + key] != 0;
    float* out = a.bias + (b * a.heads * n + i) * a.np + key;
    if (a.blocked) out = a.bias + bias_index(b * a.heads, a.np / 32, i, key);
    const int64_t hstride = a.blocked ? (int64_t)a.np * a.np : (int64_t)n * a.np;
    const float masked = a.blocked ? -INFINITY : kMaskedLogit;
    const int64_t xe = b * a.extra_sb + i * a.extra_si + key;  // head 0's extra logit
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int h = acc_row(r, g);
      if (h < a.heads) {
        float y = rstd * (acc[r] - mean * wsum_s[wave][h]);
        if (a.extra && valid) {
          const int64_t at = xe + h * a.extra_sh;
          y += kLog2e * (a.extra_bf16 ? (float)static_cast<const bf16*>(a.extra)[at]
                                      : static_cast<const float*>(a.extra)[at]);
        }
        out[h * hstride] = valid ? y : masked;
      }
    }
    t += stride;
    if (t >= a.tiles) break;
  }
}

// ---------------------------------------------------------------------------- attention
// One workgroup per (32 queries, head, batch); its four waves split the key blocks
// (wave w takes blocks w, w + 4, ...), run an online softmax each and are merged through LDS.
// Per 32-key block: S^T = K Q^T + bias^T (A = k rows, B = q rows, the bias as the MFMA
// accumulator input: lane (li, g) holds query li and keys 8 v + 4 g + e), then
// O^T += V^T P^T (A = v^T rows in the permuted key order, B = this lane's 16 weights).
// DT 32-channel tiles of the head (DT = 2: heads of 40 to 64 channels): DT 32 x 32 output
// tiles, 2 DT MFMAs of the logits per key block.
template <int DT>
__global__ __launch_bounds__(256) void apb_attention(ApbAttnArgs a) {
  __shared__ float sm[4][32], sl[4][32];
  __shared__ float so[3][64][16 * DT];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int q0 = blockIdx.x * 32, h = blockIdx.y, b = blockIdx.z;
  const int n = a.n, dh = a.dh, cs = a.cs;

  const int bb = b / a.rows_per_bias;  // the batch element of the bias and the key mask
  int any = 0;
  for (int t = threadIdx.x; t < n; t += 256) any |= a.mask[(int64_t)bb * n + t];
  const bool empty = !__syncthreads_or(any);

  const int qr = min(q0 + li, n - 1);
  const bf16* qp = a.q + ((int64_t)b * n + qr) * cs + h * dh;
  bf16x8 qf[2 * DT];
#pragma unroll
  for (int f = 0; f < 2 * DT; ++f) qf[f] = 16 * f + 8 * g < dh ? ld8(qp + 16 * f + 8 * g) : zero8();
  const float* bp = a.bias + (((int64_t)bb * a.heads + h) * n + qr) * a.np + 4 * g;
  const bf16* vp[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
    vp[t] = a.vt + (((int64_t)b * a.heads + h) * dh + min(32 * t + li, dh - 1)) * a.np + 8 * g;
  const bf16* kbase = a.k + (int64_t)b * n * cs + h * dh;

  float m = -INFINITY, l = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = zero16();
  const int nkb = a.np / 32;
  for (int kb = wave; kb < nkb; kb += 4) {
    const bf16* kp = kbase + (int64_t)min(kb * 32 + li, n - 1) * cs;
    bf16x8 kf[2 * DT];
#pragma unroll
    for (int f = 0; f < 2 * DT; ++f) kf[f] = 16 * f + 8 * g < dh ? ld8(kp + 16 * f + 8 * g) : zero8();
    f32x16 s;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(bp + kb * 32 + 8 * v);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * v + e] = bv[e];
    }
    bf16x8 vf[DT][2];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      vf[t][0] = ld8(vp[t] + kb * 32);
      vf[t][1] = ld8(vp[t] + kb * 32 + 16);
    }
#pragma unroll
    for (int f = 0; f < 2 * DT; ++f) s = mfma32(kf[f], qf[f], s);

    float bm = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bm = fmaxf(bm, s[r]);
    bm = pair_max(bm);
    const float mn = fmaxf(m, bm);
    const float alpha = fast_exp2(m - mn);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - mn);
      ps += s[r];
    }
    l = l * alpha + ps;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] *= alpha;

    if (kb * 32 + 32 > n) {  // keys past n: their v^T entries were never written
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = kb * 32 + 4 * g + 8 * (j >> 2) + (j & 3);
          if (key >= n) vf[t][0][j] = (bf16)0.f;
          if (key + 16 >= n) vf[t][1][j] = (bf16)0.f;
        }
    }
    bf16x8 p0, p1;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p0[j] = (bf16)s[j];
      p1[j] = (bf16)s[8 + j];
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      o[t] = mfma32(vf[t][0], p0, o[t]);
      o[t] = mfma32(vf[t][1], p1, o[t]);
    }
  }
  l = pair_sum(l);

  if (g == 0) {
    sm[wave][li] = m;
    sl[wave][li] = l;
  }
  __syncthreads();
  const float mx = fmaxf(fmaxf(sm[0][li], sm[1][li]), fmaxf(sm[2][li], sm[3][li]));
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) total += sl[w][li] * fast_exp2(sm[w][li] - mx);
  const float f = empty ? 0.f : fast_exp2(m - mx) / total;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] *= f;
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) so[wave - 1][lane][16 * t + r] = o[t][r];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 0; w < 3; ++w)
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[t][r] += so[w][lane][16 * t + r];
  const int qq = q0 + li;
  if (qq >= n) return;
  const int64_t row = ((int64_t)b * n + qq) * cs + h * dh;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int d0 = 32 * t + 8 * v + 4 * g;
      if (d0 < dh) {
        const bf16x4 gv = *reinterpret_cast<const bf16x4*>(a.gate + row + d0);
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = o[t][4 * v + e] * (float)gv[e];
        *reinterpret_cast<f32x4*>(a.og + row + d0) = y;
      }
    }
}

}  // namespace

template <int EPI, int XSRC, int NO>
void launch_row_gemm_t(const RowGemmArgs& a, hipStream_t stream) {
  const int otiles = a.O / 32;
  const dim3 grid((unsigned)((a.M + 31) / 32), (unsigned)((otiles + NO - 1) / NO));
  const size_t lds = row_gemm_lds(XSRC, a.K);
  // one group a wave, and workgroups to fill the second place on a CU (with fewer, the form held to 128
  // VGPRs is up to 2% slower: the output projection of 201 tokens x 384). Eight output tiles a workgroup
  // leave a wave all groups: one only at the 64 channels that just kEpiLinear brings here.
  auto kernel = row_gemm<EPI, XSRC, NO, 2>;
  if constexpr (NO < kGemmWaves || EPI == kEpiLinear)
    if (a.K / 64 <= kGemmWaves / NO && (int64_t)grid.x * grid.y > cu_count()) kernel = row_gemm<EPI, XSRC, NO, 1>;
  if (lds > 65536)  // beyond the default dynamic LDS size
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  kernel<<<grid, 64 * kGemmWaves, lds, stream>>>(a);
}

// Tile shapes: the LayerNorm-fed GEMMs give each workgroup several output tiles (the tile is
// normalised once per workgroup); the fp32-fed ones split k 8 ways when k is long, and give the
// waves separate output tiles when k has fewer groups than waves.
// Output parts: the fewest equal parts of whole tiles whose weight rows keep a workgroup's LDS at
// or below 72 KiB (two workgroups of 4 waves per CU). Measured on the
// template stacks: splitting at 56 KiB instead (three workgroups per CU, the input read twice
// for 384 outputs) was 2.5% slower per block. Rows of 256 channels or more: at most 160 KiB
// (one workgroup of 8 waves per CU), so that each part re-reads and re-normalises the input
// rows as few times as possible.
size_t row_stream_lds_cap(int K) { return (K >= 256 ? 160 : 72) * 1024; }
int row_stream_parts(int K, int O, int unit) {
  const int units = O / 32 / unit;
  int parts = 1;
  while (parts < units && (units % parts != 0 || row_stream_lds(K, O, O / parts) > row_stream_lds_cap(K))) ++parts;
  return parts;
}

// Few rows leave CUs without a workgroup, and each then takes as long as its weight rows: the parts
// are doubled until every CU has one. Not for kEpiGateResid: its out may alias the input rows, which
// only a workgroup that writes whole rows reads before it writes them.
template <int EPI, int XSRC, int K>
void launch_row_stream_t(const RowGemmArgs& a, hipStream_t stream) {
  constexpr int kStreamWaves = stream_waves(K);
  const int64_t tiles = (a.M + 31) / 32, want = (tiles + kStreamWaves - 1) / kStreamWaves;
  int parts = row_stream_parts(K, a.O, stream_unit(EPI));
  const int units = a.O / 32 / stream_unit(EPI);
  if (EPI != kEpiGateResid)
    while (units % (2 * parts) == 0 && want * parts * 2 <= cu_count()) parts *= 2;
  const size_t lds = row_stream_lds(K, a.O, a.O / parts);
  auto kernel = row_stream<EPI, XSRC, K>;
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  const int64_t per_cu =
      resident_blocks(reinterpret_cast<const void*>(kernel), 64 * kStreamWaves, lds);
  int64_t blocks = std::max<int64_t>(1, cu_count() * per_cu / parts);
  // Rows for one pass: a grid width of whole 8s puts the parts of a run of rows on one XCD (workgroups
  // go to the 8 in turn), where they share the rows in its L2 and the next kernel of the same walk finds its
  // input (the surplus workgroups leave at once): transition of 9409 x 128 rows x 2 27.7 -> 23.6 us. Not for
  // a few runs, whose parts would crowd their XCDs (500 x 256 rows x 4: 21.9 -> 33.8).
  if (blocks >= want) blocks = parts > 1 && want >= 16 ? (want + 7) / 8 * 8 : want;
  kernel<<<dim3((unsigned)std::max<int64_t>(1, blocks), (unsigned)parts), 64 * kStreamWaves, lds, stream>>>(a);
}

// The streaming kernel's cases: the pair path's short rows, a part of the weights fitting in LDS.
template <int EPI, int XSRC>
bool launch_row_stream(const RowGemmArgs& a, hipStream_t stream) {
  // k 64 or 128; bf16 rows (normalised or plain) also 256; plain bf16 rows also 512
  if (a.K != 64 && a.K != 128 && !(XSRC != kXF32 && a.K == 256) && !(XSRC == kXBf16 && a.K == 512))
    return false;
  const size_t cap = a.K >= 256 ? 160 * 1024 : 80 * 1024;
  if (row_stream_lds(a.K, a.O, a.O / row_stream_parts(a.K, a.O, stream_unit(EPI))) > cap) return false;
  if (a.K == 64) {
    launch_row_stream_t<EPI, XSRC, 64>(a, stream);
  } else if (a.K == 128) {
    launch_row_stream_t<EPI, XSRC, 128>(a, stream);
  } else if constexpr (XSRC != kXF32) {
    if (a.K == 256)
      launch_row_stream_t<EPI, XSRC, 256>(a, stream);
    else if constexpr (XSRC == kXBf16)
      launch_row_stream_t<EPI, XSRC, 512>(a, stream);
  }
  return true;
}

void launch_row_gemm(const RowGemmArgs& a, int epi, int xsrc, hipStream_t stream) {
  // short rows of the pair path: the streaming kernel (false: not a case it takes)
  if (xsrc == kXLn) {
    if (epi == kEpiApb && a.flash_rows > 0) {  // (pair widths 64, 128, 256: always a case)
      (void)launch_row_stream<kEpiApbFlash, kXLn>(a, stream);
      return;
    }
    if (epi == kEpiApb && launch_row_stream<kEpiApb, kXLn>(a, stream)) return;
    if (epi == kEpiTrimul && launch_row_stream<kEpiTrimul, kXLn>(a, stream)) return;
    if (epi == kEpiStoreY && launch_row_stream<kEpiStoreY, kXLn>(a, stream)) return;
    if (epi == kEpiGateResid && launch_row_stream<kEpiGateResid, kXLn>(a, stream)) return;
    if (epi == kEpiSwiglu && launch_row_stream<kEpiSwiglu, kXLn>(a, stream)) return;
    if (epi == kEpiResid && a.ln_plain && launch_row_stream<kEpiResid, kXBf16>(a, stream)) return;
    if (epi == kEpiResid && launch_row_stream<kEpiResid, kXLn>(a, stream)) return;
    if (epi == kEpiOpm && launch_row_stream<kEpiOpm, kXLn>(a, stream)) return;
    if (epi == kEpiPwa) {
      // tokens padded to np: the key-contiguous values leave the streaming kernel in whole 16-byte
      // pieces (512 rows x 256 tokens of 64 channels: 22 -> 19 us). row_gemm stores them 2 bytes a lane either way and takes
      // the rows as they are (192 channels, 128 x 129 tokens, 8 x 24: 83 us padded, 77 not)
      RowGemmArgs padded = a;
      padded.tmap = kMapPadKeys;
      padded.M = a.M / a.n * a.np;
      if (launch_row_stream<kEpiPwa, kXLn>(padded, stream)) return;
    }
  } else if (epi == kEpiResid && launch_row_stream<kEpiResid, kXF32>(a, stream)) {
    return;
  }
  if (epi == kEpiApb && xsrc == kXLn)
    launch_row_gemm_t<kEpiApb, kXLn, 4>(a, stream);
  else if (epi == kEpiSwiglu && xsrc == kXLn)
    launch_row_gemm_t<kEpiSwiglu, kXLn, 8>(a, stream);
  else if (epi == kEpiResid && xsrc == kXF32) {
    // k split into KS parts of whole 64-wide groups with none left idle (8 from 6 groups up)
    const int groups = a.K / 64;
    if (groups >= 6)
      launch_row_gemm_t<kEpiResid, kXF32, 1>(a, stream);
    else if (groups >= 4)
      launch_row_gemm_t<kEpiResid, kXF32, 2>(a, stream);
    else if (groups >= 2)
      launch_row_gemm_t<kEpiResid, kXF32, 4>(a, stream);
    else
      launch_row_gemm_t<kEpiResid, kXF32, 8>(a, stream);
  }
  else if (epi == kEpiResid && xsrc == kXLn) {
    if (a.O >= 256)
      launch_row_gemm_t<kEpiResid, kXLn, 8>(a, stream);
    else if (a.O >= 128)
      launch_row_gemm_t<kEpiResid, kXLn, 4>(a, stream);
    else
      launch_row_gemm_t<kEpiResid, kXLn, 2>(a, stream);
  } else if (epi == kEpiPwa && xsrc == kXLn)
    launch_row_gemm_t<kEpiPwa, kXLn, 8>(a, stream);
  else if (epi == kEpiOpm && xsrc == kXLn)
    launch_row_gemm_t<kEpiOpm, kXLn, 2>(a, stream);
  else if (epi == kEpiTrimul && xsrc == kXLn)
    launch_row_gemm_t<kEpiTrimul, kXLn, 8>(a, stream);
  else if (epi == kEpiStoreY && xsrc == kXLn) {
    if (a.O >= 256)
      launch_row_gemm_t<kEpiStoreY, kXLn, 8>(a, stream);
    else if (a.O >= 128)
      launch_row_gemm_t<kEpiStoreY, kXLn, 4>(a, stream);
    else
      launch_row_gemm_t<kEpiStoreY, kXLn, 2>(a, stream);
  } else if (epi == kEpiLinear && xsrc == kXLn) {
    if (a.O >= 256)
      launch_row_gemm_t<kEpiLinear, kXLn, 8>(a, stream);
    else if (a.O >= 128)
      launch_row_gemm_t<kEpiLinear, kXLn, 4>(a, stream);
    else
      launch_row_gemm_t<kEpiLinear, kXLn, 2>(a, stream);
  } else if (epi == kEpiGateResid && xsrc == kXLn) {
    // one workgroup column (O <= 256): a workgroup owns its rows, so out may alias the input
    if (a.O > 128)
      launch_row_gemm_t<kEpiGateResid, kXLn, 8>(a, stream);
    else if (a.O > 64)
      launch_row_gemm_t<kEpiGateResid, kXLn, 4>(a, stream);
    else
      launch_row_gemm_t<kEpiGateResid, kXLn, 2>(a, stream);
  }
}

void launch_apb_pair_bias(const PairBiasArgs& a, hipStream_t stream) {
  // pair width 128: the LDS-staged persistent kernel (two workgroups per CU), unless a
  // transposed key offset would not fit its 32-bit DMA offset
  if (a.c == 128 && (!a.transposed || (int64_t)a.n * a.n * 256 <= 0xffffffffLL)) {
    int64_t blocks = (a.tiles + 3) / 4;
    const int64_t cap = (int64_t)cu_count() * 2;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    apb_pair_bias_lds<<<dim3((unsigned)blocks), 256, 0, stream>>>(a);
    return;
  }
  auto kernel = a.c == 64 ? apb_pair_bias<64> : a.c == 256 ? apb_pair_bias<256> : apb_pair_bias<128>;
  const int64_t cap = (int64_t)cu_count() * resident_blocks(reinterpret_cast<const void*>(kernel), 256, 0);
  const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>((a.tiles + 3) / 4, cap));
  kernel<<<dim3((unsigned)blocks), 256, 0, stream>>>(a);
}

// One launch while each CU that the GEMM leaves free gets at most 42 bias tiles of 32 keys, a few per wave
// (more where more than 96 are free: the bias is then the longer kernel of the two either way): past that
// its register-fed form (32-byte pieces of 32 rows a load) falls behind the LDS-DMA kernel on every CU.
// The whole call, two launches -> one (free CUs, tiles on each): 384 channels, 201 tokens 36.3 -> 28.9 us
// (172, 8), 320 42.1 -> 34.4 (136, 24), 384 43.7 -> 42.1 (112, 41), 448 48.6 -> 51.5 (88, 71), 512 52.3 -> 71.1 (64,
// 128); 5 x 100 tokens 38.4 -> 34.3 (64, 31); 192 channels, 512 tokens 46.5 -> 45.4 (160, 51), 640 55.5 -> 59.3 (136, 94),
// 768 66.9 -> 83.2 (112, 165); 512 channels, 320 44.8 -> 39.9 (96, 33), 384 47.0 -> 51.7 (64, 72); 768 channels,
// 256 50.3 -> 41.5 (64, 32), 288 53.5 -> 56.9 (40, 65). Beside a trunk's pair track: 4 blocks of 201 / 256
// tokens 1109 -> 1094 and 1221 -> 1202 us, 320 to 384 within 0.6%.
void launch_apb_project_bias(const RowGemmArgs& a, const PairBiasArgs& p, hipStream_t stream) {
  constexpr int NO = 4;
  const int64_t gx = (a.M + 31) / 32, gy = (a.O / 32 + NO - 1) / NO, rest = cu_count() - gx * gy;
  const bool stream_case = a.K == 64 || a.K == 128 || a.K == 256;  // (row_stream's widths)
  if (stream_case || p.c != 128 || rest <= 0 || p.tiles > rest * std::max<int64_t>(42, rest / 2 - 6)) {
    launch_row_gemm(a, kEpiApb, kXLn, stream);
    launch_apb_pair_bias(p, stream);
    return;
  }
  const size_t lds = row_gemm_lds(kXLn, a.K);
  auto kernel = apb_project_bias<NO>;
  if (lds > 65536 - 8192)  // (with the bias's static LDS)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  // one workgroup per CU (registers): the bias takes the CUs that the GEMM leaves
  const int64_t bias = std::min<int64_t>((p.tiles + kGemmWaves - 1) / kGemmWaves, rest);
  kernel<<<dim3((unsigned)(gx * gy + bias)), 64 * kGemmWaves, lds, stream>>>(a, p, (int)gx, (int)gy);
}

void launch_apb_attention(const ApbAttnArgs& a, int batch, hipStream_t stream) {
  const dim3 grid((unsigned)((a.n + 31) / 32), (unsigned)a.heads, (unsigned)batch);
  if (a.dh > 32)
    apb_attention<2><<<grid, 256, 0, stream>>>(a);
  else
    apb_attention<1><<<grid, 256, 0, stream>>>(a);
}

}  // namespace ffk
