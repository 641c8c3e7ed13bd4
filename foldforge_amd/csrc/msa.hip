// MSA pair-weighted averaging on gfx950 (the MSA stack's pair-to-MSA update).
//
// Equations: src/foldforge/models/checkpoints/legacy/attention.py:203-223 (MSAAttention):
//   x = LN_msa(m); w[h, i, :] = softmax_j(LN_pair(z)[i, j] . W_b[h]) over valid keys j;
//   o[s, i, h] = sum_j w[h, i, j] v[s, j, h], v = x W_v^T; out = m + (sigmoid(x W_g^T) o) W_out^T.
// The weights do not depend on the MSA row s, so per head the average is one GEMM
//   O_h[(s, c)][i] = sum_j v^T_h[(s, c)][j] w_h[i][j]
// with all S MSA rows stacked along M. The C-ABI (api.hip) runs (the token-row GEMMs through
// launch_row_gemm, which takes the streaming row_stream where the width allows):
//   row_gemm<kEpiPwa, kXLn> (single.hip): LN_msa + value / gate projections -> v^T, gate
//   apb_pair_bias (single.hip): pair logits in log2 units, masked keys very negative
//   pwa_softmax: the softmax of every (batch, head, query) row -> bf16 weights
//   8 heads of 8, 16 or 32 channels on 64 MSA channels: pwa_fused, everything behind the softmax
//   in one kernel; other shapes: pwa_average, the per-head GEMM, gated -> bf16 (gate * o), and
//   row_gemm<kEpiResid, kXLn>, the output projection and the residual.
#include "ffk_device.h"
#include "ffk_kernels.h"

namespace ffk {

namespace {

// A row whose largest logit is below this has no valid key: its weights are all zero.
constexpr float kNoKey = -1e29f;

// One wave per row of np logits: maximum, exp2 sum, then the normalised bf16 weights.
__global__ __launch_bounds__(256) void pwa_softmax(PwaSoftmaxArgs a) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= a.rows) {
    // frag: the workgroups behind the rows pack the output projection, a 16-byte piece per thread
    const int64_t idx = ((int64_t)blockIdx.x - (a.rows + 3) / 4) * 256 + threadIdx.x;
    if (a.frag && idx >= 0 && idx < 8 * a.hd) {
      const int l = (int)idx & 63, t = (int)(idx >> 6), kt = t % (a.hd / 16), ot = t / (a.hd / 16);
      const float* src = a.w_out + (32 * ot + (l & 31)) * a.hd + 8 * kt + (a.hd / 2) * (l >> 5);
      bf16x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (bf16)src[e];
      *reinterpret_cast<bf16x8*>(a.wo + idx * 8) = v;
    }
    return;
  }
  const float* x = a.logits + row * a.np;
  bf16* w = a.w + row * a.np;
  const int64_t bh = row / a.n;
  const int q = (int)(row - bh * a.n);
  if (a.frag) w = a.w + ((bh * ((a.n + 31) / 32) + q / 32) * (a.np / 16)) * 512 + (q & 31) * 8;
  float mx = -INFINITY;
  for (int j = 4 * lane; j < a.np; j += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(x + j);
    mx = fmaxf(fmaxf(mx, fmaxf(v[0], v[1])), fmaxf(v[2], v[3]));
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  float sum = 0.f;
  for (int j = 4 * lane; j < a.np; j += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(x + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum += fast_exp2(v[e] - mx);
  }
  sum = wave_sum(sum);
  const float inv = mx > kNoKey ? 1.f / sum : 0.f;
  for (int j = 4 * lane; j < a.np; j += 256) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(x + j);
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (bf16)(fast_exp2(v[e] - mx) * inv);
    *reinterpret_cast<bf16x4*>(w + (a.frag ? (j >> 4) * 512 + ((j >> 3) & 1) * 256 + (j & 7) : j)) = o;
  }
}

// The weighted average, gate, output projection and residual for 8 heads of DH = 8, 16 or 32
// channels and 64 MSA channels. A workgroup of 8 waves takes S = 32 / DH MSA rows x 128 queries:
//   wave h: O_h[(s, d)][q] = sum_j v^T_h[(s, d)][j] w_h[q][j], one 32-row A tile (the head's S
//   rows) x 4 query tiles, both operands straight from memory in fragment order (a 16-key step of
//   a tile is one contiguous KB: [tile][k / 16][lane][8]), two steps fetched ahead;
//   the averages are gated in fp32 (a lane's gate values travel behind the key loop) and go to LDS as
//   bf16 token rows [(s, q)][8 DH] (64 KB for every DH, 16-byte pieces XOR-swizzled by row), the
//   one rounding between the average and the projection;
//   then each wave projects its share of the (token tile, 32-channel output tile) pairs: the LDS rows
//   as the B operand, W_out fragments as A (step t: channels 4 DH g + 8 t ..); residual and
//   16-byte stores.
// Rows past the depth and queries past n hold whatever the operands held: they are not stored
// and no product mixes rows or queries. This replaces a 128 x 128-tile GEMM per head, its gated
// output in memory and a token-row GEMM: 512 x 256 tokens, 8 x 8: 50 -> 20 us. Bound by the
// fragment traffic from L2 (640 KB a workgroup at 256 keys: 168 MB in all, 8.3 TB/s; matrix cores busy 7%).
template <int DH>
__global__ __launch_bounds__(512) void pwa_fused(PwaFusedArgs a) {
  constexpr int S = 32 / DH, HD = 8 * DH, KT = HD / 16, PC = HD / 8;
  constexpr int kTiles = 4 * S;                 // token tiles of 32
  constexpr int kPer = 2 * kTiles / 8;          // (token tile, output tile) pairs per wave
  __shared__ __attribute__((aligned(16))) bf16 os[S * 128 * HD];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = a.n, nqt = (n + 127) / 128, sbn = (a.depth + S - 1) / S, nk = a.np / 16;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = (int)(wg % nqt);
  const int64_t bs = wg / nqt;
  const int64_t b = bs / sbn;
  const int s0 = (int)(bs - b * sbn) * S, q0 = qt * 128;
  auto piece = [](int row, int p) { return row * HD + 8 * (p ^ (HD == 64 ? (row >> 1) & 7 : row & (PC - 1) & 15)); };

  const bf16* A = a.vt + (((b * 8 + wave) * sbn + s0 / S) * nk) * 512 + lane * 8;
  const bf16* B[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)  // query tiles past n re-read the last one
    B[t] = a.w + (((b * 8 + wave) * ((n + 31) / 32) + min(q0 / 32 + t, (n - 1) / 32)) * nk) * 512 + lane * 8;
  f32x16 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = zero16();
  bf16x8 fa[2][2], fb[2][2][4];
  auto fetch = [&](int k, bf16x8 (&x)[2], bf16x8 (&y)[2][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      x[u] = ld8(A + (k + u) * 512);
#pragma unroll
      for (int t = 0; t < 4; ++t) y[u][t] = ld8(B[t] + (k + u) * 512);
    }
  };
  auto multiply = [&](const bf16x8 (&x)[2], const bf16x8 (&y)[2][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = mfma32(x[u], y[u][t], acc[t]);
  };
  // the gate of this lane's averages, pieces 8 (2 k + g) .. of the tile's rows (s, d) at query li of
  // tile t (as acc_pieces leaves them): loaded first, so that they are there when the keys are done
  bf16x8 gv[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = 8 * (2 * k + g), s = s0 + r / DH, q = q0 + 32 * t + li;
      gv[t][k] = ld8(a.gate + ((b * a.depth + min(s, a.depth - 1)) * n + min(q, n - 1)) * HD + wave * DH + r % DH);
    }
  // np is a multiple of 64: steps in whole groups of 4
  fetch(0, fa[0], fb[0]);
#pragma unroll 1
  for (int k = 0; k < nk; k += 4) {
    fetch(k + 2, fa[1], fb[1]);
    multiply(fa[0], fb[0]);
    if (k + 4 < nk) fetch(k + 4, fa[0], fb[0]);
    multiply(fa[1], fb[1]);
  }

#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float y[2][8];
    acc_pieces(acc[t], y);  // y[k]: rows (s, d) 8 (2 k + g) .. + 7 of query li
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int r = 8 * (2 * k + g), s = r / DH, d = r % DH;
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (bf16)(y[k][e] * (float)gv[t][k][e]);
      *reinterpret_cast<bf16x8*>(&os[piece(s * 128 + 32 * t + li, (wave * DH + d) / 8)]) = o;
    }
  }
  __syncthreads();

  // this wave's token tiles and output tiles: pairs kPer wave .. + kPer - 1 of (tile, half)
  constexpr int kRt = kPer >= 2 ? kPer / 2 : 1;  // token tiles of this wave
  const int rt0 = kPer >= 2 ? wave * kRt : wave >> 1;
#pragma unroll
  for (int i = 0; i < kRt; ++i) {
    const int row = 32 * (rt0 + i) + li, sr = s0 + row / 128, qr = q0 + row % 128;
    const bool real = sr < a.depth && qr < n;
    const int64_t tok = (b * a.depth + min(sr, a.depth - 1)) * n + min(qr, n - 1);
    bf16x8 x[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) x[t] = ld8(&os[piece(row, KT * g + t)]);
#pragma unroll
    for (int u = 0; u < (kPer >= 2 ? 2 : 1); ++u) {
      const int ot = kPer >= 2 ? u : wave & 1;
      f32x16 y = zero16();
#pragma unroll
      for (int t = 0; t < KT; ++t) y = mfma32(ld8(a.wo + ((ot * KT + t) * 64 + lane) * 8), x[t], y);
      float p[2][8];
      acc_pieces(y, p);
      if (!real) continue;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int64_t at = tok * 64 + 32 * ot + 8 * (2 * k + g);
        bf16x8 o;
        if (a.res) {
          const bf16x8 r = ld8(a.res + at);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (bf16)(p[k][e] + (float)r[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (bf16)p[k][e];
        }
        *reinterpret_cast<bf16x8*>(a.out + at) = o;
      }
    }
  }
}

constexpr int kPT = 128;         // output tile: 128 (s, c) rows x 128 queries
constexpr int kPK = 32;          // keys per LDS stage
constexpr int kPKP = kPK + 8;    // LDS row stride (80 B: conflict-free 16-byte reads)
constexpr int kPOS = kPT + 4;    // epilogue fp32 row stride: 64 x kPOS floats fit in the operand stages
static_assert(64 * kPOS * 4 <= 4 * kPT * kPKP * 2, "epilogue staging exceeds the operand LDS");

// Per (batch, head): O[(s, c)][i] = sum_j v^T[(s, c)][j] w[i][j], an NT GEMM with both operands
// key-contiguous. grid: ceil(S dh / 128) * ceil(n / 128) * batch * heads workgroups (renumbered
// so that neighbours share an XCD's L2), block 256 = 2 x 2 waves of 64 x 64; operands staged
// through LDS 32 keys at a time (register prefetch two stages ahead, double buffer, one barrier per stage).
// v^T may be unwritten at keys >= n (RowGemmArgs): those operand entries are zeroed as they are staged.
// Epilogue: lane (li, g) holds query q0' + li and rows r = r0' + 8 v + 4 g + e, i.e.
// (s, c) = (r / dh, r % dh): four consecutive channels of one MSA row (dh % 4 == 0).
__global__ __launch_bounds__(256) void pwa_average(PwaAverageArgs a) {
  // operand stages xs[2] then ys[2]; after the key loop the epilogue reuses it as fp32 [64][kPOS]
  __shared__ __attribute__((aligned(16))) bf16 lds[4 * kPT * kPKP];
  bf16 (*xs)[kPT * kPKP] = reinterpret_cast<bf16 (*)[kPT * kPKP]>(lds);
  bf16 (*ys)[kPT * kPKP] = reinterpret_cast<bf16 (*)[kPT * kPKP]>(lds + 2 * kPT * kPKP);
  const int rows = a.depth * a.dh, n = a.n, np = a.np;
  const int rt = (rows + kPT - 1) / kPT, qt = (n + kPT - 1) / kPT;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t bh = wg / ((uint32_t)rt * qt);
  const int rem = (int)(wg - bh * rt * qt);
  const int r0 = (rem / qt) * kPT, q0 = (rem % qt) * kPT;
  const int64_t b = bh / a.heads;
  const int h = (int)(bh - b * a.heads);
  const bf16* X = a.vt + bh * rows * (int64_t)np;
  const bf16* Y = a.w + bh * n * (int64_t)np;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 31, g = lane >> 5;

  const bf16* xsrc[2];
  const bf16* ysrc[2];
  int soff[2], kcol[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = tid + 256 * u;
    const int row = c >> 2, kc = (c & 3) * 8;
    xsrc[u] = X + (int64_t)min(r0 + row, rows - 1) * np + kc;
    ysrc[u] = Y + (int64_t)min(q0 + row, n - 1) * np + kc;
    soff[u] = row * kPKP + kc;
    kcol[u] = kc;
  }
  // Two register sets carry the next two stages (stage s + 1 lands in LDS while stage s + 3 is
  // fetched), so a stage's global loads have two stages of MFMAs to land behind.
  bf16x8 rx0[2], ry0[2], rx1[2], ry1[2];
  auto gload = [&](bf16x8 (&rx)[2], bf16x8 (&ry)[2], int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      rx[u] = ld8(xsrc[u] + k0);
      ry[u] = ld8(ysrc[u] + k0);
    }
  };
  auto sstore = [&](bf16x8 (&rx)[2], const bf16x8 (&ry)[2], int k0, int buf) {
    if (k0 + kPK > n) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + kcol[u] + e >= n) rx[u][e] = (bf16)0.f;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      *reinterpret_cast<bf16x8*>(&xs[buf][soff[u]]) = rx[u];
      *reinterpret_cast<bf16x8*>(&ys[buf][soff[u]]) = ry[u];
    }
  };
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = zero16();
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < kPK; kk += 16) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) av[mi] = ld8(&xs[buf][(wm * 64 + mi * 32 + li) * kPKP + kk + 8 * g]);
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) bv[ni] = ld8(&ys[buf][(wn * 64 + ni * 32 + li) * kPKP + kk + 8 * g]);
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = mfma32(av[mi], bv[ni], acc[mi][ni]);
    }
  };

  // np is a multiple of 64: an even number (>= 2) of stages, taken two per iteration (buffers 0, 1)
  const int ns = np / kPK;
  gload(rx0, ry0, 0);
  sstore(rx0, ry0, 0, 0);
  gload(rx1, ry1, kPK);
  if (ns > 2) gload(rx0, ry0, 2 * kPK);
  __syncthreads();
#pragma unroll 1
  for (int st = 0; st < ns; st += 2) {
    compute(0);                   // stage st; rx1 holds stage st + 1, rx0 stage st + 2 (if any)
    sstore(rx1, ry1, (st + 1) * kPK, 1);
    if (st + 3 < ns) gload(rx1, ry1, (st + 3) * kPK);
    __syncthreads();
    compute(1);                   // stage st + 1
    if (st + 2 < ns) {
      sstore(rx0, ry0, (st + 2) * kPK, 0);
      if (st + 4 < ns) gload(rx0, ry0, (st + 4) * kPK);
    }
    __syncthreads();
  }

  const int hd = a.heads * a.dh;
  if (a.dh % 8 == 0) {
    // Staged: one half of the queries (ni) at a time goes through LDS as fp32 [query][row]; each
    // lane then gates and stores 8 consecutive rows of one query, i.e. 16 bytes of one MSA
    // row's head channels (dh % 8 == 0 keeps such a piece inside one MSA row).
    float* T = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      if (ni) __syncthreads();
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          f32x4 y;
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = acc[mi][ni][4 * v + e];
          *reinterpret_cast<f32x4*>(&T[(wn * 32 + li) * kPOS + wm * 64 + mi * 32 + 8 * v + 4 * g]) = y;
        }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int id = tid + 256 * u, ql = id >> 4, rl = (id & 15) * 8;
        const int q = q0 + (ql >> 5) * 64 + ni * 32 + (ql & 31), r = r0 + rl;
        if (q >= n || r >= rows) continue;
        const int s = r / a.dh, c = r - s * a.dh;
        const int64_t off = ((b * a.depth + s) * n + q) * hd + h * a.dh + c;
        const bf16x8 gv = ld8(a.gate + off);
        const f32x4 y0 = *reinterpret_cast<const f32x4*>(&T[ql * kPOS + rl]);
        const f32x4 y1 = *reinterpret_cast<const f32x4*>(&T[ql * kPOS + rl + 4]);
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = (bf16)(y0[e] * (float)gv[e]);
          o[4 + e] = (bf16)(y1[e] * (float)gv[4 + e]);
        }
        *reinterpret_cast<bf16x8*>(a.og + off) = o;
      }
    }
    return;
  }
#pragma unroll
  for (int ni = 0; ni < 2; ++ni) {
    const int q = q0 + wn * 64 + ni * 32 + li;
    if (q >= n) continue;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = r0 + wm * 64 + mi * 32 + 8 * v + 4 * g;
        if (r >= rows) continue;
        const int s = r / a.dh, c = r - s * a.dh;
        const int64_t off = ((b * a.depth + s) * n + q) * hd + h * a.dh + c;
        const bf16x4 gv = *reinterpret_cast<const bf16x4*>(a.gate + off);
        store4(a.og + off, acc[mi][ni][4 * v] * (float)gv[0], acc[mi][ni][4 * v + 1] * (float)gv[1],
               acc[mi][ni][4 * v + 2] * (float)gv[2], acc[mi][ni][4 * v + 3] * (float)gv[3]);
      }
  }
}

}  // namespace

void launch_pwa_softmax(const PwaSoftmaxArgs& a, hipStream_t stream) {
  const int64_t packs = a.frag ? (8 * a.hd + 255) / 256 : 0;
  pwa_softmax<<<dim3((unsigned)((a.rows + 3) / 4 + packs)), 256, 0, stream>>>(a);
}

void launch_pwa_fused(const PwaFusedArgs& a, hipStream_t stream) {
  const int S = 32 / a.dh;
  const int64_t blocks = (int64_t)((a.n + 127) / 128) * ((a.depth + S - 1) / S) * a.batch;
  if (a.dh == 8)
    pwa_fused<8><<<dim3((unsigned)blocks), 512, 0, stream>>>(a);
  else if (a.dh == 16)
    pwa_fused<16><<<dim3((unsigned)blocks), 512, 0, stream>>>(a);
  else
    pwa_fused<32><<<dim3((unsigned)blocks), 512, 0, stream>>>(a);
}

void launch_pwa_average(const PwaAverageArgs& a, hipStream_t stream) {
  const int64_t rt = ((int64_t)a.depth * a.dh + kPT - 1) / kPT, qt = (a.n + kPT - 1) / kPT;
  pwa_average<<<dim3((unsigned)(rt * qt * a.batch * a.heads)), 256, 0, stream>>>(a);
}

}  // namespace ffk
