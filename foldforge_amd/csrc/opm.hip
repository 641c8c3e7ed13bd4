// Outer product mean on gfx950 (the MSA stack's MSA-to-pair update).
//
// Equations: src/foldforge/models/checkpoints/legacy/primitives.py:40-136 (OuterProductMean)
// and legacy/reference/attention.py:57-74 (af3_outer_product_mean), in the engine's forms
// (src/foldforge/modules/engine/modules.py:184-210):
//   l[s, i] = m[s, i] (LN(msa[s, i]) W_l^T + b_l),  r[s, j] = m[s, j] (LN(msa[s, j]) W_r^T + b_r)
//   o[i, j, (c, e)] = sum_s l[s, i, c] r[s, j, e],   n[i, j] = sum_s m[s, i] m[s, j]
//   AF3: out = (o W_out^T + b) / (n + 1e-3); the clamp form divides by max(n, 1); the
//   normalize-before-projection form is (o / d) W_out^T + b.
// The C-ABI (api.hip) runs:
//   row_gemm<kEpiOpm, kXLn> (single.hip): LayerNorm + both projections, masked, stored with
//     the MSA rows contiguous (l^T, r^T [batch][n][32][sp], sp = depth padded to 64) and the
//     mask transposed
//   opm_prepare: n[i, j] as a 0/1 GEMM over the MSA rows (exact in fp32), and W_out rounded
//     to bf16 in the contraction's fragment order
//   opm_contract: per workgroup a tile of 8 x 8 tokens: the 256 x 256 outer-product block
//     summed over all MSA rows on MFMA, rounded to bf16 into LDS, projected to c_z on MFMA,
//     divided by the count, bias and residual added.
#include "ffk_device.h"
#include "ffk_kernels.h"

namespace ffk {

namespace {

constexpr int kOpmC = 32;                   // channels per side (d_hidden)
constexpr int kOpmT = 8;                    // tokens per tile side
constexpr int kOpmRows = kOpmT * kOpmC;     // (token, channel) rows of one operand tile
constexpr int kOpmBK = 64;                  // MSA rows per LDS stage (the MSA padding)
constexpr int kOpmStage = 2 * kOpmRows * kOpmBK;  // bf16 per stage: l rows, then r rows (64 KB)
constexpr int kOpmPairs = kOpmT * kOpmT;    // pairs per tile
constexpr int kOpmK2 = kOpmC * kOpmC;       // 1024: the projection's k
constexpr int kOpmCz = 128;                 // output channels
constexpr int kOpmRS = kOpmCz + 4;          // row stride (fp32) of the projection's partials
constexpr int kOpmSplit = 4;                // waves per 32 x 32 block of pair counts
static_assert(kOpmPairs * kOpmK2 <= 2 * kOpmStage, "outer products exceed the stage buffers");
static_assert(2 * kOpmPairs * kOpmRS * 4 <= 2 * kOpmStage * 2, "partials exceed the stage buffers");

// Tile order within a batch element: runs of 8 tile rows, walked column by column, so the 32
// neighbouring workgroups an XCD holds at once (consecutive ids after xcd_remap) cover 8 tile
// rows x 4 tile columns and share each operand block through that XCD's L2 (a row-major order
// gives them one tile row and 32 distinct column operands). A bijection of [0, nti * ntj).
__device__ __forceinline__ void grouped_tile(int t, int nti, int ntj, int& ti, int& tj) {
  constexpr int kRows = 8;
  const int per = kRows * ntj, first = (t / per) * kRows;
  const int rows = min(nti - first, kRows), u = t - (t / per) * per;
  ti = first + u % rows;
  tj = u / rows;
}

// k' order of the projection: piece q = k' / 8 holds the 8 products a lane (e, g) of the
// contraction has in accumulator registers 8 h .. 8 h + 7, q = 32 (2 g + h) + e, so 32 lanes
// write 32 consecutive 16-byte pieces. The weights are packed in the order of the projection's A
// fragments: wp[((f / 32) 64 + k' / 16) 64 + lane] is lane (f % 32, (k' / 8) % 2)'s 16 bytes.
__device__ __forceinline__ void opm_pack_one(const float* __restrict__ w, bf16* __restrict__ wp, int idx) {
  const int f = idx / kOpmK2, kp = idx % kOpmK2;
  const int q = kp >> 3, r = kp & 7, e = q & 31, gh = q >> 5;
  const int c = acc_row(8 * (gh & 1) + r, gh >> 1);
  const int lane = 32 * (q & 1) + (f & 31);
  wp[((((f >> 5) * (kOpmK2 / 16) + (q >> 1)) * 64 + lane) << 3) + r] =
      (bf16)w[(int64_t)f * kOpmK2 + c * kOpmC + e];
}

// The two small jobs before the contraction in one launch (each alone is a few microseconds of
// latency): workgroups below tiles * tiles * batch count the pairs, count[i][j] = sum_s mt[i][s]
// mt[j][s], one 32 x 32 block of pairs each with the MSA rows split over its 4 waves (0/1
// products: exact in fp32 in any order); the rest pack W_out.
__global__ __launch_bounds__(64 * kOpmSplit) void opm_prepare(OpmCountArgs a, const float* __restrict__ w,
                                                              bf16* __restrict__ wp) {
  const int tiles = (a.n + 31) / 32;
  const int64_t counts = (int64_t)tiles * tiles * a.batch;
  if (blockIdx.x >= counts) {
    const int idx = (int)(blockIdx.x - counts) * 64 * kOpmSplit + threadIdx.x;
    if (idx < kOpmCz * kOpmK2) opm_pack_one(w, wp, idx);
    return;
  }
  __shared__ float part[kOpmSplit][16][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int t = (int)(blockIdx.x % ((int64_t)tiles * tiles));
  const int i0 = (t / tiles) * 32, j0 = (t % tiles) * 32;
  const int64_t b = blockIdx.x / ((int64_t)tiles * tiles);
  const bf16* ar = a.mt + (b * a.n + min(i0 + li, a.n - 1)) * a.sp + 8 * g;
  const bf16* br = a.mt + (b * a.n + min(j0 + li, a.n - 1)) * a.sp + 8 * g;
  f32x16 acc = zero16();
#pragma unroll 4
  for (int k = 16 * wave; k < a.sp; k += 16 * kOpmSplit) acc = mfma32(ld8(ar + k), ld8(br + k), acc);
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
  __syncthreads();
  const int j = j0 + li;
  if (j >= a.n) return;
#pragma unroll
  for (int u = 0; u < 16 / kOpmSplit; ++u) {
    const int r = (16 / kOpmSplit) * wave + u;
    float c = 0.f;
#pragma unroll
    for (int s = 0; s < kOpmSplit; ++s) c += part[s][r][lane];
    const int i = i0 + acc_row(r, g);
    if (i < a.n) a.count[(b * a.n + i) * a.n + j] = c;
  }
}

// grid: ceil(n / 8)^2 * batch workgroups of 512 threads, one per CU (128 KB of LDS).
// Phase 1 (outer products): a 256 x 256 x depth product, rows (token i, c) x columns (token j,
// e), 8 waves of 128 x 64 (pair (i, j) is one 32 x 32 MFMA tile), so a wave reads 6 operand
// fragments for 8 MFMAs. Operand stages of 64 MSA rows (128-byte operand rows, 16-byte pieces
// XOR-swizzled by row pair) arrive by LDS DMA in two buffers, one stage ahead. Lane (li, g) ends
// with o[c = acc_row(r, g)][e = li] in acc[r].
// Phase 2 (projection): the 64 outer products go to LDS as bf16 rows of 1024 (order k' of
// opm_pack_one, pieces XOR-swizzled by pair % 16); wave (kh, fw) multiplies 32 output channels x
// all 64 pairs over half of k', so the weights come from L2 once per workgroup, fetched 8
// fragments ahead (the first behind phase 1). Phase 3: the two halves are
// joined through LDS in fp32 and leave as whole 256-byte rows.
// Measured at 512 MSA rows x 384 tokens (193 GFLOP): 183 to 186 us, 1.05 PFLOP/s, against 314 us with
// register-staged 32-row stages (an L2 latency exposed per stage) and the weights read twice per
// workgroup. Bound by the products (matrix cores busy 42% of the time) and by phases 2 and 3, which
// nothing overlaps: 128 KB of LDS leave one workgroup per CU.
__global__ __launch_bounds__(512, 2) void opm_contract(OpmContractArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 smem[2 * kOpmStage];  // 128 KB
  const int n = a.n;
  const int64_t sp = a.sp;
  const int nt = (n + kOpmT - 1) / kOpmT;
  const uint32_t t = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t b = t / ((uint32_t)nt * nt);
  int ti, tj;
  grouped_tile((int)(t - b * nt * nt), nt, nt, ti, tj);
  const int i0 = ti * kOpmT, j0 = tj * kOpmT;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // This wave's 8 one-KB pieces of a stage (pieces 0-31: l rows, 32-63: r rows; 8 rows of 128
  // bytes, all of one token: tokens past the end re-read the last one). Slot c of row r sits at
  // slot c ^ ((r >> 1) & 7). The row offset is 64 bits wide: a row is depth long.
  const int64_t row0 = (int64_t)(lane >> 3) * sp;
  const bf16* side = wave < 4 ? a.lt : a.rt;
  const int tok0 = wave < 4 ? i0 : j0;
  const bf16* src[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int piece = 8 * (wave & 3) + u;  // of this side
    const int tok = min(tok0 + (piece >> 2), n - 1);
    const int c = (lane & 7) ^ ((4 * (u & 1) + (lane >> 4)) & 7);
    src[u] = side + ((b * n + tok) * kOpmC + 8 * (piece & 3)) * sp + row0 + 8 * c;
  }
  auto stage_dma = [&](int s) {
    const uint32_t base = lds_addr(&smem[(s & 1) * kOpmStage]) + 8192 * wave;
#pragma unroll
    for (int u = 0; u < 8; ++u) dma16_at(src[u] + s * (int64_t)kOpmBK, base + 1024 * u);
  };

  const int wm = wave >> 2, wn = wave & 3;  // rows 128 wm .., columns 64 wn ..
  f32x16 acc[4][2];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = zero16();

  const int kh = wave >> 2, fw = wave & 3;  // phase 2: k' half, channels 32 fw ..
  const bf16* wfrag = a.wp + ((int64_t)(fw * (kOpmK2 / 16) + 32 * kh) * 64 + lane) * 8;
  constexpr int kWB = 8;  // weight fragments per batch
  bf16x8 wv[2][kWB];
  auto wload = [&](bf16x8 (&w)[kWB], int batch) {
#pragma unroll
    for (int s = 0; s < kWB; ++s) w[s] = ld8(wfrag + (batch * kWB + s) * 512);
  };

  const int nk = (int)(sp / kOpmBK);
  stage_dma(0);
#pragma unroll 1
  for (int s = 0; s < nk; ++s) {
    wait_vm_lds<0>();  // this wave's pieces of stage s landed
    __syncthreads();   // everyone's; the other buffer's readers are done
    if (s + 1 < nk) stage_dma(s + 1);
    const bf16* xs = &smem[(s & 1) * kOpmStage];
    const bf16* ys = xs + kOpmRows * kOpmBK;
#pragma unroll
    for (int kk = 0; kk < kOpmBK / 16; ++kk) {
      bf16x8 av[4], bv[2];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        const int r = 128 * wm + 32 * mi + li;
        av[mi] = ld8(&xs[r * kOpmBK + 8 * ((2 * kk + g) ^ ((r >> 1) & 7))]);
      }
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const int r = 64 * wn + 32 * ni + li;
        bv[ni] = ld8(&ys[r * kOpmBK + 8 * ((2 * kk + g) ^ ((r >> 1) & 7))]);
      }
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = mfma32(av[mi], bv[ni], acc[mi][ni]);
    }
  }
  wload(wv[0], 0);
  __syncthreads();  // every wave's last fragment reads are done: the buffers take the products
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      const int p = (4 * wm + mi) * kOpmT + 2 * wn + ni;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8 o;
#pragma unroll
        for (int r = 0; r < 8; ++r) o[r] = (bf16)acc[mi][ni][8 * h + r];
        const int q = 32 * (2 * g + h) + li;
        *reinterpret_cast<bf16x8*>(&smem[p * kOpmK2 + 8 * (q ^ (p & 15))]) = o;
      }
    }

  // phase 3's pair of this thread (8 threads per pair, channels 8 c8 .. and 64 + 8 c8 ..): its
  // count and residual travel during the projection
  const int pp = tid >> 3, c8 = tid & 7;
  const int i = i0 + pp / kOpmT, j = j0 + pp % kOpmT;
  const bool real = i < n && j < n;
  const int64_t pij = (b * n + min(i, n - 1)) * n + min(j, n - 1);
  const float cnt = a.count[pij];
  bf16x8 res[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (a.res) res[h] = ld8(a.res + pij * kOpmCz + 64 * h + 8 * c8);
  __syncthreads();

  f32x16 acc2[2];
  acc2[0] = zero16();
  acc2[1] = zero16();
#pragma unroll
  for (int batch = 0; batch < 32 / kWB; ++batch) {
    if (batch + 1 < 32 / kWB) wload(wv[(batch + 1) & 1], batch + 1);
#pragma unroll
    for (int s = 0; s < kWB; ++s) {
      const int q = 2 * (32 * kh + batch * kWB + s) + g;
      const int off = li * kOpmK2 + 8 * (q ^ (li & 15));
#pragma unroll
      for (int h = 0; h < 2; ++h)
        acc2[h] = mfma32(wv[batch & 1][s], ld8(&smem[off + 32 * h * kOpmK2]), acc2[h]);
    }
  }
  __syncthreads();  // the products are consumed: the buffers take the partial sums
  float* red = reinterpret_cast<float*>(smem);  // [k' half][pair][kOpmRS]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const f32x4 y = {acc2[h][4 * v], acc2[h][4 * v + 1], acc2[h][4 * v + 2], acc2[h][4 * v + 3]};
      *reinterpret_cast<f32x4*>(red + (kOpmPairs * kh + 32 * h + li) * kOpmRS + 32 * fw + 8 * v + 4 * g) = y;
    }
  __syncthreads();
  if (!real) return;
  const float d = a.count_offset >= 0.f ? cnt + a.count_offset : fmaxf(cnt, 1.f);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int f = 64 * h + 8 * c8;
    bf16x8 o;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const f32x4 y0 = *reinterpret_cast<const f32x4*>(red + pp * kOpmRS + f + 4 * v);
      const f32x4 y1 = *reinterpret_cast<const f32x4*>(red + (kOpmPairs + pp) * kOpmRS + f + 4 * v);
      const f32x4 bias = *reinterpret_cast<const f32x4*>(a.bias + f + 4 * v);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = y0[e] + y1[e];
        float x = a.normalize_before_proj ? y / d + bias[e] : (y + bias[e]) / d;
        if (a.res) x += (float)res[h][4 * v + e];
        o[4 * v + e] = (bf16)x;
      }
    }
    *reinterpret_cast<bf16x8*>(a.out + pij * kOpmCz + f) = o;
  }
}

// ---------------------------------------------------------------------------- grouped (Chai-1)
// Chai-1's grouped outer product mean (legacy/primitives.py:122-136, 8 groups of 8 channels a
// side; src/foldforge/modules/dense/spec.py:687-688): products only within each group, summed
// over the MSA rows and divided by nothing,
//   p[i, j, (g, k, l)] = sum_s l[s, i, 8 g + k] r[s, j, 8 g + l]            (512 per pair)
//   out[i, j] = LN_0.1(p[i, j]) W_out^T + b_out                 (product norm over the 512)
// grid: ceil(n / 4) * ceil(n / 8) * batch workgroups of 512 threads, one tile of 4 x 8 tokens.
// Phase 1: per group the products are one dense product, rows (token i, k) x columns (token j,
// l) over the MSA rows, so wave w takes group w: two 32 x 32 MFMA tiles, rows (i = row / 8,
// k = row % 8) for the tile's 4 tokens i, columns (j = 4 h + li / 8, l = li % 8) for h = 0, 1.
// Lane (li, g) holds row acc_row(r, g) of column li in acc[h][r]; the products go to LDS in
// fp32 in the (g, k, l) order. In the operand stages token t's 64 rows (8 groups x 8) start
// 128 t bytes later than unpadded, so the 16 lanes of a read (two neighbouring tokens' 8 rows of
// one group, 80-byte rows) cover all 64 banks.
// Phase 2: one wave per pair normalises the 512 products (two passes over 8 per lane), rounds
// them to bf16 rows; phase 3: the c_z / 32 output tiles (each over 32 pairs, k = 512; at c_z
// 128 the k range is split over two waves and summed through LDS), bias and residual added.
constexpr int kOpmKC = 32;                    // MSA rows per LDS stage (the MSA padding is 64)
constexpr int kOpmKS = kOpmKC + 8;            // LDS row stride of a stage (conflict-free reads)
constexpr int kOpmCPR = kOpmKC / 8;           // 16-byte chunks per operand row and stage
constexpr int kOgC = 64;                      // channels per side (8 groups x 8)
constexpr int kOgTI = 4, kOgTJ = 8;           // tokens per tile side
constexpr int kOgPairs = kOgTI * kOgTJ;       // 32
constexpr int kOgN = 512;                     // products per pair
constexpr int kOgNS = kOgN + 8;               // LDS row stride of a normalised pair (bf16)
constexpr int kOgXRows = kOgTI * kOgC, kOgYRows = kOgTJ * kOgC;
constexpr int kOgXPT = kOgXRows * kOpmCPR / 512, kOgYPT = kOgYRows * kOpmCPR / 512;
constexpr int kOgTokPad = 64;                 // stage rows of token t shifted by t x 128 bytes (bf16 units)
constexpr int kOgXB = kOgXRows * kOpmKS + kOgTI * kOgTokPad;  // one stage of each operand
constexpr int kOgYB = kOgYRows * kOpmKS + kOgTJ * kOgTokPad;
constexpr size_t kOgStageBytes = (size_t)2 * (kOgXB + kOgYB) * sizeof(bf16);
constexpr size_t kOgProdBytes = (size_t)kOgPairs * kOgN * sizeof(float);
constexpr size_t kOgNormBytes = (size_t)kOgPairs * kOgNS * sizeof(bf16);
constexpr size_t kOgLds = kOgStageBytes > kOgProdBytes + kOgNormBytes ? kOgStageBytes : kOgProdBytes + kOgNormBytes;

template <int CZ>
__global__ __launch_bounds__(512) void opm_contract_grouped(OpmGroupedArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  bf16* xs = reinterpret_cast<bf16*>(smem);  // [2][kOgXB]: rows (token, channel) x kOpmKS
  bf16* ys = xs + 2 * kOgXB;                 // [2][kOgYB]
  float* prod = reinterpret_cast<float*>(smem);                     // [32][512], after phase 1
  bf16* nrm = reinterpret_cast<bf16*>(smem + kOgProdBytes);         // [32][kOgNS]
  float* red = reinterpret_cast<float*>(smem);                      // phase 3 (c_z 128) partials
  const int n = a.n, sp = a.sp;
  const int nti = (n + kOgTI - 1) / kOgTI, ntj = (n + kOgTJ - 1) / kOgTJ;
  const uint32_t t = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t b = t / ((uint32_t)nti * ntj);
  int ti, tj;
  grouped_tile((int)(t - b * nti * ntj), nti, ntj, ti, tj);
  const int i0 = ti * kOgTI, j0 = tj * kOgTJ;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 31, g = lane >> 5;

  // global -> LDS: a stage is the operand rows (token, channel) x kOpmKC MSA rows, 8 bf16 a chunk
  const bf16* xsrc[kOgXPT];
  const bf16* ysrc[kOgYPT];
  int xoff[kOgXPT], yoff[kOgYPT];
#pragma unroll
  for (int u = 0; u < kOgXPT; ++u) {
    const int c = tid + 512 * u, row = c / kOpmCPR, kc = (c % kOpmCPR) * 8;
    const int tok = min(i0 + row / kOgC, n - 1);
    xsrc[u] = a.lt + ((b * n + tok) * kOgC + row % kOgC) * sp + kc;
    xoff[u] = row * kOpmKS + kc + (row / kOgC) * kOgTokPad;
  }
#pragma unroll
  for (int u = 0; u < kOgYPT; ++u) {
    const int c = tid + 512 * u, row = c / kOpmCPR, kc = (c % kOpmCPR) * 8;
    const int tok = min(j0 + row / kOgC, n - 1);
    ysrc[u] = a.rt + ((b * n + tok) * kOgC + row % kOgC) * sp + kc;
    yoff[u] = row * kOpmKS + kc + (row / kOgC) * kOgTokPad;
  }
  bf16x8 rx[kOgXPT], ry[kOgYPT];
  auto gload = [&](int k0) {
#pragma unroll
    for (int u = 0; u < kOgXPT; ++u) rx[u] = ld8(xsrc[u] + k0);
#pragma unroll
    for (int u = 0; u < kOgYPT; ++u) ry[u] = ld8(ysrc[u] + k0);
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int u = 0; u < kOgXPT; ++u)
      *reinterpret_cast<bf16x8*>(xs + buf * kOgXB + xoff[u]) = rx[u];
#pragma unroll
    for (int u = 0; u < kOgYPT; ++u)
      *reinterpret_cast<bf16x8*>(ys + buf * kOgYB + yoff[u]) = ry[u];
  };

  // this lane's operand rows: token li / 8 (i; j within each half), channel 8 w + li % 8
  const int ti8 = li >> 3, ch = 8 * wave + (li & 7);
  const int arow = (ti8 * kOgC + ch) * kOpmKS + ti8 * kOgTokPad + 8 * g;
  int brow[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) brow[h] = ((4 * h + ti8) * kOgC + ch) * kOpmKS + (4 * h + ti8) * kOgTokPad + 8 * g;
  f32x16 acc[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) acc[h] = zero16();

  gload(0);
  sstore(0);
  __syncthreads();
  int buf = 0;
#pragma unroll 1
  for (int k0 = 0; k0 < sp; k0 += kOpmKC) {
    const bool more = k0 + kOpmKC < sp;
    if (more) gload(k0 + kOpmKC);
    const bf16* xb = xs + buf * kOgXB;
    const bf16* yb = ys + buf * kOgYB;
#pragma unroll
    for (int kk = 0; kk < kOpmKC; kk += 16) {
      const bf16x8 av = ld8(xb + arow + kk);
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[h] = mfma32(av, ld8(yb + brow[h] + kk), acc[h]);
    }
    if (more) sstore(buf ^ 1);
    __syncthreads();  // also ends every read of the stages before the products land
    buf ^= 1;
  }

  // the in-group products, fp32, at p (g, k, l) order: acc[h][r] is row acc_row(r, g) =
  // (i = r / 4, k = 4 g + r % 4) of column li = (j = 4 h + li / 8, l = li % 8), group w
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int pair = (r >> 2) * kOgTJ + 4 * h + ti8;
      prod[pair * kOgN + wave * 64 + (4 * g + (r & 3)) * 8 + (li & 7)] = acc[h][r];
    }
  __syncthreads();

  // product norm: wave w normalises pairs 4 w .. 4 w + 3, lane L the products 8 L .. 8 L + 7
  {
    float nw[8], nb[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      nw[e] = a.norm_w[8 * lane + e];
      nb[e] = a.norm_b[8 * lane + e];
    }
#pragma unroll 1
    for (int u = 0; u < 4; ++u) {
      const int pair = 4 * wave + u;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(prod + pair * kOgN + 8 * lane);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(prod + pair * kOgN + 8 * lane + 4);
      float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      float s1 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s1 += x[e];
      const float mean = wave_sum(s1) * (1.f / kOgN);
      float s2 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] -= mean;
        s2 += x[e] * x[e];
      }
      const float rstd = __builtin_amdgcn_rsqf(wave_sum(s2) * (1.f / kOgN) + a.norm_eps);
      bf16x8 y;
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (bf16)(x[e] * rstd * nw[e] + nb[e]);
      *reinterpret_cast<bf16x8*>(nrm + pair * kOgNS + 8 * lane) = y;
    }
  }
  __syncthreads();

  // output projection: D[f][pair] = W_out[f] . nrm[pair] (A = bf16 weight rows, B = pair rows)
  constexpr int NT = CZ / 32;             // output tiles
  constexpr int KSPLIT = 8 / NT;          // waves per tile (k split)
  constexpr int KW = kOgN / KSPLIT;       // k per wave
  const int ft = wave % NT, kpart = wave / NT;
  const bf16* wrow = a.wp + (int64_t)(32 * ft + li) * kOgN + kpart * KW + 8 * g;
  const bf16* orow = nrm + li * kOgNS + kpart * KW + 8 * g;
  f32x16 acc2 = zero16();
#pragma unroll 4
  for (int k = 0; k < KW; k += 16) acc2 = mfma32(ld8(wrow + k), ld8(orow + k), acc2);
  if (KSPLIT > 1) {
    // (the product rows are no longer read: the partials of waves NT .. 7 go where they were)
    if (kpart > 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) red[((kpart - 1) * NT * 64 + ft * 64 + lane) * 16 + r] = acc2[r];
    }
    __syncthreads();
    if (kpart != 0) return;
#pragma unroll
    for (int w = 1; w < KSPLIT; ++w)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc2[r] += red[((w - 1) * NT * 64 + ft * 64 + lane) * 16 + r];
  }
  const int pair = li;
  const int i = i0 + pair / kOgTJ, j = j0 + pair % kOgTJ;
  if (i >= n || j >= n) return;
  const int64_t off = ((b * n + i) * n + j) * CZ;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int f = 32 * ft + 8 * v + 4 * g;
    const f32x4 bias = *reinterpret_cast<const f32x4*>(a.bias + f);
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = acc2[4 * v + e] + bias[e];
    if (a.res) {
      const bf16x4 r = *reinterpret_cast<const bf16x4*>(a.res + off + f);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += (float)r[e];
    }
    store4(a.out + off + f, y[0], y[1], y[2], y[3]);
  }
}
}  // namespace

void launch_opm_prepare(const OpmCountArgs& a, const float* w, bf16* wp, hipStream_t stream) {
  const int64_t t = (a.n + 31) / 32, threads = 64 * kOpmSplit;
  const int64_t blocks = t * t * a.batch + (kOpmCz * kOpmK2 + threads - 1) / threads;
  opm_prepare<<<dim3((unsigned)blocks), (unsigned)threads, 0, stream>>>(a, w, wp);
}

void launch_opm_contract(const OpmContractArgs& a, hipStream_t stream) {
  const int64_t nt = (a.n + kOpmT - 1) / kOpmT;
  opm_contract<<<dim3((unsigned)(nt * nt * a.batch)), 512, 0, stream>>>(a);
}

void launch_opm_contract_grouped(const OpmGroupedArgs& a, hipStream_t stream) {
  const int64_t tiles = (int64_t)((a.n + kOgTI - 1) / kOgTI) * ((a.n + kOgTJ - 1) / kOgTJ) * a.batch;
  auto kernel = a.cz == 256 ? opm_contract_grouped<256> : opm_contract_grouped<128>;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)kOgLds);
  kernel<<<dim3((unsigned)tiles), 512, kOgLds, stream>>>(a);
}

}  // namespace ffk
