// LayerNorm over the last axis on gfx950 (fp32 statistics, fp32 affine, input dtype kept).
//
// Reference: the engine LayerNorm (src/foldforge/modules/engine/modules.py:230-238) and the
// torch.nn.LayerNorm of the legacy graph (legacy/attention.py:90). HBM-bound. A row of
// L * P 16-byte pieces is held by L lanes (P pieces each), so every load and store is 16 bytes
// per lane and contiguous over the row's lanes; a lane takes 2 rows (one of three pieces; 512 / L
// or 256 / L rows per 256-thread workgroup, up to 32 workgroups per CU, larger inputs loop), fetches the
// workgroup's next rows while it normalises the current ones (two register buffers used
// alternately), keeps each row in registers between the two statistics passes (exact two-pass
// variance) and writes with non-temporal stores (128 bf16 channels at N = 512: 22.5 -> 19.6 us
// against 8 rows per lane, four persistent workgroups per CU and regular stores). Before, only
// that width had this form; the others ran one wave per row with 2-byte loads and three passes
// over the row (196608 rows of 64 bf16: 54.4 -> 6.3 us, 8.0 TB/s with the last-level cache).
#include <algorithm>

#include "ffk_device.h"
#include "ffk_kernels.h"

namespace ffk {

namespace {

// Rows a lane takes at once: two, or one where a row is three pieces a lane (with two, the row
// buffers and the affine took 159 VGPRs).
constexpr int ln_rows_per_lane(int P) { return P == 1 ? 2 : 1; }

// 16 bytes of T
template <typename T>
struct LnPiece {
  static constexpr int kN = 16 / sizeof(T);
  typedef T vec __attribute__((__vector_size__(16)));
};

// Sum over aligned groups of L lanes (every lane of the group gets the total).
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v = sum4(v);
  v += dpp_f<kDppHalfMirror>(v);
  if constexpr (L >= 16) v += dpp_f<kDppMirror>(v);
  if constexpr (L >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if constexpr (L >= 64) v = pair_sum(v);
  return v;
}

// Rows of exactly L * P pieces; x and y 16-byte aligned. grid min(ceil(rows / (R 256 / L)),
// 32 per CU); block 256.
template <typename T, int L, int P>
__global__ __launch_bounds__(256) void layer_norm_vec(const T* __restrict__ x, const float* __restrict__ w,
                                                      const float* __restrict__ b, T* __restrict__ y,
                                                      int64_t rows, float eps) {
  using V = typename LnPiece<T>::vec;
  constexpr int VE = LnPiece<T>::kN, C = L * P * VE, R = ln_rows_per_lane(P), G = 256 / L;
  const int sub = threadIdx.x % L;  // this lane's pieces: sub + L p
  auto load = [&](V (&v)[R][P], int64_t row0) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < R; ++it) {
      const int64_t row = row0 + G * it;
      if (row < rows) {
#pragma unroll
        for (int p = 0; p < P; ++p) v[it][p] = *reinterpret_cast<const V*>(x + row * C + VE * (sub + L * p));
      }
    }
  };
  float wv[P * VE], bv[P * VE];
  auto compute = [&](const V (&v)[R][P], int64_t row0) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < R; ++it) {
      const int64_t row = row0 + G * it;
      float xv[P * VE];
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < P * VE; ++i) {
        xv[i] = row < rows ? (float)v[it][i / VE][i % VE] : 0.f;
        s += xv[i];
      }
      const float mean = lanes_sum<L>(s) * (1.f / C);
      float q = 0.f;
#pragma unroll
      for (int i = 0; i < P * VE; ++i) {
        xv[i] -= mean;
        q += xv[i] * xv[i];
      }
      const float var = lanes_sum<L>(q) * (1.f / C) + eps;
      // one hardware reciprocal square root (1 ulp) where the output is rounded to bf16
      const float rstd = sizeof(T) == 2 ? __builtin_amdgcn_rsqf(var) : 1.f / sqrtf(var);
      if (row < rows) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
          V o;
#pragma unroll
          for (int e = 0; e < VE; ++e) o[e] = (T)(xv[p * VE + e] * rstd * wv[p * VE + e] + bv[p * VE + e]);
          __builtin_nontemporal_store(o, reinterpret_cast<V*>(y + row * C + VE * (sub + L * p)));
        }
      }
    }
  };
  const int64_t step = (int64_t)gridDim.x * G * R;
  const int lead = threadIdx.x / L;
  int64_t row0 = (int64_t)blockIdx.x * G * R + lead;
  V va[R][P], vb[R][P];
  load(va, row0);
  // one uniform branch per pointer (a per-element select compiles to a branch per load)
  if (w != nullptr) {
#pragma unroll
    for (int i = 0; i < P * VE; ++i) wv[i] = w[VE * (sub + L * (i / VE)) + i % VE];
  } else {
#pragma unroll
    for (int i = 0; i < P * VE; ++i) wv[i] = 1.f;
  }
  if (b != nullptr) {
#pragma unroll
    for (int i = 0; i < P * VE; ++i) bv[i] = b[VE * (sub + L * (i / VE)) + i % VE];
  } else {
#pragma unroll
    for (int i = 0; i < P * VE; ++i) bv[i] = 0.f;
  }
  // row0 - lead is the workgroup's first row: the loop condition is uniform
  while (row0 - lead < rows) {
    load(vb, row0 + step);
    compute(va, row0);
    row0 += step;
    if (row0 - lead >= rows) break;
    load(va, row0 + step);
    compute(vb, row0);
    row0 += step;
  }
}

// Any width and alignment, bf16 or fp32: one wave per row. grid min(ceil(rows / 4), 65535 * 4); block 256.
template <typename T>
__global__ __launch_bounds__(256) void layer_norm_rows(const T* __restrict__ x,
                                                       const float* __restrict__ w,
                                                       const float* __restrict__ b,
                                                       T* __restrict__ y, int64_t rows, int cols,
                                                       float eps) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float inv = 1.f / (float)cols;
  for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < rows; row += (int64_t)gridDim.x * 4) {
    const T* xr = x + row * cols;
    float s = 0.f;
    for (int c = lane; c < cols; c += 64) s += (float)xr[c];
    const float mean = wave_sum(s) * inv;
    float q = 0.f;
    for (int c = lane; c < cols; c += 64) {
      const float d = (float)xr[c] - mean;
      q += d * d;
    }
    const float rstd = 1.f / sqrtf(wave_sum(q) * inv + eps);
    T* yr = y + row * cols;
    for (int c = lane; c < cols; c += 64) {
      float v = ((float)xr[c] - mean) * rstd;
      if (w) v *= w[c];
      if (b) v += b[c];
      yr[c] = (T)v;
    }
  }
}

template <typename T, int L, int P>
void launch_vec(const T* x, const float* w, const float* b, T* y, int64_t rows, float eps, hipStream_t stream) {
  constexpr int per_block = 256 / L * ln_rows_per_lane(P);
  const int64_t blocks = std::min<int64_t>((rows + per_block - 1) / per_block, (int64_t)cu_count() * 32);
  layer_norm_vec<T, L, P><<<dim3((unsigned)blocks), 256, 0, stream>>>(x, w, b, y, rows, eps);
}

template <typename T>
void launch_typed(const T* x, const float* w, const float* b, T* y, int64_t rows, int cols, float eps,
                  hipStream_t stream) {
  // The vector kernel takes the widths whose pieces split evenly over 8 to 64 lanes with one or
  // three pieces a lane (the stacks' 64 to 768 channels) and 16-byte aligned tensors (the affine is
  // read a value at a time: any alignment); other widths, and views at odd offsets, keep the row
  // kernel.
  const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (cols % LnPiece<T>::kN == 0 && aligned(x) && aligned(y)) {
    switch (cols / LnPiece<T>::kN) {
      case 8: return launch_vec<T, 8, 1>(x, w, b, y, rows, eps, stream);
      case 16: return launch_vec<T, 16, 1>(x, w, b, y, rows, eps, stream);
      case 32: return launch_vec<T, 32, 1>(x, w, b, y, rows, eps, stream);
      case 48: return launch_vec<T, 16, 3>(x, w, b, y, rows, eps, stream);
      case 64: return launch_vec<T, 64, 1>(x, w, b, y, rows, eps, stream);
      case 96: return launch_vec<T, 32, 3>(x, w, b, y, rows, eps, stream);
      case 192: return launch_vec<T, 64, 3>(x, w, b, y, rows, eps, stream);
      default: break;
    }
  }
  const int64_t blocks = std::min<int64_t>((rows + 3) / 4, 65535 * 4);
  layer_norm_rows<T><<<dim3((unsigned)blocks), 256, 0, stream>>>(x, w, b, y, rows, cols, eps);
}

}  // namespace

void launch_layer_norm(const void* x, const float* w, const float* b, void* y, int64_t rows,
                       int cols, float eps, int dtype, hipStream_t stream) {
  if (dtype == 0)
    launch_typed(static_cast<const bf16*>(x), w, b, static_cast<bf16*>(y), rows, cols, eps, stream);
  else
    launch_typed(static_cast<const float*>(x), w, b, static_cast<float*>(y), rows, cols, eps, stream);
}

}  // namespace ffk
