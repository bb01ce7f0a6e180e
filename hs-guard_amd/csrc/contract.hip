// Unfused glue kernels with the reference engine's own kernel contracts, for callers that compose the step the way
// the reference's SlotStreamEngineV8 does (src/hs_guard/engine/slot_engine_v8.py:30-89): the variance of every
// RMSNorm arrives as an input (the caller's sq.mean(-1)), the rotary cos/sin arrive precomputed, SiLU-mul takes
// separate gate and up tensors, and q/k leave RMSNorm + RoPE in the grouped [N, Hkv, G*Lb, D] layout of the ring
// kernel. The streaming engine of this library runs the fused forms instead (glue.hip); both follow the same
// rounding points of src/hs_guard/engine/fused_kernels.py.
//
// Every kernel here is element-wise once the per-row variance is given, so each thread owns VEC consecutive
// elements of one row: the most of 8 (16-byte bf16 loads), 4 and 1 that the row width and every pointer and stride
// allow, so rows of any width and count work. Flat indices take 32 bits up to 2^31 elements (a cheap division), 64 beyond:
// SiLU-mul of 2^31 elements 1,345 us just below and above (4,350 with one element per thread).
// They move each byte once and are bound by that and, below ~10 MB, by the launch. At 1,473 tokens norm_rope over 16
// query and 4 key heads (two launches) takes 14.9 us, 38.5 with one element per thread; the others, cache-resident at
// that size, gain up to a fifth from 8 elements over 4 (rms_finish 4.2 -> 3.5 us) or stay (silu_mul 8.2).
#include <math.h>

#include <type_traits>

#include "hsg_common.h"

namespace hsg {
namespace {

constexpr int CT_THREADS = 256;

template <int VEC>
__device__ __forceinline__ void load_bf(const uint16_t* p, float* x) {
  if constexpr (VEC == 8) {
    load8_bf16(p, x);
  } else if constexpr (VEC == 4) {
    load4_bf16(p, x);
  } else {
    x[0] = bf2f(p[0]);
  }
}

template <int VEC>
__device__ __forceinline__ void store_bf(uint16_t* p, const float* x) {
  if constexpr (VEC == 8) {
    *reinterpret_cast<u32x4*>(p) = (u32x4){pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]),
                                           pack_bf16x2(x[6], x[7])};
  } else if constexpr (VEC == 4) {
    store4_bf16(p, x);
  } else {
    p[0] = f2bf(x[0]);
  }
}

template <int VEC>
__device__ __forceinline__ void store_f32(float* p, const float* x) {
  if constexpr (VEC == 1) {
    p[0] = x[0];
  } else {
#pragma unroll
    for (int e = 0; e < VEC; e += 4) *reinterpret_cast<f32x4_n*>(p + e) = (f32x4_n){x[e], x[e + 1], x[e + 2], x[e + 3]};
  }
}

// (at any 4-byte address: a weight may start anywhere in a buffer)
template <int VEC>
__device__ __forceinline__ void load_f32(const float* p, float* x) {
  if constexpr (VEC == 1) {
    x[0] = p[0];
  } else {
    typedef f32x4_n __attribute__((aligned(4))) f32x4_any;
#pragma unroll
    for (int e = 0; e < VEC; e += 4) {
      const f32x4_n v = *reinterpret_cast<const f32x4_any*>(p + e);
#pragma unroll
      for (int k = 0; k < 4; ++k) x[e + k] = v[k];
    }
  }
}

// the thread's first element, n when it has none
template <int VEC, typename I>
__device__ __forceinline__ I first_element(int64_t n) {
  const I i = ((I)blockIdx.x * CT_THREADS + threadIdx.x) * VEC;
  return i < (I)n ? i : (I)n;
}

// add_square (src/hs_guard/engine/fused_kernels.py:30-52): h = bf16(res + mix) with a plain fp32 add (no
// contraction), stored when mix is given; sq = h^2 in fp32 (of res when mix is NULL).
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void add_square_kernel(const uint16_t* res, const uint16_t* mix,
                                                                uint16_t* out, float* sq, int64_t n) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  float h[VEC];
  load_bf<VEC>(res + i, h);
  if (mix) {
    float m[VEC];
    load_bf<VEC>(mix + i, m);
#pragma unroll
    for (int e = 0; e < VEC; ++e) h[e] = rbf(__fadd_rn(h[e], m[e]));
    store_bf<VEC>(out + i, h);
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) h[e] = h[e] * h[e];
  store_f32<VEC>(sq + i, h);
}

// rms_finish (fused_kernels.py:56-72): out = bf16((x * rsqrt(var[row] + eps)) * w1[col]).
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void rms_finish_kernel(const uint16_t* x, const float* var, const float* w1,
                                                                float eps, uint16_t* out, int64_t n, int width) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  const I row = i / (I)width;
  const int col = (int)(i - row * (I)width);
  float h[VEC], wv[VEC];
  load_bf<VEC>(x + i, h);
  load_f32<VEC>(w1 + col, wv);
  const float r = rsqrtf(var[row] + eps);
#pragma unroll
  for (int e = 0; e < VEC; ++e) h[e] = (h[e] * r) * wv[e];
  store_bf<VEC>(out + i, h);
}

// silu_mul (fused_kernels.py:76-90): out = bf16(bf16(silu(gate)) * up) over two tensors of n elements.
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void silu_mul_pair_kernel(const uint16_t* gate, const uint16_t* up,
                                                                   uint16_t* out, int64_t n) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  float g[VEC], u[VEC];
  load_bf<VEC>(gate + i, g);
  load_bf<VEC>(up + i, u);
#pragma unroll
  for (int e = 0; e < VEC; ++e) g[e] = rbf(siluf_(g[e])) * u[e];
  store_bf<VEC>(out + i, g);
}

// gated_finish (fused_kernels.py:215-233): out = bf16(bf16(w[col] * bf16(x * rsqrt(var[row] + eps))) * silu(z)).
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void gated_finish_kernel(const uint16_t* x, const float* var,
                                                                  const uint16_t* w, const uint16_t* z, float eps,
                                                                  uint16_t* out, int64_t n, int width) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  const I row = i / (I)width;
  const int col = (int)(i - row * (I)width);
  float h[VEC], g[VEC], wv[VEC];
  load_bf<VEC>(x + i, h);
  load_bf<VEC>(z + i, g);
  load_bf<VEC>(w + col, wv);
  const float r = rsqrtf(var[row] + eps);
#pragma unroll
  for (int e = 0; e < VEC; ++e) h[e] = rbf(wv[e] * rbf(h[e] * r)) * siluf_(g[e]);
  store_bf<VEC>(out + i, h);
}

// square_rows (fused_kernels.py:237-249): sq[r, c] = x^2 of head r % heads of token r / heads, read from the
// strided projection rows; sq is [tokens * heads, dim] fp32.
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void square_rows_kernel(const uint16_t* src, float* sq, int heads,
                                                                 int64_t row_stride, int64_t head_stride, int dim,
                                                                 int64_t n) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  const I r = i / (I)dim;
  const int c = (int)(i - r * (I)dim);
  const int64_t token = r / (I)heads;
  const int j = (int)(r - token * heads);
  float x[VEC];
  load_bf<VEC>(src + token * row_stride + j * head_stride + c, x);
#pragma unroll
  for (int e = 0; e < VEC; ++e) x[e] = x[e] * x[e];
  store_f32<VEC>(sq + i, x);
}

// norm_rope (fused_kernels.py:252-284): per-head RMSNorm(1 + w) given var, then rotate-half RoPE on the first rot
// dims with the given bf16 cos/sin [tokens, rot]:
//   x = bf16((src[d] * rsqrt(var + eps)) * w1[d]), xp the same at d's partner (d +- rot/2),
//   out[d] = bf16(bf16(x * cos) + bf16(+-xp * sin)) for d < rot, bf16(x) beyond,
// written at out + n*out_n + (j / groups)*out_h + ((j % groups)*lb + l)*out_row + d for head j of token n*lb + l.
// A thread's VEC elements lie in one half of the rotary dims (or beyond them); their partners are a second (cached) load
// of the same row.
template <int VEC, typename I>
__global__ __launch_bounds__(CT_THREADS) void norm_rope_grouped_kernel(
    const uint16_t* src, const float* var, const float* w1, const uint16_t* cosv, const uint16_t* sinv, int rot,
    float eps, int heads, int lb, int groups, int64_t row_stride, int64_t head_stride, int dim, uint16_t* out,
    int64_t out_n, int64_t out_h, int64_t out_row, int64_t n) {
  const I i = first_element<VEC, I>(n);
  if (i == (I)n) return;
  const I r = i / (I)dim;
  const int d = (int)(i - r * (I)dim);
  const I token = r / (I)heads;
  const int j = (int)(r - token * (I)heads);
  const I nn = token / (I)lb;
  const int l = (int)(token - nn * (I)lb);
  const int half = rot / 2;
  const int partner = d < half ? d + half : (d < rot ? d - half : d);
  const float rr = rsqrtf(var[r] + eps);
  const uint16_t* base = src + (int64_t)token * row_stride + j * head_stride;
  float x[VEC], wv[VEC];
  load_bf<VEC>(base + d, x);
  load_f32<VEC>(w1 + d, wv);
#pragma unroll
  for (int e = 0; e < VEC; ++e) x[e] = rbf((x[e] * rr) * wv[e]);
  if (d < rot) {
    float xp[VEC], c[VEC], s[VEC];
    load_bf<VEC>(base + partner, xp);
    load_f32<VEC>(w1 + partner, wv);
    load_bf<VEC>(cosv + (int64_t)token * rot + d, c);
    load_bf<VEC>(sinv + (int64_t)token * rot + d, s);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      xp[e] = rbf((xp[e] * rr) * wv[e]);
      const float rh = d < half ? -xp[e] : xp[e];
      x[e] = __fadd_rn(rbf(x[e] * c[e]), rbf(rh * s[e]));
    }
  }
  store_bf<VEC>(out + (int64_t)nn * out_n + (j / groups) * out_h + ((int64_t)(j % groups) * lb + l) * out_row + d, x);
}

// Elements per thread (8 at most, or 4) of a call in rows of `width`, given its bf16 and fp32 pointers and its strides: bf16
// pieces of VEC elements and fp32 pieces of 4 are aligned to their size. 4 for the kernels that write fp32 squares: at 8 a
// wave's 16-byte stores leave gaps that its second store fills (add_square of 8,000 x 4,096 60.2 us against 56.5).
int vec_of(int most, int64_t width, std::initializer_list<const void*> bf, std::initializer_list<const void*> f32,
           std::initializer_list<int64_t> strides = {}) {
  for (const void* p : f32)
    if (p && !aligned(p, 16)) return 1;
  for (int vec : {8, 4}) {
    bool ok = width % vec == 0;
    for (const void* p : bf) ok = ok && (!p || aligned(p, 2 * vec));
    for (int64_t s : strides) ok = ok && s % vec == 0;
    if (ok && vec <= most) return vec;
  }
  return 1;
}

// Elements per thread and the type of flat indices: 32 bits (a cheap division) up to 2^31 elements
template <int VEC, typename I>
struct Form {
  static constexpr int vec = VEC;
  using index = I;
};

// launch(form, grid) for the chosen vector width over n elements
template <typename Launch>
int launch_vec(int vec, int64_t n, Launch launch) {
  const int64_t blocks = (n / vec + CT_THREADS - 1) / CT_THREADS;
  if (blocks >= (1 << 24)) return HSG_ERR_SHAPE;   // a launch holds less than 2^32 threads
  const dim3 grid((unsigned)blocks);
  const bool wide = n >= (1ll << 31);
  if (vec == 8) wide ? launch(Form<8, int64_t>{}, grid) : launch(Form<8, uint32_t>{}, grid);
  else if (vec == 4) wide ? launch(Form<4, int64_t>{}, grid) : launch(Form<4, uint32_t>{}, grid);
  else launch(Form<1, int64_t>{}, grid);
  return launch_status();
}

}  // namespace
}  // namespace hsg

using namespace hsg;

extern "C" int hsg_add_square(const void* residual, const void* mixed, void* out, float* sq, int64_t rows,
                              int32_t width, void* stream) {
  if (rows < 0 || width <= 0) return HSG_ERR_ARG;
  if (rows == 0) return HSG_OK;
  if (!residual || !sq || (mixed && !out)) return HSG_ERR_ARG;
  const int64_t n = rows * width;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* r = static_cast<const uint16_t*>(residual);
  const auto* m = static_cast<const uint16_t*>(mixed);
  auto* o = static_cast<uint16_t*>(out);
  return launch_vec(vec_of(4, width, {residual, mixed, out}, {sq}), n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((add_square_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s, r, m, o, sq, n);
  });
}

extern "C" int hsg_rms_finish(const void* x, const float* var, const float* w1, float eps, void* out, int64_t rows,
                              int32_t width, void* stream) {
  if (rows < 0 || width <= 0) return HSG_ERR_ARG;
  if (rows == 0) return HSG_OK;
  if (!x || !var || !w1 || !out) return HSG_ERR_ARG;
  const int64_t n = rows * width;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* xi = static_cast<const uint16_t*>(x);
  auto* o = static_cast<uint16_t*>(out);
  return launch_vec(vec_of(8, width, {x, out}, {}), n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((rms_finish_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s, xi, var, w1, eps, o, n, width);
  });
}

extern "C" int hsg_silu_mul_pair(const void* gate, const void* up, void* out, int64_t n, void* stream) {
  if (n < 0) return HSG_ERR_ARG;
  if (n == 0) return HSG_OK;
  if (!gate || !up || !out) return HSG_ERR_ARG;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* g = static_cast<const uint16_t*>(gate);
  const auto* u = static_cast<const uint16_t*>(up);
  auto* o = static_cast<uint16_t*>(out);
  return launch_vec(vec_of(8, n, {gate, up, out}, {}), n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((silu_mul_pair_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s, g, u, o, n);
  });
}

extern "C" int hsg_gated_finish(const void* x, const float* var, const void* weight, const void* z, float eps,
                                void* out, int64_t rows, int32_t width, void* stream) {
  if (rows < 0 || width <= 0) return HSG_ERR_ARG;
  if (rows == 0) return HSG_OK;
  if (!x || !var || !weight || !z || !out) return HSG_ERR_ARG;
  const int64_t n = rows * width;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* xi = static_cast<const uint16_t*>(x);
  const auto* w = static_cast<const uint16_t*>(weight);
  const auto* zi = static_cast<const uint16_t*>(z);
  auto* o = static_cast<uint16_t*>(out);
  return launch_vec(vec_of(8, width, {x, weight, z, out}, {}), n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((gated_finish_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s, xi, var, w, zi, eps, o, n, width);
  });
}

extern "C" int hsg_square_rows(const void* src, float* sq, int64_t tokens, int32_t heads, int64_t row_stride,
                               int64_t head_stride, int32_t dim, void* stream) {
  if (tokens < 0 || heads <= 0 || dim <= 0 || row_stride < 0 || head_stride < 0) return HSG_ERR_ARG;
  if (tokens == 0) return HSG_OK;
  if (!src || !sq) return HSG_ERR_ARG;
  const int64_t n = tokens * heads * dim;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const auto* x = static_cast<const uint16_t*>(src);
  return launch_vec(vec_of(4, dim, {src}, {sq}, {row_stride, head_stride}), n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((square_rows_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s, x, sq, heads, row_stride, head_stride, dim, n);
  });
}

extern "C" int hsg_norm_rope_grouped(const void* src, const float* var, const float* w1, const void* cos,
                                     const void* sin, int32_t rot, float eps, int32_t n_rows, int32_t lb,
                                     int32_t heads, int32_t groups, int64_t row_stride, int64_t head_stride,
                                     int32_t dim, void* out, int64_t out_n, int64_t out_h, int64_t out_row,
                                     void* stream) {
  if (n_rows < 0 || lb <= 0 || heads <= 0 || groups <= 0 || dim <= 0) return HSG_ERR_ARG;
  if (heads % groups || rot <= 0 || rot % 2 || rot > dim) return HSG_ERR_SHAPE;
  if (n_rows == 0) return HSG_OK;
  if (!src || !var || !w1 || !cos || !sin || !out) return HSG_ERR_ARG;
  const int64_t n = (int64_t)n_rows * lb * heads * dim;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return launch_vec(vec_of(8, dim, {src, cos, sin, out}, {w1}, {rot / 2, row_stride, head_stride, out_n, out_h, out_row}),
                    n, [&](auto form, dim3 grid) {
    using F = decltype(form);
    hipLaunchKernelGGL((norm_rope_grouped_kernel<F::vec, typename F::index>), grid, dim3(CT_THREADS), 0, s,
                       static_cast<const uint16_t*>(src), var, w1, static_cast<const uint16_t*>(cos),
                       static_cast<const uint16_t*>(sin), rot, eps, heads, lb, groups, row_stride, head_stride, dim,
                       static_cast<uint16_t*>(out), out_n, out_h, out_row, n);
  });
}
