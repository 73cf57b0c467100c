// The token-local steps between the products of a feedback layer
// (reference blocks/decoder_layer.py:51-72, layers/white_matter.py:105-118):
// residual add and RMS norm, query norm and RoPE, and the gated activation,
// each one kernel where the torch operations are three to twelve. A layer of
// the cyclic pass runs on a group's few hundred tokens, so its time was the
// launches: 37 a layer, about 380 us of host for some 130 us of GPU. Here a
// layer is five products, the attention and four of these kernels (small
// products take the norm, RoPE and activation into themselves, linear.hip). Each
// reads its operands once; at 1,024 tokens of width 512 they are bound by the
// launch and one round trip to memory (4 us each). A prefill of 8 x 1,024 tokens
// through four layers (8 groups, 2 passes): 28 -> 18 ms, with linear.hip 11.3
// and the pool projections there 9.7-10.4.
//
// Arithmetic and roundings are the torch operations': norms and the residual
// stream in fp32, results rounded to bf16 where the model casts.
#include "wmx_kernels.h"

namespace wmx {

namespace {

// One wave per row; lane l holds elements 512 c + 8 l + [0, 8) for c < CH.
// x' = x + delta (delta optional) to `out` (optional), and
// h = bf16(x' * rsqrt(mean(x'^2) + eps) * w) (weight optional).
template <int CH>
__global__ __launch_bounds__(256) void residual_norm_kernel(const wmx_residual_norm_args a) {
#pragma clang fp contract(off)
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= a.rows) return;  // wave-uniform
  const int lane = threadIdx.x & 63;
  float x[CH][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int d0 = 512 * c + 8 * lane;
    if (d0 >= a.hidden) continue;
    load8(a.x, r * a.x_stride + d0, false, x[c]);
    if (a.delta) {
      float y[8];
      load8(a.delta, r * a.hidden + d0, true, y);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[c][e] += y[e];
    }
    if (a.out) {
      float* o = a.out + r * a.out_stride + d0;
      *reinterpret_cast<f32x4*>(o) = f32x4{x[c][0], x[c][1], x[c][2], x[c][3]};
      *reinterpret_cast<f32x4*>(o + 4) = f32x4{x[c][4], x[c][5], x[c][6], x[c][7]};
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(x[c][e], x[c][e], ss);
  }
  if (!a.weight) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float inv = rsqrtf(ss / (float)a.hidden + a.eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int d0 = 512 * c + 8 * lane;
    if (d0 >= a.hidden) continue;
    float w[8], y[8];
    load8(a.weight, d0, a.weight_dtype == WMX_DTYPE_BF16, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (x[c][e] * inv) * w[e];
    const u32x4 p = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]), pack_bf16x2(y[6], y[7])};
    *reinterpret_cast<u32x4*>((bf16*)a.normed + r * a.hidden + d0) = p;
  }
}

// LPR lanes (D / 8 rounded up to a power of two) per (token, head) row:
// y = bf16(q * rsqrt(mean(q^2) + eps) * w), then bf16(y cos + rot(y) sin) with
// rot(y) = (-y[D/2:], y[:D/2]).
template <int D>
__global__ __launch_bounds__(256) void query_norm_rope_kernel(const wmx_query_rope_args a) {
#pragma clang fp contract(off)
  constexpr int L = D / 8, LPR = D == 96 ? 16 : L;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int l = threadIdx.x % LPR;
  const bool live = row < a.tokens * a.heads && l < L;
  const int64_t at = live ? row * D + 8 * l : 0;
  float q[8], w[8], c[8], s[8];
  load8(a.q, at, true, q);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(q[e], q[e], ss);
  ss = live ? ss : 0.f;
#pragma unroll
  for (int o = LPR / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float inv = rsqrtf(ss / (float)D + a.eps);
  const int64_t n = live ? row / a.heads : 0;
  const int64_t rope = n / a.tokens_per_row * a.rope_stride[0] + n % a.tokens_per_row * a.rope_stride[1] + (live ? 8 * l : 0);
  load8(a.weight, live ? 8 * l : 0, a.weight_dtype == WMX_DTYPE_BF16, w);
  load8(a.cos, rope, false, c);
  load8(a.sin, rope, false, s);
  float y[8], out[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = round_bf16((q[e] * inv) * w[e]);
  // the partner of element d is d +- D/2, held L / 2 lanes away
  const int lane = threadIdx.x & 63, from = l < L / 2 ? lane + L / 2 : lane - L / 2;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = __shfl(y[e], from);
    out[e] = y[e] * c[e] + (l < L / 2 ? -p : p) * s[e];
  }
  if (live)
    *reinterpret_cast<u32x4*>((bf16*)a.out + at) = u32x4{pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3]),
                                                         pack_bf16x2(out[4], out[5]), pack_bf16x2(out[6], out[7])};
}

// out = bf16(bf16(silu(gate)) * up), eight elements a thread.
__global__ __launch_bounds__(256) void silu_mul_kernel(const bf16* gate, const bf16* up, bf16* out, int64_t n8) {
#pragma clang fp contract(off)
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    float g[8], u[8], y[8];
    load8(gate, 8 * i, true, g);
    load8(up, 8 * i, true, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = round_bf16(g[e] / (1.f + expf(-g[e]))) * u[e];
    *reinterpret_cast<u32x4*>(out + 8 * i) =
        u32x4{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]), pack_bf16x2(y[6], y[7])};
  }
}

template <int CH>
void launch_norm(const wmx_residual_norm_args& a, hipStream_t stream) {
  hipLaunchKernelGGL((residual_norm_kernel<CH>), dim3((unsigned)((a.rows + 3) / 4)), dim3(256), 0, stream, a);
}

template <int D>
void launch_rope(const wmx_query_rope_args& a, hipStream_t stream) {
  constexpr int rows = 256 / (D == 96 ? 16 : D / 8);
  const int64_t n = a.tokens * a.heads;
  hipLaunchKernelGGL((query_norm_rope_kernel<D>), dim3((unsigned)((n + rows - 1) / rows)), dim3(256), 0, stream, a);
}

}  // namespace

int launch_residual_norm(const wmx_residual_norm_args& a, hipStream_t stream) {
  if ((a.rows + 3) / 4 > UINT32_MAX) return WMX_E_UNSUPPORTED;
  if (a.hidden <= 512) launch_norm<1>(a, stream);
  else if (a.hidden <= 1024) launch_norm<2>(a, stream);
  else if (a.hidden <= 2048) launch_norm<4>(a, stream);
  else launch_norm<8>(a, stream);
  return WMX_OK;
}

int launch_query_norm_rope(const wmx_query_rope_args& a, hipStream_t stream) {
  if (a.tokens * a.heads > (int64_t)UINT32_MAX) return WMX_E_UNSUPPORTED;
  switch (a.head_dim) {
    case 64: launch_rope<64>(a, stream); break;
    case 96: launch_rope<96>(a, stream); break;
    case 128: launch_rope<128>(a, stream); break;
    default: return WMX_E_UNSUPPORTED;
  }
  return WMX_OK;
}

int launch_silu_mul(const void* gate, const void* up, void* out, int64_t n, hipStream_t stream) {
  const int64_t blocks = (n / 8 + 255) / 256;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream,
                     (const bf16*)gate, (const bf16*)up, (bf16*)out, n / 8);
  return WMX_OK;
}

}  // namespace wmx
