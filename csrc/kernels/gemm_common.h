// Pieces shared by the GEMM translation units: epilogue modes and the accumulator-tile
// store (bias, bf16/fp32 output, fused SwiGLU over gate/up tiles interleaved at 16 columns).
#pragma once
#include "common.h"

namespace {

enum Epilogue : int {
  EPI_BF16 = 0,    // Y bf16 [M, ldy]  (+bias)
  EPI_F32 = 1,     // Y f32  [M, ldy]  (+bias); with split-K: slab blockIdx.y of [S, M, ldy], no bias
  EPI_SWIGLU = 2,  // n-tiles alternate gate/up; Y bf16 [M, N/2] = silu(gate)*up (+bias before act)
  EPI_RELU2 = 3,   // Y bf16 [M, ldy] = relu(. + bias)^2 (the grouped kernels, gemm256, kgemm)
  EPI_GLU_CLAMPED = 4,  // n-tiles alternate gate/up; Y bf16 [M, N/2] = clamped gated unit with a scale per row (the grouped kernels)
  EPI_GEGLU = 5,   // as EPI_SWIGLU with the tanh form of gelu instead of silu (gemm256)
  EPI_REGLU = 6,   // ... with relu (gemm256)
  EPI_XIELU = 7,   // Y bf16 [M, ldy] = xielu(. + bias) (gemm256, kgemm)
};

// Epilogues that store act(gate) * up.
constexpr bool epi_gated(int epi) { return epi == EPI_SWIGLU || epi == EPI_GEGLU || epi == EPI_REGLU; }
// Epilogues that store act(.) of single columns.
constexpr bool epi_acts(int epi) { return epi == EPI_RELU2 || epi == EPI_XIELU; }

// Constants of the clamped gated unit: with s = row_scale[row] (1 without the array), g = min(s * gate, limit),
// u = clamp(s * up, -limit, limit), the output is g * sigmoid(slope * g) * (u + shift).
struct GluClamp {
  const float* row_scale;
  float limit, slope, shift;
};

LC_DEVICE float silu(float x) { return x / (1.f + __expf(-x)); }

// 0.5 x (1 + tanh(a)) = x sigmoid(2 a), a = sqrt(2 / pi) (x + 0.044715 x^3)
LC_DEVICE float gelu_tanh(float x) { return x / (1.f + __expf(-1.5957691216057308f * (x + 0.044715f * x * x * x))); }

template <int EPI>
LC_DEVICE float gate_act(float x) { return EPI == EPI_GEGLU ? gelu_tanh(x) : EPI == EPI_REGLU ? fmaxf(x, 0.f) : silu(x); }

// xielu (common.h) for results that are rounded to bf16, without expm1f's two paths: e^x - 1 - x is x^2 times a polynomial down to
// -1 (degree 6, fitted at the Chebyshev points of [-1, 0], 1e-8 of the value in exact numbers), the difference itself
// below. Rounded to bf16 it equals the form with expm1f on 3M normal values. A
// tile's epilogue holds 128 values a lane: 2361 x 8192 x 2048 115.6 -> 109.2 us (relu^2 98.9), 40 x 8192 x 2048 10.7 -> 10.2.
LC_DEVICE float xielu_bf16(float x, float ap, float an) {
  float p = 1.6928126569837332e-05f;
  p = fmaf(p, x, 1.8832476052921265e-04f);
  p = fmaf(p, x, 1.3822416076436639e-03f);
  p = fmaf(p, x, 8.3310501649975780e-03f);
  p = fmaf(p, x, 4.1666291654109955e-02f);
  p = fmaf(p, x, 1.6666664183139801e-01f);
  p = fmaf(p, x, 0.5f);
  const float near_ = x * x * p, far_ = __expf(x) - 1.f - x;
  return (x > 0.f ? ap * x * x : an * (x > -1.f ? near_ : far_)) + 0.5f * x;
}

// The activation of an EPI_RELU2 or EPI_XIELU epilogue (ap, an: the two numbers of xIELU), v itself in the others.
template <int EPI>
LC_DEVICE float column_act(float v, float ap, float an) {
  if constexpr (EPI == EPI_RELU2) return relu2(v);
  if constexpr (EPI == EPI_XIELU) return xielu_bf16(v, ap, an);
  return v;
}

// The clamped gated unit over a gate tile and the up tile next to it (same layout as the SwiGLU store below).
// ``row_scale`` is indexed like the output rows.
LC_DEVICE void store_tile_glu_clamped(const f32x4& acc, const f32x4& acc_up, void* __restrict__ Y, const GluClamp& glu,
                                      int m0, int n0, int M, int N, int ldy, int lane) {
  const int m = m0 + (lane & 15);
  const int nb = n0 + 4 * (lane >> 4);
  if (m >= M || nb >= N) return;
  const int ob = (n0 >> 1) + 4 * (lane >> 4);
  const float s = glu.row_scale != nullptr ? glu.row_scale[m] : 1.f;
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float g = fminf(acc[r] * s, glu.limit);
    const float u = fminf(fmaxf(acc_up[r] * s, -glu.limit), glu.limit);
    v[r] = g / (1.f + expf(-glu.slope * g)) * (u + glu.shift);
  }
  u32x2 o;
  o[0] = pack_bf16x2(v[0], v[1]);
  o[1] = pack_bf16x2(v[2], v[3]);
  *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(Y) + static_cast<size_t>(m) * ldy + ob) = o;
}

// Stores one 16(n) x 16(m) accumulator tile. `n0`/`m0` are the tile origin.
template <int EPI>
LC_DEVICE void store_tile(const f32x4& acc, const f32x4* acc_up, void* __restrict__ Y,
                          const bf16_t* __restrict__ bias, int m0, int n0, int M, int N, int ldy,
                          int lane, size_t slab_off, float ap = 0.f, float an = 0.f) {
  const int m = m0 + (lane & 15);
  const int nb = n0 + 4 * (lane >> 4);
  if (m >= M) return;
  if constexpr (epi_gated(EPI)) {
    // n0 is the gate tile's origin in the interleaved space; output column = n0/2 + ...
    if (nb >= N) return;
    const int ob = (n0 >> 1) + 4 * (lane >> 4);
    float g[4], u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      g[r] = acc[r];
      u[r] = (*acc_up)[r];
      if (bias) {
        g[r] += bf16_to_f32(bias[nb + r]);
        u[r] += bf16_to_f32(bias[nb + 16 + r]);
      }
    }
    u32x2 o;
    o[0] = pack_bf16x2(gate_act<EPI>(g[0]) * u[0], gate_act<EPI>(g[1]) * u[1]);
    o[1] = pack_bf16x2(gate_act<EPI>(g[2]) * u[2], gate_act<EPI>(g[3]) * u[3]);
    *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(Y) + static_cast<size_t>(m) * ldy + ob) = o;
  } else {
    if (nb >= N) return;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = acc[r] + ((bias && nb + r < N) ? bf16_to_f32(bias[nb + r]) : 0.f);
    if constexpr (epi_acts(EPI)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = column_act<EPI>(v[r], ap, an);
    }
    if constexpr (EPI == EPI_BF16 || epi_acts(EPI)) {
      bf16_t* dst = static_cast<bf16_t*>(Y) + static_cast<size_t>(m) * ldy + nb;
      if (nb + 3 < N) {
        u32x2 o;
        o[0] = pack_bf16x2(v[0], v[1]);
        o[1] = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<u32x2*>(dst) = o;
      } else {
        for (int r = 0; r < 4 && nb + r < N; ++r) dst[r] = f32_to_bf16(v[r]);
      }
    } else {
      float* dst = static_cast<float*>(Y) + slab_off + static_cast<size_t>(m) * ldy + nb;
      if (nb + 3 < N) {
        *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
      } else {
        for (int r = 0; r < 4 && nb + r < N; ++r) dst[r] = v[r];
      }
    }
  }
}

}  // namespace
