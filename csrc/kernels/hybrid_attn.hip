// Attention of prompt portions over a paged bf16 cache at head widths in whole groups of MFMA steps: the fast form of
// attn_tile_kernel (hybrid.hip) for masks that are an interval per row (all earlier keys, a window, a chunk). Queries, scores,
// weights and sums are fp32; only the cached keys and values are 16-bit numbers.
//
// The products run on v_mfma_f32_16x16x32_bf16 all the same, without giving up a bit: a query (and a softmax weight) is cut into
// three bf16 numbers that add up to it exactly (its mantissa, eight bits at a time), keys and values are bf16 already, products
// of two bf16 numbers are exact in fp32, and the sums are fp32. Three such instructions do the work of eight
// v_mfma_f32_16x16x4_f32 of twice their length. 3001 rows over all earlier keys, 16 heads of 128 over values of 256: 755 -> 235
// us (55 GFLOP: 235 TFLOP/s where the fp32 instructions peak at 157); 2048 rows, values of 128: 233 -> 83 us; error against 64
// bits 3.4e-7 -> 2.1e-7 and 8.9e-7 -> 6.0e-7. With capped scores and four value heads side by side (700 rows, 512 value
// columns a head; 16-key tiles before) 357 -> 77 us, over latent rows (keys of 192, values of 128) 161 -> 37 us.
// (Not the same: an infinite key or value, which met a weight, now gives NaN where it gave an infinity.)
//
// A block is four waves = 64 query rows of ONE sequence and ONE query head, 16 rows a wave; keys come 32 at a time.
//   - Scores are formed transposed (keys x queries), so that a lane holds eight keys' scores of ONE row: a row's maximum is two
//     lane swaps, its rescaling one number per lane, and its weights are the operand of the second product as they stand
//     (depth 8 (lane >> 4) + j of that product is key 16 (j >> 2) + 4 (lane >> 4) + (j & 3), for weights and values alike).
//   - A wave's queries stay in registers (scaled by scale * log2 e, so that weights are powers of two).
//   - Keys and values go to LDS as they lie in the cache (16-byte copies, two buffers, one barrier per 32 keys; the loads of the
//     next keys are in flight meanwhile). The values' operand is their transpose: ds_read_b64_tr_b16 reads it so.
//   - Tiles that every row of the wave sees whole need no mask; accumulators are rescaled only when a maximum moved.
//   - GROUPS = 2: eight waves, of which the second four take every other tile of keys for the same rows; the two results are
//     joined at the end. One wave alone leaves a SIMD idle more than half of the time, and the last rows' block, which has
//     twice the mean number of keys, decides how long a small launch takes: two groups halve its chain.
#include "hybrid_common.h"

namespace {

constexpr float kLog2e = 1.4426950408889634f;

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Over the four lanes that hold a row's keys (lane, lane ^ 16, lane ^ 32, lane ^ 48).
LC_DEVICE float swap_max(float v) {
  const uint32_t b = __float_as_uint(v);
  const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(b, b, false, false));
  const uint32_t c = __float_as_uint(fmaxf(__uint_as_float(r.x), __uint_as_float(r.y)));
  const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(c, c, false, false));
  return fmaxf(__uint_as_float(t.x), __uint_as_float(t.y));
}
LC_DEVICE float swap_sum(float v) {
  const uint32_t b = __float_as_uint(v);
  const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(b, b, false, false));
  const uint32_t c = __float_as_uint(__uint_as_float(r.x) + __uint_as_float(r.y));
  const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(c, c, false, false));
  return __uint_as_float(t.x) + __uint_as_float(t.y);
}

// The upper halves of two floats' bits: two truncated bf16 numbers.
LC_DEVICE uint32_t upper_halves(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
LC_DEVICE float truncated(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// Two finite floats as three pairs of bf16 numbers that add up to them: eight bits of the mantissa each, the rest is exact.
LC_DEVICE void split3(float a, float b, uint32_t& w0, uint32_t& w1, uint32_t& w2) {
  w0 = upper_halves(a, b);
  a -= truncated(a);
  b -= truncated(b);
  w1 = upper_halves(a, b);
  a -= truncated(a);
  b -= truncated(b);
  w2 = upper_halves(a, b);
}
// The same of numbers that may not be finite: those stand in the first part alone.
LC_DEVICE void split3_any(float a, float b, uint32_t& w0, uint32_t& w1, uint32_t& w2) {
  const float fa = fabsf(a) < INFINITY ? a : 0.f, fb = fabsf(b) < INFINITY ? b : 0.f;
  split3(fa, fb, w0, w1, w2);
  const uint32_t ua = a != a ? 0x7fc0u : __float_as_uint(a) >> 16, ub = b != b ? 0x7fc0u : __float_as_uint(b) >> 16;
  w0 = ua | (ub << 16);
}

// tanh to fp32 accuracy: small arguments (capped scores mostly are) by the odd series, whose next term is 2e-10 of the result
// at 1/4; a wave with any larger one takes the library function.
LC_DEVICE float tanh_series(float x) {
  const float y = x * x;
  return x * (1.f + y * (-1.f / 3.f + y * (2.f / 15.f + y * (-17.f / 315.f + y * (62.f / 2835.f + y * (-1382.f / 155925.f))))));
}

struct TileArgs {
  const float* q;                // [T, H * D]
  const bf16_t* kc;              // planes [blocks, G, BS, k_ld], [blocks, G / v_share, BS, v_ld]
  const bf16_t* vc;
  const int32_t* block_tables;
  int MB;
  const int32_t* cu_q;
  const int32_t* positions;
  void* out;                     // row (t, h) at t * o_row + h * o_ld
  int H, G, BS;
  float scale;
  int chunk, window, k_ld, v_ld, v_share;
  const float* sinks;            // score of a silent extra entry per head (null: none)
  const float* gate;             // logits [T, ld_gate], column h: the head's result times its sigmoid (null: none)
  int ld_gate;
  float out_scale;
  int o_row, o_ld;
  int zero_sink;                 // a silent extra entry of score 0
  float softcap;                 // > 0: a scaled score s becomes softcap * tanh(s / softcap)
  int vh0, head_cols, o_col0;    // vh0 >= 0: value heads from vh0 on side by side, head_cols columns each, whatever the query head
};

constexpr int kKeys = 32;

// LDS of one group of four waves: two buffers of keys and values.
template <int DT, int VT>
constexpr int group_lds() {
  return 2 * kKeys * (16 * DT + 8 + 16 * VT + 16) * 2;
}

template <bool AF32, int DT, int VT, int GROUPS, bool CAP>
__global__ __launch_bounds__(256 * GROUPS, 2) void attn_keys32_kernel(TileArgs a) {
  constexpr int D = 16 * DT, NC = 16 * VT, DK = D / 32;
  constexpr int KS = D + 8, VS = NC + 16;            // row strides (bf16): 16 operand rows in different banks
  constexpr int KU = kKeys * D / 8 / 256, VU = kKeys * NC / 8 / 256;      // 16-byte units of a tile per thread
  static_assert(KU >= 1 && VU >= 1 && VT % 4 == 0, "tiles of at least one unit per thread");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x & 255, group = threadIdx.x >> 8;
  bf16_t* Ks = reinterpret_cast<bf16_t*>(lds + group * group_lds<DT, VT>());      // [2][kKeys * KS]
  bf16_t* Vs = Ks + 2 * kKeys * KS;                  // [2][kKeys * VS]
  const int b = blockIdx.z, h = GROUPS == 1 ? blockIdx.y : blockIdx.x;
  const int q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
  int tile;
  if (GROUPS == 1) {
    // A portion's later rows see more keys. Workgroups i and i + 256 share a CU, so every other 256 walk the row tiles
    // backwards: a long tile and a short one meet on a CU instead of two long ones.
    const bool forward = (((b * static_cast<int>(gridDim.y) + h) * static_cast<int>(gridDim.x)) >> 8) & 1;
    tile = forward ? blockIdx.x : gridDim.x - 1 - blockIdx.x;
  } else {
    tile = gridDim.y - 1 - blockIdx.y;               // a block has a CU to itself: the long tiles of all heads first
  }
  const int row0 = q0 + tile * 64;
  if (row0 >= q1) return;                            // the same for the whole block
  const int wave = tid >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int g = h / (a.H / a.G), gv = a.vh0 >= 0 ? a.vh0 : g / a.v_share, GV = a.G / a.v_share;
  const int32_t* table = a.block_tables + static_cast<size_t>(b) * a.MB;
  const int p0 = a.positions[row0];                  // rows of a portion are consecutive positions
  const int nrows = min(64, q1 - row0);
  auto first_key = [&](int p) {
    int lo = 0;
    if (a.chunk > 0) lo = (p / a.chunk) * a.chunk;
    if (a.window > 0) lo = max(lo, p - a.window + 1);
    return lo;
  };
  const int hi = p0 + nrows - 1;                     // the block's last key
  const int pw0 = p0 + 16 * wave;
  const int wave_rows = max(0, min(16, nrows - 16 * wave));
  const int wave_lo = first_key(pw0), wave_hi = pw0 + wave_rows - 1;
  const int full_lo = first_key(pw0 + 15);           // from here on to pw0 every row of the wave sees every key
  const int row_lo = first_key(pw0 + lr);            // of the row whose scores this lane holds
  bf16x8 q[3][DK];
  {
    const bool on = lr < wave_rows;                  // (rows past the portion: zero, never stored)
    const float* src = a.q + (static_cast<size_t>(row0 + 16 * wave + (on ? lr : 0)) * a.H + h) * D + 8 * lk;
    const float s = on ? a.scale * (CAP ? 1.f : kLog2e) : 0.f;
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
      const float4 x = *reinterpret_cast<const float4*>(src + 32 * kk), y = *reinterpret_cast<const float4*>(src + 32 * kk + 4);
      u32x4 w0, w1, w2;
      uint32_t c0, c1, c2;
      split3_any(x.x * s, x.y * s, c0, c1, c2);
      w0.x = c0, w1.x = c1, w2.x = c2;
      split3_any(x.z * s, x.w * s, c0, c1, c2);
      w0.y = c0, w1.y = c1, w2.y = c2;
      split3_any(y.x * s, y.y * s, c0, c1, c2);
      w0.z = c0, w1.z = c1, w2.z = c2;
      split3_any(y.z * s, y.w * s, c0, c1, c2);
      w0.w = c0, w1.w = c1, w2.w = c2;
      q[0][kk] = __builtin_bit_cast(bf16x8, w0);
      q[1][kk] = __builtin_bit_cast(bf16x8, w1);
      q[2][kk] = __builtin_bit_cast(bf16x8, w2);
    }
  }
  // staging: a tile's keys lie in one block of the cache (its size is a multiple of 32)
  u32x4 kr[KU], vr[VU];
  int k_at[KU], v_at[VU];
#pragma unroll
  for (int i = 0; i < KU; ++i) {
    const int u = tid + 256 * i;
    k_at[i] = (u / (D / 8)) * a.k_ld + (u % (D / 8)) * 8;
  }
#pragma unroll
  for (int i = 0; i < VU; ++i) {
    const int u = tid + 256 * i, col = (u % (NC / 8)) * 8, head = col / a.head_cols;     // (one value head: head 0)
    v_at[i] = (head * a.BS + u / (NC / 8)) * a.v_ld + col - head * a.head_cols;
  }
  auto block_of = [&](int j0) { return j0 <= hi ? table[j0 / a.BS] : 0; };
  auto fetch = [&](int j0, int block) {
    const bf16_t* k = a.kc + ((static_cast<size_t>(block) * a.G + g) * a.BS + j0 % a.BS) * a.k_ld;
    const bf16_t* v = a.vc + ((static_cast<size_t>(block) * GV + gv) * a.BS + j0 % a.BS) * a.v_ld;
#pragma unroll
    for (int i = 0; i < KU; ++i) kr[i] = *reinterpret_cast<const u32x4*>(k + k_at[i]);   // (keys past hi are cells of the same
#pragma unroll                                                                           // block: read, never seen)
    for (int i = 0; i < VU; ++i) vr[i] = *reinterpret_cast<const u32x4*>(v + v_at[i]);
  };
  auto stage = [&](int buf, int j0) {                // (the first use of what fetch loaded)
    if (j0 + kKeys - 1 > hi) {
#pragma unroll
      for (int i = 0; i < VU; ++i)                   // what nobody wrote may be no number, and its weight of zero times it
        if (j0 + (tid + 256 * i) / (NC / 8) > hi) vr[i] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < KU; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<u32x4*>(&Ks[buf * kKeys * KS + (u / (D / 8)) * KS + (u % (D / 8)) * 8]) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VU; ++i) {
      const int u = tid + 256 * i;
      *reinterpret_cast<u32x4*>(&Vs[buf * kKeys * VS + (u / (NC / 8)) * VS + (u % (NC / 8)) * 8]) = vr[i];
    }
  };
  float m, l;                                        // (this lane's keys only in l: summed over the row at the end)
  f32x4 o[VT];                                       // columns 16 t + 4 lk + r of row lr
  m = a.sinks != nullptr && group == 0 ? a.sinks[h] * kLog2e : a.zero_sink && group == 0 ? 0.f : -INFINITY;
  l = (a.sinks != nullptr || a.zero_sink) && group == 0 && lk == 0 ? 1.f : 0.f;
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int STEP = kKeys * GROUPS;
  const int lo_tile = (first_key(p0) / kKeys) * kKeys;
  int j0 = lo_tile + group * kKeys;                  // this group's first tile
  if (j0 <= hi) {
    fetch(j0, block_of(j0));
    stage(0, j0);
  }
  int ahead = block_of(j0 + STEP), buf = 0;
  for (int jb = lo_tile; jb <= hi; jb += STEP, j0 += STEP, buf ^= 1) {      // (all groups take the same number of turns)
    __syncthreads();                                 // this tile is in place, and nobody reads the other buffer any more
    const bool more = j0 + STEP <= hi;
    if (more) {
      fetch(j0 + STEP, ahead);
      ahead = block_of(j0 + 2 * STEP);
    }
    if (wave_rows > 0 && j0 <= wave_hi && j0 + kKeys - 1 >= wave_lo) {      // wave-uniform
      f32x4 s[2][2];                                 // [keys 16 e ..][first part of the query | the other two]
#pragma unroll
      for (int e = 0; e < 2; ++e) s[e][0] = s[e][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < DK; ++kk) {
        bf16x8 k[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
          k[e] = *reinterpret_cast<const bf16x8*>(&Ks[buf * kKeys * KS + (16 * e + lr) * KS + 32 * kk + 8 * lk]);
#pragma unroll
        for (int e = 0; e < 2; ++e) s[e][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[e], q[2][kk], s[e][1], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) s[e][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[e], q[0][kk], s[e][0], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) s[e][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[e], q[1][kk], s[e][1], 0, 0, 0);
      }
      float p[2][4];
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) p[e][r] = s[e][0][r] + s[e][1][r];
      if constexpr (CAP) {
        const float inv = 1.f / a.softcap;
        float top = 0.f;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[e][r] *= inv;
            top = fmaxf(top, fabsf(p[e][r]));
          }
        const bool series = !__any(!(top <= 0.25f));
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) p[e][r] = (series ? tanh_series(p[e][r]) : tanhf(p[e][r])) * (a.softcap * kLog2e);
      }
      if (j0 + kKeys - 1 > pw0 || j0 < full_lo) {    // some row does not see the whole tile
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = j0 + 16 * e + 4 * lk + r;
            if (j > pw0 + lr || j < row_lo) p[e][r] = -INFINITY;
          }
      }
      float top = fmaxf(fmaxf(fmaxf(p[0][0], p[0][1]), fmaxf(p[0][2], p[0][3])), fmaxf(fmaxf(p[1][0], p[1][1]), fmaxf(p[1][2], p[1][3])));
      const float mn = fmaxf(m, swap_max(top));
      const float base = mn == -INFINITY ? 0.f : mn;          // nothing visible yet: weights 0, no NaN
      const float corr = fast_exp2(m - base);
      m = mn;
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) p[e][r] = fast_exp2(p[e][r] - base);
      l = l * corr + (((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) + ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3])));
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[t][r] *= corr;
      }
      bf16x8 w[3];
      {
        u32x4 w0, w1, w2;
        uint32_t c0, c1, c2;
        split3(p[0][0], p[0][1], c0, c1, c2);
        w0.x = c0, w1.x = c1, w2.x = c2;
        split3(p[0][2], p[0][3], c0, c1, c2);
        w0.y = c0, w1.y = c1, w2.y = c2;
        split3(p[1][0], p[1][1], c0, c1, c2);
        w0.z = c0, w1.z = c1, w2.z = c2;
        split3(p[1][2], p[1][3], c0, c1, c2);
        w0.w = c0, w1.w = c1, w2.w = c2;
        w[0] = __builtin_bit_cast(bf16x8, w0);
        w[1] = __builtin_bit_cast(bf16x8, w1);
        w[2] = __builtin_bit_cast(bf16x8, w2);
      }
      // lane lr of a group of 16 addresses row 4 lk + (lr >> 2), columns 4 (lr & 3) .. + 3, and receives column lr of the four rows
      bf16_t* vs = Vs + buf * kKeys * VS + (4 * lk + (lr >> 2)) * VS + 4 * (lr & 3);
#pragma unroll
      for (int t = 0; t < VT; t += 4) {
        bf16x8 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vs + 16 * (t + i)));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vs + 16 * VS + 16 * (t + i)));
          v[i] = bf16x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
#pragma unroll
        for (int c = 2; c >= 0; --c)                 // the small parts first; four independent chains
#pragma unroll
          for (int i = 0; i < 4; ++i) o[t + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], w[c], o[t + i], 0, 0, 0);
      }
    }
    if (more) stage(buf ^ 1, j0 + STEP);
  }
  if constexpr (GROUPS == 2) {
    // the second group's sums go through LDS (the tiles are done with), register after register, to the first one's lanes
    static_assert((4 * VT + 2) * 256 * 4 <= 2 * group_lds<DT, VT>(), "the sums fit where the tiles were");
    float* xs = reinterpret_cast<float*>(lds);
    __syncthreads();
    if (group == 1) {
      xs[tid] = m;
      xs[256 + tid] = l;
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) xs[(2 + 4 * t + r) * 256 + tid] = o[t][r];
    }
    __syncthreads();
    if (group == 1) return;                          // (no barrier follows)
    const float m1 = xs[tid], mn = fmaxf(m, m1);
    const float base = mn == -INFINITY ? 0.f : mn;
    const float f0 = fast_exp2(m - base), f1 = fast_exp2(m1 - base);
    l = l * f0 + xs[256 + tid] * f1;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[t][r] = o[t][r] * f0 + xs[(2 + 4 * t + r) * 256 + tid] * f1;
  }
  const float sum = swap_sum(l);
  if (lr >= wave_rows) return;
  const size_t tok = static_cast<size_t>(row0) + 16 * wave + lr;
  const float fin = a.out_scale * (a.gate != nullptr ? sigmoidf_(a.gate[tok * a.ld_gate + h]) : 1.f) / sum;
  typename Act<AF32>::type* dst = static_cast<typename Act<AF32>::type*>(a.out) + tok * a.o_row + static_cast<size_t>(h) * a.o_ld + a.o_col0 + 4 * lk;
#pragma unroll
  for (int t = 0; t < VT; ++t) store_act4<AF32>(dst, 16 * t, make_float4(o[t][0] * fin, o[t][1] * fin, o[t][2] * fin, o[t][3] * fin));
}

}  // namespace

// Launches of up to this many row tiles run two groups of waves per tile.
constexpr long long kTwoGroupBlocks = 1024;

// Whether lc_attn_keys32 takes key width D, ``cols`` value columns and the block size (1) or not (0).
LC_EXPORT int lc_attn_keys32_ok(int D, int cols, int BS) {
  return BS % kKeys == 0 && ((D == 64 && (cols == 64 || cols == 128)) || ((D == 128 || D == 192) && (cols == 128 || cols == 256)));
}

// Sequences [0, n_seq) of cu_q, the longest of max_len rows; planes, row strides and options as for lc_attn_tile (nvh value heads
// of Dv columns from vh0 on, or with vh0 < 0 the query head's own; results from column o_col0 of a head's o_ld on).
LC_EXPORT int lc_attn_keys32(const void* q, const void* kc, const void* vc, const void* block_tables, int MB, const void* cu_q,
                             const void* positions, void* out, int act_f32, int n_seq, int max_len, int H, int G, int D, int Dv,
                             int BS, float scale, int chunk, int window, int k_ld, int v_ld, float softcap, int sink,
                             const void* sinks, const void* gate, int ld_gate, float out_scale, int o_row, int v_share, int vh0,
                             int nvh, int o_ld, int o_col0, hipStream_t st) {
  if (n_seq <= 0 || max_len <= 0) return 0;
  const int cols = nvh * Dv;
  if (H <= 0 || G <= 0 || H % G || MB <= 0 || v_share <= 0 || G % v_share || nvh <= 0 || Dv <= 0 || !lc_attn_keys32_ok(D, cols, BS)) return -1;
  if (vh0 < 0 ? nvh != 1 : (vh0 + nvh > G || v_share != 1 || Dv % 8)) return -1;
  if (k_ld < D || v_ld < Dv || k_ld % 8 || v_ld % 8 || !aligned16(q) || !aligned16(kc) || !aligned16(vc) || softcap < 0.f) return -1;
  if (o_col0 < 0 || o_col0 % 4 || o_ld < o_col0 + cols || o_row < H * o_ld || o_ld % 4 || o_row % 4 ||
      reinterpret_cast<uintptr_t>(out) % (act_f32 ? 16 : 8))
    return -1;
  if ((gate != nullptr && ld_gate < H) || (sinks != nullptr && !sink)) return -1;
  const TileArgs a{static_cast<const float*>(q), static_cast<const bf16_t*>(kc), static_cast<const bf16_t*>(vc),
                   static_cast<const int32_t*>(block_tables), MB, static_cast<const int32_t*>(cu_q),
                   static_cast<const int32_t*>(positions), out, H, G, BS, scale, chunk, window, k_ld, v_ld, v_share,
                   static_cast<const float*>(sinks), static_cast<const float*>(gate), ld_gate, out_scale, o_row, o_ld,
                   sink && sinks == nullptr, softcap, vh0, Dv, o_col0};
  const int tiles = (max_len + 63) / 64;
  if (tiles > 65535 || H > 65535 || n_seq > 65535) return -1;
  const bool two = static_cast<long long>(tiles) * H * n_seq <= kTwoGroupBlocks;
#define LC_K32_G(A32, DT, VT, CAP)                                                                                        \
  do {                                                                                                                    \
    constexpr int one_lds = group_lds<DT, VT>();                                                                          \
    static LcDeviceOnce attr_once;                                                                                        \
    attr_once.run([&] {                                                                                                   \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attn_keys32_kernel<A32, DT, VT, 1, CAP>),                   \
                                hipFuncAttributeMaxDynamicSharedMemorySize, one_lds);                                     \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attn_keys32_kernel<A32, DT, VT, 2, CAP>),                   \
                                hipFuncAttributeMaxDynamicSharedMemorySize, 2 * one_lds);                                 \
    });                                                                                                                   \
    if (two) attn_keys32_kernel<A32, DT, VT, 2, CAP><<<dim3(H, tiles, n_seq), dim3(512), 2 * one_lds, st>>>(a);           \
    else attn_keys32_kernel<A32, DT, VT, 1, CAP><<<dim3(tiles, H, n_seq), dim3(256), one_lds, st>>>(a);                   \
  } while (0)
#define LC_K32(DT, VT)                                            \
  do {                                                            \
    if (act_f32 && softcap > 0.f) LC_K32_G(true, DT, VT, true);   \
    else if (act_f32) LC_K32_G(true, DT, VT, false);              \
    else if (softcap > 0.f) LC_K32_G(false, DT, VT, true);        \
    else LC_K32_G(false, DT, VT, false);                          \
  } while (0)
  if (D == 64 && cols == 64) LC_K32(4, 4);
  else if (D == 64) LC_K32(4, 8);
  else if (D == 128 && cols == 128) LC_K32(8, 8);
  else if (D == 128) LC_K32(8, 16);
  else if (cols == 128) LC_K32(12, 8);
  else LC_K32(12, 16);
#undef LC_K32
#undef LC_K32_G
  LC_RETURN_LAST_ERROR();
}
