// Decode GEMM for small M (<= 64) and narrow outputs: Y[M,N] = X[M,K] * W[N,K]^T where
// N/128 is far below the 256 CUs of the chip (attention QKV / O / MLP-down at batch 64).
//
// Instead of splitting K across workgroups (fp32 partial slabs + a reduce launch), the K
// range is split across the 8 waves of ONE workgroup and reduced through LDS:
//   * a workgroup owns NTW consecutive 16-column n-tiles (16..64 output columns), so even
//     N = 4096 yields 256 workgroups of 8 waves;
//   * wave w streams the packed weight fragments of those n-tiles for k-tiles
//     [w*KT/8, (w+1)*KT/8) straight into VGPRs (nontemporal, read exactly once) together
//     with the matching activation fragments (L2-resident, shared by all workgroups);
//   * there is no LDS staging and no barrier in the streaming loop, so the compiler's own
//     counted vmcnt keeps loads in flight continuously;
//   * the 8 partial accumulator sets are summed through LDS (tree, 3 barriers) and wave 0..
//     apply the epilogue (bias / bf16 / fp32 / fused SwiGLU).
// Gated products with one n-tile per workgroup take half a gate tile and half of the up tile beside it as their
// 16 operand rows. Two whole tiles give 28672 columns 896 workgroups, three and a half per CU, so that CUs with
// four finish last (43.7 us at one row of 4096); 1792 of half the size are seven each: 37.0 us (6.3 TB/s).
// Same packed-weight layout and MFMA orientation as gemm.hip (weights = A operand).
#include "gemm_common.h"

namespace {

// The residual sum and norm in front of a product (rmsnorm_kernel, elementwise.hip, number for number): x = h + delta, the operand is
// x * rsqrt(mean(x^2) + eps) * gain. NORM is the number of 8-wide chunks per thread of a row of K = d (256 threads a row, two
// rows at a time), 0 for a product of X as it is. Every workgroup forms the rows for itself, into LDS, while the first weights are on
// their way; the first one stores x. h is not written: others may still read it.
struct NormIn {
  const bf16_t* h;
  const bf16_t* delta;           // or null
  const bf16_t* gain;
  bf16_t* x;                     // with delta
  float eps;
  int tiles;                     // of all workgroups
};
constexpr int kNormRows = 4, kNormPad = 8;   // most rows; elements behind a row in LDS
// Most workgroups: two per CU, which take the tiles in turn. One row, norm and product: 6144 x 4096 13.9 -> 11.9 us, 3072 x 2048 7.5 -> 6.4,
// 10240 x 8192 35.8 -> 34.2 (35.6 with 1024 groups), gated 16384 x 2048 15.3 -> 13.2, 37888 x 3584 47.0 -> 41.5 (44.3 with 256, 42.6
// with 768; the panel kernel before). Gated 28672 x 4096 stays at 41 us (one tile per workgroup 43.2), 57344 x 8192 loses 9.
constexpr int kNormGroups = 512;

template <int MT, int NTW, int EPI, int NORM = 0>
__global__ __launch_bounds__(512, NORM > 0 ? 4 : 2) void kgemm_kernel(const bf16_t* __restrict__ Wp,
                                                    const bf16_t* __restrict__ X, void* __restrict__ Y,
                                                    const bf16_t* __restrict__ bias, int M, int N, int K,
                                                    int ldy, float ap, float an, NormIn norm = {}) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NF = NTW * MT;  // accumulator fragments per wave
  // NORM: sums of squares, then the rows, behind the reduction's part
  float* const squares = reinterpret_cast<float*>(smem + 4 * NF * 64 * sizeof(f32x4));
  bf16_t* const rows = reinterpret_cast<bf16_t*>(squares + 16);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KT = K / 32;
  const int per = (KT + 7) / 8;
  const int kt_lo = wave * per, kt_hi = min(KT, kt_lo + per);
  int tile = blockIdx.x;

  f32x4 acc[NTW][MT];
#pragma unroll
  for (int n = 0; n < NTW; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // per-lane row pointers of the activation fragments (rows clamped for the M tail)
  const bf16_t* xrow[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    int row = m * 16 + (lane & 15);
    row = row < M ? row : M - 1;
    xrow[m] = NORM ? rows + row * (K + kNormPad) + 8 * (lane >> 4) : X + static_cast<size_t>(row) * K + 8 * (lane >> 4);
  }
  // HALF: 8 gate and the 8 up columns that belong to them, half a tile of each, as one operand of 16 rows
  constexpr bool HALF = EPI == EPI_SWIGLU && NTW == 1;
  auto weights = [&](int tile) {
    return HALF ? Wp + static_cast<size_t>(2 * (tile >> 1) + ((lane >> 3) & 1)) * KT * 512 + (8 * (tile & 1) + (lane & 7) + 16 * (lane >> 4)) * 8
                : Wp + static_cast<size_t>(tile * NTW) * KT * 512 + lane * 8;
  };
  const bf16_t* wbase = weights(tile);

  auto load_w = [&](bf16x8 (&wf)[NTW], int kt) {
#pragma unroll
    for (int n = 0; n < NTW; ++n)
      wf[n] = __builtin_nontemporal_load(
          reinterpret_cast<const bf16x8*>(wbase + (static_cast<size_t>(n) * KT + kt) * 512));
  };
  auto load_x = [&](bf16x8 (&xf)[MT], int kt) {
#pragma unroll
    for (int m = 0; m < MT; ++m) xf[m] = *reinterpret_cast<const bf16x8*>(xrow[m] + kt * 32);
  };
  auto load = [&](bf16x8 (&wf)[NTW], bf16x8 (&xf)[MT], int kt) {
    load_w(wf, kt);
    load_x(xf, kt);
  };
  auto fma = [&](const bf16x8 (&wf)[NTW], const bf16x8 (&xf)[MT]) {
#pragma unroll
    for (int n = 0; n < NTW; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[n], xf[m], acc[n][m], 0, 0, 0);
  };

  // register ring of four k-tiles, statically indexed (eight or twelve gain nothing: 4096 x 14336 20.5, 20.6, 20.7 us at one row)
  constexpr int R = 4;
  bf16x8 wr[R][NTW], xr[R][MT];
  if constexpr (NORM > 0) {
    const int t = threadIdx.x & 255, half = wave >> 2, chunks = K / 8;
    bf16x8 hv[NORM], dv[NORM], gain[NORM];
    auto fetch = [&](int row) {
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int c = min(t + i * 256, chunks - 1);
        hv[i] = *reinterpret_cast<const bf16x8*>(norm.h + static_cast<size_t>(row) * K + c * 8);
        if (norm.delta != nullptr) dv[i] = *reinterpret_cast<const bf16x8*>(norm.delta + static_cast<size_t>(row) * K + c * 8);
      }
    };
    fetch(min(half, M - 1));
#pragma unroll
    for (int i = 0; i < NORM; ++i) gain[i] = *reinterpret_cast<const bf16x8*>(norm.gain + min(t + i * 256, chunks - 1) * 8);
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (kt_lo + u < kt_hi) load_w(wr[u], kt_lo + u);
    for (int turn = 0; 2 * turn < M; ++turn) {
      const int row = 2 * turn + half;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int c = t + i * 256;
        if (c >= chunks) continue;
        if (norm.delta != nullptr) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            hv[i][j] = static_cast<short>(f32_to_bf16(bf16_to_f32(static_cast<bf16_t>(hv[i][j])) + bf16_to_f32(static_cast<bf16_t>(dv[i][j]))));
          if (blockIdx.x == 0 && row < M) *reinterpret_cast<bf16x8*>(norm.x + static_cast<size_t>(row) * K + c * 8) = hv[i];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = bf16_to_f32(static_cast<bf16_t>(hv[i][j]));
          ss += f * f;
        }
      }
      ss = wave_sum(ss);
      if (lane == 0) squares[8 * turn + wave] = ss;
      __syncthreads();
      const float* part = squares + 8 * turn + 4 * half;
      const float scale = rsqrtf((part[0] + part[1] + part[2] + part[3]) / static_cast<float>(K) + norm.eps);
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int c = t + i * 256;
        if (c >= chunks || row >= M) continue;
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o[j] = static_cast<short>(f32_to_bf16(bf16_to_f32(static_cast<bf16_t>(hv[i][j])) * scale * bf16_to_f32(static_cast<bf16_t>(gain[i][j]))));
        *reinterpret_cast<bf16x8*>(rows + row * (K + kNormPad) + c * 8) = o;
      }
      if (2 * turn + 2 < M) fetch(min(row + 2, M - 1));
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (kt_lo + u < kt_hi) load_x(xr[u], kt_lo + u);
  } else {
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (kt_lo + u < kt_hi) load(wr[u], xr[u], kt_lo + u);
  }
  // (NORM: a workgroup takes tiles in turn, so that the rows are formed once; the next one's first weights are requested before
  // the sums of this one meet)
  for (;;) {
    int kt = kt_lo;
    for (; kt + 2 * R <= kt_hi; kt += R) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        fma(wr[u], xr[u]);
        load(wr[u], xr[u], kt + R + u);
      }
    }
    for (; kt < kt_hi; kt += R) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        if (kt + u < kt_hi) fma(wr[u], xr[u]);
        if (kt + R + u < kt_hi) load(wr[u], xr[u], kt + R + u);
      }
    }
    const bool more = NORM > 0 && tile + static_cast<int>(gridDim.x) < norm.tiles;
    if (more) {
      wbase = weights(tile + gridDim.x);
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (kt_lo + u < kt_hi) load(wr[u], xr[u], kt_lo + u);
    }

    // ---- cross-wave reduction through LDS: 8 -> 4 -> 2 -> 1 ----
    f32x4* red = reinterpret_cast<f32x4*>(smem);  // [4 waves][NF][64 lanes]
#pragma unroll
    for (int half = 4; half >= 1; half >>= 1) {
      if (wave >= half && wave < 2 * half) {
#pragma unroll
        for (int f = 0; f < NF; ++f) red[((wave - half) * NF + f) * 64 + lane] = acc[f / MT][f % MT];
      }
      __syncthreads();
      if (wave < half) {
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f / MT][f % MT] += red[(wave * NF + f) * 64 + lane];
      }
      __syncthreads();
    }
    if (wave == 0) {
      if constexpr (HALF) {
        const int col = 8 * tile + 4 * (lane >> 4);                    // (lanes 0 .. 31: gate rows of the operand)
        const int gb = 32 * (tile >> 1) + 8 * (tile & 1) + 4 * (lane >> 4);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = acc[0][m][r], u = __shfl(g, lane + 32, 64);
            const bool in = bias != nullptr && lane < 32 && gb < N;
            v[r] = silu(g + (in ? bf16_to_f32(bias[gb + r]) : 0.f)) * (u + (in ? bf16_to_f32(bias[gb + 16 + r]) : 0.f));
          }
          const int row = 16 * m + (lane & 15);
          if (lane < 32 && row < M && gb < N) {
            u32x2 o;
            o[0] = pack_bf16x2(v[0], v[1]);
            o[1] = pack_bf16x2(v[2], v[3]);
            *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(Y) + static_cast<size_t>(row) * ldy + col) = o;
          }
        }
      } else {
#pragma unroll
        for (int n = 0; n < NTW; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            if constexpr (EPI == EPI_SWIGLU) {
              if (n & 1) continue;
              store_tile<EPI>(acc[n][m], &acc[(n + 1) % NTW][m], Y, bias, m * 16, (tile * NTW + n) * 16, M, N, ldy, lane, 0);
            } else {
              store_tile<EPI>(acc[n][m], nullptr, Y, bias, m * 16, (tile * NTW + n) * 16, M, N, ldy, lane, 0, ap, an);
            }
          }
      }
    }
    if (!more) return;
    tile += gridDim.x;
#pragma unroll
    for (int n = 0; n < NTW; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

template <int MT, int NTW>
int launch_k(int epi, const bf16_t* Wp, const bf16_t* X, void* Y, const bf16_t* bias, int M, int N, int K,
             int ldy, int n_pad, float ap, float an, hipStream_t stream) {
  const dim3 grid(n_pad / (16 * NTW)), block(512);
  const size_t lds = 4 * NTW * MT * 64 * sizeof(f32x4);
#define LC_KG(E) kgemm_kernel<MT, NTW, E><<<grid, block, lds, stream>>>(Wp, X, Y, bias, M, N, K, ldy, ap, an)
  if (epi == EPI_BF16) LC_KG(EPI_BF16);
  else if (epi == EPI_F32) LC_KG(EPI_F32);
  else if (epi == EPI_RELU2) LC_KG(EPI_RELU2);
  else if (epi == EPI_XIELU) LC_KG(EPI_XIELU);
  else if (epi == EPI_SWIGLU) LC_KG(EPI_SWIGLU);
  else return -3;
#undef LC_KG
  return static_cast<int>(hipGetLastError());
}

}  // namespace

// M <= 64, K % 32 == 0, n_pad % 128 == 0. ntw = n-tiles (16 columns) per workgroup: 1, 2 or 4 (gated, 1: two halves).
LC_EXPORT int lc_kgemm(const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K,
                       int n_pad, int ldy, int epi, int ntw, float ap, float an, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 64 || K % 32 || n_pad % 128 || N > n_pad) return -1;
  auto w = static_cast<const bf16_t*>(Wp);
  auto x = static_cast<const bf16_t*>(X);
  auto b = static_cast<const bf16_t*>(bias);
  const int mt = (M + 15) / 16;
#define LC_K(MT_)                                                                          \
  if (ntw == 1) return launch_k<MT_, 1>(epi, w, x, Y, b, M, N, K, ldy, n_pad, ap, an, stream);     \
  if (ntw == 2) return launch_k<MT_, 2>(epi, w, x, Y, b, M, N, K, ldy, n_pad, ap, an, stream);     \
  if (ntw == 4) return launch_k<MT_, 4>(epi, w, x, Y, b, M, N, K, ldy, n_pad, ap, an, stream);     \
  return -1;
  if (mt <= 1) { LC_K(1) }
  if (mt <= 2) { LC_K(2) }
  LC_K(4)
#undef LC_K
}

// Y = rmsnorm(h + delta) * W^T for up to four rows in one launch (NormIn; ``x`` receives h + delta, and is not h; without ``delta`` it is not
// written). K is the row's width, a multiple of 32 up to 8192; bf16 or gated results, one or two n-tiles per workgroup.
LC_EXPORT int lc_kgemm_norm(const void* Wp, const void* h, const void* delta, const void* gain, void* x, float eps, void* Y,
                            const void* bias, int M, int N, int K, int n_pad, int ldy, int epi, int ntw, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > kNormRows || K % 32 || K > 8192 || n_pad % 128 || N > n_pad || (epi != EPI_BF16 && epi != EPI_SWIGLU) || (ntw != 1 && ntw != 2) ||
      (delta != nullptr && (x == nullptr || x == h)))
    return -1;
  const size_t lds = 4 * ntw * 64 * sizeof(f32x4) + 64 + static_cast<size_t>(M) * (K + kNormPad) * sizeof(bf16_t);
  if (lds > 64 * 1024) return -1;
  const NormIn norm{static_cast<const bf16_t*>(h), static_cast<const bf16_t*>(delta), static_cast<const bf16_t*>(gain), static_cast<bf16_t*>(x), eps, n_pad / (16 * ntw)};
  const int groups = norm.tiles < kNormGroups ? norm.tiles : kNormGroups;
#define LC_KN(NTW, E, CH)                                                                                                              \
  kgemm_kernel<1, NTW, E, CH><<<dim3(groups), dim3(512), lds, stream>>>(static_cast<const bf16_t*>(Wp), nullptr, Y,    \
                                                                     static_cast<const bf16_t*>(bias), M, N, K, ldy, 0.f, 0.f, norm)
#define LC_KNC(NTW, E)                       \
  do {                                       \
    if (K <= 2048) LC_KN(NTW, E, 1);         \
    else if (K <= 4096) LC_KN(NTW, E, 2);    \
    else LC_KN(NTW, E, 4);                   \
  } while (0)
  if (epi == EPI_BF16) {
    if (ntw == 1) LC_KNC(1, EPI_BF16);
    else LC_KNC(2, EPI_BF16);
  } else {
    if (ntw == 1) LC_KNC(1, EPI_SWIGLU);
    else LC_KNC(2, EPI_SWIGLU);
  }
#undef LC_KNC
#undef LC_KN
  LC_RETURN_LAST_ERROR();
}
