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

template <int MT, int NTW, int EPI>
__global__ __launch_bounds__(512) void kgemm_kernel(const bf16_t* __restrict__ Wp,
                                                    const bf16_t* __restrict__ X, void* __restrict__ Y,
                                                    const bf16_t* __restrict__ bias, int M, int N, int K,
                                                    int ldy, float ap, float an) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NF = NTW * MT;  // accumulator fragments per wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KT = K / 32;
  const int per = (KT + 7) / 8;
  const int kt_lo = wave * per, kt_hi = min(KT, kt_lo + per);
  const int nt0 = blockIdx.x * NTW;

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
    xrow[m] = X + static_cast<size_t>(row) * K + 8 * (lane >> 4);
  }
  // HALF: 8 gate and the 8 up columns that belong to them, half a tile of each, as one operand of 16 rows
  constexpr bool HALF = EPI == EPI_SWIGLU && NTW == 1;
  const int pair = blockIdx.x >> 1, hf = blockIdx.x & 1;
  const bf16_t* wbase = HALF ? Wp + static_cast<size_t>(2 * pair + ((lane >> 3) & 1)) * KT * 512 + (8 * hf + (lane & 7) + 16 * (lane >> 4)) * 8
                             : Wp + static_cast<size_t>(nt0) * KT * 512 + lane * 8;

  auto load = [&](bf16x8 (&wf)[NTW], bf16x8 (&xf)[MT], int kt) {
#pragma unroll
    for (int n = 0; n < NTW; ++n)
      wf[n] = __builtin_nontemporal_load(
          reinterpret_cast<const bf16x8*>(wbase + (static_cast<size_t>(n) * KT + kt) * 512));
#pragma unroll
    for (int m = 0; m < MT; ++m) xf[m] = *reinterpret_cast<const bf16x8*>(xrow[m] + kt * 32);
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
#pragma unroll
  for (int u = 0; u < R; ++u)
    if (kt_lo + u < kt_hi) load(wr[u], xr[u], kt_lo + u);
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
  if (wave != 0) return;
  if constexpr (HALF) {
    const int col = 16 * pair + 8 * hf + 4 * (lane >> 4);          // (lanes 0 .. 31: gate rows of the operand)
    const int gb = 32 * pair + 8 * hf + 4 * (lane >> 4);
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
    return;
  }
#pragma unroll
  for (int n = 0; n < NTW; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if constexpr (EPI == EPI_SWIGLU) {
        if (n & 1) continue;
        store_tile<EPI>(acc[n][m], &acc[(n + 1) % NTW][m], Y, bias, m * 16, (nt0 + n) * 16, M, N, ldy, lane, 0);
      } else {
        store_tile<EPI>(acc[n][m], nullptr, Y, bias, m * 16, (nt0 + n) * 16, M, N, ldy, lane, 0, ap, an);
      }
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
