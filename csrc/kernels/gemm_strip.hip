// Products of up to 64 rows in one launch, whose result may pass through an activation: Y[M, .] = act(X[M, K] * W[N, K]^T).
//
// The panel kernel (gemm_panel.hip) gives a workgroup 128 columns. An output of up to 16384 columns then fills the CUs only with
// its depth split over workgroups, and the activation (or a plain result) needs another launch that adds up the fp32 slabs. Here a workgroup has
// 32 or 64 columns over the whole depth (as many as it takes for 128 to 256 workgroups), so that the activation of a
// column, or of the gate and up tiles next to each other, is applied to the accumulators.
//
// What bounds it is the way of the weights from HBM, each read once. Four waves fill a ring of LDS stages by LDS-DMA, a stage being
// one 64-deep K-tile of the weights and of the activation panel (BM = 32 or 64 rows, rows behind M repeat the last one):
//
//     columns   BM   stage            stages
//          64   32   8 + 4 KiB        6
//          64   64   8 + 8 KiB        4
//          32   32   4 + 4 KiB        6
//          32   64   4 + 8 KiB        6
//
// Rings of twice that depth, one workgroup per CU, are slower (16384 x 2048 at 32 rows 15.1 us against 13.4, 8192 x 1024 8.0 and 6.0), and a
// second workgroup finds room beside this one. With 64 columns a wave has two column tiles and half the rows, with 32
// columns half the rows and one of the two k-steps of every K-tile; the two halves of the sum meet in the LDS at the end.
// Operand conventions as in gemm_panel.hip.
//
// A plain fp32 product may come in parts of the depth (blockIdx.y), one slab each: with a quarter of a panel's columns and four times its
// depth a workgroup reads as many weights and leaves a quarter of the slabs (ops._strip_splits).
//
// One MI355X, weights from HBM (16384 x 2048: 10.3 us at 6.5 TB/s), split product and activation before, and now: gated 16384 x 2048 at
// 8, 32, 64 rows 15.6, 20.1, 21.4 us -> 13.3, 13.4, 14.3; relu^2 8192 x 2048 at 32 rows 13.6 -> 8.7.
#include "gemm_common.h"

namespace {

constexpr int GS_BK = 64, GS_NT = 2;                 // (non-temporal weights: every byte is read once, see gemm_panel.hip)

template <int NTB, int BM>
struct StripShape {
  static constexpr int WBYTES = NTB * 2048, STAGE = WBYTES + BM * 128;
  static constexpr int NSTAGE = NTB == 4 && BM == 64 ? 4 : 6, DEPTH = NSTAGE - 1;
  static constexpr int WP = NTB / 2, XP = BM / 32, P = WP + XP;      // DMA instructions per wave and K-tile
  static constexpr int MT_W = BM / 32;                               // row tiles of a wave
};

// Waits until all but the newest ``tiles`` K-tiles' requests (P each) have landed.
template <int P, int T>
LC_DEVICE void gs_wait(int tiles) {
  if constexpr (T == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (tiles >= T) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * T) : "memory");
    else gs_wait<P, T - 1>(tiles);
  }
}

template <int NTB, int BM, int EPI>
__global__ __launch_bounds__(256) void gemm_strip_kernel(const bf16_t* __restrict__ Wp, const bf16_t* __restrict__ X,
                                                         void* __restrict__ Y, const bf16_t* __restrict__ bias, int M, int N, int K,
                                                         int ldy, float ap, float an) {
  using S = StripShape<NTB, BM>;
  static_assert(S::P * S::DEPTH <= 63, "vmcnt is a 6-bit counter");
  static_assert(NTB == 2 || NTB == 4, "two column tiles per wave");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt0 = static_cast<int>(blockIdx.x) * NTB, KT = K / 32;
  const int nk = K / GS_BK / static_cast<int>(gridDim.y), kt0 = static_cast<int>(blockIdx.y) * nk;   // this workgroup's K-tiles

  // KiB piece q * 4 + wave of a stage: the weights' fragments (n-tile, k-step), then eight rows of 128 bytes each, swizzled on the source side
  const bf16_t* wsrc[S::WP];
#pragma unroll
  for (int q = 0; q < S::WP; ++q) {
    const int f = q * 4 + wave;
    wsrc[q] = Wp + (static_cast<size_t>(nt0 + (f >> 1)) * KT + 2 * kt0 + (f & 1)) * 512 + lane * 8;
  }
  const bf16_t* xsrc[S::XP];
  const int rr = lane >> 3, lc = lane & 7;
#pragma unroll
  for (int q = 0; q < S::XP; ++q) {
    int row = (q * 4 + wave) * 8 + rr;
    row = row < M ? row : M - 1;
    xsrc[q] = X + static_cast<size_t>(row) * K + kt0 * GS_BK + ((lc ^ rr) << 3);
  }
  auto issue = [&](int t) {
    if (t >= nk) return;
    char* stage = smem + (t % S::NSTAGE) * S::STAGE;
#pragma unroll
    for (int q = 0; q < S::WP; ++q)
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(wsrc[q] + static_cast<size_t>(t) * 1024), LC_LDS_PTR(stage + (q * 4 + wave) * 1024), 16, 0, GS_NT);
#pragma unroll
    for (int q = 0; q < S::XP; ++q)
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(xsrc[q] + t * GS_BK), LC_LDS_PTR(stage + S::WBYTES + (q * 4 + wave) * 1024), 16, 0, 0);
  };

  const int wp = NTB == 4 ? (wave & 1) * 2 : 0;            // first column tile of this wave
  const int mt0 = (NTB == 4 ? wave >> 1 : wave & 1) * S::MT_W;
  const int ks = wave >> 1;                                // NTB == 2: this wave's k-step
  const int r7 = lane & 7;
  f32x4 acc[2][S::MT_W];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < S::MT_W; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int t = 0; t < S::DEPTH; ++t) issue(t);
  for (int t = 0; t < nk; ++t) {
    gs_wait<S::P, S::DEPTH - 1>(nk - 1 - t);
    __builtin_amdgcn_s_barrier();                          // K-tile t is there for everybody, and nobody reads K-tile t - 1 any more
    asm volatile("" ::: "memory");
    issue(t + S::DEPTH);
    const char* stage = smem + (t % S::NSTAGE) * S::STAGE;
    const char* wimg = stage + wp * 2048 + lane * 16;
    const char* ximg = stage + S::WBYTES + mt0 * 2048 + ((lane & 15) >> 3) * 1024 + r7 * 128;
#pragma unroll
    for (int k = 0; k < (NTB == 4 ? 2 : 1); ++k) {
      const int kt = NTB == 4 ? k : ks;
      bf16x8 a[2], b[S::MT_W];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(wimg + (i * 2 + kt) * 1024);
#pragma unroll
      for (int j = 0; j < S::MT_W; ++j) b[j] = *reinterpret_cast<const bf16x8*>(ximg + j * 2048 + (((kt * 4 + (lane >> 4)) ^ r7) << 4));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < S::MT_W; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // this wave's reads are over before the stage may be written again
  }
  if constexpr (NTB == 2) {                                // the odd k-steps' half of the sum joins the even ones'
    f32x4* half = reinterpret_cast<f32x4*>(smem) + (wave & 1) * (2 * S::MT_W * 64) + lane;
    __syncthreads();
    if (ks == 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < S::MT_W; ++j) half[(i * S::MT_W + j) * 64] = acc[i][j];
    }
    __syncthreads();
    if (ks == 1) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < S::MT_W; ++j) acc[i][j] += half[(i * S::MT_W + j) * 64];
  }
  const int nbase = (nt0 + wp) * 16;
#pragma unroll
  for (int j = 0; j < S::MT_W; ++j) {
    const int m0 = (mt0 + j) * 16;
    if constexpr (epi_gated(EPI)) {
      store_tile<EPI>(acc[0][j], &acc[1][j], Y, bias, m0, nbase, M, N, ldy, lane, 0);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) store_tile<EPI>(acc[i][j], nullptr, Y, bias, m0, nbase + i * 16, M, N, ldy, lane, EPI == EPI_F32 ? static_cast<size_t>(blockIdx.y) * M * ldy : 0, ap, an);
    }
  }
}

template <int NTB, int BM>
int launch_strip(int epi, const bf16_t* w, const bf16_t* x, void* Y, const bf16_t* b, int M, int N, int K, int n_pad, int ldy, float ap, float an,
                 int splits, hipStream_t stream) {
  using S = StripShape<NTB, BM>;
  constexpr int lds = S::NSTAGE * S::STAGE;
  const dim3 grid(n_pad / (16 * NTB), splits), block(256);
#define GS_CASE(E)                                                                                                                     \
  case E: {                                                                                                                            \
    static LcDeviceOnce once;                                                                                                          \
    once.run([&] {                                                                                                                     \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_strip_kernel<NTB, BM, E>),                                    \
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);                                                      \
    });                                                                                                                                \
    gemm_strip_kernel<NTB, BM, E><<<grid, block, lds, stream>>>(w, x, Y, b, M, N, K, ldy, ap, an);                               \
    break;                                                                                                                             \
  }
  switch (epi) {
    GS_CASE(EPI_BF16)
    GS_CASE(EPI_F32)
    GS_CASE(EPI_SWIGLU)
    GS_CASE(EPI_GEGLU)
    GS_CASE(EPI_REGLU)
    GS_CASE(EPI_RELU2)
    GS_CASE(EPI_XIELU)
    default: return -2;
  }
#undef GS_CASE
  return static_cast<int>(hipGetLastError());
}

}  // namespace

// Y = act(X * W^T + bias) of 1 to 64 rows, in bf16, or plain in fp32 (the gated epilogues without a bias read n-tiles that alternate gate / up). ``tiles``: column
// tiles of 16 per workgroup, 2 or 4. ``splits`` > 1 (fp32, no bias): Y is [splits, M, ldy], the sums of as many parts of the depth. Requirements: K % 64 == 0, n_pad % 64 == 0.
LC_EXPORT int lc_gemm_strip(const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K, int n_pad, int ldy, int epi, int tiles,
                            float ap, float an, int splits, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 64 || K <= 0 || K % 64 || n_pad % 64 || N > n_pad || N <= 0 || (tiles != 2 && tiles != 4)) return -1;
  if (epi_gated(epi) && N % 32) return -1;
  if (splits < 1 || (K / GS_BK) % splits || (splits > 1 && (epi != EPI_F32 || bias != nullptr))) return -1;
  auto w = static_cast<const bf16_t*>(Wp);
  auto x = static_cast<const bf16_t*>(X);
  auto b = static_cast<const bf16_t*>(bias);
#define GS_GO(T, B) launch_strip<T, B>(epi, w, x, Y, b, M, N, K, n_pad, ldy, ap, an, splits, stream)
  if (tiles == 4) return M <= 32 ? GS_GO(4, 32) : GS_GO(4, 64);
  return M <= 32 ? GS_GO(2, 32) : GS_GO(2, 64);
#undef GS_GO
}
