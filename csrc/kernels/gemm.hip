// bf16 MFMA GEMMs for Y[M,N] = X[M,K] * W[N,K]^T on gfx950.
//
// Weights are stored pre-shuffled in MFMA-fragment order ("packed"):
//     Wp[((nt*KT + kt)*64 + lane)*8 + j] = W[nt*16 + (lane&15)][kt*32 + 8*(lane>>4) + j]
// so one wave-wide 16-byte load (or one global_load_lds_dwordx4) fetches exactly one
// 16(n) x 32(k) operand fragment as 1 KiB of contiguous memory, and the LDS image of
// a staged tile is lane-linear (conflict-free ds_read_b128, no swizzle needed).
//
// Orientation: the weight fragment is the MFMA A operand (rows = n) and the
// activation fragment the B operand (cols = m), i.e. the kernels compute Y^T tiles.
// A lane then owns 4 consecutive n of one row m: an 8-byte bf16 store.
//
// Kernels of this file:
//   * gemm_tile_kernel    -- 128x128x64 block tile, 4 waves (2x2), both operands staged
//     global->LDS with global_load_lds_dwordx4, double-buffered: outputs whose width is not
//     a multiple of 256 (tiny models); everything else goes to gemm256.hip / gemm_panel.hip.
//   * gemm_grouped_kernel -- the same tile per expert over ragged row groups (MoE).
//   * splitk_reduce_kernel -- sums the fp32 slabs of a split-K GEMM.
// Epilogues: bias add, bf16 or fp32 store, fused SwiGLU (gate/up n-tiles interleaved).
#include "gemm_common.h"

namespace {

// ---------------------------------------------------------------------------------
// Large-M kernel. Block tile 128(n) x 128(m) x 64(k); waves 2(n) x 2(m), 64x64 each.
// LDS per stage: W 8 n-tiles x 2 k-tiles x 1 KiB + X 8 m-tiles x 2 k-tiles x 1 KiB = 32 KiB.
// ---------------------------------------------------------------------------------
constexpr int GT_BN = 128, GT_BM = 128, GT_BK = 64;
constexpr int GT_STAGE_BYTES = 32 * 1024;

LC_DEVICE void gt_stage(char* stage, const bf16_t* __restrict__ Wp, const bf16_t* __restrict__ X,
                        int nt0, int m0, int m_hi, int kt0, int KT,
                        int K, int wave, int lane) {
  // 32 one-KiB pieces per stage, 8 per wave: pieces [0,16) are W, [16,32) are X.
  // X rows are clamped to m_hi-1 (tail tiles).
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int p = wave * 8 + i;
    char* dst = stage + p * 1024;  // wave-uniform; the DMA adds lane*16
    if (p < 16) {
      const int nt = p >> 1, kt = p & 1;
      const bf16_t* src = Wp + (static_cast<size_t>(nt0 + nt) * KT + (kt0 + kt)) * 512 + lane * 8;
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(src), LC_LDS_PTR(dst), 16, 0, 0);
    } else {
      const int q = p - 16;
      const int mt = q >> 1, kt = q & 1;
      int row = m0 + mt * 16 + (lane & 15);
      row = row < m_hi ? row : m_hi - 1;
      const bf16_t* src = X + static_cast<size_t>(row) * K + (kt0 + kt) * 32 + 8 * (lane >> 4);
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(src), LC_LDS_PTR(dst), 16, 0, 0);
    }
  }
}

template <int EPI>
__global__ __launch_bounds__(256) void gemm_tile_kernel(const bf16_t* __restrict__ Wp,
                                                        const bf16_t* __restrict__ X,
                                                        void* __restrict__ Y,
                                                        const bf16_t* __restrict__ bias, int M, int N,
                                                        int K, int ldy, int tiles_m, int tiles_n) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave >> 1, wm = wave & 1;

  // XCD-aware remap: blocks b and b+8 share an XCD; give each XCD a contiguous run of
  // tiles (bijective form for grids that are not a multiple of 8).
  const int nwg = tiles_m * tiles_n;
  const int orig = blockIdx.x;
  const int xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  // m fastest: consecutive tiles reuse the same 128-column weight panel from L2.
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int m0 = tm * GT_BM, nt0 = tn * (GT_BN / 16);
  const int KT = K / 32;
  const int nk = K / GT_BK;

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  gt_stage(smem, Wp, X, nt0, m0, M, 0, KT, K, wave, lane);
  __syncthreads();  // emits s_waitcnt vmcnt(0) for the LDS-DMA before the barrier

  for (int t = 0; t < nk; ++t) {
    char* cur = smem + (t & 1) * GT_STAGE_BYTES;
    if (t + 1 < nk)
      gt_stage(smem + ((t + 1) & 1) * GT_STAGE_BYTES, Wp, X, nt0, m0, M, (t + 1) * 2, KT, K, wave, lane);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      bf16x8 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(cur + ((wn * 4 + i) * 2 + kt) * 1024 + lane * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[j] = *reinterpret_cast<const bf16x8*>(cur + 16 * 1024 + ((wm * 4 + j) * 2 + kt) * 1024 + lane * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  const int nbase = tn * GT_BN + wn * 64, mbase = m0 + wm * 64;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (EPI == EPI_SWIGLU) {
        if (i & 1) continue;
        store_tile<EPI>(acc[i][j], &acc[i + 1][j], Y, bias, mbase + j * 16, nbase + i * 16, M, N, ldy, lane, 0);
      } else {
        store_tile<EPI>(acc[i][j], nullptr, Y, bias, mbase + j * 16, nbase + i * 16, M, N, ldy, lane, 0);
      }
    }
}


// ---------------------------------------------------------------------------------
// Grouped (MoE) products: rows [offsets[e], offsets[e+1]) of the expert-sorted activation matrix multiply expert e's packed
// weights. `row_index` (optional) gathers source rows, so the permutation of tokens into expert order never
// materialises a copy.
//
// Many small experts (a hundred or two rows each against a few MB of weights) are bound by the weights' way from HBM, and
// what has to be hidden is its latency: a tile's depth is only 8 to 32 K-tiles long. Block tile 128(n) x BM(m) x 64(k), a wave
// per 32 columns and 64 rows; both operands go through a ring of three LDS stages filled by LDS-DMA two K-tiles ahead, one barrier
// per K-tile, and the requests are never drained inside the loop. The two loops that were here before waited for every K-tile's
// requests at its end and fetched the activations as half lines.
//
// One MI355X, 32 experts of 512 x 2048 / 2048 x 512 (67 MB each way, 11 us at 6 TB/s), before and now: 6000 routed rows up 82 -> 29 us,
// down (fp32 out, 49 MB) 59 -> 33; 800 rows 63 -> 18 and 25 -> 15; 16384 rows 99 -> 40 and 114 -> 66.
// ---------------------------------------------------------------------------------
constexpr int GG_BN = 128, GG_BK = 64;

// Rows of a block tile, and stages of its ring (two workgroups a CU either way, 72 or 64 KiB). 64 rows (four waves) while the launch
// has a place on the CUs for every workgroup at once: the depth is a chain then, and shorter for small tiles (6000 rows up, 384
// workgroups: 29 us against 32). 128 rows (eight waves) beyond, where experts fill them: half as many readings of the weights
// (6000 rows down, 1536 workgroups of 64 rows: 39 us against 33; 8000 rows 51 and 36).
static inline int gg_rows(int rows, int E, int tiles_n) {
  const long long tiles = (static_cast<long long>(rows) + 64 * E - 1) / (64 * E) * E * tiles_n;
  return rows > 100ll * E && tiles > 512 ? 128 : 64;
}
constexpr int gg_stages(int bm) { return bm == 128 ? 2 : 3; }
constexpr int GG_W_BYTES = GG_BN * GG_BK * 2;

// Whose tile a block has: the experts' row tiles are numbered through all experts, n-tiles inside a row tile, and every XCD gets a
// contiguous run of them (blocks b and b + 8 share one), so that an expert's weights are read into one L2 and its
// rows as well. The lanes of a wave look at 64 experts at a time: a walk over the offsets is a chain of loads that costs more than
// the K-tiles of a small expert.
template <int BM>
LC_DEVICE bool gg_find(const int32_t* __restrict__ offsets, int E, int tiles_n, int lane, int& e, int& m0, int& m_hi, int& tn) {
  int used = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int x = e0 + lane;
    int n = x < E ? (offsets[x + 1] - offsets[x] + BM - 1) / BM : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    used += n;
  }
  const int nwg = __builtin_amdgcn_readfirstlane(used) * tiles_n, orig = blockIdx.x;
  if (orig >= nwg) return false;
  const int xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  int slot = tile / tiles_n;
  tn = tile % tiles_n;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int x = e0 + lane;
    const int lo = x < E ? offsets[x] : 0, hi = x < E ? offsets[x + 1] : 0;
    const int n = (hi - lo + BM - 1) / BM;
    int end = n;                                    // row tiles up to and including this expert's
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int before = __shfl_up(end, off, 64);
      if (lane >= off) end += before;
    }
    const uint64_t here = __ballot(end > slot);
    if (here != 0) {
      const int at = __builtin_ctzll(here);
      e = e0 + at;
      m0 = __builtin_amdgcn_readlane(lo, at) + (slot - (__builtin_amdgcn_readlane(end, at) - __builtin_amdgcn_readlane(n, at))) * BM;
      m_hi = __builtin_amdgcn_readlane(hi, at);
      return true;
    }
    slot -= __builtin_amdgcn_readlane(end, 63);
  }
  return false;
}

template <int EPI, int BM>
__global__ __launch_bounds__(BM * 4, 4) void gemm_grouped_kernel(const bf16_t* __restrict__ Wp_all, long long expert_stride,
                                                              const bf16_t* __restrict__ X, const int32_t* __restrict__ row_index,
                                                              const int32_t* __restrict__ offsets, int E, void* __restrict__ Y, int N,
                                                              int K, int ldy, int tiles_n, GluClamp glu) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int WAVES = BM / 16, NS = gg_stages(BM), STAGE = GG_W_BYTES + BM * 128, WPW = 16 / WAVES;       // KiB pieces of the weights per wave and K-tile
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 3, wm = wave >> 2;
  int e = 0, m0 = 0, m_hi = 0, tn = 0;
  if (!gg_find<BM>(offsets, E, tiles_n, lane, e, m0, m_hi, tn)) return;                 // block-uniform, before any barrier
  const int KT = K / 32, nk = K / GG_BK;

  // What this wave stages of a K-tile: WPW pieces of the weights (fragment f of the 16: n-tile f / 2, k-step f % 2) and two pieces
  // of eight whole 128-byte rows, swizzled on the source side as in gemm256.hip.
  const bf16_t* wsrc[WPW];
#pragma unroll
  for (int i = 0; i < WPW; ++i) {
    const int f = wave * WPW + i;
    wsrc[i] = Wp_all + static_cast<size_t>(e) * expert_stride + (static_cast<size_t>(tn * (GG_BN / 16) + (f >> 1)) * KT + (f & 1)) * 512 + lane * 8;
  }
  const bf16_t* xsrc[2];
  const int rr = lane >> 3, lc = lane & 7;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int row = m0 + (wave * 2 + i) * 8 + rr;
    row = row < m_hi ? row : m_hi - 1;
    if (row_index) row = row_index[row];
    xsrc[i] = X + static_cast<size_t>(row) * K + ((lc ^ rr) << 3);
  }
  auto request = [&](int kt) {                      // K-tile kt into its stage (behind the last one: the last one again)
    char* stage = smem + (kt % NS) * STAGE;
    const int k = kt < nk ? kt : nk - 1;
#pragma unroll
    for (int i = 0; i < WPW; ++i)
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(wsrc[i] + static_cast<size_t>(k) * 1024), LC_LDS_PTR(stage + (wave * WPW + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(xsrc[i] + k * GG_BK), LC_LDS_PTR(stage + GG_W_BYTES + (wave * 2 + i) * 1024), 16, 0, 0);
  };

  f32x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r7 = lane & 7;
  int xoff[2];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) xoff[kt] = ((lane & 15) >> 3) * 1024 + r7 * 128 + (((kt * 4 + (lane >> 4)) ^ r7) << 4);

#pragma unroll
  for (int t = 0; t + 1 < NS; ++t) request(t);
  for (int t = 0; t < nk; ++t) {
    // all but the requests of K-tile t + 1 have landed; behind the barrier everyone's have, and nobody reads K-tile t - 1 any more
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * (WPW + 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    request(t + NS - 1);
    const char* w = smem + (t % NS) * STAGE + wn * 4096 + lane * 16;
    const char* x = smem + (t % NS) * STAGE + GG_W_BYTES + wm * 8192;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      bf16x8 a[2], b[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(w + (i * 2 + kt) * 1024);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8*>(x + j * 2048 + xoff[kt]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // this wave's reads are over before it lets the stage be written again
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // (requests behind the last K-tile)

  const int nbase = tn * GG_BN + wn * 32, mbase = m0 + wm * 64;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (EPI == EPI_GLU_CLAMPED) {
      store_tile_glu_clamped(acc[0][j], acc[1][j], Y, glu, mbase + j * 16, nbase, m_hi, N, ldy, lane);
    } else if constexpr (EPI == EPI_SWIGLU) {
      store_tile<EPI>(acc[0][j], &acc[1][j], Y, nullptr, mbase + j * 16, nbase, m_hi, N, ldy, lane, 0);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) store_tile<EPI>(acc[i][j], nullptr, Y, nullptr, mbase + j * 16, nbase + i * 16, m_hi, N, ldy, lane, 0);
    }
  }
}

// Sums S fp32 slabs [S, M, N] (+bias) and writes bf16 (mode 0), fp32 (mode 1) or
// SwiGLU over gate/up n-tiles interleaved at 16 columns (mode 2, out [M, N/2]).
__global__ void splitk_reduce_kernel(const float* __restrict__ part, const bf16_t* __restrict__ bias,
                                     void* __restrict__ Y, int S, int M, int N, int ldy, int mode) {
  const size_t total4 = static_cast<size_t>(M) * (N / 4);
  const size_t slab = static_cast<size_t>(M) * N;
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total4;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t m = i / (N / 4);
    const int n = static_cast<int>(i % (N / 4)) * 4;
    f32x4 v = *reinterpret_cast<const f32x4*>(part + m * N + n);
#pragma unroll 8
    for (int s = 1; s < S; ++s) {                    // (several slabs in flight)
      const f32x4 p = *reinterpret_cast<const f32x4*>(part + s * slab + m * N + n);
      v += p;
    }
    if (bias)
      for (int r = 0; r < 4; ++r) v[r] += bf16_to_f32(bias[n + r]);
    if (mode == 0) {
      u32x2 o;
      o[0] = pack_bf16x2(v[0], v[1]);
      o[1] = pack_bf16x2(v[2], v[3]);
      *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(Y) + m * ldy + n) = o;
    } else if (mode == 1) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(Y) + m * ldy + n) = v;
    } else {
      // gate tile = even 16-column tile, up tile = the next one
      const int tile = n >> 4;
      if (tile & 1) continue;
      f32x4 u = *reinterpret_cast<const f32x4*>(part + m * N + n + 16);
      for (int s = 1; s < S; ++s) u += *reinterpret_cast<const f32x4*>(part + s * slab + m * N + n + 16);
      if (bias)
        for (int r = 0; r < 4; ++r) u[r] += bf16_to_f32(bias[n + 16 + r]);
      u32x2 o;
      o[0] = pack_bf16x2(silu(v[0]) * u[0], silu(v[1]) * u[1]);
      o[1] = pack_bf16x2(silu(v[2]) * u[2], silu(v[3]) * u[3]);
      *reinterpret_cast<u32x2*>(static_cast<bf16_t*>(Y) + m * ldy + (tile >> 1) * 16 + (n & 15)) = o;
    }
  }
}

// The same for widths that are no whole groups of 32 columns: one element per thread, bf16 or fp32.
__global__ void splitk_reduce_any_kernel(const float* __restrict__ part, const bf16_t* __restrict__ bias, void* __restrict__ Y, int S,
                                         int M, int N, int ldy, int f32) {
  const size_t slab = static_cast<size_t>(M) * N;
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < slab; i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t m = i / N;
    const int n = static_cast<int>(i - m * N);
    float v = part[i];
    for (int s = 1; s < S; ++s) v += part[s * slab + i];
    if (bias) v += bf16_to_f32(bias[n]);
    if (f32) static_cast<float*>(Y)[m * ldy + n] = v;
    else static_cast<bf16_t*>(Y)[m * ldy + n] = f32_to_bf16(v);
  }
}

}  // namespace

// Y = X * W^T with a 128x128 tile. Requirements: K % 64 == 0, n_pad % 128 == 0 (the
// packed weight buffer holds n_pad/16 n-tiles; rows >= N are zero), ldy = row stride of Y.
LC_EXPORT int lc_gemm_tile(const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K,
                           int n_pad, int ldy, int epi, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K % 64 || n_pad % 128 || N > n_pad) return -1;
  const int tiles_m = (M + GT_BM - 1) / GT_BM, tiles_n = n_pad / GT_BN;
  const dim3 grid(tiles_m * tiles_n), block(256);
  const size_t lds = 2 * GT_STAGE_BYTES;
  auto w = static_cast<const bf16_t*>(Wp);
  auto x = static_cast<const bf16_t*>(X);
  auto b = static_cast<const bf16_t*>(bias);
  if (epi == EPI_BF16)
    gemm_tile_kernel<EPI_BF16><<<grid, block, lds, stream>>>(w, x, Y, b, M, N, K, ldy, tiles_m, tiles_n);
  else if (epi == EPI_F32)
    gemm_tile_kernel<EPI_F32><<<grid, block, lds, stream>>>(w, x, Y, b, M, N, K, ldy, tiles_m, tiles_n);
  else if (epi == EPI_SWIGLU)
    gemm_tile_kernel<EPI_SWIGLU><<<grid, block, lds, stream>>>(w, x, Y, b, M, N, K, ldy, tiles_m, tiles_n);
  else
    return -2;
  LC_RETURN_LAST_ERROR();
}

LC_EXPORT int lc_splitk_reduce(const void* part, const void* bias, void* Y, int S, int M, int N, int ldy,
                               int mode, hipStream_t stream) {
  if (M <= 0) return 0;
  if (N <= 0 || S <= 0 || (N % 32 && mode == 2)) return -1;
  const size_t items = static_cast<size_t>(M) * (N % 32 ? N : N / 4);
  const int grid = static_cast<int>(std::min<size_t>((items + 255) / 256, 2048));
  if (N % 32) {
    splitk_reduce_any_kernel<<<dim3(grid), dim3(256), 0, stream>>>(static_cast<const float*>(part), static_cast<const bf16_t*>(bias), Y, S, M,
                                                                   N, ldy, mode);
    LC_RETURN_LAST_ERROR();
  }
  splitk_reduce_kernel<<<dim3(grid), dim3(256), 0, stream>>>(static_cast<const float*>(part),
                                                             static_cast<const bf16_t*>(bias), Y, S, M, N,
                                                             ldy, mode);
  LC_RETURN_LAST_ERROR();
}

// Grouped GEMM over E experts. offsets (device, int32 [E+1]) delimit each expert's rows
// in the expert-sorted order; total_rows bounds the launch (tiles beyond the used ones
// exit immediately). Output rows are in sorted order.
static int launch_gemm_grouped(const void* Wp_all, long long expert_stride, const void* X, const void* row_index,
                               const void* offsets, int E, void* Y, int total_rows, int N, int K, int n_pad, int ldy,
                               int epi, GluClamp glu, hipStream_t stream) {
  if (total_rows <= 0) return 0;
  if (K % 64 || n_pad % 128 || N > n_pad || E < 1) return -1;
  const int tiles_n = n_pad / GG_BN, bm = gg_rows(total_rows, E, tiles_n);
  const int max_tiles_m = (total_rows + bm - 1) / bm + E;
  const dim3 grid(max_tiles_m * tiles_n), block(bm * 4);
  const size_t lds = gg_stages(bm) * (GG_W_BYTES + bm * 128);
  auto w = static_cast<const bf16_t*>(Wp_all);
  auto x = static_cast<const bf16_t*>(X);
  auto ri = static_cast<const int32_t*>(row_index);
  auto off = static_cast<const int32_t*>(offsets);
#define LC_GG(EPI_)                                                                                                                     \
  do {                                                                                                                                  \
    static LcDeviceOnce once;                                                                                                           \
    once.run([&] {                                                                                                                      \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_grouped_kernel<EPI_, 64>), hipFuncAttributeMaxDynamicSharedMemorySize, \
                                gg_stages(64) * (GG_W_BYTES + 64 * 128));                                                                       \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_grouped_kernel<EPI_, 128>), hipFuncAttributeMaxDynamicSharedMemorySize, \
                                gg_stages(128) * (GG_W_BYTES + 128 * 128));                                                                      \
    });                                                                                                                                 \
    if (bm == 128) gemm_grouped_kernel<EPI_, 128><<<grid, block, lds, stream>>>(w, expert_stride, x, ri, off, E, Y, N, K, ldy, tiles_n, glu); \
    else gemm_grouped_kernel<EPI_, 64><<<grid, block, lds, stream>>>(w, expert_stride, x, ri, off, E, Y, N, K, ldy, tiles_n, glu);      \
  } while (0)
  if (epi == EPI_BF16) LC_GG(EPI_BF16);
  else if (epi == EPI_SWIGLU) LC_GG(EPI_SWIGLU);
  else if (epi == EPI_RELU2) LC_GG(EPI_RELU2);
  else if (epi == EPI_F32) LC_GG(EPI_F32);
  else if (epi == EPI_GLU_CLAMPED) LC_GG(EPI_GLU_CLAMPED);
  else return -2;
#undef LC_GG
  LC_RETURN_LAST_ERROR();
}

LC_EXPORT int lc_gemm_grouped(const void* Wp_all, long long expert_stride, const void* X,
                              const void* row_index, const void* offsets, int E, void* Y, int total_rows,
                              int N, int K, int n_pad, int ldy, int epi, hipStream_t stream) {
  if (epi == EPI_GLU_CLAMPED) return -2;
  return launch_gemm_grouped(Wp_all, expert_stride, X, row_index, offsets, E, Y, total_rows, N, K, n_pad, ldy, epi,
                             GluClamp{nullptr, 0.f, 0.f, 0.f}, stream);
}

// The gate | up product of clamped gated experts (n-tiles alternate gate / up): Y bf16 [rows, N / 2] is the gated
// unit of the product scaled by row_scale[sorted position] (fp32, may be null).
LC_EXPORT int lc_gemm_grouped_glu(const void* Wp_all, long long expert_stride, const void* X, const void* row_index,
                                  const void* offsets, int E, void* Y, int total_rows, int N, int K, int n_pad, int ldy,
                                  const void* row_scale, float limit, float slope, float shift, hipStream_t stream) {
  if (N % 32) return -1;
  return launch_gemm_grouped(Wp_all, expert_stride, X, row_index, offsets, E, Y, total_rows, N, K, n_pad, ldy,
                             EPI_GLU_CLAMPED, GluClamp{static_cast<const float*>(row_scale), limit, slope, shift}, stream);
}
