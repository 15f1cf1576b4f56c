// Large-M bf16 GEMM, 256(n) x 128..256(m) x 64(k) block tile, 8 waves, requests that stay in flight
// across barriers (counted s_waitcnt vmcnt, raw s_barrier).
//
// Same operand conventions as gemm.hip: packed weights (MFMA-fragment order) are the MFMA A
// operand, activations the B operand. Wave (wn = w&3, wm = w>>2) owns 64 n x 16 MF m of the tile =
// 4 x MF accumulator fragments. Each phase of a K-tile is
//     R (fragment reads, requests, waits) | barrier | M (MFMAs) | barrier
// and waves 4-7 run one barrier behind waves 0-3, so on every SIMD one wave is in M while its
// partner is in R. The request queue is never drained inside the loop. Weights come straight from
// global memory into registers (they are stored as fragments), one K-tile ahead; activations through
// three LDS stages filled by LDS-DMA as whole 128-byte rows in an XOR-swizzled image. Described at the loop.
//
// MF (8, 7, 6, 5, 4: tiles of 256 to 128 rows) is chosen by the caller so that the tiles fill whole
// rounds of the 256 CUs (ops.gemm256_plan, where the times of the heights stand).
#include "gemm_common.h"

namespace {

constexpr int G2_BN = 256, G2_BK = 64;
constexpr int G2_BAND = 4;

// Rows of a tile, and its LDS: three activation stages of 128 bytes a row; the epilogue stages the output tile through the same
// memory, all of its 256 columns in bf16 or half of its rows in fp32.
constexpr int g2_rows(int mf) { return 32 * mf; }
constexpr int g2_lds(int mf) { return (mf + 1) / 2 * 32 * 1024; }

struct G2Ctx {
  const bf16_t* __restrict__ Wp;
  const bf16_t* __restrict__ X;
  char* smem;
  int nt0, m0, M, K, KT, nk, wave, lane;
  int kt_lo = 0;   // first K-tile of this block's K split
};

// Byte offset, inside one m-tile's 2-KiB image, of this lane's B fragment for k-tile kt.
LC_DEVICE int g2_x_off(int kt, int lane) {
  const int r = lane & 15, rr = r & 7;
  return (r >> 3) * 1024 + rr * 128 + (((kt * 4 + (lane >> 4)) ^ rr) << 4);
}

// MFMAs of one k-step: all four n-fragments against all MF m-fragments.
#define G2_MFMA_STEP(AFR, BFR)                                                                        \
  do {                                                                                                \
    __builtin_amdgcn_s_setprio(1);                                                                    \
    _Pragma("unroll") for (int jh = 0; jh < MF; jh += 4)                                              \
      _Pragma("unroll") for (int i = 0; i < 4; ++i)                                                   \
        _Pragma("unroll") for (int j = jh; j < (jh + 4 < MF ? jh + 4 : MF); ++j)                      \
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(AFR[i], BFR[j], acc[i][j], 0, 0, 0);     \
    __builtin_amdgcn_s_setprio(0);                                                                    \
  } while (0)

#define G2_BARRIER()                         \
  do {                                       \
    asm volatile("" ::: "memory");           \
    __builtin_amdgcn_s_barrier();            \
    asm volatile("" ::: "memory");           \
  } while (0)

// GROUPED: the rows are the expert-sorted token list of a MoE layer; expert e owns rows
// offsets[e] .. offsets[e+1] and the weights at Wp + e * expert_stride. m-tiles are numbered
// through all experts (tiles_m is an upper bound: total_rows / rows of a tile + E); a block walks the E+1
// offsets to find its expert and leaves if its m-tile is past the last one in use.
template <int EPI, bool GROUPED = false, int MF = 8>
__global__ __launch_bounds__(512) void gemm256_kernel(const bf16_t* __restrict__ Wp,
                                                      const bf16_t* __restrict__ X, void* __restrict__ Y,
                                                      const bf16_t* __restrict__ bias, int M, int N, int K,
                                                      int ldy, int tiles_m, int tiles_n,
                                                      long long expert_stride = 0,
                                                      const int32_t* __restrict__ offsets = nullptr, int E = 0,
                                                      int nk_per_split = 0, float ap = 0.f, float an = 0.f) {
  constexpr int G2_BM = g2_rows(MF);
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 3, wm = wave >> 2;

  // XCD-aware remap (blocks b and b+8 share an XCD): each XCD gets a contiguous run of tiles.
  const int nwg = tiles_m * tiles_n;
  const int orig = blockIdx.x;
  const int xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  // Tiles are ordered in bands of G2_BAND n-tiles, n fastest inside a band: the ~32 tiles an
  // XCD runs at once then form an 8(m) x 4(n) patch that shares 8 activation and 4 weight
  // panels through that XCD's L2 instead of streaming 32 different activation panels.
  const int band = tile / (G2_BAND * tiles_m), idx = tile % (G2_BAND * tiles_m);
  const int bw = min(G2_BAND, tiles_n - band * G2_BAND);
  const int tn = band * G2_BAND + idx % bw, tm = idx / bw;

  int m0 = tm * G2_BM;
  if constexpr (GROUPED) {
    int gm = tm, e = 0, lo = 0, hi = 0;
    bool found = false;
    for (e = 0; e < E; ++e) {
      lo = offsets[e];
      hi = offsets[e + 1];
      const int nt = (hi - lo + G2_BM - 1) / G2_BM;
      if (gm < nt) {
        found = true;
        break;
      }
      gm -= nt;
    }
    if (!found) return;                      // block-uniform, before any barrier
    Wp += static_cast<size_t>(e) * expert_stride;
    m0 = lo + gm * G2_BM;
    M = hi;                                  // rows of this expert end here (absolute row index)
  }
  G2Ctx c{Wp, X, smem, tn * (G2_BN / 16), m0, M, K, K / 32, K / G2_BK, wave, lane};
  if (nk_per_split > 0) {   // split-K (blockIdx.y): fp32 slabs, summed by the consumer or by lc_splitk_reduce
    c.nk = nk_per_split;
    c.kt_lo = static_cast<int>(blockIdx.y) * nk_per_split;
  }

  f32x4 acc[4][MF];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The WEIGHT fragments never pass through LDS: the packed weights are stored as ready-made MFMA
  // fragments, so a wave loads its own four n-fragments of one k-step (32 deep) straight from global
  // memory into registers (one coalesced KiB per instruction), one K-tile ahead, double-buffered. LDS
  // carries the activations only (three stages; X of K-tile t+2 is requested in K-tile t into the stage
  // K-tile t-1 used): at 256 rows 128 KiB of fragment reads and 32 KiB of LDS-DMA writes per K-tile and CU
  // instead of 192 + 64. That matters because the LDS traffic of one wave slows the MFMAs of its SIMD
  // partner. Every request is issued unconditionally (indices are clamped at the end of K) so that the
  // number of memory operations between a request and its first use is the same on every path, and all
  // waits are counted by hand: left to the compiler, every wait for a register load becomes vmcnt(0),
  // because it treats a pending global_load ... lds as a FLAT access whose return order is unknown.
  //
  // A slot between two barriers carries ~75 cycles of barrier and hand-over cost on top of its MFMAs.
  // Tiles of up to 192 rows hold the activation fragments of both k-steps, so a K-tile is one phase of
  // 8 MF MFMAs; the taller ones (256 registers are all that two waves per SIMD leave) take two phases,
  // one per k-step. Every accumulator receives k0 before k1 of each K-tile in both forms.
  constexpr bool ONE = MF <= 6;
  constexpr int PP = (MF + 1) / 2;        // 8-row pieces of X a wave moves per K-tile; an odd MF repeats half of the last
  constexpr int PA = (PP + 1) / 2, PB = PP - PA;
  constexpr int XSTAGE = g2_rows(MF) * 128;
  bf16x8 A0[2][4], A1[2][4], bX[ONE ? 2 : 1][MF];
  const int xoff0 = g2_x_off(0, lane), xoff1 = g2_x_off(1, lane);
  const bf16_t* wbase = c.Wp + (static_cast<size_t>(c.nt0 + wn * 4) * c.KT + c.kt_lo * 2) * 512 + lane * 8;
  const size_t wnt = static_cast<size_t>(c.KT) * 512;      // elements between consecutive n-tiles
  // register loads from inline assembly: the compiler neither waits for them nor moves them
  auto wfrag = [&](int i, int kidx) -> bf16x8 {            // fragment of n-tile i, 32-deep k index kidx
    bf16x8 v;
    const bf16_t* ptr = wbase + i * wnt + static_cast<size_t>(kidx) * 512;
    asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(v) : "v"(ptr) : "memory");
    return v;
  };
  auto xissue = [&](int k_tile, int p, int xs) {           // this wave's piece p (8 rows) of K-tile k_tile into stage xs
    const int kk = k_tile < c.nk ? k_tile : c.nk - 1;
    int piece = p * 8 + wave;
    if (PP * 8 > 4 * MF && piece >= 4 * MF) piece -= 8;    // (past the tile: the wave's piece before, once more)
    const int rr = lane >> 3, lc = lane & 7;
    int row = c.m0 + piece * 8 + rr;
    row = row < c.M ? row : c.M - 1;
    const int koff = (c.kt_lo + kk) * G2_BK + ((lc ^ rr) << 3);
    __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(c.X + static_cast<size_t>(row) * c.K + koff),
                                     LC_LDS_PTR(smem + xs * XSTAGE + piece * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int p = 0; p < PP; ++p) xissue(0, p, 0);
#pragma unroll
  for (int p = 0; p < PP; ++p) xissue(1, p, 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    A0[0][i] = wfrag(i, 0);
    A1[0][i] = wfrag(i, 1);
  }
  // Everything: the first K-tile consumes the weight fragments requested last. With X(1) in
  // front of them, the counted waits of the loop hold from its first K-tile on.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  if (wave >= 4) G2_BARRIER();
  int xs = 0;
#define G2_KTILE(T, CUR, NXT)                                                                           \
  do {                                                                                                  \
    const int t_ = (T);                                                                                 \
    const char* ximg = smem + xs * XSTAGE + (wm * MF * 2) * 1024;                                       \
    const int xs2 = xs == 0 ? 2 : xs - 1;                                                               \
    const int kn = (t_ + 1 < c.nk ? t_ + 1 : c.nk - 1) * 2;                                             \
    if constexpr (ONE) {                                                                                \
      _Pragma("unroll") for (int j = 0; j < MF; ++j)                                                    \
        bX[0][j] = *reinterpret_cast<const bf16x8*>(ximg + j * 2048 + xoff0);                           \
      _Pragma("unroll") for (int j = 0; j < MF; ++j)                                                    \
        bX[ONE ? 1 : 0][j] = *reinterpret_cast<const bf16x8*>(ximg + j * 2048 + xoff1);                 \
      _Pragma("unroll") for (int i = 0; i < 4; ++i) A0[NXT][i] = wfrag(i, kn);                          \
      _Pragma("unroll") for (int i = 0; i < 4; ++i) A1[NXT][i] = wfrag(i, kn + 1);                      \
      _Pragma("unroll") for (int p = 0; p < PP; ++p) xissue(t_ + 2, p, xs2);                            \
      /* X(t+1): the last requests of K-tile t-1, 8 + PP operations ago; A[CUR] came before them */     \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 + PP) : "memory");                          \
      G2_BARRIER();                                                                                     \
      G2_MFMA_STEP(A0[CUR], bX[0]);                                                                     \
      G2_MFMA_STEP(A1[CUR], bX[ONE ? 1 : 0]);                                                           \
      G2_BARRIER();                                                                                     \
    } else {                                                                                            \
      /* P1 (k0, all m) */                                                                              \
      _Pragma("unroll") for (int j = 0; j < MF; ++j)                                                    \
        bX[0][j] = *reinterpret_cast<const bf16x8*>(ximg + j * 2048 + xoff0);                           \
      _Pragma("unroll") for (int i = 0; i < 4; ++i) A0[NXT][i] = wfrag(i, kn);                          \
      _Pragma("unroll") for (int p = 0; p < PA; ++p) xissue(t_ + 2, p, xs2);                            \
      /* A0[CUR]: requested at the start of P1 of K-tile t-1, PA + (4 + PB) + (4 + PA) operations ago */ \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 + 2 * PA + PB) : "memory");                 \
      G2_BARRIER();                                                                                     \
      G2_MFMA_STEP(A0[CUR], bX[0]);                                                                     \
      G2_BARRIER();                                                                                     \
      /* P2 (k1, all m) */                                                                              \
      _Pragma("unroll") for (int j = 0; j < MF; ++j)                                                    \
        bX[0][j] = *reinterpret_cast<const bf16x8*>(ximg + j * 2048 + xoff1);                           \
      _Pragma("unroll") for (int i = 0; i < 4; ++i) A1[NXT][i] = wfrag(i, kn + 1);                      \
      _Pragma("unroll") for (int p = PA; p < PP; ++p) xissue(t_ + 2, p, xs2);                           \
      /* X(t+1): the last requests of P2 of K-tile t-1, (4 + PA) + (4 + PB) operations ago; A1[CUR] */  \
      /* came before them                                                                          */   \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 + PA + PB) : "memory");                     \
      G2_BARRIER();                                                                                     \
      G2_MFMA_STEP(A1[CUR], bX[0]);                                                                     \
      G2_BARRIER();                                                                                     \
    }                                                                                                   \
    xs = xs == 2 ? 0 : xs + 1;                                                                          \
  } while (0)
  int t = 0;
  for (; t + 1 < c.nk; t += 2) {
    G2_KTILE(t, 0, 1);
    G2_KTILE(t + 1, 1, 0);
  }
  if (t < c.nk) G2_KTILE(t, 0, 1);                         // odd number of K-tiles
#undef G2_KTILE
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the clamped requests of the last K-tiles
  // The last K-tile's register loads are never consumed. Their destination registers must still
  // belong to them until the wait above: a register the compiler considered free would be handed
  // to another value and then overwritten when the load lands. These empty statements are that
  // claim (a "use" after the wait).
#pragma unroll
  for (int i = 0; i < 4; ++i)
    asm volatile("" ::"v"(A0[0][i]), "v"(A0[1][i]), "v"(A1[0][i]), "v"(A1[1][i]));
  if (wave < 4) G2_BARRIER();  // balance the stagger barrier

  const int nbase = tn * G2_BN + wn * 64, mbase = m0 + wm * (16 * MF);
  // Epilogue through LDS. Stored straight from the accumulator layout, a wave's store
  // instruction would touch 16 rows with 32 bytes each; the stores of a tile then cost as much
  // as ten K-tiles of math. Instead every wave transposes its sub-tile through a private LDS
  // region (the ring is idle by now) and writes whole rows of it: 16 bytes per lane, 8 (plain)
  // or 16 (SwiGLU) rows of 128 or 64 contiguous bytes per instruction.
  if constexpr (EPI == EPI_F32) {
    if ((ldy & 3) == 0 && (tn + 1) * G2_BN <= N) {   // uniform, as below
      G2_BARRIER();                                    // every wave is past its last ring read
      // A wave's 64 columns are 256 bytes a row, half of its rows at a time: four whole rows per store instruction. Stored
      // from the accumulator layout (16 rows of 64 bytes) 2048 x 6144 x 2048 took 61.3 us instead of 57.6, 2361 x 6720 x 2048
      // 90.4 instead of 83.3, 2048 x 2048 x 8192 in four parts 72.1 instead of 67.7.
      constexpr int JH = (MF + 1) / 2;
      char* mine = smem + wave * (JH * 16 * 256);
      const int g = lane >> 4, r16 = lane & 15;
      const bf16_t* add = gridDim.y > 1 ? nullptr : bias;
      float* out = static_cast<float*>(Y) + (static_cast<size_t>(blockIdx.y) * M + mbase) * ldy + nbase + r16 * 4;
#pragma unroll
      for (int j0 = 0; j0 < MF; j0 += JH) {
#pragma unroll
        for (int j = j0; j < (j0 + JH < MF ? j0 + JH : MF); ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4 v = acc[i][j];
            if (add != nullptr) {
#pragma unroll
              for (int r = 0; r < 4; ++r) v[r] += bf16_to_f32(add[nbase + i * 16 + 4 * g + r]);
            }
            // chunk c of row m lives at position c ^ (m mod 16)
            *reinterpret_cast<f32x4*>(mine + ((j - j0) * 16 + r16) * 256 + (((i * 4 + g) ^ r16) << 4)) = v;
          }
#pragma unroll
        for (int p = 0; p < (j0 + JH < MF ? JH : MF - j0) * 4; ++p) {
          const int row = p * 4 + g, m = j0 * 16 + row;
          const f32x4 v = *reinterpret_cast<const f32x4*>(mine + row * 256 + ((r16 ^ (row & 15)) << 4));
          if (mbase + m < M) *reinterpret_cast<f32x4*>(out + static_cast<size_t>(m) * ldy) = v;
        }
      }
      return;
    }
  } else {
    if ((ldy & 7) == 0 && (tn + 1) * G2_BN <= N) {   // uniform: the whole block tile is inside Y
      G2_BARRIER();                                    // every wave is past its last ring read
      // Staged rows are 128 bytes: a wave's 64 columns, or with SwiGLU the 32 + 32 output
      // columns of two waves that are neighbours in n (they share a region and split its rows).
      constexpr int ROWB = 128, CH = 8;
      char* mine = smem + (epi_gated(EPI) ? (wm * 2 + (wn >> 1)) : wave) * (16 * MF * ROWB);
      const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
      for (int j = 0; j < MF; ++j) {
        const int m = j * 16 + r16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          u32x2 o;
          int chunk;
          if constexpr (epi_gated(EPI)) {
            if (i & 1) continue;
            const int nb = nbase + i * 16 + 4 * g;
            float gt[4], up[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              gt[r] = acc[i][j][r] + (bias ? bf16_to_f32(bias[nb + r]) : 0.f);
              up[r] = acc[i + 1][j][r] + (bias ? bf16_to_f32(bias[nb + 16 + r]) : 0.f);
            }
            o[0] = pack_bf16x2(gate_act<EPI>(gt[0]) * up[0], gate_act<EPI>(gt[1]) * up[1]);
            o[1] = pack_bf16x2(gate_act<EPI>(gt[2]) * up[2], gate_act<EPI>(gt[3]) * up[3]);
            chunk = (wn & 1) * 4 + (i >> 1) * 2 + (g >> 1);
          } else {
            const int nb = nbase + i * 16 + 4 * g;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = column_act<EPI>(acc[i][j][r] + (bias ? bf16_to_f32(bias[nb + r]) : 0.f), ap, an);
            o[0] = pack_bf16x2(v[0], v[1]);
            o[1] = pack_bf16x2(v[2], v[3]);
            chunk = i * 2 + (g >> 1);
          }
          // chunk c of row m lives at position c ^ (m mod CH): column accesses spread over banks
          *reinterpret_cast<u32x2*>(mine + m * ROWB + ((chunk ^ (m & (CH - 1))) << 4) + (g & 1) * 8) = o;
        }
      }
      constexpr int RPI = 64 / CH;                         // rows per store instruction
      const int c16 = lane & (CH - 1), rsub = lane / CH;
      const int ncol = (epi_gated(EPI) ? tn * (G2_BN / 2) + (wn >> 1) * 64 : nbase) + c16 * 8;
      constexpr int PASSES = epi_gated(EPI) ? MF : 2 * MF;
      const int p0 = epi_gated(EPI) ? (wn & 1) * MF : 0;
      if constexpr (epi_gated(EPI)) G2_BARRIER();       // the partner wave's half rows are in place
#pragma unroll
      for (int pp = 0; pp < PASSES; ++pp) {
        const int p = p0 + pp;
        const int m = p * RPI + rsub;
        const u32x4 v = *reinterpret_cast<const u32x4*>(mine + m * ROWB + ((c16 ^ (m & (CH - 1))) << 4));
        if (mbase + m < M)
          *reinterpret_cast<u32x4*>(static_cast<bf16_t*>(Y) + static_cast<size_t>(mbase + m) * ldy + ncol) = v;
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      if constexpr (epi_gated(EPI)) {
        if (i & 1) continue;
        store_tile<EPI>(acc[i][j], &acc[i + 1][j], Y, bias, mbase + j * 16, nbase + i * 16, M, N, ldy, lane, 0);
      } else {
        const size_t slab = (EPI == EPI_F32) ? static_cast<size_t>(blockIdx.y) * M * ldy : 0;
        store_tile<EPI>(acc[i][j], nullptr, Y, gridDim.y > 1 ? nullptr : bias, mbase + j * 16, nbase + i * 16, M, N,
                        ldy, lane, slab, ap, an);
      }
    }
}


}  // namespace

// One launch over tiles of 32 MF rows.
template <int EPI, bool GROUPED, int MF>
static int g2_launch(const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K, int n_pad, int ldy, int splits,
                     long long expert_stride, const void* offsets, int E, float ap, float an, hipStream_t stream) {
  const int tiles_m = (M + g2_rows(MF) - 1) / g2_rows(MF) + (GROUPED ? E : 0), tiles_n = n_pad / G2_BN;
  static LcDeviceOnce attr_once;
  attr_once.run([&] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm256_kernel<EPI, GROUPED, MF>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, g2_lds(MF));
  });
  gemm256_kernel<EPI, GROUPED, MF><<<dim3(tiles_m * tiles_n, splits), 512, g2_lds(MF), stream>>>(
      static_cast<const bf16_t*>(Wp), static_cast<const bf16_t*>(X), Y, static_cast<const bf16_t*>(bias), M, N, K, ldy, tiles_m, tiles_n,
      expert_stride, static_cast<const int32_t*>(offsets), E, splits > 1 ? K / G2_BK / splits : 0, ap, an);
  LC_RETURN_LAST_ERROR();
}

template <int EPI>
static int g2_rows_launch(int mf, const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K, int n_pad, int ldy,
                          int splits, float ap, float an, hipStream_t stream) {
#define G2_MF(F) g2_launch<EPI, false, F>(Wp, X, Y, bias, M, N, K, n_pad, ldy, splits, 0, nullptr, 0, ap, an, stream)
  switch (mf) {
    case 8: return G2_MF(8);
    case 7: return G2_MF(7);
    case 6: return G2_MF(6);
    case 5: return G2_MF(5);
    case 4: return G2_MF(4);
  }
#undef G2_MF
  return -2;
}

// Y = X * W^T in tiles of 256 columns and 32 mf rows (mf 4 to 8). Requirements: K % 64 == 0, n_pad % 256 == 0.
LC_EXPORT int lc_gemm256(const void* Wp, const void* X, void* Y, const void* bias, int M, int N, int K,
                         int n_pad, int ldy, int epi, float ap, float an, int mf, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K % 64 || n_pad % 256 || N > n_pad) return -1;
#define G2_EPI(E) \
  case E: return g2_rows_launch<E>(mf, Wp, X, Y, bias, M, N, K, n_pad, ldy, 1, ap, an, stream)
  switch (epi) {
    G2_EPI(EPI_BF16);
    G2_EPI(EPI_F32);
    G2_EPI(EPI_SWIGLU);
    G2_EPI(EPI_GEGLU);
    G2_EPI(EPI_REGLU);
    G2_EPI(EPI_RELU2);
    G2_EPI(EPI_XIELU);
  }
#undef G2_EPI
  return -2;
}

// Grouped form over E experts for prefill-sized MoE batches: X [total_rows, K] and Y are in
// expert-sorted row order, offsets [E+1] delimit the experts' rows. Requirements as lc_gemm256. Tiles of 256 rows whatever the experts
// get: lower ones pad less, and lose all the same (8 experts of 28672 x 4096, 4316 routed rows 1018 us, 1055 with 224 rows, 1241 with 160).
LC_EXPORT int lc_gemm256_grouped(const void* Wp_all, long long expert_stride, const void* X, const void* offsets,
                                 int E, void* Y, int total_rows, int N, int K, int n_pad, int ldy, int epi,
                                 hipStream_t stream) {
  if (total_rows <= 0) return 0;
  if (K % 64 || n_pad % 256 || N > n_pad || E < 1) return -1;
  if (epi == EPI_BF16)
    return g2_launch<EPI_BF16, true, 8>(Wp_all, X, Y, nullptr, total_rows, N, K, n_pad, ldy, 1, expert_stride, offsets, E, 0.f, 0.f, stream);
  if (epi == EPI_SWIGLU)
    return g2_launch<EPI_SWIGLU, true, 8>(Wp_all, X, Y, nullptr, total_rows, N, K, n_pad, ldy, 1, expert_stride, offsets, E, 0.f, 0.f, stream);
  return -2;
}

// Split-K form for a few hundred to a few thousand rows against a narrow output, where the
// tiles alone would leave most CUs idle: Y = fp32 slabs [splits, M, ldy] (no bias).
LC_EXPORT int lc_gemm256_splitk(const void* Wp, const void* X, void* Y, int M, int N, int K, int n_pad, int ldy,
                                int splits, int mf, hipStream_t stream) {
  if (M <= 0) return 0;
  if (K % 64 || n_pad % 256 || N > n_pad || splits < 1 || (K / G2_BK) % splits) return -1;
  return g2_rows_launch<EPI_F32>(mf, Wp, X, Y, nullptr, M, N, K, n_pad, ldy, splits, 0.f, 0.f, stream);
}
