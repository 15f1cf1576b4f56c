// Products of any shape and type of the hybrid decoder designs, on the fp32 matrix instructions: C = A W^T with A, W and C
// each fp32 or bf16 (widened exactly when loaded) and fp32 accumulation. They serve what the bf16 kernels (gemm*.hip: bf16, K a
// multiple of 64) do not take: every product of the true-fp32 mode, depths that are no multiple of 64, inputs that are fp32
// column slices, products per head and, in the fp32 mode, per expert.
//
// v_mfma_f32_16x16x4_f32 takes one number per lane and operand: lane l holds row (column) l & 15 at depth l >> 4. The sum over
// the depth may run in any order, so that a lane loads FOUR neighbouring depths of its row at once (depth 4 (l >> 4) + j is the
// operand of instruction j), for A and W alike: 16-byte accesses, no transposition anywhere.
#include "hybrid_common.h"

namespace {

struct AnyGemm {
  const void* A;
  const void* W;
  const void* bias;              // [N] of W's type, or null
  void* C;
  const float* gate;             // logits, or null: outputs are scaled by the sigmoid of their row's and head's (gate_full: their own)
  int a_f32, w_f32, c_f32;
  int a_vec, w_vec;              // every row starts on a border of four elements, and K is a multiple of four
  int lda, ldc, M, N, K;
  int epi;                       // 1: square of relu
  int a_hs, c_hs;                // first column of head h in A and in C
  int ld_gate, gate_full;
  int c_vec;                     // C's rows and heads start on 16 bytes
  int splits;                    // > 1: part s of the depth leaves its sums in slab s of C (fp32, [M, ldc] each; no bias, epi or gate)
};

// Elements i .. i + 3 of p as floats, zeros from the n-th on (n may be negative).
LC_DEVICE float4 load4_any(const void* p, int f32, int vec, size_t i, int n) {
  if (vec) {
    if (n <= 0) return make_float4(0.f, 0.f, 0.f, 0.f);
    return f32 ? load_act4<true>(static_cast<const float*>(p) + i) : load_act4<false>(static_cast<const bf16_t*>(p) + i);
  }
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v[j] = j >= n ? 0.f : f32 ? static_cast<const float*>(p)[i + j] : bf16_to_f32(static_cast<const bf16_t*>(p)[i + j]);
  return make_float4(v[0], v[1], v[2], v[3]);
}

LC_DEVICE void finish_any(const AnyGemm& g, int h, int row, int col, float v, int split) {
  if (row >= g.M || col >= g.N) return;
  if (g.splits > 1) {
    static_cast<float*>(g.C)[(static_cast<size_t>(split) * g.M + row) * g.ldc + col] = v;
    return;
  }
  if (g.bias != nullptr) v += g.w_f32 ? static_cast<const float*>(g.bias)[col] : bf16_to_f32(static_cast<const bf16_t*>(g.bias)[col]);
  if (g.epi == 1) {
    v = fmaxf(v, 0.f);
    v *= v;
  }
  if (g.gate != nullptr) v *= sigmoidf_(g.gate[static_cast<size_t>(row) * g.ld_gate + (g.gate_full ? h * g.N + col : h)]);
  const size_t at = static_cast<size_t>(row) * g.ldc + static_cast<size_t>(h) * g.c_hs + col;
  if (g.c_f32)
    static_cast<float*>(g.C)[at] = v;
  else
    static_cast<bf16_t*>(g.C)[at] = f32_to_bf16(v);
}

LC_DEVICE float at4(const float4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }

// ---------------------------------------------------------------- up to 64 rows
// Bound by reading W once, and by latency where W is small. A block owns 16 outputs and splits the depth over its waves in turns
// of 32 (a row's 128 bytes per wave, 2 KB side by side over 16 waves); the partial sums meet in LDS. No staging: each wave
// multiplies what it loaded. W's rows are the first operand, so that a lane ends up with four neighbouring outputs of one row of A.
// 3 rows in fp32: 1024 x 1024 / 1024 x 4096 (outputs x depth) 10.6 us on average, 4096 x 1024 7.9 us, 32000 x 1024 32 us (4 TB/s);
// 64 x 64 tiles on the vector ALUs, as for more rows before, took 287, 136 and 172 us (their 16 .. 64 blocks left the chip idle).
template <int WAVES, int MT>
__global__ __launch_bounds__(64 * WAVES) void gemm_any_rows_kernel(AnyGemm g) {
  __shared__ f32x4 red[WAVES][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
  const int n0 = blockIdx.x * 16, h = blockIdx.z;
  const size_t w_row = (static_cast<size_t>(h) * g.N + min(n0 + lr, g.N - 1)) * g.K;
  size_t a_row[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) a_row[m] = static_cast<size_t>(min(16 * m + lr, g.M - 1)) * g.lda + static_cast<size_t>(h) * g.a_hs;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  float4 w[2], a[MT][2], wn[2], an[MT][2];
  auto fetch = [&](float4(&wd)[2], float4(&ad)[MT][2], int c) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = 32 * c + 8 * lq + 4 * s;
      wd[s] = load4_any(g.W, g.w_f32, g.w_vec, w_row + k, g.K - k);
#pragma unroll
      for (int m = 0; m < MT; ++m) ad[m][s] = load4_any(g.A, g.a_f32, g.a_vec, a_row[m] + k, g.K - k);
    }
  };
  const int chunks = (g.K + 31) / 32, per = (chunks + g.splits - 1) / g.splits;
  const int first = blockIdx.y * per + wave, last = min(static_cast<int>(blockIdx.y + 1) * per, chunks);
  if (first < last) fetch(w, a, first);
  for (int c = first; c < last; c += WAVES) {
    if (c + WAVES < last) fetch(wn, an, c + WAVES);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(w[s], j), at4(a[m][s], j), acc[m], 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      w[s] = wn[s];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m][s] = an[m][s];
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) red[wave][m][lane] = acc[m];
  __syncthreads();
  if (wave >= MT) return;
  f32x4 sum = red[0][wave][lane];
#pragma unroll
  for (int i = 1; i < WAVES; ++i) sum += red[i][wave][lane];
#pragma unroll
  for (int r = 0; r < 4; ++r) finish_any(g, h, 16 * wave + lr, n0 + 4 * lq + r, sum[r], blockIdx.y);
}

// ---------------------------------------------------------------- more rows
// 64 x 64 outputs per block, bound by the fp32 matrix rate. Four waves of 32 x 32 per depth group; KG groups split the depth
// where the tiles alone would leave CUs idle or a SIMD with a single wave, and their sums meet in LDS. Slabs of 16 depths pass
// through two LDS buffers (rows of 20 floats: the 16-byte reads of 16 rows hit all banks evenly), loads one slab ahead: a slab
// is 16 matrix instructions per wave (512 cycles) against four 16-byte LDS reads. 804 rows in fp32, 4096 x 1024: 92 us = 73 TFLOP/s,
// 1024 x 1024 / 1024 x 4096 58 us on average (vector ALUs, no depth groups: 182 and 319 us).
// GROUPED: rows are sorted positions; position p in [offsets[e], offsets[e + 1]) gives C[p] = W[e] A[row_index[p]] (A[p] without
// an index). Tile blockIdx.y belongs to the expert whose run of tiles it falls into (at most ceil(rows / 64) + E exist).
constexpr int kSlabLd = 20;

template <int KG, bool GROUPED>
__global__ __launch_bounds__(256 * KG) void gemm_any_tile_kernel(AnyGemm g, const int32_t* __restrict__ row_index,
                                                                 const int32_t* __restrict__ offsets, int E) {
  extern __shared__ __attribute__((aligned(16))) float slab[];          // [2][KG][A | W][64][kSlabLd]
  const int tid = threadIdx.x & 255, kg = threadIdx.x >> 8, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lq = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int n0 = blockIdx.x * 64;
  const int split = g.splits > 1 ? blockIdx.z : 0;     // (products per head are not split)
  int m0 = blockIdx.y * 64, h = g.splits > 1 ? 0 : blockIdx.z;
  size_t w_first = static_cast<size_t>(h) * g.N * g.K;
  if constexpr (GROUPED) {
    int e = 0, tile = blockIdx.y, lo = 0, hi = 0;
    for (; e < E; ++e) {
      lo = offsets[e];
      hi = offsets[e + 1];
      const int nt = (hi - lo + 63) >> 6;
      if (tile < nt) break;
      tile -= nt;
    }
    if (e >= E) return;                                // the same for the whole block
    m0 = lo + tile * 64;
    g.M = hi;
    w_first = static_cast<size_t>(e) * g.N * g.K;
  }
  const int sr = tid >> 2, sk = (tid & 3) * 4;         // the row and depths of a slab that this thread loads
  int a_at = min(m0 + sr, g.M - 1);
  if (GROUPED && row_index != nullptr) a_at = row_index[a_at];
  const size_t a_row = static_cast<size_t>(a_at) * g.lda + static_cast<size_t>(h) * g.a_hs;
  const size_t w_row = w_first + static_cast<size_t>(min(n0 + sr, g.N - 1)) * g.K;
  const int groups = KG * g.splits;
  const int slabs = ((g.K + 15) / 16 + groups - 1) / groups;   // per group; behind the last depth slabs are zeros
  float4 ra, rw;
  auto fetch = [&](int s) {
    const int k = 16 * ((split * KG + kg) * slabs + s) + sk;
    ra = load4_any(g.A, g.a_f32, g.a_vec, a_row + k, g.K - k);
    rw = load4_any(g.W, g.w_f32, g.w_vec, w_row + k, g.K - k);
  };
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  for (int s = 0; s < slabs; ++s) {
    float* as = slab + ((s & 1) * KG + kg) * (2 * 64 * kSlabLd);
    float* ws = as + 64 * kSlabLd;
    *reinterpret_cast<float4*>(as + sr * kSlabLd + sk) = ra;
    *reinterpret_cast<float4*>(ws + sr * kSlabLd + sk) = rw;
    __syncthreads();          // (one is enough: whoever is past it has read the other buffer, which the next slab overwrites)
    if (s + 1 < slabs) fetch(s + 1);
    float4 af[2], wf[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      af[i] = *reinterpret_cast<const float4*>(as + (32 * wm + 16 * i + lr) * kSlabLd + 4 * lq);
      wf[i] = *reinterpret_cast<const float4*>(ws + (32 * wn + 16 * i + lr) * kSlabLd + 4 * lq);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(af[i], k), at4(wf[j], k), acc[i][j], 0, 0, 0);
  }
  if constexpr (KG > 1) {
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(slab);       // [KG - 1][4][256]
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((kg - 1) * 4 + i) * 256 + tid] = acc[i >> 1][i & 1];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int q = 0; q < KG - 1; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] += red[(q * 4 + i) * 256 + tid];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        finish_any(g, h, m0 + 32 * wm + 16 * i + 4 * lq + r, n0 + 32 * wn + 16 * j + lr, acc[i][j][r], split);
}

// ---------------------------------------------------------------- more rows, fp32 throughout
// The same tiles for fp32 activations and weights whose depth is in whole lines: slabs of 32 depths go
// from memory to LDS as whole 128-byte rows (LDS-DMA, no registers in between, two stages, one barrier per slab), in an
// XOR-swizzled image (chunk c of row r lies at c ^ (r mod 8): the source addresses are permuted, the 16-byte reads of eight rows hit
// all banks). W's rows are the first operand, so that a lane holds four neighbouring outputs of a row. Four sums of every fourth depth
// keep the rounding of a sum at what up to four depth groups had above.
// 801 rows: 4096 x 1024 92 -> 82 us (82 TFLOP/s), 32000 x 1024 524 -> 471 (111; registers alone reach 154), 1024 x 4096 in eight parts 78 -> 67;
// 151 rows, 1024 x 1024 in eight parts 10.5 -> 8.0. The matrix units are busy 77 % of the time, whatever the waves per SIMD (three
// stages 1 - 3 % either way). Every wave with the whole tile for a quarter of the depth, operands straight into registers: 98 us
// for the first (256 registers do not hold the sums and two steps).
constexpr int kLineSlab = 32, kLineStage = 2 * 64 * 128;      // bytes of a stage: A | W, 64 rows of a line each

template <int KG, bool GROUPED>
__global__ __launch_bounds__(256 * KG) void gemm_f32_tile_kernel(AnyGemm g, const int32_t* __restrict__ row_index,
                                                                 const int32_t* __restrict__ offsets, int E) {
  extern __shared__ __attribute__((aligned(16))) char lines[];          // [KG][2][A | W][64][128]
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int n0 = blockIdx.x * 64;
  const int split = g.splits > 1 ? blockIdx.z : 0;     // (products per head are not split)
  int m0 = blockIdx.y * 64, h = g.splits > 1 ? 0 : blockIdx.z;
  size_t w_first = static_cast<size_t>(h) * g.N * g.K;
  if constexpr (GROUPED) {
    int e = 0, tile = blockIdx.y, lo = 0, hi = 0;
    for (; e < E; ++e) {
      lo = offsets[e];
      hi = offsets[e + 1];
      const int nt = (hi - lo + 63) >> 6;
      if (tile < nt) break;
      tile -= nt;
    }
    if (e >= E) return;                                // the same for the whole block
    m0 = lo + tile * 64;
    g.M = hi;
    w_first = static_cast<size_t>(e) * g.N * g.K;
  }
  // this wave's pieces of a slab: rows 8 wave .. + 7 and 32 + 8 wave .. of either operand
  const int rr = lane >> 3, chunk = ((lane & 7) ^ rr) * 4;
  const float *asrc[2], *wsrc[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int row = (4 * p + wave) * 8 + rr;
    int a_at = min(m0 + row, g.M - 1);
    if (GROUPED && row_index != nullptr) a_at = row_index[a_at];
    asrc[p] = static_cast<const float*>(g.A) + static_cast<size_t>(a_at) * g.lda + static_cast<size_t>(h) * g.a_hs + chunk;
    wsrc[p] = static_cast<const float*>(g.W) + w_first + static_cast<size_t>(min(n0 + row, g.N - 1)) * g.K + chunk;
  }
  const int groups = KG * g.splits, all = g.K / kLineSlab, per = (all + groups - 1) / groups;
  const int first = min((split * KG + kg) * per, all), mine = min(per, all - first);
  char* const stages = lines + kg * 2 * kLineStage;
  auto issue = [&](int s) {
    char* dst = stages + (s & 1) * kLineStage;
    const int k = (first + s) * kLineSlab;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(asrc[p] + k), LC_LDS_PTR(dst + (4 * p + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(LC_GLOBAL_PTR(wsrc[p] + k), LC_LDS_PTR(dst + 64 * 128 + (4 * p + wave) * 1024), 16, 0, 0);
    }
  };
  f32x4 part[4][2][2], acc[2][2];                       // [16 columns][16 rows]; a part sums every fourth depth
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) part[k][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (mine > 0) issue(0);
  for (int s = 0; s < mine; ++s) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                       // slab s has landed; whoever is past this has read slab s - 1
    asm volatile("" ::: "memory");
    if (s + 1 < mine) issue(s + 1);
    const char* as = stages + (s & 1) * kLineStage + (32 * wm + lr) * 128;
    const char* ws = stages + (s & 1) * kLineStage + 64 * 128 + (32 * wn + lr) * 128;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int at = ((4 * t + lq) ^ (lr & 7)) << 4;
      f32x4 af[2], wf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        af[i] = *reinterpret_cast<const f32x4*>(as + i * 2048 + at);
        wf[i] = *reinterpret_cast<const f32x4*>(ws + i * 2048 + at);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) part[k][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][k], af[j][k], part[k][i][j], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads are over before the stage may be written again
  }
  for (int s = max(mine, 0); s < per; ++s) __builtin_amdgcn_s_barrier();   // (every depth group takes every barrier)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (part[0][i][j] + part[1][i][j]) + (part[2][i][j] + part[3][i][j]);
  if constexpr (KG > 1) {
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(lines);       // [KG - 1][4][256]
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((kg - 1) * 4 + i) * 256 + tid] = acc[i >> 1][i & 1];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int q = 0; q < KG - 1; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] += red[(q * 4 + i) * 256 + tid];
  }
  const bool plain = g.bias == nullptr && g.gate == nullptr && g.c_f32 && g.c_vec;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = m0 + 32 * wm + 16 * j + lr, col = n0 + 32 * wn + 16 * i + 4 * lq;
      if (plain && col + 3 < g.N) {
        if (row >= g.M) continue;
        f32x4 v = acc[i][j];
        if (g.epi == 1) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = relu2(v[r]);
        }
        const size_t at = (static_cast<size_t>(split) * g.M + row) * g.ldc + static_cast<size_t>(h) * g.c_hs + col;
        *reinterpret_cast<f32x4*>(static_cast<float*>(g.C) + at) = v;
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) finish_any(g, h, row, col + r, acc[i][j][r], split);
    }
}

template <int KG, bool GROUPED>
int launch_tiles(const AnyGemm& g, const dim3& grid, const int32_t* row_index, const int32_t* offsets, int E, hipStream_t st) {
  constexpr size_t lds = 2 * KG * 2 * 64 * kSlabLd * sizeof(float);
  if constexpr (lds > 64 * 1024) {
    static LcDeviceOnce once;
    once.run([] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_any_tile_kernel<KG, GROUPED>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    });
  }
  gemm_any_tile_kernel<KG, GROUPED><<<grid, dim3(256 * KG), lds, st>>>(g, row_index, offsets, E);
  LC_RETURN_LAST_ERROR();
}

template <int KG, bool GROUPED>
int launch_f32_tiles(const AnyGemm& g, const dim3& grid, const int32_t* row_index, const int32_t* offsets, int E, hipStream_t st) {
  gemm_f32_tile_kernel<KG, GROUPED><<<grid, dim3(256 * KG), 2 * KG * kLineStage, st>>>(g, row_index, offsets, E);
  LC_RETURN_LAST_ERROR();
}

// Depth groups: enough waves for four on each of the 1024 SIMDs, none shorter than four slabs. Whole lines of fp32: two groups where they
// leave no CU a second block (151 rows, 4096 x 1024, 192 blocks, 22.2 -> 20.8 us; 312 blocks 37.1 -> 39.8) or where there are more
// than two and a depth to share (832 blocks of depth 1024 83.5 -> 82, of 128 10.7 -> 13.9).
template <bool GROUPED>
int tiles_any(const AnyGemm& g, int m_tiles, int heads, const int32_t* row_index, const int32_t* offsets, int E, hipStream_t st) {
  const dim3 grid((g.N + 63) / 64, m_tiles, g.splits > 1 ? g.splits : heads);
  const long long blocks = static_cast<long long>(grid.x) * grid.y * grid.z;
  if (g.a_f32 && g.w_f32 && g.a_vec && g.w_vec && g.K % kLineSlab == 0) {
    if (blocks <= 256 ? g.K / g.splits >= 256 : blocks > 512 && g.K / g.splits >= 512)
      return launch_f32_tiles<2, GROUPED>(g, grid, row_index, offsets, E, st);
    return launch_f32_tiles<1, GROUPED>(g, grid, row_index, offsets, E, st);
  }
  if (blocks <= 512 && g.K >= 256) return launch_tiles<4, GROUPED>(g, grid, row_index, offsets, E, st);
  if (blocks <= 1024 && g.K >= 128) return launch_tiles<2, GROUPED>(g, grid, row_index, offsets, E, st);
  return launch_tiles<1, GROUPED>(g, grid, row_index, offsets, E, st);
}

template <int WAVES>
int rows_any(const AnyGemm& g, int heads, hipStream_t st) {
  const dim3 grid((g.N + 15) / 16, g.splits, heads), block(64 * WAVES);
  if (g.M <= 16)
    gemm_any_rows_kernel<WAVES, 1><<<grid, block, 0, st>>>(g);
  else if (g.M <= 32)
    gemm_any_rows_kernel<WAVES, 2><<<grid, block, 0, st>>>(g);
  else
    gemm_any_rows_kernel<WAVES, 4><<<grid, block, 0, st>>>(g);
  LC_RETURN_LAST_ERROR();
}

int any_product(const AnyGemm& g, int heads, hipStream_t st) {
  if (g.M > 64) {
    const int m_tiles = (g.M + 63) / 64;
    if (m_tiles > 65535) return -1;
    return tiles_any<false>(g, m_tiles, heads, nullptr, nullptr, 0, st);
  }
  // sixteen waves give 64 blocks (1024 outputs) the loads in flight of 256 CUs; from 1024 blocks on, or where the depth is four
  // turns at most, four waves hold as many and a block ends sooner
  const bool wide = static_cast<long long>((g.N + 15) / 16) * heads >= 1024 || g.K / g.splits <= 128;
  return wide ? rows_any<4>(g, heads, st) : rows_any<16>(g, heads, st);
}

int four_border(const void* p, int f32) { return reinterpret_cast<uintptr_t>(p) % (f32 ? 16 : 8) == 0; }

}  // namespace

// ================================================================= launchers
// A may be a column slice of a wider matrix: ``lda`` is its row stride in elements. ``splits`` > 1: C is [splits, M, N] fp32, the
// sums of as many parts of the depth.
LC_EXPORT int lc_gemm_any(const void* A, int a_f32, int lda, const void* W, int w_f32, const void* bias, void* C,
                          int c_f32, int M, int N, int K, int epi, int splits, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || splits < 1 || splits > 64 || (splits > 1 && (bias != nullptr || epi != 0 || !c_f32))) return -1;
  const AnyGemm g{A, W, bias, C, nullptr, a_f32, w_f32, c_f32, K % 4 == 0 && lda % 4 == 0 && four_border(A, a_f32),
                  K % 4 == 0 && four_border(W, w_f32), lda, N, M, N, K, epi, 0, 0, 0, 0, N % 4 == 0 && four_border(C, 1), splits};
  return any_product(g, 1, st);
}

// C[m, h, :] = W[h] A[m, h, :] for H heads: W [H, N, K]; head h's inputs start at column h * a_hs of A (row stride lda), its
// outputs at column h * c_hs of C (row stride c_ld). With ``gate`` [M, H] (row stride ld_gate) the head's outputs are scaled by
// sigmoid(gate[m, h]); ``gate_full``: the gate is [M, H*N], one logit per output.
LC_EXPORT int lc_head_linear(const void* A, int a_f32, int lda, const void* W, int w_f32, void* C, int c_f32,
                             const void* gate, int ld_gate, int M, int H, int N, int K, int a_hs, int c_ld, int c_hs,
                             int gate_full, hipStream_t st) {
  if (M <= 0 || N <= 0 || H <= 0) return 0;
  if (K <= 0 || a_hs < K || lda < (H - 1) * a_hs + K || H > 65535 || c_hs < N || c_ld < (H - 1) * c_hs + N) return -1;
  if (gate != nullptr && ld_gate < (gate_full ? H * N : H)) return -1;
  if (gate == nullptr && gate_full) return -1;
  const AnyGemm g{A, W, nullptr, C, static_cast<const float*>(gate), a_f32, w_f32, c_f32,
                  K % 4 == 0 && lda % 4 == 0 && a_hs % 4 == 0 && four_border(A, a_f32), K % 4 == 0 && four_border(W, w_f32),
                  lda, c_ld, M, N, K, 0, a_hs, c_hs, ld_gate, gate_full, c_ld % 4 == 0 && c_hs % 4 == 0 && four_border(C, 1), 1};
  return any_product(g, H, st);
}

// ``rows``: an upper bound of offsets[E] known to the host (tokens x choices).
LC_EXPORT int lc_gemm_any_grouped(const void* A, int a_f32, int lda, const void* row_index, const void* offsets,
                                  const void* W, int w_f32, void* C, int c_f32, int rows, int E, int N, int K, int epi,
                                  hipStream_t st) {
  if (rows <= 0 || N <= 0 || E <= 0) return 0;
  if (K <= 0 || lda < K) return -1;
  const int tiles = (rows + 63) / 64 + E;
  if (tiles > 65535) return -1;
  const AnyGemm g{A, W, nullptr, C, nullptr, a_f32, w_f32, c_f32, K % 4 == 0 && lda % 4 == 0 && four_border(A, a_f32),
                  K % 4 == 0 && four_border(W, w_f32), lda, N, rows, N, K, epi, 0, 0, 0, 0, N % 4 == 0 && four_border(C, 1), 1};
  return tiles_any<true>(g, tiles, 1, static_cast<const int32_t*>(row_index), static_cast<const int32_t*>(offsets), E, st);
}
