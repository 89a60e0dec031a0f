// Batched products with a short inner dimension and 32-bit outputs: attention scores, K = head size up to 128.  Included by
// gemm_s8_impl.h (work order: bmm_any.h).
//
// Bound by the stores: 4 bytes of output for 2 K operations, 5.7 TB/s with whole 128-byte lines.  No pipeline: the whole of K is one
// step, a wave loads its rows of both operands, multiplies, stores 128-byte pieces of rows and ends, and what keeps the memory busy is
// many workgroups that are not in step.  Small tiles waste little where the lengths are ragged, and leave no half-empty last
// round.  us, before (persistent 256x256 tiles, or tiles by the register) / now: 160 x 512 x 512 x 128 34.9 / 29.3, 300 x 333 x 333 x 128
// 62.2 / 27.8, 100 x 301 x 301 x 80 24.6 / 11.6, 31 x 1703 x 1703 x 128 169 / 103, 101 x 1258 x 1258 x 64 329 / 169, 13 x 158 x 158 x 64 3.7 / 2.9.
#pragma once

namespace ti {

// Stores the products of a wave's rows of fragments fa with its fragments fb: rows from m0, columns from n0 on.
// STREAM: non-temporal stores.
template <int KIND, int KB, int TM, int TN, bool STREAM>
__device__ __forceinline__ void store_scores(v4i (&fa)[KB][TM], v4i (&fb)[KB][TN], const GemmParams& p, int b, int m0, int n0, int lane) {
  using E = Epi<KIND>;
  using Out = typename E::Out;
  const int r = lane & 15, g = lane >> 4, M = p.M, N = p.N;
  // Lane (r, g) gets row r and columns 4 g .. 4 g + 3 of a block.  Lanes r and r ^ 8 swap a block of each pair, so that a store writes
  // eight rows x 128 bytes.  16 bytes at any multiple of four: rows of a ragged length begin anywhere.
  typedef int v4i_dwords __attribute__((ext_vector_type(4), aligned(4)));
  Out* C = reinterpret_cast<Out*>(p.C) + (long long)b * p.strideC;
  const bool upper = r >= 8;
  const int c0 = n0 + (upper ? 16 : 0) + 4 * g;
  auto put = [&](int row, int col, v4i w) {
    if (row >= M || col >= N) return;
    Out* at = C + (long long)row * N + col;
    if (col + 4 <= N) {
      if constexpr (STREAM) __builtin_nontemporal_store(w, reinterpret_cast<v4i_dwords*>(at));
      else *reinterpret_cast<v4i_dwords*>(at) = w;
    } else {
#pragma unroll
      for (int v = 0; v < 3; ++v)
        if (col + v < N) {
          const int bits = w[v];  // a plain value: the cast must not see a vector element
          at[v] = __builtin_bit_cast(Out, bits);
        }
    }
  };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (m0 + i * 16 >= M) break;
    v4i acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[j] = v4i{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KB; ++s) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[s][j], fa[s][i], acc[j], 0, 0, 0);
    }
    const int row = m0 + i * 16 + (r & 7);
#pragma unroll
    for (int j = 0; j < TN; j += 2) {
      v4i lo, hi;  // rows 0..7 and 8..15 of the block row
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const Out x = E::apply(acc[j][v], 0.0f, p.alpha), y = E::apply(acc[j + 1][v], 0.0f, p.alpha);
        const int x0 = __builtin_bit_cast(int, x), x1 = __builtin_bit_cast(int, y);
        const int got = __builtin_amdgcn_mov_dpp(upper ? x0 : x1, 0x128, 0xf, 0xf, true);  // row_ror:8
        lo[v] = upper ? got : x0;
        hi[v] = upper ? x1 : got;
      }
      put(row, c0 + j * 16, lo);
      put(row + 8, c0 + j * 16, hi);
    }
  }
}

// A wave owns 16 TM x 16 TN outputs and loads its rows straight into matrix registers.
template <int KIND, int KB, int TM, int TN>
__global__ __launch_bounds__(256) void gemm_scores_kernel(GemmParams p, int tiles_m, int tiles_n) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int tiles = tiles_m * tiles_n;
  const long long items = (long long)tiles * p.batch;
  const long long group = item_on_xcd((items + 3) / 4);
  const long long item = group * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (group < 0 || item >= items) return;  // waves are on their own: no barrier in this kernel
  const int b = (int)(item / tiles), tile = (int)(item - (long long)b * tiles);
  const int tile_m = tile / tiles_n, tile_n = tile - tile_m * tiles_n;
  const int M = p.M, N = p.N, K = p.K, m0 = tile_m * (TM * 16), n0 = tile_n * (TN * 16);
  const int8_t* A = p.A + (long long)b * p.strideA;
  const int8_t* B = p.B + (long long)b * p.strideB;
  v4i fa[KB][TM], fb[KB][TN];
#pragma unroll
  for (int s = 0; s < KB; ++s) {
    const int k = s * 64 + g * 16;  // K % 16 == 0: a chunk is all in or all out
    const bool in = k < K;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = n0 + j * 16 + r;  // edge rows repeat the last one; never stored
      fb[s][j] = in ? *reinterpret_cast<const v4i*>(B + (size_t)(row < N ? row : N - 1) * K + k) : v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = m0 + i * 16 + r;
      fa[s][i] = in ? *reinterpret_cast<const v4i*>(A + (size_t)(row < M ? row : M - 1) * K + k) : v4i{0, 0, 0, 0};
    }
  }
  store_scores<KIND, KB, TM, TN, false>(fa, fb, p, b, m0, n0, lane);
}

// Four waves of 64 x 64 outputs share their 2 x 128 rows through the LDS, which halves the bytes loaded and loads them as whole lines
// (160 x 512 x 512 x 128: 36.3 us with waves of 64 x 64 outputs on their own, 29.3 so; 64 x 256 outputs to a workgroup 29.4).
template <int KIND, int KB, bool STREAM>
__global__ __launch_bounds__(256) void gemm_scores_lds_kernel(GemmParams p, int tiles_m, int tiles_n) {
  constexpr int BM = 128, BN = 128, ROWS = BM + BN, COPIES = ROWS / 32;
  __shared__ __attribute__((aligned(1024))) char panel[ROWS * 128];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = tiles_m * tiles_n;
  const long long item = item_on_xcd((long long)tiles * p.batch);
  if (item < 0) return;  // the whole workgroup
  const int b = (int)(item / tiles), tile = (int)(item - (long long)b * tiles);
  const int tile_m = tile / tiles_n, tile_n = tile - tile_m * tiles_n;
  const int M = p.M, N = p.N, K = p.K;
  const int8_t* A = p.A + (long long)b * p.strideA;
  const int8_t* B = p.B + (long long)b * p.strideB;
#pragma unroll
  for (int j = 0; j < COPIES; ++j) {  // copy j of a wave: eight rows of the panel, chunk c of row q at position c ^ ((q >> 1) & 7)
    const int first = (j * 4 + wave) * 8, row = first + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
    const bool in_a = first < BM;
    const int at = in_a ? tile_m * BM + row : tile_n * BN + row - BM, last = (in_a ? M : N) - 1;
    const int8_t* src = (in_a ? A : B) + (size_t)(at < last ? at : last) * K + c * 16;
    if (c * 16 < K)
      __builtin_amdgcn_global_load_lds((const TI_GLOBAL_AS void*)src, (TI_LDS_AS void*)((TI_LDS_AS char*)panel + first * 128), 16, 0, 0);
  }
  __syncthreads();
  const int wave_m = wave >> 1, wave_n = wave & 1;
  const int pos = ((g ^ (r >> 1)) & 7) << 4;
  v4i fa[KB][4], fb[KB][4];
#pragma unroll
  for (int s = 0; s < KB; ++s) {
    const bool in = s * 64 + g * 16 < K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      fa[s][i] = *reinterpret_cast<const v4i*>(panel + (((wave_m * 64 + i * 16 + r) * 128 + pos) ^ (s << 6)));
      fb[s][i] = *reinterpret_cast<const v4i*>(panel + (((BM + wave_n * 64 + i * 16 + r) * 128 + pos) ^ (s << 6)));
      if (!in) fa[s][i] = fb[s][i] = v4i{0, 0, 0, 0};
    }
  }
  store_scores<KIND, KB, 4, 4, STREAM>(fa, fb, p, b, tile_m * BM + wave_m * 64, tile_n * BN + wave_n * 64, lane);
}

// Outputs that the last-level cache does not hold, in rows of whole lines, leave with non-temporal stores.  Scores, then P.V, and the
// same with a softmax between them, us, persistent tiles / so: 40 x 2048 x 2048 x 128 201 / 179 and 390 / 359, 160 x 640 x 640 x 64 91 / 74 and
// 160 / 148, 160 x 1024 x 1024 x 128 200 / 187 and 362 / 353.  What the cache holds the softmax finds there: 64 x 768 x 768 x 64 75 us
// with plain stores, 85 with these.
static inline bool scores_stream(const GemmParams& p) { return (double)p.M * p.N * p.batch > 64e6 && p.N % 32 == 0; }

// Sizes that the tiled kernels had before these, and on which they are ahead (us, tiles / so).
static inline bool scores_left(long long batch, long long M, long long N, long long K, long long cus) {
  const long long t64 = (M + 63) / 64 * ((N + 63) / 64) * batch, t128 = (M + 127) / 128 * ((N + 127) / 128) * batch;
  const long long t256 = (M + 255) / 256 * ((N + 255) / 256) * batch;
  const double outputs = (double)M * N * batch;
  // Rows of more than 96 bytes on 64x64 tiles.  A small wave loads three times the bytes an output, which queue from a second wave to a SIMD on
  // at K = 128 (1 x 1151 x 1151 4.03 / 5.09, 65 x 116 x 116 3.76 / 4.56, 6 x 305 x 305 3.41 / 3.81; with one to a SIMD ahead, 8 x 244 x 244 3.41 / 3.16); rows
  // through the LDS are then few workgroups of 128x128 (12 x 368 x 368 x 128 4.21 / 5.45).  Not where most of those tiles is padding.
  if (K > 96 && 2 * t128 < cus) {
    if (K > 112 && (M + 15) / 16 * ((N + 31) / 32) * batch > 4 * cus && outputs > 0.5 * 4096.0 * (double)t64) return true;
    if (outputs > 1.6e6) return true;
  }
  // K that 64 does not divide, rows of whole lines: one round of 256x256 tiles with the same padding as four of 128x128 each, more than a
  // quarter of it (204 x 160 x 160 x 80 10.6 / 12.3, 228 x 223 x 192 x 80 12.4 / 13.1; full ones 16 x 1024 x 1024 x 112 14.9 / 13.6).  (128x128 tiles
  // that fill two to a CU would have some 5 % as well: 5 x 1217 x 1216 x 80 8.69 / 9.36; 27 x 512 x 512 x 80, which stays,
  // 8.67 / 8.81.)
  if (K > 64 && K % 64 != 0 && N % 32 == 0 && 4 * t256 > 3 * cus && t256 <= cus && t128 == 4 * t256 &&
      outputs < 0.72 * 65536.0 * (double)t256)
    return true;
  return false;
}

// Whether the problem is one of these (operands in aligned 16-byte chunks; the caller checked that).  Not a few hundred keys of many
// heads that fill most of that cache, in whole lines and whole steps of the persistent tiles: alone the scores are ahead here too, but they
// leave more of it dirty to the launch behind them.  Scores and P.V, and with the softmax between them, us, tiles / scores: 160 x 512 x 512 x 128
// 51.6 / 57.0 and 83.1 / 89.0, 226 x 448 x 448 x 64 60.3 / 64.5 and 98.8 / 104.3, 286 x 448 x 448 x 128 91.1 / 94.0 and 148 / 145; others of
// these sizes would be ahead, the smaller and those whose last round of tiles is short: 160 x 448 x 448 x 128 72.7 / 68.1 with the softmax, 120 x 576 x 576 x 128
// 107 / 82, 240 x 384 x 384 x 64 80.9 / 74.5.
static inline bool scores_take(const GemmParams& p) {
  if (p.M <= 16 || p.K <= 0 || p.K > 128 || p.lda != p.K || p.ldb != p.K || p.out_d != 0) return false;
  if (p.N == 128 && p.K == 128 && p.M >= 512 && (long long)((p.M + 255) / 256) * p.batch >= 2 * num_cus()) return false;  // tiles of 256x128: launch_kind
  if ((double)p.M * p.N * p.batch > 30e6 && !scores_stream(p) && p.N % 32 == 0 && p.K % 64 == 0 && p.M > 128 && p.N > 128 && p.N < 640) return false;
  return !scores_left(p.batch, p.M, p.N, p.K, num_cus());
}

enum ScoresForm { SCORES_16x32 = 0, SCORES_32x32, SCORES_LDS, SCORES_LDS_STREAM };
static constexpr const char* kScoresForms[] = {"16x32 to a wave", "32x32 to a wave", "rows through the LDS", "rows through the LDS, non-temporal stores"};

// Few outputs: the smallest waves, up to two to a SIMD (13 x 158 x 158 x 64 2.9 us, with 32 x 32 outputs to a wave 3.2, through the LDS
// 4.8; 132 x 120 x 120 x 64, four to a SIMD, 4.9 / 4.7 / 6.0).  Then 32 x 32 while the bytes loaded for each output weigh less than the LDS
// and its barrier, the sooner the longer K: 213 x 341 x 341 x 64 19.3, through the LDS 20.2, 243 x 667 x 667 x 64 157 / 131; 20 x 462 x 462 x 80
// 7.7 / 8.0, 13 x 741 x 741 x 80 9.8 / 9.5; 24 x 256 x 256 x 128 5.3 / 5.7, 245 x 87 x 87 x 128 7.0 / 6.3.
static inline ScoresForm scores_form(const GemmParams& p) {
  if ((long long)((p.M + 15) / 16) * ((p.N + 31) / 32) * p.batch <= 8LL * num_cus()) return SCORES_16x32;
  if ((double)p.M * p.N * p.batch <= (p.K <= 64 ? 24e6 : p.K <= 96 ? 5e6 : 1.6e6)) return SCORES_32x32;
  return scores_stream(p) ? SCORES_LDS_STREAM : SCORES_LDS;
}

template <int KIND, int KB>
static int launch_scores_k(const GemmParams& p, hipStream_t stream) {
  auto launch = [&](auto kern, int bm, int bn, int each) -> int {
    const int tiles_m = (p.M + bm - 1) / bm, tiles_n = (p.N + bn - 1) / bn;
    dim3 grid;
    if (int rc = xcd_grid(((long long)tiles_m * tiles_n * p.batch + each - 1) / each, 256, grid)) return rc;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, p, tiles_m, tiles_n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
    return TI_OK;
  };
  const ScoresForm form = scores_form(p);
  g_last_form = kScoresForms[form];
  if (form == SCORES_16x32) return launch(gemm_scores_kernel<KIND, KB, 1, 2>, 16, 32, 4);
  if (form == SCORES_32x32) return launch(gemm_scores_kernel<KIND, KB, 2, 2>, 32, 32, 4);
  return form == SCORES_LDS_STREAM ? launch(gemm_scores_lds_kernel<KIND, KB, true>, 128, 128, 1)
                                   : launch(gemm_scores_lds_kernel<KIND, KB, false>, 128, 128, 1);
}

template <int KIND>
static int launch_scores(const GemmParams& p, hipStream_t stream) {
  g_last_kernel = "scores";
  return p.K <= 64 ? launch_scores_k<KIND, 1>(p, stream) : launch_scores_k<KIND, 2>(p, stream);
}

}  // namespace ti
