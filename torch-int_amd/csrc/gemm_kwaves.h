// Linears of some 65 to 1024 rows whose output makes one round of small tiles: the waves of a workgroup share K, not the tile.
//
// A workgroup has one tile of 32x32 to 128x64 outputs over the whole of K, and each of its waves multiplies the WHOLE tile, over every
// NW-th step of 128 bytes.  So a wave's fragments serve as many products as the tile has (a 32x32 quarter of 64x64 reads twice the LDS
// bytes a product), its panels lie in a ring of its own, and no wave waits for another until the integer sums of all of them are
// added through the LDS at the end: no barrier in the loop, no slices of K that meet in memory, no second launch, no workspace.
//
// Bound by what the copies have in flight: a step's panels are (BM + BN) * 128 bytes for few products, 0.18 (32x32) to 0.42 us (128x64)
// a step of the workgroup with weights from HBM, 0.11 (32x64) and 0.13 (64x64) with weights that the last-level cache holds, where the
// copies of a CU alone take 0.08 and 0.11.  The tiled kernels that had these shapes take one step after the other, a barrier each, on a quarter
// of the CUs (128x128 tiles), or park and add int32 slices.  Cold weights, us, before / now: 384 x 2048 x 2048 15.7 / 6.8, 512 x 2048 x 2048
// 15.8 / 7.6, 128 x 8192 x 2048 14.5 / 8.8, 128 x 2048 x 8192 20.4 / 11.3, 128 x 4096 x 4096 15.5 / 10.0, 256 x 4096 x 4096 18.1 / 12.0,
// 256 x 2560 x 2560 13.5 / 8.1, 128 x 5120 x 5120 17.9 / 13.6, 256 x 5120 x 5120 20.9 / 17.0, 1024 x 768 x 3072 17.2 / 9.6.
//
// Row tiles begin at different steps of K (`turn`): those of one column read the same weights, and so ask HBM for different lines
// of them at a time (256 x 5120 x 5120 17.7 / 16.9, 512 x 2048 x 2048 7.85 / 7.4; 256 x 4096 x 4096 12.1 / 12.3).  Tried and left: copies spread between the
// products (level), steps turned by column tile or by workgroup (level), the same tiles with their waves side by side and up to ten stages
// (384 x 2048 x 2048 9.0, 128 x 4096 x 4096 11.7).
#pragma once

namespace ti {

// NW waves, each with a ring of STAGES steps
template <int BM_, int BN_, int NW_, int STAGES_, int KIND_, bool GROUPED_ = false>
struct KWavesCfg {
  static constexpr int BM = BM_, BN = BN_, NW = NW_, STAGES = STAGES_, KIND = KIND_;
  static constexpr bool GROUPED = GROUPED_;
  static constexpr int NT = NW * 64;
  static constexpr int TM = BM / 16, TN = BN / 16;
  static constexpr int STAGE = (BM + BN) * QBK;
  static constexpr int COPIES = STAGE / 1024;  // copy instructions a step: eight panel rows each
  static constexpr int RING = STAGES * STAGE;
  static constexpr int LDS_BYTES = NW * RING;
  // units of the epilogue: 16 rows, halves of them where that leaves waves without one
  static constexpr int PARTS = TM < NW && TM <= 2 && TN % 2 == 0 ? 2 : 1;
  static constexpr int RESIDENT = 160 * 1024 / LDS_BYTES;  // workgroups to a CU
  static constexpr int WAVES_PER_SIMD = (RESIDENT * NW + 3) / 4;
  static_assert(BM % 16 == 0 && BN % 16 == 0, "blocks of 16x16");
  static_assert(STAGES >= 1 && STAGES <= 2, "the waits know of two");
  static_assert((STAGES - 1) * COPIES <= 63, "a wait counts in six bits");
  static_assert(TM * TN * 1024 <= RING, "a wave's sums go over its ring");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

// 16 rows of the tile, as the epilogue of gemm_pipe16q_kernel knows a wave's part
template <class Cfg>
struct KWavesUnit {
  static constexpr int BM = Cfg::BM, BN = Cfg::BN, KIND = Cfg::KIND;
  static constexpr int TM = 1, TN = Cfg::TN / Cfg::PARTS, WTM = 16, WTN = TN * 16;
};

// Four consecutive columns of an fp32 output or bias; single values where it does not begin on 16 bytes.
__device__ __forceinline__ v4f load_f32x4(const float* at, bool aligned) {
  if (aligned) return *reinterpret_cast<const v4f*>(at);
  return v4f{at[0], at[1], at[2], at[3]};
}

template <class Cfg>
__global__ __launch_bounds__(Cfg::NT, (Cfg::WAVES_PER_SIMD)) void gemm_kwaves_kernel(GemmParams p, int tiles_m, int tiles_n,
                                                                                     GemmGroup grp) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, NW = Cfg::NW, S = Cfg::STAGES, COPIES = Cfg::COPIES;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = tiles_m * tiles_n;
  const int b = Cfg::GROUPED ? (int)blockIdx.x / tiles : 0;
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x - b * tiles, tiles_m, tiles_n, tile_m, tile_n, p.band);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int rows_a = p.M - m0 < BM ? p.M - m0 : BM, rows_b = p.N - n0 < BN ? p.N - n0 : BN;
  const int8_t* W = Cfg::GROUPED ? grp.B[b] : p.B;
  // the panels as buffers (launch_kind: rows at most PANEL_MAX_LD apart): rows beyond the last read as zeros, and are not stored
  const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(p.A + (size_t)m0 * p.lda), 0, (int)((unsigned)(rows_a - 1) * (unsigned)p.lda + (unsigned)p.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(W + (size_t)n0 * p.ldb), 0, (int)((unsigned)(rows_b - 1) * (unsigned)p.ldb + (unsigned)p.K), 0x00020000);
  const int steps = p.K / QBK;
  const int n = steps > wave ? (steps - wave + NW - 1) / NW : 0;  // this wave's: wave, wave + NW, ..., all turned by `turn`
  const int turn = tile_m * steps / tiles_m;

  // ---- copies: copy j of a step fills rows 8 j .. 8 j + 7 of [A panel | B panel], chunk c of row r at position c ^ ((r >> 1) & 7)
  char* ring = smem + wave * Cfg::RING;
  const int row = lane >> 3, pos = lane & 7;
  const unsigned sw[2] = {(unsigned)((pos ^ (lane >> 4)) << 4), (unsigned)((pos ^ (4 + (lane >> 4))) << 4)};  // of even and odd copies
  const unsigned a_row = (unsigned)row * (unsigned)p.lda, b_row = (unsigned)row * (unsigned)p.ldb;
  unsigned k_at = (unsigned)((wave + turn) % steps) * QBK;
  int head = 0, issued = 0;
  auto issue = [&]() {
    TI_LDS_AS char* dst = (TI_LDS_AS char*)ring + head * Cfg::STAGE;
#pragma unroll
    for (int j = 0; j < BM / 8; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, (TI_LDS_AS void*)(dst + j * 1024), 16,
                                               a_row + sw[j & 1] + k_at + (unsigned)(8 * j) * (unsigned)p.lda, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < BN / 8; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(bres, (TI_LDS_AS void*)(dst + (BM / 8 + j) * 1024), 16,
                                               b_row + sw[j & 1] + k_at + (unsigned)(8 * j) * (unsigned)p.ldb, 0, 0, 0);
    k_at += NW * QBK;
    if (k_at >= (unsigned)p.K) k_at -= (unsigned)p.K;
    head = head + 1 == S ? 0 : head + 1;
    ++issued;
  };
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < n) issue();

  // ---- fragments: lane (r, g) reads row r of a block, chunk 4 * slice + g
  const int r = lane & 15, g = lane >> 4;
  const int at = r * QBK + (((g ^ (r >> 1)) & 7) << 4);
  v4i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
  int tail = 0;
  for (int it = 0; it < n; ++it) {
    // loads complete in order: this step has landed once at most the copies of the one behind it are on their way
    if (S == 2 && issued - it == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * COPIES) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* st = ring + tail * Cfg::STAGE;
    v4i fa[2][TM], fb[2][TN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[s][i] = *reinterpret_cast<const v4i*>(st + ((at ^ (s << 6)) + i * 16 * QBK));
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[s][j] = *reinterpret_cast<const v4i*>(st + BM * QBK + ((at ^ (s << 6)) + j * 16 * QBK));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read: its stage is free for the next
    if (issued < n) issue();
    tail = tail + 1 == S ? 0 : tail + 1;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
  }

  // What an fp32 tile that is added to holds, and the bias: of all units of a wave at once, on their way while the sums meet.  Fetched unit
  // by unit behind the sums (store_tile16), each waited for memory by itself, three times on the tallest tiles: warm weights, us, so / on 64x64 tiles over the
  // whole of K, which these rows had before / now: 804 x 2048 x 2048 14.7 / 12.1 / 11.3, 324 x 3072 x 768 8.7 / 7.8 / 6.2, 300 x 4096 x 4096 13.9, now 11.5.
  using E = Epi<Cfg::KIND>;
  using Unit = KWavesUnit<Cfg>;
  constexpr bool ADDS_F32 = E::kAccumulate && sizeof(typename E::Out) == 4;
  constexpr int UNITS = ADDS_F32 ? (TM * Cfg::PARTS + NW - 1) / NW : 1;  // of a wave, one column part
  static_assert(NW % Cfg::PARTS == 0, "a wave's units have the same columns");
  const bool vec_ok = (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0;
  const int col = n0 + wave % Cfg::PARTS * Unit::WTN + 4 * g;  // whole columns (kwaves_pick)
  auto unit_at = [&](int k, int j) {
    const int m = m0 + (wave + k * NW) / Cfg::PARTS * 16 + r;
    return static_cast<float*>(p.C) + out_index(p, m < p.M ? m : p.M - 1, col + j * 16);
  };
  v4f old[UNITS][Unit::TN], bias[Unit::TN];
  if constexpr (ADDS_F32) {
#pragma unroll
    for (int j = 0; j < Unit::TN; ++j) {
      bias[j] = load_f32x4(static_cast<const float*>(p.bias) + col + j * 16, vec_ok);
#pragma unroll
      for (int k = 0; k < UNITS; ++k) old[k][j] = load_f32x4(unit_at(k, j), vec_ok);  // rows beyond the last: row M - 1, not used
    }
  }

  // ---- the waves' sums, over the rings (every copy of this wave has landed and been read)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) *reinterpret_cast<v4i*>(ring + ((i * TN + j) * 64 + lane) * 16) = acc[i][j];
  __syncthreads();
  if constexpr (ADDS_F32) {
#pragma unroll
    for (int k = 0; k < UNITS; ++k) {
      const int u = wave + k * NW, i = u / Cfg::PARTS, c = u - i * Cfg::PARTS;
      if (u >= TM * Cfg::PARTS || m0 + 16 * i >= p.M) break;
      const char* first = smem + ((i * TN + c * Unit::TN) * 64 + lane) * 16;
#pragma unroll
      for (int j = 0; j < Unit::TN; ++j) {
        v4i sum = *reinterpret_cast<const v4i*>(first + j * 1024);
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += *reinterpret_cast<const v4i*>(first + w * Cfg::RING + j * 1024);
        v4f out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out[v] = old[k][j][v] + E::apply(sum[v], E::bias_term(bias[j][v], p.beta), p.alpha);
        if (m0 + 16 * i + r < p.M) {
          float* at = unit_at(k, j);
          if (vec_ok) {
            *reinterpret_cast<v4f*>(at) = out;
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) at[v] = out[v];
          }
        }
      }
    }
    return;
  }
  GemmParams q = p;
  if constexpr (Cfg::GROUPED) {
    q.bias = grp.bias[b];
    q.C = grp.C[b];
    q.alpha = grp.alpha[b];
    q.beta = grp.beta[b];
  }
  for (int u = wave; u < TM * Cfg::PARTS; u += NW) {
    const int i = u / Cfg::PARTS, c = u - i * Cfg::PARTS;
    if (m0 + 16 * i >= p.M) break;
    const char* first = smem + ((i * TN + c * Unit::TN) * 64 + lane) * 16;
    v4i sum[1][Unit::TN];
#pragma unroll
    for (int j = 0; j < Unit::TN; ++j) sum[0][j] = *reinterpret_cast<const v4i*>(first + j * 1024);
#pragma unroll
    for (int w = 1; w < NW; ++w)
#pragma unroll
      for (int j = 0; j < Unit::TN; ++j) sum[0][j] += *reinterpret_cast<const v4i*>(first + w * Cfg::RING + j * 1024);
    store_tile16<Unit>(sum, q, 0, tile_m, tile_n, i, c, lane);
  }
}

template <class Cfg>
static int launch_kwaves_cfg(const GemmParams& p, hipStream_t stream, const GemmGroup& grp) {
  static std::atomic<unsigned long long> lds_ok{0};
  if (int rc = allow_lds(gemm_kwaves_kernel<Cfg>, Cfg::LDS_BYTES, lds_ok)) return rc;
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
  const int grid = tiles_m * tiles_n * (Cfg::GROUPED ? grp.count : 1);  // kwaves_pick: a round or two
  hipLaunchKernelGGL(gemm_kwaves_kernel<Cfg>, dim3((unsigned)grid), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, p, tiles_m, tiles_n, grp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
  return TI_OK;
}

enum KWavesTile {
  KWAVES_NONE = 0, KWAVES_32x32, KWAVES_32x64, KWAVES_48x64, KWAVES_64x64, KWAVES_64x80, KWAVES_96x64, KWAVES_80x80, KWAVES_96x80, KWAVES_128x64,
  KWAVES_64x64_PAIRS
};

// Wide outputs of a long K on which the kernels that had them are ahead, if only with weights that the last-level cache holds: several rows
// of tiles read the same long rows of weights, and the tallest tiles have few copies in flight for them.  us, those / so, cold and warm weights:
// 40 million weights of a K beyond 5120 160 x 7168 x 7680 25.2 / 27.1 and 22.4 / 23.6, in the mean of 65 to 192 rows of 7168 to 8192 on both sides 1.05 and
// 1.08 times the time.  80 columns 240 x 5120 x 7680 23.8 / 25.4 and 20.7 / 24.6, 150 x 10240 x 5120 23.2 / 23.7 and 19.5 / 22.1, 100 rows 21.5 / 20.5 and
// 17.5 / 19.3, 70 x 17920 x 2560 15.9 / 15.5 and 12.6 / 13.6, 700 x 2560 x 2048 10.7 / 11.2 and 10.7 / 10.7.  64 columns of widths that 2560 does not divide 120 x 13312 x
// 5120 24.5 / 26.0 and 19.8 / 19.7.  One row of 80x80 or 96x80 tiles of 17920 and 20480 columns at K = 5120 stays: 96 x 20480 x 5120 28.8 / 28.3 and 20.2 / 22.3.
// (The epilogue that adds to fp32 is ahead on nearly all of them: its slices do not meet in one launch.)
static inline bool kwaves_behind(KWavesTile tile, long long N, long long K) {
  if (K > 5120 && N * K >= 40000000) return true;
  switch (tile) {
    case KWAVES_64x80: return K > 7168 || (K > 4096 && N > 5120);
    case KWAVES_96x80:
      if (K < 2560) return true;
      [[fallthrough]];
    case KWAVES_80x80: return N > 5120 && (N <= 10240 ? K > 2560 : K <= 4096);
    case KWAVES_128x64: return K > 4096 && N > 5120 && N % 2560 != 0;
    default: return false;
  }
}

// The tile of such a linear (or of `problems` of one shape in one launch), or none.  The first of the list that is one round of the CUs: a
// step takes as long as the panel rows of its tile, and the round as long as its steps (us, cold weights, 0.0022 a panel row and step and some 3.5; 0.0034 where the
// outputs are wider than 10240: 96 x 16384 x 4096 20.3, 96 x 20480 x 5120 28.3).  Below
// five eighths of a round the CUs stand idle (128 x 1024 x 4096 on 32x32), and in a second round larger tiles of other kernels are ahead (cold, us: 768 x
// 4096 x 4096 24.5, 26.2 here), but for groups, whose other choice are problems one after the other: there, two workgroups of two waves share a CU (pairs;
// three 300 x 2048 x 2048 19.2 apart, 13.2 so).  The tallest tiles are where the others walk K on few CUs, too: not for a short K (512 x 3072 x 768 7.3, on
// 128x64 7.8) nor for a long one (1024 x 2048 x 8192 27.8, on 128x64 28.1); 128x80 are level with those others (128 x 20480 x 5120 32.7 / 32.2, 1024 x 2560 x 2560
// 16.2 / 16.9).
// K beyond 8192: the slices are ahead, or level (128 x 2560 x 10240 19.1 / 20, 256 x 4096 x 16384 34.6 / 34).
// Widths: multiples of 2560 and 1024 (but for those that three divides, which have 192 and 288 columns wide tiles of their own), less what kwaves_behind
// leaves, or of 768 on both sides.  K = 1024, other widths and 257 to 512 rows of K from 3072 on without an accumulating epilogue (multiples of 2560 are taken) stay
// with the kernels that had them: a line drawn where the tests of those kernels reach their forms, not by time, of which this kernel would take 0.6 to 0.9 there (384 x 4096 x 4096 17.6, 14.9 so).
// The 96x64 tiles of a K of 768 are level to behind with weights and old outputs that the cache holds, for fp32 outputs alone (324 x 3072 x 768 warm 6.1 / 6.4, cold level).
static inline KWavesTile kwaves_pick(long long M, long long N, long long K, bool accumulates, int problems = 1, bool adds_f32 = false) {
  if (M <= TI_ROWS_MAX_M || M > 4096 || N < 768 || N > 20480 || K > 8192) return KWAVES_NONE;
  if (problems > 1 && K < 2048) return KWAVES_NONE;
  const bool short_rows = N % 768 == 0 && K % 768 == 0 && K <= 3072;
  auto wide = [](long long w) { return w % 2560 == 0 || (w % 1024 == 0 && w % 3 != 0); };
  if (!short_rows && !(wide(N) && wide(K) && K >= 2048)) return KWAVES_NONE;
  if (!accumulates && K >= 3072 && N % 2560 != 0 && M > (K > 5120 ? 255 : 256) && M <= 512) return KWAVES_NONE;
  const long long cus = num_cus();
  struct Form { KWavesTile tile; int bm, bn, k_from, k_to; };
  static constexpr Form kForms[] = {
      {KWAVES_32x32, 32, 32, 0, 8192}, {KWAVES_32x64, 32, 64, 0, 8192}, {KWAVES_48x64, 48, 64, 0, 8192}, {KWAVES_64x64, 64, 64, 0, 8192},
      {KWAVES_64x80, 64, 80, 0, 8192}, {KWAVES_96x64, 96, 64, 0, 8192}, {KWAVES_80x80, 80, 80, 2048, 5120}, {KWAVES_96x80, 96, 80, 2048, 5120},
      {KWAVES_128x64, 128, 64, 2048, 5120}};
  for (const Form& f : kForms) {
    if (N % f.bn != 0) continue;
    const long long tiles = (M + f.bm - 1) / f.bm * (N / f.bn) * problems;
    if (tiles > cus || K < f.k_from || K > f.k_to) continue;
    if (problems == 1 && !adds_f32 && kwaves_behind(f.tile, N, K)) return KWAVES_NONE;
    return 8 * tiles >= 5 * cus ? f.tile : KWAVES_NONE;
  }
  return problems > 1 && (M + 63) / 64 * (N / 64) * problems <= 2 * cus ? KWAVES_64x64_PAIRS : KWAVES_NONE;
}

// Whether it goes before the weight-streaming kernel, which has narrow outputs of more than 64 rows else: from six of that kernel's blocks of rows on
// its workgroups come in twos to a CU, or with four blocks each (us, before / now: 128 x 2048 x 2048 5.1 / 4.8, 96 x 2048 x 2048 4.7 / 4.9, 96 x 2560 x 2560 8.7 / 6.2,
// 128 x 2560 x 2560 8.6 / 7.9).
static inline bool kwaves_before_rows(long long M, long long N, long long K, int problems = 1) {
  return M > (N > 2048 ? 95 : 96) && M <= 128 && K >= 2048 && K < 3072 && kwaves_pick(M, N, K, false, problems) != KWAVES_NONE;
}

template <int KIND, bool GROUPED>
static int launch_kwaves(KWavesTile tile, const GemmParams& p, hipStream_t stream, const GemmGroup& grp = GemmGroup{}) {
  g_last_form = "gemm_kwaves";
  switch (tile) {
    case KWAVES_32x32: return launch_kwaves_cfg<KWavesCfg<32, 32, 8, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_32x64: return launch_kwaves_cfg<KWavesCfg<32, 64, 8, 1, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_48x64: return launch_kwaves_cfg<KWavesCfg<48, 64, 4, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_64x64: return launch_kwaves_cfg<KWavesCfg<64, 64, 4, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_64x80: return launch_kwaves_cfg<KWavesCfg<64, 80, 4, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_96x64: return launch_kwaves_cfg<KWavesCfg<96, 64, 4, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_80x80: return launch_kwaves_cfg<KWavesCfg<80, 80, 4, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_96x80: return launch_kwaves_cfg<KWavesCfg<96, 80, 3, 2, KIND, GROUPED>>(p, stream, grp);
    case KWAVES_128x64: return launch_kwaves_cfg<KWavesCfg<128, 64, 3, 2, KIND, GROUPED>>(p, stream, grp);
    default:
      if constexpr (GROUPED) {
        g_last_form = "gemm_kwaves pairs";
        return launch_kwaves_cfg<KWavesCfg<64, 64, 2, 2, KIND, GROUPED>>(p, stream, grp);
      }
      return fail(TI_ERR_INVALID_ARG, "no tile for waves that share K");
  }
}

static inline const char* kwaves_name(KWavesTile tile) {
  static constexpr const char* kNames[] = {"", "mid_waves_32x32", "mid_waves_32x64", "mid_waves_48x64", "mid_waves_64x64", "mid_waves_64x80", "mid_waves_96x64",
                                           "mid_waves_80x80", "mid_waves_96x80", "mid_waves_128x64", "mid_waves_64x64"};
  return kNames[tile];
}

}  // namespace ti
