// Batched products of operands whose rows are not whole aligned 16-byte chunks: K that 16 does not divide (P.V over a source
// length of any value), or operands that begin anywhere.  Included by gemm_s8_impl.h (epilogues, tile order).
//
// A lane reads a run of consecutive bytes of its row as the dwords they lie in, and shifts them into place: 16-byte loads at byte
// addresses work but take 1.7 times as long (200 heads, 1 x 2003 x 128: 25.6 us, at multiples of 4 bytes 15.1).  Those dwords hold a
// byte of the run each, so a load never touches memory that the operand does not share a dword with.  What is left of a row behind
// its last whole step comes from the 16 bytes that end with the row, or from the dwords of a shorter one (byte by byte, 5 x 152 x 80 x 15 took
// 11.5 us, so 4.4), zeros behind it.
// Against a thread to an output (below 2^26 products) or copies with a padded K (four launches, the operands' bytes twice over), us:
// 18 x 130 x 64 x 130 25.5 -> 4.9, 100 x 301 x 80 x 301 32.7 -> 10.9, 160 x 517 x 128 x 517 77.4 -> 31.4, 32 x 2045 x 128 x 2045 142 -> 54;
// the copies are ahead from about M N = 1024 (M + N) on (4 x 2048 x 2048 x 4097 133 us against 142), and the callers make them there.
#pragma once

namespace ti {

typedef v4i v4i_any __attribute__((aligned(1)));

// bytes k .. k + 15 of a row of K bytes, zeros from K on
__device__ __forceinline__ v4i row_chunk(const int8_t* row, int k, int K) {
  if (k + 16 <= K) return *reinterpret_cast<const v4i_any*>(row + k);
  v4i out = {0, 0, 0, 0};
  if (k >= K) return out;
  if (K >= 16) {
    const v4i last = *reinterpret_cast<const v4i_any*>(row + K - 16);
    const unsigned __int128 bits = __builtin_bit_cast(unsigned __int128, last) >> (8 * (k + 16 - K));
    return __builtin_bit_cast(v4i, bits);
  }
  // rows shorter than a chunk (k = 0): the dwords that hold a byte of it, the last one again in the place of those behind
  const unsigned shift = (unsigned)(reinterpret_cast<uintptr_t>(row) & 3);
  const int* at = reinterpret_cast<const int*>(row - shift);
  const int last = (int)(shift + K - 1) >> 2;
  int d[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) d[i] = at[i < last ? i : last];
#pragma unroll
  for (int v = 0; v < 4; ++v) out[v] = (int)__builtin_amdgcn_alignbyte((unsigned)d[v + 1], (unsigned)d[v], shift);
  const int cut = 8 * (16 - K);
  return __builtin_bit_cast(v4i, __builtin_bit_cast(unsigned __int128, out) << cut >> cut);
}

// 4 n consecutive bytes of a row from p on: the aligned dwords that hold them, one more than n where p is not aligned.
template <int DWORDS>
struct Run {
  int d[DWORDS + 1];
  __device__ __forceinline__ void load(const int8_t* p) {  // p's low two bits: `shift` of the row
    const int8_t* at = p - (reinterpret_cast<uintptr_t>(p) & 3);
#pragma unroll
    for (int q = 0; q < DWORDS / 4; ++q) {
      typedef v4i v4i_dwords __attribute__((aligned(4)));
      const v4i w = *reinterpret_cast<const v4i_dwords*>(at + q * 16);
#pragma unroll
      for (int v = 0; v < 4; ++v) d[q * 4 + v] = w[v];
    }
    // an aligned run ends with its last dword
    d[DWORDS] = *reinterpret_cast<const int*>(at + ((reinterpret_cast<uintptr_t>(p) & 3) ? DWORDS * 4 : DWORDS * 4 - 4));
  }
  __device__ __forceinline__ void load_tail(const int8_t* row, int k, int K) {  // in place already: shift 0
#pragma unroll
    for (int q = 0; q < DWORDS / 4; ++q) {
      const v4i w = row_chunk(row, k + q * 16, K);
#pragma unroll
      for (int v = 0; v < 4; ++v) d[q * 4 + v] = w[v];
    }
    d[DWORDS] = 0;
  }
  __device__ __forceinline__ v4i chunk(int q, int shift) const {
    v4i out;
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = (int)__builtin_amdgcn_alignbyte((unsigned)d[q * 4 + v + 1], (unsigned)d[q * 4 + v], shift);
    return out;
  }
};

// Work item of a workgroup: the ids congruent modulo 8 share an XCD, whose L2 then keeps the operand that the tiles of a batch
// have in common.  -1 for the ids beyond the last item (the grid is a multiple of 8, xcd_grid).
static constexpr int XCD_ROW_BITS = 20;
__device__ __forceinline__ long long item_on_xcd(long long items) {
  const long long id = ((long long)blockIdx.y << XCD_ROW_BITS) + blockIdx.x, per = (items + 7) / 8, item = (id & 7) * per + (id >> 3);
  return (id >> 3) < per && item < items ? item : -1;
}

// Tiles of BM x BN on four waves (2 x 2), K in steps of 128 bytes through registers into two LDS stages; rows as in
// gemm_pipe16q_kernel: chunk c of row r at position c ^ ((r >> 1) & 7).
template <int BM_, int BN_, int KIND_>
struct AnyCfg {
  static constexpr int BM = BM_, BN = BN_, KIND = KIND_, WAVES_M = 2, WAVES_N = 2, NT = 256;
  static constexpr int WTM = BM / 2, WTN = BN / 2, TM = WTM / 16, TN = WTN / 16;
  static constexpr int ROWS = BM + BN, SLOTS = ROWS / 32, STAGE_BYTES = ROWS * 128, LDS_BYTES = 2 * STAGE_BYTES;
  static_assert(BM % 32 == 0 && BN % 32 == 0, "a slot is 32 rows of one operand");
};

template <class Cfg>
__global__ __launch_bounds__(256) void gemm_any_kernel(GemmParams p, int tiles_m, int tiles_n) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, SLOTS = Cfg::SLOTS;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wave_m = wave >> 1, wave_n = wave & 1;
  const int tiles = tiles_m * tiles_n;
  const long long item = item_on_xcd((long long)tiles * p.batch);
  if (item < 0) return;  // the whole workgroup, before its first barrier
  const int b = (int)(item / tiles), tile = (int)(item - (long long)b * tiles);
  const int tile_m = tile / tiles_n, tile_n = tile - tile_m * tiles_n;
  const int M = p.M, N = p.N, K = p.K;
  const int8_t* A = p.A + (long long)b * p.strideA;
  const int8_t* B = p.B + (long long)b * p.strideB;

  const int chunk = tid & 7;
  const int8_t* src[SLOTS];
  int at[SLOTS];
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int row = i * 32 + (tid >> 3);
    const bool in_a = i * 32 < BM;
    const int r = in_a ? tile_m * BM + row : tile_n * BN + row - BM;
    const int last = (in_a ? M : N) - 1;  // edge rows repeat the last one; never stored
    src[i] = (in_a ? A : B) + (size_t)(r < last ? r : last) * K;
    at[i] = row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4);
  }
  const int KT = (K + 127) / 128;
  auto load = [&](int kt, v4i (&reg)[SLOTS]) {
    if (kt * 128 + 128 <= K) {  // uniform: all steps but a last one
#pragma unroll
      for (int i = 0; i < SLOTS; ++i) reg[i] = *reinterpret_cast<const v4i_any*>(src[i] + kt * 128 + chunk * 16);
    } else {
#pragma unroll
      for (int i = 0; i < SLOTS; ++i) reg[i] = row_chunk(src[i], kt * 128 + chunk * 16, K);
    }
  };
  auto store = [&](int kt, const v4i (&reg)[SLOTS]) {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) *reinterpret_cast<v4i*>(smem + (kt & 1) * Cfg::STAGE_BYTES + at[i]) = reg[i];
  };

  const int r = lane & 15, g = lane >> 4, pos = ((g ^ (r >> 1)) & 7) << 4;
  const int a_frag = (wave_m * Cfg::WTM + r) * 128 + pos, b_frag = (BM + wave_n * Cfg::WTN + r) * 128 + pos;
  v4i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
  auto multiply = [&](int kt) {
    const char* st = smem + (kt & 1) * Cfg::STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      v4i fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = *reinterpret_cast<const v4i*>(st + ((a_frag ^ (s << 6)) + i * 2048));
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j] = *reinterpret_cast<const v4i*>(st + ((b_frag ^ (s << 6)) + j * 2048));
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
  };

  // one step ahead: what is on its way two steps ahead takes the registers of a workgroup (three workgroups of 64x128 to a CU, then one: 160 x 516 x 128 x 516 28.0 -> 53.5 us)
  v4i reg[SLOTS];
  load(0, reg);
  store(0, reg);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const bool more = kt + 1 < KT;
    if (more) load(kt + 1, reg);
    multiply(kt);
    if (more) store(kt + 1, reg);
    __syncthreads();
  }
  store_tile16<Cfg>(acc, p, b, tile_m, tile_n, wave_m, wave_n, lane);
}

// Up to 16 rows (decode steps): a workgroup owns 16 rows of B, its waves take 256-byte blocks of K in turn and meet in the LDS.
// Bound by the bytes of B: 200 heads, 1 x 128 x 2003 408 -> 13.5 us, 320 heads, 1 x 128 x 2047 79.4 (copies padded by zeros) -> 23.2.
static constexpr int ANY_BLOCKS = 2;  // blocks of a wave in flight
template <int KIND>
__global__ __launch_bounds__(1024) void gemm_any_skinny_kernel(GemmParams p, int strips) {
  extern __shared__ int red[];  // [waves - 1][256]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const long long item = item_on_xcd((long long)strips * p.batch);
  if (item < 0) return;
  const int b = (int)(item / strips), n0 = (int)(item - (long long)b * strips) * 16;
  const int M = p.M, N = p.N, K = p.K;
  const int8_t* x = p.A + (long long)b * p.strideA + (size_t)(r < M ? r : M - 1) * K;
  const int8_t* w = p.B + (long long)b * p.strideB + (size_t)(n0 + r < N ? n0 + r : N - 1) * K;
  // lane (r, g) holds bytes 64 g .. 64 g + 63 of a block of its rows, 16 to a matrix instruction: the same ones of both operands
  const int shift_w = (int)(reinterpret_cast<uintptr_t>(w) & 3), shift_x = (int)(reinterpret_cast<uintptr_t>(x) & 3);
  v4i acc = {0, 0, 0, 0};
  auto multiply = [&](const Run<16>& fw, const Run<16>& fx, int sw, int sx) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw.chunk(j, sw), fx.chunk(j, sx), acc, 0, 0, 0);
  };
  int k = wave * 256;
  const int step = waves * 256;
  for (; k + (ANY_BLOCKS - 1) * step + 256 <= K; k += ANY_BLOCKS * step) {
    Run<16> fw[ANY_BLOCKS], fx[ANY_BLOCKS];
#pragma unroll
    for (int i = 0; i < ANY_BLOCKS; ++i) fw[i].load(w + k + i * step + g * 64);
#pragma unroll
    for (int i = 0; i < ANY_BLOCKS; ++i) fx[i].load(x + k + i * step + g * 64);
#pragma unroll
    for (int i = 0; i < ANY_BLOCKS; ++i) multiply(fw[i], fx[i], shift_w, shift_x);
  }
  for (; k < K; k += step) {
    Run<16> fw, fx;
    if (k + 256 <= K) {
      fw.load(w + k + g * 64);
      fx.load(x + k + g * 64);
      multiply(fw, fx, shift_w, shift_x);
    } else {
      fw.load_tail(w, k + g * 64, K);
      fx.load_tail(x, k + g * 64, K);
      multiply(fw, fx, 0, 0);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) red[(wave - 1) * 256 + v * 64 + lane] = acc[v];
  }
  __syncthreads();
  if (wave > 0) return;
  for (int i = 0; i < waves - 1; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] += red[i * 256 + v * 64 + lane];
  if (r < M) store_skinny_tile<KIND>(acc, p, b, r, n0 + 4 * g);
}

// ------------------------------------------------------------------ host side

// The grid of so many items: one row, or rows of 2^20 workgroups where one would have 2^32 threads or more, of which a launch starts only the
// remainder, without an error (65535 batches of 16448 x 1 outputs: 65280 of 16.8 million workgroups).
static inline int xcd_grid(long long items, int threads, dim3& grid) {
  const long long groups = (items + 7) / 8 * 8, rows = (groups >> XCD_ROW_BITS) + 1;
  if (groups * threads < 1LL << 32) grid = dim3((unsigned)groups);
  else if (rows <= 65535) grid = dim3(1u << XCD_ROW_BITS, (unsigned)rows);
  else return fail(TI_ERR_INVALID_ARG, "too many output tiles (%lld)", items);
  return TI_OK;
}

template <class Cfg>
static int launch_any_tiles(const GemmParams& p, hipStream_t stream) {
  const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
  dim3 grid;
  if (int rc = xcd_grid((long long)tiles_m * tiles_n * p.batch, Cfg::NT, grid)) return rc;
  hipLaunchKernelGGL(gemm_any_kernel<Cfg>, grid, dim3(Cfg::NT), Cfg::LDS_BYTES, stream, p, tiles_m, tiles_n);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
  return TI_OK;
}

template <int KIND>
static int launch_scalar(const GemmParams& p, hipStream_t stream) {
  const long long total = (long long)p.M * p.N;
  const dim3 grid((unsigned)((total + 255) / 256), 1, p.batch);
  hipLaunchKernelGGL(gemm_scalar_kernel<KIND>, grid, dim3(256), 0, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
  return TI_OK;
}

// Forms of such a product (ti_last_kernel_form; the family is "any_skinny" up to 16 rows, else "any").
enum AnyForm { ANY_THREADS = 0, ANY_SKINNY, ANY_64x64, ANY_64x128, ANY_128x128 };
static constexpr const char* kAnyForms[] = {"a thread to an output", "strips of 16", "64x64", "64x128", "128x128"};

// Tiles: bound by latency and by what the steps of the workgroups of a CU take from one another, us a step of 128 bytes: 64x64 0.5 a
// workgroup and 0.9 at least, 64x128 0.84 and 1.1, 128x128 1.38 and 1.4 (1001 bytes of K: 4 x 2000 x 2000 64.6 / 54.1 / 44.2 us on the
// three; 2 x 1000 x 1000 x 5001 37.1 / 45.9 / 56.3; 18 x 130 x 64 x 130 4.9 / 6.6 / 9.3; 64 x 777 x 80 x 777 32.1 / 33.2 / 27.1).  Five of 64x64 to a CU for 32-bit
// outputs as well, of which registers allow four: of 6957 products, 49 to 2047 bytes of K, the choice is 1.020 times the best, priced at four 1.023.
//
// A short K of few outputs is a chain of a few latencies, which a thread to an output has fewer of: us, so / on the tiles 13 x 18 x 80 x 15
// 3.0 / 4.4, 5 x 40 x 128 x 24 3.5 / 4.1, 3 x 33 x 80 x 33 4.25 / 4.26; on the strips 64 x 1 x 128 x 7 2.5 / 3.1, 4 x 1 x 128 x 20 3.0 / 3.0.  Beyond
// that its time grows with every byte of every output: 61 x 61 outputs of 36 heads, K = 32, 9.9 / 4.7.  Fitted to 5517 products with K below 48:
// 0.80 times the time of a thread to an output everywhere, and 1.004 times the better of the two.
static inline AnyForm any_form(long long batch, long long M, long long N, long long K, int out_bytes, long long cus) {
  const long long strips = (N + 15) / 16 * batch;
  auto price = [&](int bm, int bn, int resident, double each, double least) {
    const long long tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * batch, slots = cus * resident;
    const long long rest = (tiles % slots + cus - 1) / cus;
    const double last = rest == 0 ? 0.0 : rest * each > least ? rest * each : least;
    return (double)(tiles / slots) * resident * each + last;
  };
  const double small = price(64, 64, 5, 0.5, 0.9), wide = price(64, 128, 3, 0.84, 1.1), large = price(128, 128, 2, 1.38, 1.4);
  if (K > 0 && K < 48) {
    auto longer = [](double a, double b) { return a > b ? a : b; };
    const double steps = small < wide ? (small < large ? small : large) : wide < large ? wide : large;
    const double outputs = (double)M * N * batch, threads = (double)((M * N + 255) / 256 * 256) * batch;
    const double by_threads = longer((M <= 16 ? 1.75 : 2.0) + 0.064 * K, 2.1 + threads * (0.77 + 0.74 * K) * 1e-6);
    const double others = M <= 16  ? longer(3.0, 3.1 + strips * 4e-4)
                          : K < 16 ? longer(4.2, 2.1 + 2.6 * steps + 1.5e-7 * outputs * out_bytes) * (1.0 + 1.0 / K)
                                   : longer(4.3, 2.7 + 2.0 * steps + 2.1e-7 * outputs * out_bytes);
    if (by_threads < 0.97 * others) return ANY_THREADS;
  }
  if (M <= 16) return ANY_SKINNY;
  return small <= wide && small <= large ? ANY_64x64 : wide <= large ? ANY_64x128 : ANY_128x128;
}

template <int KIND>
static int launch_any(const GemmParams& p, hipStream_t stream) {
  const AnyForm form = any_form(p.batch, p.M, p.N, p.K, (int)sizeof(typename Epi<KIND>::Out), num_cus());
  g_last_kernel = p.M <= 16 ? "any_skinny" : "any";
  g_last_form = kAnyForms[form];
  if (form == ANY_THREADS) return launch_scalar<KIND>(p, stream);
  if (form == ANY_SKINNY) {
    const int strips = (p.N + 15) / 16;
    const long long items = (long long)strips * p.batch;
    // waves to cover the latency of the loads, each with a block of K at least
    long long waves = (4096 + items - 1) / items;
    const long long most = (p.K + 255) / 256;
    waves = waves > most ? most : waves;
    waves = waves > 16 ? 16 : waves < 1 ? 1 : waves;
    dim3 grid;
    if (int rc = xcd_grid(items, (int)(64 * waves), grid)) return rc;
    hipLaunchKernelGGL(gemm_any_skinny_kernel<KIND>, grid, dim3((unsigned)(64 * waves)),
                       (size_t)(waves - 1) * 1024, stream, p, strips);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
    return TI_OK;
  }
  if (form == ANY_64x64) return launch_any_tiles<AnyCfg<64, 64, KIND>>(p, stream);
  if (form == ANY_64x128) return launch_any_tiles<AnyCfg<64, 128, KIND>>(p, stream);
  return launch_any_tiles<AnyCfg<128, 128, KIND>>(p, stream);
}

}  // namespace ti
