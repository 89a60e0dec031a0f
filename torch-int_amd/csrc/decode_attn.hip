// Attention for incremental decoding in one launch (two kernels: one for a single new token, decode_attn_one_kernel, and
// one for up to four): per (batch, head) one workgroup appends the new
// key / value rows to the KV cache, computes alpha_qk * Q.K^T over the whole cache, turns the scores into
// int8 probabilities (mask, clamp, softmax, *127, round: the arithmetic and the summation order of
// attn_softmax_q) and multiplies them with V as the cache stores it ([len, head_dim] rows).  It replaces
// the append, skinny Q.K^T, softmax and row-major P.V launches of a decode step; the scores and the
// probabilities stay in LDS.  HBM-bound on the 2 * len * head_dim bytes of cache per (batch, head).
//
// A cache row is read by head_dim/16 adjacent lanes (16 bytes each), so one load
// instruction of a wave covers 64*16/head_dim whole rows; partial dot products meet through lane
// shuffles (integers: any order gives the same bits).
#include "ti_common.h"
#include "softmax_math.h"

namespace ti {

constexpr int DA_MAX_T = 4;         // query rows per (batch, head)
constexpr int DA_LDS_LIMIT = 60 * 1024;

__device__ __forceinline__ int dot16(v4i a, v4i b, int c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_sdot4(a[i], b[i], c, false);
  return c;
}

// Sum over the LPR (4 or 8) adjacent lanes that share a cache row, through DPP lane permutes: within quads
// (lane ^ 1, lane ^ 2), then across the two quads of an 8-lane group (mirror of the half row).
template <int LPR>
__device__ __forceinline__ int row_sum(int a) {
  a += __builtin_amdgcn_mov_dpp(a, 0xB1, 0xf, 0xf, true);  // quad_perm [1,0,3,2]
  a += __builtin_amdgcn_mov_dpp(a, 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
  if (LPR == 8) a += __builtin_amdgcn_mov_dpp(a, 0x141, 0xf, 0xf, true);  // row_half_mirror
  return a;
}

// This wave's LDS traffic is done, then the workgroup's barrier; loads of the cache stay in flight across it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One new token (T == 1): the whole cache of the (batch, head) is in flight at once.  NW waves, at most NI row groups
// each; row s of the cache is row slot s % RPW of wave (s / RPW) % NW, group s / (RPW * NW).
//
// Bound by HBM for a batch of users, by the chain load - maximum - sum - product - sum for a single one, and laid out for
// both: all key loads are issued up front and all value loads before the softmax, which covers their latency;
// a lane keeps "its" scores (group u belongs to lane u % LPR of the row) in registers from the product to the
// exponential, so the maximum and the exponentials need no pass over the LDS; probabilities become the bytes of a
// v_dot4 operand and four value rows are transposed in registers (8 v_perm_b32 for 16 bytes of four rows), 12
// instructions for 16 products instead of 32; the row slots of a wave meet through v_permlane swaps, which halve the
// values left at every step.
// Measured, cold caches, us (before: decode_attn_kernel): head size 128, heads x positions, 40 x 508 10.7 -> 5.6, 32 x 108
// 7.8 -> 3.8, 128 x 904 21.5 -> 10.3, 768 x 250 20.0 -> 10.9, 768 x 904 36.5 -> 32.1 (5.5 TB/s), 128 x 2000 40.4 -> 18.3; head size
// 64, 12 x 108 7.7 -> 3.6, 576 x 500 20.0 -> 10.8.
// LDS: exponentials [Sp], maxima [NW], scale, probabilities as bytes [NW][RPW][NIP], partial outputs [NW][D].
// MOVE: the rows before the new one are read from k_past / v_past and written into the buffers on the way, which saves a pass of
// its own over the cache where it has to go to a buffer with room (the first step after a prefill, a full buffer): 768 heads x
// 901 positions 75 us (4.7 TB/s of reads and writes) instead of two strided copies of 54 us and a step of 33, eight tokens of 24
// sequences on 16 layers of OPT-6.7B's width 14.50 -> 13.50 ms.  A form of its own, so that the stores do not stand between
// the products of the other steps.
template <int D, int NW, int NI, bool PART, bool MOVE>
__global__ __launch_bounds__(NW * 64, 4) void decode_attn_one_kernel(
    const int8_t* __restrict__ q, const int8_t* __restrict__ k_new, const int8_t* __restrict__ v_new, int8_t* k_buf,
    int8_t* v_buf, const float* __restrict__ mask, int8_t* __restrict__ ctx, int8_t* __restrict__ probs_out, int S_arg,
    long long cap, int heads, float alpha_qk, float alpha_pv, const int* __restrict__ s_dev, int dr_arg,
    const int8_t* k_past, const int8_t* v_past, long long past_cap) {
  constexpr int LPR = D / 16;                // lanes per cache row
  constexpr int RPW = 64 / LPR;              // rows per wave per load
  constexpr int STEP = NW * RPW;             // rows per group
  constexpr int NJ = (NI + LPR - 1) / LPR;   // scores a lane keeps
  constexpr int NIP = (NI + 3) / 4 * 4;
  __shared__ __attribute__((aligned(16))) float ex[NI * STEP];
  __shared__ __attribute__((aligned(16))) float wmax[NW];
  __shared__ float scale_of_row;
  __shared__ __attribute__((aligned(16))) int8_t pb[NW * RPW * NIP];
  __shared__ __attribute__((aligned(16))) int red[NW * D];

  const int dr = PART ? dr_arg : D;
  int S = S_arg;
  if (s_dev != nullptr) {  // clamped to the contract, as below
    S = s_dev[0];
    S = S < 1 ? 1 : S;
    S = S > S_arg ? S_arg : S;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rs = lane / LPR, cs = lane % LPR;
  const bool in_row = !PART || cs * 16 < dr;
  const long long bh = blockIdx.x;
  const bool grow = k_new != nullptr;         // the last row comes from k_new / v_new and goes into the cache
  const int S_old = grow ? S - 1 : S;
  int8_t* kb = k_buf + bh * cap * dr;
  int8_t* vb = v_buf + bh * cap * dr;
  const int8_t* ko = MOVE ? k_past + bh * past_cap * dr : kb;  // the rows before the new one
  const int8_t* vo = MOVE ? v_past + bh * past_cap * dr : vb;
  const v4i zero = {0, 0, 0, 0};
  const int col = in_row ? cs * 16 : 0;

  const v4i qr = in_row ? *reinterpret_cast<const v4i*>(q + bh * dr + col) : zero;
  v4i fresh_k = zero, fresh_v = zero;
  if (grow) {
    fresh_k = *reinterpret_cast<const v4i*>(k_new + bh * dr + col);
    fresh_v = *reinterpret_cast<const v4i*>(v_new + bh * dr + col);
  }
  // Rows past the end re-read the last cached row (row 0 of an empty cache); groups past the end are not loaded.
  const int base = wave * RPW;
  const int last = S_old > 0 ? S_old - 1 : 0;
  auto load_rows = [&](v4i (&dst)[NI], const int8_t* buf) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      dst[u] = zero;
      if (base + u * STEP < S) {  // the same for every lane of the wave
        int s = base + u * STEP + rs;
        s = s < last ? s : last;
        dst[u] = *reinterpret_cast<const v4i*>(buf + (unsigned)(s * dr + col));
      }
    }
  };
  auto move_row = [&](int8_t* buf, int u, v4i row) {  // group u of the old rows goes into the buffer
    const int s = base + u * STEP + rs;
    if (s < S_old && in_row) *reinterpret_cast<v4i*>(buf + (unsigned)(s * dr + col)) = row;
  };
  v4i kv[NI], vv[NI];
  load_rows(kv, ko);
  // the additive mask of the scores this lane keeps, fetched together with the cache rows
  float mk[NJ];
  const float* msk = mask != nullptr ? mask + (bh / heads) * (long long)S : nullptr;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int u = j * LPR + cs, s = base + u * STEP + rs;
    mk[j] = msk != nullptr && u < NI && s < S ? msk[s] : 0.0f;
  }

  // ---- scores: max(alpha_qk * (q . k) + mask, most negative finite float)
  const float lowest = -3.402823466e+38f;
  int own[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) own[j] = 0;
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    if (base + u * STEP >= S) break;  // the same for every lane of the wave
    if (MOVE) move_row(kb, u, kv[u]);
    if (base + u * STEP <= S_old && S_old < base + u * STEP + RPW && rs == S_old - base - u * STEP) kv[u] = fresh_k;
    const int a = row_sum<LPR>(in_row ? dot16(kv[u], qr, 0) : 0);
    if (cs == u % LPR) own[u / LPR] = a;
  }
  load_rows(vv, vo);  // on their way during the softmax; together with the keys they only cost registers
  float x[NJ], m = lowest;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int u = j * LPR + cs, s = base + u * STEP + rs;
    float y = Epi<EPI_F32_SCALE>::apply(own[j], 0.0f, alpha_qk);
    if (msk != nullptr) y = y + mk[j];
    x[j] = u < NI && s < S && y > lowest ? y : lowest;
    m = m > x[j] ? m : x[j];
  }
  m = wave_max(m);
  if (lane == 0) wmax[wave] = m;
  lds_barrier();
#pragma unroll
  for (int w = 0; w < NW; ++w) m = m > wmax[w] ? m : wmax[w];

  // ---- exponentials; positions S .. the next multiple of 4 hold zeros, which change no sum
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int u = j * LPR + cs, s = base + u * STEP + rs;
    x[j] = exp_nonpos(x[j] - m);
    if (u < NI) ex[s] = s < S ? x[j] : 0.0f;
  }
  lds_barrier();
  // ---- the sum, by one wave in the order of attn_softmax_q (chunk c of four elements belongs to lane c % 64, a lane
  // adds its elements in ascending order, lanes combine with a xor butterfly 32..1)
  if (wave == 0) {
    const int nchunks = (S + 3) >> 2;
    float sum = 0.0f;
    for (int c = lane; c < nchunks; c += 64) {
      const v4f e4 = reinterpret_cast<const v4f*>(ex)[c];
#pragma unroll
      for (int j = 0; j < 4; ++j) sum = sum + e4[j];
    }
    sum = wave_sum(sum);
    if (lane == 0) scale_of_row = 127.0f / sum;
  }
  lds_barrier();
  const float scale = scale_of_row;
  // ---- probabilities: a byte per position, to the lanes of the same row of the same wave (no barrier)
  int8_t* my_pb = pb + (wave * RPW + rs) * NIP;
#pragma unroll
  for (int j = 0; j < (NIP + LPR - 1) / LPR; ++j) {
    const int u = j * LPR + cs, s = base + u * STEP + rs;
    const bool live = j < NJ && u < NI && s < S;
    const int8_t pq = live ? (int8_t)(int)__builtin_rintf(x[j < NJ ? j : 0] * scale) : (int8_t)0;
    if (u < NIP) my_pb[u] = pq;
    if (live && probs_out != nullptr) probs_out[bh * (long long)S + s] = pq;
  }
  __builtin_amdgcn_wave_barrier();

  // ---- ctx[n] = s8(alpha_pv * sum_s p[s] * v[s][n]); the lane owns columns cs*16 .. +15
  int acc[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) acc[c] = 0;
#pragma unroll
  for (int u0 = 0; u0 < NI; u0 += 4) {
    if (base + u0 * STEP >= S) break;  // the same for every lane of the wave
    const int p4 = *reinterpret_cast<const int*>(my_pb + u0);
    v4i r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = u0 + i;
      r[i] = u < NI ? vv[u < NI ? u : 0] : zero;
      if (MOVE && u < NI) move_row(vb, u, r[i]);
      if (u < NI && base + u * STEP <= S_old && S_old < base + u * STEP + RPW && rs == S_old - base - u * STEP)
        r[i] = fresh_v;
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const unsigned r0 = r[0][w], r1 = r[1][w], r2 = r[2][w], r3 = r[3][w];
      const unsigned a = __builtin_amdgcn_perm(r1, r0, 0x05010400), b = __builtin_amdgcn_perm(r3, r2, 0x05010400);
      const unsigned c = __builtin_amdgcn_perm(r1, r0, 0x07030602), d = __builtin_amdgcn_perm(r3, r2, 0x07030602);
      acc[4 * w + 0] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(b, a, 0x05040100), p4, acc[4 * w + 0], false);
      acc[4 * w + 1] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(b, a, 0x07060302), p4, acc[4 * w + 1], false);
      acc[4 * w + 2] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(d, c, 0x05040100), p4, acc[4 * w + 2], false);
      acc[4 * w + 3] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_perm(d, c, 0x07060302), p4, acc[4 * w + 3], false);
    }
  }
  // The row slots of a wave: the upper half of the lanes takes columns 8..15, the odd rows of 16 lanes 4..7 and 12..15,
  // then the lanes of a row of 16 that hold the same columns.
  int h8[8], h4[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const auto s = __builtin_amdgcn_permlane32_swap((unsigned)acc[i], (unsigned)acc[i + 8], false, false);
    h8[i] = (int)(s[0] + s[1]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto s = __builtin_amdgcn_permlane16_swap((unsigned)h8[i], (unsigned)h8[i + 4], false, false);
    h4[i] = (int)(s[0] + s[1]);
    h4[i] += __builtin_amdgcn_mov_dpp(h4[i], 0x128, 0xf, 0xf, true);                 // row_ror:8
    if (LPR == 4) h4[i] += __builtin_amdgcn_mov_dpp(h4[i], 0x124, 0xf, 0xf, true);   // row_ror:4
  }
  if ((lane & 15) < LPR) {
    const int c0 = cs * 16 + ((lane >> 4) & 1) * 4 + (lane >> 5) * 8;
    *reinterpret_cast<v4i*>(red + wave * D + c0) = v4i{h4[0], h4[1], h4[2], h4[3]};
  }
  lds_barrier();
  if (tid < dr) {
    int sum = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += red[w * D + tid];
    ctx[bh * dr + tid] = Epi<EPI_S8_SCALE>::apply(sum, 0.0f, alpha_pv);
  }
  // the new row goes into the cache last: no load of this launch reads it from there
  if (grow && rs == 0 && in_row) {
    if (wave == NW - 1) *reinterpret_cast<v4i*>(kb + (long long)S_old * dr + col) = fresh_k;
    if (wave == NW - 2) *reinterpret_cast<v4i*>(vb + (long long)S_old * dr + col) = fresh_v;
  }
}

// Bytes of dynamic LDS: fp32 scores [T][Sp], int8 probabilities [T][Sp], partial outputs [4][T][D].
__host__ __device__ inline long long decode_attn_lds(long long T, long long S, long long D) {
  const long long Sp = (S + 3) / 4 * 4;
  return T * Sp * 4 + T * Sp + 4 * T * D * 4;
}

// 256 threads.  For two to four new tokens, and for one where decode_attn_one_kernel does not apply.
// NI > 0: the whole cache of the (batch, head) is at most NI row groups per lane and all of its loads are
// issued up front (keys and values, 16 bytes each per lane), so the kernel waits for memory once.
// NI == 0: any length, four row groups in flight at a time.
// PART: the head size in memory is smaller than D, the bytes of a cache row that the lanes cover; the forms for
// head sizes 64 and 128 carry none of its tests.
// MOVE: as in decode_attn_one_kernel, a form of its own (tested at run time it cost the others up to 9 %: two tokens over 43 positions
// 8.6 -> 9.7 us).
template <int TQ, int D, int NI, bool PART, bool MOVE>
__global__ __launch_bounds__(256) void decode_attn_kernel(const int8_t* __restrict__ q, const int8_t* __restrict__ k_new,
                                                          const int8_t* __restrict__ v_new, int8_t* k_buf,
                                                          int8_t* v_buf, const float* __restrict__ mask,
                                                          int8_t* __restrict__ ctx, int8_t* __restrict__ probs_out,
                                                          int T, int S_arg, long long cap, int heads, float alpha_qk,
                                                          float alpha_pv, const int* __restrict__ s_dev, int dr_arg,
                                                          const int8_t* k_past, const int8_t* v_past, long long past_cap) {
  const int dr = PART ? dr_arg : D;
  // dr = the head size in memory, a multiple of 16 up to D (64 or 128, the lanes a cache row is spread over):
  // rows of q, the caches and ctx are dr bytes long; the lanes beyond a row hold zeros and store nothing
  // s_dev != nullptr: the number of positions is read from device memory (a launch recorded in a HIP graph is
  // replayed for a cache that has grown meanwhile; S_arg is then the largest length the launch was sized for)
  // (clamped to the contract T <= length <= S_arg: the host cannot check a value it never sees, and a length
  // outside that range would index past the LDS score rows and the cache buffers)
  int S = S_arg;
  if (s_dev != nullptr) {
    S = s_dev[0];
    S = S < T ? T : S;
    S = S > S_arg ? S_arg : S;
  }
  constexpr int LPR = D / 16;    // lanes per cache row
  constexpr int RPW = 64 / LPR;  // rows per wave per load
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int Sp = (S + 3) & ~3;
  float* scores = reinterpret_cast<float*>(smem);                              // [T][Sp]
  int8_t* probs = reinterpret_cast<int8_t*>(smem + (size_t)T * Sp * 4);        // [T][Sp]
  int* red = reinterpret_cast<int*>(smem + (size_t)T * Sp * 5);                // [4][T][D]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rs = lane / LPR, cs = lane % LPR;
  const bool in_row = !PART || cs * 16 < dr;
  const long long bh = blockIdx.x;
  const int S_old = k_new != nullptr ? S - T : S;  // rows below come from the cache, the rest from k_new / v_new
  int8_t* kb = k_buf + bh * cap * dr;
  int8_t* vb = v_buf + bh * cap * dr;
  const int8_t* ko = MOVE ? k_past + bh * past_cap * dr : kb;  // the rows before the new ones
  const int8_t* vo = MOVE ? v_past + bh * past_cap * dr : vb;
  const int8_t* kn = k_new != nullptr ? k_new + bh * T * dr : nullptr;
  const int8_t* vn = v_new != nullptr ? v_new + bh * T * dr : nullptr;

  // ---- phase 1: scores[t][s] = alpha_qk * (q[t] . k[s]); new key rows go into the cache on the way
  v4i qr[TQ];
#pragma unroll
  for (int t = 0; t < TQ; ++t)
    qr[t] = t < T && in_row ? *reinterpret_cast<const v4i*>(q + (bh * T + t) * dr + cs * 16) : v4i{0, 0, 0, 0};
  constexpr int U = NI > 0 ? NI : 4;  // row groups in flight per wave
  // Rows past the end re-read the last row (their products are never used), so the loads need no branches;
  // rows that come from k_new / v_new (or from another cache) are also written into the cache.
  auto load_rows = [&](int base, v4i (&dst)[U], int8_t* buf, const int8_t* old, const int8_t* fresh) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int s = base + u * 4 * RPW + rs;
      s = s < S ? s : S - 1;
      const int8_t* src = s < S_old ? old + (long long)s * dr : fresh + (long long)(s - S_old) * dr;
      dst[u] = in_row ? *reinterpret_cast<const v4i*>(src + cs * 16) : v4i{0, 0, 0, 0};
    }
    if (S_old < S) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = base + u * 4 * RPW + rs;
        if ((MOVE || s >= S_old) && s < S && in_row) *reinterpret_cast<v4i*>(buf + (long long)s * dr + cs * 16) = dst[u];
      }
    }
  };
  // the additive mask of the rows a lane will score, fetched together with the cache rows
  const float* msk = mask != nullptr ? mask + (bh / heads) * T * (long long)S : nullptr;
  const float lowest = -3.402823466e+38f;
  auto load_mask = [&](int base, float (&mk)[U][TQ]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = base + u * 4 * RPW + rs;
#pragma unroll
      for (int t = 0; t < TQ; ++t) mk[u][t] = (msk != nullptr && cs == 0 && s < S && t < T) ? msk[t * (long long)S + s] : 0.0f;
    }
  };
  // what the softmax reads: max(alpha_qk * acc + mask, most negative finite float)
  auto score_rows = [&](int base, v4i (&kv)[U], float (&mk)[U][TQ]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (base + u * 4 * RPW >= S) break;  // the same for every lane of the wave
      const int s = base + u * 4 * RPW + rs;
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        const int a = row_sum<LPR>(dot16(kv[u], qr[t], 0));
        if (cs == 0 && s < S && t < T) {
          float x = Epi<EPI_F32_SCALE>::apply(a, 0.0f, alpha_qk);
          if (msk != nullptr) x = x + mk[u][t];
          scores[t * Sp + s] = x > lowest ? x : lowest;
        }
      }
    }
  };
  v4i vv[U];
  if constexpr (NI > 0) {
    v4i kv[U];
    float mk[U][TQ];
    load_rows(wave * RPW, kv, kb, ko, kn);
    load_mask(wave * RPW, mk);
    load_rows(wave * RPW, vv, vb, vo, vn);
    score_rows(wave * RPW, kv, mk);
  } else {
    for (int base = wave * RPW; base < S; base += 4 * RPW * U) {
      v4i kv[U];
      float mk[U][TQ];
      load_rows(base, kv, kb, ko, kn);
      load_mask(base, mk);
      score_rows(base, kv, mk);
    }
  }
  __syncthreads();

  // ---- phase 2: int8 probabilities.  The maximum, the exponentials and the rounding use all threads;
  // the sum of a row is taken by one wave in the order of attn_softmax_q (chunk c of four elements belongs
  // to lane c % 64, a lane adds its elements in ascending order, lanes combine with a xor butterfly 32..1).
  float* wmax = reinterpret_cast<float*>(red);  // [4] per row, then [1] scale per row: red is free until phase 3
  for (int t = 0; t < T; ++t) {
    float* row = scores + t * Sp;
    float m = lowest;
    for (int i = tid; i < S; i += 256) m = m > row[i] ? m : row[i];
    m = wave_max(m);
    if (lane == 0) wmax[t * 8 + wave] = m;
  }
  __syncthreads();
  for (int t = 0; t < T; ++t) {
    float* row = scores + t * Sp;
    const float a = wmax[t * 8 + 0], b = wmax[t * 8 + 1], c = wmax[t * 8 + 2], e = wmax[t * 8 + 3];
    const float ab = a > b ? a : b, ce = c > e ? c : e;
    const float m = ab > ce ? ab : ce;
    for (int i = tid; i < S; i += 256) row[i] = exp_nonpos(row[i] - m);
  }
  __syncthreads();
  if (wave < T) {
    const float* row = scores + wave * Sp;
    const int nchunks = (S + 3) >> 2;
    float sum = 0.0f;
    for (int c = lane; c < nchunks; c += 64)
      for (int j = 0; j < 4; ++j)
        if (c * 4 + j < S) sum = sum + row[c * 4 + j];
    sum = wave_sum(sum);
    if (lane == 0) wmax[wave * 8 + 4] = 127.0f / sum;
  }
  __syncthreads();
  for (int t = 0; t < T; ++t) {
    const float* row = scores + t * Sp;
    const float scale = wmax[t * 8 + 4];
    int8_t* po = probs_out != nullptr ? probs_out + (bh * T + t) * (long long)S : nullptr;
    for (int i = tid; i < S; i += 256) {
      const int8_t pq = (int8_t)(int)__builtin_rintf(row[i] * scale);
      probs[t * Sp + i] = pq;
      if (po != nullptr) po[i] = pq;
    }
  }
  __syncthreads();

  // ---- phase 3: ctx[t][n] = s8(alpha_pv * sum_s p[t][s] * v[s][n]); the lane owns columns cs*16 .. +15
  int acc[TQ][16];
#pragma unroll
  for (int t = 0; t < TQ; ++t)
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[t][c] = 0;
  auto weigh_rows = [&](int base) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (base + u * 4 * RPW >= S) break;  // the same for every lane of the wave
      const int s = base + u * 4 * RPW + rs;
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        if (t >= T) continue;
        const int p = s < S ? (int)probs[t * Sp + s] : 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int x = vv[u][w];
          acc[t][4 * w + 0] += p * ((x << 24) >> 24);
          acc[t][4 * w + 1] += p * ((x << 16) >> 24);
          acc[t][4 * w + 2] += p * ((x << 8) >> 24);
          acc[t][4 * w + 3] += p * (x >> 24);
        }
      }
    }
  };
  if constexpr (NI > 0) {
    weigh_rows(wave * RPW);
  } else {
    for (int base = wave * RPW; base < S; base += 4 * RPW * U) {
      load_rows(base, vv, vb, vo, vn);
      weigh_rows(base);
    }
  }
  // the row slots of a wave meet through shuffles, the four waves through LDS
#pragma unroll
  for (int t = 0; t < TQ; ++t)
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      int a = acc[t][c];
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) a += __shfl_xor(a, off, 64);
      acc[t][c] = a;
    }
  if (rs == 0) {
#pragma unroll
    for (int t = 0; t < TQ; ++t)
      if (t < T) {
#pragma unroll
        for (int c = 0; c < 16; ++c) red[(wave * T + t) * D + cs * 16 + c] = acc[t][c];
      }
  }
  __syncthreads();
  for (int idx = tid; idx < T * D; idx += 256) {
    const int t = idx / D, c = idx - t * D;
    if (!PART || c < dr) {
      const int sum = red[idx] + red[T * D + idx] + red[2 * T * D + idx] + red[3 * T * D + idx];
      ctx[(bh * T + t) * dr + c] = Epi<EPI_S8_SCALE>::apply(sum, 0.0f, alpha_pv);
    }
  }
}

// D = the head size in memory: any multiple of 16 up to 128 (sizes up to 64 run on four lanes per cache row, the
// others on eight)
bool decode_attn_supported(long long T, long long S, long long D) {
  return T >= 1 && T <= DA_MAX_T && S >= 1 && D >= 16 && D <= 128 && D % 16 == 0 &&
         decode_attn_lds(T, S, D <= 64 ? 64 : 128) <= DA_LDS_LIMIT;
}

int launch_decode_attn_s8(const int8_t* q, const int8_t* k_new, const int8_t* v_new, int8_t* k_buf, int8_t* v_buf,
                          const float* mask, int8_t* ctx, int8_t* probs_out, long long BH, long long T, long long D,
                          long long cap, long long S, long long heads, float alpha_qk, float alpha_pv,
                          hipStream_t stream, const int* s_dev, const int8_t* k_past, const int8_t* v_past,
                          long long past_cap) {
  // with s_dev the kernel reads the length from device memory; S is the largest value it may find there (the LDS
  // and the kernel variant are sized for it)
  if (BH == 0) return TI_OK;
  if (!decode_attn_supported(T, S, D))
    return fail(TI_ERR_INVALID_ARG, "decode_attn: unsupported shape (T=%lld S=%lld head_dim=%lld)", T, S, D);
  if (BH > 0x7fffffffLL) return fail(TI_ERR_INVALID_ARG, "decode_attn: too many (batch, head) pairs (%lld)", BH);
  const dim3 grid((unsigned)BH), block(256);
  const int lanes_d = D <= 64 ? 64 : 128;  // the kernel variant: bytes of a cache row that its lanes cover
  const size_t lds = (size_t)decode_attn_lds(T, S, lanes_d);
  // One new token: the form with the fewest waves and groups that hold the cache (rows groups of 8 rows at head size 128, 16 at
  // 64), us, head size 128, cold: 250 positions, 768 heads: 4 waves x 8 groups 10.9, 8 x 8 11.3, 16 x 8 16.2; 500 positions,
  // 40 heads: 8 x 8 5.6, 16 x 8 5.8.  Between 96 and 128 groups sixteen waves are ahead while every workgroup has a CU to
  // itself (904 positions: 32 heads 7.3 against 8.0, 128 heads 10.2 / 10.4, 768 heads 38.0 / 32.1).  Beyond 128 groups only one
  // workgroup fits a CU, which leaves it without loads during the softmax: with more heads than two rounds of 256 the
  // streaming form, several small workgroups per CU, is level or ahead (1400 positions, 768 heads: 51.7 against 52.5; 128
  // heads 29.1 / 13.8).  So it is at head size 128 with more than one round of heads where the kernel reads the length and S is
  // only its bound: 320 heads, bound 2048, length 20 / 512 / 1024 / 2048 9.1 / 13.7 / 25.4 / 44.9 us, streaming 5.6 / 13.0 /
  // 25.0 / 44.4 (a length the host knows, 300 heads x 2040: 40.3, streaming 44.0; head size 80 keeps it, 18.0 against 25.9 at 1024).
  const long long groups = (S + 64 / (lanes_d / 16) - 1) / (64 / (lanes_d / 16));
#define TI_DA1_LAUNCH(DD, NW, NI, PART, MOVE)                                                                          \
  hipLaunchKernelGGL((decode_attn_one_kernel<DD, NW, NI, PART, MOVE>), grid, dim3(NW * 64), 0, stream, q, k_new, v_new, \
                     k_buf, v_buf, mask, ctx, probs_out, (int)S, cap, (int)heads, alpha_qk, alpha_pv, s_dev, (int)D,    \
                     k_past, v_past, past_cap)
#define TI_DA1(DD, NW, NI)                                          \
  do {                                                              \
    if (D == DD && k_past == nullptr) TI_DA1_LAUNCH(DD, NW, NI, false, false); \
    else if (D == DD) TI_DA1_LAUNCH(DD, NW, NI, false, true);       \
    else if (k_past == nullptr) TI_DA1_LAUNCH(DD, NW, NI, true, false); \
    else TI_DA1_LAUNCH(DD, NW, NI, true, true);                     \
  } while (0)
#define TI_DA1_FORMS(DD)                                            \
  do {                                                              \
    if (groups <= 8) TI_DA1(DD, 4, 2);                              \
    else if (groups <= 16) TI_DA1(DD, 4, 4);                        \
    else if (groups <= 32) TI_DA1(DD, 4, 8);                        \
    else if (groups <= 64) TI_DA1(DD, 8, 8);                        \
    else if (groups <= 96) TI_DA1(DD, 8, 12);                       \
    else if (groups <= 128 && BH > 256) TI_DA1(DD, 8, 16);          \
    else if (groups <= 128) TI_DA1(DD, 16, 8);                      \
    else if (groups <= 192) TI_DA1(DD, 16, 12);                     \
    else TI_DA1(DD, 16, 16);                                        \
  } while (0)
#define TI_DA_LAUNCH(TQ, DD, NI, PART, MOVE)                                                                            \
  hipLaunchKernelGGL((decode_attn_kernel<TQ, DD, NI, PART, MOVE>), grid, block, lds, stream, q, k_new, v_new, k_buf, v_buf, \
                     mask, ctx, probs_out, (int)T, (int)S, cap, (int)heads, alpha_qk, alpha_pv, s_dev, (int)D, k_past,  \
                     v_past, past_cap)
#define TI_DA(TQ, DD, NI)                                                \
  do {                                                                   \
    if (D == DD && k_past == nullptr) TI_DA_LAUNCH(TQ, DD, NI, false, false); \
    else if (D == DD) TI_DA_LAUNCH(TQ, DD, NI, false, true);             \
    else if (k_past == nullptr) TI_DA_LAUNCH(TQ, DD, NI, true, false);   \
    else TI_DA_LAUNCH(TQ, DD, NI, true, true);                           \
  } while (0)
  const bool one = T == 1 && (groups <= 128 || (groups <= 256 && BH <= (s_dev != nullptr && D > 96 ? 256 : 512)));
  // caches of at most 20 row groups per lane (640 positions at head size 128) with two query rows take
  // the variant that issues all loads up front
  const bool resident = T == 2 && S <= 20 * 4 * (64 / (lanes_d / 16));
  if (lanes_d == 128) {
    if (one) TI_DA1_FORMS(128);
    else if (T == 1) TI_DA(1, 128, 0);
    else if (T == 2) { if (resident) TI_DA(2, 128, 20); else TI_DA(2, 128, 0); }
    else TI_DA(4, 128, 0);
  } else {
    if (one) TI_DA1_FORMS(64);
    else if (T == 1) TI_DA(1, 64, 0);
    else if (T == 2) { if (resident) TI_DA(2, 64, 20); else TI_DA(2, 64, 0); }
    else TI_DA(4, 64, 0);
  }
#undef TI_DA1_FORMS
#undef TI_DA1
#undef TI_DA1_LAUNCH
#undef TI_DA_LAUNCH
#undef TI_DA
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "decode_attn launch: %s", hipGetErrorString(e));
  return TI_OK;
}

}  // namespace ti
