// Prefill attention with the scores of a whole row in registers: context = s8(alpha_pv round(127 softmax(max(alpha q.k^T +
// mask, lowest))) . V), up to 2048 keys (any multiple of 16) and head sizes up to 128 (any multiple of 16).  The bits are
// those of bmm_s8t_s8n_f32t -> attn_softmax_q -> bmm_s8t_s8n_s8t.
//
// One workgroup of four waves per (batch * head, 16 query rows).  The keys are cut so that a wave owns whole partial sums of
// the reference order (chunk c of four keys belongs to partial sum c % 64, which takes its chunks in ascending order): of
// every 256 keys, wave w has keys 64 w .. 64 w + 63 as four blocks of 16, and its partial sums are 16 w .. 16 w + 15.  Each
// score is computed once and stays in its accumulator register (128 of them at 2048 keys) until the row maximum and then
// the row sum are known; the waves meet twice in between, over a few KiB of LDS, and once more to add their integer
// contexts.  The three-sweep form this replaces up to 2048 keys computed scores three and exponentials up to two times, with a
// barrier and an exposed copy per tile of 256 keys and sweep.
//
// Bound by the vector ALUs (some 24 instructions a score: at 32 heads x 2048 x 128 without a mask 82 us of 126) and by waits that
// two waves to a SIMD, as many as the score registers allow, do not cover.  Causal, 32 heads x 1904 x 128, by the counters: the ALUs work in 53 % of
// the SIMDs' cycles (37 instructions a live score: dead halves of the diagonal's tiles, meetings), the matrix pipes in 10 %, the LDS in 14 %; waves
// wait for copies, LDS and one another during 37 % of their time and for an issue slot during 11 %.  What it measures against the other forms is at
// the rule that chooses (attn_fused.hip).
//
// Keys, mask values and V^T reach a wave through an LDS ring of its own, without barriers: no two waves of a workgroup use the same key, but
// a fragment load straight from global memory asks for 16 rows x 64 bytes with neighbouring lanes on different rows, a
// quarter of the rate of the copies' (32 heads x 2048 x 2048 without a mask: 264 us).  The pieces (32 keys, the mask values of 64,
// half of V^T's rows for 64 keys) follow one another in one sequence, V^T last, so that it lands under the last scores
// and the exponentials.  For P.V the four dwords of probabilities that a lane holds of 64 keys are transposed across the four
// 16-lane rows, after which a lane holds 16 consecutive keys, as a 16-byte read of V^T does.
// On V itself (VR), in pieces of 32 keys, a transposing LDS read (ds_read_b64_tr_b8) brings eight keys of a column to a lane, and any
// eight: those whose probabilities the lane has.  The kernel takes as long either way (0.98 to 1.05 times); the transpose that went
// before it is saved: 32 heads x 1904 x 128 101.6 -> 94.9 us, 160 x 528 x 128 53.5 -> 45.4, 12 x 128 x 64 7.0 -> 5.1 (2048 x 80 196 -> 198).
#include "ti_common.h"
#include "softmax_math.h"

namespace ti {

#define TI_GLOBAL_AS __attribute__((address_space(1)))
#define TI_LDS_AS __attribute__((address_space(3)))

constexpr int AR_TILE = 256;  // keys per round of the 64 partial sums
constexpr int AR_MAX_TILES = 8;
constexpr int AR_BUFFER_FLAGS = 0x00020000;  // raw buffer, 32-bit data: offsets from the descriptor's size on read as zeros
constexpr int AR_MC_ROWS = 64;  // rows to a mask class (attn_long.hip)
constexpr int AR_MC_ZERO = 1, AR_MC_UNIFORM = 2, AR_MC_LOW = 3;

typedef int v2i __attribute__((ext_vector_type(2)));

// 16-byte chunk c of row `row` of a piece whose rows hold B bytes sits at this chunk position
template <int B>
__device__ __forceinline__ int ar_swz(int row, int c) {
  return B == 128 ? (c ^ ((row >> 1) & 7)) : (c ^ ((row >> 2) & 3));
}

// chunk c of mask row `row` of a piece whose rows hold MC chunks (16 or 8)
template <int MC>
__device__ __forceinline__ int ar_mask_swz(int row, int c) {
  return MC == 16 ? c ^ row : c ^ (row >> 1);
}

template <int NT, int D>
struct AttnRows {
  static constexpr int PIECE = 32 * D;            // bytes: 32 keys, or D / 2 rows of 64 bytes of V^T, or MKEYS keys' mask
  static constexpr int COPIES = PIECE / 1024;     // copy instructions per piece
  static constexpr int MKEYS = PIECE / 64;        // 16 rows of mask values
  static constexpr int RING = 2;                  // pieces per wave (three or four: no faster, and fewer workgroups fit)
  static constexpr int WAVES = NT <= 4 ? 3 : 2;   // waves per SIMD the registers are sized for
  static constexpr int PART = 4 * RING * PIECE;   // [16][64] floats behind the rings, then [4][16]
  static constexpr int LDS = PART + 16 * 64 * 4 + 4 * 16 * 4;
  static_assert(RING * PIECE >= D / 16 * 1024, "a wave's context goes over its ring");
  static_assert(WAVES * LDS <= 160 * 1024, "resident workgroups");
};

// The ring of one wave.  A tile of `keys` puts two pieces of keys into it and, if it is one of `masked`, its mask values;
// after the last of them every tile of `vals` puts in two pieces of V^T.  The addresses are bounds-checked by the buffer
// descriptors: rows past the last key, the last query row or the head size read as zeros (and count for nothing).
// VR: V as the cache holds it, in rows of keys, whose pieces are then 32 keys as those of the keys are.
template <int NT, int D, bool VR>
struct AttnRing {
  using L = AttnRows<NT, D>;
  static constexpr int CP = L::COPIES, STAGES = 2 + 64 / L::MKEYS;
  char* ring;
  __amdgpu_buffer_rsrc_t kres, vres, mres;
  int S, dr, w;
  unsigned keys, masked, vals;
  unsigned key_off[2], v_off, m_row, m_chunk;  // a lane's offsets (keys: of even and odd copies)
  int stage = 0;                      // of the tile that comes next: 0, 1 keys or V^T, from 2 mask
  int head = 0, tail = 0, ahead = 0;  // next slot to fill, next to read, pieces between them

  __device__ __forceinline__ const char* at_tail() const { return ring + tail * L::PIECE; }
  __device__ __forceinline__ void issue() {
    if ((keys | vals) == 0) return;
    TI_LDS_AS char* dst = (TI_LDS_AS char*)ring + head * L::PIECE;
    const int tile = __builtin_ctz(keys != 0 ? keys : vals);
    const int at = tile * AR_TILE + 64 * w;
    ++stage;
    if (keys != 0) {
      if (stage <= 2) {
        const unsigned base = (unsigned)((at + 32 * (stage - 1)) * dr);
#pragma unroll
        for (int i = 0; i < CP; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(kres, (TI_LDS_AS void*)(dst + i * 1024), 16,
                                                   key_off[i & 1] + (base + (unsigned)(i * (1024 / D) * dr)), 0, 0, 0);
      } else {
        const unsigned base = (unsigned)(at + L::MKEYS * (stage - 3)) * 4u;
#pragma unroll
        for (int i = 0; i < CP; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              mres, (TI_LDS_AS void*)(dst + i * 1024), 16,
              (m_chunk ^ (unsigned)(64 * i)) + (m_row + base + (unsigned)(i * (16 / CP) * S * 4)), 0, 0, 0);
      }
      if (stage == (masked >> tile & 1 ? STAGES : 2)) {
        stage = 0;
        keys &= keys - 1;
      }
    } else {
      const unsigned base = VR ? (unsigned)((at + 32 * (stage - 1)) * dr) : (unsigned)((stage - 1) * (D / 2) * S + at);
#pragma unroll
      for (int i = 0; i < CP; ++i)
        if constexpr (VR)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(vres, (TI_LDS_AS void*)(dst + i * 1024), 16,
                                                   key_off[i & 1] + (base + (unsigned)(i * (1024 / D) * dr)), 0, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(vres, (TI_LDS_AS void*)(dst + i * 1024), 16, v_off + (base + (unsigned)(i * 16 * S)),
                                                   0, 0, 0);
      if (stage == 2) {
        stage = 0;
        vals &= vals - 1;
      }
    }
    head = head + 1 == L::RING ? 0 : head + 1;
    ++ahead;
  }
  // waits for the piece at the tail: loads complete in order, so at most the copies of the pieces behind it may be outstanding
  __device__ __forceinline__ void wait() const {
    static_assert(L::RING == 2, "at most one piece behind it");
    if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  // the piece has been read: its slot is free for the next
  __device__ __forceinline__ void release() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    tail = tail + 1 == L::RING ? 0 : tail + 1;
    --ahead;
    issue();
  }
};

// NT = tiles of 256 keys (only the last one may be cut short); D = 64 or 128, the head size in memory (dr) rounded up:
// the chunks of a query row beyond dr are zeros, so whatever the keys' copies put there adds nothing, and context columns
// beyond dr are computed and not stored.
template <int NT, int D, bool MASKED, bool VR>
__global__ __launch_bounds__(256, (AttnRows<NT, D>::WAVES)) void attn_rows_kernel(
    const int8_t* __restrict__ q, const int8_t* __restrict__ k, const float* __restrict__ mask,
    const unsigned char* __restrict__ cls, const int8_t* __restrict__ v, int8_t* __restrict__ ctx, int T, int S,
    long long stride_q, long long stride_k, int heads, int row_blocks, int n_bh, int abreast, float alpha, float alpha_pv, int dr) {
  using L = AttnRows<NT, D>;
  constexpr int KS = D / 64;  // 64-byte slices of the head dimension
  constexpr int CH = D / 16;  // blocks of 16 context columns
  constexpr int RING = L::RING, PIECE = L::PIECE;
  constexpr unsigned ALL = (1u << NT) - 1;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  char* ring = smem + w * RING * PIECE;
  float(*s_part)[64] = reinterpret_cast<float(*)[64]>(smem + L::PART);
  float(*s_max)[16] = reinterpret_cast<float(*)[16]>(smem + L::PART + 16 * 64 * 4);
  // `abreast` heads at a time (all but the last ones), and of those the heaviest rows of a causal mask first
  const int group = blockIdx.x / (abreast * row_blocks), in_group = blockIdx.x - group * (abreast * row_blocks);
  const int heads_here = n_bh - group * abreast < abreast ? n_bh - group * abreast : abreast;
  const long long bh = group * abreast + in_group % heads_here;
  const int t0 = (row_blocks - 1 - in_group / heads_here) * 16;
  const int rows = T - t0 < 16 ? T - t0 : 16;                       // rows past the end repeat the last one; never stored
  const float lowest = -3.402823466e+38f;

  v4i qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int c = 64 * s + 16 * g;
    qf[s] = *reinterpret_cast<const v4i*>(q + bh * stride_q + (long long)(t0 + (r < rows ? r : rows - 1)) * dr + (c < dr ? c : 0));
  }
  // Mask classes of this row block's tiles.  `todo`: the tiles whose keys are multiplied, all but those whose mask is low
  // throughout; `zero`: those whose mask adds nothing.  A score of a tile that is passed over is below `passed`: -1e30
  // takes no notice of any product (the launcher looks at alpha), and -6e4 or less, the mask of an fp16 model, is raised by at most the
  // largest product there can be (such tiles are multiplied like others where that is not far below it).
  unsigned todo = ALL, zero = MASKED ? 0u : ALL;
  float passed = -1e29f;
  if (MASKED && cls != nullptr) {
    const unsigned char* c = cls + ((bh / heads) * ((T + AR_MC_ROWS - 1) / AR_MC_ROWS) + t0 / AR_MC_ROWS) * NT;
    const int v = c[lane < NT ? lane : 0];
    zero = (unsigned)__builtin_amdgcn_ballot_w64(v == AR_MC_ZERO && lane < NT);
    const float product = __builtin_fabsf(alpha) * (float)(dr * 16384);
    const unsigned low = product < 3e4f ? (unsigned)__builtin_amdgcn_ballot_w64(v == AR_MC_LOW && lane < NT) : 0u;
    if (low != 0) passed = product - 5.9e4f;
    todo &= ~(low | (unsigned)__builtin_amdgcn_ballot_w64(v == AR_MC_UNIFORM && lane < NT));
  }
  AttnRing<NT, D, VR> pieces;
  pieces.ring = ring;
  pieces.S = S;
  pieces.dr = dr;
  pieces.w = w;
  pieces.kres = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(k + bh * stride_k), 0, S * dr, AR_BUFFER_FLAGS);
  pieces.vres = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(v + bh * (long long)dr * S), 0, S * dr, AR_BUFFER_FLAGS);
  pieces.mres = pieces.kres;
  if (MASKED)
    pieces.mres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(mask + ((bh / heads) * T + t0) * (long long)S), 0,
                                                    rows * S * 4, AR_BUFFER_FLAGS);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = lane / (D / 16), c = ar_swz<D>(i * (1024 / D) + row, lane % (D / 16)) * 16;
    pieces.key_off[i] = (unsigned)(row * dr + (c < dr ? c : 0));
  }
  pieces.v_off = (unsigned)((lane >> 2) * S + ar_swz<64>(lane >> 2, lane & 3) * 16);
  {
    constexpr int MC = L::MKEYS / 4;  // 16-byte chunks to a mask row
    const int row = lane / MC;
    pieces.m_row = (unsigned)(row * S * 4);
    pieces.m_chunk = (unsigned)(ar_mask_swz<MC>(row, lane % MC) * 16);
  }
  // a block past the last key (last tile only) is replaced by -infinity
  auto exists = [&](int t, int j) { return t < NT - 1 || t * AR_TILE + 64 * w + 16 * j < S; };

  v4i acc[NT][4];
  float m;
  for (;;) {  // once; a second time, without the classes, where a row needs the tiles that were passed over
    pieces.keys = pieces.vals = todo;
    pieces.masked = ~zero;
#pragma unroll
    for (int i = 0; i < RING; ++i) pieces.issue();
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[s][e] = 64 * s + 16 * g < dr ? qf[s][e] : 0;

    // ---- scores
    m = lowest;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (MASKED && !(todo >> t & 1)) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        pieces.wait();
        const char* src = pieces.at_tail();
        v4i kf[2][KS];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int s = 0; s < KS; ++s)
            kf[j][s] = *reinterpret_cast<const v4i*>(src + (16 * j + r) * D + (ar_swz<D>(16 * j + r, 4 * s + g) << 4));
        pieces.release();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          v4i a = {0, 0, 0, 0};
#pragma unroll
          for (int s = 0; s < KS; ++s) a = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf[j][s], qf[s], a, 0, 0, 0);
          acc[t][2 * h + j] = a;
        }
      }
      auto finish = [&](auto masked_, int j, v4f mk) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float x = Epi<EPI_F32_SCALE>::apply(acc[t][j][v], 0.0f, alpha);
          if constexpr (decltype(masked_)::value) x = x + mk[v];
          x = __builtin_fmaxf(x, lowest);  // NaN included
          if (t == NT - 1) x = exists(t, j) ? x : -__builtin_inff();
          m = __builtin_fmaxf(m, x);
          acc[t][j][v] = __float_as_int(x);
        }
      };
      if (MASKED && !(zero >> t & 1)) {
        constexpr int MC = L::MKEYS / 4, JP = L::MKEYS / 16;  // blocks per piece of mask
#pragma unroll
        for (int i = 0; i < 4 / JP; ++i) {
          pieces.wait();
          const char* src = pieces.at_tail();
          v4f mk[JP];
#pragma unroll
          for (int j = 0; j < JP; ++j)
            mk[j] = *reinterpret_cast<const v4f*>(src + r * (MC * 16) + ar_mask_swz<MC>(r, 4 * j + g) * 16);
          pieces.release();
#pragma unroll
          for (int j = 0; j < JP; ++j) finish(std::integral_constant<bool, true>{}, JP * i + j, mk[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) finish(std::integral_constant<bool, false>{}, j, v4f{0.f, 0.f, 0.f, 0.f});
      }
    }
    float o = __shfl_xor(m, 16, 64);
    m = m > o ? m : o;
    o = __shfl_xor(m, 32, 64);
    m = m > o ? m : o;
    if (g == 0) s_max[w][r] = m;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not for the copies of V^T)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o = s_max[i][r];
      m = m > o ? m : o;
    }
    // Beside a row maximum that is 100 above them, the scores of the tiles that were passed over add exact zeros.  A row
    // without such a maximum needs them.  (The same rows, and the same answer, in all four waves.)
    if (!MASKED || todo == ALL || __builtin_amdgcn_ballot_w64(!(m > passed + 100.0f)) == 0) break;
    todo = ALL;
    zero = 0;
    pieces.stage = pieces.head = pieces.tail = pieces.ahead = 0;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // s_max has been read, no copy is on its way
  }

  // ---- exponentials and partial sums; a block in which nothing is above exp's cut-off adds exact zeros
  unsigned live = 0;  // bit 4 t + j
  float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (MASKED && !(todo >> t & 1)) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float top = __builtin_fmaxf(__builtin_fmaxf(__int_as_float(acc[t][j][0]), __int_as_float(acc[t][j][1])),
                                        __builtin_fmaxf(__int_as_float(acc[t][j][2]), __int_as_float(acc[t][j][3])));
      if (__builtin_amdgcn_ballot_w64(top - m > -87.0f) != 0) {
        live |= 1u << (4 * t + j);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float e = exp_nonpos(__int_as_float(acc[t][j][v]) - m);
          acc[t][j][v] = __float_as_int(e);
          part[j] = part[j] + e;
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) s_part[4 * w + j][lane] = part[j];
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float all[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) all[j] = s_part[j][lane];
#pragma unroll
  for (int h = 8; h >= 1; h >>= 1)
#pragma unroll
    for (int j = 0; j < h; ++j) all[j] = all[j] + all[j + h];
  float sum = all[0];
  sum = sum + __shfl_xor(sum, 32, 64);
  sum = sum + __shfl_xor(sum, 16, 64);
  const float scale = 127.0f / sum;

  // ---- probabilities and their product with V
  v4i o[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) o[c] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (MASKED && !(todo >> t & 1)) continue;
    int pw[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned p = 0;
      if (live >> (4 * t + j) & 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v)  // in [0, 127], whole numbers
          p = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(__int_as_float(acc[t][j][v]) * scale), v, p);
      }
      pw[j] = (int)p;
    }
    if constexpr (VR) {
      // Two products of 32 keys: a lane's dwords of blocks 2 h and 2 h + 1 are the operand as they are, keys 16 j + 4 g .. +3, and the
      // transposing read of eight rows of V gives lane (r, g) the same keys of column r
      const int row = (r < 8 ? 0 : 12) + 4 * g + (r >> 1);  // the key whose 16 columns lanes 2 i and 2 i + 1 read
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        pieces.wait();
        const char* src = pieces.at_tail() + row * D + 8 * (r & 1);
        v2i vf[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c)
          vf[c] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TI_LDS_AS v2i*)(src + (ar_swz<D>(row, c) << 4)));
        pieces.release();
        const long pa = (long)((unsigned long)(unsigned)pw[2 * h] | (unsigned long)(unsigned)pw[2 * h + 1] << 32);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const long va = (long)((unsigned long)(unsigned)vf[c][0] | (unsigned long)(unsigned)vf[c][1] << 32);
          o[c] = __builtin_amdgcn_mfma_i32_16x16x32_i8(va, pa, o[c], 0, 0, 0);
        }
      }
      continue;
    }
    row_transpose4(pw);  // keys 16 j + 4 g .. +3 -> keys 16 g + 4 j .. +3
    const v4i pa = {pw[0], pw[1], pw[2], pw[3]};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      pieces.wait();
      const char* src = pieces.at_tail();
      v4i vf[CH / 2];
#pragma unroll
      for (int c = 0; c < CH / 2; ++c)
        vf[c] = *reinterpret_cast<const v4i*>(src + (16 * c + r) * 64 + (ar_swz<64>(16 * c + r, g) << 4));
      pieces.release();
#pragma unroll
      for (int c = 0; c < CH / 2; ++c)
        o[h * (CH / 2) + c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf[c], pa, o[h * (CH / 2) + c], 0, 0, 0);
    }
  }

  // ---- the four waves' contexts, over the rings (every copy of this wave has landed and been read)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int c = 0; c < CH; ++c) *reinterpret_cast<v4i*>(ring + (c * 64 + lane) * 16) = o[c];
  __syncthreads();
  if (r < rows) {
    const long long batch = bh / heads, h = bh - batch * heads;
    int8_t* crow = ctx + ((batch * T + t0 + r) * heads + h) * (long long)dr + 4 * g;
#pragma unroll
    for (int i = 0; i < CH / 4; ++i) {
      const int c = w * (CH / 4) + i;
      if (16 * c >= dr) continue;
      v4i a = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < 4; ++u) a += *reinterpret_cast<const v4i*>(smem + u * RING * PIECE + (c * 64 + lane) * 16);
      unsigned out = 0;
#pragma unroll
      for (int v = 0; v < 4; ++v) out |= (unsigned)(unsigned char)Epi<EPI_S8_SCALE>::apply(a[v], 0.0f, alpha_pv) << (8 * v);
      *reinterpret_cast<unsigned*>(crow + 16 * c) = out;
    }
  }
}

bool attn_rows_supported(long long T, long long S, long long D) {
  return T >= 1 && D >= 16 && D <= 128 && D % 16 == 0 && S >= 16 && S % 16 == 0 && S <= (long long)AR_TILE * AR_MAX_TILES;
}

template <int NT, int D, bool MASKED, bool VR, class... Args>
static void launch_ar(dim3 grid, hipStream_t stream, Args... args) {
  constexpr int lds = AttnRows<NT, D>::LDS;
  static_assert(lds <= 64 * 1024, "no larger than a launch may ask for as it is");
  hipLaunchKernelGGL((attn_rows_kernel<NT, D, MASKED, VR>), grid, dim3(256), lds, stream, args...);
}

int launch_attn_rows(const int8_t* q, const int8_t* k, const float* mask, const unsigned char* cls, const int8_t* v,
                     bool v_rows, int8_t* ctx, long long BH, long long T, long long S, long long D, long long stride_q,
                     long long stride_k, long long heads, float alpha, float alpha_pv, hipStream_t stream) {
  if (BH == 0 || T == 0) return TI_OK;
  if (mask == nullptr || !(alpha >= -1e12f && alpha <= 1e12f)) cls = nullptr;  // as in attn_long.hip
  if (!attn_rows_supported(T, S, D))
    return fail(TI_ERR_INVALID_ARG, "attn_rows: unsupported shape (T=%lld S=%lld head_dim=%lld)", T, S, D);
  const int nt = (int)((S + AR_TILE - 1) / AR_TILE);
  const long long row_blocks = (T + 15) / 16;
  if (BH * row_blocks > 0x7fffffffLL || T > 0x7fffffffLL)
    return fail(TI_ERR_INVALID_ARG, "attn_rows: too many row blocks (%lld)", BH * row_blocks);
  const dim3 grid((unsigned)(BH * row_blocks));
  // The workgroups of a head read all of its keys and values, 16 rows at a time, so those have to stay in the L2 of the XCD that
  // the head's workgroups are dealt to (one of eight, where a multiple of eight heads is abreast): 2 MiB of them to an XCD.  Us
  // with all heads abreast / so: 256 heads x 512 x 128 without a mask 133 / 73, 256 heads x 1024 x 128 523 / 230, causal 272 / 169,
  // 320 heads x 2048 x 128 2763 / 1237, causal 1565 / 979 (3 MiB to an XCD: 512 keys 87; 4 MiB: 134).
  const long long fit = 16ll * 1024 * 1024 / (2 * S * D) / 8 * 8;
  const long long abreast = fit < 8 ? 8 : fit < BH ? fit : BH;
#define TI_AR(NT, DD, MASKED, VR)                                                                                    \
  launch_ar<NT, DD, MASKED, VR>(grid, stream, q, k, mask, cls, v, ctx, (int)T, (int)S, stride_q, stride_k, (int)heads, \
                                (int)row_blocks, (int)BH, (int)abreast, alpha, alpha_pv, (int)D)
#define TI_AR_V(NT, DD, MASKED)                \
  if (v_rows) TI_AR(NT, DD, MASKED, true);     \
  else TI_AR(NT, DD, MASKED, false)
#define TI_AR_NT(NT)                           \
  case NT:                                     \
    if (D > 64) {                              \
      if (mask != nullptr) {                   \
        TI_AR_V(NT, 128, true);                \
      } else {                                 \
        TI_AR_V(NT, 128, false);               \
      }                                        \
    } else if (mask != nullptr) {              \
      TI_AR_V(NT, 64, true);                   \
    } else {                                   \
      TI_AR_V(NT, 64, false);                  \
    }                                          \
    break
  switch (nt) {
    TI_AR_NT(1);
    TI_AR_NT(2);
    TI_AR_NT(3);
    TI_AR_NT(4);
    TI_AR_NT(5);
    TI_AR_NT(6);
    TI_AR_NT(7);
    TI_AR_NT(8);
  }
#undef TI_AR_NT
#undef TI_AR_V
#undef TI_AR
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "attn_rows launch: %s", hipGetErrorString(e));
  return TI_OK;
}

}  // namespace ti
