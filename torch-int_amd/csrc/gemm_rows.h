// GEMM for a few rows of activations (2 to 64, of narrow outputs to 512): decode steps of a served batch, short prompts.  Included by
// gemm_s8_impl.h (it uses the epilogues of ti_common.h and the LDS-limit helper there).
//
// Bound by HBM: every weight byte is read from there once, for up to 64 rows of activations by one workgroup, for more by workgroups of one XCD.  What the weights cost on this
// chip is decided by two things, and the kernel is laid out for both of them:
//   - bytes in flight.  A CU has to keep some 64 KiB of weight copies outstanding to cover the round trip to HBM.  The
//     activations therefore do not share the LDS with the weights: a wave keeps the fragments of its slice of the
//     inner dimension in REGISTERS for the whole launch (16 rows x 64 bytes are 4 registers), and the whole LDS is a ring
//     of weight pieces.
//   - the shape of a copy.  A fragment load straight from global memory touches 16 rows x 64 bytes, half a cache line
//     each, and reaches a third of the rate of copies of whole lines (16384 x 4096 weights, 32 rows: 30 us against 13.4
//     with the LDS-DMA copies used here: a piece is 16 weight rows x KP * 64 bytes).
//
// Work: a workgroup of NW waves multiplies strips of 16 weight rows with one slice of the inner dimension, NW * KS * 64
// bytes long; wave w owns KS * 64 of them.  Each wave has a ring of its own, so the copy pipeline has no barriers: a
// wave waits for its own pieces with s_waitcnt.  The waves' 16 x (16 MX) partial tiles meet in the LDS (integer atomic
// adds into one of two buffers, one barrier a strip); wave (strip * MX + m) mod NW finishes row block m.  Narrow outputs
// spread their row blocks over workgroups, too (grid.y, rows_blocks_each).
//
// S slices of the inner dimension (S > 1) are spread over workgroups of one XCD, which meet as the waves of the one-launch
// split-K do (gemm_pipe16q_kernel, FUSED): partial tiles are parked in the XCD's L2, counted with an atomic that executes
// there, and the wave that arrives last adds them up.  p.arrivals == nullptr selects the two-launch form: raw partial
// products [S][M][N] for splitk_reduce_kernel.  Integer sums: the bits do not depend on any of this.
//
// LDS operations next to copies in flight are inline assembly on purpose: the compiler cannot see that an LDS access does
// not alias the copies' destination and puts a wait for ALL of them in front of it, which empties the pipeline once a strip.
//
// Measured, cold weights, us (before: the split-K, streaming and skinny kernels): 32 rows x 16384 x 4096 28.3 -> 14.6,
// 32 x 4096 x 16384 30.0 -> 17.9, 32 x 5120 x 5120 15.0 -> 10.5, 16 x 5120 x 20480 31.8 -> 20.7, 16 x 20480 x 5120 24.1 -> 19.3
// (5.4 TB/s), 8 x 20480 x 5120 22.0 -> 18.8, 48 x 768 x 768 6.0 -> 3.7; three 24 x 4096 x 4096 in one launch 84.7 -> 12.0.
#pragma once

namespace ti {

#define TI_ROWS_MAX_M 64       // of any width
#define TI_ROWS_ABREAST_M 512  // where the output is narrow (rows_blocks_each)


template <int KIND_, int MX_, int KS_, int KP_, int RING_, int NW_, bool GROUPED_ = false>
struct RowsCfg {
  static constexpr int KIND = KIND_, MX = MX_, KS = KS_, KP = KP_, RING = RING_, NW = NW_;
  static constexpr bool GROUPED = GROUPED_;
  static constexpr int NT = NW * 64;
  static constexpr int SLICE = NW * KS * 64;     // bytes of the inner dimension a workgroup covers
  static constexpr int PIECES = KS / KP;         // pieces of a strip, per wave
  static constexpr int PIECE = KP * 1024;        // 16 rows x KP * 64 bytes
  static constexpr int CW = KP * 4;              // 16-byte chunks per row of a piece
  // Chunk c of row r of a piece lies at position (c + (r >> SHIFT)) mod CW of the row, so that the 16 rows of a fragment
  // read, one chunk each, fall into 16 different 16-byte bank groups: rows are CW chunks apart, which is 4, 8, 12 or 0
  // modulo 16 as KP is 1, 2, 3 or 0 modulo 4.
  static constexpr int SHIFT = KP % 2 ? 2 : KP % 4 ? 1 : 0;
  static constexpr int RED_BYTES = 2 * MX * 1024;
  static constexpr int LDS_BYTES = NW * RING * PIECE + RED_BYTES;  // plus 64 bytes of bias per strip of a workgroup
  static constexpr int PER_CU = LDS_BYTES <= 76 * 1024 ? 2 : 1;
  static_assert(KS % KP == 0 && (RING - 1) * KP <= 63 && RING >= 2 && RING <= 8, "ring");
  static_assert((NW & (NW - 1)) == 0, "a power of two waves");
};

// `acc` = the products of row m with columns nb .. nb + 3; bt = their bias terms.  The vector stores need N % 4 == 0.
template <int KIND>
__device__ __forceinline__ void store_rows4(v4i acc, const GemmParams& p, int m, int nb, v4f bt) {
  using E = Epi<KIND>;
  using Out = typename E::Out;
  const int N = p.N;
  Out* C = reinterpret_cast<Out*>(p.C);
  Out* dst = C + out_index(p, m, nb < N ? nb : 0);
  Out o[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) o[v] = E::apply(acc[v], bt[v], p.alpha);
  const bool whole = (N & 3) == 0 && nb + 4 <= N && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  if (whole) {
    if constexpr (sizeof(Out) == 4) {
      typedef Out Out4 __attribute__((ext_vector_type(4)));
      Out4 w4 = {o[0], o[1], o[2], o[3]};
      if constexpr (E::kAccumulate) w4 = *reinterpret_cast<const Out4*>(dst) + w4;
      *reinterpret_cast<Out4*>(dst) = w4;
    } else if constexpr (sizeof(Out) == 2) {
      typedef Out Out4 __attribute__((ext_vector_type(4)));
      Out4 w4 = *reinterpret_cast<const Out4*>(dst);
#pragma unroll
      for (int v = 0; v < 4; ++v) w4[v] = accumulated<Out>(w4[v], o[v]);
      *reinterpret_cast<Out4*>(dst) = w4;
    } else {
      *reinterpret_cast<unsigned*>(dst) = (unsigned)(unsigned char)o[0] | ((unsigned)(unsigned char)o[1] << 8) |
                                          ((unsigned)(unsigned char)o[2] << 16) | ((unsigned)(unsigned char)o[3] << 24);
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (nb + v < N) dst[v] = merge_old<E>(o[v], dst + v);
  }
}

template <class Cfg>
__global__ __launch_bounds__(Cfg::NT, Cfg::NW == 16 ? 4 : 2) void gemm_rows_kernel(GemmParams p, GemmGroup grp, int strips,
                                                               int strips_per_problem) {
  constexpr int MX = Cfg::MX, KS = Cfg::KS, KP = Cfg::KP, RING = Cfg::RING, NW = Cfg::NW, PIECES = Cfg::PIECES,
                PIECE = Cfg::PIECE, CW = Cfg::CW, SHIFT = Cfg::SHIFT;
  using E = Epi<Cfg::KIND>;
  using BiasT = typename E::Bias;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int M = p.M, N = p.N, K = p.K, S = p.splits;
  const int row0 = blockIdx.y * (16 * MX);  // rows_blocks_each; 0 where S > 1

  // Workgroup -> (XCD, slice, group of strips).  Workgroup ids congruent modulo 8 share an XCD (checked below); all slices
  // of a strip go to one XCD.  Strip number o of the launch order is taken by XCD o mod 8.
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, n_groups = (int)(gridDim.x >> 3) / S;
  const int slice = local % S, group = local / S;
  if (group >= n_groups) return;
  const int first = group * 8 + xcd, step = n_groups * 8;
  const int my_strips = first < strips ? (strips - first + step - 1) / step : 0;
  if (my_strips == 0) return;  // the same for every wave, before the first barrier
  // Runs of 8 consecutive strips on one XCD, so that its L2 merges the 16-byte pieces of a line of 8-bit outputs.
  auto strip_of = [&](int i) {
    const int o = first + i * step;
    return o < (strips & ~63) ? (o & ~63) + ((o & 7) << 3) + ((o >> 3) & 7) : o;
  };
  // Placement check of the fused form: the S workgroups of a group add (1, XCC id) to the group's word and compare with
  // what was there; the last one clears it.  Device scope, so the words are 64 bytes apart: such atomics on one cache line
  // go one by one (512 workgroups on eight words of a line: 10 us).  The answer is looked at when the workgroup is done.
  unsigned xcc = 0, xcc_before = 0;
  unsigned* const xcc_word = p.xcc_seen + (group * 8 + xcd) * 16;
  const bool fused = S > 1 && p.arrivals != nullptr;
  if (fused && tid == 0) {
    xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 0xf;  // HW_REG_XCC_ID, bits 3:0
    xcc_before = __hip_atomic_fetch_add(xcc_word, (1u << 16) | xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  char* ring = smem + wave * (RING * PIECE);
  int* red = reinterpret_cast<int*>(smem + NW * RING * PIECE);  // [2][MX][4][64]
  int* bias_raw = red + 2 * MX * 256;  // [my_strips rounded up to 4][16], one element a dword
  for (int i = tid; i < 2 * MX * 256; i += Cfg::NT) red[i] = 0;
  // The bias of this workgroup's columns: copies straight into the LDS, first in line, so that no strip waits for a load
  // of its own at its end.  A lane's element lands in the lane's dword, a byte zero-extended.
  if constexpr (E::kHasBias) {
    for (int q = wave; q * 4 < my_strips; q += NW) {
      const int i = q * 4 + (lane >> 4) < my_strips ? q * 4 + (lane >> 4) : my_strips - 1;
      int strip = strip_of(i), prob = 0;
      if constexpr (Cfg::GROUPED) {
        prob = strip / strips_per_problem;
        strip -= prob * strips_per_problem;
      }
      int n = strip * 16 + r;
      n = n < N ? n : N - 1;
      const BiasT* bias = reinterpret_cast<const BiasT*>(p.bias);
      if constexpr (Cfg::GROUPED) bias = reinterpret_cast<const BiasT*>(grp.bias[prob]);
      const TI_GLOBAL_AS void* src = (const TI_GLOBAL_AS void*)(bias + n);
      if constexpr (sizeof(BiasT) == 1) __builtin_amdgcn_global_load_lds(src, (TI_LDS_AS void*)(bias_raw + q * 64), 1, 0, 0);
      else __builtin_amdgcn_global_load_lds(src, (TI_LDS_AS void*)(bias_raw + q * 64), 4, 0, 0);
    }
  }

  // ---- addresses: lane l of copy i of a piece fetches the chunk that belongs at position i * 64 + l of the piece
  const size_t k_first = (size_t)slice * Cfg::SLICE + (size_t)wave * (KS * 64);
  int row_of[KP], col_of[KP];
  unsigned off[KP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    const int c = i * 64 + lane;
    row_of[i] = c / CW;
    int col = (c % CW - (row_of[i] >> SHIFT)) % CW;
    col_of[i] = (col < 0 ? col + CW : col) * 16;
    off[i] = (unsigned)(row_of[i] * K + col_of[i]);
  }
  int frag[KP];  // byte offset of this lane's fragment of k step j inside a piece
#pragma unroll
  for (int j = 0; j < KP; ++j) frag[j] = (r * CW + (4 * j + g + (r >> SHIFT)) % CW) * 16;

  const int total = my_strips * PIECES;  // weight pieces of this wave
  int issued = 0, w_piece = 0, w_i = 0, w_slot = 0;
  auto issue_weights = [&]() {
    if (issued >= total) return;
    char* dst = ring + w_slot * PIECE;
    int strip = strip_of(w_i);
    const int8_t* B = p.B;
    if constexpr (Cfg::GROUPED) {
      const int prob = strip / strips_per_problem;
      strip -= prob * strips_per_problem;
      B = grp.B[prob];
    }
    const char* base = reinterpret_cast<const char*>(B) + (size_t)strip * 16 * K + k_first + w_piece * (KP * 64);
    const bool ragged = strip * 16 + 16 > N;  // rows past the end repeat the last row; their columns are not stored
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      unsigned o = off[i];
      if (ragged) {
        const int last = N - 1 - strip * 16;
        o = (unsigned)((row_of[i] < last ? row_of[i] : last) * K + col_of[i]);
      }
      // non-temporal: a decode step streams more weights than the last-level cache holds, each byte once
      __builtin_amdgcn_global_load_lds((const TI_GLOBAL_AS void*)(base + o), (TI_LDS_AS void*)(dst + i * 1024), 16, 0, 2);
    }
    ++issued;
    if (++w_piece == PIECES) {
      w_piece = 0;
      ++w_i;
    }
    w_slot = w_slot + 1 == RING ? 0 : w_slot + 1;
  };
  auto issue_rows = [&](int m, int piece) {
    char* dst = ring + w_slot * PIECE;
    const char* base = reinterpret_cast<const char*>(p.A) + k_first + piece * (KP * 64);
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int row = row0 + m * 16 + row_of[i];  // rows past M repeat the last one
      const unsigned o = (unsigned)((row < M ? row : M - 1) * K + col_of[i]);
      __builtin_amdgcn_global_load_lds((const TI_GLOBAL_AS void*)(base + o), (TI_LDS_AS void*)(dst + i * 1024), 16, 0, 0);
    }
    w_slot = w_slot + 1 == RING ? 0 : w_slot + 1;
  };
  // waits until at most `newer` of this wave's pieces are outstanding (copies complete in order)
  auto wait_newer = [&](int newer) {
#define TI_ROWS_WAIT(n)                                                              \
  case n:                                                                            \
    if constexpr (RING > n + 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n * KP) : "memory"); \
    break;
    if (newer >= RING - 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 1) * KP) : "memory");
      return;
    }
    switch (newer) {
      TI_ROWS_WAIT(6)
      TI_ROWS_WAIT(5)
      TI_ROWS_WAIT(4)
      TI_ROWS_WAIT(3)
      TI_ROWS_WAIT(2)
      TI_ROWS_WAIT(1)
      default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#undef TI_ROWS_WAIT
  };

  // ---- the activations pass through the ring once, into registers
  v4i x[MX][KS];
  int slot = 0;
#pragma unroll
  for (int i = 0; i < RING - 1; ++i) {
    if (i < MX * PIECES) issue_rows(i / PIECES, i % PIECES);
    else issue_weights();
  }
#pragma unroll
  for (int i = 0; i < MX * PIECES; ++i) {
    if (i + RING - 1 < MX * PIECES) issue_rows((i + RING - 1) / PIECES, (i + RING - 1) % PIECES);
    else issue_weights();
    wait_newer(MX * PIECES - 1 - i + total);
    const char* at = ring + slot * PIECE;
#pragma unroll
    for (int j = 0; j < KP; ++j) x[i / PIECES][(i % PIECES) * KP + j] = *reinterpret_cast<const v4i*>(at + frag[j]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    slot = slot + 1 == RING ? 0 : slot + 1;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // red is cleared, the bias has landed

  const unsigned red_at = (unsigned)(uintptr_t)(TI_LDS_AS int*)red + lane * 4;
  const unsigned bias_at = (unsigned)(uintptr_t)(TI_LDS_AS int*)bias_raw + g * 16;
  // the epilogue of one 16 x 16 tile: lane (r, g) holds row `row`, columns 4 g .. 4 g + 3 of the strip
  auto finish = [&](v4i sum, int si, int strip, int row) {
    int prob = 0, n0 = strip * 16;
    if constexpr (Cfg::GROUPED) {
      prob = strip / strips_per_problem;
      n0 = (strip - prob * strips_per_problem) * 16;
    }
    v4f bt = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (E::kHasBias) {
      v4i raw;
      asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(raw) : "v"(bias_at + si * 64) : "memory");
      const float beta = Cfg::GROUPED ? grp.beta[prob] : p.beta;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int element = raw[v];
        if constexpr (sizeof(BiasT) == 1) bt[v] = E::bias_term((BiasT)element, beta);
        else bt[v] = E::bias_term(__builtin_bit_cast(BiasT, element), beta);
      }
    }
    if (row >= M) return;
    if constexpr (Cfg::GROUPED) {
      GemmParams q = p;
      q.C = grp.C[prob];
      q.alpha = grp.alpha[prob];
      store_rows4<Cfg::KIND>(sum, q, row, n0 + 4 * g, bt);
    } else {
      store_rows4<Cfg::KIND>(sum, p, row, n0 + 4 * g, bt);
    }
  };
  int done = 0;
  for (int si = 0; si < my_strips; ++si) {
    v4i acc[MX];
#pragma unroll
    for (int m = 0; m < MX; ++m) acc[m] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int piece = 0; piece < PIECES; ++piece) {
      issue_weights();  // into the slot the piece before last has left
      wait_newer(total - 1 - done);
      ++done;
      const char* at = ring + slot * PIECE;
      v4i w[KP];
#pragma unroll
      for (int j = 0; j < KP; ++j) w[j] = *reinterpret_cast<const v4i*>(at + frag[j]);
#pragma unroll
      for (int j = 0; j < KP; ++j)
#pragma unroll
        for (int m = 0; m < MX; ++m)
          acc[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[j], x[m][piece * KP + j], acc[m], 0, 0, 0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
      slot = slot + 1 == RING ? 0 : slot + 1;
    }
    // ---- the waves' partial tiles add up in one of two buffers.  The compiler does not know what the assembly reads, so
    // the wait states between the last matrix instruction and the first read of its result are spelled out.
    const unsigned buf = red_at + (si & 1) * (MX * 1024);
#pragma unroll
    for (int m = 1; m < MX; ++m) asm volatile("" : "+v"(acc[m]));
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(acc[0]));
#pragma unroll
    for (int m = 0; m < MX; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        asm volatile("ds_add_u32 %0, %1 offset:%2" ::"v"(buf), "v"(acc[m][v]), "n"((m * 4 + v) * 256) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // The wave that finishes a row block takes it out of the buffer and leaves zeros; the buffer is used again two strips
    // later, beyond the next strip's barrier.
    const int strip = strip_of(si);
#pragma unroll
    for (int m = 0; m < MX; ++m) {
      if (wave != ((si * MX + m) & (NW - 1))) continue;
      v4i sum;
      {
        int s0, s1, s2, s3;
        asm volatile(
            "ds_wrxchg_rtn_b32 %0, %4, %5 offset:%6\n\tds_wrxchg_rtn_b32 %1, %4, %5 offset:%7\n\t"
            "ds_wrxchg_rtn_b32 %2, %4, %5 offset:%8\n\tds_wrxchg_rtn_b32 %3, %4, %5 offset:%9\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3)
            : "v"(buf), "v"(0), "n"((m * 4) * 256), "n"((m * 4 + 1) * 256), "n"((m * 4 + 2) * 256),
              "n"((m * 4 + 3) * 256)
            : "memory");
        sum = v4i{s0, s1, s2, s3};
      }
      const int row = row0 + m * 16 + r;
      if (S == 1) {
        finish(sum, si, strip, row);
      } else if (row < M) {
        // raw: [problem][S][M][N]; parked: [strip][row block][slice][row of the block][16] (N is a multiple of 16 here)
        int* at;
        if (fused) {
          const int rows_here = M - m * 16 < 16 ? M - m * 16 : 16;
          at = reinterpret_cast<int*>(p.parts) + (((size_t)strip * M + m * 16) * S + (size_t)slice * rows_here) * 16 + r * 16;
        } else {
          const int prob = Cfg::GROUPED ? strip / strips_per_problem : 0;
          at = reinterpret_cast<int*>(p.parts) + ((size_t)(prob * S + slice) * M + row) * N +
               (strip - prob * strips_per_problem) * 16;
        }
        *reinterpret_cast<v4i*>(at + 4 * g) = sum;
      }
    }
  }
  if (!fused) return;
  // ---- all slices of this group's strips meet once, when a workgroup is done (meeting strip by strip empties the finishing
  // wave's copy pipeline every time: 32 x 5120 x 5120 in five slices 23 us instead of 9).  Wave w of every slice parked the
  // same tiles; the one that arrives last adds them up.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the parked tiles are acknowledged by the L2
  int* counter = p.arrivals + (group * 8 + xcd) * NW + wave;
  int earlier = 0;
  if (lane == 0) earlier = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  earlier = __builtin_amdgcn_readfirstlane(earlier);
  if (earlier == S - 1) {  // uniform over the wave
    if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    for (int t = wave; t < my_strips * MX; t += NW) {
      const int si = t / MX, m = t - si * MX, row = m * 16 + r;
      const int strip = strip_of(si);
      const int rows_here = M - m * 16 < 16 ? M - m * 16 : 16;
      const int* tile = reinterpret_cast<const int*>(p.parts) + ((size_t)strip * M + m * 16) * S * 16 +
                        (r < rows_here ? r : 0) * 16 + 4 * g;
      v4i sum = {0, 0, 0, 0};
      for (int t0 = 0; t0 < S; t0 += 4) {
        // sc1: past this CU's own cache, which may hold a line shared with a tile that was not complete yet
        const int* src[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) src[u] = tile + (size_t)(t0 + u < S ? t0 + u : t0) * rows_here * 16;
        v4i q0, q1, q2, q3;
        asm volatile(
            "global_load_dwordx4 %0, %4, off sc1\n\tglobal_load_dwordx4 %1, %5, off sc1\n\t"
            "global_load_dwordx4 %2, %6, off sc1\n\tglobal_load_dwordx4 %3, %7, off sc1\n\ts_waitcnt vmcnt(0)"
            : "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(q3)
            : "v"(src[0]), "v"(src[1]), "v"(src[2]), "v"(src[3])
            : "memory");
        sum += q0;
        if (t0 + 1 < S) sum += q1;
        if (t0 + 2 < S) sum += q2;
        if (t0 + 3 < S) sum += q3;
      }
      finish(sum, si, strip, row);
    }
  }
  if (tid == 0) {
    const unsigned seen = xcc_before >> 16;
    if ((xcc_before & 0xffffu) != seen * xcc)  // a workgroup of this group ran on another XCC
      __hip_atomic_store(p.xcc_error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if ((int)seen + 1 == S) __hip_atomic_store(xcc_word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ------------------------------------------------------------------ host side

// Which tiling of the inner dimension a problem of M rows takes; 0 = none (the kernel does not take the shape).
//   A  4 waves x 512 bytes, two workgroups per CU: K % 2048 == 0
//   B  4 waves x 256 bytes, two workgroups per CU: K % 1024 == 0
//   C  8 waves x 640 bytes, one workgroup per CU: K % 5120 == 0
//   D  4 waves x 640 bytes, two per CU: K % 2560 == 0
//   E  4 waves x 192 bytes, two per CU: K % 768 == 0
//   F  16 waves x 256 bytes, one per CU: K == 4096, and pairs of A's slices (rows_paired)
//   G  8 waves x 384 bytes, one per CU: K % 3072 == 0
//   H  8 waves x 448 bytes, one per CU: K % 3584 == 0
// A divisor of K that is a whole slice comes first (C, F, H, then A, G, D, B, E): slices that meet cost 2 to 2.5 us a launch (park,
// count, add), which only a long K repays.  Several slices take the first tiling in that order; the pairs that are measured
// below compare one slice with several.  A K whose first divisor makes too many slices goes to the other kernels, also where
// another tiling would fit (36864: 18 of A, 12 of G; 49152: 24 of A, 16 of G).
// us, cold weights, 16 / 32 / 64 rows: 5120 x 5120 C 8.9 / 10.5 / 13.3, B in five slices 9.5 / 11.7 / 15.4;
// 4096 x 4096 F 6.3 / 7.8 / 9.7, A in two 7.2 / 8.7 / 10.5; 16384 x 4096 F 13.1 / 14.6 / 17.6, A in two 14.4 / 16.7 / 21.3 (F with 64
// rows: 8 waves of 512 bytes, 16 waves have too few registers for the fragments and spill, 21.8); 768 x 3072 G
// 4.6 / 5.5 / 6.8, E in four 5.1 / 5.6 / 6.5; 2048 x 2048 A 3.6 / 4.0 / 5.2, B in two 5.1 / 5.5 / 6.6.  Pieces of whole 128-byte lines where
// the tiling allows it: 36864 x 9216, 32 rows, G with pieces of 192 bytes a row 72.5, of 128 bytes 66.3.
enum RowsTiling { ROWS_NONE = 0, ROWS_A, ROWS_B, ROWS_C, ROWS_D, ROWS_E, ROWS_F, ROWS_G, ROWS_H };
struct RowsPick {
  int tiling;
  int slices;
};
// Whether several slices, `pick`, beat the kernel that would run instead.  What they cost is the end: the wave that arrives
// last adds up its tiles one after the other, four slices a round trip (64 x 20480 x 13312 in thirteen slices: 51 us of
// weights, 100 us of that).
static inline bool rows_slices_ahead(RowsPick pick, long long M, long long N, long long K, int problems, int cus) {
  // waves, workgroups per CU; us per MB of weights and per round of the end, fitted to 875 shapes within 8 %
  static constexpr struct {
    int waves, per_cu;
    double us_per_mb, us_per_round;
  } cost[] = {{0, 0, 0.0, 0.0},      {4, 2, 0.148, 0.70}, {4, 2, 0.124, 0.65}, {8, 1, 0.118, 2.20}, {4, 2, 0.125, 1.95},
              {4, 2, 0.172, 1.10},   {8, 1, 0.118, 2.00}, {8, 1, 0.123, 1.95}, {8, 1, 0.118, 2.15}};
  const auto& c = cost[pick.tiling];
  const long long strips = (N + 15) / 16 * problems, row_blocks = (M + 15) / 16;
  const long long slots = (long long)cus * c.per_cu / 8, need = (strips + 7) / 8 * pick.slices;
  const long long groups = (need < slots ? need : slots) / pick.slices * 8;
  const long long strips_each = (strips + groups - 1) / groups;
  const long long rounds = (strips_each * row_blocks + c.waves - 1) / c.waves * ((pick.slices + 3) / 4);
  const double weights_us = c.us_per_mb * N * K * problems * 1e-6, end_us = c.us_per_round * rounds;
  if (end_us <= 2.0 + 0.2 * weights_us) return true;  // an end this short: none of 475 such shapes was slower
  int tile = SPLIT_128;
  double others = -1.0;
  (void)choose_splits(M, N, K, &tile, &others);
  if (others <= 0.0) return true;  // no price to compare with
  // at these few rows that model, made for more of them, is too low for 256x256 tiles and for short runs of 128x80 ones
  if (tile == SPLIT_256) others *= 1.25;
  else if (tile == SPLIT_128x80 && others < 14.0) others *= 1.15;
  // Both prices are good to some 10 %.  Of those 875 shapes (17 to 64 rows) 96 were slower than before in slices, up to 2.6 times
  // (64 x 20480 x 13312 58.2 -> 151.4 us); of the 730 that this takes three are, by up to 8 %, the others run at 0.38 to 1.02 times.
  return 5.6 + weights_us + end_us <= 0.8 * others * problems;
}

// The same up to 16 rows, where the streaming kernel (it needs K % 1024 == 0 and 256 strips) or the skinny one would run; what the
// slices cost shows against the shortest launches and the fewest rows.  Times relative to those kernels, cold weights:
//   B's many slices (11264, 13312) 1.08 to 1.41 against the streaming kernel, whatever the rows;
//   A's eight and more at 448 strips and beyond 1.06 to 1.15 (7168 x 16384), at 256 and 320 strips 0.81 to 0.99;
//   up to 4 rows at 384 strips and beyond 1.00 to 1.12 (7168 x 7168 11.2 -> 12.3 us), from K = 20480 on 0.85 to 0.96;
//   5 to 8 rows at 384 to 448 strips of up to 7168 bytes 1.01 to 1.05;
//   E's slices (a K that 1024 does not divide) on 64 strips and more 0.93 to 1.45 against the skinny kernel, 1.18 on average (8 x
//   4096 x 1536 4.4 -> 6.2 us), K = 1536 on fewer strips too; it runs a group problem by problem, which takes twice as long.
//   Longer K on fewer than 64 strips keeps them (8 x 768 x 2304 4.6 -> 5.4 us).
static inline bool few_rows_slices_ahead(RowsPick pick, long long M, long long N, long long K, int problems) {
  const long long strips = (N + 15) / 16 * problems;
  if (K % SBK != 0 || strips < 256) return pick.tiling != ROWS_E || problems > 1 || (strips < 64 && K > 1536);
  if (pick.tiling == ROWS_B) return false;
  if (strips <= 320) return true;
  if (pick.tiling == ROWS_A && pick.slices >= 8) return false;
  if (M <= 4) return K >= 20480;
  return M > 8 || K > 7168 || strips > 512;
}

// Blocks of 16 rows to a workgroup, one slice; 0 = the rows are too many for the kernel.  As few as find a CU each: a narrow output has
// fewer strips than there are CUs, and what its launch takes is a chain: the rows' copies, then the weights', then one block's sums
// after the other.  Workgroups of one strip share an XCD, whose L2 hands the weights to the later ones.  The line is one workgroup to a CU, also
// where two fit: beyond it they share the copies' rate, or run one after the other.  Cold weights, us, all blocks in one workgroup / so / a
// block less: 48 x 768 x 768 3.81 / 3.29, 48 x 768 x 3072 6.29 / 4.65, 64 x 1024 x 5120 8.83 / 5.97, 32 x 2048 x 2048 4.04 / 3.61,
// 64 x 2048 x 2048 4.98 / 4.05 / 4.74, 64 x 2048 x 4096 7.42 / 6.56 / 9.59, 64 x 1536 x 3072 7.05 / 5.74 / 8.22; left whole: 32 x 2560 x 2560
// 5.11, split 6.20, 32 x 3072 x 1024 3.56 / 3.95, 48 x 4096 x 4096 8.43 / 12.22.
// Beyond 64 rows the tiled kernels are the others, whose few tiles walk K one after the other or meet in slices: as long as every
// workgroup is resident (two to a CU, three or four blocks each, where they fit) this is ahead of them, us before / so: 128 x 768 x 768 5.6 / 3.7,
// 144 x 768 x 3072 13.9 / 5.9, 128 x 2048 x 2048 10.6 / 5.2, 256 x 2048 x 2048 14.2 / 7.4, 144 x 2560 x 2560 12.6 / 8.9, 192 x 2304 x 768 6.3 / 5.4; not so beyond that: 256 x 2304 x 768 6.3 / 7.5, 256 x 2560 x 2560 12.2 / 13.3.
// `N`: columns of one problem; `strips`: of all of them.
static inline int rows_blocks_each(int tiling, long long M, long long N, long long strips, int cus) {
  const int blocks = (int)((M + 15) / 16);
  const long long grid = (strips + 7) / 8 * 8;
  auto fits = [&](int each, long long slots) { return grid * ((blocks + each - 1) / each) <= slots; };
  if (blocks <= 4) {
    for (int each = 1; each < blocks; ++each)
      if (fits(each, cus)) return each;
    return blocks;
  }
  // (given up, as the split products have these shapes to themselves, tests of their forms among them: 128 x 1024 x 4096 12.7 / 6.3,
  // 320 x 768 x 3072 14.8 / 7.5, three 192 x 256 x 3072 49 / 7.3)
  if (tiling == ROWS_F || N < 768 || (tiling == ROWS_G && M > 256)) return 0;
  for (int each = 1; each <= 4; ++each)
    if (fits(each, cus)) return each;
  const bool pairs = tiling == ROWS_A || tiling == ROWS_B || tiling == ROWS_D || tiling == ROWS_E;
  return !pairs ? 0 : fits(3, 2LL * cus) ? 3 : fits(4, 2LL * cus) ? 4 : 0;
}

// Six and eight slices of A run as three and four of F: half as many tiles to park, and to add at the end.  24 x 4096 x 16384 17.5 us,
// 15.9 so; 64 x 7168 x 16384 35.7 / 28.9, 5 x 2048 x 16384 10.9 / 9.8; 220 shapes of 768 to 12288 columns and 2 to 64 rows 0.92 times the time
// in the mean, worst 1.04 (33 x 768 x 12288).  Four as two are level (8192: 16 and 48 x 2048 1.03 and 1.05, 17 to 48 x 8192 0.94 to 0.96),
// twelve as six not everywhere ahead (768 columns 1.02).
static inline RowsPick rows_paired(RowsPick pick, long long K) {
  return pick.tiling == ROWS_A && (K == 12288 || K == 16384) ? RowsPick{ROWS_F, pick.slices / 2} : pick;
}

// What launches: the acceptance tests and prices are those of the slices before they are paired.
static inline RowsPick rows_pick(long long M, long long N, long long K, int cus = num_cus(), int problems = 1) {
  if (M < 1 || M > TI_ROWS_ABREAST_M || N < 1 || K < 768 || K > (1 << 20)) return {ROWS_NONE, 1};
  RowsPick pick{ROWS_NONE, 1};
  if (K == 4096) pick = {ROWS_F, 1};
  else if (K % 5120 == 0) pick = {ROWS_C, (int)(K / 5120)};
  else if (K % 3584 == 0) pick = {ROWS_H, (int)(K / 3584)};
  else if (K % 2048 == 0) pick = {ROWS_A, (int)(K / 2048)};
  else if (K % 3072 == 0) pick = {ROWS_G, (int)(K / 3072)};
  else if (K % 2560 == 0) pick = {ROWS_D, (int)(K / 2560)};
  else if (K % 1024 == 0) pick = {ROWS_B, (int)(K / 1024)};
  else if (K % 768 == 0) pick = {ROWS_E, (int)(K / 768)};
  else return {ROWS_NONE, 1};
  if (M > TI_ROWS_MAX_M && (pick.slices > 1 || rows_blocks_each(pick.tiling, M, N, (N + 15) / 16 * problems, cus) == 0)) return {ROWS_NONE, 1};
  if (cus / 8 < pick.slices) return {ROWS_NONE, 1};  // an XCD has room for one workgroup of every slice
  // The parked tiles of all slices stay a fraction of the weights; the placement words of the groups, 64 bytes apart,
  // fit a stream's block of 4096; only whole strips are parked.
  if (pick.slices > 1 &&
      (pick.slices > 16 || 2 * cus / pick.slices > 256 || 8 * pick.slices * M > K || N % 16 != 0))
    return {ROWS_NONE, 1};
  if (pick.slices > 1 && !(M <= 16 ? few_rows_slices_ahead(pick, M, N, K, problems)
                                   : rows_slices_ahead(pick, M, N, K, problems, cus)))
    return {ROWS_NONE, 1};
  return rows_paired(pick, K);
}

template <class Cfg>
static int launch_rows_cfg(const GemmParams& p, const GemmGroup& grp, int strips, int per_problem, hipStream_t stream) {
  const int slots = num_cus() * Cfg::PER_CU / 8 * 8;
  const long long need = (long long)((strips + 7) / 8) * 8 * p.splits;
  const int grid = need < slots ? (int)need : slots;
  const int groups = grid / 8 / p.splits * 8;
  const int lds = Cfg::LDS_BYTES + ((strips + groups - 1) / groups + 3) / 4 * 256;
  if (lds > 160 * 1024) return -1;  // so wide an output that the bias of a workgroup's strips leaves the ring no room
  static std::atomic<unsigned long long> lds_ok{0};
  if (int rc = allow_lds(gemm_rows_kernel<Cfg>, 160 * 1024, lds_ok)) return rc;
  const unsigned abreast = (unsigned)((p.M + 16 * Cfg::MX - 1) / (16 * Cfg::MX));  // rows_blocks_each; slices hold all rows
  hipLaunchKernelGGL(gemm_rows_kernel<Cfg>, dim3((unsigned)grid, abreast), dim3(Cfg::NT), lds, stream, p, grp, strips, per_problem);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
  return TI_OK;
}

template <int KIND, bool GROUPED, int MX>
static int launch_rows_mx(int tiling, const GemmParams& p, const GemmGroup& grp, int strips, int per_problem,
                          hipStream_t stream) {
  switch (tiling) {
    case ROWS_A: return launch_rows_cfg<RowsCfg<KIND, MX, 8, 4, 4, 4, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_B: return launch_rows_cfg<RowsCfg<KIND, MX, 4, 4, 4, 4, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_C: return launch_rows_cfg<RowsCfg<KIND, MX, 10, 2, 8, 8, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_D: return launch_rows_cfg<RowsCfg<KIND, MX, 10, 2, 8, 4, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_F:
      if constexpr (MX == 4) return launch_rows_cfg<RowsCfg<KIND, MX, 8, 4, 4, 8, GROUPED>>(p, grp, strips, per_problem, stream);
      else return launch_rows_cfg<RowsCfg<KIND, MX, 4, 2, 4, 16, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_H: return launch_rows_cfg<RowsCfg<KIND, MX, 7, 7, 2, 8, GROUPED>>(p, grp, strips, per_problem, stream);
    case ROWS_G: return launch_rows_cfg<RowsCfg<KIND, MX, 6, 2, 8, 8, GROUPED>>(p, grp, strips, per_problem, stream);
    default: return launch_rows_cfg<RowsCfg<KIND, MX, 3, 3, 5, 4, GROUPED>>(p, grp, strips, per_problem, stream);
  }
}

// Library-owned home for the parked tiles of launches of up to 16 rows, one block per stream (see gemm_s8.hip).
static constexpr long long kRowsParkBytes = 2 << 20;
int rows_split_prepare(hipStream_t stream, GemmParams& q, void** park);

// What the calling thread's last linear did here: form 0 = it ran on another kernel, 1 = one slice, 2 = slices that meet in
// one launch, 3 = two launches.
struct RowsLast {
  int form, tiling, slices;
};
extern thread_local RowsLast g_rows_last;

// The linear (or GROUPED: up to four linears of one shape on the same activations) through gemm_rows_kernel.  Returns a
// TI_* status, or -1 when the shape, the alignment or the workspace does not allow it (the caller goes on to the other
// kernels).  `workspace` as for the split-K forms: problems * slices * M * N * 4 bytes when slices > 1 and M > 16.
template <int KIND, bool GROUPED>
static int launch_rows(const GemmParams& p_in, const GemmGroup& grp, int problems, void* workspace,
                       long long workspace_bytes, hipStream_t stream) {
  if (p_in.batch != 1 || p_in.lda != p_in.K || p_in.ldb != p_in.K) return -1;
  const RowsPick pick = rows_pick(p_in.M, p_in.N, p_in.K, num_cus(), problems);
  if (pick.tiling == ROWS_NONE) return -1;
  GemmParams p = p_in;
  p.splits = pick.slices;
  p.arrivals = nullptr;
  p.parts = nullptr;
  const int per_problem = (p.N + 15) / 16, strips = per_problem * problems;
  const int mx = pick.slices > 1 ? (p.M + 15) / 16 : rows_blocks_each(pick.tiling, p.M, p.N, strips, num_cus());
  const long long park = (long long)problems * pick.slices * p.M * p.N * 4;
  bool two_launches = false;
  if (pick.slices > 1) {
    const bool given = workspace != nullptr && workspace_bytes >= park && (reinterpret_cast<uintptr_t>(workspace) & 255) == 0;
    const bool own = p.M <= 16 && park <= kRowsParkBytes;
    if (!given && !own) return -1;
    void* home = nullptr;
    const int usable = rows_split_prepare(stream, p, &home);
    if (usable < 0) return -usable;
    if (usable) {
      p.parts = given ? workspace : home;
    } else {  // without a workspace the kernels that keep no state, as in every graph: 16 x 5120 x 20480 31.8 us against 20.7
      if (!given) return -1;
      p.arrivals = nullptr;
      p.parts = workspace;
      two_launches = true;
    }
  }
  int rc;
  switch (mx) {
    case 1: rc = launch_rows_mx<KIND, GROUPED, 1>(pick.tiling, p, grp, strips, per_problem, stream); break;
    case 2: rc = launch_rows_mx<KIND, GROUPED, 2>(pick.tiling, p, grp, strips, per_problem, stream); break;
    case 3: rc = launch_rows_mx<KIND, GROUPED, 3>(pick.tiling, p, grp, strips, per_problem, stream); break;
    default: rc = launch_rows_mx<KIND, GROUPED, 4>(pick.tiling, p, grp, strips, per_problem, stream); break;
  }
  if (rc == TI_OK) g_rows_last = {two_launches ? 3 : pick.slices > 1 ? 2 : 1, pick.tiling, pick.slices};
  if (rc || !two_launches) return rc;
  for (int i = 0; i < problems; ++i) {
    GemmParams q = p_in;
    if constexpr (GROUPED) {
      q.bias = grp.bias[i];
      q.C = grp.C[i];
      q.alpha = grp.alpha[i];
      q.beta = grp.beta[i];
    }
    const long long quads = ((long long)q.M * q.N + 3) / 4;
    const int* raw = static_cast<const int*>(workspace) + (long long)i * pick.slices * q.M * q.N;
    hipLaunchKernelGGL(splitk_reduce_kernel<KIND>, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, q, raw,
                       pick.slices);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "split-K reduce launch: %s", hipGetErrorString(e));
  }
  return TI_OK;
}

}  // namespace ti
