// LayerNorm-quantise and the int8 linears that read its result, in one launch, for the few rows of a decode step:
// q = LayerNormQ(hidden) for up to 4 rows, then up to three problems of one shape out[i] = s8(fma(alpha, q . W[i], beta * bias)).
//
// By itself the LayerNorm of one row is a chain of latencies (launch, row, two sums, store: 4 us at 5120, 2.3 at 768), during
// which nothing else runs, although the weights of the linear behind it depend on nothing.  Here every workgroup normalises the
// rows itself (the row, gamma and beta come from its XCD's L2) while its first weight rows are on their way: eight waves hold
// some 120 KiB of them in registers a CU, more than the two microseconds of the chain let through.  One workgroup to a CU, so
// that the chain runs 256 times and not once for every four weight rows.
//
// Bound by HBM (each weight byte is read once).  The products are those of gemm_gemv_kernel: a wave owns one weight row at a time
// and reads it flat, 16 consecutive bytes to a lane; v_dot4 against the quantised rows in the LDS; integer sums.  The
// LayerNorm has the lanes and the order of ln_q_rows_kernel, so its bits.
// us, cold weights, LayerNorm kernel and linear apart / in one launch, launches back to back: three 1 x 5120 x 5120 18.5 / 14.5,
// 1 x 20480 x 5120 21.4 / 17.8 (5.9 TB/s), three 1 x 768 x 768 6.4 / 5.6, 1 x 10240 x 2560 10.6 / 7.7, 2 x 20480 x 5120 21.5 / 18.9,
// 1 x 36864 x 9216 53.4 / 51.3.
#include "ln_math.h"

namespace ti {

// wave sum of an int, in lane 63
__device__ __forceinline__ int wave_sum_to_63(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}

// the LDS is all that the waves exchange through: loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// NC: KiB of a weight row and, as 256 lanes hold four elements each, chunks of a lane of the LayerNorm; MX: rows of activations;
// DEPTH: weight rows of a wave in flight.
// Waves of a workgroup: four to each row that is normalised, which for four rows are sixteen where the registers allow it (two rows
// one after the other in a wave: three 4 x 768 x 768 7.5 us, 6.5 so).
template <int NC, int MX>
constexpr int ln_linear_waves() { return MX == 4 && NC <= 3 ? 16 : 8; }

template <class T, int NC, int MX>
__global__ __launch_bounds__((64 * ln_linear_waves<NC, MX>())) void ln_linear_kernel(LnLinear p) {
  constexpr int WIDE = ln_linear_waves<NC, MX>() / 8;
  constexpr int DEPTH = (NC == 1 ? 8 : NC == 2 ? 6 : NC == 3 ? 4 : NC <= 5 ? 3 : 2) / WIDE;
  constexpr int GROUPS = MX == 1 ? 1 : 2 * WIDE;   // rows normalised side by side, four waves each
  constexpr int RG = MX / GROUPS;           // rows of a group of waves
  using Raw = typename Chunk<T>::type;
  extern __shared__ __attribute__((aligned(16))) char xs[];  // [MX][NC * 1024], zeros beyond K
  __shared__ float red[2][MX][4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int K = p.K, N = p.N, M = p.M, total = N * p.problems;
  const int nchunks = K >> 2;

  // ---- the rows of this group of waves, gamma and beta: first in line
  const int t = tid & 255, group = wave >> 2;
  // (the forms beyond five serve two lengths each)
  auto in_row = [&](int i) { return i < NC - (NC > 5 ? 2 : 1) || t + i * 256 < nchunks; };
  auto chunk = [&](int i) { return in_row(i) ? t + i * 256 : nchunks - 1; };
  Raw a[RG][NC], g_raw[NC], b_raw[NC];
  const bool norm = group < GROUPS;
  if (norm) {
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      const int m = group * RG + j < M ? group * RG + j : M - 1;
      const Raw* row = reinterpret_cast<const Raw*>(static_cast<const T*>(p.hidden) + (long long)m * K);
#pragma unroll
      for (int i = 0; i < NC; ++i) a[j][i] = row[chunk(i)];
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      g_raw[i] = reinterpret_cast<const Raw*>(p.gamma)[chunk(i)];
      b_raw[i] = reinterpret_cast<const Raw*>(p.beta)[chunk(i)];
    }
  }

  // ---- weight rows: row number r of all problems, flat.  A buffer of one row (none beyond the last: no memory is read), so
  // that lanes beyond K read zeros.
  const int step = gridDim.x * waves;
  const int first = blockIdx.x * waves + wave;
  v4i w[DEPTH][NC];
  auto problem_of = [&](int r, int& n) {
    int prob = 0;
    n = r;
    if (n >= N) { n -= N; prob = 1; }
    if (n >= N) { n -= N; prob = 2; }
    return prob;
  };
  auto fetch = [&](int d, int r) {
    const bool live = r < total;
    int n;
    const int prob = problem_of(live ? r : 0, n);
    const int8_t* W = prob == 0 ? p.W[0] : prob == 1 ? p.W[1] : p.W[2];
    const __amdgpu_buffer_rsrc_t row =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(W + (long long)n * K), 0, live ? K : 0, 0x00020000);
#pragma unroll
    for (int u = 0; u < NC; ++u)
      w[d][u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(row, u * 1024 + lane * 16, 0, 2));
  };
  // lane l has the bias of this wave's weight row number l (ln_linear_takes: there are no more than 64)
  int bias = 0;
  {
    const int mine = first + lane * step;
    int n;
    const int prob = problem_of(mine < total ? mine : 0, n);
    if (mine < total) bias = (prob == 0 ? p.bias[0] : prob == 1 ? p.bias[1] : p.bias[2])[n];
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(d, first + d * step);

  // ---- LayerNorm-quantise (the arithmetic of ln_q_rows_kernel on a stream that is only read)
  const float fK = (float)K;
  v4f r[RG][NC];
  if (norm) {
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        r[j][i] = to_f32(a[j][i]);
        if (in_row(i)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s = s + r[j][i][e];
        }
      }
      s = wave_butterfly_sum(s);
      if (lane == 0) red[0][group * RG + j][wave & 3] = s;
    }
  }
  lds_barrier();
  float mu[RG];
  if (norm) {
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      const float* part = red[0][group * RG + j];
      mu[j] = (((part[0] + part[1]) + part[2]) + part[3]) / fK;
      float s2 = 0.0f;
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        if (in_row(i)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float d = r[j][i][e] - mu[j];
            const float sq = d * d;
            s2 = s2 + sq;
          }
        }
      }
      s2 = wave_butterfly_sum(s2);
      if (lane == 0) red[1][group * RG + j][wave & 3] = s2;
    }
  }
  lds_barrier();
  if (norm) {
#pragma unroll
    for (int j = 0; j < RG; ++j) {
      const float* part = red[1][group * RG + j];
      const float var = (((part[0] + part[1]) + part[2]) + part[3]) / fK;
      const float rstd = 1.0f / __builtin_sqrtf(var + p.eps);
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        const v4f g = to_f32(g_raw[i]), b = to_f32(b_raw[i]);
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = as_stored<T>(__builtin_fmaf((r[j][i][e] - mu[j]) * rstd, g[e], b[e]));
        *reinterpret_cast<int*>(xs + ((group * RG + j) * NC * 1024) + (t + i * 256) * 4) =
            in_row(i) ? pack_s8x4(y[0], y[1], y[2], y[3]) : 0;
      }
    }
  }
  lds_barrier();

  // ---- products.  The quantised rows stay in registers where they leave room for the weights (four rows of 5120 read from the
  // LDS again for every weight row: 20480 outputs 24.0 us, 21.9 so).
  constexpr bool IN_REGS = MX * NC <= 20;
  v4i xr[IN_REGS ? MX : 1][IN_REGS ? NC : 1];
  if constexpr (IN_REGS) {
#pragma unroll
    for (int m = 0; m < MX; ++m)
#pragma unroll
      for (int u = 0; u < NC; ++u) xr[m][u] = *reinterpret_cast<const v4i*>(xs + m * (NC * 1024) + u * 1024 + lane * 16);
  }
  int row_no = 0;
  for (int r0 = first; r0 < total; r0 += DEPTH * step) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int here = r0 + d * step;
      int acc[MX];
#pragma unroll
      for (int m = 0; m < MX; ++m) acc[m] = 0;
#pragma unroll
      for (int u = 0; u < NC; ++u) {
#pragma unroll
        for (int m = 0; m < MX; ++m) {
          v4i xv;
          if constexpr (IN_REGS) xv = xr[m][u];
          else xv = *reinterpret_cast<const v4i*>(xs + m * (NC * 1024) + u * 1024 + lane * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[m] = __builtin_amdgcn_sdot4(w[d][u][e], xv[e], acc[m], false);
        }
      }
      fetch(d, here + DEPTH * step);
#pragma unroll
      for (int m = 0; m < MX; ++m) acc[m] = wave_sum_to_63(acc[m]);
      const int bv = __builtin_amdgcn_readlane(bias, row_no++ & 63);
      if (here < total) {
        int n;
        const int prob = problem_of(here, n);
        const float alpha = prob == 0 ? p.alpha[0] : prob == 1 ? p.alpha[1] : p.alpha[2];
        const float beta = prob == 0 ? p.beta_s[0] : prob == 1 ? p.beta_s[1] : p.beta_s[2];
        int8_t* out = prob == 0 ? p.out[0] : prob == 1 ? p.out[1] : p.out[2];
        const float bt = beta * (float)bv;
        if (lane == 63) {
#pragma unroll
          for (int m = 0; m < MX; ++m) {
            int o = rne_sat_s32(__builtin_fmaf(alpha, (float)acc[m], bt));
            o = o < p.lo ? p.lo : o;
            o = o > 127 ? 127 : o;
            if (m < M) out[(long long)m * N + n] = (int8_t)o;
          }
        }
      }
    }
  }
}

// Three and four rows: level with two launches up to 5120 (the row's products and the LayerNorm of every row in every workgroup
// take what the launch saved: 4 x 20480 x 5120 22.0 us against 21.5, three 4 x 2560 x 2560 9.2 / 9.7) and a launch less for the
// host; beyond, where there is one launch to some 40 us, behind (4 x 36864 x 9216 57.4 / 55.1).
bool ln_linear_takes(const LnLinear& p, bool half) {
  auto al = [](const void* q, uintptr_t mask) { return (reinterpret_cast<uintptr_t>(q) & mask) == 0; };
  const uintptr_t row = half ? 7 : 15;
  if (p.M < 1 || p.M > LN_LINEAR_ROWS || p.K < 16 || p.K % 16 != 0 || p.K > 9 * 1024 || (p.M > 2 && p.K > 5 * 1024) || p.problems < 1 || p.problems > 3) return false;
  // a wave's weight rows: up to 64 of them (five waves to a CU at least)
  if (p.N < 1 || (long long)p.N * p.problems > 64LL * 5 * compute_units()) return false;
  if (!al(p.hidden, row) || !al(p.gamma, row) || !al(p.beta, row)) return false;
  for (int i = 0; i < p.problems; ++i)
    if (!al(p.W[i], 15)) return false;
  return true;
}

template <class T, int NC, int MX>
static int launch_cfg(const LnLinear& p, int cus, hipStream_t stream) {
  const long long total = (long long)p.N * p.problems;
  // One row: as many waves as leave the fewest idle in the last round of weight rows.
  int waves = ln_linear_waves<NC, MX>();
  if (MX == 1) {
    auto fill = [&](int w) {
      const long long round = (long long)cus * w;
      return (double)total / ((double)((total + round - 1) / round) * round);
    };
    for (int w = 7; w >= 5; --w)
      if (fill(w) > 1.04 * fill(waves)) waves = w;
  }
  const long long need = (total + waves - 1) / waves;
  const unsigned grid = (unsigned)(need < cus ? need : cus);
  hipLaunchKernelGGL((ln_linear_kernel<T, NC, MX>), dim3(grid), dim3(waves * 64), MX * NC * 1024, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "layernorm + linear launch: %s", hipGetErrorString(e));
  return TI_OK;
}

template <class T, int NC>
static int launch_nc(const LnLinear& p, int cus, hipStream_t stream) {
  if (p.M == 1) return launch_cfg<T, NC, 1>(p, cus, stream);
  if constexpr (NC <= 5) {
    if (p.M > 2) return launch_cfg<T, NC, 4>(p, cus, stream);
  }
  return launch_cfg<T, NC, 2>(p, cus, stream);
}

template <class T>
static int launch_t(const LnLinear& p, int cus, hipStream_t stream) {
  switch ((p.K + 1023) / 1024) {
    case 1: return launch_nc<T, 1>(p, cus, stream);
    case 2: return launch_nc<T, 2>(p, cus, stream);
    case 3: return launch_nc<T, 3>(p, cus, stream);
    case 4: return launch_nc<T, 4>(p, cus, stream);
    case 5: return launch_nc<T, 5>(p, cus, stream);
    case 6:
    case 7: return launch_nc<T, 7>(p, cus, stream);
    default: return launch_nc<T, 9>(p, cus, stream);
  }
}

int launch_ln_linear(const LnLinear& p, bool half, hipStream_t stream) {
  const int cus = compute_units();
  return half ? launch_t<_Float16>(p, cus, stream) : launch_t<float>(p, cus, stream);
}

}  // namespace ti
