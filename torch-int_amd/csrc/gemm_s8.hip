// Host-side entry of the INT8 GEMM family: dispatch over the epilogue kinds (each kind's kernels are
// compiled in a translation unit of their own, gemm_s8_kinds.hip with -DTI_KIND=n), the grouped q/k/v
// launches, the split-K slice GEMM and the workspace query.
#include <cstdlib>
#include <mutex>

#include "gemm_s8_impl.h"

namespace ti {

long long gemm_workspace_bytes(long long M, long long N, long long K, bool least) {
  if (M > 1024) {  // the rows beyond the last multiple of 256 as a small problem of their own (row_split_rows)
    long long need = 0;
    const int r = row_split_rows(M, N, K, &need);
    if (r <= 0) return 0;
    // the first rows are a problem of their own too: at exactly 1024 of them they may split K themselves
    const long long head = M - r <= 1024 ? gemm_workspace_bytes(M - r, N, K, least) : 0, rest = gemm_workspace_bytes(r, N, K, least);
    return head > need ? (head > rest ? head : rest) : need > rest ? need : rest;
  }
  const RowsPick rows = least ? RowsPick{ROWS_NONE, 1} : rows_pick(M, N, K);
  if (M > 16 && rows.tiling != ROWS_NONE && (N % 16 == 0 || K % SBK == 0)) return rows.slices > 1 ? (long long)rows.slices * M * N * 4 : 0;
  int tile = SPLIT_128;
  const int s = choose_splits(M, N, K, &tile, nullptr, 1, !least);
  if (s <= 1) return 0;
  long long one_launch = 0;
  return !least && one_launch_split(tile, s, M, N, K, &one_launch) ? one_launch : (long long)s * M * N * 4;
}

// The same for the accumulating epilogue, whose slices never meet in one launch and may be others.
long long gemm_acc_workspace_bytes(long long M, long long N, long long K) {
  long long most = gemm_workspace_bytes(M, N, K, false);
  auto more = [&](long long rows) {
    if (rows <= 16 || rows > 1024) return;
    const RowsPick pick = rows_pick(rows, N, K);
    if (pick.tiling != ROWS_NONE && (N % 16 == 0 || K % SBK == 0)) return;
    const int s = choose_splits(rows, N, K, nullptr, nullptr, 1, true, false);
    if (s > 1 && (long long)s * rows * N * 4 > most) most = (long long)s * rows * N * 4;
  };
  const int r = M > 1024 ? row_split_rows(M, N, K) : 0;
  more(r > 0 ? r : M);
  if (r > 0) more(M - r);
  return most;
}

// one per epilogue kind (EpiKind value n), each in its own translation unit
int launch_gemm_kind_0(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_1(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_2(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_3(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_4(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_5(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_6(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_7(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_8(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);
int launch_gemm_kind_9(const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream);

int compute_units() { return num_cus(); }

int gemm_row_split(long long M, long long N, long long K) { return row_split_rows(M, N, K); }

long long bmm_workspace_bytes(long long batch, long long M, long long N, long long K) {
  if (batch == 1) return gemm_workspace_bytes(M, N, K);  // one problem: the linears' split-K forms
  const int s = batched_splits(batch, M, N, K);
  return s > 1 ? (long long)s * batch * M * N * 4 : 0;
}

thread_local const char* g_last_kernel = "";
thread_local const char* g_last_form = "";
const char* last_gemm_kernel() { return g_last_kernel; }
const char* last_gemm_form() { return g_last_form; }
thread_local RowsLast g_rows_last = {0, 0, 0};
int last_rows(int* tiling, int* slices) {
  *tiling = g_rows_last.tiling;
  *slices = g_rows_last.slices;
  return g_rows_last.form;
}

// ---------------------------------------------------------------------------
// State of the one-launch split-K (the FUSED form of gemm_pipe16q_kernel), per device.
//
// Arrival counters: zero when the code object is loaded, and every launch leaves them zero (the wave that arrives
// last puts its counter back).  Launches on one stream run one after the other, so each stream that uses the
// fused form gets a block of counters of its own (kFusedStreams of them per device; further streams take the
// two-launch form).
//
// Placement: the fused form needs all workgroups whose ids are congruent mod 8 to run on one XCD.  That is how the
// hardware deals workgroups out (round robin over the XCDs; the XCD of workgroup 0 depends on the queue).  A probe
// launch records the XCC id register of 256 workgroups once per device; unless it shows one XCC per residue class,
// eight different ones, the fused form stays off.  Every fused launch checks itself as well: the workgroups of a
// tile mark their XCC in a word of the tile, and one that finds another XCC's mark raises a flag in host memory;
// the flag is looked at before every later launch and turns the fused form off with an error.
static constexpr int kFusedStreams = 8;
static constexpr int kFusedCounters = 32768;            // per stream: tiles x waves
static constexpr int kFusedTiles = kFusedCounters / 8;  // per stream: one XCC word per tile
static __device__ __align__(256) int g_fused_arrivals[kFusedStreams * (kFusedCounters + kFusedTiles)];

// State of gemm_rows_kernel's slices, apart from that of the form above: decoding goes through it on every stream, and a
// graph that holds a block of counters from above must not meet eager decoding there.  A block per stream, used by one
// launch of that stream at a time: counters and placement words, and for up to 16 rows, whose callers hold no workspace,
// the parked tiles (written in full before they are read).  A stream keeps its block for the life of the process, so
// that no launch on its way can lose it, and launches that a graph records get none: a replay is not bound to the stream
// it was recorded on.  33 blocks, as many as a program gets streams of from torch (the default one and a pool of 32);
// further streams take the other forms.
static constexpr int kRowsStreams = 33;
// rows_pick takes at most 256 groups of four or eight waves, of sixteen (half as many slices, half as many workgroups to a CU) too;
// a placement word a group, 64 bytes apart
static constexpr int kRowsCounters = 4096, kRowsWords = 4096;
static_assert(kRowsCounters >= 256 * 16 && kRowsWords >= 256 * 16, "a counter to a wave, a placement word to a group");
static __device__ __align__(256) int g_rows_arrivals[kRowsStreams * (kRowsCounters + kRowsWords)];
static __device__ __align__(256) char g_rows_park[kRowsStreams * kRowsParkBytes];

__global__ void xcc_probe_kernel(unsigned* out) {
  if (threadIdx.x == 0)
    __hip_atomic_store(out + blockIdx.x, __builtin_amdgcn_s_getreg((3 << 11) | 20) & 0xf, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);  // HW_REG_XCC_ID
}
static constexpr int kProbeWords = 256;
enum RowsSlot : signed char { ROWS_VACANT = 0, ROWS_PROBING, ROWS_USABLE, ROWS_REFUSED };

struct FusedDevice {
  std::mutex lock;
  int state = 0;  // 0 = not probed yet, 1 = usable, -1 = off
  int* arrivals = nullptr;
  int* host_words = nullptr;  // [0] = the misplacement flag, [1 .. 256] = the probe's output, then 256 words per rows slot
  int* host_words_dev = nullptr;
  int* rows_arrivals = nullptr;
  char* rows_park = nullptr;
  hipStream_t rows_streams[kRowsStreams] = {};
  RowsSlot rows_state[kRowsStreams] = {};
  hipStream_t streams[kFusedStreams] = {};
  bool live[kFusedStreams] = {};
  bool pinned[kFusedStreams] = {};  // a launch with this slot's counters was recorded into a graph: never handed on
};
static FusedDevice g_fused[64];

// -1 = not decided yet: the environment variable TORCH_INT_FUSED_SPLITK=0 switches the form off
static std::atomic<int> g_fused_on{-1};

int set_fused_split(int enable) {
  int before = g_fused_on.load(std::memory_order_relaxed);
  if (before < 0) {
    const char* v = getenv("TORCH_INT_FUSED_SPLITK");
    before = !(v && v[0] == '0');
  }
  if (enable >= 0) g_fused_on.store(enable ? 1 : 0, std::memory_order_relaxed);
  else g_fused_on.store(before, std::memory_order_relaxed);
  return before;
}
static bool fused_enabled() { return set_fused_split(-1) != 0; }

// The first use on a device allocates 35 KB of host memory and synchronises; a thread that must not allocate (the
// entry point that promises it) clears this around its call and then only uses a device that is ready.
static thread_local bool g_fused_may_probe = true;
void allow_fused_split_probe(bool allow) { g_fused_may_probe = allow; }

// While a thread records a graph in the global mode (torch's default), a query, a wait or an allocation by any other thread is
// an error there and here: it ends the recording.  Ours concern neither, so they are made in the relaxed mode.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  RelaxedCapture(const RelaxedCapture&) = delete;
  RelaxedCapture& operator=(const RelaxedCapture&) = delete;
};

// What 256 probe words say: 1 = one XCC per residue class of the workgroup id mod 8, eight different ones; -1 = another
// placement; 0 = not all of them are there yet.  Free of HIP calls so that it can be tested on the CPU.
int placement_of(const volatile int* words) {
  for (int i = 0; i < kProbeWords; ++i)
    if (words[i] == -1) return 0;
  unsigned seen = 0;
  for (int i = 0; i < kProbeWords; ++i)
    if (words[i] < 0 || words[i] > 15 || words[i] != words[i & 7]) return -1;
  for (int i = 0; i < 8; ++i) {
    if (seen & (1u << words[i])) return -1;  // two residue classes on one XCD: not the placement this needs
    seen |= 1u << words[i];
  }
  return 1;
}

// Starts the placement probe on `stream` (which must not be capturing); its words are at `at` of the host words.
static bool start_probe(FusedDevice& d, int at, hipStream_t stream) {
  for (int i = 0; i < kProbeWords; ++i) d.host_words[at + i] = -1;
  hipLaunchKernelGGL(xcc_probe_kernel, dim3(kProbeWords), dim3(64), 0, stream, reinterpret_cast<unsigned*>(d.host_words_dev + at));
  return hipGetLastError() == hipSuccess;
}
static bool probe_placement(FusedDevice& d, hipStream_t stream) {  // ... and waits for it
  RelaxedCapture relaxed;
  return start_probe(d, 1, stream) && hipStreamSynchronize(stream) == hipSuccess && placement_of(d.host_words + 1) == 1;
}

// Host words and device addresses of the current device, once.
static bool fused_memory(FusedDevice& d) {
  if (d.host_words != nullptr) return d.rows_park != nullptr;
  RelaxedCapture relaxed;
  void *arrivals = nullptr, *rows = nullptr, *park = nullptr;
  int* words = nullptr;
  if (hipGetSymbolAddress(&arrivals, HIP_SYMBOL(g_fused_arrivals)) != hipSuccess || arrivals == nullptr) return false;
  if (hipGetSymbolAddress(&rows, HIP_SYMBOL(g_rows_arrivals)) != hipSuccess || rows == nullptr) return false;
  if (hipGetSymbolAddress(&park, HIP_SYMBOL(g_rows_park)) != hipSuccess || park == nullptr) return false;
  if (hipHostMalloc(reinterpret_cast<void**>(&words), (1 + (1 + kRowsStreams) * kProbeWords) * sizeof(int),
                    hipHostMallocMapped) != hipSuccess)
    return false;
  words[0] = 0;
  if (hipHostGetDevicePointer(reinterpret_cast<void**>(&d.host_words_dev), words, 0) != hipSuccess) {
    (void)hipHostFree(words);
    return false;
  }
  d.arrivals = static_cast<int*>(arrivals);
  d.rows_arrivals = static_cast<int*>(rows);
  d.rows_park = static_cast<char*>(park);
  d.host_words = words;
  return true;
}

static bool is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) {
    (void)hipGetLastError();
    return true;  // unknown: treat as capturing (no probe, no registration)
  }
  return capturing != hipStreamCaptureStatusNone;
}

// 1 when a one-launch split-K GEMM on the current device has found a workgroup on an unexpected XCD (the output of
// that call cannot be trusted), 0 otherwise.  Reads one word of host memory; meaningful once the launches in
// question have finished.
int fused_split_faulted() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  FusedDevice& d = g_fused[dev];
  std::lock_guard<std::mutex> guard(d.lock);
  return d.host_words != nullptr && *reinterpret_cast<volatile int*>(d.host_words) != 0 ? 1 : 0;
}

// Decision logic of the fused form's bookkeeping, free of HIP calls so that it can be tested on the CPU.
// `flag` is the misplacement word, `state` the device state (0 not probed, 1 usable, -1 off).  Returns the action:
//   0 = take the two-launch form, 1 = go on (probe / slot lookup), -1 = report the misplacement and switch off.
int fused_flag_action(int state, int flag, bool enabled, long long counters, long long max_counters) {
  if (flag != 0 && state != 0) return -1;  // reported by whichever GEMM call comes next, fused or not
  if (!enabled || counters > max_counters) return 0;
  if (state < 0) return 0;
  return 1;
}

// Slot of `stream` among the `cap` slots of a device (`live[i]` = slot i holds a registered stream, `busy(i)` =
// that stream still has work queued): the stream's own slot, else a vacant one, else the first whose stream is
// idle (its counters are zero again: every launch leaves them zero), else -1.  `fresh` is set when the stream was
// not registered before.  Free of HIP calls so that it can be tested on the CPU.
template <class Busy>
static int pick_stream_slot(hipStream_t* streams, bool* live, int cap, hipStream_t stream, Busy busy, bool& fresh) {
  fresh = false;
  for (int i = 0; i < cap; ++i)
    if (live[i] && streams[i] == stream) return i;
  fresh = true;
  int slot = -1;
  for (int i = 0; i < cap && slot < 0; ++i)
    if (!live[i]) slot = i;
  for (int i = 0; i < cap && slot < 0; ++i)
    if (!busy(i)) slot = i;
  if (slot >= 0) {
    streams[slot] = stream;
    live[slot] = true;
  }
  return slot;
}

// CPU-testable face of pick_stream_slot: streams are plain integers, bit i of live_mask / busy_mask describes
// slot i; returns the slot and updates table / live_mask.
int fused_slot_for_test(long long* table, unsigned* live_mask, int cap, long long stream, unsigned busy_mask,
                        int* fresh) {
  hipStream_t tmp[32];
  bool live[32];
  if (cap > 32) cap = 32;
  for (int i = 0; i < cap; ++i) {
    tmp[i] = reinterpret_cast<hipStream_t>(table[i]);
    live[i] = (*live_mask >> i) & 1u;
  }
  bool f = false;
  const int slot = pick_stream_slot(tmp, live, cap, reinterpret_cast<hipStream_t>(stream),
                                    [&](int i) { return ((busy_mask >> i) & 1u) != 0; }, f);
  *live_mask = 0;
  for (int i = 0; i < cap; ++i) {
    table[i] = reinterpret_cast<long long>(tmp[i]);
    if (live[i]) *live_mask |= 1u << i;
  }
  *fresh = f ? 1 : 0;
  return slot;
}

static const char* kMisplacedMsg =
    "an earlier one-launch split-K GEMM on this device found a workgroup on an unexpected XCD and its result cannot "
    "be trusted (re-run it); the form is now switched off (TORCH_INT_FUSED_SPLITK=0 avoids it from the start)";

// Reports (once) a misplacement that an earlier fused launch on the current device flagged: TI_OK or TI_ERR_LAUNCH.
// Called at the start of every GEMM launch, whatever kernel it will take.
int fused_split_check() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return TI_OK;
  FusedDevice& d = g_fused[dev];
  if (d.host_words == nullptr) return TI_OK;  // never used here (written under the lock, before any fused launch)
  std::lock_guard<std::mutex> guard(d.lock);
  if (d.state == 1 && *reinterpret_cast<volatile int*>(d.host_words) != 0) {
    d.state = -1;
    return fail(TI_ERR_LAUNCH, "%s", kMisplacedMsg);
  }
  return TI_OK;
}

// counters == 0: only make the current device and `stream` ready (the probe)
int fused_split_prepare(hipStream_t stream, long long counters, GemmParams& q) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  FusedDevice& d = g_fused[dev];
  std::lock_guard<std::mutex> guard(d.lock);
  const int flag = d.host_words != nullptr ? *reinterpret_cast<volatile int*>(d.host_words) : 0;
  const int action = fused_flag_action(d.state, flag, fused_enabled(), counters, kFusedCounters);
  if (action < 0) {
    if (d.state == 1) {
      d.state = -1;
      return -fail(TI_ERR_LAUNCH, "%s", kMisplacedMsg);
    }
    return 0;  // already reported
  }
  if (action == 0) return 0;
  bool probed_now = false;  // the device's first probe ran on `stream` just now and vouches for it
  if (d.state == 0) {
    if (!g_fused_may_probe) return 0;
    // first use on this device: not while the stream records a graph (the probe allocates and synchronises)
    if (is_capturing(stream)) return 0;
    d.state = -1;
    if (!fused_memory(d) || !probe_placement(d, stream)) return 0;
    d.state = 1;
    probed_now = true;
  }
  bool fresh = false;
  const int slot = pick_stream_slot(d.streams, d.live, kFusedStreams, stream,
                                    [&](int i) {
                                      RelaxedCapture relaxed;
                                      return d.pinned[i] || hipStreamQuery(d.streams[i]) == hipErrorNotReady;
                                    },
                                    fresh);
  (void)hipGetLastError();  // a query of a destroyed stream leaves an error behind; the slot counts as idle
  if (slot < 0) return 0;
  if (fresh && !probed_now) {
    // a stream seen for the first time: the XCD on which its workgroup 0 starts may differ, and a stream made with
    // a CU mask may not deal workgroups out this way at all, so the probe runs on it once (it synchronises the
    // stream, so not during a capture or from a caller that must not wait: the slot is given back then)
    if (!g_fused_may_probe || is_capturing(stream) || !probe_placement(d, stream)) {
      d.live[slot] = false;
      return 0;
    }
  } else if (!d.pinned[slot] && is_capturing(stream)) {
    d.pinned[slot] = true;  // the recording keeps these counters for as long as the graph lives
  }
  q.arrivals = d.arrivals + (long long)slot * (kFusedCounters + kFusedTiles);
  q.xcc_seen = reinterpret_cast<unsigned*>(q.arrivals + kFusedCounters);
  q.xcc_error = d.host_words_dev;
  return 1;
}

// Slot of `stream` among `cap`: its own (fresh = false), else the first vacant one (fresh = true), else -1.  Slots are
// never handed on.  Free of HIP calls so that it can be tested on the CPU.
int pick_rows_slot(const hipStream_t* streams, const RowsSlot* state, int cap, hipStream_t stream, bool& fresh) {
  fresh = false;
  for (int i = 0; i < cap && state[i] != ROWS_VACANT; ++i)
    if (streams[i] == stream) return i;
  fresh = true;
  for (int i = 0; i < cap; ++i)
    if (state[i] == ROWS_VACANT) return i;
  return -1;
}

// Makes q ready for slices that meet in one launch of gemm_rows_kernel on `stream`: 1 = ready, *park = the stream's home
// for parked tiles; 0 = take another form; < 0 = minus the status of a misplacement to report.  Never waits for work that
// is queued: a stream's first call starts the placement probe on it and waits for that only where nothing is ahead of it
// (some 20 us); else calls take the other forms until the probe's words are there.
int rows_split_prepare(hipStream_t stream, GemmParams& q, void** park) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  FusedDevice& d = g_fused[dev];
  std::lock_guard<std::mutex> guard(d.lock);
  const int flag = d.host_words != nullptr ? *reinterpret_cast<volatile int*>(d.host_words) : 0;
  const int action = fused_flag_action(d.state, flag, fused_enabled(), 0, kFusedCounters);
  if (action < 0 && d.state == 1) {
    d.state = -1;
    return -fail(TI_ERR_LAUNCH, "%s", kMisplacedMsg);
  }
  // hipStreamPerThread is one handle for a stream of every thread
  if (action <= 0 || stream == hipStreamPerThread || is_capturing(stream)) return 0;
  if (d.host_words == nullptr && !g_fused_may_probe) return 0;  // the first use on a device allocates host memory
  if (!fused_memory(d)) {
    (void)hipGetLastError();  // not the launch's
    return 0;
  }
  bool fresh = false;
  const int slot = pick_rows_slot(d.rows_streams, d.rows_state, kRowsStreams, stream, fresh);
  if (slot < 0) return 0;
  const int words = 1 + (1 + slot) * kProbeWords;
  if (fresh) {
    RelaxedCapture relaxed;
    const bool idle = g_fused_may_probe && hipStreamQuery(stream) == hipSuccess;
    (void)hipGetLastError();  // a busy stream leaves "not ready" behind
    d.rows_streams[slot] = stream;
    d.rows_state[slot] = start_probe(d, words, stream) ? ROWS_PROBING : ROWS_REFUSED;
    if (idle) (void)hipStreamSynchronize(stream);
  }
  if (d.rows_state[slot] == ROWS_PROBING) {
    const int placement = placement_of(d.host_words + words);
    if (placement == 0) return 0;
    d.rows_state[slot] = placement > 0 ? ROWS_USABLE : ROWS_REFUSED;
    if (placement > 0 && d.state == 0) d.state = 1;  // a launch of this form reports a misplacement like any other
  }
  if (d.rows_state[slot] != ROWS_USABLE) return 0;
  q.arrivals = d.rows_arrivals + (long long)slot * (kRowsCounters + kRowsWords);
  q.xcc_seen = reinterpret_cast<unsigned*>(q.arrivals + kRowsCounters);
  q.xcc_error = d.host_words_dev;
  *park = d.rows_park + slot * kRowsParkBytes;
  return 1;
}

// CPU-testable face of rows_pick: slices (0 = the kernel does not take the shape) on a device of `cus` compute units.
int rows_pick_for_test(long long M, long long N, long long K, int cus, int* tiling) {
  const RowsPick pick = rows_pick(M, N, K, cus);
  *tiling = pick.tiling;
  return pick.tiling == ROWS_NONE ? 0 : pick.slices;
}

// CPU-testable face of pick_rows_slot: streams are plain integers, state[i] != 0 = slot i is taken; takes the slot.
int rows_slot_for_test(long long* table, signed char* state, int cap, long long stream, int* fresh) {
  bool f = false;
  static_assert(sizeof(hipStream_t) == sizeof(long long) && sizeof(RowsSlot) == 1, "plain tables");
  const int slot = pick_rows_slot(reinterpret_cast<const hipStream_t*>(table), reinterpret_cast<const RowsSlot*>(state), cap,
                                  reinterpret_cast<hipStream_t>(stream), f);
  if (slot >= 0) {
    table[slot] = stream;
    state[slot] = ROWS_USABLE;
  }
  *fresh = f ? 1 : 0;
  return slot;
}

// The probes of both forms on `stream` now rather than at its first calls.
int warm_fused_split(void* stream) {
  GemmParams unused;
  void* park = nullptr;
  const int rc = fused_split_prepare(static_cast<hipStream_t>(stream), 0, unused);
  if (rc > 0) (void)rows_split_prepare(static_cast<hipStream_t>(stream), unused, &park);
  return rc > 0 ? 1 : 0;
}

int launch_splitk_raw(int tile, const GemmParams& q, hipStream_t stream) {
  if (tile == SPLIT_128 && split_128_deep((long long)((q.M + 127) / 128) * ((q.N + 127) / 128) * q.batch, q.K, false, num_cus()))
    return launch_pipe16q<Pipe16QCfg<128, 128, 4, 2, EPI_S32_RAW, false, 5>>(q, stream);
  if (tile == SPLIT_128) return launch_pipe<PipeCfg<128, 128, 2, 2, 4, EPI_S32_RAW, false>>(q, stream);
  if (tile == SPLIT_256x160) return launch_pipe16q<Pipe16QCfg<256, 160, 4, 2, EPI_S32_RAW>>(q, stream);
  // Ten waves of 32x80 rather than four of 80x80: with one wave to a SIMD, what a wave reads and copies and what it multiplies come one after the other.
  // Cold weights, us, four / ten: 300 x 5120 x 20480 int8 51.3 / 48.6, fp32 52.3 / 49.7, 320 rows int32 53.5 / 50.4, 257 rows 47.7 / 46.3, 160 x 20480 x 5120
  // 38.7 / 38.4, 770 to 800 x 3200 x 20480 76.4 / 71.6.  Weights that the last-level cache holds are copied as fast either way, and ten waves read more
  // fragments: 1.00 to 1.03 times the time (300 x 5120 x 20480 43.7 / 44.7), 400 x 6400 x 12800 47.4 / 49.2 (cold 51.3 / 51.9).
  // 2x5 waves level, 5x1 of 32x160 behind, a fourth stage 0.3 behind.
  if (tile == SPLIT_160x160) return launch_pipe16q<Pipe16QCfg<160, 160, 5, 2, EPI_S32_RAW>>(q, stream);
  if (tile == SPLIT_128x80) return launch_pipe16q<Pipe16QCfg<128, 80, 4, 1, EPI_S32_RAW>>(q, stream);
  if (tile == SPLIT_128x160) return launch_pipe16q<Pipe16QCfg<128, 160, 4, 2, EPI_S32_RAW>>(q, stream);
  if (tile == SPLIT_128x288) return launch_pipe16q<Pipe16QCfg<128, 288, 4, 2, EPI_S32_RAW>>(q, stream);
  if (tile == SPLIT_128x192) return launch_pipe16q<Pipe16QCfg<128, 192, 4, 2, EPI_S32_RAW>>(q, stream);
  if (tile == SPLIT_256x288) return launch_pipe16q<Pipe16QCfg<256, 288, 4, 2, EPI_S32_RAW>>(q, stream);
  if (q.K % QBK == 0) return launch_pipe2<Pipe2Cfg<256, 256, 2, 4, EPI_S32_RAW, false>>(q, stream);
  return launch_pipe<PipeCfg<256, 256, 2, 4, 4, EPI_S32_RAW, false>>(q, stream);
}

// Tile width of the one persistent launch that runs a group of `count` [M,K] x [N,K] s8 linears at prefill sizes
// (160, 288, 256 or 128), or 0 when the problems run one after the other.
static int group_prefill_tile(long long M, long long N, long long K, int count) {
  if (!(M > 128 && K % QBK == 0 && K >= QBK && K <= PANEL_MAX_LD && count > 1)) return 0;
  const long long cus = num_cus();
  auto fill = [&](long long tiles) { return (double)tiles / (double)(((tiles + cus - 1) / cus) * cus); };
  const long long rows256 = (M + 255) / 256;
  const double e160 = N % 160 == 0 ? 0.88 * fill(rows256 * (N / 160) * count) : 0.0;
  const double e288 = N % 288 == 0 ? 0.95 * fill(rows256 * (N / 288) * count) : 0.0;
  // widths that only 128 divides (OPT-6.7B: 4096): 256x128 tiles, unless one problem at a time fills the CUs
  // with 256x256 tiles as well (three 2048x4096x4096: 98 -> 93 us, at 512 rows 57 -> 28 us; 2048x7168x7168
  // stays with three launches, 277 against 283 us)
  // (the line at 0.48: three 768x2048x2048 on 144 tiles 19.0 us, apart 27.4; 512 rows, 96 tiles, 20 apart)
  const double e256_alone = fill(rows256 * ((N + 255) / 256));
  double e128 = N % 128 == 0 ? 0.87 * fill(rows256 * (N / 128) * count) : 0.0;
  if (e128 < 0.48 || e128 <= e256_alone) e128 = 0.0;
  const double e = e160 > e288 ? (e160 > e128 ? e160 : e128) : (e288 > e128 ? e288 : e128);
  // Beyond 1024 rows the grouped launch and the problems one after the other are priced as price_wide prices tilings, and
  // 256x256 tiles are in the race too.  Grouped, 256x128 and 256x160 tiles take 0.97 and 0.98 times their price and 256x256 ones
  // 1.05 times, which have to be clearly ahead but in one round of a short K, where what a second round adds weighs most (three
  // 2048x2048x2048, 192 tiles: 34.6 us with weights from HBM, 34.5 on 384 of 256x128; 30.8 and 34.1 with weights that the
  // last-level cache holds).  1060 groups of three, widths 768 to 7168, 1025 to 8192 rows, weights from HBM, against the choice
  // without 256x256 tiles: 0.99 times the time, worst 1.03; at the plain price 97 of them lost more than 5 % (4096x5120x5120 266
  // -> 290 us).
  if (M > 1024 && wide_priced(M, N, K, 1)) {
    int tile = 0;
    double best = (double)count * (price_wide(M, N, K).us + 1.0);
    for (const WideRate& r : kWideRates) {
      const bool one_round = rows256 * (N / 256) * count <= cus;
      const double grouped = r.tile == WIDE_256x160 ? 0.98 : r.tile == WIDE_256x128 ? 0.97 : r.tile == WIDE_256x288 ? 1.0
                             : r.tile == WIDE_256x256 && K >= 2048 ? (one_round && K <= 2304 ? 1.03 : 1.08) : 0.0;  // 0: no such form
      if (grouped == 0.0 || N % r.bn != 0) continue;
      const double us = grouped * wide_us(r, M, N, K, count, false);
      if (us < best) {
        best = us;
        tile = r.bn;
      }
    }
    return tile;
  }
  if (e <= 0.0) return 0;
  // Up to 1024 rows a problem may have a one-round tiling of its own that needs no workspace (128x80, 128x192 or
  // 256x192 tiles over the whole of K): when the cost model prices the problems one after the other below the
  // grouped launch, they run that way (three 512x12288x12288: 260 us grouped on 256x128 tiles, 250 us apart;
  // three 512x5120x5120 stay grouped).  The group at 0.85 us per 64 bytes of K and full round of 256x256 tiles, by its efficiency.
  if (M <= 1024) {
    int tile = 0;
    double t_one = -1.0;
    const int splits = choose_splits(M, N, K, &tile, &t_one);
    if (splits == 1 && t_one > 0.0 && (tile == SPLIT_128x80 || tile == SPLIT_128x192 || tile == SPLIT_256x192)) {
      const double t_group = (double)count * M * N * (double)(K / 64) * 0.85 / (65536.0 * (double)cus * e) + 8.0;
      if ((double)count * t_one < t_group) return 0;
    }
  }
  return e160 >= e288 && e160 >= e128 ? 160 : e288 >= e128 ? 288 : 128;
}

// Whether a group call of that shape is ONE launch (the streaming kernel at decode sizes, a tiled kernel at prefill
// sizes) rather than a loop over the problems; a caller that holds a split-K workspace does better with separate
// calls in the second case.
int gemm_group_is_one_launch(long long M, long long N, long long K, int count) {
  if (M <= 16 && K % SBK == 0) return 1;
  if (M <= TI_ROWS_ABREAST_M && N % 4 == 0) {
    const RowsPick rows = rows_pick(M, N, K, num_cus(), count);
    if (rows.tiling != ROWS_NONE && rows.slices == 1) return 1;  // no workspace needed
  }
  if (M <= 16) return 0;
  if (kwaves_pick(M, N, K, false, count) != KWAVES_NONE) return 1;
  return group_prefill_tile(M, N, K, count) != 0 ? 1 : 0;
}

// q/k/v-style group of s8 linears.  One launch over all the weights: one row on the dot-product kernel, up to 64 rows (more where the outputs are narrow) on the
// weight-streaming kernel of gemm_rows.h where its tilings divide K, else up to 16 rows on the streaming kernel (K % 1024 == 0),
// and prefills whose tiles group_prefill_tile finds; anything else runs problem by problem.
int launch_gemm_group_s8(const GemmParams& shape, const GemmGroup& grp, hipStream_t stream, void* workspace,
                         long long workspace_bytes) {
  constexpr int KIND = EPI_S8_BIAS;
  if (shape.M == 0 || shape.N == 0 || grp.count == 0) return TI_OK;
  g_rows_last = {0, 0, 0};
  g_last_form = "";
  bool ptr_ok = (reinterpret_cast<uintptr_t>(shape.A) & 15) == 0;
  for (int i = 0; i < grp.count; ++i) ptr_ok = ptr_ok && (reinterpret_cast<uintptr_t>(grp.B[i]) & 15) == 0;
  const bool aligned = ptr_ok && (shape.K % SBK == 0) && shape.K > 0;
  const int spb = (shape.N + 15) / 16;
  const long long strips = (long long)spb * grp.count;
  if (ptr_ok && shape.M <= TI_ROWS_ABREAST_M && shape.N % 4 == 0 && !(gemv_takes(shape) && strips >= 256) &&
      !kwaves_before_rows(shape.M, shape.N, shape.K, grp.count)) {
    const int rc = launch_rows<KIND, true>(shape, grp, grp.count, workspace, workspace_bytes, stream);
    if (rc >= 0) {
      if (rc == TI_OK) g_last_kernel = shape.M <= 16 ? "stream_group" : "mid_stream_group";
      return rc;
    }
  }
  if (aligned && gemv_takes(shape) && strips >= 256) {
    g_last_kernel = "gemv_group";
    return launch_gemv<KIND, true>(shape, grp, grp.count, stream);
  }
  if (aligned && shape.M <= 16 && strips >= 256) {
    g_last_kernel = "stream_group";
    const int cus = num_cus();
    auto launch = [&](auto kern, int stages, int rows, int per_cu) -> int {
      const int lds = stages * rows * SBK + S_RED;
      static std::atomic<unsigned long long> lds_ok{0};
      if (int rc = allow_lds(kern, lds, lds_ok)) return rc;
      const long long slots = (long long)cus * per_cu;
      hipLaunchKernelGGL(kern, dim3((unsigned)(strips < slots ? strips : slots)), dim3(256), lds, stream, shape, spb,
                         (int)strips, grp);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return fail(TI_ERR_LAUNCH, "gemm launch: %s", hipGetErrorString(e));
      return TI_OK;
    };
    const bool deep = stream_deep_pipeline(shape.M, strips, cus);
    if (shape.M == 1)
      return deep ? launch(gemm_stream_kernel<KIND, 1, 3, true>, 3, 17, 2)
                  : launch(gemm_stream_kernel<KIND, 1, 2, true>, 2, 17, 3);
    if (shape.M <= 4) return launch(gemm_stream_kernel<KIND, 4, 2, true>, 2, 20, 3);
    return deep ? launch(gemm_stream_kernel<KIND, 16, 3, true>, 3, 32, 1)
                : launch(gemm_stream_kernel<KIND, 16, 2, true>, 2, 32, 2);
  }
  if (ptr_ok && shape.lda == shape.K && shape.ldb == shape.K) {
    const KWavesTile tile = kwaves_pick(shape.M, shape.N, shape.K, false, grp.count);
    if (tile != KWAVES_NONE) {
      g_last_kernel = "mid_waves_group";
      return launch_kwaves<KIND, true>(tile, shape, stream, grp);
    }
  }
  // Prefill shapes whose width the 256x160, 256x288, 256x256 or 256x128 tiles divide: the problems are the batches of one
  // persistent launch, so the pipeline fill and the epilogue of one projection overlap the next one's work.
  if (ptr_ok && shape.lda == shape.K && shape.ldb == shape.K) {
    const int tile = group_prefill_tile(shape.M, shape.N, shape.K, grp.count);
    if (tile != 0) {
      GemmParams q = shape;
      q.batch = grp.count;
      if (tile == 160) {
        g_last_kernel = "pipe16_256x160_group";
        return launch_pipe16q<Pipe16QCfg<256, 160, 4, 2, KIND, true>>(q, stream, grp);
      }
      if (tile == 288) {
        g_last_kernel = "pipe16_256x288_group";
        return launch_pipe16q<Pipe16QCfg<256, 288, 4, 2, KIND, true>>(q, stream, grp);
      }
      if (tile == 256) {
        g_last_kernel = "pipe16_256x256_group";
        return launch_pipe16q<Pipe16QCfg<256, 256, 4, 2, KIND, true>>(q, stream, grp);
      }
      g_last_kernel = "pipe16_256x128_group";
      return launch_pipe16q<Pipe16QCfg<256, 128, 4, 2, KIND, true>>(q, stream, grp);
    }
  }
  for (int i = 0; i < grp.count; ++i) {
    GemmParams q = shape;
    q.B = grp.B[i];
    q.bias = grp.bias[i];
    q.C = grp.C[i];
    q.alpha = grp.alpha[i];
    q.beta = grp.beta[i];
    if (int rc = launch_gemm_kind_3(q, workspace, workspace_bytes, stream)) return rc;
  }
  return TI_OK;
}

int launch_gemm(int kind, const GemmParams& p, void* ws, long long ws_bytes, hipStream_t stream) {
  if (p.M == 0 || p.N == 0 || p.batch == 0) return TI_OK;
  g_rows_last = {0, 0, 0};
  g_last_form = "";
  if (int rc = fused_split_check()) return rc;
  switch (kind) {
    case EPI_S32_BIAS: return launch_gemm_kind_0(p, ws, ws_bytes, stream);
    case EPI_S32_SCALED: return launch_gemm_kind_1(p, ws, ws_bytes, stream);
    case EPI_F32_BIAS: return launch_gemm_kind_2(p, ws, ws_bytes, stream);
    case EPI_S8_BIAS: return launch_gemm_kind_3(p, ws, ws_bytes, stream);
    case EPI_S8_RELU: return launch_gemm_kind_4(p, ws, ws_bytes, stream);
    case EPI_F32_SCALE: return launch_gemm_kind_5(p, ws, ws_bytes, stream);
    case EPI_S8_SCALE: return launch_gemm_kind_6(p, ws, ws_bytes, stream);
    case EPI_S32_RAW: return launch_gemm_kind_7(p, ws, ws_bytes, stream);
    case EPI_F32_BIAS_ACC: return launch_gemm_kind_8(p, ws, ws_bytes, stream);
    case EPI_F16_BIAS_ACC: return launch_gemm_kind_9(p, ws, ws_bytes, stream);
  }
  return fail(TI_ERR_INVALID_ARG, "unknown epilogue kind %d", kind);
}

}  // namespace ti
