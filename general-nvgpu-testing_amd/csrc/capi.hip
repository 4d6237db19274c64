// C ABI of libbeam_hip.so (declarations and reference citations: include/beam_hip.h).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include <unistd.h>

#include "../../include/beam_hip_debug.h"
#include "aux_kernels.h"
#include "kernel_set.h"
#include "tile_map.h"

using namespace beam;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(BEAM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

#define BEAM_HIP(call)                                  \
  do {                                                  \
    hipError_t e_ = (call);                             \
    if (e_ != hipSuccess) return hip_fail(e_, #call);   \
  } while (0)

struct Device {
  int status = -1;  // -1 = not probed
  char name[256] = "";
  int cus = 0;
  int clock_khz = 0;
  size_t mem = 0;
};
Device g_dev;
std::mutex g_dev_mu;
// A word of pinned host memory that a fused GEMM+LayerNorm launch sets when a workgroup in it gives up (made once, by
// beam_init; the process keeps it, and it stays set).  While it is zero no launch of the process has ever given up, and a
// checked call is done without copying the workspace header back: that blocking copy of 16 bytes cost more than a small
// call's kernel (64 x 64 x 64: 24 us of a checked call beyond its launch with the copy, 11 without, 7 as wait_for_stream waits).  After the first
// time-out every checked call reads its header.  (One word cannot tell more: launches of other streams and threads write
// it too, so comparing it before and after a launch could miss this launch's own time-out between two of another's.)
unsigned* g_ln_host_timeout = nullptr;

// Sets of words of pinned host memory, a word for each XCD in a 64-byte line of its own, through which a kernel at a stream's end
// tells a waiting thread that it has come there, and an event for each (wait_for_stream).  The words are allocated with the word
// above; a call holds a set while it waits, and without a free one waits as hipStreamSynchronize does.
constexpr int kWaitSets = 64;
unsigned* g_wait_words = nullptr;
struct WaitEvent {
  hipEvent_t event = nullptr;
  int device = -1;
} g_wait_events[kWaitSets];
std::atomic<unsigned long long> g_wait_free{~0ull};
std::atomic<unsigned> g_wait_value{0};

int take_wait_set() {
  unsigned long long free = g_wait_free.load(std::memory_order_relaxed);
  while (free != 0)
    if (g_wait_free.compare_exchange_weak(free, free & (free - 1), std::memory_order_acquire)) return __builtin_ctzll(free);
  return -1;
}
void give_wait_set(int i) { g_wait_free.fetch_or(1ull << i, std::memory_order_release); }

// Waits until everything that `st` holds has run and the host sees what it wrote; not for a stream that is being captured, and
// only on a device of kNumXcd XCDs.  hipStreamSynchronize puts a packet behind the last kernel that writes caches back for the
// host and raises a signal; a kernel of a wavefront on each XCD whose words this thread watches is 3 us shorter (a checked
// GEMM+LayerNorm of 512 x 1024 x 1024 18.4 -> 15.4 us, without the event).  The stream's kernels run one after another, and a wavefront's store is
// a release that writes back its XCD's L2: with all XCDs heard, nothing that the kernels in front wrote is left in an L2, be it
// for memory of the device or of the host.  (One wavefront on one XCD, 15.2 us, says so of that XCD's L2 only.  Eight words in
// one line, written and watched at once, 16.4 to 17.9.)  Long waits, and an XCD without a workgroup, are left to the runtime.
// The event behind that kernel, recorded while the stream works, is for the runtime: it would otherwise find kernels whose end it
// has not heard of, and put a packet of its own behind them when the caller synchronises or copies next.  us of the call and
// what follows, by hipStreamSynchronize, watched without the event, with it: the next such call 19.1, 15.7, 16.8; another
// product 22.6, 19.0, 21.1; hipDeviceSynchronize 22.3, 27.2, 21.2; a copy to the host and hipDeviceSynchronize 49.1, 52.9, 49.3.
void record_wait_event(WaitEvent* e, hipStream_t st) {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) return;
  if (e->device != device) {  // (an event belongs to a device)
    if (e->event) (void)hipEventDestroy(e->event);
    *e = WaitEvent();
    if (hipEventCreateWithFlags(&e->event, hipEventDisableTiming) != hipSuccess) {
      e->event = nullptr;
      (void)hipGetLastError();
      return;
    }
    e->device = device;
  }
  if (hipEventRecord(e->event, st) != hipSuccess) (void)hipGetLastError();
}

hipError_t wait_for_stream(hipStream_t st) {
  const int i = g_wait_words ? take_wait_set() : -1;
  if (i < 0) return hipStreamSynchronize(st);
  unsigned* const words = g_wait_words + i * kTellWords;
  const unsigned value = g_wait_value.fetch_add(1, std::memory_order_relaxed) + 1;
  int told = 0;  // XCDs
  if (launch_tell_host(words, value, st) == hipSuccess) {
    record_wait_event(&g_wait_events[i], st);
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    do {
      for (int spin = 0; spin < 32; ++spin) {
        while (told < kNumXcd && __atomic_load_n(words + told * kTellStride, __ATOMIC_ACQUIRE) == value) ++told;
        if (told == kNumXcd) {
          give_wait_set(i);
          return hipSuccess;
        }
        __builtin_ia32_pause();
      }
    } while (std::chrono::steady_clock::now() < until);
  }
  const hipError_t e = hipStreamSynchronize(st);
  if (e == hipSuccess) give_wait_set(i);  // its kernel has run; after an error it may not have, and the set stays taken
  return e;
}
// Polls before a waiting thread gives up: of statistics slots in the fused LayerNorm (3-4 us each once the pauses
// between tries have grown: about 60 ms), of a tile's flags in the one-launch split-K (about 1 us each).  What a
// workgroup legitimately waits for is resident with it and at most a tile's K loop behind, so the bound is there
// for a device that other work keeps occupied: giving up then costs milliseconds, and the caller's retry as two
// passes (beam_gemmrc_ln_checked) gives the result.
std::atomic<int> g_ln_spin_limit{16384};
// Nonces of fused GEMM+LayerNorm and one-launch split-K launches: consecutive numbers from a start that differs from process to process
// (memory recycled from another process of this library then holds tags of another sequence).
std::atomic<unsigned> g_ln_nonce{(unsigned)std::chrono::steady_clock::now().time_since_epoch().count() * 2654435761u ^
                                 (unsigned)getpid() * 40503u};

// Split-K workspace of beam_gemmrc_splitk_noalloc: device memory that exists from the moment the library's
// code is loaded on a GPU until the process ends, so the entry point never allocates.  In host code the
// array's name is only a handle for hipGetSymbolAddress; what kernels and copies get is the per-device
// address looked up below (every GPU has its own copy at its own address).
constexpr size_t kScratchPartialBytes = (size_t)16 << 20;                      // the partial sums a call may need
constexpr size_t kScratchBytes = kScratchPartialBytes + ((size_t)256 << 10);  // ... + synchronisation words of the one-launch form
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

// Address of `scratch` on the current device (looked up once per device, with that device current).
int scratch_on_current_device(void** out) {
  int dev = -1;
  BEAM_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(BEAM_ERR_UNSUPPORTED, "device index %d beyond %d", dev, kMaxDevices - 1);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    BEAM_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(BEAM_ERR_HIP, "hipGetSymbolAddress returned a null address for the scratch array");
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return BEAM_OK;
}

const std::vector<KernelSet>& kernel_sets() {
  static const std::vector<KernelSet> sets = [] {
    std::vector<KernelSet> v;
#define BEAM_PUSH(BM, BN, TM, TN) v.push_back(kernel_set_##BM##x##BN##_##TM##x##TN());
    BEAM_FOR_EACH_SET(BEAM_PUSH)
#undef BEAM_PUSH
    return v;
  }();
  return sets;
}

const KernelSet* find_set(const beam_tile_cfg& c) {
  for (const KernelSet& k : kernel_sets())
    if (k.block_m == c.block_m && k.block_n == c.block_n && k.wave_m == c.wave_m && k.wave_n == c.wave_n)
      return &k;
  return nullptr;
}

// Raster group height (tile rows that share one sweep over the columns): measured best is 4 for the
// tiles that run one workgroup per CU (8192^3: +1.7% over 8; 16384 x 16384 x 2048: +28%) and 8 for the
// smaller ones, which run two or more per CU.
constexpr int default_group_m(int block_m, int block_n) { return block_m * block_n >= 256 * 128 ? 4 : 8; }
// Largest K: the buffer descriptor of a 256-row operand tile, (255 * K + K) * 2 bytes, must stay below the
// out-of-range offset the kernels use for masked chunks (kOobOffset).
constexpr int kMaxK = (int)((kOobOffset / 512u) & ~7u) - 8;
static_assert((unsigned long long)kMaxK * 512ull < kOobOffset && kMaxK % 8 == 0, "descriptor range");

// Elements of a side-job array: its byte size must stay below the out-of-range offset the kernels use.
constexpr long long kMaxSideElems = (long long)(kOobOffset / 16) * 8;

// Validates a gemmrc problem.  *generic is set when it is well formed but outside what the tiled kernels take (K
// shorter than one 16-byte chunk, or beyond the descriptor range): such problems run on the plain kernel of
// aux_kernels.hip.
int check_problem(const void* A, const void* B, const void* C, int M, int N, int K, int dtype, bool* generic) {
  *generic = false;
  if (M < 0 || N < 0 || K < 0) return fail(BEAM_ERR_INVALID, "negative dimension (M=%d N=%d K=%d)", M, N, K);
  if (dtype != BEAM_F16 && dtype != BEAM_BF16) return fail(BEAM_ERR_UNSUPPORTED, "dtype %d: only fp16 (0) and bf16 (1)", dtype);
  if (M == 0 || N == 0) return BEAM_OK;
  if (!C) return fail(BEAM_ERR_INVALID, "null output pointer");
  if (K > 0 && (!A || !B)) return fail(BEAM_ERR_INVALID, "null input pointer");
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 1) return fail(BEAM_ERR_INVALID, "A, B and C must be aligned to their 16-bit elements");
  if ((size_t)M * (size_t)N >= ((size_t)1 << 40)) return fail(BEAM_ERR_UNSUPPORTED, "M*N too large");
  if ((M + 63) / 64 > 65535) return fail(BEAM_ERR_UNSUPPORTED, "M=%d too large", M);
  *generic = K > kMaxK || (K > 0 && K < 8);
  return BEAM_OK;
}

// Rows of A or B that do not start on 16 bytes, or C not on 8: what the kernels take at a lower rate (gemm_kernel.h:
// load_short_tile), and what may call split-K without a workspace.  No tile that a caller names is refused on them: where
// the library has no kernel for it, the plain one computes the problem.
bool rows_unaligned(const void* A, const void* B, const void* C, int K) {
  return K % 8 != 0 || (((uintptr_t)A | (uintptr_t)B) & 15) != 0 || ((uintptr_t)C & 7) != 0;
}

// Slices for `tiles` output tiles when the caller leaves the choice to the library: as many as make
// one full round of workgroups (tiles * slices = CUs), at least 4 K tiles each.  Measured at
// 256 x 256 x 32768: 16 tiles x 16 slices 15.1 us, x 24 (one and a half rounds, what the reference's
// rule gives: beam_slice_heuristic) 19.8 us, x 32 17.6 us; 8 tiles x 32 slices 14.2 us, x 16 17.0 us.
int auto_slices(long tiles, int K, int cus) {
  if (tiles * 2 > cus) return 1;
  const int ktiles = (K + kBK - 1) / kBK;
  long s = cus / (tiles < 1 ? 1 : tiles);
  if (s > ktiles / 4) s = ktiles / 4;
  if (s > 64) s = 64;  // the reduction reads every slice: 64 x 64 x 32768 takes 9.1 us with 64 slices, 11.4 with 128
  // Half a round of workgroups with 16 K tiles each beats a full round of shorter slices (every slice pays its
  // pipeline fill and adds M x N partial sums): 128 x 128 x 32768 takes 8.5 us in 32 slices, 9.6 in 64;
  // 128 x 256 x 8192 7.8 us in 16, 7.9 in 32.
  const long half_round = (cus / 2 + tiles - 1) / (tiles < 1 ? 1 : tiles);
  const long want = ktiles / 16 > half_round ? ktiles / 16 : half_round;
  if (s > want) s = want;
  return s < 1 ? 1 : (int)s;
}

// *raised (may be null): the tile's own depth is pipeline 0, and only the two K groups made it the deep pipeline.
int choose_default(int M, int N, int K, int split_req, beam_tile_cfg* cfg, int* split_k, bool* raised = nullptr);

// split_req: -1 the caller cannot run K slices (no workspace); 0 it can, and leaves the number to
// the library; > 0 it asks for that many.  The default tile is chosen for that situation.
// w4_ok: the caller has a form of the 4-wavefront kernel (gemm_w4.h); for the others the library's own choice
// of that tile means the 8-wavefront 256 x 256 tile.
int resolve_cfg(const beam_tile_cfg* in, int M, int N, int K, beam_tile_cfg* out, const KernelSet** ks,
                int split_req = -1, bool w4_ok = false) {
  if (in) {
    *out = *in;
  } else {
    int s;
    int rc = choose_default(M, N, K, split_req, out, &s);
    if (rc) return rc;
    if (!w4_ok && out->block_m == 256 && out->block_n == 256 && out->wave_m == 128 && out->wave_n == 128) out->wave_n = 64;
  }
  if (out->pipeline < 0 || out->pipeline > 2) return fail(BEAM_ERR_UNSUPPORTED, "pipeline %d: 0 (3 A + 2 B LDS slots), 1 (2 + 2) or 2 (deep)", out->pipeline);
  if (out->group_m <= 0) out->group_m = default_group_m(out->block_m, out->block_n);
  *ks = find_set(*out);
  if (!*ks)
    return fail(BEAM_ERR_UNSUPPORTED, "no kernel for workgroup tile %dx%d / wavefront tile %dx%d", out->block_m,
                out->block_n, out->wave_m, out->wave_n);
  return BEAM_OK;
}

GemmParams base_params(const void* A, const void* B, int M, int N, int K, const beam_tile_cfg& c) {
  GemmParams p;
  std::memset(&p, 0, sizeof p);
  p.A = A;
  p.B = B;
  p.M = M;
  p.N = N;
  p.K = K;
  p.tiles_m = (M + c.block_m - 1) / c.block_m;
  p.tiles_n = (N + c.block_n - 1) / c.block_n;
  p.k_slice = ((K + kBK - 1) / kBK) * kBK;
  if (p.k_slice == 0) p.k_slice = kBK;
  p.splits = 1;
  p.group_m = c.group_m;
  p.divs = make_tile_divs(p.tiles_m, p.tiles_n, p.group_m);
  return p;
}

// How a tiled kernel's 16-bit output leaves (StoreKind).  Rows on 64-byte sectors: through the L2.  Rows off them are written
// in parts of a sector by two wavefronts or workgroups: left in the L2, which puts the parts together, where that saves more
// than the write-back at the kernel's end costs.  (us, through -> cached; C in the last-level cache, then from memory.)
//   * The kernel of gemm_w4.h, 64 contiguous bytes of a row per store: always (2048 x 1992 x 4032 68 -> 67, 77 -> 74; 4096 x
//     4040 x 256 19 -> 15.5, 27 -> 18, x 1024 34 -> 31, 41 -> 33).
//   * Tiles of 64 columns: always (2048 x 1992 x 256 in 64 x 64 tiles, two K groups 14.2 -> 13.7, 14.3 -> 13.8, x 1985 14.6 ->
//     13.5; 512 x 968 x 256 4.0 -> 3.9, 4.1 -> 4.0).
//   * The others from 20 MB on (3072 x 4040 x 256 in 128 x 128 tiles 14.0 -> 12.9, 20 -> 15, in 192 x 256 13.1, 13.3, 18 -> 14;
//     4096 x 8136 x 1024 in 256 x 256 tiles 70 -> 63, 79 -> 68; 8192 x 8136 x 256 in 128 x 128 106 -> 71).  Below: 2048 x 1992 x
//     1024 in 128 x 128 tiles 11.6, cached 12.0.
//   * 256 x 256 tiles of eight wavefronts over several rounds under a short sum, one workgroup per tile, wherever rows start
//     (8192 x 8192 x 256 106 -> 65, 119 -> 62; 4096 x 8192 x 1024 58.8, 59.9; 64 -> 62; 7079 x 4544 x 1840 [K][N] 96.7, 98.5),
//     but not beside a side job (8192 x 4096 x 256 with 2^25 elements 51.9, 53.3).
//   * Rows on 32 bytes: of these only gemm_w4.h's (4096 x 4048 x 1024 33.7 -> 29.9) and the wide tiles of a plain product (5000 x
//     5008 x 1000 54.5 -> 53.8); 64 columns 1024 x 2000 x 256 4.46, cached 4.53, LayerNorm 4385 x 5232 x 392 41.9, 44.3.
// (Non-temporal stores are faster still by themselves, 8192 x 8192 x 1024 in 128 x 128 tiles 161 -> 126 us, but only put the
// cost off: with a kernel that reads the output behind it, 4096 x 4096 x 1024 takes 54.3 us written through, 56.2 so.)
int store_kind(const beam_tile_cfg& c, int wavefronts, bool w4, const void* C, int M, int N, int K, bool fused = false) {
  const size_t bytes = (size_t)M * N * 2;
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  if (!w4 && !fused && wavefronts == 8 && K < 1024 && c.block_m * c.block_n == 256 * 256 &&
      (long)((M + 255) / 256) * ((N + 255) / 256) > cus) return kStoreCached;
  if (N % 32 == 0 && ((uintptr_t)C & 63) == 0) return kStoreThrough;
  if (w4) return kStoreCached;
  if (N % 16 == 0 && ((uintptr_t)C & 31) == 0 && (fused || c.block_n == 64)) return kStoreThrough;
  return c.block_n == 64 || bytes >= ((size_t)20 << 20) ? kStoreCached : kStoreThrough;
}

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// ---- host data generation -------------------------------------------------------------

inline uint64_t mix64(uint64_t x) {  // splitmix64 finaliser
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

inline uint64_t draw(uint64_t seed, uint64_t tensor_id, uint64_t i) {
  return mix64(mix64(seed + 0x632BE59BD9B4E019ull * (tensor_id + 1)) + i);
}

inline uint32_t f32_bits(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  return u;
}

inline uint16_t to_bf16_bits(float f) {
  uint32_t x = f32_bits(f);
  if ((x & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x >> 16) | 0x40u);
  return (uint16_t)((x + 0x7fffu + ((x >> 16) & 1u)) >> 16);
}

inline uint16_t to_f16_bits(float f) {
  // Round the significand to 11 bits in float arithmetic, then repack.
  const uint32_t x = f32_bits(f);
  const uint16_t sign = (uint16_t)((x >> 16) & 0x8000u);
  const uint32_t ax = x & 0x7fffffffu;
  if (ax > 0x7f800000u) return (uint16_t)(sign | 0x7e00u);
  if (ax >= 0x477ff000u) return (uint16_t)(sign | 0x7c00u);
  float a;
  std::memcpy(&a, &ax, 4);
  if (ax < 0x38800000u) {
    // subnormal half: a / 2^-24 rounded to nearest even integer
    const float scaled = a * 16777216.0f;
    const float r = std::nearbyintf(scaled);  // default rounding mode = to nearest even
    return (uint16_t)(sign | (uint16_t)r);
  }
  uint32_t r = ax + 0xfffu + ((ax >> 13) & 1u);  // RN-even at bit 13
  return (uint16_t)(sign | ((r - 0x38000000u) >> 13));
}

template <typename F>
void parallel_for(size_t n, F f) {
  unsigned hw = std::thread::hardware_concurrency();
  unsigned nt = hw == 0 ? 4 : (hw > 16 ? 16 : hw);
  if (n < (1u << 16)) nt = 1;
  std::vector<std::thread> th;
  const size_t chunk = (n + nt - 1) / nt;
  for (unsigned t = 0; t < nt; ++t) {
    const size_t lo = t * chunk, hi = lo + chunk < n ? lo + chunk : n;
    if (lo >= hi) break;
    th.emplace_back([=] { f(lo, hi); });
  }
  for (auto& t : th) t.join();
}

}  // namespace

extern "C" {

const char* beam_last_error(void) { return g_err; }

int beam_init(void) {
  std::lock_guard<std::mutex> lk(g_dev_mu);
  if (g_dev.status >= 0) return g_dev.status == BEAM_OK ? BEAM_OK : fail(g_dev.status, "device probe failed earlier");
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0) {
    g_dev.status = BEAM_ERR_HIP;
    return fail(BEAM_ERR_HIP, "no HIP device (%s)", e == hipSuccess ? "count is zero" : hipGetErrorString(e));
  }
  hipDeviceProp_t prop;
  e = hipGetDeviceProperties(&prop, 0);
  if (e != hipSuccess) {
    g_dev.status = BEAM_ERR_HIP;
    return hip_fail(e, "hipGetDeviceProperties");
  }
  std::snprintf(g_dev.name, sizeof g_dev.name, "%s (%s)", prop.name, prop.gcnArchName);
  g_dev.cus = prop.multiProcessorCount;
  g_dev.clock_khz = prop.clockRate;
  g_dev.mem = prop.totalGlobalMem;
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    g_dev.status = BEAM_ERR_DEVICE;
    return fail(BEAM_ERR_DEVICE, "device 0 is %s; this library holds gfx950 code only", prop.gcnArchName);
  }
  g_dev.status = BEAM_OK;
  constexpr size_t kHostWordBytes = sizeof(unsigned) * (kTellStride + kWaitSets * kTellWords);
  void* word = nullptr;
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // the first call may come while a stream is being captured
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  if (hipHostMalloc(&word, kHostWordBytes, hipHostMallocPortable | hipHostMallocMapped) == hipSuccess) {
    std::memset(word, 0, kHostWordBytes);
    g_ln_host_timeout = (unsigned*)word;
    g_wait_words = (unsigned*)word + kTellStride;
  } else {
    (void)hipGetLastError();  // without it every checked call reads the header
  }
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  void* ignored;
  return scratch_on_current_device(&ignored);  // the no-allocation entry point's memory, looked up at set-up
}

int beam_device_info(char* name, int len, int* compute_units, int* clock_khz, size_t* mem_bytes) {
  int rc = beam_init();
  if (rc != BEAM_OK && rc != BEAM_ERR_DEVICE) return rc;
  if (name && len > 0) std::snprintf(name, (size_t)len, "%s", g_dev.name);
  if (compute_units) *compute_units = g_dev.cus;
  if (clock_khz) *clock_khz = g_dev.clock_khz;
  if (mem_bytes) *mem_bytes = g_dev.mem;
  return rc;
}

int beam_num_configs(void) { return (int)kernel_sets().size(); }

int beam_get_config(int index, beam_tile_cfg* out) {
  if (!out || index < 0 || index >= beam_num_configs()) return fail(BEAM_ERR_INVALID, "config index %d out of range", index);
  const KernelSet& k = kernel_sets()[index];
  out->block_m = k.block_m;
  out->block_n = k.block_n;
  out->wave_m = k.wave_m;
  out->wave_n = k.wave_n;
  out->pipeline = 0;
  out->group_m = default_group_m(out->block_m, out->block_n);
  return BEAM_OK;
}

int beam_slice_heuristic(int tiles, int compute_units) {
  if (tiles < 1) tiles = 1;
  const float units = (float)compute_units;
  int s = 1;
  if ((float)tiles < units) {
    s = (int)((units - 1.0f) / (float)tiles + 1.0f);
    float waves = (float)s * (float)tiles / units;
    float rem = waves - (float)(int)waves;
    while (rem < 0.5f) {
      ++s;
      waves = (float)s * (float)tiles / units;
      rem = waves - (float)(int)waves;
    }
  }
  return s;
}

int beam_default_config(int M, int N, int K, beam_tile_cfg* cfg, int* split_k) {
  return choose_default(M, N, K, split_k ? 0 : -1, cfg, split_k);
}

}  // extern "C"

namespace {

int choose_default(int M, int N, int K, int split_req, beam_tile_cfg* cfg, int* split_k, bool* raised) {
  if (!cfg) return fail(BEAM_ERR_INVALID, "null cfg");
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  // A small cost model picks the tile: every CU works through ceil(tiles / CUs) workgroups, `occ` of
  // them at a time (what LDS allows); a workgroup costs a fixed start-up / epilogue time plus its flops
  // at the per-CU rate of its tile shape, which is higher when several workgroups share the CU.  The
  // rates (TFLOP/s per CU, alone / with a full CU) and fixed costs (us) are fits to timings of all
  // compiled tiles on 39 shapes from 512^3 to 8192^3 (square, skinny and short-K) on an MI355X, taken
  // while the deep tiles up to 128 x 64 had one K group: they rank tiles, they are not those tiles' rates now.
  // On timings of the present kernels (beam/default_tile_timings.json), what runs for the pick is within
  // 0.8% of the best tile on average, 6.1% at worst (tile-count thresholds: 6% and 76%).  The 224- and 192-row tiles are there for what 256 rows divide badly: 3072^3 is
  // 0.75 of a round of 192 x 256 tiles against 0.56 of a round of 256 x 256 ones (49.5 against
  // 58.6 us), 7168^3 is 3.5 rounds of 224 x 256 tiles against 3.06 (546 against 613 us).
  struct Candidate {
    beam_tile_cfg cfg;
    int occ;
    double alone, full, fixed;
  };
  static const Candidate kCandidates[] = {
      {{256, 256, 128, 64, 0, default_group_m(256, 256)}, 1, 6.04, 6.04, 8.0},
      {{224, 256, 112, 64, 0, default_group_m(224, 256)}, 1, 5.95, 5.95, 8.0},
      {{192, 256, 96, 64, 0, default_group_m(192, 256)}, 1, 5.22, 5.22, 8.0},
      {{256, 128, 64, 64, 0, default_group_m(256, 128)}, 1, 4.99, 4.99, 6.0},
      {{128, 256, 64, 64, 0, default_group_m(128, 256)}, 1, 4.8, 4.8, 6.0},
      {{128, 128, 64, 64, 0, default_group_m(128, 128)}, 2, 3.8, 4.4, 3.42},
      {{128, 128, 64, 32, 2, default_group_m(128, 128)}, 1, 4.05, 4.05, 4.0},
      {{128, 64, 64, 32, 0, default_group_m(128, 64)}, 2, 2.6, 3.4, 3.5},
      {{128, 64, 64, 32, 2, default_group_m(128, 64)}, 1, 3.2, 3.2, 4.2},
      {{64, 64, 32, 32, 0, default_group_m(64, 64)}, 4, 1.87, 2.9, 2.7},
      {{64, 64, 32, 32, 2, default_group_m(64, 64)}, 1, 2.4, 2.4, 4.0},
      {{64, 128, 32, 64, 0, default_group_m(64, 128)}, 2, 3.15, 3.4, 3.5},
      {{64, 128, 32, 64, 2, default_group_m(64, 128)}, 1, 3.3, 3.3, 4.0},
  };
  // With a workspace at hand the deep-pipeline candidates are priced with their K slices: the
  // slices' workgroups fill the CUs, and the reduction costs a launch plus reading the partial sums.
  beam_tile_cfg c = kCandidates[0].cfg;
  int c_split = 1;
  double best_us = 1e300;
  for (const Candidate& k : kCandidates) {
    const long t = tiles(k.cfg.block_m, k.cfg.block_n);
    int s = 1;
    if (k.cfg.pipeline == 2 && split_req >= 0) {
      const int ktiles = (K + kBK - 1) / kBK;
      s = split_req == 0 ? auto_slices(t, K, cus) : (split_req < ktiles ? split_req : (ktiles > 0 ? ktiles : 1));
    }
    const long load = (t * s + cus - 1) / cus;  // workgroups per CU
    const long conc = load < k.occ ? load : k.occ;
    const double rate = k.occ == 1 ? k.alone : k.alone + (k.full - k.alone) * (double)(conc - 1) / (k.occ - 1);
    const double mflop = 2.0e-6 * k.cfg.block_m * k.cfg.block_n * (double)K / s;
    double us = (double)((load + k.occ - 1) / k.occ) * k.fixed + (double)load * mflop / rate;
    // the partial sums are written through to memory and read back (about 4 TB/s each way), and the reducing
    // workgroups start behind the multiplying ones
    if (s > 1) us += 2.0 + (double)s * M * N * 4.0 / 2.0e6;
    if (us < best_us) {
      best_us = us;
      c = k.cfg;
      c_split = s;
    }
  }
  *cfg = c;
  // From one full round of workgroups on, the 256 x 256 tile runs as four wavefronts of 128 x 128 (the kernel of
  // gemm_w4.h; 8192^3 fp16, same machine, in turn: 1490-1515 against 1455-1465 TFLOP/s) where that kernel's
  // shape conditions hold.
  if (c_split == 1 && c.block_m == 256 && c.block_n == 256 && tiles(256, 256) >= cus && K % kBK == 0 && K >= kW4MinK && N % 8 == 0 &&
      N <= (1 << 21)) {
    cfg->wave_m = 128;
    cfg->wave_n = 128;
  }
  // One workgroup per CU under a long sum: the deep pipeline.  Less than half the CUs busy: its long prefetch queue keeps
  // memory busy.  Tiles with two K groups: up to a full round, since a lone group's K tile is a serial chain; 64 x 128 and
  // 128 x 64 from K = 768 on (one group, two: 2048 x 1024 x 520 6.2, 6.3; x 768 8.3, 7.2; x 1024 10.0, 8.2; x 1536 13.9, 11.0;
  // 620 x 3064 x 776 9.9, 9.3; x 1600 14.6, 11.1; [K][N] 700 x 2500 x 512 7.9, 7.3; x 1024 12.5, 10.0), 64 x 64 from K = 384 on.
  // These lines are for operands that come from the last-level cache or memory, as weights that change from call to call do.
  // With the same ones in every call, which then lie in the L2s, two groups are up to 0.8 us behind (their start, and the sums'
  // way through LDS).  One group, two; 96 sets of operands in turn, 12 sets, the same ones: 1024 x 1024 x 256 4.0, 4.2; 3.8, 4.0;
  // 2.9, 3.7; x 384 5.8, 5.2; 4.6, 4.5; 3.3, 4.0; x 512 7.1, 5.7; 5.2, 4.8; 3.6, 4.2; x 1024 11.7, 7.7; 8.3, 6.2; 5.0, 5.3; x 1536
  // 16.3, 10.2; 11.2, 7.9; 6.5, 6.6; x 2048 20.8, 11.5; 14.0, 8.7; 7.9, 7.5; 2048 x 1024 x 768 11.0, 9.0; 8.2, 7.1; 5.6, 6.4; x 1024
  // 13.6, 10.1; 9.8, 7.8; 6.6, 7.3; [K][N] 1024 x 1024 x 384 6.5, 5.5; 5.1, 4.8; 4.0, 4.5.  Only from K = 2048 on: a single row of
  // those, whose form as one group is made for long sums, and at most half a round, where smaller tiles run (kw_plan).
  const long picked = tiles(c.block_m, c.block_n);
  const bool few = K >= 2048 && picked < cus / 2;
  const int area = c.block_m * c.block_n;
  const bool groups = picked <= cus && (K >= 2048 ? area <= 128 * 64 : area == 128 * 64 ? K >= 768 : area == 64 * 64 && K >= 384 && M > 64 && 2 * picked > cus);
  if (raised) *raised = false;
  if (split_req < 0 && (few || groups)) {
    if (raised) *raised = !few && c.pipeline == 0;
    cfg->pipeline = 2;
  }
  // K slices on at most half the CUs: every workgroup has the memory system of two CUs to itself, the long
  // queue's prologue costs more than it hides (64 x 128 x 65536 in 64 slices: 8.9 against 9.9 us), and the
  // reducing workgroups of the one-launch form start on the idle CUs at once.
  if (c_split > 1 && tiles(c.block_m, c.block_n) * c_split <= cus / 2) cfg->pipeline = 0;
  if (split_k) *split_k = c_split;
  return BEAM_OK;
}

// The deep pipeline of the library's own tile as one K group (KernelSet::launch_deep_one_group), or nullptr for two.  Where
// one row of 64 x 64 tiles nearly fills the chip, B is read once and memory is the bound; one ring of 8 + 7 slots then keeps
// more of it in flight than two of 5 + 4.  fp16, us, two groups -> one: [N][K] from 3/4 of a round on, 33 x 12288 x 2048
// 10.5 -> 10.1, 16 x 14336 x 8192 35.4 -> 33.9, 64 x 12288 x 16384 94.5 -> 89.6; below it 17 x 11008 x 8192 27.5, 28.4, and
// with rows off 128-byte lines, which fill LDS at half the rate, 64 x 12288 x 4104 36.9, 37.7.  [K][N] from 7/8 on:
// 16 x 16384 x 8192 45.9 -> 42.6, x 12288 81.5 -> 72.7.
GemmLauncher deep_one_group(const KernelSet& ks, const beam_tile_cfg& c, int M, int N, int K, int dtype, bool b_kmajor, int cus) {
  if (c.pipeline != 2 || M > c.block_m) return nullptr;
  const long tiles = (N + c.block_n - 1) / c.block_n;
  if (!b_kmajor && K % kBK != 0) return nullptr;
  return 8 * tiles >= (b_kmajor ? 7L : 6L) * cus ? ks.launch_deep_one_group[dtype][b_kmajor ? 1 : 0] : nullptr;
}

// The tile of gemm_kwave.h for a problem, if any.  A CU's time there is what it fills LDS with, (rows + columns) x K of its
// tile: so the tile with the smallest sum of which the problem has at most one for every CU.  (466 x 864 x 520: 32 x 64, 210
// tiles, 4.6 us; 32 x 32, 405 tiles, 5.0; 300 x 400 x 513: 32 x 16, 250 tiles, 3.7, 16 x 16, 475 tiles, 4.0, 32 x 32 4.3.
// Beyond one tile of 64 x 64 for every CU the tiled kernels are ahead: 2048 x 1024 x 2040 18.8, here 20.0.)
//   b_kmajor, ln: the form; gemm: for beam_gemmrc's or beam_matmul_nn's result, not for a split-K call; rows: where every row of A (and of B as [N][K]) starts.
enum RowStarts { kAnywhere, kOnChunks, kOnLines };  // at an element, on 16 bytes, on 128
//   side: with a SiLU job beside it.
KwPlan kw_plan(int M, int N, int K, bool b_kmajor, bool ln, bool gemm, RowStarts rows, int cus, bool side = false) {
  static const struct { int rows, cols; } kTiles[] = {{8, 16},  {16, 16}, {16, 32}, {32, 16}, {32, 32},
                                                      {8, 64},  {16, 64}, {32, 64}, {64, 32}, {64, 64}};
  const KwPlan none = {0, 0, 0, false};
  if (K < 8 || K > kMaxK) return none;
  // Longer sums of more than a handful of rows are what beam_gemmrc_splitk is for (256 x 256 x 32768: 12.2 us there, 22.0
  // here); the line is where the two are about even (256 x 256 x 8192: 8.7, here 7.1; 128 x 128 x 16384: 8.3, here 12.0).  For
  // beam_gemmrc, which has no slices, it is not a line of speed: such a sum stays on the tiled kernel at 20.2 us (256 x 256 x
  // 8192; x 8184 7.4 here) and 78.7 (x 32768), so that the two calls remain the two methods that a tuner compares.
  if (M > 64 && K >= 8192 && !b_kmajor && !ln) return none;
  // A handful of rows beside more columns than 32 for every CU: B's way from memory is the bound, and the tiled kernels' long
  // rings are ahead but for K from 512 to 4096 (16 x 11008 x 4096 19.7 us, tiled 21.2; 1 x 14704 x 9064 47.7 tiled, here 50.6;
  // 10000 x 6000 21.4, 23.0) and up to 3 * 2^24 elements of B (16384 x 4088 20.6, here 27.2; 65536 x 512 11.0, 12.1).
  if (M <= 16 && N > 32 * cus && !b_kmajor && !ln && (K < 512 || K > 4096 || (long)N * K > (3L << 24))) return none;
  for (const auto& t : kTiles) {
    if (t.rows == 8 && (M > 8 || b_kmajor || ln)) continue;
    const long tiles_n = ((long)N + t.cols - 1) / t.cols, tiles = ((long)M + t.rows - 1) / t.rows * tiles_n;
    if (tiles > cus || (ln && tiles_n > 64)) continue;
    KwPlan plan = {t.rows, t.cols, 4, false};
    // The smallest tiles have little in flight for a wavefront: eight of them from K = 2048 on (256 x 256 x 4088 6.3 -> 5.8 us;
    // x 1032 3.4, with eight 3.7).
    if (t.rows <= 16 && t.cols == 16 && K >= 2048 && !ln) plan.waves = 8;
    // Whole lines where the fills saved are more than the one that every wavefront adds: K tiles x (rows + columns) of 1200
    // (1024 x 1024 x 520, 9 x 128: 6.2 us, shifted 6.8; 466 x 864 x 1032, 17 x 96: 6.6, shifted 6.1; 256 x 256 x 2056,
    // 33 x 32: 4.4, shifted 4.5).  8 rows are bound by latency: 1 x 1024 x 9480 6.4, shifted 7.2; a row
    // of tiles of 64 columns by memory: 16 x 11944 x 1064 6.7, 7.0.  Rows off 16 bytes have chunks
    // in two lines however they are fetched: 600 x 600 x 3004 12.6 either way, x 3001 14.3, shifted 15.9.
    plan.shift = rows == kOnChunks && t.rows > 8 && !(M <= 16 && t.cols == 64) && (long)(K / kBK) * (t.rows + t.cols) >= 1200;
    // A full tile per CU with rows on lines: from K = 2048 on the deep pipeline's two K groups, whose sums cost less to bring
    // together (1024 x 1024 x 2048 8.8 us, here 9.4; 128 x 8192 x 4096 15.5, 16.6); and where one row of tiles streams B from
    // memory (64 x 16384 x 1024 8.9, here 9.6).
    if (t.rows * t.cols == 64 * 64 && rows == kOnLines && !ln && (K >= 2048 || M <= 64)) return none;
    // ... and under a short sum, wherever rows start, if C's rows are whole chunks: the sums' way through LDS is the larger part
    // (1024 columns, 12 sets of operands in turn, here -> tiled: 1024 x 256 4.7 -> 3.7, x 384 5.3 -> 4.5, x 512 5.6 -> 4.8, x 1024
    // 6.8 -> 6.1, x 1001 9.5 -> 8.5, x 1032 8.4 -> 7.9, x 1288 9.1 -> 9.0, x 1544 9.6, 9.8; rows on lines x 1536 8.2 -> 7.9, x 1792
    // 8.6 -> 8.2; [K][N] x 256 5.0 -> 4.2, x 512 5.8 -> 5.3, x 1024 7.0 -> 6.9, x 1536 8.3, 8.7; 1000 x 1003 x 1024 6.8, 7.7).
    if (t.rows * t.cols == 64 * 64 && gemm && N % 8 == 0 && M > 64 && K <= (rows != kOnLines ? 1280 : b_kmajor ? 1024 : 2047)) return none;
    // ... nor where rows are off lines but on chunks and fills would take whole lines here: so they do in the tiled kernel
    // (kFormLines; 1100 x 544 x 1352 8.9 -> 7.3, 1402 x 664 x 2216 11.9 -> 10.4, 447 x 1912 x 7504 27.8 -> 24.9; [K][N] 3393 x
    // 184 x 2168 13.0 -> 12.0, 147 x 3952 x 2824 14.6 -> 13.4).  Rows of C that are not whole chunks stay.
    if (t.rows * t.cols == 64 * 64 && plan.shift && gemm && !side && N % 8 == 0) return none;
    // ... or one row of 32 x 64 tiles streams B from nearly every CU (20 x 14000 x 1500 10.7, here 11.4; 32 x 11008 x 4096 18.8,
    // 18.1; 30 x 9000 x 3000 13.6, 12.1).
    if (t.rows == 32 && t.cols == 64 && M <= 32 && !b_kmajor && !ln && 4 * tiles > 3L * cus) return none;
    // LayerNorm on full tiles under a short sum: the sums' way through LDS is the larger part (1024 x 1024 x 520 9.1 us, here
    // 9.9; x 1000 12.7, 12.2; x 1528 15.8, 13.7).
    if (t.rows * t.cols == 64 * 64 && ln && K < 600) return none;
    return plan;
  }
  return none;
}

// What beam_gemmrc without a tile runs on where rows are off 128-byte lines but on 16-byte chunks and gemm_kwave.h is not it:
// one of the tiles whose fills take whole lines (gemm_kernel.h: Form), or one of the others, which fill at half the rate
// there (only rows of whole lines that start behind one stay as choose_default has them).  The cost model of choose_default with constants of its own, since the straight tiles' rates are lower on such rows:
// TFLOP/s per CU alone and with `occ` workgroups on the CU, us per round of workgroups and per launch, least squares on the logarithm over 280 shapes with M, N from 64
// to 8192 and K from 64 to 8192 off lines (beam/line_tile_fit.py, with the timings).  On the 241 of them that come here its pick is
// 0.9% behind the best of these on average, 16% at worst; what ran before took 14% more than the pick.  us, before -> now: 928 x 1232 x 7112 49.7 -> 27.9, 633 x
// 6536 x 2952 38.5 -> 26.3, 1228 x 1784 x 6296 59.4 -> 36.9, 7702 x 7248 x 2472 268 -> 255, 2247 x 3736 x 216 12.7 -> 10.3.
struct LineChoice {
  beam_tile_cfg cfg;
  bool lines;        // cfg is a tile of launch_gemm_lines
  double ahead = 0;  // us of what choose_default names beyond cfg's, by the model; off_lines_tile
};
LineChoice off_lines_tile(int M, int N, int K, int cus) {
  struct Candidate {
    beam_tile_cfg cfg;
    bool lines;
    int occ;
    double alone, full, round, launch;
  };
  static const Candidate kCandidates[] = {
      {{256, 256, 128, 64, 0, 0}, false, 1, 7.37, 7.37, 8.55, 0.0},
      {{224, 256, 112, 64, 0, 0}, false, 1, 6.73, 6.73, 7.33, 0.0},
      {{192, 256, 96, 64, 0, 0}, false, 1, 6.16, 6.16, 6.09, 0.0},
      {{256, 128, 64, 64, 0, 0}, false, 1, 5.17, 5.17, 4.62, 0.0},
      {{128, 256, 64, 64, 0, 0}, false, 1, 4.84, 4.84, 4.31, 0.11},
      {{128, 128, 64, 64, 0, 0}, false, 2, 3.89, 3.81, 2.88, 1.25},
      {{128, 128, 64, 64, 2, 0}, false, 1, 3.93, 3.93, 3.29, 1.13},
      {{128, 64, 64, 32, 0, 0}, false, 2, 2.62, 2.76, 1.82, 1.34},
      {{128, 64, 64, 32, 2, 0}, false, 1, 2.77, 2.77, 2.47, 1.36},
      {{64, 128, 32, 64, 0, 0}, false, 2, 2.10, 2.71, 1.90, 0.87},
      {{64, 128, 32, 64, 2, 0}, false, 1, 2.66, 2.66, 2.57, 1.09},
      {{64, 64, 32, 32, 0, 0}, false, 4, 1.57, 2.24, 1.60, 0.91},
      {{64, 64, 32, 32, 2, 0}, false, 1, 2.00, 2.00, 2.12, 0.96},
      {{64, 64, 32, 32, 2, 0}, true, 1, 2.72, 2.72, 2.45, 0.88},
      {{96, 64, 48, 32, 2, 0}, true, 1, 3.42, 3.42, 2.67, 0.96},
      {{64, 128, 32, 64, 2, 0}, true, 1, 3.72, 3.72, 3.08, 0.91},
      {{128, 64, 64, 32, 2, 0}, true, 1, 3.63, 3.63, 3.10, 1.19},
      {{96, 128, 48, 64, 2, 0}, true, 1, 4.65, 4.65, 3.90, 0.86},
      {{128, 128, 64, 64, 2, 0}, true, 1, 5.18, 5.18, 4.75, 0.82},
      {{160, 128, 80, 64, 2, 0}, true, 1, 6.07, 6.07, 4.35, 0.89},
      {{192, 128, 96, 64, 2, 0}, true, 1, 6.45, 6.45, 6.58, 0.26},
  };
  // What choose_default names stays unless another is 4% ahead by this model; 64 x 64 tiles of at most two to a CU under a sum of up
  // to five K tiles, where the model is off by as much as its picks are ahead, unless 15% (639 x 1648 x 272 in 64 x 64 tiles 4.5 us, its
  // best, 96 x 64 by lines, 4.8; 961 x 1400 x 216 4.5, 4.7; 321 x 3536 x 240 4.3, 4.5; but 559 x 2752 x 264 5.0, in 128 x 64 4.5).
  beam_tile_cfg named;
  int split;
  if (choose_default(M, N, K, -1, &named, &split) != BEAM_OK) named = kCandidates[0].cfg;
  const Candidate *best = nullptr, *stays = nullptr;
  double best_us = 0, stays_us = 0;
  for (const Candidate& k : kCandidates) {
    const long tiles = (long)((M + k.cfg.block_m - 1) / k.cfg.block_m) * ((N + k.cfg.block_n - 1) / k.cfg.block_n);
    const long load = (tiles + cus - 1) / cus;  // workgroups per CU
    const long conc = load < k.occ ? load : k.occ;
    const double rate = k.occ == 1 ? k.alone : k.alone + (k.full - k.alone) * (double)(conc - 1) / (k.occ - 1);
    const double mflop = 2.0e-6 * k.cfg.block_m * k.cfg.block_n * (double)(((long)K + kBK - 1) / kBK * kBK);
    double us = (double)((load + k.occ - 1) / k.occ) * k.round + (double)load * mflop / rate + k.launch;
    // (From 192 x 128 on, a round that nearly fills the chip moves its operands at the fabric's rate: on 159 shapes 192 x 128 tiles by
    // lines take 0.93 of the model's time with 180 tiles, 1.0 with 204, 1.1 with 240, 1.15 to 1.4 with 252, and 256 x 128 ones
    // alike.  1422 x 4040 x 528 by lines 17.0 us, in 256 x 128 tiles 11.9; 3629 x 1624 x 504 16.0, 11.9; on those shapes the picks
    // are 0.9% behind the best with this term and 1.7% without it.  Not on the tile that is named, since what would take its place in
    // two rounds is slowed by as much: 6645 x 1584 x 4192 in 245 tiles of 192 x 256 97, in 455 by lines 103.)
    const bool is_named = !k.lines && k.cfg.block_m == named.block_m && k.cfg.block_n == named.block_n && k.cfg.pipeline == named.pipeline;
    if (!is_named && load == 1 && k.cfg.block_m * k.cfg.block_n >= 192 * 128 && tiles > 0.75 * cus) us *= 1 + 0.6 * ((double)tiles / cus - 0.75);
    if (!best || us < best_us) best = &k, best_us = us;
    if (is_named) stays = &k, stays_us = us;
  }
  const bool short_sum = K < 320 && named.block_m * named.block_n == 64 * 64 && (long)((M + 63) / 64) * ((N + 63) / 64) <= 2L * cus;
  if (stays && best_us > (short_sum ? 0.85 : 0.96) * stays_us) best = stays;
  LineChoice t = {best->cfg, best->lines, best == stays ? 0 : stays ? stays_us - best_us : 1e9};
  t.cfg.group_m = default_group_m(t.cfg.block_m, t.cfg.block_n);
  return t;
}

// The same for beam_matmul_nn, where only rows of A can be off lines for K's sake: whole chunks in B's rows (N % 8 == 0), and not.
// Fitted to 120 and 90 shapes with M and N from 32 and 64 to 8192 (5001); `named` is what choose_default's tile has become there,
// and stays unless another is 8% ahead by the model.  On the 100 and 56 of them that come here the pick is 2.1% and 4.9% behind
// the best on average, 20% and 37% at worst; what ran before took 7.1% and 4.6% more than the pick.  us, before -> now: 3059 x 368
// x 7800 45.8 -> 35.5, 841 x 6176 x 1416 23.8 -> 21.6, 1369 x 957 x 208 7.6 -> 6.1, 4397 x 3888 x 280 24.2 -> 23.0.
LineChoice nn_off_lines_tile(int M, int N, int K, const beam_tile_cfg& named, int cus) {
  struct Candidate {
    beam_tile_cfg cfg;
    bool lines;
    int occ;
    double alone[2], full[2], round[2], launch[2];  // N % 8 == 0, else
  };
  static const Candidate kCandidates[] = {
      {{256, 256, 128, 64, 0, 0}, false, 1, {7.34, 7.85}, {7.34, 7.85}, {8.27, 7.56}, {0, 2.82}},
      {{224, 256, 112, 64, 0, 0}, false, 1, {7.05, 7.31}, {7.05, 7.31}, {7.45, 6.95}, {0, 2.69}},
      {{192, 256, 96, 64, 0, 0}, false, 1, {6.51, 6.92}, {6.51, 6.92}, {6.59, 6.38}, {0, 2.55}},
      {{256, 128, 64, 64, 0, 0}, false, 1, {5.14, 5.76}, {5.14, 5.76}, {4.74, 4.65}, {0, 2.96}},
      {{128, 256, 64, 64, 0, 0}, false, 1, {5.10, 5.29}, {5.10, 5.29}, {4.69, 4.52}, {0, 2.73}},
      {{128, 128, 64, 32, 0, 0}, false, 2, {3.93, 4.06}, {3.88, 3.37}, {3.50, 3.10}, {0.36, 2.98}},
      {{128, 128, 64, 32, 2, 0}, false, 1, {4.09, 4.40}, {4.09, 4.40}, {3.63, 4.90}, {0.38, 1.10}},
      {{128, 64, 64, 32, 0, 0}, false, 2, {2.25, 2.27}, {2.69, 2.76}, {2.39, 2.94}, {0.92, 0.93}},
      {{128, 64, 64, 32, 2, 0}, false, 1, {2.58, 2.79}, {2.58, 2.79}, {2.78, 3.12}, {1.18, 1.36}},
      {{64, 128, 32, 64, 0, 0}, false, 2, {1.96, 1.92}, {2.84, 2.81}, {2.46, 2.86}, {0.72, 1.90}},
      {{64, 128, 32, 64, 2, 0}, false, 1, {2.97, 2.93}, {2.97, 2.93}, {3.02, 3.44}, {1.17, 1.92}},
      {{64, 64, 32, 32, 0, 0}, false, 4, {1.29, 1.29}, {2.28, 2.52}, {2.25, 2.95}, {0.63, 0.68}},
      {{64, 64, 32, 32, 2, 0}, false, 1, {1.96, 1.96}, {1.96, 1.96}, {2.51, 2.52}, {0.82, 1.24}},
      {{64, 64, 32, 32, 2, 0}, true, 1, {2.26, 2.19}, {2.26, 2.19}, {2.43, 2.84}, {0.91, 1.19}},
      {{96, 64, 48, 32, 2, 0}, true, 1, {2.80, 2.76}, {2.80, 2.76}, {2.55, 3.18}, {0.98, 1.29}},
      {{64, 128, 32, 32, 2, 0}, true, 1, {2.74, 2.82}, {2.74, 2.82}, {2.77, 3.70}, {0.89, 1.69}},
      {{96, 128, 48, 64, 2, 0}, true, 1, {3.68, 3.85}, {3.68, 3.85}, {3.79, 5.68}, {1.00, 1.55}},
      {{128, 128, 64, 32, 2, 0}, true, 1, {4.28, 4.67}, {4.28, 4.67}, {3.43, 5.32}, {0.53, 0.93}},
      {{160, 128, 80, 64, 2, 0}, true, 1, {4.21, 4.48}, {4.21, 4.48}, {3.52, 5.15}, {1.61, 2.70}},
      {{192, 128, 96, 64, 2, 0}, true, 1, {5.15, 5.64}, {5.15, 5.64}, {5.30, 6.83}, {1.43, 2.80}},
  };
  const int odd = N % 8 != 0 ? 1 : 0;
  const Candidate *best = nullptr, *stays = nullptr;
  double best_us = 0, stays_us = 0;
  for (const Candidate& k : kCandidates) {
    const bool is_named = !k.lines && k.cfg.block_m == named.block_m && k.cfg.block_n == named.block_n && k.cfg.pipeline == named.pipeline;
    // (Rows of B that are not whole chunks under a short sum: no other wide tile.  2985 x 1381 x 360 in 128 x 128 tiles 12.7 us, by
    // lines in 160 x 128 14.0, in 256 x 128 14.3.)
    if (odd && K < 600 && k.cfg.block_n > 64 && !is_named) continue;
    const long tiles = (long)((M + k.cfg.block_m - 1) / k.cfg.block_m) * ((N + k.cfg.block_n - 1) / k.cfg.block_n);
    const long load = (tiles + cus - 1) / cus;
    const long conc = load < k.occ ? load : k.occ;
    const double rate = k.occ == 1 ? k.alone[odd] : k.alone[odd] + (k.full[odd] - k.alone[odd]) * (double)(conc - 1) / (k.occ - 1);
    const double mflop = 2.0e-6 * k.cfg.block_m * k.cfg.block_n * (double)(((long)K + kBK - 1) / kBK * kBK);
    const double us = (double)((load + k.occ - 1) / k.occ) * k.round[odd] + (double)load * mflop / rate + k.launch[odd];
    if (!best || us < best_us) best = &k, best_us = us;
    if (is_named) stays = &k, stays_us = us;
  }
  // (13% under a short sum, as in off_lines_tile, of 64 x 128 by lines a little longer: 1327 x 1320 x 264 in 64 x 64 tiles 5.9 us, by lines 6.1; 235
  // x 2872 x 272 4.4, 4.7; 401 x 3912 x 336 6.2, 6.5.)
  const bool short_sum = !odd && (K < 312 || (K < 350 && best->lines && best->cfg.block_m == 64 && best->cfg.block_n == 128));
  if (stays && best_us > (short_sum ? 0.87 : 0.92) * stays_us) return LineChoice{named, false};
  LineChoice t = {best->cfg, best->lines};
  t.cfg.group_m = default_group_m(t.cfg.block_m, t.cfg.block_n);
  return t;
}

// LDS of one of its workgroups: two slots of a K tile for each wavefront, rows in blocks of 16.
constexpr int kLdsBytes = 160 * 1024;  // of a CU
int kw_lds_bytes(const KwPlan& plan) { return plan.waves * 2 * ((plan.rows < 16 ? 16 : plan.rows) + plan.cols) * kRowBytes; }

RowStarts row_starts(const void* A, const void* B, int K, bool b_kmajor) {
  const uintptr_t at = (uintptr_t)A | (b_kmajor ? 0 : (uintptr_t)B);
  return K % kBK == 0 && (at & 127) == 0 ? kOnLines : K % 8 == 0 && (at & 15) == 0 ? kOnChunks : kAnywhere;
}

void kw_params(KwParams* p, const KwPlan& plan, const void* A, const void* B, void* C, int M, int N, int K) {
  p->A = A;
  p->B = B;
  p->C = C;
  p->M = M;
  p->N = N;
  p->K = K;
  p->tiles_m = (M + plan.rows - 1) / plan.rows;
  p->tiles_n = (N + plan.cols - 1) / plan.cols;
  p->group_m = 8;
  p->divs = make_tile_divs(p->tiles_m, p->tiles_n, p->group_m);
}

hipError_t run_kwave(const KwPlan& plan, const void* A, const void* B, void* C, int M, int N, int K, int dtype, bool b_kmajor, hipStream_t st) {
  KwParams p;
  kw_params(&p, plan, A, B, C, M, N, K);
  return dtype == BEAM_F16 ? launch_gemm_kwave<_Float16>(plan, p, b_kmajor, st) : launch_gemm_kwave<__bf16>(plan, p, b_kmajor, st);
}

}  // namespace

extern "C" {

int beam_gemmrc(const void* A, const void* B, void* C, int M, int N, int K, int dtype,
                const beam_tile_cfg* cfg, void* stream) {
  bool generic;
  int rc = check_problem(A, B, C, M, N, K, dtype, &generic);
  if (rc) return rc;
  if (M == 0 || N == 0) return BEAM_OK;
  if ((rc = beam_init())) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (K == 0) {
    BEAM_HIP(launch_zero_u16(C, (size_t)M * N, st));
    return BEAM_OK;
  }
  if (generic) {  // whatever tile was named: the tiled kernels cannot take this problem
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, false, false, st));
    return BEAM_OK;
  }
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  if (!cfg) {
    if (const KwPlan kw = kw_plan(M, N, K, false, false, true, row_starts(A, B, K, false), cus); kw.rows) {
      BEAM_HIP(run_kwave(kw, A, B, C, M, N, K, dtype, false, st));
      return BEAM_OK;
    }
  }
  beam_tile_cfg c;
  const KernelSet* ks;
  const bool off_lines = !cfg && K % kBK != 0 && row_starts(A, B, K, false) == kOnChunks;
  if (off_lines) {
    const LineChoice t = off_lines_tile(M, N, K, cus);
    c = t.cfg;
    if (t.lines) {
      GemmParams p = base_params(A, B, M, N, K, c);
      p.C = C;
      p.c_store = store_kind(c, 4, false, C, M, N, K);
      const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, 1);
      BEAM_HIP(dtype == BEAM_F16 ? launch_gemm_lines<_Float16>(c.block_m, c.block_n, p, grid, st) : launch_gemm_lines<__bf16>(c.block_m, c.block_n, p, grid, st));
      return BEAM_OK;
    }
  }
  if ((rc = resolve_cfg(off_lines ? &c : cfg, M, N, K, &c, &ks, -1, true))) {
    if (!rows_unaligned(A, B, C, K)) return rc;
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, false, false, st));
    return BEAM_OK;
  }
  // 128 x 128 tiles on the deep pipeline: four wavefronts of 64 x 64 read a third less out of LDS than eight of 64 x 32 (which
  // the library's choice names, for the [K][N] layout's sake).  us, 64 x 32 -> 64 x 64: 2048^3 20.2 -> 18.8, bf16 19.6 -> 18.3,
  // 1500 x 2500 x 2048 20.7 -> 19.4, 1792^3 14.9 -> 14.2, 1500 x 1500 x 4000 32.3 -> 32.1; [K][N] 2048^3 21.1, 21.9.
  if (!cfg && c.pipeline == 2 && c.block_m == 128 && c.block_n == 128 && c.wave_m == 64 && c.wave_n == 32) {
    c.wave_n = 64;
    if ((rc = resolve_cfg(&c, M, N, K, &c, &ks))) return rc;
  }
  GemmParams p = base_params(A, B, M, N, K, c);
  p.C = C;
  const long tiles = (long)p.tiles_m * p.tiles_n;
  // The 256 x 256 tile of four 128 x 128 wavefronts has a kernel of its own (gemm_w4.h), built for problems
  // of a round of workgroups or more: one workgroup per CU walks its tiles with the operand ring running
  // through the tile boundaries.  It is what the tile {256, 256, 128, 128} means wherever its preconditions
  // hold (elsewhere that tile is the 4-wavefront member of the gemm_kernel.h family), and what
  // beam_default_config names from one full round of workgroups on.
  const bool w4_fits = c.pipeline == 0 && K % kBK == 0 && K >= kW4MinK && N % 8 == 0 && ((uintptr_t)C & 15) == 0 && N <= (1 << 21);
  const bool w4_named = c.block_m == 256 && c.block_n == 256 && c.wave_m == 128 && c.wave_n == 128;
  if (w4_named && !w4_fits && !cfg) {  // the library's own choice, but C is only 8-byte aligned: the 8-wavefront tile
    c.wave_m = 128;
    c.wave_n = 64;
    if ((rc = resolve_cfg(&c, M, N, K, &c, &ks))) return rc;
  }
  if (w4_fits && w4_named) {
    // Non-temporal stores of C pay when C is larger than the 256 MB last-level cache (and the K loops
    // are not so short that the writes are the bound).
    p.c_store = (size_t)M * N * 2 >= ((size_t)256 << 20) && K >= 1024 ? kStoreStreaming : store_kind(c, ks->threads / 64, true, C, M, N, K);
    BEAM_HIP(launch_gemm_w4(p, dtype, dim3((unsigned)(tiles < cus ? tiles : cus), 1, 1), st));
    return BEAM_OK;
  }
  // More than one round of workgroups of another large tile: one workgroup per CU walks the tiles and
  // loads the next one's first operand tiles while it stores the current one (kEpiStoreLoop).
  // That kernel stores 16 bytes per lane through a buffer descriptor and has no short K tile.
  // Against one workgroup per tile, same machine: 16384 x 16384 x 2048 822 against 841 us,
  // 8192 x 8192 x 512 71 against 74.5 us, 8192 x 8192 x 2048 205 against 207 us, 8192^3 no difference.
  GemmLauncher loop = c.pipeline == 0 ? ks->launch[dtype][kEpiStoreLoop][0] : nullptr;
  if (loop && tiles > cus && K % kBK == 0 && N % 8 == 0 && ((uintptr_t)C & 15) == 0 && N <= (1 << 21)) {
    // Non-temporal stores of C pay when C is larger than the 256 MB last-level cache (and the K loops
    // are not so short that the writes are the bound): 16384 x 16384 x 2048 +2.5%, x 4096 +1.2%; an
    // 8192 x 8192 output (134 MB) is absorbed by that cache and loses 0.5-3% with them.
    p.c_streaming = (size_t)M * N * 2 >= ((size_t)256 << 20) && K >= 1024;
    BEAM_HIP(loop(p, dim3((unsigned)cus, 1, 1), st));
    return BEAM_OK;
  }
  p.c_store = store_kind(c, ks->threads / 64, false, C, M, N, K);
  GemmLauncher one_group = cfg ? nullptr : deep_one_group(*ks, c, M, N, K, dtype, false, cus);
  BEAM_HIP((one_group ? one_group : ks->launch[dtype][kEpiStore][c.pipeline])(p, dim3((unsigned)tiles, 1, 1), st));
  return BEAM_OK;
}

int beam_matmul_nn(const void* A, const void* B, void* C, int M, int N, int K, int dtype, const beam_tile_cfg* cfg,
                   void* stream) {
  bool generic;
  int rc = check_problem(A, B, C, M, N, K, dtype, &generic);
  if (rc) return rc;
  if (M == 0 || N == 0) return BEAM_OK;
  if ((rc = beam_init())) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (K == 0) {
    BEAM_HIP(launch_zero_u16(C, (size_t)M * N, st));
    return BEAM_OK;
  }
  // rows of B ([K][N]) shorter than a chunk of 16 bytes, or more than a descriptor spans: the plain kernel
  if (generic || N < 8 || N > (N % 8 != 0 ? 1 << 23 : 1 << 24)) {
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, true, false, st));
    return BEAM_OK;
  }
  if (!cfg) {
    if (const KwPlan kw = kw_plan(M, N, K, true, false, true, row_starts(A, B, K, true), g_dev.cus > 0 ? g_dev.cus : 256); kw.rows) {
      BEAM_HIP(run_kwave(kw, A, B, C, M, N, K, dtype, true, st));
      return BEAM_OK;
    }
  }
  beam_tile_cfg c;
  const KernelSet* ks;
  if ((rc = resolve_cfg(cfg, M, N, K, &c, &ks, -1, true))) {
    if (N % 8 == 0 && !rows_unaligned(A, B, C, K)) return rc;
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, true, false, st));
    return BEAM_OK;
  }
  if (!cfg) {
    // The library's choice is priced for B as [N][K].  In this layout a B fragment is two LDS reads, and the tiles
    // whose wavefronts are 64 columns wide pay for it: eight wavefronts of 64 x 32 instead of four of 64 x 64
    // (768 x 3072 x 768: 8.3 against 12.7 us; 2048 x 2048 x 512: 7.9 against 10.0), and 128 x 64 tiles of 64 x 32
    // instead of 64 x 128 tiles of 32 x 64 where that does not make more tiles (256 x 8192 x 8192: 57 against 71).
    // (Not where two K groups are held up by A's rows, which lie off 128-byte lines and fill LDS at half the rate: 64 of them
    // instead of 128, 2048 x 1024 x 1032 9.8 against 10.6; x 1024 9.6, 9.1.)
    auto tiles_of = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    beam_tile_cfg alt = c;
    if (c.block_m == 128 && c.block_n == 128 && c.wave_m == 64 && c.wave_n == 64) {
      alt.wave_n = 32;
    } else if (c.block_m == 64 && c.block_n == 128 && c.wave_m == 32 && c.wave_n == 64 && tiles_of(128, 64) <= tiles_of(64, 128) &&
               (c.pipeline != 2 || K % kBK == 0)) {
      alt.block_m = 128, alt.block_n = 64, alt.wave_m = 64, alt.wave_n = 32;
    }
    const KernelSet* alt_ks = nullptr;
    if ((alt.wave_n != c.wave_n) && resolve_cfg(&alt, M, N, K, &alt, &alt_ks) == BEAM_OK) c = alt, ks = alt_ks;
    if (K % kBK != 0 && row_starts(A, B, K, true) == kOnChunks) {
      const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
      const LineChoice t = nn_off_lines_tile(M, N, K, c, cus);
      c = t.cfg;
      if (t.lines) {
        GemmParams p = base_params(A, B, M, N, K, c);
        p.C = C;
        p.c_store = store_kind(c, 4, false, C, M, N, K);
        const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, 1);
        BEAM_HIP(dtype == BEAM_F16 ? launch_gemm_lines_kmajor<_Float16>(c.block_m, c.block_n, p, grid, st)
                                   : launch_gemm_lines_kmajor<__bf16>(c.block_m, c.block_n, p, grid, st));
        return BEAM_OK;
      }
      if ((rc = resolve_cfg(&c, M, N, K, &c, &ks))) return rc;
    }
  }
  // The 4-wavefront kernel, as in beam_gemmrc (its stores write whole chunks of 8 columns); the K tile's offset into B is a
  // 32-bit scalar there.
  const bool w4_fits = c.pipeline == 0 && K % kBK == 0 && K >= kW4MinK && N % 8 == 0 && ((uintptr_t)C & 15) == 0 && N <= (1 << 21) &&
                       (size_t)K * N * 2 < ((size_t)1 << 31);
  const bool w4_named = c.block_m == 256 && c.block_n == 256 && c.wave_m == 128 && c.wave_n == 128;
  if (w4_named && !w4_fits && !cfg) {
    c.wave_m = 128;
    c.wave_n = 64;
    if ((rc = resolve_cfg(&c, M, N, K, &c, &ks))) return rc;
  }
  GemmParams p = base_params(A, B, M, N, K, c);
  p.C = C;
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  if (w4_fits && w4_named) {
    const long tiles = (long)p.tiles_m * p.tiles_n;
    p.c_store = (size_t)M * N * 2 >= ((size_t)256 << 20) && K >= 1024 ? kStoreStreaming : store_kind(c, ks->threads / 64, true, C, M, N, K);
    BEAM_HIP(launch_gemm_w4_kmajor(p, dtype, dim3((unsigned)(tiles < cus ? tiles : cus), 1, 1), st));
    return BEAM_OK;
  }
  p.c_store = store_kind(c, ks->threads / 64, false, C, M, N, K);
  GemmLauncher one_group = cfg ? nullptr : deep_one_group(*ks, c, M, N, K, dtype, true, cus);
  BEAM_HIP((one_group ? one_group : ks->launch_kmajor[dtype][c.pipeline])(p, dim3((unsigned)(p.tiles_m * p.tiles_n), 1, 1), st));
  return BEAM_OK;
}

int beam_silu(const void* X, void* Y, long long count, int dtype, void* stream) {
  if (count < 0) return fail(BEAM_ERR_INVALID, "negative element count %lld", count);
  if (dtype != BEAM_F16 && dtype != BEAM_BF16) return fail(BEAM_ERR_UNSUPPORTED, "dtype %d: only fp16 (0) and bf16 (1)", dtype);
  if (count == 0) return BEAM_OK;
  if (!X || !Y) return fail(BEAM_ERR_INVALID, "null elementwise pointer");
  if (((uintptr_t)X | (uintptr_t)Y) & 15) return fail(BEAM_ERR_UNSUPPORTED, "X and Y must be 16-byte aligned");
  int rc = beam_init();
  if (rc) return rc;
  BEAM_HIP(launch_silu(X, Y, (size_t)count, dtype, (hipStream_t)stream));
  return BEAM_OK;
}

int beam_parallel_gemmrc_silu(const void* A, const void* B, void* C, int M, int N, int K, const void* X, void* Y,
                              long long count, int dtype, const beam_tile_cfg* cfg, void* stream) {
  bool generic;
  int rc = check_problem(A, B, C, M, N, K, dtype, &generic);
  if (rc) return rc;
  if (count < 0) return fail(BEAM_ERR_INVALID, "negative element count %lld", count);
  if (count > 0) {
    if (!X || !Y) return fail(BEAM_ERR_INVALID, "null elementwise pointer");
    if (((uintptr_t)X | (uintptr_t)Y) & 15) return fail(BEAM_ERR_UNSUPPORTED, "X and Y must be 16-byte aligned");
    if (count > kMaxSideElems)
      return fail(BEAM_ERR_UNSUPPORTED, "count=%lld exceeds %lld elements (one buffer descriptor)", count, kMaxSideElems);
  }
  if (M == 0 || N == 0 || K == 0 || generic) {  // no (tiled) K loop to hide anything in: the two halves run one after the other
    if ((rc = beam_gemmrc(A, B, C, M, N, K, dtype, cfg, stream))) return rc;
    return beam_silu(X, Y, count, dtype, stream);
  }
  if ((rc = beam_init())) return rc;
  beam_tile_cfg c;
  const KernelSet* ks;
  rc = resolve_cfg(cfg, M, N, K, &c, &ks);
  if (cfg && !rc && c.pipeline == 2) {
    // beam_default_config names the deep pipeline for tiles that it otherwise names with pipeline 0; passed on to here, such
    // a tile carries the job with that
    beam_tile_cfg own;
    int own_split;
    bool raised = false;
    if (choose_default(M, N, K, -1, &own, &own_split, &raised) == BEAM_OK && raised && own.block_m == c.block_m &&
        own.block_n == c.block_n && own.wave_m == c.wave_m && own.wave_n == c.wave_n)
      c.pipeline = 0;
  }
  if (cfg && (rc || c.pipeline == 2)) {  // no kernel carries a side job there
    if (!rows_unaligned(A, B, C, K)) return rc ? rc : fail(BEAM_ERR_UNSUPPORTED, "the side job runs with pipeline 0 or 1");
    if ((rc = beam_gemmrc(A, B, C, M, N, K, dtype, cfg, stream))) return rc;
    return beam_silu(X, Y, count, dtype, stream);
  }
  if (rc) return rc;
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  const long long wgs = (long long)((M + c.block_m - 1) / c.block_m) * ((N + c.block_n - 1) / c.block_n);
  const long long per_pass = wgs * ks->threads;  // units one K tile of the whole grid covers
  // With the library's tile:
  //   * Where the GEMM runs on gemm_kwave.h, the job rides in workgroups of its own behind the tiles (one launch; two launches,
  //     us: 256 x 256 x 512 with 2^18 elements 3.7, 4.6; 1000 x 1003 x 1024 with 2^22 9.5, 10.3).  Such a workgroup holds a
  //     tile's LDS, and a long job is bound by how many wavefronts of it a CU then has (operands from memory).  12 and more,
  //     tiles of up to 48 rows + columns: any length (297 x 400 x 1024 with 2^24 17.7, 20.1, with 2^26 52.6, 58.4).  8: up to
  //     2^24 elements with 64 columns or whole-line fills (3 x 8304 x 1024 20.5, 22.1; 1720 deep, 14.3 Mi, 17.0, 21.6), else up to
  //     2^23, since two accesses of a thread are in flight there and not eight (304 deep, 8.1 Mi, 9.4, 11.0; 408 deep, 13.5 Mi,
  //     19.4, 17.5).  4: up to 2^23 (512 x 1024 x 2048 17.1, 17.4; with 2^24 26.7, 25.0).
  //   * ... but not where such a workgroup is a CU's only one, not every one finds a CU without a tile, and sum and job are
  //     short: it then starts behind a tile, 1-2 us that the tiled kernel's K loop hides.  (Behind the tiles, in the loop;
  //     operands from memory, then the same in every call: 512 x 1024, 256 tiles, x 256 with 2^18 5.5, 4.5; 5.3, 3.9; with 2^20,
  //     4 passes of that kernel's grid, 6.2, 5.9; 5.7, 4.4; x 512 with 2^18 6.4, 6.2; 5.7, 4.7, with 2^20 6.7, 9.1; x 1024 with
  //     2^18 7.3, 9.1; 1000 x 1003 x 512 with 2^12 6.4, 7.1.  982 x 504 x 112, 248 tiles and 35 workgroups, 5.8, 4.7; 1241 x
  //     336 x 224, 234 tiles and 14 workgroups, 4.3, 4.4.)
  //   * A GEMM kernel that carries no side job and is the faster one by more than the second launch costs (2.5 us): the deep
  //     pipeline with less than half the CUs busy, or with tiles of 64 rows (two K groups).  One launch, two launches: 2048 x
  //     1024 x 2048 with 2^18 elements 18.9, 15.9.  Tiles of 128 rows gain less than that: 128 x 128 (one group) 496 x 5688 x
  //     1224 13.2, 15.3; 128 x 64 5813 x 312 x 6256 46.4, 47.2.  64 x 64 tiles with K below 2048: two launches
  //     from K = 1024 or 2^21 elements on (1024^3 with 2^18 9.1, 9.0, with 2^22 16.3, 11.2; 1024 x 1024 x 512 with 2^18 6.1, 7.8,
  //     with 2^22 9.9, 9.6).
  if (!cfg) {
    if (const KwPlan kw = kw_plan(M, N, K, false, false, true, row_starts(A, B, K, false), cus, true); kw.rows) {
      const long long per_wg = (long long)kw.waves * 64 * 8 * 8;  // elements of one round of a side workgroup's accesses
      const long long want = (count + per_wg - 1) / per_wg;
      const int per_cu = kLdsBytes / kw_lds_bytes(kw);  // workgroups of the launch on a CU
      const long long passes = ((count >> 3) + per_pass - 1) / per_pass;  // of the tiled kernel's grid over the job
      const bool loop = per_cu == 1 && (long long)((M + kw.rows - 1) / kw.rows) * ((N + kw.cols - 1) / kw.cols) + want > cus && passes <= 4 &&
                        passes * K <= 1024 && (K <= 256 || (K <= 512 && count >= (1 << 16)));
      if (!loop) {
        if (count > (per_cu * kw.waves >= 12 ? kMaxSideElems : per_cu * kw.waves >= 8 && (kw.shift || kw.cols == 64) ? 1 << 24 : 1 << 23)) {
          if ((rc = beam_gemmrc(A, B, C, M, N, K, dtype, nullptr, stream))) return rc;
          return beam_silu(X, Y, count, dtype, stream);
        }
        KwSideParams p;
        kw_params(&p, kw, A, B, C, M, N, K);
        p.side_x = X;
        p.side_y = Y;
        p.side_count = count;
        const int side = (int)(want < 8 * cus ? want : 8 * cus);
        BEAM_HIP(dtype == BEAM_F16 ? launch_gemm_kwave_side<_Float16>(kw, p, side, (hipStream_t)stream)
                                   : launch_gemm_kwave_side<__bf16>(kw, p, side, (hipStream_t)stream));
        return BEAM_OK;
      }
    }
    const bool two_groups = c.block_m == 64 && (K >= 2048 || (c.block_n == 64 && (K >= 1024 || count > (1 << 21))));
    if (c.pipeline == 2 && ((wgs * 2 < cus && K >= 2048) || two_groups)) {
      if ((rc = beam_gemmrc(A, B, C, M, N, K, dtype, nullptr, stream))) return rc;
      return beam_silu(X, Y, count, dtype, stream);
    }
    if (c.pipeline == 2) c.pipeline = 0;
  }
  GemmParams p = base_params(A, B, M, N, K, c);
  p.C = C;
  p.side_x = X;
  p.side_y = Y;
  p.side_count = count;
  // The narrowest unit with which the job still ends inside the K loop: the work is then spread
  // evenly over the tiles instead of crowding the first ones.  A job longer than the loop keeps
  // 16-byte units and finishes after the GEMM's epilogue.
  const long long k_tiles = ((long long)K + kBK - 1) / kBK;
  p.side_width = 16;
  for (int w = 4; w < 16; w *= 2) {
    const long long units = (count >> 3) * (16 / w);
    if ((units + per_pass - 1) / per_pass <= k_tiles) {
      p.side_width = w;
      break;
    }
  }
  p.side_iters = (int)(((count >> 3) * (16 / p.side_width) + per_pass - 1) / per_pass);
  // Two launches, where the job outlasts the loop or the GEMM alone takes its rows by whole lines, which no kernel with a side
  // job does; the second launch costs about 2.5 us and the job alone 3 us to 1 Mi elements, 8 at 9 Mi, 20 at 25 Mi.  Over 106
  // shapes from 256 x 256 x 256 to 8192^3 with 2^18 to 2^26 elements this rule took 7% off the mean of what one launch took.
  //   * Behind the loop a pass costs 0.4-1.4 us for 16 bytes per thread; a long loop's own passes are the cheaper for it.  One
  //     launch, then two, us: 1602 x 2624 x 320 with 10 Mi (14 passes behind it) 24.7, 16.8; 2156 x 3680 x 448 with 31 Mi (24)
  //     41.6, 37.2; 1226 x 7304 x 320 with 15 Mi (8) 35.6, 23.9; 5000 x 4000 x 512 with 64 Mi (18) 99.0, 82.3; but 7276 x 392 x
  //     256 with 7 Mi (1) 12.0, 13.6.  Tiles of eight wavefronts, one on a CU, move more in a pass, and their later rounds hide
  //     the earlier ones' passes: 5632 x 5632 x 256 in two rounds with 60 Mi (28) 90.5, 73.8; 8192 x 4096 x 256 in two with 64 Mi
  //     (28) 91.8, 83.6, with 32 Mi (12) 51.9, 57.3; 8192 x 8192 x 512 in four with 64 Mi (8) 127.9, 135.0.
  //   * By whole lines, with 2^20 elements or K from 2048 on: 1787 x 2648 x 744 with 38 Mi 73.8, 46.6; 1157 x 3216 x 3880 with
  //     0.5 Mi 56.0, 33.3; 679 x 3080 x 4880 with 2.3 Mi 46.5, 34.3; but 4155 x 496 x 560 with 0.6 Mi 10.4, 11.8.  Where the job
  //     ends inside the loop it is nearly free beside tiles of eight wavefronts, and the lines have to be ahead by 0.4 of what
  //     it takes alone (1908 x 4584 x 3552 with 24 Mi, 5 us ahead, 75.0, 92.4; 1539 x 3648 x 3112 with 20 Mi, 2.6, 62.3, 67.7; but
  //     1653 x 5272 x 4128 with 10 Mi, 6.7, 99.4, 92.6); by 1.1 us under a sum of up to seven K tiles (931 x 608 x 392 with 1.1 Mi,
  //     0.2 us ahead, 7.0, 8.0; 557 x 2472 x 376 with 2.1 Mi, 0.8, 9.4, 10.0; but 2115 x 456 x 392 with 3.7 Mi behind the loop 14.8, 10.1).
  bool by_lines = false;
  if (K % kBK != 0 && row_starts(A, B, K, false) == kOnChunks && (count >= (1 << 20) || K >= 2048)) {
    const LineChoice t = off_lines_tile(M, N, K, cus);
    const double alone = 2.5 + 0.7 * (double)count / (1 << 20);  // us
    const double least = p.side_iters > k_tiles ? 0 : ks->threads == 512 ? 0.4 * alone : k_tiles <= 7 ? 1.1 : 0;
    by_lines = t.lines && t.ahead > least;
  }
  const long long behind = (ks->threads == 512 ? 8 * ((wgs + cus - 1) / cus) : 4) + k_tiles / 8;
  if (!cfg && (by_lines || p.side_iters - k_tiles > behind)) {
    if ((rc = beam_gemmrc(A, B, C, M, N, K, dtype, nullptr, stream))) return rc;
    return beam_silu(X, Y, count, dtype, stream);
  }
  p.c_store = store_kind(c, ks->threads / 64, false, C, M, N, K, true);
  BEAM_HIP(ks->launch[dtype][kEpiStoreSide][c.pipeline](p, dim3((unsigned)wgs, 1, 1), (hipStream_t)stream));
  return BEAM_OK;
}

static int custom_fixed(int bm, int bn, int tm, int tn, const void* A, const void* B, void* C, int M,
                        int N, int K, void* stream) {
  beam_tile_cfg c = {bm, bn, tm, tn, 0, 0};
  return beam_gemmrc(A, B, C, M, N, K, BEAM_F16, &c, stream);
}

int beam_custom_gemmrc_128x128(const void* A, const void* B, void* C, int M, int N, int K, void* stream) {
  return custom_fixed(128, 128, 64, 64, A, B, C, M, N, K, stream);
}
int beam_custom_gemmrc_128x256(const void* A, const void* B, void* C, int M, int N, int K, void* stream) {
  return custom_fixed(128, 256, 64, 64, A, B, C, M, N, K, stream);
}
int beam_custom_gemmrc_256x128(const void* A, const void* B, void* C, int M, int N, int K, void* stream) {
  return custom_fixed(256, 128, 64, 64, A, B, C, M, N, K, stream);
}

// Workspace of a split-K call: fp32 partial sums [split_k][M][N], then (256-byte aligned) the synchronisation
// words of the one-launch form.  A workspace that only holds the partial sums still works: two launches.
static size_t splitk_partial_bytes(int M, int N, int split_k) {
  return (size_t)split_k * (size_t)M * (size_t)N * sizeof(float);
}
size_t beam_splitk_workspace_bytes(int M, int N, int split_k) {
  if (M <= 0 || N <= 0 || split_k <= 0) return 0;
  return align_up(splitk_partial_bytes(M, N, split_k), 256) + (size_t)sk_sync_bytes(M, N, split_k);
}

// 1: the fused GEMM+LayerNorm of the 4-wavefront kernel always runs one workgroup per tile (beam_set_ln_walk)
static std::atomic<int> g_ln_no_walk{[] {
  const char* e = getenv("BEAM_LN_WALK");
  return e && *e == '0' ? 1 : 0;
}()};

// 1: the one-launch split-K runs without reducing workgroups where its multiplying workgroups fit one round of the
// CUs; each of them reduces its share of its tile (beam_dbg_set_splitk_self_reduce: a measurement, off by default)
static std::atomic<int> g_splitk_self_reduce{0};

// 0: one launch where it applies, 1: always the partial kernel followed by the reduce kernel
static std::atomic<int> g_splitk_two_launches{[] {
  const char* e = getenv("BEAM_SPLITK_TWO_LAUNCHES");
  return e && *e && *e != '0' ? 1 : 0;
}()};

int beam_set_splitk_two_launches(int on) {
  g_splitk_two_launches.store(on != 0);
  return BEAM_OK;
}

static int effective_split(int M, int N, int K, const beam_tile_cfg& c, int split_k) {
  const int ktiles = (K + kBK - 1) / kBK;
  if (ktiles <= 1) return 1;
  int s = split_k;
  if (s <= 0) {
    const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
    const long t = (long)((M + c.block_m - 1) / c.block_m) * ((N + c.block_n - 1) / c.block_n);
    s = auto_slices(t, K, cus);
  }
  if (s > ktiles) s = ktiles;
  if (s < 1) s = 1;
  const int per = (ktiles + s - 1) / s;
  return (ktiles + per - 1) / per;  // drop slices that would be empty
}

// The library's own choice (no tile, no slice count) for a sum that one launch without slices is the faster for: K dealt out
// to the wavefronts of small tiles (gemm_kwave.h) where a CU then fills LDS with no more than 600 KB.  Where there is a plan
// for rows on lines there is one for rows anywhere, not the other way round; beam_splitk_effective, which does not know where
// the rows start, goes by the latter, and the call does as it says.
static KwPlan splitk_kw_plan(int M, int N, int K, const beam_tile_cfg* cfg, int split_k, RowStarts rows) {
  if (cfg || split_k > 0 || K >= 8192) return KwPlan{0, 0, 0, false};
  const KwPlan kw = kw_plan(M, N, K, false, false, false, rows, g_dev.cus > 0 ? g_dev.cus : 256);
  return (long)(kw.rows + kw.cols) * K <= 300000 ? kw : KwPlan{0, 0, 0, false};
}

int beam_splitk_effective(int M, int N, int K, const beam_tile_cfg* cfg, int split_k) {
  beam_tile_cfg c;
  const KernelSet* ks;
  if (M <= 0 || N <= 0 || K < 0) return 1;
  if ((K > 0 && K < 8) || K > kMaxK) return 1;  // the plain kernel: no slices
  if (K > 0 && splitk_kw_plan(M, N, K, cfg, split_k, kAnywhere).rows) return 1;
  if (resolve_cfg(cfg, M, N, K, &c, &ks, split_k > 0 ? split_k : 0)) return K % 8 != 0 ? 1 : -1;
  return effective_split(M, N, K, c, split_k);
}

// The once-per-shape line about a slice count the library chose (beam_set_verbose).
static std::atomic<int> g_verbose{[] {
  const char* e = getenv("BEAM_VERBOSE");
  return e && *e && *e != '0' ? 1 : 0;
}()};

int beam_set_verbose(int verbose) {
  g_verbose.store(verbose != 0);
  return BEAM_OK;
}

static void log_split_choice_once(int M, int N, int K, int dtype, const beam_tile_cfg& c, int s) {
  static std::mutex mu;
  static std::set<std::string> seen;
  const long tiles = (long)((M + c.block_m - 1) / c.block_m) * ((N + c.block_n - 1) / c.block_n);
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  char line[256];
  snprintf(line, sizeof line, "split-K [%d,%d,%d] %s: tile %dx%d, %d slices of %d K elements, %ld workgroups = %.2f rounds of %d CUs",
           M, N, K, dtype == BEAM_BF16 ? "bf16" : "fp16", c.block_m, c.block_n, s, split_k_len(K, s), tiles * s,
           (double)(tiles * s) / cus, cus);
  std::lock_guard<std::mutex> lock(mu);
  if (seen.insert(line).second) fprintf(stderr, "[beam] %s\n", line);
}

int beam_gemmrc_splitk(const void* A, const void* B, void* C, int M, int N, int K, int dtype,
                       const beam_tile_cfg* cfg, int split_k, void* ws, size_t ws_bytes, void* stream) {
  bool generic;
  int rc = check_problem(A, B, C, M, N, K, dtype, &generic);
  if (rc) return rc;
  if (M == 0 || N == 0) return BEAM_OK;
  if ((rc = beam_init())) return rc;
  hipStream_t st = (hipStream_t)stream;
  if (K == 0) {
    BEAM_HIP(launch_zero_u16(C, (size_t)M * N, st));
    return BEAM_OK;
  }
  if (generic) {  // one pass of the plain kernel, no slices (beam_splitk_effective says 1)
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, false, false, st));
    return BEAM_OK;
  }
  if (const KwPlan kw = splitk_kw_plan(M, N, K, cfg, split_k, row_starts(A, B, K, false)); kw.rows) {
    if (g_verbose.load(std::memory_order_relaxed)) log_split_choice_once(M, N, K, dtype, beam_tile_cfg{kw.rows, kw.cols, kw.rows, kw.cols, 0, 0}, 1);
    BEAM_HIP(run_kwave(kw, A, B, C, M, N, K, dtype, false, st));
    return BEAM_OK;
  }
  beam_tile_cfg c;
  const KernelSet* ks;
  if ((rc = resolve_cfg(cfg, M, N, K, &c, &ks, split_k > 0 ? split_k : 0))) {
    if (!rows_unaligned(A, B, C, K)) return rc;
    BEAM_HIP(launch_generic_gemm(A, B, C, M, N, K, dtype, false, false, st));
    return BEAM_OK;
  }
  int s = splitk_kw_plan(M, N, K, cfg, split_k, kAnywhere).rows ? 1 : effective_split(M, N, K, c, split_k);
  // Operands whose rows are not 16-byte aligned may be given without room for slices, or with it off 16 bytes (they need
  // none: one pass).
  if (rows_unaligned(A, B, C, K) && (!ws || ((uintptr_t)ws & 15) != 0 || ws_bytes < splitk_partial_bytes(M, N, s))) s = 1;
  if (split_k <= 0 && g_verbose.load(std::memory_order_relaxed)) log_split_choice_once(M, N, K, dtype, c, s);
  if (s == 1) {  // nothing to reduce: the plain kernel writes C directly
    GemmParams p = base_params(A, B, M, N, K, c);
    p.C = C;
    GemmLauncher one_group = cfg ? nullptr : deep_one_group(*ks, c, M, N, K, dtype, false, g_dev.cus > 0 ? g_dev.cus : 256);
    BEAM_HIP((one_group ? one_group : ks->launch[dtype][kEpiStore][c.pipeline])(p, dim3((unsigned)(p.tiles_m * p.tiles_n), 1, 1), st));
    return BEAM_OK;
  }
  const size_t need = splitk_partial_bytes(M, N, s);
  if (!ws || ws_bytes < need)
    return fail(BEAM_ERR_WORKSPACE, "split-K with %d slices needs %zu bytes of workspace, got %zu", s, need, ws_bytes);
  if ((uintptr_t)ws & 15) return fail(BEAM_ERR_UNSUPPORTED, "workspace must be 16-byte aligned");
  GemmParams p = base_params(A, B, M, N, K, c);
  p.ws = (float*)ws;
  p.k_slice = split_k_len(K, s);
  p.splits = s;
  // One launch: the reducing workgroups ride behind the multiplying ones in the same grid.  Needs a tile the
  // form is built for, 16-byte rows of partial sums, at most one flag per lane, a slice that fits one buffer
  // descriptor, and room for the synchronisation words behind the partial sums.
  const GemmLauncher one_launch = ks->launch_partial_fused[dtype][c.pipeline];
  if (one_launch && !g_splitk_two_launches.load(std::memory_order_relaxed) && N % 4 == 0 && s <= 64 &&
      (size_t)M * N <= ((size_t)1 << 28)) {
    // parts of 4 outputs per thread, smaller ones while the reducing workgroups are fewer than the CUs
    const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
    const long tiles = (long)p.tiles_m * p.tiles_n;
    p.sk_out = 4;
    while (p.sk_out > 1 && tiles * sk_parts_per_tile(c.block_m, c.block_n, ks->threads, p.sk_out) < cus) p.sk_out /= 2;
    const long parts = sk_parts_per_tile(c.block_m, c.block_n, ks->threads, p.sk_out);
    const size_t sync_at = align_up(need, 256);
    const size_t sync_bytes = 4 * ((size_t)kSkFlags + (size_t)(tiles * parts) * (size_t)s);
    // Many tiles make many reducing workgroups, and those carry the kernel's LDS allocation: one per CU at a time,
    // round after round behind the last multiplying workgroups.  Beyond two rounds of them the reduce kernel of the
    // two-launch form, which spreads over the CUs at once, is the faster end (2048 x 1024 x 4096 in 2 slices of
    // 128 x 128 tiles: 25.7 against 27.2 us; 1024 x 1024 x 8192 in 4: 25.9 against 24.8 the other way).
    if (ws_bytes >= sync_at + sync_bytes && tiles * parts <= 2l * cus) {
      p.C = C;
      p.sk_sync = (int*)((char*)ws + sync_at);
      p.ln_nonce = g_ln_nonce.fetch_add(1, std::memory_order_relaxed) + 1;
      p.spin_limit = g_ln_spin_limit.load();
      p.sk_self = g_splitk_self_reduce.load(std::memory_order_relaxed) && tiles * s <= cus ? 1 : 0;
      BEAM_HIP(one_launch(p, dim3((unsigned)(tiles * s + (p.sk_self ? 0 : tiles * parts)), 1, 1), st));
      return BEAM_OK;
    }
  }
  BEAM_HIP(ks->launch[dtype][kEpiPartial][c.pipeline](p, dim3((unsigned)(p.tiles_m * p.tiles_n * s), 1, 1), st));
  // Where the workspace has synchronisation words, the reduce kernel marks them "no one-launch call is the latest":
  // a time-out recorded by an earlier one-launch call on this workspace must not be read as this call's.
  const size_t hdr_at = align_up(need, 256);
  int* hdr = ws_bytes >= hdr_at + 4 * (size_t)kSkFlags ? (int*)((char*)ws + hdr_at) : nullptr;
  BEAM_HIP(launch_splitk_reduce((const float*)ws, C, (size_t)M * N, s, dtype, hdr, st));
  return BEAM_OK;
}

int beam_gemmrc_splitk_timed_out(const void* ws, size_t ws_bytes, int M, int N, int split_k_effective, void* stream,
                                 int* timed_out) {
  if (!timed_out || M <= 0 || N <= 0 || split_k_effective < 1) return fail(BEAM_ERR_INVALID, "bad argument");
  *timed_out = 0;
  BEAM_HIP(hipStreamSynchronize((hipStream_t)stream));
  int hdr[4] = {0, 0, 0, 0};
  const size_t sync_at = align_up(splitk_partial_bytes(M, N, split_k_effective), 256);
  // One slice, or a workspace that ends with the partial sums: the call had no waiting workgroups (plain kernel, or
  // partial + reduce kernel), and there are no synchronisation words to read.
  if (!ws || split_k_effective == 1 || ws_bytes < sync_at + sizeof hdr) return BEAM_OK;
  BEAM_HIP(hipMemcpy(hdr, (const char*)ws + sync_at, sizeof hdr, hipMemcpyDeviceToHost));
  *timed_out = hdr[kSkMagic] == kSkMagicValue && hdr[kSkLaunchTag] != 0 && hdr[kSkTimeout] == hdr[kSkLaunchTag];
  return BEAM_OK;
}

size_t beam_splitk_noalloc_max_bytes(void) { return kScratchPartialBytes; }

int beam_gemmrc_splitk_noalloc(const void* A, const void* B, void* C, int M, int N, int K, int dtype,
                               const beam_tile_cfg* cfg, int split_k, void* stream) {
  int rc = beam_init();
  if (rc) return rc;
  bool generic = false;
  if ((rc = check_problem(A, B, C, M, N, K, dtype, &generic))) return rc;
  if (M > 0 && N > 0 && K > 0 && !generic && !rows_unaligned(A, B, C, K)) {  // (those run without slices if need be)
    const int s = beam_splitk_effective(M, N, K, cfg, split_k);
    if (s < 0) return BEAM_ERR_UNSUPPORTED;  // the message is already set
    const size_t need = s > 1 ? splitk_partial_bytes(M, N, s) : 0;
    if (need > kScratchPartialBytes)
      return fail(BEAM_ERR_WORKSPACE, "split-K of %d x %d in %d slices needs %zu bytes; the built-in workspace of the "
                  "no-allocation entry point holds %zu (use beam_gemmrc_splitk with a workspace of your own)", M, N, s, need,
                  kScratchPartialBytes);
  }
  void* ws = nullptr;
  if ((rc = scratch_on_current_device(&ws))) return rc;
  return beam_gemmrc_splitk(A, B, C, M, N, K, dtype, cfg, split_k, ws, kScratchBytes, stream);
}

// Fused GEMM+LayerNorm workspace: [header, 256 bytes | (mean, tag) words | (M2, ~tag) words], one word of
// each kind per (row band, column tile, row).  Nothing in it is ever prepared or cleared: every fused launch
// gets a nonce that no earlier launch of this process had, and the kernel takes a statistics word for
// published only if it carries the tag made from that nonce (gemm_kernel.h: ln_launch_tag).  The library keeps
// no state about workspaces on the host either.
static size_t ln_fused_header_bytes() { return 256; }
static size_t ln_fused_set_bytes(size_t tiles_m, size_t tiles_n, int block_m) {
  return align_up(tiles_m * tiles_n * (size_t)block_m * 2 * sizeof(float), 256);
}

static size_t ln_fused_need(int M, int N, int block_m, int block_n) {
  return ln_fused_header_bytes() + 2 * ln_fused_set_bytes((size_t)(M + block_m - 1) / block_m, (size_t)(N + block_n - 1) / block_n, block_m);
}

static bool ln_fused_applies_on(const beam_tile_cfg& c, const KernelSet& ks, int N, int cus) {
  // The residency argument of the fused kernel (tile_map.h: band_block_tile) is made for 8 XCDs of 32 CUs.
  if (cus != kNumXcd * 32) return false;
  // a band's column tiles are spread over the 8 XCDs; each XCD must hold its share (<= 32) at once,
  // and the band's statistics ((tiles_n + 1) * block_m pairs) are gathered into the kernel's LDS
  const int tiles_n = (N + c.block_n - 1) / c.block_n;
  const int lds = c.pipeline ? ks.lds_bytes_shallow : ks.lds_bytes;
  return tiles_n <= 64 && (size_t)(tiles_n + 1) * c.block_m * 8 <= (size_t)lds;
}
static bool ln_fused_applies(const beam_tile_cfg& c, const KernelSet& ks, int N) { return ln_fused_applies_on(c, ks, N, g_dev.cus); }

static int ln_resolve_mode(int mode, const beam_tile_cfg& c, const KernelSet& ks, int N) {
  if (mode == BEAM_LN_AUTO) return ln_fused_applies(c, ks, N) ? BEAM_LN_FUSED : BEAM_LN_TWOPASS;
  return mode;
}

// GEMM+LayerNorm problems that run on the plain kernels, and the workspace they need (fp32 X).
static bool ln_is_generic(bool gemm_generic, const void* gamma, const void* beta) {
  return gemm_generic || ((((uintptr_t)gamma | (uintptr_t)beta) & 7) != 0);
}
static size_t ln_generic_need(int M, int N) { return align_up((size_t)M * N * sizeof(float), 256); }

// Bytes for tile `c` in `mode` (already resolved: two-pass or fused).
static size_t ln_workspace_need(int M, int N, const beam_tile_cfg& c, int mode) {
  const size_t tiles_n = (size_t)(N + c.block_n - 1) / c.block_n;
  if (mode == BEAM_LN_FUSED) return ln_fused_need(M, N, c.block_m, c.block_n);
  return align_up((size_t)M * N * sizeof(float), 256) + align_up((size_t)M * tiles_n * 2 * sizeof(float), 256);
}

// The tile a GEMM+LayerNorm call runs with: the caller's, or the library's; never the deep pipeline.
// For the one-kernel form (mode AUTO or FUSED on a device it runs on) the library does not take the plain GEMM's
// tile: every workgroup ends with the epilogue's chain of latencies, so a round of workgroups costs a fixed time
// that grows with the tile, and rounds count in whole numbers -- of bands, since a band's tiles wait for each other.
// The model is that sentence: rounds x (fixed + flops of a tile / rate), rates (TFLOP/s per CU) and fixed costs (us)
// fitted by least squares to timings of every tile on 34 shapes; on those of the present kernels
// (beam/ln_tile_timings.json) the pick is within 1.6% of the best tile in the geometric mean, 18% at worst.
struct LnCandidate {
  beam_tile_cfg cfg;
  double rate, fixed;
};
// Two candidates share the 256 x 256 tile: the 4-wavefront kernel of gemm_w4.h (the faster K loop; an epilogue in
// which nothing overlaps the vector work of its one wavefront per SIMD) and the 8-wavefront one (two wavefronts per
// SIMD cover each other's waits in the epilogue).  Measured, the first wins by 3-5% where K is 2048 and more and the
// rounds are few (4096^3: 100.3 against 105.6 us), the second by 3-14% where a tile's K loop is short (8192 x 8192 x
// 1024: 146.1 against 150.7 us; 4096 x 16384 x 1024, whose bands are too wide to walk: 166.8 against 190.8).
static const LnCandidate kLnCandidates[] = {
    {{256, 256, 128, 128, 0, 0}, 7.91, 18.17},  // (only where gemm_w4.h's conditions hold)
    {{256, 256, 128, 64, 0, 0}, 7.08, 14.13},
    {{224, 256, 112, 64, 0, 0}, 6.94, 12.35},
    {{192, 256, 96, 64, 0, 0}, 6.66, 11.01},
    {{256, 128, 64, 64, 0, 0}, 5.38, 8.00},
    {{128, 256, 64, 64, 0, 0}, 5.41, 8.17},
    {{128, 128, 64, 32, 0, 0}, 5.05, 6.65},
    {{64, 128, 32, 64, 0, 0}, 3.33, 3.54},
    {{64, 64, 32, 32, 0, 0}, 2.98, 2.76},
};
// The model's pick for a device of `cus` compute units; false if the one-kernel form applies with none of the tiles.
static bool ln_choose_tile(int M, int N, int K, int cus, beam_tile_cfg* out, const KernelSet** out_ks) {
  double best_us = 1e300;
  bool found = false;
  for (const LnCandidate& k : kLnCandidates) {
    beam_tile_cfg c = k.cfg;
    const KernelSet* ks = nullptr;
    const bool w4 = c.wave_m == 128 && c.wave_n == 128;
    if (w4 && !(K % kBK == 0 && K >= kW4MinK && N % 8 == 0)) continue;
    if (resolve_cfg(&c, M, N, K, &c, &ks, -1, w4) != BEAM_OK || !ln_fused_applies_on(c, *ks, N, cus)) continue;
    // (a band's column tiles wait for each other, so a band that straddles two rounds costs both: a round is
    // worth the whole bands it holds)
    const int tiles_m = (M + c.block_m - 1) / c.block_m, tiles_n = (N + c.block_n - 1) / c.block_n;
    const int bands_per_round = cus / tiles_n > 1 ? cus / tiles_n : 1;
    const double rounds = (double)((tiles_m + bands_per_round - 1) / bands_per_round);
    const double us = rounds * (k.fixed + 2.0e-6 * c.block_m * c.block_n * (double)K / k.rate);
    if (us < best_us) {
      best_us = us;
      *out = c;
      *out_ks = ks;
      found = true;
    }
  }
  return found;
}
static int ln_resolve_cfg(const beam_tile_cfg* cfg, int M, int N, int K, int mode, beam_tile_cfg* c, const KernelSet** ks) {
  int rc = resolve_cfg(cfg, M, N, K, c, ks, -1, true);
  if (rc) return rc;
  if (c->pipeline == 2) c->pipeline = 0;  // the deep pipeline exists for the store / split-K kernels only
  if (cfg || mode == BEAM_LN_TWOPASS || g_dev.cus <= 0) return BEAM_OK;
  beam_tile_cfg alt;
  const KernelSet* alt_ks = nullptr;
  if (ln_choose_tile(M, N, K, g_dev.cus, &alt, &alt_ks)) {
    *c = alt;
    *ks = alt_ks;
  }
  return BEAM_OK;
}

// The one-kernel form among all tiles, those whose fills take whole lines (gemm_kernel.h: Form) included, for rows on 16 bytes;
// `named` is ln_choose_tile's.  The model above with constants for rows on 128-byte lines and off them: TFLOP/s per CU, us per
// round of bands and per launch, least squares on the logarithm over 200 shapes off lines and 160 on them with M from 64 to 8192, N and K
// from 256 to 8192 (beam/line_tile_fit.py, with the timings).  `named` stays unless another tile is 4% ahead by it.  On the 145 and 115 of them
// that come here the pick is 1.9% (off lines) and 3.4% (on) behind the best tile on average, 46% and 28% at worst; what ran before
// took 11% and 9% more than the pick.  The tiles with rings deeper than 3 + 2 slots are ahead on lines too.  us, before -> now: 1978 x 2120 x
// 4888 86 -> 59 (48 with bands in groups), 2908 x 328 x 5736 51 -> 33, 1891 x 920 x 3704 40 -> 28, 6257 x 2744 x 4688 243 -> 196; on lines 1064 x 1040 x
// 3776 42 -> 29, 126 x 6720 x 1472 21.6 -> 19.0.
// 64 columns make the most column tiles, and a workgroup reads its rows' statistics of all of them: `wide`.  Without it 96 x 64 tiles
// ran 666 x 2302 x 704 in 14.0 us, 439 x 2984 x 792 in 15.5 and 301 x 3936 x 960 in 24.6; what runs now takes 11.7, 13.4 and 21.4.
static LineChoice ln_line_tile(int M, int N, int K, const beam_tile_cfg& named) {
  struct Candidate {
    beam_tile_cfg cfg;
    bool lines;
    double rate[2], round[2], launch[2];  // rows off lines, on lines
  };
  static const Candidate kCandidates[] = {
      {{256, 256, 128, 128, 0, 0}, false, {0, 7.60}, {0, 14.89}, {0, 0}},  // (only where it is `named`)
      {{256, 256, 128, 64, 0, 0}, false, {6.99, 7.79}, {16.42, 16.95}, {0, 0}},
      {{224, 256, 112, 64, 0, 0}, false, {6.59, 7.53}, {14.53, 15.39}, {0, 0}},
      {{192, 256, 96, 64, 0, 0}, false, {6.05, 7.19}, {13.07, 14.04}, {0, 0}},
      {{256, 128, 64, 64, 0, 0}, false, {4.84, 6.41}, {11.32, 12.29}, {0, 0}},
      {{128, 256, 64, 64, 0, 0}, false, {4.53, 5.74}, {9.83, 10.90}, {0, 0}},
      {{128, 128, 64, 32, 0, 0}, false, {3.77, 4.50}, {4.72, 4.60}, {4.29, 4.99}},
      {{64, 128, 32, 64, 0, 0}, false, {2.29, 2.59}, {2.04, 2.03}, {5.90, 6.00}},
      {{64, 64, 32, 32, 0, 0}, false, {1.67, 2.10}, {1.00, 1.05}, {6.00, 6.00}},
      {{96, 64, 48, 32, 2, 0}, true, {3.435, 3.396}, {8.78, 8.436}, {0, 0.369}},
      {{64, 128, 32, 64, 2, 0}, true, {3.70, 3.58}, {9.48, 9.51}, {0, 0}},
      {{128, 64, 64, 32, 2, 0}, true, {3.673, 3.692}, {9.27, 9.236}, {0.253, 0.1}},
      {{96, 128, 48, 64, 2, 0}, true, {4.52, 4.28}, {11.08, 10.91}, {0, 0}},
      {{128, 128, 64, 64, 2, 0}, true, {5.24, 5.08}, {12.33, 12.32}, {0, 0}},
      {{160, 128, 80, 64, 2, 0}, true, {5.91, 5.77}, {12.13, 12.24}, {0, 0}},
      {{192, 128, 96, 64, 2, 0}, true, {6.41, 6.03}, {15.03, 14.95}, {0, 0}},
  };
  const int on = K % kBK == 0 ? 1 : 0;
  const Candidate *best = nullptr, *stays = nullptr;
  double best_us = 0, stays_us = 0;
  for (const Candidate& k : kCandidates) {
    const beam_tile_cfg& t = k.cfg;
    const bool is_named = !k.lines && t.block_m == named.block_m && t.block_n == named.block_n && t.wave_n == named.wave_n;
    if (t.wave_m == 128 && t.wave_n == 128 && !is_named) continue;
    const int tiles_m = (M + t.block_m - 1) / t.block_m, tiles_n = (N + t.block_n - 1) / t.block_n;
    if (tiles_n > 64 || k.rate[on] == 0) continue;
    if (!k.lines) {
      beam_tile_cfg c;
      const KernelSet* ks;
      if (resolve_cfg(&t, M, N, K, &c, &ks) || !ln_fused_applies_on(c, *ks, N, kNumXcd * 32)) continue;
    }
    const int bands_per_round = kNumXcd * 32 / tiles_n;
    const double wide = k.lines && t.block_n == 64 && tiles_n > 20 ? 0.00125 * t.block_m * (tiles_n - 20) : 0;
    const double us = k.launch[on] + (double)((tiles_m + bands_per_round - 1) / bands_per_round) *
                                         (k.round[on] + wide + 2.0e-6 * t.block_m * t.block_n * (double)(((long)K + kBK - 1) / kBK * kBK) / k.rate[on]);
    if (!best || us < best_us) best = &k, best_us = us;
    if (is_named) stays = &k, stays_us = us;
  }
  if (!best || (stays && best_us > 0.96 * stays_us)) return LineChoice{named, false};
  LineChoice c = {best->cfg, best->lines};
  c.cfg.group_m = default_group_m(c.cfg.block_m, c.cfg.block_n);
  return c;
}

// The order of a GEMM+LayerNorm launch without padding (band_order_tile's group_n): plain ids, or groups of G bands where what
// the XCDs fetch, 8 / G of all rows and G times all columns, becomes less by a fifth; plain ids fetch 8 times the rows and, where
// 8 does not divide a band's column tiles, 8 times the columns.  A group is 64 workgroups at most, as a band is, 8 on each XCD.  us, plain -> so,
// in the tiles of gemm_kwave.h: 1713 x 288 x 6992 36.9 -> 21.7 (G = 4), 39 x 3680 x 7808 30.5 -> 19.1 (1), 281 x 1696 x 1880
// 16.2 -> 11.1 (1), 524 x 1440 x 3080 24.0 -> 17.9 (2), 130 x 712 x 2240 9.6 -> 6.8 (1), over 90 shapes, K from 500 to 8192, 10%
// on average; in larger ones 690 x 2904 x 5696 54.3 -> 35.4, 5161 x 1128 x 2408 47.0 -> 33.6, 2702 x 2368 x 2752 46.7 -> 38.3,
// 3959 x 419 x 424 13.9 -> 10.9, over 150 shapes 5%.  Where little is filled into LDS in all (7 Mi elements, under a short sum 12)
// the fabric is no bound, and a few instructions in front of the first load are 0.1 us (28 x 264 x 3008 6.1, 6.2; 2464 x 416 x
// 256 8.6, 8.8); nor is it for two bands of the larger tiles (84 x 5128 x 2264 20.5, 20.9).
//
// More tiles than the device holds at once: the workgroups of the group that a round cuts wait for the next one, each on its CU,
// and a longer group has more of them.  506 tiles of 224 x 256 over 256 CUs (4767 x 5736) are two rounds band after band (22 of 23: 3 wait,
// 253 start) and three in groups of two (26 wait).  So groups no longer than take the rounds of plain ids.  us in three sets of
// operands, plain ids, G = 1, 2 (4): 4755 x 5384 x 1368 84.2, 82.0, 112.9; 3283 x 6480 x 680 53.6, 51.1, 70.7; 6539 x 4352 x 1440 92.0, 83.8, 109.5;
// 7779 x 3496 x 256 44.6, 42.3, 43.7 (60.0); with the same rounds 6201 x 4672 x 2024 124.7, 117.5, 114.7.  Over 479 shapes of more than
// 256 tiles the choice was 5.6% behind the best G on average and 42% at worst, and is 0.2% and 3%.
static int order_rounds(int tiles, int group, int slots) {
  int rounds = 0, waiting = 0;
  for (int done = 0; done < tiles; ++rounds, waiting = done % group) done += std::max(1, slots - waiting);
  return rounds;
}
// slots: workgroups that the device holds at once.
static int band_group(int M, int N, int K, int rows, int cols, int slots) {
  const int tiles_m = (M + rows - 1) / rows, tiles_n = (N + cols - 1) / cols;
  if (tiles_m < (rows * cols > 64 * 64 ? 3 : 2) || (double)tiles_m * tiles_n * (rows + cols) * K < (K < 1024 ? 12e6 : 7e6)) return -1;
  const int rounds = order_rounds(tiles_m * tiles_n, tiles_n, slots);
  double most = 0.8 * (8.0 * M + (tiles_n % 8 ? 8.0 : 1.0) * N);
  int order = -1;
  for (int lg = 0; lg <= 3 && (1 << lg) <= tiles_m && (lg == 0 || tiles_n << lg <= 64); ++lg) {
    const double fetched = (8.0 * M) / (1 << lg) + (double)N * (1 << lg);
    if (fetched <= most && order_rounds(tiles_m * tiles_n, tiles_n << lg, slots) <= rounds) order = -2 - lg, most = fetched;
  }
  return order;
}

// The workgroup order of a GEMM+LayerNorm launch of the tiled kernels: group_m and group_n of band_order_tile, and the grid (returned).
// per_cu: workgroups that a CU holds at once (one of the tiles by whole lines and of gemm_w4.h's).
// Band groups: XCD x owns group_n columns of group_m bands; 8 * group_n covers a whole band and
// group_m * group_n workgroups fit the 32 CUs of an XCD even at one workgroup per CU
// ... or, when a band is short enough, whole bands per XCD (tile_map.h: band_xcd_tile)
//     if that fills every XCD, takes no more rounds of workgroups than the spread order and
//     streams no more operand panels through an XCD's L2 per round (bands + columns it touches;
//     measured: 16384 x 2048 x 2048, 4 + 8 against 32 + 1 panels, 112 against 120 us;
//     8192 x 8192 x 4096, 1 + 32 against 8 + 4, 419 against 400 us; 4096^3, 18 either way, 104.1
//     against 104.8 us)
// ... or, where those two orders' padding costs rounds of workgroups (20 column tiles are 3 per XCD on
//     seven XCDs and none on the eighth: 3000 x 5000 x 2000 in 256 x 256 tiles puts 36 workgroups on six
//     XCDs of 32 CUs), band after band with no padding: id = band * tiles_n + column, which the hardware's
//     round-robin deals out evenly.
//     So too with one column per XCD, of which every one fetches all rows and 8 - tiles_n do nothing, where groups of bands
//     (band_group) fetch less: 3061 x 384 x 1384 in 96 x 64 tiles by whole lines 17.9 -> 10.9 us, 2382 x 432 x 2600 22.5 -> 16.3,
//     3559 x 920 x 816 in 128 x 128 tiles 17.3 -> 14.8, 5240 x 1688 x 5656 in 192 x 256 117 -> 104; 48 shapes 0.53 to 1.01 of the
//     time.  (With two columns and more 0.9 to 1.07.)
// All three keep a band's workgroups together in id order, so a launch that gets only part of the device
// still finishes band by band.  (The plain kernels' raster order streams fewer operand bytes into the L2s
// when the whole grid is one round -- 4096^3: 204 against 303 MB, in the same time -- but loses exactly that.)
static unsigned ln_order(GemmParams* p, int M, int N, int K, const beam_tile_cfg& c, bool w4, int per_cu) {
  p->group_n = (p->tiles_n + kNumXcd - 1) / kNumXcd;
  p->group_m = 32 / p->group_n;
  if (p->group_m > p->tiles_m) p->group_m = p->tiles_m;
  const int bx = p->tiles_n <= 32 ? 32 / p->tiles_n : 0;
  const int rounds_spread = (p->tiles_m + p->group_m - 1) / p->group_m;
  const bool whole_bands = bx > 0 && p->tiles_m >= kNumXcd * bx && (p->tiles_m + kNumXcd * bx - 1) / (kNumXcd * bx) <= rounds_spread &&
                           bx + p->tiles_n <= p->group_m + p->group_n;
  const int rounds_grouped = whole_bands ? (p->tiles_m + kNumXcd * bx - 1) / (kNumXcd * bx) : rounds_spread;
  const long per_xcd = ((long)p->tiles_m * p->tiles_n + kNumXcd - 1) / kNumXcd;
  const int bands_grouped = band_group(M, N, K, c.block_m, c.block_n, kNumXcd * 32 * per_cu);
  if ((per_xcd + 31) / 32 < rounds_grouped || (p->group_n == 1 && !whole_bands && !w4 && bands_grouped < -1)) {
    p->group_n = bands_grouped;
    return (unsigned)(p->tiles_m * p->tiles_n);
  }
  if (whole_bands) {
    p->group_n = 0;
    p->group_m = bx;
    return (unsigned)band_xcd_grid(p->tiles_m, p->tiles_n, bx);
  }
  return (unsigned)band_block_grid(p->tiles_m, p->group_m, p->group_n);
}

// What a GEMM+LayerNorm call does and the workspace it needs: one function, so that the entry point and the
// workspace queries cannot disagree.
//   plain     the problem is outside what the tiled kernels take (K below 8 or beyond a descriptor, gamma or beta not
//             8-byte aligned): plain GEMM into fp32 X, then a row-wise LayerNorm
//   unaligned rows of A or B off 16 bytes or Y off 8 (rows_unaligned; K % 8 != 0 implies it).  The tiled kernels take
//             them; where they would refuse the call (a tile that is not compiled, BEAM_LN_FUSED where it does not apply)
//             it runs on the plain ones, which never refused such operands
//   capturing the stream is being captured: AUTO then means two passes (a replayed graph may share the device with
//             other work, which the fused kernel's residency argument does not cover); an explicit FUSED is honoured
//   wide_io   Y, gamma and beta are 16-byte aligned (the 4-wavefront kernel's vector accesses)
struct LnPlan {
  enum Kind { kPlain, kTwoPass, kFused } kind;
  beam_tile_cfg c;
  const KernelSet* ks;
  bool w4;    // fused, on the kernel of gemm_w4.h
  bool lines;  // fused, in a tile whose fills take whole lines (ks then says nothing)
  KwPlan kw;  // fused, on the kernel of gemm_kwave.h if kw.rows != 0 (c and ks then say nothing)
  size_t need;
};
// The library's own choice of gemm_kwave.h for the one-kernel form (its workgroups must be resident at once, and its order of
// bands is made for 8 XCDs of 32 CUs).
static KwPlan ln_kw_plan(int M, int N, int K, const beam_tile_cfg* cfg, int mode) {
  if (cfg || mode == BEAM_LN_TWOPASS || g_dev.cus != kNumXcd * 32) return KwPlan{0, 0, 0, false};
  return kw_plan(M, N, K, false, true, false, kOnLines, g_dev.cus);
}
static int ln_plan(int M, int N, int K, const beam_tile_cfg* cfg, int mode, bool plain, bool unaligned, bool capturing, bool wide_io,
                   LnPlan* out) {
  out->ks = nullptr;
  out->w4 = false;
  out->lines = false;
  out->kw = KwPlan{0, 0, 0, false};
  if (plain) {
    out->kind = LnPlan::kPlain;
    out->need = ln_generic_need(M, N);
    return BEAM_OK;
  }
  if (capturing && mode == BEAM_LN_AUTO) mode = BEAM_LN_TWOPASS;
  out->kw = ln_kw_plan(M, N, K, cfg, mode);
  if (out->kw.rows) {
    out->kind = LnPlan::kFused;
    out->need = ln_fused_need(M, N, out->kw.rows, out->kw.cols);
    return BEAM_OK;
  }
  int rc = ln_resolve_cfg(cfg, M, N, K, mode, &out->c, &out->ks);
  beam_tile_cfg& c = out->c;
  if ((unaligned || K % 8 != 0) && (rc || (mode == BEAM_LN_FUSED && !ln_fused_applies(c, *out->ks, N)))) {
    out->kind = LnPlan::kPlain;
    out->need = ln_generic_need(M, N);
    return BEAM_OK;
  }
  if (rc) return rc;
  if (!cfg && mode != BEAM_LN_TWOPASS && !unaligned && K >= 8 && K % 8 == 0 && g_dev.cus == kNumXcd * 32) {
    const LineChoice t = ln_line_tile(M, N, K, c);
    if (t.lines) {
      c = t.cfg;
      out->ks = nullptr;
      out->lines = true;
      out->kind = LnPlan::kFused;
      out->need = ln_fused_need(M, N, c.block_m, c.block_n);
      return BEAM_OK;
    }
    c = t.cfg;
    if ((rc = resolve_cfg(&c, M, N, K, &c, &out->ks))) return rc;
  }
  if (mode == BEAM_LN_FUSED && !ln_fused_applies(c, *out->ks, N))
    return fail(BEAM_ERR_UNSUPPORTED, "fused LayerNorm: needs a device of %d CUs and at most 64 column tiles (N=%d, block_n=%d, %d CUs)",
                kNumXcd * 32, N, c.block_n, g_dev.cus);
  mode = ln_resolve_mode(mode, c, *out->ks, N);
  // The 256 x 256 tile runs on the kernel of gemm_w4.h where that one's preconditions hold (asked for by
  // name, or as the library's own choice); where they do not, the library's own choice falls back to the
  // 8-wavefront tile of the same shape.
  const bool w4_fits = mode == BEAM_LN_FUSED && c.pipeline == 0 && c.block_m == 256 && c.block_n == 256 && K % kBK == 0 &&
                       K >= kW4MinK && N % 8 == 0 && N <= (1 << 21) && wide_io;
  if (!cfg && !w4_fits && c.block_m == 256 && c.block_n == 256 && c.wave_m == 128 && c.wave_n == 128) {
    c.wave_n = 64;
    if ((rc = resolve_cfg(&c, M, N, K, &c, &out->ks))) return rc;
  }
  out->w4 = w4_fits && c.wave_m == 128 && c.wave_n == 128;
  out->kind = mode == BEAM_LN_FUSED ? LnPlan::kFused : LnPlan::kTwoPass;
  out->need = ln_workspace_need(M, N, c, mode);
  return BEAM_OK;
}

// The plan of a call: the above for its operands and its workspace.  Unaligned rows have always got by with room for fp32 X
// on 16 bytes; a workspace that has that, and not what the tiled kernels ask for, still means the plain ones.
static int ln_plan_call(const void* A, const void* B, const void* gamma, const void* beta, const void* Y, int M, int N, int K,
                        const beam_tile_cfg* cfg, int mode, bool generic, bool capturing, const void* ws, size_t ws_bytes, LnPlan* out) {
  const bool unaligned = rows_unaligned(A, B, Y, K);
  const bool wide_io = (((uintptr_t)Y | (uintptr_t)gamma | (uintptr_t)beta) & 15) == 0;
  if (int rc = ln_plan(M, N, K, cfg, mode, ln_is_generic(generic, gamma, beta), unaligned, capturing, wide_io, out)) return rc;
  if (unaligned && out->kind != LnPlan::kPlain && (!ws || ws_bytes < out->need || ((uintptr_t)ws & 255) != 0))
    return ln_plan(M, N, K, cfg, mode, true, unaligned, capturing, wide_io, out);
  return BEAM_OK;
}

// Enough for beam_gemmrc_ln_ex(M, N, K, cfg, mode) with A, B, Y on 16 bytes and gamma, beta on 8.  AUTO covers both forms it
// can resolve to (one kernel eagerly, two passes under stream capture and as the retry of beam_gemmrc_ln_checked); two
// passes need at least what the plain kernels do.
size_t beam_gemmrc_ln_workspace_bytes_for(int M, int N, int K, const beam_tile_cfg* cfg, int mode) {
  if (M <= 0 || N <= 0 || K < 0) return 0;
  if ((K > 0 && K < 8) || K > kMaxK) return ln_generic_need(M, N);
  (void)beam_init();  // AUTO depends on the device
  LnPlan eager, captured;
  if (ln_plan(M, N, K, cfg, mode, false, false, false, true, &eager)) return 0;
  if (mode != BEAM_LN_AUTO) {
    // rows off 16 bytes have a tile of their own choice, and more column tiles perhaps
    LnPlan off;
    if (ln_plan(M, N, K, cfg, mode, false, true, false, true, &off) == BEAM_OK && off.kind == eager.kind && off.need > eager.need) return off.need;
    return eager.need;
  }
  if (ln_plan(M, N, K, cfg, mode, false, false, true, true, &captured)) return eager.need;
  return eager.need > captured.need ? eager.need : captured.need;
}

// Enough for any call with these M, N, cfg and mode: every K, every alignment, captured or not.
size_t beam_gemmrc_ln_workspace_bytes_ex(int M, int N, const beam_tile_cfg* cfg, int mode) {
  if (M <= 0 || N <= 0) return 0;
  size_t need = ln_generic_need(M, N);  // K % 8 != 0, operands aligned to an element only
  auto take = [&](size_t n) { need = n > need ? n : need; };
  // a given tile does not depend on K
  if (cfg) {
    take(beam_gemmrc_ln_workspace_bytes_for(M, N, 64, cfg, mode));
    return need;
  }
  // Without a tile the library picks one from (M, N, K), and K is not known here: the largest need over
  // every tile it can pick, in every form `mode` can resolve to.
  (void)beam_init();
  for (int i = 0; i < beam_num_configs(); ++i) {
    beam_tile_cfg c;
    const KernelSet* ks;
    if (beam_get_config(i, &c) || resolve_cfg(&c, M, N, 64, &c, &ks)) continue;
    take(ln_workspace_need(M, N, c, ln_resolve_mode(mode, c, *ks, N)));
    if (mode == BEAM_LN_AUTO) take(ln_workspace_need(M, N, c, BEAM_LN_TWOPASS));
  }
  if (const KwPlan kw = ln_kw_plan(M, N, 1024, cfg, mode); kw.rows) take(ln_fused_need(M, N, kw.rows, kw.cols));
  if (mode != BEAM_LN_TWOPASS) {
#define BEAM_LINES(BM, BN, S, KG, FORM) if ((N + BN - 1) / BN <= 64) take(ln_fused_need(M, N, BM, BN));
    BEAM_FOR_EACH_LINES_TILE(BEAM_LINES)
#undef BEAM_LINES
  }
  return need;
}

size_t beam_gemmrc_ln_workspace_bytes(int M, int N, const beam_tile_cfg* cfg) {
  return beam_gemmrc_ln_workspace_bytes_ex(M, N, cfg, BEAM_LN_AUTO);
}

size_t beam_dbg_ln_plan_bytes(int M, int N, int K, const beam_tile_cfg* cfg, int mode, int plain, int capturing, int wide_io) {
  LnPlan plan;
  if (M <= 0 || N <= 0 || K < 0 || ln_plan(M, N, K, cfg, mode, plain != 0 || (K > 0 && K < 8) || K > kMaxK, false, capturing != 0,
                                                     wide_io != 0, &plan)) return 0;
  return plan.need;
}

int beam_dbg_small_tile(int op, int M, int N, int K, int row_starts, int* rows, int* cols, int* waves, int* whole_lines) {
  if (op < 0 || op > 3 || row_starts < kAnywhere || row_starts > kOnLines || M <= 0 || N <= 0 || K < 0 || !rows || !cols || !waves || !whole_lines)
    return fail(BEAM_ERR_INVALID, "bad argument");
  const RowStarts at = (RowStarts)row_starts;
  const int cus = g_dev.cus > 0 ? g_dev.cus : 256;
  KwPlan kw = {0, 0, 0, false};
  if (op == 0) kw = kw_plan(M, N, K, false, false, true, at, cus);
  if (op == 1 && N >= 8) kw = kw_plan(M, N, K, true, false, true, at, cus);
  if (op == 2) kw = splitk_kw_plan(M, N, K, nullptr, 0, at);
  if (op == 3 && cus == kNumXcd * 32) kw = kw_plan(M, N, K, false, true, false, at, cus);
  *rows = kw.rows;
  *cols = kw.cols;
  *waves = kw.waves;
  *whole_lines = kw.shift ? 1 : 0;
  return BEAM_OK;
}

int beam_dbg_off_lines_tile(int M, int N, int K, beam_tile_cfg* cfg, int* whole_lines) {
  if (M <= 0 || N <= 0 || K < 8 || !cfg || !whole_lines) return fail(BEAM_ERR_INVALID, "null pointer or empty problem");
  const LineChoice t = off_lines_tile(M, N, K, g_dev.cus > 0 ? g_dev.cus : 256);
  *cfg = t.cfg;
  *whole_lines = t.lines ? 1 : 0;
  return BEAM_OK;
}

int beam_dbg_nn_off_lines_tile(int M, int N, int K, const beam_tile_cfg* named, beam_tile_cfg* cfg, int* whole_lines) {
  if (M <= 0 || N < 8 || K < 8 || !named || !cfg || !whole_lines) return fail(BEAM_ERR_INVALID, "null pointer or empty problem");
  const LineChoice t = nn_off_lines_tile(M, N, K, *named, g_dev.cus > 0 ? g_dev.cus : 256);
  *cfg = t.cfg;
  *whole_lines = t.lines ? 1 : 0;
  return BEAM_OK;
}

int beam_dbg_set_splitk_self_reduce(int on) {
  g_splitk_self_reduce.store(on != 0);
  return BEAM_OK;
}

int beam_set_ln_walk(int on) {
  g_ln_no_walk.store(on ? 0 : 1);
  return BEAM_OK;
}

int beam_dbg_assume_compute_units(int compute_units) {
  std::lock_guard<std::mutex> lk(g_dev_mu);
  if (g_dev.status == BEAM_OK) return fail(BEAM_ERR_INVALID, "a device has been probed: its own CU count stands");
  g_dev.cus = compute_units;
  return BEAM_OK;
}

int beam_gemmrc_ln_ex(const void* A, const void* B, const void* gamma, const void* beta, float eps, void* Y,
                      int M, int N, int K, int dtype, const beam_tile_cfg* cfg, int mode, void* ws,
                      size_t ws_bytes, void* stream) {
  bool generic;
  int rc = check_problem(A, B, Y, M, N, K, dtype, &generic);
  if (rc) return rc;
  if (M == 0 || N == 0) return BEAM_OK;
  if (!gamma || !beta) return fail(BEAM_ERR_INVALID, "null gamma/beta");
  if (((uintptr_t)gamma | (uintptr_t)beta) & 1) return fail(BEAM_ERR_INVALID, "gamma and beta must be aligned to their 16-bit elements");
  if (!(eps >= 0.0f)) return fail(BEAM_ERR_INVALID, "eps must be >= 0");
  if (mode < BEAM_LN_AUTO || mode > BEAM_LN_FUSED) return fail(BEAM_ERR_INVALID, "unknown LayerNorm mode %d", mode);
  if ((rc = beam_init())) return rc;
  hipStream_t st = (hipStream_t)stream;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (st != nullptr) (void)hipStreamIsCapturing(st, &capturing);
  LnPlan plan;
  if ((rc = ln_plan_call(A, B, gamma, beta, Y, M, N, K, cfg, mode, generic, capturing != hipStreamCaptureStatusNone, ws, ws_bytes, &plan)))
    return rc;
  const size_t need = plan.need;
  if (!ws || ws_bytes < need)
    return fail(BEAM_ERR_WORKSPACE, "GEMM+LayerNorm needs %zu bytes of workspace, got %zu", need, ws_bytes);
  if (plan.kind == LnPlan::kPlain) {
    // What the tiled kernels cannot take: the plain GEMM into fp32 X, then a row-wise LayerNorm (whatever mode was named).
    if ((uintptr_t)ws & 15) return fail(BEAM_ERR_UNSUPPORTED, "workspace must be 16-byte aligned");
    if (K == 0) BEAM_HIP(launch_fill_floats((float*)ws, (size_t)M * N, 0.0f, st));
    else BEAM_HIP(launch_generic_gemm(A, B, ws, M, N, K, dtype, false, true, st));
    BEAM_HIP(launch_ln_rows((const float*)ws, gamma, beta, Y, M, N, eps, dtype, st));
    return BEAM_OK;
  }
  if ((uintptr_t)ws & 255) return fail(BEAM_ERR_UNSUPPORTED, "workspace must be 256-byte aligned");
  if (plan.kw.rows) {
    KwPlan kw = plan.kw;
    kw.shift = kw_plan(M, N, K, false, true, false, row_starts(A, B, K, false), g_dev.cus).shift;
    KwLnParams p;
    kw_params(&p, kw, A, B, Y, M, N, K);
    p.divs = band_order_divs(p.tiles_n, 1, p.tiles_n <= kKwLnShortBand ? -1 : band_group(M, N, K, kw.rows, kw.cols, p.tiles_m * p.tiles_n));
    if (capturing != hipStreamCaptureStatusNone) BEAM_HIP(launch_ln_replay_bump((int*)ws, st));
    char* sets = (char*)ws + ln_fused_header_bytes();
    p.stats = (float*)sets;
    p.next_stats = (float*)(sets + ln_fused_set_bytes(p.tiles_m, p.tiles_n, kw.rows));
    p.timeout_flag = (int*)ws;
    p.host_timeout = g_ln_host_timeout;
    p.gamma = gamma;
    p.beta = beta;
    p.ln_nonce = g_ln_nonce.fetch_add(1, std::memory_order_relaxed) + 1;
    p.eps = eps;
    p.spin_limit = g_ln_spin_limit.load();
    BEAM_HIP(dtype == BEAM_F16 ? launch_gemm_kwave_ln<_Float16>(kw, p, st) : launch_gemm_kwave_ln<__bf16>(kw, p, st));
    return BEAM_OK;
  }
  const beam_tile_cfg& c = plan.c;
  const KernelSet* ks = plan.ks;
  GemmParams p = base_params(A, B, M, N, K, c);
  // K == 0: the kernels run with an empty K range and produce x = 0, i.e. y = beta.
  if (plan.kind == LnPlan::kFused) {
    p.C = Y;
    p.c_store = store_kind(c, plan.lines ? 4 : ks->threads / 64, plan.w4, Y, M, N, K, true);
    // Launches that share a workspace must be ordered (same stream): overlapping ones would race on the sets.
    const size_t set_bytes = ln_fused_set_bytes(p.tiles_m, p.tiles_n, c.block_m);
    float* sets = (float*)((char*)ws + ln_fused_header_bytes());
    // A recorded launch repeats its arguments on every replay: the counter in the header then makes the tag new.
    if (capturing != hipStreamCaptureStatusNone) BEAM_HIP(launch_ln_replay_bump((int*)ws, st));
    p.ln_nonce = g_ln_nonce.fetch_add(1, std::memory_order_relaxed) + 1;
    p.stats = sets;
    p.next_stats = (float*)((char*)sets + set_bytes);
    p.timeout_flag = (int*)ws;
    p.host_timeout = g_ln_host_timeout;
    p.gamma = gamma;
    p.beta = beta;
    p.eps = eps;
    p.spin_limit = g_ln_spin_limit.load();
    const unsigned grid = ln_order(&p, M, N, K, c, plan.w4, plan.lines || plan.w4 ? 1 : kLdsBytes / (c.pipeline ? ks->lds_bytes_shallow : ks->lds_bytes));
    // the band orders' divisors as multipliers (tile_map.h: band_order_divs)
    p.divs = band_order_divs(p.tiles_n, p.group_m, p.group_n);
    if (plan.w4) {
      // More ids than CUs: one workgroup per CU walks the ids w, w + CUs, ... of the same order, with the next
      // tile's first operand tiles arriving while the band's statistics are exchanged (gemm_w4.h says why no
      // chain of waits closes: a band's ids lie within fewer than 256 of each other in all three orders).  The
      // walking form keeps the epilogue's scratch inside the two LDS slots the operand ring leaves free, which
      // holds a band of up to 32 column tiles; wider bands keep one workgroup per tile.
      p.ln_ids = (int)grid;
      const unsigned cus = (unsigned)g_dev.cus;
      const bool walk = grid > cus && p.tiles_n <= kW4LnCompactTiles && !g_ln_no_walk.load(std::memory_order_relaxed);
      BEAM_HIP(launch_gemm_w4_ln(p, dtype, dim3(walk ? cus : grid, 1, 1), st));
      return BEAM_OK;
    }
    if (plan.lines) {
      BEAM_HIP(dtype == BEAM_F16 ? launch_gemm_lines_ln<_Float16>(c.block_m, c.block_n, p, dim3(grid, 1, 1), st)
                                 : launch_gemm_lines_ln<__bf16>(c.block_m, c.block_n, p, dim3(grid, 1, 1), st));
      return BEAM_OK;
    }
    BEAM_HIP(ks->launch[dtype][kEpiLnFused][c.pipeline](p, dim3(grid, 1, 1), st));
    return BEAM_OK;
  }
  p.ws = (float*)ws;
  p.stats = (float*)((char*)ws + align_up((size_t)M * N * sizeof(float), 256));
  BEAM_HIP(ks->launch[dtype][kEpiLnStats][c.pipeline](p, dim3((unsigned)(p.tiles_m * p.tiles_n), 1, 1), st));
  BEAM_HIP(launch_ln_apply(p.ws, p.stats, gamma, beta, Y, M, N, p.tiles_n, c.block_n, eps, dtype, st));
  return BEAM_OK;
}

int beam_gemmrc_ln(const void* A, const void* B, const void* gamma, const void* beta, float eps, void* Y,
                   int M, int N, int K, int dtype, const beam_tile_cfg* cfg, void* ws, size_t ws_bytes,
                   void* stream) {
  return beam_gemmrc_ln_ex(A, B, gamma, beta, eps, Y, M, N, K, dtype, cfg, BEAM_LN_AUTO, ws, ws_bytes, stream);
}

int beam_gemmrc_ln_checked(const void* A, const void* B, const void* gamma, const void* beta, float eps, void* Y,
                           int M, int N, int K, int dtype, const beam_tile_cfg* cfg, void* ws, size_t ws_bytes,
                           void* stream, int* fell_back) {
  if (fell_back) *fell_back = 0;
  hipStream_t st = (hipStream_t)stream;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (st != nullptr) (void)hipStreamIsCapturing(st, &capturing);
  // (captured: AUTO is two passes, which wait for nothing; a stream being captured cannot be waited for anyway)
  int rc = beam_gemmrc_ln_ex(A, B, gamma, beta, eps, Y, M, N, K, dtype, cfg, BEAM_LN_AUTO, ws, ws_bytes, stream);
  if (rc || capturing != hipStreamCaptureStatusNone || M == 0 || N == 0) return rc;
  bool generic;
  (void)check_problem(A, B, Y, M, N, K, dtype, &generic);
  LnPlan plan;
  if (ln_plan_call(A, B, gamma, beta, Y, M, N, K, cfg, BEAM_LN_AUTO, generic, false, ws, ws_bytes, &plan) || plan.kind != LnPlan::kFused)
    return BEAM_OK;  // nothing in the call waits for anything
  if (const volatile unsigned* word = g_ln_host_timeout; word && *word == 0) {  // (set once: the header's reader waits by itself)
    BEAM_HIP(wait_for_stream(st));
    if (*word == 0) return BEAM_OK;
  }
  int timed_out = 0;
  if ((rc = beam_gemmrc_ln_timed_out(ws, stream, &timed_out))) return rc;
  if (!timed_out) return BEAM_OK;
  if (fell_back) *fell_back = 1;
  if ((rc = beam_gemmrc_ln_ex(A, B, gamma, beta, eps, Y, M, N, K, dtype, cfg, BEAM_LN_TWOPASS, ws, ws_bytes, stream))) return rc;
  BEAM_HIP(hipStreamSynchronize(st));
  return BEAM_OK;
}

int beam_gemmrc_ln_workspace_reset(const void* ws) {
  if (!ws) return fail(BEAM_ERR_INVALID, "null workspace");
  // Forgets a recorded time-out (never needed).  The replay counter behind these words stays: it is part of the tag
  // of captured launches, and a counter that went back could hand a replay the tag of an earlier one, whose
  // statistics words would then pass for published.
  static_assert(kLnHdrTimeout < 3 && kLnHdrMagic < 3 && kLnHdrLaunchTag < 3 && kLnHdrReplay == 3, "header words");
  BEAM_HIP(hipMemset(const_cast<void*>(ws), 0, 3 * sizeof(int)));
  return BEAM_OK;
}

int beam_set_ln_spin_limit(int polls) {
  if (polls < -1) return fail(BEAM_ERR_INVALID, "spin limit must be >= -1");
  g_ln_spin_limit.store(polls);
  return BEAM_OK;
}

int beam_gemmrc_ln_timed_out(const void* ws, void* stream, int* timed_out) {
  if (!ws || !timed_out) return fail(BEAM_ERR_INVALID, "null argument");
  BEAM_HIP(hipStreamSynchronize((hipStream_t)stream));
  int hdr[4] = {0, 0, 0, 0};
  BEAM_HIP(hipMemcpy(hdr, ws, sizeof hdr, hipMemcpyDeviceToHost));
  // the header speaks of a fused launch at all, and the launch that gave up is the latest one
  *timed_out = hdr[kLnHdrMagic] == kLnMagic && hdr[kLnHdrLaunchTag] != 0 && hdr[kLnHdrTimeout] == hdr[kLnHdrLaunchTag];
  return BEAM_OK;
}

// BEAM_OP_PROBE_SPLITK_LOADS: the launch of beam_gemmrc_splitk's partial kernel, resolved the same way.
static int probe_splitk_loads(const beam_problem* q, const beam_tile_cfg* cfg, hipStream_t st) {
  bool generic;
  int rc = check_problem(q->A, q->B, q->C, q->M, q->N, q->K, q->dtype, &generic);
  if (rc) return rc;
  if ((rc = beam_init())) return rc;
  if (generic || q->dtype != BEAM_F16 || q->M == 0 || q->N == 0 || q->K == 0)
    return fail(BEAM_ERR_UNSUPPORTED, "the load probe is built for fp16 problems of the tiled kernels");
  beam_tile_cfg c;
  const KernelSet* ks;
  if ((rc = resolve_cfg(cfg, q->M, q->N, q->K, &c, &ks, q->split_k > 0 ? q->split_k : 0))) return rc;
  const bool built = c.pipeline == 2 && c.block_m == 64 && ((c.block_n == 128 && c.wave_m == 32 && c.wave_n == 64) ||
                                                            (c.block_n == 64 && c.wave_m == 32 && c.wave_n == 32));
  if (!built) return fail(BEAM_ERR_UNSUPPORTED, "the load probe is built for the deep 64x128 (wave 32x64) and 64x64 (wave 32x32) tiles");
  const int s = effective_split(q->M, q->N, q->K, c, q->split_k);
  GemmParams p = base_params(q->A, q->B, q->M, q->N, q->K, c);
  p.ws = (float*)q->ws;  // never written
  p.k_slice = split_k_len(q->K, s);
  p.splits = s;
  BEAM_HIP(launch_probe_splitk_loads(p, c.block_m, c.block_n, dim3((unsigned)(p.tiles_m * p.tiles_n * s), 1, 1), st));
  return BEAM_OK;
}

int beam_bench(int op, const beam_problem* q, const beam_tile_cfg* cfg, int warmup, int iters, void* stream,
               float* avg_ms) {
  if (!q || !avg_ms || iters < 1 || warmup < 0) return fail(BEAM_ERR_INVALID, "bad bench arguments");
  auto once = [&]() -> int {
    switch (op) {
      case BEAM_OP_GEMM:
        return beam_gemmrc(q->A, q->B, q->C, q->M, q->N, q->K, q->dtype, cfg, stream);
      case BEAM_OP_SPLITK:
        return beam_gemmrc_splitk(q->A, q->B, q->C, q->M, q->N, q->K, q->dtype, cfg, q->split_k, q->ws,
                                  q->ws_bytes, stream);
      case BEAM_OP_GEMM_LN:
        return beam_gemmrc_ln_ex(q->A, q->B, q->gamma, q->beta, q->eps, q->C, q->M, q->N, q->K, q->dtype, cfg, q->ln_mode,
                                 q->ws, q->ws_bytes, stream);
      case BEAM_OP_GEMM_SILU:
        return beam_parallel_gemmrc_silu(q->A, q->B, q->C, q->M, q->N, q->K, q->side_x, q->side_y, q->side_count,
                                         q->dtype, cfg, stream);
      case BEAM_OP_MATMUL_NN:
        return beam_matmul_nn(q->A, q->B, q->C, q->M, q->N, q->K, q->dtype, cfg, stream);
      case BEAM_OP_SILU:
        return beam_silu(q->side_x, q->side_y, q->side_count, q->dtype, stream);
      case BEAM_OP_PROBE_EMPTY:
      case BEAM_OP_PROBE_EMPTY_PAIR: {
        int rc = beam_init();
        if (rc) return rc;
        BEAM_HIP(launch_empty(256, 256, (hipStream_t)stream));
        if (op == BEAM_OP_PROBE_EMPTY_PAIR) BEAM_HIP(launch_empty(1024, 64, (hipStream_t)stream));
        return BEAM_OK;
      }
      case BEAM_OP_PROBE_SPLITK_LOADS:
        return probe_splitk_loads(q, cfg, (hipStream_t)stream);
      case BEAM_OP_PROBE_LN_APPLY: {
        // the second kernel of a two-pass GEMM+LayerNorm alone, on the fp32 X and statistics a two-pass call left in ws
        int rc = beam_init();
        if (rc) return rc;
        LnPlan plan;
        if ((rc = ln_plan(q->M, q->N, q->K, cfg, BEAM_LN_TWOPASS, q->K % 8 != 0 || q->K > kMaxK, false, false, true, &plan))) return rc;
        if (plan.kind != LnPlan::kTwoPass || !q->ws || q->ws_bytes < plan.need) return fail(BEAM_ERR_WORKSPACE, "needs the workspace of a two-pass call");
        const float* stats = (const float*)((const char*)q->ws + align_up((size_t)q->M * q->N * sizeof(float), 256));
        BEAM_HIP(launch_ln_apply((const float*)q->ws, stats, q->gamma, q->beta, q->C, q->M, q->N, (q->N + plan.c.block_n - 1) / plan.c.block_n,
                                 plan.c.block_n, q->eps, q->dtype, (hipStream_t)stream));
        return BEAM_OK;
      }
      default:
        return fail(BEAM_ERR_INVALID, "unknown op %d", op);
    }
  };
  hipStream_t st = (hipStream_t)stream;
  for (int i = 0; i < warmup; ++i) {
    int rc = once();
    if (rc) return rc;
  }
  hipEvent_t e0, e1;
  BEAM_HIP(hipEventCreate(&e0));
  BEAM_HIP(hipEventCreate(&e1));
  int rc = BEAM_OK;
  hipError_t he = hipEventRecord(e0, st);
  for (int i = 0; i < iters && rc == BEAM_OK && he == hipSuccess; ++i) rc = once();
  if (he == hipSuccess) he = hipEventRecord(e1, st);
  if (he == hipSuccess) he = hipEventSynchronize(e1);
  float ms = 0.0f;
  if (he == hipSuccess) he = hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  if (he != hipSuccess) return hip_fail(he, "event timing");
  *avg_ms = ms / (float)iters;
  return BEAM_OK;
}

int beam_probe_mfma(int dtype, int mfma_shape, int data, int passes, int warmup, int iters, void* stream, float* avg_ms,
                    double* flop_per_launch) {
  if (!avg_ms || iters < 1 || warmup < 0 || passes < 1) return fail(BEAM_ERR_INVALID, "bad probe arguments");
  if (dtype != BEAM_F16 && dtype != BEAM_BF16) return fail(BEAM_ERR_UNSUPPORTED, "dtype %d: only fp16 (0) and bf16 (1)", dtype);
  if (mfma_shape != BEAM_MFMA_16X16X32 && mfma_shape != BEAM_MFMA_32X32X16) return fail(BEAM_ERR_INVALID, "unknown MFMA shape %d", mfma_shape);
  if (data != BEAM_PROBE_DATA_NORMAL && data != BEAM_PROBE_DATA_ZEROS) return fail(BEAM_ERR_INVALID, "unknown data kind %d", data);
  int rc = beam_init();
  if (rc) return rc;
  const int cus = g_dev.cus > 0 && g_dev.cus <= 1024 ? g_dev.cus : 256;
  hipStream_t st = (hipStream_t)stream;
  for (int i = 0; i < warmup; ++i) BEAM_HIP(launch_probe_mfma(dtype, mfma_shape, cus, passes, data == BEAM_PROBE_DATA_ZEROS, st));
  hipEvent_t e0, e1;
  BEAM_HIP(hipEventCreate(&e0));
  BEAM_HIP(hipEventCreate(&e1));
  hipError_t he = hipEventRecord(e0, st);
  for (int i = 0; i < iters && he == hipSuccess; ++i) he = launch_probe_mfma(dtype, mfma_shape, cus, passes, data == BEAM_PROBE_DATA_ZEROS, st);
  if (he == hipSuccess) he = hipEventRecord(e1, st);
  if (he == hipSuccess) he = hipEventSynchronize(e1);
  float ms = 0.0f;
  if (he == hipSuccess) he = hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (he != hipSuccess) return hip_fail(he, "matrix-core probe");
  *avg_ms = ms / (float)iters;
  if (flop_per_launch) *flop_per_launch = (double)cus * 4.0 * (double)passes * 1024.0 * 1024.0;
  return BEAM_OK;
}

int beam_stream_create(void** stream) {
  if (!stream) return fail(BEAM_ERR_INVALID, "null stream pointer");
  int rc = beam_init();
  if (rc) return rc;
  hipStream_t s;
  BEAM_HIP(hipStreamCreate(&s));  // default priority
  *stream = s;
  return BEAM_OK;
}

int beam_stream_destroy(void* stream) {
  BEAM_HIP(hipStreamDestroy((hipStream_t)stream));
  return BEAM_OK;
}

int beam_graph_begin_capture(void* stream) {
  if (!stream) return fail(BEAM_ERR_INVALID, "the default stream cannot be captured");
  BEAM_HIP(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeThreadLocal));
  return BEAM_OK;
}

int beam_graph_end_capture(void* stream, void** graph_exec) {
  if (!graph_exec) return fail(BEAM_ERR_INVALID, "null graph pointer");
  hipGraph_t g = nullptr;
  BEAM_HIP(hipStreamEndCapture((hipStream_t)stream, &g));
  hipGraphExec_t e = nullptr;
  hipError_t err = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (err != hipSuccess) return hip_fail(err, "hipGraphInstantiate");
  *graph_exec = e;
  return BEAM_OK;
}

int beam_graph_launch(void* graph_exec, void* stream) {
  BEAM_HIP(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
  return BEAM_OK;
}

int beam_graph_destroy(void* graph_exec) {
  BEAM_HIP(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
  return BEAM_OK;
}

int beam_event_create(void** event) {
  if (!event) return fail(BEAM_ERR_INVALID, "null event");
  hipEvent_t e;
  BEAM_HIP(hipEventCreate(&e));
  *event = (void*)e;
  return BEAM_OK;
}
int beam_event_record(void* event, void* stream) {
  if (!event) return fail(BEAM_ERR_INVALID, "null event");
  BEAM_HIP(hipEventRecord((hipEvent_t)event, (hipStream_t)stream));
  return BEAM_OK;
}
int beam_event_elapsed_ms(void* start, void* stop, float* ms) {
  if (!start || !stop || !ms) return fail(BEAM_ERR_INVALID, "null event");
  BEAM_HIP(hipEventSynchronize((hipEvent_t)stop));
  BEAM_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return BEAM_OK;
}
int beam_event_destroy(void* event) {
  if (event) BEAM_HIP(hipEventDestroy((hipEvent_t)event));
  return BEAM_OK;
}

int beam_malloc(void** dptr, size_t bytes) {
  if (!dptr) return fail(BEAM_ERR_INVALID, "null dptr");
  *dptr = nullptr;
  if (bytes == 0) return BEAM_OK;
  BEAM_HIP(hipMalloc(dptr, bytes));
  return BEAM_OK;
}
int beam_free(void* dptr) {
  if (dptr) BEAM_HIP(hipFree(dptr));
  return BEAM_OK;
}
int beam_memcpy_h2d(void* dst, const void* src_host, size_t bytes) {
  if (bytes) BEAM_HIP(hipMemcpy(dst, src_host, bytes, hipMemcpyHostToDevice));
  return BEAM_OK;
}
int beam_memcpy_d2h(void* dst_host, const void* src, size_t bytes) {
  if (bytes) BEAM_HIP(hipMemcpy(dst_host, src, bytes, hipMemcpyDeviceToHost));
  return BEAM_OK;
}
int beam_memcpy_d2d(void* dst, const void* src, size_t bytes) {
  if (bytes) BEAM_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
  return BEAM_OK;
}
int beam_memset(void* dptr, int byte, size_t bytes) {
  if (bytes) BEAM_HIP(hipMemset(dptr, byte, bytes));
  return BEAM_OK;
}
int beam_sync(void* stream) {
  BEAM_HIP(hipStreamSynchronize((hipStream_t)stream));
  return BEAM_OK;
}

int beam_host_fill_uniform(void* dst_host, size_t n, int dtype, uint64_t seed, uint64_t tensor_id) {
  if (!dst_host && n) return fail(BEAM_ERR_INVALID, "null destination");
  if (dtype != BEAM_F16 && dtype != BEAM_BF16) return fail(BEAM_ERR_UNSUPPORTED, "dtype %d", dtype);
  uint16_t* out = (uint16_t*)dst_host;
  parallel_for(n, [=](size_t lo, size_t hi) {
    for (size_t i = lo; i < hi; ++i) {
      const uint64_t r = draw(seed, tensor_id, i);
      const float v = (float)(r >> 40) * (1.0f / 8388608.0f) - 1.0f;  // 24 bits -> [-1, 1)
      out[i] = dtype == BEAM_BF16 ? to_bf16_bits(v) : to_f16_bits(v);
    }
  });
  return BEAM_OK;
}

int beam_host_fill_normal(void* dst_host, size_t n, int dtype, uint64_t seed, uint64_t tensor_id, float mean,
                          float scale) {
  if (!dst_host && n) return fail(BEAM_ERR_INVALID, "null destination");
  if (dtype != BEAM_F16 && dtype != BEAM_BF16) return fail(BEAM_ERR_UNSUPPORTED, "dtype %d", dtype);
  uint16_t* out = (uint16_t*)dst_host;
  parallel_for(n, [=](size_t lo, size_t hi) {
    for (size_t i = lo; i < hi; ++i) {
      const uint64_t r = draw(seed, tensor_id, i);
      const double u1 = ((double)(r >> 40) + 1.0) * (1.0 / 16777216.0);      // (0, 1]
      const double u2 = (double)((r >> 8) & 0xffffffull) * (1.0 / 16777216.0);  // [0, 1)
      const double z = std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586476925 * u2);
      const float v = (float)((double)mean + (double)scale * z);
      out[i] = dtype == BEAM_BF16 ? to_bf16_bits(v) : to_f16_bits(v);
    }
  });
  return BEAM_OK;
}

int beam_dbg_tile_of_workgroup(int wg, int tiles_m, int tiles_n, int group_m, int* tm, int* tn) {
  if (tiles_m < 1 || tiles_n < 1 || group_m < 1 || wg < 0 || wg >= tiles_m * tiles_n || !tm || !tn)
    return fail(BEAM_ERR_INVALID, "bad rasterisation query");
  const TileDivs dv = make_tile_divs(tiles_m, tiles_n, group_m);
  const TileCoord t = tile_of_workgroup(wg, tiles_m, tiles_n, group_m, dv);
  *tm = t.tm;
  *tn = t.tn;
  return BEAM_OK;
}

int beam_dbg_tile_of_workgroup_by_division(int wg, int tiles_m, int tiles_n, int group_m, int* tm, int* tn) {
  if (tiles_m < 1 || tiles_n < 1 || group_m < 1 || wg < 0 || wg >= tiles_m * tiles_n || !tm || !tn)
    return fail(BEAM_ERR_INVALID, "bad rasterisation query");
  const TileCoord t = tile_of_workgroup(wg, tiles_m, tiles_n, group_m);
  *tm = t.tm;
  *tn = t.tn;
  return BEAM_OK;
}

unsigned beam_dbg_fast_div(unsigned n, unsigned d) { return fast_div(n, make_fast_div(d)); }

int beam_dbg_band_xcd_tile(int wg, int tiles_m, int tiles_n, int bx, int* tm, int* tn) {
  if (tiles_m < 1 || tiles_n < 1 || bx < 1 || wg < 0 || wg >= band_xcd_grid(tiles_m, tiles_n, bx) || !tm || !tn)
    return fail(BEAM_ERR_INVALID, "bad rasterisation query");
  const TileCoord t = band_xcd_tile(wg, tiles_m, tiles_n, bx);
  *tm = t.tm;
  *tn = t.tn;
  return BEAM_OK;
}

int beam_dbg_band_xcd_grid(int tiles_m, int tiles_n, int bx) { return band_xcd_grid(tiles_m, tiles_n, bx); }

int beam_dbg_lds_offset(int row, int chunk) { return lds_offset(row, chunk); }

int beam_dbg_kmajor_lds_offset(int k, int n, int block_n) { return kmajor_lds_offset(k, n, block_n); }

int beam_dbg_ln_default_config(int M, int N, int K, int compute_units, beam_tile_cfg* cfg) {
  if (!cfg || M <= 0 || N <= 0 || K <= 0) return fail(BEAM_ERR_INVALID, "bad argument");
  const KernelSet* ks = nullptr;
  return ln_choose_tile(M, N, K, compute_units, cfg, &ks) ? BEAM_OK : BEAM_ERR_UNSUPPORTED;
}

int beam_dbg_ln_line_tile(int M, int N, int K, beam_tile_cfg* cfg, int* whole_lines) {
  beam_tile_cfg named;
  const KernelSet* ks;
  if (M <= 0 || N <= 0 || K < 8 || K % 8 != 0 || !cfg || !whole_lines) return fail(BEAM_ERR_INVALID, "null pointer or not a problem on 16-byte rows");
  if (!ln_choose_tile(M, N, K, kNumXcd * 32, &named, &ks)) return fail(BEAM_ERR_UNSUPPORTED, "no one-kernel form for N=%d", N);
  const LineChoice t = ln_line_tile(M, N, K, named);
  *cfg = t.cfg;
  *whole_lines = t.lines ? 1 : 0;
  return BEAM_OK;
}

int beam_dbg_w4_kmajor_swizzle(int k) { return w4_kmajor_swizzle(k); }

int beam_dbg_w4_kmajor_read_offset(int wn, int b, int g, int e, int q) { return w4_kmajor_read_offset(wn, b, g, e, q); }

int beam_dbg_band_block_tile(int wg, int tiles_m, int tiles_n, int gb, int gc, int* tm, int* tn) {
  if (tiles_m < 1 || tiles_n < 1 || gb < 1 || gc < 1 || wg < 0 || wg >= band_block_grid(tiles_m, gb, gc) || !tm || !tn)
    return fail(BEAM_ERR_INVALID, "bad band-block query");
  const TileCoord t = band_block_tile(wg, tiles_m, tiles_n, gb, gc);
  *tm = t.tm;
  *tn = t.tn;
  return BEAM_OK;
}

int beam_dbg_band_block_grid(int tiles_m, int gb, int gc) { return band_block_grid(tiles_m, gb, gc); }

int beam_dbg_ln_band_order(int M, int N, int K, int rows, int cols) {
  return M < 1 || N < 1 || K < 1 || rows < 1 || cols < 1 ? 0 : band_group(M, N, K, rows, cols, kNumXcd * 32 * std::max(1, kLdsBytes / ((3 * rows + 2 * cols) * kRowBytes)));
}
int beam_dbg_ln_launch_order(int M, int N, int K, int rows, int cols, int whole_lines, int* group_m, int* group_n) {
  if (M < 1 || N < 1 || K < 1 || rows < 1 || cols < 1 || !group_m || !group_n) return 0;
  GemmParams p;
  p.tiles_m = (M + rows - 1) / rows, p.tiles_n = (N + cols - 1) / cols;
  if (p.tiles_n > 64) return 0;
  const beam_tile_cfg c = {rows, cols, 0, 0, 0, 0};
  const unsigned grid = ln_order(&p, M, N, K, c, false, whole_lines ? 1 : std::max(1, kLdsBytes / ((3 * rows + 2 * cols) * kRowBytes)));
  *group_m = p.group_m, *group_n = p.group_n;
  return (int)grid;
}
int beam_dbg_band_order_tile(int id, int tiles_m, int tiles_n, int group_m, int group_n, int* tm, int* tn) {
  if (tiles_m < 1 || tiles_n < 1 || group_m < 1 || id < 0 || !tm || !tn) return fail(BEAM_ERR_INVALID, "bad band-order query");
  const TileCoord t = band_order_tile(id, tiles_m, tiles_n, group_m, group_n, band_order_divs(tiles_n, group_m, group_n));
  *tm = t.tm;
  *tn = t.tn;
  return BEAM_OK;
}

}  // extern "C"
