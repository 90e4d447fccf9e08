// capi.cpp -- the C ABI of libcodag: contexts, decode entry points, host
// convenience wrappers, batch launch, autotuner and device helpers.
#include <fcntl.h>
#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "codag.h"
#include "internal.hpp"
#include "kernels/kernels.hpp"

namespace codag {

static thread_local std::string g_last_error;
void set_error(const std::string &msg) { g_last_error = msg; }
void clear_error() { g_last_error.clear(); }

}  // namespace codag

using namespace codag;

// A failed call's error is reported here and must not be found again by the check
// after the next launch (hipGetLastError keeps it until it is read).
#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess) {                                                             \
      (void)hipGetLastError();                                                          \
      return fail(CODAG_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
    }                                                                                   \
  } while (0)

namespace {
constexpr int kCounterSlots = 16;
constexpr uint32_t kCounterStride = 256;  // bytes between two slots' counters
}  // namespace

struct codag_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipEvent_t evs[256] = {};
  // Work-queue counters of the persistent batch launch, one slot per HIP
  // stream that launches batches: launches on one stream are ordered, so a
  // slot is never shared by two launches in flight (a slot taken over from
  // another stream first waits for that stream's last launch on it).
  uint32_t *d_counter = nullptr;  // kCounterSlots counters, kCounterStride bytes apart
  struct CounterSlot {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;  // recorded after the slot's last launch
    uint64_t last_use = 0;
    bool used = false;
  } slots[kCounterSlots];
  uint64_t use_clock = 0;
  uint32_t cu_count = 0;
  char name[256] = {0};
  codag_tune_params tune[4];
  uint32_t chunks_two_wave = 0;
  uint32_t byte_waves = 0;  // BRLE and LZSS kernels: 0 chosen by the streams, 1 or 4 waves per chunk, 2 LZSS one wave with a window (tests)
  uint32_t poll_shift = 0;  // RLE v2 queue kernel: nonzero = waits without polls (tests)
};

namespace {

struct DeviceGuard {
  int prev = -1;
  explicit DeviceGuard(int dev) {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DeviceGuard() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

hipStream_t pick(codag_ctx *ctx, codag_stream_t s) {
  return s ? static_cast<hipStream_t>(s) : ctx->stream;
}

codag_status check_rle_args(uint32_t w, uint64_t chunk_bytes) {
  if (!valid_width(w)) return fail(CODAG_ERR_INVALID, "elem_bytes must be 1, 2, 4 or 8");
  if (chunk_bytes == 0 || chunk_bytes % w)
    return fail(CODAG_ERR_INVALID, "chunk_bytes must be a positive multiple of elem_bytes");
  if (chunk_bytes / w >= (1ull << 19))
    return fail(CODAG_ERR_INVALID, "chunk_bytes/elem_bytes must be below 2^19 values");
  return CODAG_OK;
}

// RLE v1 / v2 walker + expander launch: 2 or 4 waves per chunk, 4 KiB window,
// queue_depth 2 (the double-buffered descriptor queue).
bool pc_shape(const codag_tune_params &t) {
  return t.queue_depth == 2 && t.window_bytes == 4096 &&
         (t.threads_per_group == 128 || t.threads_per_group == 256);
}

// RLE v2 also has the walker + 2 expander waves shape.
bool v2_pc_shape(const codag_tune_params &t) {
  return pc_shape(t) || (t.queue_depth == 2 && t.window_bytes == 4096 && t.threads_per_group == 192);
}

// RLE v1 pipeline launch: 8 waves per chunk, 2 KiB windows in a ring of 4.
bool pipe_shape(const codag_tune_params &t) {
  return t.threads_per_group == 512 && t.window_bytes == 2048 && t.queue_depth == 4;
}

// The shapes of a new context. For RLE v1 and v2 they leave the kernel to the
// launch's chunk count (rlev1_route, rlev2_route); another shape is launched as it
// is. The shape alone says so, so that setting what tune_get returned changes
// nothing. Deflate batches go by eight waves or one wave per stream, as their
// sizes have it, up to 12 workgroups per CU.
constexpr codag_tune_params kDefaultTune[4] = {{0, 0, 0, 0}, {512, 2048, 0, 4}, {128, 4096, 0, 2}, {128, 0, 12, 1}};

bool same_shape(const codag_tune_params &a, const codag_tune_params &b) {
  return std::memcmp(&a, &b, sizeof a) == 0;
}

enum Route : uint32_t {
  kRouteGroup = 0,  // the per-chunk kernels
  kRouteWave = 1,   // RLE v2, one wave per chunk
  kRoutePc = 2,     // walker + expander waves: kRoutePc + expanders
  kRoutePipe = 8,   // RLE v1 pipeline
  kRouteSpan = 9,   // sixteen waves that walk and expand by turns
};

// With the default shape, all waves by turns up to one chunk per CU (us, pipeline
// and turns: 256 chunks of an 8-bit table column 2448, 430, of the 64-bit benchmark
// column 76, 67; above it dense columns still gain, 512 chunks 2467, 543, but the
// benchmark column loses, 84, 95). Narrow columns of random values, literal groups
// of varints longer than the values, stay with the pipeline (256 chunks of random
// 16-bit values 192, 202; of 8-bit ones 317, 316).
uint32_t rlev1_route(const codag_tune_params &t, uint64_t n, uint32_t w, uint64_t chunk_bytes, uint64_t comp_bytes,
                     uint32_t cus) {
  const bool random = w <= 2 && comp_bytes / 5 > n * chunk_bytes / 4;
  if (same_shape(t, kDefaultTune[CODAG_RLEV1]) && n <= cus && !random) return kRouteSpan;
  if (pipe_shape(t)) return chunk_bytes / w <= (1u << 17) ? kRoutePipe : kRouteGroup;  // its descriptors' value field
  if (pc_shape(t)) return kRoutePc + t.threads_per_group / 64 - 1;
  return kRouteGroup;
}

// With the default shape, 16 waves per chunk that walk and expand by turns while
// two such groups per CU hold all chunks, as a lone walker's chain then bounds the
// launch (walker and three expanders, then 16 waves, us: 16-bit table column, 64
// chunks 917, 376, 512 chunks 1063, 486, 1024 chunks 1054, 807; 64-bit benchmark
// column, 512 chunks 153, 127, 1024 chunks 152, 232). Above that, expanders by the
// chunk count: three up to 6 chunks per CU and two up to 12 (1, 2 and 3 expanders,
// us: 16-bit table column, 1024 chunks 2276, 1276, 1051; 32-bit benchmark column,
// 1024 chunks 254, 249, 249, 2048 chunks 342, 317, 321).
// One walker and one expander where that work is not there: streams of up to 128
// bytes a chunk (16 chunks of 1024 equal values: 7.8 by one, 9.1 by 16 waves), and
// columns of wide DIRECT blocks, a few of which fill a step that 16 waves size
// byte by byte (random 64-bit values, one expander, three, and 16 waves: 256 chunks
// 180, 187, 235, 512 chunks 184, 191, 352; 40 bits, 256 chunks 137, 142, 147; 32
// bits, 16 chunks 119, 122, 124, 256 chunks 131, 135, 127; 20 bits, 256 chunks
// 118, 120, 99, 512 chunks 124, 126, 148; 16 bits, 512 chunks 114, 116, 110): from
// 3.5 stream bytes a value at one chunk per CU, from 2.25 above. comp_bytes may
// hold more than the chunks, which makes a column look wide: that is the kernel of
// one walker, not an error. `polls`: the walker's waits are as usual (a test takes
// their polls away).
uint32_t rlev2_route(const codag_tune_params &t, uint64_t n, uint32_t w, uint64_t chunk_bytes, uint64_t comp_bytes,
                     uint32_t cus, bool polls) {
  if (same_shape(t, kDefaultTune[CODAG_RLEV2])) {
    const uint64_t values = n * (chunk_bytes / w);
    const uint64_t quarters = n <= cus ? 14 : 9;  // of a stream byte, per value
    if (comp_bytes <= 128 * n || comp_bytes / quarters > values / 4) return kRoutePc + 1;
    if (n <= 2ull * cus && polls) return kRouteSpan;
    return kRoutePc + (n <= 6ull * cus ? 3 : (n <= 12ull * cus ? 2 : 1));
  }
  if (v2_pc_shape(t)) return kRoutePc + t.threads_per_group / 64 - 1;
  return t.threads_per_group == 64 ? kRouteWave : kRouteGroup;
}

// Whether a Deflate container of n chunks goes by eight waves per chunk (two such
// groups fit a CU) or one (nine fit). Eight and one wave, us, unless said otherwise
// on 128 KiB chunks of text (half its size when compressed):
//  * Up to two chunks per CU eight: 256 chunks 437, 1169, 512 chunks 547, 1266. Of
//    chunks of up to 4 KiB of very compressible or hardly compressible bytes the
//    headers and the first token are all there is to spread: one (512 chunks of 4
//    KiB: base64 text 366, 310, zeros 31, 26; text 142, 137, numbers 80, 89).
//  * Up to five, eight as well: 1280 chunks 1355, 1397 (64 KiB 822, 770; of 32-bit
//    counters 812, 1011). But one where the chunks are small (768 of 4 KiB 267,
//    141), where the output is 32 times the stream, as narrow_span then works by
//    one wave anyway (1280 chunks of zeros 958, 358), and where the stream is
//    nearly as long as the output but not stored, mostly literals that cost eight
//    waves the most (1280 chunks of base64 text 7483, 3693; stored 207, 286).
//  * Above that one: 2048 chunks 2.02 and 1.40 ms, 4096 3.90 and 3.04 ms.
// comp_bytes may hold more than the chunks; that only moves the choice.
bool inflate_many(uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes, uint32_t cus) {
  if (n > 5ull * cus) return false;
  const double ratio = (double)comp_bytes / ((double)n * (double)chunk_bytes);  // stream bytes per output byte
  if (n <= 2ull * cus) return chunk_bytes > 4096 || (ratio >= 0.125 && ratio <= 0.65);
  return chunk_bytes > 8192 && ratio > 1.0 / 32 && (ratio <= 0.65 || ratio > 0.99);
}

// Whether a BRLE container goes by one wave per chunk (19 such groups fit a CU) or
// four (five fit). Four and one wave, us: a chunk whose stream fits one wave's step
// leaves the others little (256 KiB of zeros, 4034 stream bytes, 512 chunks 183, 187,
// 2048 chunks 408, 220; 4 KiB of the benchmark column, 1024 chunks 17, 14, 16384
// chunks 231, 66), and where five groups per CU are filled several times over one
// wave's slower chunks overtake (16 KiB of it, 2048 chunks 47, 47, 4096 chunks 87,
// 63; 256 KiB, 1024 chunks 260, 580, 2048 chunks 500, 645, 4096 chunks 956, 861).
// Streams longer than their chunks are long literals, whose starts often never meet;
// then most of a step is one wave's chain (64 KiB, 1024 chunks: random bytes 220, 222,
// counters 238, 237, text 59, 113; 2048 chunks: 424, 257, 470, 272, 111, 134).
bool brle_few(uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes, uint32_t cus) {
  const uint64_t each = comp_bytes / n;  // stream bytes of a chunk
  if (each <= 4200) return true;
  return n > (each <= 24576 || (each >= chunk_bytes && each <= 98304) ? 7ull : 15ull) * cus;
}

// Whether an LZSS container goes by lzss_serial_kernel, one wave per chunk with its
// matches copied one after the other, or through a window of marks (lzss_waves),
// where every output byte costs the same. Window by four waves and this, us: text never one (512
// chunks of 128 KiB 631, 2474, 2048 chunks 1326, 3061); zeros and the like, 16 output
// bytes per stream byte, 512 chunks 157, 166, 1024 chunks 195, 170, 2048 chunks 338,
// 191, of 1 KiB 16384 chunks 97, 22; 37 bytes repeated in 4 KiB (298 stream bytes) 512
// chunks 13, 10; a log, 4 to 7 output bytes per stream byte,
// chunks of 1 KiB (253 stream bytes) 1024 chunks 12, 10, of 4 KiB (697) 1024 chunks
// 17, 23, 2048 chunks 28, 27, of 16 KiB (2476) 2048 chunks 65, 80, 4096 chunks 111,
// 102, of 128 KiB 2048 chunks 473, 579.
bool lzss_serial(uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes, uint32_t cus) {
  const uint64_t each = comp_bytes / n;  // stream bytes of a chunk
  if (each <= chunk_bytes / 10) return n > 2ull * cus || each <= 300;
  if (each > chunk_bytes / 7 * 2) return false;
  return each <= 300 || n > (each <= 1000 ? 7ull : 15ull) * cus;
}

// The kernel of an LZSS container: 0 lzss_serial_kernel, 4 waves with a window, or 1
// where there are many small chunks, whose streams are a step of one wave or two and
// leave most lanes of four idle (four waves and one, us, 1 KiB chunks of a table: 1024
// chunks 12, 14, 2048 chunks 20, 15, 4096 chunks 33, 20, 16384 chunks 114, 56; of
// random bytes 11, 15, 18, 17, 30, 22, 106, 62; 4 KiB chunks of a log 2048 chunks 28,
// 25, of random bytes 48, 68).
uint32_t lzss_waves(uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes, uint32_t cus) {
  if (lzss_serial(comp_bytes, n, chunk_bytes, cus)) return 0;
  return n > 7ull * cus && chunk_bytes <= 4096 && comp_bytes / n <= 1500 ? 1 : 4;
}

void default_tune(codag_ctx *c) {
  for (int k = 0; k < 4; k++) c->tune[k] = kDefaultTune[k];
}

// Gives a codec its shape back, however the scope ends, unless `keep` is set.
struct TuneGuard {
  codag_tune_params &shape;
  const codag_tune_params saved;
  bool keep = false;
  explicit TuneGuard(codag_tune_params &s) : shape(s), saved(s) {}
  ~TuneGuard() {
    if (!keep) shape = saved;
  }
};

// RAII device buffer used by the synchronous host wrappers.
struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  hipError_t alloc(uint64_t n) { return hipMalloc(&p, n ? n : 1); }
  template <typename T> T *as() const { return static_cast<T *>(p); }
};

// The device buffers of one call, 256-byte aligned parts of one allocation instead
// of five: a hipMalloc and its hipFree take up to 19 us, though the host call of a
// 4 MiB RLE v1 column gained less than four of them (885 us, with one 855).
struct DevPart {
  void *p = nullptr;
  template <typename T> T *as() const { return static_cast<T *>(p); }
};
struct DevSlab {
  DevBuf all;
  hipError_t alloc(std::initializer_list<std::pair<DevPart *, uint64_t>> parts) {
    constexpr uint64_t kMost = 1ull << 48;  // more than any GPU holds; the sum stays in range
    uint64_t n = 0;
    for (auto &x : parts) {
      if (x.second > kMost) return hipErrorOutOfMemory;
      n += (x.second + 255) & ~255ull;
    }
    const hipError_t e = all.alloc(n);
    if (e != hipSuccess) return e;
    n = 0;
    for (auto &x : parts) {
      x.first->p = all.as<uint8_t>() + n;
      n += (x.second + 255) & ~255ull;
    }
    return hipSuccess;
  }
};

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace

extern "C" {

const char *codag_version(void) { return "codag-mi355x 0.1 (gfx950)"; }

const char *codag_status_string(codag_status s) {
  switch (s) {
  case CODAG_OK: return "ok";
  case CODAG_ERR_INVALID: return "invalid argument";
  case CODAG_ERR_HIP: return "HIP runtime error";
  case CODAG_ERR_NOMEM: return "out of memory";
  case CODAG_ERR_IO: return "I/O error";
  case CODAG_ERR_FORMAT: return "inconsistent container";
  case CODAG_ERR_DECODE: return "decode error in at least one chunk";
  case CODAG_ERR_BUSY: return "busy";
  case CODAG_ERR_UNSUPPORTED: return "unsupported";
  case CODAG_ERR_TIMEOUT: return "timeout";
  }
  return "unknown status";
}

const char *codag_last_error(void) { return g_last_error.c_str(); }

int codag_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

codag_status codag_ctx_create(int device, codag_ctx **out) {
  if (!out) return fail(CODAG_ERR_INVALID, "ctx_create: null out");
  *out = nullptr;
  int n = codag_device_count();
  if (n <= 0) return fail(CODAG_ERR_UNSUPPORTED, "no HIP device available");
  if (device < 0 || device >= n) return fail(CODAG_ERR_INVALID, "device index out of range");
  DeviceGuard g(device);
  auto *c = new (std::nothrow) codag_ctx();
  if (!c) return fail(CODAG_ERR_NOMEM, "ctx_create");
  c->device = device;
  default_tune(c);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
    c->cu_count = (uint32_t)prop.multiProcessorCount;
    std::snprintf(c->name, sizeof c->name, "%s", prop.gcnArchName);
  }
  if (c->cu_count == 0) c->cu_count = 256;
  hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&c->ev0);
  if (e == hipSuccess) e = hipEventCreate(&c->ev1);
  if (e == hipSuccess) e = hipMalloc(&c->d_counter, kCounterSlots * kCounterStride);
  for (int i = 0; i < kCounterSlots && e == hipSuccess; i++)
    e = hipEventCreateWithFlags(&c->slots[i].done, hipEventDisableTiming);
  if (e != hipSuccess) {
    codag_ctx_destroy(c);
    return fail(CODAG_ERR_HIP, std::string("ctx_create: ") + hipGetErrorString(e));
  }
  *out = c;
  return CODAG_OK;
}

codag_status codag_ctx_destroy(codag_ctx *c) {
  if (!c) return CODAG_OK;
  DeviceGuard g(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto &sl : c->slots)
    if (sl.done) {
      if (sl.used) (void)hipEventSynchronize(sl.done);
      (void)hipEventDestroy(sl.done);
    }
  if (c->d_counter) (void)hipFree(c->d_counter);
  for (auto &e : c->evs)
    if (e) (void)hipEventDestroy(e);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return CODAG_OK;
}

codag_stream_t codag_ctx_stream(codag_ctx *c) { return c ? c->stream : nullptr; }

// ------------------------------------------------------------------ decode

codag_status codag_rlev1_decode(codag_ctx *ctx, const uint8_t *d_comp, uint64_t comp_bytes,
                                const uint64_t *d_blk_off, const uint64_t *d_col_len,
                                uint64_t n_chunks, uint32_t w, uint64_t chunk_bytes,
                                uint8_t *d_out, int32_t *d_status, codag_stream_t stream) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "rlev1_decode: null ctx");
  if (n_chunks && (!d_comp || !d_blk_off || !d_col_len || !d_out))
    return fail(CODAG_ERR_INVALID, "rlev1_decode: null device pointer");
  if (codag_status s = check_rle_args(w, chunk_bytes)) return s;
  if (n_chunks > 0x7fffffffull) return fail(CODAG_ERR_INVALID, "rlev1_decode: too many chunks");
  DeviceGuard g(ctx->device);
  const codag_tune_params &t = ctx->tune[CODAG_RLEV1];
  const uint32_t route = rlev1_route(t, n_chunks, w, chunk_bytes, comp_bytes, ctx->cu_count);
  if (route == kRouteSpan)
    HIP_TRY(launch_rlev1_span(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                              d_out, d_status, pick(ctx, stream)));
  else if (route == kRoutePipe)  // pipelined walker + helpers
    HIP_TRY(launch_rlev1_pipe(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                              d_out, d_status, pick(ctx, stream)));
  else if (route > kRoutePc)  // walker wave + expander waves per chunk
    HIP_TRY(launch_rlev1_pc(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                            d_out, d_status, route - kRoutePc, pick(ctx, stream)));
  else
    HIP_TRY(launch_rlev1_decode(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w,
                                chunk_bytes, d_out, d_status, t.threads_per_group,
                                pipe_shape(t) ? 4096 : t.window_bytes, pick(ctx, stream)));
  return CODAG_OK;
}

codag_status codag_rlev2_decode(codag_ctx *ctx, const uint8_t *d_comp, uint64_t comp_bytes,
                                const uint64_t *d_blk_off, const uint64_t *d_col_len,
                                uint64_t n_chunks, uint32_t w, uint64_t chunk_bytes,
                                uint8_t *d_out, int32_t *d_status, codag_stream_t stream) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "rlev2_decode: null ctx");
  if (n_chunks && (!d_comp || !d_blk_off || !d_col_len || !d_out))
    return fail(CODAG_ERR_INVALID, "rlev2_decode: null device pointer");
  if (codag_status s = check_rle_args(w, chunk_bytes)) return s;
  if (n_chunks > 0x7fffffffull) return fail(CODAG_ERR_INVALID, "rlev2_decode: too many chunks");
  DeviceGuard g(ctx->device);
  const codag_tune_params &t = ctx->tune[CODAG_RLEV2];
  const uint32_t route =
      rlev2_route(t, n_chunks, w, chunk_bytes, comp_bytes, ctx->cu_count, ctx->poll_shift == 0);
  if (route == kRouteSpan)
    HIP_TRY(launch_rlev2_span(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                              d_out, d_status, pick(ctx, stream)));
  else if (route > kRoutePc)  // walker wave + expander waves per chunk
    HIP_TRY(launch_rlev2_pc(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                            d_out, d_status, route - kRoutePc, ctx->poll_shift, pick(ctx, stream)));
  else if (route == kRouteWave)  // one self-contained wave per chunk
    HIP_TRY(launch_rlev2_wave(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w, chunk_bytes,
                              d_out, d_status, t.window_bytes, pick(ctx, stream)));
  else
    HIP_TRY(launch_rlev2_decode(d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w,
                                chunk_bytes, d_out, d_status, t.threads_per_group, t.window_bytes,
                                pick(ctx, stream)));
  return CODAG_OK;
}

codag_status codag_inflate_chunks(codag_ctx *ctx, const uint8_t *d_comp, uint64_t comp_bytes,
                                  const uint64_t *d_offsets, uint64_t n_chunks,
                                  uint64_t chunk_bytes, uint8_t *d_out, uint64_t *d_out_len,
                                  int32_t *d_status, uint32_t flags, codag_stream_t stream) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "inflate_chunks: null ctx");
  if (n_chunks && (!d_comp || !d_offsets || !d_out))
    return fail(CODAG_ERR_INVALID, "inflate_chunks: null device pointer");
  if (chunk_bytes == 0) return fail(CODAG_ERR_INVALID, "inflate_chunks: chunk_bytes is 0");
  if (n_chunks > 0x7fffffffull) return fail(CODAG_ERR_INVALID, "inflate_chunks: too many chunks");
  DeviceGuard g(ctx->device);
  bool many = inflate_many(comp_bytes, n_chunks, chunk_bytes, ctx->cu_count);
  if (ctx->chunks_two_wave) many = ctx->chunks_two_wave == 1;
  HIP_TRY(launch_inflate_chunks(d_comp, comp_bytes, d_offsets, n_chunks, chunk_bytes, d_out,
                                d_out_len, d_status, flags, pick(ctx, stream), many));
  return CODAG_OK;
}

static codag_status byte_codec_args(const char *what, codag_ctx *ctx, const uint8_t *d_comp,
                                     const uint64_t *d_idx, uint64_t n_chunks,
                                     uint64_t chunk_bytes, const uint8_t *d_out) {
  if (!ctx) return fail(CODAG_ERR_INVALID, std::string(what) + ": null ctx");
  if (n_chunks && (!d_comp || !d_idx || !d_out))
    return fail(CODAG_ERR_INVALID, std::string(what) + ": null device pointer");
  if (chunk_bytes == 0 || chunk_bytes >= (1ull << 31))
    return fail(CODAG_ERR_INVALID, std::string(what) + ": chunk_bytes must be in [1, 2^31)");
  if (n_chunks > 0x7fffffffull) return fail(CODAG_ERR_INVALID, std::string(what) + ": too many chunks");
  return CODAG_OK;
}

codag_status codag_brle_decode(codag_ctx *ctx, const uint8_t *d_comp, uint64_t comp_bytes,
                               const uint64_t *d_ptr, uint64_t n_chunks, uint64_t chunk_bytes,
                               uint8_t *d_out, uint64_t *d_out_len, int32_t *d_status,
                               codag_stream_t stream) {
  if (codag_status s = byte_codec_args("brle_decode", ctx, d_comp, d_ptr, n_chunks, chunk_bytes, d_out))
    return s;
  DeviceGuard g(ctx->device);
  bool few = n_chunks && brle_few(comp_bytes, n_chunks, chunk_bytes, ctx->cu_count);
  if (ctx->byte_waves) few = ctx->byte_waves == 1;
  HIP_TRY(launch_brle_chunks(d_comp, comp_bytes, d_ptr, n_chunks, chunk_bytes, d_out, d_out_len,
                             d_status, pick(ctx, stream), few));
  return CODAG_OK;
}

codag_status codag_lzss_decode(codag_ctx *ctx, const uint8_t *d_comp, uint64_t comp_bytes,
                               const uint64_t *d_ends, uint64_t n_chunks, uint64_t chunk_bytes,
                               uint8_t *d_out, uint64_t *d_out_len, int32_t *d_status,
                               codag_stream_t stream) {
  if (codag_status s = byte_codec_args("lzss_decode", ctx, d_comp, d_ends, n_chunks, chunk_bytes, d_out))
    return s;
  DeviceGuard g(ctx->device);
  uint32_t waves = n_chunks ? lzss_waves(comp_bytes, n_chunks, chunk_bytes, ctx->cu_count) : 0;
  if (ctx->byte_waves) waves = ctx->byte_waves == 1 ? 0 : (ctx->byte_waves == 2 ? 1 : 4);
  HIP_TRY(launch_lzss_chunks(d_comp, comp_bytes, d_ends, n_chunks, chunk_bytes, d_out, d_out_len,
                             d_status, pick(ctx, stream), waves));
  return CODAG_OK;
}

// The counter slot of stream s: the slot s already owns, else a free one,
// else the least recently used, after waiting for its last launch.
static codag_status counter_slot(codag_ctx *ctx, hipStream_t s, int *out) {
  int pick_i = -1;
  for (int i = 0; i < kCounterSlots; i++)
    if (ctx->slots[i].used && ctx->slots[i].stream == s) pick_i = i;
  if (pick_i < 0) {
    for (int i = 0; i < kCounterSlots && pick_i < 0; i++)
      if (!ctx->slots[i].used) pick_i = i;
  }
  if (pick_i < 0) {
    pick_i = 0;
    for (int i = 1; i < kCounterSlots; i++)
      if (ctx->slots[i].last_use < ctx->slots[pick_i].last_use) pick_i = i;
    HIP_TRY(hipEventSynchronize(ctx->slots[pick_i].done));
  }
  auto &sl = ctx->slots[pick_i];
  sl.stream = s;
  sl.used = true;
  sl.last_use = ++ctx->use_clock;
  *out = pick_i;
  return CODAG_OK;
}

codag_status codag_inflate_batch(codag_ctx *ctx, const codag_stream_desc *d_descs, uint64_t n,
                                 codag_stream_result *d_results, uint32_t flags,
                                 codag_stream_t stream) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "inflate_batch: null ctx");
  if (n && (!d_descs || !d_results)) return fail(CODAG_ERR_INVALID, "inflate_batch: null pointer");
  if (n >= 0xffffffffull) return fail(CODAG_ERR_INVALID, "inflate_batch: too many streams");
  DeviceGuard g(ctx->device);
  hipStream_t s = pick(ctx, stream);
  const codag_tune_params &t = ctx->tune[CODAG_DEFLATE];
  int slot = -1;
  if (codag_status st = counter_slot(ctx, s, &slot)) return st;
  uint32_t *counter = ctx->d_counter + slot * (kCounterStride / sizeof(uint32_t));
  HIP_TRY(launch_inflate_batch(d_descs, n, d_results, flags, counter, ctx->cu_count,
                               std::max(1u, t.groups_per_cu), s, t.threads_per_group == 128));
  HIP_TRY(hipEventRecord(ctx->slots[slot].done, s));
  return CODAG_OK;
}

codag_status codag_inflate_batch_noalloc(const codag_stream_desc *d_descs, uint64_t n,
                                         codag_stream_result *d_results, uint32_t flags,
                                         uint32_t groups_per_cu, codag_stream_t stream) {
  if (n && (!d_descs || !d_results))
    return fail(CODAG_ERR_INVALID, "inflate_batch_noalloc: null pointer");
  if (n >= 0xffffffffull)
    return fail(CODAG_ERR_INVALID,
                "inflate_batch_noalloc: at most 2^32-2 streams per call (the work-queue "
                "counter in the 256-byte static scratch array is 32 bits)");
  if (groups_per_cu > 64)
    return fail(CODAG_ERR_INVALID, "inflate_batch_noalloc: groups_per_cu must be 0..64");
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  int cus = 0;
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  uint32_t *counter = nullptr;
  HIP_TRY(inflate_scratch_ptr(&counter));
  HIP_TRY(launch_inflate_batch(d_descs, n, d_results, flags, counter, (uint32_t)(cus > 0 ? cus : 256),
                               groups_per_cu ? groups_per_cu : 28, static_cast<hipStream_t>(stream), true));
  return CODAG_OK;
}

// ------------------------------------------------------------------ host wrappers

static codag_status finish_host(codag_ctx *ctx, const DevPart &d_status, uint64_t n,
                                double *kernel_seconds) {
  HIP_TRY(hipEventSynchronize(ctx->ev1));
  float ms = 0;
  HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
  if (kernel_seconds) *kernel_seconds = ms / 1e3;
  std::vector<int32_t> st(n);
  if (n) HIP_TRY(hipMemcpy(st.data(), d_status.p, n * sizeof(int32_t), hipMemcpyDeviceToHost));
  uint64_t bad = 0;
  for (auto v : st) bad += (v != 0);
  if (bad)
    return fail(CODAG_ERR_DECODE, std::to_string(bad) + " of " + std::to_string(n) +
                                      " chunks failed to decode");
  return CODAG_OK;
}

codag_status codag_rlev1_decode_host(codag_ctx *ctx, const uint8_t *container,
                                     uint64_t container_bytes, const uint64_t *blk_off_file,
                                     uint64_t blk_off_entries, const uint64_t *col_len_file,
                                     uint64_t col_len_entries, uint32_t w, uint64_t chunk_bytes,
                                     uint8_t *out, uint64_t out_cap, uint64_t *out_bytes,
                                     double *kernel_seconds, double *total_seconds) {
  const double t0 = now_s();
  if (!ctx || !container || !blk_off_file || !col_len_file || !out_bytes)
    return fail(CODAG_ERR_INVALID, "rlev1_decode_host: null argument");
  if (codag_status s = check_rle_args(w, chunk_bytes)) return s;
  if (container_bytes < 8) return fail(CODAG_ERR_FORMAT, "container shorter than its length word");
  if (blk_off_entries < 1) return fail(CODAG_ERR_FORMAT, "empty blk_offset file");
  const uint64_t n = (blk_off_entries - 1) / 32;  // rlev1.h:469
  if (col_len_entries < n) return fail(CODAG_ERR_FORMAT, "col_len file shorter than chunk count");
  const uint64_t body = container_bytes - 8;
  for (uint64_t i = 0; i < n; i++)
    if (blk_off_file[i] > body || col_len_file[i] > body - blk_off_file[i])
      return fail(CODAG_ERR_FORMAT, "chunk " + std::to_string(i) + " lies outside the container");
  uint64_t orig = load_le(container, 8);  // rlev1.h:478
  if (orig > n * chunk_bytes) return fail(CODAG_ERR_FORMAT, "original length exceeds the chunks");
  if (!out || out_cap < orig) return fail(CODAG_ERR_INVALID, "output buffer too small");
  DeviceGuard g(ctx->device);
  DevSlab slab;
  DevPart d_in, d_off, d_len, d_out, d_st;
  HIP_TRY(slab.alloc({{&d_in, body}, {&d_off, n * 8}, {&d_len, n * 8}, {&d_out, n * chunk_bytes}, {&d_st, n * 4}}));
  HIP_TRY(hipMemcpyAsync(d_in.p, container + 8, body, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipMemcpyAsync(d_off.p, blk_off_file, n * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipMemcpyAsync(d_len.p, col_len_file, n * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
  codag_status s = codag_rlev1_decode(ctx, d_in.as<uint8_t>(), body, d_off.as<uint64_t>(),
                                      d_len.as<uint64_t>(), n, w, chunk_bytes, d_out.as<uint8_t>(),
                                      d_st.as<int32_t>(), ctx->stream);
  if (s) return s;
  HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
  HIP_TRY(hipMemcpyAsync(out, d_out.p, orig, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  *out_bytes = orig;
  s = finish_host(ctx, d_st, n, kernel_seconds);
  if (total_seconds) *total_seconds = now_s() - t0;
  return s;
}

namespace {
// Read-only map of a whole file; empty files map to nothing.
struct MapFile {
  void *p = nullptr;
  uint64_t n = 0;
  int fd = -1;
  bool open(const char *path) {
    fd = ::open(path, O_RDONLY);
    if (fd < 0) return false;
    struct stat sb;
    if (fstat(fd, &sb) != 0) return false;
    n = (uint64_t)sb.st_size;
    if (!n) return true;
    p = mmap(nullptr, n, PROT_READ, MAP_PRIVATE, fd, 0);
    if (p == MAP_FAILED) {
      p = nullptr;
      return false;
    }
    return true;
  }
  ~MapFile() {
    if (p) munmap(p, n);
    if (fd >= 0) ::close(fd);
  }
};
}  // namespace

codag_status codag_rlev1_decode_files(codag_ctx *ctx, const uint8_t *container,
                                      uint64_t container_bytes, const char *col_len_path,
                                      const char *blk_off_path, uint32_t w, uint64_t chunk_bytes,
                                      uint8_t **out, uint64_t *out_bytes, uint64_t *meta_bytes,
                                      double *kernel_seconds) {
  if (!ctx || !container || !col_len_path || !blk_off_path || !out || !out_bytes)
    return fail(CODAG_ERR_INVALID, "rlev1_decode_files: null argument");
  *out = nullptr;
  *out_bytes = 0;
  if (container_bytes < 8) return fail(CODAG_ERR_FORMAT, "container shorter than its length word");
  MapFile fc, fb;
  if (!fc.open(col_len_path)) return fail(CODAG_ERR_IO, std::string("cannot read ") + col_len_path);
  if (!fb.open(blk_off_path)) return fail(CODAG_ERR_IO, std::string("cannot read ") + blk_off_path);
  if (meta_bytes) *meta_bytes = fc.n + fb.n;  // rlev1.h:501
  const uint64_t orig = load_le(container, 8);  // rlev1.h:478
  auto *buf = static_cast<uint8_t *>(std::malloc(orig ? orig : 1));
  if (!buf) return fail(CODAG_ERR_NOMEM, "rlev1_decode_files: host output");
  uint64_t got = 0;
  codag_status s = codag_rlev1_decode_host(
      ctx, container, container_bytes, static_cast<const uint64_t *>(fb.p), fb.n / 8,
      static_cast<const uint64_t *>(fc.p), fc.n / 8, w, chunk_bytes, buf, orig, &got,
      kernel_seconds, nullptr);
  if (s) {
    std::free(buf);
    return s;
  }
  *out = buf;
  *out_bytes = got;
  return CODAG_OK;
}

codag_status codag_rlev2_decode_host(codag_ctx *ctx, const uint8_t *comp, uint64_t comp_bytes,
                                     const uint64_t *blk_off, const uint64_t *col_len,
                                     uint64_t n, uint32_t w, uint64_t chunk_bytes, uint8_t *out,
                                     uint64_t out_cap, uint64_t *out_bytes,
                                     double *kernel_seconds, double *total_seconds) {
  const double t0 = now_s();
  if (!ctx || (!comp && comp_bytes) || !blk_off || !col_len || !out_bytes)
    return fail(CODAG_ERR_INVALID, "rlev2_decode_host: null argument");
  if (codag_status s = check_rle_args(w, chunk_bytes)) return s;
  for (uint64_t i = 0; i < n; i++)
    if (blk_off[i] > comp_bytes || col_len[i] > comp_bytes - blk_off[i])
      return fail(CODAG_ERR_FORMAT, "chunk " + std::to_string(i) + " lies outside the stream");
  const uint64_t orig = blk_off[n];  // encoder_trans.h:545, decoder_trans.h:67
  if (orig > n * chunk_bytes) return fail(CODAG_ERR_FORMAT, "original length exceeds the chunks");
  if (!out || out_cap < orig) return fail(CODAG_ERR_INVALID, "output buffer too small");
  DeviceGuard g(ctx->device);
  DevSlab slab;
  DevPart d_in, d_off, d_len, d_out, d_st;
  HIP_TRY(slab.alloc({{&d_in, comp_bytes}, {&d_off, n * 8}, {&d_len, n * 8}, {&d_out, n * chunk_bytes}, {&d_st, n * 4}}));
  if (comp_bytes)
    HIP_TRY(hipMemcpyAsync(d_in.p, comp, comp_bytes, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipMemcpyAsync(d_off.p, blk_off, n * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipMemcpyAsync(d_len.p, col_len, n * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
  codag_status s = codag_rlev2_decode(ctx, d_in.as<uint8_t>(), comp_bytes, d_off.as<uint64_t>(),
                                      d_len.as<uint64_t>(), n, w, chunk_bytes, d_out.as<uint8_t>(),
                                      d_st.as<int32_t>(), ctx->stream);
  if (s) return s;
  HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
  HIP_TRY(hipMemcpyAsync(out, d_out.p, orig, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  *out_bytes = orig;
  s = finish_host(ctx, d_st, n, kernel_seconds);
  if (total_seconds) *total_seconds = now_s() - t0;
  return s;
}

codag_status codag_inflate_chunks_host(codag_ctx *ctx, const uint8_t *comp, uint64_t comp_bytes,
                                       const uint64_t *blk, uint64_t entries, uint64_t chunk_bytes,
                                       uint32_t flags, uint8_t *out, uint64_t out_cap,
                                       uint64_t *out_bytes, double *kernel_seconds,
                                       double *total_seconds) {
  const double t0 = now_s();
  if (!ctx || (!comp && comp_bytes) || !blk || !out_bytes)
    return fail(CODAG_ERR_INVALID, "inflate_chunks_host: null argument");
  if (entries < 2) return fail(CODAG_ERR_FORMAT, "blk_offset file needs at least 2 entries");
  if (chunk_bytes == 0) return fail(CODAG_ERR_INVALID, "chunk_bytes is 0");
  const uint64_t n = entries - 2;  // zlib.h:1589
  const uint64_t orig = blk[0];    // zlib.h:1590
  const uint64_t *off = blk + 1;   // zlib.h:1603
  for (uint64_t i = 0; i < n; i++)
    if (off[i] > off[i + 1] || off[i + 1] > comp_bytes)
      return fail(CODAG_ERR_FORMAT, "chunk " + std::to_string(i) + " lies outside the stream");
  if (orig > n * chunk_bytes) return fail(CODAG_ERR_FORMAT, "original length exceeds the chunks");
  if (!out || out_cap < orig) return fail(CODAG_ERR_INVALID, "output buffer too small");
  DeviceGuard g(ctx->device);
  DevSlab slab;
  DevPart d_in, d_off, d_out, d_st;
  HIP_TRY(slab.alloc({{&d_in, comp_bytes}, {&d_off, (n + 1) * 8}, {&d_out, n * chunk_bytes}, {&d_st, n * 4}}));
  if (comp_bytes)
    HIP_TRY(hipMemcpyAsync(d_in.p, comp, comp_bytes, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipMemcpyAsync(d_off.p, off, (n + 1) * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
  codag_status s =
      codag_inflate_chunks(ctx, d_in.as<uint8_t>(), comp_bytes, d_off.as<uint64_t>(), n,
                           chunk_bytes, d_out.as<uint8_t>(), nullptr, d_st.as<int32_t>(), flags,
                           ctx->stream);
  if (s) return s;
  HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
  HIP_TRY(hipMemcpyAsync(out, d_out.p, orig, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  *out_bytes = orig;
  s = finish_host(ctx, d_st, n, kernel_seconds);
  if (total_seconds) *total_seconds = now_s() - t0;
  return s;
}

// Shared tail of the BRLE / LZSS host wrappers: uploads the streams and the
// index array, decodes n chunks of chunk_bytes, checks that chunk i produced
// exactly min(chunk_bytes, orig - i*chunk_bytes) bytes and copies orig bytes
// out.
static codag_status byte_codec_host(codag_ctx *ctx, bool lzss, const uint8_t *data,
                                    uint64_t data_bytes, const uint64_t *idx, uint64_t idx_n,
                                    uint64_t n, uint64_t chunk_bytes, uint64_t orig, uint8_t *out,
                                    uint64_t *out_bytes, double *kernel_seconds) {
  DeviceGuard g(ctx->device);
  DevSlab slab;
  DevPart d_in, d_idx, d_out, d_len, d_st;
  HIP_TRY(slab.alloc({{&d_in, data_bytes}, {&d_idx, idx_n * 8}, {&d_out, n * chunk_bytes}, {&d_len, n * 8}, {&d_st, n * 4}}));
  if (data_bytes) HIP_TRY(hipMemcpyAsync(d_in.p, data, data_bytes, hipMemcpyHostToDevice, ctx->stream));
  if (idx_n) HIP_TRY(hipMemcpyAsync(d_idx.p, idx, idx_n * 8, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
  codag_status s =
      lzss ? codag_lzss_decode(ctx, d_in.as<uint8_t>(), data_bytes, d_idx.as<uint64_t>(), n,
                               chunk_bytes, d_out.as<uint8_t>(), d_len.as<uint64_t>(),
                               d_st.as<int32_t>(), ctx->stream)
           : codag_brle_decode(ctx, d_in.as<uint8_t>(), data_bytes, d_idx.as<uint64_t>(), n,
                               chunk_bytes, d_out.as<uint8_t>(), d_len.as<uint64_t>(),
                               d_st.as<int32_t>(), ctx->stream);
  if (s) return s;
  HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
  if (orig) HIP_TRY(hipMemcpyAsync(out, d_out.p, orig, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  *out_bytes = orig;
  s = finish_host(ctx, d_st, n, kernel_seconds);
  if (s) return s;
  std::vector<uint64_t> got(n);
  if (n) HIP_TRY(hipMemcpy(got.data(), d_len.p, n * 8, hipMemcpyDeviceToHost));
  for (uint64_t i = 0; i < n; i++) {
    const uint64_t want = std::min(chunk_bytes, orig - i * chunk_bytes);
    if (got[i] != want)
      return fail(CODAG_ERR_DECODE, "chunk " + std::to_string(i) + " produced " +
                                        std::to_string(got[i]) + " bytes, expected " +
                                        std::to_string(want));
  }
  return CODAG_OK;
}

codag_status codag_brle_decode_host(codag_ctx *ctx, const uint8_t *c, uint64_t cb,
                                    uint64_t chunk_bytes, uint8_t *out, uint64_t out_cap,
                                    uint64_t *out_bytes, double *kernel_seconds,
                                    double *total_seconds) {
  const double t0 = now_s();
  if (!ctx || !c || !out_bytes) return fail(CODAG_ERR_INVALID, "brle_decode_host: null argument");
  if (chunk_bytes == 0) chunk_bytes = 262144;  // brle.h:8
  // [u32 n+1][u64 ptr[n+1]][u64 original_len][streams] (brle.h:281-296, 310-316)
  if (cb < 4) return fail(CODAG_ERR_FORMAT, "brle container shorter than its header");
  uint32_t n_ptr;
  std::memcpy(&n_ptr, c, 4);
  if (n_ptr == 0 || cb < 4 + 8ull * n_ptr + 8)
    return fail(CODAG_ERR_FORMAT, "brle container shorter than its ptr array");
  const uint64_t n = n_ptr - 1;
  std::vector<uint64_t> ptr(n_ptr);
  std::memcpy(ptr.data(), c + 4, 8ull * n_ptr);
  uint64_t orig;
  std::memcpy(&orig, c + 4 + 8ull * n_ptr, 8);
  const uint64_t head = 4 + 8ull * n_ptr + 8;
  const uint8_t *data = c + head;
  const uint64_t data_bytes = cb - head;
  if (ptr[0] != 0) return fail(CODAG_ERR_FORMAT, "brle ptr[0] is not 0");
  for (uint64_t i = 0; i < n; i++)
    if (ptr[i] > ptr[i + 1] || ptr[i + 1] > data_bytes)
      return fail(CODAG_ERR_FORMAT, "chunk " + std::to_string(i) + " lies outside the stream");
  if (orig > n * chunk_bytes || (n && orig <= (n - 1) * chunk_bytes))
    return fail(CODAG_ERR_FORMAT, "original length does not match the chunk count");
  if ((!out && orig) || out_cap < orig) return fail(CODAG_ERR_INVALID, "output buffer too small");
  codag_status s = byte_codec_host(ctx, false, data, data_bytes, ptr.data(), n_ptr, n, chunk_bytes,
                                   orig, out, out_bytes, kernel_seconds);
  if (total_seconds) *total_seconds = now_s() - t0;
  return s;
}

codag_status codag_lzss_decode_host(codag_ctx *ctx, const uint8_t *c, uint64_t cb, uint8_t *out,
                                    uint64_t out_cap, uint64_t *out_bytes, double *kernel_seconds,
                                    double *total_seconds) {
  const double t0 = now_s();
  if (!ctx || !c || !out_bytes) return fail(CODAG_ERR_INVALID, "lzss_decode_host: null argument");
  // [u64 original_len][u32 chunk, n, hist, min, max][u64 ends[n]][streams]
  // (lzss.h:1100-1119, read back at 1133-1146)
  if (cb < 28) return fail(CODAG_ERR_FORMAT, "lzss container shorter than its header");
  uint64_t orig;
  uint32_t h[5];
  std::memcpy(&orig, c, 8);
  std::memcpy(h, c + 8, 20);
  const uint64_t chunk_bytes = h[0], n = h[1];
  if (h[2] != 2048 || h[3] != 3 || h[4] != 34)
    return fail(CODAG_ERR_FORMAT, "lzss parameters other than history 2048, matches 3-34");
  if (chunk_bytes == 0 && n) return fail(CODAG_ERR_FORMAT, "lzss chunk size is 0");
  if (cb < 28 + 8 * n) return fail(CODAG_ERR_FORMAT, "lzss container shorter than its lens array");
  std::vector<uint64_t> ends(n);
  if (n) std::memcpy(ends.data(), c + 28, 8 * n);
  const uint8_t *data = c + 28 + 8 * n;
  const uint64_t data_bytes = cb - 28 - 8 * n;
  for (uint64_t i = 0; i < n; i++)
    if ((i && ends[i] < ends[i - 1]) || ends[i] > data_bytes)
      return fail(CODAG_ERR_FORMAT, "chunk " + std::to_string(i) + " lies outside the stream");
  if (orig > n * chunk_bytes || (n && orig <= (n - 1) * chunk_bytes))
    return fail(CODAG_ERR_FORMAT, "original length does not match the chunk count");
  if ((!out && orig) || out_cap < orig) return fail(CODAG_ERR_INVALID, "output buffer too small");
  codag_status s = byte_codec_host(ctx, true, data, data_bytes, ends.data(), n, n,
                                   chunk_bytes ? chunk_bytes : 131072, orig, out, out_bytes,
                                   kernel_seconds);
  if (total_seconds) *total_seconds = now_s() - t0;
  return s;
}

// ------------------------------------------------------------------ tuning

// Test hook, not in the public header: codag_inflate_chunks' workgroups --
// 0 chosen by inflate_many, 1 eight waves per chunk, 2 one wave per chunk.
codag_status codag_test_chunks_two_wave(codag_ctx *ctx, uint32_t on) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "test_chunks_two_wave: null ctx");
  ctx->chunks_two_wave = on;
  return CODAG_OK;
}

// Test hook, not in the public header: the kernel (a Route) that a decode of n
// chunks is launched with.
uint32_t codag_test_route(codag_ctx *ctx, codag_codec codec, uint64_t comp_bytes, uint64_t n, uint32_t w,
                          uint64_t chunk_bytes) {
  if (!ctx || (codec != CODAG_RLEV1 && codec != CODAG_RLEV2)) return ~0u;
  const codag_tune_params &t = ctx->tune[codec];
  return codec == CODAG_RLEV1 ? rlev1_route(t, n, w, chunk_bytes, comp_bytes, ctx->cu_count)
                              : rlev2_route(t, n, w, chunk_bytes, comp_bytes, ctx->cu_count, ctx->poll_shift == 0);
}

// Test hook, not in the public header: the waves per chunk of the BRLE and LZSS
// kernels, 1 or 4, or 0 for the choice by the streams.
codag_status codag_test_byte_waves(codag_ctx *ctx, uint32_t waves) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "test_byte_waves: null ctx");
  ctx->byte_waves = waves;
  return CODAG_OK;
}

// Test hook, not in the public header: whether codag_brle_decode (codag_lzss_decode)
// of n > 0 chunks takes the kernel of one wave per chunk.
uint32_t codag_test_byte_one(codag_ctx *ctx, uint32_t lzss, uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes) {
  if (!ctx || !n) return ~0u;
  return lzss ? lzss_serial(comp_bytes, n, chunk_bytes, ctx->cu_count) : brle_few(comp_bytes, n, chunk_bytes, ctx->cu_count);
}

// Test hook, not in the public header: the kernel that LZSS chunks go by (lzss_waves).
uint32_t codag_test_lzss_waves(codag_ctx *ctx, uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes) {
  return ctx && n ? lzss_waves(comp_bytes, n, chunk_bytes, ctx->cu_count) : ~0u;
}

// Test hook, not in the public header: whether codag_inflate_chunks takes eight waves.
uint32_t codag_test_inflate_many(codag_ctx *ctx, uint64_t comp_bytes, uint64_t n, uint64_t chunk_bytes) {
  return ctx ? inflate_many(comp_bytes, n, chunk_bytes, ctx->cu_count) : ~0u;
}

// Test hook, not in the public header (no counterpart in the reference):
// `shift` nonzero switches the RLE v2 walker + expander kernel to its
// variant without polls in its bounded waits (0 restores the normal one), so
// a test can drive the waits' error path.
codag_status codag_test_poll_shift(codag_ctx *ctx, uint32_t shift) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "test_poll_shift: null ctx");
  ctx->poll_shift = shift;
  return CODAG_OK;
}

codag_status codag_tune_get(codag_ctx *ctx, codag_codec codec, codag_tune_params *out) {
  if (!ctx || !out || codec < CODAG_RLEV1 || codec > CODAG_DEFLATE)
    return fail(CODAG_ERR_INVALID, "tune_get: bad argument");
  *out = ctx->tune[codec];
  return CODAG_OK;
}

codag_status codag_tune_set(codag_ctx *ctx, codag_codec codec, const codag_tune_params *p) {
  if (!ctx || !p || codec < CODAG_RLEV1 || codec > CODAG_DEFLATE)
    return fail(CODAG_ERR_INVALID, "tune_set: bad argument");
  const bool wave_shape = (codec == CODAG_RLEV2 && p->threads_per_group == 64 &&
                           p->queue_depth == 0 &&
                           (p->window_bytes == 4096 || p->window_bytes == 8192)) ||
                          (codec != CODAG_DEFLATE && pc_shape(*p)) ||
                          (codec == CODAG_RLEV2 && v2_pc_shape(*p)) ||
                          (codec == CODAG_RLEV1 && pipe_shape(*p));
  if (codec != CODAG_DEFLATE && !wave_shape &&
      !rle_shape_supported(p->threads_per_group, p->window_bytes))
    return fail(CODAG_ERR_INVALID, "tune_set: launch shape not compiled in");
  if (codec == CODAG_DEFLATE && (p->groups_per_cu == 0 || p->groups_per_cu > 64))
    return fail(CODAG_ERR_INVALID, "tune_set: groups_per_cu must be 1..64");
  if (codec == CODAG_DEFLATE && p->threads_per_group != 64 && p->threads_per_group != 128)
    return fail(CODAG_ERR_INVALID, "tune_set: Deflate threads_per_group must be 64 or 128");
  ctx->tune[codec] = *p;
  return CODAG_OK;
}

codag_status codag_tune_run(codag_ctx *ctx, codag_codec codec, const uint8_t *d_comp,
                            uint64_t comp_bytes, const uint64_t *d_blk_off,
                            const uint64_t *d_col_len, uint64_t n_chunks, uint32_t w,
                            uint64_t chunk_bytes, uint8_t *d_out, int reps,
                            codag_tune_params *best, float *best_ms) {
  if (!ctx || codec < CODAG_RLEV1 || codec > CODAG_DEFLATE)
    return fail(CODAG_ERR_INVALID, "tune_run: bad argument");
  if (reps < 1) reps = 3;
  DeviceGuard g(ctx->device);
  std::vector<codag_tune_params> cands;
  if (codec == CODAG_DEFLATE) {
    for (uint32_t per : {8u, 16u, 20u, 24u, 28u}) cands.push_back({64, 0, per, 1});
    for (uint32_t per : {8u, 12u, 14u}) cands.push_back({128, 0, per, 1});  // by size
  } else {
    if (codec == CODAG_RLEV1) cands.push_back({512, 2048, 0, 4});  // pipelined walker + helpers
    cands.push_back({256, 4096, 0, 2});  // walker + expander shapes
    cands.push_back({128, 4096, 0, 2});
    if (codec == CODAG_RLEV2) cands.push_back({192, 4096, 0, 2});
    if (codec == CODAG_RLEV2) {  // one-wave-per-chunk shapes
      cands.push_back({64, 4096, 0, 0});
      cands.push_back({64, 8192, 0, 0});
    }
    const uint32_t shapes[][2] = {{256, 4096}, {128, 4096}, {512, 4096}, {256, 8192}, {512, 8192}};
    for (auto &sh : shapes) cands.push_back({sh[0], sh[1], 0, 0});
  }
  TuneGuard guard(ctx->tune[codec]);
  const codag_tune_params saved = guard.saved;
  const uint64_t out_bytes = n_chunks * chunk_bytes;
  std::vector<uint8_t> ref, cur;
  float bestt = 1e30f, saved_ms = 0;
  codag_tune_params bestp = saved;
  DevBuf d_st, d_descs, d_res;
  HIP_TRY(d_st.alloc(n_chunks * 8 + 8));
  if (codec == CODAG_DEFLATE) {
    // Deflate candidates differ in the persistent batch launch (one wave a stream or
    // the plan's choice, and groups per CU): time that launch on the sample's chunks.
    std::vector<uint64_t> off(n_chunks + 1);
    HIP_TRY(hipMemcpy(off.data(), d_blk_off, 8 * (n_chunks + 1), hipMemcpyDeviceToHost));
    std::vector<codag_stream_desc> descs(n_chunks);
    for (uint64_t i = 0; i < n_chunks; i++) {
      if (off[i + 1] < off[i] || off[i + 1] > comp_bytes)
        return fail(CODAG_ERR_INVALID, "tune_run: offsets out of range");
      descs[i] = {d_comp + off[i], off[i + 1] - off[i], d_out + i * chunk_bytes, chunk_bytes};
    }
    HIP_TRY(d_descs.alloc(sizeof(codag_stream_desc) * n_chunks + 8));
    HIP_TRY(d_res.alloc(sizeof(codag_stream_result) * n_chunks + 8));
    HIP_TRY(hipMemcpy(d_descs.p, descs.data(), sizeof(codag_stream_desc) * n_chunks,
                      hipMemcpyHostToDevice));
  }
  for (size_t ci = 0; ci < cands.size(); ci++) {
    ctx->tune[codec] = cands[ci];
    auto run = [&]() -> codag_status {
      if (codec == CODAG_RLEV1)
        return codag_rlev1_decode(ctx, d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w,
                                  chunk_bytes, d_out, d_st.as<int32_t>(), ctx->stream);
      if (codec == CODAG_RLEV2)
        return codag_rlev2_decode(ctx, d_comp, comp_bytes, d_blk_off, d_col_len, n_chunks, w,
                                  chunk_bytes, d_out, d_st.as<int32_t>(), ctx->stream);
      return codag_inflate_batch(ctx, d_descs.as<codag_stream_desc>(), n_chunks,
                                 d_res.as<codag_stream_result>(), 0, ctx->stream);
    };
    codag_status s = run();  // warm-up
    if (s) return s;
    HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
    for (int r = 0; r < reps; r++) run();
    HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
    HIP_TRY(hipEventSynchronize(ctx->ev1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    ms /= reps;
    // every candidate must reproduce the first candidate's output
    cur.resize(out_bytes);
    HIP_TRY(hipMemcpy(cur.data(), d_out, out_bytes, hipMemcpyDeviceToHost));
    if (ci == 0) ref = cur;
    const bool same = (cur == ref);
    if (same && ms < bestt) {
      bestt = ms;
      bestp = cands[ci];
    }
    if (same && same_shape(cands[ci], saved)) saved_ms = ms;
  }
  // the shape in use stays unless a candidate beats it by more than 2%
  // (run-to-run noise must not flip the choice)
  if (saved_ms > 0 && saved_ms <= bestt * 1.02f) {
    bestp = saved;
    bestt = saved_ms;
  }
  ctx->tune[codec] = bestp;
  guard.keep = true;
  if (best) *best = bestp;
  if (best_ms) *best_ms = bestt;
  return CODAG_OK;
}

// ------------------------------------------------------------------ plumbing

codag_status codag_dev_alloc(codag_ctx *ctx, uint64_t bytes, void **d_ptr) {
  if (!ctx || !d_ptr) return fail(CODAG_ERR_INVALID, "dev_alloc: null argument");
  DeviceGuard g(ctx->device);
  hipError_t e = hipMalloc(d_ptr, bytes ? bytes : 1);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return fail(CODAG_ERR_NOMEM, "hipMalloc: out of memory");
  }
  HIP_TRY(e);
  return CODAG_OK;
}

codag_status codag_dev_free(codag_ctx *ctx, void *d_ptr) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "dev_free: null ctx");
  if (!d_ptr) return CODAG_OK;
  DeviceGuard g(ctx->device);
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  HIP_TRY(hipFree(d_ptr));
  return CODAG_OK;
}

codag_status codag_copy_h2d(codag_ctx *ctx, void *d_dst, const void *h_src, uint64_t bytes) {
  if (!ctx || (bytes && (!d_dst || !h_src))) return fail(CODAG_ERR_INVALID, "copy_h2d");
  if (!bytes) return CODAG_OK;
  DeviceGuard g(ctx->device);
  HIP_TRY(hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  return CODAG_OK;
}

codag_status codag_copy_d2h(codag_ctx *ctx, void *h_dst, const void *d_src, uint64_t bytes) {
  if (!ctx || (bytes && (!h_dst || !d_src))) return fail(CODAG_ERR_INVALID, "copy_d2h");
  if (!bytes) return CODAG_OK;
  DeviceGuard g(ctx->device);
  HIP_TRY(hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  return CODAG_OK;
}

codag_status codag_copy_d2d(codag_ctx *ctx, void *d_dst, const void *d_src, uint64_t bytes) {
  if (!ctx || (bytes && (!d_dst || !d_src))) return fail(CODAG_ERR_INVALID, "copy_d2d");
  DeviceGuard g(ctx->device);
  HIP_TRY(launch_copy(static_cast<uint8_t *>(d_dst), static_cast<const uint8_t *>(d_src), bytes,
                      ctx->stream));
  return CODAG_OK;
}

codag_status codag_memset_d(codag_ctx *ctx, void *d_dst, int value, uint64_t bytes) {
  if (!ctx || (bytes && !d_dst)) return fail(CODAG_ERR_INVALID, "memset_d");
  if (!bytes) return CODAG_OK;
  DeviceGuard g(ctx->device);
  HIP_TRY(hipMemsetAsync(d_dst, value, bytes, ctx->stream));
  return CODAG_OK;
}

codag_status codag_stream_create(codag_ctx *ctx, codag_stream_t *out) {
  if (!ctx || !out) return fail(CODAG_ERR_INVALID, "stream_create: null argument");
  DeviceGuard g(ctx->device);
  hipStream_t s = nullptr;
  HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  *out = s;
  return CODAG_OK;
}

codag_status codag_stream_destroy(codag_ctx *ctx, codag_stream_t stream) {
  if (!ctx || !stream) return fail(CODAG_ERR_INVALID, "stream_destroy: null argument");
  DeviceGuard g(ctx->device);
  hipStream_t s = static_cast<hipStream_t>(stream);
  HIP_TRY(hipStreamSynchronize(s));
  // a counter slot bound to this stream is released with it
  for (auto &sl : ctx->slots)
    if (sl.used && sl.stream == s) {
      sl.used = false;
      sl.stream = nullptr;
    }
  HIP_TRY(hipStreamDestroy(s));
  return CODAG_OK;
}

codag_status codag_stream_sync(codag_ctx *ctx, codag_stream_t stream) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "stream_sync: null ctx");
  DeviceGuard g(ctx->device);
  HIP_TRY(hipStreamSynchronize(pick(ctx, stream)));
  return CODAG_OK;
}

codag_status codag_sync(codag_ctx *ctx) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "sync: null ctx");
  DeviceGuard g(ctx->device);
  HIP_TRY(hipStreamSynchronize(ctx->stream));
  return CODAG_OK;
}

codag_status codag_timer_start(codag_ctx *ctx) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "timer_start: null ctx");
  DeviceGuard g(ctx->device);
  HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
  return CODAG_OK;
}

codag_status codag_timer_stop(codag_ctx *ctx, float *elapsed_ms) {
  if (!ctx || !elapsed_ms) return fail(CODAG_ERR_INVALID, "timer_stop: bad argument");
  DeviceGuard g(ctx->device);
  HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
  HIP_TRY(hipEventSynchronize(ctx->ev1));
  HIP_TRY(hipEventElapsedTime(elapsed_ms, ctx->ev0, ctx->ev1));
  return CODAG_OK;
}

codag_status codag_event_record(codag_ctx *ctx, uint32_t slot, codag_stream_t stream) {
  if (!ctx || slot >= 256) return fail(CODAG_ERR_INVALID, "event_record: bad argument");
  DeviceGuard g(ctx->device);
  if (!ctx->evs[slot]) HIP_TRY(hipEventCreate(&ctx->evs[slot]));
  HIP_TRY(hipEventRecord(ctx->evs[slot], pick(ctx, stream)));
  return CODAG_OK;
}

codag_status codag_event_elapsed(codag_ctx *ctx, uint32_t a, uint32_t b, float *ms) {
  if (!ctx || a >= 256 || b >= 256 || !ms || !ctx->evs[a] || !ctx->evs[b])
    return fail(CODAG_ERR_INVALID, "event_elapsed: bad argument");
  DeviceGuard g(ctx->device);
  HIP_TRY(hipEventSynchronize(ctx->evs[b]));
  HIP_TRY(hipEventElapsedTime(ms, ctx->evs[a], ctx->evs[b]));
  return CODAG_OK;
}

codag_status codag_device_info(codag_ctx *ctx, char *name, uint32_t name_cap, uint32_t *cu_count) {
  if (!ctx) return fail(CODAG_ERR_INVALID, "device_info: null ctx");
  if (name && name_cap) std::snprintf(name, name_cap, "%s", ctx->name);
  if (cu_count) *cu_count = ctx->cu_count;
  return CODAG_OK;
}

}  // extern "C"
