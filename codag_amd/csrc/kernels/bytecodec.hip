// bytecodec.hip -- gfx950 decoders of the reference's two byte-oriented
// codecs:
//
//   BRLE  include/brle/brle.h:26-100 (brle::decode, direct path at 76-90;
//         kernel_decompress 102-110 runs one thread per chunk). A header
//         byte h > 127 is followed by h - 127 literal bytes, h <= 127 by one
//         byte repeated h + 3 times. Chunk i is data[ptr[i] .. ptr[i+1]) and
//         decodes into out + i * chunk (256 KiB in the reference, brle.h:8).
//   LZSS  include/lzss/lzss.h:234-305 (lzss::decompress_func, one thread per
//         chunk). A flag byte covers the next 8 items, least significant bit
//         first: bit 1 is a literal byte, bit 0 a 2-byte little-endian
//         reference v, length (v & 31) + 3, offset v >> 5 (11 offset bits for
//         the 2048-byte history, lzss.h:24-32), copied byte by byte from
//         offset bytes back. Chunk i is data[end[i-1] .. end[i]) and decodes
//         into out + i * chunk (128 KiB, lzss.h:21).
//
// Both formats are sequences of byte-aligned items whose sizes follow from
// one header byte (BRLE) or one flag byte per eight items (LZSS). BRLE finds
// a batch by a scalar walk over header bytes that sit in two VGPRs
// (v_readlane, no memory round trip per step), each lane then takes one
// item, and the batch's output is assembled in an LDS ring and stored to HBM
// as 16-byte aligned vectors; two waves per chunk, the walking wave one batch
// ahead of the writing wave. LZSS walks several parts of a chunk at once from
// every byte a group may begin at and resolves its output in an LDS window of
// marks; four waves per chunk. The next input window is loaded meanwhile.
//
// The reference checks nothing; these kernels report per chunk: TRUNCATED if
// the stream ends inside an item, OVERFLOW if the output would pass the
// chunk, CORRUPT for an LZSS offset of 0 or before the chunk start (or a
// chunk whose stream lies outside the input). The items before the first
// error are written; out_len gets the bytes produced.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "kernels.hpp"
#include "window.hpp"

namespace codag {
namespace bytecodec {

using namespace dev;

constexpr int32_t kOk = CODAG_CHUNK_OK;
constexpr int32_t kTrunc = CODAG_CHUNK_TRUNCATED;
constexpr int32_t kOverflow = CODAG_CHUNK_OVERFLOW;
constexpr int32_t kCorrupt = CODAG_CHUNK_CORRUPT;

// LDS input window: 64 lanes x 16 bytes from the 16-byte aligned address at
// or below the first unconsumed stream byte (`lead` bytes before it).
constexpr uint32_t kWin = 1024;
// Header bytes the walk reads lie in window bytes [0, kHead): two VGPRs.
constexpr uint32_t kHead = 512;
// Output ring. LZSS needs the last 2047 bytes as history plus one batch.
constexpr uint32_t kRing = 4096;
constexpr uint32_t kRingMask = kRing - 1;
// Batch output limits: BRLE has no history, LZSS keeps 2047 bytes of it.
// Both leave the < 16 bytes a flush keeps back intact.
constexpr uint32_t kBrleBatch = kRing - 32;
static_assert(kHead + 130 <= kWin && kHead + 17 <= kWin, "items must end inside the window");

// old with lane j's value replaced by the uniform v
__device__ __forceinline__ uint32_t wrlane(uint32_t old, uint32_t v, uint32_t j) {
  return lane_id() == j ? v : old;
}
// ------------------------------------------------------------------ input

// Stream bytes [at, at + kWin - lead) as one 16-byte load per lane. A block
// is loaded only if it holds a byte below the stream end, so no load leaves
// the 16-byte blocks (and pages) the stream occupies.
struct Window {
  uint4 v;
  uint32_t lead;
};

__device__ __forceinline__ Window window_load(const uint8_t *base, uint32_t len, uint32_t at,
                                              uint32_t lane) {
  typedef uint32_t v4u __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(1))) const v4u gvec;
  const uintptr_t a = reinterpret_cast<uintptr_t>(base) + at;
  const uintptr_t a0 = a & ~uintptr_t(15);
  const uintptr_t end = reinterpret_cast<uintptr_t>(base) + len;
  Window w;
  w.lead = (uint32_t)(a - a0);
  w.v = make_uint4(0, 0, 0, 0);
  if (a0 + 16u * lane < end) {
    const v4u q = *reinterpret_cast<gvec *>(a0 + 16u * lane);
    w.v = make_uint4(q.x, q.y, q.z, q.w);
  }
  return w;
}

// Header byte at window index q < kHead from the VGPR copies of window bytes
// [0, 256) (h0) and [256, 512) (h1); q is wave-uniform.
__device__ __forceinline__ uint32_t head_byte(uint32_t h0, uint32_t h1, uint32_t q) {
  const uint32_t l = (q >> 2) & 63u;
  const uint32_t d0 = rdlane(h0, l), d1 = rdlane(h1, l);
  return ((q < 256u ? d0 : d1) >> ((q & 3u) * 8u)) & 0xffu;
}

// ------------------------------------------------------------------ output

// Byte x of the chunk's output sits at ring[(x + mis) & kRingMask], mis =
// dst & 15, so 16-byte aligned output addresses are 16-byte aligned in LDS.
struct Out {
  uint8_t *dst;
  uint8_t *ring;
  uint32_t cap;
  uint32_t pos;      // bytes produced
  uint32_t flushed;  // bytes [0, flushed) are in HBM
  uint32_t mis;
};

__device__ __forceinline__ uint32_t ridx(const Out &o, uint32_t x) { return (x + o.mis) & kRingMask; }

// Stores ring bytes [flushed, end) to HBM: single bytes up to a 16-byte
// aligned address, then 16-byte vectors; `last` also writes the tail,
// otherwise fewer than 16 bytes stay behind.
__device__ __forceinline__ void out_store(Out &o, uint32_t lane, uint32_t end, bool last) {
  uint32_t x = o.flushed;
  uint32_t head = (16u - ((o.mis + x) & 15u)) & 15u;
  if (head > end - x) head = end - x;
  if (head) {
    if (lane < head) o.dst[x + lane] = o.ring[ridx(o, x + lane)];
    x += head;
  }
  const uint32_t nvec = (end - x) / 16u;
  for (uint32_t k = lane; k < nvec; k += kWave) {
    const uint32_t at = x + 16u * k;
    *reinterpret_cast<uint4 *>(o.dst + at) = *reinterpret_cast<const uint4 *>(o.ring + ridx(o, at));
  }
  x += nvec * 16u;
  if (last && x < end) {
    if (lane < end - x) o.dst[x + lane] = o.ring[ridx(o, x + lane)];
    x = end;
  }
  o.flushed = x;
}

__device__ __forceinline__ void chunk_bounds(const uint64_t lo, const uint64_t hi, uint64_t comp_bytes,
                                             uint64_t &len, int32_t &st) {
  st = kOk;
  len = 0;
  if (hi < lo || hi > comp_bytes || hi - lo >= (1ull << 31)) st = kCorrupt;
  else len = hi - lo;
}

// ------------------------------------------------------------------ BRLE

// Two waves per chunk, in lockstep (one workgroup barrier per batch): wave 0
// walks batch i (window staging, header chain, item checks, output offsets)
// while wave 1 writes batch i-1 into the ring and stores it to HBM. The walk
// is scalar-bound and the writing vector/LDS-bound, so the two overlap, and a
// 4096-chunk launch fills all 32 wave slots of a CU instead of 16. Batch i
// uses window buffer i % 3 (the writer still reads i-1's literal bytes while
// the walker stages i) and descriptor buffer i % 2.
struct __align__(16) BrleLds2 {
  uint8_t ring[kRing];
  uint8_t win[3][kWin];
  uint32_t item[2][kWave];  // header index | batch output offset << 16
  uint32_t nk[2];           // items in the batch
  uint32_t base[2];         // output position of the batch's first byte
  uint32_t last;            // the walker's last batch (kNoLast while walking)
};
constexpr uint32_t kNoLast = 0xffffffffu;

__global__ void __launch_bounds__(2 * kWave) brle_chunks2_kernel(const uint8_t *comp,
                                                                 uint64_t comp_bytes,
                                                                 const uint64_t *ptr, uint64_t n,
                                                                 uint64_t chunk_bytes, uint8_t *out,
                                                                 uint64_t *out_len, int32_t *status) {
  __shared__ BrleLds2 S;
  const uint32_t lane = lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x) / kWave;
  const uint64_t ci = blockIdx.x;
  if (ci >= n) return;
  uint64_t len64;
  int32_t err;
  chunk_bounds(ptr[ci], ptr[ci + 1], comp_bytes, len64, err);
  if (err != kOk) {  // both waves leave before any barrier
    if (threadIdx.x == 0) {
      if (out_len) out_len[ci] = 0;
      if (status) status[ci] = err;
    }
    return;
  }
  const uint8_t *src = comp + ptr[ci];
  const uint32_t len = (uint32_t)len64;
  uint8_t *dst = out + ci * chunk_bytes;
  const uint32_t cap = (uint32_t)chunk_bytes;
  if (threadIdx.x == 0) S.last = kNoLast;
  __syncthreads();
  // walker state
  uint32_t at = 0, pos = 0;
  Window w;
  if (wave == 0) w = window_load(src, len, 0, lane);
  // writer state
  Out o;
  o.dst = dst;
  o.ring = S.ring;
  o.cap = cap;
  o.pos = 0;
  o.flushed = 0;
  o.mis = (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 15u);
  for (uint32_t i = 0;; i++) {
    if (wave == 0 && uni(S.last) == kNoLast) {
      uint8_t *win = S.win[i % 3];
      reinterpret_cast<uint4 *>(win)[lane] = w.v;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      const uint32_t lead = uni(w.lead);
      const uint32_t h0 = reinterpret_cast<const uint32_t *>(win)[lane];
      const uint32_t h1 = reinterpret_cast<const uint32_t *>(win)[kWave + lane];
      const uint32_t qend = lead + (len - at);
      const uint32_t qlim = min(qend, kHead);
      uint32_t q = lead, nw = 0, iq = 0;
      while (nw < (uint32_t)kWave && q < qlim) {
        const uint32_t h = head_byte(h0, h1, q);
        iq = wrlane(iq, q, nw);
        nw++;
        q += h > 127u ? h - 126u : 2u;
      }
      const bool act = lane < nw;
      const uint32_t hq = act ? (uint32_t)win[iq] : 0u;
      const bool lit = hq > 127u;
      const uint32_t k = act ? (lit ? hq - 127u : hq + 3u) : 0u;
      const uint32_t inl = lit ? k + 1u : 2u;
      const uint32_t incl = wave_scan_dpp(k);
      const uint32_t bad = !act ? 0u : (iq + inl > qend ? 1u : (pos + incl > cap ? 2u : 0u));
      const uint64_t stop = __ballot(bad != 0u || (act && incl > kBrleBatch));
      uint32_t nk = nw;
      if (stop) {
        nk = (uint32_t)__builtin_ctzll(stop);
        const uint32_t why = rdlane(bad, nk);
        if (why) err = why == 1u ? kTrunc : kOverflow;
        at += rdlane(iq, nk) - lead;
      } else {
        at += q - lead;
      }
      const uint32_t T = nk ? rdlane(incl, nk - 1u) : 0u;
      S.item[i & 1][lane] = iq | ((incl - k) << 16);
      if (lane == 0) {
        S.nk[i & 1] = nk;
        S.base[i & 1] = pos;
        if (err != kOk || at >= len) S.last = i;
      }
      pos += T;
      if (err == kOk && at < len) w = window_load(src, len, at, lane);
    } else if (wave == 1 && i > 0) {
      // write batch i-1
      const uint32_t b = (i - 1) & 1;
      const uint8_t *win = S.win[(i - 1) % 3];
      const uint32_t nk = uni(S.nk[b]);
      const uint32_t it = S.item[b][lane];
      const uint32_t iq = it & 0xffffu, off = it >> 16;
      const uint32_t kk0 = lane < nk ? (uint32_t)win[iq] : 0u;
      const bool lit = kk0 > 127u;
      const uint32_t kk = lane < nk ? (lit ? kk0 - 127u : kk0 + 3u) : 0u;
      const uint32_t s0 = iq + 1u;
      const uint32_t c = kk ? (uint32_t)win[s0] : 0u;
      const uint32_t r0 = uni(S.base[b]) + off + o.mis;
      const uint32_t hb = min((4u - (r0 & 3u)) & 3u, kk);
#pragma unroll
      for (uint32_t t = 0; t < 3u; t++)
        if (t < hb) S.ring[(r0 + t) & kRingMask] = lit ? win[s0 + t] : (uint8_t)c;
      const uint32_t nd = (kk - hb) >> 2;
      const uint32_t c4 = c * 0x01010101u;
      uint32_t *ring32 = reinterpret_cast<uint32_t *>(S.ring);
      const uint32_t *win32 = reinterpret_cast<const uint32_t *>(win);
      for (uint32_t d = 0; d < nd; d++) {
        const uint32_t u = s0 + hb + 4u * d;
        uint32_t v = c4;
        if (lit) {
          const uint32_t a = u >> 2;
          v = __builtin_amdgcn_alignbit(win32[a + 1u], win32[a], (u & 3u) * 8u);
        }
        ring32[((r0 + hb + 4u * d) & kRingMask) >> 2] = v;
      }
      const uint32_t tb = hb + 4u * nd;
#pragma unroll
      for (uint32_t t = 0; t < 3u; t++)
        if (tb + t < kk) S.ring[(r0 + tb + t) & kRingMask] = lit ? win[s0 + tb + t] : (uint8_t)c;
      // the batch's last byte: the largest item end
      uint32_t e = lane < nk ? off + kk : 0u;
#pragma unroll
      for (uint32_t d = 32; d >= 1; d >>= 1) e = max(e, (uint32_t)__shfl_xor(e, (int)d, kWave));
      o.pos = uni(S.base[b]) + uni(e);
      out_store(o, lane, o.pos, false);
    }
    __syncthreads();
    const uint32_t last = uni(S.last);
    if (last != kNoLast && i >= last + 1u) break;
  }
  if (wave == 1) out_store(o, lane, o.pos, true);
  if (wave == 0 && lane == 0) {
    if (out_len) out_len[ci] = pos;
    if (status) status[ci] = err;
  }
}

// ------------------------------------------------------------------ LZSS

// Four waves per chunk. A step takes kParts parts of kPart stream bytes:
//  * Group starts. A group is a flag byte and 8 items, 9 to 17 bytes by the
//    flag's zeros, so the first group of a part starts in its first 17 bytes.
//    Lane (part, entry) walks one part from one of these 17 bytes and notes the
//    starts it passes; the exits are then chained over the parts. 15 parts of
//    17 entries fill 255 lanes, and a step's serial work is the 16 to 23 groups
//    of one part and 15 links instead of one link per group.
//  * Lane i takes group i: its item sizes follow from prefix popcounts of the
//    flag, a prefix sum of the lanes' bytes gives its output position, and it
//    marks its items in the window, which is then resolved (window.hpp).
// One wave per chunk, eight groups at a time and serial where matches overlap,
// was bound by its scalar chain and the latency of two waves a SIMD: 128 KiB
// chunks of text, before and now: 2 chunks 1.59 and 0.41 ms, 512 chunks 1.65 and
// 0.47 ms, 2048 chunks 1.95 and 1.01 ms (bound by vector issue, mostly the
// window's resolving).
constexpr int kLzWaves = 4;
constexpr uint32_t kLzThreads = kLzWaves * kWave;
constexpr uint32_t kParts = 15, kPart = 208, kEntries = 17;
constexpr uint32_t kSteps = (kPart + 8) / 9;  // groups that can start in a part
constexpr uint32_t kLzSeg = 1536, kLzWin = kLzWaves * kLzSeg;
constexpr uint32_t kLzStage = kLzThreads * 16;  // 16 bytes a thread
static_assert(kParts * kEntries <= kLzThreads && kPart < 256, "a lane per part and entry, a byte per start");
static_assert(15 + kParts * kPart + 16 + 17 + 16 <= kLzStage, "the last group of a step lies in the stage");

struct __align__(16) LzssLds {
  uint8_t stage[kLzStage];
  uint16_t win[kLzWin];
  uint8_t start[kSteps * kParts * kEntries];  // [step][part][entry]: a group's start in its part
  uint32_t exits[kLzThreads];                 // [part][entry]: groups << 8 | exit behind the part
  uint32_t part[kLzWaves];
  uint32_t err;
};

// Decodes one LZSS stream of `len` bytes into dst (at most cap bytes) by four
// waves. Every thread returns the same status and byte count.
__device__ __forceinline__ int32_t lzss_stream(const uint8_t *src, uint32_t len, uint8_t *dst, uint32_t cap,
                                               LzssLds &S, uint32_t *produced) {
  const uint32_t lane = lane_id(), tid = threadIdx.x;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid) / kWave;
  uint32_t at = 0, pos = 0, none = 0;
  int32_t err = kOk;
  Window w = window_load(src, len, 0, tid);
  while (at < len && err == kOk) {
    reinterpret_cast<uint4 *>(S.stage)[tid] = w.v;
    __syncthreads();
    const uint8_t *in = S.stage + uni(w.lead);  // stream byte `at`
    const uint32_t left = len - at;
    {
      const uint32_t part = tid / kEntries, lo = part * kPart;
      const uint32_t end = tid < kParts * kEntries ? min(lo + kPart, left) : 0u;
      uint32_t q = lo + tid - part * kEntries, n = 0;
      while (q < end) {
        S.start[n * (kParts * kEntries) + tid] = (uint8_t)(q - lo);
        n++;
        q += 17u - (uint32_t)__popc((uint32_t)in[q]);
      }
      // a part that the stream ends in has no group behind it
      S.exits[tid] = n << 8 | (q >= lo + kPart ? q - (lo + kPart) : 0u);
    }
    __syncthreads();
    // chain the parts: entry of part k and groups before it
    uint32_t x4[kLzWaves];
#pragma unroll
    for (int k = 0; k < kLzWaves; k++) x4[k] = S.exits[k * kWave + lane];
    uint32_t before[kParts], e = 0, groups = 0;
    uint32_t parts = 0;  // lane k: part k's entry, and the groups before it << 8
#pragma unroll
    for (uint32_t k = 0; k < kParts; k++) {
      before[k] = groups;
      parts = lane == k ? groups << 8 | e : parts;
      const uint32_t i = k * kEntries + e;
      const uint32_t a = rdlane(x4[k * kEntries / kWave], i & 63);
      const uint32_t b = rdlane(x4[min((k * kEntries + 16) / (uint32_t)kWave, (uint32_t)kLzWaves - 1)], i & 63);
      const uint32_t x = i / kWave == k * kEntries / kWave ? a : b;
      e = x & 255;
      groups += x >> 8;
    }
    const uint32_t next = kParts * kPart + e;  // stream bytes this step takes
    if (next < left) w = window_load(src, len, at + next, tid);
    // the groups, 256 at a time
    for (uint32_t g0 = 0; g0 < groups && err == kOk; g0 += kLzThreads) {
      const uint32_t g = g0 + tid;
      const bool have = g < groups;
      uint32_t pk = 0;
#pragma unroll
      for (uint32_t k = 1; k < kParts; k++) pk += g >= before[k] ? 1u : 0u;
      const uint32_t of = __shfl(parts, pk, kWave);
      const uint32_t q =
          have ? pk * kPart + S.start[(g - (of >> 8)) * (kParts * kEntries) + pk * kEntries + (of & 255)] : 0u;
      const uint32_t f = in[q];
      // item k: its two bytes (v) and its bytes in the output (tl), 0 past the
      // stream's end; `inside`: the stream ends inside item k
      uint32_t v[8], tl[8], n = 0, inside = 0;
      const bool tail = next >= left;  // uniform: the stream ends in this step
#pragma unroll
      for (uint32_t k = 0; k < 8; k++) {
        const uint32_t ip = q + 1 + 2 * k - (uint32_t)__popc(f & ((1u << k) - 1));
        const bool lit = (f >> k) & 1;
        v[k] = (uint32_t)in[ip] | (uint32_t)in[ip + 1] << 8;
        tl[k] = have ? (lit ? 1u : (v[k] & 31) + 3) : 0u;
        if (tail) {
          if (ip >= left) tl[k] = 0;
          else if (!lit && ip + 2 > left) inside |= 1u << k;
        }
        n += tl[k];
      }
      const uint32_t incl = wave_scan_dpp(n), sum = rdlane(incl, kWave - 1);
      __syncthreads();  // S.part is free
      if (lane == 0) S.part[wave] = sum;
      if (tid == 0) S.err = ~0u;
      __syncthreads();
      uint32_t base = incl - n, total = 0;
#pragma unroll
      for (int k = 0; k < kLzWaves; k++) {
        const uint32_t p = uni(S.part[k]);
        base += k < (int)wave ? p : 0u;
        total += p;
      }
      // the first item that is in error: cut off, without a source, too long
      {
        bool odd = inside || pos + base + n > cap;
        uint32_t x = pos + base;
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
          odd = odd || (!((f >> k) & 1) && tl[k] && (v[k] >> 5) - 1 >= x);
          x += tl[k];
        }
        if (odd) {
          x = base;
#pragma unroll 1
          for (uint32_t k = 0; k < 8; k++) {
            uint32_t vk = 0, tk = 0;
#pragma unroll
            for (uint32_t j = 0; j < 8; j++) {
              vk = j == k ? v[j] : vk;
              tk = j == k ? tl[j] : tk;
            }
            const bool lit = (f >> k) & 1;
            uint32_t bad = 0;
            if ((inside >> k) & 1) bad = (uint32_t)kTrunc;
            else if (!lit && tk && (vk >> 5) - 1 >= pos + x) bad = (uint32_t)kCorrupt;
            else if (pos + x + tk > cap) bad = (uint32_t)kOverflow;
            if (bad) {
              atomicMin(&S.err, x << 2 | bad);
              break;
            }
            x += tk;
          }
        }
      }
      uint32_t done = 0;
      while (done < total) {
        uint32_t wn = min(kLzWin, total - done);
        for (uint32_t k = tid; k < (wn + 511) / 512 * 64; k += kLzThreads)
          reinterpret_cast<uint4 *>(S.win)[k] = make_uint4(~0u, ~0u, ~0u, ~0u);
        __syncthreads();
        if (tid == 0 && wn < kLzWin) S.win[wn] = 0x8000u;
        // a group's items (at most 272 bytes) cross one segment border at most
        uint32_t x = base - done;
        const uint32_t border = base < done ? kLzSeg : (x / kLzSeg + 1) * kLzSeg;
        if (base + n > done && base < done + wn) {
#pragma unroll
          for (uint32_t k = 0; k < 8; k++) {
            const uint32_t m = (f >> k) & 1 ? 0x8000u | (v[k] & 0xff) : (v[k] >> 5) - 1;
            if (x < wn && tl[k]) S.win[x] = (uint16_t)m;
            const uint32_t to = x + tl[k];
            if ((int32_t)x < 0 && (int32_t)to > 0) S.win[0] = (uint16_t)m;  // began in the window before
            if (x < border && to > border && border < kLzWin) S.win[border] = (uint16_t)m;
            x = to;
          }
        }
        __syncthreads();
        const uint32_t es = uni(S.err);
        if (es != ~0u && (es >> 2) < done + wn) {
          wn = (es >> 2) - done;
          err = (int32_t)(es & 3);
        }
        resolve_window<kLzWaves, kLzSeg, false>(dst, S.win, pos + done, wn, wave, lane, none, none);
        __syncthreads();
        done += wn;
        if (err != kOk) break;
      }
      pos += done;
    }
    at += min(next, left);
    __syncthreads();
  }
  *produced = pos;
  return err;
}

// 80 registers: six groups per CU (2048 chunks 1.05 -> 1.01 ms against the 96 of
// five).
__global__ void __launch_bounds__(kLzThreads) __attribute__((amdgpu_waves_per_eu(6)))
lzss_chunks_kernel(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ends, uint64_t n, uint64_t chunk_bytes,
                   uint8_t *out, uint64_t *out_len, int32_t *status) {
  __shared__ LzssLds S;
  const uint64_t i = blockIdx.x;
  if (i >= n) return;
  const uint64_t lo = i ? ends[i - 1] : 0;  // lzss.h:237-238
  uint64_t len;
  int32_t st;
  chunk_bounds(lo, ends[i], comp_bytes, len, st);
  uint32_t produced = 0;
  if (st == kOk)
    st = lzss_stream(comp + lo, (uint32_t)len, out + i * chunk_bytes, (uint32_t)chunk_bytes, S, &produced);
  if (threadIdx.x == 0) {
    if (out_len) out_len[i] = produced;
    if (status) status[i] = st;
  }
}

}  // namespace bytecodec

hipError_t launch_brle_chunks(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ptr,
                              uint64_t n, uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len,
                              int32_t *status, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(bytecodec::brle_chunks2_kernel, dim3((uint32_t)n), dim3(2 * kWaveSize), 0,
                     stream, comp, comp_bytes, ptr, n, chunk_bytes, out, out_len, status);
  return hipGetLastError();
}

hipError_t launch_lzss_chunks(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ends,
                              uint64_t n, uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len,
                              int32_t *status, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(bytecodec::lzss_chunks_kernel, dim3((uint32_t)n), dim3(bytecodec::kLzThreads), 0, stream,
                     comp, comp_bytes, ends, n, chunk_bytes, out, out_len, status);
  return hipGetLastError();
}

}  // namespace codag
