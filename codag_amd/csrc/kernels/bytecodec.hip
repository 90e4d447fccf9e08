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
// one header byte (BRLE) or one flag byte per eight items (LZSS). Both decoders
// find the item starts of many parts of the stream at once: BRLE by walks from
// guessed starts that are put right until they agree, LZSS from every byte a group
// may begin at. BRLE's output is made from its items dword by dword, LZSS's
// resolved in an LDS window of marks. The next part of the stream is loaded
// meanwhile. A second LZSS kernel, one wave per chunk, copies match by match: for
// very compressible streams and many small chunks.
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

__device__ __forceinline__ void chunk_bounds(const uint64_t lo, const uint64_t hi, uint64_t comp_bytes,
                                             uint64_t &len, int32_t &st) {
  st = kOk;
  len = 0;
  if (hi < lo || hi > comp_bytes || hi - lo >= (1ull << 31)) st = kCorrupt;
  else len = hi - lo;
}

// ------------------------------------------------------------------ BRLE

// Four waves per chunk, or one (brle_few in capi.cpp has both sides' times). A step
// takes 64 blocks of 60 stream bytes per wave, one per lane:
//  * Item starts. Only a header above 128 moves on by more than two bytes, so a
//    walk visits every second byte up to the next such byte: one mask operation
//    and one header read per long literal, not one per item. Every lane walks its
//    block from a guessed start (its first byte) and keeps the starts it passes
//    in a mask. A block is entered at the greatest exit before it: a lane whose
//    entry changed walks on from there until it meets a start of its mask, where
//    its former path, and exit, hold again. In runs and text wrong starts have
//    met the right one after 40 bytes in the median and 390 at the 99th
//    percentile, nine passes a step. Where they do not (long literals of any
//    bytes), each wave in turn follows its chain block by block.
//  * Each wave lists its items, with output offsets from a prefix sum, and makes
//    its output in an LDS window: an item marks its first whole dword, a prefix
//    maximum hands each dword its item and one load its bytes; the up to three
//    bytes before and behind an item's whole dwords are then written by item.
// One wave's walk by readlane took about 250 cycles an item, with a second wave
// writing. 1024 chunks of 256 KiB, that way and now, us: runs and text 873 and 264
// (item by item through the headers 449), random bytes 1598 and 740 (by walks alone
// 1837), 16384 chunks of 4 KiB of the former 143 and 70 (by four waves and with
// entries handed on from lane to lane 799). It is bound by latency: of a step's
// cycles about two fifths are the walks and as many the output, with one chunk per
// CU or four.
// 15 dwords: lanes at the same byte of their blocks read different LDS banks
constexpr uint32_t kBrBlock = 60;
constexpr uint32_t kBrList = 512;             // items listed at a time, per wave
constexpr uint32_t kBrOut = 2048;             // a wave's output window
constexpr uint32_t kBrPasses = 24, kBrFew = 2;  // walks before a wave follows its chain block by block; see there
static_assert(kBrBlock <= 64, "the starts of a block in 64 bits");

template <int NW> struct BrCfg {
  static constexpr uint32_t kThreads = NW * kWave;
  static constexpr uint32_t kStep = kThreads * kBrBlock;  // stream bytes in which a step's items begin
  static constexpr uint32_t kStage = (15 + kStep + 129 + 8 + 15) & ~15u;
  static constexpr uint32_t kLoads = (kStage + kThreads * 16 - 1) / (kThreads * 16);
};

template <int NW> struct __align__(16) BrleLds {
  uint8_t stage[BrCfg<NW>::kStage];
  uint32_t list[NW][kBrList];  // literal << 31 | output offset in the wave << 12 | header
  uint32_t out[NW][kBrOut / 4];
  uint32_t exits[2][NW], entry[2][NW], early[NW];
  uint32_t part[NW];
  uint32_t err;
};
constexpr uint32_t kBrSpan = kWave * kBrBlock;  // stream bytes of a wave
static_assert(kBrSpan <= 4096 && kBrSpan / 2 * 130 < (1u << 19), "fields of a list entry");

// Items [0, nb) of a wave's list, their headers counted from stage byte `first`.
struct BrleItems {
  const uint8_t *stage;
  const uint32_t *list;
  uint32_t first, nb;
  struct Item {
    uint32_t at, o, k;  // stage byte of the header, output offset, output bytes (0: none)
    bool lit;
  };
  __device__ __forceinline__ Item get(uint32_t i) const {
    const uint32_t x = list[min(i, nb - 1)];
    Item t;
    t.at = first + (x & 4095u);
    t.lit = (int32_t)x < 0;
    t.o = (x >> 12) & 0x7ffffu;
    const uint32_t h = stage[t.at];
    t.k = i < nb ? (t.lit ? h - 127u : h + 3u) : 0u;
    return t;
  }
};

// Writes the items, output offset 0 being byte o0 of dst, which is 16-byte
// aligned, and their bytes [x0, x1).
template <uint32_t STAGE>
__device__ __forceinline__ void brle_write(uint8_t *dst, const BrleItems &it, uint32_t *ow, uint32_t o0, uint32_t x0,
                                           uint32_t x1, uint32_t lane) {
  uint8_t *ob = reinterpret_cast<uint8_t *>(ow);
  const uint32_t *stage32 = reinterpret_cast<const uint32_t *>(it.stage);
  uint32_t i0 = 0;  // the first item with bytes in the window
  for (uint32_t w0 = x0 & ~15u; w0 < x1; w0 += kBrOut) {
    const int32_t wn = (int32_t)min(kBrOut, x1 - w0);
    const uint32_t ow0 = o0 - w0;
#pragma unroll
    for (uint32_t r = 0; r < kBrOut / 16; r += kWave) reinterpret_cast<uint4 *>(ow)[r + lane] = make_uint4(0, 0, 0, 0);
    lds_order();
    uint32_t i1 = i0;  // behind the window's items
    BrleItems::Item t = it.get(i0 + lane);  // kept for the loop after the next
    for (;;) {
      const int32_t o = (int32_t)(ow0 + t.o), e = o + (int32_t)t.k;
      const int32_t fd = max((o + 3) >> 2, 0), ed = min(e >> 2, (int32_t)(kBrOut / 4));
      if (t.k && fd < ed) ow[fd] = i1 - i0 + lane + 1;
      i1 += kWave;
      if (i1 >= it.nb || (int32_t)rdlane((uint32_t)e, kWave - 1) >= wn) break;
      t = it.get(i1 + lane);
    }
    lds_order();
    // dwords: those not inside one item get bytes that the next loop replaces
    uint32_t carry = 1;
    for (int32_t r0 = 0; 4 * r0 < wn; r0 += 4 * kWave) {
      uint32_t m[4], x[4], a[4], lo[4], hi[4];
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) m[r] = ow[r0 + r * kWave + lane];
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) {
        m[r] = max(wave_max_dpp(m[r]), carry);
        carry = rdlane(m[r], kWave - 1);
      }
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) x[r] = it.list[i0 + m[r] - 1];
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) {
        const uint32_t in_item = 4 * (r0 + r * kWave + lane) - ow0 - ((x[r] >> 12) & 0x7ffffu);
        const int32_t b = (int32_t)(it.first + 1 + (x[r] & 4095u) + ((int32_t)x[r] < 0 ? in_item : 0u));
        a[r] = (uint32_t)min(max(b, 0), (int32_t)STAGE - 8);
        lo[r] = stage32[a[r] >> 2];
        hi[r] = stage32[(a[r] >> 2) + 1];
      }
#pragma unroll
      for (uint32_t r = 0; r < 4; r++) {
        const uint32_t v = __builtin_amdgcn_alignbyte(hi[r], lo[r], a[r] & 3u);
        ow[r0 + r * kWave + lane] = (int32_t)x[r] < 0 ? v : __builtin_amdgcn_perm(0u, v, 0u);
      }
    }
    lds_order();
    for (uint32_t i = i0;; i += kWave) {
      if (i1 - i0 > kWave) t = it.get(i + lane);
      const int32_t o = (int32_t)(ow0 + t.o), e = o + (int32_t)t.k;
      const int32_t hend = min((o + 3) & ~3, e), tbeg = max(e & ~3, hend);
      // the bytes from the item's first one on, and from its byte tbeg on
      const uint32_t ha = t.at + 1, ta = ha + (t.lit ? (uint32_t)(tbeg - o) : 0u);
      const uint32_t h0 = stage32[ha >> 2], h1 = stage32[(ha >> 2) + 1];
      const uint32_t t0 = stage32[ta >> 2], t1 = stage32[(ta >> 2) + 1];
      uint32_t hv = __builtin_amdgcn_alignbyte(h1, h0, ha & 3u), tv = __builtin_amdgcn_alignbyte(t1, t0, ta & 3u);
      hv = t.lit ? hv : __builtin_amdgcn_perm(0u, hv, 0u);
      tv = t.lit ? tv : __builtin_amdgcn_perm(0u, tv, 0u);
      const int32_t hn = o >= 0 && o < wn ? hend - o : 0, tn = tbeg >= 0 && tbeg < wn ? e - tbeg : 0;
#pragma unroll
      for (int32_t j = 0; j < 3; j++)
        if (j < hn) ob[o + j] = (uint8_t)(hv >> 8 * j);
#pragma unroll
      for (int32_t j = 0; j < 3; j++)
        if (j < tn) ob[tbeg + j] = (uint8_t)(tv >> 8 * j);
      const uint64_t past = __ballot(t.k && e > (int32_t)kBrOut);
      if (past || i + kWave >= i1) {
        i0 = min(past ? i + (uint32_t)__builtin_ctzll(past) : i1, it.nb - 1);
        break;
      }
    }
    lds_order();
    // whole vectors, then the bytes before and behind them
#pragma unroll
    for (uint32_t r = 0; r < kBrOut / 16; r += kWave) {
      const uint32_t x = w0 + 16 * (r + lane);
      if (x >= x0 && x + 16 <= x1) *reinterpret_cast<uint4 *>(dst + x) = reinterpret_cast<const uint4 *>(ow)[r + lane];
    }
    if (w0 < x0) {
      const uint32_t x = w0 + lane;
      if (lane < 16 && x >= x0 && x < x1) dst[x] = ob[lane];
    }
    const uint32_t xt = x1 & ~15u;
    if (xt >= x0 && xt >= w0 && xt - w0 < kBrOut) {
      const uint32_t x = xt + lane;
      if (x < x1) dst[x] = ob[x - w0];
    }
    lds_order();
  }
}

template <int NW>
__global__ void __launch_bounds__(NW *kWave) __attribute__((amdgpu_waves_per_eu(5)))
brle_chunks_kernel(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ptr, uint64_t n, uint64_t chunk_bytes,
                   uint8_t *out, uint64_t *out_len, int32_t *status) {
  constexpr int kBrWaves = NW;
  constexpr uint32_t kBrThreads = BrCfg<NW>::kThreads, kBrStage = BrCfg<NW>::kStage, kBrLoads = BrCfg<NW>::kLoads;
  __shared__ BrleLds<NW> S;
  const uint32_t lane = lane_id(), tid = threadIdx.x;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const uint64_t ci = blockIdx.x;
  if (ci >= n) return;
  uint64_t len64;
  int32_t err;
  chunk_bounds(ptr[ci], ptr[ci + 1], comp_bytes, len64, err);
  if (err != kOk) {  // every wave leaves before any barrier
    if (tid == 0) {
      if (out_len) out_len[ci] = 0;
      if (status) status[ci] = err;
    }
    return;
  }
  const uint8_t *src = comp + ptr[ci];
  const uint32_t len = (uint32_t)len64, cap = (uint32_t)chunk_bytes;
  uint8_t *dst = out + ci * chunk_bytes;
  const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 15u);
  uint32_t at = 0, pos = 0, lead = 0, passes = kBrPasses;
  uint4 v[kBrLoads];
  auto load = [&](uint32_t from) __attribute__((always_inline)) {
    lead = (uint32_t)(reinterpret_cast<uintptr_t>(src) + from) & 15u;
#pragma unroll
    for (uint32_t k = 0; k < kBrLoads; k++) {
      const uint32_t i = k * kBrThreads + tid;
      if (i < kBrStage / 16) v[k] = window_load(src, len, from, i).v;
    }
  };
  load(0);
  while (at < len && err == kOk) {
#pragma unroll
    for (uint32_t k = 0; k < kBrLoads; k++) {
      const uint32_t i = k * kBrThreads + tid;
      if (i < kBrStage / 16) reinterpret_cast<uint4 *>(S.stage)[i] = v[k];
    }
    if (tid == 0) S.err = ~0u;
    if (tid < kBrWaves) S.early[tid] = (tid + 1) * kBrSpan;
    __syncthreads();
    // positions are stage bytes from here on; the stream's next byte is in0, and
    // it ends at `limit`
    const uint8_t *in = S.stage;
    const uint32_t in0 = lead, limit = in0 + (len - at);
    const uint32_t lo = tid * kBrBlock, hi = min(lo + kBrBlock, limit);
    // the block's bytes above 128; every other header is two bytes before the next
    uint64_t jumps = 0;
#pragma unroll
    for (uint32_t k = 0; k < kBrBlock / 4; k++) {
      const uint32_t d = reinterpret_cast<const uint32_t *>(in + lo)[k];
      const uint32_t t = ((d & 0x7f7f7f7fu) + 0x7f7f7f7fu) & d & 0x80808080u;
      jumps |= (uint64_t)__builtin_amdgcn_udot4(t >> 7, 0x08040201u, 0u, false) << (4 * k);
    }
    uint64_t mask = 0;  // the starts of the lane's items, from byte `from` on
    uint32_t from = wave == 0 && lane == 0 ? in0 : lo, exit = 0;
    auto walk = [&]() __attribute__((always_inline)) {
      const uint64_t old = mask, every2 = (uint64_t)0x5555555555555555ull;
      mask = 0;
      uint32_t q = from;
      while (q < hi) {
        // steps of two up to and with the next byte above 128, or the block's end
        const uint64_t path = (every2 << (q - lo)) & (((uint64_t)1 << (hi - lo)) - 1), j = path & jumps;
        const uint64_t p = path & (j ^ (j - 1));
        const uint64_t met = p & old;
        if (met) {
          const uint64_t bit = met & (0 - met);
          mask |= (p & (bit - 1)) | (old & (0 - bit));
          q = exit;
          break;
        }
        mask |= p;
        if (!j) {
          q = hi + ((q ^ hi) & 1u);
        } else {
          q = lo + (uint32_t)__builtin_ctzll(j);
          q += in[q] - 126u;
        }
      }
      exit = q;
    };
    // The wave's chain from byte q on, block by block in scalars, where its lanes do
    // not find each other: the starts that count lie far apart then (long literals),
    // and many blocks are passed over.
    bool chained = false;
    auto chain = [&](uint32_t q) __attribute__((always_inline)) {
      const uint32_t base = wave * kBrSpan, stop = min(base + kBrSpan, limit), entry = q;
      mask = 0;
      from = exit = 0;
      while (q < stop) {
        const uint32_t l = (q - base) / kBrBlock, l0 = base + l * kBrBlock, l1 = min(l0 + kBrBlock, limit);
        const uint64_t js = (uint64_t)rdlane((uint32_t)(jumps >> 32), l) << 32 | rdlane((uint32_t)jumps, l);
        const uint32_t q0 = q;
        uint64_t m = 0;
        while (q < l1) {
          const uint64_t path = ((uint64_t)0x5555555555555555ull << (q - l0)) & (((uint64_t)1 << (l1 - l0)) - 1), j = path & js;
          m |= path & (j ^ (j - 1));
          if (!j) {
            q = l1 + ((q ^ l1) & 1u);
          } else {
            q = l0 + (uint32_t)__builtin_ctzll(j);
            q += uni(in[q]) - 126u;
          }
        }
        if (lane == l) {
          mask = m;
          from = q0;
          exit = q;
        }
      }
      chained = true;
      // the blocks passed over
      const uint32_t incl = wave_max_dpp(exit);
      const uint32_t x = max((uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xf, 0xf, false), entry);
      if (lo < limit && !exit) from = exit = x;
    };
    walk();
    // a block behind the stream's end has no part in what follows
    const bool mine = lo < limit;
    const uint32_t blocks = (uint32_t)__builtin_popcountll(__ballot(mine));
    exit = mine ? exit : 0u;
    uint32_t entry = wave ? wave * kBrSpan : in0, end;  // entry of the wave's first lane, exit of the step
    for (uint32_t round = 0;; round++) {
      const uint32_t r = round & 1;
      uint32_t top = 0;  // the wave's exit
      // where chains are followed one by one, a wave waits for the one before it
      const bool ready = passes == kBrPasses || wave <= round;
      for (uint32_t pass = 0; ready; pass++) {
        // Right exits grow from lane to lane, so a block is entered at the greatest exit
        // before it: an item that passes whole blocks reaches the one it ends in at once.
        const uint32_t incl = wave_max_dpp(exit);
        // what the wave before has now; the check below is made on final exits
        if (wave) entry = uni(__hip_atomic_load(&S.early[wave - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        top = max(rdlane(incl, kWave - 1), entry);
        if (lane == 0) __hip_atomic_store(&S.early[wave], top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t x = max((uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xf, 0xf, false), entry);  // wave_shr:1
        const uint64_t wrong = __ballot(mine && x != from);
        if (!wrong) break;
        // where walks meet, few blocks are left after three
        if (pass < passes && (pass < 3 || 8 * (uint32_t)__builtin_popcountll(wrong) <= 3 * blocks)) {
          if (mine && x != from) {
            from = x;
            walk();
          }
        } else {
          chain(entry);
        }
      }
      if (lane == 0) {
        S.exits[r][wave] = top;
        S.entry[r][wave] = ready ? entry : ~0u;  // no exit: another round
      }
      __syncthreads();
      bool all = true;
#pragma unroll
      for (int k = 1; k < kBrWaves; k++) {
        const uint32_t x = uni(S.exits[r][k - 1]);
        all = all && x == uni(S.entry[r][k]);
        entry = k == (int)wave ? x : entry;
      }
      end = uni(S.exits[r][kBrWaves - 1]);
      if (all) break;
    }
    if (end < limit) load(at + (end - in0));
    // while a third of the blocks and more are passed over, the next steps come to the
    // chain after kBrFew walks
    if (chained) passes = __builtin_popcountll(__ballot(mask != 0)) <= 42 ? kBrFew : kBrPasses;
    // output bytes and items, of the lane and before it: a header h is 3 + h bytes, one
    // above 127 is 130 fewer
    uint32_t n = 3 * (uint32_t)__builtin_popcountll(mask);
#pragma unroll
    for (uint32_t k = 0; k < kBrBlock / 4; k++) {
      const uint32_t d = reinterpret_cast<const uint32_t *>(in + lo)[k];
      const uint32_t ones = (((uint32_t)(mask >> (4 * k)) & 15u) * 0x204081u) & 0x01010101u;  // bytes with a start
      n = __builtin_amdgcn_udot4(d, ones, n, false) - 130u * (uint32_t)__popc(d & ones << 7);
    }
    uint32_t incl = wave_scan_dpp(n | (uint32_t)__builtin_popcountll(mask) << 20);
    if (lane == kWave - 1) S.part[wave] = incl & 0xfffffu;
    __syncthreads();
    uint32_t base = 0, total = 0;
#pragma unroll
    for (int k = 0; k < kBrWaves; k++) {
      const uint32_t p = uni(S.part[k]);
      base += k < (int)wave ? p : 0u;
      total += p;
    }
    const uint32_t room = cap - pos;
    if (end > limit || total > room) {  // items from the first error on are left out
      uint32_t o = base + (incl & 0xfffffu) - n;
      n = 0;
      for (uint64_t m = mask; m; m &= m - 1) {
        const uint32_t q = lo + (uint32_t)__builtin_ctzll(m), h = in[q];
        const uint32_t k = h > 127u ? h - 127u : h + 3u;
        const uint32_t bad =
            q + (h > 127u ? h - 126u : 2u) > limit ? (uint32_t)kTrunc : (o + k > room ? (uint32_t)kOverflow : 0u);
        if (bad) {
          atomicMin(&S.err, o << 2 | bad);
          mask &= (m & (0 - m)) - 1;
          break;
        }
        o += k;
        n += k;
      }
      incl = wave_scan_dpp(n | (uint32_t)__builtin_popcountll(mask) << 20);
    }
    const uint32_t items = rdlane(incl, kWave - 1) >> 20;
    const uint32_t o0 = pos + base + mis;
    BrleItems it{S.stage, S.list[wave], wave * kBrSpan, 0};
    for (uint32_t b0 = 0; b0 < items; b0 += kBrList) {
      uint32_t i = (incl >> 20) - (uint32_t)__builtin_popcountll(mask) - b0;
      uint32_t o = (incl & 0xfffffu) - n;
      for (uint64_t m = mask; m;) {  // the headers of four items are read together
        uint32_t q[4], h[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          q[k] = m ? lo + (uint32_t)__builtin_ctzll(m) : ~0u;
          m &= m - 1;
          h[k] = in[min(q[k], kBrStage - 1)];
        }
#pragma unroll
        for (int k = 0; k < 4; k++, i++) {
          if (q[k] != ~0u && i < kBrList) S.list[wave][i] = (h[k] & 0x80u) << 24 | o << 12 | (q[k] - wave * kBrSpan);
          o += h[k] > 127u ? h[k] - 127u : h[k] + 3u;
        }
      }
      lds_order();
      it.nb = min(items - b0, kBrList);
      const uint32_t f = uni(it.get(0).o);
      const BrleItems::Item l = it.get(it.nb - 1);
      brle_write<kBrStage>(dst - mis, it, S.out[wave], o0, o0 + f, o0 + uni(l.o + l.k), lane);
    }
    __syncthreads();
    const uint32_t es = uni(S.err);
    if (es != ~0u) err = (int32_t)(es & 3u);
    pos += es != ~0u ? es >> 2 : total;
    at += end - in0;
    __syncthreads();
  }
  if (tid == 0) {
    if (out_len) out_len[ci] = pos;
    if (status) status[ci] = err;
  }
}

// ------------------------------------------------------------------ LZSS

// Four waves per chunk, or one (lzss_waves in capi.cpp has both sides' times). A
// step takes kParts parts of kPart stream bytes (of four waves 15, of one 3):
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
// 0.47 ms, 2048 chunks 1.95 and 0.94 ms (bound by vector issue, mostly the
// window's resolving).
constexpr uint32_t kPart = 208, kEntries = 17;
constexpr uint32_t kSteps = (kPart + 8) / 9;  // groups that can start in a part
constexpr uint32_t kLzSeg = 1536;

template <int NW> struct __align__(16) LzssLds {
  static constexpr uint32_t kThreads = NW * kWave;
  static constexpr uint32_t kParts = kThreads / kEntries;
  static constexpr uint32_t kWin = NW * kLzSeg;
  static constexpr uint32_t kStage = kThreads * 16;  // 16 bytes a thread
  static_assert(kPart < 256, "a byte per start");
  static_assert(15 + kParts * kPart + 16 + 17 + 16 <= kStage, "the last group of a step lies in the stage");
  uint8_t stage[kStage];
  uint16_t win[kWin];
  uint8_t start[kSteps * kParts * kEntries];  // [step][part][entry]: a group's start in its part
  uint32_t exits[kThreads];                   // [part][entry]: groups << 8 | exit behind the part
  uint32_t part[NW];
  uint32_t err;
};

// Decodes one LZSS stream of `len` bytes into dst (at most cap bytes) by NW
// waves. Every thread returns the same status and byte count.
template <int NW>
__device__ __forceinline__ int32_t lzss_stream(const uint8_t *src, uint32_t len, uint8_t *dst, uint32_t cap,
                                               LzssLds<NW> &S, uint32_t *produced) {
  constexpr uint32_t kLzThreads = LzssLds<NW>::kThreads, kParts = LzssLds<NW>::kParts, kLzWin = LzssLds<NW>::kWin;
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
    uint32_t x4[NW];
#pragma unroll
    for (int k = 0; k < NW; k++) x4[k] = S.exits[k * kWave + lane];
    uint32_t before[kParts], e = 0, groups = 0;
    uint32_t parts = 0;  // lane k: part k's entry, and the groups before it << 8
#pragma unroll
    for (uint32_t k = 0; k < kParts; k++) {
      before[k] = groups;
      parts = lane == k ? groups << 8 | e : parts;
      const uint32_t i = k * kEntries + e;
      const uint32_t a = rdlane(x4[k * kEntries / kWave], i & 63);
      const uint32_t b = rdlane(x4[min((k * kEntries + 16) / (uint32_t)kWave, (uint32_t)NW - 1)], i & 63);
      const uint32_t x = i / kWave == k * kEntries / kWave ? a : b;
      e = x & 255;
      groups += x >> 8;
    }
    const uint32_t next = kParts * kPart + e;  // stream bytes this step takes
    if (next < left) w = window_load(src, len, at + next, tid);
    // the groups, one a thread at a time
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
      for (int k = 0; k < NW; k++) {
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
        resolve_window<NW, kLzSeg, false, true>(dst, S.win, pos + done, wn, wave, lane, none, none);
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

// 80 registers: six waves per SIMD (2048 chunks 1.05 -> 1.01 ms against the 96 of
// five).
template <int NW>
__global__ void __launch_bounds__(LzssLds<NW>::kThreads) __attribute__((amdgpu_waves_per_eu(6)))
lzss_chunks_kernel(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ends, uint64_t n, uint64_t chunk_bytes,
                   uint8_t *out, uint64_t *out_len, int32_t *status) {
  __shared__ LzssLds<NW> S;
  const uint64_t i = blockIdx.x;
  if (i >= n) return;
  const uint64_t lo = i ? ends[i - 1] : 0;  // lzss.h:237-238
  uint64_t len;
  int32_t st;
  chunk_bounds(lo, ends[i], comp_bytes, len, st);
  uint32_t produced = 0;
  if (st == kOk)
    st = lzss_stream<NW>(comp + lo, (uint32_t)len, out + i * chunk_bytes, (uint32_t)chunk_bytes, S, &produced);
  if (threadIdx.x == 0) {
    if (out_len) out_len[i] = produced;
    if (status) status[i] = st;
  }
}

// One wave per chunk, eight groups at a time, lane 8g + k holding item k of group g;
// the output goes through a ring of LDS. Literals and matches with sources before
// the eight groups are written by all lanes at once, other matches one after the
// other, a match a step. A byte costs next to nothing in a long match, and a chunk
// next to nothing in setup, so this is the kernel for very compressible streams and
// for many small chunks (see lzss_serial in capi.cpp for both kernels' times).
constexpr uint32_t kLsWin = 1024;   // staged stream bytes, 16 a lane
constexpr uint32_t kLsHead = 512;   // flag bytes the walk reads lie in these: two registers
constexpr uint32_t kLsRing = 4096;  // 2047 bytes of history, a batch, and the < 16 bytes a store keeps back
constexpr uint32_t kLsBatch = kLsRing - 2048 - 16;
static_assert(kLsHead + 17 <= kLsWin && 7 * 8 * 34 <= kLsBatch, "items end in the window; seven groups fit a batch");

struct __align__(16) LzssSerialLds {
  uint8_t ring[kLsRing];
  uint8_t win[kLsWin];
};

__global__ void __launch_bounds__(kWave)
lzss_serial_kernel(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ends, uint64_t n, uint64_t chunk_bytes,
                   uint8_t *out, uint64_t *out_len, int32_t *status) {
  __shared__ LzssSerialLds S;
  const uint32_t lane = lane_id(), g = lane >> 3, k = lane & 7u;
  const uint64_t ci = blockIdx.x;
  if (ci >= n) return;
  const uint64_t begin = ci ? ends[ci - 1] : 0;  // lzss.h:237-238
  uint64_t len64;
  int32_t err;
  chunk_bounds(begin, ends[ci], comp_bytes, len64, err);
  const uint8_t *src = comp + begin;
  const uint32_t len = (uint32_t)len64, cap = (uint32_t)chunk_bytes;
  uint8_t *dst = out + ci * chunk_bytes;
  // output byte x is ring byte (x + mis) mod kLsRing, so 16-byte aligned addresses stay so
  const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(dst) & 15u);
  auto at_ring = [&](uint32_t x) -> uint8_t & { return S.ring[(x + mis) & (kLsRing - 1)]; };
  uint32_t pos = 0, flushed = 0, at = 0;
  // bytes up to a 16-byte boundary, then vectors; the last call also writes the tail
  auto store = [&](bool last) {
    uint32_t x = flushed;
    const uint32_t head = min((0u - (mis + x)) & 15u, pos - x);
    if (lane < head) dst[x + lane] = at_ring(x + lane);
    x += head;
    const uint32_t nvec = (pos - x) / 16u;
    for (uint32_t i = lane; i < nvec; i += kWave)
      *reinterpret_cast<uint4 *>(dst + x + 16 * i) = *reinterpret_cast<const uint4 *>(&at_ring(x + 16 * i));
    x += nvec * 16u;
    if (last) {
      if (lane < pos - x) dst[x + lane] = at_ring(x + lane);
      x = pos;
    }
    flushed = x;
  };
  Window w = window_load(src, len, 0, lane);
  while (at < len && err == kOk) {
    lds_order();
    reinterpret_cast<uint4 *>(S.win)[lane] = w.v;
    lds_order();
    const uint32_t lead = uni(w.lead), qend = lead + (len - at);
    const uint32_t h0 = reinterpret_cast<const uint32_t *>(S.win)[lane];
    const uint32_t h1 = reinterpret_cast<const uint32_t *>(S.win)[kWave + lane];
    // walk over the flag bytes: group j's start -> lane j of gq
    uint32_t q = lead, ng = 0, gq = 0;
    while (ng < 8u && q < kLsHead && q < qend) {
      const uint32_t l = (q >> 2) & 63u, d0 = rdlane(h0, l), d1 = rdlane(h1, l);
      const uint32_t f = ((q < 256u ? d0 : d1) >> 8 * (q & 3u)) & 255u;
      gq = lane == ng ? q : gq;
      ng++;
      q += 17u - (uint32_t)__builtin_popcount(f);
    }
    // items (lzss.h:268-303)
    const uint32_t gs = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(g << 2), (int)gq), f = S.win[gs];
    const uint32_t ip = gs + 1u + 2u * k - (uint32_t)__builtin_popcount(f & ((1u << k) - 1u));
    const bool exists = g < ng && ip < qend;
    const bool lit = exists && ((f >> k) & 1u), mat = exists && !lit;
    const uint32_t b0 = S.win[ip], v = b0 | (uint32_t)S.win[ip + 1u] << 8;
    const uint32_t mlen = (v & 31u) + 3u, off = v >> 5;
    const uint32_t tl = lit ? 1u : (mat ? mlen : 0u);
    const uint32_t incl = wave_scan_dpp(tl);
    // an eighth group that would take the batch past kLsBatch waits
    const uint32_t keep_g = rdlane(incl, kWave - 1) > kLsBatch ? 7u : ng;
    const uint32_t x = pos + incl - tl;
    uint32_t e = 0;
    if (g < keep_g && exists) {
      if (mat && ip + 2u > qend) e = (uint32_t)kTrunc;
      else if (mat && (off == 0u || off > x)) e = (uint32_t)kCorrupt;
      else if (x + tl > cap) e = (uint32_t)kOverflow;
    }
    const uint64_t em = __ballot(e != 0u);
    uint32_t nk = keep_g * 8u;  // lanes kept (items past the stream end have tl 0)
    if (em) {
      nk = (uint32_t)__builtin_ctzll(em);
      err = (int32_t)rdlane(e, nk);
    }
    const bool keep = lane < nk;
    const uint32_t pend = pos + (nk ? rdlane(incl, nk - 1u) : 0u);
    // the kept groups are consumed (the last may end at the stream's end)
    at += (keep_g < ng ? rdlane(gq, keep_g) : min(q, qend)) - lead;
    if (err == kOk && at < len) w = window_load(src, len, at, lane);
    if (keep && lit) at_ring(x) = (uint8_t)b0;
    // matches whose source ends before the batch: all lanes at once, 4 bytes a
    // step (bytes past a match's end repeat its last byte's copy)
    const bool km = keep && mat, ind = km && (x - off) + mlen <= pos;
    if (__ballot(ind)) {
      const uint32_t sp = x - off, last = mlen - 1u;
      for (uint32_t i = 0; i < 34u; i += 4u) {
        if (!__ballot(ind && i < mlen)) break;
        if (ind && i < mlen) {
          const uint32_t k1 = min(i + 1u, last), k2 = min(i + 2u, last), k3 = min(i + 3u, last);
          const uint8_t c0 = at_ring(sp + i), c1 = at_ring(sp + k1), c2 = at_ring(sp + k2), c3 = at_ring(sp + k3);
          at_ring(x + i) = c0;
          at_ring(x + k1) = c1;
          at_ring(x + k2) = c2;
          at_ring(x + k3) = c3;
        }
      }
    }
    // the others read bytes of this batch: in stream order, one per step; byte i is
    // source byte i, or i mod oj where the match overlaps itself (lzss.h:285-288)
    for (uint64_t dm = __ballot(km && !ind); dm; dm &= dm - 1) {
      const uint32_t j = (uint32_t)__builtin_ctzll(dm);
      const uint32_t xj = rdlane(x, j), oj = rdlane(off, j), lj = rdlane(mlen, j);
      lds_order();
      if (lane < lj) {
        uint32_t m = lane;  // lane + 0.5 is at least 0.5 away from a multiple of oj: the quotient is exact
        if (oj < lj) m -= __umul24((uint32_t)(((float)lane + 0.5f) * __builtin_amdgcn_rcpf((float)oj)), oj);
        at_ring(xj + lane) = at_ring(xj - oj + m);
      }
    }
    lds_order();
    pos = pend;
    store(false);
  }
  lds_order();
  store(true);
  if (lane == 0) {
    if (out_len) out_len[ci] = pos;
    if (status) status[ci] = err;
  }
}

}  // namespace bytecodec

hipError_t launch_brle_chunks(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ptr,
                              uint64_t n, uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len,
                              int32_t *status, hipStream_t stream, bool few) {
  if (n == 0) return hipSuccess;
  if (few)
    hipLaunchKernelGGL(bytecodec::brle_chunks_kernel<1>, dim3((uint32_t)n), dim3(kWaveSize), 0, stream, comp, comp_bytes,
                       ptr, n, chunk_bytes, out, out_len, status);
  else
    hipLaunchKernelGGL(bytecodec::brle_chunks_kernel<4>, dim3((uint32_t)n), dim3(4 * kWaveSize), 0, stream, comp,
                       comp_bytes, ptr, n, chunk_bytes, out, out_len, status);
  return hipGetLastError();
}

hipError_t launch_lzss_chunks(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *ends,
                              uint64_t n, uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len,
                              int32_t *status, hipStream_t stream, uint32_t waves) {
  if (n == 0) return hipSuccess;
  if (waves == 0)
    hipLaunchKernelGGL(bytecodec::lzss_serial_kernel, dim3((uint32_t)n), dim3(kWaveSize), 0, stream, comp, comp_bytes,
                       ends, n, chunk_bytes, out, out_len, status);
  else if (waves == 1)
    hipLaunchKernelGGL(bytecodec::lzss_chunks_kernel<1>, dim3((uint32_t)n), dim3(kWaveSize), 0, stream, comp,
                       comp_bytes, ends, n, chunk_bytes, out, out_len, status);
  else
    hipLaunchKernelGGL(bytecodec::lzss_chunks_kernel<4>, dim3((uint32_t)n), dim3(4 * kWaveSize), 0, stream, comp,
                       comp_bytes, ends, n, chunk_bytes, out, out_len, status);
  return hipGetLastError();
}

}  // namespace codag
