// rlev1_pipe.hip -- ORC RLE v1 decode: one workgroup per chunk running a
// software pipeline over fixed 2 KiB windows of the chunk's stream.
//
// Segment chain in terminator numbers. Every RLE v1 segment ends on a varint
// terminator (a byte < 0x80). Number the stream's terminators 1, 2, ... and
// let 0 stand for the byte before the stream. The segment whose header
// follows terminator r ends on terminator
//   r + k                      literal group of k varints (header >= 0x80),
//   r + 2 + [delta byte < 0x80] run: the header itself (< 0x80) is r + 1,
// so the walk from header to header needs, per step, only the two bytes
// after terminator r (ent[r]). The walker holds its window's entries in its
// own registers and reads one per segment with register indexing and
// v_readlane -- no memory access on the walker's critical path.
//
// Pipeline (phase k, one workgroup barrier per phase):
//   helpers (waves 1-7; waves 1-2 load, stage and index)
//     load   : window k+2, 16 bytes per lane, into registers (HBM latency is
//              hidden behind two phases);
//     stage  : window k into an LDS ring of four windows; per 16-byte block
//              the terminator count;
//     index  : window k-1: block prefix sums number the terminators; for
//              each, sel = its ring position and ent = the two bytes after;
//     expand : window k-3, one lane per output value;
//   walker (wave 0): window k-2's part of the chain in scalar registers,
//              one descriptor per segment.
// Windows are fixed slices of the address range, so loading and indexing
// never wait for the walk. A segment may run into the next window, which is
// indexed before the segment is expanded (a well-formed segment spans at
// most 1 + 128 * 10 bytes < one window).
//
// Semantics and status follow include/rlev1/decoder.h:671-791 as restated in
// the oracle (first error in stream order): the walker reports a missing
// header byte or delta byte (TRUNCATED) and a segment that overflows the
// chunk (OVERFLOW at value index cap); the expanders report varints longer
// than 10 bytes (CORRUPT) and varints with no terminator among the indexed
// windows (TRUNCATED when the stream ends there; otherwise the varint is
// overlong and ends CORRUPT if any terminator follows, TRUNCATED if none).
#include "device.hpp"
#include "kernels.hpp"

namespace codag {
namespace rle1p {

using namespace codag::dev;

enum : int32_t { kOk = 0, kTrunc = 1, kOverflow = 2, kCorrupt = 3 };

constexpr uint32_t kWin = 2048;            // window bytes
constexpr uint32_t kBlocks = kWin / 16;    // 16-byte blocks per window
constexpr uint32_t kHelpers = 7;
constexpr uint32_t kThreads = kWave * (1 + kHelpers);
static_assert(kHelpers == 7, "expansion passes are dealt in rounds of 1 + 1 + 5 * 2");
constexpr uint32_t kRing = 4 * kWin;       // LDS byte ring
constexpr uint32_t kMirror = 32;           // copy of the ring's first bytes past its end
constexpr uint32_t kTerms = kWin + 2;      // terminators of one window (<= kWin: window 0's byte
                                           // before the stream stands for terminator 0)
constexpr uint32_t kDescs = kWin / 2 + 4;  // segments starting in one window (each spans >= 2 bytes)
constexpr uint32_t kTabRegs = kWin / 2 / kWave;  // walker registers holding a window's ent
constexpr uint32_t kMaxCap = 1u << 21;      // values per chunk (descriptor field)
constexpr uint32_t kSpare = kTerms - 1;    // sel / ent entry written for non-terminator bytes
constexpr uint32_t kNone = 0xffffffffu;

// Error keys: (value index << 2 | priority) << 32 | window. The smallest key
// is the first error in stream order; at one value index a varint read error
// comes before the overflow it would otherwise have hit.
enum : uint32_t { kPrCorrupt = 0, kPrTrunc = 1, kPrPending = 2, kPrOverflow = 3 };
constexpr uint64_t kNoKey = ~0ull;

struct Lds {
  uint8_t sbuf[kRing + kMirror];
  uint16_t sel[3][kTerms];     // ring byte offset of each terminator
  uint16_t ent[2][kTerms];     // the two stream bytes after each terminator
  uint32_t desc[2][kDescs];    // segment: r - T_w (11 bits) | first value index << 11
  uint8_t bcnt[2][kBlocks];    // terminators per 16-byte block
  uint32_t T[8];               // T[j & 7]: number of window j's first terminator
  uint32_t wnd[2][4];          // walked window: segments, first value, end value
  uint8_t mark[kHelpers][kWave];
  uint32_t last_w;             // window in which the walker stopped
  uint32_t lastterm;           // the stream's last byte is a terminator (or the stream is empty)
  uint64_t key;
};

// Bit j set where byte j of the 16-byte block is < 0x80.
__device__ __forceinline__ uint32_t term_mask16(const uint4 &x) {
  const uint32_t q[4] = {x.x, x.y, x.z, x.w};
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t n = ~q[i] & 0x80808080u;
    m |= (((n >> 7) & 1) | ((n >> 14) & 2) | ((n >> 21) & 4) | ((n >> 28) & 8)) << (4 * i);
  }
  return m;
}

// 16 bytes at window block b (offset a0 + w*kWin + 16*b) if the block holds
// a stream byte, else zeros; the last block also fetches the first dword of
// the next window. Only blocks that hold stream bytes are read, so no load
// leaves the pages the stream occupies.
__device__ __forceinline__ void load_block(uintptr_t a0, uint32_t w, uint32_t b, uintptr_t s,
                                           uintptr_t e, uint4 &d, uint32_t &dn) {
  const uintptr_t a = a0 + (uintptr_t)w * kWin + 16u * b;
  d = (a + 16 > s && a < e) ? *reinterpret_cast<const uint4 *>(a) : make_uint4(0, 0, 0, 0);
  dn = 0;
  if (b == kBlocks - 1 && a + 16 < e) dn = *reinterpret_cast<const uint32_t *>(a + 16);
}

// Value of the LEB128 varint at ring bytes [s, s + n), n in 1..10 (bits past
// 64 dropped). Reads four LDS dwords from s & ~3 (the mirror covers the wrap).
template <uint32_t W>
__device__ __forceinline__ uint64_t ring_varint(const uint8_t *sbuf, uint32_t s, uint32_t n) {
  const uint32_t *d = reinterpret_cast<const uint32_t *>(sbuf + (s & ~3u));
  const uint32_t d0 = d[0], d1 = d[1], d2 = d[2], d3 = d[3];
  const uint32_t sh = s & 3;
  const uint32_t b0 = __builtin_amdgcn_alignbyte(d1, d0, sh);  // bytes s .. s+3
  const uint32_t b1 = __builtin_amdgcn_alignbyte(d2, d1, sh);  // bytes s+4 .. s+7
  // 7-bit groups of bytes s .. s+7: pairs into 14 bits, then into 28 bits
  const uint32_t p0 = (b0 & 0x007f007fu) | ((b0 >> 1) & 0x3f803f80u);
  const uint32_t p1 = (b1 & 0x007f007fu) | ((b1 >> 1) & 0x3f803f80u);
  const uint32_t q0 = (p0 & 0x3fffu) | ((p0 >> 2) & 0x0fffc000u);
  const uint32_t q1 = (p1 & 0x3fffu) | ((p1 >> 2) & 0x0fffc000u);
  uint32_t lo = q0 | (q1 << 28);
  if (W <= 4) {  // the column keeps the low 32 bits: 5 bytes decide them
    if (n <= 4) lo &= (1u << (7 * n)) - 1;
    return lo;
  }
  uint32_t hi = q1 >> 4;
  if (n > 8) {
    const uint32_t b2 = __builtin_amdgcn_alignbyte(d3, d2, sh);  // bytes s+8 .. s+11
    hi |= (b2 & 0x7fu) << 24;
    if (n > 9) hi |= (b2 & 0x100u) << 23;
  } else if (n <= 4) {
    lo &= (1u << (7 * n)) - 1;
    hi = 0;
  } else {
    hi &= (1u << (7 * n - 32)) - 1;
  }
  return ((uint64_t)hi << 32) | lo;
}

template <uint32_t W> __device__ __forceinline__ void store_val(uint8_t *dst, uint32_t i, uint64_t v) {
  if (W == 1) dst[i] = (uint8_t)v;
  else if (W == 2) reinterpret_cast<uint16_t *>(dst)[i] = (uint16_t)v;
  else if (W == 4) reinterpret_cast<uint32_t *>(dst)[i] = (uint32_t)v;
  else reinterpret_cast<uint64_t *>(dst)[i] = v;
}

__device__ __forceinline__ void report(Lds &L, uint32_t idx, uint32_t pr, uint32_t w) {
  atomicMin(reinterpret_cast<unsigned long long *>(&L.key),
            (unsigned long long)((((uint64_t)idx << 2) | pr) << 32 | w));
}

// Waits for this wave's LDS traffic, then the workgroup barrier. Global
// loads stay in flight across it (the prefetched windows).
__device__ __forceinline__ void phase_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Four workgroups (32 waves) per CU: every chunk of a 1024-chunk column is
// resident at once, which needs <= 64 VGPRs per lane.
template <uint32_t W>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8)))
rlev1_pipe_kernel(const uint8_t *__restrict__ comp, uint64_t comp_bytes,
                  const uint64_t *__restrict__ blk_off, const uint64_t *__restrict__ col_len,
                  uint64_t chunk_bytes, uint8_t *__restrict__ out, int32_t *__restrict__ status) {
  __shared__ Lds L;
  const uint64_t chunk = blockIdx.x;
  const uint32_t lane = lane_id();
  const uint32_t wave = uni(threadIdx.x / kWave);
  const uint64_t boff = blk_off[chunk];
  const uint64_t len64 = col_len[chunk];
  if (boff > comp_bytes || len64 > comp_bytes - boff || len64 >= (1ull << 30)) {
    if (threadIdx.x == 0 && status) status[chunk] = kCorrupt;  // uniform over the workgroup
    return;
  }
  const uint32_t len = (uint32_t)len64;
  const uint32_t cap = (uint32_t)(chunk_bytes / W);
  uint8_t *dst = out + chunk * chunk_bytes;
  const uintptr_t s_addr = reinterpret_cast<uintptr_t>(comp + boff);
  const uintptr_t e_addr = s_addr + len;
  const uintptr_t a0 = (s_addr - 1) & ~uintptr_t(15);   // window 0 holds the byte before the stream
  const uint32_t lead = (uint32_t)(s_addr - a0);        // 1..16
  const uint32_t nwin = (lead + len + kWin - 1) / kWin;  // >= 1

  if (threadIdx.x == 0) {
    L.T[0] = 0;
    L.last_w = kNone;
    L.lastterm = 0;
    L.key = kNoKey;
  }

  // helper lane gl = (wave - 1) * 64 + lane loads / stages / indexes block gl
  const uint32_t gl = (wave - 1) * kWave + lane;
  const bool loader = wave >= 1 && gl < kBlocks;
  uint4 pa = make_uint4(0, 0, 0, 0), pb = pa;  // prefetched windows k and k+1
  uint32_t pna = 0, pnb = 0;
  uint4 y = pa;                                // window k-1 (indexed this phase)
  uint32_t yn = 0, ym = 0;
  if (loader) {
    load_block(a0, 0, gl, s_addr, e_addr, pa, pna);
    if (nwin > 1) load_block(a0, 1, gl, s_addr, e_addr, pb, pnb);
  }

  // walker state (wave 0, scalar); the walker is the pipeline's critical
  // path, so its instructions issue ahead of the helpers'
  uint32_t r = 0, o = 0, wdone = 0;
  if (wave == 0) __builtin_amdgcn_s_setprio(3);
  else if (wave <= 2) __builtin_amdgcn_s_setprio(2);  // the waves that also load and index

  phase_barrier();
  for (uint32_t k = 0;; k++) {
    if (wave == 0) {
      // ------------------------------------------------------------ walk window k-2
      const int32_t w = (int32_t)k - 2;
      if (w >= 0 && !wdone) {
        const uint32_t Tw = uni(L.T[w & 7]);
        const uint32_t Tn = uni(L.T[(w + 1) & 7]);
        const bool last = (uint32_t)w == nwin - 1;
        const uint32_t lastterm = last ? uni(L.lastterm) : 0u;
        // In the last window, when the stream ends on a terminator, the last
        // two candidates may lack a header or delta byte (checked from Tfast on).
        const uint32_t Tfast = lastterm ? (Tn >= 2 ? Tn - 2 : 0u) : Tn;
        // the window's step entries in registers: lane l of tab[v] holds
        // entries 2 (64 v + l) and 2 (64 v + l) + 1
        typedef uint32_t tab_t __attribute__((ext_vector_type(kTabRegs)));
        tab_t tab;
        const uint32_t *ent32 = reinterpret_cast<const uint32_t *>(L.ent[w & 1]);
#pragma unroll
        for (uint32_t v = 0; v < kTabRegs; v++) tab[v] = ent32[v * kWave + lane];
        uint32_t *desc = L.desc[w & 1];
        const uint32_t o_first = o;
        uint32_t nd = 0, stop = 0, ovf = 0;
        // Step entry of local terminator rl, from the walker's registers.
#define CODAG_ENT(rl) \
  ((__builtin_amdgcn_readlane(tab[(rl) >> 7], ((rl) >> 1) & (kWave - 1)) >> (((rl) & 1) << 4)) & 0xffff)
        // One segment: run (header h < 0x80, decoder.h:736-790) of h + 3
        // values spanning 2 + [delta byte < 0x80] terminators, or literal
        // group (decoder.h:686-733) of 256 - h values and terminators;
        // descriptor (every lane writes the same word), chunk-full /
        // overflow check, advance.
#define CODAG_STEP(e)                                                                  \
  {                                                                                    \
    const uint32_t h_ = (e) & 0xff;                                                    \
    const uint32_t cnt = h_ < 0x80 ? h_ + 3 : 256 - h_;                                \
    const uint32_t adv = h_ < 0x80 ? 2 + ((e) < 0x8000) : cnt;                         \
    desc[nd++] = (r - Tw) | (o << 11);                                                 \
    if (o + cnt >= cap) {                                                              \
      if (o + cnt > cap) { /* values past the chunk: overflow at index cap */          \
        ovf = 1;                                                                       \
        o = cap + 1; /* the expanders still read the varint at index cap */            \
      } else {                                                                         \
        o = cap;                                                                       \
      }                                                                                \
      break;                                                                           \
    }                                                                                  \
    o += cnt;                                                                          \
    r += adv;                                                                          \
  }
        r = uni(r);
        o = uni(o);
        if (r < Tfast && o < cap) {
#pragma clang loop unroll(disable)
          do {  // the step ends the loop once the chunk is full
            const uint32_t rl = r - Tw;
            const uint32_t e = CODAG_ENT(rl);
            CODAG_STEP(e)
          } while (r < Tfast);
        }
#pragma clang loop unroll(disable)
        while (!ovf && r < Tn && o < cap) {  // the stream's last two terminators
          const uint32_t rl = r - Tw;
          if (r + 1 == Tn) {  // the header would follow the stream's last byte
            if (lane == 0) report(L, o, kPrTrunc, w);
            stop = 1;
            break;
          }
          const uint32_t e = CODAG_ENT(rl);
          if ((e & 0x80) == 0 && r + 2 == Tn) {  // a run header as the last byte: no delta byte
            if (lane == 0) report(L, o, kPrTrunc, w);
            stop = 1;
            break;
          }
          CODAG_STEP(e)
        }
#undef CODAG_STEP
#undef CODAG_ENT
        if (ovf) {
          if (lane == 0) report(L, cap, kPrOverflow, w);
          stop = 1;
        }
        if (o >= cap) stop = 1;
        if (lane == 0) {
          L.wnd[w & 1][0] = nd;
          L.wnd[w & 1][1] = o_first;
          L.wnd[w & 1][2] = o;
        }
        if (stop || last) {
          wdone = 1;
          if (lane == 0) L.last_w = (uint32_t)w;
        }
      }
    } else {
      const uint32_t h = wave - 1;
      // ------------------------------------------------------------ load / stage window k
      uint4 x = pa;
      uint32_t xn = pna;
      pa = pb;
      pna = pnb;
      if (loader && k + 2 < nwin) load_block(a0, k + 2, gl, s_addr, e_addr, pb, pnb);
      // ------------------------------------------------------------ index window k-1
      {
        const int32_t w = (int32_t)k - 1;
        if (w >= 0 && (uint32_t)w < nwin) {
          if (loader) {
            // block b's first terminator: prefix over the window's block counts
            const uint32_t c_lo = L.bcnt[w & 1][lane], c_hi = L.bcnt[w & 1][kWave + lane];
            const uint32_t s_lo = wave_scan_dpp(c_lo), s_hi = wave_scan_dpp(c_hi);
            const uint32_t tot_lo = __builtin_amdgcn_readlane(s_lo, kWave - 1);
            const uint32_t tot_hi = __builtin_amdgcn_readlane(s_hi, kWave - 1);
            if (gl == 0) L.T[(w + 1) & 7] = uni(L.T[w & 7]) + tot_lo + tot_hi;
            const uint32_t slot = w & 3;
            const uint32_t b = gl;
            const uint32_t base = b < kWave ? s_lo - c_lo : tot_lo + s_hi - c_hi;
            uint32_t dn = __shfl_down(y.x, 1, kWave);
            if (lane == kWave - 1)
              dn = b == kBlocks - 1
                       ? yn
                       : *reinterpret_cast<const uint32_t *>(L.sbuf + slot * kWin + 16 * (b + 1));
            const uint32_t gx = (uint32_t)w * kWin + 16 * b;
            const uint32_t lp = lead + len - 1 - gx;  // block byte of the stream's last byte
            if (lp < 16) L.lastterm = (ym >> lp) & 1;
            uint16_t *sel = L.sel[w % 3];
            uint16_t *ent = L.ent[w & 1];
            const uint32_t xo = slot * kWin + 16 * b;
            const uint32_t by[5] = {y.x, y.y, y.z, y.w, dn};
            // branch-free: bytes that are no terminator write the spare entry
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) {
              const uint32_t ix = (ym >> j) & 1 ? base + __popc(ym & ((1u << j) - 1)) : kSpare;
              const uint32_t q = (j + 1) >> 2, sh = (j + 1) & 3;
              sel[ix] = (uint16_t)(xo + j);
              ent[ix] = (uint16_t)(sh == 0 ? by[q] : __builtin_amdgcn_alignbyte(by[q + 1], by[q], sh));
            }
          }
        } else if (w >= 0 && h == 0 && lane == 0) {
          L.T[(w + 1) & 7] = L.T[w & 7];  // past the stream: no terminators
        }
      }
      // ------------------------------------------------------------ stage window k
      if (loader && k < nwin) {
        const uint32_t slot = k & 3;
        reinterpret_cast<uint4 *>(L.sbuf + slot * kWin)[gl] = x;
        if (slot == 0 && gl < kMirror / 16) reinterpret_cast<uint4 *>(L.sbuf + kRing)[gl] = x;
        uint32_t m = term_mask16(x);
        // keep stream positions [0, len): block bytes [lead - gx, lead + len - gx)
        const int32_t gx = (int32_t)(k * kWin + 16 * gl);
        const int32_t lo = (int32_t)lead - gx, hi = (int32_t)(lead + len) - gx;
        const int32_t a = lo < 0 ? 0 : (lo > 16 ? 16 : lo);
        const int32_t z = hi < 0 ? 0 : (hi > 16 ? 16 : hi);
        const uint32_t valid = z > a ? ((0xffffu >> (16 - (z - a))) << a) : 0u;
        m &= valid;
        if (k == 0 && gl == 0) m |= 1u << (lead - 1);  // terminator 0: the byte before the stream
        L.bcnt[k & 1][gl] = (uint8_t)__popc(m);
        y = x;
        yn = xn;
        ym = m;
      }
      // ------------------------------------------------------------ expand window k-3
      const int32_t w = (int32_t)k - 3;
      if (w >= 0) {
        const uint32_t nd = uni(L.wnd[w & 1][0]);
        const uint32_t o_first = uni(L.wnd[w & 1][1]);
        const uint32_t o_end = uni(L.wnd[w & 1][2]);
        const uint32_t Tw = uni(L.T[w & 7]);
        const uint32_t n0 = uni(L.T[(w + 1) & 7]) - Tw;  // terminators of window w
        const uint32_t nk = uni(L.T[(w + 2) & 7]) - Tw;  // ... of windows w and w+1 (indexed)
        const uint32_t bad_pr = (uint32_t)w + 2 >= nwin ? kPrTrunc : kPrPending;
        const uint16_t *sel0 = L.sel[w % 3];
        // ring position of local terminator q: window w's entries, then w+1's
        const uint16_t *sel1m = L.sel[(w + 1) % 3] - n0;
        auto sel = [&](uint32_t q) -> uint32_t { return (q < n0 ? sel0 : sel1m)[q]; };
        const uint32_t *desc = L.desc[w & 1];
        // lanes exchange segment starts through these bytes (one wave's LDS
        // operations complete in order; a compiler barrier keeps the read a
        // real load after the marks)
        uint8_t *mk = L.mark[h];
        const uint32_t npass = (o_end - o_first + kWave - 1) / kWave;
        uint32_t cur = 0;
        // passes of 64 consecutive values: of every 12, helpers 0 and 1
        // (which also load, stage and index) take one each, the others two
        const uint32_t per = h < 2 ? 1u : 2u;
        const uint32_t first = h < 2 ? h : 2 * h - 2;
#pragma clang loop unroll(disable)
        for (uint32_t t = 0;; t++) {
          const uint32_t p = 12 * (t / per) + first + (t % per);
          if (p >= npass) break;
          const uint32_t ob = o_first + kWave * p;
          // cur: the last segment starting at or before value ob; lane i
          // holds segment cur + i
          uint32_t di, oi;
          bool iv;
          for (;;) {
            const uint32_t i = cur + lane;
            iv = i < nd;
            di = iv ? desc[i] : 0u;
            oi = di >> 11;
            const uint32_t c = (uint32_t)__popcll(__ballot(iv && lane >= 1 && oi <= ob));
            if (c == 0) break;
            cur += c;
          }
          // segment of value ob + lane = cur + (segments starting in (ob, ob + lane])
          mk[lane] = 0;
          if (lane >= 1 && iv && oi - ob < kWave) mk[oi - ob] = 1;
          asm volatile("" ::: "memory");
          const uint64_t starts = __ballot(mk[lane] != 0);
          const uint32_t j = __builtin_amdgcn_mbcnt_hi((uint32_t)(starts >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)starts, 0)) +
                             (uint32_t)((starts >> lane) & 1);
          const uint32_t dsc = __shfl(di, (int)j, kWave);
          const uint32_t v = ob + lane;
          const bool act = v < o_end;
          const uint32_t rl = dsc & 0x7ff;
          const uint32_t os = dsc >> 11;
          const uint32_t ii = act ? v - os : 0u;  // lanes past the window read in range
          const uint32_t s0 = sel0[rl];  // terminator before the header
          const uint32_t hb = L.sbuf[s0 + 1], db = L.sbuf[s0 + 2];
          const bool run = hb < 0x80;
          // run (decoder.h:736-790): the base starts after the delta byte,
          // ends on terminator rl + 2 + [delta byte < 0x80] and belongs to the
          // run's first value; literal group (decoder.h:686-733): varint ii
          // ends on terminator rl + 1 + ii and starts after terminator rl + ii
          // (after the header for ii = 0)
          const uint32_t qb = run ? rl + 2 + (db < 0x80) : rl + 1 + ii;
          const bool complete = qb < nk;
          const uint32_t qa = (run || ii == 0) ? rl : qb - 1;
          const uint32_t start = sel(qa) + 1 + (run ? 2u : (ii == 0 ? 1u : 0u));
          const uint32_t n = ((sel(complete ? qb : qa) - start) & (kRing - 1)) + 1;
          if (act && complete && n <= 10) {
            if (v < cap) {
              uint64_t val = ring_varint<W>(L.sbuf, start, n);
              if (run) val += (uint64_t)((int64_t)ii * (int32_t)(int8_t)db);  // delta byte
              store_val<W>(dst, v, val);
            }
          } else if (act) {  // incomplete or longer than any 64-bit varint
            report(L, run ? os : v, complete ? kPrCorrupt : bad_pr, (uint32_t)w);
          }
        }
      }
    }
    phase_barrier();
    const uint32_t lw = uni(L.last_w);
    if ((lw != kNone && k >= lw + 3) || k >= nwin + 3) break;
  }

  if (threadIdx.x == 0) {
    const uint64_t key = L.key;
    int32_t st = kOk;
    uint32_t pend_w = kNone;
    if (key != kNoKey) {
      const uint32_t pr = (uint32_t)(key >> 32) & 3;
      st = pr == kPrCorrupt ? kCorrupt : pr == kPrTrunc ? kTrunc : pr == kPrOverflow ? kOverflow : kOk;
      if (pr == kPrPending) pend_w = (uint32_t)key;
    }
    L.last_w = pend_w;
    if (pend_w == kNone && status) status[chunk] = st;
  }
  __syncthreads();
  const uint32_t pend_w = uni(L.last_w);
  if (pend_w != kNone && wave == 0) {
    // An overlong varint runs past the indexed windows: it ends CORRUPT if
    // any terminator follows window pend_w + 1, TRUNCATED if none does.
    const uintptr_t from = a0 + (uintptr_t)(pend_w + 2) * kWin;  // 16-byte aligned
    uint32_t found = 0;
    for (uintptr_t a = from + 16u * lane; a < e_addr; a += 16u * kWave) {
      const uint4 d = *reinterpret_cast<const uint4 *>(a);
      uint32_t m = term_mask16(d);
      const uintptr_t rem = e_addr - a;
      if (rem < 16) m &= (1u << rem) - 1;
      found |= m;
    }
    const uint64_t any = __ballot(found != 0);  // of all lanes: not inside lane 0's branch
    if (lane == 0 && status) status[chunk] = any ? kCorrupt : kTrunc;
  }
}

// ---------------------------------------------------------------- spans by all waves

// Walk and expansion by turns, both by every wave of a group of kSpWaves. A step
// stages 8 KiB of the stream from a segment's header on and numbers the
// terminators in it, 0 being the byte before the header.
//  * Lane i of a span of 64 terminators sizes the segment after its terminator.
//    Pointer doubling by ds_bpermute leaves every terminator the first one
//    outside its span that its chain reaches, a pass from the wave's last span to
//    its first the first one outside the wave's. A terminator whose segment is
//    not whole in the window is its own successor and ends the chain.
//  * One link per wave then gives each wave its entry, and each wave follows its
//    own spans by v_readlane.
//  * A prefix sum over the group places the segments, and the values are dealt
//    out in passes of 64, one lane per value.
// A segment that is not whole at the stream's end, or in a window of its own, is
// read value by value (one_segment), which finds its error.
// The pipeline's walker takes about 115 cycles a segment, so a column of short
// runs (3 bytes of stream each) is bound by it alone; here the chain costs the
// same whatever the segments. Latency bounds it: a step of dense segments takes
// 42 K cycles, 10 K each in the doubling, the placing and the values. 128 KiB
// chunks, pipeline and spans: 32 chunks of an 8-bit table column 2105 and 378 us,
// 64 chunks of a 64-bit one 545 and 125, benchmark columns of 64 chunks, 8 bits
// 438 and 312, 64 bits 73 and 64. With two groups per CU the benchmark columns
// are slower (512 chunks, 64 bits, 84 and 95).
constexpr uint32_t kSpBytes = 8192, kSpWaves = 16;
constexpr uint32_t kSpThreads = kSpWaves * kWave;
constexpr uint32_t kSpans = kSpBytes / kSpThreads;  // spans of a wave, at most

constexpr uint32_t kMaxSpanCap = (1u << 19) - 1;  // values per chunk (descriptor field; later ones are not read)

__device__ __forceinline__ uint32_t rdlast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
// of an inclusive prefix sum over the waves, the sum of those before this wave
__device__ __forceinline__ uint32_t before(uint32_t sums, uint32_t wave) {
  return wave ? (uint32_t)__builtin_amdgcn_readlane((int)sums, (int)wave - 1) : 0u;
}

struct SpanLds {
  uint8_t sbuf[kSpBytes + 32];
  uint16_t sel[kSpBytes];  // window byte of each terminator
  union {
    uint16_t to[kSpBytes];        // the first terminator outside its wave's that a chain reaches
    uint32_t desc[kSpBytes / 2];  // segment: terminator before it (13 bits) | first value of the step << 13
  };
  uint32_t count[kSpWaves], values[kSpWaves], segs[kSpWaves];
  uint8_t mark[kSpWaves][kWave];
  uint32_t key;   // first error: value of the step << 2 | priority
  uint32_t over;  // 1: a segment reaches past the chunk; 2: a terminator follows an overlong varint
  uint32_t pos, o, pending;  // one_segment's results
  int32_t st;
};

// Reads the segment at stream byte pos and writes its values from element o on, as
// the oracle does. Returns the status; `pending`: a varint longer than 10 bytes
// begins before pos, whose status hangs on whether any terminator follows.
template <uint32_t W>
__device__ __forceinline__ int32_t one_segment(const uint8_t *src, uint32_t len, uint32_t cap, uint8_t *dst,
                                            uint32_t &pos, uint32_t &o, uint32_t &pending) {
  pending = 0;
  if (pos >= len) return kTrunc;
  const uint32_t h = src[pos++];
  const uint32_t cnt = h < 0x80 ? h + 3 : 256 - h;
  int64_t delta = 0;
  if (h < 0x80) {
    if (pos >= len) return kTrunc;
    delta = (int8_t)src[pos++];
  }
  uint64_t v = 0;
  for (uint32_t i = 0; i < cnt; i++) {
    if (i == 0 || h >= 0x80) {
      v = 0;
      for (uint32_t n = 0;; n++) {
        if (pos >= len) return kTrunc;
        if (n == 10) {
          pending = 1;
          return kCorrupt;
        }
        const uint32_t b = src[pos++];
        v |= (uint64_t)(b & 0x7f) << (7 * n);
        if (b < 0x80) break;
      }
    }
    if (o >= cap) return kOverflow;
    store_val<W>(dst, o++, v + (uint64_t)((int64_t)i * delta));
  }
  return kOk;
}

// 64 registers: two groups per CU.
template <uint32_t W>
__global__ void __launch_bounds__(kSpThreads) __attribute__((amdgpu_waves_per_eu(8)))
rlev1_span_kernel(const uint8_t *__restrict__ comp, uint64_t comp_bytes, const uint64_t *__restrict__ blk_off,
                  const uint64_t *__restrict__ col_len, uint64_t chunk_bytes, uint8_t *__restrict__ out,
                  int32_t *__restrict__ status) {
  constexpr uint32_t kDw = kSpBytes / 4 / kSpThreads;  // window dwords a thread indexes
  __shared__ __align__(16) SpanLds L;
  const uint64_t chunk = blockIdx.x;
  const uint32_t lane = lane_id(), tid = threadIdx.x;
  const uint32_t wave = uni(tid / kWave);
  const uint64_t boff = blk_off[chunk], len64 = col_len[chunk];
  if (boff > comp_bytes || len64 > comp_bytes - boff || len64 >= (1ull << 30)) {
    if (tid == 0 && status) status[chunk] = kCorrupt;  // uniform over the workgroup
    return;
  }
  const uint32_t len = (uint32_t)len64, cap = (uint32_t)(chunk_bytes / W);
  const uint8_t *src = comp + boff;
  uint8_t *dst = out + chunk * chunk_bytes;
  const uintptr_t s_addr = reinterpret_cast<uintptr_t>(src), e_addr = s_addr + len;
  uint32_t pos = 0, o = 0;  // stream position and value index of the step's first header
  int32_t st = kOk;
  uint4 pre = make_uint4(0, 0, 0, 0);
  // the window begins at the 16-byte block of the byte before `from`; only blocks
  // with stream bytes are read
  auto load = [&](uint32_t from) __attribute__((always_inline)) {
    const uintptr_t a = ((s_addr + from - 1) & ~uintptr_t(15)) + 16u * tid;
    pre = make_uint4(0, 0, 0, 0);
    if (tid < kSpBytes / 16 && a + 16 > s_addr && a < e_addr) pre = *reinterpret_cast<const uint4 *>(a);
  };
  load(0);
  for (;;) {
    if (tid < kSpBytes / 16) reinterpret_cast<uint4 *>(L.sbuf)[tid] = pre;
    if (tid == 0) {
      L.key = ~0u;
      L.over = 0;
    }
    __syncthreads();
    const uint32_t lead = uni((uint32_t)((s_addr + pos - 1) & 15) + 1);  // window byte of stream byte pos
    const uint32_t P = min(lead + (len - pos), kSpBytes);
    const bool at_end = lead + (len - pos) <= kSpBytes;
    // ---- number the terminators
    uint32_t tm = 0;  // bit 4 i + j: byte j of the thread's dword i ends a varint
#pragma unroll
    for (uint32_t i = 0; i < kDw; i++) {
      const uint32_t at = 4 * (tid * kDw + i);
      const uint32_t t = ~reinterpret_cast<const uint32_t *>(L.sbuf)[tid * kDw + i] & 0x80808080u;
      uint32_t m = __builtin_amdgcn_udot4(t >> 7, 0x08040201u, 0u, false);
      const int32_t a = (int32_t)(lead - at), z = (int32_t)(P - at);  // stream bytes of the dword
      m &= z >= 4 ? 0xfu : (z > 0 ? (1u << z) - 1 : 0u);
      m &= a <= 0 ? 0xfu : (a < 4 ? 0xfu << a : 0u);
      m |= a >= 1 && a <= 4 ? 1u << (a - 1) : 0u;  // terminator 0
      tm |= m << (4 * i);
    }
    const uint32_t mine = (uint32_t)__popc(tm), incl0 = wave_scan_dpp(mine);
    if (lane == kWave - 1) L.count[wave] = incl0;
    __syncthreads();
    const uint32_t counts = wave_scan_dpp(lane < kSpWaves ? L.count[lane] : 0u);  // lane w: of waves 0 to w
    const uint32_t terms = rdlast(counts);
    uint32_t rank = incl0 - mine + before(counts, wave);
#pragma unroll
    for (uint32_t b = 0; b < 4 * kDw; b++) {
      if ((tm >> b) & 1) L.sel[rank++] = (uint16_t)(4 * tid * kDw + b);
    }
    __syncthreads();
    // ---- the segments after this wave's terminators
    const uint32_t spans = (terms + kSpThreads - 1) / kSpThreads, own = spans * kWave;  // of a wave
    const uint32_t w0 = wave * own, w1 = w0 + own;
    // per terminator: values << 8 | next, as a lane of its span; later the span's
    // values up to and with this segment << 8 | its own
    uint32_t sg[kSpans], ex[kSpans];
#pragma unroll
    for (uint32_t k = 0; k < kSpans; k++) {
      if (k >= spans) continue;
      const uint32_t r = w0 + k * kWave + lane;
      const uint32_t s = r < terms ? L.sel[r] : 0u;
      const uint32_t h = L.sbuf[s + 1], d = L.sbuf[s + 2];
      const bool run = h < 0x80;
      const uint32_t adv = run ? 2 + (d < 0x80) : 256 - h;
      const bool ok = r + adv < terms && s + (run ? 2u : 1u) < P;
      ex[k] = ok ? lane + adv : lane;
      sg[k] = (run ? h + 3 : adv) << 8 | ex[k];
    }
    // a chain in a span has 64 links at most
#pragma unroll
    for (uint32_t d = 0; d < 6; d++) {
#pragma unroll
      for (uint32_t k = 0; k < kSpans; k++) {
        if (k >= spans) continue;
        const uint32_t x = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(ex[k] * 4), (int)ex[k]);
        ex[k] = ex[k] < (uint32_t)kWave ? x : ex[k];
      }
    }
#pragma unroll
    for (uint32_t k = kSpans; k-- > 0;) {
      if (k >= spans) continue;
      const uint32_t b = w0 + k * kWave;
      uint32_t x = b + ex[k];
      if (k + 1 < spans) {
        const uint32_t y = L.to[min(x, w1 - 1)];
        x = x >= b + kWave && x < w1 ? y : x;
      }
      L.to[b + lane] = (uint16_t)x;
      asm volatile("" ::: "memory");  // other lanes read it; one wave's LDS operations keep their order
    }
    __syncthreads();
    // the chain over the waves; it ends at a terminator without a whole segment
    uint32_t p = 0, entry = kNone;
    bool end = false;
#pragma unroll
    for (uint32_t w = 0; w < kSpWaves; w++) {
      if (!end && p < (w + 1) * own) {
        entry = w == wave ? p : entry;
        p = uni((uint32_t)L.to[p]);
        end = p < (w + 1) * own;
      }
    }
    // this wave's segments, span by span
    uint64_t mk[kSpans];
    uint32_t values = 0, segs = 0;
    {
      uint32_t q = entry;
      bool go = entry != kNone;
#pragma unroll
      for (uint32_t k = 0; k < kSpans; k++) {
        mk[k] = 0;
        if (k >= spans) continue;
        const uint32_t b = w0 + k * kWave;
        uint64_t m = 0;
        if (go && q < b + kWave) {
          uint32_t r = q - b;
          for (;;) {
            const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)sg[k], (int)r) & 0xff;
            if (t == r) {
              go = false;
              break;
            }
            m |= 1ull << r;
            r = t;
            if (r >= (uint32_t)kWave) break;
          }
          q = b + r;
        }
        mk[k] = m;
        const uint32_t c = (m >> lane) & 1 ? sg[k] >> 8 : 0u, incl = wave_scan_dpp(c);
        sg[k] = incl << 8 | c;
        values += rdlast(incl);
        segs += (uint32_t)__builtin_popcountll(m);
      }
    }
    if (lane == 0) {
      L.values[wave] = values;
      L.segs[wave] = segs;
    }
    const uint32_t next = pos + (uni((uint32_t)L.sel[p]) + 1 - lead);
    const bool alone = at_end || p == 0;  // what follows is no whole segment
    if (!alone) load(next);
    __syncthreads();  // L.to is done with: descriptors take its place
    const uint32_t vs = wave_scan_dpp(lane < kSpWaves ? L.values[lane] : 0u);
    const uint32_t ss = wave_scan_dpp(lane < kSpWaves ? L.segs[lane] : 0u);
    const uint32_t total = rdlast(vs), nd = rdlast(ss);
    uint32_t at_o = before(vs, wave), at_n = before(ss, wave);
    const uint32_t room = cap - o;
#pragma unroll
    for (uint32_t k = 0; k < kSpans; k++) {
      if (k >= spans) continue;
      if ((mk[k] >> lane) & 1) {
        const uint32_t to = at_o + (sg[k] >> 8), os = to - (sg[k] & 0xff);
        L.desc[at_n + lanes_below(mk[k])] = (w0 + k * kWave + lane) | min(os, kMaxSpanCap) << 13;
        if (os < room && to > room) L.over = 1;
      }
      at_o += rdlast(sg[k]) >> 8;
      at_n += (uint32_t)__builtin_popcountll(mk[k]);
    }
    __syncthreads();
    // ---- values; the one at index cap is read as well, as its varint's error comes first
    const uint32_t over = uni(L.over), vend = over ? room + 1 : min(total, room);
    const uint32_t npass = (vend + kWave - 1) / kWave, per = (npass + kSpWaves - 1) / kSpWaves;
    const uint32_t pa = wave * per, pb = min(pa + per, npass);
    uint32_t cur = 0;  // the last segment that starts at or before the pass's first value
    if (pa < pb) {
      uint32_t lo = 0, hi = nd;  // by 64 probes at a time
      while (hi - lo > 1) {
        const uint32_t step = (hi - lo + kWave - 1) / kWave, i = lo + lane * step;
        const uint64_t le = __ballot(i < hi && (L.desc[min(i, nd - 1)] >> 13) <= pa * kWave);
        const uint32_t c = (uint32_t)__builtin_popcountll(le);  // lane 0 always is one
        lo += (c - 1) * step;
        hi = min(lo + step, hi);
      }
      cur = lo;
    }
    uint8_t *mkb = L.mark[wave];
#pragma clang loop unroll(disable)
    for (uint32_t t = pa; t < pb; t++) {
      const uint32_t ob = t * kWave;
      uint32_t di, oi;
      bool iv;
      for (;;) {
        const uint32_t i = cur + lane;
        iv = i < nd;
        di = iv ? L.desc[i] : 0u;
        oi = di >> 13;
        const uint32_t c = (uint32_t)__popcll(__ballot(iv && lane >= 1 && oi <= ob));
        if (c == 0) break;
        cur += c;
      }
      // segment of value ob + lane = cur + (segments starting in (ob, ob + lane])
      mkb[lane] = 0;
      if (lane >= 1 && iv && oi - ob < (uint32_t)kWave) mkb[oi - ob] = 1;
      asm volatile("" ::: "memory");
      const uint64_t starts = __ballot(mkb[lane] != 0);
      const uint32_t j = lanes_below(starts) + (uint32_t)((starts >> lane) & 1);
      const uint32_t dsc = (uint32_t)__shfl((int)di, (int)j, kWave);
      const uint32_t v = ob + lane;
      const bool act = v < vend;
      const uint32_t rl = dsc & 0x1fff, os = dsc >> 13;
      const uint32_t ii = act ? v - os : 0u;
      const uint32_t s0 = L.sel[rl];
      const uint32_t hb = L.sbuf[s0 + 1], db = L.sbuf[s0 + 2];
      const bool run = hb < 0x80;
      // the varint ends on terminator qb and follows qa, or the header (and delta
      // byte) after it
      const uint32_t qb = min(run ? rl + 2 + (db < 0x80) : rl + 1 + ii, terms - 1);
      const bool front = run || ii == 0;
      const uint32_t start = (front ? s0 : (uint32_t)L.sel[qb - 1]) + 1 + (front ? (run ? 2u : 1u) : 0u);
      const uint32_t n = L.sel[qb] + 1u - start;
      if (act && n <= 10) {
        if (v < room) {
          uint64_t val = ring_varint<W>(L.sbuf, start, n);
          if (run) val += (uint64_t)((int64_t)ii * (int32_t)(int8_t)db);
          store_val<W>(dst, o + v, val);
        }
      } else if (act) {  // longer than any 64-bit varint
        atomicMin(&L.key, (run ? os : v) << 2 | kPrCorrupt);
      }
    }
    if (over && tid == 0) atomicMin(&L.key, room << 2 | kPrOverflow);
    __syncthreads();
    const uint32_t key = uni(L.key);
    if (key != ~0u) {
      st = (key & 3) == kPrCorrupt ? kCorrupt : kOverflow;
      break;
    }
    o += min(total, room);
    pos = next;
    if (o >= cap) break;
    if (alone) {
      if (tid == 0) {
        uint32_t pending;
        L.st = one_segment<W>(src, len, cap, dst, pos, o, pending);
        L.pos = pos;
        L.o = o;
        L.pending = pending;
      }
      __syncthreads();
      st = (int32_t)uni((uint32_t)L.st);
      pos = uni(L.pos);
      o = uni(L.o);
      if (uni(L.pending)) {  // no terminator after it: the stream ends in it
        uint32_t found = 0;
        const uintptr_t from = (s_addr + pos) & ~uintptr_t(15);
        for (uintptr_t a = from + 16u * tid; a < e_addr; a += 16u * kSpThreads) {
          uint32_t m = term_mask16(*reinterpret_cast<const uint4 *>(a));
          if (a < s_addr + pos) m &= 0xffffu << (s_addr + pos - a);
          if (e_addr - a < 16) m &= (1u << (e_addr - a)) - 1;
          found |= m & 0xffffu;
        }
        if (__ballot(found != 0) && lane == 0) L.over = 2;
        __syncthreads();
        st = uni(L.over) == 2 ? kCorrupt : kTrunc;
      }
      if (st != kOk || o >= cap) break;
      load(pos);
      __syncthreads();  // every wave has read L.st
    }
  }
  if (tid == 0 && status) status[chunk] = st;
}

}  // namespace rle1p

hipError_t launch_rlev1_pipe(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *blk_off,
                             const uint64_t *col_len, uint64_t n_chunks, uint32_t w,
                             uint64_t chunk_bytes, uint8_t *out, int32_t *status,
                             hipStream_t stream) {
  if (n_chunks == 0) return hipSuccess;
  if (chunk_bytes / w > rle1p::kMaxCap) return hipErrorInvalidValue;  // descriptor value field
  const dim3 grid((uint32_t)n_chunks), block(rle1p::kThreads);
#define CODAG_V1P(W)                                                                         \
  hipLaunchKernelGGL((rle1p::rlev1_pipe_kernel<W>), grid, block, 0, stream, comp, comp_bytes, \
                     blk_off, col_len, chunk_bytes, out, status)
  switch (w) {
  case 1: CODAG_V1P(1); break;
  case 2: CODAG_V1P(2); break;
  case 4: CODAG_V1P(4); break;
  case 8: CODAG_V1P(8); break;
  default: return hipErrorInvalidValue;
  }
#undef CODAG_V1P
  return hipGetLastError();
}

hipError_t launch_rlev1_span(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *blk_off,
                             const uint64_t *col_len, uint64_t n_chunks, uint32_t w, uint64_t chunk_bytes,
                             uint8_t *out, int32_t *status, hipStream_t stream) {
  if (n_chunks == 0) return hipSuccess;
  if (chunk_bytes / w > rle1p::kMaxSpanCap) return hipErrorInvalidValue;
  const dim3 grid((uint32_t)n_chunks), block(rle1p::kSpThreads);
#define CODAG_V1S(W)                                                                         \
  hipLaunchKernelGGL((rle1p::rlev1_span_kernel<W>), grid, block, 0, stream, comp, comp_bytes, \
                     blk_off, col_len, chunk_bytes, out, status)
  switch (w) {
  case 1: CODAG_V1S(1); break;
  case 2: CODAG_V1S(2); break;
  case 4: CODAG_V1S(4); break;
  case 8: CODAG_V1S(8); break;
  default: return hipErrorInvalidValue;
  }
#undef CODAG_V1S
  return hipGetLastError();
}

}  // namespace codag
