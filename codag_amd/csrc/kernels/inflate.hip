// inflate.hip -- gfx950 zlib/Deflate (RFC 1950/1951) decoder, a group of waves per stream.
//
// Mapping onto CDNA. A stream is decoded by a group of one wave (many streams:
// throughput) or several waves (few streams: latency), in spans:
//  * Span decode. The next 64 x waves x S bits of a block are staged in LDS and
//    every lane decodes the subsequence of S bits that begins at its own bit.
//    Only lane 0's start is known to be the start of a token; Huffman codes
//    synchronise by themselves (a decoder started at a wrong bit meets the true
//    token starts after about 90 bits at the median, 430 at the 95th
//    percentile), so a lane's exit is mostly right although its entry was not.
//    Each pass hands the exits on as the next lanes' entries and decodes the
//    lanes whose entry changed, until no entry changes up to the first stop
//    (end of block, invalid code, stream end). A lane does one table lookup a
//    step: a literal takes one, a match two (length code, distance code), a
//    code longer than the root table one more.
//  * Output. The verified lanes know their byte counts; a prefix sum gives each
//    its output position. They decode once more and write a 16-bit mark at each
//    token's first byte into an LDS window (literal byte, or distance). The
//    window is then resolved 256 bytes at a time, four a lane: a DPP max scan
//    hands every byte its token's mark, sources before the window are gathered
//    from HBM a step ahead, sources inside it are followed by pointer doubling;
//    the bytes are stored and summed for the Adler-32.
//  * Codes of nearly one length do not synchronise: chain_entries finds the lanes'
//    entries from all bits at which the token before may end.
//  * Long matches: narrow_span decodes by one wave, 64 stream bits at a time.
//  * The scalar symbol loop decodes the symbol a span stopped at (end of block,
//    or the error), so statuses are exactly the serial decoder's.
// What bounds it: vector issue and its latency, not memory (without the far
// gathers and the stores the launches take the same time). 128 KiB zlib level-6
// chunks, before (one token chain per stream: 64 bit positions decoded to keep
// about seven tokens, the chain scalar) and now: 4096 chunks 9.1 and 2.96 ms, 256
// chunks 4.0 and 0.44 ms, 3 chunks 3.7 and 0.42 ms; 300 mixed streams of 4 KiB
// to 4 MiB 119 and 14.6 ms. A chunk takes 0.25 M vector instructions (0.69 M
// before): half of them passes, headers and tables, a fifth marks, a third the
// resolving. A window byte costs the same whatever token it is in, so data that
// compress to less than a thirtieth go by narrow_span (4096 chunks of zeros 1.1
// before, 0.74 ms now; with a one every 200 bytes 0.88 and 0.96).
//
// Reference counterpart: include/zlib/zlib.h:807-866 (full_warp_shared_lut),
// 531-707 (dynamic header / table build), 712-805 (symbol loop), 188-347
// (warp copy). Differences: stored blocks are decoded (the reference's branch
// is empty, zlib.h:840-842), BTYPE 11 is rejected (zlib.h:843 treats it as
// dynamic), the zlib header and Adler-32 trailer are checked as zlib does.
#include <algorithm>
#include <cstddef>
#include <mutex>

#include "device.hpp"
#include "kernels.hpp"
#include "window.hpp"

namespace codag {
namespace inflate {

using namespace codag::dev;

constexpr uint32_t kCodeBits = 7;

enum : int32_t { kOk = 0, kTrunc = 1, kOverflow = 2, kCorrupt = 3 };
constexpr int32_t kEob = 16;   // end of block (not a status)
constexpr int32_t kMore = 17;  // symbol loop: one symbol decoded (not a status)
enum : uint32_t { kTabLit = 0, kTabDist = 1, kTabCodes = 2 };

// RFC 1951 section 3.2.5 length and distance codes (the tables of
// include/zlib/zlib.h:35-51) in closed form: length code c (0..28) has
// (c - 4) / 4 extra bits from c = 8 on (none for c = 28, length 258) and base
// 3 + c below 8, else 3 + ((4 + c % 4) << extra); distance code d (0..29) has
// (d - 2) / 2 extra bits from d = 4 on and base 1 + d below 4, else
// 1 + ((2 + d % 2) << extra).
__device__ __forceinline__ uint32_t len_extra(uint32_t c) { return (c < 8 || c == 28) ? 0 : (c - 4) >> 2; }
__device__ __forceinline__ uint32_t len_base(uint32_t c, uint32_t extra) {
  return c < 8 ? c + 3 : (c == 28 ? 258 : ((4 + (c & 3)) << extra) + 3);
}
__device__ __forceinline__ uint32_t dist_extra(uint32_t d) { return d < 4 ? 0 : (d - 2) >> 1; }
__device__ __forceinline__ uint32_t dist_base(uint32_t d, uint32_t extra) {
  return d < 4 ? d + 1 : ((2 + (d & 1)) << extra) + 1;
}
// Order of the code-length code lengths (RFC 1951 3.2.7).
__constant__ uint8_t kClOrder[19] = {16, 17, 18, 0, 8, 7, 9, 6, 10, 5, 11, 4, 12, 3, 13, 2, 14, 1, 15};

template <int NSYM> struct Huff {
  uint16_t count[16];
  uint16_t first[16];
  uint16_t index[16];
  uint16_t sym[NSYM];
};

// 32-bit table entries:
//   bits 4:0   bits this lookup consumes (code and extra bits); 0 = a stop: end
//              of block, invalid symbol or no such code
//   bits 8:5   extra-bit count
//   bits 12:9  code bits this lookup consumes (the extra bits follow them)
//   bit  13    literal
//   bits 29:14 value: literal byte, length base, distance base, or, for a code
//              longer than the root table, the sub-table's descriptor
//   bits 31:30 0 the token is complete (literal, distance), 1 a length code
//              (a distance code follows), 2 a sub-table lookup follows
// A table descriptor is the table's index bits (bits 4:0, where a bit field
// extract takes its width from) and its first entry (bits 15:5).
constexpr uint32_t kLitFlag = 1u << 13;
constexpr uint32_t kLenType = 1u << 30;
constexpr uint32_t kSubType = 2u << 30;

// One shape of the decoder: NW waves per stream, SD dwords of the stream per
// lane in a span, each lane's part cut into SUB pieces for the output phase (a
// wave writes its span in SUB groups, so that a group's bytes fit the window),
// SEG window bytes per wave, root tables of LB and DB bits with room for LS and
// DS sub-table entries. 340 / 272 entries hold every sub-table of a complete
// 286 / 30 symbol code behind 9 / 7 root bits, 308 / 144 behind 10 / 8; a
// sub-table that finds no room becomes a stop, which the symbol loop decodes.
template <int NW_, int SD_, int SUB_, uint32_t SEG_, uint32_t LB_, uint32_t DB_, uint32_t LS_, uint32_t DS_>
struct Cfg {
  static constexpr int kNW = NW_, kSub = SUB_;
  static constexpr uint32_t kThreads = NW_ * 64, kSD = SD_, kSpanBits = SD_ * 32;
  static constexpr uint32_t kSeg = SEG_, kWin = NW_ * SEG_;
  static constexpr uint32_t kLB = LB_, kDB = DB_, kLS = LS_, kDS = DS_;
  static constexpr uint32_t kDistAt = (1u << LB_) + LS_, kTab = kDistAt + (1u << DB_) + DS_;
  static constexpr uint32_t kLitDesc = LB_, kDistDesc = kDistAt << 5 | DB_;
  static constexpr uint32_t kStage = kThreads * SD_ + 5;
  static_assert(kTab <= 2048, "sub-table descriptors hold 11-bit positions");
  static_assert(NW_ == 1 || SUB_ == 1, "pieces are exchanged inside one wave");
};
// Odd SD: the lanes' first reads fall on different LDS banks.
using One = Cfg<1, 13, 2, 4096, 9, 7, 340, 272>;
using Many = Cfg<8, 9, 1, 2560, 10, 8, 308, 144>;

template <class C> struct Sh {
  alignas(16) uint32_t stage[C::kStage];  // the span's stream dwords
  alignas(16) uint32_t tab[C::kTab];      // literal/length root, its sub-tables, distance root, its sub-tables
  alignas(16) uint16_t win[C::kWin + 2];  // marks of the window being written, and one for none; CRC-32 slice tables
  Huff<288> hl;
  Huff<32> hd;
  alignas(4) uint8_t lens[320];
  uint32_t err;                       // first output error of a window: position << 2 | status
  // groups of several waves
  uint32_t ex[C::kNW > 1 ? C::kThreads : 1];  // lanes' exits, bit 31 = stopped
  uint32_t mis[C::kNW], stp[C::kNW];          // per wave: first lane with a changed entry / that stopped
  uint32_t part[2][C::kNW];                   // per-wave partial sums
  uint32_t end;                               // stage bit after the span's last token
  // what the serial decoder found next (serial_step)
  uint32_t op, P, ln, val, dist, pos;
  int32_t st;
  uint32_t last;
  uint32_t stream;                            // the group's current stream
};

// LDS and global memory seen through pointers of their own address spaces:
// functions that are not inlined would else reach them by flat accesses.
template <class T> using lds = __attribute__((address_space(3))) T;
template <class T> using glob = __attribute__((address_space(1))) T;

// A wave-uniform pointer as such.
template <class T> __device__ __forceinline__ glob<T> *uni_ptr(T *p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return (glob<T> *)((uint64_t)uni((uint32_t)(a >> 32)) << 32 | uni((uint32_t)a));
}

// Orders this wave's LDS accesses around a point where its lanes exchange data
// through LDS.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The same for the whole group.
template <class C> __device__ __forceinline__ void group_sync() {
  if constexpr (C::kNW > 1) __syncthreads();
  else wave_sync();
}

// ------------------------------------------------------------- output side

// Output state, the same in every wave of the group except the per-lane
// Adler-32 partial sums: s1 = sum b, s2 = sum pos*b (mod 65521), both reduced
// after every window. Positions are 32-bit (outputs below 2^31 bytes).
struct Out {
  uint8_t *dst;
  uint32_t cap;
  uint32_t pos;  // bytes produced; all of them are stored
  uint32_t s1, s2;
};

// Eight passes that verify fewer lanes than these cost more than the chain, per lane
// (literals of 4096 chunks of text, no matches, 64 lanes: below 16 of them 11.7 ms,
// below 32 11.0 ms; base64 text 7.9 and 8.0 ms).
template <class C> constexpr uint32_t kFewLanes = C::kNW > 1 ? C::kThreads / 4 : C::kThreads / 2;
constexpr uint32_t kHard = 3;  // spans of few verified lanes before a block goes on with chain_entries

__device__ __forceinline__ void adler_add(Out &o, uint32_t at, uint32_t b) {
  o.s1 += b;
  o.s2 = (o.s2 + (at % 65521u) * b) % 65521u;
}

// One token by one wave, straight in HBM (the symbol loop's tokens).
__device__ __forceinline__ int32_t out_token(Out &o, uint32_t lane, bool lit, uint32_t val, uint32_t dist) {
  const uint32_t n = lit ? 1u : val;
  if (o.pos + n > o.cap) return kOverflow;
  if (!lit && dist > o.pos) return kCorrupt;  // zlib: "invalid distance too far back"
  for (uint32_t i = lane; i < n; i += kWave) {
    const uint32_t b = lit ? val : o.dst[o.pos - dist + i % dist];
    o.dst[o.pos + i] = (uint8_t)b;
    adler_add(o, o.pos + i, b);
  }
  o.s1 %= 65521u;
  o.pos += n;
  return kOk;
}

// Copies ln stored-block bytes from src (RFC 1951 3.2.4); thread t of T copies
// aligned output dwords, the few bytes before and after them singly.
__device__ __forceinline__ int32_t store_copy(Out &o, const uint8_t *src, uint32_t ln, uint32_t t, uint32_t T) {
  if (o.pos + ln > o.cap) return kOverflow;
  uint8_t *d = o.dst + o.pos;
  const uint32_t head = min((uint32_t)(-reinterpret_cast<uintptr_t>(d) & 3), ln);
  const uint32_t nd = (ln - head) / 4, tail = head + 4 * nd;
  if (t < head) {
    d[t] = src[t];
    adler_add(o, o.pos + t, src[t]);
  }
  if (t < ln - tail) {
    d[tail + t] = src[tail + t];
    adler_add(o, o.pos + tail + t, src[tail + t]);
  }
  for (uint32_t k = t; k < nd; k += T) {
    uint32_t v;
    __builtin_memcpy(&v, src + head + 4 * k, 4);
    *reinterpret_cast<uint32_t *>(d + head + 4 * k) = v;
    const uint32_t sum = __builtin_amdgcn_udot4(v, 0x01010101u, 0u, false);
    o.s1 += sum;
    o.s2 = (o.s2 + ((o.pos + head + 4 * k) % 65521u) * sum + __builtin_amdgcn_udot4(v, 0x03020100u, 0u, false)) % 65521u;
  }
  o.s1 %= 65521u;
  o.pos += ln;
  return kOk;
}

// The Adler-32 of the bytes written: the lanes' partial sums (each < 65521)
// over the waves of the group.
template <class C> __device__ __forceinline__ uint32_t out_adler(Out &o, Sh<C> &S, uint32_t wave) {
  uint32_t s1r = o.s1, s2r = o.s2;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    s1r += __shfl_xor(s1r, d, kWave);
    s2r += __shfl_xor(s2r, d, kWave);
  }
  uint64_t s1 = s1r, s2 = s2r;
  if constexpr (C::kNW > 1) {
    S.part[0][wave] = s1r;
    S.part[1][wave] = s2r;
    group_sync<C>();
    s1 = s2 = 0;
    for (int i = 0; i < C::kNW; i++) {
      s1 += S.part[0][i];
      s2 += S.part[1][i];
    }
  }
  s1 %= 65521u;
  s2 %= 65521u;
  const uint64_t n = o.pos % 65521u;
  const uint32_t A = (uint32_t)((1 + s1) % 65521u);
  const uint32_t B = (uint32_t)((n * ((1 + s1) % 65521u) + 65521u * 65521u - s2) % 65521u);
  return uni((B << 16) | A);
}

// ------------------------------------------------------------- table build

// cl: the code bits the lookup consumes (the code's length, less the root bits
// in a sub-table).
__device__ __forceinline__ uint32_t make_entry(uint32_t tab, uint32_t sym, uint32_t cl) {
  if (tab == kTabCodes) return cl | (sym << 14);
  if (tab == kTabDist) {
    if (sym >= 30) return 0;
    const uint32_t x = dist_extra(sym);
    return (cl + x) | (x << 5) | (cl << 9) | (dist_base(sym, x) << 14);
  }
  if (sym < 256) return cl | (cl << 9) | kLitFlag | (sym << 14);
  if (sym == 256 || sym > 285) return 0;
  const uint32_t c = sym - 257, x = len_extra(c);
  return (cl + x) | (x << 5) | (cl << 9) | (len_base(c, x) << 14) | kLenType;
}

// Builds the canonical tables for n code lengths in lens[], the root table of
// 2^bits entries at tab + at and up to `room` sub-table entries behind it.
// Applies zlib's acceptance rules (inftrees.c): an over-subscribed set is
// rejected; an incomplete set is rejected unless it has a single code of
// length 1 (literal/distance tables) or no codes at all.
// The tables are filled per entry: with the codes left-justified to 15 bits,
// lim[L] is the first value above the codes of up to L bits, so a value's code
// length is one more than the number of limits it reaches (no loop over the
// 2^(bits - L) copies of a short code, which one lane would write alone). Codes
// longer than the root share their first `bits` bits p with a range of values
// that ends below (p + 1) << (15 - bits); the longest of them is the last, so
// its length sizes p's sub-table.
// Out of line: it runs once per block.
template <int NSYM>
__device__ __noinline__ int32_t build_table(const lds<uint8_t> *lens, uint32_t n, uint32_t kind,
                                            lds<Huff<NSYM>> *h, lds<uint32_t> *tab, uint32_t at, uint32_t bits,
                                            uint32_t room) {
  const uint32_t lane = lane_id();
  lds<uint32_t> *root = tab + at;
  // lane L: the number of codes of length L
  uint32_t mycount = 0;
  for (uint32_t base = 0; base < n; base += kWave) {
    const uint32_t L = base + lane < n ? lens[base + lane] : 0u;
    const uint64_t b0 = __ballot(L & 1), b1 = __ballot(L & 2), b2 = __ballot(L & 4), b3 = __ballot(L & 8);
    const uint64_t m = (lane & 1 ? b0 : ~b0) & (lane & 2 ? b1 : ~b1) & (lane & 4 ? b2 : ~b2) & (lane & 8 ? b3 : ~b3);
    mycount += (uint32_t)__builtin_popcountll(m);
  }
  int32_t left = 1;
  uint32_t maxlen = 0, code = 0, idx = 0;
  uint32_t first_l = 0, index_l = 0;
  uint32_t lim[16];
#pragma unroll
  for (uint32_t L = 1; L < 16; L++) {
    const uint32_t c = rdlane(mycount, L);
    left = 2 * left - (int32_t)c;
    if (c) maxlen = L;
    if (L == lane) {
      first_l = code;
      index_l = idx;
    }
    lim[L] = (code + c) << (15 - L);
    code = (code + c) << 1;
    idx += c;
  }
  if (left < 0) return kCorrupt;
  if (left > 0) {
    if (kind == kTabCodes) return kCorrupt;
    if (maxlen > 1) return kCorrupt;
  }
  if (lane >= 1 && lane < 16) {
    h->count[lane] = (uint16_t)mycount;
    h->first[lane] = (uint16_t)first_l;
    h->index[lane] = (uint16_t)index_l;
  }
  // the symbols in code order: by length, then by value
  uint32_t run = index_l;  // lane L: the next place of a code of length L
  for (uint32_t base = 0; base < n; base += kWave) {
    const uint32_t L = base + lane < n ? lens[base + lane] : 0u;
    const uint64_t b0 = __ballot(L & 1), b1 = __ballot(L & 2), b2 = __ballot(L & 4), b3 = __ballot(L & 8);
    const uint64_t same = (L & 1 ? b0 : ~b0) & (L & 2 ? b1 : ~b1) & (L & 4 ? b2 : ~b2) & (L & 8 ? b3 : ~b3);
    const uint64_t mine =
        (lane & 1 ? b0 : ~b0) & (lane & 2 ? b1 : ~b1) & (lane & 4 ? b2 : ~b2) & (lane & 8 ? b3 : ~b3);
    const uint32_t place = __shfl(run, L, kWave) + (uint32_t)__builtin_popcountll(same & ((1ull << lane) - 1));
    if (L) h->sym[place] = (uint16_t)(base + lane);
    run += (uint32_t)__builtin_popcountll(mine);
  }
  lds_order();
  uint32_t limr = 0;                                   // lim[bits]
#pragma unroll
  for (uint32_t L = 1; L < 16; L++)
    if (L == bits) limr = lim[L];
  for (uint32_t k = lane; k < (1u << bits); k += kWave) {
    const uint32_t v = (__builtin_bitreverse32(k) >> (32 - bits)) << (15 - bits);
    uint32_t e = 0;
    if (v < limr) {  // else a longer code, or none
      uint32_t L = 1;
#pragma unroll
      for (uint32_t q = 1; q < 11; q++) L += v >= lim[q] ? 1u : 0u;  // bits <= 10: no longer code here
      const uint32_t c = v >> (15 - L);
      e = make_entry(kind, h->sym[h->index[L] + c - h->first[L]], L);
    }
    root[k] = e;
  }
  lds_order();
  if (maxlen <= bits) return kOk;
  // sub-tables of the prefixes from limr on, in order
  const uint32_t p0 = limr >> (15 - bits), p1 = 1u << bits;
  uint32_t used = 0;
  for (uint32_t base = p0; base < p1; base += kWave) {
    const uint32_t p = base + lane;
    uint32_t sb = 0;
    if (p < p1) {
      const uint32_t v = ((p + 1) << (15 - bits)) - 1;
      uint32_t L = 1;
#pragma unroll
      for (uint32_t q = 1; q < 15; q++) L += v >= lim[q] ? 1u : 0u;
      sb = L - bits;
    }
    const uint32_t size = sb ? 1u << sb : 0u;
    const uint32_t incl = wave_scan_dpp(size);
    const uint32_t to = used + incl - size;
    if (p < p1)
      root[__builtin_bitreverse32(p) >> (32 - bits)] =
          to + size <= room ? bits | (sb << 14) | ((at + (1u << bits) + to) << 19) | kSubType : 0u;
    used += rdlane(incl, kWave - 1);
  }
  lds_order();
  for (uint32_t i = rdlane(index_l, bits) + rdlane(mycount, bits) + lane; i < idx; i += kWave) {
    uint32_t L = bits + 1;  // the length of the i-th code
    for (uint32_t q = bits + 1; q < 15; q++) L += i >= h->index[q] + h->count[q] ? 1u : 0u;
    const uint32_t c = h->first[L] + (i - h->index[L]);
    const uint32_t sl = L - bits;  // code bits in the sub-table
    const uint32_t d = root[__builtin_bitreverse32(c >> sl) >> (32 - bits)];
    if (d == 0) continue;
    const uint32_t sb = (d >> 14) & 31, rev = __builtin_bitreverse32(c) >> (32 - L) >> bits;
    const uint32_t e = make_entry(kind, h->sym[i], sl);
    for (uint32_t k = rev; k < (1u << sb); k += 1u << sl) tab[((d >> 19) & 0x7ff) + k] = e;
  }
  lds_order();
  return kOk;
}

// Canonical decode of one code, RFC 1951 3.2.2: the code of length L is the first L stream bits read MSB-first, and
// it is valid when it lies in [first[L], first[L] + count[L]). Lane L (1..15)
// tests length L, so the tables are read once instead of once per length; the
// shortest length that hits is the code (canonical codes are prefix-free).
// Called by the whole wave. Returns the symbol or -1; *len gets the length.
template <int NSYM>
__device__ __forceinline__ int32_t slow_decode(const lds<Huff<NSYM>> *h, uint32_t buf, uint32_t *len) {
  const uint32_t lane = lane_id();
  const uint32_t L = lane & 15u;
  const uint32_t c = L ? h->count[L] : 0u, f = h->first[L], ix = h->index[L];
  const uint32_t code = __builtin_bitreverse32(buf) >> ((32u - L) & 31u);  // L = 0: unused
  const uint64_t m = __ballot(lane >= 1u && lane < 16u && code - f < c);
  if (m == 0) return -1;
  const uint32_t hit = (uint32_t)__builtin_ctzll(m);
  *len = hit;
  return (int32_t)uni(h->sym[rdlane(ix + code - f, hit)]);
}

// ------------------------------------------------------------- stream decode

// Status in the caller's convention: CODAG_CHUNK_* by default, cuDF's
// gpu_inflate_status_s codes (cudf_deflate.cuh:1243-1343: 0 ok, 1 output
// buffer too small, 2 input ended early, -1 invalid data) with
// CODAG_INFLATE_CUDF_STATUS.
__device__ __forceinline__ int32_t status_code(int32_t st, uint32_t flags) {
  if (!(flags & CODAG_INFLATE_CUDF_STATUS) || st == kOk) return st;
  return st == kOverflow ? 1 : (st == kTrunc ? 2 : -1);
}

// 32 stream bits from stage bit q on.
__device__ __forceinline__ uint32_t stage_bits(const lds<uint32_t> *stage, uint32_t q) {
  return __builtin_amdgcn_alignbit(stage[(q >> 5) + 1], stage[q >> 5], q);
}

// The chain of lengths from lane 0 on: lane j's n bits lead to lane j + n, and a
// length of 128 stops. Returns the lanes it visits; *next gets the bit behind the
// 64 that it leads to, or 128 + the lane that stops. Eight links written out with a
// fall-through test each: j is kept as j - 64, so the add's carry is the test.
__device__ __forceinline__ uint64_t chain_links(uint32_t n, uint32_t *next) {
  uint64_t M = 0;
  uint32_t j = 0u - (uint32_t)kWave;
  uint32_t t;
  asm("1:\n"
      ".rept 8\n"
      "s_bitset1_b64 %[M], %[j]\n"
      "v_readlane_b32 %[t], %[n], %[j]\n"
      "s_add_u32 %[j], %[j], %[t]\n"
      "s_cbranch_scc1 2f\n"
      ".endr\n"
      "s_branch 1b\n"
      "2:"
      : [j] "+s"(j), [M] "+s"(M), [t] "=&s"(t)
      : [n] "v"(n)
      : "scc");
  *next = j + (uint32_t)kWave;
  return M;
}

// Reads a dynamic block's code lengths (RFC 1951 3.2.7) from stage bit *q on
// and builds its tables; `limit` is the stage bit after the stream's last.
// The run-length coded lengths are decoded 64 bits at a time: lane j decodes
// the code that would start at bit q + j, a scalar chain through their lengths
// marks the true starts, a prefix sum of the repeat counts gives the positions
// and a prefix maximum the last length before each repeat. (A scalar loop, one
// code after the other, took 85 K cycles a block.)
template <class C>
__device__ __forceinline__ int32_t read_dynamic(lds<Sh<C>> *S, uint32_t *qp, uint32_t limit) {
  const uint32_t lane = lane_id();
  uint32_t q = *qp;
  const uint32_t h = uni(stage_bits(S->stage, q));
  const uint32_t nlen = (h & 31) + 257, ndist = ((h >> 5) & 31) + 1, ncode = ((h >> 10) & 15) + 4;
  q += 14;
  if (q > limit) return kTrunc;
  if (nlen > 286 || ndist > 30) return kCorrupt;  // zlib: "too many length or distance symbols"
  if (lane < 19)  // code-length code lengths, 3 bits each, in permuted order
    S->lens[kClOrder[lane]] = lane < ncode ? (uint8_t)(stage_bits(S->stage, q + 3 * lane) & 7) : (uint8_t)0;
  q += 3 * ncode;
  if (q > limit) return kTrunc;
  lds_order();
  const uint32_t total = nlen + ndist;
  // without any code zlib reads a length 0 from every bit, and no end-of-block in the end
  if (!__ballot(lane < 19 && S->lens[lane])) return q + total > limit ? kTrunc : kCorrupt;
  int32_t st = (int32_t)uni((uint32_t)build_table(S->lens, 19, kTabCodes, &S->hl, S->tab, 0, kCodeBits, 0));
  if (st != kOk) return st;
  for (uint32_t k = lane; k < sizeof(S->lens) / 4; k += kWave) reinterpret_cast<lds<uint32_t> *>(S->lens)[k] = 0;
  lds_order();
  uint32_t i = 0, prev = 0;
  while (i < total) {
    const uint32_t x = stage_bits(S->stage, q + lane);
    const uint32_t e = S->tab[x & ((1u << kCodeBits) - 1)];
    const uint32_t L = e & 31, sym = e >> 14;
    const uint32_t xb = sym < 16 ? 0u : (sym == 16 ? 2u : (sym == 17 ? 3u : 7u));
    const uint32_t rep = (sym < 16 ? 1u : (sym == 18 ? 11u : 3u)) + __builtin_amdgcn_ubfe(x, L, xb);
    const uint32_t tl = L ? L + xb : 128u;  // no such code: stops the chain
    uint32_t j;
    const uint64_t M = chain_links(tl, &j);  // the starts
    const bool start = (M >> lane) & 1 && L;
    const uint32_t incl = wave_scan_dpp(start ? rep : 0u);
    const uint32_t off = i + incl - rep;
    const bool take = start && off < total;
    // a repeat with no length before it, or past the last length: an error once it is read whole
    const uint64_t bad = __ballot(take && ((sym == 16 && off == 0) || off + rep > total));
    if (bad) return q + (uint32_t)__builtin_ctzll(bad) + rdlane(tl, (uint32_t)__builtin_ctzll(bad)) > limit ? kTrunc : kCorrupt;
    const uint32_t key = wave_max_dpp(start && sym != 16 ? ((lane + 1) << 8) | (sym < 16 ? sym : 0u) : 0u);
    const uint32_t val = key ? key & 0xff : prev;
    if (take && val)  // at most six copies of a length that is not 0
      for (uint32_t r = 0; r < rep; r++) S->lens[off + r] = (uint8_t)val;
    const uint64_t tm = __ballot(take);
    const uint32_t lastl = tm ? 63u - (uint32_t)__builtin_clzll(tm) : 0u;
    if (tm) i = rdlane(off + rep, lastl);
    prev = rdlane(val, kWave - 1);
    if (i >= total) {
      q += lastl + rdlane(tl, lastl);
    } else if (j >= 128u) {  // no such code at bit q + j - 128
      return q + (j - 128u) > limit ? kTrunc : kCorrupt;
    } else {
      q += j;
    }
  }
  if (q > limit) return kTrunc;
  lds_order();
  if (uni(S->lens[256]) == 0) return kCorrupt;  // zlib: "missing end-of-block"
  st = (int32_t)uni((uint32_t)build_table(S->lens, nlen, kTabLit, &S->hl, S->tab, 0, C::kLB, C::kLS));
  if (st != kOk) return st;
  *qp = q;
  return (int32_t)uni((uint32_t)build_table(S->lens + nlen, ndist, kTabDist, &S->hd, S->tab, C::kDistAt, C::kDB, C::kDS));
}

// The tables of the fixed codes (RFC 1951 3.2.6), entry by entry from their closed
// form: literals and lengths 256..279 have the 7-bit codes from 0 on, 0..143 the
// 8-bit codes from 48, 280..287 from 192, 144..255 the 9-bit codes from 400; the
// distances 5 bits. (Built from their lengths, as a dynamic block's, they were most
// of the time of a stream of 64 bytes.)
template <class C> __device__ __forceinline__ void load_fixed(lds<Sh<C>> *S) {
  const uint32_t lane = lane_id();
  static_assert(C::kLB >= 9 && C::kDB >= 5, "no sub-tables");
  for (uint32_t k = lane; k < (1u << C::kLB); k += kWave) {
    const uint32_t v = __builtin_bitreverse32(k) >> 23, c = v >> 1;
    const uint32_t L = v < 96 ? 7u : (v < 400 ? 8u : 9u);
    const uint32_t sym = v < 96 ? 256 + (v >> 2) : (v < 400 ? (c < 192 ? c - 48 : c + 88) : v - 256);
    S->tab[k] = make_entry(kTabLit, sym, L);
  }
  for (uint32_t k = lane; k < (1u << C::kDB); k += kWave)
    S->tab[C::kDistAt + k] = make_entry(kTabDist, __builtin_bitreverse32(k) >> 27, 5);
  for (uint32_t i = lane; i < 288; i += kWave)
    S->hl.sym[i] = (uint16_t)(i < 24 ? 256 + i : (i < 168 ? i - 24 : (i < 176 ? i + 112 : i - 32)));
  if (lane < 32) S->hd.sym[lane] = (uint16_t)lane;
  if (lane < 16) {
    S->hl.count[lane] = (uint16_t)(lane == 7 ? 24 : (lane == 8 ? 152 : (lane == 9 ? 112 : 0)));
    S->hl.first[lane] = (uint16_t)(lane == 8 ? 48 : (lane == 9 ? 400 : 0));
    S->hl.index[lane] = (uint16_t)(lane == 8 ? 24 : (lane == 9 ? 176 : 0));
    S->hd.count[lane] = (uint16_t)(lane == 5 ? 32 : 0);
    S->hd.first[lane] = 0;
    S->hd.index[lane] = 0;
  }
  lds_order();
}

// Decodes the one symbol at stage bit *q with zlib's rules: kMore and the token
// (literal: its byte, *dist = 0; else length and distance), kEob, or the status
// of an invalid symbol.
template <class C>
__device__ __forceinline__ int32_t one_symbol(const lds<Sh<C>> *S, uint32_t *q, uint32_t limit, uint32_t *len,
                                              uint32_t *dist) {
  uint32_t L = 0;
  const int32_t sym = slow_decode(&S->hl, uni(stage_bits(S->stage, *q)), &L);
  if (sym < 0) return *q >= limit ? kTrunc : kCorrupt;  // a set with such bits has one code, of one bit, or none
  *q += L;
  if (sym == 256) return kEob;
  if (sym > 285) return kCorrupt;
  *len = (uint32_t)sym;
  *dist = 0;
  if (sym < 256) return kMore;
  const uint32_t c = (uint32_t)sym - 257, lx = len_extra(c);
  *len = len_base(c, lx) + __builtin_amdgcn_ubfe(uni(stage_bits(S->stage, *q)), 0, lx);
  *q += lx;
  const int32_t ds = slow_decode(&S->hd, uni(stage_bits(S->stage, *q)), &L);
  if (ds < 0) return *q >= limit ? kTrunc : kCorrupt;
  *q += L;
  if (ds >= 30) return kCorrupt;
  const uint32_t dx = dist_extra((uint32_t)ds);
  *dist = dist_base((uint32_t)ds, dx) + __builtin_amdgcn_ubfe(uni(stage_bits(S->stage, *q)), 0, dx);
  *q += dx;
  return kMore;
}

enum : uint32_t { kOpEnd = 0, kOpSpan = 1, kOpStored = 2, kOpToken = 3 };

// The serial part of the decode, by one wave: with `symbol`, decodes the symbol
// at bit P that a span stopped at; outside a block, reads the next block header
// and builds its tables. *S gets what comes next: the operation (a span from
// bit P on; a stored block of ln bytes at bit P; one token; the end), its
// status and whether the block is the stream's last. Out of line, with its
// results in LDS, so that its scalars do not crowd the span decoder's.
// At most 4096 bits from P on are read: a dynamic header has less than 105 +
// 316 * 7 + 14 (each length costs at most 7 bits, a repeat of at least three 14).
template <class C>
__device__ __noinline__ void serial_step(const uint32_t *w, uint32_t nw, uint32_t limit_bits,
                                         uint32_t P, bool symbol, bool last, lds<Sh<C>> *S) {
  const uint32_t lane = lane_id();
  const uint32_t d0 = P >> 5;
  static_assert(C::kStage >= 130, "stage holds a block header");
  for (uint32_t k = lane; k < 130; k += kWave) S->stage[k] = d0 + k < nw ? w[d0 + k] : 0u;
  lds_order();
  const uint32_t limit = limit_bits - d0 * 32;
  uint32_t q = P & 31, op = kOpEnd, ln = 0, val = 0, dist = 0;
  int32_t st = kOk;
  bool inside = symbol;
  if (symbol) {
    st = one_symbol<C>(S, &q, limit, &val, &dist);
    if (q > limit) st = kTrunc;
    if (st == kMore) {
      st = kOk;
      op = kOpToken;
    } else if (st == kEob) {
      st = kOk;
      inside = false;
    }
  }
  if (st == kOk && !inside && !last) {
    const uint32_t h = uni(stage_bits(S->stage, q));
    q += 3;
    last = h & 1;
    const uint32_t type = (h >> 1) & 3;
    if (q > limit) {
      st = kTrunc;
    } else if (type == 0) {  // stored (RFC 1951 3.2.4)
      q = (q + 7) & ~7u;
      const uint32_t lw = uni(stage_bits(S->stage, q));
      q += 32;
      ln = lw & 0xffff;
      if (q > limit) st = kTrunc;
      else if (ln != (~lw >> 16)) st = kCorrupt;
      else if (q + ln * 8 > limit) st = kTrunc;
      else op = kOpStored;
    } else if (type == 1) {  // fixed Huffman
      load_fixed<C>(S);
      op = kOpSpan;
    } else if (type == 2) {  // dynamic Huffman
      st = read_dynamic<C>(S, &q, limit);
      if (st == kOk) op = kOpSpan;
    } else {
      st = kCorrupt;  // zlib: "invalid block type"
    }
  }
  if (lane == 0) {
    S->op = st == kOk ? op : (uint32_t)kOpEnd;
    S->P = d0 * 32 + q;
    S->ln = ln;
    S->val = val;
    S->dist = dist;
    S->st = st;
    S->last = last;
  }
  lds_order();
}

// ------------------------------------------------------------- span decode

// A lane's place in the staged stream: the two dwords at its bit and the one
// after them, which is read a lookup ahead, so that a lookup waits for one LDS
// read (its table) and not for two.
struct Place {
  uint32_t at, w0, w1, w2;
};

template <class Dwords> __device__ __forceinline__ Place place_at(Dwords stage, uint32_t q) {
  const Dwords s = stage + (q >> 5);
  return Place{q, s[0], s[1], s[2]};
}

// The 32 stream bits from the place on.
__device__ __forceinline__ uint32_t place_bits(const Place &p) { return __builtin_amdgcn_alignbit(p.w1, p.w0, p.at); }

// Moves the place on by n <= 31 bits.
template <class Dwords> __device__ __forceinline__ void place_move(Place &p, Dwords stage, uint32_t n) {
  const uint32_t to = p.at + n;
  const bool cross = to > (p.at | 31);
  p.w0 = cross ? p.w1 : p.w0;
  p.w1 = cross ? p.w2 : p.w1;
  p.w2 = stage[(to >> 5) + 2];
  p.at = to;
}

// The entry of bits x in the table of descriptor d.
template <class Dwords> __device__ __forceinline__ uint32_t look(Dwords tab, uint32_t x, uint32_t d) {
  return tab[(d >> 5) + __builtin_amdgcn_ubfe(x, 0, d)];  // the field's width is d's low five bits
}

// The value of a length or distance code: its base and extra bits.
__device__ __forceinline__ uint32_t entry_value(uint32_t e, uint32_t x) {
  return __builtin_amdgcn_ubfe(e, 14, 16) + __builtin_amdgcn_ubfe(x, __builtin_amdgcn_ubfe(e, 9, 4), __builtin_amdgcn_ubfe(e, 5, 4));
}

template <class C> __device__ __forceinline__ uint32_t next_table(uint32_t e) {
  const uint32_t sub = __builtin_amdgcn_ubfe(e, 14, 16), root = e >= kLenType ? C::kDistDesc : C::kLitDesc;
  return e >= kSubType ? sub : root;
}

// Decodes tokens from bit q on until one starts at or after `bound`: q becomes
// that start (on a stop, the start of the token that stops). A token that ends
// past `limit` stops. With Count, n gets the bytes the tokens produce. One
// lookup a step in straight-line code: one LDS latency and about 30 vector
// instructions; a branch per kind of entry doubled that in scalar mask
// work.
template <class C, bool Count, class Dwords>
__device__ __forceinline__ bool run_tokens(Dwords stage, Dwords tab, uint32_t &q, uint32_t bound, uint32_t limit,
                                           uint32_t &n) {
  uint32_t d = C::kLitDesc, pend = 1, end = bound;
  Place p = place_at(stage, q);
  while (q < end) {
    const uint32_t x = place_bits(p), e = look(tab, x, d);
    place_move(p, stage, e & 31);
    const bool good = (e & 31) != 0 && p.at <= limit;
    const bool whole = good && e < kLenType;
    if (Count) {
      uint32_t v = entry_value(e, x);
      asm("" : "+v"(v));  // every lane computes it: no branch
      n += whole ? pend : 0u;
      v = e < kLenType ? 1u : v;
      pend = e < kSubType ? v : pend;
    }
    q = whole ? p.at : q;
    end = good ? end : 0u;
    d = next_table<C>(e);
  }
  return end != bound;
}

// Writes the tokens of the group's lanes, in lane order: this lane's begin at
// stage bit q and produce n bytes. The lanes mark the bytes of one window after
// the other. The first output error in stream order ends it: the tokens before
// it are written.
template <class C>
__device__ __forceinline__ int32_t emit(Out &o, Sh<C> &S, uint32_t q, uint32_t n, uint32_t wave, uint32_t lane) {
  const uint32_t tid = wave * kWave + lane;
  const uint32_t incl = wave_scan_dpp(n);
  uint32_t x = incl - n, total = rdlane(incl, kWave - 1);
  if constexpr (C::kNW > 1) {
    if (lane == 0) S.part[0][wave] = total;
    __syncthreads();
    total = 0;
    for (uint32_t k = 0; k < (uint32_t)C::kNW; k++) {
      const uint32_t p = uni(S.part[0][k]);
      if (k < wave) x += p;
      total += p;
    }
  }
  const uint32_t end = x + n;  // this lane's bytes: [x, end) from o.pos on
  const bool check = o.pos < 32768u || o.pos + total > o.cap;
  uint32_t lastx = ~0u, lastm = 0;  // this lane's last token
  Place p = place_at(&S.stage[0], q);
  uint32_t done = 0;
  int32_t st = kOk;
  while (done < total) {
    uint32_t wn = min(C::kWin, total - done);
    for (uint32_t k = tid; k < (wn + 511) / 512 * 64; k += C::kThreads)
      reinterpret_cast<uint4 *>(S.win)[k] = uint4{~0u, ~0u, ~0u, ~0u};
    if (check && tid == 0) S.err = ~0u;
    group_sync<C>();
    // the bytes behind the last one count as literals
    if (tid == 0 && wn < C::kWin) S.win[wn] = 0x8000u;
    if (x > done && lastx < done) S.win[0] = (uint16_t)lastm;  // a token that began before this window
    const uint32_t stopx = min(end, done + wn);
    // One lookup a step without branches: a lookup that completes no token writes
    // its mark behind the window (with a branch for each kind of entry, 25 scalar
    // instructions more a step, 4096 chunks took 3.20 ms and 3 chunks 445 us, without
    // 3.09 and 419; both before the window was resolved four bytes a lane).
    uint32_t d = C::kLitDesc, mlen = 0, bad = ~0u;
    uint32_t goal = stopx;
    while (x < goal) {
      const uint32_t bits = place_bits(p), e = look(&S.tab[0], bits, d);
      place_move(p, &S.stage[0], e & 31);
      d = next_table<C>(e);
      const uint32_t v = entry_value(e, bits);
      const bool whole = e < kLenType, lit = e & kLitFlag;
      mlen = (int32_t)e >= (int32_t)kLenType ? v : mlen;
      const uint32_t tl = lit ? 1u : mlen;
      const uint32_t m = lit ? 0x8000u | v : v - 1;
      if (check) {
        const uint32_t at = o.pos + x;
        const uint32_t why =
            at + tl > o.cap ? (uint32_t)kOverflow : (!lit && v > at ? (uint32_t)kCorrupt : 0u);  // distance too far back
        bad = whole && why ? min(bad, x << 2 | why) : bad;
      }
      S.win[whole ? x - done : C::kWin] = (uint16_t)m;
      if constexpr (C::kNW > 1) {  // a mark for the next segment's wave, too
        const uint32_t b = (x - done + tl - 1) / C::kSeg * C::kSeg;
        if (whole && b > x - done && b < C::kWin) S.win[b] = (uint16_t)m;
      }
      lastx = whole ? x : lastx;
      lastm = whole ? m : lastm;
      x += whole ? tl : 0u;
      goal = (e & 31) ? goal : 0u;  // no stop in a counted range
    }
    if (check && bad != ~0u) atomicMin(&S.err, bad);
    group_sync<C>();
    if (check) {
      const uint32_t e = uni(S.err);
      if (e != ~0u) {
        wn = (e >> 2) - done;
        st = (int32_t)(e & 3);
      }
    }
    resolve_window<C::kNW, C::kSeg, true, C::kNW == 1>(o.dst, S.win, o.pos + done, wn, wave, lane, o.s1, o.s2);
    group_sync<C>();
    done += wn;
    if (st != kOk) break;
  }
  o.pos += done;
  return st;
}

// ------------------------------------------------------------- narrow decode

typedef uint32_t __attribute__((aligned(1))) unaligned_dword;

// What the narrow decoder leaves: the next stream bit, the output position and
// this lane's Adler-32 sums; whether a symbol at P needs the symbol loop.
struct Narrow {
  uint32_t P, pos, s1, s2, stopped;
  int32_t st;
};

// Output bytes per stream byte from which the narrow decoder is the faster. In a
// group of eight waves it leaves seven idle, so spans hold on longer there (128 KiB
// chunks of zeros with a one every 200 bytes, 78 output bytes per stream byte, spans
// and narrow, us: 512 chunks by eight waves 321, 577 (an earlier copy loop), 4096
// chunks by one wave 1998, 958).
template <class C> constexpr uint32_t kNarrowRatio = C::kNW > 1 ? 200 : 32;

// Decodes tokens from stream bit P on by one wave, 64 bits at a time: lane j looks
// up the token that would start at bit j, a scalar chain through their lengths
// marks those that do, and each is written at once: literals by their lanes,
// matches one after the other by all lanes, into the window's LDS as a ring of the
// last H bytes, which is stored in blocks of 1024 bytes. It is for long matches: a
// span costs about 200 instructions per 256 output bytes, whatever the tokens, and
// keeps two or three lanes busy with all of them, several times over; here a match
// of 258 bytes is five reads and writes. It is bound by latency, about 1.2 K cycles
// a match and 1.5 K per 64 bits. 128 KiB chunks of zeros, spans and this, us: 4096
// chunks 2593, 738, 512 chunks 540, 325, one 449, 303; of a repeated 300 bytes, 4096
// chunks 1656, 670; 600 streams of 4 MiB of zeros 23.8 and 10.0 ms.
// It goes on while the output is kNarrowRatio times the stream's bytes, or still
// promises to be by the room that is left, for 3072 bits at most. At most kTake
// bytes are produced from one set of 64 bits, so the ring's last H - kTake bytes are
// there for matches; sources before them, or before the first byte that is produced
// here, come from HBM, where all but the last 1024 bytes are.
template <class C>
__device__ __noinline__ Narrow narrow_span(const uint32_t *w_, uint32_t nw, uint32_t limit_bits, uint32_t P,
                                           uint8_t *dst_, uint32_t pos, uint32_t cap, uint32_t s1, uint32_t s2,
                                           lds<Sh<C>> *S) {
  constexpr uint32_t H = C::kNW == 1 ? 8192 : 32768, kTake = 2048, kStaged = 256;
  static_assert(H < sizeof(S->win) && kStaged <= C::kStage, "the ring fits the window, the dwords the stage");
  const uint32_t lane = lane_id();
  lds<uint8_t> *ring = reinterpret_cast<lds<uint8_t> *>(S->win);
  const glob<const uint32_t> *w = uni_ptr(w_);
  glob<uint8_t> *dst = uni_ptr(dst_);
  P = uni(P);
  pos = uni(pos);
  nw = uni(nw);
  limit_bits = uni(limit_bits);
  cap = uni(cap);
  const uint32_t enter = pos;
  uint32_t fl = pos;                   // bytes stored
  uint32_t d0 = 0, staged = 0;         // the stage holds dwords [d0, d0 + staged)
  uint32_t P1 = P, pos1 = pos;         // where the ratio is measured from
  uint32_t stopped = 0;
  int32_t st = kOk;
  auto store = [&](uint32_t to) __attribute__((always_inline)) {  // bytes [fl, to), to - fl <= 1024 + 3
    lds_order();
    const uint32_t head = min((0u - fl) & 3, to - fl);
    if (head) {
      if (lane < head) {
        const uint32_t b = ring[(fl + lane) & (H - 1)];
        dst[fl + lane] = (uint8_t)b;
        s1 += b;
        s2 = (s2 + ((fl + lane) % 65521u) * b) % 65521u;
      }
      fl += head;
    }
    uint32_t a1 = 0, a2 = 0;
    for (uint32_t k = 4 * lane; k < to - fl; k += 4 * kWave) {
      uint32_t b = *reinterpret_cast<lds<uint32_t> *>(ring + ((fl + k) & (H - 1)));
      glob<uint8_t> *d = dst + (fl + k);
      if (k + 4 <= to - fl) {
        *reinterpret_cast<glob<unaligned_dword> *>(d) = b;
      } else {
        b &= (1u << 8 * (to - fl - k)) - 1;
        for (uint32_t j = 0; j < to - fl - k; j++) d[j] = (uint8_t)(b >> 8 * j);
      }
      const uint32_t sum = __builtin_amdgcn_udot4(b, 0x01010101u, 0u, false);
      a1 += sum;
      a2 += k * sum + __builtin_amdgcn_udot4(b, 0x03020100u, 0u, false);
    }
    s1 = (s1 + a1) % 65521u;
    s2 = (s2 + (fl % 65521u) * a1 + a2) % 65521u;
    fl = to;
    lds_order();
  };
  for (;;) {
    if ((P >> 5) + 8 > d0 + staged) {  // 64 positions, a token of 48 bits and the dword behind it
      d0 = P >> 5;
      staged = kStaged;
      lds_order();
#pragma unroll
      for (uint32_t k = 0; k < kStaged; k += kWave) S->stage[k + lane] = d0 + k + lane < nw ? w[d0 + k + lane] : 0u;
      lds_order();
    }
    const uint32_t a = P - d0 * 32 + lane, limit = limit_bits - d0 * 32;
    // the token at bit a: `at` its end, len and val or dist. It has 48 bits at most,
    // and its last lookup begins at its 28th: all from the 64 bits at a
    const lds<uint32_t> *bits = S->stage + (a >> 5);
    const uint32_t b0 = bits[0], b1 = bits[1], b2 = bits[2];
    const uint32_t x0 = __builtin_amdgcn_alignbit(b1, b0, a), x1 = __builtin_amdgcn_alignbit(b2, b1, a);
    auto from_bit = [&](uint32_t q) __attribute__((always_inline)) { return __builtin_amdgcn_alignbit(x1, x0, q - a); };
    uint32_t x = x0, e = look((const lds<uint32_t> *)S->tab, x, C::kLitDesc), at = a + (e & 31);
    bool ok = (e & 31) != 0;
    const bool sub = ok && e >= kSubType;
    if (__ballot(sub)) {
      const uint32_t x2 = from_bit(at);
      const uint32_t e2 = look((const lds<uint32_t> *)S->tab, x2, sub ? __builtin_amdgcn_ubfe(e, 14, 16) : C::kLitDesc);
      x = sub ? x2 : x;
      e = sub ? e2 : e;
      at += sub ? e2 & 31 : 0u;
      ok = ok && (e & 31) != 0;
    }
    const bool lit = e & kLitFlag, match = ok && !lit;
    const uint32_t val = entry_value(e, x), len = lit ? 1u : val;
    uint32_t dist = 0;
    if (__ballot(match)) {
      uint32_t y = from_bit(at), f = look((const lds<uint32_t> *)S->tab, y, C::kDistDesc);
      uint32_t to = at + (f & 31);
      bool fine = (f & 31) != 0;
      const bool dsub = match && fine && f >= kSubType;
      if (__ballot(dsub)) {
        const uint32_t y2 = from_bit(to);
        const uint32_t f2 = look((const lds<uint32_t> *)S->tab, y2, dsub ? __builtin_amdgcn_ubfe(f, 14, 16) : C::kDistDesc);
        y = dsub ? y2 : y;
        f = dsub ? f2 : f;
        to += dsub ? f2 & 31 : 0u;
        fine = fine && (f & 31) != 0;
      }
      dist = match ? entry_value(f, y) : 0u;
      at = match ? to : at;
      ok = match ? fine : ok;
    }
    ok = ok && at <= limit;
    uint32_t next;
    const uint64_t M = chain_links(ok ? at - a : 128u, &next);
    const bool start = (M >> lane) & 1 && ok;
    const uint32_t incl = wave_scan_dpp(start ? len : 0u), off = incl - (start ? len : 0u);
    bool take = start && incl <= kTake;
    const uint64_t left = __ballot(start && !take);
    const uint32_t last = left ? (uint32_t)__builtin_ctzll(left) : 64u;  // the first token left for the next turn
    const bool over = take && pos + incl > cap, wrong = take && dist > pos + off;  // distance too far back
    const uint64_t bad = __ballot(over || wrong);
    uint64_t taken = __ballot(take);
    if (bad) {  // the tokens before the first error are written
      const uint32_t f = (uint32_t)__builtin_ctzll(bad);
      st = rdlane(over, f) ? kOverflow : kCorrupt;
      taken &= (1ull << f) - 1;
      take = take && lane < f;
    }
    const uint32_t total = taken ? rdlane(incl, 63u - (uint32_t)__builtin_clzll(taken)) : 0u;
    if (take && lit) ring[(pos + off) & (H - 1)] = (uint8_t)val;
    const uint32_t lo = max(enter, pos + kTake > H ? pos + kTake - H : 0u);  // the ring's first byte
    for (uint64_t mm = __ballot(take && !lit); mm; mm &= mm - 1) {
      const uint32_t l = (uint32_t)__builtin_ctzll(mm);
      const uint32_t n = rdlane(len, l), d = rdlane(dist, l), t = pos + rdlane(off, l), from = t - d;
      // ROWS rows of 64 bytes; the lanes behind the match write behind the ring
      auto copy = [&]<uint32_t ROWS>() __attribute__((always_inline)) {
        uint32_t src[ROWS], b[ROWS];
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) src[r] = from + r * kWave + lane;
        if (d < n) {
          // a match longer than its distance repeats its first d bytes; i + 0.5 is at
          // least 0.5 away from a multiple of d < 258, so the quotient is exact
          const float rc = __builtin_amdgcn_rcpf((float)d);
#pragma unroll
          for (uint32_t r = 0; r < ROWS; r++)
            src[r] -= __umul24((uint32_t)(((float)(r * kWave + lane) + 0.5f) * rc), d);
        }
        lds_order();
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) b[r] = ring[src[r] & (H - 1)];
        if (from < lo) {
#pragma unroll
          for (uint32_t r = 0; r < ROWS; r++)
            if (r * kWave + lane < n && src[r] < lo) b[r] = dst[src[r]];
          // waits here, and not on the other path, where it would wait for the stores
#pragma unroll
          for (uint32_t r = 0; r < ROWS; r++) asm volatile("" : "+v"(b[r]));
        }
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++)
          ring[r * kWave + lane < n ? (t + r * kWave + lane) & (H - 1) : H] = (uint8_t)b[r];
      };
      if (n <= kWave) copy.template operator()<1>();
      else if (n <= 3 * kWave) copy.template operator()<3>();
      else copy.template operator()<5>();
    }
    pos += total;
    if (bad) break;
    while (pos - fl >= 1024) store(fl + 1024 - (fl & 3));
    if (left) {
      P += last;
    } else {
      P += next >= 128 ? next - 128 : next;
      if (next >= 128) {
        stopped = 1;
        break;
      }
    }
    if (P - P1 >= 1024) {
      if ((pos - pos1) * 8 >= kNarrowRatio<C> * (P - P1)) {
        P1 = P;
        pos1 = pos;
      } else if (P - P1 >= 3072 || (uint64_t)(cap - pos) * 8 < (uint64_t)kNarrowRatio<C> * (limit_bits - P)) {
        break;
      }
    }
  }
  while (fl < pos) store(min(pos, fl + 1024 - (fl & 3)));
  return Narrow{P, pos, s1, s2, stopped, st};
}

// Where a span's lanes do not find each other's token starts (codes of nearly one
// length keep a wrong phase: 128 equally frequent bytes, say), lane j decodes its
// part from each of the 16 bits at which the token before it may end, and a chain
// through these exits gives every lane its entry. A candidate whose first token ends
// at another one has its exit (of 7-bit literals, 7 or 8 of the 16 are decoded). A
// part that begins further behind, after a match, is decoded from there when the
// chain comes to it. Returns the lanes that have an entry, all up to the first that
// stops, and this lane's entry in the low half. 128 KiB chunks of 7-bit literals, by
// passes where the chain broke at a match, all 16 decoded, and now: 4096 chunks by
// one wave each 24.3 and 11.1 ms, 512 by eight waves 11.9 and 2.3 ms; base64 text,
// 512 chunks 4.9 and 3.1 ms.
template <class C>
__device__ __noinline__ uint64_t chain_entries(lds<Sh<C>> *S, uint32_t lo, uint32_t bound, uint32_t limit, uint32_t wave) {
  const uint32_t lane = lane_id();
  const lds<uint32_t> *stage = S->stage, *tab = S->tab;
  if constexpr (C::kNW > 1) __syncthreads();  // mis and stp are free
  // the exit behind `bound` of entry q, 255 = stop
  auto exit_of = [&](uint32_t q) __attribute__((always_inline)) {
    uint32_t n = 0;
    const bool stop = run_tokens<C, false, const lds<uint32_t> *>(stage, tab, q, bound, limit, n);
    return stop ? 255u : q - bound;
  };
  uint32_t exits[4] = {0, 0, 0, 0};  // byte c: of entry lo + c
#pragma unroll 1
  for (uint32_t c = 16; c-- > 0;) {
    // a literal that the root table holds leads to candidate `to`
    const uint32_t e = look(tab, stage_bits(stage, lo + c), C::kLitDesc), to = c + (e & 31);
    const bool known = (e & 31) && e < kLenType && to < 16 && lo + to <= limit;
    const uint32_t m = to < 4 ? exits[0] : to < 8 ? exits[1] : to < 12 ? exits[2] : exits[3];
    uint32_t x = (m >> 8 * (to & 3)) & 255;
    if (__ballot(!known)) {
      const uint32_t y = exit_of(lo + c);
      x = known ? x : y;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) exits[k] |= c / 4 == k ? x << 8 * (c & 3) : 0u;
  }
  uint32_t entry = lo, off = 0, have = 0;
  for (uint32_t w = 0; w < (uint32_t)C::kNW; w++) {
    if (w == wave) {
      for (; have < (uint32_t)kWave && off != 255; have++) {
        if (lane == have) entry = lo + off;
        uint32_t m;
        if (off < 16) {
          const uint32_t k = off / 4;
          m = (k == 0 ? exits[0] : k == 1 ? exits[1] : k == 2 ? exits[2] : exits[3]) >> 8 * (off & 3);
        } else {
          m = exit_of(lo + off);
        }
        off = rdlane(m, have) & 255;
      }
    }
    if constexpr (C::kNW > 1) {
      if (w == wave && lane == 0) {
        S->mis[w] = have;
        S->stp[w] = off;
      }
      __syncthreads();
      have = uni(S->mis[w]);
      off = uni(S->stp[w]);
      if (off == 255) return (uint64_t)(w * kWave + have) << 32 | entry;
      have = 0;
    }
  }
  return (uint64_t)(C::kNW > 1 ? C::kThreads : have) << 32 | entry;
}

// Decodes and writes the tokens of one span from stream bit P on; P becomes the
// bit after the last token written. *stopped: a symbol there needs the symbol
// loop. Returns the first output error.
template <class C>
__device__ __forceinline__ int32_t span(const uint32_t *w, uint32_t nw, uint32_t limit_bits, uint32_t &P, bool &stopped,
                                        uint32_t &hard, Out &o, Sh<C> &S, uint32_t wave, uint32_t lane) {
  constexpr uint32_t max_pass = 8;  // pass k verifies at least k lanes
  const uint32_t tid = wave * kWave + lane;
  const uint32_t d0 = P >> 5, off0 = P & 31;
  {
    constexpr uint32_t N = (C::kStage + C::kThreads - 1) / C::kThreads;
    const __amdgpu_buffer_rsrc_t rsrc = buffer_of(w, nw * 4);
    uint32_t v[N];
#pragma unroll
    for (uint32_t k = 0; k < N; k++)
      v[k] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (d0 + k * C::kThreads + tid) * 4, 0, 0);
#pragma unroll
    for (uint32_t k = 0; k < N; k++)
      if (k * C::kThreads + tid < C::kStage) S.stage[k * C::kThreads + tid] = v[k];
  }
  const uint32_t limit = limit_bits - d0 * 32;
  group_sync<C>();
  const uint32_t lo = off0 + tid * C::kSpanBits, bound = lo + C::kSpanBits;
  uint32_t entry = lo, q = lo, n = 0;
  uint32_t sq[C::kSub], sn[C::kSub];
#pragma unroll
  for (int k = 0; k < C::kSub; k++) sq[k] = sn[k] = 0;
  bool stop = false;
  uint32_t valid;  // lanes verified
  if (hard == kHard) {
    const uint64_t r = chain_entries<C>((lds<Sh<C>> *)&S, lo, bound, limit, wave);
    valid = uni((uint32_t)(r >> 32));
    q = (uint32_t)r;
#pragma unroll
    for (int k = 0; k < C::kSub; k++) {
      sq[k] = q;
      n = 0;
      if (!stop) stop = run_tokens<C, true>(&S.stage[0], &S.tab[0], q, lo + (k + 1) * C::kSpanBits / C::kSub, limit, n);
      sn[k] = n;
    }
  } else {
    stop = run_tokens<C, false>(&S.stage[0], &S.tab[0], q, bound, limit, n);
    for (uint32_t pass = 2;; pass++) {
      const uint32_t mine = q | (stop ? 0x80000000u : 0u);
      uint32_t up = __shfl_up(mine, 1, kWave);
      if constexpr (C::kNW > 1) {
        if (lane == kWave - 1) S.ex[wave] = mine;
        __syncthreads();
        if (lane == 0 && wave) up = S.ex[wave - 1];
      }
      const uint32_t next = tid == 0 ? off0 : (up >> 31 ? entry : up);
      const uint64_t mm = __ballot(next != entry), sm = __ballot(stop);
      uint32_t fm = mm ? wave * kWave + (uint32_t)__builtin_ctzll(mm) : C::kThreads;
      uint32_t fs = sm ? wave * kWave + (uint32_t)__builtin_ctzll(sm) : C::kThreads;
      if constexpr (C::kNW > 1) {
        if (lane == 0) {
          S.mis[wave] = fm;
          S.stp[wave] = fs;
        }
        __syncthreads();
        for (uint32_t k = 0; k < (uint32_t)C::kNW; k++) {
          fm = min(fm, uni(S.mis[k]));
          fs = min(fs, uni(S.stp[k]));
        }
      }
      if (pass > 2 && (fm > fs || fm == C::kThreads)) {
        valid = min(fs + 1, C::kThreads);
        break;
      }
      if (pass > max_pass) {
        valid = fm;  // the verified lanes make the span
        if (valid < kFewLanes<C>) hard++;
        break;
      }
      // every lane counts its bytes in pass 2; later only lanes with a new entry
      // (those behind a stop, too: most stops before the last pass are not real)
      if (pass == 2 || next != entry) {
        const uint32_t q0 = q;
        const bool stop0 = stop;
        bool met = false;  // back on the tokens of the pass before
        entry = q = next;
        stop = false;
#pragma unroll
        for (int k = 0; k < C::kSub; k++) {
          if (k && pass > 2 && q == sq[k]) met = true;
          if (!met) {
            sq[k] = q;
            n = 0;
            if (!stop) stop = run_tokens<C, true>(&S.stage[0], &S.tab[0], q, lo + (k + 1) * C::kSpanBits / C::kSub, limit, n);
            sn[k] = n;
          }
        }
        if (met) {
          q = q0;
          stop = stop0;
        }
      }
    }
  }
  if (tid >= valid) {
#pragma unroll
    for (int k = 0; k < C::kSub; k++) sn[k] = 0;
  }
  // the exit of the last verified lane, and whether it stopped there
  uint32_t endq = rdlane(q | (stop ? 0x80000000u : 0u), (valid - 1) & (kWave - 1));
  if constexpr (C::kNW > 1) {
    if (wave == (valid - 1) / kWave && lane == 0) S.end = endq;  // read after emit's barriers
  }
  int32_t st = kOk;
#pragma unroll 1
  for (int g = 0; g < C::kSub && st == kOk; g++) {
    uint32_t eq = sq[0], en = sn[0];
    if constexpr (C::kSub > 1) {
      const uint32_t l = g * (kWave / C::kSub) + lane / C::kSub;
      eq = en = 0;
#pragma unroll
      for (int k = 0; k < C::kSub; k++) {
        const uint32_t a = __shfl(sq[k], l, kWave), b = __shfl(sn[k], l, kWave);
        if ((int)(lane % C::kSub) == k) {
          eq = a;
          en = b;
        }
      }
    }
    st = emit<C>(o, S, eq, en, wave, lane);
  }
  if constexpr (C::kNW > 1) endq = uni(S.end);
  stopped = endq >> 31;
  P = d0 * 32 + (endq & 0x7fffffffu);
  return st;
}

struct Result {
  int32_t status;
  uint64_t bytes;
  uint32_t adler;
};

// ------------------------------------------------------------- CRC-32 (gzip)

// CRC-32 of RFC 1952 (reflected polynomial 0xEDB88320). Polynomials mod P are
// held bit-reflected: bit 31 is x^0. mulmod multiplies two of them (shift
// and add over GF(2)); kX2n[k] is x^(2^k) mod P, so x^(8n) mod P is a product
// of kX2n entries over the bits of n (the combination rule zlib's
// crc32_combine uses: crc(A B) = crc(A) * x^(8|B|) + crc(B)).
constexpr uint32_t kCrcPoly = 0xEDB88320u;

__host__ __device__ constexpr uint32_t crc_mulmod(uint32_t a, uint32_t b) {
  uint32_t m = 1u << 31, p = 0;
  for (;;) {
    if (a & m) {
      p ^= b;
      if ((a & (m - 1)) == 0) break;
    }
    m >>= 1;
    b = (b & 1) ? (b >> 1) ^ kCrcPoly : b >> 1;
  }
  return p;
}

struct X2nTable {
  uint32_t t[32];
  constexpr X2nTable() : t() {
    uint32_t p = 1u << 30;  // x^1
    t[0] = p;
    for (int k = 1; k < 32; k++) t[k] = p = crc_mulmod(p, p);
  }
};
__constant__ X2nTable kX2n = X2nTable();

// b * a mod P for a wave-uniform a.
__device__ __forceinline__ uint32_t crc_scale(uint32_t a, uint32_t b) {
  uint32_t p = 0;
#pragma unroll 4
  for (uint32_t k = 0; k < 32; k++) {
    p ^= (a >> 31) ? b : 0u;
    a <<= 1;
    b = (b >> 1) ^ ((b & 1) ? kCrcPoly : 0u);
  }
  return p;
}

// Builds the four 256-entry slice tables in `tab` (4 KiB of LDS) by T threads;
// sync() orders the threads.
template <class F> __device__ __forceinline__ void crc_tables(uint32_t *tab, uint32_t t, uint32_t T, F sync) {
  for (uint32_t i = t; i < 256; i += T) {
    uint32_t c = i;
#pragma unroll
    for (int k = 0; k < 8; k++) c = (c & 1) ? (c >> 1) ^ kCrcPoly : c >> 1;
    tab[i] = c;
  }
  sync();
#pragma unroll
  for (int k = 1; k < 4; k++) {
    for (uint32_t i = t; i < 256; i += T) {
      const uint32_t c = tab[(k - 1) * 256 + i];
      tab[k * 256 + i] = (c >> 8) ^ tab[c & 0xff];
    }
    sync();
  }
}

__device__ __forceinline__ uint32_t crc_dword(const uint32_t *tab, uint32_t c, uint32_t v) {
  c ^= v;
  return tab[768 + (c & 0xff)] ^ tab[512 + ((c >> 8) & 0xff)] ^ tab[256 + ((c >> 16) & 0xff)] ^ tab[c >> 24];
}

// The CRC register, begun at 0, after this wave's part of the n bytes at p:
// thread t of T takes 2^lg bytes, the last thread the last ones, so that the
// bytes missing to T * 2^lg stand at the front, where zeros leave the register
// at 0. Neighbours are combined pairwise (crc(A B) = crc(A) * x^(8|B|) +
// crc(B), all B of a step of one length), 6 products for 64 lanes; combined one
// lane after the other, with a length of its own each, 64 lanes took about 80.
__device__ __forceinline__ uint32_t crc_part(const uint8_t *p, uint32_t n, uint32_t lg, const uint32_t *tab,
                                             uint32_t t, uint32_t T) {
  const uint64_t behind = (uint64_t)(T - 1 - t) << lg;  // bytes after this thread's
  uint32_t c = 0;
  if (behind < n) {
    const uint32_t hi = n - (uint32_t)behind, len = min(hi, 1u << lg);
    uint32_t i = hi - len;
    for (; i < hi && ((hi - i) & 15); i++) c = tab[(c ^ p[i]) & 0xff] ^ (c >> 8);
    for (; i < hi; i += 16) {
      uint4 v;
      __builtin_memcpy(&v, p + i, 16);
      c = crc_dword(tab, crc_dword(tab, crc_dword(tab, crc_dword(tab, c, v.x), v.y), v.z), v.w);
    }
  }
#pragma unroll 1
  for (uint32_t k = 0; k < 6; k++) c ^= crc_scale(kX2n.t[(3 + lg + k) & 31], __shfl_up(c, 1u << k, kWave));
  return rdlane(c, kWave - 1);
}

// x^(8n) times the register's first value, all ones: what the bytes before the
// first one contribute.
__device__ __forceinline__ uint32_t crc_begin(uint32_t n) {
  uint32_t c = 0xFFFFFFFFu;
  for (uint32_t k = 3; n; n >>= 1, k++)
    if (n & 1) c = crc_scale(kX2n.t[k & 31], c);
  return c;
}

// Log2 of the bytes per thread, at least 16 (n < 2^31).
__device__ __forceinline__ uint32_t crc_share(uint32_t n, uint32_t T) {
  const uint32_t each = max((n + T - 1) / T, 16u);
  return 32u - (uint32_t)__builtin_clz(each - 1);
}

// CRC-32 of n bytes at global address p by one wave; `tab`: 4 KiB of LDS.
__device__ __forceinline__ uint32_t wave_crc32(const uint8_t *p, uint32_t n, uint32_t *tab) {
  const uint32_t lane = lane_id();
  wave_sync();
  crc_tables(tab, lane, kWave, [] { wave_sync(); });
  const uint32_t c = crc_part(p, n, crc_share(n, kWave), tab, lane, kWave);
  wave_sync();
  return uni(~(c ^ crc_begin(n)));
}

// The same by the whole group, which has written the bytes.
template <class C>
__device__ __forceinline__ uint32_t group_crc32(const uint8_t *p, uint32_t n, Sh<C> &S, uint32_t wave, uint32_t lane) {
  uint32_t *tab = reinterpret_cast<uint32_t *>(S.win);
  const uint32_t tid = wave * kWave + lane, lg = crc_share(n, C::kThreads);
  group_sync<C>();
  crc_tables(tab, tid, C::kThreads, [] { group_sync<C>(); });
  uint32_t c = crc_part(p, n, lg, tab, tid, C::kThreads);
  if constexpr (C::kNW > 1) {
    if (lane == 0) S.part[0][wave] = c;
    __syncthreads();
    c = S.part[0][0];
    for (uint32_t k = 1; k < (uint32_t)C::kNW; k++) c = crc_scale(kX2n.t[(9 + lg) & 31], c) ^ S.part[0][k];
    __syncthreads();
  }
  return uni(~(c ^ crc_begin(n)));
}

// gzip member header (RFC 1952 2.3), checked as zlib's inflate() checks it:
// ID1 ID2 = 1f 8b, CM = 8, no reserved FLG bits, FEXTRA / FNAME / FCOMMENT
// skipped, FHCRC compared with the low 16 bits of the header's CRC-32.
// Returns the header length, or -kTrunc / -kCorrupt.
__device__ __forceinline__ int64_t gzip_header(const uint8_t *src, uint64_t len, uint32_t *tab) {
  const uint32_t lane = lane_id();
  if (len < 10) {
    // zlib reports a short header as truncated unless a byte it has already
    // read is wrong
    const uint32_t b0 = len > 0 ? uni(src[0]) : 0x1f, b1 = len > 1 ? uni(src[1]) : 0x8b;
    const uint32_t b2 = len > 2 ? uni(src[2]) : 8, b3 = len > 3 ? uni(src[3]) : 0;
    if (b0 != 0x1f || b1 != 0x8b || b2 != 8 || (b3 & 0xe0)) return -kCorrupt;
    return -kTrunc;
  }
  if (uni(src[0]) != 0x1f || uni(src[1]) != 0x8b || uni(src[2]) != 8) return -kCorrupt;
  const uint32_t flg = uni(src[3]);
  if (flg & 0xe0) return -kCorrupt;
  uint64_t at = 10;
  if (flg & 0x04) {  // FEXTRA
    if (at + 2 > len) return -kTrunc;
    const uint32_t xlen = uni(src[at]) | (uni(src[at + 1]) << 8);
    at += 2 + xlen;
    if (at > len) return -kTrunc;
  }
  for (uint32_t f = 0x08; f <= 0x10; f <<= 1) {  // FNAME, FCOMMENT: zero-terminated
    if (!(flg & f)) continue;
    for (;;) {
      if (at >= len) return -kTrunc;
      const uint64_t q = at + lane;
      const bool z = q < len && src[q] == 0;
      const uint64_t m = __ballot(z);
      if (m) {
        at += (uint64_t)__builtin_ctzll(m) + 1;
        break;
      }
      at += kWave;
    }
  }
  if (flg & 0x02) {  // FHCRC
    if (at + 2 > len) return -kTrunc;
    const uint32_t want = uni(src[at]) | (uni(src[at + 1]) << 8);
    if ((wave_crc32(src, (uint32_t)at, tab) & 0xffff) != want) return -kCorrupt;
    at += 2;
  }
  return (int64_t)at;
}

// ------------------------------------------------------------- streams

// Decodes one zlib / raw / gzip stream by the whole group. Wave 0 reads the
// headers, builds the tables and decodes the symbols that stop a span; spans
// and stored blocks are done by all waves. The result is wave 0's.
template <class C>
__device__ __forceinline__ Result inflate_group(const uint8_t *src, uint64_t len, uint8_t *dst, uint64_t cap,
                                                uint32_t flags, Sh<C> &S) {
  const uint32_t lane = lane_id();
  const uint32_t wave = C::kNW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x) / kWave : 0u;
  Result res{kOk, 0, 1};
  // 32-bit bit positions bound the stream to < 2^28 bytes; outputs are
  // capped below 2^31 bytes.
  if (len >= (1ull << 28)) {
    res.status = kCorrupt;
    return res;
  }
  if (cap > 0x7fffffffull) cap = 0x7fffffffull;
  const uintptr_t a = reinterpret_cast<uintptr_t>(src);
  const uint32_t lead = (uint32_t)(a & 3);
  const uint32_t *w = reinterpret_cast<const uint32_t *>(a - lead);  // bit positions count from here
  const uint32_t limit = (uint32_t)((lead + len) * 8);               // one past the stream's last bit
  const uint32_t nw = (uint32_t)((lead + len + 3) / 4);
  Out o;
  o.dst = dst;
  o.cap = (uint32_t)cap;
  o.pos = 0;
  o.s1 = 0;
  o.s2 = 0;
  const bool gzip = flags & CODAG_INFLATE_GZIP;
  const bool raw = (flags & CODAG_INFLATE_RAW) && !gzip;
  uint32_t *crc_tab = reinterpret_cast<uint32_t *>(S.win);
  int32_t st = kOk;
  uint64_t start = 0;
  if (wave == 0) {
    if (gzip) {
      const int64_t h = gzip_header(src, len, crc_tab);
      if (h < 0) st = (int32_t)(-h);
      else start = (uint64_t)h;
    } else if (!raw) {
      if (len < 2) {
        st = kTrunc;
      } else {
        const uint32_t cmf = uni(src[0]), flg = uni(src[1]);
        // zlib inflate.c: method 8, window <= 32K, header check, no preset dictionary
        if ((cmf & 15) != 8 || (cmf >> 4) > 7 || ((cmf << 8) | flg) % 31 != 0 || (flg & 0x20)) st = kCorrupt;
        start = 2;
      }
    }
  }
  const bool headed = st == kOk;  // the stream's header is accepted
  uint32_t P = (uint32_t)((lead + start) * 8);
  bool last = false, inside = false, stopped = false;
  uint32_t hard = 0;     // the block's spans in which few lanes were verified
  // the block goes on by narrow_span; the output's room has nothing to do with its bytes (wave 0)
  bool narrow = false, roomy = false;
  for (;;) {
    uint32_t op = kOpEnd;
    if (wave == 0) {
      while (st == kOk) {
        if (inside && !stopped) {
          if (!narrow) {
            op = kOpSpan;
            break;
          }
          const Narrow r = narrow_span<C>(w, nw, limit, P, o.dst, o.pos, o.cap, o.s1, o.s2, (lds<Sh<C>> *)&S);
          P = uni(r.P);
          o.pos = uni(r.pos);
          o.s1 = r.s1;
          o.s2 = r.s2;
          st = (int32_t)uni((uint32_t)r.st);
          stopped = uni(r.stopped);
          narrow = stopped;  // else it left for want of long matches: the sizes promised too much
          roomy = roomy || !stopped;
        } else if (inside || !last) {
          const bool symbol = inside;
          serial_step<C>(w, nw, limit, P, symbol, last, (lds<Sh<C>> *)&S);
          op = uni(S.op);
          P = uni(S.P);
          st = (int32_t)uni((uint32_t)S.st);
          last = uni(S.last);
          inside = op == kOpSpan || op == kOpToken;
          stopped = false;
          if (op == kOpToken) {
            const uint32_t val = uni(S.val), dist = uni(S.dist);
            st = out_token(o, lane, dist == 0, val, dist);
          }
          if (op == kOpStored || op == kOpEnd) break;
          if (op == kOpSpan) {  // a new block: by the bytes that the stream's rest has to give
            narrow = !roomy && (uint64_t)(o.cap - o.pos) * 8 >= (uint64_t)kNarrowRatio<C> * (limit - P);
          }
        } else {
          op = kOpEnd;
          break;
        }
      }
      if (st != kOk) op = kOpEnd;
    }
    if constexpr (C::kNW > 1) {
      if (threadIdx.x == 0) {
        S.op = op;
        S.P = P;
        S.pos = o.pos;
      }
      __syncthreads();
      op = uni(S.op);
      P = uni(S.P);
      o.pos = uni(S.pos);
    }
    if (op == kOpEnd) break;
    if (op == kOpSpan) {
      const uint32_t P0 = P, pos0 = o.pos;
      const int32_t e = span<C>(w, nw, limit, P, stopped, hard, o, S, wave, lane);
      if (wave == 0) st = e;
      // a block after one of equal code lengths is expected to be another
      hard = stopped ? (hard == kHard ? kHard - 1 : 0u) : hard;
      narrow = (uint64_t)(o.pos - pos0) * 8 >= (uint64_t)kNarrowRatio<C> * (P - P0);
    } else {
      const uint32_t ln = uni(S.ln);
      const int32_t e = store_copy(o, reinterpret_cast<const uint8_t *>(w) + P / 8, ln, wave * kWave + lane, C::kThreads);
      if (wave == 0) st = e;
      P += 8 * ln;
      group_sync<C>();  // the command is read by all
    }
  }
  const uint32_t check = gzip ? group_crc32<C>(dst, o.pos, S, wave, lane) : out_adler<C>(o, S, wave);
  if (wave != 0) return res;
  if (!headed) {
    res.status = st;
    return res;
  }
  res.adler = check;
  res.bytes = o.pos;
  if (gzip) {
    // RFC 1952 trailer on the next byte boundary: CRC-32 and ISIZE, both
    // little-endian; zlib checks the CRC first ("incorrect data check"),
    // then the length ("incorrect length check")
    if (st == kOk) {
      const uint64_t at = (P + 7) / 8 - lead;
      if (at + 8 > len) {
        st = kTrunc;
      } else {
        const uint32_t crc = uni(src[at]) | (uni(src[at + 1]) << 8) | (uni(src[at + 2]) << 16) |
                             (uni(src[at + 3]) << 24);
        const uint32_t isize = uni(src[at + 4]) | (uni(src[at + 5]) << 8) |
                               (uni(src[at + 6]) << 16) | (uni(src[at + 7]) << 24);
        if (!(flags & CODAG_INFLATE_SKIP_ADLER) && crc != res.adler) st = kCorrupt;
        else if (isize != (uint32_t)res.bytes) st = kCorrupt;
      }
    }
  } else if (st == kOk && !raw) {
    // RFC 1950 trailer: Adler-32, big-endian, on the next byte boundary
    const uint64_t at = (P + 7) / 8 - lead;
    if (at + 4 > len) {
      st = kTrunc;
    } else if (!(flags & CODAG_INFLATE_SKIP_ADLER)) {
      const uint32_t t = (uni(src[at]) << 24) | (uni(src[at + 1]) << 16) |
                         (uni(src[at + 2]) << 8) | uni(src[at + 3]);
      if (t != res.adler) st = kCorrupt;
    }
  }
  res.status = st;
  return res;
}

// Decodes and writes chunk c of a container; the group's result goes to its
// length and status words.
template <class C>
__device__ __forceinline__ void inflate_chunk(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *off,
                                              uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len, int32_t *status,
                                              uint32_t flags, Sh<C> &S) {
  const uint64_t c = blockIdx.x;
  const uint64_t o0 = off[c], o1 = off[c + 1];
  Result r{kCorrupt, 0, 0};
  if (o1 >= o0 && o1 <= comp_bytes)
    r = inflate_group<C>(comp + o0, o1 - o0, out + c * chunk_bytes, chunk_bytes, flags, S);
  if (threadIdx.x == 0) {
    if (status) status[c] = status_code(r.status, flags);
    if (out_len) out_len[c] = r.bytes;
  }
}

__global__ void __launch_bounds__(One::kThreads) __attribute__((amdgpu_waves_per_eu(3)))
inflate_chunks_kernel(const uint8_t *__restrict__ comp, uint64_t comp_bytes,
                      const uint64_t *__restrict__ off, uint64_t chunk_bytes, uint8_t *out,
                      uint64_t *__restrict__ out_len, int32_t *__restrict__ status, uint32_t flags) {
  __shared__ Sh<One> S;
  inflate_chunk<One>(comp, comp_bytes, off, chunk_bytes, out, out_len, status, flags, S);
}

__global__ void __launch_bounds__(Many::kThreads)
inflate_chunks_many_kernel(const uint8_t *__restrict__ comp, uint64_t comp_bytes,
                           const uint64_t *__restrict__ off, uint64_t chunk_bytes, uint8_t *out,
                           uint64_t *__restrict__ out_len, int32_t *__restrict__ status, uint32_t flags) {
  __shared__ Sh<Many> S;
  inflate_chunk<Many>(comp, comp_bytes, off, chunk_bytes, out, out_len, status, flags, S);
}

// The queue of a batch, in device memory: its next stream and whether groups of
// eight waves or of one decode it.
//  * The plan's constants are fits to zlib streams of text and numbers on 256 CUs:
//    one wave takes about 20 ns per compressed byte of its stream and the GPU's
//    one-wave groups together 1/85 ns; its eight-wave groups together take about
//    150 ns per stream and 1/78 ns per compressed byte. (gzip members also pay
//    their CRC-32: 3000 small ones go by eight waves, 0.93 ms, and would take 0.78
//    by one.) So eight waves win until
//    there are many streams of about one size. Mixed zlib streams from 4 KiB on
//    (one wave / eight waves, ms): 700 of up to 64 KiB 0.77 / 0.37, 3000 of up
//    to 64 KiB 0.86 / 0.90, of up to 1 MiB 11.2 / 4.5, 6000 of up to 16 KiB
//    0.49 / 1.08, of up to 256 KiB 3.19 / 3.39. (The large streams by eight
//    waves and then the small ones by one wave each was never the faster.)
//  * Streams that the narrow decoder takes keep one wave busy in either group: one
//    (600 streams of 128 KiB of zeros 0.33 / 0.63).
struct BatchQueue {
  uint32_t next;
  uint32_t many;
};
constexpr uint32_t kPlanThreads = 1024, kPlanSample = 1u << 16;

// Resets the queue and chooses the groups by the streams' sizes (of evenly
// spaced streams, where there are more than kPlanSample). `shape`: 0 chosen
// here, 1 one wave, 2 eight waves.
__global__ void __launch_bounds__(kPlanThreads)
plan_batch_kernel(const codag_stream_desc *__restrict__ descs, uint64_t n, BatchQueue *q, uint32_t shape) {
  __shared__ uint64_t sums[kPlanThreads / kWave], tops[kPlanThreads / kWave], rooms[kPlanThreads / kWave];
  const uint64_t m = min(n, (uint64_t)kPlanSample);
  uint64_t sum = 0, top = 0, room = 0;
  if (shape == 0)
    for (uint64_t k = threadIdx.x; k < m; k += blockDim.x) {
      const uint64_t b = min(descs[k * n / m].src_bytes, (uint64_t)1 << 28);
      sum += b;
      room += min(descs[k * n / m].dst_cap, (uint64_t)1 << 31);
      top = max(top, b);
    }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    sum += __shfl_xor(sum, d, kWave);
    room += __shfl_xor(room, d, kWave);
    top = max(top, __shfl_xor(top, d, kWave));
  }
  if (lane_id() == 0) {
    sums[threadIdx.x / kWave] = sum;
    tops[threadIdx.x / kWave] = top;
    rooms[threadIdx.x / kWave] = room;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  sum = top = room = 0;
  for (uint32_t i = 0; i < blockDim.x / kWave; i++) {
    sum += sums[i];
    top = max(top, tops[i]);
    room += rooms[i];
  }
  const bool small = room < kNarrowRatio<One> * sum;  // outputs below so many times their streams
  if (m) sum = sum / m * n;
  const uint64_t one = max(200000 + 20 * top, sum / 85), many = 150 * n + sum / 78;  // ns
  q->next = 0;
  q->many = shape == 0 ? small && many <= one : shape == 2;
}

// Persistent loop over a batch: each group takes the next stream from the queue
// until none is left.
template <class C>
__device__ __forceinline__ void inflate_batch(const codag_stream_desc *descs, uint64_t n, codag_stream_result *results,
                                              uint32_t flags, BatchQueue *q, Sh<C> &S) {
  if (q->many != (C::kNW > 1)) return;
  for (;;) {
    group_sync<C>();
    if (threadIdx.x == 0) S.stream = atomicAdd(&q->next, 1u);
    group_sync<C>();
    const uint32_t i = uni(S.stream);
    if ((uint64_t)i >= n) break;
    const codag_stream_desc d = descs[i];
    // In an uneven batch the largest streams set the finish time: their waves
    // issue first (wave priority by output size), the small streams fill the
    // remaining issue slots.
    const uint64_t big = d.dst_cap;
    if (big >= (2u << 20)) __builtin_amdgcn_s_setprio(3);
    else if (big >= (1u << 20)) __builtin_amdgcn_s_setprio(2);
    else if (big >= (512u << 10)) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    const Result r = inflate_group<C>(d.src, d.src_bytes, d.dst, d.dst_cap, flags, S);
    if (threadIdx.x == 0) {
      results[i].bytes_written = r.bytes;
      results[i].status = status_code(r.status, flags);
      results[i].adler32 = r.adler;
    }
  }
}

__global__ void __launch_bounds__(One::kThreads) __attribute__((amdgpu_waves_per_eu(3)))
inflate_batch_kernel(const codag_stream_desc *__restrict__ descs, uint64_t n,
                     codag_stream_result *__restrict__ results, uint32_t flags, BatchQueue *q) {
  __shared__ Sh<One> S;
  inflate_batch<One>(descs, n, results, flags, q, S);
}

__global__ void __launch_bounds__(Many::kThreads)
inflate_batch_many_kernel(const codag_stream_desc *__restrict__ descs, uint64_t n,
                          codag_stream_result *__restrict__ results, uint32_t flags, BatchQueue *q) {
  __shared__ Sh<Many> S;
  inflate_batch<Many>(descs, n, results, flags, q, S);
}

// Device memory of the allocation-free batch entry point: its queue. Every GPU holds its own copy for the life of the
// process; all calls on one GPU share it.
constexpr uint32_t kScratchWords = 64;  // 256 bytes
static __device__ __align__(256) uint32_t scratch[kScratchWords];
constexpr int kScratchDevices = 64;
static_assert(sizeof(BatchQueue) <= 256, "a queue fits a counter slot and the static array");

}  // namespace inflate

// Device address of `scratch` on the current device, looked up once per
// device with that device current (the host-side name is not a device
// address and must never reach a kernel).
hipError_t inflate_scratch_ptr(uint32_t **out) {
  static std::mutex mu;
  static uint32_t *ptrs[inflate::kScratchDevices] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= inflate::kScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(inflate::scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    ptrs[dev] = static_cast<uint32_t *>(p);
  }
  *out = ptrs[dev];
  return hipSuccess;
}

// many: eight waves per chunk, else one (inflate_many).
hipError_t launch_inflate_chunks(const uint8_t *comp, uint64_t comp_bytes, const uint64_t *off,
                                 uint64_t n, uint64_t chunk_bytes, uint8_t *out, uint64_t *out_len,
                                 int32_t *status, uint32_t flags, hipStream_t stream, bool many) {
  if (n == 0) return hipSuccess;
  if (many)
    hipLaunchKernelGGL(inflate::inflate_chunks_many_kernel, dim3((uint32_t)n), dim3(inflate::Many::kThreads), 0,
                       stream, comp, comp_bytes, off, chunk_bytes, out, out_len, status, flags);
  else
    hipLaunchKernelGGL(inflate::inflate_chunks_kernel, dim3((uint32_t)n), dim3(kWaveSize), 0,
                       stream, comp, comp_bytes, off, chunk_bytes, out, out_len, status, flags);
  return hipGetLastError();
}

// Batches that all fit the GPU at once (two eight-wave groups per CU) go to
// eight-wave groups; for larger ones the queue's plan picks one of two launches,
// and the other's groups leave at once. !by_size: one wave per stream.
hipError_t launch_inflate_batch(const codag_stream_desc *descs, uint64_t n,
                                codag_stream_result *results, uint32_t flags, uint32_t *counter,
                                uint32_t cus, uint32_t per_cu, hipStream_t stream, bool by_size) {
  using namespace inflate;
  auto *q = reinterpret_cast<BatchQueue *>(counter);
  const uint32_t shape = !by_size ? 1u : (n <= 2ull * cus ? 2u : 0u);
  hipLaunchKernelGGL(plan_batch_kernel, dim3(1), dim3(shape ? kWaveSize : kPlanThreads), 0, stream, descs, n, q, shape);
  if (n == 0) return hipGetLastError();
  if (shape != 1) {
    const uint64_t groups = std::min<uint64_t>(n, (uint64_t)cus * std::min(per_cu, 2u));
    hipLaunchKernelGGL(inflate_batch_many_kernel, dim3((uint32_t)groups), dim3(Many::kThreads), 0, stream, descs, n,
                       results, flags, q);
  }
  if (shape != 2) {
    const uint64_t groups = std::min<uint64_t>(n, (uint64_t)cus * per_cu);
    hipLaunchKernelGGL(inflate_batch_kernel, dim3((uint32_t)groups), dim3(kWaveSize), 0, stream, descs, n, results,
                       flags, q);
  }
  return hipGetLastError();
}

}  // namespace codag
