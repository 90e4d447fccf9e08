// window.hpp -- the output side shared by the Deflate and LZSS decoders: an LDS
// window of 16-bit marks, one per output byte, resolved into bytes by a group of
// NW waves and stored to HBM.
#pragma once

#include "device.hpp"

namespace codag {
namespace dev {

__device__ __forceinline__ uint32_t rdlane(uint32_t v, uint32_t j) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)j);
}

// Keeps the compiler from moving LDS accesses across it; a wave's LDS
// instructions are executed in order, so no wait is needed.
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Inclusive wave64 prefix maximum with DPP row shifts and row broadcasts.
__device__ __forceinline__ uint32_t wave_max_dpp(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return v;
}

// Buffer loads: a lane whose offset is not below the size takes no part in the
// load and gets 0, so no branch stands around it and the loads of several rows
// stay in flight together.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

// The bytes [0, wn) of the window at output position w0 are marked; resolves
// them, stores them and, with SUM, adds them to this lane's Adler-32 sums (sum b
// and sum pos*b, mod 65521). A mark is a literal (0x8000 | byte) or a match's
// distance - 1; a byte without one (0xffff) continues the token of the byte
// before it (a literal then repeats); a token also has a mark where it crosses
// into another wave's segment of SEG bytes. The window is initialised up to the
// next multiple of 512 bytes and has a literal mark behind its last byte.
// Each wave resolves its segment in groups of 256 bytes; the far sources of the
// next group are loaded while this one's near sources are followed. Nothing is
// stored before the segment is done: a wait for loads would also wait for the
// stores before them.
// A lane has one byte of each of the group's four rows of 64, or, with QUADS, four
// consecutive bytes: one prefix maximum a group instead of four and half the LDS
// instructions, but LDS gathers of a lane stride and far loads over four times
// the cache lines. Rows and quads, us: LZSS, 2048 chunks, 1000 and 932; one-wave Deflate,
// 4096 chunks, 3092 and 2963; eight-wave groups, 3000 gzip members, 912 and 962.
// A group's bytes first get 0x8000 | byte where the byte is known (literals,
// far sources) and else the window index of their source; a byte then takes
// what its source holds, byte or index, until it is a byte (pointer doubling).
template <int NW, uint32_t SEG, bool SUM, bool QUADS>
__device__ __forceinline__ void resolve_window(uint8_t *dst, uint16_t *win, uint32_t w0, uint32_t wn, uint32_t wave,
                                               uint32_t lane, uint32_t &adler1, uint32_t &adler2) {
  static_assert(SEG % 512 == 0 && SEG <= 4096, "a segment is whole pairs of row groups, tracked in one 64-bit mask");
  static_assert(NW * SEG <= 32768, "distances inside the window stay below the literal flag");
  constexpr uint32_t R = 4, G = R * kWave;
  const uint32_t s0 = wave * SEG, s1 = min(s0 + SEG, wn);
  uint32_t carry = 0x8000u;
  uint64_t late = 0;  // groups with bytes whose source lies in another wave's segment
  const __amdgpu_buffer_rsrc_t rsrc = buffer_of(dst, 0x80000000u);
  auto at = [&](uint32_t g, uint32_t r) { return QUADS ? g + R * lane + r : g + r * kWave + lane; };
  auto read4 = [&](uint32_t g, uint32_t *v) __attribute__((always_inline)) {
    const uint2 m = *reinterpret_cast<const uint2 *>(win + g + R * lane);
    v[0] = m.x & 0xffff, v[1] = m.x >> 16, v[2] = m.y & 0xffff, v[3] = m.y >> 16;
  };
  auto write4 = [&](uint32_t g, const uint32_t *v) __attribute__((always_inline)) {
    *reinterpret_cast<uint2 *>(win + g + R * lane) =
        make_uint2(__builtin_amdgcn_perm(v[1], v[0], 0x05040100u), __builtin_amdgcn_perm(v[3], v[2], 0x05040100u));
  };
  // reads the marks of a group and loads its far sources
  auto open = [&](uint32_t row, uint32_t *c, uint32_t *f) __attribute__((always_inline)) {
    if constexpr (QUADS) {
      uint32_t m[R];
      read4(row, m);
      uint32_t last = m[0];
#pragma unroll
      for (uint32_t r = 1; r < R; r++) last = m[r] != 0xffffu ? m[r] : last;
      const uint32_t key = wave_max_dpp(last != 0xffffu ? ((lane + 1) << 16) | last : 0u);
      const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key, 0x138, 0xf, 0xf, false);  // wave_shr:1
      uint32_t t = up ? up & 0xffff : carry;
#pragma unroll
      for (uint32_t r = 0; r < R; r++) t = c[r] = m[r] != 0xffffu ? m[r] : t;
      carry = rdlane(t, kWave - 1);
    } else {
      uint32_t k[R];
#pragma unroll
      for (uint32_t r = 0; r < R; r++) {
        const uint32_t m = win[at(row, r)];
        k[r] = m == 0xffffu ? 0u : ((lane + 1) << 16) | m;
      }
#pragma unroll
      for (uint32_t r = 0; r < R; r++) {
        k[r] = wave_max_dpp(k[r]);
        c[r] = k[r] ? k[r] & 0xffff : carry;
        carry = rdlane(c[r], kWave - 1);
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < R; r++) {
      const uint32_t i = at(row, r);
      // a distance beyond the window; past the stored bytes it may be anything,
      // and an offset below 0 lies outside the buffer
      const bool isfar = c[r] >= i && c[r] < 0x8000u;
      f[r] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rsrc, isfar ? w0 + (i - 1 - c[r]) : ~0u, 0, 0);
    }
  };
  auto close = [&](uint32_t row, const uint32_t *c, const uint32_t *f) __attribute__((always_inline)) {
    uint32_t v[R];
#pragma unroll
    for (uint32_t r = 0; r < R; r++) {
      const uint32_t i = at(row, r);
      v[r] = c[r] < i ? i - 1 - c[r] : (c[r] >= 0x8000u ? c[r] : 0x8000u | f[r]);
      if constexpr (!QUADS) win[i] = (uint16_t)v[r];
    }
    if constexpr (QUADS) write4(row, v);
    // an index in another wave's segment waits for the second pass
    for (;;) {
      bool go[R], more = false;
#pragma unroll
      for (uint32_t r = 0; r < R; r++) {
        go[r] = NW == 1 ? v[r] < 0x8000u : v[r] - s0 < 0x8000u - s0;
        more |= go[r];
      }
      if (!__ballot(more)) break;
      lds_order();
      uint32_t t[R];
#pragma unroll
      for (uint32_t r = 0; r < R; r++) t[r] = win[v[r] & 0x7fff];
#pragma unroll
      for (uint32_t r = 0; r < R; r++) {
        v[r] = go[r] ? t[r] : v[r];
        if constexpr (!QUADS) win[at(row, r)] = (uint16_t)v[r];
      }
      if constexpr (QUADS) write4(row, v);
    }
    if constexpr (NW > 1) {
      uint32_t low = v[0];
#pragma unroll
      for (uint32_t r = 1; r < R; r++) low = min(low, v[r]);
      if (__ballot(low < 0x8000u)) late |= 1ull << ((row - s0) / G);
    }
  };
  // two sets of registers in turn: a copy from one to the other would wait for
  // the loads (rows from s1 to the next pair of groups are literals)
  uint32_t ca[R], fa[R], cb[R], fb[R];
  if (s0 < s1) open(s0, ca, fa);
  for (uint32_t row = s0; row < s1; row += 2 * G) {
    open(row + G, cb, fb);
    close(row, ca, fa);
    open(min(row + 2 * G, s0 + SEG - G), ca, fa);
    close(row + G, cb, fb);
  }
  if constexpr (NW > 1) {
    // every byte now is resolved or holds an index; the chains end at resolved
    // bytes, so no wave waits for another
    __syncthreads();
    while (late) {
      const uint32_t row = s0 + (uint32_t)__builtin_ctzll(late) * G;
      late &= late - 1;
      uint32_t v[R];
      if constexpr (QUADS) {
        read4(row, v);
      } else {
#pragma unroll
        for (uint32_t r = 0; r < R; r++) v[r] = win[at(row, r)];
      }
      for (;;) {
        uint32_t low = v[0];
#pragma unroll
        for (uint32_t r = 1; r < R; r++) low = min(low, v[r]);
        if (!__ballot(low < 0x8000u)) break;
        lds_order();
        uint32_t t[R];
#pragma unroll
        for (uint32_t r = 0; r < R; r++) t[r] = win[v[r] & 0x7fff];
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
          v[r] = v[r] < 0x8000u ? t[r] : v[r];
          if constexpr (!QUADS) win[at(row, r)] = (uint16_t)v[r];
        }
        if constexpr (QUADS) write4(row, v);
      }
    }
  }
  lds_order();
  // the segment to HBM, four bytes a lane
  uint32_t a1 = 0, a2 = 0;
  (void)a1, (void)a2;
  const uint32_t len = s1 > s0 ? s1 - s0 : 0u;
  for (uint32_t k = 4 * lane; k < len; k += 4 * kWave) {
    const uint2 w = *reinterpret_cast<const uint2 *>(win + s0 + k);
    uint32_t b = __builtin_amdgcn_perm(w.y, w.x, 0x06040200u);
    uint8_t *d = dst + (w0 + s0 + k);
    if (k + 4 <= len) {
      __builtin_memcpy(d, &b, 4);
    } else {
      b &= (1u << 8 * (len - k)) - 1;
      for (uint32_t j = 0; j < len - k; j++) d[j] = (uint8_t)(b >> 8 * j);
    }
    if constexpr (SUM) {
      const uint32_t sum = __builtin_amdgcn_udot4(b, 0x01010101u, 0u, false);
      a1 += sum;
      a2 += k * sum + __builtin_amdgcn_udot4(b, 0x03020100u, 0u, false);
    }
  }
  if constexpr (SUM) {
    // a1 = sum b <= 16320 (SEG 4096), a2 = sum of (position - w0 - s0) * b < 2^27
    adler1 = (adler1 + a1) % 65521u;
    adler2 = (adler2 + ((w0 + s0) % 65521u) * a1 + a2) % 65521u;
  }
}

}  // namespace dev
}  // namespace codag
