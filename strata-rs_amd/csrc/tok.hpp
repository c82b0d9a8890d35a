// Weight rows against many token vectors on f16 MFMA with f32-class
// precision (tok_mm.hip): the operand formats.
//
// Activations. Per 256-element super-block of a token a power of two 2^k
// brings its largest |x| into [2^14, 2^15), and every y = x * 2^k is held as
// hi + 2^-11 lo, hi = f16(y) and lo = f16(2^11 (y - hi)): y to within 2^-23 of
// itself (a remainder has 12 bits and a sign, an f16 11: the last of the 24 is
// lost in one element of four), whatever its size beside its neighbours down
// to 2^-27 of the maximum, and below to within 2^-50 of that (lo's own scale
// keeps it off f16's subnormals, where hi + lo would fall short from 2^-17 of
// the maximum on). Both enter v_mfma_f32_*_f16, whose products are exact and
// whose sums are f32; lo's factor 2^-11 is in the weights it meets (or, where
// hi and lo are rows of one fragment, joins with the sums).
// Weights. Codes become exact f16 integers: Q4_K / Q5_K codes times their
// 6-bit sub-block scale (<= 63 * 31, 11 bits), the others the codes alone,
// their sub-block scale applied to each sub-block's f32 sums. The block's d
// (and the K-quants' min term, sum_j m_j * sum_j x on one more MFMA) joins
// once per super-block.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace sh {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// 16 / 8 bytes from a 2-byte aligned address (34- and 210-byte blocks start
// at even addresses): one global load on gfx950.
typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2a2 __attribute__((ext_vector_type(2), aligned(2)));
__device__ __forceinline__ u32x4 ld16h(const uint8_t* p) {
  const u32x4a2 v = *reinterpret_cast<const u32x4a2*>(p);
  return u32x4{v.x, v.y, v.z, v.w};
}
// The same through whole dwords, sh = p & 2 known when it is used: the load
// unit takes a 16-byte load off the dword grid in twice as many accesses
// (Q6_K down of 96 tokens x 8 of 128 experts: 65 -> 36 M accesses, 102 -> 88
// us). The last dword is read again where sh is 0, so no byte outside a dword
// that p[0, 16) touches is.
struct Win16 {
  u32x4 v;
  uint32_t e;
};
__device__ __forceinline__ Win16 ld16w(const uint8_t* p, uint32_t sh) {
  typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
  const uint8_t* a = p - sh;
  const u32x4a4 v = *reinterpret_cast<const u32x4a4*>(a);
  return {u32x4{v.x, v.y, v.z, v.w}, *reinterpret_cast<const uint32_t*>(a + 12 + 2 * sh)};
}
__device__ __forceinline__ u32x4 win16(const Win16& r, uint32_t sh) {
  return u32x4{__builtin_amdgcn_alignbyte(r.v.y, r.v.x, sh), __builtin_amdgcn_alignbyte(r.v.z, r.v.y, sh),
               __builtin_amdgcn_alignbyte(r.v.w, r.v.z, sh), __builtin_amdgcn_alignbyte(r.e, r.v.w, sh)};
}
__device__ __forceinline__ u32x2 ld8h(const uint8_t* p) {
  const u32x2a2 v = *reinterpret_cast<const u32x2a2*>(p);
  return u32x2{v.x, v.y};
}

__device__ __forceinline__ f16x2_t as_h2(uint32_t v) { return __builtin_bit_cast(f16x2_t, v); }
__device__ __forceinline__ f16x2_t h2_dup(float v) {
  const _Float16 h = static_cast<_Float16>(v);
  return f16x2_t{h, h};
}

// A B fragment (the lane's 8 weights of one k step): word pairs hold bytes
// (0, 2) and (1, 3) of a code word, so slot order within 4 columns is
// 0, 2, 1, 3 (tok_slot); the activations are stored in the same order.
constexpr float kTokLo = 0x1p-11f;  // of a lo limb
union TokFrag {
  f16x2_t h[4];
  f16x8_t v;
};

// Four codes < 64 (one a byte) times sc plus c = -1024 sc: 1024 + q is the
// f16 with bits 0x6400 | q, and the fused product is exact.
__device__ __forceinline__ void tok_scaled4(uint32_t w, f16x2_t sc, f16x2_t c, f16x2_t& a, f16x2_t& b) {
  a = __builtin_elementwise_fma(as_h2((w & 0x003F003Fu) | 0x64006400u), sc, c);
  b = __builtin_elementwise_fma(as_h2(((w >> 8) & 0x003F003Fu) | 0x64006400u), sc, c);
}
// Four signed bytes as f16.
__device__ __forceinline__ void tok_signed4(uint32_t w, f16x2_t& a, f16x2_t& b) {
  const uint32_t u = w ^ 0x80808080u;
  const f16x2_t bias = as_h2(0xE480E480u);  // -(1024 + 128)
  a = as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04020400u)) + bias;
  b = as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)) + bias;
}

// A format: a row's super-block (256 columns) is taken in four groups g of
// 64 columns (32-column sub-blocks 2g and 2g + 1), each four MFMA k steps
// (sub-block jj, step i). load<g> issues group g's loads into Raw; take<g>
// moves what they brought into Sb (the next super-block's loads then go into
// Raw); frags<g, jj> forms the two B fragments of sub-block jj, and sub<g> is
// the scale of a k step (kSub 1) or sub-block (kSub 2) of the group. kSub 0:
// the scales are in the weights. `left`: Q8_0 blocks from the super-block's
// first to the row's last.
// take_lds<g>: take<g> from the row's bytes in LDS (kPieces 16-byte pieces
// from the dword at or below the super-block, `sh` bytes below it).
// kPerm 0: step i of lane half h is columns 16 h + 8 i + [0, 8) of the
// sub-block; 1: columns 16 i + 8 h + [0, 8).
template <int Q>
struct TokQ4Q5 {  // Q4_K, Q5_K
  static constexpr int kSub = 0, kPerm = 0, kSbBytes = Q == kQ5_K ? 176 : 144;
  static constexpr bool kMin = true;
  struct Raw {
    u32x4 h, qh, q[4];
  };
  struct Sb {
    u32x4 h, qh, q;
    uint32_t sc03, sc47;
  };
  template <int G>
  __device__ static __forceinline__ void load(const uint8_t* sb, int half, Raw& r, int) {
    if constexpr (G == 0) {
      r.h = ld16h(sb);
      if constexpr (Q == kQ5_K) r.qh = ld16h(sb + 16 + 16 * half);
    }
    r.q[G] = ld16h(sb + (Q == kQ5_K ? 48 : 16) + 32 * G + 16 * half);
  }
  template <int G>
  __device__ static __forceinline__ void take(const Raw& r, Sb& s) {
    s.q = r.q[G];
    if constexpr (G == 0) {
      s.h = r.h;
      if constexpr (Q == kQ5_K) s.qh = r.qh;
      s.sc03 = s.h.y & 0x3F3F3F3Fu;
      s.sc47 = (s.h.w & 0x0F0F0F0Fu) | ((s.h.y >> 2) & 0x30303030u);
    }
  }
  static constexpr int kPieces = kSbBytes / 16;
  template <int G>
  __device__ static __forceinline__ void take_lds(const uint8_t* row, uint32_t, uint32_t, int half, Sb& s) {
    s.q = *reinterpret_cast<const u32x4*>(row + (Q == kQ5_K ? 48 : 16) + 32 * G + 16 * half);
    if constexpr (G == 0) {
      s.h = *reinterpret_cast<const u32x4*>(row);
      if constexpr (Q == kQ5_K) s.qh = *reinterpret_cast<const u32x4*>(row + 16 + 16 * half);
      s.sc03 = s.h.y & 0x3F3F3F3Fu;
      s.sc47 = (s.h.w & 0x0F0F0F0Fu) | ((s.h.y >> 2) & 0x30303030u);
    }
  }
  __device__ static __forceinline__ float d(const Sb& s) { return h2f(s.h.x); }
  __device__ static __forceinline__ float dmin(const Sb& s) { return h2f(s.h.x >> 16); }
  // m_j of the eight sub-blocks (either lane half)
  __device__ static __forceinline__ f16x8_t mins(const Sb& s) {
    const uint32_t m03 = s.h.z & 0x3F3F3F3Fu;
    const uint32_t m47 = ((s.h.w >> 4) & 0x0F0F0F0Fu) | ((s.h.z >> 2) & 0x30303030u);
    f16x8_t v;
    v[0] = static_cast<_Float16>(ubyte<0>(m03));
    v[1] = static_cast<_Float16>(ubyte<1>(m03));
    v[2] = static_cast<_Float16>(ubyte<2>(m03));
    v[3] = static_cast<_Float16>(ubyte<3>(m03));
    v[4] = static_cast<_Float16>(ubyte<0>(m47));
    v[5] = static_cast<_Float16>(ubyte<1>(m47));
    v[6] = static_cast<_Float16>(ubyte<2>(m47));
    v[7] = static_cast<_Float16>(ubyte<3>(m47));
    return v;
  }
  template <int G, int JJ>
  __device__ static __forceinline__ void frags(const Sb& s, TokFrag (&f)[2]) {
    const f16x2_t sc = h2_dup(ubyte<2 * (G & 1) + JJ>(G < 2 ? s.sc03 : s.sc47));
    // Q4_K's high nibbles stay in place: 64 + q is the f16 with bits
    // 0x5400 | q << 4
    constexpr bool kHigh = Q != kQ5_K && JJ == 1;
    const f16x2_t c = sc * h2_dup(kHigh ? -64.f : -1024.f);
    const uint32_t q[4] = {s.q.x, s.q.y, s.q.z, s.q.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f16x2_t* o = f[k >> 1].h + 2 * (k & 1);
      if constexpr (Q == kQ5_K) {
        const uint32_t qh[4] = {s.qh.x, s.qh.y, s.qh.z, s.qh.w};
        uint32_t code[2];
        q5k_codes(q[k], qh[k], G, code[0], code[1]);
        tok_scaled4(code[JJ], sc, c, o[0], o[1]);
      } else {
        constexpr uint32_t kMask = kHigh ? 0x00F000F0u : 0x000F000Fu, kBits = kHigh ? 0x54005400u : 0x64006400u;
        o[0] = __builtin_elementwise_fma(as_h2((q[k] & kMask) | kBits), sc, c);
        o[1] = __builtin_elementwise_fma(as_h2(((q[k] >> 8) & kMask) | kBits), sc, c);
      }
    }
  }
  template <int G>
  __device__ static __forceinline__ float sub(const Sb&, int, int, int) {
    return 1.f;
  }
};

// Q6_K: 16-element sub-blocks are the k steps. A lane half reads whole
// 16-byte runs (the sub-block of its own half of l) and the halves exchange
// 8 of them (permlane32_swap), so each k step has columns l of one sub-block.
struct TokQ6 {
  static constexpr int kSub = 1, kPerm = 1, kSbBytes = 210;
  static constexpr bool kMin = false;
  struct Raw {
    Win16 sc, qh[2], ql[4];  // by half of the super-block
    uint32_t d, sh;
  };
  struct Sb {
    u32x4 sc;
    uint32_t d;
    u32x4 qh, ql[2];
  };
  template <int G>
  __device__ static __forceinline__ void load(const uint8_t* sb, int half, Raw& r, int) {
    if constexpr (G == 0) {
      r.sh = uint32_t(reinterpret_cast<uintptr_t>(sb)) & 2u;
      r.sc = ld16w(sb + 192, r.sh);
      r.d = *reinterpret_cast<const uint16_t*>(sb + 208);
    }
    if constexpr ((G & 1) == 0) {
      constexpr int H = G >> 1;
      r.qh[H] = ld16w(sb + 128 + 32 * H + 16 * half, r.sh);
      r.ql[2 * H] = ld16w(sb + 64 * H + 16 * half, r.sh);
      r.ql[2 * H + 1] = ld16w(sb + 64 * H + 32 + 16 * half, r.sh);
    }
  }
  // words (0, 1 | 2, 3) of each half's run -> the lane's 8 bytes of the
  // first half's run (.x .y) and of the second's (.z .w)
  __device__ static __forceinline__ u32x4 halves(u32x4 w) {
    const auto a = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
    return u32x4{a[0], b[0], a[1], b[1]};
  }
  static constexpr int kPieces = 13;  // 208 bytes; the last dword is the row's `tail`
  __device__ static __forceinline__ u32x4 lds16(const uint8_t* p, uint32_t sh) {
    return win16({*reinterpret_cast<const u32x4*>(p), *reinterpret_cast<const uint32_t*>(p + 16)}, sh);
  }
  template <int G>
  __device__ static __forceinline__ void take_lds(const uint8_t* row, uint32_t sh, uint32_t tail, int half, Sb& s) {
    if constexpr (G == 0) {
      s.sc = win16({*reinterpret_cast<const u32x4*>(row + 192), tail}, sh);
      s.d = (tail >> (8 * sh)) & 0xFFFFu;
    }
    if constexpr ((G & 1) == 0) {
      constexpr int H = G >> 1;
      s.qh = halves(lds16(row + 128 + 32 * H + 16 * half, sh));
      s.ql[0] = halves(lds16(row + 64 * H + 16 * half, sh));
      s.ql[1] = halves(lds16(row + 64 * H + 32 + 16 * half, sh));
    }
  }
  __device__ static __forceinline__ float d(const Sb& s) { return h2f(s.d); }
  template <int G>
  __device__ static __forceinline__ void take(const Raw& r, Sb& s) {
    if constexpr (G == 0) {
      s.sc = win16(r.sc, r.sh);
      s.d = r.d;
    }
    if constexpr ((G & 1) == 0) {
      s.qh = halves(win16(r.qh[G >> 1], r.sh));
      s.ql[0] = halves(win16(r.ql[G], r.sh));
      s.ql[1] = halves(win16(r.ql[G + 1], r.sh));
    }
  }
  template <int G, int JJ>
  __device__ static __forceinline__ void frags(const Sb& s, TokFrag (&f)[2]) {
    const f16x2_t bias = as_h2(0xE420E420u);  // -(1024 + 32)
    // 32-column group I = 2 (G & 1) + JJ of the half: ql run JJ, nibble G & 1,
    // bit pair I of qh
    constexpr int I = 2 * (G & 1) + JJ;
    const uint32_t q[4] = {s.ql[JJ].x, s.ql[JJ].y, s.ql[JJ].z, s.ql[JJ].w};
    const uint32_t qh[4] = {s.qh.x, s.qh.y, s.qh.z, s.qh.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t lo = (G & 1) ? (q[k] >> 4) & 0x0F0F0F0Fu : q[k] & 0x0F0F0F0Fu;
      uint32_t t;
      if constexpr (I < 2)
        t = qh[k] << (4 - 2 * I);
      else
        t = qh[k] >> (2 * I - 4);
      const uint32_t w = lo | (t & 0x30303030u);
      f16x2_t* o = f[k >> 1].h + 2 * (k & 1);
      o[0] = as_h2((w & 0x003F003Fu) | 0x64006400u) + bias;
      o[1] = as_h2(((w >> 8) & 0x003F003Fu) | 0x64006400u) + bias;
    }
  }
  template <int G>
  __device__ static __forceinline__ float sub(const Sb& s, int k, int q6_signed, int) {
    const uint32_t w = (G == 0 ? s.sc.x : G == 1 ? s.sc.y : G == 2 ? s.sc.z : s.sc.w) >> (8 * k);
    return q6_signed ? float(int8_t(w & 0xFFu)) : ubyte<0>(w);
  }
};

// Q8_0: eight 34-byte blocks stand for a super-block; a row's last one may
// hold fewer (`left` blocks from this super-block on): blocks past the row
// read its last one and get scale 0.
struct TokQ8 {
  static constexpr int kSub = 2, kPerm = 0, kSbBytes = 272;
  static constexpr bool kMin = false;
  struct Raw {
    u32x4 q[8];
    uint32_t d[8];
  };
  struct Sb {
    u32x4 q[2];
    uint32_t d[2];
  };
  template <int G>
  __device__ static __forceinline__ void load(const uint8_t* sb, int half, Raw& r, int left) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      const uint8_t* b = sb + 34 * min(2 * G + jj, left - 1);
      r.q[2 * G + jj] = ld16h(b + 2 + 16 * half);
      r.d[2 * G + jj] = *reinterpret_cast<const uint16_t*>(b);
    }
  }
  template <int G>
  __device__ static __forceinline__ void take(const Raw& r, Sb& s) {
    s.q[0] = r.q[2 * G];
    s.q[1] = r.q[2 * G + 1];
    s.d[0] = r.d[2 * G];
    s.d[1] = r.d[2 * G + 1];
  }
  static constexpr int kPieces = 17;  // rows of whole super-blocks
  template <int G>
  __device__ static __forceinline__ void take_lds(const uint8_t* row, uint32_t, uint32_t, int half, Sb& s) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      constexpr int J = 2 * G;
      const uint32_t* p = reinterpret_cast<const uint32_t*>(row + ((34 * (J + jj) + 2) & ~3) + 16 * half);
      const uint32_t sh = (34 * (J + jj) + 2) & 2;
      s.q[jj] = win16({u32x4{p[0], p[1], p[2], p[3]}, sh ? p[4] : 0u}, sh);
      s.d[jj] = *reinterpret_cast<const uint16_t*>(row + 34 * (J + jj));
    }
  }
  __device__ static __forceinline__ float d(const Sb&) { return 1.f; }
  template <int G, int JJ>
  __device__ static __forceinline__ void frags(const Sb& s, TokFrag (&f)[2]) {
    const u32x4 q = s.q[JJ];
    tok_signed4(q.x, f[0].h[0], f[0].h[1]);
    tok_signed4(q.y, f[0].h[2], f[0].h[3]);
    tok_signed4(q.z, f[1].h[0], f[1].h[1]);
    tok_signed4(q.w, f[1].h[2], f[1].h[3]);
  }
  template <int G>
  __device__ static __forceinline__ float sub(const Sb& s, int jj, int, int left) {
    return 2 * G + jj < left ? h2f(s.d[jj]) : 0.f;
  }
};

// IQ4_XS in either reading of the code bytes (GGML: sub-block ib reads
// qs[16 ib ..); else every sub-block reads qs[0..16)).
template <bool GGML>
struct TokIQ4 {
  static constexpr int kSub = 2, kPerm = 1, kSbBytes = 136;
  static constexpr bool kMin = false;
  struct Raw {
    u32x2 h, q[8];
  };
  struct Sb {
    u32x2 h, q[2];
  };
  template <int G>
  __device__ static __forceinline__ void load(const uint8_t* sb, int half, Raw& r, int) {
    if constexpr (G == 0) r.h = ld8h(sb);
    if constexpr (GGML) {
      r.q[2 * G] = ld8h(sb + 8 + 32 * G + 8 * half);
      r.q[2 * G + 1] = ld8h(sb + 24 + 32 * G + 8 * half);
    } else if constexpr (G == 0) {
      r.q[0] = ld8h(sb + 8 + 8 * half);
    }
  }
  template <int G>
  __device__ static __forceinline__ void take(const Raw& r, Sb& s) {
    if constexpr (G == 0) s.h = r.h;
    if constexpr (GGML || G == 0) {
      s.q[0] = r.q[2 * G];
      s.q[1] = r.q[GGML ? 2 * G + 1 : 0];
    }
  }
  __device__ static __forceinline__ float d(const Sb& s) { return h2f(s.h.x); }
  template <int G, int JJ>
  __device__ static __forceinline__ void frags(const Sb& s, TokFrag (&f)[2]) {
    const u32x2 q = s.q[JJ];
    tok_signed4(iq4_lut(q.x & 0x0F0F0F0Fu), f[0].h[0], f[0].h[1]);
    tok_signed4(iq4_lut(q.y & 0x0F0F0F0Fu), f[0].h[2], f[0].h[3]);
    tok_signed4(iq4_lut((q.x >> 4) & 0x0F0F0F0Fu), f[1].h[0], f[1].h[1]);
    tok_signed4(iq4_lut((q.y >> 4) & 0x0F0F0F0Fu), f[1].h[2], f[1].h[3]);
  }
  template <int G>
  __device__ static __forceinline__ float sub(const Sb& s, int jj, int, int) {
    return iq4xs_scale(s.h.x, s.h.y, 2 * G + jj);
  }
};

}  // namespace sh
