// Weight rows against many token vectors: y[t][r] = sum_c W[r][c] x[t][c]
// as `tokens` calls of ops::gemv (crates/strata-core/src/ops.rs:14-28), for
// 9 tokens to thousands and for an expert's, at the matvecs' precision
// (tok.hpp's operands).
//
// The launches: tok_prep_kernel converts the tokens once per call into the
// MFMA's A fragments (a super-block of a token group is one contiguous run,
// the order the matmul's LDS ring takes them in), tok_mm_kernel multiplies,
// and rows whose columns were split over workgroups are added by the launch
// that reads them (a fixed order, so results do not depend on timing).
//
// tok_mm_kernel: workgroup = 4 waves x 32 weight rows against one token
// group, over its share of the super-blocks. A wave forms the B fragments of
// its own 32 rows from registers, each packed byte loaded and decoded once
// per token group, a super-block ahead; the group's A fragments come
// through a ring of three LDS buffers (global_load_lds, two stages ahead)
// that the four waves share. A group is
//   32, 64 or 96 tokens: hi and lo limbs are fragments of their own, lo's
//     against 2^-11 of the weights into hi's f32 sums or, where registers
//     allow, into sums of their own (a stage is 64 columns);
//   8 or 16 tokens: the hi limbs are A rows [0, T) and the lo limbs rows
//     [T, 2 T) of one fragment, so no matrix work is done for padding at 16,
//     and their sums are added at the end (a stage is a whole super-block).
// Bound: weights are read and decoded once per group, so few tokens are
// bound by the weight stream and many by MFMA (two f16 products per weight
// and token). Per launch in a kernel trace: gate and up of 4096 x 12288 Q4_K
// (two matrices) 25 us at 24 tokens, 58 us at 77 (MFMA 29% busy, VALU 25), 285
// us at 512 (363 TFLOP/s of x, twice that of f16); down of 12288 x 4096 Q6_K
// 25, 47 and 252 us (its 16-column sub-blocks cost 16 scalings per MFMA pair).
// v_mfma_f32_32x32x16_f16: A row / B column = lane % 32, k = 8 (lane / 32) +
// [0, 8); D column (weight row) = lane % 32, D row (token) = 8 (i / 4) + 4
// (lane / 32) + i % 4.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "tok.hpp"

namespace sh {

constexpr int kTokRows = 128;  // weight rows per workgroup
constexpr int kTokThreads = 256;

// The image of a token group's super-block: 16 k steps (pieces per step:
// tiles x limbs), the sub-block sums of x (one fragment a tile), and the
// 2^-k of its tokens; whole KiB.
template <int TOK>
struct TokShape {
  static constexpr bool kPacked = TOK <= 16;  // hi and lo limbs in one fragment
  static constexpr int kTiles = kPacked ? 1 : TOK / 32;
  static constexpr int kLimbs = kPacked ? 1 : 2;
  static constexpr int kPiece = TOK == 8 ? 512 : 1024;
  static constexpr int kGroup = 4 * kTiles * kLimbs * kPiece;  // 64 columns
  static constexpr int kSums = kTiles * kPiece;
  static constexpr int kSb = 4 * kGroup + kSums + (TOK == 8 ? 512 : 1024);
};
constexpr int tok_sb_bytes(int tok) {
  return tok == 8 ? TokShape<8>::kSb : tok == 16 ? TokShape<16>::kSb : tok == 32 ? TokShape<32>::kSb
       : tok == 64 ? TokShape<64>::kSb : TokShape<96>::kSb;
}

// Byte of piece (row m of the fragment, lane half h): a fragment of 32 rows
// (16 at 8 tokens, whose rows 16 to 31 repeat them and are not used).
__device__ __forceinline__ int tok_row_byte(int tok, int m, int h) { return ((tok == 8 ? 16 : 32) * h + m) * 16; }

// ------------------------------------------------------------------- prep --
// A wave per (token, super-block): lane l holds columns 4 l .. 4 l + 3.
// SILU: the values are silu(g) * u of the partial sums g = sum_s part[s][t]
// [c], u = sum_s part[s][t][cols + c] (ops.rs:85-87, in order of s), else
// x[t][c]. Columns past the row are zero.
struct TokPrep {
  const float* x;
  int64_t ld;    // floats between tokens of x (or of a partial sum)
  int64_t part;  // floats between partial sums
  int nsplit;
  int cols, nsb, tokens, tok, perm;
  uint8_t* img;
  const int* src;   // value t is row src[t] of x, and goes to
  const int* slot;  // place slot[t] of the groups (null: t)
};

template <bool SILU>
__global__ void __launch_bounds__(256) tok_prep_kernel(TokPrep a) {
  const int lane = threadIdx.x & 63;
  const int sb = blockIdx.x * 4 + (threadIdx.x >> 6), t = blockIdx.y;
  if (sb >= a.nsb) return;
  const int c0 = 256 * sb + 4 * lane;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (c0 < a.cols) {  // whole 4-column pieces: cols is a multiple of 32
    typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // x of any float alignment
    const float* p = a.x + int64_t(a.src ? a.src[t] : t) * a.ld + c0;
    v = *reinterpret_cast<const f32x4a4*>(p);
    if constexpr (SILU) {
      f32x4 u = *reinterpret_cast<const f32x4a4*>(p + a.cols);
      for (int s = 1; s < a.nsplit; ++s) {
        v += *reinterpret_cast<const f32x4a4*>(p + s * a.part);
        u += *reinterpret_cast<const f32x4a4*>(p + s * a.part + a.cols);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = v[k] / (1.f + expf(-v[k])) * u[k];
    }
  }
  float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
  float s = (v.x + v.y) + (v.z + v.w);
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) {
    m = fmaxf(m, __shfl_xor(m, off, kWave));
    s += __shfl_xor(s, off, kWave);
  }
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, kWave));
  // 2^k with max |x| 2^k in [2^14, 2^15); a maximum that is not finite makes
  // every sum of the token NaN (a NaN element does so by itself)
  int e = 0;
  (void)frexpf(m, &e);
  const int k = m > 0.f ? min(15 - e, 126) : 0;
  const float up = ldexpf(1.f, k);
  const float down = (m - m == 0.f) ? ldexpf(1.f, -k) : __builtin_nanf("");

  const int tok = a.tok;
  const int sl = a.slot ? a.slot[t] : t;
  const int group = sl / tok, tg = sl - group * tok;  // this token in its group
  const bool packed = tok <= 16;
  const int tile = packed ? 0 : tg >> 5, row = packed ? tg : tg & 31;
  const int tiles = packed ? 1 : tok / 32, limbs = packed ? 1 : 2;
  const int piece = tok == 8 ? 512 : 1024;
  const int gbytes = 4 * tiles * limbs * piece;
  uint8_t* base = a.img + (int64_t(group) * a.nsb + sb) * tok_sb_bytes(tok);

  f16x2_t h01, h23, l01, l23;  // columns (0, 2) and (1, 3): tok.hpp's slot order
  const float y0 = v.x * up, y1 = v.y * up, y2 = v.z * up, y3 = v.w * up;
  h01[0] = static_cast<_Float16>(y0);
  h01[1] = static_cast<_Float16>(y2);
  h23[0] = static_cast<_Float16>(y1);
  h23[1] = static_cast<_Float16>(y3);
  auto low = [](float y, _Float16 h) { return static_cast<_Float16>((y - static_cast<float>(h)) * (1.f / kTokLo)); };
  l01[0] = low(y0, h01[0]);
  l01[1] = low(y2, h01[1]);
  l23[0] = low(y1, h23[0]);
  l23[1] = low(y3, h23[1]);

  const int j = lane >> 3, c = (4 * lane) & 31;  // sub-block, column in it
  const int i = a.perm ? c >> 4 : (c >> 3) & 1, half = a.perm ? (c >> 3) & 1 : c >> 4;
  const int step = 2 * (j & 1) + i;
  uint8_t* p = base + (j >> 1) * gbytes + (tile * 4 + step) * limbs * piece + 2 * (c & 7);
  const u32x2 hi = {__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23)};
  const u32x2 lo = {__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23)};
  *reinterpret_cast<u32x2*>(p + tok_row_byte(tok, row, half)) = hi;
  if (packed)
    *reinterpret_cast<u32x2*>(p + tok_row_byte(tok, row + tok, half)) = lo;
  else
    *reinterpret_cast<u32x2*>(p + piece + tok_row_byte(tok, row, half)) = lo;

  // sub-block sums of x as hi and lo of sum * 2^(k - 5), against the mins in
  // both lane halves (lo's times 2^-11): apart in the k slots, or (packed) in
  // the A rows
  uint8_t* sums = base + 4 * gbytes + tile * piece;
  if ((lane & 7) == 0) {
    const float y = ldexpf(s, k - 5);
    const _Float16 sh = static_cast<_Float16>(y), sl = low(y, sh);
    *reinterpret_cast<_Float16*>(sums + tok_row_byte(tok, row, 0) + 2 * j) = sh;
    if (packed) {
      *reinterpret_cast<_Float16*>(sums + tok_row_byte(tok, row + tok, 0) + 2 * j) = sl;
      *reinterpret_cast<_Float16*>(sums + tok_row_byte(tok, row, 1) + 2 * j) = _Float16(0);
      *reinterpret_cast<_Float16*>(sums + tok_row_byte(tok, row + tok, 1) + 2 * j) = _Float16(0);
    } else {
      *reinterpret_cast<_Float16*>(sums + tok_row_byte(tok, row, 1) + 2 * j) = sl;
    }
  }
  if (lane == 0) reinterpret_cast<float*>(base + 4 * gbytes + tiles * piece)[tg] = down;
}

// ----------------------------------------------------------------- matmul --
struct TokMm {
  const uint8_t *w0, *w1;  // two matrices of the same shape (w1 null: one)
  int rows, tiles;         // rows of each, 128-row tiles of both
  int64_t rb;              // bytes per row
  int nsb, sb_per, nsplit; // super-blocks of a row, of a workgroup's share, shares
  int nblk;                // 32-column blocks of a row
  const uint8_t* img;
  float* out;              // [nsplit][tokens][ld]; w1's rows follow w0's
  int64_t ld, part;        // floats between tokens, between shares
  int tokens, groups, q6s;
  TokItems items;
};

struct TokNone {};
template <class F>
constexpr bool tok_lds_format() {
  return !std::is_same<F, TokIQ4<true>>::value && !std::is_same<F, TokIQ4<false>>::value;
}
// A wave's 32 rows of a super-block on their way through its LDS: load()
// requests them in whole 16-byte pieces, row after row (adjacent lanes read
// adjacent bytes), store() writes the pieces that came to the wave's slot, in
// the order they were read, and the lanes take their rows from there. Loads
// straight to the lanes (32 rows x 32 bytes each) cost an access or two per
// lane: Q6_K down of 96 tokens x 8 of 128 experts took 36 M accesses for 165
// MB, and the load unit bound it; this way it takes 11. Routed FFN, 128 x 2048 x 768 Q4_K / Q6_K: 16
// tokens 111 -> 98 us, 64 189 -> 155 to 170, 96 204 -> 169 to 186, 256 231 ->
// 214; dense FFN
// 2048 / 6144 Q5_K / Q8_0, 12 tokens 43 -> 34.
template <class F, bool CO>
struct TokWave {
  static constexpr int kN = (32 * F::kPieces + 63) / 64, kLds = kN * 1024;
  static constexpr bool kTail = F::kSbBytes % 16 != 0;  // a dword past the pieces, rows off the dword grid
  uint8_t* slot;
  const uint8_t* base;  // a dword boundary at or below the wave's first row's share
  uint32_t off[kN];     // of the lane's pieces (their rows') from it
  uint32_t toff;        // of the lane's row
  u32x4 v[kN];
  uint32_t t;
  uint32_t sh, tail;  // of the super-block in the slot: the lane's row
  __device__ __forceinline__ TokWave(const uint8_t* w, int row0, int rows, int64_t rb, int sb0, uint8_t* l, int wave,
                                     int lane) {
    slot = l + wave * kLds;
    const uint8_t* p = w + int64_t(min(row0, rows - 1)) * rb + int64_t(sb0) * F::kSbBytes;
    const uint32_t b = uint32_t(reinterpret_cast<uintptr_t>(p)) & 3u;
    base = p - b;
    const int most = max(rows - 1 - row0, 0);  // rows past the matrix: its last
#pragma unroll
    for (int k = 0; k < kN; ++k) {
      const int q = min(lane + 64 * k, 32 * F::kPieces - 1), r = q / F::kPieces;
      off[k] = b + uint32_t(min(r, most)) * uint32_t(rb) + (kTail ? 0 : 16 * (q - r * F::kPieces));
    }
    toff = b + uint32_t(min(lane & 31, most)) * uint32_t(rb);
  }
  __device__ __forceinline__ void load(int s) {
    const uint8_t* p = base + int64_t(s) * (kTail ? 0 : F::kSbBytes);
    const uint32_t add = kTail ? uint32_t(s) * F::kSbBytes : 0;
#pragma unroll
    for (int k = 0; k < kN; ++k) {
      typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
      uint32_t o = off[k];
      if constexpr (kTail) {  // the dword at or below the row's super-block, then the piece
        const int q = min(int(threadIdx.x & 63) + 64 * k, 32 * F::kPieces - 1);
        o = ((o + add) & ~3u) + 16 * (q % F::kPieces);
      }
      const u32x4a4 x = *reinterpret_cast<const u32x4a4*>(p + o);
      v[k] = u32x4{x.x, x.y, x.z, x.w};
    }
    if constexpr (kTail) t = *reinterpret_cast<const uint32_t*>(p + ((toff + add) & ~3u) + 16 * F::kPieces);
  }
  __device__ __forceinline__ void store(int s) {
    const int lane = threadIdx.x & 63;
    // (a wave's LDS operations run in order: its reads below see every
    // lane's pieces, its next writes come after them)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < kN; ++k) *reinterpret_cast<u32x4*>(slot + 1024 * k + 16 * lane) = v[k];
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    sh = kTail ? (toff + uint32_t(s) * F::kSbBytes) & 3u : 0;
    tail = t;
  }
  __device__ __forceinline__ const uint8_t* row(int r32) const { return slot + r32 * (16 * F::kPieces); }
};
template <class F>
struct TokWave<F, false> {
  uint32_t sh, tail;
  __device__ __forceinline__ TokWave(const uint8_t*, int, int, int64_t, int, uint8_t*, int, int) {}
  __device__ __forceinline__ void load(int) {}
  __device__ __forceinline__ void store(int) {}
  __device__ __forceinline__ const uint8_t* row(int) const { return nullptr; }
};

// CO: the wave's weights by way of its own LDS (TokWave) instead of one
// 16-byte load a lane from 32 rows at a time.
template <class F, int TOK, bool CO>
__global__ void __launch_bounds__(kTokThreads, 2) tok_mm_kernel(TokMm a) {
  using S = TokShape<TOK>;
  constexpr int NT = S::kTiles;
  constexpr int kAcc = TOK == 8 ? 8 : 16;  // D values of a tile that are used
  // lo limbs into sums of their own, up to 64 tokens where a super-block's
  // sums stay in the MFMA's accumulators: fewer instructions than 2^-11 of
  // every weight (4096 / 12288 Q4_K, 24 tokens: 58.0 us, else 59.4; lo on hi's
  // own scale, short of bits beside large neighbours, 57.2)
  constexpr bool kOwnLo = F::kSub == 0 && !S::kPacked && NT <= 2;
  constexpr int kSums = kOwnLo ? 2 * NT : NT;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int r32 = lane & 31, half = lane >> 5;

  // workgroup -> (share, 8 row tiles, token group, row tile): the groups of
  // a row tile run on one XCD (workgroup i on XCD i % 8), near in time, and
  // share the weights in its L2
  int id = blockIdx.x;
  const int t8 = id & 7;
  id >>= 3;
  int group, share, tile, p0, cnt;
  int64_t we = 0;
  if (a.items.e) {
    // groups are an expert's tokens: the row tiles of a group run on one
    // XCD, near in time, and share its fragments in the L2
    group = id / a.tiles * 8 + t8;
    tile = id - group / 8 * a.tiles;
    share = 0;
    if (group >= *a.items.n) return;
    we = a.items.e[group] * a.items.stride;
    p0 = a.items.off[group];
    cnt = a.items.cnt[group];
  } else {
    group = id % a.groups;
    id /= a.groups;
    const int nt8 = (a.tiles + 7) >> 3;
    share = id / nt8;
    tile = (id - share * nt8) * 8 + t8;
    if (tile >= a.tiles) return;
    p0 = group * TOK;
    cnt = min(TOK, a.tokens - p0);
  }
  const int per_mat = a.w1 ? a.tiles >> 1 : a.tiles;
  const int mat = tile >= per_mat;
  const int row0 = (tile - mat * per_mat) * kTokRows + 32 * wave;
  const int sb0 = share * a.sb_per, n = min(a.sb_per, a.nsb - sb0);
  const uint8_t* wr = (mat ? a.w1 : a.w0) + we + int64_t(min(row0 + r32, a.rows - 1)) * a.rb + int64_t(sb0) * F::kSbBytes;
  const uint8_t* img = a.img + (int64_t(group) * a.nsb + sb0) * S::kSb;
  const int blk0 = a.nblk - 8 * sb0;  // blocks from this share's first

  using Raw = typename std::conditional<CO, TokNone, typename F::Raw>::type;
  Raw raw0, raw1;  // even and odd super-blocks: no copies between them
  TokWave<F, CO> wv((mat ? a.w1 : a.w0) + we, row0, a.rows, a.rb, sb0,
                    lds + (S::kPacked ? 3 * S::kSb : 3 * S::kGroup + S::kSums + 1024), wave, lane);
  typename F::Sb sb;
  f32x16_t y[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) y[t] = f32x16_t{};

  // one 64-column group: its k steps into acc (kSub 0, over the super-block)
  // or scaled by sub-block into acc
  auto group_mma = [&](auto G, const uint8_t* A, f32x16_t (&acc)[kSums], int left) {
    constexpr int g = decltype(G)::value;
    // fragments of one sub-block at a time, or (32-column scales) of both
    constexpr bool kBoth = F::kSub == 2;
    TokFrag f[2][2];
    auto frags = [&](int jj) {
      if (jj == 0)
        F::template frags<g, 0>(sb, f[0]);
      else
        F::template frags<g, 1>(sb, f[kBoth]);
    };
    auto frag_a = [&](int t, int k, int limb) {
      const int at = TOK == 8 ? (16 * half + (lane & 15)) * 16 : 16 * lane;
      return *reinterpret_cast<const f16x8_t*>(A + ((t * 4 + k) * S::kLimbs + limb) * S::kPiece + at);
    };
    // the weights of k step k that a limb meets: integers up to 2^11, so
    // 2^-11 of them is exact
    auto frag_b = [&](int k, int limb) {
      const f16x8_t w = f[kBoth ? k >> 1 : 0][k & 1].v;
      return limb && !kOwnLo ? w * static_cast<_Float16>(kTokLo) : w;
    };
    if constexpr (F::kSub == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k % 2 == 0) frags(k / 2);
#pragma unroll
        for (int limb = 0; limb < S::kLimbs; ++limb)
#pragma unroll
          for (int t = 0; t < NT; ++t)
          {
            f32x16_t& d = acc[kOwnLo && limb ? NT + t : t];
            d = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag_a(t, k, limb), frag_b(k, limb), d, 0, 0, 0);
          }
      }
    } else {
      // unit u = (k steps of a sub-block, tile): its MFMAs go out before unit
      // u - 1's sums are scaled, so the two overlap and only two units' sums
      // are held (the barriers keep the compiler from batching the MFMAs)
      constexpr int kSteps = F::kSub == 1 ? 1 : 2, kUnits = 4 / kSteps * NT;
      f32x16_t dd[2];
      float sc = 0.f;
#pragma unroll
      for (int u = 0; u <= kUnits; ++u) {
        if (u < kUnits) {
          const int k = u / NT * kSteps, t = u % NT;
          if (t == 0 && (kBoth ? k == 0 : k % 2 == 0)) {
            frags(k / 2);
            if constexpr (kBoth) frags(1);
          }
          f32x16_t v = {};
#pragma unroll
          for (int k2 = 0; k2 < kSteps; ++k2)
#pragma unroll
            for (int limb = 0; limb < S::kLimbs; ++limb)
              v = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag_a(t, k + k2, limb), frag_b(k + k2, limb), v, 0, 0, 0);
          dd[u & 1] = v;
        }
        if (u > 0) {
          const int t = (u - 1) % NT;
          if (t == 0) sc = F::template sub<g>(sb, (u - 1) / NT, a.q6s, left);
#pragma unroll
          for (int i = 0; i < kAcc; ++i) acc[t][i] = __builtin_fmaf(dd[(u - 1) & 1][i], sc, acc[t][i]);
          asm volatile("" : "+v"(acc[t]));  // here and not where the sums are used
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // a super-block's sums into y: y += 2^-k (d acc - dmin 2^5 mn)
  auto finish_sb = [&](const uint8_t* sums, f32x16_t (&acc)[kSums]) {
    const float d = F::d(sb);
    const float* pk = reinterpret_cast<const float*>(sums + S::kSums);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x16_t mn = {};
      float dm = 0.f;
      if constexpr (F::kMin) {
        dm = -32.f * F::dmin(sb);
        const int at = TOK == 8 ? (16 * half + (lane & 15)) * 16 : 16 * lane;
        const _Float16 lo = static_cast<_Float16>(!S::kPacked && half ? kTokLo : 1.f);
        mn = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8_t*>(sums + t * S::kPiece + at),
                                                    F::mins(sb) * lo, mn, 0, 0, 0);
      }
#pragma unroll
      for (int i4 = 0; i4 < kAcc / 4; ++i4) {
        const int tk = TOK == 8 ? 4 * half : TOK == 16 ? 8 * (i4 & 1) + 4 * half : 32 * t + 8 * i4 + 4 * half;
        const f32x4 p = *reinterpret_cast<const f32x4*>(pk + tk);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[t][4 * i4 + i];
          if constexpr (kOwnLo) v = __builtin_fmaf(kTokLo, acc[NT + t][4 * i4 + i], v);
          v *= d;
          if constexpr (F::kMin) v = __builtin_fmaf(dm, mn[4 * i4 + i], v);
          y[t][4 * i4 + i] = __builtin_fmaf(p[i], v, y[t][4 * i4 + i]);
        }
      }
    }
  };
  auto load_sb = [&](int s, auto G, Raw& raw) {
    const int sc = min(s, n - 1);
    if constexpr (!CO)
      F::template load<decltype(G)::value>(wr + int64_t(sc) * F::kSbBytes, half, raw, blk0 - 8 * sc);
    else if constexpr (decltype(G)::value == 0)
      wv.load(sc);
    asm volatile("" ::: "memory");  // the loads stay here, a super-block ahead of their use
  };
  using std::integral_constant;
  const integral_constant<int, 0> g0;
  const integral_constant<int, 1> g1;
  const integral_constant<int, 2> g2;
  const integral_constant<int, 3> g3;

  auto take = [&](auto G, const Raw& cur) {
    constexpr int g = decltype(G)::value;
    if constexpr (CO)
      F::template take_lds<g>(wv.row(r32), wv.sh, wv.tail, half, sb);
    else
      F::template take<g>(cur, sb);
  };
  if constexpr (S::kPacked) {
    // stage = super-block: kCopies copies a wave (past the image: its last
    // KiB again, the same bytes to the same place)
    constexpr int kKib = S::kSb / 1024, kCopies = (kKib + 3) / 4;
    auto stage = [&](int s, int slot) {
      const uint8_t* src = img + int64_t(min(s, n - 1)) * S::kSb;
      uint8_t* dst = lds + slot * S::kSb;
#pragma unroll
      for (int k = 0; k < kCopies; ++k) {
        const int q = min(wave + 4 * k, kKib - 1);
        copy16_to_lds(src + q * 1024 + 16 * lane, dst + q * 1024);
      }
    };
    load_sb(0, g0, raw0);
    load_sb(0, g1, raw0);
    load_sb(0, g2, raw0);
    load_sb(0, g3, raw0);
    stage(0, 0);
    stage(1, 1);
    wait_vmem<kCopies>();
    int slot = 0;
    auto super_block = [&](int s, Raw& cur, Raw& next) {
      // weights of s and stage s have landed when no more than the newest
      // kCopies operations, stage s + 1's copies, are outstanding. The next
      // weights go out ahead of the next copies: a wait for them with copies
      // behind would be a wait for everything (the compiler counts no vector
      // memory operation past a pending LDS copy)
      wait_vmem<kCopies>();
      lds_barrier();
      if constexpr (CO) wv.store(s);
      load_sb(s + 1, g0, next);
      load_sb(s + 1, g1, next);
      load_sb(s + 1, g2, next);
      load_sb(s + 1, g3, next);
      stage(s + 2, slot == 0 ? 2 : slot - 1);
      const uint8_t* A = lds + slot * S::kSb;
      const int left = blk0 - 8 * s;
      f32x16_t acc[kSums] = {};
      take(g0, cur);
      group_mma(g0, A, acc, left);
      take(g1, cur);
      group_mma(g1, A + S::kGroup, acc, left);
      take(g2, cur);
      group_mma(g2, A + 2 * S::kGroup, acc, left);
      take(g3, cur);
      group_mma(g3, A + 3 * S::kGroup, acc, left);
      finish_sb(A + 4 * S::kGroup, acc);
      slot = slot == 2 ? 0 : slot + 1;
    };
    for (int s = 0; s < n; s += 2) {
      super_block(s, raw0, raw1);
      if (s + 1 < n) super_block(s + 1, raw1, raw0);
    }
  } else {
    // stage = 64 columns: 2 NT copies a wave; the sums and 2^-k of a
    // super-block go to an area of their own in its first stage
    constexpr int kCopies = 2 * NT;
    uint8_t* tail = lds + 3 * S::kGroup;
    auto stage = [&](int c, int slot) {
      const int cc = min(c, 4 * n - 1);
      const uint8_t* src = img + int64_t(cc >> 2) * S::kSb + (cc & 3) * S::kGroup;
      uint8_t* dst = lds + slot * S::kGroup;
#pragma unroll
      for (int k = 0; k < kCopies; ++k) {
        const int q = wave + 4 * k;
        copy16_to_lds(src + q * 1024 + 16 * lane, dst + q * 1024);
      }
    };
    load_sb(0, g0, raw0);
    load_sb(0, g1, raw0);
    load_sb(0, g2, raw0);
    load_sb(0, g3, raw0);
    stage(0, 0);
    stage(1, 1);
    wait_vmem<kCopies>();
    int slot = 0;
    auto super_block = [&](int s, Raw& cur, Raw& next) {
      f32x16_t acc[kSums] = {};
      const int left = blk0 - 8 * s;
      auto step = [&](auto G) {
        constexpr int g = decltype(G)::value;
        // stage 4 s + g has landed when no more than the newest kCopies
        // operations are outstanding; every wave is past the slot that the
        // next copies overwrite
        wait_vmem<kCopies>();
        lds_barrier();
        if constexpr (CO && g == 0) {
          wv.store(s);
          load_sb(s + 1, G, next);
        }
        if constexpr (g == 0) {
          const int q = min(wave, NT);  // NT fragments and one KiB of 2^-k
          copy16_to_lds(img + int64_t(s) * S::kSb + 4 * S::kGroup + q * 1024 + 16 * lane, tail + q * 1024);
        }
        stage(4 * s + g + 2, slot == 0 ? 2 : slot - 1);
        take(G, cur);
        if constexpr (!CO) load_sb(s + 1, G, next);
        group_mma(G, lds + slot * S::kGroup, acc, left);
        slot = slot == 2 ? 0 : slot + 1;
      };
      step(g0);
      step(g1);
      step(g2);
      step(g3);
      finish_sb(tail, acc);
    };
    for (int s = 0; s < n; s += 2) {
      super_block(s, raw0, raw1);
      if (s + 1 < n) super_block(s + 1, raw1, raw0);
    }
  }

  wait_vmem<0>();  // no copy into this workgroup's LDS outlives it
  // ---- the share's sums
  const int r = row0 + r32;
  if (r >= a.rows) return;
  float* o = a.out + share * a.part + int64_t(p0) * a.ld + int64_t(mat) * a.rows + r;
  if constexpr (S::kPacked) {
#pragma unroll
    for (int i = 0; i < TOK / 2; ++i) {
      const int t = TOK == 8 ? 4 * half + i : 8 * (i >> 2) + 4 * half + (i & 3);
      if (t < cnt) o[int64_t(t) * a.ld] = __builtin_fmaf(kTokLo, y[0][i + TOK / 2], y[0][i]);
    }
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tk = 32 * t + 8 * (i >> 2) + 4 * half + (i & 3);
        if (tk < cnt) o[int64_t(tk) * a.ld] = y[t][i];
      }
  }
}

// out[i] = res[i] + sum_s part[s][i], in order of s (res optional); V floats
// a thread.
template <int V>
__global__ void __launch_bounds__(256) tok_sum_kernel(const float* __restrict__ part, int64_t stride, int nsplit,
                                                      const float* res, float* out, int64_t n) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const int64_t i = V * (blockIdx.x * int64_t(blockDim.x) + threadIdx.x);
  if (i >= n) return;
  vec v = *reinterpret_cast<const vec*>(part + i);
  for (int s = 1; s < nsplit; ++s) v += *reinterpret_cast<const vec*>(part + s * stride + i);
  if (res) v = *reinterpret_cast<const vec*>(res + i) + v;
  *reinterpret_cast<vec*>(out + i) = v;
}

// ------------------------------------------------------------------- host --
bool tok_ok(uint32_t quant, int64_t rows, int64_t cols) {
  return device_quant(quant) && rows > 0 && rows <= (int64_t(1) << 24) && cols > 0 && cols <= (int64_t(1) << 20) &&
         cols % geometry(quant).block == 0;
}

TokPlan tok_plan(int64_t rows, int mats, int64_t cols, int tokens, int cu, int max_split) {
  TokPlan p{};
  if (tokens <= 16) {  // (fewer than 9 stay with the matvecs)
    p.tok = 16;
  } else {
    const int g = (tokens + 95) / 96;
    p.tok = ((tokens + g - 1) / g + 31) / 32 * 32;
  }
  p.groups = (tokens + p.tok - 1) / p.tok;
  p.nsb = int((cols + 255) / 256);
  p.tiles = int((rows + kTokRows - 1) / kTokRows) * mats;
  // workgroups a round: two per CU (what LDS holds) from 64 tokens. Below it
  // holds one to three with the weights' slots, and four are counted: fewer,
  // longer shares took up to 9% more (three matrices of 5120 / 17408 Q6_K, 17
  // tokens 124 us, counting two 135; 3584 / 8192, 9 tokens, 58 / 56)
  const int64_t slots = int64_t(cu) * (p.tok >= 64 ? 2 : 4);
  // shares of the columns: the fewest rounds of workgroups, each round as
  // long as a share plus about two super-blocks of start and end
  double best = 0;
  for (int s = 1; s <= std::min(max_split, p.nsb); ++s) {
    const int per = (p.nsb + s - 1) / s;
    if ((p.nsb + per - 1) / per != s) continue;
    const int64_t wg = int64_t(p.tiles) * p.groups * s;
    const double t = std::max(1.0, double(wg) / double(slots)) * (per + 2) + 0.25 * s;
    if (p.nsplit == 0 || t < best) {
      best = t;
      p.nsplit = s;
      p.sb_per = per;
    }
  }
  return p;
}

size_t tok_image_bytes(const TokPlan& p) { return size_t(p.groups) * p.nsb * size_t(tok_sb_bytes(p.tok)); }

static int tok_perm(uint32_t quant) { return quant == kQ6_K || quant == kIQ4_XS; }

hipError_t launch_tok_prep(const TokPlan& p, uint32_t quant, const float* x, int64_t ld, int cols, int tokens,
                           void* img, hipStream_t s, const int* src, const int* slot) {
  const TokPrep a{x, ld, 0, 1, cols, p.nsb, tokens, p.tok, tok_perm(quant), static_cast<uint8_t*>(img), src, slot};
  hipLaunchKernelGGL(tok_prep_kernel<false>, dim3(unsigned((p.nsb + 3) / 4), unsigned(tokens)), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_tok_prep_silu(const TokPlan& p, uint32_t quant, const float* gu, int64_t ld, int64_t part,
                                int nsplit, int cols, int tokens, void* img, hipStream_t s, const int* slot) {
  const TokPrep a{gu, ld, part, nsplit, cols, p.nsb, tokens, p.tok, tok_perm(quant), static_cast<uint8_t*>(img), nullptr,
                  slot};
  hipLaunchKernelGGL(tok_prep_kernel<true>, dim3(unsigned((p.nsb + 3) / 4), unsigned(tokens)), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <class F, int TOK>
static void launch_tok(const TokMm& a, int64_t blocks, hipStream_t s) {
  using S = TokShape<TOK>;
  const size_t lds = S::kPacked ? 3 * size_t(S::kSb) : 3 * size_t(S::kGroup) + S::kSums + 1024;
  // weights by way of LDS: up to 32 tokens (with more a super-block's MFMAs
  // cover its loads, and the LDS costs a workgroup on the CU: 77 tokens of the
  // dense FFN 116 us direct, 127 by way of LDS), pieces on the dword grid
  // (Q6_K: realigned as they are read), rows of whole super-blocks
  if constexpr (tok_lds_format<F>() && TOK <= 32) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(a.w0) | reinterpret_cast<uintptr_t>(a.w1) | uintptr_t(a.items.stride);
    if (F::kSbBytes % 4 != 0 || ((at & 3u) == 0 && a.rb % F::kSbBytes == 0)) {
      hipLaunchKernelGGL((tok_mm_kernel<F, TOK, true>), dim3(unsigned(blocks)), dim3(kTokThreads),
                         (lds + 4 * TokWave<F, true>::kLds), s, a);
      return;
    }
  }
  hipLaunchKernelGGL((tok_mm_kernel<F, TOK, false>), dim3(unsigned(blocks)), dim3(kTokThreads), lds, s, a);
}
template <class F>
static void launch_tok_f(int tok, const TokMm& a, int64_t blocks, hipStream_t s) {
  switch (tok) {
    case 8: launch_tok<F, 8>(a, blocks, s); break;
    case 16: launch_tok<F, 16>(a, blocks, s); break;
    case 32: launch_tok<F, 32>(a, blocks, s); break;
    case 64: launch_tok<F, 64>(a, blocks, s); break;
    default: launch_tok<F, 96>(a, blocks, s);
  }
}

hipError_t launch_tok_mm(const TokPlan& p, uint32_t quant, const void* w0, const void* w1, int64_t rows, int64_t cols,
                         const void* img, float* out, int64_t ld, int64_t part, int tokens, int reading,
                         hipStream_t s, const TokItems* items) {
  TokMm a{};
  a.w0 = static_cast<const uint8_t*>(w0);
  a.w1 = static_cast<const uint8_t*>(w1);
  a.rows = int(rows);
  a.tiles = p.tiles;
  a.rb = byte_size(quant, cols);
  a.nsb = p.nsb;
  a.sb_per = p.sb_per;
  a.nsplit = p.nsplit;
  a.nblk = int(cols / 32);
  a.img = static_cast<const uint8_t*>(img);
  a.out = out;
  a.ld = ld;
  a.part = part;
  a.tokens = tokens;
  a.groups = p.groups;
  a.q6s = reading;
  if (items) a.items = *items;
  if (items && p.nsplit != 1) return hipErrorInvalidValue;
  const int64_t blocks = items ? int64_t(p.groups + 7) / 8 * 8 * p.tiles
                               : int64_t(p.nsplit) * ((p.tiles + 7) / 8) * p.groups * 8;
  if (blocks > (int64_t(1) << 31) - 1) return hipErrorInvalidValue;
  switch (quant) {
    case kQ4_K: launch_tok_f<TokQ4Q5<kQ4_K>>(p.tok, a, blocks, s); break;
    case kQ5_K: launch_tok_f<TokQ4Q5<kQ5_K>>(p.tok, a, blocks, s); break;
    case kQ6_K: launch_tok_f<TokQ6>(p.tok, a, blocks, s); break;
    case kQ8_0: launch_tok_f<TokQ8>(p.tok, a, blocks, s); break;
    case kIQ4_XS:
      if (reading) launch_tok_f<TokIQ4<true>>(p.tok, a, blocks, s);
      else launch_tok_f<TokIQ4<false>>(p.tok, a, blocks, s);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_tok_sum(const float* part, int64_t stride, int nsplit, const float* res, float* out, int64_t n,
                          hipStream_t s) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(part) | reinterpret_cast<uintptr_t>(res) |
                       reinterpret_cast<uintptr_t>(out) | uintptr_t(4 * n) | uintptr_t(4 * stride);
  if (at & 15u)
    hipLaunchKernelGGL(tok_sum_kernel<1>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, part, stride, nsplit, res,
                       out, n);
  else
    hipLaunchKernelGGL(tok_sum_kernel<4>, dim3(unsigned((n / 4 + 255) / 256)), dim3(256), 0, s, part, stride, nsplit,
                       res, out, n);
  return hipGetLastError();
}

}  // namespace sh
