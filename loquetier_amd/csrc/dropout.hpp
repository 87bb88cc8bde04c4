// Dropout of the training rows of x, applied where x (or dX) passes through registers.
//
// The reference drops x before the LoRA term, one nn.Dropout(p) per adapter
// (src/loquetier_src/models/mixed_lora.py:185-192): a dropped copy of every training partition
// plus a torch.cat of the whole batch, and autograd's mask multiply on the way back.  Here no
// dropped copy of x exists.  The mask is a pure function of (seed, offset, row, column): the
// shrink kernels generate it for the x fragments they load and leave its keep bits behind (one
// byte per eight columns, 1/16 of x's bytes); the backward brings those bits -- or the same bits
// made again by drop_bits_kernel -- into the order of the plan's tiles and applies them to the x rows
// the weight-gradient kernel stages and to the dX values the expand kernel stores.
//
// Mask: the eight 16-bit pieces of philox4x32_10(counter = (row, col / 8, offset), key = seed)
// decide elements col .. col + 7 of a row; an element is dropped when its piece is below
// floor(p * 65536).  Kept elements become round(x * (1 / (1 - p))) (float product, as torch's
// dropout computes it), dropped ones +0.  Rows at or past `rows` (inference rows) and segments
// with p <= 0 pass through untouched.
#pragma once
#include "smlm_common.hpp"

namespace smlm {

struct DropArgs {
  const float* seg_p;  // [S] dropout probability of each segment's adapter; nullptr: no dropout
  int rows;            // training rows are [0, rows)
  uint32_t k0, k1;     // seed
  uint32_t o0, o1;     // offset (distinguishes layers / steps)
  uint8_t* bits;       // optional [rows, bits_pitch]: keep bits, one byte per eight columns of a row;
  long bits_pitch;     //   written by the forward's shrink, read by the backward instead of regenerating
};

// the arguments of projection pj of a launch over several projections: offset + pj
__device__ __forceinline__ DropArgs drop_proj(DropArgs d, int pj) {
  const uint64_t off = (((uint64_t)d.o1 << 32) | d.o0) + (uint32_t)pj;
  d.o0 = (uint32_t)off;
  d.o1 = (uint32_t)(off >> 32);
  return d;
}

struct DropRow {
  uint32_t thresh;  // pieces below it are dropped
  float scale;      // factor of kept elements
  bool on;
};

// threshold and factor of dropout probability p (p <= 0: off, thresh 0 and factor 1)
__device__ __forceinline__ DropRow drop_params(float p) {
  DropRow r;
  r.on = p > 0.0f;
  r.thresh = p >= 1.0f ? 65536u : (r.on ? (uint32_t)(p * 65536.0f) : 0u);
  r.scale = p >= 1.0f ? 0.0f : (r.on ? 1.0f / (1.0f - p) : 1.0f);
  return r;
}

// The dropout probability of a row of segment `seg` (either -1: none), 0 for rows that are not training rows.  A load
// without a branch, so that the loads behind it need not wait for it (zero: readable, holds 0.0f).
__device__ __forceinline__ float drop_prob(const DropArgs& d, int row, int seg, const uint16_t* zero) {
  const bool ok = row >= 0 && row < d.rows && seg >= 0;
  return *(const SMLM_GLOBAL float*)(ok ? d.seg_p + seg : reinterpret_cast<const float*>(zero));
}

__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                              uint32_t k1, uint32_t (&out)[4]) {
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    if (i) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    // (three-way exclusive or: truth table 0x96)
    const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
    const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
    c1 = (uint32_t)p1;
    c3 = (uint32_t)p0;
    c0 = n0;
    c2 = n2;
  }
  out[0] = c0, out[1] = c1, out[2] = c2, out[3] = c3;
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Which of the eight elements at columns 8*colblk .. +7 of a row are kept, two to a word as the elements are: 1 in the half
// of a kept element, 0 in a dropped one's.  Two elements an instruction: thresh - piece, saturating at zero, is nonzero
// exactly where the piece is below thresh.  A thresh of 65536 (p >= 1) does not fit a half: the caller's last AND, with
// drop_none_kept, takes what is left.
__device__ __forceinline__ u32x4 drop_keep_pairs(const DropArgs& d, uint32_t thresh, int row, int colblk) {
  uint32_t w[4];
  philox4x32_10((uint32_t)row, (uint32_t)colblk, d.o0, d.o1, d.k0, d.k1, w);
  const uint16_t t16 = (uint16_t)(thresh < 65535u ? thresh : 65535u);
  uint32_t ones = 0x00010001u;
  asm("" : "+s"(ones));  // (knowing the value, the compiler turns this back into compares and selects, an element each)
  const u16x2 t = {t16, t16}, one = __builtin_bit_cast(u16x2, ones);
  u32x4 k;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    k[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(
                                            one, __builtin_elementwise_sub_sat(t, __builtin_bit_cast(u16x2, w[e]))));
  return k;
}
__device__ __forceinline__ uint32_t drop_none_kept(uint32_t thresh) { return thresh > 65535u ? 0u : ~0u; }

// the same as keep bits: bit e = element e is kept
__device__ __forceinline__ uint32_t keep_bits8(u32x4 k, uint32_t limit) {
  const uint32_t b = k[0] | (k[1] << 2) | (k[2] << 4) | (k[3] << 6);
  return (b | (b >> 15)) & 0xffu & limit;
}
__device__ __forceinline__ uint32_t drop_keep8(const DropArgs& d, uint32_t thresh, int row, int colblk) {
  return keep_bits8(drop_keep_pairs(d, thresh, row, colblk), drop_none_kept(thresh));
}

// Whether a projection's keep bits can be stored U (2 or 4) bytes at a time: rows and addresses in multiples of U.
template <int U>
__device__ __forceinline__ bool drop_words(const uint8_t* bits, long pitch) {
  return ((reinterpret_cast<uintptr_t>(bits) | (uintptr_t)pitch) & (U - 1)) == 0;
}

// The masks of U x-fragments of a wave, lane (c, g) holding columns 8 (colblk0 + 4 u + g) .. +7 of row c in fragment u.
// They need nothing of x: the shrink kernels make them while x is on its way, U generators side by side, whose ten rounds
// each wait for the one before.  One generator at a time behind x's arrival, a byte stored for each, and so, us: forward
// of 2786 rows, two projections 4096 -> 4096 at rank 32 50.5 and 47.1, 900 rows 27.1 and 25.9, 8000 rows at rank 16 108.2
// and 96.6 (without dropout 83).  Most of that is the stores: rows of the mask that only take single bytes gain nothing.
template <int U>
struct DropMasks {
  u32x4 m[U];  // 0xffff in the half of a kept element, 0 in a dropped one's

  // bits_out (may be nullptr): the row's keep bits, one byte per eight columns, are left there for a later pass that reads
  // them instead of running the generator again; blocks at or past colblk_end are not.  words: drop_words<U> of them; the
  // bytes of a row then go out U from each of its four lanes instead of one at a time.
  __device__ __forceinline__ void make(const DropArgs& d, const DropRow& r, int row, int colblk0, int g, uint8_t* bits_out,
                                       long pitch, int colblk_end, bool words) {
    const uint32_t limit = drop_none_kept(r.thresh);
    uint32_t b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u32x4 k = drop_keep_pairs(d, r.thresh, row, colblk0 + 4 * u + g);
      b[u] = keep_bits8(k, limit);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t ke = k[e];  // (a vector's element cast in place reads element 0: clang)
        m[u][e] = __builtin_bit_cast(uint32_t, (u16x2)(u16x2{0, 0} - __builtin_bit_cast(u16x2, ke)));
      }
    }
    if (!bits_out) return;  // uniform over the wave
    uint8_t* const at = bits_out + (long)row * pitch + colblk0;
    static_assert(U == 2 || U == 4, "");
    if (words) {  // uniform over the wave
      // lane g holds bytes 4 u + g of the row's 4 U and stores bytes U g + j
      if constexpr (U == 4) {  // halves change places with the lane two groups away, then bytes with the lane next door
        const uint32_t w = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
        const auto h = __builtin_amdgcn_permlane32_swap(w, w, false, false);  // the words of groups g & 1 and (g & 1) + 2
        const uint32_t v = __builtin_amdgcn_perm(h[1], h[0], g & 2 ? 0x07060302u : 0x05040100u);
        const auto q = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // ... of the even and the odd group
        const uint32_t o = __builtin_amdgcn_perm(q[1], q[0], g & 1 ? 0x07030501u : 0x06020400u);
        if (r.on && colblk0 + 4 * g < colblk_end) *(SMLM_GLOBAL uint32_t*)(at + 4 * g) = o;
      } else {  // the pairs of neighbours together, then the pair and the fragment the lane stores
        const uint32_t w = b[0] | (b[1] << 8);
        const auto q = __builtin_amdgcn_permlane16_swap(w, w, false, false);
        const uint32_t v = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u);
        const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // of pairs 0 and 1
        const uint32_t o = (g & 1 ? h[1] : h[0]) >> (g & 2 ? 16 : 0);
        if (r.on && colblk0 + 2 * g < colblk_end) *(SMLM_GLOBAL uint16_t*)(at + 2 * g) = (uint16_t)o;
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r.on && colblk0 + 4 * u + g < colblk_end) *(SMLM_GLOBAL uint8_t*)(at + 4 * u + g) = (uint8_t)b[u];
  }

  // fragment u of x: kept elements times the factor (float product, rounded to the 16-bit type), dropped ones +0.  Rows
  // that are not dropped have thresh 0 and factor 1: the product is the element.
  template <int DT>
  __device__ __forceinline__ u32x4 apply(u32x4 v, int u, const DropRow& r) const {
    const uint32_t limit = drop_none_kept(r.thresh);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = __builtin_amdgcn_bitop3_b32(pack2<DT>(Num<DT>::lo(v[e]) * r.scale, Num<DT>::hi(v[e]) * r.scale), m[u][e],
                                         limit, 0x80);  // (three-way and)
    return o;
  }
};

// Eight elements of a row from their stored keep bits: kept ones times the factor, dropped ones +0; rows that are not
// dropped keep everything, times 1.
template <int DT>
__device__ __forceinline__ u32x4 drop8_bits(u32x4 v, const DropRow& r, uint32_t keep) {
  const float scale = r.on ? r.scale : 1.0f;
  const int k = r.on ? (int)keep : 0xff;
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_sbfe(k, 2 * e, 1), hi = (uint32_t)__builtin_amdgcn_sbfe(k, 2 * e + 1, 1);
    o[e] = pack2<DT>(Num<DT>::lo(v[e]) * scale, Num<DT>::hi(v[e]) * scale) & ((lo & 0xffffu) | (hi & 0xffff0000u));
  }
  return o;
}

// Keep bits as dX and the weight gradients read them, by tile slot: [tile][64 columns][8 pairs of slots][8 bytes][2], a
// line for 64 columns of a tile.  A pair is the slots s and s + 4 that a lane of the weight gradients stages one after the
// other, so that their two bytes are one load and one register.  (Read by row, the bits of 64 columns are eight bytes of a
// line a row, fetched by every XCD: under dropout at rank 32 the weight gradients of two adapters of 1024 rows, two
// projections, took 25.5 us, without 18.9.)
__device__ __forceinline__ long tile_bits(int tile, int chunk, int chunks, int slot, int byte) {
  return (((long)tile * chunks + chunk) * 8 + ((slot & 3) | (slot >> 3) << 2)) * 16 + 2 * byte + (slot >> 2 & 1);
}

// The bits the forward left by row, by tile slot: an item of 256 threads is a tile and 1024 columns.
struct TileBits {
  const uint8_t* rows_bits[8];  // [rows, pitch] of each projection
  uint8_t* out[8];
  int pitch[8], chunks[8];      // bytes of a row; ceil(columns / 64)
  int first[9];                 // items of projection i: [first[i], first[i + 1])
  int n, rows, tiles;           // projections (0: nothing to do), training rows, bound of the plan's tiles
};
__device__ __forceinline__ void tile_bits_item(const TileBits& z, const int32_t* tile_row, int item, int thread) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < 8; ++j) i += (j < z.n && item >= z.first[j]) ? 1 : 0;
  const int in = item - z.first[i], tile = in % z.tiles;
  // a wave takes two pairs of slots, the second of each 16 lanes after the first
  const int pair = thread >> 5, second = thread >> 4 & 1, slot = (pair & 3) + 4 * second + 8 * (pair >> 2);
  const int chunk = in / z.tiles * 16 + (thread & 15);
  const int row = tile_row[tile * kTileRows + slot];
  const bool ok = row >= 0 && row < z.rows && chunk < z.chunks[i];
  u32x2 v = {0u, 0u};
  if (ok) {
    const uint8_t* from = z.rows_bits[i] + (long)row * z.pitch[i] + 8 * chunk;
    if (((reinterpret_cast<uintptr_t>(z.rows_bits[i]) | (uintptr_t)z.pitch[i]) & 7u) == 0) {  // uniform over the workgroup
      v = *(const SMLM_GLOBAL u32x2*)from;
    } else {
      const int left = z.pitch[i] - 8 * chunk;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < left) v[e >> 2] |= (uint32_t)*(const SMLM_GLOBAL uint8_t*)(from + e) << (8 * (e & 3));
    }
  }
  const bool write = ok | (__shfl_xor((int)ok, 16) != 0);
  const uint32_t own = second ? v[1] : v[0], got = (uint32_t)__shfl_xor((int)(second ? v[0] : v[1]), 16);
  const uint32_t lo = second ? got : own, hi = second ? own : got;  // four bytes of the first slot, of the second
  if (write)
    *(SMLM_GLOBAL u32x2*)(z.out[i] + tile_bits(tile, chunk, z.chunks[i], slot & ~4, 4 * second)) =
        u32x2{__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u)};
}
struct TileBitsArgs {
  TileBits bits;
  const int32_t* tile_row;
};
__global__ __launch_bounds__(256) void tile_bits_kernel(TileBitsArgs a) {
  tile_bits_item(a.bits, a.tile_row, (int)blockIdx.x, threadIdx.x);
}

// The same bits made anew, where the caller of a backward has none: workgroup -> tile, thread -> (row slot, column
// blocks slot-strided by 16).
struct DropBitsArgs {
  const int32_t* hdr;        // plan header: [0] = number of tiles
  const int32_t* tile_row;
  const int32_t* tile_rseg;
  DropArgs drop;             // bits: the output, by tile slot; bits_pitch: column blocks of a row
};

__global__ __launch_bounds__(256) void drop_bits_kernel(DropBitsArgs a) {
  const int tile = blockIdx.x;
  if (tile >= a.hdr[0]) return;
  const int slot = threadIdx.x >> 4, chunks = (int)((a.drop.bits_pitch + 7) / 8);
  const int row = a.tile_row[tile * kTileRows + slot];
  const DropRow r = drop_params(drop_prob(a.drop, row, a.tile_rseg[tile * kTileRows + slot],
                                          reinterpret_cast<const uint16_t*>(a.hdr + kHdrZeros)));
  if (!r.on) return;  // rows that are not dropped never have their byte applied
  for (int cb = threadIdx.x & 15; cb < a.drop.bits_pitch; cb += 16)
    a.drop.bits[tile_bits(tile, cb >> 3, chunks, slot, cb & 7)] = (uint8_t)drop_keep8(a.drop, r.thresh, row, cb);
}

}  // namespace smlm
