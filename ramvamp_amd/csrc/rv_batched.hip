// rv_batched.hip — the batched GEMVs of a prefill chunk (gemv.rs:444-543,
// :616-651) on int8 MFMA, bit-identical to the scalar dots.
//
// out[i][a] = row(row_lo + i) . act_row(a). Every output is the scalar dot's
// f32 value bit for bit: the integer sums are exact and the per-block float
// expression and the block order are the scalar kernel's. A launch runs up to
// three matrices (a chunk's k, v and q projections) over the same activations.
//
// The k-quant sums go through v_mfma_i32_16x16x64_i8 with the sub-block scales
// folded into two int8 planes of the weights. sc * q does not fit in int8;
// it is split so that each plane is a packed product with no carries:
//   Q4_K: sc = 8 sh + sl (sh, sl <= 7), q <= 15: planes sh*q, sl*q (<= 105),
//     sumi = 8 H + L;
//   Q5_K: sh*q and sl*q reach 217, so the planes hold them less 128 (the top
//     bit flipped) and sumi = 8 H + L + 9 * 128 A, A the sum of the block's
//     activations;
//   Q6_K: sum_s sc_s (sum q a - 32 bsum_s) (dot.rs:150-179) is exactly
//     sum sc (q - 32) a; sc (q - 32) = 64 hi + lo (lo < 64): sumi = 64 H + L;
//   Q8_0: the weight bytes themselves, one 16x16x32 MFMA per 32-weight block.
// The mins' sum (and A) is one f16 MFMA a block: its 16 k slots are the sums
// of 16 consecutive activations (at most 2048 in magnitude, exact in f16)
// against their sub-block's min (against ones), every product and sum an
// integer below 2^24, so exact in f32.
//
// A workgroup of 8 waves owns 16 weight rows x 128 activation rows. It
// unpacks the planes of KC blocks of its rows into LDS, then every wave runs
// its own tile of 16 activation rows against all of them without a barrier;
// the packed bytes of the next KC blocks are loaded meanwhile. What bounds it
// is instruction issue: a wave issues at most one instruction in about 5
// cycles, so it is kept to 128 registers (four waves per SIMD). Measured for
// a 512-row chunk at hidden 2048, q_dim 4096 (q Q4_K, k Q8_0, v Q6_K, o
// Q5_K): 53 us in two launches, against 118 us in four with the planes built
// per block behind two barriers and scattered loads; 77 rows 25 us against 97.
// Not faster: two or four tiles a wave with fewer waves (within 8 %), all of a
// row's blocks unpacked before the products (64 KiB of LDS: 512 rows 34 against
// 30 us), operands built in each wave's registers (53 against 33 us), one
// tile's float work issued between the next one's MFMAs.
// Loads go to consecutive lanes at dword-aligned addresses: a 64-lane load
// whose neighbouring lanes fall into different rows takes 64 cycles of the
// CU's address unit whatever its width, and one of 16 bytes a lane at odd
// 2-byte offsets 140-280, against 16 for 1 KiB contiguous. A prefill chunk's
// activations come in operand order from the rows quantizer (PackedActs,
// rv_quant.hpp), 1 KiB contiguous per load; those of the public calls are blocks
// row by row, turned around on the way (TurnedActs) unless they are few.
#include <type_traits>

#include "rv_device.hpp"
#include "rv_internal.hpp"
#include "rv_quant.hpp"

namespace rv {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
// Global accesses at the alignment the packed rows have (2 or 4 bytes).
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 f16x4a __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float f16_bits(uint32_t bits) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits & 0xFFFFu));
}

// ---- weights: unpacking into LDS ------------------------------------------------

constexpr int kW = 8;   // waves, each with one activation tile
constexpr int kR = 16;  // weight rows
constexpr int KC = 4;   // 256-weight blocks unpacked at a time

// Byte of a block's plane where the 16-byte chunk c (values 16 c .. + 15) of
// row r lies: chunks permuted by the row, so that 16 rows' reads of one chunk
// and the unpacking's writes each fall on all 64 banks.
__device__ __forceinline__ int chunk_at(int r, int c) { return 256 * r + 16 * (c ^ (r & 15)); }

// The unpacked weights of KC blocks (Q8_0: groups of eight blocks) of kR rows.
struct Planes {
  int8_t p[KC][2][kR * 256];
  _Float16 mins[KC][kR][8];  // [4 (j % 2) + j / 2]: sub-block j's min
  float d[KC][2][kR];        // d, dmin
};
struct Planes0 {
  int8_t p[KC][kR * 256];
  float d[KC][8][kR];  // block c's d
};

// What a thread unpacks at a time. k-quants: 16 bytes of quants (piece p of
// eight, 32 weights) of one block; Q8_0: 8 bytes (piece p of 32) of a group.
template <int FMT>
struct Raw;
template <>
struct Raw<RV_QF_Q4_K> {
  u32x4a hdr, q;
};
template <>
struct Raw<RV_QF_Q5_K> {
  u32x4a hdr, q, h;
};
template <>
struct Raw<RV_QF_Q6_K> {
  u32x4a q, h;  // from the dword below when the block starts 2 past one,
  uint32_t q4, h4;  // and the dword after each
  int s0, s1;
  uint32_t d, odd;
};
template <>
struct Raw<RV_QF_Q8_0> {
  uint32_t a, b, c;
  uint32_t d, odd;
};

template <int FMT>
__device__ __forceinline__ void load_raw(Raw<FMT>& w, const uint8_t* __restrict__ row, int nb, int blk, int p) {
  if constexpr (FMT == RV_QF_Q8_0) {
    const uint8_t* b = row + (size_t)min(8 * blk + (p >> 2), nb - 1) * 34;
    const uint8_t* q = b + 2 + 8 * (p & 3);
    w.odd = (uint32_t)(uintptr_t)q & 2;
    const uint32_t* qa = reinterpret_cast<const uint32_t*>(q - w.odd);
    w.a = qa[0];
    w.b = qa[1];
    w.c = *reinterpret_cast<const uint16_t*>(q + 6);  // the last two bytes (in c's low half)
    w.d = *reinterpret_cast<const uint16_t*>(b);
  } else if constexpr (FMT == RV_QF_Q6_K) {
    const uint8_t* b = row + (size_t)min(blk, nb - 1) * 210;
    w.odd = (uint32_t)(uintptr_t)b & 2;
    const uint8_t* q = b + 16 * p - w.odd;
    const uint8_t* h = b + 128 + 32 * (p >> 2) + 16 * (p & 1) - w.odd;
    w.q = *reinterpret_cast<const u32x4a*>(q);
    w.q4 = *reinterpret_cast<const uint32_t*>(q + 16);
    w.h = *reinterpret_cast<const u32x4a*>(h);
    w.h4 = *reinterpret_cast<const uint32_t*>(h + 16);
    const int8_t* sc = reinterpret_cast<const int8_t*>(b + 192 + 8 * (p >> 2) + (p & 3));
    w.s0 = sc[0];
    w.s1 = sc[4];
    w.d = *reinterpret_cast<const uint16_t*>(b + 208);
  } else {
    constexpr bool kQ5 = FMT == RV_QF_Q5_K;
    const uint8_t* b = row + (size_t)min(blk, nb - 1) * (kQ5 ? 176 : 144);
    w.hdr = *reinterpret_cast<const u32x4a*>(b);
    w.q = *reinterpret_cast<const u32x4a*>(b + (kQ5 ? 48 : 16) + 16 * p);
    if constexpr (kQ5) w.h = *reinterpret_cast<const u32x4a*>(b + 16 + 16 * (p & 1));
  }
}

// q's four bytes times s, no carry between bytes (q * s <= 255).
__device__ __forceinline__ uint32_t mul_bytes(uint32_t q, uint32_t s) {
  const unsigned short f = (unsigned short)s;
  return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, q) * u16x2{f, f}));
}

// Four 6-bit weights (bytes of q, 0..63) times sc after subtracting 32: v =
// 64 hi + lo, hi and lo packed as bytes.
__device__ __forceinline__ void split_q6(uint32_t q, int sc, int& hi, int& lo) {
  const short f = (short)sc, m = (short)(-32 * sc);
  const s16x2 e = __builtin_bit_cast(s16x2, q & 0x00FF00FFu) * s16x2{f, f} + s16x2{m, m};
  const s16x2 o = __builtin_bit_cast(s16x2, (q >> 8) & 0x00FF00FFu) * s16x2{f, f} + s16x2{m, m};
  const uint32_t he = __builtin_bit_cast(uint32_t, (s16x2)(e >> 6)), ho = __builtin_bit_cast(uint32_t, (s16x2)(o >> 6));
  // bytes (0, 2) of the even pair beside bytes (0, 2) of the odd one
  hi = (int)__builtin_amdgcn_perm(ho, he, 0x06020400u);
  lo = (int)(__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, e), 0x06020400u) &
             0x3F3F3F3Fu);
}

__device__ __forceinline__ void put16(int8_t* at, i32x4 v) { *reinterpret_cast<i32x4*>(at) = v; }

// Piece p of row r's k-th block into the planes, whose bytes are in the
// weights' own order.
template <int FMT>
__device__ __forceinline__ void build(const Raw<FMT>& w, Planes& pl, int r, int k, int p) {
  i32x4 h0, l0, h1, l1;  // the low nibbles' weights, the high nibbles'
  if constexpr (FMT == RV_QF_Q6_K) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t q = __builtin_amdgcn_alignbyte(e < 3 ? w.q[e + 1] : w.q4, w.q[e], w.odd);
      const uint32_t t = __builtin_amdgcn_alignbyte(e < 3 ? w.h[e + 1] : w.h4, w.h[e], w.odd) >> (p & 2);
      int a, b;
      split_q6((q & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u), w.s0, a, b);
      h0[e] = a, l0[e] = b;
      split_q6(((q >> 4) & 0x0F0F0F0Fu) | (t & 0x30303030u), w.s1, a, b);
      h1[e] = a, l1[e] = b;
    }
    const int c0 = chunk_at(r, 8 * (p >> 2) + (p & 3)), c1 = chunk_at(r, 8 * (p >> 2) + (p & 3) + 4);
    put16(&pl.p[k][0][c0], h0);
    put16(&pl.p[k][1][c0], l0);
    put16(&pl.p[k][0][c1], h1);
    put16(&pl.p[k][1][c1], l1);
    if (p == 0) pl.d[k][0][r] = f16_bits(w.d);
  } else {
    constexpr bool kQ5 = FMT == RV_QF_Q5_K;
    const int jj = p >> 1;
    // get_scale_min_k4 (quants/blocks.rs:158-167) of sub-blocks 2 jj, 2 jj + 1.
    const uint32_t t0 = w.hdr[1], t1 = w.hdr[2], t2 = w.hdr[3];
    const uint32_t s4 = jj < 2 ? t0 & 0x3F3F3F3Fu : (t2 & 0x0F0F0F0Fu) | ((t0 >> 2) & 0x30303030u);
    const uint32_t m4 = jj < 2 ? t1 & 0x3F3F3F3Fu : ((t2 >> 4) & 0x0F0F0F0Fu) | ((t1 >> 2) & 0x30303030u);
    const uint32_t s2 = s4 >> (16 * (jj & 1)), m2 = m4 >> (16 * (jj & 1));
    const uint32_t sa = s2 & 0xFFu, sb = (s2 >> 8) & 0xFFu;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t q0 = w.q[e] & 0x0F0F0F0Fu, q1 = (w.q[e] >> 4) & 0x0F0F0F0Fu;
      if constexpr (kQ5) {
        const uint32_t t = w.h[e] >> (2 * jj);  // bits 0, 1: the two sub-blocks' fifth bits
        q0 |= (t << 4) & 0x10101010u;
        q1 |= (t << 3) & 0x10101010u;
      }
      const uint32_t f = kQ5 ? 0x80808080u : 0u;
      h0[e] = (int)(mul_bytes(q0, sa >> 3) ^ f);
      l0[e] = (int)(mul_bytes(q0, sa & 7u) ^ f);
      h1[e] = (int)(mul_bytes(q1, sb >> 3) ^ f);
      l1[e] = (int)(mul_bytes(q1, sb & 7u) ^ f);
    }
    const int c0 = chunk_at(r, 4 * jj + (p & 1)), c1 = chunk_at(r, 4 * jj + (p & 1) + 2);
    put16(&pl.p[k][0][c0], h0);
    put16(&pl.p[k][1][c0], l0);
    put16(&pl.p[k][0][c1], h1);
    put16(&pl.p[k][1][c1], l1);
    if ((p & 1) == 0) {
      pl.mins[k][r][jj] = (_Float16)(float)(m2 & 0xFFu);
      pl.mins[k][r][4 + jj] = (_Float16)(float)((m2 >> 8) & 0xFFu);
    }
    if (p == 0) {
      pl.d[k][0][r] = f16_bits(w.hdr[0]);
      pl.d[k][1][r] = f16_bits(w.hdr[0] >> 16);
    }
  }
}

// Q8_0: piece p = 4 c + kq (8 bytes) of row r's k-th group into operand order.
__device__ __forceinline__ void build0(const Raw<RV_QF_Q8_0>& w, Planes0& pl, int r, int k, int p) {
  const int c = p >> 2, kq = p & 3;
  // odd: a, b hold bytes -2 .. 5 and c bytes 6, 7; else a, b are the eight.
  const uint32_t x = __builtin_amdgcn_alignbyte(w.b, w.a, w.odd), y = w.odd ? (w.b >> 16) | (w.c << 16) : w.b;
  *reinterpret_cast<i32x2*>(&pl.p[k][chunk_at(r, 4 * (c >> 1) + kq) + 8 * (c & 1)]) = i32x2{(int)x, (int)y};
  if (kq == 0) pl.d[k][c][r] = f16_bits(w.d);
}

// ---- activations -----------------------------------------------------------

// One block's (Q8_0: eight blocks') operands of a 16-row tile: lane (col, kq)
// holds column col's 16 bytes of each 64-value chunk, and the sums of those.
template <int FMT>
struct Act {
  i32x4 q[4];
  f16x4 bs;
  float d[FMT == RV_QF_Q8_0 ? 8 : 1];
};

// How a wave gets its activation tile, one block (Q8_0: a group of eight) after
// another: packed operands as they are; public blocks in operand order straight
// from memory (k-quants); or public blocks turned around in LDS (TurnedActs).
enum ActSrc { kPacked, kDirect, kTurned };

// Packed and direct: where a lane finds its tile's operands, the tile's (packed)
// or its first row's bytes, wave-uniform, and the lane's offsets from there. The
// next block's are loaded while one is used.
struct ActAt {
  const char* base;
  int nt, step;  // step: bytes to the next block
  uint32_t q, bs, d;
};

template <int FMT, int SRC>
__device__ __forceinline__ ActAt act_at(const BatchedArgs& a, int tile, int col, int kq) {
  constexpr bool kQ80 = FMT == RV_QF_Q8_0;
  static_assert(SRC == kPacked || (SRC == kDirect && !kQ80), "packed, or public k-quants");
  constexpr int kUnit = kQ80 ? kPacked0Bytes : kPackedKBytes;  // also a public block's size (k-quants)
  const char* acts = reinterpret_cast<const char*>(kQ80 ? a.acts_0 : a.acts_k);
  const int left = a.n_acts - 16 * tile;
  ActAt r;
  r.nt = min(16, left);
  const uint32_t i = (uint32_t)min(col, r.nt - 1);
  r.base = acts + (size_t)tile * 16 * (a.in_dim / 256) * kUnit;
  if constexpr (SRC == kPacked) {
    r.step = r.nt * kUnit;
    r.q = ((uint32_t)kq * r.nt + i) * 16;
    r.bs = 256 * r.nt + ((uint32_t)kq * r.nt + i) * 8;
    r.d = kQ80 ? 256 * r.nt + 32 * i : 288 * r.nt + 4 * i;
  } else {
    r.step = kUnit;
    r.d = i * (uint32_t)(a.in_dim / 256) * kUnit;  // the lane's own row
    r.q = r.d + 4 + 16 * kq;
    r.bs = 0;
  }
  return r;
}

template <int FMT, int SRC>
__device__ __forceinline__ void load_act(Act<FMT>& y, const ActAt& at) {
  const char* base = at.base;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const u32x4a v = *reinterpret_cast<const u32x4a*>(base + (SRC == kPacked ? 64 * c * at.nt : 64 * c) + at.q);
    y.q[c] = i32x4{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
  }
  if constexpr (FMT == RV_QF_Q8_0) {
    const f32x4a d0 = *reinterpret_cast<const f32x4a*>(base + at.d);
    const f32x4a d1 = *reinterpret_cast<const f32x4a*>(base + at.d + 16);
#pragma unroll
    for (int c = 0; c < 4; ++c) y.d[c] = d0[c], y.d[4 + c] = d1[c];
  } else {
    if constexpr (FMT != RV_QF_Q6_K && SRC == kPacked) y.bs = *reinterpret_cast<const f16x4a*>(base + at.bs);
    y.d[0] = *reinterpret_cast<const float*>(base + at.d);
  }
}

// Public blocks (a row's after one another): loaded 256 contiguous bytes of a
// row at a time and turned around through the wave's own LDS, written a block
// ahead of its use and loaded two ahead. In operand order straight from the
// blocks, a row per lane, each load takes 64 cycles or more of the CU's address
// unit, for every 16 weight rows again: 4096 x 2048 weights by 512 activations
// Q4_K 32.8 -> 30.9 us a call, Q8_0 135 -> 40; 8192 x 8192 by 1024 611 -> 390,
// 1908 -> 491. What binds Q4_K and Q6_K then is the LDS, 16 16-byte accesses a
// block and wave, so that two row groups share each block (launch_batched).
constexpr int kTurnRow = 272;  // bytes per row of 256 (16-byte reads of 16 rows and writes of a row: all banks)
constexpr int kTurnD = 12;     // floats per row of the Q8_0 scales (16-byte reads of 16 rows: all banks)
constexpr int kTurnScales = 16 * kTurnRow;
constexpr int kTurnBytes = kTurnScales + 2 * 16 * kTurnD * (int)sizeof(float);  // scales of two groups
template <int FMT>
struct TurnedActs {
  static constexpr bool kQ80 = FMT == RV_QF_Q8_0;
  const char* base;  // the tile's first row (K: the block last loaded of it): wave-uniform
  uint32_t off[4];   // the lane's 16 bytes of rows 4 i + lane / 16
  uint32_t doff[kQ80 ? 2 : 1];
  int lane, nb;
  char* lds;
  u32x4a raw[4];
  float rd[kQ80 ? 2 : 1], dk;

  __device__ __forceinline__ TurnedActs(const BatchedArgs& a, int tile, int lane_, char* lds_) : lane(lane_), lds(lds_) {
    nb = a.in_dim / (kQ80 ? 32 : 256);
    const uint32_t row = (uint32_t)nb * (kQ80 ? sizeof(rv_block_q8_0) : sizeof(rv_block_q8_k));
    const int nt = min(16, a.n_acts - 16 * tile);
    base = reinterpret_cast<const char*>(kQ80 ? a.acts_0 : a.acts_k) + (size_t)tile * 16 * row;
    // Rows past the tile repeat its last. K: chunk lane % 16 of the block. Q8_0:
    // half lane % 2 of block lane / 2 % 8 of the group (its offset by load).
#pragma unroll
    for (int i = 0; i < 4; ++i)
      off[i] = row * min(4 * i + (lane >> 4), nt - 1) + 4 + 16 * (kQ80 ? lane & 1 : lane & 15);
    if constexpr (kQ80) {
#pragma unroll
      for (int i = 0; i < 2; ++i) doff[i] = row * min(8 * i + (lane >> 3), nt - 1);
    } else {
      doff[0] = row * min(lane & 15, nt - 1);
    }
    load(0);
    if constexpr (kQ80) {
      put(0, raw, rd);
      load(1);
    } else {  // the first two in flight together
      u32x4a first[4];
      const float fd[1] = {rd[0]};
#pragma unroll
      for (int i = 0; i < 4; ++i) first[i] = raw[i];
      if (nb > 1) base += sizeof(rv_block_q8_k);
      load(1);
      put(0, first, fd);
    }
  }
  // Block b (K: the one at base) of the tile's rows; Q8_0: blocks 8 b .. + 7,
  // those past the row its last.
  __device__ __forceinline__ void load(int b) {
    uint32_t at = 0;
    if constexpr (kQ80) at = (uint32_t)min(8 * b + ((lane >> 1) & 7), nb - 1) * sizeof(rv_block_q8_0);
#pragma unroll
    for (int i = 0; i < 4; ++i) raw[i] = *reinterpret_cast<const u32x4a*>(base + (off[i] + at));
    if constexpr (kQ80) {
      const uint32_t dat = (uint32_t)min(8 * b + (lane & 7), nb - 1) * sizeof(rv_block_q8_0);
#pragma unroll
      for (int i = 0; i < 2; ++i) rd[i] = *reinterpret_cast<const float*>(base + (doff[i] + dat));
    } else {
      rd[0] = *reinterpret_cast<const float*>(base + doff[0]);
    }
  }
  __device__ __forceinline__ float* dd(int k) const {
    return reinterpret_cast<float*>(lds + kTurnScales) + 16 * kTurnD * (k & 1);
  }
  __device__ __forceinline__ void put(int k, const u32x4a (&w)[4], const float (&wd)[kQ80 ? 2 : 1]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * i + (lane >> 4);
      if constexpr (kQ80) {  // as build0 lays the weights
        const int c = (lane >> 1) & 7, at = 4 * (c >> 1) + 2 * (lane & 1);
        *reinterpret_cast<i32x2*>(lds + kTurnRow * r + 16 * at + 8 * (c & 1)) = i32x2{(int)w[i][0], (int)w[i][1]};
        *reinterpret_cast<i32x2*>(lds + kTurnRow * r + 16 * at + 16 + 8 * (c & 1)) = i32x2{(int)w[i][2], (int)w[i][3]};
      } else {
        *reinterpret_cast<i32x4*>(lds + kTurnRow * r + 16 * (lane & 15)) =
            i32x4{(int)w[i][0], (int)w[i][1], (int)w[i][2], (int)w[i][3]};
      }
    }
    if constexpr (kQ80) {
#pragma unroll
      for (int i = 0; i < 2; ++i) dd(k)[kTurnD * (8 * i + (lane >> 3)) + (lane & 7)] = wd[i];
    } else {
      dk = wd[0];
    }
  }
  // Block b of n into y; b % 2 == k % 2.
  __device__ __forceinline__ void next(Act<FMT>& y, int k, int b, int n) {
    const int col = lane & 15, kq = lane >> 4;
    wave_lds_order();
#pragma unroll
    for (int c = 0; c < 4; ++c) y.q[c] = *reinterpret_cast<const i32x4*>(lds + kTurnRow * col + 64 * c + 16 * kq);
    if constexpr (!kQ80) y.d[0] = dk;
    wave_lds_order();  // read before the next block goes over it
    put(k + 1, raw, rd);
    if (!kQ80 && b + 2 < n) base += sizeof(rv_block_q8_k);
    load(b + 2);
  }
  // Q8_0: the four scales c .. + 3 of the group last taken (which was k).
  __device__ __forceinline__ f32x4 scales(int k, int c) const {
    return *reinterpret_cast<const f32x4*>(dd(k) + kTurnD * (lane & 15) + c);
  }
};

struct NoTurn {
  __device__ __forceinline__ NoTurn(const BatchedArgs&, int, int, char*) {}
};
template <int FMT, int SRC>
using Turned = std::conditional_t<SRC == kTurned, TurnedActs<FMT>, NoTurn>;

// The sums of the lane's 16 values of each chunk (carried by the packed
// layout, formed here from public blocks).
template <int FMT, int SRC>
__device__ __forceinline__ f16x4 act_sums(const Act<FMT>& y) {
  if constexpr (SRC == kPacked) return y.bs;
  f16x4 r;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    int s = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) s = __builtin_amdgcn_sdot4(y.q[c][k], 0x01010101, s, false);
    r[c] = (_Float16)(float)s;
  }
  return r;
}

// Stores rows i .. i + 3 (those below n_rows) of activation ao.
__device__ __forceinline__ void store4(const BatchedArgs& a, const BatchedSeg& sg, int i, int ao, f32x4 v) {
  if (ao >= a.n_acts) return;
  if (a.transposed) {
    float* o = sg.out + (size_t)ao * sg.ldo + i;
    if (i + 3 < sg.n_rows) {
      if (a.accumulate) v = *reinterpret_cast<const f32x4a*>(o) + v;
      *reinterpret_cast<f32x4a*>(o) = v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (i + r < sg.n_rows) o[r] = a.accumulate ? o[r] + v[r] : v[r];
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (i + r < sg.n_rows) {
        float* o = sg.out + (size_t)(i + r) * sg.ldo + ao;
        *o = a.accumulate ? *o + v[r] : v[r];
      }
  }
}

// ---- the products ----------------------------------------------------------------

// A k-quant segment's rows 16 RG rg .. against activation tile kW ag + wave of
// each wave. RG row groups share each block's operands; the planes' KC slots
// then hold KC / RG blocks of each.
template <int FMT, int SRC, int RG>
__device__ __forceinline__ void kq_body(const BatchedArgs& a, const BatchedSeg& sg, int rg, int ag, Planes& pl,
                                        char* turn) {
#pragma clang fp contract(off)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, kq = lane >> 4;
  const int nb = a.in_dim / 256, n_tiles = (a.n_acts + 15) / 16, tile = ag * kW + wave;
  // Unpacking: piece tid % 8 (eight lanes read a block's 128 quant bytes) of
  // row (tid / 8) % 16 and slot tid / 128 of the planes: row group slot % RG
  // and block slot / RG of the chunk. The rows are taken in
  // the order that gives neighbouring groups of eight lanes the two halves of
  // the banks: Q6_K's pieces fill chunks 0-3 and 8-11 of a row (swizzled: the
  // others of row ^ 4), the others' 0, 1, 4, 5, .. (of row ^ 2). Rows past the
  // range re-read its last (their outputs are not stored), blocks past the
  // row its last.
  constexpr int KB = KC / RG;
  const int bp = tid & 7, i8 = (tid >> 3) & 15, slot = wave >> 1, bk = slot / RG;
  const int br = FMT == RV_QF_Q6_K ? ((i8 & 1) << 2) | ((i8 & 6) >> 1) | (i8 & 8)
                                   : ((i8 & 1) << 1) | ((i8 & 2) >> 1) | (i8 & 12);
  const uint8_t* wrow = sg.w + (size_t)(sg.row_lo + min(kR * (RG * rg + slot % RG) + br, sg.n_rows - 1)) * sg.row_bytes;
  Raw<FMT> raw;
  load_raw<FMT>(raw, wrow, nb, bk, bp);
  Turned<FMT, SRC> turned(a, min(tile, n_tiles - 1), lane, turn + wave * kTurnBytes);
  ActAt at;
  Act<FMT> act[SRC == kTurned ? 1 : 2];
  if constexpr (SRC != kTurned) {
    at = act_at<FMT, SRC>(a, min(tile, n_tiles - 1), col, kq);
    load_act<FMT, SRC>(act[0], at);
  }
  f32x4 sumf[RG]{};
  for (int b0 = 0; b0 < nb; b0 += KB) {
    if (b0) __syncthreads();  // every wave is done with the previous chunk's planes
    build<FMT>(raw, pl, br, slot, bp);
    load_raw<FMT>(raw, wrow, nb, b0 + KB + bk, bp);
    __syncthreads();
    if (tile >= n_tiles) continue;  // wave-uniform: a wave without activations only unpacks
    f16x4 bs;
#pragma unroll
    for (int p = 0; p < KC; ++p) {  // the planes' slots
      const int k = p / RG, g = p % RG;
      if (g == 0 && b0 + k >= nb) break;
      if (g == 0) {
        if constexpr (SRC == kTurned) {
          turned.next(act[0], k, b0 + k, nb);
        } else {
          if (b0 + k + 1 < nb) at.base += at.step;  // the last block is loaded again, unused
          load_act<FMT, SRC>(act[(k + 1) & 1], at);
        }
      }
      const Act<FMT>& y = act[SRC == kTurned ? 0 : k & 1];
      i32x4 hi{}, lo{};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const i32x4 wh = *reinterpret_cast<const i32x4*>(&pl.p[p][0][chunk_at(col, 4 * c + kq)]);
        const i32x4 wl = *reinterpret_cast<const i32x4*>(&pl.p[p][1][chunk_at(col, 4 * c + kq)]);
        hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, y.q[c], hi, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, y.q[c], lo, 0, 0, 0);
      }
      const f32x4 dw = *reinterpret_cast<const f32x4*>(&pl.d[p][0][4 * kq]);
      const float da = y.d[0];
      if constexpr (FMT == RV_QF_Q6_K) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int sumi = 64 * hi[r] + lo[r];
          sumf[g][r] += dw[r] * da * (float)sumi;
        }
      } else {
        const f32x4 dm = *reinterpret_cast<const f32x4*>(&pl.d[p][1][4 * kq]);
        const f16x4 m4 = *reinterpret_cast<const f16x4*>(&pl.mins[p][col][4 * (kq >> 1)]);
        if (g == 0) bs = act_sums<FMT, SRC>(y);
        const f32x4 mins = __builtin_amdgcn_mfma_f32_16x16x16f16(m4, bs, f32x4{}, 0, 0, 0);
        int extra = 0;
        if constexpr (FMT == RV_QF_Q5_K) {
          static_assert(RG == 1, "Q5_K takes one row group");
          const f16x4 one = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
          extra = 1152 * (int)__builtin_amdgcn_mfma_f32_16x16x16f16(one, bs, f32x4{}, 0, 0, 0)[0];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int sumi = 8 * hi[r] + lo[r] + extra;
          const float d = dw[r] * da, dmin = dm[r] * da;
          sumf[g][r] += d * (float)sumi - dmin * mins[r];
        }
      }
      if constexpr (RG == 2) __builtin_amdgcn_sched_barrier(0);
    }
  }
  store4(a, sg, kR * RG * rg + 4 * kq, 16 * tile + col, sumf[0]);
  if constexpr (RG == 2) store4(a, sg, kR * (RG * rg + 1) + 4 * kq, 16 * tile + col, sumf[1]);
}

// A Q8_0 segment's 16 rows 16 rg .. against one activation tile per wave.
template <int SRC>
__device__ __forceinline__ void q80_body(const BatchedArgs& a, const BatchedSeg& sg, int rg, int ag, Planes0& pl,
                                         char* turn) {
#pragma clang fp contract(off)
  constexpr int FMT = RV_QF_Q8_0, NI = kR * KC * 32 / (64 * kW);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, kq = lane >> 4;
  const int nb = a.in_dim / 32, steps = (nb + 7) / 8, n_tiles = (a.n_acts + 15) / 16, tile = ag * kW + wave;
  // Piece tid % 32 of group (tid / 32) % KC of row tid / 128 + 4 u.
  const int bp = tid & 31, bk = (tid >> 5) % KC, br = tid / (32 * KC);
  const uint8_t* wrow[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u)
    wrow[u] = sg.w + (size_t)(sg.row_lo + min(kR * rg + br + kR / NI * u, sg.n_rows - 1)) * sg.row_bytes;
  Raw<FMT> raw[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) load_raw<FMT>(raw[u], wrow[u], nb, bk, bp);
  Turned<FMT, SRC> turned(a, min(tile, n_tiles - 1), lane, turn + wave * kTurnBytes);
  ActAt at;
  Act<FMT> act[SRC == kTurned ? 1 : 2];
  if constexpr (SRC != kTurned) {
    at = act_at<FMT, SRC>(a, min(tile, n_tiles - 1), col, kq);
    load_act<FMT, SRC>(act[0], at);
  }
  f32x4 sumf{};
  for (int s0 = 0; s0 < steps; s0 += KC) {
    if (s0) __syncthreads();
#pragma unroll
    for (int u = 0; u < NI; ++u) build0(raw[u], pl, br + kR / NI * u, bk, bp);
#pragma unroll
    for (int u = 0; u < NI; ++u) load_raw<FMT>(raw[u], wrow[u], nb, s0 + KC + bk, bp);
    __syncthreads();
    if (tile >= n_tiles) continue;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      const int s = s0 + k;
      if (s >= steps) break;
      if constexpr (SRC == kTurned) {
        turned.next(act[0], k, s, steps);
      } else {
        if (s + 1 < steps) at.base += at.step;
        load_act<FMT, SRC>(act[(k + 1) & 1], at);
      }
      const Act<FMT>& y = act[SRC == kTurned ? 0 : k & 1];
      const int nblk = min(8, nb - 8 * s);
      f32x4 dy;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if constexpr (SRC == kTurned) {
          if (c % 4 == 0) dy = turned.scales(k, c);
        } else {
          dy[c % 4] = y.d[c];
        }
        const i32x2 w2 = *reinterpret_cast<const i32x2*>(&pl.p[k][chunk_at(col, 4 * (c >> 1) + kq) + 8 * (c & 1)]);
        const i32x2 y2 = {y.q[c >> 1][2 * (c & 1)], y.q[c >> 1][2 * (c & 1) + 1]};
        const i32x4 acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, w2), __builtin_bit_cast(long, y2),
                                                                i32x4{}, 0, 0, 0);
        const f32x4 dw = *reinterpret_cast<const f32x4*>(&pl.d[k][c][4 * kq]);
        if (SRC == kPacked || c < nblk) {
#pragma unroll
          for (int r = 0; r < 4; ++r) sumf[r] += (float)acc[r] * (dw[r] * dy[c % 4]);
        }
      }
    }
  }
  store4(a, sg, kR * rg + 4 * kq, 16 * tile + col, sumf);
}

template <int SRC, int RG>
__global__ __launch_bounds__(64 * kW) __attribute__((amdgpu_waves_per_eu(4))) void batched_kernel(BatchedArgs a) {
  constexpr int kPlaneBytes = sizeof(Planes) > sizeof(Planes0) ? sizeof(Planes) : sizeof(Planes0);
  static_assert(kPlaneBytes % 16 == 0 && kTurnBytes % 16 == 0, "16-byte LDS accesses");
  __shared__ __attribute__((aligned(16))) char lds[kPlaneBytes + (SRC == kTurned ? kW * kTurnBytes : 0)];
  int b = (int)blockIdx.x, si = 0;
  while (si + 1 < a.n_seg && b >= a.seg[si].blocks) b -= a.seg[si++].blocks;
  const BatchedSeg& sg = a.seg[si];
  // Row group rg and activation group ag: a row group's activation groups
  // take block indices equal mod 8, so they read its weights through one
  // XCD's L2.
  const int n_ag = a.n_ag, q8 = b / (8 * n_ag), rem = b % (8 * n_ag);
  const int rg = 8 * q8 + rem % 8, ag = rem / 8;
  if (rg >= sg.n_rg) return;  // uniform: the last eight row groups may be partial
  auto& pl = *reinterpret_cast<Planes*>(lds);
  char* const turn = lds + kPlaneBytes;  // each wave's activations (turned)
  // (The launch takes Q8_0 and Q5_K to the instantiations that have them.)
  switch (sg.fmt) {
    case RV_QF_Q8_0:
      if constexpr (RG == 1 && SRC != kDirect) q80_body<SRC>(a, sg, rg, ag, *reinterpret_cast<Planes0*>(lds), turn);
      return;
    case RV_QF_Q4_K: return kq_body<RV_QF_Q4_K, SRC, RG>(a, sg, rg, ag, pl, turn);
    case RV_QF_Q5_K:
      if constexpr (RG == 1) kq_body<RV_QF_Q5_K, SRC, RG>(a, sg, rg, ag, pl, turn);
      return;
    default: return kq_body<RV_QF_Q6_K, SRC, RG>(a, sg, rg, ag, pl, turn);
  }
}

}  // namespace

HipStatus launch_batched(BatchedArgs a, bool packed, hipStream_t s) {
  HipStatus st;
  if (a.n_acts == 0 || a.in_dim == 0) return st;
  unsigned grid = 0;
  a.n_ag = (a.n_acts + 16 * kW - 1) / (16 * kW);
  // Public blocks (one segment). With up to two working waves a CU the turn's
  // latency shows, and k-quants load in operand order. Turned vs not, us per
  // call: Q4_K 4096 x 2048 weights, 1 activation 7.7 vs 7.2, 32 (512 waves) 8.3
  // vs 8.0, 128 11.3 vs 12.0; 8192 x 8192, 16 (512) 23.6 vs 23.0, 32 27.6 vs 30.8.
  // Q8_0's scattered 8-byte loads lose there too (4096 x 2048, 1 12.2 vs 13.1).
  const BatchedSeg& s0 = a.seg[0];
  const long waves = (long)((s0.n_rows + kR - 1) / kR) * ((a.n_acts + 15) / 16);
  const bool direct = !packed && s0.fmt != RV_QF_Q8_0 && waves <= 512;
  // Otherwise Q4_K and Q6_K take two row groups a workgroup once one would put
  // two workgroups on a CU, with at least half of the waves at work. One vs
  // two: Q4_K 4096 x 2048, 128 activations (256 workgroups) 11.3 vs 14.3, 256
  // 17.0 vs 14.8, 512 30.9 vs 23.2; 8192 x 8192, 32 27.6 vs 30.0, 64 34.2 either
  // way, 1024 390 vs 283; Q6_K 410 vs 297. (Q5_K's registers do not allow it;
  // Q8_0 is bound by its float work.)
  const long pairs = (long)((s0.n_rows + 2 * kR - 1) / (2 * kR)) * a.n_ag;
  const bool two = !packed && !direct && (s0.fmt == RV_QF_Q4_K || s0.fmt == RV_QF_Q6_K) && pairs > 128 && a.n_acts >= 64;
  const int rows = two ? 2 * kR : kR;
  for (int i = 0; i < a.n_seg; ++i) {
    BatchedSeg& g = a.seg[i];
    g.n_rg = (g.n_rows + rows - 1) / rows;
    g.blocks = (g.n_rg + 7) / 8 * 8 * a.n_ag;
    grid += (unsigned)g.blocks;
  }
  if (grid == 0) return st;
#define RV_BATCHED(SRC, RG) hipLaunchKernelGGL((batched_kernel<SRC, RG>), dim3(grid), dim3(64 * kW), 0, s, a)
  if (packed)
    RV_BATCHED(kPacked, 1);
  else if (direct)
    RV_BATCHED(kDirect, 1);
  else if (two)
    RV_BATCHED(kTurned, 2);
  else
    RV_BATCHED(kTurned, 1);
#undef RV_BATCHED
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "batched gemv launch";
  return st;
}

}  // namespace rv
