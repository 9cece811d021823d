// rv_quant.hip — the quantized projections either side of attention on gfx950:
// Q8_K / Q8_0 activation quantizers and the k-quant / Q8_0 GEMVs.
//
// Replaces quantize_row_q8_k / quantize_row_q8_0
// (crates/core/src/kernels/quants/quantize.rs:37-106) and the row-range GEMVs
// gemv_q8_k_rows / gemv_q8_0_rows (kernels/gemv.rs:296-615) over the scalar
// dots vec_dot_{q4_k,q5_k,q6_k}_q8_k / vec_dot_q8_0_q8_0 (quants/dot.rs),
// as called at model/forward.rs:2574-2646.
//
// Results are bit-identical to the reference's scalar kernels:
//  - quantizers: one wave per 256-value Q8_K block (the first value of
//    largest magnitude found by a lane-ordered wave reduction, RNE rounding,
//    the scalar code's f32 divisions) and 32 lanes per Q8_0 block;
//  - GEMVs: one wave per output row. Lanes split each super-block's
//    sub-blocks and form the integer sub-block sums with v_dot4_i32_i8
//    (exact, in any order), a block's integer totals come from an exact
//    8-lane reduction, the block's float contribution is the scalar dot's
//    expression, and the row's sum adds the blocks in order.
// The GEMVs stream each weight byte once (HBM-bound); activations are
// re-read per row from L2.
#include "rv_device.hpp"
#include "rv_internal.hpp"
#include "rv_quant.hpp"

namespace rv {
namespace {

__device__ __forceinline__ float f16_bits_to_f32(uint32_t bits) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits & 0xFFFFu));
}

// 32 bytes at a 2-byte-aligned address as raw dwords: aligned-down reads plus
// a 2-byte tail, reading nothing outside [a, a + 32) except the two bytes
// before `a` (which the callers' layouts guarantee belong to the same block).
// fix32 realigns them, so the loads can be issued ahead of their use.
struct Raw32 {
  uint32_t e[8];
  uint32_t tail, odd;
};
__device__ __forceinline__ Raw32 raw32_a2(const uint8_t* a) {
  Raw32 r;
  r.odd = (uint32_t)(uintptr_t)a & 2;
  const uint32_t* p = reinterpret_cast<const uint32_t*>(a - r.odd);
#pragma unroll
  for (int k = 0; k < 8; ++k) r.e[k] = p[k];
  r.tail = *reinterpret_cast<const uint16_t*>(a + 30);
  return r;
}
__device__ __forceinline__ void fix32(const Raw32& r, uint32_t (&w)[8]) {
#pragma unroll
  for (int k = 0; k < 7; ++k) w[k] = __builtin_amdgcn_alignbyte(r.e[k + 1], r.e[k], r.odd);
  w[7] = r.odd ? (r.e[7] >> 16) | (r.tail << 16) : r.e[7];
}

// Sum over the 8 lanes of an aligned lane group (exact for integers).
__device__ __forceinline__ int sum8_lanes(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_XOR1, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, DPP_QUAD_XOR2, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_HALF_MIRROR, 0xF, 0xF, false);
  return v;
}

__device__ __forceinline__ int dot4(uint32_t w, int a, int acc) {
  return __builtin_amdgcn_sdot4((int)w, a, acc, false);
}

__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// get_scale_min_k4 (quants/blocks.rs:158-167) from the 12 scale bytes as
// three little-endian dwords.
__device__ __forceinline__ void scale_min_k4(int j, const uint32_t (&s)[3], int& sc, int& m) {
  auto byte = [&](int i) { return (int)((s[i >> 2] >> (8 * (i & 3))) & 0xFF); };
  if (j < 4) {
    sc = byte(j) & 63;
    m = byte(j + 4) & 63;
  } else {
    sc = (byte(j + 4) & 0xF) | ((byte(j - 4) >> 6) << 4);
    m = (byte(j + 4) >> 4) | ((byte(j) >> 6) << 4);
  }
}

// 16 bytes at a 4-byte-aligned global address (global_load_dwordx4 needs
// only dword alignment).
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));

// Lane j's view of one Q8_K activation block: qs[32j .. 32j+31] packed 4
// per int, the scale d, and bsums[2j], bsums[2j+1].
struct ActK {
  int a[8];
  float d;
  int bs_lo, bs_hi;
};

__device__ __forceinline__ ActK act_from_block(const rv_block_q8_k* __restrict__ y, int j) {
  ActK r;
  const int* q = reinterpret_cast<const int*>(y->qs + 32 * j);
#pragma unroll
  for (int k = 0; k < 8; ++k) r.a[k] = q[k];
  const uint32_t bs = *reinterpret_cast<const uint32_t*>(y->bsums + 2 * j);
  r.bs_lo = (int)(int16_t)(bs & 0xFFFFu);
  r.bs_hi = (int)(int16_t)(bs >> 16);
  r.d = y->d;
  return r;
}

// What a lane loads of its weight block: k-quants, lane j of the block's 8;
// Q8_0, the whole 32-weight block.
template <int FMT>
struct BlockRaw;
template <>
struct BlockRaw<RV_QF_Q4_K> {
  u32x4a hdr, q[2];
};
template <>
struct BlockRaw<RV_QF_Q5_K> {
  u32x4a hdr, q[2], h[2];
};
template <>
struct BlockRaw<RV_QF_Q6_K> {
  Raw32 ql, qh;
  uint32_t sc, d;
};
template <>
struct BlockRaw<RV_QF_Q8_0> {
  Raw32 q;
  uint32_t d;
};

template <int FMT>
__device__ __forceinline__ void load_block(BlockRaw<FMT>& w, const uint8_t* __restrict__ blk, int j) {
  if constexpr (FMT == RV_QF_Q8_0) {
    w.d = *reinterpret_cast<const uint16_t*>(blk);
    w.q = raw32_a2(blk + 2);
  } else if constexpr (FMT == RV_QF_Q6_K) {
    const int half = j >> 2, grp = j & 3;
    w.ql = raw32_a2(blk + 64 * half + 32 * (grp & 1));
    w.qh = raw32_a2(blk + 128 + 32 * half);
    w.sc = *reinterpret_cast<const uint16_t*>(blk + 192 + 2 * j);
    w.d = *reinterpret_cast<const uint16_t*>(blk + 208);
  } else {
    constexpr bool kQ5 = FMT == RV_QF_Q5_K;
    w.hdr = *reinterpret_cast<const u32x4a*>(blk);
    const u32x4a* qp = reinterpret_cast<const u32x4a*>(blk + (kQ5 ? 48 : 16) + 32 * (j >> 1));
    w.q[0] = qp[0], w.q[1] = qp[1];
    if constexpr (kQ5) {
      const u32x4a* hp = reinterpret_cast<const u32x4a*>(blk + 16);
      w.h[0] = hp[0], w.h[1] = hp[1];
    }
  }
}

// One super-block's float contribution for the k-quants, computed by the 8
// lanes of a group, lane j owning sub-block j (Q4_K/Q5_K: 32 weights) or
// the two 16-weight sub-blocks 2j, 2j+1 (Q6_K); every lane of the group
// returns the same value.
//  - Q4_K / Q5_K: k_quant_affine_block with the expansions (dot.rs:56-143):
//    d*sumi - dmin*sumi_mins, d = f16(d)*y.d, dmin = f16(dmin)*y.d.
//  - Q6_K: vec_dot_q6_k_q8_k (dot.rs:150-179): lane j = 4 half + group holds
//    weights 32j .. 32j+31: ql nibbles (byte l + 32 (group & 1) of the half,
//    high nibble for groups 2, 3) and two qh bits (2 group). The stored values
//    are q + 32 in 0..63; sum (q+32)a - 32 sum a, with sum a the activation
//    bsums.
template <int FMT>
__device__ __forceinline__ float kq_block(const BlockRaw<FMT>& w, const ActK& y, int j) {
#pragma clang fp contract(off)
  if constexpr (FMT == RV_QF_Q6_K) {
    const int grp = j & 3;
    uint32_t ql[8], qh[8];
    fix32(w.ql, ql);
    fix32(w.qh, qh);
    int lo = 0, hi = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t nib = (grp >> 1) ? (ql[k] >> 4) & 0x0F0F0F0Fu : ql[k] & 0x0F0F0F0Fu;
      const uint32_t v = nib | (((qh[k] >> (2 * grp)) & 0x03030303u) << 4);
      if (k < 4)
        lo = dot4(v, y.a[k], lo);
      else
        hi = dot4(v, y.a[k], hi);
    }
    lo -= 32 * y.bs_lo;
    hi -= 32 * y.bs_hi;
    const int sc_lo = (int)(int8_t)(w.sc & 0xFF), sc_hi = (int)(int8_t)(w.sc >> 8);
    const int sumi = sum8_lanes(sc_lo * lo + sc_hi * hi);
    const float d = f16_bits_to_f32(w.d);
    return d * y.d * (float)sumi;
  } else {
    const uint32_t s[3] = {w.hdr[1], w.hdr[2], w.hdr[3]};
    int acc = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint32_t v = (w.q[k >> 2][k & 3] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
      if constexpr (FMT == RV_QF_Q5_K) v |= ((w.h[k >> 2][k & 3] >> j) & 0x01010101u) << 4;
      acc = dot4(v, y.a[k], acc);
    }
    int sc, m;
    scale_min_k4(j, s, sc, m);
    const int sumi = sum8_lanes(sc * acc);
    const int sumi_mins = sum8_lanes(m * (y.bs_lo + y.bs_hi));
    const float d = f16_bits_to_f32(w.hdr[0]) * y.d;
    const float dmin = f16_bits_to_f32(w.hdr[0] >> 16) * y.d;
    return d * (float)sumi - dmin * (float)sumi_mins;
  }
}

// One row against its activation blocks (global memory or LDS), every lane
// returning the row's sum, added in block order. k-quants: 8 super-blocks per
// pass (lane group b); Q8_0 (vec_dot_q8_0_q8_0, dot.rs:185-201): lane per
// 32-weight block, 64 per pass, sumf += sumi * (f16(d) * y.d). The first P
// passes' weights come in `pre` (row_prefetch), loaded ahead.
template <int FMT>
constexpr int kPassBlocks = FMT == RV_QF_Q8_0 ? 64 : 8;
template <int FMT>
constexpr int kBlockBytes = FMT == RV_QF_Q4_K ? 144 : FMT == RV_QF_Q5_K ? 176 : FMT == RV_QF_Q6_K ? 210 : 34;

template <int FMT>
__device__ __forceinline__ void load_pass(BlockRaw<FMT>& w, const uint8_t* __restrict__ row, int nb, int b0, int lane) {
  // Groups past the row re-read its last block (unused).
  const int b = min(b0 + (FMT == RV_QF_Q8_0 ? lane : lane >> 3), nb - 1);
  load_block<FMT>(w, row + (size_t)b * kBlockBytes<FMT>, lane & 7);
}

template <int FMT>
__device__ __forceinline__ float pass_value(const BlockRaw<FMT>& w, int nb, int b0, const void* __restrict__ acts,
                                            int lane) {
#pragma clang fp contract(off)
  if constexpr (FMT == RV_QF_Q8_0) {
    const rv_block_q8_0* y = reinterpret_cast<const rv_block_q8_0*>(acts) + min(b0 + lane, nb - 1);
    uint32_t q[8];
    fix32(w.q, q);
    const int* a = reinterpret_cast<const int*>(y->qs);
    int s = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) s = dot4(q[k], a[k], s);
    return (float)s * (f16_bits_to_f32(w.d) * y->d);
  } else {
    const rv_block_q8_k* y = reinterpret_cast<const rv_block_q8_k*>(acts) + min(b0 + (lane >> 3), nb - 1);
    return kq_block<FMT>(w, act_from_block(y, lane & 7), lane & 7);
  }
}

template <int FMT>
__device__ __forceinline__ float add_pass(float sumf, float c, int nb, int b0) {
  constexpr int N = kPassBlocks<FMT>, S = 64 / N;
  if (b0 + N <= nb) {
#pragma unroll
    for (int k = 0; k < N; ++k) sumf += lane_f(c, S * k);
  } else {
    for (int k = 0; k < nb - b0; ++k) sumf += lane_f(c, S * k);
  }
  return sumf;
}

template <int FMT, int P>
__device__ __forceinline__ float row_sum(const BlockRaw<FMT> (&pre)[P], const uint8_t* __restrict__ row, int nb,
                                         const void* __restrict__ acts, int lane) {
  constexpr int N = kPassBlocks<FMT>;
  float sumf = 0.f;
#pragma unroll
  for (int p = 0; p < P; ++p)
    if (N * p < nb) sumf = add_pass<FMT>(sumf, pass_value<FMT>(pre[p], nb, N * p, acts, lane), nb, N * p);
  for (int b0 = N * P; b0 < nb; b0 += N) {
    BlockRaw<FMT> w;
    load_pass<FMT>(w, row, nb, b0, lane);
    sumf = add_pass<FMT>(sumf, pass_value<FMT>(w, nb, b0, acts, lane), nb, b0);
  }
  return sumf;
}

template <int FMT, int P>
__device__ __forceinline__ void row_prefetch(BlockRaw<FMT> (&pre)[P], const uint8_t* __restrict__ row, int nb,
                                             int lane) {
#pragma unroll
  for (int p = 0; p < P; ++p) load_pass<FMT>(pre[p], row, nb, kPassBlocks<FMT> * p, lane);
}

// quantize_row_q8_k (quantize.rs:71-106) of one block by one wave, lane l
// holding values 4l .. 4l+3: the first value of largest magnitude (the
// maximum over the wave, then the lowest lane that holds it and that lane's
// first such value; NaN never wins, as `av > amax` never takes it), RNE
// rounding, the clamp, the sums of 16 values and the scalar code's f32
// divisions. A block whose maximum is 0 is all zeros.
struct Q8KLane {
  uint32_t q;  // the lane's four quants
  int sum16;   // the sum over its aligned group of four lanes (16 values)
  float d;
};
__device__ __forceinline__ Q8KLane quantize_lane_q8_k(const float (&v)[4]) {
  float amax = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(v[e]));
  amax = swap_max<32>(swap_max<16>(group_max<16>(amax)));
  Q8KLane r{0u, 0, 0.f};
  if (amax == 0.f) return r;  // wave-uniform
  float first = 0.f;
  bool any = false;
#pragma unroll
  for (int e = 3; e >= 0; --e)
    if (fabsf(v[e]) == amax) {
      first = v[e];
      any = true;
    }
  const float mx = lane_f(first, __builtin_ctzll(__ballot(any)));
  const float iscale = -127.f / mx;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = min(max((int)__builtin_rintf(iscale * v[e]), -128), 127);
    r.q |= (uint32_t)(n & 0xFF) << (8 * e);
    r.sum16 += n;
  }
  r.sum16 += __builtin_amdgcn_update_dpp(0, r.sum16, DPP_QUAD_XOR1, 0xF, 0xF, false);
  r.sum16 += __builtin_amdgcn_update_dpp(0, r.sum16, DPP_QUAD_XOR2, 0xF, 0xF, false);
  r.d = 1.f / iscale;
  return r;
}

__device__ __forceinline__ void store_q8_k(const Q8KLane& r, rv_block_q8_k* blk, int lane) {
  *reinterpret_cast<uint32_t*>(blk->qs + 4 * lane) = r.q;
  if ((lane & 3) == 0) blk->bsums[lane >> 2] = (int16_t)r.sum16;
  if (lane == 0) blk->d = r.d;
}

__device__ __forceinline__ void quantize_block_q8_k(const float* __restrict__ xs, rv_block_q8_k* blk, int lane) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = xs[4 * lane + e];
  store_q8_k(quantize_lane_q8_k(v), blk, lane);
}

// quantize_row_q8_0 (quantize.rs:37-55) of one block by the 32 lanes of a
// half-wave, lane i holding value i: d = amax/127, q = round(v/d) half away
// from zero, d stored f16-rounded.
__device__ __forceinline__ void quantize_block_q8_0(const float* __restrict__ xs, rv_block_q8_0* blk, int i) {
  const float v = xs[i];
  float amax = fabsf(v);
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  const float d = amax / 127.f;
  const float id = d != 0.f ? 1.f / d : 0.f;
  blk->qs[i] = (int8_t)roundf(v * id);
  if (i == 0) blk->d = (float)(_Float16)d;
}

// The same of one block by an aligned group of 8 lanes, lane i holding
// values 4i .. 4i+3.
struct Q80Lane {
  uint32_t q;
  float d;
};
__device__ __forceinline__ Q80Lane quantize_lane_q8_0(const float (&v)[4]) {
  float amax = fabsf(v[0]);
#pragma unroll
  for (int e = 1; e < 4; ++e) amax = fmaxf(amax, fabsf(v[e]));
  amax = group_max<8>(amax);
  const float d = amax / 127.f;
  const float id = d != 0.f ? 1.f / d : 0.f;
  Q80Lane r{0u, (float)(_Float16)d};
#pragma unroll
  for (int e = 0; e < 4; ++e) r.q |= (uint32_t)(uint8_t)(int8_t)roundf(v[e] * id) << (8 * e);
  return r;
}

__global__ __launch_bounds__(256) void quantize_q8_k_kernel(const float* __restrict__ x, rv_block_q8_k* __restrict__ out,
                                                           int n_blocks) {
  const int b = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= n_blocks) return;  // wave-uniform
  quantize_block_q8_k(x + (size_t)b * 256, out + b, threadIdx.x & 63);
}

__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float* __restrict__ x, rv_block_q8_0* __restrict__ out,
                                                           int n_blocks) {
  const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int b = t >> 5;
  if (b >= n_blocks) return;  // whole 32-lane halves
  quantize_block_q8_0(x + (size_t)b * 32, out + b, t & 31);
}

// Both forms in one launch: wave b quantizes 256-value block b to Q8_K and
// its eight 32-value blocks to Q8_0 (each half-wave four of them), with the
// same per-block code as the two kernels above, so the same bytes.
__global__ __launch_bounds__(256) void quantize_both_kernel(const float* __restrict__ x, rv_block_q8_k* __restrict__ ok,
                                                            rv_block_q8_0* __restrict__ o0, int n_blocks) {
  const int b = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= n_blocks) return;  // wave-uniform
  const int lane = threadIdx.x & 63;
  const float* xb = x + (size_t)b * 256;
  quantize_block_q8_k(xb, ok + b, lane);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int sb = 2 * i + (lane >> 5);
    quantize_block_q8_0(xb + 32 * sb, o0 + (size_t)b * 8 + sb, lane & 31);
  }
}

constexpr int kRowsPerWG = 4;

// out[i] = row(row_lo + i) . acts for i < n_rows, acts quantized blocks in
// global memory; one wave per row.
template <int FMT>
__global__ __launch_bounds__(64 * kRowsPerWG) void gemv_rows_kernel(const uint8_t* __restrict__ w, size_t row_bytes,
                                                                    int nb, const void* __restrict__ acts, long row_lo,
                                                                    int n_rows, float* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int i = (int)blockIdx.x * kRowsPerWG + (threadIdx.x >> 6);
  if (i >= n_rows) return;  // wave-uniform
  const uint8_t* row = w + (size_t)(row_lo + i) * row_bytes;
  BlockRaw<FMT> pre[1];
  row_prefetch<FMT, 1>(pre, row, nb, lane);
  const float v = row_sum<FMT, 1>(pre, row, nb, acts, lane);
  if (lane == 0) out[i] = v;
}

// Sum over the wave in the order of a shuffle tree over lanes 32, 16, .., 1
// apart, by swaps and DPP (after the first three steps the values repeat every
// eight lanes, so a rotation by 4 reaches the lane 4 apart).
__device__ __forceinline__ double wave_sum_tree_f64(double x) {
  x = swap_sum_f64<32>(x);
  x = swap_sum_f64<16>(x);
  x += dpp_f64<0x128>(x);  // row_ror:8
  x += dpp_f64<0x124>(x);  // row_ror:4
  x += dpp_f64<DPP_QUAD_XOR2>(x);
  x += dpp_f64<DPP_QUAD_XOR1>(x);
  return x;
}

// One workgroup of a fused projection, eight rows of a segment, one per wave:
// the wave's weight row is loaded while the workgroup (normalizes and)
// quantizes x into LDS, NB 256-value blocks of x per wave, in the form that FMT
// takes (the same per-block code as the quantizer kernels, so bit-identical).
// All rows of a workgroup are of one segment, so its waves run one FMT and pass
// the same barriers; a wave past the segment's last row has live false.
template <int FMT, bool NORM, int NB>
__device__ __forceinline__ void fused_rows(const FusedProjArgs& a, const FusedSeg& s, int i, bool live, int wave,
                                           int lane, void* lds, double* red) {
#pragma clang fp contract(off)
  typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int P = FMT != RV_QF_Q8_0 && NB > 1 ? 2 : 1;  // passes whose weights are loaded ahead
  constexpr bool kQ80 = FMT == RV_QF_Q8_0;
  const int nbw = kQ80 ? a.nb0 : a.nbk;
  // The lane's four values of each of the wave's blocks (blocks past the row
  // re-read its last), straight into the quantizers' registers; with the norm
  // also its weight and, for the sum of squares, the values in the summing
  // order (thread t: t, t + 512, ..). They are issued ahead of the weights,
  // since loads retire in order.
  f32x4a xv[NB], wv[NB];
  float xs[NORM ? 4 * NB : 1];
  const int n = a.nbk * 256;
  if constexpr (NORM) {
#pragma unroll
    for (int r = 0; r < 4 * NB; ++r) xs[r] = a.x[min((int)threadIdx.x + 64 * kFusedWaves * r, n - 1)];
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int at = 256 * min(wave + kFusedWaves * u, a.nbk - 1) + 4 * lane;
    xv[u] = *reinterpret_cast<const f32x4a*>(a.x + at);
    if constexpr (NORM) wv[u] = *reinterpret_cast<const f32x4a*>(a.norm_w + at);
  }
  asm volatile("" ::: "memory");
  const uint8_t* row = s.w + (size_t)i * s.row_bytes;
  BlockRaw<FMT> pre[P];
  row_prefetch<FMT, P>(pre, row, nbw, lane);
  float addv = 0.f;  // the residual the output row is added to
  if (s.add && lane == 0) addv = s.add[i];
  const uint32_t gate = a.gate_pos ? *a.gate_pos : 0u;
  asm volatile("" ::: "memory");  // issued before the barriers
  float inv = 1.f;
  if constexpr (NORM) {
    // norm.rs:55-57: x * inv * w left to right in f32.
    double ss = 0.0;
#pragma unroll
    for (int r = 0; r < 4 * NB; ++r) {
      const double v = (int)threadIdx.x + 64 * kFusedWaves * r < n ? (double)xs[r] : 0.0;
      ss += v * v;
    }
    ss = wave_sum_tree_f64(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < kFusedWaves; ++w) tot += red[w];
    inv = (float)(1.0 / sqrt(tot / (double)n + (double)a.eps));
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int b = wave + kFusedWaves * u;
    if (b >= a.nbk) break;  // wave-uniform
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = NORM ? xv[u][e] * inv * wv[u][e] : xv[u][e];
    if constexpr (kQ80) {
      const Q80Lane z = quantize_lane_q8_0(v);
      rv_block_q8_0* blk = reinterpret_cast<rv_block_q8_0*>(lds) + 8 * b + (lane >> 3);
      *reinterpret_cast<uint32_t*>(blk->qs + 4 * (lane & 7)) = z.q;
      if ((lane & 7) == 0) blk->d = z.d;
    } else {
      store_q8_k(quantize_lane_q8_k(v), reinterpret_cast<rv_block_q8_k*>(lds) + b, lane);
    }
  }
  __syncthreads();
  if (!live || gate > a.gate_max) return;  // (the whole grid's decode step was refused: nothing is written)
  const float v = row_sum<FMT, P>(pre, row, nbw, lds, lane);
  if (lane == 0) s.out[i] = s.add ? addv + v : v;
}

// Workgroups of a segment of n rows.
__host__ __device__ constexpr int fused_groups(int n) { return (n + kFusedWaves - 1) / kFusedWaves; }

// NB: 256-value blocks per wave (x holds at most 256 * kFusedWaves * NB values).
template <bool NORM, int NB>
__global__ __launch_bounds__(64 * kFusedWaves) void fused_proj_kernel(FusedProjArgs a) {
  // x as Q8_K blocks or as eight times as many Q8_0 blocks.
  static_assert(sizeof(rv_block_q8_k) >= 8 * sizeof(rv_block_q8_0), "the Q8_0 form fits the Q8_K form's bytes");
  __shared__ rv_block_q8_k lds[kFusedWaves * NB];
  __shared__ double red[kFusedWaves];
  // The wave index as a scalar: the row, its segment and the segment's
  // fields are then wave-uniform, read with scalar loads from the kernel
  // arguments (indexed from a vector register, each was a vector load of
  // the argument segment that every later load waited behind).
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int b = (int)blockIdx.x, sg = 0;
  while (sg + 1 < a.n_seg && b >= fused_groups(a.n_rows[sg])) b -= fused_groups(a.n_rows[sg++]);
  const bool live = b * kFusedWaves + wave < a.n_rows[sg];
  // A wave past the last row quantizes beside the others, on that row's bytes.
  const int i = min(b * kFusedWaves + wave, a.n_rows[sg] - 1);
  const FusedSeg& s = a.seg[sg];
  switch (s.fmt) {  // workgroup-uniform
    case RV_QF_Q4_K: return fused_rows<RV_QF_Q4_K, NORM, NB>(a, s, i, live, wave, lane, lds, red);
    case RV_QF_Q5_K: return fused_rows<RV_QF_Q5_K, NORM, NB>(a, s, i, live, wave, lane, lds, red);
    case RV_QF_Q6_K: return fused_rows<RV_QF_Q6_K, NORM, NB>(a, s, i, live, wave, lane, lds, red);
    default: return fused_rows<RV_QF_Q8_0, NORM, NB>(a, s, i, live, wave, lane, lds, red);
  }
}

// norm.rs:18-58: 1 / sqrt(mean(x^2) + eps) with the squares summed in f64 (here
// per thread, then over lanes and waves in a fixed order, so every thread gets
// the same value), sqrt and reciprocal in f64, rounded once to f32.
__global__ __launch_bounds__(1024) void rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       float eps, int n, float* __restrict__ out) {
  __shared__ double red[16];
  double ss = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const double v = (double)x[i];
    ss += v * v;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  double tot = 0.0;
#pragma unroll
  for (int v = 0; v < 16; ++v) tot += red[v];
  const float inv = (float)(1.0 / sqrt(tot / (double)n + (double)eps));
  for (int j = threadIdx.x; j < n; j += 1024) {
#pragma clang fp contract(off)
    out[j] = x[j] * inv * w[j];
  }
}

// A chunk's rows quantized into the batched GEMVs' operand order (PackedActs,
// rv_quant.hpp), to Q8_K and, with Q0, to Q8_0; with NORM each row is
// RMS-normalized first (norm.rs:18-58). blockIdx.x is the row, wave w takes
// its blocks W blockIdx.y + w, then W * gridDim.y on. The normed row never
// goes through memory: as separate launches (norm, then both quantizations
// with one wave per block and four 6-step shuffle reductions) a 512-row chunk
// of 2048 values took 7.0 + 7.6 us.
template <bool NORM, bool Q0, int W>
__global__ __launch_bounds__(64 * W) void quantize_rows_kernel(const float* __restrict__ x, int n_rows, int n,
                                                               const float* __restrict__ norm_w, float eps,
                                                               char* __restrict__ pk, char* __restrict__ p0) {
#pragma clang fp contract(off)
  typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));
  const int row = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nb = n / 256, tile = row >> 4, a = row & 15, nt = min(16, n_rows - 16 * tile);
  const float* xr = x + (size_t)row * n;
  char* tk = pk + (size_t)tile * 16 * nb * kPackedKBytes;
  char* t0 = Q0 ? p0 + (size_t)tile * 16 * nb * kPacked0Bytes : nullptr;
  const int b0 = W * (int)blockIdx.y + wave;
  // The wave's first block, loaded ahead of the norm's reduction.
  f32x4a xv{}, wv{};
  const int bc = min(b0, nb - 1);
  xv = *reinterpret_cast<const f32x4a*>(xr + 256 * bc + 4 * lane);
  if constexpr (NORM) wv = *reinterpret_cast<const f32x4a*>(norm_w + 256 * bc + 4 * lane);
  float inv = 1.f;
  if constexpr (NORM) {
    __shared__ double red[4];
    // The squares in f64: thread t < 256 takes t, t + 256, .., then each wave's
    // sum, then the four waves' in order.
    if (wave < 4) {
      double ss = 0.0;
      for (int i = threadIdx.x; i < n; i += 256) {
        const double v = (double)xr[i];
        ss += v * v;
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
      if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) tot += red[w];
    inv = (float)(1.0 / sqrt(tot / (double)n + (double)eps));
  }
  for (int b = b0; b < nb; b += W * (int)gridDim.y) {
    if (b != b0) {
      xv = *reinterpret_cast<const f32x4a*>(xr + 256 * b + 4 * lane);
      if constexpr (NORM) wv = *reinterpret_cast<const f32x4a*>(norm_w + 256 * b + 4 * lane);
    }
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = NORM ? xv[e] * inv * wv[e] : xv[e];
    // Values 4 lane .. + 3: bytes 4 (lane % 4) of piece lane / 4.
    const Q8KLane k = quantize_lane_q8_k(v);
    char* ub = tk + (size_t)b * nt * kPackedKBytes;
    const int piece = lane >> 2;
    *reinterpret_cast<uint32_t*>(ub + (piece * nt + a) * 16 + 4 * (lane & 3)) = k.q;
    if ((lane & 3) == 0)
      *reinterpret_cast<_Float16*>(ub + 256 * nt + ((piece & 3) * nt + a) * 8 + 2 * (piece >> 2)) =
          (_Float16)(float)k.sum16;
    if (lane == 0) *reinterpret_cast<float*>(ub + 288 * nt + 4 * a) = k.d;
    if constexpr (Q0) {
      const Q80Lane z = quantize_lane_q8_0(v);
      char* zb = t0 + (size_t)b * nt * kPacked0Bytes;
      const int blk = lane >> 3, i = lane & 7;  // values 4 i .. + 3 of the block: byte 4 (i % 2) of its piece i / 2
      *reinterpret_cast<uint32_t*>(zb + ((4 * (blk >> 1) + (i >> 1)) * nt + a) * 16 + 8 * (blk & 1) + 4 * (i & 1)) = z.q;
      if (i == 0) *reinterpret_cast<float*>(zb + 256 * nt + 32 * a + 4 * blk) = z.d;
    }
  }
}

__global__ __launch_bounds__(256) void vec_add_kernel(float* __restrict__ a, const float* __restrict__ b, long n) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) a[i] += b[i];
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float* __restrict__ out, long n) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = 0.f;
}

template <int FMT>
void launch_rows_t(const uint8_t* w, size_t row_bytes, int nb, const void* acts, size_t row_lo, size_t n_rows,
                   float* out, hipStream_t s) {
  const unsigned grid = (unsigned)((n_rows + kRowsPerWG - 1) / kRowsPerWG);
  hipLaunchKernelGGL((gemv_rows_kernel<FMT>), dim3(grid), dim3(64 * kRowsPerWG), 0, s, w, row_bytes, nb, acts,
                     (long)row_lo, (int)n_rows, out);
}


}  // namespace

HipStatus launch_quantize_q8_k(const float* x, rv_block_q8_k* out, size_t n_blocks, hipStream_t s) {
  HipStatus st;
  if (n_blocks == 0) return st;
  hipLaunchKernelGGL(quantize_q8_k_kernel, dim3((unsigned)((n_blocks + 3) / 4)), dim3(256), 0, s, x, out,
                     (int)n_blocks);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "quantize_q8_k launch";
  return st;
}

HipStatus launch_quantize_q8_0(const float* x, rv_block_q8_0* out, size_t n_blocks, hipStream_t s) {
  HipStatus st;
  if (n_blocks == 0) return st;
  hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((n_blocks * 32 + 255) / 256)), dim3(256), 0, s, x, out,
                     (int)n_blocks);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "quantize_q8_0 launch";
  return st;
}

HipStatus launch_gemv_rows(uint32_t fmt, const uint8_t* w, size_t row_bytes, size_t in_dim, const void* acts,
                           size_t row_lo, size_t n_rows, float* out, hipStream_t s) {
  HipStatus st;
  if (n_rows == 0 || in_dim == 0) return st;
  const int nb = (int)(in_dim / (fmt == RV_QF_Q8_0 ? 32 : 256));
  switch (fmt) {
    case RV_QF_Q4_K: launch_rows_t<RV_QF_Q4_K>(w, row_bytes, nb, acts, row_lo, n_rows, out, s); break;
    case RV_QF_Q5_K: launch_rows_t<RV_QF_Q5_K>(w, row_bytes, nb, acts, row_lo, n_rows, out, s); break;
    case RV_QF_Q6_K: launch_rows_t<RV_QF_Q6_K>(w, row_bytes, nb, acts, row_lo, n_rows, out, s); break;
    default: launch_rows_t<RV_QF_Q8_0>(w, row_bytes, nb, acts, row_lo, n_rows, out, s);
  }
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "gemv launch";
  return st;
}

HipStatus launch_fill_zero(float* out, size_t n, hipStream_t s) {
  HipStatus st;
  if (n == 0) return st;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out, (long)n);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "fill launch";
  return st;
}

HipStatus launch_fused_proj(const FusedProjArgs& a, hipStream_t s) {
  HipStatus st;
  unsigned groups = 0;
  for (int i = 0; i < a.n_seg; ++i) groups += (unsigned)fused_groups(a.n_rows[i]);
  if (groups == 0) return st;
  const dim3 grid(groups), block(64 * kFusedWaves);
#define RV_FUSED(NB)                                                          \
  if (a.norm_w)                                                               \
    hipLaunchKernelGGL((fused_proj_kernel<true, NB>), grid, block, 0, s, a);  \
  else                                                                        \
    hipLaunchKernelGGL((fused_proj_kernel<false, NB>), grid, block, 0, s, a)
  if (a.nbk <= kFusedWaves) {
    RV_FUSED(1);
  } else if (a.nbk <= 2 * kFusedWaves) {
    RV_FUSED(2);
  } else {
    RV_FUSED(4);
  }
#undef RV_FUSED
  static_assert(kFusedMaxKBlocks == 4 * kFusedWaves, "the widest row");
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "fused projection launch";
  return st;
}

HipStatus launch_rmsnorm(const float* x, const float* w, float eps, size_t n, float* out, hipStream_t s) {
  HipStatus st;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(1), dim3(1024), 0, s, x, w, eps, (int)n, out);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "rmsnorm launch";
  return st;
}

HipStatus launch_vec_add(float* a, const float* b, size_t n, hipStream_t s) {
  HipStatus st;
  if (n == 0) return st;
  hipLaunchKernelGGL(vec_add_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, b, (long)n);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "vec_add launch";
  return st;
}

HipStatus launch_quantize_rows(const float* x, size_t n_rows, size_t n, const float* norm_w, float eps, void* packed_k,
                               void* packed_0, hipStream_t s) {
  HipStatus st;
  if (n_rows == 0 || n == 0) return st;
  if (norm_w && !packed_0) {  // the normed form writes both
    st.e = hipErrorInvalidValue;
    st.what = "quantize rows: the norm without the Q8_0 rows";
    return st;
  }
  char *pk = (char*)packed_k, *p0 = (char*)packed_0;
  const unsigned nb = (unsigned)(n / 256);
  if (norm_w)
    hipLaunchKernelGGL((quantize_rows_kernel<true, true, 8>), dim3((unsigned)n_rows), dim3(512), 0, s, x, (int)n_rows,
                       (int)n, norm_w, eps, pk, p0);
  else if (p0)
    hipLaunchKernelGGL((quantize_rows_kernel<false, true, 4>), dim3((unsigned)n_rows, (nb + 3) / 4), dim3(256), 0, s, x,
                       (int)n_rows, (int)n, norm_w, eps, pk, p0);
  else
    hipLaunchKernelGGL((quantize_rows_kernel<false, false, 4>), dim3((unsigned)n_rows, (nb + 3) / 4), dim3(256), 0, s,
                       x, (int)n_rows, (int)n, norm_w, eps, pk, p0);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "quantize rows launch";
  return st;
}

HipStatus launch_quantize_both(const float* x, rv_block_q8_k* ok, rv_block_q8_0* o0, size_t n_k_blocks,
                               hipStream_t s) {
  HipStatus st;
  if (n_k_blocks == 0) return st;
  hipLaunchKernelGGL(quantize_both_kernel, dim3((unsigned)((n_k_blocks + 3) / 4)), dim3(256), 0, s, x, ok, o0,
                     (int)n_k_blocks);
  st.e = hipGetLastError();
  if (st.e != hipSuccess) st.what = "quantize launch";
  return st;
}

}  // namespace rv

