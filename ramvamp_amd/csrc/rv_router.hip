// rv_router.hip — the MoE router's decision (include/ramvamp_router.h;
// model/forward.rs:2658-2705), bit for bit.
//
// Every expert's logit is one serial f32 sum in index order, each product
// rounded before it is added (dot_f32, forward.rs:1231-1238; contraction off),
// so the order binds it: a dependent f32 addition takes 9 cycles, 18.4 k (7.7
// us) for a 2048-wide row.
//
// At most 128 experts (staged_kernel): two waves per row, lane = expert, take
// the sums from 64-value chunks of all weight rows that four more waves bring
// through LDS; each value costs one multiplication (x broadcast from a
// register by DPP) and one addition, the pair 5.4 ns (13 cycles). Each row's softmax and top-k then run in one wave with
// two experts per lane.
//
// Otherwise (router_kernel): each thread streams its own experts' rows with
// 16-byte loads, chunks ahead of the sums (rows 16-byte aligned; otherwise
// 4-byte loads in the same order), the rows staged in LDS.
//
// The softmax (softmax.rs:18-40) takes the max over the logits, each
// exponential in f64, the f64 sum in expert order and the f32 reciprocal. The
// top-k (strict >: the first index wins ties; the winner set to -inf) is an
// argmax over a wave that prefers the larger probability and then the lower
// index, which is the serial scan's choice; the renormalization is an f32 sum
// in selection order, then one division each.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/ramvamp_router.h"
#include "rv_device.hpp"
#include "rv_internal.hpp"

namespace rv {
namespace {

constexpr int kRouterThreads = 256;
constexpr int kMaxExperts = 1024;
constexpr int kMaxHidden = 16384;
constexpr int kChunk = 32;  // weight values per prefetched chunk

// Dynamic LDS per row: x [hidden], the logits [n_experts + 1], then the f64
// exponentials [n_experts]; rounded to 4 floats so every row's x starts
// 16-byte aligned for the chunked reads.
__host__ __device__ constexpr size_t router_lds_floats(size_t hidden, size_t n_experts) {
  return (((hidden + n_experts + 2) & ~(size_t)1) + 2 * n_experts + 3) & ~(size_t)3;
}

// The x values of chunk c for rows 0..R-1, read from LDS (row r's region
// starts row_stride floats after row r-1's).
template <int R>
__device__ __forceinline__ void load_x(f32x4 (&xv)[R][kChunk / 4], const float* __restrict__ xs, int row_stride,
                                       int c) {
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < kChunk / 4; ++q)
      xv[r][q] = *reinterpret_cast<const f32x4*>(xs + (size_t)r * row_stride + c * kChunk + 4 * q);
}

// acc[r] += w[j] * x_r[j] for one 32-value chunk of R rows, in order: the
// chunk's products first (independent, each rounded), then each row's
// dependent additions, so the sums' chains wait on additions only.
template <int R>
__device__ __forceinline__ void chunk_sum(float (&acc)[R], const f32x4 (&w)[kChunk / 4],
                                          const f32x4 (&xv)[R][kChunk / 4]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float p[kChunk];
#pragma unroll
    for (int q = 0; q < kChunk / 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) p[4 * q + e] = w[q][e] * xv[r][q][e];
#pragma unroll
    for (int k = 0; k < kChunk; ++k) acc[r] += p[k];
  }
}

// R rows per workgroup (blockIdx.x * R ..), each with its LDS region of
// router_lds_floats(hidden, n_experts) floats; every weight chunk a thread
// loads feeds all R rows' sums.
template <int R>
__global__ __launch_bounds__(kRouterThreads) void router_kernel(const float* __restrict__ x, int n_rows, int hidden,
                                                                const float* __restrict__ router, int n_experts,
                                                                int top_k, int norm, uint32_t* __restrict__ experts,
                                                                float* __restrict__ weights) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int rs = (int)router_lds_floats(hidden, n_experts);  // floats per row region (a multiple of 4)
  const int row0 = (int)blockIdx.x * R, nr = min(R, n_rows - row0);
  auto xs_of = [&](int r) { return smem + (size_t)r * rs; };                 // [hidden]
  auto prob_of = [&](int r) { return smem + (size_t)r * rs + hidden; };      // [n_experts + 1]
  auto ex_of = [&](int r) {                                                  // [n_experts], 8-byte aligned
    return reinterpret_cast<double*>(smem + (size_t)r * rs + ((hidden + n_experts + 2) & ~1));
  };
  const int tid = threadIdx.x;
  for (int r = 0; r < R; ++r) {
    const float* xr = x + (size_t)(row0 + min(r, nr - 1)) * hidden;  // rows past the batch repeat its last
    for (int i = tid; i < hidden; i += kRouterThreads) xs_of(r)[i] = xr[i];
  }
  __syncthreads();
  const bool vec = hidden % 4 == 0 && ((uintptr_t)router & 15) == 0;
  const int nc = vec ? hidden / kChunk : 0;  // whole chunks; the rest one value at a time
  for (int g0 = 0; g0 < n_experts; g0 += kRouterThreads) {
    const int e = min(g0 + tid, n_experts - 1);
    const float* w = router + (size_t)e * hidden;
    const f32x4* wv = reinterpret_cast<const f32x4*>(w);
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    // Chunk c of the weight row (clamped to the last: every prefetch is
    // issued, so the wait before each chunk's use counts only newer chunks'
    // loads), three ahead of its sums. Up to 2 rows, x is read from LDS one
    // chunk ahead too; 4 rows' worth would not fit the registers, so there
    // it is read just before its sums.
    constexpr bool x_ahead = R <= 2;
    auto fetch = [&](int c, f32x4 (&dst)[kChunk / 4]) {
      c = min(c, nc - 1);
#pragma unroll
      for (int q = 0; q < kChunk / 4; ++q) dst[q] = wv[c * (kChunk / 4) + q];
    };
    auto pre = [&](f32x4 (&xv)[R][kChunk / 4], int c) {
      if constexpr (x_ahead) load_x<R>(xv, smem, rs, c);
    };
    auto use = [&](const f32x4 (&wc)[kChunk / 4], f32x4 (&xv)[R][kChunk / 4], int c) {
      if constexpr (!x_ahead) load_x<R>(xv, smem, rs, c);
      chunk_sum<R>(acc, wc, xv);
    };
    if (nc > 0) {
      f32x4 r0[kChunk / 4], r1[kChunk / 4], r2[kChunk / 4], r3[kChunk / 4];
      f32x4 xa[R][kChunk / 4], xb[R][kChunk / 4];
      fetch(0, r0);
      fetch(1, r1);
      fetch(2, r2);
      pre(xa, 0);
      int c = 0;
      for (; c + 4 <= nc; c += 4) {
        fetch(c + 3, r3);
        pre(xb, c + 1);
        use(r0, xa, c);
        fetch(c + 4, r0);
        pre(xa, c + 2);
        use(r1, xb, c + 1);
        fetch(c + 5, r1);
        pre(xb, c + 3);
        use(r2, xa, c + 2);
        fetch(c + 6, r2);
        pre(xa, min(c + 4, nc - 1));
        use(r3, xb, c + 3);
      }
      // Up to three chunks left, already in r0, r1, r2 (x of the first in xa).
      if (c < nc) use(r0, xa, c);
      if (c + 1 < nc) {
        pre(xb, c + 1);
        use(r1, xb, c + 1);
      }
      if (c + 2 < nc) {
        pre(xa, c + 2);
        use(r2, xa, c + 2);
      }
    }
    for (int i = nc * kChunk; i < hidden; ++i) {
      const float wi = w[i];
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] += wi * xs_of(r)[i];
    }
    if (g0 + tid < n_experts) {
#pragma unroll
      for (int r = 0; r < R; ++r) prob_of(r)[g0 + tid] = acc[r];
    }
  }
  __syncthreads();
  if (tid < nr) {  // thread r: row r's maximum
    const float* pr = prob_of(tid);
    float mx = -INFINITY;
    for (int e = 0; e < n_experts; ++e)
      if (pr[e] > mx) mx = pr[e];
    prob_of(tid)[n_experts] = mx;  // the slot after the logits (the f64 array starts past it)
  }
  __syncthreads();
  for (int r = 0; r < nr; ++r) {
    const double m = (double)prob_of(r)[n_experts];
    for (int e = tid; e < n_experts; e += kRouterThreads) ex_of(r)[e] = exp((double)prob_of(r)[e] - m);
  }
  __syncthreads();
  __shared__ float inv_sh[R];
  if (tid < nr) {  // thread r: row r's f64 sum in expert order
    const double* er = ex_of(tid);
    double sum = 0.0;
    for (int e = 0; e < n_experts; ++e) sum += er[e];
    inv_sh[tid] = (float)(1.0 / sum);
  }
  __syncthreads();
  for (int r = 0; r < nr; ++r) {
    const float inv = inv_sh[r];
    for (int e = tid; e < n_experts; e += kRouterThreads) prob_of(r)[e] = (float)ex_of(r)[e] * inv;
  }
  __syncthreads();
  // Wave r (< nr): row r's top_k rounds of an argmax, each lane over experts
  // lane, lane + 64, ... (in order, strict >), then across lanes preferring
  // the larger value and then the lower index; with nothing above -inf,
  // expert 0 at -inf.
  const int wave = tid >> 6, lane = tid & 63;
  if (wave >= nr) return;
  float* prob = prob_of(wave);
  uint32_t* eo = experts + (size_t)(row0 + wave) * top_k;
  float* wo = weights + (size_t)(row0 + wave) * top_k;
  float s = 0.f;
  for (int k = 0; k < top_k; ++k) {
    float bp = -INFINITY;
    int be = 1 << 30;
    for (int e = lane; e < n_experts; e += 64)
      if (prob[e] > bp) {
        bp = prob[e];
        be = e;
      }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float p2 = __shfl_xor(bp, off, 64);
      const int e2 = __shfl_xor(be, off, 64);
      if (p2 > bp || (p2 == bp && e2 < be)) {
        bp = p2;
        be = e2;
      }
    }
    if (be == (1 << 30)) be = 0;  // every probability -inf or NaN: the scan keeps expert 0
    if (lane == 0) {
      eo[k] = (uint32_t)be;
      wo[k] = bp;
      prob[be] = -INFINITY;
    }
    s += bp;  // the selection-order f32 sum, identical on every lane
    wave_lds_order();  // lane 0's -inf before the next round's reads
  }
  if (norm && lane == 0) {
    for (int k = 0; k < top_k; ++k) wo[k] = wo[k] / s;
  }
}

// ---- the staged form ---------------------------------------------------------
constexpr int kStagedExperts = 128;
constexpr int kStagedChunk = 64;               // weight values per chunk
constexpr int kStagedRow = kStagedChunk + 4;   // floats per staged expert row (16-byte reads of 16 rows: all banks)
constexpr int kStagers = 4;                    // waves that bring the weights
constexpr int kRing = 3;                       // chunks in LDS, and in the waves' registers (4: no faster)

template <int R>
struct StagedLds {
  float w[kRing][kStagedExperts][kStagedRow];
  double ex[R][kStagedExperts];
  float logit[R][kStagedExperts];
};

// x of the lane that holds value K of its 16-lane row, in every lane.
template <int K>
__device__ __forceinline__ float row_bcast(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + K, 0xF, 0xF, true));
}

// One serial f32 sum over 16-value groups, its products three values ahead of
// its additions: an addition depends on the previous one (9 cycles), and a
// product adjacent to the addition that takes it would double that. Group g's
// weights are in w[g % 3], read from LDS two groups ahead (the stagers' writes
// hold the LDS up to 256 cycles at a time); p holds the products of a group's
// first three values.
struct Chain {
  float acc = 0.f;
  float p[4];
  f32x4 w[3][4];
};

__device__ __forceinline__ void load_group(f32x4 (&w)[4], const float* __restrict__ at) {
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const f32x4*>(at + 4 * i);
}

template <int K>
__device__ __forceinline__ void chain_step(Chain& c, const f32x4 (&w)[4], const f32x4 (&nw)[4], float xv, float nx) {
#pragma clang fp contract(off)
  constexpr int J = (K + 3) % 16;
  c.acc += c.p[K % 4];
  c.p[(K + 3) % 4] = K + 3 < 16 ? row_bcast<J>(xv) * w[J / 4][J % 4] : row_bcast<J>(nx) * nw[J / 4][J % 4];
  __builtin_amdgcn_sched_barrier(0);  // the order is the point
}

// Adds group G's 16 products (x in xv), forms the next group's first three (x
// in nx) and reads the weights of the one after it from `ahead`.
template <int G>
__device__ __forceinline__ void chain_group(Chain& c, const float* __restrict__ ahead, float xv, float nx) {
  const f32x4(&w)[4] = c.w[G % 3];
  const f32x4(&nw)[4] = c.w[(G + 1) % 3];
  load_group(c.w[(G + 2) % 3], ahead);
  __builtin_amdgcn_sched_barrier(0);
  chain_step<0>(c, w, nw, xv, nx);
  chain_step<1>(c, w, nw, xv, nx);
  chain_step<2>(c, w, nw, xv, nx);
  chain_step<3>(c, w, nw, xv, nx);
  chain_step<4>(c, w, nw, xv, nx);
  chain_step<5>(c, w, nw, xv, nx);
  chain_step<6>(c, w, nw, xv, nx);
  chain_step<7>(c, w, nw, xv, nx);
  chain_step<8>(c, w, nw, xv, nx);
  chain_step<9>(c, w, nw, xv, nx);
  chain_step<10>(c, w, nw, xv, nx);
  chain_step<11>(c, w, nw, xv, nx);
  chain_step<12>(c, w, nw, xv, nx);
  chain_step<13>(c, w, nw, xv, nx);
  chain_step<14>(c, w, nw, xv, nx);
  chain_step<15>(c, w, nw, xv, nx);
}

__device__ __forceinline__ float wave_max(float v) { return swap_max<32>(swap_max<16>(group_max<16>(v))); }

// One row's softmax and top-k by one wave, lane l holding experts l and l +
// 64 (those below n_experts).
template <int R>
__device__ __forceinline__ void choose(StagedLds<R>& s, int r, int lane, int n_experts, int top_k, int norm,
                                       uint32_t* __restrict__ eo, float* __restrict__ wo) {
#pragma clang fp contract(off)
  float p[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) p[h] = lane + 64 * h < n_experts ? s.logit[r][lane + 64 * h] : -INFINITY;
  const double m = (double)wave_max(fmaxf(fmaxf(-INFINITY, p[0]), p[1]));  // NaN never is the maximum
  double e[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    e[h] = exp((double)p[h] - m);
    s.ex[r][lane + 64 * h] = lane + 64 * h < n_experts ? e[h] : 0.0;
  }
  wave_lds_order();  // the other lanes' exponentials below
  // The sum in expert order (every lane the same); slots past n_experts hold
  // +0, which leaves a sum of exponentials as it is.
  double sum = 0.0;
  const int n16 = (n_experts + 15) & ~15;
  for (int i = 0; i < n16; i += 16) {
    double t[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) t[k] = s.ex[r][i + k];
#pragma unroll
    for (int k = 0; k < 16; ++k) sum += t[k];
  }
  const float inv = (float)(1.0 / sum);
#pragma unroll
  for (int h = 0; h < 2; ++h) p[h] = lane + 64 * h < n_experts ? (float)e[h] * inv : -INFINITY;
  float total = 0.f, mine = 0.f;
  uint32_t mine_e = 0;
  for (int k = 0; k < top_k; ++k) {
    // The first of the largest: slot 0 holds the lower indices. With nothing
    // above -inf (or NaN only) the scan keeps expert 0 at -inf.
    const float best = wave_max(fmaxf(fmaxf(-INFINITY, p[0]), p[1]));
    const uint64_t b0 = __ballot(p[0] == best), b1 = __ballot(p[1] == best);
    int be = 0;
    float bp = -INFINITY;
    if (best > -INFINITY) {  // wave-uniform
      const int l = __builtin_ctzll(b0 ? b0 : b1);
      be = b0 ? l : l + 64;
      bp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b0 ? p[0] : p[1]), l));
    }
    if (lane == be) p[0] = -INFINITY;
    if (lane + 64 == be) p[1] = -INFINITY;
    if (lane == (k & 63)) {
      mine = bp;
      mine_e = (uint32_t)be;
    }
    total += bp;  // the selection-order f32 sum
    if ((k & 63) == 63 || k == top_k - 1) {
      if (lane <= (k & 63)) {
        eo[(k & ~63) + lane] = mine_e;
        wo[(k & ~63) + lane] = mine;
      }
    }
  }
  if (norm)
    for (int k = lane; k < top_k; k += 64) wo[k] = wo[k] / total;
}

// R rows per workgroup: waves 2 r and 2 r + 1 sum row r's experts 0-63 and
// 64-127, the last kStagers waves bring the weights. Bound by the sums' order:
// an addition beside the next product takes 5.4 ns, so 11.1 us for 2048 values,
// of 18.3 us a call for 1 row, 21.3 for 512 and 26.9 for 1024 (31.4, 47.0 and
// 58.7 when two waves both staged and summed, each product beside the addition
// that takes it, one thread took the maximum and the f64 sum, and the top-k
// went through LDS). Products formed by the stagers, so that the sum waves only
// add, measured the same.
template <int R>
__global__ __launch_bounds__(64 * (2 * R + kStagers)) void staged_kernel(const float* __restrict__ x, int n_rows,
                                                                         int hidden, const float* __restrict__ router,
                                                                         int n_experts, int top_k, int norm,
                                                                         uint32_t* __restrict__ experts,
                                                                         float* __restrict__ weights) {
  extern __shared__ __attribute__((aligned(16))) char staged_smem[];
  auto& s = *reinterpret_cast<StagedLds<R>*>(staged_smem);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int row0 = (int)blockIdx.x * R, nc = hidden / kStagedChunk;
  const bool stager = wave >= 2 * R;
  // Stagers: chunk c's 2048 16-byte quads, eight a thread (a wave: 16 quads
  // each of 4 rows), in registers from three chunks before they are stashed.
  // Chunks past the last and experts past n_experts repeat the last one.
  const int st = (int)threadIdx.x - 128 * R;
  f32x4 wq[kRing][8];
  auto fetch = [&](int c, int slot) {
    c = min(c, nc - 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int f = 64 * kStagers * k + st, e = min(f >> 4, n_experts - 1);
      wq[slot][k] = *reinterpret_cast<const f32x4*>(router + (size_t)e * hidden + c * kStagedChunk + 4 * (f & 15));
    }
  };
  auto stash = [&](int slot) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int f = 64 * kStagers * k + st;
      *reinterpret_cast<f32x4*>(&s.w[slot][f >> 4][4 * (f & 15)]) = wq[slot][k];
    }
  };
  // Sum waves: the row's x, 16 values per register in every 16-lane row, two
  // to three chunks ahead (rows past the batch repeat its last).
  const int r = wave >> 1, ex = 64 * (wave & 1) + lane;
  const float* xr = x + (size_t)min(row0 + r, n_rows - 1) * hidden;  // wave-uniform
  const uint32_t x16 = lane & 15;
  float xv[kRing][4];
  auto fetch_x = [&](int c, float (&dst)[4]) {
    const float* at = xr + min(c, nc - 1) * kStagedChunk;
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = (at + 16 * k)[x16];
  };
  // Chunk c lies in slot c % kRing. While it is summed (and the next one's first
  // groups read), chunk c + 2 goes into the slot of chunk c - 1, last read
  // before the previous barrier. The two roles run loops of their own, so each
  // one's waits count its own loads, and pass the same nc + 1 barriers.
  auto meet = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  if (stager) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) fetch(u, u);
    stash(0);
    fetch(kRing, 0);
    stash(1);
    fetch(kRing + 1, 1);
    meet();
    for (int c0 = 0; c0 < nc; c0 += kRing) {
#pragma unroll
      for (int u = 0; u < kRing; ++u) {
        if (c0 + u >= nc) break;
        stash((u + 2) % kRing);
        fetch(c0 + u + 2 + kRing, (u + 2) % kRing);
        meet();
      }
    }
  } else {
#pragma clang fp contract(off)
#pragma unroll
    for (int u = 0; u < kRing; ++u) fetch_x(u, xv[u]);
    meet();
    Chain ch;
    load_group(ch.w[0], &s.w[0][ex][0]);
    load_group(ch.w[1], &s.w[0][ex][16]);
    ch.p[0] = row_bcast<0>(xv[0][0]) * ch.w[0][0][0];
    ch.p[1] = row_bcast<1>(xv[0][0]) * ch.w[0][0][1];
    ch.p[2] = row_bcast<2>(xv[0][0]) * ch.w[0][0][2];
    auto chunk = [&](auto U, int c) {  // U = c % kRing
      constexpr int u = decltype(U)::value;
      const float* w = &s.w[u][ex][0];
      const float* nw = &s.w[(u + 1) % kRing][ex][0];
      chain_group<4 * u>(ch, w + 32, xv[u][0], xv[u][1]);
      chain_group<4 * u + 1>(ch, w + 48, xv[u][1], xv[u][2]);
      chain_group<4 * u + 2>(ch, nw, xv[u][2], xv[u][3]);
      chain_group<4 * u + 3>(ch, nw + 16, xv[u][3], xv[(u + 1) % kRing][0]);
      fetch_x(c + kRing, xv[u]);
      meet();
    };
    for (int c = 0; c < nc; c += kRing) {
      chunk(std::integral_constant<int, 0>{}, c);
      if (c + 1 >= nc) break;
      chunk(std::integral_constant<int, 1>{}, c + 1);
      if (c + 2 >= nc) break;
      chunk(std::integral_constant<int, 2>{}, c + 2);
    }
    s.logit[r][ex] = ch.acc;
  }
  __syncthreads();
  if (wave < R && row0 + wave < n_rows)
    choose<R>(s, wave, lane, n_experts, top_k, norm, experts + (size_t)(row0 + wave) * top_k,
              weights + (size_t)(row0 + wave) * top_k);
}

template <int R>
hipError_t launch_staged(const float* x, size_t n_rows, size_t hidden, const float* router, size_t n_experts,
                         size_t top_k, int norm, uint32_t* experts, float* weights, hipStream_t s) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&staged_kernel<R>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(StagedLds<R>));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(staged_kernel<R>, dim3((unsigned)((n_rows + R - 1) / R)), dim3(64 * (2 * R + kStagers)),
                     sizeof(StagedLds<R>), s, x, (int)n_rows, (int)hidden, router, (int)n_experts, (int)top_k, norm,
                     experts, weights);
  return hipGetLastError();
}

int32_t fail(rv_error* err, int32_t code, uint64_t a, uint64_t b, const char* what) {
  if (err) *err = rv_error{code, a, b, 0, 0, what};
  return code;
}

}  // namespace
}  // namespace rv

extern "C" int32_t rv_router_topk(const float* x, size_t n_rows, size_t hidden, const float* router,
                                  size_t router_len, size_t n_experts, size_t top_k, int norm_topk_prob,
                                  uint32_t* experts, float* weights, void* stream, uint32_t flags, rv_error* err) {
  using rv::fail;
  // forward.rs:774-777 validates top_k against the expert count first.
  if (top_k == 0 || top_k > n_experts) return fail(err, RV_FWD_INVALID_TOP_K, top_k, n_experts, "router top_k");
  if (hidden == 0) return fail(err, RV_PRIM_EMPTY, 0, 0, "router dot");
  size_t want;
  if (__builtin_mul_overflow(n_experts, hidden, &want) || want != router_len)
    return fail(err, RV_PRIM_LENGTH_MISMATCH, router_len, want, "router: weights vs n_experts x hidden");
  if (n_experts > (size_t)rv::kMaxExperts || hidden > (size_t)rv::kMaxHidden)
    return fail(err, RV_ERR_UNSUPPORTED, n_experts, hidden, "router above 1024 experts or 16384 values");
  if (flags & RV_HOST_PTRS) return fail(err, RV_ERR_UNSUPPORTED, flags, 0, "RV_HOST_PTRS (device pointers only)");
  const hipStream_t s = (hipStream_t)stream;
  if (n_rows > 0) {
    for (const void* p : {(const void*)x, (const void*)router, (const void*)experts, (const void*)weights})
      if (!p || ((uintptr_t)p & 3)) return fail(err, p ? RV_ERR_UNSUPPORTED : RV_ERR_NULL_ARG, (uintptr_t)p, 0, "router pointer");
    hipError_t e;
    const int norm = norm_topk_prob ? 1 : 0;
    if (n_experts <= (size_t)rv::kStagedExperts && hidden % rv::kStagedChunk == 0 && ((uintptr_t)router & 15) == 0) {
      // As many rows per workgroup as leave one workgroup a CU: the weights
      // (1 MiB at 128 x 2048) pass each CU's LDS once for all of them.
      if (n_rows <= 256)
        e = rv::launch_staged<1>(x, n_rows, hidden, router, n_experts, top_k, norm, experts, weights, s);
      else if (n_rows <= 512)
        e = rv::launch_staged<2>(x, n_rows, hidden, router, n_experts, top_k, norm, experts, weights, s);
      else
        e = rv::launch_staged<4>(x, n_rows, hidden, router, n_experts, top_k, norm, experts, weights, s);
    } else {
      // Rows per workgroup: as many as keep at least 256 workgroups (up to 4)
      // and fit the LDS; each weight chunk a thread loads then feeds them all.
      const size_t row_bytes = rv::router_lds_floats(hidden, n_experts) * sizeof(float);
      const size_t lds_cap = 160 * 1024 - 1024;
      int R = 1;
      while (R < 4 && n_rows >= (size_t)(2 * R) * 256 && (size_t)(2 * R) * row_bytes <= lds_cap) R *= 2;
      const unsigned grid = (unsigned)((n_rows + R - 1) / R);
#define RV_ROUTER(RR)                                                                                             \
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&rv::router_kernel<RR>),                               \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_cap);                           \
  hipLaunchKernelGGL((rv::router_kernel<RR>), dim3(grid), dim3(rv::kRouterThreads), (unsigned)(RR * row_bytes), s, x, \
                     (int)n_rows, (int)hidden, router, (int)n_experts, (int)top_k, norm, experts, weights)
      if (R == 4) {
        RV_ROUTER(4);
      } else if (R == 2) {
        RV_ROUTER(2);
      } else {
        RV_ROUTER(1);
      }
#undef RV_ROUTER
      e = hipGetLastError();
    }
    if (e != hipSuccess) return fail(err, RV_ERR_HIP, (uint64_t)e, 0, "router launch");
  }
  if (flags & RV_SYNC) {
    const hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(err, RV_ERR_HIP, (uint64_t)e, 0, "hipStreamSynchronize");
  }
  if (err) *err = rv_error{RV_OK, 0, 0, 0, 0, nullptr};
  return RV_OK;
}
