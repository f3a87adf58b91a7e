// k_add_rmsnorm.hip -- fused residual-add + RMSNorm for gfx950.
//
// Reference: v7s_fused_add_rmsnorm(o, residual, add, weight, dim),
// src/asm/add_rmsnorm_kernel.inc:15-129.
//   Pass 1: residual = residual + add (stored in place); the sum of squares is
//           accumulated in four 8-lane YMM accumulators A..D by FMA.  Blocks of
//           8 floats that do not fill a 4-way group (blocks % 4) go first, all
//           into A; then each group of 4 blocks feeds A, B, C, D.
//   Reduce: (A+B)+(C+D) lane-wise, then HADD_YMM (v7_macros.inc:38-45).
//   Scale:  1/sqrt(sumsq/dim + eps), four IEEE operations.
//   Pass 2: o = (scale * residual) * weight.
// This kernel reproduces that order exactly, so its output is bit-identical.
// One workgroup per row: each thread keeps its float4 chunks of the row in
// registers (4*(tid + k*TPR) for k < KMAX), so pass 1 issues every load of
// residual and add together and pass 2 needs no second read; residual, add
// and o move as streaming loads and stores, the weight row stays cached.  The
// updated residual also goes to LDS, where 32 lanes of wave 0 replay the 32
// FMA chains, chain by chain (ChainLayout), and reduce them with DPP row
// shifts in the (A+B)+(C+D) + HADD_YMM pairing.
// Bound: many rows by HBM ([8192, 4096] add+RMSNorm 85-86 us, 79% of the peak;
// [1000, 16384] 50.5 -> 46.5 us with 1024 threads per row in place of 256); few
// rows by latency: the loads, the chain (128 dependent FMAs at 4096 floats),
// the scale's divisions and square root, the stores ([8, 4096] RMSNorm 3.29 ->
// 2.67 us, add+RMSNorm -> Q8 3.49 -> 3.36, [8, 5376] add+RMSNorm 5.4 -> 3.4).
//
// The same row body serves the neighbours of this kernel in the reference:
//   v7s_rmsnorm (src/asm/rmsnorm_kernel.inc:12-75): no add, same order;
//   v7s_rmsnorm_quantize (src/asm/rmsnorm_quantize_kernel.inc:62-218): the
//     normalised row quantized per group of 64 exactly as v7d_quantize does;
//   and the Q8 decode step v7s_add_inplace -> v7s_rmsnorm_quantize
//     (src/asm/forward_q8.inc:386-387), fused here into one pass.
#include <type_traits>

#include "v7g_device.h"
#include "v7g_internal.h"

namespace v7g {

// The chain lane lam runs YMM accumulator q = v >> 3, lane j = v & 7 with
// v = chain_of_lane(lam), chosen so that lam = 8*q0 + 4*q1 + 2*j2 + j0 + 16*j1
// (q0, q1, j0..j2 the bits of q and j): the reduction's pairs are then lanes
// lam, lam+8 (A+B, C+D), lam, lam+4 ((A+B)+(C+D)), lam, lam+2 (v_i + v_{i+4}),
// lam, lam+1 (w0+w1, w2+w3) and lanes 0, 16 (the final sum).
__device__ __forceinline__ int chain_of_lane(int lam) {
  const int q = ((lam >> 3) & 1) | (((lam >> 2) & 1) << 1);
  const int j = (lam & 1) | (((lam >> 4) & 1) << 1) | (((lam >> 1) & 1) << 2);
  return 8 * q + j;
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// The reference's reduction of the 32 chains (lane lam holds chain
// chain_of_lane(lam)) as DPP row shifts; the same value in every lane.
__device__ __forceinline__ float chain_reduce(float acc) {
  acc = acc + dpp_f<0x108>(acc);  // row_shl:8   A+B, C+D
  acc = acc + dpp_f<0x104>(acc);  // row_shl:4   (A+B)+(C+D)
  acc = acc + dpp_f<0x102>(acc);  // row_shl:2   HADD_YMM: v_i + v_{i+4}
  acc = acc + dpp_f<0x101>(acc);  // row_shl:1   w0+w1, w2+w3
  const float lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, acc), 0));
  const float hi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, acc), 16));
  return lo + hi;
}

// Sum of squares of a row of dim floats (dim % 32 == 0) staged at the padded
// layout, in the reference's order; called by a whole wave, returns the same
// value in every lane.  U: chain elements per register set (2U VGPRs).  RING:
// how lengths that are no whole pair of sets are read; for a length known at
// compile time the three-set form ([300, 3840] RMSNorm -> Q8 4.72 -> 4.20 us,
// [2000, 3840] 10.9 -> 10.3, [300, 2560] 3.88 -> 3.66), else the plain loop, which
// the compiler batches by 16 (the three-set form with run-time bounds: 2-3%
// slower at 576, 1088, 1536 and 7808, 1-2% faster at 832 and 2304).
template <int U, bool RING, bool LEFT = false>
__device__ __forceinline__ float padded_row_sumsq(const float *row, int dim) {
  const int lane = __lane_id();
  float acc = 0.0f;
  if (lane < 32) {
    const int v = chain_of_lane(lane);
    // element 32g + v sits at float 40g + v + 4*(v >> 4)
    const float *p = row + v + 4 * (v >> 4);
    const int steps = dim >> 5;
    if constexpr (LEFT) {
      // the (dim/8) % 4 leftover blocks, all into A; element 8*left + 32g + v is then at
      // float 40g + 8*left + v + 4*((2*left + (v >> 2)) >> 2)
      const int left = (dim >> 3) & 3;
      if (v < 8)
        for (int b = 0; b < left; ++b) {
          const float e = row[8 * b + v + 4 * ((2 * b + (v >> 2)) >> 2)];
          acc = __builtin_fmaf(e, e, acc);
        }
      p = row + 8 * left + v + 4 * ((2 * left + (v >> 2)) >> 2);
    }
    if (steps % (2 * U) == 0 && (!LEFT || steps > 0)) {
      // Two register sets of U chain elements: the LDS reads of one set are
      // in flight while the FMAs consume the other, so the chain waits on
      // LDS once instead of once per U steps.  Same FMAs, same order.  The
      // empty asm statements pass the accumulator through a point after each
      // set of reads, so the compiler neither sinks a read down to its use
      // nor hoists the FMAs above the reads of the other set.
      float a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = p[40 * u];
      int g0 = 0;
      for (; g0 + 2 * U < steps; g0 += 2 * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) b[u] = p[40 * (g0 + U + u)];
        asm volatile("" : "+v"(acc)::"memory");
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_fmaf(a[u], a[u], acc);
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = p[40 * (g0 + 2 * U + u)];
        asm volatile("" : "+v"(acc)::"memory");
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_fmaf(b[u], b[u], acc);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) b[u] = p[40 * (g0 + U + u)];
      asm volatile("" : "+v"(acc)::"memory");
#pragma unroll
      for (int u = 0; u < U; ++u) acc = __builtin_fmaf(a[u], a[u], acc);
#pragma unroll
      for (int u = 0; u < U; ++u) acc = __builtin_fmaf(b[u], b[u], acc);
    } else if constexpr (!RING) {
#pragma unroll 16
      for (int g = 0; g < steps; ++g) {
        const float e = p[40 * g];
        acc = __builtin_fmaf(e, e, acc);
      }
    } else {
      // Three sets of 8, two in flight while the third is consumed, then the
      // last elements one by one.
      constexpr int V = 8;
      const int sets = steps / V;
      float a[V], b[V], d[V];
      auto get = [&](float(&v)[V], int set) {
        if (set < sets) {  // uniform
#pragma unroll
          for (int u = 0; u < V; ++u) v[u] = p[40 * (V * set + u)];
        }
        asm volatile("" : "+v"(acc)::"memory");
      };
      auto eat = [&](const float(&v)[V]) {
#pragma unroll
        for (int u = 0; u < V; ++u) acc = __builtin_fmaf(v[u], v[u], acc);
        asm volatile("" : "+v"(acc)::"memory");
      };
      get(a, 0);
      get(b, 1);
      for (int s = 0; s < sets; s += 3) {
        get(d, s + 2);
        eat(a);
        if (s + 1 >= sets) break;
        get(a, s + 3);
        eat(b);
        if (s + 2 >= sets) break;
        get(b, s + 4);
        eat(d);
      }
      for (int g = sets * V; g < steps; ++g) {
        const float e = p[40 * g];
        acc = __builtin_fmaf(e, e, acc);
      }
    }
  }
  return chain_reduce(acc);
}

// A workgroup barrier for LDS only: unlike __syncthreads() it does not wait
// for the wave's global loads and stores (s_waitcnt lgkmcnt(0), not vmcnt).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ int padded(int m) { return 4 * (m + (m >> 2)); }

// Where the row kernels stage a row: chain by chain.  Chain lane lam's
// elements, in the order its FMAs take them, lie one behind another at float
// lam * STRIDE, so the lane reads four of them with one 16-byte LDS load.
// Element 8b + j of the row (block b, YMM lane j) is step left + g of its chain
// for block left + 4g + q; the leftover blocks b < left = (dim/8) % 4, which
// the reference takes first, all into A, are steps b of chain (A, j).  Steps a
// chain has no element for (past the row's end; B, C and D during the leftover
// blocks) hold zeros: fma(0, 0, acc) is acc for every sum of squares, so they
// change nothing, and every row of up to 4*TPR*KMAX floats runs the same
// compiled chain.
// U: 16-byte reads per register set of the chain.
template <int TPR, int KMAX, bool LEFT, int U>
struct ChainLayout {
  static constexpr int kSteps = TPR * KMAX / 8 + (LEFT ? 3 : 0);  // room for three leftover blocks
  static constexpr int kSets = (kSteps + 4 * U - 1) / (4 * U);
  static constexpr int kStride = 4 * U * kSets + 4 * (1 + (U * kSets) % 2);
  static_assert(kStride % 8 == 4, "the 16-byte reads of 16 lanes, and a wave's 4-byte writes, fall on distinct banks");
  // two sets behind the last chain, which the chain's prefetch touches; then the scale
  static constexpr int kScale = 32 * kStride + 8 * U;
  static constexpr unsigned kBytes = 4u * (kScale + 4);
};

// The row's sum of squares in the reference's order, from the chain layout;
// called by a whole wave, the same value in every lane.  Three register sets of
// U 16-byte reads: two sets are in flight while the FMAs consume the third (LDS
// answers in about 130 cycles, a set of U = 4 is 16 dependent FMAs of 4 cycles).
// The empty asm statements pass the accumulator through a point after each set
// of reads, so the compiler neither sinks a read to its use nor hoists the FMAs
// above the reads of another set.  Reads run up to two sets past the chain's
// end, into the next chain or the space behind the last.
template <int SETS, int STRIDE, int U>
__device__ __forceinline__ float chain_sumsq(const float *row) {
  const int lane = __lane_id();
  float acc = 0.0f;
  if (lane < 32) {
    const float4 *p = reinterpret_cast<const float4 *>(row + lane * STRIDE);
    float4 a[U], b[U], d[U];
    auto get = [&](float4(&v)[U], int set) {
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = p[U * set + u];
      asm volatile("" : "+v"(acc)::"memory");
    };
    auto eat = [&](const float4(&v)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        acc = __builtin_fmaf(v[u].x, v[u].x, acc);
        acc = __builtin_fmaf(v[u].y, v[u].y, acc);
        acc = __builtin_fmaf(v[u].z, v[u].z, acc);
        acc = __builtin_fmaf(v[u].w, v[u].w, acc);
      }
      asm volatile("" : "+v"(acc)::"memory");
    };
    get(a, 0);
    get(b, 1);
    for (int s = 0;; s += 3) {
      get(d, s + 2);
      eat(a);
      if (s + 1 >= SETS) break;
      get(a, s + 3);
      eat(b);
      if (s + 2 >= SETS) break;
      get(b, s + 4);
      eat(d);
      if (s + 3 >= SETS) break;
    }
  }
  return chain_reduce(acc);
}

// One row of dim floats, 4*TPR*(KMAX-1) < dim <= 4*TPR*KMAX.  ADD: the input
// is residual + add (residual updated in place), else x.  QGS == 0:
// o = (s*x)*w; QGS = 32 or 64: the normalised row is quantized in groups of
// QGS (codes q, scales q_s) and o is not written.  o may alias residual (the
// row then ends as o, as in the reference).  LEFT: dim % 32 != 0.
// Each of TPR threads holds KMAX float4 chunks in registers from the loads to
// the results.  Only the last chunk is tested against the row's end: its loads
// are clamped to the row's first floats, its LDS stores are zeros, its global
// stores predicated (a branch around a load would put a wait at its merge).
// When the weights are requested (vector memory operations retire in issue
// order, so a weight load behind the residual's stores waits for them):
//  - FEW, at most one row per CU and the shapes of more rows that launch_row and
//    launch_q8_row name: once the row is staged, ahead of the residual's stores, so
//    that they travel during the chain and delay neither the row nor the result
//    ([1, 8192] add+RMSNorm 4.85 -> 4.02 us, with the chain's new layout);
//  - many rows, ADD: right behind the row's loads;
//  - many rows without ADD: after the chain, so that the other rows on the CU
//    get their loads first ([1024, 4096] 6.9 -> 6.2 us); with four and more
//    chunks one by one, each store waiting for the one before (and so with ADD
//    beyond 8192 floats at two rows per CU).  Where all rows are resident at
//    once, unpaced stores of the first rows hold up the loads of the last: [1000,
//    8192] 14.4 us, paced 11.4.
// FEW uses as many registers as the chain can use; otherwise at most 64 VGPRs
// (row_waves), so that a CU's waves are full, with smaller chain sets.
static constexpr int row_chain_u(int kmax, bool few) { return few || kmax == 1 ? 4 : (kmax == 2 ? 3 : 2); }

template <int TPR, int KMAX, bool ADD, int QGS, bool LEFT, bool FEW>
__device__ __forceinline__ void rms_row(float *o, int8_t *q, float *q_s, float *xin, const float *add,
                                        const float *weight, int dim, float eps) {
  constexpr int U = row_chain_u(KMAX, FEW);
  using L = ChainLayout<TPR, KMAX, LEFT, U>;
  constexpr int STRIDE = L::kStride;
  constexpr bool LATE_W = !FEW && (!ADD || (KMAX == 8 && TPR > 256));
  extern __shared__ __attribute__((aligned(16))) float row[];
  const int tid = threadIdx.x;
  const size_t r = blockIdx.x;
  float *xr = xin + r * (size_t)dim;
  const float *ar = ADD ? add + r * (size_t)dim : nullptr;
  const bool last = 4 * (tid + (KMAX - 1) * TPR) < dim;  // the last chunk is live
  auto live = [&](int k) { return LEFT ? 4 * (tid + k * TPR) < dim : k < KMAX - 1 || last; };
  // A chunk's address as a uniform base and a 32-bit lane offset (scalar-base loads and stores).
  const unsigned t4 = 4u * (unsigned)tid;
  const unsigned t4_last = last ? t4 + 4u * (KMAX - 1) * TPR : 0u;
  auto src = [&](const float *p, int k) {
    if constexpr (LEFT) return p + (live(k) ? t4 + 4u * k * TPR : 0u);
    return k < KMAX - 1 ? (p + 4 * k * TPR) + t4 : p + t4_last;
  };

  float4 x[KMAX], b[KMAX], w[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    x[k] = ld_stream4(src(xr, k));
    if constexpr (ADD) b[k] = ld_stream4(src(ar, k));
  }
  auto load_w = [&]() {
#pragma unroll
    for (int k = 0; k < KMAX; ++k) w[k] = *reinterpret_cast<const float4 *>(src(weight, k));
  };
  if constexpr (ADD && !FEW && !LATE_W) load_w();
  const int left = LEFT ? (dim >> 3) & 3 : 0;
  {  // zeros for the steps no chunk writes
    constexpr int first = LEFT ? 0 : TPR * KMAX / 8, end = 4 * U * L::kSets;
    for (int i = tid + 32 * first; i < 32 * end; i += TPR) {
      const int lam = i & 31, step = i >> 5;
      const bool zero = !LEFT || (step < left && chain_of_lane(lam) >= 8) || step >= left + (dim >> 5);
      if (zero) row[lam * STRIDE + step] = 0.f;
    }
  }
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    if constexpr (ADD) x[k] = make_float4(x[k].x + b[k].x, x[k].y + b[k].y, x[k].z + b[k].z, x[k].w + b[k].w);
    // chunk m is the half (m & 1) of block m >> 1: chains 8q + 4(m & 1) + {0, 1, 2, 3}, which
    // chain_of_lane gives to lanes lam + {0, 1, 16, 17}
    const int m = tid + k * TPR, blk = m >> 1;
    int qa = blk & 3, step = blk >> 2;
    if constexpr (LEFT) {
      const bool lo = blk < left;
      qa = lo ? 0 : (blk - left) & 3;
      step = lo ? blk : left + ((blk - left) >> 2);
    }
    float *p = row + (8 * (qa & 1) + 4 * (qa >> 1) + 2 * (m & 1)) * STRIDE + step;
    if (!LEFT || live(k)) {
      p[0] = live(k) ? x[k].x : 0.f;
      p[STRIDE] = live(k) ? x[k].y : 0.f;
      p[16 * STRIDE] = live(k) ? x[k].z : 0.f;
      p[17 * STRIDE] = live(k) ? x[k].w : 0.f;
    }
  }
  if constexpr (ADD) {
    if constexpr (FEW) {
      asm volatile("" ::: "memory");
      load_w();
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
      if (live(k)) st_stream4((xr + 4 * k * TPR) + t4, x[k]);
  }
  lds_barrier();
  if constexpr (!ADD && FEW) load_w();
  if (tid < 64) {
    const float s0 = rms_scale(chain_sumsq<L::kSets, STRIDE, U>(row), (float)dim, eps);
    if (tid == 0) row[L::kScale] = s0;
  }
  lds_barrier();
  if constexpr (LATE_W && KMAX < 4) load_w();
  const float s = row[L::kScale];

  // n = (s * x) * w, then either stored or quantized.
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const unsigned i = 4u * (unsigned)(tid + k * TPR);
    if constexpr (LATE_W && KMAX >= 4) {  // one chunk's weights, and the stores so far done, before its store
      w[k] = *reinterpret_cast<const float4 *>(src(weight, k));
      asm volatile("s_waitcnt vmcnt(0)" : "+v"(w[k].x), "+v"(w[k].y), "+v"(w[k].z), "+v"(w[k].w)::"memory");
    }
    const float4 n =
        make_float4((s * x[k].x) * w[k].x, (s * x[k].y) * w[k].y, (s * x[k].z) * w[k].z, (s * x[k].w) * w[k].w);
    if constexpr (QGS == 0) {
      if (live(k)) st_stream4((o + r * (size_t)dim + 4 * k * TPR) + t4, n);
    } else {
      // QGS/4 consecutive lanes hold one group (dim % QGS == 0 and whole waves:
      // a group is entirely live or entirely past the row); every lane takes
      // part in the DPP butterfly, or, in a wave holding a NaN or an Inf, in
      // the reference's ordered vmaxps tree (rmsnorm_quantize_kernel.inc:158-186).
      constexpr int LPG = QGS / 4;
      float m = lane_absmax4(n);
      float scale, recip;
      uint32_t codes;
      if (!wave_any_nonfinite(m)) {
        m = (LPG == 8) ? group8_max(m) : group16_max(m);
        q8_scale_finite(m, scale, recip);
        codes = pack4_codes_finite(n, recip);
      } else {
        q8_scale(q8_floor(group_absmax_tree<QGS>(n)), scale, recip);
        codes = pack4_codes_full(n, recip);
      }
      if (live(k)) {
        const size_t cw = (r * (size_t)dim + i) >> 2;  // dword of 4 codes
        st_stream_u32(reinterpret_cast<uint32_t *>(q) + cw, codes);
        if ((tid & (LPG - 1)) == 0) st_stream_f32(q_s + r * (size_t)(dim / QGS) + (i / QGS), scale);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// RMSNorm -> Q8 (and its fused-add form) for dim % 32 == 0, 512 <= dim <= 12288.
//
// One row per workgroup of dim/16 threads.  The row is read with coalesced
// dwordx4 loads (thread t: float4 chunks t + k*T, k < 4) and staged in LDS,
// chunk m at float 4*(m + m/4): 16 bytes of padding after every 64, so that
// the quantizer's reads below are free of bank conflicts.  Lanes 0..31 of
// wave 0 replay the reference's 32 FMA chains from LDS, then the exact
// (A+B)+(C+D) + HADD_YMM reduction runs as DPP row shifts (chain_of_lane
// places each partial sum where the shift finds its partner).  Each thread
// then quantizes 16 consecutive elements read back from LDS: the group max is
// a lane-local max and one or two quad DPP steps (4 or 2 lanes per group),
// the scale and reciprocal are computed once per 16 elements, and the 16
// codes leave as one 16-byte store.  The fused-add form writes the updated
// residual back with the loads' layout.  Same operations and order as
// rms_row, so the same bits; with many rows less time than rms_row, whose
// quantizer takes the lanes' steps once per 4 elements ([5000, 4096] RMSNorm ->
// Q8 19.7 us against 21.6, with the add 44.2 against 45.6).  The LDS array is
// declared 16-byte aligned:
// with the element type's 4-byte alignment the compiler splits every float4
// access into two 8-byte ones.  The chains read their elements one register
// set ahead (16 elements; 8 in the fused-add form, which keeps the weights
// live across the chain and would otherwise exceed 64 VGPRs).

// TPB > 0: the block size, known at compile time (the common widths); 0: blockDim.x.
template <int TPB, int QGS, bool ADD>
__global__ __launch_bounds__(TPB ? TPB : 1024) void norm_q8_row16_kernel(int8_t *q, float *q_s, float *x,
                                                                         const float *add, const float *weight,
                                                                         int dim, float eps) {
  extern __shared__ __attribute__((aligned(16))) float row[];  // dim + dim/4 floats; floats 16..19 (padding) hold the scale
  const int t = threadIdx.x;
  const int T = TPB ? TPB : (int)blockDim.x;  // dim / 16
  if constexpr (TPB > 0) dim = 16 * TPB;
  const size_t r = blockIdx.x;
  float *xr = x + r * (size_t)dim;
  float4 w[4], v[4];
  // With the residual add, the weights are requested first: vector memory
  // counters retire in order, and a weight load issued after the residual's
  // stores would wait for them.  Without it they follow the staging.
  if constexpr (ADD) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = *reinterpret_cast<const float4 *>(weight + 16 * t + 4 * k);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = ld_stream4(xr + 4 * (t + k * T));
  if constexpr (ADD) {
    float4 b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) b[k] = ld_stream4(add + r * (size_t)dim + 4 * (t + k * T));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = make_float4(v[k].x + b[k].x, v[k].y + b[k].y, v[k].z + b[k].z, v[k].w + b[k].w);
      st_stream4(xr + 4 * (t + k * T), v[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) *reinterpret_cast<float4 *>(row + padded(t + k * T)) = v[k];
  lds_barrier();
  if (t < 64) {
    const float s0 = rms_scale(padded_row_sumsq<ADD ? 8 : 16, (TPB > 0)>(row, dim), (float)dim, eps);
    if (t == 0) row[16] = s0;
  }
  if constexpr (!ADD) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = *reinterpret_cast<const float4 *>(weight + 16 * t + 4 * k);
  }
  lds_barrier();
  const float s = row[16];
  float n[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 xv = *reinterpret_cast<const float4 *>(row + 20 * t + 4 * k);  // chunks 4t .. 4t+3
    n[4 * k + 0] = (s * xv.x) * w[k].x;
    n[4 * k + 1] = (s * xv.y) * w[k].y;
    n[4 * k + 2] = (s * xv.z) * w[k].z;
    n[4 * k + 3] = (s * xv.w) * w[k].w;
  }
  // Group max: NaN-propagating lane max, then (no NaN or Inf in the wave) an
  // unsigned max over the group's 4 (GS 64) or 2 (GS 32) lanes, else the
  // reference's ordered vmaxps tree.
  float m = __builtin_elementwise_maximum(__builtin_fabsf(n[0]), __builtin_fabsf(n[1]));
#pragma unroll
  for (int i = 2; i < 16; ++i) m = __builtin_elementwise_maximum(m, __builtin_fabsf(n[i]));
  float scale, recip;
  uint32_t c[4];
  if (!wave_any_nonfinite(m)) {
    uint32_t u = __builtin_bit_cast(uint32_t, m);
    u = umax(u, dpp_u<DPP_QUAD_XOR1>(u));
    if constexpr (QGS == 64) u = umax(u, dpp_u<DPP_QUAD_XOR2>(u));
    q8_scale_finite(__builtin_bit_cast(float, u), scale, recip);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      c[k] = pack4_codes_finite(make_float4(n[4 * k], n[4 * k + 1], n[4 * k + 2], n[4 * k + 3]), recip);
  } else {
    q8_scale(q8_floor(group_absmax_tree16<QGS>(n)), scale, recip);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      c[k] = pack4_codes_full(make_float4(n[4 * k], n[4 * k + 1], n[4 * k + 2], n[4 * k + 3]), recip);
  }
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 cv = {c[0], c[1], c[2], c[3]};
  __builtin_nontemporal_store(cv, reinterpret_cast<u4 *>(q + r * (size_t)dim) + t);
  // every lane of the group stores the same scale to the same address (one store, no branch)
  st_stream_f32(q_s + r * (size_t)(dim / QGS) + t / (QGS / 16), scale);
}

// Waves per SIMD: full CUs for many rows; 8 chunks of residual, add and weights need 128 VGPRs.
static constexpr int row_waves(int kmax, bool add, bool few) { return few ? 1 : (kmax == 8 && add ? 4 : 8); }

template <int TPR, int KMAX, bool ADD, bool LEFT, bool FEW>
__global__ __launch_bounds__(TPR, row_waves(KMAX, ADD, FEW)) void rmsnorm_row_kernel(float *o, float *x,
                                                                                     const float *add,
                                                                                     const float *weight, int dim,
                                                                                     float eps) {
  rms_row<TPR, KMAX, ADD, 0, LEFT, FEW>(o, nullptr, nullptr, x, add, weight, dim, eps);
}

template <int TPR, int KMAX, int QGS, bool ADD, bool FEW>
__global__ __launch_bounds__(TPR, FEW ? 1 : 8) void rmsnorm_q8_row_kernel(int8_t *q, float *q_s, float *x,
                                                                          const float *add, const float *weight,
                                                                          int dim, float eps) {
  rms_row<TPR, KMAX, ADD, QGS, false, FEW>(nullptr, q, q_s, x, add, weight, dim, eps);
}

// Many rows, staged at the padded layout with one 16-byte LDS store per chunk,
// which costs the other rows on the CU less than rms_row's four 4-byte ones and
// its zeros; their waves hide the longer chain.  FIX: dim == 4*TPR*KMAX, every
// chunk live (1024, 2048, 3072 and 4096 at 256 threads; with the add the weights
// are requested ahead of the residual's stores).  Otherwise any dim up to
// 4*TPR*KMAX, each chunk tested against the row's end and the weights read behind
// the scale; LEFT: dim % 32 != 0.  launch_row says which rows take it.
template <int TPR, int KMAX, bool ADD, bool FIX, bool LEFT>
__global__ __launch_bounds__(TPR, 1) void rmsnorm_padded_row_kernel(float *o, float *xin, const float *add,
                                                                 const float *weight, int dim, float eps) {
  static_assert(!(FIX && LEFT), "4*TPR*KMAX is a multiple of 32");
  constexpr bool EARLY_W = FIX && ADD;
  if constexpr (FIX) dim = 4 * TPR * KMAX;
  extern __shared__ __attribute__((aligned(16))) float row[];
  const int tid = threadIdx.x;
  const size_t r = blockIdx.x;
  float *xr = xin + r * (size_t)dim;
  float4 x[KMAX], b[KMAX], w[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int i = 4 * (tid + k * TPR);
    if (FIX || i < dim) {
      x[k] = ld_stream4(xr + i);
      if constexpr (ADD) b[k] = ld_stream4(add + r * (size_t)dim + i);
    }
  }
  if constexpr (EARLY_W) {
#pragma unroll
    for (int k = 0; k < KMAX; ++k) w[k] = *reinterpret_cast<const float4 *>(weight + 4 * (tid + k * TPR));
  }
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int i = 4 * (tid + k * TPR);
    if (FIX || i < dim) {
      if constexpr (ADD) {
        x[k] = make_float4(x[k].x + b[k].x, x[k].y + b[k].y, x[k].z + b[k].z, x[k].w + b[k].w);
        st_stream4(xr + i, x[k]);
        // With a single live chunk the compiler rewrites this store into an ordinary one unless it is
        // pinned here ([513, 1024] 3.16 us, as an ordinary store 3.46).
        if constexpr (FIX && KMAX == 1) asm volatile("" ::: "memory");
      }
      *reinterpret_cast<float4 *>(row + padded(tid + k * TPR)) = x[k];
    }
  }
  __syncthreads();
  // floats 16..19 of the padded layout are padding: the scale goes there
  if (tid < 64) {
    const float s0 = rms_scale(padded_row_sumsq<8, false, LEFT>(row, dim), (float)dim, eps);
    if (tid == 0) row[16] = s0;
  }
  __syncthreads();
  const float s = row[16];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int i = 4 * (tid + k * TPR);
    if (FIX || i < dim) {
      if constexpr (!EARLY_W) w[k] = *reinterpret_cast<const float4 *>(weight + i);
      st_stream4(o + r * (size_t)dim + i, make_float4((s * x[k].x) * w[k].x, (s * x[k].y) * w[k].y,
                                                      (s * x[k].z) * w[k].z, (s * x[k].w) * w[k].w));
    }
  }
}

// LDS bytes of the padded layout: up to the last chunk, and at least the scale's place.
static unsigned padded_bytes(int dim) {
  const int m = dim / 4 - 1, end = 4 * (m + (m >> 2)) + 4, last_pad = dim % 16 ? end : dim + dim / 4;
  return 4u * (unsigned)(last_pad < 20 ? 20 : last_pad);
}

// Calls go(tpr, kmax) with the shape as compile-time constants: kmax chunks per
// thread, the fewest whole waves that hold dim floats.  False, and no call,
// where that leaves more than the last chunk partly past the row's end
// (rms_row tests only the last one) or the waves are outside [MIN_WAVES,
// MAX_WAVES], the ones built.
template <int KMAX, int MIN_WAVES, int MAX_WAVES, typename Go>
static bool with_threads(int dim, Go go) {
  const int waves = (dim / 4 + 64 * KMAX - 1) / (64 * KMAX);
  if (waves < MIN_WAVES || waves > MAX_WAVES || 64 * waves * (KMAX - 1) > dim / 4) return false;
  using std::integral_constant;
  constexpr integral_constant<int, KMAX> k{};
  auto call = [&](auto tpr) {
    constexpr int waves_c = decltype(tpr)::value / 64;
    if constexpr (waves_c >= MIN_WAVES && waves_c <= MAX_WAVES) go(tpr, k);
  };
  switch (waves) {
    case 1: call(integral_constant<int, 64>{}); break;
    case 2: call(integral_constant<int, 128>{}); break;
    case 3: call(integral_constant<int, 192>{}); break;
    case 4: call(integral_constant<int, 256>{}); break;
    case 5: call(integral_constant<int, 320>{}); break;
    case 6: call(integral_constant<int, 384>{}); break;
    case 7: call(integral_constant<int, 448>{}); break;
    case 8: call(integral_constant<int, 512>{}); break;
    case 9: call(integral_constant<int, 576>{}); break;
    case 10: call(integral_constant<int, 640>{}); break;
    case 11: call(integral_constant<int, 704>{}); break;
    case 12: call(integral_constant<int, 768>{}); break;
    case 13: call(integral_constant<int, 832>{}); break;
    case 14: call(integral_constant<int, 896>{}); break;
    case 15: call(integral_constant<int, 960>{}); break;
    default: call(integral_constant<int, 1024>{}); break;
  }
  return true;
}

// Calls launch(first row, rows) over all rows, one workgroup of tpr threads per
// row.  HIP refuses a grid dimension of 2^32 threads or more, so more rows than
// that go in several launches.
template <typename Launch>
static void by_rows(int rows, int tpr, Launch launch) {
  const int most = (int)(0xFFFFFFFFu / (unsigned)tpr);
  for (int first = 0; first < rows;) {
    const int n = rows - first < most ? rows - first : most;
    launch(first, n);
    first += n;
  }
}

// At most one row per CU: what counts is a row's own latency.
constexpr int kFewRows = 256;

template <int N>
using Int = std::integral_constant<int, N>;

// The row's shape.  Each line follows the times of [rows, dim] on one MI355X (cold
// rows, launches from a graph; in brackets the form it is preferred to).
//
// dim % 32 == 0, at most 256 rows: chains, one chunk per thread up to 1024
// floats, two up to 8192, four beyond and at 4096 and 8192 (fewer waves to gather
// at the barriers: [8, 4096] 3.03 us against 3.22 with two).
//
// More rows: chains where a row still waits mostly for itself, the padded layout,
// whose rows cost the CU less LDS and fewer instructions, where a CU's rows wait for
// each other:
//  - 1024, 2048, 3072 and 4096 floats: the fixed length (so 256 without the add:
//    its one chunk per thread needs no test);
//  - below 1024 with the add: chains with the few-row registers up to six rows per
//    CU ([1300, 832] 4.6 us [many-row registers 4.9]), then padded, 256 threads up to
//    eight rows per CU ([1700, 640] 4.5 [4.8]), a wave per row ([2500, 896] 7.4 [8.5],
//    [5000, 544] 8.5 [9.4]) until 8192 one-wave rows fill the GPU, chains beyond;
//    without it chains, and a padded wave per row above 5000 rows ([8192, 640] 7.5
//    [8.7]; 320 and 480 floats: at 6145 to 8191 rows);
//  - below 2048: one chunk per thread, without the add two from four rows per CU on;
//    with it padded, 256 threads, while a round of rows is more than 4 MB and at most
//    eight share a CU ([1500, 1984] 9.4 [10.3], [1500, 1792] 8.4 [9.5], [769, 1152] 4.0
//    [4.3]);
//  - below 4096: two chunks; padded, 256 threads of four, where that makes all rows
//    resident at once: at two to eight rows per CU with the add (six above 3072
//    floats, [1000, 2304] 7.7 [8.4]), four to eight without ([1500, 4032] 8.2 [10.8],
//    2560 and less from five on); three chunks and the few-row registers with
//    the add at up to two rows per CU ([400, 2304] 4.1 [5.0]);
//  - below 8192: two chunks; padded, 256 threads of eight, where that makes all rows
//    resident, with the add at 449 to 1024 rows and, up to 5376 floats, again in the
//    last part of the second round ([1000, 5376] 15.8 [17.1], [1280, 4288] 15.9 [17.6]),
//    without it up to the rows whose LDS fits ([1300, 5376] 9.9 [12.3], [1000, 4864]
//    7.7 [9.7]); eight chunks of chains below those where the width allows it;
//  - beyond: four chunks; with the add up to two rows per CU padded, 256 threads of
//    16 ([400, 12288] 16.2 [17.7]; at 8192 and 16384 eight chunks of chains), and
//    above three rows per CU and 12288 floats the few-row registers ([1000, 14336] 42.8
//    [46.8]; 2% slower at 16384); eight chunks at two to three rows per CU where
//    two rows of 1024 threads leave a third waiting ([700, 10112] RMSNorm 9.9 [13.8],
//    with the add 21.2 [23.2]).
//
// dim % 32 != 0 (add only; no model has such a width): padded, with half the
// threads where that makes all rows resident ([1000, 5000] 16.0 us [17.1 with natural
// layout, 18.9 with chains], [1500, 1032] 6.5 [8.5 with 512 threads and chains]);
// chains from 136 to 1024 floats at up to six rows per CU ([600, 904] 3.7 [4.3]),
// at 2056 to 8184 and above 14336 at up to one row per CU ([1, 16376] 8.8 [10.5]).
template <bool ADD>
static bool launch_row(float *o, float *x, const float *add, const float *weight, int rows, int dim, float eps,
                       hipStream_t stream) {
  auto launch = [&](auto kernel, int tpr, unsigned lds) {
    by_rows(rows, tpr, [&](int first, int n) {
      const size_t at = (size_t)first * (size_t)dim;
      enqueue(kernel, dim3(n), dim3(tpr), lds, stream, o + at, x + at, ADD ? add + at : add, weight, dim, eps);
    });
    return true;
  };
  auto chains = [&](auto tpr, auto kmax, auto leftover, auto regs) {
    constexpr int TPR = decltype(tpr)::value, K = decltype(kmax)::value;
    constexpr bool LEFT = decltype(leftover)::value, FEW = decltype(regs)::value;
    return launch(rmsnorm_row_kernel<TPR, K, ADD, LEFT, FEW>, TPR,
                  ChainLayout<TPR, K, LEFT, row_chain_u(K, FEW)>::kBytes);
  };
  auto padded_rows = [&](auto tpr, auto kmax, auto leftover) {
    constexpr int TPR = decltype(tpr)::value, K = decltype(kmax)::value;
    return launch(rmsnorm_padded_row_kernel<TPR, K, ADD, false, decltype(leftover)::value>, TPR, padded_bytes(dim));
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  if constexpr (ADD) {
    if (dim % 32) {
      auto pad = [&](auto tpr, auto kmax) { return padded_rows(tpr, kmax, yes); };
      auto left = [&](auto tpr, auto kmax) { return chains(tpr, kmax, yes, no); };
      if (dim <= 256) return dim <= 128 || rows == 1 ? pad(Int<64>{}, Int<1>{}) : left(Int<64>{}, Int<1>{});
      if (dim <= 1024) {
        if (rows <= 6 * kFewRows ? rows > 1 || dim > 704 : rows > 6144 && dim > 512) return left(Int<256>{}, Int<1>{});
        if (rows <= 2048) return pad(Int<256>{}, Int<1>{});
        return dim <= 512 ? pad(Int<64>{}, Int<2>{}) : pad(Int<64>{}, Int<4>{});
      }
      if (dim <= 2048) return rows <= 4 * kFewRows ? pad(Int<512>{}, Int<1>{}) : pad(Int<256>{}, Int<2>{});
      const bool half = rows > 2 * kFewRows && rows <= 8 * kFewRows;
      if (dim <= 4096) {
        if (rows <= kFewRows) return left(Int<512>{}, Int<2>{});
        return half ? pad(Int<256>{}, Int<4>{}) : pad(Int<512>{}, Int<2>{});
      }
      if (dim <= 8192) {
        if (rows <= kFewRows) return left(Int<1024>{}, Int<2>{});
        return half ? pad(Int<256>{}, Int<8>{}) : pad(Int<512>{}, Int<4>{});
      }
      if (rows <= kFewRows && dim > 14336) return left(Int<1024>{}, Int<4>{});
      return rows > 384 && rows <= 576 ? pad(Int<256>{}, Int<16>{}) : pad(Int<1024>{}, Int<4>{});
    }
  }
  auto few = [&](auto tpr, auto kmax) { return chains(tpr, kmax, no, yes); };
  auto many = [&](auto tpr, auto kmax) { return chains(tpr, kmax, no, no); };
  auto pad = [&](auto tpr, auto kmax) { return padded_rows(tpr, kmax, no); };
  if (rows <= kFewRows) {
    if (dim <= 1024) return with_threads<1, 1, 4>(dim, few);
    if (dim == 4096) return few(Int<256>{}, Int<4>{});
    if (dim == 8192) return few(Int<512>{}, Int<4>{});
    return dim < 8192 ? with_threads<2, 3, 16>(dim, few) : with_threads<4, 9, 16>(dim, few);
  }
  auto fixed = [&](auto tpr, auto kmax) {
    constexpr int TPR = decltype(tpr)::value;
    return launch(rmsnorm_padded_row_kernel<TPR, decltype(kmax)::value, ADD, true, false>, TPR, padded_bytes(dim));
  };
  if constexpr (ADD) {
    if (dim <= 1024 && rows <= 6 * kFewRows) return with_threads<1, 1, 4>(dim, few);
  } else {
    if (dim == 256) return fixed(Int<64>{}, Int<1>{});
  }
  switch (dim) {
    case 1024: return fixed(Int<256>{}, Int<1>{});
    case 2048: return fixed(Int<256>{}, Int<2>{});
    case 3072: return fixed(Int<256>{}, Int<3>{});
    case 4096: return fixed(Int<256>{}, Int<4>{});
  }
  if (dim < 1024) {
    if constexpr (ADD)
      if (dim > 512 && rows <= 2048) return pad(Int<256>{}, Int<1>{});
    if (dim > 512 && (ADD ? rows < 8192 : rows > 5000)) return pad(Int<64>{}, Int<4>{});
    if (rows > 2048 && dim > 256) {
      if constexpr (!ADD)
        if (dim <= 512 && rows > 6144 && rows < 8192) return pad(Int<64>{}, Int<2>{});
      if (dim <= 512) return many(Int<64>{}, Int<2>{});
      if (dim <= 768) return many(Int<64>{}, Int<3>{});
      if constexpr (!ADD) return many(Int<64>{}, Int<4>{});
    }
    if constexpr (ADD)
      return dim <= 512 ? with_threads<1, 1, 2>(dim, many) : many(Int<256>{}, Int<1>{});
    else
      return with_threads<1, 1, 4>(dim, many);
  }
  if (dim < 2048) {
    if constexpr (ADD)
      return rows > 2 * kFewRows && rows <= 8 * kFewRows && rows * dim > 1 << 20 ? pad(Int<256>{}, Int<2>{})
                                                                                 : with_threads<1, 5, 8>(dim, many);
    else
      return rows <= 4 * kFewRows ? with_threads<1, 5, 8>(dim, many) : with_threads<2, 3, 4>(dim, many);
  }
  if (dim < 4096) {
    if (rows > (ADD ? 2 : dim <= 2560 ? 5 : 4) * kFewRows && rows <= (ADD && dim > 3072 ? 6 : 8) * kFewRows)
      return pad(Int<256>{}, Int<4>{});
    if constexpr (ADD)
      if (rows <= 2 * kFewRows && dim <= 3840) return with_threads<3, 3, 6>(dim, few);
    return with_threads<2, 5, 8>(dim, many);
  }
  if (dim < 8192) {
    // rows of the padded layout that are resident at once: 5 bytes of LDS a float, 68 VGPRs (seven workgroups)
    const int on_cu = 160 * 1024 / (5 * dim), resident = kFewRows * (on_cu < 7 ? on_cu : 7);
    if (ADD ? (rows > 448 && rows <= 4 * kFewRows) ||
                  (dim < 5632 && rows > 1152 && rows <= (dim <= 5120 ? 1536 : 1280))
            : rows <= resident && rows > (dim <= 4608 ? 3 : dim < 5376 ? 2 : 4) * kFewRows)
      return pad(Int<256>{}, Int<8>{});
    if ((ADD ? rows <= 448 : rows > 2 * kFewRows && rows <= 4 * kFewRows) && with_threads<8, 3, 4>(dim, many))
      return true;
    return with_threads<2, 9, 16>(dim, many);
  }
  if constexpr (ADD) {
    if (rows <= 2 * kFewRows) {
      if (dim == 8192) return many(Int<256>{}, Int<8>{});
      if (dim == 16384) return many(Int<512>{}, Int<8>{});
      return pad(Int<256>{}, Int<16>{});
    }
    if (rows <= 3 * kFewRows && dim > 8192 && dim <= 10240 && with_threads<8, 5, 5>(dim, many)) return true;
    if (rows > 3 * kFewRows && dim > 12288 && dim < 16384) return with_threads<4, 13, 16>(dim, few);
  } else {
    if (rows > 2 * kFewRows && rows <= 3 * kFewRows && dim > 9216 && dim < 12288 && with_threads<8, 5, 6>(dim, many))
      return true;
  }
  return with_threads<4, 8, 16>(dim, many);
}

bool launch_fused_add_rmsnorm(float *o, float *residual, const float *add, const float *weight, int rows, int dim,
                              float eps, hipStream_t stream) {
  return launch_row<true>(o, residual, add, weight, rows, dim, eps, stream);
}

bool launch_rmsnorm(float *o, const float *x, const float *weight, int rows, int dim, float eps, hipStream_t stream) {
  return launch_row<false>(o, const_cast<float *>(x), nullptr, weight, rows, dim, eps, stream);
}

// RMSNorm -> Q8 as one row of chains: at most 256 rows, and more where
// norm_q8_row16_kernel cannot (below 512 or above 12288 floats, codes off their
// 16-byte boundary).  More rows, from [rows, dim] with unaligned codes (in brackets
// the shape that the line is preferred to):
//  - one chunk per thread, up to 4096 floats with the add and while few rows share a
//    CU without it, keeps the few-row registers at any row count ([100000, 256]
//    28.9 us [many-row registers 31.8], [20000, 1024] 23.2 [25.5]);
//  - without the add then two chunks up to 2048 floats and four beyond, many-row
//    registers ([2048, 3840] 9.8 [one chunk 13.0], [1000, 8192] 9.9 [two 15.3]);
//  - with the add two chunks up to 5632 floats, four beyond, with the few-row
//    registers up to 8192 ([5000, 8192] 91 [two chunks 104]), at 16384 ([400, 16384]
//    21.7 [24.1]), above 12288 from three rows per CU on and below it at GS 32.
template <int QGS, bool ADD>
static bool launch_q8_row(int8_t *q, float *q_s, float *x, const float *add, const float *weight, int rows, int dim,
                          float eps, hipStream_t stream) {
  auto go = [&](auto tpr, auto kmax, auto regs) {
    constexpr int TPR = decltype(tpr)::value, K = decltype(kmax)::value;
    constexpr bool FEW = decltype(regs)::value;
    by_rows(rows, TPR, [&](int first, int n) {
      const size_t at = (size_t)first * (size_t)dim;
      enqueue(rmsnorm_q8_row_kernel<TPR, K, QGS, ADD, FEW>, dim3(n), dim3(TPR),
              ChainLayout<TPR, K, false, row_chain_u(K, FEW)>::kBytes, stream, q + at, q_s + at / QGS, x + at,
              ADD ? add + at : add, weight, dim, eps);
    });
    return true;
  };
  auto few = [&](auto tpr, auto kmax) { return go(tpr, kmax, std::true_type{}); };
  auto many = [&](auto tpr, auto kmax) { return go(tpr, kmax, std::false_type{}); };
  if (rows > 2048 && dim > 256 && dim <= 512) return many(Int<64>{}, Int<2>{});
  if (dim <= 4096) {
    if constexpr (!ADD) {
      if (dim > 1024 && dim <= 2048 && rows > 4 * kFewRows) return with_threads<2, 3, 4>(dim, many);
      if (dim > 2048 && rows > 2 * kFewRows)
        return with_threads<4, 3, 4>(dim, many) || with_threads<2, 5, 5>(dim, many);
    }
    return with_threads<1, 1, 16>(dim, few);
  }
  if (dim <= 8192) {
    if (rows <= (ADD ? 1 : 2) * kFewRows) return with_threads<2, 9, 16>(dim, few);
    if constexpr (ADD)
      return dim <= 5632 ? with_threads<2, 9, 11>(dim, few) : with_threads<4, 6, 8>(dim, few);
    else
      return with_threads<4, 5, 8>(dim, many);
  }
  const bool few_regs = dim == 16384 || (dim > 12288 && rows > 3 * kFewRows) || (dim < 12288 && QGS == 32);
  if (rows <= kFewRows || (ADD && few_regs)) return with_threads<4, 9, 16>(dim, few);
  return with_threads<4, ADD && QGS == 32 ? 12 : 9, 16>(dim, many);
}

bool launch_rmsnorm_quantize(int8_t *q, float *q_s, float *x, const float *add, const float *weight, int rows,
                             int dim, int gs, float eps, hipStream_t stream) {
  // At most one row per CU takes the row kernel, whose chain is shorter and whose
  // results need no second pass through LDS ([1, 2304] 2.84 -> 2.21 us with the
  // add, [8, 4096] 3.49 -> 3.36); beyond that norm_q8_row16_kernel's quantizer,
  // with a quarter of the instructions, wins ([512, 2560] 5.31 us against 5.59).
  // The 16-elements-per-thread kernel needs the 32 chain lanes (dim >= 512), whole
  // 32-element blocks, 16-byte aligned codes and at most 64 KiB of LDS (5 bytes per element).
  if (rows > kFewRows && dim % 32 == 0 && dim >= 512 && dim <= 12288 && ((uintptr_t)q & 15u) == 0) {
    const dim3 grid(rows), block(dim / 16);
    const unsigned lds = (unsigned)(dim + dim / 4) * sizeof(float);
    auto go = [&](auto kernel) { enqueue(kernel, grid, block, lds, stream, q, q_s, x, add, weight, dim, eps); };
    const bool g32 = gs == 32;
    auto go_tpb = [&](auto tpb) {
      constexpr int TPB = decltype(tpb)::value;
      if (add)
        go(g32 ? norm_q8_row16_kernel<TPB, 32, true> : norm_q8_row16_kernel<TPB, 64, true>);
      else
        go(g32 ? norm_q8_row16_kernel<TPB, 32, false> : norm_q8_row16_kernel<TPB, 64, false>);
    };
    // The block size compiled in for the common model widths: 0.2 to 2.7 points
    // of the HBM peak above the run-time block size at [8192, dim].
    switch (dim) {
      case 2048: go_tpb(std::integral_constant<int, 128>{}); break;
      case 2560: go_tpb(std::integral_constant<int, 160>{}); break;
      case 3072: go_tpb(std::integral_constant<int, 192>{}); break;
      case 3584: go_tpb(std::integral_constant<int, 224>{}); break;
      case 3840: go_tpb(std::integral_constant<int, 240>{}); break;
      case 4096: go_tpb(std::integral_constant<int, 256>{}); break;
      case 5120: go_tpb(std::integral_constant<int, 320>{}); break;
      case 6144: go_tpb(std::integral_constant<int, 384>{}); break;
      case 8192: go_tpb(std::integral_constant<int, 512>{}); break;
      default: go_tpb(std::integral_constant<int, 0>{}); break;
    }
    return true;
  }
  if (add)
    return gs == 32 ? launch_q8_row<32, true>(q, q_s, x, add, weight, rows, dim, eps, stream)
                    : launch_q8_row<64, true>(q, q_s, x, add, weight, rows, dim, eps, stream);
  return gs == 32 ? launch_q8_row<32, false>(q, q_s, x, add, weight, rows, dim, eps, stream)
                  : launch_q8_row<64, false>(q, q_s, x, add, weight, rows, dim, eps, stream);
}

}  // namespace v7g
