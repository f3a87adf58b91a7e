// k_swiglu_q8.hip -- elementwise SwiGLU, SwiGLU -> Q8 and Q8 block quantization, gfx950.
//
// References:
//   .pq_ffn_silu (src/asm/prefill_q8.inc:1159-1166): out = (sigmoid(g)*g)*u
//     with EVAL_SIGMOID (src/asm/v7_macros.inc:98-160);
//   v7d_quantize / v7s_quantize_chunk (src/asm/utility_dispatch.inc:108-212,
//     src/asm/quantize_kernel.inc:44-159): per group of GS floats,
//     wmax = max|x| floored at 127*2^-126, scale = wmax/127 (stored),
//     recip = 1/scale, code = sat(rne(x*recip)) raised to -127; a partial
//     tail group uses the same arithmetic.
//   The SwiGLU -> Q8 chain (src/asm/prefill_q8.inc:1154-1183) quantizes the
//   SwiGLU row; here the SwiGLU values never leave registers.
// The reference group size is 64 (src/asm/v7_core.inc:120); 32-element blocks
// and the other group sizes use the same algorithm.
//
// Vector layout: lane owns 4 consecutive floats (streaming dwordx4 loads of
// gate and up, or x), a power of two of consecutive lanes (1 to 64) forms one
// group, the group max is a lane butterfly inside them (for full groups of 32
// and 64 the reference's ordered vmaxps tree in a wave that holds a NaN or an
// Inf), each lane stores its 4 codes as one dword, and the first lane of the
// group stores the scale.  The divisions of
// the reference (sigmoid's 1/(1+e), wmax/127, 1/scale) are the shorter
// sequences of v7g_device.h that give the same bits for every reachable input.
#include <type_traits>

#include "v7g_device.h"
#include "v7g_internal.h"

namespace v7g {

// One float4 chunk per thread and a grid that covers the array once, with no
// loop: a thread's loads are issued together, many waves keep them in flight,
// and a wave carries no loop or grid-stride bookkeeping (a grid-stride loop
// cost the SwiGLU -> Q8 kernel 20 vector instructions per wave and about 2%
// of its time).  Addresses are the block's uniform base plus a 32-bit lane
// offset (scalar base, vector offset loads).  The element counts the entries
// accept (below 2^40) keep the grid below 2^31 blocks.
constexpr unsigned kStreamBlock = 256;

static unsigned stream_blocks(long long n4) { return (unsigned)((n4 + kStreamBlock - 1) / kStreamBlock); }

__global__ __launch_bounds__(kStreamBlock) void swiglu_f32_kernel(float *out, const float *gate, const float *up,
                                                                  long long n4) {
  const long long c0 = (long long)blockIdx.x * kStreamBlock;  // the block's first chunk (uniform)
  if (c0 + threadIdx.x >= n4) return;
  const unsigned t4 = 4u * threadIdx.x;
  const float4 g = ld_stream4((gate + 4 * c0) + t4);
  const float4 u = ld_stream4((up + 4 * c0) + t4);
  st_stream4((out + 4 * c0) + t4,
             make_float4(swiglu_v7(g.x, u.x), swiglu_v7(g.y, u.y), swiglu_v7(g.z, u.z), swiglu_v7(g.w, u.w)));
}

// Elements n - n%4 .. n-1 (fewer than 4), one thread each.
__global__ void swiglu_f32_tail_kernel(float *out, const float *gate, const float *up, long long start, long long n) {
  long long i = start + threadIdx.x;
  if (i < n) out[i] = swiglu_v7(gate[i], up[i]);
}

void launch_swiglu_f32(float *out, const float *gate, const float *up, long long n, hipStream_t stream) {
  long long n4 = n / 4;
  if (n4 > 0)
    enqueue(swiglu_f32_kernel, dim3(stream_blocks(n4)), dim3(kStreamBlock), 0, stream, out, gate, up, n4);
  if (n % 4)
    enqueue(swiglu_f32_tail_kernel, dim3(1), dim3(4), 0, stream, out, gate, up, n4 * 4, n);
}

// v7s_add_inplace (src/asm/add_kernel.inc:26-49): x = x + y, one vaddps per
// element; streamed like the kernels above.
__global__ __launch_bounds__(kStreamBlock) void add_inplace_kernel(float *x, const float *y, long long n4) {
  const long long c0 = (long long)blockIdx.x * kStreamBlock;
  if (c0 + threadIdx.x >= n4) return;
  const unsigned t4 = 4u * threadIdx.x;
  const float4 a = ld_stream4((x + 4 * c0) + t4);
  const float4 b = ld_stream4((y + 4 * c0) + t4);
  st_stream4((x + 4 * c0) + t4, make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w));
}

__global__ void add_inplace_tail_kernel(float *x, const float *y, long long start, long long n) {
  long long i = start + threadIdx.x;
  if (i < n) x[i] = x[i] + y[i];
}

void launch_add_inplace(float *x, const float *y, long long n, hipStream_t stream) {
  long long n4 = n / 4;
  if (n4 > 0)
    enqueue(add_inplace_kernel, dim3(stream_blocks(n4)), dim3(kStreamBlock), 0, stream, x, y, n4);
  if (n % 4) enqueue(add_inplace_tail_kernel, dim3(1), dim3(4), 0, stream, x, y, n4 * 4, n);
}

// |v| with NaN as zero, as an unsigned integer (orders as the magnitudes do).
__device__ __forceinline__ uint32_t abs_bits_no_nan(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
  return u > 0x7f800000u ? 0u : u;
}

// The largest u over the aligned P lanes of a group, in every lane of it.
template <int P>
__device__ __forceinline__ uint32_t group_umax(uint32_t u) {
  if constexpr (P >= 2) u = umax(u, dpp_u<DPP_QUAD_XOR1>(u));
  if constexpr (P >= 4) u = umax(u, dpp_u<DPP_QUAD_XOR2>(u));
  if constexpr (P >= 8) u = umax(u, dpp_u<DPP_ROW_HALF_MIRROR>(u));
  if constexpr (P >= 16) u = umax(u, dpp_u<DPP_ROW_MIRROR>(u));
  if constexpr (P >= 32)
    u = umax(u, (uint32_t)__builtin_amdgcn_ds_bpermute((__lane_id() ^ 16) << 2, (int)u));
  if constexpr (P >= 64)
    u = umax(u, (uint32_t)__builtin_amdgcn_ds_bpermute((__lane_id() ^ 32) << 2, (int)u));
  return u;
}

__device__ __forceinline__ uint32_t lane_absmax4_no_nan(float4 v) {
  return umax(umax(abs_bits_no_nan(v.x), abs_bits_no_nan(v.y)), umax(abs_bits_no_nan(v.z), abs_bits_no_nan(v.w)));
}

// Flat path: every row length is a multiple of GS (16, 32, 64, 128 or 256: 4 to
// 64 lanes of a wave, powers of two) and the arrays sit on 16-byte (codes:
// 4-byte) boundaries, so groups tile the flat array and group g covers elements
// [g*GS, (g+1)*GS).  GS/4 consecutive lanes hold one group (aligned inside the
// wave, so a group never straddles two waves); their max is a lane butterfly.
// Every other call goes through quantize_q8_group_kernel, whose row arithmetic
// and per-lane bounds would cost 8% here (2048 x 4096 at GS 128: 10.0 us
// against 9.2, and 93.5 us for one thread per group; back to back over buffers
// past the Infinity Cache, one MI355X).
template <int GS, bool SWIGLU>
__global__ __launch_bounds__(kStreamBlock) void quantize_q8_flat_kernel(int8_t *__restrict__ out_q,
                                                                        float *__restrict__ out_s,
                                                                        const float *__restrict__ x,
                                                                        const float *__restrict__ gate,
                                                                        const float *__restrict__ up, long long n4) {
  constexpr int LPG = GS / 4;  // lanes per group
  {
    const long long c0 = (long long)blockIdx.x * kStreamBlock;  // the block's first chunk (uniform)
    const long long c = c0 + threadIdx.x;
    if (c >= n4) return;
    const unsigned t4 = 4u * threadIdx.x;
    float4 v;
    if constexpr (SWIGLU) {
      const float4 g = ld_stream4((gate + 4 * c0) + t4);
      const float4 u = ld_stream4((up + 4 * c0) + t4);
      v = make_float4(swiglu_v7(g.x, u.x), swiglu_v7(g.y, u.y), swiglu_v7(g.z, u.z), swiglu_v7(g.w, u.w));
    } else {
      v = ld_stream4((x + 4 * c0) + t4);
    }
    // absmax: without NaN the vmaxps tree is a plain maximum, a DPP butterfly
    // here; a wave holding a NaN takes the reference's ordered tree instead,
    // and one holding an Inf the same general path (scale Inf, codes 0 / -127).
    float m = lane_absmax4(v);
    float scale, recip;
    uint32_t codes;
    if (!wave_any_nonfinite(m)) {
      m = __builtin_bit_cast(float, group_umax<LPG>(__builtin_bit_cast(uint32_t, m)));
      q8_scale_finite(m, scale, recip);
      codes = pack4_codes_finite(v, recip);
    } else {
      float wmax;
      if constexpr (GS == 32 || GS == 64)
        wmax = group_absmax_tree<GS>(v);
      else
        wmax = __builtin_bit_cast(float, group_umax<LPG>(lane_absmax4_no_nan(v)));
      q8_scale(q8_floor(wmax), scale, recip);
      codes = pack4_codes_full(v, recip);
    }
    st_stream_u32((reinterpret_cast<uint32_t *>(out_q) + c0) + threadIdx.x, codes);
    if ((threadIdx.x & (LPG - 1)) == 0) st_stream_f32((out_s + c0 / LPG) + threadIdx.x / LPG, scale);
  }
}

// Every other row length, group size and alignment: GS in [1, 4096], rows that
// end in a partial group, x off its 16-byte and codes off their 4-byte
// boundary.  P consecutive lanes (a power of two, P >= gs/4 up to 64) hold one
// group of one row, 4 consecutive floats each: one 16-byte load at the float's
// own alignment, the group max over P lanes by lane exchanges, 4 codes as one
// dword at the byte's own alignment.  A lane at the end of a partial group
// reads and writes its last 1 to 3 elements one by one, lanes past it hold
// zeros, which leave the group's max as it is.  LOOP (gs > 256, P = 64): each
// lane walks the group in steps of 256 floats, twice (max, then codes; the
// second read comes from the caches).
//
// The group max of a partial group, and of a full group of any size but 32
// and 64, is the reference's in-order scan (quantize_kernel.inc:119-152:
// vmaxss |x|, wmax), which drops a NaN element and is otherwise the plain
// maximum: order-free.  A full group of 32 or 64 takes the ordered vmaxps tree
// where its wave holds a NaN or an Inf, as in the flat kernel.  The codes of a
// tail group cannot leave [-127.00002, 127.00002] except as NaN, where the
// tail's vmaxss/vminss/vcvtss2si and the vector conversion both give -127, so
// one conversion serves both.
//
// WIDE: 2^31 lanes or more; 64-bit group indices and a grid-stride loop.
//
// Bound by HBM as the flat kernel is, plus the rows' misaligned lines.  One
// thread per group with scalar loads and byte stores (the form before) left
// each wave 64 separate lines per load.  Measured back to back over buffers past
// the Infinity Cache, quantize, one MI355X: rows of 5185 x 2431 at GS 64
// 365 -> 13.9 us (4.6 TB/s), 4096 x 4096 at GS 100 377 -> 21.3 us, at GS 512
// 328 -> 18.7 us, 8192 x 4096 at GS 64 with x off its boundary 997 -> 31.9 us
// (the flat kernel on aligned x: 28.5); 8 x 1119 at GS 32 15.0 -> 4.1 us.
typedef float v7g_f4u __attribute__((ext_vector_type(4), aligned(4)));

template <int P, bool SWIGLU, bool LOOP, bool WIDE>
__global__ __launch_bounds__(kStreamBlock) void quantize_q8_group_kernel(
    int8_t *__restrict__ out_q, float *__restrict__ out_s, const float *__restrict__ x,
    const float *__restrict__ gate, const float *__restrict__ up, unsigned long long magic, unsigned spr, int gs,
    long long row_len, unsigned long long groups) {
  using idx_t = typename std::conditional<WIDE, unsigned long long, unsigned>::type;
  constexpr idx_t kGroupsPerBlock = kStreamBlock / P;
  const int l = threadIdx.x & (P - 1);
  idx_t g0 = (idx_t)blockIdx.x * kGroupsPerBlock;
  do {
    const idx_t gid_raw = g0 + threadIdx.x / P;
    const bool live = gid_raw < (idx_t)groups;
    const idx_t gid = live ? gid_raw : (idx_t)groups - 1;
    idx_t r = gid;  // gid / spr
    if constexpr (WIDE)
      r = gid / spr;
    else if (spr > 1)
      r = (idx_t)__umul64hi((unsigned long long)gid, magic);
    const long long in_row = (long long)(gid - r * spr) * gs;
    const long long start = (long long)r * row_len + in_row;
    const int len = row_len - in_row < gs ? (int)(row_len - in_row) : gs;

    auto chunk = [&](int i) {  // elements i .. i+3 of the group; zeros past its end
      auto ld = [&](const float *p) {
        if (i + 4 <= len) {
          v7g_f4u a;
          if constexpr (LOOP)
            a = *reinterpret_cast<const v7g_f4u *>(p + start + i);
          else
            a = __builtin_nontemporal_load(reinterpret_cast<const v7g_f4u *>(p + start + i));
          return make_float4(a.x, a.y, a.z, a.w);
        }
        return make_float4(i < len ? p[start + i] : 0.f, i + 1 < len ? p[start + i + 1] : 0.f,
                           i + 2 < len ? p[start + i + 2] : 0.f, 0.f);
      };
      if constexpr (SWIGLU) {
        const float4 g = ld(gate), u = ld(up);
        return make_float4(swiglu_v7(g.x, u.x), swiglu_v7(g.y, u.y), swiglu_v7(g.z, u.z), swiglu_v7(g.w, u.w));
      } else {
        return ld(x);
      }
    };
    auto store = [&](int i, uint32_t c) {
      int8_t *q = out_q + start + i;
      if (i + 4 <= len) {
        __builtin_memcpy(q, &c, 4);
      } else {
        if (i < len) q[0] = (int8_t)c;
        if (i + 1 < len) q[1] = (int8_t)(c >> 8);
        if (i + 2 < len) q[2] = (int8_t)(c >> 16);
      }
    };

    float4 v = chunk(4 * l);
    float m = lane_absmax4(v);
    if constexpr (LOOP)
      for (int i = 4 * (l + P); i < len; i += 4 * P) m = __builtin_elementwise_maximum(m, lane_absmax4(chunk(i)));
    float scale, recip;
    const bool finite = !wave_any_nonfinite(m);
    if (finite) {
      q8_scale_finite(__builtin_bit_cast(float, group_umax<P>(__builtin_bit_cast(uint32_t, m))), scale, recip);
    } else {
      uint32_t u = lane_absmax4_no_nan(v);
      if constexpr (LOOP)
        for (int i = 4 * (l + P); i < len; i += 4 * P) u = umax(u, lane_absmax4_no_nan(chunk(i)));
      float wmax = __builtin_bit_cast(float, group_umax<P>(u));
      if constexpr (P == 8 || P == 16) {  // gs 32 or 64: full groups follow the tree
        const float tree = group_absmax_tree<4 * P>(v);
        if (gs == 4 * P && len == gs) wmax = tree;
      }
      q8_scale(q8_floor(wmax), scale, recip);
    }
    if (live) {
      store(4 * l, finite ? pack4_codes_finite(v, recip) : pack4_codes_full(v, recip));
      if constexpr (LOOP)
        for (int i = 4 * (l + P); i < len; i += 4 * P) store(i, pack4_codes_full(chunk(i), recip));
      if (l == 0) out_s[gid] = scale;
    }
    g0 += (idx_t)gridDim.x * kGroupsPerBlock;
  } while (WIDE && g0 < (idx_t)groups);
}

template <int P, bool LOOP>
static void launch_group(int8_t *out_q, float *out_s, const float *x, const float *gate, const float *up, int rows,
                         int row_len, int gs, hipStream_t stream) {
  unsigned long long groups = (unsigned long long)rows * (unsigned)((row_len + (long long)gs - 1) / gs);
  // Without partial groups the rows are one long row.
  const bool one_row = row_len % gs == 0;
  const long long len = one_row ? (long long)rows * row_len : row_len;
  const bool wide = groups * P >= (1ull << 31);
  const unsigned spr = (one_row && !wide) ? (unsigned)groups : (unsigned)((row_len + (long long)gs - 1) / gs);
  const long long arg_len = (one_row && !wide) ? len : row_len;
  const unsigned long long magic = ~0ull / spr + 1ull;  // n / spr == umulhi64(n, magic) for n < 2^32 (spr > 1)
  const unsigned long long per = kStreamBlock / P, all = (groups + per - 1) / per;
  const dim3 grid((unsigned)(all < (1ull << 23) ? all : (1ull << 23)));
  auto go = [&](auto kernel) {
    enqueue(kernel, grid, dim3(kStreamBlock), 0, stream, out_q, out_s, x, gate, up, magic, spr, gs, arg_len, groups);
  };
  if (wide)
    gate ? go(quantize_q8_group_kernel<P, true, LOOP, true>) : go(quantize_q8_group_kernel<P, false, LOOP, true>);
  else
    gate ? go(quantize_q8_group_kernel<P, true, LOOP, false>) : go(quantize_q8_group_kernel<P, false, LOOP, false>);
}

template <int GS>
static void launch_flat(int8_t *out_q, float *out_s, const float *x, const float *gate, const float *up, long long n,
                        hipStream_t stream) {
  const long long n4 = n / 4;
  const dim3 grid(stream_blocks(n4));
  if (gate)
    enqueue((quantize_q8_flat_kernel<GS, true>), grid, dim3(kStreamBlock), 0, stream, out_q, out_s, x, gate,
                       up, n4);
  else
    enqueue((quantize_q8_flat_kernel<GS, false>), grid, dim3(kStreamBlock), 0, stream, out_q, out_s, x,
                       gate, up, n4);
}

static bool aligned(const void *p, size_t a) { return p == nullptr || ((uintptr_t)p % a) == 0; }

void launch_quantize_q8(int8_t *out_q, float *out_s, const float *x, const float *gate, const float *up, int rows,
                        int row_len, int gs, hipStream_t stream) {
  const long long n = (long long)rows * row_len;
  // one lane per 4 elements, fewer than 2^32 (HIP's limit of a grid); beyond it the group kernel's grid-stride loop
  const bool flat = row_len % gs == 0 && n / 4 < (1LL << 32) - 256 && aligned(out_q, 4) && aligned(x, 16) &&
                    aligned(gate, 16) && aligned(up, 16);
  if (flat) {
    auto go = [&](auto g) { launch_flat<decltype(g)::value>(out_q, out_s, x, gate, up, n, stream); };
    switch (gs) {
      case 16: go(std::integral_constant<int, 16>{}); return;
      case 32: go(std::integral_constant<int, 32>{}); return;
      case 64: go(std::integral_constant<int, 64>{}); return;
      case 128: go(std::integral_constant<int, 128>{}); return;
      case 256: go(std::integral_constant<int, 256>{}); return;
    }
  }
  const int widest = gs < row_len ? gs : row_len;  // the longest group
  auto go = [&](auto p, auto loop) {
    launch_group<decltype(p)::value, decltype(loop)::value>(out_q, out_s, x, gate, up, rows, row_len, gs, stream);
  };
  using std::integral_constant;
  if (widest > 256)
    go(integral_constant<int, 64>{}, std::true_type{});
  else if (widest > 128)
    go(integral_constant<int, 64>{}, std::false_type{});
  else if (widest > 64)
    go(integral_constant<int, 32>{}, std::false_type{});
  else if (widest > 32)
    go(integral_constant<int, 16>{}, std::false_type{});
  else if (widest > 16)
    go(integral_constant<int, 8>{}, std::false_type{});
  else if (widest > 8)
    go(integral_constant<int, 4>{}, std::false_type{});
  else if (widest > 4)
    go(integral_constant<int, 2>{}, std::false_type{});
  else
    go(integral_constant<int, 1>{}, std::false_type{});
}

}  // namespace v7g
