// gfx950 (CDNA4, wave64) kernels of the NeuZip bf16 codec.
//
//   nz_split_unpacked_kernel   Manager::split            cuda/high_level.cu:265-321
//   nz_encode_kernel           kernel_aligned_split      cuda/kernels.cuh:62-156
//   nz_encode_long_kernel      + per-chunk exponent histogram, 12-bit frequency
//                              table and its serialized form, then
//                              nvcomp ANS compress       cuda/high_level.cu:103-115
//   nz_compact_kernel          exact-size compaction     cuda/high_level.cu:117-124
//                              (on the device: every record finds its own place)
//   nz_decode_kernel           nvcomp ANS decompress + kernel_aligned_merge fused:
//                              cuda/high_level.cu:184-201, cuda/kernels.cuh:167-217
//
// The whole path is byte/integer work bound by HBM traffic; there is no dense
// contraction, hence no MFMA.  One wavefront decodes one segment with 64
// interleaved rANS states; the exponent never exists in HBM on the decode side.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "nz_format.h"
#include "nz_lookback.h"

#define NZ_RING_WORDS 1024u  // per-wave LDS ring of renormalisation words (NzWaveDec) ...
#define NZ_RING_DWORDS (NZ_RING_WORDS / 2)
#define NZ_RING_WIDE 512u    // ... or of 8-byte entries prepared from them (NzWaveDecOne)
#define NZ_RING_NARROW 256u

// ----------------------------------------------------------------------------
// element-wise split / merge arithmetic
// ----------------------------------------------------------------------------

// Exponent byte and (sign | kept mantissa) field of one bf16 value.  This is the
// closed form of cuda/kernels.cuh:122-137,153-155: round the 15-bit magnitude
// half-up to S kept mantissa bits, the carry running into the exponent and the
// exponent byte wrapping 255 -> 0 exactly like the reference's uint8 store.
template <int S>
__device__ __forceinline__ void nz_split_one(uint32_t v, uint32_t& exp, uint32_t& repr) {
  if constexpr (S == 7) {
    exp = (v >> 7) & 0xFFu;
    repr = ((v >> 8) & 0x80u) | (v & 0x7Fu);
  } else {
    uint32_t a = ((v & 0x7FFFu) + (1u << (6 - S))) & 0x7FFFu;
    exp = a >> 7;
    repr = ((v >> 15) << S) | ((a >> (7 - S)) & ((1u << S) - 1u));
  }
}

// Position of element j (0..7) of an 8-element group inside the group's S+1
// packed bytes, MSB first (cuda/kernels.cuh:86-89): bit offset inside the
// little-endian integer that holds those bytes.
template <int S>
__device__ __forceinline__ constexpr uint32_t nz_field_shift(int j) {
  return 8u * ((uint32_t)(j * (S + 1)) >> 3) + (7u - S - ((uint32_t)(j * (S + 1)) & 7u));
}

// cuda/kernels.cuh:197-206 for a non-NaN result (the float multiply by +-1.0f of
// :213-216 only moves the sign bit into place).
template <int S>
__device__ __forceinline__ uint32_t nz_merge_one(uint32_t exp, uint32_t repr) {
  uint32_t frac = (repr & ((1u << S) - 1u)) << (7 - S);
  uint32_t sign = (repr >> S) & 1u;
  return (sign << 15) | (exp << 7) | frac;
}

__device__ __forceinline__ float nz_bf16_to_f32(uint32_t h) { return __uint_as_float(h << 16); }
// two floats -> two bf16 in one word, round to nearest even, NaN stays NaN: the
// conversion instruction of gfx950 (v_cvt_pk_bf16_f32)
typedef __bf16 nz_bf16x2 __attribute__((ext_vector_type(2)));
typedef float nz_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t nz_f32_to_bf16x2(float lo, float hi) {
  const nz_f32x2 v = {lo, hi};
  const nz_bf16x2 r = __builtin_convertvector(v, nz_bf16x2);
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t nz_f32_to_bf16(float f) { return nz_f32_to_bf16x2(f, 0.0f) & 0xFFFFu; }

// ----------------------------------------------------------------------------
// block normalizers (cuda/kernels.cuh:94-118 on the split side, :208-216 on the
// merge side): every group of 2^log2n consecutive elements is divided by
// 1.m, m = the 7 mantissa bits of the group's largest magnitude, before the
// split, and multiplied by it again after the merge.  The group stores m << 1
// (the top 8 of the 23 fraction bits of the float 1.m).  Division and product
// run in fp32 and round to bf16, nearest even, and give what the reference's
// float expressions give: the exact quotient A / B of two 8-bit significands
// is never closer to a bf16 rounding boundary (odd / 2^k, k <= 8) than
// 1 / (256 B) > 2^-16 of its value (256 A = odd * B has no solution with
// B < 256), gradual underflow included, so an fp32 quotient that is off by a
// few units in its last place rounds to the same bf16 as the correctly rounded
// one.  The division is therefore a multiplication by the hardware reciprocal
// of 1.m (one unit in the last place).
// ----------------------------------------------------------------------------
struct NzNorm {
  const uint8_t* bytes;  // one per group, null when the tensor is not normalized
  uint32_t log2n;
};

__device__ __forceinline__ float nz_norm_base(uint32_t byte) {
  return __uint_as_float(0x3F800000u | (byte << 15));
}
__device__ __forceinline__ uint32_t nz_norm_div(uint32_t h, uint32_t byte) {
  return nz_f32_to_bf16(nz_bf16_to_f32(h) * __builtin_amdgcn_rcpf(nz_norm_base(byte)));
}
__device__ __forceinline__ uint32_t nz_norm_mul(uint32_t h, uint32_t byte) {
  return nz_f32_to_bf16(nz_bf16_to_f32(h) * nz_norm_base(byte));
}

// The group bytes of the 8 consecutive elements that start at e0 (a multiple of
// 8), one per element: byte j of the result belongs to element e0 + j.  With
// groups of 8 elements or more there is only one, in byte 0.
__device__ __forceinline__ uint64_t nz_norm_load8(const NzNorm& nm, uint64_t e0) {
  if (nm.log2n >= 3) return nm.bytes[e0 >> nm.log2n];
  if (nm.log2n == 0) return *reinterpret_cast<const uint64_t*>(nm.bytes + e0);
  if (nm.log2n == 1) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(nm.bytes + (e0 >> 1));
    return (uint64_t)__builtin_amdgcn_perm(w, w, 0x01010000u) |
           ((uint64_t)__builtin_amdgcn_perm(w, w, 0x03030202u) << 32);
  }
  const uint32_t w = *reinterpret_cast<const uint16_t*>(nm.bytes + (e0 >> 2));
  return (uint64_t)((w & 0xFFu) * 0x01010101u) | ((uint64_t)((w >> 8) * 0x01010101u) << 32);
}

// 8 bf16 values times (MUL) or divided by their group factors; `nb` holds the
// group byte of every element (all the same when a group has 8 elements or more:
// `same`, which saves seven of the eight factor set-ups)
template <bool MUL>
__device__ __forceinline__ uint4 nz_scale8(const uint4 v, const uint64_t nb, const bool same) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t o[4];
  const auto factor = [](uint32_t byte) {
    const float base = nz_norm_base(byte);
    return MUL ? base : __builtin_amdgcn_rcpf(base);
  };
  if (same) {
    const float f = factor((uint32_t)nb & 0xFFu);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float lo = __uint_as_float(w[k] << 16), hi = __uint_as_float(w[k] & 0xFFFF0000u);
      o[k] = nz_f32_to_bf16x2(lo * f, hi * f);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float f0 = factor((uint32_t)(nb >> (16 * k)) & 0xFFu);
      const float f1 = factor((uint32_t)(nb >> (16 * k + 8)) & 0xFFu);
      const float lo = __uint_as_float(w[k] << 16), hi = __uint_as_float(w[k] & 0xFFFF0000u);
      o[k] = nz_f32_to_bf16x2(lo * f0, hi * f1);
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

#ifndef NZ_TEMPLATES_ONLY
// One byte per group: the mantissa of the largest magnitude (patterns of |x|
// order like the values).  A workgroup covers 2048 elements, a multiple of
// every group size.
__global__ __launch_bounds__(256) void nz_absmax_kernel(const uint16_t* __restrict__ in, uint64_t n,
                                                        uint32_t log2n, uint8_t* __restrict__ norm) {
  __shared__ uint32_t smax[256];
  const uint32_t tid = threadIdx.x;
  const uint64_t blk0 = (uint64_t)blockIdx.x * 2048;
  const uint64_t e0 = blk0 + (uint64_t)tid * 8;
  uint32_t mag[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) mag[j] = 0;
  if (e0 + 8 <= n) {
    const uint4 v = *reinterpret_cast<const uint4*>(in + e0);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) mag[j] = (w[j >> 1] >> (16 * (j & 1))) & 0x7FFFu;
  } else {
    for (uint32_t j = 0; j < 8 && e0 + j < n; ++j) mag[j] = in[e0 + j] & 0x7FFFu;
  }
  if (log2n < 3) {
    const uint32_t gs = 1u << log2n;
    for (uint32_t q = 0; q < 8; q += gs) {
      if (e0 + q >= n) break;
      uint32_t m = 0;
      for (uint32_t j = 0; j < gs; ++j) m = mag[q + j] > m ? mag[q + j] : m;
      norm[(e0 + q) >> log2n] = (uint8_t)((m & 0x7Fu) << 1);
    }
    return;
  }
  uint32_t m8 = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) m8 = mag[j] > m8 ? mag[j] : m8;
  // a group is `per` consecutive threads: butterfly inside the wavefront, then
  // (groups of 1024 elements: two wavefronts) through LDS
  const uint32_t per = 1u << (log2n - 3);
  for (uint32_t o = 1; o < per && o < 64; o <<= 1) {
    const uint32_t other = (uint32_t)__shfl_xor((int)m8, (int)o, 64);
    m8 = other > m8 ? other : m8;
  }
  if (per > 64) {
    if ((tid & 63) == 0) smax[tid >> 6] = m8;
    __syncthreads();
    const uint32_t other = smax[(tid >> 6) ^ 1u];
    m8 = other > m8 ? other : m8;
  }
  if ((tid & (per - 1)) == 0 && e0 < n) norm[e0 >> log2n] = (uint8_t)((m8 & 0x7Fu) << 1);
}

#endif  // NZ_TEMPLATES_ONLY

__device__ __forceinline__ uint32_t nz_lane_id() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

__device__ __forceinline__ uint32_t nz_rank_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// inclusive prefix sum over the 64 lanes of a wavefront
// Inclusive prefix sum over the 64 lanes with data-parallel-primitive moves:
// four shifted adds inside each row of 16 lanes, then the last lane of row 0
// and 2 is added to rows 1 and 3, and lane 31 to rows 2 and 3.
__device__ __forceinline__ uint32_t nz_wave_scan(uint32_t v, uint32_t lane) {
  (void)lane;
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  // row_bcast:31
  return v;
}
// the next power of two
__host__ __device__ __forceinline__ constexpr uint32_t nz_pow2(uint32_t v) { return v <= 1 ? 1u : v <= 2 ? 2u : v <= 4 ? 4u : 8u; }

// Sums of MR (up to 8) floats over the 64 lanes, all at once; the lane for which nz_sum_lane
// holds gets the total of v[nz_sum_index(lane)], where there is one.
// Lanes 1 apart are added first, then those 2, 4, 8, 16 and 32 apart: one tree for every MR,
// so a value's total does not depend on how many are summed beside it, and it stays
// the same from version to version.  The steps of 1, 2 and 16 put one half of the values that are
// left into each half of the lanes (eight values: 25 instructions or so instead of eight times seven).
// Those of 4 and 8 are rotations of the row, which make the right pairs in the lanes with bit 2 set.
// (Eight rows through the Linears of a block of width 4096: 243.6 us.  Steps of 32, 16, 8, 1, 2
// and 4, all of the first three exchanges, took 243.0 and gave other bits.)
template <int MR>
__device__ __forceinline__ float nz_wave_sums(const float (&v)[MR], uint32_t lane) {
  static_assert(MR >= 1 && MR <= 8, "");
  const auto dpp = [](float f, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(f), decltype(ctrl)::value, 0xF, 0xF, true));
  };
  constexpr int P = nz_pow2(MR), A = P > 1 ? P / 2 : 1, B = A > 1 ? A / 2 : 1;
  // lo + its partner's in the lower half of the lanes, hi + its partner's in the upper
  const auto halves = [&](float lo, float hi, bool upper, auto ctrl) {
    const float own = upper ? hi : lo, other = upper ? lo : hi;
    return own + dpp(other, ctrl);
  };
  using Pair = std::integral_constant<int, 0xB1>;  // quad_perm:[1,0,3,2]
  using Quad = std::integral_constant<int, 0x4E>;  // quad_perm:[2,3,0,1]
  float a[A], b[B];
#pragma unroll
  for (int m = 0; m < A; ++m)
    if (P > 1 && m + A < MR) a[m] = halves(v[m], v[m + A < MR ? m + A : m], lane & 1u, Pair{});
    else a[m] = v[m] + dpp(v[m], Pair{});
#pragma unroll
  for (int m = 0; m < B; ++m) {
    if (A > 1) b[m] = halves(a[m], a[m + B < A ? m + B : m], lane & 2u, Quad{});
    else b[m] = a[m] + dpp(a[m], Quad{});
    b[m] += dpp(b[m], std::integral_constant<int, 0x124>{});  // row_ror:4
    b[m] += dpp(b[m], std::integral_constant<int, 0x128>{});  // row_ror:8
  }
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(b[0]), __float_as_uint(b[B - 1]), false, false);
  const uint32_t t = __float_as_uint(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(t, t, false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
// the value whose total a lane has, and whether it is the lane that is asked for it
template <int MR>
__device__ __forceinline__ uint32_t nz_sum_index(uint32_t lane) {
  constexpr uint32_t P = nz_pow2(MR);
  return P == 8   ? 4 * (lane & 1) + (lane & 2) + (lane >> 4 & 1)
         : P == 4 ? 2 * (lane & 1) + (lane >> 1 & 1)
         : P == 2 ? lane & 1
                  : 0u;
}
template <int MR>
__device__ __forceinline__ bool nz_sum_lane(uint32_t lane) {
  constexpr uint32_t P = nz_pow2(MR), which = P == 8 ? 0x13u : P == 4 ? 3u : P == 2 ? 1u : 0u;
  return (lane & ~which) == 4u && nz_sum_index<MR>(lane) < (uint32_t)MR;
}

__device__ __forceinline__ uint32_t nz_get12(const uint8_t* p, uint32_t i) {
  uint32_t bit = 12u * i;
  const uint8_t* q = p + (bit >> 3);
  uint32_t w = (uint32_t)q[0] | ((uint32_t)q[1] << 8);
  return (w >> (bit & 4u)) & 0xFFFu;
}

#ifndef NZ_TEMPLATES_ONLY
// ----------------------------------------------------------------------------
// Manager::split: unpacked exponent and sign|mantissa bytes, precision 7 always
// (cuda/high_level.cu:289-296 forces f_bits_save = 7).
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void nz_split_unpacked_kernel(const uint16_t* __restrict__ in,
                                                                uint64_t n,
                                                                uint8_t* __restrict__ exps,
                                                                uint8_t* __restrict__ fracs,
                                                                const NzNorm nm) {
  uint64_t i0 = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i0 >= n) return;
  if (i0 + 8 <= n) {
    uint4 v = *reinterpret_cast<const uint4*>(in + i0);
    if (nm.bytes) v = nz_scale8<false>(v, nz_norm_load8(nm, i0), nm.log2n >= 3);
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint64_t e = 0, f = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t h = (w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu, ex, rp;
      nz_split_one<7>(h, ex, rp);
      e |= (uint64_t)ex << (8 * j);
      f |= (uint64_t)rp << (8 * j);
    }
    *reinterpret_cast<uint64_t*>(exps + i0) = e;
    *reinterpret_cast<uint64_t*>(fracs + i0) = f;
  } else {
    for (uint64_t i = i0; i < n; ++i) {
      uint32_t ex, rp, h = in[i];
      if (nm.bytes) h = nz_norm_div(h, nm.bytes[i >> nm.log2n]);
      nz_split_one<7>(h, ex, rp);
      exps[i] = (uint8_t)ex;
      fracs[i] = (uint8_t)rp;
    }
  }
}

#endif  // NZ_TEMPLATES_ONLY

// ----------------------------------------------------------------------------
// encode: one workgroup per chunk
// ----------------------------------------------------------------------------
//
// Two kernels share the pieces below.  nz_encode_kernel (segments of up to
// NZ_ENC_MAX_LANE_SYMS symbols per lane, which covers every geometry the
// library picks by itself): wavefront k of the workgroup splits segment k of
// the chunk, keeps the exponent bytes of its lanes in registers, and codes
// them from there once the chunk's table exists: the exponents never reach
// memory.  nz_encode_long_kernel (longer segments): all wavefronts split the
// chunk and park the exponents in scratch, then one wavefront per segment
// codes them from there.

#define NZ_ENC_MAX_LANE_SYMS 288u  // 36 groups of 8 symbols per lane: what fits the registers of four wavefronts per SIMD
#define NZ_ENC_LONG_THREADS 1024u

// f(constant I) for I = FROM, FROM + STEP, ... while I < TO (or, with a negative
// step, while I >= TO): straight-line code with compile-time indices, so that
// a register array indexed by I never needs an address
template <int I>
struct NzConst {
  static constexpr int value = I;
};
template <int FROM, int TO, int STEP, class F>
__device__ __forceinline__ void nz_static_for(F&& f) {
  if constexpr ((STEP > 0 && FROM < TO) || (STEP < 0 && FROM >= TO)) {
    f(NzConst<FROM>{});
    nz_static_for<FROM + STEP, TO, STEP>(f);
  }
}

// sums / maxima over the workgroup (at most 16 wavefronts), two at a time; `red`: two words per wavefront
template <class Op>
__device__ __forceinline__ void nz_block_pair(uint32_t& a, uint32_t& b, uint32_t* red, Op second) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b = second(b, (uint32_t)__shfl_xor(b, o, 64));
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) reinterpret_cast<uint2*>(red)[threadIdx.x >> 6] = make_uint2(a, b);
  __syncthreads();
  a = b = 0;
  for (uint32_t w = 0; w < blockDim.x / 64; ++w) {
    const uint2 v = reinterpret_cast<const uint2*>(red)[w];
    a += v.x;
    b = second(b, v.y);
  }
}
__device__ __forceinline__ void nz_block_sum_max(uint32_t& a, uint32_t& b, uint32_t* red) {
  nz_block_pair(a, b, red, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
}
__device__ __forceinline__ void nz_block_sum2(uint32_t& a, uint32_t& b, uint32_t* red) {
  nz_block_pair(a, b, red, [](uint32_t x, uint32_t y) { return x + y; });
}

__device__ __forceinline__ uint32_t nz_block_max(uint32_t v, uint32_t* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    uint32_t t = __shfl_xor(v, o, 64);
    v = t > v ? t : v;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t t = 0;
  for (uint32_t w = 0; w < blockDim.x / 64; ++w) t = red[w] > t ? red[w] : t;
  return t;
}

// Histogram of a workgroup, in the dynamic LDS that later holds the word staging:
// 2^copies_log2 copies of 256 counters, one per lane modulo their number, the copies
// of a symbol next to each other.  A wavefront's atomics then fall on banks by lane
// and not by symbol, whatever the exponents: with 32 copies two lanes at most meet on
// a bank, and eight atomics of a wavefront take 35 cycles of the compute unit's LDS
// (8 copies side by side at an odd stride, where lanes with the same symbol wait for
// each other: 144; 32 of those: 55; 64 copies of this kind: 34).
#define NZ_HIST_COPIES_LOG2 5u
struct NzHist {
  uint32_t* mine;       // this lane's copy
  uint32_t copies_log2;

  static __device__ __forceinline__ void clear(uint32_t* all, uint32_t copies_log2) {
    for (uint32_t i = threadIdx.x; i < (64u << copies_log2); i += blockDim.x)
      reinterpret_cast<uint4*>(all)[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  __device__ __forceinline__ void count(uint32_t symbol) const { atomicAdd(&mine[symbol << copies_log2], 1u); }
  // a symbol's counters, 16 bytes at a time; neighbouring symbols begin at different ones (banks again)
  static __device__ __forceinline__ uint32_t sum(const uint32_t* all, uint32_t copies_log2, uint32_t symbol) {
    const uint4* at = reinterpret_cast<const uint4*>(all + (symbol << copies_log2));
    const uint32_t quads = 1u << (copies_log2 - 2);
    uint32_t c = 0;
    for (uint32_t k = 0; k < quads; ++k) {
      const uint4 v = at[(k + symbol) & (quads - 1)];
      c += v.x + v.y + v.z + v.w;
    }
    return c;
  }
};

// LDS of an encode workgroup (besides histogram and word staging).
struct NzEncLds {
  uint32_t red[32];
  uint32_t scan_s[4];
  uint64_t mw[4];
  uint32_t cf[256];
  uint4 tab[256];  // per symbol: nz_quot_entry
  uint32_t ser[NZ_TABLE_MAX_BYTES / 4];  // the serialized table
  uint32_t sbuf[NZ_MAX_SEGS_PER_CHUNK][NZ_STATE_MAX_BYTES / 4];
  uint32_t pad_sym, raw;
  // for records that go straight to their place: the chunk's record sizes, the
  // sum over the chunks before it, whether the wait for those was given up
  uint32_t seg_units[NZ_MAX_SEGS_PER_CHUNK];
  // what the wavefronts found for their segments (words, state bytes) and the table's length, for
  // the thread that sizes the records: the copies in scratch memory are for the kernels that follow
  uint32_t seg_w[NZ_MAX_SEGS_PER_CHUNK], seg_sb[NZ_MAX_SEGS_PER_CHUNK], tab_len;
  uint32_t chunk_total, gave_up;
  uint32_t redo;  // a wavefront ran out of staging room: the chunk is coded again, into the slots
  uint32_t lb[2];  // the two words of the scratch's announcement state, as thread 0 read them
  uint64_t red64[NZ_ENC_LONG_THREADS / 64];
};

// Split one element group: 8 bf16 values -> 8 exponent bytes (byte j of `e` =
// element j) and the S+1 packed bytes (`f`, little-endian).  Two elements at a
// time, both halves of a dword in parallel: the rounding add cannot carry
// from the low half into the high one (0x7FFF + 2^(6-S) < 2^16), so the closed
// form of nz_split_one holds for both halves at once.
template <int S>
__device__ __forceinline__ void nz_split_group(const uint4 v, uint64_t& e, uint64_t& f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t t[4], p[4];  // per dword: exponents in bytes 0 and 2 | the two (S+1)-bit fields, first element on top
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (S == 7) {
      t[k] = (w[k] >> 7) & 0x00FF00FFu;
      p[k] = ((w[k] >> 8) & 0x00800080u) | (w[k] & 0x007F007Fu);  // sign | mantissa in bytes 0 and 2
    } else {
      const uint32_t a = ((w[k] & 0x7FFF7FFFu) + (0x00010001u << (6 - S))) & 0x7FFF7FFFu;
      t[k] = (a >> 7) & 0x00FF00FFu;
      const uint32_t fld = ((w[k] >> (15 - S)) & (0x00010001u << S)) | ((a >> (7 - S)) & (0x00010001u * ((1u << S) - 1u)));
      p[k] = ((fld << (S + 1)) | (fld >> 16)) & ((1u << (2 * S + 2)) - 1u);
    }
  }
  // bytes 0 and 2 of two dwords -> four consecutive bytes
  const uint32_t e_lo = __builtin_amdgcn_perm(t[1], t[0], 0x06040200u), e_hi = __builtin_amdgcn_perm(t[3], t[2], 0x06040200u);
  e = ((uint64_t)e_hi << 32) | e_lo;
  if constexpr (S == 7) {
    const uint32_t f_lo = __builtin_amdgcn_perm(p[1], p[0], 0x06040200u), f_hi = __builtin_amdgcn_perm(p[3], p[2], 0x06040200u);
    f = ((uint64_t)f_hi << 32) | f_lo;
  } else if constexpr (S == 3) {
    f = p[0] | (p[1] << 8) | (p[2] << 16) | (p[3] << 24);  // one byte per pair of elements
  } else if constexpr (S == 1) {
    f = ((p[0] << 4) | p[1]) | (((p[2] << 4) | p[3]) << 8);  // one nibble per pair
  } else {
    f = (p[0] << 6) | (p[1] << 4) | (p[2] << 2) | p[3];      // two bits per pair, element 0 on top
  }
}

template <int S>
__device__ __forceinline__ void nz_store_packed(uint8_t* pp, uint64_t f) {
  if constexpr (S == 7) __builtin_nontemporal_store(f, reinterpret_cast<uint64_t*>(pp));
  else if constexpr (S == 3) __builtin_nontemporal_store((uint32_t)f, reinterpret_cast<uint32_t*>(pp));
  else if constexpr (S == 1) __builtin_nontemporal_store((uint16_t)f, reinterpret_cast<uint16_t*>(pp));
  else __builtin_nontemporal_store((uint8_t)f, pp);
}

// The last elements of the tensor (fewer than 8 in this lane's group): missing
// ones contribute zero bits (cuda/kernels.cuh:92), and only ceil(rem*(S+1)/8)
// packed bytes exist.  -> the exponent bytes, zero above `rem`.
template <int S>
__device__ __forceinline__ uint64_t nz_split_tail(const uint16_t* __restrict__ in, uint64_t gi, uint32_t rem,
                                                  uint8_t* pp, const NzNorm& nm) {
  uint64_t e = 0, f = 0;
  for (uint32_t j = 0; j < rem; ++j) {
    uint32_t h = in[gi + j], ex, rp;
    if (nm.bytes) h = nz_norm_div(h, nm.bytes[(gi + j) >> nm.log2n]);
    nz_split_one<S>(h, ex, rp);
    e |= (uint64_t)ex << (8 * j);
    const uint32_t bit = j * (S + 1);
    f |= (uint64_t)rp << (8u * (bit >> 3) + (7u - S - (bit & 7u)));
  }
  const uint32_t nb = (rem * (S + 1) + 7) / 8;
  for (uint32_t b = 0; b < nb; ++b) pp[b] = (uint8_t)(f >> (8 * b));
  return e;
}

// x / f in one instruction.  The 32 bits of x, taken as those of a double, are the
// subnormal x * 2^-1074; the table's multiplier is 2^1023 * r with r a little above
// 1 / f (nz_quot_entry), so the fused multiply-add forms x * r * 2^-51 + 2 - 2^-52 exactly
// and rounds once, to a multiple of 2^-51: the low word of the result is x * r - 1/2
// rounded to nearest, which is floor(x / f) for 16 <= x < f << 20 (x * r exceeds x / f by
// less than 2^-18, so it is never a whole number and never reaches the next one; pinned
// on the host for every f, tests/test_quotient_fma.py).  FP64 multiply-adds run at the rate
// of the 32-bit integer ones here, subnormals included.
__device__ __forceinline__ uint32_t nz_quot(uint32_t x, uint32_t r_lo, uint32_t r_hi) {
  const double xd = __builtin_bit_cast(double, (uint64_t)x);
  const double r = __builtin_bit_cast(double, ((uint64_t)r_hi << 32) | r_lo);
  return (uint32_t)__builtin_bit_cast(uint64_t, __builtin_fma(xd, r, 2.0 - 0x1p-52));
}

// The encoder's entry of a symbol: x = freq << 20 (renormalisation threshold), y = 4096 - freq,
// z and w = the multiplier of nz_quot, whose 12 lowest bits give way to cum: the multiplier
// is made 1 + 2^-39 times too large first, so that it stays above 1 / freq whatever they are.
__device__ __forceinline__ uint4 nz_quot_entry(uint32_t f, uint32_t cum) {
  const uint64_t r = f ? __builtin_bit_cast(uint64_t, (1.0 + 0x1p-39) / (double)f) + (1023ull << 52) : 0ull;
  return make_uint4(f << 20, NZ_M - f, ((uint32_t)r & ~(NZ_M - 1)) | cum, (uint32_t)(r >> 32));
}

// From the chunk's histogram (cn symbols): the 12-bit frequency table (sum
// exactly 4096), the encoder's per-symbol entries in LDS, the serialized table (in LDS, and in
// `out` for the kernels that follow) and the chunk record.  Run by the whole workgroup (at least 256 threads).
// -> an estimate of the chunk's coded length in bits (sum of count x -log2 of
// the quantised probability), the same in every thread.
__device__ __forceinline__ uint32_t nz_build_table(NzEncLds& L, const uint32_t* hist, const uint32_t copies_log2,
                                                   const uint32_t cn, uint8_t* __restrict__ out,
                                                   NzChunkInfo* __restrict__ info_c) {
  const uint32_t tid = threadIdx.x;
  // threads 0..255 own one symbol each; the others take part in the reductions
  // with neutral values
  const bool own = tid < 256;
  const uint32_t cnt = own ? NzHist::sum(hist, copies_log2, tid) : 0u;
  const uint32_t live = cnt > 0;
  // live symbols; most frequent symbol, lowest index on ties (cnt <= 2^24 fits above the index byte)
  uint32_t k = live, key = own ? ((cnt << 8) | (255u - tid)) : 0u;
  nz_block_sum_max(k, key, L.red);
  const uint32_t imax = 255u - (key & 0xFFu);
  // cnt * (4096 - k) fits 32 bits for chunks of up to 2^19 symbols (every geometry the library
  // chooses itself): a 32-bit division then, a fraction of the 64-bit one's instructions
  uint32_t f = 0;
  if (cn <= (1u << 19)) f = live ? 1u + (cnt * (NZ_M - k)) / cn : 0u;
  else f = live ? 1u + (uint32_t)(((uint64_t)cnt * (NZ_M - k)) / cn) : 0u;
  // (the estimate does without what the most frequent symbol is still given)
  uint32_t sum = f, est_bits = live ? (uint32_t)((float)cnt * (12.0f - __log2f((float)f))) + 1u : 0u;
  nz_block_sum2(sum, est_bits, L.red);
  if (tid == imax) f += NZ_M - sum;
  if (k == 1) f = (tid == imax) ? (NZ_M - 1) : ((tid == (imax ^ 1u)) ? 1u : 0u);

  // exclusive prefix sum over the 256 symbols
  uint32_t incl = f;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t t = __shfl_up(incl, o, 64);
    if ((tid & 63) >= (uint32_t)o) incl += t;
  }
  if (own && (tid & 63) == 63) L.scan_s[tid >> 6] = incl;
  __syncthreads();
  if (own) {
    uint32_t woff = 0;
    for (uint32_t w = 0; w < (tid >> 6); ++w) woff += L.scan_s[w];
    const uint32_t cum = woff + incl - f;
    L.tab[tid] = nz_quot_entry(f, cum);
  }

  // ---- serialise the table, in parallel ----
  // 256-bit live mask from the ballots of the four owning waves; the rank of a
  // live symbol is the number of live symbols below it.
  const uint64_t bal = __ballot(own && f != 0);
  if (own && (tid & 63) == 0) L.mw[tid >> 6] = bal;
  __syncthreads();
  const uint64_t m0 = L.mw[0], m1 = L.mw[1], m2 = L.mw[2], m3 = L.mw[3];
  const uint32_t kk = (uint32_t)(__popcll(m0) + __popcll(m1) + __popcll(m2) + __popcll(m3));
  if (own && f != 0) {
    const uint32_t w = tid >> 6;
    const uint32_t below = (w > 0 ? (uint32_t)__popcll(m0) : 0u) + (w > 1 ? (uint32_t)__popcll(m1) : 0u) +
                           (w > 2 ? (uint32_t)__popcll(m2) : 0u) +
                           (uint32_t)__popcll(bal & ((1ull << (tid & 63)) - 1ull));
    L.cf[below] = f;
  }
  // a run starts at a live symbol whose predecessor is not live
  const uint64_t s0 = m0 & ~(m0 << 1);
  const uint64_t s1 = m1 & ~((m1 << 1) | (m0 >> 63));
  const uint64_t s2 = m2 & ~((m2 << 1) | (m1 >> 63));
  const uint64_t s3 = m3 & ~((m3 << 1) | (m2 >> 63));
  const uint32_t runs = (uint32_t)(__popcll(s0) + __popcll(s1) + __popcll(s2) + __popcll(s3));
  const bool run_form = runs >= 1 && runs <= NZ_MAX_RUNS;
  const uint32_t head = run_form ? 1u + 2u * runs : 33u;
  __syncthreads();
  uint8_t* ser = reinterpret_cast<uint8_t*>(L.ser);
  // 12-bit fields, two per three bytes
  for (uint32_t pj = tid; 2 * pj < kk; pj += blockDim.x) {
    const uint32_t a = L.cf[2 * pj];
    const bool two = 2 * pj + 1 < kk;
    const uint32_t b = two ? L.cf[2 * pj + 1] : 0u;
    uint8_t* fp = ser + head + 3 * pj;
    fp[0] = (uint8_t)(a & 0xFF);
    fp[1] = (uint8_t)((a >> 8) | ((b & 0xF) << 4));
    if (two) fp[2] = (uint8_t)(b >> 4);
  }
  if (!run_form && tid < 32) {
    const uint64_t mq = tid < 8 ? m0 : (tid < 16 ? m1 : (tid < 24 ? m2 : m3));
    ser[1 + tid] = (uint8_t)(mq >> (8 * (tid & 7)));
  }
  if (tid == 0) {
    if (run_form) {
      ser[0] = (uint8_t)runs;
      const uint64_t mm[4] = {m0, m1, m2, m3};
      const uint64_t ss[4] = {s0, s1, s2, s3};
      uint32_t r = 0;
      for (int w = 0; w < 4; ++w) {
        uint64_t sm = ss[w];
        while (sm) {
          const uint32_t b = (uint32_t)__builtin_ctzll(sm);
          sm &= sm - 1;
          // first symbol at or after the start that is not live
          uint32_t end = 256;
          uint64_t dead = ~mm[w] & ~((b ? (1ull << b) : 1ull) - 1ull);
          if (b == 0) dead = ~mm[w];
          for (int v = w; v < 4; ++v) {
            if (v > w) dead = ~mm[v];
            if (dead) {
              end = 64u * v + (uint32_t)__builtin_ctzll(dead);
              break;
            }
          }
          ser[1 + 2 * r] = (uint8_t)(64u * w + b);
          ser[2 + 2 * r] = (uint8_t)(end - (64u * w + b) - 1u);
          ++r;
        }
      }
    } else {
      ser[0] = NZ_MODE_BITMAP;
    }
    const uint32_t bytes = head + (12 * kk + 7) / 8;
    const uint32_t padded = (bytes + 3) & ~3u;
    for (uint32_t b = bytes; b < padded; ++b) ser[b] = 0;
    NzChunkInfo ci;
    ci.tab_len = padded;
    ci.pad_sym = imax;
    ci.raw = 0;
    ci.reserved = 0;
    *info_c = ci;
    L.pad_sym = imax;
    L.tab_len = padded;
  }
  __syncthreads();
  for (uint32_t i = tid; i < L.tab_len / 4; i += blockDim.x) reinterpret_cast<uint32_t*>(out)[i] = L.ser[i];
  return est_bits;
}

// ----------------------------------------------------------------------------
// per chunk: coded or raw, and the record size of each of its segments (run by one
// wavefront of the encode kernel, a lane per segment, once all segments of the chunk
// are coded)
// ----------------------------------------------------------------------------
__device__ __forceinline__ bool nz_chunk_finalize(uint64_t c, uint64_t n, uint32_t chunk_syms,
                                                  uint32_t seg_syms, uint32_t spc, NzChunkInfo* info,
                                                  const uint32_t* lds_words, const uint32_t* lds_state_bytes,
                                                  uint32_t tab_len, uint32_t* seg_units, uint32_t* chunk_units,
                                                  uint32_t* lds_seg_units, uint32_t* lds_chunk_total) {
  const uint32_t k = nz_lane_id();
  const uint64_t base = c * chunk_syms;
  const uint32_t cn = (uint32_t)((n - base) < chunk_syms ? (n - base) : chunk_syms);
  const uint32_t nseg = (cn + seg_syms - 1) / seg_syms;
  uint32_t rans = 0, raws = 0;  // bytes; a record has at most ~2^23, a chunk eight records
  if (k < nseg) {
    const uint32_t sn = (cn - k * seg_syms) < seg_syms ? (cn - k * seg_syms) : seg_syms;
    rans = lds_state_bytes[k] + 2u * ((lds_words[k] + 1) & ~1u);
    raws = ((sn + 3) & ~3u) + (sn == nz_seg_nominal(chunk_syms, seg_syms, spc, k) ? NZ_CARRY_BYTES : 0u);
  }
  const uint32_t rans_total = tab_len + __builtin_amdgcn_readlane(nz_wave_scan(rans, k), 63);
  const uint32_t raw_total = 4u + __builtin_amdgcn_readlane(nz_wave_scan(raws, k), 63);
  const bool raw = rans_total >= raw_total;
  if (k < nseg) {
    const uint32_t units = (raw ? raws + (k == 0 ? 4u : 0u) : rans + (k == 0 ? tab_len : 0u)) / 4;
    seg_units[c * spc + k] = units;
    lds_seg_units[k] = units;
  }
  if (k == 0) {
    info[c].raw = raw ? 1u : 0u;
    chunk_units[c] = (raw ? raw_total : rans_total) / 4;
    *lds_chunk_total = (raw ? raw_total : rans_total) / 4;
  }
  return raw;
}

// ----------------------------------------------------------------------------
// rANS encode of one segment by one wavefront
// ----------------------------------------------------------------------------
//
// The 64 lanes run backwards over their symbols.  Per symbol: emit the low 16
// state bits when the state is at or above freq << 20 (ranked into the word
// slot back to front, so that the decoder reads front to back), then
// x = (x / f) << 12 | (x % f) + cum.  A segment's slot holds one word per
// symbol, the most any input can emit, so there is no overflow path; a chunk
// that codes to more than its raw size is stored raw (decided at the end of the
// kernel, once all segments of the chunk are coded).

// Table entries on their way to the encoder: four of them, those of the symbols that are coded
// next, entry of symbol j in v[j & 3].  They do not depend on the state, so each is read four
// steps before its use, across groups as well.
typedef uint32_t nz_u32x4 __attribute__((ext_vector_type(4)));
struct NzEncAhead {
  nz_u32x4 v[4];

  __device__ __forceinline__ void fetch(const uint4* __restrict__ tab, const uint64_t sy, const int j) {
    v[j & 3] = reinterpret_cast<const nz_u32x4*>(tab)[(uint32_t)(sy >> (8 * j)) & 0xFFu];
  }
  // the first four of a group
  __device__ __forceinline__ void start(const uint4* __restrict__ tab, const uint64_t sy) {
#pragma unroll
    for (int j = 7; j >= 4; --j) fetch(tab, sy, j);
  }
};

// The 8 symbols of one group (byte j of `sy` = symbol j), last symbol first; `sy_next`: those
// of the group that is coded after it.
// Words go downwards from `pos`, a byte offset into the segment's slot in scratch memory or,
// with LDS, an LDS byte address in the wavefront's staging area.  There every lane stores: a
// lane without a word writes one of the 64 places below the words of the step (each lane its
// own), which the words that follow overwrite.  That keeps the execution mask out of the step's
// chain; the caller leaves 64 words of room below.
template <bool LDS>
__device__ __forceinline__ void nz_enc_group(uint32_t& x, uint32_t& pos, const uint64_t sy, const uint64_t sy_next,
                                             NzEncAhead& ahead, const uint4* __restrict__ tab,
                                             uint16_t* __restrict__ slot, const uint32_t below) {
  typedef __attribute__((address_space(3))) uint16_t lds_u16;
#pragma unroll
  for (int j = 7; j >= 0; --j) {
    nz_u32x4 e = ahead.v[j & 3];
    asm("" : "+v"(e));  // one 16-byte read, not two of 8
    const bool need = x >= e.x;
    const uint64_t m = __ballot(need);
    const uint32_t word = x;
    x = need ? (x >> 16) : x;
    // x < f << 20 here; with q = x / f the new state is (q << 12) + (x - q f) + cum
    const uint32_t q = nz_quot(x, e.z, e.w);
    uint32_t t = x + (e.z & (NZ_M - 1));
    asm("" : "+v"(t));  // then one multiply-add
    x = __umul24(q, e.y) + t;
    ahead.fetch(tab, j >= 4 ? sy : sy_next, j ^ 4);
    pos -= 2u * (uint32_t)__popcll(m);
    if constexpr (LDS) {
      uint32_t zero = 0;
      asm("" : "+v"(zero));  // a vector register: the short form of the select
      const uint32_t at = __builtin_amdgcn_mbcnt_hi(
          (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, need ? zero : below));
      *(lds_u16*)(uintptr_t)((at << 1) + pos) = (uint16_t)word;
    } else if (need) {
      *reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(slot) + ((nz_rank_below(m) << 1) + pos)) = (uint16_t)word;
    }
  }
}

// Final states, variable length: 64 two-bit codes (code c = 5 + c nibbles),
// then the states as a little-endian nibble stream in lane order.  A state
// is >= 2^16, so it takes 20..32 bits; a flat 32 would waste ~4 more per lane.
__device__ __forceinline__ void nz_enc_finish(const uint32_t x, const uint32_t words, const uint64_t seg,
                                              uint32_t* __restrict__ sb, const uint32_t lane,
                                              uint32_t* __restrict__ states, uint32_t* __restrict__ seg_words,
                                              uint32_t* __restrict__ seg_state_bytes, uint32_t* lds_words,
                                              uint32_t* lds_state_bytes) {
  const uint32_t code = (x >> 20 ? 1u : 0u) + (x >> 24 ? 1u : 0u) + (x >> 28 ? 1u : 0u);
  const uint32_t nn = 5u + code;
  const uint32_t incl = nz_wave_scan(nn, lane);
  const uint32_t at = incl - nn;  // nibble offset of this lane's field
  const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
  const uint32_t sbytes = 16u + ((((total + 1u) >> 1) + 3u) & ~3u);
  for (uint32_t i = lane; i < NZ_STATE_MAX_BYTES / 4; i += 64) sb[i] = 0;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  atomicOr(&sb[lane >> 4], code << (2 * (lane & 15)));
  const uint64_t field = (uint64_t)x << (4 * (at & 7));
  atomicOr(&sb[4 + (at >> 3)], (uint32_t)field);
  if (field >> 32) atomicOr(&sb[5 + (at >> 3)], (uint32_t)(field >> 32));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  uint32_t* sdst = states + seg * (NZ_STATE_MAX_BYTES / 4);
  for (uint32_t i = lane; i < sbytes / 4; i += 64) sdst[i] = sb[i];
  if (lane == 0) {
    seg_words[seg] = words;
    seg_state_bytes[seg] = sbytes;
    *lds_words = words;
    *lds_state_bytes = sbytes;
  }
}

// The tensors of one encode call ride in the kernel argument block (as the
// items of a decode batch do): the grid of an encode kernel is the
// concatenation of their chunks, that of the scan kernel one workgroup per
// tensor, that of the compaction the concatenation of their segments.
#define NZ_ENC_BATCH_MAX 16
struct NzEncItem {
  const uint16_t* in;   // dense input
  uint8_t* packed;      // stored sign|mantissa stream
  uint8_t* ws;          // this tensor's slice of the scratch; the offsets below are into it
  uint8_t* comp;        // the container: header, directory, records
  uint64_t comp_cap;    // capacity the container size is checked against
  uint64_t* d_total;    // container size
  uint32_t* d_status;   // bit 0: the container does not fit
  NzNorm nm;            // normalizer bytes (nullptr: none)
  NzGeom g;
  uint64_t exps, tab_ser, info, carry, slots, states, seg_words, seg_sbytes, seg_units, chunk_units;
  uint32_t chunk_end, seg_end;  // running totals over the batch
  // records straight to their place (nz_encode_kernel, `direct` != 0): where the
  // chunks announce their sizes (two words per chunk, offset into ws), the
  // number that marks this call's announcements, how often a chunk looks for
  // an announcement before it gives up, and where it says so (may be null)
  uint64_t pub, nonce;
  uint64_t* d_gave_up;
  uint32_t direct, spin_limit;
  uint64_t lb_state;  // NzLbWords (offset into ws)
  // `placed`: one byte per segment (offset into ws), left by a direct encode: 1 =
  // the record is in the container and not in the scratch (its words went there
  // from LDS).  nz_compact_kernel with `use_placed` takes such records from
  // `old_comp`, where they lie at the offsets they keep.
  uint64_t placed;
  const uint8_t* old_comp;
  uint32_t use_placed, reserved;
};
struct NzEncBatch {
  uint32_t count;
  uint32_t stage_words;  // nz_encode_kernel: 16-bit words of LDS staging per wavefront (dynamic LDS), 0 = none
  uint32_t copies_log2;  // histogram copies (NzHist; dynamic LDS as well, used before the staging)
  uint32_t reserved;
  NzEncItem item[NZ_ENC_BATCH_MAX];
};

__device__ __forceinline__ void nz_write_header(uint8_t* comp, const NzGeom& g, uint64_t total) {
  uint32_t* h = reinterpret_cast<uint32_t*>(comp);
  h[0] = NZ_MAGIC;
  h[1] = NZ_FORMAT_VERSION;
  h[2] = (uint32_t)(g.n & 0xFFFFFFFFu);
  h[3] = (uint32_t)(g.n >> 32);
  h[4] = g.chunk_syms;
  h[5] = g.lane_syms;
  h[6] = (uint32_t)g.n_chunks;
  h[7] = (uint32_t)g.n_segs;
  h[8] = (uint32_t)g.dir_off;
  h[9] = (uint32_t)g.rec_off;
  h[10] = (uint32_t)(total & 0xFFFFFFFFu);
  h[11] = (uint32_t)(total >> 32);
  h[12] = h[13] = h[14] = h[15] = 0;
  // the alignment gap between directory and records
  for (uint64_t b = g.dir_off + 4 * (g.n_segs + 1); b < g.rec_off; ++b) comp[b] = 0;
}


// ----------------------------------------------------------------------------
// move a segment record to its final place
// ----------------------------------------------------------------------------
// NT threads (t = 0 .. NT-1) move the record of segment `seg` = segment k of
// chunk c to o0, counted in 4-byte units from the start of the record area
// (`mine` = its size in the same units; ci, sbytes, w: the chunk's info, the
// size of the coder states, the number of words; `table`, `states`, `words`: where the
// record's parts are, in scratch memory or in LDS; the words at the end of the segment's
// slot or in a staging area).  With `whole` the
// record is not assembled from its parts but copied from there (the same record
// in another container).  They write the segment's directory entry; those of
// the last segment add the closing entry, the header, the container size and
// the overflow flag.  -> whether the record fits the container (if not, nothing
// of it is written).
template <uint32_t NT>
__device__ __forceinline__ bool nz_move_record(const NzEncItem& it, const uint64_t seg, const uint64_t c,
                                               const uint32_t k, const uint64_t o0, const uint32_t mine,
                                               const NzChunkInfo ci, const uint32_t sbytes, const uint32_t w,
                                               const uint32_t* table, const uint32_t* states, const uint16_t* words,
                                               const uint8_t* whole, const uint32_t t) {
  static_assert(NT >= NZ_TAIL_PAD, "too few threads for the closing zeros");
  const NzGeom& g = it.g;
  const uint8_t* __restrict__ carry = it.ws + it.carry;
  const uint16_t* __restrict__ slots = reinterpret_cast<const uint16_t*>(it.ws + it.slots);
  uint8_t* __restrict__ comp = it.comp;
  const uint64_t o1 = o0 + mine;
  const bool fits = o1 <= 0xFFFFFFFFull && g.rec_off + 4 * o1 + NZ_TAIL_PAD <= it.comp_cap;
  if (seg + 1 == g.n_segs && t == 0) {
    const uint64_t total = g.rec_off + 4 * o1 + NZ_TAIL_PAD;
    *it.d_total = total;
    if (!fits) atomicOr(it.d_status, 1u);
  }
  if (!fits) return false;  // (a record before this one may still fit and be written: harmless)
  uint32_t* dir = reinterpret_cast<uint32_t*>(comp + g.dir_off);
  if (t == 0) dir[seg] = (uint32_t)o0;
  uint8_t* dst = comp + g.rec_off + 4 * o0;
  if (seg + 1 == g.n_segs) {
    if (t == 0) {
      dir[g.n_segs] = (uint32_t)o1;
      nz_write_header(comp, g, g.rec_off + 4 * o1 + NZ_TAIL_PAD);
    }
    if (t < NZ_TAIL_PAD) comp[g.rec_off + 4 * o1 + t] = 0;  // closing zeros
  }
  if (whole) {
    if (whole != dst)
      for (uint32_t i = t; i < mine; i += NT)
        reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(whole)[i];
    return true;
  }
  const uint64_t seg_base = c * g.chunk_syms + (uint64_t)k * g.seg_syms;
  const uint32_t nom = nz_seg_nominal(g.chunk_syms, g.seg_syms, g.spc, k);
  const uint32_t sn = (uint32_t)((g.n - seg_base) < nom ? (g.n - seg_base) : nom);
  if (ci.raw) {
    uint32_t off = 0;
    if (k == 0) {
      if (t < 4) dst[t] = t == 0 ? NZ_MODE_RAW : 0;
      off = 4;
    }
    const uint32_t padded = (sn + 3) & ~3u;
    const uint8_t* rawp = reinterpret_cast<const uint8_t*>(slots + seg * g.seg_syms);  // left there by the encode kernel
    for (uint32_t i = t; i < padded; i += NT) dst[off + i] = i < sn ? rawp[i] : 0;
    if (sn == nom)
      for (uint32_t i = t; i < NZ_CARRY_BYTES; i += NT) dst[off + padded + i] = carry[seg * NZ_CARRY_BYTES + i];
    return true;
  }
  uint32_t off = 0;
  if (k == 0) {
    for (uint32_t i = t; i < ci.tab_len / 4; i += NT) reinterpret_cast<uint32_t*>(dst)[i] = table[i];
    off = ci.tab_len;
  }
  uint32_t* sdst = reinterpret_cast<uint32_t*>(dst + off);
  for (uint32_t i = t; i < sbytes / 4; i += NT) sdst[i] = states[i];
  // the words are 2-byte aligned; they are moved as dwords (two aligned loads and a
  // funnel shift when the source is off by one word; the load past the last word
  // stays inside the scratch buffer or the staging area)
  const uint16_t* src = words;
  const uint32_t mis = (uint32_t)((reinterpret_cast<uintptr_t>(src) >> 1) & 1u);
  const uint32_t* s32 = reinterpret_cast<const uint32_t*>(src - mis);
  uint32_t* wdst = reinterpret_cast<uint32_t*>(dst + off + sbytes);
  const uint32_t nd = (w + 1) / 2;
  const uint32_t nd4 = nd & ~3u;  // four dwords per thread and turn, then the last one to three singly
  for (uint32_t i = 4 * t; i < nd4; i += 4 * NT) {
    const uint32_t a0 = s32[i], a1 = s32[i + 1], a2 = s32[i + 2], a3 = s32[i + 3];
    uint4 v = make_uint4(a0, a1, a2, a3);
    if (mis) {
      const uint32_t a4 = s32[i + 4];
      v = make_uint4(__builtin_amdgcn_alignbit(a1, a0, 16), __builtin_amdgcn_alignbit(a2, a1, 16),
                     __builtin_amdgcn_alignbit(a3, a2, 16), __builtin_amdgcn_alignbit(a4, a3, 16));
    }
    if ((w & 1) && i + 4 == nd) v.w &= 0xFFFFu;  // the padding word of an odd count is zero
    wdst[i] = v.x;
    wdst[i + 1] = v.y;
    wdst[i + 2] = v.z;
    wdst[i + 3] = v.w;
  }
  for (uint32_t i = nd4 + t; i < nd; i += NT) {
    uint32_t v = mis ? __builtin_amdgcn_alignbit(s32[i + 1], s32[i], 16) : s32[i];
    if ((w & 1) && i == nd - 1) v &= 0xFFFFu;
    wdst[i] = v;
  }
  return true;
}

// Wavefronts per SIMD unit that the kernel for NG groups is compiled for: what its registers (72, 96,
// 128 and 128 for the four NG) allow without spilling.  The host sizes the dynamic LDS by the same number.
// (64 Mi elements in chunks of 16384 with 64 symbols per lane and of 65536 with 128: 100.8 and 77.5 us;
// with LDS cut for 8 and 6 wavefronts and two registers spilled 104.9 and 79.0.)
static constexpr int NZ_ENC_GROUPS[4] = {8, 16, 32, NZ_ENC_MAX_LANE_SYMS / NZ_GROUP};  // NG of the classes
__host__ __device__ constexpr uint32_t nz_enc_waves(int ng) { return ng <= 8 ? 7u : ng <= 16 ? 5u : 4u; }
// four wavefronts of the largest classes: four workgroups to a compute unit, each with 32 histogram copies
static_assert(sizeof(NzEncLds) + (1024u << NZ_HIST_COPIES_LOG2) <= 160u * 1024u / nz_enc_waves(32), "");

// Segments of up to 8 * NG symbols per lane: the exponents stay in registers.
// Workgroup = max(4, segments per chunk) wavefronts; wavefront k owns segment k.
// dynamic LDS of the encode kernels: the histogram (NzHist), then the word staging of
// nz_encode_kernel (stage_words / 2 dwords per wavefront + 4)
extern __shared__ __attribute__((aligned(16))) uint32_t nz_enc_stage[];
#ifdef NZ_PROBE_PHASES
__device__ unsigned long long nz_probe_acc[8];
#define NZ_PROBE_MARK(k)                                        \
  do {                                                          \
    if (threadIdx.x == 0) {                                     \
      const unsigned long long now = __builtin_readcyclecounter(); \
      atomicAdd(&nz_probe_acc[k], now - probe_t);               \
      probe_t = now;                                            \
    }                                                           \
  } while (0)
#else
#define NZ_PROBE_MARK(k)
#endif

template <int S, int NG>
__global__ __launch_bounds__(64 * NZ_MAX_SEGS_PER_CHUNK, nz_enc_waves(NG)) void nz_encode_kernel(const NzEncBatch b) {
  __shared__ NzEncLds L;
#ifdef NZ_PROBE_PHASES
  unsigned long long probe_t = __builtin_readcyclecounter();
#endif
  uint32_t t = 0, first = 0;
  while (t + 1 < b.count && blockIdx.x >= b.item[t].chunk_end) {
    first = b.item[t].chunk_end;
    ++t;
  }
  const NzEncItem& it = b.item[t];
  const NzGeom& g = it.g;
  const uint64_t c = blockIdx.x - first;
  const uint64_t n = g.n;
  const uint32_t chunk_syms = g.chunk_syms, seg_syms = g.seg_syms, spc = g.spc;
  const uint16_t* __restrict__ in = it.in;
  const NzNorm nm = it.nm;
  NzChunkInfo* info = reinterpret_cast<NzChunkInfo*>(it.ws + it.info);
  uint32_t* seg_words = reinterpret_cast<uint32_t*>(it.ws + it.seg_words);
  uint32_t* seg_state_bytes = reinterpret_cast<uint32_t*>(it.ws + it.seg_sbytes);
  uint32_t* seg_units = reinterpret_cast<uint32_t*>(it.ws + it.seg_units);

  const uint32_t tid = threadIdx.x;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lane = tid & 63;
  const uint64_t base = c * chunk_syms;
  const uint32_t cn = (uint32_t)((n - base) < chunk_syms ? (n - base) : chunk_syms);
  const uint64_t seg = c * spc + wave;
  const uint64_t seg_base = base + (uint64_t)wave * seg_syms;
  const bool has_seg = wave < spc && seg_base < n;
  const uint32_t nom = nz_seg_nominal(chunk_syms, seg_syms, spc, wave < spc ? wave : 0u);
  const uint32_t seg_n = has_seg ? (uint32_t)((n - seg_base) < nom ? (n - seg_base) : nom) : 0u;
  const uint32_t ngroups = (seg_n + NZ_GROUP_SYMS - 1) / NZ_GROUP_SYMS;  // at most NG
  const bool seg_full = has_seg && seg_n == nom;

  // State of the scratch's size announcements (see NzEncItem::lb_state): read
  // once, by one thread, long before it is needed, and handed to the others
  // through LDS, so that every thread of the workgroup acts on the same values
  // (another workgroup may change the words while this one starts).
  NzLbWords* lb_state = reinterpret_cast<NzLbWords*>(it.ws + it.lb_state);
  if (tid == 0) {
    L.lb[0] = it.direct ? __hip_atomic_load(&lb_state->runs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    L.lb[1] = it.direct ? __hip_atomic_load(&lb_state->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    L.redo = 0;
  }
  NzHist::clear(nz_enc_stage, b.copies_log2);
  __syncthreads();
  // this run places its records itself (read again where it is asked: kept, it takes registers of the coding phase)
  const auto places = [&] { return it.direct && L.lb[1] != NZ_LOOKBACK_ABORT; };
  const NzHist hist{nz_enc_stage + (lane & ((1u << b.copies_log2) - 1u)), b.copies_log2};

  // ---- phase 1: split.  Packed bytes go to the stored layout: segment k of a
  // chunk starts at k * seg_keep, and the last NZ_CARRY_BYTES of a full segment
  // go to carry[seg] instead (they ride in the rANS start states).
  const uint32_t seg_keep = seg_syms / 8 * (S + 1) - NZ_CARRY_BYTES;  // of a segment of nominal length
  const uint64_t chunk_keep = (uint64_t)chunk_syms / 8 * (S + 1) - (uint64_t)NZ_CARRY_BYTES * spc;
  const uint32_t keep = nom / 8 * (S + 1) - NZ_CARRY_BYTES;
  uint8_t* pk = it.packed + c * chunk_keep + (uint64_t)wave * seg_keep;
  uint8_t* carry_seg = it.ws + it.carry + seg * NZ_CARRY_BYTES;
  const uint32_t whole = seg_n / NZ_GROUP_SYMS;  // groups in which every lane has 8 elements
  uint64_t ex[NG];
  const auto dest = [&](uint32_t g8) {  // where the packed bytes of this lane's group g8 go
    const uint32_t sb = (g8 * NZ_LANES + lane) * (S + 1);
    return (seg_full && sb >= keep) ? carry_seg + (sb - keep) : pk + sb;
  };
  const auto count8 = [&](uint64_t e) {
#ifndef NZ_PROBE_NO_HIST
#pragma unroll
    for (int j = 0; j < 8; ++j) hist.count((uint32_t)(e >> (8 * j)) & 0xFFu);
#else  // measurement build: the split phase without its histogram (the kernel ends after the phase)
    asm volatile("" ::"v"((uint32_t)e), "v"((uint32_t)(e >> 32)));
#endif
  };
  // Four groups at a time, and the loads of the next eight (short segments: four) are
  // issued before the current four are split: twelve 16-byte loads per lane in flight.
  // (The registers are there: the exponents of the groups in flight do not exist yet.)
  constexpr int AHEAD = NG >= 32 ? 2 : 1;
  uint4 vn[AHEAD][4];  // block b of four groups in vn[b % AHEAD]
  const auto load4 = [&](uint4 (&v)[4], uint32_t gv) {
    const uint16_t* src = in + seg_base + (gv * NZ_LANES + lane) * NZ_GROUP;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const nz_u32x4 r = __builtin_nontemporal_load(reinterpret_cast<const nz_u32x4*>(src + q * NZ_GROUP_SYMS));
      v[q] = make_uint4(r.x, r.y, r.z, r.w);
    }
  };
  if (4 <= whole) load4(vn[0], 0);
  if (AHEAD > 1 && 8 <= whole) load4(vn[AHEAD - 1], 4);
  nz_static_for<0, NG, 4>([&](auto g4c) {
    constexpr int g4 = decltype(g4c)::value;
    // the group number as a run-time value for all address arithmetic: with
    // constants the compiler precomputes the addresses of all groups up front
    // and runs out of registers; ex[] keeps its compile-time index
    uint32_t gv = (uint32_t)g4;
    asm volatile("" : "+s"(gv));
    if (gv + 4 <= whole) {
      uint4 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = vn[g4 / 4 % AHEAD][q];
      if (gv + 4 * AHEAD + 4 <= whole) load4(vn[g4 / 4 % AHEAD], gv + 4 * AHEAD);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (nm.bytes)
          v[q] = nz_scale8<false>(v[q], nz_norm_load8(nm, seg_base + ((gv + q) * NZ_LANES + lane) * NZ_GROUP),
                                  nm.log2n >= 3);
        uint64_t f;
        nz_split_group<S>(v[q], ex[g4 + q], f);
        nz_store_packed<S>(dest(gv + q), f);
        count8(ex[g4 + q]);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t g8 = gv + q;
        ex[g4 + q] = 0;
        if (g8 < ngroups) {
          const uint32_t idx0 = (g8 * NZ_LANES + lane) * NZ_GROUP;
          const uint64_t gi = seg_base + idx0;
          if (idx0 + 8 <= seg_n) {
            uint4 v = *reinterpret_cast<const uint4*>(in + gi);
            if (nm.bytes) v = nz_scale8<false>(v, nz_norm_load8(nm, gi), nm.log2n >= 3);
            uint64_t f;
            nz_split_group<S>(v, ex[g4 + q], f);
            nz_store_packed<S>(dest(g8), f);
            count8(ex[g4 + q]);
          } else if (idx0 < seg_n) {
            const uint32_t rem = seg_n - idx0;
            ex[g4 + q] = nz_split_tail<S>(in, gi, rem, dest(g8), nm);
            for (uint32_t j = 0; j < rem; ++j) hist.count((uint32_t)(ex[g4 + q] >> (8 * j)) & 0xFFu);
          }
        }
      }
    }
  });
  __threadfence_block();  // the carried bytes are read back below
  __syncthreads();
  NZ_PROBE_MARK(0);
#ifdef NZ_PROBE_NO_HIST
  return;
#endif

  // ---- the chunk's table ----
  const uint32_t est_bits = nz_build_table(L, nz_enc_stage, b.copies_log2, cn, it.ws + it.tab_ser + c * NZ_TABLE_MAX_BYTES, info + c);
  NZ_PROBE_MARK(1);

  // ---- phase 2: code the segment from the registers, last group first ----
  // The words go to the segment's slot in scratch memory, or, when the records
  // are placed by this kernel and the estimate says they fit, to the wavefront's
  // staging area in LDS (the last `stage_w` words of the slot), from where they
  // are written once, to their final place.  A wavefront that would run out of
  // staging stops; the chunk is then coded again into the slots (the exponents
  // are still in registers).
  const uint32_t cap_words = seg_syms;
  uint16_t* slot = reinterpret_cast<uint16_t*>(it.ws + it.slots) + seg * cap_words;
  const uint32_t stage_w = b.stage_words < cap_words ? b.stage_words : cap_words;
  const uint32_t stage_lo = cap_words - stage_w;  // first word of the slot that has a place in the staging area
  const uint32_t est_seg_words = (uint32_t)(((uint64_t)est_bits * seg_syms / cn) >> 4);
  bool staged = places() && stage_w >= 1024 && est_seg_words + (est_seg_words >> 4) + 64 <= stage_w;
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  uint32_t* stage = nz_enc_stage + wave * (b.stage_words / 2);
  const uint32_t stage_lds = (uint32_t)(uintptr_t)((lds_u32*)stage);
  uint32_t pos_end = cap_words;  // where the segment's words begin in its slot
  const auto code_segment = [&](auto lds_tag) -> bool {
    constexpr bool LDS = decltype(lds_tag)::value != 0;
    const uint32_t pad = L.pad_sym;
    // a full segment starts from 2^16 | 16 carried bits of the packed stream
    uint32_t x = NZ_L | (seg_full ? (uint32_t)reinterpret_cast<const uint16_t*>(carry_seg)[lane] : 0u);
    // byte position of the words: the staging area stands for the last stage_w words of the slot
    const uint32_t pos_lo = LDS ? stage_lds : 0u, pos_hi = pos_lo + 2u * (LDS ? stage_w : cap_words);
    uint32_t pos = pos_hi;
    bool out_of_room = false;
    NzEncAhead ahead;
    nz_static_for<NG - 1, 0, -1>([&](auto g8c) {
      constexpr int g8 = decltype(g8c)::value;
      uint32_t gv = (uint32_t)g8;
      asm volatile("" : "+s"(gv));
      if (gv < ngroups && !out_of_room) {
        // a group emits at most 512 words and writes over the 64 places below them
        if (LDS && pos - pos_lo < 2 * (NZ_GROUP * NZ_LANES + NZ_LANES)) {
          out_of_room = true;
        } else {
          uint64_t sy = ex[g8];
          if (gv >= whole) {  // the tensor ends inside this group: the most frequent symbol stands in
            const uint32_t idx0 = (gv * NZ_LANES + lane) * NZ_GROUP;
            const uint32_t have = idx0 < seg_n ? seg_n - idx0 : 0u;  // < 8 in some lane
            if (have < 8) {
              const uint64_t keepm = have ? (~0ull >> (64 - 8 * have)) : 0ull;
              sy = (sy & keepm) | ((0x0101010101010101ull * pad) & ~keepm);
            }
          }
          if (!LDS || gv + 1 == ngroups) ahead.start(L.tab, sy);  // (across groups it would cost the slot form registers)
          nz_enc_group<LDS>(x, pos, sy, ex[g8 ? g8 - 1 : 0], ahead, L.tab, slot, ~lane);
        }
      }
    });
    if (out_of_room) return true;
    nz_enc_finish(x, (pos_hi - pos) / 2, seg, L.sbuf[wave], lane, reinterpret_cast<uint32_t*>(it.ws + it.states),
                  seg_words, seg_state_bytes, &L.seg_w[wave], &L.seg_sb[wave]);
    pos_end = cap_words - (pos_hi - pos) / 2;
    return false;
  };
#pragma nounroll
  for (int pass = 0; pass < 2; ++pass) {
    if (has_seg) {
      if (staged) {
        if (code_segment(NzConst<1>{})) L.redo = 1;
      } else {
        code_segment(NzConst<0>{});
      }
    }
    // every segment of the chunk is coded (or one has run out of staging)
    __threadfence_block();
    __syncthreads();
    if (!(staged && L.redo)) break;
    staged = false;
  }
  NZ_PROBE_MARK(2);
  // decide coded-or-raw and size the records
  if (wave == 0) {
    const bool raw = nz_chunk_finalize(c, n, chunk_syms, seg_syms, spc, info, L.seg_w, L.seg_sb, L.tab_len, seg_units,
                                       reinterpret_cast<uint32_t*>(it.ws + it.chunk_units), L.seg_units,
                                       &L.chunk_total);
    if (lane == 0) {
      L.raw = raw;
      L.gave_up = 0;
    }
  }
  __syncthreads();
  if (L.raw && has_seg) {
    // a chunk that does not compress: its exponent bytes take the place of the words
    uint8_t* rawp = reinterpret_cast<uint8_t*>(slot);
    nz_static_for<0, NG, 1>([&](auto g8c) {
      constexpr int g8 = decltype(g8c)::value;
      uint32_t gv = (uint32_t)g8;
      asm volatile("" : "+s"(gv));
      const uint32_t idx0 = (gv * NZ_LANES + lane) * NZ_GROUP;
      if (idx0 < seg_n) *reinterpret_cast<uint64_t*>(rawp + idx0) = ex[g8];
    });
  }
  if (!it.direct) return;  // the records are placed by nz_compact_kernel
  const uint32_t lb_gen = L.lb[0];  // (only now: kept since the beginning, it was spilled for the coding phase)
  uint8_t* placed = it.ws + it.placed;  // per segment: its record is in the container and nowhere else
  const bool last_chunk = c + 1 == g.n_chunks;
  if (!places()) {
    // the run before this one ended with a workgroup giving up: nothing is
    // placed, the caller is told, and the mark is taken away for the next run
    if (tid == 0) {
      atomicOr(it.d_status, 4u);
      if (it.d_gave_up) *it.d_gave_up = it.nonce;
      nz_lb_unplaced(lb_state, it.nonce, lb_gen, last_chunk);
    }
    if (has_seg && lane == 0) placed[seg] = 0;
    return;
  }

  // ---- the records go straight to their place ----
  // The chunk announces the size of its records: two words, each with half of
  // the run's 64-bit mark on top and the size (or its complement) below, so
  // that whatever the scratch memory held before cannot pass for an
  // announcement.  Then it adds up the announcements of the chunks before it,
  // waiting for those that are not there yet.  Workgroups of one launch are
  // observed to start in the order of their numbers, so a chunk waited for is
  // normally running or done, and none of them waits before it has announced;
  // nothing guarantees that order across the dies of the device or next to
  // another kernel that fills the compute units, so the wait is bounded
  // (`spin_limit` looks per announcement): a chunk that gives up says so and
  // leaves its records where they are, for nz_compact_kernel.  Nothing but
  // the announcements passes between workgroups: relaxed device-scope
  // accesses, no fences.
  typedef unsigned long long nz_u64;
  nz_u64* pub = reinterpret_cast<nz_u64*>(it.ws + it.pub);  // four words per chunk: size pair, running-total pair
  const uint32_t mark_a = (uint32_t)(it.nonce >> 32) ^ lb_gen, mark_b = (uint32_t)it.nonce ^ (lb_gen * 0x9E3779B1u);
  const uint32_t mark_pa = mark_a ^ 0xA5A5A5A5u, mark_pb = mark_b ^ 0x3C3C3C3Cu;  // a size can never pass for a total
  if (tid == 0) {
    const uint32_t u = L.chunk_total;
    __hip_atomic_store(pub + 4 * c, ((nz_u64)mark_a << 32) | u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(pub + 4 * c + 1, ((nz_u64)mark_b << 32) | (uint32_t)~u, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  NZ_PROBE_MARK(3);
  // The chunks before this one, a window of one per thread at a time, nearest first.  A chunk
  // that has already placed its records has also announced the running total up to and
  // including itself (below); the nearest such chunk ends the walk, so a workgroup reads the
  // announcements of the chunks that ran beside it and one total, not those of every chunk
  // of the tensor.
  uint64_t part = 0;
  bool lost = false;
  if (c <= blockDim.x) {
    // every chunk before this one has a thread of its own: their sizes, nothing else
    if (tid < c) {
      for (uint32_t tries = 0;; ++tries) {
        const nz_u64 a = __hip_atomic_load(pub + 4 * tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const nz_u64 q = __hip_atomic_load(pub + 4 * tid + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)(a >> 32) == mark_a && (uint32_t)(q >> 32) == mark_b && (uint32_t)a == (uint32_t)~(uint32_t)q) {
          part = (uint32_t)a;
          break;
        }
        if (tries >= it.spin_limit) {
          lost = true;
          break;
        }
        __builtin_amdgcn_s_sleep(8);
      }
    }
  } else
  for (uint64_t hi = c; hi > 0;) {
    const uint64_t lo = hi > blockDim.x ? hi - blockDim.x : 0;
    const uint64_t i = lo + tid;
    uint32_t val = 0, key = 0;  // key: position in the window + 1 of an entry that carries a running total
    if (i < hi) {
      for (uint32_t tries = 0;; ++tries) {
        // all four words in flight at once: one round trip per look
        const nz_u64 a = __hip_atomic_load(pub + 4 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const nz_u64 q = __hip_atomic_load(pub + 4 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const nz_u64 pa = __hip_atomic_load(pub + 4 * i + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const nz_u64 pq = __hip_atomic_load(pub + 4 * i + 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)(pa >> 32) == mark_pa && (uint32_t)(pq >> 32) == mark_pb &&
            (uint32_t)pa == (uint32_t)~(uint32_t)pq) {
          val = (uint32_t)pa;
          key = (uint32_t)(i - lo) + 1u;
          break;
        }
        if ((uint32_t)(a >> 32) == mark_a && (uint32_t)(q >> 32) == mark_b && (uint32_t)a == (uint32_t)~(uint32_t)q) {
          val = (uint32_t)a;
          break;
        }
        if (tries >= it.spin_limit) {
          lost = true;
          break;
        }
        __builtin_amdgcn_s_sleep(8);
      }
    }
    // the same verdict for every thread: did anybody give up, and where is the nearest total
    const uint32_t verdict = nz_block_max(lost ? 0x80000000u : key, L.red);
    if (verdict & 0x80000000u) {
      lost = true;
      break;
    }
    const uint32_t at = (uint32_t)(i - lo) + 1u;  // sizes of the entries after the total, and the total itself
    if (i < hi && (key ? key == verdict : at > verdict)) part += val;
    if (verdict) break;
    hi = lo;
  }
  if (lost) L.gave_up = 1;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor((nz_u64)part, o, 64);
  if (lane == 0) L.red64[wave] = part;
  __threadfence_block();  // also: the raw bytes above are read back by the move
  __syncthreads();
  NZ_PROBE_MARK(4);
  // staged words of this wavefront to their slot, for the kernel that places records afterwards
  const auto unstage = [&]() {
    const uint16_t* sw = reinterpret_cast<const uint16_t*>(stage);
    for (uint32_t p = pos_end + lane; p < cap_words; p += NZ_LANES) slot[p] = sw[p - stage_lo];
  };
  if (L.gave_up) {
    if (tid == 0) {
      atomicOr(it.d_status, 4u);
      if (it.d_gave_up) *it.d_gave_up = it.nonce;
      nz_lb_gave_up(lb_state, it.nonce, lb_gen, last_chunk);
    }
    if (has_seg) {
      if (staged && !L.raw) unstage();
      if (lane == 0) placed[seg] = 0;
    }
    return;
  }
  if (tid == 0) {
    nz_lb_placed(lb_state, lb_gen, last_chunk);
    // the running total up to and including this chunk, for the chunks that come later (32 bits
    // of 4-byte units: a container beyond 16 GiB announces none, and its chunks walk on)
    uint64_t upto = L.chunk_total;
    for (uint32_t q = 0; q < blockDim.x / 64; ++q) upto += L.red64[q];
    if (upto <= 0xFFFFFFFFull) {
      const uint32_t p32 = (uint32_t)upto;
      __hip_atomic_store(pub + 4 * c + 2, ((nz_u64)mark_pa << 32) | p32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(pub + 4 * c + 3, ((nz_u64)mark_pb << 32) | (uint32_t)~p32, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (has_seg) {
    uint64_t o0 = 0;
    for (uint32_t q = 0; q < blockDim.x / 64; ++q) o0 += L.red64[q];
    for (uint32_t q = 0; q < wave; ++q) o0 += L.seg_units[q];
    const bool from_stage = staged && !L.raw;
    const uint16_t* words = from_stage ? reinterpret_cast<const uint16_t*>(stage) + (pos_end - stage_lo) : slot + pos_end;
    NzChunkInfo ci;  // as nz_build_table and nz_chunk_finalize left it in scratch memory, from LDS
    ci.tab_len = L.tab_len;
    ci.pad_sym = L.pad_sym;
    ci.raw = L.raw ? 1u : 0u;
    ci.reserved = 0;
    const bool fits = nz_move_record<64>(it, seg, c, wave, o0, L.seg_units[wave], ci, L.seg_sb[wave],
                                         cap_words - pos_end, L.ser, L.sbuf[wave], words, nullptr, lane);
    if (from_stage && !fits) unstage();
    if (lane == 0) {
      placed[seg] = (from_stage && fits) ? 1 : 0;
      if (!fits) nz_lb_left_out(lb_state, it.nonce);
    }
  }
  NZ_PROBE_MARK(5);
}

// Longer segments: all wavefronts split the chunk into scratch, then one
// wavefront per segment codes from there.
template <int S>
__global__ __launch_bounds__(NZ_ENC_LONG_THREADS) void nz_encode_long_kernel(const NzEncBatch b) {
  __shared__ NzEncLds L;
  uint32_t t = 0, first = 0;
  while (t + 1 < b.count && blockIdx.x >= b.item[t].chunk_end) {
    first = b.item[t].chunk_end;
    ++t;
  }
  const NzEncItem& it = b.item[t];
  const NzGeom& g = it.g;
  const uint64_t c = blockIdx.x - first;
  const uint64_t n = g.n;
  const uint32_t chunk_syms = g.chunk_syms, seg_syms = g.seg_syms, spc = g.spc;
  const uint16_t* __restrict__ in = it.in;
  const NzNorm nm = it.nm;
  uint8_t* carry = it.ws + it.carry;
  uint8_t* exps = it.ws + it.exps;
  NzChunkInfo* info = reinterpret_cast<NzChunkInfo*>(it.ws + it.info);
  uint32_t* seg_words = reinterpret_cast<uint32_t*>(it.ws + it.seg_words);
  uint32_t* seg_state_bytes = reinterpret_cast<uint32_t*>(it.ws + it.seg_sbytes);
  uint32_t* seg_units = reinterpret_cast<uint32_t*>(it.ws + it.seg_units);

  const uint32_t tid = threadIdx.x;
  const uint64_t base = c * chunk_syms;
  const uint32_t cn = (uint32_t)((n - base) < chunk_syms ? (n - base) : chunk_syms);

  NzHist::clear(nz_enc_stage, b.copies_log2);
  __syncthreads();
  const NzHist hist{nz_enc_stage + (tid & ((1u << b.copies_log2) - 1u)), b.copies_log2};

  const uint32_t seg_keep = seg_syms / 8 * (S + 1) - NZ_CARRY_BYTES;     // of a segment of nominal length
  const uint64_t chunk_keep = (uint64_t)chunk_syms / 8 * (S + 1) - (uint64_t)NZ_CARRY_BYTES * spc;
  const uint64_t seg0 = c * spc;
  for (uint32_t i = tid * 8; i < cn; i += blockDim.x * 8) {
    const uint64_t gi = base + i;
    const uint32_t sk = i / seg_syms;                       // segment inside the chunk
    const uint32_t sb = (i - sk * seg_syms) / 8 * (S + 1);  // byte inside the segment
    const uint32_t nom = nz_seg_nominal(chunk_syms, seg_syms, spc, sk);
    const uint32_t keep = nom / 8 * (S + 1) - NZ_CARRY_BYTES;
    const bool seg_full = base + (uint64_t)sk * seg_syms + nom <= n;
    uint8_t* pp = (seg_full && sb >= keep) ? carry + (seg0 + sk) * NZ_CARRY_BYTES + (sb - keep)
                                           : it.packed + c * chunk_keep + (uint64_t)sk * seg_keep + sb;
    const uint32_t rem = cn - i;
    uint64_t e;
    if (rem >= 8) {
      uint4 v = *reinterpret_cast<const uint4*>(in + gi);
      if (nm.bytes) v = nz_scale8<false>(v, nz_norm_load8(nm, gi), nm.log2n >= 3);
      uint64_t f;
      nz_split_group<S>(v, e, f);
      nz_store_packed<S>(pp, f);
      *reinterpret_cast<uint64_t*>(exps + gi) = e;
#pragma unroll
      for (int j = 0; j < 8; ++j) hist.count((uint32_t)(e >> (8 * j)) & 0xFFu);
    } else {
      e = nz_split_tail<S>(in, gi, rem, pp, nm);
      for (uint32_t j = 0; j < rem; ++j) {
        exps[gi + j] = (uint8_t)(e >> (8 * j));
        hist.count((uint32_t)(e >> (8 * j)) & 0xFFu);
      }
    }
  }
  __syncthreads();
  nz_build_table(L, nz_enc_stage, b.copies_log2, cn, it.ws + it.tab_ser + c * NZ_TABLE_MAX_BYTES, info + c);
  // exponents and carried bytes of this chunk are read back below
  __threadfence_block();
  __syncthreads();

  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lane = tid & 63;
  const uint64_t seg = seg0 + wave;
  const uint64_t seg_base = base + (uint64_t)wave * seg_syms;
  const uint32_t cap_words = seg_syms;
  uint16_t* slot = reinterpret_cast<uint16_t*>(it.ws + it.slots) + seg * cap_words;
  const bool has_seg = wave < spc && seg_base < n;
  uint32_t seg_n = 0;
  if (has_seg) {
    const uint32_t nom = nz_seg_nominal(chunk_syms, seg_syms, spc, wave);
    seg_n = (uint32_t)((n - seg_base) < nom ? (n - seg_base) : nom);
    const uint32_t ngroups = (seg_n + NZ_GROUP_SYMS - 1) / NZ_GROUP_SYMS;
    const uint32_t pad = L.pad_sym;
    const uint8_t* src = exps + seg_base;
    uint32_t x = NZ_L | (seg_n == nom ? (uint32_t)reinterpret_cast<const uint16_t*>(carry)[seg * NZ_LANES + lane] : 0u);
    uint32_t pos = 2 * cap_words;
    const auto group_syms = [&](uint32_t gq) {
      const uint32_t idx0 = (gq * NZ_LANES + lane) * NZ_GROUP;
      uint64_t sy = 0;
      if (idx0 + 8 <= seg_n) return *reinterpret_cast<const uint64_t*>(src + idx0);
      for (int j = 0; j < 8; ++j) {
        uint32_t bb = (idx0 + j < seg_n) ? src[idx0 + j] : pad;
        sy |= (uint64_t)bb << (8 * j);
      }
      return sy;
    };
    uint64_t sy = group_syms(ngroups - 1);
    NzEncAhead ahead;
    ahead.start(L.tab, sy);
    for (uint32_t gq = ngroups; gq-- > 0;) {
      const uint64_t sy_next = group_syms(gq ? gq - 1 : 0);
      nz_enc_group<false>(x, pos, sy, sy_next, ahead, L.tab, slot, 0u);
      sy = sy_next;
    }
    nz_enc_finish(x, cap_words - pos / 2, seg, L.sbuf[wave], lane, reinterpret_cast<uint32_t*>(it.ws + it.states),
                  seg_words, seg_state_bytes, &L.seg_w[wave], &L.seg_sb[wave]);
  }
  __threadfence_block();
  __syncthreads();
  if (tid < 64) {
    const bool raw = nz_chunk_finalize(c, n, chunk_syms, seg_syms, spc, info, L.seg_w, L.seg_sb, L.tab_len, seg_units,
                                       reinterpret_cast<uint32_t*>(it.ws + it.chunk_units), L.seg_units,
                                       &L.chunk_total);
    if (tid == 0) L.raw = raw;
  }
  __syncthreads();
  if (L.raw && has_seg) {
    // a chunk that does not compress: its exponent bytes take the place of the words
    uint8_t* rawp = reinterpret_cast<uint8_t*>(slot);
    const uint8_t* src = exps + seg_base;
    for (uint32_t i = lane; i < seg_n; i += 64) rawp[i] = src[i];
  }
}

// ----------------------------------------------------------------------------
// container size, header
// ----------------------------------------------------------------------------

// sum of v over the 256 threads of the workgroup, in every thread
__device__ __forceinline__ uint64_t nz_block_sum64(uint64_t v, uint64_t* red4) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor((unsigned long long)v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = v;
  __syncthreads();
  return red4[0] + red4[1] + red4[2] + red4[3];
}

#ifndef NZ_TEMPLATES_ONLY
// Container size of every tensor of the batch from the record sizes of its
// chunks (one workgroup of 256 threads per tensor): for a caller that wants the
// size before it provides the container's memory.  A tensor without elements
// has no compaction workgroup: its (header-only) container is written here
// when `comp` is known.
__global__ __launch_bounds__(256) void nz_total_kernel(const NzEncBatch b) {
  __shared__ uint64_t red4[4];
  const NzEncItem& it = b.item[blockIdx.x];
  const NzGeom& g = it.g;
  const uint32_t* __restrict__ chunk_units = reinterpret_cast<const uint32_t*>(it.ws + it.chunk_units);
  uint64_t part = 0;
  for (uint64_t i = threadIdx.x; i < g.n_chunks; i += 256) part += chunk_units[i];
  const uint64_t units = nz_block_sum64(part, red4);
  if (threadIdx.x == 0) {
    const uint64_t total = g.rec_off + 4 * units + NZ_TAIL_PAD;
    *it.d_total = total;
    if (total > it.comp_cap || units > 0xFFFFFFFFull) atomicOr(it.d_status, 1u);
    if (g.n_segs == 0 && it.comp && total <= it.comp_cap) {
      nz_write_header(it.comp, g, total);
      reinterpret_cast<uint32_t*>(it.comp + g.dir_off)[0] = 0;
      for (uint32_t q = 0; q < NZ_TAIL_PAD; ++q) it.comp[g.rec_off + q] = 0;
    }
  }
}

// ----------------------------------------------------------------------------
// move every segment record to its final place: one workgroup per segment
// ----------------------------------------------------------------------------
// The workgroup of segment k of chunk c finds where its record goes by itself:
// the record sizes of all chunks before c (one number per chunk, left by the
// encode kernel) plus those of the segments before k in c.
__device__ __forceinline__ void nz_compact_segment(const NzEncItem& it, const uint64_t seg, uint64_t* red4) {
  const NzGeom& g = it.g;
  const NzChunkInfo* __restrict__ info = reinterpret_cast<const NzChunkInfo*>(it.ws + it.info);
  const uint32_t* __restrict__ seg_words = reinterpret_cast<const uint32_t*>(it.ws + it.seg_words);
  const uint32_t* __restrict__ seg_state_bytes = reinterpret_cast<const uint32_t*>(it.ws + it.seg_sbytes);
  const uint32_t* __restrict__ seg_units = reinterpret_cast<const uint32_t*>(it.ws + it.seg_units);
  const uint32_t* __restrict__ chunk_units = reinterpret_cast<const uint32_t*>(it.ws + it.chunk_units);
  const uint64_t c = seg / g.spc;
  const uint32_t k = (uint32_t)(seg - c * g.spc);
  const uint32_t tid = threadIdx.x;
  // everything the move depends on is fetched at once: one round of memory latency
  uint64_t part = 0;
  for (uint64_t i = tid; i < c; i += 256) part += chunk_units[i];
  if (tid < k) part += seg_units[c * g.spc + tid];
  const uint32_t mine = seg_units[seg];
  const NzChunkInfo ci = info[c];
  const uint32_t sbytes = seg_state_bytes[seg];
  const uint32_t w = seg_words[seg];
  const bool in_old = it.use_placed && (it.ws + it.placed)[seg] != 0;
  const uint64_t o0 = nz_block_sum64(part, red4);
  const uint16_t* words = reinterpret_cast<const uint16_t*>(it.ws + it.slots) + seg * g.seg_syms + (g.seg_syms - w);
  nz_move_record<256>(it, seg, c, k, o0, mine, ci, sbytes, w,
                      reinterpret_cast<const uint32_t*>(it.ws + it.tab_ser + c * NZ_TABLE_MAX_BYTES),
                      reinterpret_cast<const uint32_t*>(it.ws + it.states) + seg * (NZ_STATE_MAX_BYTES / 4), words,
                      in_old ? it.old_comp + g.rec_off + 4 * o0 : nullptr, tid);
}
__global__ __launch_bounds__(256) void nz_compact_kernel(const NzEncBatch b) {
  __shared__ uint64_t red4[4];
  uint32_t t = 0, first = 0;
  while (t + 1 < b.count && blockIdx.x >= b.item[t].seg_end) {
    first = b.item[t].seg_end;
    ++t;
  }
  nz_compact_segment(b.item[t], blockIdx.x - first, red4);
}
// Between an in-place write and a read that the host enqueues before it knows how the write went:
// the tensors of which the write has left a record out of the container (it outgrew its buffer, or
// a chunk gave up waiting) are put together again in a buffer that holds any container, and the read
// goes by the same mark (NzBatchItem::late).  There is next to never anything to do, so the grid
// is small, and the marks of all tensors are looked at together: 1.5 to 4 us (64 workgroups that look at one
// tensor after the other: 4.3).
__global__ __launch_bounds__(256) void nz_late_kernel(const NzEncBatch b) {
  __shared__ uint64_t red4[4];
  const uint32_t lane = threadIdx.x & 63, mine = lane < b.count ? lane : 0;  // all tensors' marks at once
  const NzLbWords* words = reinterpret_cast<const NzLbWords*>(b.item[mine].ws + b.item[mine].lb_state);
  const bool not_whole = nz_lb_not_whole(words, b.item[mine].nonce);
  for (uint64_t todo = __ballot(lane < b.count && not_whole); todo; todo &= todo - 1) {
    const NzEncItem& it = b.item[__builtin_ctzll(todo)];
    for (uint64_t seg = blockIdx.x; seg < it.g.n_segs; seg += gridDim.x) nz_compact_segment(it, seg, red4);
  }
}

#endif  // NZ_TEMPLATES_ONLY

// ----------------------------------------------------------------------------
// fused rANS decode + merge: one workgroup per chunk, one wavefront per segment
// ----------------------------------------------------------------------------
//
// LDS: a 4096-entry slot table of 8-byte entries (32 KiB)
//          lo = freq | nz_rot_exp(symbol) << 24      hi = slot - cum[symbol]
//      (so that one v_mad_u32_u24 of lo's low 24 bits gives the next state and
//      the symbol is a whole byte for v_perm_b32), and per wavefront a ring that
//      slides over the segment's record and first holds the record's head
//      (table, coder states, first words).  What the table parse leaves for the
//      fill lies under the table's last slots.
// A rANS step per lane: x = freq * (x >> 12) + hi, and when the state falls below
// 2^16 a 16-bit word taken at (words consumed so far by the wave + rank of the
// lane among the lanes that need one).  Two forms:
//   NzWaveDec     slot read, then the word's read: the ring holds 1024 words
//                 (2 KiB); a workgroup of eight wavefronts has 48 KiB, three
//                 share the 160 KiB of a CU
//   NzWaveDecOne  one read, of a slot or of an entry prepared from the word: the
//                 ring holds the entries of 512 words (4 KiB; 64 KiB, two
//                 workgroups to a CU) in launches of at most one workgroup per
//                 CU (nz_one_read), of 256 in fused products of more.

// What the table parse leaves for the slot-table fill (runs, windows, flags)
// lies in the last slots of the table itself; those are filled last, from
// registers.
#define NZ_TMETA_DWORDS (512 + 256 + 4)
#define NZ_TMETA_SLOT ((uint32_t)(NZ_M - 416))  /* first slot under it; a multiple of 32 */
static_assert(2 * (NZ_M - NZ_TMETA_SLOT) >= NZ_TMETA_DWORDS && NZ_TMETA_SLOT % 32 == 0, "parse results fit under the tail");
// dynamic LDS of a decode workgroup whose chunks have up to `spc` segments
#define NZ_DEC_LDS_BYTES(spc, one) ((size_t)8 * (NZ_M + (spc) * ((one) ? NZ_RING_WIDE : NZ_RING_NARROW)))
// Fused products of that many rows stage activations behind the rings, in launches of more than one
// workgroup per compute unit whose chunks have a segment for each row (two groups' worth; 64 KiB in
// all for eight rows and eight segments).
#define NZ_STAGED_ROWS 6
#define NZ_GEMV_LDS_BYTES(spc, one, rows) \
  (NZ_DEC_LDS_BYTES(spc, one) + (!(one) && (rows) >= NZ_STAGED_ROWS && (spc) >= (rows) ? (size_t)2048 * (rows) : 0))
// Launches of at most one workgroup per compute unit decode with NzWaveDecOne and its
// wide ring, unless their output is written with streaming stores.  (Fused products of more
// workgroups take it too, with the narrow ring and in any case: the two-read step took
// 184.5 us for the one-row products of a block of width 4096, this one 168.2.  Exponents of
// six bits, two or three times what weights have, cost it a refill per group: one row times
// 50257 x 1024 of those took 45.0 us and takes 46.6, 14336 x 4096 42.9 and 42.0.)  The line lies
// where the figures of dense output crossed for the default chunk (eight wavefronts, 256 symbols
// per lane; MI355X, 256 compute units; two-read against one-read step, microseconds, taken when
// the one-read step was some 5 % longer than it is):
//   read     8 workgroups 29.7 / 25.2, 128: 33.6 / 29.7, 256: 34.6 / 31.7,
//            257: 40.7 / 40.7, 320: 41.2 / 41.2, 512: 42.9 / 44.4, 768: 62.6 / 67.1
//   gather   1 row 32.5 / 27.8, 256 rows 40.5 / 38.1, 320 rows 48.2 / 47.8, 512 rows 52.4 / 53.3
// It counts workgroups and not wavefronts: chunks of four wavefronts (65536 / 256)
// would still gain above it (320: 34.6 / 30.8, 512: 35.5 / 32.4, 768: 39.4 / 38.3)
// and lose at 1024 (45.2 / 61.1).  Those keep the two-read step, and so do reads with normalizers (narrow
// ring; precision 3, groups of 64: 320 chunks 45.0 / 45.3, 512: 49.7 / 51.3, precision 7: 45.5 / 44.7, 52.2 / 52.5).
// Below the line it costs where a wavefront
// takes many words (6 bits per exponent, 256 workgroups: 36.3 / 36.9; 8 workgroups:
// 29.8 / 27.1) and where four streams launch 256 workgroups each at the same time
// (342 / 370 for sixteen reads: two workgroups to a compute unit and not three;
// two such streams 206 / 204, eight of 128 workgroups 486 / 459).
NZ_HD static inline bool nz_one_read(uint64_t workgroups, uint32_t compute_units, bool stream_out) {
  return !stream_out && workgroups <= compute_units;
}
// Workgroups that share a chunk, where a launch would leave compute units idle: each builds the slot
// table, and decodes an equal part of the segments.  A wavefront with a SIMD unit to itself takes its
// steps faster than one of two, of which the younger waits for the older (140 and 158 cycles per step in a
// workgroup of eight), and the wavefronts of a compute unit share its LDS and vector L1.  Reads of 8, 32,
// 64 and 128 chunks 25.1, 24.9, 26.2, 27.9 -> 22.3, 22.2, 23.8, 25.1 us, products of eight
// rows 36.4, 35.1, 32.6, 33.0 -> 30.2, 29.1, 27.3, 27.9; 160 chunks, which stay whole, 28.4 and 33.4.  Four and
// eight streams with 128 chunks each, at once: 212 and 419 us either way; with rings for whole chunks 239 and 484.
#define NZ_MAX_PARTS 8u
NZ_HD static inline uint32_t nz_parts(uint64_t chunks, uint32_t spc, uint32_t compute_units, bool stream_out) {
  uint32_t parts = 1;
  while (!stream_out && 2 * parts <= spc && 2 * parts <= NZ_MAX_PARTS && 2 * parts * chunks <= compute_units) parts *= 2;
  return parts;
}
// rings that a workgroup needs: its segments', and the first one's for the table
NZ_HD static inline uint32_t nz_part_rings(uint32_t spc, uint32_t parts) {
  return parts > 1 ? (spc + parts - 1) / parts + 1 : spc;
}

// S+1 packed bytes of one 8-element group, as a little-endian integer
template <int S>
__device__ __forceinline__ uint64_t nz_load_sm(const uint8_t* p) {
  if constexpr (S == 7) return *reinterpret_cast<const uint64_t*>(p);
  else if constexpr (S == 3) return *reinterpret_cast<const uint32_t*>(p);
  else if constexpr (S == 1) return *reinterpret_cast<const uint16_t*>(p);
  else return *p;
}

// 8 decoded values to the dense output as a streaming (non-temporal) 16-byte
// store: for outputs too large to stay in the last-level cache until their
// consumer runs (nz_stream_output).
__device__ __forceinline__ void nz_stream_store(uint16_t* p, const uint4 v) {
  typedef uint32_t nz_u32x4 __attribute__((ext_vector_type(4)));
  const nz_u32x4 q = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(q, reinterpret_cast<nz_u32x4*>(p));
}

// Output policy of a decode.  A tensor whose dense form is at most half of the
// 256 MB last-level cache is written with ordinary stores: the GEMM that
// consumes the weight right after finds it there (decode + matrix-vector
// product of a 128 MiB weight: 66 us instead of 75), and a reused output buffer
// costs nothing extra.  A larger tensor cannot stay resident anyway; writing it
// with streaming stores keeps it from churning the cache (448 MiB: 145 us
// instead of 167).
#ifndef NZ_STREAM_OUT_BYTES
#define NZ_STREAM_OUT_BYTES (128ull << 20)
#endif
NZ_HD static inline bool nz_stream_output(uint64_t n) { return 2 * n > NZ_STREAM_OUT_BYTES; }

// S+1 packed bytes of one group from the stored stream in global memory,
// which a decode reads exactly once: a streaming (non-temporal) load, so that
// the bytes do not displace what the caches could keep.  `off`: where the lane's
// bytes are in the stream of its segment.  One and two bytes come with the 32-bit word
// around them (which the lanes of the group share: stream and groups are multiples of 64 bytes) and
// are shifted down where they are used.  Loaded by themselves, they are kept as a byte or half word until that use,
// groups later, and the compiler masks them to 32 bits wherever it likes: in front of the steps that the load was
// to be under way for, which then wait for memory (one-read step, 256 chunks, precision 1: 33.5 or 36.0 us with
// what else was in the kernel, 31.0 with the word; two-read step, 512 chunks: 51.0 and 45.6).
// ALONE: by themselves all the same.  The row gather, which is bound by one wavefront's steps, needs 16 vector
// registers more with the words and normalizers, and then has room for three workgroups to a compute unit, not four.
template <int S, bool ALONE>
using NzPacked = std::conditional_t<S == 7 || ALONE, uint64_t, uint32_t>;
template <int S, bool ALONE>
__device__ __forceinline__ NzPacked<S, ALONE> nz_stream_sm(const uint8_t* stream, uint32_t off) {
  const uint8_t* p = stream + (S < 3 && !ALONE ? off & ~3u : off);
  if constexpr (S == 7) return __builtin_nontemporal_load(reinterpret_cast<const uint64_t*>(p));
  else if constexpr (S == 3 || !ALONE) return __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p));
  else if constexpr (S == 1) return __builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(p));
  else return __builtin_nontemporal_load(p);
}
// bits that the lane's bytes lie above the word's lowest
template <int S, bool ALONE>
__device__ __forceinline__ uint32_t nz_packed_shift(uint32_t lane) {
  return ALONE ? 0u : S == 1 ? 16 * (lane & 1) : S == 0 ? 8 * (lane & 3) : 0u;
}
// The same for the one normalizer byte of a group of eight elements: the four bytes at `at`, or at `last`, the last
// place that has four, and how far up the byte is.  (256 chunks, precision 3, groups of 64: 35.5 or 38 us with the byte
// alone, 33.0 with the word; two-read step, 512 chunks, precision 0, groups of 8: 53.3 and 49.9.)
struct NzNormByte {
  uint32_t word, up;
  __device__ __forceinline__ uint32_t get() const { return __builtin_amdgcn_ubfe(word, 8 * up, 8); }
};
template <bool ALONE>
__device__ __forceinline__ NzNormByte nz_stream_norm(const uint8_t* bytes, uint32_t at, uint32_t last) {
  if constexpr (ALONE) return NzNormByte{bytes[at], 0u};
  const uint32_t from = at < last ? at : last;
  NzNormByte b;
  __builtin_memcpy(&b.word, bytes + from, 4);
  b.up = at - from;
  return b;
}

// The exponent byte as the decoder's tables hold it: rotated right by one.  An exponent lies across
// the bytes of a bf16 value, seven bits below the sign and one above the mantissa; the rotated
// byte, put into both bytes of the value, has all eight of them in place, so that merging
// needs no shift.
__device__ __forceinline__ constexpr uint32_t nz_rot_exp(uint32_t e) { return (e >> 1) | ((e & 1u) << 7); }
__device__ __forceinline__ constexpr uint32_t nz_unrot_exp(uint32_t r) { return ((r << 1) & 0xFFu) | (r >> 7); }

// Merge 8 exponents (rotated, byte 3 of ew[j]) with the group's packed bytes into 8
// bf16 values.
template <int S>
__device__ __forceinline__ uint4 nz_merge_group(uint64_t sm, const uint32_t (&ew)[8]) {
  uint32_t o[4];
  if constexpr (S == 7) {
    // out16 = sign << 15 | exp << 7 | mant, byte b = sign << 7 | mant.  Per pair:
    //   t = bytes [e0 e0 e1 e1]: exponents on bits 7..14 and 23..30
    //   u = bytes [b0 b0 b1 b1]: sign lands on bit 15 / 31, mantissa on 0..6 / 16..22
    //   out = bitfield insert of t's exponent bits into u
    // (13.4 cycles of the vector ALU per pair; with a shift of t, 17.9)
    const uint32_t lo = (uint32_t)sm, hi = (uint32_t)(sm >> 32);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t t = __builtin_amdgcn_perm(ew[2 * k + 1], ew[2 * k], 0x07070303u);
      const uint32_t w = k < 2 ? lo : hi;
      const uint32_t u = __builtin_amdgcn_perm(0u, w, (k & 1) ? 0x03030202u : 0x01010000u);
      // bitfield insert: (mask & t) | (~mask & u)
      asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(o[k]) : "s"(0x7F807F80u), "v"(t), "v"(u));
    }
  } else {
    // Fewer mantissa bits: the same shape.  A byte that holds an element's sign
    // in bit 7 and its mantissa bits right below goes into both bytes of the
    // element's half (sign on bit 15, mantissa from bit 6 down); what else the
    // byte holds is masked away, and the exponents' bits are or-ed in.
    const uint32_t lo = (uint32_t)sm;
    constexpr uint32_t keep = 0x80008000u | (((0x7Fu << (7 - S)) & 0x7Fu) * 0x00010001u);
    constexpr int NV = S == 3 ? 2 : (S == 1 ? 4 : 8);
    uint32_t v[NV];  // v[i]: the packed bytes shifted left by i fields
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = lo << (i * (S + 1));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t t = __builtin_amdgcn_perm(ew[2 * k + 1], ew[2 * k], 0x07070303u);
      uint32_t u;
      if constexpr (S == 3) {
        // byte k holds elements 2k (high nibble) and 2k + 1
        u = __builtin_amdgcn_perm(v[1], v[0], (uint32_t)(4 + k) * 0x01010000u + (uint32_t)k * 0x0101u);
      } else if constexpr (S == 1) {
        // byte k / 2 holds elements 4 (k / 2) .. + 3, two bits each
        const uint32_t b = (uint32_t)k >> 1;
        u = __builtin_amdgcn_perm(v[2 * (k & 1) + 1], v[2 * (k & 1)], (4 + b) * 0x01010000u + b * 0x0101u);
      } else {
        // one byte holds the eight signs, element 0 in bit 7
        u = __builtin_amdgcn_perm(v[2 * k + 1], v[2 * k], 0x04040000u);
      }
      o[k] = (u & keep) | (t & 0x7F807F80u);
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// ----------------------------------------------------------------------------
// y = W x for one activation row, W decoded on the fly and never written out
// ----------------------------------------------------------------------------
// A group is 512 consecutive weights, 8 in each lane.  The row length is a multiple of 8 and at
// least 512, so a lane's weights lie in one row of W and a group in at most two (in one, always,
// where the row length is a multiple of 512).  A
// lane keeps an fp32 partial sum of its 8-element dot products; what happens
// when the wave leaves a row is described at NzGemvWalk.  Where rows are whole groups, row r owns
// acc[2r] (fixed-point sum) and acc[2r + 1] (contribution count in the low half, flag
// in bit 32).
// 40 fraction bits: an absolute resolution of 9e-13 per partial sum; up to 16
// partial sums below 2^18 in magnitude cannot overflow 64 bits.
#define NZ_GEMV_FRAC_BITS 40
#define NZ_GEMV_PART_MAX 262144.0f /* 2^18 */

struct NzGemv {
  const uint16_t* x;      // as many activation rows as the kernel is for, in_features bf16 values each, 16-byte aligned
  long long* acc;         // accumulators of this tensor, all zero between calls: rows that are whole groups, two words per row
                          // and activation row (sum | count and flag); else acc_words words of 32 bits (count, a partial
                          // sum of each segment that a row can touch)
  uint16_t* y;            // for each activation row one bf16 per row of the tensor
  const uint16_t* bias;   // one bf16 per row of the tensor, or null
  uint32_t in_features;   // multiple of 8, at least 512
  uint32_t acc_words;
};
// 32-bit words of a row's accumulator where rows are not whole groups, in fours: a row of L elements that
// touches k segments holds k - 2 of them, of the shortest `min_seg` elements, and an element of two more
NZ_HD static inline uint32_t nz_row_acc_words(uint32_t in_features, uint32_t min_seg) {
  return (1u + (in_features - 2u) / min_seg + 2u + 3u) & ~3u;
}

struct NzNoLds {};  // the activations of a group are not in LDS

// what a lane holds of the activation rows for one group of 8 weights
template <int MR>
struct NzXq {
  uint4 v[MR];
};

typedef __attribute__((ext_vector_type(2))) __bf16 nz_bf16x2;

__device__ __forceinline__ float nz_dot8(const uint4 w, const uint4 x, float acc) {
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(nz_bf16x2, w.x), __builtin_bit_cast(nz_bf16x2, x.x), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(nz_bf16x2, w.y), __builtin_bit_cast(nz_bf16x2, x.y), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(nz_bf16x2, w.z), __builtin_bit_cast(nz_bf16x2, x.z), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(nz_bf16x2, w.w), __builtin_bit_cast(nz_bf16x2, x.w), acc, false);
  return acc;
}

// Position of a wavefront inside W while it walks its segment group by group.
//
// Rows need not be WHOLE groups.  Where one ends inside a group, the lanes up to there bring their
// last products to it and the lanes behind begin the next row's sums.  Rows that are whole groups
// have kernels of their own, because the other step costs them 4 % (one row through the Linears of
// a block of width 4096: 163 us, 170 with a look at the row's end in every group).
//
// When the wave leaves a row it adds its 64 partial sums in a fixed order.  A row that lies inside the wave's segment is complete then: bias
// added, rounded, stored.  A row shared with other segments goes through the
// row's accumulator: the partial sums of its segments, and a counter of contributions; the wave that brings
// the count to the number of segments the row touches finishes the row and returns the words to zero.
// Where rows are whole groups, the partial sums are added in 24.40 fixed point (integer addition is
// associative, so the result does not depend on which wave arrives first; a
// partial sum that is NaN, infinite or beyond 2^18 sets a flag instead and the
// row comes out as NaN).  Where they are not, each segment leaves its fp32 sum in a word of its own and
// the last wave adds them in the order of the segments: such Linears are products of the GEMM library
// where this kernel does not serve them, so the sums keep fp32's range, infinities and small values.
// (Fixed point brought zero for sums below 2^-41 and NaN for infinite ones.  A block of width 4224, one and
// eight rows: 164.0 and 269.7 us in fixed point, 163.8 and 271.6 with words.)
template <int MR, bool WHOLE>
struct NzGemvWalk {
  NzGemv gv;
  uint64_t row;
  uint64_t seg_first, seg_end;  // elements of the tensor this wave covers
  uint32_t col;        // column of the current group's first element (uniform)
  uint32_t pending;    // groups added since the last flush, or whether there are any (uniform)
  uint32_t seg_syms, last_syms, spc, k;  // segment lengths of a chunk, this wave's segment inside it
  uint32_t lane_off;   // bytes from a group's first activation to this lane's
  uint64_t w_rows;     // rows of the tensor (= elements between two output rows)
  float sum[MR];

  __device__ __forceinline__ void start(const NzGemv& g, const NzGeom& geom, uint64_t first_elem,
                                        uint32_t seg_n, uint32_t wave_in_chunk, uint32_t lane) {
    gv = g;
    lane_off = 16u * lane;
    w_rows = geom.n / g.in_features;
    row = first_elem / g.in_features;
    col = (uint32_t)(first_elem - row * g.in_features);
    seg_first = first_elem;
    seg_end = first_elem + seg_n;
    seg_syms = geom.seg_syms;
    spc = geom.spc;
    last_syms = geom.chunk_syms - (geom.spc - 1) * geom.seg_syms;  // the chunk's (shorter) last segment
    k = wave_in_chunk;
    pending = 0;
#pragma unroll
    for (int m = 0; m < MR; ++m) sum[m] = 0.f;
  }
  __device__ __forceinline__ uint32_t next_col() const {
    if constexpr (WHOLE) return col + NZ_GROUP_SYMS == gv.in_features ? 0u : col + NZ_GROUP_SYMS;
    return col + NZ_GROUP_SYMS >= gv.in_features ? col + NZ_GROUP_SYMS - gv.in_features : col + NZ_GROUP_SYMS;
  }
  // the lane's 8 activations of every row for the group at column c: a scalar address that goes
  // from row to row and the lane's offset.  (Addresses made of row number and stride in each lane took 30 vector
  // instructions per group of eight rows; addresses kept, all scalar registers there are.  Eight
  // rows through the Linears of a block of width 4096: 305 -> 264 us, with flush() below.)
  __device__ __forceinline__ NzXq<MR> load(uint32_t c) const {
    NzXq<MR> r;
    uint32_t stride = 2 * gv.in_features, off = lane_off;
    const uint8_t* p = reinterpret_cast<const uint8_t*>(gv.x + c);
    if constexpr (!WHOLE) {  // the lanes behind the end of the row are at the next one's beginning
      p = reinterpret_cast<const uint8_t*>(gv.x);
      off += 2 * c;
      off = off - stride < off ? off - stride : off;
    }
    asm volatile("" : "+s"(stride), "+v"(off));  // made anew for every group; 32 bits for the offset
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      r.v[m] = *reinterpret_cast<const uint4*>(p + off);
      p += stride;
    }
    return r;
  }
  // Segments the row [first, last] touches, this wave's included, and how many of them come before it: walk
  // over the segment boundaries to the left and to the right (a row rarely spans more
  // than two or three segments; no division).
  __device__ __forceinline__ uint32_t segments_of_row(uint64_t first, uint64_t last, uint32_t* before) const {
    uint32_t count = 1;
    uint64_t at = seg_first;
    uint32_t kk = k;
    while (at > first) {  // the segment before `at` also holds part of the row
      kk = kk ? kk - 1 : spc - 1;
      at -= kk == spc - 1 ? last_syms : seg_syms;
      ++count;
    }
    *before = count - 1;
    at = seg_end;
    kk = k;
    while (at <= last) {  // so does the segment that starts at `at`
      kk = kk + 1 == spc ? 0 : kk + 1;
      at += kk == spc - 1 ? last_syms : seg_syms;
      ++count;
    }
    return count;
  }
  __device__ __forceinline__ void store_row(float v, uint32_t m) const {
    if (gv.bias) v += nz_bf16_to_f32(gv.bias[row]);
    gv.y[(uint64_t)m * w_rows + row] = (uint16_t)nz_f32_to_bf16(v);
  }
  // the row's results, one lane per activation row (for a shared row of eight activations one
  // chain of atomics, not eight after each other)
  __device__ __forceinline__ void flush(uint32_t lane) {
    asm volatile("" : "+v"(lane));  // which lane takes which value is worked out here, not kept across the groups
    const float t = nz_wave_sums<MR>(sum, lane);
    const uint32_t m = nz_sum_index<MR>(lane);
    if (nz_sum_lane<MR>(lane)) {
      const uint64_t first = row * gv.in_features, last = first + gv.in_features - 1;
      if (first >= seg_first && last < seg_end) {
        store_row(t, m);
      } else {
        // Device-scope atomics execute at the L2 in the order they are issued by
        // this lane when each one waits for the value the previous returned, so
        // no cache flush is needed: the count is issued only after the sum's old
        // value has come back, the exchanges only after the count's.
        uint32_t place;
        const uint32_t expected = segments_of_row(first, last, &place);
        uint32_t zero;  // 0, but only the hardware knows: ties the next atomic to the returned value
        if constexpr (WHOLE) {
          unsigned long long* slot = reinterpret_cast<unsigned long long*>(gv.acc + 2 * (row * MR + m));
          unsigned long long r0;
          if (fabsf(t) < NZ_GEMV_PART_MAX)  // false for NaN as well
            r0 = atomicAdd(slot, (unsigned long long)__float2ll_rn(t * (float)(1ull << NZ_GEMV_FRAC_BITS)));
          else
            r0 = atomicOr(slot + 1, 1ull << 32);
          asm volatile("v_and_b32 %0, 0, %1" : "=v"(zero) : "v"((uint32_t)r0));
          const unsigned long long before = atomicAdd(slot + 1, 1ull + zero);
          if ((uint32_t)before + 1u == expected) {
            const long long a = (long long)atomicExch(slot, 0ull);
            const unsigned long long f = atomicExch(slot + 1, 0ull);
            store_row((f >> 32) ? __uint_as_float(0x7FC00000u)
                                : (float)((double)a * (1.0 / (double)(1ull << NZ_GEMV_FRAC_BITS))),
                      m);
          }
        } else {
          uint32_t* slot = reinterpret_cast<uint32_t*>(gv.acc) + (row * MR + m) * gv.acc_words;
          const uint32_t r0 = atomicExch(slot + 1 + place, __float_as_uint(t));
          asm volatile("v_and_b32 %0, 0, %1" : "=v"(zero) : "v"(r0));
          if (atomicAdd(slot, 1u + zero) + 1u == expected) {
            double a = 0.0;  // (exact for two partial sums of like size, so that the rounding below is the only one)
            for (uint32_t q = 0; q < expected; ++q) a += (double)__uint_as_float(atomicExch(slot + 1 + q, 0u));
            atomicExch(slot, 0u);
            store_row((float)a, m);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < MR; ++k) sum[k] = 0.f;
    pending = 0;
  }
  // add the dot products of the current group, then step to the next group
  __device__ __forceinline__ void add(const uint4 w, const NzXq<MR>& x, uint32_t lane) {
    if constexpr (WHOLE) {
#pragma unroll
      for (int m = 0; m < MR; ++m) sum[m] = nz_dot8(w, x.v[m], sum[m]);
      next(lane);
    } else {
      const uint32_t left = gv.in_features - col;
      col = next_col();
      if (left > NZ_GROUP_SYMS) {
#pragma unroll
        for (int m = 0; m < MR; ++m) sum[m] = nz_dot8(w, x.v[m], sum[m]);
        pending = 1;
      } else {
        const bool ends = NZ_GROUP * lane < left;  // this lane's weights still belong to the row
        float behind[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          const float t = nz_dot8(w, x.v[m], ends ? sum[m] : 0.f);
          sum[m] = ends ? t : sum[m];
          behind[m] = ends ? 0.f : t;
        }
        flush(lane);
        ++row;
#pragma unroll
        for (int m = 0; m < MR; ++m) sum[m] = behind[m];
        pending = left < NZ_GROUP_SYMS && row < w_rows;  // (behind the last row there are no weights)
      }
    }
  }
  // the same with the group's activations in LDS, 64 x 16 bytes per row
  __device__ __forceinline__ void add(const uint4 w, const uint4* x, uint32_t lane) {
    static_assert(WHOLE, "");
#pragma unroll
    for (int m = 0; m < MR; ++m) sum[m] = nz_dot8(w, x[NZ_LANES * m + lane], sum[m]);
    next(lane);
  }
  __device__ __forceinline__ void next(uint32_t lane) {
    ++pending;
    col = next_col();
    if (col == 0) {
      flush(lane);
      ++row;
    }
  }
};

// The activations of a workgroup's next group of weights, in LDS, for chunks whose wavefronts are at
// the same column all the time.  Each of the first MR wavefronts brings one activation row's
// part (two buffers, one barrier per group).
template <int MR>
struct NzXStage {
  uint4* buf;
  const uint16_t* row;  // this lane's place in the activation row that the wavefront brings
  uint32_t at;          // ... and in a buffer (16-byte units)
  bool mine;            // whether it brings one

  // Every segment of the chunk begins a row of the matrix and all have the same length.
  static __device__ __forceinline__ bool fits(const NzGeom& g, const NzGemv& gv, uint32_t cn) {
    return g.seg_syms % gv.in_features == 0 && g.chunk_syms == g.spc * g.seg_syms && cn == g.chunk_syms &&
           g.spc >= (uint32_t)MR;
  }
  __device__ __forceinline__ void start(uint4* behind_rings, const NzGemv& gv, uint32_t wave, uint32_t lane) {
    buf = behind_rings;
    mine = wave < (uint32_t)MR;
    at = NZ_LANES * wave + lane;
    row = gv.x + (uint64_t)(mine ? wave : 0u) * gv.in_features + NZ_GROUP * lane;
  }
  __device__ __forceinline__ const uint4* buffer(uint32_t b) const { return buf + b * (NZ_LANES * MR); }
  __device__ __forceinline__ uint4 fetch(uint32_t col) const { return *reinterpret_cast<const uint4*>(row + col); }
  __device__ __forceinline__ void put(uint32_t b, const uint4 x) const {
    if (mine) buf[b * (NZ_LANES * MR) + at] = x;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
};

// A wavefront's record and its ring: where the record lies, what may be loaded of it, and the
// staging of its head.
struct NzRecord {
  uint32_t* ring32;       // at least 512 dwords
  const uint8_t* words;   // start of the record (uniform); word indices count from here
  uint32_t lim;           // largest byte offset from `words` that may be loaded: container end - 16 (uniform)
  uint32_t nwords;        // 16-bit units the record holds, table and states included
  uint32_t lane;

  // record at comp + pos of a container of comp_bytes (pos + 16 <= comp_bytes)
  __device__ __forceinline__ void attach(const uint8_t* comp, uint64_t comp_bytes, uint64_t pos, uint32_t* ring) {
    ring32 = ring;
    words = comp + pos;
    const uint64_t room = comp_bytes - NZ_TAIL_PAD - pos;
    lim = room < 0xFFFFFFF0ull ? (uint32_t)room : 0xFFFFFFF0u;
  }

  // Address of byte `off` of the record, clamped to the container's closing
  // padding: every load of up to 16 bytes through it is in bounds, so the loads
  // are unconditional; words past the record are never consumed by a valid stream.
  __device__ __forceinline__ const uint8_t* at(uint32_t off) const { return words + (off < lim ? off : lim); }

  // 16 bytes of the record at dword index d
  __device__ __forceinline__ uint4 fetch(uint32_t d) const {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(at(4u * d));
    return make_uint4(q[0], q[1], q[2], q[3]);
  }

  // Stage the first 512 dwords of the record (table of a chunk's first record,
  // coder states, first words) where the ring is.
  __device__ __forceinline__ void stage() {
    uint4 v[2];
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) v[q] = fetch(256 * q + 4 * lane);
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) *reinterpret_cast<uint4*>(ring32 + 256 * q + 4 * lane) = v[q];
  }
};

// Decoder state of one wavefront, for dense output in launches of more than one workgroup per
// compute unit, which are bound by memory: the ring holds 1024 words, a window of the record, and
// the loads behind it have six groups to arrive.
struct NzWaveDec : NzRecord {
  static_assert(NZ_RING_DWORDS == 2 * NZ_RING_NARROW, "one size of ring in larger launches");
  const uint2* lut;
  uint32_t ring_lds;      // LDS byte address of the ring (the same in all lanes, kept in a vector register)
  uint32_t x;             // this lane's rANS state
  uint32_t base;          // words consumed by the wave (the same in all lanes, kept in a vector register)
  uint32_t filled;        // dwords staged into the ring (multiple of 256; uniform)
  uint32_t sel_keep, sel_shift;  // byte selectors of the renormalisation (vector registers)
  uint4 r;                // 8 words per lane fetched during the previous group

  __device__ __forceinline__ void commit(uint32_t d, const uint4& v) {
    *reinterpret_cast<uint4*>(ring32 + (d & (NZ_RING_DWORDS - 1))) = v;
  }

  __device__ __forceinline__ void stage() {
    NzRecord::stage();
    filled = 512;
  }

  // Start decoding from state x0; the words begin `first_word` 16-bit units
  // into the record (at most 348, so at least 676 words are staged ahead).
  __device__ __forceinline__ void start(uint32_t x0, uint32_t first_word) {
    x = x0;
    base = first_word;
    filled = __builtin_amdgcn_readfirstlane(filled);
    r = fetch(filled + 4 * lane);  // the 512 words behind the staged window
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    ring_lds = (uint32_t)(uintptr_t)((lds_u32*)ring32);
    // keep the three per-lane constants in vector registers of their own (an
    // instruction can name only one scalar register or literal)
    sel_keep = 0x07060504u;
    sel_shift = 0x05040100u;
    asm volatile("" : "+v"(sel_keep), "+v"(sel_shift), "+v"(ring_lds), "+v"(base));
  }

  // Ring upkeep, before every group: the 512 words that follow the staged window wait in
  // registers (`r`, fetched right after the previous commit, addresses clamped
  // to the container); at the start of a group they are committed to the ring
  // if no more than 512 words are still ahead of `base`, and the next 512 are
  // fetched.  A group consumes at most 8 * 64 = 512 words, so at least 512
  // words are ahead at every group start, the window [base, filled) never
  // exceeds the 1024 ring words, and a fetch has at least one group (for
  // exponent data about six) to arrive before its commit.
  __device__ __forceinline__ void look() {
    const uint32_t ahead = __builtin_amdgcn_readfirstlane(base);
    if ((2 * filled - ahead) <= 512u) {
      commit(filled + 4 * lane, r);
      filled += 256;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      r = fetch(filled + 4 * lane);
    }
  }

  // Decode the next 8 symbols of every lane into byte 3 of ew[0..7] (rotated, nz_rot_exp).
  //
  // A step issues: slot read, multiply-add, compare, the lane's word index
  // (words consumed by the wave + its rank among the lanes that renormalise:
  // the two mbcnt instructions add the rank to `base`), the index wrapped into
  // the ring, the word read, and one byte permute whose selector either keeps
  // the state or shifts the word in; `base` advances by the ballot's
  // popcount.  No execution-mask changes and three scalar instructions per
  // step (popcount and the two waits).
  __device__ __forceinline__ void group(uint32_t (&ew)[8]) {
    typedef __attribute__((address_space(3))) const uint16_t lds_cu16;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint2 e = lut[x & (NZ_M - 1)];
      x = __umul24(e.x, x >> NZ_PROB_BITS) + e.y;
      ew[j] = e.x;
      const bool need = x < NZ_L;
      const uint64_t m = __ballot(need);
      const uint32_t widx = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
      uint32_t ring_word = widx & (NZ_RING_WORDS - 1);
      asm volatile("" : "+v"(ring_word));  // mask, then one shift-add (not shift, mask, add)
      const uint32_t at = (ring_word << 1) + ring_lds;
      uint32_t w = *(lds_cu16*)(uintptr_t)at;
      // keep the word read unconditional: straight-line code, no exec-mask branch
      asm volatile("" : "+v"(w));
      const uint32_t sel = need ? sel_shift : sel_keep;
      x = __builtin_amdgcn_perm(x, w, sel);  // x << 16 | w where the state fell below 2^16
      base += (uint32_t)__popcll(m);
    }
  }
  __device__ __forceinline__ void finish() {}  // the state is complete after every step
};

// Decoder state of one wavefront, for launches that are not bound by memory: those of at most one
// workgroup per compute unit and all fused products.
//
// There a step is bound by its chain of dependent operations where few wavefronts share a
// SIMD, and by its vector instructions where many do.  In NzWaveDec the chain holds two LDS round
// trips: the renormalisation word (its place depends on the ballot of the fresh states),
// then the slot entry that the state with the word shifted in selects.  But a
// state that takes a word w becomes x << 16 | w, so its slot is w & 4095, which
// the word alone decides, and
//   f * ((x << 16 | w) >> 12) + bias = (f << 4) * x + (f * (w >> 12) + bias).
// The ring therefore holds, per word, the slot entry that the word selects with
// its frequency times 16 and f * (w >> 12) added to its bias (it is below 16 f: 16 bits), and
// a step is ONE read: from the ring at the lane's rank where the state fell below
// 2^16, from the slot table otherwise, then one multiply-add.  Table and rings are
// numbered through in entries of 8 bytes (a ring begins at a multiple of its size), so that
// one select and one shift make the address.  A wavefront makes the entries of
// RING / 2 words at a time with independent reads; a weight's exponents take one word
// per six symbols or so.
template <uint32_t RING>
struct NzWaveDecOne : NzRecord {
  // An entry's number is its LDS address over 8: the slot table is the first NZ_M of them (the dynamic LDS
  // begins at address 0, nz_decode_chunk), a ring's number and a word's place in it are or-ed, and the
  // address is made by a 16-bit shift.
  static_assert(NZ_M % RING == 0 && (NZ_M + NZ_MAX_SEGS_PER_CHUNK * RING) * 8 <= 1u << 16, "");
  static constexpr uint32_t BLOCK = RING / 2;  // words the ring is refilled by
  static constexpr uint32_t PER_LANE = BLOCK / NZ_LANES;
  // the wide ring is looked at every so many steps, the most its block can feed; the narrow one per group
  static constexpr int STEPS = RING == NZ_RING_WIDE ? (int)(BLOCK / NZ_LANES) : NZ_GROUP;

  const uint2* lut;
  uint32_t ring_at;       // number of the ring's first entry (the same in all lanes, kept in a vector register)
  uint32_t x;             // this lane's rANS state, before the word it may still have to take
  uint32_t top;           // what the next frequency is multiplied with: x with a word to take, x >> 12 without
  uint32_t widx;          // index of that word
  uint2 e;                // entry of the next step
  uint32_t base;          // words consumed by the wave (the same in all lanes, kept in a vector register)
  uint32_t used;          // the same number, as of the last look at the ring (uniform)
  uint32_t filled;        // words entered into the ring (multiple of 4; uniform)
  uint32_t r[PER_LANE / 2];  // the lane's words of the next block, fetched after the previous refill

  __device__ __forceinline__ void fetch_block(uint32_t first) {  // (first a multiple of 4)
    const uint32_t* q = reinterpret_cast<const uint32_t*>(at(2 * first + 2 * PER_LANE * lane));
#pragma unroll
    for (uint32_t k = 0; k < PER_LANE / 2; ++k) r[k] = q[k];
  }
  // the entries of words first + PER_LANE * lane ... into the ring
  __device__ __forceinline__ void enter(uint32_t first, const uint32_t (&v)[PER_LANE / 2]) {
    uint32_t w[PER_LANE];
    uint2 t[PER_LANE];
#pragma unroll
    for (uint32_t k = 0; k < PER_LANE; ++k) w[k] = k & 1 ? v[k / 2] >> 16 : v[k / 2] & 0xFFFFu;
#pragma unroll
    for (uint32_t k = 0; k < PER_LANE; ++k) t[k] = lut[w[k] & (NZ_M - 1)];
#pragma unroll
    for (uint32_t k = 0; k < PER_LANE; ++k) {
      t[k].y += __umul24(t[k].x, w[k] >> NZ_PROB_BITS);
      t[k].x += __umul24(t[k].x, 15u);  // the symbol stays in byte 3: f << 4 has 16 bits
    }
    uint4* to = reinterpret_cast<uint4*>(ring32 + 2 * ((first + PER_LANE * lane) & (RING - 1)));
#pragma unroll
    for (uint32_t k = 0; k < PER_LANE / 2; ++k) to[k] = make_uint4(t[2 * k].x, t[2 * k].y, t[2 * k + 1].x, t[2 * k + 1].y);
  }
  __device__ __forceinline__ void lds_order() const {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // Start decoding from state x0; the words begin `first_word` 16-bit units
  // into the record (at most 348, so the first RING from a multiple of 4 are staged).
  __device__ __forceinline__ void start(uint32_t x0, uint32_t first_word) {
    const uint32_t from = __builtin_amdgcn_readfirstlane(first_word) & ~3u;
    filled = from + RING;
    fetch_block(filled);  // the block behind the ring's
    uint32_t v[2][PER_LANE / 2];
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h)
#pragma unroll
      for (uint32_t k = 0; k < PER_LANE / 2; ++k) v[h][k] = ring32[(from + h * BLOCK + PER_LANE * lane) / 2 + k];
    lds_order();
    enter(from, v[0]);
    enter(from + BLOCK, v[1]);
    lds_order();
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    ring_at = (uint32_t)(uintptr_t)((lds_u32*)ring32) / 8;
    x = x0;
    top = x0 >> NZ_PROB_BITS;
    widx = first_word;
    e = lut[x0 & (NZ_M - 1)];
    base = used = __builtin_amdgcn_readfirstlane(first_word);
    // keep the per-lane constants in vector registers of their own
    asm volatile("" : "+v"(ring_at), "+v"(base));
  }

  // the block that waits in registers into the ring, the one behind it on its way
  __device__ __forceinline__ void refill() {
    lds_order();  // entries of words already taken are written over
    enter(filled, r);
    filled += BLOCK;
    lds_order();
    fetch_block(filled);
  }

  // Ring upkeep, before every group: when no more than BLOCK words are left ahead of `base`, so that the
  // window [base, filled) never exceeds the ring.
  // Wide ring: looked at again inside a group, before every four steps, which consume at most BLOCK words; for
  // exponent data a fetch then has some three groups to arrive.
  // Narrow ring: looked at once per group.  A group takes 80 words or so of exponent
  // data; one that takes more than there are finds that out by scalar instructions in every step,
  // and refills then.  (Where many wavefronts share a SIMD those cost next to nothing, while a refill
  // every two steps would wait not only for its words but for the loads that the same
  // group has issued: 173 us for the Linears of a block of width 4096, and 167 us this way.  With
  // the wide ring and few wavefronts it is the other way round: 25.5 and 26.8 us for 8 chunks.)
  //
  // [base - 64, base) may just have been read when a refill writes over it: LDS
  // operations of a wavefront run in order, and the fences keep them so.
  //
  // The look before a group comes ahead of the group's loads: a refill waits for its words, and,
  // because loads return in order and their number differs from way to way, for every other load
  // under way, those from memory too.  (Four rows through the Linears of a block of width
  // 4096: 191 -> 188 us; read of 5003 x 3001, precision 3, normalizers: 32.3 -> 31.4 us.)
  __device__ __forceinline__ void look() {
    if constexpr (STEPS < NZ_GROUP) used = __builtin_amdgcn_readfirstlane(base);
    if (filled - used <= BLOCK) refill();
  }

  // Decode the next 8 symbols of every lane into byte 3 of ew[0..7] (rotated, nz_rot_exp).
  __device__ __forceinline__ void group(uint32_t (&ew)[8]) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) const u32x2 lds_cu64;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j % STEPS == 0 && j) look();
      x = __umul24(e.x, top) + e.y;
      ew[j] = e.x;
      const bool need = x < NZ_L;
      const uint64_t m = __ballot(need);
      widx = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
      const uint32_t entry = need ? ((widx & (RING - 1)) | ring_at) : (x & (NZ_M - 1));
      uint32_t addr;  // entry * 8; the numbers stay below 8192.  (The 16-bit shift runs at twice the rate.)
      asm("v_lshlrev_b16 %0, 3, %1" : "=v"(addr) : "v"(entry));
      const uint32_t taken = (uint32_t)__popcll(m);
      if constexpr (STEPS == NZ_GROUP) {
        used += taken;
        if (__builtin_expect(used > filled, 0)) refill();
      }
      const u32x2 v = *(lds_cu64*)(uintptr_t)addr;
      e = make_uint2(v.x, v.y);
      top = need ? x : x >> NZ_PROB_BITS;
      base += taken;
    }
  }

  // The state after the last step, with the word it took: the ring does not
  // hold the words themselves, so that one comes from the record again.
  __device__ __forceinline__ void finish() {
    if (x < NZ_L) x = (x << 16) | *reinterpret_cast<const uint16_t*>(at(2u * widx));
  }
};

// The part of the tensor that a row gather takes from a chunk: elements [first, last] go to out[0] ...
struct NzRowOut {
  uint16_t* out;
  uint64_t first, last;
  bool vec;  // out 16-byte aligned and first a multiple of 8: groups of 8 can be stored whole

  __device__ __forceinline__ bool overlaps(uint64_t from, uint32_t count) const {
    return from <= last && from + count > first;
  }
  __device__ __forceinline__ void store1(uint64_t e, uint32_t h) const {
    if (e >= first && e <= last) out[e - first] = (uint16_t)h;
  }
  __device__ __forceinline__ void store8(uint64_t e, const uint4 v) const {
    if (vec && e >= first && e + 7 <= last) {
      *reinterpret_cast<uint4*>(out + (e - first)) = v;
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) store1(e + j, w[j >> 1] >> (16 * (j & 1)) & 0xFFFFu);
    }
  }
};

// One workgroup decodes chunk `c` of one tensor; wavefront k of the workgroup
// takes segment k of the chunk (wavefronts beyond the chunk's segments only
// help to build the slot table).
// With GEMV the decoded values are not stored: they are multiplied with the
// activation `gv.x` and summed into `gv.acc` (the tensor is a row-major matrix
// with rows of gv.in_features elements, a multiple of 8: a lane's 8 weights exist
// all or not at all, and belong to one row).
// With NORM every merged value is multiplied by its group's factor (`nm`)
// before it is stored or used.
// Where several workgroups share the chunk, this one's segments are from first_seg to before end_seg.
// With ROWS only the segments that hold elements of `row` are decoded, and only those elements
// stored; the wavefronts of the others help with the table, and LDS has rings for the first
// segment's record and for as many segments as a row can touch.
template <int S, int GEMV, bool NORM, bool STREAM, bool ONE, bool WHOLE = true, bool ROWS = false>
__device__ __forceinline__ void nz_decode_chunk(
    const uint8_t* __restrict__ comp, const uint64_t comp_bytes, const uint8_t* __restrict__ packed,
    uint16_t* __restrict__ out, const NzGeom& g, uint32_t* __restrict__ d_status, const uint64_t c,
    const NzGemv& gv, const NzNorm& nm, const uint32_t first_seg, const uint32_t end_seg,
    const NzRowOut& row = NzRowOut{}) {
  constexpr bool ONE_READ = ONE || GEMV || ROWS;
  // At LDS address 0: a kernel that decodes has no static LDS (pinned in tests/test_kernel_resources.py),
  // because NzWaveDecOne numbers table and rings through from there.
  extern __shared__ uint32_t lds[];
  uint2* lut = reinterpret_cast<uint2*>(lds);                   // 4096 x 8 bytes
  uint32_t* rings = lds + 2 * NZ_M;                             // spc rings
  uint32_t* tmeta = lds + 2 * NZ_TMETA_SLOT;                    // what the table parse leaves for the fill:
  uint2* runs = reinterpret_cast<uint2*>(tmeta);                //   per live symbol (freq | rotated symbol << 24, first slot)
  uint2* wins = runs + 256;                                     //   per 32 slots (bitmap of run starts, runs before)
  uint32_t* tflag = reinterpret_cast<uint32_t*>(wins + 128);    //   [0] frequencies sum to 4096, [1] table bytes
  const uint8_t* tb = reinterpret_cast<const uint8_t*>(rings);  // table bytes: start of the first record

  const uint32_t tid = threadIdx.x;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keep it scalar
  const uint32_t lane = tid & 63;
  const uint64_t seg0 = c * g.spc;
  const uint64_t chunk_base = c * g.chunk_syms;
  const uint32_t cn =
      (uint32_t)((g.n - chunk_base) < g.chunk_syms ? (g.n - chunk_base) : g.chunk_syms);
  const uint32_t nseg = (cn + g.seg_syms - 1) / g.seg_syms;
  const uint32_t* dir = reinterpret_cast<const uint32_t*>(comp + g.dir_off);

  // the container must be the one the caller's geometry describes
  if (c == 0 && tid == 0) {
    const uint32_t* h = reinterpret_cast<const uint32_t*>(comp);
    if (h[0] != NZ_MAGIC || h[1] != NZ_FORMAT_VERSION || h[2] != (uint32_t)g.n || h[3] != (uint32_t)(g.n >> 32) ||
        h[4] != g.chunk_syms || h[5] != g.lane_syms)
      atomicOr(d_status, 16u);
  }

  // Two rounds of global loads, then only LDS: every wavefront reads the
  // chunk's directory entries itself, then stages the first 2 KiB of its
  // record into its ring (for the chunk's first record that window begins with
  // the table, which all wavefronts parse from there) and fetches the packed
  // bytes of its first group.
  const uint32_t dv = lane <= nseg ? dir[seg0 + lane] : 0u;
  const uint64_t f0 = __builtin_amdgcn_readlane(dv, 0), f1 = __builtin_amdgcn_readlane(dv, 1);
  if (f1 <= f0 || g.rec_off + 4 * f1 + NZ_TAIL_PAD > comp_bytes) {
    if (tid == 0) atomicOr(d_status, 2u);
    return;
  }
  bool has_seg = wave < nseg;
  uint32_t ring = wave;  // the first segment's record, with the table, has the first one
  if constexpr (ONE && !ROWS) {
    has_seg = has_seg && wave >= first_seg && wave < end_seg;
    ring = wave - first_seg + (first_seg ? 1u : 0u);
  }
  if constexpr (ROWS) {
    const uint32_t from = row.first > chunk_base ? (uint32_t)((row.first - chunk_base) / g.seg_syms) : 0u;
    has_seg = has_seg && row.overlaps(chunk_base + (uint64_t)wave * g.seg_syms, g.seg_syms);
    ring = wave - (from > 1 ? from - 1 : 0u);
  }
  const uint32_t wk = has_seg ? wave : 0u;  // wavefronts without a segment only help with the table
  if (wk == 0) ring = 0;
  const uint64_t seg_base = chunk_base + (uint64_t)wk * g.seg_syms;
  const uint32_t nom = nz_seg_nominal(g.chunk_syms, g.seg_syms, g.spc, wk);
  const uint32_t seg_n = (uint32_t)((g.n - seg_base) < nom ? (g.n - seg_base) : nom);
  const uint32_t ngroups = (seg_n + NZ_GROUP_SYMS - 1) / NZ_GROUP_SYMS;
  const uint64_t o0 = __builtin_amdgcn_readlane(dv, wk), o1 = __builtin_amdgcn_readlane(dv, wk + 1);
  const bool bad_rec = o1 < o0 || g.rec_off + 4 * o1 + NZ_TAIL_PAD > comp_bytes;
  const uint64_t rec_pos = g.rec_off + 4 * o0;  // uniform: the readlanes above are scalar
  const uint32_t rec_all = (uint32_t)(4 * (o1 - o0));
  // stored packed layout: every full segment keeps seg_p - 128 bytes, its last
  // 128 bytes ride in the coder states (or behind the symbols of a raw record)
  const bool carry = seg_n == nom;
  const uint32_t keep = nom / 8 * (S + 1) - NZ_CARRY_BYTES;
  const uint64_t chunk_keep = (uint64_t)g.chunk_syms / 8 * (S + 1) - (uint64_t)NZ_CARRY_BYTES * g.spc;
  const uint8_t* pk = packed + c * chunk_keep + (uint64_t)wk * (g.seg_syms / 8 * (S + 1) - NZ_CARRY_BYTES);
  uint16_t* dst = out + seg_base;
  const auto store1 = [&](uint32_t at, uint32_t h) __attribute__((always_inline)) {
    if constexpr (ROWS) row.store1(seg_base + at, h);
    else dst[at] = (uint16_t)h;
  };
  const auto store8 = [&](uint32_t at, const uint4 v) __attribute__((always_inline)) {
    if constexpr (ROWS) row.store8(seg_base + at, v);
    else *reinterpret_cast<uint4*>(dst + at) = v;
  };
  // groups whose packed bytes are (partly) carried are merged after the loop
  const uint32_t tailg = carry ? (S == 0 ? 2u : 1u) : 0u;
  const uint32_t body = ngroups - tailg;
  // Groups in which every lane has 8 elements run without any predicate; the
  // packed bytes are fetched one group ahead of their use (the address of the
  // fetch past the last group is clamped, its value unused).
  const uint32_t whole = seg_n / NZ_GROUP_SYMS < body ? seg_n / NZ_GROUP_SYMS : body;
  const uint32_t lane_off = lane * (S + 1);
  const uint32_t last_off = whole ? (whole - 1) * NZ_LANES * (S + 1) + lane_off : 0u;
  constexpr uint32_t RING = ONE ? NZ_RING_WIDE : NZ_RING_NARROW;
  std::conditional_t<ONE_READ, NzWaveDecOne<RING>, NzWaveDec> w;
  w.lut = lut;
  w.attach(comp, comp_bytes, bad_rec ? 0 : rec_pos, rings + ring * 2 * RING);
  w.nwords = rec_all / 2;
  w.lane = lane;
  const uint64_t norm_bytes = NORM ? ((g.n - 1) >> nm.log2n) + 1 : 0;
  const bool wide_norm = nm.log2n >= 3 && norm_bytes >= 4;
  // Normalizer bytes, where a lane needs one for each of its groups: counted from the segment's first one, or
  // from the last place that has four, in 32 bits.
  const uint64_t norm_first = seg_base >> nm.log2n, norm_four = norm_bytes - 4;
  const uint64_t norm_from = norm_first < norm_four ? norm_first : norm_four;
  const uint8_t* const norm_at = nm.bytes + norm_from;
  const uint32_t norm_off = (uint32_t)(seg_base - (norm_from << nm.log2n)) + lane * NZ_GROUP;
  const uint32_t norm_last = (uint32_t)(norm_four - norm_from < seg_n ? norm_four - norm_from : seg_n);
  NzPacked<S, ROWS> sm_next = 0;
  NzNormByte nb_next{};
  constexpr int MR = GEMV ? GEMV : 1;  // activation rows a lane multiplies with (GEMV: 0 = plain decode)
  // The activation of the next group is fetched a group ahead.  Of several rows it is this
  // group's: the registers of the next ones' cost a workgroup per compute unit where there would
  // be three, and gain nothing where there are two (four rows through the Linears of a block of
  // width 4096: 188 us ahead, 185 us not; eight: 255 and 256 us).
  constexpr bool X_AHEAD = MR == 1;
  NzXq<X_AHEAD ? MR : 1> xq_next{};
  NzGemvWalk<MR, WHOLE> walk;
  if constexpr (ONE || ROWS)
    if (wave == 0 && !has_seg && !bad_rec) w.stage();  // the table
  if (has_seg && !bad_rec) {
    w.stage();
    if constexpr (GEMV) {
      walk.start(gv, g, seg_base, seg_n, wk, lane);
      if constexpr (X_AHEAD) xq_next = walk.load(walk.col);
    }
    if (whole) {
      sm_next = nz_stream_sm<S, ROWS>(pk, lane_off);
      if (NORM && wide_norm) nb_next = nz_stream_norm<ROWS>(norm_at, norm_off >> nm.log2n, norm_last);
    }
  }
  __syncthreads();
  // the first 32 table bytes hold the mode and all run descriptors there can be
  const uint4 h0 = reinterpret_cast<const uint4*>(tb)[0], h1 = reinterpret_cast<const uint4*>(tb)[1];
  const uint32_t bm_byte = tb[1 + (lane >> 1)];  // bitmap mode: the byte with this lane's four symbols
  const uint32_t mode = (uint32_t)__builtin_amdgcn_readfirstlane(h0.x & 0xFFu);
  uint32_t tab_len = 4;

  if (mode != NZ_MODE_RAW) {
    if (mode > NZ_MAX_RUNS) {
      if (tid == 0) atomicOr(d_status, 2u);
      return;
    }
    // Wavefront 0 parses the table, four symbols per lane, and leaves for the
    // fill below: the live symbols in order (`runs`: frequency, symbol, first
    // slot) and, per window of 32 slots, which slots start a run and how many
    // runs start before the window (`wins`).
    if (wave == 0) {
      wins[lane] = make_uint2(0u, 0u);
      wins[lane + 64] = make_uint2(0u, 0u);
      uint32_t head, kk = 0, live4 = 0;
      uint32_t rk[4] = {0, 0, 0, 0};  // rank of the symbol among those the table lists
      if (mode == NZ_MODE_BITMAP) {
        head = 33;
        live4 = (bm_byte >> (4 * (lane & 1))) & 15u;
        const uint32_t c = (uint32_t)__popc(live4);
        const uint32_t ci = nz_wave_scan(c, lane);
        kk = __builtin_amdgcn_readlane(ci, 63);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) rk[j] = ci - c + (uint32_t)__popc(live4 & ((1u << j) - 1u));
      } else {
        head = 1 + 2 * mode;
        uint32_t acc = 0;
        // the run descriptors, 16 bits each from the second byte on, move down through scalar registers
        const auto pair = [](uint32_t lo, uint32_t hi) {
          return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(lo) | ((uint64_t)__builtin_amdgcn_readfirstlane(hi) << 32);
        };
        uint64_t q0 = pair(h0.x, h0.y), q1 = pair(h0.z, h0.w), q2 = pair(h1.x, h1.y), q3 = pair(h1.z, h1.w);
#pragma nounroll
        for (uint32_t r = 0; r < mode; ++r) {
          const uint32_t st = (uint32_t)(q0 >> 8) & 0xFFu, ln = ((uint32_t)(q0 >> 16) & 0xFFu) + 1u;
          q0 = q0 >> 16 | q1 << 48;
          q1 = q1 >> 16 | q2 << 48;
          q2 = q2 >> 16 | q3 << 48;
          q3 >>= 16;
#pragma unroll
          for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t d = 4 * lane + j - st;
            if (d < ln) {
              live4 |= 1u << j;
              rk[j] = acc + d;
            }
          }
          acc += ln;
        }
        kk = acc;
      }
      if (kk > 256) kk = 256;  // corrupt input: stay inside the staged bytes
      uint32_t fr[4], tot = 0, nz4 = 0;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t f = nz_get12(tb + head, rk[j] > 255 ? 255u : rk[j]);  // read in any case: no branch
        fr[j] = ((live4 >> j) & 1u) ? f : 0u;
        tot += fr[j];
        nz4 += fr[j] ? 1u : 0u;
      }
      // one scan for both the cumulative frequency (below 2^20) and the number of
      // symbols with a nonzero frequency (from bit 20 up)
      const uint32_t mine = tot | (nz4 << 20);
      const uint32_t incl = nz_wave_scan(mine, lane);
      const uint32_t all = __builtin_amdgcn_readlane(incl, 63);
      const bool sums = (all & 0xFFFFFu) == NZ_M;
      if (lane == 0) {
        tflag[0] = sums ? 1u : 0u;
        tflag[1] = (head + (12 * kk + 7) / 8 + 3) & ~3u;
      }
      if (sums) {  // only then do the first slots stay below 4096
        uint32_t first = (incl - mine) & 0xFFFFFu, k = (incl - mine) >> 20;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
          if (fr[j]) {
            runs[k] = make_uint2(fr[j] | (nz_rot_exp(4 * lane + j) << 24), first);
            atomicOr(&wins[first >> 5].x, 1u << (first & 31));
            ++k;
            first += fr[j];
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // runs that start before each window: prefix of the bitmap's popcounts
        const uint32_t b0 = wins[2 * lane].x, b1 = wins[2 * lane + 1].x;
        const uint32_t c0 = (uint32_t)__popc(b0), c1 = (uint32_t)__popc(b1);
        const uint32_t pi = nz_wave_scan(c0 + c1, lane);
        wins[2 * lane].y = pi - c0 - c1;
        wins[2 * lane + 1].y = pi - c1;
      }
    }
    __syncthreads();
    // Slot table: a thread fills eight consecutive slots, in pairs of 16 bytes.  The run of a slot is the
    // number of runs that start at or before it, minus one; the eight lie in one window, and rarely
    // does a pair hold the start of a run in its second slot.  (Of a table whose frequencies
    // do not sum to 4096 nothing was written: the fill then reads zeros and the chunk is given up
    // right after.)  The last slots lie under the parse results: the threads' last entries wait
    // in registers until all have read what they need.  Neighbouring lanes' pairs are in turn: eight lanes
    // write to different banks.  (One slot at a time, two LDS reads and a write of 8 bytes for each, the
    // fill took 2900 cycles, of some 50000 that a chunk of 256 symbols per lane takes.  With this, and the
    // run descriptors in scalar registers above: read of 1024 x 1024 22.2 -> 21.5 us, gather of a row 21.8 -> 21.2,
    // one and eight rows through the Linears of a block of width 4096 160.6 -> 158.4, 237.4 -> 234.0; reads of 128
    // chunks, precision 0, 26.0 -> 25.1, precision 7 with normalizers of 64 27.6 -> 27.0, of 512 chunks, two-read
    // step, precision 1, 46.4 -> 45.9.)
    {
      const auto slot_at = [&](uint32_t at, uint32_t i) { return at + 2u * ((i + (lane >> 2)) & 3u); };
      const auto entries = [&](uint32_t at, uint4 (&en)[4]) {
        const uint2 wn = wins[at >> 5];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
          const uint32_t slot = slot_at(at, i), bit = slot & 31;
          const uint32_t k = wn.y + (uint32_t)__popc(wn.x & ((2u << bit) - 1u)) - 1u;
          const uint2 a = runs[k & 255u];
          uint2 b = a;
          if ((wn.x >> (bit + 1)) & 1u) b = runs[(k + 1u) & 255u];
          en[i] = make_uint4(a.x, slot - a.y, b.x, slot + 1u - b.y);
        }
      };
      const auto put = [&](uint32_t at, const uint4 (&en)[4]) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(lut + slot_at(at, i)) = en[i];
      };
      uint4 en[4];
      // (whole rounds end at slot 3584 at the latest, with 64, 128, ... 512 threads)
      static_assert(NZ_M - 8 * NZ_LANES <= NZ_TMETA_SLOT, "");
      uint32_t at = 8 * tid;
      for (uint32_t done = 8 * blockDim.x; done < NZ_M; done += 8 * blockDim.x, at += 8 * blockDim.x) {
        entries(at, en);
        put(at, en);
      }
      if (at < NZ_M) entries(at, en);
      const uint32_t table_ok = tflag[0], table_len = tflag[1];
      __syncthreads();
      if (at < NZ_M) put(at, en);
      if (!table_ok) {
        if (tid == 0) atomicOr(d_status, 2u);
        return;
      }
      tab_len = table_len;
    }
  }
  __syncthreads();

  if (!has_seg) return;
  // the chunk's first record begins with the table
  const uint32_t rec_skip = wave == 0 ? tab_len : 0u;
  const bool damaged = bad_rec || rec_all < rec_skip;
  const uint64_t rec_start = rec_pos + rec_skip;
  const uint32_t rec_bytes = rec_all - rec_skip;

  if (mode == NZ_MODE_RAW) {
    const uint32_t padded = (seg_n + 3) & ~3u;
    if (damaged || rec_bytes < padded + (carry ? NZ_CARRY_BYTES : 0u)) {
      if (lane == 0) atomicOr(d_status, 2u);
      return;
    }
    const uint8_t* raw = comp + rec_start;
    const uint8_t* tailp = raw + padded;
    const auto whole8 = [&](uint32_t idx0) __attribute__((always_inline)) {  // 8 elements of the tensor
      const uint32_t b = idx0 / 8 * (S + 1);
      uint64_t sy = (uint64_t)reinterpret_cast<const uint32_t*>(raw + idx0)[0] |
                    ((uint64_t)reinterpret_cast<const uint32_t*>(raw + idx0)[1] << 32);
      const uint64_t sm = (carry && b >= keep) ? nz_load_sm<S>(tailp + (b - keep)) : nz_load_sm<S>(pk + b);
      uint32_t ew[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) ew[j] = nz_rot_exp((uint32_t)(sy >> (8 * j)) & 0xFFu) << 24;
      uint4 mv = nz_merge_group<S>(sm, ew);
      if constexpr (NORM) mv = nz_scale8<true>(mv, nz_norm_load8(nm, seg_base + idx0), nm.log2n >= 3);
      return mv;
    };
    for (uint32_t gq = 0; gq < ngroups; ++gq) {
      const uint32_t idx0 = (gq * NZ_LANES + lane) * NZ_GROUP;
      if constexpr (GEMV) {  // every lane takes part in the sums, behind the tensor's end with zeros
        uint4 mv = make_uint4(0u, 0u, 0u, 0u);
        if (WHOLE || idx0 < seg_n) mv = whole8(idx0);
        walk.add(mv, walk.load(walk.col), lane);
        continue;
      }
      if (idx0 >= seg_n) continue;
      const uint32_t rem = seg_n - idx0;
      if (rem >= 8) {
        store8(idx0, whole8(idx0));
      } else {
        for (uint32_t j = 0; j < rem; ++j) {
          const uint32_t bit = (idx0 + j) * (S + 1);
          const uint32_t rp = ((uint32_t)pk[bit >> 3] >> (7u - S - (bit & 7u))) & ((2u << S) - 1u);
          uint32_t h = nz_merge_one<S>(raw[idx0 + j], rp);
          if constexpr (NORM) h = nz_norm_mul(h, nm.bytes[(seg_base + idx0 + j) >> nm.log2n]);
          store1(idx0 + j, h);
        }
      }
    }
    if constexpr (GEMV)
      if (walk.pending) walk.flush(lane);
    return;
  }

  // final encoder states, read from the staged window: 64 two-bit length
  // codes, then a nibble stream
  const uint32_t* rec32 = w.ring32 + rec_skip / 4;
  const uint32_t nn = 5u + ((rec32[lane >> 4] >> (2 * (lane & 15))) & 3u);
  const uint32_t incl = nz_wave_scan(nn, lane);
  const uint32_t at = incl - nn;
  const uint32_t sbytes = 16u + ((((__builtin_amdgcn_readlane(incl, 63) + 1u) >> 1) + 3u) & ~3u);
  constexpr bool STAGED = GEMV >= NZ_STAGED_ROWS && !ONE && !NORM && WHOLE;
  uint4* const xbuf = reinterpret_cast<uint4*>(rings + 2 * RING * g.spc);
  if (damaged || rec_bytes < sbytes) {
    if (lane == 0) atomicOr(d_status, 2u);
    if constexpr (STAGED) {
      // the other segments of the chunk are multiplied with the activation row that this wavefront brings
      if (NzXStage<MR>::fits(g, gv, cn)) {
        NzXStage<MR> xs;
        xs.start(xbuf, gv, wave, lane);
        uint32_t col = 0;
        xs.put(0, xs.fetch(0));
        for (uint32_t k = 1; k <= (whole & ~1u); ++k) {  // as often as a wavefront that decodes
          col = col + NZ_GROUP_SYMS == gv.in_features ? 0u : col + NZ_GROUP_SYMS;
          xs.put(k & 1u, xs.fetch(col));
        }
      }
    }
    return;
  }
  // the 8 bytes read here may reach into the words: still inside the window
  const uint32_t fb = 16u + (at >> 1);
  const uint64_t win = (uint64_t)rec32[fb >> 2] | ((uint64_t)rec32[(fb >> 2) + 1] << 32);
  const uint32_t x0 = (uint32_t)(win >> (8 * (fb & 3) + 4 * (at & 1))) & (0xFFFFFFFFu >> (32 - 4 * nn));
  w.start(x0, (rec_skip + sbytes) / 2);

  // Groups in which every lane has 8 elements.  Packed bytes (and normalizer
  // bytes) are fetched TWO groups before their use, alternately into two
  // registers, so that the wait in front of a merge is for a load issued two
  // groups (about two microseconds) earlier and for nothing younger: neither
  // the latency of a load that misses every cache nor the previous group's
  // store is waited for.
  const auto sm_at = [&](uint32_t gq) {
    const uint32_t off = gq * NZ_LANES * (S + 1) + lane_off;
    return nz_stream_sm<S, ROWS>(pk, off < last_off ? off : last_off);
  };
  // `wide`: groups of 8 elements or more, one byte per lane and group (where there are four in all).  The
  // walk over the full groups exists once per case, so that the common one has
  // no branch between the byte's load and its use two groups later (a load
  // behind a branch is waited for at the join, with every store before it).
  const auto nb_at = [&](uint32_t gq, auto wide) {
    const uint32_t e = (gq < whole ? gq : whole - 1) * NZ_GROUP_SYMS;
    if constexpr (decltype(wide)::value) {
      return nz_stream_norm<ROWS>(norm_at, (e + norm_off) >> nm.log2n, norm_last);
    } else {
      const uint64_t v = nz_norm_load8(nm, seg_base + e + lane * NZ_GROUP);
      return nm.log2n >= 3 ? v * 0x0101010101010101ull : v;  // (fewer than four normalizers in all)
    }
  };
  // (`xl`: the group's activations in LDS, or NzNoLds)
  const auto full_group = [&](uint32_t gq, const NzPacked<S, ROWS> sm, const auto nb, auto wide, auto fetch_ahead,
                              auto xl) __attribute__((always_inline)) {
    constexpr bool X_LDS = !std::is_same_v<decltype(xl), NzNoLds>;
    if constexpr (ONE_READ) w.look();  // before the group's loads: a refill waits for all that are under way
    NzXq<MR> xq;
    if constexpr (GEMV && X_AHEAD) {
      xq = xq_next;
      xq_next = walk.load(walk.next_col());  // always inside x
    } else if constexpr (GEMV && !X_LDS) {
      xq = walk.load(walk.col);
    }
    fetch_ahead();  // behind the activations: their wait is then not for bytes from memory as well (eight rows: 265 -> 260 us)
    if constexpr (!ONE_READ) w.look();  // (behind them here: 143 us for 8192 x 28672, before them 145)
    uint32_t ew[8];
    w.group(ew);
    // the merge starts only here: its wait for the packed bytes (and the normalizers' bytes) must not be
    // hoisted in front of the rANS steps
    constexpr bool WIDE = decltype(wide)::value;
    uint32_t sml, smh = 0, nbl = 0, nbh = 0;
    if constexpr (sizeof(sm) == 8) {
      sml = (uint32_t)sm, smh = (uint32_t)(sm >> 32);
      asm volatile("" : "+v"(sml), "+v"(smh), "+v"(ew[7]));
    } else {
      sml = sm;
      asm volatile("" : "+v"(sml), "+v"(ew[7]));
      sml >>= nz_packed_shift<S, ROWS>(lane);
    }
    if constexpr (NORM && WIDE) {
      NzNormByte byte = nb;
      asm volatile("" : "+v"(byte.word), "+v"(ew[7]));
      nbl = byte.get();
    } else if constexpr (NORM) {
      nbl = (uint32_t)nb, nbh = (uint32_t)(nb >> 32);
      asm volatile("" : "+v"(nbl), "+v"(nbh), "+v"(ew[7]));
    }
    if constexpr (ROWS)
      if (!row.overlaps(seg_base + gq * NZ_GROUP_SYMS, NZ_GROUP_SYMS)) return;
    uint4 mv = nz_merge_group<S>(((uint64_t)smh << 32) | sml, ew);
    if constexpr (NORM) mv = nz_scale8<true>(mv, ((uint64_t)nbh << 32) | nbl, WIDE);
    if constexpr (X_LDS) walk.add(mv, xl, lane);
    else if constexpr (GEMV) walk.add(mv, xq, lane);
    else if constexpr (STREAM) nz_stream_store(dst + (gq * NZ_LANES + lane) * NZ_GROUP, mv);
    else store8((gq * NZ_LANES + lane) * NZ_GROUP, mv);
  };
  const auto full_groups = [&](auto wide) __attribute__((always_inline)) {
    NzPacked<S, ROWS> sm_a = sm_next, sm_b = 0;
    std::conditional_t<decltype(wide)::value, NzNormByte, uint64_t> nb_a{}, nb_b{};
    if constexpr (NORM && decltype(wide)::value) nb_a = nb_next;
    else if constexpr (NORM) nb_a = whole ? nb_at(0, wide) : 0;
    uint32_t gq = 0;
    const auto fetch_a = [&] {
      sm_a = sm_at(gq + 2);
      if constexpr (NORM) nb_a = nb_at(gq + 2, wide);
    };
    const auto fetch_b = [&] {
      sm_b = sm_at(gq + 1);
      if constexpr (NORM) nb_b = nb_at(gq + 1, wide);
    };
    if constexpr (STAGED) {
      // Every wavefront by itself reads MR KiB per group, and beside a wavefront at another
      // column the vector L1 (32 KiB) holds too little of them: with all rows at one address
      // eight rows through the Linears of a block of width 4096 took 192 us, not 256.  Staged
      // (gate and up projection; the others keep the loads): six, seven and eight rows
      // 222, 239, 256 -> 219, 229, 242 us.  Up to five rows a third workgroup per compute unit
      // is worth more than that; launches of one workgroup lose 6 to 9 us to the barriers.
      if (NzXStage<MR>::fits(g, gv, cn)) {
        NzXStage<MR> xs;
        xs.start(xbuf, gv, wave, lane);
        xs.put(0, xs.fetch(0));
        for (; gq + 1 < whole; gq += 2) {
          const uint4 next_b = xs.fetch(walk.next_col());  // always inside x
          full_group(gq, sm_a, nb_a, wide, fetch_b, xs.buffer(0));
          xs.put(1, next_b);
          const uint4 next_a = xs.fetch(walk.next_col());
          full_group(gq + 1, sm_b, nb_b, wide, fetch_a, xs.buffer(1));
          xs.put(0, next_a);
        }
        if (gq < whole) full_group(gq, sm_a, nb_a, wide, [] {}, xs.buffer(0));
        return;
      }
    }
    for (; gq + 1 < whole; gq += 2) {
      full_group(gq, sm_a, nb_a, wide, fetch_b, NzNoLds{});
      full_group(gq + 1, sm_b, nb_b, wide, fetch_a, NzNoLds{});
    }
    if (gq < whole) full_group(gq, sm_a, nb_a, wide, [] {}, NzNoLds{});
  };
  if (!NORM || wide_norm) full_groups(NzConst<1>{});
  else {
    full_groups(NzConst<0>{});
    // What was fetched for groups that are not there has to come, too: the compiler lets this path run into the other
    // walk, and would have that wait in every turn for a register that such a load might still be under way to.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  }
  if ((!GEMV || !WHOLE) && whole < body) {  // the ragged last group of the tensor
    const uint32_t idx0 = (whole * NZ_LANES + lane) * NZ_GROUP;
    uint32_t ew[8];
    w.look();
    w.group(ew);
    if constexpr (GEMV) {  // (rows of eights: a lane has all of its 8 elements or none)
      const bool in = idx0 < seg_n;
      uint4 mv = nz_merge_group<S>(in ? nz_load_sm<S>(pk + idx0 / 8 * (S + 1)) : 0ull, ew);
      if constexpr (NORM) mv = nz_scale8<true>(mv, in ? nz_norm_load8(nm, seg_base + idx0) : 0ull, nm.log2n >= 3);
      walk.add(mv, walk.load(walk.col), lane);
    } else if (idx0 < seg_n) {
      const uint32_t rem = seg_n - idx0 < 8 ? seg_n - idx0 : 8;
      for (uint32_t j = 0; j < rem; ++j) {
        const uint32_t bit = (idx0 + j) * (S + 1);
        const uint32_t rp = ((uint32_t)pk[bit >> 3] >> (7u - S - (bit & 7u))) & ((2u << S) - 1u);
        uint32_t sym = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) sym = (uint32_t)q == j ? nz_unrot_exp(ew[q] >> 24) : sym;
        uint32_t h = nz_merge_one<S>(sym, rp);
        if constexpr (NORM) h = nz_norm_mul(h, nm.bytes[(seg_base + idx0 + j) >> nm.log2n]);
        store1(idx0 + j, h);
      }
    }
  }
  uint32_t ext[2][8];
#pragma unroll
  for (uint32_t t = 0; t < 2; ++t)
    if (t < tailg) {
      w.look();
      w.group(ext[t]);
    }

  // every lane must be back at the encoder's start state (2^16 | carried bits)
  // and the wave must not have read past its record
  w.finish();
  const bool bad = (carry ? (w.x >> 16) != 1u : w.x != NZ_L) || (w.base > w.nwords);
  if (__ballot(bad) != 0 && lane == 0) atomicOr(d_status, 4u);

  if (carry) {
    // the ring is dead now: park the 128 carried bytes at its start
    reinterpret_cast<uint16_t*>(w.ring32)[lane] = (uint16_t)(w.x & 0xFFFFu);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint8_t* tailp = reinterpret_cast<const uint8_t*>(w.ring32);
#pragma unroll
    for (uint32_t t = 0; t < 2; ++t) {
      if (t < tailg) {
        const uint32_t idx0 = ((body + t) * NZ_LANES + lane) * NZ_GROUP;
        const uint32_t b = idx0 / 8 * (S + 1);
        const uint64_t sm = b >= keep ? nz_load_sm<S>(tailp + (b - keep)) : nz_load_sm<S>(pk + b);
        uint4 mv = nz_merge_group<S>(sm, ext[t]);
        if constexpr (NORM) mv = nz_scale8<true>(mv, nz_norm_load8(nm, seg_base + idx0), nm.log2n >= 3);
        if constexpr (GEMV) walk.add(mv, walk.load(walk.col), lane);
        else store8(idx0, mv);
      }
    }
  }
  if constexpr (GEMV)
    if (walk.pending) walk.flush(lane);
}

// Workgroup b of a launch in which `parts` share a chunk: which chunk (of the launch), which of its segments.
struct NzPart {
  uint32_t chunk, first, end;
  __device__ __forceinline__ NzPart(uint32_t b, uint32_t parts, uint32_t spc) {
    const uint32_t l = 31u - (uint32_t)__builtin_clz(parts);  // (a power of two)
    chunk = b >> l;
    const uint32_t per = (spc + parts - 1) >> l;
    first = (b & (parts - 1)) * per;
    end = first + per;
  }
};

template <int S, bool NORM, bool STREAM, bool ONE>
__global__ __launch_bounds__(64 * NZ_MAX_SEGS_PER_CHUNK) void nz_decode_kernel(
    const uint8_t* __restrict__ comp, uint64_t comp_bytes, const uint8_t* __restrict__ packed,
    uint16_t* __restrict__ out, NzGeom g, uint32_t* __restrict__ d_status, const NzNorm nm, const uint32_t parts) {
  const NzPart p(blockIdx.x, ONE ? parts : 1u, g.spc);
  nz_decode_chunk<S, 0, NORM, STREAM, ONE>(comp, comp_bytes, packed, out, g, d_status, p.chunk, NzGemv{}, nm, p.first, p.end);
}

// Several tensors in one launch: the grid is the concatenation of their
// chunks, `chunk_end` the running total.  The items ride in the kernel
// argument block, so a launch needs no device-side table.
#define NZ_BATCH_MAX 16
struct NzBatchItem {
  const uint8_t* comp;
  uint64_t comp_bytes;
  const uint8_t* packed;
  uint16_t* out;       // dense output (decode) ...
  long long* acc;      // ... or the row accumulators, output and bias (matrix-vector product)
  uint16_t* y;
  const uint16_t* bias;
  const uint8_t* norm; // group bytes of a normalized tensor
  NzGeom g;
  uint32_t chunk_end;
  uint32_t acc_words;  // NzGemv
  // dense output of a tensor whose last write is not known to have fitted its buffer: the words in that
  // write's scratch (null: all is known), its nonce, and the container to take if they say it is not whole
  const NzLbWords* late;
  uint64_t late_nonce;
  const uint8_t* late_comp;
  uint64_t late_bytes;
};
struct NzBatch {
  uint32_t count;
  uint32_t in_features;  // matrix-vector product only
  const uint16_t* x;     // matrix-vector product only
  uint32_t log2n;        // normalized tensors only
  uint32_t x_rows;       // matrix-vector product only: activation rows (1..8)
  NzBatchItem item[NZ_BATCH_MAX];
  uint32_t parts;        // workgroups that share a chunk (nz_parts)
};

template <int S, bool NORM, bool STREAM, bool ONE>
__global__ __launch_bounds__(64 * NZ_MAX_SEGS_PER_CHUNK) void nz_decode_batch_kernel(
    const NzBatch b, uint32_t* __restrict__ d_status) {
  uint32_t t = 0, first = 0;
  const uint32_t parts = ONE ? b.parts : 1u, at = blockIdx.x >> (31u - (uint32_t)__builtin_clz(parts));
  while (t + 1 < b.count && at >= b.item[t].chunk_end) {
    first = b.item[t].chunk_end;
    ++t;
  }
  const NzBatchItem& it = b.item[t];
  const NzPart p(blockIdx.x, parts, it.g.spc);
  const bool other = it.late && nz_lb_not_whole(it.late, it.late_nonce);
  nz_decode_chunk<S, 0, NORM, STREAM, ONE>(other ? it.late_comp : it.comp, other ? it.late_bytes : it.comp_bytes,
                                          it.packed, it.out, it.g, d_status, at - first, NzGemv{},
                                          NzNorm{it.norm, b.log2n}, p.first, p.end);
}

// The same walk over several matrices that multiply MR activation rows (each
// decoded weight is used MR times before it is dropped).
template <int S, bool NORM, int MR, bool ONE, bool WHOLE>
__global__ __launch_bounds__(64 * NZ_MAX_SEGS_PER_CHUNK) void nz_decode_gemv_kernel(
    const NzBatch b, uint32_t* __restrict__ d_status) {
  uint32_t t = 0, first = 0;
  const uint32_t parts = ONE ? b.parts : 1u, at = blockIdx.x >> (31u - (uint32_t)__builtin_clz(parts));
  while (t + 1 < b.count && at >= b.item[t].chunk_end) {
    first = b.item[t].chunk_end;
    ++t;
  }
  const NzBatchItem& it = b.item[t];
  const NzPart p(blockIdx.x, parts, it.g.spc);
  const NzGemv gv{b.x, it.acc, it.y, it.bias, b.in_features, it.acc_words};
  nz_decode_chunk<S, MR, NORM, false, ONE, WHOLE>(it.comp, it.comp_bytes, it.packed, nullptr, it.g, d_status,
                                        at - first, gv, NzNorm{it.norm, b.log2n}, p.first, p.end);
}

// ----------------------------------------------------------------------------
// row gather (embedding lookup): decode only the segments that hold the rows asked
// for.  Workgroup (i, k) takes the k-th chunk touched by row indices[i] and stores
// what the row has of it; those of the first chunks come first, because few rows reach into
// another.  An index outside the table sets status bit 8 and yields a row of zeros.
//
// Bound by the chain of one segment's steps, whatever the number of rows up to four workgroups per
// compute unit (rows that lie in one segment take two rings, 40 KiB of LDS).  All segments
// of a chunk, stored in a slot and copied from there by a second kernel, took 26.8 us for one row of
// 128256 x 4096, 36.5 for 256, 51.6 for 512 and 107.6 for 1024; this takes 22.1, 23.5, 28.7 and 38.0.
// One-read steps for any number of rows (with an eighth of the wavefronts decoding, the chain is
// what counts), with the narrow ring where there are more workgroups than compute units.
// ----------------------------------------------------------------------------
template <int S, bool NORM, bool WIDE>
__global__ __launch_bounds__(64 * NZ_MAX_SEGS_PER_CHUNK) void nz_decode_rows_kernel(
    const uint8_t* __restrict__ comp, uint64_t comp_bytes, const uint8_t* __restrict__ packed,
    uint16_t* __restrict__ out, NzGeom g, uint32_t* __restrict__ d_status, const NzNorm nm,
    const long long* __restrict__ indices, uint32_t row_len, uint32_t cpr) {
  const uint32_t count = gridDim.x / cpr, k = blockIdx.x / count, i = blockIdx.x - k * count;
  const long long idx = indices[i];
  uint16_t* dst = out + (uint64_t)i * row_len;
  if (idx < 0 || (uint64_t)idx >= g.n / row_len) {
    if (k == 0) {
      for (uint32_t e = threadIdx.x; e < row_len; e += blockDim.x) dst[e] = 0;
      if (threadIdx.x == 0) atomicOr(d_status, 8u);
    }
    return;
  }
  const uint64_t first = (uint64_t)idx * row_len, last = first + row_len - 1;
  const uint64_t c = first / g.chunk_syms + k;
  if (c > last / g.chunk_syms) return;
  const NzRowOut row{dst, first, last, ((uintptr_t)dst & 15u) == 0 && first % NZ_GROUP == 0};
  nz_decode_chunk<S, 0, NORM, false, WIDE, true, true>(comp, comp_bytes, packed, nullptr, g, d_status, c, NzGemv{}, nm, 0, g.spc,
                                                          row);
}
