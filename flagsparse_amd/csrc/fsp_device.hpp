// Device-side building blocks shared by every flagsparse_amd kernel (gfx950).
//
// Wave64 throughout: a workgroup is FSP_WG_THREADS threads = FSP_WAVES waves of
// 64 lanes.  Cross-lane sums use DPP inside a 16-lane row (quad_perm, row
// half-mirror, row mirror), ds_swizzle across the two rows of a 32-lane half
// and ds_bpermute across the two halves.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#define FSP_WG_THREADS 256
#define FSP_WAVES (FSP_WG_THREADS / 64)

namespace fsp {

// ---------------------------------------------------------------- value types
// Storage types and their accumulation types.  f16 / bf16 use clang's native
// _Float16 / __bf16 (hardware conversions on gfx950).
template <typename T> struct acc_of { using type = float; };
template <> struct acc_of<double> { using type = double; };

// SpMV of f32 accumulates in f64 (the reference promotes f32 SpMV to f64).
template <typename T> struct spmv_acc_of { using type = float; };
template <> struct spmv_acc_of<float> { using type = double; };
template <> struct spmv_acc_of<double> { using type = double; };

// One rounding per term: c + a * b as a fused multiply-add, written out so
// every loop variant accumulates identically whatever the contraction mode.
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename A, typename T> __device__ __forceinline__ A to_acc(T v) {
  return static_cast<A>(v);
}
template <typename T, typename A> __device__ __forceinline__ T from_acc(A v) {
  return static_cast<T>(v);
}

// ------------------------------------------------------------ vector loads
// VEC consecutive elements of T loaded / stored as one access of
// VEC*sizeof(T) bytes (<= 16), aligned to one element only: gfx950 runs with
// unaligned global access on, so the compiler emits the same dwordx4 for any
// element-aligned address and a row of any length or stride is read 16 bytes
// per lane.
template <typename T, int VEC> struct vec_t {
  T v[VEC];
};

// ---------------------------------------------------------- cross-lane moves
// DPP control codes (GCN/CDNA ISA): quad_perm selectors, row mirrors.
constexpr int DPP_QUAD_XOR1 = 0xB1;   // quad_perm [1,0,3,2]
constexpr int DPP_QUAD_XOR2 = 0x4E;   // quad_perm [2,3,0,1]
constexpr int DPP_ROW_HALF_MIRROR = 0x141;
constexpr int DPP_ROW_MIRROR = 0x140;

template <int CTRL> __device__ __forceinline__ int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, dpp_i32<CTRL>(__builtin_bit_cast(int, v)));
}
template <int CTRL> __device__ __forceinline__ double dpp(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = dpp_i32<CTRL>(static_cast<int>(static_cast<uint32_t>(u)));
  const int hi = dpp_i32<CTRL>(static_cast<int>(static_cast<uint32_t>(u >> 32)));
  return __builtin_bit_cast(
      double, (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                  static_cast<uint32_t>(lo));
}

// Lane exchange with lane ^ mask (mask < 32) through ds_swizzle bit mode:
// offset = xor_mask << 10 | or_mask << 5 | and_mask, and_mask = 0x1F.
__device__ __forceinline__ int swz_xor_i32(int v, int mask) {
  // ds_swizzle needs an immediate pattern; dispatch the handful of masks used.
  switch (mask) {
    case 1: return __builtin_amdgcn_ds_swizzle(v, (1 << 10) | 0x1F);
    case 2: return __builtin_amdgcn_ds_swizzle(v, (2 << 10) | 0x1F);
    case 4: return __builtin_amdgcn_ds_swizzle(v, (4 << 10) | 0x1F);
    case 8: return __builtin_amdgcn_ds_swizzle(v, (8 << 10) | 0x1F);
    default: return __builtin_amdgcn_ds_swizzle(v, (16 << 10) | 0x1F);
  }
}
// Lane exchange with lane ^ mask for any mask < 64 through ds_bpermute.
__device__ __forceinline__ int bperm_xor_i32(int v, int mask) {
  const int lane = __lane_id();
  return __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, v);
}

__device__ __forceinline__ int xor_i32(int v, int mask) {
  return mask < 32 ? swz_xor_i32(v, mask) : bperm_xor_i32(v, mask);
}
__device__ __forceinline__ float shfl_xor(float v, int mask) {
  return __builtin_bit_cast(float, xor_i32(__builtin_bit_cast(int, v), mask));
}
__device__ __forceinline__ double shfl_xor(double v, int mask) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = xor_i32(static_cast<int>(static_cast<uint32_t>(u)), mask);
  const int hi = xor_i32(static_cast<int>(static_cast<uint32_t>(u >> 32)), mask);
  return __builtin_bit_cast(
      double, (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                  static_cast<uint32_t>(lo));
}

// Sum over aligned groups of `lanes` consecutive lanes (power of two, 1..64);
// every lane of a group receives the group total, bitwise identical across
// the group (each step adds two partial sums that are exchanged pairwise).
// `lanes` is wave-uniform, so the guards are uniform branches.
template <typename A> __device__ __forceinline__ A group_sum(A v, int lanes) {
  if (lanes >= 2) v += dpp<DPP_QUAD_XOR1>(v);
  if (lanes >= 4) v += dpp<DPP_QUAD_XOR2>(v);
  if (lanes >= 8) v += dpp<DPP_ROW_HALF_MIRROR>(v);
  if (lanes >= 16) v += dpp<DPP_ROW_MIRROR>(v);
  if (lanes >= 32) v += shfl_xor(v, 16);
  if (lanes >= 64) v += shfl_xor(v, 32);
  return v;
}

// Broadcast inside a lane group: every lane receives the value of lane U of
// its quad (LANES 4) or of its row of 16 lanes (LANES 16).  One DPP move that
// the compiler folds into an integer add where it can.
template <int LANES, int U> __device__ __forceinline__ int bcast_i32(int v) {
  static_assert((LANES == 4 || LANES == 16) && U >= 0 && U < LANES, "a quad or a row of 16 lanes");
  constexpr int ctrl = LANES == 4 ? U * 0x55 : 0x150 + U;  // quad_perm [U,U,U,U] / row_newbcast:U
  return __builtin_amdgcn_mov_dpp(v, ctrl, 0xF, 0xF, true);
}
template <int LANES, int U, typename V> __device__ __forceinline__ V bcast(V v) {
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(V, bcast_i32<LANES, U>(__builtin_bit_cast(int, v)));
  } else {
    static_assert(sizeof(V) == 8, "32- or 64-bit values");
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = static_cast<uint32_t>(bcast_i32<LANES, U>(static_cast<int>(static_cast<uint32_t>(u))));
    const uint32_t hi = static_cast<uint32_t>(bcast_i32<LANES, U>(static_cast<int>(static_cast<uint32_t>(u >> 32))));
    return __builtin_bit_cast(V, (static_cast<uint64_t>(hi) << 32) | lo);
  }
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop
// whose index is a constant expression (DPP controls are immediates).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Byte-offset addressing: 32-bit offsets from a uniform base when OFF32.
template <bool OFF32> struct addr;
// (char-pointer arithmetic keeps the global address space visible to the
// compiler, so the loads stay global_load with a scalar base.)
template <> struct addr<true> {
  using off_t = uint32_t;
  template <typename P> static __device__ __forceinline__ P* at(P* base, off_t byte_off) {
    using C = typename std::conditional<std::is_const<P>::value, const char, char>::type;
    return reinterpret_cast<P*>(reinterpret_cast<C*>(base) + static_cast<uint64_t>(byte_off));
  }
};
template <> struct addr<false> {
  using off_t = uint64_t;
  template <typename P> static __device__ __forceinline__ P* at(P* base, off_t byte_off) {
    using C = typename std::conditional<std::is_const<P>::value, const char, char>::type;
    return reinterpret_cast<P*>(reinterpret_cast<C*>(base) + byte_off);
  }
};

template <bool OFF32, typename P>
__device__ __forceinline__ const P& elem(const P* base, typename addr<OFF32>::off_t i) {
  return *addr<OFF32>::at(base, i * static_cast<typename addr<OFF32>::off_t>(sizeof(P)));
}

// Third word of a raw buffer descriptor (32-bit elements, no swizzle).
constexpr int kRawBuffer = 0x00020000;

// ------------------------------------------------------------ index helpers
template <typename I> __device__ __forceinline__ int64_t ld_idx(const I* p, int64_t i) {
  return static_cast<int64_t>(p[i]);
}

}  // namespace fsp
