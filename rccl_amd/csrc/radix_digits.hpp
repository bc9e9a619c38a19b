// Key images, digits and the wave helpers that the radix sort's kernels share
// (onesweep passes, block sorts and rank merges).
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "radix_plan.hpp"

namespace rccl_hip {
namespace radix {

struct NoValue {};

enum class KeyClass { Unsigned, Signed, Float };

// Order-preserving bit image of a key, with the float +-0 collapse applied
// for digit extraction. Transforms: rccl-cub/src/ordering_backend/radix.rs:75-235
// (unsigned identity, signed sign flip, float: negative -> all bits inverted,
// otherwise sign flipped; descending = complement); collapse: :257-337 (the
// ordered value 0x7f..f is read as 0x80..0, so -0.0 and +0.0 share every
// digit). Stored keys are never rewritten.
template <class Bits, KeyClass KC, bool DESC>
struct KeyOps {
  using SBits = typename std::make_signed<Bits>::type;
  static constexpr int NBITS = int(sizeof(Bits) * 8);
  static constexpr Bits SIGN = Bits(1) << (NBITS - 1);

  // The order-preserving bijection, before the collapse. Onesweep passes keep
  // keys in this form between passes: the first converts its raw input
  // (image), the last its output back (raw), and every digit in between
  // needs only the collapse (image_digit): about half the ALU work per digit
  // for float keys.
  __device__ static __forceinline__ Bits image(Bits raw) {
    Bits x = raw;
    if constexpr (KC == KeyClass::Signed) x ^= SIGN;
    if constexpr (KC == KeyClass::Float)
      x ^= static_cast<Bits>(static_cast<SBits>(raw) >> (NBITS - 1)) | SIGN;
    if constexpr (DESC) x = ~x;
    return x;
  }
  __device__ static __forceinline__ Bits raw(Bits x) {
    if constexpr (DESC) x = ~x;
    if constexpr (KC == KeyClass::Signed) x ^= SIGN;
    // A set top bit marks a non-negative float (sign flipped), a clear one a
    // negative float (all bits inverted).
    if constexpr (KC == KeyClass::Float)
      x ^= static_cast<Bits>(~(static_cast<SBits>(x) >> (NBITS - 1))) | SIGN;
    return x;
  }
  __device__ static __forceinline__ Bits collapse(Bits x) {
    if constexpr (KC == KeyClass::Float) return x == SIGN - 1 ? SIGN : x;
    else return x;
  }

  __device__ static __forceinline__ Bits digit_source(Bits raw) { return collapse(image(raw)); }

  __device__ static __forceinline__ uint32_t digit(Bits raw, uint32_t bit, uint32_t mask) {
    return static_cast<uint32_t>(digit_source(raw) >> bit) & mask;
  }
  __device__ static __forceinline__ uint32_t image_digit(Bits y, uint32_t bit, uint32_t mask) {
    return static_cast<uint32_t>(collapse(y) >> bit) & mask;
  }
};

// How keys of one digit get their order within a wave (see onesweep_tile).
enum class Rank : int { LaneAtomic = 0, MatchAny = 1 };

// Opaque copy: the compiler must assume the value changed here, so it cannot
// carry values derived from it across this point. Aggregate keys (record
// rows) overload it in their own namespace, found by argument-dependent
// lookup.
template <class T>
__device__ __forceinline__ void launder(T &x) {
  asm volatile("" : "+v"(x));
}

// True when every lane of the (fully active) wave holds the same value.
__device__ __forceinline__ bool wave_uniform(uint32_t v) {
  return __ballot(v == __builtin_amdgcn_readfirstlane(v)) == ~uint64_t(0);
}

// Whether at least 8 lanes of the (fully active) wave share lane 0's value.
__device__ __forceinline__ bool hot_wave(uint32_t v) {
  return __builtin_popcountll(__ballot(v == __builtin_amdgcn_readfirstlane(v))) >= 8;
}

// Lanes of the fully active wave whose value of `d` equals this lane's, over
// the bits set in `bits` (one ballot per bit; the digits differ in no other
// bit).
__device__ __forceinline__ uint64_t peer_lanes(uint32_t d, uint32_t bits) {
  uint64_t m = ~uint64_t(0);
#pragma unroll
  for (int b = 0; b < 9; ++b) {
    if (bits & (1u << b)) {
      const bool set = ((d >> b) & 1u) != 0;
      const uint64_t bal = __ballot(set);
      m &= set ? bal : ~bal;
    }
  }
  return m;
}

// Lowest set lane of a non-zero mask.
__device__ __forceinline__ uint32_t lowest_lane(uint64_t m) {
  return static_cast<uint32_t>(__builtin_ctzll(m));
}

} // namespace radix
} // namespace rccl_hip
