// Block radix sort and rank merge for gfx950: the short sorts.
//
// An onesweep sort is a chain of dependent launches (init, histogram, scan,
// one pass per key byte); below a few hundred thousand items each of them
// costs its launch (about 4 us) whatever it moves. Short inputs take one or
// two launches instead:
//   block_sort  one block per tile sorts its tile by every 8-bit digit of the
//               bit window, keys in registers, exchanged through LDS
//   rank_merge  the sorted tiles become one sorted range: an item's final
//               position is its position in its own tile plus, for every
//               other tile, the number of that tile's items before it
//               (binary searches, the top levels over samples in LDS)
// Both are stable, so together they give the LSD sort's permutation.
// Reference behaviour: the single-tile route (rccl-cub/src/radix.rs:470-492,
// ordering_backend/radix.rs:366-715) and the pass control of radix.rs:364-876,
// whose results (and selector flips) these sorts keep.
#pragma once

#include "radix_digits.hpp"

namespace rccl_hip {
namespace radix {

// What moves with a key through LDS: values of up to 4 bytes themselves,
// wider ones as the 16-bit index of their item (gathered once at the end).
template <class Val>
struct BlockPayload {
  static constexpr bool PAIRS = !std::is_same<Val, NoValue>::value;
  static constexpr bool INDEXED = PAIRS && sizeof(Val) > 4;
  using type = typename std::conditional<
      INDEXED, uint16_t, typename std::conditional<PAIRS, Val, char>::type>::type;
};

// The bits of a digit source that a sort of [begin_bit, end_bit) orders by.
template <class Bits>
__device__ __forceinline__ Bits window_key(Bits source, uint32_t begin_bit, uint32_t end_bit) {
  constexpr uint32_t NBITS = sizeof(Bits) * 8;
  return static_cast<Bits>(source << (NBITS - end_bit)) >> (NBITS - end_bit + begin_bit);
}

// OR of a value over the lanes of a fully active wave, in every lane.
template <class Bits>
__device__ __forceinline__ Bits wave_or(Bits x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) x |= __shfl_xor(x, o, 64);
  return x;
}

// `width` (at most 8) bits of x from bit `bit` on, bit and width uniform. The
// 64-bit form works on the two words: a 64-bit shift costs four instructions.
__device__ __forceinline__ uint32_t bits_at(uint32_t x, uint32_t bit, uint32_t width) {
  return __builtin_amdgcn_ubfe(x, bit, width);
}
__device__ __forceinline__ uint32_t bits_at(uint64_t x, uint32_t bit, uint32_t width) {
  const uint32_t lo = static_cast<uint32_t>(x), hi = static_cast<uint32_t>(x >> 32);
  const uint32_t a = bit < 32 ? lo : hi, b = bit < 32 ? hi : 0u;
  return __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(b, a, bit & 31u), 0, width);
}

// One block per tile of `tile` items (a multiple of 64, at most BLOCK_THREADS
// x ITEMS): tile b is [b * tile, b * tile + len). Every input of a tile is read
// before any of its outputs is written, and blocks share no item, so the
// output may be the input. With `samples`, the digit source of every chunk of
// SAMPLE sorted items' last one goes to samples[item / SAMPLE] for the rank
// merge (the largest key where the last tile has no such item).
//
// What bounds it: one CU's LDS and vector issue. The block is as wide as the
// CU allows (16 waves) and a key's pass is one returning LDS atomic (its rank
// within its wave and digit), one read of its wave's digit start, and one
// write and one read of the exchange. Slots past the tile's end hold the
// largest key, which stays behind every item of the tile, so no item is
// tested. Digits that do not vary in the tile take no pass.
template <class Bits, class Val, class Ops, int ITEMS, Rank RANK>
__global__ void __launch_bounds__(BLOCK_THREADS)
block_sort_kernel(const Bits *keys_in, Bits *keys_out, const Val *vals_in, Val *vals_out,
                  uint32_t n, uint32_t tile, uint32_t begin_bit, uint32_t end_bit,
                  Bits *__restrict__ samples) {
  using Payload = BlockPayload<Val>;
  using Pay = typename Payload::type;
  constexpr bool PAIRS = Payload::PAIRS;
  constexpr int WAVES = BLOCK_THREADS / 64;
  constexpr int TILE = BLOCK_THREADS * ITEMS;
  constexpr int QUARTERS = BLOCK_THREADS / BINS;    // threads per digit
  constexpr int QWAVES = WAVES / QUARTERS;          // waves counted by each of them
  // Row stride: QWAVES rows apart is 16 banks apart, so the QUARTERS threads
  // of a digit read different banks.
  constexpr int ROW = BINS + 4;
  static_assert(QUARTERS * BINS == BLOCK_THREADS && QUARTERS * QWAVES == WAVES, "digit threads");
  static_assert(WAVES <= 64, "one lane per wave total");
  static_assert(TILE <= 65536, "item indices are 16-bit");
  __shared__ Bits s_keys[TILE];
  __shared__ Pay s_pay[PAIRS ? TILE : 1];
  __shared__ uint32_t cnt[WAVES][ROW];  // digit counts, then starts, of each wave
  __shared__ uint32_t wave_sum[WAVES];
  __shared__ Bits s_first;
  __shared__ uint32_t s_vary[2];  // bits that differ between items of the tile

  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t base = blockIdx.x * tile;
  const uint32_t len = min(tile, n - base);
  // Wave-contiguous, lane-striped: item j of a lane is first + 64 j, so (wave,
  // item, lane) order is source order. `rows` items per lane hold the tile.
  const uint32_t rows = (len + BLOCK_THREADS - 1) / BLOCK_THREADS;
  const uint32_t first = wave * rows * 64u + lane;
  Bits key[ITEMS];
  Pay pay[PAIRS ? ITEMS : 1];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (uint32_t(j) >= rows) continue;
    const uint32_t i = min(first + uint32_t(j) * 64u, len - 1u);
    key[j] = keys_in[base + i];
    if constexpr (Payload::INDEXED) pay[j] = static_cast<Pay>(i);
    else if constexpr (PAIRS) pay[j] = vals_in[base + i];
  }
  if (tid < 2) s_vary[tid] = 0;
  // The bits that vary, against the tile's first item (a slot past the end
  // repeats the last item here).
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (uint32_t(j) >= rows) continue;
    key[j] = Ops::image(key[j]);
  }
  if (tid == 0) s_first = Ops::collapse(key[0]);
  lds_barrier();
  Bits vary = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (uint32_t(j) >= rows) continue;
    vary |= Ops::collapse(key[j]) ^ s_first;
    if (first + uint32_t(j) * 64u >= len) key[j] = ~Bits(0);
  }
  vary = wave_or(vary);
  if (lane == 0) {
    atomicOr(&s_vary[0], static_cast<uint32_t>(vary));
    if constexpr (sizeof(Bits) == 8) atomicOr(&s_vary[1], static_cast<uint32_t>(vary >> 32));
  }
  lds_barrier();
  // (readfirstlane returns an int: not to be sign-extended.)
  vary = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(s_vary[0]));
  if constexpr (sizeof(Bits) == 8)
    vary |= static_cast<Bits>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(s_vary[1])))
            << 32;

  uint32_t *wcnt = cnt[wave];
  for (uint32_t bit = begin_bit; bit < end_bit; bit += 8) {
    const uint32_t width = min(8u, end_bit - bit);
    const uint32_t mask = (1u << width) - 1u;
    if ((static_cast<uint32_t>(vary >> bit) & mask) == 0) continue;
    // A wave clears and counts in its own row only: no barrier between.
#pragma unroll
    for (int k = 0; k < BINS / 64; ++k) wcnt[uint32_t(k) * 64u + lane] = 0;
    uint32_t dig[ITEMS], rank[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (uint32_t(j) >= rows) continue;
      dig[j] = bits_at(Ops::collapse(key[j]), bit, width);
    }
    if constexpr (RANK == Rank::MatchAny) {
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        if (uint32_t(j) >= rows) continue;
        const uint64_t m = peer_lanes(dig[j], mask);
        const uint32_t below = popc_below(m);
        const uint32_t got =
            below == 0
                ? __hip_atomic_fetch_add(&wcnt[dig[j]],
                                         static_cast<uint32_t>(__builtin_popcountll(m)),
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)
                : 0u;
        rank[j] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(
                      static_cast<int>(lowest_lane(m) << 2), static_cast<int>(got))) +
                  below;
      }
    } else if (hot_wave(dig[0]) || (rows > ITEMS / 2 && hot_wave(dig[ITEMS / 2]))) {
      // Lanes on one counter are served one after another. Where many share
      // a digit, those with lane 0's take one atomic together.
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        if (uint32_t(j) >= rows) continue;
        const uint64_t m = __ballot(dig[j] == __builtin_amdgcn_readfirstlane(dig[j]));
        const bool in = ((m >> lane) & 1u) != 0;
        const uint32_t below = popc_below(m);
        uint32_t got = 0;
        if (!in || lane == 0)
          got = __hip_atomic_fetch_add(
              &wcnt[dig[j]], in ? static_cast<uint32_t>(__builtin_popcountll(m)) : 1u,
              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t group = __builtin_amdgcn_readfirstlane(got);
        rank[j] = in ? group + below : got;
      }
    } else {
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        if (uint32_t(j) >= rows) continue;
        rank[j] = __hip_atomic_fetch_add(&wcnt[dig[j]], 1u, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    lds_barrier();
    // Thread t holds waves [q * QWAVES, (q + 1) * QWAVES) of digit t /
    // QUARTERS, q = t % QUARTERS: thread order is (digit, wave) order, the
    // order of the pass's output.
    const uint32_t d = tid / QUARTERS, q0 = tid % QUARTERS * QWAVES;
    uint32_t c[QWAVES], sum = 0;
#pragma unroll
    for (int w = 0; w < QWAVES; ++w) {
      c[w] = cnt[q0 + w][d];
      sum += c[w];
    }
    const uint32_t inc = wave_inclusive_sum(sum, lane);
    if (lane == 63) wave_sum[wave] = inc;
    lds_barrier();
    // Exclusive start of this wave's digits: the earlier waves' totals.
    const uint32_t before = wave_inclusive_sum(lane < wave ? wave_sum[lane % WAVES] : 0u, lane);
    uint32_t run = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(before), 63)) +
                   inc - sum;
#pragma unroll
    for (int w = 0; w < QWAVES; ++w) {
      cnt[q0 + w][d] = run;
      run += c[w];
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (uint32_t(j) >= rows) continue;
      // Below rows * BLOCK_THREADS <= TILE: the counters counted these slots.
      const uint32_t pos = wcnt[dig[j]] + rank[j];
      s_keys[pos] = key[j];
      if constexpr (PAIRS) s_pay[pos] = pay[j];
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (uint32_t(j) >= rows) continue;
      const uint32_t i = first + uint32_t(j) * 64u;
      key[j] = s_keys[i];
      if constexpr (PAIRS) pay[j] = s_pay[i];
    }
    // The next pass scatters into LDS only after three more barriers, which
    // every read above has passed; its counters are its own wave's.
  }
  if constexpr (Payload::INDEXED) {
    Val v[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (uint32_t(j) >= rows) continue;
      v[j] = vals_in[base + min(uint32_t(pay[j]), len - 1u)];
    }
    __syncthreads();  // every value is read before any is written (in place)
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (uint32_t(j) >= rows) continue;
      const uint32_t i = first + uint32_t(j) * 64u;
      if (i < len) vals_out[base + i] = v[j];
    }
  }
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (uint32_t(j) >= rows) continue;
    const uint32_t i = first + uint32_t(j) * 64u;
    if (i < len) {
      keys_out[base + i] = Ops::raw(key[j]);
      if constexpr (PAIRS && !Payload::INDEXED) vals_out[base + i] = pay[j];
    }
    // i >= len holds the largest key, which window_key keeps largest.
    if (samples && i % SAMPLE == SAMPLE - 1u && i - (SAMPLE - 1u) < len)
      samples[(base + i) / SAMPLE] = window_key<Bits>(Ops::collapse(key[j]), begin_bit, end_bit);
  }
}

// Merges `tiles` sorted tiles of TILE items (the last may be short), one
// item per thread.
//
// What bounds it: issue and latency of the searches, one per item and tile.
// Two thirds of a search's levels run over the samples in LDS (3 vector
// instructions each), the others in the SAMPLE - 1 items before the chunk's
// last, in one or two lines that the wave's neighbouring items share; RM_WAYS
// searches overlap. The work grows with the number of tiles.
template <class Bits, class Val, class Ops, uint32_t TILE>
__global__ void __launch_bounds__(RM_THREADS)
rank_merge_kernel(const Bits *__restrict__ keys_in, Bits *__restrict__ keys_out,
                  const Val *__restrict__ vals_in, Val *__restrict__ vals_out, uint32_t n,
                  uint32_t tiles, uint32_t begin_bit, uint32_t end_bit,
                  const Bits *__restrict__ samples) {
  constexpr bool PAIRS = !std::is_same<Val, NoValue>::value;
  constexpr uint32_t CHUNKS = TILE / SAMPLE;  // per tile
  static_assert((CHUNKS & (CHUNKS - 1)) == 0 && (SAMPLE & (SAMPLE - 1)) == 0, "binary searches");
  static_assert(TILE % RM_THREADS == 0, "a block's items are one tile's");
  extern __shared__ __attribute__((aligned(16))) unsigned char rm_smem[];
  Bits *s_samples = reinterpret_cast<Bits *>(rm_smem);  // tiles rounded up to RM_WAYS
  const uint32_t tid = threadIdx.x;
  const uint32_t g = blockIdx.x * RM_THREADS + tid;
  const uint32_t at = min(g, n - 1u);
  const Bits raw = keys_in[at];
  typename std::conditional<PAIRS, Val, char>::type val{};
  if constexpr (PAIRS) val = vals_in[at];
  const uint32_t sample_count = (n + SAMPLE - 1) / SAMPLE;
  const uint32_t slots = (tiles + RM_WAYS - 1) / RM_WAYS * RM_WAYS * CHUNKS;
  for (uint32_t i = tid; i < slots; i += RM_THREADS)
    s_samples[i] = i < sample_count ? samples[i] : ~Bits(0);
  auto source = [&](Bits r) { return window_key<Bits>(Ops::digit_source(r), begin_bit, end_bit); };
  const Bits x = source(raw);
  const uint32_t mine = blockIdx.x / (TILE / RM_THREADS);  // the whole block's tile
  uint32_t pos = at - mine * TILE;
  __syncthreads();
  for (uint32_t t0 = 0; t0 < tiles; t0 += RM_WAYS) {
    // Items of tile t before x: smaller ones, and equal ones of earlier tiles.
    // Only the last tile can be short, and no tile is later than it: a slot
    // past its end (the largest key) is never before x.
    auto before = [&](int w, Bits y) { return t0 + w < mine ? !(x < y) : y < x; };
    uint32_t c[RM_WAYS];  // first the chunks whose last item is before x
#pragma unroll
    for (int w = 0; w < RM_WAYS; ++w) c[w] = 0;
#pragma unroll
    for (uint32_t step = CHUNKS / 2; step; step >>= 1) {
#pragma unroll
      for (int w = 0; w < RM_WAYS; ++w)
        if (before(w, s_samples[(t0 + w) * CHUNKS + c[w] + step - 1u])) c[w] += step;
    }
#pragma unroll
    for (int w = 0; w < RM_WAYS; ++w)
      if (before(w, s_samples[(t0 + w) * CHUNKS + c[w]])) ++c[w];
    // Then the items of the chunk after them. A tile past the end and the
    // item's own count none.
#pragma unroll
    for (int w = 0; w < RM_WAYS; ++w) c[w] *= SAMPLE;
#pragma unroll
    for (uint32_t step = SAMPLE / 2; step; step >>= 1) {
#pragma unroll
      for (int w = 0; w < RM_WAYS; ++w) {
        const uint32_t k = (t0 + w) * TILE + c[w] + step - 1u;
        if (before(w, source(keys_in[min(k, n - 1u)]))) c[w] += step;
      }
    }
#pragma unroll
    for (int w = 0; w < RM_WAYS; ++w) {
      const uint32_t t = t0 + w;
      const uint32_t count = t < tiles && t != mine ? min(TILE, n - t * TILE) : 0u;
      pos += min(c[w], count);
    }
  }
  if (g >= n) return;
  pos = min(pos, n - 1u);
  keys_out[pos] = raw;
  if constexpr (PAIRS) vals_out[pos] = val;
}

} // namespace radix
} // namespace rccl_hip
