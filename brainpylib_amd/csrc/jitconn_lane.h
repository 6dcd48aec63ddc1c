// A std::mt19937 stream to a lane: 64 short streams walked by one wave, for the jitconn kernels.
//
// Word t of a generator, t < 227, is made of the seeded state alone: of x[t], x[t + 1] and x[t + 397], where x is the
// recurrence that seeds.  So a lane that holds x[t] and x[t + 397] and advances both draws these words with no state in
// memory: 397 steps to begin with instead of a seeded state's 624, which goes through memory (2,496 bytes out and back)
// and takes a wave's turn for a handful of synapses.  Words 227 to 453 need the new word 227 before them, which is made
// once more: two recurrences and a twist on top.
//
// Bound by the vector unit's issue: 1,600 instructions to begin with and, with homogeneous weights, 56 for every synapse
// of the longest of 64 streams (85 from word 227 on), where walk_stream() spends 59 on a batch of up to 64 and as many
// again on a stream's begin and end.  Row walks of 20,000 inputs, a wave to a stream / a lane: 400,000 rows of 3 / 44 / 130
// synapses 296 / 295 / 296 us, now 32 / 66 / 150; 20,000 of them 32 / 32 / 33, now 12 / 23 / (33: by wave); uniform weights
// 400,000 298 / 296 / 317, now 34 / 84 / (317); normal ones 300 / 317 / 413, now 43 / 162 / (413).  Normal weights take the
// logarithm, division and square root of an accepted attempt with every unit, for some lane has accepted one.
#pragma once

#include "jitconn_stream.h"

namespace bpl {

// the words a lane can draw, and those of them that need no new word
constexpr uint32_t kLaneWords = 2u * (kMtN - kMtM), kLaneFirst = kMtN - kMtM;

struct LaneGenerator {
  uint32_t near_, far_;      // x[t], x[t + 397]; from word 227 on x[t], x[t + 170]
  uint32_t start_, middle_;  // x[0], x[397]; from word 227 on x[t - 227]
  uint32_t t;                // wave uniform
  static __device__ __forceinline__ uint32_t step(uint32_t x, uint32_t i) { return 1812433253u * (x ^ (x >> 30)) + i; }
  __device__ __forceinline__ explicit LaneGenerator(uint32_t seed) : near_(seed), far_(seed), start_(seed), t(0) {
#pragma unroll 4
    for (uint32_t i = 1; i < kMtM; ++i) far_ = step(far_, i);
    far_ = step(far_, kMtM);
    middle_ = far_;
  }
  // the next word, not yet tempered; kAny: it may be one from word 227 on
  template <bool kAny>
  __device__ __forceinline__ uint32_t raw() {
    const uint32_t next = step(near_, t + 1u);
    uint32_t w;
    if (!kAny || t < kLaneFirst) {
      w = mt_twist(near_, next, far_);
      far_ = step(far_, t + kMtM + 1u);
    } else {
      // (made of the new word t - 227, which is made once more)
      if (t == kLaneFirst) far_ = middle_;
      const uint32_t behind = step(start_, t - kLaneFirst + 1u);
      w = mt_twist(near_, next, mt_twist(start_, behind, far_));
      start_ = behind;
      far_ = step(far_, t - kLaneFirst + kMtM + 1u);
    }
    near_ = next;
    ++t;
    return w;
  }
  template <bool kAny>
  __device__ __forceinline__ uint32_t word() { return mt_temper(raw<kAny>()); }
};

// Walks stream std::mt19937{stream_seed} of each lane over [0, n): calls f(index, weight, valid) with the whole wave converged,
// one synapse of every lane that has one (`valid`; the others get index 0) per call, in the order of each stream.  Returns the lanes
// whose stream needs more than kLaneWords words: they gave what lies in front of their position `pos`.
// The skips fit: sp.narrow and n <= 0xf0000000, so that a position never leads around 2^32.
template <typename T1, int W, typename F>
__device__ __forceinline__ uint64_t walk_lane_streams(uint32_t stream_seed, bool alive, uint32_t n, const SkipParams &sp,
                                                      T1 wa, T1 wb, uint32_t &pos, F &&f) {
  LaneGenerator gen(stream_seed);
  {
    const uint32_t lo = gen.raw<false>(), hi = gen.word<false>();
    pos = skip_from_words<true, false>(lo, hi, sp, __builtin_amdgcn_ballot_w64(alive));
  }
  alive = alive && pos < n;
  uint64_t left = __builtin_amdgcn_ballot_w64(alive);
  uint32_t state = 0;  // (normal weights)
  T1 x = T1(0), first = T1(0), second = T1(0);
  auto walk = [&](auto any, uint32_t most) {
    constexpr bool kAny = decltype(any)::value;
    if constexpr (W != kNormal) {
      // homogeneous  K K K ..., uniform  K (w K) (w K) ...: a synapse at the position behind each K
      constexpr uint32_t WW = W == kUniform ? WeightWords<T1>::value : 0;
      while (left != 0 && gen.t + WW + 2u <= most) {
        T1 weight = T1(1);
        if constexpr (W == kUniform) {
          uint32_t w[WW];
  #pragma unroll
          for (uint32_t i = 0; i < WW; ++i) w[i] = gen.template word<kAny>();
          weight = uniform_weight(w, wa, wb);
        }
        f(alive ? pos : 0u, weight, alive);
        const uint32_t lo = gen.template raw<kAny>(), hi = gen.template word<kAny>();
        pos += skip_from_words<true, false>(lo, hi, sp, left);
        alive = alive && pos < n;
        left = __builtin_amdgcn_ballot_w64(alive);
      }
    } else {
      // K (A..A K) (K) ... with attempts A (walk_stream()); state: 0 attempt, 1 first and 2 second skip behind an accepted
      // one.  Double: the units are one canonical double each, the attempts X Y; state 3: Y expected.
      constexpr bool kWide = sizeof(T1) == 8;
      while (left != 0 && gen.t + 2u <= most) {
        const uint32_t lo = gen.template word<kAny>(), hi = gen.template word<kAny>();
        float upper;
        bool accepted;
        T1 y;
        const bool skips = state == 1u || state == 2u;
        if constexpr (!kWide) {
          const PolarF32 a = polar_attempt(lo, hi);
          upper = a.u1;
          accepted = a.ok && state == 0u;
          if (!skips) x = a.x;
          y = a.y;
        } else {
          upper = static_cast<float>(hi);
          y = __dsub_rn(__dmul_rn(2.0, canonical_f64(lo, hi)), 1.0);
          const double r2 = __dadd_rn(__dmul_rn(x, x), __dmul_rn(y, y));
          accepted = state == 3u && !(r2 > 1.0 || r2 == 0.0);
          if (state == 0u) x = y;
        }
        f(alive && skips ? pos : 0u, state == 1u ? first : second, alive && skips);
        const uint32_t skip = skip_from_words<true, true>(lo, hi, upper, sp, __builtin_amdgcn_ballot_w64(alive && skips));
        if (skips) pos += skip;
        if (accepted) polar_weights(x, y, wa, wb, first, second);
        if constexpr (!kWide) state = accepted ? 1u : state == 1u ? 2u : 0u;
        else state = accepted ? 1u : state == 1u ? 2u : state == 0u ? 3u : 0u;
        alive = alive && pos < n;
        left = __builtin_amdgcn_ballot_w64(alive);
      }
    }
  };
  walk(std::false_type(), kLaneFirst);
  walk(std::true_type(), kLaneWords);
  return left;
}

}  // namespace bpl
