// Generator-stream walker shared by the jitconn kernels: one wave64 walks one std::mt19937
// stream (mt_wave.h) and hands the synapses it finds, 64 lanes at a time, to a callback.
#pragma once

#include <cmath>
#include <type_traits>

#include "common.h"
#include "mt_wave.h"

namespace bpl {

enum : int { kHomo = 0, kUniform = 1, kNormal = 2 };
enum : int { kInEvent = 0, kInDense = 1 };

// weight draws ----------------------------------------------------------------------------------
// std::uniform_real_distribution<T>{a,b} computes canonical * (b - a) + a; the descriptor carries
// a and the range b - a (as the reference's GPU descriptors do, lib/gpu_jitconn_event_matvec.cu:
// 221-222), so the range is formed by the caller.  No contraction.
__device__ __forceinline__ float uniform_weight(const uint32_t *w, float a, float range) {
  return __fadd_rn(__fmul_rn(canonical_f32(w[0]), range), a);
}
__device__ __forceinline__ double uniform_weight(const uint32_t *w, double a, double range) {
  return __dadd_rn(__dmul_rn(canonical_f64(w[0], w[1]), range), a);
}

template <typename T1>
struct WeightWords {
  static constexpr int value = sizeof(T1) == 4 ? 1 : 2;  // mt19937 words per uniform weight
};

// Normal weights: a wave queues the accepted polar attempts and the positions of their synapses in LDS and
// works the attempts off `drain` at a time, a lane each (the logarithm, division and square root of a weight
// are two thirds of the instructions of a unit, and three units of ten are accepted attempts: evaluated in
// place they ran for all 64 lanes of every batch: matvec and its gradient over 1.5e8 synapses 2.35 -> 1.87
// ms; matmat of 128 rows with 1e7 synapses 234 -> 214 us).  A batch of 64 units accepts at most 22 attempts (an
// attempt and its two skips are three units; of double coordinates four, 17), and the positions lag behind the
// attempts by two at most.  `drain` in double is what leaves 16 waves their 64 KB of static LDS.
template <typename T1>
struct NormalQueue {
  static constexpr uint32_t drain = sizeof(T1) == 4 ? 64 : 40;           // attempts worked off together
  static constexpr uint32_t attempts = drain + (sizeof(T1) == 4 ? 24 : 18);  // slots
  static constexpr uint32_t spill = 2 * (attempts - drain);             // positions that may outlast a drain
  static constexpr int words = static_cast<int>(attempts * (2 * sizeof(T1) / 4 + 2));
  static_assert(spill <= kWave && 2 * drain <= 2 * kWave, "one lane per attempt and per position moved");
};

// Words a lane takes from the generator per batch, and how many lanes take some.
template <typename T1, int W>
struct StreamBatch {
  static constexpr int K = W == kUniform ? WeightWords<T1>::value + 2 : 2;
  static constexpr int NL = K <= 3 ? kWave : 56;  // K * NL <= 227
};

// LDS words one wave needs: the generator state and, for normal weights, the queue behind it.  kShort: the state with the
// least mirror (mt_wave.h).
template <typename T1, int W, bool kShort = false>
struct StreamLds {
  static constexpr int mirror = kShort ? kMtLeastMirror : StreamBatch<T1, W>::K * StreamBatch<T1, W>::NL;
  static constexpr int state_words = kMtN + mirror;
  static constexpr int words = state_words + (W == kNormal ? NormalQueue<T1>::words : 0);
  static_assert(words % 2 == 0, "the queue of the next wave stays aligned");
};

__device__ __forceinline__ double read_lane_f64(double v, int l) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v));
  const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(b), l));
  const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(b >> 32), l));
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// Lane l receives lane l - 1's value, across the whole wave, in one data-parallel move (lane 0
// keeps its own); the general shuffle goes through the LDS crossbar and a dozen index instructions.
__device__ __forceinline__ uint32_t wave_shift_up1(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), 0x138 /* wave_shr:1 */,
                                                           0xf, 0xf, false));
}
__device__ __forceinline__ double wave_shift_up1(double v) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v));
  const uint32_t lo = wave_shift_up1(static_cast<uint32_t>(b)), hi = wave_shift_up1(static_cast<uint32_t>(b >> 32));
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// std::normal_distribution<float> (libstdc++, Marsaglia polar): candidate pair from two words
struct PolarF32 {
  float x, y, r2, u1;  // u1: the second word (capped) as a float
  bool ok;
};
__device__ __forceinline__ PolarF32 polar_attempt(uint32_t w0, uint32_t w1) {
  PolarF32 a;
  // 2 * canonical - 1: the scalings by powers of two are exact, so one fused multiply-add rounds where
  // the subtraction of the CPU code rounds
  a.u1 = canonical_f32_scaled(w1);
  a.x = fmaf(canonical_f32_scaled(w0), 0x1p-31f, -1.0f);
  a.y = fmaf(a.u1, 0x1p-31f, -1.0f);
  a.r2 = __fadd_rn(__fmul_rn(a.x, a.x), __fmul_rn(a.y, a.y));
  a.ok = !(a.r2 > 1.0f || a.r2 == 0.0f);
  return a;
}

// Roles of the 64 two-word units of one batch of a normal-weight stream: which are polar attempts and which
// are skips follows from a small automaton over the units' "this attempt would be accepted" bits.  A unit is a
// map of the automaton's four states, one byte per state, and one byte permutation composes two maps, so a
// prefix scan over the lanes gives every lane the state behind its unit.  (On the scalar unit, eight units at
// a time through a table, the automaton took 64 scalar instructions a batch; a CU issues one of those a cycle
// for its 32 waves, as many as vector instructions: matvec and its gradient over 1.5e8 synapses 2.58 ms, with
// the scan 1.87.)
// float: 0 attempt expected (the last one was rejected), 1 first skip expected, 2 second skip expected, 3 attempt expected
// (the second skip was the last unit).
// double (a unit is one coordinate): 0 X expected, 1 Y expected, 2 first skip, 3 second skip expected.
constexpr uint32_t state_map(uint32_t from0, uint32_t from1, uint32_t from2, uint32_t from3) {
  return from0 | from1 << 8 | from2 << 16 | from3 << 24;
}
template <bool kWide>
struct UnitMaps {
  static constexpr uint32_t accepts = kWide ? state_map(1, 2, 3, 0) : state_map(1, 2, 3, 1);
  static constexpr uint32_t rejects = kWide ? state_map(1, 0, 3, 0) : state_map(0, 2, 3, 0);
};
template <int kDpp, int kRows>
__device__ __forceinline__ uint32_t compose_behind(uint32_t map, uint32_t &before) {
  before = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(before), static_cast<int>(map), kDpp, kRows, 0xf, false));
  return __builtin_amdgcn_perm(map, map, before);
}
// What a lane composes its map with in each step.  A step's move leaves the lanes without a lane so far below as they
// were: they hold the identity for the whole walk (else a register is set to it in front of each of the six moves).
struct ScanBefore {
  uint32_t at[6] = {state_map(0, 1, 2, 3), state_map(0, 1, 2, 3), state_map(0, 1, 2, 3),
                    state_map(0, 1, 2, 3), state_map(0, 1, 2, 3), state_map(0, 1, 2, 3)};
  // (each in a register of its own from the start)
  __device__ __forceinline__ ScanBefore() {
#pragma unroll
    for (int i = 0; i < 6; ++i) asm volatile("" : "+v"(at[i]));
  }
};
// the state behind this lane's unit; `entered` is the state in front of lane 0's and becomes the one behind lane 63's
template <bool kWide>
__device__ __forceinline__ uint32_t state_behind(bool ok, uint32_t &entered, ScanBefore &before) {
  uint32_t map = ok ? UnitMaps<kWide>::accepts : UnitMaps<kWide>::rejects;
  map = compose_behind<0x111, 0xf>(map, before.at[0]);  // row_shr:1, 2, 4, 8, then the rows' totals (wave_inclusive_scan_u32)
  map = compose_behind<0x112, 0xf>(map, before.at[1]);
  map = compose_behind<0x114, 0xf>(map, before.at[2]);
  map = compose_behind<0x118, 0xf>(map, before.at[3]);
  map = compose_behind<0x142, 0xa>(map, before.at[4]);
  map = compose_behind<0x143, 0xc>(map, before.at[5]);
  const uint32_t state = __builtin_amdgcn_ubfe(map, 8u * entered, 8u);
  entered = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(state), kWave - 1));
  return state;
}

// The two weights of an accepted attempt (libstdc++: y * mult first, then the saved x * mult)
__device__ __forceinline__ void polar_weights(float x, float y, float mean, float sigma, float &w_first, float &w_second) {
  const float r2 = __fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y));
  const float mult = __fsqrt_rn(__fdiv_rn(__fmul_rn(-2.0f, logf(r2)), r2));
  w_first = __fadd_rn(__fmul_rn(__fmul_rn(y, mult), sigma), mean);
  w_second = __fadd_rn(__fmul_rn(__fmul_rn(x, mult), sigma), mean);
}
__device__ __forceinline__ void polar_weights(double x, double y, double mean, double sigma, double &w_first, double &w_second) {
  const double r2 = __dadd_rn(__dmul_rn(x, x), __dmul_rn(y, y));
  const double mult = sqrt(-2 * log(r2) / r2);
  w_first = __dadd_rn(__dmul_rn(__dmul_rn(y, mult), sigma), mean);
  w_second = __dadd_rn(__dmul_rn(__dmul_rn(x, mult), sigma), mean);
}

// number of lanes below this one in `mask`, plus `base`
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask, uint32_t base) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), base));
}

// Walks stream std::mt19937{stream_seed} over [0, n): calls f(index, weight, valid, partial) once per
// batch with the whole wave converged; `valid` marks the lanes that hold a synapse of the row: the first
// lanes of the wave, their indices rising from lane to lane; all of them unless `partial` (wave uniform); the others
// get index 0.  Normal weights come two at a time: synapses
// 2 l and 2 l + 1 of a group are lane l's.  f is called for the first and then for the second ones, or, if
// it can be called so, f(index, weight, valid, index, weight, valid) for both.
//
// `pre` points at the stream's 624 seeded state words when they were prepared by
// launch_seed_streams(); with nullptr the wave seeds the generator itself on the scalar unit.
//
// kQuick: skips are first tried on the upper words alone (skip_quick).
//
// `loaded()` is called once, when the generator state is in LDS and `pre` is no longer read.
//
// `start`: what the indices are counted from (the walk ends at `n`, counted alike).  The ends are found in positions without
// it: a skip may lead to a position just under 2^32, which is beyond every row, and `start` more would lead around.
struct NoLoadHook {
  __device__ __forceinline__ void operator()() const {}
};
template <typename T1, int W, bool kQuick = false, bool kShort = false, typename F, typename L = NoLoadHook>
__device__ __forceinline__ void walk_stream(uint32_t *st, int lane, uint32_t stream_seed, const uint32_t *pre,
                                            uint32_t n, const SkipParams &sp, T1 wa, T1 wb, F &&f, L &&loaded = L(),
                                            uint32_t start = 0u) {
  constexpr int K = StreamBatch<T1, W>::K, NL = StreamBatch<T1, W>::NL, kMirror = StreamLds<T1, W, kShort>::mirror;
  if (pre != nullptr) mt_load<kMirror>(st, pre, lane);
  else mt_seed<kMirror>(st, stream_seed, lane);
  loaded();
  uint32_t pos = 0;
  LdsWord *const base = mt_base<K, NL, kMirror>(st, lane);
  // (Every skip is at least 1 (log_p is validated on the host), but for U = 0; a walk that does not get on all the same ends.)
  // A batch's last position says on the scalar unit whether the row goes on behind it, unless 64 skips of up to 64 *
  // |inv_log2| could lead around 2^32: then every batch is looked at lane by lane.
  uint32_t whole_below = !sp.narrow || n > 0xf0000000u ? 0u : n;
  asm volatile("" : "+s"(whole_below));  // (one comparison per batch instead of three)
  if constexpr (W == kHomo) {
    // stream: K K K ...   synapse s sits at K_0 + ... + K_s
    uint32_t carry = start;
    for (;;) {
      uint32_t w[K];
      mt_generate<K, NL, kMirror, kQuick ? 0 : -1>(base, pos, lane, w);
      uint32_t incl = wave_inclusive_scan_u32(skip_from_words<kQuick, !kQuick>(w[0], w[1], sp));
      asm volatile("" : "+v"(incl));  // (else the last step of the scan and this addition become three instructions)
      uint32_t idx = carry + incl;
      const uint32_t before = carry;
      carry = __builtin_amdgcn_readlane(idx, kWave - 1);
      const bool partial = carry >= whole_below;
      bool valid = true;
      uint64_t done = 0;
      if (partial) {
        // (the positions rise from lane to lane: the lanes of the row are those below the first one at or past n)
        done = __builtin_amdgcn_ballot_w64(idx - start >= n - start);
        valid = done == 0 || lane < static_cast<int>(__builtin_ctzll(done));
        idx = valid ? idx : 0u;
        asm volatile("" : "+v"(idx));  // (a branch, not a select in every batch)
      }
      f(idx, T1(1), valid, partial);
      if (done || carry == before) break;
    }
  } else if constexpr (W == kUniform) {
    // stream: K  (w K) (w K) ...   synapse s sits at K_0 + ... + K_s, its weight precedes K_{s+1}
    constexpr int WW = WeightWords<T1>::value;
    uint32_t w0[2] = {1u, 1u};
    mt_generate<2, 1, kMirror>(mt_base<2, 1, kMirror>(st, lane), pos, lane, w0);
    uint32_t carry = start + __builtin_amdgcn_readfirstlane(skip_from_words<false, true>(w0[0], w0[1], sp, 1ull));
    for (;;) {
      uint32_t w[K];
#pragma unroll
      for (int i = 0; i < K; ++i) w[i] = 1u;
      mt_generate<K, NL, kMirror, kQuick ? WW : -1>(base, pos, lane, w);
      const T1 weight = uniform_weight(w, wa, wb);
      uint32_t skip = skip_from_words<kQuick, !kQuick>(w[WW], w[WW + 1], sp, ~0ull >> (kWave - NL));
      if (NL < kWave && lane >= NL) skip = 0;
      uint32_t incl = wave_inclusive_scan_u32(skip);
      asm volatile("" : "+v"(incl));
      const uint32_t behind = carry + incl;
      uint32_t idx = behind - skip;
      const uint32_t before = carry;
      carry = __builtin_amdgcn_readlane(behind, kWave - 1);
      const bool partial = NL < kWave || carry >= whole_below;
      bool valid = true;
      uint64_t done = 0;
      if (partial) {
        done = __builtin_amdgcn_ballot_w64(idx - start >= n - start) & (~0ull >> (kWave - NL));
        valid = lane < (done ? static_cast<int>(__builtin_ctzll(done)) : NL);
        idx = valid ? idx : 0u;
        asm volatile("" : "+v"(idx));
      }
      f(idx, weight, valid, partial);
      if (done || carry == before) break;
    }
  } else {
    // float: the stream in 2-word units is  K  (A..A K) (K) (A..A K) (K) ...   A = polar attempt (x word, y
    // word), the last A of a group is the accepted one.  double: every draw is one canonical double, so the
    // units are  K  (X Y .. X Y K) (K) ...   X, Y = the two coordinates of an attempt.  The first K after an
    // accepted attempt belongs to the synapse that receives y*mult, the second K to the one that receives the
    // saved x*mult.  Every lane evaluates its unit both ways; state_behind() assigns the roles.  Synapses 2 a
    // and 2 a + 1 of the stream so belong to its accepted attempt a.
    //
    // Bound by the issue of vector instructions: 107 per batch of 64 units (39 synapses), a fifth of them the attempts
    // worked off; 130 before a skip was tried on its upper word, the scan of the roles kept its identities and one count of
    // lanes gave the queue slots of attempts and positions (row walk of 1.5e8 synapses 841 -> 771 us, double with events 1,847 -> 1,593).
    using Q = NormalQueue<T1>;
    constexpr bool kWide = sizeof(T1) == 8;
    uint32_t *const queue = st + StreamLds<T1, W, kShort>::state_words;
    T1 *const q_attempt = reinterpret_cast<T1 *>(queue);              // x, y of the attempts queued
    uint32_t *const q_pos = queue + Q::attempts * (2 * sizeof(T1) / 4);  // their synapses' positions
    uint32_t n_attempt = 0, n_pos = 0;
    uint32_t w0[2] = {1u, 1u};
    mt_generate<2, 1, kMirror>(mt_base<2, 1, kMirror>(st, lane), pos, lane, w0);
    uint32_t carry = start + __builtin_amdgcn_readfirstlane(skip_from_words<false, true>(w0[0], w0[1], sp, 1ull));
    uint32_t entered = 0;
    ScanBefore scan_before;
    double prev_v63 = 0.0;
    const uint32_t max_batches = n / 16u + 1024u;
    for (uint32_t b = 0; b < max_batches; ++b) {
      uint32_t w[2] = {1u, 1u};
      mt_generate<2, kWave, kMirror>(base, pos, lane, w);
      T1 x, y;
      float upper = 0.0f;  // the upper word of a unit that is a skip
      bool ok;
      if constexpr (!kWide) {
        const PolarF32 a = polar_attempt(w[0], w[1]);
        x = a.x, y = a.y, upper = a.u1, ok = a.ok;
      } else {
        y = __dsub_rn(__dmul_rn(2.0, canonical_f64(w[0], w[1])), 1.0);
        x = wave_shift_up1(y);
        if (lane == 0) x = prev_v63;
        prev_v63 = read_lane_f64(y, kWave - 1);
        const double r2 = __dadd_rn(__dmul_rn(x, x), __dmul_rn(y, y));
        ok = !(r2 > 1.0 || r2 == 0.0);  // an attempt (lane - 1, lane) would be accepted
      }
      const uint32_t before = entered;
      const uint32_t state = state_behind<kWide>(ok, entered, scan_before);
      const bool accepted = state == (kWide ? 2u : 1u);
      uint64_t skips;
      if constexpr (kWide) {
        const uint64_t k1 = __ballot(state == 3u);
        skips = k1 | (k1 << 1) | (before == 3u ? 1ull : 0ull);
      } else {
        skips = __ballot(state >= 2u);
      }
      const bool is_k = __builtin_amdgcn_inverse_ballot_w64(skips);
      if constexpr (kWide) upper = static_cast<float>(w[1]);
      const uint32_t skip_any = skip_from_words<kQuick, true>(w[0], w[1], upper, sp, skips);  // wave-converged call
      const uint32_t skip = is_k ? skip_any : 0u;
      uint32_t incl = wave_inclusive_scan_u32(skip);
      asm volatile("" : "+v"(incl));  // (else the last step of the scan and the addition behind it become three instructions)
      const uint32_t idx = incl + (carry - skip);
      const uint64_t acc = __ballot(accepted);
      // Attempt a is in slot a of the queue and its two synapses' positions in slots 2 a and 2 a + 1: the attempts
      // accepted below a lane give its slot, whichever of the two it holds.
      const uint32_t attempt = lanes_below(acc, n_attempt);
      if (accepted) {
        T1 *const q = q_attempt + 2u * attempt;
        q[0] = x;
        q[1] = y;
      }
      if (is_k) {  // (of the attempt before: attempt - 1)
        if constexpr (kWide) q_pos[2u * attempt - (state == 3u ? 2u : 1u)] = idx;
        else q_pos[2u * attempt + state - 4u] = idx;
      }
      carry += __builtin_amdgcn_readlane(incl, kWave - 1);
      uint64_t done = 0;
      if (carry >= whole_below) {
        done = __ballot(idx - start >= n - start) & skips;
        // (the positions rise: the synapses of the row are the skips below the first one at or past n)
        if (done) skips &= (done ^ (done - 1u)) & ~done;
      }
      n_attempt += static_cast<uint32_t>(__popcll(acc));
      n_pos += static_cast<uint32_t>(__popcll(skips));
      while (n_pos >= 2u * Q::drain || (done && n_pos != 0u)) {
        __builtin_amdgcn_wave_barrier();
        const uint32_t at = static_cast<uint32_t>(lane);
        const bool have = kWave == static_cast<int>(Q::drain) || at < Q::drain;
        const bool valid0 = have && 2u * at < n_pos, valid1 = have && 2u * at + 1u < n_pos;
        T1 first = T1(0), second = T1(0);
        uint32_t idx0 = 0, idx1 = 0;
        if (valid0) {
          polar_weights(q_attempt[2u * at], q_attempt[2u * at + 1u], wa, wb, first, second);
          idx0 = q_pos[2u * at], idx1 = q_pos[2u * at + 1u];
          if (!valid1) idx1 = 0;
        }
        if constexpr (std::is_invocable_v<F &, uint32_t, T1, bool, uint32_t, T1, bool>) {
          f(idx0, first, valid0, idx1, second, valid1);
        } else {
#pragma unroll kWide ? 1 : 2
          for (int h = 0; h < 2; ++h) f(h ? idx1 : idx0, h ? second : first, h ? valid1 : valid0, true);
        }
        if (n_pos <= 2u * Q::drain && done) break;
        // what the group left goes to the front
        __builtin_amdgcn_wave_barrier();
        if (at < Q::spill) {
          const T1 a = q_attempt[2u * Q::drain + at];
          const uint32_t p = q_pos[2u * Q::drain + at];
          __builtin_amdgcn_wave_barrier();
          q_attempt[at] = a;
          q_pos[at] = p;
        }
        __builtin_amdgcn_wave_barrier();
        n_attempt -= Q::drain;
        n_pos -= 2u * Q::drain;
      }
      if (done) break;
    }
  }
}

// Seeds `count` generators std::mt19937{seed + first + i} and stores their 624-word states at
// states[i * 624].  One lane per stream: the 623-step recurrence of 64 streams advances in
// lock step on the vector unit, and LDS transposes 64 x 64 tiles so that every state is written
// with contiguous 256-byte stores.  The scalar unit (one per CU) can seed only one stream per
// wave at a time and saturates when every row of a large matrix needs its own generator.
void launch_seed_streams(hipStream_t stream, uint32_t seed, uint32_t first, uint32_t count, uint32_t *states);

// Streams seeded per launch_seed_streams() call by the operators that use it, and the number
// of streams from which they do.
constexpr uint32_t kSeedChunk = 131072;
constexpr uint32_t kSeedAheadMin = 8192;

}  // namespace bpl
