// Just-in-time-connectivity operators for gfx950: the matrix is never stored, its rows are
// regenerated in registers on every call from per-stream std::mt19937 generators (mt_wave.h)
// with geometric skip sampling, exactly the loop of the reference's CPU kernels
//   first = ceil(log(U)/log_p);  while (i < n) { [w = weight draw;] use(i, w); i += ceil(log(U)/log_p); }
// (lib/cpu_jitconn_event_matvec.cpp:20-31, lib/cpu_jitconn_matvec.cpp:20-29 and their *_atomic
// twins).  Stream `o` is std::mt19937{seed + o}.
//
// One wave64 owns one stream.  Each lane draws one synapse of the next batch (its skip and its
// weight), a DPP prefix sum over the skips places the 64 synapses, a ballot finds where the row
// ends.  The only memory traffic is the input vector (events are packed into an LDS bitmap when
// it fits) and the output.
//
//   row walk  ("outdim_parallel"):  stream per output element, inputs gathered, one store.
//   column walk ("atomic"):         stream per input element, silent inputs are skipped
//                                   entirely (compacted per workgroup), outputs by atomics.
//
// Reference boundary: lib/gpu_jitconn_event_matvec.cu:111-135,432-522,
// lib/gpu_jitconn_event_matvec_atomic.cu:61-85, lib/gpu_jitconn_matvec.cu:115-138,
// lib/gpu_jitconn_matvec_atomic.cu:53-77 (buffers = [input, out]; descriptors; target names).
#include <cmath>

#include <type_traits>

#include "bins.h"
#include "common.h"
#include "jitconn_lane.h"
#include "jitconn_stream.h"
#include "targets.h"

namespace bpl {
namespace {

// ---- row walk -------------------------------------------------------------------------------------
// LDS the row walk gives to an event bitmap when it wants two 16-wave workgroups per CU (each wave
// can issue one instruction every four cycles, so the number of resident waves bounds the VALU
// utilisation: 1,000,000 streams of 1,000 synapses, 32 waves per CU, 650 G synapses/s).
// What two workgroups leave of a CU's 160 KB beside their 16 waves' states and queues (homogeneous weights 33,536 bytes,
// uniform ones 29,440, double 27,392, normal ones 18,944, double 11,264: the share of events hardly matters to those, the
// second probe hides behind the weights), this at most.
constexpr uint32_t kRowwalkCoarseMost = 38912;
// Float normal weights with events keep the state with the least mirror: wrapping a batch's addresses lane by lane costs
// eight instructions, and the LDS that it saves holds twice the events' bitmap (1e5 streams of 1,000 to 1,500 synapses over
// 40,000 / 130,000 / 150,000 / 900,000 inputs: 590 / 637 / 726 / 693 us, with the long mirror 600 / 675 / 835 / 705).  Not double, whose
// batches cost more than the probes (818 / 868 / 987 / 910 with the long mirror, else 837 / 902 / 1,033 / 928), nor a dense vector
// (matvec and its gradient 1,769 us, else 1,780).
template <typename T1, int IN, int W>
constexpr bool rowwalk_short() { return IN == kInEvent && W == kNormal && sizeof(T1) == 4; }
template <typename T1, int W, bool kShort>
constexpr uint32_t rowwalk_bytes_for_two() {
  const uint32_t left = (80u * 1024u - 16u * 4u * StreamLds<T1, W, kShort>::words - 64u) / 256u * 256u;
  return left < kRowwalkCoarseMost ? left : kRowwalkCoarseMost;
}
template <typename T1, int W>
constexpr uint32_t rowwalk_coarse_bytes() { return rowwalk_bytes_for_two<T1, W, rowwalk_short<T1, kInEvent, W>()>(); }

// BITS: where the event probes go.  0: the event vector in global memory; 1: its bitmap in LDS;
// 2: a coarse bitmap in LDS (one bit per 2^g positions, at most rowwalk_coarse_bytes<T1, W>()) and, where its
// bit is set, the exact packed bitmap in global memory (`in`, the coarse one behind it).  Positions count from
// kRowwalkLead: the first word of the exact bitmap is empty, and a lane that has nothing to look up reads it.
constexpr uint32_t kRowwalkLead = 32;
// (With the coarse bitmap two 16-wave workgroups are meant to share a CU: 8 waves per SIMD, which
// the register allocation has to leave room for; the normal-weight walk needs 66 otherwise.)
// Register budget: eight waves per SIMD need at most 64 vector AND at most 80 scalar registers per
// wave here (with 81..96 scalar registers only seven fit, so a second 16-wave workgroup does not).
constexpr uint32_t kFuseBatch = 64;   // streams seeded together, one per lane
constexpr uint32_t kFuseSlots = 3;    // batches of seeded states in a workgroup's ring
constexpr uint32_t kFuseNumbers = 8;  // batch numbers a row-walk workgroup remembers (more than a wave can fall behind)
constexpr uint32_t kFuseLdsWords = 16;  // the row walk's counters and numbers, in front of the states
constexpr uint32_t kFuseRoundBits = 5;  // a number's place in the eight is told from its last use by this many bits below it
static_assert(1 + 2 * kFuseSlots + kFuseNumbers <= kFuseLdsWords, "room for them");
constexpr uint32_t kFuseSpin = 1u << 22;           // polls of a flag in LDS before a wave stops waiting
constexpr uint32_t kFuseNotSeeded = 0x80000000u;   // flag bit: the batch's rows seed their own generators
constexpr size_t kFuseRingBytes = static_cast<size_t>(kFuseSlots) * kFuseBatch * kMtN * sizeof(uint32_t);  // per workgroup
static_assert(kMtSeedTileWords <= kMtN, "the seeding wave transposes through its own state buffer");

// (The self-check's waves give up waiting for a seeded state after no poll or after three: kNoPolls, kThreePolls added to BITS.)
constexpr int kNoPolls = 4, kThreePolls = 8;
template <typename T1, typename VT, int IN, int W, int FORM, bool FUSED>
__global__ __launch_bounds__(1024, (FORM == 2 || (W == kNormal && sizeof(T1) == 4)) ? 8 : 4)
    __attribute__((amdgpu_num_sgpr(80))) void jitconn_rowwalk_kernel(const VT *__restrict__ in, T1 *__restrict__ out,
                                                               uint32_t n_out, uint32_t n_in, uint32_t seed,
                                                               SkipParams skips, T1 wa, T1 wb, uint32_t *next,
                                                               uint32_t *states) {
  constexpr int BITS = FORM & 3;
  constexpr uint32_t SPIN = (FORM & kNoPolls) ? 0u : (FORM & kThreePolls) ? 3u : kFuseSpin;
  // `states` (optional) holds the outputs' generators' seeded states.  FUSED: `states` is the workgroups' rings
  // (kFuseRingBytes each), `next` (optional) two counters that are zero.
  extern __shared__ __attribute__((aligned(8))) uint32_t smem_raw[];
  uint32_t *smem = smem_raw + (FUSED ? kFuseLdsWords : 0u);
  const int lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t nwaves = blockDim.x / kWave;
  constexpr bool kShort = rowwalk_short<T1, IN, W>();
  constexpr int kWords = StreamLds<T1, W, kShort>::words;
  uint32_t *st = smem + wave * kWords;
  const uint32_t *bits = smem + nwaves * kWords;
  constexpr uint32_t kLead = BITS == 2 ? kRowwalkLead : 0u;  // positions in front of the first input
  const uint8_t *coarse_bytes = reinterpret_cast<const uint8_t *>(smem + 16 * kWords);  // (BITS == 2: sixteen waves)
  uint32_t coarse_g = 0, coarse_g3 = 3;
  if constexpr (BITS == 2) {
    uint32_t *wbits = smem + 16 * kWords;
    coarse_g = coarse_shift(n_in + kLead, rowwalk_coarse_bytes<T1, W>());
    coarse_g3 = coarse_g + 3u;
    const uint32_t words = (coarse_bits(n_in + kLead, coarse_g) + 31u) >> 5;
    const uint32_t *coarse = reinterpret_cast<const uint32_t *>(in) + coarse_offset_words(n_in + kLead);
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) wbits[i] = coarse[i];
    __syncthreads();
    // (a shift by a scalar register takes twice the cycles; the other weights have no vector registers to spare)
    if constexpr (W == kHomo) asm volatile("" : "+v"(coarse_g), "+v"(coarse_g3));
  } else if constexpr (BITS == 1) {
    uint32_t *wbits = smem + nwaves * kWords;
    const uint32_t words = (n_in + 31u) >> 5;
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) wbits[i] = pack_events32<VT>(in, i << 5, n_in);
    __syncthreads();
  }
  // output o from stream seed + o, whose seeded state is at `pre` (or nullptr: the wave seeds it itself)
  auto walk_row = [&](uint32_t o, const uint32_t *pre, auto &&loaded) {
    double acc = 0.0;
    uint32_t cnt = 0;
    // two-level bitmap: the exact word of a batch is requested when the batch is drawn and looked
    // at when the next one is, so that no wave waits for it
    uint32_t late_word = 0, late_idx = 0;
    T1 late_w = T1(0);
    auto count_event = [&](uint32_t bit, T1 w) {  // bit: 0 or 1
      if (W == kHomo) cnt += bit;
      else if (bit) acc += static_cast<double>(w);
    };
    auto settle = [&]() { count_event(__builtin_amdgcn_ubfe(late_word, late_idx, 1u), late_w); };
    walk_stream<T1, W, true, kShort>(st, lane, seed + o, pre, n_in + kLead, skips, wa, wb,
                                     [&](uint32_t idx, T1 w, bool valid, bool partial) {
      if constexpr (IN == kInEvent && BITS == 2) {
        settle();
        // position idx: bit (idx >> g) of the coarse bitmap, bit idx of the exact one, whose word 0 holds no input: it is
        // what lanes beyond the row (position 0) and lanes without a coarse hit read
        const uint32_t byte = coarse_bytes[idx >> coarse_g3];
        const uint32_t hit = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(byte), (idx >> coarse_g) & 7u, 1u));
        const uint32_t off = __builtin_amdgcn_bitop3_b32(idx >> 3, ~3u, hit, 0x80);  // a & b & c
        late_word = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(in) + off);
        late_idx = idx;
        late_w = w;
      } else if constexpr (IN == kInEvent && BITS == 1) {
        uint32_t bit = __builtin_amdgcn_ubfe(reinterpret_cast<const uint8_t *>(bits)[idx >> 3], idx & 7u, 1u);
        if (partial) {
          bit = valid ? bit : 0u;
          asm volatile("" : "+v"(bit));  // (a branch, not a select in every batch)
        }
        count_event(bit, w);
      } else if constexpr (IN == kInEvent) {
        if (valid) count_event(probe_event(in, idx) ? 1u : 0u, w);
      } else {
        auto add = [&]() {
          const T1 v = static_cast<T1>(in[idx]);
          acc += static_cast<double>(W == kHomo ? v : static_cast<T1>(w * v));
        };
        if (!partial) add();
        else if (valid) add();
      }
    }, loaded, kLead);
    if constexpr (IN == kInEvent && BITS == 2) settle();
    if (IN == kInEvent && W == kHomo) {
      cnt = wave_inclusive_scan_u32(cnt);
      if (lane == kWave - 1) out[o] = static_cast<T1>(cnt);
    } else {
      acc = wave_sum(acc);
      if (lane == 0) out[o] = static_cast<T1>(acc);
    }
  };

  if constexpr (!FUSED) {
    for (uint32_t i = blockIdx.x * nwaves + wave; i < n_out; i += gridDim.x * nwaves)
      walk_row(i, states ? states + static_cast<size_t>(i) * kMtN : nullptr, NoLoadHook());
  } else {
    // The generators are seeded inside the kernel, 64 streams at a time on the vector unit (the scalar
    // unit, one per CU, cannot seed a stream per wave fast enough), while the other waves walk: the
    // workgroup takes batches of 64 consecutive outputs, its waves take (batch, row) tasks from a counter in LDS, and the
    // wave that takes the first row of the workgroup's batch j first takes batch j + 1 and seeds it into slot (j + 1) % 3 of
    // the workgroup's ring of seeded states in
    // device memory (`states`), which stays in the L2.  A slot is written again only after all 64 rows
    // of its previous batch have copied their state to LDS, and read only after its flag says which
    // batch it holds; these waits are bounded, and a wave that gives up seeds its own generator instead.
    //
    // Which batch is next comes from a counter of the device (`next`: batches taken, workgroups at their end): of two
    // workgroups on a CU the older one gets more of the issue slots, and with equal shares the younger one worked
    // alone, four waves to a SIMD, for the last fifth (1,000,000 streams of 1,000 synapses: 1,665 us, with the counter 1,552).  Without one
    // (`next` null), batch blockIdx.x + j * gridDim.x.  A wave knows its rows by these numbers, whatever became of the
    // seeding.  Number j + 1 is taken by the wave that seeds: from the counter as soon as batch j is ready or the wave has given up
    // on it, so that it comes before twice that wait is over (taken before, a workgroup that is behind has one more batch to
    // do).  Without one at once where rows are so short that the walk waits for the seeding alone, so that a workgroup's first
    // two batches are seeded side by side (homogeneous weights, rows of 30, 33,000 / 38,000 / 45,000 / 60,000 of them 42 / 42 / 42.6 / 52.3 us,
    // now 37 / 37 / 40.6 / 53; rows of 400 would lose, 45,000 of them 51 -> 55, and so would other weights, 60,000 rows of 30 with
    // uniform ones 55 -> 59).
    uint32_t &s_task = smem_raw[0], *const s_ready = smem_raw + 1, *const s_loaded = s_ready + kFuseSlots,
             *const s_batch = s_loaded + kFuseSlots;
    const uint32_t n_batches = (n_out + kFuseBatch - 1u) / kFuseBatch;
    // (`states` is neither const nor restrict: other waves write what this one reads behind a flag)
    uint32_t *ring = states + static_cast<size_t>(blockIdx.x) * kFuseSlots * kFuseBatch * kMtN;
    if (threadIdx.x == 0) {
      s_task = 0;
      for (uint32_t k = 0; k < kFuseSlots; ++k) s_ready[k] = 0, s_loaded[k] = 0;
      for (uint32_t k = 0; k < kFuseNumbers; ++k) s_batch[k] = 0;
    }
    __syncthreads();
    const bool early = W == kHomo && next == nullptr && static_cast<double>(n_in) * skips.log_p > -64.0;
    auto round_of = [&](uint32_t j) { return (j / kFuseNumbers + 1u) & ((1u << kFuseRoundBits) - 1u); };
    auto take_batch = [&](uint32_t j) {
      uint32_t b = blockIdx.x + j * gridDim.x;
      if (next != nullptr) {
        if (lane == 0) b = atomicAdd(&next[0], 1u);
        b = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(b)));
      }
      b = min(b, n_batches);  // (at most 2^26)
      __hip_atomic_store(&s_batch[j % kFuseNumbers], b << kFuseRoundBits | round_of(j), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      return b;
    };
    auto seed_batch = [&](uint32_t j, uint32_t b) {
      const uint32_t slot = j % kFuseSlots;
      mt_seed_batch(st, lane, seed + b * kFuseBatch + static_cast<uint32_t>(lane), ring + static_cast<size_t>(slot) * kFuseBatch * kMtN);
      __hip_atomic_store(&s_ready[slot], j + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (wave == 0) {
      const uint32_t b = take_batch(0);
      if (b < n_batches) seed_batch(0, b);
    }
    for (;;) {
      // Every lane adds one, so the counter advances by 64 per task and any lane's old value / 64 is the
      // task.  (With the add under `if (lane == 0)` the compiler split the loop by lane: lane 0 went back
      // to the add alone and the other lanes stayed behind with task 0 for ever.)
      const uint32_t t = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                             static_cast<int>(atomicAdd(&s_task, 1u)))) / kWave;
      const uint32_t j = t / kFuseBatch, r = t % kFuseBatch;
      const uint32_t slot = j % kFuseSlots;
      uint32_t number = 0, flag = 0;  // (read together: a wave that waits for neither spends one turn of the LDS on them)
      // (twice as long as a wave waits for a batch before it takes the next number: the polls there are four times as long)
      for (uint32_t spin = 0; spin < 8u * kFuseSpin; ++spin) {
        number = __hip_atomic_load(&s_batch[j % kFuseNumbers], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        flag = __hip_atomic_load(&s_ready[slot], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if ((number & ((1u << kFuseRoundBits) - 1u)) == round_of(j)) break;
        __builtin_amdgcn_s_sleep(2);
      }
      number = __builtin_amdgcn_readfirstlane(number);
      const uint32_t batch = number >> kFuseRoundBits;
      // (every wave's first task of the batch behind the last one)
      if (batch >= n_batches || (number & ((1u << kFuseRoundBits) - 1u)) != round_of(j)) break;
      auto await_states = [&]() {
        for (uint32_t spin = 0; spin < SPIN; ++spin) {
          // (A break, not a condition of the loop, which took eleven instructions a poll instead of four, and one poll in 512 cycles:
          // those of the seeding's ten microseconds take the issue slots of the wave that seeds.  100,000 streams of 20 synapses
          // 88.4 -> 86.0 us, uniform weights 94.5 -> 91.5, normal ones 98.8 -> 95.4.)
          if ((flag & ~kFuseNotSeeded) >= j + 1u) break;
          __builtin_amdgcn_s_sleep(8);
          flag = __hip_atomic_load(&s_ready[slot], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        if ((flag & ~kFuseNotSeeded) < j + 1u) flag = kFuseNotSeeded;
      };
      if (!early) await_states();
      const uint32_t behind = r == 0 ? take_batch(j + 1u) : n_batches;  // (the batch that this wave is to seed)
      if (behind < n_batches) {
        // slot (j + 1) % 3 last held batch j - 2: (j + 1) / 3 batches have used it, 64 loads each, and its flag is j - 1
        // (a wave that gave up on batch j - 2 counts as one that has loaded, also while the states are still being written)
        const uint32_t slot1 = (j + 1u) % kFuseSlots, need = ((j + 1u) / kFuseSlots) * kFuseBatch;
        bool free_ = false;
        for (uint32_t spin = 0; spin < SPIN && !free_; ++spin) {
          free_ = __hip_atomic_load(&s_loaded[slot1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) >= need &&
                  (__hip_atomic_load(&s_ready[slot1], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) & ~kFuseNotSeeded) + 3u >= j + 2u;
          if (!free_) __builtin_amdgcn_s_sleep(2);
        }
        if (free_) seed_batch(j + 1u, behind);
        else __hip_atomic_store(&s_ready[slot1], kFuseNotSeeded | (j + 2u), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      if (early) await_states();
      const uint32_t *pre = (flag & kFuseNotSeeded) ? nullptr : ring + (static_cast<size_t>(slot) * kFuseBatch + r) * kMtN;
      auto loaded = [&]() {
        if (lane == 0) __hip_atomic_fetch_add(&s_loaded[slot], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      };
      const uint32_t o = batch * kFuseBatch + r;
      if (o < n_out) walk_row(o, pre, loaded);
      else loaded();
    }
    // (the last workgroup to take a batch behind the last one leaves the counter as it was found)
    if (next != nullptr) {
      __syncthreads();
      if (threadIdx.x == 0 && atomicAdd(&next[1], 1u) == gridDim.x - 1u) next[0] = 0u, next[1] = 0u;
    }
  }
}

// ---- row walk of short streams ------------------------------------------------------------------------
// A lane per output (jitconn_lane.h): workgroups of one wave, 64 outputs each, the events probed where they lie.  The rare
// stream that is longer than its lane can draw is walked again by the whole wave, which seeds it itself.
template <typename T1, typename VT, int IN, int W>
__global__ __launch_bounds__(kWave, 8) void jitconn_rows_by_lane_kernel(const VT *__restrict__ in, T1 *__restrict__ out,
                                                                        uint32_t n_out, uint32_t n_in, uint32_t seed,
                                                                        SkipParams skips, T1 wa, T1 wb) {
  __shared__ __attribute__((aligned(8))) uint32_t st[StreamLds<T1, W, true>::words];
  const int lane = lane_id();
  const uint32_t o = blockIdx.x * kWave + static_cast<uint32_t>(lane);
  double acc = 0.0, lost = 0.0;
  uint32_t cnt = 0;
  // what a synapse meets is looked at when the next one is drawn
  VT late = VT();
  T1 late_w = T1(0);
  bool late_valid = false;
  // A wave adds a row in 64 parts and a tree; one chain of a lane would be up to four times as far off.  Double: what every
  // addition rounds away is added up beside it (Knuth's two-sum), so that the result is the rounded sum but for its last place
  // (400,000 rows of 44, dense: 70.6 -> 77.2 us; uniform weights, 20: 67.2 -> 70.1).  (Float results round the 64-bit sum to 24 bits.)
  auto plus = [&](double v) {
    if constexpr (sizeof(T1) == 8) {
      const double sum = acc + v, part = sum - acc;
      lost += (acc - (sum - part)) + (v - part);
      acc = sum;
    } else {
      acc += v;
    }
  };
  auto total = [&]() { return sizeof(T1) == 8 && lost == lost ? acc + lost : acc; };  // (an infinite sum loses NaN)
  auto use = [&](bool valid, VT v, T1 w) {
    if constexpr (IN == kInEvent) {
      const bool on = is_event(v) && valid;
      if (W == kHomo) cnt += on ? 1u : 0u;
      else plus(on ? static_cast<double>(w) : 0.0);
    } else {
      const T1 x = static_cast<T1>(v);
      if (valid) plus(static_cast<double>(W == kHomo ? x : static_cast<T1>(w * x)));
    }
  };
  auto result = [&]() { return (IN == kInEvent && W == kHomo) ? static_cast<T1>(cnt) : static_cast<T1>(total()); };
  uint32_t pos;
  uint64_t longer = walk_lane_streams<T1, W>(seed + o, o < n_out, n_in, skips, wa, wb, pos, [&](uint32_t idx, T1 w, bool valid) {
    use(late_valid, late, late_w);
    late = in[idx], late_w = w, late_valid = valid;
  });
  use(late_valid, late, late_w);
  if (o < n_out && !__builtin_amdgcn_inverse_ballot_w64(longer)) out[o] = result();
  for (; longer != 0; longer &= longer - 1ull) {
    const uint32_t row = blockIdx.x * kWave + static_cast<uint32_t>(__builtin_ctzll(longer));
    acc = 0.0, lost = 0.0, cnt = 0;
    walk_stream<T1, W, true, true>(st, lane, seed + row, nullptr, n_in, skips, wa, wb,
                                   [&](uint32_t idx, T1 w, bool valid, bool) { use(valid, in[idx], w); });
    if (IN == kInEvent && W == kHomo) cnt = wave_inclusive_scan_u32(cnt);
    else acc = wave_sum(total()), lost = 0.0;
    if (lane == ((IN == kInEvent && W == kHomo) ? kWave - 1 : 0)) out[row] = result();
  }
}

// ---- column walk ------------------------------------------------------------------------------------
constexpr int kColThreads = 256;

template <typename T1, typename VT, int IN, int W>
__global__ __launch_bounds__(kColThreads) void jitconn_colwalk_kernel(const VT *__restrict__ in,
                                                                      T1 *__restrict__ out, uint32_t n_out,
                                                                      uint32_t n_in, uint32_t seed, SkipParams skips,
                                                                      T1 wa, T1 wb) {
  constexpr int kWaves = kColThreads / kWave;
  constexpr int kWords = StreamLds<T1, W>::words;
  __shared__ __attribute__((aligned(8))) uint32_t s_state[kWaves * kWords];
  __shared__ uint32_t s_col[kColThreads];
  __shared__ T1 s_val[kColThreads];
  __shared__ uint32_t s_wave_cnt[kWaves];

  const int lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t c = blockIdx.x * kColThreads + threadIdx.x;
  T1 v = T1(0);
  bool on = false;
  if (c < n_in) {
    const VT x = in[c];
    on = is_event(x);
    v = static_cast<T1>(x);
  }
  const uint64_t mask = __ballot(on);
  if (lane == 0) s_wave_cnt[wave] = static_cast<uint32_t>(__popcll(mask));
  __syncthreads();
  uint32_t base = 0, count = 0;
#pragma unroll
  for (uint32_t i = 0; i < kWaves; ++i) {
    if (i < wave) base += s_wave_cnt[i];
    count += s_wave_cnt[i];
  }
  if (on) {
    const uint32_t k = base + static_cast<uint32_t>(__popcll(mask & ((1ull << lane) - 1ull)));
    s_col[k] = c;
    s_val[k] = v;
  }
  __syncthreads();

  uint32_t *st = s_state + wave * kWords;
  for (uint32_t k = wave; k < count; k += kWaves) {
    const uint32_t col = s_col[k];
    const T1 val = s_val[k];
    walk_stream<T1, W>(st, lane, seed + col, nullptr, n_out, skips, wa, wb, [&](uint32_t idx, T1 w, bool valid, bool) {
      if (valid) {
        T1 add;
        if (IN == kInDense) add = (W == kHomo) ? val : static_cast<T1>(w * val);
        else add = w;  // homo: w == 1
        atomic_add(&out[idx], add);
      }
    });
  }
}

// Active input columns of an event vector, gathered into a list in device memory (any order): the
// column and its value.  A workgroup lists the active ones among its kCollectCols columns in LDS
// first, so that one atomic reserves all their positions (atomics of many workgroups on the one
// counter are served one after the other).
constexpr uint32_t kCollectCols = 4096;
constexpr double kColBinEventMin = 1.0e7;  // synapses of all columns from which a walk of event columns has bins (launch_colwalk)

template <typename T1, typename VT>
__global__ __launch_bounds__(1024) void collect_active_columns_kernel(const VT *__restrict__ in, uint32_t n_in,
                                                                      uint32_t *__restrict__ counter,
                                                                      uint32_t *__restrict__ list_col,
                                                                      T1 *__restrict__ list_val,
                                                                      uint32_t *__restrict__ clear, uint32_t n_clear,
                                                                      T1 *__restrict__ zero, uint32_t n_zero) {
  // (also clears the bins' counters and the output, which the kernels behind this one add to: two launches less)
  __shared__ uint32_t s_col[kCollectCols];
  __shared__ T1 s_val[kCollectCols];
  __shared__ uint32_t s_count, s_base;
  const uint32_t tid = threadIdx.x, lane = tid % kWave;
  if (tid == 0) s_count = 0;
  for (uint32_t i = blockIdx.x * 1024u + tid; i < n_clear; i += gridDim.x * 1024u) clear[i] = 0u;
  for (uint32_t i = blockIdx.x * 1024u + tid; i < n_zero; i += gridDim.x * 1024u) zero[i] = T1(0);
  __syncthreads();
  const uint32_t c0 = blockIdx.x * kCollectCols;
  for (uint32_t t = 0; t < kCollectCols; t += 1024) {
    const uint32_t c = c0 + t + tid;
    bool on = false;
    T1 v = T1(0);
    if (c < n_in) {
      const VT x = in[c];
      on = is_event(x);
      v = static_cast<T1>(x);
    }
    const uint64_t mask = __ballot(on);
    uint32_t base = 0;
    if (lane == 0 && mask) base = atomicAdd(&s_count, static_cast<uint32_t>(__popcll(mask)));
    base = __builtin_amdgcn_readfirstlane(base);
    if (on) {
      const uint32_t k = base + static_cast<uint32_t>(__popcll(mask & ((1ull << lane) - 1ull)));
      s_col[k] = c;
      s_val[k] = v;
    }
  }
  __syncthreads();
  const uint32_t count = s_count;
  if (tid == 0) s_base = count ? atomicAdd(counter, count) : 0u;
  __syncthreads();
  const uint32_t base = s_base;
  for (uint32_t i = tid; i < count; i += 1024) {
    list_col[base + i] = s_col[i];
    list_val[base + i] = s_val[i];
  }
}

// Column walk that appends its (output, value) pairs to bins instead of adding them to `out` one
// global atomic at a time (about 21 G/s on this device).  The streams to walk are entries
// [0, n_list) of a list: column list_col[k] with value list_val[k] (event input: the active
// columns), or, without a list, column first + k with value in[first + k] (dense input).  Waves
// take entries round robin over the whole grid, so every wave walks the same number of streams.
// A wave seeding its own generator does it on the CU's one scalar unit, about 2 us each, and a
// CU's waves queue up for it.  A pair for output window b (2^shift outputs) of workgroup p goes to
// place (p * n_win + b) * cap + position of the bins; the positions continue from `counts` (zero before
// the first launch of a call), so that a call may be split into several launches; a pair that finds
// its bin full is added to `out` directly.  add_uniform_bins() then adds the bins window by window.
// The bins hold n_pairs places: `packed` (windows of at most 2^16 outputs) as an array of values with an
// array of 16-bit positions within the window behind it, 6 bytes a pair instead of 8 (10 instead of 16):
// the pairs are written once and read once, and that traffic is what a walk over a dense vector costs.
constexpr int kColBinThreads = 1024;  // 16 waves share one set of bins: 4 times fewer, 4 times larger bins
constexpr size_t kColBinBytesMax = static_cast<size_t>(3) << 30;  // bins of the dense column walk (scratch memory)

//
// So the generators are seeded inside this kernel on the vector unit, as in the row walk: workgroup p takes the
// entries p, p + G, p + 2 G, ... (G workgroups), 64 of them are a batch, its waves take (batch, entry) tasks
// from a counter in LDS, and the wave that takes the first entry of batch j first seeds batch j + 1 on the
// vector unit (lane per stream) into slot (j + 1) % 3 of the workgroup's ring of seeded states in device
// memory (`states`, kFuseRingBytes per workgroup), which the other waves read back from the L2.  Only the
// first batch of a workgroup is waited for.
template <typename T1, typename VT, int IN, int W>
__global__ __launch_bounds__(kColBinThreads, sizeof(T1) == 4 ? 8 : 4) void jitconn_colwalk_bins_kernel(
    const VT *__restrict__ in, T1 *__restrict__ out, uint32_t n_out, uint32_t seed, SkipParams skips, T1 wa, T1 wb,
    uint32_t first, uint32_t n_list_host, const uint32_t *__restrict__ n_list_dev,
    const uint32_t *__restrict__ list_col, const T1 *__restrict__ list_val, uint32_t *states,
    uint32_t n_win, uint32_t shift, uint32_t cap, void *__restrict__ pairs, uint64_t n_pairs,
    uint32_t packed, uint32_t *__restrict__ counts) {
  constexpr int kWaves = kColBinThreads / kWave;
  constexpr bool kShort = W == kNormal;  // (sixteen waves' states and queues within 64 KB of static LDS)
  constexpr int kWords = StreamLds<T1, W, kShort>::words;
  __shared__ __attribute__((aligned(8))) uint32_t s_state[kWaves * kWords];
  __shared__ uint32_t s_cnt[kBinMaxWindows];
  __shared__ uint32_t s_task, s_ready[kFuseSlots], s_loaded[kFuseSlots];

  const int lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t p = blockIdx.x;
  if (threadIdx.x < n_win) s_cnt[threadIdx.x] = counts[static_cast<size_t>(threadIdx.x) * gridDim.x + p];
  if (threadIdx.x == 0) {
    s_task = 0;
    for (uint32_t k = 0; k < kFuseSlots; ++k) s_ready[k] = 0, s_loaded[k] = 0;
  }
  __syncthreads();
  const uint64_t region = static_cast<uint64_t>(p) * n_win * cap;  // first place of this workgroup's bins
  unsigned char *const region_val = static_cast<unsigned char *>(pairs) + region * (packed ? sizeof(T1) : sizeof(BinPair<T1>));
  unsigned char *const region_rel = static_cast<unsigned char *>(pairs) + n_pairs * sizeof(T1) + region * 2u;  // (packed)
  uint32_t *st = s_state + wave * kWords;
  const uint32_t n_list = n_list_dev ? *n_list_dev : n_list_host;

  // list entry k: its stream, seeded at `pre` (or nullptr: the wave seeds it itself)
  auto walk_entry = [&](uint32_t k, const uint32_t *pre, auto &&loaded) {
    uint32_t col;
    T1 val;
    if (list_col != nullptr) {
      col = list_col[k];
      val = list_val[k];
    } else {
      col = first + k;
      val = static_cast<T1>(in[col]);
      if (!is_event(val)) {  // a zero input adds nothing (wave uniform)
        loaded();
        return;
      }
    }
    walk_stream<T1, W, true, kShort>(st, lane, seed + col, pre, n_out, skips, wa, wb, [&](uint32_t idx, T1 w, bool valid, bool partial) {
      const uint32_t b = idx >> shift;
      // The positions rise from lane to lane and the lanes that hold a synapse are the first ones of the
      // wave, so the lanes of a batch that meet in one window are neighbours (sixteen of them with
      // 16,384-output windows and conn_prob 0.001, all 64 with a dense matrix).  A returning addition
      // of several lanes to ONE counter occupies the CU's LDS for 64 cycles (measured; 7 when every lane
      // has a counter of its own), so the first lane of every run of equal windows reserves the places
      // of the whole run and the others fetch its answer (12 cycles with the shuffle): 3 to 6 % of the
      // walk, whose larger cost is the scattered stores of the pairs.  Lanes 0 and 32 begin runs of their
      // own, which keeps the masks at 32 bits, and so does the first lane without a synapse: run lengths then need no bound.
      const uint64_t valids = partial ? __builtin_amdgcn_ballot_w64(valid) : ~0ull;
      const uint64_t heads = __builtin_amdgcn_ballot_w64(b != wave_shift_up1(b)) | 0x100000001ull | (valids + 1ull);
      const uint32_t half = lane < 32 ? static_cast<uint32_t>(heads) : static_cast<uint32_t>(heads >> 32);
      const uint32_t in_half = static_cast<uint32_t>(lane) & 31u;
      const uint32_t rank = static_cast<uint32_t>(__builtin_clz(half << (31u - in_half)));  // lanes from the run's first to this one
      uint32_t first_slot = 0;
      if (__builtin_amdgcn_inverse_ballot_w64(heads & valids)) {
        // the next run begins `run` lanes above this one (a run ends with its half at the latest)
        const uint32_t above = (half >> in_half) & ~1u;
        const uint32_t run = above != 0u ? static_cast<uint32_t>(__builtin_ctz(above)) : 32u - in_half;
        first_slot = atomicAdd(&s_cnt[b], run);
      }
      const uint32_t slot = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>(4u * (static_cast<uint32_t>(lane) - rank)),
                                                                              static_cast<int>(first_slot))) + rank;
      if (valid) {
        T1 add;
        if (IN == kInDense) add = (W == kHomo) ? val : static_cast<T1>(w * val);
        else add = w;  // homo: w == 1
        if (slot < cap) {
          // (within the workgroup's region, whose bytes are counted in 32 bits; a window's number has seven, `cap` at most 24)
          const uint32_t at = static_cast<uint32_t>(__umul24(b, cap)) + slot;
          const uint32_t rel = idx & ((1u << shift) - 1u);
          if (packed) {
            *reinterpret_cast<T1 *>(region_val + at * static_cast<uint32_t>(sizeof(T1))) = add;
            *reinterpret_cast<uint16_t *>(region_rel + at * 2u) = static_cast<uint16_t>(rel);
          } else {
            BinPair<T1> e;
            e.rel = rel;
            e.val = add;
            *reinterpret_cast<BinPair<T1> *>(region_val + at * static_cast<uint32_t>(sizeof(BinPair<T1>))) = e;
          }
        } else {
          atomic_add(&out[idx], add);
        }
      }
    }, loaded);
  };

  // this workgroup's entries: p + i * G for i < mine
  const uint32_t mine = n_list > p ? (n_list - p + gridDim.x - 1u) / gridDim.x : 0u;
  const uint32_t batches = (mine + kFuseBatch - 1u) / kFuseBatch;
  uint32_t *ring = states + static_cast<size_t>(p) * kFuseSlots * kFuseBatch * kMtN;
  auto seed_batch = [&](uint32_t j) {
    const uint32_t slot = j % kFuseSlots;
    const uint32_t i = j * kFuseBatch + static_cast<uint32_t>(lane);
    uint32_t col = 0;
    if (i < mine) {
      const uint32_t k = p + i * gridDim.x;
      col = list_col != nullptr ? list_col[k] : first + k;
    }
    const uint32_t left = mine - j * kFuseBatch;
    uint32_t *const to = ring + static_cast<size_t>(slot) * kFuseBatch * kMtN;
    // (a short last batch: the quick form, for it is soon waited for; not the second of two with normal weights, whose walk of the
    // first lasts longer than the seeding: 65,000 columns of 20 116.2 -> 113.0 us)
    if (left >= kFuseBatch || (W == kNormal && j != 0u && batches == 2u)) mt_seed_batch(st, lane, seed + col, to, left);
    else mt_seed_batch<true>(st, lane, seed + col, to, left);
    __hip_atomic_store(&s_ready[slot], j + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  if (wave == 0 && batches != 0) seed_batch(0);
  // (One batch: the others wait at the barrier, where they take no issue slots from the wave that seeds.  More: the wave that
  // takes the first entry seeds batch 1 beside it; 1,000,000 streams of 18 synapses, both walks, 1,908 us, behind the barrier 1,950.)
  if (batches <= 1u) __syncthreads();
  for (;;) {
    // (every lane adds one: the counter advances by 64 per task, any lane's old value / 64 is the task)
    const uint32_t t = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                           static_cast<int>(atomicAdd(&s_task, 1u)))) / kWave;
    const uint32_t j = t / kFuseBatch, r = t % kFuseBatch;
    if (j >= batches) break;
    if (r == 0 && j + 1 < batches) {
      // slot (j + 1) % 3 last held batch j - 2: (j + 1) / 3 batches have used it, 64 loads each
      const uint32_t slot = (j + 1u) % kFuseSlots, need = ((j + 1u) / kFuseSlots) * kFuseBatch;
      bool free_ = false;
      for (uint32_t spin = 0; spin < kFuseSpin && !free_; ++spin) {
        free_ = __hip_atomic_load(&s_loaded[slot], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) >= need;
        if (!free_) __builtin_amdgcn_s_sleep(2);
      }
      if (free_) seed_batch(j + 1u);
      else __hip_atomic_store(&s_ready[slot], kFuseNotSeeded | (j + 2u), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    const uint32_t slot = j % kFuseSlots;
    uint32_t flag = 0;
    for (uint32_t spin = 0; spin < kFuseSpin; ++spin) {
      flag = __hip_atomic_load(&s_ready[slot], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
      if ((flag & ~kFuseNotSeeded) >= j + 1u) break;
      __builtin_amdgcn_s_sleep(8);
    }
    if ((flag & ~kFuseNotSeeded) < j + 1u) flag = kFuseNotSeeded;
    const uint32_t *pre = (flag & kFuseNotSeeded) ? nullptr : ring + (static_cast<size_t>(slot) * kFuseBatch + r) * kMtN;
    auto loaded = [&]() {
      if (lane == 0) __hip_atomic_fetch_add(&s_loaded[slot], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const uint32_t i = j * kFuseBatch + r;
    if (i < mine) walk_entry(p + i * gridDim.x, pre, loaded);
    else loaded();
  }
  __syncthreads();
  if (threadIdx.x < n_win) counts[static_cast<size_t>(threadIdx.x) * gridDim.x + p] = s_cnt[threadIdx.x];
}

// ---- column walk of short streams ---------------------------------------------------------------------
// The same with a lane to a column (jitconn_lane.h): batches of 64 entries, one to a workgroup before any has a second.
// The synapses that 64 columns have at one time lie anywhere, so every lane reserves a place for itself, or, where there is
// one window, the wave for all.  The rare stream that is longer than its lane can draw is finished by the whole wave.
template <typename T1, typename VT, int IN, int W>
__global__ __launch_bounds__(kColBinThreads, sizeof(T1) == 4 ? 8 : 4) void jitconn_columns_by_lane_kernel(
    const VT *__restrict__ in, T1 *__restrict__ out, uint32_t n_out, uint32_t seed, SkipParams skips, T1 wa, T1 wb,
    uint32_t first, uint32_t n_list_host, const uint32_t *__restrict__ n_list_dev,
    const uint32_t *__restrict__ list_col, const T1 *__restrict__ list_val, uint32_t n_win, uint32_t shift, uint32_t cap,
    void *__restrict__ pairs, uint64_t n_pairs, uint32_t *__restrict__ counts) {
  constexpr uint32_t kWaves = kColBinThreads / kWave;
  constexpr int kStateWords = StreamLds<T1, W, true>::words;
  __shared__ __attribute__((aligned(8))) uint32_t s_state[kWaves * kStateWords];
  __shared__ uint32_t s_cnt[kBinMaxWindows];
  const int lane = lane_id();
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave))), p = blockIdx.x;
  if (threadIdx.x < n_win) s_cnt[threadIdx.x] = counts[static_cast<size_t>(threadIdx.x) * gridDim.x + p];
  __syncthreads();
  const uint64_t region = static_cast<uint64_t>(p) * n_win * cap;  // first place of this workgroup's bins
  unsigned char *const region_val = static_cast<unsigned char *>(pairs) + region * sizeof(T1);
  unsigned char *const region_rel = static_cast<unsigned char *>(pairs) + n_pairs * sizeof(T1) + region * 2u;
  uint32_t *const st = s_state + wave * kStateWords;
  const uint32_t n_list = n_list_dev ? *n_list_dev : n_list_host;
  auto append = [&](uint32_t idx, T1 add, bool valid) {  // (the whole wave)
    const uint32_t b = idx >> shift;
    uint32_t slot = cap;
    if (cap != 0) {
      if (n_win == 1) {
        const uint64_t valids = __builtin_amdgcn_ballot_w64(valid);
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&s_cnt[0], static_cast<uint32_t>(__popcll(valids)));
        slot = lanes_below(valids, static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(base))));
      } else if (valid) {
        slot = atomicAdd(&s_cnt[b], 1u);
      }
    }
    if (!valid) return;
    if (slot < cap) {
      const uint32_t at = static_cast<uint32_t>(__umul24(b, cap)) + slot;
      const uint32_t rel = idx & ((1u << shift) - 1u);
      *reinterpret_cast<T1 *>(region_val + at * static_cast<uint32_t>(sizeof(T1))) = add;
      *reinterpret_cast<uint16_t *>(region_rel + at * 2u) = static_cast<uint16_t>(rel);
    } else {
      atomic_add(&out[idx], add);
    }
  };
  for (uint32_t batch = p + wave * gridDim.x; batch < (n_list + kWave - 1u) / kWave; batch += kWaves * gridDim.x) {
    const uint32_t k = batch * kWave + static_cast<uint32_t>(lane);
    bool on = k < n_list;
    uint32_t col = 0;
    T1 val = T1(0);
    if (on) {
      col = list_col != nullptr ? list_col[k] : first + k;
      val = list_col != nullptr ? list_val[k] : static_cast<T1>(in[col]);
      on = is_event(val);  // (a zero input adds nothing)
    }
    auto addend = [&](T1 w, T1 v) { return IN == kInDense ? (W == kHomo ? v : static_cast<T1>(w * v)) : w; };  // (homo: w == 1)
    uint32_t pos;
    uint64_t longer = walk_lane_streams<T1, W>(seed + col, on, n_out, skips, wa, wb, pos,
                                               [&](uint32_t idx, T1 w, bool valid) { append(idx, addend(w, val), valid); });
    for (; longer != 0; longer &= longer - 1ull) {
      const int of = static_cast<int>(__builtin_ctzll(longer));
      const uint32_t its_col = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(col), of));
      const uint32_t from = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(pos), of));
      const T1 its_val = list_col != nullptr ? list_val[batch * kWave + of] : static_cast<T1>(in[its_col]);
      walk_stream<T1, W, true, true>(st, lane, seed + its_col, nullptr, n_out, skips, wa, wb, [&](uint32_t idx, T1 w, bool valid, bool) {
        append(idx, addend(w, its_val), valid && idx >= from);
      });
    }
  }
  __syncthreads();
  uint32_t win = threadIdx.x;
  asm volatile("" : "+v"(win));  // (else the address from above is kept, in memory with normal weights)
  if (win < n_win) counts[static_cast<size_t>(win) * gridDim.x + p] = s_cnt[win];
}

// ---- seeding ahead ------------------------------------------------------------------------------------
constexpr int kSeedThreads = 128;

// Stream s of the launch is seed + first + s, or, with a list, seed + ids[s]; `count_dev` (optional)
// holds the number of list entries, of which at most `count` are seeded.
__global__ __launch_bounds__(kSeedThreads) void mt_seed_streams_kernel(uint32_t seed, uint32_t first, uint32_t count,
                                                                      uint32_t *__restrict__ states,
                                                                      const uint32_t *__restrict__ ids,
                                                                      const uint32_t *__restrict__ count_dev) {
  __shared__ __attribute__((aligned(8))) uint32_t s_tile[kSeedThreads / kWave][kMtSeedTileWords];
  const int lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t base = (blockIdx.x * (kSeedThreads / kWave) + wave) * kWave;  // first stream of this wave
  if (count_dev != nullptr && *count_dev < count) count = *count_dev;
  if (base >= count) return;
  const uint32_t mine = base + static_cast<uint32_t>(lane);  // lane l seeds stream base + l
  uint32_t x = seed + first + mine;
  if (ids != nullptr) x = seed + (mine < count ? ids[mine] : 0u);
  mt_seed_batch(s_tile[wave], lane, x, states + static_cast<size_t>(base) * kMtN,
                count - base < static_cast<uint32_t>(kWave) ? count - base : static_cast<uint32_t>(kWave));
}

}  // namespace

void launch_seed_streams(hipStream_t stream, uint32_t seed, uint32_t first, uint32_t count, uint32_t *states) {
  if (count == 0) return;
  hipLaunchKernelGGL(mt_seed_streams_kernel, dim3(div_up(count, kSeedThreads)), dim3(kSeedThreads), 0, stream, seed,
                     first, count, states, static_cast<const uint32_t *>(nullptr),
                     static_cast<const uint32_t *>(nullptr));
}

namespace {

// ---- launchers ----------------------------------------------------------------------------------------
bool valid_log_p(const char *target, double log_p) {
  if (!(log_p < 0.0) || std::isinf(log_p)) {
    set_error("%s: log_p must be finite and negative (conn_prob in (0, 1]), got %g", target, log_p);
    return false;
  }
  return true;
}

// Scratch memory of one row-walk call, taken with ONE request so that its parts cannot move apart:
//   [packed event bitmap, the coarse bitmap behind it (only where the launcher packs one)]
//   [rings of seeded generator states, kFuseRingBytes per workgroup (only from kSeedAheadMin outputs)]
struct RowwalkScratch {
  unsigned char *base = nullptr;
  size_t bitmap_bytes = 0;   // a multiple of 256
  uint32_t ring_groups = 0;  // workgroups that have a ring
  bool refused = false;      // the stream is being captured and the memory is not there yet: the call fails
  uint32_t *bitmap() const { return bitmap_bytes && base ? reinterpret_cast<uint32_t *>(base) : nullptr; }
  uint32_t *rings() const { return ring_groups && base ? reinterpret_cast<uint32_t *>(base + bitmap_bytes) : nullptr; }
};

// At most four row-walk workgroups share a CU (eight waves each; sixteen-wave ones two).
inline uint32_t rowwalk_max_groups() { return 4u * static_cast<uint32_t>(device_info().num_cu); }

// `optional`: a capture that finds none goes on without.
inline RowwalkScratch rowwalk_scratch(hipStream_t stream, uint32_t n_out, size_t bitmap_bytes, bool optional) {
  RowwalkScratch sc;
  sc.bitmap_bytes = (bitmap_bytes + 255) / 256 * 256;
  if (n_out >= kSeedAheadMin) {
    const uint32_t batches = div_up(n_out, kFuseBatch);
    sc.ring_groups = batches < rowwalk_max_groups() ? batches : rowwalk_max_groups();
  }
  const size_t want = sc.bitmap_bytes + sc.ring_groups * kFuseRingBytes;
  if (want == 0) return sc;
  sc.base = static_cast<unsigned char *>(stream_workspace(stream, want, optional));
  if (sc.base == nullptr && !scratch_refused_by_capture() && sc.ring_groups != 0 && sc.bitmap_bytes != 0) {
    // no room for the rings: the bitmap alone (the waves then seed their own generators)
    bpl_clear_error();
    sc.ring_groups = 0;
    sc.base = static_cast<unsigned char *>(stream_workspace(stream, sc.bitmap_bytes));
  }
  if (sc.base == nullptr) {
    sc.refused = scratch_refused_by_capture();
    if (!sc.refused) bpl_clear_error();  // (an allocation failed: paths that need no scratch memory remain)
    sc.ring_groups = 0;
  }
  return sc;
}

template <typename T1, typename VT, int IN, int W, int BITS>
void launch_rowwalk_impl(hipStream_t stream, const VT *in, T1 *out, uint32_t n_out, uint32_t n_in, uint32_t seed,
                         double log_p, T1 wa, T1 wb, int nwaves, size_t lds_bytes, const RowwalkScratch &sc) {
  const bool fused = sc.rings() != nullptr;
  auto kernel = fused ? jitconn_rowwalk_kernel<T1, VT, IN, W, BITS, true> : jitconn_rowwalk_kernel<T1, VT, IN, W, BITS, false>;
  const int block = nwaves * kWave;
  struct Cached {
    size_t lds_bytes;
    int block;
    int per_cu;
  };
  static thread_local Cached cached_for[2] = {{~size_t(0), 0, 0}, {~size_t(0), 0, 0}};
  if (fused) lds_bytes += kFuseLdsWords * sizeof(uint32_t);
  Cached &cached = cached_for[fused];
  if (cached.lds_bytes != lds_bytes || cached.block != block) {
    if (lds_bytes > 64 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(lds_bytes));
    int q = 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&q, reinterpret_cast<const void *>(kernel), block, lds_bytes) !=
            hipSuccess || q < 1) {
      (void)hipGetLastError();
      q = 1;
    }
    cached = {lds_bytes, block, q};
  }
  const unsigned resident = static_cast<unsigned>(device_info().num_cu) * static_cast<unsigned>(cached.per_cu);
  // From kSeedAheadMin outputs the generators are seeded inside the kernel, 64 at a time on the vector
  // unit, into the workgroups' rings (one launch for the whole walk); smaller walks seed in place.
  unsigned needed = fused ? div_up(n_out, kFuseBatch) : div_up(n_out, nwaves);
  if (fused && needed > sc.ring_groups) needed = sc.ring_groups;
  const unsigned grid = needed < resident ? needed : resident;
  // Batches are taken as they come from four for a workgroup on, rows of 200 synapses and more from two and a half; fewer are
  // shared out evenly, for then the workgroups that finish first, two to a CU, would take a last batch together while other CUs are
  // idle (20,000 inputs, even shares / taken: rows of 100, 45,000 of them 43.7 / 52 us, 60,000 54 / 61, 75,000 66.6 / 75, 90,000 76.3 / 82,
  // 120,000 99.6 / 104, 150,000 122.5 / 125.7, 200,000 159 / 157, normal weights 45,000 54.7 / 69, 90,000 98 / 106, 120,000 125 / 123, 200,000 196 / 192; rows of
  // 1,000, 60,000 of them 113 / 116, 75,000 133 / 136, 90,000 162 / 154, 150,000 259 / 248, normal weights 75,000 379 / 383, 90,000 468 / 446).
  // A capture that finds no counters shares them out, too.
  uint32_t *next = nullptr;
  const double per_row = -log_p * static_cast<double>(n_in);
  if (fused && 2u * div_up(n_out, kFuseBatch) >= (per_row < 200.0 ? 8u : 5u) * grid) {
    next = stream_counters(stream, true);
    if (next != nullptr) next += kWalkCounters;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), lds_bytes, stream, in, out, n_out, n_in, seed,
                     make_skip_params(log_p), wa, wb, next, sc.rings());
}

// Event probes from an LDS bitmap when it fits beside the generator states, else from global memory.
template <typename T1, typename VT, int IN, int W>
void launch_rowwalk_plain(hipStream_t stream, const VT *in, T1 *out, uint32_t n_out, uint32_t n_in, uint32_t seed,
                          double log_p, T1 wa, T1 wb, const RowwalkScratch &sc) {
  const size_t state_bytes = StreamLds<T1, W, rowwalk_short<T1, IN, W>()>::words * 4;
  const size_t cap = static_cast<size_t>(160) * 1024 - 512;
  // With the generators seeded inside the kernel every workgroup has a ring of seeded states in device
  // memory: 16-wave workgroups, so that the rings in use together are half as many and stay in the L2
  // and the memory-side cache.
  const int fused_waves = sc.rings() != nullptr ? 16 : 8;
  if (IN == kInEvent) {
    const size_t bitmap = (static_cast<size_t>(n_in) + 31) / 32 * 4;
    if (bitmap + 4 * state_bytes <= cap) {
      // Small bitmaps: 8-wave workgroups, several per CU.  Large ones: one workgroup per CU with
      // as many waves as fit beside the bitmap (each wave can issue one instruction every four
      // cycles, so the number of resident waves bounds the VALU utilisation).
      int nw = fused_waves;
      if (bitmap > 16 * 1024) {
        nw = static_cast<int>((cap - bitmap) / state_bytes);
        if (nw > 16) nw = 16;
        // Rows that seed in place and are more than one workgroup a CU works on: two workgroups of fewer waves, if they
        // hold them all (300,000 inputs, 6,000 rows of 300: 59.5 -> 58.1 us, uniform weights 61.6 -> 57.9, double 64.2 -> 59.7;
        // 8,000 rows in two turns 80).
        const size_t half = cap / 2 > bitmap ? (cap / 2 - bitmap) / state_bytes : 0, cus = static_cast<size_t>(device_info().num_cu);
        if (sc.rings() == nullptr && half < 16 && n_out > 16 * cus && n_out <= 2 * half * cus)
          nw = static_cast<int>(half);
      }
      launch_rowwalk_impl<T1, VT, IN, W, 1>(stream, in, out, n_out, n_in, seed, log_p, wa, wb, nw,
                                            bitmap + nw * state_bytes, sc);
      return;
    }
  }
  launch_rowwalk_impl<T1, VT, IN, W, 0>(stream, in, out, n_out, n_in, seed, log_p, wa, wb, fused_waves,
                                        fused_waves * state_bytes, sc);
}

// The longest event bitmap that is kept whole in LDS.  Rows that one workgroup a CU works on: kRowwalkCoarseMost, for the two
// levels take two launches more and save nothing (4,000 rows of 20 and of 300, 300,000 inputs: 32 / 34 us, in two levels 36 / 38,
// uniform weights 32 / 35 and 36 / 39, normal ones 33 / 39 and 37 / 44, double 34 / 47 and 38 / 51; 16,000 rows, seeded in the
// kernel, 29 / 35 and 33 / 39, normal ones 33 / 55 and 37 / 60).  More rows: what leaves room for two workgroups
// (20,000 / 100,000 rows of 1,000, 300,000 inputs: 76 / 195 us, 85 / 222 with one workgroup), which for rows that seed in
// place is counted with the least mirror, as the scalar unit bounds those (8,000 rows of 20 and of 300, 300,000 inputs:
// 55 / 60 us, in two levels 58 / 61).
template <typename T1, int W>
uint32_t rowwalk_exact_bytes(uint32_t n_out) {
  const uint32_t cus = static_cast<uint32_t>(device_info().num_cu);
  const bool fused = n_out >= kSeedAheadMin;
  if (n_out <= (fused ? kFuseBatch : 16u) * cus) return kRowwalkCoarseMost;
  return fused ? rowwalk_coarse_bytes<T1, W>() : rowwalk_bytes_for_two<T1, W, true>();
}

// Whether a lane walks a stream (jitconn_lane.h) rather than a wave: where its time, in us, is the smaller one by these fits of
// both (every kernel with either walk over 1,000 to 1,000,000 streams of 3 to 165 synapses, 3,000 to 600,000 places), and no more
// than one stream in 10^5 is expected to need more words than a lane can draw (4.5 standard deviations of the synapses of a row).
//
// By lane a wave takes what its longest stream takes, 2.4 standard deviations over the mean, from word 227 on more: a begin
// and a share for each of its synapses, while they wait for their own instructions, longer from one wave to a SIMD on.  By wave the
// seeding counts: on the CU's scalar unit, 11.3 us for 2,048 streams, or, from kSeedAheadMin on, for 64 streams a CU at a time.
//
// Rows, by wave / by lane at the line, floats: 4,000 of 55, 3,000 inputs 28.1 / 26.2 us, of 75 28.3 / 30.9; 10,000 of 25 22.0 / 17.9, of 55
// 22.5 / 26.9; 20,000 of 55 29.9 / 27.0, of 75 31.8 / 33.0; 80,000 of 130 70 / 66, of 165 72 / 81; uniform weights 16,000 of 25 24.1 / 17.4,
// of 55 24.3 / 28.5; normal ones 10,000 of 8 24.4 / 21.5, of 15 24.4 / 27.4, 80,000 of 40 72 / 62, of 55 73.5 / 80; in double 20,000 of 15
// 45.7 / 42.1, of 25 48 / 58.  Events whose vector the L2s do not hold lose what the walk by wave gains from their bitmap
// (500,000 rows of 167, 1,500,000 inputs of doubles 418 / 470).
//
// Columns of a dense vector: a synapse's place in the bins and its store come on top, and a walk by wave has bins from 1,048,576
// synapses on.  5,000 outputs: 4,000 columns of 25 26.6 / 25.8 us, of 40 30.5 / 40.2; 10,000 of 100 96 / 69, of 130 36 / 83; 60,000 of 55 71 / 62,
// of 100 78 / 87; doubles, whose 512 workgroups do not fit the device at once, 20,000 of 40 75 / 66, of 55 53 / 79; normal ones 8,000 of 3 36 / 26, of 15 39 / 50.
//
// Those of the events only: their number is not known here, and a wave to each of a few takes 20 us (5,000 outputs, 15 columns
// of 15 21.2 / 20.1 us, of 25 21.4 / 23.5; normal ones of 3 19.3 / 17.4, of 8 19.0 / 20.8).
enum StreamUse { kGathers, kScatters, kScattersSome };
template <typename T1, int W>
bool streams_by_lane(uint32_t streams, uint32_t n, double log_p, const SkipParams &sp, StreamUse use, uint64_t event_bytes = 0) {
  constexpr bool wide = sizeof(T1) == 8;
  const double mean = -std::expm1(log_p) * static_cast<double>(n), count = streams;
  constexpr double words = W == kHomo ? 2.0 : W == kUniform ? 2.0 + WeightWords<T1>::value : wide ? 4.55 : 3.27;
  if (!sp.narrow || n > 0xf0000000u || words * (mean + 4.5 * std::sqrt(mean)) > kLaneWords - 2.0) return false;
  const double longest = mean + 2.4 * std::sqrt(mean), steps = longest + 0.5 * std::fmax(0.0, longest - kLaneFirst / words);
  // the share of a wave's steps whose skips the upper word alone does not decide
  const double undecided = sp.quick ? -std::expm1(-128.0 * 0x1p-33 * sp.quick_band) : 1.0;
  auto of = [](double homo, double uniform, double uniform_wide, double normal, double normal_wide) {
    return W == kHomo ? homo : W == kUniform ? (wide ? uniform_wide : uniform) : wide ? normal_wide : normal;
  };
  if (use == kGathers) {
    if (event_bytes > (8u << 20)) return false;
    const double turns = std::ceil(count / 65536.0);  // waves of 64 to a SIMD
    const double step = of(wide ? 0.262 : 0.25, 0.33, 0.42, 0.73, 1.25) * (1.0 + undecided * of(0.4, 0.15, 0.1, 0.1, 0.05));
    const double by_lane = of(8.0, 6.0, 6.0, 9.0, 10.5) + step * steps * (1.0 + of(0.32, 0.42, 0.42, 0.42, 0.6) * (turns - 1.0));
    double by_wave = streams < kSeedAheadMin ? of(5.5, 4.0, 4.3, 4.7, 5.5) + 11.3 * std::ceil(count / 2048.0)
                     : streams <= 16384u     ? of(21.6, 21.3, 23.3, 24.0, 29.0) + (streams > 12288u ? 1.5 : 0.0)
                     : streams <= 32768u     ? of(29.6, 29.4, 33.0, 33.0, 45.0) + (streams > 24576u ? 1.5 : 0.0)
                                             : of(10.0, 10.0, 11.0, 11.0, 24.0) + count * (W == kNormal && wide ? 0.91e-3 : 0.75e-3);
    if (event_bytes != 0) {
      by_wave += 1.9;  // (the bitmap; one in two levels)
      if (n > 8u * kRowwalkCoarseMost) by_wave = streams <= 4096u ? 37.0 : streams < kSeedAheadMin ? 59.0 : by_wave + 5.0;
    } else if (static_cast<uint64_t>(n) * sizeof(T1) > (2u << 20) && streams > 32768u) {
      by_wave *= of(1.4, 1.25, 1.25, 1.25, 1.1);  // (a vector that the L2s hardly hold)
    }
    return by_lane < by_wave;
  }
  if (use == kScattersSome) {
    // (without bins the synapses that lanes have at one time meet few outputs in any order, a wave's are neighbours: 200,000 columns of
    // 16, 10 / 30 % events, 5,000 outputs 49 / 107, by lane 56 / 135, 20,000 outputs 43 / 90, by lane 35 / 74)
    if (!wide && n <= 10000u && mean >= 11.0 && mean * count >= 2.0e6 && mean * count < kColBinEventMin) return false;
    return steps * of(0.27, 0.31, 0.33, 0.8, 1.0) < 7.2;
  }
  const double synapses = mean * count, outs = 26e-6 * n, slower = 1.0 + 0.1 * undecided;
  double by_lane;
  if (synapses < 131072.0) {  // (no bins)
    by_lane = of(16.0, 13.0, 14.5, 15.0, 16.5) + of(0.28, 0.34, 0.41, 0.82, 1.35) * slower * steps;
  } else if (streams <= (wide ? 16384u : 32768u)) {
    by_lane = of(21.0, 19.0, 20.0, 22.0, 22.0) + outs + of(0.42, 0.43, 0.56, 0.92, 1.55) * slower * steps;
  } else {
    const double step = of(wide ? 0.85 : 0.55, 0.62, 1.08, 1.17, 2.95) * slower;
    by_lane = of(wide ? 26.0 : 22.5, 22.0, 26.0, 24.0, 36.0) + (wide && n > 16384u ? 7.0 : 0.0) + outs + 45e-6 * count + step * std::fmax(1.0, count / 220e3) * steps;
  }
  double by_wave;
  if (synapses < 1048576.0) {
    const double begin = streams <= 4096u ? of(20.0, 18.5, 18.5, 18.5, 19.5) : wide ? 33.0 : of(22.0, 20.5, 20.5, 20.5, 20.5);
    const double each = n <= 16384u ? (wide ? 0.05e-3 : 0.06e-3) : wide ? 0.035e-3 : 0.04e-3;  // (fewer outputs: more atomics to one)
    by_wave = std::fmax(begin + each * synapses, 12.0 + 0.79e-3 * count + 0.025e-3 * synapses);
  } else {
    by_wave = 0.75 * outs + (streams <= 32768u ? (wide ? 42.0 : 29.0) + 0.35e-3 * count + 0.06 * mean : (wide ? 16.0 : 10.0) + 0.9e-3 * count + mean * (streams <= 98304u ? 0.14 : 4e-6 * count));
  }
  return by_lane < by_wave;
}

template <typename T1, typename VT, int IN, int W>
void launch_rowwalk(hipStream_t stream, const VT *in, T1 *out, uint32_t n_out, uint32_t n_in, uint32_t seed,
                    double log_p, T1 wa, T1 wb) {
  if (n_out == 0) return;
  const SkipParams sp = make_skip_params(log_p);
  if (streams_by_lane<T1, W>(n_out, n_in, log_p, sp, kGathers, IN == kInEvent ? n_in * sizeof(VT) : 0)) {
    hipLaunchKernelGGL((jitconn_rows_by_lane_kernel<T1, VT, IN, W>), dim3(div_up(n_out, kWave)), dim3(kWave), 0, stream, in,
                       out, n_out, n_in, seed, sp, wa, wb);
    return;
  }
  constexpr bool kEvents = IN == kInEvent;
  const size_t words = (static_cast<size_t>(n_in) + 31) / 32;
  // A longer event bitmap (rowwalk_exact_bytes): two levels, the exact bitmap packed into global memory and a
  // coarse one made for LDS.  Wide event types: the vector is packed to one bit per element once, instead of once per workgroup.
  const uint32_t exact_most = rowwalk_exact_bytes<T1, W>(n_out);
  const bool two_level = kEvents && words * 4 > exact_most && n_in <= 0xffffffffu - kRowwalkLead;
  const bool packed = kEvents && (two_level || sizeof(VT) > 1);
  uint32_t g = 0, off = 0, c_words = 0;
  size_t bitmap_ws = 0;
  if (two_level) {
    g = coarse_shift(n_in + kRowwalkLead, rowwalk_coarse_bytes<T1, W>());
    off = coarse_offset_words(n_in + kRowwalkLead);
    c_words = (coarse_bits(n_in + kRowwalkLead, g) + 31u) / 32u;
    bitmap_ws = (static_cast<size_t>(off) + c_words + 1) * sizeof(uint32_t);
  } else if (packed) {
    bitmap_ws = (words + 1) * sizeof(uint32_t);
  }
  // (Refused in a capture, the call ends with the error: a graph must not record a slower path.  But for byte events whose
  // bitmap is no longer than what LDS may keep of one: without rings such a walk is captured without scratch memory.)
  const bool optional = kEvents && sizeof(VT) == 1 && n_out < kSeedAheadMin && words * 4 <= kRowwalkCoarseMost;
  const RowwalkScratch sc = rowwalk_scratch(stream, n_out, bitmap_ws, optional);
  if (sc.refused && !optional) return;
  if constexpr (kEvents) {
    if (uint32_t *bits = sc.bitmap()) {
      pack_event_bitmap<VT>(stream, in, n_in, bits, two_level ? kRowwalkLead / 32u : 0u);
      const PackedBits *pin = reinterpret_cast<const PackedBits *>(bits);
      if (two_level) {
        hipLaunchKernelGGL(coarsen_bitmap_kernel, dim3(div_up(c_words, 256)), dim3(256), 0, stream, bits,
                           static_cast<uint32_t>(words + kRowwalkLead / 32u), g, bits + off, c_words);
        const size_t state_bytes = StreamLds<T1, W, rowwalk_short<T1, IN, W>()>::words * 4;
        launch_rowwalk_impl<T1, PackedBits, IN, W, 2>(stream, pin, out, n_out, n_in, seed, log_p, wa, wb, 16,
                                                      static_cast<size_t>(c_words) * 4 + 16 * state_bytes, sc);
      } else {
        launch_rowwalk_plain<T1, PackedBits, IN, W>(stream, pin, out, n_out, n_in, seed, log_p, wa, wb, sc);
      }
      return;
    }
  }
  launch_rowwalk_plain<T1, VT, IN, W>(stream, in, out, n_out, n_in, seed, log_p, wa, wb, sc);
}

template <typename T1, typename VT, int IN, int W>
void launch_colwalk(hipStream_t stream, const VT *in, T1 *out, uint32_t n_out, uint32_t n_in, uint32_t seed,
                    double log_p, T1 wa, T1 wb) {
  if (n_in == 0 || n_out == 0) {
    fill_zero(stream, out, n_out);
    return;
  }
  bool out_cleared = false;  // (with event input and bins, the kernel that lists the active columns clears it)
  // Many pairs: bins (also for a narrow output: seeding on the vector unit and the even spread of the streams pay).  The number of pairs is n_in * n_out * p for a
  // dense input; for events it depends on the activity, which the host does not know: bins are sized
  // for one column in eight being active (fuller bins overflow into direct atomics) and used when
  // one active column in a hundred already means a hundred thousand pairs (10,000 x 10,000 with
  // conn_prob 0.1: 44, 54 and 61 us at 0.1, 1 and 20 % activity; without bins 40, 44 and 152 us).
  const uint32_t shift = bin_window_shift(n_out);
  const uint32_t n_win = div_up(n_out, 1u << shift);
  const double p_conn = -std::expm1(log_p);
  const double full = static_cast<double>(n_in) * static_cast<double>(n_out) * p_conn;
  const SkipParams sp = make_skip_params(log_p);
  // (streams that a lane can draw reach windows of 2^16 outputs at most, which streams_by_lane() has seen to: positions of 16 bits)
  const bool by_lane = (IN == kInDense || n_in >= 2048) && shift <= 16u && streams_by_lane<T1, W>(n_in, n_out, log_p, sp, IN == kInDense ? kScatters : kScattersSome);
  const bool bins = n_win <= kBinMaxWindows && full >= (IN == kInEvent ? kColBinEventMin : by_lane ? 131072.0 : 1048576.0);
  // Event input and fewer pairs: the same list of active columns and the same seeding on the vector unit, but
  // the walk adds its pairs to `out` with atomics.  (A wave that seeds its own stream spends 2 us of the CU's one
  // scalar unit on it: with 200,000 active columns of ten synapses each the walk without a list took 1.2 ms.)
  // A dense input with fewer pairs takes the same walk over all its columns, chunk by chunk (4,000 x
  // 4,000 with conn_prob 0.02: 0.5 ms where every lane seeded the generator of its own column).
  // (Event input with fewer than 2,048 columns stays with the walk below: at 1 % activity its one launch takes 26 us
  // against the 35 us of list, seeds and walk, though 125 against 47 us at 20 %.)
  const bool listed = !bins && (IN == kInDense || n_in >= 2048);
  if (bins || listed) {
    const uint32_t n_win = bins ? div_up(n_out, 1u << bin_window_shift(n_out)) : 1u;  // (no bins: every pair overflows)
    const uint32_t shift = bins ? bin_window_shift(n_out) : 31u;
    uint32_t producers = 2u * static_cast<uint32_t>(device_info().num_cu);
    const uint32_t least = by_lane ? kWave : kColBinThreads / kWave;  // columns that occupy a producer
    if (producers > div_up(n_in, least)) producers = div_up(n_in, least);
    auto round_up = [](size_t v) { return (v + 255) / 256 * 256; };
    // Dense input: the bins are emptied (added to `out`) after every `group` chunks of kSeedChunk columns,
    // the largest number of chunks whose pairs fit kColBinBytesMax of scratch memory (every column of a
    // 1,000,000 x 1,000,000 matrix with conn_prob 0.001 at once would take 10.7 GB).
    const bool packed = shift <= 16;
    const size_t pair_size = packed ? sizeof(T1) + 2 : sizeof(BinPair<T1>);
    const uint32_t chunks = div_up(n_in, kSeedChunk);
    uint32_t group = chunks;
    double cap_d = 0.0;
    size_t pair_bytes = 0;
    for (;;) {
      const double share = (group >= chunks) ? 1.0 : static_cast<double>(group) * kSeedChunk / static_cast<double>(n_in);
      double per_bin = full * share / (static_cast<double>(producers) * n_win);  // every column active
      // (by lane a producer has whole batches)
      const double batch = full / n_in * kWave / n_win;
      if (by_lane && IN == kInDense) per_bin = std::ceil(std::ceil(share * n_in / kWave) / producers) * batch;
      cap_d = 1.25 * per_bin + 6.0 * std::sqrt(per_bin) + 128.0;
      if (IN == kInEvent) cap_d = std::fmax(cap_d / 8.0, by_lane ? std::fmax(512.0, 2.0 * batch + 128.0) : 512.0);
      cap_d = std::floor(cap_d / 4.0) * 4.0;  // (packed bins begin at multiples of four places)
      pair_bytes = round_up(static_cast<size_t>(producers) * n_win * static_cast<size_t>(cap_d) * pair_size);
      if (IN == kInEvent || group == 1 || pair_bytes <= kColBinBytesMax) break;
      group = (group + 1u) / 2u;
    }
    // no bins (every pair goes to `out` with an atomic): nothing to size and nothing to empty between the chunks
    if (!bins) cap_d = 0.0, pair_bytes = 0, group = chunks;
    const size_t count_bytes = round_up(static_cast<size_t>(n_win) * producers * sizeof(uint32_t));
    // the workgroups' rings of generator states, seeded inside the walk
    const size_t state_bytes = by_lane ? 0 : round_up(static_cast<size_t>(producers) * kFuseRingBytes);
    const size_t list_bytes = (IN == kInEvent) ? round_up(static_cast<size_t>(n_in) * 4) : 0;
    const size_t val_bytes = (IN == kInEvent) ? round_up(static_cast<size_t>(n_in) * sizeof(T1)) : 0;
    uint32_t *list_count = (IN == kInEvent) ? stream_counters(stream) : nullptr;
    if (cap_d < 4.0e9 && pair_bytes <= (static_cast<size_t>(32) << 30) && (IN == kInDense || list_count != nullptr)) {
      // (a producer's region is addressed with 32 bits of bytes, a bin's places with 24: more than scratch memory holds, but
      // for a handful of producers)
      const double addressable = 4294967040.0 / (static_cast<double>(n_win) * sizeof(BinPair<T1>));
      cap_d = std::fmin(cap_d, std::floor(std::fmin(addressable, 16777212.0) / 4.0) * 4.0);
      const uint32_t cap = static_cast<uint32_t>(cap_d);
      unsigned char *ws = static_cast<unsigned char *>(
        stream_workspace(stream, pair_bytes + count_bytes + state_bytes + list_bytes + val_bytes));
      if (ws != nullptr) {
        void *pairs = ws;
        const uint64_t n_pairs = static_cast<uint64_t>(producers) * n_win * cap;
        uint32_t *counts = reinterpret_cast<uint32_t *>(ws + pair_bytes);
        uint32_t *states = reinterpret_cast<uint32_t *>(ws + pair_bytes + count_bytes);
        uint32_t *list_col = list_bytes ? reinterpret_cast<uint32_t *>(ws + pair_bytes + count_bytes + state_bytes) : nullptr;
        T1 *list_val = val_bytes ? reinterpret_cast<T1 *>(ws + pair_bytes + count_bytes + state_bytes + list_bytes) : nullptr;
        auto walk = jitconn_colwalk_bins_kernel<T1, VT, IN, W>;
        auto walk_lanes = jitconn_columns_by_lane_kernel<T1, VT, IN, W>;
        out_cleared = true;
        if (IN == kInEvent) {
          // the active columns, then one walk that seeds their generators as it goes
          hipLaunchKernelGGL((collect_active_columns_kernel<T1, VT>), dim3(div_up(n_in, kCollectCols)), dim3(1024), 0, stream,
                             in, n_in, list_count, list_col, list_val, counts, n_win * producers, out, n_out);
          if (by_lane) {
            hipLaunchKernelGGL(walk_lanes, dim3(producers), dim3(kColBinThreads), 0, stream, in, out, n_out, seed, sp, wa,
                               wb, 0u, 0u, static_cast<const uint32_t *>(list_count), static_cast<const uint32_t *>(list_col),
                               static_cast<const T1 *>(list_val), n_win, shift, cap, pairs, n_pairs, counts);
          } else {
            hipLaunchKernelGGL(walk, dim3(producers), dim3(kColBinThreads), 0, stream, in, out, n_out, seed, sp, wa, wb,
                               0u, 0u, static_cast<const uint32_t *>(list_count), static_cast<const uint32_t *>(list_col),
                               static_cast<const T1 *>(list_val), states, n_win, shift, cap, pairs, n_pairs, packed ? 1u : 0u, counts);
          }
        } else {
          // every column, a chunk at a time; the bins are emptied after every `group` chunks (by lane: after every launch)
          fill_zero(stream, out, n_out);
          fill_zero(stream, counts, n_win * producers);
          uint32_t in_bins = 0;
          const uint64_t span = by_lane ? static_cast<uint64_t>(group) * kSeedChunk : kSeedChunk;
          if (by_lane) group = 1;
          for (uint64_t at = 0; at < n_in; at += span) {
            const uint32_t first = static_cast<uint32_t>(at);
            const uint32_t count = static_cast<uint32_t>(n_in - at < span ? n_in - at : span);
            if (by_lane) {
              hipLaunchKernelGGL(walk_lanes, dim3(producers), dim3(kColBinThreads), 0, stream, in, out, n_out, seed, sp, wa,
                                 wb, first, count, static_cast<const uint32_t *>(nullptr),
                                 static_cast<const uint32_t *>(nullptr), static_cast<const T1 *>(nullptr), n_win, shift, cap,
                                 pairs, n_pairs, counts);
            } else {
              hipLaunchKernelGGL(walk, dim3(producers), dim3(kColBinThreads), 0, stream, in, out, n_out, seed, sp, wa,
                                 wb, first, count, static_cast<const uint32_t *>(nullptr),
                                 static_cast<const uint32_t *>(nullptr), static_cast<const T1 *>(nullptr), states,
                                 n_win, shift, cap, pairs, n_pairs, packed ? 1u : 0u, counts);
            }
            if (++in_bins == group && at + span < n_in) {
              if (!add_uniform_bins<T1>("jitconn column walk", stream, out, n_out, shift, producers, cap, pairs, packed, counts,
                                        static_cast<uint32_t *>(nullptr)))
                return;  // (the error stands: part of the pairs is in `out` already)
              fill_zero(stream, counts, n_win * producers);
              in_bins = 0;
            }
          }
        }
        if (!bins) {
          if (list_count != nullptr) fill_zero(stream, list_count, 1u);  // (the list's counter goes back to zero for the next call)
          return;
        }
        if (add_uniform_bins<T1>("jitconn column walk", stream, out, n_out, shift, producers, cap, pairs, packed, counts, list_count))
          return;
        // (the bins could not be added: nothing reached `out` yet except overflow pairs; start over)
        if (list_count != nullptr) fill_zero(stream, list_count, 1u);
        out_cleared = false;
      } else {
        if (scratch_refused_by_capture()) return ensure_error("jitconn column walk", "nothing was enqueued: the path that the scratch memory at hand allows could not be launched");
        bpl_clear_error();
      }
    }
  }
  if (!out_cleared) fill_zero(stream, out, n_out);
  hipLaunchKernelGGL((jitconn_colwalk_kernel<T1, VT, IN, W>), dim3(div_up(n_in, kColThreads)), dim3(kColThreads), 0,
                     stream, in, out, n_out, n_in, seed, make_skip_params(log_p), wa, wb);
}

// buffers = [input, out].  RAW_PROB: the descriptor's probability field holds conn_prob itself, as the
// reference packs it for its first-generation dense-vector targets (matvec.py:338-343); the walk then uses
// the log_p its CPU path derives from it (matvec.py:298), so that both versions give one matrix.
template <typename T1, typename VT, int IN, int W, bool COLWALK, bool RAW_PROB = false>
void jitconn_entry(const char *target, hipStream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  uint32_t n_row, n_col, seed;
  double log_p, a = 0, b = 0;
  if (W == kHomo) {
    bpl_jitconn_prob_homo_descriptor d;
    if (!unpack(target, opaque, opaque_len, &d)) return;
    n_row = d.n_row, n_col = d.n_col, seed = d.seed, log_p = d.log_p;
  } else {
    bpl_jitconn_prob_weight_descriptor d;
    if (!unpack(target, opaque, opaque_len, &d)) return;
    n_row = d.n_row, n_col = d.n_col, seed = d.seed, log_p = d.log_p, a = d.w_a, b = d.w_b;
  }
  if (RAW_PROB) {
    const double p = log_p;
    if (!(p > 0.0) || std::isinf(p)) {
      set_error("%s: conn_prob must be in (0, 1], got %g", target, p);
      return;
    }
    log_p = std::log(p < 1.0 ? 1.0 - p : 1e-40);
  }
  if (!valid_log_p(target, log_p)) return;
  if (buffers == nullptr) {
    set_error("%s: null buffer table", target);
    return;
  }
  const VT *in = static_cast<const VT *>(buffers[0]);
  T1 *out = static_cast<T1 *>(buffers[1]);
  if (COLWALK) launch_colwalk<T1, VT, IN, W>(stream, in, out, n_row, n_col, seed, log_p, static_cast<T1>(a), static_cast<T1>(b));
  else launch_rowwalk<T1, VT, IN, W>(stream, in, out, n_row, n_col, seed, log_p, static_cast<T1>(a), static_cast<T1>(b));
  check_launch(target);
}

// ---- self-check of the skip computation -------------------------------------------------------------
// Draw t of the check: mode 0, two hashed words; mode 1, the canonical value next to a ceil() boundary:
// U * 2^64 = exp(k * log_p) * 2^64 + j * 2^11 for k = t / 64 + 1, j = t % 64 - 32 (2^11: one unit in the
// last place of a double in [0.5, 1)).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__global__ __launch_bounds__(256) void check_skips_kernel(uint32_t seed, uint64_t n, int mode, SkipParams sp,
                                                          unsigned long long *__restrict__ counts,
                                                          unsigned long long *__restrict__ levels) {
  unsigned long long differ = 0, untrusted = 0, untrusted_close = 0, untrusted_quick = 0;
  for (uint64_t t = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x; t < n;
       t += static_cast<uint64_t>(gridDim.x) * 256u) {
    uint64_t bits;
    if (mode == 0) {
      bits = mix64(t + (static_cast<uint64_t>(seed) << 32));
    } else {
      const double edge = exp(static_cast<double>(t / 64u + 1u) * sp.log_p) * 0x1p64;
      bits = (edge < 0x1p64 ? static_cast<uint64_t>(edge) : ~0ull) +
             static_cast<uint64_t>((static_cast<int64_t>(t % 64u) - 32) * 2048);
    }
    const uint32_t lo = static_cast<uint32_t>(bits), hi = static_cast<uint32_t>(bits >> 32);
    uint64_t unsafe;
    const uint64_t me = 1ull << lane_id();
    const uint32_t fast = skip_fast(lo, hi, sp, unsafe);
    const uint32_t exact = skip_exact(lo, hi, sp);
    if (unsafe & me) ++untrusted;
    else if (fast != exact) ++differ;
    const uint32_t close = skip_close(lo, hi, sp, unsafe);
    if (unsafe & me) ++untrusted_close;
    else if (close != exact) ++differ;
    const float uppers[] = {static_cast<float>(hi), canonical_f32_scaled(hi)};
    for (const float upper : uppers) {
      const uint32_t quick = skip_quick(hi, upper, sp, unsafe);
      if (unsafe & me) ++untrusted_quick;
      else if (sp.quick && quick != exact) ++differ;
    }
  }
  if (counts != nullptr && differ) atomicAdd(&counts[0], differ);
  if (counts != nullptr && untrusted) atomicAdd(&counts[1], untrusted);
  if (levels != nullptr) {
    if (untrusted_quick) atomicAdd(&levels[0], untrusted_quick);
    if (untrusted) atomicAdd(&levels[1], untrusted);
    if (untrusted_close) atomicAdd(&levels[2], untrusted_close);
    if (blockIdx.x == 0 && threadIdx.x == 0) levels[3] = sp.quick ? 1u : 0u;
  }
}

// |hardware log2 - log2| over every fp32 in [0.5, 1): the largest, as the bits of a double; and over those in
// [2^-10, 1) against what the quick path allows it, counted with the draws that differ
__global__ __launch_bounds__(256) void check_log2_kernel(unsigned long long *__restrict__ worst,
                                                         unsigned long long *__restrict__ differ) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;  // < 2^23
  for (uint32_t e = 0; e < 10u; ++e) {
    const float u = __uint_as_float((0x3f000000u - (e << 23)) | t);
    const double off = fabs(static_cast<double>(__builtin_amdgcn_logf(u)) - log2(static_cast<double>(u)));
    if (!(off <= 9.6e-7)) atomicAdd(differ, 1ull);
  }
  const float m = __uint_as_float(0x3f000000u | t);
  const double err = fabs(static_cast<double>(__log2f(m)) - log2(static_cast<double>(m)));
  double wave_worst = err;
  for (int d = kWave / 2; d > 0; d >>= 1) wave_worst = fmax(wave_worst, __shfl_xor(wave_worst, d, kWave));
  if (lane_id() == 0) atomicMax(worst, static_cast<unsigned long long>(__double_as_longlong(wave_worst)));
  if (t == 0) worst[1] = static_cast<unsigned long long>(__double_as_longlong(kSkipLog2Error));
}

}  // namespace

void jitconn_seed_streams(hipStream_t stream, uint32_t seed, uint32_t first, uint32_t count, uint32_t *states) {
  launch_seed_streams(stream, seed, first, count, states);
}

}  // namespace bpl

using namespace bpl;

extern "C" int bpl_selfcheck_jitconn_skips(bpl_stream_t stream, uint32_t seed, uint64_t n_draws, int near_boundaries,
                                           double log_p, uint64_t *counts) {
  if (counts == nullptr || !(log_p < 0.0)) {
    set_error("bpl_selfcheck_jitconn_skips: counts must be device memory for four words and log_p negative");
    return 1;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned long long *c = reinterpret_cast<unsigned long long *>(counts);
  hipLaunchKernelGGL(check_skips_kernel, dim3(2048), dim3(256), 0, s, seed, n_draws, near_boundaries ? 1 : 0, make_skip_params(log_p), c,
                     static_cast<unsigned long long *>(nullptr));
  hipLaunchKernelGGL(check_log2_kernel, dim3((1u << 23) / 256u), dim3(256), 0, s, c + 2, c);
  return check_launch("bpl_selfcheck_jitconn_skips") ? 0 : 1;
}

extern "C" int bpl_selfcheck_jitconn_trust(bpl_stream_t stream, uint32_t seed, uint64_t n_draws, double log_p, uint64_t *counts) {
  if (counts == nullptr || !(log_p < 0.0)) {
    set_error("bpl_selfcheck_jitconn_trust: counts must be device memory for four words and log_p negative");
    return 1;
  }
  hipLaunchKernelGGL(check_skips_kernel, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream), seed, n_draws, 0,
                     make_skip_params(log_p), static_cast<unsigned long long *>(nullptr),
                     reinterpret_cast<unsigned long long *>(counts));
  return check_launch("bpl_selfcheck_jitconn_trust") ? 0 : 1;
}

extern "C" int bpl_selfcheck_jitconn_rowwalk(bpl_stream_t stream, const uint8_t *events, float *out, uint32_t n_out,
                                             uint32_t n_in, uint32_t seed, double log_p, uint32_t polls, uint32_t groups,
                                             int counter) {
  const char *const name = "bpl_selfcheck_jitconn_rowwalk";
  const uint32_t batches = div_up(n_out, kFuseBatch);
  if (events == nullptr || out == nullptr || !(log_p < 0.0) || n_in == 0 || n_in > 131072u || groups == 0 ||
      groups > batches || groups > rowwalk_max_groups() || (polls != 0 && polls != 3)) {
    set_error("%s: up to 131,072 inputs, no more workgroups than batches of %u outputs, 0 or 3 polls", name, kFuseBatch);
    return 1;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  void *const rings = stream_workspace(s, static_cast<size_t>(groups) * kFuseRingBytes);
  uint32_t *const counters = counter ? stream_counters(s) : nullptr;
  if (rings == nullptr || (counter && counters == nullptr)) return 1;
  auto kernel = polls == 0 ? jitconn_rowwalk_kernel<float, uint8_t, kInEvent, kHomo, 1 + kNoPolls, true>
                           : jitconn_rowwalk_kernel<float, uint8_t, kInEvent, kHomo, 1 + kThreePolls, true>;
  const size_t lds = (kFuseLdsWords + 16 * StreamLds<float, kHomo>::words + div_up(n_in, 32)) * sizeof(uint32_t);
  if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          static_cast<int>(lds)) != hipSuccess) {
    (void)hipGetLastError();
    set_error("%s: %zu bytes of LDS are not to be had", name, lds);
    return 1;
  }
  hipLaunchKernelGGL(kernel, dim3(groups), dim3(1024), lds, s, events, out, n_out, n_in, seed, make_skip_params(log_p),
                     0.0f, 0.0f, counters ? counters + kWalkCounters : nullptr, static_cast<uint32_t *>(rings));
  return check_launch(name) ? 0 : 1;
}

extern "C" int bpl_selfcheck_jitconn_by_lane(uint32_t weights, uint32_t value_bytes, uint32_t streams, uint32_t n, double log_p,
                                             uint32_t use, uint32_t event_bytes) {
  if (weights > 2u || (value_bytes != 4u && value_bytes != 8u) || use > 2u) {
    set_error("bpl_selfcheck_jitconn_by_lane: no such weights, values or use");
    return -1;
  }
  auto ask = [&](auto value, auto kind) {
    return streams_by_lane<decltype(value), decltype(kind)::value>(streams, n, log_p, make_skip_params(log_p), static_cast<StreamUse>(use),
                                                                 static_cast<uint64_t>(event_bytes) * n);
  };
  auto of = [&](auto value) {
    return weights == 0u ? ask(value, std::integral_constant<int, kHomo>())
                         : weights == 1u ? ask(value, std::integral_constant<int, kUniform>())
                                         : ask(value, std::integral_constant<int, kNormal>());
  };
  return value_bytes == 4u ? of(0.0f) : of(0.0);
}

#define BPL_DEFINE(name, ...)                                                                      \
  extern "C" void name(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) { \
    jitconn_entry<__VA_ARGS__>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len); \
  }

// event input: <result type, event type, kInEvent, weight kind, column walk>
#define BPL_EVENT_FAMILY(wname, W)                                                                           \
  BPL_DEFINE(gpu_event_matvec_prob_##wname##_v2_float_bool, float, uint8_t, kInEvent, W, false)               \
  BPL_DEFINE(gpu_event_matvec_prob_##wname##_v2_float_float, float, float, kInEvent, W, false)                \
  BPL_DEFINE(gpu_event_matvec_prob_##wname##_v2_double_bool, double, uint8_t, kInEvent, W, false)             \
  BPL_DEFINE(gpu_event_matvec_prob_##wname##_v2_double_double, double, double, kInEvent, W, false)            \
  BPL_DEFINE(gpu_event_matvec_atomic_prob_##wname##_v2_float_bool, float, uint8_t, kInEvent, W, true)         \
  BPL_DEFINE(gpu_event_matvec_atomic_prob_##wname##_v2_float_float, float, float, kInEvent, W, true)          \
  BPL_DEFINE(gpu_event_matvec_atomic_prob_##wname##_v2_double_bool, double, uint8_t, kInEvent, W, true)       \
  BPL_DEFINE(gpu_event_matvec_atomic_prob_##wname##_v2_double_double, double, double, kInEvent, W, true)

#define BPL_DENSE_FAMILY(wname, W)                                                           \
  BPL_DEFINE(gpu_matvec_prob_##wname##_v2_float, float, float, kInDense, W, false)            \
  BPL_DEFINE(gpu_matvec_prob_##wname##_v2_double, double, double, kInDense, W, false)         \
  BPL_DEFINE(gpu_matvec_atomic_prob_##wname##_v2_float, float, float, kInDense, W, true)      \
  BPL_DEFINE(gpu_matvec_atomic_prob_##wname##_v2_double, double, double, kInDense, W, true)

// the reference's first-generation names (lib/gpu_ops.cc:143-148): row walk only, conn_prob in the descriptor
#define BPL_DENSE_V1_FAMILY(wname, W)                                                        \
  BPL_DEFINE(gpu_matvec_prob_##wname##_v1_float, float, float, kInDense, W, false, true)      \
  BPL_DEFINE(gpu_matvec_prob_##wname##_v1_double, double, double, kInDense, W, false, true)

BPL_EVENT_FAMILY(homo, kHomo)
BPL_EVENT_FAMILY(uniform, kUniform)
BPL_DENSE_FAMILY(homo, kHomo)
BPL_DENSE_FAMILY(uniform, kUniform)
BPL_EVENT_FAMILY(normal, kNormal)
BPL_DENSE_FAMILY(normal, kNormal)
BPL_DENSE_V1_FAMILY(homo, kHomo)
BPL_DENSE_V1_FAMILY(uniform, kUniform)
BPL_DENSE_V1_FAMILY(normal, kNormal)
