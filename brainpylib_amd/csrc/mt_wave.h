// A std::mt19937 stream generated cooperatively by one wave64, state in LDS.
//
// The jitconn operators draw one generator stream per output row (or per input column):
// stream i is std::mt19937{seed + i}, the generator of the reference's CPU backend
// (lib/cpu_jitconn_event_matvec.cpp:20-21), restarted per stream the way the reference's GPU
// backend restarts its generator per row (lib/gpu_jitconn_event_matvec.cu:94-96).  A row is
// then exactly what the reference CPU code produces for a one-row matrix seeded `seed + i`.
//
// MT19937 produces word t from words t-624, t-623 and t-227, so up to 227 consecutive words can
// be produced at once from the previous 624: each lane computes K consecutive words
// (64*K <= 227) of the next batch and the 624-word state is a circular buffer in LDS, followed by
// a copy of its first words so that a run of consecutive words never wraps.
// Seeding is a serial 623-step recurrence; it runs on the scalar unit (the seed is wave
// uniform) and the values are packed 64 at a time into a vector register with v_writelane.
#pragma once

#include <cmath>

#include "common.h"

namespace bpl {

constexpr int kMtN = 624;
constexpr int kMtM = 397;
// st[624 + i] repeats st[i] for i < kMirror, so that a run of kMirror + 1 words from any slot on is contiguous.  Either the
// least, what a lane reads (then every lane wraps its own two addresses), or what a whole batch reads: the batch begins
// at a wave-uniform slot and its addresses are two additions instead of eight instructions.
constexpr int kMtLeastMirror = 4;

template <int kMirror>
__device__ __forceinline__ void mt_seed(uint32_t *st, uint32_t seed, int lane) {
  uint32_t x = __builtin_amdgcn_readfirstlane(seed);
#pragma unroll 1
  for (int base = 0; base < kMtN; base += kWave) {
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < kWave; ++i) {
      // lane i of v <- x  (x lives in a scalar register)
      asm volatile("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(x), "n"(i));
      x = 1812433253u * (x ^ (x >> 30)) + static_cast<uint32_t>(base + i + 1);
    }
    if (base + lane < kMtN) st[base + lane] = v;
    if (base + lane < kMirror) st[kMtN + base + lane] = v;
  }
}

// Copies a state seeded elsewhere (624 words at `src`) into the wave's LDS buffer.  All its loads are in flight
// together: in a walk over short streams this latency is what is waited for, and the compiler, left to itself, put the last
// load behind the wait for the others and, where registers are scarce, waited for every other one (row and column walk of
// 400,000 x 9,000 with 18 synapses a row 878 -> 821 us, of 100,000 x 7,000 with 140 339 -> 328, of 50,000 x 3,000 with 600
// 266 -> 256; normal weights with every other load waited for: 100,000 rows of 140 403 us, now 371).
template <int kMirror>
__device__ __forceinline__ void mt_load(uint32_t *st, const uint32_t *__restrict__ src, int lane) {
  constexpr int kLoads = (kMtN + kWave - 1) / kWave;
  uint32_t v[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) v[i] = src[i + 1 < kLoads ? i * kWave + lane : min(i * kWave + lane, kMtN - 1)];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int at = i * kWave + lane;
    if (i + 1 == kLoads) asm volatile("" : "+v"(v[i]));  // (else its load goes behind the others' wait, to the lanes that store it)
    if (at < kMtN) st[at] = v[i];
    if (at < kMirror) st[kMtN + at] = v[i];
  }
}

// Seeds 64 generators at once, lane l the stream std::mt19937{lane_seed}, and stores the states of
// the first n_streams of them at dst[l * 624 .. + 624).  The 623-step recurrence of the 64 streams
// advances in lock step on the vector unit (a few dozen instructions per stream instead of the
// scalar unit's 3,100 for one); every eight steps the words pass through `tile` (LDS of the calling
// wave, four pairs of words apart) so that they leave as 32-byte runs per stream instead of 4-byte words 2,496
// bytes apart.  (Plain stores: the states are read back soon, by waves of the same workgroup, and do
// best when they stay in the L2; with nontemporal stores and loads the 1e6-row walk took 3.6 instead
// of 3.1 ms.)  `dst` is wave uniform: the stores take it as a buffer whose lane offset never changes.
constexpr int kMtSeedPairStride = 160;  // words from a pair of words of the 64 streams to the next: neighbours in other banks
constexpr int kMtSeedTileWords = 3 * kMtSeedPairStride + 2 * kWave;

// The first n_streams are stored.  Otherwise than SOON: a branch around every store of a batch of fewer than 64: 78 * 4 of them,
// 12.5 to 15 us a batch for a wave alone.  SOON: by a buffer that ends with the last one's state (the hardware leaves out what
// lies behind it), and three rounds to a turn of the loop: 8.6 us (10.1 with one round; the recurrence alone takes 5.3), for
// batches that are waited for.  (Where batch after batch is seeded beside waves that walk, throughput counts, and the branches
// are the better form: column walk of 1,000,000 streams of 18 synapses with the row walk 1,907 us, without them 1,945.)
template <bool SOON = false>
__device__ __forceinline__ void mt_seed_batch(uint32_t *tile, int lane, uint32_t lane_seed, uint32_t *dst,
                                              uint32_t n_streams = kWave) {
  typedef uint32_t Pair __attribute__((ext_vector_type(2)));
  uint32_t x = lane_seed;
  const uint32_t sub = static_cast<uint32_t>(lane) >> 2, pair = static_cast<uint32_t>(lane) & 3u;  // stream within 16, word pair
  Pair *const put = reinterpret_cast<Pair *>(tile) + lane;
  const Pair *const get = reinterpret_cast<const Pair *>(tile) + (pair * (kMtSeedPairStride / 2) + sub);
  const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
      dst, 0, static_cast<int>(SOON ? n_streams * (kMtN * 4u) : kWave * kMtN * 4u), 0x00027000);
  // (streams 16 q + sub; the 16 q are added on the scalar unit, but where they have to count in the lane's offset)
  constexpr uint32_t kRow16 = 16u * kMtN * 4u;
  const uint32_t lane_offset = (sub * kMtN + 2u * pair) * 4u;
  auto store = [&](uint32_t q, uint32_t w0, Pair v) {  // streams 16 q + sub: words w0 + 2 pair, + 1
    if (!SOON && !(16u * q + sub < n_streams)) return;
    __builtin_amdgcn_raw_buffer_store_b64(v, out, static_cast<int>(lane_offset + (SOON ? kRow16 * q : 0u)),
                                          static_cast<int>(SOON ? w0 * 4u : (16u * q * kMtN + w0) * 4u), 0);
  };
  // The words of a tile are read back from LDS at the end of a round and stored at the start of the next
  // one, behind its eight steps of the recurrence, so that the chain of multiplications does not wait for
  // the LDS (a wave's LDS operations complete in order: the next round's writes cannot overtake the reads).
  Pair v[4];
#pragma unroll (SOON ? 3 : 1)
  for (uint32_t w0 = 0; w0 < kMtN; w0 += 8) {
#pragma unroll
    for (uint32_t i = 0; i < 8; i += 2) {  // words w0 + i and w0 + i + 1 of stream `lane`
      Pair p;
      p.x = x;
      p.y = 1812433253u * (p.x ^ (p.x >> 30)) + (w0 + i + 1);
      put[i / 2 * (kMtSeedPairStride / 2)] = p;
      x = 1812433253u * (p.y ^ (p.y >> 30)) + (w0 + i + 2);
    }
    __builtin_amdgcn_wave_barrier();
    if (w0 != 0) {
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) store(q, w0 - 8u, v[q]);
    }
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) v[q] = get[16u * q];
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) store(q, kMtN - 8u, v[q]);
}

// gfx950 evaluates any function of three words bit by bit in one instruction; 0x6c is (a & c) ^ b,
// 0x96 is a ^ b ^ c (the compiler finds the first only now and then).
__device__ __forceinline__ uint32_t and_xor(uint32_t a, uint32_t c, uint32_t b) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x6c);
}

__device__ __forceinline__ uint32_t mt_twist(uint32_t a, uint32_t b, uint32_t c) {
  // y = (a & 0x80000000) | (b & 0x7fffffff) in one bit-field insert (the compiler makes two instructions of it)
  uint32_t y;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(y) : "s"(0x7fffffffu), "v"(b), "v"(a));
  const uint32_t odd = static_cast<uint32_t>(-static_cast<int32_t>(b & 1u));  // all ones when y is odd
  return and_xor(odd, 0x9908b0dfu, c) ^ (y >> 1);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y) {
  y ^= y >> 11;
  y = and_xor(y << 7, 0x9d2c5680u, y);
  y = and_xor(y << 15, 0xefc60000u, y);
  y ^= y >> 18;
  return y;
}

// Produces the next K * NL words of the stream; lane l < NL receives words
// K*l .. K*l + K-1 of them (tempered) in w[].  `pos` is the state slot of the first new word
// (wave uniform, < 624) and is advanced.  Word kRaw of each lane's is left untempered.
//
// A lane reads the K + 1 old words from its first slot s on and the K words from slot
// (s + 397) mod 624 on, and writes K new words from s on.  With the words that follow the 624th repeated
// (kMirror), all three runs are contiguous, and only a batch that touches the first kMirror words or runs past
// the 624th (wave-uniform tests on `pos`) has copies to keep equal.
//
// `base` is mt_base<K, NL, kMirror>(st, lane): the state, at the lane's first word of it where the addresses of a batch do
// not wrap lane by lane.
typedef __attribute__((address_space(3))) uint32_t LdsWord;
typedef uint32_t LdsPair __attribute__((ext_vector_type(2)));
template <int K, int NL, int kMirror>
__device__ __forceinline__ LdsWord *mt_base(uint32_t *st, int lane) {
  if (kMirror < K * NL) return (LdsWord *)st;
  LdsWord *p = (LdsWord *)(st + K * lane);
  asm volatile("" : "+v"(p));  // (else it is split up again and added in every batch)
  return p;
}
template <int K, int NL, int kMirror, int kRaw = -1>
__device__ __forceinline__ void mt_generate(LdsWord *base, uint32_t &pos, int lane, uint32_t (&w)[K]) {
  constexpr uint32_t kSpan = static_cast<uint32_t>(K * NL);
  static_assert(K >= 1 && K <= kMtLeastMirror && kSpan <= 227, "words per lane and batch");
  constexpr bool kLinear = kMirror >= static_cast<int>(kSpan);  // (a batch's addresses need not wrap lane by lane)
  if (NL == kWave || lane < NL) {
    LdsWord *near_at, *far_at;
    if constexpr (kLinear) {
      near_at = base + pos;
      far_at = base + (pos + kMtM < kMtN ? pos + kMtM : pos + kMtM - kMtN);
    } else {
      uint32_t s = pos + static_cast<uint32_t>(K * lane);
      s = min(s, s - kMtN);  // (unsigned: s - 624 wraps to a huge value while s < 624)
      uint32_t f = s + kMtM;
      f = min(f, f - kMtN);
      near_at = base + s, far_at = base + f;
    }
    uint32_t near_[K + 1], far_[K], fresh[K];
    // (Two words a lane: `pos` is even, the pairs lie at multiples of 8 bytes and pass in one operation each; as two
    // operations on every other word they would take twice the time of the LDS.)
    constexpr bool kPairs = K == 2 && kLinear;
    if constexpr (kPairs) {
      const LdsPair a = *(const __attribute__((address_space(3))) LdsPair *)near_at;
      near_[0] = a.x, near_[1] = a.y, near_[K] = near_at[K];
    } else {
#pragma unroll
      for (int i = 0; i <= K; ++i) near_[i] = near_at[i];
    }
#pragma unroll
    for (int i = 0; i < K; ++i) far_[i] = far_at[i];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      fresh[i] = mt_twist(near_[i], near_[i + 1], far_[i]);
      w[i] = i == kRaw ? fresh[i] : mt_temper(fresh[i]);
    }
    auto put = [&](LdsWord *at, int i0, int n) {
      if constexpr (kPairs) {
        *(__attribute__((address_space(3))) LdsPair *)at = LdsPair{fresh[0], fresh[1]};
      } else {
#pragma unroll
        for (int i = i0; i < i0 + n; ++i) at[i] = fresh[i];
      }
    };
    put(near_at, 0, K);
    if constexpr (kLinear) {
      constexpr int kStep = kPairs ? 2 : 1;  // (a pair lies on one side)
      if (pos + kSpan > static_cast<uint32_t>(kMtN)) {
        LdsWord *const low = near_at - kMtN;
#pragma unroll
        for (int i = 0; i < K; i += kStep) {
          if (lane >= static_cast<int>((kMtN - pos - i + K - 1) / K)) put(low, i, kStep);
        }
      } else if (pos < static_cast<uint32_t>(kMirror)) {
#pragma unroll
        for (int i = 0; i < K; i += kStep) {
          if (lane < static_cast<int>((kMirror - pos - i + K - 1) / K)) put(near_at + kMtN, i, kStep);  // (what the mirror repeats)
        }
        __builtin_amdgcn_wave_barrier();  // (keeps the stores of the two branches from being made one behind both)
      }
    } else if (pos < static_cast<uint32_t>(kMirror) || pos + kSpan > static_cast<uint32_t>(kMtN)) {
      uint32_t s = pos + static_cast<uint32_t>(K * lane);
      s = min(s, s - kMtN);
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const uint32_t a = s + i;
        if (a >= kMtN) near_at[i - kMtN] = fresh[i];
        else if (a < static_cast<uint32_t>(kMirror)) near_at[i + kMtN] = fresh[i];
      }
    }
  }
  pos += kSpan;
  if (pos >= kMtN) pos -= kMtN;
}

// libstdc++ generate_canonical<double,53>(mt19937): low word first, the 64-bit sum rounded once
// to double, scaled by 2^-64, clamped below 1.
__device__ __forceinline__ double canonical_f64(uint32_t lo, uint32_t hi) {
  const double s = __dadd_rn(static_cast<double>(lo), __dmul_rn(static_cast<double>(hi), 4294967296.0));
  const double r = s * 0x1p-64;  // exact scaling
  return r >= 1.0 ? 0x1.fffffffffffffp-1 : r;  // nextafter(1, 0)
}

// libstdc++ generate_canonical<float,24>(mt19937): one word rounded to float, scaled by 2^-32, and a
// result of 1 replaced by nextafterf(1, 0).  The word rounds up to 2^32 from 0xffffff80 on, and every
// word from 0xffffff00 to 0xffffff7f rounds to 0xffffff00 = nextafterf(1, 0) * 2^32: capping the WORD
// at 0xffffff7f gives the same floats with one integer minimum instead of a compare and a select.
__device__ __forceinline__ float canonical_f32_scaled(uint32_t word) {  // canonical * 2^32
  return static_cast<float>(min(word, 0xffffff7fu));
}
__device__ __forceinline__ float canonical_f32(uint32_t word) { return canonical_f32_scaled(word) * 0x1p-32f; }

// (unsigned int) of a double as x86-64 compiles it: truncate to int64, keep the low 32 bits;
// out of range and NaN give 0.
__device__ __forceinline__ uint32_t f64_to_u32_x86(double x) {
  if (x >= 0.0 && x < 4294967296.0) return static_cast<uint32_t>(x);  // the only case seen in practice
  if (!(x > -9223372036854775808.0 && x < 9223372036854775808.0)) return 0u;
  return static_cast<uint32_t>(static_cast<uint64_t>(static_cast<long long>(x)));
}

// Parameters of the skip computation, derived from log_p by the launchers (a kernel argument).
//
// q + 1 = log2(U) * inv_log2 + 1 is formed in fixed point by one fused multiply-add: with 3/2 * 2^20 added, the
// low word of the double is the fraction in units of 2^-32 and the low 19 bits of the high one are the integer part,
// so that its fraction is tested by one comparison of words and truncated by one AND (with v_fract_f64, a subtraction,
// a comparison of doubles and a conversion: four instructions of the vector unit's slower half instead of two, one of them
// of its faster).  Skips that may be longer than 19 bits (conn_prob under 8.5e-5): 3/2 * 2^33 instead, 19 bits of fraction.
// The band within `guard` of an integer, where the exact path decides, begins at fraction 0 of q + 1 + guard.
constexpr double kSkipFixed = 0x1.8p20, kSkipFixedWide = 0x1.8p33;
constexpr uint32_t kSkipIntegerMask = (1u << 19) - 1u;
struct SkipParams {
  double log_p;      // log(1 - p)
  double inv_log2;   // ln(2) / log_p: skip = ceil(log2(U) * inv_log2)
  double offset;     // 1 - 32 * inv_log2 (the fast path works on log2(U * 2^32) and truncates instead of ceil()) + guard + 3/2 * 2^k
  uint32_t band;     // the fast path is trusted from this fraction on (never 0: q = inf has fraction 0)
  double close_offset;  // the same for the close path, which needs the smaller band close_band
  uint32_t close_band;
  double quick_offset;  // the same for the quick path
  uint32_t quick_band;
  bool quick;        // the quick path is worth trying
  bool narrow;       // every skip fits 19 bits
};

// Error of the fast path's log2(U): U * 2^32 is formed in fp32 from the two words (two roundings,
// 2^-23 relative, 1.72e-7 on the logarithm) and the hardware fp32 log2 of its mantissa in [0.5, 1) is
// documented to 1 ulp, 2^-24 = 5.96e-8 on a result in [-1, 0] (bpl_selfcheck_jitconn_skips measures
// it over all 2^23 mantissas): 2.32e-7 together, the rest is margin.
constexpr double kSkipLog2Error = 3e-7;

// Quick path: log2(U) from the upper word alone, at least kQuickMin, and without the split into exponent and
// mantissa.  The lower word left out, at most 2^-22 relative: up to 3.44e-7 too little on the logarithm, so half of it
// is added and 1.72e-7 remains on either side; the upper one rounded to fp32
// (2^-24 relative): 0.86e-7; the hardware log2 of a value in [2^-10, 1), 1 ulp of a result of at most 10 in size: 9.54e-7
// (measured over all of them by bpl_selfcheck_jitconn_skips); together 1.212e-6, the rest is margin.  It saves
// 13 of 22 instructions, the tempering of the lower word among them, wherever all of a batch's draws can be trusted: at
// conn_prob 0.001 in 80 % of the batches (row walk of 1e6 streams of 1,000 synapses: 2,060 -> 1,998 us; 1e5 streams of
// 1,000 with conn_prob 0.03: 236 -> 215 us, uniform weights 303 -> 279).  Normal weights have tempered both words of a unit
// and the upper one as a float for the polar attempt: 6 instructions instead of 14.
constexpr double kQuickLog2Error = 1.4e-6, kQuickLog2Short = 1.72e-7;
constexpr uint32_t kQuickMin = 1u << 22;
// Above this guard (conn_prob below about 3e-4) more than half of the batches would take the fast path after it.
constexpr double kQuickGuardMax = 0.004;

// Error of the close path's log2(U): 64-bit arithmetic (a few 1e-15) and a series cut off at 2e-14; the rest is margin.
constexpr double kCloseLog2Error = 1e-12;

inline SkipParams make_skip_params(double log_p) {
  SkipParams sp;
  sp.log_p = log_p;
  sp.inv_log2 = 0.6931471805599453094 / log_p;
  // The quotient is off by at most kSkipLog2Error * |inv_log2| plus fp64 rounding and, in fixed point, the rounding of the
  // offset and of the multiply-add (half a unit of the fraction each); inside that band
  // around an integer the exact path decides.  Quotients that could leave the range of uint32
  // (log2(U) >= -64): always the exact path, which converts as x86-64 does.
  const double size = std::fabs(sp.inv_log2);
  sp.narrow = size * 64.0 + 2.0 < 524288.0;
  const double rounding = sp.narrow ? 1e-9 : 0x1p-18;
  double guard = kSkipLog2Error * size + rounding, close_guard = kCloseLog2Error * size + rounding;
  if (!(size * 64.0 + 2.0 < 4.0e9)) guard = close_guard = 1.0;
  sp.offset = 1.0 - 32.0 * sp.inv_log2 + guard + (sp.narrow ? kSkipFixed : kSkipFixedWide);
  sp.band = static_cast<uint32_t>(std::fmin(std::ceil(guard * 0x1p33), 4294967295.0));
  sp.close_offset = 1.0 + close_guard + (sp.narrow ? kSkipFixed : kSkipFixedWide);
  sp.close_band = static_cast<uint32_t>(std::fmin(std::ceil(close_guard * 0x1p33), 4294967295.0));
  const double quick_guard = kQuickLog2Error * size + 1e-9;
  sp.quick_offset = 1.0 + kQuickLog2Short * sp.inv_log2 + quick_guard + kSkipFixed;
  sp.quick_band = static_cast<uint32_t>(std::fmin(std::ceil(quick_guard * 0x1p33), 4294967295.0));
  sp.quick = sp.narrow && quick_guard < kQuickGuardMax;
  return sp;
}

// One geometric skip: (unsigned) ceil(log(U) / log_p)  (lib/cpu_jitconn_event_matvec.cpp:24),
// U = canonical double of two generator words (low word first).
//
// Exact path: fp64 log and IEEE division, as the CPU code.
__device__ __forceinline__ uint32_t skip_exact(uint32_t lo, uint32_t hi, const SkipParams &sp) {
  return f64_to_u32_x86(ceil(log(canonical_f64(lo, hi)) / sp.log_p));
}

// A quotient in fixed point: its integer part, and the lanes whose fraction lies in the band.
__device__ __forceinline__ uint32_t fixed_skip(double z, bool narrow, uint32_t band, uint64_t &unsafe) {
  const uint32_t z_lo = static_cast<uint32_t>(__double2loint(z)), z_hi = static_cast<uint32_t>(__double2hiint(z));
  unsafe = __builtin_amdgcn_ballot_w64((narrow ? z_lo : z_lo << 13) < band);
  return narrow ? z_hi & kSkipIntegerMask : __builtin_amdgcn_alignbit(z_hi, z_lo, 19);
}

// Fast path: log2(U * 2^32) = exponent + v_log_f32(mantissa) of the fp32 value of the two words, one
// fused multiply-add to q + 1 = log2(U) * inv_log2 + 1, truncation.  `unsafe`: the lanes where q is within the guard
// of an integer, i.e. where a rounding of the exact path could land on another ceil() (or q = inf, U = 0).
__device__ __forceinline__ uint32_t skip_fast(uint32_t lo, uint32_t hi, const SkipParams &sp, uint64_t &unsafe) {
  const float f = fmaf(static_cast<float>(lo), 0x1p-32f, static_cast<float>(hi));
  int e;
  const float m = frexpf(f, &e);  // f = m * 2^e, m in [0.5, 1)
  const double l2 = static_cast<double>(e) + static_cast<double>(__log2f(m));
  return fixed_skip(fma(l2, sp.inv_log2, sp.offset), sp.narrow, sp.band, unsafe);
}

// A constant made where it is used: the compiler keeps those of a rarely taken path in registers of the whole loop.
constexpr uint64_t bits_of(double v) { return __builtin_bit_cast(uint64_t, v); }
template <uint64_t kBits>
__device__ __forceinline__ double scalar_constant() {
  int lo, hi;
  asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "n"(static_cast<uint32_t>(kBits)));
  asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "n"(static_cast<uint32_t>(kBits >> 32)));
  return __hiloint2double(hi, lo);
}

// Close path: where the fast one cannot decide, log2(U) in 64 bits to about 1e-14, from the series of the inverse
// hyperbolic tangent (log m = 2 artanh((m - 1) / (m + 1)), m within sqrt(1/2) .. sqrt(2)).  A third of the exact path's
// instructions, which then is left with a draw in 10^8; the share of the batches that come here is 2.7 % at conn_prob 0.001
// (1,000,000 streams of 1,000 synapses: 1,597 -> 1,551 us) and a quarter at 0.0001.
__device__ __forceinline__ uint32_t skip_close(uint32_t lo, uint32_t hi, const SkipParams &sp, uint64_t &unsafe) {
  const double u = fma(static_cast<double>(hi), 0x1p32, static_cast<double>(lo));
  int e;
  double m = frexp(u, &e);  // u = m * 2^e, m in [0.5, 1)
  const bool low = m < scalar_constant<bits_of(0.70710678118654752)>();
  m = low ? m + m : m;
  e -= low ? 65 : 64;
  // 1 / (m + 1): the hardware's approximation (2^-24) and one Newton step
  const double d = m + 1.0, r0 = __builtin_amdgcn_rcp(d), r = fma(fma(-d, r0, 1.0), r0, r0);
  const double t = (m - 1.0) * r, t2 = t * t;
  double s = scalar_constant<bits_of(1.0 / 15.0)>();
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 13.0)>());
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 11.0)>());
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 9.0)>());
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 7.0)>());
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 5.0)>());
  s = fma(s, t2, scalar_constant<bits_of(1.0 / 3.0)>());
  s = fma(s, t2, 1.0);
  const double l2 = fma(t * scalar_constant<bits_of(2.885390081777926815)>(), s, static_cast<double>(e));  // 2 / ln 2
  const uint32_t skip = fixed_skip(fma(l2, sp.inv_log2, sp.close_offset), sp.narrow, sp.close_band, unsafe);
  unsafe |= __builtin_amdgcn_ballot_w64((lo | hi) == 0u);  // (the series knows no infinity)
  return skip;
}

// `upper`: `hi` as a float, or that of `hi` capped at 0xffffff7f (canonical_f32_scaled), which is 2^-24 too little at most.
__device__ __forceinline__ uint32_t skip_quick(uint32_t hi, float upper, const SkipParams &sp, uint64_t &unsafe) {
  const float l2 = __builtin_amdgcn_logf(upper * 0x1p-32f);
  const double z = fma(static_cast<double>(l2), sp.inv_log2, sp.quick_offset);
  const uint32_t skip = fixed_skip(z, true, sp.quick_band, unsafe);
  unsafe |= __builtin_amdgcn_ballot_w64(hi < kQuickMin);
  return skip;
}

// If any lane of the wave is inside the band, the whole wave takes the next path (wave-uniform
// branches): the fast, the close and the exact one.  Only the lanes in `needed` have to be right.  kQuick: the quick path is
// tried first.  kTempered: `lo` is a word of the stream; else it is still to be tempered.
// `upper`: see skip_quick.
template <bool kQuick, bool kTempered>
__device__ __forceinline__ uint32_t skip_from_words(uint32_t lo, uint32_t hi, float upper, const SkipParams &sp,
                                                    uint64_t needed = ~0ull) {
  uint64_t unsafe;
  if (kQuick && sp.quick) {
    const uint32_t quick = skip_quick(hi, upper, sp, unsafe);
    if ((unsafe & needed) == 0) return quick;
  }
  if (!kTempered) lo = mt_temper(lo);
  const uint32_t fast = skip_fast(lo, hi, sp, unsafe);
  if ((unsafe & needed) == 0) return fast;
  const uint32_t close = skip_close(lo, hi, sp, unsafe);
  if ((unsafe & needed) == 0) return close;
  return skip_exact(lo, hi, sp);
}
template <bool kQuick, bool kTempered>
__device__ __forceinline__ uint32_t skip_from_words(uint32_t lo, uint32_t hi, const SkipParams &sp, uint64_t needed = ~0ull) {
  return skip_from_words<kQuick, kTempered>(lo, hi, static_cast<float>(hi), sp, needed);
}

}  // namespace bpl
