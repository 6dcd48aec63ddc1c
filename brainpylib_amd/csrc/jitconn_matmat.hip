// jitconn matmat for gfx950:  Y[m,n] = X[m,k] @ M[k,n],  M regenerated on the fly.
//
// Column j of M is generator stream std::mt19937{seed + j} walked over the k inputs, the same
// stream the matvec operators use for output j with transpose=True, so that
// matmat(X)[i,:] == matvec(X[i,:], transpose=True) -- the identity the reference's tests assert
// (brainpylib/_src/jitconn_ops/tests/matmat_testcase.py:133-138).
//
// The reference kernel (lib/gpu_jitconn_matmat.cu:236-276) gives each thread a few rows of X for
// one column and reads X[row*k + id] with unrelated ids in neighbouring threads.  Here one
// wave64 owns a column: X is first transposed into a scratch buffer XT[k][m] (rows padded to a
// multiple of 64), then for every synapse (id, w) of the column the wave reads the contiguous
// row XT[id][0..m) and each lane accumulates its own output rows, in stream order, with the same
// multiply-then-add the CPU path performs.  The synapses of a batch pass from the lanes that drew
// them to the whole wave through LDS (one broadcast read each).
//
// Reference boundary: lib/gpu_jitconn_matmat.cu:279-317,364-455 (buffers = [X, Y], descriptor
// MatMatJITProbDescriptor1, target names lib/gpu_ops.cc:161-174).
#include "common.h"
#include "jitconn_stream.h"
#include "targets.h"

namespace bpl {
namespace {

constexpr int kTile = 32;

constexpr int kPrepareThreads = kTile * 8;
constexpr uint32_t kPrepareGroups = 1u << 22;  // workgroups that transpose, at most

// XT[r / pass_rows][c][r % pass_rows] = X[r][c] for r < m: the transposed operand in slices of pass_rows rows of
// X (a multiple of 32), every slice contiguous, its rows pass_rows entries long; rows m .. m_pad - 1 are zero.
// (In one array of rows of m_pad entries the pieces that a pass reads lie m_pad entries apart and share a
// fraction of the L2's sets.)
// Float64: 64 rows at a time, the low words of the 64 and then the high words, for the walk reads XT word by word.
// The first seed_groups workgroups do not transpose: one wave of each seeds the generators of 64 of the `count` columns,
// which it does in 8.6 us, beside the transposition (128 x 10,000: the launch takes 12.5 us, without the seeding 6.1).
// The others take the tiles in turn: a launch has fewer than 2^32 threads, an X of 2^34 entries as many tiles as 2^32 threads.
template <typename T>
__global__ __launch_bounds__(kPrepareThreads) void matmat_prepare_kernel(const T *__restrict__ X, T *__restrict__ XT,
                                                                         uint32_t m, uint32_t k, uint32_t m_pad,
                                                                         uint32_t pass_rows, uint32_t col_tiles, uint32_t tiles,
                                                                         uint32_t seed, uint32_t count,
                                                                         uint32_t seed_groups,
                                                                         uint32_t *__restrict__ states) {
  constexpr size_t kTileBytes = sizeof(T) * kTile * (kTile + 1), kSeedBytes = sizeof(uint32_t) * kMtSeedTileWords;
  __shared__ __attribute__((aligned(16))) unsigned char s_mem[kTileBytes > kSeedBytes ? kTileBytes : kSeedBytes];
  if (blockIdx.x < seed_groups) {
    const uint32_t base = blockIdx.x * kWave;
    const int lane = lane_id();
    if (threadIdx.x < kWave)
      mt_seed_batch<true>(reinterpret_cast<uint32_t *>(s_mem), lane, seed + base + static_cast<uint32_t>(lane),
                          states + static_cast<size_t>(base) * kMtN,
                          count - base < static_cast<uint32_t>(kWave) ? count - base : static_cast<uint32_t>(kWave));
    return;
  }
  T(*tile)[kTile + 1] = reinterpret_cast<T(*)[kTile + 1]>(s_mem);
  const uint32_t tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;  // 32 x 8
  for (uint32_t at = blockIdx.x - seed_groups;;) {
    const uint32_t c0 = at % col_tiles * kTile, r0 = at / col_tiles * kTile;
    for (uint32_t i = ty; i < kTile; i += 8) {
      const uint32_t r = r0 + i, c = c0 + tx;
      tile[i][tx] = (r < m && c < k) ? X[static_cast<size_t>(r) * k + c] : T(0);
    }
    __syncthreads();
    for (uint32_t i = ty; i < kTile; i += 8) {
      const uint32_t c = c0 + i, r = r0 + tx;
      if (c < k && r < m_pad) {
        constexpr uint32_t kWords = sizeof(T) / 4;
        uint32_t *to = reinterpret_cast<uint32_t *>(XT + (static_cast<size_t>(r / pass_rows) * k + c) * pass_rows) +
                       r % pass_rows / kWave * (kWave * kWords) + r % kWave;
        uint32_t w[kWords];
        __builtin_memcpy(w, &tile[tx][i], sizeof(T));
#pragma unroll
        for (uint32_t part = 0; part < kWords; ++part) to[part * kWave] = w[part];
      }
    }
    at += gridDim.x - seed_groups;
    if (at >= tiles) break;
    __syncthreads();  // the tile is read
  }
}

__device__ __forceinline__ float mul_rn(float a, float b) { return __fmul_rn(a, b); }
__device__ __forceinline__ double mul_rn(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ float add_rn(float a, float b) { return __fadd_rn(a, b); }
__device__ __forceinline__ double add_rn(double a, double b) { return __dadd_rn(a, b); }

// one synapse of a batch: where its row of XT starts (bytes) and its weight
template <typename T1>
struct __attribute__((aligned(2 * sizeof(T1)))) Synapse {
  uint32_t off;
  T1 w;
};

// MT = 64-row tiles of Y one wave accumulates; a launch is one pass over MT * 64 rows of X (pass number `pass`).
// (The passes are launches of their own, one after the other: as the second dimension of one grid the
// workgroups of two passes run side by side nearly all the time, two slices of XT compete for the L2s, and
// eight passes of 256 rows took 5.7 ms instead of 3.8.)
template <typename T1, int W, int MT>
__global__ __launch_bounds__(256) void jitconn_matmat_kernel(const T1 *__restrict__ XT, T1 *__restrict__ Y,
                                                             uint32_t m, uint32_t k, uint32_t n, uint32_t m_pad,
                                                             uint32_t seed, SkipParams skips, T1 wa, T1 wb,
                                                             uint32_t first, uint32_t count,
                                                             const uint32_t *__restrict__ states, uint32_t pass) {
  constexpr int kWaves = 4;
  constexpr int kStreamWords = StreamLds<T1, W>::words;
  __shared__ __attribute__((aligned(8))) uint32_t s_state[kWaves * kStreamWords];
  constexpr int kSlots = W == kNormal ? 2 * kWave : kWave;  // normal weights come two to a lane
  __shared__ __attribute__((aligned(16))) Synapse<T1> s_syn[kWaves * kSlots];
  const int lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  uint32_t *st = s_state + wave * kStreamWords;
  Synapse<T1> *syn = s_syn + wave * kSlots;
  const uint32_t row_base = pass * (MT * kWave);  // first row of Y of this pass
  // The walk is bound by these reads, 512 bytes per synapse and pass of 128 float32 rows, at 27 of the 33 TB/s that 64 bytes
  // per clock and CU come to, with the vector issue (0.6 of its rate) beside them.  A load takes the wave-uniform byte offset
  // of a row of the slice (32 bits, checked by the host), an immediate one, and four times the lane, which the buffer's
  // descriptor adds (stride 4, thread number enabled): no address arithmetic per synapse, one instruction less, 6.9 now: 10,000 x
  // 10,000 of 1,000 synapses x 128 203 -> 200 us, 1,000 x 200,000 of 20 396 -> 390.  Loads of 4 bytes a lane reach that
  // rate; of 8 bytes 17.6 TB/s, as they did the float64 rows before these were stored as two words apart (5,000 x 10,000 of
  // 250 x 100: 166 -> 124 us; with 16 bytes a lane 124 too, but there 64 rows are half a wave) and float32 rows of 128 as pairs (300 us).
  constexpr uint32_t kWords = sizeof(T1) / 4;
  constexpr uint32_t row_bytes = MT * kWave * static_cast<uint32_t>(sizeof(T1));
  const __amdgpu_buffer_rsrc_t slice = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T1 *>(XT + static_cast<size_t>(pass) * k * (MT * kWave)), 4, static_cast<int>(k * row_bytes), 0x00807000);
  auto load = [&](uint32_t off, uint32_t t) {  // tile t of the row at byte `off`: the lane's entry
    uint32_t w[kWords];
#pragma unroll
    for (uint32_t i = 0; i < kWords; ++i)
      w[i] = __builtin_amdgcn_raw_buffer_load_b32(slice, static_cast<int>(off + (t * kWords + i) * kWave * 4), 0, 0);
    T1 x;
    __builtin_memcpy(&x, w, sizeof(T1));
    return x;
  };
  // columns first .. first + count - 1 of M; states[c]: the generator of column first + c, if they are seeded ahead
  for (uint32_t c = blockIdx.x * kWaves + wave; c < count; c += gridDim.x * kWaves) {
    const uint32_t j = first + c;
    T1 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = T1(0);
    const uint32_t *pre = states != nullptr ? states + static_cast<size_t>(c) * kMtN : nullptr;
    // Every valid lane leaves its synapses (the byte offset of their rows of XT, their weights) in the
    // wave's LDS slots, in lane order (which is stream order); every lane then reads the slots
    // one after the other (one address per read: a broadcast), so a synapse costs one LDS read,
    // its loads and MT multiply-adds, with U synapses' loads in flight.
    auto take = [&](uint32_t count) {
      constexpr int U = 8;
      uint32_t i = 0;
      for (; i + U <= count; i += U) {
        T1 ws[U];
        T1 x[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const Synapse<T1> e = syn[i + u];
          ws[u] = e.w;
#pragma unroll
          for (int t = 0; t < MT; ++t) x[u][t] = load(e.off, t);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t] = add_rn(acc[t], mul_rn(ws[u], x[u][t]));
        }
      }
      for (; i < count; ++i) {
        const Synapse<T1> e = syn[i];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = add_rn(acc[t], mul_rn(e.w, load(e.off, t)));
      }
    };
    auto put = [&](uint32_t slot, uint32_t idx, T1 w) {
      syn[slot].off = idx * row_bytes;
      syn[slot].w = w;
    };
    if constexpr (W == kNormal) {
      walk_stream<T1, W, true>(st, lane, seed + j, pre, k, skips, wa, wb,
                         [&](uint32_t idx0, T1 w0, bool valid0, uint32_t idx1, T1 w1, bool valid1) {
        __builtin_amdgcn_wave_barrier();  // the reads of the batch before are done
        if (valid0) {
          put(2u * static_cast<uint32_t>(lane), idx0, w0);
          put(2u * static_cast<uint32_t>(lane) + 1u, idx1, w1);  // (not counted where only the first is valid)
        }
        __builtin_amdgcn_wave_barrier();
        take(static_cast<uint32_t>(__popcll(__ballot(valid0)) + __popcll(__ballot(valid1))));
      });
    } else {
      walk_stream<T1, W, true>(st, lane, seed + j, pre, k, skips, wa, wb, [&](uint32_t idx, T1 w, bool valid, bool) {
        __builtin_amdgcn_wave_barrier();
        if (valid) put(static_cast<uint32_t>(lane), idx, w);
        __builtin_amdgcn_wave_barrier();
        take(static_cast<uint32_t>(__popcll(__ballot(valid))));
      });
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const uint32_t r = row_base + t * kWave + lane;
      if (r < m) Y[static_cast<size_t>(r) * n + j] = acc[t];
    }
  }
}

template <typename T1, int W>
void matmat_entry(const char *target, hipStream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  bpl_matmat_jit_prob_descriptor d;
  if (!unpack(target, opaque, opaque_len, &d)) return;
  if (!(d.log_p < 0.0) || std::isinf(d.log_p)) {
    set_error("%s: log_p must be finite and negative (conn_prob in (0, 1]), got %g", target, d.log_p);
    return;
  }
  if (buffers == nullptr) {
    set_error("%s: null buffer table", target);
    return;
  }
  const T1 *X = static_cast<const T1 *>(buffers[0]);
  T1 *Y = static_cast<T1 *>(buffers[1]);
  const uint32_t m = d.m, k = d.k, n = d.n;
  if (m == 0 || n == 0) return;
  // rows of X are padded to what the passes of the kernel read: one pass of 64 or 128 rows, or several of 128.
  // (A pass regenerates the matrix, but its slice of XT, 5 MB for 10,000 inputs, stays in the L2s: 2,048 rows of X
  // against a 10,000 x 10,000 matrix take 3.2 ms with uniform and 3.7 ms with normal weights in 16 passes of 128,
  // 3.7 and 3.8 ms in 8 passes of 256, whose slices do not.)
  uint32_t m_pad = (m + kWave - 1) / kWave * kWave;
  const uint32_t pass_rows = m_pad > 2 * kWave ? 2 * kWave : m_pad;
  m_pad = (m + pass_rows - 1) / pass_rows * pass_rows;
  if (k == 0) {
    fill_zero(stream, Y, m * n);  // m * n fits 32 bits whenever Y is addressable by the kernels below
    check_launch(target);
    return;
  }
  if (static_cast<uint64_t>(k) * pass_rows * sizeof(T1) > 0xffffffffull) {
    set_error("%s: a slice of the transposed operand (%u x %u) exceeds 4 GiB", target, k, pass_rows);
    return;
  }
  // scratch memory: [XT][the generator states of a chunk of columns, seeded ahead on the vector unit]
  const size_t xt_bytes = (static_cast<size_t>(k) * m_pad * sizeof(T1) + 255) / 256 * 256;
  // Seeded ahead where a CU has more columns than one workgroup's: its one scalar unit seeds a generator in 1.3 us (and
  // no wave in less than 5), all columns together on the vector units take 8.6 us.  Float32, in place / ahead:
  // 1,000 inputs 1,024 columns 16.3 / 18.4 us, 1,500 21.1 / 19.3, 3,000 26.5 / 20.8; 20,000 inputs of 4 rows, 20,000 columns
  // of 100 synapses 132.7 / 49.4; 10,000 columns of 1,000 synapses 209 / 204, with normal weights 241 / 233.
  const uint32_t chunk = n < kSeedChunk ? n : kSeedChunk;
  const size_t state_bytes = static_cast<size_t>(chunk) * kMtN * sizeof(uint32_t);
  bool ahead = n > 4u * static_cast<uint32_t>(device_info().num_cu);
  // From 32,768 columns on (in place a million columns of 20 synapses take 5.6 ms, ahead 3.3) the states are required;
  // with fewer a call that finds no room for them, a captured one above all, goes on without.
  const bool optional = ahead && n < 32768;
  unsigned char *ws =
      static_cast<unsigned char *>(stream_workspace(stream, xt_bytes + (ahead ? state_bytes : 0), optional));
  if (ws == nullptr && optional) {
    bpl_clear_error();
    ahead = false;
    ws = static_cast<unsigned char *>(stream_workspace(stream, xt_bytes));
  }
  if (ws == nullptr) return;
  T1 *XT = reinterpret_cast<T1 *>(ws);
  uint32_t *states = reinterpret_cast<uint32_t *>(ws + xt_bytes);
  const uint32_t col_tiles = div_up(k, kTile), seed_groups = ahead ? div_up(chunk, kWave) : 0;
  // (an X that fits the device has fewer than 2^32 tiles)
  const uint32_t all_tiles = static_cast<uint32_t>(static_cast<uint64_t>(col_tiles) * div_up(m_pad, kTile));
  hipLaunchKernelGGL(matmat_prepare_kernel<T1>, dim3(seed_groups + (all_tiles < kPrepareGroups ? all_tiles : kPrepareGroups)),
                     dim3(kPrepareThreads), 0, stream, X, XT, m, k, m_pad, pass_rows, col_tiles, all_tiles, d.seed, chunk,
                     seed_groups, states);
  const T1 wa = static_cast<T1>(d.w_a), wb = static_cast<T1>(d.w_b);
  const uint32_t tiles = pass_rows / kWave, passes = m_pad / pass_rows;
  for (uint32_t first = 0; first < n; first += chunk) {
    const uint32_t count = n - first < chunk ? n - first : chunk;
    if (ahead && first != 0) jitconn_seed_streams(stream, d.seed, first, count, states);
    const unsigned grid_x = div_up(count, 4);
    const uint32_t *pre = ahead ? states : nullptr;
    for (uint32_t pass = 0; pass < passes; ++pass) {
      if (tiles == 1) {
        hipLaunchKernelGGL((jitconn_matmat_kernel<T1, W, 1>), dim3(grid_x), dim3(256), 0, stream, XT, Y, m, k, n, m_pad,
                           d.seed, make_skip_params(d.log_p), wa, wb, first, count, pre, pass);
      } else {
        hipLaunchKernelGGL((jitconn_matmat_kernel<T1, W, 2>), dim3(grid_x), dim3(256), 0, stream, XT, Y, m, k, n, m_pad,
                           d.seed, make_skip_params(d.log_p), wa, wb, first, count, pre, pass);
      }
    }
  }
  check_launch(target);
}

}  // namespace
}  // namespace bpl

using namespace bpl;

#define BPL_DEFINE(name, T1, W)                                                                    \
  extern "C" void name(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) { \
    matmat_entry<T1, W>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len);   \
  }

BPL_DEFINE(gpu_matmat_prob_prob_normal_float_v1, float, kNormal)
BPL_DEFINE(gpu_matmat_prob_prob_normal_double_v1, double, kNormal)
BPL_DEFINE(gpu_matmat_prob_prob_uniform_float_v1, float, kUniform)
BPL_DEFINE(gpu_matmat_prob_prob_uniform_double_v1, double, kUniform)
