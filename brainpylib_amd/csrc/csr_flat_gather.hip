// csr_matvec (no transpose) with the dense vector gathered from L2, walked FLAT: every wave owns a contiguous
// range of the nonzeros, whatever rows they belong to, so that every lane of every load and gather carries a
// nonzero.  (A row-wise walk, groups of lanes taking whole rows in steps of 16-byte loads, pads each row to
// whole steps of its group: with 100 nonzeros per row a fifth of the lanes of its gather instructions lie
// beyond the row, and a gather instruction costs the address unit the same whether its lanes are masked or
// not.  That walk took 633 us at 1e8 nonzeros in rows of 100, this one 546; rows of 30: 449 against 315.)
//
// Measured on this device: a product that reads one 4-byte element of a 4 MB vector per nonzero is bound by
// the rate at which a CU's vector cache takes misses (about one 128-byte line per 3.2 clocks and CU, whatever
// the occupancy), and the index and weight streams go through the same cache.  What helps is fewer, wider
// stream requests (every lane loads FOUR consecutive nonzeros, 16 bytes of indices and 16 or 32 of weights,
// per request), the nontemporal hint on the streams, so that the 800 MB that pass through do not push the
// vector out of the L2s, and sixteen gathers in flight per lane.
//
// A wave takes its range in steps of U * 64 quads (1,024 nonzeros of float, 512 of double): 16-byte loads of
// the index and weight streams (nontemporal), sixteen gathers per lane, the products formed in F and widened
// as the reference's CPU loop does (brainpylib/_src/sparse_ops/sparse_csr_matvec.py:116-119).  Which row a
// nonzero belongs to comes from a window of 65 consecutive entries of indptr in LDS, beginning at the row the
// step begins in: a six-step search per quad, then a walk over the quad's four elements.  A lane adds a run of
// elements of one row to that row's float64 accumulator in LDS with one atomic.  Rows that end inside the step
// are stored; the partial sum of the row that is still open moves to accumulator 0 of the next step.  A step
// that meets more than 64 rows (empty rows, very short ones) takes further windows over the same registers.
//
// Rows across the ranges of two or more waves: a wave never stores a row that began before its range; it
// leaves that row's partial sum in head[wave], and the partial sum of the row still open at the end of its
// range in tail[wave] with the row's number.  A second, small kernel adds tail[w] and the heads of the waves
// that follow, as far as their ranges begin within the row, and stores the row.  The arrays hold one entry per wave of
// the launch (the nonzero count is known on the device only; the number of waves is the launcher's).
//
// OUT: what the walk leaves behind.  kFlatSums: y = A x.  kFlatProducts: products[j] = v[row of j] * x[column of j]
// for every nonzero j (the gradient of the weights), stored with the quads' own 16-byte width; the rows of the
// nonzeros are at hand in the window anyway, v's 64 elements of the window lie beside it.  Both at once read the
// indices and gather x once.  Measured: 1e7 nonzeros, both, x of 30,011 floats in LDS: 33 us, 3.6 TB/s of the 120 MB it
// must move; 3e7 nonzeros, products alone, x of 120,011 floats: 122 us, bound by the lines that the gathers move out
// of the L2s (2.7 GB, 54 us without those gathers).  An expanded list of the rows, two gathers and a product as
// passes of their own took 215 and 850 us.
// STAGED: one workgroup of 1,024 threads per CU keeps the first elements of x (139 to 151 KB) in LDS and gathers only the
// rest from L2 (flat_stages()).  Every gather it spares counts: with 147 instead of 138 KB 1,000,000 x 50,000 with 100 per row
// takes 221 instead of 234 us, 200,000 x 50,000 56 instead of 58.
#include <type_traits>

#include "common.h"
#include "csr_flat_gather.h"

namespace bpl {
namespace {

// (aligned to their elements: the arrays may begin anywhere, and a 16-byte load of an address that is not a multiple
// of 16 costs what it touches)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64x2 __attribute__((ext_vector_type(2), aligned(8)));

enum : int { kFlatSums = 1, kFlatProducts = 2 };
// 16 waves per CU either way: two workgroups, or one that has the LDS to itself (STAGED)
constexpr int flat_threads(bool staged) { return staged ? 1024 : 512; }
constexpr unsigned flat_per_cu(bool staged) { return staged ? 1u : 2u; }
constexpr uint32_t kFlatRows = 64;  // rows of an indptr window (one per lane)
// bytes of x in LDS: what the windows, accumulators and v's elements of the 16 waves leave (147 KB beside the sums, 139 to
// 143 beside both)
template <typename F, int OUT>
constexpr uint32_t flat_staged_bytes() {
  const uint32_t sums = (OUT & kFlatSums) ? 16u * kFlatRows * 8u : kFlatRows * 8u;
  const uint32_t v = ((OUT & kFlatProducts) ? 16u : 1u) * (kFlatRows + 1u) * static_cast<uint32_t>(sizeof(F));
  return (160u * 1024u - 16u * (kFlatRows + 2u) * 4u - sums - v - 64u) / 1024u * 1024u;
}
constexpr uint32_t kNoRow = 0xffffffffu;

// quads per lane and step, as many as 128 registers hold (with sums and products of floats at once two as well: the
// elements of x and the weights both live until the rows are known)
template <typename F, int OUT>
struct FlatQuads {
  static constexpr int value = sizeof(F) == 4 && OUT != (kFlatSums | kFlatProducts) ? 4 : 2;
};

// The least a wave takes, in nonzeros and rows: a wavefront of quads.  (The plain sums of x in L2 whole steps: a gather
// costs the address unit the same however many of its lanes hold a nonzero.)
template <typename F, int OUT, bool STAGED>
constexpr uint32_t flat_min_share() {
  return 4u * kWave * ((OUT == kFlatSums && !STAGED) ? FlatQuads<F, OUT>::value : 1);
}

// Four consecutive indices / weights, whole quad q of the array.
__device__ __forceinline__ u32x4 flat_index_quad(const uint32_t *__restrict__ p, uint32_t q) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p) + q);
}
__device__ __forceinline__ void flat_data_quad(const float *__restrict__ p, uint32_t q, float (&v)[4]) {
  const f32x4 t = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p) + q);
  v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
}
__device__ __forceinline__ void flat_data_quad(const double *__restrict__ p, uint32_t q, double (&v)[4]) {
  const f64x2 a = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(p) + 2u * q);
  const f64x2 b = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(p) + 2u * q + 1u);
  v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y;
}
__device__ __forceinline__ void flat_store_quad(float *__restrict__ p, const float (&v)[4]) {
  __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4 *>(p));
}
__device__ __forceinline__ void flat_store_quad(double *__restrict__ p, const double (&v)[4]) {
  __builtin_nontemporal_store(f64x2{v[0], v[1]}, reinterpret_cast<f64x2 *>(p));
  __builtin_nontemporal_store(f64x2{v[2], v[3]}, reinterpret_cast<f64x2 *>(p) + 1);
}

// Where the waves' ranges begin.  Rows and nonzeros are one list, each row's end behind its nonzeros, and a wave takes
// an equal piece of that list: a range balanced by nonzeros alone leaves a long block of empty or nearly empty rows to
// one wave, a window of 64 rows after the other (1,000,000 rows and 5e6 nonzeros, all in the first tenth of the rows: 21 ms,
// now 70 us; 2,000 rows of 20,000 among as many of 0.1: 5.8 ms, now 0.61; the weights' gradient with 100 nonzeros: 26 ms,
// now 80 us).  Even matrices: 0.91 to 1.02 of the time before, 1.05 with doubles of 30,000 columns and ten per row.
// A row's end counts as four nonzeros: 64 empty rows are a window with its dependent load, 2.5 us, where a step of 1,024
// nonzeros takes some 10 (346,000 rows of 870 in the first tenth, x 42,500: 300 us with one, 87 with four or eight; from eight
// on a long row among many of one nonzero per step is the last to end: 988,000 x 116,000 57 -> 66 us, with sixteen 91).
// row, pos: of the first `diag` entries of the list, how many are rows (= the row the next nonzero belongs to or the next
// end is of) and how many nonzeros; two places side by side, 64 probes a round (four rounds for a million rows).
// A place moves back to a multiple of 32 nonzeros (a line of indices) where the row that holds that one is among the
// last round's probes: the loads of a wave then cover whole lines.  (A function of `diag` alone and monotone in it: the
// last round's probes are a fixed division of the rows.)
constexpr uint32_t kFlatRowWeight = 4;
__device__ __forceinline__ uint64_t flat_list(uint32_t n_row, uint32_t nnz) {  // entries of the list
  return static_cast<uint64_t>(kFlatRowWeight) * n_row + nnz;
}
__device__ __forceinline__ void flat_split(const uint32_t *__restrict__ indptr, uint32_t n_row, uint32_t nnz,
                                           const uint64_t (&diag)[2], uint32_t lane, uint32_t (&row)[2],
                                           uint32_t (&pos)[2]) {
  const uint64_t total = flat_list(n_row, nnz);
  uint32_t lo[2] = {0, 0}, first[2], ptr[2];
  uint64_t hi[2] = {n_row, n_row};
  for (uint32_t stride = n_row / kWave + (n_row % kWave ? 1u : 0u);; stride = stride / kWave + (stride % kWave ? 1u : 0u)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint64_t probe = static_cast<uint64_t>(lo[k]) + static_cast<uint64_t>(lane) * stride;
      ptr[k] = probe < hi[k] ? indptr[probe] : 0xffffffffu;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint64_t probe = static_cast<uint64_t>(lo[k]) + static_cast<uint64_t>(lane) * stride;
      const bool below = lane == 0 || (probe < hi[k] && kFlatRowWeight * probe + ptr[k] <= diag[k]);  // (a prefix of the lanes)
      first[k] = lo[k];
      lo[k] += (static_cast<uint32_t>(__popcll(__ballot(below))) - 1u) * stride;
      const uint64_t top = static_cast<uint64_t>(lo[k]) + stride;
      hi[k] = top < hi[k] ? top : hi[k];
    }
    if (stride == 1u) break;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (diag[k] >= total) {
      row[k] = n_row, pos[k] = nnz;
      continue;
    }
    const uint32_t at = lo[k] - first[k];
    uint32_t row_end = at + 1u < kWave ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ptr[k]), at + 1u)) : 0xffffffffu;
    if (row_end == 0xffffffffu) row_end = indptr[lo[k] + 1u];  // (not among the probes)
    const uint64_t p = diag[k] - static_cast<uint64_t>(kFlatRowWeight) * lo[k];
    row[k] = lo[k], pos[k] = p < row_end ? static_cast<uint32_t>(p) : row_end;
    const uint32_t back = pos[k] & ~31u;
    const uint32_t rows = static_cast<uint32_t>(__popcll(__ballot(lane <= at && ptr[k] <= back)));
    if (rows != 0u) row[k] = first[k] + rows - 1u, pos[k] = back;
  }
}

template <typename F, bool HETER, int OUT, bool STAGED>
__global__ __launch_bounds__(flat_threads(STAGED), 4) void csr_flat_gather_kernel(
    const F *__restrict__ data, const uint32_t *__restrict__ indices, const uint32_t *__restrict__ indptr,
    const F *__restrict__ x, F *__restrict__ y, uint32_t n_row, uint32_t n_col, uint32_t min_mean,
    double *__restrict__ head, double *__restrict__ tail, uint32_t *__restrict__ tail_row, uint32_t *__restrict__ range,
    const F *__restrict__ v, F *__restrict__ products, uint32_t n_products) {
  constexpr int U = FlatQuads<F, OUT>::value;
  constexpr uint32_t kStepQuads = U * kWave;
  constexpr int kFlatWaves = flat_threads(STAGED) / kWave;
  constexpr bool kSums = (OUT & kFlatSums) != 0, kProducts = (OUT & kFlatProducts) != 0;
  constexpr bool kWeights = kSums && HETER;  // (the products of v and x alone do not need them)
  extern __shared__ __attribute__((aligned(16))) unsigned char s_staged[];
  __shared__ uint32_t s_ptr_all[kFlatWaves][kFlatRows + 2];  // (entry 65: a sentinel)
  __shared__ double s_sum_all[kSums ? kFlatWaves : 1][kFlatRows];
  __shared__ F s_v_all[kProducts ? kFlatWaves : 1][kFlatRows + 1];  // v of the window's rows (entry 64: never used)
  const uint32_t nnz = indptr[n_row];
  const uint32_t mean = nnz / n_row;
  if (mean < min_mean || nnz > kFlatMaxNnz) return;  // (the launcher's other kernel takes those matrices)
  if constexpr (kProducts) {  // (index arrays longer than indptr says: nothing depends on what lies beyond)
    for (uint64_t i = nnz + static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n_products;
         i += gridDim.x * blockDim.x)
      products[i] = F(0);
  }
  const uint32_t lane = static_cast<uint32_t>(lane_id()), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  uint32_t *s_ptr = s_ptr_all[wv];
  double *s_sum = s_sum_all[kSums ? wv : 0];
  F *s_v = s_v_all[kProducts ? wv : 0];
  F *s_x = reinterpret_cast<F *>(s_staged);
  uint32_t staged = 0;
  if constexpr (STAGED) {
    constexpr uint32_t kFits = flat_staged_bytes<F, OUT>() / sizeof(F);
    staged = n_col < kFits ? n_col : kFits;
    copy_to_lds(s_x, x, staged);
    __syncthreads();
  }
  const uint32_t waves = gridDim.x * kFlatWaves, w = blockIdx.x * kFlatWaves + wv;
  // the wave owns the nonzeros [begin, end) and stores the rows [r, row_end), but for one that began before `begin`
  uint32_t share = nnz / waves + kFlatRowWeight * (n_row / waves + 1u) + 1u;
  if (share < flat_min_share<F, OUT, STAGED>()) share = flat_min_share<F, OUT, STAGED>();
  const uint64_t diag[2] = {static_cast<uint64_t>(w) * share, (static_cast<uint64_t>(w) + 1u) * share};
  uint32_t split_row[2], split_pos[2];
  if (diag[0] >= flat_list(n_row, nnz)) {
    if (kSums && lane == 0) head[w] = 0.0, tail[w] = 0.0, tail_row[w] = kNoRow, range[w] = nnz;
    return;
  }
  flat_split(indptr, n_row, nnz, diag, lane, split_row, split_pos);
  const uint32_t begin = split_pos[0], end = split_pos[1], row_end = split_row[1];
  if (kSums && lane == 0) head[w] = 0.0, tail[w] = 0.0, tail_row[w] = kNoRow, range[w] = begin;
  const F w_homo = (HETER || !kSums) ? F(0) : data[0];

  // Invariant at the start of a step [s0, s1): r is the first row whose end is not behind the wave; s_sum[0] holds what
  // row r has gathered in this wave so far, s_sum[1..63] are zero.
  uint32_t r = split_row[0];
  if (kSums) s_sum[lane] = 0.0;
  if (lane == 0) s_ptr[kFlatRows + 1] = 0xffffffffu;

  // Two steps are under way at a time: the index and weight streams of step i + 1 are requested before the
  // gathers of step i are consumed (568 against 609 us at 1e8 nonzeros).  A step's window of indptr is
  // requested first of all: waiting for a load means waiting for every load issued before it.  (Keeping the
  // next step's gathers in flight as well needs more registers than two workgroups per CU leave: the
  // compiler spills, and a reloaded register is a load that waits for every gather before it: 750 us.)
  // The loads carry no condition (a branch per load keeps the compiler from leaving them in flight): a lane beyond
  // the array's last whole quad reads that one again and its elements are masked by their position, and the one to
  // three nonzeros behind it are read where they are used.
  constexpr uint32_t kStep = 4u * kStepQuads;
  const uint32_t whole = nnz / 4u;
  auto load_streams = [&](uint32_t s0, u32x4 (&ci)[U], F (&cd)[U][4]) {  // lane l: quads s0 / 4 + l, + 64, ...
    if (s0 >= end || whole == 0) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t q = s0 / 4u + static_cast<uint32_t>(u) * kWave + lane;
      ci[u] = flat_index_quad(indices, q < whole ? q : whole - 1u);
    }
    if constexpr (kWeights) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = s0 / 4u + static_cast<uint32_t>(u) * kWave + lane;
        flat_data_quad(data, q < whole ? q : whole - 1u, cd[u]);
      }
    }
  };
  u32x4 ci[U] = {};
  F cd[U][4] = {};
  load_streams(begin & ~3u, ci, cd);
  // (a range without nonzeros has one step, for its rows)
  for (uint32_t s0 = begin & ~3u;; s0 += kStep) {
    const uint32_t s1 = (end - s0 > kStep) ? s0 + kStep : end;
    uint32_t ptr_lane, ptr_last;
    F v_lane = F(0);
    auto load_window = [&]() {
      const uint64_t k = static_cast<uint64_t>(r) + lane;
      if constexpr (kProducts) v_lane = k < n_row ? v[k] : F(0);
      ptr_lane = k <= n_row ? indptr[k] : 0xffffffffu;
      // (a load of the vector unit: one of the scalar unit would be waited for together with every LDS read)
      uint32_t last = r + kFlatRows;
      asm volatile("" : "+v"(last));
      ptr_last = static_cast<uint64_t>(r) + kFlatRows <= n_row ? indptr[last] : 0xffffffffu;
    };
    load_window();
    if (s1 > 4u * whole) {  // (the array's last one to three nonzeros)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane != whole) continue;
        const uint32_t p0 = 4u * whole;
        ci[u] = u32x4{indices[p0], p0 + 1u < nnz ? indices[p0 + 1u] : 0u, p0 + 2u < nnz ? indices[p0 + 2u] : 0u, 0u};
        if constexpr (kWeights) {
          cd[u][0] = data[p0];
          if (p0 + 1u < nnz) cd[u][1] = data[p0 + 1u];
          if (p0 + 2u < nnz) cd[u][2] = data[p0 + 2u];
        }
      }
    }
    F prod[U][4];  // (the vector's elements first, then the products: in F, as the reference forms them)
    auto column = [&](int u, int t) {  // (beyond the step: element 0, unused)
      const uint32_t p = 4u * (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane) + static_cast<uint32_t>(t);
      return p < s1 ? ci[u][t] : 0u;
    };
    if constexpr (STAGED) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t c = column(u, t);
          prod[u][t] = s_x[c < staged ? c : 0u];
        }
      }
      if (staged < n_col) {  // (uniform)
        // (all LDS reads first: without the empty statements each would be moved into the branch around the load)
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(prod[u][t]));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const uint32_t c = column(u, t);
            if (c >= staged) prod[u][t] = x[c];
          }
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) prod[u][t] = x[column(u, t)];
      }
    }
    F cw[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int t = 0; t < 4; ++t) cw[u][t] = kWeights ? cd[u][t] : w_homo;
    }
    load_streams(s1, ci, cd);  // (a step at or beyond the end of the range loads nothing)
    if constexpr (!kProducts) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) prod[u][t] = static_cast<F>(prod[u][t] * cw[u][t]);
      }
    }
    // (with products the elements of x are kept: this is the addend of the row's sum)
    auto addend = [&](int u, int t) {
      return static_cast<double>(kProducts ? static_cast<F>(prod[u][t] * cw[u][t]) : prod[u][t]);
    };
    // windows of 64 rows from r on, until one reaches beyond the step
    for (;;) {
      s_ptr[lane] = ptr_lane;
      if constexpr (kProducts) s_v[lane] = v_lane;
      if (lane == 0) s_ptr[kFlatRows] = ptr_last;
      __builtin_amdgcn_wave_barrier();
      const uint32_t lo = s_ptr[0] > begin ? s_ptr[0] : begin, hi = ptr_last;  // this window takes [lo, hi) of the step
      // The row of every quad's first nonzero and the ends of that row and of the next one, for the U quads
      // together (the LDS reads of different quads do not wait for each other); then, without a branch, the
      // quads that lie in one row or in two; a loop only for quads that meet three rows or more.
      uint32_t kq[U], e1[U], e2[U];
#pragma unroll
      for (int u = 0; u < U; ++u) kq[u] = 0;  // the last k < 64 with s_ptr[k] <= max(p0, lo) (s_ptr[0] <= lo)
#pragma unroll
      for (uint32_t step = kFlatRows / 2; step != 0; step >>= 1) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t p0 = 4u * (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane);
          const uint32_t pe = p0 > lo ? p0 : lo;
          if (s_ptr[kq[u] + step] <= pe) kq[u] += step;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) e1[u] = s_ptr[kq[u] + 1u], e2[u] = s_ptr[kq[u] + 2u];  // (s_ptr[65] is a sentinel)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t p0 = 4u * (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane);
        const uint32_t top = hi < s1 ? hi : s1;  // the window takes the nonzeros [lo, top)
        if (e2[u] > p0 + 3u || e1[u] >= top) {
          // one row, or two (what lies at e1 or behind belongs to row k + 1, unless that is the next window's)
          if constexpr (kProducts) {
            const F v0 = s_v[kq[u]], v1 = s_v[kq[u] + 1u];
            F g[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) g[t] = (p0 + static_cast<uint32_t>(t) < e1[u] ? v0 : v1) * prod[u][t];
            if (p0 >= lo && p0 + 3u < top) {
              flat_store_quad(products + p0, g);
            } else {
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const uint32_t p = p0 + static_cast<uint32_t>(t);
                if (p >= lo && p < top) products[p] = g[t];
              }
            }
          }
          if constexpr (kSums) {
            double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const uint32_t p = p0 + static_cast<uint32_t>(t);
              const double a = (p >= lo && p < top) ? addend(u, t) : 0.0;
              acc0 += p < e1[u] ? a : 0.0;
              acc1 += p < e1[u] ? 0.0 : a;
            }
            if (acc0 != 0.0) atomicAdd(&s_sum[kq[u]], acc0);
            if (acc1 != 0.0) atomicAdd(&s_sum[kq[u] + 1u], acc1);
          }
        } else if (p0 < top && p0 + 3u >= lo) {
          uint32_t k = kq[u];
          double acc = 0.0;
          uint32_t kacc = k;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const uint32_t p = p0 + static_cast<uint32_t>(t);
            if (p >= lo && p < top) {
              while (s_ptr[k + 1u] <= p) ++k;  // (ends below 64: p < hi = s_ptr[64])
              if constexpr (kProducts) products[p] = s_v[k] * prod[u][t];
              if constexpr (kSums) {
                if (k != kacc) {
                  if (acc != 0.0) atomicAdd(&s_sum[kacc], acc);
                  acc = 0.0, kacc = k;
                }
                acc += addend(u, t);
              }
            }
          }
          if (kSums && acc != 0.0) atomicAdd(&s_sum[kacc], acc);
        }
      }
      __builtin_amdgcn_wave_barrier();
      // rows of the window that end inside the step (a prefix of the window): stored, or, the one that began
      // before this wave's range, left in head[]
      const uint64_t row = static_cast<uint64_t>(r) + lane;
      const bool ended = lane < row_end - r && s_ptr[lane + 1u] <= s1;
      const uint32_t n_ended = static_cast<uint32_t>(__popcll(__ballot(ended)));
      if (kSums && ended) {
        const double total = s_sum[lane];
        if (ptr_lane < begin) head[w] = total;
        else y[row] = static_cast<F>(total);
      }
      double open = 0.0;
      if constexpr (kSums) open = n_ended < kFlatRows ? s_sum[n_ended] : 0.0;  // (wave uniform address: a broadcast)
      __builtin_amdgcn_wave_barrier();
      if constexpr (kSums) s_sum[lane] = 0.0;
      r += n_ended;
      if (n_ended < kFlatRows || r >= n_row) {
        if (kSums && lane == 0) s_sum[0] = open;
        break;
      }
      load_window();
    }
    __builtin_amdgcn_wave_barrier();
    if (s1 == end) break;
  }
  // the row that is still open at the end of the range (if it has nonzeros in it)
  if (kSums && lane == 0 && r < n_row) {
    const uint32_t rs = indptr[r];
    if (rs < end) {
      if (rs < begin) head[w] = s_sum[0];
      else tail[w] = s_sum[0], tail_row[w] = r;
    }
  }
}

// One wave per wave of the walk: the row left open at the end of range w = its tail + the heads of the ranges
// it runs through, in a fixed order.
template <typename F>
__global__ __launch_bounds__(kWave) void csr_flat_finish_kernel(const uint32_t *__restrict__ indptr, F *__restrict__ y,
                                                                uint32_t n_row, uint32_t min_mean,
                                                                uint32_t waves, const double *__restrict__ head,
                                                                const double *__restrict__ tail,
                                                                const uint32_t *__restrict__ tail_row,
                                                                const uint32_t *__restrict__ range) {
  const uint32_t nnz = indptr[n_row];
  const uint32_t mean = nnz / n_row;
  if (mean < min_mean || nnz > kFlatMaxNnz) return;
  const uint32_t w = blockIdx.x, lane = threadIdx.x;
  const uint32_t row = tail_row[w];
  if (row == kNoRow) return;
  const uint32_t row_end = indptr[row + 1u];
  double acc = 0.0;
  for (uint32_t v = w + 1u + lane; v < waves && range[v] < row_end; v += kWave) acc += head[v];
  acc = wave_sum(acc);
  if (lane == 0) y[row] = static_cast<F>(tail[w] + acc);
}

}  // namespace

// Whether the walk keeps the first elements of x in LDS: up to 552 KB, a quarter and more of which fit.  What a gather from L2 costs
// is the 128-byte line it moves (about 29 TB/s from all L2s, 230 G gathers/s): staging takes its share of them away,
// 120,000 floats and 2e7 nonzeros in rows of 100: 97 us, 155 us gathered from L2 alone.
template <typename F>
bool flat_stages(uint32_t n_col) {
  return static_cast<uint64_t>(n_col) * sizeof(F) <= 552ull * 1024u;
}

template <typename F, bool HETER, int OUT, bool STAGED>
static bool launch_flat(const char *target, hipStream_t stream, const F *data, const uint32_t *indices,
                        const uint32_t *indptr, const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t min_mean,
                        const F *v, F *products, uint32_t n_products) {
  constexpr bool kSums = (OUT & kFlatSums) != 0;
  const unsigned grid = static_cast<unsigned>(device_info().num_cu) * flat_per_cu(STAGED);
  const uint32_t waves = grid * (flat_threads(STAGED) / kWave);
  double *head = nullptr, *tail = nullptr;
  uint32_t *tail_row = nullptr, *range = nullptr;
  if (kSums) {
    // [head: waves doubles][tail: waves doubles][tail_row: waves words][range: waves words]
    unsigned char *ws = static_cast<unsigned char *>(stream_workspace(stream, static_cast<size_t>(waves) * 24u));
    if (ws == nullptr) return false;
    head = reinterpret_cast<double *>(ws), tail = head + waves;
    tail_row = reinterpret_cast<uint32_t *>(tail + waves), range = tail_row + waves;
  }
  auto kernel = csr_flat_gather_kernel<F, HETER, OUT, STAGED>;
  size_t lds = 0;
  if (STAGED) {
    constexpr uint32_t kMost = flat_staged_bytes<F, OUT>();
    lds = static_cast<size_t>(n_col) * sizeof(F) < kMost ? static_cast<size_t>(n_col) * sizeof(F) : kMost;
    static thread_local bool attr_set = false;  // (per instantiation)
    if (!attr_set) {
      if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(kMost)) != hipSuccess) {
        (void)hipGetLastError();
        set_error("%s: the device does not give a workgroup %u bytes of LDS", target, kMost);
        return false;
      }
      attr_set = true;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(flat_threads(STAGED)), lds, stream, data, indices, indptr, x, y, n_row,
                     n_col, min_mean, head, tail, tail_row, range, v, products, n_products);
  if (kSums)
    hipLaunchKernelGGL(csr_flat_finish_kernel<F>, dim3(waves), dim3(kWave), 0, stream, indptr, y, n_row, min_mean,
                       waves, static_cast<const double *>(head), static_cast<const double *>(tail),
                       static_cast<const uint32_t *>(tail_row), static_cast<const uint32_t *>(range));
  return check_launch(target);
}

template <typename F>
bool csr_flat_gather(const char *target, hipStream_t stream, const F *data, bool heter, const uint32_t *indices,
                     const uint32_t *indptr, const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t min_mean) {
  if (n_row == 0) return true;
  auto launch = [&](auto h, auto staged) {
    return launch_flat<F, decltype(h)::value, kFlatSums, decltype(staged)::value>(
      target, stream, data, indices, indptr, x, y, n_row, n_col, min_mean, nullptr, nullptr, 0u);
  };
  if (flat_stages<F>(n_col)) return heter ? launch(std::true_type(), std::true_type()) : launch(std::false_type(), std::true_type());
  return heter ? launch(std::true_type(), std::false_type()) : launch(std::false_type(), std::false_type());
}

template <typename F>
bool csr_gradient(const char *target, hipStream_t stream, const F *data, const uint32_t *indices, const uint32_t *indptr,
                  const F *v, const F *x, F *products, F *sums, uint32_t n_row, uint32_t n_col, uint32_t nnz) {
  if (n_row == 0) {
    fill_zero(stream, products, nnz);
    return check_launch(target);
  }
  if (nnz > kFlatMaxNnz) {
    set_error("%s: %u nonzeros are more than the walk's positions can number", target, nnz);
    return false;
  }
  auto launch = [&](auto out, auto staged) {
    return launch_flat<F, true, decltype(out)::value, decltype(staged)::value>(target, stream, data, indices, indptr, x, sums,
                                                                               n_row, n_col, 0u, v, products, nnz);
  };
  using Products = std::integral_constant<int, kFlatProducts>;
  using Both = std::integral_constant<int, kFlatSums | kFlatProducts>;
  if (flat_stages<F>(n_col)) return sums != nullptr ? launch(Both(), std::true_type()) : launch(Products(), std::true_type());
  return sums != nullptr ? launch(Both(), std::false_type()) : launch(Products(), std::false_type());
}

// csr_matvec_gradient: buffers = [data, indices, indptr, row vector, column vector, products, sums (or null)]
template <typename F>
static void csr_matvec_gradient_entry(const char *target, hipStream_t stream, void **buffers, const char *opaque,
                                      size_t opaque_len) {
  bpl_csr_transpose_descriptor d;
  if (!unpack(target, opaque, opaque_len, &d)) return;
  if (buffers == nullptr) {
    set_error("%s: null buffer table", target);
    return;
  }
  csr_gradient<F>(target, stream, static_cast<const F *>(buffers[0]), static_cast<const uint32_t *>(buffers[1]),
                  static_cast<const uint32_t *>(buffers[2]), static_cast<const F *>(buffers[3]),
                  static_cast<const F *>(buffers[4]), static_cast<F *>(buffers[5]), static_cast<F *>(buffers[6]), d.n_row,
                  d.n_col, d.nnz);
}

template bool flat_stages<float>(uint32_t);
template bool flat_stages<double>(uint32_t);
template bool csr_flat_gather<float>(const char *, hipStream_t, const float *, bool, const uint32_t *, const uint32_t *,
                                     const float *, float *, uint32_t, uint32_t, uint32_t);
template bool csr_flat_gather<double>(const char *, hipStream_t, const double *, bool, const uint32_t *, const uint32_t *,
                                      const double *, double *, uint32_t, uint32_t, uint32_t);

}  // namespace bpl

extern "C" void csr_matvec_gradient_float(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  bpl::csr_matvec_gradient_entry<float>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len);
}
extern "C" void csr_matvec_gradient_double(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  bpl::csr_matvec_gradient_entry<double>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len);
}
