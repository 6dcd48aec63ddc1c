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
// kStaged: one workgroup of 1,024 threads per CU keeps the first elements of x (139 to 151 KB) in LDS and gathers only the
// rest from L2 (flat_stages()).  Every gather it spares counts: with 147 instead of 138 KB 1,000,000 x 50,000 with 100 per row
// takes 221 instead of 234 us, 200,000 x 50,000 56 instead of 58.
// kSwept: x passes through the LDS of every CU in windows of 147 KB, once per round; a round is what the CU's 16 waves hold
// in registers, 24 to 48 nonzeros a lane.  A CU then requests x in whole lines, 3,750 of them for 120,000 floats and 24,576
// nonzeros, instead of a line per nonzero.  The rounds' other traffic is under way meanwhile: a step's registers are
// filled with the next round's indices as soon as its rows are done.  Bound by what of a round does not overlap: staging
// (1.5 us a window), the test of every place against every window (three instructions), the rows (flat_vector() has the times).
// A workgroup whose columns lie together has no use for that: it looks at sixteen columns of every wave's first step, and
// where one window of x holds them or nearly so (the threshold below), it walks step by step with that window in LDS and
// gathers what it misses.  Which of the two a matrix wants is known on the device only: 300,000 rows of 100 and 120,000 floats,
// columns within 300 / 3,000 of the row's place 70 / 71 us, with all windows passing by 109 / 109, with the first 147 KB staged
// 69 / 99; a tenth of them anywhere 78, 109 and 72.  Slower than gathers from L2 that hit: one weight and
// 180,000 floats, columns within 300, 65 us (59), 30,000 rows of 1,000 and 150,000 floats 74 (64), and gathered so by this kernel,
// too (65 and 70, but 73 instead of 70 with 120,000).  What the look costs where the windows pass by: 0 to 2 us of 85 to 140 (from loads
// of its own, spread over the workgroup's nonzeros, 2 to 5).
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
enum class FlatVector { kL2, kStaged, kSwept };
// 16 waves per CU either way: two workgroups, or one that has the LDS to itself
constexpr int flat_threads(FlatVector from) { return from == FlatVector::kL2 ? 512 : 1024; }
constexpr unsigned flat_per_cu(FlatVector from) { return from == FlatVector::kL2 ? 2u : 1u; }
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
enum : int { kStepIndices = 1, kStepWeights = 2 };  // what is loaded of a step

// quads per lane and step, as many as 128 registers hold (with sums and products of floats at once two as well: the
// elements of x and the weights both live until the rows are known)
template <typename F, int OUT, FlatVector FROM>
struct FlatQuads {
  static constexpr int value = sizeof(F) == 4 && OUT != (kFlatSums | kFlatProducts) && FROM != FlatVector::kSwept ? 4 : 2;
};

// A lane's index quads of a step.
template <int N>
struct FlatIndices {
  static constexpr int count = N;
  u32x4 q[N];
};

// The least a wave takes, in nonzeros and rows: a wavefront of quads.  (The plain sums of x in L2 whole steps: a gather
// costs the address unit the same however many of its lanes hold a nonzero.)
template <typename F, int OUT, FlatVector FROM>
constexpr uint32_t flat_min_share() {
  return 4u * kWave * ((OUT == kFlatSums && FROM == FlatVector::kL2) ? FlatQuads<F, OUT, FROM>::value : 1);
}

// kSwept: steps whose nonzeros a wave keeps in registers while the windows of x pass by, as many as 128 registers hold.
template <typename F, bool HETER, int OUT>
struct FlatHeld {
  static constexpr int value = (OUT == kFlatProducts ? 6 : HETER && sizeof(F) == 4 ? 3 : 4) /
                               static_cast<int>(sizeof(F) / 4);
};

// (Sums and products of doubles at once: the registers hold one step, and no size pays for the windows.  Doubles with one
// weight: 150,000 to 500,000 rows of 100 with 37,500 columns take as long either way, more columns longer.)
template <typename F, bool HETER, int OUT>
constexpr bool flat_sweeps() { return sizeof(F) == 4 || (HETER && OUT != (kFlatSums | kFlatProducts)); }

// kSwept: a nonzero's register holds where its element of x lies until a window brings the element itself.  The place is
// written as a NaN with its sign set, one that no element has in LDS: those are stored as the NaN without a payload.
__device__ __forceinline__ float flat_place(float, uint32_t c) { return __uint_as_float(0xff800004u + 4u * c); }
__device__ __forceinline__ double flat_place(double, uint32_t c) {
  return __hiloint2double(static_cast<int>(0xfff00001u + c), 0);
}
__device__ __forceinline__ float flat_no_place(float v) {
  return __float_as_uint(v) > 0xff800000u ? __uint_as_float(0x7fc00000u) : v;
}
__device__ __forceinline__ double flat_no_place(double v) {
  return static_cast<uint32_t>(__double2hiint(v)) > 0xfff00000u ? __hiloint2double(0x7ff80000, 0) : v;
}
// v = the element whose place it holds, if that lies among the n in LDS, which begin with element `first`.  (origin: kept
// in one scalar register, so that a nonzero costs a subtraction, a comparison and a read of the lanes concerned.)
typedef __attribute__((address_space(3))) const unsigned char *flat_lds;
__device__ __forceinline__ uint32_t flat_origin(float, uint32_t first) { return 0xff800004u + 4u * first; }
__device__ __forceinline__ uint32_t flat_origin(double, uint32_t first) { return 0xfff00001u + first; }
__device__ __forceinline__ void flat_take(float &v, flat_lds window, uint32_t origin, uint32_t bytes) {
  const uint32_t at = __float_as_uint(v) - origin;
  if (at < bytes) v = *reinterpret_cast<__attribute__((address_space(3))) const float *>(window + at);
}
__device__ __forceinline__ void flat_take(double &v, flat_lds window, uint32_t origin, uint32_t bytes) {
  const uint32_t at = static_cast<uint32_t>(__double2hiint(v)) - origin;
  if (at < bytes / 8u) v = *reinterpret_cast<__attribute__((address_space(3))) const double *>(window + 8u * at);
}
// Columns that have a place: the places of both types end in front of 2^32, behind which the words of zeros and denormals begin.
constexpr uint32_t kFlatMostPlaces = (1u << 20) - 1u;
static_assert(0xfff00001ull + kFlatMostPlaces - 1u <= 0xffffffffull && 0xff800004ull + 4ull * (kFlatMostPlaces - 1u) <= 0xffffffffull,
              "no place is taken for a number");

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {  // (of all 64 lanes, to all of them)
#pragma unroll
  for (int d = 1; d < kWave; d *= 2) v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), d, kWave)));
  return __builtin_amdgcn_readfirstlane(v);
}

// The n elements of x to LDS, three 16-byte loads of every thread in flight.
template <typename F>
__device__ __forceinline__ void flat_stage_window(F *to, const F *__restrict__ x, uint32_t n) {
  constexpr uint32_t kPer = 16 / sizeof(F), kUnroll = 3;
  typedef F piece __attribute__((ext_vector_type(kPer), aligned(sizeof(F))));
  typedef F lds_piece __attribute__((ext_vector_type(kPer)));
  const uint32_t pieces = n / kPer;
  for (uint32_t i0 = threadIdx.x; i0 < pieces; i0 += kUnroll * blockDim.x) {
    piece v[kUnroll];
#pragma unroll
    for (uint32_t k = 0; k < kUnroll; ++k) {
      const uint32_t i = i0 + k * blockDim.x;
      v[k] = reinterpret_cast<const piece *>(x)[i < pieces ? i : pieces - 1u];
    }
#pragma unroll
    for (uint32_t k = 0; k < kUnroll; ++k) {
      const uint32_t i = i0 + k * blockDim.x;
      lds_piece t;
#pragma unroll
      for (uint32_t j = 0; j < kPer; ++j) t[j] = flat_no_place(v[k][j]);
      if (i < pieces) reinterpret_cast<lds_piece *>(to)[i] = t;
    }
  }
  const uint32_t rest = pieces * kPer + threadIdx.x;
  if (rest < n) to[rest] = flat_no_place(x[rest]);
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

template <typename F, bool HETER, int OUT, FlatVector FROM>
__global__ __launch_bounds__(flat_threads(FROM), 4) void csr_flat_gather_kernel(
    const F *__restrict__ data, const uint32_t *__restrict__ indices, const uint32_t *__restrict__ indptr,
    const F *__restrict__ x, F *__restrict__ y, uint32_t n_row, uint32_t n_col, uint32_t min_mean,
    double *__restrict__ head, double *__restrict__ tail, uint32_t *__restrict__ tail_row, uint32_t *__restrict__ range,
    const F *__restrict__ v, F *__restrict__ products, uint32_t n_products, uint32_t least) {
  constexpr int kFlatWaves = flat_threads(FROM) / kWave;
  constexpr bool kStaged = FROM == FlatVector::kStaged, kSwept = FROM == FlatVector::kSwept;
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
  constexpr uint32_t kFits = flat_staged_bytes<F, OUT>() / sizeof(F);  // elements of x in LDS
  const uint32_t staged = n_col < kFits ? n_col : kFits;       // (kStaged)
  if constexpr (kStaged) {
    copy_to_lds(s_x, x, staged);
    __syncthreads();
  }
  const uint32_t waves = gridDim.x * kFlatWaves, w = blockIdx.x * kFlatWaves + wv;
  static_assert(sizeof(s_ptr_all) + (kSums ? sizeof(s_sum_all) : 0u) + (kProducts ? sizeof(s_v_all) : 0u) +
                  (kWave + 4u) * sizeof(uint32_t) + flat_staged_bytes<F, OUT>() <= 160u * 1024u, "LDS of a CU");
  // (kSwept: how many of the columns looked at lie in each half of a window, the first and the last of them, their number)
  constexpr uint32_t kHalf = kFits / 2u;
  __shared__ uint32_t s_half[kSwept ? kWave : 1], s_lowest, s_highest, s_sampled, s_rounds;
  if constexpr (kSwept) {
    if (threadIdx.x < kWave) s_half[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_lowest = kNoRow, s_highest = 0, s_sampled = 0, s_rounds = 0;
    __syncthreads();
  }
  // the wave owns the nonzeros [begin, end) and stores the rows [r, row_end), but for one that began before `begin`
  uint32_t share = nnz / waves + kFlatRowWeight * (n_row / waves + 1u) + 1u;
  if (share < flat_min_share<F, OUT, FROM>()) share = flat_min_share<F, OUT, FROM>();
  const uint64_t diag[2] = {static_cast<uint64_t>(w) * share, (static_cast<uint64_t>(w) + 1u) * share};
  uint32_t split_row[2], split_pos[2];
  const bool idle = diag[0] >= flat_list(n_row, nnz);
  if (idle) {
    if (kSums && lane == 0) head[w] = 0.0, tail[w] = 0.0, tail_row[w] = kNoRow, range[w] = nnz;
    if constexpr (!kSwept) return;
    split_row[0] = split_row[1] = n_row, split_pos[0] = split_pos[1] = nnz;  // (it helps to bring the windows)
  } else {
    flat_split(indptr, n_row, nnz, diag, lane, split_row, split_pos);
  }
  const uint32_t begin = split_pos[0], end = split_pos[1], row_end = split_row[1];
  if (kSums && !idle && lane == 0) head[w] = 0.0, tail[w] = 0.0, tail_row[w] = kNoRow, range[w] = begin;
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
  const uint32_t whole = nnz / 4u;
  auto load_step = [&](uint32_t s0, auto which, auto &ci, auto &cd) {  // lane l: quads s0 / 4 + l, + 64, ...
    constexpr int kWhich = decltype(which)::value, U = std::remove_reference_t<decltype(ci)>::count;
    if (s0 >= end || whole == 0) {
      // (what is not loaded is not kept either: its registers are free)
#pragma unroll
      for (int u = 0; kSwept && (kWhich & kStepIndices) && u < U; ++u) ci.q[u] = u32x4{};
      return;
    }
    if constexpr ((kWhich & kStepIndices) != 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = s0 / 4u + static_cast<uint32_t>(u) * kWave + lane;
        ci.q[u] = flat_index_quad(indices, q < whole ? q : whole - 1u);
      }
    }
    if constexpr (kWeights && (kWhich & kStepWeights) != 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = s0 / 4u + static_cast<uint32_t>(u) * kWave + lane;
        flat_data_quad(data, q < whole ? q : whole - 1u, cd[u]);
      }
    }
  };
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
  // The window's loads are waited for here, where the number of loads behind them is known: at the head of the loop over the
  // windows the compiler waits for every load that either way in may have left.
  auto await_window = [&]() {
    if constexpr (FROM == FlatVector::kL2) return;
    asm volatile("" : "+v"(ptr_lane), "+v"(ptr_last));
    if constexpr (kProducts) asm volatile("" : "+v"(v_lane));
  };
  // The array's last one to three nonzeros, where the step holds them.
  auto load_last = [&](uint32_t s0, auto which, auto &ci, auto &cd) {
    constexpr int kWhich = decltype(which)::value, U = std::remove_reference_t<decltype(ci)>::count;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane != whole) continue;
      const uint32_t p0 = 4u * whole;
      if constexpr ((kWhich & kStepIndices) != 0)
        ci.q[u] = u32x4{indices[p0], p0 + 1u < nnz ? indices[p0 + 1u] : 0u, p0 + 2u < nnz ? indices[p0 + 2u] : 0u, 0u};
      if constexpr (kWeights && (kWhich & kStepWeights) != 0) {
        cd[u][0] = data[p0];
        if (p0 + 1u < nnz) cd[u][1] = data[p0 + 1u];
        if (p0 + 2u < nnz) cd[u][2] = data[p0 + 2u];
      }
    }
  };
  using Indices = std::integral_constant<int, kStepIndices>;
  using Weights = std::integral_constant<int, kStepWeights>;
  using Both = std::integral_constant<int, kStepIndices | kStepWeights>;
  // The rows of the step [s0, s1).  prod: its products, with products to store (kProducts) the elements of x; cw: its weights.
  auto walk_rows = [&](uint32_t s0, uint32_t s1, const auto &prod, const auto &cw) {
    constexpr int U = static_cast<int>(std::extent_v<std::remove_reference_t<decltype(prod)>>);
    auto addend = [&](int u, int t) {
      return static_cast<double>(kProducts ? static_cast<F>(prod[u][t] * cw[u][t]) : prod[u][t]);
    };
    await_window();
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
      await_window();
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto multiply = [&](auto &prod, const auto &cw) {
    constexpr int U = static_cast<int>(std::extent_v<std::remove_reference_t<decltype(prod)>>);
    if constexpr (!kProducts) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) prod[u][t] = static_cast<F>(prod[u][t] * (kWeights ? cw[u][t] : w_homo));
      }
    }
  };
  // Step by step, with the n_lds elements of x from `origin` on in LDS (kInLds).
  auto walk_steps = [&](auto in_lds, auto origin, uint32_t n_lds, auto &&stage) {
    constexpr bool kInLds = decltype(in_lds)::value;
    constexpr int U = FlatQuads<F, OUT, kInLds ? FlatVector::kStaged : FlatVector::kL2>::value;
    constexpr uint32_t kStep = 4u * U * kWave;
    FlatIndices<U> ci = {};
    F cd[U][4] = {};
    load_step(begin & ~3u, Both(), ci, cd);
    stage();
    // (a range without nonzeros has one step, for its rows)
    for (uint32_t s0 = begin & ~3u;; s0 += kStep) {
      const uint32_t s1 = (end - s0 > kStep) ? s0 + kStep : end;
      load_window();
      if (s1 > 4u * whole) load_last(s0, Both(), ci, cd);
      F prod[U][4];  // (the vector's elements first, then the products: in F, as the reference forms them)
      auto column = [&](int u, int t) {  // (beyond the step: one that costs nothing, unused)
        const uint32_t p = 4u * (s0 / 4u + static_cast<uint32_t>(u) * kWave + lane) + static_cast<uint32_t>(t);
        return p < s1 ? ci.q[u][t] : static_cast<uint32_t>(origin);
      };
      auto place = [&](uint32_t c) {  // (in a window that may run on at element 0)
        if constexpr (std::is_same_v<decltype(origin), uint32_t>) return min(c - origin, c - origin + n_col);
        else return c;
      };
      if constexpr (kInLds) {
        const uint32_t last = n_lds - 1u;
        uint32_t furthest = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const uint32_t at = place(column(u, t));
            prod[u][t] = s_x[min(at, last)];
            furthest = max(furthest, at);
          }
        }
        if (__builtin_amdgcn_ballot_w64(furthest > last) != 0) {
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
              if (place(c) > last) prod[u][t] = x[c];
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
        for (int t = 0; t < 4; ++t) cw[u][t] = cd[u][t];
      }
      load_step(s1, Both(), ci, cd);  // (a step at or beyond the end of the range loads nothing)
      multiply(prod, cw);
      walk_rows(s0, s1, prod, cw);
      if (s1 == end) break;
    }
  };
  constexpr int kHeldSteps = FlatHeld<F, HETER, OUT>::value, kHeldQuads = FlatQuads<F, OUT, FROM>::value;
  constexpr uint32_t kHeld = 4u * kHeldQuads * kWave * kHeldSteps;  // nonzeros of a wave's round
  const uint32_t own = idle ? 0u : (begin & ~3u) < end ? (end - (begin & ~3u) - 1u) / kHeld + 1u : 1u;  // its rounds
  uint32_t origin = kNoRow, n_lds = kFits;
  FlatIndices<kHeldQuads> first_step = {};
  if constexpr (kSwept) {
    F unused[kHeldQuads][4];
    load_step(begin & ~3u, Indices(), first_step, unused);  // (under way meanwhile)
    if ((begin & ~3u) < end && whole != 0) {  // sixteen columns of every wave
      const uint32_t column = first_step.q[0][0];
      const bool sampled = lane % 4u == 0;
      if (sampled) atomicAdd(&s_half[column / kHalf < kWave ? column / kHalf : kWave - 1u], 1u);
      const uint32_t lowest = ~wave_max_u32(sampled ? ~column : 0u), highest = wave_max_u32(sampled ? column : 0u);
      if (lane == 0) atomicMin(&s_lowest, lowest), atomicMax(&s_highest, highest), atomicAdd(&s_sampled, kWave / 4u);
    }
    if (lane == 0) atomicMax(&s_rounds, own);
    __syncthreads();
    // One window for all columns looked at, with room for those between and beyond them; else the two neighbouring halves
    // that hold most (the last and the first element are neighbours: a ring's first and last rows), if what they miss is at
    // most half of what the launcher takes to be worth the windows (where every column is as likely, 256 columns tell a
    // share of 0.3 to 0.03, and one workgroup that gathers a third of its elements is the last of all: a threshold of
    // three quarters took 60,000,000 nonzeros over 200,000 floats from 250 to 259 us).
    const uint32_t lowest = s_lowest, highest = s_highest;
    if (lowest <= highest && highest < n_col) {
      const uint32_t pad = (highest - lowest) / 16u + 64u;
      const uint32_t from = (lowest > pad ? lowest - pad : 0u) & ~3u, to = n_col - highest > pad ? highest + pad : n_col;
      if (to - from <= kFits) {
        origin = from, n_lds = to - from;
      } else {
        const uint32_t halves = (n_col - 1u) / kHalf + 1u;
        const uint32_t both = lane < halves ? s_half[lane] + s_half[lane + 1u < halves ? lane + 1u : 0u] : 0u;
        const uint32_t most = wave_max_u32(both), sampled = s_sampled;
        const uint32_t first = kHalf * static_cast<uint32_t>(__builtin_ctzll(__builtin_amdgcn_ballot_w64(both == most)));
        if (2u * (sampled - most) * static_cast<uint64_t>(nnz) < sampled * static_cast<uint64_t>(least))
          origin = first + (n_col - first) % 4u;  // (what lies behind the last element is a multiple of 16 bytes from the first)
      }
      origin = __builtin_amdgcn_readfirstlane(origin), n_lds = __builtin_amdgcn_readfirstlane(n_lds);
    }
  }
  if constexpr (!kSwept) {
    walk_steps(std::integral_constant<bool, kStaged>(), std::integral_constant<uint32_t, 0u>(), staged, []() {});
  } else if (origin != kNoRow) {
    auto stage = [&]() {
      const uint32_t to_end = n_col - origin;
      copy_to_lds(s_x, x + origin, n_lds < to_end ? n_lds : to_end);
      if (n_lds > to_end) copy_to_lds(s_x + to_end, x, n_lds - to_end);
      __syncthreads();
    };
    if (idle) stage();
    else walk_steps(std::true_type(), origin, n_lds, stage);
  } else {
    constexpr int H = kHeldSteps, U = kHeldQuads;
    constexpr uint32_t kStep = 4u * U * kWave;
    FlatIndices<U> ci[H] = {};
    F cd[2][U][4] = {};  // weights, a step ahead
    uint32_t s0 = begin & ~3u;  // the round takes [s0, s0 + H * kStep)
    ci[0] = first_step;
#pragma unroll
    for (int h = 1; h < H; ++h) load_step(s0 + static_cast<uint32_t>(h) * kStep, Indices(), ci[h], cd[0]);
    load_step(s0, Weights(), ci[0], cd[0]);
    const uint32_t rounds = __builtin_amdgcn_readfirstlane(s_rounds);
    const uint32_t windows = (n_col - 1u) / kFits + 1u;
    const uint32_t width = ((n_col - 1u) / windows + 4u) & ~3u;  // (at most kFits, a multiple of 4)
    uint32_t here = kNoRow;                                      // the window in LDS
    for (uint32_t round = 0; round < rounds; ++round) {
      const bool work = round < own;  // (uniform over the wave; without work it brings its part of the windows)
      F prod[H][U][4];
      if (work) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const uint32_t sh = s0 + static_cast<uint32_t>(h) * kStep;
          if (sh < end && end - sh <= kStep && end > 4u * whole) load_last(sh, Indices(), ci[h], cd[0]);
#pragma unroll
          for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const uint32_t p = 4u * (sh / 4u + static_cast<uint32_t>(u) * kWave + lane) + static_cast<uint32_t>(t);
              prod[h][u][t] = p < end ? flat_place(F(0), ci[h].q[u][t]) : F(0);
            }
          }
        }
      }
      // (there and back: a round begins with the window that the one before ended with)
      for (uint32_t i = 0; i < windows; ++i) {
        const uint32_t window = (round & 1u) ? windows - 1u - i : i;
        const uint32_t first = window * width, n = n_col - first < width ? n_col - first : width;
        if (window != here) {
          if (here != kNoRow) __syncthreads();
          flat_stage_window(s_x, x + first, n);
          here = window;
          __syncthreads();
        }
        if (work) {
          uint32_t origin = flat_origin(F(0), first), bytes = n * static_cast<uint32_t>(sizeof(F));
          asm volatile("" : "+s"(origin), "+s"(bytes));
#pragma unroll
          for (int h = 0; h < H; ++h) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
              for (int t = 0; t < 4; ++t) flat_take(prod[h][u][t], (flat_lds)s_staged, origin, bytes);
            }
          }
        }
      }
      if (work) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const uint32_t sh = s0 + static_cast<uint32_t>(h) * kStep;
          const bool step = h == 0 || sh < end;
          if (step) load_window();
          load_step(sh + kStep, Weights(), ci[0], cd[(h + 1) % 2]);
          // (the steps behind are done with their registers: the next round's indices are requested)
          if (h != 0) load_step(sh + (H - 1u) * kStep, Indices(), ci[h - 1], cd[0]);
          if (step) {
            const uint32_t s1 = end - sh > kStep ? sh + kStep : end;
            if (s1 > 4u * whole) load_last(sh, Weights(), ci[0], cd[h % 2]);
            multiply(prod[h], cd[h % 2]);
            walk_rows(sh, s1, prod[h], cd[h % 2]);
          }
        }
        load_step(s0 + (2u * H - 1u) * kStep, Indices(), ci[H - 1], cd[0]);
        s0 += H * kStep;
        if constexpr (H % 2 != 0) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < 4; ++t) cd[0][u][t] = cd[1][u][t];
          }
        }
      }
    }
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

// Where the walk takes x from, if its columns lie anywhere (the kernel itself looks whether they do).  A visit of a window (147 KB staged
// and a test of every place held, 3 us with nothing beside it) has to spare 1.15 million gathers (double 0.7; with one weight
// 1.4: no weights to request meanwhile), a call a million (one weight 2.0), and x has to be longer than what fits by as much as makes a gather cost a
// line of its own (weights 1.5 times, one weight twice: 50,000 floats and 1e8 nonzeros in rows of 100 220 us, by windows 242, one weight and 75,000
// 241 and 241).  Measured without windows and now (300,000 rows of 100 where not said): 60,000 / 120,000 / 180,000 floats 92 / 130 / 152
// -> 86 / 107 / 122 us, the weights' gradient 91 / 118 / 144 -> 71 / 85 / 97, both gradients 123 / 159 / 172 -> 102 / 123 / 139, one weight
// 120,000 / 180,000 106 / 139 -> 100 / 113, doubles 30,000 / 60,000 / 90,000 123 / 158 / 183 -> 104 / 137 / 160, their gradient 140 / 166 / 183 ->
// 106 / 127 / 142; 30,000 rows of 1,000 and 150,000 floats 150 -> 114.  On the other side of the line, with and without:
// 260,000 floats 148 and 154, 200,000 with 1e7 nonzeros 58 and 59, 5e6 37 and 36; one weight and 60,000 84 and 73, 260,000 135 and 141.
template <typename F, bool HETER, int OUT>
static FlatVector flat_vector(uint32_t n_col, uint32_t nnz, uint32_t *least) {
  constexpr uint32_t kFits = flat_staged_bytes<F, OUT>() / sizeof(F);
  constexpr FlatVector kSwept = FlatVector::kSwept;
  if (n_col <= kFits) return FlatVector::kStaged;
  if constexpr (flat_sweeps<F, HETER, OUT>()) {
    const uint64_t waves = static_cast<uint64_t>(device_info().num_cu) * (flat_threads(kSwept) / kWave);
    const uint64_t round = waves * kWave * 4u * FlatQuads<F, OUT, kSwept>::value * FlatHeld<F, HETER, OUT>::value;
    const uint64_t visits = 1u + static_cast<uint64_t>((n_col - 1u) / kFits) * (nnz / round + 1u);
    const uint64_t gathers = flat_stages<F>(n_col) ? nnz - static_cast<uint64_t>(nnz) * kFits / n_col : nnz;
    constexpr uint32_t kPerVisit = !HETER ? 1400000u : sizeof(F) == 4 ? 1150000u : 700000u;
    constexpr uint32_t kPerCall = !HETER ? 2000000u : 1000000u;
    constexpr uint32_t kLeast = !HETER ? 2u * kFits : OUT == kFlatSums && sizeof(F) == 4 ? kFits + kFits / 2u : kFits;
    const uint64_t worth = visits * kPerVisit + kPerCall;
    *least = static_cast<uint32_t>(worth);  // (gathers is below 2^32)
    constexpr uint32_t kHalves = kFits / 2u * kWave;  // (the kernel's histogram of the columns)
    constexpr uint32_t kMost = kHalves < kFlatMostPlaces ? kHalves : kFlatMostPlaces;
    if (n_col > kLeast && n_col <= kMost && gathers >= worth) return kSwept;
  }
  return flat_stages<F>(n_col) ? FlatVector::kStaged : FlatVector::kL2;
}

template <typename F, bool HETER, int OUT, FlatVector FROM>
static bool launch_flat(const char *target, hipStream_t stream, const F *data, const uint32_t *indices,
                        const uint32_t *indptr, const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t min_mean,
                        const F *v, F *products, uint32_t n_products, uint32_t least) {
  constexpr bool kSums = (OUT & kFlatSums) != 0;
  const unsigned grid = static_cast<unsigned>(device_info().num_cu) * flat_per_cu(FROM);
  const uint32_t waves = grid * (flat_threads(FROM) / kWave);
  double *head = nullptr, *tail = nullptr;
  uint32_t *tail_row = nullptr, *range = nullptr;
  if (kSums) {
    // [head: waves doubles][tail: waves doubles][tail_row: waves words][range: waves words]
    unsigned char *ws = static_cast<unsigned char *>(stream_workspace(stream, static_cast<size_t>(waves) * 24u));
    if (ws == nullptr) return false;
    head = reinterpret_cast<double *>(ws), tail = head + waves;
    tail_row = reinterpret_cast<uint32_t *>(tail + waves), range = tail_row + waves;
  }
  auto kernel = csr_flat_gather_kernel<F, HETER, OUT, FROM>;
  size_t lds = 0;
  if (FROM != FlatVector::kL2) {
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
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(flat_threads(FROM)), lds, stream, data, indices, indptr, x, y, n_row,
                     n_col, min_mean, head, tail, tail_row, range, v, products, n_products, least);
  if (kSums)
    hipLaunchKernelGGL(csr_flat_finish_kernel<F>, dim3(waves), dim3(kWave), 0, stream, indptr, y, n_row, min_mean,
                       waves, static_cast<const double *>(head), static_cast<const double *>(tail),
                       static_cast<const uint32_t *>(tail_row), static_cast<const uint32_t *>(range));
  return check_launch(target);
}

template <typename F, bool HETER, int OUT>
static bool flat_walk(const char *target, hipStream_t stream, const F *data, const uint32_t *indices, const uint32_t *indptr,
                      const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t nnz, uint32_t min_mean, const F *v,
                      F *products) {
  uint32_t least = 0;
  const FlatVector from = flat_vector<F, HETER, OUT>(n_col, nnz, &least);
  auto launch = [&](auto from) {
    return launch_flat<F, HETER, OUT, decltype(from)::value>(target, stream, data, indices, indptr, x, y, n_row, n_col,
                                                             min_mean, v, products, (OUT & kFlatProducts) ? nnz : 0u, least);
  };
  switch (from) {
    case FlatVector::kStaged: return launch(std::integral_constant<FlatVector, FlatVector::kStaged>());
    case FlatVector::kSwept:
      if constexpr (flat_sweeps<F, HETER, OUT>()) return launch(std::integral_constant<FlatVector, FlatVector::kSwept>());
    default: return launch(std::integral_constant<FlatVector, FlatVector::kL2>());
  }
}

template <typename F>
bool csr_flat_gather(const char *target, hipStream_t stream, const F *data, bool heter, const uint32_t *indices,
                     const uint32_t *indptr, const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t nnz,
                     uint32_t min_mean) {
  if (n_row == 0) return true;
  auto walk = heter ? flat_walk<F, true, kFlatSums> : flat_walk<F, false, kFlatSums>;
  return walk(target, stream, data, indices, indptr, x, y, n_row, n_col, nnz, min_mean, nullptr, nullptr);
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
  auto walk = sums != nullptr ? flat_walk<F, true, kFlatSums | kFlatProducts> : flat_walk<F, true, kFlatProducts>;
  return walk(target, stream, data, indices, indptr, x, sums, n_row, n_col, nnz, 0u, v, products);
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
                                     const float *, float *, uint32_t, uint32_t, uint32_t, uint32_t);
template bool csr_flat_gather<double>(const char *, hipStream_t, const double *, bool, const uint32_t *, const uint32_t *,
                                      const double *, double *, uint32_t, uint32_t, uint32_t, uint32_t);

}  // namespace bpl

extern "C" void csr_matvec_gradient_float(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  bpl::csr_matvec_gradient_entry<float>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len);
}
extern "C" void csr_matvec_gradient_double(bpl_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
  bpl::csr_matvec_gradient_entry<double>(__func__, static_cast<hipStream_t>(stream), buffers, opaque, opaque_len);
}
