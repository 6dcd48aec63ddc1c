// csr_matvec without transpose for vectors that are gathered from L2 (csr_flat_gather.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace bpl {

// The flat walk computes positions of nonzeros one step beyond the end of a wave's range in 32 bits: matrices
// with more nonzeros than this are left to the caller's other kernel, whatever their mean.
constexpr uint32_t kFlatMaxNnz = 0xffffffffu - 8192u;

// y = A x, walked flat: every wave owns a contiguous range of the nonzeros and tells the rows apart through
// windows of indptr in LDS.  For matrices with min_mean <= nnz / n_row and nnz <= kFlatMaxNnz; for others the kernels
// return at once and write nothing (the mean is known on the device only, so the caller enqueues its kernel
// for short rows behind this one).  x must have at least one element.
// nnz: the number of nonzeros as far as the caller knows it (0: not), for the choice of a kernel alone.  Takes 24 bytes of the stream's scratch
// memory per wave of its launch.  false: no scratch memory, or the launch failed (error recorded).
template <typename F>
bool csr_flat_gather(const char *target, hipStream_t stream, const F *data, bool heter, const uint32_t *indices,
                     const uint32_t *indptr, const F *x, F *y, uint32_t n_row, uint32_t n_col, uint32_t nnz,
                     uint32_t min_mean);

// Whether the walk keeps a part of x in LDS (one of up to four times what fits).
template <typename F>
bool flat_stages(uint32_t n_col);

// The same walk for the gradients of a product with a matrix of one weight per nonzero:
// products[j] = v[row of j] * x[column of j] and, if `sums` is given, sums = A x.  `products` has nnz elements; those
// beyond indptr[n_row], if that is less, become zero.
template <typename F>
bool csr_gradient(const char *target, hipStream_t stream, const F *data, const uint32_t *indices, const uint32_t *indptr,
                  const F *v, const F *x, F *products, F *sums, uint32_t n_row, uint32_t n_col, uint32_t nnz);

}  // namespace bpl
