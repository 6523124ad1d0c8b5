// Contraction entry points shared by the library's HIP translation units (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sbi {

// Row and job tables of the Jacobian contraction (device arrays).  Rows of dim z: off[z] .. end[z] - 1;
// off[z + 1] is end[z] rounded up to a multiple of four (the records in between are valid and
// unused).  Jobs cover the dims in groups of kJacGroup: either all rows of the group that starts at
// dim job[2] (rows job[0] .. job[1] - 1, none for a group without rows, whose J is zero; slot job[3] =
// -1), or a part of a group's rows with its own slot of partial sums; groups of several parts are listed
// in `red`.  Parts start at multiples of four rows after the group's first.
constexpr int kJacGroup = 8;
struct JacRows {
  const int32_t* row;  // [2 * off[nz]] {row of A, row of S}
  const int32_t* off;  // [nz + 1]
  const int32_t* end;  // [nz]
  const int32_t* job;  // [4 * n_jobs]
  const int32_t* red;  // [3 * n_red] {first dim, first slot, slots}
  int n_jobs, n_red;
};

// Jacobian contraction (gemm.hip), FP64 matrix cores: for each input dim z < nz, p < P, c < n,
//   J[(p * n + c) * nz + z] = sum over the rows q of dim z of A[row[2 q] * lda + p] *
//                                                            S[row[2 q + 1] * lds + c].
// A dim with no rows gets zeros.  A is 16-byte aligned, lda even and at least P rounded up to two.
// padded: the caller promises that every row of S, the last one included, is readable up to n rounded
// up to two.  part: P * n * kJacGroup doubles per slot.
int contract_jacobian_f64(const double* A, int64_t lda, const double* S, int64_t lds, bool padded,
                          const JacRows& t, int nz, double* J, int64_t P, int64_t n, double* part,
                          hipStream_t st);

}  // namespace sbi
