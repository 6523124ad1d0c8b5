// Shared host-side helpers: thread-local error message, HIP status checks.
#pragma once

#include <cstdint>
#include <string>

namespace sbi {

void set_error(const std::string& msg);

// Jacobian contraction (gemm.hip): whether the rows of S may be copied 16 bytes at a time.  They start
// on 16 bytes, and for an odd n the element after a row's last one is there (padded: without that
// promise the last row may be the end of its allocation, whatever lds is).
inline bool jac_wide_rows(const double* S, int64_t lds, int64_t n, bool padded) {
  return ((uintptr_t)S & 15) == 0 && lds % 2 == 0 && (n % 2 == 0 || (padded && lds > n));
}

}  // namespace sbi

// Return SBI_ERR_HIP with the HIP error text recorded when a HIP runtime call fails (used by the
// HIP translation units only).
#define SBI_HIP_CHECK(expr)                                                              \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess) {                                                              \
      sbi::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));                 \
      return SBI_ERR_HIP;                                                                \
    }                                                                                    \
  } while (0)
