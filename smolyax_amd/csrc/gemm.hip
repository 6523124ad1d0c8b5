// Coefficient-by-basis contraction on the matrix cores (gfx950 MFMA), for many outputs.
//
//   Y[p, j] = offset[j] + sum_k A[k, p] * B[k, j]        p < P, j < n, k < K
//
// A is the basis matrix written by the basis kernels (K x P, points contiguous: the Newton basis
// H^T or the barycentric entry weights W^T); B is the coefficient matrix (K x n, outputs
// contiguous: Newton surpluses or zeta-scaled node values).  Y is FP64, row stride ldy.
//
// Every workgroup is independent (no inter-workgroup waits, no atomics), so any number of these
// launches may run concurrently on several streams, and each Y row is a function of its own column
// of A only, summed in a fixed order: a point's result does not depend on P, on its position in
// the batch or on the batch's other points (bit for bit).
//
// FP64 operands: contract_f64_kernel; FP32 with k interleaved by four and more than 32 outputs:
// contract_k4_kernel (both stage their operands in LDS).  Other FP32 calls: contract_kernel below.
// The staged loops' raw barriers wait for the wave's copies (vmcnt) and for its LDS reads (lgkmcnt): a
// buffer that other waves copy into after the barrier has then been read.
//
// contract_kernel, work split: a workgroup of 4 waves owns a 64-point x (32*FN)-output tile of Y;
// each wave a 32 x 16*FN sub-tile made of 2 x FN MFMA 16x16 fragments.
//
// k order: MFMA 16x16x4 takes k = lane/16 from lane group g; within a 16-wide chunk of k, step s
// of the four MFMAs takes k = k0 + 4g + s, so each lane walks four consecutive rows of A and B.
// A and B are read with one dword per lane (plain layout); the 16 lanes of a group read 16
// consecutive points (outputs) of one row: 64-byte segments.  Edges are handled by clamped loads
// (rows beyond P or n are computed and discarded) and, in the last chunk, by zeroing terms with
// k >= K.
//
// Accumulation: the FP32 MFMA accumulators (v_mfma_f32_16x16x4) hold partial sums of kFlushK terms
// of k that are added into FP64 accumulators (in LDS), so the accumulation error stays that of a
// 256-term sum and the result's error is dominated by the FP32 rounding of the operands.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "../../include/smolyax_amd.h"
#include "common.h"
#include "gemm.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kWaves = 4;
constexpr int kBlockM = 64;   // points per workgroup
constexpr int kChunk = 16;    // k per main-loop iteration
constexpr int kFlushK = 256;  // FP32 partial sums are flushed into FP64 every kFlushK terms

__device__ __forceinline__ v4f mfma(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4d mfma(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// FP64 head rows k < K64 of A64 (K64 x P) and B64 (K64 x n) into h with the FP64 MFMA (lane group
// g supplies row k0 + g of each 4-row step; lane li point ph[fm] and output jcol[fn]).  Four steps
// per iteration: all their loads are issued before their MFMAs (one memory round trip per 16
// rows instead of per 4), and the MFMAs run in row order, steps past K64 skipped.
template <int WM, int WN>
__device__ __forceinline__ void head_fp64(const double* __restrict__ A64, int64_t lda64,
                                          const double* __restrict__ B64, int64_t ldb64,
                                          int64_t K64, int g, const int64_t (&ph)[WM],
                                          const int64_t (&jcol)[WN], v4d (&h)[WM][WN]) {
  for (int64_t k0 = 0; k0 < K64; k0 += 16) {
    double ha[4][WM], hb[4][WN];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t k = k0 + 4 * u + g;
      const bool in = k < K64;
      const int64_t kc = in ? k : K64 - 1;
#pragma unroll
      for (int fm = 0; fm < WM; ++fm) {
        const double v = A64[kc * lda64 + ph[fm]];
        ha[u][fm] = in ? v : 0.0;
      }
#pragma unroll
      for (int fn = 0; fn < WN; ++fn) {
        const double v = B64[kc * ldb64 + jcol[fn]];
        hb[u][fn] = in ? v : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (k0 + 4 * u >= K64) break;
#pragma unroll
      for (int fm = 0; fm < WM; ++fm)
#pragma unroll
        for (int fn = 0; fn < WN; ++fn) h[fm][fn] = mfma(ha[u][fm], hb[u][fn], h[fm][fn]);
    }
  }
}

// Optional FP64 head (FP32 operands only): rows k < K64 of A64 (K64 x P) and B64 (K64 x n) are
// contracted first with the FP64 MFMA, straight into the FP64 accumulators.  Lane li supplies the
// A row of point 4*(li & 3) + (li >> 2) of its 16-point block, which puts the FP64 MFMA's result
// (row g + 4r in register r of lane group g) into the FP32 layout (row 4g + r).
template <int FN, bool kK4 = false>
__global__ __launch_bounds__(64 * kWaves) void contract_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    const double* __restrict__ offset, double* __restrict__ Y, int64_t ldy, int64_t P, int64_t n,
    int64_t K, const double* __restrict__ A64, int64_t lda64, const double* __restrict__ B64,
    int64_t ldb64, int64_t K64) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, g = lane >> 4;

  const int64_t m_base = (int64_t)blockIdx.x * kBlockM + wm * 32;
  const int64_t n_base = (int64_t)blockIdx.y * (32 * FN) + wn * (16 * FN);
  int64_t pcol[2], jcol[FN];
#pragma unroll
  for (int fm = 0; fm < 2; ++fm) pcol[fm] = min(m_base + fm * 16 + li, P - 1);
#pragma unroll
  for (int fn = 0; fn < FN; ++fn) jcol[fn] = min(n_base + fn * 16 + li, n - 1);

  v4f acc[2][FN];
  // FP64 sums of the partial tiles of kFlushK terms: in LDS (one column per thread, no sharing),
  // which keeps the register count low enough for two waves per SIMD.
  __shared__ double acc64s[2 * FN * 4][64 * kWaves];
  auto acc64 = [&](int fm, int fn, int r) -> double& {
    return acc64s[(fm * FN + fn) * 4 + r][threadIdx.x];
  };
#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      acc[fm][fn] = v4f{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) acc64(fm, fn, r) = 0.0;
    }

  if (K64 > 0) {
    int64_t ph[2];
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
      ph[fm] = min(m_base + fm * 16 + 4 * (li & 3) + (li >> 2), P - 1);
    v4d h[2][FN];
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) h[fm][fn] = v4d{0, 0, 0, 0};
    head_fp64<2, FN>(A64, lda64, B64, ldb64, K64, g, ph, jcol, h);
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc64(fm, fn, r) = h[fm][fn][r];
  }

  const int64_t K16 = K & ~(int64_t)(kChunk - 1);
  float a[2][4], b[FN][4];
  auto load = [&](int64_t k0) {
    if constexpr (kK4) {
      // k-interleaved operands: the four k of a lane's steps are one 16-byte vector
      const int64_t kq = (k0 >> 2) + g;
#pragma unroll
      for (int fm = 0; fm < 2; ++fm) {
        const v4f v = *reinterpret_cast<const v4f*>(A + (kq * lda + pcol[fm]) * 4);
        a[fm][0] = v.x;
        a[fm][1] = v.y;
        a[fm][2] = v.z;
        a[fm][3] = v.w;
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const v4f v = *reinterpret_cast<const v4f*>(B + (kq * ldb + jcol[fn]) * 4);
        b[fn][0] = v.x;
        b[fn][1] = v.y;
        b[fn][2] = v.z;
        b[fn][3] = v.w;
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int64_t k = k0 + 4 * g + s;
        const float* __restrict__ ar = A + k * lda;
        const float* __restrict__ br = B + k * ldb;
#pragma unroll
        for (int fm = 0; fm < 2; ++fm) a[fm][s] = ar[pcol[fm]];
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) b[fn][s] = br[jcol[fn]];
      }
    }
  };
  auto step = [&]() {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int fm = 0; fm < 2; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = mfma(a[fm][s], b[fn][s], acc[fm][fn]);
  };
  auto flush = [&]() {
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc64(fm, fn, r) += (double)acc[fm][fn][r];
        acc[fm][fn] = v4f{0, 0, 0, 0};
      }
  };

  auto chunk = [&](int64_t k0) {
    float ca[2][4], cb[FN][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int fm = 0; fm < 2; ++fm) ca[fm][s] = a[fm][s];
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) cb[fn][s] = b[fn][s];
    }
    if (k0 + kChunk < K16) load(k0 + kChunk);  // next chunk in flight during this one
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int fm = 0; fm < 2; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = mfma(ca[fm][s], cb[fn][s], acc[fm][fn]);
  };
  if (K16 > 0) {
    load(0);
    if constexpr (kK4) {
      // the chunks of one kFlushK run form an inner loop with the flush after it, so the MFMA
      // accumulators stay in the matrix-core registers across the run (a flush test inside the
      // chunk loop made the compiler copy them to and from ordinary registers at every chunk).  The
      // plain FP32 layout keeps the flat loop (3.73 ms flat, 4.53 ms nested).  Same sums.
      for (int64_t kc = 0; kc < K16; kc += kFlushK) {
        const int64_t kce = min(K16, kc + (int64_t)kFlushK);
        for (int64_t k0 = kc; k0 < kce; k0 += kChunk) chunk(k0);
        if (kce % kFlushK == 0) flush();  // a run cut short by K16 is flushed after the tail
      }
    } else {
      for (int64_t k0 = 0; k0 < K16; k0 += kChunk) {
        chunk(k0);
        if (((k0 + kChunk) % kFlushK) == 0) flush();
      }
    }
  }
  if (!kK4 && K16 < K) {  // last partial chunk: rows k >= K contribute zero (K4: K % 16 == 0)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t k = K16 + 4 * g + s;
      const bool in = k < K;
      const int64_t kc = in ? k : K - 1;
#pragma unroll
      for (int fm = 0; fm < 2; ++fm) {
        const float v = A[kc * lda + pcol[fm]];
        a[fm][s] = in ? v : 0.0f;
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const float v = B[kc * ldb + jcol[fn]];
        b[fn][s] = in ? v : 0.0f;
      }
    }
    step();
  }
  flush();

#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      const int64_t col = n_base + fn * 16 + li;
      if (col >= n) continue;
      const double off = offset ? offset[col] : 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // result layout: row 4g + r in register r of lane group g, column lane % 16
        const int64_t row = m_base + fm * 16 + (4 * g + r);
        const double v = acc64(fm, fn, r);
        if (row < P) Y[row * ldy + col] = off + v;
      }
    }
}

// Outputs per workgroup tile (32 * FN): 128 for wide outputs, 64 when 128-wide tiles would leave
// fewer than two workgroups per CU (8192 points x 256 outputs: 0.337 ms for the mixed step
// against 0.371 ms); a tile's results do not depend on its width (same bits).
inline int64_t tile_n(int64_t P, int64_t n) {
  if (n <= 32) return 32;
  if (n <= 64) return 64;
  const int64_t gm = (P + kBlockM - 1) / kBlockM;
  return gm * ((n + 127) / 128) < 512 ? 64 : 128;
}

// ------------------------------------------------------------------------------------------
// Split-k form of contract_kernel for small batches: the kFlushK-chunks of k are spread over
// blockIdx.z (chunks [z * cps, (z + 1) * cps) per slice) and slice z = nsplit computes the FP64
// head; every chunk's partial tile (the MFMA accumulators of its kFlushK terms, exactly what
// contract_kernel adds into its FP64 sums at that flush) is written to `part`, the head to
// `head`, and contract_reduce_kernel adds them in contract_kernel's order: the same bits.
// ------------------------------------------------------------------------------------------
template <int FN, bool kK4>
__global__ __launch_bounds__(64 * kWaves) void contract_split_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb, int64_t P,
    int64_t n, int64_t K, const double* __restrict__ A64, int64_t lda64,
    const double* __restrict__ B64, int64_t ldb64, int64_t K64, int64_t cps, int nsplit,
    float* __restrict__ part, double* __restrict__ head) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, g = lane >> 4;
  const int64_t m_base = (int64_t)blockIdx.x * kBlockM + wm * 32;
  const int64_t n_base = (int64_t)blockIdx.y * (32 * FN) + wn * (16 * FN);
  const int64_t Pn = P * n;
  int64_t pcol[2], jcol[FN];
#pragma unroll
  for (int fm = 0; fm < 2; ++fm) pcol[fm] = min(m_base + fm * 16 + li, P - 1);
#pragma unroll
  for (int fn = 0; fn < FN; ++fn) jcol[fn] = min(n_base + fn * 16 + li, n - 1);
  // element (fm, fn, r) of this lane: row and column of Y
  auto out_at = [&](int fm, int fn, int r, int64_t& row, int64_t& col) {
    row = m_base + fm * 16 + (4 * g + r);
    col = n_base + fn * 16 + li;
  };

  if ((int)blockIdx.z == nsplit) {  // the FP64 head
    int64_t ph[2];
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
      ph[fm] = min(m_base + fm * 16 + 4 * (li & 3) + (li >> 2), P - 1);
    v4d h[2][FN];
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) h[fm][fn] = v4d{0, 0, 0, 0};
    head_fp64<2, FN>(A64, lda64, B64, ldb64, K64, g, ph, jcol, h);
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int64_t row, col;
          out_at(fm, fn, r, row, col);
          if (row < P && col < n) head[row * n + col] = h[fm][fn][r];
        }
    return;
  }

  const int64_t nch = (K + kFlushK - 1) / kFlushK;
  const int64_t c0 = (int64_t)blockIdx.z * cps, c1 = min(nch, c0 + cps);
  if (c0 >= c1) return;
  const int64_t K16 = K & ~(int64_t)(kChunk - 1);
  v4f acc[2][FN];
#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = v4f{0, 0, 0, 0};
  int64_t cur = c0;  // chunk whose partial tile is accumulating
  auto emit = [&]() {
#pragma unroll
    for (int fm = 0; fm < 2; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          int64_t row, col;
          out_at(fm, fn, r, row, col);
          if (row < P && col < n) part[cur * Pn + row * n + col] = acc[fm][fn][r];
        }
        acc[fm][fn] = v4f{0, 0, 0, 0};
      }
    ++cur;
  };

  float a[2][4], b[FN][4];
  auto load = [&](int64_t k0) {
    if constexpr (kK4) {
      const int64_t kq = (k0 >> 2) + g;
#pragma unroll
      for (int fm = 0; fm < 2; ++fm) {
        const v4f v = *reinterpret_cast<const v4f*>(A + (kq * lda + pcol[fm]) * 4);
        a[fm][0] = v.x;
        a[fm][1] = v.y;
        a[fm][2] = v.z;
        a[fm][3] = v.w;
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const v4f v = *reinterpret_cast<const v4f*>(B + (kq * ldb + jcol[fn]) * 4);
        b[fn][0] = v.x;
        b[fn][1] = v.y;
        b[fn][2] = v.z;
        b[fn][3] = v.w;
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int64_t k = k0 + 4 * g + s;
        const float* __restrict__ ar = A + k * lda;
        const float* __restrict__ br = B + k * ldb;
#pragma unroll
        for (int fm = 0; fm < 2; ++fm) a[fm][s] = ar[pcol[fm]];
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) b[fn][s] = br[jcol[fn]];
      }
    }
  };

  const int64_t kb = c0 * kFlushK, ke = min(c1 * kFlushK, K16);
  if (kb < ke) {
    load(kb);
    // one inner loop per kFlushK chunk, emitted after it (accumulators stay in place)
    for (int64_t kc = kb; kc < ke; kc += kFlushK) {
      const int64_t kce = min(ke, kc + (int64_t)kFlushK);
      for (int64_t k0 = kc; k0 < kce; k0 += kChunk) {
        float ca[2][4], cb[FN][4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
          for (int fm = 0; fm < 2; ++fm) ca[fm][s] = a[fm][s];
#pragma unroll
          for (int fn = 0; fn < FN; ++fn) cb[fn][s] = b[fn][s];
        }
        if (k0 + kChunk < ke) load(k0 + kChunk);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int fm = 0; fm < 2; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn)
              acc[fm][fn] = mfma(ca[fm][s], cb[fn][s], acc[fm][fn]);
      }
      if (kce % kFlushK == 0) emit();
    }
  }
  if (!kK4 && c1 == nch && K16 < K) {  // last partial chunk of 16: rows k >= K contribute zero
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t k = K16 + 4 * g + s;
      const bool in = k < K;
      const int64_t kc = in ? k : K - 1;
#pragma unroll
      for (int fm = 0; fm < 2; ++fm) {
        const float v = A[kc * lda + pcol[fm]];
        a[fm][s] = in ? v : 0.0f;
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        const float v = B[kc * ldb + jcol[fn]];
        b[fn][s] = in ? v : 0.0f;
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int fm = 0; fm < 2; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = mfma(a[fm][s], b[fn][s], acc[fm][fn]);
  }
  if (cur < c1) emit();  // the slice's last chunk when K ends inside it
}

// Y[p, j] = offset[j] + (((head + part_0) + part_1) + ...) (+ 0.0 when K is a multiple of
// kFlushK: contract_kernel's final flush then adds an empty partial tile), head = 0 without one.
// kGrouped (FP64 chains): the sums of `per` chains first, then theirs.
template <typename E, bool kGrouped>
__global__ __launch_bounds__(256) void contract_reduce_kernel(const E* __restrict__ part,
                                                              int64_t nch, int64_t per,
                                                              const double* __restrict__ head,
                                                              const double* __restrict__ offset,
                                                              double* __restrict__ Y, int64_t ldy,
                                                              int64_t P, int64_t n, int64_t K) {
  const int64_t Pn = P * n;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < Pn;
       i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / n, col = i - row * n;
    double v = head ? head[i] : 0.0;
    if constexpr (!kGrouped) {
      for (int64_t c = 0; c < nch; c += 4) {  // four loads in flight, also where fewer are left
        E q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = part[min(c + u, nch - 1) * Pn + i];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (c + u < nch) v += (double)q[u];
      }
    } else {
      for (int64_t c = 0; c < nch; c += per) {
        double s = 0.0;
#pragma unroll 8
        for (int64_t u = c; u < min(nch, c + per); ++u) s += (double)part[u * Pn + i];
        v += s;
      }
    }
    if (K % kFlushK == 0) v += 0.0;
    const double off = offset ? offset[col] : 0.0;
    Y[row * ldy + col] = off + v;
  }
}

// Split plan for a contraction of P points x n outputs: the slices of k (0: no split) and chunks
// per slice.  A launch of fewer than kSplitMinGroups workgroups is split so that about
// kSplitTarget workgroups run (small batches: the k loop of one workgroup is the latency).
constexpr int64_t kSplitMinGroups = 256;
constexpr int64_t kSplitTarget = 512;
constexpr int64_t kSplitMaxBytes = int64_t(256) << 20;  // workspace of one split call
struct SplitPlan {
  int64_t nsplit = 0, cps = 0, nch = 0, part_bytes = 0, head_bytes = 0;
};
SplitPlan split_plan(int64_t P, int64_t n, int64_t K, int64_t K64) {
  SplitPlan sp;
  const int64_t gm = (P + kBlockM - 1) / kBlockM;
  const int64_t tn = tile_n(P, n);
  const int64_t groups = gm * ((n + tn - 1) / tn);
  sp.nch = (K + kFlushK - 1) / kFlushK;
  if (P <= 0 || n <= 0 || groups >= kSplitMinGroups || (sp.nch < 2 && K64 == 0)) return sp;
  int64_t want = (kSplitTarget + groups - 1) / groups;
  if (want > sp.nch) want = sp.nch;
  if (want < 1) want = 1;
  sp.cps = sp.nch > 0 ? (sp.nch + want - 1) / want : 0;
  sp.nsplit = sp.cps > 0 ? (sp.nch + sp.cps - 1) / sp.cps : 0;
  if (sp.nsplit + (K64 > 0 ? 1 : 0) < 2) {  // one slice: nothing to gain
    sp = SplitPlan{};
    return sp;
  }
  sp.part_bytes = (sp.nch * P * n * (int64_t)sizeof(float) + 255) / 256 * 256;
  sp.head_bytes = K64 > 0 ? P * n * 8 : 0;
  if (sp.part_bytes + sp.head_bytes > kSplitMaxBytes || sp.nsplit >= 65535) sp = SplitPlan{};
  return sp;
}

template <bool kK4>
int contract_split_launch(const SplitPlan& sp, const float* A, int64_t lda, const float* B, int64_t ldb,
                          const double* offset, double* Y, int64_t ldy, int64_t P, int64_t n,
                          int64_t K, const double* A64, int64_t lda64, const double* B64,
                          int64_t ldb64, int64_t K64, void* ws, hipStream_t st) {
  float* part = (float*)ws;
  double* head = K64 > 0 ? (double*)((char*)ws + sp.part_bytes) : nullptr;
  const dim3 block(64 * kWaves);
  const unsigned gm = (unsigned)((P + kBlockM - 1) / kBlockM);
  const unsigned gz = (unsigned)(sp.nsplit + (K64 > 0 ? 1 : 0));
  const int ns = (int)sp.nsplit;
  const int64_t tn = tile_n(P, n);
  if (tn == 32) {
    hipLaunchKernelGGL((contract_split_kernel<1, kK4>), dim3(gm, (unsigned)((n + 31) / 32), gz),
                       block, 0, st, A, lda, B, ldb, P, n, K, A64, lda64, B64, ldb64, K64, sp.cps,
                       ns, part, head);
  } else if (tn == 64) {
    hipLaunchKernelGGL((contract_split_kernel<2, kK4>), dim3(gm, (unsigned)((n + 63) / 64), gz),
                       block, 0, st, A, lda, B, ldb, P, n, K, A64, lda64, B64, ldb64, K64, sp.cps,
                       ns, part, head);
  } else {
    hipLaunchKernelGGL((contract_split_kernel<4, kK4>),
                       dim3(gm, (unsigned)((n + 127) / 128), gz), block, 0, st, A, lda, B, ldb, P,
                       n, K, A64, lda64, B64, ldb64, K64, sp.cps, ns, part, head);
  }
  SBI_HIP_CHECK(hipGetLastError());
  const int64_t Pn = P * n;
  int64_t rg = (Pn + 255) / 256;
  if (rg > 4096) rg = 4096;
  hipLaunchKernelGGL((contract_reduce_kernel<float, false>), dim3((unsigned)rg), dim3(256), 0, st, part,
                     sp.nch, int64_t(1), head, offset, Y, ldy, P, n, K);
  SBI_HIP_CHECK(hipGetLastError());
  return SBI_OK;
}

// ------------------------------------------------------------------------------------------
// FP64 contraction.  Bound: v_mfma_f64_16x16x4, 64 cycles of a SIMD per 2048 operations (measured
// ceiling of a large library product on this card: 72 TFLOP/s).  The operands need only 16 bytes
// per cycle and CU, so what matters is that several waves per SIMD always have their fragments at
// hand: operands are staged in LDS, three buffers of 16 k, copied two chunks ahead by direct
// global -> LDS loads (one barrier per chunk), and the register count allows three waves per SIMD.
// 8192 points x 256 outputs, K 5000: 340-376 us (matrix cores busy 85 % of the time, 2.15 GHz) against
// 402-412 us with each wave loading its own fragments from L2 one chunk ahead; 5000 x 160, K 10 002 (k
// over workgroups): 478 -> 305 us; 5000 x 8192, K 256: 487 -> 380-430 us.  Requesting a whole
// chunk's fragments before its first MFMA costs a wave per SIMD's worth of registers (5730 us).
//
// Work split: a workgroup of 4 waves owns a (32 * WM)-point x (32 * WN)-output tile, each wave 16 * WM
// points x 16 * WN outputs; the last output tile with at most 32 outputs left is cut into four waves of
// 16 points x 32 outputs instead, so that no wave works on outputs past the edge (160 outputs:
// 17 % less matrix work).  WN = 1 for at most 32 outputs; WM = 1 (32 points) where that fills the CUs
// better (f64_plan).  The output tiles of one point tile run
// on one XCD (its L2 serves their A rows).
//
// LDS image of a chunk: rows of the tile's width; the 16-byte slot q of row r holds the elements
// of slot q ^ (8 * ((r >> 2) & 1)) (step s multiplies rows s, 4 + s, 8 + s, 12 + s), so the two rows that half a wave reads together lie in different
// halves of the banks.  kDirect = false: row strides, widths or bases that are not multiples of
// 16 bytes go through registers (8-byte loads one chunk ahead); the same image, the same bits.
//
// Sums: the MFMA accumulators hold a chain of kFlushK terms, the chains are added into the sum of a
// slice (a third of K), the three slice sums in order, so the rounding grows with kFlushK + K / (3
// kFlushK) + 3 terms.  Grids that would leave CUs idle spread k over workgroups (f64_plan), a
// slice or some chains each; they write the sums of these units to `part` and
// contract_reduce_kernel adds them in the same order: the same bits for any P, alone or in a batch.
// `ordered` (sbi_contract): one slice, the chains added in order, never spread.
// ------------------------------------------------------------------------------------------
constexpr int kF64Slices = 3;
constexpr int kF64Buf = 3;
constexpr int kPanel = 4;  // point tiles an XCD works on side by side (contract_k4_kernel)
// k per slice (the last one may be shorter): whole chunks, one slice up to three chains
inline int64_t f64_slice(int64_t K) {
  if (K <= kF64Slices * kFlushK) return std::max<int64_t>(K, 1);
  const int64_t third = (K + kF64Slices - 1) / kF64Slices;
  return (third + kChunk - 1) / kChunk * kChunk;
}
enum { kWhole = 0, kBySlice = 1, kByChain = 2 };  // how k is spread over workgroups (kSplit)

template <int WM, int WN, bool kDirect, int kSplit>
__global__ __launch_bounds__(64 * kWaves, WM * WN < 4 ? 4 : 3) void contract_f64_kernel(
    const double* __restrict__ A, int64_t lda, const double* __restrict__ B, int64_t ldb,
    const double* __restrict__ offset, double* __restrict__ Y, int64_t ldy, int64_t P, int64_t n,
    int64_t K, int ntm, int ntn, int nz, int64_t slice, int upz, double* __restrict__ part) {
  constexpr int TM = 32 * WM, TN = 32 * WN;
  constexpr int kA = kChunk * TM * 8, kStep = kA + kChunk * TN * 8;  // bytes of a chunk: A, then B
  constexpr int nA = kA / 1024, kPer = kStep / 4096;                 // 1 KB copies: of A, per wave
  static_assert(kStep % 4096 == 0, "whole copies per wave");
  __shared__ __attribute__((aligned(16))) char smem[kF64Buf * kStep];
  const int L = blockIdx.x;
  const int idx = L >> 3;
  const int tn = idx % ntn;
  const int pair = (idx / ntn) * 8 + (L & 7);
  if (pair >= ntm * nz) return;
  const int tm = pair % ntm, z = pair / ntm;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;
  const bool thin = WM == 2 && WN == 2 && n - n0 <= 32;  // 4 x 1 waves of 16 x 32 instead of 2 x 2 of 32 x 32
  const int mw = thin ? wave * 16 : (wave & 1) * (16 * WM);
  const int nw = thin ? 0 : (wave >> 1) * (16 * WN);
  // k in chunks: KC of them, sc per slice; chain u (kByChain: upz of them per workgroup, in slices
  // of `per`) starts at chunk c_of(u); this workgroup takes [cb, ce)
  const int KC = (int)((K + kChunk - 1) / kChunk), KF = (int)(K / kChunk);
  const int sc = (int)((slice + kChunk - 1) / kChunk), cpc = kFlushK / kChunk;
  const int per = (sc + cpc - 1) / cpc;
  auto c_of = [&](int u) { return min(KC, (u / per) * sc + (u % per) * cpc); };
  const int cb = kSplit == kWhole ? 0 : kSplit == kBySlice ? z * sc : c_of(z * upz);
  const int ce = kSplit == kWhole ? KC : kSplit == kBySlice ? min(KC, cb + sc) : c_of((z + 1) * upz);

  // copy i of this wave: 128 consecutive elements of the LDS image, two per lane (columns past
  // the edge re-read the last pair or element, rows past K row K - 1: never used).  The address is
  // a scalar base that advances by a chunk plus this lane's fixed offset: every vector instruction
  // in the loop takes time from the matrix cores (23 per chunk: 437 us, 4 per chunk: 400 us, 8192 x
  // 256, K 5000).
  typedef typename std::conditional<kDirect, uint32_t, uint64_t>::type off_t;
  const char* baseA = (const char*)(A + m0 + (int64_t)cb * kChunk * lda);  // of the next chunk
  const char* baseB = (const char*)(B + n0 + (int64_t)cb * kChunk * ldb);
  auto krow = [&](int i) {
    const int c = wave + 4 * i;
    return 4 * i < nA ? (c * 128 + lane * 2) / TM : ((c - nA) * 128 + lane * 2) / TN;
  };
  off_t col[kPer], voff[kPer];  // bytes from the base to this lane's pair: in its row, in all
  uint32_t odd = 0;  // bit i: the pair's second element is past the edge (kDirect = false)
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = wave + 4 * i;
    const bool isA = 4 * i < nA;
    const int T = isA ? TM : TN;
    const int pos = (isA ? c : c - nA) * 128 + lane * 2;
    const int64_t org = isA ? m0 : n0;
    const int64_t at = org + (((pos % T) / 2) ^ (8 * ((krow(i) >> 2) & 1))) * 2, end = isA ? P : n;
    if (!kDirect && at + 1 >= end) odd |= 1u << i;
    col[i] = (off_t)((min(at, kDirect ? (end - 1) & ~(int64_t)1 : end - 1) - org) * 8);
    voff[i] = col[i] + (off_t)krow(i) * (off_t)((isA ? lda : ldb) * 8);
  }
  int ci = cb;  // the next chunk to be copied
  double pend[kDirect ? 1 : 2 * kPer];
  auto advance = [&](auto&& put) {
    if (ci >= KF) {  // the last rows of K
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        voff[i] = col[i] + (off_t)min(krow(i), (int)(K - 1 - (int64_t)ci * kChunk)) *
                               (off_t)((4 * i < nA ? lda : ldb) * 8);
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) put(i, (const double*)((4 * i < nA ? baseA : baseB) + voff[i]));
    baseA += kChunk * 8 * lda;
    baseB += kChunk * 8 * ldb;
    ++ci;
  };
  auto fetch = [&] {  // kDirect = false: the next chunk into registers
    if (ci < ce)
      advance([&](int i, const double* p) {
        pend[2 * i] = p[0];
        pend[2 * i + 1] = p[(odd >> i) & 1 ? 0 : 1];
      });
  };
  auto issue = [&](int b) {  // the next chunk into buffer b
    char* dst = smem + b * kStep + wave * 1024;
    if constexpr (kDirect) {
      if (ci < ce)
        advance([&](int i, const double* p) {
          __builtin_amdgcn_global_load_lds((const void*)p, (lds_void*)(dst + i * 4096), 16, 0, 0);
        });
    } else {
      typedef double v2d __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        *(v2d*)(dst + i * 4096 + lane * 16) = v2d{pend[2 * i], pend[2 * i + 1]};
      fetch();
    }
  };
  // chunk c has landed in every wave (the copies of the next one may be in flight)
  auto wait = [&](int c) {
    if constexpr (kDirect) {
      if (c + 1 < ce) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kPer) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
    } else {
      __syncthreads();
    }
  };

  int bi = 0;  // buffer of the chunk being computed
  const int sw = 16 * (g & 1);
  if (cb < ce) {
    if constexpr (kDirect) {
      issue(0);
      issue(1);
    } else {
      fetch();
      issue(0);
    }
  }
  // the walk over k, once for whole tiles and once for thin ones: a test inside a chunk would cut its
  // matrix instructions into pairs that each wait for their LDS reads
  auto walk = [&](auto thin_tile) {
    constexpr bool kThin = decltype(thin_tile)::value;
    constexpr int M = kThin ? 1 : WM;
    v4d total[M][WN], sum[M][WN], acc[M][WN];
    auto each = [&](auto&& f) {  // the fragments of this wave
#pragma unroll
      for (int fm = 0; fm < M; ++fm)
#pragma unroll
        for (int fn = 0; fn < WN; ++fn) f(fm, fn);
    };
    each([&](int fm, int fn) { total[fm][fn] = v4d{0, 0, 0, 0}; });
    uint32_t pa[M], pb[WN];  // byte offsets of this lane's elements in a buffer
#pragma unroll
    for (int fm = 0; fm < M; ++fm) pa[fm] = (uint32_t)(4 * g * TM + ((mw + fm * 16 + li) ^ sw)) * 8;
#pragma unroll
    for (int fn = 0; fn < WN; ++fn) pb[fn] = (uint32_t)(kA + (4 * g * TN + ((nw + fn * 16 + li) ^ sw)) * 8);
    auto compute = [&](int c, bool tail) {
      const char* buf = smem + bi * kStep;
#pragma unroll
      for (int s = 0; s < kChunk / 4; ++s) {
        double a[M], b[WN];
#pragma unroll
        for (int fm = 0; fm < M; ++fm) a[fm] = *(const double*)(buf + pa[fm] + s * 8 * TM);
#pragma unroll
        for (int fn = 0; fn < WN; ++fn) b[fn] = *(const double*)(buf + pb[fn] + s * 8 * TN);
        if (tail && (int64_t)c * kChunk + 4 * g + s >= K) {
#pragma unroll
          for (int fm = 0; fm < M; ++fm) a[fm] = 0.0;
#pragma unroll
          for (int fn = 0; fn < WN; ++fn) b[fn] = 0.0;
        }
        // a wave with its operands at hand goes ahead of those that address and wait (400 -> 375 us)
        __builtin_amdgcn_s_setprio(1);
        each([&](int fm, int fn) { acc[fm][fn] = mfma(a[fm], b[fn], acc[fm][fn]); });
        __builtin_amdgcn_s_setprio(0);
      }
    };
    auto chain = [&](int c0, int c1) {  // acc = the sum over the chunks [c0, c1)
      each([&](int fm, int fn) { acc[fm][fn] = v4d{0, 0, 0, 0}; });
      const int cf = min(c1, KF);
      for (int c = c0; c < cf; ++c) {
        wait(c);
        issue(kDirect ? (bi == 0 ? kF64Buf - 1 : bi - 1) : (bi + 1 == kF64Buf ? 0 : bi + 1));
        compute(c, false);
        bi = bi + 1 == kF64Buf ? 0 : bi + 1;
      }
      if (cf < c1) {
        wait(cf);
        compute(cf, true);
      }
    };
    auto row_of = [&](int fm, int r) { return m0 + mw + fm * 16 + g + 4 * r; };
    auto col_of = [&](int fn) { return n0 + nw + fn * 16 + li; };
    auto emit = [&](int64_t unit, v4d(&v)[M][WN]) {
      double* __restrict__ out = part + unit * P * n;
      each([&](int fm, int fn) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int64_t row = row_of(fm, r), col = col_of(fn);
          if (row < P && col < n) out[row * n + col] = v[fm][fn][r];
        }
      });
    };
    if constexpr (kSplit == kByChain) {
      for (int u = z * upz; c_of(u) < ce; ++u) {
        chain(c_of(u), c_of(u + 1));
        emit(u, acc);
      }
      return;
    }
    for (int c0 = cb; c0 < ce; c0 += sc) {
      const int c1 = min(ce, c0 + sc);
      each([&](int fm, int fn) { sum[fm][fn] = v4d{0, 0, 0, 0}; });
      for (int c = c0; c < c1; c += cpc) {
        chain(c, min(c1, c + cpc));
        each([&](int fm, int fn) { sum[fm][fn] += acc[fm][fn]; });
      }
      if constexpr (kSplit == kWhole) each([&](int fm, int fn) { total[fm][fn] += sum[fm][fn]; });
      else emit(z, sum);
    }
    if constexpr (kSplit != kWhole) return;
    each([&](int fm, int fn) {
      const int64_t col = col_of(fn);
      const double off = offset ? offset[min(col, n - 1)] : 0.0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = row_of(fm, r);
        if (row < P && col < n) Y[row * ldy + col] = off + total[fm][fn][r];
      }
    });
  };
  if constexpr (WM == 2 && WN == 2) {
    if (thin) return walk(std::true_type{});
  }
  walk(std::false_type{});
}

// How contract_f64_kernel spreads the work: tiles of 64 or 32 points, and k not at all (nz = 1, no
// workspace), a slice per workgroup, or upz chains each, whichever takes least by this estimate.
// A CU holds three workgroups of the larger tile (four of the smaller, 16 % slower per point); alone
// one reaches about half of the matrix cores' rate, two 0.8 of it.  So a CU that gets q workgroups
// takes as long as q of them at the full rate, and more for the last one or two.  The partial
// sums are written and read once, at about 4.5 TB/s, by a second launch.
// 5000 x 160, K 10 002: 388 us with slices of 2048 dealt to equal numbers of workgroups, 315 us by
// thirds; 8192 x 256, K 5000: 435 and 376 us; 2000 x 2000 of an evaluation with K 660: 272 us with
// tiles of 64 points (1024 tiles, four per CU), 248 us of 32; 500 x 64, K 9986: 472 us unsplit, 104
// us by slices, 31 us by chains.
struct F64Plan {
  int64_t nz = 1, units = 0, per = 1, bytes = 0;
  int split = kWhole, upz = 1, wm = 2;  // wm: 32 wm points per tile
};
inline int64_t f64_tile_n(int64_t n) { return n <= 32 ? 32 : 64; }
F64Plan f64_plan(int64_t P, int64_t n, int64_t K, bool may_split = true) {
  F64Plan best;
  if (P <= 0 || n <= 0) return best;
  const int64_t tn = f64_tile_n(n), tiles = (P + kBlockM - 1) / kBlockM * ((n + tn - 1) / tn);
  const int64_t slice = f64_slice(K), slices = (K + slice - 1) / slice;
  const int64_t per = (slice + kFlushK - 1) / kFlushK;
  const int64_t chains = (slices - 1) * per + (K - (slices - 1) * slice + kFlushK - 1) / kFlushK;
  // microseconds of `each` chains in every one of nz workgroups per tile, and of the partial sums
  auto cost = [&](int64_t nz, double each, int64_t units) {
    const double chain = 64.0 * tn * 2 * kFlushK / (72e6 / 256);
    const int64_t q = (tiles * nz + 255) / 256, rest = q % 3;
    const double rounds = (double)(q - rest) + (rest == 1 ? 2.0 : rest == 2 ? 2.5 : 0.0);
    const double bytes = (double)units * P * n * 16;
    return rounds * (each * chain + 2.0) + (units ? 6.0 + bytes / 4.5e6 : 0.0);
  };
  double least = cost(1, (double)K / kFlushK, 0);
  {
    const int64_t q = ((P + 31) / 32 * ((n + tn - 1) / tn) + 255) / 256, rest = q % 4;
    const double half[4] = {0.0, 1.0, 1.25, 1.7};
    const double chain = 64.0 * tn * 2 * kFlushK / (72e6 / 256);
    const double c = (0.58 * (double)(q - rest) + half[rest]) * ((double)K / kFlushK * chain + 2.0);
    if (c < least) {
      least = c;
      best.wm = 1;
    }
  }
  if (K <= kFlushK || !may_split) return best;
  auto consider = [&](int split, int64_t nz, double each, int64_t units, int64_t upz) {
    if (nz < 2 || units * P * n * 8 > kSplitMaxBytes) return;
    const double c = cost(nz, each, units);
    if (c >= least) return;
    least = c;
    best.wm = 2;
    best.split = split;
    best.nz = nz;
    best.units = units;
    best.per = split == kByChain ? per : 1;
    best.upz = (int)upz;
    best.bytes = units * P * n * 8;
  };
  consider(kBySlice, slices, (double)slice / kFlushK, slices, 1);
  for (int64_t upz = 1; upz <= std::min<int64_t>(chains, 64); ++upz)
    consider(kByChain, (chains + upz - 1) / upz, (double)upz, chains, upz);
  return best;
}

typedef void (*f64_kernel_t)(const double*, int64_t, const double*, int64_t, const double*, double*,
                             int64_t, int64_t, int64_t, int64_t, int, int, int, int64_t, int, double*);
template <int WN, bool kDirect>
f64_kernel_t f64_kernel(int wm, int split) {
  if (split == kBySlice) return contract_f64_kernel<2, WN, kDirect, kBySlice>;
  if (split == kByChain) return contract_f64_kernel<2, WN, kDirect, kByChain>;
  return wm == 1 ? contract_f64_kernel<1, WN, kDirect, kWhole>
                 : contract_f64_kernel<2, WN, kDirect, kWhole>;
}

// padded: every row of A (B) is readable up to P (n) rounded up to a multiple of two.
int contract_f64(const double* A, int64_t lda, const double* B, int64_t ldb, const double* offset,
                 double* Y, int64_t ldy, int64_t P, int64_t n, int64_t K, bool padded, bool ordered,
                 void* ws, int64_t ws_bytes, hipStream_t st) {
  F64Plan pl = f64_plan(P, n, K, !ordered);
  if (!ws || ws_bytes < pl.bytes) pl = f64_plan(P, n, K, false);
  const bool direct = K == 0 || (((uintptr_t)A | (uintptr_t)B) % 16 == 0 && lda % 2 == 0 &&
                                 ldb % 2 == 0 && std::max(lda, ldb) < (1 << 24) &&  // 32-bit offsets
                                 (padded || (P % 2 == 0 && n % 2 == 0)));
  const int64_t tn = f64_tile_n(n), ntn = (n + tn - 1) / tn;
  const int wm = pl.wm;
  const int64_t ntm = (P + 32 * wm - 1) / (32 * wm);
  const int64_t grid = ((ntm * pl.nz + 7) / 8) * 8 * ntn;
  if (grid > 0x7fffffff) {
    sbi::set_error("sbi_contract: launch too large");
    return SBI_ERR_INVALID;
  }
  const f64_kernel_t kernel = tn == 32 ? (direct ? f64_kernel<1, true>(wm, pl.split)
                                                 : f64_kernel<1, false>(wm, pl.split))
                                       : (direct ? f64_kernel<2, true>(wm, pl.split)
                                                 : f64_kernel<2, false>(wm, pl.split));
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * kWaves), 0, st, A, lda, B, ldb, offset,
                     Y, ldy, P, n, K, (int)ntm, (int)ntn, (int)pl.nz, ordered ? std::max<int64_t>(K, 1) : f64_slice(K), pl.upz, (double*)ws);
  SBI_HIP_CHECK(hipGetLastError());
  if (pl.nz > 1) {
    const int64_t rg = std::min<int64_t>((P * n + 255) / 256, 4096);
    const auto reduce = pl.per > 1 ? contract_reduce_kernel<double, true>
                                   : contract_reduce_kernel<double, false>;
    hipLaunchKernelGGL(reduce, dim3((unsigned)rg), dim3(256), 0, st, (const double*)ws, pl.units,
                       pl.per, nullptr, offset, Y, ldy, P, n, K);
    SBI_HIP_CHECK(hipGetLastError());
  }
  return SBI_OK;
}

// ------------------------------------------------------------------------------------------
// FP32 contraction with k-interleaved operands, staged in LDS: contract_kernel<., true> with
// other tiles and the same sums (the FP64 head first, chains of kFlushK terms from the FP32
// MFMA added into FP64 in order), so the same bits.  Bound: v_mfma_f32_16x16x4, 32 cycles of a SIMD.
// A workgroup of 4 waves (2 x 2) owns 32 WM points x 32 WN outputs; a chunk of 4 KQ k is copied into
// one of three LDS buffers by direct 16-byte loads two chunks ahead (one barrier per chunk, as in
// contract_f64_kernel), and one 16-byte LDS read gives a lane its operand of four steps.
// The output tiles run over XCDs by point tile, four point tiles at a time, so that the chunks of A
// and B that an XCD's workgroups read at about the same time fit its L2.
// 4096 x 4096, K 9986: 3.24 ms with each wave loading its own fragments from L2, 2.78 ms with 4 x 4
// fragments per wave (matrix cores busy 85 % of the time at 2.15 GHz), 2.95 with 4 x 2, 3.08 with 2 x
// 2 and chunks of 32 k; 5000 x 256, K 5000 (316 tiles of 2 x 2): 232 -> 212 us.  No gain from four to
// eight buffers or from reading the next chunk's fragments ahead of the MFMAs.
// ------------------------------------------------------------------------------------------
template <int WM, int WN, int KQ>
__global__ __launch_bounds__(64 * kWaves, WM * WN > 8 ? 2 : 3) void contract_k4_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    const double* __restrict__ offset, double* __restrict__ Y, int64_t ldy, int64_t P, int64_t n,
    int64_t K, const double* __restrict__ A64, int64_t lda64, const double* __restrict__ B64,
    int64_t ldb64, int64_t K64, int ntm, int ntn) {
  constexpr int TM = 32 * WM, TN = 32 * WN;
  constexpr int kA = KQ * TM * 16, kStep = kA + KQ * TN * 16;  // bytes of a chunk: A, then B
  constexpr int nA = kA / 1024, kPer = kStep / 4096;         // 1 KB copies: of A, per wave
  static_assert(nA % 4 == 0 && kStep % 4096 == 0, "whole copies per wave");
  __shared__ __attribute__((aligned(16))) char smem[kF64Buf * kStep];
  // tile t of this XCD's: its point tiles in panels (the last one may be narrower), a panel's tiles
  // output by output; no workgroup without a tile but at the end, so that none of the CUs, which
  // take the workgroups in turn, is left with those
  const int xcd = blockIdx.x & 7, t = blockIdx.x >> 3;
  const int own = (ntm - xcd + 7) / 8;
  if (t >= own * ntn) return;
  const int first = t / (kPanel * ntn) * kPanel, width = min(kPanel, own - first);
  const int in_panel = t - first * ntn;
  const int tn = in_panel / width, tm = (first + in_panel % width) * 8 + xcd;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;
  const int mw = (wave & 1) * (16 * WM), nw = (wave >> 1) * (16 * WN);

  // copies: scalar base plus this lane's fixed offset (columns past the edge re-read the last one)
  const char* baseA = (const char*)(A + m0 * 4);
  const char* baseB = (const char*)(B + n0 * 4);
  const int KR = (int)(K / 4), KC = (KR + KQ - 1) / KQ;  // rows of four k, chunks
  uint64_t voff[kPer];
  auto offsets = [&](int rows) {  // rows of the chunk (all but the last one: KQ)
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const bool isA = 4 * i < nA;
      const int idx = (isA ? wave + 4 * i : wave + 4 * i - nA) * 64 + lane;
      const int T = isA ? TM : TN;
      const int64_t at = min((isA ? m0 : n0) + idx % T, (isA ? P : n) - 1) - (isA ? m0 : n0);
      voff[i] = (uint64_t)(min(idx / T, rows - 1) * (isA ? lda : ldb) + at) * 16;
    }
  };
  offsets(KQ);
  int ci = 0;  // the next chunk to be copied
  auto issue = [&](int b) {
    if (ci >= KC) return;
    if (KQ > 4 && (ci + 1) * KQ > KR) offsets(KR - ci * KQ);
    char* dst = smem + b * kStep + wave * 1024;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      __builtin_amdgcn_global_load_lds((const void*)((4 * i < nA ? baseA : baseB) + voff[i]),
                                       (lds_void*)(dst + i * 4096), 16, 0, 0);
    baseA += lda * (16 * KQ);
    baseB += ldb * (16 * KQ);
    ++ci;
  };

  issue(0);
  issue(1);

  v4d sum[WM][WN];
#pragma unroll
  for (int fm = 0; fm < WM; ++fm)
#pragma unroll
    for (int fn = 0; fn < WN; ++fn) sum[fm][fn] = v4d{0, 0, 0, 0};
  if (K64 > 0) {
    int64_t ph[WM], jcol[WN];
#pragma unroll
    for (int fm = 0; fm < WM; ++fm)
      ph[fm] = min(m0 + mw + fm * 16 + 4 * (li & 3) + (li >> 2), P - 1);
#pragma unroll
    for (int fn = 0; fn < WN; ++fn) jcol[fn] = min(n0 + nw + fn * 16 + li, n - 1);
    head_fp64<WM, WN>(A64, lda64, B64, ldb64, K64, g, ph, jcol, sum);
  }

  uint32_t pa[WM], pb[WN];  // byte offsets of this lane's operands in a buffer
#pragma unroll
  for (int fm = 0; fm < WM; ++fm) pa[fm] = (uint32_t)(g * TM + mw + fm * 16 + li) * 16;
#pragma unroll
  for (int fn = 0; fn < WN; ++fn) pb[fn] = (uint32_t)(kA + (g * TN + nw + fn * 16 + li) * 16);
  v4f acc[WM][WN];
  int bi = 0;
  for (int c0 = 0; c0 < KC; c0 += kFlushK / (4 * KQ)) {
    const int c1 = min(KC, c0 + kFlushK / (4 * KQ));
#pragma unroll
    for (int fm = 0; fm < WM; ++fm)
#pragma unroll
      for (int fn = 0; fn < WN; ++fn) acc[fm][fn] = v4f{0, 0, 0, 0};
    for (int c = c0; c < c1; ++c) {
      if (c + 1 < KC) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kPer) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
      issue(bi == 0 ? kF64Buf - 1 : bi - 1);
#pragma unroll
      for (int h = 0; h < KQ / 4; ++h) {  // 16 k
        if (h && c * KQ + 4 * h >= KR) break;
        const char* buf = smem + bi * kStep;
        v4f a[WM], b[WN];
#pragma unroll
        for (int fm = 0; fm < WM; ++fm) a[fm] = *(const v4f*)(buf + pa[fm] + h * (64 * TM));
#pragma unroll
        for (int fn = 0; fn < WN; ++fn) b[fn] = *(const v4f*)(buf + pb[fn] + h * (64 * TN));
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int fm = 0; fm < WM; ++fm)
#pragma unroll
            for (int fn = 0; fn < WN; ++fn) acc[fm][fn] = mfma(a[fm][s], b[fn][s], acc[fm][fn]);
        __builtin_amdgcn_s_setprio(0);
      }
      bi = bi + 1 == kF64Buf ? 0 : bi + 1;
    }
#pragma unroll
    for (int fm = 0; fm < WM; ++fm)
#pragma unroll
      for (int fn = 0; fn < WN; ++fn)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[fm][fn][r] += (double)acc[fm][fn][r];
  }
#pragma unroll
  for (int fn = 0; fn < WN; ++fn) {
    const int64_t col = n0 + nw + fn * 16 + li;
    if (col >= n) continue;
    const double off = offset ? offset[col] : 0.0;
#pragma unroll
    for (int fm = 0; fm < WM; ++fm)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = m0 + mw + fm * 16 + 4 * g + r;
        if (row < P) Y[row * ldy + col] = off + sum[fm][fn][r];
      }
  }
}

template <int WM, int WN, int KQ>
void contract_k4_launch(const float* A, int64_t lda, const float* B, int64_t ldb,
                        const double* offset, double* Y, int64_t ldy, int64_t P, int64_t n,
                        int64_t K, const double* A64, int64_t lda64, const double* B64,
                        int64_t ldb64, int64_t K64, hipStream_t st) {
  const int64_t ntm = (P + 32 * WM - 1) / (32 * WM), ntn = (n + 32 * WN - 1) / (32 * WN);
  const int64_t grid = (ntm + 7) / 8 * 8 * ntn;
  hipLaunchKernelGGL((contract_k4_kernel<WM, WN, KQ>), dim3((unsigned)grid), dim3(64 * kWaves), 0, st, A,
                     lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64, K64, (int)ntm,
                     (int)ntn);
}

template <bool kK4 = false>
int contract_launch(const float* A, int64_t lda, const float* B, int64_t ldb, const double* offset,
                    double* Y, int64_t ldy, int64_t P, int64_t n, int64_t K, const double* A64,
                    int64_t lda64, const double* B64, int64_t ldb64, int64_t K64, hipStream_t st) {
  const dim3 block(64 * kWaves);
  const unsigned gm = (unsigned)((P + kBlockM - 1) / kBlockM);
  const int64_t tn = tile_n(P, n);
  if (tn == 32) {
    hipLaunchKernelGGL((contract_kernel<1, kK4>), dim3(gm, (unsigned)((n + 31) / 32)), block, 0, st,
                       A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64, K64);
  } else if constexpr (kK4) {
    // the tile that takes least: workgroups per CU that run side by side at the full rate, fewer at
    // the end at less (4 x 4 fragments: two per CU, one alone at 0.7; else three, two at 0.7, one at
    // 0.6), the smaller tiles at 0.94 and 0.88 of the largest one's rate.  12 000 x 900, K 5000: 1.36
    // ms with 4 x 4 fragments (752 workgroups, three per CU), 1.19 with 4 x 2 (whole evaluations).
    auto cost = [&](int64_t tm, int64_t tn, double size, int slots, double one, double two) {
      const int64_t q = ((P + tm - 1) / tm * ((n + tn - 1) / tn) + 255) / 256, rest = q % slots;
      return size * ((double)(q - rest) + (rest == 1 ? one : rest == 2 ? two : 0.0));
    };
    const double c44 = cost(128, 128, 4.0, 2, 1.4, 0.0), c42 = cost(128, 64, 2.0 / 0.94, 3, 1.6, 2.8),
                 c22 = cost(64, 64, 1.0 / 0.88, 3, 1.7, 2.8);
    // a short K is over before the staged tiles' pipeline pays: where two 64 x 128 tiles per CU cover
    // the whole result, contract_kernel's direct loads reach 0.79 of that rate (16 384 x 200, K 336 and
    // 64 head rows: 78 us, a whole evaluation, against 82 to 84 with 2 x 2 fragments and 4 tiles per
    // CU; K 640: 104 and 106; 9000 x 200, K 336: 72 and 67)
    const int64_t direct = (int64_t)gm * ((n + 127) / 128);
    if (K <= 512 && direct > 480 && direct <= 512 && 4.0 / 0.79 < std::min(c44, std::min(c42, c22)))
      hipLaunchKernelGGL((contract_kernel<4, true>), dim3(gm, (unsigned)((n + 127) / 128)), block, 0, st,
                         A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64, K64);
    else if (c44 <= std::min(c42, c22))
      contract_k4_launch<4, 4, 4>(A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64,
                                  K64, st);
    else if (c42 <= c22)
      contract_k4_launch<4, 2, 4>(A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64,
                                  K64, st);
    else
      contract_k4_launch<2, 2, 8>(A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64,
                                  K64, st);
  } else if (tn == 64) {
    hipLaunchKernelGGL((contract_kernel<2, false>), dim3(gm, (unsigned)((n + 63) / 64)), block, 0,
                       st, A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64, K64);
  } else {
    hipLaunchKernelGGL((contract_kernel<4, false>), dim3(gm, (unsigned)((n + 127) / 128)), block, 0,
                       st, A, lda, B, ldb, offset, Y, ldy, P, n, K, A64, lda64, B64, ldb64, K64);
  }
  SBI_HIP_CHECK(hipGetLastError());
  return SBI_OK;
}

// ------------------------------------------------------------------------------------------
// BF16 contraction (gfx950 v_mfma_f32_16x16x32_bf16): Y = offset + A64^T B64 + A^T B with A and B
// in BF16, k-interleaved by 8 (element (k, p) of A at A[((k / 8) * lda + p) * 8 + k % 8], the same
// for B; K a multiple of 32, zero rows pad it), and an optional FP64 head of K64 rows in the plain
// layout (FP64 MFMA, as in contract_kernel).  BF16 products are exact in FP32; the FP32 partial
// sums are added into FP64 registers every kBfFlush k.
//
// Work split: a workgroup of 4 waves (2 x 2) owns a tile of TM = 32 * kBfWM points x TN =
// 32 * kBfWN outputs; each wave a sub-tile of kBfWM x kBfWN MFMA 16x16 fragments (4 x 4 for the
// largest grids, 4 x 2 for large ones, 2 x 2 otherwise).  Per 32-k step the workgroup
// copies the step's 16-byte A vectors (4 k-groups x TM points) and B vectors (4 x TN outputs)
// into LDS with direct-to-LDS loads, kBfBuf buffers in rotation, the copies issued two steps
// ahead and one barrier per step (a buffer is rewritten two steps after it was read, and every
// wave has passed the barrier of the step in between); each wave then reads its fragments with
// 16-byte LDS reads.  Lane group g = lane / 16 supplies k = 8g .. 8g + 7 of the step to both
// operands.  The steps of one kBfFlush chunk form an inner loop with the flush after it, so the
// FP32 accumulators stay in the matrix-core registers across the chunk (a flush test inside the
// step loop made the compiler copy them to and from ordinary registers at every step).
// Measured (same bits as each wave loading its own fragments from global memory): 4096 points x
// 4096 outputs, K 10 016: 0.42 ms against 0.66-0.71 ms (4 x 2 fragments; 0.32-0.35 ms with 4 x 4);
// 8192 x 256, K 5 024: 39 us against 66 us.
// Every workgroup is independent and each Y row depends only on its own column of A (fixed order).
// ------------------------------------------------------------------------------------------
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v8bf lds_v8bf;
constexpr int kBfFlush = 1024;  // k per FP32 partial sum
constexpr int kBfBuf = 4;       // LDS buffers of one 32-k step each

// kBfWM x kBfWN fragments per wave (points, outputs); 2 x 2 waves per workgroup (the body of the
// kernels below; each has its own LDS buffers)
template <int kBfWM, int kBfWN>
__device__ __forceinline__ void contract_bf16_body(
    const uint4* __restrict__ A, int64_t lda, const uint4* __restrict__ B, int64_t ldb,
    int64_t K, const double* __restrict__ A64, int64_t lda64, const double* __restrict__ B64,
    int64_t ldb64, int64_t K64, const double* __restrict__ offset, double* __restrict__ Y,
    int64_t ldy, int64_t P, int64_t n) {
  constexpr int TM = 32 * kBfWM, TN = 32 * kBfWN;
  constexpr int kAB = 4 * TM * 16, kStep = kAB + 4 * TN * 16;  // bytes per step: A, then B
  constexpr int nA = kAB / 1024, nI = kStep / 1024, kPer = nI / 4;  // 1 KB copies
  static_assert(TM % 64 == 0 && TN % 64 == 0 && nI % 4 == 0 && kPer >= 2 && kPer <= 4,
                "tile shape");
  __shared__ __attribute__((aligned(16))) char smem[kBfBuf * kStep];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 15, g = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * TM, n0 = (int64_t)blockIdx.y * TN;
  const int64_t m_base = m0 + wm * (16 * kBfWM);
  const int64_t n_base = n0 + wn * (16 * kBfWN);
  int64_t jcol[kBfWN];
#pragma unroll
  for (int fn = 0; fn < kBfWN; ++fn) jcol[fn] = min(n_base + fn * 16 + li, n - 1);

  v4d acc64[kBfWM][kBfWN];
#pragma unroll
  for (int fm = 0; fm < kBfWM; ++fm)
#pragma unroll
    for (int fn = 0; fn < kBfWN; ++fn) acc64[fm][fn] = v4d{0, 0, 0, 0};

  if (K64 > 0) {  // FP64 head: lane li supplies point 4 * (li & 3) + (li >> 2) of its block, so
                  // the FP64 MFMA's rows land in the FP32 layout (row 4g + r in register r)
    int64_t ph[kBfWM];
#pragma unroll
    for (int fm = 0; fm < kBfWM; ++fm)
      ph[fm] = min(m_base + fm * 16 + 4 * (li & 3) + (li >> 2), P - 1);
    head_fp64<kBfWM, kBfWN>(A64, lda64, B64, ldb64, K64, g, ph, jcol, acc64);
  }

  v4f acc[kBfWM][kBfWN];
#pragma unroll
  for (int fm = 0; fm < kBfWM; ++fm)
#pragma unroll
    for (int fn = 0; fn < kBfWN; ++fn) acc[fm][fn] = v4f{0, 0, 0, 0};
  auto flush = [&]() {
#pragma unroll
    for (int fm = 0; fm < kBfWM; ++fm)
#pragma unroll
      for (int fn = 0; fn < kBfWN; ++fn) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc64[fm][fn][r] += (double)acc[fm][fn][r];
        acc[fm][fn] = v4f{0, 0, 0, 0};
      }
  };
  // copy c of a step (this wave: c = wave + 4 i): c < nA -> A vectors of k-group c / (TM / 64),
  // points 64 (c % (TM / 64)) .., else B vectors likewise; it lands at LDS byte c * 1024 +
  // 16 lane, i.e. [k-group][point] then [k-group][output].  Points and outputs past the edge
  // re-read the last one (their results are not stored).
  const uint4* src[kPer];
  int64_t sstep[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = wave + 4 * i;
    if (c < nA) {
      const int kq = c / (TM / 64), part = c % (TM / 64);
      src[i] = A + (int64_t)kq * lda + min(m0 + part * 64 + lane, P - 1);
      sstep[i] = 4 * lda;
    } else {
      const int kq = (c - nA) / (TN / 64), part = (c - nA) % (TN / 64);
      src[i] = B + (int64_t)kq * ldb + min(n0 + part * 64 + lane, n - 1);
      sstep[i] = 4 * ldb;
    }
  }
  auto issue = [&](int s) {
    char* buf = smem + (s % kBfBuf) * kStep;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      __builtin_amdgcn_global_load_lds((const void*)(src[i] + (int64_t)s * sstep[i]),
                                       (lds_void*)(buf + (wave + 4 * i) * 1024), 16, 0, 0);
  };
  const int S = (int)(K / 32);
  if (S > 0) {
    issue(0);
    if (S > 1) issue(1);
    for (int sc = 0; sc < S; sc += kBfFlush / 32) {
      const int se = min(S, sc + kBfFlush / 32);
      for (int s = sc; s < se; ++s) {
        // this wave's copies of step s have landed once at most those of s + 1, s + 2 remain
        if (s + 2 < S) {
          issue(s + 2);
          if constexpr (kPer == 4) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
          else if constexpr (kPer == 3) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
          else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
        } else if (s + 1 < S) {
          if constexpr (kPer == 4) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
          else if constexpr (kPer == 3) asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)" ::: "memory");
          else asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        }
        asm volatile("s_barrier" ::: "memory");  // every wave's copies of step s have landed
        const lds_v8bf* LA = (const lds_v8bf*)(smem + (s % kBfBuf) * kStep);
        const lds_v8bf* LB = (const lds_v8bf*)(smem + (s % kBfBuf) * kStep + kAB);
        v8bf a[kBfWM], b[kBfWN];
#pragma unroll
        for (int fm = 0; fm < kBfWM; ++fm) a[fm] = LA[g * TM + wm * (16 * kBfWM) + fm * 16 + li];
#pragma unroll
        for (int fn = 0; fn < kBfWN; ++fn) b[fn] = LB[g * TN + wn * (16 * kBfWN) + fn * 16 + li];
#pragma unroll
        for (int fm = 0; fm < kBfWM; ++fm)
#pragma unroll
          for (int fn = 0; fn < kBfWN; ++fn)
            acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[fm], b[fn], acc[fm][fn], 0, 0,
                                                                  0);
      }
      flush();
    }
  }

#pragma unroll
  for (int fn = 0; fn < kBfWN; ++fn) {
    const int64_t col = n_base + fn * 16 + li;
    if (col >= n) continue;
    const double off = offset ? offset[col] : 0.0;
#pragma unroll
    for (int fm = 0; fm < kBfWM; ++fm)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = m_base + fm * 16 + (4 * g + r);
        if (row < P) Y[row * ldy + col] = off + acc64[fm][fn][r];
      }
  }
}

#define SBI_BF16_ARGS                                                                          \
  const uint4 *__restrict__ A, int64_t lda, const uint4 *__restrict__ B, int64_t ldb, int64_t K, \
      const double *__restrict__ A64, int64_t lda64, const double *__restrict__ B64,             \
      int64_t ldb64, int64_t K64, const double *__restrict__ offset, double *__restrict__ Y,     \
      int64_t ldy, int64_t P, int64_t n
template <int kBfWM, int kBfWN>
__global__ __launch_bounds__(256) void contract_bf16_kernel(SBI_BF16_ARGS) {
  contract_bf16_body<kBfWM, kBfWN>(A, lda, B, ldb, K, A64, lda64, B64, ldb64, K64, offset, Y, ldy,
                                   P, n);
}
// 4 x 4 fragments per wave (workgroup 128 x 128), asked for two waves per SIMD: 243 registers
// and no scratch (one wave per SIMD otherwise).  4096 points x 4096 outputs, K 10 016: 323-350 us
// against 416-485 us for 4 x 2 fragments; same bits.  (The request on the 4 x 2 and 2 x 2 forms
// measured no gain, so it is this kernel's alone.)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void
contract_bf16_wide_kernel(SBI_BF16_ARGS) {
  contract_bf16_body<4, 4>(A, lda, B, ldb, K, A64, lda64, B64, ldb64, K64, offset, Y, ldy, P, n);
}
#undef SBI_BF16_ARGS

// ------------------------------------------------------------------------------------------
// Jacobian contraction: for each input dim z, J[p, c, z] = sum over the rows q of dim z of
// A[e_q, p] S[v_q, c].  Rows are listed dim by dim, each dim padded to a multiple of four, so every
// 4-row MFMA step belongs to one dim (steps spanning dims would run once per dim: 2-4 x the
// matrix work of the many dims with a handful of rows).
//
// A workgroup of 4 waves takes one job for 64 points x 32 outputs: the rows of a group of kJacDims
// consecutive dims (one accumulator tile per dim in registers), or one part of a group with many
// rows: the first dims of an index set hold most of them (the first 8 of 200: 5594 of 11 506), so
// the host cuts such a group into parts, which jac_group_reduce_kernel adds in order.  Bound: the
// FP64 matrix cores (75 us at 999 points x 256 outputs x 200 dims) and, for the many short groups,
// the latency of a job's start; measured there 268 us + 27 us for the parts (466 us with masked
// chunks across dims, each wave loading from L2 and every lane writing its own 64 bytes).  (Groups
// with few rows joined into longer jobs were slower, 542 us: a wave's stores of a finished group hold
// up its next loads, which complete in order behind them.)
//
// Operands are staged in LDS in chunks of 32 rows, three buffers, copied two chunks ahead by direct
// global -> LDS loads (16-byte slots of odd rows rotated by 8, as in contract_f64_kernel); the row
// table is copied the same way three chunks ahead of that, into each wave's own ring, and read
// into registers a chunk before it is needed.  Every wave issues the same number of copies per
// chunk, past the last one too (rows clamped), so the waits are counts.  kWide = false: S rows that do not start on 16 bytes, or an odd number of outputs
// without the promise of a spare element (jac_wide_rows), are copied in 4-byte pieces.
//
// The tile is written through LDS, one accumulator register of every dim at a time, so that eight
// consecutive lanes write the kJacDims consecutive doubles of one (point, output): a lane writing
// them itself makes eight requests of 8 bytes where one of 64 does.
// ------------------------------------------------------------------------------------------
constexpr int kJacDims = sbi::kJacGroup;  // dims per job
constexpr int kJacN = 32;                 // outputs per job
constexpr int kJacChunk = 32;             // rows per chunk
constexpr int kJacRing = 8;               // row-table chunks on chip (six in use)
constexpr int kJacT = 68;  // doubles between dims of a tile being written (the 8 dims of 4 outputs
                           // fall into all banks)

template <bool kWide>
__global__ __launch_bounds__(64 * kWaves, 2) void jac_contract_kernel(
    const double* __restrict__ A, uint32_t lda, const double* __restrict__ S, int64_t lds,
    sbi::JacRows t, int nz, double* __restrict__ J, int64_t P, int64_t n, int ntp, int ntn,
    double* __restrict__ part) {
  constexpr int C = kJacChunk;
  constexpr int kA = C * kBlockM * 8, kB = C * kJacN * 8, kRec = C * 8;  // bytes of a chunk
  constexpr int kNA = kA / 4096, kNB = kB / 4096 * (kWide ? 1 : 4);      // copies per wave
  constexpr int kPer = kNA + kNB + 1;
  static_assert(kRec == 64 * 4, "one copy per row-table chunk");
  __shared__ __attribute__((aligned(16))) char smem[3 * (kA + kB) + kWaves * kJacRing * kRec];
  static_assert(kWaves * kJacDims * kJacT * 8 <= 3 * (kA + kB), "the tile being written");
  const int L = blockIdx.x, idx = L >> 3;
  const int tn = idx % ntn;
  const int pair = (idx / ntn) * 8 + (L & 7);
  if (pair >= ntp * t.n_jobs) return;
  const int tp = pair % ntp;
  const int32_t* __restrict__ job = t.job + 4 * (pair / ntp);
  const int r0 = job[0], r1 = job[1], slot = job[3];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, g = lane >> 4;
  const int mw = (wave & 1) * 32, nw = (wave >> 1) * 16;
  const int64_t m0 = (int64_t)tp * kBlockM, n0 = (int64_t)tn * kJacN;
  char* const ring = smem + 3 * (kA + kB) + wave * kJacRing * kRec;

  // copies of this wave: LDS rows 2 i, 2 i + 1 of A for i = wave + 4 u (lane: row 2 i + lane / 32, pair
  // lane % 32); S rows 4 i .. 4 i + 3 for i = wave + 4 u, four at a time (lane: row lane / 16, pair
  // lane % 16) or one at a time in words (lane: word lane of the row's 64)
  const int ar = lane >> 5;
  const double* __restrict__ ap =
      A + min(m0 + (((lane & 31) ^ (8 * ar)) * 2), (P - 1) & ~(int64_t)1);
  const int br = kWide ? lane >> 4 : 0;
  const int64_t bcol = n0 + (((lane & 15) ^ (8 * (br & 1))) * 2);
  const double* __restrict__ bp = S + min(bcol, (n - 1) & ~(int64_t)1);
  int ra[kNA], rs[kNB];  // rows of A and S of the next chunk to be copied
  auto copy_rec = [&](int c) {  // row-table chunk c
    const int64_t w = (int64_t)min(r0 + c * C + (lane >> 1), r1 - 1) * 2 + (lane & 1);
    __builtin_amdgcn_global_load_lds((const void*)(t.row + w),
                                     (lds_void*)(ring + (c % kJacRing) * kRec), 4, 0, 0);
  };
  auto read_rec = [&](int c) {  // (row-table chunk c has landed)
    const int2* rec = (const int2*)(ring + (c % kJacRing) * kRec);
#pragma unroll
    for (int u = 0; u < kNA; ++u) ra[u] = rec[2 * (wave + 4 * u) + ar].x;
#pragma unroll
    for (int u = 0; u < kNB; ++u)
      rs[u] = kWide ? rec[4 * (wave + 4 * u) + br].y : rec[4 * (wave + 4 * (u / 4)) + u % 4].y;
  };
  auto copy = [&](int b) {  // the next chunk of A and S into buffer b
    char* da = smem + b * kA + wave * 1024;
#pragma unroll
    for (int u = 0; u < kNA; ++u)
      __builtin_amdgcn_global_load_lds((const void*)(ap + (uint64_t)(uint32_t)ra[u] * lda),
                                       (lds_void*)(da + u * 4096), 16, 0, 0);
    char* ds = smem + 3 * kA + b * kB + wave * 1024;
#pragma unroll
    for (int u = 0; u < kNB; ++u) {
      if constexpr (kWide) {
        __builtin_amdgcn_global_load_lds((const void*)(bp + (int64_t)rs[u] * lds),
                                         (lds_void*)(ds + u * 4096), 16, 0, 0);
      } else {
        const int64_t col = n0 + ((lane >> 1) ^ (16 * (u & 1)));
        const double* row = S + (int64_t)rs[u] * lds + min(col, n - 1);
        __builtin_amdgcn_global_load_lds((const void*)((const int*)row + (lane & 1)),
                                         (lds_void*)(ds + u / 4 * 4096 + u % 4 * 256), 4, 0, 0);
      }
    }
  };
  const int sw = 16 * (g & 1);
  v4d cur[2];
  // one 4-row step at row 4 s of the chunk in buffer b; rows at and past `end` (relative to the
  // chunk) count as zero
  auto step = [&](int b, int s, int end) {
    const int r = 4 * s + g;
    const double* sa = (const double*)(smem + b * kA) + r * kBlockM;
    double a0 = sa[(mw + li) ^ sw], a1 = sa[(mw + 16 + li) ^ sw];
    double bv = ((const double*)(smem + 3 * kA + b * kB))[r * kJacN + ((nw + li) ^ sw)];
    if (4 * s + 4 > end && r >= end) a0 = a1 = bv = 0.0;
    cur[0] = mfma(a0, bv, cur[0]);
    cur[1] = mfma(a1, bv, cur[1]);
  };

  v4d acc[kJacDims][2];
  const int z0 = job[2];
  if (r0 < r1) {
    copy_rec(0);
    copy_rec(1);
    copy_rec(2);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    read_rec(0);
    copy(0);
    copy_rec(3);
    read_rec(1);
    copy(1);
    copy_rec(4);
    read_rec(2);
  }
  // lane l: first row of the group's dim l, end of its real rows
  const int offv = t.off[min(z0 + min(lane, kJacDims), nz)];
  const int endv = t.end[min(z0 + min(lane, kJacDims - 1), nz - 1)];
  int q = r0, c = 0, q0 = r0, b = 0;  // next row; its chunk, the chunk's first row and buffer
  auto begin = [&] {  // chunk c has landed in every wave (and row-table chunk c + 3); c + 2 is copied
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kPer) : "memory");
    asm volatile("s_barrier" ::: "memory");
    copy(b == 0 ? 2 : b - 1);
    copy_rec(c + 5);
    read_rec(c + 3);
  };
  auto advance = [&](int rows) {
    q += rows;
    if (q == q0 + C) {
      ++c;
      q0 = q;
      b = b == 2 ? 0 : b + 1;
    }
  };
  for (int jj = 0; jj < kJacDims; ++jj) {
    const int end = min(__builtin_amdgcn_readlane(offv, jj + 1), r1);
    const int real = __builtin_amdgcn_readlane(endv, jj);
    const int whole = min(end, real);
    cur[0] = cur[1] = v4d{0, 0, 0, 0};
    while (q < end) {
      // (whole chunks in a loop of their own: the accumulators stay in place)
      while (q == q0 && q + C <= whole) {
        begin();
#pragma unroll
        for (int s = 0; s < C / 4; ++s) step(b, s, C);
        advance(C);
      }
      if (q >= end) break;
      if (q == q0) begin();
      const int stop = min(end, q0 + C);
      for (; q < stop; q += 4) step(b, (q - q0) >> 2, real - q0);
      advance(0);
    }
    switch (jj) {  // (register arrays take constant indices)
#define SBI_KEEP(i)      \
  case i:                \
    acc[i][0] = cur[0];  \
    acc[i][1] = cur[1];  \
    break;
      SBI_KEEP(0) SBI_KEEP(1) SBI_KEEP(2) SBI_KEEP(3) SBI_KEEP(4) SBI_KEEP(5) SBI_KEEP(6) SBI_KEEP(7)
#undef SBI_KEEP
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the last chunk
  __syncthreads();

  // FP64 16x16x4 result: row (point) g + 4r in register r, column (output) = lane % 16.  Register r of
  // all dims goes through LDS; lanes l = 8 i + (lane >> 3) of it are written in step i, so a step has
  // one point and 8 outputs, the points follow each other, and the address is a scalar that advances
  // plus the lane's own fixed offset (with an address per element a call on one job of a few rows took
  // 1.5 us more, and 999 points x 256 outputs x 200 dims 351 instead of 346 us).
  double* __restrict__ tr = (double*)smem + wave * kJacDims * kJacT;
  const int jj = lane & 7, sub = lane >> 3;
  const double* __restrict__ from = tr + jj * kJacT + sub;
  const int64_t row0 = m0 + mw, col0 = n0 + nw;
  const int rows = (int)min(P - row0, (int64_t)32);
  const int64_t ldo = slot >= 0 ? kJacDims : nz;
  const uint32_t own = (uint32_t)sub * (uint32_t)ldo + jj;
  const bool in0 = col0 + sub < n, in1 = col0 + 8 + sub < n;
  typedef __attribute__((address_space(1))) double gdouble;
  gdouble* out = (gdouble*)(slot >= 0 ? part + (int64_t)slot * P * n * kJacDims : J + z0) +
                 (row0 * n + col0) * ldo;
  const bool mine = slot >= 0 || z0 + jj < nz;
#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int u = 0; u < kJacDims; ++u) tr[u * kJacT + lane] = acc[u][fm][r];
      double v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = from[8 * i];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        if (fm * 16 + 4 * r + h < rows) {
          if (mine && in0) out[own] = v[2 * h];
          if (mine && in1) (out + 8 * ldo)[own] = v[2 * h + 1];
        }
        out += n * ldo;
        asm volatile("" : "+s"(out));  // (or the 32 addresses are computed and kept first)
      }
    }
}

// J of the dim groups that several jobs share: the sum of their parts in order (blockIdx.y: the
// shared group).
__global__ __launch_bounds__(256) void jac_group_reduce_kernel(const double* __restrict__ part,
                                                              const int32_t* __restrict__ red,
                                                              int nz, double* __restrict__ J,
                                                              int64_t Pn) {
  const int z0 = red[3 * blockIdx.y], slot = red[3 * blockIdx.y + 1], count = red[3 * blockIdx.y + 2];
  const int nd = min(kJacDims, nz - z0);
  for (int64_t i8 = (int64_t)blockIdx.x * 256 + threadIdx.x; i8 < Pn * kJacDims;
       i8 += (int64_t)gridDim.x * 256) {
    const int jj = (int)(i8 % kJacDims);
    double v = 0.0;
#pragma unroll 4
    for (int u = 0; u < count; ++u) v += part[((int64_t)slot + u) * Pn * kJacDims + i8];
    if (jj < nd) J[i8 / kJacDims * nz + z0 + jj] = v;
  }
}

}  // namespace

namespace sbi {

int contract_jacobian_f64(const double* A, int64_t lda, const double* S, int64_t lds, bool padded,
                          const JacRows& t, int nz, double* J, int64_t P, int64_t n, double* part,
                          hipStream_t st) {
  if (P <= 0 || n <= 0 || nz <= 0) return SBI_OK;
  const int64_t ntp = (P + kBlockM - 1) / kBlockM, ntn = (n + kJacN - 1) / kJacN;
  const int64_t grid = ntn * ((ntp * t.n_jobs + 7) / 8) * 8;
  if (grid > 0x7fffffff || t.n_red > 65535) {
    set_error("contract_jacobian_f64: launch too large");
    return SBI_ERR_INVALID;
  }
  const bool wide = jac_wide_rows(S, lds, n, padded);
  hipLaunchKernelGGL(wide ? jac_contract_kernel<true> : jac_contract_kernel<false>,
                     dim3((unsigned)grid), dim3(64 * kWaves), 0, st, A, (uint32_t)lda, S, lds, t, nz,
                     J, P, n, (int)ntp, (int)ntn, part);
  SBI_HIP_CHECK(hipGetLastError());
  if (t.n_red > 0) {
    const int64_t rg = std::min<int64_t>((P * n * kJacDims + 255) / 256, 4096);
    hipLaunchKernelGGL(jac_group_reduce_kernel, dim3((unsigned)rg, (unsigned)t.n_red), dim3(256), 0,
                       st, part, t.red, nz, J, P * n);
    SBI_HIP_CHECK(hipGetLastError());
  }
  return SBI_OK;
}

}  // namespace sbi

extern "C" int sbi_contract(const void* A, int64_t lda, const void* B, int64_t ldb,
                            const double* offset, double* Y, int64_t ldy, int64_t P, int64_t n,
                            int64_t K, int32_t dtype, void* stream) {
  if (P < 0 || n < 0 || K < 0 || (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K > 0 && (!A || !B || lda < P || ldb < n)) ||
      P > (int64_t)65535 * kBlockM || n > (int64_t)65535 * 32) {
    sbi::set_error("sbi_contract: invalid argument");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == 0)
    return contract_f64((const double*)A, lda, (const double*)B, ldb, offset, Y, ldy, P, n, K,
                        false, true, nullptr, 0, st);
  if (dtype == 1)
    return contract_launch<false>((const float*)A, lda, (const float*)B, ldb, offset, Y, ldy, P,
                                  n, K, nullptr, 0, nullptr, 0, 0, st);
  sbi::set_error("sbi_contract: dtype must be 0 (f64) or 1 (f32)");
  return SBI_ERR_INVALID;
}

extern "C" int sbi_contract_f64_workspace(int64_t P, int64_t n, int64_t K, int64_t* bytes) {
  if (P < 0 || n < 0 || K < 0 || !bytes) {
    sbi::set_error("sbi_contract_f64_workspace: invalid argument");
    return SBI_ERR_INVALID;
  }
  *bytes = f64_plan(P, n, K).bytes;
  return SBI_OK;
}

extern "C" int sbi_contract_f64_ws(const double* A, int64_t lda, const double* B, int64_t ldb,
                                   const double* offset, double* Y, int64_t ldy, int64_t P,
                                   int64_t n, int64_t K, void* workspace, int64_t ws_bytes,
                                   void* stream) {
  if (P < 0 || n < 0 || K < 0 || ws_bytes < 0 || (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K > 0 && (!A || !B || lda < P || ldb < n)) ||
      ((uintptr_t)workspace & 15) || P > (int64_t)65535 * kBlockM || n > (int64_t)65535 * 32) {
    sbi::set_error("sbi_contract_f64_ws: invalid argument");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  const bool padded = lda >= P + (P & 1) && ldb >= n + (n & 1);
  return contract_f64(A, lda, B, ldb, offset, Y, ldy, P, n, K, padded, false, workspace, ws_bytes,
                      (hipStream_t)stream);
}

extern "C" int sbi_contract_split_k4(const double* A64, int64_t lda64, const double* B64,
                                     int64_t ldb64, int64_t K64, const float* A32, int64_t lda32,
                                     const float* B32, int64_t ldb32, int64_t K32,
                                     const double* offset, double* Y, int64_t ldy, int64_t P,
                                     int64_t n, void* stream) {
  if (P < 0 || n < 0 || K64 < 0 || K32 < 0 || K32 % 16 != 0 ||
      (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K64 > 0 && (!A64 || !B64 || lda64 < P || ldb64 < n)) ||
      (P > 0 && n > 0 && K32 > 0 &&
       (!A32 || !B32 || lda32 < P || ldb32 < n || ((uintptr_t)A32 & 15) || ((uintptr_t)B32 & 15))) ||
      P > (int64_t)65535 * kBlockM || n > (int64_t)65535 * 32) {
    sbi::set_error("sbi_contract_split_k4: invalid argument (K32 must be a multiple of 16, the "
                   "k-interleaved operands 16-byte aligned)");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  return contract_launch<true>(A32, lda32, B32, ldb32, offset, Y, ldy, P, n, K32, A64,
                                      lda64, B64, ldb64, K64, (hipStream_t)stream);
}

extern "C" int64_t sbi_contract_split_k4_workspace(int64_t P, int64_t n, int64_t K64,
                                                   int64_t K32) {
  if (P < 0 || n < 0 || K64 < 0 || K32 < 0 || K32 % 16 != 0) {
    sbi::set_error("sbi_contract_split_k4_workspace: invalid argument");
    return -1;
  }
  const SplitPlan sp = split_plan(P, n, K32, K64);
  return sp.nsplit ? sp.part_bytes + sp.head_bytes : 0;
}

extern "C" int sbi_contract_split_k4_ws(const double* A64, int64_t lda64, const double* B64,
                                        int64_t ldb64, int64_t K64, const float* A32,
                                        int64_t lda32, const float* B32, int64_t ldb32,
                                        int64_t K32, const double* offset, double* Y, int64_t ldy,
                                        int64_t P, int64_t n, void* workspace, int64_t ws_bytes,
                                        void* stream) {
  if (P < 0 || n < 0 || K64 < 0 || K32 < 0 || K32 % 16 != 0 || ws_bytes < 0 ||
      (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K64 > 0 && (!A64 || !B64 || lda64 < P || ldb64 < n)) ||
      (P > 0 && n > 0 && K32 > 0 &&
       (!A32 || !B32 || lda32 < P || ldb32 < n || ((uintptr_t)A32 & 15) || ((uintptr_t)B32 & 15))) ||
      ((uintptr_t)workspace & 255) || P > (int64_t)65535 * kBlockM || n > (int64_t)65535 * 32) {
    sbi::set_error("sbi_contract_split_k4_ws: invalid argument (K32 must be a multiple of 16, the "
                   "k-interleaved operands 16-byte aligned, the workspace 256-byte aligned)");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  const SplitPlan sp = split_plan(P, n, K32, K64);
  if (sp.nsplit == 0 || !workspace || ws_bytes < sp.part_bytes + sp.head_bytes)
    return contract_launch<true>(A32, lda32, B32, ldb32, offset, Y, ldy, P, n, K32, A64,
                                        lda64, B64, ldb64, K64, (hipStream_t)stream);
  return contract_split_launch<true>(sp, A32, lda32, B32, ldb32, offset, Y, ldy, P, n,
                                            K32, A64, lda64, B64, ldb64, K64, workspace,
                                            (hipStream_t)stream);
}

extern "C" int sbi_contract_split(const double* A64, int64_t lda64, const double* B64,
                                  int64_t ldb64, int64_t K64, const float* A32, int64_t lda32,
                                  const float* B32, int64_t ldb32, int64_t K32,
                                  const double* offset, double* Y, int64_t ldy, int64_t P,
                                  int64_t n, void* stream) {
  if (P < 0 || n < 0 || K64 < 0 || K32 < 0 || (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K64 > 0 && (!A64 || !B64 || lda64 < P || ldb64 < n)) ||
      (P > 0 && n > 0 && K32 > 0 && (!A32 || !B32 || lda32 < P || ldb32 < n)) ||
      P > (int64_t)65535 * kBlockM || n > (int64_t)65535 * 32) {
    sbi::set_error("sbi_contract_split: invalid argument");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  return contract_launch<false>(A32, lda32, B32, ldb32, offset, Y, ldy, P, n, K32, A64, lda64,
                                B64, ldb64, K64, (hipStream_t)stream);
}

extern "C" int sbi_contract_bf16_k8(const double* A64, int64_t lda64, const double* B64,
                                    int64_t ldb64, int64_t K64, const void* A16, int64_t lda16,
                                    const void* B16, int64_t ldb16, int64_t K16,
                                    const double* offset, double* Y, int64_t ldy, int64_t P,
                                    int64_t n, void* stream) {
  if (P < 0 || n < 0 || K64 < 0 || K16 < 0 || K16 % 32 != 0 ||
      (P > 0 && n > 0 && (!Y || ldy < n)) ||
      (P > 0 && n > 0 && K64 > 0 && (!A64 || !B64 || lda64 < P || ldb64 < n)) ||
      (P > 0 && n > 0 && K16 > 0 &&
       (!A16 || !B16 || lda16 < P || ldb16 < n || ((uintptr_t)A16 & 15) || ((uintptr_t)B16 & 15))) ||
      (P + 63) / 64 > 0x7fffffff || (n + 63) / 64 > 65535) {
    sbi::set_error("sbi_contract_bf16_k8: invalid argument (K16 must be a multiple of 32, the "
                   "k-interleaved operands 16-byte aligned)");
    return SBI_ERR_INVALID;
  }
  if (P == 0 || n == 0) return SBI_OK;
  // per-wave tiles: 64 x 64 (workgroup 128 x 128, LDS 64 KB) while that gives at least 1024
  // workgroups, else 64 x 32 (128 x 64, 48 KB) likewise, else 32 x 32 (64 x 64, 32 KB): the
  // smaller tiles spread small grids further (2 and 4 waves per SIMD); every element's sum is the
  // same (same bits)
  const int64_t g44 = ((P + 127) / 128) * ((n + 127) / 128);
  const int64_t g42 = ((P + 127) / 128) * ((n + 63) / 64);
  if (g44 >= 1024) {
    const dim3 grid((unsigned)((P + 127) / 128), (unsigned)((n + 127) / 128));
    hipLaunchKernelGGL(contract_bf16_wide_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                       (const uint4*)A16, lda16, (const uint4*)B16, ldb16, K16, A64, lda64, B64,
                       ldb64, K64, offset, Y, ldy, P, n);
  } else if (g42 >= 1024) {
    const dim3 grid((unsigned)((P + 127) / 128), (unsigned)((n + 63) / 64));
    hipLaunchKernelGGL((contract_bf16_kernel<4, 2>), grid, dim3(256), 0, (hipStream_t)stream,
                       (const uint4*)A16, lda16, (const uint4*)B16, ldb16, K16, A64, lda64, B64,
                       ldb64, K64, offset, Y, ldy, P, n);
  } else {
    const dim3 grid((unsigned)((P + 63) / 64), (unsigned)((n + 63) / 64));
    hipLaunchKernelGGL((contract_bf16_kernel<2, 2>), grid, dim3(256), 0, (hipStream_t)stream,
                       (const uint4*)A16, lda16, (const uint4*)B16, ldb16, K16, A64, lda64, B64,
                       ldb64, K64, offset, Y, ldy, P, n);
  }
  SBI_HIP_CHECK(hipGetLastError());
  return SBI_OK;
}
