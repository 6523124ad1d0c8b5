// Barycentric combination technique for 2 to 16 outputs, FP64, gfx950.
//
//   y(x) = offset + sum over entries e of F[e, :] prod_{factors (slot s, index mu) of e} Lhat^s_mu(x_s)
//
// (src/smolyax/barycentric.py:69-123, summed over the blocks of interpolation.py:264-304).  The
// entries of all blocks form one list, so the sum is a product of the entry weights W (points x
// entries, made here and never stored) with F on v_mfma_f64_16x16x4: 64 cycles of a SIMD per 4
// entries x 16 points x 16 outputs, beside 1 to 8 LDS reads and products per 64 weights.
//
// The host cuts the list into shares of about 1500 entries whose factors need at most 318 rows
// of 1D basis values; a workgroup of 8 waves (two per CU) takes 64 points and one or more shares, one after
// another: the share's basis rows for the 64 points in LDS, the entries in steps of four (one per
// lane group) dealt over the waves, the waves' sums added in wave order.  When the 64-point tiles
// are few, the shares are spread over workgroups that write their sums to a workspace, and a second
// kernel adds them in share order: the same bits for any batch.
//
// 500 points x 40 inputs x 10 outputs, 95 956 entries: 1830 us for one workgroup per 64 points and 4
// outputs walking the blocks through scalar loads, 54 us a call here, one after another (a kernel trace
// has 54 us for this kernel and 6 for the sum over shares; matrix cores alone: 20 us); with 8-byte reads of the basis rows 18 us more (LDS-bound), one workgroup of 16 waves
// 5 us more, four of 4 waves 10 us more.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/smolyax_amd.h"
#include "common.h"
#include "launch.h"

namespace {

constexpr int kTile = 64;    // points per workgroup
constexpr int kWaves = 8;
constexpr int kOut = 16;     // outputs of a matrix fragment
constexpr int kHdr = 16;     // int32 per share header
constexpr int kSlotBatch = 4;  // slots per wave whose coordinates are requested together

typedef double v4d __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) double lds_f64;
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ cptr<T> C(const T* p) {
  return (cptr<T>)(p);
}

// First-form basis of degree deg at x into rows row0 .. row0 + deg for this lane (exact one-hot at
// a node): the products in the order of the other barycentric kernels.
__device__ __forceinline__ void basis_rows(double x, cptr<double> xi, cptr<double> w, int deg,
                                           lds_f64* tab, int row0, int lane) {
  double s = 1.0;
  for (int m = deg; m >= 0; --m) {
    tab[(row0 + m) * kTile + lane] = s;
    s *= (x - xi[m]);
  }
  double pre = 1.0;
  int hit = -1;
  for (int m = 0; m <= deg; ++m) {
    const double dm = x - xi[m];
    if (dm == 0.0) hit = m;
    tab[(row0 + m) * kTile + lane] *= w[m] * pre;
    pre *= dm;
  }
  if (hit >= 0) {
    for (int m = 0; m <= deg; ++m) tab[(row0 + m) * kTile + lane] = (m == hit) ? 1.0 : 0.0;
  }
}

// u16 rows per entry in the record stream of K factors
constexpr int rec_stride(int K) { return K <= 2 ? 2 : K <= 4 ? 4 : 8; }

// The steps of a share whose entries have K factors: step s holds entries 4 s + g for lane group g.
// Lane (li, g) computes the weights of its entry at the points 32 h + 2 li + c of the four fragments
// f = 2 h + c, two neighbouring points per 16-byte LDS read (a lane group reads 256 contiguous
// bytes of a row: no bank conflicts whatever the rows).
// A wave takes a contiguous run of steps, and every two steps are summed from zero before they are
// added: a block's entries are neighbours and largely cancel, and a sum that follows them loses
// less.  (Steps dealt over the waves and one running sum: 48 us instead of 54 us at the size
// above, but up to 12 % more error than the walk over blocks: 1.0e-13 against 0.9e-13, 3.7e-13
// against 3.4e-13; here 0.9e-13 and 3.2e-13.)
template <int K>
__device__ __forceinline__ void run_steps(int n, const uint16_t* __restrict__ rec,
                                          const double* __restrict__ F, int64_t d_out, int wave,
                                          int lane, const lds_f64* tab, v4d (&acc)[4]) {
  constexpr int R = rec_stride(K);
  const int li = lane & 15, g = lane >> 4;
  typedef double v2d __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) v2d lds_v2d;
  const double* __restrict__ Fl = F + (int64_t)g * d_out + min((int64_t)li, d_out - 1);
  const int begin = n * wave / kWaves, end = n * (wave + 1) / kWaves;
  if (begin >= end) return;
  uint32_t rw[2][R / 2];
  double b[2];
  auto fetch = [&](int q, int s) {
    const uint32_t* __restrict__ r = (const uint32_t*)(rec + ((int64_t)s * 4 + g) * R);
#pragma unroll
    for (int i = 0; i < R / 2; ++i) rw[q][i] = r[i];
    b[q] = Fl[(int64_t)s * 4 * d_out];
  };
  v4d run[4];
  auto step = [&](int q, int next) {
    int off[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const uint32_t r = i & 1 ? rw[q][i >> 1] >> 16 : rw[q][i >> 1] & 0xffff;
      off[i] = (int)r * kTile + 2 * li;
    }
    const double bs = b[q];
    fetch(q, min(next, end - 1));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v2d u = *(const lds_v2d*)(tab + off[0] + 32 * h);
#pragma unroll
      for (int i = 1; i < K; ++i) {
        const v2d t = *(const lds_v2d*)(tab + off[i] + 32 * h);
        u.x *= t.x;
        u.y *= t.y;
      }
      const v4d zero = {0, 0, 0, 0};
      run[2 * h] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, bs, q ? run[2 * h] : zero, 0, 0, 0);
      run[2 * h + 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, bs, q ? run[2 * h + 1] : zero, 0, 0, 0);
    }
  };
  fetch(0, begin);
  fetch(1, min(begin + 1, end - 1));
  int s = begin;
  for (; s + 2 <= end; s += 2) {
    step(0, s + 2);
    step(1, s + 3);
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] += run[f];
  }
  if (s < end) {
    step(0, s);
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] += run[f];
  }
}

__global__ __launch_bounds__(kTile* kWaves, 4) void bary_few_kernel(sbi_bary_desc d,
                                                                const double* __restrict__ x,
                                                                int64_t P, int64_t ldx,
                                                                double* __restrict__ y,
                                                                double* __restrict__ part,
                                                                int shares_per_wg) {
  extern __shared__ double lds_raw[];
  lds_f64* tab = (lds_f64*)lds_raw;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p = min((int64_t)blockIdx.x * kTile + lane, P - 1);
  const double* __restrict__ xp = x + p * ldx;
  const int n = (int)d.d_out;
  const int sh0 = blockIdx.y * shares_per_wg, sh1 = min(d.n_share, sh0 + shares_per_wg);
  // this thread's element of the tile after the waves' sums are added: point tid / 16, output tid % 16
  const int64_t prow = (int64_t)blockIdx.x * kTile + (threadIdx.x >> 4);
  const int pcol = threadIdx.x & 15;
  constexpr int kE = 16 / kWaves;  // elements per thread: points prow + 4 kWaves i
  double total[kE];
#pragma unroll
  for (int i = 0; i < kE; ++i) total[i] = 0.0;

  for (int sh = sh0; sh < sh1; ++sh) {
    cptr<int32_t> h = C(d.share) + (int64_t)sh * kHdr;
    const int ns = h[1];
    cptr<int32_t> slots = C(d.share_slot) + 2 * (int64_t)h[0];
    __syncthreads();  // the previous share's sums have been read
    for (int s0 = wave; s0 < ns; s0 += kSlotBatch * kWaves) {
      int sl[kSlotBatch], row[kSlotBatch];
      double xv[kSlotBatch];
#pragma unroll
      for (int u = 0; u < kSlotBatch; ++u) {
        const int s = min(s0 + u * kWaves, ns - 1);
        sl[u] = slots[2 * s];
        row[u] = slots[2 * s + 1];
      }
#pragma unroll
      for (int u = 0; u < kSlotBatch; ++u) xv[u] = xp[C(d.slot_dim)[sl[u]]];
#pragma unroll
      for (int u = 0; u < kSlotBatch; ++u)
        if (s0 + u * kWaves < ns)
          basis_rows(xv[u], C(d.slot_nodes) + (int64_t)sl[u] * d.dmax1,
                     C(d.slot_w) + (int64_t)sl[u] * d.dmax1, C(d.slot_deg)[sl[u]], tab, row[u],
                     lane);
    }
    if (wave == kWaves - 1) tab[h[2] * kTile + lane] = 1.0;  // the row of padding factors
    __syncthreads();

    v4d acc[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] = v4d{0, 0, 0, 0};
    const uint16_t* __restrict__ rec = (const uint16_t*)d.share_rec + (int64_t)h[4];
    const double* __restrict__ F = d.share_F + (int64_t)h[3] * n;
#define SBI_STEPS(K)                                               \
  {                                                                \
    const int ks = h[4 + K];                                       \
    run_steps<K>(ks, rec, F, n, wave, lane, tab, acc);             \
    rec += (int64_t)ks * 4 * rec_stride(K);                        \
    F += (int64_t)ks * 4 * n;                                      \
  }
    SBI_STEPS(1) SBI_STEPS(2) SBI_STEPS(3) SBI_STEPS(4)
    SBI_STEPS(5) SBI_STEPS(6) SBI_STEPS(7) SBI_STEPS(8)
#undef SBI_STEPS
    __syncthreads();  // the table is done with
    // result layout: register r of lane group g holds row g + 4 r of the fragment, output li
    const int li = lane & 15, g = lane >> 4;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        tab[(wave * kTile + 32 * (f >> 1) + 2 * (g + 4 * r) + (f & 1)) * kOut + li] = acc[f][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kE; ++i) {
      const int64_t row = prow + 4 * kWaves * i;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
        s += tab[w * kTile * kOut + kTile * kWaves * i + threadIdx.x];
      if (!part) total[i] += s;
      else if (row < P && pcol < n) part[((int64_t)sh * P + row) * n + pcol] = s;
    }
  }
#pragma unroll
  for (int i = 0; i < kE; ++i) {
    const int64_t row = prow + 4 * kWaves * i;
    if (!part && row < P && pcol < n) y[row * n + pcol] = d.offset[pcol] + total[i];
  }
}

// y = offset + the shares' sums in share order.
__global__ __launch_bounds__(256) void bary_few_reduce_kernel(const double* __restrict__ part,
                                                             int n_share,
                                                             const double* __restrict__ offset,
                                                             double* __restrict__ y, int64_t Pn,
                                                             int n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= Pn) return;
  double v = 0.0;
#pragma unroll 8
  for (int s = 0; s < n_share; ++s) v += part[(int64_t)s * Pn + i];
  y[i] = offset[i % n] + v;
}

// Shares per workgroup: one, spread by the workspace, unless the tiles alone are eight workgroups per
// CU (131 072 points) or the workspace would exceed 256 MB: then all, without a workspace.  Fewer,
// longer workgroups leave CUs idle at the end: 16 384 points, 14 shares, 40 inputs: 298 us one by
// one, 351 us with all 14 in a workgroup (9000 points: 182 and 222 us).
int shares_per_wg(const sbi_bary_desc& d, int64_t P) {
  const bool alone = (P + kTile - 1) / kTile >= 2048 || d.n_share > 65535 ||  // (launch limit)
                     d.n_share * P * d.d_out * 8 > (int64_t(256) << 20);
  return alone ? d.n_share : 1;
}

}  // namespace

extern "C" int sbi_bary_plan_desc(const sbi_plan* plan, const sbi_bary_desc** out);

extern "C" int64_t sbi_bary_eval_few_workspace(const sbi_plan* plan, int64_t P) {
  const sbi_bary_desc* d = nullptr;
  if (sbi_bary_plan_desc(plan, &d) != SBI_OK || P < 0 || d->n_share <= 0) {
    sbi::set_error("sbi_bary_eval_few_workspace: null plan, negative P or a plan without shares");
    return -1;
  }
  return P == 0 || shares_per_wg(*d, P) >= d->n_share ? 0 : d->n_share * P * d->d_out * 8;
}

extern "C" int sbi_bary_eval_few_f64(const sbi_plan* plan, const double* x, int64_t P, int64_t ldx,
                                     double* y, void* workspace, int64_t ws_bytes, void* stream) {
  const sbi_bary_desc* dp = nullptr;
  if (sbi_bary_plan_desc(plan, &dp) != SBI_OK || !x || !y || P < 0 || ldx < dp->d_in ||
      ws_bytes < 0 || ((uintptr_t)workspace & 7)) {
    sbi::set_error("sbi_bary_eval_few_f64: invalid argument");
    return SBI_ERR_INVALID;
  }
  const sbi_bary_desc& d = *dp;
  if (d.n_share <= 0) {
    sbi::set_error("sbi_bary_eval_few_f64: the plan has no shares (more than 16 outputs, or a block "
                   "of more than 8 factors or too many basis rows)");
    return SBI_ERR_CAPACITY;
  }
  if (P == 0) return SBI_OK;
  if ((P + kTile - 1) / kTile > 0x7fffffff) {
    sbi::set_error("sbi_bary_eval_few_f64: too many points for one call");
    return SBI_ERR_INVALID;
  }
  int per = shares_per_wg(d, P);
  double* part = per < d.n_share ? (double*)workspace : nullptr;
  if (per < d.n_share && (!workspace || ws_bytes < d.n_share * P * d.d_out * 8)) {
    per = d.n_share;  // no room for the shares' sums: one workgroup per tile, the same bits
    part = nullptr;
  }
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = (size_t)std::max(d.share_rows, kWaves * kOut) * kTile * sizeof(double);
  sbi::allow_lds((const void*)bary_few_kernel);
  const dim3 grid((unsigned)((P + kTile - 1) / kTile), (unsigned)((d.n_share + per - 1) / per));
  hipLaunchKernelGGL(bary_few_kernel, grid, dim3(kTile * kWaves), lds, st, d, x, P, ldx, y, part,
                     per);
  SBI_HIP_CHECK(hipGetLastError());
  if (part) {
    const int64_t Pn = P * d.d_out;
    hipLaunchKernelGGL(bary_few_reduce_kernel, dim3((unsigned)((Pn + 255) / 256)), dim3(256), 0, st,
                       part, d.n_share, d.offset, y, Pn, (int)d.d_out);
    SBI_HIP_CHECK(hipGetLastError());
  }
  return SBI_OK;
}
