// float64 path: slogdet / slogpf forward and their gradients (A^-T, S^-1) for
// 0 <= n <= 8192: one workgroup per matrix up to n = 128, the blocked kernels of lu64_impl.inc
// above.
//
// The reference takes float64 through the same entry points as float32 (dtype check
// `_prep`, src/fermix/api.py:24-31; 64-bit fields in src/fermix/_field.py:20-120, where
// "tf32x3" is rejected for 64-bit types, :265-275). Its arithmetic for these types is
// the generic path: LU with partial pivoting (`_slogdet_generic` / `_slog_from_lu`,
// src/fermix/_fallback.py:36-60), the inverse for the gradient (`_lu_parts_generic`,
// :63-97) and Parlett-Reid with the pivot swapped into column c + 1 and the rank-2
// update tau w^T - w tau^T (`_slogpf_generic`, :266-300).
//
// n <= 128 (fx_tune.f64_reg_max_n): the matrix in LDS, one workgroup or wave per matrix
// (field_small.inc); above, the blocked kernels of lu64_impl.inc. The value and the gradient
// call of one order run the same factorisation, so their sign / logabs agree bit for bit.
#include <algorithm>

#include "common.h"
#include "fermix_internal.h"
#include "field.h"

namespace fx {
namespace {

constexpr int F64_MAXN = 8192;
size_t align_up_256(size_t x) { return (x + 255) / 256 * 256; }

// Above f64_reg_max_n the values come from the blocked LU (lu64_impl.inc) and the gradient's
// A^-T from the blocked solves of the same factorisation.
bool lu64_path(int n) { return n > tune().f64_reg_max_n; }

// slogdet values for n <= TINY64_MAXN with several matrices per wave: G = 16 lanes per matrix,
// lane r of a group holding row r in registers, no workgroup barrier: the pivot is the exact
// 64-bit argmax (the high words' maximum, then the low words' among the lanes holding it,
// then the lowest such row), l = a[r][j] * (1 / piv) and one fma per entry of the unassigned
// rows, the logs summed in pivot order, the sign from the negative pivots and the
// permutation's parity. The pivot row reaches the group through LDS. Kept beside the
// LDS-resident kernel, which gives a whole wave to a matrix, where it wins: B = 16384, n = 8
// 23 against 41 us, n = 16 35 against 69,; at n = 32 (G = 32) it lost,
// 136 against 125 us.
constexpr int TINY64_MAXN = 16;

template <int G>
__global__ __launch_bounds__(256) void lutiny64_kernel(const double* __restrict__ a, int n, int64_t batch,
                                                       double* __restrict__ sign_out,
                                                       double* __restrict__ logabs_out) {
  constexpr int MPW = 256 / G;  // matrices per workgroup
  __shared__ double ubuf[256], pbuf[256];
  __shared__ int ibuf[256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = tid % G;       // row within the matrix
  const int gbase = lane - r;  // first lane of the group
  double* const ub = ubuf + (tid - r);  // the group's pivot row
  double* const pv = pbuf + (tid - r);  // its pivots, in column order
  int* const pi = ibuf + (tid - r);     // and their rows
  const int64_t mi = (int64_t)blockIdx.x * MPW + tid / G;
  const bool live = mi < batch;
  const double* Ab = a + (live ? mi : 0) * (int64_t)n * n;
  double M[G];
  const int rr = min(r, n - 1);
#pragma unroll
  for (int c = 0; c < G; ++c) M[c] = Ab[(int64_t)rr * n + min(c, n - 1)];
#pragma unroll
  for (int c = 0; c < G; ++c) M[c] = (r < n && c < n) ? M[c] : 0.0;
  bool asg = false, singular = false;
  double sgn = 1.0;
  static_for<0, G>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if (j < n) {
      const unsigned long long k = (r < n && !asg) ? key64(M[j]) : 0ull;
      const unsigned hi = (unsigned)(k >> 32), lo = (unsigned)k;
      const unsigned mh = group_max_u32<G>(hi);
      const unsigned ml = group_max_u32<G>(hi == mh ? lo : 0u);
      const int p = group_first<G>(k != 0 && hi == mh && lo == ml, gbase);
      const double piv = __shfl(M[j], gbase + p);
      double rinv = 0.0;
      if (piv == 0.0) {
        singular = true;
      } else {
        rinv = 1.0 / piv;
        if (piv < 0.0) sgn = -sgn;
      }
      if (r == p) {
#pragma unroll
        for (int c = j + 1; c < G; ++c) ub[c] = M[c];
        pv[j] = piv;
        pi[j] = p;
      }
      wave_lds_fence();
      if (r < n && r != p && !asg) {
        const double l = M[j] * rinv;
#pragma unroll
        for (int c = j + 1; c < G; ++c) M[c] = fma(-l, ub[c], M[c]);
      }
      if (r == p) asg = true;
      wave_lds_fence();  // every read of ub precedes the next step's writes
    }
  });
  if (live && r == 0) {
    double logabs = 0.0;
    if (!singular)
      for (int j = 0; j < n; ++j) logabs += log(fabs(pv[j]));
    unsigned seen = 0;  // parity of j -> pi[j] from its cycles
    int cycles = 0;
    for (int s0 = 0; s0 < n; ++s0) {
      if ((seen >> s0) & 1u) continue;
      ++cycles;
      for (int u = s0; !((seen >> u) & 1u); u = pi[u]) seen |= 1u << u;
    }
    if ((n - cycles) & 1) sgn = -sgn;
    sign_out[mi] = singular ? 0.0 : sgn;
    logabs_out[mi] = singular ? -INFINITY : logabs;
  }
}

// Argument checks shared by the float64 entry points: the alignment contract of the ABI
// (matrix-shaped and workspace pointers 16-byte aligned, sign / logabs 8-byte aligned).
int check_f64_args(const void* a, int64_t batch, int n, const void* sign, const void* logabs, const void* out,
                   const void* ws) {
  if (batch < 0 || n < 0) return FX_ERR_INVALID_ARGUMENT;
  if (n > F64_MAXN) return FX_ERR_UNSUPPORTED;
  if (batch > 0 && (!sign || !logabs || (n > 0 && !a))) return FX_ERR_INVALID_ARGUMENT;
  auto mis = [](const void* p, uintptr_t m) { return ((uintptr_t)p & m) != 0; };
  if (mis(a, 15) || mis(out, 15) || mis(ws, 15) || mis(sign, 7) || mis(logabs, 7)) return FX_ERR_INVALID_ARGUMENT;
  if (batch > 0x7fffffff) return FX_ERR_UNSUPPORTED;
  return FX_OK;
}

}  // namespace

// The gradient's matrix of n <= TINY64_MAXN comes from its own factorisation, gated by the
// values' sign, so that a gradient call returns the values' bits.
int launch_lu64_small(const double* a, int n, int64_t batch, double* sign, double* logabs, double* out, bool det,
                      hipStream_t s) {
  if (n < 1 || n > TINY64_MAXN)
    return fsmall_lu<double>(a, n, 0, batch, sign, logabs, nullptr, det ? sign : nullptr, logabs, out, 1, s);
  lutiny64_kernel<16><<<dim3((unsigned)((batch + 15) / 16)), 256, 0, s>>>(a, n, batch, sign, logabs);
  if (hipGetLastError() != hipSuccess) return FX_ERR_LAUNCH;
  if (!out) return FX_OK;
  return fsmall_lu<double>(a, n, 0, batch, nullptr, nullptr, sign, det ? sign : nullptr, logabs, out, 1, s);
}

}  // namespace fx

using namespace fx;

extern "C" {

size_t fx_slogdet_f64_workspace(int64_t batch, int32_t n) {
  fx::TunePin pin_;
  if (n > F64_MAXN) return 0;
  return lu64_path(n) ? lu64_workspace(batch, n) : 0;
}

int fx_slogdet_f64(const double* a, int64_t batch, int32_t n, double* sign, double* logabs, void* workspace,
                   size_t workspace_bytes, fx_stream_t stream) {
  fx::TunePin pin_;
  const int st = check_f64_args(a, batch, n, sign, logabs, nullptr, workspace);
  if (st != FX_OK || batch == 0) return st;
  if (lu64_path(n)) return launch_lu64(a, n, batch, sign, logabs, workspace, workspace_bytes, (hipStream_t)stream);
  return launch_lu64_small(a, n, batch, sign, logabs, nullptr, false, (hipStream_t)stream);
}

size_t fx_slogdet_parts_f64_workspace(int64_t batch, int32_t n) {
  fx::TunePin pin_;
  if (n > F64_MAXN) return 0;
  return lu64_path(n) ? lu64_inverse_workspace(batch, n) : 0;
}

int fx_slogdet_parts_f64(const double* a, int64_t batch, int32_t n, double* sign, double* logabs, double* inv_t,
                         void* workspace, size_t workspace_bytes, fx_stream_t stream) {
  fx::TunePin pin_;
  const int st = check_f64_args(a, batch, n, sign, logabs, inv_t, workspace);
  if (st != FX_OK || batch == 0) return st;
  if (!inv_t) return fx_slogdet_f64(a, batch, n, sign, logabs, workspace, workspace_bytes, stream);
  hipStream_t s = (hipStream_t)stream;
  if (!lu64_path(n)) return launch_lu64_small(a, n, batch, sign, logabs, inv_t, false, s);
  return launch_lu64_inverse(a, n, 0, batch, sign, logabs, nullptr, nullptr, nullptr, inv_t, 1, workspace,
                             workspace_bytes, s);
}

size_t fx_slogpf_f64_workspace(int64_t batch, int32_t n) {
  fx::TunePin pin_;
  return n > F64_MAXN || !lu64_path(n) ? 0 : pr64_workspace(batch, n);
}

int fx_slogpf_f64(const double* a, int64_t batch, int32_t n, int32_t skew_symmetrize, double* sign, double* logabs,
                  void* workspace, size_t workspace_bytes, fx_stream_t stream) {
  fx::TunePin pin_;
  const int st = check_f64_args(a, batch, n, sign, logabs, nullptr, workspace);
  if (st != FX_OK || batch == 0) return st;
  hipStream_t s = (hipStream_t)stream;
  if (!lu64_path(n)) return fsmall_pr<double>(a, n, skew_symmetrize != 0, batch, sign, logabs, s);
  return launch_pr64_blocked(a, n, skew_symmetrize != 0, batch, sign, logabs, workspace, workspace_bytes, s);
}

size_t fx_slogpf_parts_f64_workspace(int64_t batch, int32_t n) {
  fx::TunePin pin_;
  if (n > F64_MAXN || batch <= 0) return 0;
  const size_t pr = fx_slogpf_f64_workspace(batch, n);
  const size_t inv = (lu64_path(n) ? align_up_256(lu64_inverse_workspace(batch, n)) : 0) +
                     align_up_256((size_t)batch * 2 * sizeof(double));
  // + the blocked Parlett-Reid run's pair-pivot spread (the adjugate's route gate)
  return align_up_256(pr) + std::max(inv, pf_adjugate_f64_ws(batch, n)) +
         (lu64_path(n) ? align_up_256((size_t)batch * sizeof(double)) : 0);
}

int fx_slogpf_parts_f64(const double* a, int64_t batch, int32_t n, int32_t skew_symmetrize, int32_t adjugate,
                        double* sign, double* logabs, double* g, void* workspace, size_t workspace_bytes,
                        fx_stream_t stream) {
  fx::TunePin pin_;
  int st = check_f64_args(a, batch, n, sign, logabs, g, workspace);
  if (st != FX_OK || batch == 0) return st;
  hipStream_t s = (hipStream_t)stream;
  if (!g) return fx_slogpf_f64(a, batch, n, skew_symmetrize, sign, logabs, workspace, workspace_bytes, stream);
  const size_t need = fx_slogpf_parts_f64_workspace(batch, n);
  if (workspace_bytes < need || (!workspace && need)) return FX_ERR_WORKSPACE;
  const size_t pr = align_up_256(fx_slogpf_f64_workspace(batch, n));
  char* base = (char*)workspace;
  double* spread = lu64_path(n) ? (double*)(base + need - align_up_256((size_t)batch * sizeof(double))) : nullptr;
  SideStream side(s, !adjugate && lu64_path(n) && pf_parts_overlap(batch, n));
  if (side.ok() && (st = side.fork()) != FX_OK) return st;
  st = lu64_path(n) ? launch_pr64_blocked(a, n, skew_symmetrize != 0, batch, sign, logabs, base, pr, side.side(), spread)
                    : fsmall_pr<double>(a, n, skew_symmetrize != 0, batch, sign, logabs, s);
  if (st != FX_OK || n == 0) return st;
  // the Pfaffian adjugate (cplx.hip): the LU route, or the pivot-replaced Parlett-Reid
  // formula for pf = 0 and numerically singular members
  if (adjugate)
    return pf_adjugate_f64(a, batch, n, skew_symmetrize != 0, g, sign, logabs, spread, base + pr,
                           need - pr - (spread ? align_up_256((size_t)batch * sizeof(double)) : 0), s);
  // S^-1 from an LU of the same S, zeroed where the Parlett-Reid run found pf = 0 (every
  // member for odd n)
  if (lu64_path(n)) {
    const size_t lw = align_up_256(lu64_inverse_workspace(batch, n));
    double* gsign = (double*)(base + pr + lw);
    return launch_lu64_inverse(a, n, skew_symmetrize != 0, batch, gsign, gsign + batch, sign, nullptr, nullptr, g, 0,
                               base + pr, lw, s, &side);
  }
  double* gsign = (double*)(base + pr);
  return fsmall_lu<double>(a, n, skew_symmetrize != 0, batch, gsign, gsign + batch, sign, nullptr, nullptr, g, 0, s);
}

}  // extern "C"
