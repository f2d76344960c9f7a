// A^-T from the packed LU of P A' (the slogdet backward), N > 128 (smaller orders:
// small_inverse.hip): the factors are embedded in T (Ninv x Ninv, Ninv = 32 * 2^k >= N,
// identity padded) and
//   1. the 128x128 diagonal blocks are inverted in place in LDS: strictly-lower part of
//      L^-1, upper part of U~^-1 (U~ = U with exact zero pivots replaced by 1, so singular
//      inputs stay finite);
//   2. the block-recursive levels s = 128, 256, .., Ninv/2 complete L^-1 and U~^-1 with
//      four batched MFMA GEMMs per level (all block pairs of a level in one launch):
//        X21 = -X22 (L21 X11),   Y12 = -Y11 (U12 Y22);
//   3. Z = U~^-1 L^-1 by one GEMM whose tiles only run over k >= max(row, col), its
//      epilogue storing invT[g0[c]][i] = Z[i][c] (transpose + row permutation through
//      LDS) and flagging tiles with a non-finite value; Z itself is never stored;
//   4. invT is zeroed for members with a non-finite Z or, if requested, an exactly zero
//      pivot.
// Total 4/3 N^3 of MFMA work (L^-1 and U^-1 N^3/3 each, the triangular product 2N^3/3).
//
// Reference roles replaced (ChenAo-Phys/fermix): _packed_lu / _diag_kernel leaf
// inverses (src/fermix/_inverse.py:75-221), _inv_unit_lower (:429-452), _solve_upper
// (:455-474) and _permT with the singular guard (:478-531).
#include "common.h"
#include "fermix_internal.h"

namespace fx {

// 32-bit index math (Ninv <= 2048).
__global__ void embed_kernel(const float* __restrict__ src, int N, float* __restrict__ T, int Ninv) {
  const int64_t b = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= Ninv * Ninv) return;
  const int r = e / Ninv, c = e - r * Ninv;
  T[b * Ninv * Ninv + e] = (r < N && c < N) ? src[b * (int64_t)N * N + r * N + c] : (r == c ? 1.0f : 0.0f);
}

typedef float v16f __attribute__((ext_vector_type(16)));

// op values of the packed block in LDS: the unit-lower factor (strictly lower entries,
// 1 on the diagonal) and the upper factor (upper entries incl. the diagonal)
__device__ __forceinline__ float lunit_at(const float* Ts, int ld, int r, int c) {
  return r > c ? Ts[r * ld + c] : (r == c ? 1.0f : 0.0f);
}
__device__ __forceinline__ float upper_at(const float* Ts, int ld, int r, int c) {
  return r <= c ? Ts[r * ld + c] : 0.0f;
}

constexpr int D = 128;  // order of the diagonal blocks that are inverted whole in LDS

// In-place inverses of the D x D diagonal blocks of the packed T:
// the strictly-lower part becomes L^-1, and with upper the upper part U~^-1, over the
// whole block, in one workgroup with the block in LDS:
//   1. the 32x32 leaves by substitution, one wave per leaf: lane c (< 32) forms column c
//      of L^-1 by forward substitution, lane 32 + c column c of U~^-1 by back
//      substitution (zero pivots divided as 1);
//   2. the recursion levels s = 32, 64 < D on MFMA (32x32x2): X21 = -X22 (L21 X11) and
//      Y12 = -Y11 (U12 Y22), one (pair, factor, 32-column block) per wave. The inner
//      product stays in registers and enters the outer one as it stands (lane (h, c)
//      holding rows 8 (v / 4) + 4 h + v % 4: one MFMA per v over those K indices, the
//      left operand read from LDS in that order); a barrier separates the reads of
//      L21 / U12 from the in-place stores of X21 / Y12.
__global__ __launch_bounds__(256) void diag_inverse_kernel(float* __restrict__ T, int Ninv,
                                                           const int* __restrict__ active, int upper) {
  constexpr int LDT = D + 1;
  __shared__ float Ts[D * LDT];
  const int64_t b = blockIdx.y;
  if (active && !active[b]) return;
  const int t0 = D * blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  float* base = T + b * (int64_t)Ninv * Ninv + (int64_t)t0 * Ninv + t0;
  {
    constexpr int NV = D * D / 4, PER = NV / 256;
    float4 v[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + 256 * u;
      v[u] = *reinterpret_cast<const float4*>(base + (e / (D / 4)) * Ninv + 4 * (e % (D / 4)));
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + 256 * u;
      float* d = Ts + (e / (D / 4)) * LDT + 4 * (e % (D / 4));
      d[0] = v[u].x;
      d[1] = v[u].y;
      d[2] = v[u].z;
      d[3] = v[u].w;
    }
  }
  __syncthreads();
  // 1. leaves
  {
    const int lo = 32 * wave, c = lane & 31;
    float x[32];
    if (lane < 32) {
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < i; ++k) acc = fmaf(Ts[(lo + i) * LDT + lo + k], x[k], acc);
        x[i] = (i == c) ? 1.0f : (i > c ? -acc : 0.0f);
      }
    } else if (upper) {
#pragma unroll
      for (int i = 31; i >= 0; --i) {
        float acc = (i == c) ? 1.0f : 0.0f;
#pragma unroll
        for (int k = i + 1; k < 32; ++k) acc = fmaf(-Ts[(lo + i) * LDT + lo + k], x[k], acc);
        const float dg = Ts[(lo + i) * LDT + lo + i];
        x[i] = (i > c) ? 0.0f : acc / (dg == 0.0f ? 1.0f : dg);
      }
    }
    // both halves of the wave have read the leaf (the branches run one after the other)
    if (lane < 32 || upper) {
#pragma unroll
      for (int i = 0; i < 32; ++i)
        if (lane < 32 ? (i > c) : (i <= c)) Ts[(lo + i) * LDT + lo + c] = x[i];
    }
  }
  __syncthreads();
  // 2. levels s = 32, 64 below D
  const int l32 = lane & 31, lh = lane >> 5;
  static_for<0, 2>([&](auto lc) {
    constexpr int s = 32 << decltype(lc)::value;
    if constexpr (s < D) {
      constexpr int NCB = s / 32;  // 32-column blocks (and 32-row tiles) of an s x s block
      const int chains = upper ? 2 : 1;
      const int items = (D / (2 * s)) * chains * NCB;  // <= 4
      const bool act = wave < items;
      const int J = wave % NCB, rest = wave / NCB;
      const int chain = rest % chains, o = (rest / chains) * 2 * s;
      v16f tacc[NCB];
#pragma unroll
      for (int I = 0; I < NCB; ++I)
#pragma unroll
        for (int v = 0; v < 16; ++v) tacc[I][v] = 0.0f;
      if (act) {
        if (chain == 0) {
          // T = L21 X11, column block J: k >= 32 J (X11 unit lower)
          for (int k0 = 32 * J; k0 < s; k0 += 2) {
            const float bv = lunit_at(Ts, LDT, o + k0 + lh, o + 32 * J + l32);
#pragma unroll
            for (int I = 0; I < NCB; ++I)
              tacc[I] = __builtin_amdgcn_mfma_f32_32x32x2f32(Ts[(o + s + 32 * I + l32) * LDT + o + k0 + lh], bv,
                                                              tacc[I], 0, 0, 0);
          }
        } else {
          // T = U12 Y22, column block J: k < 32 J + 32 (Y22 upper)
          for (int k0 = 0; k0 < 32 * J + 32; k0 += 2) {
            const float bv = upper_at(Ts, LDT, o + s + k0 + lh, o + s + 32 * J + l32);
#pragma unroll
            for (int I = 0; I < NCB; ++I)
              tacc[I] = __builtin_amdgcn_mfma_f32_32x32x2f32(Ts[(o + 32 * I + l32) * LDT + o + s + k0 + lh], bv,
                                                              tacc[I], 0, 0, 0);
          }
        }
      }
      __syncthreads();  // every read of L21 / U12 is done
      if (act) {
#pragma unroll
        for (int I = 0; I < NCB; ++I) {
          v16f out;
#pragma unroll
          for (int v = 0; v < 16; ++v) out[v] = 0.0f;
          if (chain == 0) {
            // X21 = -X22 T, row tile I: k <= 32 I + 31 (X22 unit lower)
#pragma unroll
            for (int K = 0; K <= I; ++K)
#pragma unroll
              for (int v = 0; v < 16; ++v) {
                const int k = 32 * K + 8 * (v >> 2) + 4 * lh + (v & 3);
                out = __builtin_amdgcn_mfma_f32_32x32x2f32(lunit_at(Ts, LDT, o + s + 32 * I + l32, o + s + k),
                                                           tacc[K][v], out, 0, 0, 0);
              }
#pragma unroll
            for (int v = 0; v < 16; ++v)
              Ts[(o + s + 32 * I + 8 * (v >> 2) + 4 * lh + (v & 3)) * LDT + o + 32 * J + l32] = -out[v];
          } else {
            // Y12 = -Y11 T, row tile I: k >= 32 I (Y11 upper)
#pragma unroll
            for (int K = I; K < NCB; ++K)
#pragma unroll
              for (int v = 0; v < 16; ++v) {
                const int k = 32 * K + 8 * (v >> 2) + 4 * lh + (v & 3);
                out = __builtin_amdgcn_mfma_f32_32x32x2f32(upper_at(Ts, LDT, o + 32 * I + l32, o + k), tacc[K][v],
                                                           out, 0, 0, 0);
              }
#pragma unroll
            for (int v = 0; v < 16; ++v)
              Ts[(o + 32 * I + 8 * (v >> 2) + 4 * lh + (v & 3)) * LDT + o + s + 32 * J + l32] = -out[v];
          }
        }
      }
      __syncthreads();
    }
  });
  for (int e = tid; e < D * D; e += 256) base[(e / D) * Ninv + e % D] = Ts[(e / D) * LDT + e % D];
}

// bad[b] = any tile flag, or (zero_singular and sign[b] == 0)
__global__ void reduce_bad_kernel(const int* __restrict__ flags, int ntiles, const float* __restrict__ sign,
                                  int zero_singular, int* __restrict__ bad, int64_t batch) {
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= batch) return;
  bool f = false;
  for (int k = lane; k < ntiles; k += 64) f = f || flags[b * ntiles + k] != 0;
  const bool any = __ballot(f) != 0ull;
  if (lane == 0) bad[b] = (any || (zero_singular && sign[b] == 0.0f)) ? 1 : 0;
}

// invT[b] = 0 for the flagged members (one workgroup per member; others exit at once).
__global__ __launch_bounds__(256) void zero_bad_kernel(const int* __restrict__ bad, float* __restrict__ invT,
                                                       int64_t nn) {
  const int64_t b = blockIdx.x;
  if (!bad[b]) return;
  float* o = invT + b * nn;
  for (int64_t e = threadIdx.x; e < nn; e += 256) o[e] = 0.0f;
}

// In-place inverses of the unit-lower L (strictly lower part) and, with upper, of the
// upper U~ (upper part incl. diagonal) packed in T (B, Ninv, Ninv), the identity from order N
// on: the diagonal blocks and tiles past N are left as they are. The two factors' levels are
// independent: where a level leaves the chip partly idle the upper one's run on the side
// stream (one level's products are 128 x 128 tiles of about 30 us each, alone on a CU or
// not). Measured, slogdet + gradient: B = 95, n = 354 867 -> 751 us, B = 30, n = 700 1628 ->
// 1411, B = 8, n = 900 1732 -> 1609; from 512 tiles per level on one stream serves as well.
int launch_tri_inverse(float* T, int Ninv, int N, int64_t batch, float* Tmp, float* Tmp2, bool upper, hipStream_t s,
                       const int* active, int x3) {
  const int64_t NN = (int64_t)Ninv * Ninv;
  hipLaunchKernelGGL(diag_inverse_kernel, dim3((N + D - 1) / D, (unsigned)batch), dim3(256), 0, s, T, Ninv,
                     active, (int)upper);
  if (hipGetLastError() != hipSuccess) return FX_ERR_LAUNCH;
  SideStream side(s, upper && !active && batch * (Ninv / 256) * (Ninv / 256) <= 512);
  if (side.ok() && side.fork() != FX_OK) return FX_ERR_LAUNCH;
  // C (sz x sz, all pairs of a level) = alpha op(A) op(B)
  auto product = [&](const float* A, int maskA, bool tmpA, const float* B, int maskB, bool tmpB, float* C, bool tmpC,
                     float alpha, int sz, bool rows, hipStream_t st) {
    const int pairs = Ninv / (2 * sz);
    const int64_t dstride = (int64_t)2 * sz * (Ninv + 1);  // next pair along the diagonal
    const int64_t tall = (int64_t)pairs * sz * sz, tone = (int64_t)sz * sz;
    GemmDesc d = {};
    d.active = active;
    d.x3 = x3;
    d.M = d.N = d.K = sz;
    d.A = A;
    d.maskA = maskA;
    d.lda = tmpA ? sz : Ninv;
    d.sA = tmpA ? tall : NN;
    d.sA2 = tmpA ? tone : dstride;
    d.B = B;
    d.maskB = maskB;
    d.ldb = tmpB ? sz : Ninv;
    d.sB = tmpB ? tall : NN;
    d.sB2 = tmpB ? tone : dstride;
    d.C = C;
    d.ldc = tmpC ? sz : Ninv;
    d.sC = tmpC ? tall : NN;
    d.sC2 = tmpC ? tone : dstride;
    d.alpha = alpha;
    d.beta = 0.0f;
    // rows (L) or columns (U) sz .. of a pair's block that lie past N
    d.rlim = rows ? N - sz : 1 << 30;
    d.clim = rows ? 1 << 30 : N - sz;
    d.lim_step = 2 * sz;
    return launch_gemm(d, batch, pairs, st);
  };
  for (int sz = D; sz < Ninv; sz *= 2) {
    float* const T21 = T + (int64_t)sz * Ninv;
    float* const T12 = T + sz;
    float* const T22 = T21 + sz;
    // L: Tmp = L21 X11, X21 = -X22 Tmp
    int st = product(T21, MASK_NONE, false, T, MASK_LOWER_UNIT, false, Tmp, true, 1.0f, sz, true, s);
    if (st == FX_OK) st = product(T22, MASK_LOWER_UNIT, false, Tmp, MASK_NONE, true, T21, false, -1.0f, sz, true, s);
    if (st != FX_OK) return st;
    if (!upper) continue;
    // U: Tmp2 = U12 Y22, Y12 = -Y11 Tmp2
    const hipStream_t su = side.side();
    st = product(T12, MASK_NONE, false, T22, MASK_UPPER, false, Tmp2, true, 1.0f, sz, false, su);
    if (st == FX_OK) st = product(T, MASK_UPPER, false, Tmp2, MASK_NONE, true, T12, false, -1.0f, sz, false, su);
    if (st != FX_OK) return st;
  }
  return side.join();
}

int launch_unit_lower_inverse(float* T, int Ninv, int N, int64_t batch, float* Tmp, hipStream_t s,
                              const int* active, int x3) {
  return launch_tri_inverse(T, Ninv, N, batch, Tmp, nullptr, false, s, active, x3);
}

int inv_padded(int N) {
  int p = 32;
  while (p < N) p *= 2;
  return p;
}

size_t lu_inverse_workspace(int64_t batch, int N, bool need_copy) {
  // small_inverse.hip leaves it unused; the entry points ask for a workspace at every order
  if (N <= SMALL_INV_MAXN) return ((size_t)batch * 32 + 255) / 256 * 256;
  const int Ninv = inv_padded(N);
  const int nt = (N + 63) / 64;  // 64x64 tiles of the Z product
  size_t bytes = 0;
  auto add = [&](size_t x) { bytes += (x + 255) / 256 * 256; };
  if (need_copy) add((size_t)batch * Ninv * Ninv * 4);  // T
  add((size_t)batch * Ninv * Ninv / 4 * 4);              // Tmp (largest level: Ninv/2 x Ninv/2)
  add((size_t)batch * nt * nt * 4);                      // flags
  add((size_t)batch * 4);                                // bad
  return bytes;
}

int launch_lu_inverse(float* LU, const int* g0, int N, int n, int64_t batch, const float* sign,
                      int zero_singular, float* invT, bool in_place, void* ws, size_t ws_bytes,
                      hipStream_t s, const float* scale, int x3) {
  const int Ninv = inv_padded(N);
  const bool need_copy = !(in_place && Ninv == N);
  if (!ws || ws_bytes < lu_inverse_workspace(batch, N, need_copy)) return FX_ERR_WORKSPACE;
  if (N <= SMALL_INV_MAXN)
    return launch_lu_inv_small(LU, g0, N, n, batch, sign, scale, zero_singular, false, invT, s);
  char* p = (char*)ws;
  auto take = [&](size_t x) {
    char* q = p;
    p += (x + 255) / 256 * 256;
    return (void*)q;
  };
  float* T = need_copy ? (float*)take((size_t)batch * Ninv * Ninv * 4) : LU;
  float* Tmp = (float*)take((size_t)batch * Ninv * Ninv / 4 * 4);
  const int nt = (N + 63) / 64;  // 64x64 tiles of the Z product, one non-finite flag each
  int* flags = (int*)take((size_t)batch * nt * nt * 4);
  int* bad = (int*)take((size_t)batch * 4);
  const int64_t NN = (int64_t)Ninv * Ninv;
  if (need_copy) {
    hipLaunchKernelGGL(embed_kernel, dim3((unsigned)((NN + 255) / 256), (unsigned)batch), dim3(256), 0, s,
                       LU, N, T, Ninv);
    if (hipGetLastError() != hipSuccess) return FX_ERR_LAUNCH;
  }
  // the output, unused so far and at least Ninv^2 / 4 floats a member (n > Ninv / 2), holds Tmp2
  int st0 = launch_tri_inverse(T, Ninv, N, batch, Tmp, invT, true, s, nullptr, x3);
  if (st0 != FX_OK) return st0;
  // Z = U~^-1 L^-1 (the leading N x N block) stored straight as invT = P^T Z^T:
  // invT[g0[c]][i] = Z[i][c] for i < n and g0[c] < n, with the non-finite tile flags
  {
    GemmDesc d = {};
    d.x3 = x3;
    d.M = d.N = d.K = N;
    d.A = T;
    d.maskA = MASK_UPPER;
    d.B = T;
    d.maskB = MASK_LOWER_UNIT;
    d.lda = d.ldb = Ninv;
    d.sA = d.sB = NN;
    d.alpha = 1.0f;
    d.beta = 0.0f;
    d.tout = invT;
    d.g0 = g0;
    d.nout = n;
    d.scale = scale;
    d.flags = flags;
    const int st = launch_gemm(d, batch, 1, s);
    if (st != FX_OK) return st;
  }
  // the flagged members (and, with zero_singular, those with a zero pivot) are cleared
  hipLaunchKernelGGL(reduce_bad_kernel, dim3((unsigned)((batch + 3) / 4)), dim3(256), 0, s, flags, nt * nt,
                     sign, zero_singular, bad, batch);
  if (hipGetLastError() != hipSuccess) return FX_ERR_LAUNCH;
  hipLaunchKernelGGL(zero_bad_kernel, dim3((unsigned)batch), dim3(256), 0, s, bad, invT, (int64_t)n * n);
  return hipGetLastError() == hipSuccess ? FX_OK : FX_ERR_LAUNCH;
}

}  // namespace fx
