// The gradients' matrices for padded orders N <= 128 in one launch each, a matrix per
// workgroup (four per workgroup for N <= 32), straight from the forward's exported
// factors: A^-T or adj(A)^T from the packed LU (lu_inv_small_kernel), S^-1 or pf(S) S^-1
// from the Parlett-Reid factors (pf_inv_small_kernel).
//
// Both solve for whole 16-column blocks of the inverse. The factor sits in LDS (row stride
// N + 4: the 16-byte reads of 16 consecutive rows at four consecutive 16-byte columns fall
// on each bank four times, the least for 1 KiB), a wave owns the block columns w and
// NB - 1 - w (equal work), and a block column of the unknown stays in registers in the
// accumulator layout of v_mfma_f32_16x16x4f32 (lane (g, c) holds rows 4 g + v): register v
// of a block is the right operand of the MFMA over the K indices {4 g + v} as it stands,
// and the left operand over these indices is one 16-byte read of the factor. So between
// the inversion of the 16 x 16 diagonal blocks and the output no wave waits for another.
// Bound: the fp32 MFMAs (2/3 NB^3 + O(NB^2) block products of four 32-cycle MFMAs for the
// LU, 1/3 NB^3 for the Parlett-Reid) and the diagonal blocks' substitution chain.
//
// Reference roles replaced (ChenAo-Phys/fermix): _lu_parts / _permT with the singular guard
// (src/fermix/_inverse.py:478-531), _det_gradT (src/fermix/_diff.py:205-246) and _pf_parts
// (src/fermix/_pfinv.py:196-269) with _pf_adj_coeffs / _second_zero / _lifted_mean
// (src/fermix/_fallback.py:101-176), for the orders of the fused kernels.
#include "common.h"
#include "fermix_internal.h"

namespace fx {

namespace {

template <int NB>
struct SmallInv {
  static constexpr int N = 16 * NB;
  static constexpr int LD = N + 4;
  static constexpr int NW = (NB + 1) / 2;       // waves per matrix
  static constexpr int MW = NB <= 2 ? 4 : 1;    // matrices per workgroup (one wave each)
  static constexpr int NT = 64 * NW * MW;       // threads per workgroup
  // waves per SIMD that the LDS (16 NB rows of 16 NB + 4) and the registers allow together
  static constexpr int WPE = NB == 8 ? 2 : NB >= 6 ? 3 : 4;
};

// Ordering point of the NW waves of one matrix.
template <int NW>
__device__ __forceinline__ void mat_sync() {
  if constexpr (NW == 1) wave_lds_fence();
  else __syncthreads();
}

// Whether p holds on any thread of the matrix (every thread calls it; an ordering point).
template <int NW>
__device__ __forceinline__ bool mat_any(bool p) {
  if constexpr (NW == 1) {
    wave_lds_fence();
    return __ballot(p) != 0ull;
  } else {
    return __syncthreads_or(p ? 1 : 0) != 0;
  }
}

// In-place inverses of the 16 x 16 diagonal blocks of the packed factor in LDS, a block per
// 16 lanes (lane c forms column c by substitution), every block of the matrix at once:
// the unit-lower blocks (strictly lower part) and, with UPPER, the upper blocks (zero
// pivots divided as 1). An upper block is the lower one read backwards from its last
// entry, so both run the same instructions.
template <int NB, bool UPPER>
__device__ __forceinline__ void invert_diagonals(float* T, int wave, int lane) {
  constexpr int LD = SmallInv<NB>::LD;
  const int q = lane >> 4, c = lane & 15;
  const int blk = UPPER ? 2 * wave + (q & 1) : 4 * wave + q;
  const bool up = UPPER && (q >> 1);
  if (blk >= NB) return;
  float* const p0 = T + (16 * blk) * LD + 16 * blk + (up ? 15 * LD + 15 : 0);
  const int sg = up ? -1 : 1;
  // row i + 1 is read while row i is formed (the fence keeps the scheduler from raising all
  // 136 reads, and their registers, to the top)
  float x[16], e[2][16];
  auto read_row = [&](auto ic_) {
    constexpr int i = decltype(ic_)::value;
    static_for<0, (UPPER ? i + 1 : i)>([&](auto kc) { e[i & 1][kc.value] = p0[sg * (i * LD + kc.value)]; });
  };
  read_row(ic<0>{});
  static_for<0, 16>([&](auto ic_) {
    constexpr int i = decltype(ic_)::value;
    if constexpr (i < 15) read_row(ic<i + 1>{});
    float acc = i == c ? 1.0f : 0.0f;
    static_for<0, i>([&](auto kc) { acc = fmaf(-e[i & 1][kc.value], x[kc.value], acc); });
    if constexpr (UPPER) {
      const float d = up ? e[i & 1][i] : 1.0f;
      acc = acc / (d == 0.0f ? 1.0f : d);
    }
    x[i] = opaque(i < c ? 0.0f : acc);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  });
  // the block's 16 lanes have read its entries (one wave, in order)
  wave_lds_fence();
  static_for<0, 16>([&](auto ic_) {
    constexpr int i = decltype(ic_)::value;
    if (up ? i >= c : i > c) p0[sg * (i * LD + c)] = x[i];
  });
}

// Left operand of block (i, k): row 16 i + li, columns 16 k + 4 g + v.
template <int LD>
__device__ __forceinline__ v4f left_op(const float* T, int i, int k, int li, int g) {
  return *reinterpret_cast<const v4f*>(T + (16 * i + li) * LD + 16 * k + 4 * g);
}
// ... of the inverted diagonal blocks: unit lower, upper.
template <int LD>
__device__ __forceinline__ v4f left_lower(const float* T, int i, int li, int g) {
  v4f a = left_op<LD>(T, i, i, li, g);
#pragma unroll
  for (int v = 0; v < 4; ++v) a[v] = 4 * g + v < li ? a[v] : (4 * g + v == li ? 1.0f : 0.0f);
  return a;
}
template <int LD>
__device__ __forceinline__ v4f left_upper(const float* T, int i, int li, int g) {
  v4f a = left_op<LD>(T, i, i, li, g);
#pragma unroll
  for (int v = 0; v < 4; ++v) a[v] = 4 * g + v >= li ? a[v] : 0.0f;
  return a;
}

__device__ __forceinline__ v4f opaque4(v4f x) {
  return v4f{opaque(x[0]), opaque(x[1]), opaque(x[2]), opaque(x[3])};
}

__device__ __forceinline__ v4f mul16(v4f a, v4f b, v4f acc) {
#pragma unroll
  for (int v = 0; v < 4; ++v) acc = mfma16(a[v], b[v], acc);
  return acc;
}

// a b from zero, its four K-steps added in pairs: the roundings of a chain of sixteen products, and
// of a sum over blocks that runs through one accumulator, put slogpf's gradient 3 % (n = 16)
// to 7 % (n = 128) further from 64-bit results than the substitution and GEMMs before.
__device__ __forceinline__ v4f mul16_pairs(v4f a, v4f b) {
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  return (mfma16(a[0], b[0], zero) + mfma16(a[1], b[1], zero)) + (mfma16(a[2], b[2], zero) + mfma16(a[3], b[3], zero));
}

// Block columns j[0] < j[1] (two == false: j[0] only) of -L^-1: z[c][i], block row i, zero
// above the diagonal. Forward substitution by block rows.
template <int NB>
__device__ __forceinline__ void solve_lower(const float* T, const int (&j)[2], bool two, int li, int g,
                                            v4f (&z)[2][NB]) {
  constexpr int LD = SmallInv<NB>::LD;
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  static_for<0, NB>([&](auto ic_) {
    constexpr int i = decltype(ic_)::value;
    v4f a[i > 0 ? i : 1];
    static_for<0, i>([&](auto kc) { a[kc.value] = left_op<LD>(T, i, kc.value, li, g); });
    const v4f inv = left_lower<LD>(T, i, li, g);
    v4f acc[2] = {zero, zero};
    static_for<0, i>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      if (k >= j[0]) {
        acc[0] = mul16(a[k], z[0][k], acc[0]);
        if (two && k >= j[1]) acc[1] = mul16(a[k], z[1][k], acc[1]);
      }
    });
    static_for<0, 2>([&](auto cc_) {
      constexpr int c = decltype(cc_)::value;
      z[c][i] = zero;
      if (i == j[c]) {
        // the diagonal block itself, rows 4 g + v of column li
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float t = T[(16 * i + 4 * g + v) * LD + 16 * i + li];
          z[c][i][v] = 4 * g + v > li ? -t : (4 * g + v == li ? -1.0f : 0.0f);
        }
      } else if (i > j[c] && (c == 0 || two)) {
        z[c][i] = -mul16(inv, acc[c], zero);
      }
    });
  });
}

// ------------------------------------------------------------------ LU

// out[b] = scale[b] A^-T (zero for members with a non-finite value or, with zero_singular,
// sign[b] = 0) from the packed LU of P A (B, N, N) and the row map g0: U~ X = L^-1 solved
// block column by block column (U~: exact zero pivots as 1), out[g0[c]][i] = X[i][c].
// With DET out[b] = adj(A)^T instead: det A^-T for the regular members (the factors' own
// determinant), and for exactly zero pivots the rank-1 continuation
//   s A~^-T[:, k2] (x) U~^-1 e_k1,  s = sgn(P) d_K (one zero pivot k1 = k2),
//   sgn(P) d_K (U~^-1)[k1][k2] (two),  0 (more),
// d_K the product of the nonzero pivots.
// Measured, forward + gradient in one process against the embed, diagonal-block inverse, product
// and guard launches (det: also the parity and pivot launches) that did this before: slogdet
// B = 4096, n = 100 940 -> 392 us, det B = 16384, n = 24 619 -> 102 us.
template <int NB, bool DET>
__global__ __launch_bounds__(SmallInv<NB>::NT, SmallInv<NB>::WPE) void lu_inv_small_kernel(
    const float* __restrict__ LU, const int* __restrict__ g0, int n, int64_t batch, const float* __restrict__ sign,
    const float* __restrict__ scale, int zero_singular, float* __restrict__ out) {
  using C = SmallInv<NB>;
  constexpr int N = C::N, LD = C::LD, NW = C::NW, TM = 64 * NW;
  __shared__ __align__(16) float Ts[C::MW][N * LD];
  __shared__ float vecs[DET ? C::MW : 1][DET ? 2 * N + 16 : 1];
  const int m = C::MW > 1 ? threadIdx.x >> 6 : 0;
  const int64_t b = (int64_t)blockIdx.x * C::MW + m;
  if (C::MW > 1 && b >= batch) return;  // whole waves; no workgroup barrier is used then
  float* const T = Ts[m];
  const int tid = C::MW > 1 ? threadIdx.x & 63 : threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g = lane >> 4;
  {
    constexpr int NV = N * N / 4, PER = (NV + TM - 1) / TM;
    const float4* src = reinterpret_cast<const float4*>(LU + b * (int64_t)N * N);
    float4 v[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + TM * u;
      v[u] = src[NV % TM == 0 ? e : min(e, NV - 1)];
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + TM * u;
      if (NV % TM == 0 || e < NV) *reinterpret_cast<float4*>(T + (e / (N / 4)) * LD + 4 * (e % (N / 4))) = v[u];
    }
  }
  const int j[2] = {wave, NB - 1 - wave};
  const bool two = j[1] > j[0];
  const int row[2] = {g0[b * N + 16 * j[0] + li], g0[b * N + 16 * j[1] + li]};
  const float sgn = sign[b];
  mat_sync<NW>();

  // DET, singular members: the zero pivots, their count and s (wave-uniform, formed alike by
  // every wave from the untouched diagonal)
  int k1 = 0, k2 = 0, nz = 0;
  float s1 = 0.0f;
  float det = 1.0f;
  if constexpr (DET) {
    constexpr int H = (N + 63) / 64;
    // |det| as the product of the pivots' mantissas and the sum of their exponents: exp of a float
    // logabs has the log's rounding, 2^-25 of it, in every entry (det's gradient B = 20000, n = 14
    // against 64-bit results 4.4e-7 -> 2.9e-7, B = 400, n = 128 to 0.37 of the error)
    double pm = 1.0;
    int px = 0;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int i = lane + 64 * h;
      const double d = i < N ? (double)T[i * LD + i] : 1.0;
      pm *= __builtin_amdgcn_frexp_mant(d);
      px += __builtin_amdgcn_frexp_exp(d);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      pm *= __shfl_xor(pm, o);
      px += __shfl_xor(px, o);
    }
    det = (float)ldexp(fabs(pm), px);
    if (sgn == 0.0f) {
      float lg = 0.0f;
      int odd = 0, last = -1;
      k1 = N;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const int i = lane + 64 * h;
        const float d = i < N ? T[i * LD + i] : 1.0f;
        const unsigned long long z = __ballot(d == 0.0f);
        nz += __popcll(z);
        odd += __popcll(__ballot(d < 0.0f));
        if (z) {
          k1 = min(k1, 64 * h + (int)__builtin_ctzll(z));
          last = 64 * h + 63 - (int)__builtin_clzll(z);
        }
        lg += d != 0.0f ? logf(fabsf(d)) : 0.0f;
      }
      k2 = last;
      lg = wave_sum_f32(lg);
      // parity of P by its inversions
      for (int h = 0; h < H; ++h) {
        const int i = lane + 64 * h;
        const int pi = i < N ? g0[b * N + i] : -1;
#pragma unroll 1
        for (int q = 0; q < N; ++q) odd += __popcll(__ballot(i < N && q < i && g0[b * N + q] > pi));
      }
      s1 = (nz >= 3 || k2 >= n || k2 < 0) ? 0.0f : ((odd & 1) ? -1.0f : 1.0f) * expf(lg);
      mat_sync<NW>();
    }
  }

  invert_diagonals<NB, true>(T, wave, lane);
  mat_sync<NW>();

  // z = -L^-1, then -X by back substitution, in place
  v4f z[2][NB];
  solve_lower<NB>(T, j, two, li, g, z);
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  static_for<0, NB>([&](auto ic_) {
    constexpr int i = NB - 1 - decltype(ic_)::value;
    v4f a[NB - i];
    static_for<i + 1, NB>([&](auto kc) { a[kc.value - i - 1] = left_op<LD>(T, i, kc.value, li, g); });
    const v4f inv = left_upper<LD>(T, i, li, g);
#pragma unroll
    for (int c = 0; c < 2; ++c) z[c][i] = -z[c][i];
    static_for<i + 1, NB>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      z[0][i] = mul16(a[k - i - 1], z[0][k], z[0][i]);
      if (two) z[1][i] = mul16(a[k - i - 1], z[1][k], z[1][i]);
    });
    z[0][i] = -mul16(inv, z[0][i], zero);
    if (two) z[1][i] = -mul16(inv, z[1][i], zero);
  });

  bool nf = zero_singular && sgn == 0.0f;
  static_for<0, NB>([&](auto ic_) {
    constexpr int i = decltype(ic_)::value;
#pragma unroll
    for (int v = 0; v < 4; ++v) nf = nf | !isfinite(z[0][i][v]) | !isfinite(z[1][i][v]);
  });

  float* const ob = out + b * (int64_t)n * n;
  if constexpr (DET) {
    if (sgn == 0.0f) {
      // u = U~^-1 e_k1 (and (U~^-1)[k1][k2]) by blocks, on the matrix's first wave
      float* const u = vecs[m];
      float* const col = u + N;
      float* const ts = col + N;
      if (wave == 0 && s1 != 0.0f) {
        for (int pass = nz == 2 ? 0 : 1; pass < 2; ++pass) {
          const int kt = pass ? k1 : k2;
          for (int i = lane; i < N; i += 64) u[i] = 0.0f;
          wave_lds_fence();
          for (int i = kt >> 4; i >= 0; --i) {
            float t = 16 * i + li == kt ? 1.0f : 0.0f;
            for (int c = 16 * (i + 1); c <= kt; ++c) t = fmaf(-T[(16 * i + li) * LD + c], u[c], t);
            if (lane < 16) ts[li] = t;
            wave_lds_fence();
            float x = 0.0f;
#pragma unroll 1
            for (int c = 0; c < 16; ++c) x = c >= li ? fmaf(T[(16 * i + li) * LD + 16 * i + c], ts[c], x) : x;
            if (lane < 16) u[16 * i + li] = x;
            wave_lds_fence();
          }
          if (!pass) s1 *= u[k1];
          wave_lds_fence();
        }
      }
      // column k2 of A~^-T
      const int i2 = (k2 < 0 ? 0 : k2) >> 4, r2 = k2 & 15;
      static_for<0, NB>([&](auto ic_) {
        constexpr int i = decltype(ic_)::value;
        if (i == i2 && g == r2 >> 2) {
          static_for<0, 2>([&](auto cc_) {
            constexpr int c = decltype(cc_)::value;
            const v4f zz = opaque4(z[c][i]);
            const float x = (r2 & 2) ? ((r2 & 1) ? zz[3] : zz[2]) : ((r2 & 1) ? zz[1] : zz[0]);
            if ((c == 0 || two) && row[c] < N) col[row[c]] = -x;
          });
        }
      });
      if (wave == 0 && lane == 0) ts[0] = s1;
      const bool bad = mat_any<NW>(nf);
      const float sv = ts[0];
      for (int e = tid; e < n * n; e += TM) {
        const int r = e / n, c = e - r * n;
        ob[e] = bad || sv == 0.0f ? 0.0f : sv * col[r] * u[c];
      }
      return;
    }
  }
  const bool bad = mat_any<NW>(nf);  // also: every wave is done with T
  const float sc = DET ? -sgn * det : (scale ? -scale[b] : -1.0f);
  if ((n & 3) == 0) {
    // a lane's four rows of one column of X: 16 consecutive bytes of an output row
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if ((c == 0 || two) && row[c] < n) {
        float* o = ob + (int64_t)row[c] * n + 4 * g;
#pragma unroll
        for (int i = 0; i < NB; ++i)
          if (16 * i + 4 * g < n) *reinterpret_cast<v4f*>(o + 16 * i) = bad ? zero : sc * opaque4(z[c][i]);
      }
    }
  } else {
    // rows of the output are not 16-byte aligned: through LDS, whole rows per wave
#pragma unroll
    for (int c = 0; c < 2; ++c)
      if ((c == 0 || two) && row[c] < n) {
#pragma unroll
        for (int i = 0; i < NB; ++i) *reinterpret_cast<v4f*>(T + row[c] * LD + 16 * i + 4 * g) = bad ? zero : sc * opaque4(z[c][i]);
      }
    mat_sync<NW>();
    if ((n & 1) == 0) {
      for (int r = wave; r < n; r += NW)
        if (2 * lane < n)
          *reinterpret_cast<float2*>(ob + (int64_t)r * n + 2 * lane) = *reinterpret_cast<const float2*>(T + r * LD + 2 * lane);
    } else {
      for (int r = wave; r < n; r += NW)
        for (int e = lane; e < n; e += 64) ob[(int64_t)r * n + e] = T[r * LD + e];
    }
  }
}

// ------------------------------------------------------------------ Parlett-Reid

// w_x v_y - v_x w_y, both products rounded alike (no fma), so exactly odd under x <-> y.
__device__ __forceinline__ float wedge(float wx, float vy, float vx, float wy) {
#pragma clang fp contract(off)
  return wx * vy - vx * wy;
}

// out[b] = scale[b] S^-1, or scale[b] pf(S) S^-1 with adjugate, from the Parlett-Reid factors
// (gbuf in chunks of PB columns by original row, pivots d, final position -> row perm):
// with d~ = d, d_K (the smallest) and exact zeros replaced by 1, L~ = L with the a-columns
// scaled by 1 / d~, Y = L~^-1 and R = Y^T D~^-1 Y,
//   G = -P^T [a1 R + a2 (w v^T - v w^T)] P,  w = R e_2K, v = Y^T e_2K,
// inverse (a1, a2) = (1, (1 - d_K) / d_K), zero for d_K = 0 or a non-finite result;
// adjugate (a1, a2) = sgn(P) D_K (d_K, 1 - d_K), a second exact zero pivot z lifted: the
// mean of the evaluations with d_z = +1 and -1 (the second only for such members).
// Y's block columns stay in registers (DY, the right operand, is a swap of a lane's own
// rows) and are exchanged once through LDS as left operands, 16 bytes per lane; R's lower
// tiles go back to LDS mirrored and in the output's order. Measured, slogpf forward + gradient
// B = 2000, n = 90: 520 us as six launches (assembly, inverse, product, vectors, gather,
// guard) -> 134 us.
template <int NB>
__global__ __launch_bounds__(SmallInv<NB>::NT, SmallInv<NB>::WPE) void pf_inv_small_kernel(
    const float* __restrict__ gbuf, int PB, const float* __restrict__ d, const int* __restrict__ perm, int n,
    int64_t batch, int adjugate, const float* __restrict__ scale, float* __restrict__ out) {
  using C = SmallInv<NB>;
  constexpr int N = C::N, LD = C::LD, NW = C::NW, TM = 64 * NW;
  __shared__ __align__(16) float Ts[C::MW][N * LD];
  __shared__ __align__(16) float dis[C::MW][N / 2], dts[C::MW][NB == 1 ? N / 2 : 1];
  __shared__ __align__(16) int ps[C::MW][N];
  __shared__ __align__(16) float ws[C::MW][N], vs[C::MW][N];
  __shared__ int inv_odd[C::MW][NW];
  const int m = C::MW > 1 ? threadIdx.x >> 6 : 0;
  const int64_t b = (int64_t)blockIdx.x * C::MW + m;
  if (C::MW > 1 && b >= batch) return;  // whole waves; no workgroup barrier is used then
  float* const T = Ts[m];
  float* const di = dis[m];
  int* const p = ps[m];
  int tid = C::MW > 1 ? threadIdx.x & 63 : threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63;
  for (int f = tid; f < N; f += TM) p[f] = perm[b * N + f];
  mat_sync<NW>();

  // K, the coefficients and 1 / d~: every wave forms them alike (at most one pair per lane)
  constexpr int H = N / 2;
  const float dl = lane < H ? d[b * H + lane] : 1.0f;
  const unsigned key = lane < n / 2 ? __float_as_uint(fabsf(dl)) : 0xffffffffu;
  const unsigned kmin = ~wave_max_u32(~key);
  const int K = first_lane(key == kmin);
  const float dK = readlane_f(dl, K);
  const bool other = lane < H && lane != K;
  float dt = (lane == K || dl == 0.0f) ? 1.0f : dl;
  float dinv = 1.0f / dt;
  float a1 = 1.0f, a2 = dK != 0.0f ? (1.0f - dK) / dK : 0.0f;
  int lift = -1;
  if (adjugate) {
    // parity of P by its inversions: one row per thread
    const int f = tid;
    bool odd = false;
    if (f < N) {
      const int pf = p[f];
#pragma unroll 1
      for (int q = 0; q < N; q += 4) {
        const int4 pq = *reinterpret_cast<const int4*>(p + q);
        odd ^= (q < f && pq.x > pf) ^ (q + 1 < f && pq.y > pf) ^ (q + 2 < f && pq.z > pf) ^ (q + 3 < f && pq.w > pf);
      }
    }
    int cnt = __popcll(__ballot(odd));
    if constexpr (NW > 1) {
      if (lane == 0) inv_odd[m][wave] = cnt;
      __syncthreads();
      cnt = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) cnt += inv_odd[m][w];
    }
    const float lg = wave_sum_f32(other && dl != 0.0f ? logf(fabsf(dl)) : 0.0f);
    const unsigned long long zm = __ballot(other && dl == 0.0f);
    cnt += __popcll(__ballot(other && dl < 0.0f));
    lift = zm ? (int)__builtin_ctzll(zm) : -1;
    const float D = __popcll(zm) > 1 ? 0.0f : ((cnt & 1) ? -1.0f : 1.0f) * expf(lg) * (zm ? 0.5f : 1.0f);
    a1 = D * dK;
    a2 = D * (1.0f - dK);
  }
  const float sc = scale ? scale[b] : 1.0f;
  const int j[2] = {wave, NB - 1 - wave};
  const bool two = j[1] > j[0];
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float* const ob = out + b * (int64_t)n * n;

  for (int pass = 0; pass < (lift >= 0 ? 2 : 1); ++pass) {
    // lane-derived masks and addresses are formed anew in each evaluation, not held across
    asm volatile("" : "+v"(tid), "+v"(lane));
    const int li = lane & 15, g = lane >> 4;
    if (pass) {
      if (lane == lift) dinv = dt = -1.0f;
      a1 = -a1;
      a2 = -a2;
      mat_sync<NW>();  // the first evaluation's output has been read from LDS
    }
    if (wave == 0 && lane < H) {
      di[lane] = dinv;
      if constexpr (NB == 1) dts[m][lane] = dt;
    }
    mat_sync<NW>();
    // L~ by 16 x 16 blocks (I, J), J <= I, a block per wave step: lane (r, c) moves columns
    // 4 c .. 4 c + 3 of row r (original row p[f]). Column a = 2 s holds w / d~ (G column
    // 2 t + 1), column p = 2 s + 1 holds tau
    {
      constexpr int NBLK = NB * (NB + 1) / 2, PER = (NBLK + NW - 1) / NW;
      const float* gb = gbuf + b * (int64_t)N * N;
      float4 v[PER];
      int f[PER], c[PER];
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        int J = NBLK % NW == 0 ? wave + NW * u : min(wave + NW * u, NBLK - 1), I = 0;
        while (J > I) J -= ++I;
        f[u] = 16 * I + (lane >> 2);
        c[u] = 16 * J + 4 * (lane & 3);
        v[u] = *reinterpret_cast<const float4*>(gb + ((int64_t)(c[u] / PB) * N + p[f[u]]) * PB + c[u] % PB);
      }
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const float2 dd = *reinterpret_cast<const float2*>(di + (c[u] >> 1));
        float4 w;
        float wx = v[u].y * dd.x, wz = v[u].w * dd.y;
        if constexpr (NB == 1) {  // divided: in sums of at most 16 the reciprocals' roundings show
          const float2 e = *reinterpret_cast<const float2*>(dts[m] + (c[u] >> 1));
          wx = v[u].y / e.x;
          wz = v[u].w / e.y;
        }
        w.x = f[u] > (c[u] | 1) ? wx : 0.0f;
        w.y = f[u] > (c[u] | 1) ? v[u].x : 0.0f;
        w.z = f[u] > ((c[u] + 2) | 1) ? wz : 0.0f;
        w.w = f[u] > ((c[u] + 2) | 1) ? v[u].z : 0.0f;
        *reinterpret_cast<float4*>(T + f[u] * LD + c[u]) = w;
      }
    }
    mat_sync<NW>();
    invert_diagonals<NB, false>(T, wave, lane);
    mat_sync<NW>();
    v4f z[2][NB];
    solve_lower<NB>(T, j, two, li, g, z);
    mat_sync<NW>();
    // Y's blocks (k, jj), k >= jj, as left operands of Y^T: the lane's own four rows
    static_for<0, NB>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      float* const f = T + k * (k + 1) / 2 * 256 + 4 * lane;
      if (k >= j[0]) *reinterpret_cast<v4f*>(f + 256 * j[0]) = -opaque4(z[0][k]);
      if (two && k >= j[1]) *reinterpret_cast<v4f*>(f + 256 * j[1]) = -opaque4(z[1][k]);
    });
    mat_sync<NW>();
    // v = Y^T e_2K by position
    float vpos = 0.0f;
    if (tid < N) {
      const int kb = (2 * K) >> 4, r = (2 * K) & 15;
      if ((tid >> 4) <= kb) vpos = T[(kb * (kb + 1) / 2 + (tid >> 4)) * 256 + 4 * (16 * (r >> 2) + (tid & 15)) + (r & 3)];
    }
    // DY = rows (Y[p_s], -Y[a_s]) / d~_s; z holds -Y
    static_for<0, NB>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const float2 dd = *reinterpret_cast<const float2*>(di + 8 * k + 2 * g);
      static_for<0, 2>([&](auto cc_) {
        constexpr int c = decltype(cc_)::value;
        const v4f y = z[c][k];
        if constexpr (NB == 1) {
          const float2 e = *reinterpret_cast<const float2*>(dts[m] + 2 * g);
          z[c][k] = v4f{-y[1] / e.x, y[0] / e.x, -y[3] / e.y, y[2] / e.y};
        } else {
          z[c][k] = v4f{-y[1] * dd.x, y[0] * dd.x, -y[3] * dd.y, y[2] * dd.y};
        }
      });
    });
    // R(i, j) = sum_{k >= i} Y(k, i)^T DY(k, j), tiles i >= j
    v4f r[2][NB];
    static_for<0, NB>([&](auto ic_) {
      constexpr int i = decltype(ic_)::value;
      r[0][i] = zero;
      r[1][i] = zero;
      if (i >= j[0]) {
        v4f a[NB - i];
        static_for<i, NB>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          a[k - i] = *reinterpret_cast<const v4f*>(T + (k * (k + 1) / 2 + i) * 256 + 4 * lane);
        });
        static_for<i, NB>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          r[0][i] += mul16_pairs(a[k - i], z[0][k]);
          if (two && i >= j[1]) r[1][i] += mul16_pairs(a[k - i], z[1][k]);
        });
      }
    });
    mat_sync<NW>();
    // R and the two vectors in the output's order; the diagonal is exactly zero
    if (tid < N) vs[m][p[tid]] = vpos;
    static_for<0, 2>([&](auto cc_) {
      constexpr int c = decltype(cc_)::value;
      if (c == 0 || two) {
        const int cc = 16 * j[c] + li, pc = p[cc];
        static_for<0, NB>([&](auto ic_) {
          constexpr int i = decltype(ic_)::value;
          if (i >= j[c]) {
            const int4 pf = *reinterpret_cast<const int4*>(p + 16 * i + 4 * g);
            const int pr[4] = {pf.x, pf.y, pf.z, pf.w};
            const v4f t = opaque4(r[c][i]);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int f = 16 * i + 4 * g + v;
              if (f >= cc) {
                const float x = f > cc ? t[v] : 0.0f;
                T[pr[v] * LD + pc] = x;
                T[pc * LD + pr[v]] = -x;
              }
            }
          }
        });
      }
    });
    mat_sync<NW>();
    const int pK = p[2 * K];
    for (int x = tid; x < N; x += TM) ws[m][x] = T[x * LD + pK];
    mat_sync<NW>();
    bool nf = dK == 0.0f;
    if ((n & 3) == 0) {
      const int n4 = n >> 2;
      for (int e = tid; e < n * n4; e += TM) {
        const int x = e / n4, y = 4 * (e - x * n4);
        const float wx = ws[m][x], vx = vs[m][x];
        const v4f rr = *reinterpret_cast<const v4f*>(T + x * LD + y);
        const v4f wy = *reinterpret_cast<const v4f*>(&ws[m][y]), vy = *reinterpret_cast<const v4f*>(&vs[m][y]);
        v4f val;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          val[v] = -(a1 * rr[v] + a2 * wedge(wx, vy[v], vx, wy[v]));
          nf = nf || !isfinite(val[v]);
        }
        v4f* o = reinterpret_cast<v4f*>(ob + 4 * e);
        *o = pass ? *o + sc * val : sc * val;
      }
    } else {  // n is even: 8-byte rows
      const int n2 = n >> 1;
      for (int e = tid; e < n * n2; e += TM) {
        const int x = e / n2, y = 2 * (e - x * n2);
        const float wx = ws[m][x], vx = vs[m][x];
        const float2 rr = *reinterpret_cast<const float2*>(T + x * LD + y);
        const float2 wy = *reinterpret_cast<const float2*>(&ws[m][y]), vy = *reinterpret_cast<const float2*>(&vs[m][y]);
        const float v0 = -(a1 * rr.x + a2 * wedge(wx, vy.x, vx, wy.x));
        const float v1 = -(a1 * rr.y + a2 * wedge(wx, vy.y, vx, wy.y));
        nf = nf || !isfinite(v0) || !isfinite(v1);
        float2* o = reinterpret_cast<float2*>(ob + 2 * e);
        const float2 old = pass ? *o : make_float2(0.0f, 0.0f);
        *o = make_float2(old.x + sc * v0, old.y + sc * v1);
      }
    }
    // inverse mode: a member with d_K = 0 or a non-finite value is cleared (each thread
    // rewrites entries of its own)
    if (!adjugate && mat_any<NW>(nf)) {
      if ((n & 3) == 0) {
        for (int e = tid; e < n * (n >> 2); e += TM) *reinterpret_cast<v4f*>(ob + 4 * e) = zero;
      } else {
        for (int e = tid; e < n * (n >> 1); e += TM) *reinterpret_cast<float2*>(ob + 2 * e) = make_float2(0.0f, 0.0f);
      }
    }
  }
}

template <int NB>
void launch_lu(const float* LU, const int* g0, int n, int64_t batch, const float* sign, const float* scale,
               int zero_singular, bool det, float* out, hipStream_t s) {
  using C = SmallInv<NB>;
  const dim3 grid((unsigned)((batch + C::MW - 1) / C::MW));
  if (det)
    hipLaunchKernelGGL((lu_inv_small_kernel<NB, true>), grid, dim3(C::NT), 0, s, LU, g0, n, batch, sign, scale,
                       zero_singular, out);
  else
    hipLaunchKernelGGL((lu_inv_small_kernel<NB, false>), grid, dim3(C::NT), 0, s, LU, g0, n, batch, sign, scale,
                       zero_singular, out);
}

template <int NB>
void launch_pf(const float* gbuf, int PB, const float* d, const int* perm, int n, int64_t batch, int adjugate,
               const float* scale, float* out, hipStream_t s) {
  using C = SmallInv<NB>;
  hipLaunchKernelGGL((pf_inv_small_kernel<NB>), dim3((unsigned)((batch + C::MW - 1) / C::MW)), dim3(C::NT), 0, s, gbuf,
                     PB, d, perm, n, batch, adjugate, scale, out);
}

}  // namespace

int launch_lu_inv_small(const float* LU, const int* g0, int N, int n, int64_t batch, const float* sign,
                        const float* scale, int zero_singular, bool det, float* out, hipStream_t s) {
  if (N % 16 || N > SMALL_INV_MAXN || n > N) return FX_ERR_UNSUPPORTED;
  switch (N / 16) {
    case 1: launch_lu<1>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 2: launch_lu<2>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 3: launch_lu<3>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 4: launch_lu<4>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 5: launch_lu<5>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 6: launch_lu<6>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    case 7: launch_lu<7>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
    default: launch_lu<8>(LU, g0, n, batch, sign, scale, zero_singular, det, out, s); break;
  }
  return hipGetLastError() == hipSuccess ? FX_OK : FX_ERR_LAUNCH;
}

int launch_pf_inv_small(const float* gbuf, int PB, const float* d, const int* perm, int N, int n, int64_t batch,
                        int adjugate, const float* scale, float* out, hipStream_t s) {
  if (N % 16 || N > SMALL_INV_MAXN || n > N) return FX_ERR_UNSUPPORTED;
  switch (N / 16) {
    case 1: launch_pf<1>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 2: launch_pf<2>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 3: launch_pf<3>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 4: launch_pf<4>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 5: launch_pf<5>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 6: launch_pf<6>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    case 7: launch_pf<7>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
    default: launch_pf<8>(gbuf, PB, d, perm, n, batch, adjugate, scale, out, s); break;
  }
  return hipGetLastError() == hipSuccess ? FX_OK : FX_ERR_LAUNCH;
}

}  // namespace fx
