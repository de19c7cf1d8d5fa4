// Device stages fused around the FFT passes: the directional-stiffness
// product K : p before the forward transform, the Green-operator projection
// per wave vector between the transforms, and block reductions for the
// p . Ap partial sums after the inverse transform.
#pragma once
#include "mugpu_internal.hpp"

namespace mugpu {

// ---- symmetric fields (small strain) ---------------------------------------------
// The small-strain projection takes and gives symmetric tensors, and K : p of
// an isotropic tangent is symmetric: the spectra between the passes then hold
// the dim (dim + 1) / 2 independent components (Voigt order: the diagonal, then
// yz, xz, xy) instead of dim^2, 2/3 (3D) or 3/4 (2D) of the bytes and of the
// transforms.  The projection of a field is that of its symmetric part, which
// is taken when a field enters.  Measured per launch at 128^3 FP64: middle axis
// 56 + 46 -> 38 + 32 us, first axis 62 -> 44 (in the variant best for six lines),
// c2r 98 -> 76.
__host__ __device__ constexpr int sym_lines(int dim) { return dim * (dim + 1) / 2; }
// lines per row or k-point: packed or one per component
__host__ __device__ constexpr int nb_lines(int dim, bool packed) {
  return packed ? sym_lines(dim) : dim * dim;
}
template <int DIM>
__host__ __device__ constexpr int sym_line(int i, int j) {
  return i == j ? i : DIM == 3 ? 6 - (i + j) : 2;
}
// line of component c = i + dim j
template <int DIM, bool PK>
__host__ __device__ constexpr int line_of(int c) {
  return PK ? sym_line<DIM>(c % DIM, c / DIM) : c;
}
// components i + DIM j and j + DIM i of line c
template <int DIM>
__host__ __device__ __forceinline__ void sym_pair(int c, int& a, int& b) {
  a = DIM == 3 ? (0x367840 >> (4 * c)) & 15 : (0x230 >> (4 * c)) & 15;
  b = DIM == 3 ? (0x125840 >> (4 * c)) & 15 : (0x130 >> (4 * c)) & 15;
}
template <typename T, int DIM>
__device__ __forceinline__ void unpack_lines(const T* q, T* f) {
#pragma unroll
  for (int c = 0; c < DIM * DIM; ++c) f[c] = q[line_of<DIM, true>(c)];
}
template <typename T, int DIM, bool PK>
__device__ __forceinline__ void pack_lines(const T* f, T* q) {
  if constexpr (PK) {
#pragma unroll
    for (int j = 0; j < DIM; ++j)
#pragma unroll
      for (int i = 0; i <= j; ++i)
        q[sym_line<DIM>(i, j)] = i == j ? f[i + DIM * i] : T(0.5) * (f[i + DIM * j] + f[j + DIM * i]);
  } else {
#pragma unroll
    for (int c = 0; c < DIM * DIM; ++c) q[c] = f[c];
  }
}

// ---- tangents kept as factors ------------------------------------------------------
// LEF: q holds F, S and (lambda, mu); p, dp at i + DIM j
template <typename T, int DIM>
__host__ __device__ __forceinline__ void lef_product(const T* q, const T* p, T* dp) {
  constexpr int NC = DIM * DIM, NL = sym_lines(DIM);
  const T *F = q, *S = q + NC;
  const T lam = q[NC + NL], mu = q[NC + NL + 1];
  T e[NC], tr = 0;  // F^T dF
#pragma unroll
  for (int j = 0; j < DIM; ++j)
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      T s = 0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) s += F[k + DIM * i] * p[k + DIM * j];
      e[i + DIM * j] = s;
      if (i == j) tr += s;
    }
#pragma unroll
  for (int j = 0; j < DIM; ++j)
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      T s = 0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) {
        const T t = (k == j ? lam * tr : T(0)) + mu * (e[k + DIM * j] + e[j + DIM * k]);
        s += p[i + DIM * k] * S[sym_line<DIM>(k, j)] + F[i + DIM * k] * t;
      }
      dp[i + DIM * j] = s;
    }
}

// HCT: the consistent HEP1 tangent (materials.hip) in the eigenbasis V of the
// trial b_e.  With H = V^T F^-T, D = V^T dF, Q = D H^T and t, n the eigenvalues of
// tau and N, b those of b_e and g the divided differences of ln:
//   dP = V [C(M) - diag(t) Q^T] H,  M_mm = 2 Q_mm,
//   M_mn = g_mn (b_n Q_mn + b_m Q_nm),
//   C(M) = c1 tr(M) I + c2 M + c3 diag(n) (n . diag M),  t_m = t0 + t1 n_m
// q: [0, 4) V as a unit quaternion, [4, 13) H, [13, 19) g_mn b_n for (m, n) =
// 01, 10, 02, 20, 12, 21, [19] c1, [20] c2, [21] c3, [22] n_0, [23] n_1 (n is
// traceless), [24] t0, [25] t1
template <typename T>
__host__ __device__ __forceinline__ void hct_product(const T* q, const T* p, T* dp) {
  T V[9];
  {
    const T w = q[0], x = q[1], y = q[2], z = q[3];
    V[0] = 1 - 2 * (y * y + z * z);
    V[1] = 2 * (x * y + w * z);
    V[2] = 2 * (x * z - w * y);
    V[3] = 2 * (x * y - w * z);
    V[4] = 1 - 2 * (x * x + z * z);
    V[5] = 2 * (y * z + w * x);
    V[6] = 2 * (x * z + w * y);
    V[7] = 2 * (y * z - w * x);
    V[8] = 1 - 2 * (x * x + y * y);
  }
  const T* H = q + 4;
  T D[9], Q[9], A[9];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int m = 0; m < 3; ++m) D[m + 3 * j] = V[3 * m] * p[3 * j] + V[1 + 3 * m] * p[1 + 3 * j] + V[2 + 3 * m] * p[2 + 3 * j];
#pragma unroll
  for (int n = 0; n < 3; ++n)
#pragma unroll
    for (int m = 0; m < 3; ++m) Q[m + 3 * n] = D[m] * H[n] + D[m + 3] * H[n + 3] + D[m + 6] * H[n + 6];
  const T n0 = q[22], n1 = q[23], n2 = -n0 - n1;
  const T m0 = 2 * Q[0], m1 = 2 * Q[4], m2 = 2 * Q[8];
  const T ct = q[19] * (m0 + m1 + m2), c2 = q[20], nm = q[21] * (n0 * m0 + n1 * m1 + n2 * m2);
  const T m01 = c2 * (q[13] * Q[3] + q[14] * Q[1]);
  const T m02 = c2 * (q[15] * Q[6] + q[16] * Q[2]);
  const T m12 = c2 * (q[17] * Q[7] + q[18] * Q[5]);
  const T t0 = q[24] + q[25] * n0, t1 = q[24] + q[25] * n1, t2 = q[24] + q[25] * n2;
  // A = C(M) - diag(t) Q^T
  A[0] = ct + c2 * m0 + n0 * nm - t0 * Q[0];
  A[4] = ct + c2 * m1 + n1 * nm - t1 * Q[4];
  A[8] = ct + c2 * m2 + n2 * nm - t2 * Q[8];
  A[3] = m01 - t0 * Q[1];
  A[1] = m01 - t1 * Q[3];
  A[6] = m02 - t0 * Q[2];
  A[2] = m02 - t2 * Q[6];
  A[7] = m12 - t1 * Q[5];
  A[5] = m12 - t2 * Q[7];
  // dP = V (A H)
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    T b[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) b[m] = A[m] * H[3 * j] + A[m + 3] * H[1 + 3 * j] + A[m + 6] * H[2 + 3 * j];
#pragma unroll
    for (int i = 0; i < 3; ++i) dp[i + 3 * j] = V[i] * b[0] + V[i + 3] * b[1] + V[i + 6] * b[2];
  }
}

// dp = K : p for voxel v in the cell's tangent representation (blocked
// layout of tan_off(); lanes on consecutive voxels read contiguous runs)
template <typename T, int DIM>
__device__ __forceinline__ void tangent_product(int kind, const T* __restrict__ tan,
                                                int64_t v, const T* p, T* dp) {
  constexpr int NC = DIM * DIM;
  if (kind == TAN_ISO) {
    const T lam = tan[tan_off(v, 0, 2)], mu = tan[tan_off(v, 1, 2)];
    T tr = 0;
#pragma unroll
    for (int i = 0; i < DIM; ++i) tr += p[i * (DIM + 1)];
#pragma unroll
    for (int j = 0; j < DIM; ++j)
#pragma unroll
      for (int i = 0; i < DIM; ++i)
        dp[i + DIM * j] = (i == j ? lam * tr : T(0)) + mu * (p[i + DIM * j] + p[j + DIM * i]);
  } else if (sizeof(T) == 8 && kind == TAN_LEF) {
    constexpr int S = NC + sym_lines(DIM) + 2;
    const T* K = tan + tan_off(v, 0, S);
    T q[S];
#pragma unroll
    for (int i = 0; i < S; ++i) q[i] = K[i * kTanBlock];
    lef_product<T, DIM>(q, p, dp);
  } else if (sizeof(T) == 8 && DIM == 3 && kind == TAN_HCT) {
    const T* K = tan + tan_off(v, 0, kHct);
    T q[kHct];
#pragma unroll
    for (int i = 0; i < kHct; ++i) q[i] = K[i * kTanBlock];
    if constexpr (DIM == 3) hct_product<T>(q, p, dp);
  } else if (kind == TAN_HEP) {
    constexpr int S = DIM * DIM * DIM;
    const T* M = tan + tan_off(v, 0, S);
    T s[DIM];
#pragma unroll
    for (int n = 0; n < DIM; ++n) {
      T a = 0;
#pragma unroll
      for (int j = 0; j < DIM; ++j) a += p[j + DIM * n];
      s[n] = a;
    }
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      T a = 0;
#pragma unroll
      for (int n = 0; n < DIM; ++n) a += M[(q + NC * n) * kTanBlock] * s[n];
      dp[q] = a;
    }
  } else if (kind == TAN_SYM) {
    constexpr int S = NC * (NC + 1) / 2;
    const T* K = tan + tan_off(v, 0, S);
#pragma unroll
    for (int r = 0; r < NC; ++r) dp[r] = T(0);
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      const T kd = K[sym_index(r, r, NC) * kTanBlock];
      dp[r] += kd * p[r];
#pragma unroll
      for (int c = r + 1; c < NC; ++c) {
        const T k = K[sym_index(r, c, NC) * kTanBlock];
        dp[r] += k * p[c];
        dp[c] += k * p[r];
      }
    }
  } else {
    const T* K = tan + tan_off(v, 0, NC * NC);
#pragma unroll
    for (int r = 0; r < NC; ++r) {
      T a = 0;
#pragma unroll
      for (int c = 0; c < NC; ++c) a += K[(r + NC * c) * kTanBlock] * p[c];
      dp[r] = a;
    }
  }
}

template <typename T>
__device__ __forceinline__ T fft_freq(int c, int n, double L) {
  // numpy fftfreq(n)*n order divided by the length (src/fft/fft_utils.cc:41-56)
  const int npos = (n - 1) / 2 + 1;
  return T((double)(c < npos ? c : c - n) / L);
}

// Green-operator projection of the nc complex components of one wave
// vector, f[(i + DIM j) * stride], in place, with unit wave vector xi and the
// normalisation 1/N folded in:
//   small strain (src/fft/projection_small_strain.cc:61-85):
//     G f = (xi_i a_j + xi_i b_j + xi_j a_i + xi_j b_i)/2 - xi_i xi_j s,
//     a = f xi, b = f^T xi, s = xi^T f xi
//   finite strain (projection_finite_strain_fast.cc:65-85 and the full-G
//   variant, projection_finite_strain.cc:61-95, which is the same operator):
//     f_ij <- (sum_k f_ik xi_k) xi_j
template <typename T, int DIM>
__device__ __forceinline__ void project_point(c_t<T>* f, int stride, const T* xi, int kind,
                                              T norm) {
  constexpr int NC = DIM * DIM;
  T fr[NC], fi[NC];
#pragma unroll
  for (int r = 0; r < NC; ++r) {
    const c_t<T> v = f[r * stride];
    fr[r] = v.x;
    fi[r] = v.y;
  }
  if (kind == MUGPU_PROJ_SMALL_STRAIN) {
    T ar[DIM], br[DIM], ai[DIM], bi[DIM];
    T sr_ = 0, si_ = 0;
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      T a1 = 0, b1 = 0, a2 = 0, b2 = 0;
#pragma unroll
      for (int m = 0; m < DIM; ++m) {
        a1 += fr[i + DIM * m] * xi[m];
        a2 += fi[i + DIM * m] * xi[m];
        b1 += fr[m + DIM * i] * xi[m];
        b2 += fi[m + DIM * i] * xi[m];
      }
      ar[i] = a1;
      ai[i] = a2;
      br[i] = b1;
      bi[i] = b2;
      sr_ += xi[i] * a1;
      si_ += xi[i] * a2;
    }
#pragma unroll
    for (int j = 0; j < DIM; ++j)
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        const T gr = T(0.5) * (xi[i] * ar[j] + xi[i] * br[j] + xi[j] * ar[i] + xi[j] * br[i]) -
                     xi[i] * xi[j] * sr_;
        const T gi = T(0.5) * (xi[i] * ai[j] + xi[i] * bi[j] + xi[j] * ai[i] + xi[j] * bi[i]) -
                     xi[i] * xi[j] * si_;
        c_t<T> g;
        g.x = norm * gr;
        g.y = norm * gi;
        f[(i + DIM * j) * stride] = g;
      }
  } else {
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      T s1 = 0, s2 = 0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) {
        s1 += fr[i + DIM * k] * xi[k];
        s2 += fi[i + DIM * k] * xi[k];
      }
#pragma unroll
      for (int j = 0; j < DIM; ++j) {
        c_t<T> g;
        g.x = norm * (s1 * xi[j]);
        g.y = norm * (s2 * xi[j]);
        f[(i + DIM * j) * stride] = g;
      }
    }
  }
}

// the small-strain projection of packed lines: with a = f xi, s = xi . a,
//   G f = xi_i a_j + xi_j a_i - xi_i xi_j s
template <typename T, int DIM>
__device__ __forceinline__ void project_point_sym(c_t<T>* f, const T* xi, T norm) {
  constexpr int NL = sym_lines(DIM);
  c_t<T> v[NL];
#pragma unroll
  for (int r = 0; r < NL; ++r) v[r] = f[r];
  T ar[DIM], ai[DIM], sr_ = 0, si_ = 0;
#pragma unroll
  for (int i = 0; i < DIM; ++i) {
    T a1 = 0, a2 = 0;
#pragma unroll
    for (int m = 0; m < DIM; ++m) {
      a1 += v[sym_line<DIM>(i, m)].x * xi[m];
      a2 += v[sym_line<DIM>(i, m)].y * xi[m];
    }
    ar[i] = a1;
    ai[i] = a2;
    sr_ += xi[i] * a1;
    si_ += xi[i] * a2;
  }
#pragma unroll
  for (int j = 0; j < DIM; ++j)
#pragma unroll
    for (int i = 0; i <= j; ++i) {
      c_t<T> g;
      g.x = norm * (xi[i] * ar[j] + xi[j] * ar[i] - xi[i] * xi[j] * sr_);
      g.y = norm * (xi[i] * ai[j] + xi[j] * ai[i] - xi[i] * xi[j] * si_);
      f[sym_line<DIM>(i, j)] = g;
    }
}

// unit wave vector of Fourier point c (first DIM coordinates) of the grid
// res with lengths L; false for k = 0 and, under the even-grid policy, for a
// Nyquist index on an even axis (the operator is zero there).  |xi|^2 is
// summed without contraction into fused multiply-adds: left to the compiler,
// whether it contracts depends on the kernel the function is inlined into,
// and the serving and single-cell first-axis kernels then differ in the last
// bit of xi wherever 1/L is inexact (lengths like 7 or 5)
template <typename T, int DIM>
__device__ __forceinline__ bool unit_wave_vector(const int* c, const int* res, const double* L,
                                                 int allow_even, T* xi) {
#pragma clang fp contract(off)
  T n2 = 0;
  bool zero = true, nyq = false;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    xi[d] = fft_freq<T>(c[d], res[d], L[d]);
    n2 += xi[d] * xi[d];
    if (c[d] != 0) zero = false;
    if (allow_even && (res[d] % 2 == 0) && 2 * c[d] == res[d]) nyq = true;
  }
  if (zero || nyq) return false;
  const T inv = T(1) / sqrt(n2);
#pragma unroll
  for (int d = 0; d < DIM; ++d) xi[d] *= inv;
  return true;
}

// deterministic sum over the NT threads of a block (any NT <= 1024); red
// holds NT doubles; every thread must call it
template <int NT>
__device__ double block_sum_any(double v, double* red) {
  constexpr int P2 = NT <= 64 ? 64 : NT <= 128 ? 128 : NT <= 256 ? 256 : NT <= 512 ? 512 : 1024;
  red[threadIdx.x] = v;
  __syncthreads();
#pragma unroll
  for (int s = P2 / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s && threadIdx.x + s < NT) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  return red[0];
}

// the same for a workgroup of NT threads (any NT <= 1024) by lane halving in
// each wavefront, then over the wavefronts, in a fixed order; red holds 16
// doubles; the result is valid in thread 0.  Every thread must call it.
__device__ __forceinline__ double block_sum_waves(double v, double* red, int NT) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lanes = NT - 64 * wave < 64 ? NT - 64 * wave : 64;
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const double o = __shfl_down(v, s, 64);
    if (lane + s < lanes) v += o;
  }
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < (NT + 63) / 64; ++w) t += red[w];
  return t;
}

// sum of up to kFoldMax partials by the first wavefront, in an order that does
// not depend on the workgroup: lane l adds l, l + 64, ..., then lane halving;
// the result is in every thread.  Every thread must call it (a barrier inside);
// red holds one double
__device__ __forceinline__ double fold_sum(const double* __restrict__ part, int count, double* red) {
  if (threadIdx.x < 64) {
    double v = 0.0;
    for (int i0 = 0; i0 < count; i0 += 64 * 4) {
      double t[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = i0 + 64 * k + (int)threadIdx.x;
        t[k] = part[i < count ? i : count - 1];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i0 + 64 * k + (int)threadIdx.x < count) v += t[k];
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v += __shfl_down(v, s, 64);
    if (threadIdx.x == 0) red[0] = v;
  }
  __syncthreads();
  return red[0];
}

// ---- packed symmetric CG vectors ----------------------------------------------------
// In a packed run p and r of a chunk of iterations hold the dim (dim + 1) / 2
// components too (48 instead of 72 B per voxel in 3D, five sweeps per iteration);
// the chunk's first iteration reads them from the full fields (the mean of two
// mirrored components) and its last one writes r back to them.  Per launch at
// 128^3, with x no longer in the r2c pass: r2c 168 -> 94 us, c2r 76 -> 69; at
// 125^3 128 -> 96 and 102 -> 78.

// of `tot` packed values from `base` on, those that lie before `lim`; <= 0 where
// the rows are all beyond the last one (the later row pairs of a last workgroup)
__host__ __device__ __forceinline__ int sym_left(int64_t base, int64_t lim, int tot) {
  return lim - base < tot ? (int)(lim - base) : tot;
}
// the two entries of a field of dim^2 components that hold packed value base + e
// (base: a multiple of dim (dim + 1) / 2)
template <int DIM>
__host__ __device__ __forceinline__ void sym_entries(int64_t base, int e, int64_t& a, int64_t& b) {
  constexpr int NC = DIM * DIM, NL = sym_lines(DIM);
  const int m = e / NL;
  int ca, cb;
  sym_pair<DIM>(e - m * NL, ca, cb);
  const int64_t g = (base / NL + m) * NC;
  a = g + ca;
  b = g + cb;
}

// p (packed) of `tot` values from `base` on, at most KB per thread in flight,
// stored and staged in sp; with SYM_UPDATE p = -r + beta p.  Values at and beyond
// `lim` are staged as zeros; nothing is read there.
template <typename T, int DIM, int KB>
__device__ __forceinline__ void sym_stage(const T* in, const T* rvec, T* pout, int flags, T beta,
                                          int64_t base, int64_t lim, int tot, int NT, T* sp) {
  const bool upd = flags & SYM_UPDATE, full = flags & SYM_SRC_FULL;
  const int last = sym_left(base, lim, tot) - 1;
  if (last < 0) {
    for (int e = threadIdx.x; e < tot; e += NT) sp[e] = T(0);
    return;
  }
  for (int e0 = 0; e0 < tot; e0 += KB * NT) {
    T pv[KB], rv[KB];
    if (full) {
      T pw[KB], rw[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        int e = e0 + i * NT + (int)threadIdx.x;
        if (e > last) e = last;
        int64_t a, b;
        sym_entries<DIM>(base, e, a, b);
        pv[i] = in[a];
        pw[i] = in[b];
        rv[i] = rvec[a];
        rw[i] = rvec[b];
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        pv[i] = T(0.5) * (pv[i] + pw[i]);
        rv[i] = T(0.5) * (rv[i] + rw[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        int e = e0 + i * NT + (int)threadIdx.x;
        if (e > last) e = last;
        pv[i] = in[base + e];
        rv[i] = rvec[base + e];
      }
    }
#pragma unroll
    for (int i = 0; i < KB; ++i) {
      const int e = e0 + i * NT + (int)threadIdx.x;
      if (e < tot) {
        T x = T(0);
        if (e <= last) {
          x = upd ? -rv[i] + beta * pv[i] : pv[i];
          pout[base + e] = x;
        }
        sp[e] = x;
      }
    }
  }
}

// r += alpha A p over `tot` packed values from `base` on (A p of value e from
// get(voxel, line)); returns this thread's part of r . r over all dim^2
// components
template <typename T, int DIM, int KB, typename G>
__device__ __forceinline__ double sym_rupd(const T* rin, T* out, T* ap, int flags, T al, int64_t base,
                                           int tot, int NT, const G& get) {
  constexpr int NC = DIM * DIM, NL = sym_lines(DIM);
  const bool sfull = flags & SYM_SRC_FULL, ofull = flags & SYM_OUT_FULL;
  const int64_t vox0 = base / NL;
  double acc = 0.0;
  for (int e0 = 0; e0 < tot; e0 += KB * NT) {
    T dv[KB];
    if (sfull) {
      T dw[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        int e = e0 + i * NT + (int)threadIdx.x;
        if (e >= tot) e = tot - 1;
        const int m = e / NL;
        int ca, cb;
        sym_pair<DIM>(e - m * NL, ca, cb);
        const int64_t g = (vox0 + m) * NC;
        dv[i] = rin[g + ca];
        dw[i] = rin[g + cb];
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) dv[i] = T(0.5) * (dv[i] + dw[i]);
    } else {
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int e = e0 + i * NT + (int)threadIdx.x;
        dv[i] = rin[base + (e < tot ? e : tot - 1)];
      }
    }
#pragma unroll
    for (int i = 0; i < KB; ++i) {
      const int e = e0 + i * NT + (int)threadIdx.x;
      if (e < tot) {
        const int m = e / NL, c = e - m * NL;
        const T val = get(m, c);
        const T rv = dv[i] + al * val;
        int ca, cb;
        sym_pair<DIM>(c, ca, cb);
        const int64_t g = (vox0 + m) * NC;
        if (ofull) {
          out[g + ca] = rv;
          out[g + cb] = rv;
        } else {
          out[base + e] = rv;
        }
        if (ap) {
          ap[g + ca] = val;
          ap[g + cb] = val;
        }
        acc += (c < DIM ? 1.0 : 2.0) * ((double)rv * (double)rv);
      }
    }
  }
  return acc;
}

// r2c: beta and SolverCG's loop test after the previous iteration, from the sum s
// of its r . r partials; false: the loop has stopped (workgroup 0 says so to the
// later kernels)
__device__ __forceinline__ bool fold_beta_test(const ScalarFold& f, double s, double& beta) {
  const double old = f.scal[(f.iter - 1) & 1 ? SC_RDR1 : SC_RDR];
  const bool go = s > f.scal[SC_TOL2];  // (false for NaN)
  beta = s / old;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    f.scal[f.iter & 1 ? SC_RDR1 : SC_RDR] = s;
    f.scal[SC_NEWRDR] = s;
    f.scal[SC_BETA] = beta;
    // an iteration whose r . r is NaN is not counted here (the host does)
    if (s == s) f.ctl[CTL_ITER] = f.iter;
    if (!go) f.ctl[CTL_ACTIVE] = 0;
  }
  return go;
}
// The whole of it: whether the iteration runs, with its beta.  Workgroup 0 of this
// very launch clears the flag, so the wavefronts of another workgroup may read
// different values of it: none returns before all have summed the partials,
// and where the flag was cleared by this launch the test fails for everyone.
// Every thread must call it (barriers inside); red holds one double and is free
// again on return
__device__ __forceinline__ bool fold_goes_on(const ScalarFold& f, const int* active, double* red,
                                             double& beta) {
  const int on = active ? active[0] : 1;
  const double s = fold_sum(f.rr, f.nrr, red);
  if (!on || !fold_beta_test(f, s, beta)) return false;
  __syncthreads();
  return true;
}
// c2r: alpha from the sum s of the p . K p partials
__device__ __forceinline__ double fold_alpha(const ScalarFold& f, double s) {
  const double al = f.scal[f.iter & 1 ? SC_RDR1 : SC_RDR] / s;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    f.scal[SC_PAP] = s;
    f.scal[SC_ALPHA] = al;
    if (f.aring) f.aring[f.iter & (kRing - 1)] = al;
  }
  return al;
}

}  // namespace mugpu
