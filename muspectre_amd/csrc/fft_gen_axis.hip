// Strided passes along an axis of run-time length: c2c along
// the middle axis (or the first one, for the engine's transforms), and the
// first axis with the projection between its two transforms.  The plans'
// shapes are made here too.
#include "fft_gen.hpp"

namespace mugpu {

namespace {

// ---- plan: radices, threads per line, workgroup shapes ---------------------------
// threads per line without which a thread would hold too much, and the most
// that a pass can use
int min_threads(const GenAxis& ax) {
  int P = 1;
  for (int i = 0; i < ax.np; ++i) {
    const int R = ax.ps[i].R, nb = ax.ps[i].nb;
    const bool prime = !gen_compiled(R);
    const int need = prime ? (nb * (((R - 1) / 2 + kGenQ) / kGenQ) + kGenTB - 1) / kGenTB
                           : (nb + gen_held(R) - 1) / gen_held(R);
    if (need > P) P = need;
  }
  const int hold = (ax.n + kGenVals - 1) / kGenVals;
  return P > hold ? P : hold;
}
int max_threads(const GenAxis& ax) {
  int P = 1;
  for (int i = 0; i < ax.np; ++i) {
    const int R = ax.ps[i].R, nb = ax.ps[i].nb;
    const int use = gen_compiled(R) ? nb : nb * (((R - 1) / 2 + kGenQ) / kGenQ);
    if (use > P) P = use;
  }
  return P;
}

// threads per line for L lines: as near kGenThreads threads as the passes allow
bool threads_for(const GenAxis& ax, int L, GenShape& g) {
  const int lo = min_threads(ax), hi = max_threads(ax);
  int P = kGenThreads / L;
  if (P > hi) P = hi;
  if (P < lo) P = lo;
  if (L * P > kGenMaxNT) return false;
  g.L = L;
  g.P = P;
  g.NT = (L * P + 63) / 64 * 64;
  return g.NT <= kGenMaxNT;
}

}  // namespace

bool gen_radices(int n, GenAxis& ax) {
  ax = GenAxis{};
  if (n < 2) return false;
  ax.n = n;
  int f[kGenMaxPass * 2], nf = 0, m = n;
  for (int r : {17, 13, 11, 9, 8, 7, 5, 4, 3, 2})
    while (m % r == 0 && nf < kGenMaxPass * 2) {
      f[nf++] = r;
      m /= r;
    }
  // the primes without a compiled butterfly go first (no twiddles there)
  int q[kGenMaxPass * 2], nq = 0;
  for (int r = 19; m > 1 && nq < kGenMaxPass; r += 2)
    while (m % r == 0) {
      q[nq++] = r;
      m /= r;
    }
  for (int i = 0; i < nf; ++i) q[nq++] = f[i];
  if (m != 1 || nq > kGenMaxPass) return false;
  int NS = 1;
  ax.np = nq;
  for (int i = 0; i < nq; ++i) {
    GenPass& ps = ax.ps[i];
    ps.R = q[i];
    ps.NS = NS;
    ps.nb = n / q[i];
    ps.step = n / (NS * q[i]);
    ps.magic = NS > 1 ? (unsigned)(((uint64_t)1 << 32) / (uint64_t)NS + 1) : 0u;
    if (q[i] > 9) ax.cls = 1;
    NS *= q[i];
  }
  return true;
}

GenShape gen_last_shape(const GenAxis& ax, int nc, int nl, int64_t rows) {
  // pairs of rows per workgroup: more while the grid keeps 1024 workgroups
  // and the LDS leaves room for four of them per CU.  The staging area counted is
  // that of full fields; packed CG vectors stage two thirds of it (2D: three
  // quarters) and are launched with as much less LDS, but in the same shape
  GenShape best{};
  const int n = ax.n;
  for (int mult = 1; mult <= 8; ++mult) {
    GenShape g{};
    const int L = mult * nl;
    if (!threads_for(ax, L, g)) break;
    const size_t lines = (size_t)n * (L | 1) * 16, tw = (size_t)n * 16;
    const size_t fwd = lines + tw + (size_t)2 * n * nc * 8;
    const size_t half = (size_t)2 * mult * (n / 2 + 1) * nl * 16;
    const size_t bwd = (lines > half ? lines : half) + tw;
    g.mult = mult;
    // threads beyond the transforms' share the sweeps over the staged rows
    // (four values each): up to 256 where the grid leaves the chip idle anyway
    // (33x27x35: r2c 22.6 -> 16.0, c2r 10.6 -> 8.9 us), else only in the r2c
    // pass, which stages most, and at most twice as many (125^3: 144 -> 128 us;
    // four times as many cost 22.5 -> 26.0 us at 63^3)
    const bool idle = rows / (2 * mult) < 1024;
    int sweep = (2 * n * nc / 4 + 63) / 64 * 64;
    if (sweep > kGenThreads) sweep = kGenThreads;
    g.NT_bwd = idle && sweep > g.NT ? sweep : g.NT;
    if (!idle && sweep > 2 * g.NT) sweep = 2 * g.NT;
    if (sweep > g.NT) g.NT = sweep;
    g.lds = fwd;
    g.lds_bwd = bwd;
    if (fwd > kGenMaxLds || bwd > kGenMaxLds) break;
    if (mult > 1 && (g.lds > kGenLds || L > 40 || rows / (2 * mult) < 1024)) break;
    best = g;
  }
  return best;
}

GenShape gen_axis0_shape(const GenAxis& ax, int nl, int64_t plane) {
  GenShape best{};
  for (int mult = 1; mult <= 4; mult *= 2) {
    GenShape g{};
    const int L = mult * nl;
    if (!threads_for(ax, L, g)) break;
    g.mult = mult;
    g.lds = (size_t)ax.n * ((L | 1) + 1) * 16;
    if (g.lds > kGenMaxLds) break;
    if (mult > 1 && (g.lds > kGenLds || L > 40 || plane / mult < 1024)) break;
    best = g;
  }
  return best;
}

GenShape gen_strided_shape(const GenAxis& ax, int64_t inner, int64_t outer) {
  GenShape best{};
  for (int L = 4; L <= 16; L *= 2) {
    GenShape g{};
    if (!threads_for(ax, L, g)) break;
    g.mult = 1;
    g.lds = (size_t)ax.n * ((L | 1) + 1) * 16;
    if (g.lds > kGenMaxLds) break;
    if (L > 4 && (g.lds > 2 * kGenLds || (inner + L - 1) / L * outer < 512)) break;
    best = g;
  }
  return best;
}

namespace {

template <typename T>
struct GStr {
  c_t<T>* data;
  int64_t inner;
  int L, P, LS;
  GenAxis ax;
  const c_t<T>* tw;
  const int* active;  // FftPlan::active
};

// data[(o * n + m) * inner + w]: the workgroup transforms L consecutive lines w
// of plane o; HBM is read by the first pass and written by the last
template <typename T, int CLS, int SG>
__global__ __launch_bounds__(kGenMaxNT) void k_gen_strided(GStr<T> a) {
  if (a.active && !a.active[0]) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int n = a.ax.n, LS = a.LS;
  c_t<T>* s = reinterpret_cast<c_t<T>*>(smem);
  c_t<T>* tw = s + n * LS;
  gen_twiddles<T>(tw, a.tw, n);
  const int p = threadIdx.x / a.L, l = threadIdx.x - p * a.L;
  const int64_t gx = gridDim.x;
  const int64_t t = xcd_tile(blockIdx.y * gx + blockIdx.x, gx * gridDim.y);
  const int64_t o = t / gx;
  const int64_t w = (t - o * gx) * a.L + l;
  const bool act = p < a.P && w < a.inner;
  c_t<T>* base = a.data + o * n * a.inner + (w < a.inner ? w : a.inner - 1);
  const int64_t inner = a.inner;
  gen_fft<T, CLS, SG, true, true>(
      a.ax, a.P, p, act, s + l, LS, tw, [&](int m) { return base[m * inner]; },
      [&](int m, c_t<T> x) { base[m * inner] = x; });
}

template <typename T>
struct GAxis0 {
  c_t<T>* data;
  int64_t plane;  // k-points per first-axis index
  int KP, L, P, LS;
  GenAxis ax;
  const c_t<T>* tw;
  int kind, allow_even, res[3], hlast;
  double Lc[3];
  T norm;
  const int* active;  // FftPlan::active
};

template <typename T, int CLS, int DIM, bool PK>
__global__ __launch_bounds__(kGenMaxNT) void k_gen_axis0(GAxis0<T> a) {
  if (a.active && !a.active[0]) return;
  constexpr int NC = nb_lines(DIM, PK);
  extern __shared__ __align__(16) unsigned char smem[];
  const int n = a.ax.n, LS = a.LS, KP = a.KP;
  c_t<T>* s = reinterpret_cast<c_t<T>*>(smem);
  c_t<T>* tw = s + n * LS;
  gen_twiddles<T>(tw, a.tw, n);
  const int p = threadIdx.x / a.L, l = threadIdx.x - p * a.L;
  const int64_t q0 = xcd_tile(blockIdx.x, gridDim.x) * KP;
  const int64_t inner = a.plane * NC;
  const int64_t w = q0 * NC + l;
  const bool act = p < a.P, valid = w < inner;
  c_t<T>* base = a.data + (valid ? w : inner - 1);
  auto ld = [&](int m) { return base[m * inner]; };
  auto st = [&](int m, c_t<T> x) {
    if (valid) base[m * inner] = x;
  };
  gen_fft<T, CLS, -1, true, false>(a.ax, a.P, p, act, s + l, LS, tw, ld, st);
  // projection per wave vector (k0, q0 + kp); KP is 1, 2 or 4 and divides the
  // thread count, so a thread keeps one kp
  const int sh = KP >> 1;  // log2 of KP
  const int kp = threadIdx.x & (KP - 1);
  const int64_t q = q0 + kp;
  int c[3] = {0, 0, 0};
  if (DIM == 3) {
    c[1] = (int)q / a.hlast;
    c[2] = (int)q - c[1] * a.hlast;
  } else {
    c[1] = (int)q;
  }
  for (int k0 = threadIdx.x >> sh; k0 < n && q < a.plane; k0 += blockDim.x >> sh) {
    c[0] = k0;
    T xi[DIM];
    c_t<T>* f = s + k0 * LS + kp * NC;
    if (!unit_wave_vector<T, DIM>(c, a.res, a.Lc, a.allow_even, xi)) {
#pragma unroll
      for (int r = 0; r < NC; ++r) f[r] = c_t<T>{};
      continue;
    }
    if constexpr (PK) project_point_sym<T, DIM>(f, xi, a.norm);
    else project_point<T, DIM>(f, 1, xi, a.kind, a.norm);
  }
  __syncthreads();
  gen_fft<T, CLS, +1, false, true>(a.ax, a.P, p, act, s + l, LS, tw, ld, st);
}

template <typename T>
int strided_t(FftPlan& p, int ax, void* spec, int sign) {
  GStr<T> a{};
  a.data = static_cast<c_t<T>*>(spec);
  a.inner = p.lines();
  for (int d = ax + 1; d < p.dim; ++d) a.inner *= p.hres[d];
  int64_t outer = 1;
  for (int d = 0; d < ax; ++d) outer *= p.hres[d];
  const GenShape& g = p.gen_str[ax][p.packed ? 1 : 0];
  a.L = g.L;
  a.P = g.P;
  a.LS = g.L | 1;
  a.ax = p.gen[ax];
  a.tw = static_cast<const c_t<T>*>(sizeof(T) == 8 ? p.tw64[ax] : p.tw32[ax]);
  a.active = p.active;
  const dim3 grid((unsigned)((a.inner + a.L - 1) / a.L), (unsigned)outer), block((unsigned)g.NT);
  if (a.ax.cls == 0) {
    if (sign < 0) hipLaunchKernelGGL((k_gen_strided<T, 0, -1>), grid, block, g.lds, stream(), a);
    else hipLaunchKernelGGL((k_gen_strided<T, 0, +1>), grid, block, g.lds, stream(), a);
  } else {
    if (sign < 0) hipLaunchKernelGGL((k_gen_strided<T, 1, -1>), grid, block, g.lds, stream(), a);
    else hipLaunchKernelGGL((k_gen_strided<T, 1, +1>), grid, block, g.lds, stream(), a);
  }
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

template <typename T, int DIM, bool PK>
int axis0_t(FftPlan& p, const ProjParams& pj, void* spec) {
  GAxis0<T> a{};
  a.data = static_cast<c_t<T>*>(spec);
  a.plane = p.kpts / p.res[0];
  const GenShape& g = p.gen_axis0[PK ? 1 : 0];
  a.KP = g.mult;
  a.L = g.L;
  a.P = g.P;
  a.LS = g.L | 1;
  a.ax = p.gen[0];
  a.tw = static_cast<const c_t<T>*>(sizeof(T) == 8 ? p.tw64[0] : p.tw32[0]);
  a.kind = pj.kind;
  a.allow_even = pj.allow_even;
  for (int d = 0; d < 3; ++d) {
    a.res[d] = p.res[d];
    a.Lc[d] = pj.L[d];
  }
  a.hlast = p.hres[p.dim - 1];
  a.norm = (T)pj.norm;
  a.active = p.active;
  const dim3 grid((unsigned)((a.plane + a.KP - 1) / a.KP)), block((unsigned)g.NT);
  if (a.ax.cls == 0) hipLaunchKernelGGL((k_gen_axis0<T, 0, DIM, PK>), grid, block, g.lds, stream(), a);
  else hipLaunchKernelGGL((k_gen_axis0<T, 1, DIM, PK>), grid, block, g.lds, stream(), a);
  MUGPU_HIP(hipGetLastError());
  return MUGPU_OK;
}

}  // namespace

int gen_strided(FftPlan& p, int prec, int ax, void* spec, int sign) {
  return prec == MUGPU_FP64 ? strided_t<double>(p, ax, spec, sign) : strided_t<float>(p, ax, spec, sign);
}

int gen_axis0_project(FftPlan& p, int prec, const ProjParams& pj, void* spec) {
  if (prec != MUGPU_FP64)
    return p.dim == 3 ? axis0_t<float, 3, false>(p, pj, spec) : axis0_t<float, 2, false>(p, pj, spec);
  if (p.packed) return p.dim == 3 ? axis0_t<double, 3, true>(p, pj, spec) : axis0_t<double, 2, true>(p, pj, spec);
  return p.dim == 3 ? axis0_t<double, 3, false>(p, pj, spec) : axis0_t<double, 2, false>(p, pj, spec);
}

}  // namespace mugpu
