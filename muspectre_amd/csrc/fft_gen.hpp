// Passes for axis lengths known at run time (any length without a
// compile-time instantiation; the odd lengths that the reference's
// projections ask for are all of this kind): building blocks of the kernels in
// fft_gen_last.hip and fft_gen_axis.hip.
//
// Layout as in fft_fast.hpp: a workgroup owns L lines, thread (l, p) works on
// line l, consecutive lanes on consecutive lines, so that LDS and strided HBM
// accesses are unit stride across lanes and every index computation of a
// butterfly (j, j mod NS, the twiddle exponent) is shared by all lanes of a
// line group.  What is known only at run time is the length, the number P of
// threads per line and the sequence of radices; each radix is compiled:
// 2, 3, 4, 5, 7, 8, 9 (class 0) and 11, 13, 17 (class 1, which costs registers
// and is a kernel of its own), and a pass for any other prime.  A thread holds
// the inputs of up to gen_held(R) butterflies in registers between the reads
// and the writes of a pass, so one LDS buffer serves.  No integer division by
// a run-time value is left inside a pass of a compiled radix: j / NS is a
// multiplication by a reciprocal made with the plan.  The pass for other primes
// divides once per task, which forms (R - 1) / 2 products for each output pair.
//
// Bound by HBM from about 64^3 on, by latency below.  Measured per launch on a
// 125^3 small-strain CG iteration, against the passes of fft_passes.hip that
// served every such length before (element-wise integer divisions, radices 7
// and above as direct sums with table loads from memory): r2c 125 us (301),
// middle axis 57 (266), first axis with the projection 74 (384), c2r with the
// dot product 115 (403); on 51^2, where no workgroup count fills the chip,
// 7.1 (8.4), -, 8.3 (14.3) and 7.1 us (9.1).
#pragma once
#include <type_traits>

#include "mugpu_internal.hpp"
#include "op_stages.hpp"

namespace mugpu {

namespace {

// ---- butterflies of the odd radices ------------------------------------------
// With a_t = x_t + x_{R-t}, b_t = x_t - x_{R-t}, t = 1..h, h = (R-1)/2:
//   X_q, X_{R-q} = x_0 + sum_t a_t cos(2 pi t q / R) -+ i sum_t b_t sin(2 pi t q / R)
// (signs of the forward transform), half the multiplications of the direct
// sum, all by real constants
template <int R>
struct OddRoots;
template <>
struct OddRoots<5> {
    static constexpr double c[2] = {0.309016994374947424102293417182819059,
      -0.809016994374947424102293417182819059};
    static constexpr double s[2] = {0.951056516295153572116439333379382143,
      0.587785252292473129168705954639072769};
};
template <>
struct OddRoots<7> {
    static constexpr double c[3] = {0.623489801858733530525004884004239811,
      -0.222520933956314404288902564496794759, -0.900968867902419126236102319507445051};
    static constexpr double s[3] = {0.78183148246802980870844452667405775,
      0.974927912181823607018131682993931217, 0.433883739117558120475768332848358755};
};
template <>
struct OddRoots<11> {
    static constexpr double c[5] = {0.841253532831181168861811648919367718,
      0.415415013001886425529274149229623204, -0.142314838273285140443792668616369669,
      -0.654860733945285064056925072466293553, -0.959492973614497389890368057066327699};
    static constexpr double s[5] = {0.540640817455597582107635954318691695,
      0.90963199535451837141171538307902846, 0.989821441880932732376092037776718787,
      0.75574957435425828377403584397234442, 0.281732556841429697711417915346616899};
};
template <>
struct OddRoots<13> {
    static constexpr double c[6] = {0.885456025653209895900375522015098879,
      0.568064746731155802511807559127516625, 0.120536680255323053349067687452543582,
      -0.354604887042535625969637892600018474, -0.748510748171101098634630599701351384,
      -0.970941817426052027156982276293789227};
    static constexpr double s[6] = {0.464723172043768545656015335133104778,
      0.822983865893656394579617423439381991, 0.992708874098053992800751649492520179,
      0.935016242685414823439784599837830729, 0.66312265824079520237678549266676628,
      0.239315664287557767148753726260211895};
};
template <>
struct OddRoots<17> {
    static constexpr double c[8] = {0.932472229404355804573115891821563386,
      0.739008917220659115924534309872648106, 0.445738355776538267396457549379486855,
      0.0922683594633019952396511071545064804, -0.273662990072082863539077935436813432,
      -0.602634636379256389178588154986840622, -0.850217135729614152134143922949352058,
      -0.982973099683901778281948844855198716};
    static constexpr double s[8] = {0.361241666187152948744714596183700164,
      0.673695643646557211712691912425694616, 0.895163291355062322067016499753785457,
      0.995734176295034521871191178905481784, 0.96182564317281907040879629073151855,
      0.798017227280239503332805112796261369, 0.526432162877355800244607799140699566,
      0.183749517816570331574408839620727582};
};
template <typename T, int R, int SG>
__device__ __forceinline__ void odd_bfly(c_t<T>* v) {
  constexpr int h = (R - 1) / 2;
#pragma unroll
  for (int t = 1; t <= h; ++t) {
    const c_t<T> x = v[t], y = v[R - t];
    v[t] = cadd(x, y);
    v[R - t] = csub(x, y);
  }
  c_t<T> u[R];
  u[0] = v[0];
#pragma unroll
  for (int t = 1; t <= h; ++t) u[0] = cadd(u[0], v[t]);
#pragma unroll
  for (int q = 1; q <= h; ++q) {
    c_t<T> C = v[0], S;
    S.x = S.y = T(0);
#pragma unroll
    for (int t = 1; t <= h; ++t) {
      const int m = t * q % R;
      const T c = T(OddRoots<R>::c[(m <= h ? m : R - m) - 1]);
      const T s = m <= h ? T(OddRoots<R>::s[m - 1]) : -T(OddRoots<R>::s[R - m - 1]);
      C.x += c * v[t].x;
      C.y += c * v[t].y;
      S.x += s * v[R - t].x;
      S.y += s * v[R - t].y;
    }
    // X_q = C - i S forward, C + i S backward
    c_t<T> a, b;
    a.x = C.x + S.y;
    a.y = C.y - S.x;
    b.x = C.x - S.y;
    b.y = C.y + S.x;
    u[q] = SG < 0 ? a : b;
    u[R - q] = SG < 0 ? b : a;
  }
#pragma unroll
  for (int q = 0; q < R; ++q) v[q] = u[q];
}

// radix 9 as 3 x 3: n = 3 n1 + n2, k = k1 + 3 k2
template <typename T, int SG>
__device__ __forceinline__ void bfly9(c_t<T>* v) {
  // cos and sin of 2 pi m / 9 for m = 1, 2, 4
  const T wc[3] = {T(0.766044443118978035202392650555416674), T(0.173648177666930348851716626769314796),
                   T(-0.93969262078590838405410927732473147)};
  const T ws[3] = {T(0.642787609686539326322643409907263433), T(0.984807753012208059366743024589523014),
                   T(0.342020143325668733044099614682259581)};
  c_t<T> a[3][3];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
    c_t<T> x[3] = {v[n2], v[3 + n2], v[6 + n2]};
    Butterfly<T, 3>::run(x, SG, nullptr, 0);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      const int m = n2 * k1;  // 0, 1, 2 or 4
      if (m == 0) {
        a[n2][k1] = x[k1];
      } else {
        const int i = m == 4 ? 2 : m - 1;
        c_t<T> w;
        w.x = wc[i];
        w.y = SG < 0 ? -ws[i] : ws[i];
        a[n2][k1] = cmul(x[k1], w);
      }
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    c_t<T> y[3] = {a[0][k1], a[1][k1], a[2][k1]};
    Butterfly<T, 3>::run(y, SG, nullptr, 0);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = y[k2];
  }
}

template <typename T, int R, int SG>
__device__ __forceinline__ void gen_bfly(c_t<T>* v) {
  if constexpr (R == 9) bfly9<T, SG>(v);
  else if constexpr (R == 2 || R == 3 || R == 4 || R == 8) Butterfly<T, R>::run(v, SG, nullptr, 0);
  else odd_bfly<T, R, SG>(v);
}

// ---- passes ---------------------------------------------------------------------
// One Stockham pass of radix R on the line whose element m is col[m * LS], by
// the P threads p of the line (`act` is false for the surplus threads of the
// workgroup, which only keep the barriers).  `first`: the inputs come from
// ld(m) instead; `last`: the outputs go to st(m, value).  Inputs are read from
// clamped butterfly indices, so that all loads of a thread go out together.
template <typename T, int R, int SG, bool GIN, bool GOUT, class Ld, class St>
__device__ __forceinline__ void gen_pass(const GenPass& ps, int P, int p, bool act, bool first, bool last,
                                         c_t<T>* col, int LS, const c_t<T>* tw, Ld ld, St st) {
  constexpr int B = gen_held(R);
  c_t<T> v[B][R];
  const int nb = ps.nb;
  if (GIN && first) {
#pragma unroll
    for (int b = 0; b < B; ++b)
      if (b * P < nb) {
        const int j = p + b * P < nb ? p + b * P : nb - 1;
#pragma unroll
        for (int t = 0; t < R; ++t) v[b][t] = ld(j + t * nb);
      }
  } else {
#pragma unroll
    for (int b = 0; b < B; ++b)
      if (b * P < nb) {
        const int j = p + b * P < nb ? p + b * P : nb - 1;
#pragma unroll
        for (int t = 0; t < R; ++t) v[b][t] = col[(j + t * nb) * LS];
      }
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < B; ++b)
    if (b * P < nb) {
      const int j = p + b * P < nb ? p + b * P : nb - 1;
      int q = j, k = 0;
      if (ps.NS > 1) {
        q = (int)__umulhi((unsigned)j, ps.magic);
        k = j - q * ps.NS;
        const int e = k * ps.step;
#pragma unroll
        for (int t = 1; t < R; ++t) {
          c_t<T> w = tw[t * e];
          if (SG > 0) w.y = -w.y;
          v[b][t] = cmul(v[b][t], w);
        }
      }
      gen_bfly<T, R, SG>(v[b]);
      const int o = q * ps.NS * R + k;
      if (act && p + b * P < nb) {
        if (GOUT && last) {
#pragma unroll
          for (int t = 0; t < R; ++t) st(o + t * ps.NS, v[b][t]);
        } else {
#pragma unroll
          for (int t = 0; t < R; ++t) col[(o + t * ps.NS) * LS] = v[b][t];
        }
      }
    }
  if (!(GOUT && last)) __syncthreads();
}

// The pass of any other prime R: the twiddled inputs are replaced in place by
// x_0, a_t (at t) and b_t (at R - t), then a task forms kGenQ output pairs
// (q, R - q) at once, so that an a_t, b_t read from LDS serves kGenQ pairs; a
// thread holds the outputs of up to kGenTB tasks until every input has been
// read.  The roots come from the twiddle table in LDS (one exponent per lane
// group: broadcasts).
template <typename T, int SG, bool GIN, bool GOUT, class Ld, class St>
__device__ __forceinline__ void gen_prime(const GenPass& ps, int P, int p, bool act, bool first, bool last,
                                          c_t<T>* col, int LS, const c_t<T>* tw, Ld ld, St st) {
  const int nb = ps.nb, R = ps.R, NS = ps.NS, h = (R - 1) / 2;
  if (act) {
    for (int it = p; it < nb * (h + 1); it += P) {
      const int t = it / nb, j = it - t * nb;
      const int k = NS > 1 ? j - (int)__umulhi((unsigned)j, ps.magic) * NS : 0;
      c_t<T> x = GIN && first ? ld(j + t * nb) : col[(j + t * nb) * LS];
      if (t == 0) {
        if (GIN && first) col[j * LS] = x;
        continue;
      }
      c_t<T> y = GIN && first ? ld(j + (R - t) * nb) : col[(j + (R - t) * nb) * LS];
      if (NS > 1) {
        c_t<T> w = tw[t * k * ps.step], z = tw[(R - t) * k * ps.step];
        if (SG > 0) {
          w.y = -w.y;
          z.y = -z.y;
        }
        x = cmul(x, w);
        y = cmul(y, z);
      }
      col[(j + t * nb) * LS] = cadd(x, y);
      col[(j + (R - t) * nb) * LS] = csub(x, y);
    }
  }
  __syncthreads();
  const int tasks = nb * ((h + kGenQ) / kGenQ);
  c_t<T> C[kGenTB][kGenQ], S[kGenTB][kGenQ];
#pragma unroll
  for (int b = 0; b < kGenTB; ++b)
    if (b * P < tasks) {
      const int it = p + b * P < tasks ? p + b * P : tasks - 1;
      const int u = it / nb, j = it - u * nb;
      int q[kGenQ], m[kGenQ];
      const c_t<T> x0 = col[j * LS];
#pragma unroll
      for (int i = 0; i < kGenQ; ++i) {
        q[i] = u * kGenQ + i < h ? u * kGenQ + i : h;
        m[i] = 0;
        C[b][i] = x0;
        S[b][i].x = S[b][i].y = T(0);
      }
      for (int t = 1; t <= h; ++t) {
        const c_t<T> a = col[(j + t * nb) * LS], d = col[(j + (R - t) * nb) * LS];
#pragma unroll
        for (int i = 0; i < kGenQ; ++i) {
          m[i] += q[i];
          if (m[i] >= R) m[i] -= R;
          const c_t<T> w = tw[m[i] * nb];  // cos, -sin
          C[b][i].x += w.x * a.x;
          C[b][i].y += w.x * a.y;
          S[b][i].x += w.y * d.x;
          S[b][i].y += w.y * d.y;
        }
      }
    }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int b = 0; b < kGenTB; ++b)
      if (p + b * P < tasks) {
        const int it = p + b * P;
        const int u = it / nb, j = it - u * nb;
        const int g = NS > 1 ? (int)__umulhi((unsigned)j, ps.magic) : j;
        const int o = g * NS * R + (j - g * NS);
#pragma unroll
        for (int i = 0; i < kGenQ; ++i) {
          const int q = u * kGenQ + i;
          if (q <= h) {
            // S holds -sum b_t sin: X_q = C + i S forward, C - i S backward
            c_t<T> x, y;
            x.x = C[b][i].x - S[b][i].y;
            x.y = C[b][i].y + S[b][i].x;
            y.x = C[b][i].x + S[b][i].y;
            y.y = C[b][i].y - S[b][i].x;
            const c_t<T> lo = SG < 0 ? x : y, hi = SG < 0 ? y : x;
            if (GOUT && last) {
              st(o + q * NS, lo);
              if (q > 0) st(o + (R - q) * NS, hi);
            } else {
              col[(o + q * NS) * LS] = lo;
              if (q > 0) col[(o + (R - q) * NS) * LS] = hi;
            }
          }
        }
      }
  }
  if (!(GOUT && last)) __syncthreads();
}

// the whole transform of a workgroup's lines; GIN: the first pass reads ld(m),
// GOUT: the last one writes st(m, value); otherwise from LDS (written and a
// barrier passed before the call) and to LDS (a barrier passed on return)
template <typename T, int CLS, int SG, bool GIN, bool GOUT, class Ld, class St>
__device__ __forceinline__ void gen_fft(const GenAxis& ax, int P, int p, bool act, c_t<T>* col, int LS,
                                        const c_t<T>* tw, Ld ld, St st) {
  for (int i = 0; i < ax.np; ++i) {
    const GenPass& ps = ax.ps[i];
    const bool first = i == 0, last = i + 1 == ax.np;
#define MUGPU_GP(R) \
  case R: gen_pass<T, R, SG, GIN, GOUT>(ps, P, p, act, first, last, col, LS, tw, ld, st); break;
    if constexpr (CLS == 0) {
      switch (ps.R) {
        MUGPU_GP(2) MUGPU_GP(3) MUGPU_GP(4) MUGPU_GP(5) MUGPU_GP(7) MUGPU_GP(8) MUGPU_GP(9)
        default: break;
      }
    } else {
      switch (ps.R) {
        MUGPU_GP(2) MUGPU_GP(3) MUGPU_GP(4) MUGPU_GP(5) MUGPU_GP(7) MUGPU_GP(8) MUGPU_GP(9)
        MUGPU_GP(11) MUGPU_GP(13) MUGPU_GP(17)
        default: gen_prime<T, SG, GIN, GOUT>(ps, P, p, act, first, last, col, LS, tw, ld, st); break;
      }
    }
#undef MUGPU_GP
  }
}

// copy of the twiddle table behind the lines
template <typename T>
__device__ __forceinline__ void gen_twiddles(c_t<T>* dst, const c_t<T>* __restrict__ tw, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) dst[i] = tw[i];
}

}  // namespace
}  // namespace mugpu
