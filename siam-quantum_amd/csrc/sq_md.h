// sq_md.h - device-side building blocks of the two-electron kernels.
//
// Integrals are evaluated with the McMurchie-Davidson scheme: Hermite
// expansion coefficients E^{ij}_t per Cartesian axis, the Hermite Coulomb
// tensor R_{tuv} from the Boys function, and the contraction
//   (ab|cd) = 2 pi^{5/2}/(p q sqrt(p+q)) K_ab K_cd
//             sum_{tuv} E^{ab}_{tuv} sum_{TUV} (-1)^{T+U+V} E^{cd}_{TUV} R_{t+T,u+U,v+V}.
// Every loop bound is a template parameter, so the whole primitive-quartet
// evaluation unrolls into straight-line code with all intermediates in
// registers.  The Boys function F_m(T) is read from a table that each
// workgroup keeps in LDS (Taylor expansion about the nearest grid point plus
// downward recursion).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include <utility>

namespace sqmd {

// ---------------------------------------------------------------- basics
template <int V> using ic = std::integral_constant<int, V>;

template <typename F, int... I>
__host__ __device__ __forceinline__ void sfor_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(ic<I>{}), ...);
}
// compile-time for: f(ic<0>), ..., f(ic<N-1>)
template <int N, typename F>
__host__ __device__ __forceinline__ void sfor(F&& f) {
  sfor_impl(f, std::make_integer_sequence<int, N>{});
}

__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }
// number of (t,u,v) with t+u+v <= L
__host__ __device__ constexpr int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// Cartesian component order used by the GAMESS reader of the reference
// (src/basis.c:464-498): s; x y z; xx yy zz xy xz yz; f in that file's order.
struct Cart { int x, y, z; };
// Component i of angular momentum l, by arithmetic only (no lookup arrays,
// so that the value is the same in every compilation context).
__host__ __device__ constexpr Cart cart(int l, int i) {
  return l == 0 ? Cart{0, 0, 0}
       : l == 1 ? Cart{i == 0 ? 1 : 0, i == 1 ? 1 : 0, i == 2 ? 1 : 0}
       : l == 2 ? (i < 3 ? Cart{i == 0 ? 2 : 0, i == 1 ? 2 : 0, i == 2 ? 2 : 0}
                         : Cart{i == 5 ? 0 : 1, i == 4 ? 0 : 1, i == 3 ? 0 : 1})
       : (i == 0 ? Cart{3, 0, 0} : i == 1 ? Cart{0, 3, 0} : i == 2 ? Cart{0, 0, 3}
        : i == 3 ? Cart{2, 1, 0} : i == 4 ? Cart{1, 2, 0} : i == 5 ? Cart{2, 0, 1}
        : i == 6 ? Cart{1, 0, 2} : i == 7 ? Cart{0, 2, 1} : i == 8 ? Cart{0, 1, 2}
        : Cart{1, 1, 1});
}

// compact index of (t,u,v), t+u+v <= L, grouped by total order
__host__ __device__ constexpr int hidx(int t, int u, int v) {
  const int n = t + u + v;
  // entries of lower total order, then position inside order n
  const int below = n * (n + 1) * (n + 2) / 6;
  const int m = u + v;           // t = n - m
  return below + m * (m + 1) / 2 + v;
}

constexpr double kTwoPi25 = 34.986836655249725;  // 2 pi^{5/2}
constexpr double kPrimCutoff = 1.0e-15;            // bare prefactor cut

// ---------------------------------------------------------------- Boys
// Table: F_m(k*kBoysStep) for k in [0,kBoysNT), m in [0,kBoysNM), then
// exp(-k*kBoysStep) in column kBoysNM (row stride kBoysCols).
constexpr int kBoysNT = 651;
constexpr double kBoysStep = 0.1;
constexpr double kBoysTMax = (kBoysNT - 1) * kBoysStep;  // 65
constexpr int kBoysNM = 28;
constexpr int kBoysCols = kBoysNM + 1;
constexpr int kBoysTaylor = 9;  // terms of the Taylor expansion
constexpr int kBoysLdsW = kBoysTaylor + 1;  // LDS row: F_L .. F_{L+8}, exp(-T_k)

// Large-T branch of boys<L>: from T >= kBoysTCut[L] - 0.05 on, F_0 =
// sqrt(pi/T)/2 and the upward recursion without the exp(-T) term are within
// 2e-17 relative of F_m for every m <= L (checked against mpmath in steps of
// 0.5), so a class of total angular momentum L needs table rows up to
// kBoysTCut[L] only.  L = 9 is the (dd|dd) energy gradient.
constexpr double kBoysTCut[10] = {36.5, 40.5, 44.0, 47.0, 50.0, 52.5, 55.0, 57.5, 60.0, 62.5};
template <int L>
constexpr int boys_rows() {
  static_assert(L >= 0 && L <= 9, "Boys table cut-offs cover L <= 9");
  return (int)(kBoysTCut[L] / kBoysStep + 0.5) + 1;
}
static_assert(boys_rows<9>() <= kBoysNT, "table shorter than the largest cut-off");

// 1/j!
__host__ __device__ constexpr double inv_fact(int j) {
  double f = 1.0;
  for (int i = 2; i <= j; ++i) f *= i;
  return 1.0 / f;
}

// LDS copy for a class of total angular momentum L: per grid point the
// Taylor coefficients F_{L+j}/j!, j = 0..8, and exp(-T_k).  Dividing here
// makes each Taylor term of boys<L> one FMA instead of a product and an FMA.
template <int L>
__device__ __forceinline__ void boys_load_lds(double* lds, const double* __restrict__ tab) {
  // 16 threads a row (10 of them load), so that a thread keeps its column
  const int tid = threadIdx.x + threadIdx.y * blockDim.x, j = tid & 15;
  if (j >= kBoysLdsW) return;
  double f = 1.0;
  for (int i = 2; i <= j && j < kBoysTaylor; ++i) f *= i;
  const double inv = 1.0 / f;
  const double* col = tab + (j < kBoysTaylor ? L + j : kBoysNM);
  for (int k = tid >> 4; k < boys_rows<L>(); k += (blockDim.x * blockDim.y) >> 4)
    lds[k * kBoysLdsW + j] = col[k * kBoysCols] * inv;
}

// Nearest integer k of x in [0, 2^20] and the same as R, by adding 1.5 2^52
// (2^23 in float): two full-rate additions instead of two conversions.
__host__ __device__ __forceinline__ int round_near(double x, double& k) {
  const double t = x + 6755399441055744.0;
  k = t - 6755399441055744.0;
#ifdef __HIP_DEVICE_COMPILE__
  return __double2loint(t);
#else
  return (int)k;
#endif
}
__host__ __device__ __forceinline__ int round_near(float x, float& k) {
  const float t = x + 12582912.0f;
  k = t - 12582912.0f;
#ifdef __HIP_DEVICE_COMPILE__
  return __float_as_int(t) - 0x4b400000;
#else
  return (int)k;
#endif
}

// In an FP32 evaluation the rounding of a constant leans the same way in every
// integral, and a J element sums millions of them, so constants enter with a
// second FP32 part there: 0.1 of the table step is 1.5e-8 too large, 1/3, 1/5
// and 1/7 of the recursion 3e-8, 1.5e-8 and 4e-8, which left F_0 at L = 6
// 1.2e-7 too large on average over T < 30 (now 7e-10).
// T_k - T for the grid point k:
__host__ __device__ __forceinline__ double grid_offset(double k, double T) { return k * kBoysStep - T; }
__host__ __device__ __forceinline__ float grid_offset(float k, float T) {
  constexpr float hi = (float)kBoysStep, lo = (float)(kBoysStep - (double)hi);
  return fmaf(k, lo, fmaf(k, hi, -T));
}
// x / (2 M + 1):
template <int M>
__host__ __device__ __forceinline__ double div_odd(double x) { return x * (1.0 / (2 * M + 1)); }
template <int M>
__host__ __device__ __forceinline__ float div_odd(float x) {
  constexpr float hi = (float)(1.0 / (2 * M + 1)), lo = (float)(1.0 / (2 * M + 1) - (double)hi);
  return M == 0 ? x : fmaf(x, hi, x * lo);
}
// x sqrt(pi) / 2:
constexpr double kHalfSqrtPi = 0.88622692545275801365;
__host__ __device__ __forceinline__ double mul_half_sqrt_pi(double x) { return kHalfSqrtPi * x; }
__host__ __device__ __forceinline__ float mul_half_sqrt_pi(float x) {
  constexpr float hi = (float)kHalfSqrtPi, lo = (float)(kHalfSqrtPi - (double)hi);
  return fmaf(x, hi, x * lo);
}

// 1/sqrt(s) for s > 0: the hardware estimate refined by two Newton steps
// y <- y (3/2 - s/2 y^2), each of which squares the relative error.
__host__ __device__ __forceinline__ double rsqrt_nr(double s) {
#ifdef __HIP_DEVICE_COMPILE__
  double y = __builtin_amdgcn_rsq(s);
  const double h = 0.5 * s;
  y = y * fma(-h * y, y, 1.5);
  y = y * fma(-h * y, y, 1.5);
  return y;
#else
  return 1.0 / sqrt(s);
#endif
}
__host__ __device__ __forceinline__ float rsqrt_nr(float s) {
#ifdef __HIP_DEVICE_COMPILE__
  float y = __builtin_amdgcn_rsqf(s);  // hardware estimate, then one Newton step
  return y * (1.5f - 0.5f * s * y * y);
#else
  return 1.0f / sqrtf(s);
#endif
}


// F_0..F_L at T, evaluated in precision R (the table itself is FP64).
// T < kBoysTCut[L] - 0.05: F_L by Taylor expansion about the nearest grid point T_k,
// exp(-T) = exp(-T_k) exp(T_k - T) with the second factor by its Taylor
// series (|T_k - T| <= 0.05), then downward recursion.  Larger T: F_0 =
// sqrt(pi/T)/2 from the refined reciprocal square root (erfc(sqrt(T)) <
// 1e-27), and the upward recursion F_{m+1} = (2m+1) F_m / (2T) without the
// exp(-T) term, which changes F_m (m <= L) by less than 2e-17 relative
// there, so no exponential is evaluated on this branch.  FP32 evaluation
// needs fewer Taylor terms for the same relative accuracy.
template <int L, typename R = double>
__host__ __device__ __forceinline__ void boys(R T, R (&F)[L + 1], const double* lds) {
  constexpr int NT = sizeof(R) == 4 ? 5 : kBoysTaylor;  // 0.05^5/5! ~ 2.6e-9
  if (T < R(kBoysTCut[L] - 0.5 * kBoysStep)) {
    R kr;
    const int k = round_near(T * R(1.0 / kBoysStep), kr);
    const R d = grid_offset(kr, T);  // expansion in (T_k - T)
    const double* row = lds + k * kBoysLdsW;
    // F_L(T) = sum_j F_{L+j}(T_k) (T_k - T)^j / j!
    R s = R(row[NT - 1]);
    sfor<NT - 1>([&](auto jj) {
      constexpr int j = NT - 2 - decltype(jj)::value;
      s = s * d + R(row[j]);
    });
    F[L] = s;
    if constexpr (L > 0) {
      // exp(d) = sum_j d^j / j!, same number of terms as above
      R x = R(inv_fact(NT - 1));
      sfor<NT - 1>([&](auto jj) {
        constexpr int j = NT - 2 - decltype(jj)::value;
        x = x * d + R(inv_fact(j));
      });
      const R e = R(row[kBoysTaylor]) * x, t2 = T + T;
      sfor<L>([&](auto mm) {
        constexpr int m = L - 1 - decltype(mm)::value;
        F[m] = div_odd<m>(t2 * F[m + 1] + e);
      });
    }
  } else {
    // large T: F_0 = sqrt(pi/T)/2, F_{m+1} = (2m+1) F_m / (2T)
    const R y = rsqrt_nr(T);
    F[0] = mul_half_sqrt_pi(y);
    if constexpr (L > 0) {
      const R h = R(0.5) * y * y;
      sfor<L>([&](auto mm) {
        constexpr int m = decltype(mm)::value;
        F[m + 1] = (R(2 * m + 1) * h) * F[m];
      });
    }
  }
}

// ------------------------------------------------------ Hermite coefficients
// E[i][j][t], i<=LI, j<=LJ, t<=i+j  (unit K_ab factored out)
template <int LI, int LJ, typename R = double>
struct Herm1 {
  R e[LI + 1][LJ + 1][LI + LJ + 1];
};

template <int LI, int LJ, typename R>
__host__ __device__ __forceinline__ void herm_coef(Herm1<LI, LJ, R>& E, R xpa, R xpb, R h2p) {
  E.e[0][0][0] = R(1);
  sfor<LI>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    sfor<i + 2>([&](auto tt) {
      constexpr int t = decltype(tt)::value;
      R v = R(0);
      if constexpr (t >= 1) v += h2p * E.e[i][0][t - 1];
      if constexpr (t <= i) v += xpa * E.e[i][0][t];
      if constexpr (t + 1 <= i) v += R(t + 1) * E.e[i][0][t + 1];
      E.e[i + 1][0][t] = v;
    });
  });
  sfor<LI + 1>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    sfor<LJ>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      sfor<i + j + 2>([&](auto tt) {
        constexpr int t = decltype(tt)::value;
        R v = R(0);
        if constexpr (t >= 1) v += h2p * E.e[i][j][t - 1];
        if constexpr (t <= i + j) v += xpb * E.e[i][j][t];
        if constexpr (t + 1 <= i + j) v += R(t + 1) * E.e[i][j][t + 1];
        E.e[i][j + 1][t] = v;
      });
    });
  });
}

// ------------------------------------------------------ Hermite Coulomb R
// Which axis the recursion lowers for every entry (n; t,u,v), and which
// entries are needed at all.  An entry needs (t-1) at level n+1 and, for
// t > 1, (t-2) there too; taking for each the axis whose parents are already
// in use (and an index of at most 2, which costs one FMA instead of two
// operations) leaves fewer entries than lowering the first non-zero index
// everywhere: 102 instead of 120 at L = 5, in 120 operations instead of 151;
// 166 of 203 at L = 6.
template <int L>
struct RPlan {
  signed char axis[L + 1][nherm(L)];  // -1: not needed
  constexpr RPlan() : axis() {
    int tt[nherm(L)] = {}, uu[nherm(L)] = {}, vv[nherm(L)] = {};
    for (int o = 0; o <= L; ++o)
      for (int m = 0; m <= o; ++m)
        for (int v = 0; v <= m; ++v) {
          const int i = hidx(o - m, m - v, v);
          tt[i] = o - m; uu[i] = m - v; vv[i] = v;
        }
    for (int n = 0; n <= L; ++n)
      for (int i = 0; i < nherm(L); ++i) axis[n][i] = -1;
    bool need[L + 2][nherm(L)] = {};
    for (int i = 0; i < nherm(L); ++i) need[0][i] = true;
    for (int n = 0; n <= L; ++n)
      for (int o = L - n; o >= 1; --o)
        for (int nz = 1; nz <= 3; ++nz)  // entries with the fewest choices first
          for (int i = (o * (o + 1) * (o + 2)) / 6; i < ((o + 1) * (o + 2) * (o + 3)) / 6; ++i) {
            const int e[3] = {tt[i], uu[i], vv[i]};
            if (!need[n][i] || (e[0] > 0) + (e[1] > 0) + (e[2] > 0) != nz) continue;
            int best = -1, cost = 1 << 20, p1b = 0, p2b = -1;
            for (int a = 0; a < 3; ++a) {
              if (e[a] == 0) continue;
              const int p1 = hidx(e[0] - (a == 0), e[1] - (a == 1), e[2] - (a == 2));
              const int p2 = e[a] > 1 ? hidx(e[0] - 2 * (a == 0), e[1] - 2 * (a == 1), e[2] - 2 * (a == 2)) : -1;
              const int c = (need[n + 1][p1] ? 0 : 1) + (p2 >= 0 && !need[n + 1][p2] ? 1 : 0) + (e[a] > 2 ? 1 : 0);
              if (c < cost) { cost = c; best = a; p1b = p1; p2b = p2; }
            }
            axis[n][i] = (signed char)best;
            need[n + 1][p1b] = true;
            if (p2b >= 0) need[n + 1][p2b] = true;
          }
  }
};

// pref R^{(0)}_{tuv} for t+u+v <= L, built level by level from
// R^{(n)}_{000} = (-2 alpha)^n F_n.  alpha and its powers are FP64 in an FP32
// evaluation too: alpha is the same for all quartets of a kind, so its
// rounding would lean the same way in all of them.
template <int L, typename Rl = double>
__host__ __device__ __forceinline__ void herm_R(Rl (&R)[nherm(L)], const Rl (&F)[L + 1],
                                       double alpha, Rl X, Rl Y, Rl Z, double pref = 1.0) {
  constexpr RPlan<L> plan{};
  Rl lev[L + 1][nherm(L)];
  double m2a = -2.0 * alpha, pw = pref;
  sfor<L + 1>([&](auto nn) {
    constexpr int n = decltype(nn)::value;
    lev[n][0] = Rl(pw) * F[n];
    pw *= m2a;
  });
  // level n holds orders up to L-n; build from n = L-1 down to 0
  sfor<L>([&](auto kk) {
    constexpr int n = L - 1 - decltype(kk)::value;
    constexpr int top = L - n;
    sfor<top>([&](auto oo) {
      constexpr int o = decltype(oo)::value + 1;  // total order 1..top
      sfor<o + 1>([&](auto mm) {
        constexpr int m = decltype(mm)::value;     // u+v
        sfor<m + 1>([&](auto vv) {
          constexpr int v = decltype(vv)::value;
          constexpr int u = m - v, t = o - m;
          constexpr int ax = plan.axis[n][hidx(t, u, v)];
          if constexpr (ax >= 0) {
            constexpr int k = ax == 0 ? t : ax == 1 ? u : v;
            Rl r = (ax == 0 ? X : ax == 1 ? Y : Z) * lev[n + 1][hidx(t - (ax == 0), u - (ax == 1), v - (ax == 2))];
            if constexpr (k > 1)
              r += Rl(k - 1) * lev[n + 1][hidx(t - 2 * (ax == 0), u - 2 * (ax == 1), v - 2 * (ax == 2))];
            lev[n][hidx(t, u, v)] = r;
          }
        });
      });
    });
  });
  sfor<nherm(L)>([&](auto ii) { R[decltype(ii)::value] = lev[0][decltype(ii)::value]; });
}

}  // namespace sqmd
