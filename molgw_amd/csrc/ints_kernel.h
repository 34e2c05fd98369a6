// Device code of the two- and three-centre Coulomb integrals over contracted
// Gaussian shells on the GPU (one launcher per translation unit, ints_l*.hip), for the RI tensor of the integral front end:
//   (mu nu|P)  of calculate_integrals_eri_3center_scalapack (src/m_eri_calculate.f90:1266-1580),
//   (P|Q)      of calculate_integrals_eri_2center_scalapack (src/m_eri_calculate.f90:703-945),
// which the reference takes from libcint (cint3c2e / cint2c2e,
// src/m_libcint_tools.f90:54-260). Written from the McMurchie-Davidson
// scheme:
//   (ab|c) = 2 pi^(5/2) / (p q sqrt(p + q)) sum_tuv E^ab_tuv sum_tau,nu,phi
//            (-1)^(tau+nu+phi) E^c_(tau nu phi) R_(t+tau, u+nu, v+phi)(alpha, P - C)
// with E the Hermite expansion coefficients of the bra product and of the
// single ket Gaussian, alpha = p q / (p + q), and R the Hermite Coulomb
// integrals from the Boys function.
//
// Work decomposition. Shell pairs are grouped by (l_a, l_b), ket functions
// (shell, function) by l_c; one launch per class (l_a, l_b, l_c) with the
// three angular momenta as template parameters, so every index into R, E and
// the accumulators is a compile-time constant. A workgroup owns one bra shell
// pair and 128 ket functions of one l_c; the bra's primitive pairs are expanded
// (E coefficients, P, p) cooperatively into LDS in batches and read as
// broadcasts. Each thread keeps, per ket primitive, R in one in-place array
// (levels n = L .. 0, sums t+u+v processed from high to low so that level n + 1
// is read before it is overwritten), the ket's Hermite coefficients of its final
// function, and the Cartesian bra block of its function in registers; the bra is
// transformed to the final functions once at the end.
//
// What bounds it: FP64 instructions in the deeply contracted (s s|, (p s|
// classes (64 primitive pairs a bra), registers and code size in the others,
// where a bra has one primitive pair and every instruction is fetched for one
// use. So divisions by constants are products, a primitive takes one division
// and one square root, an uncontracted ket's coefficients (half of them zero by
// parity, and skipped) are found once, E is read again from LDS rather than
// held, and the transform at the end is a loop. All classes of an 8-carbon
// alkane in cc-pVDZ / cc-pVDZ-RI (202 functions): 2.02 -> 0.93 ms, of which
// (s s|f) 0.42 -> 0.07 (its coefficients were in scratch memory) and the four
// (d d| 0.32 -> 0.10.
//
// Boys function: F_L(T) by a 7-term Taylor series around the nearest point
// of a table F_n(k h), h = 0.05, T <= 36 (error below 2e-15 relative), then
// downward recursion; above T = 36, F_0 = sqrt(pi / T) / 2 (the neglected
// tail is e^-T < 3e-16) and upward recursion. The recursions' divisions are
// products with a reciprocal and a correction by the residual, as accurate as
// divisions (0.3 % of the alkane's time; without it the rounding of the one
// reciprocal adds up over the orders, 2.2 -> 5.3e-16 for F_10).
#pragma once
#include "mgw_internal.h"

#include <cmath>
#include <type_traits>
#include <utility>

namespace mgw {
namespace eri {

// f(0), .., f(N - 1) with the index as a constant expression: the loops below
// nest four deep with bounds of one another, which the compiler's unroller gives
// up on at the higher angular momenta; indices it does not know put an array
// into scratch memory
template <class F, int... I>
__device__ __attribute__((always_inline)) inline void unroll_seq(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __attribute__((always_inline)) inline void unroll(F&& f) {
  unroll_seq(f, std::make_integer_sequence<int, N>{});
}
#define MGW_UNROLL(i, n) unroll<(n)>([&](auto i) __attribute__((always_inline))

constexpr int BOYS_N = 17;          // orders 0 .. 16 in the table (L <= 10 plus 6 Taylor terms)
constexpr int BOYS_TAYLOR = 6;
constexpr double BOYS_H = 0.05;
constexpr double BOYS_TMAX = 36.0;
constexpr int BOYS_NT = 721;        // points 0, h, .., 36

__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
// R_{t,u,v}, t + u + v <= L: sums s in increasing order, then (u + v, v)
__host__ __device__ constexpr int hidx(int t, int u, int v) {
  const int s = t + u + v, r = u + v;
  return s * (s + 1) * (s + 2) / 6 + r * (r + 1) / 2 + v;
}
// and back: the sum s and r = u + v of an index, then t, u, v
__host__ __device__ constexpr int herm_s(int m) {
  int s = 0;
  while (nherm(s) <= m) ++s;
  return s;
}
__host__ __device__ constexpr int herm_r(int m) {
  const int s = herm_s(m), k = s > 0 ? m - nherm(s - 1) : 0;
  int r = 0;
  while ((r + 1) * (r + 2) / 2 <= k) ++r;
  return r;
}
__host__ __device__ constexpr int herm_t(int m) { return herm_s(m) - herm_r(m); }
__host__ __device__ constexpr int herm_v(int m) {
  const int s = herm_s(m), r = herm_r(m);
  return m - (s > 0 ? nherm(s - 1) : 0) - r * (r + 1) / 2;
}
__host__ __device__ constexpr int herm_u(int m) { return herm_r(m) - herm_v(m); }
// Cartesian component c of a shell of angular momentum l: (l - i, i - k, k)
// for i = 0 .. l, k = 0 .. i (x power decreasing first), as the basis module
// orders them
__host__ __device__ constexpr int cart_i(int c) {
  int i = 0;
  while ((i + 1) * (i + 2) / 2 <= c) ++i;
  return i;
}
__host__ __device__ constexpr int cart_x(int l, int c) { return l - cart_i(c); }
__host__ __device__ constexpr int cart_y(int l, int c) { return cart_i(c) - (c - cart_i(c) * (cart_i(c) + 1) / 2); }
__host__ __device__ constexpr int cart_z(int l, int c) { return c - cart_i(c) * (cart_i(c) + 1) / 2; }

struct ShellsDev {
  const int32_t* l;
  const double* center;
  const int32_t* poff;
  const double* exps;
  const double* coefs;
  const int32_t* toff;
  const double* tmat;
  const int32_t* foff;
};

struct EriArgs {
  ShellsDev A, B, C;
  const int2* pairs;       // bra shell pairs (sa in A, sb in B) of the class
  const int2* kfun;        // ket functions (sc, f) of the class
  int nkfun;
  const int32_t* kshell;   // ket shells of the class
  int nkshell, lanes;      // lanes: of a workgroup, side by side on ket shells (power of two)
  const double* boys;      // [BOYS_NT][BOYS_N]
  int metric;              // 0: packed (mu nu|P); 1: (P|Q) with B the unit shells
  const int32_t* pairmap;  // 0: pair index of (mu, nu) (nbf x nbf) or -1
  int nbf;
  int64_t npair;
  int naux;                // 1: leading dimension of (P|Q)
  double* out;
};

// a / b for a given rounded r = 1 / b: one product and the residual's correction,
// as accurate as a division; r alone would leave its own rounding in every
// order of the recursions below
__device__ inline double corrected_quotient(double a, double b, double r) {
  const double q = a * r;
  return fma(fma(-b, q, a), r, q);
}

template <int L>
__device__ inline void boys_eval(double T, const double* __restrict__ tab, double* f) {
  if (T < BOYS_TMAX) {
    const int k = (int)(T * (1.0 / BOYS_H) + 0.5);
    const double d = k * BOYS_H - T;
    const double* __restrict__ row = tab + k * BOYS_N + L;
    // F_L(T) = sum_j F_{L+j}(t_k) (t_k - T)^j / j!
    double s = row[BOYS_TAYLOR];
#pragma unroll
    for (int j = BOYS_TAYLOR - 1; j >= 0; --j) s = row[j] + s * (d * (1.0 / (double)(j + 1)));
    f[L] = s;
    const double e = exp(-T);
#pragma unroll
    for (int n = L - 1; n >= 0; --n)
      f[n] = corrected_quotient(2.0 * T * f[n + 1] + e, (double)(2 * n + 1), 1.0 / (double)(2 * n + 1));
  } else {
    const double e = exp(-T), h = 0.5 / T;
    f[0] = 0.5 * sqrt(corrected_quotient(6.28318530717958647693, 2.0 * T, h));
#pragma unroll
    for (int n = 0; n < L; ++n) f[n + 1] = corrected_quotient((double)(2 * n + 1) * f[n] - e, 2.0 * T, h);
  }
}

// Hermite expansion of one dimension of a primitive pair into e[(i (LB+1) + j) (LAB+1) + t]
// (i <= LA, j <= LB, t <= i + j); e[0] carries exp(-mu X_AB^2).
template <int LA, int LB>
__device__ inline void hermite_pair(double a, double b, double xab, double* __restrict__ e) {
  constexpr int LAB = LA + LB, LD = LAB + 1;
  const double p = a + b, mu = a * b / p;
  const double xpa = -b * xab / p, xpb = a * xab / p, h = 0.5 / p;
  for (int n = 0; n < (LA + 1) * (LB + 1) * LD; ++n) e[n] = 0.0;
  e[0] = exp(-mu * xab * xab);
  for (int i = 0; i <= LA; ++i)
    for (int j = 0; j <= LB; ++j) {
      if (i == 0 && j == 0) continue;
      const double* src;
      double x;
      if (i > 0) {
        src = e + ((i - 1) * (LB + 1) + j) * LD;
        x = xpa;
      } else {
        src = e + (j - 1) * LD;
        x = xpb;
      }
      double* dst = e + (i * (LB + 1) + j) * LD;
      const int top = i + j - 1;
      for (int t = 0; t <= i + j; ++t) {
        double v = (t <= top ? x * src[t] : 0.0);
        if (t > 0 && t - 1 <= top) v += h * src[t - 1];
        if (t + 1 <= top) v += (t + 1) * src[t + 1];
        dst[t] = v;
      }
    }
}

// R_tuv(alpha, P - C), t + u + v <= L, in place: level L, then down to level 0
template <int L>
__device__ __attribute__((always_inline)) inline void hermite_coulomb(double alpha, double xpc, double ypc, double zpc,
                                                                      const double* __restrict__ boys, double* R) {
  double f[L + 1];
  boys_eval<L>(alpha * (xpc * xpc + ypc * ypc + zpc * zpc), boys, f);
  // level L, then down to level 0 in place
  double pw[L + 1];
  pw[0] = 1.0;
#pragma unroll
  for (int n = 1; n <= L; ++n) pw[n] = pw[n - 1] * (-2.0 * alpha);
  R[0] = pw[L] * f[L];
  MGW_UNROLL(step, L) {
    constexpr int n = L - 1 - step, top = nherm(L - n) - 1;
    MGW_UNROLL(i, top) {
      constexpr int m = top - i, t = herm_t(m), u = herm_u(m), v = herm_v(m);
      double val;
      if constexpr (t > 0) {
        val = xpc * R[hidx(t - 1, u, v)];
        if constexpr (t > 1) val += (t - 1) * R[hidx(t - 2, u, v)];
      } else if constexpr (u > 0) {
        val = ypc * R[hidx(t, u - 1, v)];
        if constexpr (u > 1) val += (u - 1) * R[hidx(t, u - 2, v)];
      } else {
        val = zpc * R[hidx(t, u, v - 1)];
        if constexpr (v > 1) val += (v - 1) * R[hidx(t, u, v - 2)];
      }
      R[m] = val;
    });
    R[0] = pw[n] * f[n];
  });
}

// Hermite coefficients of one final function of a ket primitive (1 / 2q = h):
// K(tau nu phi) = (-1)^(tau+nu+phi) sum_c tc[c] Ec[cx][tau] Ec[cy][nu] Ec[cz][phi];
// zero unless tau + nu + phi has the parity of LC
template <int LC>
__device__ inline void ket_hermite(const double* tc, double h, double* K) {
  double ec[LC + 1][LC + 1];
#pragma unroll
  for (int i = 0; i <= LC; ++i)
#pragma unroll
    for (int t = 0; t <= LC; ++t) ec[i][t] = 0.0;
  ec[0][0] = 1.0;
#pragma unroll
  for (int i = 1; i <= LC; ++i)
#pragma unroll
    for (int t = 0; t <= i; ++t) {
      double v = 0.0;
      if (t > 0) v += h * ec[i - 1][t - 1];
      if (t + 1 <= i - 1) v += (t + 1) * ec[i - 1][t + 1];
      ec[i][t] = v;
    }
#pragma unroll
  for (int n = 0; n < nherm(LC); ++n) K[n] = 0.0;
  MGW_UNROLL(c, ncart(LC)) {
    constexpr int ex = cart_x(LC, c), ey = cart_y(LC, c), ez = cart_z(LC, c);
    MGW_UNROLL(m, nherm(LC)) {
      constexpr int t = herm_t(m), u = herm_u(m), v = herm_v(m);
      if constexpr (t <= ex && u <= ey && v <= ez && !(((ex - t) | (ey - u) | (ez - v)) & 1)) {   // else zero
        constexpr double sg = (LC & 1) ? -1.0 : 1.0;
        K[m] += sg * tc[c] * ec[ex][t] * ec[ey][u] * ec[ez][v];
      }
    });
  });
}

constexpr int WG = 128;   // ket functions per workgroup
constexpr int NPB = 8;    // bra primitive pairs expanded per LDS batch

template <int LA, int LB, int LC>
__global__ void __launch_bounds__(WG) eri_kernel(EriArgs g) {
  constexpr int LAB = LA + LB, L = LAB + LC;
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC);
  constexpr int LD = LAB + 1;
  constexpr int NE = (LA + 1) * (LB + 1) * LD;
  __shared__ double sE[NPB][3][NE];
  __shared__ double sQ[NPB][5];   // p, P (3), contraction weight / p

  const int2 pr = g.pairs[blockIdx.x];
  const int sa = pr.x, sb = pr.y;
  const int kf = blockIdx.y * WG + threadIdx.x;
  int sc = 0, fc = 0;
  bool active = kf < g.nkfun;
  if (active) {
    const int2 t = g.kfun[kf];
    sc = t.x;
    fc = t.y;
    // the metric is symmetric: shell blocks with sc > sa are the mirror of another thread's
    if (g.metric && sc > sa) active = false;
  }
  const double ax = g.A.center[3 * sa], ay = g.A.center[3 * sa + 1], az = g.A.center[3 * sa + 2];
  const double bx = g.B.center[3 * sb], by = g.B.center[3 * sb + 1], bz = g.B.center[3 * sb + 2];
  const int ia0 = g.A.poff[sa], nia = g.A.poff[sa + 1] - ia0;
  const int ib0 = g.B.poff[sb], nib = g.B.poff[sb + 1] - ib0;
  const int nprim = nia * nib;

  double cx = 0.0, cy = 0.0, cz = 0.0;
  int k0 = 0, k1 = 0;
  double tc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) tc[c] = 0.0;
  if (active) {
    cx = g.C.center[3 * sc];
    cy = g.C.center[3 * sc + 1];
    cz = g.C.center[3 * sc + 2];
    k0 = g.C.poff[sc];
    k1 = g.C.poff[sc + 1];
    const double* __restrict__ t = g.C.tmat + g.C.toff[sc] + fc * NC;
#pragma unroll
    for (int c = 0; c < NC; ++c) tc[c] = t[c];
  }

  // of a ket of one primitive (an uncontracted auxiliary shell), once for all
  // bra primitives
  const bool one = k1 - k0 == 1;
  double K[nherm(LC)], qe = 1.0, qw = 0.0;
  if (one) {
    qe = g.C.exps[k0];
    qw = 2.0 * 17.493418327624862 / qe * g.C.coefs[k0];   // 2 pi^(5/2)
    ket_hermite<LC>(tc, 0.5 / qe, K);
  }

  double acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = 0.0;

  for (int base = 0; base < nprim; base += NPB) {
    const int nb = min(NPB, nprim - base);
    __syncthreads();   // previous batch consumed
    if (threadIdx.x < 3 * nb) {
      const int q = threadIdx.x / 3, d = threadIdx.x % 3;
      const int ip = base + q;
      const double a = g.A.exps[ia0 + ip / nib], b = g.B.exps[ib0 + ip % nib];
      const double xab = d == 0 ? ax - bx : d == 1 ? ay - by : az - bz;
      hermite_pair<LA, LB>(a, b, xab, &sE[q][d][0]);
      if (d == 0) {
        const double p = a + b;
        sQ[q][0] = p;
        sQ[q][1] = (a * ax + b * bx) / p;
        sQ[q][2] = (a * ay + b * by) / p;
        sQ[q][3] = (a * az + b * bz) / p;
        sQ[q][4] = g.A.coefs[ia0 + ip / nib] * g.B.coefs[ib0 + ip % nib] / p;
      }
    }
    __syncthreads();
    if (!active) continue;
    for (int q = 0; q < nb; ++q) {
      const double p = sQ[q][0], px = sQ[q][1], py = sQ[q][2], pz = sQ[q][3], wab = sQ[q][4];
      for (int k = k0; k < k1; ++k) {
        if (!one) {
          qe = g.C.exps[k];
          qw = 2.0 * 17.493418327624862 / qe * g.C.coefs[k];
          ket_hermite<LC>(tc, 0.5 / qe, K);
        }
        const double rpq = 1.0 / (p + qe), alpha = p * qe * rpq;
        const double xpc = px - cx, ypc = py - cy, zpc = pz - cz;
        double R[nherm(L)];
        hermite_coulomb<L>(alpha, xpc, ypc, zpc, g.boys, R);
        // ket-contracted Hermite integrals G(tuv), t + u + v <= LAB
        double G[nherm(LAB)];
        MGW_UNROLL(m, nherm(LAB)) {
          constexpr int t = herm_t(m), u = herm_u(m), v = herm_v(m);
          double sum = 0.0;
          MGW_UNROLL(m2, nherm(LC)) {
            if constexpr ((herm_s(m2) & 1) == (LC & 1))   // else K = 0
              sum += K[m2] * R[hidx(t + herm_t(m2), u + herm_u(m2), v + herm_v(m2))];
          });
          G[m] = sum;
        });
        const double pref = sqrt(rpq) * wab * qw;
        // bra: acc[a][b] += pref sum_tuv Ex Ey Ez G
        MGW_UNROLL(ab, NA * NB) {
          constexpr int a = ab / NB, b = ab % NB;
          // from (p p| on, E is read again for each function of a: kept for all
          // of them it takes the registers of acc and G
          if constexpr (LAB >= 2 && b == 0) __asm__ __volatile__("" ::: "memory");
          constexpr int ix = cart_x(LA, a), iy = cart_y(LA, a), iz = cart_z(LA, a);
          constexpr int jx = cart_x(LB, b), jy = cart_y(LB, b), jz = cart_z(LB, b);
          const double* __restrict__ ex = &sE[q][0][(ix * (LB + 1) + jx) * LD];
          const double* __restrict__ ey = &sE[q][1][(iy * (LB + 1) + jy) * LD];
          const double* __restrict__ ez = &sE[q][2][(iz * (LB + 1) + jz) * LD];
          double sum = 0.0;
          MGW_UNROLL(t, ix + jx + 1) {
            MGW_UNROLL(u, iy + jy + 1) {
              const double etu = ex[t] * ey[u];
              MGW_UNROLL(v, iz + jz + 1) { sum += etu * ez[v] * G[hidx(t, u, v)]; });
            });
          });
          acc[a][b] += pref * sum;
        });
      }
    }
  }
  if (!active) return;

  // final functions of the bra: V(fa, fb) = sum_ab Ta[fa][a] Tb[fb][b] acc[a][b].
  // The loops over the functions stay loops: code that runs once costs its
  // fetch from memory (unrolled, this part was most of the (d d|c) classes' time)
  const int nfa = g.A.foff[sa + 1] - g.A.foff[sa], nfb = g.B.foff[sb + 1] - g.B.foff[sb];
  const double* __restrict__ ta = g.A.tmat + g.A.toff[sa];
  const double* __restrict__ tb = g.B.tmat + g.B.toff[sb];
  double half[NB];
  auto half_row = [&](int fa) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      double s = 0.0;
#pragma unroll
      for (int a = 0; a < NA; ++a) s += ta[fa * NA + a] * acc[a][b];
      half[b] = s;
    }
  };
  auto value = [&](int fb) __attribute__((always_inline)) {
    double s = 0.0;
#pragma unroll
    for (int b = 0; b < NB; ++b) s += tb[fb * NB + b] * half[b];
    return s;
  };

  if (g.metric) {
    // (P|Q): the bra's second shell is the unit function; write both triangles
    const int64_t Q = g.C.foff[sc] + fc;
#pragma unroll 1
    for (int fa = 0; fa < nfa; ++fa) {
      if (sc == sa && fa < fc) continue;   // one writer per element of a diagonal block
      half_row(fa);
      const double v = value(0);
      const int64_t P = g.A.foff[sa] + fa;
      g.out[P + Q * g.naux] = v;
      g.out[Q + P * g.naux] = v;
    }
    return;
  }
  const int64_t P = g.C.foff[sc] + fc;
  const bool same = sa == sb && g.A.l == g.B.l;
#pragma unroll 1
  for (int fa = 0; fa < nfa; ++fa)
#pragma unroll 1
    for (int fb = 0; fb < nfb; ++fb) {
      const int mu = g.A.foff[sa] + fa, nu = g.B.foff[sb] + fb;
      const int32_t ip = g.pairmap[(int64_t)mu * g.nbf + nu];
      if (ip < 0) continue;
      half_row(fa);
      double v = value(fb);
      if (same) {
        if constexpr (NA == NB) {
          half_row(fb);
          v = 0.5 * (v + value(fa));
        }
        if (mu == nu) v *= 0.5;   // diagonal pairs stored x1/2
      }
      g.out[ip + P * g.npair] = v;
    }
}

// Number of ways h^((i + t) / 2) enters E^i_t of a single Gaussian (h = 1 / 2q):
// i! / (t! m! 2^m), m = (i - t) / 2; zero for odd i - t
__host__ __device__ constexpr double ket_weight(int i, int t) {
  if (t > i || ((i - t) & 1)) return 0.0;
  double w = 1.0;
  for (int k = t + 1; k <= i; ++k) w *= k;
  for (int k = 1; k <= (i - t) / 2; ++k) w /= 2.0 * k;
  return w;
}

constexpr int NPS = 16;   // bra primitive pairs expanded per LDS batch

// The classes (s s|c) and (p s|c), whose time is the Coulomb integrals R of up to
// 64 primitive pairs a bra: a thread owns a ket shell instead of one of its
// 2 l_c + 1 functions, forms R once for all of them and accumulates the ket's
// Cartesian components (at most 15 x 3 sums); each component is a few terms of R
// times a power of h. Few ket shells of one l_c leave lanes over (16 f shells in
// an 8-carbon alkane): the workgroup is lanes shells wide and its 128 / lanes
// slices share the primitive pairs, summed through LDS in a fixed order; that also
// cuts the chain of 64 primitive pairs that a launch ends on. The eight classes
// of that alkane: 0.52 -> 0.32 ms (0.35 with up to 128 lanes, 0.39 with 16).
template <int LA, int LC>
__global__ void __launch_bounds__(WG) eri_shell_kernel(EriArgs g) {
  constexpr int L = LA + LC, NA = ncart(LA), NC = ncart(LC), LD = LA + 1, NE = (LA + 1) * LD;
  __shared__ double sE[NPS][3][NE];
  __shared__ double sQ[NPS][5];   // p, P (3), contraction weight / p
  __shared__ double red[WG];

  const int2 pr = g.pairs[blockIdx.x];
  const int sa = pr.x, sb = pr.y;
  const int lane = threadIdx.x & (g.lanes - 1), slice = threadIdx.x / g.lanes, nslice = WG / g.lanes;
  const int ks = blockIdx.y * g.lanes + lane;
  bool active = ks < g.nkshell;
  int sc = 0;
  if (active) {
    sc = g.kshell[ks];
    // the metric is symmetric: shell blocks with sc > sa are the mirror of another thread's
    if (g.metric && sc > sa) active = false;
  }
  const double ax = g.A.center[3 * sa], ay = g.A.center[3 * sa + 1], az = g.A.center[3 * sa + 2];
  const double bx = g.B.center[3 * sb], by = g.B.center[3 * sb + 1], bz = g.B.center[3 * sb + 2];
  const int ia0 = g.A.poff[sa], nia = g.A.poff[sa + 1] - ia0;
  const int ib0 = g.B.poff[sb], nib = g.B.poff[sb + 1] - ib0;
  const int nprim = nia * nib;
  double cx = 0.0, cy = 0.0, cz = 0.0, qe = 1.0, qw = 0.0;
  int k0 = 0, k1 = 0;
  if (active) {
    cx = g.C.center[3 * sc];
    cy = g.C.center[3 * sc + 1];
    cz = g.C.center[3 * sc + 2];
    k0 = g.C.poff[sc];
    k1 = g.C.poff[sc + 1];
  }
  const bool one = k1 - k0 == 1;
  if (one) {
    qe = g.C.exps[k0];
    qw = 2.0 * 17.493418327624862 / qe * g.C.coefs[k0];   // 2 pi^(5/2)
  }

  double acc[NC][NA];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[c][a] = 0.0;

  for (int base = 0; base < nprim; base += NPS) {
    const int nb = min(NPS, nprim - base);
    __syncthreads();   // previous batch consumed
    if (threadIdx.x < 3 * nb) {
      const int q = threadIdx.x / 3, d = threadIdx.x % 3;
      const int ip = base + q;
      const double a = g.A.exps[ia0 + ip / nib], b = g.B.exps[ib0 + ip % nib];
      const double xab = d == 0 ? ax - bx : d == 1 ? ay - by : az - bz;
      hermite_pair<LA, 0>(a, b, xab, &sE[q][d][0]);
      if (d == 0) {
        const double p = a + b;
        sQ[q][0] = p;
        sQ[q][1] = (a * ax + b * bx) / p;
        sQ[q][2] = (a * ay + b * by) / p;
        sQ[q][3] = (a * az + b * bz) / p;
        sQ[q][4] = g.A.coefs[ia0 + ip / nib] * g.B.coefs[ib0 + ip % nib] / p;
      }
    }
    __syncthreads();
    for (int q = slice; q < nb; q += nslice) {
      const double p = sQ[q][0], px = sQ[q][1], py = sQ[q][2], pz = sQ[q][3], wab = sQ[q][4];
      for (int k = k0; k < k1; ++k) {
        if (!one) {
          qe = g.C.exps[k];
          qw = 2.0 * 17.493418327624862 / qe * g.C.coefs[k];
        }
        const double rpq = 1.0 / (p + qe), alpha = p * qe * rpq;
        double R[nherm(L)];
        hermite_coulomb<L>(alpha, px - cx, py - cy, pz - cz, g.boys, R);
        // pref h^((LC + s) / 2), signed: the weight of the terms R with ket sum s
        double hp[LC + 1];
        {
          const double h = 0.5 / qe;
          double w = ((LC & 1) ? -1.0 : 1.0) * sqrt(rpq) * wab * qw;
#pragma unroll
          for (int n = 0; n < (LC + 1) / 2; ++n) w *= h;
#pragma unroll
          for (int s = LC & 1; s <= LC; s += 2) {
            hp[s] = w;
            w *= h;
          }
        }
        MGW_UNROLL(c, NC) {
          constexpr int ex = cart_x(LC, c), ey = cart_y(LC, c), ez = cart_z(LC, c);
          double G[nherm(LA)];
          MGW_UNROLL(m, nherm(LA)) {
            constexpr int t = herm_t(m), u = herm_u(m), v = herm_v(m);
            double sum = 0.0;
            MGW_UNROLL(s, LC + 1) {
              if constexpr (!((s ^ LC) & 1)) {
                double part = 0.0;
                MGW_UNROLL(m2, nherm(LC)) {
                  if constexpr (herm_s(m2) == s) {
                    constexpr double w = ket_weight(ex, herm_t(m2)) * ket_weight(ey, herm_u(m2)) * ket_weight(ez, herm_v(m2));
                    if constexpr (w != 0.0) part += w * R[hidx(t + herm_t(m2), u + herm_u(m2), v + herm_v(m2))];
                  }
                });
                sum += hp[s] * part;
              }
            });
            G[m] = sum;
          });
          MGW_UNROLL(a, NA) {
            constexpr int ix = cart_x(LA, a), iy = cart_y(LA, a), iz = cart_z(LA, a);
            double sum = 0.0;
            MGW_UNROLL(t, ix + 1) {
              MGW_UNROLL(u, iy + 1) {
                const double etu = sE[q][0][ix * LD + t] * sE[q][1][iy * LD + u];
                MGW_UNROLL(v, iz + 1) { sum += etu * sE[q][2][iz * LD + v] * G[hidx(t, u, v)]; });
              });
            });
            acc[c][a] += sum;
          });
        });
      }
    }
  }
  if (nslice > 1 && nprim > 1) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        __syncthreads();
        red[threadIdx.x] = acc[c][a];
        __syncthreads();
        if (slice == 0)
          for (int s = 1; s < nslice; ++s) acc[c][a] += red[s * g.lanes + lane];
      }
  }
  if (!active || slice > 0) return;

  // final functions, as in eri_kernel: V(fa, f) = Tb sum_a Ta[fa][a] sum_c Tc[f][c] acc[c][a]
  const int nfa = g.A.foff[sa + 1] - g.A.foff[sa], nfc = g.C.foff[sc + 1] - g.C.foff[sc];
  const double* __restrict__ ta = g.A.tmat + g.A.toff[sa];
  const double* __restrict__ tc = g.C.tmat + g.C.toff[sc];
  const double tb = g.B.tmat[g.B.toff[sb]];
#pragma unroll 1
  for (int fa = 0; fa < nfa; ++fa) {
    const int mu = g.A.foff[sa] + fa, nu = g.B.foff[sb];
    const int32_t ip = g.metric ? 0 : g.pairmap[(int64_t)mu * g.nbf + nu];
    if (ip < 0) continue;
    double half[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      double s = 0.0;
#pragma unroll
      for (int a = 0; a < NA; ++a) s += ta[fa * NA + a] * acc[c][a];
      half[c] = s;
    }
#pragma unroll 1
    for (int f = 0; f < nfc; ++f) {
      double v = 0.0;
#pragma unroll
      for (int c = 0; c < NC; ++c) v += tc[f * NC + c] * half[c];
      v *= tb;
      const int64_t P = g.C.foff[sc] + f;
      if (g.metric) {
        if (sc == sa && fa < f) continue;   // one writer per element of a diagonal block
        g.out[mu + P * g.naux] = v;
        g.out[P + (int64_t)mu * g.naux] = v;
      } else {
        g.out[ip + P * g.npair] = (sa == sb && LA == 0) ? 0.5 * v : v;   // diagonal pairs stored x1/2
      }
    }
  }
}

// launch one class of the translation unit that holds it
int launch_la0(int lb, int lc, dim3 grid, const EriArgs& g, hipStream_t s);
int launch_la1(int lb, int lc, dim3 grid, const EriArgs& g, hipStream_t s);
int launch_la2(int lb, int lc, dim3 grid, const EriArgs& g, hipStream_t s);
int launch_la3(int lb, int lc, dim3 grid, const EriArgs& g, hipStream_t s);
int launch_la4(int lb, int lc, dim3 grid, const EriArgs& g, hipStream_t s);

}  // namespace eri
}  // namespace mgw
