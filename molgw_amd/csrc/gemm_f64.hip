// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4_f64), gfx950.
//
// One kernel serves every dense FP64 contraction of the RI G0W0 path:
//   AO->MO half transforms ((P|mu nu) . C), the Casida SYRK (B^T B scaled by
//   sqrt(de)), w_s = B (X+Y), the self-energy products w_s^T (P|p i), the
//   imaginary-axis chi0 = X diag(s(iw)) X^T batched over frequencies,
//   chi(iw) (P|p m) with a fused column-dot epilogue, and the Hartree /
//   exchange products of the RI-HF.
//
// What bounds it: the matrix cores (one 16x16x4 MFMA takes 64 cycles of a
// SIMD), so everything else only has to stay out of their way.
//   * A workgroup of WM x WN wave64s owns a BM x BN tile of C and walks K in
//     slabs of BK = 16 through LDS, the next slab's global loads in flight
//     during the MFMAs of the current one. What keeps the matrix cores busy is
//     other workgroups on the same CU: their MFMAs run under this one's
//     barriers, LDS writes and epilogue. 128x128 tiles (accumulators of 128
//     registers) fit twice, with two LDS buffers and one barrier per slab;
//     smaller tiles take one buffer and two barriers and fit three or four
//     times (128x80 of long K: 46 -> 58 TFLOP/s with three instead of two).
//     A wave issues its MFMAs at raised priority (128-wide tiles: 64 -> 67
//     TFLOP/s at 8192 x 8192 x 4096; the copy-bound narrow tiles lose 5 %).
//   * Global loads are pairs of doubles (16 bytes a lane) along the operand's
//     contiguous dimension. Rows past the edge read the last row again (their
//     results are not stored), so only a last slab that is cut by K tests its
//     elements, and it reads zeros there.
//   * A wave whose part of the tile lies past the edge or above the diagonal of
//     a symmetric update leaves the matrix cores to the others.
//   * With fewer tiles than the GPU's slots, or a last round of workgroups that
//     would be mostly empty, the K range of that round's tiles is split
//     (split_plan): their partial products go to a workspace and
//     gemm_f64_reduce_kernel sums them in order and applies the epilogue. The
//     whole rounds before it run as they are, so the workspace holds two
//     rounds' tiles at most (128 MiB), whatever the product's size.
//
// Fragment layout of v_mfma_f64_16x16x4_f64 (checked on gfx950): operand "a"
// lane l = a[i = l & 15][k = l >> 4], operand "b" lane l = b[k = l >> 4][j = l & 15],
// result lane l register r = d[i = (l >> 4) + 4 r][j = l & 15]. The kernel
// feeds a = B^T and b = A^T so that d[i][j] = C(m = j, n = i): the 16 lanes of
// a row group hold 16 consecutive rows m of one column of the column-major C
// and every store is a 128-byte contiguous segment.
#include "mgw_internal.h"
#include "tile_order.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

namespace mgw {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
// two doubles at an address that is only 8-byte aligned (odd leading
// dimensions): global memory takes 16-byte accesses at any dword address
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int BK = 16;         // k per slab
// LDS row length of a tile of b rows (columns): consecutive k start 144 bytes
// apart modulo the 256 bytes of the banks, so that neither the 4 k of a
// fragment read nor the 8 pairs of k that a transposing store writes share
// banks; even, so that pairs stay 16-byte aligned
constexpr int lds_row(int b) { return b + (b % 32 == 0 ? 18 : 34); }
constexpr int GROUP_M = 8;     // tile rows per group of the grouped ordering

struct GemmDev {
  int M, N, K;
  const double* A; int64_t lda, strideA;
  const double* B; int64_t ldb, strideB;
  double* C; int64_t ldc, strideC;
  const double* kscale; int64_t strideK;
  const double* rowscale;
  const double* colscale;
  const double* diag_add; int64_t strideDiag;
  double alpha, beta;
  int lower_only;
  int no_mirror;       // lower_only: leave the strict upper triangle untouched
  int upper_zero;      // lower_only: write zeros above the diagonal instead of the mirror
  int tri_a;           // A (not transposed) is lower triangular, zeros stored above the diagonal
  int batch_outer;     // walk the tiles of one batch entry before the next
  int tiles_m, tiles_n;
  unsigned tiles, batch;      // tiles of one batch entry
  // the tiles (over all batch entries) behind the first `whole` take `splits`
  // workgroups of kchunk (a multiple of BK) along K each
  unsigned whole, rest;
  int splits, kchunk;
  double* part;        // splits > 1: part[tile - whole][split][n - n0][m - m0], else null
  const double* dotB; int64_t lddot;
  double dot_cc, dot_cd;
  double* dotpart; int64_t strideDot;
  const double* dot_w; int64_t strideDotW;
};

// C(m, n) of the product: scales, diagonal and beta, the mirror or the zero
// above the diagonal
__device__ inline void store_result(const GemmDev& g, double* __restrict__ C, const double* __restrict__ dg, int m,
                                    int n, double acc) {
  double v = g.alpha * acc;
  if (g.rowscale) v *= g.rowscale[m];
  if (g.colscale) v *= g.colscale[n];
  if (dg && m == n) v += dg[m];
  const int64_t idx = m + (int64_t)n * g.ldc;
  if (g.beta != 0.0) v += g.beta * C[idx];
  C[idx] = v;
  if (g.lower_only && m > n && !g.no_mirror) C[n + (int64_t)m * g.ldc] = g.upper_zero ? 0.0 : v;
}

// First row and column of a tile: square tiles of a symmetric update walk the
// lower triangle, the others groups of GROUP_M tile rows.
template <int BM, int BN>
__device__ inline void tile_origin(const GemmDev& g, int tile, int& m0, int& n0) {
  int bm, bn;
  if (g.lower_only && BM == BN) {
    tri_grouped(tile, g.tiles_m, bm, bn);
  } else {
    const int per_group = GROUP_M * g.tiles_n;
    const int group = tile / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(g.tiles_m - first_m, GROUP_M);
    const int in_group = tile - group * per_group;
    bm = first_m + in_group % gsize;
    bn = in_group / gsize;
  }
  m0 = bm * BM;
  n0 = bn * BN;
}

// Tile and batch entry of the u-th tile over all batch entries: batch fastest
// when the entries share operands (the frequencies of one chi0 tile read the
// same panels), batch slowest when they do not.
__device__ inline void tile_of_unit(const GemmDev& g, unsigned u, int& tile, int& batch) {
  const unsigned d = g.batch_outer ? g.tiles : g.batch, q = u / d, r = u - q * d;
  batch = (int)(g.batch_outer ? q : r);
  tile = (int)(g.batch_outer ? r : q);
}

template <int BM, int BN, int WM, int WN, bool TA, bool TB, bool DOT, int KLASS>
__global__ void __launch_bounds__(64 * WM * WN, WM * WN > 4 ? WM * WN / 4 : BM * BN <= 128 * 64 ? 4 : BM * BN <= 128 * 96 ? 3 : 2)
gemm_f64_kernel(GemmDev g) {
  constexpr int NT = 64 * WM * WN;
  constexpr int TM = BM / WM;
  constexpr int TN = BN / WN;
  constexpr int FM = TM / 16;
  constexpr int FN = TN / 16;
  static_assert(TM % 16 == 0 && TN % 16 == 0, "wave tile");
  constexpr bool PRIO = BN >= 128;          // raised priority during the MFMAs
  constexpr int NBUF = BM * BN <= 128 * 96 ? 1 : 2;
  // pairs of doubles of a slab, and the walk of a thread over them: an
  // operand whose contiguous dimension is m (n) has BM / 2 pairs per k, one
  // whose contiguous dimension is k has BK / 2 per row
  constexpr int PA = BM * BK / 2, PB = BN * BK / 2;
  constexpr int LA = (PA + NT - 1) / NT, LB = (PB + NT - 1) / NT;
  constexpr int ACOLS = TA ? BK / 2 : BM / 2, BCOLS = TB ? BN / 2 : BK / 2;

  __shared__ __attribute__((aligned(16))) double As[NBUF][BK][lds_row(BM)];
  __shared__ __attribute__((aligned(16))) double Bs[NBUF][BK][lds_row(BN)];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave % WM;
  const int wn = wave / WM;

  // logical block: the whole tiles, then the K splits of the others, one split
  // of all of them before the next (they share its range of the panels)
  const bool in_split = blockIdx.x >= g.whole;
  const unsigned L = in_split ? xcd_logical32(blockIdx.x - g.whole, g.rest * g.splits) : xcd_logical32(blockIdx.x, g.whole);
  const int split = in_split ? (int)(L / g.rest) : 0;
  const unsigned unit = in_split ? g.whole + L % g.rest : L;
  int tile, batch, m0, n0;
  tile_of_unit(g, unit, tile, batch);
  tile_origin<BM, BN>(g, tile, m0, n0);
  // symmetric rank-k update: tiles strictly above the diagonal have nothing to do
  if (g.lower_only && m0 + BM - 1 < n0) return;

  const double* __restrict__ A = g.A + (int64_t)batch * g.strideA;
  const double* __restrict__ B = g.B + (int64_t)batch * g.strideB;
  const double* __restrict__ ks = g.kscale ? g.kscale + (int64_t)batch * g.strideK : nullptr;

  // K range: a lower-triangular A has no terms beyond the tile's last row
  const int kall = g.tri_a ? min(g.K, m0 + BM) : g.K;
  const int kb = split * g.kchunk;
  const int ke = in_split ? min(kall, kb + g.kchunk) : kall;
  const int nslab = ke > kb ? (ke - kb + BK - 1) / BK : 0;

  // this thread's pair i of the A slab: column c of ACOLS, row r + i * NT / ACOLS
  const int ac = tid % ACOLS, ar = tid / ACOLS;
  const int bc = tid % BCOLS, br = tid / BCOLS;
  constexpr int AR = NT / ACOLS, BR = NT / BCOLS;
  static_assert(NT % ACOLS == 0 && NT % BCOLS == 0, "walk");
  // pairs past the edge of an operand read its last row again: the element
  // distance of a pair along m (n) is then 0
  const bool full = m0 + BM <= g.M && n0 + BN <= g.N;
  const int am = min(m0 + 2 * ac, g.M - 1), bnn = min(n0 + 2 * bc, g.N - 1);
  const int a2 = m0 + 2 * ac + 1 < g.M ? 1 : 0, b2 = n0 + 2 * bc + 1 < g.N ? 1 : 0;
  // running pointers to this thread's first pair of the next slab
  const double* __restrict__ pa =
      TA ? A + kb + 2 * ac + (int64_t)(m0 + ar) * g.lda : A + am + (int64_t)(kb + ar) * g.lda;
  const double* __restrict__ pb =
      TB ? B + bnn + (int64_t)(kb + br) * g.ldb : B + kb + 2 * bc + (int64_t)(n0 + br) * g.ldb;
  const int64_t aslab = TA ? BK : BK * g.lda, bslab = TB ? BK * g.ldb : BK;
  const int64_t astep = AR * g.lda, bstep = BR * g.ldb;

  // the slab's values on their way from memory to LDS; the scales of k are
  // applied there, so that no load is waited for before the MFMAs it runs under
  d2 ra[LA], rb[LB], rk[LB];
  auto load_slab = [&](int k0) __attribute__((always_inline)) {
    if (k0 + BK <= ke && full) {
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        if (PA % NT != 0 && tid + i * NT >= PA) break;
        ra[i] = *reinterpret_cast<const d2u*>(pa + i * astep);
      }
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        if (PB % NT != 0 && tid + i * NT >= PB) break;
        rb[i] = *reinterpret_cast<const d2u*>(pb + i * bstep);
      }
      if (ks) {
#pragma unroll
        for (int i = 0; i < LB; ++i) {
          if (TB) rk[i] = d2{ks[k0 + br + i * BR], 0.0};
          else rk[i] = d2{ks[k0 + 2 * bc], ks[k0 + 2 * bc + 1]};
        }
      }
    } else if (k0 + BK <= ke) {
      // a tile at the edge
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        if (PA % NT != 0 && tid + i * NT >= PA) break;
        if (TA) {
          ra[i] = *reinterpret_cast<const d2u*>(A + k0 + 2 * ac + (int64_t)min(m0 + ar + i * AR, g.M - 1) * g.lda);
        } else {
          const double* __restrict__ q = pa + i * astep;
          ra[i] = d2{q[0], q[a2]};
        }
      }
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        if (PB % NT != 0 && tid + i * NT >= PB) break;
        if (TB) {
          const double* __restrict__ q = pb + i * bstep;
          rb[i] = d2{q[0], q[b2]};
          if (ks) rk[i] = d2{ks[k0 + br + i * BR], 0.0};
        } else {
          rb[i] = *reinterpret_cast<const d2u*>(B + k0 + 2 * bc + (int64_t)min(n0 + br + i * BR, g.N - 1) * g.ldb);
          if (ks) rk[i] = d2{ks[k0 + 2 * bc], ks[k0 + 2 * bc + 1]};
        }
      }
    } else {
      // the slab cut by the end of K: zeros past it, in both operands
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        const int r = ar + i * AR;
        if (PA % NT != 0 && tid + i * NT >= PA) break;
        ra[i] = d2{0.0, 0.0};
        if (TA) {
          const int k = k0 + 2 * ac;
          const double* __restrict__ q = A + k + (int64_t)min(m0 + r, g.M - 1) * g.lda;
          if (k < ke) ra[i][0] = q[0];
          if (k + 1 < ke) ra[i][1] = q[1];
        } else if (k0 + r < ke) {
          const double* __restrict__ q = pa + i * astep;
          ra[i] = d2{q[0], q[a2]};
        }
      }
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int r = br + i * BR;
        if (PB % NT != 0 && tid + i * NT >= PB) break;
        rb[i] = d2{0.0, 0.0};
        rk[i] = d2{0.0, 0.0};
        if (TB) {
          if (k0 + r < ke) {
            const double* __restrict__ q = pb + i * bstep;
            rb[i] = d2{q[0], q[b2]};
            if (ks) rk[i][0] = ks[k0 + r];
          }
        } else {
          const int k = k0 + 2 * bc;
          const double* __restrict__ q = B + k + (int64_t)min(n0 + r, g.N - 1) * g.ldb;
          if (k < ke) {
            rb[i][0] = q[0];
            if (ks) rk[i][0] = ks[k];
          }
          if (k + 1 < ke) {
            rb[i][1] = q[1];
            if (ks) rk[i][1] = ks[k + 1];
          }
        }
      }
    }
    pa += aslab;
    pb += bslab;
  };
  auto store_slab = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int r = ar + i * AR;
      if (PA % NT != 0 && tid + i * NT >= PA) break;
      if (TA) {
        As[buf][2 * ac][r] = ra[i][0];
        As[buf][2 * ac + 1][r] = ra[i][1];
      } else {
        *reinterpret_cast<d2*>(&As[buf][r][2 * ac]) = ra[i];
      }
    }
    if (ks) {
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        rb[i][0] *= rk[i][0];
        rb[i][1] *= TB ? rk[i][0] : rk[i][1];
      }
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int r = br + i * BR;
      if (PB % NT != 0 && tid + i * NT >= PB) break;
      if (TB) {
        *reinterpret_cast<d2*>(&Bs[buf][r][2 * bc]) = rb[i];
      } else {
        Bs[buf][2 * bc][r] = rb[i][0];
        Bs[buf][2 * bc + 1][r] = rb[i][1];
      }
    }
  };

  d4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

  // a wave whose tile lies past the edge or above the diagonal of a symmetric
  // update only helps to load
  const int mw = m0 + wm * TM, nw = n0 + wn * TN;
  const bool active = __builtin_amdgcn_readfirstlane(mw < g.M && nw < g.N && (!g.lower_only || mw + TM - 1 >= nw));

  const int fr = lane & 15;
  const int fk = lane >> 4;
  auto compute = [&](int buf) __attribute__((always_inline)) {
    if (!active) return;
    if (PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k4 = 0; k4 < BK / 4; ++k4) {
      double af[FM], bf[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) af[i] = As[buf][k4 * 4 + fk][wm * TM + i * 16 + fr];
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[j] = Bs[buf][k4 * 4 + fk][wn * TN + j * 16 + fr];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j], af[i], acc[i][j], 0, 0, 0);
    }
    if (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  if (nslab > 0) {
    load_slab(kb);
    if constexpr (NBUF == 2) {
      store_slab(0);
      __syncthreads();
      for (int s = 0; s < nslab; ++s) {
        if (s + 1 < nslab) load_slab(kb + (s + 1) * BK);
        compute(s & 1);
        if (s + 1 < nslab) store_slab((s & 1) ^ 1);
        __syncthreads();
      }
    } else {
      for (int s = 0; s < nslab; ++s) {
        store_slab(0);
        __syncthreads();
        if (s + 1 < nslab) load_slab(kb + (s + 1) * BK);
        compute(0);
        __syncthreads();
      }
    }
  }

  // ------------------------------------------------------------ epilogue
  if constexpr (DOT) {
    // Column dots of this row block: sum_m C(m,n) (cc C(m,n) + cd D(m,n)),
    // or sum_m w(m) C(m,n)^2 without D (w = 1 without row weights).
    __shared__ double red[WM][BN];
    const double* __restrict__ D = g.dotB ? g.dotB + (int64_t)batch * g.strideB : nullptr;  // batched as B
    const double* __restrict__ W = g.dot_w ? g.dot_w + (int64_t)batch * g.strideDotW : nullptr;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      // the loads of a column group go out together: no bounds check around
      // each, but indices held to the last row and column
      double dv[4][FM], wv[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int m = min(m0 + wm * TM + i * 16 + fr, g.M - 1);
        wv[i] = W ? W[m] : 1.0;
        if (D) {
#pragma unroll
          for (int r = 0; r < 4; ++r) dv[r][i] = D[m + (int64_t)min(n0 + wn * TN + j * 16 + fk + 4 * r, g.N - 1) * g.lddot];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int nl = wn * TN + j * 16 + fk + 4 * r;
        double part = 0.0;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const double c = g.alpha * acc[i][j][r];
          if (m0 + wm * TM + i * 16 + fr < g.M) part += D ? c * (g.dot_cc * c + g.dot_cd * dv[r][i]) : wv[i] * c * c;
        }
        part += __shfl_xor(part, 8, 16);
        part += __shfl_xor(part, 4, 16);
        part += __shfl_xor(part, 2, 16);
        part += __shfl_xor(part, 1, 16);
        if (fr == 0) red[wm][nl] = part;
      }
    }
    __syncthreads();
    double* __restrict__ out = g.dotpart + (int64_t)batch * g.strideDot;
    for (int nl = tid; nl < BN; nl += NT) {
      const int n = n0 + nl;
      if (n < g.N) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < WM; ++w) sum += red[w][nl];
        out[(int64_t)(m0 / BM) * g.N + n] = sum;
      }
    }
    return;
  }

  double* __restrict__ C = g.C + (int64_t)batch * g.strideC;
  const double* __restrict__ dg = g.diag_add ? g.diag_add + (int64_t)batch * g.strideDiag : nullptr;
  double* __restrict__ P =
      in_split ? g.part + ((int64_t)(unit - g.whole) * g.splits + split) * (BM * BN) - (m0 + (int64_t)n0 * BM) : nullptr;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + wm * TM + i * 16 + fr;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + wn * TN + j * 16 + fk + 4 * r;
        if (m >= g.M || n >= g.N) continue;
        if (g.lower_only && m < n) continue;
        if (in_split) P[m + (int64_t)n * BM] = acc[i][j][r];
        else store_result(g, C, dg, m, n, acc[i][j][r]);
      }
    }
  }
}

// Sum of the K splits in order, then the epilogue. Memory-bound: a thread owns
// one (m, n) of one tile, consecutive threads consecutive m.
template <int B>
__global__ void __launch_bounds__(256) gemm_f64_reduce_kernel(GemmDev g) {
  int tile, batch, m0, n0;
  tile_of_unit(g, g.whole + blockIdx.y, tile, batch);
  tile_origin<B, B>(g, tile, m0, n0);
  const int e = blockIdx.x * 256 + threadIdx.x;
  const int m = m0 + e % B, n = n0 + e / B;
  if (m >= g.M || n >= g.N || (g.lower_only && m < n)) return;
  const double* __restrict__ p = g.part + (int64_t)blockIdx.y * g.splits * (B * B) + e;
  double s = 0.0;
  for (int q = 0; q < g.splits; ++q) s += p[(int64_t)q * (B * B)];
  store_result(g, g.C + (int64_t)batch * g.strideC,
               g.diag_add ? g.diag_add + (int64_t)batch * g.strideDiag : nullptr, m, n, s);
}

// Column tiles (NB): B not transposed only, and of each class the form of A that
// occurs; the other forms run under the symbol of GEMM_OTHER
constexpr bool narrow_form(int klass, bool ta) {
  return klass == MGW_KCLASS_GEMM_OTHER || klass == MGW_KCLASS_GEMM_SIGMA ? klass == MGW_KCLASS_GEMM_OTHER || ta : !ta;
}

template <int BM, int BN, int WM, int WN, bool DOT, int KLASS, bool NB = false>
int launch_cfg(const GemmF64& h, hipStream_t stream, int splits = 1, int64_t whole = 0) {
  GemmDev g;
  g.M = h.M; g.N = h.N; g.K = h.K;
  g.A = h.A; g.lda = h.lda; g.strideA = h.strideA;
  g.B = h.B; g.ldb = h.ldb; g.strideB = h.strideB;
  g.C = h.C; g.ldc = h.ldc; g.strideC = h.strideC;
  g.kscale = h.kscale; g.strideK = h.strideK;
  g.rowscale = h.rowscale; g.colscale = h.colscale;
  g.diag_add = h.diag_add; g.strideDiag = h.strideDiag;
  g.alpha = h.alpha; g.beta = h.beta;
  g.lower_only = h.lower_only ? 1 : 0;
  g.no_mirror = h.no_mirror ? 1 : 0;
  g.upper_zero = h.upper_zero ? 1 : 0;
  g.tri_a = h.tri_a ? 1 : 0;
  g.batch_outer = h.batch_outer ? 1 : 0;
  g.tiles_m = (h.M + BM - 1) / BM;
  g.tiles_n = (h.N + BN - 1) / BN;
  g.batch = (unsigned)h.batch;
  g.dotB = h.dotB; g.lddot = h.lddot; g.dotpart = h.dotpart; g.strideDot = h.strideDot;
  g.dot_cc = h.dot_cc; g.dot_cd = h.dot_cd;
  g.dot_w = h.dot_w; g.strideDotW = h.strideDotW;
  // square-tile symmetric updates enumerate the lower triangle of tiles only;
  // other lower-only shapes launch the full grid and skip upper tiles
  const int64_t tiles = (h.lower_only && BM == BN) ? (int64_t)g.tiles_m * (g.tiles_m + 1) / 2
                                                   : (int64_t)g.tiles_m * g.tiles_n;
  const int64_t units = tiles * h.batch;
  MGW_REQUIRE(units < (1ll << 31), MGW_ERR_ARG, "gemm_f64: too many tiles");
  g.splits = splits;
  g.tiles = (unsigned)tiles;
  g.whole = (unsigned)(splits > 1 ? whole : units);
  g.rest = (unsigned)units - g.whole;
  g.kchunk = (int)(((h.K + (int64_t)splits - 1) / splits + BK - 1) / BK * BK);
  g.part = splits > 1 ? h.split_work : nullptr;
  MGW_REQUIRE(h.batch >= 1, MGW_ERR_ARG, "gemm_f64: batch out of range");
  dim3 grid(g.whole + g.rest * splits, 1, 1);
  dim3 block(64 * WM * WN, 1, 1);
  const int ta = h.transA ? 1 : 0, tb = h.transB ? 1 : 0;
#define MGW_GEMM_CASE(TA_, TB_)                                                                        \
  if constexpr (!NB || (!TB_ && narrow_form(KLASS, TA_)))                                              \
    if (ta == TA_ && tb == TB_)                                                                        \
      hipLaunchKernelGGL((gemm_f64_kernel<BM, BN, WM, WN, TA_, TB_, DOT, KLASS>), grid, block, 0,      \
                         stream, g);
  MGW_GEMM_CASE(0, 0)
  MGW_GEMM_CASE(0, 1)
  MGW_GEMM_CASE(1, 0)
  MGW_GEMM_CASE(1, 1)
#undef MGW_GEMM_CASE
  MGW_HIP(hipGetLastError());
  if constexpr (BM == BN && !DOT)
    if (splits > 1) {
      hipLaunchKernelGGL(gemm_f64_reduce_kernel<BM>, dim3(BM * BM / 256, g.rest), dim3(256), 0,
                         stream, g);
      MGW_HIP(hipGetLastError());
    }
  return MGW_OK;
}

}  // namespace

// Row blocks of the dot epilogue: 64x64 tiles, whose triangular K ranges stop
// closer to the diagonal and of which four share a CU (naux 1372, 6304 columns,
// 16 frequencies: 3.86 ms against 4.53 for 128x128 and 4.15 for 128x64).
int gemm_f64_dot_rowblocks(int M) { return (M + 63) / 64; }

// ------------------------------------------------------------------ autotuner
// Candidate tile configurations (all FP64 MFMA, BK = 16):
//   0: 256x128, 16 waves   1: 128x128, 8 waves   2: 128x128, 4 waves   3: 64x64, 4 waves
//      128 x 16 fn, 4 waves, for products of few columns
// The defaults (split_plan's 2 or 3; column_tiles' 0, 2 or 3) were measured on
// MI355X. With tuning on, the first product of a new (class, transposes, lower
// or few columns, log2 M/N/K bucket) times every candidate on
// the actual operands and keeps the fastest; the table can be persisted.
namespace {

constexpr int NCFG = 4;
constexpr int TUNE_COLUMNS = 2;    // products of few columns: candidate 0 is their column tiles
constexpr int TUNE_SPLIT = 4;      // products with a split K, of candidates of their own

struct TuneKey {
  int klass, ta, tb, lower, mb, nb, kb;   // lower: plus what tells candidate lists of one family apart
  bool operator<(const TuneKey& o) const {
    return std::tie(klass, ta, tb, lower, mb, nb, kb) < std::tie(o.klass, o.ta, o.tb, o.lower, o.mb, o.nb, o.kb);
  }
};

struct Tuner {
  std::mutex mu;
  std::map<TuneKey, int> table;
  int mode = 0;           // 0 off, 1 tune unseen shapes
  std::string file;       // persisted table (appended as entries are found)
  bool loaded = false;
};

Tuner& tuner() {
  static Tuner t;
  return t;
}

int log2_bucket(int64_t v) {
  int b = 0;
  while (v > 1) { v >>= 1; ++b; }
  return b;
}

void load_table(Tuner& t) {
  if (t.loaded) return;
  t.loaded = true;
  const char* f = std::getenv("MGW_TUNE_FILE");
  if (!f || !*f) return;
  t.file = f;
  FILE* fp = std::fopen(f, "r");
  if (!fp) return;
  TuneKey k;
  int cfg;
  while (std::fscanf(fp, "%d %d %d %d %d %d %d %d", &k.klass, &k.ta, &k.tb, &k.lower, &k.mb, &k.nb, &k.kb, &cfg) == 8)
    if (cfg >= 0 && cfg < 16) t.table[k] = cfg;   // each family checks its own candidate count
  std::fclose(fp);
}

template <int KLASS>
int launch_candidate(int cfg, const GemmF64& h, hipStream_t stream) {
  switch (cfg) {
    case 0: return launch_cfg<256, 128, 4, 4, false, KLASS>(h, stream);
    case 1: return launch_cfg<128, 128, 4, 2, false, KLASS>(h, stream);
    case 2: return launch_cfg<128, 128, 2, 2, false, KLASS>(h, stream);
    default: return launch_cfg<64, 64, 2, 2, false, KLASS>(h, stream);
  }
}

// Tiles of a product of few columns (the transforms, half transforms and
// self-energy products of a window of states, the blocks of a factorisation): 128
// rows by 16 fn columns (cfg 0), 64x64 (cfg 3) or 128x128 (cfg 2), whichever is
// estimated to take the least time; fn: the best of the column tiles.
//
// A round of workgroups, `share` per CU, takes (K + fixed) steps, each at the
// tile's rate; the last round costs 0.15 and a part for the workgroups it has, a
// lone one 0.33. Rates (TFLOP/s of the tile's area), fixed costs and these parts
// are fitted to the times of 965 products on random operands: both transforms and
// the half transform of 50 to 768 functions, 75 to 2688 auxiliary ones and 1 to 768
// states, self-energy and factorisation products, 65536 rows with K to 4096. Over
// them the estimate's choice takes 0.6 % more than the best tile on average and
// 18 % at most. By rows of 128 and the columns' fit alone, with 64x64 below 512
// workgroups, it was 15 % on average and up to 89 %: rows past the edge, few full
// rounds and a lone workgroup's latency count as much as columns. 64x64 tiles read
// their operands twice as often and end at 8 rounds (up to 19 % off beyond); 96
// columns pay for a long K (2064384 x 90 x 768: 5.9 ms, 6.3 on tiles of 48).
void column_tiles(const GemmF64& h, int* cfg, int* fn) {
  struct Tile {
    int cfg, bm, bn, share;
    double rate, fixed;
  };
  static constexpr Tile TILES[] = {{2, 128, 128, 2, 70.4, 126.0}, {3, 64, 64, 4, 63.9, 84.8},
                                   {0, 128, 16, 4, 43.0, 31.6}, {0, 128, 32, 4, 52.7, 43.0},
                                   {0, 128, 48, 4, 65.7, 78.9}, {0, 128, 64, 4, 66.2, 88.7},
                                   {0, 128, 80, 3, 68.9, 96.2}, {0, 128, 96, 3, 67.0, 95.0}};
  double best = 0.0, best_columns = 0.0;
  for (const Tile& t : TILES) {
    const int64_t wgs = (int64_t)((h.M + t.bm - 1) / t.bm) * ((h.N + t.bn - 1) / t.bn) * h.batch;
    const int64_t slots = 256 * t.share, full = wgs / slots;
    if (t.cfg == 3 && full >= 8) continue;
    const double part = (double)(wgs % slots) / slots;
    const double rounds = full == 0 ? 0.33 + 0.67 * part : full + (part > 0.0 ? 0.15 + 0.85 * part : 0.0);
    const double cost = (double)t.bm * t.bn * slots / t.rate * (h.K + t.fixed) * rounds;
    if (best == 0.0 || cost < best) {
      best = cost;
      *cfg = t.cfg;
    }
    if (t.cfg == 0 && (best_columns == 0.0 || cost < best_columns)) {
      best_columns = cost;
      *fn = t.bn / 16;
    }
  }
}

template <int KLASS>
int launch_narrow(int fn, const GemmF64& h, hipStream_t stream) {
  switch (fn) {
    case 1: return launch_cfg<128, 16, 4, 1, false, KLASS, true>(h, stream);
    case 2: return launch_cfg<128, 32, 4, 1, false, KLASS, true>(h, stream);
    case 3: return launch_cfg<128, 48, 4, 1, false, KLASS, true>(h, stream);
    case 4: return launch_cfg<128, 64, 2, 2, false, KLASS, true>(h, stream);
    case 5: return launch_cfg<128, 80, 4, 1, false, KLASS, true>(h, stream);
    default: return launch_cfg<128, 96, 2, 2, false, KLASS, true>(h, stream);
  }
}

// fn > 0: cfg 0 is the column tiles of 16 fn. Of the classes, only the forms that occur have
// kernels of their own there (narrow_form).
int launch_by_class(int cfg, int fn, const GemmF64& h, hipStream_t stream) {
  if (fn > 0 && cfg == 0) {
    if (narrow_form(h.klass, h.transA)) {
      switch (h.klass) {
        case MGW_KCLASS_GEMM_AO2MO: return launch_narrow<MGW_KCLASS_GEMM_AO2MO>(fn, h, stream);
        case MGW_KCLASS_GEMM_CASIDA: return launch_narrow<MGW_KCLASS_GEMM_CASIDA>(fn, h, stream);
        case MGW_KCLASS_GEMM_SIGMA: return launch_narrow<MGW_KCLASS_GEMM_SIGMA>(fn, h, stream);
        case MGW_KCLASS_CHOLESKY: return launch_narrow<MGW_KCLASS_CHOLESKY>(fn, h, stream);
      }
    }
    return launch_narrow<MGW_KCLASS_GEMM_OTHER>(fn, h, stream);
  }
  switch (h.klass) {
    case MGW_KCLASS_GEMM_AO2MO: return launch_candidate<MGW_KCLASS_GEMM_AO2MO>(cfg, h, stream);
    case MGW_KCLASS_GEMM_CASIDA: return launch_candidate<MGW_KCLASS_GEMM_CASIDA>(cfg, h, stream);
    case MGW_KCLASS_GEMM_SIGMA: return launch_candidate<MGW_KCLASS_GEMM_SIGMA>(cfg, h, stream);
    case MGW_KCLASS_GEMM_CHI0: return launch_candidate<MGW_KCLASS_GEMM_CHI0>(cfg, h, stream);
    case MGW_KCLASS_CHOLESKY: return launch_candidate<MGW_KCLASS_CHOLESKY>(cfg, h, stream);
    default: return launch_candidate<MGW_KCLASS_GEMM_OTHER>(cfg, h, stream);
  }
}

int64_t tile_count(int M, int N, int batch, bool lower, int b) {
  const int64_t tm = (M + b - 1) / b, tn = (N + b - 1) / b;
  return (lower ? tm * (tm + 1) / 2 : tm * tn) * batch;
}

// How a plain product runs on b x b tiles (128 or 64): the first `whole` tiles
// by one workgroup each, the others by `splits` workgroups along K.
struct SplitPlan {
  int b, splits;
  int64_t whole, rest;
};

// The cheapest plan in cycles. Two workgroups of 128x128 or four of 64x64 share
// a CU's four SIMDs; a round of them lasts as long as its K range plus a fixed
// prologue and epilogue. A k step takes the cycles below by the workgroups that
// share a CU, so a last round that does not fill the slots is cheaper than a whole
// one. They are those of the parts of the peak that tiles reach together (128x128:
// 0.55 alone, 0.85 for two; 64x64: 0.25, 0.45, 0.6, 0.68), but for long-K symmetric
// products (may_split: chi0, exchange) fitted to 90 of them, of 420 to 1900 rows and
// 5 to 32 frequencies: there the 64-wide tiles are up to 22 % faster than those parts
// say (1036 rows, 32 frequencies: 8.5 ms, 10.5 on 128-wide ones), and the choice is
// 1.1 % from the best on average, 7 % at most; 8 and 41 % with the others. A single
// product whose operand does not stay in the 256 MiB last-level cache has the first
// ones: 64-wide tiles read it twice as often, and no other frequency's product does
// at the same time (exchange, 768 functions, 430080 rows: 16.9 ms a call, 17.4 on them).
//
// With `room` the K range of the last round's tiles may be split, into at most two
// rounds of workgroups (64x64: 64, 128x128: 128 MiB of partial products); those are
// written and read once at HBM's copy rate (1.9 KB per cycle). Equal costs take
// the smaller tiles, also when a product fits one of them: the larger one only
// adds idle waves.
SplitPlan split_plan(int M, int N, int K, int batch, bool lower, bool may_split, bool room) {
  struct Cost {
    double step128[3], step64[5], fixed128, fixed64;
  };
  static constexpr Cost PLAIN{{0.0, 256.0 / 0.55, 512.0 / 0.85},
                              {0.0, 64.0 / 0.25, 128.0 / 0.45, 192.0 / 0.6, 256.0 / 0.68}, 48.0, 48.0};
  static constexpr Cost LONG_K{{0.0, 390.0, 618.0}, {0.0, 160.0, 200.0, 262.0, 310.0}, 40.0, 30.0};
  const bool streamed = batch == 1 && 8.0 * std::max(M, N) * K > 256.0 * (1 << 20);
  const Cost& t = may_split && !streamed ? LONG_K : PLAIN;
  SplitPlan best{};
  double cost = 0.0;
  for (const int b : {64, 128}) {
    const double* step = b == 128 ? t.step128 : t.step64;
    const double fixed = b == 128 ? t.fixed128 : t.fixed64;
    const int share = b == 128 ? 2 : 4, slots = 256 * share;
    const int64_t tiles = tile_count(M, N, batch, lower, b);
    const int64_t rest = tiles % slots, whole = tiles - rest;
    const double full = (K + fixed) * (double)(whole / slots) * step[share];
    // 8 bytes of a partial product written and read, cycles per split
    const double traffic = 16.0 * M * (double)N * batch * (lower ? 0.5 : 1.0) * rest / tiles / 1900.0;
    for (int s = 1; s == 1 || (may_split && room && rest > 0 && K / s >= 64 && s * rest <= 2 * slots); ++s) {
      const int64_t wgs = s * rest;
      double c = full + ((double)K / s + fixed) *
                            ((double)(wgs / slots) * step[share] + step[(wgs % slots + 255) / 256]);
      if (s > 1) c += 7000.0 + s * traffic;
      else if (may_split && room) c *= 0.95;      // a split has to gain one part in twenty
      if (best.b == 0 || c < cost) {
        cost = c;
        best = SplitPlan{b, s, s > 1 ? whole : tiles, s > 1 ? rest : 0};
      }
    }
  }
  return best;
}

template <int KLASS>
int launch_split_cfg(const SplitPlan& p, int cfg, const GemmF64& h, hipStream_t stream) {
  if (p.b == 64) return launch_cfg<64, 64, 2, 2, false, KLASS>(h, stream, p.splits, p.whole);
  if (cfg == 0) return launch_cfg<128, 128, 2, 2, false, KLASS>(h, stream, p.splits, p.whole);
  return launch_cfg<128, 128, 4, 2, false, KLASS>(h, stream, p.splits, p.whole);
}

// The tuner may pick the waves of a 128-wide tile (0: four, 1: eight), not the
// tile, which decides what is split.
int launch_split(const SplitPlan& p, const GemmF64& h, hipStream_t stream) {
  MGW_REQUIRE(!h.dotpart && !h.no_tune && h.beta == 0.0, MGW_ERR_ARG, "gemm_f64: a split K needs a plain output");
  auto launch = [&](int cfg) {
    return h.klass == MGW_KCLASS_GEMM_CHI0 ? launch_split_cfg<MGW_KCLASS_GEMM_CHI0>(p, cfg, h, stream)
                                           : launch_split_cfg<MGW_KCLASS_GEMM_OTHER>(p, cfg, h, stream);
  };
  if (p.b == 64) return launch(0);
  return autotune_select(h.klass, h.transA ? 1 : 0, h.transB ? 1 : 0, log2_bucket(h.M), log2_bucket(h.N),
                         log2_bucket((int64_t)h.K * h.batch), 2, 0, launch, stream, TUNE_SPLIT + (h.lower_only ? 1 : 0));
}

int tune(const GemmF64& h, int fn, hipStream_t stream, int* best) {
  hipEvent_t a, b;
  MGW_HIP(hipEventCreate(&a));
  MGW_HIP(hipEventCreate(&b));
  float best_ms = 1e30f;
  *best = -1;
  for (int cfg = 0; cfg < NCFG; ++cfg) {
    MGW_HIP(hipEventRecord(a, stream));
    MGW_TRY(launch_by_class(cfg, fn, h, stream));
    MGW_HIP(hipEventRecord(b, stream));
    MGW_HIP(hipEventSynchronize(b));
    float ms = 0.0f;
    MGW_HIP(hipEventElapsedTime(&ms, a, b));
    if (ms < best_ms) { best_ms = ms; *best = cfg; }
  }
  MGW_HIP(hipEventDestroy(a));
  MGW_HIP(hipEventDestroy(b));
  return MGW_OK;
}

}  // namespace

size_t gemm_f64_split_doubles(int M, int N, int K, int batch, bool lower) {
  const SplitPlan p = split_plan(M, N, K, batch, lower, true, true);
  return p.splits > 1 ? (size_t)p.rest * p.splits * p.b * p.b : 0;
}

int gemm_autotune_mode(int mode) {
  Tuner& t = tuner();
  std::lock_guard<std::mutex> lk(t.mu);
  load_table(t);
  const int old = t.mode;
  if (mode >= 0) t.mode = mode;
  return old;
}

int autotune_select(int family, int ns, int h, int mb, int nb, int kb, int ncand, int fallback,
                    const std::function<int(int)>& launch, hipStream_t stream, int list) {
  Tuner& t = tuner();
  const TuneKey key{family, ns, h, list, mb, nb, kb};
  int choice = fallback;
  bool need_tune = false;
  {
    std::lock_guard<std::mutex> lk(t.mu);
    load_table(t);
    auto it = t.table.find(key);
    if (it != t.table.end() && it->second < ncand) choice = it->second;
    else need_tune = t.mode == 1;
  }
  if (!need_tune) return launch(choice);
  hipEvent_t a, b;
  MGW_HIP(hipEventCreate(&a));
  MGW_HIP(hipEventCreate(&b));
  // two rounds over the candidates, the best time of each (other streams of
  // the device may run meanwhile); another candidate replaces the fallback
  // only if it is at least 3 % faster
  std::vector<float> ms(ncand, 1e30f);
  auto time_all = [&]() -> int {
    for (int round = 0; round < 2; ++round)
      for (int cand = 0; cand < ncand; ++cand) {
        MGW_HIP(hipEventRecord(a, stream));
        MGW_TRY(launch(cand));
        MGW_HIP(hipEventRecord(b, stream));
        MGW_HIP(hipEventSynchronize(b));
        float e = 0.0f;
        MGW_HIP(hipEventElapsedTime(&e, a, b));
        ms[cand] = std::min(ms[cand], e);
      }
    return MGW_OK;
  };
  const int rc = time_all();
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  MGW_TRY(rc);
  int best = fallback;
  for (int cand = 0; cand < ncand; ++cand)
    if (ms[cand] < ms[best] && ms[cand] < 0.97f * ms[fallback]) best = cand;
  std::lock_guard<std::mutex> lk(t.mu);
  if (!t.table.emplace(key, best).second) return MGW_OK;   // another stream tuned it meanwhile
  if (!t.file.empty()) {
    if (FILE* fp = std::fopen(t.file.c_str(), "a")) {
      std::fprintf(fp, "%d %d %d %d %d %d %d %d\n", key.klass, key.ta, key.tb, key.lower, key.mb, key.nb, key.kb,
                   best);
      std::fclose(fp);
    }
  }
  return MGW_OK;   // every candidate wrote the same result
}

int gemm_f64(const GemmF64& h, hipStream_t stream) {
  if (h.M <= 0 || h.N <= 0 || h.batch <= 0) return MGW_OK;
  // MGW_BF16X6 and MGW_FP16X3 split only the chi0 and imaginary-axis
  // self-energy operands (chi0_split.hip, wb_split.hip); every other product
  // of those modes stays FP64
  MGW_REQUIRE(h.dot_w == nullptr || h.precision == MGW_FP64, MGW_ERR_ARG, "gemm_f64: row-weighted dots are FP64 only");
  if (h.precision == MGW_FP32 || h.precision == MGW_BF16X3) return gemm_lowp(h, h.precision, stream);
  // FP16x3 products need the operand maxima; without them the product stays FP64
  if (h.precision == MGW_FP16X3 && h.amax && h.bmax) return gemm_lowp(h, h.precision, stream);
  MGW_REQUIRE(h.K >= 0, MGW_ERR_ARG, "gemm_f64: negative K");
  MGW_REQUIRE(!h.lower_only || h.M == h.N, MGW_ERR_ARG, "gemm_f64: lower_only needs M == N");
  MGW_REQUIRE(h.dotpart == nullptr || !h.lower_only, MGW_ERR_ARG, "gemm_f64: dot epilogue needs a full tile grid");
  MGW_REQUIRE(!h.tri_a || (!h.transA && h.M == h.K), MGW_ERR_ARG,
              "gemm_f64: a triangular A must be square and not transposed");
  MGW_REQUIRE(h.dotpart != nullptr || h.C != nullptr, MGW_ERR_ARG, "gemm_f64: no output");
  if (h.dotpart) return launch_cfg<64, 64, 2, 2, true, MGW_KCLASS_GEMM_WB>(h, stream);
  const SplitPlan plan = split_plan(h.M, h.N, h.K, h.batch, h.lower_only, h.may_split, h.split_work != nullptr);
  if (plan.splits > 1) return launch_split(plan, h, stream);
  int cfg = plan.b == 64 ? 3 : 2, fn = 0;
  if (!h.transB && !h.lower_only && h.N < 1024) column_tiles(h, &cfg, &fn);
  Tuner& t = tuner();
  const TuneKey key{h.klass, h.transA ? 1 : 0, h.transB ? 1 : 0, fn > 0 ? TUNE_COLUMNS : h.lower_only ? 1 : 0,
                    log2_bucket(h.M), log2_bucket(h.N), log2_bucket((int64_t)h.K * h.batch)};
  bool need_tune = false;
  {
    std::lock_guard<std::mutex> lk(t.mu);
    load_table(t);
    auto it = t.table.find(key);
    if (it != t.table.end() && it->second < NCFG) cfg = it->second;
    else need_tune = t.mode == 1 && h.beta == 0.0 && !h.no_tune;   // candidates overwrite C: only pure products
  }
  if (need_tune) {
    int best = cfg;
    MGW_TRY(tune(h, fn, stream, &best));
    std::lock_guard<std::mutex> lk(t.mu);
    t.table[key] = best;
    cfg = best;
    if (!t.file.empty()) {
      if (FILE* fp = std::fopen(t.file.c_str(), "a")) {
        std::fprintf(fp, "%d %d %d %d %d %d %d %d\n", key.klass, key.ta, key.tb, key.lower, key.mb, key.nb, key.kb,
                     best);
        std::fclose(fp);
      }
    }
  }
  return launch_by_class(cfg, fn, h, stream);
}

}  // namespace mgw
