// The hop of few sites: a workgroup's 8 waves take one direction each (gfx950).
//
// On a small lattice the gathering kernel (wc_hop.h) has less than a wave per
// SIMD and each wave waits for the loads of 8 directions one after another:
// 8^4 in FP64 took 11 us a hop, 10 of them latency.  Here a workgroup covers
// 64 (site, right-hand side) items with 512 threads, wave w handles direction
// w of all 64: the loads of all directions, of the epilogue's clover rows and
// operands are under way at once.  The half spinors of the 8 directions meet
// in LDS, where wave s < 4 adds them up for spin s in the gathering kernel's
// order, and the rows of the clover blocks are shared out the same way: the
// same bits.
#pragma once
#include "wc_hop.h"

namespace wck {

constexpr int kSplitItems = 64;
constexpr int kSplitThreads = 8 * kSplitItems;
// most items (site, right-hand side): the workgroups that the chip holds at
// once, one per CU in FP64 and two in FP32.  Up to there this form is 1.3-2
// times as fast as the gathering kernel with its best shape (8^4 FP64: hop 10.1
// -> 5.5 us, Mpc^dag Mpc 45.6 -> 31.8, M 18.8 -> 14.1; 16^4 FP32 12-real: 13.2 ->
// 7.1, 67 -> 44, 30 -> 20); beyond, the other one has waves enough to hide the
// loads and needs no LDS round trip (16^4 FP64: Mpc^dag Mpc 79 against 83 us,
// 24^3 x 48: 580 against 782).
template <typename R> constexpr long split_most() { return sizeof(R) == 8 ? 256 * kSplitItems : 512 * kSplitItems; }

// U h of direction (MU, FB) for the gathered spinor psi, link entries raw in u
template <typename R, int NL, int DAG, int MU, int FB>
__device__ __forceinline__ void split_dir(const HopLaunch &a, const int c[4], typename c2<R>::t u[9],
                                          const typename c2<R>::t psi[12], typename c2<R>::t ch[2][3]) {
  using C = typename c2<R>::t;
  constexpr int S = ((FB == 0) != (DAG != 0)) ? 1 : -1;
  prepare_link<R, NL>(a, MU, FB, c, u);
  C hs[2][3];
#pragma unroll
  for (int col = 0; col < 3; ++col)
    project<MU, S>(psi[col], psi[3 + col], psi[6 + col], psi[9 + col], hs[0][col], hs[1][col]);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      C t = cmul(u[3 * i + 0], hs[s][0]);
      t = cmadd(t, u[3 * i + 1], hs[s][1]);
      ch[s][i] = cmadd(t, u[3 * i + 2], hs[s][2]);
    }
}

// acc += direction DIR's part of spin w, from its upper spins c0, c1
template <typename C, int DAG, int DIR>
__device__ __forceinline__ void split_add(int w, const C c0, const C c1, C &acc) {
  constexpr int S = (((DIR & 1) == 0) != (DAG != 0)) ? 1 : -1;
  if (w == 0) {
    acc = cadd(acc, c0);
  } else if (w == 1) {
    acc = cadd(acc, c1);
  } else {
    C a2 = acc, a3 = acc;
    accum_lower<DIR / 2, S>(a2, a3, c0, c1);
    acc = w == 2 ? a2 : a3;
  }
}

// row i (0..5) of a packed Hermitian block: its diagonal entry and the five
// others in column order, as stored
template <typename R> struct CloverRow {
  R d;
  typename c2<R>::t e[5];
};
template <typename R>
__device__ __forceinline__ void row_load(const typename c2<R>::t *block, int i, CloverRow<R> &q) {
  q.d = ((const R *)(block + (long)(i >> 1) * kBlk))[i & 1];
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const int col = j < i ? j : j + 1;
    const int slot = col < i ? tri(i, col) : tri(col, i);
    q.e[j] = block[(long)slot * kBlk];
  }
}
// (A v)_i, summed as clov_mul6 does, v[col] at p[col * kSplitItems]
template <typename R>
__device__ __forceinline__ typename c2<R>::t row_mul(const CloverRow<R> &q, int i, const typename c2<R>::t *p) {
  using C = typename c2<R>::t;
  C acc = cscale(p[i * kSplitItems], q.d);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    if (j < i) acc = cmadd(acc, q.e[j], p[j * kSplitItems]);
    else acc = cmaddc(acc, q.e[j], p[(j + 1) * kSplitItems]);
  }
  return acc;
}

template <typename R, int NL, int DAG, int EPI>
__global__ __launch_bounds__(kSplitThreads, 2) void k_hop_split(const HopLaunch a) {
  using C = typename c2<R>::t;
  if (a.halt && *a.halt) return;
  constexpr int W = kSplitItems;
  const Geom &g = a.g;
  const int N = a.nrhs;
  __shared__ C part[8 * 6 * W];  // [direction][2 spins x 3 colours][item]
  __shared__ C vec[12 * W];      // [component][item]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t items = (uint32_t)g.Vh * (uint32_t)N;
  const uint32_t q0 = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * W + (uint32_t)lane;
  const bool live = q0 < items;
  const uint32_t q = live ? q0 : items - 1;
  const uint32_t h = N == 1 ? q : q / (uint32_t)N;
  const int r = (int)(q - h * (uint32_t)N);
  int c[4];
  half_coords(g, h, a.pout, c);
  const bool zb = a.open_bc && (c[3] == 0 || c[3] == g.L[3] - 1);

  // direction w: link and neighbour spinor
  C u[9], psi[12];
  {
    const uint32_t nb = hop_neighbour(g, h, c[0], c[1], c[2], c[3], w);
    const wc_rsrc in = make_rsrc(a.in, 12u * (uint32_t)g.Vh * (uint32_t)N * (uint32_t)sizeof(C));
    const uint32_t vo = ((uint32_t)aidx_site(nb, 12) * (uint32_t)N + (uint32_t)r) * (uint32_t)sizeof(C);
    const C *wl = (const C *)a.W + aidx(w * NL, h, 8 * NL);
#pragma unroll
    for (int e = 0; e < NL; ++e) u[e] = wl[e * kBlk];
#pragma unroll
    for (int k = 0; k < 12; ++k)
      psi[k] = bload<C>(in, vo, (uint32_t)k * (uint32_t)(kBlk * N) * (uint32_t)sizeof(C));
  }
  // waves 0..3, spin w: what its three components need in the epilogue
  const int ch = w >> 1, i0 = 3 * (w & 1);
  const C *blocks = (const C *)((EPI & EPI_CLOV) ? a.clov : a.diag_clov);
  constexpr bool kRows = (EPI & (EPI_CLOV | EPI_DIAG)) != 0;
  CloverRow<R> row[3];
  C y[3];
  if (w < 4) {
    if (kRows && blocks) {
      if ((EPI & EPI_CLOV) && a.clov_roff) blocks += a.clov_roff[r];
      const C *b = blocks + aidx(ch * 18, h, 36);
#pragma unroll
      for (int k = 0; k < 3; ++k) row_load(b, i0 + k, row[k]);
    }
    if (EPI & (EPI_DIAG | EPI_AXPY)) {
      const C *p = (const C *)a.y + aidx(3 * w, h, 12) * N + r;
#pragma unroll
      for (int k = 0; k < 3; ++k) y[k] = p[(long)k * kBlk * N];
    }
  }
  // wave 4 forms the inner product: its left vector lies where waves 0..3 have
  // their rows
  if ((EPI & EPI_DOT) && w == 4) {
    const C *p = (const C *)a.dotv + aidx_site(h, 12) * N + r;
#pragma unroll
    for (int k = 0; k < 12; ++k) row[k / 5].e[k % 5] = p[(long)k * kBlk * N];
  }
  {
    C x[2][3];
    switch (w) {
      case 0: split_dir<R, NL, DAG, 0, 0>(a, c, u, psi, x); break;
      case 1: split_dir<R, NL, DAG, 0, 1>(a, c, u, psi, x); break;
      case 2: split_dir<R, NL, DAG, 1, 0>(a, c, u, psi, x); break;
      case 3: split_dir<R, NL, DAG, 1, 1>(a, c, u, psi, x); break;
      case 4: split_dir<R, NL, DAG, 2, 0>(a, c, u, psi, x); break;
      case 5: split_dir<R, NL, DAG, 2, 1>(a, c, u, psi, x); break;
      case 6: split_dir<R, NL, DAG, 3, 0>(a, c, u, psi, x); break;
      default: split_dir<R, NL, DAG, 3, 1>(a, c, u, psi, x); break;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 3; ++i) part[(w * 6 + s * 3 + i) * W + lane] = x[s][i];
  }
  if ((EPI & EPI_DIAG) && w < 4)
#pragma unroll
    for (int i = 0; i < 3; ++i) vec[(3 * w + i) * W + lane] = y[i];
  __syncthreads();
  // the sums of spin w, direction by direction
  C acc[3];
  if (w < 4) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      acc[i] = cmk<C>(0, 0);
      const C *p = part + i * W + lane;
      split_add<C, DAG, 0>(w, p[0 * W], p[3 * W], acc[i]);
      split_add<C, DAG, 1>(w, p[6 * W], p[9 * W], acc[i]);
      split_add<C, DAG, 2>(w, p[12 * W], p[15 * W], acc[i]);
      split_add<C, DAG, 3>(w, p[18 * W], p[21 * W], acc[i]);
      split_add<C, DAG, 4>(w, p[24 * W], p[27 * W], acc[i]);
      split_add<C, DAG, 5>(w, p[30 * W], p[33 * W], acc[i]);
      split_add<C, DAG, 6>(w, p[36 * W], p[39 * W], acc[i]);
      split_add<C, DAG, 7>(w, p[42 * W], p[45 * W], acc[i]);
      if (zb) acc[i] = cmk<C>(0, 0);
    }
  }
  if (EPI & EPI_CLOV) {
    if (w < 4)
#pragma unroll
      for (int i = 0; i < 3; ++i) vec[(3 * w + i) * W + lane] = acc[i];
    __syncthreads();
    if (w < 4 && !zb) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        if (blocks)
          acc[i] = row_mul<R>(row[i], i0 + i, vec + 6 * ch * W + lane);
        else
          acc[i] = cscale(acc[i], (R)a.clov_scalar);
      }
    }
  }
  if (w < 4) {
    if (EPI & EPI_DIAG) {
      if (!zb) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const C d = blocks ? row_mul<R>(row[i], i0 + i, vec + 6 * ch * W + lane) : cscale(y[i], (R)a.diag);
          acc[i] = cadd(acc[i], d);
        }
      }
    } else if (EPI & EPI_AXPY) {
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] = csub(y[i], acc[i]);
    }
    if (live) {
      C *o = (C *)a.out + aidx(3 * w, h, 12) * N + r;
#pragma unroll
      for (int i = 0; i < 3; ++i) o[(long)i * kBlk * N] = acc[i];
    }
  }
  if (EPI & EPI_DOT) {
    // the item's product, its components in order; with one right-hand side
    // also the sum over the workgroup's 64-site block, in site order
    // (k_dot_blocks)
    __syncthreads();
    if (w < 4)
#pragma unroll
      for (int i = 0; i < 3; ++i) vec[(3 * w + i) * W + lane] = acc[i];
    __syncthreads();
    if (w == 4) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        const C v = vec[k * W + lane];
        const C d = row[k / 5].e[k % 5];
        s = fma((double)d.y, (double)v.y, fma((double)d.x, (double)v.x, s));
      }
      if (live) a.dots[(long)h * N + r] = s;
      if (N == 1 && a.dot_partials) {
        double *ds = (double *)part;
        ds[lane] = s;
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
          double t = 0.0;
#pragma unroll
          for (int i = 0; i < W; ++i) t += ds[i];
          a.dot_partials[h >> 6] = t;
        }
      }
    }
  }
}

template <typename R> bool split_applies(const HopLaunch &a) {
  if (!a.split || a.half_in || a.half_out || a.skip_t_faces) return false;
  return a.g.Vh * a.nrhs <= split_most<R>();
}

template <typename R, int NL, int DAG> static bool split_epi(const HopLaunch &a, unsigned grid, hipStream_t s) {
  switch (a.epi) {
#define WC_EPI(E)                                                      \
  case E:                                                              \
    k_hop_split<R, NL, DAG, E><<<grid, kSplitThreads, 0, s>>>(a);      \
    return true;
    WC_EPI(0)
    WC_EPI(EPI_CLOV)
    WC_EPI(EPI_DIAG)
    WC_EPI(EPI_AXPY)
    WC_EPI(EPI_CLOV | EPI_AXPY)
    WC_EPI(EPI_CLOV | EPI_AXPY | EPI_DOT)
    WC_EPI(EPI_AXPY | EPI_DOT)
#undef WC_EPI
    default: return false;
  }
}

template <typename R> bool hop_split(const HopLaunch &a, hipStream_t s) {
  const unsigned grid = (unsigned)((a.g.Vh * a.nrhs + kSplitItems - 1) / kSplitItems);
  if (a.nl == 9) return a.dag ? split_epi<R, 9, 1>(a, grid, s) : split_epi<R, 9, 0>(a, grid, s);
  return a.dag ? split_epi<R, 6, 1>(a, grid, s) : split_epi<R, 6, 0>(a, grid, s);
}

}  // namespace wck
