// The hop of many right-hand sides, marching in t (gfx950).
//
// What bounds the gathering kernel (wc_hop.h) with 12 right-hand sides is the
// fabric behind the L2s: an XCD's sites in flight and their neighbours (10 MB
// in FP64) are far beyond its 4 MB L2, so an input spinor is fetched 5-7
// times (24^3 x 48, FP64: 5.5 GB of reads against 1.15 GB compulsory; with the
// stores 7.5 TB/s, what the fabric gives).  Visiting the sites in another order, occupancy
// caps and cache hints changed that by 10 % at most.  Here a wave owns 64
// items (site of a t-slice, group of RB right-hand sides; 16 bytes a
// component in FP64 and FP32) and walks through t with them:
//   - a site's +-t neighbours have its own place h3 in their slices, and so
//     has one of its +-x neighbours: the wave loads a slice's own spinors
//     once, when they are the +t neighbours, and keeps them in LDS until they
//     have been the x and the -t neighbours.  8 gathers a site become 6, one
//     of them from HBM;
//   - the waves of an XCD own one compact patch of the slice (rows in blocks of
//     kMarchRows in y, XCDs along the order) and walk together, so the y, z and
//     other x neighbours were loaded by another wave one step before and are
//     often in L2 (24^3 x 48 FP64: reads 5.5 -> 3.1 GB, 3.6 fetches a spinor);
//   - the 6 x 12 loads of a step are issued up to a step ahead into registers
//     (512 a lane: one wave per SIMD), the links and clover blocks of the next
//     slice too.  A workgroup is one wave: nothing waits for other waves.
// Everything is added in the gathering kernel's order: the same bits.
//
// Measured against the gathering kernel (Meooe, 12 right-hand sides): FP64
// 24^3 x 48 826 -> 553 us, 16^3 x 32 156 -> 94 us; FP32 32^3 x 64 1078 -> 828 us
// (12-real links 1027 -> 769 us); also on the smallest lattices (8^4 FP64 14 ->
// 10 us: a step's loads are all under way at once, where the other kernel
// waits for each direction).  On large lattices the texture addresser (87 %
// busy, 24^3 x 48 FP64) and the fabric (7.0 TB/s of reads and stores) then bound
// it together; its waves wait for a tenth of their time, the other kernel's for
// half.
#pragma once
#include "wc_hop.h"

namespace wck {

constexpr int kMarchItems = 64;  // one wave, one workgroup
constexpr int kMarchSlots = 128;  // waves an XCD holds: one per SIMD of 32 CUs
constexpr int kMarchRows = 4;  // rows (y) of a block of the visiting order
// sites a wave's items can lie in (links and clover blocks in LDS: 13.8 KB
// beside 24.6 KB of spinors, four waves per CU)
template <typename R> constexpr int march_sites() { return sizeof(R) == 8 ? 8 : 16; }
template <typename R> constexpr int march_rb() { return 16 / (2 * (int)sizeof(R)); }  // right-hand sides per item

// loads of values that are read once
typedef double nt_d2 __attribute__((ext_vector_type(2)));
typedef float nt_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 load_once(const double2 *p) {
  return __builtin_bit_cast(double2, __builtin_nontemporal_load((const nt_d2 *)p));
}
__device__ __forceinline__ float2 load_once(const float2 *p) {
  return __builtin_bit_cast(float2, __builtin_nontemporal_load((const nt_f2 *)p));
}

// raw values of RB right-hand sides -> spinors
template <typename R, int RB>
__device__ __forceinline__ void march_unpack(const wc_v4i q[12], typename c2<R>::t psi[RB][12]) {
  using C = typename c2<R>::t;
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    const rhs_pack<C, RB> v = __builtin_bit_cast(rhs_pack<C, RB>, q[k]);
#pragma unroll
    for (int j = 0; j < RB; ++j) psi[j][k] = v.v[j];
  }
}

// acc += the direction's link (entry e at lw[((2 MU + FB) * 9 + e) * LS]) times
// the half spinors, with the lower spins rebuilt
template <typename R, int DAG, int MU, int FB, int RB>
__device__ __forceinline__ void march_mul(const typename c2<R>::t hs[RB][2][3], const typename c2<R>::t *lw,
                                          typename c2<R>::t acc[RB][12]) {
  using C = typename c2<R>::t;
  constexpr int S = ((FB == 0) != (DAG != 0)) ? 1 : -1;
  constexpr int LS = march_sites<R>();
  const C *u = lw + (2 * MU + FB) * 9 * LS;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const C u0 = u[(3 * i) * LS], u1 = u[(3 * i + 1) * LS], u2 = u[(3 * i + 2) * LS];
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      C ch[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        C t = cmul(u0, hs[j][s][0]);
        t = cmadd(t, u1, hs[j][s][1]);
        ch[s] = cmadd(t, u2, hs[j][s][2]);
      }
      acc[j][i] = cadd(acc[j][i], ch[0]);
      acc[j][3 + i] = cadd(acc[j][3 + i], ch[1]);
      accum_lower<MU, S>(acc[j][6 + i], acc[j][9 + i], ch[0], ch[1]);
    }
  }
  // The sums are made here: left to itself the compiler moves all eight
  // directions into the epilogue's branches, with all their operands live.
#pragma unroll
  for (int j = 0; j < RB; ++j)
#pragma unroll
    for (int k = 0; k < 12; ++k) asm volatile("" : "+v"(acc[j][k].x), "+v"(acc[j][k].y));
  __builtin_amdgcn_sched_barrier(0);
}

// the half spinors of colour col from the four spins' raw values
template <typename R, int DAG, int MU, int FB, int RB>
__device__ __forceinline__ void march_project(const wc_v4i q0, const wc_v4i q1, const wc_v4i q2, const wc_v4i q3, int col,
                                              typename c2<R>::t hs[RB][2][3]) {
  using C = typename c2<R>::t;
  constexpr int S = ((FB == 0) != (DAG != 0)) ? 1 : -1;
  const rhs_pack<C, RB> p0 = __builtin_bit_cast(rhs_pack<C, RB>, q0), p1 = __builtin_bit_cast(rhs_pack<C, RB>, q1),
                        p2 = __builtin_bit_cast(rhs_pack<C, RB>, q2), p3 = __builtin_bit_cast(rhs_pack<C, RB>, q3);
#pragma unroll
  for (int j = 0; j < RB; ++j) project<MU, S>(p0.v[j], p1.v[j], p2.v[j], p3.v[j], hs[j][0][col], hs[j][1][col]);
}

template <typename R, int DAG, int MU, int FB, int RB>
__device__ __forceinline__ void march_dir(const wc_v4i q[12], const typename c2<R>::t *lw,
                                          typename c2<R>::t acc[RB][12]) {
  using C = typename c2<R>::t;
  __builtin_amdgcn_sched_barrier(0);
  C hs[RB][2][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) march_project<R, DAG, MU, FB, RB>(q[c], q[3 + c], q[6 + c], q[9 + c], c, hs);
  march_mul<R, DAG, MU, FB, RB>(hs, lw, acc);
}

// Links, clover blocks and spinors of a wave in LDS: 38.4 KB, four waves per CU.
template <typename R, int NL, int DAG, int EPI>
__global__ __launch_bounds__(kMarchItems, 1) void k_hop_march(const HopLaunch a) {
  using C = typename c2<R>::t;
  if (a.halt && *a.halt) return;
  constexpr int W = kMarchItems, RB = march_rb<R>(), LS = march_sites<R>();
  constexpr int kPart = W / LS;                        // directions or slots the wave handles at once
  constexpr int kTasks = 8 / kPart;                    // directions of a lane
  constexpr int kClov = (36 + kPart - 1) / kPart;      // clover slots of a lane
  constexpr bool kHasClov = (EPI & (EPI_CLOV | EPI_DIAG)) != 0;
  const Geom &g = a.g;
  const int N = a.nrhs, G = (N + RB - 1) / RB;
  const int Lt = g.L[3], S3 = (int)(g.Vh / Lt), items = S3 * G;
  // XCD k gets the k-th eighth of the slice's tiles, all their t-segments
  const int ntiles = (items + W - 1) / W, tpx = (ntiles + 7) >> 3;
  const int ib = blockIdx.x >> 3, xcd = blockIdx.x & 7, seg = ib / tpx;
  const int tile = xcd * ntiles / 8 + (ib - seg * tpx);
  if (tile >= (xcd + 1) * ntiles / 8) return;
  const int t0 = seg * Lt / a.march_segs, t1 = (seg + 1) * Lt / a.march_segs;
  // site of the slice at place v of the visiting order: rows in blocks of
  // kMarchRows in y, so that the patch of an XCD is compact in y and z
  auto place = [&](int v) {
    const int row = v / g.Lxh, x = v - row * g.Lxh;
    const int per = kMarchRows * g.L[2], blk = row / per, r = row - blk * per;
    const int yb = min(kMarchRows, g.L[1] - blk * kMarchRows);
    const int z = r / yb, y = blk * kMarchRows + (r - z * yb);
    return (z * g.L[1] + y) * g.Lxh + x;
  };
  const int tid = threadIdx.x;
  const int j0 = tile * W, v0 = j0 / G, nsv = min((j0 + W - 1) / G, S3 - 1) - v0 + 1;  // the wave's sites
  // lanes beyond the last item repeat it; the last group of a site overlaps
  // its neighbour when RB does not divide N: the same bits are stored twice
  const int j = min(j0 + tid, items - 1), v = j / G, rb = min((j - v * G) * RB, N - RB);
  const int h3 = place(v);
  const int row = h3 / g.Lxh, xh = h3 - row * g.Lxh, cz = row / g.L[1], cy = row - cz * g.L[1];
  const int sy = g.Lxh, sz = g.Lxh * g.L[1];
  const int h_yp = cy == g.L[1] - 1 ? h3 - (g.L[1] - 1) * sy : h3 + sy;
  const int h_ym = cy == 0 ? h3 + (g.L[1] - 1) * sy : h3 - sy;
  const int h_zp = cz == g.L[2] - 1 ? h3 - (g.L[2] - 1) * sz : h3 + sz;
  const int h_zm = cz == 0 ? h3 + (g.L[2] - 1) * sz : h3 - sz;
  // x = 2 xh + b: b = 0 has its +x neighbour at its own place, b = 1 its -x
  // neighbour; the other one is the place before (b = 0) or after (b = 1)
  const int par = (cy + cz + a.pout) & 1;
  auto h_xo = [&](int t) {
    if ((par + t) & 1) return xh == g.Lxh - 1 ? h3 - xh : h3 + 1;
    return xh == 0 ? h3 + g.Lxh - 1 : h3 - 1;
  };
  const uint32_t fbytes = 12u * (uint32_t)g.Vh * (uint32_t)N * (uint32_t)sizeof(C);
  const wc_rsrc in = make_rsrc(a.in, fbytes);
  const uint32_t ks = (uint32_t)kBlk * (uint32_t)N * (uint32_t)sizeof(C);
  auto gather_of = [&](wc_rsrc f, int t, int h, wc_v4i q[12]) {
    const uint32_t vo = ((uint32_t)aidx_site((long)t * S3 + h, 12) * (uint32_t)N + (uint32_t)rb) * (uint32_t)sizeof(C);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 12; ++k) q[k] = __builtin_amdgcn_raw_buffer_load_b128(f, (int)vo, (int)((uint32_t)k * ks), 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto gather = [&](int t, int h, wc_v4i q[12]) { gather_of(in, t, h, q); };

  extern __shared__ __align__(16) char wc_dyn_lds[];
  wc_v4i *sp = (wc_v4i *)wc_dyn_lds;               // own spinors of two slices [2][12][W]
  C *lk = (C *)(wc_dyn_lds + 2 * 12 * W * 16);     // prepared links [dir * 9 + e][LS]
  C *cl = lk + 72 * LS;                            // clover blocks [36][LS]
  // A lane's share of a slice's links and blocks: the wave's site lsi,
  // directions ldir, ldir + kPart, ... and slots likewise.  Loaded raw a step
  // ahead (lu, lc), prepared into LDS when the step before is done.
  const void *blocks = (EPI & EPI_CLOV) ? a.clov : a.diag_clov;
  const C *cb = (const C *)(blocks ? blocks : a.W);  // no clover term: any values
  C lu[kTasks][NL], lc[kClov];
  const int lsi = tid & (LS - 1), ldir = tid / LS;
  const int lh = place(v0 + min(lsi, nsv - 1));
  int lc4[4];
  half_coords(g, lh, a.pout, lc4);  // in slice 0
  const int lxh = lc4[0] >> 1, lpar = lc4[0] & 1;
  auto link_load = [&](int t) {
    const long H = (long)t * S3 + lh;
    const C *p = (const C *)a.W + aidx(ldir * NL, H, 8 * NL);
#pragma unroll
    for (int w = 0; w < kTasks; ++w)
#pragma unroll
      for (int e = 0; e < NL; ++e) lu[w][e] = load_once(p + (w * kPart * NL + e) * kBlk);
    if (kHasClov) {
      const C *q = cb + aidx(ldir, H, 36);
#pragma unroll
      for (int w = 0; w < kClov; ++w)
        if (36 % kPart == 0 || ldir + w * kPart < 36) lc[w] = load_once(q + w * kPart * kBlk);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // what prepare_link folds into a link, per direction of the lane: the
  // coefficient, the boundary's factor, and the x or t where that applies
  // (y, z: -2 always, -1 never)
  R lcoef[kTasks];
  C lph[kTasks];
  int lwhen[kTasks];
#pragma unroll
  for (int w = 0; w < kTasks; ++w) {
    const int dir = ldir + w * kPart, mu = dir >> 1, fb = dir & 1;
    C f = cmk<C>((R)a.ph[0][0], (R)a.ph[0][1]);
    int last = g.L[0] - 1;
    if (mu == 1) f = cmk<C>((R)a.ph[1][0], (R)a.ph[1][1]), last = g.L[1] - 1;
    if (mu == 2) f = cmk<C>((R)a.ph[2][0], (R)a.ph[2][1]), last = g.L[2] - 1;
    if (mu == 3) f = cmk<C>((R)a.ph[3][0], (R)a.ph[3][1]), last = g.L[3] - 1;
    if (fb) f.y = -f.y, last = 0;
    lcoef[w] = (R)(mu == 3 ? a.ct : a.cs);
    lph[w] = cscale(f, lcoef[w]);
    lwhen[w] = (mu == 0 || mu == 3) ? last : ((mu == 1 ? lc4[1] : lc4[2]) == last ? -2 : -1);
  }
  auto link_stage = [&](int t) {
    const int x = 2 * lxh + ((lpar + t) & 1);
#pragma unroll
    for (int w = 0; w < kTasks; ++w) {
      const int dir = ldir + w * kPart;
      C u[9];
#pragma unroll
      for (int e = 0; e < NL; ++e) u[e] = lu[w][e];
      if (NL == 6) link_third_row(u);
      if (lwhen[w] == -2 || lwhen[w] == ((dir >> 1) == 3 ? t : x)) {
#pragma unroll
        for (int e = 0; e < 9; ++e) u[e] = cmul(lph[w], u[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 9; ++e) u[e] = cscale(u[e], lcoef[w]);
      }
#pragma unroll
      for (int e = 0; e < 9; ++e) lk[(dir * 9 + e) * LS + lsi] = u[e];
    }
    if (kHasClov) {
#pragma unroll
      for (int w = 0; w < kClov; ++w)
        if (36 % kPart == 0 || ldir + w * kPart < 36) cl[(ldir + w * kPart) * LS + lsi] = lc[w];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto wrap = [&](int t) { return t < 0 ? t + Lt : (t >= Lt ? t - Lt : t); };

  // X: own place in slice t + 1; qa, qb, qc: the other neighbours in turn.
  // Before the first step: slices t0 - 1 and t0 to LDS, its loads under way.
  wc_v4i X[12], qa[12], qb[12], qc[12];
  link_load(t0);
  gather(wrap(t0 - 1), h3, X);
  gather(t0, h3, qa);
  gather(t0, h_yp, qb);
  gather(t0, h_ym, qc);
  {
    wc_v4i *A = sp + (t0 & 1) * 12 * W + tid, *B = sp + ((t0 + 1) & 1) * 12 * W + tid;
#pragma unroll
    for (int k = 0; k < 12; ++k) B[k * W] = X[k];
#pragma unroll
    for (int k = 0; k < 12; ++k) A[k * W] = qa[k];
  }
  gather(t0, h_xo(t0), qa);
  gather(wrap(t0 + 1), h3, X);
  link_stage(t0);
  link_load(wrap(t0 + 1));
  const C *lw = lk + (v - v0);
#pragma unroll 1
  for (int t = t0; t < t1; ++t) {
    // A: own spinors of slice t, B: of slice t - 1 (a lane reads and writes
    // its own only; the barrier, of one wave, orders the links' LDS accesses)
    wc_v4i *A = sp + (t & 1) * 12 * W + tid, *B = sp + ((t + 1) & 1) * 12 * W + tid;
    const int tn = wrap(t + 1);
    const long h = (long)t * S3 + h3;
    __syncthreads();
    C acc[RB][12];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int k = 0; k < 12; ++k) acc[i][k] = cmk<C>(0, 0);
    const bool own_p = ((par + t) & 1) == 0;
    {
      C hp[RB][2][3], hm[RB][2][3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        wc_v4i o[4], x[4], y[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = A[(3 * k + c) * W];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          x[k] = own_p ? o[k] : qa[3 * k + c];
          y[k] = own_p ? qa[3 * k + c] : o[k];
        }
        march_project<R, DAG, 0, 0, RB>(x[0], x[1], x[2], x[3], c, hp);
        march_project<R, DAG, 0, 1, RB>(y[0], y[1], y[2], y[3], c, hm);
      }
      __builtin_amdgcn_sched_barrier(0);
      march_mul<R, DAG, 0, 0, RB>(hp, lw, acc);
      march_mul<R, DAG, 0, 1, RB>(hm, lw, acc);
    }
    // Each buffer is loaded again as soon as it is read; loads complete in
    // order, so each is issued in the order of use.  The epilogue's operands
    // take the places of the next step's +y (y) and -y (dotv) neighbours.
    gather(t, h_zp, qa);
    march_dir<R, DAG, 1, 0, RB>(qb, lw, acc);
    gather(t, h_zm, qb);
    march_dir<R, DAG, 1, 1, RB>(qc, lw, acc);
    if (EPI & EPI_DOT) gather_of(make_rsrc(a.dotv, fbytes), t, h3, qc);
    else gather(tn, h_ym, qc);
    march_dir<R, DAG, 2, 0, RB>(qa, lw, acc);
    gather(tn, h_xo(tn), qa);
    march_dir<R, DAG, 2, 1, RB>(qb, lw, acc);
    if (EPI & (EPI_DIAG | EPI_AXPY)) gather_of(make_rsrc(a.y, fbytes), t, h3, qb);
    else gather(tn, h_yp, qb);
    march_dir<R, DAG, 3, 0, RB>(X, lw, acc);
    {
      C hs[RB][2][3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        march_project<R, DAG, 3, 1, RB>(B[c * W], B[(3 + c) * W], B[(6 + c) * W], B[(9 + c) * W], c, hs);
      march_mul<R, DAG, 3, 1, RB>(hs, lw, acc);
    }
#pragma unroll
    for (int k = 0; k < 12; ++k) B[k * W] = X[k];
    gather(wrap(t + 2), h3, X);
    const bool zb = a.open_bc && (t == 0 || t == Lt - 1);
    hop_epilogue<R, EPI, RB, C>(
        a, h, rb, zb, blocks ? cl + (v - v0) : nullptr, (long)LS, acc,
        [&](C y[RB][12]) { march_unpack<R, RB>(qb, y); }, [&](C dv[RB][12]) { march_unpack<R, RB>(qc, dv); });
    if (EPI & (EPI_DIAG | EPI_AXPY)) gather(tn, h_yp, qb);
    if (EPI & EPI_DOT) gather(tn, h_ym, qc);
    __syncthreads();
    link_stage(tn);
    link_load(wrap(t + 2));
  }
}

// t-segments of ntiles tiles: whole rounds of an XCD's waves against what a
// segment costs beyond its steps (two slices more to load and the first
// latencies, about 3 steps: 16^3 x 32 FP64, 12 right-hand sides, 1 round of 2
// segments 94 us, 2 rounds of 5 117 us; 24^3 x 48, 4 rounds of 3 557 us, 2 of 1
// 692 us)
inline int march_segments(int ntiles, int Lt) {
  const long tpx = (ntiles + 7) / 8;
  int best = 1;
  long cost = -1;
  for (int n = 1; n <= Lt; ++n) {
    const long rounds = (tpx * n + kMarchSlots - 1) / kMarchSlots;
    const long c = rounds * ((Lt + n - 1) / n + 3);
    if (cost < 0 || c < cost) cost = c, best = n;
  }
  return best;
}

// tiles of a t-slice: waves of 64 items (site, group of RB right-hand sides)
template <typename R> inline int march_tiles(const HopLaunch &a) {
  const long items = a.g.Vh / a.g.L[3] * ((a.nrhs + march_rb<R>() - 1) / march_rb<R>());
  return (int)((items + kMarchItems - 1) / kMarchItems);
}

// Where the t-marching form applies: a wave's 64 items within march_sites
// sites (FP64 from 8 right-hand sides, except 9; FP32 from 7), working
// precision, fields within one buffer descriptor, one set of clover blocks.
// Its rule where neither the tuner nor the caller has decided (times against the
// gathering kernel, Meooe / M / Mpc^dag Mpc):
// - slices of 2048 half-sites or more walked 4 or more at a time, 1.0-1.7 / 0.92-1.5
//   / 0.93-1.5 times as fast.  Not with 15 to 17 groups of right-hand sides on x-y
//   planes of two 64-site blocks, where its patch just outgrows an L2 and the
//   gathering kernel's sites do not: 16 right-hand sides, FP64 16^3 x 32 12-real 0.91
//   / 0.89 / 0.95, 16 x 16 x 32^2 1.07 / 0.93 / 0.95 (12 of them 1.6 / 1.4 / 1.3).
// - lattices of at most 384 waves in all, with whole links: 8^4 FP64, 12 right-hand
//   sides, 1.21 / 1.32 / 1.11.  With 12-real links the gathering kernel has so much
//   less to load that it wins in the bare hop and in M (0.74-0.97 / 0.8-1.04), not in
//   the hops of Mpc with their clover and axpy (even counts 0.98-1.18; 8^3 x 16 FP32,
//   12: 71 -> 63 us).  Odd counts in FP32 cost a group that is half idle (8^3 x 12,
//   13: 0.99 / 1.03 / 0.93).
// Between, fields are in the caches and slices small enough that the gathering
// kernel finds most neighbours there.
template <typename R> bool march_applies(const HopLaunch &a) {
  constexpr int RB = march_rb<R>(), W = kMarchItems;
  if (!a.march || a.half_in || a.half_out || a.skip_t_faces || a.nrhs < RB || a.nrhs > 64) return false;
  if ((a.epi & EPI_CLOV) && a.clov_roff) return false;
  if (12.0 * (double)a.g.Vh * a.nrhs * 2.0 * sizeof(R) >= 4294967296.0) return false;
  const int G = (a.nrhs + RB - 1) / RB;
  if ((W % G == 0 ? W / G : (W - 1) / G + 2) > march_sites<R>()) return false;
  if (a.march == 1) return true;
  const int ntiles = march_tiles<R>(a), Lt = a.g.L[3];
  if ((long)ntiles * Lt <= 384) return a.nrhs % RB == 0 && (a.nl == 9 || (a.epi & (EPI_CLOV | EPI_AXPY)));
  if (G >= 15 && G <= 17 && a.g.Lxh * a.g.L[1] == 2 * kBlk) return false;
  const int n = march_segments(ntiles, Lt);
  return a.g.Vh / Lt >= 2048 && (Lt + n - 1) / n >= 4;
}

template <typename R, int NL, int DAG> static bool march_epi(const HopLaunch &a, unsigned grid, hipStream_t s) {
  constexpr size_t lds = 2 * 12 * kMarchItems * 16 + (size_t)108 * march_sites<R>() * 2 * sizeof(R);
  switch (a.epi) {
#define WC_EPI(E)                                                         \
  case E:                                                                 \
    k_hop_march<R, NL, DAG, E><<<grid, kMarchItems, lds, s>>>(a);         \
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

template <typename R> bool hop_march(const HopLaunch &a0, hipStream_t s) {
  HopLaunch a = a0;
  a.big = 0;
  const int ntiles = march_tiles<R>(a);
  a.march_segs = march_segments(ntiles, a.g.L[3]);
  const unsigned grid = (unsigned)(8 * ((ntiles + 7) / 8) * a.march_segs);
  if (a.nl == 9) return a.dag ? march_epi<R, 9, 1>(a, grid, s) : march_epi<R, 9, 0>(a, grid, s);
  return a.dag ? march_epi<R, 6, 1>(a, grid, s) : march_epi<R, 6, 0>(a, grid, s);
}

}  // namespace wck
