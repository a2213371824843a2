// Downward pass on the device (taichi_with_jerks/traverse_eager.h:272-292):
// L2L from each internal cell into its children, one launch per level from the
// root down, then L2P at every leaf, then the results are scattered back to
// the caller's body order.
//
//   L2L (kernel_fast_lean.h:1001-1058): for each child,
//       L_child[n,m] += sum_{k<=p-n} sum_{|l|<=k} L[n+k, m+l] conj Y_k^l(X - X_child)
//       one block per child, with the harmonic table and the parent's
//       expansions in LDS (8 KB at p = 12); each thread takes a share of the
//       output terms, whose sums run over contiguous runs of both tables, two
//       terms at a time into two partial sums.  The levels are a chain, and a
//       level of a few blocks takes the latency of one thread's sums, so there
//       are two shapes:
//       * one wave per child.  Beside a long P2P launch only blocks that fit
//         the slot of one finished P2P wave get in: levels of 256-thread
//         blocks waited for P2P's last blocks (at N = 2^20 the pass ended
//         1.4 ms after P2P; now it ends 4 ms before P2P does).
//       * 512 threads per child, two per output, on levels of at most 1,024
//         cells where P2P is short: a level 35 -> 13 us at p = 12; and above
//         p = 13 everywhere.
//   L2P (kernel_fast_lean.h:1060-1128): two leaves per wave, 32 lanes each
//       (leaves average ~19 bodies: one leaf per wave left 70% of the lanes
//       idle); lane = body, Y = Y(X_c - x_b) and
//       dY/dt with velocity -v_b, streamed order by order (three harmonic
//       rows in registers); only n <= 1 of the local field is formed:
//       p += Re Phi_0^0, a -= (Re Phi_1^1, Im Phi_1^1, Re Phi_1^0),
//       j -= the same of Phidot = L conj dY + Ldot conj Y.
#include "tc_common.h"
#include "tc_harm.h"
#include "tc_kernels.h"

#ifndef TC_SHARD
#error "compiled once per order shard, with -DTC_SHARD=k (see TC_NSHARDS in tc_kernels.h)"
#endif

namespace tcfmm {
namespace TC_SHARD_NS(TC_SHARD) {

// T threads per child, S of them sharing each output's sum (over every S-th
// source order).  ids (or null): parents, eight blocks each, block 8 i + k for
// child k; otherwise the blocks are the cells from `first` on.
template <int P, int T, int S>
__global__ __launch_bounds__(T) void k_l2l(CellsDev c, const int *__restrict__ ids, int first) {
  constexpr int NT = nterm(P);
  constexpr int NO = tri(P, P) + 1;
  static_assert(P + 1 <= T && T % kWave == 0 && (S == 1 || S == 2), "shape");
  __shared__ cplx G[NT], cl[NT], cld[NT];
  const int u = threadIdx.x;
  int ci, ch;
  if (ids) {
    ci = ids[blockIdx.x >> 3];
    if ((int)(blockIdx.x & 7) >= c.nchild[ci]) return;
    ch = c.child[ci] + (blockIdx.x & 7);
  } else {
    ch = first + blockIdx.x;
    ci = c.parent[ch];
  }
  const double *Lp = c.L + (size_t)ci * NT;
  const double *Ldp = c.Ld + (size_t)ci * NT;
  for (int t = u; t < NT; t += T) {
    int n = 0;
    while ((n + 1) * (n + 1) <= t) n++;
    const int m = t - n * n - n;
    cl[t] = packed_to_c(Lp, n, m);
    cld[t] = packed_to_c(Ldp, n, m);
  }
  harm_table_col<P>(u, c.X[3 * ci] - c.X[3 * ch], c.X[3 * ci + 1] - c.X[3 * ch + 1],
                    c.X[3 * ci + 2] - c.X[3 * ch + 2], G);
  __syncthreads();
  double *Lc = c.L + (size_t)ch * NT;
  double *Ldc = c.Ld + (size_t)ch * NT;
  // tasks (output term, L or Ldot), strided over the block
  const int part = S > 1 ? u & 1 : 0;
  for (int j = u / S; j < 2 * NO; j += T / S) {
    const int which = j >= NO, o = j - which * NO;
    int n = 0;
    while (tri(n + 1, 0) <= o) n++;
    const int m = o - tri(n, 0);
    const cplx *src = which ? cld : cl;
    cplx a = {0, 0}, a2 = {0, 0};
    for (int kk = part; kk <= P - n; kk += S) {
      // l = -kk..kk: src[ixnm(n + kk, m + l)] and G[ixnm(kk, l)] run contiguously
      const cplx *sr = src + ixnm(n + kk, m - kk), *gr = G + ixnm(kk, -kk);
      const int len = 2 * kk + 1;
      int t = 0;
      for (; t + 1 < len; t += 2) {
        a = cadd(a, cmul(sr[t], cconj(gr[t])));
        a2 = cadd(a2, cmul(sr[t + 1], cconj(gr[t + 1])));
      }
      if (t < len) a = cadd(a, cmul(sr[t], cconj(gr[t])));
    }
    a = cadd(a, a2);
    if (S > 1) {
      a.re += dpp_move<0xb1>(a.re);  // the neighbour's part (lanes 2 i, 2 i + 1)
      a.im += dpp_move<0xb1>(a.im);
    }
    if (part == 0) {
      double *dst = which ? Ldc : Lc;
      const int s = n * n + n;
      dst[s + m] += a.re;
      if (m > 0) dst[s - m] += a.im;
    }
  }
}

// Orders K..P of L2P for one body: row K of Y(X_c - x_b) (compile-time K, no
// case tests) and its time derivative, contracted with L / Ldot of orders K
// and K+1 for the n <= 1 part of the local field.  l = -m uses
// Y_k^{-m} = (-1)^m conj(Y_k^m), and the same of L, Ldot and dY/dt, so the
// terms of the outputs of order m = 0 that are read as real parts (Phi_0^0,
// Phi_1^0 and its time derivative) come in equal pairs: only l >= 0 is
// formed, the l > 0 sums (h00, h10, e10) counting twice at the end.
// Phi_1^1 and its derivative keep both l = +m and l = -m.  A scheduling
// barrier per order keeps the later orders' coefficient reads from being
// hoisted (which multiplies the live registers).
struct L2PAcc {
  double p00, h00, p10, h10, d10, e10;  // Re parts: l = 0 terms, l > 0 terms
  cplx p11, d11;
};

template <int P, int K>
__device__ __forceinline__ void l2p_orders(double dx, double dy, double dz, double r2, double vx,
                                           double vy, double vz, const cplx *cl, const cplx *cld,
                                           cplx *y1, cplx *y2, L2PAcc &a) {
  __builtin_amdgcn_sched_barrier(0);
  cplx yk[P + 1];
  harm_row_c<K>(dx, dy, dz, r2, y1, y2, yk);
  const cplx *L0 = cl + K * K + K;
  const cplx *L1 = cl + (K + 1) * (K + 1) + (K + 1);
  const cplx *D1 = cld + (K + 1) * (K + 1) + (K + 1);
  constexpr bool up = K < P;
  auto redot = [](cplx u, cplx v) { return u.re * v.re + u.im * v.im; };  // Re(u conj v)
#pragma unroll
  for (int m = 0; m <= K; m++) {
    cplx dy_m = {0.0, 0.0};
    if constexpr (K > 0) {
      const cplx eta = {-vx * 0.5, vy * 0.5}, xi = {vx * 0.5, vy * 0.5};
      if (m <= K - 2) dy_m = cadd(dy_m, cmul(y1[m + 1 <= P ? m + 1 : P], eta));
      if (m <= K - 1) dy_m = cadd(dy_m, cscale(vz, y1[m]));
      if (m >= 1) {
        dy_m = cadd(dy_m, cmul(y1[m >= 1 ? m - 1 : 0], xi));
      } else if (K >= 2) {
        const cplx c1 = cconj(y1[1]);
        dy_m = cadd(dy_m, cmul({-c1.re, -c1.im}, xi));
      }
    }
    const cplx y = yk[m];
    if (m == 0) {
      a.p00 += redot(L0[0], y);
      if (up) {
        a.p10 += redot(L1[0], y);
        a.d10 += redot(L1[0], dy_m) + redot(D1[0], y);
      }
    } else {
      a.h00 += redot(L0[m], y);
      if (up) {
        a.h10 += redot(L1[m], y);
        a.e10 += redot(L1[m], dy_m) + redot(D1[m], y);
      }
    }
    if (up) {
      const cplx g = cconj(y), gd = cconj(dy_m);
      a.p11 = cadd(a.p11, cmul(L1[m + 1], g));
      a.d11 = cadd(a.d11, cadd(cmul(L1[m + 1], gd), cmul(D1[m + 1], g)));
      if (m > 0) {
        const double sg = (m & 1) ? -1.0 : 1.0;
        const cplx g2 = cscale(sg, y), gd2 = cscale(sg, dy_m);
        a.p11 = cadd(a.p11, cmul(L1[1 - m], g2));
        a.d11 = cadd(a.d11, cadd(cmul(L1[1 - m], gd2), cmul(D1[1 - m], g2)));
      }
    }
  }
  if constexpr (K < P) {
#pragma unroll
    for (int m = 0; m <= K; m++) {
      y2[m] = y1[m];
      y1[m] = yk[m];
    }
    l2p_orders<P, K + 1>(dx, dy, dz, r2, vx, vy, vz, cl, cld, y1, y2, a);
  }
}

// kAdd: into the results (which the caller cleared or already holds sums in);
// otherwise every body's far-field results are written, zeros for bodies that
// are not sinks, and nothing has to be cleared before.
//
// Up to p = 12 the kernel is held to three waves per SIMD (168 VGPRs; at
// p = 12 that spills 14 of its 196, 60 bytes per lane, and still runs the
// downward pass 0.02-0.08 ms sooner per 2^20-body evaluation than two waves).
template <int P, bool kAdd>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(P <= 12 ? 3 : 1))) void k_l2p(
    CellsDev c, BodiesDev b, ResultsDev r, const int *__restrict__ leaf_ids, int nleaves) {
  constexpr int NT = nterm(P);
  constexpr int kHalf = kWave / 2;  // lanes per leaf: two leaves per wave
  __shared__ cplx cl[2][NT], cld[2][NT];
  const int lane = threadIdx.x, h = lane / kHalf, u = lane - h * kHalf;
  const int li = 2 * (int)blockIdx.x + h;
  const int ci = li < nleaves ? leaf_ids[li] : -1;
  const bool on = ci >= 0 && c.has_sink[ci];
  if (on) {
    const double *Lp = c.L + (size_t)ci * NT;
    const double *Ldp = c.Ld + (size_t)ci * NT;
    for (int t = u; t < NT; t += kHalf) {
      int n = 0;
      while ((n + 1) * (n + 1) <= t) n++;
      int m = t - n * n - n;
      cl[h][t] = packed_to_c(Lp, n, m);
      cld[h][t] = packed_to_c(Ldp, n, m);
    }
  }
  __syncthreads();
  if (ci < 0) return;
  const int b0 = c.body[ci], nb = c.nbody[ci];
  if (!on) {
    if (!kAdd)
      for (int i = b0 + u; i < b0 + nb; i += kHalf)
        r.pot[i] = r.ax[i] = r.ay[i] = r.az[i] = r.jx[i] = r.jy[i] = r.jz[i] = 0.0;
    return;
  }
  const double X0 = c.X[3 * ci], X1 = c.X[3 * ci + 1], X2 = c.X[3 * ci + 2];
  for (int base = 0; base < nb; base += kHalf) {
    const int i = b0 + base + u;
    if (base + u >= nb) continue;
    if (!(b.flags[i] & kSink)) {
      if (!kAdd) r.pot[i] = r.ax[i] = r.ay[i] = r.az[i] = r.jx[i] = r.jy[i] = r.jz[i] = 0.0;
      continue;
    }
    const double vx = -b.vx[i], vy = -b.vy[i], vz = -b.vz[i];
    const double dx = X0 - b.x[i], dy = X1 - b.y[i], dz = X2 - b.z[i];
    const double r2 = dx * dx + dy * dy + dz * dz;
    cplx y1[P + 1], y2[P + 1];
    L2PAcc a = {0, 0, 0, 0, 0, 0, {0, 0}, {0, 0}};
    l2p_orders<P, 0>(dx, dy, dz, r2, vx, vy, vz, cl[h], cld[h], y1, y2, a);
    r.pot[i] = (kAdd ? r.pot[i] : 0.0) + (a.p00 + 2.0 * a.h00);
    r.ax[i] = (kAdd ? r.ax[i] : 0.0) - a.p11.re;
    r.ay[i] = (kAdd ? r.ay[i] : 0.0) - a.p11.im;
    r.az[i] = (kAdd ? r.az[i] : 0.0) - (a.p10 + 2.0 * a.h10);
    r.jx[i] = (kAdd ? r.jx[i] : 0.0) - a.d11.re;
    r.jy[i] = (kAdd ? r.jy[i] : 0.0) - a.d11.im;
    r.jz[i] = (kAdd ? r.jz[i] : 0.0) - (a.d10 + 2.0 * a.e10);
  }
}

template <int P>
static void l2l_go(CellsDev c, const int *ids, int first, int nblocks, bool wide, hipStream_t s) {
  if (wide)
    hipLaunchKernelGGL((k_l2l<P, 512, 2>), dim3(nblocks), dim3(512), 0, s, c, ids, first);
  else
    hipLaunchKernelGGL((k_l2l<P, 64, 1>), dim3(nblocks), dim3(64), 0, s, c, ids, first);
}
template <int P>
static void l2p_go(CellsDev c, BodiesDev b, ResultsDev r, const int *ids, int n, bool add,
                   hipStream_t s) {
  const dim3 g((n + 1) / 2), t(64);
  if (add)
    hipLaunchKernelGGL((k_l2p<P, true>), g, t, 0, s, c, b, r, ids, n);
  else
    hipLaunchKernelGGL((k_l2p<P, false>), g, t, 0, s, c, b, r, ids, n);
}

// Whether a level of `cells` takes 512 threads per cell: up to 1,024 cells
// (four blocks a CU) where no long P2P runs beside it, and always above p = 13,
// where the tables (48 bytes a coefficient) leave room for few one-wave blocks
// on a CU and for none in a finished P2P wave's slot (13 KB).  One wave / eight
// waves per cell: p = 20, N = 2^17, the three widest levels 108, 197, 207 / 52,
// 80, 109 us; evaluations beside a long P2P, N = 2^18 (theta 0.4) p = 13 8.74 /
// 8.84 ms, 14 10.48 / 10.47, 16 13.04 / 12.89, 20 25.35 / 24.83, 24 41.0 / 39.4.
template <int P>
constexpr bool l2l_wide(int cells, bool beside) {
  return (cells <= 1024 && !beside) || 48 * nterm(P) > 10 * 1024;
}

int launch_l2l(int p, CellsDev c, int ls, int le, bool beside, hipStream_t s) {
  if (le <= ls) return 0;
  switch (p) {
#define TC_CASE(P)\
  case P:\
    if constexpr (in_shard(P, TC_SHARD)) {\
      l2l_go<P>(c, nullptr, ls, le - ls, l2l_wide<P>(le - ls, beside), s);\
      return 0;\
    } else {\
      return -1;\
    }
    TC_FOR_EACH_P(TC_CASE)
#undef TC_CASE
    default:
      return -1;
  }
}

int launch_l2l_ids(int p, CellsDev c, const int *ids, int nids, hipStream_t s) {
  if (nids <= 0) return 0;
  switch (p) {
#define TC_CASE(P)\
  case P:\
    if constexpr (in_shard(P, TC_SHARD)) {\
      l2l_go<P>(c, ids, 0, 8 * nids, l2l_wide<P>(8 * nids, false), s);\
      return 0;\
    } else {\
      return -1;\
    }
    TC_FOR_EACH_P(TC_CASE)
#undef TC_CASE
    default:
      return -1;
  }
}

int launch_l2p(int p, CellsDev c, BodiesDev b, ResultsDev r, const int *leaf_ids, int nleaves,
               hipStream_t s, bool add) {
  if (nleaves <= 0) return 0;
  switch (p) {
#define TC_CASE(P)\
  case P:\
    if constexpr (in_shard(P, TC_SHARD)) {\
      l2p_go<P>(c, b, r, leaf_ids, nleaves, add, s);\
      return 0;\
    } else {\
      return -1;\
    }
    TC_FOR_EACH_P(TC_CASE)
#undef TC_CASE
    default:
      return -1;
  }
}

}  // namespace TC_SHARD_NS(TC_SHARD)
}  // namespace tcfmm
