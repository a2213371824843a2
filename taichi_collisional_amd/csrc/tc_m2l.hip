// M2L: rotation-based multipole-to-local translation, FP64, gfx950.
//
// Follows M2L_rotate (taichi_with_jerks/kernel_fast_lean.h:1130-1371): per
// (target Ci, source Cj) pair the source moments are scaled to homogeneous
// form, rotated about z by alpha_z, x<->z swapped, rotated by alpha_x, swapped
// back (so the pair axis lies along z), translated along z, and rotated back
// with the same four steps in reverse; the result is added to Ci's local
// expansion.  The same operator maps Mdot to Ldot.
//
// GPU form.  The swap S_n is the same matrix for every pair, so it is applied
// as a product of constant sparse blocks against each lane's coefficients:
// one lane = one (target, source) pair, the swap entries are folded into the
// instruction stream as constant operands of v_fma_f64, and only the per-pair
// z-rotations and translation factors live in registers.  The forward half's
// scaling by (n+|m|)!(n-|m|)! is folded into its two swaps' constants.  Work that the translation cannot see is skipped: after the
// second forward swap only components |m| <= min(n, p-n) are formed, and the
// first backward swap only reads those.  The quirk of the reference's
// factorial table (factorial_table[2p] == 0, kernel_fast_lean.h:129) removes
// M_p^{+-p} from the sum; with quirk=1 those inputs are zeroed.
//
// The order P of a launch is the truncation order of its pairs: the cells'
// coefficient rows may be longer (stride >= (P+1)^2 doubles, an expansion of
// a higher order), and only the terms up to order P are read and added, so
// one set of coefficient arrays serves pairs of different orders.
//
// Work decomposition: one wave = one chunk of <= 64 sources of a single target
// cell (the chunk list is grouped by target) for one array (M -> L or Mdot ->
// Ldot); each XCD takes a contiguous range of the (array, chunk) items so
// neighbouring targets share its L2.  The contributions are summed across the
// wave on the matrix unit (WaveSum); the chunk adds its sum into the target's
// L with one atomic per coefficient.
//
// Bound by FP64 issue, with the gathers close behind (p = 12, N = 2^20, under
// the counters: vector instructions 77 % of the cycles, matrix ones 15 %, the
// texture data unit 87 % busy, at 1.87 GHz).  One launch, before -> after the
// sums left the vector unit and LDS, the four-wave blocks and the two parts:
// p = 12, N = 2^20 (theta 0.4, 35.2 M pairs) 14.06 -> 13.2 ms; N = 2^17 (theta
// 0.5, 1.98 M pairs) p = 16: 3.18 -> 2.11, 18: 4.82 -> 2.79, 20: 11.70 ->
// 4.94, 24: 37.0 -> 8.29 ms.
#include "tc_common.h"
#include "tc_kernels.h"
#include "swap_tables.h"

#include <algorithm>

#ifndef TC_SHARD
#error "compiled once per order shard, with -DTC_SHARD=k (see TC_NSHARDS in tc_kernels.h)"
#endif

namespace tcfmm {
namespace TC_SHARD_NS(TC_SHARD) {

// n! for the translation factors, loaded with scalar loads (uniform across the
// wave).  Filled by m2l_init_tables().
__constant__ double c_fact[2 * kMaxP + 2];

// z-rotation of one order by e^{i m alpha} (forward) or e^{-i m alpha}
// (backward), m = 1..N.  The powers come from the recurrence
// e^{i(m+1)a} = e^{ima} e^{ia} (kernel_fast_lean.h:1163-1169).
//
// rotate(): the chain is recomputed inside the call from an opaque copy of
// e^{ia}.  Without the copy the compiler merges the identical chains of all
// unrolled orders into one table of 4p powers that stays live across the
// kernel (p = 12: ~90 extra registers, one wave per SIMD instead of two).
// The forward half uses it: its orders run p..0, so a table would be largest
// exactly where the working set is.  The backward half runs 0..p and grows a
// table by one power per order instead (rotate_tab), while the rotated
// moments it consumes die off.
template <int N, bool kBack>
__device__ __forceinline__ void rotate(double *v, double c1, double s1) {
  asm volatile("" : "+v"(c1), "+v"(s1));
  // Chebyshev form of the power recurrence: cos((m+1)a) = 2 cos a cos(ma) -
  // cos((m-1)a), and the same for sin, one FMA per component per power
  const double t = c1 + c1;
  double cq = 1.0, sq = 0.0, c = c1, s = s1;
#pragma unroll
  for (int m = 1; m <= N; m++) {
    double im = v[N - m], re = v[N + m];
    if (kBack) {
      v[N - m] = c * im - s * re;
      v[N + m] = c * re + s * im;
    } else {
      v[N - m] = c * im + s * re;
      v[N + m] = c * re - s * im;
    }
    if (m < N) {
      const double cn = fma(t, c, -cq), sn = fma(t, s, -sq);
      cq = c;
      sq = s;
      c = cn;
      s = sn;
    }
  }
}

template <int N, bool kBack>
__device__ __forceinline__ void rotate_tab(double *v, const double *cp, const double *sp) {
#pragma unroll
  for (int m = 1; m <= N; m++) {
    const double c = cp[m], s = sp[m];
    double im = v[N - m], re = v[N + m];
    if (kBack) {
      v[N - m] = c * im - s * re;
      v[N + m] = c * re + s * im;
    } else {
      v[N - m] = c * im + s * re;
      v[N + m] = c * re - s * im;
    }
  }
}

// Powers e^{iNa} from the two below (the Chebyshev recurrence rotate() uses),
// stored at index N; index 0 holds e^0.
template <int N>
__device__ __forceinline__ void extend_powers(double *cp, double *sp, double c1, double s1) {
  if constexpr (N == 1) {
    cp[0] = 1.0;
    sp[0] = 0.0;
    cp[1] = c1;
    sp[1] = s1;
  } else if constexpr (N > 1) {
    const double t = c1 + c1;
    cp[N] = fma(t, cp[N - 1], -cp[N - 2]);
    sp[N] = fma(t, sp[N - 1], -sp[N - 2]);
  }
}

// out rows |r-N| <= QR from input columns |c-N| <= QC (everything else 0).
// S_n only couples components of one parity class (Re/Im part and parity of
// m); rows are produced class by class so each class's inputs die early.
// kScaled: D^-1 S_n D with D = diag((n+|m|)!(n-|m|)!) instead of S_n.
template <int N, int QR, int QC, bool kScaled = false>
__device__ __forceinline__ void swap_block(const double *in, double *out) {
#pragma unroll
  for (int cls = 0; cls < 4; cls++) {
#pragma unroll
    for (int r = 0; r < 2 * N + 1; r++) {
      const int m = r - N;
      const int rc = (m >= 0 ? 0 : 2) + ((m < 0 ? -m : m) & 1);
      if (rc != cls) continue;
      double acc = 0.0;
      if (m <= QR && -m <= QR) {
#pragma unroll
        for (int e = kSwapRowPtr[N * N + r]; e < kSwapRowPtr[N * N + r + 1]; e++) {
          const int c = kSwapCol[e];
          if (c - N <= QC && N - c <= QC) acc += (kScaled ? kSwapValScaled[e] : kSwapVal[e]) * in[c];
        }
      }
      out[r] = acc;
    }
  }
}

// Waves per block, one chunk each.  From p = 14 on the kernel's straight-line
// code is larger than the 64 KB instruction cache (p = 15: 77 KB, 20: 175 KB,
// 24: 310 KB); the four waves of a block then go through it together, kept in
// step by a barrier per order, so that each line is fetched once for four.
constexpr int m2l_waves(int p) { return p >= 14 ? 4 : 1; }

// Waves per SIMD the registers are cut for (0: as they come, two or more).
// Two up to p = 19 (p = 19: 3.43 ms against 4.63 with one, N = 2^17), one
// above, where the second wave's share spills (p = 20: 4.94 against 5.26 with
// two, p = 24: 8.29 against 12.9).
constexpr int m2l_occ(int p) { return p < 13 ? 0 : p <= 19 ? 2 : 1; }

// The source orders are taken in two parts, k > m2l_split(p) and then the
// rest, each rotated, translated and rotated back (the operator is linear):
// the first part reaches only the target orders n < p - m2l_split, whose
// backward half costs an eighth of the whole, and each part's rotated moments
// are about half of all (p = 20: 100 and 121 of 221 doubles, which with the
// working set would be over 512 registers).  -1: one part, up to p = 13, whose
// moments fit (p = 12 in two parts: 14.4 ms against 13.2, N = 2^20; p = 14:
// 1.52 ms in two parts, 1.71 in one, N = 2^17).
constexpr int m2l_split(int p) { return p >= 14 ? p / 2 : -1; }

// Where the rotated moments M_k^m, |m| <= q(k) = min(k, P - k), of the source
// orders k = LO..HI are kept between the halves: a register each, and in the
// orders of four-wave blocks (where LDS is free and registers are not) an LDS
// slot for those with P - k - |m| <= reach, which the translation reads at
// most reach + 1 times: as many as fit (80 or 40 KB a SIMD's wave).
template <int P>
struct M2LStore {
  // register index, or -1 - slot; at k^2 + k + m
  short at[(P + 1) * (P + 1)];
  int regs, slots;
};
constexpr int m2l_q(int p, int k) { return k < p - k ? k : p - k; }
template <int P>
constexpr M2LStore<P> m2l_store(int lo, int hi) {
  const int room = m2l_waves(P) == 1 ? 0 : m2l_occ(P) == 2 ? 39 : 80;
  int reach = -1;
  for (int u = 0; u <= P; u++) {
    int c = 0;
    for (int k = lo; k <= hi; k++)
      for (int m = -m2l_q(P, k); m <= m2l_q(P, k); m++) c += P - k - (m < 0 ? -m : m) <= u;
    if (c > room) break;
    reach = u;
  }
  M2LStore<P> s = {};
  for (int k = lo; k <= hi; k++)
    for (int m = -m2l_q(P, k); m <= m2l_q(P, k); m++) {
      if (P - k - (m < 0 ? -m : m) <= reach)
        s.at[k * k + k + m] = (short)(-1 - s.slots++);
      else
        s.at[k * k + k + m] = (short)s.regs++;
    }
  return s;
}
template <int P, int LO, int HI>
struct M2LPart {
  static constexpr M2LStore<P> store = m2l_store<P>(LO, HI);
  // largest |m| that reaches target order n, and the largest such order
  static constexpr int q(int n) {
    int q = 0;
    for (int k = LO; k <= HI && k <= P - n; k++) q = m2l_q(P, k) > q ? m2l_q(P, k) : q;
    return n < q ? n : q;
  }
  static constexpr int top = P - LO;
};
template <int P, int LO, int HI>
constexpr M2LStore<P> M2LPart<P, LO, HI>::store;

// M_k^m (compile-time k, m) from where it is kept; ml: the lane's LDS column
template <class Part>
__device__ __forceinline__ double kept(const double *mp, const double *ml, int k, int m) {
  const int w = Part::store.at[k * k + k + m];
  return w < 0 ? ml[(-1 - w) * kWave] : mp[w];
}

template <int N>
__device__ __forceinline__ void load_order(const double *__restrict__ src, double *v) {
#pragma unroll
  for (int r = 0; r < 2 * N + 1; r++) v[r] = src[N * N + r];
}

// Forward half for the orders N..LO of the source moments, one after another:
// rotate by alpha_z, swap, rotate by alpha_x, swap (rows |m| <= min(N, p-N)
// only), into the rotated-moment store.  b0 holds order N; the gather of order
// N-1 is issued first, fenced with scheduling barriers so the compiler neither
// hoists every order's gathers to the top nor sinks them to their use (deeper
// prefetch made no difference).
template <int P, int LO, int HI, int N>
__device__ __forceinline__ void m2l_forward_order(const double *__restrict__ src, bool quirk,
                                                  double ezr, double ezi, double exr,
                                                  double exi, const double *b0, double *mp,
                                                  double *ml) {
  using Part = M2LPart<P, LO, HI>;
  constexpr int K = 2 * N + 1;
  constexpr int Q = m2l_q(P, N);
  if constexpr (m2l_waves(P) > 1) __syncthreads();
  double nb[N > LO ? 2 * N - 1 : 1];
  if constexpr (N > LO) {
    __builtin_amdgcn_sched_barrier(0);
    load_order<N - 1>(src, nb);
    __builtin_amdgcn_sched_barrier(0);
  }
  // D^-1 S Rx S D Rz with D = diag((n+|m|)!(n-|m|)!) (the reference's scale
  // and unscale, kernel_fast_lean.h:1175-1181, 1247-1251): the z-rotations
  // only mix +-m, so they commute with D, and the product is
  // (D^-1 S D) Rx (D^-1 S D) Rz -- the scaling lives in the swap constants
  double v[K], w[K];
#pragma unroll
  for (int r = 0; r < K; r++) v[r] = b0[r];
  if (N == P && quirk) {
    v[0] = 0.0;
    v[2 * N] = 0.0;
  }
  rotate<N, false>(v, ezr, ezi);
  swap_block<N, N, N, true>(v, w);
  rotate<N, false>(w, exr, exi);
  swap_block<N, Q, N, true>(w, v);
#pragma unroll
  for (int m = -Q; m <= Q; m++) {
    const int at = Part::store.at[N * N + N + m];
    if (at < 0)
      ml[(-1 - at) * kWave] = v[N + m];
    else
      mp[at] = v[N + m];
  }
  if constexpr (N > LO)
    m2l_forward_order<P, LO, HI, N - 1>(src, quirk, ezr, ezi, exr, exi, nb, mp, ml);
}

// The sums over the wave's pairs, by the FP64 matrix unit: with one operand
// the lanes' values u and the other a 0 / 1 selector, a product of four 4 x 4
// blocks adds lanes l, l + 16, l + 32, l + 48 of one coefficient and puts the
// sum in one of four columns, so four coefficients share a register; a second
// product, from the other side, adds the four rows of that register into one
// row, so sixteen coefficients share one (each summed over 16 lanes), and two
// rotations within rows of 16 lanes finish them.  Exact selectors: the sums
// round as additions do.  Coefficients are taken in their storage order t =
// n^2 + n + m, whatever their order n.
//
// Lane layout of v_mfma_f64_4x4x4_4b (b = block): A[i][k] in lane i + 4 b +
// 16 k, B[k][j] in lane j + 4 b + 16 k, D[i][j] in lane j + 4 b + 16 i.
struct WaveSum {
  double sel[4];  // sel[i]: 1 in lanes with lane % 4 == i
  double four, sixteen, out;

  __device__ __forceinline__ void start(int lane) {
#pragma unroll
    for (int i = 0; i < 4; i++) sel[i] = (lane & 3) == i ? 1.0 : 0.0;
    four = sixteen = out = 0.0;
  }
  // coefficient T of NT (compile-time, increasing); dst: the target's row
  template <int T, int NT>
  __device__ __forceinline__ void add(double u, double *dst, bool write, int lane) {
    four = __builtin_amdgcn_mfma_f64_4x4x4f64(u, sel[T % 4], T % 4 == 0 ? 0.0 : four, 0, 0, 0);
    if constexpr (T % 4 == 3 || T == NT - 1) {
      constexpr int G = T / 4;
      sixteen = __builtin_amdgcn_mfma_f64_4x4x4f64(sel[G % 4], four,
                                                   G % 4 == 0 ? 0.0 : sixteen, 0, 0, 0);
      if constexpr (G % 4 == 3 || T == NT - 1) {
        // lane j + 4 b + 16 i: block b's part of coefficient 16 H + 4 i + j
        constexpr int H = G / 4;
        double v = sixteen + dpp_move<0x124>(sixteen);
        v += dpp_move<0x128>(v);
        out = ((lane >> 2) & 3) == H % 4 ? v : out;
        if constexpr (H % 4 == 3 || T == NT - 1) {
          const int t = 64 * (H / 4) + 16 * ((lane >> 2) & 3) + 4 * (lane >> 4) + (lane & 3);
          if (write && t <= T) atomicAdd(dst + t, out);
        }
      }
    }
  }
};

template <int N, int NT, int R = 0>
__device__ __forceinline__ void sum_order(WaveSum &ws, const double *u, double *dst, bool write,
                                          int lane) {
  ws.template add<N * N + R, NT>(u[R], dst, write, lane);
  if constexpr (R < 2 * N) sum_order<N, NT, R + 1>(ws, u, dst, write, lane);
}

// f: translation factors f[j] = j! r^-(j+1), one table for all orders (order N
// reads j = N..P, so the entries die off as the rotation powers grow).  Up to
// p = 15 the powers of both angles are such growing tables; above, they would
// take 4 p doubles and are formed again in every order, as in the forward half.
template <int P, int LO, int HI, int N>
__device__ __forceinline__ void m2l_backward_order(const double *mp, const double *ml,
                                                   const double *f, double ezr, double ezi,
                                                   double exr, double exi, double *czp,
                                                   double *szp, double *cxp, double *sxp,
                                                   WaveSum &ws, double *dst, bool write,
                                                   int lane) {
  using Part = M2LPart<P, LO, HI>;
  constexpr int K = 2 * N + 1;
  constexpr int Q = Part::q(N);
  constexpr int TOP = HI < P - N ? HI : P - N;  // source orders LO..TOP reach order N
  if constexpr (m2l_waves(P) > 1) __syncthreads();
  // one order at a time: keeps the scheduler from interleaving the
  // register-only work of several orders (which multiplies live state)
  __builtin_amdgcn_sched_barrier(0);
  double u[K], w[K];
#pragma unroll
  for (int r = 0; r < K; r++) u[r] = 0.0;
  // translation along z (kernel_fast_lean.h:1253-1295):
  // L_n^{+-m} += (-1)^m sum_{k=m}^{p-n} M_k^{+-m} (n+k)! r^-(n+k+1)
#pragma unroll
  for (int k = LO; k <= TOP; k++) u[N] += kept<Part>(mp, ml, k, 0) * f[N + k];
#pragma unroll
  for (int m = 1; m <= Q; m++) {
#pragma unroll
    for (int k = LO; k <= TOP; k++) {
      if (m > m2l_q(P, k)) continue;
      const double fk = (m & 1) ? -f[N + k] : f[N + k];
      u[N - m] += kept<Part>(mp, ml, k, -m) * fk;
      u[N + m] += kept<Part>(mp, ml, k, m) * fk;
    }
  }
  constexpr bool kTab = P <= 15;
  if constexpr (kTab) {
    extend_powers<N>(cxp, sxp, exr, exi);
    extend_powers<N>(czp, szp, ezr, ezi);
  }
  swap_block<N, N, Q>(u, w);
  if constexpr (kTab)
    rotate_tab<N, true>(w, cxp, sxp);
  else
    rotate<N, true>(w, exr, exi);
  swap_block<N, N, N>(w, u);
  if constexpr (kTab)
    rotate_tab<N, true>(u, czp, szp);
  else
    rotate<N, true>(u, ezr, ezi);
  sum_order<N, (Part::top + 1) * (Part::top + 1)>(ws, u, dst, write, lane);
}

template <int P, int LO, int HI, int... Ns>
__device__ __forceinline__ void m2l_backward_all(const double *mp, const double *ml,
                                                 const double *f, double ezr, double ezi,
                                                 double exr, double exi, double *dst, bool write,
                                                 int lane, IntSeq<Ns...>) {
  WaveSum ws;
  ws.start(lane);
  double czp[P + 1], szp[P + 1], cxp[P + 1], sxp[P + 1];
  (m2l_backward_order<P, LO, HI, Ns>(mp, ml, f, ezr, ezi, exr, exi, czp, szp, cxp, sxp, ws, dst,
                                     write, lane),
   ...);
}

// Source orders LO..HI of the chunk's pairs, added to the target's row dst.
template <int P, int LO, int HI>
__device__ __forceinline__ void m2l_part(const double *__restrict__ src, bool quirk, double ezr,
                                         double ezi, double exr, double exi, double ri,
                                         bool active, double *dst, bool write, int lane,
                                         double *ml) {
  using Part = M2LPart<P, LO, HI>;
  // Orders run from HI down: the large orders (biggest working set) run while
  // few rotated moments are live.
  double mp[Part::store.regs], v0[2 * HI + 1];
  load_order<HI>(src, v0);
  m2l_forward_order<P, LO, HI, HI>(src, quirk, ezr, ezi, exr, exi, v0, mp, ml);
  // Fence the rotated moments: without it, IR-level code motion interleaves
  // the forward and backward halves and roughly doubles the live registers
  // (p = 12: 512 registers plus scratch spills instead of ~310, no spills).
#pragma unroll
  for (int t = 0; t < Part::store.regs; t++) asm volatile("" : "+v"(mp[t]));
  __builtin_amdgcn_sched_barrier(0);
  // translation factors j! r^-(j+1); zero on idle lanes, which zeroes their
  // whole contribution
  double f[P + 1];
  {
    double rp = active ? ri : 0.0;
#pragma unroll
    for (int k = 0; k <= P; k++) {
      f[k] = c_fact[k] * rp;
      rp *= ri;
    }
  }
  m2l_backward_all<P, LO, HI>(mp, ml, f, ezr, ezi, exr, exi, dst, write, lane,
                              MakeIntSeq<Part::top + 1>{});
}

template <int P>
__global__ __launch_bounds__(64 * m2l_waves(P))
    __attribute__((amdgpu_waves_per_eu(m2l_occ(P) > 0 ? m2l_occ(P) : 1))) void k_m2l(
    const int4 *__restrict__ chunks, int nchunk, const int *__restrict__ src_list,
    const double *__restrict__ cX, const unsigned char *__restrict__ has_sink,
    const double *__restrict__ M, const double *__restrict__ Md, double *__restrict__ L,
    double *__restrict__ Ld, int quirk, int stride) {
  constexpr int W = m2l_waves(P);
  const int lane = threadIdx.x & (kWave - 1);
  // (chunk, array) from the linear block id, contiguous per XCD; waves past
  // the last item, or whose target has no sink, repeat a chunk and write
  // nothing (a block of such waves ends at once)
  const int first = xcd_contiguous(blockIdx.x, gridDim.x) * W;
  auto live = [&](int k) { return k < 2 * nchunk && has_sink[chunks[k % nchunk].x]; };
  bool any = false;
#pragma unroll
  for (int k = 0; k < W; k++) any |= live(first + k);
  if (!any) return;
  const int mine = first + __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const bool write = W == 1 || live(mine);
  const int item = min(mine, 2 * nchunk - 1);
  const int which = item >= nchunk;
  const int4 ch = chunks[item - which * nchunk];
  const int tgt = ch.x, start = ch.y, cnt = ch.z;
  const double *Msrc = which ? Md : M;
  double *Lout = which ? Ld : L;
  const bool active = lane < cnt;
  const int j = src_list[start + (active ? lane : 0)];

  double dx = cX[3 * tgt + 0] - cX[3 * j + 0];
  double dy = cX[3 * tgt + 1] - cX[3 * j + 1];
  double dz = cX[3 * tgt + 2] - cX[3 * j + 2];
  double rxy2 = dx * dx + dy * dy;
  double rxy = sqrt(rxy2);
  double r = sqrt(rxy2 + dz * dz);
  double ri = 1.0 / r;
  // e^{i alpha_z} = (dY + i dX)/r_xy (1 on the z axis), e^{i alpha_x} = (dZ - i r_xy)/r
  double ezr = 1.0, ezi = 0.0;
  const double exr = dz * ri, exi = -rxy * ri;
  if (rxy > 0) {
    double q = 1.0 / rxy;
    ezr = dy * q;
    ezi = dx * q;
  }
  constexpr int S = m2l_split(P);
  constexpr int kSlots = std::max(M2LPart<P, S + 1, P>::store.slots,
                                  S >= 0 ? M2LPart<P, 0, S >= 0 ? S : P>::store.slots : 0);
  __shared__ double s_mp[kSlots > 0 ? W * kSlots * kWave : 1];
  double *ml = s_mp + (kSlots > 0 ? ((int)threadIdx.x / kWave) * kSlots * kWave + lane : 0);
  const double *src = Msrc + (size_t)j * stride;
  double *dst = Lout + (size_t)tgt * stride;
  m2l_part<P, S + 1, P>(src, quirk != 0, ezr, ezi, exr, exi, ri, active, dst, write, lane, ml);
  if constexpr (S >= 0) {
    __builtin_amdgcn_sched_barrier(0);
    m2l_part<P, 0, S>(src, false, ezr, ezi, exr, exi, ri, active, dst, write, lane, ml);
  }
}

void m2l_init_tables(int p, int quirk) {
  static int done_p = -1, done_q = -1;
  if (done_p == p && done_q == quirk) return;
  double fact[2 * kMaxP + 2];
  fact[0] = 1.0;
  for (int i = 1; i < 2 * kMaxP + 2; i++) fact[i] = fact[i - 1] * i;
  hipMemcpyToSymbol(HIP_SYMBOL(c_fact), fact, sizeof(fact));
  done_p = p;
  done_q = quirk;
}

template <int P>
static void launch(const M2LArgs &a, hipStream_t s) {
  if (a.nchunks <= 0) return;
  constexpr int W = m2l_waves(P);
  const dim3 grid((2 * a.nchunks + W - 1) / W);
  hipLaunchKernelGGL(k_m2l<P>, grid, dim3(64 * W), 0, s, a.chunks, a.nchunks, a.src, a.cX, a.has_sink, a.M,
                     a.Md, a.L, a.Ld, a.quirk, a.stride > 0 ? a.stride : nterm(P));
}

int launch_m2l(int p, const M2LArgs &a, hipStream_t s) {
  m2l_init_tables(p, a.quirk);
  switch (p) {
#define TC_CASE(P)\
  case P:\
    if constexpr (in_shard(P, TC_SHARD)) {\
      launch<P>(a, s);\
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
