// Spin-weighted Legendre ring transforms on gfx950 (FP64).  See legendre.h for the conventions.
//
// Replaces the reference's SHTns synth / analys / synth_grad calls
// (cunusht/sht/GPU_sht_transformer.py:56-96) with per-m three-term recursions:
//   synthesis : one wave per (m, one to three groups of 64 ring pairs); coefficients are wave-uniform
//               and arrive through the scalar cache (small transforms: as vector loads and DPP row
//               broadcasts); the l-loop runs in two phases, first with underflow rescaling while any
//               lane is still below 2^-300, then plain.
//   adjoint   : one wave per (m, one to four groups); per-l sums over the lanes are formed in registers (halving steps over
//               lane swaps) and added up over an m's waves in LDS (up to 512 ring pairs) or, with atomics, in the output,
//               which a last pass scales.
#include "legendre.h"

#include "timing.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <cmath>

namespace nusht {
namespace {

// What a kernel transforms: a spin-0 field, the E component of a spin-s field alone, or E and B.
enum FieldMode { kScalar, kGrad, kFull };

__host__ __device__ inline int l0_of(int m, int s) { return m > s ? m : s; }

constexpr double kThresh = 0x1p300;   // rescale when a scaled value exceeds this
constexpr double kSmall = 0x1p-600;   // one scale step
constexpr double kSeedLo = 0x1p-300;

// ------------------------------------------------------------------ tables
__global__ void k_rec_tables(int lmax, int s, const long* __restrict__ mofs, double2* __restrict__ rec,
                             double* __restrict__ cnorm) {
  int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m > lmax) return;
  int l0 = l0_of(m, s);
  if (l0 > lmax) return;
  long base = mofs[m];
  double cprev = 1.0, ccur = 1.0;
  cnorm[base] = 1.0;
  for (int l = l0; l < lmax; ++l) {
    double alpha, b, gamma;
    if (l == 0) {
      alpha = sqrt(3.0); b = 0.0; gamma = 0.0;
    } else {
      double d1 = sqrt(((l + 1.0) * (l + 1) - (double)m * m) * ((l + 1.0) * (l + 1) - (double)s * s));
      double d0 = sqrt(((double)l * l - (double)m * m) * ((double)l * l - (double)s * s));
      double f = sqrt((2.0 * l + 3) * (2.0 * l + 1));
      alpha = f * (l + 1) / d1;
      b = f * (double)m * s / (l * d1);
      gamma = sqrt((2.0 * l + 3) / (2.0 * l - 1)) * (l + 1) * d0 / (l * d1);
    }
    double cnext = (l == l0) ? 1.0 : gamma * cprev;
    rec[base + (l - l0)] = double2{alpha * ccur / cnext, b * ccur / cnext};
    cnorm[base + (l - l0) + 1] = cnext;
    cprev = ccur;
    ccur = cnext;
  }
}

__device__ inline void renorm(double& v, double& k) {
  while (v != 0.0 && fabs(v) < kSeedLo) { v *= 0x1p600; k -= 1.0; }
}

// Starting values at l0 = max(m, s): u = N_l0 d^l0_{m,-s}, v = N_l0 d^l0_{m,+s}, with scale exponents.
__global__ __launch_bounds__(64) void k_seeds(int lmax, int s, int nslot, int sstride,
                                              const double* __restrict__ slot_theta, double2* __restrict__ st_mu,
                                              double2* __restrict__ st_p, double2* __restrict__ st_k) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nslot) return;
  const double th = slot_theta[i];
  const double sh = sin(0.5 * th), ch = cos(0.5 * th);
  const double ns = sqrt((2.0 * s + 1) / (4.0 * M_PI));
  double u = 0, v = 0, ku = 0, kv = 0;
  // m < s: closed form at l0 = s
  for (int m = 0; m < s && m <= lmax; ++m) {
    double lg = 0.5 * (lgamma(2.0 * s + 1) - lgamma(s + m + 1.0) - lgamma(s - m + 1.0));
    double bin = exp(lg);
    double uu = ns * bin * pow(ch, (double)(s - m)) * pow(sh, (double)(s + m));
    if ((m + s) & 1) uu = -uu;
    double vv = ns * bin * pow(ch, (double)(s + m)) * pow(sh, (double)(s - m));
    const long q = (long)m * sstride + i;
    st_mu[q] = double2{uu, vv};
    st_p[q] = double2{0.0, 0.0};
    st_k[q] = double2{0.0, 0.0};
  }
  if (s > lmax) return;
  // m = s: u = N_s sin^{2s}(th/2), v = N_s cos^{2s}(th/2); then the product recursion in m.
  u = ns; v = ns;
  for (int j = 0; j < 2 * s; ++j) { u *= sh; v *= ch; }
  renorm(u, ku);
  renorm(v, kv);
  {
    const long q = (long)s * sstride + i;
    st_mu[q] = double2{u, v};
    st_p[q] = double2{0.0, 0.0};
    st_k[q] = double2{ku, kv};
  }
  for (int m = s + 1; m <= lmax; ++m) {
    double f = -sqrt(2.0 * m * (2.0 * m + 1) / ((double)m * m - (double)s * s)) * sh * ch;
    u *= f;
    v *= f;
    renorm(u, ku);
    renorm(v, kv);
    const long q = (long)m * sstride + i;
    st_mu[q] = double2{u, v};
    st_p[q] = double2{0.0, 0.0};
    st_k[q] = double2{ku, kv};
  }
}

// Advance each (m, 64-slot group) through the l-range in which every value of the group is
// below 2^-300, in steps of kStartAlign, and store the state at the first l that may contribute.
// Scale exponents never decrease, so a group that is still all-under after a step of kStartAlign
// was all-under at every l inside it; otherwise the step is undone.
constexpr int kStartAlign = 8;

template <bool SP>
__global__ __launch_bounds__(64) void k_advance(int lmax, int s, int nslot, int sstride, int ngroups,
                                                const double* __restrict__ slot_theta, const long* __restrict__ mofs,
                                                const double2* __restrict__ rec_all, double2* __restrict__ st_mu,
                                                double2* __restrict__ st_p, double2* __restrict__ st_k,
                                                int* __restrict__ start) {
  const int m = blockIdx.x / ngroups;
  const int g = blockIdx.x - m * ngroups;
  const int l0 = l0_of(m, s);
  if (l0 > lmax) return;
  const int slot = g * 64 + (int)threadIdx.x;
  const bool valid = slot < nslot;
  const long q = (long)m * sstride + slot;
  double x = 0, mu = 0, mv = 0, pu = 0, pv = 0, ku = 0, kv = 0;
  if (valid) {
    x = cos(slot_theta[slot]);
    const double2 a = st_mu[q], k = st_k[q];
    mu = a.x; ku = k.x;
    if (SP) { mv = a.y; kv = k.y; }
  }
  auto dead = [&]() { return !__any(valid && (ku == 0.0 || (SP && kv == 0.0))); };
  const double2* __restrict__ rec = rec_all + mofs[m];
  int lc = l0;
  while (lc + kStartAlign - 1 <= lmax && dead()) {
    const double smu = mu, smv = mv, spu = pu, spv = pv, sku = ku, skv = kv;
#pragma unroll
    for (int i = 0; i < kStartAlign; ++i) {
      const double2 rc = rec[lc - l0 + i];
      const double t = rc.x * x;
      const double nu = fma(t + rc.y, mu, -pu);
      pu = mu; mu = nu;
      if (SP) {
        const double nv = fma(t - rc.y, mv, -pv);
        pv = mv; mv = nv;
      }
      if (ku < 0.0 && fabs(mu) > kThresh) { mu *= kSmall; pu *= kSmall; ku += 1.0; }
      if (SP && kv < 0.0 && fabs(mv) > kThresh) { mv *= kSmall; pv *= kSmall; kv += 1.0; }
    }
    if (dead()) { lc += kStartAlign; continue; }
    mu = smu; mv = smv; pu = spu; pv = spv; ku = sku; kv = skv;
    break;
  }
  if (valid && lc > l0) {
    st_mu[q] = double2{mu, mv};
    st_p[q] = double2{pu, pv};
    st_k[q] = double2{ku, kv};
  }
  if (threadIdx.x == 0) start[(long)m * ngroups + g] = lc;
}

// ------------------------------------------------------------------ synthesis prep
// coef layout per map b, (m, l):  spin 0: coef[(mofs[m]+l-l0)*NB + b] = a_lm c_l fl_l
//                                 spin s: coef[((mofs[m]+l-l0)*NB + b)*2 + {0,1}] = (W', Wt')
//                                 spin s, E only (ncomp 1): coef[(mofs[m]+l-l0)*NB + b] = W'
//   W' = -(-1)^s c_l (E + iB),  Wt' = -c_l (conj E + i conj B);  with B = 0, Wt' = (-1)^s conj(W').
__global__ void k_prep(int lmax, int s, int nmaps, int nbpad, int ncomp, const double2* __restrict__ alm, long stride_map,
                       const double* __restrict__ fl, const long* __restrict__ mofs,
                       const double* __restrict__ cnorm, double2* __restrict__ coef) {
  const int m = blockIdx.y;
  const int l0 = l0_of(m, s);
  if (l0 > lmax) return;
  const long nalm = (long)(lmax + 1) * (lmax + 2) / 2;
  const long mbase = (long)m * (2 * lmax + 1 - m) / 2;
  const double sg = (s & 1) ? 1.0 : -1.0;  // -(-1)^s
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j <= lmax - l0; j += gridDim.x * blockDim.x) {
    const int l = l0 + j;
    const long q = mofs[m] + j;
    double c = cnorm[q];
    if (fl) c *= fl[l];
    for (int b = 0; b < nbpad; ++b) {
      double2 e{0.0, 0.0}, bb{0.0, 0.0};
      if (b < nmaps) {
        const double2* ab = alm + b * stride_map;
        e = ab[mbase + l];
        if (s != 0 && ncomp > 1) bb = ab[nalm + mbase + l];
      }
      if (s == 0) {
        coef[q * nbpad + b] = double2{e.x * c, e.y * c};
      } else if (ncomp == 1) {
        coef[q * nbpad + b] = double2{sg * c * e.x, sg * c * e.y};
      } else {
        double2 w{e.x - bb.y, e.y + bb.x};
        double2 wt{e.x + bb.y, -e.y + bb.x};
        coef[(q * nbpad + b) * 2] = double2{sg * c * w.x, sg * c * w.y};
        coef[(q * nbpad + b) * 2 + 1] = double2{-c * wt.x, -c * wt.y};
      }
    }
  }
}

// ------------------------------------------------------------------ synthesis kernel
__device__ __forceinline__ void fma2(double2& acc, double2 c, double w) {
  acc.x = fma(c.x, w, acc.x);
  acc.y = fma(c.y, w, acc.y);
}

struct SynthArgs {
  int lmax, s, nslot, sstride, nsb, nmaps;
  const double* slot_theta;
  const int* slot_north;
  const int* slot_south;
  const long* mofs;
  const double2* rec;
  const double2* st_mu;
  const double2* st_p;
  const double2* st_k;
  const int* start;
  const double2* coef;
  double2* G;
  long sm, sr, smap;
};

// Entries a chunked, prefetching l-loop may read past the last l of the last m: three chunks of 8 l (k_synth_row).
constexpr int kSynPad = 32;

// Every 8 l of the slow phase (some lane of the wave still below 2^-300): a chain whose scaled value passed 2^200
// moves up one scale step.  A step of the recursion grows a value by at most sqrt(2 l + 3), so between two checks a
// scaled value stays below 2^300, and what is masked until the next check is below 2^-300.
constexpr double kRescale = 0x1p200;
constexpr int kRescaleL = 8;
static_assert(kStartAlign % kRescaleL == 0, "ring groups join the l-loop at a rescale check");

__device__ __forceinline__ double rescaled_weight(double& mu, double& p, float& k) {
  if (k < 0.f && fabs(mu) > kRescale) { mu *= kSmall; p *= kSmall; k += 1.f; }
  return k == 0.f ? 1.0 : 0.0;
}

// One wave per (m, R groups of 64 ring pairs); each group joins the l-loop at its first contributing l.  The
// coefficients are wave-uniform and arrive through the scalar cache in chunks of CH l, the next chunk's loads issued
// before the current chunk's arithmetic (the tables are padded).  What bounds it: FP64 VALU issue.  Per l and ring pair
// a spin-s E + B map takes 8 FMAs of contraction and 4 of recursion; the chip sustains one FP64 instruction per
// 4.7 - 5.3 cycles and SIMD (clock and operand mix), and the loop runs at 5.6.  R: with one group per wave the
// scalar-cache misses of the coefficient stream were the bound (loads from one fixed address: 8.0 -> 4.6 ms at lmax
// 4095 spin 2), and R groups share one stream.  Measured at lmax 4095, one map, ms: spin 2 R = 1 / 2 / 3 / 4:
// 7.1 / 6.07 / 6.7 / 8.1 (7.4 before, R = 1); spin-1 gradient 4.96 / 4.01 / 4.2 / 4.4 (4.66 before); spin 0 (chunks of
// 4 l) R = 2 / 3 / 4: 3.2 / 2.84 / 2.76 (4.3 before, R = 1).  More groups lengthen the slow phase (4 % of the steps at
// R = 1, 8 % at 2, 15 % at 4) and cost waves per SIMD.
// GR (spin s, E only): the coefficient stream holds W' alone.  Since Wt' = (-1)^s conj(W') and the
// recursion values are real, the -m sums are conjugates of the +m ones: the kernel accumulates
// sum W' mu_u and sum W' mu_v split by the parity of l - l0 (half the contraction of the E + B case) and
// forms the four ring coefficients at the end.
// Two maps (NB = 2) leave registers for one group per wave, and its waves wait for the coefficient stream again.  While
// all of a launch's waves fit the GPU at once, blocks of WPB = 8 waves take neighbouring groups of one m, and seven of
// them find its coefficients in the CU's scalar cache; a longer launch is better off with free blocks, for spin 0 of two
// groups.  Two maps, ms, measured variant of the kernels before (2 or 4 l per chunk, blocks of 1, 4 or 8) / one wave per
// block, 2 l per chunk / now: spin 0 lmax 511 0.061 / 0.078 / 0.054, 900 0.115 / 0.153 / 0.116, 2047 0.88 / 0.98 / 0.68,
// 4095 5.69 / 7.00 / 4.14; spin 2 lmax 511 0.100 / 0.094 / 0.091, 900 0.214 / 0.233 / 0.211, 2047 1.66 / 1.44 / 1.44.
template <bool SP, int NB, int R, int CH, bool GR, int MINW, int WPB = 1>
__global__ __launch_bounds__(64 * WPB, MINW) void k_synth(SynthArgs a) {
  static_assert(SP || !GR, "the gradient-only contraction is a spin-s case");
  static_assert(kRescaleL % CH == 0, "rescale checks fall on chunk starts");
  constexpr int K = (SP && !GR) ? 2 * NB : NB;
  // Blocks are dealt to the XCDs round-robin (block b runs on XCD b % 8).  XCD x takes
  // m = x, x + 8, x + 16, ... with all blocks of one m in a row, so each m's coefficient stream
  // is read through one XCD's L2, and every XCD still starts with its longest m.
  const int blk = blockIdx.x;
  const int j = blk / kNumXcd;
  const int m = (blk - j * kNumXcd) + kNumXcd * (j / a.nsb);
  const int sb = (j % a.nsb) * WPB + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int L = a.lmax;
  if (m > L) return;
  const int l0 = l0_of(m, a.s);
  // the launch may carry empty slot groups (odd block count per m, see launch_synth)
  if (l0 > L || sb * 64 * R >= a.nslot) return;
  const int lane = threadIdx.x & 63;
  const int ng = (a.nslot + 63) >> 6;

  double x[R], mu_u[R], mu_v[R], pu[R], pv[R];
  float ku[R], kv[R];
  int lst[R];  // first contributing l of each group (past lmax: never)
  int lc = L + 1, lall = l0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int g = sb * R + r;
    const int slot = g * 64 + lane;
    lst[r] = __builtin_amdgcn_readfirstlane(g < ng ? a.start[(long)m * ng + g] : L + 1);
    lc = min(lc, lst[r]);
    if (lst[r] <= L) lall = max(lall, lst[r]);
    x[r] = slot < a.nslot ? cos(a.slot_theta[slot]) : 0.0;
    mu_u[r] = mu_v[r] = pu[r] = pv[r] = 0.0;
    ku[r] = kv[r] = 0.f;
  }
  lc = __builtin_amdgcn_readfirstlane(lc);
  lall = __builtin_amdgcn_readfirstlane(lall);

  const long base = a.mofs[m];
  const double2* __restrict__ rec = a.rec + base;
  const double2* __restrict__ cf = a.coef + base * K;

  // spin 0: P / A even / odd sums.  Spin s: P (+m north), N (-m north), A (+m south), B (-m south), the south-ring
  // sign alternation inside.  GR: sums of W' mu_u over even / odd l - l0 in P / N, of W' mu_v in A / B.
  double2 P[R][NB], N[R][NB], A[R][NB], B[R][NB];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) P[r][b] = N[r][b] = A[r][b] = B[r][b] = double2{0.0, 0.0};

  struct Buf {
    double2 rc[CH];
    double2 cw[CH][K];
  };
  auto load = [&](int l, Buf& b) {
    const int j0 = l - l0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      b.rc[i] = rec[j0 + i];
#pragma unroll
      for (int k = 0; k < K; ++k) b.cw[i][k] = cf[(long)(j0 + i) * K + k];
    }
  };
  double fu[R], fv[R];  // 1, or 0 while the lane's chain is below range (slow phase)
  // groups starting at l load their state; chains that left their scale step move up
  auto join = [&](int l) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (l == lst[r]) {
        const int slot = (sb * R + r) * 64 + lane;
        if (slot < a.nslot) {
          const long q = (long)m * a.sstride + slot;
          const double2 sm = a.st_mu[q], sp = a.st_p[q], sk = a.st_k[q];
          mu_u[r] = sm.x; pu[r] = sp.x; ku[r] = (float)sk.x;
          if (SP) { mu_v[r] = sm.y; pv[r] = sp.y; kv[r] = (float)sk.y; }
        }
      }
      fu[r] = rescaled_weight(mu_u[r], pu[r], ku[r]);
      fv[r] = SP ? rescaled_weight(mu_v[r], pv[r], kv[r]) : 0.0;
    }
  };
  // One chunk (the first l at even l - l0).  SLOW: some lane may still be below the
  // representable range (masked contributions); FULL: all CH l <= L.
  auto chunk = [&](int l, const Buf& bf, auto slow_tag, auto full_tag) {
    constexpr bool SLOW = decltype(slow_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (!FULL && l + i > L) break;
      const bool odd = (i & 1) != 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double wu = mu_u[r], wv = mu_v[r];
        if (SLOW) { wu *= fu[r]; if (SP) wv *= fv[r]; }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if (!SP) {
            if (odd) fma2(A[r][b], bf.cw[i][b], wu); else fma2(P[r][b], bf.cw[i][b], wu);
          } else if (GR) {
            const double2 w = bf.cw[i][b];
            if (odd) { fma2(N[r][b], w, wu); fma2(B[r][b], w, wv); }
            else { fma2(P[r][b], w, wu); fma2(A[r][b], w, wv); }
          } else {
            const double2 w = bf.cw[i][2 * b], wt = bf.cw[i][2 * b + 1];
            fma2(P[r][b], w, wu);
            fma2(N[r][b], wt, wv);
            if (odd) { fma2(A[r][b], w, -wv); fma2(B[r][b], wt, -wu); }
            else { fma2(A[r][b], w, wv); fma2(B[r][b], wt, wu); }
          }
        }
        // the step past l = lmax reads a padded table entry; its result is never used
        const double t = bf.rc[i].x * x[r];
        const double nu = SP ? fma(t + bf.rc[i].y, mu_u[r], -pu[r]) : fma(t, mu_u[r], -pu[r]);
        pu[r] = mu_u[r]; mu_u[r] = nu;
        if (SP) {
          const double nv = fma(t - bf.rc[i].y, mu_v[r], -pv[r]);
          pv[r] = mu_v[r]; mu_v[r] = nv;
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // keeps the next l's products out of this one's registers
    }
  };
  auto any_under = [&]() {
    bool under = false;
#pragma unroll
    for (int r = 0; r < R; ++r) under |= (ku[r] < 0.f) || (kv[r] < 0.f);
    return __any(under);
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  if (lc <= L) {
    Buf cur, nxt;
    load(lc, cur);
    // slow phase: while a group has still to join or some lane is below 2^-300
    while (lc <= L && (lc <= lall || any_under())) {
      if (((lc - l0) & (kRescaleL - 1)) == 0) join(lc);
      load(lc + CH, nxt);
      if (lc + CH - 1 <= L) chunk(lc, cur, T_{}, T_{});
      else chunk(lc, cur, T_{}, F_{});
      cur = nxt;
      lc += CH;
    }
    // fast phase, two chunks per iteration so that the two buffers alternate without copies
    while (lc + 2 * CH - 1 <= L) {
      load(lc + CH, nxt);
      chunk(lc, cur, F_{}, T_{});
      load(lc + 2 * CH, cur);
      chunk(lc + CH, nxt, F_{}, T_{});
      lc += 2 * CH;
    }
    if (lc + CH - 1 <= L) {
      load(lc + CH, nxt);
      chunk(lc, cur, F_{}, T_{});
      cur = nxt;
      lc += CH;
    }
    if (lc <= L) chunk(lc, cur, F_{}, F_{});
  }

  const double sg0 = ((l0 + m) & 1) ? -1.0 : 1.0;  // (-1)^{l+m} for even (l - l0)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int slot = (sb * R + r) * 64 + lane;
    if (slot >= a.nslot) continue;
    const int rn = a.slot_north[slot];
    const int rs = a.slot_south[slot];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b >= a.nmaps) break;
      double2* Gb = a.G + b * a.smap;
      if (!SP) {
        Gb[(long)m * a.sm + (long)rn * a.sr] = cadd(P[r][b], A[r][b]);
        if (rs >= 0) Gb[(long)m * a.sm + (long)rs * a.sr] = cscale(csub(P[r][b], A[r][b]), sg0);
      } else {
        double2 pN, mN, pS, mS;
        if (GR) {
          // north +m: sum W' mu_u; north -m: (-1)^s conj(sum W' mu_v); south +m: sg0 (even - odd of sum W' mu_v);
          // south -m: sg0 (-1)^s conj(even - odd of sum W' mu_u)
          const double ss = (a.s & 1) ? -1.0 : 1.0;
          pN = cadd(P[r][b], N[r][b]);
          mN = cscale(cconj(cadd(A[r][b], B[r][b])), ss);
          pS = cscale(csub(A[r][b], B[r][b]), sg0);
          mS = cscale(cconj(csub(P[r][b], N[r][b])), sg0 * ss);
        } else {
          pN = P[r][b];
          mN = N[r][b];
          pS = cscale(A[r][b], sg0);
          mS = cscale(B[r][b], sg0);
        }
        const long rowp = (long)(L + m) * a.sm, rowm = (long)(L - m) * a.sm;
        Gb[rowp + (long)rn * a.sr] = pN;
        if (rs >= 0) Gb[rowp + (long)rs * a.sr] = pS;
        if (m > 0) {
          Gb[rowm + (long)rn * a.sr] = mN;
          if (rs >= 0) Gb[rowm + (long)rs * a.sr] = mS;
        }
      }
    }
  }
}

// ------------------------------------------------------------------ synthesis with few waves
// Broadcast of lane I of each 16-lane row to the whole row.
template <int I>
__device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + I, 0xF, 0xF, true);
}

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// acc += (c of lanes I, I + 1 of the row) * w: the complex coefficient is the DPP operand of the two FMAs.  A DPP
// read needs two wait states after a VALU write of its source (the buffers are copied in the slow phase).
template <int I, bool NEG>
__device__ __forceinline__ void row_fma2(double2& acc, double c, double w) {
  if constexpr (NEG)
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, -%2, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
        : "+v"(acc.x), "+v"(acc.y) : "v"(c), "v"(w), "n"(I), "n"(I + 1));
  else
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %2, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
        : "+v"(acc.x), "+v"(acc.y) : "v"(c), "v"(w), "n"(I), "n"(I + 1));
}

// One map, one wave per (m, group of 64 ring pairs) and, for spin s, chain (u: north +m and south -m; v: north -m and
// south +m), for launches that leave SIMDs with one or two waves: there a wave issues one FP64 instruction per
// 8 - 9 cycles and nothing hides a scalar load, which returns out of order, so every wait covers all of them.  The
// coefficients come as vector loads instead, 16 doubles per register in each 16-lane row (8 l of the recursion
// table, 4 or 8 of the map's), three chunks of 8 l deep, and reach the arithmetic as DPP row broadcasts; the two
// chains run side by side in two waves.  With the coefficient preparation, ms, against the faster of k_synth with few
// and with more groups: lmax 255 spin 2 0.033 -> 0.015, spin-1 gradient 0.027 -> 0.017, spin 0 0.022 -> 0.013;
// lmax 1000 0.218 -> 0.160, 0.182 -> 0.125, 0.118 -> 0.070.  For spin s k_synth is the faster one from lmax 1200 on
// (two broadcasts per l and chain less): kernel alone, spin 2, here / few / more groups, lmax 1200 0.291 / 0.292 / 0.346,
// 1500 0.53 / 0.49 / 0.52, 2047 1.16 / 1.04 / 1.07, 4095 7.5 / 7.1 / 6.1; spin 0 4095 2.49 / 3.23 / 2.74.
template <int MODE>
__global__ __launch_bounds__(64) void k_synth_row(SynthArgs a) {
  constexpr bool SP = MODE != kScalar;
  constexpr int NC = SP ? 2 : 1;              // chains
  constexpr int CW = MODE == kFull ? 4 : 2;  // coefficient doubles per l
  constexpr int CH = 8;
  const int blk = blockIdx.x;
  const int j = blk / kNumXcd;
  const int m = (blk - j * kNumXcd) + kNumXcd * (j / (a.nsb * NC));
  const int sc = j % (a.nsb * NC);
  const int sb = sc / NC;
  const bool vch = SP && (sc % NC);
  const int L = a.lmax;
  if (m > L) return;
  const int l0 = l0_of(m, a.s);
  if (l0 > L || sb * 64 >= a.nslot) return;
  const int lane = threadIdx.x, row = lane & 15;
  int lc = a.start[(long)m * ((a.nslot + 63) >> 6) + sb];
  const int slot = sb * 64 + lane;
  double x = 0.0, mu = 0.0, p = 0.0;
  float kk = 0.f;
  if (slot < a.nslot) {
    const long q = (long)m * a.sstride + slot;
    x = cos(a.slot_theta[slot]);
    const double2 sm = a.st_mu[q], sp = a.st_p[q], sk = a.st_k[q];
    mu = vch ? sm.y : sm.x;
    p = vch ? sp.y : sp.x;
    kk = (float)(vch ? sk.y : sk.x);
  }
  const long base = a.mofs[m];
  const double* __restrict__ rec = reinterpret_cast<const double*>(a.rec + base) + row;
  // the v chain takes (W~', W') where the u chain takes (W', W~')
  const double* __restrict__ cf =
      reinterpret_cast<const double*>(a.coef) + base * CW + (MODE == kFull && vch ? row ^ 2 : row);
  const bool flip = vch && (row & 1);  // the v chain's -B_l
  double2 P{0.0, 0.0}, Q{0.0, 0.0};    // full: north and (sign alternating) south sums; else even and odd sums
  struct Buf {
    double rc, cw[CW / 2];
  };
  auto load = [&](int l, Buf& b) {
    const long j0 = l - l0;
    b.rc = rec[2 * j0];
#pragma unroll
    for (int k = 0; k < CW / 2; ++k) b.cw[k] = cf[j0 * CW + 16 * k];
  };
  auto chunk = [&](int l, const Buf& bf, double f, auto slow_tag, auto full_tag) {
    constexpr bool SLOW = decltype(slow_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
    const double rc = flip ? -bf.rc : bf.rc;
    static_for<0, CH>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr bool odd = (i & 1) != 0;
      if (!FULL && l + i > L) return;
      const double w = SLOW ? mu * f : mu;
      if constexpr (MODE == kFull) {
        row_fma2<(i & 3) * 4, false>(P, bf.cw[i >> 2], w);
        row_fma2<(i & 3) * 4 + 2, odd>(Q, bf.cw[i >> 2], w);
      } else {
        row_fma2<2 * i, false>(odd ? Q : P, bf.cw[0], w);
      }
      const double t = SP ? fma(row_bcast<2 * i>(rc), x, row_bcast<2 * i + 1>(rc)) : row_bcast<2 * i>(rc) * x;
      const double nu = fma(t, mu, -p);
      p = mu;
      mu = nu;
    });
    __builtin_amdgcn_sched_barrier(0);  // the next chunk's waits stay behind this chunk
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  if (lc <= L) {
    Buf b0, b1, b2;
    load(lc, b0);
    load(lc + CH, b1);
    while (lc <= L && __any(kk < 0.f)) {
      const double f = rescaled_weight(mu, p, kk);
      load(lc + 2 * CH, b2);
      if (lc + CH - 1 <= L) chunk(lc, b0, f, T_{}, T_{});
      else chunk(lc, b0, f, T_{}, F_{});
      b0 = b1;
      b1 = b2;
      lc += CH;
    }
    while (lc + 3 * CH - 1 <= L) {
      load(lc + 2 * CH, b2);
      chunk(lc, b0, 1.0, F_{}, T_{});
      load(lc + 3 * CH, b0);
      chunk(lc + CH, b1, 1.0, F_{}, T_{});
      load(lc + 4 * CH, b1);
      chunk(lc + 2 * CH, b2, 1.0, F_{}, T_{});
      lc += 3 * CH;
    }
    while (lc + CH - 1 <= L) {
      load(lc + 2 * CH, b2);
      chunk(lc, b0, 1.0, F_{}, T_{});
      b0 = b1;
      b1 = b2;
      lc += CH;
    }
    if (lc <= L) chunk(lc, b0, 1.0, F_{}, F_{});
  }
  if (slot >= a.nslot) return;
  const double sg0 = ((l0 + m) & 1) ? -1.0 : 1.0;
  const int rn = a.slot_north[slot], rs = a.slot_south[slot];
  double2 north, south;
  if constexpr (MODE == kFull) {
    north = P;
    south = cscale(Q, sg0);
  } else {
    north = cadd(P, Q);
    south = cscale(csub(P, Q), sg0);
    if constexpr (MODE == kGrad) {  // the -m rows (north of the v chain, south of the u chain): (-1)^s conj
      const double ss = (a.s & 1) ? -1.0 : 1.0;
      if (vch) north = cscale(cconj(north), ss);
      else south = cscale(cconj(south), ss);
    }
  }
  const long rowp = (long)(SP ? L + m : m) * a.sm, rowm = (long)(L - m) * a.sm;
  if (!vch || m > 0) a.G[(vch ? rowm : rowp) + (long)rn * a.sr] = north;
  if (rs >= 0 && (!SP || vch || m > 0)) a.G[((SP && !vch) ? rowm : rowp) + (long)rs * a.sr] = south;
}

// ------------------------------------------------------------------ synthesis on the matrix cores
// For 4 maps per launch the contraction over l is a GEMM per m: per chunk of 4 l,
// (64 ring pairs x 4 l) x (4 l x 16 columns), done with v_mfma_f64_16x16x4_f64 while the VALU
// runs the recursion.  Columns, 4 per map b, with s_l = (-1)^{l+m}:
//   spin s, u chain: Re W_b, Im W_b, Re s_l Wt_b, Im s_l Wt_b    (north +m, south -m)
//           v chain: Re Wt_b, Im Wt_b, Re s_l W_b, Im s_l W_b    (north -m, south +m)
//   spin 0, u chain: Re a_b, Im a_b, Re s_l a_b, Im s_l a_b      (north, south)
// A launch takes 4 NS maps (NS = 1 or 2 groups of 16 columns; the recursion and the A tiles serve both groups).
// The table holds, per m and per block q of 4 l (l = l0 + 4q + k), the values once: spin s
// [k][b][Re W, Im W, Re Wt, Im Wt] (64 NS doubles), spin 0 [k][b][Re a, Im a] (32 NS), b < 4 NS.  Lane j + 16k of
// group g's B operand (column j = 4b' + c of map b = 4g + b' at l0 + 4q + k) reads entry (k, b, c) for the u
// chain and (k, b, c ^ 2) for the v chain (spin s), (k, b, c & 1) for spin 0, and negates it when c >= 2 and
// l + m is odd; blocks start at l0 + 4q, so that sign is fixed per lane.  Entries past lmax are zero.

// Operand layouts of v_mfma_f64_16x16x4_f64 on gfx950 (64 lanes):
//   A[i][k] in lane i + 16k, B[k][j] in lane j + 16k, D[i][j] in register i / 4 of lane j + 16 (i % 4).

// One thread per (block q of 4 l, k, map b): map b's entry at l = l0 + 4q + k, one 32-byte store (16 for spin 0;
// consecutive threads write consecutive entries).  Block row y serves m = y and m = lmax - y, whose tables together
// have about lmax + 2 rows of l, so no block row is idle.
template <int NS>
__global__ void k_prep4(int lmax, int s, int nmaps, int ncomp, AlmPtrs8 alm,
                        const double* __restrict__ fl, const long* __restrict__ mofs, const long* __restrict__ mblk,
                        const double* __restrict__ cnorm, double* __restrict__ coef) {
  const int nc = s ? 2 : 1;
  const long nalm = (long)(lmax + 1) * (lmax + 2) / 2;
  const double sg = (s & 1) ? 1.0 : -1.0;  // -(-1)^s
  for (int pass = 0; pass < 2; ++pass) {
    const int m = pass == 0 ? (int)blockIdx.y : lmax - (int)blockIdx.y;
    if (pass == 1 && m <= (int)blockIdx.y) break;  // the middle m has no partner
    const int l0 = l0_of(m, s);
    if (l0 > lmax) continue;
    const int nl = lmax - l0 + 1;
    constexpr int NM = 4 * NS, LNM = NS == 1 ? 2 : 3;  // maps per launch and log2
    const long nthr = (long)((nl + 3) >> 2) * 4 * NM;
    const long mbase = (long)m * (2 * lmax + 1 - m) / 2;
    double* out = coef + mblk[m] * nc * 32 * NS;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < nthr; t += (long)gridDim.x * blockDim.x) {
      const int b = (int)(t & (NM - 1)), k = (int)((t >> LNM) & 3);
      const long q = t >> (LNM + 2);
      const int jj = (int)(4 * q + k);
      const int l = l0 + jj;
      double2 w{0.0, 0.0}, wt{0.0, 0.0};  // spin 0: w = a_lm c_l
      if (l <= lmax && b < nmaps) {
        double cl = cnorm[mofs[m] + jj];
        if (fl) cl *= fl[l];
        const double2* ab = alm.p[0];  // selects, not an indexed read of the argument array
#pragma unroll
        for (int u = 1; u < NM; ++u) ab = b == u ? alm.p[u] : ab;
        const double2 ev = ab[mbase + l];
        if (s == 0) {
          w = double2{cl * ev.x, cl * ev.y};
        } else {
          const double2 bv = ncomp > 1 ? ab[nalm + mbase + l] : double2{0.0, 0.0};
          w = double2{sg * cl * (ev.x - bv.y), sg * cl * (ev.y + bv.x)};
          wt = double2{-cl * (ev.x + bv.y), -cl * (-ev.y + bv.x)};
        }
      }
      double2* o = reinterpret_cast<double2*>(out + q * nc * 32 * NS + (k * NM + b) * nc * 2);
      o[0] = w;
      if (s != 0) o[1] = wt;
    }
  }
}

typedef double v4d_t __attribute__((ext_vector_type(4)));

// 4 x 4 transpose of (register k, row g of 16 lanes): afterwards register g holds in lane i + 16k
// what register k held in lane 16g + i (the A-operand tile of ring pairs 16g .. 16g + 15).
__device__ __forceinline__ void transpose_rows(double (&u)[4]) {
  unsigned lo[4], hi[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    lo[k] = (unsigned)__double2loint(u[k]);
    hi[k] = (unsigned)__double2hiint(u[k]);
  }
  auto sw32 = [](unsigned& x, unsigned& y) {
    auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);  // x upper half <-> y lower half
    x = r[0]; y = r[1];
  };
  auto sw16 = [](unsigned& x, unsigned& y) {
    auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);  // x odd rows <-> y even rows
    x = r[0]; y = r[1];
  };
  sw32(lo[0], lo[2]); sw32(lo[1], lo[3]); sw16(lo[0], lo[1]); sw16(lo[2], lo[3]);
  sw32(hi[0], hi[2]); sw32(hi[1], hi[3]); sw16(hi[0], hi[1]); sw16(hi[2], hi[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k) u[k] = __hiloint2double((int)hi[k], (int)lo[k]);
}

template <bool SP, int NS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NS == 1 ? 3 : 2))) void k_synth_mfma(
    SynthArgs a, const double* __restrict__ coef4, const long* __restrict__ mblk) {
  constexpr int NC = SP ? 2 : 1;
  // same block -> (m, slot group) mapping as k_synth with one wave per block
  const int blk = blockIdx.x;
  const int j = blk / kNumXcd;
  const int m = (blk - j * kNumXcd) + kNumXcd * (j / a.nsb);
  const int sb = j % a.nsb;
  const int L = a.lmax;
  if (m > L) return;
  const int l0 = l0_of(m, a.s);
  if (l0 > L || sb * 64 >= a.nslot) return;
  const int lane = threadIdx.x & 63;
  const int lstart = a.start[(long)m * ((a.nslot + 63) >> 6) + sb];

  const int slot = sb * 64 + lane;
  double x = 0, mu_u = 0, mu_v = 0, pu = 0, pv = 0, ku = 0, kv = 0;
  if (slot < a.nslot) {
    const long q = (long)m * a.sstride + slot;
    x = cos(a.slot_theta[slot]);
    const double2 sm = a.st_mu[q], sp = a.st_p[q], sk = a.st_k[q];
    mu_u = sm.x; pu = sp.x; ku = sk.x;
    if (SP) { mu_v = sm.y; pv = sp.y; kv = sk.y; }
  }
  const double2* __restrict__ rec = a.rec + a.mofs[m];
  const double* __restrict__ cb = coef4 + mblk[m] * NC * 32 * NS;
  // this lane's B entries in a block for group 0 (u chain, v chain; group g adds 16 g, 8 g for spin 0) and their
  // sign bit: column c = lane & 3 >= 2 at odd l + m, l = l0 + 4q + (lane >> 4)
  const int c4 = lane & 3;
  const int eu = SP ? (lane >> 4) * 16 * NS + (lane & 15) : (lane >> 4) * 8 * NS + ((lane & 15) >> 2) * 2 + (c4 & 1);
  const int ev = eu ^ 2;
  const unsigned sgnb = (c4 >= 2 && ((l0 + (lane >> 4) + m) & 1)) ? 0x80000000u : 0u;
  auto sgn = [&](double v) {
    return __hiloint2double(__double2hiint(v) ^ (int)sgnb, __double2loint(v));
  };

  v4d_t Du[NS][4], Dv[NS][4];
#pragma unroll
  for (int h = 0; h < NS; ++h)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      Du[h][g] = v4d_t{0.0, 0.0, 0.0, 0.0};
      Dv[h][g] = v4d_t{0.0, 0.0, 0.0, 0.0};
    }
  struct Buf {
    double2 rc[4];
    double bu[NS], bv[NS];
  };
  auto load = [&](int lc, Buf& b) {
    const int jl = lc - l0;
#pragma unroll
    for (int i = 0; i < 4; ++i) b.rc[i] = rec[jl + 1 + i];  // the steps from l + 1 (state one step ahead)
    const double* blkp = cb + (long)(jl >> 2) * NC * 32 * NS;
#pragma unroll
    for (int h = 0; h < NS; ++h) {
      b.bu[h] = blkp[eu + h * (SP ? 16 : 8)];
      if (SP) b.bv[h] = blkp[ev + h * 16];
    }
  };
  // GRP: the map groups a chunk accumulates (-1 all, else that group alone)
  auto chunk = [&](int lc, const Buf& bf, auto slow_tag, auto full_tag, auto grp_tag) {
    constexpr bool SLOW = decltype(slow_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
    constexpr int GRP = decltype(grp_tag)::value;
    double U[4], V[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!FULL && lc + i > L) { U[i] = 0.0; V[i] = 0.0; continue; }  // zero weight past lmax
      double wu = pu, wv = pv;  // the value at lc + i
      if (SLOW) { wu = ku == 0.0 ? wu : 0.0; wv = kv == 0.0 ? wv : 0.0; }
      U[i] = wu; V[i] = wv;
      const double t = bf.rc[i].x * x;
      const double nu = fma(t + bf.rc[i].y, mu_u, -pu);
      pu = mu_u; mu_u = nu;
      if (SP) {
        const double nv = fma(t - bf.rc[i].y, mu_v, -pv);
        pv = mu_v; mu_v = nv;
      }
      if (SLOW) {
        if (ku < 0.0 && fabs(mu_u) > kThresh) { mu_u *= kSmall; pu *= kSmall; ku += 1.0; }
        if (SP && kv < 0.0 && fabs(mu_v) > kThresh) { mu_v *= kSmall; pv *= kSmall; kv += 1.0; }
      }
    }
    transpose_rows(U);
#pragma unroll
    for (int h = 0; h < NS; ++h) {
      if (GRP >= 0 && h != GRP) continue;
      const double bu = sgn(bf.bu[h]);
#pragma unroll
      for (int g = 0; g < 4; ++g) Du[h][g] = __builtin_amdgcn_mfma_f64_16x16x4f64(U[g], bu, Du[h][g], 0, 0, 0);
    }
    if (SP) {
      transpose_rows(V);
#pragma unroll
      for (int h = 0; h < NS; ++h) {
        if (GRP >= 0 && h != GRP) continue;
        const double bv = sgn(bf.bv[h]);
#pragma unroll
        for (int g = 0; g < 4; ++g) Dv[h][g] = __builtin_amdgcn_mfma_f64_16x16x4f64(V[g], bv, Dv[h][g], 0, 0, 0);
      }
    }
  };
  auto any_under = [&]() { return __any((ku < 0.0) || (kv < 0.0)); };
  using T_ = std::true_type;
  using F_ = std::false_type;
  // The l-loop runs one recursion step ahead: at the first l of a chunk it holds (mu, p) = (mu_{l+1}, mu_l), and
  // the chunk's four A values are p before each step, so none of them is still part of the recursion state when
  // the transposes overwrite them in place (no register copies).  The step to l + 1 is made here; a step past
  // lmax reads a padded or neighbouring table entry and its result is never used.
  {
    const double2 rc0 = rec[lstart - l0];
    const double t = rc0.x * x;
    const double nu = fma(t + rc0.y, mu_u, -pu);
    pu = mu_u; mu_u = nu;
    if (SP) {
      const double nv = fma(t - rc0.y, mu_v, -pv);
      pv = mu_v; mu_v = nv;
    }
    if (ku < 0.0 && fabs(mu_u) > kThresh) { mu_u *= kSmall; pu *= kSmall; ku += 1.0; }
    if (SP && kv < 0.0 && fabs(mu_v) > kThresh) { mu_v *= kSmall; pv *= kSmall; kv += 1.0; }
  }
  using GA_ = std::integral_constant<int, -1>;
  int lc = lstart;
  Buf cur, nxt;
  load(lc, cur);
  // slow phase (some lane below 2^-300); the next chunk's coefficients are loaded before the current chunk is
  // computed.  With two map groups it runs once per group, the recursion restarting from its saved state for the
  // second: a group's accumulators are then either still zero or untouched in the loop, and the loop keeps only
  // the other group's in registers (both together with the rescaling state exceed the two-wave register budget).
  // The second pass runs the same number of chunks, since the phase's end depends on the recursion alone.
  auto slow_phase = [&](auto grp_tag, int lend) {
    while (lend < 0 ? (lc <= L && any_under()) : lc < lend) {
      load(lc + 4, nxt);
      if (lc + 3 <= L) chunk(lc, cur, T_{}, T_{}, grp_tag);
      else chunk(lc, cur, T_{}, F_{}, grp_tag);
      cur = nxt;
      lc += 4;
    }
  };
  if constexpr (NS == 1) {
    slow_phase(GA_{}, -1);
  } else {
    const double s_mu_u = mu_u, s_pu = pu, s_mu_v = mu_v, s_pv = pv, s_ku = ku, s_kv = kv;
    slow_phase(std::integral_constant<int, 0>{}, -1);
    const int lend = lc;
    if (lend > lstart) {
      mu_u = s_mu_u; pu = s_pu; mu_v = s_mu_v; pv = s_pv; ku = s_ku; kv = s_kv;
      lc = lstart;
      load(lc, cur);
      slow_phase(std::integral_constant<int, 1>{}, lend);
    }
  }
  // two chunks per iteration, so the two buffers alternate without copies (loads reach at most one 4-l block
  // past lmax, as the single-chunk step does)
  while (lc + 7 <= L) {
    load(lc + 4, nxt);
    chunk(lc, cur, F_{}, T_{}, GA_{});
    load(lc + 8, cur);
    chunk(lc + 4, nxt, F_{}, T_{}, GA_{});
    lc += 8;
  }
  if (lc + 3 <= L) {
    load(lc + 4, nxt);
    chunk(lc, cur, F_{}, T_{}, GA_{});
    cur = nxt;
    lc += 4;
  }
  if (lc <= L) chunk(lc, cur, F_{}, F_{}, GA_{});

  // epilogue: lane = jc + 16 qq holds column jc of group h (map 4 h + jc / 4) for ring pairs 16 g + 4 r + qq
  // (register r)
  const int jc = lane & 15, qq = lane >> 4;
  const int c = jc & 3;
  const int part = c & 1;
#pragma unroll
  for (int h = 0; h < NS; ++h) {
    const int b = 4 * h + (jc >> 2);
    if (b >= a.nmaps) continue;
    double* Gd = reinterpret_cast<double*>(a.G + b * a.smap);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int sl = sb * 64 + 16 * g + 4 * r + qq;
        if (sl >= a.nslot) continue;
        const int rn = a.slot_north[sl];
        const int rs = a.slot_south[sl];
        const double du = Du[h][g][r];
        if (!SP) {
          if (c < 2) Gd[((long)m * a.sm + (long)rn * a.sr) * 2 + part] = du;
          else if (rs >= 0) Gd[((long)m * a.sm + (long)rs * a.sr) * 2 + part] = du;
        } else {
          const double dv = Dv[h][g][r];
          const long rowp = (long)(L + m) * a.sm, rowm = (long)(L - m) * a.sm;
          if (c < 2) {
            Gd[(rowp + (long)rn * a.sr) * 2 + part] = du;                        // north +m
            if (m > 0) Gd[(rowm + (long)rn * a.sr) * 2 + part] = dv;            // north -m
          } else if (rs >= 0) {
            Gd[(rowp + (long)rs * a.sr) * 2 + part] = dv;                        // south +m
            if (m > 0) Gd[(rowm + (long)rs * a.sr) * 2 + part] = du;            // south -m
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------ adjoint kernel
// Lane exchanges of the sums over a wave's 64 ring pairs.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, false);
  hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
constexpr int kDppQuadXor2 = 0x4E, kDppQuadXor1 = 0xB1, kDppQuadSame = 0xE4;
constexpr int kDppRowRor8 = 0x128, kDppRowShl4 = 0x104, kDppRowShr4 = 0x114;

// a + (a of lane ^ OFF) in the lanes with (lane & OFF) == 0, b + (b of lane ^ OFF) in the others.
// OFF = 32 or 16: one swap of the register pair per half does it.  permlane32_swap(x, y) leaves x = (own x | y of
// lane - 32) and y = (x of lane + 32 | own y) over the two halves, permlane16_swap the same over the row pairs, so
// x + y is the wanted sum in every lane.  OFF = 8 or 4: DPP moves inside the 16-lane row, the bank mask (groups of 4
// lanes) choosing whose value a lane takes.
template <int OFF>
__device__ __forceinline__ double pair_sum(double a, double b) {
  static_assert(OFF == 32 || OFF == 16 || OFF == 8 || OFF == 4, "lane exchanges at offsets 32, 16, 8 and 4");
  const int alo = __double2loint(a), ahi = __double2hiint(a), blo = __double2loint(b), bhi = __double2hiint(b);
  if constexpr (OFF == 32) {
    const auto rl = __builtin_amdgcn_permlane32_swap((unsigned)alo, (unsigned)blo, false, false);
    const auto rh = __builtin_amdgcn_permlane32_swap((unsigned)ahi, (unsigned)bhi, false, false);
    return __hiloint2double((int)rh[0], (int)rl[0]) + __hiloint2double((int)rh[1], (int)rl[1]);
  } else if constexpr (OFF == 16) {
    const auto rl = __builtin_amdgcn_permlane16_swap((unsigned)alo, (unsigned)blo, false, false);
    const auto rh = __builtin_amdgcn_permlane16_swap((unsigned)ahi, (unsigned)bhi, false, false);
    return __hiloint2double((int)rh[0], (int)rl[0]) + __hiloint2double((int)rh[1], (int)rl[1]);
  } else {
    constexpr int kFromUp = OFF == 8 ? kDppRowRor8 : kDppRowShl4;    // the value of lane + OFF
    constexpr int kFromDown = OFF == 8 ? kDppRowRor8 : kDppRowShr4;  // the value of lane - OFF
    constexpr int kLow = OFF == 8 ? 0x3 : 0x5, kHigh = OFF == 8 ? 0xC : 0xA;
    const auto partner = [&](int x, int y) {
      const int t = __builtin_amdgcn_update_dpp(0, x, kFromUp, 0xF, kLow, false);
      return __builtin_amdgcn_update_dpp(t, y, kFromDown, 0xF, kHigh, false);
    };
    const auto own = [&](int x, int y) { return __builtin_amdgcn_update_dpp(x, y, kDppQuadSame, 0xF, kHigh, false); };
    return __hiloint2double(own(ahi, bhi), own(alo, blo)) + __hiloint2double(partner(ahi, bhi), partner(alo, blo));
  }
}

// Sums of 16 values per lane over the wave: halving steps (each lane keeps half of the values, added to its
// partner's) over lane bits 5 to 2, then plain sums over the quad; lane ln ends up with the sum of value ln >> 2.
__device__ __forceinline__ double wave_sums(double (&v)[16]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = pair_sum<32>(v[i], v[i + 8]);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pair_sum<16>(v[i], v[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) v[i] = pair_sum<8>(v[i], v[i + 2]);
  double r = pair_sum<4>(v[0], v[1]);
  r += dpp_mov<kDppQuadXor2>(r);
  r += dpp_mov<kDppQuadXor1>(r);
  return r;
}

struct AdjArgs {
  int lmax, s, nslot, sstride, ngroups, nsb;
  const double* slot_theta;
  const int* slot_north;
  const int* slot_south;
  const long* mofs;
  const double2* rec;
  const double2* st_mu;
  const double2* st_p;
  const double2* st_k;
  const int* start;
  const double2* G;
  long sm, sr;
  const double* cnorm;
  double2* alm;
};

// The sums over ring pairs -> alm, c the coefficient's norm (see k_adjoint).
template <int MODE>
__device__ __forceinline__ double2 adjoint_coef(int m, double c, double2 t) {
  if constexpr (MODE == kScalar) return double2{c * t.x, m == 0 ? 0.0 : c * t.y};
  else return cscale(t, -0.5 * c);
}
__device__ __forceinline__ void adjoint_coef(int s, double c, double2 x, double2 y, double2& e, double2& b) {
  const double2 X = cscale(x, (s & 1) ? -c : c), Y = cscale(y, c);
  e = double2{-0.5 * (X.x + Y.x), -0.5 * (X.y + Y.y)};
  b = double2{-0.5 * (X.y - Y.y), 0.5 * (X.x - Y.x)};
}

constexpr int kAdjointAllWaves = 4;  // of a workgroup that holds all of an m's waves

// One wave per (m, R groups of 64 ring pairs), as in the synthesis: every wave runs its own l-range, so polar groups,
// which contribute late or never, hold nobody up.  (One workgroup per m with all its ring pairs and an LDS sum per l
// filled a CU at lmax 4095 and waited for its equatorial waves.)  Per K l the wave adds up its ring pairs' products in
// registers, sums them over its lanes (wave_sums) and adds the 16 totals to the output array with one atomic each
// (128 bytes, or 64 bytes of E and of B): the array (cleared before) holds, per (l, m),
//   spin 0: sum, E alone: (-1)^s X + Y, E + B: X in E's place and Y in B's,
// X and Y the sums over the u and v halves; k_adjoint_finish turns them into alm.  The recursion table comes as
// vector loads, 8 l per register and 16-lane row, two chunks ahead, broadcast by DPP.
// What bounds it: FP64 VALU issue.  Per l and ring pair a spin-s E + B map takes 8 FMAs and 4 of recursion, and the
// lane sums (12 permlane swap pairs, 21 DPP and 14 adds per 4 l, a swap taking two issue slots) cost 7.5 / R more.
// Times, ms, with the clearing and finishing passes (0.16 at lmax 4095): spin 2 lmax 4095 R = 1 / 2 / 3 / 4:
// 13.4 / 10.2 / 9.3 / 9.6 (13.9 before), spin 0 6.1 / 4.2 / 3.65 / 3.7 (10.1 before); lmax 300 spin 2 0.040 / 0.047 /
// 0.053 (0.131 before): few waves want the shorter l-step.
// ALL: the waves of one m form a workgroup and keep their totals in LDS; it adds them up in wave order and writes alm
// itself, without the passes before and after, and repeats bit for bit.  Us, with atomics and three launches / now: spin 2
// lmax 64 19.7 / 10.9, 300 47 / 31, 511 86 / 87, 700 173 / 137, 766 198 / 192; spin 0 35 / 19 at 300, 88 / 68 at 700.
template <int MODE, int R, bool ALL = false>
__global__ __launch_bounds__(ALL ? 64 * kAdjointAllWaves : 64) void k_adjoint(AdjArgs a) {
  extern __shared__ double adj_sums[];  // ALL: [wave][l - l0][NA]
  constexpr bool SP = MODE != kScalar;
  constexpr int NA = MODE == kFull ? 4 : 2;  // doubles per (l, m)
  constexpr int K = 16 / NA;                 // l per lane sum
  constexpr int CH = 8;
  const int blk = blockIdx.x;
  const int j = blk / kNumXcd;
  const int m = (blk - j * kNumXcd) + kNumXcd * (j / a.nsb);
  const int wave = ALL ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
  const int sb = ALL ? wave : j % a.nsb;
  const int L = a.lmax;
  if (m > L) return;
  const int l0 = l0_of(m, a.s);
  const int lane = threadIdx.x & 63;
  const long nalm = (long)(L + 1) * (L + 2) / 2;
  const long row = (long)m * (2 * L + 1 - m) / 2;  // of (l, m) = (0, m) in alm
  const int nl = L + 1 - l0;
  if (!ALL && (l0 > L || sb * 64 * R >= a.nslot)) return;
  const long base = a.mofs[m];
  const double* __restrict__ rec = reinterpret_cast<const double*>(a.rec + base) + (lane & 15);

  // C[r]: the ring pair's factors.  The south-ring sign (-1)^{l+m} is sgA at even l - l0 and -sgA at odd ones:
  //   spin 0: C0 / C1 = north +- south (even / odd l - l0)
  //   E + B:  X = sum C0 u +- C1 v, Y = sum C2 v +- C3 u
  //   E:      Z = (-1)^s X + Y = sum (C0 or C1) u + (C2 or C3) v (even or odd l - l0)
  double x[R], mu[R], pm[R], nv[R], pv[R];
  float ku[R], kv[R];
  double2 C0[R], C1[R], C2[R], C3[R];
  int lst[R];
  int lc = L + 1, lall = l0;
  const double sgA = ((l0 + m) & 1) ? -1.0 : 1.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int g = sb * R + r;
    lst[r] = __builtin_amdgcn_readfirstlane(g < a.ngroups && nl > 0 ? a.start[(long)m * a.ngroups + g] : L + 1);
    lc = min(lc, lst[r]);
    if (lst[r] <= L) lall = max(lall, lst[r]);
    const int slot = g * 64 + lane;
    x[r] = mu[r] = pm[r] = nv[r] = pv[r] = 0.0;
    ku[r] = kv[r] = 0.f;
    C0[r] = C1[r] = C2[r] = C3[r] = double2{0.0, 0.0};
    if (slot < a.nslot && lst[r] <= L) {
      x[r] = cos(a.slot_theta[slot]);
      const int rn = a.slot_north[slot];
      const int rs = a.slot_south[slot];
      const double2 zero{0.0, 0.0};
      if constexpr (!SP) {
        const double2* g0 = a.G + (long)m * a.sm;
        const double2 gn = g0[(long)rn * a.sr];
        const double2 gs = rs >= 0 ? cscale(g0[(long)rs * a.sr], sgA) : zero;
        C0[r] = cadd(gn, gs);
        C1[r] = csub(gn, gs);
      } else {
        const double2* gp = a.G + (long)(L + m) * a.sm;
        const double2* gm = a.G + (long)(L - m) * a.sm;
        const double2 pn = gp[(long)rn * a.sr], qn = cconj(gm[(long)rn * a.sr]);
        const double2 ps = rs >= 0 ? cscale(gp[(long)rs * a.sr], sgA) : zero;
        const double2 qs = rs >= 0 ? cscale(cconj(gm[(long)rs * a.sr]), sgA) : zero;
        if constexpr (MODE == kFull) {
          C0[r] = pn; C1[r] = ps; C2[r] = qn; C3[r] = qs;
        } else {
          const double ss = (a.s & 1) ? -1.0 : 1.0;
          C0[r] = cadd(cscale(pn, ss), qs);
          C1[r] = csub(cscale(pn, ss), qs);
          C2[r] = cadd(qn, cscale(ps, ss));
          C3[r] = csub(qn, cscale(ps, ss));
        }
      }
    }
  }
  lc = __builtin_amdgcn_readfirstlane(lc);
  lall = __builtin_amdgcn_readfirstlane(lall);
  if (!ALL && lc > L) return;

  // where this lane's total goes (one lane of each quad writes)
  const int wl = (lane >> 2) / NA, wc = (lane >> 2) % NA;
  const bool writer = (lane & 3) == 0;
  double* __restrict__ out = reinterpret_cast<double*>(a.alm + row + l0 + wl + (wc >> 1) * nalm) + (wc & 1);
  double* sums = adj_sums + wave * nl * NA;
  if constexpr (ALL)
    for (int i = lane; i < min(lc - l0, nl) * NA; i += 64) sums[i] = 0.0;

  // One chunk of 8 l.  SLOW: a group may join, some lane may be below range; FULL: all 8 l <= L.
  auto chunk = [&](int l, double rc, auto slow_tag, auto full_tag) {
    constexpr bool SLOW = decltype(slow_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
    double fu[R], fv[R];
    if constexpr (SLOW) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (l == lst[r]) {
          const int slot = (sb * R + r) * 64 + lane;
          if (slot < a.nslot) {
            const long q = (long)m * a.sstride + slot;
            const double2 sm = a.st_mu[q], sp = a.st_p[q], sk = a.st_k[q];
            mu[r] = sm.x; pm[r] = sp.x; ku[r] = (float)sk.x;
            if (SP) { nv[r] = sm.y; pv[r] = sp.y; kv[r] = (float)sk.y; }
          }
        }
        fu[r] = rescaled_weight(mu[r], pm[r], ku[r]);
        fv[r] = SP ? rescaled_weight(nv[r], pv[r], kv[r]) : 0.0;
      }
    }
    static_for<0, CH / K>([&](auto hc) {
      constexpr int h = decltype(hc)::value;
      double v[16];
      static_for<0, K>([&](auto ic) {
        constexpr int i = decltype(ic)::value, li = h * K + i;
        constexpr bool odd = (i & 1) != 0;
        const double ra = row_bcast<2 * li>(rc), rb = SP ? row_bcast<2 * li + 1>(rc) : 0.0;
        double2 X{0.0, 0.0}, Y{0.0, 0.0};
#pragma unroll
        for (int r = 0; r < R; ++r) {
          double wu = mu[r], wv = nv[r];
          if (SLOW) { wu *= fu[r]; if (SP) wv *= fv[r]; }
          if constexpr (MODE == kFull) {
            fma2(X, C0[r], wu);
            fma2(Y, C2[r], wv);
            fma2(X, C1[r], odd ? -wv : wv);
            fma2(Y, C3[r], odd ? -wu : wu);
          } else {
            fma2(X, odd ? C1[r] : C0[r], wu);
            if (SP) fma2(X, odd ? C3[r] : C2[r], wv);
          }
          // a step past lmax reads a padded or neighbouring table entry; its result is never used
          const double t = SP ? fma(ra, x[r], rb) : ra * x[r];
          const double nu = fma(t, mu[r], -pm[r]);
          pm[r] = mu[r]; mu[r] = nu;
          if (SP) {
            const double nn = fma(fma(ra, x[r], -rb), nv[r], -pv[r]);
            pv[r] = nv[r]; nv[r] = nn;
          }
        }
        v[i * NA] = X.x;
        v[i * NA + 1] = X.y;
        if constexpr (MODE == kFull) { v[i * NA + 2] = Y.x; v[i * NA + 3] = Y.y; }
      });
      const double total = wave_sums(v);
      const int lh = l + h * K;
      if (writer && (FULL || lh + wl <= L)) {
        if constexpr (ALL) sums[(lh - l0) * NA + (lane >> 2)] = total;
        else atomicAdd(out + 2 * (lh - l0), total);
      }
    });
  };
  auto any_under = [&]() {
    bool under = false;
#pragma unroll
    for (int r = 0; r < R; ++r) under |= (ku[r] < 0.f) || (kv[r] < 0.f);
    return __any(under);
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  auto load = [&](int l) { return rec[2 * (long)(l - l0)]; };
  double b0 = 0.0, b1 = 0.0;
  if (lc <= L) { b0 = load(lc); b1 = load(lc + CH); }
  while (lc <= L && (lc <= lall || any_under())) {
    const double b2 = load(lc + 2 * CH);
    if (lc + CH - 1 <= L) chunk(lc, b0, T_{}, T_{});
    else chunk(lc, b0, T_{}, F_{});
    b0 = b1;
    b1 = b2;
    lc += CH;
  }
  while (lc + 2 * CH - 1 <= L) {
    chunk(lc, b0, F_{}, T_{});
    b0 = load(lc + 2 * CH);
    chunk(lc + CH, b1, F_{}, T_{});
    b1 = load(lc + 3 * CH);
    lc += 2 * CH;
  }
  if (lc + CH - 1 <= L) {
    chunk(lc, b0, F_{}, T_{});
    b0 = b1;
    lc += CH;
  }
  if (lc <= L) chunk(lc, b0, F_{}, F_{});
  if constexpr (ALL) {
    __syncthreads();
    const int nw = blockDim.x >> 6;
    for (int l = m + (int)threadIdx.x; l <= L; l += blockDim.x) {
      double2* e = a.alm + row + l;
      if (l < l0) {
        e[0] = double2{0.0, 0.0};
        if constexpr (MODE == kFull) e[nalm] = double2{0.0, 0.0};
        continue;
      }
      double t[NA];
#pragma unroll
      for (int k = 0; k < NA; ++k) t[k] = 0.0;
      for (int w = 0; w < nw; ++w)
#pragma unroll
        for (int k = 0; k < NA; ++k) t[k] += adj_sums[(w * nl + l - l0) * NA + k];
      const double c = a.cnorm[base + l - l0];
      if constexpr (MODE == kFull) adjoint_coef(a.s, c, double2{t[0], t[1]}, double2{t[2], t[3]}, e[0], e[nalm]);
      else e[0] = adjoint_coef<MODE>(m, c, double2{t[0], t[1]});
    }
  }
}

__global__ void k_adjoint_clear(double2* __restrict__ p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    p[i] = double2{0.0, 0.0};
}

// The sums of k_adjoint -> alm, in place.  Block row y serves m = y and m = lmax - y, which together have lmax + 2 l.
template <int MODE>
__global__ __launch_bounds__(256) void k_adjoint_finish(int L, int s, const long* __restrict__ mofs,
                                                        const double* __restrict__ cnorm, double2* __restrict__ alm) {
  const long nalm = (long)(L + 1) * (L + 2) / 2;
  for (int pass = 0; pass < 2; ++pass) {
    const int m = pass == 0 ? (int)blockIdx.y : L - (int)blockIdx.y;
    if (pass == 1 && m <= (int)blockIdx.y) break;  // the middle m has no partner
    const int l0 = l0_of(m, s);
    const long mbase = (long)m * (2 * L + 1 - m) / 2;
    for (int l = l0 + blockIdx.x * blockDim.x + threadIdx.x; l <= L; l += gridDim.x * blockDim.x) {
      const double c = cnorm[mofs[m] + (l - l0)];
      double2* e = alm + mbase + l;
      if constexpr (MODE == kFull) adjoint_coef(s, c, *e, e[nalm], *e, e[nalm]);
      else *e = adjoint_coef<MODE>(m, c, *e);
    }
  }
}

}  // namespace

// ------------------------------------------------------------------ host
void LegendreTables::build(int L, int s, const std::vector<double>& theta, hipStream_t st) {
  NUSHT_REQUIRE(L >= 0 && s >= 0 && s <= 3, kErrArg, "legendre: bad lmax/spin");
  if (const char* e = getenv("NUSHT_LEGENDRE_MFMA"); e && e[0] == '0') mfma = false;
  lmax = L;
  spin = s;
  nring = (int)theta.size();
  n_prep = "legendre_prep_" + tag + "_s" + std::to_string(s);
  n_synth = "legendre_synth_" + tag + "_s" + std::to_string(s);
  n_adj = "legendre_adjoint_" + tag + "_s" + std::to_string(s);
  // pair rings symmetric about the equator
  std::vector<int> order(nring);
  for (int i = 0; i < nring; ++i) order[i] = i;
  std::sort(order.begin(), order.end(), [&](int a, int b) { return theta[a] < theta[b]; });
  std::vector<char> used(nring, 0);
  std::vector<double> sth;
  std::vector<int> sn, ss;
  int lo = 0, hi = nring - 1;
  while (lo <= hi) {
    int a = order[lo], b = order[hi];
    if (lo == hi) {
      sth.push_back(theta[a]); sn.push_back(a); ss.push_back(a);
      break;
    }
    if (std::fabs(theta[a] + theta[b] - M_PI) < 1e-13) {
      sth.push_back(theta[a]); sn.push_back(a); ss.push_back(b);
      ++lo; --hi;
    } else if (theta[a] + theta[b] < M_PI) {
      sth.push_back(theta[a]); sn.push_back(a); ss.push_back(-1);
      ++lo;
    } else {
      sth.push_back(theta[b]); sn.push_back(b); ss.push_back(-1);
      --hi;
    }
  }
  // an equator ring paired with itself: keep it as north only
  for (size_t i = 0; i < sn.size(); ++i)
    if (ss[i] == sn[i]) ss[i] = -1;
  nslot = (int)sth.size();
  upload(slot_theta, sth);
  upload(slot_north, sn);
  upload(slot_south, ss);

  std::vector<long> mo(L + 2, 0);
  for (int m = 0; m <= L; ++m) {
    int l0 = l0_of(m, s);
    mo[m + 1] = mo[m] + (l0 <= L ? (L - l0 + 1) : 0);
  }
  nlm = mo[L + 1];
  upload(mofs, mo);
  std::vector<long> mb(L + 1, 0);
  nblk = 0;
  for (int m = 0; m <= L; ++m) {
    mb[m] = nblk;
    nblk += ceil_div((long)(mo[m + 1] - mo[m]), 4L);
  }
  upload(mblk, mb);
  // padded so that a chunked, prefetching l-loop may read past the last l of the last m
  rec.alloc(sizeof(double2) * (size_t)(std::max<long>(nlm, 1) + kSynPad));
  cnorm.alloc(sizeof(double) * (size_t)(std::max<long>(nlm, 1) + kSynPad));
  sstride = nslot;
  ngroups = ceil_div(nslot, 64);
  const size_t nst = (size_t)(L + 1) * sstride;
  st_mu.alloc(sizeof(double2) * nst);
  st_p.alloc(sizeof(double2) * nst);
  st_k.alloc(sizeof(double2) * nst);
  start.alloc(sizeof(int) * (size_t)(L + 1) * ngroups);
  hipLaunchKernelGGL(k_rec_tables, dim3(ceil_div(L + 1, 128)), dim3(128), 0, st, L, s, mofs.as<long>(),
                     rec.as<double2>(), cnorm.as<double>());
  NUSHT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_seeds, dim3(ceil_div(nslot, 64)), dim3(64), 0, st, L, s, nslot, sstride,
                     slot_theta.as<double>(), st_mu.as<double2>(), st_p.as<double2>(), st_k.as<double2>());
  NUSHT_LAUNCH_CHECK();
  const dim3 grid((unsigned)((long)ngroups * (L + 1)));
  if (s > 0)
    hipLaunchKernelGGL(k_advance<true>, grid, dim3(64), 0, st, L, s, nslot, sstride, ngroups,
                       slot_theta.as<double>(), mofs.as<long>(), rec.as<double2>(), st_mu.as<double2>(),
                       st_p.as<double2>(), st_k.as<double2>(), start.as<int>());
  else
    hipLaunchKernelGGL(k_advance<false>, grid, dim3(64), 0, st, L, s, nslot, sstride, ngroups,
                       slot_theta.as<double>(), mofs.as<long>(), rec.as<double2>(), st_mu.as<double2>(),
                       st_p.as<double2>(), st_k.as<double2>(), start.as<int>());
  NUSHT_LAUNCH_CHECK();
  // work actually run by a synthesis (reported with the plan; synchronizes once)
  std::vector<int> hs((size_t)(L + 1) * ngroups);
  NUSHT_HIP(hipMemcpyAsync(hs.data(), start.get(), sizeof(int) * hs.size(), hipMemcpyDeviceToHost, st));
  NUSHT_HIP(hipStreamSynchronize(st));
  pair_steps = 0;
  for (int m = 0; m <= L; ++m) {
    if (l0_of(m, s) > L) continue;
    for (int g = 0; g < ngroups; ++g)
      pair_steps += (long)(L + 1 - hs[(size_t)m * ngroups + g]) * std::min(64, nslot - 64 * g);
  }
}

static int padded_maps(int nmaps) { return nmaps <= 1 ? 1 : nmaps <= 2 ? 2 : nmaps <= 4 ? 4 : 8; }

size_t legendre_coef_bytes(const LegendreTables& t, int nmaps) {
  // padded by kSynPad entries (chunked, prefetching reads past the last l of the last m)
  const size_t vec = sizeof(double2) * (size_t)(std::max<long>(t.nlm, 1) + kSynPad) * padded_maps(nmaps) *
                     (t.spin ? 2 : 1);
  if (nmaps < 3) return vec;
  // matrix-core layout: 32 doubles per chain, map group and block of 4 l, 2 blocks of padding (prefetch)
  const int ns = nmaps >= kLegendreMfma8Min ? 2 : 1;
  const size_t mf = sizeof(double) * 32 * ns * (t.spin ? 2 : 1) * (size_t)(t.nblk + 2);
  return std::max(vec, mf);
}

// Synthesis variants of one map, in order of the launch size they suit: k_synth_row, k_synth with few and with more
// ring groups per wave; the autotuner picks one per table.  Launches of two maps go by their waves (kTwoMapWaves).
static const char* const kSynVariants[] = {"row broadcasts", "few groups per wave", "more groups per wave"};
constexpr int kNumSynVariants = 3;

// Waves of 64 ring pairs (m times ring groups) from which launches of two maps take free blocks, spin 0 two groups per
// wave: about those the GPU holds (256 CUs, 4 SIMDs, 8 waves).  Blocks of 8 waves / free blocks, ms: lmax 900 (7208 waves)
// spin 0 0.115 / 0.129, spin 2 0.210 / 0.231; lmax 1000 (9009) 0.148 / 0.163, 0.27 / 0.27; lmax 1200 (12010) 0.237 / 0.209,
// 0.42 / 0.39.
constexpr long kTwoMapWaves = 10000;

template <bool SP, int NB, bool GR = false>
static void launch_synth(const SynthArgs& a, int variant, hipStream_t st) {
  // Odd number of blocks per m: blocks are handed to XCDs and shader engines round-robin, and
  // with a power-of-two count every engine would see the same slot groups for every m, so the
  // polar groups (long underflow phases) would pile up on a few engines.
  SynthArgs b = a;
  const auto blocks = [&](int groups, int chains) {
    b.nsb = ceil_div(a.nslot, 64 * groups) | 1;
    return dim3((unsigned)(b.nsb * chains * ceil_div(a.lmax + 1, kNumXcd) * kNumXcd));
  };
  if constexpr (NB > 1) {
    constexpr int CH = SP ? 2 : 4;
    if ((long)(a.lmax + 1) * ceil_div(a.nslot, 64) < kTwoMapWaves) {
      const dim3 grid = blocks(8, 1);
      hipLaunchKernelGGL((k_synth<SP, NB, 1, CH, GR, 1, 8>), grid, dim3(64 * 8), 0, st, b);
    } else {
      constexpr int R = SP ? 1 : 2;
      const dim3 grid = blocks(R, 1);
      hipLaunchKernelGGL((k_synth<SP, NB, R, CH, GR, 1>), grid, dim3(64), 0, st, b);
    }
  } else if (variant == 0) {
    constexpr int MODE = !SP ? kScalar : GR ? kGrad : kFull;
    const dim3 grid = blocks(1, SP ? 2 : 1);
    hipLaunchKernelGGL(k_synth_row<MODE>, grid, dim3(64), 0, st, b);
  } else if constexpr (SP) {
    const dim3 grid = blocks(variant, 1);
    if (variant == 1) hipLaunchKernelGGL((k_synth<SP, 1, 1, 2, GR, 8>), grid, dim3(64), 0, st, b);
    else hipLaunchKernelGGL((k_synth<SP, 1, 2, 2, GR, 6>), grid, dim3(64), 0, st, b);
  } else {
    const dim3 grid = blocks(variant + 1, 1);
    if (variant == 1) hipLaunchKernelGGL((k_synth<SP, 1, 2, 4, GR, 6>), grid, dim3(64), 0, st, b);
    else hipLaunchKernelGGL((k_synth<SP, 1, 3, 4, GR, 4>), grid, dim3(64), 0, st, b);
  }
  NUSHT_LAUNCH_CHECK();
}

static void legendre_synth_chunk(const LegendreTables& t, int nmaps, int ncomp, const double2* alm,
                                 long alm_stride_map, const double* fl, double2* coef_ws, double2* G, long sm, long sr,
                                 long smap, hipStream_t st);

static void legendre_synth_mfma(const LegendreTables& t, int nmaps, int ncomp, const AlmPtrs8& alm,
                                const double* fl, double2* coef_ws, double2* G, long sm, long sr, long smap,
                                hipStream_t st);

static AlmPtrs8 strided_maps(const double2* alm, long stride, int nmaps) {
  AlmPtrs8 a{};
  for (int b = 0; b < 8; ++b) a.p[b] = alm + (b < nmaps ? b : 0) * stride;
  return a;
}

// maps of the next matrix-core launch for `left` remaining maps (>= 3); NUSHT_LEGENDRE_MFMA8=0 keeps 4 per launch
static int mfma_maps(int left) {
  const char* e = getenv("NUSHT_LEGENDRE_MFMA8");
  const bool eight = !(e && e[0] == '0');
  return eight && left >= kLegendreMfma8Min ? std::min(8, left) : std::min(kLegendreMfmaMaps, left);
}

void legendre_synth(const LegendreTables& t, int nmaps, int ncomp, const double2* alm, long alm_stride_map,
                    const double* fl, double2* coef_ws, double2* G, long sm, long sr, long smap, hipStream_t st) {
  NUSHT_REQUIRE(nmaps >= 1 && nmaps <= 8, kErrArg, "legendre_synth: nmaps must be in [1, 8]");
  const int ch = std::max(1, std::min(t.chunk, 2));
  int b = 0;
  while (b < nmaps) {
    const int left = nmaps - b;
    if (t.mfma && left >= 3) {
      const int nb = mfma_maps(left);
      legendre_synth_mfma(t, nb, ncomp, strided_maps(alm + b * alm_stride_map, alm_stride_map, nb), fl, coef_ws,
                          G + b * smap, sm, sr, smap, st);
      b += nb;
    } else {
      const int nb = std::min(ch, left);
      legendre_synth_chunk(t, nb, ncomp, alm + b * alm_stride_map, alm_stride_map, fl, coef_ws, G + b * smap, sm,
                           sr, smap, st);
      b += nb;
    }
  }
}

void legendre_synth_maps(const LegendreTables& t, int nmaps, int ncomp, const double2* const* alm, double2* coef_ws,
                         double2* G, long sm, long sr, long smap, hipStream_t st) {
  NUSHT_REQUIRE(nmaps >= 1 && nmaps <= 8, kErrArg, "legendre_synth_maps: nmaps must be in [1, 8]");
  int b = 0;
  while (b < nmaps) {
    const int left = nmaps - b;
    if (t.mfma && left >= 3) {
      const int nb = mfma_maps(left);
      AlmPtrs8 ap{};
      for (int k = 0; k < 8; ++k) ap.p[k] = alm[b + (k < nb ? k : 0)];
      legendre_synth_mfma(t, nb, ncomp, ap, nullptr, coef_ws, G + b * smap, sm, sr, smap, st);
      b += nb;
    } else {
      legendre_synth(t, 1, ncomp, alm[b], 0, nullptr, coef_ws, G + b * smap, sm, sr, smap, st);
      b += 1;
    }
  }
}

static void legendre_synth_mfma(const LegendreTables& t, int nmaps, int ncomp, const AlmPtrs8& alm,
                                const double* fl, double2* coef_ws, double2* G, long sm, long sr, long smap,
                                hipStream_t st) {
  NUSHT_REQUIRE(nmaps >= 1 && nmaps <= 8, kErrArg, "matrix-core synthesis: 1 to 8 maps per launch");
  const int L = t.lmax;
  const int ns = nmaps > kLegendreMfmaMaps ? 2 : 1;  // 16-column map groups
  double* coef4 = reinterpret_cast<double*>(coef_ws);
  {
    StageScope sc(t.n_prep.c_str(), st);
    // block row y covers m = y and m = L - y; its x extent is sized for m = 0 (the longest table)
    dim3 grid(ceil_div((L + 4) / 4 * 16 * ns, 256), L / 2 + 1);
    if (ns == 1)
      hipLaunchKernelGGL(k_prep4<1>, grid, dim3(256), 0, st, L, t.spin, nmaps, ncomp, alm, fl, t.mofs.as<long>(),
                         t.mblk.as<long>(), t.cnorm.as<double>(), coef4);
    else
      hipLaunchKernelGGL(k_prep4<2>, grid, dim3(256), 0, st, L, t.spin, nmaps, ncomp, alm, fl, t.mofs.as<long>(),
                         t.mblk.as<long>(), t.cnorm.as<double>(), coef4);
    NUSHT_LAUNCH_CHECK();
  }
  SynthArgs a;
  a.lmax = L; a.s = t.spin; a.nslot = t.nslot; a.sstride = t.sstride; a.nmaps = nmaps;
  a.nsb = ceil_div(a.nslot, 64) | 1;
  a.slot_theta = t.slot_theta.as<double>();
  a.slot_north = t.slot_north.as<int>();
  a.slot_south = t.slot_south.as<int>();
  a.mofs = t.mofs.as<long>();
  a.rec = t.rec.as<double2>();
  a.st_mu = t.st_mu.as<double2>();
  a.st_p = t.st_p.as<double2>();
  a.st_k = t.st_k.as<double2>();
  a.start = t.start.as<int>();
  a.coef = coef_ws;
  a.G = G; a.sm = sm; a.sr = sr; a.smap = smap;
  const int nblocks = a.nsb * ceil_div(L + 1, kNumXcd) * kNumXcd;
  StageScope sc(t.n_synth.c_str(), st);
  if (t.spin > 0 && ns == 1)
    hipLaunchKernelGGL((k_synth_mfma<true, 1>), dim3(nblocks), dim3(64), 0, st, a, coef4, t.mblk.as<long>());
  else if (t.spin > 0)
    hipLaunchKernelGGL((k_synth_mfma<true, 2>), dim3(nblocks), dim3(64), 0, st, a, coef4, t.mblk.as<long>());
  else if (ns == 1)
    hipLaunchKernelGGL((k_synth_mfma<false, 1>), dim3(nblocks), dim3(64), 0, st, a, coef4, t.mblk.as<long>());
  else
    hipLaunchKernelGGL((k_synth_mfma<false, 2>), dim3(nblocks), dim3(64), 0, st, a, coef4, t.mblk.as<long>());
  NUSHT_LAUNCH_CHECK();
}

// Variant of a table that was not measured (point sets: no mirrored rings, so up to 64 points per group).  Spin s,
// points at lmax, us, row broadcasts / few / more groups: 300 at 2000 390 / 471 / 540, 1000 at 300 39 / 51 / 57, 1000 at
// 1000 306 / 248 / 302, 700 at 2000 757 / 655 / 699, 3000 at 1000 806 / 647 / 629, 1000 at 4000 3967 / 3858 / 3033.  Spin 0
// is within 15 % of its best with row broadcasts, 1.3 to 2 times ahead below 1000 points.
static int untuned_variant(const LegendreTables& t) {
  const long waves = (long)(t.lmax + 1) * t.ngroups;
  if (t.spin == 0 || t.ngroups < 8 || waves < 12000) return 0;
  return waves < 40000 ? 1 : 2;
}

static void legendre_synth_chunk(const LegendreTables& t, int nmaps, int ncomp, const double2* alm,
                                 long alm_stride_map, const double* fl, double2* coef_ws, double2* G, long sm, long sr,
                                 long smap, hipStream_t st) {
  const int L = t.lmax;
  const int nbpad = padded_maps(nmaps);
  {
    StageScope sc(t.n_prep.c_str(), st);
    dim3 grid(ceil_div(L + 1, 256), L + 1);
    hipLaunchKernelGGL(k_prep, grid, dim3(256), 0, st, L, t.spin, nmaps, nbpad, ncomp, alm, alm_stride_map, fl,
                       t.mofs.as<long>(), t.cnorm.as<double>(), coef_ws);
    NUSHT_LAUNCH_CHECK();
  }
  SynthArgs a;
  a.lmax = L; a.s = t.spin; a.nslot = t.nslot; a.sstride = t.sstride; a.nsb = 0; a.nmaps = nmaps;
  a.slot_theta = t.slot_theta.as<double>();
  a.slot_north = t.slot_north.as<int>();
  a.slot_south = t.slot_south.as<int>();
  a.mofs = t.mofs.as<long>();
  a.rec = t.rec.as<double2>();
  a.st_mu = t.st_mu.as<double2>();
  a.st_p = t.st_p.as<double2>();
  a.st_k = t.st_k.as<double2>();
  a.start = t.start.as<int>();
  a.coef = coef_ws;
  a.G = G; a.sm = sm; a.sr = sr; a.smap = smap;
  const bool sp = t.spin > 0;
  const bool gr = sp && ncomp == 1;  // E only: the gradient-only contraction
  const int tv = gr ? t.variant_grad : t.variant;
  const int var = (tv >= 0 && tv < kNumSynVariants) ? tv : untuned_variant(t);
  StageScope sc(t.n_synth.c_str(), st);
  switch (nbpad) {  // the kernel's NB must equal the coefficient stride written by k_prep
    case 1:
      if (gr) launch_synth<true, 1, true>(a, var, st);
      else if (sp) launch_synth<true, 1>(a, var, st);
      else launch_synth<false, 1>(a, var, st);
      break;
    case 2:
      if (gr) launch_synth<true, 2, true>(a, var, st);
      else if (sp) launch_synth<true, 2>(a, var, st);
      else launch_synth<false, 2>(a, var, st);
      break;
    default: throw Error{kErrUnsupported, "legendre_synth: at most 2 maps per launch"};
  }
}

int legendre_variant_count() { return kNumSynVariants; }

// Waves of a one-group launch (m times ring groups) below which a table takes the row-broadcast synthesis without
// measuring the others.  At lmax 255 (768 waves, spin 0) it takes 10 us against 22, at lmax 1000 (8008) 0.070 to
// 0.160 ms against 0.118 to 0.218; between 20 us launches the measurement took the slower one in one process of four.
// Few rings at a high lmax are the same case: 24 rings at lmax 4000 (4001 waves) 0.39 ms against 1.04 (spin 2), 0.22
// against 0.66 (spin 0).
constexpr long kRowWaves = 4096;

// Coefficients to measure on, of order one: on zeros the clock runs higher (2.33 GHz at lmax 4095, 2.05 on data), by
// more for the denser kernels.  In three processes each over lmax 64 to 4095, measured on zeros and one kernel after the
// other the tuner took row broadcasts at lmax 1500 spin 2 (0.51 ms, few groups 0.47) in two and more groups at lmax 4095
// spin 0 (2.73 ms, row broadcasts 2.45) in one; on data, with every kernel run before the first is timed, in none.
static __global__ void k_tuning_alm(double2* __restrict__ alm, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const unsigned h = (unsigned)i * 2654435761u;
    alm[i] = double2{(h >> 16) * 0x1p-15 - 1.0, (h & 0xffffu) * 0x1p-15 - 1.0};
  }
}

void legendre_autotune(LegendreTables& t, int ncomp, double2* coef_ws, double2* G, long sm, long sr, hipStream_t st) {
  // NUSHT_LEGENDRE_VARIANT=k fixes the variant (tests run every variant this way)
  if (const char* fv = getenv("NUSHT_LEGENDRE_VARIANT"); fv && fv[0]) {
    const int v = atoi(fv);
    NUSHT_REQUIRE(v >= 0 && v < kNumSynVariants, kErrArg, "NUSHT_LEGENDRE_VARIANT out of range");
    t.variant = t.variant_grad = v;
    t.tuned_ms = 0.f;
    return;
  }
  const bool gr = t.spin > 0 && ncomp == 1;
  int& slot = gr ? t.variant_grad : t.variant;
  const int nvar = (long)(t.lmax + 1) * t.ngroups < kRowWaves ? 1 : kNumSynVariants;
  // one measurement per (lmax, spin, ring pairs) and process
  static std::mutex mu;
  static std::map<std::tuple<int, int, int, int>, std::pair<int, float>> cache;
  const auto key = std::make_tuple(t.lmax, t.spin, t.nslot, ncomp);
  {
    std::lock_guard<std::mutex> g(mu);
    auto it = cache.find(key);
    if (it != cache.end()) {
      slot = it->second.first;
      if (!gr) t.tuned_ms = it->second.second;
      return;
    }
  }
  const long nalm = (long)(t.lmax + 1) * (t.lmax + 2) / 2 * ncomp;
  DevBuf dummy(sizeof(double2) * (size_t)nalm);
  hipLaunchKernelGGL(k_tuning_alm, dim3((unsigned)std::min<long>(4096, ceil_div(nalm, 256L))), dim3(256), 0, st,
                     dummy.as<double2>(), nalm);
  NUSHT_LAUNCH_CHECK();
  const double2* alm = dummy.as<double2>();
  hipEvent_t e0, e1;
  NUSHT_HIP(hipEventCreate(&e0));
  NUSHT_HIP(hipEventCreate(&e1));
  float best = 1e30f;
  int bestv = 0;
  const char* env = getenv("NUSHT_VERBOSE");
  const bool verbose = env && env[0] && env[0] != '0';
  for (int v = 0; v < nvar; ++v) {  // all of them first, or the one timed first is timed while the clock settles
    slot = v;
    legendre_synth(t, 1, ncomp, alm, 0, nullptr, coef_ws, G, sm, sr, 0, st);
  }
  for (int v = 0; v < nvar; ++v) {
    slot = v;
    NUSHT_HIP(hipEventRecord(e0, st));
    for (int k = 0; k < 2; ++k) legendre_synth(t, 1, ncomp, alm, 0, nullptr, coef_ws, G, sm, sr, 0, st);
    NUSHT_HIP(hipEventRecord(e1, st));
    NUSHT_HIP(hipEventSynchronize(e1));
    float ms = 0;
    NUSHT_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (verbose)
      fprintf(stderr, "[nusht] legendre autotune %s lmax %d spin %d ncomp %d pairs %d: variant %d (%s) %.3f ms\n",
              t.tag.c_str(), t.lmax, t.spin, ncomp, t.nslot, v, kSynVariants[v], ms / 2);
    if (ms < best) { best = ms; bestv = v; }
  }
  slot = bestv;
  if (!gr) t.tuned_ms = best / 2;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  std::lock_guard<std::mutex> g(mu);
  cache[key] = {bestv, best / 2};
}

// Ring groups per wave of the adjoint where its waves add to the output.  Up to 384 ring pairs (512 for spin 0) one or two
// waves hold an m: their sums on a cleared output come out the same in either order, so the adjoint repeats bit for bit.
// Above, three or more waves add in any order, and the choice is by time: three groups once a launch with three has
// kAdjointMinWaves waves; below it a SIMD has one or two waves, and the shorter l-step of one group is worth more than the
// shared lane sums.  Measured, ms, one / three groups: lmax 700 spin 0 0.090 / 0.096, spin 2 0.167 / 0.174 (1402 waves);
// lmax 850 0.120 / 0.122, 0.224 / 0.231 (2553); lmax 1000 0.170 / 0.148, 0.296 / 0.276 (3003).
constexpr long kAdjointMinWaves = 2600;

static int adjoint_groups(int mode, int lmax, int ngroups) {
  if (ngroups <= (mode == kScalar ? 8 : 6)) return ceil_div(ngroups, 2);
  return (long)(lmax + 1) * ceil_div(ngroups, 3) < kAdjointMinWaves ? 1 : 3;
}

template <int MODE>
static void launch_adjoint(const LegendreTables& t, AdjArgs a, hipStream_t st) {
  const int L = t.lmax;
  // All of an m's waves in one workgroup, up to 512 ring pairs and as long as their totals in LDS leave a CU five waves (us,
  // in LDS / added to the output: 24 rings at lmax 1000 spin 2, five waves, 98 / 131; 256 rings at lmax 2000 spin 0, four,
  // 307 / 247); one group per wave up to four, two above (one / two: spin 2 lmax 300 31 / 38, 511 97 / 87, 700 182 / 137).
  const int RA = t.ngroups <= kAdjointAllWaves ? 1 : 2, nw = ceil_div(t.ngroups, RA);
  const size_t lds = sizeof(double) * (MODE == kFull ? 4 : 2) * (size_t)nw * (L + 1);
  if (nw <= kAdjointAllWaves && nw * (160 * 1024 / lds) >= 5) {
    a.nsb = 1;
    const auto kern = RA == 1 ? k_adjoint<MODE, 1, true> : k_adjoint<MODE, 2, true>;
    if (lds > 64 * 1024)
      NUSHT_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)(ceil_div(L + 1, kNumXcd) * kNumXcd)), dim3(64 * nw), lds, st, a);
    NUSHT_LAUNCH_CHECK();
    return;
  }
  const long n = (long)(L + 1) * (L + 2) / 2 * (MODE == kFull ? 2 : 1);
  hipLaunchKernelGGL(k_adjoint_clear, dim3((unsigned)std::min<long>(4096, (n + 255) / 256)), dim3(256), 0, st, a.alm, n);
  NUSHT_LAUNCH_CHECK();
  const int R = adjoint_groups(MODE, L, t.ngroups);
  a.nsb = ceil_div(t.ngroups, R) | 1;  // odd, as in launch_synth
  const dim3 grid((unsigned)(a.nsb * ceil_div(L + 1, kNumXcd) * kNumXcd));
  if (R == 1) hipLaunchKernelGGL((k_adjoint<MODE, 1>), grid, dim3(64), 0, st, a);
  else if (R == 2) hipLaunchKernelGGL((k_adjoint<MODE, 2>), grid, dim3(64), 0, st, a);
  else if (MODE == kScalar && R == 4) hipLaunchKernelGGL((k_adjoint<kScalar, 4>), grid, dim3(64), 0, st, a);
  else hipLaunchKernelGGL((k_adjoint<MODE, 3>), grid, dim3(64), 0, st, a);
  NUSHT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_adjoint_finish<MODE>, dim3(ceil_div(L + 1, 1024), L / 2 + 1), dim3(256), 0, st, L, t.spin,
                     t.mofs.as<long>(), t.cnorm.as<double>(), a.alm);
  NUSHT_LAUNCH_CHECK();
}

void legendre_adjoint(const LegendreTables& t, int ncomp, const double2* G, long sm, long sr, double2* alm,
                      hipStream_t st) {
  AdjArgs a;
  a.lmax = t.lmax; a.s = t.spin; a.nslot = t.nslot; a.sstride = t.sstride; a.ngroups = t.ngroups; a.nsb = 0;
  a.slot_theta = t.slot_theta.as<double>();
  a.slot_north = t.slot_north.as<int>();
  a.slot_south = t.slot_south.as<int>();
  a.mofs = t.mofs.as<long>();
  a.rec = t.rec.as<double2>();
  a.st_mu = t.st_mu.as<double2>();
  a.st_p = t.st_p.as<double2>();
  a.st_k = t.st_k.as<double2>();
  a.start = t.start.as<int>();
  a.G = G; a.sm = sm; a.sr = sr; a.alm = alm; a.cnorm = t.cnorm.as<double>();
  // the limits of the range this entry point takes; nothing above them is tested
  NUSHT_REQUIRE(t.lmax <= (t.spin ? 5119 : 10239), kErrUnsupported, "legendre_adjoint: lmax too large");
  StageScope sc(t.n_adj.c_str(), st);
  if (t.spin == 0) launch_adjoint<kScalar>(t, a, st);
  else if (ncomp == 1) launch_adjoint<kGrad>(t, a, st);
  else launch_adjoint<kFull>(t, a, st);
}

}  // namespace nusht
