// SHT on iso-latitude rings (see ring.h).
//
// Replaces the reference's GL-grid SHTns calls (synthesis_cupy / adjoint_synthesis_cupy /
// synthesis_der1_cupy, cunusht/sht/GPU_sht_transformer.py:56-96) and, for spin 1, the pointing
// kernel launched after synth_grad (cunusht/deflection/GPU_nufft_transformer.py:83-101).
#include "ring.h"

#include "stages.h"
#include "timing.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <set>
#include <utility>

namespace nusht {
namespace {

// Workgroup sizes by the values a ring's DFT holds in LDS.  Every thread keeps about eight values in registers (106 -
// 128 VGPRs, four waves per SIMD; three of the largest workgroup), so a workgroup of the largest size fills a CU whatever
// its ring's length; with smaller ones four rings of up to 2048 values, or two of up to 4160, run on a CU and cover each
// other's barriers and loads.  Measured with 768 threads for every ring and now: 301 rings of 625 values (lmax 300)
// 28 -> 21 us; 1501 rings of 3072 values (lmax 1500), synthesis 100 -> 70 us, adjoint 94 -> 78 us.
// Registers spilled at the small sizes: none or a few for direct and Bluestein transforms (13 to 30 where rings alias),
// 30 to 112 for Rader's and for the launches of any method.
constexpr int kRingClasses = 3;
constexpr int kRingNT[kRingClasses] = {256, 512, kDftNT};
constexpr int kRingNMax[kRingClasses] = {2048, 4160, kDftNMAX};

// A plan of at most kFewRings rings, the longest above kFewRingsValues, runs as one launch of its longest ring's size and
// at least 512 threads: at most two workgroups come to a CU, so a launch lasts as long as its slowest ring.  Adjoint /
// synthesis, us, by each ring's size and now: 500 rings of 1001 to 2048 pixels 73 / 81 -> 48 / 53, 300 of 401 to 2000
// 57 / 64 -> 36 / 39, 100 rings of 2000 15.3 / 16.0 -> 13.7 / 15.6.
constexpr int kFewRings = 512, kFewRingsValues = 1024;

// LDS values of a ring's workgroup: its DFT and, for a ring shorter than its band, the rows that alias onto it
// (those of a band that does not fit are read term by term)
int ring_values(const RingLen& d, int nrow, int band) {
  return d.n >= band || nrow > kDftNMAX ? d.lds_values() : std::max(d.lds_values(), nrow);
}

int ring_class(int values) {
  int c = 0;
  while (values > kRingNMax[c]) ++c;
  return c;
}

struct RingArgs {
  int lmax, spin, gstride, mode;
  int stage;              // rings shorter than their band: their rows fit the launch's LDS
  RingLen one;            // the ring length of a launch whose rings all share one length
  const int* rings;       // rings of this launch
  const int* lenidx;      // per ring: index into lens
  const RingLen* lens;
  const double* theta;
  const double* phi0;
  const long* ofs;
  double2* G;
  double* o0;
  double* o1;
  double* o2;
  const double* i0;
  const double* i1;
  const double* wt;  // per-ring weights applied to the adjoint's input (null: none)
};

// G_m e^{i m phi0} for row m of this ring
__device__ __forceinline__ double2 ring_coef(const double2* g, int m, int L, int spin, long gstride, double ph0) {
  double2 v = g[(long)(spin ? m + L : m) * gstride];
  if (ph0 != 0.0) {
    double s, c;
    sincos(m * ph0, &s, &c);
    v = cmul(v, double2{c, s});
  }
  return v;
}

constexpr int kAnyMethod = -1;

// What a launch does: rows -> rings, every ring at least as long as its band; rows -> rings of any length; or the
// transpose.  Each has a kernel of its own: the sums over aliased rows hold more registers than the rest.
enum RingPass { kFullBand, kAliased, kToRows };

// UNIFORM: every ring of the launch has the length a.one (read from the kernel arguments) and the DFT method METHOD;
// otherwise each ring reads its description from a.lens and, with kAnyMethod, takes its own method (all but the split).
// The transforms of every launch are inlined: called, they saved 160 to 250 bytes of registers per thread and shared
// nothing with the loads around them (HEALPix nside 512, lmax 1000, spin 2: synthesis 166 -> 117 us, adjoint 154 -> 103).
template <int METHOD, int NT, int NMAX>
__device__ __forceinline__ void ring_dft(double2* buf, const RingLen& Ld) {
  if constexpr (METHOD == kAnyMethod) {
    if (Ld.method == (int)DftMethod::Direct) dft_lds<0, double, NT, NMAX>(buf, Ld);
    else if (Ld.method == (int)DftMethod::Bluestein) dft_lds<2, double, NT, NMAX>(buf, Ld);
    else dft_lds<1, double, NT, NMAX>(buf, Ld);
  } else {
    dft_lds<METHOD, double, NT, NMAX>(buf, Ld);
  }
}

template <int METHOD, bool UNIFORM, RingPass PASS, int NT, int NMAX>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT < kDftNT ? 4 : 3))) void k_ring(RingArgs a) {
  constexpr int E = (NMAX + NT - 1) / NT;
  extern __shared__ unsigned char smem_raw[];
  double2* buf = reinterpret_cast<double2*>(smem_raw);
  // neighbouring rings run on the same XCD at the same time, so the m-major G columns they read
  // share that XCD's L2 lines
  const int ring = a.rings[xcd_remap(blockIdx.x, gridDim.x)];
  const RingLen& Ld = UNIFORM ? a.one : a.lens[a.lenidx[ring]];
  const int n = Ld.n;
  const int L = a.lmax;
  const double ph0 = a.phi0[ring];
  const long ofs = a.ofs[ring];
  const double2* g = a.G + ring;  // G[row][ring], row stride gstride
  if constexpr (PASS != kToRows) {
    // conjugated spectrum for the inverse DFT: X[m mod n] = sum conj(G_m e^{i m phi0}) over the m that alias there
    const int mlo = a.spin ? -L : 0;
    if (PASS == kFullBand || n >= 2 * L + 1) {
      for (int k = threadIdx.x; k < n; k += NT) buf[k] = double2{0.0, 0.0};
      // The thread's rows (at most E: L - mlo < n <= NMAX) are loaded unconditionally, from rows
      // clamped to L, so that every load is in flight before the first LDS write.
      double2 gv[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int m = min(mlo + (int)threadIdx.x + i * NT, L);
        gv[i] = g[(long)(a.spin ? m + L : m) * a.gstride];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int m = mlo + (int)threadIdx.x + i * NT;
        if (m <= L) {
          double2 v = gv[i];
          if (ph0 != 0.0) {
            double s, c;
            sincos(m * ph0, &s, &c);
            v = cmul(v, double2{c, s});
          }
          const int k = m >= 0 ? m : m + n;
          buf[k] = cconj(v);
          if (!a.spin && m > 0) buf[n - m] = v;
        }
      }
    } else if (a.stage) {
      // The ring is shorter than its band: X[k] sums the m = k mod n.  All rows are loaded at once, as above, and staged
      // in LDS in order of m (the launch has room for max(L - mlo + 1, DFT values)); then every k adds its terms up, for
      // short rings split over P threads (a ring of four pixels has 2 lmax / 4 terms per k).  One loop over k and its
      // terms, each loaded when its turn came, made the polar rings the launch's whole time: 2047 HEALPix rings at
      // nside 512, lmax 1000, spin 2, took 295 us, with staged rows 166 and inlined transforms 117.
      const int nrow = L - mlo + 1;
      double2 gv[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int m = min(mlo + (int)threadIdx.x + i * NT, L);
        gv[i] = g[(long)(a.spin ? m + L : m) * a.gstride];
      }
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int q = threadIdx.x + i * NT;
        if (q < nrow) {
          double2 v = gv[i];
          if (ph0 != 0.0) {
            double s, c;
            sincos((mlo + q) * ph0, &s, &c);
            v = cmul(v, double2{c, s});
          }
          buf[q] = v;
        }
      }
      __syncthreads();
      // terms p, p + P, p + 2 P, ... of k
      auto terms = [&](int k, int p, int P) {
        double2 acc{0.0, 0.0};
        for (int m = mlo + ((k - mlo) % n + n) % n + p * n; m <= L; m += P * n) acc = cadd(acc, cconj(buf[m - mlo]));
        if (!a.spin)  // the m < 0 half of a real field: conj(G_{-m}) = G_m at k = -m mod n
          for (int m = ((n - k) % n == 0 ? n : (n - k) % n) + p * n; m <= L; m += P * n) acc = cadd(acc, buf[m]);
        return acc;
      };
      if (2 * n <= NT) {
        const int P = NT / n;
        const int p = (int)threadIdx.x / n, k = (int)threadIdx.x - p * n;
        double2 part{0.0, 0.0};
        if (p < P) part = terms(k, p, P);
        __syncthreads();
        if (p < P) buf[threadIdx.x] = part;
        __syncthreads();
        if ((int)threadIdx.x < n)
          for (int q = 1; q < P; ++q) part = cadd(part, buf[q * n + threadIdx.x]);
        __syncthreads();
        if ((int)threadIdx.x < n) buf[threadIdx.x] = part;
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const int k = threadIdx.x + i * NT;
          if (k < n) gv[i] = terms(k, 0, 1);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const int k = threadIdx.x + i * NT;
          if (k < n) buf[k] = gv[i];
        }
      }
    } else {
      for (int k = threadIdx.x; k < n; k += NT) {
        double2 acc{0.0, 0.0};
        for (int m = mlo + ((k - mlo) % n + n) % n; m <= L; m += n)
          acc = cadd(acc, cconj(ring_coef(g, m, L, a.spin, a.gstride, ph0)));
        if (!a.spin)  // the m < 0 half of a real field: conj(G_{-m}) = G_m at k = -m mod n
          for (int m = (n - k) % n == 0 ? n : (n - k) % n; m <= L; m += n)
            acc = cadd(acc, ring_coef(g, m, L, 0, a.gstride, ph0));
        buf[k] = acc;
      }
    }
    __syncthreads();
    ring_dft<METHOD, NT, NMAX>(buf, Ld);
    const double th = a.theta[ring];
    const double sth = sin(th), cth = cos(th);  // constant along the ring
    for (int k = threadIdx.x; k < n; k += NT) {
      double2 f = cconj(buf[k]);
      if (a.mode == 0) {
        a.o0[ofs + k] = f.x;
      } else if (a.mode == 1) {
        a.o0[ofs + k] = f.x;
        a.o1[ofs + k] = f.y;
      } else {
        double tp, pp;
        deflect_point_sc(sth, cth, ph0 + k * (2.0 * M_PI / n), f.x, f.y, tp, pp, a.o2 ? &a.o2[ofs + k] : nullptr);
        a.o0[ofs + k] = tp;
        a.o1[ofs + k] = pp;
      }
    }
  } else {
    const double w = a.wt ? a.wt[ring] : 1.0;
    for (int k = threadIdx.x; k < n; k += NT)
      buf[k] = double2{w * a.i0[ofs + k], (a.spin && a.i1) ? w * a.i1[ofs + k] : 0.0};
    __syncthreads();
    ring_dft<METHOD, NT, NMAX>(buf, Ld);
    const int mlo = a.spin ? -L : 0;
    for (int m = mlo + (int)threadIdx.x; m <= L; m += NT) {
      const int k = (m % n + n) % n;
      double2 v = buf[k];
      if (ph0 != 0.0) {
        double s, c;
        sincos(-m * ph0, &s, &c);
        v = cmul(v, double2{c, s});
      }
      a.G[ring + (long)(a.spin ? m + L : m) * a.gstride] = v;
    }
  }
}

using RingKernel = void (*)(RingArgs);

template <int CLASS, RingPass PASS>
RingKernel ring_kernel(int method, bool uniform) {
  constexpr int NT = kRingNT[CLASS], NMAX = kRingNMax[CLASS];
  constexpr int kDirect = (int)DftMethod::Direct, kRader = (int)DftMethod::Rader, kBlue = (int)DftMethod::Bluestein,
                kSplit = (int)DftMethod::Split;
  if constexpr (PASS != kFullBand) {  // (rings of several lengths take the kernel of any length)
    if (!uniform) {
      if constexpr (CLASS == kRingClasses - 1)
        if (method == kSplit) return k_ring<kSplit, false, PASS, NT, NMAX>;
      return method == kDirect ? k_ring<kDirect, false, PASS, NT, NMAX>
             : method == kRader ? k_ring<kRader, false, PASS, NT, NMAX>
             : method == kBlue ? k_ring<kBlue, false, PASS, NT, NMAX> : k_ring<kAnyMethod, false, PASS, NT, NMAX>;
    }
  }
  if constexpr (CLASS == kRingClasses - 1)
    if (method == kSplit) return k_ring<kSplit, true, PASS, NT, NMAX>;
  return method == kDirect ? k_ring<kDirect, true, PASS, NT, NMAX>
         : method == kRader ? k_ring<kRader, true, PASS, NT, NMAX> : k_ring<kBlue, true, PASS, NT, NMAX>;
}

template <RingPass PASS>
RingKernel ring_kernel(int cls, int method, bool uniform) {
  return cls == 0 ? ring_kernel<0, PASS>(method, uniform)
         : cls == 1 ? ring_kernel<1, PASS>(method, uniform) : ring_kernel<2, PASS>(method, uniform);
}

RingKernel ring_kernel(RingPass pass, int cls, int method, bool uniform) {
  return pass == kFullBand ? ring_kernel<kFullBand>(cls, method, uniform)
         : pass == kAliased ? ring_kernel<kAliased>(cls, method, uniform) : ring_kernel<kToRows>(cls, method, uniform);
}

__global__ void k_sqrt_ll(int lmax, double* out) {
  int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l <= lmax) out[l] = sqrt((double)l * (l + 1));
}

}  // namespace

RingPlan::RingPlan(int lmax, int spin, const std::vector<double>& theta, const std::vector<double>& phi0,
                   const std::vector<long>& nph, const std::vector<long>& ofs, const std::vector<double>& weight,
                   hipStream_t st)
    : lmax_(lmax), spin_(spin), nring_((int)theta.size()) {
  NUSHT_REQUIRE(nring_ >= 1, kErrArg, "ringplan: no rings");
  NUSHT_REQUIRE(phi0.size() == theta.size() && nph.size() == theta.size() && ofs.size() == theta.size(), kErrArg,
                "ringplan: ring arrays differ in length");
  NUSHT_REQUIRE(weight.empty() || weight.size() == theta.size(), kErrArg, "ringplan: one weight per ring");
  for (int i = 0; i < nring_; ++i) {
    NUSHT_REQUIRE(theta[i] >= 0.0 && theta[i] <= M_PI, kErrArg, "ringplan: theta outside [0, pi]");
    NUSHT_REQUIRE(nph[i] >= 1 && ofs[i] >= 0, kErrArg, "ringplan: bad nph or ofs");
  }
  npix_ = 0;
  for (int i = 0; i < nring_; ++i) npix_ = std::max(npix_, ofs[i] + nph[i]);
  // one DFT description per distinct ring length
  std::vector<int> lidx(nring_);
  int longest = 0;
  for (int i = 0; i < nring_; ++i) {
    lidx[i] = dft_.add((int)nph[i], st);
    if (nph[i] > nph[longest]) longest = i;
  }
  method_ = (RingMethod)dft_.at(lidx[longest]).method;
  std::vector<RingLen> lv;
  for (int i = 0; i < dft_.size(); ++i) lv.push_back(dft_.at(i));
  upload(lens_, lv);
  upload(lenidx_, lidx);
  nrows_ = spin ? 2 * lmax + 1 : lmax + 1;
  gstride_ = nring_;
  group_rings(lidx, true);
  group_rings(lidx, false);
  upload(theta_, theta);
  upload(phi0_, phi0);
  upload(ofs_, ofs);
  if (!weight.empty()) upload(weight_, weight);
  tab_.tag = "ring";
  tab_.build(lmax, spin, theta, st);
  G_.alloc(sizeof(double2) * (size_t)gstride_ * nrows_);
  coef_.alloc(legendre_coef_bytes(tab_, 1));
  sqll_.alloc(sizeof(double) * (lmax + 1));
  hipLaunchKernelGGL(k_sqrt_ll, dim3(ceil_div(lmax + 1, 256)), dim3(256), 0, st, lmax, sqll_.as<double>());
  NUSHT_LAUNCH_CHECK();
  legendre_autotune(tab_, spin ? 2 : 1, coef_.as<double2>(), G_.as<double2>(), gstride_, 1, st);
  if (spin) legendre_autotune(tab_, 1, coef_.as<double2>(), G_.as<double2>(), gstride_, 1, st);  // E only
}

// Launches of one direction (to_rings: rows -> rings).  Rings are grouped by workgroup size and, above the smallest, by DFT
// method: of the short rings of a ragged grid one launch takes all methods, since every launch lasts as long as its
// slowest ring (HEALPix nside 32, lmax 64: 16 us, 26 with one launch per method), while long ones gain more from a
// kernel of their own (nside 2048, lmax 2500, synthesis: 2.00 ms, 2.19 in one launch).
void RingPlan::group_rings(const std::vector<int>& lidx, bool to_rings) {
  const int band = 2 * lmax_ + 1;
  std::vector<int> values(nring_);
  int most = 0;
  for (int i = 0; i < nring_; ++i) {
    const RingLen& d = dft_.at(lidx[i]);
    values[i] = to_rings ? ring_values(d, nrows_, band) : d.lds_values();
    most = std::max(most, values[i]);
  }
  const bool few = nring_ <= kFewRings && most > kFewRingsValues;
  std::map<int, std::set<int>> methods;  // of each size
  const auto size_of = [&](int i) { return few ? std::max(1, ring_class(most)) : ring_class(values[i]); };
  for (int i = 0; i < nring_; ++i)
    if (dft_.at(lidx[i]).method != (int)DftMethod::Split) methods[size_of(i)].insert(dft_.at(lidx[i]).method);
  std::map<std::pair<int, int>, std::vector<int>> launches;
  for (int i = 0; i < nring_; ++i) {
    int cls = size_of(i), method = dft_.at(lidx[i]).method;
    if (method == (int)DftMethod::Split) cls = kRingClasses - 1;  // long rings only
    else if (methods[cls].size() > 1 && (few || cls == 0)) method = kAnyMethod;
    launches[{cls, method}].push_back(i);
  }
  for (const auto& [key, ids] : launches) {
    RingGroup g;
    g.cls = key.first;
    g.method = key.second;
    g.n = (int)ids.size();
    bool one = true, full = true;
    int v = kRingNT[g.cls];  // (the sums over aliased rows hold one value per thread)
    for (int i : ids) {
      one &= lidx[i] == lidx[ids[0]];
      full &= dft_.at(lidx[i]).n >= band;
      v = std::max(v, values[i]);
    }
    g.one = one ? lidx[ids[0]] : -1;
    if (one) g.method = dft_.at(g.one).method;
    g.pass = !to_rings ? kToRows : one && full ? kFullBand : kAliased;
    g.lds = sizeof(double2) * (size_t)v;
    // Rows that alias are staged in LDS if they fit.  One or two terms per value are as well read in turn where a ring
    // fills a CU (3001 rings of 6000 pixels, lmax 3000, spin 2: 408 us, 442 staged).
    g.stage = nrows_ <= kDftNMAX && !(one && g.cls == kRingClasses - 1 && dft_.at(g.one).n > lmax_);
    upload(g.ids, ids);
    NUSHT_HIP(hipFuncSetAttribute((const void*)ring_kernel((RingPass)g.pass, g.cls, g.method, one),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)(sizeof(double2) * kRingNMax[g.cls])));
    groups_.push_back(std::move(g));
  }
}

size_t RingPlan::bytes() const {
  size_t b = tab_.bytes() + theta_.bytes() + phi0_.bytes() + ofs_.bytes() + weight_.bytes() + sqll_.bytes() +
             G_.bytes() + coef_.bytes() + lens_.bytes() + lenidx_.bytes();
  b += dft_.bytes();
  for (const RingGroup& g : groups_) b += g.ids.bytes();
  return b;
}

void RingPlan::ring_pass(int mode, double* o0, double* o1, double* o2, hipStream_t st, const double* wt) {
  RingArgs a;
  a.lmax = lmax_; a.spin = spin_; a.gstride = gstride_; a.mode = mode;
  a.lenidx = lenidx_.as<int>();
  a.lens = lens_.as<RingLen>();
  a.theta = theta_.as<double>(); a.phi0 = phi0_.as<double>(); a.ofs = ofs_.as<long>();
  a.G = G_.as<double2>();
  a.o0 = o0; a.o1 = o1; a.o2 = o2;
  a.i0 = o0; a.i1 = o1;
  a.wt = wt;
  static const char* names[4] = {"ring_dft_synth_s0", "ring_dft_synth_spin", "ring_dft_pointing", "ring_dft_adjoint"};
  StageScope sc(names[mode], st);
  for (const RingGroup& g : groups_) {
    if ((g.pass == kToRows) != (mode == 3)) continue;
    a.rings = g.ids.as<int>();
    a.stage = g.stage;
    if (g.one >= 0) a.one = dft_.at(g.one);
    hipLaunchKernelGGL(ring_kernel((RingPass)g.pass, g.cls, g.method, g.one >= 0), dim3(g.n), dim3(kRingNT[g.cls]),
                       g.lds, st, a);
    NUSHT_LAUNCH_CHECK();
  }
}

void RingPlan::synthesis(const double2* alm, int ncomp, double* map0, double* map1, hipStream_t st) {
  legendre_synth(tab_, 1, ncomp, alm, 0, nullptr, coef_.as<double2>(), G_.as<double2>(), gstride_, 1, 0, st);
  ring_pass(spin_ ? 1 : 0, map0, map1, nullptr, st);
}

void RingPlan::adjoint(const double* map0, const double* map1, double2* alm, int ncomp, hipStream_t st) {
  ring_pass(3, const_cast<double*>(map0), const_cast<double*>(map1), nullptr, st);
  legendre_adjoint(tab_, ncomp, G_.as<double2>(), gstride_, 1, alm, st);
}

void RingPlan::analysis(const double* map0, const double* map1, double2* alm, int ncomp, hipStream_t st) {
  NUSHT_REQUIRE(has_weights(), kErrState, "ring plan created without ring weights: no analysis");
  ring_pass(3, const_cast<double*>(map0), const_cast<double*>(map1), nullptr, st, weight_.as<double>());
  legendre_adjoint(tab_, ncomp, G_.as<double2>(), gstride_, 1, alm, st);
}

void RingPlan::synthesis_grad(const double2* alm, double* dtheta, double* dphi, hipStream_t st) {
  NUSHT_REQUIRE(spin_ == 1, kErrState, "gradient synthesis needs a spin-1 ring plan");
  legendre_synth(tab_, 1, 1, alm, 0, sqll_.as<double>(), coef_.as<double2>(), G_.as<double2>(), gstride_, 1, 0, st);
  ring_pass(1, dtheta, dphi, nullptr, st);
}

void RingPlan::dlm2pointing(const double2* dlm_scaled, double* ptheta, double* pphi, double* gamma, hipStream_t st) {
  NUSHT_REQUIRE(spin_ == 1, kErrState, "dlm2pointing needs a spin-1 ring plan");
  legendre_synth(tab_, 1, 1, dlm_scaled, 0, sqll_.as<double>(), coef_.as<double2>(), G_.as<double2>(), gstride_, 1, 0,
                 st);
  ring_pass(2, ptheta, pphi, gamma, st);
}

}  // namespace nusht
