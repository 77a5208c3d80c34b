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

namespace nusht {
namespace {

// Workgroup sizes by the values a ring's DFT holds in LDS.  Every thread keeps about eight values in registers (105 -
// 127 VGPRs, four waves per SIMD), so a workgroup of the largest size fills a CU whatever its ring's length; with
// smaller ones four rings of up to 2048 values, or two of up to 4160, run on a CU and cover each other's barriers
// and loads.  Measured with 768 threads for every ring and now: 301 rings of 625 values (lmax 300)
// 28 -> 21 us; 1501 rings of 3072 values (lmax 1500), synthesis 100 -> 70 us, adjoint 94 -> 78 us.
constexpr int kRingClasses = 3;
constexpr int kRingNT[kRingClasses] = {256, 512, kDftNT};
constexpr int kRingNMax[kRingClasses] = {2048, 4160, kDftNMAX};

// LDS values of a ring's workgroup: its DFT and, for a ring shorter than its band, the rows that alias onto it
// (those of a band that does not fit are read term by term)
int ring_values(const RingLen& d, int nrow, int band) {
  return d.n >= band || nrow > kDftNMAX ? d.lds_values() : std::max(d.lds_values(), nrow);
}

int ring_class(const RingLen& d, int values) {
  if (d.method == (int)DftMethod::Split) return kRingClasses - 1;  // long rings only
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

// UNIFORM: every ring of the launch has the length a.one >= 2 lmax + 1 (read from the kernel arguments) and the DFT method
// METHOD; otherwise each ring reads its description from a.lens, may be shorter than its band and, with kAnyMethod,
// takes its own method (all but the split): ragged grids run as one launch per workgroup size, since every launch
// lasts as long as its slowest ring (HEALPix nside 512, lmax 1000: 218 us, 241 us with one launch per DFT method).
constexpr int kAnyMethod = -1;

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

template <int METHOD, bool UNIFORM, int NT, int NMAX>
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
  if (a.mode < 3) {
    // conjugated spectrum for the inverse DFT: X[m mod n] = sum conj(G_m e^{i m phi0}) over the m that alias there
    const int mlo = a.spin ? -L : 0;
    if (UNIFORM || n >= 2 * L + 1) {
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
      // nside 512, lmax 1000, took 347 us in three launches (one per DFT method), now 218 us.
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

template <int CLASS>
RingKernel ring_kernel(int method, bool uniform) {
  constexpr int NT = kRingNT[CLASS], NMAX = kRingNMax[CLASS];
  if constexpr (CLASS == kRingClasses - 1) {
    if (method == (int)DftMethod::Split) return uniform ? k_ring<3, true, NT, NMAX> : k_ring<3, false, NT, NMAX>;
  }
  if (!uniform) return k_ring<kAnyMethod, false, NT, NMAX>;
  if (method == (int)DftMethod::Direct) return k_ring<0, true, NT, NMAX>;
  return method == (int)DftMethod::Rader ? k_ring<1, true, NT, NMAX> : k_ring<2, true, NT, NMAX>;
}

RingKernel ring_kernel(int cls, int method, bool uniform) {
  return cls == 0 ? ring_kernel<0>(method, uniform)
         : cls == 1 ? ring_kernel<1>(method, uniform) : ring_kernel<2>(method, uniform);
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
  // one DFT description per distinct ring length; rings grouped by workgroup size, the split DFTs apart
  static_assert(kRingGroups == kRingClasses + 1, "one launch per workgroup size and one for the split DFTs");
  std::vector<int> lidx(nring_);
  std::vector<std::vector<int>> by_group(kRingGroups);
  int longest = 0;
  for (int i = 0; i < nring_; ++i) {
    lidx[i] = dft_.add((int)nph[i], st);
    const RingLen& d = dft_.at(lidx[i]);
    const int values = ring_values(d, spin ? 2 * lmax + 1 : lmax + 1, 2 * lmax + 1);
    const int cls = ring_class(d, values);
    const int grp = d.method == (int)DftMethod::Split ? kRingClasses : cls;
    by_group[grp].push_back(i);
    // (the sums over aliased rows hold one value per thread)
    lds_[grp] = std::max(lds_[grp], sizeof(double2) * (size_t)std::max(values, kRingNT[cls]));
    if (nph[i] > nph[longest]) longest = i;
  }
  method_ = (RingMethod)dft_.at(lidx[longest]).method;
  std::vector<RingLen> lv;
  for (int i = 0; i < dft_.size(); ++i) lv.push_back(dft_.at(i));
  upload(lens_, lv);
  upload(lenidx_, lidx);
  for (int m = 0; m < kRingGroups; ++m) {
    nrings_m_[m] = (int)by_group[m].size();
    if (nrings_m_[m]) upload(rings_[m], by_group[m]);
    uniform_[m] = -1;
    for (int i : by_group[m]) {
      if (uniform_[m] == -1) uniform_[m] = lidx[i];
      else if (uniform_[m] != lidx[i]) { uniform_[m] = -2; break; }
    }
  }
  for (int cls = 0; cls < kRingClasses; ++cls)
    for (int method = 0; method < (cls == kRingClasses - 1 ? kDftMethods : (int)DftMethod::Split); ++method)
      for (bool uni : {false, true})
        NUSHT_HIP(hipFuncSetAttribute((const void*)ring_kernel(cls, method, uni),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)(sizeof(double2) * kRingNMax[cls])));
  upload(theta_, theta);
  upload(phi0_, phi0);
  upload(ofs_, ofs);
  if (!weight.empty()) upload(weight_, weight);
  tab_.tag = "ring";
  tab_.build(lmax, spin, theta, st);
  nrows_ = spin ? 2 * lmax + 1 : lmax + 1;
  gstride_ = nring_;
  G_.alloc(sizeof(double2) * (size_t)gstride_ * nrows_);
  coef_.alloc(legendre_coef_bytes(tab_, 1));
  sqll_.alloc(sizeof(double) * (lmax + 1));
  hipLaunchKernelGGL(k_sqrt_ll, dim3(ceil_div(lmax + 1, 256)), dim3(256), 0, st, lmax, sqll_.as<double>());
  NUSHT_LAUNCH_CHECK();
  legendre_autotune(tab_, spin ? 2 : 1, coef_.as<double2>(), G_.as<double2>(), gstride_, 1, st);
  if (spin) legendre_autotune(tab_, 1, coef_.as<double2>(), G_.as<double2>(), gstride_, 1, st);  // E only
}

size_t RingPlan::bytes() const {
  size_t b = tab_.bytes() + theta_.bytes() + phi0_.bytes() + ofs_.bytes() + weight_.bytes() + sqll_.bytes() +
             G_.bytes() + coef_.bytes() + lens_.bytes() + lenidx_.bytes();
  b += dft_.bytes();
  for (int m = 0; m < kRingGroups; ++m) b += rings_[m].bytes();
  return b;
}

void RingPlan::ring_pass(int mode, double* o0, double* o1, double* o2, hipStream_t st, const double* wt) {
  RingArgs a;
  a.lmax = lmax_; a.spin = spin_; a.gstride = gstride_; a.mode = mode;
  a.stage = nrows_ <= kDftNMAX ? 1 : 0;
  a.lenidx = lenidx_.as<int>();
  a.lens = lens_.as<RingLen>();
  a.theta = theta_.as<double>(); a.phi0 = phi0_.as<double>(); a.ofs = ofs_.as<long>();
  a.G = G_.as<double2>();
  a.o0 = o0; a.o1 = o1; a.o2 = o2;
  a.i0 = o0; a.i1 = o1;
  a.wt = wt;
  static const char* names[4] = {"ring_dft_synth_s0", "ring_dft_synth_spin", "ring_dft_pointing", "ring_dft_adjoint"};
  StageScope sc(names[mode], st);
  for (int m = 0; m < kRingGroups; ++m) {
    if (!nrings_m_[m]) continue;
    a.rings = rings_[m].as<int>();
    const bool uni = uniform_[m] >= 0 && dft_.at(uniform_[m]).n >= 2 * lmax_ + 1;
    if (uni) a.one = dft_.at(uniform_[m]);
    const int cls = std::min(m, kRingClasses - 1);
    const int method = m == kRingClasses ? (int)DftMethod::Split : uni ? a.one.method : (int)DftMethod::Direct;
    const RingKernel k = ring_kernel(cls, method, uni);
    hipLaunchKernelGGL(k, dim3(nrings_m_[m]), dim3(kRingNT[cls]), lds_[m], st, a);
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
