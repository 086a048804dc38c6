// qnb_fep.hip -- Qfep6's free-energy analysis on the device, over the energy
// frames a batch has recorded (one window per instance, in instance order):
//
//  * Part 1, free-energy perturbation (src/qfep.f90:587-648): per window i the
//    forward average dgf_i = -kT ln <exp(-(V.lam_{i+1} - V.lam_i)/kT)>_i and the
//    reverse dgr_i towards window i-1, then dG_i = dG_{i-1} + (dgf_{i-1} -
//    dgr_i)/2;
//  * Part 2, reaction free energy per window and energy-gap bin (:700-795):
//    the EVB ground state E_g of two states (:492-500), the gap sum_s c_s V_s
//    binned between the smallest and largest gap of all windows, per bin the
//    averages of E_g - eps and V_s - eps (eps = V.lam_i) and the exponential
//    averages about them, dGg = dG_i - kT ln <exp(-(E_g - eps - av)/kT)> + av;
//  * Part 3 (:797-827): per bin the point-weighted averages over windows.
//
// State energies are formed from each frame as pot_energy forms EQ(s)%total
// (src/potene.f90:224-231: Q bonded terms, then qx = qq + qp + qw, el and
// vdW), plus the alpha shifts (qfep.f90:447-452).  Every sum runs over the
// frames in order, as the reference's loops do (its terms formed in parallel,
// one thread per sum), with no contraction of multiply-add pairs, so the results differ from Qfep6's only
// by the last bits of exp and log.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "qnb_host.h"

#pragma clang fp contract(off)

namespace qnb {

// V_s of frame f (alpha applied), the ground state, c1 and the gap
__device__ void fep_frame(const FepWin& W, const FepPar& P, int f, double* v, double& vg, double& c1, double& gap,
                          double& r) {
  if (W.V) {
    for (int s = 0; s < P.ns; s++) v[s] = W.V[(size_t)f * P.ns + s] + (s == 0 ? 0.0 : P.alpha[s]);
    r = W.noffd > 0 ? W.rkl[f] : 0.0;
  } else {
    const double* h = W.hist + (size_t)f * QNB_FRAME_LEN;
    for (int s = 0; s < P.ns; s++) {
      const double* q = h + QNB_F_Q0 + 6 * s;
      const double* b = h + QNB_F_QB0 + 4 * s;
      const double qxel = q[0] + q[2] + q[4];
      const double qxvdw = q[1] + q[3] + q[5];
      const double total = b[0] + b[1] + b[2] + b[3] + qxel + qxvdw + 0.0;  // + EQ(s)%restraint (none)
      v[s] = total + (s == 0 ? 0.0 : P.alpha[s]);
    }
    r = W.noffd > 0 ? h[QNB_F_OFFD + 1] : 0.0;
  }
  vg = 0.0;
  c1 = 0.0;
  if (P.ns == 2) {
    const double dr = r - P.r0;
    const double H = P.A * exp(-P.mu * dr) * exp(-P.eta * (dr * dr));
    vg = 0.5 * (v[0] + v[1]) - 0.5 * sqrt((v[0] - v[1]) * (v[0] - v[1]) + 4.0 * (H * H));
    if (W.noffd > 0) {
      const double t = (vg - v[0]) / H;
      c1 = 1.0 / (1.0 + t * t);
    }
  }
  gap = 0.0;
  for (int s = 0; s < P.ns; s++) gap = gap + v[s] * P.coeff[s];
}

__device__ double veff_of(const double* lam, const double* v, int ns) {
  double e = 0.0;
  for (int s = 0; s < ns; s++) e = e + lam[s] * v[s];
  return e;
}

// Part 1 sums and the gap range of window blockIdx.x.  The Boltzmann factors
// are formed by every thread, FW_CH frames at a time, and one thread per sum
// adds them from LDS in frame order: 1,000 additions are 8 us of latency, where
// one thread that also formed them took 586 us (51 windows of 1,000 frames),
// 15 us now.
#define FW_CH 1024
__global__ __launch_bounds__(256) void k_fep_window(const FepWin* __restrict__ wins, int n, FepPar P, double* dgf,
                                                    double* dgr, double* wmin, double* wmax) {
  const int i = blockIdx.x, t = threadIdx.x;
  const FepWin& W = wins[i];
  __shared__ double e[2][FW_CH];
  __shared__ double ends[2][4];
  double v[QNB_MAX_STATES], vg, c1, gap, r;
  double lo = INFINITY, hi = -INFINITY, sum = 0.0;
  const bool fwd = i + 1 < n, rev = i > 0;
  const int which = t / QNB_WAVE;  // wave 0 adds the forward sum, wave 1 the reverse one
  for (int f0 = P.nskip; f0 < W.nf; f0 += FW_CH) {
    const int nk = min(FW_CH, W.nf - f0);
    __syncthreads();
    for (int k = t; k < nk; k += blockDim.x) {
      fep_frame(W, P, f0 + k, v, vg, c1, gap, r);
      lo = fmin(lo, gap);
      hi = fmax(hi, gap);
      const double veff1 = veff_of(W.lam, v, P.ns);
      if (fwd) {
        const double dv = veff_of(wins[i + 1].lam, v, P.ns) - veff1;
        e[0][k] = exp(-dv / P.kT);
      }
      if (rev) {
        const double dv = veff_of(wins[i - 1].lam, v, P.ns) - veff1;
        e[1][k] = exp(-dv / P.kT);
      }
    }
    __syncthreads();
    if (t % QNB_WAVE == 0 && ((which == 0 && fwd) || (which == 1 && rev))) {
#pragma unroll 16
      for (int k = 0; k < nk; k++) sum = sum + e[which][k];
    }
  }
  if (t % QNB_WAVE == 0 && which < 2) {
    double out = NAN;
    if (which == 0 ? fwd : rev) {
      sum = sum / (double)(W.nf - P.nskip);
      out = -P.kT * log(sum);
    }
    (which == 0 ? dgf : dgr)[i] = out;
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off));
    hi = fmax(hi, __shfl_xor(hi, off));
  }
  if (t % QNB_WAVE == 0) ends[0][which] = lo, ends[1][which] = hi;
  __syncthreads();
  if (t == 0) {
    wmin[i] = fmin(fmin(ends[0][0], ends[0][1]), fmin(ends[0][2], ends[0][3]));
    wmax[i] = fmax(fmax(ends[1][0], ends[1][1]), fmax(ends[1][2], ends[1][3]));
  }
}

// dG chain and the overall gap range, one wave: the windows' values are read
// 64 at a time, and lane 0 adds them up in order
__global__ __launch_bounds__(64) void k_fep_chain(int n, const double* dgf, const double* dgr, const double* wmin,
                                                  const double* wmax, double* dG, double* range) {
  const int lane = threadIdx.x;
  double lo = INFINITY, hi = -INFINITY, g = 0.0;
  for (int i0 = 0; i0 < n; i0 += QNB_WAVE) {
    const int i = i0 + lane;
    double step = 0.0;
    if (i < n) {
      if (i > 0) step = 0.5 * (dgf[i - 1] - dgr[i]);
      lo = fmin(lo, wmin[i]);
      hi = fmax(hi, wmax[i]);
    }
    double mine = 0.0;
    for (int k = 0; k < min(QNB_WAVE, n - i0); k++) {
      if (i0 + k > 0) g = g + lane_value(step, k);
      if (lane == k) mine = g;
    }
    if (i < n) dG[i] = mine;
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off));
    hi = fmax(hi, __shfl_xor(hi, off));
  }
  if (lane == 0) {
    range[0] = lo;
    range[1] = hi;
  }
}

// Part 2 of window blockIdx.x: thread t owns bin t of a tile of 256 bins and
// takes the window's frames in order.  FB_CH frames at a time are formed by all
// threads into LDS, with the frames of each bin as one bit mask per 64 frames
// (lanes that hold the same bin, by ballots over the bits of its number); a
// bin's thread then walks its masks.  A thread that formed every frame itself
// to find its own took 2,040 us at 51 windows of 1,000 frames and 50 bins; 64
// us now, the length of the walks.  Per (window, bin) rec[] holds dGg, c1, c2,
// r, then dGv of each state; npts the points.  Two states (fep_params).
#define FEP_REC (4 + QNB_MAX_STATES)
#define FB_CH 512
#define FB_BINS 256
struct FepBinLds {
  double val[6][FB_CH];
  uint64_t frames[FB_CH / QNB_WAVE][FB_BINS];
  double av[3][FB_BINS];
};
// adds the N staged values of bin t's frames, in order; clears the masks
template <int N>
__device__ __forceinline__ int fep_bin_walk(FepBinLds& L, int t, double (&s)[N]) {
  int cnt = 0;
  for (int g = 0; g < FB_CH / QNB_WAVE; g++) {
    uint64_t m = L.frames[g][t];
    if (m == 0) continue;
    L.frames[g][t] = 0;
    cnt += __popcll(m);
    while (m != 0) {
      const int f = g * QNB_WAVE + __ffsll((long long)m) - 1;
      m &= m - 1;
#pragma unroll
      for (int c = 0; c < N; c++) s[c] = s[c] + L.val[c][f];
    }
  }
  return cnt;
}
__global__ __launch_bounds__(FB_BINS) void k_fep_bins(const FepWin* __restrict__ wins, FepPar P, const double* dG,
                                                      const double* range, double* rec, int* npts) {
  const int i = blockIdx.x, t = threadIdx.x, lane = t % QNB_WAVE;
  const FepWin& W = wins[i];
  const int ns = P.ns;
  if (!(range[1] > range[0])) return;  // no bins to fill: the host refuses the result
  const double gapmin = range[0];
  const double xint = (range[1] - range[0]) / (double)P.nbins;
  __shared__ FepBinLds L;
  for (int g = 0; g < FB_CH / QNB_WAVE; g++) L.frames[g][t] = 0;
  for (int k0 = 0; k0 < P.nbins; k0 += FB_BINS) {
    const int k = k0 + t, nk = min(FB_BINS, P.nbins - k0);
    // the frames from f0 on into LDS: sums = false, the values to average;
    // true, the exponentials about the averages
    auto stage = [&](int f0, bool sums) {
      for (int u = t; u < FB_CH; u += FB_BINS) {
        const int f = f0 + u;
        double v[QNB_MAX_STATES], vg, c1, gap, r;
        int b = -1;
        if (f < W.nf) {
          fep_frame(W, P, f, v, vg, c1, gap, r);
          const int bin = (int)((gap - gapmin) / xint);
          if (bin >= k0 && bin < k0 + nk) b = bin - k0;
        }
        uint64_t same = __ballot(b >= 0);
        for (int bit = 1; bit < nk; bit <<= 1) {
          const uint64_t m = __ballot(b & bit);
          same &= (b & bit) ? m : ~m;
        }
        if (b >= 0) {
          if ((same & ((1ull << lane) - 1ull)) == 0) L.frames[u / QNB_WAVE][b] = same;
          const double veff = veff_of(W.lam, v, ns);
          if (sums) {
            for (int s = 0; s < 2; s++) L.val[s][u] = exp(-(v[s] - veff - L.av[s][b]) / P.kT);
            L.val[2][u] = exp(-(vg - veff - L.av[2][b]) / P.kT);
          } else {
            for (int s = 0; s < 2; s++) L.val[s][u] = v[s] - veff;
            L.val[2][u] = vg - veff;
            L.val[3][u] = c1;
            L.val[4][u] = r;
            L.val[5][u] = W.noffd > 0 ? 1.0 - c1 : 0.0;
          }
        }
      }
    };
    // per bin: V_s - eps, E_g - eps, c1, r, c2
    double av[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, sum[3] = {0.0, 0.0, 0.0};
    int cnt = 0;
    for (int f0 = P.nskip; f0 < W.nf; f0 += FB_CH) {
      __syncthreads();
      stage(f0, false);
      __syncthreads();
      if (t < nk) cnt += fep_bin_walk(L, t, av);
    }
    if (cnt != 0)
      for (int c = 0; c < 6; c++) av[c] = av[c] / (double)cnt;
    for (int c = 0; c < 3; c++) L.av[c][t] = av[c];
    for (int f0 = P.nskip; f0 < W.nf; f0 += FB_CH) {
      __syncthreads();
      stage(f0, true);
      __syncthreads();
      if (t < nk) fep_bin_walk(L, t, sum);
    }
    if (t < nk) {
      double* o = rec + ((size_t)i * P.nbins + k) * FEP_REC;
      npts[(size_t)i * P.nbins + k] = cnt;
      if (cnt > 0 && cnt >= P.nmin) {
        for (int s = 0; s < 2; s++) o[4 + s] = dG[i] + (-P.kT * log(sum[s] / (double)cnt) + av[s]);
        o[0] = dG[i] + (-P.kT * log(sum[2] / (double)cnt) + av[2]);
        o[1] = av[3];
        o[2] = av[5];
        o[3] = av[4];
      } else {
        for (int z = 0; z < FEP_REC; z++) o[z] = NAN;
      }
    }
  }
}

// Part 3: per bin, the windows in order, FP3_U of them requested at a time
#define FP3_U 8
__global__ __launch_bounds__(256) void k_fep_part3(int n, FepPar P, const double* range, const double* rec,
                                                   const int* npts, double* bins, int* ptsum) {
  if (!(range[1] > range[0])) return;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < P.nbins; k += gridDim.x * blockDim.x) {
    double b[4] = {0.0, 0.0, 0.0, 0.0};
    int pt = 0;
    for (int i0 = 0; i0 < n; i0 += FP3_U) {
      int c[FP3_U];
      double o[FP3_U][4];
#pragma unroll
      for (int u = 0; u < FP3_U; u++) {
        const size_t w = (size_t)min(i0 + u, n - 1) * P.nbins + k;
        c[u] = i0 + u < n ? npts[w] : 0;
        for (int z = 0; z < 4; z++) o[u][z] = rec[w * FEP_REC + z];
      }
#pragma unroll
      for (int u = 0; u < FP3_U; u++) {
        if (c[u] == 0 || c[u] < P.nmin) continue;
        pt += c[u];
        for (int z = 0; z < 4; z++) b[z] = b[z] + o[u][z] * (double)c[u];
      }
    }
    ptsum[k] = pt;
    const bool ok = pt > 0 && pt >= P.nmin;
    for (int z = 0; z < 4; z++) bins[4 * k + z] = ok ? b[z] / (double)pt : NAN;
  }
}

// Scratch layout: one device buffer of fep_scratch_doubles(n, nbins)
// doubles holds every intermediate and output, at the offsets fep_layout
// gives (the last region holds the int32 point counts).
void fep_layout(int n, int nbins, size_t off[8]) {
  off[0] = 0;                                  // dgf [n]
  off[1] = off[0] + n;                         // dgr [n]
  off[2] = off[1] + n;                         // dG [n]
  off[3] = off[2] + n;                         // wmin, wmax [2n]
  off[4] = off[3] + 2 * (size_t)n;             // range [2]
  off[5] = off[4] + 2;                         // rec [n][nbins][FEP_REC]
  off[6] = off[5] + (size_t)n * nbins * FEP_REC;  // bins [nbins][4]
  off[7] = off[6] + 4 * (size_t)nbins;         // ints follow: npts [n][nbins], ptsum [nbins]
}
size_t fep_scratch_doubles(int n, int nbins) {
  size_t off[8];
  fep_layout(n, nbins, off);
  return off[7] + ((size_t)n * nbins + nbins + 1) / 2 + 1;
}
size_t fep_rec_len() { return FEP_REC; }

// Part 1 and the gap range
void launch_fep_part1(hipStream_t st, const FepWin* wins, int n, const FepPar& P, double* scratch) {
  size_t off[8];
  fep_layout(n, P.nbins, off);
  double* sd = scratch;
  hipLaunchKernelGGL(k_fep_window, dim3(n), dim3(256), 0, st, wins, n, P, sd + off[0], sd + off[1], sd + off[3],
                     sd + off[3] + n);
  hipLaunchKernelGGL(k_fep_chain, dim3(1), dim3(64), 0, st, n, sd + off[0], sd + off[1], sd + off[3], sd + off[3] + n,
                     sd + off[2], sd + off[4]);
}

// Parts 2 and 3 (P.nbins > 0); nothing is written where the gap range is empty
void launch_fep_bins(hipStream_t st, const FepWin* wins, int n, const FepPar& P, double* scratch) {
  size_t off[8];
  fep_layout(n, P.nbins, off);
  double* sd = scratch;
  int* npts = reinterpret_cast<int*>(sd + off[7]);
  hipLaunchKernelGGL(k_fep_bins, dim3(n), dim3(FB_BINS), 0, st, wins, P, sd + off[2], sd + off[4], sd + off[5], npts);
  hipLaunchKernelGGL(k_fep_part3, dim3((P.nbins + 255) / 256), dim3(256), 0, st, n, P, sd + off[4], sd + off[5], npts,
                     sd + off[6], npts + (size_t)n * P.nbins);
}

// Runs the analysis and copies the results out.  hw: the window records, whose
// data sit in device memory already or come with the tables of `pack`.
int fep_run(hipStream_t st, std::vector<FepWin>& hw, const FepPar& P, qnb_fep_out* out, DevPack& pack) {
  const int n = (int)hw.size();
  DevAlloc mem;
  const FepWin* dw = nullptr;
  double* sd = nullptr;
  size_t off[8];
  fep_layout(n, P.nbins, off);
  const size_t nd = fep_scratch_doubles(n, P.nbins);
  pack.add(&dw, (const FepWin*)hw.data(), hw.size());
  pack.space(&sd, nd);
  if (int rc = pack.alloc(mem)) return rc;
  if (int rc = pack.copy()) return rc;
  launch_fep_part1(st, dw, n, P, sd);
  if (P.nbins > 0) launch_fep_bins(st, dw, n, P, sd);
  HIPCHK(hipGetLastError());
  std::unique_ptr<double[]> host(new (std::nothrow) double[nd]);
  if (!host) return fail(QNB_ENOMEM, "no host memory for %zu results", nd);
  const double* h = host.get();
  HIPCHK(hipMemcpyAsync(host.get(), sd, nd * sizeof(double), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  const double* range = h + off[4];
  if (P.nbins > 0 && !(range[1] > range[0])) return fail(QNB_EINVAL, "energy gap range is empty: no bins to fill");
  auto put = [](double* dst, const double* src, size_t k) {
    if (dst) memcpy(dst, src, k * sizeof(double));
  };
  put(out->dgf, h + off[0], n);
  put(out->dgr, h + off[1], n);
  put(out->dG, h + off[2], n);
  put(out->gap_range, range, 2);
  const size_t nb = (size_t)n * P.nbins;
  const double *rec = h + off[5], *bins = h + off[6];
  const int32_t* ints = reinterpret_cast<const int32_t*>(h + off[7]);
  for (size_t w = 0; w < nb; w++) {
    const double* o = rec + w * FEP_REC;
    if (out->dGg) out->dGg[w] = o[0];
    if (out->c1) out->c1[w] = o[1];
    if (out->c2) out->c2[w] = o[2];
    if (out->r) out->r[w] = o[3];
    if (out->dGv)
      for (int s2 = 0; s2 < P.ns; s2++) out->dGv[w * P.ns + s2] = o[4 + s2];
    if (out->npts) out->npts[w] = ints[w];
  }
  for (int k = 0; k < P.nbins; k++) {
    if (out->bin_dGg) out->bin_dGg[k] = bins[4 * k];
    if (out->bin_c1) out->bin_c1[k] = bins[4 * k + 1];
    if (out->bin_c2) out->bin_c2[k] = bins[4 * k + 2];
    if (out->bin_r) out->bin_r[k] = bins[4 * k + 3];
    if (out->ptsum) out->ptsum[k] = ints[nb + k];
  }
  return 0;
}

int fep_params(const qnb_fep_params* p, int ns, FepPar* P) {
  if (!p) return fail(QNB_EINVAL, "no parameters");
  if (!(p->kT > 0.0)) return fail(QNB_EINVAL, "kT must be positive");
  if (ns < 1 || ns > QNB_MAX_STATES) return fail(QNB_EINVAL, "nstates must be 1..%d", QNB_MAX_STATES);
  if (p->nskip < 0 || p->nbins < 0 || p->nmin < 0) return fail(QNB_EINVAL, "nskip, nbins and nmin must be >= 0");
  if (p->nbins > 0 && ns != 2)
    return fail(QNB_EINVAL, "the reaction free energy (nbins > 0) needs the 2-state EVB ground state");
  P->kT = p->kT;
  P->nskip = p->nskip;
  P->nbins = p->nbins;
  P->nmin = p->nmin;
  P->ns = ns;
  for (int s = 0; s < QNB_MAX_STATES; s++) {
    P->alpha[s] = s == 0 ? 0.0 : p->alpha[s];  // alfa(1) = zero (qfep.f90:447)
    P->coeff[s] = p->coeff[s];
  }
  P->A = p->A;
  P->mu = p->mu;
  P->eta = p->eta;
  P->r0 = p->r0;
  return 0;
}

}  // namespace qnb

using namespace qnb;

extern "C" int32_t qnb_free_energy(int32_t nwin, int32_t nstates, const int32_t* nframes, const double* const* V,
                                   const double* const* rkl, const double* lambdas, const qnb_fep_params* p,
                                   qnb_fep_out* out) {
  if (nwin < 1 || !nframes || !V || !lambdas || !out) return fail(QNB_EINVAL, "bad arguments");
  FepPar P;
  if (int rc = fep_params(p, nstates, &P)) return rc;
  DevPack pack;
  std::vector<FepWin> hw(nwin);
  for (int w = 0; w < nwin; w++) {
    if (!V[w] || nframes[w] <= P.nskip)
      return fail(QNB_EINVAL, "window %d has no frames after the %d skipped", w, P.nskip);
    FepWin& W = hw[w];
    W.hist = nullptr;
    W.nf = nframes[w];
    W.noffd = (rkl && rkl[w]) ? 1 : 0;
    W.rkl = nullptr;
    pack.add(&W.V, V[w], (size_t)nframes[w] * nstates);
    if (W.noffd) pack.add(&W.rkl, rkl[w], (size_t)nframes[w]);
    for (int s = 0; s < QNB_MAX_STATES; s++) W.lam[s] = s < nstates ? lambdas[(size_t)w * nstates + s] : 0.0;
  }
  return fep_run(nullptr, hw, P, out, pack);
}
