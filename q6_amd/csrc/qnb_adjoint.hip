// qnb_adjoint.hip -- adjoint of the per-state Q-atom energies over stored
// frames: for every frame f, state s and Q-atom iq the kernel returns
//   dE_s/d(charge of iq in s), dE_s/d(LJ A and B factors of iq in s) for
//   normal and 1-4 pairs, and iq's share of E_s (el, vdw),
// where E_s = EQ(s)%qq + %qp + %qw (src/potene.f90:224-229) recomputed from the
// frame.  Each Q table entry is a product of a Q-side parameter and a partner
// factor (precompute_set_values_qp/qq/qw, src/simprep.f90:3420-3589); the
// caller passes the derivative of every entry with respect to its Q-side
// parameter (the tangent tables), so the kernel only sums tangent x radial
// function over the pairs.  The Q lists are recomputed per frame with the
// criteria of nbqplist/nbqwlist (src/nonbondene.f90:3647-3742, 3862-3944):
// nothing from the MD's lists is stored.  Pair math in R (float for the
// FP32 backward, double for validation), every sum in FP64.
#include <hip/hip_runtime.h>

#include "qnb_host.h"

namespace qnb {

// one pair's parameters in one state: LJ and Coulomb, soft core, tangents
template <typename R>
struct AdjPar {
  R A, B, el, sc, tq, tA, tB;
};

template <typename R>
__device__ __forceinline__ void adj_pair(double (&g)[QNB_ADJ_NV], R r2, R r, const AdjPar<R>& p, bool is14, bool lj,
                                         bool energy) {
  g[ADJ_DQ] += (double)(p.tq * r);
  if (energy) g[ADJ_EEL] += (double)(p.el * r);
  if (!lj) return;
  R r6 = r2 * r2 * r2;
  if (p.sc != R(0)) r6 = recip(recip(r6) + p.sc);
  const R r12 = r6 * r6;
  const double gA = (double)(p.tA * r12), gB = (double)(p.tB * r6);
  if (is14) {
    g[ADJ_DA14] += gA;
    g[ADJ_DB14] -= gB;
  } else {
    g[ADJ_DA] += gA;
    g[ADJ_DB] -= gB;
  }
  if (energy) g[ADJ_EVDW] += (double)(p.A * r12) - (double)(p.B * r6);
}

// One block per (frame, Q-atom), its four waves taking every fourth 64 waters,
// solute atoms and Q pairs; grid.y = instance, rows of blocks along z.  A wave's pass is a few dozen
// iterations of dependent loads, so the kernel is bound by their latency until
// the waves fill the chip: four waves per sum instead of one, the Q-water
// tables of a site held over the waters, and each solute atom's list test from
// its own word (qp_test) instead of through group, switch atom and exclusion
// take 6 instances x 20 frames x 30 Q-atoms of 1,200 + 3,100 atoms from 175 to
// 158 us (FP32 pairs), and a water read once for its three sites to 100; 24
// frames x 18 Q-atoms from 50 to 20 and 17 us (FP64).
#define ADJ_WPB 4
template <typename R, int NS>
__global__ __launch_bounds__(QNB_WAVE* ADJ_WPB) void k_adjoint(const DevSys* __restrict__ systems,
                                                               const AdjDev* __restrict__ adjs) {
  const DevSys& S = systems[blockIdx.y];
  const AdjDev& A = adjs[blockIdx.y];
  const int nq = S.nqat, ns = S.nstates, sa = S.sa, nsol = S.nat_solute;
  if (nq <= 0) return;
  const int t0 = threadIdx.x, lane = t0 % QNB_WAVE;
  const uint32_t blk = blockIdx.z * gridDim.x + blockIdx.x;
  const int f = (int)(blk / (uint32_t)nq), iq = (int)(blk % (uint32_t)nq);
  if (f >= A.nframes) return;
  const auto x = gp(A.frames + (size_t)f * 3 * S.natom);
  const int i = S.iqseq[iq];
  const double xi0 = x[3 * i], xi1 = x[3 * i + 1], xi2 = x[3 * i + 2];
  const double xp0 = S.xp[0], xp1 = S.xp[1], xp2 = S.xp[2], rcq2 = S.rcq2;
  double g[NS][QNB_ADJ_NV];
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int c = 0; c < QNB_ADJ_NV; c++) g[s][c] = 0.0;
  auto inv = [&](double ax, double ay, double az, double bx, double by, double bz, R& r2, R& r) {
    const R ux = (R)(ax - bx), uy = (R)(ay - by), uz = (R)(az - bz);
    rinv(ux * ux + uy * uy + uz * uz, r2, r);
  };
  // dist4p's sum for the point (a, b, c) and the Q-list centre
  auto dist2 = [&](double a, double b, double c) {
#pragma clang fp contract(off)
    const double dx = xp0 - a, dy = xp1 - b, dz = xp2 - c;
    double d = dx * dx;
    d = d + dy * dy;
    d = d + dz * dz;
    return d;
  };

  // Q-water: every water whose oxygen lies within Rcq of the Q-list centre; one
  // whose position is not a number is not left out, so that its frame's results
  // show it
  const auto qw_par = [&](int k, int s) {
    const size_t t = (size_t)iq + (size_t)nq * ((size_t)k + (size_t)sa * s);
    return AdjPar<R>{(R)ldg(S.qwA + t), (R)ldg(S.qwB + t), (R)ldg(S.qwEl + t), (R)ldg(S.qwSc + t),
                     (R)ldg(A.qw_dq + t), (R)ldg(A.qw_dA + t), (R)ldg(A.qw_dB + t)};
  };
  if (sa == 3) {
    // a water's nine coordinates in one run, the parameters of its sites in LDS
    // (the same for every lane): the loads' 72-byte strides, not the pairs, are
    // what a pass per site waits for
    __shared__ AdjPar<R> par[3][NS];
    if (t0 < 3 * ns && S.nwat > 0) par[t0 / ns][t0 % ns] = qw_par(t0 / ns, t0 % ns);
    __syncthreads();
    for (int w = t0; w < S.nwat; w += QNB_WAVE * ADJ_WPB) {
      const int o = nsol + 3 * w;
      double xw[3][3];
      for (int k = 0; k < 3; k++)
        for (int c = 0; c < 3; c++) xw[k][c] = x[3 * (o + k) + c];
      if (ldg(S.excl + o) || dist2(xw[0][0], xw[0][1], xw[0][2]) > rcq2) continue;
      __asm__ volatile("" ::: "memory");  // the parameters stay in LDS, not in registers over the loop
#pragma unroll
      for (int k = 0; k < 3; k++) {
        R r2, r;
        inv(xw[k][0], xw[k][1], xw[k][2], xi0, xi1, xi2, r2, r);
#pragma unroll
        for (int s = 0; s < NS; s++) {
          if (s >= ns) break;
          adj_pair<R>(g[s], r2, r, par[k][s], false, k == 0 || !S.spc, true);
        }
      }
    }
  } else {
    for (int k = 0; k < sa; k++) {
      AdjPar<R> p[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        if (s >= ns || S.nwat <= 0) break;
        p[s] = qw_par(k, s);
      }
      const bool lj = k == 0 || !S.spc;
      for (int w = t0; w < S.nwat; w += QNB_WAVE * ADJ_WPB) {
        const int o = nsol + sa * w, j = o + k;
        const double ox = x[3 * o], oy = x[3 * o + 1], oz = x[3 * o + 2];
        const double jx = x[3 * j], jy = x[3 * j + 1], jz = x[3 * j + 2];
        if (ldg(S.excl + o) || dist2(ox, oy, oz) > rcq2) continue;
        R r2, r;
        inv(jx, jy, jz, xi0, xi1, xi2, r2, r);
#pragma unroll
        for (int s = 0; s < NS; s++) {
          if (s >= ns) break;
          adj_pair<R>(g[s], r2, r, p[s], false, lj, true);
        }
      }
    }
  }
  // the Q tables' entry t of the Q-solute pairs
  auto qp_par = [&](size_t t) {
    return AdjPar<R>{(R)ldg(S.qpA + t), (R)ldg(S.qpB + t), (R)ldg(S.qpEl + t), (R)ldg(S.qpSc + t),
                     (R)ldg(A.qp_dq + t), (R)ldg(A.qp_dA + t), (R)ldg(A.qp_dB + t)};
  };
  // Q-solute: atoms of solute groups inside Rcq (switch atom, or any atom
  // with iuse_switch_atom = 0), not 1-2/1-3 bonded to any Q-atom
#pragma unroll 2
  for (int j = t0; j < nsol; j += QNB_WAVE * ADJ_WPB) {
    const int sw = ldg(S.qp_test + j);
    if (sw < 0) continue;
    if (S.any_atom) {
      if (!qp_group_in(S, A.frames + (size_t)f * 3 * S.natom, ldg(S.atom_group + j))) continue;
    } else if (!(dist2(x[3 * sw], x[3 * sw + 1], x[3 * sw + 2]) <= rcq2)) {
      continue;
    }
    R r2, r;
    inv(x[3 * j], x[3 * j + 1], x[3 * j + 2], xi0, xi1, xi2, r2, r);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if (s >= ns) break;
      const size_t t = (size_t)j + (size_t)nsol * ((size_t)iq + (size_t)nq * s);
      adj_pair<R>(g[s], r2, r, qp_par(t), ldg(A.qp_is14 + t) != 0, true, true);
    }
  }
  // Q-Q pairs with iq as either member; the energy is counted by the lower one
  for (int q = t0; q < S.nqq; q += QNB_WAVE * ADJ_WPB) {
    const int ia = S.qq_iq[q], ja = S.qq_jq[q];
    if (ia != iq && ja != iq) continue;
    const int st = S.qq_st[q];
    const int a = S.iqseq[ia], b = S.iqseq[ja];
    R r2, r;
    inv(x[3 * b], x[3 * b + 1], x[3 * b + 2], x[3 * a], x[3 * a + 1], x[3 * a + 2], r2, r);
    const double* pr = S.qq_par + 4 * q;
    const size_t t = (size_t)ia + (size_t)nq * ((size_t)ja + (size_t)nq * st);
    const bool mine = ia == iq;
    const R tq = (R)(mine ? A.qq_dq_i[t] : A.qq_dq_j[t]);
    const bool soft = S.qq_soft[q], is14 = A.qq_is14[t] != 0;
    const R tA = (R)(mine ? A.qq_dA_i[t] : A.qq_dA_j[t]);
    const R tB = (R)(mine ? A.qq_dB_i[t] : A.qq_dB_j[t]);
#pragma unroll
    for (int k = 0; k < NS; k++) {
      if (k != st) continue;
      if (soft) {
        // exponential soft pair: its A, B are not LJ factors (no LJ tangent)
        g[k][ADJ_DQ] += (double)(tq * r);
        if (mine) {
          g[k][ADJ_EEL] += (double)((R)pr[2] * r);
          g[k][ADJ_EVDW] += (double)((R)pr[0] * exp(-(R)pr[1] / r));
        }
      } else {
        adj_pair<R>(g[k], r2, r, AdjPar<R>{(R)pr[0], (R)pr[1], (R)pr[2], (R)pr[3], tq, tA, tB}, is14, true, mine);
      }
    }
  }
  // Q-bonded-neighbour pairs of iq (entries of the qp tables)
  for (int q = t0; q < S.nqqp; q += QNB_WAVE * ADJ_WPB) {
    if (S.qqp_iq[q] != iq) continue;
    const int j = S.qqp_j[q], st = S.qqp_st[q];
    R r2, r;
    inv(x[3 * j], x[3 * j + 1], x[3 * j + 2], xi0, xi1, xi2, r2, r);
    const double* pr = S.qqp_par + 4 * q;
    const size_t t = (size_t)j + (size_t)nsol * ((size_t)iq + (size_t)nq * st);
    const AdjPar<R> p{(R)pr[0], (R)pr[1], (R)pr[2], (R)pr[3], (R)A.qp_dq[t], (R)A.qp_dA[t], (R)A.qp_dB[t]};
#pragma unroll
    for (int k = 0; k < NS; k++)
      if (k == st) adj_pair<R>(g[k], r2, r, p, A.qp_is14[t] != 0, true, true);
  }
  // the block's sums, in wave order
  constexpr int NV = NS * QNB_ADJ_NV;
  __shared__ double part[ADJ_WPB][64];
  double v[NV];
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int c = 0; c < QNB_ADJ_NV; c++) v[s * QNB_ADJ_NV + c] = g[s][c];
  const double sum = wave_sum_tr<double, NV>(v, lane);
  if (wave_sum_tr_writer<NV>(lane)) part[t0 / QNB_WAVE][wave_sum_tr_index<NV>(lane)] = sum;
  __syncthreads();
  if (t0 < ns * QNB_ADJ_NV) {
    const int s = t0 / QNB_ADJ_NV, c = t0 % QNB_ADJ_NV;
    double e = part[0][t0];
    for (int w = 1; w < ADJ_WPB; w++) e += part[w][t0];
    A.out[(((size_t)f * ns + s) * nq + iq) * QNB_ADJ_NV + c] = e;
  }
}

// Adds a caller's tangent tables to a pack (sizes from the system); A, whose
// pointers the pack sets, and the tables stay in place until it is copied.
int adjoint_pack(DevPack& M, const DevSys& S, const qnb_qtangent* t, AdjDev& A) {
  if (!t) return fail(QNB_EINVAL, "null tangent tables");
  const size_t nq = S.nqat, ns = S.nstates, nsol = S.nat_solute, sa = S.sa;
  const size_t np = nsol * nq * ns, nw = S.nwat > 0 ? nq * sa * ns : 0, nqq = nq * nq * ns;
#define UPT(field, n)                                                                     \
  do {                                                                                    \
    if ((n) > 0 && !t->field) return fail(QNB_EINVAL, "tangent table " #field " missing"); \
    M.add(&A.field, (n) > 0 ? t->field : nullptr, (n));                                   \
  } while (0)
  UPT(qp_dq, np);
  UPT(qp_dA, np);
  UPT(qp_dB, np);
  UPT(qp_is14, np);
  UPT(qw_dq, nw);
  UPT(qw_dA, nw);
  UPT(qw_dB, nw);
  UPT(qq_dq_i, nqq);
  UPT(qq_dA_i, nqq);
  UPT(qq_dB_i, nqq);
  UPT(qq_dq_j, nqq);
  UPT(qq_dA_j, nqq);
  UPT(qq_dB_j, nqq);
  UPT(qq_is14, nqq);
#undef UPT
  return 0;
}

// A launch holds fewer than 2^32 threads along x: 16.7 million blocks, which
// 84,000 frames of 200 Q-atoms pass; more than 2^22 blocks are laid out in
// several rows along z.
template <typename R>
static void launch_adj_r(hipStream_t st, int ns_max, long blocks, int B, const DevSys* dsys, const AdjDev* dadj) {
  const long most = 1l << 22, rows = (blocks + most - 1) / most;
  dim3 grid((unsigned)((blocks + rows - 1) / rows), B, (unsigned)rows), block(QNB_WAVE * ADJ_WPB);
  if (ns_max <= 1) hipLaunchKernelGGL((k_adjoint<R, 1>), grid, block, 0, st, dsys, dadj);
  else if (ns_max <= 2) hipLaunchKernelGGL((k_adjoint<R, 2>), grid, block, 0, st, dsys, dadj);
  else if (ns_max <= 4) hipLaunchKernelGGL((k_adjoint<R, 4>), grid, block, 0, st, dsys, dadj);
  else hipLaunchKernelGGL((k_adjoint<R, 8>), grid, block, 0, st, dsys, dadj);
}

// blocks = max over instances of nframes * nqat
void launch_adjoint(hipStream_t st, int prec, int ns_max, long blocks, int B, const DevSys* dsys, const AdjDev* dadj) {
  if (blocks <= 0 || B <= 0) return;
  if (prec == QNB_PREC_MIXED) launch_adj_r<float>(st, ns_max, blocks, B, dsys, dadj);
  else launch_adj_r<double>(st, ns_max, blocks, B, dsys, dadj);
}

}  // namespace qnb
