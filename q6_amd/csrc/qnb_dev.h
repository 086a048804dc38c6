// qnb_dev.h -- device-side data layout and pair arithmetic of the MI355X
// nonbonded engine (gfx950, wave64).
//
// Layout in HBM (one record per system instance; topology arrays may be shared
// between instances of a batch, per-instance state is private):
//   x, d        natom x {x,y,z} float64 (reference qr_vec layout)
//   lrf         ncgp x 43 float64 (centre, phi0, phi1, phi2(3x3), phi3(9x3),
//               the reference's LRF_TYPE order)
//   nbr/nnbr    full neighbour lists in ELL form: row g holds every charge group
//               within the cut-off of group g (both directions of a pair),
//               nnbr[g] entries, row stride `cap`
//   epart       per-wave energy partials [slot][QNB_NE] reduced in fixed order
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qnb.h"

#define QNB_WAVE 64
#define QNB_NLRF 43
#define QNB_MAXST 8
#define QNB_MAXSH 8

// energy slots
enum {
  E_PP_EL = 0, E_PP_VDW, E_PW_EL, E_PW_VDW, E_WW_EL, E_WW_VDW, E_LRF, E_RAD, E_POL,
  E_Q0  // then per state s: qq_el, qq_vdw, qp_el, qp_vdw, qw_el, qw_vdw at E_Q0 + 6*s
};
#define QNB_NE (E_Q0 + 6 * QNB_MAXST)
// blocks per system of the energy reduction's first pass (k_reduce_part)
#define QNB_RED_BLOCKS 64

// a bond or angle as one of its atoms sees it: its role (place in the term),
// the other atoms in the term's order, and the parameters, so that an atom's
// terms are one load away from their partners' positions
struct alignas(8) BondRec {
  int role, other;
  double r0, k;
};
struct alignas(8) AngleRec {
  int role, o1, o2, pad;
  double t0, k;
};

struct DevSys {
  // sizes
  int natom, nat_solute, nwat, sa, ncgp, ncgp_solute, nqat, nstates, ntypes, ivdw_rule, spc;
  // 1: every solute-water LJ parameter of solvent atoms 1.. is zero (their
  // pw pairs reduce exactly to Coulomb)
  int pw_coul_h;
  int any_atom;  // iuse_switch_atom = 0: group cut-off tests take any atom pair
  int use_lrf, prec, quirk;
  double rcpp2, rcpw2, rcww2, rcq2, rclrf2, rexcl2;
  double lambda[QNB_MAXST];
  double el14;
  double xp[3], xw[3];
  // SCAAS
  double rwat, fk_wsphere, Dwmz, awmz, Boltz, fkwpol, itdis;
  int wpol, nshell;
  double sh_rout[QNB_MAXSH], sh_dr[QNB_MAXSH], sh_cstb[QNB_MAXSH];

  // topology (may be shared across a batch)
  const double* crg;
  const int* iac;
  const int* iqatom;
  const uint8_t* excl;
  const uint8_t* heavy;
  const int* gfirst;   // into cgpatom
  const int* glast;    // into cgpatom (inclusive)
  const int* gswitch;  // atom
  const int* cgpatom;
  const int* atom_group;
  // per group-ordered atom k (cgpatom order; groups are consecutive runs):
  // the bit of the atom's group (its index modulo 64) in the far-group ballot
  // word of the list sweep's 64-group chunk
  const uint64_t* gbit;
  int ncgpat;
  const int* cgentry;  // per group-ordered atom: its index, with AL_SKIP for a Q-atom (expand_row)
  const double* avdw;  // [t*3+k]
  const double* bvdw;
  const int* ljcod;    // [ti + tj*ntypes], 1-based code
  const uint32_t* exmask;  // [nat_solute] bit k-1: pair (i, i+k) excluded; bit 31: i has long partners
  const uint32_t* m14mask; // [nat_solute] bit k-1: pair (i, i+k) is 1-4
  const int* lx_off;       // [nat_solute+1] long exclusion/1-4 partners of the lower atom
  const int* lx_j;
  const uint8_t* lx_kind;  // 0 excluded, 1 1-4
  // solute-receiver fast path (k_sforces): a partner group b whose atom
  // indices lie more than 25 from every atom of the receiver group a, with
  // no long-range exclusion or 1-4 partner in either group, holds no
  // excluded or 1-4 pair with a; with the geometric rule and LJ code 1 for
  // every type pair, A, B and qq of such a pair are products of per-atom
  // factors
  const int* gspan;       // [ncgp_solute][2]: smallest and largest atom index of the group
  const uint8_t* glong;   // [ncgp_solute]: an atom of the group has long-range exclusion / 1-4 partners
  int ppfast;             // geometric rule and ljcod = 1 throughout
  const double* ppd;      // [nat_solute][PP_REC]: avdw(t, 1), bvdw(t, 1), charge, 0, avdw(t, 3), bvdw(t, 3), 0, 0 (FP64 path)
  const float* ppf;       // the same in FP32 (mixed path)
  const double* pwA;       // [i + j*nat_solute]
  const double* pwB;
  const double* pwEl;
  const float* pw_f;  // mixed path: [i][PW_REC] A, B, el of atom i with solvent sites 0..2 (FP32)
  const double* wwA;       // [la + ka*sa]
  const double* wwB;
  const double* wwEl;
  // pairs inside each solvent molecule (nonbond_solvent_internal): offsets
  // [n_sint][2] and A, B, charge product [n_sint][3]
  int n_sint;
  const int* sint_ij;
  const double* sint_par;
  const int* iqseq;
  const int* iq_of;  // [nat_solute] the atom's place in iqseq, -1 where it has none
  const uint8_t* qconn3;
  // per solute atom: the switch atom that decides whether its group is on the
  // Q-solute list, or -1 where no group test can put it there (within two
  // bonds of a Q-atom, in no group, excluded switch atom)
  const int* qp_test;
  const double* qpA;  // [i + nsol*(iq + nq*s)]
  const double* qpB;
  const double* qpEl;
  const double* qpSc;
  const float* qpA_f;  // FP32 copies of qpA, qpB, qpEl, qpSc for the mixed path
  const float* qpB_f;
  const float* qpEl_f;
  const float* qpSc_f;
  // the Q-solvent table packed for the force kernels, [iq][k][s] {A, B, el,
  // soft-core score}; FP64 path / mixed path
  const double* qw_d;
  const float* qw_f;
  const double* qwA;  // [iq + nq*(j + sa*s)]
  const double* qwB;
  const double* qwEl;
  const double* qwSc;
  // static Q-Q and Q-bonded-neighbour lists, all states concatenated
  const int* qq_iq;
  const int* qq_jq;
  const int* qq_st;
  const uint8_t* qq_soft;
  const double* qq_par;  // [p*4]: A, B, el, score
  int nqq;
  const int* qqp_iq;
  const int* qqp_j;
  const int* qqp_st;
  const double* qqp_par;
  int nqqp;
  // atom-centred view of the two lists (Q-atoms, then the distinct partners
  // of the Q-neighbour pairs): items {first atom, second atom, pair,
  // (state << 2) | (kind << 1) | side}
  const int* qe_atom;
  const int* qe_off;
  const int* qe_item;  // [4 * items]
  int nqe;
  const int* qe_of;    // [nat_solute] the atom's entity, -1 where it has none

  // per-instance state
  double* x;
  // LRF sources in cgpatom order, packed before each list update: x, y, z
  // and the charge (0 for Q-atoms, which take no part in the expansion);
  // FP32 for the mixed path, FP64 for the plain one (the other is null)
  float* xqg;
  double* xqgd;
  // [ncgp][4] per group, packed with them: its reference atom's position
  // (switch atom of a solute group, oxygen of a water) and 0 if that atom is
  // excluded, else 1
  double* gref;
  double* d;
  // gradient rows of the Q-atom side [nqat][3] and of the Q-Q entities
  // [nqe][3] where these run beside the solute receivers (QROWS_*), added to
  // d by the per-atom pass; dq is zero between steps, dqq stored anew
  double* dq;
  double* dqq;
  double* lrf;
  int* nbr;
  int* nnbr;
  // partner atoms of receivers 0 .. atom_rows - 1 (expand_row; a solvent other
  // than 3-site water has none, solvent_receiver walks its groups): rows of acap
  // slots; [ncgp][2] the slots in use and the groups they hold; slots per batch of
  // groups; slots a group takes where a row was too short (partner_row)
  int* alist;
  int* alist_end;
  int acap, al_batch, al_group, atom_rows;
  int* nnsol;  // [ncgp] length of the row's solute prefix (rows are sorted)
  // reference test-point reuse of the LRF-off switch-atom solute-water list
  // (quirk bit 0 with use_lrf = 0): per solute group, the first water within
  // the cut-off of the switch atom (nwat when none); later waters are tested
  // against atom glast + 1
  int* pw_first;
  int cap;
  int* need;        // [2] most groups of a row seen, and most slots of an atom row that did not fit
  uint8_t* qw_in;   // [nwat] water on the Q-water list
  uint8_t* qp_in;   // [ncgp_solute] group on the Q-solute list
  int* qw_list;     // compacted waters on the Q list
  int* qp_list;     // compacted solute atoms on the Q list
  int* nq_lists;    // [2]: n_qw, n_qp
  double* epart;    // [nslots][QNB_NE]
  int nslots;
  double* ered_part;  // [QNB_RED_BLOCKS][QNB_NE] partial sums of k_reduce_part
  double* ered;     // [QNB_NE]
  double* eatom;    // [natom][2]: per-atom LRF and radial-restraint energies
  // polarisation restraint state
  double* sh_state;  // [3*QNB_MAXSH]: theta_corr, avtheta, avn_insh
  int* sh_list;      // [QNB_MAXSH][nwat] members of each shell
  double* sh_lth;    // [QNB_MAXSH][nwat] their theta
  int* sh_n;         // [QNB_MAXSH] members per shell
  // atom-centred bonded terms of the MD path: for atom i, records
  // boff[i]..boff[i+1]-1 of brec and aoff[i]..aoff[i+1]-1 of arec; atoms
  // [0, nbat) carry all of them, with gradient rows brow (k_pol_bonded)
  const int* boff;
  const BondRec* brec;
  const int* aoff;
  const AngleRec* arec;
  double* brow;
  int nbat;
  double* wp_rank;   // [QNB_MAXSH][nwat][2] restraint energy and theta of each member, by rank
  // energy sampling: energies are accumulated when ene_every <= 0 or when
  // the instance's step counter is a multiple of ene_every
  const int* step_ptr;
  int ene_every;
};

// Q-atom bonded terms of one instance (qbond, qangle, qurey_bradley,
// qtorsion, qimproper, src/bondene.f90:387-685), resolved per state on the
// host.  Terms are numbered bonds, angles, torsions, impropers; each writes
// its gradient contributions into fixed slots (zeros where absent), and every
// atom the terms touch sums its slots in a fixed order.
struct QbDev {
  int nb, na, nt, ni, ns, urey;
  int nslot, nat;
  const int* atoms;     // term atoms: 2 per bond, 3 per angle, 4 per torsion / improper
  const double* par;    // [nterm][ns][4] the state's library row
  const uint8_t* pres;  // [nterm][ns] 1 = term present in the state
  const int* cpl;       // [na + nt + ni][4]: bond, flag, Urey-Bradley bond, flag (bond -1 = uncoupled)
  const int* slot0;     // [nterm] first slot of the term
  const int* coff;      // [nat + 1] slots of distinct atom a: cslot[coff[a] .. coff[a+1])
  const int* cslot;
  const int* catom;     // [nat] atom number
  double* morse;        // [nb][4] EMorseD, dMorse_i (x, y, z): kept between calls
  double* snap;         // [nb][ns][4] the same as evaluated in each state of this call
  double* eterm;        // [nterm][ns] energy of each term in each state
  double* slots;        // [ns][nslot][3] gradient shares of each state's terms
  double* e;            // [ns][4] bond, angle, torsion, improper of the last call
  double lambda[QNB_MAXST];
};

__device__ __forceinline__ bool want_energies(const DevSys& S) {
  return S.ene_every <= 0 || (*S.step_ptr % S.ene_every) == 0;
}

// ---------------------------------------------------------------- helpers

// load through the global address space: the DevSys arrays are reached
// through generic pointers, whose loads (flat) the compiler can neither
// separate from LDS traffic in its wait counts nor batch as freely
template <typename T>
__device__ __forceinline__ T ldg(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}
// a Q-solute table in the pair arithmetic's type: on the mixed path its FP32
// copy (the same values the FP64 table gives after rounding to float)
template <typename R>
__device__ __forceinline__ const R* qp_tab(const double* d, const float* f) {
  if constexpr (sizeof(R) == 4) return f;
  else return d;
}

template <typename T>
using gptr_t = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr_t<T> gp(const T* p) {
  return (gptr_t<T>)p;
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gpm(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}
// a value that is the same in every lane, in a scalar register: loop bounds
// and branches on it are the wave's and not each lane's
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename T>
__device__ __forceinline__ void stg(T* p, T v) {
  *(__attribute__((address_space(1))) T*)p = v;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, QNB_WAVE);
  return v;
}

// Sum over the wavefront without LDS instructions, for call sites where every
// lane is active: DPP moves within each row of 16 lanes (quad_perm xor 1 and
// xor 2, row_half_mirror, row_mirror), then the four row sums are read with
// v_readlane and added in a fixed order, so the result (the same in every
// lane) is deterministic.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum_all(double v) {
  v += dpp_move<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);  // row_half_mirror
  v += dpp_move<0x140>(v);  // row_mirror
  return ((lane_value(v, 0) + lane_value(v, 16)) + lane_value(v, 32)) + lane_value(v, 48);
}

// Sums N per-lane values over the wave at once ("transposed" reduction): a
// step pairs every lane with a partner and, while each lane still holds
// several values, the lane keeps half of them (the half its lane bit names)
// and adds the partner's copy of that half, so the number of values per
// lane halves each step.  Pairings: row_mirror (lane bit 3), row_half_mirror
// (bit 2), quad_perm xor 2 (bit 1), xor 1 (bit 0), then v_permlane16_swap
// (bit 4: rows 0<->1, 2<->3) and v_permlane32_swap (bit 5: halves); the
// mirrors come first because they also flip the lower bits, which must not
// yet decide anything.  Once a lane holds one value the remaining steps are
// plain butterflies.  Returns, in every lane, the full sum of value
// wave_sum_tr_index<N>(lane).  About 7 VALU per value (13% of N separate
// wave_sum_all reductions for N = 30).
__host__ __device__ constexpr int pow2_ceil(int n) { return n <= 1 ? 1 : 2 * pow2_ceil((n + 1) / 2); }
__host__ __device__ constexpr int log2_exact(int p) { return p <= 1 ? 0 : 1 + log2_exact(p / 2); }

template <int CTRL, int C>
__device__ __forceinline__ void tr_dpp_step(double* v, bool upper) {
  if constexpr (C >= 2) {
#pragma unroll
    for (int j = 0; j < C / 2; j++) {
      const double x = v[j], y = v[j + C / 2];
      const double send = upper ? x : y;  // the half the partner keeps
      const double keep = upper ? y : x;
      v[j] = keep + dpp_move<CTRL>(send);
    }
  } else {
    v[0] += dpp_move<CTRL>(v[0]);
  }
}

__device__ __forceinline__ void swap16(double& x, double& y) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(x), (unsigned)__double2loint(y), false,
                                                   false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y), false,
                                                   false);
  x = __hiloint2double((int)hi[0], (int)lo[0]);
  y = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ void swap32(double& x, double& y) {
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(x), (unsigned)__double2loint(y), false,
                                                   false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y), false,
                                                   false);
  x = __hiloint2double((int)hi[0], (int)lo[0]);
  y = __hiloint2double((int)hi[1], (int)lo[1]);
}

// rows (lane bit 4) or halves (bit 5): after the swap, x + y holds in every
// lane the pair's sum of the half that lane keeps
template <int C, bool HALVES>
__device__ __forceinline__ void tr_swap_step(double* v) {
  if constexpr (C >= 2) {
#pragma unroll
    for (int j = 0; j < C / 2; j++) {
      double x = v[j], y = v[j + C / 2];
      if constexpr (HALVES) swap32(x, y);
      else swap16(x, y);
      v[j] = x + y;
    }
  } else {
    double x = v[0], y = v[0];
    if constexpr (HALVES) swap32(x, y);
    else swap16(x, y);
    v[0] = x + y;
  }
}

template <int CTRL>
__device__ __forceinline__ float dpp_move_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// per-lane partials of type T (float or double); the first step exchanges
// them in T and adds in FP64 ((double)a + (double)b, exact conversions), so
// float partials are never summed in float and the wide FP64 copy of the N
// values is never live at once
template <typename T, int N>
__device__ __forceinline__ double wave_sum_tr(const T (&in)[N], int lane) {
  constexpr int P = pow2_ceil(N);
  static_assert(P <= 64, "at most 64 values");
  static_assert(QNB_NE <= 64, "one energy record per wave store");
  double v[P];
  const bool up = lane & 8;
  if constexpr (P >= 2) {
#pragma unroll
    for (int j = 0; j < P / 2; j++) {
      const T x = in[j], y = j + P / 2 < N ? in[j + P / 2] : T(0);
      const T send = up ? x : y;
      const T keep = up ? y : x;
      T got;
      if constexpr (sizeof(T) == 4) got = dpp_move_f<0x140>(send);
      else got = dpp_move<0x140>(send);
      v[j] = (double)keep + (double)got;
    }
  } else {
    T got;
    if constexpr (sizeof(T) == 4) got = dpp_move_f<0x140>(in[0]);
    else got = dpp_move<0x140>(in[0]);
    v[0] = (double)in[0] + (double)got;
  }
  tr_dpp_step<0x141, (P >= 2 ? P / 2 : 1)>(v, lane & 4);
  tr_dpp_step<0x4E, (P >= 4 ? P / 4 : 1)>(v, lane & 2);
  tr_dpp_step<0xB1, (P >= 8 ? P / 8 : 1)>(v, lane & 1);
  tr_swap_step<(P >= 16 ? P / 16 : 1), false>(v);
  tr_swap_step<(P >= 32 ? P / 32 : 1), true>(v);
  return v[0];
}

// the value whose sum lane `lane` holds after wave_sum_tr<N>, and whether
// the lane is that value's one writer (its bits that decided nothing are 0)
template <int N>
__device__ __forceinline__ int wave_sum_tr_index(int lane) {
  constexpr int L = log2_exact(pow2_ceil(N));
  const int bits[6] = {3, 2, 1, 0, 4, 5};
  int j = 0;
#pragma unroll
  for (int s = 0; s < L; s++) j = (j << 1) | ((lane >> bits[s]) & 1);
  return j;
}
template <int N>
__device__ __forceinline__ bool wave_sum_tr_writer(int lane) {
  constexpr int L = log2_exact(pow2_ceil(N));
  constexpr int bits[6] = {3, 2, 1, 0, 4, 5};
  int decided = 0;
#pragma unroll
  for (int s = 0; s < L; s++) decided |= 1 << bits[s];
  return (lane & ~decided) == 0 && wave_sum_tr_index<N>(lane) < N;
}

// the lane that holds value j after wave_sum_tr<N> and writes it
template <int N>
__host__ __device__ constexpr int wave_sum_tr_lane(int j) {
  constexpr int L = log2_exact(pow2_ceil(N));
  constexpr int bits[6] = {3, 2, 1, 0, 4, 5};
  int lane = 0;
  for (int s = 0; s < L; s++) lane |= ((j >> (L - 1 - s)) & 1) << bits[s];
  return lane;
}

// A wave's energy record ep[0 .. QNB_NE) in one coalesced store from lanes
// 0 .. QNB_NE-1: `sum` holds wave_sum_tr<N>'s sums of the N partials, each is
// read from its lane, and entry slot[j] takes sum j, every other entry 0.
template <int N>
__device__ __forceinline__ void store_energy_record(double* ep, double sum, const int (&slot)[N], int lane) {
  double v = 0.0;
#pragma unroll
  for (int j = 0; j < N; j++) {
    const double vj = lane_value(sum, wave_sum_tr_lane<N>(j));
    if (lane == slot[j]) v = vj;
  }
  if (lane < QNB_NE) *(__attribute__((address_space(1))) double*)(ep + lane) = v;
}
// energy records of the Q-Q pairs after the charge groups' ones: one when k_qq
// wrote them, one per four entities when k_forces_small did
__host__ __device__ __forceinline__ int qq_slots(const DevSys& S) { return S.nqe > 4 ? (S.nqe + 3) / 4 : 1; }
enum { QQ_ONE_RECORD = 1, QQ_RECORD_PER_BLOCK = 2 };

// shell members per block of the polarisation-restraint force kernel
#define WP_WATERS 64
// waves per block of that kernel in a small step
#define POL_SMALL_WAVES 16
__host__ __device__ __forceinline__ bool has_pol(const DevSys& S) { return S.nwat > 0 && S.wpol && S.nshell > 0; }
// restraint energy (c = 0) or theta (c = 1) of shell is, added over its n
// members by one wave (every lane active): lane l takes ranks l, l + 64, ...,
// then a fixed tree
__device__ __forceinline__ double watpol_sum(const DevSys& S, int is, int n, int c) {
  const auto p = gp(S.wp_rank + 2 * (size_t)is * S.nwat);
  double v = 0.0;
#pragma unroll 4
  for (int k = threadIdx.x % QNB_WAVE; k < n; k += QNB_WAVE) v += p[2 * (size_t)k + c];
  return wave_sum(v);
}

// Last phase of the polarisation restraint, `waves` waves of one block per
// system (wave `w` takes shells w, w + waves, ...): accumulates avtheta and
// avn_insh and clears the shell counts for the next step's angle kernel.
__device__ __forceinline__ void watpol_finish(const DevSys& S, int w, int waves) {
  if (!has_pol(S)) return;
  for (int is = w; is < S.nshell; is += waves) {
    const int n = ldg(S.sh_n + is);
    if (n == 0) continue;
    const double s = watpol_sum(S, is, n, 1);
    if (threadIdx.x % QNB_WAVE == 0) {
      S.sh_n[is] = 0;
      S.sh_state[QNB_MAXSH + is] += s / (double)n;
      S.sh_state[2 * QNB_MAXSH + is] += (double)n;
    }
  }
}

// Second pass of the energy reduction, one block of 256 threads: lane k of
// wave c adds energy k of every fourth partial from c on, wave 0 adds the four
// sums, the Q-Q record and the polarisation record, and writes ered.
__device__ __forceinline__ void reduce_final(const DevSys& S, int with_qq, int with_pol) {
  __shared__ double part[4][QNB_WAVE];
  const int k = threadIdx.x % QNB_WAVE, c = threadIdx.x / QNB_WAVE;
  double s = 0.0;
  if (k < QNB_NE) {
    const auto p = gp(S.ered_part);
#pragma unroll
    for (int g = 0; g < QNB_RED_BLOCKS / 4; g++) s += p[(size_t)(c + 4 * g) * QNB_NE + k];
  }
  part[c][k] = s;
  __shared__ double pol;
  if (c == 1 && with_pol && has_pol(S)) {
    double e = 0.0;
    for (int is = 0; is < S.nshell; is++) e += watpol_sum(S, is, ldg(S.sh_n + is), 0);
    if (k == 0) pol = e;
  }
  __syncthreads();
  if (c == 0 && k < QNB_NE) {
    double t = ((part[0][k] + part[1][k]) + part[2][k]) + part[3][k];
    if (with_qq && S.nqat > 0)
      for (int m = 0, nm = with_qq == QQ_ONE_RECORD ? 1 : qq_slots(S); m < nm; m++)
        t += ldg(S.epart + (size_t)(S.ncgp + m) * QNB_NE + k);
    if (k == E_POL && with_pol && has_pol(S)) t += pol;
    S.ered[k] = t;
  }
  __syncthreads();
}

// group contributions (calculate_exc): one pair of an energy array's list,
// kind 0 Q-Q (nbe_qq; soft: the exponential soft pair), 1 Q-solute (nbe_qx);
// i the Q-atom's index, j the partner's; the pair's A, B, el and soft-core
// score as the Q tables hold them
struct ExcEnt {
  int kind, i, j, soft;
  double A, B, el, sc;
};
// one system's arrays: off[a*ns + s] .. off[a*ns + s + 1] the pairs of array
// a in state s, type[a] (QNB_GC_*); hist: the batch's per-frame results
// [frame][narr][ns][QNB_GC_NV]
struct ExcDev {
  int narr, ns, max_frames;
  const int* off;
  const ExcEnt* ent;
  const int* type;
  double* hist;
};

// the walk of one (array, state): e[11] the state's energies (qq el, vdW, qp
// el, vdW, qw el, vdW, Q bond, angle, torsion, improper, restraint), o[7]
__device__ __forceinline__ void exc_walk(const ExcDev& D, const double* __restrict__ x, int a, int st,
                                         const double* e, double* o) {
#pragma clang fp contract(off)
  double qqel = e[0], qqvdw = e[1], qpel = e[2], qpvdw = e[3];
  const int ty = D.type[a];
  const int p0 = D.off[a * D.ns + st], p1 = D.off[a * D.ns + st + 1];
  for (int p = p0; p < p1; p++) {
    const ExcEnt& t = D.ent[p];
    const double ux = x[3 * t.j] - x[3 * t.i], uy = x[3 * t.j + 1] - x[3 * t.i + 1], uz = x[3 * t.j + 2] - x[3 * t.i + 2];
    const double r2 = 1.0 / (ux * ux + uy * uy + uz * uz), r = sqrt(r2), r6d = r2 * r2 * r2;
    const double r6_hc = 1.0 / r6d;
    double r6 = r6_hc + t.sc;
    r6 = 1.0 / r6;
    const double r12 = r6 * r6;
    const double Vel = t.el * r;
    double Va, Vb;
    if (t.soft) {  // nbe_qq's exponential soft pair (nonbonded.f90:138-141)
      Vb = 0.0;
      Va = t.A * exp(-t.B / r);
    } else {
      Va = t.A * r12;
      Vb = t.B * r6;
    }
    double* el = t.kind == 0 ? &qqel : &qpel;
    double* vdw = t.kind == 0 ? &qqvdw : &qpvdw;
    if (ty == QNB_GC_FULL) {
      *el = *el - Vel;
      *vdw = *vdw - (Va - Vb);
    } else if (ty == QNB_GC_ELECTRO) {
      *el = *el - Vel;
    } else {
      *vdw = *vdw - (Va - Vb);
    }
  }
  o[0] = qqel;
  o[1] = qqvdw;
  o[2] = qpel;
  o[3] = qpvdw;
  o[4] = qqel + qpel + e[4];
  o[5] = qqvdw + qpvdw + e[5];
  o[6] = e[6] + e[7] + e[8] + e[9] + o[4] + o[5] + e[10];
}

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// the LRF-off switch-atom solute-water list takes nbpwlist's test-point reuse
__host__ __device__ __forceinline__ bool pw_quirk(const DevSys& S) {
  return (S.quirk & 1) && !S.use_lrf && !S.any_atom && S.nwat > 0 && S.ncgp_solute > 0;
}

// q_dist4 (math.f90:254-262): |b - a|^2, ((dx^2 + dy^2) + dz^2), no contraction
__device__ __forceinline__ double dist4(const double* __restrict__ x, int a, int b) {
#pragma clang fp contract(off)
  double dx = ldg(x + 3 * b) - ldg(x + 3 * a);
  double dy = ldg(x + 3 * b + 1) - ldg(x + 3 * a + 1);
  double dz = ldg(x + 3 * b + 2) - ldg(x + 3 * a + 2);
  double r = dx * dx;
  r = r + dy * dy;
  r = r + dz * dz;
  return r;
}

__device__ __forceinline__ double dist4p(const double* __restrict__ x, int a, const double* p) {
#pragma clang fp contract(off)
  double dx = p[0] - x[3 * a];
  double dy = p[1] - x[3 * a + 1];
  double dz = p[2] - x[3 * a + 2];
  double r = dx * dx;
  r = r + dy * dy;
  r = r + dz * dz;
  return r;
}

// Adds an atom's per-atom terms to its gradient.  A solute atom in no charge
// group (an excluded atom of a topology cut to a sphere) is reached by no pair
// kernel, so this pass is the first writer of its gradient and stores it.
__device__ __forceinline__ void store_atom_gradient(const DevSys& S, int i, const double* f) {
  const auto d = gpm(S.d);
  if (i < S.nat_solute && ldg(S.atom_group + i) < 0) {
    d[3 * i] = f[0];
    d[3 * i + 1] = f[1];
    d[3 * i + 2] = f[2];
  } else {
    d[3 * i] += f[0];
    d[3 * i + 1] += f[1];
    d[3 * i + 2] += f[2];
  }
}

// which gradient rows of the Q kernels hold this step's sums
enum { QROWS_SIDE = 1, QROWS_QQ = 2 };
// adds atom i's rows to f; the Q-atom side's row is cleared for the next step
__device__ __forceinline__ void add_qrows(const DevSys& S, int i, int rows, double* f) {
  if (rows == 0 || i >= S.nat_solute || S.nqat <= 0) return;
  const int iq = (rows & QROWS_SIDE) ? ldg(S.iq_of + i) : -1;
  if (iq >= 0) {
    const auto q = gpm(S.dq) + 3 * iq;
    for (int c = 0; c < 3; c++) {
      f[c] += q[c];
      q[c] = 0.0;
    }
  }
  const int e = (rows & QROWS_QQ) ? ldg(S.qe_of + i) : -1;
  if (e >= 0)
    for (int c = 0; c < 3; c++) f[c] += ldg(S.dqq + 3 * e + c);
}

// harmonic bonds and angles of the solute (bond, angle: src/bondene.f90:41-246)
// One thread per atom sums the terms of every bond and angle it belongs to
// (each term is evaluated once per member atom), so the gradient needs no
// atomics and does not depend on scheduling.  A bond's energy is counted by
// its first atom, an angle's by its vertex; each block's energy sums go to
// bpart[block] and k_record adds them in block order.  bonded_atom is the
// per-atom part, used by k_bonded (the minimiser), k_atom_step (MD steps that
// record energies) and k_pol_bonded (the others).
// An atom has a few terms, each a chain of loads: BA_U records and then their
// partners' positions are requested together.
#define BA_U 2
__device__ __forceinline__ void bonded_atom(const DevSys& S, int i, double* f, double& eb, double& ea) {
  const auto x = gp(S.x);
  const int b0 = ldg(S.boff + i), b1 = ldg(S.boff + i + 1), a0 = ldg(S.aoff + i), a1 = ldg(S.aoff + i + 1);
  const double xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
  for (int it = b0; it < b1; it += BA_U) {
    BondRec r[BA_U];
    double xo[BA_U][3];
#pragma unroll
    for (int u = 0; u < BA_U; u++) {
      const auto p = gp(S.brec + min(it + u, b1 - 1));
      r[u] = BondRec{p->role, p->other, p->r0, p->k};
    }
#pragma unroll
    for (int u = 0; u < BA_U; u++)
      for (int c = 0; c < 3; c++) xo[u][c] = x[3 * r[u].other + c];
#pragma unroll
    for (int u = 0; u < BA_U; u++) {
      if (it + u >= b1) break;
      const bool first = r[u].role == 0;
      // from the bond's first atom to its second
      double v[3];
      for (int c = 0; c < 3; c++) v[c] = first ? xo[u][c] - xi[c] : xi[c] - xo[u][c];
      const double d = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
      const double db = d - r[u].r0;
      const double dv = r[u].k * db / d;
      const double sg = first ? -dv : dv;
      for (int c = 0; c < 3; c++) f[c] += v[c] * sg;
      if (first) eb += 0.5 * r[u].k * db * db;
    }
  }
  for (int it = a0; it < a1; it += BA_U) {
    AngleRec r[BA_U];
    double x1[BA_U][3], x2[BA_U][3];
#pragma unroll
    for (int u = 0; u < BA_U; u++) {
      const auto p = gp(S.arec + min(it + u, a1 - 1));
      r[u] = AngleRec{p->role, p->o1, p->o2, 0, p->t0, p->k};
    }
#pragma unroll
    for (int u = 0; u < BA_U; u++)
      for (int c = 0; c < 3; c++) {
        x1[u][c] = x[3 * r[u].o1 + c];
        x2[u][c] = x[3 * r[u].o2 + c];
      }
#pragma unroll
    for (int u = 0; u < BA_U; u++) {
      if (it + u >= a1) break;
      const int role = r[u].role;
      // the angle's atoms i, j (vertex), k
      double v[3], w[3];
      for (int c = 0; c < 3; c++) {
        const double pi = role == 0 ? xi[c] : x1[u][c];
        const double pj = role == 0 ? x1[u][c] : (role == 1 ? xi[c] : x2[u][c]);
        const double pk = role == 2 ? xi[c] : x2[u][c];
        v[c] = pi - pj;
        w[c] = pk - pj;
      }
      const double ru = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
      const double rw = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
      double ct = (v[0] * w[0] + v[1] * w[1] + v[2] * w[2]) / (ru * rw);
      ct = fmin(1.0, fmax(-1.0, ct));
      const double th = acos(ct);
      // sin(theta) from the cross product, consistent with the numerator of
      // the derivative below even for nearly linear angles, where
      // sin(acos(ct)) loses all digits; at a linear angle the derivative has
      // no direction
      const double cx = v[1] * w[2] - v[2] * w[1], cy = v[2] * w[0] - v[0] * w[2], cz = v[0] * w[1] - v[1] * w[0];
      const double st = sqrt(cx * cx + cy * cy + cz * cz) / (ru * rw);
      const double da = th - r[u].t0;
      if (role == 1) ea += 0.5 * r[u].k * da * da;
      if (!(st > 1.0e-8)) continue;
      const double dv = r[u].k * da;
      // dtheta/dx_i = -(w/(ru rw) - ct u/ru^2)/sin(theta), likewise for k; j balances
      for (int c = 0; c < 3; c++) {
        const double gi = -(w[c] / (ru * rw) - ct * v[c] / (ru * ru)) / st;
        const double gk = -(v[c] / (ru * rw) - ct * w[c] / (rw * rw)) / st;
        f[c] += dv * (role == 0 ? gi : (role == 2 ? gk : -(gi + gk)));
      }
    }
  }
}

// A charge group's LRF expansion, its symmetric tensors by their independent
// components (xx xy xz yy yz zz; xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz): 23
// of the 43 stored numbers, all requested at once.
struct LrfGroup {
  double c[3], phi0, p1[3], p2[6], p3[10];
};
__device__ __forceinline__ void lrf_load(const DevSys& S, int group, LrfGroup& g) {
  const auto L = gp(S.lrf + (size_t)QNB_NLRF * group);
  for (int k = 0; k < 3; k++) g.c[k] = L[k], g.p1[k] = L[4 + k];
  g.phi0 = L[3];
  constexpr int i2[6] = {0, 1, 2, 4, 5, 8};
  constexpr int i3[10] = {0, 1, 2, 4, 5, 8, 13, 14, 17, 26};
#pragma unroll
  for (int k = 0; k < 6; k++) g.p2[k] = L[7 + i2[k]];
#pragma unroll
  for (int k = 0; k < 10; k++) g.p3[k] = L[16 + i3[k]];
}
// LRF Taylor application for one atom at x (lrf_taylor, nonbondene.f90:507-571)
__device__ __forceinline__ void lrf_taylor(const LrfGroup& g, double x, double y, double z, double q, double* f,
                                           double& e) {
  const double d[3] = {g.c[0] - x, g.c[1] - y, g.c[2] - z};
  constexpr int s2[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
  constexpr int s3[3][3][3] = {{{0, 1, 2}, {1, 3, 4}, {2, 4, 5}},
                               {{1, 3, 4}, {3, 6, 7}, {4, 7, 8}},
                               {{2, 4, 5}, {4, 7, 8}, {5, 8, 9}}};
  double t[3], df[3];
#pragma unroll
  for (int k = 0; k < 3; k++) t[k] = d[0] * g.p2[s2[k][0]] + d[1] * g.p2[s2[k][1]] + d[2] * g.p2[s2[k][2]];
  const double V = g.phi0 + (d[0] * g.p1[0] + d[1] * g.p1[1] + d[2] * g.p1[2]) +
                   0.5 * (d[0] * t[0] + d[1] * t[1] + d[2] * t[2]);
  e += 0.5 * q * V;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double u[3];
#pragma unroll
    for (int j = 0; j < 3; j++)
      u[j] = d[0] * g.p3[s3[k][j][0]] + d[1] * g.p3[s3[k][j][1]] + d[2] * g.p3[s3[k][j][2]];
    df[k] = g.p1[k] + t[k] + 0.5 * (d[0] * u[0] + d[1] * u[1] + d[2] * u[2]);
    f[k] -= df[k] * q;
  }
}
__device__ __forceinline__ void lrf_taylor_atom(const DevSys& S, int i, int group, double* f, double& e) {
  LrfGroup g;
  lrf_load(S, group, g);
  const auto x = gp(S.x);
  lrf_taylor(g, x[3 * i], x[3 * i + 1], x[3 * i + 2], ldg(S.crg + i), f, e);
}

// SCAAS radial restraint on one water oxygen (restrain_solvent,
// nonbondene.f90:6466-6544, 3-site branch)
__device__ __forceinline__ void radial_restraint(const DevSys& S, double x, double y, double z, double shift, double* f,
                                                 double& e) {
  double vx = x - S.xw[0], vy = y - S.xw[1], vz = z - S.xw[2];
  double b = sqrt(vx * vx + vy * vy + vz * vz);
  double db = b - (S.rwat - shift);
  double erst, dv;
  if (db > 0.0) {
    erst = 0.5 * S.fk_wsphere * (db * db) - S.Dwmz;
    dv = S.fk_wsphere * db / b;
  } else if (b > 0.0) {
    double fexp = exp(S.awmz * db);
    erst = S.Dwmz * (fexp * fexp - 2.0 * fexp);
    dv = -2.0 * S.Dwmz * S.awmz * (fexp - fexp * fexp) / b;
  } else {
    erst = 0.0;
    dv = 0.0;
  }
  f[0] += vx * dv;
  f[1] += vy * dv;
  f[2] += vz * dv;
  e += erst;
}

__device__ __forceinline__ void radial_restraint(const DevSys& S, int src, double shift, double* f, double& e) {
  const auto x = gp(S.x);
  radial_restraint(S, x[3 * src], x[3 * src + 1], x[3 * src + 2], shift, f, e);
}

// The atom whose distance from xwcent drives atom i's SCAAS radial term
// (restrain_solvent, nonbondene.f90:6466-6544), or -1: a 3-site water's first
// atom acts on itself; in other solvents every heavy atom (by the first
// molecule's pattern, is_heavy_solv) of a non-excluded molecule takes the
// term at the distance of the molecule's first atom, as the reference
// measures it.
__device__ __forceinline__ int radial_source(const DevSys& S, int i) {
  const int w = i - S.nat_solute;
  if (w < 0) return -1;
  const int isolv = w % S.sa, first = i - isolv;
  if (ldg(S.excl + first)) return -1;
  if (S.sa == 3) return isolv == 0 ? i : -1;
  return ldg(S.heavy + S.nat_solute + isolv) ? first : -1;
}

// Q-solute group test (nbqplist, nonbondene.f90:3647-3742): the group's
// switch atom within Rcq of xpcent; with any_atom (nbqplis2 :3408-3500) any
// atom of the group, scanned in group order
__device__ __forceinline__ bool qp_group_in(const DevSys& S, const double* __restrict__ x, int g) {
  const int sw = S.gswitch[g];
  if (S.excl[sw]) return false;
  if (!S.any_atom) return dist4p(x, sw, S.xp) <= S.rcq2;
  for (int k = S.gfirst[g]; k <= S.glast[g]; k++)
    if (dist4p(x, S.cgpatom[k], S.xp) <= S.rcq2) return true;
  return false;
}

// 1/|u|^2 and 1/|u| from |u|^2.  FP32: the hardware reciprocal square root
// (v_rsq_f32, 1 ulp), the usual pair-kernel form.  FP64: the hardware's
// reciprocal root (about 26 bits) with one third-order step,
// y (1 + e/2 + 3 e^2/8) with e = 1 - d2 y^2, and 1/d2 from its square with one
// Newton step: 15 slots and no branch, a division and a root took about 32.
// At the limits (d2 = 0: y infinite; d2 = inf: y = 0) both steps' residuals are
// 0 inf = NaN, and v_min_f64 takes its other operand then: 1, with which each
// step leaves its limit as it is (a residual proper is about 0, and a NaN d2
// still gives NaN through y).  That is 2 slots; the LRF sweep, whose
// q/r^3 r^2 is NaN at both limits in any case, does without (rinv_inner).
template <bool LIMITS>
__device__ __forceinline__ void rinv_steps(double d2, double& r2, double& r) {
  const double y = __builtin_amdgcn_rsq(d2);
  double e = __builtin_fma(-d2 * y, y, 1.0);
  if (LIMITS) e = __builtin_fmin(e, 1.0);
  r = __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
  const double s = r * r;
  double f = __builtin_fma(-d2, s, 1.0);
  if (LIMITS) f = __builtin_fmin(f, 1.0);
  r2 = __builtin_fma(s, f, s);
}
__device__ __forceinline__ void rinv_inner(double d2, double& r2, double& r) { rinv_steps<false>(d2, r2, r); }
__device__ __forceinline__ void rinv(double d2, double& r2, double& r) { rinv_steps<true>(d2, r2, r); }
__device__ __forceinline__ void rinv_inner(float d2, float& r2, float& r) {
  r = __builtin_amdgcn_rsqf(d2);
  r2 = r * r;
}
__device__ __forceinline__ void rinv(float d2, float& r2, float& r) {
  r = __builtin_amdgcn_rsqf(d2);
  r2 = r * r;
}
// |u|^2; in FP32 with the multiply-adds written out, so that its rounding does
// not depend on which of them the compiler would fuse at a call site
__device__ __forceinline__ double norm2(double x, double y, double z) { return x * x + y * y + z * z; }
__device__ __forceinline__ float norm2(float x, float y, float z) {
  return __builtin_fmaf(z, z, __builtin_fmaf(x, x, y * y));
}
// 1/v: IEEE in FP64, hardware reciprocal (v_rcp_f32, 1 ulp) in FP32
__device__ __forceinline__ double recip(double v) { return 1.0 / v; }
__device__ __forceinline__ float recip(float v) { return __builtin_amdgcn_rcpf(v); }

// Pair arithmetic in precision R (double: plain path; float: mixed path).
// u = x_j - x_i arrives in FP64 (the difference of FP64 positions), is rounded
// to R, and the returned scalar dv is in R; callers accumulate u*dv in FP64.
template <typename R>
struct PairMath {
  // nbe (nonbonded.f90:45-75): LJ + Coulomb.  Adds V_el, V_a - V_b to the
  // accumulators (type T: FP64, or R for a short per-partner partial).
  // `want`: accumulate the energies (only the sampled steps need them)
  template <typename T>
  static __device__ __forceinline__ R nbe(R ux, R uy, R uz, R A, R B, R q, T& el, T& vdw, bool want = true) {
    R r2, r;
    rinv(norm2(ux, uy, uz), r2, r);
    R r6 = r2 * r2 * r2;
    R r12 = r6 * r6;
    R Vel = q * r, Va = A * r12, Vb = B * r6;
    if (want) {
      el += (T)Vel;
      vdw += (T)Va - (T)Vb;
    }
    return r2 * (-Vel - R(12) * Va + R(6) * Vb);
  }
  // nbe_spc (nonbonded.f90:247-267): Coulomb only
  template <typename T>
  static __device__ __forceinline__ R nbe_spc(R ux, R uy, R uz, R q, T& el, bool want = true) {
    R r2, r;
    rinv(norm2(ux, uy, uz), r2, r);
    R Vel = q * r;
    if (want) el += (T)Vel;
    return -r2 * Vel;
  }
  // nbe_qx (nonbonded.f90:200-222), soft-core score sc, state weight lam
  static __device__ __forceinline__ R nbe_qx(R r2, R r, R r6in, R A, R B, R q, R sc, R lam, double& el,
                                             double& vdw, bool want = true) {
    R r6_hc = R(1), r6 = r6in;
    // FP64: without a soft core 1/(1/r6) and r6/r6 are r6 and 1; FP32 keeps the
    // rounding of the two reciprocals
    if (sizeof(R) == 4 || sc != R(0)) {
      r6_hc = recip(r6in);
      r6 = recip(r6_hc + sc);
    }
    R r12 = r6 * r6;
    R Vel = q * r, Va = A * r12, Vb = B * r6;
    if (want) {
      el += (double)Vel;
      vdw += (double)Va - (double)Vb;
    }
    if (sizeof(R) == 8 && sc == R(0)) return r2 * (-Vel - (R(12) * Va - R(6) * Vb)) * lam;
    return r2 * (-Vel - (R(12) * Va - R(6) * Vb) * r6 * r6_hc) * lam;
  }
};

// floats per solute atom in the FP32 solute-water table (3 sites x A, B, el,
// padded to 16-byte records)
#define PW_REC 12
// values per solute atom in the solute-solute factor tables (ppd, ppf)
#define PP_REC 8

// partners per wave of the Q-atom force kernel (the Q-atom's partners are
// split into chunks of about this many)
#ifndef QF_PART
#define QF_PART 512
#endif
// grid.x of the Q-atom force kernel: per XCD (8) and per Q-atom group of 8,
// the blocks of one Q-atom's chunks (W waves per block)
inline int qforces_blocks(int nq, int chunks, int W) { return 8 * ((chunks + W - 1) / W) * ((nq + 7) / 8); }

// the same inside k_forces_small: more, shorter waves (as launches of their own
// the Q-atom side took 11-13 us at 8 partners per lane)
#define QF_PART_SMALL 192

// blocks of each role of k_forces_small, and the chunks of a Q-atom's partners
struct SmallGrid {
  int solute, solvent, qside, qq, theta, qchunks;
  int blocks() const { return solute + solvent + qside + qq + theta; }
};

// threads of the Q-Q kernel's block (one block per system)
#define QQ_THREADS 1024
// polarisation restraint: threads per block of the angle kernel (one per
// water); shell members staged in LDS at a time by the force kernel
#define WP_THREADS 256
#define WP_CHUNK 1024

// at most FC_WPB wavefronts per block of the solvent-receiver kernels
#define FC_WPB 8
// largest charge group (atoms)
#ifndef FC_CAP
#define FC_CAP 384
#endif
// partner-atom entries (DevSys::alist): atom index and flags; slots per batch
// of groups where every solute group fits in them, else FC_CAP
enum : int { AL_ATOM = (1 << 28) - 1, AL_OWN = 1 << 28, AL_FAR = 1 << 29, AL_SKIP = 1 << 30 };
#define AL_BATCH 128
// Solute receivers (solute_receiver): atoms per sweep, whose values (an index and
// 6 of R each) are the same in every lane, and per-wave LDS
template <typename R>
__host__ __device__ constexpr int so_ch() { return sizeof(R) == 4 ? 10 : 5; }
template <typename R>
__host__ __device__ constexpr size_t so_wave_bytes() {
  return (so_ch<R>() * (5 * sizeof(double) + 12 * sizeof(R) + 4 * sizeof(int)) + 15) / 16 * 16;
}

// Placement of a batch's blocks on the XCDs.  Blocks are dealt to the 8 XCDs
// round-robin in linear block order.  imap 0: grid (nb, ninst), block x of
// every instance on the same XCD (instances share the topology's rows in
// L2).  imap 1: a 1-D grid of 8 * ceil(nb * ninst / 8) blocks whose k-th
// block on XCD x takes work item x * per + k of the instance-major order, so
// each instance's blocks run on one or two XCDs and its coordinates stay in
// their L2.  Returns false for padding blocks.
__device__ __forceinline__ bool map_block(int imap, int nb, int ninst, int& inst, int& blk) {
  if (imap == 0) {
    inst = blockIdx.y;
    blk = blockIdx.x;
    return blk < nb;
  }
  const long total = (long)nb * ninst, per = (total + 7) / 8, L = blockIdx.x;
  const long g = (L % 8) * per + L / 8;
  if (g >= total) return false;
  inst = (int)(g / nb);
  blk = (int)(g % nb);
  return true;
}

// Adjoint of the per-state Q-atom energies over a set of frames: tangent
// tables (derivative of each Q table entry with respect to the Q-side
// parameter of that entry) and the per-frame output.
#define QNB_ADJ_NV 7
enum { ADJ_DQ = 0, ADJ_DA, ADJ_DB, ADJ_DA14, ADJ_DB14, ADJ_EEL, ADJ_EVDW };

struct AdjDev {
  const double* frames;  // [nframes][natom*3]
  int nframes;
  const double* qp_dq;   // layout of qpA: [j + nsol*(iq + nq*s)]
  const double* qp_dA;
  const double* qp_dB;
  const uint8_t* qp_is14;
  const double* qw_dq;   // layout of qwA: [iq + nq*(k + sa*s)]
  const double* qw_dA;
  const double* qw_dB;
  const double* qq_dq_i;  // layout of the qq tables: [iq + nq*(jq + nq*s)]
  const double* qq_dA_i;
  const double* qq_dB_i;
  const double* qq_dq_j;
  const double* qq_dA_j;
  const double* qq_dB_j;
  const uint8_t* qq_is14;
  double* out;  // [nframes][nstates][nqat][QNB_ADJ_NV]
};
