// qnb_kernels.hip -- HIP kernels of the nonbonded engine for gfx950.
//
// Work decomposition is receiver-centric: one wavefront owns one charge group
// (a solute group or a water) and computes every interaction of its atoms with
// all partners, so pair forces need no atomics and the result does not depend
// on scheduling.  Each unordered pair is evaluated from both sides; its energy
// is counted once, on the side that owns the pair under the reference's parity
// rule (nonbondene.f90:1589-1591), which also decides which side's list the
// pair is exported in.  Q-atoms, whose partners are all waters and solute
// atoms within Rcq, are the one many-to-one case: their forces are summed per
// wavefront and added with one atomic per wave and component.
#include "qnb_host.h"

namespace qnb {

__device__ __forceinline__ int group_ref_atom(const DevSys& S, int g) {
  return g < S.ncgp_solute ? ldg(S.gswitch + g) : S.nat_solute + S.sa * (g - S.ncgp_solute);
}

// Group test of the iuse_switch_atom = 0 builders for a pair with a solute
// group: true when any atom pair (solute-solute, nbpplis2(_lrf)
// nonbondene.f90:950-1089, 1369-1488) or any solute atom and the water's
// first atom (nbpwlis2(_lrf) :2137-2230, 2493-2620) lies within cut2;
// otherwise r2 is the squared distance of the last pair the reference scans
// (the groups' last atoms; symmetric, so either group may be the receiver),
// which its _lrf forms compare with RcLRF^2
__device__ __forceinline__ bool any_atom_pair(const DevSys& S, const double* __restrict__ x, int a, int b, bool a_sol,
                                            bool b_sol, int ra, int rb, double cut2, double& r2) {
  r2 = 1.0;
  if (a_sol && b_sol) {
    const int a1 = ldg(S.glast + a), b0 = ldg(S.gfirst + b), b1 = ldg(S.glast + b);
    for (int ia = ldg(S.gfirst + a); ia <= a1; ia++) {
      const int i = ldg(S.cgpatom + ia);
      for (int jb = b0; jb <= b1; jb++) {
        r2 = dist4(x, i, ldg(S.cgpatom + jb));
        if (r2 <= cut2) return true;
      }
    }
    return false;
  }
  const int g = a_sol ? a : b, w = a_sol ? rb : ra;
  const int g1 = ldg(S.glast + g);
  for (int k = ldg(S.gfirst + g); k <= g1; k++) {
    r2 = dist4(x, ldg(S.cgpatom + k), w);
    if (r2 <= cut2) return true;
  }
  return false;
}

// First water (index order) within the cut-off of each solute group's switch
// atom, for the LRF-off switch-atom solute-water list: nbpwlist
// (nonbondene.f90:2665-2691) reuses its switch-atom variable `ia` as the loop
// index over the group's atoms, so once a water is inside, the distance test
// of every later water is made from atom cgp(ig)%last + 1.  One wavefront per
// solute group; excluded groups and waters are skipped as the reference does.
__global__ __launch_bounds__(256) void k_pw_first(const DevSys* __restrict__ systems) {
  const DevSys& S = systems[blockIdx.y];
  const int g = blockIdx.x * (blockDim.x / QNB_WAVE) + threadIdx.x / QNB_WAVE;
  if (g >= S.ncgp_solute || !pw_quirk(S)) return;
  const int lane = threadIdx.x % QNB_WAVE;
  const int ia = ldg(S.gswitch + g);
  int first = S.nwat;
  if (!ldg(S.excl + ia)) {
    for (int w0 = 0; w0 < S.nwat; w0 += QNB_WAVE) {
      const int w = w0 + lane;
      bool in = false;
      if (w < S.nwat) {
        const int ja = S.nat_solute + S.sa * w;
        in = !ldg(S.excl + ja) && dist4(S.x, ia, ja) <= S.rcpw2;
      }
      const uint64_t m = __ballot(in);
      if (m) {
        first = w0 + __ffsll((long long)m) - 1;
        break;
      }
    }
  }
  if (lane == 0) S.pw_first[g] = first;
}

// the owner side of a charge-group pair (a != b) under the parity rule
__device__ __forceinline__ bool owns(int a, int b) {
  return (a < b && ((a + b) & 1) == 0) || (a > b && ((a + b) & 1) == 1);
}

// ---------------------------------------------------------------------------
// LRF expansion (lrf_update, nonbondene.f90:628-725), restated on raw sums that
// need no per-atom constant or subtraction:
//   p[0] = sum q/r,  p[1..3] = sum f0 d_a,  p[4..9] = sum w1 d_a d_b,
//   p[10..19] = sum w2 d_a d_b d_c
// with d = x_i - centre, f0 = q/r^3, w1 = f0/r^2, w2 = w1/r^2; components xx xy
// xz yy yz zz, then xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz.  lrf_update's
// field1 = 3 f0/r^2 and its 5 field2 d d d term (field2 = -field1/r^2) give
// phi2_ab = 3 p_ab - delta_ab sum f0 and phi3_abc = -15 p_abc +
// 3 (delta_ab H_c + delta_ac H_b + delta_bc H_a), H_a = sum w1 d_a; as
// w1 r^2 = f0 and w2 r^2 = w1, sum f0 is the trace of p[4..9] and H_a the trace
// of p[10..19] over the other two indices: lrf_tensors, once per receiver.
#define LRF_NF 20
typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));
template <typename R>
__device__ __forceinline__ void lrf_accumulate(R* p, R dx, R dy, R dz, R q) {
  R ri2, ri;
  rinv_inner(norm2(dx, dy, dz), ri2, ri);
  const R qri = q * ri;
  p[0] += qri;
  const R f0 = qri * ri2;
  const R w1 = f0 * ri2;
  const R w2 = w1 * ri2;
  p[1] += dx * f0;
  p[2] += dy * f0;
  p[3] += dz * f0;
  const R xx = dx * dx, xy = dx * dy, xz = dx * dz, yy = dy * dy, yz = dy * dz, zz = dz * dz;
  p[4] += xx * w1;
  p[5] += xy * w1;
  p[6] += xz * w1;
  p[7] += yy * w1;
  p[8] += yz * w1;
  p[9] += zz * w1;
  const R gx = w2 * dx, gy = w2 * dy, gz = w2 * dz;
  p[10] += gx * xx;
  p[11] += gx * xy;
  p[12] += gx * xz;
  p[13] += gx * yy;
  p[14] += gx * yz;
  p[15] += gx * zz;
  p[16] += gy * yy;
  p[17] += gy * yz;
  p[18] += gy * zz;
  p[19] += gz * zz;
}

// raw sums -> phi0, phi1[3], phi2[6], phi3[10] (lrf_update's tensors)
__device__ __forceinline__ void lrf_tensors(double* acc, const double* q) {
  const double s0 = q[4] + q[7] + q[9];
  const double hx = q[10] + q[13] + q[15], hy = q[11] + q[16] + q[18], hz = q[12] + q[17] + q[19];
  acc[0] = q[0];
  acc[1] = -q[1];
  acc[2] = -q[2];
  acc[3] = -q[3];
  acc[4] = 3.0 * q[4] - s0;
  acc[5] = 3.0 * q[5];
  acc[6] = 3.0 * q[6];
  acc[7] = 3.0 * q[7] - s0;
  acc[8] = 3.0 * q[8];
  acc[9] = 3.0 * q[9] - s0;
  acc[10] = 9.0 * hx - 15.0 * q[10];
  acc[11] = 3.0 * hy - 15.0 * q[11];
  acc[12] = 3.0 * hz - 15.0 * q[12];
  acc[13] = 3.0 * hx - 15.0 * q[13];
  acc[14] = -15.0 * q[14];
  acc[15] = 3.0 * hx - 15.0 * q[15];
  acc[16] = 9.0 * hy - 15.0 * q[16];
  acc[17] = 3.0 * hz - 15.0 * q[17];
  acc[18] = 3.0 * hy - 15.0 * q[18];
  acc[19] = 9.0 * hz - 15.0 * q[19];
}

// Raw buffer loads (32-bit byte offsets from a base in scalar registers; an
// offset at or past `bytes` reads 0): the sweep's packed arrays are indexed
// without 64-bit address arithmetic or clamping.
typedef unsigned int u4v __attribute__((vector_size(16)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ f4v buf_f4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ d4v buf_d4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const d2v lo = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  const d2v hi = __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, 0, 0));
  return d4v{lo.x, lo.y, hi.x, hi.y};
}
typedef unsigned int u2v __attribute__((vector_size(8)));
__device__ __forceinline__ u2v buf_u2(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u2v, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
// through the scalar cache: a table that no kernel writes, at an index that is
// the same in every lane
__device__ __forceinline__ int ldc(const int* p) {
  return *(const __attribute__((address_space(4))) int*)(uintptr_t)p;
}

// Packs the LRF sources before a list update, one record per atom in
// cgpatom order (a charge group's atoms are one run): x, y, z and the charge,
// 0 for Q-atoms (lrf_update skips them); FP32 for the mixed path (each
// coordinate rounded once), FP64 for the plain one.  Also packs each group's
// reference atom for the group tests of the sweep, with 0 if it is excluded.
__global__ __launch_bounds__(256) void k_pack_xq(const DevSys* __restrict__ systems) {
  const DevSys& S = systems[blockIdx.y];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= S.ncgpat) return;
  const int i = ldg(S.cgpatom + k);
  const auto x = gp(S.x);
  const double q = ldg(S.iqatom + i) != 0 ? 0.0 : ldg(S.crg + i);
  if (S.xqg) {
    const auto o = gpm(S.xqg);
    o[4 * k] = (float)x[3 * i];
    o[4 * k + 1] = (float)x[3 * i + 1];
    o[4 * k + 2] = (float)x[3 * i + 2];
    o[4 * k + 3] = (float)q;
  }
  if (S.xqgd) {
    const auto o = gpm(S.xqgd);
    o[4 * k] = x[3 * i];
    o[4 * k + 1] = x[3 * i + 1];
    o[4 * k + 2] = x[3 * i + 2];
    o[4 * k + 3] = q;
  }
  if (k < S.ncgp) {  // thread k also packs group k's reference atom
    const int rb = group_ref_atom(S, k);
    const auto o = gpm(S.gref);
    o[4 * k] = x[3 * rb];
    o[4 * k + 1] = x[3 * rb + 1];
    o[4 * k + 2] = x[3 * rb + 2];
    o[4 * k + 3] = ldg(S.excl + rb) ? 0.0 : 1.0;
  }
}

// index of the symmetric third-rank component (a<=b<=c sorted) in acc[10..]
__device__ __forceinline__ int t3index(int a, int b, int c) {
  // sort three indices
  if (a > b) { int t = a; a = b; b = t; }
  if (b > c) { int t = b; b = c; c = t; }
  if (a > b) { int t = a; a = b; b = t; }
  // lexicographic rank among (000 001 002 011 012 022 111 112 122 222)
  const int base[3] = {0, 6, 9};
  if (a == 0) {
    const int r0[3][3] = {{0, 1, 2}, {0, 3, 4}, {0, 0, 5}};
    return 10 + r0[b][c];
  }
  if (a == 1) return 10 + (b == 1 ? (c == 1 ? 6 : 7) : 8);
  (void)base;
  return 19;
}

// one packed LRF source record: FP32 on the mixed path, FP64 on the plain one
template <typename R>
__device__ __forceinline__ auto lrf_rec(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(R) == 4) return buf_f4(r, off);
  else return buf_d4(r, off);
}

// dist4 on packed reference positions: |b - a|^2, ((dx^2 + dy^2) + dz^2)
__device__ __forceinline__ double dist4v(const d4v& a, const d4v& b) {
#pragma clang fp contract(off)
  const double dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
  double r = dx * dx;
  r = r + dy * dy;
  r = r + dz * dz;
  return r;
}

// ---------------------------------------------------------------------------
// Partner atoms of receiver group a, written by its wave at the end of a list
// update (nsr: the solute groups of its row) and read by the force kernels of
// every step until the next one: the solute groups of the row's prefix as
// atoms.  Lane = partner group; the groups are taken in batches of up to 64 whose atoms fit
// in `batch` slots (al_batch) and every batch ends at a multiple of 64 slots,
// so lane l of the force kernels, taking slots l, l + 64, ..., always adds the
// same partners in the same order.  An entry is the atom's index with AL_OWN
// (the receiver owns the energy of the two groups' pairs) and AL_FAR (a solute
// receiver and a group that can hold no excluded or 1-4 pair with it: every
// index more than 25 from the receiver's, no long-range partners in either);
// AL_SKIP marks Q-atoms (their pairs belong to the Q kernels) and the padding.
// The force kernels then read one coalesced list per receiver instead of
// walking group -> atoms -> positions through LDS at every step.  A launch of
// its own cost a list update 7 us.  A row longer than acap slots ends before
// the batch that does not fit (alist_end: slots and groups stored) and its length
// goes to need[1], as a neighbour row's does to need[0]; the force kernels take
// the groups after it from the neighbour row (row_tail).  With acap 0 the call
// only counts.
#define LS_WPB 8  // waves per block of the list sweep at most
__device__ __forceinline__ void expand_row(const DevSys& S, int a, int nsr, int lane, int w) {
  const int batch = S.al_batch;
  const bool a_sol = a < S.ncgp_solute;
  const int* row = S.nbr + (size_t)a * S.cap;
  const int acap = S.acap;
  int* out = S.alist + (size_t)a * acap;
  const bool along = a_sol && ldg(S.glong + a);
  const int alo = a_sol ? ldg(S.gspan + 2 * a) : 0, ahi = a_sol ? ldg(S.gspan + 2 * a + 1) : 0;
  __shared__ int s_incl[LS_WPB][QNB_WAVE], s_src[LS_WPB][QNB_WAVE], s_tag[LS_WPB][QNB_WAVE];
  int n = 0, stored = 0, groups = 0;
  for (int p0 = 0, ng = 0; p0 < nsr; p0 += ng) {
    const int p = p0 + lane;
    int f0 = 0, cnt = 0, tag = 0;
    if (p < nsr) {
      const int b = ldg(row + p);
      f0 = ldg(S.gfirst + b);
      cnt = ldg(S.glast + b) - f0 + 1;
      const bool blong = ldg(S.glong + b);
      const int blo = ldg(S.gspan + 2 * b), bhi = ldg(S.gspan + 2 * b + 1);
      tag = owns(a, b) ? AL_OWN : 0;
      if (a_sol && !along && !blong && (blo - ahi > 25 || alo - bhi > 25)) tag |= AL_FAR;
    }
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < QNB_WAVE; o <<= 1) {
      const int u = __shfl_up(incl, o, QNB_WAVE);
      if (lane >= o) incl += u;
    }
    // inclusive sums never decrease, so the groups that fit are a prefix (a
    // group always fits)
    ng = min(__popcll(__ballot(incl <= batch)), nsr - p0);
    const int total = __shfl(incl, ng - 1, QNB_WAVE);
    const int end = uni((total + QNB_WAVE - 1) / QNB_WAVE * QNB_WAVE);
    n += end;
    if (n > acap) continue;
    // lane = slot: its group is the first whose inclusive count passes it
    s_incl[w][lane] = incl;
    s_src[w][lane] = f0 - (incl - cnt);
    s_tag[w][lane] = tag;
    __builtin_amdgcn_wave_barrier();
    for (int s = lane; s < end; s += QNB_WAVE) {
      int e = AL_SKIP;
      if (s < total) {
        int g = 0;
#pragma unroll
        for (int h = 32; h > 0; h >>= 1)
          if (s_incl[w][g + h - 1] <= s) g += h;
        e = ldg(S.cgentry + s_src[w][g] + s) | s_tag[w][g];
      }
      stg(out + stored + s, e);
    }
    __builtin_amdgcn_wave_barrier();
    stored = n;
    groups = p0 + ng;
  }
  if (lane == 0) {
    S.alist_end[2 * a] = stored;
    S.alist_end[2 * a + 1] = groups;
    if (n > acap) atomicMax(S.need + 1, n);
  }
}

// ---------------------------------------------------------------------------
// Pair-list update with LRF (make_pair_lists, nonbondene.f90:749-837, SPH):
// one wavefront per receiver charge group a, sweeping the other groups in
// chunks of 64 (lane = group b; reference atoms are L2-resident).  A pair
// inside its class cut-off goes to a's neighbour row through a ballot/prefix
// compaction; the pairs beyond it (and inside RcLRF) form the chunk's far
// word, and the wave then adds the charges of those groups' atoms to a's
// expansion lane by atom over the chunk's run of packed records (lrf_update,
// nonbondene.f90:628-725), so every lane has an atom whatever the group sizes.
// ANY: some system of the launch has iuse_switch_atom = 0 (any_atom), whose
// group tests scan atom pairs; the switch-atom form is compiled without it.
//
// Bound by the vector unit: an atom costs 43 FP32 slots (about 55 FP64 ones)
// for its 20 sums.  Around them: the run is read LRF_U records per lane at a
// time (64 waters are three), the first before the group tests, from a base
// that moves in scalar registers; FP32 has the next batch in flight while one
// is summed, FP64 the next chunk's groups.  A record's group is
// one bit of a 64-bit word, so a test is two ANDs and reads past the run find
// 0; FP64 takes the sums raw too, with rinv_inner in place of a root and three
// divisions.  Measured, the partner-atom rows included: 2,620 -> 2,330 us for 51
// windows of 11,056 atoms in FP32, 6,970 -> 3,420 us in FP64; 19,440 atoms in
// FP64 710 -> 331 us.
// LRF: for the systems that want the expansion, the others leave at once (and
// the other way round): without it the sweep reads no records and has the next
// chunk's groups in flight.  ANY reads a batch of records when it sums it: held
// over the group tests, which loop over atom pairs, they leave three waves per
// SIMD (51 windows of 11,056 atoms in FP32 6.6 ms, 6.15 so).
#define LRF_U 3
template <typename R, bool ANY, bool LRF>
__global__ __launch_bounds__(64 * LS_WPB) void k_lists_lrf(const DevSys* __restrict__ systems) {
  const DevSys& S = systems[blockIdx.y];
  const int a = uni(blockIdx.x * (blockDim.x / QNB_WAVE) + threadIdx.x / QNB_WAVE);
  if (a >= S.ncgp || (S.use_lrf != 0) != LRF) return;
  const int lane = threadIdx.x % QNB_WAVE;
  const double* __restrict__ x = S.x;
  const int ra = group_ref_atom(S, a);
  const bool a_sol = a < S.ncgp_solute;
  // centre of a (cgp_centers, nonbondene.f90:43-78): sum in atom order, then divide
  double cx = 0.0, cy = 0.0, cz = 0.0;
  const int ga0 = ldc(S.gfirst + a), ga1 = ldc(S.glast + a);
  for (int k = ga0; k <= ga1; k++) {
    int at = ldc(S.cgpatom + k);
    cx = cx + ldg(x + 3 * at);
    cy = cy + ldg(x + 3 * at + 1);
    cz = cz + ldg(x + 3 * at + 2);
  }
  double nat = (double)(ga1 - ga0 + 1);
  cx = cx / nat;
  cy = cy / nat;
  cz = cz / nat;
  const R cxr = (R)cx, cyr = (R)cy, czr = (R)cz;
  double acc[LRF_NF];
#pragma unroll
  for (int k = 0; k < LRF_NF; k++) acc[k] = 0.0;
  int count = 0, count_sol = 0;
  int* row = S.nbr + (size_t)a * S.cap;
  // mixed path: the lane's FP32 sums since the last flush to FP64, flushed
  // after a chunk once a lane has been offered LRF_FLUSH atoms (at most
  // LRF_FLUSH - 1 plus one chunk's share)
  constexpr int LRF_FLUSH = 16;
  constexpr bool F32 = sizeof(R) == 4;
  float pf[LRF_NF];
#pragma unroll
  for (int k = 0; k < LRF_NF; k++) pf[k] = 0.0f;
  int offered = 0;
  if (!ldg(S.excl + ra)) {
    const int ncgp = S.ncgp, nsol = S.ncgp_solute;
    const auto grs = buf_rsrc(S.gref, (size_t)ncgp * 32);
    const d4v A = buf_d4(grs, (uint32_t)a * 32);
    constexpr uint32_t RB = F32 ? 16 : 32;
    const char* recs = F32 ? (const char*)S.xqg : (const char*)S.xqgd;
    const char* bits = (const char*)S.gbit;
    // the cut-off of a pair with a solute group and with a water, given a
    const double cut_sol = a_sol ? S.rcpp2 : S.rcpw2, cut_wat = a_sol ? S.rcpw2 : S.rcww2;
    const bool quirk = pw_quirk(S), any_atom = ANY && S.any_atom;
    const double rclrf2 = LRF ? S.rclrf2 : -1.0;
    constexpr bool AHEAD = !F32 || !LRF;  // next chunk's groups in flight
    using Rec = decltype(lrf_rec<R>(grs, 0));
    // the chunk's atoms: the run from b0's first to its last group's last; FP64
    // requests the next chunk's groups while it sums this one (FP32 has no
    // registers for that beside the sums at four waves per SIMD)
    int k1 = ldc(S.gfirst);
    d4v Gn = buf_d4(grs, (uint32_t)lane * 32);
    for (int b0 = 0; b0 < ncgp; b0 += QNB_WAVE) {
      const int b = b0 + lane;
      const d4v G = AHEAD ? Gn : buf_d4(grs, (uint32_t)b * 32);  // 0 past the last group
      const int k0 = ldc(S.gfirst + b0);
      k1 = ldc(S.glast + min(b0 + QNB_WAVE, ncgp) - 1) + 1;
      if constexpr (AHEAD) Gn = buf_d4(grs, (uint32_t)(b + QNB_WAVE) * 32);
      Rec r[LRF_U];
      u2v s[LRF_U];
      auto fetch = [&](int k, Rec* rr, u2v* ss) {
        // 0 past the end of the run
        const auto rs = buf_rsrc(recs + (size_t)k * RB, (size_t)(k1 - k) * RB);
        const auto bs = buf_rsrc(bits + (size_t)k * 8, (size_t)(k1 - k) * 8);
#pragma unroll
        for (int u = 0; u < LRF_U; u++) {
          rr[u] = lrf_rec<R>(rs, (uint32_t)(lane + u * QNB_WAVE) * RB);
          ss[u] = buf_u2(bs, (uint32_t)(lane + u * QNB_WAVE) * 8);
        }
      };
      if constexpr (LRF && !ANY) fetch(k0, r, s);
      bool in = false, far = false;
      if (G.w != 0.0 && b != a) {
        const bool b_sol = b < nsol;
        const double cut2 = b_sol ? cut_sol : cut_wat;
        double r2;
        bool inside;
        if (any_atom && (a_sol || b_sol)) {
          inside = any_atom_pair(S, x, a, b, a_sol, b_sol, ra, group_ref_atom(S, b), cut2, r2);
        } else if (quirk && a_sol != b_sol) {
          // nbpwlist's test point: the switch atom up to the group's first
          // water inside, atom glast + 1 after it (LRF off: r2 unused)
          const int g = a_sol ? a : b, w = (a_sol ? b : a) - nsol;
          const int wf = ldg(S.pw_first + g);
          r2 = 0.0;
          inside = w == wf ||
                   (w > wf && dist4(x, ldg(S.glast + g) + 1, a_sol ? group_ref_atom(S, b) : ra) <= cut2);
        } else {
          r2 = dist4v(A, G);
          inside = r2 <= cut2;
        }
        in = inside;
        far = !inside && r2 <= rclrf2;
      }
      const uint64_t m = __ballot(in);
      if (m != 0) {
        const int pos = count + __popcll(m & ((1ull << lane) - 1ull));
        if (in && pos < S.cap) stg(row + pos, b);
        count += __popcll(m);
        if (b0 < nsol) count_sol += __popcll(__ballot(in && b < nsol));
      }
      if constexpr (!LRF) continue;
      const uint64_t fw = __ballot(far);
      if (fw == 0) continue;
      if constexpr (ANY) fetch(k0, r, s);
      const uint32_t f0 = (uint32_t)fw, f1 = (uint32_t)(fw >> 32);
      auto sum = [&](const Rec* rr, const u2v* ss) {
#pragma unroll
        for (int u = 0; u < LRF_U; u++)
          if (((ss[u][0] & f0) | (ss[u][1] & f1)) != 0) {
            if constexpr (F32) lrf_accumulate<float>(pf, rr[u].x - cxr, rr[u].y - cyr, rr[u].z - czr, rr[u].w);
            else lrf_accumulate<double>(acc, rr[u].x - cxr, rr[u].y - cyr, rr[u].z - czr, rr[u].w);
          }
      };
      if constexpr (F32 && !ANY) {
        for (int k = k0 + LRF_U * QNB_WAVE; k < k1; k += LRF_U * QNB_WAVE) {
          Rec rn[LRF_U];
          u2v sn[LRF_U];
          fetch(k, rn, sn);
          sum(r, s);
#pragma unroll
          for (int u = 0; u < LRF_U; u++) r[u] = rn[u], s[u] = sn[u];
        }
        sum(r, s);
      } else {
        sum(r, s);
        for (int k = k0 + LRF_U * QNB_WAVE; k < k1; k += LRF_U * QNB_WAVE) {
          fetch(k, r, s);
          sum(r, s);
        }
      }
      if constexpr (F32) {
        offered += (k1 - k0 + QNB_WAVE - 1) / QNB_WAVE;
        if (offered >= LRF_FLUSH) {
#pragma unroll
          for (int c = 0; c < LRF_NF; c++) {
            acc[c] += (double)pf[c];
            pf[c] = 0.0f;
          }
          offered = 0;
        }
      }
    }
  }
  if constexpr (LRF) {
    if constexpr (F32)
#pragma unroll
      for (int c = 0; c < LRF_NF; c++) acc[c] += (double)pf[c];
    const double tr = wave_sum_tr<double, LRF_NF>(acc, lane);
#pragma unroll
    for (int k = 0; k < LRF_NF; k++) acc[k] = lane_value(tr, wave_sum_tr_lane<LRF_NF>(k));
  }
  if (lane == 0) {
    double t[LRF_NF];
    lrf_tensors(t, acc);
    S.nnbr[a] = count;
    S.nnsol[a] = count_sol;
    if (count > S.cap) atomicMax(S.need, count);
    double* L = S.lrf + (size_t)QNB_NLRF * a;
    L[0] = cx;
    L[1] = cy;
    L[2] = cz;
    L[3] = t[0];
    L[4] = t[1];
    L[5] = t[2];
    L[6] = t[3];
    const int p2[3][3] = {{4, 5, 6}, {5, 7, 8}, {6, 8, 9}};
    for (int k = 0; k < 3; k++)
      for (int c = 0; c < 3; c++) L[7 + 3 * k + c] = t[p2[k][c]];
    for (int n = 0; n < 3; n++)
      for (int j = 0; j < 3; j++)
        for (int c = 0; c < 3; c++) L[16 + 3 * (j + 3 * n) + c] = t[t3index(n, j, c)];
  }
  if (a < S.atom_rows) {
    __threadfence_block();  // the row's stores before its loads
    expand_row(S, a, min(count_sol, S.cap), lane, threadIdx.x / QNB_WAVE);
  }
}

// ---------------------------------------------------------------------------
// Q-atom lists (nbqplist nonbondene.f90:3647-3742, nbqwlist 3862-3944): flags
// and ordered compaction of the waters and solute atoms within Rcq of xpcent.
// One block of 1024 threads per system; each thread takes a contiguous chunk
// so the compacted order is the reference's append order.
__global__ __launch_bounds__(1024) void k_qlists(const DevSys* __restrict__ systems) {
  const DevSys& S = systems[blockIdx.x];
  __shared__ int scan[1024];
  const int t = threadIdx.x, nt = blockDim.x;
  // waters
  {
    const int per = (S.nwat + nt - 1) / nt, w0 = t * per, w1 = min(S.nwat, w0 + per);
    int c = 0;
    for (int w = w0; w < w1; w++) {
      int o = S.nat_solute + S.sa * w;
      bool in = !S.excl[o] && dist4p(S.x, o, S.xp) <= S.rcq2;
      S.qw_in[w] = in;
      c += in;
    }
    scan[t] = c;
    __syncthreads();
    for (int off = 1; off < nt; off <<= 1) {
      int v = t >= off ? scan[t - off] : 0;
      __syncthreads();
      scan[t] += v;
      __syncthreads();
    }
    int pos = scan[t] - c;
    for (int w = w0; w < w1; w++)
      if (S.qw_in[w]) S.qw_list[pos++] = w;
    if (t == nt - 1) S.nq_lists[0] = scan[t];
    __syncthreads();
  }
  // solute atoms, group by group
  {
    const int per = (S.ncgp_solute + nt - 1) / nt, g0 = t * per, g1 = min(S.ncgp_solute, g0 + per);
    int c = 0;
    for (int g = g0; g < g1; g++) {
      const bool in = qp_group_in(S, S.x, g);
      S.qp_in[g] = in;
      if (in)
        for (int k = S.gfirst[g]; k <= S.glast[g]; k++) c += !S.qconn3[S.cgpatom[k]];
    }
    scan[t] = c;
    __syncthreads();
    for (int off = 1; off < nt; off <<= 1) {
      int v = t >= off ? scan[t - off] : 0;
      __syncthreads();
      scan[t] += v;
      __syncthreads();
    }
    int pos = scan[t] - c;
    for (int g = g0; g < g1; g++)
      if (S.qp_in[g])
        for (int k = S.gfirst[g]; k <= S.glast[g]; k++) {
          int i = S.cgpatom[k];
          if (!S.qconn3[i]) S.qp_list[pos++] = i;
        }
    if (t == nt - 1) S.nq_lists[1] = scan[t];
  }
}

// term bits (include/qnb.h enum qnb_term)
enum : uint32_t { T_WW = QNB_T_WW, T_QW = QNB_T_QW, T_PW = QNB_T_PW, T_PP = QNB_T_PP, T_QP = QNB_T_QP,
                  T_LRF = QNB_T_LRF, T_QQ = QNB_T_QQ, T_QQP = QNB_T_QQP, T_RAD = QNB_T_RAD, T_POL = QNB_T_POL,
                  T_SINT = QNB_T_SINT };

// ---------------------------------------------------------------------------
// Receiver-side forces: one wavefront per charge group a (or four, see
// solute_receiver) walks its partners, every lane one partner atom at a time:
// solute partners from the receiver's atom list (expand_row), so lanes stay
// balanced however large the groups are, waters from the neighbour row.  A lane
// forms the partner's position relative to the receiver's reference atom once in
// FP64, rounds it to R and evaluates it against the receiver atoms (offsets from
// the same reference point), accumulating per-lane forces in R; the wave reduces
// them in FP64.  Pair forms: water-water as nonbond_ww_spc / nonbond_ww
// (nonbondene.f90:5886-5975, 5509-5573: O-O LJ + Coulomb, the other 8
// Coulomb only for SPC), pw from the pw table (nonbond_pw 4856-4916), pp from
// pp_pair (nonbond_pp 4694-4760).  Writes (not adds) d for every atom of a,
// and the wave's energy partials into epart[a] on the sampled steps.

// the pair (lo, hi) in lo's long exclusion / 1-4 list: 1 excluded, 2 1-4,
// 0 neither (kept out of line: rare, and its loop would stop the callers'
// receiver-atom loops from unrolling)
__device__ __noinline__ int long_pair_kind(const DevSys& S, int lo, int hi) {
  bool ex = false, is14 = false;
  for (int m = ldg(S.lx_off + lo); m < ldg(S.lx_off + lo + 1); m++)
    if (ldg(S.lx_j + m) == hi) {
      if (ldg(S.lx_kind + m) == 0) ex = true;
      else is14 = true;
    }
  return ex ? 1 : (is14 ? 2 : 0);
}

// the pair (i, j) from the atoms' exclusion and 1-4 masks: 1 excluded, 2 1-4,
// 0 neither
__device__ __forceinline__ int pair_kind(const DevSys& S, int i, uint32_t xi, uint32_t mi, int j, uint32_t xj,
                                         uint32_t mj) {
  const bool il = i < j;
  const int dk = il ? j - i : i - j;
  const uint32_t xm = il ? xi : xj, m14 = il ? mi : mj;
  if (dk <= 25) {
    const uint32_t bit = 1u << (dk - 1);
    return (xm & bit) ? 1 : ((m14 & bit) ? 2 : 0);
  }
  return (xm >> 31) ? long_pair_kind(S, il ? i : j, il ? j : i) : 0;
}

// Solute-solute pair parameters from the two atoms' types, charges and exclusion
// masks (bit 31: partners beyond the 25-atom window, looked up in the long
// list), as pp_int_comp / precompute_set_values_pp (simprep.f90:2952-3065,
// 3321-3350) would tabulate them; false: the pair does not interact.
struct PPAtom {
  int i, t;
  uint32_t xm, m14;
  double q;
};
__device__ __forceinline__ bool pp_pair(const DevSys& S, const PPAtom& P, const PPAtom& Q, double& A, double& B,
                                        double& el) {
  const int kind = pair_kind(S, P.i, P.xm, P.m14, Q.i, Q.xm, Q.m14);
  if (kind == 1) return false;
  const bool is14 = kind == 2;
  const int vdw = is14 ? 3 : ldg(S.ljcod + (P.t + Q.t * S.ntypes));
  const int kp = P.t * 3 + vdw - 1, kq = Q.t * 3 + vdw - 1;
  if (S.ivdw_rule == 1) {
    A = ldg(S.avdw + kp) * ldg(S.avdw + kq);
    B = ldg(S.bvdw + kp) * ldg(S.bvdw + kq);
  } else {
    double tA = ldg(S.avdw + kp) + ldg(S.avdw + kq);
    tA = tA * tA;
    tA = tA * tA * tA;
    double tB = ldg(S.bvdw + kp) * ldg(S.bvdw + kq);
    A = (tA * tA) * tB;
    B = 2.0 * tA * tB;
  }
  el = P.q * Q.q;
  const bool set = fabs(A) > 1.0e-10 || fabs(B) > 1.0e-10 || fabs(el) > 1.0e-10;
  if (vdw == 3) el = el * S.el14;
  return set;
}

// ---------------------------------------------------------------------------
// The lambda-weighted dv of a Q pair over its states (nbe_qx per state,
// nonbonded.f90:200-222): `par(s)` gives state s's A, B, el and soft-core score.
// Without a soft core the force is linear in A, B and el, so on the steps that
// sample no energies the FP64 path weights and sums the states' parameters
// first and evaluates the pair once.  The mixed path keeps the states apart,
// as every FP32 sum of these kernels keeps its terms and their order: a run of
// many windows meets a group pair at its cut-off at every list update, and
// another rounding of the forces would take such a pair the other way.
template <typename R>
struct QPar {
  R A, B, q, sc;
};
template <typename R, int NS, typename F>
__device__ __forceinline__ R qx_states(const DevSys& S, R r2, R r, int ns, double* eq, bool want, F par) {
  const R r6 = r2 * r2 * r2;
  if constexpr (sizeof(R) == 4) {
    R dvs = R(0);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if (s >= ns) break;
      const QPar<R> p = par(s);
      dvs += PairMath<R>::nbe_qx(r2, r, r6, p.A, p.B, p.q, p.sc, (R)S.lambda[s], eq[2 * s], eq[2 * s + 1], want);
    }
    return dvs;
  }
  QPar<R> p[NS];
  R A = R(0), B = R(0), q = R(0);
  bool soft = false;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    if (s >= ns) break;
    p[s] = par(s);
    const R lam = (R)S.lambda[s];
    A += lam * p[s].A;
    B += lam * p[s].B;
    q += lam * p[s].q;
    soft = soft || p[s].sc != R(0);
  }
  if (!want && !soft) return r2 * (r6 * (R(6) * B - R(12) * A * r6) - q * r);
  R dvs = R(0);
#pragma unroll
  for (int s = 0; s < NS; s++) {
    if (s >= ns) break;
    dvs += PairMath<R>::nbe_qx(r2, r, r6, p[s].A, p[s].B, p[s].q, p[s].sc, (R)S.lambda[s], eq[2 * s], eq[2 * s + 1],
                               want);
  }
  return dvs;
}
// Coulomb only (nbe_qspc, nonbonded.f90:226-243: an SPC hydrogen)
template <typename R, int NS, typename F>
__device__ __forceinline__ R qspc_states(const DevSys& S, R r2, R r, int ns, double* eq, bool want, F el) {
  R dvs = R(0);
#pragma unroll
  for (int s = 0; s < NS; s++) {
    if (s >= ns) break;
    const R Vel = el(s) * r;
    if (want) eq[2 * s] += (double)Vel;
    dvs += -r2 * Vel * (R)S.lambda[s];
  }
  return dvs;
}
// entry (iq, k, s) of the Q-solvent table in the pair arithmetic's type
template <typename R>
__device__ __forceinline__ QPar<R> qw_par(const DevSys& S, int iq, int k, int s) {
  const R* t = qp_tab<R>(S.qw_d, S.qw_f) + 4 * ((size_t)(iq * S.sa + k) * S.nstates + s);
  return QPar<R>{ldg(t), ldg(t + 1), ldg(t + 2), ldg(t + 3)};
}
template <typename R>
__device__ __forceinline__ R qw_el(const DevSys& S, int iq, int k, int s) {
  return ldg(qp_tab<R>(S.qw_d, S.qw_f) + 4 * ((size_t)(iq * S.sa + k) * S.nstates + s) + 2);
}

// A receiver's partner atoms as its force kernel reads them: `stored` slots of its
// atom row, then, where the row was too short, al_group slots for each further
// group, its atoms from the neighbour row.  `n` slots in all.
struct PartnerRow {
  const int* al;
  int stored, groups, n;
};
__device__ __forceinline__ PartnerRow partner_row(const DevSys& S, int a, int nsr) {
  PartnerRow r;
  r.al = S.alist + (size_t)a * S.acap;
  r.stored = uni(ldg(S.alist_end + 2 * a));
  r.groups = uni(ldg(S.alist_end + 2 * a + 1));
  r.n = r.stored + (nsr - r.groups) * S.al_group;
  return r;
}
// slot q past the stored ones
__device__ __forceinline__ int row_tail(const DevSys& S, int a, int groups, int q) {
  const int p = groups + q / S.al_group, m = q % S.al_group;
  const int b = ldg(S.nbr + (size_t)a * S.cap + p);
  const int f0 = ldg(S.gfirst + b), cnt = ldg(S.glast + b) - f0 + 1;
  return m < cnt ? ldg(S.cgentry + f0 + m) | (owns(a, b) ? AL_OWN : 0) : (int)AL_SKIP;
}
// out of line for the solute receivers: rare, and their loops call in any case
// (long_pair_kind); a call would cost the water receivers two waves per SIMD
__device__ __noinline__ int row_tail_call(const DevSys& S, int a, int groups, int q) {
  return row_tail(S, a, groups, q);
}

// ---------------------------------------------------------------------------
// Solute receivers: one wavefront per solute charge group a, or, in a small
// launch (SPLIT), the four waves of a block, each with a quarter of a's
// partners.  a's atoms are taken in sweeps of up to so_ch; they are the same
// for every lane and are read into scalar registers (70 values in FP32 beside the
// pointers: about 118 words of them the compiler keeps in lanes of vector
// registers and reads back), and a lane takes one partner at a time against
// them, the next partner's data in flight meanwhile:
//  * solute partners from the receiver's atom list (expand_row; nonbond_pp,
//    nonbondene.f90:4694-4760): those of a group without an excluded or 1-4
//    pair (AL_FAR) take A, B and qq as products of per-atom factors when the
//    system uses the geometric rule with LJ code 1 throughout (ppfast): the
//    products pp_pair forms for such a pair, same operands; every other pair
//    goes through the exclusion masks and pp_pair's rules;
//  * partner waters with the fixed mapping of k_wforces (lane l takes site
//    l % 3 of water l / 3 of the round; nonbond_pw 4856-4916);
//  * the pairs inside the group (ig == jgr, i < j, nonbondene.f90:1610) and
//    the receiver side of the Q-atom - solute pairs (nonbond_qp 5157-5230).
// Writes d of the group's atoms, and the pp, pw and qp energy partials on the
// sampled steps (a pp pair's energy on its owner side).
//
// Bound by VALU issue at 51 windows and by the latency of one row in a small
// launch.  Staging 128 partners at a time through LDS, with ten receiver atoms
// in vector registers (167 of them, three waves per SIMD), took 213 us at 51
// windows of 400 ten-atom groups and 52 us for one FP64 window; staging by
// blocks of four waves 310 us at 51 windows (its barriers wait on four chains
// of loads); from the atom lists it takes 145 us, and about 20
// us split four ways.

__device__ __forceinline__ float lane_get(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_get(double v, int lane) { return lane_value(v, lane); }
__device__ __forceinline__ int lane_get(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// the sum of each lane's value over waves w0 .. w0 + n - 1 of the block, in
// wave order; every wave of the block takes part
__device__ __forceinline__ double waves_sum(double (*comb)[QNB_WAVE], double v, int w0, int n, int lane) {
  __syncthreads();
  comb[threadIdx.x / QNB_WAVE][lane] = v;
  __syncthreads();
  double s = comb[w0][lane];
  for (int w = 1; w < n; w++) s += comb[w0 + w][lane];
  return s;
}

template <typename R, int NS, bool E, bool SPLIT>
__device__ __forceinline__ void solute_receiver(const DevSys& S, uint32_t mask, int a, int wave, int waves,
                                                unsigned char* wbase, double (*comb)[QNB_WAVE]) {
  constexpr int CH = so_ch<R>();
  const int lane = threadIdx.x % QNB_WAVE;
  // the sweep's receiver data in LDS for the pairs that take it by lane:
  // charge, LJ factors of codes 1 and 3, solute-solvent parameters of the
  // three water sites, offset, index, type, masks
  double* s_rq = reinterpret_cast<double*>(wbase);
  double(*s_r3)[4] = reinterpret_cast<double(*)[4]>(s_rq + CH);
  R(*s_pw)[3][3] = reinterpret_cast<R(*)[3][3]>(s_r3 + CH);
  R(*s_o)[3] = reinterpret_cast<R(*)[3]>(s_pw + CH);
  int* s_ia = reinterpret_cast<int*>(s_o + CH);
  int* s_rt = s_ia + CH;
  uint32_t* s_rx = reinterpret_cast<uint32_t*>(s_rt + CH);
  uint32_t* s_rm = s_rx + CH;
  const double* __restrict__ x = S.x;
  const auto d = gpm(S.d);
  const int nn = uni(min(ldg(S.nnbr + a), S.cap)), nsr = uni(min(ldg(S.nnsol + a), nn));
  const int* __restrict__ row = S.nbr + (size_t)a * S.cap;
  const bool want_e = E && want_energies(S);
  const int nsol = S.nat_solute, sa = S.sa, ncs = S.ncgp_solute;
  const int ra = uni(ldg(S.gswitch + a));
  const bool aexcl = uni(ldg(S.excl + ra));
  const bool fast = S.ppfast != 0, coul_h = S.pw_coul_h != 0;
  double e_ppel = 0.0, e_ppvdw = 0.0, e_pwel = 0.0, e_pwvdw = 0.0;
  double eq[2 * NS];  // per state: qp_el, qp_vdw
#pragma unroll
  for (int k = 0; k < 2 * NS; k++) eq[k] = 0.0;
  const double xr0 = ldg(x + 3 * ra), xr1 = ldg(x + 3 * ra + 1), xr2 = ldg(x + 3 * ra + 2);
  const int g0 = uni(ldg(S.gfirst + a)), na = uni(ldg(S.glast + a)) - g0 + 1;
  const int nq = S.nqat, ns = S.nstates;
  const bool qin = (mask & T_QP) && nq > 0 && uni(ldg(S.qp_in + a));
  const bool pp = (mask & T_PP) && !aexcl;
  PartnerRow partners = partner_row(S, a, nsr);
  if (!pp) partners.stored = partners.n = 0;
  const int nsl = partners.n;
  const bool pw = (mask & T_PW) && !aexcl && nsr < nn;
  // SPLIT: sets of waves with receiver atoms of their own (nset), the waves of
  // a set sharing the partners
  const int nset = !SPLIT || na <= CH ? 1 : (na <= 2 * CH ? 2 : 4), parts = SPLIT ? waves / nset : 1;
  const int set = SPLIT ? wave / parts : 0, part = SPLIT ? wave % parts : 0;
  // the first two rounds' entries are requested before the receiver's own
  // chain of loads
  // (every count of slots is a multiple of 64, so a round's place is the wave's)
  const int t0 = QNB_WAVE * part, ts = QNB_WAVE * parts;
  auto entry = [&](int t) {
    if (t < partners.stored) return ldg(partners.al + t + lane);
    return t < nsl ? row_tail_call(S, a, partners.groups, t + lane - partners.stored) : (int)AL_SKIP;
  };
  const int e0 = entry(t0), e1 = entry(t0 + ts);
  for (int cb = 0; cb < na; cb += nset * CH) {
    const int c0 = cb + set * CH, nk = max(0, min(CH, na - c0));
    // receiver atoms: lane k loads atom c0 + k (index -1: takes no pair
    // terms), then each value is read into scalar registers
    int il = -1, i_own = 0;
    R ol0 = R(0), ol1 = R(0), ol2 = R(0), fa = R(0), fb = R(0), fc = R(0);
    if (lane < nk) {
      const int i = ldg(S.cgpatom + (g0 + c0 + lane));
      i_own = i;
      il = (!aexcl && ldg(S.iqatom + i) == 0) ? i : -1;
      ol0 = (R)(ldg(x + 3 * i) - xr0);
      ol1 = (R)(ldg(x + 3 * i + 1) - xr1);
      ol2 = (R)(ldg(x + 3 * i + 2) - xr2);
      s_ia[lane] = il;
      s_o[lane][0] = ol0;
      s_o[lane][1] = ol1;
      s_o[lane][2] = ol2;
      const R* pf = qp_tab<R>(S.ppd, S.ppf) + PP_REC * (size_t)i;
      fa = ldg(pf);
      fb = ldg(pf + 1);
      fc = ldg(pf + 2);
      s_rt[lane] = ldg(S.iac + i);
      s_rx[lane] = ldg(S.exmask + i);
      s_rm[lane] = ldg(S.m14mask + i);
      s_rq[lane] = ldg(S.crg + i);
      s_r3[lane][0] = ldg(S.ppd + PP_REC * (size_t)i);
      s_r3[lane][1] = ldg(S.ppd + PP_REC * (size_t)i + 1);
      s_r3[lane][2] = ldg(S.ppd + PP_REC * (size_t)i + 4);
      s_r3[lane][3] = ldg(S.ppd + PP_REC * (size_t)i + 5);
      if (pw && sa == 3)
#pragma unroll
        for (int kb = 0; kb < 3; kb++) {
          const size_t tt = (size_t)i + (size_t)nsol * kb;
          s_pw[lane][kb][0] = (R)ldg(S.pwA + tt);
          s_pw[lane][kb][1] = (R)ldg(S.pwB + tt);
          s_pw[lane][kb][2] = (R)ldg(S.pwEl + tt);
        }
    }
    __builtin_amdgcn_wave_barrier();
    int ri[CH];
    R ro[CH][3], rA[CH], rB[CH], rQ[CH], f[CH][3];
#pragma unroll
    for (int k = 0; k < CH; k++) {
      ri[k] = lane_get(il, k);
      ro[k][0] = lane_get(ol0, k);
      ro[k][1] = lane_get(ol1, k);
      ro[k][2] = lane_get(ol2, k);
      rA[k] = lane_get(fa, k);
      rB[k] = lane_get(fb, k);
      rQ[k] = lane_get(fc, k);
      f[k][0] = f[k][1] = f[k][2] = R(0);
    }
    // A, B and qq of sweep atom k with atom j (pp_pair); false: no pair
    auto general = [&](int k, int i, int j, const double* qf, double qc, uint32_t qx, uint32_t qm, R& A, R& B,
                       R& el) {
      double Ad, Bd, eld;
      if (fast) {
        // code 1, or 3 for a 1-4 pair
        const int kind = pair_kind(S, i, s_rx[k], s_rm[k], j, qx, qm);
        if (kind == 1) return false;
        const bool is14 = kind == 2;
        Ad = is14 ? s_r3[k][2] * qf[2] : s_r3[k][0] * qf[0];
        Bd = is14 ? s_r3[k][3] * qf[3] : s_r3[k][1] * qf[1];
        eld = s_rq[k] * qc;
        if (!(fabs(Ad) > 1.0e-10 || fabs(Bd) > 1.0e-10 || fabs(eld) > 1.0e-10)) return false;
        if (is14) eld = eld * S.el14;
      } else {
        const PPAtom P{i, s_rt[k], s_rx[k], s_rm[k], s_rq[k]};
        const PPAtom Q{j, ldg(S.iac + j), qx, qm, qc};
        if (!pp_pair(S, P, Q, Ad, Bd, eld)) return false;
      }
      A = (R)Ad;
      B = (R)Bd;
      el = (R)eld;
      return true;
    };
    // ---- partner solute atoms, one list slot per lane; the next slot's
    // position and factors load while this one is evaluated
    if (nk > 0 && nsl > 0) {
      int e = e0, en = e1;
      double px, py, pz;
      R pA, pB, pQ;
      auto fetch = [&](int entry) {
        const int j = entry & AL_ATOM;
        px = ldg(x + 3 * j);
        py = ldg(x + 3 * j + 1);
        pz = ldg(x + 3 * j + 2);
        const R* pf = qp_tab<R>(S.ppd, S.ppf) + PP_REC * (size_t)j;
        pA = ldg(pf);
        pB = ldg(pf + 1);
        pQ = ldg(pf + 2);
      };
      fetch(e);
      for (int t = t0; t < nsl; t += ts) {
        const R dx = (R)(px - xr0), dy = (R)(py - xr1), dz = (R)(pz - xr2);
        const R qA = pA, qB = pB, qQ = pQ;
        const int ec = e;
        e = en;
        fetch(e);
        en = entry(t + 2 * ts);
        if (ec & AL_SKIP) continue;
        const bool acc = want_e && (ec & AL_OWN);
        R pel = R(0), pvdw = R(0);
        // AL_FAR: no exclusion or 1-4 pair possible, A, B, qq from the factors
        const bool far = fast && (ec & AL_FAR);
        const int j = ec & AL_ATOM;
        double qf[4], qc = 0.0;
        uint32_t qx = 0u, qm = 0u;
        // the receiver data in LDS is read where it is used: hoisted out of the
        // loop it would fill the registers that the other partners need
        __asm__ volatile("" ::: "memory");
        if (!far) {
          const double* pf = S.ppd + PP_REC * (size_t)j;
          qf[0] = ldg(pf), qf[1] = ldg(pf + 1), qf[2] = ldg(pf + 4), qf[3] = ldg(pf + 5);
          qc = ldg(S.crg + j);
          qx = ldg(S.exmask + j);
          qm = ldg(S.m14mask + j);
        }
#pragma unroll
        for (int k = 0; k < CH; k++) {
          if (ri[k] < 0) continue;
          R A = rA[k] * qA, B = rB[k] * qB, el = rQ[k] * qQ;
          if (far) {
            // pp_pair's `set` test (QREAL_EPS, src/sizes.f90:50); in FP32
            // a pair of zero parameters adds exactly zero, so it is skipped
            // only on the FP64 path
            if constexpr (sizeof(R) == 8)
              if (!(fabs(A) > R(1.0e-10) || fabs(B) > R(1.0e-10) || fabs(el) > R(1.0e-10))) continue;
          } else if (!general(k, ri[k], j, qf, qc, qx, qm, A, B, el)) {
            continue;
          }
          const R ux = dx - ro[k][0], uy = dy - ro[k][1], uz = dz - ro[k][2];
          const R dv = PairMath<R>::nbe(ux, uy, uz, A, B, el, pel, pvdw, acc);
          f[k][0] += ux * dv;
          f[k][1] += uy * dv;
          f[k][2] += uz * dv;
        }
        if (acc) {
          e_ppel += (double)pel;
          e_ppvdw += (double)pvdw;
        }
      }
    }
    // ---- partner solvent molecules: lane l takes site kb = l % sa of molecule
    // l / sa of the round, M = 64 / sa molecules per round
    if (pw && nk > 0) {
      const int M = sa == 3 ? QNB_WAVE / 3 : QNB_WAVE / sa;
      const int kb = sa == 3 ? lane % 3 : lane % sa, m = sa == 3 ? lane / 3 : lane / sa;
      if (m < M)
        for (int p = nsr + m + M * part; p < nn; p += M * parts) {
          const int j = nsol + sa * (ldg(row + p) - ncs) + kb;
          const R dx = (R)(ldg(x + 3 * j) - xr0), dy = (R)(ldg(x + 3 * j + 1) - xr1),
                  dz = (R)(ldg(x + 3 * j + 2) - xr2);
          R pel = R(0), pvdw = R(0);
          __asm__ volatile("" ::: "memory");
#pragma unroll
          for (int k = 0; k < CH; k++) {
            if (ri[k] < 0) continue;
            R A, B, el;
            if (sa == 3) {
              A = s_pw[k][kb][0];
              B = s_pw[k][kb][1];
              el = s_pw[k][kb][2];
            } else {
              const size_t tt = (size_t)ri[k] + (size_t)nsol * kb;
              A = (R)ldg(S.pwA + tt);
              B = (R)ldg(S.pwB + tt);
              el = (R)ldg(S.pwEl + tt);
            }
            const R ux = dx - ro[k][0], uy = dy - ro[k][1], uz = dz - ro[k][2];
            const R dv = PairMath<R>::nbe(ux, uy, uz, A, B, el, pel, pvdw, want_e);
            f[k][0] += ux * dv;
            f[k][1] += uy * dv;
            f[k][2] += uz * dv;
          }
          if (want_e) {
            e_pwel += (double)pel;
            e_pwvdw += (double)pvdw;
          }
        }
    }
    // ---- pairs inside the group: lane (g, kq) = (lane / nk, lane % nk)
    // takes receiver atom kq against group atoms q = g, g + G, ...
    // (G = 64 / nk); an atom of this sweep has its data in LDS, others
    // (groups larger than one sweep) are read from memory
    if (pp && nk > 0) {
      const int G = QNB_WAVE / nk, kq = lane % nk, g = lane / nk;
      const int i = s_ia[kq];
      R fq[3] = {R(0), R(0), R(0)};
      if (g < G && i >= 0) {
        const R ox = s_o[kq][0], oy = s_o[kq][1], oz = s_o[kq][2];
        for (int q = g + G * part; q < na; q += G * parts) {
          const int ql = q - c0;
          const bool in_sweep = ql >= 0 && ql < nk;
          int j;
          R dx, dy, dz;
          if (in_sweep) {
            j = s_ia[ql];  // -1: a Q-atom, whose pairs belong to the Q kernels
            dx = s_o[ql][0];
            dy = s_o[ql][1];
            dz = s_o[ql][2];
          } else {
            j = ldg(S.cgpatom + (g0 + q));
            if (ldg(S.iqatom + j) != 0) continue;
            dx = (R)(ldg(x + 3 * j) - xr0);
            dy = (R)(ldg(x + 3 * j + 1) - xr1);
            dz = (R)(ldg(x + 3 * j + 2) - xr2);
          }
          if (j < 0 || j == i) continue;
          R A, B, el;
          bool ok;
          if (in_sweep) {
            ok = general(kq, i, j, s_r3[ql], s_rq[ql], s_rx[ql], s_rm[ql], A, B, el);
          } else {
            const double* pf = S.ppd + PP_REC * (size_t)j;
            const double qf[4] = {ldg(pf), ldg(pf + 1), ldg(pf + 4), ldg(pf + 5)};
            ok = general(kq, i, j, qf, ldg(S.crg + j), ldg(S.exmask + j), ldg(S.m14mask + j), A, B, el);
          }
          if (!ok) continue;
          const R ux = dx - ox, uy = dy - oy, uz = dz - oz;
          const R dv = PairMath<R>::nbe(ux, uy, uz, A, B, el, e_ppel, e_ppvdw, want_e && i < j);
          fq[0] += ux * dv;
          fq[1] += uy * dv;
          fq[2] += uz * dv;
        }
      }
#pragma unroll
      for (int k = 0; k < CH; k++)
        if (k == kq) {
          f[k][0] += fq[0];
          f[k][1] += fq[1];
          f[k][2] += fq[2];
        }
    }
    // ---- Q-atom - solute atom, receiver side: lane (g, kq) = (lane / nk,
    // lane % nk) takes receiver atom kq against Q-atoms g, g + G, ... (G = 64
    // / nk)
    if (qin && nk > 0) {
      const R *qtA = qp_tab<R>(S.qpA, S.qpA_f), *qtB = qp_tab<R>(S.qpB, S.qpB_f);
      const R *qtE = qp_tab<R>(S.qpEl, S.qpEl_f), *qtS = qp_tab<R>(S.qpSc, S.qpSc_f);
      const int G = QNB_WAVE / nk, kq = lane % nk, g = lane / nk;
      const int i = __shfl(il, kq, QNB_WAVE);
      const R ox = __shfl(ol0, kq, QNB_WAVE), oy = __shfl(ol1, kq, QNB_WAVE), oz = __shfl(ol2, kq, QNB_WAVE);
      R fq[3] = {R(0), R(0), R(0)};
      if (g < G && i >= 0 && !ldg(S.qconn3 + i)) {
        for (int iq = g + G * part; iq < nq; iq += G * parts) {
          const int q = ldg(S.iqseq + iq);
          const R ux = (R)(ldg(x + 3 * q) - xr0) - ox, uy = (R)(ldg(x + 3 * q + 1) - xr1) - oy,
                  uz = (R)(ldg(x + 3 * q + 2) - xr2) - oz;
          R r2, r;
          rinv(norm2(ux, uy, uz), r2, r);
          const R dvs = qx_states<R, NS>(S, r2, r, ns, eq, want_e, [&](int s) {
            const size_t t = (size_t)i + (size_t)nsol * ((size_t)iq + (size_t)nq * s);
            return QPar<R>{ldg(qtA + t), ldg(qtB + t), ldg(qtE + t), ldg(qtS + t)};
          });
          fq[0] += ux * dvs;
          fq[1] += uy * dvs;
          fq[2] += uz * dvs;
        }
      }
#pragma unroll
      for (int k = 0; k < CH; k++)
        if (k == kq) {
          f[k][0] += fq[0];
          f[k][1] += fq[1];
          f[k][2] += fq[2];
        }
    }
    // reduce all 3 CH force components of the wave at once; component c of
    // sweep atom k is value 3k + c
    R fv[3 * CH];
#pragma unroll
    for (int k = 0; k < CH; k++)
#pragma unroll
      for (int c = 0; c < 3; c++) fv[3 * k + c] = f[k][c];
    double fs = wave_sum_tr(fv, lane);
    if constexpr (SPLIT) fs = waves_sum(comb, fs, set * parts, parts, lane);
    const int j = wave_sum_tr_index<3 * CH>(lane);
    const int iw = __shfl(i_own, j / 3, QNB_WAVE);
    if (part == 0 && wave_sum_tr_writer<3 * CH>(lane) && j / 3 < nk) d[3 * iw + j % 3] = -fs;
    __builtin_amdgcn_wave_barrier();
  }
  if (!want_e) return;
  // pp and pw energies, then each state's qp el and vdW
  double en[4 + 2 * NS];
  int slot[4 + 2 * NS];
  en[0] = e_ppel, slot[0] = E_PP_EL;
  en[1] = e_ppvdw, slot[1] = E_PP_VDW;
  en[2] = e_pwel, slot[2] = E_PW_EL;
  en[3] = e_pwvdw, slot[3] = E_PW_VDW;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    en[4 + 2 * s] = eq[2 * s], slot[4 + 2 * s] = E_Q0 + 6 * s + 2;
    en[5 + 2 * s] = eq[2 * s + 1], slot[5 + 2 * s] = E_Q0 + 6 * s + 3;
  }
  double sum = wave_sum_tr(en, lane);
  if constexpr (SPLIT) sum = waves_sum(comb, sum, 0, waves, lane);
  if (!SPLIT || wave == 0) store_energy_record<4 + 2 * NS>(S.epart + (size_t)a * QNB_NE, sum, slot, lane);
}

template <typename R, int NS, bool E>
__global__ __launch_bounds__(64 * FC_WPB) void k_sforces(const DevSys* __restrict__ systems, uint32_t mask, int imap,
                                                         int nb, int ninst) {
  int inst, blk;
  if (!map_block(imap, nb, ninst, inst, blk)) return;
  const DevSys& S = systems[inst];
  const int wib = threadIdx.x / QNB_WAVE;
  const int a = uni(blk * (int)(blockDim.x / QNB_WAVE) + wib);
  if (a >= S.ncgp_solute) return;
  extern __shared__ __align__(16) unsigned char so_smem[];
  solute_receiver<R, NS, E, false>(S, mask, a, 0, 1, so_smem + (size_t)wib * so_wave_bytes<R>(), nullptr);
}

// ---------------------------------------------------------------------------
// Water receivers (rigid 3-site solvent): one wavefront per water a.  Its
// neighbour row is sorted, so the solute groups (indices below ncgp_solute)
// come first, then the waters.  Solute partners come from the receiver's atom
// list (expand_row), one partner atom per lane against the three receiver atoms with
// the pw parameters (nonbond_pw, nonbondene.f90:4856-4916; energy counted on
// the solute side).  Partner waters need no staging: their atoms are
// consecutive, so in each round lane l takes atom l % 3 of the row's water
// (l / 3) of the round, 21 waters per round (lane 63 idle), reading the
// position straight from x, and evaluates it against the three receiver
// atoms (nonbond_ww_spc nonbondene.f90:5886-5975: O-O LJ + Coulomb, the
// other pairs Coulomb only; nonbond_ww 5509-5573 for other solvents).  Then
// the receiver side of the Q-atom - water pairs.  Writes d of the three
// atoms, and the wave's ww and qw energy partials on the sampled steps.
template <typename R, int NS, bool E>
__device__ __forceinline__ void water_receiver(const DevSys& S, uint32_t mask, int a) {
  const int lane = threadIdx.x % QNB_WAVE;
  const double* __restrict__ x = S.x;
  const auto d = gpm(S.d);
  const int nn = uni(min(ldg(S.nnbr + a), S.cap));
  const int* __restrict__ row = S.nbr + (size_t)a * S.cap;
  const bool want_e = E && want_energies(S);
  const int nsol = S.nat_solute, sa = S.sa, ncs = S.ncgp_solute;
  const int ra = nsol + sa * (a - ncs);
  const bool aexcl = uni(ldg(S.excl + ra));
  const int nq = S.nqat, ns = S.nstates;
  double e_el = 0.0, e_vdw = 0.0;
  double eq[2 * NS];  // per state: qw_el, qw_vdw
#pragma unroll
  for (int k = 0; k < 2 * NS; k++) eq[k] = 0.0;
  const double xr0 = ldg(x + 3 * ra), xr1 = ldg(x + 3 * ra + 1), xr2 = ldg(x + 3 * ra + 2);
  R o[3][3], f[3][3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    o[k][0] = (R)(ldg(x + (3 * (ra + k))) - xr0);
    o[k][1] = (R)(ldg(x + (3 * (ra + k) + 1)) - xr1);
    o[k][2] = (R)(ldg(x + (3 * (ra + k) + 2)) - xr2);
    f[k][0] = f[k][1] = f[k][2] = R(0);
  }
  if (!aexcl) {
    const int nsr = uni(min(ldg(S.nnsol + a), nn));  // length of the row's solute prefix
    // solute partners from the receiver's atom list, one per lane, the next
    // one's data in flight
    if (mask & T_PW) {
      const PartnerRow partners = partner_row(S, a, nsr);
      const int n = partners.stored;
      const int* __restrict__ al = partners.al;
      int e = lane < n ? ldg(al + lane) : 0;
      int en = lane + QNB_WAVE < n ? ldg(al + lane + QNB_WAVE) : 0;
      double px = 0.0, py = 0.0, pz = 0.0;
      R pl[9];
      auto fetch = [&](int i) {
        px = ldg(x + 3 * i);
        py = ldg(x + 3 * i + 1);
        pz = ldg(x + 3 * i + 2);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          if constexpr (sizeof(R) == 4) {
            pl[3 * k] = ldg(S.pw_f + PW_REC * i + 3 * k);
            pl[3 * k + 1] = ldg(S.pw_f + PW_REC * i + 3 * k + 1);
            pl[3 * k + 2] = ldg(S.pw_f + PW_REC * i + 3 * k + 2);
          } else {
            const size_t tt = (size_t)i + (size_t)nsol * k;
            pl[3 * k] = (R)ldg(S.pwA + tt);
            pl[3 * k + 1] = (R)ldg(S.pwB + tt);
            pl[3 * k + 2] = (R)ldg(S.pwEl + tt);
          }
        }
      };
      auto pairs = [&](R dx, R dy, R dz, const R* pw) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const R ux = dx - o[k][0], uy = dy - o[k][1], uz = dz - o[k][2];
          R ee = R(0), ev = R(0);
          // sites without LJ: nbe with A = B = 0 is nbe_spc exactly
          const R dv = (k > 0 && S.pw_coul_h)
                           ? PairMath<R>::nbe_spc(ux, uy, uz, pw[3 * k + 2], ee, false)
                           : PairMath<R>::nbe(ux, uy, uz, pw[3 * k], pw[3 * k + 1], pw[3 * k + 2], ee, ev, false);
          f[k][0] += ux * dv;
          f[k][1] += uy * dv;
          f[k][2] += uz * dv;
        }
      };
      if (n > 0) fetch(e & AL_ATOM);
      for (int t = lane; t < n; t += QNB_WAVE) {
        const R dx = (R)(px - xr0), dy = (R)(py - xr1), dz = (R)(pz - xr2);
        R pw[9];
#pragma unroll
        for (int k = 0; k < 9; k++) pw[k] = pl[k];
        const int ec = e;
        e = en;
        fetch(e & AL_ATOM);
        en = t + 2 * QNB_WAVE < n ? ldg(al + t + 2 * QNB_WAVE) : 0;
        if (!(ec & AL_SKIP)) pairs(dx, dy, dz, pw);
      }
      // groups that the row had no room for
      for (int q = lane; q < partners.n - n; q += QNB_WAVE) {
        const int ec = row_tail(S, a, partners.groups, q);
        if (ec & AL_SKIP) continue;
        fetch(ec & AL_ATOM);
        pairs((R)(px - xr0), (R)(py - xr1), (R)(pz - xr2), pl);
      }
    }
    // partner waters: lane l takes atom kb = l % 3 of water (l / 3) of the round
    if (mask & T_WW) {
      R wel[3], wA = R(0), wB = R(0), gA[3], gB[3];
      const int kb = lane % 3, pw0 = lane / 3;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        wel[k] = (R)ldg(S.wwEl + k + 3 * kb);  // receiver atom k with partner atom kb
        gA[k] = (R)ldg(S.wwA + k + 3 * kb);
        gB[k] = (R)ldg(S.wwB + k + 3 * kb);
      }
      if (S.spc && kb == 0) {
        // SPC: LJ for O-O only; the other lanes take the same path with zero
        // LJ parameters, so the k = 0 pair does not branch on kb
        wA = (R)ldg(S.wwA);
        wB = (R)ldg(S.wwB);
      }
      for (int p = nsr + pw0; p < nn; p += QNB_WAVE / 3) {
        if (lane >= 3 * (QNB_WAVE / 3)) break;
        const int b = ldg(row + p);
        const int j = nsol + sa * (b - ncs) + kb;
        const R dx = (R)(ldg(x + 3 * j) - xr0), dy = (R)(ldg(x + 3 * j + 1) - xr1), dz = (R)(ldg(x + 3 * j + 2) - xr2);
        const bool acc = want_e && owns(a, b);
        R pel = R(0), pvdw = R(0);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const R ux = dx - o[k][0], uy = dy - o[k][1], uz = dz - o[k][2];
          R dv;
          if (S.spc) {
            if (k == 0) dv = PairMath<R>::nbe(ux, uy, uz, wA, wB, wel[0], pel, pvdw, acc);
            else dv = PairMath<R>::nbe_spc(ux, uy, uz, wel[k], pel, acc);
          } else {
            dv = PairMath<R>::nbe(ux, uy, uz, gA[k], gB[k], wel[k], pel, pvdw, acc);
          }
          f[k][0] += ux * dv;
          f[k][1] += uy * dv;
          f[k][2] += uz * dv;
        }
        if (acc) {
          e_el += (double)pel;
          e_vdw += (double)pvdw;
        }
      }
    }
  }
  // Q-atom - water, receiver side (nonbond_qw_spc nonbondene.f90:5658-5767;
  // nonbond_qw 5339-5418): lane per Q-atom, the water's three sites in turn
  // (an SPC hydrogen takes the Coulomb-only nbe_qspc, nonbonded.f90:226-243)
  if ((mask & T_QW) && nq > 0 && ldg(S.qw_in + (a - ncs))) {
    for (int iq = lane; iq < nq; iq += QNB_WAVE) {
      const int q = ldg(S.iqseq + iq);
      const R qx = (R)(ldg(x + 3 * q) - xr0), qy = (R)(ldg(x + 3 * q + 1) - xr1), qz = (R)(ldg(x + 3 * q + 2) - xr2);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const R ux = qx - o[k][0], uy = qy - o[k][1], uz = qz - o[k][2];
        R r2, r;
        rinv(norm2(ux, uy, uz), r2, r);
        const R dvs = k == 0 || !S.spc
                          ? qx_states<R, NS>(S, r2, r, ns, eq, want_e, [&](int s) { return qw_par<R>(S, iq, k, s); })
                          : qspc_states<R, NS>(S, r2, r, ns, eq, want_e, [&](int s) { return qw_el<R>(S, iq, k, s); });
        f[k][0] += ux * dvs;
        f[k][1] += uy * dvs;
        f[k][2] += uz * dvs;
      }
    }
  }
  {
    // the nine force components in one transposed reduction; component c of
    // atom k is value 3k + c, i.e. d[3 * ra + j]
    R fv[9];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int c = 0; c < 3; c++) fv[3 * k + c] = f[k][c];
    const double fs = wave_sum_tr(fv, lane);
    if (wave_sum_tr_writer<9>(lane)) d[3 * ra + wave_sum_tr_index<9>(lane)] = -fs;
  }
  if (!want_e) return;
  // ww energies, then each state's qw el and vdW
  double part[2 + 2 * NS];
  int slot[2 + 2 * NS];
  part[0] = e_el, slot[0] = E_WW_EL;
  part[1] = e_vdw, slot[1] = E_WW_VDW;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    part[2 + 2 * s] = eq[2 * s], slot[2 + 2 * s] = E_Q0 + 6 * s + 4;
    part[3 + 2 * s] = eq[2 * s + 1], slot[3 + 2 * s] = E_Q0 + 6 * s + 5;
  }
  store_energy_record<2 + 2 * NS>(S.epart + (size_t)a * QNB_NE, wave_sum_tr(part, lane), slot, lane);
}

template <typename R, int NS, bool E>
__global__ __launch_bounds__(64 * FC_WPB) void k_wforces(const DevSys* __restrict__ systems, uint32_t mask,
                                                         int imap, int nb, int ninst) {
  int inst, blk;
  if (!map_block(imap, nb, ninst, inst, blk)) return;
  const DevSys& S = systems[inst];
  const int wib = threadIdx.x / QNB_WAVE;
  const int a = __builtin_amdgcn_readfirstlane(S.ncgp_solute + blk * (int)(blockDim.x / QNB_WAVE) + wib);
  if (a < S.ncgp) water_receiver<R, NS, E>(S, mask, a);
}

// ---------------------------------------------------------------------------
// Receivers of a solvent other than 3-site water (any solv_atom up to 64):
// one wavefront per solvent molecule a; lane l takes receiver atom
// k = l % sa and, with M = 64 / sa lanes per atom, every M-th partner atom
// from m = l / sa on, in the partner order of the reference's loops:
//  * solute partner groups (the row's prefix): their non-Q atoms with the pw
//    parameters (nonbond_pw, nonbondene.f90:4856-4916; energy counted on the
//    solute side);
//  * partner molecules: the sa x sa atom pairs with ww_precomp
//    (nonbond_ww 5509-5573), energy on the owner side of the pair;
//  * the Q-atoms (receiver side of nonbond_qw 5339-5418);
//  * the pairs inside the molecule (nonbond_solvent_internal 6082-6154),
//    excluded molecules included: the lane of each end atom evaluates the
//    pair, the first end counts its energy.
// The lanes of an atom add their FP64 partials in lane order (LDS); writes d
// of the molecule's atoms and the wave's ww and qw energy partials on the
// sampled steps.
template <typename R, int NS>
__device__ __forceinline__ void solvent_receiver(const DevSys& S, uint32_t mask, int a, double (*s_f)[3]) {
  const int lane = threadIdx.x % QNB_WAVE;
  const int sa = S.sa, M = QNB_WAVE / sa;
  const int k = lane % sa, m = lane / sa;
  const bool active = m < M;
  const double* __restrict__ x = S.x;
  const int nsol = S.nat_solute, ncs = S.ncgp_solute, nq = S.nqat, ns = S.nstates;
  const int base = nsol + sa * (a - ncs), ia = base + k;
  const bool aexcl = ldg(S.excl + base);
  const bool want_e = want_energies(S);
  const int nn = uni(min(ldg(S.nnbr + a), S.cap));
  const int* __restrict__ row = S.nbr + (size_t)a * S.cap;
  const double xi0 = ldg(x + 3 * ia), xi1 = ldg(x + 3 * ia + 1), xi2 = ldg(x + 3 * ia + 2);
  double f[3] = {0.0, 0.0, 0.0};
  double e_el = 0.0, e_vdw = 0.0;
  double eq[2 * NS];
#pragma unroll
  for (int c = 0; c < 2 * NS; c++) eq[c] = 0.0;
  if (active && !aexcl) {
    for (int p = 0; p < nn; p++) {
      const int b = ldg(row + p);
      if (b < ncs) {
        if (!(mask & T_PW)) continue;
        const int t1 = ldg(S.glast + b);
        for (int t = ldg(S.gfirst + b) + m; t <= t1; t += M) {
          const int j = ldg(S.cgpatom + t);
          if (ldg(S.iqatom + j) != 0) continue;
          const R ux = (R)(ldg(x + 3 * j) - xi0), uy = (R)(ldg(x + 3 * j + 1) - xi1),
                  uz = (R)(ldg(x + 3 * j + 2) - xi2);
          const size_t tt = (size_t)j + (size_t)nsol * k;
          R ee = R(0), ev = R(0);
          const R dv = PairMath<R>::nbe(ux, uy, uz, (R)ldg(S.pwA + tt), (R)ldg(S.pwB + tt), (R)ldg(S.pwEl + tt),
                                        ee, ev, false);
          f[0] += (double)(ux * dv);
          f[1] += (double)(uy * dv);
          f[2] += (double)(uz * dv);
        }
      } else {
        if (!(mask & T_WW)) continue;
        const bool own = want_e && owns(a, b);
        const int jb = nsol + sa * (b - ncs);
        for (int kb = m; kb < sa; kb += M) {
          const int j = jb + kb;
          const R ux = (R)(ldg(x + 3 * j) - xi0), uy = (R)(ldg(x + 3 * j + 1) - xi1),
                  uz = (R)(ldg(x + 3 * j + 2) - xi2);
          const int t = k + kb * sa;
          R ee = R(0), ev = R(0);
          const R dv = (S.spc && (k != 0 || kb != 0))
                           ? PairMath<R>::nbe_spc(ux, uy, uz, (R)ldg(S.wwEl + t), ee, own)
                           : PairMath<R>::nbe(ux, uy, uz, (R)ldg(S.wwA + t), (R)ldg(S.wwB + t), (R)ldg(S.wwEl + t),
                                              ee, ev, own);
          f[0] += (double)(ux * dv);
          f[1] += (double)(uy * dv);
          f[2] += (double)(uz * dv);
          if (own) {
            e_el += (double)ee;
            e_vdw += (double)ev;
          }
        }
      }
    }
    if ((mask & T_QW) && nq > 0 && ldg(S.qw_in + (a - ncs))) {
      for (int iq = m; iq < nq; iq += M) {
        const int q = ldg(S.iqseq + iq);
        const R ux = (R)(ldg(x + 3 * q) - xi0), uy = (R)(ldg(x + 3 * q + 1) - xi1), uz = (R)(ldg(x + 3 * q + 2) - xi2);
        R r2, r;
        rinv(norm2(ux, uy, uz), r2, r);
        const R dvs = k == 0 || !S.spc
                          ? qx_states<R, NS>(S, r2, r, ns, eq, want_e, [&](int s) { return qw_par<R>(S, iq, k, s); })
                          : qspc_states<R, NS>(S, r2, r, ns, eq, want_e, [&](int s) { return qw_el<R>(S, iq, k, s); });
        f[0] += (double)(ux * dvs);
        f[1] += (double)(uy * dvs);
        f[2] += (double)(uz * dvs);
      }
    }
  }
  if ((mask & T_SINT) && S.n_sint > 0 && active && m == 0) {
    for (int ip = 0; ip < S.n_sint; ip++) {
      const int oa = ldg(S.sint_ij + 2 * ip), ob = ldg(S.sint_ij + 2 * ip + 1);
      if (oa != k && ob != k) continue;
      const int i0 = base + oa, i1 = base + ob;
      const R vx = (R)(ldg(x + 3 * i1) - ldg(x + 3 * i0)), vy = (R)(ldg(x + 3 * i1 + 1) - ldg(x + 3 * i0 + 1)),
              vz = (R)(ldg(x + 3 * i1 + 2) - ldg(x + 3 * i0 + 2));
      R r2, r;
      rinv(vx * vx + vy * vy + vz * vz, r2, r);
      const R r6 = r2 * r2 * r2, r12 = r6 * r6;
      const R Vel = (R)ldg(S.sint_par + 3 * ip + 2) * r, Va = (R)ldg(S.sint_par + 3 * ip) * r12,
              Vb = (R)ldg(S.sint_par + 3 * ip + 1) * r6;
      const R dv = r2 * (-Vel) + r2 * (R(-12) * Va + R(6) * Vb);
      // d(ia) -= v dv, d(ib) += v dv; the lane holds the negative gradient
      // part f (d = -f), as for the pairs above (u = partner - receiver)
      const double sgn = oa == k ? 1.0 : -1.0;
      if (oa == k && ob == k) continue;  // a self pair carries no force
      f[0] += sgn * (double)(vx * dv);
      f[1] += sgn * (double)(vy * dv);
      f[2] += sgn * (double)(vz * dv);
      if (want_e && oa == k) {
        e_el += (double)Vel;
        e_vdw += (double)(Va - Vb);
      }
    }
  }
  s_f[lane][0] = f[0];
  s_f[lane][1] = f[1];
  s_f[lane][2] = f[2];
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  if (lane < sa) {
    double t0 = 0.0, t1 = 0.0, t2 = 0.0;
    for (int mm = 0; mm < M; mm++) {
      t0 += s_f[lane + sa * mm][0];
      t1 += s_f[lane + sa * mm][1];
      t2 += s_f[lane + sa * mm][2];
    }
    const auto d = gpm(S.d);
    d[3 * ia] = -t0;
    d[3 * ia + 1] = -t1;
    d[3 * ia + 2] = -t2;
  }
  if (!want_e) return;
  double part[2 + 2 * NS];
  int slot[2 + 2 * NS];
  part[0] = e_el, slot[0] = E_WW_EL;
  part[1] = e_vdw, slot[1] = E_WW_VDW;
#pragma unroll
  for (int st = 0; st < NS; st++) {
    part[2 + 2 * st] = eq[2 * st], slot[2 + 2 * st] = E_Q0 + 6 * st + 4;
    part[3 + 2 * st] = eq[2 * st + 1], slot[3 + 2 * st] = E_Q0 + 6 * st + 5;
  }
  store_energy_record<2 + 2 * NS>(S.epart + (size_t)a * QNB_NE, wave_sum_tr(part, lane), slot, lane);
}

template <typename R, int NS>
__global__ __launch_bounds__(64 * FC_WPB) void k_gforces(const DevSys* __restrict__ systems, uint32_t mask,
                                                         int imap, int nb, int ninst) {
  int inst, blk;
  if (!map_block(imap, nb, ninst, inst, blk)) return;
  const DevSys& S = systems[inst];
  const int wib = threadIdx.x / QNB_WAVE;
  const int a = __builtin_amdgcn_readfirstlane(S.ncgp_solute + blk * (int)(blockDim.x / QNB_WAVE) + wib);
  if (a >= S.ncgp) return;
  __shared__ double s_f[FC_WPB][QNB_WAVE][3];
  solvent_receiver<R, NS>(S, mask, a, s_f[wib]);
}

// ---------------------------------------------------------------------------
// Per-atom terms after the pair kernels, one thread per atom: the LRF Taylor
// term (lrf_taylor, nonbondene.f90:507-571) of every non-Q, non-excluded
// atom and the SCAAS radial restraint (restrain_solvent, 6466-6544) of the
// solvent atoms radial_source names; adds to d (store_atom_gradient).  On the
// sampled steps the atom's two energies go to eatom[2i], eatom[2i+1] for the
// fixed-order reduction.
__global__ __launch_bounds__(256) void k_atom_terms(const DevSys* __restrict__ systems, uint32_t mask,
                                                    const double* __restrict__ tfree, int rows) {
  const DevSys& S = systems[blockIdx.y];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= S.natom) return;
  double f[3] = {0.0, 0.0, 0.0};
  double el = 0.0, er = 0.0;
  if ((mask & T_LRF) && S.use_lrf && !ldg(S.excl + i) && ldg(S.iqatom + i) == 0) lrf_taylor_atom(S, i, ldg(S.atom_group + i), f, el);
  const int src = (mask & T_RAD) ? radial_source(S, i) : -1;
  if (src >= 0) {
    const double T = tfree[blockIdx.y];
    const double shift = S.fk_wsphere != 0.0 ? sqrt(S.Boltz * T / S.fk_wsphere) : 0.0;
    radial_restraint(S, src, shift, f, er);
  }
  add_qrows(S, i, rows, f);
  store_atom_gradient(S, i, f);
  if (want_energies(S)) {
    stg(S.eatom + 2 * i, el);
    stg(S.eatom + 2 * i + 1, er);
  }
}

// ---------------------------------------------------------------------------
// Q-atom side of the Q-water and Q-solute pairs: wave = (Q-atom iq, every
// chunks-th 64 of its partners from 64 ch on); the wave's sum is added with
// atomics (a few per Q-atom) to the Q-atom's gradient, or, with rows, to its
// row of S.dq (launches that run beside or inside the solute receivers' one,
// which store the same atoms' gradients; the per-atom pass adds dq).
template <typename R, int NS>
__device__ __forceinline__ void qatom_side(const DevSys& S, uint32_t mask, int iq, int ch, int chunks, int rows) {
  const int lane = threadIdx.x % QNB_WAVE;
  const int nqw = ldg(S.nq_lists + 0), nqp = ldg(S.nq_lists + 1);
  const int nw_ch = (mask & T_QW) ? (nqw + QNB_WAVE - 1) / QNB_WAVE : 0;
  const int np_ch = (mask & T_QP) ? (nqp + QNB_WAVE - 1) / QNB_WAVE : 0;
  const double* __restrict__ x = S.x;
  const int i = ldg(S.iqseq + iq);
  const int nq = S.nqat, ns = S.nstates, sa = S.sa;
  const double xi0 = ldg(x + 3 * i), xi1 = ldg(x + 3 * i + 1), xi2 = ldg(x + 3 * i + 2);
  // per-lane partials in R (a lane takes one partner per chunk), summed over
  // the wave in FP64
  R f[3] = {R(0), R(0), R(0)};
  double dummy[2 * NS];
  const R *qtA = qp_tab<R>(S.qpA, S.qpA_f), *qtB = qp_tab<R>(S.qpB, S.qpB_f);
  const R *qtE = qp_tab<R>(S.qpEl, S.qpEl_f), *qtS = qp_tab<R>(S.qpSc, S.qpSc_f);
  for (int c = ch; c < nw_ch + np_ch; c += chunks) {
    const int p = c * QNB_WAVE + lane;
    if (c < nw_ch) {
      if (p >= nqw) continue;
      const int o = S.nat_solute + sa * ldg(S.qw_list + p);
      for (int k = 0; k < sa; k++) {
        const int j = o + k;
        const double ux = ldg(x + 3 * j) - xi0, uy = ldg(x + 3 * j + 1) - xi1, uz = ldg(x + 3 * j + 2) - xi2;
        const R rux = (R)ux, ruy = (R)uy, ruz = (R)uz;
        R r2, r;
        rinv(norm2(rux, ruy, ruz), r2, r);
        const R dvs = k == 0 || !S.spc
                          ? qx_states<R, NS>(S, r2, r, ns, dummy, false, [&](int s) { return qw_par<R>(S, iq, k, s); })
                          : qspc_states<R, NS>(S, r2, r, ns, dummy, false, [&](int s) { return qw_el<R>(S, iq, k, s); });
        f[0] -= rux * dvs;
        f[1] -= ruy * dvs;
        f[2] -= ruz * dvs;
      }
    } else {
      const int pp = p - nw_ch * QNB_WAVE;
      if (pp >= nqp) continue;
      const int j = ldg(S.qp_list + pp);
      const double ux = ldg(x + 3 * j) - xi0, uy = ldg(x + 3 * j + 1) - xi1, uz = ldg(x + 3 * j + 2) - xi2;
      const R rux = (R)ux, ruy = (R)uy, ruz = (R)uz;
      R r2, r;
      rinv(norm2(rux, ruy, ruz), r2, r);
      auto par = [&](int s) {
        const size_t t = (size_t)j + (size_t)S.nat_solute * ((size_t)iq + (size_t)nq * s);
        return QPar<R>{ldg(qtA + t), ldg(qtB + t), ldg(qtE + t), ldg(qtS + t)};
      };
      if constexpr (sizeof(R) == 8) {
        const R dvs = qx_states<R, NS>(S, r2, r, ns, dummy, false, par);
        f[0] -= rux * dvs;
        f[1] -= ruy * dvs;
        f[2] -= ruz * dvs;
      } else {
        const R r6 = r2 * r2 * r2;
#pragma unroll
        for (int s = 0; s < NS; s++) {
          if (s >= ns) break;
          const QPar<R> p = par(s);
          const R dv = PairMath<R>::nbe_qx(r2, r, r6, p.A, p.B, p.q, p.sc, (R)S.lambda[s], dummy[0], dummy[1], false);
          f[0] -= rux * dv;
          f[1] -= ruy * dv;
          f[2] -= ruz * dv;
        }
      }
    }
  }
  const double fs = wave_sum_tr(f, lane);
  const int c = wave_sum_tr_index<3>(lane);
  if (wave_sum_tr_writer<3>(lane) && fs != 0.0)
    unsafeAtomicAdd(rows ? S.dq + 3 * iq + c : S.d + 3 * i + c, fs);
}

template <typename R, int NS>
__global__ __launch_bounds__(256) void k_qforces(const DevSys* __restrict__ systems, uint32_t mask,
                                                 int chunks_per_q, int rows) {
  const DevSys& S = systems[blockIdx.y];
  // block x runs on XCD x % 8 and takes Q-atom iq = x % 8 + 8 * (x / 8 / bq),
  // chunks (x / 8 % bq) * W .. + W - 1 (W waves per block, bq blocks per
  // Q-atom): an XCD serves only the Q-atoms iq = its index mod 8, so the rows
  // of the Q tables it reads stay in its L2 across the instances
  const int W = blockDim.x / QNB_WAVE, bq = (chunks_per_q + W - 1) / W;
  const int m = blockIdx.x / 8;
  const int iq = blockIdx.x % 8 + 8 * (m / bq), ch = uni((m % bq) * W + threadIdx.x / QNB_WAVE);
  if (iq < S.nqat && ch < chunks_per_q) qatom_side<R, NS>(S, mask, iq, ch, chunks_per_q, rows);
}

// ---------------------------------------------------------------------------
// Static Q-Q (nonbond_qq, nonbondene.f90:5013-5082, pair kernel nbe_qq
// nonbonded.f90:111-150) and Q-bonded-neighbour (nonbond_qqp, 5085-5153)
// lists: a wavefront per atom of the lists (entity) whose lanes evaluate the
// pairs the atom belongs to; the wave's sum goes to the atom's gradient once (no atomics; each pair is
// evaluated from both sides).  A pair's energy is counted by its first atom;
// per state the energies are summed per wave and then over the waves in
// order.
template <int NS>
__device__ __forceinline__ void qq_add(double (&eq)[NS][4], int s, int c0, double v0, double v1) {
#pragma unroll
  for (int k = 0; k < NS; k++)
    if (k == s) {
      eq[k][c0] += v0;
      eq[k][c0 + 1] += v1;
    }
}

// Wave `wave` takes entities wave, wave + stride, ..., its lanes the entity's
// pairs; the block's energies go to record `slot`.  rows: the sums go to the
// entities' rows of S.dqq (stored, not added), which the per-atom pass adds.
template <typename R, int NS>
__device__ __forceinline__ void qq_pairs(const DevSys& S, uint32_t mask, int wave, int stride, int slot, int rows,
                                         double* red) {
  const int lane = threadIdx.x % QNB_WAVE, wid = threadIdx.x / QNB_WAVE;
  const auto x = gp(S.x);
  const auto d = gpm(S.d);
  const bool want_e = want_energies(S);
  double eq[NS][4];
#pragma unroll
  for (int s = 0; s < NS; s++) eq[s][0] = eq[s][1] = eq[s][2] = eq[s][3] = 0.0;
  for (int e = wave; e < S.nqe; e += stride) {
    const int me = ldg(S.qe_atom + e);
    double f[3] = {0.0, 0.0, 0.0};
    for (int it = ldg(S.qe_off + e) + lane, end = ldg(S.qe_off + e + 1); it < end; it += QNB_WAVE) {
      const int i = ldg(S.qe_item + 4 * it), j = ldg(S.qe_item + 4 * it + 1), p = ldg(S.qe_item + 4 * it + 2);
      const int w = ldg(S.qe_item + 4 * it + 3), s = w >> 2, side = w & 1;
      const bool qq = (w & 2) == 0;
      if (!(mask & (qq ? T_QQ : T_QQP))) continue;
      const double* pr = (qq ? S.qq_par : S.qqp_par) + 4 * p;
      const double ux = x[3 * j] - x[3 * i], uy = x[3 * j + 1] - x[3 * i + 1], uz = x[3 * j + 2] - x[3 * i + 2];
      const R rux = (R)ux, ruy = (R)uy, ruz = (R)uz;
      R r2, r;
      rinv(norm2(rux, ruy, ruz), r2, r);
      const R pA = (R)ldg(pr), pB = (R)ldg(pr + 1), pel = (R)ldg(pr + 2), psc = (R)ldg(pr + 3);
      const R lam = (R)S.lambda[s];
      R dv;
      if (qq) {
        R r6d = r2 * r2 * r2;
        R r6_hc = recip(r6d);
        R r6 = recip(r6_hc + psc);
        R r12 = r6 * r6;
        R Vel = pel * r, Va, Vb;
        if (ldg(S.qq_soft + p)) {
          Vb = R(0);
          Va = pA * exp(-pB / r);
          dv = r2 * (-Vel - pB * Va / r) * lam;
        } else {
          Va = pA * r12;
          Vb = pB * r6;
          dv = r2 * (-Vel - (R(12) * Va - R(6) * Vb) * r6 * r6_hc) * lam;
        }
        if (want_e && side == 0) qq_add<NS>(eq, s, 0, (double)Vel, (double)Va - (double)Vb);
      } else {
        double el = 0.0, vdw = 0.0;
        dv = PairMath<R>::nbe_qx(r2, r, r2 * r2 * r2, pA, pB, pel, psc, lam, el, vdw, want_e && side == 0);
        if (want_e && side == 0) qq_add<NS>(eq, s, 2, el, vdw);
      }
      // the pair's gradient is -u dv on its first atom, +u dv on the second
      const double sg = side == 0 ? -1.0 : 1.0;
      f[0] += sg * (double)(rux * dv);
      f[1] += sg * (double)(ruy * dv);
      f[2] += sg * (double)(ruz * dv);
    }
    f[0] = wave_sum(f[0]);
    f[1] = wave_sum(f[1]);
    f[2] = wave_sum(f[2]);
    if (lane == 0) {
      if (rows) {
        const auto o = gpm(S.dqq) + 3 * e;
        o[0] = f[0];
        o[1] = f[1];
        o[2] = f[2];
      } else {
        d[3 * me] += f[0];
        d[3 * me + 1] += f[1];
        d[3 * me + 2] += f[2];
      }
    }
  }
  if (!want_e) return;
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const double v = wave_sum(eq[s][c]);
      if (lane == 0) red[4 * (wid * NS + s) + c] = v;
    }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const int nw = blockDim.x / QNB_WAVE;
  double* ep = S.epart + (size_t)slot * QNB_NE;
  for (int k = 0; k < QNB_NE; k++) ep[k] = 0.0;
  for (int s = 0; s < NS; s++)
    for (int c = 0; c < 4; c++) {
      double v = 0.0;
      for (int w = 0; w < nw; w++) v += red[4 * (w * NS + s) + c];
      ep[E_Q0 + 6 * s + c] = v;
    }
}

template <typename R, int NS>
__global__ __launch_bounds__(QQ_THREADS) void k_qq(const DevSys* __restrict__ systems, uint32_t mask) {
  const DevSys& S = systems[blockIdx.x];
  constexpr int NW = QQ_THREADS / QNB_WAVE;
  __shared__ double red[NW * NS * 4];
  qq_pairs<R, NS>(S, mask, threadIdx.x / QNB_WAVE, NW, S.ncgp, 0, red);
}

// ---------------------------------------------------------------------------
// SCAAS polarisation restraint (watpol, nonbondene.f90:6548-6746,
// md = .true.): the angles and shells (watpol_theta), the ranks and forces
// (pol_forces, blocks of 64 members of one shell), the per-shell sums
// (watpol_finish).  The reference's per-shell selection sort by theta is a
// stable ascending sort; here each member's rank is counted directly (ties
// broken by water index, as the selection sort does).
//
// Dipole and radial directions of the molecule whose first atom is i
// (nonbondene.f90:6572-6604): a 3-site solvent takes H1 + H2 - 2 O and the
// radial vector of O; any other the charge-weighted sum of its positions
// (charges of the first solvent molecule) and its centroid's radial vector.
__device__ __forceinline__ void wat_vectors(const DevSys& S, int i, double* rmu, double& rm, double* rcu,
                                            double& rc) {
  const double* x = S.x;
  const int sa = S.sa;
  double m[3], v[3];
  if (sa == 3) {
    for (int c = 0; c < 3; c++) m[c] = (x[3 * (i + 1) + c] + x[3 * (i + 2) + c]) - x[3 * i + c] * 2.0;
    for (int c = 0; c < 3; c++) v[c] = x[3 * i + c] - S.xw[c];
  } else {
    const double* chg = S.crg + S.nat_solute;
    double g[3] = {0.0, 0.0, 0.0};
    m[0] = m[1] = m[2] = 0.0;
    for (int k = 0; k < sa; k++) {
      const double q = ldg(chg + k);
      for (int c = 0; c < 3; c++) {
        g[c] = g[c] + x[3 * (i + k) + c];
        m[c] = m[c] + x[3 * (i + k) + c] * q;
      }
    }
    for (int c = 0; c < 3; c++) v[c] = g[c] / (double)sa - S.xw[c];
  }
  rm = sqrt(m[0] * m[0] + m[1] * m[1] + m[2] * m[2]);
  for (int c = 0; c < 3; c++) rmu[c] = m[c] / rm;
  rc = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  for (int c = 0; c < 3; c++) rcu[c] = v[c] / rc;
}

// Phase 1, one thread per water: theta and shell (-1: inside the innermost
// shell, or excluded); the members of each shell are appended to its list
// (slot order is immaterial: ranks are counted by value).  Block 0 first
// applies the theta_corr feedback of the steps that are multiples of itdis
// (nonbondene.f90:6653-6666).  The shell counts start at zero (set at
// creation and cleared by watpol_finish).
__device__ __forceinline__ void watpol_theta(const DevSys& S, int blk, int step) {
  if (!has_pol(S)) return;
  const int t = threadIdx.x, nsh = S.nshell, nw = S.nwat;
  if (blk == 0 && t == 0) {
    double* st = S.sh_state;  // theta_corr[8], avtheta[8], avn_insh[8]
    const int itd = (int)llround(S.itdis);
    if (step > 0 && itd > 0 && step % itd == 0) {
      for (int is = 0; is < nsh; is++) {
        st[QNB_MAXSH + is] = st[QNB_MAXSH + is] / S.itdis;
        st[2 * QNB_MAXSH + is] = st[2 * QNB_MAXSH + is] / S.itdis;
        st[is] = st[is] + st[QNB_MAXSH + is] - acos(S.sh_cstb[is]);
        st[QNB_MAXSH + is] = 0.0;
        st[2 * QNB_MAXSH + is] = 0.0;
      }
    }
  }
  const int w = blk * WP_THREADS + t;
  if (w >= nw) return;
  const int i = S.nat_solute + S.sa * w;
  int sh = -1;
  double th = 0.0;
  if (!ldg(S.excl + i)) {
    double rmu[3], rcu[3], rm, rc;
    wat_vectors(S, i, rmu, rm, rcu, rc);
    double scp = rmu[0] * rcu[0] + rmu[1] * rcu[1] + rmu[2] * rcu[2];
    scp = scp > 1.0 ? 1.0 : (scp < -1.0 ? -1.0 : scp);
    th = acos(scp);
    if (rc > S.sh_rout[nsh - 1] - S.sh_dr[nsh - 1]) {
      int is;
      for (is = nsh - 1; is >= 1; is--)
        if (rc <= S.sh_rout[is]) break;
      if (is < 1) is = 0;
      sh = is;
    }
  }
  // append to the shell lists with one atomic per (wave, shell): the lanes of
  // a shell take consecutive places (ranks are counted by (theta, water index),
  // so the order of appending does not matter)
  const int lane = t % QNB_WAVE;
  int pending = sh;
  for (;;) {
    const uint64_t act = __ballot(pending >= 0);
    if (act == 0) break;
    const int lead = __ffsll((unsigned long long)act) - 1;
    const int s0 = __shfl(pending, lead, QNB_WAVE);
    const uint64_t m = __ballot(pending == s0);
    int base = 0;
    if (lane == lead) base = atomicAdd(S.sh_n + s0, __popcll(m));
    base = __shfl(base, lead, QNB_WAVE);
    if (pending == s0) {
      const int pos = base + __popcll(m & ((1ull << lane) - 1ull));
      stg(S.sh_list + (size_t)s0 * nw + pos, w);
      stg(S.sh_lth + (size_t)s0 * nw + pos, th);
      pending = -1;
    }
  }
}

__global__ __launch_bounds__(WP_THREADS) void k_watpol_theta(const DevSys* __restrict__ systems,
                                                             const int* __restrict__ istep) {
  watpol_theta(systems[blockIdx.y], blockIdx.x, istep[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// All force kernels of a step in one launch, for launches too small to fill
// the chip (small_launch): blocks of four waves take, in this order, one
// solute receiver (its row split over the four waves), four solvent receivers,
// four chunks of a Q-atom's partners, four Q-Q entities, or WP_THREADS waters'
// polarisation angles.  Everything they read is there before the launch and
// they write disjoint rows (the Q kernels' sums go to dq and dqq), so no order
// between them is needed.  What bounds such a step is the latency of each
// launch and of one wave walking one row: as launches of their own on two
// streams a step of one 3,342-atom window took 78 us and one of an FP64 window
// of 11,056 atoms 122 us, with this kernel 62 and 111.
template <typename R, int NS, bool E>
__global__ __launch_bounds__(256) void k_forces_small(const DevSys* __restrict__ systems, uint32_t mask,
                                                                  SmallGrid G, const int* __restrict__ istep) {
  const DevSys& S = systems[blockIdx.y];
  const int wib = threadIdx.x / QNB_WAVE;
  extern __shared__ __align__(16) unsigned char small_smem[];
  int b = blockIdx.x;
  if (b < G.solute) {
    __shared__ double comb[4][QNB_WAVE];
    if (b < S.ncgp_solute)
      solute_receiver<R, NS, E, true>(S, mask, b, uni(wib), 4, small_smem + (size_t)wib * so_wave_bytes<R>(), comb);
    return;
  }
  b -= G.solute;
  if (b < G.solvent) {
    const int a = __builtin_amdgcn_readfirstlane(S.ncgp_solute + 4 * b + wib);
    if (a >= S.ncgp) return;
    if (S.sa == 3)
      water_receiver<R, NS, E>(S, mask, a);
    else
      solvent_receiver<R, NS>(S, mask, a, reinterpret_cast<double(*)[3]>(small_smem) + QNB_WAVE * wib);
    return;
  }
  b -= G.solvent;
  if (b < G.qside) {
    const int bq = (G.qchunks + 3) / 4, iq = b / bq, ch = uni(4 * (b % bq) + wib);
    if (iq < S.nqat && ch < G.qchunks) qatom_side<R, NS>(S, mask, iq, ch, G.qchunks, 1);
    return;
  }
  b -= G.qside;
  if (b < G.qq) {
    if (b < qq_slots(S))
      qq_pairs<R, NS>(S, mask, 4 * b + wib, 4 * qq_slots(S), S.ncgp + b, 1, reinterpret_cast<double*>(small_smem));
    return;
  }
  watpol_theta(S, b - G.qq, istep[blockIdx.y]);
}

// Phase 2, WP_WATERS members of one shell per block, WAVES waves on the same
// members: each member's rank in its shell's stable ascending order of theta
// (the reference's selection sort; ties by water index) is the number of
// members before it, counted against the shell's list staged in LDS, an equal
// part of it per wave (equal angles, which only coincidence brings, in a second
// pass of the members concerned; an angle that is not a number, of a water
// without a dipole direction, counts as the largest, so every member has a rank
// of its own and its NaN reaches the sums); wave 0 then forms the target angle from the
// rank, the restraint energy and the forces (adds to d), and writes energy and
// theta at the member's rank (wp_rank), so the sums over a shell do not depend
// on the order the angle kernel appended its members in.  Counting is n^2
// compares, but over all blocks it is a few microseconds of latency at n = 700,
// where one block per shell running a bitonic network over its 55 steps took
// 14-23 us and was a launch of its own.  Blocks take the members of one shell,
// not the waters in index order, so a wave counts one list: the index order,
// where every block holds every shell, cost 51 windows of 2,352 waters 22 us
// per step more.
// WAVES: a small step waits for this kernel, so 16 waves share a count (1,110
// waters 10.5 -> 8.2 us, 2,352 waters 17 -> 8.5 us against 4); beside full
// force kernels, whose blocks leave four wave slots sooner than 16, 4 do.
__device__ __forceinline__ double pol_key(double theta) { return __builtin_fmin(theta, __builtin_inf()); }
template <int WAVES>
__device__ __forceinline__ void pol_forces(const DevSys& S) {
  const int lane = threadIdx.x % QNB_WAVE, wid = threadIdx.x / QNB_WAVE;
  if (!has_pol(S)) return;
  const int nsh = S.nshell, nw = S.nwat;
  // block x of the system takes members 64 x' .. of shell sh, the blocks of
  // the shells laid end to end
  int cnt[QNB_MAXSH];
#pragma unroll
  for (int is = 0; is < QNB_MAXSH; is++) cnt[is] = is < nsh ? ldg(S.sh_n + is) : 0;
  int sh = -1, xb = blockIdx.x, n = 0;
#pragma unroll
  for (int is = 0; is < QNB_MAXSH; is++) {
    const int nb = (cnt[is] + WP_WATERS - 1) / WP_WATERS;
    if (sh < 0) {
      if (xb < nb) sh = is, n = cnt[is];
      else xb -= nb;
    }
  }
  if (sh < 0) return;
  __shared__ double c_th[WP_CHUNK];
  __shared__ int s_cnt[WAVES][QNB_WAVE], s_eq[WAVES][QNB_WAVE];
  const int m = xb * WP_WATERS + lane;
  const double* L_th = S.sh_lth + (size_t)sh * nw;
  const int* L_w = S.sh_list + (size_t)sh * nw;
  const int w = m < n ? ldg(L_w + m) : 0;
  const double th = m < n ? ldg(L_th + m) : 0.0, key = pol_key(th);
  int before = 0, equal = 0;
  for (int k0 = 0; k0 < n; k0 += WP_CHUNK) {
    const int nk = min(WP_CHUNK, n - k0);
    __syncthreads();
    for (int k = threadIdx.x; k < nk; k += blockDim.x) c_th[k] = pol_key(ldg(L_th + k0 + k));
    __syncthreads();
    const int q0 = nk * wid / WAVES, q1 = nk * (wid + 1) / WAVES;
#pragma unroll 8
    for (int k = q0; k < q1; k++) {
      before += c_th[k] < key;
      equal += c_th[k] == key;
    }
  }
  s_cnt[wid][lane] = before;
  s_eq[wid][lane] = equal;
  __syncthreads();
  if (wid != 0 || m >= n) return;
  int il = 1;
  equal = 0;
  for (int u = 0; u < WAVES; u++) {
    il += s_cnt[u][lane];
    equal += s_eq[u][lane];
  }
  if (equal > 1)  // members with the same angle: by water index
    for (int k = 0; k < n; k++) il += pol_key(ldg(L_th + k)) == key && ldg(L_w + k) < w;
  const double pi = 3.141592653589793;
  const double tc = S.sh_state[sh];
  double arg = 1.0 + (1.0 - 2.0 * (double)il) / (double)n;
  double th0 = acos(arg);
  // sin(acos(c)) = sqrt((1 - c)(1 + c)), here and below
  th0 = th0 - 3.0 * sqrt((1.0 - arg) * (1.0 + arg)) * S.sh_cstb[sh] / 2.0;
  if (th0 < 0.0) th0 = 0.0;
  if (th0 > pi) th0 = pi;
  const double dth = th - th0 + tc;
  const double epol = 0.5 * S.fkwpol * (dth * dth);
  const double dv = S.fkwpol * dth;
  const int i = S.nat_solute + S.sa * w;
  double rmu[3], rcu[3], rm, rc;
  wat_vectors(S, i, rmu, rm, rcu, rc);
  double scp = rmu[0] * rcu[0] + rmu[1] * rcu[1] + rmu[2] * rcu[2];
  scp = scp > 1.0 ? 1.0 : (scp < -1.0 ? -1.0 : scp);
  double f0 = sqrt((1.0 - scp) * (1.0 + scp));
  if (fabs(f0) < 1.0e-10) f0 = 1.0e-10;
  f0 = -1.0 / f0;
  f0 = dv * f0;
  const auto d = gpm(S.d);
  for (int c = 0; c < 3; c++) {
    const double av = rcu[c] - rmu[c] * scp;
    const double f1 = (av * (-2.0)) / rm, f3 = av / rm, f2 = (rmu[c] - rcu[c] * scp) / rc;
    d[3 * i + c] += (f1 + f2) * f0;
    for (int k = 1; k < S.sa; k++) d[3 * (i + k) + c] += f3 * f0;
  }
  double* o = S.wp_rank + 2 * ((size_t)sh * nw + il - 1);
  stg(o, epol);
  stg(o + 1, th);
}

// the bonded terms of atom i into its rows, for k_integrate
__device__ __forceinline__ void bonded_rows(const DevSys& S, int i) {
  if (i >= S.nbat) return;
  double f[3] = {0.0, 0.0, 0.0}, eb = 0.0, ea = 0.0;
  bonded_atom(S, i, f, eb, ea);
  for (int c = 0; c < 3; c++) stg(S.brow + 3 * i + c, f[c]);
}

// In a small step the bonded terms (blocks from pol on) share the launch of the
// polarisation blocks, whose latency is the longer one; where the restraint
// runs beside full force kernels the two are launches of their own, because the
// 106 registers of the bonded terms (32 without) keep those from the CUs: 51
// windows of 11,056 atoms, 847 us per step in one launch, 834 in two.  A block of
// the small launch takes the atoms of one wave: 16 waves of FP64 angles on one
// CU took 21 us for 4,000 atoms, spread 9 us.
__global__ __launch_bounds__(64 * POL_SMALL_WAVES) void k_pol_bonded(const DevSys* __restrict__ systems, int pol) {
  const DevSys& S = systems[blockIdx.y];
  if ((int)blockIdx.x < pol) pol_forces<POL_SMALL_WAVES>(S);
  else if (threadIdx.x < QNB_WAVE) bonded_rows(S, ((int)blockIdx.x - pol) * QNB_WAVE + threadIdx.x);
}
__global__ __launch_bounds__(256) void k_pol_forces(const DevSys* __restrict__ systems) {
  pol_forces<4>(systems[blockIdx.y]);
}
__global__ __launch_bounds__(256) void k_bonded_rows(const DevSys* __restrict__ systems) {
  bonded_rows(systems[blockIdx.y], blockIdx.x * blockDim.x + threadIdx.x);
}

// Phase 3 on its own, one wave per system (watpol_finish): the minimiser's
// step; the MD step runs it in k_integrate, a single evaluation in
// k_reduce_final.
__global__ __launch_bounds__(64) void k_watpol_finish(const DevSys* __restrict__ systems) {
  watpol_finish(systems[blockIdx.x], 0, 1);
}

// ---------------------------------------------------------------------------
// Fixed-order reduction of the energy partials on the sampled steps, in two
// passes: block g of QNB_RED_BLOCKS per system sums its share of the per-wave
// records (a wave reads one 57-double record per iteration, lane k on energy
// k) and of the per-atom LRF and radial energies into ered_part[g]; one block
// per system then adds the QNB_RED_BLOCKS partials (reduce_final, qnb_dev.h;
// the MD step does that inside k_record).  The records are written all over
// the chip, so each read is a miss in this CU's caches and the pass is bound
// by how many reads are in flight: one block of 1,024 threads per system,
// whose thread 0 also added 1,024 atom sums in turn, took 68 us for 2,752
// records and 11,056 atoms; with 64 blocks and the final pass a whole
// evaluation of that system takes 62 us less (344 to 281 us).
__global__ __launch_bounds__(256) void k_reduce_part(const DevSys* __restrict__ systems) {
  const DevSys& S = systems[blockIdx.y];
  if (!want_energies(S)) return;
  const int g = blockIdx.x, lane = threadIdx.x % QNB_WAVE, c = threadIdx.x / QNB_WAVE;
  constexpr int NP = 4 * QNB_RED_BLOCKS;  // waves of a system
  const int p = 4 * g + c;
  const auto ep = gp(S.epart);
  const int a0 = (int)((long)S.ncgp * p / NP), a1 = (int)((long)S.ncgp * (p + 1) / NP);
  double s = 0.0;
  if (lane < QNB_NE) {
#pragma unroll 4
    for (int a = a0; a < a1; a++) s += ep[(size_t)a * QNB_NE + lane];
  }
  const auto ea = gp(S.eatom);
  const int i0 = (int)((long)S.natom * p / NP), i1 = (int)((long)S.natom * (p + 1) / NP);
  double l = 0.0, r = 0.0;
  for (int i = i0 + lane; i < i1; i += QNB_WAVE) {
    l += ea[2 * i];
    r += ea[2 * i + 1];
  }
  l = wave_sum(l);
  r = wave_sum(r);
  if (lane == E_LRF) s += l;
  if (lane == E_RAD) s += r;
  __shared__ double part[4][QNB_WAVE];
  part[c][lane] = s;
  __syncthreads();
  if (c == 0 && lane < QNB_NE)
    stg(S.ered_part + (size_t)g * QNB_NE + lane, ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane]);
}

// the second pass alone (single-system evaluations)
__global__ __launch_bounds__(256) void k_reduce_final(const DevSys* __restrict__ systems, int with_qq, int with_pol) {
  const DevSys& S = systems[blockIdx.x];
  if (want_energies(S)) reduce_final(S, with_qq, with_pol);
  if (with_pol) watpol_finish(S, threadIdx.x / QNB_WAVE, 4);
}

void launch_sweep(hipStream_t st, int prec, bool any, int lrf, int groups, int wpb, int B, const DevSys* dsys) {
  const dim3 g((groups + wpb - 1) / wpb, B), t(QNB_WAVE * wpb);
  if (lrf & SWEEP_PLAIN) {
    if (any) hipLaunchKernelGGL((k_lists_lrf<double, true, false>), g, t, 0, st, dsys);
    else hipLaunchKernelGGL((k_lists_lrf<double, false, false>), g, t, 0, st, dsys);
  }
  if (!(lrf & SWEEP_LRF)) return;
  if (prec == QNB_PREC_MIXED) {
    if (any) hipLaunchKernelGGL((k_lists_lrf<float, true, true>), g, t, 0, st, dsys);
    else hipLaunchKernelGGL((k_lists_lrf<float, false, true>), g, t, 0, st, dsys);
  } else {
    if (any) hipLaunchKernelGGL((k_lists_lrf<double, true, true>), g, t, 0, st, dsys);
    else hipLaunchKernelGGL((k_lists_lrf<double, false, true>), g, t, 0, st, dsys);
  }
}

SmallGrid small_grid(int solute_groups, int nwat, int sa, int nqat, int nat_solute, int nqe, uint32_t mask, bool pol) {
  SmallGrid G{};
  G.solute = solute_groups;
  G.solvent = (nwat + 3) / 4;
  if (nqat > 0 && (mask & (QNB_T_QW | QNB_T_QP))) {
    G.qchunks = std::max(1, std::min((nwat + nat_solute + QF_PART_SMALL - 1) / QF_PART_SMALL, 64));
    G.qside = nqat * ((G.qchunks + 3) / 4);
  }
  if (nqat > 0 && (mask & (QNB_T_QQ | QNB_T_QQP))) G.qq = (std::max(nqe, 1) + 3) / 4;
  if (pol) G.theta = (nwat + WP_THREADS - 1) / WP_THREADS;
  return G;
}

template <typename R, int NS, bool E>
static void launch_small(hipStream_t st, const SmallGrid& G, int B, const DevSys* dsys, uint32_t mask,
                         const int* istep) {
  const size_t lds = std::max(4 * so_wave_bytes<R>(),
                              std::max(sizeof(double) * 4 * NS * 4, sizeof(double) * 3 * 4 * QNB_WAVE));
  hipLaunchKernelGGL((k_forces_small<R, NS, E>), dim3(G.blocks(), B), dim3(256), lds, st, dsys, mask, G, istep);
}

template <typename R, bool E>
static void launch_small_ns(int ns, hipStream_t st, const SmallGrid& G, int B, const DevSys* dsys, uint32_t mask,
                            const int* istep) {
  if (ns <= 1) launch_small<R, 1, E>(st, G, B, dsys, mask, istep);
  else if (ns <= 2) launch_small<R, 2, E>(st, G, B, dsys, mask, istep);
  else if (ns <= 4) launch_small<R, 4, E>(st, G, B, dsys, mask, istep);
  else launch_small<R, 8, E>(st, G, B, dsys, mask, istep);
}

void launch_forces_small(hipStream_t st, int prec, int ns_max, bool energy, const SmallGrid& G, int B,
                         const DevSys* dsys, uint32_t mask, const int* istep) {
  if (G.blocks() <= 0) return;
  if (prec == QNB_PREC_MIXED) {
    if (energy) launch_small_ns<float, true>(ns_max, st, G, B, dsys, mask, istep);
    else launch_small_ns<float, false>(ns_max, st, G, B, dsys, mask, istep);
  } else {
    if (energy) launch_small_ns<double, true>(ns_max, st, G, B, dsys, mask, istep);
    else launch_small_ns<double, false>(ns_max, st, G, B, dsys, mask, istep);
  }
}

// explicit instantiations used by the host code
#define QNB_INST(R, NS)                                                            \
  template __global__ void k_qforces<R, NS>(const DevSys*, uint32_t, int, int);                       \
  template __global__ void k_sforces<R, NS, true>(const DevSys*, uint32_t, int, int, int); \
  template __global__ void k_sforces<R, NS, false>(const DevSys*, uint32_t, int, int, int); \
  template __global__ void k_wforces<R, NS, true>(const DevSys*, uint32_t, int, int, int); \
  template __global__ void k_wforces<R, NS, false>(const DevSys*, uint32_t, int, int, int); \
  template __global__ void k_gforces<R, NS>(const DevSys*, uint32_t, int, int, int);
QNB_INST(double, 1)
QNB_INST(double, 2)
QNB_INST(double, 4)
QNB_INST(double, 8)
QNB_INST(float, 1)
QNB_INST(float, 2)
QNB_INST(float, 4)
QNB_INST(float, 8)
#define QNB_INST_QQ(NS)                                           \
  template __global__ void k_qq<double, NS>(const DevSys*, uint32_t); \
  template __global__ void k_qq<float, NS>(const DevSys*, uint32_t);
QNB_INST_QQ(1)
QNB_INST_QQ(2)
QNB_INST_QQ(4)
QNB_INST_QQ(8)

}  // namespace qnb
