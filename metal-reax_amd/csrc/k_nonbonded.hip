// Tapered van der Waals + shielded Coulomb + polarization, and the charge-equilibration matrix H.
//
// One 64-lane wave per owned atom walks that atom's full skin list; every pair (i, j, s) with r <= nonb_cut is evaluated from both
// ends, each end keeping only its own gradient (-CE dvec on i) and half of the pair energy, so no atom writes another atom's force
// (atomic-free, bitwise repeatable: fixed lane assignment + fixed butterfly reduction). The distance is the canonical one, so both
// ends agree on the cut-off decision and on r. Reference: src/cpu/nonbonded.cpp:18-82 (pair loop, owner-computes counting: a
// physical pair counted once = half from each end here), include/reaxmetal/terms.hpp:262-325 (formulas), terms_host.hpp:17-39
// (taper). FP64 mode uses the reference's Horner taper and its exponents (pow(x, 0.33333333333333) for the cube root), each
// pow evaluated as exp(y log x); FP32 terms use the algebraically equal t-form of the taper (no cancellation of O(10)
// coefficients in float) and the float cube root. Both precisions run the same two passes: over the skin list with the pairs
// within the cutoff compacted into full waves, and over the charge-matrix rows when those are current.
//
// H (stock fix qeq/reaxff compute_H / calculate_H, LAMMPS fix_qeq_reaxff.cpp): H_ij = 14.4 Tap_q(r) / (r^3 + (g_i g_j)^-1.5)^(1/3) for
// r^2 <= swb^2, stored as full rows (both directions, every image): FP64 values in FP64 mode, FP32 values otherwise; 16-bit
// column indices when the system has at most 65535 atoms.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace rxa {
namespace {

struct NbAcc { double gx = 0, gy = 0, gz = 0, ev = 0, ee = 0, v[6] = {0, 0, 0, 0, 0, 0}; };

// this end's gradient -CE dvec, half of the pair energies and half of the pair virial r_ij (x) f_j = -CE dvec (x) dvec
__device__ inline void nb_acc(NbAcc& a, double ce, double evdw, double eel, double dx, double dy, double dz) {
  a.gx += -ce * dx; a.gy += -ce * dy; a.gz += -ce * dz;
  a.ev += 0.5 * evdw;
  a.ee += 0.5 * eel;
  const double hv = -0.5 * ce;
  a.v[0] += hv * dx * dx; a.v[1] += hv * dy * dy; a.v[2] += hv * dz * dz; a.v[3] += hv * dx * dy; a.v[4] += hv * dx * dz; a.v[5] += hv * dy * dz;
}

// FP64 terms of one pair (i, j) within nonb_cut at distance r, dvec = x_j - x_i: the reference's formulas in double with its
// Horner taper in r and its exponents (0.33333333333333 for the shielded Coulomb's cube root as written), pow(x, y) evaluated
// as exp(y log x) (a few ulp), the type pair's (1 / gamma_w)^p_vdW1 and the reciprocals of r_vdW and rcore from the table,
// e1 = e2^2 for the two Morse exponentials, and one division for 1 / r
template <class Row>
__device__ inline void nb_pair_d(const Globals& g, const Row* __restrict__ row, double qi, double qj, int tj, double r,
                                 double dx, double dy, double dz, NbAcc& a) {
  const Row& P = row[tj];
  const double p_vdW1 = g.p_vdW1, p1i = 1.0 / g.p_vdW1;
  const int vt = g.vdw_type;
  const double ir = 1.0 / r;
  const double* c = g.tap;
  double Tap = c[7] * r + c[6];
  Tap = Tap * r + c[5]; Tap = Tap * r + c[4]; Tap = Tap * r + c[3]; Tap = Tap * r + c[2]; Tap = Tap * r + c[1]; Tap = Tap * r + c[0];
  double dTap = 7 * c[7] * r + 6 * c[6];
  dTap = dTap * r + 5 * c[5]; dTap = dTap * r + 4 * c[4]; dTap = dTap * r + 3 * c[3]; dTap = dTap * r + 2 * c[2];
  dTap += c[1] * ir;
  const double alpha = P.alpha, D = P.D, a_r = alpha * P.irvdw;
  double evdw, CEvd;
  if (vt == 1 || vt == 3) {
    const double pr = exp(p_vdW1 * log(r)), S = pr + P.pgw;
    const double fn13 = exp(p1i * log(S));
    const double e2 = exp(0.5 * alpha * (1.0 - fn13 * P.irvdw)), e1 = e2 * e2;
    const double e0 = D * (e1 - 2.0 * e2);
    evdw = Tap * e0;
    const double dfn13 = fn13 / S * pr * (ir * ir);
    CEvd = dTap * e0 - Tap * D * a_r * (e1 - e2) * dfn13;
  } else {
    const double e2 = exp(0.5 * alpha * (1.0 - r * P.irvdw)), e1 = e2 * e2;
    const double e0 = D * (e1 - 2.0 * e2);
    evdw = Tap * e0;
    CEvd = dTap * e0 - Tap * D * a_r * (e1 - e2) * ir;
  }
  if (vt == 2 || vt == 3) {
    const double ec = P.ecore * exp(P.acore * (1.0 - r * P.ircore));
    evdw += Tap * ec;
    CEvd += dTap * ec + Tap * (-(P.acore * P.ircore) * ec) * ir;
    if (g.lg) {
      const double r6 = (r * r * r) * (r * r * r), idn = 1.0 / (r6 + P.re6);
      const double elg = -P.lgcij * idn;
      evdw += Tap * elg;
      CEvd += dTap * elg + Tap * (-6.0 * elg * (r6 * ir) * idn) * ir;
    }
  }
  const double d1 = r * r * r + P.gamma, id3 = 1.0 / exp(0.33333333333333 * log(d1));
  const double qq = 332.06371 * qi * qj;
  const double eel = qq * Tap * id3;
  const double CE = CEvd + qq * (dTap - Tap * r / d1) * id3;
  nb_acc(a, CE, evdw, eel, dx, dy, dz);
}

// Single-precision terms (mixed and FP32 modes): the same pair loop with the hardware base-2 exponential and logarithm
// (v_exp_f32 / v_log_f32, about 1 ulp) for exp, pow and the cube root, e1 = e2^2 for the two Morse exponentials, a pair table
// in float with (1/gamma_w)^p_vdW1 precomputed, and a squared-distance pre-test before the FP64 square root of the cut-off test.
__device__ inline float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ inline float flog2(float x) { return __builtin_amdgcn_logf(x); }

// one pair (i, j) within nonb_cut at distance rd, dvec = x_j - x_i: this end's gradient, half of the pair energy and virial
__device__ inline void nb_pair_f(const Globals& g, const NbPairF* __restrict__ row, float qi, float qj, int tj, double rd, double dx,
                             double dy, double dz, NbAcc& a) {
  // divisions by constants are products with reciprocals (table or loop-invariant), divisions by pair quantities use the
  // hardware reciprocal (1 ulp): single-precision terms, within their own rounding
  const float p_vdW1 = (float)g.p_vdW1, p1i = (float)(1.0 / g.p_vdW1);
  const int vt = g.vdw_type, lg = g.lg;
  const float swa = (float)g.nonb_low, itw = (float)(1.0 / (g.nonb_cut - g.nonb_low));
  const float L2E = 1.4426950408889634f;
  const NbPairF P = row[tj];
  const float r = (float)rd, ir = __builtin_amdgcn_rcpf(r);
  const float x = (r - swa) * itw, x2 = x * x, x3 = x2 * x, x4 = x2 * x2;
  const float Tap = 1.0f - x4 * (35.0f - 84.0f * x + 70.0f * x2 - 20.0f * x3);
  const float dTap = (x3 * (-140.0f + 420.0f * x - 420.0f * x2 + 140.0f * x3)) * (itw * ir);
  float evdw, CEvd;
  if (vt == 1 || vt == 3) {
    const float pr = fexp2(p_vdW1 * flog2(r)), S = pr + P.pgw;
    const float fn13 = fexp2(p1i * flog2(S));
    const float e2 = fexp2((0.5f * L2E) * P.alpha * (1.0f - fn13 * P.irvdw)), e1 = e2 * e2;
    const float e0 = P.D * (e1 - 2.0f * e2);
    evdw = Tap * e0;
    const float dfn13 = fn13 * __builtin_amdgcn_rcpf(S) * pr * (ir * ir);
    CEvd = dTap * e0 - Tap * P.D * P.a_r * (e1 - e2) * dfn13;
  } else {
    const float e2 = fexp2((0.5f * L2E) * P.alpha * (1.0f - r * P.irvdw)), e1 = e2 * e2;
    const float e0 = P.D * (e1 - 2.0f * e2);
    evdw = Tap * e0;
    CEvd = dTap * e0 - Tap * P.D * P.a_r * (e1 - e2) * ir;
  }
  if (vt == 2 || vt == 3) {
    const float ec = P.ecore * fexp2(L2E * P.acore * (1.0f - r * P.ircore));
    evdw += Tap * ec;
    CEvd += dTap * ec + Tap * (-P.ac_r * ec) * ir;
    if (lg) {
      const float r3 = r * r * r, r6 = r3 * r3, idn = __builtin_amdgcn_rcpf(r6 + P.re6);
      const float elg = -P.lgcij * idn;
      evdw += Tap * elg;
      CEvd += dTap * elg + Tap * (-6.0f * elg * (r6 * ir) * idn) * ir;
    }
  }
  const float d1 = r * r * r + P.gamma, rc = fexp2(flog2(d1) * (-1.0f / 3.0f));   // d1^(-1/3)
  const float qq = 332.06371f * qi * qj;
  const float eel = qq * Tap * rc;
  const float CE = CEvd + qq * (dTap - Tap * r * __builtin_amdgcn_rcpf(d1)) * rc;
  const double ce = (double)CE;
  a.gx += -ce * dx; a.gy += -ce * dy; a.gz += -ce * dz;
  a.ev += 0.5 * (double)evdw;
  a.ee += 0.5 * (double)eel;
  const double hv = -0.5 * ce;
  a.v[0] += hv * dx * dx; a.v[1] += hv * dy * dy; a.v[2] += hv * dz * dz; a.v[3] += hv * dx * dy; a.v[4] += hv * dx * dz; a.v[5] += hv * dy * dz;
}

// the per-precision parts of the non-bonded kernels below: the charges' type, the pair table row, the pair evaluation and the
// polarization energy
template <bool D> struct NbPrec;
template <> struct NbPrec<false> {
  using Q = float;
  using Row = NbPairF;
  using Tab = NbPairF;
  static __device__ Tab tab(const Row& P) { return P; }
  static __device__ const NbPairF* row(const Globals& g, const Tables& t, int ti) { return t.nbf + ti * g.ntypes; }
  static __device__ void pair(const Globals& g, const NbPairF* row, float qi, float qj, int tj, double rd, double dx, double dy,
                              double dz, NbAcc& a) {
    nb_pair_f(g, row, qi, qj, tj, rd, dx, dy, dz, a);
  }
  static __device__ double pol(const DevSpecies& sp, double qd) {
    const float q = (float)qd;
    return (double)(23.02f * ((float)sp.chi * q + ((float)sp.eta / 2.0f) * (q * q)));
  }
};
// the non-bonded part of DevPair
struct NbPairD { double D, alpha, irvdw, pgw, ecore, acore, ircore, gamma, lgcij, re6; };
template <> struct NbPrec<true> {
  using Q = double;
  using Row = DevPair;
  using Tab = NbPairD;
  static __device__ Tab tab(const Row& P) { return {P.D, P.alpha, P.irvdw, P.pgw, P.ecore, P.acore, P.ircore, P.gamma, P.lgcij, P.re6}; }
  static __device__ const DevPair* row(const Globals& g, const Tables& t, int ti) { return t.pair + ti * g.ntypes; }
  template <class R>
  static __device__ void pair(const Globals& g, const R* row, double qi, double qj, int tj, double rd, double dx, double dy,
                              double dz, NbAcc& a) {
    nb_pair_d(g, row, qi, qj, tj, rd, dx, dy, dz, a);
  }
  static __device__ double pol(const DevSpecies& sp, double q) { return 23.02 * (sp.chi * q + (sp.eta / 2.) * (q * q)); }
};

// wave sums in a fixed butterfly order, then lane 0 stores the atom's gradient, energies and virial
template <bool D>
__device__ inline void nb_finish(const State& st, const Tables& t, int i, int ti, int lane, const NbAcc& a) {
  // four sums at a time, row r of 16 lanes holding the r-th: its first lane stores it (the arrays' strides are n)
  const int n = st.n, row = lane >> 4;
  const bool first = (lane & 15) == 0;
  const double s0 = wave_sum4_rows(a.gx, a.gy, a.gz, a.ev);
  const double s1 = wave_sum4_rows(a.ee, a.v[0], a.v[1], a.v[2]);
  const double s2 = wave_sum4_rows(a.v[3], a.v[4], a.v[5], 0.0);
  if (!first) return;
  double* const p0 = row < 2 ? (row == 0 ? st.gnb_x : st.gnb_y) : (row == 2 ? st.gnb_z : st.eatom + T_VDW * n);
  p0[i] = s0;
  double* const p1 = row == 0 ? st.eatom + T_ELE * n : st.vatom + (size_t)(row - 1) * n;
  p1[i] = s1;
  if (row < 3) st.vatom[(size_t)(3 + row) * n + i] = s2;
  else st.eatom[T_POL * n + i] = ti >= 0 ? NbPrec<D>::pol(t.sp[ti], st.q[i]) : 0.0;
}

// Wave per atom over the skin list: the distance test runs on all lanes, pairs within nonb_cut are compacted (list order) into
// a per-wave LDS ring, and the term arithmetic runs on full waves of 64 pairs.
constexpr int kNbWaves = 4;
constexpr int kNbRing = 128;

template <bool D>
__device__ inline void nb_list_wave(const State& st, const Globals& g, const Tables& t, int i, int* rj, int* rt, double* rx,
                                    double* ry, double* rz, double* rr) {
  using Q = typename NbPrec<D>::Q;
  const int lane = lane_id();
  const int ti = st.type[i];
  NbAcc a;
  if (ti >= 0) {
    const size_t base = (size_t)i * st.maxnb;
    const int cnt = min(st.nb_cnt[i], st.maxnb);
    const Q qi = (Q)st.q[i];
    const double4 pi = st.pos[i];
    const double cut = g.nonb_cut, cut2 = cut * cut * (1.0 + 1e-12);
    const typename NbPrec<D>::Row* __restrict__ row = NbPrec<D>::row(g, t, ti);
    int head = 0, fill = 0;
    auto batch = [&](int m) {
      if (lane < m) {
        const int e = (head + lane) & (kNbRing - 1);
        const int j = rj[e];
        NbPrec<D>::pair(g, row, qi, (Q)st.q[j], rt[e], rr[e], rx[e], ry[e], rz[e], a);
      }
    };
    for (int k0 = 0; k0 < cnt; k0 += 64) {
      const int k = k0 + lane;
      bool keep = false;
      int j = 0, tj = -1;
      double dx = 0, dy = 0, dz = 0, rd = 0;
      if (k < cnt) {
        j = st.nb_j[base + k];
        const double r2 = pair_dvec_list(st, pi, j, st.nb_s[base + k], dx, dy, dz, tj);
        if (tj >= 0 && r2 <= cut2) {
          rd = sqrt(r2);
          keep = rd <= cut;
        }
      }
      const unsigned long long mk = __ballot(keep);
      if (keep) {
        const int e = (head + fill + lanes_below(mk)) & (kNbRing - 1);
        rj[e] = j; rt[e] = tj; rx[e] = dx; ry[e] = dy; rz[e] = dz; rr[e] = rd;
      }
      fill += __popcll(mk);
      __builtin_amdgcn_wave_barrier();
      if (fill >= 64) {
        batch(64);
        head = (head + 64) & (kNbRing - 1);
        fill -= 64;
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (fill > 0) batch(fill);
  }
  nb_finish<D>(st, t, i, ti, lane, a);
}

__global__ void __launch_bounds__(64 * kNbWaves) k_nonbonded_f(State st, Globals g, Tables t) {
  __shared__ int rj_[kNbWaves][kNbRing], rt_[kNbWaves][kNbRing];
  __shared__ double rx_[kNbWaves][kNbRing], ry_[kNbWaves][kNbRing], rz_[kNbWaves][kNbRing], rr_[kNbWaves][kNbRing];
  const int w = threadIdx.x >> 6;
  const int i = wave_atom();
  if (i >= st.n) return;
  nb_list_wave<false>(st, g, t, i, rj_[w], rt_[w], rx_[w], ry_[w], rz_[w], rr_[w]);
}

__global__ void __launch_bounds__(64 * kNbWaves) k_nonbonded_d(State st, Globals g, Tables t) {
  __shared__ int rj_[kNbWaves][kNbRing], rt_[kNbWaves][kNbRing];
  __shared__ double rx_[kNbWaves][kNbRing], ry_[kNbWaves][kNbRing], rz_[kNbWaves][kNbRing], rr_[kNbWaves][kNbRing];
  const int w = threadIdx.x >> 6;
  const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);   // not wave_atom: it spills here
  if (i >= st.n) return;
  nb_list_wave<true>(st, g, t, i, rj_[w], rt_[w], rx_[w], ry_[w], rz_[w], rr_[w]);
}

// What every pair of a row looks up, in LDS (one wave): the shift vectors and the row type's parameters. Read from memory in the
// pair loop they cost as much address traffic as the positions, and, loads returning in order, a wait for all that is in flight for the
// next pairs. The non-bonded pass over the rows took 81 us at 24,000 atoms and 661 us at 192,000; with chunks that have no shift taken
// without one 76 and 588, with these tables 62 and 466, with the row's own data in scalar registers (wave_atom) 58 and 411. Two
// capacities: with its ring the matrix build takes 20 KB per block with 32 shifts and 29 KB (5 blocks per CU, as many as its registers
// allow) with 128. A single periodic cell has 27 shifts from three list radii per side on (the cell search) and at least 125 below (one
// image more than reaches); packed systems have 27 where all are wider than two radii, 125 down to two thirds of one: 40 of them with
// 125 shifts, one capacity of 64 (tables in memory) 23.2 ms for 20 steps, with 128 22.7 ms. Cells with more shifts (thin ones) or
// force fields with more types read them from memory.
constexpr int kTabTypes = 16;
// the tables' capacity in shift vectors (0: no tables)
inline int row_table_shifts(const State& st, const Globals& g) {
  const long long ns = (long long)(2 * st.smx0 + 1) * (2 * st.smx1 + 1) * (2 * st.smx2 + 1);
  return g.ntypes > kTabTypes || ns > 128 ? 0 : ns > 32 ? 128 : 32;
}
// calls f(integral_constant c) for the capacity
template <class F>
inline void with_row_tables(const State& st, const Globals& g, F&& f) {
  switch (row_table_shifts(st, g)) {
    case 32: f(std::integral_constant<int, 32>{}); break;
    case 128: f(std::integral_constant<int, 128>{}); break;
    default: f(std::integral_constant<int, 0>{}); break;
  }
}
template <class P, int kTab>
struct RowTables {
  double x[kTab ? kTab : 1], y[kTab ? kTab : 1], z[kTab ? kTab : 1];
  P par[kTabTypes];
  __device__ void fill_shifts(const State& st, const double4* __restrict__ shv) {
    const int ns = 2 * shift_index(st, 0) + 1;
    for (int k = lane_id(); k < ns; k += 64) {
      const double4 S = shv[k];
      x[k] = S.x; y[k] = S.y; z[k] = S.z;
    }
  }
  __device__ double4 shift(int k) const { return make_double4(x[k], y[k], z[k], 0.0); }
};

// pair_dvec_list for a charge-matrix entry: the same operands in the same order, the shift vector found through the entry's key
// (zero: the key's index of the zero shift)
template <class F>
__device__ inline double pair_dvec_key(F&& shift, const double4 pi, const double4 pj, int key, int zero, double& dx, double& dy, double& dz) {
  const int k = key & 0x7FFF;
  if (!__any(k != zero)) return pair_dvec_plain(pi, pj, dx, dy, dz);
  return pair_dvec_shift(pi, pj, (key & 0x8000) != 0, shift(k), dx, dy, dz);
}

// The non-bonded terms over the charge-matrix rows: the rows hold, in skin-list order, exactly the pairs within the matrix
// cutoff, so every lane carries a pair (no distance pre-pass, no compaction) and a row costs its column and key (4 bytes per
// pair with 16-bit columns) instead of the 8-byte skin entries of all pairs out to the list radius. Lane l takes entries l,
// l + 64, ..., the assignment of the skin-list kernel's compacted batches, so the sums are the same.
template <bool D, int kTab, class TC>
__device__ inline void nb_rows_wave(const State& st, const Globals& g, const Tables& t, const TC* __restrict__ col,
                                    const unsigned short* __restrict__ key, const int* __restrict__ rcnt, int stride, int i,
                                    RowTables<typename NbPrec<D>::Tab, kTab>& L) {
  using Q = typename NbPrec<D>::Q;
  const int lane = lane_id();
  const int ti = st.type[i];
  NbAcc a;
  if (ti >= 0) {
    const size_t base = (size_t)i * stride;   // keys in list order, columns as row_slot puts them
    const int cnt = rcnt[i], zero = shift_index(st, 0);
    const Q qi = (Q)st.q[i];
    const double4 pi = st.pos[i];
    const double cut = g.nonb_cut, cut2 = cut * cut * (1.0 + 1e-12);
    const typename NbPrec<D>::Row* __restrict__ row = NbPrec<D>::row(g, t, ti);
    const double4* __restrict__ shv = st.shv + pos_sys(pi.w) * st.shv_stride;
    if (kTab) {
      L.fill_shifts(st, shv);
      if (lane < g.ntypes) L.par[lane] = NbPrec<D>::tab(row[lane]);
      __builtin_amdgcn_wave_barrier();
    }
    // two-deep software pipeline as in the matrix build: columns/keys two strides ahead, positions and charges one ahead
    // (lanes past the row's end carry the row atom itself and key 0, valid indices never used)
    int jB = i, kyB = 0, jC = i, kyC = 0;
    if (lane < cnt) { jC = (int)col[base + row_slot(lane)]; kyC = key[base + lane]; }
    double4 pC = st.pos[jC];
    Q qC = (Q)st.q[jC];
    if (lane + 64 < cnt) { jB = (int)col[base + row_slot(lane + 64)]; kyB = key[base + lane + 64]; }
    for (int k = lane; k < cnt; k += 64) {
      const double4 pj = pC;
      const Q qj = qC;
      const int ky = kyC;
      jC = jB; kyC = kyB;
      pC = st.pos[jC];
      qC = (Q)st.q[jC];
      jB = i; kyB = 0;
      if (k + 128 < cnt) { jB = (int)col[base + row_slot(k + 128)]; kyB = key[base + k + 128]; }
      double dx, dy, dz;
      const double r2 = pair_dvec_key([&](int s) { return kTab ? L.shift(s) : shv[s]; }, pi, pj, ky, zero, dx, dy, dz);
      if (r2 <= cut2) {
        const double rd = sqrt(r2);
        if (rd <= cut) {
          if constexpr (kTab) NbPrec<D>::pair(g, L.par, qi, qj, pos_type(pj.w), rd, dx, dy, dz, a);
          else NbPrec<D>::pair(g, row, qi, qj, pos_type(pj.w), rd, dx, dy, dz, a);
        }
      }
    }
  }
  nb_finish<D>(st, t, i, ti, lane, a);
}

// (asked for 5 waves per SIMD: with the row's data in vector registers 96 VGPRs without spills, where the compiler's own choice of 106 and 4
// waves was slower; 79 and 6 waves since it is in scalar ones)
template <class TC, int kTab>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_nonbonded_rows(State st, Globals g, Tables t, const TC* __restrict__ col,
                                                        const unsigned short* __restrict__ key, const int* __restrict__ rcnt, int stride) {
  __shared__ RowTables<NbPairF, kTab> L[kTab ? 4 : 1];
  const int i = wave_atom();
  if (i >= st.n) return;
  nb_rows_wave<false, kTab, TC>(st, g, t, col, key, rcnt, stride, i, L[kTab ? threadIdx.x >> 6 : 0]);
}
template <class TC, int kTab>
__global__ void __launch_bounds__(256) k_nonbonded_rows_d(State st, Globals g, Tables t, const TC* __restrict__ col,
                                                          const unsigned short* __restrict__ key, const int* __restrict__ rcnt, int stride) {
  __shared__ RowTables<NbPairD, kTab> L[kTab ? 4 : 1];
  const int i = wave_atom();
  if (i >= st.n) return;
  nb_rows_wave<true, kTab, TC>(st, g, t, col, key, rcnt, stride, i, L[kTab ? threadIdx.x >> 6 : 0]);
}

constexpr int kQbWaves = 4, kQbRing = 256;

// One wave per row atom over its skin list, 128 entries at a time: a filter pass (distance only) pushes the pairs within the matrix
// cutoff, in list order, into a per-wave LDS ring; every 64 of them are finished together (taper, shielded 1/r, stores), so the
// costly part runs on full waves. Bound by the latency of a wave's chain of loads: doing the arithmetic, the position gathers or the
// stores twice adds 0 to 5 %. So two chunks go through the chain at once, each round's loads go out in the order in which they are
// waited for (the guess gathers of the batches, the next positions, the entries after those), and the row's own data sit in scalar
// registers. 24,000 / 192,000 atoms of water: 138 / 1064 us a chunk at a time with the tables in memory, 137 / 1075 with the tables in
// LDS, 123 / 945 two chunks at a time, 117 / 915 us with the row's data in scalar registers (79 VGPRs, 6 waves per SIMD), 113 / 872 us with
// the stores in whole groups (81 VGPRs, 5 waves). Row entries are kept in skin-list
// order: slot m of the row is the m-th pair of the list within the cutoff. The 16-bit key is the canonical flag and the
// shift-table index the distance used.
// fuse: the row also forms the charge solve's start from the guess in x (k_cg_guess ran before): y = H x with the values as
// built (FP64, or the FP32 values a non-refined FP32 solve iterates with), r = b - (y + eta x), p = r / eta, and the row's
// b.b and r.p for the block partials; this replaces a separate product pass over the rows.
template <int kTab>
__device__ inline void qeq_build_row(const State& st, const Globals& g, const Tables& t, const QeqBuffers& qb, int i, int fuse,
                                     int* rj, int* rk, double* rr, RowTables<double, kTab>& L, double (&acc)[4]) {
  const int lane = lane_id();
  const int ti = st.type[i];
  const size_t base = (size_t)i * st.maxnb, rbase = (size_t)i * qb.stride;
  const int cnt = ti >= 0 ? min(st.nb_cnt[i], st.maxnb) : 0;
  const double swb2 = g.q_swb * g.q_swb;
  const double* T = g.qtap;
  const double4 pi = st.pos[i];
  const double4* __restrict__ shv = st.shv + pos_sys(pi.w) * st.shv_stride;
  const double* __restrict__ shld = t.qeq_shld + max(ti, 0) * g.ntypes;
  const double eta = ti >= 0 ? t.qeq_eta[ti] : 1.0, chi = ti >= 0 ? t.qeq_chi[ti] : 0.0;
  const double2* __restrict__ x2 = reinterpret_cast<const double2*>(qb.x);
  const double2 xi = fuse ? x2[i] : make_double2(0.0, 0.0);
  const int zero = shift_index(st, 0);
  const int* __restrict__ lj = st.nb_j + base;
  const int* __restrict__ ls = st.nb_s + base;
  // entry k of the list (past its end the last one, which no lane uses)
  const int last = max(cnt - 1, 0);
  auto entry = [&](int k, int& j, int& e) { const int q = min(k, last); j = cnt ? lj[q] : i; e = cnt ? ls[q] : 0; };
  int jn[2], en[2], jc[2], ec[2];   // the next two chunks' entries, this pair's
  double4 pc[2];
  for (int u = 0; u < 2; ++u) {   // with the count in flight (entries past it are cleared)
    const int q = min(64 * u + lane, st.maxnb - 1);
    jc[u] = lj[q]; ec[u] = ls[q];
  }
  for (int u = 0; u < 2; ++u)
    if (64 * u + lane >= cnt) { jc[u] = i; ec[u] = 0; }
  for (int u = 0; u < 2; ++u) entry(64 * (2 + u) + lane, jn[u], en[u]);
  if (kTab) {
    L.fill_shifts(st, shv);
    if (lane < g.ntypes) L.par[lane] = shld[lane];
    __builtin_amdgcn_wave_barrier();
  }
  for (int u = 0; u < 2; ++u) pc[u] = st.pos[jc[u]];
  int m = 0, head = 0, fill = 0;
  double lo_sum = 0.0;   // this lane's part of sum_j |lo_ij| (refinement)
  double y0 = 0.0, y1 = 0.0;   // fuse: this lane's part of (H x) of both systems
  // the lane's entry of a batch taken from the ring: column, key | type, squared distance, then the matrix entry
  struct Batch { int j, k; double h; double2 x; };
  auto take = [&](int count, Batch& b) {
    const int e = (head + lane) & (kQbRing - 1);
    b.j = i;
    if (lane < count) { b.j = rj[e]; b.k = rk[e]; b.h = rr[e]; }
    if (fuse) b.x = x2[b.j];
    head = (head + count) & (kQbRing - 1);
    fill -= count;
  };
  // h - (float)h is exact in FP64; rounded to FP32 it leaves the two parts within about 2^-48 (relative) of h
  auto low = [](double h) { return (float)(h - (double)(float)h); };
  auto evaluate = [&](int count, Batch& b) {
    if (lane < count) {
      const double r = sqrt(b.h);
      double Tap = T[7] * r + T[6];
      Tap = Tap * r + T[5]; Tap = Tap * r + T[4]; Tap = Tap * r + T[3]; Tap = Tap * r + T[2]; Tap = Tap * r + T[1]; Tap = Tap * r + T[0];
      double sh;
      if constexpr (kTab) sh = L.par[b.k >> 16]; else sh = shld[b.k >> 16];
      b.h = (Tap * 14.4) * rcbrt_f64(r * r * r + sh);
      double hv = b.h;   // the value the start's product uses
      if (qb.fp32) {
        if (qb.refine) lo_sum += fabs((double)low(b.h));
        else hv = (double)(float)b.h;
      }
      if (fuse) {
        y0 += hv * b.x.x;
        y1 += hv * b.x.y;
      }
    }
  };
  auto store = [&](int count, const Batch& b) {   // places past the row's end: the row's own column (take) and zero
    const size_t o = rbase + m + group_slot(lane);   // row_slot: m counts full groups
    const double h = lane < count ? b.h : 0.0;
    if (qb.narrow) qb.col16[o] = (unsigned short)b.j; else qb.col[o] = b.j;
    if (qb.fp32) {
      qb.val32[o] = (float)h;
      if (qb.refine) qb.lo32[o] = low(h);
    } else {
      qb.val[o] = h;
    }
    if (qb.keyed && lane < count) qb.key[rbase + m + lane] = (unsigned short)(b.k & 0xFFFF);
    m += count;
  };
  for (int k0 = 0; k0 < cnt; k0 += 128) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = k0 + 64 * u + lane, j = jc[u], e = ec[u];
      const double4 pj = pc[u];
      bool keep = false;
      double r2 = 0;
      int kt = 0;
      if (k < cnt) {
        const bool canon = (e & kCanon) != 0;
        int sidx = zero;
        double dx, dy, dz;
        if (!__any(entry_code(e) != 0)) {
          r2 = pair_dvec_plain(pi, pj, dx, dy, dz);
        } else {
          sidx = entry_shift_index(st, e);
          r2 = pair_dvec_shift(pi, pj, canon, kTab ? L.shift(sidx) : shv[sidx], dx, dy, dz);
        }
        const int tj = pos_type(pj.w);
        keep = tj >= 0 && r2 <= swb2;
        kt = (qb.keyed ? (canon ? 0x8000 : 0) | sidx : 0) | (tj << 16);   // a keyed table has at most 32768 entries
      }
      const unsigned long long msk = __ballot(keep);
      if (keep) {
        const int e2 = (head + fill + lanes_below(msk)) & (kQbRing - 1);
        rj[e2] = j; rk[e2] = kt; rr[e2] = r2;
      }
      fill += __popcll(msk);
    }
    __builtin_amdgcn_wave_barrier();
    // the full batches leave the ring; their guess values, then the next chunks' positions, then the entries after those go out
    Batch b0, b1;
    const int nfull = fill >> 6;
    if (nfull > 0) take(64, b0);
    if (nfull > 1) take(64, b1);
    __builtin_amdgcn_wave_barrier();
    for (int u = 0; u < 2; ++u) { jc[u] = jn[u]; ec[u] = en[u]; pc[u] = st.pos[jc[u]]; }
    for (int u = 0; u < 2; ++u) entry(k0 + 64 * (4 + u) + lane, jn[u], en[u]);
    if (nfull > 0) evaluate(64, b0);
    if (nfull > 1) evaluate(64, b1);
    // what was loaded has come back here, before the stores go out: loads and stores are waited for in order, so a wait at the
    // top of the loop would be one for the stores
    for (int u = 0; u < 2; ++u)
      asm volatile("" : "+v"(pc[u].x), "+v"(pc[u].y), "+v"(pc[u].z), "+v"(pc[u].w), "+v"(jn[u]), "+v"(en[u]));
    if (nfull > 0) store(64, b0);
    if (nfull > 1) store(64, b1);
  }
  if (fill > 0 || m == 0) {   // (an empty row gets one group of such places: the product reads a row's last group again)
    Batch b;
    const int count = fill;
    take(count, b);
    evaluate(count, b);
    store(count, b);
  }
  {
    double s[3] = {lo_sum, y0, y1};
    wave_sums<3>(s);
    lo_sum = s[0]; y0 = s[1]; y1 = s[2];
  }
  if (lane == 0) {
    qb.cnt[i] = m;
    if (qb.refine) qb.lorow[i] = lo_sum;
    const double hinv = 1.0 / eta;
    qb.eta[i] = eta;
    qb.hinv[i] = hinv;
    qb.chi[i] = chi;
    if (fuse) {   // the start of k_spmv2's kMode 1 for this row (b from this build's chi: the guess kernel ran before it)
      const double wv[2] = {y0 + eta * xi.x, y1 + eta * xi.y};
      for (int s = 0; s < 2; ++s) {
        const double b = s == 0 ? -chi : -1.0;
        qb.b[2 * i + s] = b;
        const double r = b - wv[s];
        const double d = r * hinv;
        qb.r[2 * i + s] = r;
        qb.p[2 * i + s] = d;
        acc[s] = b * b;
        acc[2 + s] = r * d;
      }
    }
  }
}

template <int kTab>
__global__ void __launch_bounds__(256) k_qeq_build(State st, Globals g, Tables t, QeqBuffers qb, int fuse) {
  __shared__ RowTables<double, kTab> L[kTab ? kQbWaves : 1];
  __shared__ int ring_j[kQbWaves][kQbRing];
  __shared__ int ring_k[kQbWaves][kQbRing];   // key | neighbour type << 16
  __shared__ double ring_r2[kQbWaves][kQbRing];
  __shared__ double sh[4 * kQbWaves];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = wave_atom();
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  if (i < st.n) qeq_build_row<kTab>(st, g, t, qb, i, fuse, ring_j[wv], ring_k[wv], ring_r2[wv], L[kTab ? wv : 0], acc);
  if (fuse) {   // the block's partials of b.b and r.p, its rows in wave order (a fixed order)
    if (lane_id() == 0)
      for (int k = 0; k < 4; ++k) sh[k * kQbWaves + wv] = acc[k];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int k = 0; k < 4; ++k) {
        double v = sh[k * kQbWaves];
        for (int w = 1; w < kQbWaves; ++w) v += sh[k * kQbWaves + w];
        qb.partial_qb[blockIdx.x * 4 + k] = v;
      }
  }
}

// Census of the non-bonded cut-off decision: per atom, the pairs its skin list holds at the counted (canonical) end within
// nonb_cut. The test is the one every non-bonded kernel takes (the FP64 square root of the canonical squared distance <=
// nonb_cut, in all precisions), on the same list entries, so the count is the number of pairs those kernels evaluate there.
__global__ void __launch_bounds__(256) k_census_nb(State st, Globals g) {
  const int i = wave_atom();
  if (i >= st.n) return;
  const int lane = lane_id();
  const int ti = st.type[i];
  int c = 0;
  if (ti >= 0) {
    const size_t base = (size_t)i * st.maxnb;
    const int cnt = min(st.nb_cnt[i], st.maxnb);
    const double4 pi = st.pos[i];
    for (int k = lane; k < cnt; k += 64) {
      const int e = st.nb_s[base + k];
      if (!(e & kCanon)) continue;
      double dx, dy, dz;
      int tj;
      const double r2 = pair_dvec_list(st, pi, st.nb_j[base + k], e, dx, dy, dz, tj);
      if (tj >= 0 && sqrt(r2) <= g.nonb_cut) ++c;
    }
  }
  c = wave_sum_int(c);
  if (lane == 0) st.cen[kCenNonbonded * st.n + i] = c;
}

inline int nblk(long long items, int per) { return (int)((items + per - 1) / per); }

}  // namespace

void launch_census_nb(const State& st, const Globals& g, hipStream_t s) {
  hipLaunchKernelGGL(k_census_nb, dim3(nblk((long long)st.n * 64, 256)), dim3(256), 0, s, st, g);
}

void launch_nonbonded(Precision p, const State& st, const Cell& c, const Globals& g, const Tables& t, hipStream_t s) {
  const dim3 grid(nblk((long long)st.n * 64, 256)), blk(256);
  (void)c;
  if (p == Precision::FP64) hipLaunchKernelGGL(k_nonbonded_d, grid, blk, 0, s, st, g, t);
  else hipLaunchKernelGGL(k_nonbonded_f, grid, blk, 0, s, st, g, t);
}

void launch_nonbonded_rows(Precision p, const State& st, const Globals& g, const Tables& t, const QeqBuffers& qb, hipStream_t s) {
  const dim3 grid(nblk((long long)st.n * 64, 256)), blk(256);
  with_row_tables(st, g, [&](auto tab) {
    constexpr int kTab = decltype(tab)::value;
    if (p == Precision::FP64) {
      if (qb.narrow) hipLaunchKernelGGL((k_nonbonded_rows_d<unsigned short, kTab>), grid, blk, 0, s, st, g, t, qb.col16, qb.key, qb.cnt, qb.stride);
      else hipLaunchKernelGGL((k_nonbonded_rows_d<int, kTab>), grid, blk, 0, s, st, g, t, qb.col, qb.key, qb.cnt, qb.stride);
    } else {
      if (qb.narrow) hipLaunchKernelGGL((k_nonbonded_rows<unsigned short, kTab>), grid, blk, 0, s, st, g, t, qb.col16, qb.key, qb.cnt, qb.stride);
      else hipLaunchKernelGGL((k_nonbonded_rows<int, kTab>), grid, blk, 0, s, st, g, t, qb.col, qb.key, qb.cnt, qb.stride);
    }
  });
}

void launch_qeq_build(const State& st, const Cell& c, const Globals& g, const Tables& t, QeqBuffers& qb, int fuse, hipStream_t s) {
  (void)c;
  const dim3 grid(qeq_build_blocks(st.n)), blk(256);
  with_row_tables(st, g, [&](auto tab) {
    hipLaunchKernelGGL(k_qeq_build<decltype(tab)::value>, grid, blk, 0, s, st, g, t, qb, fuse);
  });
}

}  // namespace rxa
