// Host-side launchers of the device kernels (one translation unit per kernel family; engine.hip orchestrates them).
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace rxa {

enum class Precision { FP64 = 0, MIXED = 1, FP32 = 2 };

struct BinGrid {
  int nc[3] = {1, 1, 1};
  int ncells() const { return nc[0] * nc[1] * nc[2]; }
};
struct BinBuffers {
  unsigned *keys = nullptr, *skeys = nullptr, *atom_key = nullptr;
  int *idx = nullptr, *sidx = nullptr, *cstart = nullptr, *cend = nullptr;
  void* temp = nullptr;
  size_t temp_bytes = 0;
};

// ---- neighbour search (k_neighbor.hip)
void launch_wrap(const State& st, const Cell& c, hipStream_t s);
void launch_fill_int(int* p, int n, int v, hipStream_t s);
void launch_flags_out(const int* flags, int* host, hipStream_t s);   // the 8 capacity flags into pinned host memory
size_t bin_temp_bytes(int n);
void launch_bin(const State& st, const Cell& c, const BinGrid& g, BinBuffers& b, hipStream_t s);
// skin list and sub-lists of every atom (radii rs, rb for bond and rh for H-bond candidates). sorted: the atoms are in the order of
// their cells, so an atom's key is b.skeys of its index and the order needs no index
SubCut sub_cut(double rb, double rh);
void launch_nbr_cells(const State& st, const Globals& gl, const Tables& t, const Cell& c, const BinGrid& g, const BinBuffers& b, bool sorted,
                      double rs, double rb, double rh, hipStream_t s);
void launch_nbr_brute(const State& st, const Globals& g, const Tables& t, const Cell& c, const int sm[3], double rs, double rb, double rh,
                      hipStream_t s);
void launch_pos4(const State& st, hipStream_t s);                                   // pos = (x, y, z, type)
struct PermuteSet {   // per-atom arrays moved together by launch_permute
  int n = 0, nd = 0, ni = 0, nl = 0;
  double* d[24];
  int* i[4];
  long long* l[2];
};
void launch_permute(const PermuteSet& ps, const int* src, double* sd, int* si, long long* sl, hipStream_t s);
void launch_positions_in(const State& st, const double* ux, const int* perm, hipStream_t s);
void launch_shift_table(const Cell& c, double4* shv, const int smx[3], hipStream_t s);
// the sub-lists of all atoms from the skin list (packed systems, and after a sub-list's capacity grew); the acceptors' rows of the H-bond candidates
void launch_sublists(const State& st, const Globals& g, const Tables& t, double rb, double rh, hipStream_t s);
void launch_acceptor_rows(const State& st, const Globals& g, const Tables& t, hipStream_t s);

// ---- bond-order chain and bonded terms (k_bonded.hip)
void launch_bond_build(Precision p, const State& st, const Globals& g, const Tables& t, hipStream_t s);
// (limit8: also the number of atoms with more than 8 bonds, exact up to this limit, see both_sizes_limit; -1: not counted)
void launch_bo_correct(Precision p, const State& st, const Globals& g, const Tables& t, int limit8, hipStream_t s);
void launch_atom_terms(Precision p, const State& st, const Globals& g, const Tables& t, hipStream_t s);
// The angle kernels take 8 and 16 lanes per atom in one launch where at most this many atoms have more than 8 bonds (and none more than
// 16); -1: never. With 16 lanes for all a wave takes 4 atoms: up to 12,288 of them (3 waves on each of the 1,024 SIMDs, FP32 terms) run
// at once, and nothing is gained. Beyond that, the three term kernels of disordered carbon, 16 lanes for all against both (a group of 8
// atoms with one of those atoms costs as before, and its launch finds the others by their counts):
//   FP32 terms, 12,000 atoms 0.4 % 133 / 138 us, 1.1 % 135 / 151; 12,400 0.3 % 149 / 138, 1.3 % 163 / 154; 16,000 0.2 % 161 / 135, 1.6 %
//   189 / 186; 30,000 0.4 % 244 / 209, 1.3 % 264 / 242, 2.1 % 273 / 283. (24,000, two rounds of waves either way: 0.7 % 206 / 207,
//   1.4 % 220 / 229.)
//   FP64 terms, 12,400 atoms 0.3 % 173 / 144 us, 0.7 % 180 / 188; 14,000 0.2 % 175 / 165, 1.2 % 199 / 215; 16,000 0.2 % 182 / 181, 1.3 %
//   210 / 219; 18,000 0.3 % 209 / 188, 1.6 % 248 / 235; 20,000 1.4 % 264 / 245; 30,000 1.3 % 342 / 331, 2.1 % 354 / 377.
inline int both_sizes_limit(Precision p, int n) { return n <= 12288 ? -1 : p == Precision::FP64 && n < 18000 ? n / 256 : n / 64; }
void launch_angle_terms(Precision p, const State& st, const Globals& g, const Tables& t, int bmax, bool both, hipStream_t s);
// BO-derivative pass (CdDelta, then the per-atom bond sums); the final gather adds the non-bonded gradient and the virial
void launch_bond_derivatives(const State& st, hipStream_t s);
void launch_gather(const State& st, hipStream_t s);
void launch_eatom_ref(const State& st, hipStream_t s);   // per-atom energies of the reference's attribution (peratom calls)
void launch_vatom_ref(const State& st, hipStream_t s);   // per-atom virials of the reference's split (peratom calls, before the gather)

// ---- non-bonded terms and the charge-equilibration matrix (k_nonbonded.hip)
void launch_nonbonded(Precision p, const State& st, const Cell& c, const Globals& g, const Tables& t, hipStream_t s);

// Place of the k-th entry of a charge-matrix row in the row's storage: a group of 64 entries puts side by side the four entries
// k = l, l + 16, l + 32, l + 48 that lane l of the product's 16 lanes per row adds in turn, so the lane reads them as one vector (8
// bytes of 16-bit columns, 16 bytes of FP32 values). The last group's places past the row's end hold the row's own column and zero; an
// empty row has one group of such places.
// Rows are a multiple of 64 entries apart and start on 128-byte lines.
constexpr int kRowGroup = 64;
__host__ __device__ inline int group_slot(int r) { return ((r & 15) << 2) | ((r >> 4) & 3); }
__host__ __device__ inline int row_slot(int k) { return (k & ~(kRowGroup - 1)) | group_slot(k); }
inline int row_stride(int maxnb) { return (maxnb + kRowGroup - 1) / kRowGroup * kRowGroup; }

struct QeqBuffers {
  int stride = 0;            // entries from row to row (row_stride of the skin list's capacity)
  int* cnt = nullptr;        // n: entries per row
  // the rows are stored in exactly one column format and one value format, entry k of row i at i * stride + row_slot(k):
  int* col = nullptr;               // n * stride: column (owned atom index), when narrow == 0
  unsigned short* col16 = nullptr;  // n * stride: the same in 16 bits, when narrow == 1 (n <= 65535)
  double* val = nullptr;            // n * stride: H_ij in FP64 (FP64 mode)
  float* val32 = nullptr;           // n * stride: H_ij in FP32 (mixed and FP32 modes)
  // n * stride: the FP32 remainder H_ij - (double)val32 (written when refine == 1), so that (double)val32 + (double)lo32
  // carries H_ij to about 48 bits for the FP64 residuals of the iterative refinement
  float* lo32 = nullptr;
  int narrow = 0;
  // FP64 iterative refinement of the FP32-valued solve: initial and verification residuals with the two-float matrix, CG
  // restarted from the true residual while it exceeds the tolerance (mixed mode; FP32 mode with the fix's 'resident' keyword)
  int refine = 0;
  // n * stride (entries in list order): how the pair of each entry is reached from the row's atom, for the non-bonded pass over the same rows: bit 15 set
  // if the row's atom is the pair's canonical end, bits 0-14 the index in the shift-vector table of the lattice shift applied to
  // the canonical end's partner. Written when keyed == 1 (shift table of at most 32768 vectors).
  unsigned short* key = nullptr;
  int keyed = 0;
  double* eta = nullptr;     // n: diagonal (fix eta, 2 x ffield)
  double* hinv = nullptr;    // n: 1 / eta
  double* chi = nullptr;     // n
  // CG state, two systems (s: b = -chi, t: b = -1) interleaved per atom: [2*i + sys]
  double *b, *x, *r, *d, *p, *q;
  double* partial;           // 4 * kCgBlocks: per-block partials of the element-wise CG kernels
  double* partial_mv;        // 4 * qeq_mv_partials(n): per-block partials of the matrix-vector product
  double* partial_rs;        // 4 * qeq_mv_partials(n): per-block partials of the refinement's verification residual
  double* partial_qb;        // 4 * qeq_build_blocks(n): per-block partials of the solve's start fused into the matrix build
  // refinement's bound (k_qeq.hip gate_partials): the FP32 remainders' row sums sum_j |lo_ij| (n), the CG start x0 (2 n, same
  // layout as x) and the gate's per-block partials (3 * qeq_gate_partials(), pinned host memory)
  double* lorow = nullptr;
  double* x0 = nullptr;
  double* gate_host = nullptr;
  int fp32 = 0;              // the matrix values are val32 (mixed and FP32 modes) instead of val
  double* scal;              // device scalars and activity flags per iteration (see k_qeq.hip), own allocation sized by imax
  double* scal_host = nullptr;   // the same in pinned host memory, written by the kernels that set them
  double *s_hist, *t_hist;   // 4 * n each, [k * n + i], k = 0 most recent
};
constexpr int kCgBlocks = 256;
// doubles per iteration slot of QeqBuffers::scal after its 8-double header (sig of s and t, the activity pair, the restart-record
// pair); the scalars of iterations 0 .. imax + 1 take 8 + kScalSlot (imax + 2) doubles
constexpr int kScalSlot = 4;
inline size_t qeq_scal_doubles(int imax) { return 8 + (size_t)kScalSlot * (size_t)(imax + 2); }
// several independent systems packed in one engine: per-system CG scalars and row scratch (k_qeq.hip)
struct PackedQeq {
  int S = 0;
  const int* sys_start = nullptr;   // S + 1 row offsets
  const int* sysid = nullptr;       // n: system of each row
  double* pk = nullptr;             // 10 S: per solve |b|, r.p, alpha, beta; sums of s and t
  int* pki = nullptr;               // 4 S: per solve state (1 active, 0 stopped, 2 stopped and verified by the refinement
                                    // check), stock loop index
  double* rowv = nullptr;           // 4 n: per-row d.q and r.p of both solves
  int* any = nullptr;               // imax + 2, pinned host memory: some system active for iteration it + 1 (set to 1 by iteration
                                    // it, [0] by the start; cleared by the host)
};
void launch_pk_qeq_init(const State& st, QeqBuffers& qb, const PackedQeq& pq, int imax, double tol, int use_hist, hipStream_t s);
void launch_pk_qeq_iteration(const State& st, QeqBuffers& qb, const PackedQeq& pq, int it, int imax, double tol, hipStream_t s);
// refinement check after iteration it (qb.refine): every solve that has stopped and is not yet verified gets its true residual
// with the two-float matrix; a solve above tol restarts (beta 0) for iteration it + 1, the others are verified
void launch_pk_qeq_restart(const State& st, QeqBuffers& qb, const PackedQeq& pq, int it, int imax, double tol, hipStream_t s);
void launch_pk_qeq_finish(const State& st, QeqBuffers& qb, const PackedQeq& pq, hipStream_t s);
// packed systems: neighbour search, integrator and energy sums per system (k_packed.hip)
void launch_pk_shift_table(const Cell* cells, int S, double4* shv, const int smx[3], hipStream_t s);
void launch_pk_wrap(const State& st, const Cell* cells, const int* reb, hipStream_t s);
void launch_pk_nbr(const State& st, const Cell* cells, const int* sys_start, const int4* ext, const int* reb, double rs,
                   hipStream_t s);   // the skin list only (launch_sublists follows)
// fuse = 1: also the charge solve's start from the guess in x (launch_qeq_guess before it), finished by launch_qeq_init_fused
void launch_qeq_build(const State& st, const Cell& c, const Globals& g, const Tables& t, QeqBuffers& qb, int fuse, hipStream_t s);
inline int qeq_build_blocks(int n) { return (int)(((long long)n * 64 + 255) / 256); }
void launch_qeq_guess(const State& st, QeqBuffers& qb, int use_hist, hipStream_t s);
void launch_qeq_init_fused(const State& st, QeqBuffers& qb, int imax, double tol, hipStream_t s);
// census of the non-bonded cut-off decision (st.cen, category kCenNonbonded)
void launch_census_nb(const State& st, const Globals& g, hipStream_t s);
// Non-bonded terms over the charge-matrix rows instead of the skin list: valid while the rows belong to the current positions,
// carry keys, and the matrix cutoff covers nonb_cut.
void launch_nonbonded_rows(Precision p, const State& st, const Globals& g, const Tables& t, const QeqBuffers& qb, hipStream_t s);
void launch_qeq_matvec1(const State& st, const QeqBuffers& qb, const double* x, double* y, hipStream_t s);
void launch_qeq_init(const State& st, QeqBuffers& qb, int imax, double tol, int use_hist, hipStream_t s);
void launch_qeq_mvdir(const State& st, QeqBuffers& qb, int it, int imax, double tol, hipStream_t s);   // beta, d, q = A d, d.q partials
// alpha, x, r, p, r.p partials; gate: also, when both systems have stopped, the partials of the refinement's bound
void launch_qeq_update(const State& st, QeqBuffers& qb, int it, bool gate, hipStream_t s);
int qeq_gate_partials();
// refinement check when both systems have stopped before iteration it: the true residual b - (diag(eta) + H) x with the two-float
// matrix and each system's restart flag (slot `it` of the scalars); the next product takes them up (launch_qeq_mvdir_chk)
void launch_qeq_restart(const State& st, QeqBuffers& qb, int it, int imax, double tol, hipStream_t s);
void launch_qeq_mvdir_chk(const State& st, QeqBuffers& qb, int it, int imax, double tol, hipStream_t s);
int qeq_mv_partials(int n);                                                                             // partials per product
void launch_qeq_finish(const State& st, QeqBuffers& qb, hipStream_t s);

// ---- reductions and integration (k_md.hip)
void launch_energy_reduce(const State& st, double* out /*kTerms + 6 + 1*/, hipStream_t s);
struct MdBuffers {
  double *vx, *vy, *vz, *mass;   // per atom (mass from type)
  double* nh;                    // thermostat state (see k_md.hip)
  double *x0, *y0, *z0;          // positions at the last rebuild
  double* partial;               // reduction scratch
};
void launch_md_half_kick(const State& st, MdBuffers& md, double dtf, hipStream_t s);
void launch_md_drift(const State& st, MdBuffers& md, double dt, hipStream_t s);
void launch_md_ref_positions(const State& st, MdBuffers& md, hipStream_t s);
// fused step kernels: see k_md.hip
void launch_md_step_start(const State& st, MdBuffers& md, double dtf, double dt, bool thermostat, bool pending,
                          double* disp /* pinned: md_disp_partials() */, hipStream_t s);
int md_disp_partials();   // per-block partials of the kick-drift kernel's largest squared displacement
void launch_md_gather_step_end(const State& st, MdBuffers& md, double dtf, bool thermostat, hipStream_t s);
void launch_md_scale(const State& st, MdBuffers& md, hipStream_t s);
void launch_pk_ref(const State& st, MdBuffers& md, const int* reb, hipStream_t s);
void launch_pk_disp(const State& st, MdBuffers& md, const int* sys_start, int S, double lim, int* reb, int* any /* pinned */,
                    double* disp, hipStream_t s);
void launch_pk_thermostat(const State& st, MdBuffers& md, const int* sys_start, int S, double* nh_all, hipStream_t s);
void launch_pk_energy(const State& st, const int* sys_start, int S, double* out, hipStream_t s);

void launch_stream_copy(const void* src, void* dst, size_t bytes, hipStream_t s);   // bytes a multiple of 16

}  // namespace rxa
