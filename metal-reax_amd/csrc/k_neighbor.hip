// Neighbour search on the device: wrap into the cell, cell binning (stable radix sort of cell keys), and the full "skin" list of
// every owned atom: all images (j, s) with |x_j + s.L - x_i| <= nonb_cut + skin, in a deterministic order (cells in a fixed stencil
// order, atoms ascending inside a cell). One 64-lane wave per atom; the lanes test 64 candidates at once and compact the hits with a
// ballot, so the list is written in candidate order without atomics.
//
// Reference semantics: the far list of src/neighbor/neighbor.cpp:180-212 (pairs within the row cut-off, measured as x_j - x_i) over
// the image-expanded set of neighbor.cpp:18-88. Here both directions of every pair are kept (a full list), measured from the pair's
// canonical end (common.hpp), and the consumers apply their own cut-offs (nonb_cut, swb, bond_cut, hbond_cut) to that distance.
#include <hipcub/hipcub.hpp>

#include "common.hpp"
#include "launch.hpp"

namespace rxa {

namespace {

#pragma clang fp contract(off)
__global__ void k_wrap(State st, Cell c) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st.n) return;
  double r[3] = {st.x[i], st.y[i], st.z[i]};
  double k[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < 3; ++d)
    if (c.per[d]) k[d] = floor(frac_coord(c, d, r[0], r[1], r[2]));
  for (int d = 0; d < 3; ++d)
    if (k[d] != 0.0)
      for (int e = 0; e < 3; ++e) r[e] -= k[d] * c.v[d][e];
  st.x[i] = r[0];
  st.y[i] = r[1];
  st.z[i] = r[2];
  st.pos[i] = make_double4(r[0], r[1], r[2], pos_w(st, i));
}

// lattice shift vectors of all codes in [-smx, smx]^3, accumulated exactly as shift_vec does
__global__ void k_shift_table(Cell c, double4* shv, int smx0, int smx1, int smx2) {
  const int d0 = 2 * smx0 + 1, d1 = 2 * smx1 + 1, d2 = 2 * smx2 + 1;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= d0 * d1 * d2) return;
  const int s0 = k % d0 - smx0, s1 = (k / d0) % d1 - smx1, s2 = k / (d0 * d1) - smx2;
  double sx, sy, sz;
  shift_vec(c, shift_code(s0, s1, s2), sx, sy, sz);
  shv[k] = make_double4(sx, sy, sz, 0.0);
}
#pragma clang fp contract(on)

__global__ void k_pos4(State st) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st.n) return;
  st.pos[i] = make_double4(st.x[i], st.y[i], st.z[i], pos_w(st, i));
}

__global__ void k_cell_keys(State st, Cell c, int nc0, int nc1, int nc2, unsigned* keys, int* idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st.n) return;
  const int nc[3] = {nc0, nc1, nc2};
  int q[3];
  for (int d = 0; d < 3; ++d) {
    const double f = frac_coord(c, d, st.x[i], st.y[i], st.z[i]);
    int t = (int)floor(f * nc[d]);
    q[d] = t < 0 ? 0 : (t >= nc[d] ? nc[d] - 1 : t);
  }
  keys[i] = (unsigned)((q[2] * nc1 + q[1]) * nc0 + q[0]);
  idx[i] = i;
}

__global__ void k_fill_int(int* p, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_flags_out(const int* flags, int* host) {
  if (threadIdx.x < 8) host[threadIdx.x] = flags[threadIdx.x];
}

__global__ void k_cell_ranges(int n, const unsigned* skeys, int* cstart, int* cend, unsigned* atom_key, const int* sidx) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const unsigned k = skeys[p];
  if (p == 0 || skeys[p - 1] != k) cstart[k] = p;
  if (p == n - 1 || skeys[p + 1] != k) cend[k] = p + 1;
  atom_key[sidx[p]] = k;
}

// Lower bound of the distance between an atom and a block of the periodic cell (another image of the cell, or a neighbouring
// search cell), given per direction as gap[d], the perpendicular distance to the block's nearer face (0 inside its slab): the
// faces' normals are orthogonal in an untilted cell, where the gaps add in squares; otherwise the largest holds.
__device__ inline double block_gap2(bool ortho, const double gap[3]) {
  const double a = gap[0] * gap[0], b = gap[1] * gap[1], c = gap[2] * gap[2];
  return ortho ? a + b + c : fmax(a, fmax(b, c));
}
__device__ inline bool untilted(const Cell& c) { return c.v[1][0] == 0.0 && c.v[2][0] == 0.0 && c.v[2][1] == 0.0; }
constexpr double kGapSlack = 1e-6;   // subtracted from every gap (Angstrom): far above the rounding of wrapped coordinates

// One wave per atom. The 27 cells of the stencil are looked at by 27 lanes at once (image, range of atoms, distance of the cell
// from the atom); the cells within the list radius are then searched one after another, 64 atoms at a time, in stencil order.
// Bound by vector issue (a chunk of 64 candidates costs about 100 instructions). At 24,000 atoms (cells of 12.4 A, radius 12 A)
// 19 of the 27 cells remain, and the sub-lists are filled from the distances at hand: 222 us, against 261 us with all cells and
// 107 us for the sub-lists in a pass of their own.
// (sidx: atoms in the order of their cells; null when the atoms themselves are in that order)
__global__ void __launch_bounds__(256) k_nbr_cells(State st, Globals g, Tables t, Cell c, int nc0, int nc1, int nc2, const int* sidx,
                                                   const int* cstart, const int* cend, const unsigned* atom_key, double rs2, SubCut cut) {
  const int i = wave_atom();
  if (i >= st.n) return;
  const int lane = lane_id();
  const double4 pi = st.pos[i];
  ListRow row = list_row(st, g, t, i);
  // this lane's cell
  int first = 0, last = 0, code = 0;
  bool near = false;
  if (lane < 27) {
    const int nc[3] = {nc0, nc1, nc2}, off[3] = {lane % 3 - 1, lane / 3 % 3 - 1, lane / 9 - 1};
    const unsigned key = atom_key[i];
    const int home[3] = {(int)(key % (unsigned)nc0), (int)((key / (unsigned)nc0) % (unsigned)nc1), (int)(key / (unsigned)(nc0 * nc1))};
    int q[3], s[3];
    double gap[3];
    for (int d = 0; d < 3; ++d) {
      q[d] = home[d] + off[d];
      s[d] = q[d] < 0 ? -1 : (q[d] >= nc[d] ? 1 : 0);
      q[d] -= s[d] * nc[d];
      const double u = fmin(fmax(frac_coord(c, d, pi.x, pi.y, pi.z) * nc[d] - home[d], 0.0), 1.0);   // place within the home cell
      gap[d] = off[d] == 0 ? 0.0 : fmax((off[d] < 0 ? u : 1.0 - u) * (c.h[d] / nc[d]) - kGapSlack, 0.0);
    }
    const int cell = (q[2] * nc1 + q[1]) * nc0 + q[0];
    first = cstart[cell];
    last = cend[cell];
    code = shift_code(s[0], s[1], s[2]);
    near = first < last && block_gap2(untilted(c), gap) <= rs2;
  }
  for (unsigned long long left = __ballot(near); left; left &= left - 1) {
    const int from = __ffsll((long long)left) - 1;
    const int pe = __builtin_amdgcn_readlane(last, from), sc = __builtin_amdgcn_readlane(code, from);
    // the image's shift vector is the same for the whole cell; the list radius lies a skin beyond every consumer's cut-off, so
    // the test takes the image from this side (no canonical orientation) and only kept entries need the tags that decide
    // their canonical end
    const double4 S = st.shv[pos_sys(pi.w) * st.shv_stride + shift_index(st, sc)];
    for (int p0 = __builtin_amdgcn_readlane(first, from); p0 < pe; p0 += 64) {
      const int p = p0 + lane;
      bool keep = false;
      int j = 0, tj = -1;
      double d2 = 0;
      if (p < pe) {
        j = sidx ? sidx[p] : p;
        if (!(j == i && sc == 0)) {
          const double4 pj = st.pos[j];
          const double ex = (pj.x + S.x) - pi.x, ey = (pj.y + S.y) - pi.y, ez = (pj.z + S.z) - pi.z;
          d2 = ex * ex + ey * ey + ez * ez;
          keep = d2 <= rs2;
          tj = pos_type(pj.w);
        }
      }
      append_entries(st, t, cut, row, keep, j, sc, tj, d2);
    }
  }
  close_skin(st, row);
  close_sub(st, row);
}

// Direct search for cells narrower than three list radii: one wave per atom over the images of the cell in shift order, 64 images
// at a time: each lane takes one image and keeps it if the image of the cell comes within the list radius of the atom; the
// atoms of the kept images are then searched as one sequence (image by image, atoms ascending), 64 at a time, so small cells
// fill the wave with several images. The shift table enumerates every image that could matter to any atom; for one atom most
// are out of reach (31 A cell, 12 A radius: 6 of 125 remain). Bound by the serial walk of a wave over its candidates: 3000 atoms in
// a 31 A cell 185 us (3522 us over all images and with the canonical orientation formed for every candidate), 24 atoms in a
// 6.2 A cell 32 us (163).
constexpr int kBruteWaves = 4;
__global__ void __launch_bounds__(64 * kBruteWaves) k_nbr_brute(State st, Globals g, Tables t, Cell c, int sm0, int sm1, int sm2, double rs2,
                                                                SubCut cut) {
  __shared__ int codes_[kBruteWaves][64];
  const int i = wave_atom();
  if (i >= st.n) return;
  const int lane = lane_id(), n = st.n;
  int* codes = codes_[threadIdx.x >> 6];
  const double4 pi = st.pos[i];
  ListRow row = list_row(st, g, t, i);
  const int w[3] = {2 * sm0 + 1, 2 * sm1 + 1, 2 * sm2 + 1};
  const int images = w[0] * w[1] * w[2];
  const bool ortho = untilted(c);
  double f[3];
  for (int d = 0; d < 3; ++d) f[d] = frac_coord(c, d, pi.x, pi.y, pi.z);
  for (int m0 = 0; m0 < images; m0 += 64) {
    const int m = m0 + lane;
    const int s[3] = {m % w[0] - sm0, m / w[0] % w[1] - sm1, m / (w[0] * w[1]) - sm2};
    bool near = m < images;
    if (near) {
      double gap[3];
      for (int d = 0; d < 3; ++d) gap[d] = s[d] == 0 ? 0.0 : fmax((s[d] > 0 ? s[d] - f[d] : f[d] - s[d] - 1.0) * c.h[d] - kGapSlack, 0.0);
      near = block_gap2(ortho, gap) <= rs2;
    }
    const unsigned long long mk = __ballot(near);
    __builtin_amdgcn_wave_barrier();
    if (near) codes[lanes_below(mk)] = shift_code(s[0], s[1], s[2]);
    __builtin_amdgcn_wave_barrier();
    const int total = __popcll(mk) * n;
    int q = lane / n, j = lane % n;   // this lane's image and atom of the sequence
    for (int k = lane; k - lane < total; k += 64) {
      bool keep = false;
      int sc = 0, tj = -1;
      double d2 = 0;
      if (k < total) {
        sc = codes[q];
        if (!(j == i && sc == 0)) {
          const double4 pj = st.pos[j], S = st.shv[pos_sys(pi.w) * st.shv_stride + shift_index(st, sc)];
          const double ex = (pj.x + S.x) - pi.x, ey = (pj.y + S.y) - pi.y, ez = (pj.z + S.z) - pi.z;
          d2 = ex * ex + ey * ey + ez * ez;
          keep = d2 <= rs2;
          tj = pos_type(pj.w);
        }
      }
      append_entries(st, t, cut, row, keep, j, sc, tj, d2);
      j += 64;
      if (j >= n) { q += j / n; j %= n; }
    }
  }
  close_skin(st, row);
  close_sub(st, row);
}

// Bond and H-bond candidate sub-lists of the skin list (entry order kept): candidates within bond_cut + skin of every typed atom,
// and for H-bond donors (p_hbond 1) the acceptors (p_hbond 2) within hbond_cut + skin. Per-step kernels scan
// these instead of the whole skin list and apply the exact cut-offs to the current distance. The single-system searches above
// fill them along with the skin list; this pass lists them from it with packed systems, and again when a sub-list's capacity has
// grown. Entries two chunks ahead and positions one chunk ahead are loaded while a chunk is tested (the walk is latency-bound).
__global__ void __launch_bounds__(256) k_sublists(State st, Globals g, Tables t, SubCut cut) {
  const int i = wave_atom();
  if (i >= st.n) return;
  const int lane = lane_id();
  ListRow row = list_row(st, g, t, i);
  const double4 pi = st.pos[i];
  const double4* __restrict__ shv = st.shv + (size_t)pos_sys(pi.w) * st.shv_stride;
  const int* __restrict__ lj = st.nb_j + (size_t)i * st.maxnb;
  const int* __restrict__ ls = st.nb_s + (size_t)i * st.maxnb;
  const int cnt = row.ti >= 0 ? min(st.nb_cnt[i], st.maxnb) : 0;
  int jB = i, eB = 0, jC = i, eC = 0;   // lanes past the row's end carry the row atom itself, never listed
  if (lane < cnt) { jC = lj[lane]; eC = ls[lane]; }
  double4 pC = st.pos[jC];
  if (64 + lane < cnt) { jB = lj[64 + lane]; eB = ls[64 + lane]; }
  for (int k0 = 0; k0 < cnt; k0 += 64) {
    const int k = k0 + lane;
    const int j = jC, e = eC;
    const double4 pj = pC;
    jC = jB; eC = eB;
    if (k0 + 64 < cnt) pC = st.pos[jC];
    jB = i; eB = 0;
    if (k + 128 < cnt) { jB = lj[k + 128]; eB = ls[k + 128]; }
    // list radii with a skin beyond the consumers' cut-offs: the image from this side, no canonical orientation
    const double4 S = shv[shift_index(st, entry_code(e))];
    const double ex = (pj.x + S.x) - pi.x, ey = (pj.y + S.y) - pi.y, ez = (pj.z + S.z) - pi.z;
    append_sub(st, t, cut, row, k < cnt, j, e, pos_type(pj.w), ex * ex + ey * ey + ez * ez);
  }
  close_sub(st, row);
}

// Acceptor lists as the transpose of the donor lists: every donor candidate slot (flat index j * maxhc + h) is appended to its
// acceptor's row in arrival order (an integer atomic claims the position), then each row is put in ascending slot order by
// rank counting (the slot indices are distinct), so the acceptor's later force gather runs in a fixed order.
__global__ void __launch_bounds__(256) k_hc_transpose(State st, Globals g, Tables t) {
  const int j = wave_atom();
  if (j >= st.n) return;
  const int tj = st.type[j];
  if (tj < 0 || t.sp[tj].p_hbond != 1) return;
  const int nc = min(st.hc_cnt[j], st.maxhc);
  const size_t jb = (size_t)j * st.maxhc;
  for (int h = lane_id(); h < nc; h += 64) {
    const int k = st.hc_j[jb + h];
    const int p = atomicAdd(&st.hc_cnt[k], 1);
    if (p < st.maxhc) st.hc_m[(size_t)k * st.maxhc + p] = (int)(jb + h);
    else atomicMax(&st.flags[5], p + 1);
  }
}

// (kLds: the row's keys staged in the wave's share of dynamic LDS, maxhc ints per wave, so the rank loop reads LDS broadcasts;
// rows too long for LDS read the keys from global memory)
// Each pass over the keys ranks four of the lane's keys (a row of up to 256 slots takes one pass).
template <bool kLds>
__global__ void __launch_bounds__(256) k_hc_sort(State st, Globals g, Tables t) {
  extern __shared__ int hc_keys[];
  const int k = wave_atom();
  if (k >= st.n) return;
  const int tk = st.type[k];
  if (tk < 0 || t.sp[tk].p_hbond != 2) return;
  const int m = min(st.hc_cnt[k], st.maxhc);
  const size_t kb = (size_t)k * st.maxhc;
  const int* keys = st.hc_m + kb;
  if (kLds) {
    int* lk = hc_keys + (threadIdx.x >> 6) * st.maxhc;
    for (int h = lane_id(); h < m; h += 64) lk[h] = st.hc_m[kb + h];
    __builtin_amdgcn_wave_barrier();
    keys = lk;
  }
  constexpr int kEach = 4;
  for (int h0 = lane_id(); h0 - lane_id() < m; h0 += 64 * kEach) {
    int key[kEach], rank[kEach];
    for (int u = 0; u < kEach; ++u) { key[u] = h0 + 64 * u < m ? keys[h0 + 64 * u] : 0; rank[u] = 0; }
#pragma unroll 4
    for (int q = 0; q < m; ++q) {
      const int other = keys[q];
      for (int u = 0; u < kEach; ++u) rank[u] += other < key[u] ? 1 : 0;
    }
    for (int u = 0; u < kEach; ++u)
      if (h0 + 64 * u < m) st.hc_j[kb + rank[u]] = key[u];
  }
}

// Gather of every persistent per-atom array into a new atom order: new[i] = old[src[i]] (through a scratch area, one kernel to
// gather, one to copy back). Used to keep atoms in cell order (spatial locality of every neighbour gather) and to carry state
// across a change of the caller's atom order.
__global__ void k_permute_gather(PermuteSet ps, const int* src, double* sd, int* si, long long* sl) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ps.n) return;
  const int j = src[i];
  for (int k = 0; k < ps.nd; ++k) sd[(size_t)k * ps.n + i] = ps.d[k][j];
  for (int k = 0; k < ps.ni; ++k) si[(size_t)k * ps.n + i] = ps.i[k][j];
  for (int k = 0; k < ps.nl; ++k) sl[(size_t)k * ps.n + i] = ps.l[k][j];
}

__global__ void k_permute_scatter(PermuteSet ps, const double* sd, const int* si, const long long* sl) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ps.n) return;
  for (int k = 0; k < ps.nd; ++k) ps.d[k][i] = sd[(size_t)k * ps.n + i];
  for (int k = 0; k < ps.ni; ++k) ps.i[k][i] = si[(size_t)k * ps.n + i];
  for (int k = 0; k < ps.nl; ++k) ps.l[k][i] = sl[(size_t)k * ps.n + i];
}

// positions from a caller's device arrays (x[n], y[n], z[n] in the caller's order) into the engine's order
__global__ void k_positions_in(State st, const double* ux, const int* perm) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st.n) return;
  const int u = perm[i];
  const double x = ux[u], y = ux[st.n + u], z = ux[2 * (size_t)st.n + u];
  st.x[i] = x; st.y[i] = y; st.z[i] = z;
  st.pos[i] = make_double4(x, y, z, pos_w(st, i));
}

inline int blocks_for(long long items, int per_block) { return (int)((items + per_block - 1) / per_block); }

}  // namespace

void launch_wrap(const State& st, const Cell& c, hipStream_t s) {
  if (st.n == 0) return;
  hipLaunchKernelGGL(k_wrap, dim3(blocks_for(st.n, 256)), dim3(256), 0, s, st, c);
}

void launch_permute(const PermuteSet& ps, const int* src, double* sd, int* si, long long* sl, hipStream_t s) {
  if (ps.n == 0) return;
  hipLaunchKernelGGL(k_permute_gather, dim3(blocks_for(ps.n, 256)), dim3(256), 0, s, ps, src, sd, si, sl);
  hipLaunchKernelGGL(k_permute_scatter, dim3(blocks_for(ps.n, 256)), dim3(256), 0, s, ps, sd, si, sl);
}

void launch_positions_in(const State& st, const double* ux, const int* perm, hipStream_t s) {
  hipLaunchKernelGGL(k_positions_in, dim3(blocks_for(st.n, 256)), dim3(256), 0, s, st, ux, perm);
}

void launch_pos4(const State& st, hipStream_t s) {
  if (st.n == 0) return;
  hipLaunchKernelGGL(k_pos4, dim3(blocks_for(st.n, 256)), dim3(256), 0, s, st);
}

void launch_shift_table(const Cell& c, double4* shv, const int smx[3], hipStream_t s) {
  const int m = (2 * smx[0] + 1) * (2 * smx[1] + 1) * (2 * smx[2] + 1);
  hipLaunchKernelGGL(k_shift_table, dim3(blocks_for(m, 256)), dim3(256), 0, s, c, shv, smx[0], smx[1], smx[2]);
}

SubCut sub_cut(double rb, double rh) {
  const double m = 1.0 + 1e-12;
  return SubCut{rb * rb * m, rh * rh * m};
}

void launch_sublists(const State& st, const Globals& g, const Tables& t, double rb, double rh, hipStream_t s) {
  hipLaunchKernelGGL(k_sublists, dim3(blocks_for((long long)st.n * 64, 256)), dim3(256), 0, s, st, g, t, sub_cut(rb, rh));
}

void launch_acceptor_rows(const State& st, const Globals& g, const Tables& t, hipStream_t s) {
  if (!(g.hbond_cut > 0)) return;
  const dim3 grid(blocks_for((long long)st.n * 64, 256)), blk(256);
  hipLaunchKernelGGL(k_hc_transpose, grid, blk, 0, s, st, g, t);
  const size_t lds = 4 * (size_t)st.maxhc * sizeof(int);   // four waves per block
  if (lds <= 64 * 1024) hipLaunchKernelGGL(k_hc_sort<true>, grid, blk, lds, s, st, g, t);
  else hipLaunchKernelGGL(k_hc_sort<false>, grid, blk, 0, s, st, g, t);
}

void launch_fill_int(int* p, int n, int v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_int, dim3(blocks_for(n, 256)), dim3(256), 0, s, p, n, v);
}

void launch_flags_out(const int* flags, int* host, hipStream_t s) {
  hipLaunchKernelGGL(k_flags_out, dim3(1), dim3(64), 0, s, flags, host);
}

size_t bin_temp_bytes(int n) {
  size_t bytes = 0;
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const unsigned*)nullptr, (unsigned*)nullptr, (const int*)nullptr, (int*)nullptr, n);
  return bytes;
}

void launch_bin(const State& st, const Cell& c, const BinGrid& g, BinBuffers& b, hipStream_t s) {
  const int n = st.n;
  hipLaunchKernelGGL(k_cell_keys, dim3(blocks_for(n, 256)), dim3(256), 0, s, st, c, g.nc[0], g.nc[1], g.nc[2], b.keys, b.idx);
  size_t bytes = b.temp_bytes;
  int bits = 1;
  while ((1u << bits) < (unsigned)g.ncells()) ++bits;
  (void)hipcub::DeviceRadixSort::SortPairs(b.temp, bytes, b.keys, b.skeys, b.idx, b.sidx, n, 0, bits, s);
  launch_fill_int(b.cstart, g.ncells(), 0, s);
  launch_fill_int(b.cend, g.ncells(), 0, s);
  hipLaunchKernelGGL(k_cell_ranges, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, b.skeys, b.cstart, b.cend, b.atom_key, b.sidx);
}

void launch_nbr_cells(const State& st, const Globals& gl, const Tables& t, const Cell& c, const BinGrid& g, const BinBuffers& b, bool sorted,
                      double rs, double rb, double rh, hipStream_t s) {
  hipLaunchKernelGGL(k_nbr_cells, dim3(blocks_for((long long)st.n * 64, 256)), dim3(256), 0, s, st, gl, t, c, g.nc[0], g.nc[1], g.nc[2],
                     sorted ? (const int*)nullptr : (const int*)b.sidx, b.cstart, b.cend,
                     (const unsigned*)(sorted ? b.skeys : b.atom_key), rs * rs, sub_cut(rb, rh));
}

void launch_nbr_brute(const State& st, const Globals& g, const Tables& t, const Cell& c, const int sm[3], double rs, double rb, double rh,
                      hipStream_t s) {
  // (the image is taken from the listing atom's side: the slack keeps every pair the canonical side has within the radius)
  hipLaunchKernelGGL(k_nbr_brute, dim3(blocks_for(st.n, kBruteWaves)), dim3(64 * kBruteWaves), 0, s, st, g, t, c, sm[0], sm[1], sm[2],
                     rs * rs * (1.0 + 1e-12), sub_cut(rb, rh));
}

}  // namespace rxa
