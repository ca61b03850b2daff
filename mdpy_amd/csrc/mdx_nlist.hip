// Wrapping, mdpy-compatible cell binning, and the per-atom neighbour list (gfx950).
//
// Reference behaviour restated here:
//   wrap_positions            mdpy/utils/pbc.py:28-36
//   CellList grid + binning   mdpy/core/cell_list.py:56-116
//   27-cell stencil           mdpy/constraint/__init__.py:12-19 and
//                             mdpy/constraint/charmm_nonbonded_constraint.py:75-100
// The force kernels do not walk the reference's dense cell table: atoms are binned into a
// periodic grid of cells at least (rc + skin)/2 wide, sorted by cell (ascending original id
// inside a cell, so every order is deterministic), and each atom gets a full neighbour list
// (one row of entries per atom). In REFERENCE mode the list also drops
// pairs whose mdpy cells are not stencil neighbours, reproducing the reference's pair set.
#include "mdx_internal.h"
#include <algorithm>
#include <cmath>

#define NL_BLOCK 256

// ============================================================== wrap / reference binning
__global__ void k_wrap(double* __restrict__ pos, int n, double Lx, double Ly, double Lz, double ix,
                       double iy, double iz, DevState* st) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double L[3] = {Lx, Ly, Lz}, inv[3] = {ix, iy, iz};
  bool lost = false;
  double out[3];
  for (int d = 0; d < 3; ++d) {
    double x = pos[3 * i + d];
    double m = -rint(x * inv[d]);  // np.round: half to even
    if (fabs(m) >= 2.0) lost = true;
    out[d] = x + m * L[d];
  }
  if (lost) {
    atomicOr(&st->flags, MDX_FLAG_LOSS);
    return;
  }
  for (int d = 0; d < 3; ++d) pos[3 * i + d] = out[d];
}

__global__ void k_minpos(const double* __restrict__ pos, int n, DevState* st) {
  __shared__ unsigned long long sm[3][NL_BLOCK / 64];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long e[3] = {~0ull, ~0ull, ~0ull};
  if (i < n)
    for (int d = 0; d < 3; ++d) e[d] = enc_double_order(pos[3 * i + d]);
  for (int d = 0; d < 3; ++d) {
    unsigned long long v = e[d];
    for (int off = 32; off > 0; off >>= 1) {
      unsigned long long o = __shfl_xor(v, off, 64);
      v = o < v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) sm[d][threadIdx.x >> 6] = v;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned long long v = ~0ull;
    for (int w = 0; w < NL_BLOCK / 64; ++w) v = sm[threadIdx.x][w] < v ? sm[threadIdx.x][w] : v;
    atomicMin(&st->minpos[threadIdx.x], v);
  }
}

__global__ void k_ref_bin(const double* __restrict__ pos, int n, int nx, int ny, int nz, double ix,
                          double iy, double iz, DevState* st, int* __restrict__ cell_index,
                          int* __restrict__ cell_lin, int* __restrict__ counts) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double mn[3] = {dec_double_order(st->minpos[0]), dec_double_order(st->minpos[1]),
                  dec_double_order(st->minpos[2])};
  double inv[3] = {ix, iy, iz};
  int nn[3] = {nx, ny, nz};
  int c[3];
  for (int d = 0; d < 3; ++d) {
    double s = (pos[3 * i + d] - mn[d]) * inv[d];  // (x - min x) . cell_inv, diagonal
    const double f = floor(s);
    // range decided before the conversion (NaN or runaway positions flag and clamp)
    if (!(f >= 0.0 && f < (double)nn[d])) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
    const int k = clamped_floor_index(f, nn[d]);
    c[d] = k;
    if (cell_index) cell_index[3 * i + d] = k;
  }
  int lin = (c[0] * ny + c[1]) * nz + c[2];
  if (cell_lin) cell_lin[i] = lin;
  int cnt = atomicAdd(&counts[lin], 1) + 1;
  atomicMax(&st->maxpc, cnt);
}

__global__ void k_ref_scatter(const int* __restrict__ cell_lin, int n, int* __restrict__ cursor,
                              int* __restrict__ table, int maxpc) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int c = cell_lin[i];
  int slot = atomicAdd(&cursor[c], 1);
  if (slot < maxpc) table[(long long)c * maxpc + slot] = i;
}

// Sort each row ascending (bitonic sort in LDS); entries >= valid are padding -1.
__global__ void k_sort_rows(int* __restrict__ table, const int* __restrict__ counts, int width) {
  __shared__ int buf[SORT_MAX];
  int row = blockIdx.x;
  int cnt = counts[row];
  int P = 1;
  while (P < cnt) P <<= 1;
  for (int t = threadIdx.x; t < P; t += blockDim.x)
    buf[t] = t < cnt ? table[(long long)row * width + t] : 0x7fffffff;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < P; t += blockDim.x) {
        int u = t ^ j;
        if (u > t) {
          bool up = (t & k) == 0;
          int a = buf[t], b = buf[u];
          if ((a > b) == up) {
            buf[t] = b;
            buf[u] = a;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int t = threadIdx.x; t < width; t += blockDim.x)
    table[(long long)row * width + t] = t < cnt ? buf[t] : -1;
}

__global__ void k_fill_i32(int* __restrict__ p, int v, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// reset the reference-binning reductions (minimum position per axis, largest population,
// flags) and the per-cell counts
__global__ void k_ref_reset(DevState* st, int* __restrict__ counts, int nc) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nc) counts[i] = 0;
  if (i == 0) {
    st->minpos[0] = st->minpos[1] = st->minpos[2] = ~0ull;
    st->maxpc = 0;
    st->flags = 0;
  }
}

extern "C" int mdx_wrap_positions(mdx_ctx* c) {
  MDX_CHECK(c && c->pos, MDX_ERR_INVALID, "mdx_wrap_positions: no system bound");
  MDX_ENTER();
  c->forces_current = false;
  double inv[3];
  for (int d = 0; d < 3; ++d) inv[d] = 1.0 / c->box[d];
  MDX_HIP(hipMemsetAsync(&c->dstate.p->flags, 0, sizeof(unsigned), c->stream));
  k_wrap<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(c->pos, c->n, c->box[0], c->box[1], c->box[2],
                                                            inv[0], inv[1], inv[2], c->dstate.p);
  MDX_LAUNCH_CHECK();
  unsigned flags = 0;
  MDX_HIP(hipMemcpyAsync(&flags, &c->dstate.p->flags, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream));
  MDX_HIP(hipStreamSynchronize(c->stream));
  int h1 = 1;
  MDX_HIP(hipMemcpy(&c->dstate.p->rebuild, &h1, sizeof(int), hipMemcpyHostToDevice));
  MDX_CHECK(!(flags & MDX_FLAG_LOSS), MDX_ERR_PARTICLE_LOSS, "atom(s) moved beyond 2 PBC images");
  MDX_LEAVE_RET(0);
}

// Reference grid for a cell-list cutoff (cell_list.py:74-81).
void mdx_ref_grid(const double* box, double rc, int* n, double* w, double* inv) {
  for (int d = 0; d < 3; ++d) {
    int k = (int)std::floor((box[d] + 2.0) / rc);
    if (k < 3) k = 3;
    n[d] = k;
    w[d] = (box[d] + 2.0) / (double)k;
    inv[d] = 1.0 / w[d];
  }
}

static int ref_bin_enqueue(mdx_ctx* c, double cell_cutoff, int* d_cell_index) {
  mdx_ref_grid(c->box, cell_cutoff, c->ref_n, c->ref_w, c->ref_inv);
  int nc = c->ref_n[0] * c->ref_n[1] * c->ref_n[2];
  int rc;
  if ((rc = c->ref_cell_lin.ensure(c->n))) return rc;
  if ((rc = c->ref_counts.ensure(nc))) return rc;
  if ((rc = c->ref_cursor.ensure(nc))) return rc;
  k_ref_reset<<<div_up(nc, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(c->dstate.p, c->ref_counts.p, nc);
  MDX_LAUNCH_CHECK();
  k_minpos<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(c->pos, c->n, c->dstate.p);
  MDX_LAUNCH_CHECK();
  k_ref_bin<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(
      c->pos, c->n, c->ref_n[0], c->ref_n[1], c->ref_n[2], c->ref_inv[0], c->ref_inv[1], c->ref_inv[2],
      c->dstate.p, d_cell_index, c->ref_cell_lin.p, c->ref_counts.p);
  MDX_LAUNCH_CHECK();
  return 0;
}

extern "C" int mdx_celllist_reference(mdx_ctx* c, double cell_cutoff, int* d_cell_index, int* h_n, int* h_maxpc) {
  MDX_CHECK(c && c->pos, MDX_ERR_INVALID, "mdx_celllist_reference: no system bound");
  MDX_CHECK(cell_cutoff > 0, MDX_ERR_CELL_CUTOFF, "cutoff radius is poor defined");
  for (int d = 0; d < 3; ++d)
    MDX_CHECK(std::floor(c->box[d] / cell_cutoff) >= 2, MDX_ERR_CELL_CUTOFF,
              "the cutoff_radius is too large to create cell list");
  MDX_ENTER();
  MDX_HIP(hipMemsetAsync(&c->dstate.p->flags, 0, sizeof(unsigned), c->stream));
  int rc = ref_bin_enqueue(c, cell_cutoff, d_cell_index);
  if (rc) return rc;
  int maxpc = 0;
  unsigned flags = 0;
  MDX_HIP(hipMemcpyAsync(&maxpc, &c->dstate.p->maxpc, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  MDX_HIP(hipMemcpyAsync(&flags, &c->dstate.p->flags, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream));
  MDX_HIP(hipStreamSynchronize(c->stream));
  MDX_CHECK(!(flags & MDX_FLAG_OVERFLOW), MDX_ERR_OVERFLOW, "reference binning produced an out-of-range cell");
  for (int d = 0; d < 3; ++d) h_n[d] = c->ref_n[d];
  *h_maxpc = maxpc;
  MDX_LEAVE_RET(0);
}

extern "C" int mdx_celllist_table(mdx_ctx* c, int* d_table, int maxpc) {
  MDX_CHECK(c && d_table && maxpc > 0, MDX_ERR_INVALID, "mdx_celllist_table: bad arguments");
  MDX_CHECK(maxpc <= SORT_MAX * 8, MDX_ERR_OVERFLOW, "cell population %d too large", maxpc);
  int nc = c->ref_n[0] * c->ref_n[1] * c->ref_n[2];
  MDX_CHECK(nc > 0, MDX_ERR_INVALID, "mdx_celllist_table before mdx_celllist_reference");
  MDX_CHECK(maxpc <= SORT_MAX, MDX_ERR_OVERFLOW, "cell population %d exceeds %d", maxpc, SORT_MAX);
  MDX_ENTER();
  MDX_HIP(hipMemsetAsync(c->ref_cursor.p, 0, nc * sizeof(int), c->stream));
  MDX_HIP(hipMemsetAsync(d_table, 0xff, (size_t)nc * maxpc * sizeof(int), c->stream));
  k_ref_scatter<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(c->ref_cell_lin.p, c->n, c->ref_cursor.p,
                                                                   d_table, maxpc);
  MDX_LAUNCH_CHECK();
  k_sort_rows<<<nc, 256, 0, c->stream>>>(d_table, c->ref_counts.p, maxpc);
  MDX_LAUNCH_CHECK();
  MDX_LEAVE_RET(0);
}

// ============================================================== neighbour-list grid

__global__ void k_check_disp(const double* __restrict__ pos, const double* __restrict__ pos_build, int n,
                             double Lx, double Ly, double Lz, DevState* st) {
  __shared__ double sm[NL_BLOCK / 64];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d2 = 0.0;
  bool bad = false;
  if (i < n) {
    double L[3] = {Lx, Ly, Lz};
    for (int d = 0; d < 3; ++d) {
      double x = pos[3 * i + d];
      if (!isfinite(x)) bad = true;
      double dd = x - pos_build[3 * i + d];
      dd -= L[d] * rint(dd / L[d]);
      d2 += dd * dd;
    }
  }
  if (bad) atomicOr(&st->flags, MDX_FLAG_NONFINITE);
  if (d2 != d2) d2 = INFINITY;  // a position that is not finite, now or at the build: the list is due
  for (int off = 32; off > 0; off >>= 1) d2 = fmax(d2, __shfl_xor(d2, off, 64));
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = 0;
    for (int w = 0; w < NL_BLOCK / 64; ++w) v = fmax(v, sm[w]);
    atomicMax(&st->max_disp2_bits, enc_double_order(v));
  }
}

struct GridArgs {
  int nx, ny, nz;
  double Lx, Ly, Lz;
  double wx, wy, wz;  // cell widths
};

// Each atom's cell and its place among the cell's atoms (any order: k_grid_sort_fill sorts). Atomics on
// few cells bound it, so a run of lanes in one cell counts with one, and the place it returns spares
// the scatter its own. 23,328 atoms, 512 cells (us, with the scatter): 21 -> 7.6, 30,021 atoms,
// 1,331 cells: 11.4 -> 7.3.
__global__ void k_grid_bin(const double* __restrict__ pos, int n, GridArgs g, const DevState* st, double thr2,
                           int* __restrict__ atom_cell, int* __restrict__ atom_place, int* __restrict__ cell_count) {
  if (!need_rebuild(st, thr2)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
  const int j = min(i, n - 1);  // every lane stays for the exchanges below
  double L[3] = {g.Lx, g.Ly, g.Lz}, w[3] = {g.wx, g.wy, g.wz};
  int nn[3] = {g.nx, g.ny, g.nz};
  int c[3];
  for (int d = 0; d < 3; ++d) {
    double x = pos[3 * j + d];
    x -= L[d] * floor(x / L[d]);
    c[d] = clamped_floor_index(x / w[d], nn[d]);
  }
  const int lin = i < n ? (c[0] * g.ny + c[1]) * g.nz + c[2] : -1;
  const int before = __shfl_up(lin, 1, 64);
  const unsigned long long heads = __ballot(lane == 0 || lin != before);  // first lanes of the runs
  const int head = 63 - __clzll(heads & (~0ull >> (63 - lane)));
  const unsigned long long later = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
  int base = 0;
  if (lane == head && i < n) base = atomicAdd(&cell_count[lin], (later ? __ffsll((long long)later) - 1 : 64) - lane);
  base = __shfl(base, head, 64);
  if (i >= n) return;
  atom_cell[i] = lin;
  atom_place[i] = base + lane - head;
}

// single-block exclusive scan over cells, with the check of the sort limit: a lane sums its run of
// cells, waves scan their lanes, every lane adds the waves before its own (one lane adding 1,024 sums
// took most of 12-13 us; 2.8 now)
#define SCAN_THREADS 1024
__global__ __launch_bounds__(SCAN_THREADS) void k_cell_scan(const int* __restrict__ cell_count, int* __restrict__ cell_start,
                                                            int ncell, DevState* st, double thr2) {
  if (!need_rebuild(st, thr2)) return;
  __shared__ int wsum[SCAN_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int per = (ncell + SCAN_THREADS - 1) / SCAN_THREADS;
  const int b = tid * per, e = min(ncell, b + per);
  int s = 0;
  bool over = false;
  for (int k = b; k < e; ++k) {
    const int v = cell_count[k];
    over |= v > SORT_MAX;
    s += v;
  }
  if (over) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
  int incl = s;
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, 64);
    if (lane >= off) incl += v;
  }
  if (lane == 63) wsum[tid >> 6] = incl;
  __syncthreads();
  int acc = incl - s;
  for (int w = 0; w < (tid >> 6); ++w) acc += wsum[w];
  for (int k = b; k < e; ++k) {
    cell_start[k] = acc;
    acc += cell_count[k];
  }
}

__global__ void k_grid_scatter(const int* __restrict__ atom_cell, const int* __restrict__ atom_place, int n,
                               const int* __restrict__ cell_start, int* __restrict__ sorted_orig, const DevState* st,
                               double thr2) {
  if (!need_rebuild(st, thr2)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  sorted_orig[cell_start[atom_cell[i]] + atom_place[i]] = i;
}

__global__ void k_grid_sort_fill(FillArgs f) {
  if (!need_rebuild(f.st, f.thr2)) return;
  grid_sort_fill_block(f, blockIdx.x);
}

FillArgs fill_args(mdx_ctx* c, double thr2) {
  FillArgs f;
  f.cell_start = c->cell_start.p;
  f.cell_count = c->cell_count.p;
  f.sorted_orig = c->sorted_orig.p;
  f.orig_sorted = c->orig_sorted.p;
  f.pos = c->pos;
  f.pos_build = c->pos_at_build.p;
  f.lj64 = c->has_lj ? c->lj64.p : nullptr;
  f.ljs = c->ljs.p;
  f.ljs14 = c->ljs14.p;
  const bool ref = c->pair_mode == MDX_PAIRS_REFERENCE;
  f.ref_lin = ref ? c->ref_cell_lin.p : nullptr;
  f.ref_cell_sorted = c->ref_cell_sorted.p;
  f.rny = c->ref_n[1];
  f.rnz = c->ref_n[2];
  f.st = c->dstate.p;
  f.thr2 = thr2;
  f.qs = c->has_charges ? c->charge_s.p : nullptr;
  f.xq = c->xq.p;
  f.xf = c->xf.p;
  f.pos_sorted = c->pos_sorted.p;
  for (int d = 0; d < 3; ++d) {
    f.L[d] = c->box[d];
    f.iL[d] = 1.0 / c->box[d];
  }
  f.ncell = c->ncell;
  return f;
}

// every evaluation: the sorted-order copies of pack_atom
__global__ void k_pack(FillArgs f, int n) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int o = f.sorted_orig[s];
  pack_atom(f.pos[3 * o], f.pos[3 * o + 1], f.pos[3 * o + 2], f.qs ? f.qs[o] : 0.f, f.L, f.iL, &f.xq[s], &f.xf[s],
            &f.pos_sorted[3 * s]);
}

struct ListArgs {
  GridArgs g;
  int n;
  int cap;
  float rl2;          // list radius squared (float pre-filter)
  double rc;
  int ref_mode;       // REFERENCE stencil filter
  int rnx, rny, rnz;  // reference grid
  int nstencil;
  int shifted;        // staged candidates are shifted into the home frame (no minimum image)
};

__device__ __forceinline__ int cyc_dist(int a, int b, int n) {
  int d = a > b ? a - b : b - a;
  return min(d, n - d);
}

// One workgroup per home cell: the candidates of every stencil cell (identical for all atoms of
// the home cell) are staged in LDS in chunks, then each NB_G-lane group scans them for one home
// atom at a time and compacts the accepted ones with a wave ballot. Same candidate order, hence
// the same lists, as a per-atom walk of the stencil; global memory is read once per cell. The
// next chunk's candidates are fetched into registers while the current one is scanned.
// Staged candidates are shifted into the home cell's periodic frame (when the stencil holds each
// periodic cell once, on no more than one side), so the scan needs no minimum-image arithmetic.
// Exclusions and 1-4 partners within 32 atom indices of the home atom are bits of two 64-bit
// masks; an atom with a partner outside that window scans its CSR lists (staged in LDS) instead.
// Each lane tests BL_U candidates per pass, all LDS reads issued first; r <= rc is decided in float64
// (lists without a skin). FAST instantiations (shifted candidates, exact pair mode, masks present)
// compile out the reference-mode filter and the minimum image.
#ifndef BL_CH
#define BL_CH 1024  // candidates staged per chunk (a multiple of the fast kernel's pass)
#endif
#define BL_MAXST 512
#define BL_MAXEX 32  // exclusions (and 1-4 partners) per atom
#define BL_HMAX 192  // home atoms staged in LDS (more: their data is read from global memory)
#define BL_POOL 1024 // exclusion / 1-4 entries of a cell's home atoms staged in LDS
#define BL_THREADS 512
#define BL_SLOTS ((BL_CH + BL_THREADS - 1) / BL_THREADS)  // staged candidates per lane per chunk
#define BL_U 4       // candidates per lane per pass
#define BL_WIN 32    // index window of the exclusion masks: partners i-32 .. i+31

// The arguments of one context's list-build launch (passed by value to the single-context
// kernels, or one replica's record of a batched launch).
struct ListCall {
  ListArgs a;
  const float4* xq;
  const int4* xf;
  const int* sorted_orig;
  const int* cell_start;
  const int* cell_count;
  const int* stencil;
  const int* excl_ptr;
  const int* excl_idx;
  const int* s14_ptr;
  const int* s14_idx;
  const unsigned long long* ex_win;
  const unsigned long long* s4_win;
  const unsigned char* win_bad;
  const int* ref_cell_sorted;
  const double* pos;
  int* nbr_count;
  unsigned* nbr_list;
  DevState* st;
  double thr2;
  int split;  // fast build: workgroups per home cell
};

// the build of home cell `cell`
template <bool FAST>
__device__ __forceinline__ void build_list_cell_body(const ListCall& L, const int cell) {
  const ListArgs& a = L.a;
  const float4* __restrict__ xq = L.xq;
  const int* __restrict__ sorted_orig = L.sorted_orig;
  const int* __restrict__ cell_start = L.cell_start;
  const int* __restrict__ cell_count = L.cell_count;
  const int* __restrict__ stencil = L.stencil;
  const int* __restrict__ excl_ptr = L.excl_ptr;
  const int* __restrict__ excl_idx = L.excl_idx;
  const int* __restrict__ s14_ptr = L.s14_ptr;
  const int* __restrict__ s14_idx = L.s14_idx;
  const unsigned long long* __restrict__ ex_win = L.ex_win;
  const unsigned long long* __restrict__ s4_win = L.s4_win;
  const unsigned char* __restrict__ win_bad = L.win_bad;
  const int* __restrict__ ref_cell_sorted = L.ref_cell_sorted;
  const double* __restrict__ pos = L.pos;
  int* __restrict__ nbr_count = L.nbr_count;
  unsigned* __restrict__ nbr_list = L.nbr_list;
  DevState* st = L.st;
  const double thr2 = L.thr2;
  if (!need_rebuild(st, thr2)) return;
  __shared__ float4 cxq[BL_CH];
  __shared__ int2 cto[BL_CH];      // (sorted slot, original atom id)
  __shared__ int cr[FAST ? 1 : BL_CH];
  __shared__ int sb[BL_MAXST], sp[BL_MAXST + 1];
  __shared__ unsigned char shc[BL_MAXST];  // periodic shift of each stencil cell: 2 bits per axis
  __shared__ int acnt[SORT_MAX];
  __shared__ int exl[BL_THREADS / NB_G][BL_MAXEX], s4l[BL_THREADS / NB_G][BL_MAXEX];
  // home atoms staged once per block: position, atom id, window masks, exclusion / 1-4 lists
  __shared__ float4 hxi[BL_HMAX];
  __shared__ int ho[BL_HMAX], hex0[BL_HMAX + 1], hs40[BL_HMAX + 1];
  __shared__ unsigned long long hexm[BL_HMAX], hs4m[BL_HMAX];
  __shared__ unsigned char hbad[BL_HMAX];
  __shared__ int pool_ex[BL_POOL], pool_s4[BL_POOL];
  __shared__ int fast;
  const GridArgs& gr = a.g;
  const int hb = cell_start[cell], hn = cell_count[cell];
  if (hn > SORT_MAX) {  // oversize cells are flagged where the cells are counted: empty lists
    for (int t = threadIdx.x; t < hn; t += blockDim.x) nbr_count[hb + t] = 0;
    return;
  }
  if (hn == 0) return;
  const int tid = threadIdx.x;
  const int hz = cell % gr.nz, hy = (cell / gr.nz) % gr.ny, hx = cell / (gr.nz * gr.ny);
  const bool shifted = FAST || a.shifted;
  for (int k = tid; k < a.nstencil; k += blockDim.x) {
    int p = stencil[k];
    int nx = hx + ((p >> 16) & 0xff) - 128, ny = hy + ((p >> 8) & 0xff) - 128, nz = hz + (p & 0xff) - 128;
    // a neighbour reached across the box edge is the periodic image one box length away
    // (code per axis: 0 = -L, 1 = 0, 2 = +L)
    const int cx = nx < 0 ? 0 : (nx >= gr.nx ? 2 : 1);
    const int cy = ny < 0 ? 0 : (ny >= gr.ny ? 2 : 1);
    const int cz = nz < 0 ? 0 : (nz >= gr.nz ? 2 : 1);
    shc[k] = (unsigned char)(cx | (cy << 2) | (cz << 4));
    nx += nx < 0 ? gr.nx : (nx >= gr.nx ? -gr.nx : 0);
    ny += ny < 0 ? gr.ny : (ny >= gr.ny ? -gr.ny : 0);
    nz += nz < 0 ? gr.nz : (nz >= gr.nz ? -gr.nz : 0);
    const int nc = (nx * gr.ny + ny) * gr.nz + nz;
    sb[k] = cell_start[nc];
    sp[k + 1] = cell_count[nc];
  }
  for (int j = tid; j < hn; j += blockDim.x) acnt[j] = 0;
  const bool fit = hn <= BL_HMAX;
  if (fit) {
    for (int h = tid; h < hn; h += blockDim.x) {
      const int o = sorted_orig[hb + h];
      ho[h] = o;
      hxi[h] = xq[hb + h];
      hex0[h + 1] = excl_ptr ? excl_ptr[o + 1] - excl_ptr[o] : 0;
      hs40[h + 1] = s14_ptr ? s14_ptr[o + 1] - s14_ptr[o] : 0;
      hexm[h] = ex_win ? ex_win[o] : 0ull;
      hs4m[h] = s4_win ? s4_win[o] : 0ull;
      hbad[h] = win_bad ? win_bad[o] : (unsigned char)1;
    }
  }
  __syncthreads();
  if (tid == 0) {
    sp[0] = 0;
    for (int k = 0; k < a.nstencil; ++k) sp[k + 1] += sp[k];
    if (fit) {
      hex0[0] = 0;
      hs40[0] = 0;
      for (int h = 0; h < hn; ++h) {
        hex0[h + 1] += hex0[h];
        hs40[h + 1] += hs40[h];
      }
    }
    fast = fit && hex0[fit ? hn : 0] <= BL_POOL && hs40[fit ? hn : 0] <= BL_POOL;
  }
  __syncthreads();
  if (fast) {
    for (int h = tid; h < hn; h += blockDim.x) {
      const int o = ho[h];
      if (excl_ptr)
        for (int r = 0; r < hex0[h + 1] - hex0[h]; ++r) pool_ex[hex0[h] + r] = excl_idx[excl_ptr[o] + r];
      if (s14_ptr)
        for (int r = 0; r < hs40[h + 1] - hs40[h]; ++r) pool_s4[hs40[h] + r] = s14_idx[s14_ptr[o] + r];
    }
  }
  const int total = sp[a.nstencil];
  const float Lx = (float)gr.Lx, Ly = (float)gr.Ly, Lz = (float)gr.Lz;
  // a lane's share of one chunk's candidates, fetched from global memory into registers
  float4 pv[BL_SLOTS];
  int2 pt[BL_SLOTS];
  int pr[BL_SLOTS];
  auto fetch = [&](int base) {
    const int nch = min(BL_CH, total - base);
#pragma unroll
    for (int r = 0; r < BL_SLOTS; ++r) {
      const int c = tid + r * BL_THREADS;
      if (c < nch) {
        const int idx = base + c;
        int lo = 0, hi = a.nstencil - 1;  // last stencil cell whose prefix <= idx
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (sp[mid] <= idx) lo = mid;
          else hi = mid - 1;
        }
        const int t = sb[lo] + (idx - sp[lo]);
        float4 v = xq[t];
        if (shifted) {
          const int code = shc[lo];
          v.x += (float)((code & 3) - 1) * Lx;
          v.y += (float)(((code >> 2) & 3) - 1) * Ly;
          v.z += (float)(((code >> 4) & 3) - 1) * Lz;
        }
        pv[r] = v;
        pt[r] = make_int2(t, sorted_orig[t]);
        if (!FAST && a.ref_mode) pr[r] = ref_cell_sorted[t];
      }
    }
  };
  auto store = [&](int base) {
    const int nch = min(BL_CH, total - base);
#pragma unroll
    for (int r = 0; r < BL_SLOTS; ++r) {
      const int c = tid + r * BL_THREADS;
      if (c < nch) {
        cxq[c] = pv[r];
        cto[c] = pt[r];
        if (!FAST && a.ref_mode) cr[c] = pr[r];
      }
    }
  };
  __syncthreads();  // sp, pools
  if (total > 0) fetch(0);
  store(0);
  __syncthreads();
  const int lane = tid & 63;
  const int q = tid / NB_G, g = tid & (NB_G - 1);
  const int ngroups = blockDim.x / NB_G;
  const unsigned long long gmask = (NB_G == 64 ? ~0ull : ((1ull << NB_G) - 1ull)) << (lane & ~(NB_G - 1));
  const unsigned long long below = (1ull << lane) - 1ull;
  const float ix = 1.0f / Lx, iy = 1.0f / Ly, iz = 1.0f / Lz;
  int* my_ex = exl[q];
  int* my_s4 = s4l[q];
  for (int base = 0; base < total; base += BL_CH) {
    const int nch = min(BL_CH, total - base);
    const bool more = base + BL_CH < total;
    if (more) fetch(base + BL_CH);  // in flight during this chunk's scan
    for (int h = q; h < hn; h += ngroups) {  // uniform per group
      const int s = hb + h;
      int o, nex_all, ns4_all;
      const int* src_ex;
      const int* src_s4;
      float4 xi;
      bool masked;
      unsigned long long exm, s4m;
      if (fast) {  // everything from LDS
        o = ho[h];
        xi = hxi[h];
        nex_all = hex0[h + 1] - hex0[h];
        ns4_all = hs40[h + 1] - hs40[h];
        src_ex = pool_ex + hex0[h];
        src_s4 = pool_s4 + hs40[h];
        masked = hbad[h] == 0;
        exm = hexm[h];
        s4m = hs4m[h];
      } else {     // crowded cell: read the home atom's data from global memory
        o = sorted_orig[s];
        xi = xq[s];
        const int e0 = excl_ptr ? excl_ptr[o] : 0, t0s = s14_ptr ? s14_ptr[o] : 0;
        nex_all = excl_ptr ? excl_ptr[o + 1] - e0 : 0;
        ns4_all = s14_ptr ? s14_ptr[o + 1] - t0s : 0;
        src_ex = excl_idx + e0;
        src_s4 = s14_idx + t0s;
        masked = win_bad && win_bad[o] == 0;
        exm = ex_win ? ex_win[o] : 0ull;
        s4m = s4_win ? s4_win[o] : 0ull;
      }
      // index-window masks, or the CSR lists for an atom with a partner outside the window
      const int nex = masked ? 0 : min(nex_all, BL_MAXEX), ns4 = masked ? 0 : min(ns4_all, BL_MAXEX);
      if (!masked) {
        if (g < nex) my_ex[g] = src_ex[g];
        if (g < ns4) my_s4[g] = src_s4[g];
        if (g == 0 && (nex_all > BL_MAXEX || ns4_all > BL_MAXEX)) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
      }
      const int rci = (!FAST && a.ref_mode) ? ref_cell_sorted[s] : 0;
      const double pi[3] = {pos[3 * o], pos[3 * o + 1], pos[3 * o + 2]};
      wave_lds_sync();  // the group's lanes are in one wave
      unsigned* row = nbr_list + (long long)s * a.cap;
      int cnt = acnt[h];
      for (int cb = 0; cb < nch; cb += BL_U * NB_G) {
        float4 xj[BL_U];
        int2 tj[BL_U];
        int rcj[BL_U];
#pragma unroll
        for (int u = 0; u < BL_U; ++u) {
          const int ci = min(cb + u * NB_G + g, nch - 1);
          xj[u] = cxq[ci];
          tj[u] = cto[ci];
          rcj[u] = (!FAST && a.ref_mode) ? cr[ci] : 0;
        }
#pragma unroll
        for (int u = 0; u < BL_U; ++u) {
          const int jo = tj[u].y;
          float dx = xj[u].x - xi.x, dy = xj[u].y - xi.y, dz = xj[u].z - xi.z;
          if (!shifted) {
            dx -= Lx * rintf(dx * ix);
            dy -= Ly * rintf(dy * iy);
            dz -= Lz * rintf(dz * iz);
          }
          bool acc = (cb + u * NB_G + g < nch) & (tj[u].x != s) & (dx * dx + dy * dy + dz * dz < a.rl2);
          bool s14;
          if (masked) {
            const int dw = jo - o + BL_WIN;
            const bool win = (unsigned)dw < 2u * BL_WIN;
            const int sh = dw & (2 * BL_WIN - 1);
            acc &= !(win && ((exm >> sh) & 1ull));
            s14 = win && ((s4m >> sh) & 1ull);
          } else {
            s14 = false;
            for (int r = 0; r < nex; ++r) acc &= (my_ex[r] != jo);
            for (int r = 0; r < ns4; ++r) s14 |= (my_s4[r] == jo);
          }
          if (!FAST && a.ref_mode) {
            const int ax = cyc_dist(rci >> 20, rcj[u] >> 20, a.rnx);
            const int ay = cyc_dist((rci >> 10) & 1023, (rcj[u] >> 10) & 1023, a.rny);
            const int az = cyc_dist(rci & 1023, rcj[u] & 1023, a.rnz);
            acc &= (ax <= 1) & (ay <= 1) & (az <= 1);
          }
          if (acc) {  // float64 decision with the reference's sequence (pbc.py:40-44)
            double d[3];
            const double L[3] = {gr.Lx, gr.Ly, gr.Lz};
            for (int r = 0; r < 3; ++r) {
              double v = pos[3 * jo + r] - pi[r];
              double sv = v * (1.0 / L[r]);
              sv -= rint(sv);
              d[r] = sv * L[r];
            }
            acc = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) <= a.rc;
          }
          const unsigned long long m = __ballot(acc) & gmask;
          const int slot = cnt + __popcll(m & below);
          if (acc && slot < a.cap) row[slot] = nbr_entry(tj[u].x, s14);
          cnt += __popcll(m);
        }
      }
      if (g == 0) acnt[h] = cnt;
      wave_lds_sync();  // the next home atom of this group overwrites my_ex / my_s4
    }
    __syncthreads();
    if (more) {
      store(base + BL_CH);
      __syncthreads();
    }
  }
  for (int h = tid; h < hn; h += blockDim.x) {
    const int cnt = acnt[h];
    nbr_count[hb + h] = min(cnt, a.cap);
    if (cnt > a.cap) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
  }
}

template <bool FAST>
__global__ __launch_bounds__(BL_THREADS) void k_build_list_cell(ListCall L) {
  build_list_cell_body<FAST>(L, blockIdx.x);
}

// The common case of the build above as its own kernel: exact pair mode, float32 list radius, and
// either no exclusions or window masks present.
//
// Vector-instruction bound (the distance tests), so a test is made as short as it can be:
// - positions are 32-bit box fractions, staged relative to the home cell's centre with their squared
//   length, so "inside the list radius" is three fma and a compare, |b|^2 - 2 a.b < r^2 - |a|^2.
//   Rounding moves r^2 by less than 3.2e-6 r_l^2 (cells of r_l/3 to r_l, at most 2.1 r_l from the
//   centre to a listed atom); rl2 carries 1e-5 on top of r_l^2, so no pair inside r_l is missed.
//   WRAP (a stencil that wraps onto itself, where one image per cell isn't enough) takes each
//   pair's wrapped integer difference instead;
// - a wave holds BLF_H home atoms in scalar registers and tests each staged candidate it reads from
//   LDS against all of them, without a branch: lanes with nothing to store get an offset past the
//   rows, and a row has room for one whole group after its capacity;
// - exclusions, the atom itself and 1-4 partners are bits of window masks; 64 candidates of which none
//   is near any of the home atoms both in space and in index (all but a few) skip them;
// - candidates farther than the list radius from the home cell's box (3 of 10) are dropped as they
//   are staged.
// Home atoms with a partner outside the window scan their CSR lists. A grid of few cells gives each
// cell to `split` workgroups (a share of its home atoms each). The lists are in the order of
// k_build_list_cell.
// Before (one home atom per wave pass, 40 vector and scalar instructions with 6 branches per test,
// small boxes by k_build_list_cell) / now (us): 648 atoms 23 / 11, 2,592 r_c 12 92 / 24, 3,000 r_c 9
// 75 / 23, 23,328 r_c 12 86 / 69, 98,304 r_c 12 285 / 226. The vector unit issues in 82 % of the
// busy cycles (23,328 atoms, 24.1 M of 29.5 M).
#define BLF_H 4
#define BLF_WAVES (BL_THREADS / 64)
struct BlfShared {
  float4 x[BL_CH];  // (x, y, z, |.|^2) from the home cell's centre; WRAP: box fractions and 0
  int2 e[BL_CH];    // (list entry, original atom id)
  int2 sc[BL_MAXST + 1];  // stencil cells: (first candidate, sorted slot of candidate 0 if it were in this cell)
  int kept[BL_CH / 64];   // candidates kept of each 64
  int acnt[SORT_MAX];
  int exl[BLF_WAVES][BL_MAXEX], s4l[BLF_WAVES][BL_MAXEX];
  int4 hx[BL_HMAX];
  int ho[BL_HMAX];
  unsigned long long hexm[BL_HMAX], hs4m[BL_HMAX];
  unsigned char hbad[BL_HMAX];
};

// One chunk of nch staged candidates against H home atoms; lane k of the *l arguments holds home
// atom k's position terms (WRAP: fractions), limit, atom id, count and masks. Returns the counts.
template <int H, bool WRAP>
__device__ __forceinline__ int blf_scan(const float4* __restrict__ x, const int2* __restrict__ e, int nch, float al,
                                        float bl, float cl, float rl, int ol, int cntl, unsigned long long exl,
                                        unsigned long long s4l, unsigned* rows_p, int cap, float sx, float sy, float sz) {
  const int lane = threadIdx.x & 63, lim = cap - MDX_LIST_PAD;
  int ia[H], ib[H], ic[H], cnt[H];
  unsigned o32[H];
  float rhs[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    ia[k] = __builtin_amdgcn_readlane(__float_as_int(al), k);
    ib[k] = __builtin_amdgcn_readlane(__float_as_int(bl), k);
    ic[k] = __builtin_amdgcn_readlane(__float_as_int(cl), k);
    rhs[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rl), k));
    o32[k] = (unsigned)__builtin_amdgcn_readlane(ol, k) - 32u;
    cnt[k] = __builtin_amdgcn_readlane(cntl, k);
  }
  // the rows of these home atoms; a store past their end is dropped
  __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(rows_p, 0, H * cap * 4, 0x00020000);
  float4 xn = x[lane];
  int2 en = e[lane];
  for (int cb = 0; cb < nch; cb += 64) {
    const float4 xj = xn;
    const int2 ej = en;
    const int nb = cb + 64 < nch ? cb + 64 : 0;  // the next 64, in flight
    xn = x[nb + lane];
    en = e[nb + lane];
    unsigned long long m[H], any = 0;
#pragma unroll
    for (int k = 0; k < H; ++k) {
      bool near;
      if (WRAP) {
        const float dx = (float)(int)(__float_as_uint(xj.x) - (unsigned)ia[k]) * sx;
        const float dy = (float)(int)(__float_as_uint(xj.y) - (unsigned)ib[k]) * sy;
        const float dz = (float)(int)(__float_as_uint(xj.z) - (unsigned)ic[k]) * sz;
        near = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, xj.w))) < rhs[k];
      } else {
        near = fmaf(xj.x, __int_as_float(ia[k]),
                    fmaf(xj.y, __int_as_float(ib[k]), fmaf(xj.z, __int_as_float(ic[k]), xj.w))) < rhs[k];
      }
      m[k] = __ballot(near);
      any |= m[k] & __ballot((unsigned)ej.y - o32[k] < 64u);
    }
    int entry[H];
#pragma unroll
    for (int k = 0; k < H; ++k) entry[k] = ej.x;
    if (any != 0) {  // scalar: some candidate is near a home atom in space and in index
#pragma unroll
      for (int k = 0; k < H; ++k) {
        const unsigned dw = min((unsigned)ej.y - o32[k], 63u);  // bit 63 is always clear
        const unsigned long long exm = (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(exl >> 32), k) << 32 |
                                       (unsigned)__builtin_amdgcn_readlane((int)exl, k);
        const unsigned long long s4m = (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(s4l >> 32), k) << 32 |
                                       (unsigned)__builtin_amdgcn_readlane((int)s4l, k);
        m[k] &= __ballot(!((exm >> dw) & 1ull));
        entry[k] |= (int)((s4m >> dw) & 1ull);
      }
    }
#pragma unroll
    for (int k = 0; k < H; ++k) {
      int slot4 = 4 * (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m[k] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m[k], 0u));
      asm volatile("" : "+v"(slot4));  // computed for every lane: a select follows, not a branch
      const int off = __builtin_amdgcn_inverse_ballot_w64(m[k]) ? slot4 : (int)0x80000000;
      __builtin_amdgcn_raw_buffer_store_b32((unsigned)entry[k], rows, off, (k * cap + min(cnt[k], lim)) * 4, 0);
      cnt[k] += __popcll(m[k]);
    }
  }
  int out = 0;
#pragma unroll
  for (int k = 0; k < H; ++k) out = lane == k ? cnt[k] : out;
  return out;
}

template <bool WRAP>
__device__ __forceinline__ void build_list_fast_body(const ListCall& L, const int block, BlfShared& sh) {
  static_assert(BL_CH % BL_THREADS == 0 && BL_CH / 64 <= 64, "a lane per 64 of a chunk");
  const ListArgs& a = L.a;
  const int4* __restrict__ xf = L.xf;
  const int* __restrict__ sorted_orig = L.sorted_orig;
  const int* __restrict__ excl_ptr = L.excl_ptr;
  const int* __restrict__ excl_idx = L.excl_idx;
  const int* __restrict__ s14_ptr = L.s14_ptr;
  const int* __restrict__ s14_idx = L.s14_idx;
  int* __restrict__ nbr_count = L.nbr_count;
  unsigned* __restrict__ nbr_list = L.nbr_list;
  DevState* st = L.st;
  if (!need_rebuild(st, L.thr2)) return;
  const int cell = block / L.split, part = block - cell * L.split;
  const GridArgs& gr = a.g;
  const int hb = L.cell_start[cell], hn_all = L.cell_count[cell];
  // this workgroup's share of the home atoms
  const int p0 = (int)((long long)hn_all * part / L.split), p1 = (int)((long long)hn_all * (part + 1) / L.split);
  const int tid = threadIdx.x;
  if (hn_all > SORT_MAX) {  // oversize cells are flagged where the cells are counted: empty lists
    for (int t = p0 + tid; t < p1; t += BL_THREADS) nbr_count[hb + t] = 0;
    return;
  }
  if (p0 == p1) return;
  const int s0 = hb + p0, hn = p1 - p0;
  const int hz = cell % gr.nz, hy = (cell / gr.nz) % gr.ny, hx = cell / (gr.nz * gr.ny);
  for (int k = tid; k < a.nstencil; k += BL_THREADS) {
    const int p = L.stencil[k];
    int nx = hx + ((p >> 16) & 0xff) - 128, ny = hy + ((p >> 8) & 0xff) - 128, nz = hz + (p & 0xff) - 128;
    nx += nx < 0 ? gr.nx : (nx >= gr.nx ? -gr.nx : 0);
    ny += ny < 0 ? gr.ny : (ny >= gr.ny ? -gr.ny : 0);
    nz += nz < 0 ? gr.nz : (nz >= gr.nz ? -gr.nz : 0);
    const int nc = (nx * gr.ny + ny) * gr.nz + nz;
    sh.sc[k] = make_int2(L.cell_count[nc], L.cell_start[nc]);
  }
  for (int j = tid; j < hn; j += BL_THREADS) sh.acnt[j] = 0;
  const bool fit = hn <= BL_HMAX;
  if (fit) {
    for (int h = tid; h < hn; h += BL_THREADS) {
      const int o = sorted_orig[s0 + h];
      sh.ho[h] = o;
      sh.hx[h] = xf[s0 + h];
      sh.hexm[h] = L.ex_win ? L.ex_win[o] : 1ull << 32;
      sh.hs4m[h] = L.s4_win ? L.s4_win[o] : 0ull;
      sh.hbad[h] = L.win_bad ? L.win_bad[o] : (unsigned char)0;
    }
  }
  __syncthreads();
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar registers
  if (w == 0) {  // prefix sums of the stencil cells' sizes, a run of them per lane
    const int per = (a.nstencil + 63) >> 6, k0 = lane * per, k1 = min(a.nstencil, k0 + per);
    int sum = 0;
    for (int k = k0; k < k1; ++k) sum += sh.sc[k].x;
    int incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    int run = incl - sum;
    for (int k = k0; k < k1; ++k) {
      const int2 v = sh.sc[k];
      sh.sc[k] = make_int2(run, v.y - run);
      run += v.x;
    }
    if (lane == 63) sh.sc[a.nstencil] = make_int2(incl, 0);
  }
  __syncthreads();
  const int total = sh.sc[a.nstencil].x;
  const float sx = (float)(gr.Lx * 0x1p-32), sy = (float)(gr.Ly * 0x1p-32), sz = (float)(gr.Lz * 0x1p-32);
  // centre of the home cell as box fractions, and its half widths
  const int ccx = (int)(unsigned)((hx + 0.5) / gr.nx * 4294967296.0), ccy = (int)(unsigned)((hy + 0.5) / gr.ny * 4294967296.0),
            ccz = (int)(unsigned)((hz + 0.5) / gr.nz * 4294967296.0);
  const float hwx = 0.5f * (float)gr.wx, hwy = 0.5f * (float)gr.wy, hwz = 0.5f * (float)gr.wz;
  const float reach2 = a.rl2 * 1.0001f;
  auto relative = [&](const int4& f) {
    float4 v;
    v.x = (float)(int)((unsigned)f.x - (unsigned)ccx) * sx;
    v.y = (float)(int)((unsigned)f.y - (unsigned)ccy) * sy;
    v.z = (float)(int)((unsigned)f.z - (unsigned)ccz) * sz;
    v.w = fmaf(v.x, v.x, fmaf(v.y, v.y, v.z * v.z));
    return v;
  };
  int4 pv[BL_SLOTS];
  int2 pt[BL_SLOTS];
  auto fetch = [&](int base) {
#pragma unroll
    for (int r = 0; r < BL_SLOTS; ++r) {
      const int first = base + w * 64 + r * BL_THREADS, idx = first + lane;  // the wave's candidates: first ..
      if (first >= total) break;
      // the cell of the first one, by counting the cells that begin at or before it; then on from cell
      // to cell while they begin inside the wave's 64
      int k = -1;
      for (int b = 0; b < a.nstencil; b += 64)
        k += __popcll(__ballot(b + lane < a.nstencil && sh.sc[min(b + lane, a.nstencil)].x <= first));
      int off = sh.sc[k].y;
      for (++k; k < a.nstencil; ++k) {
        const int2 v = sh.sc[k];
        if (__builtin_amdgcn_readfirstlane(v.x) > first + 63) break;
        if (idx >= v.x) off = v.y;
      }
      if (idx < total) {
        const int t = off + idx;
        pv[r] = xf[t];
        pt[r] = make_int2((int)nbr_entry(t, false), sorted_orig[t]);
      }
    }
  };
  // the fetched candidates within the list radius of the home cell's box
  float4 sv[BL_SLOTS];
  unsigned long long keep[BL_SLOTS];
  auto select = [&](int base) {
#pragma unroll
    for (int r = 0; r < BL_SLOTS; ++r) {
      const float4 v = relative(pv[r]);
      const float dx = fmaxf(fabsf(v.x) - hwx, 0.f), dy = fmaxf(fabsf(v.y) - hwy, 0.f), dz = fmaxf(fabsf(v.z) - hwz, 0.f);
      keep[r] = __ballot(base + tid + r * BL_THREADS < total && fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < reach2);
      sv[r] = WRAP ? make_float4(__int_as_float(pv[r].x), __int_as_float(pv[r].y), __int_as_float(pv[r].z), 0.f) : v;
      if (lane == 0) sh.kept[r * BLF_WAVES + w] = __popcll(keep[r]);
    }
  };
  // staged in order, behind the candidates kept of the 64s before; padded to whole passes with
  // candidates far away from everything. Returns their number.
  auto store = [&]() {
    int incl = lane < BL_CH / 64 ? sh.kept[lane] : 0;
    for (int d = 1; d < BL_CH / 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    const int n = __builtin_amdgcn_readlane(incl, BL_CH / 64 - 1);
#pragma unroll
    for (int r = 0; r < BL_SLOTS; ++r) {
      const int c0 = __builtin_amdgcn_readlane(incl, r * BLF_WAVES + w) - __popcll(keep[r]);
      const int c = c0 + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(keep[r] >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((unsigned)keep[r], 0u));
      if (__builtin_amdgcn_inverse_ballot_w64(keep[r])) {
        sh.x[c] = sv[r];
        sh.e[c] = pt[r];
      }
    }
    if (n + tid < ((n + 63) & ~63)) {
      sh.x[n + tid] = make_float4(0.f, 0.f, 0.f, 1e30f);
      sh.e[n + tid] = make_int2(0, 0);
    }
    return n;
  };
  fetch(0);
  select(0);
  __syncthreads();
  int nch = store();
  __syncthreads();
  int* my_ex = sh.exl[w];
  int* my_s4 = sh.s4l[w];
  const int lim = a.cap - MDX_LIST_PAD;  // capacity of a row: a group's 64 entries fit after it
  const int hw0 = hn * w / BLF_WAVES, hw1 = hn * (w + 1) / BLF_WAVES;  // this wave's home atoms
  for (int base = 0; base < total; base += BL_CH) {
    const bool more = base + BL_CH < total;
    if (more) fetch(base + BL_CH);  // in flight during this chunk's scan
    for (int h0 = hw0, nh; h0 < hw1; h0 += nh) {
      const int rounds = (hw1 - h0 + BLF_H - 1) / BLF_H;
      nh = (hw1 - h0 + rounds - 1) / rounds;
      // one lane per home atom reads its data
      const int hl = h0 + min(lane, nh - 1), sl = s0 + hl;
      int4 fl;
      int ol;
      unsigned long long exm, s4m;
      bool bad;
      if (fit) {
        fl = sh.hx[hl];
        ol = sh.ho[hl];
        exm = sh.hexm[hl];
        s4m = sh.hs4m[hl];
        bad = sh.hbad[hl] != 0;
      } else {
        fl = xf[sl];
        ol = sorted_orig[sl];
        exm = L.ex_win ? L.ex_win[ol] : 1ull << 32;
        s4m = L.s4_win ? L.s4_win[ol] : 0ull;
        bad = L.win_bad && L.win_bad[ol] != 0;
      }
      const float4 rel = relative(fl);
      const float ha = WRAP ? __int_as_float(fl.x) : -2.f * rel.x, hbb = WRAP ? __int_as_float(fl.y) : -2.f * rel.y,
                  hc = WRAP ? __int_as_float(fl.z) : -2.f * rel.z, hr = WRAP ? a.rl2 : a.rl2 - rel.w;
      const float rhs = bad ? -3e38f : hr;  // no candidate is inside: done below
      const int before = sh.acnt[hl];
      unsigned* rows = nbr_list + (long long)(s0 + h0) * a.cap;
      int after;
#define BLF_SCAN(H_) after = blf_scan<H_, WRAP>(sh.x, sh.e, nch, ha, hbb, hc, rhs, ol, before, exm, s4m, rows, a.cap, sx, sy, sz)
      if (nh == 4) BLF_SCAN(4);
      else if (nh == 3) BLF_SCAN(3);
      else if (nh == 2) BLF_SCAN(2);
      else BLF_SCAN(1);
#undef BLF_SCAN
      if (lane < nh) sh.acnt[hl] = after;
      for (unsigned left = (unsigned)__ballot(bad && lane < nh); left; left &= left - 1u) {
        // a partner outside the index window: the CSR lists
        const int k = __builtin_amdgcn_readfirstlane(__ffs(left) - 1);
        const int o = __builtin_amdgcn_readlane(ol, k), s = s0 + h0 + k;
        int count = __builtin_amdgcn_readlane(before, k);
        const int e0 = excl_ptr ? excl_ptr[o] : 0, t0s = s14_ptr ? s14_ptr[o] : 0;
        const int nex_all = excl_ptr ? excl_ptr[o + 1] - e0 : 0, ns4_all = s14_ptr ? s14_ptr[o + 1] - t0s : 0;
        const int nex = min(nex_all, BL_MAXEX), ns4 = min(ns4_all, BL_MAXEX);
        if (lane < nex) my_ex[lane] = excl_idx[e0 + lane];
        if (lane < ns4) my_s4[lane] = s14_idx[t0s + lane];
        if (lane == 0 && (nex_all > BL_MAXEX || ns4_all > BL_MAXEX)) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
        wave_lds_sync();
        unsigned* row = nbr_list + (long long)s * a.cap;
        const float kx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ha), k)),
                    ky = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hbb), k)),
                    kz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hc), k)),
                    kr = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hr), k));
        for (int cb = 0; cb < nch; cb += 64) {
          const float4 xj = sh.x[cb + lane];
          const int2 ej = sh.e[cb + lane];
          float r2;
          if (WRAP) {
            const float dx = (float)(int)(__float_as_uint(xj.x) - __float_as_uint(kx)) * sx;
            const float dy = (float)(int)(__float_as_uint(xj.y) - __float_as_uint(ky)) * sy;
            const float dz = (float)(int)(__float_as_uint(xj.z) - __float_as_uint(kz)) * sz;
            r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, xj.w)));
          } else {
            r2 = fmaf(xj.x, kx, fmaf(xj.y, ky, fmaf(xj.z, kz, xj.w)));
          }
          bool acc = r2 < kr && ej.y != o;
          bool s14 = false;
          for (int r = 0; r < nex; ++r) acc &= (my_ex[r] != ej.y);
          for (int r = 0; r < ns4; ++r) s14 |= (my_s4[r] == ej.y);
          const unsigned long long m = __ballot(acc);
          const int slot = count + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
          if (acc && slot < lim) row[slot] = (unsigned)(ej.x | (int)s14);
          count += __popcll(m);
        }
        if (lane == 0) sh.acnt[h0 + k] = count;
        wave_lds_sync();  // the wave's next home atom overwrites my_ex / my_s4
      }
    }
    if (more) select(base + BL_CH);
    __syncthreads();
    if (more) {
      nch = store();
      __syncthreads();
    }
  }
  for (int h = tid; h < hn; h += BL_THREADS) {
    const int cnt = sh.acnt[h];
    nbr_count[s0 + h] = min(cnt, lim);
    if (cnt > lim) atomicOr(&st->flags, MDX_FLAG_OVERFLOW);
  }
}

template <bool WRAP>
__global__ __launch_bounds__(BL_THREADS) void k_build_list_fast(ListCall L) {
  __shared__ BlfShared sh;
  build_list_fast_body<WRAP>(L, blockIdx.x, sh);
}

// every replica's list build in one launch
__global__ __launch_bounds__(BL_THREADS) void k_build_list_fast_batch(BatchMap map, const ListCall* __restrict__ calls) {
  __shared__ BlfShared sh;
  int block;
  const int r = batch_replica(map, &block);
  if (calls[r].a.shifted) build_list_fast_body<false>(calls[r], block, sh);
  else build_list_fast_body<true>(calls[r], block, sh);
}

__global__ void k_request_rebuild(DevState* st) { st->rebuild = 1; }

int mdx_enqueue_request_rebuild(mdx_ctx* c) {
  k_request_rebuild<<<1, 1, 0, c->stream>>>(c->dstate.p);
  MDX_LAUNCH_CHECK();
  return 0;
}

__global__ void k_clear_rebuild(DevState* st) {
  st->rebuild = 0;
  st->max_disp2_bits = 0;
}

// zero the per-cell counts of the list grid when a rebuild is due (a kernel, not a memset, so
// the step stays safe to capture in a hipGraph) and count rebuilds; `force`: a rebuild is due
__global__ void k_prep_rebuild(DevState* st, double thr2, int* __restrict__ cell_count, int ncell, bool force) {
  if (!force && !need_rebuild(st, thr2)) return;
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ncell) cell_count[i] = 0;
  if (i == 0) {
    if (force) st->rebuild = 1;
    st->nrebuild += 1;
  }
}


// ============================================================== host side
static void make_grid(mdx_ctx* c, GridArgs* g) {
  g->nx = c->gn[0];
  g->ny = c->gn[1];
  g->nz = c->gn[2];
  g->Lx = c->box[0];
  g->Ly = c->box[1];
  g->Lz = c->box[2];
  g->wx = c->box[0] / c->gn[0];
  g->wy = c->box[1] / c->gn[1];
  g->wz = c->box[2] / c->gn[2];
}

int mdx_nlist_prepare(mdx_ctx* c) {
  double rl = c->rc + c->skin;
  for (int d = 0; d < 3; ++d) {
    int k = (int)std::floor(c->box[d] * c->cells_per_rl / rl);
    if (k < 1) k = 1;
    c->gn[d] = k;
  }
  c->ncell = c->gn[0] * c->gn[1] * c->gn[2];
  // stencil: offsets whose cells can hold an atom within rl of the home cell, each distinct
  // periodic cell once
  c->stencil.clear();
  int lo[3], hi[3];
  double w[3];
  for (int d = 0; d < 3; ++d) {
    w[d] = c->box[d] / c->gn[d];
    int r = (int)std::ceil(rl / w[d]);
    if (2 * r + 1 >= c->gn[d]) {
      lo[d] = -((c->gn[d] - 1) / 2);
      hi[d] = c->gn[d] / 2;
    } else {
      lo[d] = -r;
      hi[d] = r;
    }
    c->reach[d] = r;
  }
  for (int dx = lo[0]; dx <= hi[0]; ++dx)
    for (int dy = lo[1]; dy <= hi[1]; ++dy)
      for (int dz = lo[2]; dz <= hi[2]; ++dz) {
        double mx = std::max(0, std::abs(dx) - 1) * w[0];
        double my = std::max(0, std::abs(dy) - 1) * w[1];
        double mz = std::max(0, std::abs(dz) - 1) * w[2];
        if (mx * mx + my * my + mz * mz > rl * rl) continue;
        c->stencil.push_back(((dx + 128) << 16) | ((dy + 128) << 8) | (dz + 128));
      }
  int rc;
  if ((rc = c->d_stencil.ensure(c->stencil.size()))) return rc;
  MDX_HIP(hipMemcpy(c->d_stencil.p, c->stencil.data(), c->stencil.size() * sizeof(int), hipMemcpyHostToDevice));
  if ((rc = c->cell_count.ensure(c->ncell)) || (rc = c->cell_start.ensure(c->ncell)) ||
      (rc = c->atom_place.ensure(c->n)) || (rc = c->atom_cell.ensure(c->n)) ||
      (rc = c->sorted_orig.ensure(c->n)) || (rc = c->orig_sorted.ensure(c->n)) || (rc = c->xq.ensure(c->n)) || (rc = c->xf.ensure(c->n)) ||
      (rc = c->ljs.ensure(c->n)) || (rc = c->ljs14.ensure(c->n)) || (rc = c->ref_cell_sorted.ensure(c->n)) ||
      (rc = c->pos_at_build.ensure(3 * (size_t)c->n)) || (rc = c->nbr_count.ensure(c->n)) ||
      (rc = c->pos_sorted.ensure(3 * (size_t)c->n)))
    return rc;
  // capacity: expected neighbours in a sphere of radius rl at the system density, with margin
  double vol = c->box[0] * c->box[1] * c->box[2];
  double dens = c->n / vol;
  double expect = 4.0 / 3.0 * M_PI * rl * rl * rl * dens;
  int cap = (int)(expect * 1.5 + 64);
  if (cap > c->n) cap = c->n;
  cap += MDX_LIST_PAD;
  if (cap < c->nbr_cap) cap = c->nbr_cap;
  c->nbr_cap = cap;
  c->list_stride = cap;
  // slack after the last row: the nonbonded kernel loads the next chunk's indices ahead
  if ((rc = c->nbr_list.ensure((size_t)cap * c->n + MDX_LIST_SLACK))) return rc;
  MDX_HIP(hipMemset(c->pos_at_build.p, 0, 3 * sizeof(double) * c->n));
  int one = 1;
  MDX_HIP(hipMemcpy(&c->dstate.p->rebuild, &one, sizeof(int), hipMemcpyHostToDevice));
  c->list_valid = true;
  return 0;
}

int mdx_nlist_enqueue_pack(mdx_ctx* c) {
  k_pack<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(fill_args(c, 0.0), c->n);
  MDX_LAUNCH_CHECK();
  return 0;
}

// squared displacement that triggers a rebuild; skin == 0 (reference pair set or no buffer):
// rebuild every evaluation
static double rebuild_thr2(const mdx_ctx* c) {
  const double half = 0.5 * c->skin;
  return c->skin > 0 ? half * half : -1.0;
}

// Enqueue: displacement check, conditional rebuild of the list, pack. Leaves the rebuild flag set
// for the consumer (k_clear_rebuild is enqueued by the caller after the last reader).
int mdx_nlist_update(mdx_ctx* c, bool force_rebuild) {
  int rc = mdx_nlist_update_order(c, force_rebuild);
  return rc ? rc : mdx_nlist_update_list(c);
}

// First part: displacement check and, on a rebuild, binning, per-cell sort and fill of the
// sorted-order arrays; then the pack. Everything the PME plane kernels read is final after it.
int mdx_nlist_update_order(mdx_ctx* c, bool force_rebuild) {
  MDX_CHECK(c->nb_configured, MDX_ERR_INVALID, "nonbonded not configured");
  const double thr2 = rebuild_thr2(c);
  GridArgs g;
  make_grid(c, &g);
  int nb = div_up(c->n, NL_BLOCK);
  DevState* st = c->dstate.p;
  const bool pro = c->prologue_done;  // displacement, rebuild decision and packing already done
  if (!pro) {
    k_check_disp<<<nb, NL_BLOCK, 0, c->stream>>>(c->pos, c->pos_at_build.p, c->n, c->box[0], c->box[1], c->box[2], st);
    MDX_LAUNCH_CHECK();
    k_prep_rebuild<<<div_up(c->ncell, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(st, thr2, c->cell_count.p, c->ncell, force_rebuild);
    MDX_LAUNCH_CHECK();
  }
  // reference cells are needed for the REFERENCE stencil filter; they depend on the minimum
  // position, so REFERENCE mode runs with skin 0 (rebuild every evaluation) and re-bins here.
  if (c->pair_mode == MDX_PAIRS_REFERENCE) {
    int rc = ref_bin_enqueue(c, c->cell_cutoff, nullptr);
    if (rc) return rc;
  }
  if (!c->prologue_binned) {  // else the step prologue's last workgroup binned the atoms
    k_grid_bin<<<nb, NL_BLOCK, 0, c->stream>>>(c->pos, c->n, g, st, thr2, c->atom_cell.p, c->atom_place.p, c->cell_count.p);
    MDX_LAUNCH_CHECK();
    k_cell_scan<<<1, SCAN_THREADS, 0, c->stream>>>(c->cell_count.p, c->cell_start.p, c->ncell, st, thr2);
    MDX_LAUNCH_CHECK();
    k_grid_scatter<<<nb, NL_BLOCK, 0, c->stream>>>(c->atom_cell.p, c->atom_place.p, c->n, c->cell_start.p,
                                                   c->sorted_orig.p, st, thr2);
    MDX_LAUNCH_CHECK();
  }
  const FillArgs fa = fill_args(c, thr2);
  k_grid_sort_fill<<<c->ncell, 256, 0, c->stream>>>(fa);
  MDX_LAUNCH_CHECK();
  return pro || force_rebuild ? 0 : mdx_nlist_enqueue_pack(c);  // a rebuild's fill packs every atom
}

// Fast build: workgroups per home cell. Grids of few cells leave the chip idle: up to 8 workgroups
// share a cell's atoms until there's about one per compute unit (each stages the cell's candidates,
// so more cost more than they give). One / by this rule (us): 648 atoms r_c 9 (27 cells) 14.6 / 11.4,
// 2,592 r_c 12 (64 cells) 41 / 24, 3,000 r_c 9 (125 cells) 29 / 23.
static int blf_split(const mdx_ctx* c) {
  int s = 1;
  while (s < 8 && 2 * s * c->ncell <= c->ncu) s *= 2;
  return s;
}

// The list-build launch of a context: its arguments and kernel (0: the fast build, of every list with a
// skin; 1, 2: the cell build, general and FAST).
static int list_call(mdx_ctx* c, ListCall* L, int* kind) {
  const bool ref = c->pair_mode == MDX_PAIRS_REFERENCE;
  ListArgs& a = L->a;
  make_grid(c, &a.g);
  a.n = c->n;
  a.cap = c->nbr_cap;
  double rl = c->rc + c->skin;
  a.rl2 = (float)(rl * rl) * (1.0f + 1e-5f);
  a.rc = c->rc;
  a.ref_mode = ref ? 1 : 0;
  a.rnx = c->ref_n[0];
  a.rny = c->ref_n[1];
  a.rnz = c->ref_n[2];
  a.nstencil = (int)c->stencil.size();
  MDX_CHECK(a.nstencil <= BL_MAXST, MDX_ERR_INVALID, "stencil of %d cells exceeds %d", a.nstencil, BL_MAXST);
  // each periodic cell appears once in the stencil, on one side only: a fixed shift per stencil
  // cell maps its atoms to the image nearest the home cell
  a.shifted = 1;
  for (int d = 0; d < 3; ++d)
    if (2 * c->reach[d] + 1 >= c->gn[d]) a.shifted = 0;
  const bool win = c->win_ready && c->h_win_bad.size() == (size_t)c->n;
  // set with the exclusions and 1-4 pairs; without either only the atom itself is masked
  MDX_CHECK(win || !(c->has_excl || c->has_s14), MDX_ERR_INVALID, "exclusions without their window masks");
  L->xq = c->xq.p;
  L->xf = c->xf.p;
  L->sorted_orig = c->sorted_orig.p;
  L->cell_start = c->cell_start.p;
  L->cell_count = c->cell_count.p;
  L->stencil = c->d_stencil.p;
  L->excl_ptr = c->has_excl ? c->excl_ptr.p : nullptr;
  L->excl_idx = c->excl_idx.p;
  L->s14_ptr = c->has_s14 ? c->s14_ptr.p : nullptr;
  L->s14_idx = c->s14_idx.p;
  L->ex_win = win ? c->ex_win.p : nullptr;
  L->s4_win = win ? c->s4_win.p : nullptr;
  L->win_bad = win ? c->win_bad.p : nullptr;
  L->ref_cell_sorted = c->ref_cell_sorted.p;
  L->pos = c->pos;
  L->nbr_count = c->nbr_count.p;
  L->nbr_list = c->nbr_list.p;
  L->st = c->dstate.p;
  L->thr2 = rebuild_thr2(c);
  L->split = blf_split(c);
  *kind = c->skin > 0 ? 0 : (win && a.shifted && !a.ref_mode ? 2 : 1);  // reference mode has no skin
  return 0;
}

// Second part: the neighbour-list build (its workgroups return at once unless rebuilding).
int mdx_nlist_update_list(mdx_ctx* c) {
  ListCall L;
  int kind, rc = list_call(c, &L, &kind);
  if (rc) return rc;
  dim3 grid(c->ncell), block(BL_THREADS);
  switch (kind) {
    case 0: {
      grid.x *= L.split;
      if (L.a.shifted) k_build_list_fast<false><<<grid, block, 0, c->stream>>>(L);
      else k_build_list_fast<true><<<grid, block, 0, c->stream>>>(L);
      break;
    }
    case 1: k_build_list_cell<false><<<grid, block, 0, c->stream>>>(L); break;
    default: k_build_list_cell<true><<<grid, block, 0, c->stream>>>(L); break;
  }
  MDX_LAUNCH_CHECK();
  return 0;
}

// ---- batched replicas: the sort/fill and list-build launches of every replica
__global__ __launch_bounds__(256) void k_grid_sort_fill_batch(BatchMap map, const FillArgs* __restrict__ calls) {
  int cell;
  const int r = batch_replica(map, &cell);
  const FillArgs& f = calls[r];
  if (!need_rebuild(f.st, f.thr2)) return;
  grid_sort_fill_block(f, cell);
}

int mdx_batch_prepare_list(mdx_ctx* const* cs, int n, BatchKind* fill, BatchKind* list) {
  std::vector<FillArgs> fa;
  std::vector<ListCall> lc;
  std::vector<int> bfa, bl;
  for (int r = 0; r < n; ++r) {
    mdx_ctx* c = cs[r];
    fa.push_back(fill_args(c, rebuild_thr2(c)));
    bfa.push_back(c->ncell);
    ListCall L;
    int kind, rc = list_call(c, &L, &kind);
    if (rc) return rc;
    MDX_CHECK(kind == 0, MDX_ERR_INVALID, "replica %d: batched steps need a list radius larger than the pair cutoff", r);
    lc.push_back(L);
    bl.push_back(c->ncell * L.split);
  }
  int rc;
  if ((rc = batch_kind_upload(fill, fa, bfa, 0)) || (rc = batch_kind_upload(list, lc, bl, 0))) return rc;
  return 0;
}

int mdx_batch_launch_fill(const BatchKind& k, hipStream_t s) {
  if (!k.blocks) return 0;
  k_grid_sort_fill_batch<<<k.blocks, 256, 0, s>>>(k.map, (const FillArgs*)k.calls);
  MDX_LAUNCH_CHECK();
  return 0;
}

int mdx_batch_launch_list(const BatchKind& k, hipStream_t s) {
  k_build_list_fast_batch<<<k.blocks, BL_THREADS, 0, s>>>(k.map, (const ListCall*)k.calls);
  MDX_LAUNCH_CHECK();
  return 0;
}

int mdx_nlist_enqueue_clear(mdx_ctx* c) {
  k_clear_rebuild<<<1, 1, 0, c->stream>>>(c->dstate.p);
  MDX_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- pair enumeration (parity)
__global__ void k_emit_pairs(int n, int cap, const int* __restrict__ nbr_count, const unsigned* __restrict__ nbr_list,
                             const int* __restrict__ sorted_orig, const float4* __restrict__ xq, const double* __restrict__ pos,
                             double Lx, double Ly, double Lz, double rc, int* __restrict__ out,
                             long long out_cap, unsigned long long* __restrict__ counter) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int o = sorted_orig[s];
  int cnt = nbr_count[s];
  double L[3] = {Lx, Ly, Lz};
  for (int k = 0; k < cnt; ++k) {
    unsigned e = nbr_list[(long long)s * cap + k];
    int t = nbr_slot(e);
    int jo = sorted_orig[t];
    if (jo <= o) continue;  // unique pairs, i < j (original ids)
    double d[3];
    for (int q = 0; q < 3; ++q) {
      double v = pos[3 * jo + q] - pos[3 * o + q];
      double sv = v * (1.0 / L[q]);
      sv -= rint(sv);
      d[q] = sv * L[q];
    }
    double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    if (!(r <= rc)) continue;
    unsigned long long slot = atomicAdd(counter, 1ull);
    if ((long long)slot < out_cap) {
      out[2 * slot] = o;
      out[2 * slot + 1] = jo;
    }
  }
}

extern "C" int mdx_neighbor_pairs(mdx_ctx* c, int* d_pairs, int64_t capacity, int64_t* h_count) {
  MDX_CHECK(c && c->pos && c->nb_configured, MDX_ERR_INVALID, "mdx_neighbor_pairs: system/nonbonded not set");
  MDX_ENTER();
  c->forces_current = false;
  MDX_HIP(hipMemsetAsync(&c->dstate.p->flags, 0, sizeof(unsigned), c->stream));
  int rc = mdx_nlist_update(c, true);
  if (rc) return rc;
  if ((rc = c->tmp64.ensure(1))) return rc;
  MDX_HIP(hipMemsetAsync(c->tmp64.p, 0, sizeof(long long), c->stream));
  k_emit_pairs<<<div_up(c->n, NL_BLOCK), NL_BLOCK, 0, c->stream>>>(
      c->n, c->nbr_cap, c->nbr_count.p, c->nbr_list.p, c->sorted_orig.p, c->xq.p, c->pos, c->box[0], c->box[1],
      c->box[2], c->rc, d_pairs, capacity, (unsigned long long*)c->tmp64.p);
  MDX_LAUNCH_CHECK();
  rc = mdx_nlist_enqueue_clear(c);
  if (rc) return rc;
  long long cnt = 0;
  unsigned flags = 0;
  MDX_HIP(hipMemcpyAsync(&cnt, c->tmp64.p, sizeof(long long), hipMemcpyDeviceToHost, c->stream));
  MDX_HIP(hipMemcpyAsync(&flags, &c->dstate.p->flags, sizeof(unsigned), hipMemcpyDeviceToHost, c->stream));
  MDX_HIP(hipStreamSynchronize(c->stream));
  MDX_CHECK(!(flags & MDX_FLAG_OVERFLOW), MDX_ERR_OVERFLOW, "neighbour list or cell capacity exceeded");
  *h_count = cnt;
  MDX_LEAVE_RET(0);
}
