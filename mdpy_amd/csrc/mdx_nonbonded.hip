// Nonbonded launch (the pair evaluation of mdx_nonbonded_body.h, with the bonded terms as
// trailing workgroups), the Ewald-correction table, and the plain all-pairs Coulomb kernel
// (mdpy/constraint/electrostatic_constraint.py:52-79), gfx950.
#include "mdx_bonded_terms.h"
#include "mdx_nonbonded_body.h"

#define NB_BLOCK 256

// G(z) of the forces-only Coulomb path and its derivative, float64, for the table
static void coulomb_correction(double beta, double z, double* G, double* dG) {
  const double k = 2.0 * beta * beta * beta / sqrt(M_PI);
  const double x2 = beta * beta * z;
  if (x2 < 2.0) {
    // G = k sum_{n>=1} (-1)^(n+1) 2n / (n! (2n+1)) x^(2n-2): the series of erf(x)/x^3 minus
    // that of exp(-x^2)/x^2, without their cancellation at small z
    double s = 0, sp = 0, fact = 1, xp = 1, xpm = 0;  // xp = x2^(n-1), xpm = x2^(n-2)
    for (int n = 1; n <= 40; ++n) {
      fact *= n;
      const double cn = ((n & 1) ? 2.0 : -2.0) * n / (fact * (2 * n + 1));
      s += cn * xp;
      if (n >= 2) sp += cn * (n - 1) * beta * beta * xpm;
      xpm = xp;
      xp *= x2;
    }
    *G = k * s;
    *dG = k * sp;
    return;
  }
  const double r = sqrt(z), e = exp(-x2), er = erf(beta * r), c = 2.0 * beta / sqrt(M_PI);
  *G = er / (z * r) - c * e / z;
  *dG = beta * e / (sqrt(M_PI) * z * z) - 1.5 * er / (z * z * r) + c * (beta * beta * e / z + e / (z * z));
}

int mdx_coulomb_table_update(mdx_ctx* c) {
  if (!(c->beta > 0 && c->rc > 0) || (c->ctab.p && c->ctab_beta == c->beta && c->ctab_rc == c->rc)) return 0;
  const int N = MDX_CTAB_N;
  const double zmax = c->rc * c->rc * (1.0 + 1e-3);  // the float64 cutoff re-decision may accept r2 a hair above rc^2
  const double h = zmax / N;
  std::vector<float4> tab(N);
  double g0, d0;
  coulomb_correction(c->beta, 0.0, &g0, &d0);
  for (int k = 0; k < N; ++k) {
    double g1, d1;
    coulomb_correction(c->beta, (k + 1) * h, &g1, &d1);
    const double a0 = g0, a1 = d0 * h, a2 = 3.0 * (g1 - g0) - (2.0 * d0 + d1) * h, a3 = 2.0 * (g0 - g1) + (d0 + d1) * h;
    tab[k] = make_float4((float)a0, (float)a1, (float)a2, (float)a3);
    g0 = g1;
    d0 = d1;
  }
  int rc = c->ctab.ensure(N);
  if (rc) return rc;
  MDX_HIP(hipMemcpy(c->ctab.p, tab.data(), N * sizeof(float4), hipMemcpyHostToDevice));
  c->ctab_beta = c->beta;
  c->ctab_rc = c->rc;
  c->ctab_scale = (float)(N / zmax);
  mdx_invalidate_graph(c);
  return 0;
}

// Workgroups [0, nres) loop over the nb_blocks nonbonded workgroup indices (nres == nb_blocks:
// one each); the trailing ones evaluate the bonded terms. Blocks are numbered in cell order, so
// a contiguous range of them is a compact region of the box.
//
// At most 128 VGPRs (4 waves per SIMD) instead of the 132 the compiler picks by itself: the cap
// costs two 8-byte spills outside the pair loop (reloaded once per atom), leaves the kernel's own
// time unchanged and measured the whole PME-concurrent step ~1.3 % faster on water23328.
template <bool LJ, bool COUL, bool ENERGY, int G, bool S14>
__global__ __launch_bounds__(NB_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_nonbonded(NbArgs a, NbPtrs P, BondedArgs ba, int nb_blocks, int nres) {
  if ((int)blockIdx.x >= nres) {  // trailing workgroups: bonded terms
    bonded_block(ba, blockIdx.x - nres);
    return;
  }
  if (nres % 8 == 0 && nres < nb_blocks) {
    // workgroups are dealt to the 8 XCDs round-robin: give each XCD a contiguous (spatially
    // compact) range of the blocks, its nres/8 workgroups striding through it
    const int x = blockIdx.x & 7, per = nres >> 3;
    const int b1 = (int)((long long)nb_blocks * (x + 1) / 8);
    for (int vb = (int)((long long)nb_blocks * x / 8) + (blockIdx.x >> 3); vb < b1; vb += per)
      nb_block<LJ, COUL, ENERGY, G, NB_BLOCK, S14>(a, P, vb);
    return;
  }
  if (nres == nb_blocks) {  // one unit each, in the same contiguous ranges per XCD
    const int x = blockIdx.x & 7, q = nb_blocks >> 3, rem = nb_blocks & 7;
    nb_block<LJ, COUL, ENERGY, G, NB_BLOCK, S14>(a, P, x * q + min(x, rem) + (blockIdx.x >> 3));
    return;
  }
  for (int vb = blockIdx.x; vb < nb_blocks; vb += nres) nb_block<LJ, COUL, ENERGY, G, NB_BLOCK, S14>(a, P, vb);
}

// Lanes per atom. Fewer lanes leave less of a row's last chunk empty and share the reduction and
// the row set-up among more atoms of a wave; more lanes give small systems enough waves. Measured
// alone with 16 / 32 / 64 lanes (us): 648 atoms r_c 9 A 7.3 / 5.3 / 4.5, 2,592 r_c 12 12.4 / 9.4 / 8.4,
// 3,000 r_c 9 8.0 / 6.5 / 5.9, 9,000 r_c 9 11.8 / 12.1 / 13.6, r_c 12 21.0 / 21.2 / 22.6,
// 23,328 r_c 12 40.8 / 43.2 / 50.9, 98,304 r_c 12 188 / 207 / 259.
int mdx_nb_lanes(const mdx_ctx* c) {
  if (c->nb_lanes_set) return c->nb_lanes;
  return c->n >= 8192 ? 16 : (c->n >= 3072 ? 32 : 64);
}

NbArgs nb_args(const mdx_ctx* c) {
  NbArgs a;
  a.n = c->n;
  a.cap = c->nbr_cap;
  const double s[3] = {c->box[0] * 0x1p-32, c->box[1] * 0x1p-32, c->box[2] * 0x1p-32};
  a.sx = (float)s[0];
  a.sy = (float)s[1];
  a.sz = (float)s[2];
  a.sx2 = (float)(s[0] * s[0]);
  a.sy2 = (float)(s[1] * s[1]);
  a.sz2 = (float)(s[2] * s[2]);
  a.rc2 = (float)(c->rc * c->rc);
  // float32 r^2 carries ~5e-7 of itself in error (the box fractions hold 32 bits): re-decide within
  // a band of more than 20x that in float64
  a.guard2 = (float)(c->rc * 2e-4);
  a.beta = (float)c->beta;
  a.twob_sqrtpi = (float)(2.0 * c->beta / sqrt(M_PI));
  a.ct_scale = c->ctab_scale;
  a.ctab = c->ctab.p;
  a.Lxd = c->box[0];
  a.Lyd = c->box[1];
  a.Lzd = c->box[2];
  a.rcd = c->rc;
  return a;
}

NbPtrs nb_ptrs(const mdx_ctx* c) {
  NbPtrs P;
  P.xf = c->xf.p;
  P.ljs = c->ljs.p;
  P.ljs14 = c->ljs14.p;
  P.nbr_count = c->nbr_count.p;
  P.nbr_list = c->nbr_list.p;
  P.sorted_orig = c->sorted_orig.p;
  P.pos = c->pos;
  P.ffix = c->ffix.p;
  P.efix = c->efix.p;
  P.st = c->dstate.p;
  return P;
}

int mdx_enqueue_nonbonded(mdx_ctx* c, bool lj, bool coul, bool energy, unsigned bonded_terms) {
  const NbArgs a = nb_args(c);
  const NbPtrs P = nb_ptrs(c);
  MDX_CHECK(!coul || (a.ctab && c->ctab_beta == c->beta && c->ctab_rc == c->rc), MDX_ERR_INVALID,
            "Ewald-correction table not built for the current beta and cutoff");
  const int lanes = mdx_nb_lanes(c);
  static_assert(NB_BLOCK == BD_BLOCK, "bonded workgroups share the nonbonded launch");
  BondedArgs ba{};
  const int nbb = (int)div_up((long long)c->n * lanes, NB_BLOCK);
  const int nbo = bonded_terms ? mdx_bonded_args(c, bonded_terms, &ba) : 0;
  // resident workgroups: all of them, or nb_persist per compute unit looping over the rest (so
  // that the concurrent PME kernels find room on every compute unit). Unless set, 3 per compute unit
  // when that gives each at most two units of work, else one workgroup per unit: with more units
  // the dispatcher's balancing is worth more. A whole step with 3 per unit / one each (us): 23,328
  // atoms (1,458 units) 88.1 / 89.4, 31,200 (1,950) 106.6 / 102.3, 98,304 (6,144) 375 / 324.
  const int per = c->nb_persist >= 0 ? c->nb_persist : (nbb > 6 * c->ncu ? 0 : 3);
  const int nres = per > 0 ? std::min(nbb, per * c->ncu) : nbb;
  dim3 grid(nres + nbo);
#define NB_LAUNCH4(L_, C_, E_, S_)                                                                     \
  do {                                                                                                 \
    if (lanes == 16)                                                                                   \
      k_nonbonded<L_, C_, E_, 16, S_><<<grid, NB_BLOCK, 0, c->stream>>>(NB_ARGS);                      \
    else if (lanes == 64)                                                                              \
      k_nonbonded<L_, C_, E_, 64, S_><<<grid, NB_BLOCK, 0, c->stream>>>(NB_ARGS);                      \
    else                                                                                               \
      k_nonbonded<L_, C_, E_, 32, S_><<<grid, NB_BLOCK, 0, c->stream>>>(NB_ARGS);                      \
  } while (0)
  // the list holds 1-4 pairs only if the system has scaled pairs
#define NB_LAUNCH(L_, C_, E_)                                                                          \
  do {                                                                                                 \
    if (c->has_s14) NB_LAUNCH4(L_, C_, E_, true); else NB_LAUNCH4(L_, C_, E_, false);                  \
  } while (0)
#define NB_ARGS a, P, ba, nbb, nres
  if (lj && coul) {
    if (energy) NB_LAUNCH(true, true, true); else NB_LAUNCH(true, true, false);
  } else if (lj) {
    if (energy) NB_LAUNCH(true, false, true); else NB_LAUNCH(true, false, false);
  } else {
    if (energy) NB_LAUNCH(false, true, true); else NB_LAUNCH(false, true, false);
  }
#undef NB_LAUNCH
#undef NB_LAUNCH4
#undef NB_ARGS
  MDX_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------------
// Plain Coulomb (mdpy ElectrostaticConstraint): every i < j not excluded, minimum image, no
// cutoff, E = q_i q_j / (4 pi eps0 r). float64, a full double loop (each pair from both ends).
//
// FP64 VALU bound: ~32 float64 instructions per ordered pair. A workgroup takes PC_BLOCK atoms (one
// lane each) against one of S slices of the partners, staged PC_TILE at a time in LDS; S is chosen
// so that the launch has about 4 waves per SIMD however few atoms there are. The slices' partial
// sums stay float64 in scratch and are added in slice order by k_coulomb_reduce, which rounds
// each atom's force to fixed point once (the result does not depend on S beyond float64 rounding).
// 1/r is v_rsq_f64 (relative error e0 < 2^-22) with one third-order step y (1 + e/2 + 3 e^2/8),
// e = 1 - r^2 y^2, which leaves 5/16 e0'^3 < 2^-60: float64 accurate, in 5 instructions instead of a
// square root and a division. Exclusions (and the atom itself) are a 64-bit mask per lane and tile,
// built from the atom's list once per tile; tiles without any for the whole wave skip the test and
// evaluate PC_U partners at a time (independent chains: the estimate and the rounding are slow).
// 12,000 atoms: 4,830 -> 192 + 10 us (before: one 256-lane workgroup per 256 atoms, a square root, a
// division and a walk of the exclusion list per pair). Rounding by adding and subtracting 1.5 2^52
// instead of v_rndne_f64: 190 us, no gain.
#define PC_BLOCK 256
#define PC_TILE 64
#define PC_U 4  // partners in flight per lane
#define PC_WAVES_PER_SIMD 4

// 1/sqrt(x) in float64 from the hardware estimate. The estimate is of the smallest normal where x = 0, so
// coincident charges give the huge energy and NaN force that 1/0 gives; the step takes x itself, so
// NaN (which fmax would replace) stays NaN.
__device__ __forceinline__ double rsqrt64(double x) {
  const double y = __builtin_amdgcn_rsq(fmax(x, 2.2250738585072014e-308));
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

__global__ __launch_bounds__(PC_BLOCK) void k_coulomb_plain(int n, const double* __restrict__ pos,
                                                            const double* __restrict__ q, double Lx, double Ly,
                                                            double Lz, const int* __restrict__ excl_ptr,
                                                            const int* __restrict__ excl_idx, int per_slice,
                                                            double* __restrict__ part) {
  __shared__ double4 tile[PC_TILE];
  const int i = blockIdx.x * PC_BLOCK + threadIdx.x;
  const bool on = i < n;
  double xi = 0, yi = 0, zi = 0;
  int e0 = 0, e1 = 0;
  if (on) {
    xi = pos[3 * i];
    yi = pos[3 * i + 1];
    zi = pos[3 * i + 2];
    if (excl_ptr) {
      e0 = excl_ptr[i];
      e1 = excl_ptr[i + 1];
    }
  }
  double fx = 0, fy = 0, fz = 0, en = 0;
  const double ix = 1.0 / Lx, iy = 1.0 / Ly, iz = 1.0 / Lz;
  auto pair = [&](const double4& pj, double qj) {
    double dx = pj.x - xi, dy = pj.y - yi, dz = pj.z - zi;
    dx = fma(-Lx, rint(dx * ix), dx);
    dy = fma(-Ly, rint(dy * iy), dy);
    dz = fma(-Lz, rint(dz * iz), dz);
    const double rinv = rsqrt64(fma(dx, dx, fma(dy, dy, dz * dz)));
    const double e = qj * rinv;
    const double fr = e * (rinv * rinv);
    fx = fma(fr, dx, fx);
    fy = fma(fr, dy, fy);
    fz = fma(fr, dz, fz);
    en += e;
  };
  const int j0 = blockIdx.y * per_slice, j1 = min(n, j0 + per_slice);
  for (int base = j0; base < j1; base += PC_TILE) {
    __syncthreads();
    if (threadIdx.x < PC_TILE) {
      // zero charges (and the places past the end) sit at the origin: whatever their distance they
      // add exactly 0, as rinv is finite
      const int j = base + threadIdx.x;
      const double qj = j < j1 ? q[j] : 0.0;
      tile[threadIdx.x] = qj != 0.0 ? make_double4(pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], qj)
                                    : make_double4(0, 0, 0, 0);
    }
    __syncthreads();
    unsigned long long skip = 0;  // partners of this tile the lane's atom does not see
    if ((unsigned)(i - base) < (unsigned)PC_TILE) skip = 1ull << (i - base);
    for (int k = e0; k < e1; ++k) {
      const unsigned d = (unsigned)(excl_idx[k] - base);
      if (d < PC_TILE) skip |= 1ull << d;
    }
    if (__ballot(skip != 0) == 0) {
#pragma unroll 1
      for (int t = 0; t < PC_TILE; t += PC_U) {
        double4 pj[PC_U];
#pragma unroll
        for (int u = 0; u < PC_U; ++u) pj[u] = tile[t + u];
#pragma unroll
        for (int u = 0; u < PC_U; ++u) pair(pj[u], pj[u].w);
      }
    } else {
      for (int t = 0; t < PC_TILE; ++t) {
        const double4 pj = tile[t];
        if (!((skip >> t) & 1ull)) pair(pj, pj.w);
      }
    }
  }
  if (!on) return;
  double* p = part + 4ll * n * blockIdx.y;
  p[i] = fx;
  p[n + i] = fy;
  p[2 * n + i] = fz;
  p[3 * n + i] = en;
}

// the slices' sums of one atom per lane, in slice order, then force and energy in fixed point
__global__ __launch_bounds__(PC_BLOCK) void k_coulomb_reduce(int n, int slices, const double* __restrict__ part,
                                                             const double* __restrict__ q, double ke,
                                                             long long* __restrict__ ffix,
                                                             long long* __restrict__ efix) {
  const int i = blockIdx.x * PC_BLOCK + threadIdx.x;
  double v[4] = {0, 0, 0, 0};
  if (i < n && q[i] != 0.0) {
    for (int s = 0; s < slices; ++s)
      for (int d = 0; d < 4; ++d) v[d] += part[4ll * n * s + (long long)d * n + i];
    const double qk = q[i] * ke;
    // force on i = -q_i q_j ke / r^3 (x_j - x_i)
    for (int d = 0; d < 3; ++d)
      atomicAdd((unsigned long long*)&ffix[(long long)d * n + i], (unsigned long long)to_fix(-qk * v[d]));
    v[3] *= qk;
  }
  __shared__ double sm[PC_BLOCK / 64];
  const double en = wave_sum(v[3]);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = en;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < PC_BLOCK / 64; ++w) s += sm[w];
    atomicAdd((unsigned long long*)&efix[7], (unsigned long long)to_fix(0.5 * s));
  }
}

// partner slices of an n-atom launch: enough workgroups for PC_WAVES_PER_SIMD waves on every SIMD,
// whole tiles per slice
static int coulomb_slices(const mdx_ctx* c, int* per_slice) {
  const int blocks = div_up(c->n, PC_BLOCK), tiles = div_up(c->n, PC_TILE);
  const int want = div_up((long long)PC_WAVES_PER_SIMD * std::max(c->ncu, 1), blocks);  // PC_BLOCK lanes: 1 wave a SIMD
  const int per = div_up(tiles, std::max(1, std::min(want, tiles)));
  *per_slice = per * PC_TILE;
  return div_up(tiles, per);
}

int mdx_coulomb_plain_prepare(mdx_ctx* c) {
  int per;
  return c->pc_part.ensure(4 * (size_t)c->n * coulomb_slices(c, &per));
}

int mdx_enqueue_coulomb_plain(mdx_ctx* c) {
  const double ke = 1.0 / (4.0 * M_PI * 0.5727652348434076);  // 1/(4 pi eps0), internal units
  int per;
  const int slices = coulomb_slices(c, &per);
  const int rc = mdx_coulomb_plain_prepare(c);  // already sized when the step is being captured
  if (rc) return rc;
  const int blocks = div_up(c->n, PC_BLOCK);
  k_coulomb_plain<<<dim3(blocks, slices), PC_BLOCK, 0, c->stream>>>(
      c->n, c->pos, c->charge64.p, c->box[0], c->box[1], c->box[2], c->has_excl ? c->excl_ptr.p : nullptr,
      c->excl_idx.p, per, c->pc_part.p);
  MDX_LAUNCH_CHECK();
  k_coulomb_reduce<<<blocks, PC_BLOCK, 0, c->stream>>>(c->n, slices, c->pc_part.p, c->charge64.p, ke, c->ffix.p,
                                                       c->efix.p);
  MDX_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------------
// Batched replicas: every replica's nonbonded workgroups (one per unit of work, no persistent
// loop) followed by its bonded ones, in one launch.
struct NbCall {
  NbArgs a;
  NbPtrs P;
  BondedArgs ba;
  int nb_blocks;  // the replica's nonbonded workgroups; the rest of its workgroups are bonded
  int lanes;      // the replica's lanes per atom
};

template <bool LJ, bool COUL, bool ENERGY, bool S14>
__global__ __launch_bounds__(NB_BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_nonbonded_batch(
    BatchMap map, const NbCall* __restrict__ calls) {
  int b;
  const NbCall& k = calls[batch_replica(map, &b)];
  if (b >= k.nb_blocks) {
    bonded_block(k.ba, b - k.nb_blocks);
    return;
  }
  if (k.lanes == 16) nb_block<LJ, COUL, ENERGY, 16, NB_BLOCK, S14>(k.a, k.P, b);
  else if (k.lanes == 64) nb_block<LJ, COUL, ENERGY, 64, NB_BLOCK, S14>(k.a, k.P, b);
  else nb_block<LJ, COUL, ENERGY, 32, NB_BLOCK, S14>(k.a, k.P, b);
}

int mdx_batch_prepare_nb(mdx_ctx* const* cs, int n, unsigned bonded_terms, BatchKind* out) {
  std::vector<NbCall> calls;
  std::vector<int> blocks;
  bool any_set = false;
  for (int r = 0; r < n; ++r) any_set |= cs[r]->nb_lanes_set;
  const int want = cs[0]->nb_lanes_set ? cs[0]->nb_lanes : 32;
  for (int r = 0; r < n; ++r) {
    mdx_ctx* c = cs[r];
    NbCall k;
    k.lanes = mdx_nb_lanes(c);
    k.a = nb_args(c);
    k.P = nb_ptrs(c);
    MDX_CHECK(k.a.ctab && c->ctab_beta == c->beta && c->ctab_rc == c->rc, MDX_ERR_INVALID,
              "replica %d: Ewald-correction table not built for the current beta and cutoff", r);
    // lanes chosen by the caller have to agree (32 where another replica's were chosen and this
    // one's not); the ones each system gets by itself may differ
    MDX_CHECK((!any_set || (c->nb_lanes_set ? c->nb_lanes : 32) == want) && c->has_s14 == cs[0]->has_s14,
              MDX_ERR_INVALID, "replica %d: batched replicas need the same lanes per atom and 1-4 pair mode", r);
    k.ba = BondedArgs{};
    k.nb_blocks = (int)div_up((long long)c->n * k.lanes, NB_BLOCK);
    const int nbo = bonded_terms ? mdx_bonded_args(c, bonded_terms, &k.ba) : 0;
    calls.push_back(k);
    blocks.push_back(k.nb_blocks + nbo);
  }
  return batch_kind_upload(out, calls, blocks, 0);
}

// LJ + direct-space Coulomb, the batched step's pair terms
int mdx_batch_launch_nb(const BatchKind& k, bool s14, bool energy, hipStream_t s) {
  const NbCall* calls = (const NbCall*)k.calls;
#define NBB(E_, S_) k_nonbonded_batch<true, true, E_, S_><<<k.blocks, NB_BLOCK, 0, s>>>(k.map, calls)
  if (energy) {
    if (s14) NBB(true, true); else NBB(true, false);
  } else {
    if (s14) NBB(false, true); else NBB(false, false);
  }
#undef NBB
  MDX_LAUNCH_CHECK();
  return 0;
}
