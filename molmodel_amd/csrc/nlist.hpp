// nlist.hpp -- the block-wide parts of a neighbour-list build that several
// kernels carry: those of nbrlist.hip, and the reciprocal-space kernels of
// small systems, which take them along (kspace.hip).  FP64 as the reference
// forms it: no contraction.
#pragma once
#include "engine.hpp"
#include "reduce.hpp"

namespace mmamd {

__device__ __forceinline__ double min_image_sq(double ax, double ay, double az, double bx,
                                               double by, double bz, double L, double invL) {
#pragma clang fp contract(off)
  double x = ax - bx, y = ay - by, z = az - bz;
  x -= L * floor(x * invL + 0.5);
  y -= L * floor(y * invL + 0.5);
  z -= L * floor(z * invL + 0.5);
  return x * x + y * y + z * z;
}

// The skin test (nbrlist.cpp:64-76) on the largest and second largest
// first-site displacement since the last build, merged from per-block
// partials in the finish kernel's layout (FIN_TB groups a block).  Every
// thread of the block calls it and gets the outcome.
__device__ __forceinline__ bool skin_fires(const SysParams &P, int s, const double *__restrict__ part,
                                           int maxblk) {
  __shared__ double w1[16], w2[16];
  __shared__ int fire;
  const int nb = (P.ngroup + FIN_TB - 1) / FIN_TB;
  double t1 = 0, t2 = 0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    const double *q = part + ((long)s * maxblk + b) * FIN_NPART + FIN_TOP;
    top2_merge(t1, t2, load_coherent(q), load_coherent(q + 1));
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const double b1 = __shfl_xor(t1, o), b2 = __shfl_xor(t2, o);
    top2_merge(t1, t2, b1, b2);
  }
  if ((threadIdx.x & 63) == 0) { w1[threadIdx.x >> 6] = t1; w2[threadIdx.x >> 6] = t2; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double u1 = w1[0], u2 = w2[0];
    for (int k = 1; k < (int)(blockDim.x >> 6); k++) top2_merge(u1, u2, w1[k], w2[k]);
    fire = u1 + u2 > P.skin;   // nbrlist.cpp:75-76
  }
  __syncthreads();
  return fire;
}

// the stored cell of a first site at (x, y, z), -1 for a position that is not
// finite or so far out that a cell index would leave int range (an error)
__device__ __forceinline__ int stored_cell(const SysParams &P, double x, double y, double z,
                                           const int *__restrict__ cell_rank) {
#pragma clang fp contract(off)
  const double lim = 1e9 * P.lc;
  if (!(fabs(x) <= lim && fabs(y) <= lim && fabs(z) <= lim)) return -1;
  const int n = P.ncell;
  const int ix = (int)floor(x / P.lc + 0.5);
  const int iy = (int)floor(y / P.lc + 0.5);
  const int iz = (int)floor(z / P.lc + 0.5);
  // stored at the cell's position along the Hilbert curve
  return cell_rank[P.cell0 + (mod_nonneg(ix, n) * n + mod_nonneg(iy, n)) * n + mod_nonneg(iz, n)];
}

// groups one cell may hold: far above any physical density (cells hold
// about two groups on average), low enough that the serial sort stays short
constexpr int NL_SORT_MAX = 512;
constexpr int NL_CELL_REGS = 8;   // cells up to this size are sorted in registers

// A cell's n groups (v: the first NL_CELL_REGS of them; all of them already in
// order[b ..] if there are more) into ascending group order at order[b ..],
// so that the sorted order is deterministic, and their first-site positions
// into the pair kernel's gpos.
__device__ __forceinline__ void place_cell(int b, int n, int *v, int *__restrict__ order,
                                           const double *__restrict__ last,
                                           double4 *__restrict__ gpos) {
  if (n <= NL_CELL_REGS) {
#pragma unroll
    for (int k = 0; k < NL_CELL_REGS; k++) v[k] = k < n ? v[k] : 0x7fffffff;
#pragma unroll
    for (int p = 0; p < NL_CELL_REGS; p++)   // odd-even transpositions
#pragma unroll
      for (int k = p & 1; k + 1 < NL_CELL_REGS; k += 2) {
        const int lo = min(v[k], v[k + 1]);
        v[k + 1] = max(v[k], v[k + 1]);
        v[k] = lo;
      }
    double4 p[NL_CELL_REGS];
#pragma unroll
    for (int k = 0; k < NL_CELL_REGS; k++)
      if (k < n) p[k] = make_double4(last[3 * v[k]], last[3 * v[k] + 1], last[3 * v[k] + 2], 0.0);
#pragma unroll
    for (int k = 0; k < NL_CELL_REGS; k++)
      if (k < n) {
        order[b + k] = v[k];
        gpos[b + k] = p[k];
      }
    return;
  }
  for (int i = b + 1; i < b + n; i++) {
    const int x = order[i];
    int j = i - 1;
    while (j >= b && order[j] > x) { order[j + 1] = order[j]; j--; }
    order[j + 1] = x;
  }
  for (int i = b; i < b + n; i++) {
    const int g = order[i];
    gpos[i] = make_double4(last[3 * g], last[3 * g + 1], last[3 * g + 2], 0.0);
  }
}

// Skin test, cells, counts, sorted order and gpos of one system in one block,
// with the cells' counts in LDS (cnt, P.ncell^3 of them).
template <int TB>
__device__ __forceinline__ void nl_bin_block(
    const SysParams &P, int s, int *cnt, const int *__restrict__ gfirst,
    const double *__restrict__ r, int N, int *__restrict__ rebuild, int *__restrict__ gcell,
    double *__restrict__ last, int *__restrict__ cell_start, int *__restrict__ order,
    double4 *__restrict__ gpos, unsigned long long *__restrict__ builds, int *__restrict__ err,
    const double *__restrict__ part, int maxblk, int from_part, const int *__restrict__ cell_rank) {
#pragma clang fp contract(off)
  __shared__ int wsum[TB / 64], bad;
  const int tid = threadIdx.x;
  int want = rebuild[s];
  if (from_part && skin_fires(P, s, part, maxblk)) {
    if (tid == 0) rebuild[s] = 1;
    want = 1;
  }
  if (!want) return;
  const int nc = P.ncell * P.ncell * P.ncell, G = P.ngroup;
  if (tid == 0) {
    builds[s] += 1;
    // another system's error leaves this one's rows empty too (k_nl_pairs)
    bad = (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_NAN) != 0;
  }
  for (int c = tid; c < nc; c += TB) cnt[c] = 0;
  __syncthreads();
  constexpr int U = 4;   // groups in flight per thread
  for (int i0 = tid; i0 < G; i0 += U * TB) {
    int site[U];
    double x[U][3];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * TB;
      site[u] = gfirst[P.group0 + (i < G ? i : 0)];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int d = 0; d < 3; d++) x[u][d] = r[(long)d * N + site[u]];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * TB, g = P.group0 + i;
      if (i >= G) break;
      int c = stored_cell(P, x[u][0], x[u][1], x[u][2], cell_rank);
      if (c < 0) {
        atomicOr(err, ERR_NAN);   // reported; the group is parked in cell 0
        bad = 1;
        c = 0;
      }
      gcell[g] = P.cell0 + c;
      last[3 * g] = x[u][0];
      last[3 * g + 1] = x[u][1];
      last[3 * g + 2] = x[u][2];
      atomicAdd(&cnt[c], 1);
    }
  }
  __syncthreads();
  // exclusive scan: each thread its own run of cells, then over the block
  const int per = (nc + TB - 1) / TB, c0 = min(tid * per, nc), c1 = min(c0 + per, nc);
  int sum = 0;
  for (int c = c0; c < c1; c++) sum += cnt[c];
  int incl = sum;
  const int lane = tid & 63, wid = tid >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  int at = P.group0 + incl - sum;
  for (int w = 0; w < wid; w++) at += wsum[w];
  for (int c = c0; c < c1; c++) {
    const int n = cnt[c];
    cell_start[P.cell0 + c] = at;
    cnt[c] = at;   // the next free slot of the cell
    at += n;
  }
  if (tid == 0) cell_start[P.cell0 + nc] = P.group0 + G;
  __syncthreads();
  for (int i0 = tid; i0 < G; i0 += U * TB) {
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * TB;
      c[u] = i < G ? gcell[P.group0 + i] - P.cell0 : 0;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * TB;
      if (i < G) order[atomicAdd(&cnt[c[u]], 1)] = P.group0 + i;
    }
  }
  __syncthreads();
  if (bad) return;   // the rows of an error are discarded, so skip the sort
  for (int c = tid; c < nc; c += TB) {
    // cnt[c] is now the end of cell c and the start of cell c + 1
    const int b = c ? cnt[c - 1] : P.group0, n = cnt[c] - b;
    if (n > NL_SORT_MAX) {   // collapsed positions: reported, not sorted
      atomicOr(err, ERR_CELL);
      continue;
    }
    int v[NL_CELL_REGS];
#pragma unroll
    for (int k = 0; k < NL_CELL_REGS; k++)
      if (k < n) v[k] = order[b + k];
    place_cell(b, n, v, order, last, gpos);
  }
}

// One wavefront per sorted group.  The stencil cells that can hold a pair
// (the group's own cell and those whose box lies within rc + skin of it)
// are compacted into a per-wavefront list with their counts' prefix sums;
// their candidates are then laid end to end, each lane takes one, and the
// accepted ones are compacted with a ballot.  The row lists the stencil
// cells in order and each cell's groups in sorted order.
constexpr int NL_SEG = 256;   // listed cells per wavefront before a flush
constexpr int NL_LDS = 3 * NL_SEG + 1;

template <int NW>
__device__ __forceinline__ void nl_pairs_block(
    const SysParams &P, int blk, int nblk, int *lds,
    const int *__restrict__ order, const int *__restrict__ gcell,
    const int *__restrict__ cell_start, const int4 *__restrict__ sten, int nbcap,
    int *__restrict__ nbr, int *__restrict__ nnb, int *__restrict__ err,
    const double *__restrict__ r, int N, const double *__restrict__ q,
    const int *__restrict__ gfirst, const int *__restrict__ gns, const int *__restrict__ ginfo,
    const double4 *__restrict__ gpos, float4 *__restrict__ spk, int2 *__restrict__ gmeta,
    const int *__restrict__ gexcl, int4 *__restrict__ gslot, const int *__restrict__ cell_rank,
    const int *__restrict__ cell_unrank, int *__restrict__ gslot_inv) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int *cs = lds + wv * NL_LDS, *co = cs + NL_SEG, *cc = co + NL_SEG + 1;
  const unsigned long long below = (1ull << lane) - 1ull;
  // one wavefront per sorted group (the loop strides only if the grid is
  // smaller); more waves in flight hide the candidate loads of a rebuild
  // better than a grid-stride over a small grid (measured, and the empty
  // launches of the steps that do not rebuild cost no more)
  const int nwave = nblk * NW;
  // after a non-finite or collapsed position the cells are meaningless (all
  // groups may share one): leave the rows empty
  const bool bad =
      (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & (ERR_NAN | ERR_CELL)) != 0;
  for (int wave = blk * NW + wv; wave < P.ngroup; wave += nwave) {
    const int gs = P.group0 + wave;
    const int g = order[gs];
    // the finish kernel's per-slot indices in the new order
    if (lane == 0) {
      gslot[gs] = make_int4(g, gfirst[g], gns[g], gexcl[g]);
      gslot_inv[g] = gs;
    }
    if (bad) {   // the error is reported; the rows stay empty
      if (lane == 0) nnb[gs] = 0;
      continue;
    }
    const int n = P.ncell;
    // A, B: cell indices (ix*n + iy)*n + iz, as the reference numbers them;
    // cells are stored at their Hilbert positions (cell_rank)
    const int A = cell_unrank[gcell[g]];
    const int ax = A / (n * n), ay = (A / n) % n, az = A % n;
    const double4 pg = gpos[gs];
    const double L = P.L, invL = 1 / P.L;
    const double c2 = P.nl_c2;
    int cnt = 0;
    int *row = nbr + (long)gs * nbcap;
    int nseg = 0, tot = 0;   // listed cells and their candidates (wave-uniform)
    if (lane == 0) co[0] = 0;
    // test the listed cells' candidates and append the accepted ones
    auto flush = [&]() {
      __builtin_amdgcn_wave_barrier();
      for (int u0 = 0; u0 < tot; u0 += 64) {
        const int u = u0 + lane;
        bool take = false;
        int hs = -1;
        if (u < tot) {
          int lo = 0, hi = nseg - 1;   // last cell with co[k] <= u
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (co[mid] <= u) lo = mid; else hi = mid - 1;
          }
          hs = cs[lo] + (u - co[lo]);
          const int B = cc[lo];
          if (hs != gs) {
            if (B == A) {
              take = true;
            } else {
              // the cell that owns the (A,B) row supplies the first argument
              int ra = A, rb = B;
              canonical_pair(ra, rb);
              const double4 ph = gpos[hs];
              const double d2 = (ra == A) ? min_image_sq(pg.x, pg.y, pg.z, ph.x, ph.y, ph.z, L, invL)
                                          : min_image_sq(ph.x, ph.y, ph.z, pg.x, pg.y, pg.z, L, invL);
              take = d2 < c2;
            }
          }
        }
        const unsigned long long bal = __ballot(take);
        if (take) {
          const int pos = cnt + __popcll(bal & below);
          if (pos < nbcap) row[pos] = hs;
        }
        cnt += __popcll(bal);
      }
      __builtin_amdgcn_wave_barrier();   // the cell list is rewritten next
      nseg = 0;
      tot = 0;
    };
    for (int t0 = 0; t0 < P.nsten; t0 += 64) {
      const int t = t0 + lane;
      int nb = 0, start = 0, B = -1;
      if (t < P.nsten) {
        const int4 o = sten[P.sten0 + t];
        const int bxx = (ax + o.x) % n, byy = (ay + o.y) % n, bzz = (az + o.z) % n;
        B = (bxx * n + byy) * n + bzz;
        const int Bs = P.cell0 + cell_rank[P.cell0 + B];
        start = cell_start[Bs];
        nb = cell_start[Bs + 1] - start;
        // a cell whose box (cell b holds x in [(b - 1/2) lc, (b + 1/2) lc)
        // mod L) lies farther than rc + skin from this group holds no pair;
        // the margin covers the rounding of the cell assignment
        if (B != A) {
          const double lc = P.lc, h = 0.5 * P.lc;
          double dx = pg.x - bxx * lc, dy = pg.y - byy * lc, dz = pg.z - bzz * lc;
          dx = fabs(dx - L * floor(dx * invL + 0.5)) - h;
          dy = fabs(dy - L * floor(dy * invL + 0.5)) - h;
          dz = fabs(dz - L * floor(dz * invL + 0.5)) - h;
          dx = dx > 0 ? dx : 0;
          dy = dy > 0 ? dy : 0;
          dz = dz > 0 ? dz : 0;
          if (dx * dx + dy * dy + dz * dz > c2 * (1 + 1e-9) + 1e-9) nb = 0;
        }
      }
      const unsigned long long keep = __ballot(nb > 0);
      const int k = __popcll(keep);
      if (nseg + k > NL_SEG) flush();
      int incl = nb;   // inclusive scan of the kept counts over the wave
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
      }
      if (nb > 0) {
        const int at = nseg + __popcll(keep & below);
        cs[at] = start;
        cc[at] = B;
        co[at + 1] = tot + incl;
      }
      tot += __shfl(incl, 63);
      nseg += k;
    }
    if (nseg > 0) flush();
    if (lane == 0) {
      if (cnt > nbcap) {
        atomicOr(err, ERR_NL_OVERFLOW);
        cnt = nbcap;
      }
      nnb[gs] = cnt;
    }
    // the pair kernel's packed site inputs in the new sorted order (as
    // k_pack; the first-site positions were written with the order)
    const int s0 = gfirst[g], ns = gns[g];
    if (lane == 0) gmeta[gs] = make_int2(ns, ginfo[g]);
    if (lane < MAXS) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (lane < ns) {
        const int sk = s0 + lane;
        v = make_float4((float)(r[sk] - pg.x), (float)(r[N + sk] - pg.y), (float)(r[2 * N + sk] - pg.z),
                        ((ginfo[g] >> (8 * lane)) & SITE_HAS_Q) ? (float)q[sk] : 0.f);
      }
      spk[(long)gs * MAXS + lane] = v;
    }
  }
}

// what both parts read and write
struct NlArgs {
  const int *gfirst, *gns, *ginfo, *gexcl;
  const double *r, *q;
  int N;
  int *rebuild, *gcell;
  double *last;
  int *cell_start, *order;
  double4 *gpos;
  unsigned long long *builds;
  int *err;
  const double *part;
  int maxblk, from_part;
  const int *cell_rank, *cell_unrank;
  const int4 *sten;
  int nbcap;
  int *nbr, *nnb;
  float4 *spk;
  int2 *gmeta;
  int4 *gslot;
  int *gslot_inv;

  template <int TB>
  __device__ __forceinline__ void bin(const SysParams &P, int s, int *cnt) const {
    nl_bin_block<TB>(P, s, cnt, gfirst, r, N, rebuild, gcell, last, cell_start, order, gpos, builds,
                     err, part, maxblk, from_part, cell_rank);
  }
  template <int NW>
  __device__ __forceinline__ void pairs(const SysParams &P, int s, int blk, int nblk, int *lds) const {
    if (!rebuild[s]) return;
    nl_pairs_block<NW>(P, blk, nblk, lds, order, gcell, cell_start, sten, nbcap, nbr, nnb, err, r, N,
                       q, gfirst, gns, ginfo, gpos, spk, gmeta, gexcl, gslot, cell_rank, cell_unrank,
                       gslot_inv);
  }
};

// one block per system up to these sizes (nbrlist.hip)
constexpr int NL_BIN_CELLS = 12000;    // 47 KB of counts
constexpr int NL_BIN_GROUPS = 8192;

// launch arguments; sets the rebuild flags if force
int nl_prepare(Engine &e, int force, int from_partials, NlArgs &a, int &maxc);

}  // namespace mmamd
