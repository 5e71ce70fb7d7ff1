// nbrlist.hip -- device cell neighbor list over groups.
//
// Reproduces the pair set of NeighborList::rebuild_periodic
// (nbrlist.cpp:222-251) bit for bit:
//   * cell of a group = cell_index(floor(x/lc + 0.5), ...) of its first site,
//     FP64, lc = L*(1.0/ncell) (nbrlist.cpp:97, 228-231; pbc.h:25-31);
//   * same-cell pairs are always listed (nbrlist.cpp:243-244);
//   * pairs in distinct neighbouring cells are listed iff the FP64
//     minimum-image distance^2 < (rc+skin)^2 (nbrlist.cpp:245-248,
//     bcond.hpp:56-60, pbc.h:8-14), evaluated in the order the reference
//     evaluates it: first argument in the cell that owns the cell pair row
//     (pbin.c:6), no FMA contraction.
// Layout: groups are counting-sorted by cell (deterministic order within a
// cell), and each sorted group gets a full list (both directions) of sorted
// neighbour indices in a fixed-capacity row, for the pair kernel.
#include "engine.hpp"
#include "scan.hpp"
#include "reduce.hpp"
#include "pack.hpp"

#pragma clang fp contract(off)

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

// Skin test, cells, counts and the cells' lists of groups (head, next); the
// last block to finish scans the counts into sorted group offsets.  Only a
// step that rebuilds pays for the fence and the counter.
// from_part: the skin test on the partials of the kernel that moved the
// positions; every block forms the same outcome, a rebuild already requested
// stays requested, and block 0 records it for the rest of the chain.
__global__ void __launch_bounds__(256) k_nl_assign(
    const SysParams *__restrict__ sp, const int *__restrict__ gfirst,
    const double *__restrict__ r, int nsite_total, int *__restrict__ rebuild,
    int *__restrict__ gcell, double *__restrict__ last, int *__restrict__ cell_count,
    int *__restrict__ cell_start, int *__restrict__ head, int *__restrict__ next,
    int *__restrict__ done, unsigned long long *__restrict__ builds, int *__restrict__ err,
    const double *__restrict__ part, int maxblk, int from_part, const int *__restrict__ cell_rank) {
  __shared__ int lastblk;
  const int s = blockIdx.y;
  const SysParams &P = sp[s];
  const int nblk = (P.ngroup + 255) / 256;
  if ((int)blockIdx.x >= nblk) return;
  int want = rebuild[s];
  if (from_part) {
    const bool fire = skin_fires(P, s, part, maxblk);
    want |= fire;
    if (blockIdx.x == 0 && threadIdx.x == 0 && fire) rebuild[s] = 1;
  }
  if (!want) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) builds[s] += 1;
  if (i < P.ngroup) {
    const int g = P.group0 + i;
    const int site = gfirst[g];
    const double x = r[site], y = r[nsite_total + site], z = r[2 * nsite_total + site];
    int c = stored_cell(P, x, y, z, cell_rank);
    if (c < 0) {
      atomicOr(err, ERR_NAN);   // reported; the group is parked in cell 0
      c = 0;
    }
    c += P.cell0;
    gcell[g] = c;
    last[3 * g] = x;
    last[3 * g + 1] = y;
    last[3 * g + 2] = z;
    next[g] = atomicExch(&head[c], g);
    atomicAdd(&cell_count[c], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    lastblk = atomicAdd(&done[s], 1) == nblk - 1;
  }
  __syncthreads();
  if (!lastblk) return;
  __threadfence();
  if (threadIdx.x == 0) done[s] = 0;
  block_scan_clear(cell_count + P.cell0, cell_start + P.cell0, P.ncell * P.ncell * P.ncell, P.group0);
}

// The groups of each cell from its list, in ascending order, one thread per
// cell; the lists are cleared for the next build.  After a non-finite
// position (its group parked in cell 0) or in a collapsed cell the list is
// not walked: the rows of an error are discarded, and the slots keep the
// order of the last build.
__global__ void k_nl_order(const SysParams *__restrict__ sp, const int *__restrict__ rebuild,
                           const int *__restrict__ cell_start, int *__restrict__ head,
                           const int *__restrict__ next, int *__restrict__ order,
                           const double *__restrict__ last, double4 *__restrict__ gpos,
                           int *__restrict__ err) {
  const int s = blockIdx.y;
  if (!rebuild[s]) return;
  const SysParams &P = sp[s];
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= P.ncell * P.ncell * P.ncell) return;
  int g = head[P.cell0 + c];
  head[P.cell0 + c] = -1;
  if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_NAN) return;
  const int b = cell_start[P.cell0 + c], n = cell_start[P.cell0 + c + 1] - b;
  if (n > NL_SORT_MAX) {   // collapsed positions: reported, not sorted
    atomicOr(err, ERR_CELL);
    return;
  }
  int v[NL_CELL_REGS];
  if (n <= NL_CELL_REGS) {
#pragma unroll
    for (int k = 0; k < NL_CELL_REGS; k++) {
      if (k >= n) break;
      v[k] = g;
      g = next[g];
    }
  } else {
    for (int k = 0; k < n; k++, g = next[g]) order[b + k] = g;
  }
  place_cell(b, n, v, order, last, gpos);
}

// The same for one system in one block, with the cells' counts in LDS: one
// launch less, which a step that does not rebuild saves about 2.5 us by.  A
// rebuild takes one block 27 us for 4 096 groups (20 in the two kernels
// above) and 200 for 32 768 (45), so with a rebuild every 25 to 30 steps the
// line lies near 8 000 groups.
constexpr int NL_BIN_TB = 1024;
constexpr int NL_BIN_CELLS = 12000;    // 47 KB of counts
constexpr int NL_BIN_GROUPS = 8192;

__global__ void __launch_bounds__(NL_BIN_TB) k_nl_bin(
    const SysParams *__restrict__ sp, const int *__restrict__ gfirst,
    const double *__restrict__ r, int N, int *__restrict__ rebuild, int *__restrict__ gcell,
    double *__restrict__ last, int *__restrict__ cell_start, int *__restrict__ order,
    double4 *__restrict__ gpos, unsigned long long *__restrict__ builds, int *__restrict__ err,
    const double *__restrict__ part, int maxblk, int from_part, const int *__restrict__ cell_rank) {
  extern __shared__ int cnt[];
  __shared__ int wsum[NL_BIN_TB / 64], bad;
  const int s = blockIdx.x, tid = threadIdx.x;
  const SysParams &P = sp[s];
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
  for (int c = tid; c < nc; c += NL_BIN_TB) cnt[c] = 0;
  __syncthreads();
  constexpr int U = 4;   // groups in flight per thread
  for (int i0 = tid; i0 < G; i0 += U * NL_BIN_TB) {
    int site[U];
    double x[U][3];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * NL_BIN_TB;
      site[u] = gfirst[P.group0 + (i < G ? i : 0)];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int d = 0; d < 3; d++) x[u][d] = r[(long)d * N + site[u]];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * NL_BIN_TB, g = P.group0 + i;
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
  const int per = (nc + NL_BIN_TB - 1) / NL_BIN_TB, c0 = min(tid * per, nc), c1 = min(c0 + per, nc);
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
  for (int i0 = tid; i0 < G; i0 += U * NL_BIN_TB) {
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * NL_BIN_TB;
      c[u] = i < G ? gcell[P.group0 + i] - P.cell0 : 0;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + u * NL_BIN_TB;
      if (i < G) order[atomicAdd(&cnt[c[u]], 1)] = P.group0 + i;
    }
  }
  __syncthreads();
  if (bad) return;   // the rows of an error are discarded, so skip the sort
  for (int c = tid; c < nc; c += NL_BIN_TB) {
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

__global__ void __launch_bounds__(256) k_nl_pairs(
    const SysParams *__restrict__ sp, const int *__restrict__ rebuild,
    const int *__restrict__ order, const int *__restrict__ gcell,
    const int *__restrict__ cell_start, const int4 *__restrict__ sten, int nbcap,
    int *__restrict__ nbr, int *__restrict__ nnb, int *__restrict__ err,
    const double *__restrict__ r, int N, const double *__restrict__ q,
    const int *__restrict__ gfirst, const int *__restrict__ gns, const int *__restrict__ ginfo,
    const double4 *__restrict__ gpos, float4 *__restrict__ spk, int2 *__restrict__ gmeta,
    const int *__restrict__ gexcl, int4 *__restrict__ gslot, const int *__restrict__ cell_rank,
    const int *__restrict__ cell_unrank, int *__restrict__ gslot_inv) {
#pragma clang fp contract(off)
  __shared__ int c_start[4][NL_SEG], c_off[4][NL_SEG + 1], c_cell[4][NL_SEG];
  const int s = blockIdx.y;
  if (!rebuild[s]) return;
  const SysParams &P = sp[s];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int *cs = c_start[wv], *co = c_off[wv], *cc = c_cell[wv];
  const unsigned long long below = (1ull << lane) - 1ull;
  // one wavefront per sorted group (the loop strides only if the grid is
  // smaller); more waves in flight hide the candidate loads of a rebuild
  // better than a grid-stride over a small grid (measured, and the empty
  // launches of the steps that do not rebuild cost no more)
  const int nwave = (int)((gridDim.x * blockDim.x) >> 6);
  // after a non-finite or collapsed position the cells are meaningless (all
  // groups may share one): leave the rows empty
  const bool bad =
      (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & (ERR_NAN | ERR_CELL)) != 0;
  for (int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); wave < P.ngroup;
       wave += nwave) {
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
    // k_pack; the first-site positions were written by k_nl_sortcell)
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

__global__ void k_set_flags(int *f, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) f[i] = v;
}

// Externally supplied positions: the pair kernel's packed inputs in the
// present sorted order (as k_pack) and the displacements since the last build
// (nbrlist.cpp:64-76) as per-block partials that the build check merges.  One
// block per FIN_TB groups; a block per system alone took 35 us for 32 768
// groups, and the packing was a kernel of its own (6.5 us): 6.3 us for both
__global__ void __launch_bounds__(FIN_TB) k_skin_pack(
    const SysParams *__restrict__ sp, const int *__restrict__ order, const int *__restrict__ gfirst,
    const int *__restrict__ gns, const int *__restrict__ ginfo, const double *__restrict__ r,
    const double *__restrict__ q, int N, const double *__restrict__ last,
    double4 *__restrict__ gpos, float4 *__restrict__ spk, int2 *__restrict__ gmeta,
    double *__restrict__ part, int maxblk) {
  __shared__ double red[FIN_TB / 64][2];
  const int s = blockIdx.y;
  const SysParams &P = sp[s];
  const int i = blockIdx.x * FIN_TB + threadIdx.x;
  if ((int)(blockIdx.x * FIN_TB) >= P.ngroup) return;
  double top[2] = {0, 0};
  if (i < P.ngroup) {
    const int gs = P.group0 + i;
    const int g = order[gs];
    const double4 p = pack_group(gs, gfirst[g], gns[g], ginfo[g], r, q, N, gpos, spk, gmeta);
    const double dx = p.x - last[3 * g], dy = p.y - last[3 * g + 1], dz = p.z - last[3 * g + 2];
    const double d = sqrt(dx * dx + dy * dy + dz * dz);
    top[0] = d <= 1e300 ? d : 1e300;   // a non-finite position (or a list built from one) rebuilds
  }
  block_reduce<2, 0, FIN_TB>(top, red);
  if (threadIdx.x == 0) {
    double *o = part + ((long)s * maxblk + blockIdx.x) * FIN_NPART + FIN_TOP;
    o[0] = top[0];
    o[1] = top[1];
  }
}

// after it, launch_nl_build takes the partials
int launch_skin_pack(Engine &e) {
  hipLaunchKernelGGL(k_skin_pack, dim3((e.maxg + FIN_TB - 1) / FIN_TB, e.nsys), dim3(FIN_TB), 0,
                     e.stream, e.d_sp, e.d_order, e.d_gfirst, e.d_gns, e.d_ginfo, e.d_r, e.d_q,
                     e.nsite, e.d_last, e.d_gpos, e.d_spk, e.d_gmeta, e.d_fpart, e.nblk_part);
  MM_HIP(hipGetLastError());
  return 0;
}

int launch_set_rebuild(Engine &e, int value) {
  hipLaunchKernelGGL(k_set_flags, dim3((e.nsys + 63) / 64), dim3(64), 0, e.stream, e.d_rebuild,
                     e.nsys, value);
  MM_HIP(hipGetLastError());
  return 0;
}

int launch_nl_build(Engine &e, int force, int from_partials) {
  if (force) {
    int rc = launch_set_rebuild(e);
    if (rc) return rc;
  }
  const int tb = 256;
  dim3 gg((e.maxg + tb - 1) / tb, e.nsys);
  const double *r = e.d_r;
  int maxc = 0;
  for (auto &p : e.hsp) maxc = std::max(maxc, p.ncell * p.ncell * p.ncell);
  if (maxc <= NL_BIN_CELLS && e.maxg <= NL_BIN_GROUPS) {
    hipLaunchKernelGGL(k_nl_bin, dim3(e.nsys), dim3(NL_BIN_TB), sizeof(int) * maxc, e.stream, e.d_sp,
                       e.d_gfirst, r, e.nsite, e.d_rebuild, e.d_gcell, e.d_last, e.d_cell_start,
                       e.d_order, e.d_gpos, e.d_nlb, e.d_err, e.d_fpart, e.nblk_part, from_partials,
                       e.d_cell_rank);
  } else {
    hipLaunchKernelGGL(k_nl_assign, gg, dim3(tb), 0, e.stream, e.d_sp, e.d_gfirst, r, e.nsite,
                       e.d_rebuild, e.d_gcell, e.d_last, e.d_cell_count, e.d_cell_start,
                       e.d_cell_head, e.d_gnext, e.d_done + 3 * e.nsys, e.d_nlb, e.d_err, e.d_fpart,
                       e.nblk_part, from_partials, e.d_cell_rank);
    hipLaunchKernelGGL(k_nl_order, dim3((maxc + tb - 1) / tb, e.nsys), dim3(tb), 0, e.stream,
                       e.d_sp, e.d_rebuild, e.d_cell_start, e.d_cell_head, e.d_gnext, e.d_order,
                       e.d_last, e.d_gpos, e.d_err);
  }
  hipLaunchKernelGGL(k_nl_pairs, dim3((e.maxg + 3) / 4, e.nsys), dim3(256), 0,
                     e.stream, e.d_sp, e.d_rebuild, e.d_order, e.d_gcell, e.d_cell_start,
                     e.d_sten, e.nbcap, e.d_nbr, e.d_nnb, e.d_err, e.d_r, e.nsite, e.d_q,
                     e.d_gfirst, e.d_gns, e.d_ginfo, e.d_gpos, e.d_spk, e.d_gmeta, e.d_gexcl,
                     e.d_gslot, e.d_cell_rank, e.d_cell_unrank, e.d_gslot_inv);
  MM_HIP(hipGetLastError());
  return 0;
}

}  // namespace mmamd
