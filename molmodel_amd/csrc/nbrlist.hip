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
#include "nlist.hpp"
#include "scan.hpp"
#include "reduce.hpp"
#include "pack.hpp"

#pragma clang fp contract(off)

namespace mmamd {

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
  // Every wave waits until its own counts have been made (vmcnt 0) before the
  // barrier, which waits for no memory, and thread 0's fence only for its own
  // wave's: the last block must not scan while a count is on its way.  (A fence
  // in every wave does it too, and writes the L2 back four times as often: 51
  // us a rebuild of 32768 groups instead of 40)
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    lastblk = atomicAdd(&done[s], 1) == nblk - 1;
  }
  __syncthreads();
  if (!lastblk) return;
  __threadfence();
  if (threadIdx.x == 0) done[s] = 0;
  if (block_scan_clear(cell_count + P.cell0, cell_start + P.cell0, P.ncell * P.ncell * P.ncell,
                       P.group0, NL_SORT_MAX))
    atomicOr(err, ERR_CELL);   // collapsed positions: reported, not sorted
}

// The groups of each cell from its list, in ascending order, one thread per
// cell; the lists are cleared for the next build.  After a non-finite
// position (its group parked in cell 0) or a collapsed cell no list is
// walked: the rows of an error are discarded, and the slots keep the order of
// the last build, so that every group has one whatever was reported (the next
// skin test walks them).
__global__ void k_nl_order(const SysParams *__restrict__ sp, const int *__restrict__ rebuild,
                           const int *__restrict__ cell_start, int *__restrict__ head,
                           const int *__restrict__ next, int *__restrict__ order,
                           const double *__restrict__ last, double4 *__restrict__ gpos,
                           const int *__restrict__ err) {
  const int s = blockIdx.y;
  if (!rebuild[s]) return;
  const SysParams &P = sp[s];
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= P.ncell * P.ncell * P.ncell) return;
  int g = head[P.cell0 + c];
  head[P.cell0 + c] = -1;
  if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & (ERR_NAN | ERR_CELL)) return;
  const int b = cell_start[P.cell0 + c], n = cell_start[P.cell0 + c + 1] - b;
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

__global__ void __launch_bounds__(NL_BIN_TB) k_nl_bin(const SysParams *__restrict__ sp, NlArgs a) {
  extern __shared__ int cnt[];
  a.bin<NL_BIN_TB>(sp[blockIdx.x], blockIdx.x, cnt);
}

__global__ void __launch_bounds__(256) k_nl_pairs(const SysParams *__restrict__ sp, NlArgs a) {
  __shared__ int lds[4 * NL_LDS];
  a.pairs<4>(sp[blockIdx.y], blockIdx.y, blockIdx.x, gridDim.x, lds);
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

int nl_prepare(Engine &e, int force, int from_partials, NlArgs &a, int &maxc) {
  if (force) {
    int rc = launch_set_rebuild(e);
    if (rc) return rc;
  }
  maxc = 0;
  for (auto &p : e.hsp) maxc = std::max(maxc, p.ncell * p.ncell * p.ncell);
  a = {e.d_gfirst, e.d_gns, e.d_ginfo, e.d_gexcl, e.d_r, e.d_q, e.nsite, e.d_rebuild, e.d_gcell,
       e.d_last, e.d_cell_start, e.d_order, e.d_gpos, e.d_nlb, e.d_err, e.d_fpart, e.nblk_part,
       from_partials, e.d_cell_rank, e.d_cell_unrank, e.d_sten, e.nbcap, e.d_nbr, e.d_nnb, e.d_spk,
       e.d_gmeta, e.d_gslot, e.d_gslot_inv};
  return 0;
}

int launch_nl_build(Engine &e, int force, int from_partials) {
  NlArgs a;
  int maxc;
  if (int rc = nl_prepare(e, force, from_partials, a, maxc)) return rc;
  const int tb = 256;
  if (maxc <= NL_BIN_CELLS && e.maxg <= NL_BIN_GROUPS) {
    hipLaunchKernelGGL(k_nl_bin, dim3(e.nsys), dim3(NL_BIN_TB), sizeof(int) * maxc, e.stream, e.d_sp,
                       a);
  } else {
    hipLaunchKernelGGL(k_nl_assign, dim3((e.maxg + tb - 1) / tb, e.nsys), dim3(tb), 0, e.stream,
                       e.d_sp, e.d_gfirst, e.d_r, e.nsite,
                       e.d_rebuild, e.d_gcell, e.d_last, e.d_cell_count, e.d_cell_start,
                       e.d_cell_head, e.d_gnext, e.d_done + 3 * e.nsys, e.d_nlb, e.d_err, e.d_fpart,
                       e.nblk_part, from_partials, e.d_cell_rank);
    hipLaunchKernelGGL(k_nl_order, dim3((maxc + tb - 1) / tb, e.nsys), dim3(tb), 0, e.stream,
                       e.d_sp, e.d_rebuild, e.d_cell_start, e.d_cell_head, e.d_gnext, e.d_order,
                       e.d_last, e.d_gpos, e.d_err);
  }
  hipLaunchKernelGGL(k_nl_pairs, dim3((e.maxg + 3) / 4, e.nsys), dim3(256), 0, e.stream, e.d_sp, a);
  MM_HIP(hipGetLastError());
  return 0;
}

}  // namespace mmamd
