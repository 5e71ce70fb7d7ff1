// kspace.hip -- plain Ewald reciprocal-space sum, FP64 (kspace.c:87-174).
//
// Half-space integer vectors |n| <= kc (kspace.c:35-58), a_k =
// (4 pi / V) exp(-k^2 / 4 eta^2) / k^2 (kspace.c:96-103), structure factors
// S_k = sum q sin(k.r), C_k = sum q cos(k.r) (kspace.c:147-155), then
// phi_i += sum 2 a_k (S s_i + C c_i) and E_i += sum 2 a_k (C s_i - S c_i) k
// (kspace.c:156-173).  Wave vectors come in rows: all nz of one (nx, ny), and
// k.r = (nx b1 + ny b2).r + nz b3.r, so a row's sines and cosines follow from
// those of its (nx, ny) part and of nz b3.r by the addition theorems.
// Everything is FP64.  What bounds both kernels is latency at the sizes plain
// Ewald is used for (hundreds to a few thousand sites): a sincos is about 100
// FP64 instructions, so each kernel keeps the number of them per thread small
// and spreads rows and sites over the chip.
//   k_ks_sf     one block per row (and per eight |nz| of it), one thread per
//               site: two sincos per site and row, then a rotation per |nz|;
//               648 sites, 709 wave vectors: 6.4 us (5.3 with a sincos per site
//               and wave vector), 3 120 sites: 10.2 (12.2), 12 288: 27 (34),
//               41 472: 79 (115), 65 856: 123 (177); its 80 or so blocks leave
//               most CUs idle there, and are still faster than 709 that each walk the sites
//   k_ks_field  a block serves 16 sites and its 64 16-lane teams take a row
//               each; the sites' e^{i n b.r} for every n are formed once, in
//               LDS, and so are the wave vectors' coefficients; 6.5 us for 648
//               and for 2 920 sites (8.7 and 8.2 with the coefficients read from
//               memory in the loop, 38 with 16 waves that walk the wave vectors
//               with a sincos each, 64 sites a block), 48 for 41 472 (107)
// The k-sum energy and virial
// (W_ab = sum a_k |rho_k|^2 (delta_ab - 2 k_a k_b (1/k^2 + 1/(4 eta^2))))
// are formed by a block of its own beside the field kernel's.
#include "engine.hpp"
#include "nlist.hpp"

namespace mmamd {

// A row of the half space: (first wave vector, nx, ny, m): nz = -m .. m, or
// 1 .. m for nx = ny = 0.
struct KRow {
  int k0, nx, ny, m;
  bool half;
  __device__ __forceinline__ explicit KRow(int4 v)
      : k0(v.x), nx(v.y), ny(v.z), m(v.w), half(v.y == 0 && v.z == 0) {}
  __device__ __forceinline__ int at(int nz) const { return k0 + nz + (half ? -1 : m); }
};

constexpr int KS_NZ = 8;       // |nz| values a structure-factor block serves
constexpr int SF_TB = 512;

__global__ void __launch_bounds__(SF_TB) k_ks_sf(const SysParams *__restrict__ sp,
                                               const int4 *__restrict__ krow,
                                               const double *__restrict__ r, const double *__restrict__ q,
                                               int N, double *__restrict__ ksc, NlArgs nl, int nlb) {
  before_pairs();
  const int s = blockIdx.y;
  const SysParams &P = sp[s];
  if ((int)blockIdx.x < nlb) {
    extern __shared__ int cnt[];
    if (blockIdx.z == 0) nl.bin<SF_TB>(P, s, cnt);
    return;
  }
  const int rw = blockIdx.x - nlb;
  if (P.kmode != 0 || rw >= P.nkrow) return;
  const KRow row(krow[P.krow0 + rw]);
  const int z0 = blockIdx.z * KS_NZ;
  if (z0 > row.m) return;
  const double *B = P.RL;
  const double b0 = row.nx * B[0] + row.ny * B[3], b1 = row.nx * B[1] + row.ny * B[4],
               b2 = row.nx * B[2] + row.ny * B[5];
  // per |nz|: sums of q times cos cos, sin sin, sin cos, cos sin of the
  // (nx, ny) and nz parts
  double a[4 * KS_NZ];
#pragma unroll
  for (int c = 0; c < 4 * KS_NZ; c++) a[c] = 0;
  for (int i = threadIdx.x; i < P.nsite; i += SF_TB) {
    const int si = P.site0 + i;
    const double x = r[si], y = r[N + si], z = r[2 * N + si], qi = q[si];
    double xs, xc, s1, c1, sz = 0, cz = 1;
    sincos(b0 * x + b1 * y + b2 * z, &xs, &xc);
    const double tz = B[6] * x + B[7] * y + B[8] * z;
    sincos(tz, &s1, &c1);
    if (z0) sincos(z0 * tz, &sz, &cz);
    xs *= qi;
    xc *= qi;
#pragma unroll
    for (int j = 0; j < KS_NZ; j++) {
      if (z0 + j > row.m) break;
      a[4 * j] += xc * cz;
      a[4 * j + 1] += xs * sz;
      a[4 * j + 2] += xs * cz;
      a[4 * j + 3] += xc * sz;
      const double t = cz * c1 - sz * s1;
      sz = sz * c1 + cz * s1;
      cz = t;
    }
  }
  // the wave's 32 sums over 64 lanes: at each step a lane hands half of its
  // values to its partner and keeps the other half (31 exchanges instead of
  // the 192 of a reduction value by value, which took longer than the sums)
  __shared__ double red[SF_TB / 64][4 * KS_NZ];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 2 * KS_NZ; h >= 1; h >>= 1) {
    const bool up = lane & (2 * h);
#pragma unroll
    for (int c = 0; c < h; c++) {
      const double mine = up ? a[c + h] : a[c], other = up ? a[c] : a[c + h];
      a[c] = mine + __shfl_xor(other, 2 * h);
    }
  }
  a[0] += __shfl_xor(a[0], 1);
  if (!(lane & 1)) red[w][lane >> 1] = a[0];
  __syncthreads();
  const int j = threadIdx.x, nz = z0 + j;
  if (j >= KS_NZ || nz > row.m) return;
  double t[4];
  for (int c = 0; c < 4; c++) {
    t[c] = 0;
    for (int k = 0; k < SF_TB / 64; k++) t[c] += red[k][4 * j + c];
  }
  if (!(row.half && nz == 0)) {
    double *o = ksc + 2L * (P.k0 + row.at(nz));
    o[0] = t[2] + t[3];
    o[1] = t[0] - t[1];
  }
  if (!row.half && nz > 0) {
    double *o = ksc + 2L * (P.k0 + row.at(-nz));
    o[0] = t[2] - t[3];
    o[1] = t[0] + t[1];
  }
}

constexpr int KS_SITES = 16, KS_SPLIT = 64, KS_TB = KS_SITES * KS_SPLIT;
constexpr int KS_MAXTAB = 31;   // largest |n| whose table fits beside the partial sums
// wave vectors whose coefficients 2 a_k (S, C) a block keeps in LDS: read from
// memory inside the loop over nz, each cost its trip there one after the other
constexpr int KS_STAGE = 1536;

// Each team of 16 lanes (one per site) takes rows team, team + KS_SPLIT, ...;
// the teams' sums are added in team order (deterministic).  TABLE false: wave
// vectors beyond KS_MAXTAB, whose factors are formed where they are used.
// LIST: the first nlb blocks of a system carry a neighbour-list build's pair
// search (16 wavefronts each); without it the kernel needs 69 registers
// instead of 124, which leaves room on a CU for the pair kernel beside it.
template <bool TABLE, bool LIST>
__global__ void __launch_bounds__(KS_TB) k_ks_field(const SysParams *__restrict__ sp,
                                                    const double4 *__restrict__ kvec,
                                                    const int4 *__restrict__ krow,
                                                    const double *__restrict__ ksc,
                                                    const double *__restrict__ r, int N,
                                                    double *__restrict__ kres,
                                                    double *__restrict__ acc, int want_virial,
                                                    NlArgs nl, int nlb) {
  before_pairs();
  extern __shared__ double2 tab[];   // [axis][n][site]: (cos, sin)
  __shared__ double part[KS_SPLIT][4 * KS_SITES];
  const int s = blockIdx.y;
  const SysParams &P = sp[s];
  if (LIST && (int)blockIdx.x < nlb) {
    nl.pairs<KS_TB / 64>(P, s, blockIdx.x, nlb, (int *)tab);
    return;
  }
  const int blk = blockIdx.x - nlb;
  if (P.kmode != 0) return;
  const int nblk = (P.nsite + KS_SITES - 1) / KS_SITES;
  if (blk > nblk) return;
  if (blk == nblk) {
    if (!acc) return;
    // k-sum energy and virial of this system
    double e = 0, w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const double c4 = 0.25 / (P.eta * P.eta);
    for (int k = threadIdx.x; k < P.nk; k += KS_TB) {
      const double4 kv = kvec[P.k0 + k];
      const double S = ksc[2 * (P.k0 + k)], C = ksc[2 * (P.k0 + k) + 1];
      const double ek = kv.w * (S * S + C * C);
      e += ek;
      if (want_virial) {
        const double k2 = kv.x * kv.x + kv.y * kv.y + kv.z * kv.z;
        const double f = 2 * (1 / k2 + c4);
        const double kk[3] = {kv.x, kv.y, kv.z};
        for (int a = 0; a < 3; a++)
          for (int b = 0; b < 3; b++) w[3 * a + b] += ek * ((a == b ? 1.0 : 0.0) - f * kk[a] * kk[b]);
      }
    }
    for (int o = 32; o >= 1; o >>= 1) {
      e += __shfl_xor(e, o);
      if (want_virial)
        for (int c = 0; c < 9; c++) w[c] += __shfl_xor(w[c], o);
    }
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      part[wid][0] = e;
      for (int c = 0; c < 9; c++) part[wid][1 + c] = w[c];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double t[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      for (int ww = 0; ww < KS_TB / 64; ww++)
        for (int c = 0; c < 10; c++) t[c] += part[ww][c];
      acc[s * NACC + ACC_KSPACE_E] = t[0];
      // reciprocal virial kept beside the per-site results; finish adds it
      for (int c = 0; c < 9; c++) kres[(long)4 * N + 9 * s + c] = want_virial ? t[1 + c] : 0.0;
    }
    return;
  }
  const int site = threadIdx.x & (KS_SITES - 1), team = threadIdx.x / KS_SITES;
  const int i = blk * KS_SITES + site;
  const int si = P.site0 + (i < P.nsite ? i : 0);
  const double *B = P.RL;
  double th[3];
  {
    const double x = r[si], y = r[N + si], z = r[2 * N + si];
#pragma unroll
    for (int a = 0; a < 3; a++) th[a] = B[3 * a] * x + B[3 * a + 1] * y + B[3 * a + 2] * z;
  }
  const int nm = P.nkmax;
  double2 *coef = tab + (TABLE ? 3 * (nm + 1) * KS_SITES : 0);
  const bool staged = P.nk <= KS_STAGE;
  auto form = [&](int k) {
    const double a = 2 * kvec[P.k0 + k].w;
    return make_double2(a * ksc[2 * (P.k0 + k)], a * ksc[2 * (P.k0 + k) + 1]);
  };
  if (staged)
    for (int k = threadIdx.x; k < P.nk; k += KS_TB) coef[k] = form(k);
  if (TABLE) {
    for (int t = team; t < 3 * (nm + 1); t += KS_SPLIT) {
      const int a = t / (nm + 1), n = t - a * (nm + 1);
      double sn, cs;
      sincos(n * (a == 0 ? th[0] : a == 1 ? th[1] : th[2]), &sn, &cs);
      tab[t * KS_SITES + site] = make_double2(cs, sn);
    }
  }
  if (TABLE || staged) __syncthreads();
  auto factor = [&](int a, int n) {
    if (TABLE) return tab[(a * (nm + 1) + n) * KS_SITES + site];
    double2 f;
    sincos(n * th[a], &f.y, &f.x);
    return f;
  };
  double p = 0, g1 = 0, g2 = 0, g3 = 0;   // phi; field components along b1, b2, b3
  for (int rw = team; rw < P.nkrow; rw += KS_SPLIT) {
    const KRow row(krow[P.krow0 + rw]);
    const double2 ex = factor(0, row.nx);
    double2 ey = factor(1, row.ny < 0 ? -row.ny : row.ny);
    if (row.ny < 0) ey.y = -ey.y;
    const double xc = ex.x * ey.x - ex.y * ey.y, xs = ex.x * ey.y + ex.y * ey.x;
    double t0 = 0;
    const int first = row.half ? 1 : 0;
    for (int nz = first; nz <= row.m; nz++) {
      const double2 ez = factor(2, nz);
      const double cc = xc * ez.x, ss = xs * ez.y, sc = xs * ez.x, cs = xc * ez.y;
      const int kp = row.at(nz);
      const double2 ap = staged ? coef[kp] : form(kp);
      const double snp = sc + cs, csp = cc - ss;
      double t = ap.y * snp - ap.x * csp;
      p += ap.x * snp + ap.y * csp;
      t0 += t;
      g3 += nz * t;
      if (!row.half && nz > 0) {
        const int km = row.at(-nz);
        const double2 am = staged ? coef[km] : form(km);
        const double snm = sc - cs, csm = cc + ss;
        t = am.y * snm - am.x * csm;
        p += am.x * snm + am.y * csm;
        t0 += t;
        g3 -= nz * t;
      }
    }
    g1 += row.nx * t0;
    g2 += row.ny * t0;
  }
  double *o = &part[team][site];
  o[0] = p;
  o[KS_SITES] = g1 * B[0] + g2 * B[3] + g3 * B[6];
  o[2 * KS_SITES] = g1 * B[1] + g2 * B[4] + g3 * B[7];
  o[3 * KS_SITES] = g1 * B[2] + g2 * B[5] + g3 * B[8];
  __syncthreads();
  // sixteen waves add four teams each, then one wave the sixteen sums
  const int at = threadIdx.x & 63, w = threadIdx.x >> 6;
  const double t = part[4 * w][at] + part[4 * w + 1][at] + part[4 * w + 2][at] + part[4 * w + 3][at];
  __syncthreads();
  part[w][at] = t;
  __syncthreads();
  if (w == 0) {
    double u = 0;
#pragma unroll
    for (int k = 0; k < KS_TB / 64; k++) u += part[k][at];
    const int c = at / KS_SITES, j = blk * KS_SITES + (at & (KS_SITES - 1));
    if (j < P.nsite) kres[4L * (P.site0 + j) + c] = u;
  }
}

// f(first wave vector, nx, ny, largest |nz|) for the rows of |n| <= kc
// (kspace.c:35-58), in the lexicographic order of the wave vectors; returns
// the number of wave vectors
template <class F> static int each_row(double kc, F f) {
  const double nsqmax = kc * kc + 1e-8;
  const int nm = (int)floor(kc);
  int nk = 0;
  for (int nx = 0; nx <= nm; nx++)
    for (int ny = (nx == 0) ? 0 : -nm; ny <= nm; ny++) {
      int m = -1;
      while (m < nm && nx * nx + ny * ny + (m + 1) * (m + 1) <= nsqmax) m++;
      const bool half = nx == 0 && ny == 0;
      if (m < (half ? 1 : 0)) continue;
      f(nk, nx, ny, m);
      nk += half ? m : 2 * m + 1;
    }
  return nk;
}

int kspace_rows(double kc, std::vector<int4> &rows) {
  return each_row(kc, [&](int k0, int nx, int ny, int m) { rows.push_back(make_int4(k0, nx, ny, m)); });
}

int kspace_count(double kc, int &nrow) {
  nrow = 0;
  return each_row(kc, [&](int, int, int, int) { nrow++; });
}

// a neighbour-list build that goes along: nl null without one
struct WithList {
  const NlArgs *nl = nullptr;
  int maxg = 0, maxc = 0;
};

static void launch_sf(dim3 rows_sys, int nm, hipStream_t st, const SysParams *sp,
                      const int4 *krow, const double *r, const double *q, int N, double *ksc,
                      const WithList &l = {}) {
  const int nlb = l.nl ? 1 : 0;
  rows_sys.x += nlb;
  rows_sys.z = nm / KS_NZ + 1;
  hipLaunchKernelGGL(k_ks_sf, rows_sys, dim3(SF_TB), sizeof(int) * l.maxc, st, sp, krow, r, q, N,
                     ksc, l.nl ? *l.nl : NlArgs{}, nlb);
}

static int staged_nk(int nk) { return nk <= KS_STAGE ? nk : 0; }

// acc null: energy and virial are not formed; nk: wave vectors to stage
static void launch_field(int nsite, int nsys, int nm, int nk, hipStream_t st, const SysParams *sp,
                         const double4 *kvec, const int4 *krow, const double *ksc,
                         const double *r, int N, double *kres, double *acc, int want_virial,
                         const WithList &l = {}) {
  constexpr int NW = KS_TB / 64;
  const int nlb = (l.maxg + NW - 1) / NW;
  const dim3 grid((nsite + KS_SITES - 1) / KS_SITES + (acc ? 1 : 0) + nlb, nsys);
  const NlArgs a = l.nl ? *l.nl : NlArgs{};
  const size_t list = nlb ? sizeof(int) * NL_LDS * NW : 0;
  const bool tab = nm <= KS_MAXTAB;
  const size_t lds = std::max(list, sizeof(double2) * ((tab ? 3 * (nm + 1) * KS_SITES : 0) + nk));
#define FIELD(T, L)                                                                             \
  hipLaunchKernelGGL((k_ks_field<T, L>), grid, dim3(KS_TB), lds, st, sp, kvec,                  \
                     krow, ksc, r, N, kres, acc, want_virial, a, nlb)
  if (tab && nlb) FIELD(true, true);
  else if (tab) FIELD(true, false);
  else if (nlb) FIELD(false, true);
  else FIELD(false, false);
#undef FIELD
}

static int launch_ewald(Engine &e, int want_virial, hipStream_t st, int energies, const WithList &l) {
  int maxrow = 0, maxn = 0, nm = 0, nk = 0;   // nk: the most that a block stages
  for (auto &p : e.hsp)
    if (p.kmode == 0) {
      maxrow = std::max(maxrow, p.nkrow);
      maxn = std::max(maxn, p.nsite);
      nm = std::max(nm, p.nkmax);
      nk = std::max(nk, staged_nk(p.nk));
    }
  if (maxrow == 0) return 0;
  launch_sf(dim3(maxrow, e.nsys), nm, st, e.d_sp, e.d_krow, e.d_r, e.d_q, e.nsite, e.d_ksc, l);
  launch_field(maxn, e.nsys, nm, nk, st, e.d_sp, (const double4 *)e.d_kvec, e.d_krow, e.d_ksc, e.d_r,
               e.nsite, e.d_kres, energies ? e.d_acc : nullptr, want_virial, l);
  MM_HIP(hipGetLastError());
  return 0;
}

int launch_kspace(Engine &e, int want_virial, hipStream_t st, int energies) {
  return launch_ewald(e, want_virial, st, energies, {});
}

// Small plain-Ewald engines: the two launches of a neighbour-list build, which
// in most steps find nothing to do, ride in those of the reciprocal sum, and
// everything stays on one stream.  A launch of its own costs 3 us whatever it
// does, a fork to the second stream and back 10.  A step of 216 waters took
// 36.3 us forked, 36.3 in a line and 30.5 like this, 960 waters with ions
// 44.9, 46.9 and 42.4 (28.4 and 40.0 with the field's coefficients in LDS).
// Beyond PAIR_WIDE_GROUPS the pair kernel fills the chip and the sums beside
// it are the longer part, so the fork pays.
bool kspace_takes_list(const Engine &e) {
  bool ewald = false;
  for (auto &p : e.hsp) {
    if (p.kmode == 1 || p.ncell * p.ncell * p.ncell > NL_BIN_CELLS) return false;
    ewald |= p.kmode == 0 && p.nkrow > 0;
  }
  return ewald && e.pair_lanes == 64;
}

int launch_kspace_list(Engine &e, int want_virial, int energies, int force, int from_partials) {
  NlArgs a;
  WithList l;
  if (int rc = nl_prepare(e, force, from_partials, a, l.maxc)) return rc;
  l.nl = &a;
  l.maxg = e.maxg;
  return launch_ewald(e, want_virial, e.stream, energies, l);
}

// Structure factors and field of one system whose parameters, wave vectors,
// rows (nkrow of them, |n| up to nm), SoA positions and result buffers the
// caller provides (kspace_field_noalloc keeps them in its own device array):
// ksc 2 nk, kres 4 nsite.
int launch_kspace_raw(const SysParams *sp, const double4 *kvec, const int4 *krow, int nkrow,
                      int nm, int nk, int nsite, const double *r, const double *q, double *ksc,
                      double *kres, hipStream_t st) {
  launch_sf(dim3(nkrow, 1), nm, st, sp, krow, r, q, nsite, ksc);
  launch_field(nsite, 1, nm, staged_nk(nk), st, sp, kvec, krow, ksc, r, nsite, kres, nullptr, 0);
  MM_HIP(hipGetLastError());
  return 0;
}

// the field kernel of one system with other structure factors and outputs
// (the adjoint pass): kres_out needs 4 N entries
int launch_kspace_field_only(Engine &e, int sys, const double *ksc, double *kres_out) {
  const SysParams &P = e.hsp[sys];
  if (P.kmode != 0) return 0;
  launch_field(P.nsite, 1, P.nkmax, staged_nk(P.nk), e.stream, e.d_sp + sys, (const double4 *)e.d_kvec, e.d_krow,
               ksc, e.d_r, e.nsite, kres_out, nullptr, 0);
  MM_HIP(hipGetLastError());
  return 0;
}

}  // namespace mmamd
