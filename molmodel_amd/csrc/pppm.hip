// pppm.hip -- P3M on the device (pppm.c:498-641).
//
// Steps, each its own kernel on one stream:
//   bin      s = diag(n) L^-1 r in FP64, nearest/lower mesh point and the
//            fractional offset as the reference forms them (pppm.c:523-548),
//            and a copy of each site in the slots of the mesh column-block
//            bin that holds its base point (a per-block LDS rank per bin and
//            one global claim of slots per bin the block touches);
//   spread   one workgroup per column block (bx x by columns), as 64-bit
//            fixed point in LDS (exact, so independent of the order of the
//            atomics), no global atomics, one of two ways (a shape choice):
//            pulling -- the block takes the sites of its own and the
//            neighbouring bins and accumulates q w_x w_y w_z into the
//            points it owns, then writes them once; or by owner -- the
//            block takes only its own bin's sites, accumulates their whole
//            stencils into a halo of (bx + P - 1) x (by + P - 1) columns
//            and writes the halo to its own slice, which the z pass sums;
//            pulling re-reads every site for each block its stencil
//            reaches, the halos cost their traffic, so columns holding many
//            sites favour pulling and few sites the halos;
//   fft      in-place mixed-radix line FFTs in LDS (fft.hpp): z (real to half
//            spectrum; by the pulling blocks themselves where their columns
//            come in pairs), then per kz plane y and x forward, the influence
//            function (and the mesh energy/virial), x and y inverse, then z
//            (half spectrum to real), unnormalised like FFTW;
//   gather   phi_i = sum w phi_m and, with real-space differentiation (the
//            reference default), E_i = (diag(n) L^-1)^T (sum -dw phi_m)
//            (pppm.c:603-640); with the field formed on the mesh (ik), the
//            planes also form E_a = -i k_a phi_k, the inverse z pass runs
//            over four components and E_i = sum w E_m (pppm.c:577-626).
// Assignment weights are the cardinal B-splines that the reference's
// polynomial tables tabulate (pppm.c:69-275), evaluated by recursion in FP32.
#include "engine.hpp"
#include "reduce.hpp"
#include "fft.hpp"
#include <cmath>
#include <cstring>

namespace mmamd {

constexpr float FIX_SCALE = 4294967296.0f;   // 2^32
constexpr double FIX_INV = 1.0 / 4294967296.0;
// A contribution in fixed point, to the nearest even: adding 1.5 2^20 to the
// FP64 value leaves it in units of 2^-32 in the low bits (three instructions;
// the conversion of a scaled float to 64 bits takes about ten).  Exact for
// contributions below 2^19: sites with larger charges take the conversion.
constexpr double FIX_MAGIC = 1572864.0;
constexpr float FIX_MAXQ = 262144.f;
template <bool WIDE = false>
__device__ __forceinline__ unsigned long long to_fix(float x) {
  if (WIDE) return (unsigned long long)__float2ll_rn(x * FIX_SCALE);
  return (unsigned long long)(__double_as_longlong((double)x + FIX_MAGIC) -
                              __double_as_longlong(FIX_MAGIC));
}

template <int P>
__device__ __forceinline__ void bspline_w(float s, float *w, float *ndw) {
  // w[k] = M_P(u + P - 1 - k), u = s + 1/2; ndw[k] = -dw/ds (cardinal
  // B-spline recursion, all loops unrolled for the compile-time order)
  const float u = s + 0.5f;
  float m[P + 1];
#pragma unroll
  for (int k = 0; k <= P; k++) m[k] = 0.f;
  m[0] = 1.f;
#pragma unroll
  for (int p = 2; p <= P; p++) {
    if (p == P && ndw) {
#pragma unroll
      for (int k = 0; k < P; k++) {
        const float a = k < p - 1 ? m[k] : 0.f;
        const float b = k >= 1 ? m[k - 1] : 0.f;
        ndw[P - 1 - k] = b - a;
      }
    }
    constexpr float dummy = 0.f;
    (void)dummy;
    const float inv = 1.f / (float)(p - 1);
#pragma unroll
    for (int k = p - 1; k >= 0; k--) {
      const float x = u + (float)k;
      const float a = k < p - 1 ? m[k] : 0.f;
      const float b = k >= 1 ? m[k - 1] : 0.f;
      m[k] = (x * a + ((float)p - x) * b) * inv;
    }
  }
  if (P == 1 && ndw) ndw[0] = 0.f;
#pragma unroll
  for (int k = 0; k < P; k++) w[P - 1 - k] = m[k];
}

// wrap j + off into [0, n) for |off| < n (no integer division)
__device__ __forceinline__ int wrap(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

// Grid coordinates of each site (pppm.c:540-557) and its copy in the slots
// of its mesh column bin (bx x by columns).  A block ranks its sites per bin
// in LDS and claims each bin's slots with one global atomic; the order
// inside a bin varies from run to run, and the spreading's 64-bit
// fixed-point sums do not depend on it.  The gather clears the counters.
// A site beyond a bin's capacity raises ERR_BIN_OVERFLOW and records in
// *need the slot count that bin would have needed, so the host can grow the
// bins and evaluate again.
constexpr int MAXBINS = 4096;
__global__ void __launch_bounds__(256) k_p3m_bin(const SysParams *__restrict__ sp,
                                                 const double *__restrict__ r,
                                                 const double *__restrict__ q, int N,
                                                 int4 *__restrict__ sgrid,
                                                 float4 *__restrict__ sfrac,
                                                 int *__restrict__ fill, int bcap,
                                                 int4 *__restrict__ bgrid,
                                                 float4 *__restrict__ bfrac,
                                                 int *__restrict__ err, int *__restrict__ need) {
  before_pairs();
  __shared__ int cnt[MAXBINS];
  const int s = blockIdx.y;
  const SysParams &P = sp[s];
  if (P.kmode != 1) return;
  if ((int)(blockIdx.x * blockDim.x) >= P.nsite) return;
  const int nb = P.nbx * P.nby;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) cnt[t] = 0;
  __syncthreads();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool on = i < P.nsite;
  const int si = P.site0 + (on ? i : 0);
  const double x = r[si], y = r[N + si], z = r[2 * N + si];
  const double *T = P.T;
  double sx = T[0] * x + T[3] * y + T[6] * z;
  double sy = T[1] * x + T[4] * y + T[7] * z;
  double sz = T[2] * x + T[5] * y + T[8] * z;
  int jx, jy, jz;
  if (P.order & 1) {
    jx = (int)floor(sx + 0.5); jy = (int)floor(sy + 0.5); jz = (int)floor(sz + 0.5);
    sx -= jx; sy -= jy; sz -= jz;
  } else {
    jx = (int)floor(sx); jy = (int)floor(sy); jz = (int)floor(sz);
    sx -= jx + 0.5; sy -= jy + 0.5; sz -= jz + 0.5;
  }
  jx = mod_nonneg(jx, P.nx); jy = mod_nonneg(jy, P.ny); jz = mod_nonneg(jz, P.nz);
  const int lb = (jx / P.bx) * P.nby + jy / P.by;
  const int b = P.bin0 + lb;
  const float4 f = make_float4((float)sx, (float)sy, (float)sz, (float)q[si]);
  int rank = 0;
  if (on) {
    sgrid[si] = make_int4(jx, jy, jz, b);
    sfrac[si] = f;
    rank = atomicAdd(&cnt[lb], 1);
  }
  __syncthreads();
  // one claim per bin this block touches; the base replaces the count
  for (int t = threadIdx.x; t < nb; t += blockDim.x)
    if (cnt[t]) cnt[t] = atomicAdd(&fill[P.bin0 + t], cnt[t]);
  __syncthreads();
  if (!on) return;
  const int slot = cnt[lb] + rank;
  if (slot < bcap) {
    bgrid[(long)b * bcap + slot] = make_int4(jx, jy, jz, si);
    bfrac[(long)b * bcap + slot] = f;
  } else {
    atomicOr(err, ERR_BIN_OVERFLOW);   // reported; the site is left out of the mesh
    atomicMax(need, slot + 1);
  }
}

__device__ __forceinline__ int floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// The sites whose stencils reach a spreading block's columns: the bins of the
// neighbouring column blocks (at most 8 per axis for P <= 7), flattened into
// one list so that all threads work whatever the bins' sizes: thread t < nbin
// takes bin t, wave 0 scans the counts.
struct ReachedSites {
  int start[64], off[65], nbin;

  template <int P>
  __device__ __forceinline__ void collect(const SysParams &Q, int X0, int Y0,
                                          const int *__restrict__ fill, int bcap) {
    constexpr int istart = -((P + 1) / 2 - 1);
    const int bx = Q.bx, by = Q.by;
    int xlo = floor_div(X0 - istart - P + 1, bx), xhi = floor_div(X0 + bx - 1 - istart, bx);
    int ylo = floor_div(Y0 - istart - P + 1, by), yhi = floor_div(Y0 + by - 1 - istart, by);
    if (xhi - xlo + 1 >= Q.nbx) { xlo = 0; xhi = Q.nbx - 1; }
    if (yhi - ylo + 1 >= Q.nby) { ylo = 0; yhi = Q.nby - 1; }
    const int ncy = yhi - ylo + 1, n = (xhi - xlo + 1) * ncy;   // <= 64
    if (threadIdx.x < 64) {
      int cnt = 0;
      const int t = threadIdx.x;
      if (t < n) {
        const int ccx = mod_nonneg(xlo + t / ncy, Q.nbx), ccy = mod_nonneg(ylo + t % ncy, Q.nby);
        const int b = Q.bin0 + ccx * Q.nby + ccy;
        start[t] = b * bcap;
        cnt = min(fill[b], bcap);
      }
      int incl = cnt;   // inclusive scan over the wave
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o);
        if (t >= o) incl += y;
      }
      off[t + 1] = incl;
      if (t == 0) { off[0] = 0; nbin = n; }
    }
    __syncthreads();
  }
  __device__ __forceinline__ int total() const { return off[nbin]; }
  // where site u of the list is kept
  __device__ __forceinline__ int slot(int u) const {
    int lo = 0, hi = nbin - 1;   // last bin with off[bin] <= u
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (off[mid] <= u) lo = mid; else hi = mid - 1;
    }
    return start[lo] + (u - off[lo]);
  }
};

constexpr int FFT_MAXN = 128;
// an axis' factors exp(-2 pi i t / n), and (pos) each frequency's place and
// each place's signed frequency, from the system's tables (p3m_twiddles)
__device__ __forceinline__ void load_tw(float2 *stw, const float2 *tw, int n) {
  for (int t = threadIdx.x; t < n; t += blockDim.x) stw[t] = tw[t];
}
__device__ __forceinline__ void load_pos(int *pos, const float2 *tw, int n) {
  for (int t = threadIdx.x; t < n; t += blockDim.x) pos[t] = __float_as_int(tw[3 * FFT_MAXN + t].x);
}
__device__ __forceinline__ void load_freq(short *f, const float2 *tw, int n) {
  for (int t = threadIdx.x; t < n; t += blockDim.x)
    f[t] = (short)__float_as_int(tw[3 * FFT_MAXN + t].y);
}

// half spectrum of two real lines a + i b from their transform at k and -k
__device__ __forceinline__ float2 half_a(float2 zp, float2 zm) {
  return make_float2(0.5f * (zp.x + zm.x), 0.5f * (zp.y - zm.y));
}
__device__ __forceinline__ float2 half_b(float2 zp, float2 zm) {
  return make_float2(0.5f * (zp.y + zm.y), 0.5f * (zm.x - zp.x));
}

// A pulling block holds whole z lines, so it transforms them itself, where its
// columns come in the pairs that k_fft_z makes one complex line of: an even
// number of y columns a block and on the mesh.  (The bound keeps the LDS of a
// block at 24 KB.)  One launch and a trip of the mesh through memory less, the
// writes in runs of two columns: spreading and z pass of 12 288 sites on 48^3
// took 7.0 and 5.7 us and take 9.5 together, of 98 304 on 64^3 17.2 and 7.0, now 20.3.
constexpr int FUSE_POINTS = 2048;
__host__ __device__ __forceinline__ bool spread_transforms(const SysParams &Q) {
  return !(Q.by & 1) && !(Q.ny & 1) && Q.bx * Q.by * Q.nz <= FUSE_POINTS;
}
__device__ __forceinline__ void transform_columns(const SysParams &Q, const unsigned long long *acc,
                                                  float2 *buf, const float2 *stw, const int *pos,
                                                  int X0, int Y0, float2 *__restrict__ cmesh) {
  const int nz = Q.nz, nzh = nz / 2 + 1, ls = nz | 1, nl = Q.bx * Q.by / 2, half = Q.by / 2;
  float *fb = reinterpret_cast<float *>(buf);
  const float inv = 1.f / (float)nz, inv_nl = 1.f / (float)nl, inv_half = 1.f / (float)half;
  for (int t = threadIdx.x; t < 2 * nl * nz; t += blockDim.x) {
    const int c = div_small(t, inv), z = t - c * nz;
    fb[2 * ((c >> 1) * ls + z) + (c & 1)] = (float)((double)(long long)acc[t] * FIX_INV);
  }
  __syncthreads();
  fft_forward(buf, nl, ls, 1, nz, Q.rad[2], stw);
  float2 *dst = cmesh + Q.cmesh0 + (long)X0 * Q.ny + Y0;
  const long plane = (long)Q.nx * Q.ny;
  for (int t = threadIdx.x; t < nzh * nl; t += blockDim.x) {
    const int k = div_small(t, inv_nl), l = t - k * nl;
    const int ox = div_small(l, inv_half), oy = 2 * (l - ox * half);
    const float2 zp = buf[l * ls + pos[k]], zm = buf[l * ls + pos[k ? nz - k : 0]];
    float2 *o = dst + k * plane + ox * Q.ny + oy;
    o[0] = half_a(zp, zm);
    o[1] = half_b(zp, zm);
  }
}

// the block's points out to the mesh
__device__ __forceinline__ void store_columns(const SysParams &Q, const unsigned long long *acc,
                                              int X0, int Y0, float *__restrict__ mesh) {
  const int nz = Q.nz, by = Q.by;
  for (int t = threadIdx.x; t < Q.bx * by * nz; t += blockDim.x) {
    const int gz = t % nz, gy = (t / nz) % by, gx = t / (nz * by);
    mesh[Q.mesh0 + ((long)(X0 + gx) * Q.ny + (Y0 + gy)) * nz + gz] =
        (float)((double)(long long)acc[t] * FIX_INV);
  }
}

// Spreading by pulling.  One site per thread, which runs over the block's own
// columns and takes the weights that its stencil has there, if any (with 2 x
// 2 columns a reached site has on average 2.8 of the four; running over the
// 25 columns of its stencil and testing each took 1 250 instructions a site).
// What bounds it is instruction issue (72% of the cycles at 98 304 sites on
// 64^3): every site is weighted again for each block that it reaches.  17.2
// us there (24.2 before), 7.0 for 12 288 on 48^3 (11.1).
//
// stencil offset of the column k past the one at offset a (n columns round)
__device__ __forceinline__ unsigned column_offset(unsigned a, unsigned k, unsigned n) {
  const unsigned v = a + k, w = v - n;   // w is huge unless v >= n
  return v < w ? v : w;
}

// swx, swy: this thread's columns of the block's staged weights, 256 apart
template <int P, bool WIDE>
__device__ __forceinline__ void spread_site(const SysParams &Q, int X0, int Y0, const int4 &g,
                                            const float4 &f, float *swx, float *swy,
                                            unsigned long long *acc) {
  constexpr int istart = -((P + 1) / 2 - 1);
  const int nz = Q.nz, bx = Q.bx, by = Q.by;
  float wx[P], wy[P], wz[P];
  bspline_w<P>(f.x, wx, nullptr);
  bspline_w<P>(f.y, wy, nullptr);
  bspline_w<P>(f.z, wz, nullptr);
#pragma unroll
  for (int k = 0; k < P; k++) {
    swx[256 * k] = f.w * wx[k];
    swy[256 * k] = wy[k];
  }
  int iz[P];
#pragma unroll
  for (int c = 0; c < P; c++) iz[c] = wrap(g.z + istart + c, nz);
  const unsigned a0 = wrap(X0 - g.x - istart, Q.nx), b0 = wrap(Y0 - g.y - istart, Q.ny);
  for (int ox = 0; ox < bx; ox++) {
    const unsigned a = column_offset(a0, ox, Q.nx);
    if (a >= P) continue;
    const float wa = swx[256 * a];
    unsigned long long *col = acc + ox * by * nz;
    for (int oy = 0; oy < by; oy++, col += nz) {
      const unsigned b = column_offset(b0, oy, Q.ny);
      if (b >= P) continue;
      const float w = wa * swy[256 * b];
#pragma unroll
      for (int c = 0; c < P; c++) atomicAdd(col + iz[c], to_fix<WIDE>(w * wz[c]));
    }
  }
}

template <int P>
__global__ void __launch_bounds__(256) k_p3m_spread(const SysParams *__restrict__ sp,
                                                    const int *__restrict__ fill, int bcap,
                                                    const int4 *__restrict__ bgrid,
                                                    const float4 *__restrict__ bfrac,
                                                    float *__restrict__ mesh,
                                                    const float2 *__restrict__ twid_all,
                                                    float2 *__restrict__ cmesh) {
  before_pairs();
  extern __shared__ unsigned long long acc[];
  __shared__ ReachedSites reached;
  __shared__ float swx[P * 256], swy[P * 256];   // staged so that an offset can index them
  __shared__ float2 stw[FFT_MAXN];
  __shared__ int pos[FFT_MAXN];
  const int s = blockIdx.y;
  const SysParams &Q = sp[s];
  if (Q.kmode != 1 || Q.order != P) return;
  const int blk = blockIdx.x;
  if (blk >= Q.nbx * Q.nby) return;
  const int X0 = blk / Q.nby * Q.bx, Y0 = blk % Q.nby * Q.by;
  const int npts = Q.bx * Q.by * Q.nz;
  for (int t = threadIdx.x; t < npts; t += blockDim.x) acc[t] = 0ull;
  const bool z = spread_transforms(Q);
  if (z) {
    load_tw(stw, twid_all + Q.twid0 + 2 * FFT_MAXN, Q.nz);
    load_pos(pos, twid_all + Q.twid0 + 2 * FFT_MAXN, Q.nz);
  }
  reached.collect<P>(Q, X0, Y0, fill, bcap);
  const int total = reached.total();
  // a site is loaded while the one before it is spread
  float *wx = swx + threadIdx.x, *wy = swy + threadIdx.x;
  int4 gn = make_int4(0, 0, 0, 0);
  float4 fn = make_float4(0.f, 0.f, 0.f, 0.f);
  auto load = [&](int u) {
    if (u >= total) return;
    const int t = reached.slot(u);
    gn = bgrid[t];
    fn = bfrac[t];
  };
  load(threadIdx.x);
  for (int u = threadIdx.x; u < total; u += blockDim.x) {
    const int4 g = gn;
    const float4 f = fn;
    load(u + blockDim.x);
    if (fabsf(f.w) < FIX_MAXQ) spread_site<P, false>(Q, X0, Y0, g, f, wx, wy, acc);
    else spread_site<P, true>(Q, X0, Y0, g, f, wx, wy, acc);
  }
  __syncthreads();
  if (z) transform_columns(Q, acc, reinterpret_cast<float2 *>(acc + npts), stw, pos, X0, Y0, cmesh);
  else store_columns(Q, acc, X0, Y0, mesh);
}

// The transpose of the gather's field instead of the charge: site i
// contributes src_i . (dw_x w_y w_z, w_x dw_y w_z, w_x w_y dw_z) with dw the
// negated weight derivatives the gather uses and src_i = q_i (R_i T) (the
// adjoint of E_i = T^T sum_m dw phi_m for a given R_i), so that the
// convolution and an ordinary gather of the result give
// sum_i q_i R_i . dE_i/dq_j at every site j.  The caller scales src to at
// most about one.
template <int P>
__global__ void __launch_bounds__(256) k_p3m_spread_adj(const SysParams *__restrict__ sp,
                                                        const int *__restrict__ fill, int bcap,
                                                        const int4 *__restrict__ bgrid,
                                                        const float4 *__restrict__ bfrac,
                                                        float *__restrict__ mesh,
                                                        const float4 *__restrict__ src) {
  extern __shared__ unsigned long long acc[];
  __shared__ ReachedSites reached;
  const SysParams &Q = sp[0];
  if (Q.kmode != 1 || Q.order != P) return;
  const int blk = blockIdx.x;
  if (blk >= Q.nbx * Q.nby) return;
  const int nz = Q.nz, X0 = blk / Q.nby * Q.bx, Y0 = blk % Q.nby * Q.by;
  for (int t = threadIdx.x; t < Q.bx * Q.by * nz; t += blockDim.x) acc[t] = 0ull;
  reached.collect<P>(Q, X0, Y0, fill, bcap);
  const int total = reached.total();
  constexpr int istart = -((P + 1) / 2 - 1);
  for (int u = threadIdx.x; u < total; u += blockDim.x) {
    const int t = reached.slot(u);
    const int4 g = bgrid[t];
    const float4 f = bfrac[t];
    float wx[P], wy[P], wz[P], dwx[P], dwy[P], dwz[P];
    bspline_w<P>(f.x, wx, dwx);
    bspline_w<P>(f.y, wy, dwy);
    bspline_w<P>(f.z, wz, dwz);
    int iz[P];
#pragma unroll
    for (int c = 0; c < P; c++) iz[c] = wrap(g.z + istart + c, nz);
    const float4 sv = src[g.w];
    for (int ox = 0; ox < Q.bx; ox++) {
      const int a = wrap(X0 + ox - g.x - istart, Q.nx);
      if (a >= P) continue;
      float wa = wx[0], da = dwx[0];
#pragma unroll
      for (int k = 1; k < P; k++) {
        wa = a == k ? wx[k] : wa;
        da = a == k ? dwx[k] : da;
      }
      for (int oy = 0; oy < Q.by; oy++) {
        const int b = wrap(Y0 + oy - g.y - istart, Q.ny);
        if (b >= P) continue;
        float wb = wy[0], db = dwy[0];
#pragma unroll
        for (int k = 1; k < P; k++) {
          wb = b == k ? wy[k] : wb;
          db = b == k ? dwy[k] : db;
        }
        const float al = sv.x * da * wb + sv.y * wa * db;
        const float be = sv.z * wa * wb;
        unsigned long long *col = acc + (ox * Q.by + oy) * nz;
#pragma unroll
        for (int c = 0; c < P; c++) atomicAdd(col + iz[c], to_fix(al * wz[c] + be * dwz[c]));
      }
    }
  }
  __syncthreads();
  store_columns(Q, acc, X0, Y0, mesh);
}

// Spreading by owner: the block of column block k takes only the sites
// binned to it (base point in its bx x by columns), so every site is read
// and weighted once, and accumulates all P^3 weights of each into an LDS
// halo of (bx + P - 1) x (by + P - 1) columns of nz points (halo column
// (hx, hy) is mesh column (X0 + istart + hx, Y0 + istart + hy) mod n) as
// 64-bit fixed point, exact and so independent of the order of the
// atomics.  The halo goes out whole to the block's own slice of `halo`;
// the z pass adds the halos that cover each mesh column (integer sums, so
// the mesh equals that of a single accumulator).  One work item per (site,
// z offset c): the P lanes of a site write P consecutive points of a
// column, in different LDS banks.
template <int P>
__global__ void __launch_bounds__(512) k_p3m_spread_halo(const SysParams *__restrict__ sp,
                                                         const int *__restrict__ fill, int bcap,
                                                         const int4 *__restrict__ bgrid,
                                                         const float4 *__restrict__ bfrac,
                                                         unsigned long long *__restrict__ halo) {
  before_pairs();
  extern __shared__ unsigned long long hacc[];
  const int s = blockIdx.y;
  const SysParams &Q = sp[s];
  if (Q.kmode != 1 || Q.order != P) return;
  const int blk = blockIdx.x;
  if (blk >= Q.nbx * Q.nby) return;
  const int nz = Q.nz, HX = Q.bx + P - 1, HY = Q.by + P - 1;
  const int npts = HX * HY * nz;
  for (int t = threadIdx.x; t < npts; t += blockDim.x) hacc[t] = 0ull;
  __syncthreads();
  const int X0 = (blk / Q.nby) * Q.bx, Y0 = (blk % Q.nby) * Q.by;
  const int b = Q.bin0 + blk;
  const int n = min(fill[b], bcap);
  constexpr int istart = -((P + 1) / 2 - 1);
  for (int u = threadIdx.x; u < n * P; u += blockDim.x) {
    const int site = u / P, c = u - site * P;
    const int4 g = bgrid[(long)b * bcap + site];
    const float4 f = bfrac[(long)b * bcap + site];
    float wx[P], wy[P], wz[P];
    bspline_w<P>(f.x, wx, nullptr);
    bspline_w<P>(f.y, wy, nullptr);
    bspline_w<P>(f.z, wz, nullptr);
    float wc = wz[0];
#pragma unroll
    for (int k = 1; k < P; k++)
      if (c == k) wc = wz[k];
    const int iz = wrap(g.z + istart + c, nz);
    unsigned long long *base = hacc + ((g.x - X0) * HY + (g.y - Y0)) * nz + iz;
    if (fabsf(f.w) < FIX_MAXQ) {
#pragma unroll
      for (int a = 0; a < P; a++) {
        const float qa = f.w * wx[a];
#pragma unroll
        for (int bb = 0; bb < P; bb++)
          atomicAdd(base + (a * HY + bb) * nz, to_fix(qa * wy[bb] * wc));
      }
    } else {
      for (int a = 0; a < P; a++) {
        float wa = wx[0];
#pragma unroll
        for (int k = 1; k < P; k++) wa = a == k ? wx[k] : wa;
#pragma unroll
        for (int bb = 0; bb < P; bb++)
          atomicAdd(base + (a * HY + bb) * nz, to_fix<true>(f.w * wa * wy[bb] * wc));
      }
    }
  }
  __syncthreads();
  unsigned long long *dst = halo + Q.halo0 + (long)blk * npts;
  for (int t = threadIdx.x; t < npts; t += blockDim.x) dst[t] = hacc[t];
}

// ---------------- transforms ----------------
// Half spectra are stored plane by plane, [kz][x][y], the influence function
// likewise but with x and y in the digit-reversed order the forward
// transforms leave (fft.hpp), so that its factors line up with the spectrum.
constexpr int FZ_LINES = 16;                 // complex lines per z block: 32 mesh lines
constexpr int FZ_TB = 256;
constexpr int FP_TB = 512;                   // plane block

// Mesh line `line` (column xi = line / ny, yi = line % ny) of a P3M system is
// the sum of the spreading blocks' halo columns that cover it: halo column
// (dx, dy) of block (bi, bj) is mesh column (bi bx + istart + dx,
// bj by + istart + dy) mod n, so the covering blocks have
// dx = xi - istart (mod bx), dy likewise.  The block's threads first list the
// covering columns of its lines, one (line, column) each, and then sum them,
// one point each with four loads in flight: integer sums, then the
// conversion a single accumulator would make.  (Sixteen threads per line that
// each worked out the line's columns took 35 us for 32 meshes of 30^3 and
// 36^3 at order 6, and take 15 this way)
constexpr int HALO_MAXCOV = (MAXORDER + 1) * (MAXORDER + 1);   // blocks of one column each
struct HaloLists {
  int off[2 * FZ_LINES][HALO_MAXCOV], n[2 * FZ_LINES];
};

__device__ __forceinline__ void halo_lines(const SysParams &P, const unsigned long long *__restrict__ halo,
                                           int l0, int nl, int ls, float *fb, HaloLists &L) {
  const int nz = P.nz, ny = P.ny, bxs = P.bx, bys = P.by;
  const int istart = -((P.order + 1) / 2 - 1), HX = bxs + P.order - 1, HY = bys + P.order - 1;
  const int hpts = HX * HY * nz;
  const int mx = (HX + bxs - 1) / bxs, my = (HY + bys - 1) / bys;   // most per axis
  for (int t = threadIdx.x; t < 2 * FZ_LINES * mx * my; t += FZ_TB) {
    const int l = t / (mx * my), e = t - l * mx * my, i = e / my, j = e - i * my;
    if (l >= nl) {
      if (e == 0) L.n[l] = 0;
      continue;
    }
    const int xi = (l0 + l) / ny, yi = (l0 + l) - xi * ny;
    const int dx0 = mod_nonneg(xi - istart, bxs), dy0 = mod_nonneg(yi - istart, bys);
    const int ni = (HX - dx0 + bxs - 1) / bxs, nj = (HY - dy0 + bys - 1) / bys;
    if (e == 0) L.n[l] = ni * nj;
    if (i >= ni || j >= nj) continue;
    const int dx = dx0 + i * bxs, dy = dy0 + j * bys;
    const int bi = mod_nonneg(xi - istart - dx, P.nx) / bxs, bj = mod_nonneg(yi - istart - dy, ny) / bys;
    L.off[l][i * nj + j] = (bi * P.nby + bj) * hpts + (dx * HY + dy) * nz;
  }
  __syncthreads();
  const unsigned long long *h = halo + P.halo0;
  const float inv = 1.f / (float)nz;
  for (int t = threadIdx.x; t < 2 * FZ_LINES * nz; t += FZ_TB) {
    const int l = div_small(t, inv), z = t - l * nz, n = L.n[l];
    unsigned long long sum = 0ull;
    for (int e = 0; e < n; e += 4) {
      unsigned long long v[4];
#pragma unroll
      for (int k = 0; k < 4; k++) v[k] = e + k < n ? h[L.off[l][e + k] + z] : 0ull;
      sum += (v[0] + v[1]) + (v[2] + v[3]);
    }
    fb[2 * ((l >> 1) * ls + z) + (l & 1)] = (float)((double)(long long)sum * FIX_INV);
  }
}

// z lines, real to half spectrum.  Two neighbouring mesh lines are one complex
// line (a in the real, b in the imaginary part) whose transform Z separates
// as a_k = (Z_k + conj Z_-k) / 2, b_k = (Z_k - conj Z_-k) / 2i, so a block
// takes 32 lines.  Its four waves share the loads and stores; a stage has
// 16 nz / R butterflies (96 or 128 at 48 and 64 points), at most one a thread
// where nz <= 16 R.
// HALO: a line is the sum of the spreading blocks' halo columns that cover it
// (halo_lines) instead of the real mesh.  What bounds it is the launch and one
// trip to memory: 5.7 us at 48^3, 6.7 at 64^3, and the inverse 5.9 and 7
// (5.65 and 6 with one line per transform, 16 lines a block).
template <bool HALO>
__global__ void __launch_bounds__(FZ_TB) k_fft_z(
    const SysParams *__restrict__ sp, const float2 *__restrict__ twid_all,
    const float *__restrict__ mesh, float2 *__restrict__ cmesh,
    const unsigned long long *__restrict__ halo, int spread_does) {
  before_pairs();
  __shared__ float2 buf[FZ_LINES * (FFT_MAXN + 1)], stw[FFT_MAXN];
  __shared__ int pos[FFT_MAXN];
  const SysParams &P = sp[blockIdx.y];
  if (P.kmode != 1 || (spread_does && spread_transforms(P))) return;
  const int nz = P.nz, nzh = nz / 2 + 1, ls = nz | 1;
  const int nlines = P.nx * P.ny, l0 = blockIdx.x * 2 * FZ_LINES, nl = min(2 * FZ_LINES, nlines - l0);
  if (nl <= 0) return;
  load_tw(stw, twid_all + P.twid0 + 2 * FFT_MAXN, nz);
  load_pos(pos, twid_all + P.twid0 + 2 * FFT_MAXN, nz);
  float *fb = reinterpret_cast<float *>(buf);
  if constexpr (HALO) {
    __shared__ HaloLists lists;
    halo_lines(P, halo, l0, nl, ls, fb, lists);
  } else {
    const float *src = mesh + P.mesh0 + (long)l0 * nz;
    const float inv = 1.f / (float)nz;
    batched<8>(2 * FZ_LINES * nz, [&](int t) { return t < nl * nz ? src[t] : 0.f; },
               [&](int t, float v) {
                 const int l = div_small(t, inv), z = t - l * nz;
                 fb[2 * ((l >> 1) * ls + z) + (l & 1)] = v;
               });
  }
  __syncthreads();
  fft_forward(buf, FZ_LINES, ls, 1, nz, P.rad[2], stw);
  float2 *dst = cmesh + P.cmesh0 + l0;
  for (int t = threadIdx.x; t < nzh * FZ_LINES; t += blockDim.x) {
    const int k = t / FZ_LINES, l = t % FZ_LINES;
    const float2 zp = buf[l * ls + pos[k]], zm = buf[l * ls + pos[k ? nz - k : 0]];
    float2 *o = dst + (long)k * nlines + 2 * l;
    if (2 * l < nl) o[0] = half_a(zp, zm);
    if (2 * l + 1 < nl) o[1] = half_b(zp, zm);
  }
}

// z lines, half spectrum to real, two lines in one complex line as above.
// The potential's lines are followed by their first order - 1 points again,
// so that a site's run along z is contiguous for the gather; with the field
// on the mesh (blockIdx.z: phi, Ex, Ey, Ez) the components are interleaved
// per point instead.
__global__ void __launch_bounds__(FZ_TB) k_fft_zinv(const SysParams *__restrict__ sp,
                                                    const float2 *__restrict__ twid_all,
                                                    const float2 *__restrict__ cmesh,
                                                    float *__restrict__ mesh) {
  before_pairs();
  __shared__ float2 buf[FZ_LINES * (FFT_MAXN + 1)], stw[FFT_MAXN];
  __shared__ int pos[FFT_MAXN];
  const SysParams &P = sp[blockIdx.y];
  if (P.kmode != 1) return;
  const int comp = blockIdx.z;
  if (comp > 0 && !P.ik) return;
  const int nz = P.nz, nzh = nz / 2 + 1, ls = nz | 1;
  const int nlines = P.nx * P.ny, l0 = blockIdx.x * 2 * FZ_LINES, nl = min(2 * FZ_LINES, nlines - l0);
  if (nl <= 0) return;
  load_tw(stw, twid_all + P.twid0 + 2 * FFT_MAXN, nz);
  load_pos(pos, twid_all + P.twid0 + 2 * FFT_MAXN, nz);
  __syncthreads();
  const float2 *src = cmesh + P.cmesh0 + (P.ik ? comp + 1 : 0) * (long)nlines * nzh + l0;
  batched<4>(nzh * FZ_LINES,
             [&](int t) {
               const int k = t / FZ_LINES, l = t % FZ_LINES;
               const float2 *o = src + (long)k * nlines + 2 * l;
               float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
               if (2 * l < nl) { const float2 a = o[0]; v.x = a.x; v.y = a.y; }
               if (2 * l + 1 < nl) { const float2 b = o[1]; v.z = b.x; v.w = b.y; }
               return v;
             },
             [&](int t, float4 v) {
               const int k = t / FZ_LINES;
               float2 *x = buf + (t % FZ_LINES) * ls;
               if (k == 0 || 2 * k == nz) {
                 x[pos[k]] = make_float2(v.x, v.z);   // real lines: no imaginary part here
               } else {
                 x[pos[k]] = make_float2(v.x - v.w, v.y + v.z);
                 x[pos[nz - k]] = make_float2(v.x + v.w, v.z - v.y);
               }
             });
  __syncthreads();
  fft_inverse(buf, FZ_LINES, ls, 1, nz, P.rad[2], stw);
  const float *fb = reinterpret_cast<const float *>(buf);
  const int out = P.ik ? nz : P.mzs;
  const float inv = 1.f / (float)out;
  for (int t = threadIdx.x; t < nl * out; t += blockDim.x) {
    const int l = div_small(t, inv), z = t - l * out;
    const float v = fb[2 * ((l >> 1) * ls + (z < nz ? z : z - nz)) + (l & 1)];
    if (P.ik) mesh[P.omesh0 + 4 * ((long)l0 * nz + t) + comp] = v;
    else mesh[P.omesh0 + (long)l0 * out + t] = v;
  }
}

// The x transforms of a tile of one kz plane in LDS (its ncol columns y0 ..
// of the plane's ny, x points ls apart): forward, the influence function,
// inverse, and what the points add to the mesh energy 1/2 sum G |rho_k|^2
// and its virial W_ab = sum e_k (delta_ab - 2 k_a k_b (1/k^2 + 1/(4 eta^2)))
// (ENER, VIR).  comp > 0: E_a = -i k_a phi_k, a = comp - 1, k from the signed
// x, y index and the half-spectrum z index (pppm.c:577-594).
// fx, fy: signed frequencies of the places along x and y.
template <bool VIR, bool ENER, bool IK>
__device__ __forceinline__ void convolve_x(const SysParams &P, float2 *buf, int ls, int ncol, int y0,
                                           int kz, int comp, const float2 *twx, const short *fx,
                                           const short *fy, const float *__restrict__ green,
                                           double &e, double *w) {
  const float *g = green + P.green0 + (long)kz * P.nx * P.ny + y0;
  const int ny = P.ny;
  const double mult = (kz == 0 || 2 * kz == P.nz) ? 1.0 : 2.0;
  const double c4 = 0.25 / (P.eta * P.eta);
  fft_forward<false>(buf, ncol, 1, ls, P.nx, P.rad[0], twx);
  fft_middle(
      buf, ncol, 1, ls, P.nx, P.rad[0], [&](int c, int px) { return g[px * ny + c]; },
      [&](int c, int px, float gg, float2 &v) {
        if (ENER && comp == 0) {
          const double ek = 0.5 * mult * (double)gg * ((double)v.x * v.x + (double)v.y * v.y);
          e += ek;
          if (VIR && gg != 0.f) {
            double k[3];
            for (int a = 0; a < 3; a++)
              k[a] = P.RL[a] * fx[px] + P.RL[3 + a] * fy[y0 + c] + P.RL[6 + a] * kz;
            const double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
            const double f = 2 * (1 / k2 + c4);
            for (int a = 0; a < 3; a++)
              for (int b = 0; b < 3; b++)
                w[3 * a + b] += ek * ((a == b ? 1.0 : 0.0) - f * k[a] * k[b]);
          }
        }
        {   // rounded here in every variant of the kernel, not fused into the butterfly
#pragma clang fp contract(off)
          v = make_float2(v.x * gg, v.y * gg);
          if (IK && comp > 0) {
            const int a = comp - 1;
            const float k = (float)(P.RL[a] * fx[px] + P.RL[3 + a] * fy[y0 + c] + P.RL[6 + a] * kz);
            v = make_float2(k * v.y, -k * v.x);
          }
        }
      });
  fft_inverse<false>(buf, ncol, 1, ls, P.nx, P.rad[0], twx);
}

template <int NV, int TB>
__device__ __forceinline__ void mesh_energy(double e, const double *w, int s, int nblk, int blk,
                                            double *part, int *done, double *acc, double *kvir,
                                            int maxblk) {
  __shared__ double red[TB / 64][NV];
  __shared__ int last;
  double vals[NV];
  vals[0] = e;
  for (int c = 1; c < NV; c++) vals[c] = w[c - 1];
  if (finish_partials<NV, NV, TB>(vals, part + (long)s * maxblk * NV, nblk, blk, &done[s], red, &last)) {
    acc[s * NACC + ACC_KSPACE_E] = vals[0];
    for (int c = 0; c < 9; c++) kvir[9 * s + c] = NV > 1 ? vals[c + 1] : 0.0;
  }
}

// One kz plane of a system: forward y and x, the influence function, inverse
// x and y, all in LDS, where the four line passes of a mesh used to go to
// memory and back and cost a launch each.  One block per plane (and per
// component with the field on the mesh, which repeats the forward transforms
// rather than wait for them); 512 threads of at most 64 registers and up to
// 46 KB of LDS, so that a block fits beside three blocks of the pair kernel
// on a CU.  What bounds it is the chain of nine LDS round trips, about 1 us
// each: 12 us at 48^3 and 16 at 64^3, against 21 and 22 us and two launches
// more for a pass per axis (39 against 14 at 45 x 42 x 48 with the field on
// the mesh).  Pairing the z and y lines of an x slab in one block instead and
// leaving x alone takes as long (9 + 7 + 9 us at 48^3 against 6 + 12 + 6).
template <bool VIR, bool ENER, bool IK>
__global__ void __launch_bounds__(FP_TB, (VIR || ENER) ? 4 : 8) k_fft_plane(const SysParams *__restrict__ sp,
                                                        const float2 *__restrict__ twid_all,
                                                        const float *__restrict__ green,
                                                        float2 *__restrict__ cmesh,
                                                        double *__restrict__ part,
                                                        int *__restrict__ done,
                                                        double *__restrict__ acc,
                                                        double *__restrict__ kvir, int maxblk) {
  before_pairs();
  extern __shared__ float2 plane[];
  __shared__ float2 twx[FFT_MAXN], twy[FFT_MAXN];
  __shared__ short fx[FFT_MAXN], fy[FFT_MAXN];
  const int s = blockIdx.y, kz = blockIdx.x, comp = IK ? blockIdx.z : 0;
  const SysParams &P = sp[s];
  if (P.kmode != 1 || !P.plane) return;
  const int nx = P.nx, ny = P.ny, nzh = P.nz / 2 + 1, ls = ny | 1;
  if (kz >= nzh || (IK && comp > 0 && !P.ik)) return;
  load_tw(twx, twid_all + P.twid0, nx);
  load_tw(twy, twid_all + P.twid0 + FFT_MAXN, ny);
  if (VIR || IK) {
    load_freq(fx, twid_all + P.twid0, nx);
    load_freq(fy, twid_all + P.twid0 + FFT_MAXN, ny);
  }
  float2 *src = cmesh + P.cmesh0 + (long)kz * nx * ny;
  const float inv = 1.f / (float)ny;
  batched<8>(nx * ny, [&](int t) { return src[t]; },
             [&](int t, float2 v) { plane[t + div_small(t, inv) * (ls - ny)] = v; });
  __syncthreads();
  fft_forward(plane, nx, ls, 1, ny, P.rad[1], twy);
  double e = 0, w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  convolve_x<VIR, ENER, IK>(P, plane, ls, ny, 0, kz, comp, twx, fx, fy, green, e, w);
  fft_inverse(plane, nx, ls, 1, ny, P.rad[1], twy);
  // the field's components go beside the density's spectrum, which the
  // blocks of the other components read
  float2 *dst = src + (IK && P.ik ? (comp + 1) * (long)nx * ny * nzh : 0);
  for (int t = threadIdx.x; t < nx * ny; t += FP_TB) {
    const int x = div_small(t, inv);
    dst[t] = plane[t + x * (ls - ny)];
  }
  if (ENER && comp == 0)
    mesh_energy<VIR ? 10 : 1, FP_TB>(e, w, s, nzh, kz, part, done, acc, kvir, maxblk);
}

// Planes too large for that: y lines forward and inverse in passes of their
// own, and x lines with the influence function between them, 16 lines a block.
constexpr int FL_LINES = 16, FL_TB = 256;

template <bool INV>
__global__ void __launch_bounds__(FL_TB, 4) k_fft_y(const SysParams *__restrict__ sp,
                                                    const float2 *__restrict__ twid_all,
                                                    float2 *__restrict__ cmesh) {
  before_pairs();
  __shared__ float2 buf[FL_LINES * (FFT_MAXN + 1)], twy[FFT_MAXN];
  const SysParams &P = sp[blockIdx.y];
  if (P.kmode != 1 || P.plane) return;
  const int comp = blockIdx.z;
  if (comp > 0 && !P.ik) return;
  const int ny = P.ny, ls = ny | 1, nlines = P.nx * (P.nz / 2 + 1);
  const int l0 = blockIdx.x * FL_LINES, nl = min(FL_LINES, nlines - l0);
  if (nl <= 0) return;
  load_tw(twy, twid_all + P.twid0 + FFT_MAXN, ny);
  float2 *src = cmesh + P.cmesh0 + (INV && P.ik ? comp + 1 : 0) * (long)nlines * ny + (long)l0 * ny;
  const float inv = 1.f / (float)ny;
  batched<8>(nl * ny, [&](int t) { return src[t]; },
             [&](int t, float2 v) { buf[t + div_small(t, inv) * (ls - ny)] = v; });
  __syncthreads();
  if (INV) fft_inverse(buf, nl, ls, 1, ny, P.rad[1], twy);
  else fft_forward(buf, nl, ls, 1, ny, P.rad[1], twy);
  for (int t = threadIdx.x; t < nl * ny; t += FL_TB) src[t] = buf[t + div_small(t, inv) * (ls - ny)];
}

template <bool VIR, bool ENER, bool IK>
__global__ void __launch_bounds__(FL_TB, 4) k_fft_x(const SysParams *__restrict__ sp,
                                                    const float2 *__restrict__ twid_all,
                                                    const float *__restrict__ green,
                                                    float2 *__restrict__ cmesh,
                                                    double *__restrict__ part,
                                                    int *__restrict__ done,
                                                    double *__restrict__ acc,
                                                    double *__restrict__ kvir, int maxblk) {
  before_pairs();
  constexpr int LS = FL_LINES + 1;
  __shared__ float2 buf[LS * FFT_MAXN], twx[FFT_MAXN];
  __shared__ short fx[FFT_MAXN], fy[FFT_MAXN];
  const int s = blockIdx.y, comp = IK ? blockIdx.z : 0;
  const SysParams &P = sp[s];
  if (P.kmode != 1 || P.plane || (IK && comp > 0 && !P.ik)) return;
  const int nx = P.nx, ny = P.ny, nzh = P.nz / 2 + 1, nt = (ny + FL_LINES - 1) / FL_LINES;
  if ((int)blockIdx.x >= nzh * nt) return;
  const int kz = blockIdx.x / nt, y0 = blockIdx.x % nt * FL_LINES, nl = min(FL_LINES, ny - y0);
  load_tw(twx, twid_all + P.twid0, nx);
  if (VIR || IK) {
    load_freq(fx, twid_all + P.twid0, nx);
    load_freq(fy, twid_all + P.twid0 + FFT_MAXN, ny);
  }
  float2 *src = cmesh + P.cmesh0 + (long)kz * nx * ny + y0;
  batched<8>(nx * FL_LINES,
             [&](int t) {
               const int c = t % FL_LINES;
               return c < nl ? src[t / FL_LINES * ny + c] : make_float2(0.f, 0.f);
             },
             [&](int t, float2 v) { buf[t / FL_LINES * LS + t % FL_LINES] = v; });
  __syncthreads();
  double e = 0, w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  convolve_x<VIR, ENER, IK>(P, buf, LS, nl, y0, kz, comp, twx, fx, fy, green, e, w);
  float2 *dst = src + (IK && P.ik ? (comp + 1) * (long)nx * ny * nzh : 0);
  for (int t = threadIdx.x; t < nx * FL_LINES; t += FL_TB) {
    const int x = t / FL_LINES, c = t % FL_LINES;
    if (c < nl) dst[(long)x * ny + c] = buf[x * LS + c];
  }
  if (ENER && comp == 0)
    mesh_energy<VIR ? 10 : 1, FL_TB>(e, w, s, nzh * nt, blockIdx.x, part, done, acc, kvir, maxblk);
}

// Mesh buffers of one system, whose sizes, order and ik are set: the charge
// mesh at mesh0, the mesh the gather reads at omesh0, the half spectra at
// cmesh0; mesh and cmesh (floats and complex numbers so far) advance.
// A plane goes through k_fft_plane if it leaves three pair blocks of a CU
// their LDS (48 KB of 160 free beside them).
int p3m_mesh_layout(SysParams &P, long &mesh, long &cmesh) {
  const int n[3] = {P.nx, P.ny, P.nz};
  for (int d = 0; d < 3; d++)
    if (n[d] > FFT_MAXN || !fft_plan(n[d], P.rad[d])) return -1;
  const long M = (long)P.nx * P.ny * P.nz, Mc = (long)P.nx * P.ny * (P.nz / 2 + 1);
  P.plane = P.nx * (P.ny | 1) <= FFT_PLANE_MAX;
  P.mzs = P.nz + P.order - 1;
  P.mesh0 = mesh;
  mesh = (mesh + M + 3) & ~3L;   // 16-byte aligned: an ik system's points are float4
  P.omesh0 = mesh;
  mesh = (mesh + (P.ik ? 4 * M : (long)P.nx * P.ny * P.mzs) + 3) & ~3L;
  P.cmesh0 = cmesh;
  cmesh += (P.ik ? 5 : 1) * Mc;   // the density's, then phi, Ex, Ey, Ez of an ik system
  return 0;
}

// The system's tables: exp(-2 pi i t / n) for each axis (128 entries), then
// for each axis (place of frequency t, signed frequency of place t) as ints
// (128 entries).
void p3m_twiddles(const SysParams &P, std::vector<float2> &tw) {
  const int n[3] = {P.nx, P.ny, P.nz};
  const size_t at = tw.size();
  tw.resize(at + P3M_TWIDDLES);
  for (int d = 0; d < 3; d++)
    for (int t = 0; t < FFT_MAXN; t++) {
      const double a = -2 * M_PI * (t % n[d]) / n[d];
      tw[at + d * FFT_MAXN + t] = make_float2((float)cos(a), (float)sin(a));
    }
  for (int d = 0; d < 3; d++) {
    float2 *f = &tw[at + (3 + d) * FFT_MAXN];
    for (int k = 0; k < n[d]; k++) {
      const int p = fft_pos(k, n[d], P.rad[d]), sg = k > n[d] / 2 ? k - n[d] : k;
      memcpy(&f[k].x, &p, sizeof p);
      memcpy(&f[p].y, &sg, sizeof sg);
    }
  }
}

// where the influence function's value at (ix, iy, kz) is stored, relative to green0
long p3m_green_at(const SysParams &P, int ix, int iy, int kz) {
  return ((long)kz * P.nx + fft_pos(ix, P.nx, P.rad[0])) * P.ny + fft_pos(iy, P.ny, P.rad[1]);
}

// partial sums of the mesh energy: one per block of the x transforms
int p3m_energy_blocks(const SysParams &P) {
  return (P.nz / 2 + 1) * (P.plane ? 1 : (P.ny + FL_LINES - 1) / FL_LINES);
}

// IK: systems whose field was formed on the mesh; phi and E_a are
// interpolated from their four meshes with the assignment weights
// (pppm.c:618-626), E already Cartesian
template <int P, bool IK = false>
__global__ void __launch_bounds__(256, 4) k_p3m_gather(const SysParams *__restrict__ sp,
                                                    const int4 *__restrict__ sgrid,
                                                    const float4 *__restrict__ sfrac,
                                                    const float *__restrict__ mesh,
                                                    double *__restrict__ kres,
                                                    int *__restrict__ fill) {
  before_pairs();
  const int s = blockIdx.y;
  const SysParams &Q = sp[s];
  if (Q.kmode != 1 || Q.order != P || Q.ik != (int)IK) return;
  if (blockIdx.x == 0)   // the spreading has read the bin counters: clear them
    for (int t = threadIdx.x; t < Q.nbx * Q.nby; t += blockDim.x) fill[Q.bin0 + t] = 0;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Q.nsite) return;
  const int si = Q.site0 + i;
  const int4 g = sgrid[si];
  const float4 f = sfrac[si];
  const int nx = Q.nx, ny = Q.ny, nz = Q.nz;
  constexpr int istart = -((P + 1) / 2 - 1);
  float wx[P], wy[P], wz[P], dx[P], dy[P], dz[P];
  bspline_w<P>(f.x, wx, IK ? nullptr : dx);
  bspline_w<P>(f.y, wy, IK ? nullptr : dy);
  bspline_w<P>(f.z, wz, IK ? nullptr : dz);
  int ix[P], iy[P], iz[P];
#pragma unroll
  for (int a = 0; a < P; a++) {
    ix[a] = wrap(g.x + istart + a, nx);
    iy[a] = wrap(g.y + istart + a, ny);
    iz[a] = wrap(g.z + istart + a, nz);
  }
  const float *m0 = mesh + Q.omesh0;
  float ph = 0.f, e0 = 0.f, e1 = 0.f, e2 = 0.f;
  if constexpr (IK) {
    // the last inverse pass leaves (phi, Ex, Ey, Ez) interleaved per point
    const float4 *m4 = reinterpret_cast<const float4 *>(m0);
#pragma unroll
    for (int a = 0; a < P; a++) {
#pragma unroll
      for (int b = 0; b < P; b++) {
        const float4 *col = m4 + ((long)ix[a] * ny + iy[b]) * nz;
        const float wxy = wx[a] * wy[b];
#pragma unroll
        for (int c = 0; c < P; c++) {
          const float w = wxy * wz[c];
          const float4 v = col[iz[c]];
          ph += w * v.x;
          e0 += w * v.y;
          e1 += w * v.z;
          e2 += w * v.w;
        }
      }
    }
    kres[4 * si] = (double)ph;
    kres[4 * si + 1] = (double)e0;
    kres[4 * si + 2] = (double)e1;
    kres[4 * si + 3] = (double)e2;
    return;
  }
#pragma unroll
  for (int a = 0; a < P; a++) {
#pragma unroll
    for (int b = 0; b < P; b++) {
      // the run of P points along z, contiguous in the padded line (the
      // compiler makes it wide loads: two instead of five at order 5)
      float run[P];
      __builtin_memcpy(run, m0 + (ix[a] * ny + iy[b]) * Q.mzs + iz[0], sizeof run);
      float cp = 0.f, cz = 0.f;
#pragma unroll
      for (int c = 0; c < P; c++) {
        cp += wz[c] * run[c];
        cz += dz[c] * run[c];
      }
      const float wxy = wx[a] * wy[b];
      ph += wxy * cp;
      e0 += dx[a] * wy[b] * cp;
      e1 += wx[a] * dy[b] * cp;
      e2 += wxy * cz;
    }
  }
  const double *T = Q.T;
  kres[4 * si] = (double)ph;
  kres[4 * si + 1] = (double)e0 * T[0] + (double)e1 * T[1] + (double)e2 * T[2];
  kres[4 * si + 2] = (double)e0 * T[3] + (double)e1 * T[4] + (double)e2 * T[5];
  kres[4 * si + 3] = (double)e0 * T[6] + (double)e1 * T[7] + (double)e2 * T[8];
}

// The convolution: forward z, the kz planes, inverse z.  sp / nsg: the systems
// the grid's y extent covers (all of them, or one system's parameters with
// nsg = 1), hp their host copies; halo: the spreading blocks' partials the z
// pass sums (null: the real mesh holds the charges).
template <bool VIR, bool ENER, bool IK>
static void launch_planes(Engine &e, hipStream_t st, const SysParams *sp, const SysParams *hp, int nsg) {
  int np = 0, lds = 0, ny = 0, nx = 0;
  for (int s = 0; s < nsg; s++) {
    const SysParams &P = hp[s];
    if (P.kmode != 1) continue;
    const int nzh = P.nz / 2 + 1;
    if (P.plane) {
      np = std::max(np, nzh);
      lds = std::max(lds, P.nx * (P.ny | 1));
    } else {
      ny = std::max(ny, (P.nx * nzh + FL_LINES - 1) / FL_LINES);
      nx = std::max(nx, p3m_energy_blocks(P));
    }
  }
  const int nc = IK ? 4 : 1;
  if (np)
    hipLaunchKernelGGL((k_fft_plane<VIR, ENER, IK>), dim3(np, nsg, nc), dim3(FP_TB),
                       lds * sizeof(float2), st, sp, e.d_twid, e.d_green, e.d_cmesh, e.d_part,
                       e.d_done + e.nsys, e.d_acc, e.d_kres + 4L * e.nsite, e.nblk_part);
  if (nx) {
    hipLaunchKernelGGL(k_fft_y<false>, dim3(ny, nsg), dim3(FL_TB), 0, st, sp, e.d_twid, e.d_cmesh);
    hipLaunchKernelGGL((k_fft_x<VIR, ENER, IK>), dim3(nx, nsg, nc), dim3(FL_TB), 0, st, sp, e.d_twid,
                       e.d_green, e.d_cmesh, e.d_part, e.d_done + e.nsys, e.d_acc,
                       e.d_kres + 4L * e.nsite, e.nblk_part);
    hipLaunchKernelGGL(k_fft_y<true>, dim3(ny, nsg, nc), dim3(FL_TB), 0, st, sp, e.d_twid, e.d_cmesh);
  }
}

static void launch_fft(Engine &e, int want_virial, int energies, hipStream_t st, const SysParams *sp,
                       const SysParams *hp, int nsg, const unsigned long long *halo,
                       bool spread_does) {
  int nz = 0;
  bool ik = false, left = false;   // left: z lines that the spreading did not transform
  for (int s = 0; s < nsg; s++)
    if (hp[s].kmode == 1) {
      left |= !(spread_does && spread_transforms(hp[s]));
      nz = std::max(nz, (hp[s].nx * hp[s].ny + 2 * FZ_LINES - 1) / (2 * FZ_LINES));
      ik |= hp[s].ik != 0;
    }
  if (halo)
    hipLaunchKernelGGL(k_fft_z<true>, dim3(nz, nsg), dim3(FZ_TB), 0, st, sp, e.d_twid, e.d_mesh,
                       e.d_cmesh, halo, 0);
  else if (left)
    hipLaunchKernelGGL(k_fft_z<false>, dim3(nz, nsg), dim3(FZ_TB), 0, st, sp, e.d_twid, e.d_mesh,
                       e.d_cmesh, halo, spread_does ? 1 : 0);
#define PLANES(V, E)                                             \
  if (ik) launch_planes<V, E, true>(e, st, sp, hp, nsg);         \
  else launch_planes<V, E, false>(e, st, sp, hp, nsg);
  if (want_virial) { PLANES(true, true) }
  else if (energies) { PLANES(false, true) }
  else { PLANES(false, false) }
#undef PLANES
  hipLaunchKernelGGL(k_fft_zinv, dim3(nz, nsg, ik ? 4 : 1), dim3(FZ_TB), 0, st, sp, e.d_twid,
                     e.d_cmesh, e.d_mesh);
}

// LDS of a pulling block's complex lines
static size_t pull_lines(const SysParams &p) {
  return spread_transforms(p) ? sizeof(float2) * p.bx * p.by / 2 * (p.nz | 1) : 0;
}

int launch_p3m(Engine &e, int want_virial, hipStream_t st, int energies) {
  int maxn = 0, maxbins = 0;
  for (auto &p : e.hsp)
    if (p.kmode == 1) {
      maxn = std::max(maxn, p.nsite);
      maxbins = std::max(maxbins, p.nbx * p.nby);
    }
  if (maxn == 0) return 0;
  const int tb = 256;
  dim3 gs((maxn + tb - 1) / tb, e.nsys);
  hipLaunchKernelGGL(k_p3m_bin, gs, dim3(tb), 0, st, e.d_sp, e.d_r, e.d_q, e.nsite,
                     e.d_sgrid, e.d_sfrac, e.d_bin_fill, e.bcap, e.d_bgrid, e.d_bfrac, e.d_err,
                     e.d_bin_fill + e.nbin_total);
  bool used[MAXORDER + 1] = {false}, used_ad[MAXORDER + 1] = {false},
       used_ik[MAXORDER + 1] = {false};
  for (auto &p : e.hsp)
    if (p.kmode == 1) {
      used[p.order] = true;
      (p.ik ? used_ik : used_ad)[p.order] = true;
    }
  // LDS of the spreading: the largest halo, or block, of the systems of each order
  size_t hbytes[MAXORDER + 1] = {0};
  const int h = e.spread_halo ? 1 : 0;
  int htb = 256;   // by owner: a second round of work items costs more than idle threads
  for (auto &p : e.hsp)
    if (p.kmode == 1)
      hbytes[p.order] = std::max(hbytes[p.order], sizeof(unsigned long long) * p.nz *
                                                      (p.bx + h * (p.order - 1)) *
                                                      (p.by + h * (p.order - 1)) +
                                                      (h ? 0 : pull_lines(p)));
  for (auto &p : e.hsp)
    if (p.kmode == 1 && (long)p.nsite * p.order > 384L * p.nbx * p.nby) htb = 512;
#define SPREAD(PO)                                                                           \
  if (used[PO] && e.spread_halo)                                                             \
    hipLaunchKernelGGL(k_p3m_spread_halo<PO>, dim3(maxbins, e.nsys), dim3(htb), hbytes[PO],   \
                       st, e.d_sp, e.d_bin_fill, e.bcap, e.d_bgrid, e.d_bfrac, e.d_halo);     \
  else if (used[PO])                                                                         \
    hipLaunchKernelGGL(k_p3m_spread<PO>, dim3(maxbins, e.nsys), dim3(256), hbytes[PO], st,    \
                       e.d_sp, e.d_bin_fill, e.bcap, e.d_bgrid, e.d_bfrac, e.d_mesh, e.d_twid,  \
                       e.d_cmesh);
  SPREAD(1) SPREAD(2) SPREAD(3) SPREAD(4) SPREAD(5) SPREAD(6) SPREAD(7)
#undef SPREAD
  launch_fft(e, want_virial, energies, st, e.d_sp, e.hsp.data(), e.nsys,
             e.spread_halo ? e.d_halo : nullptr, !e.spread_halo);
#define GATHER(PO)                                                                        \
  if (used_ad[PO])                                                                        \
    hipLaunchKernelGGL(k_p3m_gather<PO>, gs, dim3(tb), 0, st, e.d_sp, e.d_sgrid,     \
                       e.d_sfrac, e.d_mesh, e.d_kres, e.d_bin_fill);                      \
  if (used_ik[PO])                                                                        \
    hipLaunchKernelGGL((k_p3m_gather<PO, true>), gs, dim3(tb), 0, st, e.d_sp, e.d_sgrid, \
                       e.d_sfrac, e.d_mesh, e.d_kres, e.d_bin_fill);
  GATHER(1) GATHER(2) GATHER(3) GATHER(4) GATHER(5) GATHER(6) GATHER(7)
#undef GATHER
  MM_HIP(hipGetLastError());
  return 0;
}

// The mesh adjoint of one P3M system: bin its sites again (the last gather
// cleared the counters; positions are those of the last evaluation), spread
// the adjoint source src (per site, global site index), convolve with the
// influence function (no energy), and gather the potential of the result
// into kres[4 i] of the system's sites (kres[4 i + 1..3] receive its
// field, unused).
int launch_p3m_adjoint(Engine &e, int sys, const float4 *src, hipStream_t st) {
  const SysParams &P = e.hsp[sys];
  if (P.kmode != 1) return 0;
  const SysParams *sp = e.d_sp + sys;
  const int tb = 256;
  const dim3 gs((P.nsite + tb - 1) / tb, 1);
  hipLaunchKernelGGL(k_p3m_bin, gs, dim3(tb), 0, st, sp, e.d_r, e.d_q, e.nsite, e.d_sgrid,
                     e.d_sfrac, e.d_bin_fill, e.bcap, e.d_bgrid, e.d_bfrac, e.d_err,
                     e.d_bin_fill + e.nbin_total);
  const dim3 gb(P.nbx * P.nby, 1);
  const size_t blds = sizeof(unsigned long long) * P.bx * P.by * P.nz;
#define ADJ_ORDER(PO)                                                                        \
  case PO:                                                                                   \
    hipLaunchKernelGGL(k_p3m_spread_adj<PO>, gb, dim3(256), blds, st, sp, e.d_bin_fill,      \
                       e.bcap, e.d_bgrid, e.d_bfrac, e.d_mesh, src);                         \
    break;
  switch (P.order) {
    ADJ_ORDER(1) ADJ_ORDER(2) ADJ_ORDER(3) ADJ_ORDER(4) ADJ_ORDER(5) ADJ_ORDER(6) ADJ_ORDER(7)
    default: set_last_error("assignment order out of range"); return -1;
  }
#undef ADJ_ORDER
  launch_fft(e, 0, 0, st, sp, &P, 1, nullptr, false);
#define ADJ_GATHER(PO)                                                                      \
  case PO:                                                                                  \
    hipLaunchKernelGGL(k_p3m_gather<PO>, gs, dim3(tb), 0, st, sp, e.d_sgrid, e.d_sfrac,     \
                       e.d_mesh, e.d_kres, e.d_bin_fill);                                   \
    break;
  switch (P.order) {
    ADJ_GATHER(1) ADJ_GATHER(2) ADJ_GATHER(3) ADJ_GATHER(4) ADJ_GATHER(5) ADJ_GATHER(6)
    ADJ_GATHER(7)
    default: break;
  }
#undef ADJ_GATHER
  MM_HIP(hipGetLastError());
  return 0;
}

// One forward ik pass of one system with the charges q (global site index)
// in place of its own: bin, spread by pulling, the ik convolution (no
// energy) and the ik gather, which leaves (phi, E) of the pass in kres[4 i]
// of the system's sites.  The ik field operator is a real circulant whose
// multiplier -i k_a G(k) is odd, so its transpose is its negative; the
// adjoint of the ik force therefore needs nothing but forward passes.
int launch_p3m_ik_pass(Engine &e, int sys, const double *q, hipStream_t st) {
  const SysParams &P = e.hsp[sys];
  if (P.kmode != 1 || !P.ik) return 0;
  const SysParams *sp = e.d_sp + sys;
  const int tb = 256;
  const dim3 gs((P.nsite + tb - 1) / tb, 1);
  hipLaunchKernelGGL(k_p3m_bin, gs, dim3(tb), 0, st, sp, e.d_r, q, e.nsite, e.d_sgrid,
                     e.d_sfrac, e.d_bin_fill, e.bcap, e.d_bgrid, e.d_bfrac, e.d_err,
                     e.d_bin_fill + e.nbin_total);
  const dim3 gb(P.nbx * P.nby, 1);
  const size_t blds = sizeof(unsigned long long) * P.bx * P.by * P.nz + pull_lines(P);
#define IK_SPREAD(PO)                                                                        \
  case PO:                                                                                   \
    hipLaunchKernelGGL(k_p3m_spread<PO>, gb, dim3(256), blds, st, sp, e.d_bin_fill, e.bcap,  \
                       e.d_bgrid, e.d_bfrac, e.d_mesh, e.d_twid, e.d_cmesh);                  \
    break;
  switch (P.order) {
    IK_SPREAD(1) IK_SPREAD(2) IK_SPREAD(3) IK_SPREAD(4) IK_SPREAD(5) IK_SPREAD(6) IK_SPREAD(7)
    default: set_last_error("assignment order out of range"); return -1;
  }
#undef IK_SPREAD
  launch_fft(e, 0, 0, st, sp, &P, 1, nullptr, true);
#define IK_GATHER(PO)                                                                       \
  case PO:                                                                                  \
    hipLaunchKernelGGL((k_p3m_gather<PO, true>), gs, dim3(tb), 0, st, sp, e.d_sgrid,        \
                       e.d_sfrac, e.d_mesh, e.d_kres, e.d_bin_fill);                        \
    break;
  switch (P.order) {
    IK_GATHER(1) IK_GATHER(2) IK_GATHER(3) IK_GATHER(4) IK_GATHER(5) IK_GATHER(6) IK_GATHER(7)
    default: break;
  }
#undef IK_GATHER
  MM_HIP(hipGetLastError());
  return 0;
}

}  // namespace mmamd
