// fft.hpp -- complex FFTs of lines held in LDS, in place, by mixed radices.
//
// A line of n points is transformed by up to three stages of radix 2..10
// (decimation in frequency): at a stage of sub-length m, the butterfly of
// block b and offset j takes the points b m + j + k m/R, k < R, transforms
// them in registers, multiplies the k-th by exp(-2 pi i j k / m) and puts
// them back where they came from.  No second buffer is needed, a stage costs
// one read and one write of LDS, and the transform ends in digit-reversed
// order (fft_pos gives a frequency's place).  The inverse runs the stages
// backwards (conjugate factors before the butterfly), from that order to the
// natural one, so a convolution needs no reordering at all.
#pragma once
#include <hip/hip_runtime.h>

namespace mmamd {

constexpr int FFT_STAGES = 3;

// radices of a length n (<= 128, factors 2, 3, 5, 7): as few stages as
// possible, and among those the smallest largest radix (registers)
inline bool fft_plan(int n, int *rad) {
  int best = 99;
  for (int a = 1; a <= 10; a++)
    for (int b = a; b <= 10; b++)
      for (int c = b; c <= 10; c++) {
        if (a * b * c != n) continue;
        const int cost = 16 * ((a > 1) + (b > 1) + (c > 1)) + c;
        if (cost < best) {
          best = cost;
          int k = 0;
          for (int r : {a, b, c})
            if (r > 1) rad[k++] = r;
          while (k < FFT_STAGES) rad[k++] = 0;
        }
      }
  return best < 99;
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// the place of frequency k in a transformed line of length n
inline int fft_pos(int k, int n, const int *rad) {
  int p = 0;
  for (int s = 0; s < FFT_STAGES && rad[s]; s++) {
    const int R = rad[s];
    n /= R;
    p += k % R * n;
    k /= R;
  }
  return p;
}

// cos and sin of 2 pi k / n for the butterflies' constants, by series
constexpr double fft_pi = 3.14159265358979323846;
constexpr double fft_cos(int k, int n) {
  k %= n;
  if (2 * k > n) k = n - k;
  const double x = 2 * fft_pi * k / n;
  double t = 1, s = 1;
  for (int i = 1; i < 20; i++) { t *= -x * x / ((2 * i - 1) * (2 * i)); s += t; }
  return s;
}
constexpr double fft_sin(int k, int n) {
  k %= n;
  const bool neg = 2 * k > n;
  if (neg) k = n - k;
  const double x = 2 * fft_pi * k / n;
  double t = x, s = x;
  for (int i = 1; i < 20; i++) { t *= -x * x / ((2 * i) * (2 * i + 1)); s += t; }
  return neg ? -s : s;
}
template <int N> struct FftConst {
  float c[N] = {}, s[N] = {};
  constexpr FftConst() {
    for (int k = 0; k < N; k++) { c[k] = (float)fft_cos(k, N); s[k] = (float)fft_sin(k, N); }
  }
};

// R-point transform of v in registers, natural order in and out
template <int R, bool INV>
__device__ __forceinline__ void dft(float2 *v) {
  if constexpr (R == 2) {
    const float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const float2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
    const float2 c = cadd(v[1], v[3]), d = csub(v[1], v[3]);
    const float2 di = INV ? make_float2(-d.y, d.x) : make_float2(d.y, -d.x);
    v[0] = cadd(a, c);
    v[2] = csub(a, c);
    v[1] = cadd(b, di);
    v[3] = csub(b, di);
  } else if constexpr (R == 3 || R == 5 || R == 7) {
    // symmetric and antisymmetric pairs: X_k, X_{R-k} = C_k -+ i S_k
    constexpr FftConst<R> T;
    constexpr int H = (R - 1) / 2;
    float2 p[H], m[H];
#pragma unroll
    for (int j = 0; j < H; j++) {
      p[j] = cadd(v[j + 1], v[R - 1 - j]);
      m[j] = csub(v[j + 1], v[R - 1 - j]);
    }
    const float2 x0 = v[0];
    float2 sum = x0;
#pragma unroll
    for (int j = 0; j < H; j++) sum = cadd(sum, p[j]);
    v[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; k++) {
      float2 c = x0, s = make_float2(0.f, 0.f);
#pragma unroll
      for (int j = 0; j < H; j++) {
        const int e = (j + 1) * k % R;
        c.x += T.c[e] * p[j].x;
        c.y += T.c[e] * p[j].y;
        s.x += T.s[e] * m[j].x;
        s.y += T.s[e] * m[j].y;
      }
      const float2 is = INV ? make_float2(-s.y, s.x) : make_float2(s.y, -s.x);
      v[k] = cadd(c, is);
      v[R - k] = csub(c, is);
    }
  } else {   // composite: A x B
    constexpr int A = R % 3 == 0 ? 3 : 2, B = R / A;
    constexpr FftConst<R> T;
    float2 u[R];
#pragma unroll
    for (int b = 0; b < B; b++) {
      float2 t[A];
#pragma unroll
      for (int a = 0; a < A; a++) t[a] = v[B * a + b];
      dft<A, INV>(t);
#pragma unroll
      for (int a = 0; a < A; a++)
        u[B * a + b] = a * b == 0 ? t[a]
                                  : cmul(t[a], make_float2(T.c[a * b % R], INV ? T.s[a * b % R] : -T.s[a * b % R]));
    }
#pragma unroll
    for (int a = 0; a < A; a++) {
      dft<B, INV>(u + B * a);
#pragma unroll
      for (int b = 0; b < B; b++) v[a + A * b] = u[B * a + b];
    }
  }
}

// quotient u / d for u < 2^22, inv = 1 / d
__device__ __forceinline__ int div_small(int u, float inv) { return (int)(((float)u + 0.5f) * inv); }

// One stage over nlines lines (line l at buf + l ls, its points es apart):
// consecutive threads take consecutive lines, then the next butterfly.
// tw: exp(-2 pi i t / n).
template <int R, bool INV>
__device__ __forceinline__ void fft_stage(float2 *buf, int nlines, int ls, int es, int n, int m,
                                          const float2 *tw) {
  const int sub = m / R, total = nlines * (n / R);
  const float inv_lines = 1.f / (float)nlines, inv_sub = 1.f / (float)sub;
  const unsigned ks = sub * es, step = n / m;
  for (int u = threadIdx.x; u < total; u += blockDim.x) {
    const unsigned b = div_small(u, inv_lines), l = u - __umul24(b, nlines);
    const unsigned blk = div_small(b, inv_sub), j = b - __umul24(blk, sub);
    float2 *x = buf + (__umul24(l, ls) + __umul24(__umul24(blk, m) + j, es));
    const float2 *t = tw;
    const unsigned jt = __umul24(j, step);
    float2 v[R];
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = x[__umul24(k, ks)];
    if (INV && sub > 1) {
#pragma unroll
      for (int k = 1; k < R; k++) {
        const float2 w = *(t += jt);
        v[k] = cmul(v[k], make_float2(w.x, -w.y));
      }
    }
    dft<R, INV>(v);
    if (!INV && sub > 1) {
#pragma unroll
      for (int k = 1; k < R; k++) v[k] = cmul(v[k], *(t += jt));
    }
#pragma unroll
    for (int k = 0; k < R; k++) x[__umul24(k, ks)] = v[k];
  }
  __syncthreads();
}

template <bool INV>
__device__ __forceinline__ void fft_stage_any(int R, float2 *buf, int nlines, int ls, int es, int n,
                                              int m, const float2 *tw) {
  switch (R) {
    case 2: fft_stage<2, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 3: fft_stage<3, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 4: fft_stage<4, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 5: fft_stage<5, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 6: fft_stage<6, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 7: fft_stage<7, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 8: fft_stage<8, INV>(buf, nlines, ls, es, n, m, tw); break;
    case 9: fft_stage<9, INV>(buf, nlines, ls, es, n, m, tw); break;
    default: fft_stage<10, INV>(buf, nlines, ls, es, n, m, tw); break;
  }
}

// All stages; every thread of the block calls them, the lines already
// visible to all; they end with a barrier.  INNER false leaves out the last
// forward and the first inverse stage, which fft_middle runs together.
template <bool INNER = true>
__device__ __forceinline__ void fft_forward(float2 *buf, int nlines, int ls, int es, int n,
                                            const int *rad, const float2 *tw) {
  int m = n;
  for (int s = 0; s < FFT_STAGES && rad[s]; s++) {
    if (!INNER && (s + 1 == FFT_STAGES || !rad[s + 1])) break;
    fft_stage_any<false>(rad[s], buf, nlines, ls, es, n, m, tw);
    m /= rad[s];
  }
}
template <bool INNER = true>
__device__ __forceinline__ void fft_inverse(float2 *buf, int nlines, int ls, int es, int n,
                                            const int *rad, const float2 *tw) {
  int s = 0, m = 1;
  while (s < FFT_STAGES && rad[s]) s++;
  while (--s >= 0) {
    m *= rad[s];
    if (INNER || s + 1 < FFT_STAGES && rad[s + 1])
      fft_stage_any<true>(rad[s], buf, nlines, ls, es, n, m, tw);
  }
}

// The last forward stage, f on every point of the transform, and the first
// inverse stage, in registers: both work on the same R points and neither has
// factors.  load(l, p) is issued with the points' reads; f(l, p, loaded, v)
// changes the point of line l at place p.
template <int R, class Load, class F>
__device__ __forceinline__ void fft_middle_r(float2 *buf, int nlines, int ls, int es, int n,
                                             Load load, F f) {
  const int total = nlines * (n / R);
  const float inv_lines = 1.f / (float)nlines;
  for (int u = threadIdx.x; u < total; u += blockDim.x) {
    const int b = div_small(u, inv_lines), l = u - b * nlines;
    float2 *x = buf + l * ls + b * R * es;
    float g[R];
#pragma unroll
    for (int k = 0; k < R; k++) g[k] = load(l, b * R + k);
    float2 v[R];
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = x[k * es];
    dft<R, false>(v);
#pragma unroll
    for (int k = 0; k < R; k++) f(l, b * R + k, g[k], v[k]);
    dft<R, true>(v);
#pragma unroll
    for (int k = 0; k < R; k++) x[k * es] = v[k];
  }
  __syncthreads();
}

template <class Load, class F>
__device__ __forceinline__ void fft_middle(float2 *buf, int nlines, int ls, int es, int n,
                                           const int *rad, Load load, F f) {
  int R = rad[0];
  for (int s = 1; s < FFT_STAGES && rad[s]; s++) R = rad[s];
  switch (R) {
    case 2: fft_middle_r<2>(buf, nlines, ls, es, n, load, f); break;
    case 3: fft_middle_r<3>(buf, nlines, ls, es, n, load, f); break;
    case 4: fft_middle_r<4>(buf, nlines, ls, es, n, load, f); break;
    case 5: fft_middle_r<5>(buf, nlines, ls, es, n, load, f); break;
    case 6: fft_middle_r<6>(buf, nlines, ls, es, n, load, f); break;
    case 7: fft_middle_r<7>(buf, nlines, ls, es, n, load, f); break;
    case 8: fft_middle_r<8>(buf, nlines, ls, es, n, load, f); break;
    case 9: fft_middle_r<9>(buf, nlines, ls, es, n, load, f); break;
    default: fft_middle_r<10>(buf, nlines, ls, es, n, load, f); break;
  }
}

// dst(t, src(t)) for every t < n over the block, U reads in flight per thread
template <int U, class Src, class Dst>
__device__ __forceinline__ void batched(int n, Src src, Dst dst) {
  for (int t0 = threadIdx.x; t0 < n; t0 += U * blockDim.x) {
    decltype(src(0)) v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int t = t0 + u * blockDim.x;
      if (t < n) v[u] = src(t);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int t = t0 + u * blockDim.x;
      if (t < n) dst(t, v[u]);
    }
  }
}

}  // namespace mmamd
