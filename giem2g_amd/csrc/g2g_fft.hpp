// g2g_fft.hpp -- batched complex FFTs held in LDS: radix-4 Stockham for
// powers of two, and a factor-plan Stockham for other lengths (below).
//
// NR independent rows of length L sit in LDS at buf[row*LS + i] (LS >= L, a
// padded row stride).  The transform is an in-place Stockham autosort FFT
// with radix-4 stages (plus one radix-2 stage when log2 L is odd): every
// thread loads its butterflies into registers, the block synchronises, and
// the outputs are written back to the same buffer.  Twiddles come from an
// LDS table tw[t] = exp(-2*pi*i*t/L).  DIR = -1 is the forward transform
// (exp(-i)), DIR = +1 the unnormalised inverse.
#pragma once
#include "g2g_common.hpp"

namespace g2g {

template <int R, int DIR, typename T2> __device__ inline void dft_small(T2* v) {
  if constexpr (R == 2) {
    T2 a = v[0], b = v[1];
    v[0] = a + b;
    v[1] = a - b;
  } else {
    T2 a0 = v[0] + v[2], a1 = v[0] - v[2];
    T2 a2 = v[1] + v[3], d = v[1] - v[3];
    T2 a3 = (DIR < 0) ? mul_mi(d) : mul_pi(d);
    v[0] = a0 + a2;
    v[2] = a0 - a2;
    v[1] = a1 + a3;
    v[3] = a1 - a3;
  }
}

template <typename T2, int L, int NR, int LS, int NT, int R, int DIR>
__device__ inline void stockham_stage(T2* buf, const T2* tw, int Ns) {
  constexpr int NBR = L / R;
  constexpr int NB = NR * NBR;
  constexpr int PER = (NB + NT - 1) / NT;
  T2 v[PER][R];
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int bi = tid + q * NT;
    if (NB % NT == 0 || bi < NB) {
      const int row = bi / NBR, j = bi % NBR;
      const int k = j & (Ns - 1);
#pragma unroll
      for (int r = 0; r < R; r++) v[q][r] = buf[row * LS + j + r * NBR];
      if (Ns > 1) {
        const int tstep = L / (Ns * R);
#pragma unroll
        for (int r = 1; r < R; r++) {
          T2 w = tw[k * r * tstep];
          if (DIR > 0) w.y = -w.y;
          v[q][r] = v[q][r] * w;
        }
      }
      dft_small<R, DIR>(v[q]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int bi = tid + q * NT;
    if (NB % NT == 0 || bi < NB) {
      const int row = bi / NBR, j = bi % NBR;
      const int k = j & (Ns - 1);
      const int idxD = (j - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; r++) buf[row * LS + idxD + r * Ns] = v[q][r];
    }
  }
  __syncthreads();
}

// Full transform.  Caller must __syncthreads() after filling buf and tw.
template <typename T2, int L, int NR, int LS, int NT, int DIR>
__device__ inline void lds_fft(T2* buf, const T2* tw) {
  constexpr int LOG = (L <= 1) ? 0 : (31 - __builtin_clz(L));
  constexpr int N4 = LOG / 2;
  int Ns = 1;
#pragma unroll
  for (int s = 0; s < N4; s++) {
    stockham_stage<T2, L, NR, LS, NT, 4, DIR>(buf, tw, Ns);
    Ns *= 4;
  }
  if constexpr (LOG & 1) stockham_stage<T2, L, NR, LS, NT, 2, DIR>(buf, tw, Ns);
}

// ------------------------------------------------------- any length ------
// Lengths that are not powers of two (any even Nx, Ny) run a Stockham autosort
// FFT over the length's factors -- fours, then twos, then the odd primes -- in
// the same LDS layout.  The plan is made on the host, with multipliers for the
// stages' divisions by runtime numbers.
struct FftPlan {
  int L = 0, nst = 0;
  int rad[8] = {};
  // q = umulhi(x, m) = x / d for x d < 2^32: d = L / rad, and d = the product
  // of the radices before (stage 0: not used)
  unsigned mb[8] = {}, mn[8] = {};
};

inline unsigned div_mul(int d) { return d > 1 ? (unsigned)(((uint64_t(1) << 32) + d - 1) / d) : 0; }

inline FftPlan fft_plan(int L) {
  FftPlan p;
  p.L = L;
  int n = L, ns = 1;
  auto push = [&](int r) {
    if (p.nst >= 8) throw Error(-3, "FFT length has too many factors");
    p.rad[p.nst] = r;
    p.mb[p.nst] = div_mul(L / r);
    p.mn[p.nst++] = div_mul(ns);
    ns *= r;
    n /= r;
  };
  while (n % 4 == 0) push(4);
  while (n % 2 == 0) push(2);
  for (int f = 3; n > 1; f += 2)
    while (n % f == 0) push(f);
  return p;
}

// x / d with m = div_mul(d)
__device__ inline int fast_div(int x, int d, unsigned m) { return d > 1 ? (int)__umulhi((unsigned)x, m) : x; }

// R-point DFT of an odd prime R: the inputs j and R - j enter every output as
// their sum times a cosine and their difference times a sine, shared by the
// outputs k and R - k.  cs[m - 1] = exp(-2 pi i m/R), m = 1 .. (R-1)/2.
template <int R, int DIR, typename T2> __device__ inline void dft_odd(T2* v, const T2* cs) {
  constexpr int H = (R - 1) / 2;
  T2 t[H], d[H];
  T2 x0 = v[0], sum = x0;
#pragma unroll
  for (int j = 1; j <= H; j++) {
    t[j - 1] = v[j] + v[R - j];
    d[j - 1] = v[j] - v[R - j];
    sum = sum + t[j - 1];
  }
  v[0] = sum;
#pragma unroll
  for (int k = 1; k <= H; k++) {
    T2 a = x0, b = mk<T2>(0, 0);
#pragma unroll
    for (int j = 1; j <= H; j++) {
      const int m = j * k % R;
      const T2 w = cs[(m <= H ? m : R - m) - 1];
      const auto sn = m <= H ? w.y : -w.y;  // -sin(2 pi m/R)
      a.x = fma(t[j - 1].x, w.x, a.x);
      a.y = fma(t[j - 1].y, w.x, a.y);
      b.x = fma(d[j - 1].x, sn, b.x);
      b.y = fma(d[j - 1].y, sn, b.y);
    }
    const T2 ib = mul_pi(b);  // i times the sines' part of the forward transform
    v[k] = DIR < 0 ? a + ib : a - ib;
    v[R - k] = DIR < 0 ? a - ib : a + ib;
  }
}

// One stage of a compile-time radix: butterflies in registers as in
// stockham_stage, at runtime length L and runtime product Ns of the radices
// before.  (Every output summed over its butterfly's R inputs on its own, with
// divisions by runtime numbers for each: forward and inverse passes together
// 184 us at 96x96x32 FP64, now 99; 417 -> 247 us at 176x224x16.)
template <typename T2, int R, int PER, int NT, int DIR>
__device__ inline void stockham_stage_rt(T2* buf, const T2* tw, int L, int NR, int LS, int Ns, unsigned mb, unsigned mn) {
  const int NBR = L / R, NB = NR * NBR, sK = NBR / Ns;
  T2 v[PER][R];
  int dst[PER];
  T2 cs[R > 4 || R == 3 ? (R - 1) / 2 : 1];
  if constexpr (R > 4 || R == 3) {
#pragma unroll
    for (int m = 1; m <= (R - 1) / 2; m++) cs[m - 1] = tw[m * NBR];
  }
#pragma unroll
  for (int p = 0; p < PER; p++) {
    const int bi = threadIdx.x + p * NT;
    if (bi < NB) {
      const int row = fast_div(bi, NBR, mb), j = bi - row * NBR;
      const int jq = fast_div(j, Ns, mn), k = j - jq * Ns;
      const T2* src = buf + row * LS + j;
      dst[p] = row * LS + jq * Ns * R + k;
#pragma unroll
      for (int r = 0; r < R; r++) v[p][r] = src[r * NBR];
      if (Ns > 1) {
        const int e = k * sK;
#pragma unroll
        for (int r = 1; r < R; r++) {
          T2 w = tw[r * e];
          if (DIR > 0) w.y = -w.y;
          v[p][r] = v[p][r] * w;
        }
      }
      if constexpr (R == 2 || R == 4) dft_small<R, DIR>(v[p]);
      else dft_odd<R, DIR>(v[p], cs);
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PER; p++) {
    if ((int)threadIdx.x + p * NT < NB) {
#pragma unroll
      for (int r = 0; r < R; r++) buf[dst[p] + r * Ns] = v[p][r];
    }
  }
  __syncthreads();
}

// 16x16x4 matrix products: lane l supplies A[row l%16][k l/16] and B[k
// l/16][col l%16] and holds four rows of column l%16 of the result: rows 4*kq +
// q (FP32) or kq + 4*q (FP64), kq = l/16 (both measured)
template <typename R> struct v4t;
template <> struct v4t<double> { typedef double t __attribute__((ext_vector_type(4))); };
template <> struct v4t<float> { typedef float t __attribute__((ext_vector_type(4))); };
__device__ inline v4t<double>::t mma4(double a, double b, v4t<double>::t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline v4t<float>::t mma4(float a, float b, v4t<float>::t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename R> __device__ inline int mma_row(int kq, int q);
template <> __device__ inline int mma_row<float>(int kq, int q) { return 4 * kq + q; }
template <> __device__ inline int mma_row<double>(int kq, int q) { return kq + 4 * q; }

// result tiles per wave of a prime stage: at most, over the primes from 11
constexpr int prime_tiles(int tot, int lc, int waves) {
  int most = 1;
  for (int r = 11; r <= lc / 2; r += 2) {
    const int items = (tot / r + 7) / 8 * (((r - 1) / 2 + 16) / 16);
    const int per = (items + waves - 1) / waves;
    if (per > most) most = per;
  }
  return most;
}

// A stage of a prime radix from 11 up, on the matrix cores: the sums t_q = x_q
// + x_{R-q} and differences d_q (q = 1 .. H = (R-1)/2, after the twiddles) take
// the inputs' places in LDS; then [cos 2 pi qk/R] t and [sin] d for k = 0 .. H are
// real matrix products with eight butterflies (16 real columns) per tile, and
// the outputs k and R - k are their sum and difference.  4 H (H + 1), about R^2,
// real products per butterfly (with k padded to tiles of 16 rows) where a sum
// over all inputs for every output takes 4 R^2 (both directions at 148x172x27,
// primes 37 and 43: FP64 706 -> 360 us, complex64 880 -> 289 us; eight vectors
// at 194x194x19, prime 97: 13.8 -> 5.9 ms a batch).  (The rows in batches of
// four tiles per wave, for fewer registers, made the complex64 passes 1.4-2.4
// times as long.)
template <typename T2, int LC, int NR, int NT, int DIR>
__device__ inline void stockham_stage_prime(T2* buf, const T2* tw, int L, int LS, int R, int Ns) {
  using RR = decltype(T2::x);
  using V4 = typename v4t<RR>::t;
  constexpr int NW = NT / 64, MAXI = prime_tiles(NR * LC, LC, NW);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kq = lane >> 4;
  const int H = (R - 1) / 2, NBR = L / R, NB = NR * NBR, sK = NBR / Ns;
  for (int e = threadIdx.x; e < NB * H; e += NT) {
    const int q1 = e / NB, c = e - q1 * NB, q = q1 + 1, row = c / NBR, j = c - row * NBR;
    T2* p = buf + row * LS + j;
    T2 x = p[q * NBR], y = p[(R - q) * NBR];
    if (Ns > 1) {
      const int f = j % Ns * sK;
      T2 wx = tw[q * f], wy = tw[(R - q) * f];
      if (DIR > 0) {
        wx.y = -wx.y;
        wy.y = -wy.y;
      }
      x = x * wx;
      y = y * wy;
    }
    p[q * NBR] = x + y;
    p[(R - q) * NBR] = x - y;
  }
  __syncthreads();
  const int MT = (H + 16) / 16;
  const int items = (NB + 7) / 8 * MT;
  const RR sg = ((col & 1) != 0) == (DIR < 0) ? RR(1) : RR(-1);  // of i b in output k
  V4 a[MAXI], b[MAXI];
#pragma unroll
  for (int it = 0; it < MAXI; it++) {
    const int item = wave + NW * it;
    if (item < items) {
      const int nt = item / MT, mt = item - nt * MT;
      const int c = min(8 * nt + (col >> 1), NB - 1), row = c / NBR, j = c - row * NBR;
      const RR* p = reinterpret_cast<const RR*>(buf + row * LS + j) + (col & 1);
      const int k = 16 * mt + col, step = 4 * k % R;
      int idx = (kq + 1) * k % R;
      const RR x0 = p[0];
      V4 va = {x0, x0, x0, x0}, vb = {0, 0, 0, 0};
      for (int q = kq + 1; q <= H + kq; q += 4) {  // (the same count in every lane)
        const bool ok = q <= H;
        const T2 w = tw[idx * NBR];
        const int qc = ok ? q : 1;
        const RR t = p[2 * qc * NBR], d = p[2 * (R - qc) * NBR];
        va = mma4(ok ? w.x : RR(0), ok ? t : RR(0), va);
        vb = mma4(ok ? w.y : RR(0), ok ? d : RR(0), vb);
        idx += step;
        if (idx >= R) idx -= R;
      }
      a[it] = va;
      b[it] = vb;
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < MAXI; it++) {
    const int item = wave + NW * it;
    if (item < items) {
      const int nt = item / MT, mt = item - nt * MT, c = 8 * nt + (col >> 1);
      const int row = c / NBR, j = c - row * NBR, jq = j / Ns;
      RR* p = reinterpret_cast<RR*>(buf + row * LS + jq * Ns * R + (j - jq * Ns)) + (col & 1);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int k = 16 * mt + mma_row<RR>(kq, i);
        const RR ib = sg * __shfl_xor(b[it][i], 1);  // the other part of b
        if (k <= H && c < NB) {
          p[2 * k * Ns] = a[it][i] + ib;
          if (k > 0) p[2 * (R - k) * Ns] = a[it][i] - ib;
        }
      }
    }
  }
  __syncthreads();
}

// Full transform of NR rows of length plan.L <= LC (the capacity the
// buffers were sized for).  RT = false: LC itself, a power of two, with
// lds_fft.  Caller must __syncthreads() after filling buf and tw.
template <typename T2, int LC, int NR, int LS, int NT, int DIR, bool RT>
__device__ inline void lds_fft_any(T2* buf, const T2* tw, const FftPlan& plan) {
  if constexpr (!RT) {
    lds_fft<T2, LC, NR, LS, NT, DIR>(buf, tw);
  } else {
    constexpr int TOT = NR * LC;  // butterflies of radix R: at most TOT / R
    auto per = [](int r) { return (TOT / r + NT - 1) / NT; };
    int Ns = 1;
    for (int s = 0; s < plan.nst; s++) {
#define G2G_STAGE(r)                                                                                       \
  case r:                                                                                                  \
    if constexpr (r <= LC / 2)                                                                             \
      stockham_stage_rt<T2, r, per(r), NT, DIR>(buf, tw, plan.L, NR, LS, Ns, plan.mb[s], plan.mn[s]);      \
    break;
      switch (plan.rad[s]) {
        G2G_STAGE(2) G2G_STAGE(3) G2G_STAGE(4) G2G_STAGE(5) G2G_STAGE(7)
        default: stockham_stage_prime<T2, LC, NR, NT, DIR>(buf, tw, plan.L, LS, plan.rad[s], Ns);
      }
#undef G2G_STAGE
      Ns *= plan.rad[s];
    }
  }
}

}  // namespace g2g
