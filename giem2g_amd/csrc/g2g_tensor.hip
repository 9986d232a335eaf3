// g2g_tensor.hip -- FP64 Green-tensor build and tensor spectrum on the GPU.
//
// Reference path replaced: CalcIntegralGreenTensor ->
// CalcIntegralGreenTensor3dElementGeneral -> {COMPUTE_WEIGHTS ->
// VBTransformWeightsAllDoubleInt, Calc_Double_Integral_U}
// (calc_ie_tensor_module.F90:54-352, VolumeBesselTransforms.F90:89-403,
// ie_kernel_hankel_module.F90:44-197, apq_module.F90:31-312) and
// CalcFFTofIETensorGeneral (Integral_Equation_Module.F90:319-471).
//
// The reference evaluates the layered vertical kernel U(lambda_K, W) once per
// (offset, tap).  U is linear in the six filter weights with coefficients
// that depend on lambda only, so here:
//   1. k_weights   : one block per lateral offset computes the 501x6 digital
//                    filter weights (1024-point FFT deconvolution in LDS),
//                    the 1e-12 tap mask and the lambda scaling;  these are
//                    frequency independent and cached;
//   2. k_lambda    : one block per tap K evaluates the weight-free kernel
//                    tables a,b,c (packed symmetric) and d (full) of
//                    Calc_Double_Integral_U;
//   3. k_wgemm     : G(offset, entry) = sum_K w(offset,K) * table(K, entry),
//                    FP64 (NxNy x taps) x (taps x Nz^2) matrix products;
//   4. k_tfft_y/x  : symmetric extension with per-component signs, 2-D FFT,
//                    Nyquist cancellation, in place.
#include "g2g_fft.hpp"
#include "g2g_op.hpp"

#include <cmath>
#include <vector>

namespace g2g {

constexpr int NTAPS = 501, NFIRST = 212, VBN = 1024;
constexpr double VB_YSTEP = 1e-1 * 2e0;
constexpr double VB_XI = -4.82205425726955430357775925664462079e-2 * 2e0;
constexpr double VB_Q = VB_YSTEP / 2.0;
constexpr double VB_P = VB_Q + VB_XI;
constexpr double PI_D = 3.1415926535897932384626433832795028841971693993751;
enum { IE_DXX = 0, IE_DXY = 1, IE_DYY = 2, IE_DX = 3, IE_DY = 4, IE_D0 = 5 };

// ------------------------------------------------------------ weights ---
__device__ inline double vb_inputfunction(double t) {
  const double y = exp(-t), y2 = y * y, y4 = y2 * y2;
  return 8.0 * exp(-y2) * (y4 - 4.0 * y2 + 2.0) * y;
}

// spectrum of the input function (VBTransformInit, VolumeBesselTransforms.F90:89-109)
__global__ __launch_bounds__(256) void k_f1(zd* f1out, const zd* twg) {
  __shared__ zd buf[VBN + 1];
  __shared__ zd tw[VBN];
  for (int i = threadIdx.x; i < VBN; i += 256) tw[i] = twg[i];
  for (int i = threadIdx.x; i < VBN; i += 256) {
    const int i0 = i & ~1;
    double y1 = (double)(i0 - 512) * VB_YSTEP + VB_Q;
    if (i & 1) y1 = y1 + VB_YSTEP;
    const double v = vb_inputfunction(y1);
    buf[i] = mkz((i & 1) ? -v : v, 0.0);
  }
  __syncthreads();
  lds_fft<zd, VBN, 1, VBN + 1, 256, +1>(buf, tw);
  for (int i = threadIdx.x; i < VBN; i += 256) f1out[i] = buf[i];
}

struct WParams {
  int Nx, Ny;
  double dx, dy, rmin, log_rmin;
};

// outfunc_int4_all for knot I (VolumeBesselTransforms.F90:304-550)
__device__ inline void outfunc4(double explt, double cphi, double sphi, double alpha, double beta,
                                double* R) {
  double f[2][3][3];  // [x/y][D0,D1,D2][1..3]
#pragma unroll
  for (int J = 0; J < 2; J++) {
    const double c = J == 0 ? cphi : sphi, h = J == 0 ? alpha : beta;
    double x1 = explt * c;
    const double dd = h * explt;
    x1 = x1 - dd * 0.5;
    double x[3] = {x1, x1 + dd, x1 - dd}, x2[3], ex[3], er[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      x[k] = x[k] * 0.5;
      x2[k] = x[k] * x[k];
      ex[k] = exp(-x2[k]);
      er[k] = erf(x[k]);
    }
#define D2(a) ((a)[1] + (a)[2] - 2.0 * (a)[0])
    double t[3], r0, r1, r2;
    // DOUBLE_INT_D0 via INT_2d_edt
    for (int k = 0; k < 3; k++) t[k] = x[k] * er[k];
    r0 = D2(t) * sqrt(PI_D) * 0.25;
    r1 = D2(ex);
    for (int k = 0; k < 3; k++) t[k] = ex[k] * x2[k] / 4.0;
    r2 = D2(t);
    f[J][0][0] = 32.0 * (1.5 * r0 + r1 + r2);
    f[J][0][1] = 8.0 * r0 + 4.0 * r1;
    f[J][0][2] = 4.0 * r0 + r1;
    // DOUBLE_INT_D1 via INT_1d_edt
    r0 = D2(er) * sqrt(PI_D) * 0.5;
    for (int k = 0; k < 3; k++) t[k] = ex[k] * x[k];
    r1 = D2(t);
    for (int k = 0; k < 3; k++) t[k] = t[k] * x2[k];
    r2 = D2(t);
    f[J][1][0] = -8.0 * r2 - 12.0 * r1 + 12.0 * r0;
    f[J][1][1] = -2.0 * r1 + 2.0 * r0;
    f[J][1][2] = r0;
    // DOUBLE_INT_D2
    double e2[3];
    for (int k = 0; k < 3; k++) e2[k] = ex[k] / 2.0;
    for (int k = 0; k < 3; k++) t[k] = x2[k] * e2[k] * 4.0;
    f[J][2][1] = D2(t);
    for (int k = 0; k < 3; k++) t[k] = x2[k] * t[k] * 4.0;
    f[J][2][0] = D2(t);
    f[J][2][2] = D2(e2);
#undef D2
  }
#define CMB(a, b) (f[0][a][2] * f[1][b][0] + f[0][a][0] * f[1][b][2] + 2.0 * f[0][a][1] * f[1][b][1])
  const double e2 = explt * explt, e3 = e2 * explt;
  R[0] = CMB(0, 0) / e3;
  R[1] = CMB(2, 0) / explt;
  R[2] = CMB(1, 1) / explt;
  R[3] = CMB(1, 0) / e2;
  R[4] = CMB(0, 2) / explt;
  R[5] = CMB(0, 1) / e2;
#undef CMB
}

__device__ inline double block_max(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  double r = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); i++) r = fmax(r, red[i]);
  return r;
}

// Window of taps [x, y) outside which every weight of an offset is zero:
// every thread reports its taps that are on
__device__ inline void tap_window(int* kw, int K, bool on) {
  if (!on) return;
  atomicMin(&kw[0], K);
  atomicMax(&kw[1], K + 1);
}

// One block per offset b = lx + Nx*ly.  Output wts[c][K][b] (IE order) and
// the offset's window of taps win[b].  A thread keeps the weights of its taps K =
// threadIdx.x + 256 u in registers and the twiddles stay in global memory:
// with the transforms' 49 KB of LDS two blocks share a CU (with weights and
// twiddles in LDS, 89 KB, one did: one wave per SIMD).  128x128 offsets: 3.61 ->
// 2.19 ms; twiddles in LDS 2.30, registers for three blocks 2.26.
__global__ __launch_bounds__(256) void k_weights(double* __restrict__ wts, int2* __restrict__ win,
                                                 const zd* __restrict__ f1,
                                                 const zd* __restrict__ twg,
                                                 const double* __restrict__ lms, WParams P) {
  constexpr int NRW = 3, LS = VBN + 1;
  __shared__ zd buf[NRW * LS];
  double wt[6][2];
  __shared__ double red[8];
  const int b = blockIdx.x, lx = b % P.Nx, ly = b / P.Nx;
  const double x = lx * P.dx + P.dx / 2.0, y = ly * P.dy + P.dy / 2.0;
  const double rho = sqrt(x * x + y * y);
  const double rp[6] = {rho * rho * rho, rho, rho, rho * rho, rho, rho * rho};
  const double alpha = P.dx / rho, beta = P.dy / rho, phi = atan2(y, x);
  const double cphi = cos(phi), sphi = sin(phi);
  const double s = log(rho) - P.log_rmin;
  for (int half = 0; half < 2; half++) {
    __syncthreads();
    for (int i = threadIdx.x; i < VBN; i += 256) {
      const int i0 = i & ~1;
      double y2 = (double)(i0 - 512) * VB_YSTEP + VB_P + s;
      if (i & 1) y2 = y2 + VB_YSTEP;
      const double explt = exp(y2);
      double R[6];
      outfunc4(explt, cphi, sphi, alpha, beta, R);
      const double sg = (i & 1) ? -1.0 : 1.0;
      for (int c = 0; c < NRW; c++) buf[c * LS + i] = mkz(sg * R[half * 3 + c], 0.0);
    }
    __syncthreads();
    lds_fft<zd, VBN, NRW, LS, 256, +1>(buf, twg);
    for (int i = threadIdx.x; i < NRW * VBN; i += 256) {
      const int c = i / VBN, J = i - c * VBN;
      const zd h = cdiv(buf[c * LS + J], f1[J]);
      buf[c * LS + J] = (J & 1) ? -h : h;
    }
    __syncthreads();
    lds_fft<zd, VBN, NRW, LS, 256, -1>(buf, twg);
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int K = threadIdx.x + 256 * u, J = K + NFIRST;
      // reference output order D0,DXX,DXY,DX,DYY,DY
      auto tap = [&](int c) {
        if (K >= NTAPS) return 0.0;
        double h = buf[c * LS + J].x / (double)VBN;
        if (J & 1) h = -h;
        return h / P.dx / P.dy * rp[half * 3 + c];
      };
      if (half == 0) {
        wt[IE_D0][u] = tap(0);
        wt[IE_DXX][u] = tap(1);
        wt[IE_DXY][u] = tap(2);
      } else {
        wt[IE_DX][u] = tap(0);
        wt[IE_DYY][u] = tap(1);
        wt[IE_DY][u] = tap(2);
      }
    }
  }
  // COMPUTE_WEIGHTS W0 logic (calc_ie_tensor_module.F90:327-351)
  double W0[6];
  auto colmax = [&](int c) { return block_max(fmax(fabs(wt[c][0]), fabs(wt[c][1])), red); };
  W0[IE_DXX] = colmax(IE_DXX);
  if (lx != 0 && ly != 0) {
    double m = fmax(fmax(colmax(IE_DXY), colmax(IE_DYY)), fmax(colmax(IE_DX), colmax(IE_DY)));
    W0[IE_DXY] = W0[IE_DYY] = W0[IE_DX] = W0[IE_DY] = m;
  } else if (lx == 0) {
    W0[IE_DXY] = -W0[IE_DXX];
    W0[IE_DYY] = colmax(IE_DYY);
    W0[IE_DX] = -W0[IE_DXX];
    W0[IE_DY] = (ly != 0) ? colmax(IE_DY) : -W0[IE_DXX];
  } else {
    W0[IE_DXY] = -W0[IE_DXX];
    W0[IE_DYY] = colmax(IE_DYY);
    W0[IE_DX] = colmax(IE_DX);
    W0[IE_DY] = -W0[IE_DXX];
  }
  W0[IE_D0] = colmax(IE_D0);
  const int64_t M = (int64_t)P.Nx * P.Ny;
  __shared__ int kw[2];
  if (threadIdx.x < 2) kw[threadIdx.x] = threadIdx.x == 0 ? NTAPS : 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int K = threadIdx.x + 256 * u;
    if (K >= NTAPS) break;
    double w[6];
    for (int c = 0; c < 6; c++) w[c] = wt[c][u];
    if (lx == 0) {  // :330-342
      w[IE_DXY] = 0;
      w[IE_DX] = 0;
      if (ly == 0) w[IE_DY] = 0;
    } else if (ly == 0) {  // :343-349
      w[IE_DXY] = 0;
      w[IE_DY] = 0;
    }
    double Wm = 0;
    for (int c = 0; c < 6; c++) {
      const double t = fabs(w[c] / W0[c]);
      if (c == 0 || t > Wm) Wm = t;
    }
    const bool on = Wm > 1e-12;
    const double lm = lms[K];
    double o[6];
    o[IE_DXX] = w[IE_DXX] / lm;
    o[IE_DYY] = w[IE_DYY] / lm;
    o[IE_DXY] = w[IE_DXY] / lm;
    o[IE_DX] = w[IE_DX] * lm;
    o[IE_DY] = w[IE_DY] * lm;
    o[IE_D0] = w[IE_D0] * lm;
    for (int c = 0; c < 6; c++) wts[((int64_t)c * NTAPS + K) * M + b] = on ? o[c] : 0.0;
    tap_window(kw, K, on);
  }
  __syncthreads();
  if (threadIdx.x == 0) win[b] = make_int2(kw[0], kw[1]);
}

// ------------------------------------------------------ lambda tables ---
struct LParams {
  int Nl, Nz;
  zd iwm;
  const zd* bk;  // [csigma 0..Nl | k2 0..Nl | (thick, depth) 0..Nl as zd]
};


__device__ inline zd cz2(double a, double b) { return mkz(a, b); }
__device__ inline zd cadd(zd a, double b) { return mkz(a.x + b, a.y); }
__device__ inline zd csqrt_d(zd z) {
  // principal square root
  const double r = hypot(z.x, z.y);
  if (r == 0.0) return mkz(0.0, 0.0);
  double t = sqrt(0.5 * (r + fabs(z.x)));
  if (z.x >= 0.0) return mkz(t, z.y / (2.0 * t));
  return mkz(fabs(z.y) / (2.0 * t), z.y >= 0 ? t : -t);
}
__device__ inline zd cexp_d(zd z) {
  const double e = exp(z.x);
  double s, c;
  sincos(z.y, &s, &c);
  return mkz(e * c, e * s);
}
__device__ inline zd operator/(zd a, zd b) { return cdiv(a, b); }
__device__ inline zd rdiv(double a, zd b) { return cdiv(mkz(a, 0.0), b); }

// Calc_Apq without the A matrix (apq_module.F90:230-249): eta, el, p, q and
// Arr of the layered background for one lambda; arrays indexed by layer
// 1..Nl.  cs, k2: csigma and k^2 (0..Nl); td: (thickness, depth) per layer.
__device__ inline void layer_apq(double lm, int Nl, const zd* sh_cs, const zd* sh_k2, const zd* sh_td,
                                 zd* eta, zd* el, zd (*p)[2], zd (*q)[2], zd (*Arr)[2]) {
  for (int i = 1; i <= Nl; i++) eta[i] = csqrt_d(cz2(lm * lm - sh_k2[i].x, -sh_k2[i].y));
  for (int i = 1; i <= Nl - 1; i++) el[i] = cexp_d(eta[i] * (-2.0 * sh_td[i].x));
  el[Nl] = cz2(0, 0);
  // Calc_p
  {
    zd eta0 = csqrt_d(cz2(lm * lm - sh_k2[0].x, -sh_k2[0].y));
    zd ceta = eta0 / eta[1];
    p[1][0] = cz2(1.0 - ceta.x, -ceta.y) / cadd(ceta, 1.0);
    zd cg = sh_cs[0] / sh_cs[1];
    p[1][1] = (cg - ceta) / (cg + ceta);
    for (int i = 2; i <= Nl; i++) {
      zd a0 = eta[i - 1] / eta[i];
      zd a1 = a0 * sh_cs[i] / sh_cs[i - 1];
      for (int k = 0; k < 2; k++) {
        zd w = el[i - 1] * p[i - 1][k];
        w = cadd(w, -1.0) / cadd(w, 1.0);
        w = w * (k == 0 ? a0 : a1);
        p[i][k] = cadd(w, 1.0) / cz2(1.0 - w.x, -w.y);
      }
    }
  }
  // Calc_q
  {
    q[Nl][0] = q[Nl][1] = cz2(0, 0);
    if (Nl > 1) {
      zd a0 = eta[Nl] / eta[Nl - 1];
      zd a1 = a0 * sh_cs[Nl - 1] / sh_cs[Nl];
      q[Nl - 1][0] = cz2(1.0 - a0.x, -a0.y) / cadd(a0, 1.0);
      q[Nl - 1][1] = cz2(1.0 - a1.x, -a1.y) / cadd(a1, 1.0);
      for (int i = Nl - 2; i >= 1; i--) {
        zd b0 = eta[i + 1] / eta[i];
        zd b1 = b0 * sh_cs[i] / sh_cs[i + 1];
        for (int k = 0; k < 2; k++) {
          zd w = el[i + 1] * q[i + 1][k];
          w = cadd(w, -1.0) / cadd(w, 1.0);
          w = w * (k == 0 ? b0 : b1);
          q[i][k] = cadd(w, 1.0) / cz2(1.0 - w.x, -w.y);
        }
      }
    }
  }
  for (int i = 1; i <= Nl; i++)
    for (int k = 0; k < 2; k++)
      Arr[i][k] = rdiv(1.0, eta[i]) / cz2(1.0 - (p[i][k] * q[i][k] * el[i]).x,
                                           -(p[i][k] * q[i][k] * el[i]).y);
}

// expz per cell, Calc_pexpz_All and Calc_qexpz_All (apq_module.F90:112-177);
// pez, qez at [2*I + k].
__device__ inline void layer_pqexpz(int Nz, int Nl, const int* lnumg, const double* zg,
                                    const double* dzg, const zd* sh_td, const zd* eta,
                                    const zd (*p)[2], const zd (*q)[2], zd* expz, zd* pez, zd* qez) {
  for (int I = 1; I <= Nz; I++) expz[I] = cexp_d(eta[lnumg[I]] * (-dzg[I]));
  // Calc_pexpz_All
  int l = lnumg[0];
  zd e;
  if (l > 1) e = cexp_d(eta[l] * (-2.0 * (zg[0] - sh_td[l - 1].y)));
  else if (l == 1) e = cexp_d(eta[1] * (-2.0 * zg[0]));
  else e = cz2(1, 0);
  for (int I = 1; I <= Nz; I++) {
    if (l != lnumg[I]) e = cz2(1, 0);
    l = lnumg[I];
    pez[2 * I] = e * p[l][0];
    pez[2 * I + 1] = e * p[l][1];
    e = e * expz[I] * expz[I];
  }
  // Calc_qexpz_All
  l = lnumg[Nz];
  if (l != Nl) e = cexp_d(eta[l] * (-2.0 * (sh_td[l].y - zg[Nz])));
  else e = cz2(0, 0);
  for (int I = Nz; I >= 1; I--) {
    if (l != lnumg[I]) e = cz2(1, 0);
    l = lnumg[I];
    qez[2 * I] = e * q[l][0];
    qez[2 * I + 1] = e * q[l][1];
    e = e * expz[I] * expz[I];
  }
}

// tables per tap K: a[P], b[P], c[P] packed upper (i<=j at i + j(j+1)/2), d[Nz*Nz] column-major
__global__ __launch_bounds__(64) void k_lambda(zd* __restrict__ tabs,
                                               const double* __restrict__ lms,
                                               const double* __restrict__ dzg,
                                               const double* __restrict__ zg,
                                               const int* __restrict__ lnumg, LParams L) {
  extern __shared__ unsigned char sm_raw[];
  const int Nz = L.Nz, Nl = L.Nl;
  zd* expz = reinterpret_cast<zd*>(sm_raw);  // 1..Nz
  zd* pez = expz + (Nz + 1);                       // [I][2]
  zd* qez = pez + 2 * (Nz + 1);
  zd* fct = qez + 2 * (Nz + 1);  // fcont_t [I][2]
  zd* tfr = fct + 2 * (Nz + 1);  // t_frame [I][3]
  zd* fcb = tfr + 3 * (Nz + 1);
  zd* bfr = fcb + (Nz + 1);
  zd* Ft = bfr + (Nz + 1);  // [I][3]
  zd* Fb = Ft + 3 * (Nz + 1);
  zd* GII = Fb + (Nz + 1);  // [I][4]
  __shared__ zd eta[65], p[65][2], q[65][2], Arr[65][2];
  __shared__ zd sh_cs[65], sh_k2[65], sh_td[65];
  for (int i = threadIdx.x; i <= Nl; i += blockDim.x) {
    sh_cs[i] = L.bk[i];
    sh_k2[i] = L.bk[Nl + 1 + i];
    sh_td[i] = L.bk[2 * (Nl + 1) + i];
  }
  __syncthreads();
  const int K = blockIdx.x;
  const double lm = lms[K];
  const int P = Nz * (Nz + 1) / 2;
  zd* ta = tabs + (int64_t)K * (3 * P + Nz * Nz);
  zd* tb = ta + P;
  zd* tc = tb + P;
  zd* td = tc + P;
  __shared__ zd el[65];  // thread 0 only (a private array would live in scratch)
  if (threadIdx.x == 0) {
    layer_apq(lm, Nl, sh_cs, sh_k2, sh_td, eta, el, p, q, Arr);
    layer_pqexpz(Nz, Nl, lnumg, zg, dzg, sh_td, eta, p, q, expz, pez, qez);
  }
  __syncthreads();
  for (int I = 1 + threadIdx.x; I <= Nz; I += blockDim.x) {
    const int l = lnumg[I];
    const zd ez = expz[I], et = eta[l], sg = sh_cs[l];
    if (I <= Nz - 1) {  // Calc_tframe_p (apq_module.F90:83-110)
      zd a[2], bb[2], c[2];
      for (int k = 0; k < 2; k++) {
        a[k] = pez[2 * I + k];
        bb[k] = a[k] * ez;
        c[k] = bb[k] * ez;
        a[k] = cadd(a[k], 1.0);
        bb[k] = cadd(bb[k], 1.0);
        c[k] = cadd(c[k], 1.0);
      }
      const zd w = cz2(1.0 - ez.x, -ez.y) / et;
      for (int k = 0; k < 2; k++) fct[2 * I + k] = ez * a[k] / c[k];
      tfr[3 * I + 0] = w * bb[0] / c[0];
      tfr[3 * I + 1] = cz2(1.0 - fct[2 * I + 1].x, -fct[2 * I + 1].y) / sg;
      tfr[3 * I + 2] = (w * bb[1] / c[1]) / sg;
    }
    if (I >= 2) {  // Calc_bframe_q (138-153)
      zd a = qez[2 * I + 1];
      const zd d = cadd(a * ez * ez, 1.0);
      a = cadd(a, 1.0);
      fcb[I] = ez * a / d;
      bfr[I] = cadd(fcb[I], -1.0) / sg;
    }
    // Calc_FtFb (31-79)
    zd a[2], a1[2], a2[2], p1[2], p2[2], pe1[2], pe2[2], q1[2], q2[2], qe1[2], qe2[2], Fb3[3],
        w[2];
    for (int k = 0; k < 2; k++) {
      a[k] = cz2(1.0 - ez.x, -ez.y) * Arr[l][k];
      a1[k] = a[k] / et;
      a2[k] = a1[k] / et;
      const zd pz = pez[2 * I + k], qz = qez[2 * I + k];
      p1[k] = cadd(pz, 1.0);
      p2[k] = cz2(1.0 - pz.x, -pz.y);
      pe1[k] = cadd(pz * ez, 1.0);
      pe2[k] = cadd(pz * ez, -1.0);
      q1[k] = cadd(qz, 1.0);
      q2[k] = cz2(1.0 - qz.x, -qz.y);
      qe1[k] = cadd(qz * ez, 1.0);
      qe2[k] = cz2(1.0 - (qz * ez).x, -(qz * ez).y);
    }
    const zd eta2 = et * et;
    for (int k = 0; k < 2; k++) {
      Ft[3 * I + k] = a1[k] * p1[k] * qe1[k];
      Fb3[k] = a1[k] * pe1[k] * q1[k];
      w[k] = -(a2[k] * (p2[k] * qe1[k] + pe1[k] * q2[k]));
    }
    Ft[3 * I + 2] = a[1] * p1[1] * qe2[1];
    Fb3[2] = a[1] * pe2[1] * q1[1];
    const zd dzt = rdiv(2.0, eta2) * dzg[I];
    GII[4 * I + 0] = w[0] + dzt;
    GII[4 * I + 1] = Fb3[1] - Ft[3 * I + 1];
    GII[4 * I + 2] = (w[1] + dzt) * L.iwm + eta2 / sg * w[1];
    GII[4 * I + 3] = Fb3[2] - Ft[3 * I + 2] - eta2 * w[0];
    Fb[I] = Fb3[1];
  }
  __syncthreads();
  // tables: one thread per source layer Izs (column)
  const double lm2 = lm * lm;
  for (int Izs = 1 + threadIdx.x; Izs <= Nz; Izs += blockDim.x) {
    const int js = Izs - 1;
    const zd sg = sh_cs[lnumg[Izs]];
    const zd* g4 = GII + 4 * Izs;
    const int dia = js + js * (js + 1) / 2;
    ta[dia] = (g4[0] * lm2 + g4[3]) / sg;  // coefficient of W_DXX (diag, :89-103)
    tb[dia] = g4[0] * L.iwm;               // coefficient of W_D0
    tc[dia] = g4[2];                       // EZZ
    td[js + Nz * js] = g4[1] / sg;         // EXZ/EYZ
    // GoByShellsU (ie_kernel_hankel_module.F90:125-173)
    zd u1 = Ft[3 * Izs + 0] * L.iwm, u2 = Ft[3 * Izs + 1], u3 = Ft[3 * Izs + 2];
    for (int Izr = Izs - 1; Izr >= 1; Izr--) {
      const int ir = Izr - 1, pi = ir + js * (js + 1) / 2;
      const zd* fr = tfr + 3 * Izr;
      const zd t1 = u1 * fr[0];
      ta[pi] = t1 + u3 * fr[1];
      tb[pi] = t1;
      tc[pi] = (u2 * lm2) * fr[2];
      td[ir + Nz * js] = u2 * fr[1];
      u1 = u1 * fct[2 * Izr];
      u2 = u2 * fct[2 * Izr + 1];
      u3 = u3 * fct[2 * Izr + 1];
    }
    // GoByShellsL (175-197)
    zd v = Fb[Izs];
    for (int Izr = Izs + 1; Izr <= Nz; Izr++) {
      td[(Izr - 1) + Nz * js] = v * bfr[Izr];
      v = v * fcb[Izr];
    }
  }
}

// --------------------------------------------------------- weighted sum ---
// C[o][coff + e] = scale * sum_seg sum_K A_seg[K][o] * B_seg[K][e] for every
// offset o and entry e (A real weights, B complex tables): FP64 matrix
// products (offsets x taps) (taps x 2 entries) on v_mfma_f64_16x16x4, all
// jobs (tensor components) of a build in one launch.  A large FP64 product
// reaches 71 TFLOP/s on this card; the tiles here, with a barrier per 8 taps,
// 42 to 59.  Three things keep the work below the (offsets x 501 x entries)
// of the plain sum:
//   - the taps: a block sums the window in which one of its offsets has a
//     weight (the 1e-12 mask of the weights leaves 210 to 370 of 501 taps);
//   - the x-y mirror (TRI): on a square grid with dx = dy the block at
//     (ly,lx) is that at (lx,ly) with x and y exchanged, so offsets lx >= ly
//     are summed and stored in both places (coff2: the exchanged component);
//   - a tile is 128 offsets x 32 complex entries, double-buffered in LDS by
//     chunks of 8 taps, so that the loads of a chunk run beside the matrix
//     products of the one before.
// Measured (128x128x32): six launches on the vector unit, every tap and offset,
// 4830 us (35 TFLOP/s) -> 980 to 1080 us (46 to 42 TFLOP/s of the sums that are
// left); with two receivers, thirty launches 5930 us (27 TFLOP/s) -> 1400 us
// (59 TFLOP/s).
struct WJob {
  int coff, coff2, Ne, nseg;  // coff or coff2 < 0: not stored there
  const double *A0, *A1;  // [K][lda]
  const zd *B0, *B1;      // [K][ldb], entry e at B[K*ldb + e]
};
struct WJobs {
  int n;
  WJob j[15];
};
typedef double f64x4 __attribute__((ext_vector_type(4)));

// (at least three waves per SIMD asked for: below two the compiler keeps the
// accumulators in the second register file and copies them every chunk)
template <bool TRI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_wgemm(zd* __restrict__ C, int64_t rows, int64_t lda, int64_t BS, int64_t ldb,
                                               const int2* __restrict__ win, int Nx, double scale, WJobs jobs) {
  constexpr int TM = 128, TE = 32, TK = 8, LA = TM + 16, LB = 2 * TE + 16;
  __shared__ double As[2][TK][LA];
  __shared__ __align__(16) double Bs[2][TK][LB];
  __shared__ int64_t mo[TM], mt[TM];
  __shared__ int kw[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, kq = lane >> 4;
  // job and entry tile of this block
  int jt = blockIdx.y, ji = 0;
  while (jt >= (jobs.j[ji].Ne + TE - 1) / TE) {
    jt -= (jobs.j[ji].Ne + TE - 1) / TE;
    ji++;
  }
  const WJob job = jobs.j[ji];
  const int n0 = jt * TE;
  if (tid < 2) kw[tid] = tid == 0 ? NTAPS : 0;
  __syncthreads();
  if (tid < TM) {
    const int64_t t = (int64_t)blockIdx.x * TM + tid;
    int64_t o = -1, ot = -1;
    if (t < rows) {
      if constexpr (TRI) {
        // rows ly = r (lx = r .. Nx-1) and ly = Nx-1-r together have Nx+1 offsets
        const int r = (int)(t / (Nx + 1)), c = (int)(t - (int64_t)r * (Nx + 1));
        const int ly = c < Nx - r ? r : Nx - 1 - r, lx = c < Nx - r ? r + c : c - 1;
        o = lx + (int64_t)Nx * ly;
        if (lx != ly) ot = ly + (int64_t)Nx * lx;
      } else {
        o = t;
      }
      const int2 w = win[o];
      atomicMin(&kw[0], w.x);
      atomicMax(&kw[1], w.y);
    }
    mo[tid] = o;
    mt[tid] = ot;
  }
  __syncthreads();
  const int klo = kw[0], khi = kw[1];
  const int nch = khi > klo ? (khi - klo + TK - 1) / TK : 0, nct = nch * job.nseg;
  // loads: offset tid % 128 of taps tid / 128 + 2 i; entry tid % 32 of tap tid / 32
  const int am = tid & (TM - 1), ak = tid >> 7, bn = tid & (TE - 1), bk = tid >> 5;
  // (rows and entries past the end read the first ones and are not stored;
  // taps past the window count as zero weights.  No branch: with one per load
  // or chunk the compiler moved the accumulators between register files in
  // every chunk, 1180 us against 980)
  const int64_t ao = mo[am] < 0 ? 0 : mo[am];
  const int bo = n0 + bn < job.Ne ? n0 + bn : n0;
  double ra[4];
  zd rb;
  auto load = [&](int c) {
    const bool second = c >= nch;
    const int k0 = klo + (second ? c - nch : c) * TK;
    const double* A = second ? job.A1 : job.A0;
    const zd* B = second ? job.B1 : job.B0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int K = k0 + ak + 2 * i;
      const double v = A[(int64_t)min(K, NTAPS - 1) * lda + ao];
      ra[i] = K < khi ? v : 0.0;
    }
    rb = B[(int64_t)min(k0 + bk, NTAPS - 1) * ldb + bo];
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; i++) As[buf][ak + 2 * i][am] = ra[i];
    *reinterpret_cast<zd*>(&Bs[buf][bk][2 * bn]) = rb;
  };
  f64x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = f64x4{0, 0, 0, 0};
  if (nct > 0) {
    load(0);
    stash(0);
    __syncthreads();
    for (int c = 0; c < nct; c++) {
      const int buf = c & 1;
      load(min(c + 1, nct - 1));
#pragma unroll
      for (int s = 0; s < TK / 4; s++) {
        double a[2], b[4];
#pragma unroll
        for (int i = 0; i < 2; i++) a[i] = As[buf][s * 4 + kq][wave * 32 + i * 16 + col];
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = Bs[buf][s * 4 + kq][j * 16 + col];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      stash(buf ^ 1);
      __syncthreads();
    }
  }
  // lane (col, kq) holds real column 16 j + col of offsets 16 i + kq + 4 q
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = wave * 32 + i * 16 + kq + 4 * q;
      if (mo[r] < 0) continue;
      double* d0 = !TRI || job.coff >= 0 ? reinterpret_cast<double*>(C + mo[r] * BS + job.coff + n0) + col : nullptr;
      double* d1 =
          TRI && job.coff2 >= 0 && mt[r] >= 0 ? reinterpret_cast<double*>(C + mt[r] * BS + job.coff2 + n0) + col : nullptr;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (n0 + j * 8 + (col >> 1) >= job.Ne) continue;
        const double v = acc[i][j][q] * scale;
        if (!TRI || d0) d0[j * 16] = v;
        if (TRI && d1) d1[j * 16] = v;
      }
    }
}
static dim3 wgemm_grid(int64_t rows, const WJobs& w) {
  unsigned nt = 0;
  for (int i = 0; i < w.n; i++) nt += (unsigned)((w.j[i].Ne + 31) / 32);
  return dim3((unsigned)((rows + 127) / 128), nt);
}

// ------------------------------------------------------------ tensor FFT ---
__device__ inline void entry_signs(int Nz, int64_t e, double* sx, double* sy) {
  const int64_t P = (int64_t)Nz * (Nz + 1) / 2;
  if (e < P) { *sx = 1; *sy = 1; }
  else if (e < 2 * P) { *sx = -1; *sy = -1; }
  else if (e < 4 * P) { *sx = 1; *sy = 1; }
  else if (e < 4 * P + (int64_t)Nz * Nz) { *sx = -1; *sy = 1; }
  else { *sx = 1; *sy = -1; }
}

template <int L> constexpr int ne_for() { return L <= 64 ? 32 : (L <= 128 ? 16 : (L <= 512 ? 8 : 4)); }

// AXIS 0: transform along y for a fixed lx (blockIdx.x); AXIS 1: along x for fixed ky.
// L is the buffer capacity; with RT the transform length is plan.L <= L.
// MIR (the half tensor of op_build_tensor): yy and yz are xx and xz with the
// axes exchanged, so only xx, xy, zz and xz are read and transformed, and the
// second pass stores xx and xz of (kx,ky) also as yy and yz of (ky,kx): 0.72
// of the bytes.  HBM bound (128x128x32: 1180 -> 790 to 830 us for the two passes,
// 4.0 to 3.8 TB/s).
template <int L, int AXIS, bool RT, bool MIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RT ? 2 : 1))) void k_tfft(zd* __restrict__ G, const zd* __restrict__ twg,
                                              int Nx, int Ny, int Nz, int64_t BS, FftPlan plan) {
  constexpr int NE = ne_for<L>(), LS = L + 1, NT = 256;
  __shared__ zd buf[NE * LS];
  __shared__ zd tw[L];
  const int Lr = RT ? plan.L : L;
  const int N = Lr / 2;  // Ny (AXIS 0) or Nx (AXIS 1)
  const int fixed = blockIdx.x;
  const int64_t e0 = (int64_t)blockIdx.y * NE;
  const int64_t P = (int64_t)Nz * (Nz + 1) / 2, NN = (int64_t)Nz * Nz, ne = MIR ? 3 * P + NN : BS;
  for (int i = threadIdx.x; i < Lr; i += NT) tw[i] = twg[i];
  auto gidx = [&](int l) -> int64_t {
    return AXIS == 0 ? ((int64_t)fixed + (int64_t)Nx * l) * BS : ((int64_t)l + (int64_t)Nx * fixed) * BS;
  };
  auto entry = [&](int64_t e) -> int64_t { return MIR && e >= 2 * P ? e + P : e; };
  for (int i = threadIdx.x; i < NE * N; i += NT) {
    const int l = i / NE, s = i - l * NE;
    zd g = mkz(0, 0);
    double sx = 1, sy = 1;
    if (e0 + s < ne) {
      const int64_t e = entry(e0 + s);
      g = G[gidx(l) + e];
      entry_signs(Nz, e, &sx, &sy);
    }
    const double sgn = AXIS == 0 ? sy : sx;
    buf[s * LS + l] = g;
    if (l > 0) buf[s * LS + Lr - l] = g * sgn;
    else buf[s * LS + N] = mkz(0, 0);
  }
  __syncthreads();
  lds_fft_any<zd, L, NE, LS, NT, -1, RT>(buf, tw, plan);
  for (int i = threadIdx.x; i < NE * N; i += NT) {
    const int k = i / NE, s = i - k * NE;
    if (e0 + s < ne) {
      const int64_t e = entry(e0 + s);
      const zd t = buf[s * LS + N];
      const double sg = (k & 1) ? -1.0 : 1.0;
      const zd r = buf[s * LS + k] - t * sg;
      G[gidx(k) + e] = r;
      if constexpr (MIR && AXIS == 1) {
        if (e < P) G[((int64_t)fixed + (int64_t)Nx * k) * BS + e + 2 * P] = r;
        else if (e >= 4 * P) G[((int64_t)fixed + (int64_t)Nx * k) * BS + e + NN] = r;
      }
    }
  }
}

static void make_tw64(int L, zd** d) {
  std::vector<zd> h(L);
  for (int t = 0; t < L; t++) {
    long double a = -2.0L * 3.14159265358979323846264338327950288L * t / L;
    h[t] = mkz((double)cosl(a), (double)sinl(a));
  }
  G2G_HIP(hipMalloc(d, sizeof(zd) * L));
  G2G_HIP(hipMemcpy(*d, h.data(), sizeof(zd) * L, hipMemcpyHostToDevice));
}

void op_tensor_fft(Operator& op, zd* G, bool mir) {
  const int Nx2 = 2 * op.Nx, Ny2 = 2 * op.Ny;
  const zd *twx = op.d64.twx, *twy = op.d64.twy;
  const FftPlan &py = op.py, &px = op.px;
  const int64_t P = (int64_t)op.Nz * (op.Nz + 1) / 2, ne = mir ? 3 * P + (int64_t)op.Nz * op.Nz : op.BS;
  auto pass = [&](auto LC, auto AX, auto MR, const zd* tw, const FftPlan& plan) {
    constexpr int LL = decltype(LC)::value, axis = decltype(AX)::value;
    constexpr int NE = ne_for<LL>();
    hipLaunchKernelGGL((k_tfft<LL, axis, decltype(LC)::rt, decltype(MR)::value>),
                       dim3(axis == 0 ? op.Nx : op.Ny, (unsigned)((ne + NE - 1) / NE)), dim3(256), 0, op.stream, G, tw,
                       op.Nx, op.Ny, op.Nz, op.BS, plan);
  };
  using std::integral_constant;
  len_dispatch(Ny2, [&](auto LC) {
    if (mir) pass(LC, integral_constant<int, 0>{}, std::true_type{}, twy, py);
    else pass(LC, integral_constant<int, 0>{}, std::false_type{}, twy, py);
  });
  len_dispatch(Nx2, [&](auto LC) {
    if (mir) pass(LC, integral_constant<int, 1>{}, std::true_type{}, twx, px);
    else pass(LC, integral_constant<int, 1>{}, std::false_type{}, twx, px);
  });
  G2G_HIP(hipGetLastError());
}

void op_free_tensor_scratch(Operator& op) {
  op.par.release();
  op.spar.release();
  if (op.wts) (void)hipFree(op.wts);
  if (op.tabs) (void)hipFree(op.tabs);
  op.wts = nullptr;
  op.tabs = nullptr;
  op.have_wts = false;
}

// Tables of a tensor build on the device: the taps' lambda, layer thicknesses
// (1-based), borders, layer numbers and the background's arrays
struct BuildTables {
  const double *lms, *dz, *z;
  const int* ln;
  const zd* bk;  // sigma, i sigma mu0 w, (thickness, depth): Nl + 1 each
  double mw;
};
static BuildTables build_tables(const Operator& op, DevTables& t, double rmin) {
  const int Nz = op.Nz;
  std::vector<double> lms(NTAPS), dz1(Nz + 1, 0.0);
  for (int j = 0; j < NTAPS; j++) lms[j] = std::exp(VB_XI + (double)(j + NFIRST - 512) * VB_YSTEP) / rmin;
  for (int i = 1; i <= Nz; i++) dz1[i] = op.dz[i - 1];
  const double mw = 4.0 * PI_D * 1e-7 * op.omega;
  std::vector<zd> bk(3 * (op.Nl + 1), mkz(0, 0));
  for (int i = 0; i <= op.Nl; i++) {
    bk[i] = op.csigma[i];
    bk[op.Nl + 1 + i] = mkz(-op.csigma[i].y * mw, op.csigma[i].x * mw);  // i*sigma*mu0*w
  }
  {
    double depth = 0;
    for (int i = 1; i <= op.Nl - 1; i++) {
      depth += op.thick[i];
      bk[2 * (op.Nl + 1) + i] = mkz(op.thick[i], depth);
    }
  }
  t.h.clear();
  const size_t o0 = t.add(lms.data(), NTAPS), o1 = t.add(dz1.data(), Nz + 1), o2 = t.add(op.z.data(), Nz + 1),
               o3 = t.add(op.lnum.data(), Nz + 1), o4 = t.add(bk.data(), bk.size());
  t.send();
  return {t.at<double>(o0), t.at<double>(o1), t.at<double>(o2), t.at<int>(o3), t.at<zd>(o4), mw};
}

void op_build_tensor(Operator& op, bool half) {
  G2G_CHECK(op.have_bkg, -4, "background not set");
  G2G_CHECK(op.Nl <= 64 && op.Nz <= MAX_NZ, -3, "tensor build supports Nl <= 64 and Nz <= 256");
  const int64_t M = (int64_t)op.Nx * op.Ny;
  const int Nz = op.Nz, P = Nz * (Nz + 1) / 2;
  const double rmin = std::sqrt(op.dx * op.dx + op.dy * op.dy) / 2.0;  // :102
  const BuildTables bt = build_tables(op, op.par, rmin);
  G2G_HIP(hipEventRecord(op.ev[0], op.stream));
  if (!op.have_wts) {
    zd *tw, *f1;
    make_tw64(VBN, &tw);
    G2G_HIP(hipMalloc(&f1, sizeof(zd) * VBN));
    // the weights, then every offset's window of taps
    if (!op.wts) G2G_HIP(hipMalloc(&op.wts, sizeof(double) * 6 * NTAPS * M + sizeof(int2) * M));
    hipLaunchKernelGGL(k_f1, dim3(1), dim3(256), 0, op.stream, f1, tw);
    WParams wp{op.Nx, op.Ny, op.dx, op.dy, rmin, std::log(rmin)};
    hipLaunchKernelGGL(k_weights, dim3((unsigned)M), dim3(256), 0, op.stream, op.wts,
                       (int2*)(op.wts + 6 * NTAPS * M), f1, tw, bt.lms, wp);
    G2G_HIP(hipGetLastError());
    G2G_HIP(hipStreamSynchronize(op.stream));
    (void)hipFree(tw);
    (void)hipFree(f1);
    op.have_wts = true;
  }
  // lambda tables
  LParams lp;
  lp.Nl = op.Nl;
  lp.Nz = Nz;
  lp.iwm = mkz(0.0, bt.mw);
  lp.bk = bt.bk;
  const size_t tab_n = (size_t)NTAPS * (3 * P + Nz * Nz);
  if (!op.tabs || op.tabs_bytes < tab_n * sizeof(zd)) {
    if (op.tabs) (void)hipFree(op.tabs);
    G2G_HIP(hipMalloc(&op.tabs, tab_n * sizeof(zd)));
    op.tabs_bytes = tab_n * sizeof(zd);
  }
  const size_t sm = sizeof(zd) * (size_t)(Nz + 1) * 20;
  if (sm > 65536)
    G2G_HIP(hipFuncSetAttribute((const void*)k_lambda, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm));
  hipLaunchKernelGGL(k_lambda, dim3(NTAPS), dim3(64), sm, op.stream, (zd*)op.tabs, bt.lms, bt.dz,
                     bt.z, bt.ln, lp);
  G2G_HIP(hipGetLastError());
  // weighted sums into the real-space tensor (stored in d64.G), x 1/(4 pi)
  const zd* T = (const zd*)op.tabs;
  const int64_t ldb = 3 * P + (int64_t)Nz * Nz;
  const double* W = op.wts;
  auto Wc = [&](int c) { return W + (int64_t)c * NTAPS * M; };
  const double scale = 1.0 / PI_D / 4.0;
  const int NN = Nz * Nz, xz = 4 * P, yz = 4 * P + NN;
  // half: only xx, xy, zz and xz, summed for the offsets lx >= ly and stored
  // at both places of the x-y mirror (the sums of yy and yz at (lx,ly) are xx
  // and xz at (ly,lx)).  The weights' mask is not symmetric in x and y: at 28%
  // of the offsets lx < ly (34x34) it keeps other taps than at the mirrored one,
  // most often one more or less at its threshold, so these blocks differ from
  // sums of their own by up to 1.2e2 eps of their weight-error scale.  Against sums of
  // extended-precision weights with taps down to 1e-15 they are no further off:
  // mean error of the blocks lx < ly 21 eps of that scale against 23 (34x34x6),
  // 24 against 27 (64x64x2)
  const WJobs jobs = {6,
                      {{0, -1, P, 2, Wc(IE_DXX), Wc(IE_D0), T, T + P},
                       {P, P, P, 1, Wc(IE_DXY), nullptr, T, nullptr},
                       {half ? -1 : 2 * P, 0, P, 2, Wc(IE_DYY), Wc(IE_D0), T, T + P},
                       {3 * P, 3 * P, P, 1, Wc(IE_D0), nullptr, T + 2 * P, nullptr},
                       {xz, -1, NN, 1, Wc(IE_DX), nullptr, T + 3 * P, nullptr},
                       {half ? -1 : yz, xz, NN, 1, Wc(IE_DY), nullptr, T + 3 * P, nullptr}}};
  const int2* win = (const int2*)(W + 6 * NTAPS * M);
  if (half) {
    const int64_t rows = (int64_t)op.Nx * (op.Nx + 1) / 2;
    hipLaunchKernelGGL(k_wgemm<true>, wgemm_grid(rows, jobs), dim3(256), 0, op.stream, op.d64.G, rows, M, op.BS, ldb, win,
                       op.Nx, scale, jobs);
  } else {
    hipLaunchKernelGGL(k_wgemm<false>, wgemm_grid(M, jobs), dim3(256), 0, op.stream, op.d64.G, M, M, op.BS, ldb, win,
                       op.Nx, scale, jobs);
  }
  G2G_HIP(hipGetLastError());
  G2G_HIP(hipEventRecord(op.ev[1], op.stream));
}

// ====================================================================== //
// Receiver continuation tensor (CalcRecalculationGreenTensor,              //
// calc_rc_tensor_module.F90:37-230, with VBTransformWeightsAllSingleInt,   //
// VolumeBesselTransforms.F90:198-229, and Calc_Integral_U,                 //
// rc_kernel_hankel_module.F90:56-254).  The same factorisation as above:   //
// per-(offset, receiver) weights, per-(tap, receiver) weight-free tables   //
// of the 13 kernel functions of (lambda, z), and their weighted tap sums   //
// on k_wgemm.  Then the full 2-D FFT of every tensor column               //
// (CalcFFTofRCTensor, Continuation_Function_Module.F90:349-383).          //
// ====================================================================== //

// outfunc_int2_all for one knot (VolumeBesselTransforms.F90:342-371, 407-434, 553-603)
__device__ inline void outfunc2(double explt, double cphi, double sphi, double alpha, double beta,
                                double* R) {
  double f[2][3][3];  // [x/y][D0,D1,D2][1..3]
#pragma unroll
  for (int J = 0; J < 2; J++) {
    const double c = J == 0 ? cphi : sphi, h = J == 0 ? alpha : beta;
    double x[2], x2[2], ex[2], er[2], t[2];
    x[0] = explt * c * 0.5;
    x[1] = x[0] + h * explt * 0.5;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      x2[k] = x[k] * x[k];
      ex[k] = exp(-x2[k]);
      er[k] = erf(x[k]);
    }
    // SINGLE_INT_D0
    const double a0 = er[1] * sqrt(PI_D) - er[0] * sqrt(PI_D);
    for (int k = 0; k < 2; k++) t[k] = x[k] * ex[k];
    double b = t[1] - t[0];
    for (int k = 0; k < 2; k++) t[k] = t[k] * x2[k];
    double cc = t[1] - t[0];
    f[J][0][0] = a0 * 0.5;
    f[J][0][1] = a0 - 2.0 * b;
    f[J][0][2] = 6.0 * a0 - 12.0 * b - 8.0 * cc;
    // SINGLE_INT_D1
    for (int k = 0; k < 2; k++) t[k] = ex[k];
    f[J][1][0] = (t[1] - t[0]) / 2.0;
    for (int k = 0; k < 2; k++) t[k] = t[k] * x2[k];
    f[J][1][1] = (t[1] - t[0]) * 2.0;
    for (int k = 0; k < 2; k++) t[k] = t[k] * x2[k];
    f[J][1][2] = (t[1] - t[0]) * 8.0;
    // SINGLE_INT_D2
    for (int k = 0; k < 2; k++) t[k] = x[k] * ex[k];
    const double a2 = t[1] - t[0];
    for (int k = 0; k < 2; k++) t[k] = t[k] * x2[k];
    b = t[1] - t[0];
    for (int k = 0; k < 2; k++) t[k] = t[k] * x2[k];
    cc = t[1] - t[0];
    f[J][2][0] = -a2 * 0.5;
    f[J][2][1] = 2.0 * (a2 - b);
    f[J][2][2] = 16.0 * b - 8.0 * cc;
  }
#define CMB(a, b) (f[0][a][2] * f[1][b][0] + f[0][a][0] * f[1][b][2] + 2.0 * f[0][a][1] * f[1][b][1])
  R[0] = CMB(0, 0) / explt;
  R[1] = CMB(2, 0) * explt;
  R[2] = CMB(1, 1) * explt;
  R[3] = CMB(1, 0);
  R[4] = CMB(0, 2) * explt;
  R[5] = CMB(0, 1);
#undef CMB
}

struct RcWParams {
  int Nx, Ny;
  double dx, dy, xs, ys, log_rmin;
};

// One block per offset point p = ix*2Ny + iy of one receiver.  Output
// wts[c][K][p] in IE order, masked (1e-12 of the largest weight of the
// offset, calc_rc_tensor_module.F90:202-212) and lambda-scaled (:214-219);
// zero on the ix = Nx and iy = Ny offsets.  LDS and registers as in k_weights
// (65536 offsets: 12.1 -> 7.1 ms).
__global__ __launch_bounds__(256) void k_rc_weights(double* __restrict__ wts, int2* __restrict__ win,
                                                    const zd* __restrict__ f1,
                                                    const zd* __restrict__ twg,
                                                    const double* __restrict__ lms, RcWParams P) {
  constexpr int NRW = 3, LS = VBN + 1;
  __shared__ zd buf[NRW * LS];
  double wt[6][2];
  __shared__ double red[8];
  const int Ny2 = 2 * P.Ny;
  const int64_t NP = (int64_t)4 * P.Nx * P.Ny;
  const int p = blockIdx.x, ix = p / Ny2, iy = p - ix * Ny2;
  if (ix == P.Nx || iy == P.Ny) {
    for (int i = threadIdx.x; i < 6 * NTAPS; i += 256) wts[(int64_t)i * NP + p] = 0.0;
    if (threadIdx.x == 0) win[p] = make_int2(NTAPS, 0);
    return;
  }
  const int lx = ix < P.Nx ? ix : ix - 2 * P.Nx, ly = iy < P.Ny ? iy : iy - Ny2;
  const double x = lx * P.dx - P.dx / 2.0 + P.xs, y = ly * P.dy - P.dy / 2.0 + P.ys;
  const double rho = sqrt(x * x + y * y);
  const double alpha = P.dx / rho, beta = P.dy / rho, phi = atan2(y, x);
  const double cphi = cos(phi), sphi = sin(phi);
  const double s = log(rho) - P.log_rmin;
  for (int half = 0; half < 2; half++) {
    __syncthreads();
    for (int i = threadIdx.x; i < VBN; i += 256) {
      const int i0 = i & ~1;
      double y2 = (double)(i0 - 512) * VB_YSTEP + VB_P + s;
      if (i & 1) y2 = y2 + VB_YSTEP;
      const double explt = exp(y2);
      double R[6];
      outfunc2(explt, cphi, sphi, alpha, beta, R);
      const double sg = (i & 1) ? -1.0 : 1.0;
      for (int c = 0; c < NRW; c++) buf[c * LS + i] = mkz(sg * R[half * 3 + c], 0.0);
    }
    __syncthreads();
    lds_fft<zd, VBN, NRW, LS, 256, +1>(buf, twg);
    for (int i = threadIdx.x; i < NRW * VBN; i += 256) {
      const int c = i / VBN, J = i - c * VBN;
      const zd h = cdiv(buf[c * LS + J], f1[J]);
      buf[c * LS + J] = (J & 1) ? -h : h;
    }
    __syncthreads();
    lds_fft<zd, VBN, NRW, LS, 256, -1>(buf, twg);
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int K = threadIdx.x + 256 * u, J = K + NFIRST;
      auto tap = [&](int c) {
        if (K >= NTAPS) return 0.0;
        double h = buf[c * LS + J].x / (double)VBN;
        return (J & 1) ? -h : h;
      };
      // reference output order D0,DXX,DXY,DX,DYY,DY; scalings of
      // VolumeBesselTransforms.F90:222-228
      if (half == 0) {
        wt[IE_D0][u] = tap(0) * rho;
        wt[IE_DXX][u] = tap(1) / rho;
        wt[IE_DXY][u] = tap(2) / rho;
      } else {
        wt[IE_DX][u] = tap(0);
        wt[IE_DYY][u] = tap(1) / rho;
        wt[IE_DY][u] = tap(2);
      }
    }
  }
  double m = 0;
#pragma unroll
  for (int c = 0; c < 6; c++) m = fmax(m, fmax(fabs(wt[c][0]), fabs(wt[c][1])));
  const double W0 = block_max(m, red);
  __shared__ int kw[2];
  if (threadIdx.x < 2) kw[threadIdx.x] = threadIdx.x == 0 ? NTAPS : 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int K = threadIdx.x + 256 * u;
    if (K >= NTAPS) break;
    double Wm = 0;
    for (int c = 0; c < 6; c++) Wm = fmax(Wm, fabs(wt[c][u] / W0));
    const bool on = Wm > 1e-12;
    const double lm = lms[K];
    double o[6];
    o[IE_DXX] = wt[IE_DXX][u] / lm;
    o[IE_DYY] = wt[IE_DYY][u] / lm;
    o[IE_DXY] = wt[IE_DXY][u] / lm;
    o[IE_DX] = wt[IE_DX][u] * lm;
    o[IE_DY] = wt[IE_DY][u] * lm;
    o[IE_D0] = wt[IE_D0][u] * lm;
    for (int c = 0; c < 6; c++) wts[((int64_t)c * NTAPS + K) * NP + p] = on ? o[c] : 0.0;
    tap_window(kw, K, on);
  }
  __syncthreads();
  if (threadIdx.x == 0) win[p] = make_int2(kw[0], kw[1]);
}

// kernel functions of one receiver per tap, table [K][f][z]
enum { RF_G11 = 0, RF_G3DZ_G11, RF_G2DZ, RF_G2DZ0, RF_G2G2DZZ, RF_G3, RF_G1DZ, RF_G2, RF_G1,
       RF_NG1DZ, RF_NG3, RF_NG2, RF_NG1, RF_COUNT };

struct RcLParams {
  int Nl, Nz, rl, cell;
  double zr;
  zd iwm;
  const zd* bk;  // [csigma 0..Nl | k2 0..Nl | (thick, depth) 0..Nl]
};

// One block per tap K: Calc_Apq with the receiver row of A, Calc_Recv_Part,
// Calc_Ftb and Calc_G_not_match for every source layer (one lane each).
__global__ __launch_bounds__(64) void k_rc_lambda(zd* __restrict__ tabs,
                                                  const double* __restrict__ lms,
                                                  const double* __restrict__ dzg,
                                                  const double* __restrict__ zg,
                                                  const int* __restrict__ lnumg, RcLParams L) {
  const int Nz = L.Nz, Nl = L.Nl, rl = L.rl, N = L.cell;
  __shared__ zd eta[65], p[65][2], q[65][2], Arr[65][2], wlay[65][2], Arl[65][2];
  __shared__ zd sh_cs[65], sh_k2[65], sh_td[65];
  __shared__ zd expz[MAX_NZ + 1], pez[2 * (MAX_NZ + 1)], qez[2 * (MAX_NZ + 1)];
  for (int i = threadIdx.x; i <= Nl; i += blockDim.x) {
    sh_cs[i] = L.bk[i];
    sh_k2[i] = L.bk[Nl + 1 + i];
    sh_td[i] = L.bk[2 * (Nl + 1) + i];
  }
  __syncthreads();
  const int K = blockIdx.x;
  const double lm = lms[K];
  __shared__ zd el[65];  // thread 0 only (a private array would live in scratch)
  if (threadIdx.x == 0) {
    layer_apq(lm, Nl, sh_cs, sh_k2, sh_td, eta, el, p, q, Arr);
    // the receiver row A(rl, l) of the layer-coupling matrix (apq_module.F90:250-264)
    for (int i = 1; i <= Nl - 1; i++) {
      zd tmp = sh_k2[i] - sh_k2[i + 1];
      tmp = tmp * sh_td[i].y;
      tmp = tmp / (eta[i + 1] + eta[i]);
      const zd et = cexp_d(tmp);
      for (int k = 0; k < 2; k++) wlay[i][k] = cadd(p[i + 1][k], 1.0) / cadd(p[i][k] * el[i], 1.0) * et;
    }
    for (int l = 1; l <= Nl; l++) {
      const int hi = l > rl ? l : rl, lo = l > rl ? rl : l;
      zd a0 = Arr[hi][0], a1 = Arr[hi][1];
      for (int j = hi - 1; j >= lo; j--) {
        a0 = a0 * wlay[j][0];
        a1 = a1 * wlay[j][1];
      }
      Arl[l][0] = a0;
      Arl[l][1] = rl > l ? a1 * sh_cs[rl] / sh_cs[l] : a1;
    }
    layer_pqexpz(Nz, Nl, lnumg, zg, dzg, sh_td, eta, p, q, expz, pez, qez);
  }
  __syncthreads();
  zd* T = tabs + (int64_t)K * RF_COUNT * Nz;
  const zd eta_r = eta[rl], eta_zr = eta_r * L.zr, sr = sh_cs[rl];
  for (int I = 1 + threadIdx.x; I <= Nz; I += blockDim.x) {
    const int l = lnumg[I];
    const zd ez = expz[I], et = eta[l];
    const bool above = I <= N;  // cell above the receiver
    // Calc_Recv_Part (rc_kernel_hankel_module.F90:187-230)
    zd w1[2], w2[2];
    if (!above) {
      const zd eta_dr = rl > 1 ? eta_r * (sh_td[rl - 1].y * 2.0) : cz2(0, 0);
      const zd e1 = cexp_d(et * (-zg[I - 1]) + eta_zr);
      const zd e2 = cexp_d(et * (-zg[I - 1]) - eta_zr + eta_dr);
      w1[0] = e2 * p[rl][0] + e1;
      w1[1] = (e1 - e2 * p[rl][0]) * eta_r;
      w2[0] = e2 * p[rl][1] + e1;
      w2[1] = (e1 - e2 * p[rl][1]) * eta_r;
    } else {
      const zd e1 = cexp_d(et * zg[I] - eta_zr);
      // below the last layer the reflected term vanishes (eta_dr = HUGE, :219)
      const zd e2 = rl < Nl ? cexp_d(et * zg[I] + eta_zr - eta_r * (sh_td[rl].y * 2.0)) : cz2(0, 0);
      w1[0] = e2 * q[rl][0] + e1;
      w1[1] = (e2 * q[rl][0] - e1) * eta_r;
      w2[0] = e2 * q[rl][1] + e1;
      w2[1] = (e2 * q[rl][1] - e1) * eta_r;
    }
    // Calc_Ftb (:232-254): p above the receiver with sign -1, q below with +1
    const zd* pq = above ? pez : qez;
    const double sgn = above ? -1.0 : 1.0;
    const zd a = cz2(1.0 - ez.x, -ez.y), a1 = a / et;
    const zd F0 = a1 * cadd(pq[2 * I] * ez, 1.0);
    const zd F1 = a1 * cadd(pq[2 * I + 1] * ez, 1.0);
    const zd pe = pq[2 * I + 1] * ez;
    const zd F2 = a * (cz2(1.0 - pe.x, -pe.y) * sgn);
    // Calc_G_not_match (:152-186)
    const zd A1 = Arl[l][0], A2 = Arl[l][1];
    const zd G1 = A1 * F0 * w1[0];
    const zd G3DZ = (A2 * F2 * w2[1]) / sr;
    const zd G2DZ = (A2 * F1 * w2[1]) / sr;
    const zd G2DZ0 = (A2 * F2 * w2[0]) / sr;
    const zd G2G2DZZ = (A2 * F1 * w2[0]) * (lm * lm) / sr;
    const zd G3 = A2 * F2 * w2[0] - A1 * F0 * w1[1];
    const zd G1DZ = A1 * F0 * w1[1];
    const zd G2 = A2 * F1 * w2[0];
    const zd G11 = G1 * L.iwm;
    const int z = I - 1;
    T[RF_G11 * Nz + z] = G11;
    T[RF_G3DZ_G11 * Nz + z] = G3DZ + G11;
    T[RF_G2DZ * Nz + z] = G2DZ;
    T[RF_G2DZ0 * Nz + z] = G2DZ0;
    T[RF_G2G2DZZ * Nz + z] = G2G2DZZ;
    T[RF_G3 * Nz + z] = G3;
    T[RF_G1DZ * Nz + z] = G1DZ;
    T[RF_G2 * Nz + z] = G2;
    T[RF_G1 * Nz + z] = G1;
    T[RF_NG1DZ * Nz + z] = -G1DZ;
    T[RF_NG3 * Nz + z] = -G3;
    T[RF_NG2 * Nz + z] = -G2;
    T[RF_NG1 * Nz + z] = -G1;
  }
}

// In-place forward FFT of every tensor column along y for a fixed ix
// (AXIS 0) or along x for a fixed iy (AXIS 1), points p = ix*Ny2 + iy.
template <int L, int AXIS, bool RT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RT ? 2 : 1))) void k_rc_tfft(zd* __restrict__ G, const zd* __restrict__ twg, int Ny2,
                                                 int64_t BS, FftPlan plan) {
  constexpr int NE = ne_for<L>(), LS = L + 1, NT = 256;
  __shared__ zd buf[NE * LS];
  __shared__ zd tw[L];
  const int Lr = RT ? plan.L : L;
  const int fixed = blockIdx.x;
  const int64_t e0 = (int64_t)blockIdx.y * NE;
  for (int i = threadIdx.x; i < Lr; i += NT) tw[i] = twg[i];
  auto gidx = [&](int l) -> int64_t {
    return AXIS == 0 ? ((int64_t)fixed * Ny2 + l) * BS : ((int64_t)l * Ny2 + fixed) * BS;
  };
  for (int i = threadIdx.x; i < NE * Lr; i += NT) {
    const int l = i / NE, s = i - l * NE;
    buf[s * LS + l] = (e0 + s < BS) ? G[gidx(l) + e0 + s] : mkz(0, 0);
  }
  __syncthreads();
  lds_fft_any<zd, L, NE, LS, NT, -1, RT>(buf, tw, plan);
  for (int i = threadIdx.x; i < NE * Lr; i += NT) {
    const int k = i / NE, s = i - k * NE;
    if (e0 + s < BS) G[gidx(k) + e0 + s] = buf[s * LS + k];
  }
}

// PrepareRecvs (data_types_module.F90:124-152) against the current background
void rc_prepare_receivers(RcOperator& rc) {
  const Operator& op = *rc.op;
  G2G_CHECK(op.have_bkg, -4, "background not set");
  const int Nz = op.Nz;
  rc.zr.resize(rc.Nr);
  rc.layer.resize(rc.Nr);
  rc.cell.resize(rc.Nr);
  for (int r = 0; r < rc.Nr; r++) {
    const double z = rc.depth[r];
    rc.layer[r] = std::max(op_layer(op, z), 1);
    rc.zr[r] = z;
    if (z <= op.z[0]) {
      rc.cell[r] = 0;
    } else if (z >= op.z[Nz]) {
      rc.cell[r] = Nz + 1;
    } else {
      for (int Iz = 1; Iz <= Nz; Iz++) {
        if (std::fabs(z / op.z[Iz] - 1.0) < 1e-7) {
          rc.cell[r] = Iz;
          break;
        } else if (z > op.z[Iz - 1] && z < op.z[Iz]) {
          rc.zr[r] = op.z[Iz - 1];
          rc.cell[r] = Iz - 1;
          break;
        }
      }
    }
  }
}

void rc_build_tensor(RcOperator& rc) {
  Operator& op = *rc.op;
  G2G_CHECK(op.have_bkg, -4, "background not set");
  G2G_CHECK(op.Nl <= 64 && op.Nz <= MAX_NZ, -3, "tensor build supports Nl <= 64 and Nz <= 256");
  // weights of other cell sizes (the operator's geometry has changed since) are made anew
  if (rc.wts_dx != op.dx || rc.wts_dy != op.dy) {
    rc_check_corners(op, rc.Nr, rc.xs.data(), rc.ys.data());
    rc.have_wts = false;
  }
  rc_prepare_receivers(rc);
  const int Nz = op.Nz, Nr = rc.Nr;
  const int64_t NP = rc.NP, BS = rc.BS, WS = (int64_t)6 * NTAPS * NP + NP;  // weights per receiver, then the points' windows of taps
  const double rmin = std::sqrt(op.dx * op.dx + op.dy * op.dy) / 2.0;  // :67
  const BuildTables bt = build_tables(op, rc.par, rmin);
  G2G_HIP(hipEventRecord(rc.ev[0], op.stream));
  // The weights do not depend on frequency: all receivers' weights are kept
  // when they fit in 8 GB, else one receiver's are recomputed per build.
  const bool cache = (double)Nr * WS * sizeof(double) <= 8.0 * (1 << 30);
  zd *tw = nullptr, *f1 = nullptr;
  if (!rc.have_wts) {
    make_tw64(VBN, &tw);
    G2G_HIP(hipMalloc(&f1, sizeof(zd) * VBN));
    hipLaunchKernelGGL(k_f1, dim3(1), dim3(256), 0, op.stream, f1, tw);
    if (!rc.wts) {
      G2G_HIP(hipMalloc(&rc.wts, sizeof(double) * WS * (cache ? Nr : 1)));
      rc.bytes += sizeof(double) * WS * (cache ? Nr : 1);
    }
  }
  auto weights = [&](int r, double* dst) {
    RcWParams wp{op.Nx, op.Ny, op.dx, op.dy, rc.xs[r], rc.ys[r], std::log(rmin)};
    hipLaunchKernelGGL(k_rc_weights, dim3((unsigned)NP), dim3(256), 0, op.stream, dst,
                       (int2*)(dst + 6 * NTAPS * NP), f1, tw, bt.lms, wp);
  };
  if (!rc.have_wts && cache)
    for (int r = 0; r < Nr; r++) weights(r, rc.wts + r * WS);
  if (!rc.tabs) {
    G2G_HIP(hipMalloc(&rc.tabs, sizeof(zd) * NTAPS * RF_COUNT * Nz));
    rc.bytes += sizeof(zd) * NTAPS * RF_COUNT * Nz;
  }
  const double scale = 1.0 / PI_D / 4.0;  // :223-224
  const int64_t ldb = RF_COUNT * Nz;
  for (int r = 0; r < Nr; r++) {
    double* W = rc.wts + (cache ? r * WS : 0);
    if (!cache) weights(r, W);
    RcLParams lp{op.Nl, Nz, rc.layer[r], rc.cell[r], rc.zr[r], mkz(0.0, bt.mw), bt.bk};
    hipLaunchKernelGGL(k_rc_lambda, dim3(NTAPS), dim3(64), 0, op.stream, rc.tabs, bt.lms, bt.dz, bt.z, bt.ln, lp);
    auto Wc = [&](int c) { return W + (int64_t)c * NTAPS * NP; };
    auto Tf = [&](int f) { return (const zd*)rc.tabs + (int64_t)f * Nz; };
    auto J1 = [&](int e, int c, int f) {
      const int o = (e * Nr + r) * Nz;
      return WJob{o, o, Nz, 1, Wc(c), nullptr, Tf(f), nullptr};
    };
    auto J2 = [&](int e, int c, int f, int c2, int f2) {
      const int o = (e * Nr + r) * Nz;
      return WJob{o, o, Nz, 2, Wc(c), Wc(c2), Tf(f), Tf(f2)};
    };
    // Calc_Integral_U accumulation (rc_kernel_hankel_module.F90:116-145)
    const WJobs jobs = {15,
                        {J2(0, IE_D0, RF_G11, IE_DXX, RF_G3DZ_G11),   // REXX
                         J1(1, IE_DXY, RF_G3DZ_G11),                  // REXY
                         J1(2, IE_DX, RF_G2DZ),                       // REXZ
                         J2(3, IE_D0, RF_G11, IE_DYY, RF_G3DZ_G11),   // REYY
                         J1(4, IE_DY, RF_G2DZ),                       // REYZ
                         J1(5, IE_DX, RF_G2DZ0),                      // REZX
                         J1(6, IE_DY, RF_G2DZ0),                      // REZY
                         J1(7, IE_D0, RF_G2G2DZZ),                    // REZZ
                         J1(8, IE_DXY, RF_G3),                        // RHXX
                         J2(9, IE_DYY, RF_G3, IE_D0, RF_NG1DZ),       // RHXY
                         J1(10, IE_DY, RF_G2),                        // RHXZ
                         J2(11, IE_D0, RF_G1DZ, IE_DXX, RF_NG3),      // RHYX
                         J1(12, IE_DX, RF_NG2),                       // RHYZ
                         J1(13, IE_DY, RF_NG1),                       // RHZX
                         J1(14, IE_DX, RF_G1)}};                      // RHZY
    hipLaunchKernelGGL(k_wgemm<false>, wgemm_grid(NP, jobs), dim3(256), 0, op.stream, rc.G, NP, NP, BS, ldb,
                       (const int2*)(W + 6 * NTAPS * NP), 0, scale, jobs);
  }
  G2G_HIP(hipGetLastError());
  G2G_HIP(hipEventRecord(rc.ev[1], op.stream));
  G2G_HIP(hipStreamSynchronize(op.stream));
  float ms = 0;
  G2G_HIP(hipEventElapsedTime(&ms, rc.ev[0], rc.ev[1]));
  rc.t_tensor = ms * 1e-3;
  rc.have_wts = rc.have_wts || cache;
  rc.wts_dx = op.dx;
  rc.wts_dy = op.dy;
  rc.have_tensor = true;
  rc.spectral = false;
  rc.tensor_version = op.bkg_version;
  if (tw) (void)hipFree(tw);
  if (f1) (void)hipFree(f1);
}

void rc_tensor_fft(RcOperator& rc) {
  Operator& op = *rc.op;
  G2G_CHECK(rc.have_tensor && !rc.spectral, -4, "receiver tensor not built (or already transformed)");
  const int Nx2 = 2 * op.Nx, Ny2 = 2 * op.Ny;
  const zd *twx = op.d64.twx, *twy = op.d64.twy;
  const FftPlan &py = op.py, &px = op.px;
  G2G_HIP(hipEventRecord(rc.ev[0], op.stream));
  len_dispatch(Ny2, [&](auto LC) {
    constexpr int LL = decltype(LC)::value;
    constexpr int NE = ne_for<LL>();
    hipLaunchKernelGGL((k_rc_tfft<LL, 0, decltype(LC)::rt>), dim3(Nx2, (unsigned)((rc.BS + NE - 1) / NE)),
                       dim3(256), 0, op.stream, rc.G, twy, Ny2, rc.BS, py);
  });
  len_dispatch(Nx2, [&](auto LC) {
    constexpr int LL = decltype(LC)::value;
    constexpr int NE = ne_for<LL>();
    hipLaunchKernelGGL((k_rc_tfft<LL, 1, decltype(LC)::rt>), dim3(Ny2, (unsigned)((rc.BS + NE - 1) / NE)),
                       dim3(256), 0, op.stream, rc.G, twx, Ny2, rc.BS, px);
  });
  G2G_HIP(hipGetLastError());
  G2G_HIP(hipEventRecord(rc.ev[1], op.stream));
  G2G_HIP(hipStreamSynchronize(op.stream));
  float ms = 0;
  G2G_HIP(hipEventElapsedTime(&ms, rc.ev[0], rc.ev[1]));
  rc.t_fft = ms * 1e-3;
  rc.spectral = true;
}

}  // namespace g2g
