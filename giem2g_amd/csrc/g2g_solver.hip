// g2g_solver.hip -- device-resident nested FGMRES.
//
// Reference path replaced: SolveEquation -> GIEM2G_FGMRES -> SEQ_FGMRES_SOLVE
// -> GMRES_SOLVE (ie_solver_module.F90:43-258; GFGMRES/gmres.F90:110-549;
// GFGMRES/seq_fgmres.F90:109-226).  The algorithm is kept step for step --
// depth-2 nesting (flexible outer FGMRES, one cycle of plain GMRES with
// x0 = b as the right preconditioner), iterated classical Gram-Schmidt with
// the 2|w| > |h| test and at most 3 re-orthogonalisations, Givens rotations
// (reference-BLAS ZROTG/ZROT semantics), restart from the Arnoldi residual,
// final true residual -- so iteration counts compare with the reference.
// Krylov vectors live in HBM; the (m+1)x(m+1) Hessenberg matrix and the
// rotations stay on the host.  The inner solver can run on complex64
// vectors with the complex64 operator (mixed precision; the outer stays FP64
// and acts as iterative refinement).
#include <chrono>
#include <cstdlib>
#include <complex>
#include <functional>
#include <vector>

#include "g2g_op.hpp"
#include <condition_variable>
#include <exception>
#include <mutex>
#include <thread>

#include "g2g_solver.hpp"

namespace g2g {

using zc = std::complex<double>;
constexpr int BT = 256;
// blocks of the Krylov reductions and updates: two per CU (C2 solves, against
// 1024 blocks: FP64 1.2% and complex64-inner 0.6% faster; 256 made the
// complex64 solve 5% slower, 768 and 2048 were slower than 512)
constexpr int NBLK = 512;
constexpr int KC = 8;       // columns per multi-dot block row
constexpr int MAXK = 64;    // columns of one multi-dot call (Krylov basis size bound)


template <typename A> __device__ inline A wave_sum(A v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Sums over the wave of 2KC values at once: each step halves the values a lane
// carries (17 shuffles instead of 6 for each value, the additions of each sum
// the same as wave_sum's).  Lanes 4j .. 4j+3 return the sum of value j.  The
// shuffles bound the short dot products: with six each, k_mdot took 6.3 us at
// 32x32x8 in FP64 and k_reduce 5.3, now 4.0 and 2.4.
template <int N, typename A> __device__ inline void wave_halve(A (&v)[2 * KC]) {
  const bool up = threadIdx.x & (4 * N);
#pragma unroll
  for (int k = 0; k < N; k++) {
    const A keep = up ? v[k + N] : v[k], give = up ? v[k] : v[k + N];
    v[k] = keep + __shfl_xor(give, 4 * N);
  }
}
template <typename A> __device__ inline A wave_sums(A (&v)[2 * KC]) {
  static_assert(KC == 8, "the halving is for 16 values");
  wave_halve<8>(v);
  wave_halve<4>(v);
  wave_halve<2>(v);
  wave_halve<1>(v);
  v[0] += __shfl_xor(v[0], 2);
  return v[0] + __shfl_xor(v[0], 1);
}

// Partial sums of conj(V[:,k]) . w for k < K: block row blockIdx.y takes
// columns KC*y .. KC*y + KC - 1 and writes part[(y*gridDim.x + x)*2KC + j]
template <typename T2, typename A>
__global__ __launch_bounds__(BT) void k_mdot(const T2* __restrict__ V, int64_t N, int K,
                                             const T2* __restrict__ w, A* __restrict__ part) {
  const int k0 = blockIdx.y * KC, kc = K - k0 < KC ? K - k0 : KC;
  V += (int64_t)k0 * N;
  part += (int64_t)blockIdx.y * gridDim.x * 2 * KC;
  A acc[2 * KC];
#pragma unroll
  for (int k = 0; k < 2 * KC; k++) acc[k] = 0;
  // all KC loads issued before the products: the column index is clamped to
  // kc - 1 instead of a branch per column (with a branch each load waited for
  // the one before, about 2 TB/s); sums past kc are never read
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT) {
    const T2 wv = w[i];
    T2 v[KC];
#pragma unroll
    for (int k = 0; k < KC; k++) v[k] = ld_stream(V + (int64_t)(k < kc ? k : kc - 1) * N + i);
#pragma unroll
    for (int k = 0; k < KC; k++) {
      acc[2 * k] += (A)v[k].x * (A)wv.x + (A)v[k].y * (A)wv.y;
      acc[2 * k + 1] += (A)v[k].x * (A)wv.y - (A)v[k].y * (A)wv.x;
    }
  }
  __shared__ A red[BT / 64][2 * KC];
  const A sum = wave_sums(acc);
  if ((threadIdx.x & 3) == 0) red[threadIdx.x >> 6][(threadIdx.x & 63) >> 2] = sum;
  __syncthreads();
  if (threadIdx.x < 2 * KC) {
    A s = 0;
    for (int q = 0; q < BT / 64; q++) s += red[q][threadIdx.x];
    part[blockIdx.x * 2 * KC + threadIdx.x] = s;
  }
}

// out[2KC*y + j] = sum_b part[(y*nb + b)*2KC + j]; block y, 2*KC outputs (as double)
template <typename A>
__global__ __launch_bounds__(BT) void k_reduce(const A* __restrict__ part, int nb, double* out) {
  part += (int64_t)blockIdx.x * nb * 2 * KC;
  out += blockIdx.x * 2 * KC;
  __shared__ double red[BT / 64][2 * KC];
  double acc[2 * KC];
  for (int j = 0; j < 2 * KC; j++) acc[j] = 0;
  for (int b = threadIdx.x; b < nb; b += BT)
    for (int j = 0; j < 2 * KC; j++) acc[j] += (double)part[b * 2 * KC + j];
  const double sum = wave_sums(acc);
  if ((threadIdx.x & 3) == 0) red[threadIdx.x >> 6][(threadIdx.x & 63) >> 2] = sum;
  __syncthreads();
  if (threadIdx.x < 2 * KC) {
    double s = 0;
    for (int q = 0; q < BT / 64; q++) s += red[q][threadIdx.x];
    out[threadIdx.x] = s;
  }
}

// w -= sum_k V[:,k] h[k]; part[b] = partial |w|^2
template <typename T2, typename A>
__global__ __launch_bounds__(BT) void k_update_norm(T2* __restrict__ w, const T2* __restrict__ V,
                                                    int64_t N, int K, const zd* __restrict__ h,
                                                    A* __restrict__ part) {
  // coefficients past K are zero, so the columns go in groups of KC with
  // all loads of a group in flight (index clamped to K - 1); the terms are
  // added in the same order as one at a time, and the zero ones change nothing
  __shared__ T2 hs[MAXK];
  for (int k = threadIdx.x; k < MAXK; k += BT) hs[k] = k < K ? mk<T2>(h[k].x, h[k].y) : mk<T2>(0, 0);
  __syncthreads();
  A nrm = 0;
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT) {
    T2 acc = w[i];
    for (int k0 = 0; k0 < K; k0 += KC) {
      T2 v[KC];
#pragma unroll
      for (int j = 0; j < KC; j++) v[j] = ld_stream(V + (int64_t)(k0 + j < K ? k0 + j : K - 1) * N + i);
#pragma unroll
      for (int j = 0; j < KC; j++) {
        const T2 hk = hs[k0 + j];
        acc.x -= v[j].x * hk.x - v[j].y * hk.y;
        acc.y -= v[j].x * hk.y + v[j].y * hk.x;
      }
    }
    w[i] = acc;
    nrm += (A)acc.x * (A)acc.x + (A)acc.y * (A)acc.y;
  }
  __shared__ A red[BT / 64];
  A a = wave_sum(nrm);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    A s = 0;
    for (int q = 0; q < BT / 64; q++) s += red[q];
    part[blockIdx.x] = s;
  }
}

// x = sum_k B[:,k] y[k] (+ x if accumulate)
template <typename T2>
__global__ __launch_bounds__(BT) void k_lincomb(T2* __restrict__ x, const T2* __restrict__ B,
                                                int64_t N, int K, const zd* __restrict__ y,
                                                int accumulate) {
  __shared__ T2 ys[64];
  for (int k = threadIdx.x; k < K; k += BT) ys[k] = mk<T2>(y[k].x, y[k].y);
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT) {
    T2 acc = accumulate ? x[i] : mk<T2>(0, 0);
    for (int k = 0; k < K; k++) cmac(acc, B[(int64_t)k * N + i], ys[k]);
    x[i] = acc;
  }
}

template <typename T2, typename R>
__global__ void k_scale(T2* __restrict__ dst, const T2* __restrict__ src, int64_t N, R s) {
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT)
    dst[i] = src[i] * s;
}
template <typename T2> __global__ void k_bminus(T2* __restrict__ r, const T2* __restrict__ b, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT)
    r[i] = b[i] - r[i];
}
template <typename T2> __global__ void k_add(T2* __restrict__ x, const T2* __restrict__ a, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT)
    x[i] = x[i] + a[i];
}
template <typename Ti, typename To>
__global__ void k_convert(To* __restrict__ o, const Ti* __restrict__ a, int64_t N) {
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT)
    o[i] = mk<To>((decltype(To::x))a[i].x, (decltype(To::x))a[i].y);
}
// rhs / guess scaling of SolveEquation (ie_solver_module.F90:64-97)
__global__ void k_rhs_scale(zd* __restrict__ out, const zd* __restrict__ in,
                            const zd* __restrict__ asiga, const double* __restrict__ sq,
                            int64_t ncxy, int Nz, int64_t N, int mode) {
  // mode 0: out = sq*in; 1: out = in/asiga; 2: out = asiga*in
  for (int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x; i < N; i += (int64_t)gridDim.x * BT) {
    const int64_t ci = i % (ncxy * Nz);
    const int z = (int)(ci / ncxy);
    if (mode == 0) out[i] = in[i] * sq[z];
    else if (mode == 1) out[i] = cdiv(in[i], asiga[ci]);
    else out[i] = asiga[ci] * in[i];
  }
}

static inline dim3 gridN(int64_t N) {
  int64_t b = (N + BT - 1) / BT;
  return dim3((unsigned)(b < 4096 ? b : 4096));
}

// Results the host reads (dot products, a Gram-Schmidt pass's coefficients
// and norm) reach it through a mailbox in pinned host memory: one wave
// copies them there and then raises a sequence number, which the host polls.
// The host sees them a few microseconds after the kernel ends; a copy and a
// blocking stream synchronisation took about 50 us per Gram-Schmidt pass.
struct Mailbox {
  unsigned seq;
  unsigned pad[63];
  double v[2 * MAXK + 2 * KC];
};
__global__ __launch_bounds__(64) void k_publish(const double* __restrict__ src, int n, Mailbox* mb,
                                                unsigned seq) {
  for (int i = threadIdx.x; i < n; i += 64) mb->v[i] = src[i];
  __threadfence_system();  // the values are visible to the host before the number
  if (threadIdx.x == 0) __hip_atomic_store(&mb->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// How long the host polls before it falls back to a blocking
// synchronisation: GIEM2G_POLL_MS milliseconds (0: block at once), else 200
static int poll_limit_ms() {
  const char* e = std::getenv("GIEM2G_POLL_MS");
  if (!e || !*e) return 200;
  const int v = std::atoi(e);
  return v < 0 ? 0 : v;
}

// The end of a Gram-Schmidt pass: |w|^2 from the update's partial sums and the
// pass's test 2|w| > |h| (accepted also when `force`, the fourth pass), which
// every block makes for itself (the sums of nb <= NBLK blocks, from the
// caches), then the next basis vector dst = src / |w| where the pass was
// accepted (queued before the host has read the results) and nothing
// otherwise.  Block 0 publishes |w|^2, the test and the pass's coefficients h
// (res[0 .. 2K)) in the host mailbox.  Launches bound it at small grids: with
// the sum and the test in a kernel of one block before it 6.6 us at 32x32x8,
// now 3.8.
template <typename T2, typename R>
__global__ __launch_bounds__(BT) void k_scale_pass(T2* __restrict__ dst, const T2* __restrict__ src, int64_t N,
                                                    const R* __restrict__ npart, int nb, const double* __restrict__ res,
                                                    int K, int force, Mailbox* mb, unsigned seq) {
  static_assert(2 * MAXK <= BT, "one thread per coefficient");
  __shared__ double red[BT / 64], hred[2 * MAXK];
  const int t = threadIdx.x;
  int64_t i = (int64_t)blockIdx.x * BT + t;
  T2 x = src[i < N ? i : N - 1];
  double acc = 0;
  for (int b = t; b < nb; b += BT) acc += (double)npart[b];
  const double h = t < 2 * K ? res[t] : 0.0;
  acc = wave_sum(acc);
  if ((t & 63) == 0) red[t >> 6] = acc;
  if (t < 2 * MAXK) hred[t] = h;
  __syncthreads();
  double w2 = 0;
  for (int q = 0; q < BT / 64; q++) w2 += red[q];
  double h2 = 0;
  for (int k = 0; k < K; k++) h2 += hred[2 * k] * hred[2 * k] + hred[2 * k + 1] * hred[2 * k + 1];
  const bool ok = force || 2.0 * sqrt(w2) > sqrt(h2);
  if (blockIdx.x == 0 && t < 64) {
    for (int k = t; k < 2 * K; k += 64) mb->v[k] = hred[k];
    if (t == 0) {
      mb->v[2 * MAXK] = w2;
      mb->v[2 * MAXK + 1] = ok ? 1.0 : 0.0;
    }
    __threadfence_system();  // the values are visible to the host before the number
    if (t == 0) __hip_atomic_store(&mb->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (!ok) return;
  const R f = (R)(1.0 / sqrt(w2));
  while (i < N) {
    dst[i] = x * f;
    i += (int64_t)gridDim.x * BT;
    if (i < N) x = src[i];
  }
}
// Waits until the work queued on s so far has ended, polling an event for
// at most ms milliseconds
static void poll_event(hipEvent_t ev, hipStream_t s, int ms) {
  G2G_HIP(hipEventRecord(ev, s));
  const auto t0 = std::chrono::steady_clock::now();
  for (unsigned i = 1; ms > 0; i++) {
    const hipError_t e = hipEventQuery(ev);
    if (e == hipSuccess) return;
    if (e != hipErrorNotReady) G2G_HIP(e);
    if ((i & 255) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(ms)) break;
    __builtin_ia32_pause();
  }
  G2G_HIP(hipEventSynchronize(ev));
}

// ---------------------------------------------------------------- BLAS ---
struct DevBlas {
  hipStream_t s;
  void* part = nullptr;  // (MAXK/KC) * NBLK * 2KC doubles
  double* res = nullptr; // 2*MAXK dot products (complex pairs) + 2KC for a norm
  zd* hbuf = nullptr; // 64
  Mailbox* mail = nullptr;   // pinned host memory
  Mailbox* dmail = nullptr;  // its device address
  const double* hres = nullptr;  // mail->v
  int poll_ms = 200;             // poll_limit_ms() when the solve began
  // counts of this solver (merged into the operator's counters by the caller)
  int64_t dots = 0, passes = 0;
  double bytes = 0;  // bytes the Krylov kernels read and write
  Prof* prof = nullptr;  // event log of the profiling mode (dot products), or null
  int prof_start() { return prof && prof->on ? prof->record(s) : -1; }
  void prof_end(int a) {
    if (a >= 0) prof->mark(Prof::DOT, 0, 0, a, prof->record(s));
  }
  void init(hipStream_t st, Arena& ws) {
    s = st;
    part = ws.get(WS_PART, sizeof(double) * (MAXK / KC) * NBLK * 2 * KC);
    res = (double*)ws.get(WS_RES, sizeof(double) * (2 * MAXK + 2 * KC));
    hbuf = (zd*)ws.get(WS_HBUF, sizeof(zd) * 64);
    mail = (Mailbox*)ws.get_pinned(0, sizeof(Mailbox));
    G2G_HIP(hipHostGetDevicePointer((void**)&dmail, mail, 0));
    hres = mail->v;
    poll_ms = poll_limit_ms();
  }
  static int nblocks(int64_t N) { return (int)std::min<int64_t>(NBLK, (N + BT - 1) / BT); }
  // res[0 .. 2K) = V[:,k]^H w for k < K, on the device (no host round trip)
  template <typename T2, typename A> void mdot_dev(const T2* V, int64_t N, int K, const T2* w) {
    G2G_CHECK(K >= 1 && K <= MAXK, -3, "multi-dot of more than 64 columns");
    const int nb = nblocks(N), nrow = (K + KC - 1) / KC;
    bytes += (double)sizeof(T2) * N * (K + 1);
    hipLaunchKernelGGL((k_mdot<T2, A>), dim3(nb, nrow), dim3(BT), 0, s, V, N, K, w, (A*)part);
    hipLaunchKernelGGL((k_reduce<A>), dim3(nrow), dim3(BT), 0, s, (const A*)part, nb, res);
  }
  // res[0 .. n) to hres; everything queued on the stream before has ended
  void fetch(int n) {
    // the last number published has been seen, so it cannot change meanwhile
    const unsigned seq = __atomic_load_n(&mail->seq, __ATOMIC_ACQUIRE) + 1;
    hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, s, (const double*)res, n, dmail, seq);
    G2G_HIP(hipGetLastError());
    wait_mail(seq);
  }
  // until the mailbox holds number seq
  void wait_mail(unsigned seq) {
    const auto t0 = std::chrono::steady_clock::now();
    for (unsigned i = 1; poll_ms > 0; i++) {
      if (__atomic_load_n(&mail->seq, __ATOMIC_ACQUIRE) == seq) return;
      if ((i & 4095) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(poll_ms))
        break;
      __builtin_ia32_pause();
    }
    // a long queue (or an error, which the synchronisation reports)
    G2G_HIP(hipStreamSynchronize(s));
    G2G_CHECK(__atomic_load_n(&mail->seq, __ATOMIC_ACQUIRE) == seq, -1,
              "the reduction results did not reach the host");
  }
  // out[k] = V[:,k]^H w for k < K
  template <typename T2, typename A>
  void mdot(const T2* V, int64_t N, int K, const T2* w, zc* out) {
    const int pa = prof_start();
    mdot_dev<T2, A>(V, N, K, w);
    prof_end(pa);
    fetch(2 * K);
    for (int k = 0; k < K; k++) out[k] = zc(hres[2 * k], hres[2 * k + 1]);
    dots += K;
  }
  // One classical Gram-Schmidt pass: h = V^H w, w -= V h, returns |w|; h goes
  // from the reduction straight to the update kernel, one host round trip.
  // The device also makes the pass's test 2|w| > |h| (accepted when `force`)
  // and, when it passes, writes vnext = w/|w| before the host has read the
  // results; *accepted tells the host which it was.
  template <typename T2, typename A>
  double ortho_pass(T2* w, const T2* V, int64_t N, int K, zc* h, T2* vnext, bool force, bool* accepted) {
    const int pa = prof_start();
    mdot_dev<T2, A>(V, N, K, w);
    const int nb = nblocks(N);
    hipLaunchKernelGGL((k_update_norm<T2, A>), dim3(nb), dim3(BT), 0, s, w, V, N, K, (const zd*)res,
                       (A*)part);
    const unsigned seq = __atomic_load_n(&mail->seq, __ATOMIC_ACQUIRE) + 1;
    hipLaunchKernelGGL((k_scale_pass<T2, A>), gridN(N), dim3(BT), 0, s, vnext, (const T2*)w, N, (const A*)part, nb,
                       (const double*)res, K, force ? 1 : 0, dmail, seq);
    G2G_HIP(hipGetLastError());
    prof_end(pa);
    bytes += (double)sizeof(T2) * N * (K + 2);
    wait_mail(seq);
    for (int k = 0; k < K; k++) h[k] = zc(hres[2 * k], hres[2 * k + 1]);
    *accepted = hres[2 * MAXK + 1] != 0.0;
    if (*accepted) bytes += 2.0 * sizeof(T2) * N;
    dots += K + 1;
    passes++;
    return std::sqrt(hres[2 * MAXK]);
  }
  template <typename T2, typename A> double norm(const T2* v, int64_t N) {
    zc t;
    mdot<T2, A>(v, N, 1, v, &t);
    return std::sqrt(t.real());
  }
  template <typename T2>
  void lincomb(T2* x, const T2* B, int64_t N, int K, const zc* y, bool acc) {
    bytes += (double)sizeof(T2) * N * (K + (acc ? 2 : 1));
    G2G_HIP(hipMemcpyAsync(hbuf, y, sizeof(zd) * K, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL((k_lincomb<T2>), gridN(N), dim3(BT), 0, s, x, B, N, K, hbuf, acc ? 1 : 0);
  }
  template <typename T2, typename R> void scale(T2* d, const T2* src, int64_t N, R f) {
    bytes += 2.0 * sizeof(T2) * N;
    hipLaunchKernelGGL((k_scale<T2, R>), gridN(N), dim3(BT), 0, s, d, src, N, f);
  }
  template <typename T2> void copy(T2* d, const T2* src, int64_t N) {
    bytes += 2.0 * sizeof(T2) * N;
    G2G_HIP(hipMemcpyAsync(d, src, sizeof(T2) * N, hipMemcpyDeviceToDevice, s));
  }
  template <typename T2> void bminus(T2* r, const T2* b, int64_t N) {
    bytes += 3.0 * sizeof(T2) * N;
    hipLaunchKernelGGL((k_bminus<T2>), gridN(N), dim3(BT), 0, s, r, b, N);
  }
  template <typename T2> void add(T2* x, const T2* a, int64_t N) {
    bytes += 3.0 * sizeof(T2) * N;
    hipLaunchKernelGGL((k_add<T2>), gridN(N), dim3(BT), 0, s, x, a, N);
  }
  template <typename Ti, typename To> void convert(To* o, const Ti* a, int64_t N) {
    bytes += (double)(sizeof(Ti) + sizeof(To)) * N;
    hipLaunchKernelGGL((k_convert<Ti, To>), gridN(N), dim3(BT), 0, s, o, a, N);
  }
};

// reference BLAS ZROTG / ZROT
static void zrotg(zc& ca, zc cb, double& c, zc& sn) {
  if (std::abs(ca) == 0.0) {
    c = 0.0;
    sn = 1.0;
    ca = cb;
  } else {
    const double scale = std::abs(ca) + std::abs(cb);
    const double a1 = std::abs(ca / scale), b1 = std::abs(cb / scale);
    const double nrm = scale * std::sqrt(a1 * a1 + b1 * b1);
    const zc alpha = ca / std::abs(ca);
    c = std::abs(ca) / nrm;
    sn = alpha * std::conj(cb) / nrm;
    ca = alpha * nrm;
  }
}
static void zrot(zc& cx, zc& cy, double c, zc s) {
  const zc t = c * cx + s * cy;
  cy = c * cy - std::conj(s) * cx;
  cx = t;
}

// ------------------------------------------------------------- GMRES ---
template <typename R> struct Gmres {
  using T2 = cx_t<R>;
  using Apply = std::function<void(const T2*, T2*)>;
  int64_t N = 0;
  int M = 0;
  bool flex = false;
  int maxit = 1;
  double tol = 1e-8;
  T2 *x = nullptr, *r0 = nullptr, *w = nullptr, *V = nullptr, *Z = nullptr;
  std::vector<zc> H, gs, y, dp;
  std::vector<double> gc;
  int iternum = 0;
  double cur_res = 1;  // relative residual after the last Arnoldi step
  // FinalActions recomputes the true residual (one more product); an inner
  // solve whose caller only takes the solution can skip it
  bool true_residual = true;
  Apply A;
  Apply precond;  // right preconditioner (flex only); identity when empty
  // optional check of a variable preconditioner: accept_step(v, A z) false
  // replaces z by fallback(v) before the Gram-Schmidt step
  std::function<bool(const T2*, const T2*)> accept_step;
  Apply fallback;
  DevBlas* blas = nullptr;
  int64_t* matvecs = nullptr;
  std::vector<double>* hist = nullptr;
  size_t bytes = 0;

  zc& HH(int i, int j) { return H[(size_t)i + (size_t)(M + 1) * j]; }

  // buffers from arena slots slot0 .. slot0+4 (kept for the next solve)
  void alloc(int64_t n, int m, bool f, Arena& ws, int slot0) {
    N = n;
    M = m;
    flex = f;
    auto Al = [&](T2** p, int64_t cnt, int k) {
      *p = (T2*)ws.get(slot0 + k, sizeof(T2) * cnt);
      bytes += sizeof(T2) * cnt;
    };
    Al(&x, N, 0);
    Al(&r0, N, 1);
    Al(&w, N, 2);
    Al(&V, N * (M + 1), 3);
    if (flex) Al(&Z, N * M, 4);
    H.assign((size_t)(M + 1) * (M + 1), 0);
    gs.assign(M + 1, 0);
    gc.assign(M + 1, 0);
    y.assign(M + 1, 0);
    dp.assign(M + 1, 0);
  }
  void apply(const T2* in, T2* out) {
    A(in, out);
    if (matvecs) (*matvecs)++;
  }
  double norm(const T2* v) { return blas->norm<T2, R>(v, N); }
  T2* Vc(int k) { return V + (int64_t)k * N; }

  // ApplyRightPreconditioner (gmres.F90:491-506)
  void right_precond(const T2* vin, T2* vout, int K) {
    if (precond) precond(vin, vout);
    else blas->copy(vout, vin, N);
    if (flex) blas->copy(Z + (int64_t)K * N, vout, N);
  }
  // ConstructCurrentSolution (:423-458)
  void construct(int jH, T2* solution) {
    const int L = jH - 1;
    for (int i = 0; i < L; i++) y[i] = HH(i, M);
    for (int i = L - 1; i >= 0; i--) {
      zc t = y[i];
      for (int j = i + 1; j < L; j++) t -= HH(i, j) * y[j];
      y[i] = t / HH(i, i);
    }
    if (L > 0) {
      blas->lincomb(x, flex ? Z : V, N, L, y.data(), false);
      // non-flexible: right preconditioner is the identity here
      blas->add(solution, x, N);
    }
    blas->copy(x, solution, N);
  }
  // FinalActions (:382-421)
  double final_actions(int jH, double sPb, const T2* rhs, T2* solution, int* stat, double bea) {
    construct(jH, solution);
    if (!true_residual) {
      *stat = bea >= tol ? 2 : 1;
      return bea;
    }
    blas->copy(w, solution, N);
    apply(w, r0);
    blas->bminus(r0, rhs, N);
    const double tr = norm(r0);
    const double res = tr / sPb;
    *stat = res >= tol ? 2 : 1;
    return res;
  }
  // KrylovSubspaceConstruction (:216-329)
  double krylov(double bn, int* jHp) {
    int jH = *jHp;
    double bea = -1;
    for (;;) {
      const int j = jH - 1;
      // without a preconditioner (plain inner GMRES) the operator takes the
      // basis vector itself
      const T2* zj = Vc(j);
      if (precond || flex) {
        right_precond(Vc(j), w, j);
        zj = w;
      }
      apply(zj, r0);
      if (accept_step && !accept_step(Vc(j), r0)) {
        // the variable preconditioner's step is rejected: redo it with the fallback
        fallback(Vc(j), w);
        if (flex) blas->copy(Z + (int64_t)j * N, w, N);
        apply(w, r0);
      }
      std::swap(w, r0);
      for (int i = 0; i < jH; i++) HH(i, j) = 0;
      // iterated classical Gram-Schmidt: passes until 2|w| > |h| of the
      // last pass, at most four; the device makes the test and writes the
      // next basis vector w/|w| after the accepted pass
      int northo = 0;
      double dnormw = 0;
      for (;;) {
        northo++;
        bool accepted = false;
        dnormw = blas->ortho_pass<T2, R>(w, V, N, jH, dp.data(), Vc(jH), northo > 3, &accepted);
        for (int i = 0; i < jH; i++) HH(i, j) += dp[i];
        if (accepted) break;
      }
      HH(jH, j) = dnormw;
      for (int i = 0; i < j; i++) zrot(HH(i, j), HH(i + 1, j), gc[i], gs[i]);
      zc h1 = HH(j, j), h2 = HH(j + 1, j);
      zrotg(h1, h2, gc[j], gs[j]);
      zrot(HH(j, M), HH(j + 1, M), gc[j], gs[j]);
      zrot(HH(j, j), HH(j + 1, j), gc[j], gs[j]);
      HH(j + 1, j) = 0;
      bea = std::abs(HH(j + 1, M)) / bn;
      cur_res = bea;
      iternum++;
      if (hist) hist->push_back(bea);
      jH++;
      if (bea < tol || jH > M) break;
    }
    *jHp = jH;
    return bea;
  }
  // PrepareRestart (:333-379), iterative residual
  double restart(T2* solution, int jH) {
    construct(jH, solution);
    const double beta = std::abs(HH(M, M));
    for (int J = M - 1; J >= 0; J--) {
      HH(J, M) = 0;
      zrot(HH(J, M), HH(J + 1, M), gc[J], -gs[J]);
    }
    std::vector<zc> col(M + 1);
    for (int J = 0; J <= M; J++) col[J] = HH(J, M);
    blas->lincomb(w, V, N, M + 1, col.data(), false);
    return beta;
  }
  // GMRES_SOLVE (:110-213)
  SolveResult solve(T2* xo, const T2* x0, const T2* b) {
    SolveResult r;
    std::fill(H.begin(), H.end(), zc(0));
    iternum = 0;
    const double bn = norm(b);
    if (bn < 1e-14) {
      G2G_HIP(hipMemsetAsync(xo, 0, sizeof(T2) * N, blas->s));
      r.stat = 1;
      return r;
    }
    const double sPb = bn;
    blas->copy(xo, x0, N);
    apply(x0, r0);
    blas->bminus(r0, b, N);
    blas->copy(w, r0, N);
    double beta = norm(w);
    if (beta / bn < tol) {
      r.stat = 1;
      r.be = r.bea = beta / bn;
      return r;
    }
    int iter = 0, jH = 1, stat = -1;
    double bea = -1;
    for (;;) {
      HH(0, M) = beta;
      cur_res = beta / bn;
      blas->scale(V, w, N, (R)(1.0 / beta));
      for (int i = 0; i < M; i++) HH(i + 1, M) = 0;
      jH = 1;
      bea = krylov(bn, &jH);
      if (bea < tol) {
        r.be = final_actions(jH, sPb, b, xo, &stat, bea);
        r.stat = stat;
        r.iterations = iternum;
        r.bea = bea;
        return r;
      }
      iter++;
      if (iter >= maxit) break;
      beta = restart(xo, jH);
    }
    r.be = final_actions(jH, sPb, b, xo, &stat, bea);
    r.bea = bea;
    r.iterations = iternum;
    r.stat = -1;
    return r;
  }
};

// ------------------------------------------------------- nested solve ---
// res = v - alpha w with the least-squares alpha = <w, v>/<w, w>; returns
// ||res|| (res may alias w)
template <typename T2, typename A>
static double fit_residual(DevBlas& blas, const T2* v, const T2* w, T2* res, int64_t N, zc* alpha) {
  zc t, ww;
  blas.mdot<T2, A>(w, N, 1, v, &t);
  blas.mdot<T2, A>(w, N, 1, w, &ww);
  *alpha = ww.real() > 0 ? t / ww.real() : zc(0);
  blas.lincomb(res, w, N, 1, alpha, false);
  blas.bminus(res, v, N);
  return blas.norm<T2, A>(res, N);
}

SolveResult nested_solve(Operator& op, const zd* b, const zd* x0, zd* xout,
                         const SolveParams& p, std::vector<double>* hist,
                         const PrecondHook* learned, const SolveEnv* env) {
  const int64_t N = op.nvec();
  const hipStream_t st = env ? env->stream : op.stream;
  G2G_CHECK(!env || p.precond == 0, -3, "the learned preconditioner runs only in single solves");
  Arena& ws = env ? *env->ws : op.ws[0];
  DevBlas blas;
  blas.init(st, ws);
  blas.prof = &op.prof;
  Gmres<double> outer;
  outer.blas = &blas;
  outer.maxit = p.max_restart;
  outer.tol = p.tol;
  outer.alloc(N, p.outer_m, true, ws, WS_OUTER);
  outer.matvecs = env ? env->mv64 : &op.cnt.matvecs;
  outer.hist = hist;
  if (env) outer.A = env->A64;
  else outer.A = [&](const zd* in, zd* out) { op_apply<double>(op, op.d64, in, out, op.stream, false); };
  // inner tolerance: p.inner_tol when set; by default the reference's shared
  // tolerance for FP64 inner solves and the relaxed rule with factor 1 for
  // complex64 ones (their accuracy is judged by the FP64 outer's residual,
  // not by iteration counts that compare with the reference; at 256x256x32
  // 96 -> 79 complex64 products for the same 3 outer iterations, at
  // 128x128x64 unchanged)
  const double itol = p.inner_tol != 0 ? p.inner_tol : (p.inner_precision == 1 ? -1.0 : 0.0);
  Gmres<double> in64;
  Gmres<float> in32;
  zf *b32 = nullptr, *x32 = nullptr, *r32 = nullptr;
  zd *tmp = nullptr, *tmp2 = nullptr;
  SolveResult res;
  try {
    if (p.inner_precision == 0) {
      in64.blas = &blas;
      in64.maxit = 1;
      in64.tol = itol > 0 ? itol : p.tol;
      in64.alloc(N, p.inner_m, false, ws, WS_IN64);
      in64.matvecs = env ? env->mv64 : &op.cnt.matvecs;
      in64.A = outer.A;
    } else {
      if (!op.have_g32) op_make_g32(op);
      in32.blas = &blas;
      in32.maxit = 1;
      in32.tol = itol > 0 ? itol : p.tol;
      // the complex64 inner solve's own true residual is never used (the
      // FP64 outer judges the step); the FP64 inner keeps the reference's
      in32.true_residual = false;
      in32.alloc(N, p.inner_m, false, ws, WS_IN32);
      in32.matvecs = env ? env->mv32 : &op.cnt.matvecs32;
      if (env) in32.A = env->A32;
      else in32.A = [&](const zf* in, zf* out) { op_apply<float>(op, op.d32, in, out, op.stream, false); };
      b32 = (zf*)ws.get(WS_B32, sizeof(zf) * N);
      x32 = (zf*)ws.get(WS_X32, sizeof(zf) * N);
      if (p.precond == 1) r32 = (zf*)ws.get(WS_R32, sizeof(zf) * N);
    }
    tmp = (zd*)ws.get(WS_TMP, sizeof(zd) * N);
    if (p.precond == 1 && p.inner_precision == 0) tmp2 = (zd*)ws.get(WS_TMP2, sizeof(zd) * N);
    // FGMRES_BASED_PRECONDITIONER (seq_fgmres.F90:216-226): inner GMRES with x0 = b = v
    // relaxed inner tolerance (inner_tol < 0): an outer step whose residual
    // is already r needs its preconditioner only to tol / r, the relaxation
    // of inexact Krylov methods (Simoncini and Szyld, SIAM J. Sci. Comput.
    // 25, 2003): |inner_tol| tol / r, kept between tol and 0.1
    auto set_inner_tol = [&]() {
      if (itol >= 0) return;
      const double eta = std::min(0.1, std::max(p.tol, -itol * p.tol / std::max(outer.cur_res, 1e-300)));
      in64.tol = in32.tol = eta;
    };
    auto inner_gmres = [&](const zd* v, zd* z) {
      set_inner_tol();
      if (p.inner_precision == 0) {
        in64.solve(z, v, v);
      } else {
        blas.convert<zd, zf>(b32, v, N);
        in32.solve(x32, b32, b32);
        blas.convert<zf, zd>(z, x32, N);
      }
    };
    G2G_CHECK(p.precond == 0 || (learned && learned->apply), -4,
              "learned preconditioner requested but none is attached");
    // after `patience` learned steps in a row are rejected, the network is
    // not called again in this solve (the steps it would propose cost an
    // operator application and a network application each)
    int rejected_run = 0;
    bool learned_on = true, learned_used = false;
    auto note = [&](bool accepted) {
      rejected_run = accepted ? 0 : rejected_run + 1;
      if (p.learned_patience > 0 && rejected_run >= p.learned_patience) learned_on = false;
    };
    if (p.precond == 1) {
      // learned start + inner GMRES: c = M(v), scaled by the least-squares
      // factor alpha = <A c, v>/<A c, A c>; accepted when it cuts the
      // residual, ||v - alpha A c|| < accept ||v|| (inner precision), then
      // z = alpha c + inner GMRES on v - alpha A c; else plain inner GMRES.
      outer.precond = [&](const zd* v, zd* z) {
        if (!learned_on) {
          inner_gmres(v, z);
          return;
        }
        set_inner_tol();
        res.precond_calls++;
        learned->apply(learned->ctx, v, z);
        zc alpha;
        if (p.inner_precision == 0) {
          op_apply<double>(op, op.d64, z, tmp, op.stream, false);
          op.cnt.matvecs++;
          const double rn = fit_residual<zd, double>(blas, v, tmp, tmp, N, &alpha);
          const double vn = blas.norm<zd, double>(v, N);
          if (!(rn < learned->accept * vn)) {
            res.precond_fallbacks++;
            note(false);
            in64.solve(z, v, v);
            return;
          }
          note(true);
          blas.lincomb(z, z, N, 1, &alpha, false);
          in64.solve(tmp2, tmp, tmp);
          blas.add(z, tmp2, N);
        } else {
          blas.convert<zd, zf>(b32, v, N);
          blas.convert<zd, zf>(x32, z, N);
          op_apply<float>(op, op.d32, x32, r32, op.stream, false);
          op.cnt.matvecs32++;
          const double rn = fit_residual<zf, float>(blas, b32, r32, r32, N, &alpha);
          const double vn = blas.norm<zf, float>(b32, N);
          if (!(rn < learned->accept * vn)) {
            res.precond_fallbacks++;
            note(false);
            in32.solve(x32, b32, b32);
            blas.convert<zf, zd>(z, x32, N);
            return;
          }
          note(true);
          blas.lincomb(z, z, N, 1, &alpha, false);
          in32.solve(x32, r32, r32);
          blas.convert<zf, zd>(tmp, x32, N);
          blas.add(z, tmp, N);
        }
      };
    } else if (p.precond == 2) {
      // learned step only, z = M(v); the outer checks, with the A z it
      // computes anyway, that min_alpha ||v - alpha A z|| < accept ||v||
      // (FGMRES does not depend on the scale of z) and otherwise replaces
      // z by inner GMRES(v).
      outer.precond = [&](const zd* v, zd* z) {
        learned_used = learned_on;
        if (!learned_on) {
          inner_gmres(v, z);
          return;
        }
        res.precond_calls++;
        learned->apply(learned->ctx, v, z);
      };
      outer.accept_step = [&](const zd* v, const zd* Az) {
        if (!learned_used) return true;  // the step came from the inner GMRES
        zc alpha;
        const double rn = fit_residual<zd, double>(blas, v, Az, tmp, N, &alpha);
        const double vn = blas.norm<zd, double>(v, N);
        const bool ok = rn < learned->accept * vn;
        note(ok);
        if (!ok) res.precond_fallbacks++;
        return ok;
      };
      outer.fallback = inner_gmres;
    } else {
      outer.precond = inner_gmres;
    }
    SolveResult r = outer.solve(xout, x0, b);
    r.precond_calls = res.precond_calls;
    r.precond_fallbacks = res.precond_fallbacks;
    res = r;
    res.dots = blas.dots;
    res.passes = blas.passes;
    res.krylov_bytes = blas.bytes;
    if (!env) {
      op.cnt.dotprods += blas.dots;
      op.cnt.gs_passes += blas.passes;
      op.cnt.krylov_bytes += blas.bytes;
    }
  } catch (...) {
    (void)hipStreamSynchronize(st);  // nothing may still use the arena's buffers
    throw;
  }
  G2G_HIP(hipStreamSynchronize(st));
  return res;
}

// ------------------------------------------------------- paired solve ---
// Two independent solves with the same operator (the two polarizations of
// one frequency) run on two host threads, each with its own stream for the
// Krylov BLAS.  Their matrix-vector products meet in a rendezvous: when both
// wait for a product of the same precision, one two-vector apply serves both
// (op_apply2: the tensor is read once for two right-hand sides on the matrix
// cores); a thread whose partner has finished or waits for the other
// precision goes alone.  A requester's queued work ends before its request
// is posted, and the issuer waits for the product before either thread goes
// on; both waits poll an event (measured: event waits between the streams
// instead of host waits made the paired solves 5% slower, and blocking
// synchronisations wake the host about 50 us after the work ends).
namespace {
struct PairBatcher {
  Operator* op = nullptr;
  std::mutex mu;
  std::condition_variable cv;
  struct Req {
    const void* in = nullptr;
    void* out = nullptr;
    int prec = 0;
    bool pending = false, done = false;
    hipStream_t s = nullptr;     // the requester's stream
    hipEvent_t ready = nullptr;  // polled before the request is posted
  } r[2];
  hipEvent_t served = nullptr;   // polled after each product
  int poll_ms = poll_limit_ms();
  bool active[2] = {true, true};
  long long paired = 0, alone = 0;

  void run_one(const Req& q) {
    if (q.prec == 0) op_apply<double>(*op, op->d64, (const zd*)q.in, (zd*)q.out, op->stream, false);
    else op_apply<float>(*op, op->d32, (const zf*)q.in, (zf*)q.out, op->stream, false);
  }
  void apply(int me, const void* in, void* out, int prec) {
    poll_event(r[me].ready, r[me].s, poll_ms);  // s and ready do not change while the threads run
    std::unique_lock<std::mutex> lk(mu);
    Req& m = r[me];
    m.in = in;
    m.out = out;
    m.prec = prec;
    m.pending = true;
    m.done = false;
    const int ot = 1 - me;
    for (;;) {
      if (m.done) {
        m.done = false;
        return;
      }
      if (r[ot].pending || !active[ot]) {
        if (r[ot].pending && r[ot].prec == prec && op_pair_supported(*op)) {
          const Req& a = r[0];
          const Req& b = r[1];
          if (prec == 0)
            op_apply2<double>(*op, op->d64, (const zd*)a.in, (const zd*)b.in, (zd*)a.out, (zd*)b.out, op->stream);
          else
            op_apply2<float>(*op, op->d32, (const zf*)a.in, (const zf*)b.in, (zf*)a.out, (zf*)b.out, op->stream);
          paired++;
        } else {
          if (r[ot].pending) {
            run_one(r[ot]);
            alone++;
          }
          run_one(m);
          alone++;
        }
        poll_event(served, op->stream, poll_ms);
        if (r[ot].pending) {
          r[ot].pending = false;
          r[ot].done = true;
        }
        m.pending = false;
        cv.notify_all();
        return;
      }
      cv.wait(lk);
    }
  }
  // a worker that returns (or throws) withdraws any request it left, so the
  // other never runs a product on buffers that are freed
  void finish(int me) {
    std::lock_guard<std::mutex> lk(mu);
    active[me] = false;
    r[me].pending = false;
    r[me].done = false;
    cv.notify_all();
  }
};
}  // namespace

PairResult nested_solve_pair(Operator& op, const zd* const b[2], const zd* const x0[2], zd* const xout[2],
                             const SolveParams& p) {
  G2G_CHECK(p.precond == 0, -3, "paired solves use the inner GMRES preconditioner only");
  if (p.inner_precision != 0 && !op.have_g32) op_make_g32(op);
  G2G_HIP(hipStreamSynchronize(op.stream));
  PairBatcher pb;
  pb.op = &op;
  PairResult out;
  std::exception_ptr err[2];
  // streams and events exist before either thread starts (a request reads its
  // partner's); they are released after both threads have drained
  auto release = [&]() {
    for (auto& q : pb.r) {
      if (q.s) (void)hipStreamSynchronize(q.s);
      if (q.ready) (void)hipEventDestroy(q.ready);
      if (q.s) (void)hipStreamDestroy(q.s);
      q.s = nullptr;
      q.ready = nullptr;
    }
    if (pb.served) (void)hipEventDestroy(pb.served);
    pb.served = nullptr;
  };
  try {
    for (auto& q : pb.r) {
      G2G_HIP(hipStreamCreate(&q.s));
      G2G_HIP(hipEventCreateWithFlags(&q.ready, hipEventDisableTiming));
    }
    G2G_HIP(hipEventCreateWithFlags(&pb.served, hipEventDisableTiming));
  } catch (...) {
    release();
    throw;
  }
  auto worker = [&](int me) {
    const hipStream_t s = pb.r[me].s;
    try {
      SolveEnv env;
      env.stream = s;
      env.ws = &op.ws[me];
      env.mv64 = &out.mv64[me];
      env.mv32 = &out.mv32[me];
      env.A64 = [&, me](const zd* in, zd* o) { pb.apply(me, in, o, 0); };
      env.A32 = [&, me](const zf* in, zf* o) { pb.apply(me, in, o, 1); };
      out.r[me] = nested_solve(op, b[me], x0[me], xout[me], p, &out.hist[me], nullptr, &env);
    } catch (...) {
      err[me] = std::current_exception();
    }
    pb.finish(me);
  };
  std::thread t0(worker, 0), t1(worker, 1);
  t0.join();
  t1.join();
  (void)hipStreamSynchronize(op.stream);
  release();
  for (auto& e : err)
    if (e) std::rethrow_exception(e);
  out.paired = pb.paired;
  out.alone = pb.alone;
  op.cnt.matvecs += out.mv64[0] + out.mv64[1];
  op.cnt.matvecs32 += out.mv32[0] + out.mv32[1];
  for (int k = 0; k < 2; k++) {
    op.cnt.dotprods += out.r[k].dots;
    op.cnt.gs_passes += out.r[k].passes;
    op.cnt.krylov_bytes += out.r[k].krylov_bytes;
  }
  return out;
}

void solve_scale(Operator& op, zd* out, const zd* in, int mode) {
  const int64_t N = op.nvec();
  hipLaunchKernelGGL(k_rhs_scale, gridN(N), dim3(BT), 0, op.stream, out, in, op.d64.asiga, op.d64.sq,
                     (int64_t)op.Nx * op.Ny, op.Nz, N, mode);
  G2G_HIP(hipGetLastError());
}

}  // namespace g2g
