// g2g_unet.hip -- the learned right preconditioner on MI355X (gfx950).
//
// Network: 3-level 3D U-Net, widths 16/32/64, input 8 channels (residual
// re/im x 3, log10 contrast, log10 of the cell size in background
// wavenumbers), output 6 channels; 3x3x3
// convolutions with bias and ReLU, 2x2x2 average pooling, nearest
// upsampling, concatenation [upsampled, skip], a 1x1 output convolution.
// Volumes are channels-last [batch][z][y][x][C] in bf16.
//
// Convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16:
//   out[co][p] = bias[co] + sum_k W[co][k] X[k][p],  k = tap*Cin + ci,
// A = weights (16 output channels x 32 k), B = input (32 k x 16 voxels).
// Lane l of a wave holds A row l%16 / B column l%16 and the 8 consecutive
// k = 8*(l/16) .. 8*(l/16)+7, which is one 16-byte read of 8 channels of one
// tap (Cin is a multiple of 8) from the tile's copy in LDS; the FP32 result of lane l is rows
// 4*(l/16) .. 4*(l/16)+3 of column l%16 -- four consecutive output channels
// of one voxel, stored as one 8-byte bf16 write.  The data gradient is the
// same kernel run on the transposed, tap-flipped weights; the weight
// gradient (k_dw) takes exact products and FP32 sums.  No reference counterpart:
// GFGMRES/seq_fgmres.F90:142-152 preconditions with an inner GMRES.
#include <cmath>
#include <complex>
#include <cstring>
#include <vector>

#include "g2g_op.hpp"
#include "g2g_unet.hpp"

namespace g2g {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int UB = 256;

int64_t up_to(int64_t a, int64_t m) { return (a + m - 1) / m * m; }
unsigned nblk(int64_t n, int b = UB) { return (unsigned)((n + b - 1) / b); }

struct Src {
  const bf16* p;
  int C;
  int up;  // 1: the source is at half resolution (nearest upsampling)
  int64_t bstride;
};

struct ConvArgs {
  Src s1, s2;
  const bf16* w;
  int kp, ntap, cin;
  const float* bias;
  int cout, relu;
  bf16* ybf;
  float* yf;
  int ldy;
  int64_t ybstride;
  int nx, ny, nz;
  // input layer: the caller's FP32 volume instead of s1.p (or null)
  const float* xf;
  // the 1x1 output layer applied to this layer's result (16 channels): its
  // weight fragment, bias and FP32 result of cout2 channels (or null)
  const bf16* w2;
  const float* bias2;
  float* y2;
  int cout2;
};

// bias, ReLU and store of four consecutive output channels of one voxel (all
// outputs stored here have a multiple of four channels, conv_launch)
__device__ inline void conv_store(const ConvArgs& a, f32x4 c, int co0, int64_t p, int bat) {
  if (co0 >= a.cout) return;
  float o[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    o[q] = c[q] + ((a.bias && co0 + q < a.cout) ? a.bias[co0 + q] : 0.f);
    if (a.relu) o[q] = fmaxf(o[q], 0.f);
  }
  if (a.ybf) {
    const bf16x4 b = {(bf16)o[0], (bf16)o[1], (bf16)o[2], (bf16)o[3]};
    *reinterpret_cast<bf16x4*>(a.ybf + bat * a.ybstride + p * a.ldy + co0) = b;
  } else {
    *reinterpret_cast<f32x4*>(a.yf + bat * a.ybstride + p * a.ldy + co0) = f32x4{o[0], o[1], o[2], o[3]};
  }
}

// A convolution tile of (1 << lx, 1 << ly, 1 << lz) voxels: tile counts, the
// voxels with the rim, the plane stride of the LDS copy, and multipliers for
// division by the rim's row and plane sizes (exact for v < 2048); the same
// for an upsampled source's rim at half resolution.  Matrix column group
// n = sum of s[k] over the set bits k of (wave, g): the groups of one wave
// share the parities of their voxels' coordinates.
struct ConvBox {
  int hx, hy, hvox, hv;
  unsigned mx, mxy;
};
struct ConvTile {
  int lx, ly, lz, ntx, nty, nt;
  ConvBox f, h;
  int sg[2], sw[2];
};

// 1x1 convolutions (27-tap ones: k_conv3 below).  One wave: 16 output
// channels x 64 voxels (4 MFMA columns), one k-step; HBM bound.
__global__ __launch_bounds__(UB) void k_conv1x1(ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kq = lane >> 4;
  const int nvox = a.nx * a.ny * a.nz;
  const int pbase = (blockIdx.x * 4 + wave) * 64;
  const int cb = blockIdx.y, bat = blockIdx.z;
  const bf16* x1 = a.s1.p + bat * a.s1.bstride;
  const bf16x8 af = *reinterpret_cast<const bf16x8*>(a.w + ((int64_t)cb * 64 + lane) * 8);
  const int k0 = kq * 8;
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int p = pbase + s * 16 + col;
    bf16x8 bfr = {0, 0, 0, 0, 0, 0, 0, 0};
    if (k0 < a.cin && p < nvox) bfr = *reinterpret_cast<const bf16x8*>(x1 + (int64_t)p * a.cin + k0);
    f32x4 c = {0, 0, 0, 0};
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr, c, 0, 0, 0);
    if (p < nvox) conv_store(a, c, cb * 16 + kq * 4, (int64_t)p, bat);
  }
}

// FP32 input rounded to bf16 on the way
__device__ inline bf16x8 to_bf16x8(const float* x) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(x), b = *reinterpret_cast<const f32x4*>(x + 4);
  return bf16x8{(bf16)a[0], (bf16)a[1], (bf16)a[2], (bf16)a[3], (bf16)b[0], (bf16)b[1], (bf16)b[2], (bf16)b[3]};
}

// Copies the tile's box at (X0, Y0, Z0) of a source to planes of 8 channels, zero outside the volume
template <int NCH, typename T>
__device__ inline void conv_stage(bf16x8* xs, const ConvBox& b, const T* x, int X0, int Y0, int Z0, int nx, int ny,
                                  int nz, int tid) {
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
  for (int e = tid; e < b.hvox * NCH; e += UB) {
    const int v = e / NCH, ch = e - v * NCH;
    const int vz = (int)(((unsigned)v * b.mxy) >> 20), vr = v - vz * b.hx * b.hy;
    const int vy = (int)(((unsigned)vr * b.mx) >> 20), vx = vr - vy * b.hx;
    const int X = X0 + vx, Y = Y0 + vy, Z = Z0 + vz;
    const bool in = X >= 0 && X < nx && Y >= 0 && Y < ny && Z >= 0 && Z < nz;
    // the load is unconditional, from a clamped voxel, so that several are in flight
    const int Xc = min(max(X, 0), nx - 1), Yc = min(max(Y, 0), ny - 1), Zc = min(max(Z, 0), nz - 1);
    const T* xp = x + (((int64_t)Zc * ny + Yc) * nx + Xc) * (NCH * 8) + ch * 8;
    bf16x8 val;
    if constexpr (sizeof(T) == 4) val = to_bf16x8(xp);
    else val = *reinterpret_cast<const bf16x8*>(xp);
    xs[ch * b.hv + v] = in ? val : zero;
  }
}

constexpr int conv_g(int cin) { return cin >= 64 ? 2 : 4; }

// 3x3x3 convolution, CIN input channels, CT x 16 output channels, a tile of
// 64 G voxels (4 waves of 16 G voxels x all output channels).
// The tile with its one-voxel rim is copied to LDS once, zero outside the
// volume, concatenated and upsampled on the way, in planes of 8 channels
// ([chunk][voxel], 16 bytes each): the 16 lanes of a matrix column then read
// 16 neighbouring voxels without bank conflicts, and a tap is an offset added
// to the lane's own voxel (a 4-byte table entry per k-step and lane quarter)
// instead of the three bounds checks, the address and the global gather that
// each fragment took when every wave read its input from memory: that kernel
// ran at 0.10-0.17 of the matrix rate with the vector unit busy on addresses.
// Every fragment read from LDS feeds the CT output tiles.  LDS bandwidth
// bounds it (16 bytes a lane per CT products).  Measured at 256x256x32, all
// layers of one forward pass: 1508 -> 585 us (251 GFLOP, 0.17 -> 0.43
// PFLOP/s; 48 -> 16 channels 0.60 PFLOP/s); the whole pass 1541 -> 597 us
// with the input conversion and the 1x1 output layer done on the way.  The
// sums run over k in the same order and instruction as before, so the results
// are the same bit for bit.
// Weights: fragment order [co tile][k-step][lane][8], one contiguous 1 KB
// load per k-step and tile.
// An upsampled source (its first UPC channels) is kept in LDS at half
// resolution: a quarter to an eighth of the bytes, so that three to five
// blocks share a CU instead of one or two (48 channels 270 -> 143 us, 96
// channels 173 -> 81 us).  Its offset of a tap depends on the parity of the
// voxel's coordinates (eight table entries per k-step).
template <int CIN, int CT, int UPC>
__global__ __launch_bounds__(UB) void k_conv3(ConvArgs a, ConvTile t) {
  constexpr int G = conv_g(CIN), NKS = (27 * CIN + 31) / 32, NU = UPC / 8, NF = CIN / 8 - NU;
  constexpr int NPAR = UPC ? 8 : 1;
  constexpr bool TAIL = (27 * CIN) % 32 != 0;
  extern __shared__ unsigned char conv_sm[];
  bf16x8* xs = reinterpret_cast<bf16x8*>(conv_sm);  // half-resolution planes, then the full ones
  const int full0 = NU * t.h.hv;
  // offset of the k-step's chunk and tap for lane quarter kq and voxel
  // parity; bit 15: of an upsampled source; 0xffff: past the last tap
  unsigned short* tab = reinterpret_cast<unsigned short*>(conv_sm + sizeof(bf16x8) * (full0 + NF * t.f.hv));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, kq = lane >> 4;
  // consecutive workgroups go round-robin to the eight XCDs: each XCD gets a
  // run of neighbouring tiles, whose rims meet in its L2
  int tile;
  {
    const int n = gridDim.x, q = n >> 3, r = n & 7, x = blockIdx.x & 7, i = blockIdx.x >> 3;
    tile = x * q + (x < r ? x : r) + i;
  }
  const int bat = tile / t.nt;
  tile -= bat * t.nt;
  const int tz0 = tile / (t.ntx * t.nty), ty0 = (tile / t.ntx) % t.nty, tx0 = tile % t.ntx;
  const int x0 = tx0 << t.lx, y0 = ty0 << t.ly, z0 = tz0 << t.lz;
  for (int i = tid; i < NKS * 4 * NPAR; i += UB) {
    const int par = i % NPAR, e = i / NPAR, k0 = (e >> 2) * 32 + (e & 3) * 8, tap = k0 / CIN, ch = (k0 - tap * CIN) >> 3;
    const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;
    int off = 0xffff;
    if (tap < 27) {
      if (ch < NU)  // voxel 2a + p with tap d reads half voxel a + (p + d + 1) / 2 of the rim
        off = 0x8000 | (ch * t.h.hv + ((((par >> 2) + dz + 1) >> 1) * t.h.hy + ((((par >> 1) & 1) + dy + 1) >> 1)) * t.h.hx +
                        (((par & 1) + dx + 1) >> 1));
      else
        off = full0 + (ch - NU) * t.f.hv + (dz * t.f.hy + dy) * t.f.hx + dx;
    }
    tab[i] = (unsigned short)off;
  }
  if constexpr (UPC > 0) {
    conv_stage<NU>(xs, t.h, a.s1.p + bat * a.s1.bstride, (x0 >> 1) - 1, (y0 >> 1) - 1, (z0 >> 1) - 1, a.nx >> 1,
                   a.ny >> 1, a.nz >> 1, tid);
    conv_stage<NF>(xs + full0, t.f, a.s2.p + bat * a.s2.bstride, x0 - 1, y0 - 1, z0 - 1, a.nx, a.ny, a.nz, tid);
  } else {
    if (CIN == 8 && a.xf)
      conv_stage<NF>(xs, t.f, a.xf + bat * a.s1.bstride, x0 - 1, y0 - 1, z0 - 1, a.nx, a.ny, a.nz, tid);
    else
      conv_stage<NF>(xs, t.f, a.s1.p + bat * a.s1.bstride, x0 - 1, y0 - 1, z0 - 1, a.nx, a.ny, a.nz, tid);
  }
  __syncthreads();
  int base[G], baseh[G], vx[G], vy[G], vz[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int n = (g & 1) * t.sg[0] + (g >> 1) * t.sg[1] + (wave & 1) * t.sw[0] + (wave >> 1) * t.sw[1];
    const int v = n * 16 + col;
    vx[g] = v & ((1 << t.lx) - 1);
    vy[g] = (v >> t.lx) & ((1 << t.ly) - 1);
    vz[g] = v >> (t.lx + t.ly);
    base[g] = (vz[g] * t.f.hy + vy[g]) * t.f.hx + vx[g];
    baseh[g] = ((vz[g] >> 1) * t.h.hy + (vy[g] >> 1)) * t.h.hx + (vx[g] >> 1);
  }
  const int par = UPC ? (vx[0] & 1) + 2 * (vy[0] & 1) + 4 * (vz[0] & 1) : 0;  // the same for every g
  f32x4 acc[CT][G];
#pragma unroll
  for (int c = 0; c < CT; c++)
#pragma unroll
    for (int g = 0; g < G; g++) acc[c][g] = f32x4{0, 0, 0, 0};
  const bf16x8* wf = reinterpret_cast<const bf16x8*>(a.w) + lane;
  constexpr int NFULL = TAIL ? NKS - 1 : NKS;
#pragma unroll 3
  for (int ks = 0; ks < NFULL; ks++) {
    const int off = tab[(ks * 4 + kq) * NPAR + par], o = off & 0x7fff;
    const bool up = UPC > 0 && (off & 0x8000);
    bf16x8 af[CT];
#pragma unroll
    for (int c = 0; c < CT; c++) af[c] = wf[(c * NKS + ks) * 64];
#pragma unroll
    for (int g = 0; g < G; g++) {
      const bf16x8 b = xs[(up ? baseh[g] : base[g]) + o];
#pragma unroll
      for (int c = 0; c < CT; c++) acc[c][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[c], b, acc[c][g], 0, 0, 0);
    }
  }
  if constexpr (TAIL) {  // k past the 27th tap: zero input
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    const int off = tab[(NFULL * 4 + kq) * NPAR + par];
    const bool past = off == 0xffff, up = UPC > 0 && !past && (off & 0x8000);
    const int o = past ? 0 : off & 0x7fff;
#pragma unroll
    for (int g = 0; g < G; g++) {
      const bf16x8 v = xs[(up ? baseh[g] : base[g]) + o];
      const bf16x8 b = past ? zero : v;
#pragma unroll
      for (int c = 0; c < CT; c++)
        acc[c][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[(c * NKS + NFULL) * 64], b, acc[c][g], 0, 0, 0);
    }
  }
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int X = x0 + vx[g], Y = y0 + vy[g], Z = z0 + vz[g];
    const bool in = X < a.nx && Y < a.ny && Z < a.nz;
    const int64_t p = ((int64_t)Z * a.ny + Y) * a.nx + X;
    if (in && (a.ybf || a.yf)) {
#pragma unroll
      for (int c = 0; c < CT; c++) conv_store(a, acc[c][g], c * 16 + kq * 4, p, bat);
    }
    if constexpr (CIN == 16 && CT == 1) {
      if (a.w2) {
        // the 1x1 layer's operand: lane quarter kq < 2 takes channels 8 kq ..
        // 8 kq + 7 of its voxel from quarters 2 kq and 2 kq + 1
        bf16x4 o;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float v = acc[0][g][q] + (a.bias ? a.bias[kq * 4 + q] : 0.f);
          o[q] = (bf16)(a.relu ? fmaxf(v, 0.f) : v);
        }
        const int2 w = __builtin_bit_cast(int2, o);
        const int l0 = (col + 32 * kq) & 63, l1 = (l0 + 16) & 63;
        const int4 u = {__shfl(w.x, l0), __shfl(w.y, l0), __shfl(w.x, l1), __shfl(w.y, l1)};
        const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
        const bf16x8 b = kq < 2 ? __builtin_bit_cast(bf16x8, u) : zero;
        f32x4 r = {0, 0, 0, 0};
        r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(reinterpret_cast<const bf16x8*>(a.w2)[lane], b, r, 0, 0, 0);
        if (in) {
          float* y = a.y2 + ((int64_t)bat * a.nx * a.ny * a.nz + p) * a.cout2;
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (kq * 4 + q < a.cout2) y[kq * 4 + q] = r[q] + a.bias2[kq * 4 + q];
        }
      }
    }
  }
}

// Weight gradient dW[co][t][ci] = sum_p dZ[p][co] X[p+off(t)][ci] and db[co] =
// sum_p dZ[p][co] on v_mfma_f32_16x16x32_bf16: 16 co x 16 ci tiles, 32 voxels
// (two x rows of 16) per instruction.  X is bf16; dZ is FP32 and enters as
// three bf16 numbers of 8 bits each (h + m + l = dZ exactly), so every product
// is exact and the sums are FP32, as in the FP32 vector kernel this replaces.
// A tile of 16 x 4 x 2 voxels is transposed into LDS once, [ci][row][x] and
// [part][co][row][x], 8 voxels per 16-byte read; the x taps of a row are its
// 16-byte chunk shifted by one element into or out of the neighbouring dwords,
// the y and z taps other rows.  Wave (dz, ci tile) accumulates its 9 taps x
// NCO tiles in registers over all tiles of the block; each block writes its
// sums to a slot of its own, which k_dw_reduce adds in a fixed order (the
// sums no longer depend on the order of atomics).  The parts m and l have
// accumulators of their own, which keeps their roundings out of the large
// sums.  A part is often zero where dZ is not, and the places of a tile outside
// the volume have dZ = 0, so an infinite or NaN activation would turn sums into
// NaN there that have none: from a block's first tile with such an X on, the
// sums are taken over the voxels of the volume with FP32 dZ itself (gradient at
// 8 x 64x64x16 1435 us without, 1411 us with the check of the exponents on
// their way to LDS).  Strides of an odd number of 16-byte units spread the 16 channels of a
// read over the banks.  The transposition and the LDS reads bound it (matrix
// cores about a fifth busy).  Measured at 8 x 64x64x16, all layers: 7910 us on
// the FP32 vector unit with atomics -> 520 us; error of the sums against FP64
// 4.4e-7 -> 0.6e-7.
struct DwArgs {
  const float* dz;
  int ldz, cout;
  Src s1, s2;
  int cin, ntap;
  float* part;
  int64_t pstride;  // cout*ntap*cin + cout
  int nx, ny, nz, ntx, nty, nt, ntot;
};
constexpr int DW_XROW = 24;                 // 16 voxels, then (-, x = -1), (x = 16, -) of a row
constexpr int DW_XST = 24 * DW_XROW + 8;    // 24 rows (6 y, 4 z) of a channel
constexpr int DW_ZST = 8 * 16 + 8;          // 8 rows (4 y, 2 z) of a channel

template <int NCO, int NCI, bool ONE>
__global__ __launch_bounds__(192 * NCI) void k_dw(DwArgs a) {
  constexpr int NT = 192 * NCI, NCH = 2 * NCI;
  extern __shared__ __align__(16) unsigned char dw_sm[];
  bf16* xs = reinterpret_cast<bf16*>(dw_sm);
  bf16* zs = xs + NCI * 16 * DW_XST;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, kq = lane >> 4, half = kq & 1;
  const int dzi = ONE ? 1 : wave % 3, cit = ONE ? 0 : wave / 3;
  const int c0 = blockIdx.y * NCI * 16, o0 = blockIdx.z * NCO * 16;
  const int nxh = a.nx >> 1, nyh = a.ny >> 1;
  const bool bias = ONE || (dzi == 1 && cit == 0 && blockIdx.y == 0);
  constexpr int NTAP = ONE ? 1 : 9;
  f32x4 acc[2][NTAP][NCO], bacc[2][NCO];  // [0]: the leading part h, [1]: m and l
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int t = 0; t < NCO; t++) {
      bacc[h][t] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < NTAP; k++) acc[h][k][t] = f32x4{0, 0, 0, 0};
    }
  __shared__ int special;  // a tile had an infinite or NaN activation
  if (tid == 0) special = 0;
  __syncthreads();
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16 one1 = (bf16)1.f;
  const bf16x8 ones = {one1, one1, one1, one1, one1, one1, one1, one1};
  const int first = (int)((int64_t)a.ntot * blockIdx.x / gridDim.x);
  const int last = (int)((int64_t)a.ntot * (blockIdx.x + 1) / gridDim.x);
  for (int tile = first; tile < last; tile++) {
    const int bat = tile / a.nt, tt = tile - bat * a.nt;
    const int z0 = tt / (a.ntx * a.nty) * 2, y0 = (tt / a.ntx) % a.nty * 4, x0 = tt % a.ntx * 16;
    // one voxel's 8 channels of chunk c (zero outside the volume); the load is
    // unconditional, from a clamped voxel
    auto ldx = [&](int c, int X, int Y, int Z) -> bf16x8 {
      const int ci = c0 + c * 8;
      const bool in = ci < a.cin && X >= 0 && X < a.nx && Y >= 0 && Y < a.ny && Z >= 0 && Z < a.nz;
      const int Xc = min(max(X, 0), a.nx - 1), Yc = min(max(Y, 0), a.ny - 1), Zc = min(max(Z, 0), a.nz - 1);
      const int cc = ci < a.cin ? ci : 0;
      const bool f = cc < a.s1.C;
      const Src& sr = f ? a.s1 : a.s2;
      const int64_t q = sr.up ? ((int64_t)(Zc >> 1) * nyh + (Yc >> 1)) * nxh + (Xc >> 1)
                              : ((int64_t)Zc * a.ny + Yc) * a.nx + Xc;
      const bf16x8 v =
          *reinterpret_cast<const bf16x8*>(sr.p + bat * sr.bstride + q * sr.C + (f ? cc : cc - a.s1.C));
      return in ? v : zero;
    };
    unsigned exps = 0;  // bit 15 of a half: an exponent of all ones was there
    auto check = [&](const bf16x8& v) {
      const uint4 u = __builtin_bit_cast(uint4, v);
      exps |= ((u.x & 0x7f807f80u) + 0x00800080u) | ((u.y & 0x7f807f80u) + 0x00800080u) |
              ((u.z & 0x7f807f80u) + 0x00800080u) | ((u.w & 0x7f807f80u) + 0x00800080u);
    };
    for (int e = tid; e < 48 * NCH; e += NT) {
      const int c = e % NCH, r = e / NCH, h8 = (r & 1) * 8, row = r >> 1, hy = row % 6, hz = row / 6;
      bf16x8 v[8];
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = ldx(c, x0 + h8 + j, y0 + hy - 1, z0 + hz - 1);
#pragma unroll
      for (int j = 0; j < 8; j++) check(v[j]);
      bf16* dst = xs + c * 8 * DW_XST + row * DW_XROW + h8;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const bf16x8 o = {v[0][k], v[1][k], v[2][k], v[3][k], v[4][k], v[5][k], v[6][k], v[7][k]};
        *reinterpret_cast<bf16x8*>(dst + k * DW_XST) = o;
      }
    }
    if constexpr (!ONE) {
      for (int e = tid; e < 48 * NCH; e += NT) {
        const int c = e % NCH, r = e / NCH, side = r & 1, row = r >> 1, hy = row % 6, hz = row / 6;
        const bf16x8 v = ldx(c, side ? x0 + 16 : x0 - 1, y0 + hy - 1, z0 + hz - 1);
        check(v);
        bf16* dst = xs + c * 8 * DW_XST + row * DW_XROW + 17 + side;
#pragma unroll
        for (int k = 0; k < 8; k++) dst[k * DW_XST] = v[k];
      }
    }
    for (int e = tid; e < 64 * NCO; e += NT) {
      const int q = e % (4 * NCO), r = e / (4 * NCO), h8 = (r & 1) * 8, row = r >> 1, co = o0 + q * 4;
      const int Y = y0 + (row & 3), Z = z0 + (row >> 2);
      const bool in = co < a.ldz && Y < a.ny && Z < a.nz;
      const float* src = a.dz + (((int64_t)bat * a.nz + min(Z, a.nz - 1)) * a.ny + min(Y, a.ny - 1)) * a.nx * a.ldz +
                         (co < a.ldz ? co : 0);
      f32x4 v[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int X = x0 + h8 + j;
        const f32x4 g = *reinterpret_cast<const f32x4*>(src + (int64_t)min(X, a.nx - 1) * a.ldz);
        v[j] = in && X < a.nx ? g : f32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        bf16x8 p0, p1, p2;
#pragma unroll
        for (int j = 0; j < 8; j++) {
          // h, m: the leading 8 bits of v and of the rest (truncated, so that
          // both rests are exact); an infinity or NaN goes into h alone
          const float x = v[j][i];
          const unsigned u = __float_as_uint(x);
          const bool fin = (u & 0x7f800000u) != 0x7f800000u;
          const float h = __uint_as_float(u & 0xffff0000u);
          const float r1 = fin ? x - h : 0.f;
          const float m = __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
          p0[j] = (bf16)(fin ? h : x);
          p1[j] = (bf16)m;
          p2[j] = (bf16)(r1 - m);
        }
        bf16* dst = zs + (q * 4 + i) * DW_ZST + row * 16 + h8;
        *reinterpret_cast<bf16x8*>(dst) = p0;
        *reinterpret_cast<bf16x8*>(dst + NCO * 16 * DW_ZST) = p1;
        *reinterpret_cast<bf16x8*>(dst + 2 * NCO * 16 * DW_ZST) = p2;
      }
    }
    if (exps & 0x80008000u) special = 1;
    __syncthreads();
    const bool plain = __builtin_amdgcn_readfirstlane(special) == 0;
    if (!plain) {
      for (int row = 0; row < 8; row++) {
        const int y = row & 3, z = row >> 2;
        if (y0 + y >= a.ny || z0 + z >= a.nz || (ONE && (row >> 1) % 3 != wave)) continue;
        for (int x = 0; x < 16 && x0 + x < a.nx; x++) {
          const float* d =
              a.dz + ((((int64_t)bat * a.nz + z0 + z) * a.ny + y0 + y) * a.nx + x0 + x) * a.ldz + o0 + kq * 4;
          f32x4 g[NCO];
#pragma unroll
          for (int t = 0; t < NCO; t++)
            g[t] = o0 + t * 16 + kq * 4 < a.ldz ? *reinterpret_cast<const f32x4*>(d + t * 16) : f32x4{0, 0, 0, 0};
#pragma unroll
          for (int k = 0; k < NTAP; k++) {
            const int dy = ONE ? 1 : k / 3, xx = ONE ? x : x + k % 3 - 1;
            const bf16* r = xs + (cit * 16 + col) * DW_XST + ((z + dzi) * 6 + y + dy) * DW_XROW;
            const float v = (float)r[xx < 0 ? 17 : (xx > 15 ? 18 : xx)];
#pragma unroll
            for (int t = 0; t < NCO; t++) acc[0][k][t] += g[t] * v;
          }
          if (bias) {
#pragma unroll
            for (int t = 0; t < NCO; t++) bacc[0][t] += g[t];
          }
        }
      }
    }
    for (int s = plain ? (ONE ? wave : 0) : 4; s < 4; s += ONE ? 3 : 1) {
      const int z = s >> 1, y = (s & 1) * 2 + (kq >> 1);
      bf16x8 af[3][NCO];
#pragma unroll
      for (int p = 0; p < 3; p++)
#pragma unroll
        for (int t = 0; t < NCO; t++)
          af[p][t] = *reinterpret_cast<const bf16x8*>(zs + ((p * NCO + t) * 16 + col) * DW_ZST + (z * 4 + y) * 16 + half * 8);
#pragma unroll
      for (int dy = ONE ? 1 : 0; dy < (ONE ? 2 : 3); dy++) {
        const bf16* row = xs + (cit * 16 + col) * DW_XST + ((z + dzi) * 6 + y + dy) * DW_XROW;
        const bf16x8 bc = *reinterpret_cast<const bf16x8*>(row + half * 8);
        if constexpr (ONE) {
#pragma unroll
          for (int t = 0; t < NCO; t++)
#pragma unroll
            for (int p = 2; p >= 0; p--) acc[p > 0][0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[p][t], bc, acc[p > 0][0][t], 0, 0, 0);
        } else {
          const unsigned prev = *reinterpret_cast<const unsigned*>(row + (half ? 6 : 16));
          const unsigned next = *reinterpret_cast<const unsigned*>(row + (half ? 18 : 8));
          const uint4 c = __builtin_bit_cast(uint4, bc);
          const unsigned m0 = __builtin_amdgcn_alignbit(c.x, prev, 16), m1 = __builtin_amdgcn_alignbit(c.y, c.x, 16),
                         m2 = __builtin_amdgcn_alignbit(c.z, c.y, 16), m3 = __builtin_amdgcn_alignbit(c.w, c.z, 16),
                         m4 = __builtin_amdgcn_alignbit(next, c.w, 16);
          const bf16x8 bx[3] = {__builtin_bit_cast(bf16x8, uint4{m0, m1, m2, m3}), bc,
                                __builtin_bit_cast(bf16x8, uint4{m1, m2, m3, m4})};
#pragma unroll
          for (int p = 2; p >= 0; p--)
#pragma unroll
            for (int dx = 0; dx < 3; dx++)
#pragma unroll
              for (int t = 0; t < NCO; t++)
                acc[p > 0][dy * 3 + dx][t] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[p][t], bx[dx], acc[p > 0][dy * 3 + dx][t], 0, 0, 0);
        }
      }
      if (bias) {
#pragma unroll
        for (int t = 0; t < NCO; t++)
#pragma unroll
          for (int p = 2; p >= 0; p--)
            bacc[p > 0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[p][t], ones, bacc[p > 0][t], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // lane (col, kq) holds input channel col and output channels 4 kq + q of each tile
  float* part = a.part + (ONE ? (int64_t)blockIdx.x * 3 + wave : (int64_t)blockIdx.x) * a.pstride;
  const int ci = c0 + cit * 16 + col;
#pragma unroll
  for (int t = 0; t < NCO; t++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int co = o0 + t * 16 + kq * 4 + q;
      if (co >= a.cout) continue;
      if (ci < a.cin) {
#pragma unroll
        for (int k = 0; k < NTAP; k++) part[((int64_t)co * a.ntap + (ONE ? 0 : dzi * 9 + k)) * a.cin + ci] = acc[0][k][t][q] + acc[1][k][t][q];
      }
      if (bias && col == 0) part[(int64_t)a.cout * a.ntap * a.cin + co] = bacc[0][t][q] + bacc[1][t][q];
    }
}

// g[i] = sum over the np slots of part[slot][i], in a fixed order, in double:
// 64 sums per block, 16 threads each (4 threads each left most of the chip
// idle: 123 us a gradient at 8 x 64x64x16, 8 threads 83, 16 threads 76)
constexpr int DWR = 16;
__global__ __launch_bounds__(64 * DWR) void k_dw_reduce(const float* __restrict__ part, int np, int64_t n, float* __restrict__ g) {
  __shared__ double red[DWR][64];
  const int t = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + t;
  double s = 0;
  if (i < n) {
#pragma unroll 8
    for (int k = w; k < np; k += DWR) s += (double)part[k * n + i];
  }
  red[w][t] = s;
  __syncthreads();
  if (w == 0 && i < n) {
    double sum = 0;
    for (int k = 0; k < DWR; k++) sum += red[k][t];
    g[i] = (float)sum;
  }
}

// forward weights w[co][tap*cin+ci] and transposed weights
// wt[ci][tap'*coutT+co] = W[co][ntap-1-tap'][ci] (bf16, zero padded), both in
// fragment order: element j of lane l in k-step s of output tile c, at
// ((c*nks + s)*64 + l)*8 + j, is row 16c + l%16, column 32s + 8(l/16) + j
__device__ inline void frag_rc(int64_t i, int kp, int* row, int* k) {
  const int j = (int)(i & 7), l = (int)(i >> 3) & 63, nks = kp / 32;
  const int cs = (int)(i >> 9), s = cs % nks, c = cs / nks;
  *row = c * 16 + (l & 15);
  *k = s * 32 + (l >> 4) * 8 + j;
}
__global__ void k_wprep(const float* __restrict__ W, int cout, int cin, int ntap, bf16* w, int coutP,
                        int kp, bf16* wt, int cinP, int coutT, int kpT) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n1 = (int64_t)coutP * kp, n2 = (int64_t)cinP * kpT;
  if (i < n1) {
    int co, k;
    frag_rc(i, kp, &co, &k);
    const int t = k / cin, ci = k % cin;
    float v = 0.f;
    if (co < cout && t < ntap) v = W[((int64_t)co * ntap + t) * cin + ci];
    w[i] = (bf16)v;
  } else if (i < n1 + n2) {
    const int64_t j = i - n1;
    int ci, k;
    frag_rc(j, kpT, &ci, &k);
    const int tp = k / coutT, co = k % coutT;
    float v = 0.f;
    if (ci < cin && tp < ntap && co < cout) v = W[((int64_t)co * ntap + (ntap - 1 - tp)) * cin + ci];
    wt[j] = (bf16)v;
  }
}

// 2x2x2 average pooling, 8 channels per thread
__global__ void k_pool(const bf16* __restrict__ src, bf16* __restrict__ dst, int C, int nx, int ny,
                       int nz, int64_t nb) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nxh = nx / 2, nyh = ny / 2, nzh = nz / 2;
  const int C8 = C / 8;
  const int64_t nc = (int64_t)nxh * nyh * nzh;
  if (i >= nb * nc * C8) return;
  const int c8 = (int)(i % C8);
  const int64_t q = (i / C8) % nc, bat = i / (C8 * nc);
  const int x = (int)(q % nxh), y = (int)((q / nxh) % nyh), z = (int)(q / ((int64_t)nxh * nyh));
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16* sb = src + bat * (int64_t)nx * ny * nz * C;
  for (int d = 0; d < 8; d++) {
    const int X = 2 * x + (d & 1), Y = 2 * y + ((d >> 1) & 1), Z = 2 * z + (d >> 2);
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(sb + (((int64_t)Z * ny + Y) * nx + X) * C + c8 * 8);
#pragma unroll
    for (int k = 0; k < 8; k++) s[k] += (float)v[k];
  }
  bf16x8 o;
#pragma unroll
  for (int k = 0; k < 8; k++) o[k] = (bf16)(s[k] * 0.125f);
  *reinterpret_cast<bf16x8*>(dst + (bat * nc + q) * C + c8 * 8) = o;
}

// dz = g * (y > 0) (or g when y is null), FP32 and bf16 copies, four channels
// per thread; channels c >= C of the copies (row length Cp = 4 << sh) are zero.
// The gradient g of the layer's output, taken from where the other layers left
// it, so that it needs no pass of its own:
//   GradPlain     g = dy (rows of ldy)
//   GradUpsample  the output went, upsampled, into a concatenation: the sum of
//                 its eight children in dy, the concatenation's gradient
//   GradPool      the output went into a concatenation and a pooling: dy (the
//                 concatenation's part) plus an eighth of dc, the pooled one's
// Memory bounds it: with the sums and copies in kernels of their own, an
// element and two 64-bit divisions per thread, 240 us of a gradient at 8 x
// 64x64x16, now 132.
enum GradSource { GradPlain, GradUpsample, GradPool };
// The grid's y axis takes the layers z, so the rows beyond its limit (GRID_Y_MAX,
// long volumes) are a second turn of the loop.
constexpr int GRID_Y_MAX = 65535;
template <GradSource SRC>
__global__ void k_relu_back(const float* __restrict__ dy, int ldy, const float* __restrict__ dc, const bf16* __restrict__ y,
                            int C, int sh, float* __restrict__ dzf, bf16* __restrict__ dzb, int nx, int ny, int nz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int xy = i >> sh, c = (i & ((1 << sh) - 1)) * 4;
  if (xy >= nx * ny) return;
  const int64_t bat = blockIdx.z;
  for (int z = blockIdx.y; z < nz; z += gridDim.y) {
    const int64_t p = (bat * nz + z) * nx * ny + xy;
    f32x4 g;
    if constexpr (SRC == GradUpsample) {
      const int yy = xy / nx, x = xy - yy * nx;
      g = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int d = 0; d < 8; d++) {
        const int X = 2 * x + (d & 1), Y = 2 * yy + ((d >> 1) & 1), Z = 2 * z + (d >> 2);
        g += *reinterpret_cast<const f32x4*>(dy + (((bat * 2 * nz + Z) * 2 * ny + Y) * 2 * nx + X) * ldy + c);
      }
    } else {
      g = *reinterpret_cast<const f32x4*>(dy + p * ldy + c);
      if constexpr (SRC == GradPool) {
        const int yy = xy / nx, x = xy - yy * nx;
        const int64_t q = ((bat * (nz / 2) + z / 2) * (ny / 2) + yy / 2) * (nx / 2) + x / 2;
        g += 0.125f * *reinterpret_cast<const f32x4*>(dc + q * C + c);
      }
    }
    if (y) {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(y + p * C + c);
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (!((float)v[k] > 0.f)) g[k] = 0.f;
    }
    bf16x4 o;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (c + k >= C) g[k] = 0.f;
      o[k] = (bf16)g[k];
    }
    const int64_t at = (p << (sh + 2)) + c;
    *reinterpret_cast<f32x4*>(dzf + at) = g;
    *reinterpret_cast<bf16x4*>(dzb + at) = o;
  }
}

// n voxels of 8 channels; VEC: a is 16-byte aligned
template <bool VEC> __global__ void k_f32_to_bf16(const float* __restrict__ a, bf16* __restrict__ b, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bf16x8 o;
  if constexpr (VEC) {
    o = to_bf16x8(a + i * 8);
  } else {
#pragma unroll
    for (int k = 0; k < 8; k++) o[k] = (bf16)a[i * 8 + k];
  }
  *reinterpret_cast<bf16x8*>(b + i * 8) = o;
}

// MSE: loss += sum (o-t)^2 / n; dout[p][0..7] = 2 (o-t)/n (channels 6, 7 zero)
__global__ void k_mse(const float* __restrict__ o, const float* __restrict__ t, float* __restrict__ dout,
                      int64_t nvox, double inv_n, double* loss) {
  __shared__ double red[UB];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0;
  if (i < nvox * 8) {
    const int64_t p = i / 8;
    const int c = (int)(i % 8);
    float g = 0.f;
    if (c < 6) {
      const float d = o[p * 6 + c] - t[p * 6 + c];
      s = (double)d * d * inv_n;
      g = (float)(2.0 * d * inv_n);
    }
    dout[i] = g;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o2 = UB / 2; o2 > 0; o2 >>= 1) {
    if (threadIdx.x < o2) red[threadIdx.x] += red[threadIdx.x + o2];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, int64_t n, float lr, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = 0.9f * m1[i] + 0.1f * gi;
  const float b = 0.999f * m2[i] + 0.001f * gi * gi;
  m1[i] = a;
  m2[i] = b;
  p[i] -= lr * (a * c1) / (sqrtf(b * c2) + 1e-8f);
}

// ------------------------------------------------------------- features --
// sum of |v|^2 into per-block partials
__global__ void k_sumsq(const zd* __restrict__ v, int64_t n, double* part) {
  __shared__ double red[UB];
  double s = 0;
  for (int64_t i = (int64_t)blockIdx.x * UB + threadIdx.x; i < n; i += (int64_t)gridDim.x * UB)
    s += v[i].x * v[i].x + v[i].y * v[i].y;
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = UB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
// scale = [rms, 1/rms] with rms = ||v|| / sqrt(n) (1 for a zero vector)
__global__ void k_scale_fin(const double* part, int nb, int64_t n, double* scale) {
  __shared__ double red[UB];
  double s = 0;
  for (int i = threadIdx.x; i < nb; i += UB) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = UB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double rms = sqrt(red[0] / (double)n);
    if (!(rms > 0)) rms = 1.0;
    scale[0] = rms;
    scale[1] = 1.0 / rms;
  }
}

// logc = log10(Re sa / Re sb) with sa recovered from a = 2 sqrt(Re sb)/(sa + conj sb)
__global__ void k_logc(const zd* __restrict__ asiga, const zd* __restrict__ csigb, const double* sq,
                       int64_t ncxy, int Nz, float* logc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncxy * Nz) return;
  const int z = (int)(i / ncxy);
  const zd a = asiga[i], sb = csigb[z];
  const zd sa = cdiv(mkz(2.0 * sq[z], 0.0), a) - mkz(sb.x, -sb.y);
  const double r = fmax(sa.x, 1e-12) / sb.x;
  logc[i] = (float)log10(r);
}

// x[p][8] from a residual r (slots s0,s1,s2 hold physical x,y,z); bf16 or FP32
__global__ void k_pack(const zd* __restrict__ r, int64_t ncell, int64_t ncxy, int s0, int s1, int s2,
                       const double* __restrict__ scale, const float* __restrict__ logc,
                       const float* __restrict__ logk, bf16* xb, float* xf) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ncell) return;
  const double is = scale[1];
  const zd a = r[s0 * ncell + p], b = r[s1 * ncell + p], c = r[s2 * ncell + p];
  float v[8] = {(float)(a.x * is), (float)(a.y * is), (float)(b.x * is), (float)(b.y * is),
                (float)(c.x * is), (float)(c.y * is), logc[p], logk[p / ncxy]};
  if (xb) {
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 8; k++) o[k] = (bf16)v[k];
    *reinterpret_cast<bf16x8*>(xb + p * 8) = o;
  } else {
#pragma unroll
    for (int k = 0; k < 8; k++) xf[p * 8 + k] = v[k];
  }
}

// target t[p][6] = a(p) e_c(p) / rms
__global__ void k_target(const zd* __restrict__ e, const zd* __restrict__ asiga, int64_t ncell, int s0,
                         int s1, int s2, const double* __restrict__ scale, float* t) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ncell) return;
  const double is = scale[1];
  const zd a = asiga[p];
  const zd ex = a * e[s0 * ncell + p], ey = a * e[s1 * ncell + p], ez = a * e[s2 * ncell + p];
  t[p * 6 + 0] = (float)(ex.x * is);
  t[p * 6 + 1] = (float)(ex.y * is);
  t[p * 6 + 2] = (float)(ey.x * is);
  t[p * 6 + 3] = (float)(ey.y * is);
  t[p * 6 + 4] = (float)(ez.x * is);
  t[p * 6 + 5] = (float)(ez.y * is);
}

// z_c(p) = rms * (o[p][2c] + i o[p][2c+1]) / a(p)
__global__ void k_unpack(const float* __restrict__ o, const zd* __restrict__ asiga, int64_t ncell,
                         int s0, int s1, int s2, const double* __restrict__ scale, zd* z) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ncell) return;
  const double rms = scale[0];
  const zd ia = cdiv(mkz(rms, 0.0), asiga[p]);
  z[s0 * ncell + p] = ia * mkz(o[p * 6 + 0], o[p * 6 + 1]);
  z[s1 * ncell + p] = ia * mkz(o[p * 6 + 2], o[p * 6 + 3]);
  z[s2 * ncell + p] = ia * mkz(o[p * 6 + 4], o[p * 6 + 5]);
}

}  // namespace

// ------------------------------------------------------------------ host --
// (name, cin, cout, taps, relu): the architecture of the network
static const int kArch[11][4] = {{8, 16, 27, 1},  {16, 16, 27, 1}, {16, 32, 27, 1}, {32, 32, 27, 1},
                                 {32, 64, 27, 1}, {64, 64, 27, 1}, {96, 32, 27, 1}, {32, 32, 27, 1},
                                 {48, 16, 27, 1}, {16, 16, 27, 1}, {16, 6, 1, 0}};

int64_t unet_param_count() {
  int64_t c = 0;
  for (auto& a : kArch) c += (int64_t)a[1] * a[2] * a[0] + a[1];
  return c;
}

void unet_init(UNet& n, int) {
  n.L.clear();
  int64_t po = 0, wo = 0, wto = 0;
  for (auto& a : kArch) {
    UNetLayer l;
    l.cin = a[0];
    l.cout = a[1];
    l.ntap = a[2];
    l.relu = a[3];
    l.poff = po;
    po += (int64_t)l.cout * l.ntap * l.cin + l.cout;
    l.coutP = (int)up_to(l.cout, 16);
    l.kp = (int)up_to((int64_t)l.ntap * l.cin, 32);
    l.coutT = (int)up_to(l.cout, 8);
    l.cinP = (int)up_to(l.cin, 16);
    l.kpT = (int)up_to((int64_t)l.ntap * l.coutT, 32);
    l.woff = wo;
    l.wtoff = wto;
    wo += up_to((int64_t)l.coutP * l.kp, 128);
    wto += up_to((int64_t)l.cinP * l.kpT, 128);
    n.L.push_back(l);
  }
  n.nparams = po;
  n.nw = wo;
  n.nwt = wto;
  G2G_HIP(hipStreamCreate(&n.stream));
  G2G_HIP(hipMalloc(&n.params, sizeof(float) * po));
  G2G_HIP(hipMalloc(&n.grads, sizeof(float) * po));
  G2G_HIP(hipMalloc(&n.m1, sizeof(float) * po));
  G2G_HIP(hipMalloc(&n.m2, sizeof(float) * po));
  G2G_HIP(hipMalloc(&n.w, sizeof(bf16) * wo));
  G2G_HIP(hipMalloc(&n.wt, sizeof(bf16) * wto));
  G2G_HIP(hipMalloc(&n.dscal, sizeof(double) * 4));
  G2G_HIP(hipMemsetAsync(n.params, 0, sizeof(float) * po, n.stream));
  G2G_HIP(hipMemsetAsync(n.grads, 0, sizeof(float) * po, n.stream));
  G2G_HIP(hipMemsetAsync(n.m1, 0, sizeof(float) * po, n.stream));
  G2G_HIP(hipMemsetAsync(n.m2, 0, sizeof(float) * po, n.stream));
  G2G_HIP(hipStreamSynchronize(n.stream));
  n.adam_t = 0;
  n.wdirty = true;
}

void unet_free(UNet& n) {
  for (void* p : {(void*)n.params, (void*)n.grads, (void*)n.m1, (void*)n.m2, (void*)n.w, (void*)n.wt,
                  (void*)n.dscal, n.ws})
    if (p) (void)hipFree(p);
  if (n.stream) (void)hipStreamDestroy(n.stream);
  n = UNet();
}

// tiles of the weight gradient at a level
static int dw_tiles(int B, int nx, int ny, int nz) { return B * ((nx + 15) / 16) * ((ny + 3) / 4) * ((nz + 1) / 2); }

// Slots of a layer's weight gradient (one per block), one tile or more each, at
// least 64: as many as 32 MB of partial sums hold for up to 16 output channels
// (three 64-thread waves a block: 60 -> 47 us a layer against 16 MB), 16 MB
// for wider ones (42 us against 49 with 32 MB: the sums' traffic)
static int dw_slots(const UNetLayer& l, int tiles) {
  const int64_t per = (int64_t)l.cout * l.ntap * l.cin + l.cout;
  return (int)std::min<int64_t>(tiles, std::min<int64_t>(1024, std::max<int64_t>(64, (int64_t(l.cout <= 16 ? 8 : 4) << 20) / per)));
}

// floats of the partial sums of every layer of a training step
static int64_t dw_part_size(const UNet& n, int B, int nx, int ny, int nz) {
  int64_t most = 0;
  static const int level[11] = {0, 0, 1, 1, 2, 2, 1, 1, 0, 0, 0};
  for (int i = 0; i < 11; i++) {
    const UNetLayer& l = n.L[i];
    const int64_t per = (int64_t)l.cout * l.ntap * l.cin + l.cout;
    const int t = dw_tiles(B, nx >> level[i], ny >> level[i], nz >> level[i]);
    most = std::max<int64_t>(most, per * dw_slots(l, t) * (l.ntap == 1 ? 3 : 1));
  }
  return most;
}

void unet_reserve(UNet& n, int B, int nx, int ny, int nz, bool training) {
  G2G_CHECK(nx % 4 == 0 && ny % 4 == 0 && nz % 4 == 0 && nx > 0 && ny > 0 && nz > 0, -2,
            "U-Net volume dimensions must be positive multiples of 4");
  G2G_CHECK(B >= 1, -2, "batch must be >= 1");
  if (n.ws && n.B == B && n.nx == nx && n.ny == ny && n.nz == nz && (n.training || !training)) return;
  if (n.ws) {
    G2G_HIP(hipStreamSynchronize(n.stream));
    (void)hipFree(n.ws);
    n.ws = nullptr;
  }
  const int64_t n0 = (int64_t)B * nx * ny * nz, n1 = n0 / 8, n2 = n0 / 64;
  size_t off = 0;
  std::vector<std::pair<void**, size_t>> plan;
  auto add = [&](void** p, size_t bytes) {
    plan.push_back({p, off});
    off += (bytes + 255) / 256 * 256;
  };
  add((void**)&n.in, 2 * n0 * 8);
  const int64_t lvl[11] = {n0, n0, n1, n1, n2, n2, n1, n1, n0, n0, n0};
  for (int i = 0; i < 10; i++) add((void**)&n.act[i], 2 * lvl[i] * n.L[i].cout);
  n.act[10] = nullptr;
  add((void**)&n.p1, 2 * n1 * 16);
  add((void**)&n.p2, 2 * n2 * 32);
  add((void**)&n.out, 4 * n0 * 6);
  if (training) {
    add((void**)&n.dout, 4 * n0 * 8);
    add((void**)&n.f48, 4 * n0 * 48);
    add((void**)&n.fa, 4 * n0 * 16);
    add((void**)&n.fb, 4 * n0 * 4);
    add((void**)&n.f96, 4 * n1 * 96);
    add((void**)&n.dzf, 4 * n0 * 16);
    add((void**)&n.dzb, 2 * n0 * 16);
    add((void**)&n.dwp, 4 * dw_part_size(n, B, nx, ny, nz));
  } else {
    n.dout = n.f48 = n.fa = n.fb = n.f96 = n.dzf = n.dwp = nullptr;
    n.dzb = nullptr;
  }
  void* base = nullptr;
  G2G_HIP(hipMalloc(&base, off));
  for (auto& pr : plan) *pr.first = (char*)base + pr.second;
  n.ws = base;
  n.ws_bytes = off;
  n.B = B;
  n.nx = nx;
  n.ny = ny;
  n.nz = nz;
  n.training = training;
}

void unet_prepare_weights(UNet& n, hipStream_t s) {
  if (!n.wdirty) return;
  for (auto& l : n.L) {
    const int64_t tot = (int64_t)l.coutP * l.kp + (int64_t)l.cinP * l.kpT;
    hipLaunchKernelGGL(k_wprep, dim3(nblk(tot)), dim3(UB), 0, s, n.params + l.poff, l.cout, l.cin, l.ntap,
                       n.w + l.woff, l.coutP, l.kp, n.wt + l.wtoff, l.cinP, l.coutT, l.kpT);
  }
  G2G_HIP(hipGetLastError());
  n.wdirty = false;
}

static Src src(const bf16* p, int C, int up, int64_t bstride) {
  Src r;
  r.p = p;
  r.C = C;
  r.up = up;
  r.bstride = bstride;
  return r;
}

static ConvBox conv_box(int hx, int hy, int hz) {
  ConvBox b;
  b.hx = hx;
  b.hy = hy;
  b.hvox = hx * hy * hz;
  b.hv = b.hvox | 1;  // planes start on different banks
  b.mx = ((1u << 20) + hx - 1) / hx;
  b.mxy = ((1u << 20) + hx * hy - 1) / (hx * hy);
  return b;
}

// Tile of 64 G voxels: 16 long in x, or 8 or 4 where that covers the volume
// with fewer tiles
static ConvTile conv_tile(int G, int nx, int ny, int nz) {
  // log2 sides, then the group strides of bits (g0, g1, w0, w1)
  static const int shapes[2][3][7] = {{{4, 2, 1, 2, 0, 1, 4}, {3, 2, 2, 1, 0, 2, 4}, {2, 3, 2, 1, 0, 2, 4}},
                                      {{4, 2, 2, 2, 8, 1, 4}, {3, 3, 2, 1, 2, 4, 8}, {2, 3, 3, 1, 4, 2, 8}}};
  ConvTile best{};
  int64_t least = -1;
  for (auto& sh : shapes[G == 4]) {
    ConvTile t;
    t.lx = sh[0];
    t.ly = sh[1];
    t.lz = sh[2];
    auto up = [](int n, int l) { return (n + (1 << l) - 1) >> l; };
    t.ntx = up(nx, t.lx);
    t.nty = up(ny, t.ly);
    t.nt = t.ntx * t.nty * up(nz, t.lz);
    t.f = conv_box((1 << t.lx) + 2, (1 << t.ly) + 2, (1 << t.lz) + 2);
    t.h = conv_box((1 << t.lx) / 2 + 2, (1 << t.ly) / 2 + 2, (1 << t.lz) / 2 + 2);
    t.sg[0] = sh[3];
    t.sg[1] = sh[4];
    t.sw[0] = sh[5];
    t.sw[1] = sh[6];
    if (least < 0 || t.nt < least) {
      least = t.nt;
      best = t;
    }
  }
  return best;
}

template <int CIN, int CT, int UPC> static void conv3_go(const ConvArgs& a, int B, hipStream_t s) {
  G2G_CHECK(UPC ? a.s1.up == 1 && a.s1.C == UPC && a.s2.up == 0 && a.s2.C == CIN - UPC : a.s1.up == 0 && a.s2.C == 0, -1,
            "convolution sources do not match the layer");
  const ConvTile t = conv_tile(conv_g(CIN), a.nx, a.ny, a.nz);
  constexpr int NKS = (27 * CIN + 31) / 32, NU = UPC / 8;
  const size_t lds = (size_t)16 * (NU * t.h.hv + (CIN / 8 - NU) * t.f.hv) + sizeof(short) * NKS * 4 * (UPC ? 8 : 1);
  if (lds > 65536)
    G2G_HIP(hipFuncSetAttribute((const void*)k_conv3<CIN, CT, UPC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  hipLaunchKernelGGL((k_conv3<CIN, CT, UPC>), dim3((unsigned)(t.nt * B)), dim3(UB), lds, s, a, t);
}

// the network's widths (forward, and the data gradient's transposed ones)
static void conv_launch(const ConvArgs& a, int coutP, int B, hipStream_t s) {
  G2G_CHECK(a.cout % 4 == 0 && a.ldy % 4 == 0, -1, "convolution outputs of a multiple of four channels");
  const int64_t nvox = (int64_t)a.nx * a.ny * a.nz;
  if (a.ntap == 1) {
    G2G_CHECK(a.kp == 32 && a.s2.C == 0 && a.s1.up == 0, -1, "1x1 convolution of more than 32 channels");
    hipLaunchKernelGGL(k_conv1x1, dim3(nblk(nvox, 256), coutP / 16, B), dim3(UB), 0, s, a);
    return;
  }
  const int ct = coutP / 16;
#define G2G_CONV(ci, c, u) \
  if (a.cin == ci && ct == c) return conv3_go<ci, c, u>(a, B, s);
  G2G_CONV(8, 1, 0) G2G_CONV(16, 1, 0) G2G_CONV(16, 2, 0) G2G_CONV(16, 3, 0) G2G_CONV(32, 1, 0) G2G_CONV(32, 2, 0)
  G2G_CONV(32, 4, 0) G2G_CONV(32, 6, 0) G2G_CONV(48, 1, 32) G2G_CONV(64, 2, 0) G2G_CONV(64, 4, 0) G2G_CONV(96, 2, 64)
#undef G2G_CONV
  G2G_CHECK(false, -1, "no convolution kernel for this layer width");
}

// y = conv(x) at level dims (nx, ny, nz), batch B
static void conv_fwd(UNet& n, int li, Src s1, Src s2, int nx, int ny, int nz, bf16* ybf, hipStream_t s,
                     const float* xf = nullptr, float* y2 = nullptr) {
  const UNetLayer& l = n.L[li];
  ConvArgs a{};
  a.s1 = s1;
  a.s2 = s2;
  a.w = n.w + l.woff;
  a.kp = l.kp;
  a.ntap = l.ntap;
  a.cin = l.cin;
  a.bias = n.params + l.poff + (int64_t)l.cout * l.ntap * l.cin;
  a.cout = l.cout;
  a.relu = l.relu;
  a.ybf = ybf;
  a.ldy = l.cout;
  a.ybstride = (int64_t)nx * ny * nz * l.cout;
  a.xf = xf;
  if (y2) {
    const UNetLayer& o = n.L[10];
    G2G_CHECK(l.cin == 16 && l.cout == 16 && o.cin == 16 && o.ntap == 1 && o.kp == 32 && o.coutP == 16, -1,
              "the output layer does not follow a 16-channel layer");
    a.w2 = n.w + o.woff;
    a.bias2 = n.params + o.poff + (int64_t)o.cout * o.cin;
    a.y2 = y2;
    a.cout2 = o.cout;
  }
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  G2G_CHECK(s1.C + s2.C == l.cin, -1, "U-Net layer input width mismatch");
  conv_launch(a, l.coutP, n.B, s);
}

// data gradient: dx[p][ci] (FP32, row length cin) from dzb[p][coutT] (bf16)
static void conv_dx(UNet& n, int li, const bf16* dzb, int nx, int ny, int nz, float* dx, hipStream_t s) {
  const UNetLayer& l = n.L[li];
  const int64_t nvox = (int64_t)nx * ny * nz;
  ConvArgs a{};
  a.s1 = src(dzb, l.coutT, 0, nvox * l.coutT);
  a.s2 = src(nullptr, 0, 0, 0);
  a.w = n.wt + l.wtoff;
  a.kp = l.kpT;
  a.ntap = l.ntap;
  a.cin = l.coutT;
  a.bias = nullptr;
  a.cout = l.cin;
  a.relu = 0;
  a.ybf = nullptr;
  a.yf = dx;
  a.ldy = l.cin;
  a.ybstride = nvox * l.cin;
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  conv_launch(a, l.cinP, n.B, s);
}

template <int NCO, int NCI, bool ONE> static void dw_go(const DwArgs& a, int slots, int gy, int gz, hipStream_t s) {
  const size_t lds = sizeof(bf16) * (NCI * 16 * DW_XST + 3 * NCO * 16 * DW_ZST);
  if (lds > 65536)
    G2G_HIP(hipFuncSetAttribute((const void*)k_dw<NCO, NCI, ONE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  hipLaunchKernelGGL((k_dw<NCO, NCI, ONE>), dim3(slots, gy, gz), dim3(192 * NCI), lds, s, a);
}

static void conv_dw(UNet& n, int li, const float* dzf, int ldz, Src s1, Src s2, int nx, int ny, int nz,
                    hipStream_t s) {
  const UNetLayer& l = n.L[li];
  DwArgs a;
  a.dz = dzf;
  a.ldz = ldz;
  a.cout = l.cout;
  a.s1 = s1;
  a.s2 = s2.p ? s2 : s1;
  a.cin = l.cin;
  a.ntap = l.ntap;
  a.part = n.dwp;
  a.pstride = (int64_t)l.cout * l.ntap * l.cin + l.cout;
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  a.ntx = (nx + 15) / 16;
  a.nty = (ny + 3) / 4;
  a.ntot = dw_tiles(n.B, nx, ny, nz);
  a.nt = a.ntot / n.B;
  const int slots = dw_slots(l, a.ntot);
  G2G_CHECK(ldz % 4 == 0 && l.cin % 8 == 0 && s1.C + s2.C == l.cin, -1, "weight gradient: layer widths");
  // tiles of 16 channels: one by one or two by two in a block; wider layers
  // take blocks side by side (48 input channels: 135 us as three blocks, 166
  // us as one of nine waves, which left a third of the CUs idle)
  const int no = (l.cout + 15) / 16, ni = (l.cin + 15) / 16;
  if (l.ntap == 1) {
    G2G_CHECK(no == 1 && ni == 1, -1, "weight gradient: 1x1 layer of more than 16 channels");
    dw_go<1, 1, true>(a, slots, 1, 1, s);
  } else if (no == 1) dw_go<1, 1, false>(a, slots, ni, 1, s);
  else if (no % 2 == 0 && ni == 1) dw_go<2, 1, false>(a, slots, 1, no / 2, s);
  else if (no % 2 == 0 && ni % 2 == 0) dw_go<2, 2, false>(a, slots, ni / 2, no / 2, s);
  else G2G_CHECK(false, -1, "no weight-gradient kernel for this layer width");
  hipLaunchKernelGGL(k_dw_reduce, dim3(nblk(a.pstride, 64)), dim3(64 * DWR), 0, s, n.dwp, slots * (l.ntap == 1 ? 3 : 1),
                     a.pstride, n.grads + l.poff);
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

void unet_load_input(UNet& n, const float* x, hipStream_t s) {
  const int64_t cnt = (int64_t)n.B * n.nx * n.ny * n.nz;
  if (aligned16(x)) hipLaunchKernelGGL(k_f32_to_bf16<true>, dim3(nblk(cnt)), dim3(UB), 0, s, x, n.in, cnt);
  else hipLaunchKernelGGL(k_f32_to_bf16<false>, dim3(nblk(cnt)), dim3(UB), 0, s, x, n.in, cnt);
}

void unet_forward(UNet& n, hipStream_t s, const float* x, float* y) {
  G2G_CHECK(n.ws != nullptr, -4, "U-Net workspace not reserved");
  unet_prepare_weights(n, s);
  const int X0 = n.nx, Y0 = n.ny, Z0 = n.nz, X1 = X0 / 2, Y1 = Y0 / 2, Z1 = Z0 / 2, X2 = X1 / 2,
            Y2 = Y1 / 2, Z2 = Z1 / 2;
  const int64_t v0 = (int64_t)X0 * Y0 * Z0, v1 = v0 / 8, v2 = v0 / 64;
  const Src none = src(nullptr, 0, 0, 0);
  bf16** A = n.act;
  conv_fwd(n, 0, src(n.in, 8, 0, v0 * 8), none, X0, Y0, Z0, A[0], s, x);
  conv_fwd(n, 1, src(A[0], 16, 0, v0 * 16), none, X0, Y0, Z0, A[1], s);
  hipLaunchKernelGGL(k_pool, dim3(nblk((int64_t)n.B * v1 * 2)), dim3(UB), 0, s, A[1], n.p1, 16, X0, Y0, Z0,
                     (int64_t)n.B);
  conv_fwd(n, 2, src(n.p1, 16, 0, v1 * 16), none, X1, Y1, Z1, A[2], s);
  conv_fwd(n, 3, src(A[2], 32, 0, v1 * 32), none, X1, Y1, Z1, A[3], s);
  hipLaunchKernelGGL(k_pool, dim3(nblk((int64_t)n.B * v2 * 4)), dim3(UB), 0, s, A[3], n.p2, 32, X1, Y1, Z1,
                     (int64_t)n.B);
  conv_fwd(n, 4, src(n.p2, 32, 0, v2 * 32), none, X2, Y2, Z2, A[4], s);
  conv_fwd(n, 5, src(A[4], 64, 0, v2 * 64), none, X2, Y2, Z2, A[5], s);
  conv_fwd(n, 6, src(A[5], 64, 1, v2 * 64), src(A[3], 32, 0, v1 * 32), X1, Y1, Z1, A[6], s);
  conv_fwd(n, 7, src(A[6], 32, 0, v1 * 32), none, X1, Y1, Z1, A[7], s);
  conv_fwd(n, 8, src(A[7], 32, 1, v1 * 32), src(A[1], 16, 0, v0 * 16), X0, Y0, Z0, A[8], s);
  // the 1x1 output layer runs on the last layer's registers; its bf16 input
  // is stored only for a backward pass
  conv_fwd(n, 9, src(A[8], 16, 0, v0 * 16), none, X0, Y0, Z0, n.training ? A[9] : nullptr, s, nullptr,
           y ? y : n.out);
  G2G_HIP(hipGetLastError());
}

// one layer of the backward pass: dz = g*(y>0), weight gradient, data gradient into dx
template <GradSource SRC = GradPlain>
static void layer_back(UNet& n, int li, const float* dy, int ldy, const bf16* y, Src s1, Src s2, int nx,
                       int ny, int nz, float* dx, hipStream_t s, const float* dc = nullptr) {
  const UNetLayer& l = n.L[li];
  int sh = 0;
  while ((4 << sh) < l.coutT) sh++;
  G2G_CHECK((4 << sh) == l.coutT && (!l.relu || l.cout == l.coutT), -3, "layer widths are powers of two");
  hipLaunchKernelGGL(k_relu_back<SRC>, dim3(nblk((int64_t)(nx * ny) << sh), std::min(nz, GRID_Y_MAX), n.B), dim3(UB), 0,
                     s, dy, ldy, dc, l.relu ? y : nullptr, l.cout, sh, n.dzf, n.dzb, nx, ny, nz);
  conv_dw(n, li, n.dzf, l.coutT, s1, s2, nx, ny, nz, s);
  if (dx) conv_dx(n, li, n.dzb, nx, ny, nz, dx, s);
}

void unet_backward(UNet& n, hipStream_t s) {
  G2G_CHECK(n.training, -4, "U-Net workspace not reserved for training");
  const int X0 = n.nx, Y0 = n.ny, Z0 = n.nz, X1 = X0 / 2, Y1 = Y0 / 2, Z1 = Z0 / 2, X2 = X1 / 2,
            Y2 = Y1 / 2, Z2 = Z1 / 2;
  const int64_t v0 = (int64_t)X0 * Y0 * Z0, v1 = v0 / 8, v2 = v0 / 64;
  const Src none = src(nullptr, 0, 0, 0);
  bf16** A = n.act;
  layer_back(n, 10, n.dout, 8, nullptr, src(A[9], 16, 0, v0 * 16), none, X0, Y0, Z0, n.fa, s);
  layer_back(n, 9, n.fa, 16, A[9], src(A[8], 16, 0, v0 * 16), none, X0, Y0, Z0, n.fa, s);
  layer_back(n, 8, n.fa, 16, A[8], src(A[7], 32, 1, v1 * 32), src(A[1], 16, 0, v0 * 16), X0, Y0, Z0, n.f48,
             s);
  layer_back<GradUpsample>(n, 7, n.f48, 48, A[7], src(A[6], 32, 0, v1 * 32), none, X1, Y1, Z1, n.fb, s);
  layer_back(n, 6, n.fb, 32, A[6], src(A[5], 64, 1, v2 * 64), src(A[3], 32, 0, v1 * 32), X1, Y1, Z1, n.f96,
             s);
  layer_back<GradUpsample>(n, 5, n.f96, 96, A[5], src(A[4], 64, 0, v2 * 64), none, X2, Y2, Z2, n.fb, s);
  layer_back(n, 4, n.fb, 64, A[4], src(n.p2, 32, 0, v2 * 32), none, X2, Y2, Z2, n.fb, s);
  layer_back<GradPool>(n, 3, n.f96 + 64, 96, A[3], src(A[2], 32, 0, v1 * 32), none, X1, Y1, Z1, n.fb, s, n.fb);
  layer_back(n, 2, n.fb, 32, A[2], src(n.p1, 16, 0, v1 * 16), none, X1, Y1, Z1, n.fb, s);
  layer_back<GradPool>(n, 1, n.f48 + 32, 48, A[1], src(A[0], 16, 0, v0 * 16), none, X0, Y0, Z0, n.fa, s, n.fb);
  layer_back(n, 0, n.fa, 16, A[0], src(n.in, 8, 0, v0 * 8), none, X0, Y0, Z0, nullptr, s);
  G2G_HIP(hipGetLastError());
}

double unet_mse(UNet& n, const float* target, hipStream_t s) {
  const int64_t nv = (int64_t)n.B * n.nx * n.ny * n.nz;
  G2G_HIP(hipMemsetAsync(n.dscal, 0, sizeof(double), s));
  hipLaunchKernelGGL(k_mse, dim3(nblk(nv * 8)), dim3(UB), 0, s, n.out, target, n.dout, nv,
                     1.0 / (double)(nv * 6), n.dscal);
  G2G_HIP(hipGetLastError());
  double loss = 0;
  G2G_HIP(hipMemcpyAsync(&loss, n.dscal, sizeof(double), hipMemcpyDeviceToHost, s));
  G2G_HIP(hipStreamSynchronize(s));
  return loss;
}

void unet_adam(UNet& n, float lr, hipStream_t s) {
  n.adam_t++;
  const float c1 = 1.0f / (1.0f - powf(0.9f, (float)n.adam_t));
  const float c2 = 1.0f / (1.0f - powf(0.999f, (float)n.adam_t));
  hipLaunchKernelGGL(k_adam, dim3(nblk(n.nparams)), dim3(UB), 0, s, n.params, n.grads, n.m1, n.m2, n.nparams,
                     lr, c1, c2);
  G2G_HIP(hipGetLastError());
  n.wdirty = true;
}

// ------------------------------------------------------------ features --
void learned_prepare(LearnedCtx& c, Operator& op, UNet& net) {
  G2G_CHECK(op.have_sigma, -4, "conductivity not set");
  if (c.ncell != op.ncell()) learned_free(c);
  c.net = &net;
  c.op = &op;
  c.ncell = op.ncell();
  if (!c.logc) {
    G2G_HIP(hipMalloc(&c.logc, sizeof(float) * c.ncell));
    G2G_HIP(hipMalloc(&c.logk, sizeof(float) * op.Nz));
    G2G_HIP(hipMalloc(&c.scale, sizeof(double) * 2));
    G2G_HIP(hipMalloc(&c.part, sizeof(double) * 1024));
  }
  // frequency feature per layer: log10(|k_b| dx), |k_b|^2 = omega mu0 |sigma_b|
  std::vector<float> lk(op.Nz);
  for (int z = 0; z < op.Nz; z++) {
    const double kk = op.omega * (4e-7 * 3.14159265358979323846) * std::abs(std::complex<double>(op.csigb[z].x, op.csigb[z].y));
    lk[z] = (float)std::log10(std::sqrt(kk) * op.dx);
  }
  G2G_HIP(hipMemcpyAsync(c.logk, lk.data(), sizeof(float) * op.Nz, hipMemcpyHostToDevice, op.stream));
  zd* d_csigb = nullptr;
  G2G_HIP(hipMalloc(&d_csigb, sizeof(zd) * op.Nz));
  G2G_HIP(hipMemcpyAsync(d_csigb, op.csigb.data(), sizeof(zd) * op.Nz, hipMemcpyHostToDevice, op.stream));
  hipLaunchKernelGGL(k_logc, dim3(nblk(c.ncell)), dim3(UB), 0, op.stream, op.d64.asiga, d_csigb, op.d64.sq,
                     (int64_t)op.Nx * op.Ny, op.Nz, c.logc);
  G2G_HIP(hipGetLastError());
  G2G_HIP(hipStreamSynchronize(op.stream));
  (void)hipFree(d_csigb);
}

void learned_free(LearnedCtx& c) {
  for (void* p : {(void*)c.logc, (void*)c.logk, (void*)c.scale, (void*)c.part})
    if (p) (void)hipFree(p);
  c.logc = c.logk = nullptr;
  c.scale = c.part = nullptr;
  c.ncell = 0;
}

static void residual_scale(LearnedCtx& c, const zd* r, hipStream_t s) {
  const int64_t n = 3 * c.ncell;
  const int nb = (int)std::min<int64_t>(1024, (n + UB - 1) / UB);
  hipLaunchKernelGGL(k_sumsq, dim3(nb), dim3(UB), 0, s, r, n, c.part);
  hipLaunchKernelGGL(k_scale_fin, dim3(1), dim3(UB), 0, s, c.part, nb, n, c.scale);
}

void learned_features(LearnedCtx& c, const zd* r, const zd* e, float* x, float* t, hipStream_t s) {
  Operator& op = *c.op;
  residual_scale(c, r, s);
  const int* sl = op.comp_slot;
  hipLaunchKernelGGL(k_pack, dim3(nblk(c.ncell)), dim3(UB), 0, s, r, c.ncell, (int64_t)op.Nx * op.Ny, sl[0],
                     sl[1], sl[2], c.scale, c.logc, c.logk, (bf16*)nullptr, x);
  if (e && t)
    hipLaunchKernelGGL(k_target, dim3(nblk(c.ncell)), dim3(UB), 0, s, e, op.d64.asiga, c.ncell, sl[0], sl[1],
                       sl[2], c.scale, t);
  G2G_HIP(hipGetLastError());
}

void learned_apply(LearnedCtx& c, const zd* v, zd* z, hipStream_t s) {
  Operator& op = *c.op;
  UNet& n = *c.net;
  unet_reserve(n, 1, op.Nx, op.Ny, op.Nz, false);
  residual_scale(c, v, s);
  const int* sl = op.comp_slot;
  hipLaunchKernelGGL(k_pack, dim3(nblk(c.ncell)), dim3(UB), 0, s, v, c.ncell, (int64_t)op.Nx * op.Ny, sl[0],
                     sl[1], sl[2], c.scale, c.logc, c.logk, n.in, (float*)nullptr);
  unet_forward(n, s);
  hipLaunchKernelGGL(k_unpack, dim3(nblk(c.ncell)), dim3(UB), 0, s, n.out, op.d64.asiga, c.ncell, sl[0], sl[1],
                     sl[2], c.scale, z);
  G2G_HIP(hipGetLastError());
}

}  // namespace g2g
