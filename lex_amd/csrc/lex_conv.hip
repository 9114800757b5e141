// X4: the 3x3x3 'SAME' convolutions of the SGS correction net on BF16 MFMA with FP32
// accumulation.  The architecture follows simpleCNN (dl_models.py:19-30): four Conv
// layers (kernel 3x3x3, stride 1, zero 'SAME' padding, bias) with the tanh-approximate
// GELU (flax nn.gelu's default) between them.
//
// Layout: activations channels-last (x, y, z, c) with the channel count padded to a
// multiple of 16 (CIN, COUT template arguments, 16 or 32).  Weights are kept in FP32 as
// W[tap][cin][cout] (flax's (3,3,3,in,out) kernel, tap = kx*9 + ky*3 + kz) and packed
// for the kernels into BF16 rows Wp[cout][step*32 + k] (one MFMA K-step per 32 k).
//
// MFMA: v_mfma_f32_16x16x32_bf16.  Lane l supplies A[row l%16][k 8(l/16)..+7],
// B[k 8(l/16)..+7][col l%16] and receives D[row 4(l/16)+i][col l%16], i = 0..3.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "lex_common.hpp"

namespace lex {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// the same in memory at any element's address: callers' buffers are views as they come
typedef bf16x8 bf16x8_any __attribute__((aligned(2)));
typedef bf16x4 bf16x4_any __attribute__((aligned(2)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));

constexpr int CTX = 4, CTY = 4, CTZ = 16;  // output tile of one workgroup (4 waves)
constexpr int HX = CTX + 2, HY = CTY + 2, HZ = CTZ + 2;

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// tanh for the GELU of BF16 activations: 1 - 2 / (1 + e^(2y)) from the hardware
// exponential and reciprocal (a few instructions instead of the library's tens).  It
// saturates to +-1 with e^(2y) at inf / 0; near 0 its absolute error is ~1e-7, which the
// GELU's factor x makes a relative error of the same size, far below BF16's 4e-3.
__device__ __forceinline__ float tanh_fast(float y) {
  const float e = __expf(2.0f * y);
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e);
}
// tanh-approximate GELU and its derivative.  0.5 x (1 + tanh(y)) = x / (1 + e^(-2y)) with
// y = k0 (x + k1 x^3): seven instructions, e^(-2y) = 2^(x (c0 + c1 x^2)) with
// c0 = -2 k0 log2(e), c1 = -2 k0 k1 log2(e); it saturates to x and to -0 like the tanh form.
__device__ __forceinline__ float gelu_t(float x) {
  const float c0 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634);
  const float c1 = (float)(-2.0 * 0.7978845608028654 * 0.044715 * 1.4426950408889634);
  const float e = __builtin_amdgcn_exp2f(x * fmaf(c1, x * x, c0));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu_t_grad(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  float t = tanh_fast(k0 * (x + k1 * x * x * x));
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * k0 * (1.0f + 3.0f * k1 * x * x);
}

// Element stride of one cell in an LDS halo tile: the CIN channels plus 8 (16 bytes) of
// padding.  An MFMA operand read takes 16 bytes from each of 16 consecutive cells (one z
// run); with a stride of CIN elements (32 or 64 bytes for 16 or 32 channels) those reads
// fall on 2 or 4 distinct bank groups of the 256-byte bank row, with CIN + 8 (48 or 80
// bytes, an odd multiple of 16) on 16 distinct ones.
__host__ __device__ constexpr int conv_cell_stride(int cin) { return cin + 8; }

// K-steps of 32 over (tap, channel): CIN <= 32 packs 32 / CIN taps per step; CIN = 64
// spends two steps per tap (channels 0..31, then 32..63).
template <int CIN>
struct ConvSteps {
  static constexpr int TPS = CIN <= 32 ? 32 / CIN : 1;              // taps per K-step
  static constexpr int SPT = CIN <= 32 ? 1 : CIN / 32;              // K-steps per tap
  static constexpr int NSTEP = CIN <= 32 ? (27 + TPS - 1) / TPS : 27 * SPT;
};
// tap and first channel of a lane's 8 k values (kl = 8 * (lane / 16)) in step s
__host__ __device__ __forceinline__ void conv_step_k(int cinp, int s, int kl, int& tap, int& ch) {
  if (cinp <= 32) {
    tap = s * (32 / cinp) + kl / cinp;
    ch = kl % cinp;
  } else {
    tap = s / (cinp / 32);
    ch = (s % (cinp / 32)) * 32 + kl;
  }
}

// Forward convolution.  mode bit 0: GELU after the bias; bit 1: FP32 output Yf with
// cout_real channels (else BF16 Y with COUT channels); bit 2: periodic x and y.  pre (optional): FP32
// pre-activation, COUT channels.
template <int CIN, int COUT>
__global__ __launch_bounds__(256) void k_conv3_fwd(int nx, int ny, int nz, const __bf16* __restrict__ X,
                                                   const __bf16* __restrict__ Wp, const float* __restrict__ bias,
                                                   int mode, int cout_real, __bf16* __restrict__ Y,
                                                   float* __restrict__ Yf, float* __restrict__ pre) {
  constexpr int NSTEP = ConvSteps<CIN>::NSTEP, NT = COUT / 16, CS = conv_cell_stride(CIN);
  __shared__ __attribute__((aligned(16))) __bf16 tile[HX * HY * HZ * CS];
  // neighbouring tiles (which share halo cells) on one XCD: z tiles fastest, then y, x
  const TileId tb = xcd_tile();
  const int z0 = tb.x * CTZ, y0 = tb.y * CTY, x0 = tb.z * CTX;
  constexpr int nchunk = HX * HY * HZ * CIN / 8;
  const bool circ = (mode & 4) != 0;  // periodic x and y (flax padding 'CIRCULAR' there), zero z
  for (int c = threadIdx.x; c < nchunk; c += 256) {
    int cell = c / (CIN / 8), g = c % (CIN / 8);
    int hz = cell % HZ, hy = (cell / HZ) % HY, hx = cell / (HZ * HY);
    int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
    if (circ) {
      gx = gx < 0 ? gx + nx : (gx >= nx ? gx - nx : gx);
      gy = gy < 0 ? gy + ny : (gy >= ny ? gy - ny : gy);
    }
    bf16x8 v;
    if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz) {
      v = *(const bf16x8_any*)(X + (((long)gx * ny + gy) * nz + gz) * CIN + 8 * g);
    } else {
      for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.0f;
    }
    *(bf16x8*)(tile + cell * CS + 8 * g) = v;
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, m = l & 15, g = l >> 4;
  f32x4 acc[CTY][NT];
  for (int a = 0; a < CTY; ++a)
    for (int b = 0; b < NT; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int kl = 8 * g;  // this lane's first k within a step
  // the weight fragments of step s+1 are fetched while step s runs
  bf16x8 bw[NT], bwn[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) bw[nt] = *(const bf16x8*)(Wp + (long)(nt * 16 + m) * (NSTEP * 32) + kl);
  for (int s = 0; s < NSTEP; ++s) {
    int tap, ch0;
    conv_step_k(CIN, s, kl, tap, ch0);
    if (tap > 26) tap = 26;              // padded K-step: weights are zero there
    const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
    const int sn = (s + 1 < NSTEP) ? s + 1 : s;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      bwn[nt] = *(const bf16x8*)(Wp + (long)(nt * 16 + m) * (NSTEP * 32) + sn * 32 + kl);
    bf16x8 a[CTY];
#pragma unroll
    for (int mt = 0; mt < CTY; ++mt) {
      const int cell = ((w + 1 + dx) * HY + (mt + 1 + dy)) * HZ + (m + 1 + dz);
      a[mt] = *(const bf16x8*)(tile + cell * CS + ch0);
    }
#pragma unroll
    for (int mt = 0; mt < CTY; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = mfma16(a[mt], bw[nt], acc[mt][nt]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) bw[nt] = bwn[nt];
  }
  const int xc = x0 + w;
#pragma unroll
  for (int mt = 0; mt < CTY; ++mt) {
    const int yc = y0 + mt;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = nt * 16 + m;
      const float bn = bias[n];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int zc = z0 + 4 * g + i;
        if (xc < nx && yc < ny && zc < nz) {
          const long cell = ((long)xc * ny + yc) * nz + zc;
          float v = acc[mt][nt][i] + bn;
          if (pre) pre[cell * COUT + n] = v;
          if (mode & 1) v = gelu_t(v);
          if (mode & 2) {
            if (n < cout_real) Yf[cell * cout_real + n] = v;
          } else {
            Y[cell * COUT + n] = (__bf16)v;
          }
        }
      }
    }
  }
}

// The forward convolution for COUT a multiple of 32 on v_mfma_f32_32x32x16_bf16: one
// MFMA covers 32 cells x 32 output channels, so each A fragment read from LDS (32 cells x
// 16 k) feeds 32 (or 64) output channels, half the LDS bytes per flop of the 16x16x32
// form, whose A fragments feed 16.  Output tile 4 x 4 x 16 (x, y, z) per 4-wave
// workgroup, as k_conv3_fwd (the same 52 KB halo tile for 32 channels): wave w owns
// x = x0 + w and two accumulator blocks, each 2 y rows x 16 z cells as the 32 MFMA rows
// (row m: y offset m / 16, z offset m % 16).  Operand layout: lane l supplies A[row l%32][k 8(l/32)..+7]
// and B[k 8(l/32)..+7][col l%32] and receives D[row 8(i/4) + 4(l/32) + i%4][col l%32]
// in accumulator i = 0..15.  Same arguments and results as k_conv3_fwd.
constexpr int CT2X = 4, CT2Y = 4, CT2Z = 16;
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int CIN, int COUT>
__global__ __launch_bounds__(256) void k_conv3_fwd32(int nx, int ny, int nz, const __bf16* __restrict__ X,
                                                     const __bf16* __restrict__ Wp, const float* __restrict__ bias,
                                                     int mode, int cout_real, __bf16* __restrict__ Y,
                                                     float* __restrict__ Yf, float* __restrict__ pre) {
  constexpr int NSTEP = ConvSteps<CIN>::NSTEP, NT = COUT / 32, NK = 2 * NSTEP;   // 16-wide K steps
  constexpr int GX = CT2X + 2, GY = CT2Y + 2, GZ = CT2Z + 2, CS = conv_cell_stride(CIN);
  __shared__ __attribute__((aligned(16))) __bf16 tile[GX * GY * GZ * CS];
  const TileId tb = xcd_tile();  // neighbouring tiles on one XCD (shared halo cells in its L2)
  const int z0 = tb.x * CT2Z, y0 = tb.y * CT2Y, x0 = tb.z * CT2X;
  constexpr int nchunk = GX * GY * GZ * CIN / 8;
  const bool circ = (mode & 4) != 0;  // periodic x and y (flax padding 'CIRCULAR' there), zero z
  for (int c = threadIdx.x; c < nchunk; c += 256) {
    int cell = c / (CIN / 8), g = c % (CIN / 8);
    int hz = cell % GZ, hy = (cell / GZ) % GY, hx = cell / (GZ * GY);
    int gx = x0 + hx - 1, gy = y0 + hy - 1, gz = z0 + hz - 1;
    if (circ) {
      gx = gx < 0 ? gx + nx : (gx >= nx ? gx - nx : gx);
      gy = gy < 0 ? gy + ny : (gy >= ny ? gy - ny : gy);
    }
    bf16x8 v;
    if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz) {
      v = *(const bf16x8_any*)(X + (((long)gx * ny + gy) * nz + gz) * CIN + 8 * g);
    } else {
      for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.0f;
    }
    *(bf16x8*)(tile + cell * CS + 8 * g) = v;
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, m = l & 31, h = l >> 5;
  f32x16 acc[CT2Y / 2][NT];
#pragma unroll
  for (int a = 0; a < CT2Y / 2; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  // fully unrolled: the tap of a K step does not depend on the lane (a step of 16 k is
  // one tap's channels 16 s' .. 16 s' + 15), so every tap offset is a constant and only
  // the channel offset 8 (l / 32) varies by lane
  const __bf16* tw = tile + ((w + 1) * GY + 1) * GZ * CS + (((m >> 4) * GZ + (m & 15) + 1) * CS) + 8 * h;
  const __bf16* wl = Wp + (long)m * (NSTEP * 32) + 8 * h;
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    const int kk0 = s * 16;          // the step's first k (lane half 0)
    int tap, ch0;
    conv_step_k(CIN, kk0 / 32, kk0 % 32, tap, ch0);
    if (tap > 26) tap = 26;          // padded K: weights are zero there
    const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
    bf16x8 b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[nt] = *(const bf16x8*)(wl + (long)nt * 32 * (NSTEP * 32) + kk0);
#pragma unroll
    for (int mt = 0; mt < CT2Y / 2; ++mt) {
      // cell ((w + 1 + dx), (2 mt + m/16 + 1 + dy), (m%16 + 1 + dz)), channel ch0 + 8 h
      const int off = ((dx * GY + 2 * mt + dy) * GZ + dz) * CS + ch0;
      const bf16x8 a = *(const bf16x8*)(tw + off);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[nt], acc[mt][nt], 0, 0, 0);
    }
  }
  const int xc = x0 + w;
#pragma unroll
  for (int mt = 0; mt < CT2Y / 2; ++mt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = nt * 32 + m;
      const float bn = bias[n];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 8 * (i / 4) + 4 * h + (i % 4);   // MFMA row of accumulator i
        const int yc = y0 + 2 * mt + (row >> 4), zc = z0 + (row & 15);
        if (xc < nx && yc < ny && zc < nz) {
          const long cell = ((long)xc * ny + yc) * nz + zc;
          float v = acc[mt][nt][i] + bn;
          if (pre) pre[cell * COUT + n] = v;
          if (mode & 1) v = gelu_t(v);
          if (mode & 2) {
            if (n < cout_real) Yf[cell * cout_real + n] = v;
          } else {
            Y[cell * COUT + n] = (__bf16)v;
          }
        }
      }
    }
  }
}

// The forward convolution for CIN <= 32 and 16 or 32 output channels (every layer of the SGS
// net and simpleCNN, both directions): a march along x with the weights in registers.
//
// A workgroup of 4 waves owns a column of 4 y rows and 16 z cells and a run of x planes, which
// it advances 4 at a time.  A wave owns 16 output channels (the MFMA's rows) and, of the four
// planes, WX (2 with 32 output channels, where two waves share a plane, 1 with 16) of 4 y rows
// of 16 z cells (the MFMA's columns).  An operand read from LDS (16 cells of one z run x 32 k)
// is used for every (x, y) tap that reaches it: 3 (WX 2) or 2 MFMAs per read on average; one
// per read, as with the cells as rows of one plane, needs all the LDS bandwidth there is.
// Half the output channels per wave is half the weights (108 VGPRs for 32 input channels),
// which leaves two waves per SIMD.
//
// LDS is a ring of 10 halo planes (6 rows x 18 cells): 6 that the step reads and the next 4,
// which arrive straight from memory (no registers) under the step's MFMAs.  The results are
// stored after the wait for them, so that no wait covers a store just issued.  The march
// reads each x plane once (108 cells per 64 outputs; a stand-alone 8 x 4 x 16 tile 135), and
// neighbouring columns, on one XCD, read their common rows at about the same time.
//
// Neither unit is saturated: at 240 x 240 x 120 the 32 -> 32 layer takes 366 us, its MFMAs
// alone 240 (a third of them 112, so 192 for the MFMAs themselves, 2.0 GHz under that load)
// and its memory traffic alone (0.52 GB read, 0.43 written) 215.  One wave per SIMD with all
// the weights, 4 x 4 x 16 tiles and 32 x 32 MFMAs took 575 there and 42 (now 31) at 96 x 96 x
// 48; 5 -> 32 277 (now 236) and 32 -> 5 287 (220).  No gain from wave priorities, from
// non-temporal stores (pre-activations 20 % slower) or from three waves per SIMD for 16
// input channels (365 us: spills).
//
// K: for 32 input channels one step per tap; for 16 a step is two z taps, (-1, 0) and (+1, -),
// lanes 0-31 reading the first and 32-63 the second (zeros where there is none).  Cells lie unpadded in LDS; for 32
// channels the upper and lower 32 bytes of a cell change places where bit 2 of its z position
// is set, which puts the 16 lanes that an operand read serves at a time (0-3, 12-15, 20-27 and
// 4-11, 16-19, 28-31 of each half wave) on all 64 banks.
//
// MODE: bit 0 GELU after the bias, bit 1 FP32 output Yf with cout_real channels (else BF16
// Y), bit 2 periodic x and y, bit 3 GELU gradient: `pre` is read (the FP32 pre-activation of
// the layer below, COUT channels) and Y = BF16((acc + bias) * gelu'(pre)), the data gradient
// and the k_gelu_bwd pass after it in one (bits 0-2 clear).
// ALIGNED: X starts at a 16-byte boundary, as the copies into LDS need; else the planes go
// through registers (240 x 240 x 120, 32 -> 32: 366 and 498 us; moving such an X to an
// aligned scratch copy first took 630 and memory that a caller may not have).
constexpr int RSX = 4, RTY = 4, RTZ = 16;   // planes per step; rows and cells of a column
constexpr int RRING = 2 * RSX + 2;          // halo planes in LDS

__device__ const unsigned k_zero_chunk[4] __attribute__((aligned(16))) = {0, 0, 0, 0};

template <int CIN, int COUT, int MODE, bool ALIGNED>
__global__ __launch_bounds__(256, 2) void k_conv3_rows(int nx, int ny, int nz, int run, const __bf16* __restrict__ X,
                                                       const __bf16* __restrict__ Wp, const float* __restrict__ bias,
                                                       int cout_real, __bf16* __restrict__ Y, float* __restrict__ Yf,
                                                       float* __restrict__ pre) {
  static_assert((CIN == 16 || CIN == 32) && (COUT == 16 || COUT == 32), "weights and accumulators fit 256 VGPRs");
  constexpr bool GELU = (MODE & 1) != 0, F32 = (MODE & 2) != 0, CIRC = (MODE & 4) != 0, GGRAD = (MODE & 8) != 0;
  static_assert(!GGRAD || (MODE & 7) == 0, "the GELU-gradient epilogue writes BF16 without GELU");
  constexpr int NH = COUT / 16, WX = NH;                        // channel halves; planes per wave and step
  constexpr int GY = RTY + 2, GZ = RTZ + 2, NCH = CIN / 8;      // halo rows, cells; 16-byte chunks of a cell
  constexpr int PLC = GY * GZ * NCH, GP = (PLC + 63) / 64;      // chunks of a plane; wave accesses that fetch it
  constexpr int PLANE = GP * 64 * 8;                            // LDS elements of a plane
  constexpr int NPF = (RSX * GP + 3) / 4;                       // accesses per wave and step
  constexpr int NZG = CIN == 32 ? 3 : 2;                        // K steps per (x, y) tap
  constexpr int KROW = ConvSteps<CIN>::NSTEP * 32;              // packed weights of one output channel
  // 16 input channels: zeros for the lanes of the second K step that have no tap, which read
  // them at the offset of every row (a zero weight times an infinity would be NaN)
  constexpr int ZEROS = CIN == 16 ? (GY - 1) * GZ * CIN + 8 : 0;
  __shared__ __attribute__((aligned(16))) __bf16 ring[RRING * PLANE + ZEROS];
  for (int e = threadIdx.x; e < ZEROS; e += 256) ring[RRING * PLANE + e] = (__bf16)0.0f;
  // workgroups: z tile, then row, then run of planes (conv_rows_grid)
  const TileId tb = xcd_tile();
  const unsigned tz = (nz + RTZ - 1) / RTZ, ty = (ny + RTY - 1) / RTY;
  const unsigned id = tb.x + gridDim.x * tb.y, col = id / tz, part = col / ty;
  const int z0 = (int)(id - col * tz) * RTZ, y0 = (int)(col - part * ty) * RTY;
  const int xa = (int)part * run, xb = min(xa + run, nx);
  if (xa >= nx) return;   // past the last workgroup of a grid in two dimensions
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, m = l & 15, g = l >> 4;
  const int ch = (w % NH) * 16 + 4 * g, xw = (w / NH) * WX;     // first output channel of the lane; first plane
  auto swz = [](int z) { return CIN == 32 ? (z >> 1) & 2 : 0; };
  // weights: rows are output channels, k this lane's 8 channels of the step's tap (CIN 16:
  // tap slot 27 of the packed rows is zero)
  bf16x8 wr[9][NZG];
  {
    const __bf16* wl = Wp + (long)((w % NH) * 16 + m) * KROW + 8 * (g % NCH);
#pragma unroll
    for (int xy = 0; xy < 9; ++xy)
#pragma unroll
      for (int zg = 0; zg < NZG; ++zg) {
        const int tap = CIN == 32 ? xy * 3 + zg : (zg == 0 ? xy * 3 + (g >> 1) : (g < 2 ? xy * 3 + 2 : 27));
        wr[xy][zg] = *(const bf16x8*)(wl + tap * CIN);
      }
  }
  const f32x4 bn = {bias[ch], bias[ch + 1], bias[ch + 2], bias[ch + 3]};
  // LDS element of this lane's operand in step zg of row 0 of a plane
  int lb[NZG];
#pragma unroll
  for (int zg = 0; zg < NZG; ++zg) {
    const int z = m + (CIN == 32 ? zg : (zg == 0 ? (g >> 1) : 2));
    lb[zg] = z * CIN + 8 * ((g % NCH) ^ swz(z));
  }
  // Fetch access q of a run of planes: 64 consecutive chunks q % GP of plane q / GP.  The
  // lane's chunk: row hy, cell hz, source chunk of the cell.
  auto chunk = [&](int q, int& hy, int& hz) {
    const int c = (q % GP) * 64 + l, cell = c / NCH;
    hy = cell / GZ;
    hz = cell - hy * GZ;
    return 8 * ((c % NCH) ^ swz(hz));
  };
  auto put = [&](int q, int slot, const void* src) {
    if (PLC % 64 == 0 || (q % GP) * 64 + l < PLC) {
      if constexpr (ALIGNED)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(ring + slot * PLANE + (q % GP) * 512),
                                         16, 0, 0);
      else
        *(bf16x8*)(ring + slot * PLANE + (q % GP) * 512 + 8 * l) = *(const bf16x8_any*)src;
    }
  };
  // byte offsets of the lane's chunks of a step's planes from (plane, y0 - 1, z0 - 1)
  uint32_t off[NPF];
#pragma unroll
  for (int j = 0; j < NPF; ++j) {
    const int q = w + 4 * j;
    int hy, hz;
    const int e = chunk(q, hy, hz);
    off[j] = (uint32_t)(((q / GP) * ny + hy) * nz + hz) * (CIN * 2) + 2 * e;
  }
  const bool inside = y0 > 0 && z0 > 0 && y0 + RTY < ny && z0 + RTZ < nz && (long)RRING * ny * nz * CIN * 2 < (1L << 32);
  // n planes from x = px on (cells outside the domain: zero, or their periodic image) into
  // the ring slots from `slot` on
  auto fetch = [&](int px, int n, int slot) {
    if (inside && n == RSX && px >= 0 && px + RSX <= nx) {   // uniform
      const char* corner = (const char*)(X + (((long)px * ny + (y0 - 1)) * nz + (z0 - 1)) * CIN);
#pragma unroll
      for (int j = 0; j < NPF; ++j) {
        const int q = w + 4 * j, s = slot + q / GP;
        if ((RSX * GP) % 4 == 0 || q < RSX * GP) put(q, s >= RRING ? s - RRING : s, corner + (size_t)off[j]);
      }
    } else {
      for (int q = w; q < n * GP; q += 4) {
        int hy, hz;
        const int e = chunk(q, hy, hz);
        int gx = px + q / GP, gy = y0 + hy - 1;
        const int gz = z0 + hz - 1, s = slot + q / GP;
        if (CIRC) {
          gx = gx < 0 ? gx + nx : (gx >= nx ? gx - nx : gx);
          gy = gy < 0 ? gy + ny : (gy >= ny ? gy - ny : gy);
        }
        const void* src = X + (((long)gx * ny + gy) * nz + gz) * CIN + e;
        if (!((unsigned)gx < (unsigned)nx && (unsigned)gy < (unsigned)ny && (unsigned)gz < (unsigned)nz)) src = k_zero_chunk;
        put(q, s >= RRING ? s - RRING : s, src);
      }
    }
  };
  fetch(xa - 1, RSX + 2, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int zc = z0 + m;
  int slot = 0;   // ring slot of plane x - 1
  for (int x = xa; x < xb; x += RSX) {
    __syncthreads();   // the step's planes are in LDS, and the slots of the next are no longer read
    if (x + RSX < xb) fetch(x + RSX + 1, RSX, slot + RSX + 2 >= RRING ? slot + RSX + 2 - RRING : slot + RSX + 2);
    f32x4 acc[WX][RTY];
#pragma unroll
    for (int a = 0; a < WX; ++a)
#pragma unroll
      for (int b = 0; b < RTY; ++b) acc[a][b] = bn;
    // operand groups (halo plane, step), one group of GY rows read ahead
    constexpr int NG = NZG * (WX + 2);
    bf16x8 f[2][GY];
    auto read = [&](int gi, bf16x8(&d)[GY]) {
      const int s = slot + xw + gi / NZG;
      int e = (s >= RRING ? s - RRING : s) * PLANE + lb[gi % NZG];
      if (CIN == 16 && gi % NZG == 1 && g >= 2) e = RRING * PLANE;
      const __bf16* r = ring + e;
#pragma unroll
      for (int y = 0; y < GY; ++y) d[y] = *(const bf16x8*)(r + y * GZ * CIN);
    };
    read(0, f[0]);
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
      if (gi + 1 < NG) read(gi + 1, f[(gi + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);  // the reads ahead of this group's MFMAs, not after them
      const int xp = gi / NZG, zg = gi % NZG;
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) {
          if (xp - kx < 0 || xp - kx >= WX) continue;
#pragma unroll
          for (int y = 0; y < RTY; ++y)
            acc[xp - kx][y] = mfma16(wr[kx * 3 + ky][zg], f[gi & 1][y + ky], acc[xp - kx][y]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = slot + RSX >= RRING ? slot + RSX - RRING : slot + RSX;
    // epilogue: accumulator i of (a, b) is cell (x + xw + a, y0 + b, z0 + m), channel ch + i
    auto rows = [&](auto&& f) {
#pragma unroll
      for (int a = 0; a < WX; ++a) {
        const int xc = x + xw + a;
        if (xc >= xb) continue;  // uniform over the wave
#pragma unroll
        for (int b = 0; b < RTY; ++b) {
          if (y0 + b >= ny) continue;  // uniform
          if (zc < nz) f(a, b, ((long)xc * ny + y0 + b) * nz + zc);
        }
      }
    };
    bf16x4 res[WX][RTY];
    if constexpr (GGRAD) {
      rows([&](int a, int b, long c0) {
        const f32x4 pa = *(const f32x4_any*)(pre + c0 * COUT + ch);
#pragma unroll
        for (int i = 0; i < 4; ++i)   // padded channels: +0
          res[a][b][i] = (__bf16)(ch + i < cout_real ? acc[a][b][i] * gelu_t_grad(pa[i]) : 0.f);
      });
    } else if constexpr (!F32) {
#pragma unroll
      for (int a = 0; a < WX; ++a)
#pragma unroll
        for (int b = 0; b < RTY; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) res[a][b][i] = (__bf16)(GELU ? gelu_t(acc[a][b][i]) : acc[a][b][i]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of the next planes
    rows([&](int a, int b, long c0) {
      const f32x4 v = acc[a][b];
      if (!GGRAD && pre) *(f32x4_any*)(pre + c0 * COUT + ch) = v;
      if constexpr (F32) {
        float* o = Yf + c0 * cout_real + ch;
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = GELU ? gelu_t(v[i]) : v[i];
        if (cout_real == COUT) {
          *(f32x4_any*)o = r;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (ch + i < cout_real) o[i] = r[i];
        }
      } else {
        *(bf16x4_any*)(Y + c0 * COUT + ch) = res[a][b];
      }
    });
  }
}

// x planes per workgroup: whole steps, so many that the workgroups fill the device evenly.
// A run costs its planes and about one step more (the first planes, the weights).
inline int conv_run(int nx, long cols, int resident) {
  int best = 0;
  double cost = 0.0;
  for (int runs = 1; runs <= (nx + RSX - 1) / RSX && runs <= 256; ++runs) {
    const int len = ((nx + runs - 1) / runs + RSX - 1) / RSX * RSX;
    const long n = cols * ((nx + len - 1) / len);
    const double c = (double)((n + resident - 1) / resident) * (len + RSX);
    if (best == 0 || c < cost) {
      best = len;
      cost = c;
    }
  }
  return best;
}

// One dimension up to 2^20 workgroups, as rows or z tiles in the grid's second or third would
// bound them at 2^16; more in rows of 2^20.
inline dim3 conv_rows_grid(int nx, int ny, int nz, int run) {
  const long n = (long)((nz + RTZ - 1) / RTZ) * ((ny + RTY - 1) / RTY) * ((nx + run - 1) / run);
  const long rows = (n + (1L << 20) - 1) >> 20;
  return dim3((unsigned)(rows > 1 ? 1L << 20 : n), (unsigned)rows);
}

// workgroups the device holds at once (occupancy from the runtime)
template <int CIN, int COUT, int MODE>
inline int conv_rows_resident() {
  static const int per_cu = [] {
    int per = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_conv3_rows<CIN, COUT, MODE, true>, 256, 0);
    return per > 0 ? per : 1;
  }();
  return device_cus() * per_cu;
}

// Weight gradient: dW[tap][c][n] += sum_p X[p + o(tap)][c] * G[p][n] over the cells of
// the grid (G: BF16 gradient of the pre-activation, COUT channels).  Workgroups loop
// over output tiles and store their FP32 partial sums (all 27 CIN COUT of them) in the
// slot of part that belongs to the workgroup; k_partial_sum then adds the slots in
// workgroup order, so the result does not depend on the order the workgroups ran in.
//
// The reduction runs over cells, so an MFMA operand lane needs 8 consecutive cells of
// one channel: both tiles are transposed into channel rows in LDS, the X rows as z-runs
// of XR = 24 elements per (c, hx, hy): the CTZ interior cells at 8..8+CTZ-1, the lower
// halo at 7 and the upper halo at 0.  A tap's z offset dz then shifts the 8-cell window
// by one element, which is rebuilt from one aligned 16-byte read and one neighbouring
// dword with byte-align (the upper halo read for dz = +1 at the end of the run wraps to
// offset 0, where it is stored).
constexpr int XR = 24;

// Eight waves; tile t + 1 is on its way to registers while tile t is multiplied.  The cells of
// a tile are halved between waves 0-3 and 4-7; within a half a wave takes some of the nine
// (dx, dy) pairs and, with 32 input channels, one of the two 16-channel groups: the three dz of
// a pair come from the same aligned read and its two neighbouring dwords, and the G operands
// serve all of a wave's taps.  The two waves of a SIMD hold the larger and the smaller share of
// pairs.  Neighbouring cells are transposed two at a time, so that LDS takes 4-byte writes.
// Four waves, one per SIMD (487 VGPRs), that took single taps waited for the tile's loads, read
// G again for every tap and wrote 2-byte scatters: us of the kernel at 96x96x48, 16->16, 16->32,
// 32->16 and 32->32 channels, 55, 61, 95 and 112; now 25, 31, 34 and 42.
// Workgroup b stores its partial sums at part + b * (27 CIN COUT + COUT): the weights' (the two
// halves added through LDS), then (with_bias) the bias gradient's, which rides along: once a G
// tile is in LDS, the 512 / COUT threads of each channel row add their consecutive cells of it,
// in order, to one running FP32 sum each; at the end the sums of a channel are added in thread
// order.
// element j of lo and of hi in one word
__device__ __forceinline__ unsigned pair16(const bf16x8& lo, const bf16x8& hi, int j) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 a = __builtin_bit_cast(u32x4, lo), b = __builtin_bit_cast(u32x4, hi);
  return __builtin_amdgcn_perm(b[j >> 1], a[j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
}

template <int CIN, int COUT>
__global__ __launch_bounds__(512) void k_conv3_wgrad(int nx, int ny, int nz, const __bf16* __restrict__ X,
                                                     const __bf16* __restrict__ G, float* __restrict__ part,
                                                     int with_bias) {
  static_assert(CTZ == 16 && XR == 24, "z-run layout assumes a 16-cell z tile");
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  constexpr int NCELL = CTX * CTY * CTZ, NL = HX * HY, NTH = 512;
  constexpr int MT = COUT / 16, NT = CIN / 16, NG = 4 / NT, PP = (9 + NG - 1) / NG;
  constexpr int TPC = NTH / COUT;   // bias: threads per channel row
  static_assert(NCELL == 256 && NCELL % (8 * TPC) == 0, "bias sums: whole 16-byte reads of a 256-cell row");
  // channel rows padded to an odd multiple of 16 bytes (modulo 256): the 16 lanes of an
  // operand read take 16 different channel rows at one offset, which then fall on 16
  // distinct bank groups instead of 1 (G rows of 512 bytes) or 4 (X rows of 1728)
  constexpr int XS = NL * XR + 8, GS = NCELL + 8;   // row strides in elements
  static_assert((XS * 2) % 32 == 16 && (GS * 2) % 32 == 16, "odd multiples of 16 bytes");
  __shared__ __attribute__((aligned(16))) __bf16 xt[CIN * XS];  // [c][hx][hy][z-run]
  __shared__ __attribute__((aligned(16))) __bf16 gt[COUT * GS];  // [n][cell]
  static_assert(4 * 64 * 3 * MT * 4 * sizeof(float) <= sizeof(xt), "the halves are added through the X tile");
  const int tid = threadIdx.x, l = tid & 63, m = l & 15, g = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), half = w >> 2, ct = NT == 2 ? w & 1 : 0;
  const int pg0 = NT == 2 ? (w >> 1) & 1 : w & 3, pg = half ? NG - 1 - pg0 : pg0;
  f32x4 acc[PP][3][MT];
#pragma unroll
  for (int i = 0; i < PP; ++i)
    for (int z = 0; z < 3; ++z)
      for (int mt = 0; mt < MT; ++mt) acc[i][z][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float bsum = 0.f;

  // items of a tile: pairs of cells along z, and the two z ends of every halo line
  constexpr int XP = NL * (CTZ / 2) * (CIN / 8), XE = NL * 2 * (CIN / 8), GP = NCELL / 2 * (COUT / 8);
  constexpr int NXP = (XP + NTH - 1) / NTH, NXE = (XE + NTH - 1) / NTH, NGP = (GP + NTH - 1) / NTH;
  bf16x8 xp[NXP][2], xe[NXE], gp[NGP][2];
  const int tz = (nz + CTZ - 1) / CTZ, ty = (ny + CTY - 1) / CTY, tx = (nx + CTX - 1) / CTX;
  const int ntiles = tx * ty * tz;
  auto ld = [&](const __bf16* f, int ch, int x, int y, int z, int c0) {
    bf16x8 v = {};
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz)
      v = *(const bf16x8_any*)(f + (((long)x * ny + y) * nz + z) * ch + c0);
    return v;
  };
  auto fetch = [&](int tile) {
    const int z0 = (tile % tz) * CTZ, y0 = ((tile / tz) % ty) * CTY, x0 = (tile / (tz * ty)) * CTX;
#pragma unroll
    for (int q = 0; q < NXP; ++q) {
      const int e = tid + q * NTH;
      if (e >= XP) break;
      const int zp = e % (CTZ / 2), line = (e / (CTZ / 2)) % NL, cg = e / (CTZ / 2 * NL);
      const int x = x0 + line / HY - 1, y = y0 + line % HY - 1, z = z0 + 2 * zp;
      xp[q][0] = ld(X, CIN, x, y, z, 8 * cg);
      xp[q][1] = ld(X, CIN, x, y, z + 1, 8 * cg);
    }
#pragma unroll
    for (int q = 0; q < NXE; ++q) {
      const int e = tid + q * NTH;
      if (e >= XE) break;
      const int hi = e & 1, line = (e >> 1) % NL, cg = (e >> 1) / NL;
      xe[q] = ld(X, CIN, x0 + line / HY - 1, y0 + line % HY - 1, hi ? z0 + CTZ : z0 - 1, 8 * cg);
    }
#pragma unroll
    for (int q = 0; q < NGP; ++q) {
      const int e = tid + q * NTH;
      if (e >= GP) break;
      const int cell = 2 * (e % (NCELL / 2)), ng = e / (NCELL / 2);
      const int x = x0 + cell / (CTY * CTZ), y = y0 + (cell / CTZ) % CTY, z = z0 + cell % CTZ;
      gp[q][0] = ld(G, COUT, x, y, z, 8 * ng);
      gp[q][1] = ld(G, COUT, x, y, z + 1, 8 * ng);
    }
  };
  auto place = [&]() {
#pragma unroll
    for (int q = 0; q < NXP; ++q) {
      const int e = tid + q * NTH;
      if (e >= XP) break;
      const int zp = e % (CTZ / 2), line = (e / (CTZ / 2)) % NL, cg = e / (CTZ / 2 * NL);
      __bf16* dst = xt + (8 * cg) * XS + line * XR + 8 + 2 * zp;
#pragma unroll
      for (int j = 0; j < 8; ++j) *(unsigned*)(dst + j * XS) = pair16(xp[q][0], xp[q][1], j);
    }
#pragma unroll
    for (int q = 0; q < NXE; ++q) {
      const int e = tid + q * NTH;
      if (e >= XE) break;
      const int hi = e & 1, line = (e >> 1) % NL, cg = (e >> 1) / NL;
      __bf16* dst = xt + (8 * cg) * XS + line * XR + (hi ? 0 : 7);
#pragma unroll
      for (int j = 0; j < 8; ++j) dst[j * XS] = xe[q][j];
    }
#pragma unroll
    for (int q = 0; q < NGP; ++q) {
      const int e = tid + q * NTH;
      if (e >= GP) break;
      const int cell = 2 * (e % (NCELL / 2)), ng = e / (NCELL / 2);
#pragma unroll
      for (int j = 0; j < 8; ++j) *(unsigned*)(gt + (8 * ng + j) * GS + cell) = pair16(gp[q][0], gp[q][1], j);
    }
  };
  const int step = gridDim.x;
  fetch(blockIdx.x);
  for (int tile = blockIdx.x; tile < ntiles; tile += step) {
    place();
    __syncthreads();
    if (tile + step < ntiles) fetch(tile + step);
    if (with_bias) {   // uniform
      const __bf16* row = gt + (tid / TPC) * GS + (tid % TPC) * (NCELL / TPC);
#pragma unroll
      for (int r = 0; r < NCELL / TPC / 8; ++r) {
        const bf16x8 v = *(const bf16x8*)(row + 8 * r);
#pragma unroll
        for (int j = 0; j < 8; ++j) bsum += (float)v[j];
      }
    }
#pragma unroll 1
    for (int ks = 4 * half; ks < 4 * half + 4; ++ks) {
      const int k0 = ks * 32 + 8 * g;  // 8 consecutive cells along z of one (hx, hy) line
      const int hx = ks >> 1, hy = 2 * (ks & 1) + (g >> 1), hz = 8 * (g & 1);
      bf16x8 a[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[mt] = *(const bf16x8*)(gt + (mt * 16 + m) * GS + k0);
      const __bf16* xc = xt + (ct * 16 + m) * XS + (hx * HY + hy) * XR;
#pragma unroll
      for (int i = 0; i < PP; ++i) {
        const int p = pg + i * NG;
        if (p >= 9) break;   // uniform over the wave
        const __bf16* row = xc + ((p / 3) * HY + p % 3) * XR;
        const u32x4 c = *(const u32x4*)(row + 8 + hz);
        const unsigned lo = *(const unsigned*)(row + 6 + hz);         // elements 6 + hz, 7 + hz
        const unsigned hi = *(const unsigned*)(row + (hz ? 0 : 16));  // element 16 + hz, or the upper halo
        u32x4 wl, wh;
        wl[0] = __builtin_amdgcn_alignbyte(c[0], lo, 2);
        wh[3] = __builtin_amdgcn_alignbyte(hi, c[3], 2);
#pragma unroll
        for (int j = 0; j < 3; ++j) wl[j + 1] = wh[j] = __builtin_amdgcn_alignbyte(c[j + 1], c[j], 2);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[i][0][mt] = mfma16(a[mt], __builtin_bit_cast(bf16x8, wl), acc[i][0][mt]);
          acc[i][1][mt] = mfma16(a[mt], __builtin_bit_cast(bf16x8, c), acc[i][1][mt]);
          acc[i][2][mt] = mfma16(a[mt], __builtin_bit_cast(bf16x8, wh), acc[i][2][mt]);
        }
      }
    }
    __syncthreads();
  }
  float* dW = part + (long)blockIdx.x * (27 * CIN * COUT + COUT);
  float* red = reinterpret_cast<float*>(xt);   // the X tile is no longer read
  if (with_bias) {
    red[tid] = bsum;
    __syncthreads();
    if (tid < COUT) {
      float s = 0.f;
      for (int i = 0; i < TPC; ++i) s += red[tid * TPC + i];
      dW[27 * CIN * COUT + tid] = s;
    }
    __syncthreads();
  }
  // D[row = n][col = c]: lane holds rows 4g+i of the M-tile, column m of the N-tile
  f32x4* share = reinterpret_cast<f32x4*>(red) + ((pg * NT + ct) * 3 * MT) * 64 + l;
#pragma unroll
  for (int i = 0; i < PP; ++i) {
    const int p = pg + i * NG;
    if (half) {
#pragma unroll
      for (int z = 0; z < 3; ++z)
        for (int mt = 0; mt < MT; ++mt) share[(z * MT + mt) * 64] = acc[i][z][mt];
    }
    __syncthreads();
    if (!half && p < 9) {
#pragma unroll
      for (int z = 0; z < 3; ++z)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const f32x4 s = acc[i][z][mt] + share[(z * MT + mt) * 64];
          *(f32x4*)(dW + ((long)(3 * p + z) * CIN + ct * 16 + m) * COUT + mt * 16 + 4 * g) = s;
        }
    }
    __syncthreads();
  }
}

// out[e] += sum over b < nb of part[b * stride + e], in order of b (e < n); the loads are
// issued 16 at a time ahead of their additions, so a thread waits for one memory round
// trip per 16 partial sums, not per partial sum
__global__ void k_partial_sum(int nb, int n, int stride, const float* __restrict__ part, float* __restrict__ out,
                              int n2, float* __restrict__ out2) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n + n2) return;
  float s = 0.f;
  int b = 0;
  for (; b + 16 <= nb; b += 16) {
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = part[(long)(b + q) * stride + e];
#pragma unroll
    for (int q = 0; q < 16; ++q) s += v[q];
  }
  for (; b < nb; ++b) s += part[(long)b * stride + e];
  if (e < n) {
    out[e] += s;
  } else {
    out2[e - n] += s;
  }
}

// channels n0 .. n0+7 of one FP32 row (zero from c_real on); vec: the row is 16-byte
// aligned (two 16-byte loads when all 8 channels are real)
__device__ __forceinline__ void load_row8(const float* __restrict__ src, int n0, int c_real, bool vec, float (&v)[8]) {
  if (vec && n0 + 8 <= c_real) {
    const float4 a = *(const float4*)(src + n0), b = *(const float4*)(src + n0 + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = n0 + j < c_real ? src[n0 + j] : 0.f;
  }
}

// k_gelu_bwd with one thread per 8 output channels of a cell (one 16-byte store), as
// k_to_bf16_cl8: nch = cp / 8, nchunk = ncell * nch < 2^31, gpre 16-byte aligned
// (vec bit 0: gpost rows 16-byte aligned, bit 1: pre rows)
__global__ void k_gelu_bwd8(unsigned nchunk, unsigned nch, int c_real, int cpre, const float* __restrict__ gpost,
                            int gstride, const float* __restrict__ pre, int gelu, int vec, __bf16* __restrict__ gpre) {
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nchunk) return;
  const unsigned p = t / nch;
  const int n0 = 8 * (int)(t - p * nch);
  float g[8], x[8];
  load_row8(gpost + (long)p * gstride, n0, c_real, (vec & 1) != 0, g);
  if (gelu) load_row8(pre + (long)p * cpre, n0, c_real, (vec & 2) != 0, x);
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float v = 0.f;
    if (n0 + j < c_real) {
      v = g[j];
      if (gelu) v *= gelu_t_grad(x[j]);
    }
    o[j] = (__bf16)v;
  }
  *(bf16x8*)(gpre + 8L * t) = o;
}

// g_pre = g_post * gelu'(pre) (or g_post when gelu is 0) -> BF16, cp channels (the
// channels >= c_real are zero)
__global__ void k_gelu_bwd(long ncell, int cp, int c_real, int cpre, const float* __restrict__ gpost, int gstride,
                           const float* __restrict__ pre, int gelu, __bf16* __restrict__ gpre) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ncell * cp) return;
  long p = t / cp;
  int n = (int)(t % cp);
  float v = 0.f;
  if (n < c_real) {
    v = gpost[p * gstride + n];
    if (gelu) v *= gelu_t_grad(pre[p * cpre + n]);
  }
  gpre[t] = (__bf16)v;
}

// Pack FP32 W[tap][cin][cout] into BF16 rows Wp[n][s*32 + k] of a CINP -> COUTP
// convolution.  flip = 1 packs the transposed convolution of the data gradient:
// input channels = cout, output channels = cin, taps mirrored (tap -> 26 - tap).
__global__ void k_conv3_pack(const float* __restrict__ W, int cin, int cout, int cinp, int coutp, int nstep,
                             int flip, __bf16* __restrict__ Wp) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)coutp * nstep * 32) return;
  int n = (int)(t / (nstep * 32));
  int k = (int)(t % (nstep * 32));
  int s = k / 32, kl = k % 32;
  int tap, ch;
  conv_step_k(cinp, s, kl, tap, ch);
  float v = 0.f;
  if (tap < 27) {
    if (!flip) {
      if (ch < cin && n < cout) v = W[((long)tap * cin + ch) * cout + n];
    } else {  // input channel ch is a forward output channel, output n a forward input channel
      if (ch < cout && n < cin) v = W[((long)(26 - tap) * cin + n) * cout + ch];
    }
  }
  Wp[t] = (__bf16)v;
}

// The same with one thread per 8 output channels of a cell (one 16-byte store) and 32-bit
// indexing: nch = cp / 8 chunks per cell, nchunk = ncell * nch < 2^31, out 16-byte aligned;
// vec: in and cs keep every row 16-byte aligned.
__global__ void k_to_bf16_cl8(unsigned nchunk, unsigned nch, int c_real, int cs, int vec, const float* __restrict__ in,
                              __bf16* __restrict__ out) {
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nchunk) return;
  const unsigned p = t / nch;
  const int n0 = 8 * (int)(t - p * nch);
  float x[8];
  load_row8(in + (long)p * cs, n0, c_real, vec != 0, x);
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (__bf16)x[j];
  *(bf16x8*)(out + 8L * t) = v;
}

// FP32 channels-last (c_real channels, stride cs) -> BF16 padded to cp channels
__global__ void k_to_bf16_cl(long ncell, int c_real, int cs, int cp, const float* __restrict__ in,
                             __bf16* __restrict__ out) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ncell * cp) return;
  long p = t / cp;
  int n = (int)(t % cp);
  out[t] = (__bf16)(n < c_real ? in[p * cs + n] : 0.f);
}

}  // namespace lex
