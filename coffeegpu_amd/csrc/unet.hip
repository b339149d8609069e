// U-Net building blocks for gfx950 (include/coffee_unet.h): BF16 activations
// and weights, FP32 accumulation on the matrix cores.
//
// The 3x3 convolution is an implicit GEMM.  With Cin % 32 == 0 it runs on
// v_mfma_f32_16x16x32_bf16, the input tile and the weights staged in LDS
// (conv3x3_tile; Cin = 16 too) or, where the images fill the tiles badly, the input
// from the caches (conv3x3_k32); otherwise, or with operands that are not 16-byte
// aligned, on v_mfma_f32_16x16x16_bf16 from global memory: the M dimension is
// 16 pixels per wavefront (4 wavefronts = 64 pixels per workgroup), N is 16*NB
// output channels, K runs over the 9 taps times the input channels in steps of
// 16.  NHWC with channels padded to 16 makes every A and B fragment one 8-byte
// load per lane (4 consecutive BF16 channels).
// Operand layout of the 16x16x16 instruction (wave64):
//   A[i][k] from lane i + 16*(k/4), element k%4;
//   B[k][j] from lane j + 16*(k/4), element k%4;
//   D[i][j] in lane j + 16*(i/4), element i%4.
// The backward data pass is the same kernel with the taps mirrored and the
// transposed weights.  The weight gradient reduces over pixels (K = pixels),
// split into ranges whose FP32 partial tiles are summed in a second pass, so
// results do not depend on scheduling.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "coffee_hip.h"
#include "coffee_unet.h"
#include "ctx.hpp"

namespace coffee {
namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // at any float's address
typedef uint16_t bf16;
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf2f(bf16 v) { return __uint_as_float((uint32_t)v << 16); }

__device__ __forceinline__ bf16 f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (bf16)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (bf16)(u >> 16);
}

int launch_check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(nullptr, COFFEE_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return COFFEE_OK;
}

// Operand layout of the 16x16x32 instruction (wave64):
//   A[i][k] from lane i + 16*(k/8), element k%8;
//   B[k][j] from lane j + 16*(k/8), element k%8;
//   D[i][j] in lane j + 16*(i/4), element i%4.
enum ConvForm { kOut, kMasked, kPoolBack, kUpBack };  // see conv_epilogue

struct ConvArgs {
  const bf16* in;
  const bf16* w;
  const float* bias;
  bf16* out;
  float* out32;
  int N, H, W, Cin, Cout, flip, relu;
  // input forms (conv3x3_tile)
  const bf16* in2;  // channels c1 .. Cin - 1 (concatenation)
  int c1, up;       // c1 = Cin without
  // output forms
  int form, csplit;
  const bf16* mask;
  const bf16* skip;
  bf16* out2;
  bf16* pool;
};

template <int NB>
__global__ void __launch_bounds__(256) conv3x3_mfma(const ConvArgs a) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const long P = (long)a.N * a.H * a.W;
  const long pix0 = ((long)blockIdx.x * 4 + wave) * 16;
  const int co0 = blockIdx.y * 16 * NB;
  const long pa = pix0 + li;
  int n = 0, y = 0, x = 0;
  const bool pvalid = pa < P;
  if (pvalid) {
    x = (int)(pa % a.W);
    const long t = pa / a.W;
    y = (int)(t % a.H);
    n = (int)(t / a.H);
  }
  f4 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) acc[b] = f4{0.f, 0.f, 0.f, 0.f};
  bool cvalid[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) cvalid[b] = co0 + b * 16 + li < a.Cout;
  for (int tap = 0; tap < 9; tap++) {
    int dy = tap / 3 - 1, dx = tap % 3 - 1;
    if (a.flip) {
      dy = -dy;
      dx = -dx;
    }
    const int yy = y + dy, xx = x + dx;
    const bool ok = pvalid && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W;
    const bf16* src = a.in + ((long)(n * a.H + (ok ? yy : 0)) * a.W + (ok ? xx : 0)) * a.Cin + 4 * lk;
    const bf16* wt = a.w + (long)tap * a.Cout * a.Cin + 4 * lk;
    for (int c0 = 0; c0 < a.Cin; c0 += 16) {
      s4 av = s4{0, 0, 0, 0};
      if (ok) av = *(const s4*)(src + c0);
#pragma unroll
      for (int b = 0; b < NB; b++) {
        s4 bv = s4{0, 0, 0, 0};
        if (cvalid[b]) bv = *(const s4*)(wt + (long)(co0 + b * 16 + li) * a.Cin + c0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc[b], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int co = co0 + b * 16 + li;
    if (!cvalid[b]) continue;
    const float bb = a.bias ? a.bias[co] : 0.f;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const long p = pix0 + 4 * lk + v;
      if (p >= P) continue;
      float val = acc[b][v] + bb;
      if (a.relu) val = val > 0.f ? val : 0.f;
      if (a.out) a.out[p * a.Cout + co] = f2bf(val);
      if (a.out32) a.out32[p * a.Cout + co] = val;
    }
  }
}

// The same convolution on v_mfma_f32_16x16x32_bf16 (twice the K of the
// 16x16x16 instruction per issue) for Cin % 32 == 0.  A workgroup of 4
// wavefronts computes 64*MB pixels x 16*NB output channels; K runs over the 9
// taps x Cin in steps of 32.  The weight slice of a step (16*NB channels x 32
// input channels) is staged in LDS, double-buffered and shared by the 4
// wavefronts; each wavefront's input fragments (16 B per lane) and the next
// weight slice are requested one step ahead.  Operand layout (wave64):
//   A[i][k] from lane i + 16*(k/8), element k%8;
//   B[k][j] from lane j + 16*(k/8), element k%8;
//   D[i][j] in lane j + 16*(i/4), element i%4.
template <int NB, int MB>
__global__ void __launch_bounds__(256) conv3x3_k32(const ConvArgs a) {
  constexpr int LDW = 40;  // LDS row: 32 input channels + 8 of padding (bank spread)
  __shared__ __attribute__((aligned(16))) bf16 wl[2][16 * NB * LDW];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const long P = (long)a.N * a.H * a.W;
  const long pixw = ((long)blockIdx.x * 4 + wave) * (16 * MB);
  const int co0 = blockIdx.y * 16 * NB;
  int pn[MB], py[MB], px[MB];
  bool pv[MB];
#pragma unroll
  for (int m = 0; m < MB; m++) {
    const long pa = pixw + m * 16 + li;
    pv[m] = pa < P;
    pn[m] = py[m] = px[m] = 0;
    if (pv[m]) {
      px[m] = (int)(pa % a.W);
      const long t = pa / a.W;
      py[m] = (int)(t % a.H);
      pn[m] = (int)(t / a.H);
    }
  }
  // weight staging: thread t loads 8 input channels (16 B) of row t/4
  const int wrow = threadIdx.x >> 2, wpart = threadIdx.x & 3;
  const bool wload = wrow < 16 * NB;
  const bool wvalid = wload && co0 + wrow < a.Cout;
  const int nci = a.Cin / 32, nk = 9 * nci;
  auto load_w = [&](int s) {
    s8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    const int tap = s / nci, c0 = (s - tap * nci) * 32;
    if (wvalid) v = *(const s8*)(a.w + ((long)tap * a.Cout + co0 + wrow) * a.Cin + c0 + 8 * wpart);
    return v;
  };
  auto load_a = [&](int s, s8 (&av)[MB]) {
    const int tap = s / nci, c0 = (s - tap * nci) * 32;
    int dy = tap / 3 - 1, dx = tap % 3 - 1;
    if (a.flip) {
      dy = -dy;
      dx = -dx;
    }
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const int yy = py[m] + dy, xx = px[m] + dx;
      av[m] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (pv[m] && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
        av[m] = *(const s8*)(a.in + ((long)(pn[m] * a.H + yy) * a.W + xx) * a.Cin + c0 + 8 * lk);
    }
  };
  f4 acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[m][b] = f4{0.f, 0.f, 0.f, 0.f};
  s8 acur[MB], anext[MB];
  s8 wnext = load_w(0);
  load_a(0, acur);
  if (wload) *(s8*)&wl[0][wrow * LDW + 8 * wpart] = wnext;
  __syncthreads();
  for (int s = 0; s < nk; s++) {
    if (s + 1 < nk) {
      wnext = load_w(s + 1);
      load_a(s + 1, anext);
    }
    const bf16* wb = wl[s & 1];
    bf8 bfr[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
      bfr[b] = __builtin_bit_cast(bf8, *(const s8*)&wb[(b * 16 + li) * LDW + 8 * lk]);
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const bf8 af = __builtin_bit_cast(bf8, acur[m]);
#pragma unroll
      for (int b = 0; b < NB; b++)
        acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[b], acc[m][b], 0, 0, 0);
    }
    if (s + 1 < nk) {
      // buffer (s + 1) & 1 was last read in step s - 1, before its barrier
      if (wload) *(s8*)&wl[(s + 1) & 1][wrow * LDW + 8 * wpart] = wnext;
#pragma unroll
      for (int m = 0; m < MB; m++) acur[m] = anext[m];
    }
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int co = co0 + b * 16 + li;
    if (co >= a.Cout) continue;
    const float bb = a.bias ? a.bias[co] : 0.f;
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const long p = pixw + m * 16 + 4 * lk + v;
        if (p >= P) continue;
        float val = acc[m][b][v] + bb;
        if (a.relu) val = val > 0.f ? val : 0.f;
        if (a.out) a.out[p * a.Cout + co] = f2bf(val);
        if (a.out32) a.out32[p * a.Cout + co] = val;
      }
  }
}

// Output forms of conv3x3_tile, from a wavefront's accumulators: acc[m][b][v] is
// image row y0 + m, column x0 + lane % 16, channel co0 + 16 b + 4 (lane / 16) + v,
// so a lane holds 4 consecutive channels of a pixel (one 8-byte store each) and
// needs no LDS; the pixel beside it is in lane ^ 1, the one below in acc[m + 1].
// The values rounded to BF16 between the operations are those the separate
// kernels store, so the fused forms give the same bits.
//   kOut: bias and ReLU, to `out` (BF16) and `out32`; with `pool`, also the 2x2
//     averages of the stored values (coffee_unet_pool2).
//   kMasked (backward data): the first csplit channels to `out` (stride
//     csplit), zero where `mask` (the ReLU output they are the gradient of) is not
//     positive; the others to `out2` unmasked (coffee_unet_combine).
//   kPoolBack: the gradient of a 2x2 average pool, a quarter of the value to
//     each of the four pixels of the finer grid, plus `skip`, masked
//     (coffee_unet_pool2_bwd, then combine).
//   kUpBack: the gradient of a nearest 2x upsampling, the sum of 2x2 stored
//     values, masked (coffee_unet_up2_bwd, then combine).
template <int MB, int NB>
__device__ __forceinline__ void conv_epilogue(const ConvArgs& a, const f4 (&acc)[MB][NB],
                                              const f4 (&bias)[NB], int img, int y0, int x, int co0) {
  const int lk = ((int)threadIdx.x & 63) >> 4;
  auto masked = [&](s4 o, const bf16* m) {
    const s4 mv = *(const s4*)m;
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (!(bf2f((bf16)mv[e]) > 0.f)) o[e] = 0;
    return o;
  };
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int c = co0 + 16 * b + 4 * lk;
    s4 o[MB];
#pragma unroll
    for (int m = 0; m < MB; m++) {
      const int y = y0 + m;
      const bool live = y < a.H && x < a.W;
      const long p = (long)(img * a.H + y) * a.W + x;
      f4 v = acc[m][b];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v[e] += bias[b][e];
        if (a.relu) v[e] = v[e] > 0.f ? v[e] : 0.f;
        o[m][e] = (short)f2bf(v[e]);
      }
      if (a.form == kOut && live) {
        if (a.out) *(s4*)(a.out + p * a.Cout + c) = o[m];
        if (a.out32) *(f4*)(a.out32 + p * a.Cout + c) = v;
      } else if (a.form == kMasked && live) {
        const bool first = c < a.csplit;
        const long w = first ? p * a.csplit + c : p * (a.Cout - a.csplit) + c - a.csplit;
        *(s4*)((first ? a.out : a.out2) + w) = first && a.mask ? masked(o[m], a.mask + w) : o[m];
      } else if (a.form == kPoolBack && live) {
        s4 d;
#pragma unroll
        for (int e = 0; e < 4; e++) d[e] = (short)f2bf(0.25f * bf2f((bf16)o[m][e]));
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const long w = ((2L * (img * a.H + y) + q / 2) * (2L * a.W) + 2 * x + q % 2) * a.Cout + c;
          s4 r = d;
          if (a.skip) {
            const s4 sk = *(const s4*)(a.skip + w);
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = (short)f2bf(bf2f((bf16)d[e]) + bf2f((bf16)sk[e]));
          }
          *(s4*)(a.out + w) = a.mask ? masked(r, a.mask + w) : r;
        }
      }
    }
    if constexpr (MB % 2 == 0) {
      if (a.form == kUpBack || a.pool) {
        bf16* const dst = a.form == kUpBack ? a.out : a.pool;
#pragma unroll
        for (int m = 0; m < MB; m += 2) {
          s4 r;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float u = bf2f((bf16)o[m][e]), d = bf2f((bf16)o[m + 1][e]);
            const float s = (u + __shfl_xor(u, 1)) + (d + __shfl_xor(d, 1));
            r[e] = (short)f2bf(a.form == kUpBack ? s : 0.25f * s);
          }
          const int y = y0 + m;
          if (y >= a.H || x >= a.W || (x & 1)) continue;
          const long w = ((long)(img * (a.H >> 1) + (y >> 1)) * (a.W >> 1) + (x >> 1)) * a.Cout + c;
          *(s4*)(dst + w) = a.form == kUpBack && a.mask ? masked(r, a.mask + w) : r;
        }
      }
    }
  }
}

// 16-byte chunk swizzle of the LDS rows of conv3x3_tile: chunk c of row k lives
// at c ^ csw(k).  On gfx950 a ds_read_b128 whose 64 lanes read chunk lane / 16 of
// 64-byte rows base + lane % 16 then runs as fast as a contiguous 1 KiB read,
// for every base (measured); unswizzled 64-byte rows, rows padded to 80 bytes
// and the swizzles (k >> 2) & 3 or k & 3 took 1.35x as long, and the forward
// convolution counted a third of its LDS cycles as bank conflicts with the
// padded rows.  Rows of 64 channels or more swizzle each 8 chunks.
template <int PARTS>
__device__ __forceinline__ int csw(int k) {
  return PARTS >= 8 ? k & 7 : PARTS == 4 ? (k >> 1) & 3 : (k >> 2) & 1;
}

// The convolution with the input tile in LDS.  A workgroup (4 wavefronts)
// computes a tile of TR image rows x 16 columns of one image x 16 NB output channels.
// For each chunk of CP input channels it stages the (TR + 2) x 18 input pixels
// (zero outside the image) and the 9 x 16 NB x CP weights in LDS once, so every
// input value crosses the memory hierarchy once per chunk instead of once per
// tap.  The next chunk's global loads are in flight, in registers, during the
// current chunk's MFMAs; the LDS is single-buffered, so that two workgroups share
// a CU (double-buffered, one workgroup per CU, measured 25-35 % slower).
//
// The order in which an output value takes its products is part of the result
// (the BF16 rounding of a layer feeds the next ones): chunks of 32 channels, and
// the taps within a chunk, for images of whole 16-pixel rows and whole 64-channel
// blocks (CP = 32, any Cin % 32 == 0); the taps, and the 32-channel chunks within
// a tap, otherwise, as conv3x3_k32 (CP = Cin = 32, 64, 128 or 256 here); Cin = 16
// takes the taps with v_mfma_f32_16x16x16_bf16, as conv3x3_mfma.  So every shape of
// less than 2^31 pixels has one result, whatever tile or kernel computes it, as long
// as in, w, out and out32 are 16-byte aligned (conv_tiled): others go to the kernels
// that sum by taps, 32 channels at a time or, with in or w off, 16.
//
// With few output channels the LDS read rate counts: one 16-byte-per-lane read
// takes 8 cycles of the CU's LDS, in which its SIMDs finish two MFMAs.  Where the
// registers allow (SHARE) a wavefront (rows wave MB .. + MB - 1) reads each input
// fragment of its MB + 2 rows and three column shifts once and applies all row
// shifts of the taps to it: 3 (MB + 2) + 9 NB reads per 9 MB NB MFMAs instead of 9
// (MB + NB).
//
// Input forms: `in2` continues the channels of `in` (concatenation without a
// copy); `up` reads the input of a nearest 2x upsampling at its coarse pixels.
// Output forms: conv_epilogue.
template <int TR, int NB, int CP, bool FLIP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CP > 64 ? 1 : TR == 16 || NB == 4 || CP == 64 ? 2 : 4)))
    conv3x3_tile(const ConvArgs a) {
  constexpr int TW = 16, IH = TR + 2, IW = TW + 2, NIN = IH * IW;
  constexpr int PARTS = CP / 8;                 // 16-byte chunks of an LDS row
  constexpr int SUB = CP < 32 ? 1 : CP / 32;    // MFMA steps per tap
  constexpr int MB = TR / 4, COB = 16 * NB, NW = 9 * COB * PARTS;
  constexpr int IN_E = NIN * CP, W_E = 9 * COB * CP;
  constexpr int IN_LD = (NIN * PARTS + 255) / 256;  // 16-byte input loads per thread
  constexpr int W_LD = (NW + 255) / 256;            // 16-byte weight loads per thread
  constexpr bool SHARE = CP >= 32 && NB > 1 && 3 * (MB + 2) * SUB <= (NB == 2 ? 12 : 24);
  static_assert(TR % 4 == 0, "rows per wavefront");
  __shared__ __attribute__((aligned(16))) bf16 lds[IN_E + W_E];

  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int tiles_x = (a.W + TW - 1) / TW, tiles_y = (a.H + TR - 1) / TR;
  const int tile = blockIdx.x;
  const int img = tile / (tiles_x * tiles_y);
  const int rest = tile - img * tiles_x * tiles_y;
  const int y0 = (rest / tiles_x) * TR, x0 = (rest % tiles_x) * TW;
  const int co0 = blockIdx.y * COB;
  const int nch = a.Cin / CP;

  int ipix[IN_LD];  // input pixel of this thread's u-th load, -1 outside the image
#pragma unroll
  for (int u = 0; u < IN_LD; u++) {
    const int idx = t + 256 * u, pix = idx / PARTS;
    const int yy = y0 - 1 + pix / IW, xx = x0 - 1 + pix % IW;
    ipix[u] = -1;
    if (idx < NIN * PARTS && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
      ipix[u] = a.up ? (img * (a.H >> 1) + (yy >> 1)) * (a.W >> 1) + (xx >> 1)
                     : (img * a.H + yy) * a.W + xx;
  }
  s8 rin[IN_LD], rw[W_LD];
  auto load_chunk = [&](int ch) __attribute__((always_inline)) {
    const int c0 = ch * CP;
#pragma unroll
    for (int u = 0; u < IN_LD; u++) {
      const int part = (t + 256 * u) % PARTS, c = c0 + 8 * part;
      const bool second = c >= a.c1;
      rin[u] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (ipix[u] >= 0)
        rin[u] = *(const s8*)(second ? a.in2 + (long)ipix[u] * (a.Cin - a.c1) + c - a.c1
                                     : a.in + (long)ipix[u] * a.c1 + c);
    }
#pragma unroll
    for (int u = 0; u < W_LD; u++) {
      const int idx = t + 256 * u;
      const int row = idx / PARTS, part = idx % PARTS;  // row = tap * COB + co
      const int tap = row / COB, co = row % COB;
      if (NW % 256 == 0 || idx < NW)
        rw[u] = *(const s8*)(a.w + ((long)tap * a.Cout + co0 + co) * a.Cin + c0 + 8 * part);
    }
  };
  auto store_chunk = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < IN_LD; u++) {
      const int idx = t + 256 * u, k = idx / PARTS;
      if (idx < NIN * PARTS) *(s8*)&lds[k * CP + 8 * ((idx % PARTS) ^ csw<PARTS>(k))] = rin[u];
    }
#pragma unroll
    for (int u = 0; u < W_LD; u++) {
      const int idx = t + 256 * u, k = idx / PARTS;
      if (NW % 256 == 0 || idx < NW)
        *(s8*)&lds[IN_E + k * CP + 8 * ((idx % PARTS) ^ csw<PARTS>(k))] = rw[u];
    }
  };
  // 16-byte fragment of row k, channels 32 s + 8 lk ..
  auto frag = [&](const bf16* base, int k, int s) {
    return __builtin_bit_cast(bf8, *(const s8*)&base[k * CP + 8 * ((4 * s + lk) ^ csw<PARTS>(k))]);
  };

  // D[i = channel][j = pixel]: the weights are operand A, so that a lane ends
  // up with consecutive channels of one pixel (conv_epilogue)
  f4 acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[m][b] = f4{0.f, 0.f, 0.f, 0.f};

  load_chunk(0);
  f4 bias[NB];
  auto load_bias = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; b++)
      bias[b] = a.bias ? (f4)*(const f4u*)(a.bias + co0 + 16 * b + 4 * lk) : f4{0.f, 0.f, 0.f, 0.f};
  };
  if constexpr (NB < 4) load_bias();  // where the registers are free, not after the MFMAs
  store_chunk();
  __syncthreads();
  for (int ch = 0; ch < nch; ch++) {
    if (ch + 1 < nch) load_chunk(ch + 1);
    bf8 shared[SHARE ? SUB : 1][3][SHARE ? MB + 2 : 1];
    if constexpr (SHARE) {
#pragma unroll
      for (int s = 0; s < SUB; s++)
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int r = 0; r < MB + 2; r++)
            shared[s][dx][r] = frag(lds, (wave * MB + r) * IW + li + dx, s);
    }
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
      // input offset (0..2, 0..2) of the tap's weights
      const int dy = FLIP ? 2 - tap / 3 : tap / 3, dx = FLIP ? 2 - tap % 3 : tap % 3;
      if constexpr (CP == 16) {
        // 8-byte fragments: channels 4 lk .. of a 32-byte row
        auto frag4 = [&](const bf16* base, int k) {
          return *(const s4*)&base[k * CP + 8 * ((lk >> 1) ^ csw<PARTS>(k)) + 4 * (lk & 1)];
        };
        s4 bfr[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) bfr[b] = frag4(lds + IN_E, tap * COB + b * 16 + li);
#pragma unroll
        for (int m = 0; m < MB; m++) {
          const s4 af = frag4(lds, (wave * MB + m + dy) * IW + li + dx);
#pragma unroll
          for (int b = 0; b < NB; b++)
            acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bfr[b], af, acc[m][b], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int s = 0; s < SUB; s++) {
          bf8 bfr[NB];
#pragma unroll
          for (int b = 0; b < NB; b++) bfr[b] = frag(lds + IN_E, tap * COB + b * 16 + li, s);
#pragma unroll
          for (int m = 0; m < MB; m++) {
            bf8 af;
            if constexpr (SHARE) af = shared[s][dx][m + dy];
            else af = frag(lds, (wave * MB + m + dy) * IW + li + dx, s);
#pragma unroll
            for (int b = 0; b < NB; b++)
              acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[b], af, acc[m][b], 0, 0, 0);
          }
        }
      }
    }
    if (ch + 1 < nch) {
      __syncthreads();  // every wavefront is done with this chunk
      store_chunk();
      __syncthreads();
    }
  }

  if constexpr (NB == 4) load_bias();
  conv_epilogue<MB, NB>(a, acc, bias, img, y0 + wave * MB, x0 + li, co0);
}

// One wavefront per (pixel range, tap, 16x16 tile of (co, ci)).
__global__ void __launch_bounds__(64)
    wgrad_mfma(const bf16* __restrict__ x, const bf16* __restrict__ dz, float* __restrict__ part,
               int N, int H, int W, int Cin, int Cout, long chunk) {
  const int lane = threadIdx.x;
  const int li = lane & 15, lk = lane >> 4;
  const int split = blockIdx.x, tap = blockIdx.y;
  const int ncib = Cin / 16;
  const int cob = blockIdx.z / ncib, cib = blockIdx.z % ncib;
  const int dy = tap / 3 - 1, dx = tap % 3 - 1;
  const long P = (long)N * H * W;
  const long p_begin = (long)split * chunk;
  const long p_end = p_begin + chunk < P ? p_begin + chunk : P;
  const int co = cob * 16 + li, ci = cib * 16 + li;
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  for (long p0 = p_begin; p0 < p_end; p0 += 16) {
    short av[4], bv[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const long p = p0 + 4 * lk + v;
      av[v] = 0;
      bv[v] = 0;
      if (p < p_end) {
        av[v] = (short)dz[p * Cout + co];
        const int px = (int)(p % W);
        const long t = p / W;
        const int py = (int)(t % H);
        const int pn = (int)(t / H);
        const int yy = py + dy, xx = px + dx;
        if (yy >= 0 && yy < H && xx >= 0 && xx < W)
          bv[v] = (short)x[((long)(pn * H + yy) * W + xx) * Cin + ci];
      }
    }
    const s4 a4 = s4{av[0], av[1], av[2], av[3]};
    const s4 b4 = s4{bv[0], bv[1], bv[2], bv[3]};
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a4, b4, acc, 0, 0, 0);
  }
  // D[i = co][j = ci]: lane holds co = cob*16 + 4*lk + v, ci = cib*16 + li
  float* dst = part + ((long)split * 9 + tap) * Cout * Cin;
#pragma unroll
  for (int v = 0; v < 4; v++) dst[(long)(cob * 16 + 4 * lk + v) * Cin + cib * 16 + li] = acc[v];
}

// Weight gradient on v_mfma_f32_16x16x32_bf16: for one tap and one pixel
// range a workgroup (4 wavefronts) computes a 64 (co) x 64 (ci) tile of
// dW[tap][co][ci] = sum_p dz[p][co] x[p + tap][ci] (GEMM with K = pixels).
// Each step stages 32 pixels of dz and of the shifted input in LDS, transposed
// to channel-major rows so that a lane's 8 consecutive pixels (one MFMA
// fragment) are one 16-byte read; the global loads (16 B = 8 channels of one
// pixel per thread) for the next step are issued before the current step's
// MFMAs.  Wavefront w computes channels co0 + 16 w .. + 15 against the 64
// input channels (4 MFMAs per step).  Channels beyond Cout / Cin and pixels
// beyond the range or the image are zero.  The sums of kLinear in the same order
// (wgrad_linear), for the calls that wgrad_taps_pays names and for 2^31 pixels and more.
__global__ void __launch_bounds__(256)
    wgrad_k32(const bf16* __restrict__ x, const bf16* __restrict__ dz, float* __restrict__ part,
              int N, int H, int W, int Cin, int Cout, long chunk) {
  constexpr int LDP = 40;  // LDS row: 32 pixels + 8 of padding (bank spread)
  __shared__ __attribute__((aligned(16))) bf16 dzt[2][64 * LDP];
  __shared__ __attribute__((aligned(16))) bf16 xt[2][64 * LDP];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int split = blockIdx.x, tap = blockIdx.y;
  const int ncib = (Cin + 63) / 64;
  const int co0 = (blockIdx.z / ncib) * 64, ci0 = (blockIdx.z % ncib) * 64;
  const int dy = tap / 3 - 1, dx = tap % 3 - 1;
  const long P = (long)N * H * W;
  const long p_begin = (long)split * chunk;
  const long p_end = p_begin + chunk < P ? p_begin + chunk : P;
  // staging: thread t moves 8 channels (16 B) of pixel t % 32 of the step,
  // channels 8 (t / 32) ..; consecutive lanes write consecutive LDS columns
  const int sp = threadIdx.x & 31, sc = (threadIdx.x >> 5) * 8;
  const bool dz_ok = co0 + sc < Cout, x_ok = ci0 + sc < Cin;
  auto fetch = [&](long k0, s8& vdz, s8& vx) {
    vdz = s8{0, 0, 0, 0, 0, 0, 0, 0};
    vx = s8{0, 0, 0, 0, 0, 0, 0, 0};
    const long p = k0 + sp;
    if (p >= p_end) return;
    if (dz_ok) vdz = *(const s8*)(dz + p * Cout + co0 + sc);
    const int px = (int)(p % W);
    const long t = p / W;
    const int py = (int)(t % H), pn = (int)(t / H);
    const int yy = py + dy, xx = px + dx;
    if (x_ok && yy >= 0 && yy < H && xx >= 0 && xx < W)
      vx = *(const s8*)(x + ((long)(pn * H + yy) * W + xx) * Cin + ci0 + sc);
  };
  auto stage = [&](int buf, const s8& vdz, const s8& vx) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
      dzt[buf][(sc + e) * LDP + sp] = (bf16)vdz[e];
      xt[buf][(sc + e) * LDP + sp] = (bf16)vx[e];
    }
  };
  f4 acc[4];
#pragma unroll
  for (int b = 0; b < 4; b++) acc[b] = f4{0.f, 0.f, 0.f, 0.f};
  s8 ndz, nx;
  fetch(p_begin, ndz, nx);
  stage(0, ndz, nx);
  __syncthreads();
  int buf = 0;
  for (long k0 = p_begin; k0 < p_end; k0 += 32) {
    const bool more = k0 + 32 < p_end;
    if (more) fetch(k0 + 32, ndz, nx);
    const bf8 af = __builtin_bit_cast(bf8, *(const s8*)&dzt[buf][(wave * 16 + li) * LDP + 8 * lk]);
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const bf8 bfr = __builtin_bit_cast(bf8, *(const s8*)&xt[buf][(b * 16 + li) * LDP + 8 * lk]);
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr, acc[b], 0, 0, 0);
    }
    // buffer buf ^ 1 was last read in the previous step, before its barrier
    if (more) stage(buf ^ 1, ndz, nx);
    __syncthreads();
    buf ^= 1;
  }
  // D[i = co][j = ci]: lane holds co = co0 + 16 wave + 4 lk + v, ci = ci0 + 16 b + li
  float* dst = part + ((long)split * 9 + tap) * Cout * Cin;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const int ci = ci0 + b * 16 + li;
    if (ci >= Cin) continue;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int co = co0 + wave * 16 + 4 * lk + v;
      if (co < Cout) dst[(long)co * Cin + ci] = acc[b][v];
    }
  }
}

// Transposing 64-bit LDS read of gfx950 (ds_read_b64_tr_b16).  Within each
// group of 16 lanes, lane 4 r + q names 4 consecutive 16-bit values (columns
// 4 q .. 4 q + 3 of "row" r); lane i of the group receives column i of rows
// 0 .. 3.  Two such reads give the 8 K values of a 16x16x32 MFMA operand
// from a matrix stored K-major (pixels as rows, channels contiguous).
typedef __attribute__((address_space(3))) s4 lds_s4;
__device__ __forceinline__ s4 lds_read_tr(const bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
}

template <int CIB, int COB, bool LIN>
constexpr int wgrad_lds() {  // bf16 values of its tiles
  return 128 * COB + (LIN ? 391 : 180) * (CIB + 8);
}

// 16-byte chunk swizzle of the dz tile of wgrad_block (pixel rows of C8 chunks):
// chunk c of pixel k lives at c ^ wswz(k).  With 32 or 64 channels it puts the 32 lanes of every transposing read (pixel rows 8 g + 4 h + r of a
// 32-pixel step) on distinct banks with no padding; the bits it uses (1 and 3) come
// only from the lane's own part of the pixel index.
template <int C8>
__device__ __forceinline__ int wswz(int k) {
  return C8 == 8 ? (k & 2) | ((k >> 1) & 4) : C8 == 4 ? (k & 2) | ((k >> 3) & 1) : 0;
}

// Order of the pixels of a weight gradient (part of its FP32 result): tiles of 8 x
// 16 or 4 x 16 pixels, or the pixels as they lie in memory.
enum WgradOrder { kTile8, kTile4, kLinear };

struct WgradArgs {
  const bf16* x;
  const bf16* dz;
  float* part;
  float* bpart;    // bias partials, or null
  const bf16* x2;  // input forms, as ConvArgs
  int N, H, W, Cin, Cout, c1, up;
  int order, ranges, per, ntiles;  // per: tiles (kLinear: pixels) per range
  int bblocks, bchunk;             // kept apart from the ranges: bias_part
  int split;                       // kLinear: workgroups that share out the taps (1 or 3)
};

// Layers of one launch (at most MAX: a single layer has no table to send and search,
// 1 us of its two launches), with the first workgroup of each (first[n] = total).
constexpr int kWgradLayers = 20;
template <int MAX>
struct WgradMany {
  int n, first[MAX + 1];
  WgradArgs l[MAX];
};

// Entry k of ascending first workgroups that workgroup b belongs to.
__device__ __forceinline__ int entry_of(const int* first, int n, int b) {
  int k = 0;
  while (k + 1 < n && b >= first[k + 1]) k++;
  return k;
}

// v / d for 0 <= v < d + 130, mul = 2^20 / d + 1 (exact for d < 256; from there on v /
// d is 0 or 1).
__device__ __forceinline__ int small_div(int v, int d, int mul) {
  return d < 256 ? (int)((unsigned)v * (unsigned)mul >> 20) : (int)(v >= d);
}

// Weight gradient with the pixels staged in LDS: a workgroup computes the 9 x COB
// (co) x CIB (ci) block of dW[tap][co][ci] = sum_p dz[p][co] x[p + tap][ci] over a
// range of pixels (GEMM with K = pixels), TP at a time.  dz (TP pixels x COB) and
// the input with its one-pixel halo lie in LDS as in memory (pixel rows, channels
// contiguous; 16-byte stores), and both MFMA operands are read with the transposing
// LDS read, so a tap's shift is only another row address and every staged value
// serves all nine taps.  Input rows are padded by 8 values.  The next tile's global
// loads are in flight during the current tile's MFMAs.
//
// The pixels are summed in the order `order` names, 32 per instruction
// (v_mfma_f32_16x16x32_bf16) and one chain per range, so that a training step gives
// the same gradients whatever the block shape: a sum in another order moves a BF16
// weight of the next step now and then, and with it every activation.
//   TR rows x 16 columns: the halo tile is (TR + 2) x 18 pixels.
//   kLinear: TP consecutive pixels; three strips of them, a row of the image above
//   and below (zero outside the image); where a tap leaves the row, or the pixel
//   the range, the lane reads a row of zeros instead.
// A wavefront owns 16 input channels against all COB output channels: with CIB = 64
// for all nine taps; with 32 or 16, 2 or 4 wavefronts share them out.  With DY (kLinear)
// a workgroup takes the three taps of row dy, one strip, and the wavefronts share
// out the output channels.  FORMS: x2 and up are looked at.  Pixels beyond
// the image are zero.  Partial blocks go to part[range][tap][co][ci] (summed in
// range order by wgrad_reduce); in the tile orders with bpart given, the workgroups
// of the first input-channel block also sum dz over their range, per output channel
// in a fixed order, into bpart[range][co].
template <int CIB, int COB, int ORDER, bool FORMS, bool DY = false>
__device__ __forceinline__ void wgrad_block(const WgradArgs& a, int range, int block, bf16* lds,
                                            int row0 = 0) {
  constexpr bool LIN = ORDER == kLinear;
  constexpr int TR = ORDER == kTile4 ? 4 : 8, TW = 16, TP = TR * TW;
  constexpr int XW = LIN ? TP + 2 : TW + 2, XP = (DY ? 1 : LIN ? 3 : TR + 2) * XW, XS = CIB + 8;
  constexpr int D8 = COB / 8, X8 = CIB / 8;       // 16-byte chunks per pixel
  constexpr int NDZ = (TP * D8 + 255) / 256;      // 16-byte dz loads per thread
  constexpr int NX = (XP * X8 + 255) / 256;       // 16-byte input loads per thread
  constexpr int WC = CIB / 16, TG = 4 / WC;       // wavefronts along ci, groups of taps
  constexpr int MC = DY ? 1 : COB / 16, NT = DY ? 3 : (9 + TG - 1) / TG;
  bf16* const dzs = lds;
  bf16* const xs = lds + TP * COB;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int wc = wave % WC, tg = wave / WC, m0 = DY ? tg : 0;  // m0: first 16 of COB
  const bool works = m0 < COB / 16;
  const int li = lane & 15, lk = lane >> 4;
  const int g = lane >> 4, r = (lane >> 2) & 3, q = lane & 3;
  const int ncib = a.Cin / CIB;
  const int co0 = (block / ncib) * COB, ci0 = (block % ncib) * CIB;
  const bool do_bias = !LIN && a.bpart && !a.bblocks && block % ncib == 0;
  const int H = a.H, W = a.W, Cin = a.Cin, Cout = a.Cout;
  const int tiles_x = LIN ? 1 : W / TW, tiles_y = (H + TR - 1) / TR;
  // kLinear: pixels, at most 2^31 - 1
  const int begin = range * a.per;
  const int end = (int)min((long)begin + a.per, (long)a.ntiles), stride = LIN ? TP : 1;
  const int mulW = (1 << 20) / W + 1, mulH = (1 << 20) / H + 1;

  s8 rdz[NDZ], rx[NX];
  int col0 = 0;  // column of the first pixel of the tile being loaded (kLinear)
  auto load_tile = [&](int tile) __attribute__((always_inline)) {
    // first pixel (kLinear) or corner of the tile
    int img, y0, x0;
    if constexpr (LIN) {
      const unsigned row = (unsigned)tile / (unsigned)W;
      col0 = x0 = (int)((unsigned)tile - row * W);
      img = (int)(row / (unsigned)H);
      y0 = (int)row - img * H;
    } else {
      img = tile / (tiles_x * tiles_y);
      const int rest = tile - img * tiles_x * tiles_y;
      y0 = (rest / tiles_x) * TR;
      x0 = (rest % tiles_x) * TW;
    }
#pragma unroll
    for (int u = 0; u < NDZ; u++) {
      const int idx = t + 256 * u, px = idx / D8, c8 = idx % D8;
      const int yy = y0 + px / TW, xx = x0 + px % TW;
      const bool in = LIN ? px < end - tile : yy < H;
      const long p = LIN ? (long)tile + px : (long)(img * H + yy) * W + xx;
      rdz[u] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if ((TP * D8 % 256 == 0 || idx < TP * D8) && in)
        rdz[u] = *(const s8*)(a.dz + p * Cout + co0 + 8 * c8);
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int idx = t + 256 * u;
      rx[u] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (idx < XP * X8) {
        const int pix = idx / X8, c = ci0 + 8 * (idx % X8);
        int yy, xx, im = img;
        bool in;
        if constexpr (LIN) {
          // pixel tile - 1 + pix % XW of the strip, a row up or down; the one
          // before column 0 serves no tap
          const int v = x0 + pix % XW - 1, down = small_div(max(v, 0), W, mulW);
          const int rr = y0 + down, next = small_div(rr, H, mulH);
          im += next;
          yy = rr - next * H + pix / XW + row0 - 1;
          xx = v - down * W;
          in = v >= 0 && im < a.N && yy >= 0 && yy < H;
        } else {
          yy = y0 - 1 + pix / XW;
          xx = x0 - 1 + pix % XW;
          in = yy >= 0 && yy < H && xx >= 0 && xx < W;
        }
        if (in) {
          const long p = FORMS && a.up ? (long)(im * (H >> 1) + (yy >> 1)) * (W >> 1) + (xx >> 1)
                                       : (long)(im * H + yy) * W + xx;
          if (FORMS && c >= a.c1) rx[u] = *(const s8*)(a.x2 + p * (Cin - a.c1) + c - a.c1);
          else rx[u] = *(const s8*)(a.x + p * (FORMS ? a.c1 : Cin) + c);
        }
      }
    }
  };
  auto store_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NDZ; u++) {
      const int idx = t + 256 * u, px = idx / D8, c8 = idx % D8;
      if (TP * D8 % 256 == 0 || idx < TP * D8)
        *(s8*)&dzs[px * COB + 8 * (c8 ^ wswz<D8>(px))] = rdz[u];
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int idx = t + 256 * u;
      if (idx < XP * X8) *(s8*)&xs[(idx / X8) * XS + 8 * (idx % X8)] = rx[u];
    }
  };
  // A: K index 8 g + 4 h + r of step st is pixel 32 st + 8 g + 4 h + r; the lane's
  // part ka fixes the swizzle, st and h add whole rows.
  const int ka = 8 * g + r;
  int abase[MC];  // offsets in dzs, as xbase and zero in xs
#pragma unroll
  for (int m = 0; m < MC; m++)
    abase[m] = (ka * COB + 8 * ((2 * (works ? m0 + m : 0) + (q >> 1)) ^ wswz<D8>(ka)) + 4 * (q & 1));
  // B: the same pixel, in the middle of the haloed input
  const int xchunk = 8 * (2 * wc + (q >> 1)) + 4 * (q & 1);
  const int xbase = xchunk + (LIN ? (DY ? 0 : XW) + ka + 1
                                  : ((g >> 1) + 1) * XW + 8 * (g & 1) + r + 1) * XS;
  const int zero = XP * XS + xchunk;
  if (LIN && t < CIB) xs[XP * XS + t] = 0;

  f4 acc[NT][MC];
#pragma unroll
  for (int k = 0; k < NT; k++)
#pragma unroll
    for (int m = 0; m < MC; m++) acc[k][m] = f4{0.f, 0.f, 0.f, 0.f};
  float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (begin < end) load_tile(begin);
  for (int tile = begin; tile < end; tile += stride) {
    const int left = LIN ? end - tile : TP;  // pixels of the tile in the range
    const int colt = col0;
    __syncthreads();  // every wavefront is done with the previous tile
    store_tile();
    __syncthreads();
    if (LIN ? left > TP : tile + 1 < end) load_tile(tile + stride);
    if (do_bias && t < 32 * D8) {
      // thread (pixel group t / D8, chunk t % D8): pixels t / D8, t / D8 + 32, ...
#pragma unroll
      for (int i = 0; i < TP / 32; i++) {
        const int px = t / D8 + 32 * i, c8 = t % D8;
        const s8 v = *(const s8*)&dzs[px * COB + 8 * (c8 ^ wswz<D8>(px))];
#pragma unroll
        for (int e = 0; e < 8; e++) bsum[e] += bf2f((bf16)v[e]);
      }
    }
#pragma unroll 1
    for (int st = 0; st < TP / 32 && 32 * st < left && works; st++) {
      bf8 af[MC];
#pragma unroll
      for (int m = 0; m < MC; m++) {
        const s4 lo = lds_read_tr(dzs + abase[m] + (32 * st) * COB);
        const s4 hi = lds_read_tr(dzs + abase[m] + (32 * st + 4) * COB);
        af[m] = __builtin_bit_cast(bf8, s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
      }
      // whether the lane's two pixels in the step have a neighbour to the left and
      // right
      const int row = (LIN ? 32 * st : 2 * st * XW) * XS;
      bool mid[2], lft[2], rgt[2];
      if constexpr (LIN) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int k = 32 * st + ka + 4 * h, v = colt + k, col = v - small_div(v, W, mulW) * W;
          mid[h] = k < left;
          lft[h] = mid[h] && col > 0;
          rgt[h] = mid[h] && col < W - 1;
        }
      }
#pragma unroll
      for (int i = 0; i < NT; i++) {
        const int tap = DY ? i : tg + TG * i;
        if (!DY && TG > 1 && tap >= 9) continue;
        const int dy = DY ? 0 : tap / 3 - 1, dx = tap % 3 - 1, off = (dy * XW + dx) * XS;
        auto from = [&](int h) {
          const int at = xbase + (row + off) + 4 * h * XS;
          if constexpr (!LIN) return at;
          const bool ok = dx == 0 ? mid[h] : (dx < 0 ? lft[h] : rgt[h]);
          return ok ? at : zero;
        };
        const s4 lo = lds_read_tr(xs + from(0)), hi = lds_read_tr(xs + from(1));
        const bf8 bfr = __builtin_bit_cast(bf8, s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
#pragma unroll
        for (int m = 0; m < MC; m++)
          acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[m], bfr, acc[i][m], 0, 0, 0);
      }
    }
  }
  // D[i = co][j = ci]: lane holds co = co0 + 16 m + 4 lk + v, ci = ci0 + 16 wc + li
  const int ci = ci0 + wc * 16 + li;
#pragma unroll
  for (int i = 0; i < NT; i++) {
    const int tap = DY ? 3 * row0 + i : tg + TG * i;
    if (tap >= 9 || !works) continue;
    float* dst = a.part + ((long)range * 9 + tap) * Cout * Cin;
#pragma unroll
    for (int m = 0; m < MC; m++)
#pragma unroll
      for (int v = 0; v < 4; v++) dst[(long)(co0 + (m0 + m) * 16 + 4 * lk + v) * Cin + ci] = acc[i][m][v];
  }
  if (do_bias) {
    // the 32 pixel groups' sums of each channel, added in group order
    __syncthreads();  // every wavefront is done with the last tile
    float* red = (float*)lds;
    if (t < 32 * D8)
#pragma unroll
      for (int e = 0; e < 8; e++) red[(t / D8) * COB + 8 * (t % D8) + e] = bsum[e];
    __syncthreads();
    if (t < COB) {
      float b = 0.f;
      for (int k = 0; k < 32; k++) b += red[k * COB + t];
      a.bpart[(long)range * Cout + co0 + t] = b;
    }
  }
}

// Bias gradient db[c] = sum_p dz[p][c] in two deterministic passes, for the orders
// that do not sum it with the weights.  Pass 1: block b sums the pixels [b chunk, (b
// + 1) chunk) of every channel, threads laid out channel-fastest so that a pixel's
// channels are one coalesced row (channel groups of up to 256; 256 / group pixel
// rows in parallel, summed in a fixed order).  Pass 2 adds the block partials in
// block order.
__device__ __forceinline__ void bias_part(const bf16* __restrict__ dz, float* __restrict__ part,
                                          long P, int C, long chunk, int b, float* red) {
  const long p0 = b * chunk;
  const long p1 = p0 + chunk < P ? p0 + chunk : P;
  for (int cb = 0; cb < C; cb += 256) {
    const int cw = C - cb < 256 ? C - cb : 256;
    const int rows = 256 / cw;
    const int c = (int)threadIdx.x % cw, r = (int)threadIdx.x / cw;
    float s = 0.f;
    if (r < rows)
      for (long p = p0 + r; p < p1; p += rows) s += bf2f(dz[p * C + cb + c]);
    red[threadIdx.x] = s;
    __syncthreads();
    if ((int)threadIdx.x < cw) {
      float t = 0.f;
      for (int k = 0; k < rows; k++) t += red[k * cw + threadIdx.x];
      part[(long)b * C + cb + threadIdx.x] = t;
    }
    __syncthreads();
  }
}

// Workgroups of a layer in the launch of its order: its bias_part
// blocks, then ranges x channel blocks.
template <int MAX, int ORDER>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
    wgrad_tiles(const WgradMany<MAX> m) {
  __shared__ __attribute__((aligned(16))) bf16 lds[wgrad_lds<64, 32, false>()];
  const int k = MAX > 1 ? entry_of(m.first, m.n, blockIdx.x) : 0;
  const WgradArgs a = m.l[k];
  const int b = blockIdx.x - m.first[k] - a.bblocks;
  if (b < 0) {
    bias_part(a.dz, a.bpart, (long)a.N * a.H * a.W, a.Cout, a.bchunk, b + a.bblocks, (float*)lds);
    return;
  }
  const int range = b % a.ranges, block = b / a.ranges;
  wgrad_block<64, 32, ORDER, true>(a, range, block, lds);
}

template <int MAX>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
    wgrad_linear(const WgradMany<MAX> m) {
  __shared__ __attribute__((aligned(16))) bf16 lds[wgrad_lds<32, 32, true>()];
  const int k = MAX > 1 ? entry_of(m.first, m.n, blockIdx.x) : 0;
  const WgradArgs a = m.l[k];
  const int b = blockIdx.x - m.first[k] - a.bblocks;
  if (b < 0) {
    bias_part(a.dz, a.bpart, (long)a.N * a.H * a.W, a.Cout, a.bchunk, b + a.bblocks, (float*)lds);
    return;
  }
  const int range = b % a.ranges, block = b / a.ranges;
  constexpr bool F = MAX > 1;
  if (MAX == 1 && a.split == 3) {
    if (a.Cin % 32 == 0) {
      if (a.Cout % 32 == 0) wgrad_block<32, 32, kLinear, F, true>(a, range, block / 3, lds, block % 3);
      else wgrad_block<32, 16, kLinear, F, true>(a, range, block / 3, lds, block % 3);
    } else {
      if (a.Cout % 32 == 0) wgrad_block<16, 32, kLinear, F, true>(a, range, block / 3, lds, block % 3);
      else wgrad_block<16, 16, kLinear, F, true>(a, range, block / 3, lds, block % 3);
    }
  } else if (a.Cin % 32 == 0) {
    if (a.Cout % 32 == 0) wgrad_block<32, 32, kLinear, F>(a, range, block, lds);
    else wgrad_block<32, 16, kLinear, F>(a, range, block, lds);
  } else {
    if (a.Cout % 32 == 0) wgrad_block<16, 32, kLinear, F>(a, range, block, lds);
    else wgrad_block<16, 16, kLinear, F>(a, range, block, lds);
  }
}

// One layer in a tile order, blocks of 64 x 64 channels (wgrad_block's chains, bit for
// bit; from it they spill 17 registers, and with 64 x 32 blocks 1.6 times the bytes are
// staged: 16 x 64 x 128, 128 -> 64 45 -> 62 and 72 us), for Cin % 64 == 0, Cout % 64 == 0
// and W % 16 == 0: a workgroup computes the 9 x 64 (co) x 64 (ci) block of
// dW[tap][co][ci] = sum_p dz[p][co] x[p + tap][ci] over a range of tiles of
// TR image rows x 16 columns.  dz (TR x 16 pixels x 64 co) and the input
// with its one-pixel halo are staged in LDS as they lie in memory (pixel
// rows, channels contiguous; 16-byte stores), and both MFMA operands are read
// with the transposing LDS read, so a tap's shift is only another row
// address (a constant offset from the lane's base) and every staged value
// serves all nine taps.  Input rows are padded to XS = 72 values.  Wavefront
// w owns input channels ci0 + 16 w .. + 15 against the 64 output channels:
// per 32-pixel step it reads 4 A fragments (shared by the taps) and 9 B
// fragments for 36 MFMAs (v_mfma_f32_16x16x32_bf16).  The next tile's
// global loads are in flight during the current tile's MFMAs.  Pixels beyond
// the image are zero.  Partial blocks per range go to
// part[range][tap][co][ci] (summed by wgrad_reduce in range order); when
// bpart is given, the workgroups of the first input-channel block also sum dz
// over their range, per output channel in a fixed order, into
// bpart[range][co].
template <int TR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
    wgrad_tr(const bf16* __restrict__ x, const bf16* __restrict__ dz, float* __restrict__ part,
             float* __restrict__ bpart, int N, int H, int W, int Cin, int Cout,
             int tiles_per_range, int ntiles) {
  constexpr int TW = 16, TP = TR * TW, XW = TW + 2, XP = (TR + 2) * XW, XS = 72;
  constexpr int NDZ = TP * 8 / 256;            // 16-byte dz loads per thread
  constexpr int NX = (XP * 8 + 255) / 256;     // 16-byte input loads per thread
  static_assert(TP % 32 == 0, "whole 32-pixel steps per tile");
  static_assert(32 * 64 <= XP * XS, "bias reduction fits in the input tile");
  __shared__ __attribute__((aligned(16))) bf16 dzs[TP * 64];
  __shared__ __attribute__((aligned(16))) bf16 xs[XP * XS];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int g = lane >> 4, r = (lane >> 2) & 3, q = lane & 3;
  const int range = blockIdx.x;
  const int ncib = Cin / 64;
  const int co0 = (blockIdx.y / ncib) * 64, ci0 = (blockIdx.y % ncib) * 64;
  const bool do_bias = bpart && blockIdx.y % ncib == 0;
  const int tiles_x = W / TW, tiles_y = (H + TR - 1) / TR;
  const int t_begin = range * tiles_per_range;
  const int t_end = min(t_begin + tiles_per_range, ntiles);

  s8 rdz[NDZ], rx[NX];
  auto load_tile = [&](int tile) __attribute__((always_inline)) {
    const int img = tile / (tiles_x * tiles_y);
    const int rest = tile - img * tiles_x * tiles_y;
    const int y0 = (rest / tiles_x) * TR, x0 = (rest % tiles_x) * TW;
#pragma unroll
    for (int u = 0; u < NDZ; u++) {
      const int idx = t + 256 * u, px = idx >> 3, c8 = idx & 7;
      const int yy = y0 + px / TW, xx = x0 + px % TW;
      rdz[u] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (yy < H) rdz[u] = *(const s8*)(dz + ((long)(img * H + yy) * W + xx) * Cout + co0 + 8 * c8);
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int idx = t + 256 * u;
      rx[u] = s8{0, 0, 0, 0, 0, 0, 0, 0};
      if (idx < XP * 8) {
        const int pix = idx >> 3, c8 = idx & 7;
        const int yy = y0 - 1 + pix / XW, xx = x0 - 1 + pix % XW;
        if (yy >= 0 && yy < H && xx >= 0 && xx < W)
          rx[u] = *(const s8*)(x + ((long)(img * H + yy) * W + xx) * Cin + ci0 + 8 * c8);
      }
    }
  };
  auto store_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NDZ; u++) {
      const int idx = t + 256 * u, px = idx >> 3, c8 = idx & 7;
      *(s8*)&dzs[px * 64 + 8 * (c8 ^ wswz<8>(px))] = rdz[u];
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int idx = t + 256 * u;
      if (idx < XP * 8) *(s8*)&xs[(idx >> 3) * XS + 8 * (idx & 7)] = rx[u];
    }
  };
  // A: K index 8 g + 4 h + r of step st is pixel 32 st + 16 (g / 2) + 8 (g % 2)
  // + 4 h + r; the lane's part ka fixes the swizzle, st and h add 64-value rows.
  const int ka = 16 * (g >> 1) + 8 * (g & 1) + r;
  const bf16* abase[4];
#pragma unroll
  for (int m = 0; m < 4; m++) abase[m] = &dzs[ka * 64 + 8 * ((2 * m + (q >> 1)) ^ wswz<8>(ka)) + 4 * (q & 1)];
  // B: the same pixel shifted by the tap, in the haloed input tile
  const bf16* xbase = &xs[(((g >> 1) + 1) * XW + 8 * (g & 1) + r + 1) * XS + 8 * (2 * wave + (q >> 1)) +
                          4 * (q & 1)];

  f4 acc[9][4];
#pragma unroll
  for (int k = 0; k < 9; k++)
#pragma unroll
    for (int m = 0; m < 4; m++) acc[k][m] = f4{0.f, 0.f, 0.f, 0.f};
  float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (t_begin < t_end) load_tile(t_begin);
  for (int tile = t_begin; tile < t_end; tile++) {
    __syncthreads();  // every wavefront is done with the previous tile
    store_tile();
    __syncthreads();
    if (tile + 1 < t_end) load_tile(tile + 1);
    if (do_bias) {
      // thread (pixel group t / 8, chunk t % 8): pixels t / 8, t / 8 + 32, ...
#pragma unroll
      for (int i = 0; i < TP / 32; i++) {
        const int px = (t >> 3) + 32 * i, c8 = t & 7;
        const s8 v = *(const s8*)&dzs[px * 64 + 8 * (c8 ^ wswz<8>(px))];
#pragma unroll
        for (int e = 0; e < 8; e++) bsum[e] += bf2f((bf16)v[e]);
      }
    }
#pragma unroll 1
    for (int st = 0; st < TP / 32; st++) {
      bf8 af[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const s4 lo = lds_read_tr(abase[m] + (32 * st) * 64);
        const s4 hi = lds_read_tr(abase[m] + (32 * st + 4) * 64);
        af[m] = __builtin_bit_cast(bf8, s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
      }
#pragma unroll
      for (int tap = 0; tap < 9; tap++) {
        const int dy = tap / 3 - 1, dx = tap % 3 - 1;
        const int off = ((2 * st + dy) * XW + dx) * XS;
        const s4 lo = lds_read_tr(xbase + off);
        const s4 hi = lds_read_tr(xbase + off + 4 * XS);
        const bf8 bfr = __builtin_bit_cast(bf8, s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
#pragma unroll
        for (int m = 0; m < 4; m++)
          acc[tap][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[m], bfr, acc[tap][m], 0, 0, 0);
      }
    }
  }
  // D[i = co][j = ci]: lane holds co = co0 + 16 m + 4 lk + v, ci = ci0 + 16 wave + li
  const int ci = ci0 + wave * 16 + li;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    float* dst = part + ((long)range * 9 + k) * Cout * Cin;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int v = 0; v < 4; v++) dst[(long)(co0 + m * 16 + 4 * lk + v) * Cin + ci] = acc[k][m][v];
  }
  if (do_bias) {
    // the 32 pixel groups' sums of each channel, added in group order
    __syncthreads();  // every wavefront is done with the last tile
    float* red = (float*)xs;  // 32 x 64 floats, inside the input tile
#pragma unroll
    for (int e = 0; e < 8; e++) red[(t >> 3) * 64 + 8 * (t & 7) + e] = bsum[e];
    __syncthreads();
    if (t < 64) {
      float b = 0.f;
      for (int k = 0; k < 32; k++) b += red[k * 64 + t];
      bpart[(long)range * Cout + co0 + t] = b;
    }
  }
}

// Sum of m values v(k), k = 0 .. m-1, as 8 interleaved partial sums (k mod 8)
// combined pairwise: a fixed order (deterministic results) whose loads do
// not wait on each other.
template <typename F>
__device__ __forceinline__ float sum8(int m, F&& v) {
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int k = 0;
  for (; k + 8 <= m; k += 8)
#pragma unroll
    for (int u = 0; u < 8; u++) s[u] += v(k + u);
  for (int u = 0; k + u < m; u++) s[u] += v(k + u);
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// Pass 2 of the bias: 4 partial rows x 64 channels per block, each thread adding
// every 4th block partial (sum8), then the 4 row sums in row order.
__device__ __forceinline__ void bias_sum(const float* __restrict__ part, float* __restrict__ db,
                                         int nb, int C, int block) {
  __shared__ float red[256];
  const int cl = (int)threadIdx.x & 63, r = (int)threadIdx.x >> 6;
  const int c = block * 64 + cl;
  float s = 0.f;
  if (c < C) {
    const int m = nb > r ? (nb - r + 3) / 4 : 0;  // partials r, r + 4, ...
    s = sum8(m, [&](int k) { return part[(long)(r + 4 * k) * C + c]; });
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (r == 0 && c < C) db[c] = ((red[cl] + red[64 + cl]) + red[128 + cl]) + red[192 + cl];
}

struct ReduceArgs {
  const float* part;
  const float* bpart;
  float* dW;
  float* db;
  long n;
  int nb, ranges;
  int bblocks, sums;  // bias_sum of bblocks partials, in `sums` workgroups
};
template <int MAX>
struct ReduceMany {
  int n, first[MAX + 1];
  ReduceArgs l[MAX];
};

// dW[i] = sum over ranges of part[range][i], and db[c] = sum over ranges of
// bpart[range][c] (threads n .. n + nb - 1 of a layer), in range order.
template <int MAX>
__global__ void __launch_bounds__(256) wgrad_reduce(const ReduceMany<MAX> m) {
  const int k = MAX > 1 ? entry_of(m.first, m.n, blockIdx.x) : 0;
  const ReduceArgs& a = m.l[k];
  const int b = blockIdx.x - m.first[k];
  if (b < a.sums) {
    bias_sum(a.bpart, a.db, a.bblocks, a.nb, b);
    return;
  }
  const long i = (b - a.sums) * 256L + threadIdx.x;
  if (i < a.n) a.dW[i] = sum8(a.ranges, [&](int r) { return a.part[r * a.n + i]; });
  else if (!a.sums && i < a.n + a.nb)
    a.db[i - a.n] = sum8(a.ranges, [&](int r) { return a.bpart[(long)r * a.nb + (i - a.n)]; });
}

__global__ void __launch_bounds__(256) bias_grad_part(const bf16* __restrict__ dz,
                                                      float* __restrict__ part, long P, int C,
                                                      long chunk) {
  __shared__ float red[256];
  bias_part(dz, part, P, C, chunk, blockIdx.x, red);
}

__global__ void __launch_bounds__(256) bias_grad_sum(const float* __restrict__ part,
                                                     float* __restrict__ db, int nb, int C) {
  bias_sum(part, db, nb, C, blockIdx.x);
}

__global__ void combine_kernel(bf16* __restrict__ out, int ost, int ooff, const bf16* __restrict__ a,
                               int ast, int aoff, const bf16* __restrict__ b, int bst, int boff,
                               const bf16* __restrict__ mask, int mst, int moff, int nc, long npix) {
  const long total = npix * nc;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long p = i / nc;
    const int c = (int)(i % nc);
    float v = bf2f(a[p * ast + aoff + c]);
    if (b) v += bf2f(b[p * bst + boff + c]);
    if (mask && !(bf2f(mask[p * mst + moff + c]) > 0.f)) v = 0.f;
    out[p * ost + ooff + c] = f2bf(v);
  }
}

// h, w: sizes of the fine grid.
__global__ void pool2_kernel(const bf16* __restrict__ in, bf16* __restrict__ out, int N, int h, int w,
                             int C) {
  const int h2 = h / 2, w2 = w / 2;
  const long total = (long)N * h2 * w2 * C;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    long t = i / C;
    const int x = (int)(t % w2);
    t /= w2;
    const int y = (int)(t % h2);
    const int n = (int)(t / h2);
    const long b = ((long)(n * h + 2 * y) * w + 2 * x) * C + c;
    const float s = (bf2f(in[b]) + bf2f(in[b + C])) + (bf2f(in[b + (long)w * C]) + bf2f(in[b + (long)w * C + C]));
    out[i] = f2bf(0.25f * s);
  }
}

__global__ void pool2_bwd_kernel(const bf16* __restrict__ dy, bf16* __restrict__ dx, int N, int h,
                                 int w, int C) {
  const long total = (long)N * h * w * C;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    long t = i / C;
    const int x = (int)(t % w);
    t /= w;
    const int y = (int)(t % h);
    const int n = (int)(t / h);
    dx[i] = f2bf(0.25f * bf2f(dy[((long)(n * (h / 2) + y / 2) * (w / 2) + x / 2) * C + c]));
  }
}

__global__ void up2_kernel(const bf16* __restrict__ in, bf16* __restrict__ out, int N, int h, int w,
                           int C) {
  const long total = (long)N * h * w * C;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    long t = i / C;
    const int x = (int)(t % w);
    t /= w;
    const int y = (int)(t % h);
    const int n = (int)(t / h);
    out[i] = in[((long)(n * (h / 2) + y / 2) * (w / 2) + x / 2) * C + c];
  }
}

__global__ void up2_bwd_kernel(const bf16* __restrict__ dy, bf16* __restrict__ dx, int N, int h,
                               int w, int C) {
  const int h2 = h / 2, w2 = w / 2;
  const long total = (long)N * h2 * w2 * C;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int c = (int)(i % C);
    long t = i / C;
    const int x = (int)(t % w2);
    t /= w2;
    const int y = (int)(t % h2);
    const int n = (int)(t / h2);
    const long b = ((long)(n * h + 2 * y) * w + 2 * x) * C + c;
    const float s = (bf2f(dy[b]) + bf2f(dy[b + C])) + (bf2f(dy[b + (long)w * C]) + bf2f(dy[b + (long)w * C + C]));
    dx[i] = f2bf(s);
  }
}

constexpr int kMseBlocks = COFFEE_UNET_MSE_WORK;

double mse_sum(const double* part, long npix, int nc) {
  double tot = 0.0;
  for (int b = 0; b < kMseBlocks; b++) tot += part[b];
  return tot / ((double)npix * nc);
}

__global__ void __launch_bounds__(256)
    mse_kernel(const float* __restrict__ out32, int cst, const float* __restrict__ target, int nc,
               long npix, bf16* __restrict__ dout, double* __restrict__ part) {
  __shared__ double red[256];
  const double scale = 2.0 / ((double)npix * nc);
  double s = 0.0;
  const long total = npix * cst;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long p = i / cst;
    const int c = (int)(i % cst);
    float g = 0.f;
    if (c < nc) {
      const double d = (double)out32[i] - (double)target[p * nc + c];
      s += d * d;
      g = (float)(scale * d);
    }
    dout[i] = f2bf(g);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int m = 128; m > 0; m >>= 1) {
    if ((int)threadIdx.x < m) red[threadIdx.x] += red[threadIdx.x + m];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, long n, float lr, float b1, float b2, float eps,
                            float c1, float c2) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

struct AdamArgs {
  float* p;
  const float* g;
  float* m;
  float* v;
  bf16* wb;  // [9][cout][cin] and its transpose, or null
  bf16* wbt;
  int n, cout, cin;
};
constexpr int kAdamTensors = 48;
struct AdamMany {
  int n, first[kAdamTensors + 1];
  float lr, b1, b2, eps, c1, c2;
  AdamArgs l[kAdamTensors];
};

// Adam step of many tensors and the BF16 copies of their new weights: a
// workgroup takes 32 x 32 channels of one tap (1024 values of a bias), whose
// transpose goes through LDS so that both copies are stored along their rows.
__global__ void __launch_bounds__(256) adam_many_kernel(const AdamMany t) {
  __shared__ bf16 tile[32][34];
  const int k = entry_of(t.first, t.n, blockIdx.x);
  const AdamArgs& a = t.l[k];
  const int b = blockIdx.x - t.first[k];
  auto step = [&](int i) {
    const float gi = a.g[i];
    const float mi = t.b1 * a.m[i] + (1.f - t.b1) * gi;
    const float vi = t.b2 * a.v[i] + (1.f - t.b2) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    const float p = a.p[i] - t.lr * (mi / t.c1) / (sqrtf(vi / t.c2) + t.eps);
    a.p[i] = p;
    return p;
  };
  if (!a.wb) {
    for (int i = b * 1024 + threadIdx.x; i < min(a.n, (b + 1) * 1024); i += 256) step(i);
    return;
  }
  const int nci = (a.cin + 31) / 32, nco = (a.cout + 31) / 32;
  const int ci0 = (b % nci) * 32, co0 = (b / nci % nco) * 32, tap = b / (nci * nco);
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int co = co0 + y + 8 * u, ci = ci0 + x;
    if (co >= a.cout || ci >= a.cin) continue;
    const int i = (tap * a.cout + co) * a.cin + ci;
    const bf16 w = f2bf(step(i));
    a.wb[i] = w;
    tile[y + 8 * u][x] = w;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int ci = ci0 + y + 8 * u, co = co0 + x;
    if (co < a.cout && ci < a.cin) a.wbt[(tap * a.cin + ci) * a.cout + co] = tile[x][y + 8 * u];
  }
}

__global__ void weights_bf16_kernel(const float* __restrict__ w32, bf16* __restrict__ wb,
                                    bf16* __restrict__ wbt, int Cout, int Cin) {
  const long total = 9L * Cout * Cin;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int ci = (int)(i % Cin);
    const long t = i / Cin;
    const int co = (int)(t % Cout);
    const int tap = (int)(t / Cout);
    const bf16 v = f2bf(w32[i]);
    wb[i] = v;
    wbt[((long)tap * Cin + ci) * Cout + co] = v;
  }
}

__global__ void to_bf16_kernel(const float* __restrict__ in, bf16* __restrict__ out, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    out[i] = f2bf(in[i]);
}

__global__ void from_bf16_kernel(const bf16* __restrict__ in, float* __restrict__ out, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    out[i] = bf2f(in[i]);
}

template <typename T>
__global__ void pack_kernel(const T* f0, const T* f1, const T* f2, const T* f3, const T* f4_,
                            const T* f5, int dims0, int g0, int g1, int n0, int n1, double x0,
                            double dx, double dy, double rpow, double extra, void* out, int out32,
                            int cst, long base) {
  const long total = (long)n0 * n1 * cst;
  const T* F[6] = {f0, f1, f2, f3, f4_, f5};
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
    const int c = (int)(t % cst);
    const long pix = t / cst;
    const int i = (int)(pix % n0);
    const int j = (int)(pix / n0);
    double v = 0.0;
    if (c < 6) {
      const double r = exp(x0 + dx * i);
      const double th = dy * j;
      const double h = (c % 3 == 2) ? r * sin(th) : r;
      v = (double)F[c][(long)(i + g0) + (long)(j + g1) * dims0] * h * pow(r, rpow);
    } else if (c == 6) {
      v = extra;
    }
    const long o = base + t;
    if (out32) ((float*)out)[o] = (float)v;
    else ((bf16*)out)[o] = f2bf((float)v);
  }
}

template <typename T>
__global__ void unpack_kernel(const float* in, int cst, long base, T* f0, T* f1, T* f2, T* f3,
                              T* f4_, T* f5, int dims0, int g0, int g1, int n0, int n1, double x0,
                              double dx, double dy, double rpow) {
  const long total = (long)n0 * n1 * 6;
  T* F[6] = {f0, f1, f2, f3, f4_, f5};
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
    const int c = (int)(t % 6);
    const long pix = t / 6;
    const int i = (int)(pix % n0);
    const int j = (int)(pix / n0);
    const double r = exp(x0 + dx * i);
    const double th = dy * j;
    const double h = (c % 3 == 2) ? r * sin(th) : r;
    const double den = h * pow(r, rpow);
    const double v = fabs(den) > 1e-12 ? (double)in[base + pix * cst + c] / den : 0.0;
    F[c][(long)(i + g0) + (long)(j + g1) * dims0] = (T)v;
  }
}

// Corotation: E = -(Omega x r) x B with v = Omega r sin(theta) (phi direction),
// in upper components of x = ln r, theta: E^x = v B^theta, E^theta = -v B^x,
// E^phi = 0 (boundary_pulsar_sph applies the same relation inside the star).
template <typename T>
__global__ void corotate_kernel(T* ex, T* ey, T* ez, const T* bx, const T* by, int dims0, int g0,
                                int g1, int n0, int n1, double x0, double dx, double dy,
                                double omega) {
  const long total = (long)n0 * n1;
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
    const int i = (int)(t % n0), j = (int)(t / n0);
    const long c = (long)(i + g0) + (long)(j + g1) * dims0;
    const double v = omega * exp(x0 + dx * i) * sin(dy * j);
    ex[c] = (T)(v * (double)by[c]);
    ey[c] = (T)(-v * (double)bx[c]);
    ez[c] = T(0);
  }
}

int grid_for(long total, int block = 256) {
  long b = (total + block - 1) / block;
  return (int)(b < 1 ? 1 : (b > 65535 ? 65535 : b));
}

bool aligned16(const void* p) { return (uintptr_t)p % 16 == 0; }

// The order of products of a shape (see conv3x3_tile): by 32-channel chunks, or
// by taps.
bool conv_by_chunks(const ConvArgs& a) {
  return a.Cin % 32 == 0 && a.Cout % 64 == 0 && a.W % 16 == 0;
}

// Whether conv3x3_tile takes the convolution: 16-byte aligned arrays, pixel
// indices of its input in 32 bits, and a channel count it has the shape's order for.
bool conv_tiled(const ConvArgs& a) {
  return (conv_by_chunks(a) || a.Cin == 16 || a.Cin == 32 || a.Cin == 64 || a.Cin == 128 ||
          a.Cin == 256) &&
         (long)a.N * a.H * a.W <= 2147483647L && aligned16(a.in) && aligned16(a.w) &&
         aligned16(a.out) && aligned16(a.out32);
}

// Outputs of 2 x 2 pixels: a wavefront has to hold both rows (tiles of 8 rows).
bool conv_pairs(const ConvArgs& a) { return a.form == kUpBack || a.pool; }

// Tile of conv3x3_tile: image rows, 16-channel blocks of the output, channels
// staged at once.
struct ConvTile {
  int tr, nb, cp;
};

long conv_groups(const ConvArgs& a, int tr, int nb) {
  return (long)a.N * ((a.W + 15) / 16) * ((a.H + tr - 1) / tr) * (a.Cout / (16 * nb));
}

// The largest (most MFMAs per LDS read, least halo) that still gives two
// workgroups per CU, else one with more workgroups; 4 rows for images of no more
// (8 x 1 x 16384, 32 -> 64 83 us with 8 rows and 64 channels, 62 with 4 and 32).
ConvTile conv_tile(const ConvArgs& a) {
  const int cp = conv_by_chunks(a) ? 32 : a.Cin;
  const bool c32 = a.Cout % 32 == 0, pairs = conv_pairs(a);
  if (cp == 256) return {4, 1, 256};  // all channels staged at once: 126 KiB of LDS
  if (cp == 128) return {pairs ? 8 : 4, c32 ? 2 : 1, 128};  // 63 to 117 KiB
  if (a.Cout % 64 == 0 && cp == 32 && (a.H > 4 || pairs)) {
    if (a.H > 8 && conv_groups(a, 16, 4) >= 512) return {16, 4, 32};
    if (conv_groups(a, 8, 4) >= 512) return {8, 4, 32};
  }
  if (c32 && (pairs || (a.H > 4 && conv_groups(a, 8, 2) >= 256))) return {8, 2, cp};
  if (c32) return {4, 2, cp};
  return {8, 1, cp};
}

// 64 or 128 pixels (mb = 1 or 2) x 16 nb channels per workgroup of the kernels that
// sum by taps from global memory: conv3x3_k32 takes two 16-pixel row blocks per
// wavefront when that still leaves two workgroups per CU.
struct ConvTaps {
  int nb, mb;
  long groups;
};
ConvTaps conv_taps(const ConvArgs& a) {
  const long P = (long)a.N * a.H * a.W;
  const int nb = a.Cout % 64 == 0 ? 4 : a.Cout % 32 == 0 ? 2 : 1;
  const long cb = a.Cout / (16 * nb);
  const int mb = a.Cin % 32 == 0 && (P + 127) / 128 * cb >= 512 ? 2 : 1;
  return {nb, mb, (P + 64 * mb - 1) / (64 * mb) * cb};
}

// Arguments that are sizes alone (pairs: outputs of 2 x 2 pixels).
ConvArgs conv_sizes(int n, int h, int w, int cin, int cout, bool pairs) {
  ConvArgs a{};
  a.N = n;
  a.H = h;
  a.W = w;
  a.Cin = cin;
  a.Cout = cout;
  a.form = pairs ? kUpBack : kOut;
  return a;
}

// Estimated microseconds of conv3x3_tile and of conv3x3_k32 (Cin = 16: conv3x3_mfma)
// on a shape that both sum by taps, to the same bits.  Both are a start-up and a
// time per round of resident workgroups, fitted to 430 shapes (N 1 to 65536, H and W
// 1 to 16384, 16 to 256 channels; most within 10 %, the worst 40 % off).  What decides:
// a tile works on whole 16 x 4 .. 16 x 16 pixels, whatever the image fills of them,
// and with 128 or 256 channels one workgroup has the CU to itself and restages its
// input for every 16 or 32 output channels; the others read every tap from the
// caches, a long chain that a few workgroups wait out.  Of the tile and the other kernel:
// 256 -> 256 8 x 16 x 8 9 and 42 us, 16 x 78 x 89 931 and 336, 65536 images of 1 x 1 27554
// and 127; 128 -> 128 12 x 48 x 134 122 and 65; 64 -> 64 6 x 73 x 40 7.5 and 16.3.
double conv_tile_us(const ConvArgs& a) {
  const ConvTile t = conv_tile(a);
  const double base = t.cp == 16 ? 0.3 : t.cp == 32 ? 0.6 : t.cp == 64 ? 0.5 : t.cp == 128 ? 3.3 : 6.0;
  const double slope = t.cp == 16 ? 0.105 : t.cp == 32 ? 0.125 : 0.265;
  const double slots = t.cp == 256 || (t.cp == 128 && t.tr * t.nb > 4) ? 256 : 512;
  return 3.5 + (base + slope * t.tr * t.nb) * std::max(1.0, conv_groups(a, t.tr, t.nb) / slots);
}

double conv_taps_us(const ConvArgs& a) {
  const ConvTaps t = conv_taps(a);
  const double rounds = std::max(1.0, t.groups / 512.0);
  if (a.Cin == 16) return 3 + t.nb + (0.5 + 0.75 * t.nb) * rounds;
  if (t.mb == 1) return 4 + a.Cin * (0.07 + (t.nb == 4 ? 0.11 : 0.09) * rounds);
  return 5 + a.Cin * (0.11 + (t.nb == 4 ? 0.145 : t.nb == 2 ? 0.105 : 0.08) * rounds);
}

// Whether the tile is the faster kernel for a convolution that conv_tiled takes (in
// doubt, within 5 %, the other one: tiny images are faster than its estimate).
bool conv_tile_pays(const ConvArgs& a) {
  return conv_by_chunks(a) || 1.05 * conv_tile_us(a) <= conv_taps_us(a);
}

template <int TR, int NB, int CP>
void launch_conv_tile(const ConvArgs& a, hipStream_t s) {
  const dim3 g((unsigned)(conv_groups(a, TR, NB) / (a.Cout / (16 * NB))), (unsigned)(a.Cout / (16 * NB)));
  if (a.flip) conv3x3_tile<TR, NB, CP, true><<<g, 256, 0, s>>>(a);
  else conv3x3_tile<TR, NB, CP, false><<<g, 256, 0, s>>>(a);
}

template <int CP>
void launch_conv(const ConvArgs& a, const ConvTile& t, hipStream_t s) {
  if (t.nb == 2 && t.tr == 8) launch_conv_tile<8, 2, CP>(a, s);
  else if (t.nb == 2) launch_conv_tile<4, 2, CP>(a, s);
  else if (CP == 128 && t.tr == 4) launch_conv_tile<4, 1, 128>(a, s);
  else launch_conv_tile<8, 1, CP>(a, s);
}

int launch_conv_tiled(const ConvArgs& a, hipStream_t s) {
  const ConvTile t = conv_tile(a);
  if (t.cp == 256) launch_conv_tile<4, 1, 256>(a, s);
  else if (t.cp == 128) launch_conv<128>(a, t, s);
  else if (t.cp == 64) launch_conv<64>(a, t, s);
  else if (t.cp == 16) launch_conv<16>(a, t, s);
  else if (t.nb == 4 && t.tr == 16) launch_conv_tile<16, 4, 32>(a, s);
  else if (t.nb == 4) launch_conv_tile<8, 4, 32>(a, s);
  else launch_conv<32>(a, t, s);
  return launch_check("conv3x3");
}

// Workgroups of a layer per range: blocks of 64 x 64 channels (many layers in one
// launch: 64 x 32) in the tile orders, of 32 x 32, or 16 where the count asks for it, in
// kLinear, where `split` workgroups share out the taps of a block.
int wgrad_blocks(const WgradArgs& a, bool many) {
  if (a.order != kLinear) return (a.Cin / 64) * (a.Cout / (many ? 32 : 64));
  return (a.Cin / (a.Cin % 32 == 0 ? 32 : 16)) * (a.Cout / (a.Cout % 32 == 0 ? 32 : 16)) * a.split;
}

// Whether wgrad_k32 sums a planned layer of order kLinear sooner than wgrad_linear, to
// the same bits: its workgroups take a tap and 64 x 64 channels, so where the
// channels fill them it stages less than 32 x 32 blocks that read all nine taps' pixels
// per block.  Both times as steps (of 32 and of 128 pixels) of a workgroup, over rounds of
// resident ones.  The factors are fitted to 770 calls: the chosen kernel is within 5 % of
// the faster one on nearly all, 14 % off on images of a few columns or 16 rows.  Of k32
// and linear: 64 -> 64 16 x 91 x 79 71 and 97 us, 256 -> 64 10 x 99 x 44 90 and 122, 96 -> 48 1 x 256 x 256 62 and 74;
// 16 -> 16 1 x 256 x 256 37 and 26, 256 -> 256 16 x 78 x 89 811 and 645.
bool wgrad_taps_pays(const WgradArgs& a) {
  const long taps = 9L * ((a.Cout + 63) / 64) * ((a.Cin + 63) / 64) * a.ranges;
  const long blocks = (long)wgrad_blocks(a, false) * a.ranges;
  const double k32 = 0.52 * ((a.per + 31) / 32) * std::max(1.0, taps / 1536.0);
  const double lin = (a.split == 3 ? 0.85 : 1.32) * ((a.per + 127) / 128) * std::max(1.0, blocks / 512.0);
  return k32 < lin;
}

// Blocks and pixels per block of the two-pass bias sum, whose partials may take cap
// rows of cout values.
long bias_blocks(long P, int cout, long cap, long* chunk) {
  *chunk = 256 / (cout < 256 ? cout : 256) * 64;  // 64 pixels per thread row
  long nb = (P + *chunk - 1) / *chunk;
  if (nb > cap) {
    *chunk = (P + cap - 1) / cap;
    nb = (P + *chunk - 1) / *chunk;
  }
  return nb;
}

// Order and ranges of a layer split over at most nsplit ranges of pixels: tiles for
// channels in multiples of 64 and whole tiles across, of 4 rows where the image is
// lower than 8.  Returns whether the bias is summed with the weights (the ranges
// then leave room after their partials for one row of cout values each).
bool wgrad_plan(WgradArgs& a, int nsplit, bool bias) {
  const long P = (long)a.N * a.H * a.W;
  a.split = 1;
  if (a.Cin % 64 || a.Cout % 64 || a.W % 16) {
    a.order = kLinear;
    a.ntiles = (int)P;
    a.per = (int)(((P + nsplit - 1) / nsplit + 15) / 16 * 16);
    a.ranges = (int)((P + a.per - 1) / a.per);
    return false;
  }
  a.order = a.H >= 8 ? kTile8 : kTile4;
  const int tr = a.H >= 8 ? 8 : 4;
  a.ntiles = (int)((long)a.N * (a.W / 16) * ((a.H + tr - 1) / tr));
  const bool fused = bias && nsplit >= 2 && nsplit - 1 <= 9 * a.Cin;
  const long nr = fused ? nsplit - 1 : nsplit;
  a.per = (int)((a.ntiles + nr - 1) / nr);
  a.ranges = (a.ntiles + a.per - 1) / a.per;
  return fused;
}

// Partials of planned layers, one launch per kind of order, then their sums in one.
// Base 32, 4 levels on 8 x 64 x 128: 44 + 60 us and 22 us of sums for the 18 layers,
// against 522 one layer at a time (two to four launches each; before kLinear read
// strips of pixels from LDS, one tap per workgroup, 585).
// db: bias gradients, of the layers with bpart.
template <int MAX>
int launch_wgrad(const WgradArgs* l, float* const* dW, float* const* db, int n, hipStream_t s) {
  WgradMany<MAX> m;
  ReduceMany<MAX> r;
  m.n = r.n = n;
  m.first[0] = r.first[0] = 0;
  for (int k = 0; k < n; k++) {
    const WgradArgs& a = m.l[k] = l[k];
    const long nw = 9L * a.Cout * a.Cin;
    const int nb = a.bpart ? a.Cout : 0, sums = a.bblocks ? (a.Cout + 63) / 64 : 0;
    r.first[k + 1] = r.first[k] + sums + (int)((nw + (sums ? 0 : nb) + 255) / 256);
    r.l[k] = {a.part, a.bpart, dW[k], db[k], nw, nb, a.ranges, a.bblocks, sums};
  }
  for (const int order : {kTile8, kTile4, kLinear}) {
    for (int k = 0; k < n; k++)
      m.first[k + 1] = m.first[k] + (l[k].order == order
                                         ? l[k].bblocks + l[k].ranges * wgrad_blocks(l[k], MAX > 1) : 0);
    if (!m.first[n]) continue;
    if (order == kLinear) wgrad_linear<MAX><<<m.first[n], 256, 0, s>>>(m);
    else if constexpr (MAX == 1) {
      const WgradArgs& a = l[0];
      const dim3 g((unsigned)a.ranges, (unsigned)wgrad_blocks(a, false));
      if (order == kTile8)
        wgrad_tr<8><<<g, 256, 0, s>>>(a.x, a.dz, a.part, a.bpart, a.N, a.H, a.W, a.Cin, a.Cout, a.per, a.ntiles);
      else
        wgrad_tr<4><<<g, 256, 0, s>>>(a.x, a.dz, a.part, a.bpart, a.N, a.H, a.W, a.Cin, a.Cout, a.per, a.ntiles);
    } else if (order == kTile8) wgrad_tiles<MAX, kTile8><<<m.first[n], 256, 0, s>>>(m);
    else wgrad_tiles<MAX, kTile4><<<m.first[n], 256, 0, s>>>(m);
    const int rc = launch_check("conv3x3_wgrad");
    if (rc) return rc;
  }
  wgrad_reduce<MAX><<<r.first[n], 256, 0, s>>>(r);
  return launch_check("wgrad_reduce");
}

}  // namespace
}  // namespace coffee

using namespace coffee;

extern "C" {

int coffee_unet_conv3x3(const void* in, const void* w, const float* bias, void* out, float* out32,
                        int n, int h, int wd, int cin, int cout, int flip, int relu, void* stream) {
  if (!in || !w || (!out && !out32) || n < 1 || h < 1 || wd < 1 || cin < 16 || cout < 16 ||
      cin % 16 || cout % 16)
    return fail(nullptr, COFFEE_ERR_INVALID, "conv3x3: bad arguments (channels must be multiples of 16)");
  ConvArgs a{};
  a.in = (const bf16*)in;
  a.w = (const bf16*)w;
  a.bias = bias;
  a.out = (bf16*)out;
  a.out32 = out32;
  a.N = n;
  a.H = h;
  a.W = wd;
  a.Cin = a.c1 = cin;
  a.Cout = a.csplit = cout;
  a.flip = flip;
  a.relu = relu;
  const hipStream_t s = (hipStream_t)stream;
  const long P = (long)n * h * wd;
  const long bx = (P + 63) / 64;
  if (bx > 2147483647L) return fail(nullptr, COFFEE_ERR_SIZE, "conv3x3: too many pixels");
  if (conv_tiled(a) && conv_tile_pays(a)) return launch_conv_tiled(a, s);
  if (cin % 32 == 0 && aligned16(in) && aligned16(w)) {
    const ConvTaps t = conv_taps(a);
    const long cb = cout / (16 * t.nb);
    const dim3 g((unsigned)(t.groups / cb), (unsigned)cb);
#define COFFEE_CONV32(NBV)                                              \
  do {                                                                  \
    if (t.mb == 2) conv3x3_k32<NBV, 2><<<g, 256, 0, s>>>(a);           \
    else conv3x3_k32<NBV, 1><<<g, 256, 0, s>>>(a);                     \
  } while (0)
    if (t.nb == 4) COFFEE_CONV32(4);
    else if (t.nb == 2) COFFEE_CONV32(2);
    else COFFEE_CONV32(1);
#undef COFFEE_CONV32
  } else if (cout % 64 == 0) {
    conv3x3_mfma<4><<<dim3((unsigned)bx, cout / 64), 256, 0, s>>>(a);
  } else if (cout % 32 == 0) {
    conv3x3_mfma<2><<<dim3((unsigned)bx, cout / 32), 256, 0, s>>>(a);
  } else {
    conv3x3_mfma<1><<<dim3((unsigned)bx, cout / 16), 256, 0, s>>>(a);
  }
  return launch_check("conv3x3");
}

int coffee_unet_conv3x3_fusable(int n, int h, int wd, int cin, int cout, int pairs) {
  if (n < 1 || h < 1 || wd < 1 || cin < 16 || cout < 16 || cin % 16 || cout % 16) return 0;
  const ConvArgs a = conv_sizes(n, h, wd, cin, cout, false);
  // all of 256 channels leave no room for tiles of 8 rows
  return conv_tiled(a) && (!pairs || conv_by_chunks(a) || cin != 256);
}

double coffee_unet_conv3x3_excess(int n, int h, int wd, int cin, int cout, int pairs) {
  if (!coffee_unet_conv3x3_fusable(n, h, wd, cin, cout, pairs)) return 0.0;
  const ConvArgs a = conv_sizes(n, h, wd, cin, cout, pairs != 0);
  return conv_by_chunks(a) ? 0.0 : std::max(0.0, conv_tile_us(a) - conv_taps_us(a));
}

int coffee_unet_conv3x3_fused(const coffee_unet_conv* c, void* stream) {
  if (!c || !c->in || !c->w || (!c->out && !c->out32) ||
      !coffee_unet_conv3x3_fusable(c->n, c->h, c->wd, c->cin, c->cout,
                                   c->form == kUpBack || c->pool != nullptr))
    return fail(nullptr, COFFEE_ERR_INVALID, "conv3x3_fused: bad arguments");
  const bool even = c->h % 2 == 0 && c->wd % 2 == 0;
  if (c->form < kOut || c->form > kUpBack || c->cin1 < 16 || c->cin1 % 16 || c->cin1 > c->cin ||
      (c->cin1 < c->cin && !c->in2) || ((c->up || c->form == kUpBack || c->pool) && !even) ||
      (c->form != kOut && (!c->out || c->out32 || c->pool)) ||
      (c->form == kMasked && (c->csplit < 16 || c->csplit % 16 || c->csplit > c->cout ||
                              (c->csplit < c->cout && !c->out2))))
    return fail(nullptr, COFFEE_ERR_INVALID, "conv3x3_fused: inconsistent forms");
  for (const void* p : {c->in, c->in2, c->w, (const void*)c->bias, (const void*)c->out,
                        (const void*)c->out2, (const void*)c->out32, c->mask, c->skip,
                        (const void*)c->pool})
    if (!aligned16(p)) return fail(nullptr, COFFEE_ERR_INVALID, "conv3x3_fused: 16-byte alignment required");
  ConvArgs a{};
  a.in = (const bf16*)c->in;
  a.in2 = (const bf16*)c->in2;
  a.c1 = c->cin1;
  a.up = c->up;
  a.w = (const bf16*)c->w;
  a.bias = c->bias;
  a.out = (bf16*)c->out;
  a.out2 = (bf16*)c->out2;
  a.out32 = c->out32;
  a.mask = (const bf16*)c->mask;
  a.skip = (const bf16*)c->skip;
  a.pool = (bf16*)c->pool;
  a.form = c->form;
  a.csplit = c->csplit;
  a.N = c->n;
  a.H = c->h;
  a.W = c->wd;
  a.Cin = c->cin;
  a.Cout = c->cout;
  a.flip = c->flip;
  a.relu = c->relu;
  return launch_conv_tiled(a, (hipStream_t)stream);
}

int coffee_unet_conv3x3_wgrad(const void* x, const void* dz, float* partial, int nsplit, float* dW,
                              float* db, int n, int h, int wd, int cin, int cout, void* stream) {
  if (!x || !dz || !partial || !dW || nsplit < 1 || cin % 16 || cout % 16 || cin < 16 || cout < 16)
    return fail(nullptr, COFFEE_ERR_INVALID, "conv3x3_wgrad: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  const long P = (long)n * h * wd;
  WgradArgs a{};
  a.x = (const bf16*)x;
  a.dz = (const bf16*)dz;
  a.N = n;
  a.H = h;
  a.W = wd;
  a.Cin = a.c1 = cin;
  a.Cout = cout;
  const long nw = 9L * cout * cin;
  const bool aligned = aligned16(x) && aligned16(dz);
  bool tiles = aligned && P < 2147483647L - 256, fused = false;
  if (tiles) {
    fused = wgrad_plan(a, nsplit, db != nullptr);
    // a third of the taps per workgroup, which then stages one strip of three, until
    // the chip is full several times over: 8 x 64 x 128, 32 -> 32 39.5 -> 30.9 us; 8 x 16
    // x 8, 256 -> 256 35.7 -> 27.0; 16 x 128 x 256, 32 -> 32 112 -> 82 (with the sums)
    if (a.order == kLinear && (long)a.ranges * wgrad_blocks(a, false) < 2048) a.split = 3;
    tiles = a.order != kLinear || !wgrad_taps_pays(a);
  }
  if (tiles) {
    a.part = partial;
    a.bpart = fused ? partial + a.ranges * nw : nullptr;
    const int rc = launch_wgrad<1>(&a, &dW, &db, 1, s);
    if (rc || !db || fused) return rc;
  } else {
    long chunk = (P + nsplit - 1) / nsplit;
    chunk = (chunk + 15) / 16 * 16;
    const int used = (int)((P + chunk - 1) / chunk);
    if (aligned)
      wgrad_k32<<<dim3(used, 9, ((cout + 63) / 64) * ((cin + 63) / 64)), 256, 0, s>>>(
          (const bf16*)x, (const bf16*)dz, partial, n, h, wd, cin, cout, chunk);
    else
      wgrad_mfma<<<dim3(used, 9, (cout / 16) * (cin / 16)), 64, 0, s>>>(
          (const bf16*)x, (const bf16*)dz, partial, n, h, wd, cin, cout, chunk);
    int rc = launch_check("conv3x3_wgrad");
    if (rc) return rc;
    ReduceMany<1> r;
    r.n = 1;
    r.first[0] = 0;
    r.first[1] = (int)((nw + 255) / 256);
    r.l[0] = {partial, nullptr, dW, nullptr, nw, 0, used, 0, 0};
    wgrad_reduce<1><<<r.first[1], 256, 0, s>>>(r);
    rc = launch_check("wgrad_reduce");
    if (rc || !db) return rc;
  }
  // the weight partials have been reduced: their buffer holds the bias partials
  long bchunk;
  const long nbb = bias_blocks(P, cout, (long)nsplit * 9 * cin, &bchunk);
  bias_grad_part<<<(unsigned)nbb, 256, 0, s>>>((const bf16*)dz, partial, P, cout, bchunk);
  int rc = launch_check("bias_grad_part");
  if (rc) return rc;
  bias_grad_sum<<<(cout + 63) / 64, 256, 0, s>>>(partial, db, (int)nbb, cout);
  return launch_check("bias_grad_sum");
}

int coffee_unet_wgrad_many(const coffee_unet_wgrad* l, int count, float* partial, long floats,
                           long* need, void* stream) {
  if (!l || count < 1 || (!partial && !need))
    return fail(nullptr, COFFEE_ERR_INVALID, "wgrad_many: bad arguments");
  std::vector<WgradArgs> a(count);
  std::vector<float*> dW(count), db(count);
  long used = 0;
  for (int k = 0; k < count; k++) {
    const coffee_unet_wgrad& q = l[k];
    if (!q.x || !q.dz || !q.dw || !q.db || q.n < 1 || q.h < 1 || q.wd < 1 || q.cin < 16 ||
        q.cout < 16 || q.cin % 16 || q.cout % 16 || q.cin1 < 16 || q.cin1 % 16 || q.cin1 > q.cin ||
        (q.cin1 < q.cin && !q.x2) || (q.up && (q.h % 2 || q.wd % 2)) || q.nsplit < 1 ||
        !aligned16(q.x) || !aligned16(q.x2) || !aligned16(q.dz))
      return fail(nullptr, COFFEE_ERR_INVALID, "wgrad_many: bad arguments of layer " + std::to_string(k));
    const long P = (long)q.n * q.h * q.wd, nw = 9L * q.cout * q.cin;
    if (P >= 2147483647L - 256) return fail(nullptr, COFFEE_ERR_SIZE, "wgrad_many: too many pixels");
    WgradArgs& w = a[k];
    w = WgradArgs{};
    w.x = (const bf16*)q.x;
    w.x2 = (const bf16*)q.x2;
    w.dz = (const bf16*)q.dz;
    w.N = q.n;
    w.H = q.h;
    w.W = q.wd;
    w.Cin = q.cin;
    w.Cout = q.cout;
    w.c1 = q.cin1;
    w.up = q.up;
    const bool fused = wgrad_plan(w, q.nsplit, true);
    if (!fused) {
      long chunk;
      w.bblocks = (int)bias_blocks(P, q.cout, (long)q.nsplit * 9 * q.cin, &chunk);
      w.bchunk = (int)chunk;
    }
    w.part = partial + used;
    w.bpart = w.part + w.ranges * nw;
    used += w.ranges * nw + (long)(fused ? w.ranges : w.bblocks) * q.cout;
    dW[k] = q.dw;
    db[k] = q.db;
  }
  if (need) *need = used;
  if (!partial) return COFFEE_OK;
  if (floats < used) return fail(nullptr, COFFEE_ERR_INVALID, "wgrad_many: workspace too small");
  for (int k = 0; k < count; k += kWgradLayers) {
    const int rc = launch_wgrad<kWgradLayers>(&a[k], &dW[k], &db[k], std::min(count - k, kWgradLayers),
                                              (hipStream_t)stream);
    if (rc) return rc;
  }
  return COFFEE_OK;
}

int coffee_unet_combine(void* out, int ost, int ooff, const void* a, int ast, int aoff,
                        const void* b, int bst, int boff, const void* mask, int mst, int moff,
                        int nc, long npix, void* stream) {
  if (!out || !a || nc < 1 || npix < 1 || ooff + nc > ost || aoff + nc > ast ||
      (b && boff + nc > bst) || (mask && moff + nc > mst))
    return fail(nullptr, COFFEE_ERR_INVALID, "combine: bad arguments");
  combine_kernel<<<grid_for(npix * nc), 256, 0, (hipStream_t)stream>>>(
      (bf16*)out, ost, ooff, (const bf16*)a, ast, aoff, (const bf16*)b, bst, boff,
      (const bf16*)mask, mst, moff, nc, npix);
  return launch_check("combine");
}

int coffee_unet_pool2(const void* in, void* out, int n, int h, int wd, int c, void* stream) {
  if (!in || !out || h % 2 || wd % 2) return fail(nullptr, COFFEE_ERR_INVALID, "pool2: even sizes required");
  pool2_kernel<<<grid_for((long)n * h * wd * c / 4), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)in, (bf16*)out, n, h, wd, c);
  return launch_check("pool2");
}

int coffee_unet_pool2_bwd(const void* dy, void* dx, int n, int h, int wd, int c, void* stream) {
  if (!dy || !dx || h % 2 || wd % 2) return fail(nullptr, COFFEE_ERR_INVALID, "pool2_bwd: even sizes required");
  pool2_bwd_kernel<<<grid_for((long)n * h * wd * c), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)dy, (bf16*)dx, n, h, wd, c);
  return launch_check("pool2_bwd");
}

int coffee_unet_up2(const void* in, void* out, int n, int h, int wd, int c, void* stream) {
  if (!in || !out || h % 2 || wd % 2) return fail(nullptr, COFFEE_ERR_INVALID, "up2: even sizes required");
  up2_kernel<<<grid_for((long)n * h * wd * c), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)in, (bf16*)out, n, h, wd, c);
  return launch_check("up2");
}

int coffee_unet_up2_bwd(const void* dy, void* dx, int n, int h, int wd, int c, void* stream) {
  if (!dy || !dx || h % 2 || wd % 2) return fail(nullptr, COFFEE_ERR_INVALID, "up2_bwd: even sizes required");
  up2_bwd_kernel<<<grid_for((long)n * h * wd * c / 4), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)dy, (bf16*)dx, n, h, wd, c);
  return launch_check("up2_bwd");
}

int coffee_unet_mse(const float* out32, int cst, const float* target, int nc, long npix,
                    void* dout, double* loss, void* stream) {
  if (!out32 || !target || !dout || !loss || nc < 1 || nc > cst)
    return fail(nullptr, COFFEE_ERR_INVALID, "mse: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  double* part = nullptr;
  if (hipMalloc(&part, sizeof(double) * kMseBlocks) != hipSuccess)
    return fail(nullptr, COFFEE_ERR_HIP, "mse: hipMalloc failed");
  mse_kernel<<<kMseBlocks, 256, 0, s>>>(out32, cst, target, nc, npix, (bf16*)dout, part);
  hipError_t e = hipGetLastError();
  double h[kMseBlocks];
  if (e == hipSuccess) e = hipMemcpyAsync(h, part, sizeof(h), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFree(part);
  if (e != hipSuccess) return fail(nullptr, COFFEE_ERR_HIP, std::string("mse: ") + hipGetErrorString(e));
  *loss = mse_sum(h, npix, nc);
  return COFFEE_OK;
}

int coffee_unet_mse_pinned(const float* out32, int cst, const float* target, int nc, long npix,
                           void* dout, double* work, double* loss, void* stream) {
  if (!out32 || !target || !dout || !work || !loss || nc < 1 || nc > cst || npix < 1)
    return fail(nullptr, COFFEE_ERR_INVALID, "mse_pinned: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  mse_kernel<<<kMseBlocks, 256, 0, s>>>(out32, cst, target, nc, npix, (bf16*)dout, work);
  int rc = launch_check("mse_pinned");
  if (rc) return rc;
  const hipError_t e = hipStreamSynchronize(s);
  if (e != hipSuccess) return fail(nullptr, COFFEE_ERR_HIP, std::string("mse_pinned: ") + hipGetErrorString(e));
  *loss = mse_sum(work, npix, nc);
  return COFFEE_OK;
}

int coffee_unet_adam(float* p, const float* g, float* m, float* v, long n, float lr, float beta1,
                     float beta2, float eps, int t, void* wb, void* wbt, int cout, int cin,
                     void* stream) {
  if (!p || !g || !m || !v || n < 1 || t < 1) return fail(nullptr, COFFEE_ERR_INVALID, "adam: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  const float c1 = 1.f - powf(beta1, (float)t), c2 = 1.f - powf(beta2, (float)t);
  adam_kernel<<<grid_for(n), 256, 0, s>>>(p, g, m, v, n, lr, beta1, beta2, eps, c1, c2);
  int rc = launch_check("adam");
  if (rc || !wb) return rc;
  if (!wbt || 9L * cout * cin != n) return fail(nullptr, COFFEE_ERR_INVALID, "adam: weight shape mismatch");
  weights_bf16_kernel<<<grid_for(n), 256, 0, s>>>(p, (bf16*)wb, (bf16*)wbt, cout, cin);
  return launch_check("weights_bf16");
}

int coffee_unet_adam_many(const coffee_unet_tensor* l, int count, float lr, float beta1, float beta2,
                          float eps, int t, void* stream) {
  if (!l || count < 1 || t < 1) return fail(nullptr, COFFEE_ERR_INVALID, "adam_many: bad arguments");
  for (int k = 0; k < count; k++)
    if (!l[k].p || !l[k].g || !l[k].m || !l[k].v || l[k].n < 1 ||
        (l[k].wb && (!l[k].wbt || l[k].cout < 1 || l[k].cin < 1 || 9L * l[k].cout * l[k].cin != l[k].n)))
      return fail(nullptr, COFFEE_ERR_INVALID, "adam_many: bad arguments of tensor " + std::to_string(k));
  AdamMany a;
  a.lr = lr;
  a.b1 = beta1;
  a.b2 = beta2;
  a.eps = eps;
  a.c1 = 1.f - powf(beta1, (float)t);
  a.c2 = 1.f - powf(beta2, (float)t);
  auto launch = [&]() -> int {
    if (!a.n) return COFFEE_OK;
    adam_many_kernel<<<a.first[a.n], 256, 0, (hipStream_t)stream>>>(a);
    a.n = 0;
    return launch_check("adam_many");
  };
  a.n = a.first[0] = 0;
  for (int k = 0; k < count; k++) {
    const coffee_unet_tensor& q = l[k];
    int rc = COFFEE_OK;
    if (q.n > 1L << 30) {  // beyond the 32-bit indices of the kernel for many
      rc = coffee_unet_adam(q.p, q.g, q.m, q.v, q.n, lr, beta1, beta2, eps, t, q.wb, q.wbt, q.cout, q.cin,
                            stream);
    } else {
      a.l[a.n] = {q.p, q.g, q.m, q.v, (bf16*)q.wb, (bf16*)q.wbt, (int)q.n, q.cout, q.cin};
      a.first[a.n + 1] = a.first[a.n] + (q.wb ? 9 * ((q.cout + 31) / 32) * ((q.cin + 31) / 32)
                                              : (int)((q.n + 1023) / 1024));
      if (++a.n == kAdamTensors) rc = launch();
    }
    if (rc) return rc;
  }
  return launch();
}

int coffee_unet_weights_bf16(const float* w32, void* wb, void* wbt, int cout, int cin, void* stream) {
  if (!w32 || !wb || !wbt) return fail(nullptr, COFFEE_ERR_INVALID, "weights_bf16: null argument");
  weights_bf16_kernel<<<grid_for(9L * cout * cin), 256, 0, (hipStream_t)stream>>>(
      w32, (bf16*)wb, (bf16*)wbt, cout, cin);
  return launch_check("weights_bf16");
}

int coffee_unet_to_bf16(const float* in, void* out, long n, void* stream) {
  if (!in || !out) return fail(nullptr, COFFEE_ERR_INVALID, "to_bf16: null argument");
  to_bf16_kernel<<<grid_for(n), 256, 0, (hipStream_t)stream>>>(in, (bf16*)out, n);
  return launch_check("to_bf16");
}

int coffee_unet_from_bf16(const void* in, float* out, long n, void* stream) {
  if (!in || !out) return fail(nullptr, COFFEE_ERR_INVALID, "from_bf16: null argument");
  from_bf16_kernel<<<grid_for(n), 256, 0, (hipStream_t)stream>>>((const bf16*)in, out, n);
  return launch_check("from_bf16");
}

int coffee_unet_pack(void* const fields[6], int scalar_bytes, int dims0, int g0, int g1, int n0,
                     int n1, double x0, double dx, double dy, double rpow, double extra_channel,
                     void* out, int out_fp32, int cst, int image, void* stream) {
  if (!fields || !out || cst < 6 || n0 < 1 || n1 < 1 || image < 0)
    return fail(nullptr, COFFEE_ERR_INVALID, "pack: bad arguments");
  for (int q = 0; q < 6; q++)
    if (!fields[q]) return fail(nullptr, COFFEE_ERR_INVALID, "pack: null field");
  const long base = (long)image * n0 * n1 * cst;
  const int blocks = grid_for((long)n0 * n1 * cst);
  hipStream_t s = (hipStream_t)stream;
  if (scalar_bytes == 4) {
    float* const* f = (float* const*)fields;
    pack_kernel<float><<<blocks, 256, 0, s>>>(f[0], f[1], f[2], f[3], f[4], f[5], dims0, g0, g1, n0,
                                              n1, x0, dx, dy, rpow, extra_channel, out, out_fp32,
                                              cst, base);
  } else {
    double* const* f = (double* const*)fields;
    pack_kernel<double><<<blocks, 256, 0, s>>>(f[0], f[1], f[2], f[3], f[4], f[5], dims0, g0, g1,
                                               n0, n1, x0, dx, dy, rpow, extra_channel, out,
                                               out_fp32, cst, base);
  }
  return launch_check("pack");
}

int coffee_unet_unpack(const float* in, int cst, int image, void* const fields[6], int scalar_bytes,
                       int dims0, int g0, int g1, int n0, int n1, double x0, double dx, double dy,
                       double rpow, void* stream) {
  if (!in || !fields || cst < 6 || n0 < 1 || n1 < 1 || image < 0)
    return fail(nullptr, COFFEE_ERR_INVALID, "unpack: bad arguments");
  for (int q = 0; q < 6; q++)
    if (!fields[q]) return fail(nullptr, COFFEE_ERR_INVALID, "unpack: null field");
  const long base = (long)image * n0 * n1 * cst;
  const int blocks = grid_for((long)n0 * n1 * 6);
  hipStream_t s = (hipStream_t)stream;
  if (scalar_bytes == 4) {
    float* const* f = (float* const*)fields;
    unpack_kernel<float><<<blocks, 256, 0, s>>>(in, cst, base, f[0], f[1], f[2], f[3], f[4], f[5],
                                                dims0, g0, g1, n0, n1, x0, dx, dy, rpow);
  } else {
    double* const* f = (double* const*)fields;
    unpack_kernel<double><<<blocks, 256, 0, s>>>(in, cst, base, f[0], f[1], f[2], f[3], f[4], f[5],
                                                 dims0, g0, g1, n0, n1, x0, dx, dy, rpow);
  }
  return launch_check("unpack");
}

int coffee_unet_corotate(void* const fields[6], int scalar_bytes, int dims0, int g0, int g1,
                         int n0, int n1, double x0, double dx, double dy, double omega,
                         void* stream) {
  if (!fields || n0 < 1 || n1 < 1 || dims0 < n0 + 2 * g0 || g0 < 0 || g1 < 0)
    return fail(nullptr, COFFEE_ERR_INVALID, "corotate: bad arguments");
  for (int q = 0; q < 5; q++)
    if (!fields[q]) return fail(nullptr, COFFEE_ERR_INVALID, "corotate: null field");
  const int blocks = grid_for((long)n0 * n1);
  hipStream_t s = (hipStream_t)stream;
  if (scalar_bytes == 4) {
    float* const* f = (float* const*)fields;
    corotate_kernel<float><<<blocks, 256, 0, s>>>(f[0], f[1], f[2], f[3], f[4], dims0, g0, g1, n0,
                                                  n1, x0, dx, dy, omega);
  } else if (scalar_bytes == 8) {
    double* const* f = (double* const*)fields;
    corotate_kernel<double><<<blocks, 256, 0, s>>>(f[0], f[1], f[2], f[3], f[4], dims0, g0, g1,
                                                   n0, n1, x0, dx, dy, omega);
  } else {
    return fail(nullptr, COFFEE_ERR_INVALID, "corotate: scalar_bytes must be 4 or 8");
  }
  return launch_check("corotate");
}

}  // extern "C"
