// Kernels of the learned initialiser: a 3D U-Net whose convolutions run on
// gfx950's BF16 matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulate).
//
// The reference has no counterpart: its stage 0 starts from zero
// (XT_ICD_update.c:549-553) and its initICD = 1 path reads an object from a
// file without interpolation (XT_ICD_update.c:558-571).  The network's output
// enters the ICD stage the same way, as the stage's starting object.
//
// Layouts.  Activations and their gradients are bf16, channels last:
// [N][D][H][W][C] with C a multiple of 32.  Convolution weights are bf16
// [27][Cout][Cin] (tap = (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1)), so one
// lane's eight consecutive input channels are one 16-byte load.  Biases,
// master weights, optimiser state and weight gradients are fp32.  Every
// 3x3x3 convolution pads with zeros ("same" size).
//
// Matrix-core lane layout of v_mfma_f32_16x16x32_bf16 (64 lanes, l = lane):
//   A (16 x 32, M x K): lane l holds A[l % 16][8 (l / 16) + i], i = 0..7
//   B (32 x 16, K x N): lane l holds B[8 (l / 16) + i][l % 16]
//   D (16 x 16):        lane l holds D[4 (l / 16) + j][l % 16], j = 0..3
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "timbir_dev.h"

namespace tbnn {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTaps = 27;
constexpr int kWavesPerBlock = 4;

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; i++) z[i] = (bf16)0.0f;
  return z;
}

// ---------------------------------------------------------------------------
// 3x3x3 convolution, forward: out[v][co] = bias[co] + sum_tap sum_ci
// in[v + off(tap)][ci] w[tap][co][ci], then ReLU when relu != 0.  A wave owns
// 16 MB voxels of one (n, d, h) row and 16 NB output channels; its K loop runs
// over the 27 taps and the input channels in chunks of 32.  Taps whose
// (d, h) neighbour row lies outside the volume are skipped (uniform over the
// wave); voxels whose x neighbour lies outside read zeros.  CAT: the first Ca
// input channels are those of `ina`, of half the size, nearest x2 upsampled.
// ---------------------------------------------------------------------------
template <int MB, int NB, bool CAT>
__device__ __forceinline__ void conv_strip(const bf16 *__restrict__ ina, int Ca,
                                           const bf16 *__restrict__ in,
                                           const bf16 *__restrict__ w,
                                           const float *__restrict__ bias, void *__restrict__ out,
                                           int D, int H, int W, int Cin, int Cout, int relu,
                                           int out_f32, int n, int d, int h, int w0, int co0) {
  const int lane = threadIdx.x & 63;
  const int row = lane & 15, kq = lane >> 4;
  const int Cb = CAT ? Cin - Ca : Cin;  // channels of `in`
  f32x4 acc[MB][NB];
#pragma unroll
  for (int a = 0; a < MB; a++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nchunk = Cin / 32;
  for (int tap = 0; tap < kTaps; tap++) {
    const int zz = d + tap / 9 - 1, yy = h + (tap / 3) % 3 - 1, dx = tap % 3 - 1;
    if (zz < 0 || zz >= D || yy < 0 || yy >= H) continue;
    const bf16 *inrow = in + (((size_t)n * D + zz) * H + yy) * (size_t)W * Cb;
    const bf16 *wt_tap = w + (size_t)tap * Cout * Cin;
    for (int c = 0; c < nchunk; c++) {
      const bf16 *src = inrow + c * 32;
      int ch = Cb, sh = 0;
      if constexpr (CAT) {
        if (c * 32 < Ca) {
          src = ina + (((size_t)n * (D / 2) + zz / 2) * (H / 2) + yy / 2) * (size_t)(W / 2) * Ca +
                c * 32;
          ch = Ca;
          sh = 1;
        } else {
          src -= Ca;
        }
      }
      bf16x8 av[MB], bv[NB];
#pragma unroll
      for (int a = 0; a < MB; a++) {
        const int xx = w0 + 16 * a + row + dx;
        av[a] = (xx >= 0 && xx < W)
                    ? *reinterpret_cast<const bf16x8 *>(src + (size_t)(xx >> sh) * ch + kq * 8)
                    : zero8();
      }
#pragma unroll
      for (int b = 0; b < NB; b++)
        bv[b] = *reinterpret_cast<const bf16x8 *>(wt_tap + (size_t)(co0 + 16 * b + row) * Cin +
                                                  c * 32 + kq * 8);
#pragma unroll
      for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[a][b] = mfma(av[a], bv[b], acc[a][b]);
    }
  }
  const size_t orow = (((size_t)n * D + d) * H + h) * (size_t)W;
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int co = co0 + 16 * b + row;
    const float bb = bias ? bias[co] : 0.f;
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int x = w0 + 16 * a + 4 * kq + j;
        if (x >= W) continue;
        float v = acc[a][b][j] + bb;
        if (relu) v = fmaxf(v, 0.f);
        const size_t o = (orow + x) * Cout + co;
        if (out_f32) static_cast<float *>(out)[o] = v;
        else static_cast<bf16 *>(out)[o] = (bf16)v;
      }
  }
}

template <int MB, int NB>
__global__ __launch_bounds__(64 * kWavesPerBlock) void k_conv3d_fwd(
    const bf16 *__restrict__ in, const bf16 *__restrict__ w, const float *__restrict__ bias,
    void *__restrict__ out, int N, int D, int H, int W, int Cin, int Cout, int relu,
    int out_f32) {
  const long long g = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  const int WT = (W + 16 * MB - 1) / (16 * MB);
  const int CT = Cout / (16 * NB);
  const long long total = (long long)N * D * H * WT * CT;
  if (g >= total) return;
  long long r = g;
  const int ct = (int)(r % CT); r /= CT;
  const int wt = (int)(r % WT); r /= WT;
  const int h = (int)(r % H); r /= H;
  const int d = (int)(r % D);
  const int n = (int)(r / D);
  conv_strip<MB, NB, false>(nullptr, 0, in, w, bias, out, D, H, W, Cin, Cout, relu, out_f32, n, d,
                            h, wt * 16 * MB, ct * 16 * NB);
}

// The same convolution with the input staged in LDS.  The input's channels are
// 32 CA of a tensor at half size, nearest x2 upsampled (`ina`, CA may be 0),
// then 32 CB of one at full size (`in`): the concatenation of a U-Net's skip
// connection need not exist in memory.  Tile: 64 SP voxels per wave as strips
// of WT x (64 / WT), 4 waves side by side in h, 16 NB output channels.  One
// input plane (dz) at a time is staged with its halo, in the order of the taps,
// and each of its values serves 9 taps from LDS; without it every tap read
// every value through the L1 (192 B a cycle wanted, 64 there).
//   Weights are the A operand (M = output channel; row m of fragment b is
// channel (m / 4) 4 NB + 4 b + m % 4, so a lane ends with 4 NB consecutive
// channels of a voxel and stores them whole), activations the B operand (N =
// voxel).  Fragment a holds the voxels x = 4 q + a, so the three x taps of four
// fragments are six reads instead of twelve, and four of the half-size tensor
// (a voxel's parent is x / 2); LDS keeps x modulo 4 (parents modulo 2) apart,
// which makes each read one contiguous KB.
//   The sums run over (tap, channel chunk) as in k_conv3d_fwd, one MFMA each:
// the bits are the same.  Rows above and below the volume are zeros in LDS; a
// weight that is infinite or NaN makes those NaN, so a wave that finds such a
// sum in the volume's first or last row takes conv_strip for its strips, which
// leaves those taps out.
//   What bounds it: staging and sums take turns behind barriers with two or three
// waves a SIMD; matrix cores, other vector instructions and LDS are each busy for
// less than a third of the cycles.  2 x 16 x 256 x 256 voxels, before and now: 32
// -> 32 channels 0.38 and 0.19 ms (600 TFLOP/s); 64 + 32 -> 32 with its
// concatenation 1.6 and 0.47 ms (710 TFLOP/s).
template <int CA, int CB, int SP, int WT>
struct ConvTile {
  static constexpr int RPS = 64 / WT, HT = 4 * SP * RPS;
  static constexpr int HR = HT + 2, QW = WT / 4 + 1;  // full size: s[CB][HR][4][QW][32]
  static constexpr int HC = HT / 2 + 2;               // half size: s[CA][HC][2][QW][32]
  static constexpr int kFull = CB * HR * 4 * QW * 32, kHalf = CA * HC * 2 * QW * 32;
  static constexpr size_t kBytes = (size_t)(kFull + kHalf) * sizeof(bf16);
};

template <int CA, int CB, int NB, int SP, int WT>
__global__ __launch_bounds__(256) void k_conv3d_tile(
    const bf16 *__restrict__ ina, const bf16 *__restrict__ in, const bf16 *__restrict__ w,
    const float *__restrict__ bias, void *__restrict__ out, int N, int D, int H, int W, int Cout,
    int relu, int out_f32) {
  using T = ConvTile<CA, CB, SP, WT>;
  constexpr int C = CA + CB, Cin = 32 * C, RPS = T::RPS, HT = T::HT, HR = T::HR, HC = T::HC,
                QW = T::QW;
  constexpr bool HOLD = C <= 3;  // a row's fragments of every chunk fit the registers
  extern __shared__ bf16 s_in[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & 15, kq = lane >> 4;
  const int WB = (W + WT - 1) / WT, HB = (H + HT - 1) / HT, CT = Cout / (16 * NB);
  // neighbouring tiles on one XCD (block b runs on XCD b mod 8): they share halos
  unsigned g = blockIdx.x;
  if ((gridDim.x & 7) == 0) g = (g & 7) * (gridDim.x >> 3) + (g >> 3);
  const int ct = g % CT; g /= CT;
  const int w0 = (int)(g % WB) * WT; g /= WB;
  const int h0 = (int)(g % HB) * HT; g /= HB;
  const int d = g % D, n = g / D;
  const int co0 = ct * 16 * NB;
  const int hw = h0 + __builtin_amdgcn_readfirstlane(wave) * SP * RPS;  // the wave's first row
  const int xq = row % (WT / 4), yr = row / (WT / 4);
  f32x4 acc[SP][4][NB];
#pragma unroll
  for (int s = 0; s < SP; s++)
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < NB; b++) acc[s][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16 *wl = w + (size_t)(co0 + (row >> 2) * 4 * NB + (row & 3)) * Cin + kq * 8;
  int held = -1;  // the half-size plane in LDS
  for (int dz = 0; dz < 3; dz++) {
    const int zz = d + dz - 1;
    if (zz < 0 || zz >= D) continue;
    __syncthreads();
    if constexpr (CB > 0) {
      const bf16 *plane = in + ((size_t)n * D + zz) * H * W * (32 * CB);
#pragma unroll 4
      for (int i = threadIdx.x; i < HR * (WT + 2) * 4 * CB; i += 256) {
        const int part = i % (4 * CB), vox = i / (4 * CB), xi = vox % (WT + 2), y = vox / (WT + 2);
        const int yy = h0 + y - 1, xx = w0 + xi - 1;
        bf16x8 v = zero8();
        if (yy >= 0 && yy < H && xx >= 0 && xx < W)
          v = *reinterpret_cast<const bf16x8 *>(plane + ((size_t)yy * W + xx) * (32 * CB) + part * 8);
        *reinterpret_cast<bf16x8 *>(
            s_in + ((((part >> 2) * HR + y) * 4 + (xi & 3)) * QW + (xi >> 2)) * 32 + (part & 3) * 8) =
            v;
      }
    }
    if constexpr (CA > 0) {
      const int H2 = H / 2, W2 = W / 2;
      if (held != (zz >> 1)) {
        held = zz >> 1;
        const bf16 *plane = ina + ((size_t)n * (D / 2) + held) * H2 * W2 * (32 * CA);
#pragma unroll 4
        for (int i = threadIdx.x; i < HC * (WT / 2 + 2) * 4 * CA; i += 256) {
          const int part = i % (4 * CA), vox = i / (4 * CA);
          const int xi = vox % (WT / 2 + 2), y = vox / (WT / 2 + 2);
          const int yy = h0 / 2 + y - 1, xx = w0 / 2 + xi - 1;
          bf16x8 v = zero8();
          if (yy >= 0 && yy < H2 && xx >= 0 && xx < W2)
            v = *reinterpret_cast<const bf16x8 *>(plane + ((size_t)yy * W2 + xx) * (32 * CA) +
                                                  part * 8);
          *reinterpret_cast<bf16x8 *>(s_in + T::kFull +
                                      ((((part >> 2) * HC + y) * 2 + (xi & 1)) * QW + (xi >> 1)) * 32 +
                                      (part & 3) * 8) = v;
        }
      }
    }
    __syncthreads();
    // a wave past a volume of fewer rows than a tile (not of a last tile alone: its
    // waves' early end costs the tall volumes' launches more than it saves, 64 -> 64
    // channels of 16 planes of 114 x 106 144 us with it and 136 without)
    if (h0 == 0 && hw >= H) continue;
#pragma unroll 1
    for (int dy = 0; dy < 3; dy++) {
      const bf16 *wt = wl + (size_t)(dz * 9 + dy * 3) * Cout * Cin;
      // voxels 4 q + t - 1 of chunk c, t = 0 .. 5; of the half-size tensor
      // their parents 2 q + u - 1, u = (t + 1) / 2
      auto frag = [&](int s, int c, int t) -> bf16x8 {
        const int y = (wave * SP + s) * RPS + yr + dy;
        const bf16 *p;
        if (c < CA) {
          const int u = (t + 1) >> 1;
          p = s_in + T::kFull + (((c * HC + ((y + 1) >> 1)) * 2 + (u & 1)) * QW + xq + (u >> 1)) * 32;
        } else {
          p = s_in + ((((c - CA) * HR + y) * 4 + (t & 3)) * QW + xq + (t >> 2)) * 32;
        }
        return *reinterpret_cast<const bf16x8 *>(p + kq * 8);
      };
      bf16x8 fr[SP][HOLD ? C : 1][6];
      if constexpr (HOLD) {
#pragma unroll
        for (int s = 0; s < SP; s++)
#pragma unroll
          for (int c = 0; c < C; c++)
#pragma unroll
            for (int t = 0; t < 6; t++)
              fr[s][c][t] = c < CA && t > 0 && (t & 1) == 0 ? fr[s][c][t - 1] : frag(s, c, t);
      }
#pragma unroll
      for (int dx = 0; dx < 3; dx++)
#pragma unroll
        for (int c = 0; c < C; c++) {
          bf16x8 wv[NB];
#pragma unroll
          for (int b = 0; b < NB; b++)
            wv[b] = *reinterpret_cast<const bf16x8 *>(wt + (size_t)dx * Cout * Cin +
                                                      (size_t)b * 4 * Cin + c * 32);
#pragma unroll
          for (int s = 0; s < SP; s++) {
            bf16x8 x[4];
#pragma unroll
            for (int a = 0; a < 4; a++)
              x[a] = HOLD ? fr[s][HOLD ? c : 0][a + dx]
                     : c < CA && a > 0 && ((a + dx) & 1) == 0 ? x[a - 1]
                                                              : frag(s, c, a + dx);
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
              for (int b = 0; b < NB; b++) acc[s][a][b] = mfma(wv[b], x[a], acc[s][a][b]);
          }
        }
    }
  }
  if (hw == 0 || hw + SP * RPS >= H) {
    bool bad = false;
#pragma unroll
    for (int s = 0; s < SP; s++) {
      const int h = hw + s * RPS + yr;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const bool in_edge = (h == 0 || h == H - 1) && w0 + 4 * xq + a < W;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int k = 0; k < 4; k++) bad |= in_edge & !(fabsf(acc[s][a][b][k]) < INFINITY);
      }
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0ull, 0)) {
#pragma unroll 1
      for (int i = 0; i < SP * RPS * (WT / 16) * NB; i++) {
        const int h = hw + i / (WT / 16 * NB), x = w0 + i / NB % (WT / 16) * 16;
        if (h < H && x < W)
          conv_strip<1, 1, (CA > 0)>(ina, 32 * CA, in, w, bias, out, D, H, W, Cin, Cout, relu,
                                     out_f32, n, d, h, x, co0 + i % NB * 16);
      }
      return;
    }
  }
  // lane: channels co .. co + 4 NB - 1 of voxel x = w0 + 4 xq + a
  const int co = co0 + kq * 4 * NB;
  float bb[4 * NB];
#pragma unroll
  for (int k = 0; k < 4 * NB; k++) bb[k] = bias ? bias[co + k] : 0.f;
#pragma unroll
  for (int s = 0; s < SP; s++) {
    const int h = h0 + (wave * SP + s) * RPS + yr;
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const int x = w0 + 4 * xq + a;
      if (h >= H || x >= W) continue;
      const size_t o = ((((size_t)n * D + d) * H + h) * W + x) * Cout + co;
#pragma unroll
      for (int b = 0; b < NB; b += 2) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
          v[k] = acc[s][a][b + k / 4][k % 4] + bb[4 * b + k];
          if (relu) v[k] = fmaxf(v[k], 0.f);
        }
        if (out_f32) {
          float4 *p = reinterpret_cast<float4 *>(static_cast<float *>(out) + o + 4 * b);
          p[0] = make_float4(v[0], v[1], v[2], v[3]);
          p[1] = make_float4(v[4], v[5], v[6], v[7]);
        } else {
          bf16x8 q;
#pragma unroll
          for (int k = 0; k < 8; k++) q[k] = (bf16)v[k];
          *reinterpret_cast<bf16x8 *>(static_cast<bf16 *>(out) + o + 4 * b) = q;
        }
      }
    }
  }
}

// wt[t][ci][co] = w[26 - t][co][ci]: the weights of the gradient with respect
// to the input, which is the forward convolution of the output gradient with
// the spatially flipped, transposed kernel
__global__ void k_conv_flip(const bf16 *__restrict__ w, bf16 *__restrict__ wt, int Cin, int Cout) {
  const size_t n = (size_t)kTaps * Cin * Cout;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const int co = (int)(i % Cout);
    const int ci = (int)((i / Cout) % Cin);
    const int t = (int)(i / ((size_t)Cout * Cin));
    wt[i] = w[((size_t)(kTaps - 1 - t) * Cout + co) * Cin + ci];
  }
}

// ---------------------------------------------------------------------------
// 3x3x3 convolution, weight gradient: gw[tap][co][ci] = sum_v gout[v][co]
// in[v + off(tap)][ci].  M = co, N = ci, K = 32 voxels of a row.
//   A block takes 32 output and 32 input channels and walks units of kGH x 32
// pixels by a run of planes: LDS holds three planes of the input (with a halo
// pixel) and one of the output gradient, so every value read from memory
// serves its 27 taps; the next planes are in registers while one is computed.
// Channels are the contiguous axis in memory but the matrix cores want the
// voxels of K in a lane: ds_read_b64_tr_b16 transposes 4 voxels x 16 channels
// on the way from LDS.  K index 8 kq + i is the voxel x = 4 kq + i % 4 + 16 (i
// / 4) of the row in both operands, which makes each such read 512 contiguous
// bytes.
//   Wave (dz, co half, row group): 9 taps x (16 x 32) channels of sums; it
// walks the input rows, holding the gradient rows of the three y taps, so a
// row costs 7 fragments for 18 MFMAs (97 B a cycle of LDS per CU at the matrix
// cores' rate).  The two row groups are added at the end, the slices by
// k_sum_parts: the order is fixed.  Reading 2 bytes per lane and load from
// global memory, one tap at a time, took 654 us on average over the layers of
// a training step on 4 x 8 x 128 x 128 voxels, in this form 45 (580 TFLOP/s).
// ---------------------------------------------------------------------------
constexpr int kGH = 16, kGW = 32, kGThreads = 768;
typedef short s16x4 __attribute__((ext_vector_type(4)));

struct WgradUnits {
  int hb, wb, zc, per, units;  // tiles in h and w, runs of `per` planes, units in all
};

template <bool VEC>
__device__ __forceinline__ bf16x8 load8(const bf16 *p) {
  if constexpr (VEC) return *reinterpret_cast<const bf16x8 *>(p);
  bf16x8 v;
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = p[i];
  return v;
}

// 8 values of K for this lane's column from 16 channels at p (voxel x = 0,
// channel 0 of the 16): rows x = 4 kq .. + 3 and 16 further
__device__ __forceinline__ bf16x8 tr_frag(const bf16 *p, int lane) {
  const bf16 *q = p + (4 * (lane >> 4) + ((lane & 15) >> 2)) * 16 + (lane & 3) * 4;
  typedef __attribute__((address_space(3))) s16x4 *lds4;
  union {
    s16x4 h[2];
    bf16x8 v;
  } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)q);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(q + 16 * 16));
  return u.v;
}

template <bool VEC>
__global__ __launch_bounds__(kGThreads) void k_conv3d_wgrad(
    const bf16 *__restrict__ in, const bf16 *__restrict__ gout, float *__restrict__ part, int N,
    int D, int H, int W, int Cin, int Cout, int S, WgradUnits U) {
  constexpr int HR = kGH + 2, WR = kGW + 2;
  constexpr int kIn = 2 * HR * WR * 16, kOut = 2 * kGH * kGW * 16;  // bf16 of a plane
  constexpr int NI = (HR * WR * 4 + kGThreads - 1) / kGThreads;
  constexpr int NO = (kGH * kGW * 4 + kGThreads - 1) / kGThreads;
  extern __shared__ bf16 s_w[];  // input planes [3][2][HR][WR][16], gradient [2][kGH][kGW][16]
  bf16 *s_g = s_w + 3 * kIn;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int dz = wave % 3, half = (wave / 3) & 1, rg = wave / 6;
  const int IT = Cin / 32, OT = Cout / 32;
  const int s = blockIdx.x / (IT * OT), io = blockIdx.x - s * (IT * OT);
  const int ci0 = io % IT * 32, co0 = io / IT * 32;
  f32x4 acc[9][2];
#pragma unroll
  for (int t = 0; t < 9; t++) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int u = s; u < U.units; u += S) {
    int q = u;
    const int zi = q % U.zc; q /= U.zc;
    const int w0 = q % U.wb * kGW; q /= U.wb;
    const int h0 = q % U.hb * kGH, n = q / U.hb;
    const int za = zi * U.per, zb = min(za + U.per, D);
    // plane z of the input (out of range: zeros) and of the gradient
    auto fetch_in = [&](int z, bf16x8 (&r)[NI]) {
      const bf16 *plane = in + ((size_t)n * D + max(z, 0)) * H * W * Cin + ci0;
#pragma unroll
      for (int k = 0; k < NI; k++) {
        const int i = threadIdx.x + k * kGThreads, vox = i >> 2;
        const int yy = h0 + vox / WR - 1, xx = w0 + vox % WR - 1;
        r[k] = zero8();
        if (i < HR * WR * 4 && z >= 0 && z < D && yy >= 0 && yy < H && xx >= 0 && xx < W)
          r[k] = load8<VEC>(plane + ((size_t)yy * W + xx) * Cin + (i & 3) * 8);
      }
    };
    auto fetch_out = [&](int z, bf16x8 (&r)[NO]) {
      const bf16 *plane = gout + ((size_t)n * D + z) * H * W * Cout + co0;
#pragma unroll
      for (int k = 0; k < NO; k++) {
        const int i = threadIdx.x + k * kGThreads, vox = i >> 2;
        const int yy = h0 + vox / kGW, xx = w0 + vox % kGW;
        r[k] = zero8();
        if (i < kGH * kGW * 4 && z < zb && yy < H && xx < W)
          r[k] = load8<VEC>(plane + ((size_t)yy * W + xx) * Cout + (i & 3) * 8);
      }
    };
    auto put_in = [&](int z, const bf16x8 (&r)[NI]) {
      bf16 *slot = s_w + (z + 1) % 3 * kIn;
#pragma unroll
      for (int k = 0; k < NI; k++) {
        const int i = threadIdx.x + k * kGThreads, vox = i >> 2;
        if (i < HR * WR * 4)
          *reinterpret_cast<bf16x8 *>(slot + (((i >> 1) & 1) * HR * WR + vox) * 16 + (i & 1) * 8) =
              r[k];
      }
    };
    auto put_out = [&](const bf16x8 (&r)[NO]) {
#pragma unroll
      for (int k = 0; k < NO; k++) {
        const int i = threadIdx.x + k * kGThreads, vox = i >> 2;
        if (i < kGH * kGW * 4)
          *reinterpret_cast<bf16x8 *>(s_g + (((i >> 1) & 1) * kGH * kGW + vox) * 16 + (i & 1) * 8) =
              r[k];
      }
    };
    bf16x8 ri[NI], ro[NO];
    __syncthreads();  // the unit before is done with LDS
    fetch_in(za - 1, ri);
    put_in(za - 1, ri);
    fetch_in(za, ri);
    put_in(za, ri);
    fetch_in(za + 1, ri);
    fetch_out(za, ro);
    for (int z = za; z < zb; z++) {
      if (z > za) __syncthreads();  // plane z - 1 is done
      put_in(z + 1, ri);
      put_out(ro);
      __syncthreads();
      if (z + 1 < zb) {
        fetch_in(z + 2, ri);
        fetch_out(z + 1, ro);
      }
      // input row y (0 .. HR - 1 of the tile) meets gradient row y - dy, dy = 0 .. 2
      const bf16 *pi = s_w + (z + dz) % 3 * kIn;
      const bf16 *pg = s_g + half * kGH * kGW * 16;
      constexpr int RR = kGH / 2;
      const int r0 = rg * RR;
      bf16x8 ga[3];
#pragma unroll
      for (int y = 0; y < RR + 2; y++) {
        if (y < RR) ga[y % 3] = tr_frag(pg + (r0 + y) * kGW * 16, lane);
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int f = 0; f < 2; f++) {
            const bf16x8 x = tr_frag(pi + ((f * HR + r0 + y) * WR + dx) * 16, lane);
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
              if (y - dy >= 0 && y - dy < RR)
                acc[dy * 3 + dx][f] = mfma(ga[(y - dy) % 3], x, acc[dy * 3 + dx][f]);
          }
      }
    }
  }
  // the second row group's sums join the first's through LDS
  __syncthreads();
  f32x4 *sh = reinterpret_cast<f32x4 *>(s_w) + (size_t)(wave % 6) * 18 * 64 + lane;
  if (rg == 1) {
#pragma unroll
    for (int t = 0; t < 18; t++) sh[t * 64] = acc[t / 2][t % 2];
  }
  __syncthreads();
  if (rg == 0) {
    float *dst = part + ((size_t)s * kTaps + dz * 9) * Cout * Cin;
#pragma unroll
    for (int t = 0; t < 18; t++) {
      const f32x4 v = acc[t / 2][t % 2] + sh[t * 64];
#pragma unroll
      for (int j = 0; j < 4; j++)
        dst[((size_t)(t / 2) * Cout + co0 + 16 * half + 4 * (lane >> 4) + j) * Cin + ci0 +
            16 * (t % 2) + (lane & 15)] = v[j];
    }
  }
}

// The same for volumes whose tiles would be mostly empty (short rows, few of
// them): a wave owns one tap, 16 MBO output and 16 NBI input channels and one of S
// slices of the voxels in their order, 32 at a time, whatever row they lie in; its
// sums go to part[s][tap][co][ci].
template <int MBO, int NBI>
__global__ __launch_bounds__(64 * kWavesPerBlock) void k_conv3d_wgrad_flat(
    const bf16 *__restrict__ in, const bf16 *__restrict__ gout, float *__restrict__ part,
    int N, int D, int H, int W, int Cin, int Cout, int S) {
  const int lane = threadIdx.x & 63;
  const long long g = (long long)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  const int OT = Cout / (16 * MBO), IT = Cin / (16 * NBI);
  const long long total = (long long)S * kTaps * OT * IT;
  if (g >= total) return;
  long long r = g;
  const int it = (int)(r % IT); r /= IT;
  const int ot = (int)(r % OT); r /= OT;
  const int tap = (int)(r % kTaps);
  const int s = (int)(r / kTaps);
  const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
  const int row = lane & 15, kq = lane >> 4;
  const int co0 = ot * 16 * MBO, ci0 = it * 16 * NBI;
  const long long nvox = (long long)N * D * H * W;
  const long long nch = (nvox + 31) / 32;
  const long long c_begin = nch * s / S, c_end = nch * (s + 1) / S;
  f32x4 acc[MBO][NBI];
#pragma unroll
  for (int a = 0; a < MBO; a++)
#pragma unroll
    for (int b = 0; b < NBI; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (long long c = c_begin; c < c_end; c++) {
    bf16x8 av[MBO], bv[NBI];
#pragma unroll
    for (int a = 0; a < MBO; a++) av[a] = zero8();
#pragma unroll
    for (int b = 0; b < NBI; b++) bv[b] = zero8();
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const long long v = c * 32 + kq * 8 + i;
      if (v >= nvox) break;
      long long q = v;
      const int x = (int)(q % W); q /= W;
      const int y = (int)(q % H); q /= H;
      const int z = (int)(q % D);
      const int nn = (int)(q / D);
#pragma unroll
      for (int a = 0; a < MBO; a++) av[a][i] = gout[(size_t)v * Cout + co0 + 16 * a + row];
      const int zz = z + dz, yy = y + dy, xx = x + dx;
      if (zz >= 0 && zz < D && yy >= 0 && yy < H && xx >= 0 && xx < W) {
        const size_t u = (((size_t)nn * D + zz) * H + yy) * (size_t)W + xx;
#pragma unroll
        for (int b = 0; b < NBI; b++) bv[b][i] = in[u * Cin + ci0 + 16 * b + row];
      }
    }
#pragma unroll
    for (int a = 0; a < MBO; a++)
#pragma unroll
      for (int b = 0; b < NBI; b++) acc[a][b] = mfma(av[a], bv[b], acc[a][b]);
  }
  float *dst = part + ((size_t)s * kTaps + tap) * Cout * Cin;
#pragma unroll
  for (int a = 0; a < MBO; a++)
#pragma unroll
    for (int b = 0; b < NBI; b++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        dst[(size_t)(co0 + 16 * a + 4 * kq + j) * Cin + ci0 + 16 * b + row] = acc[a][b][j];
}

// out[i] = sum_s part[s][i]: RUNS runs of slices side by side, each in order with
// eight loads in flight, then the runs in order.  Block: E entries.
template <int RUNS, int E>
__global__ __launch_bounds__(E *RUNS) void k_sum_parts(const float *__restrict__ part,
                                                       float *__restrict__ out, size_t n, int S) {
  __shared__ float sh[RUNS][E];
  const int col = threadIdx.x % E, run = threadIdx.x / E;
  const int per = (S + RUNS - 1) / RUNS;
  const int s0 = min(run * per, S), s1 = min(s0 + per, S);
  for (size_t i0 = blockIdx.x * (size_t)E; i0 < n; i0 += (size_t)gridDim.x * E) {
    const size_t i = i0 + col;
    float acc = 0.f;
    if (i < n) {
      int s = s0;
      for (; s + 8 <= s1; s += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = part[(size_t)(s + k) * n + i];
#pragma unroll
        for (int k = 0; k < 8; k++) acc += v[k];
      }
#pragma unroll 1
      for (; s < s1; s++) acc += part[(size_t)s * n + i];
    }
    if constexpr (RUNS > 1) {
      __syncthreads();
      sh[run][col] = acc;
      __syncthreads();
      if (run == 0) {
#pragma unroll
        for (int r = 1; r < RUNS; r++) acc += sh[r][col];
      }
    }
    if (run == 0 && i < n) out[i] = acc;
  }
}

// The elementwise kernels below move 8 channels (16 bytes) per thread.  Those
// over voxels take one item (V channels of one voxel) after another and divide
// its index by high products, so a 64-bit division costs nothing where they
// are large and small or narrow volumes fill the chip too.  With one channel
// per thread the network input took 156 us, the head 147, the pooling 36 on
// average for 2 x 16 x 256 x 256 voxels; now 39, 23 and 16.
// V: 8, or 1 where the channels or an address do not allow 16-byte accesses.
template <int V>
__device__ __forceinline__ void ldv(const bf16 *p, float (&o)[V]) {
  if constexpr (V == 8) {
    const bf16x8 v = *reinterpret_cast<const bf16x8 *>(p);
#pragma unroll
    for (int k = 0; k < 8; k++) o[k] = (float)v[k];
  } else {
    o[0] = (float)p[0];
  }
}
template <int V>
__device__ __forceinline__ void stv(bf16 *p, const float (&o)[V]) {
  if constexpr (V == 8) {
    bf16x8 v;
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = (bf16)o[k];
    *reinterpret_cast<bf16x8 *>(p) = v;
  } else {
    p[0] = (bf16)o[0];
  }
}

// Division of a flat index by one of the sizes behind it.  32 bits, for indices
// below 2^31: one high product with the divisor's reciprocal rounded up (with
// 2^s < d <= 2^(s+1), m d exceeds 2^(32+s) by less than d, so the error stays
// below one step of the quotient); else the plain 64-bit division.
template <class Ix>
struct Div {
  Ix d;
  __device__ __forceinline__ Ix operator()(Ix n) const { return n / d; }
};
template <>
struct Div<uint32_t> {
  uint32_t d, m, s;
  __device__ __forceinline__ uint32_t operator()(uint32_t n) const {
    return m ? __umulhi(n, m) >> s : n;
  }
};
template <class Ix>
static Div<Ix> make_div(long long d) {
  Div<Ix> r{};
  r.d = (Ix)std::max<long long>(d, 1);
  if constexpr (sizeof(Ix) == 4) {
    if (r.d > 1) {
      r.s = 31 - __builtin_clz(r.d - 1);
      r.m = (uint32_t)(((1ull << (32 + r.s)) + r.d - 1) / r.d);
    }
  }
  return r;
}

// A block's sums by channel: thread t holds V channels of group t % nc of one of
// the block's vs voxels, t / nc, of which the first nd have any.  All its channels
// go through LDS at once, then as many threads an output as the block has add
// parts of the voxels, and one adds the parts: two short chains.  (A channel at a
// time and one thread an output, a head's backward pass of 64 voxels took 40 us, 5
// so.)  sh: BS V + BS floats.
template <int V, int BS>
__device__ __forceinline__ void block_channel_sum(const float (&acc)[V], int nc, int nd, float *sh,
                                                  float *out) {
  const int t = threadIdx.x, no = nc * V;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < V; k++) sh[t * V + k] = acc[k];
  __syncthreads();
  const int parts = min(min(BS / no, 16), nd);
  if (parts <= 1) {
    for (int o = t; o < no; o += BS) {
      float s = 0.f;
      for (int d = 0; d < nd; d++) s += sh[d * no + o];
      out[o] = s;
    }
    return;
  }
  float *sp = sh + BS * V;
  const int o = t % no, p = t / no;
  if (p < parts) {
    float s = 0.f;
#pragma unroll 4
    for (int d = p; d < nd; d += parts) s += sh[d * no + o];
    sp[t] = s;
  }
  __syncthreads();
  if (p == 0) {
    float s = sp[o];
#pragma unroll 4
    for (int q = 1; q < parts; q++) s += sp[q * no + o];
    out[o] = s;
  }
}

// part[s][c] = sum over the voxels of slice s of g[v][c] (bias gradient): the
// block's threads hold channel groups and step over the slice's voxels side by
// side (one thread per channel, all voxels in turn: 163 us on average over the
// layers of a training step on 4 x 8 x 128 x 128 voxels, 6 in this form)
template <int V>
__global__ __launch_bounds__(256) void k_channel_sum(const bf16 *__restrict__ g,
                                                     float *__restrict__ part, long long nvox,
                                                     int C, int S) {
  __shared__ float sh[256 * V + 256];
  const int s = blockIdx.x, CG = C / V;
  const long long v0 = nvox * s / S, v1 = nvox * (s + 1) / S;
  for (int c0 = 0; c0 < CG; c0 += 256) {
    const int nc = min(256, CG - c0), vs = 256 / nc;
    const int c = (int)threadIdx.x % nc, dv = (int)threadIdx.x / nc;
    float acc[V] = {};
    if (dv < vs) {
#pragma unroll 4
      for (long long v = v0 + dv; v < v1; v += vs) {
        float x[V];
        ldv<V>(g + (size_t)v * C + (c0 + c) * V, x);
#pragma unroll
        for (int k = 0; k < V; k++) acc[k] += x[k];
      }
    }
    block_channel_sum<V, 256>(acc, nc, (int)min((long long)vs, v1 - v0), sh,
                              part + (size_t)s * C + c0 * V);
  }
}

// g[i] = y[i] > 0 ? g[i] : 0 (ReLU backward through the stored output)
__global__ void k_relu_bwd(const bf16 *__restrict__ y, bf16 *__restrict__ g, size_t n, int vec) {
  const size_t n8 = vec ? n / 8 : 0;
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = tid; i < n8; i += step) {
    const bf16x8 a = reinterpret_cast<const bf16x8 *>(y)[i];
    bf16x8 v = reinterpret_cast<bf16x8 *>(g)[i];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = (float)a[k] > 0.f ? v[k] : (bf16)0.f;
    reinterpret_cast<bf16x8 *>(g)[i] = v;
  }
  for (size_t i = n8 * 8 + tid; i < n; i += step)
    if (!((float)y[i] > 0.f)) g[i] = (bf16)0.f;
}

// 2x2x2 average pooling, forward and backward.  An item is V channels of an
// output voxel; wo, ho, dp divide by the output's sides.
template <int V, class Ix>
__global__ __launch_bounds__(256) void k_avgpool2(const bf16 *__restrict__ in,
                                                  bf16 *__restrict__ out, int C, Ix total,
                                                  Div<Ix> cg, Div<Ix> wo, Div<Ix> ho, Div<Ix> dp) {
  for (Ix j = blockIdx.x * (Ix)blockDim.x + threadIdx.x; j < total;
       j += (Ix)gridDim.x * blockDim.x) {
    const Ix p = cg(j), q = wo(p), r = ho(q), n = dp(r);
    const Ix c = (j - p * cg.d) * V, x = p - q * wo.d, y = q - r * ho.d, z = r - n * dp.d;
    const Ix row = 2 * wo.d * (Ix)C, plane = 2 * ho.d * row;
    const bf16 *src = in + ((n * dp.d + z) * 2 * plane + 2 * y * row + 2 * x * C + c);
    float s[V] = {};
#pragma unroll
    for (int k = 0; k < 8; k++) {
      float v[V];
      ldv<V>(src + ((k >> 2) * plane + ((k >> 1) & 1) * row + (Ix)((k & 1) * C)), v);
#pragma unroll
      for (int u = 0; u < V; u++) s[u] += v[u];
    }
#pragma unroll
    for (int u = 0; u < V; u++) s[u] *= 0.125f;
    stv<V>(out + (size_t)j * V, s);
  }
}

template <int V, class Ix>
__global__ __launch_bounds__(256) void k_avgpool2_bwd(const bf16 *__restrict__ gout,
                                                      bf16 *__restrict__ gin, int C, Ix total,
                                                      Div<Ix> cg, Div<Ix> wo, Div<Ix> ho,
                                                      Div<Ix> dp) {
  for (Ix j = blockIdx.x * (Ix)blockDim.x + threadIdx.x; j < total;
       j += (Ix)gridDim.x * blockDim.x) {
    const Ix p = cg(j), q = wo(p), r = ho(q), n = dp(r);
    const Ix c = (j - p * cg.d) * V, x = p - q * wo.d, y = q - r * ho.d, z = r - n * dp.d;
    float v[V];
    const Ix parent = ((n * (dp.d / 2) + z / 2) * (ho.d / 2) + y / 2) * (wo.d / 2) + x / 2;
    ldv<V>(gout + (parent * C + c), v);
#pragma unroll
    for (int u = 0; u < V; u++) v[u] *= 0.125f;
    stv<V>(gin + (size_t)j * V, v);
  }
}

// out[v][0:Ca] = a[parent(v)][:] (nearest x2 upsampling of the coarse
// features), out[v][Ca:Ca+Cb] = b[v][:] (the skip connection)
template <int V, class Ix>
__global__ __launch_bounds__(256) void k_up2_concat(const bf16 *__restrict__ a,
                                                    const bf16 *__restrict__ b,
                                                    bf16 *__restrict__ out, int Ca, int Cb,
                                                    Ix total, Div<Ix> cg,
                                                    Div<Ix> wo, Div<Ix> ho, Div<Ix> dp) {
  for (Ix j = blockIdx.x * (Ix)blockDim.x + threadIdx.x; j < total;
       j += (Ix)gridDim.x * blockDim.x) {
    const Ix p = cg(j), q = wo(p), r = ho(q), n = dp(r);
    const Ix c = (j - p * cg.d) * V, x = p - q * wo.d, y = q - r * ho.d, z = r - n * dp.d;
    const Ix parent = ((n * (dp.d / 2) + z / 2) * (ho.d / 2) + y / 2) * (wo.d / 2) + x / 2;
    const bf16 *src = c < (Ix)Ca ? a + (parent * Ca + c) : b + (p * Cb + (c - Ca));
    if constexpr (V == 8)
      *reinterpret_cast<bf16x8 *>(out + (size_t)j * 8) = *reinterpret_cast<const bf16x8 *>(src);
    else
      out[j] = *src;
  }
}

// backward of k_up2_concat: ga[p][c] = sum over the 8 children of g[v][c],
// gb[v][c] = g[v][Ca + c]; the na groups of V channels of ga, then those of gb.
// Each output has an item of its own, so every row of gb is written, also the
// last ones of an odd size, which no parent covers.
template <int V, class Ix>
__global__ __launch_bounds__(256) void k_up2_concat_bwd(const bf16 *__restrict__ g,
                                                        bf16 *__restrict__ ga,
                                                        bf16 *__restrict__ gb, int D, int H, int W,
                                                        int Ca, int Cb, Ix na, Ix total,
                                                        Div<Ix> ag, Div<Ix> bg, Div<Ix> wc,
                                                        Div<Ix> hc, Div<Ix> dc) {
  const int C = Ca + Cb;
  for (Ix j = blockIdx.x * (Ix)blockDim.x + threadIdx.x; j < total;
       j += (Ix)gridDim.x * blockDim.x) {
    if (j < na) {
      const Ix p = ag(j), q = wc(p), r = hc(q), n = dc(r);
      const Ix c = (j - p * ag.d) * V, x = p - q * wc.d, y = q - r * hc.d, z = r - n * dc.d;
      const bf16 *src = g + ((((n * D + 2 * z) * H + 2 * y) * W + 2 * x) * C + c);
      float s[V] = {};
#pragma unroll
      for (int k = 0; k < 8; k++) {
        float v[V];
        ldv<V>(src + (((Ix)(k >> 2) * H + ((k >> 1) & 1)) * W + (k & 1)) * C, v);
#pragma unroll
        for (int u = 0; u < V; u++) s[u] += v[u];
      }
      stv<V>(ga + (size_t)j * V, s);
    } else {
      const Ix i = j - na, v = bg(i);
      const bf16 *src = g + (v * C + Ca + (i - v * bg.d) * V);
      if constexpr (V == 8)
        *reinterpret_cast<bf16x8 *>(gb + (size_t)i * 8) = *reinterpret_cast<const bf16x8 *>(src);
      else
        gb[i] = *src;
    }
  }
}

// network input: x[v][0] = s * fbp[v], x[v][1] = s * mean over frames of
// fbp[v], channels 2..31 zero; the volumes are fp32 [N][D][H][W] (one
// sample per frame) and mean is [D][H][W] (shared by all samples)
__global__ void k_make_input(const float *__restrict__ fbp, const float *__restrict__ mean,
                             bf16 *__restrict__ x, long long nvox, long long per, float scale,
                             int vec) {
  const bool small = nvox <= 0x7fffffffLL && per <= 0x7fffffffLL;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)nvox * 4;
       i += (size_t)gridDim.x * blockDim.x) {
    const size_t v = i >> 2;
    bf16x8 o = zero8();
    if ((i & 3) == 0) {
      o[0] = (bf16)(scale * fbp[v]);
      if (mean) o[1] = (bf16)(scale * mean[small ? (uint32_t)v % (uint32_t)per : v % (size_t)per]);
    }
    bf16 *p = x + v * 32 + (i & 3) * 8;
    if (vec) {
      *reinterpret_cast<bf16x8 *>(p) = o;
    } else {
#pragma unroll
      for (int k = 0; k < 8; k++) p[k] = o[k];
    }
  }
}

// mean[q] = sum over frames f of x[f * per + q] / nframes (fp32, frames in
// order): the temporal mean of a 4D object, the network's second input
__global__ void k_frame_mean(const float *__restrict__ x, float *__restrict__ mean,
                             long long nframes, long long per) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < (size_t)per;
       q += (size_t)gridDim.x * blockDim.x) {
    float s = 0.f;
    for (long long f = 0; f < nframes; f++) s += x[(size_t)f * per + q];
    mean[q] = s / (float)nframes;
  }
}

// output head: out[v] = fbp[v] + (b + sum_c w[c] h[v][c]) / scale (a 1x1x1
// convolution to one channel, a residual on the filtered back-projection)
__global__ void k_head_fwd(const bf16 *__restrict__ h, const float *__restrict__ w,
                           const float *__restrict__ b, const float *__restrict__ fbp,
                           float *__restrict__ out, long long nvox, int C, float inv_scale,
                           int vec) {
  for (size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x; v < (size_t)nvox;
       v += (size_t)gridDim.x * blockDim.x) {
    float s = b[0];
    if (vec) {
      for (int c = 0; c < C; c += 32) {
        bf16x8 x[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
          x[k] = *reinterpret_cast<const bf16x8 *>(h + v * C + c + 8 * k);
#pragma unroll
        for (int k = 0; k < 32; k++) s += w[c + k] * (float)x[k / 8][k % 8];
      }
    } else {
      for (int c = 0; c < C; c++) s += w[c] * (float)h[v * C + c];
    }
    out[v] = fbp[v] + s * inv_scale;
  }
}

// mean squared error over nvox voxels: part[block] = partial sums of
// (out - target)^2; gout[v] = 2 (out - target) / nvox (fp32)
__global__ void k_mse(const float *__restrict__ out, const float *__restrict__ target,
                      float *__restrict__ gout, double *__restrict__ part, long long nvox) {
  __shared__ double sh[256];
  double s = 0.0;
  for (size_t v = blockIdx.x * (size_t)blockDim.x + threadIdx.x; v < (size_t)nvox;
       v += (size_t)gridDim.x * blockDim.x) {
    const float e = out[v] - target[v];
    s += (double)e * e;
    gout[v] = 2.f * e / (float)nvox;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = blockDim.x / 2; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// head backward: gh[v][c] = gout[v] w[c] / scale (bf16); the head's weight
// and bias gradients per slice of voxels: part[s][c] = sum gout[v] h[v][c] /
// scale (c < C), part[s][C] = sum gout[v] / scale.  One pass, block = slice:
// the weight sums, once a thread per channel walking the slice's voxels, were
// the whole of its 417 us for 4 x 8 x 128 x 128 voxels; now 17.
// S 0: gh alone, the blocks sharing its voxels; C 0: the bias gradient alone.
template <int V, int BS>
__global__ __launch_bounds__(BS) void k_head_bwd(const bf16 *__restrict__ h,
                                                 const float *__restrict__ w,
                                                 const float *__restrict__ gout,
                                                 bf16 *__restrict__ gh, float *__restrict__ part,
                                                 long long nvox, int C, int S, float inv_scale) {
  __shared__ float sh[BS * V + BS];
  const int s = blockIdx.x, CG = C / V;
  const long long v0 = nvox * s / gridDim.x, v1 = nvox * (s + 1) / gridDim.x;
  for (int c0 = 0; c0 == 0 || c0 < CG; c0 += BS) {
    const int nc = max(min(BS, CG - c0), 1), vs = BS / nc;
    const int cg = (int)threadIdx.x % nc, dv = (int)threadIdx.x / nc, c = (c0 + cg) * V;
    const int nd = (int)min((long long)vs, v1 - v0);
    const long long begin = dv < vs ? v0 + dv : v1;
    float gs = 0.f;
    if (CG > 0) {
      float acc[V] = {}, wc[V];
#pragma unroll
      for (int k = 0; k < V; k++) wc[k] = w[c + k];
#pragma unroll 4
      for (long long v = begin; v < v1; v += vs) {
        const float g = gout[v] * inv_scale;
        float x[V], o[V];
        ldv<V>(h + (size_t)v * C + c, x);
#pragma unroll
        for (int k = 0; k < V; k++) {
          o[k] = g * wc[k];
          acc[k] += g * x[k];
        }
        stv<V>(gh + (size_t)v * C + c, o);
        gs += g;
      }
      if (S > 0) block_channel_sum<V, BS>(acc, nc, nd, sh, part + (size_t)s * (C + 1) + c0 * V);
    } else {
      for (long long v = begin; v < v1; v += vs) gs += gout[v] * inv_scale;
    }
    if (c0 == 0 && S > 0) {
      // the bias, which the first thread of each voxel has
      __syncthreads();
      if (cg == 0) sh[dv] = gs;
      __syncthreads();
      const float bias[1] = {sh[threadIdx.x]};
      block_channel_sum<1, BS>(bias, 1, nd, sh, part + (size_t)s * (C + 1) + C);
    }
  }
}

// Adam with bias correction on fp32 master weights; bf16 copies for the
// kernels (wb may be null)
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ gr, float *__restrict__ m,
                       float *__restrict__ v, bf16 *__restrict__ wb, size_t n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    if (wb) wb[i] = (bf16)pi;
  }
}

// a[i] = a[i] + b[i] (bf16, the sum rounded once): gradients reaching one
// activation from two consumers
__global__ void k_add_bf16(bf16 *__restrict__ a, const bf16 *__restrict__ b, size_t n, int vec) {
  const size_t n8 = vec ? n / 8 : 0;
  const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = tid; i < n8; i += step) {
    bf16x8 x = reinterpret_cast<bf16x8 *>(a)[i];
    const bf16x8 y = reinterpret_cast<const bf16x8 *>(b)[i];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = (bf16)((float)x[k] + (float)y[k]);
    reinterpret_cast<bf16x8 *>(a)[i] = x;
  }
  for (size_t i = n8 * 8 + tid; i < n; i += step) a[i] = (bf16)((float)a[i] + (float)b[i]);
}

__global__ void k_to_bf16(const float *__restrict__ a, bf16 *__restrict__ b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    b[i] = (bf16)a[i];
}

}  // namespace tbnn

using namespace tbnn;

// ---------------------------------------------------------------------------
// C ABI (declared in include/timbir_dev.h)
// ---------------------------------------------------------------------------
static thread_local std::string g_nn_err;

static int nn_fail(const char *msg, hipError_t e = hipSuccess) {
  g_nn_err = msg;
  if (e != hipSuccess) {
    g_nn_err += ": ";
    g_nn_err += hipGetErrorString(e);
  }
  return -1;
}

#define NNCHK(what)                                     \
  do {                                                  \
    hipError_t e_ = hipGetLastError();                  \
    if (e_ != hipSuccess) return nn_fail(what, e_);     \
  } while (0)

static int grid1d(size_t n) {
  size_t g = (n + 255) / 256;
  if (g < 1) g = 1;
  if (g > 65535 * 8) g = 65535 * 8;
  return (int)g;
}

// blocks of 256 threads in a launch: its threads are counted in 32 bits
constexpr long long kMaxBlocks = 0xffffffffLL / 256;

static bool al16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

extern "C" const char *tb_nn_last_error(void) { return g_nn_err.c_str(); }

// Device memory for the callers of these kernels, from this library's HIP
// runtime (so that the kernels and the copies are ordered on its streams).
extern "C" int tb_dev_malloc(uint64_t bytes, void **ptr) {
  *ptr = nullptr;
  hipError_t e = hipMalloc(ptr, bytes ? bytes : 1);
  if (e != hipSuccess) return nn_fail("tb_dev_malloc", e);
  return 0;
}

extern "C" int tb_dev_free(void *ptr) {
  hipError_t e = hipFree(ptr);
  if (e != hipSuccess) return nn_fail("tb_dev_free", e);
  return 0;
}

extern "C" int tb_dev_copy(void *dst, const void *src, uint64_t bytes, int32_t kind) {
  // kind: 0 host to device, 1 device to host, 2 device to device; blocking
  const hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice
                          : kind == 1 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
  hipError_t e = hipMemcpy(dst, src, bytes, k);
  if (e != hipSuccess) return nn_fail("tb_dev_copy", e);
  return 0;
}

extern "C" int tb_dev_zero(void *ptr, uint64_t bytes, void *stream) {
  hipError_t e = hipMemsetAsync(ptr, 0, bytes, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return nn_fail("tb_dev_zero", e);
  return 0;
}

extern "C" int tb_dev_synchronize(void) {
  hipError_t e = hipDeviceSynchronize();
  if (e != hipSuccess) return nn_fail("tb_dev_synchronize", e);
  return 0;
}

template <int CA, int CB, int NB, int SP, int WT>
static int conv_tile(const void *a, const void *in, const void *w, const float *bias, void *out,
                     int n, int d, int h, int wd, int cout, int relu, int out_f32, hipStream_t s) {
  using T = ConvTile<CA, CB, SP, WT>;
  auto fn = k_conv3d_tile<CA, CB, NB, SP, WT>;
  const long long blocks = (long long)n * d * ((h + T::HT - 1) / T::HT) * ((wd + WT - 1) / WT) *
                           (cout / (16 * NB));
  if (blocks > kMaxBlocks) return nn_fail("tb_nn_conv3d: volume too large");
  if (T::kBytes > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)T::kBytes);
    if (e != hipSuccess) return nn_fail("tb_nn_conv3d", e);
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(256), T::kBytes, s,
                     static_cast<const bf16 *>(a), static_cast<const bf16 *>(in),
                     static_cast<const bf16 *>(w), bias, out, n, d, h, wd, cout, relu, out_f32);
  NNCHK("tb_nn_conv3d");
  return 0;
}

using conv_fn = int (*)(const void *, const void *, const void *, const float *, void *, int, int,
                        int, int, int, int, int, hipStream_t);
// A staged form: its launch, workgroups, and voxels of a plane with its rows and
// columns filled up to whole tiles.  Strips of 64 x 1 voxels, or 32 x 2 where
// that leaves fewer lanes without a voxel (and for 128 + 64 input channels,
// whose tile of 64 leaves one workgroup per CU).
struct ConvForm {
  conv_fn fn;
  long long blocks, slots;
};
template <int CA, int CB, int NB, int SP>
static ConvForm conv_form(long long planes, int h, int wd, int cout) {
  const bool narrow = CA == 4 || (wd + 31LL) / 32 * 32 < (wd + 63LL) / 64 * 64;
  const long long WT = narrow ? 32 : 64, HT = 4 * SP * (64 / WT);
  const long long th = (h + HT - 1) / HT, tw = (wd + WT - 1) / WT;
  return {narrow ? conv_tile<CA, CB, NB, SP, 32> : conv_tile<CA, CB, NB, SP, 64>,
          planes * th * tw * (cout / (16 * NB)), th * HT * tw * WT};
}
// More output channels a wave use a staged value more often, but a wave's chain
// is longer: 32 channels while that leaves the chip with at most three workgroups
// a CU (one where LDS holds one, from 128 input channels on), else 64, else 96.
// 64 -> 64 channels, 16 planes of 16 x 16 voxels: 36 us with 64 channels a wave,
// 23 with 32; 128 -> 128, 64 planes of 16 x 32: 66 and 82.  Two strips per wave for
// 32 channels of 32 inputs, where the weights' share of the L1 would otherwise
// bound, unless they fill up a quarter more rows.
template <int CA, int CB>
static ConvForm conv_pick(long long planes, int h, int wd, int cout) {
  constexpr long long few = CA + CB >= 4 ? 256 : 768;
  ConvForm f = conv_form<CA, CB, 2, 1>(planes, h, wd, cout);
  if constexpr (CA == 0 && CB == 1) {
    if (f.blocks > few && cout % 64 && cout % 96) {
      const ConvForm g = conv_form<CA, CB, 2, 2>(planes, h, wd, cout);
      if (g.slots <= f.slots * 5 / 4) f = g;
    }
  }
  if (f.blocks > few && cout % 64 == 0) f = conv_form<CA, CB, 4, 1>(planes, h, wd, cout);
  if (f.blocks > few && cout % 96 == 0) f = conv_form<CA, CB, 6, 1>(planes, h, wd, cout);
  return f;
}

extern "C" int tb_nn_conv3d(const void *in, const void *w, const float *bias, void *out,
                            int32_t n, int32_t d, int32_t h, int32_t wd, int32_t cin,
                            int32_t cout, int32_t relu, int32_t out_f32, void *stream) {
  if (n <= 0 || d <= 0 || h <= 0 || wd <= 0 || cin % 32 || cout % 32 || cin <= 0 || cout <= 0)
    return nn_fail("tb_nn_conv3d: sizes must be positive, channels multiples of 32");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long planes = (long long)n * d;
  const ConvForm f = cin == 32    ? conv_pick<0, 1>(planes, h, wd, cout)
                     : cin == 64  ? conv_pick<0, 2>(planes, h, wd, cout)
                     : cin == 96  ? conv_pick<0, 3>(planes, h, wd, cout)
                     : cin == 128 ? conv_pick<0, 4>(planes, h, wd, cout)
                     : cin == 192 ? conv_pick<0, 6>(planes, h, wd, cout)
                                  : ConvForm{nullptr, 0, 0};
  // Unstaged: planes of one row, two thirds of whose taps lie outside (4 planes of
  // one voxel, 128 -> 128 channels: 27 us staged, 16 unstaged; not one long row
  // alone), volumes of two or three rows that fill the chip, whose tiles are empty
  // by half and more (512 planes of 2 x 4, 128 -> 64: 74 and 42), other channels, an
  // output that 16-byte stores do not allow, and more tiles than a launch holds.
  const long long strips = (wd + 63LL) / 64 * 64 * h;
  const bool empty = f.slots > 2 * strips || (f.slots == 2 * strips && (cin >= 96 || wd <= 8));
  const bool unstaged = (h == 1 && (planes > 1 || wd <= 32)) || (empty && f.blocks >= 512);
  if (f.fn && al16(out) && !unstaged && f.blocks <= kMaxBlocks)
    return f.fn(nullptr, in, w, bias, out, n, d, h, wd, cout, relu, out_f32, s);
  const int MB = 4, NB = 2;
  const long long waves = planes * h * ((wd + 16 * MB - 1) / (16 * MB)) * (cout / (16 * NB));
  const long long blocks = (waves + kWavesPerBlock - 1) / kWavesPerBlock;
  if (blocks > kMaxBlocks) return nn_fail("tb_nn_conv3d: volume too large");
  hipLaunchKernelGGL((k_conv3d_fwd<4, 2>), dim3((unsigned)blocks), dim3(64 * kWavesPerBlock), 0,
                     s, static_cast<const bf16 *>(in), static_cast<const bf16 *>(w), bias, out, n,
                     d, h, wd, cin, cout, relu, out_f32);
  NNCHK("tb_nn_conv3d");
  return 0;
}

extern "C" int tb_nn_conv3d_up2cat(const void *a, const void *b, const void *w, const float *bias,
                                   void *out, int32_t n, int32_t d, int32_t h, int32_t wd,
                                   int32_t ca, int32_t cb, int32_t cout, int32_t relu,
                                   void *stream) {
  if (n <= 0 || d <= 0 || h <= 0 || wd <= 0 || d % 2 || h % 2 || wd % 2 || cout <= 0 || cout % 32)
    return nn_fail("tb_nn_conv3d_up2cat: sizes must be positive and even, channels multiples of 32");
  const long long planes = (long long)n * d;
  const conv_fn fn = ca == 64 && cb == 32    ? conv_pick<2, 1>(planes, h, wd, cout).fn
                     : ca == 128 && cb == 64 ? conv_pick<4, 2>(planes, h, wd, cout).fn
                                             : nullptr;
  if (!fn) return nn_fail("tb_nn_conv3d_up2cat: 64 + 32 or 128 + 64 input channels");
  if (!al16(a) || !al16(b) || !al16(w) || !al16(out))
    return nn_fail("tb_nn_conv3d_up2cat: a, b, w and out must be 16-byte aligned");
  return fn(a, b, w, bias, out, n, d, h, wd, cout, relu, 0, static_cast<hipStream_t>(stream));
}

extern "C" int tb_nn_conv3d_flip(const void *w, void *wt, int32_t cin, int32_t cout,
                                 void *stream) {
  hipLaunchKernelGGL(k_conv_flip, dim3(grid1d((size_t)kTaps * cin * cout)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const bf16 *>(w),
                     static_cast<bf16 *>(wt), cin, cout);
  NNCHK("tb_nn_conv3d_flip");
  return 0;
}

template <int RUNS, int E>
static void sum_parts_runs(const float *part, float *out, size_t n, int slices, hipStream_t s) {
  const unsigned blocks =
      (unsigned)std::min<size_t>(std::max<size_t>((n + E - 1) / E, 1), 65536);
  hipLaunchKernelGGL((k_sum_parts<RUNS, E>), dim3(blocks), dim3(E * RUNS), 0, s, part, out, n,
                     slices);
}
// As many runs as give the chip its 2^19 threads: 27648 entries of 256 slices take
// 9 us in one run, 4 in 16; 331776 entries of 32 slices 8 in one, 20 in 16.  (One
// thread per entry and one load at a time took 26 and 11.)
static void sum_parts(const float *part, float *out, size_t n, int slices, hipStream_t s) {
  if (n <= (1u << 19) / 16) sum_parts_runs<16, 64>(part, out, n, slices, s);
  else if (n <= (1u << 19) / 4) sum_parts_runs<4, 64>(part, out, n, slices, s);
  else sum_parts_runs<1, 256>(part, out, n, slices, s);
}

extern "C" int tb_nn_conv3d_wgrad(const void *in, const void *gout, float *gw, float *part,
                                  int32_t slices, int32_t n, int32_t d, int32_t h, int32_t wd,
                                  int32_t cin, int32_t cout, void *stream) {
  if (cin % 32 || cout % 32 || slices <= 0)
    return nn_fail("tb_nn_conv3d_wgrad: channels must be multiples of 32");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t nw = (size_t)kTaps * cin * cout;
  // about two blocks per CU over the 32 x 32 channel pairs; planes are split
  // into runs (each reads two planes more) only where tiles alone are fewer
  const long long pairs = (long long)(cin / 32) * (cout / 32);
  const long long want = std::max<long long>(1, 512 / std::max<long long>(pairs, 1));
  WgradUnits U;
  U.hb = (h + kGH - 1) / kGH;
  U.wb = (wd + kGW - 1) / kGW;
  const long long tiles = std::max<long long>((long long)n * U.hb * U.wb, 1);
  const long long runs = std::min<long long>(std::max<long long>(want / tiles, 1), (d + 3) / 4);
  U.per = std::max<int>((int)((d + runs - 1) / std::max<long long>(runs, 1)), 1);
  U.zc = (d + U.per - 1) / U.per;
  const long long units = (long long)n * U.hb * U.wb * U.zc;
  if (units > 0x7fffffffLL) return nn_fail("tb_nn_conv3d_wgrad: volume too large");
  U.units = (int)units;
  // partial sums: as many as have work, the units shared out evenly
  long long S = std::max<long long>(1, std::min<long long>({(long long)slices, units, want}));
  S = std::max<long long>(1, (units + (units + S - 1) / S - 1) / std::max<long long>((units + S - 1) / S, 1));
  // A workgroup stages a plane (a unit of several has one and a half more) in about
  // the time in which a wave of the flat kernel walks 1.25 chunks of 32 voxels (4.6
  // and 3.7 us); 256 workgroups run at once, and about 2000 such waves.  Volumes of
  // short rows, few rows or few slices are sooner done by chunks: 512 planes of 1 x 2
  // voxels, 4 slices, 32 -> 32 channels take 663 us in tiles and 37 by chunks; 16
  // planes of 48 x 48, 256 slices, 30 and 75.
  const long long chunks = ((long long)n * d * h * wd + 31) / 32;
  const long long SF = std::max<long long>(1, std::min<long long>(slices, chunks));
  const double flat = 1.25 * (double)((chunks + SF - 1) / SF) *
                      std::max(1.0, (double)(SF * kTaps * pairs) / 2000.0);
  const double tile = (double)((units + S - 1) / S) * (U.per + (d > 1 ? 1.5 : 0.5)) *
                      (double)((S * pairs + 255) / 256);
  const long long flat_blocks = (SF * kTaps * pairs + kWavesPerBlock - 1) / kWavesPerBlock;
  if (flat < tile && flat_blocks <= kMaxBlocks) {
    hipLaunchKernelGGL((k_conv3d_wgrad_flat<2, 2>), dim3((unsigned)flat_blocks),
                       dim3(64 * kWavesPerBlock), 0, s, static_cast<const bf16 *>(in),
                       static_cast<const bf16 *>(gout), part, n, d, h, wd, cin, cout, (int)SF);
    sum_parts(part, gw, nw, (int)SF, s);
    NNCHK("tb_nn_conv3d_wgrad");
    return 0;
  }
  const size_t lds = (size_t)(3 * 2 * (kGH + 2) * (kGW + 2) + 2 * kGH * kGW) * 16 * sizeof(bf16);
  auto fn = al16(in) && al16(gout) ? k_conv3d_wgrad<true> : k_conv3d_wgrad<false>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return nn_fail("tb_nn_conv3d_wgrad", e);
  hipLaunchKernelGGL(fn, dim3((unsigned)(S * pairs)), dim3(kGThreads), lds, s,
                     static_cast<const bf16 *>(in), static_cast<const bf16 *>(gout), part, n, d, h,
                     wd, cin, cout, (int)S, U);
  sum_parts(part, gw, nw, (int)S, s);
  NNCHK("tb_nn_conv3d_wgrad");
  return 0;
}

extern "C" int tb_nn_channel_sum(const void *g, float *out, float *part, int32_t slices,
                                 int64_t nvox, int32_t c, void *stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto fn = c % 8 == 0 && al16(g) ? k_channel_sum<8> : k_channel_sum<1>;
  hipLaunchKernelGGL(fn, dim3(slices), dim3(256), 0, s, static_cast<const bf16 *>(g), part,
                     (long long)nvox, c, slices);
  sum_parts(part, out, (size_t)c, slices, s);
  NNCHK("tb_nn_channel_sum");
  return 0;
}

extern "C" int tb_nn_relu_bwd(const void *y, void *g, int64_t count, void *stream) {
  hipLaunchKernelGGL(k_relu_bwd, dim3(grid1d((count + 7) / 8)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const bf16 *>(y),
                     static_cast<bf16 *>(g), (size_t)count, al16(y) && al16(g));
  NNCHK("tb_nn_relu_bwd");
  return 0;
}

// Blocks of the kernels over voxels' items: 32 a CU at most, so a thread of a
// large volume takes several (concatenation's backward pass, 2 x 16 x 256 x 256
// voxels, 32 + 32 channels: 111 us with a block for every 256 items, 95 so).
static int item_grid(size_t n) { return std::min(grid1d(n), 8192); }

// The kernels over voxels, by index type and channels a thread.  32-bit indices
// serve volumes below 2^31 items.
static bool small_index(int n, int d, int h, int wd, long long c) {
  return (double)n * d * h * wd * (double)c < 2147483647.0;
}

template <int V, class Ix>
static void avgpool2(const void *in, void *out, int n, int d, int h, int wd, int c, bool backward,
                     hipStream_t s) {
  const int k = backward ? 1 : 2;
  d /= k, h /= k, wd /= k;  // the output's size
  const size_t total = (size_t)n * d * h * wd * (c / V);
  hipLaunchKernelGGL((backward ? k_avgpool2_bwd<V, Ix> : k_avgpool2<V, Ix>), dim3(item_grid(total)),
                     dim3(256), 0, s, static_cast<const bf16 *>(in), static_cast<bf16 *>(out), c,
                     (Ix)total, make_div<Ix>(c / V), make_div<Ix>(wd), make_div<Ix>(h),
                     make_div<Ix>(d));
}

extern "C" int tb_nn_avgpool2(const void *in, void *out, int32_t n, int32_t d, int32_t h,
                              int32_t wd, int32_t c, int32_t backward, void *stream) {
  if (d % 2 || h % 2 || wd % 2) return nn_fail("tb_nn_avgpool2: odd size");
  if (n <= 0 || d <= 0 || h <= 0 || wd <= 0 || c <= 0) return 0;
  const bool vec = c % 8 == 0 && al16(in) && al16(out);
  const bool small = small_index(n, d, h, wd, c);
  auto fn = vec ? (small ? avgpool2<8, uint32_t> : avgpool2<8, uint64_t>)
                : (small ? avgpool2<1, uint32_t> : avgpool2<1, uint64_t>);
  fn(in, out, n, d, h, wd, c, backward != 0, static_cast<hipStream_t>(stream));
  NNCHK("tb_nn_avgpool2");
  return 0;
}

template <int V, class Ix>
static void up2_concat(const void *a, const void *b, void *out, int n, int d, int h, int wd, int ca,
                       int cb, hipStream_t s) {
  const size_t total = (size_t)n * d * h * wd * ((ca + cb) / V);
  hipLaunchKernelGGL((k_up2_concat<V, Ix>), dim3(item_grid(total)), dim3(256), 0, s,
                     static_cast<const bf16 *>(a), static_cast<const bf16 *>(b),
                     static_cast<bf16 *>(out), ca, cb, (Ix)total, make_div<Ix>((ca + cb) / V),
                     make_div<Ix>(wd), make_div<Ix>(h), make_div<Ix>(d));
}

extern "C" int tb_nn_up2_concat(const void *a, const void *b, void *out, int32_t n, int32_t d,
                                int32_t h, int32_t wd, int32_t ca, int32_t cb, void *stream) {
  if (n <= 0 || d <= 0 || h <= 0 || wd <= 0 || ca + cb <= 0) return 0;
  const bool vec = ca % 8 == 0 && cb % 8 == 0 && al16(a) && al16(b) && al16(out);
  const bool small = small_index(n, d, h, wd, (long long)ca + cb);
  auto fn = vec ? (small ? up2_concat<8, uint32_t> : up2_concat<8, uint64_t>)
                : (small ? up2_concat<1, uint32_t> : up2_concat<1, uint64_t>);
  fn(a, b, out, n, d, h, wd, ca, cb, static_cast<hipStream_t>(stream));
  NNCHK("tb_nn_up2_concat");
  return 0;
}

template <int V, class Ix>
static void up2_concat_bwd(const void *g, void *ga, void *gb, int n, int d, int h, int wd, int ca,
                           int cb, hipStream_t s) {
  const size_t na = (size_t)n * (d / 2) * (h / 2) * (wd / 2) * (ca / V);
  const size_t total = na + (size_t)n * d * h * wd * (cb / V);
  hipLaunchKernelGGL((k_up2_concat_bwd<V, Ix>), dim3(item_grid(total)), dim3(256), 0, s,
                     static_cast<const bf16 *>(g), static_cast<bf16 *>(ga),
                     static_cast<bf16 *>(gb), d, h, wd, ca, cb, (Ix)na, (Ix)total,
                     make_div<Ix>(ca / V), make_div<Ix>(cb / V), make_div<Ix>(wd / 2),
                     make_div<Ix>(h / 2), make_div<Ix>(d / 2));
}

extern "C" int tb_nn_up2_concat_bwd(const void *g, void *ga, void *gb, int32_t n, int32_t d,
                                    int32_t h, int32_t wd, int32_t ca, int32_t cb, void *stream) {
  if (n <= 0 || d <= 0 || h <= 0 || wd <= 0 || ca + cb <= 0) return 0;
  const bool vec = ca % 8 == 0 && cb % 8 == 0 && al16(g) && al16(ga) && al16(gb);
  const bool small = small_index(n, d, h, wd, (long long)ca + cb);
  auto fn = vec ? (small ? up2_concat_bwd<8, uint32_t> : up2_concat_bwd<8, uint64_t>)
                : (small ? up2_concat_bwd<1, uint32_t> : up2_concat_bwd<1, uint64_t>);
  fn(g, ga, gb, n, d, h, wd, ca, cb, static_cast<hipStream_t>(stream));
  NNCHK("tb_nn_up2_concat_bwd");
  return 0;
}

extern "C" int tb_nn_add(void *a, const void *b, int64_t count, void *stream) {
  hipLaunchKernelGGL(k_add_bf16, dim3(grid1d((count + 7) / 8)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<bf16 *>(a),
                     static_cast<const bf16 *>(b), (size_t)count, al16(a) && al16(b));
  NNCHK("tb_nn_add");
  return 0;
}

extern "C" int tb_nn_make_input(const float *fbp, const float *mean, void *x, int64_t nvox,
                                int64_t per_sample, float scale, void *stream) {
  hipLaunchKernelGGL(k_make_input, dim3(grid1d((size_t)nvox * 4)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), fbp, mean, static_cast<bf16 *>(x),
                     (long long)nvox, (long long)per_sample, scale, al16(x));
  NNCHK("tb_nn_make_input");
  return 0;
}

extern "C" int tb_nn_frame_mean(const float *x, float *mean, int64_t nframes, int64_t per,
                                void *stream) {
  hipLaunchKernelGGL(k_frame_mean, dim3(grid1d(per)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, mean, (long long)nframes,
                     (long long)per);
  NNCHK("tb_nn_frame_mean");
  return 0;
}

extern "C" int tb_nn_head(const void *h, const float *w, const float *b, const float *fbp,
                          float *out, int64_t nvox, int32_t c, float scale, void *stream) {
  hipLaunchKernelGGL(k_head_fwd, dim3(grid1d(nvox)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const bf16 *>(h), w, b, fbp,
                     out, (long long)nvox, c, 1.f / scale, c % 32 == 0 && al16(h));
  NNCHK("tb_nn_head");
  return 0;
}

extern "C" int tb_nn_head_bwd(const void *h, const float *w, const float *gout, void *gh,
                              float *part, int32_t slices, int64_t nvox, int32_t c, float scale,
                              void *stream) {
  // one wave a slice where it has no more to do (2048 slices of 5000 voxels x 32
  // channels: 9 us with eight, 4 with one)
  const bool vec = c % 8 == 0 && al16(h) && al16(gh);
  const int blocks = slices > 0 ? slices : grid1d((size_t)(nvox + 127) / 128);
  const bool one = (nvox / blocks + 1) * (double)(vec ? c / 8 : c) <= 64.0;
  auto fn = vec ? (one ? k_head_bwd<8, 64> : k_head_bwd<8, 512>)
                : (one ? k_head_bwd<1, 64> : k_head_bwd<1, 512>);
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(one ? 64 : 512), 0, static_cast<hipStream_t>(stream),
                     static_cast<const bf16 *>(h), w, gout, static_cast<bf16 *>(gh), part,
                     (long long)nvox, c, slices, 1.f / scale);
  NNCHK("tb_nn_head_bwd");
  return 0;
}

extern "C" int tb_nn_mse(const float *out, const float *target, float *gout, double *part,
                         int32_t blocks, int64_t nvox, void *stream) {
  hipLaunchKernelGGL(k_mse, dim3(blocks), dim3(256), 0, static_cast<hipStream_t>(stream), out,
                     target, gout, part, (long long)nvox);
  NNCHK("tb_nn_mse");
  return 0;
}

extern "C" int tb_nn_sum_parts(const float *part, float *out, int64_t count, int32_t slices,
                               void *stream) {
  sum_parts(part, out, (size_t)count, slices, static_cast<hipStream_t>(stream));
  NNCHK("tb_nn_sum_parts");
  return 0;
}

extern "C" int tb_nn_adam(float *p, const float *g, float *m, float *v, void *wb, int64_t count,
                          float lr, float b1, float b2, float eps, int32_t step, void *stream) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(grid1d(count)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     p, g, m, v, static_cast<bf16 *>(wb), (size_t)count, lr, b1, b2, eps, c1, c2);
  NNCHK("tb_nn_adam");
  return 0;
}

extern "C" int tb_nn_to_bf16(const float *a, void *b, int64_t count, void *stream) {
  hipLaunchKernelGGL(k_to_bf16, dim3(grid1d(count)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a, static_cast<bf16 *>(b), (size_t)count);
  NNCHK("tb_nn_to_bf16");
  return 0;
}
