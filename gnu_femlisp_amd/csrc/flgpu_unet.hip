// Learned coarse correction: a 3-level 3D U-Net (16/32/64 channels, 3x3x3
// kernels) with BF16 weights and FP32 accumulation on MFMA, trained on the
// GPU by its own forward and backward kernels with Adam.
//
// No femlisp counterpart: femlisp has no learned components.  The network is
// used by flgpu_solve as an extra correction inside the flexible CG: after
// the V-cycle z1 = V(r), the residual r1 = r - A z1 is fed to the network and
// z = z1 + N(r1); plain GMG-FCG takes over when the defect stalls.
//
// Tensors are channels-last [batch][z][y][x][c] in FP32.  Convolutions are
// implicit GEMMs on v_mfma_f32_16x16x16bf16_1k over voxels (tiles of 16),
// output channels (tiles of 16) and 27 taps x input channels (chunks of
// 16); activations and weights are rounded to BF16 when they enter the
// matrix cores, products accumulate in FP32.  Weight gradients are implicit
// GEMMs on the same instruction (voxels as K) with per-block partials reduced
// in a fixed order.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "flgpu_learned.h"

namespace flgpu {

constexpr int NL = 9;
static const int L_CIN[NL] = {-1, 16, 16, 32, 32, 64, 96, 48, 16};
static const int L_COUT[NL] = {16, 16, 32, 32, 64, 64, 32, 16, 1};
static const int L_LEVEL[NL] = {0, 0, 1, 1, 2, 2, 1, 0, 0};

typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short bf16_bits(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}

// ---- tiles of the convolutions ----------------------------------------------------------------
// A workgroup works on a box of bz x by x bx voxels of one sample; the input channels of the box
// and of the one-voxel halo around it are staged in LDS as BF16, one plane of 16 channels after
// another: lds[chunk][halo voxel][16].  With 32 bytes per voxel the 16 lanes of an MFMA operand
// (16 voxels) times its four channel groups read 512 consecutive bytes wherever the tap shifts
// them, so no tap has bank conflicts and every value is rounded to BF16 once per box instead of
// once per tap.
struct ConvGeom {
  int n;                   // voxels per axis
  int bz, by, bx;          // box
  int vol, hvol;           // voxels of the box, of the box with its halo
  int nbox;                // boxes of all samples
  Div1 dnx, dny, dnz;      // boxes per axis
  Div1 dbx, dby, dhx, dhy; // box and halo extents
};

// how a convolution's blocks are split (conv_plan)
struct ConvPlan {
  ConvGeom g;
  int mt, nt, wm;  // voxel and channel tiles per wave, waves along the voxels
  int nch, ntt;    // chunks of input channels, tiles of output channels
};

// The input of a convolution: channels [0, c0) from p0, [c0, c0 + c1) from p1.  up: p0 lives
// on the grid of n / 2 voxels per axis and is upsampled (nearest), the decoder's concatenation
// [upsampled, skip], which is then never stored.
struct ConvIn {
  const float *p0, *p1;
  int c0, c1, up;
};

// box `t` of the geometry: sample and first voxel
__device__ __forceinline__ void conv_box(const ConvGeom &G, int t, int &b, int &z0, int &y0,
                                         int &x0) {
  unsigned u = (unsigned)t, q = fdiv(u, G.dnx);
  x0 = (int)(u - q * G.dnx.f.d) * G.bx;
  u = q;
  q = fdiv(u, G.dny);
  y0 = (int)(u - q * G.dny.f.d) * G.by;
  u = q;
  q = fdiv(u, G.dnz);
  z0 = (int)(u - q * G.dnz.f.d) * G.bz;
  b = (int)q;
}

// Stages channels [16 ch0, 16 (ch0 + nch)) of the box at (b, z0, y0, x0) and its halo; zero
// outside the grid and beyond the last channel.  Four entries of four channels per thread in
// flight together.
__device__ __forceinline__ void conv_stage(const ConvGeom &G, const ConvIn &in, int ch0, int nch,
                                           Div1 dq, int b, int z0, int y0, int x0, short *lds) {
  const int Q = nch * 4, total = G.hvol * Q, ct = in.c0 + in.c1, n = G.n, h = n >> 1;
  constexpr int U = 4;
  auto run = [&](auto vec) {
    for (int e0 = threadIdx.x; e0 < total; e0 += U * 256) {
      float4 f[U];
      int dst[U], left[U];  // channels from the entry's first on, 0: nothing there
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * 256;
        const unsigned ec = (unsigned)min(e, total - 1);
        const unsigned pos = fdiv(ec, dq), q = ec - pos * (unsigned)Q;
        const unsigned t = fdiv(pos, G.dhx);
        const int hx = (int)(pos - t * G.dhx.f.d);
        const unsigned hz = fdiv(t, G.dhy);
        const int hy = (int)(t - hz * G.dhy.f.d);
        const int z = z0 + (int)hz - 1, y = y0 + hy - 1, x = x0 + hx - 1;
        const int c = ch0 * 16 + (int)q * 4;
        dst[u] = e < total ? (int)(((q >> 2) * (unsigned)G.hvol + pos) * 16u + (q & 3u) * 4u) : -1;
        const bool live = (unsigned)z < (unsigned)n && (unsigned)y < (unsigned)n &&
                          (unsigned)x < (unsigned)n && c < ct;
        left[u] = live ? ct - c : 0;
        // unconditional loads, of the first values where there is nothing to load: a load in a
        // branch of its own waits for the one before it
        const bool second = live && c >= in.c0;
        const int cs = second ? in.c1 : in.c0, cc = second ? c - in.c0 : c;
        const int sh = in.up && !second ? 1 : 0, m = sh ? h : n;
        const long vox = (((long)b * m + (z >> sh)) * m + (y >> sh)) * m + (x >> sh);
        const float *src = (second ? in.p1 : in.p0) + (live ? vox * cs + cc : 0);
        if (vec) {
          f[u] = *(const float4 *)src;
        } else {  // channel counts that are no multiple of 4 (one source)
          f[u].x = src[0];
          f[u].y = src[left[u] > 1 ? 1 : 0];
          f[u].z = src[left[u] > 2 ? 2 : 0];
          f[u].w = src[left[u] > 3 ? 3 : 0];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (dst[u] >= 0) {
          v4s s;
          s[0] = left[u] > 0 ? bf16_bits(f[u].x) : (short)0;
          s[1] = left[u] > 1 ? bf16_bits(f[u].y) : (short)0;
          s[2] = left[u] > 2 ? bf16_bits(f[u].z) : (short)0;
          s[3] = left[u] > 3 ? bf16_bits(f[u].w) : (short)0;
          *(v4s *)(lds + dst[u]) = s;
        }
    }
  };
  if (((in.c0 | in.c1) & 3) == 0) run(std::true_type());
  else run(std::false_type());
}

// The voxel of every position of the box at (b, z0, y0, x0) and its halo, -1 outside the grid; of
// an upsampled input also the half grid's, behind them.
__device__ __forceinline__ void conv_table(const ConvGeom &G, int up, int b, int z0, int y0,
                                           int x0, int *tab) {
  const int n = G.n, h = n >> 1;
  for (int pos = threadIdx.x; pos < G.hvol; pos += 256) {
    const unsigned t = fdiv((unsigned)pos, G.dhx), hz = fdiv(t, G.dhy);
    const int x = x0 + pos - (int)(t * G.dhx.f.d) - 1, y = y0 + (int)(t - hz * G.dhy.f.d) - 1,
              z = z0 + (int)hz - 1;
    const bool in = (unsigned)z < (unsigned)n && (unsigned)y < (unsigned)n &&
                    (unsigned)x < (unsigned)n;
    tab[pos] = in ? ((b * n + z) * n + y) * n + x : -1;
    if (up) tab[G.hvol + pos] = in ? ((b * h + (z >> 1)) * h + (y >> 1)) * h + (x >> 1) : 0;
  }
}

// conv_stage of all chunks with the voxels from conv_table: several channel quads share a
// position, whose division and multiplications are then formed once (the weight gradients, which
// stage one chunk at a time, are faster without: 74 against 93 us)
__device__ __forceinline__ void conv_stage_table(const ConvGeom &G, const ConvIn &in, int nch,
                                                 Div1 dq, const int *tab, short *lds) {
  const int Q = nch * 4, total = G.hvol * Q, ct = in.c0 + in.c1, hv = in.up ? G.hvol : 0;
  constexpr int U = 4;
  auto run = [&](auto vec) {
    for (int e0 = threadIdx.x; e0 < total; e0 += U * 256) {
      float4 f[U];
      int dst[U], left[U];  // channels from the entry's first on, 0: nothing there
      int vox[U], vup[U];   // read together, without a branch
#pragma unroll
      for (int u = 0; u < U; u++) {
        const unsigned pos = fdiv((unsigned)min(e0 + u * 256, total - 1), dq);
        vox[u] = tab[pos];
        vup[u] = tab[hv + pos];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * 256;
        const unsigned ec = (unsigned)min(e, total - 1);
        const unsigned pos = fdiv(ec, dq), q = ec - pos * (unsigned)Q;
        const int c = (int)q * 4, v = vox[u];
        dst[u] = e < total ? (int)(((q >> 2) * (unsigned)G.hvol + pos) * 16u + (q & 3u) * 4u) : -1;
        const bool live = v >= 0 && c < ct, second = c >= in.c0;
        left[u] = live ? ct - c : 0;
        // unconditional loads, of the first values where there is nothing to load
        const unsigned w = live ? (unsigned)(second ? v : vup[u]) : 0u;
        const unsigned cs = (unsigned)(second ? in.c1 : in.c0),
                       cc = live ? (unsigned)(second ? c - in.c0 : c) : 0u;
        const float *src = (live && second ? in.p1 : in.p0) + (size_t)w * cs + cc;
        if (vec) {
          f[u] = *(const float4 *)src;
        } else {  // channel counts that are no multiple of 4 (one source)
          f[u].x = src[0];
          f[u].y = src[left[u] > 1 ? 1 : 0];
          f[u].z = src[left[u] > 2 ? 2 : 0];
          f[u].w = src[left[u] > 3 ? 3 : 0];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (dst[u] >= 0) {
          v4s s;
          s[0] = left[u] > 0 ? bf16_bits(f[u].x) : (short)0;
          s[1] = left[u] > 1 ? bf16_bits(f[u].y) : (short)0;
          s[2] = left[u] > 2 ? bf16_bits(f[u].z) : (short)0;
          s[3] = left[u] > 3 ? bf16_bits(f[u].w) : (short)0;
          *(v4s *)(lds + dst[u]) = s;
        }
    }
  };
  if (((in.c0 | in.c1) & 3) == 0) run(std::true_type());
  else run(std::false_type());
}

// ---- convolution forward / input gradient (implicit GEMM on MFMA) --------------------

// out[v][o] = bias[o] + sum_t sum_c in[v + off(t) * sgn][c] * W[t][c][o]
// with W as MFMA fragments wf[t][chunk of 16 c][tile of 16 o][lane][4] (k_wfrag).  sgn = +1 for
// the forward convolution; sgn = -1 with the transposed weights' fragments computes the input
// gradient (taps mirrored).  mask (an activation of the output's layout): the result is zero
// where it is <= 0, the ReLU's backward pass.
//
// The weights are the MFMA's row operand and the voxels its column operand, so a lane ends with
// four consecutive channels of one voxel and stores them with one 16-byte access.  A wave holds
// MT x NT tiles of 16 voxels x 16 channels, which share each voxel operand (LDS) and each weight
// fragment (512 contiguous bytes, from L1/L2, fetched a group of iterations ahead).  Products
// accumulate tap by tap and, within a tap, 16 channels at a time in ascending order.
// Batch 32, 32^3, [32 up, 16 skip] -> 16 channels: 178 us, 244 TFLOP/s (227 us without conv_table),
// bound by LDS reads and the staging (2559 us and 215 us for the concatenation as one wave per
// 16 voxels without LDS, which rounded the inputs and fetched single 2-byte weights anew for each
// of the 27 taps).
template <int MT, int NT>
__global__ __launch_bounds__(256) void k_conv(ConvGeom G, ConvIn in, int nch, Div1 dq, int no,
                                              int ntt, const short *__restrict__ wf,
                                              const float *__restrict__ bias,
                                              const float *__restrict__ mask,
                                              float *__restrict__ out, int relu, int sgn,
                                              int wm) {
  extern __shared__ __align__(16) short lds[];
  const int box = (int)xcd_block(blockIdx.x, gridDim.x);
  if (box >= G.nbox) return;  // the whole block
  int b, z0, y0, x0;
  conv_box(G, box, b, z0, y0, x0);
  int *tab = (int *)(lds + (long)nch * G.hvol * 16);
  conv_table(G, in.up, b, z0, y0, x0, tab);
  __syncthreads();
  conv_stage_table(G, in, nch, dq, tab, lds);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int mw = w % wm, nw = w / wm;
  const int hx = (int)G.dhx.f.d, hy = (int)G.dhy.f.d;
  int abase[MT];
  long vout[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int m = (mw * MT + mt) * 16 + i;
    const unsigned mc = (unsigned)(m < G.vol ? m : 0);
    const unsigned t = fdiv(mc, G.dbx);
    const int xx = (int)(mc - t * G.dbx.f.d);
    const unsigned zz = fdiv(t, G.dby);
    const int yy = (int)(t - zz * G.dby.f.d);
    abase[mt] = ((((int)zz + 1) * hy + yy + 1) * hx + xx + 1) * 16 + 4 * g;
    const int z = z0 + (int)zz, y = y0 + yy, x = x0 + xx;
    vout[mt] = m < G.vol && z < G.n && y < G.n && x < G.n
                   ? (((long)b * G.n + z) * G.n + y) * G.n + x
                   : -1;
  }
  v4f acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[mt][t] = (v4f){0.f, 0.f, 0.f, 0.f};
  const int nit = 27 * nch;
  const v4s *wp = (const v4s *)wf + (long)nw * NT * 64 + lane;
  // weight fragments of PF iterations (tap, chunk) are in flight ahead of their use
  constexpr int PF = MT == 1 || NT == 1 ? 9 : 3;  // divides the 27 taps
  // iterations whose voxels are read from LDS together: read one by one, a wave with one tile
  // waits for LDS at every product (one sample of 32^3: convolutions of 10.4..12.9 us, together
  // 9.5..11.0; more weights ahead, or fetched before the staging, gave nothing)
  constexpr int PA = MT == 1 ? 9 : 3;
  static_assert(PF % PA == 0, "a group of weights holds whole groups of voxels");
  v4s bw[PF][NT];
#pragma unroll
  for (int u = 0; u < PF; u++)
#pragma unroll
    for (int t = 0; t < NT; t++) bw[u][t] = wp[((long)min(u, nit - 1) * ntt + t) * 64];
  __syncthreads();
  int tz = -1, ty = -1, tx = -1, ch = 0;  // offset of the tap, channel chunk
  for (int it = 0; it < nit; it += PF) {
#pragma unroll
    for (int u0 = 0; u0 < PF; u0 += PA) {
      v4s a[PA][MT];
#pragma unroll
      for (int u = 0; u < PA; u++) {
        const int off = (((tz * hy + ty) * hx + tx) * sgn + ch * G.hvol) * 16;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) a[u][mt] = *(const v4s *)(lds + abase[mt] + off);
        if (++ch == nch) {
          ch = 0;
          if (++tx == 2) {
            tx = -1;
            if (++ty == 2) {
              ty = -1;
              tz++;
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < PA; u++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int t = 0; t < NT; t++)
            acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bw[u0 + u][t], a[u][mt],
                                                                   acc[mt][t], 0, 0, 0);
        const int nx = min(it + u0 + u + PF, nit - 1);
#pragma unroll
        for (int t = 0; t < NT; t++) bw[u0 + u][t] = wp[((long)nx * ntt + t) * 64];
      }
    }
  }
  // D[4g + q][i]: channel 4g + q of the tile, voxel i
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    if (vout[mt] < 0) continue;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int o = (nw * NT + t) * 16 + 4 * g;
      if ((no & 3) == 0) {
        if (o >= no) continue;
        float4 r = make_float4(acc[mt][t][0], acc[mt][t][1], acc[mt][t][2], acc[mt][t][3]);
        if (bias) {
          r.x += bias[o];
          r.y += bias[o + 1];
          r.z += bias[o + 2];
          r.w += bias[o + 3];
        }
        if (relu) {
          if (r.x < 0.f) r.x = 0.f;
          if (r.y < 0.f) r.y = 0.f;
          if (r.z < 0.f) r.z = 0.f;
          if (r.w < 0.f) r.w = 0.f;
        }
        if (mask) {
          const float4 k = *(const float4 *)(mask + vout[mt] * no + o);
          if (k.x <= 0.f) r.x = 0.f;
          if (k.y <= 0.f) r.y = 0.f;
          if (k.z <= 0.f) r.z = 0.f;
          if (k.w <= 0.f) r.w = 0.f;
        }
        *(float4 *)(out + vout[mt] * no + o) = r;
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if (o + q >= no) continue;
          float r = acc[mt][t][q] + (bias ? bias[o + q] : 0.f);
          if (relu && r < 0.f) r = 0.f;
          if (mask && mask[vout[mt] * no + o + q] <= 0.f) r = 0.f;
          out[vout[mt] * no + o + q] = r;
        }
      }
    }
  }
}

// ---- weight gradients: gW[t][c][o] = sum_v in[v + off(t)][c] * gout[v][o] -------------
// An implicit GEMM on v_mfma_f32_16x16x16bf16_1k: M = 16 input channels, N = output channels,
// K = voxels.  A block takes 16 input channels and every P-th box: it stages the box's inputs
// with their halo as the convolution does and the box's output gradients, both rounded to BF16,
// and accumulates the 16 x co products of all 27 taps in FP32 registers, 7 taps to a wave, over
// its boxes.  The operands need four voxels of one channel per lane while LDS holds 16 channels
// of a voxel: ds_read_tr16 transposes on the way (a lane reads four channels of voxel
// 4g + lane % 16 / 4; it receives channel lane % 16 of voxels 4g .. 4g + 3).  So an input value
// is read from device memory once (2.5 times with its halo) instead of once per tap, and a
// wave's gradient operand serves its seven taps.  The blocks of the first channel chunk also sum
// gout in FP32 (the bias gradient).  Every block writes its sums as a partial
// [block][27 ci co + co]; k_wgrad_reduce adds them in a fixed order.
// Bound by latency: four blocks a CU (128 registers a thread; with three 208 us), whose staging
// loads are issued four at a time and whose seven taps' operands are read together.
// Batch 32, 32^3, 48 x 16 channels: 185 us, 16 x 16 channels 66 (213 and 73 with every staging
// load and every operand waited for by itself; 3592 us with one tap per block, which read the
// inputs 27 times and gathered the operands from LDS two bytes at a time).

constexpr int kWgVox = 256;  // voxels of a box, 16 K steps

typedef __attribute__((address_space(3))) v4s lds_v4s;
__device__ __forceinline__ v4s lds_read_tr(const short *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
}

template <int NTO>
__global__ __launch_bounds__(256, NTO <= 2 ? 4 : 2) void k_conv_wgrad(
    ConvGeom G, ConvIn in, int ncc, int co, const float *__restrict__ gout, int P,
    float *__restrict__ partial) {
  extern __shared__ __align__(16) short lds[];
  constexpr int Q = NTO * 4;
  short *sa = lds;                                // [halo voxel][16]
  short *sg = sa + (long)G.hvol * 16;             // [o tile][voxel of the box][16]
  short *sz = sg + NTO * kWgVox * 16;             // 4 zeros: the input of voxels outside the grid
  float *sb = (float *)(sz + 8);                  // [256][4] bias partial sums
  unsigned short *pt = (unsigned short *)(sb + 1024);  // halo position of a voxel, 0xffff: none
  const int cc = (int)(blockIdx.x % (unsigned)ncc), p = (int)(blockIdx.x / (unsigned)ncc);
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
  const int hx = (int)G.dhx.f.d, hy = (int)G.dhy.f.d, ct = in.c0 + in.c1;
  if (tid < 4) sz[tid] = 0;
  v4f acc[7][NTO];
  int toff[7];
#pragma unroll
  for (int t = 0; t < 7; t++) {
    const int tap = min(w + 4 * t, 26);
    toff[t] = (((tap / 9 - 1) * hy + (tap / 3) % 3 - 1) * hx + tap % 3 - 1) * 16;
#pragma unroll
    for (int k = 0; k < NTO; k++) acc[t][k] = (v4f){0.f, 0.f, 0.f, 0.f};
  }
  float bs[4] = {0.f, 0.f, 0.f, 0.f};
  const Div1 d4 = Div1{FastDiv{4u, 0x80000000u, 1}};  // (n * 2^31 >> 32) >> 1 = n / 4
  for (int box = p; box < G.nbox; box += P) {
    int b, z0, y0, x0;
    conv_box(G, box, b, z0, y0, x0);
    __syncthreads();  // the previous box has been read
    conv_stage(G, in, cc, 1, d4, b, z0, y0, x0, sa);
    // the output gradients: thread tid takes the channels 4 (tid % Q) .. + 3 of every box voxel
    // tid / Q + k 256 / Q
    const int q = tid % Q;
    constexpr int U = 4;  // loads in flight together
    auto run = [&](auto vec) {
      for (int m0 = tid / Q; m0 < kWgVox; m0 += U * (256 / Q)) {
        float4 fr[U];
        int hp[U];  // the voxel's halo position, -1: outside the grid
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int m = m0 + u * (256 / Q);
          const unsigned mc = (unsigned)(m < G.vol ? m : 0), t = fdiv(mc, G.dbx);
          const int xx = (int)(mc - t * G.dbx.f.d);
          const unsigned zz = fdiv(t, G.dby);
          const int yy = (int)(t - zz * G.dby.f.d);
          const int z = z0 + (int)zz, y = y0 + yy, x = x0 + xx;
          const bool ok = m < G.vol && z < G.n && y < G.n && x < G.n;
          const long v = (((long)b * G.n + z) * G.n + y) * G.n + x;
          hp[u] = ok ? (((int)zz + 1) * hy + yy + 1) * hx + xx + 1 : -1;
          const int left = ok ? co - 4 * q : 0;
          const float *src = gout + (left > 0 ? v * co + 4 * q : 0);
          if (vec) {
            fr[u] = *(const float4 *)src;
          } else {
            fr[u].x = src[0];
            fr[u].y = src[left > 1 ? 1 : 0];
            fr[u].z = src[left > 2 ? 2 : 0];
            fr[u].w = src[left > 3 ? 3 : 0];
          }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int m = m0 + u * (256 / Q), left = hp[u] >= 0 ? co - 4 * q : 0;
          const float f[4] = {left > 0 ? fr[u].x : 0.f, left > 1 ? fr[u].y : 0.f,
                              left > 2 ? fr[u].z : 0.f, left > 3 ? fr[u].w : 0.f};
          v4s s;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            bs[j] += f[j];
            s[j] = bf16_bits(f[j]);
          }
          *(v4s *)(sg + ((long)(q >> 2) * kWgVox + m) * 16 + (q & 3) * 4) = s;
          if (q == 0) pt[m] = hp[u] >= 0 ? (unsigned short)hp[u] : (unsigned short)0xffff;
        }
      }
    };
    if ((co & 3) == 0) run(std::true_type());
    else run(std::false_type());
    __syncthreads();
#pragma unroll 2
    for (int ks = 0; ks < kWgVox; ks += 16) {
      const int m = ks + 4 * g + (l16 >> 2);
      const unsigned pos = pt[m];
      const short *ab = sa + (int)pos * 16 + 4 * (l16 & 3);
      v4s bb[NTO];
#pragma unroll
      for (int k = 0; k < NTO; k++)
        bb[k] = lds_read_tr(sg + ((long)k * kWgVox + m) * 16 + 4 * (l16 & 3));
      v4s a[7];
#pragma unroll
      for (int t = 0; t < 7; t++) a[t] = lds_read_tr(pos == 0xffffu ? sz : ab + toff[t]);
      __builtin_amdgcn_sched_barrier(0);  // else each is read when its product needs it
#pragma unroll
      for (int t = 0; t < 7; t++)
#pragma unroll
        for (int k = 0; k < NTO; k++)
          acc[t][k] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[t], bb[k], acc[t][k], 0, 0, 0);
    }
  }
  const long npair = (long)ct * co, stride = 27 * npair + co;
  float *part = partial + (long)p * stride;
  // D[4g + q][l16]: input channel 16 cc + 4g + q, output channel 16 k + l16
#pragma unroll
  for (int t = 0; t < 7; t++) {
    const int tap = w + 4 * t;
    if (tap >= 27) break;
#pragma unroll
    for (int k = 0; k < NTO; k++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int c = cc * 16 + 4 * g + q, o = k * 16 + l16;
        if (c < ct && o < co) part[tap * npair + (long)c * co + o] = acc[t][k][q];
      }
  }
  if (cc == 0) {  // bias: the threads of one channel group summed in thread order
#pragma unroll
    for (int j = 0; j < 4; j++) sb[tid * 4 + j] = bs[j];
    __syncthreads();
    if (tid < co) {
      float s = 0.f;
      for (int k = tid >> 2; k < 256; k += Q) s += sb[k * 4 + (tid & 3)];
      part[27 * npair + tid] = s;
    }
  }
}

// The gradients of all layers from their partials, one launch: grad[off + e] = the sum over the
// layer's P partials in a fixed order (eight consecutive ranges, each in ascending order).
struct WgLayer {
  long part, off;  // first partial value, first gradient value
  int np, P, blk;  // values per partial, partials, first block of the layer
};
struct WgTable {
  WgLayer l[9];
};
constexpr int kWrSeg = 8;

__global__ __launch_bounds__(64 * kWrSeg) void k_wgrad_reduce(WgTable T,
                                                              const float *__restrict__ partial,
                                                              float *__restrict__ grad) {
  __shared__ float s[kWrSeg][64];
  int l = 0;
  while (l < 8 && (int)blockIdx.x >= T.l[l + 1].blk) l++;
  const WgLayer L = T.l[l];
  const int e = ((int)blockIdx.x - L.blk) * 64 + (threadIdx.x & 63), seg = threadIdx.x >> 6;
  const int per = (L.P + kWrSeg - 1) / kWrSeg, c1 = min((seg + 1) * per, L.P);
  float a = 0.f;
  if (e < L.np) {
    const float *q = partial + L.part + e;
    int c = seg * per;
    for (; c + 8 <= c1; c += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = q[(long)(c + u) * L.np];
#pragma unroll
      for (int u = 0; u < 8; u++) a += v[u];
    }
    for (; c < c1; c++) a += q[(long)c * L.np];
  }
  s[seg][threadIdx.x & 63] = a;
  __syncthreads();
  if (seg == 0 && e < L.np) {
    float r = 0.f;
#pragma unroll
    for (int k = 0; k < kWrSeg; k++) r += s[k][threadIdx.x & 63];
    grad[L.off + e] = r;
  }
}

// ---- elementwise / resampling (four channels per thread) -----------------------------------

// voxel v of the grid of n per axis: batch, z, y, x
__device__ __forceinline__ void vox_coords(long v, int n, long &b, int &z, int &y, int &x) {
  long t = v / n;
  x = (int)(v - t * n);
  long u = t / n;
  y = (int)(t - u * n);
  b = u / n;
  z = (int)(u - b * n);
}

// average pool 2x2x2: out (n/2) from in (n), c channels (a multiple of 4)
__global__ void k_pool(int batch, int n, int c, const float *in, float *out) {
  const int h = n / 2, c4 = c / 4;
  const long total = (long)batch * h * h * h * c4;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int k = (int)(e % c4);
  long b;
  int z, y, x;
  vox_coords(e / c4, h, b, z, y, x);
  float4 f[8];
#pragma unroll
  for (int d = 0; d < 8; d++) {
    const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
    f[d] = *(const float4 *)(in + (((b * n + zz) * n + yy) * n + xx) * c + 4 * k);
  }
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int d = 0; d < 8; d++) {
    s.x += f[d].x;
    s.y += f[d].y;
    s.z += f[d].z;
    s.w += f[d].w;
  }
  *(float4 *)(out + e * 4) = make_float4(0.125f * s.x, 0.125f * s.y, 0.125f * s.z, 0.125f * s.w);
}

// gradient of an upsampled layer (n/2, cu) from that of the concatenation (n, cu + cs): the sum
// over the 8 children, zero where the layer's activation is <= 0
__global__ void k_up_bwd(int batch, int n, int cu, int cs, const float *gcat, const float *act,
                         float *gup) {
  const int h = n / 2, c4 = cu / 4;
  const long total = (long)batch * h * h * h * c4;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int k = (int)(e % c4);
  long b;
  int z, y, x;
  vox_coords(e / c4, h, b, z, y, x);
  float4 f[8];
#pragma unroll
  for (int d = 0; d < 8; d++) {
    const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
    f[d] = *(const float4 *)(gcat + (((b * n + zz) * n + yy) * n + xx) * (cu + cs) + 4 * k);
  }
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int d = 0; d < 8; d++) {
    s.x += f[d].x;
    s.y += f[d].y;
    s.z += f[d].z;
    s.w += f[d].w;
  }
  const float4 a = *(const float4 *)(act + e * 4);
  if (a.x <= 0.f) s.x = 0.f;
  if (a.y <= 0.f) s.y = 0.f;
  if (a.z <= 0.f) s.z = 0.f;
  if (a.w <= 0.f) s.w = 0.f;
  *(float4 *)(gup + e * 4) = s;
}

// gradient of a layer that feeds the skip connection and the pool: the skip part of gcat
// (n, cu + cs) plus gpool (n/2, cs) / 8, zero where the layer's activation is <= 0
__global__ void k_skip_bwd(int batch, int n, int cu, int cs, const float *gcat,
                           const float *gpool, const float *act, float *g) {
  const int h = n / 2, c4 = cs / 4;
  const long total = (long)batch * n * n * n * c4;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int k = (int)(e % c4);
  const long v = e / c4;
  long b;
  int z, y, x;
  vox_coords(v, n, b, z, y, x);
  float4 s = *(const float4 *)(gcat + v * (cu + cs) + cu + 4 * k);
  const float4 p = *(const float4 *)(gpool + (((b * h + z / 2) * h + y / 2) * h + x / 2) * cs +
                                     4 * k);
  const float4 a = *(const float4 *)(act + e * 4);
  s.x += 0.125f * p.x;
  s.y += 0.125f * p.y;
  s.z += 0.125f * p.z;
  s.w += 0.125f * p.w;
  if (a.x <= 0.f) s.x = 0.f;
  if (a.y <= 0.f) s.y = 0.f;
  if (a.z <= 0.f) s.z = 0.f;
  if (a.w <= 0.f) s.w = 0.f;
  *(float4 *)(g + e * 4) = s;
}

// MSE: g = 2 (y - t) / m; per-block partial sums of (y - t)^2
__global__ __launch_bounds__(256) void k_mse(long m, const float *y, const float *t, float *g,
                                             double *partial) {
  __shared__ double s[256];
  double acc = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < m; i += (long)gridDim.x * 256) {
    float d = y[i] - t[i];
    g[i] = 2.f * d / (float)m;
    acc += (double)d * d;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// *out = scale * the sum of 256 partials, by pairs
__global__ __launch_bounds__(256) void k_sum_partials(const double *p, double *out, double scale) {
  __shared__ double s[256];
  s[threadIdx.x] = p[threadIdx.x];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0] * scale;
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters
__global__ void k_adam(long np, float *theta, const float *g, float *m, float *v, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.f - b1) * gi;
  float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  theta[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// The BF16 weight fragments of k_conv, all layers in one launch, zero beyond ci and co:
// forward   wf[t][chunk of c][tile of o][lane][j] = W[t][c = 16 chunk + 4 (lane / 16) + j]
//                                                    [o = 16 tile + lane % 16]
// transposed wg[t][chunk of o][tile of c][lane][j] = W[t][c = 16 tile + lane % 16]
//                                                    [o = 16 chunk + 4 (lane / 16) + j]
struct WfLayer {
  long w, f;        // first weight, first fragment value
  int ci, co, blk;  // channels, first block of the layer
};
struct WfTable {
  WfLayer l[9];
};
__global__ __launch_bounds__(256) void k_wfrag(WfTable T, const float *__restrict__ theta,
                                               short *wf, short *wg) {
  int l = 0;
  while (l < 8 && (int)blockIdx.x >= T.l[l + 1].blk) l++;
  const WfLayer L = T.l[l];
  const int nc = (L.ci + 15) / 16, no = (L.co + 15) / 16;
  const int e = ((int)blockIdx.x - L.blk) * 256 + threadIdx.x;
  if (e >= 27 * nc * no * 256) return;
  const int j = e & 3, lane = (e >> 2) & 63, f = e >> 8;
  const int k = 4 * (lane >> 4) + j, i = lane & 15;
  const float *W = theta + L.w;
  {
    const int ot = f % no, ch = (f / no) % nc, t = f / (no * nc), c = ch * 16 + k, o = ot * 16 + i;
    wf[L.f + e] =
        c < L.ci && o < L.co ? bf16_bits(W[((long)t * L.ci + c) * L.co + o]) : (short)0;
  }
  {
    const int tt = f % nc, ch = (f / nc) % no, t = f / (no * nc), c = tt * 16 + i, o = ch * 16 + k;
    wg[L.f + e] =
        c < L.ci && o < L.co ? bf16_bits(W[((long)t * L.ci + c) * L.co + o]) : (short)0;
  }
}

}  // namespace flgpu

// ---- network object ---------------------------------------------------------------------

struct flgpu_unet {
  flgpu_ctx *ctx = nullptr;
  int cin = 2;
  long np = 0;
  long woff[flgpu::NL], boff[flgpu::NL];
  long foff[flgpu::NL];  // first weight fragment value of a layer
  flgpu::WfTable wft;
  unsigned wf_blocks = 0;
  float *theta = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
  short *wf = nullptr, *wg = nullptr;  // BF16 weight fragments (k_wfrag)
  int step = 0;
  // activation storage and launch plans for the current (batch, n)
  int cap_batch = 0, cap_n = 0;
  float *a[flgpu::NL] = {}, *p0 = nullptr, *p1 = nullptr;
  float *g[flgpu::NL] = {}, *gp0 = nullptr, *gp1 = nullptr, *gc1 = nullptr, *gc0 = nullptr;
  float *partial = nullptr;
  flgpu::ConvPlan fwd[flgpu::NL], bwd[flgpu::NL];
  flgpu::ConvGeom wgeom[3];
  flgpu::WgTable wgt;
  unsigned wr_blocks = 0;
  double *lpart = nullptr;
};

namespace flgpu {

flgpu_ctx *unet_ctx(const flgpu_unet *u) { return u->ctx; }

static long vox(int batch, int n) { return (long)batch * n * n * n; }

static int layer_cin(const flgpu_unet *u, int l) { return l == 0 ? u->cin : L_CIN[l]; }
static int tiles16(int c) { return (c + 15) / 16; }

// The box of at most vcap voxels, with at most hcap voxels including its halo, that costs least
// for n voxels per axis: every block costs its vcap voxels of products, also where the box or
// its part inside the grid is smaller, and about 0.3 of that per halo voxel staged.  Extents
// that divide the grid evenly win, so odd grids get boxes of their own.
static ConvGeom conv_geom(int batch, int n, int vcap, int hcap) {
  std::vector<int> ext;
  for (int k = 1; k <= n; k++) {
    const int e = (n + k - 1) / k;
    if (ext.empty() || ext.back() != e) ext.push_back(e);
  }
  double best = -1.0;
  int bz = 1, by = 1, bx = 1;
  for (int ex : ext)
    for (int ey : ext)
      for (int ez : ext) {
        if ((long)ex * ey * ez > vcap) continue;
        const long hv = (long)(ex + 2) * (ey + 2) * (ez + 2);
        if (hv > hcap) continue;
        const double boxes = (double)((n + ex - 1) / ex) * ((n + ey - 1) / ey) * ((n + ez - 1) / ez);
        const double cost = boxes * (vcap + 0.3 * hv);
        if (best < 0.0 || cost < best) {
          best = cost;
          bz = ez;
          by = ey;
          bx = ex;
        }
      }
  ConvGeom G;
  G.n = n;
  G.bz = bz;
  G.by = by;
  G.bx = bx;
  G.vol = bz * by * bx;
  G.hvol = (bz + 2) * (by + 2) * (bx + 2);
  const int nx = (n + bx - 1) / bx, ny = (n + by - 1) / by, nz = (n + bz - 1) / bz;
  const long nbox = (long)batch * nx * ny * nz;
  FLGPU_REQUIRE(nbox < 0x7fffffffL / 27, "too many voxels for the convolution's index range");
  G.nbox = (int)nbox;
  G.dnx = div1(nx);
  G.dny = div1(ny);
  G.dnz = div1(nz);
  G.dbx = div1(bx);
  G.dby = div1(by);
  G.dhx = div1(bx + 2);
  G.dhy = div1(by + 2);
  return G;
}

// bytes of LDS per block: two blocks fit a CU's 160 KB
constexpr int kConvLds = 80 * 1024;

// How a convolution with nch chunks of input channels and ntt tiles of output channels is
// split: four waves share a box, wm of them along its voxels and 4 / wm along its channel tiles.
// A wave with more voxel tiles (mt) reuses a weight fragment more often, so the largest mt is
// taken that still gives every CU two blocks; grids too small for that (one sample: 64 boxes
// of 64 voxels at 16^3, 8 at 8^3) are split further, over the channel tiles too.
static ConvPlan conv_plan(const flgpu_unet *u, int batch, int n, int nch, int ntt) {
  const int hcap = kConvLds / (32 * nch), cus = u->ctx->cus;
  ConvPlan p;
  for (p.mt = 4; p.mt >= 1; p.mt /= 2) {
    if (p.mt * ntt > 16 && p.mt > 1) continue;  // registers of the accumulators
    p.wm = 4;
    p.nt = ntt;
    p.g = conv_geom(batch, n, 64 * p.mt, hcap);
    if (p.g.nbox >= 2 * cus || p.mt == 1) break;
  }
  while (p.mt == 1 && p.g.nbox < cus && p.wm > 1 && p.nt % 2 == 0) {
    p.wm /= 2;
    p.nt /= 2;
    p.g = conv_geom(batch, n, 16 * p.wm, hcap);
  }
  p.nch = nch;
  p.ntt = ntt;
  return p;
}

static void unet_free_acts(flgpu_unet *u) {
  for (int l = 0; l < NL; l++) {
    dev_free(u->a[l]);
    dev_free(u->g[l]);
    u->a[l] = u->g[l] = nullptr;
  }
  for (float **p : {&u->p0, &u->p1, &u->gp0, &u->gp1, &u->gc1, &u->gc0, &u->partial}) {
    dev_free(*p);
    *p = nullptr;
  }
  u->cap_batch = u->cap_n = 0;
}

static void unet_alloc_acts(flgpu_unet *u, int batch, int n, bool train) {
  if (u->cap_batch == batch && u->cap_n == n && (!train || u->g[0])) return;
  unet_free_acts(u);
  int nl[3] = {n, n / 2, n / 4};
  auto fa = [](long cnt) { return (float *)dev_alloc(sizeof(float) * cnt); };
  for (int l = 0; l < NL; l++) {
    const int nn = nl[L_LEVEL[l]], ci = tiles16(layer_cin(u, l)), co = tiles16(L_COUT[l]);
    u->fwd[l] = conv_plan(u, batch, nn, ci, co);
    u->bwd[l] = conv_plan(u, batch, nn, co, ci);
    u->a[l] = fa(vox(batch, nn) * L_COUT[l]);
  }
  u->p0 = fa(vox(batch, nl[1]) * 16);
  u->p1 = fa(vox(batch, nl[2]) * 32);
  if (train) {
    for (int l = 0; l < NL; l++) u->g[l] = fa(vox(batch, nl[L_LEVEL[l]]) * L_COUT[l]);
    u->gp0 = fa(vox(batch, nl[1]) * 16);
    u->gp1 = fa(vox(batch, nl[2]) * 32);
    u->gc1 = fa(vox(batch, nl[1]) * 96);
    u->gc0 = fa(vox(batch, nl[0]) * 48);
    for (int k = 0; k < 3; k++)
      u->wgeom[k] = conv_geom(batch, nl[k], kWgVox, kConvLds / 64);
    // P blocks per chunk of input channels: about four blocks per CU (two: 2197 us for a
    // batch of 32 x 32^3 instead of 1999), all with the same number
    // of boxes but for the last few
    long off = 0;
    int blk = 0;
    for (int l = 0; l < NL; l++) {
      const int nbox = u->wgeom[L_LEVEL[l]].nbox, ncc = tiles16(layer_cin(u, l));
      const int pmax = std::max(1, std::min(nbox, 4 * u->ctx->cus / ncc));
      const int per = (nbox + pmax - 1) / pmax;
      WgLayer &W = u->wgt.l[l];
      W.P = (nbox + per - 1) / per;
      W.np = 27 * layer_cin(u, l) * L_COUT[l] + L_COUT[l];
      W.part = off;
      W.off = u->woff[l];
      W.blk = blk;
      off += (long)W.P * W.np;
      blk += (W.np + 63) / 64;
    }
    u->partial = fa(off);
    u->wr_blocks = (unsigned)blk;
  }
  u->cap_batch = batch;
  u->cap_n = n;
}

template <int MT, int NT>
static void conv_launch(flgpu_unet *u, const ConvPlan &p, const ConvIn &in, int no,
                        const short *wf, const float *bias, const float *mask, float *out,
                        int relu, int sgn) {
  const size_t lds = (size_t)p.g.hvol * (p.nch * 32 + (in.up ? 8 : 4));
  if (lds > 64 * 1024)
    FLGPU_HIP(hipFuncSetAttribute((const void *)k_conv<MT, NT>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_conv<MT, NT><<<xcd_grid(p.g.nbox), 256, lds, u->ctx->stream>>>(
      p.g, in, p.nch, div1(p.nch * 4), no, p.ntt, wf, bias, mask, out, relu, sgn, p.wm);
  FLGPU_HIP(hipGetLastError());
}

static void conv_run(flgpu_unet *u, const ConvPlan &p, const ConvIn &in, int no, const short *wf,
                     const float *bias, const float *mask, float *out, int relu, int sgn) {
#define FLGPU_CONV(MT, NT)                                                     \
  if (p.mt == MT && p.nt == NT) {                                              \
    conv_launch<MT, NT>(u, p, in, no, wf, bias, mask, out, relu, sgn);         \
    return;                                                                    \
  }
  FLGPU_CONV(4, 1)
  FLGPU_CONV(4, 2)
  FLGPU_CONV(4, 3)
  FLGPU_CONV(4, 4)
  FLGPU_CONV(2, 1)
  FLGPU_CONV(2, 2)
  FLGPU_CONV(2, 3)
  FLGPU_CONV(2, 4)
  FLGPU_CONV(2, 6)
  FLGPU_CONV(1, 1)
  FLGPU_CONV(1, 2)
  FLGPU_CONV(1, 3)
  FLGPU_CONV(1, 4)
  FLGPU_CONV(1, 6)
#undef FLGPU_CONV
  FLGPU_REQUIRE(false, "no convolution kernel for this layer");
}

// out = relu(conv(in) + bias) of layer l
static void conv(flgpu_unet *u, int l, const ConvIn &in, float *out, int relu) {
  conv_run(u, u->fwd[l], in, L_COUT[l], u->wf + u->foff[l], u->theta + u->boff[l], nullptr, out,
           relu, 1);
}

// gin = conv^T(gout) through the transposed weights (taps mirrored), zero where mask <= 0
static void conv_gin(flgpu_unet *u, int l, const float *gout, const float *mask, float *gin) {
  const ConvIn in = {gout, nullptr, L_COUT[l], 0, 0};
  conv_run(u, u->bwd[l], in, layer_cin(u, l), u->wg + u->foff[l], nullptr, mask, gin, 0, -1);
}

// the partial sums of layer l's weight and bias gradients
static void conv_wgrad(flgpu_unet *u, int l, const ConvIn &in, const float *gout) {
  const ConvGeom &G = u->wgeom[L_LEVEL[l]];
  const WgLayer &W = u->wgt.l[l];
  const int co = L_COUT[l], nto = tiles16(co), ncc = tiles16(in.c0 + in.c1);
  const size_t lds = (size_t)G.hvol * 32 + (size_t)nto * kWgVox * 32 + 16 + 4096 + kWgVox * 2;
  const unsigned grid = (unsigned)(W.P * ncc);
  float *part = u->partial + W.part;
  hipStream_t s = u->ctx->stream;
  auto launch = [&](auto kern) {
    if (lds > 64 * 1024)
      FLGPU_HIP(hipFuncSetAttribute((const void *)kern,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kern<<<grid, 256, lds, s>>>(G, in, ncc, co, gout, W.P, part);
    FLGPU_HIP(hipGetLastError());
  };
  switch (nto) {
    case 1: launch(k_conv_wgrad<1>); break;
    case 2: launch(k_conv_wgrad<2>); break;
    case 4: launch(k_conv_wgrad<4>); break;
    default: FLGPU_REQUIRE(false, "no weight-gradient kernel for this layer");
  }
}

static void refresh_bf16(flgpu_unet *u) {
  k_wfrag<<<u->wf_blocks, 256, 0, u->ctx->stream>>>(u->wft, u->theta, u->wf, u->wg);
  FLGPU_HIP(hipGetLastError());
}

static unsigned ew(long m) { return grid_for(m, 256); }

// the decoder's inputs [upsampled, skip] and the plain ones
static ConvIn conv_in(const float *p, int c) { return ConvIn{p, nullptr, c, 0, 0}; }
static ConvIn conv_cat(const float *up, int cu, const float *skip, int cs) {
  return ConvIn{up, skip, cu, cs, 1};
}

// y: the network's output (FP32, batch n^3 values)
void unet_forward(flgpu_unet *u, int batch, int n, const float *x, float *y) {
  hipStream_t s = u->ctx->stream;
  int nl[3] = {n, n / 2, n / 4};
  conv(u, 0, conv_in(x, u->cin), u->a[0], 1);
  conv(u, 1, conv_in(u->a[0], 16), u->a[1], 1);
  k_pool<<<ew(vox(batch, nl[1]) * 4), 256, 0, s>>>(batch, n, 16, u->a[1], u->p0);
  conv(u, 2, conv_in(u->p0, 16), u->a[2], 1);
  conv(u, 3, conv_in(u->a[2], 32), u->a[3], 1);
  k_pool<<<ew(vox(batch, nl[2]) * 8), 256, 0, s>>>(batch, nl[1], 32, u->a[3], u->p1);
  conv(u, 4, conv_in(u->p1, 32), u->a[4], 1);
  conv(u, 5, conv_in(u->a[4], 64), u->a[5], 1);
  conv(u, 6, conv_cat(u->a[5], 64, u->a[3], 32), u->a[6], 1);
  conv(u, 7, conv_cat(u->a[6], 32, u->a[1], 16), u->a[7], 1);
  conv(u, 8, conv_in(u->a[7], 16), y, 0);
  FLGPU_HIP(hipGetLastError());
}

// loss (device slot) and gradients of all parameters into u->grad
void unet_backward(flgpu_unet *u, int batch, int n, const float *x, const float *t) {
  hipStream_t s = u->ctx->stream;
  int nl[3] = {n, n / 2, n / 4};
  long v0 = vox(batch, n), v1 = vox(batch, nl[1]), v2 = vox(batch, nl[2]);
  k_mse<<<256, 256, 0, s>>>(v0, u->a[8], t, u->g[8], u->lpart);
  k_sum_partials<<<1, 256, 0, s>>>(u->lpart, u->ctx->red_out + 8, 1.0 / (double)v0);
  conv_wgrad(u, 8, conv_in(u->a[7], 16), u->g[8]);
  conv_gin(u, 8, u->g[8], u->a[7], u->g[7]);
  conv_wgrad(u, 7, conv_cat(u->a[6], 32, u->a[1], 16), u->g[7]);
  conv_gin(u, 7, u->g[7], nullptr, u->gc0);
  k_up_bwd<<<ew(v1 * 8), 256, 0, s>>>(batch, n, 32, 16, u->gc0, u->a[6], u->g[6]);
  conv_wgrad(u, 6, conv_cat(u->a[5], 64, u->a[3], 32), u->g[6]);
  conv_gin(u, 6, u->g[6], nullptr, u->gc1);
  k_up_bwd<<<ew(v2 * 16), 256, 0, s>>>(batch, nl[1], 64, 32, u->gc1, u->a[5], u->g[5]);
  conv_wgrad(u, 5, conv_in(u->a[4], 64), u->g[5]);
  conv_gin(u, 5, u->g[5], u->a[4], u->g[4]);
  conv_wgrad(u, 4, conv_in(u->p1, 32), u->g[4]);
  conv_gin(u, 4, u->g[4], nullptr, u->gp1);
  // a3 feeds the pool and the skip: gradients add
  k_skip_bwd<<<ew(v1 * 8), 256, 0, s>>>(batch, nl[1], 64, 32, u->gc1, u->gp1, u->a[3], u->g[3]);
  conv_wgrad(u, 3, conv_in(u->a[2], 32), u->g[3]);
  conv_gin(u, 3, u->g[3], u->a[2], u->g[2]);
  conv_wgrad(u, 2, conv_in(u->p0, 16), u->g[2]);
  conv_gin(u, 2, u->g[2], nullptr, u->gp0);
  k_skip_bwd<<<ew(v0 * 4), 256, 0, s>>>(batch, n, 32, 16, u->gc0, u->gp0, u->a[1], u->g[1]);
  conv_wgrad(u, 1, conv_in(u->a[0], 16), u->g[1]);
  conv_gin(u, 1, u->g[1], u->a[0], u->g[0]);
  conv_wgrad(u, 0, conv_in(x, u->cin), u->g[0]);
  k_wgrad_reduce<<<u->wr_blocks, 64 * kWrSeg, 0, s>>>(u->wgt, u->partial, u->grad);
  FLGPU_HIP(hipGetLastError());
}

// Standard normal values from 64-bit random words by Marsaglia's polar method (1964), in the
// sequence std::normal_distribution<double> gives over std::mt19937_64, so a seed keeps its
// weights.  The library's version takes two long double logarithms per word to find how many
// words a double needs (one), 12 to 21 ms for a network; this takes 4.
struct Normal {
  std::mt19937_64 rng;
  bool saved = false;
  double save = 0.0;
  explicit Normal(unsigned long seed) : rng(seed) {}
  double canonical() {
    const double u = (double)rng() / 18446744073709551616.0;
    return u >= 1.0 ? std::nextafter(1.0, 0.0) : u;
  }
  void reset() { saved = false; }
  double next() {
    if (saved) {
      saved = false;
      return save;
    }
    double x, y, r2;
    do {
      x = 2.0 * canonical() - 1.0;
      y = 2.0 * canonical() - 1.0;
      r2 = x * x + y * y;
    } while (r2 > 1.0 || r2 == 0.0);
    const double m = std::sqrt(-2.0 * std::log(r2) / r2);
    save = x * m;
    saved = true;
    return y * m;
  }
};

// He-normal weights for the ReLU layers (a tenth of that for the output layer), zero biases
static std::vector<float> initial_parameters(int cin, unsigned long seed) {
  std::vector<float> h;
  Normal nd(seed);
  for (int l = 0; l < NL; l++) {
    const int ci = l == 0 ? cin : L_CIN[l], co = L_COUT[l];
    const long nw = 27L * ci * co;
    const double sd = std::sqrt(2.0 / (27.0 * ci));
    nd.reset();  // each layer has a distribution of its own
    h.reserve(h.size() + nw + co);
    for (long i = 0; i < nw; i++) {
      const double v = nd.next() * sd;
      h.push_back((float)(l == NL - 1 ? 0.1 * v : v));
    }
    h.insert(h.end(), co, 0.f);
  }
  return h;
}

static void check_shape(const flgpu_unet *u, const flgpu_vec *vec, int batch, int n, int ch,
                        const char *what) {
  FLGPU_REQUIRE(vec && vec->ctx == u->ctx, std::string(what) + " missing or of another context");
  FLGPU_REQUIRE(vec->prec == FLGPU_F32, std::string(what) + " must be an FP32 vector");
  FLGPU_REQUIRE(vec->n == vox(batch, n) * ch, std::string(what) + " has the wrong length");
}

}  // namespace flgpu

using namespace flgpu;

extern "C" int flgpu_unet_create(flgpu_ctx *ctx, int cin, unsigned long seed, flgpu_unet **out) {
  return guard([&] {
    FLGPU_REQUIRE(ctx && out, "arguments must not be NULL");
    FLGPU_REQUIRE(cin >= 1 && cin <= 16, "cin must be in 1..16");
    CTX_LOCK(ctx);
    flgpu_unet *u = new flgpu_unet;
    u->ctx = ctx;
    u->cin = cin;
    const std::vector<float> h = initial_parameters(cin, seed);
    long off = 0;
    for (int l = 0; l < NL; l++) {
      u->woff[l] = off;
      u->boff[l] = off + 27L * layer_cin(u, l) * L_COUT[l];
      off = u->boff[l] + L_COUT[l];
    }
    u->np = off;
    long fo = 0;
    for (int l = 0; l < NL; l++) {
      const int ci = layer_cin(u, l), co = L_COUT[l], nf = 27 * tiles16(ci) * tiles16(co);
      u->foff[l] = fo;
      u->wft.l[l] = WfLayer{u->woff[l], fo, ci, co, (int)u->wf_blocks};
      u->wf_blocks += nf;
      fo += 256L * nf;
    }
    u->theta = (float *)dev_alloc(sizeof(float) * off);
    u->m = (float *)dev_alloc(sizeof(float) * off);
    u->v = (float *)dev_alloc(sizeof(float) * off);
    u->grad = (float *)dev_alloc(sizeof(float) * off);
    u->wf = (short *)dev_alloc(sizeof(short) * fo);
    u->wg = (short *)dev_alloc(sizeof(short) * fo);
    u->lpart = (double *)dev_alloc(sizeof(double) * 256);
    FLGPU_HIP(hipMemcpyAsync(u->theta, h.data(), sizeof(float) * off, hipMemcpyHostToDevice,
                             ctx->stream));
    vfill(ctx, off, FLGPU_F32, u->m, 0.0);
    vfill(ctx, off, FLGPU_F32, u->v, 0.0);
    vfill(ctx, off, FLGPU_F32, u->grad, 0.0);
    refresh_bf16(u);
    FLGPU_HIP(hipStreamSynchronize(ctx->stream));
    *out = u;
    return 0;
  });
}

extern "C" int flgpu_unet_destroy(flgpu_unet *u) {
  return guard([&] {
    if (!u) return 0;
    CTX_LOCK(u->ctx);
    FLGPU_HIP(hipStreamSynchronize(u->ctx->stream));
    unet_free_acts(u);
    for (void *p : {(void *)u->theta, (void *)u->m, (void *)u->v, (void *)u->grad, (void *)u->wf,
                    (void *)u->wg, (void *)u->lpart})
      dev_free(p);
    delete u;
    return 0;
  });
}

extern "C" int flgpu_unet_nparams(const flgpu_unet *u, long *np) {
  return guard([&] {
    FLGPU_REQUIRE(u && np, "arguments must not be NULL");
    *np = u->np;
    return 0;
  });
}

// parameters (and Adam state) as doubles: checkpoint / restore
extern "C" int flgpu_unet_get_params(const flgpu_unet *u, double *theta, double *m, double *v,
                                     int *step) {
  return guard([&] {
    FLGPU_REQUIRE(u, "network must not be NULL");
    CTX_LOCK(u->ctx);
    std::vector<float> h(u->np);
    const float *src[3] = {u->theta, u->m, u->v};
    double *dst[3] = {theta, m, v};
    for (int k = 0; k < 3; k++) {
      if (!dst[k]) continue;
      FLGPU_HIP(hipMemcpy(h.data(), src[k], sizeof(float) * u->np, hipMemcpyDeviceToHost));
      for (long i = 0; i < u->np; i++) dst[k][i] = h[i];
    }
    if (step) *step = u->step;
    return 0;
  });
}

extern "C" int flgpu_unet_set_params(flgpu_unet *u, const double *theta, const double *m,
                                     const double *v, int step) {
  return guard([&] {
    FLGPU_REQUIRE(u && theta, "network and theta must not be NULL");
    CTX_LOCK(u->ctx);
    FLGPU_HIP(hipStreamSynchronize(u->ctx->stream));
    std::vector<float> h(u->np);
    const double *src[3] = {theta, m, v};
    float *dst[3] = {u->theta, u->m, u->v};
    for (int k = 0; k < 3; k++) {
      if (src[k]) {
        for (long i = 0; i < u->np; i++) h[i] = (float)src[k][i];
        FLGPU_HIP(hipMemcpy(dst[k], h.data(), sizeof(float) * u->np, hipMemcpyHostToDevice));
      } else if (k > 0) {
        vfill(u->ctx, u->np, FLGPU_F32, dst[k], 0.0);
      }
    }
    u->step = step;
    refresh_bf16(u);
    FLGPU_HIP(hipStreamSynchronize(u->ctx->stream));
    return 0;
  });
}

extern "C" int flgpu_unet_forward(flgpu_unet *u, int batch, int n, const flgpu_vec *x,
                                  flgpu_vec *y) {
  return guard([&] {
    FLGPU_REQUIRE(u, "network must not be NULL");
    FLGPU_REQUIRE(batch >= 1 && n >= 4 && n % 4 == 0, "n must be a multiple of 4");
    check_shape(u, x, batch, n, u->cin, "x");
    check_shape(u, y, batch, n, 1, "y");
    CTX_LOCK(u->ctx);
    unet_alloc_acts(u, batch, n, false);
    unet_forward(u, batch, n, (const float *)x->d, (float *)y->d);
    return 0;
  });
}

// loss and gradient without an update (gradient check)
extern "C" int flgpu_unet_loss_grad(flgpu_unet *u, int batch, int n, const flgpu_vec *x,
                                    const flgpu_vec *t, double *loss, double *grad) {
  return guard([&] {
    FLGPU_REQUIRE(u && loss, "arguments must not be NULL");
    FLGPU_REQUIRE(batch >= 1 && n >= 4 && n % 4 == 0, "n must be a multiple of 4");
    check_shape(u, x, batch, n, u->cin, "x");
    check_shape(u, t, batch, n, 1, "t");
    CTX_LOCK(u->ctx);
    unet_alloc_acts(u, batch, n, true);
    unet_forward(u, batch, n, (const float *)x->d, u->a[8]);
    unet_backward(u, batch, n, (const float *)x->d, (const float *)t->d);
    fetch_slots(u->ctx, 9);
    *loss = u->ctx->host_out[8];
    if (grad) {
      std::vector<float> h(u->np);
      FLGPU_HIP(hipMemcpy(h.data(), u->grad, sizeof(float) * u->np, hipMemcpyDeviceToHost));
      for (long i = 0; i < u->np; i++) grad[i] = h[i];
    }
    return 0;
  });
}

// one Adam training step on a batch: returns the batch loss before the update
extern "C" int flgpu_unet_train_step(flgpu_unet *u, int batch, int n, const flgpu_vec *x,
                                     const flgpu_vec *t, double lr, double *loss) {
  return guard([&] {
    FLGPU_REQUIRE(u, "network must not be NULL");
    FLGPU_REQUIRE(batch >= 1 && n >= 4 && n % 4 == 0, "n must be a multiple of 4");
    check_shape(u, x, batch, n, u->cin, "x");
    check_shape(u, t, batch, n, 1, "t");
    CTX_LOCK(u->ctx);
    unet_alloc_acts(u, batch, n, true);
    unet_forward(u, batch, n, (const float *)x->d, u->a[8]);
    unet_backward(u, batch, n, (const float *)x->d, (const float *)t->d);
    u->step += 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float c1 = 1.f - std::pow(b1, (float)u->step), c2 = 1.f - std::pow(b2, (float)u->step);
    k_adam<<<grid_for(u->np, 256), 256, 0, u->ctx->stream>>>(u->np, u->theta, u->grad, u->m, u->v,
                                                             (float)lr, b1, b2, eps, c1, c2);
    FLGPU_HIP(hipGetLastError());
    refresh_bf16(u);
    if (loss) {
      fetch_slots(u->ctx, 9);
      *loss = u->ctx->host_out[8];
    }
    return 0;
  });
}

// ---- lattice <-> network grid -------------------------------------------------------------

namespace flgpu {

// network input of sample s: channel 0 = r / rms(r) on nodes (z,y,x) < n of
// the (n+1)^3 lattice, channel 1 = log(kappa) / 4 of the cell with that lower
// corner (0 without kappa).  rms from the dot in *ss: sqrt(ss / n^3).
template <class T>
__global__ void k_pack(int n, const T *__restrict__ r, const double *__restrict__ kappa,
                       const double *ss, float *x, long sample) {
  long nv = (long)n * n * n;
  long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  int xx = (int)(v % n), yy = (int)((v / n) % n), zz = (int)(v / ((long)n * n));
  long idx = ((long)zz * (n + 1) + yy) * (n + 1) + xx;
  double rms = sqrt(*ss / (double)nv);
  double inv = rms > 0.0 ? 1.0 / rms : 0.0;
  float *o = x + (sample * nv + v) * 2;
  o[0] = (float)((double)r[idx] * inv);
  o[1] = kappa ? (float)(log(kappa[v]) * 0.25) : 0.f;
}

// target of sample s: e / rms(e) on the network grid
__global__ void k_pack_target(int n, const double *__restrict__ e, const double *ss, float *t,
                              long sample) {
  long nv = (long)n * n * n;
  long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  int xx = (int)(v % n), yy = (int)((v / n) % n), zz = (int)(v / ((long)n * n));
  long idx = ((long)zz * (n + 1) + yy) * (n + 1) + xx;
  double rms = sqrt(*ss / (double)nv);
  t[sample * nv + v] = (float)(rms > 0.0 ? e[idx] / rms : 0.0);
}

// lattice vector from the network output (zero on Dirichlet nodes)
template <class T>
__global__ void k_unpack(int n, const float *__restrict__ y, T *q) {
  long M = n + 1;
  long N = M * M * M;
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  int xx = (int)(idx % M), yy = (int)((idx / M) % M), zz = (int)(idx / (M * M));
  bool interior = xx > 0 && yy > 0 && zz > 0 && xx < n && yy < n && zz < n;
  q[idx] = interior ? (T)y[((long)zz * n + yy) * n + xx] : (T)0;
}

// q += beta c with beta = (c . r1) / (c . A c), the energy-optimal step along c, when that step
// adds at least min_gain of the energy of the cycle's own step: (c . r1)^2 / (c . A c) >=
// min_gain (z1 . r).  d = {c . r1, c . A c, z1 . r}; *flag = 1 when added, else 0.
template <class T>
__global__ void k_add_opt(long N, const double *__restrict__ d, double min_gain, double *flag,
                          const T *c, T *q) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const double num = d[0], den = d[1], zr = d[2];
  const bool add = den > 0.0 && zr > 0.0 && num * num / den >= min_gain * zr;
  if (i == 0) *flag = add ? 1.0 : 0.0;
  if (i >= N || !add) return;
  const T beta = (T)(num / den);
  q[i] += beta * c[i];
}

// The network's correction inside flexible CG.  After the V-cycle z1 = q, the residual
// r1 = r - A z1 is taken to the level the network runs on (the cycle's own restrictions, in
// the cycle's precision), the network maps it to an error estimate there, the cycle's
// prolongations bring that back (c), and q += beta c with the energy-optimal beta, when that
// step carries enough energy (k_add_opt).  On the top level this is z = z1 + beta N(r1).
struct UnetHook : LearnedHook {
  flgpu_ctx *ctx;
  flgpu_mg *mg;
  const flgpu_mat *A;
  flgpu_unet *u;
  const flgpu_vec *kappa;
  int n, lc, top, mprec;
  long N;
  int prec;
  void *r1 = nullptr, *c = nullptr, *Ac = nullptr;
  std::vector<void *> lv;  // levels lc..top in the cycle's precision (below the top)
  float *xin = nullptr;
  ~UnetHook() override {
    dev_free(r1);
    dev_free(c);
    dev_free(Ac);
    for (void *p : lv) dev_free(p);
    dev_free(xin);
  }
  void correct(void *r, void *q, double min_gain, int flag) override {
    hipStream_t s = ctx->stream;
    FLGPU_REQUIRE(prec == FLGPU_F64, "the learned correction runs inside an FP64 outer iteration");
    spmv(A, -1.0, q, 1.0, r, r1);
    long nv = (long)n * n * n;
    const double *kd = kappa ? (const double *)kappa->d : nullptr;
    unet_alloc_acts(u, 1, n, false);
    if (lc == top) {
      vdot_dev(ctx, N, prec, r1, r1, 10);
      k_pack<double><<<grid_for(nv, 256), 256, 0, s>>>(n, (const double *)r1, kd,
                                                       ctx->red_out + 10, xin, 0);
      unet_forward(u, 1, n, xin, u->a[8]);
      k_unpack<double><<<grid_for(N, 256), 256, 0, s>>>(n, u->a[8], (double *)c);
    } else {
      vcopy(ctx, N, FLGPU_F64, r1, mprec, lv[top - lc]);
      for (int l = top; l > lc; l--) mg_restrict(mg, l, lv[l - lc], lv[l - 1 - lc]);
      long Nc = mg_level_rows(mg, lc);
      vdot_dev(ctx, Nc, mprec, lv[0], lv[0], 10);
      if (mprec == FLGPU_F64)
        k_pack<double><<<grid_for(nv, 256), 256, 0, s>>>(n, (const double *)lv[0], kd,
                                                         ctx->red_out + 10, xin, 0);
      else
        k_pack<float><<<grid_for(nv, 256), 256, 0, s>>>(n, (const float *)lv[0], kd,
                                                        ctx->red_out + 10, xin, 0);
      unet_forward(u, 1, n, xin, u->a[8]);
      if (mprec == FLGPU_F64)
        k_unpack<double><<<grid_for(Nc, 256), 256, 0, s>>>(n, u->a[8], (double *)lv[0]);
      else
        k_unpack<float><<<grid_for(Nc, 256), 256, 0, s>>>(n, u->a[8], (float *)lv[0]);
      for (int l = lc + 1; l <= top; l++) mg_prolong(mg, l, lv[l - 1 - lc], lv[l - lc]);
      vcopy(ctx, N, mprec, lv[top - lc], FLGPU_F64, c);
    }
    spmv(A, 1.0, c, 0.0, Ac, Ac);
    {  // c . r1, c . A c and the cycle step's z1 . r, one pass
      const void *dx[3] = {c, c, q}, *dy[3] = {r1, Ac, r};
      const int slots[3] = {11, 12, 13};
      vdot_multi_dev(ctx, N, prec, dx, dy, slots);
    }
    k_add_opt<double><<<grid_for(N, 256), 256, 0, s>>>(N, ctx->red_out + 11, min_gain,
                                                       ctx->red_out + flag, (const double *)c,
                                                       (double *)q);
    FLGPU_HIP(hipGetLastError());
  }
};

std::unique_ptr<LearnedHook> learned_hook(flgpu_mg *mg, const flgpu_mat *A) {
  FLGPU_REQUIRE(mg, "the learned correction needs a hierarchy");
  flgpu_unet *u;
  const flgpu_vec *kappa;
  int n;
  mg_unet(mg, &u, &kappa, &n);
  FLGPU_REQUIRE(u, "no learned network is attached to the hierarchy (flgpu_mg_attach_unet)");
  FLGPU_REQUIRE(n % 4 == 0, "the network grid needs n divisible by 4");
  std::unique_ptr<UnetHook> h(new UnetHook);
  h->ctx = A->ctx;
  h->mg = mg;
  h->A = A;
  h->u = u;
  h->kappa = kappa;
  h->n = n;
  h->N = A->nrows;
  h->prec = A->prec;
  h->lc = mg_level_cells(mg, n);
  h->top = mg_top_level(mg);
  h->mprec = mg_precision(mg);
  FLGPU_REQUIRE(h->lc >= 0, "the network's grid is no level of the hierarchy");
  FLGPU_REQUIRE(mg_level_rows(mg, h->lc) == (long)(n + 1) * (n + 1) * (n + 1),
                "the network's level is not a 3D Q1 lattice of n cells per axis");
  FLGPU_REQUIRE(mg_level_rows(mg, h->top) == h->N, "A does not match the hierarchy");
  size_t b = prec_bytes(A->prec) * h->N;
  h->r1 = dev_alloc(b);
  h->c = dev_alloc(b);
  h->Ac = dev_alloc(b);
  if (h->lc < h->top)
    for (int l = h->lc; l <= h->top; l++)
      h->lv.push_back(dev_alloc(prec_bytes(h->mprec) * mg_level_rows(mg, l)));
  h->xin = (float *)dev_alloc(sizeof(float) * 2 * (long)n * n * n);
  return std::unique_ptr<LearnedHook>(h.release());
}

}  // namespace flgpu

extern "C" int flgpu_unet_pack(const flgpu_vec *r, const flgpu_vec *kappa, int n, flgpu_vec *x,
                               long sample, int target) {
  return guard([&] {
    FLGPU_REQUIRE(r && x, "arguments must not be NULL");
    FLGPU_REQUIRE(r->prec == FLGPU_F64 && r->n == (long)(n + 1) * (n + 1) * (n + 1),
                  "r must be an FP64 lattice vector of (n+1)^3 values");
    FLGPU_REQUIRE(!kappa || (kappa->prec == FLGPU_F64 && kappa->n == (long)n * n * n),
                  "kappa must be an FP64 vector of n^3 cell values");
    long nv = (long)n * n * n;
    int ch = target ? 1 : 2;
    FLGPU_REQUIRE(x->prec == FLGPU_F32 && sample >= 0 && (sample + 1) * nv * ch <= x->n,
                  "x too small for this sample");
    flgpu_ctx *ctx = r->ctx;
    CTX_LOCK(ctx);
    vdot_dev(ctx, r->n, FLGPU_F64, r->d, r->d, 14);
    if (target)
      k_pack_target<<<grid_for(nv, 256), 256, 0, ctx->stream>>>(n, (const double *)r->d,
                                                                ctx->red_out + 14, (float *)x->d,
                                                                sample);
    else
      k_pack<double><<<grid_for(nv, 256), 256, 0, ctx->stream>>>(
          n, (const double *)r->d, kappa ? (const double *)kappa->d : nullptr, ctx->red_out + 14,
          (float *)x->d, sample);
    FLGPU_HIP(hipGetLastError());
    return 0;
  });
}

// dst[k] = src rows idx[k] (rows of row_len values), k = 0..count-1
extern "C" int flgpu_vec_gather_rows(const flgpu_vec *src, long row_len, const long *idx,
                                     int count, flgpu_vec *dst) {
  return guard([&] {
    FLGPU_REQUIRE(src && dst && idx && row_len > 0 && count >= 0, "bad arguments");
    FLGPU_REQUIRE(src->prec == dst->prec && src->ctx == dst->ctx, "precision/context mismatch");
    FLGPU_REQUIRE(dst->n >= (long)count * row_len, "dst too small");
    long rows = src->n / row_len;
    flgpu_ctx *ctx = src->ctx;
    CTX_LOCK(ctx);
    size_t eb = prec_bytes(src->prec);
    for (int k = 0; k < count; k++) {
      FLGPU_REQUIRE(idx[k] >= 0 && idx[k] < rows, "row index out of range");
      FLGPU_HIP(hipMemcpyAsync((char *)dst->d + (size_t)k * row_len * eb,
                               (const char *)src->d + (size_t)idx[k] * row_len * eb, row_len * eb,
                               hipMemcpyDeviceToDevice, ctx->stream));
    }
    return 0;
  });
}
