// cmi_net.hip -- the learned warm start: a 4-layer 3-D convolutional network
// (3x3x3 kernels, 32 channels, ReLU) that maps (log n_H, log of the
// first-pass photoionization rate) to the logit of the converged neutral
// fraction.  Trained and run on the GPU by the kernels below:
//
//   conv_block_kernel   implicit-GEMM 3-D convolution on BF16 MFMA
//                  (v_mfma_f32_16x16x32_bf16, FP32 accumulation) over 8^3
//                  blocks of a dilation sub-lattice staged in LDS.  Serves the
//                  forward pass (weights [tap][cout][cin], bias, ReLU) and the
//                  input gradient (the same convolution over the output
//                  gradient with the flipped, transposed weights, masked by
//                  the ReLU of the layer below).
//   conv3_kernel   the same convolution without LDS, one wave per run of 16
//                  voxels: for volumes that leave the blocks mostly empty
//                  (dilations near the volume's edges), and for all forward
//                  passes after cmi_net_set_tiled(0).  The same outputs bit for
//                  bit.
//   wgrad_block_kernel  weight and bias gradient dW[tap][cout][cin] = sum_v
//                  dy[v][cout] * x[v + tap][cin] on the same MFMA, K = voxels,
//                  all 27 taps of a workgroup's blocks kept in registers.
//   wgrad_first_kernel, wgrad_last_kernel, dgrad_last_kernel  the layers with
//                  2 inputs and 1 output, taps as a matrix dimension.
//   plus the loss (mean squared error on logits), Adam on FP32 master weights
//   with the packing to BF16, crop sampling and input normalisation.
//
// Activations are BF16, channels-last with 32 channels ([B][D][H][W][32]); the
// network's 2 input channels are stored as [B][D][H][W][2] and the gradient of
// its single output as [B][D][H][W], and padded to the MFMA shapes in LDS.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <string>
#include <type_traits>
#include <vector>

#include "../../include/cmi.h"
#include "cmi_ctx.hpp"
#include "cmi_device.hpp"

namespace cmi {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kC = 32;        // channels of every activation tensor
constexpr int kTaps = 27;
constexpr int kLayers = 4;
// real input / output channels of each layer
__host__ __device__ constexpr int layer_cin(int l) { return l == 0 ? 2 : 32; }
__host__ __device__ constexpr int layer_cout(int l) { return l == kLayers - 1 ? 1 : 32; }

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }
__device__ __forceinline__ __bf16 f2bf(float v) { return (__bf16)v; }

// A voxel's 2 input channels (packed) as its MFMA operand: channels 8*kg ..
// 8*kg+7 of 32, zeros beyond the second.
__device__ __forceinline__ bf16x8 feat_operand(uint32_t two, int kg) {
  union {
    uint32_t u[4];
    bf16x8 v;
  } f;
  f.u[0] = kg == 0 ? two : 0u;
  f.u[1] = f.u[2] = f.u[3] = 0u;
  return f.v;
}

// ---------------------------------------------------------------------------
// 3-D convolution (padding 1) as implicit GEMM on MFMA 16x16x32 BF16.
// Lane l of a wave: A rows (voxels) l%16, A/B k-group (input channels)
// 8*(l/16)..+7, B column (output channel) l%16; accumulator rows (voxels)
// 4*(l/16)..+3, column l%16.
// ---------------------------------------------------------------------------
// kFeat: x is the network's input, 2 channels per voxel.
template <int NB, bool kFeat>
__global__ void __launch_bounds__(256) conv3_kernel(
    const __bf16 *__restrict__ x, const __bf16 *__restrict__ w,
    const float *__restrict__ bias, int nrun, int D, int H, int W, int dil,
    __bf16 *__restrict__ y, float *__restrict__ yf, const __bf16 *__restrict__ mask,
    int relu) {
  const int lane = threadIdx.x & 63;
  const int run = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (run >= nrun) return;  // whole wave leaves together
  // run -> (b, d, h, w0): 16 voxels along the last axis
  const int wr = W >> 4;
  int t = run;
  const int w0 = (t % wr) << 4;
  t /= wr;
  const int h = t % H;
  t /= H;
  const int d = t % D;
  const int b = t / D;
  const int vl = lane & 15;   // voxel (A row) / output channel (B column)
  const int kg = lane >> 4;   // k group: channels 8*kg .. 8*kg+7
  f32x4 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int NOUT = 16 * NB;
#pragma unroll 1
  for (int tap = 0; tap < kTaps; ++tap) {
    const int kd = tap / 9, kh = (tap / 3) % 3, kw = tap % 3;
    const int zd = d + (kd - 1) * dil, zh = h + (kh - 1) * dil,
              zw = w0 + vl + (kw - 1) * dil;
    bf16x8 a;
    if ((unsigned)zd < (unsigned)D && (unsigned)zh < (unsigned)H &&
        (unsigned)zw < (unsigned)W) {
      const size_t vox = (((size_t)b * D + zd) * H + zh) * W + zw;
      if (kFeat)
        a = feat_operand(reinterpret_cast<const uint32_t *>(x)[vox], kg);
      else
        a = *reinterpret_cast<const bf16x8 *>(x + vox * kC + 8 * kg);
    } else {
      a = bf16x8{};
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const bf16x8 bw = *reinterpret_cast<const bf16x8 *>(
          w + ((size_t)tap * NOUT + nb * 16 + vl) * kC + 8 * kg);
      acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bw, acc[nb], 0, 0, 0);
    }
  }
  const size_t vbase = (((size_t)b * D + d) * H + h) * W + w0;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int co = nb * 16 + vl;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t v = vbase + 4 * kg + i;
      float r = acc[nb][i] + (bias ? bias[co] : 0.f);
      if (mask) r = bf2f(mask[v * kC + co]) > 0.f ? r : 0.f;
      if (relu) r = fmaxf(r, 0.f);
      if (y) y[v * kC + co] = f2bf(r);
      if (yf && co == 0) yf[v] = r;
    }
  }
}

// ---------------------------------------------------------------------------
// Blocks.  A convolution with dilation d is d^3 ordinary 3x3x3 convolutions on
// the sub-lattices of voxels with equal coordinates mod d.  A workgroup takes a
// block of one sub-lattice, kBZ x 8 x 8 voxels, and stages it with its
// one-voxel halo in LDS, so that each input voxel is read from memory once per
// block instead of once per tap.  Any volume and dilation: a block may reach
// past its sub-lattice (zeros in, nothing out).  8^3 rather than rows of 16
// voxels along the last axis, because the sub-lattices of the 64^3 training
// crops at dilation 8 are 8^3.
//
// Packed blocks (kPack).  Along an axis where a whole sub-lattice has at most 3
// voxels a block holds several sub-lattices of consecutive residues, one empty
// position between neighbours: all that a tap past a sub-lattice's end meets is
// the zero padding, and one position of it serves both.  One sub-lattice a block
// would fill 1/512 of it at a dilation beyond the volume; packed, an axis is at
// least half filled.  Four training steps of two 64^3 crops at dilations of 32 and
// of 64: 35.4 and 253 ms before, 4.4 and 5.8 with packed blocks (and convolutions
// run by run where those are sparse).
// ---------------------------------------------------------------------------
constexpr int kE = 8;        // block edge
constexpr int kHE = kE + 2;  // with the halo

// Residues along an axis: `res` of them, `per_block` to a block, each with
// `period` positions (its voxels and an empty one); inv: 1 / period in 1/256,
// exact over a block's positions.  Not packed: 1, 0, 0.
struct Residues {
  int res, per_block, period, inv;
};

struct BlockGeo {
  int D, H, W, dil;
  int nrz, nry, nrx;  // residues per axis (packed: groups of residues)
  int nbz, nby, nbx;  // blocks per axis of the largest sub-lattice
  int nblocks;
  bool packed;        // some axis has several residues to a block
  // for the choice between blocks and runs (block_geo)
  bool sparse;    // few of the blocks' positions hold voxels
  bool few_runs;  // about a run per SIMD
  bool one_wave;  // all blocks at a time
  Residues pz, py, px;
};

// One block: its sample, (first) residues, first voxel and the extents of
// (the first) sub-lattice.
struct Block {
  int b, rz, ry, rx, z0, y0, x0, Ds, Hs, Ws;
};

template <int kBZ, bool kPack>
__device__ __forceinline__ Block block_of(const BlockGeo &G, int t) {
  Block k;
  k.x0 = (t % G.nbx) * kE;
  t /= G.nbx;
  k.y0 = (t % G.nby) * kE;
  t /= G.nby;
  k.z0 = (t % G.nbz) * kBZ;
  t /= G.nbz;
  k.rx = t % G.nrx;
  t /= G.nrx;
  k.ry = t % G.nry;
  t /= G.nry;
  k.rz = t % G.nrz;
  k.b = t / G.nrz;
  if (kPack) {
    k.rx *= G.px.per_block;
    k.ry *= G.py.per_block;
    k.rz *= G.pz.per_block;
  }
  k.Ds = (G.D - k.rz + G.dil - 1) / G.dil;
  k.Hs = (G.H - k.ry + G.dil - 1) / G.dil;
  k.Ws = (G.W - k.rx + G.dil - 1) / G.dil;
  return k;
}

// Coordinate of a block's position u along a packed axis, or -1 where it holds
// no voxel of the volume (extent cells).
__device__ __forceinline__ int packed_coord(const Residues &P, int r0, int x0, int extent,
                                            int dil, int u) {
  const int s = (u * P.inv) >> 8;  // which of the block's residues (-1 before the first)
  const int o = x0 + u - s * P.period;
  const int c = r0 + s + dil * o;  // past the volume for a residue's empty position
  return (unsigned)s < (unsigned)min(P.per_block, P.res - r0) && o >= 0 && c < extent ? c : -1;
}
// Positions of a block that hold voxels along an axis, as bits.
__device__ __forceinline__ unsigned packed_positions(const Residues &P, int r0, int x0,
                                                     int extent, int dil) {
  unsigned m = 0;
  for (int u = 0; u < kE; ++u)
    if (packed_coord(P, r0, x0, extent, dil, u) >= 0) m |= 1u << u;
  return m;
}

// Voxel number at position (uz, uy, ux) of a block, counted from its first
// voxel, or -1 outside the volume.
template <bool kPack>
__device__ __forceinline__ long long block_voxel(const BlockGeo &G, const Block &k, int uz,
                                                 int uy, int ux) {
  if (kPack) {
    const int z = packed_coord(G.pz, k.rz, k.z0, G.D, G.dil, uz);
    const int y = packed_coord(G.py, k.ry, k.y0, G.H, G.dil, uy);
    const int x = packed_coord(G.px, k.rx, k.x0, G.W, G.dil, ux);
    if ((z | y | x) < 0) return -1;
    return ((long long)(k.b * G.D + z) * G.H + y) * G.W + x;
  }
  const int sz = k.z0 + uz, sy = k.y0 + uy, sx = k.x0 + ux;
  if ((unsigned)sz >= (unsigned)k.Ds || (unsigned)sy >= (unsigned)k.Hs ||
      (unsigned)sx >= (unsigned)k.Ws)
    return -1;
  return ((long long)(k.b * G.D + k.rz + G.dil * sz) * G.H + k.ry + G.dil * sy) * G.W + k.rx +
         G.dil * sx;
}
// Halo voxel v (of (kBZ + 2) x 10 x 10) and inner voxel o (of kBZ x 8 x 8).
template <bool kPack>
__device__ __forceinline__ long long halo_voxel(const BlockGeo &G, const Block &k, int v) {
  return block_voxel<kPack>(G, k, v / (kHE * kHE) - 1, (v / kHE) % kHE - 1, v % kHE - 1);
}
template <bool kPack>
__device__ __forceinline__ long long inner_voxel(const BlockGeo &G, const Block &k, int o) {
  return block_voxel<kPack>(G, k, o >> 6, (o >> 3) & 7, o & 7);
}

// ---------------------------------------------------------------------------
// Convolution over 8^3 blocks: the same outputs as conv3_kernel bit for bit
// (every output voxel's 27 taps go through the same MFMAs with the same
// operands in the same order).  A wave computes two rows of 8 voxels in each
// of the block's planes, 8 MFMA rows of 16 voxels, and loads the weights of
// three taps at a time, one group ahead, once for all of them; 32-channel
// outputs leave through LDS in 16-byte pieces.  An LDS read of 16 B per lane
// feeds NB MFMAs, which puts the LDS at the pace of the matrix cores for NB =
// 2; two workgroups a CU (64 KB of LDS each) overlap one's loads with the
// other's products.  2^20 voxels (4 crops of 64^3), 32 -> 32 channels: 77 us
// (63 without the block's loads, 50 without its products), 87 for the rows of
// 16 voxels it replaces where those divided the volume and 290 for the per-run
// kernel that the other volumes and the input gradient took.
// mask: outputs of voxels and channels where it is not positive become 0 (the
// ReLU of the layer below, for the input gradient).
// ---------------------------------------------------------------------------
constexpr int kConvThreads = 256;

template <int NB, bool kFeat, bool kPack>
__global__ void __launch_bounds__(kConvThreads, 2) conv_block_kernel(
    BlockGeo G, const __bf16 *__restrict__ x, const __bf16 *__restrict__ w,
    const float *__restrict__ bias, __bf16 *__restrict__ y, float *__restrict__ yf,
    const __bf16 *__restrict__ mask, int relu) {
  constexpr int kHalo = kHE * kHE * kHE;
  constexpr int kInBytes = kHalo * (kFeat ? 4 : 64);
  constexpr int kOutBytes = NB == 2 ? kE * kE * kE * 64 : 0;
  __shared__ __align__(16) unsigned char lds[kInBytes > kOutBytes ? kInBytes : kOutBytes];
  const Block k = block_of<kE, kPack>(G, blockIdx.x);
  if (k.z0 >= k.Ds || k.y0 >= k.Hs || k.x0 >= k.Ws) return;
  // every thread issues all of its loads before its first LDS store, so the
  // block's memory latency is paid once, not once per load
  if (kFeat) {
    constexpr int kLoads = (kHalo + kConvThreads - 1) / kConvThreads;
    uint32_t vals[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int v = (int)threadIdx.x + i * kConvThreads;
      const long long g = v < kHalo ? halo_voxel<kPack>(G, k, v) : -1;
      vals[i] = g >= 0 ? reinterpret_cast<const uint32_t *>(x)[g] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int v = (int)threadIdx.x + i * kConvThreads;
      if (v < kHalo) reinterpret_cast<uint32_t *>(lds)[v] = vals[i];
    }
  } else {
    constexpr int kLoads = (4 * kHalo + kConvThreads - 1) / kConvThreads;
    bf16x8 vals[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int p = (int)threadIdx.x + i * kConvThreads;  // 16-byte piece
      const long long g = p < 4 * kHalo ? halo_voxel<kPack>(G, k, p >> 2) : -1;
      vals[i] = bf16x8{};
      if (g >= 0) vals[i] = *reinterpret_cast<const bf16x8 *>(x + g * kC + 8 * (p & 3));
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int p = (int)threadIdx.x + i * kConvThreads;
      if (p < 4 * kHalo) reinterpret_cast<bf16x8 *>(lds)[p] = vals[i];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int vl = lane & 15;  // voxel (A row) / output channel (B column)
  const int kg = lane >> 4;  // k group: channels 8*kg .. 8*kg+7
  const int NOUT = 16 * NB;
  const int first = (2 * wave + (vl >> 3)) * kHE + (vl & 7);  // halo voxel of tap 0
  const int nz = min(kE, k.Ds - k.z0);
  bool rows = 2 * wave < k.Hs - k.y0;  // the wave has voxels
  unsigned planes = 0;                 // planes with voxels (packed)
  if (kPack) {
    planes = packed_positions(G.pz, k.rz, k.z0, G.D, G.dil);
    rows = ((packed_positions(G.py, k.ry, k.y0, G.H, G.dil) >> (2 * wave)) & 3u) != 0;
  }
  f32x4 acc[kE][NB];
#pragma unroll
  for (int r = 0; r < kE; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[r][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto products = [&](auto whole) {
    bf16x8 bw[3][NB], bn[3][NB];
    auto load_weights = [&](int group) {
#pragma unroll
      for (int kw = 0; kw < 3; ++kw)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          bn[kw][nb] = *reinterpret_cast<const bf16x8 *>(
              w + ((size_t)(3 * group + kw) * NOUT + nb * 16 + vl) * kC + 8 * kg);
    };
    load_weights(0);
#pragma unroll 1
    for (int group = 0; group < 9; ++group) {
#pragma unroll
      for (int kw = 0; kw < 3; ++kw)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) bw[kw][nb] = bn[kw][nb];
      if (group + 1 < 9) load_weights(group + 1);
      const int at = first + ((group / 3) * kHE + group % 3) * kHE;
#pragma unroll
      for (int kw = 0; kw < 3; ++kw) {
#pragma unroll
        for (int r = 0; r < kE; ++r) {
          if (kPack) {
            if (((planes >> r) & 1u) == 0) continue;
          } else if (!decltype(whole)::value && r >= nz) {
            break;
          }
          const int v = at + kw + r * kHE * kHE;
          bf16x8 a;
          if (kFeat)
            a = feat_operand(reinterpret_cast<const uint32_t *>(lds)[v], kg);
          else
            a = *reinterpret_cast<const bf16x8 *>(lds + (size_t)v * 64 + 16 * kg);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[r][nb] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bw[kw][nb], acc[r][nb], 0, 0, 0);
        }
      }
    }
  };
  if (rows) {
    if (!kPack && nz == kE)
      products(std::true_type{});
    else
      products(std::false_type{});
  }
  if (NB == 2) {
    // through the (now free) LDS block as [voxel][32 channels]
    __bf16 *out = reinterpret_cast<__bf16 *>(lds);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kE; ++r)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int co = nb * 16 + vl;
        const float add = bias ? bias[co] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int vrow = 4 * kg + i;
          float o = acc[r][nb][i] + add;
          if (relu) o = fmaxf(o, 0.f);
          out[((r * kE + 2 * wave + (vrow >> 3)) * kE + (vrow & 7)) * kC + co] = f2bf(o);
        }
      }
    __syncthreads();
    constexpr int kOut = kE * kE * kE * 4 / kConvThreads;  // 16-byte pieces per thread
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      const int p = (int)threadIdx.x + i * kConvThreads;
      const long long g = inner_voxel<kPack>(G, k, p >> 2);
      if (g < 0) continue;
      bf16x8 o = reinterpret_cast<const bf16x8 *>(lds)[p];
      if (mask) {
        const bf16x8 m = *reinterpret_cast<const bf16x8 *>(mask + g * kC + 8 * (p & 3));
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = bf2f(m[e]) > 0.f ? o[e] : f2bf(0.f);
      }
      *reinterpret_cast<bf16x8 *>(y + g * kC + 8 * (p & 3)) = o;
    }
  } else if (vl == 0) {
    // the network's output: channel 0 only
#pragma unroll
    for (int r = 0; r < kE; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vrow = 4 * kg + i;
        const long long g =
            block_voxel<kPack>(G, k, r, 2 * wave + (vrow >> 3), vrow & 7);
        if (g >= 0) yf[g] = acc[r][0][i] + (bias ? bias[0] : 0.f);
      }
  }
}

// ---------------------------------------------------------------------------
// Weight gradients.  K of the MFMA runs over voxels, so both operands are
// columns of channels-last data: the LDS transpose read (ds_read_b64_tr_b16,
// 4 voxels x 16 channels per 16 lanes) forms them, two reads for the 8
// consecutive voxels of a lane.
// ---------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));

union Operand {
  s16x4 h[2];
  bf16x8 v;
};

// p: the lane's share of voxels x .. x+3 (its voxel (lane % 16) / 4, channels
// 4 (lane % 4) ..); step: elements from voxel x to voxel x+4.
__device__ __forceinline__ bf16x8 voxels_operand(const __bf16 *p, int step) {
  Operand o;
  o.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4 *)p);
  o.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4 *)(p + step));
  return o.v;
}

// Workgroups add their sums into kCopies copies of the gradient in turn
// (grad_copy), which the optimiser sums up.  Adds of many workgroups to one
// cache line pass one at a time: 512 workgroups on one copy cost 35 to 42 us
// of a 32-channel layer's 125, on 16 copies 2 to 3.
constexpr int kCopies = 16;
__device__ __forceinline__ float *grad_copy(float *g, size_t stride) {
  return g + (blockIdx.x % kCopies) * stride;
}

constexpr int kGZ = 4;  // planes of a weight-gradient block
constexpr int kGVox = kGZ * kE * kE;
constexpr int kGHalo = (kGZ + 2) * kHE * kHE;
constexpr int kGThreads = 256;
constexpr int kTapsPerWave = 7;

// The 32 -> 32 channel layers.  A wave owns 7 taps (the last wave 6 and the
// bias, whose second operand is ones) and keeps their 32 x 32 gradients in
// registers over all blocks of its workgroup; one FP32 atomic add per weight
// and workgroup at the end.  Per 32 voxels a wave reads 32 operand halves
// from LDS for 28 MFMAs, so LDS and matrix cores are about level; the next
// block's loads are in flight under them.  2^20 voxels: 100 us (16 of them the
// final adds; 76 with an eighth of the products), against 970 for one wave per
// tap, channel block and 16 runs with 2-byte operand loads.
template <bool kPack>
__global__ void __launch_bounds__(kGThreads, 2) wgrad_block_kernel(
    BlockGeo G, const __bf16 *__restrict__ dy, const __bf16 *__restrict__ x,
    float *__restrict__ grad, size_t stride, size_t off_w, size_t off_b) {
  float *const dW = grad_copy(grad, stride) + off_w, *const db = grad_copy(grad, stride) + off_b;
  __shared__ __align__(16) __bf16 xs[kGHalo * kC];
  __shared__ __align__(16) __bf16 ds[kGVox * kC];
  constexpr int kXL = (4 * kGHalo + kGThreads - 1) / kGThreads, kDL = 4 * kGVox / kGThreads;
  bf16x8 px[kXL], pd[kDL];
  auto load = [&](int blk) {
    const Block k = block_of<kGZ, kPack>(G, blk);
#pragma unroll
    for (int i = 0; i < kXL; ++i) {
      const int p = (int)threadIdx.x + i * kGThreads;
      const long long g = p < 4 * kGHalo ? halo_voxel<kPack>(G, k, p >> 2) : -1;
      px[i] = bf16x8{};
      if (g >= 0) px[i] = *reinterpret_cast<const bf16x8 *>(x + g * kC + 8 * (p & 3));
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i) {
      const int p = (int)threadIdx.x + i * kGThreads;
      const long long g = inner_voxel<kPack>(G, k, p >> 2);
      pd[i] = bf16x8{};
      if (g >= 0) pd[i] = *reinterpret_cast<const bf16x8 *>(dy + g * kC + 8 * (p & 3));
    }
  };
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ml = lane & 15, kg = lane >> 4, r4 = ml >> 2, c4 = lane & 3;
  const __bf16 *const dl = ds + ((kg * kE + r4) * kC + 4 * c4);
  const __bf16 *const xl = xs + ((kg * kHE + r4) * kC + 4 * c4);
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = f2bf(1.f);
  f32x4 acc[kTapsPerWave][2][2];
#pragma unroll
  for (int t = 0; t < kTapsPerWave; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[t][q >> 1][q & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  int blk = blockIdx.x;
  if (blk < G.nblocks) load(blk);
  for (; blk < G.nblocks; blk += gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kXL; ++i) {
      const int p = (int)threadIdx.x + i * kGThreads;
      if (p < 4 * kGHalo) reinterpret_cast<bf16x8 *>(xs)[p] = px[i];
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i)
      reinterpret_cast<bf16x8 *>(ds)[threadIdx.x + i * kGThreads] = pd[i];
    __syncthreads();
    if (blk + (int)gridDim.x < G.nblocks) load(blk + gridDim.x);
    // 32 voxels at a time: 4 rows of 8, row kg the lane's
#pragma unroll 1
    for (int s = 0; s < kGVox / 32; ++s) {
      const __bf16 *const dp = dl + s * (4 * kE) * kC;
      const __bf16 *const xp = xl + ((s >> 1) * kHE * kHE + (s & 1) * 4 * kHE) * kC;
      bf16x8 a[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) a[m] = voxels_operand(dp + 16 * m, 4 * kC);
#pragma unroll
      for (int t = 0; t < kTapsPerWave; ++t) {
        const int tap = wave * kTapsPerWave + t;
        if (t + 1 < kTapsPerWave || tap < kTaps) {
          const int off = ((tap / 9) * kHE + (tap / 3) % 3) * kHE + tap % 3;
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const bf16x8 b = voxels_operand(xp + off * kC + 16 * n, 4 * kC);
#pragma unroll
            for (int m = 0; m < 2; ++m)
              acc[t][m][n] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b, acc[t][m][n], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int m = 0; m < 2; ++m)
            acc[t][m][0] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], ones, acc[t][m][0], 0, 0, 0);
        }
      }
    }
  }
  // accumulator: rows (cout) 4*kg..+3, column (cin) ml
#pragma unroll
  for (int t = 0; t < kTapsPerWave; ++t) {
    const int tap = wave * kTapsPerWave + t;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int co = 16 * m + 4 * kg + i;
        if (tap < kTaps) {
          atomicAdd(&dW[((size_t)tap * kC + co) * kC + ml], acc[t][m][0][i]);
          atomicAdd(&dW[((size_t)tap * kC + co) * kC + 16 + ml], acc[t][m][1][i]);
        } else if (ml == 0) {
          atomicAdd(&db[co], acc[t][m][0][i]);
        }
      }
  }
}

// The first layer (2 input channels): tap and input channel together are the
// MFMA's columns, 54 of 64 (16 to a wave), with the bias (ones) as column 54.
// The input is staged as planes shifted by each tap of the last axis, so that
// an operand's 8 voxels are one aligned read.  Bound by reading dy once and
// the final adds (42 us for 2^20 voxels; 59 with twice the workgroups).
template <bool kPack>
__global__ void __launch_bounds__(kGThreads) wgrad_first_kernel(
    BlockGeo G, const __bf16 *__restrict__ dy, const uint32_t *__restrict__ feat,
    float *__restrict__ grad, size_t stride, size_t off_w, size_t off_b) {
  float *const dW = grad_copy(grad, stride) + off_w, *const db = grad_copy(grad, stride) + off_b;
  constexpr int kPlane = (kGZ + 2) * kHE * kE;  // one channel, one shift
  __shared__ __align__(16) __bf16 ds[kGVox * kC];
  __shared__ __align__(16) uint16_t pl[3 * 2 * kPlane];
  constexpr int kFL = (kGHalo + kGThreads - 1) / kGThreads, kDL = 4 * kGVox / kGThreads;
  uint32_t pf[kFL];
  bf16x8 pd[kDL];
  auto load = [&](int blk) {
    const Block k = block_of<kGZ, kPack>(G, blk);
#pragma unroll
    for (int i = 0; i < kFL; ++i) {
      const int v = (int)threadIdx.x + i * kGThreads;
      const long long g = v < kGHalo ? halo_voxel<kPack>(G, k, v) : -1;
      pf[i] = g >= 0 ? feat[g] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i) {
      const int p = (int)threadIdx.x + i * kGThreads;
      const long long g = inner_voxel<kPack>(G, k, p >> 2);
      pd[i] = bf16x8{};
      if (g >= 0) pd[i] = *reinterpret_cast<const bf16x8 *>(dy + g * kC + 8 * (p & 3));
    }
  };
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ml = lane & 15, kg = lane >> 4, r4 = ml >> 2, c4 = lane & 3;
  const __bf16 *const dl = ds + ((kg * kE + r4) * kC + 4 * c4);
  const int n = 16 * wave + ml, tap = n >> 1, c = n & 1;
  const bool real = tap < kTaps;
  const uint16_t *const fl =
      pl + (real ? (((tap % 3) * 2 + c) * kPlane + ((tap / 9) * kHE + (tap / 3) % 3) * kE) : 0) +
      kg * kE;
  bf16x8 fixed;  // the operand of a column that is no tap
#pragma unroll
  for (int j = 0; j < 8; ++j) fixed[j] = f2bf(n == 2 * kTaps ? 1.f : 0.f);
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  int blk = blockIdx.x;
  if (blk < G.nblocks) load(blk);
  for (; blk < G.nblocks; blk += gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFL; ++i) {
      const int v = (int)threadIdx.x + i * kGThreads;
      const int hx = v % kHE, row = v / kHE;
      if (v < kGHalo) {
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          if ((unsigned)(hx - s) < (unsigned)kE) {
            pl[(2 * s) * kPlane + row * kE + hx - s] = (uint16_t)pf[i];
            pl[(2 * s + 1) * kPlane + row * kE + hx - s] = (uint16_t)(pf[i] >> 16);
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i)
      reinterpret_cast<bf16x8 *>(ds)[threadIdx.x + i * kGThreads] = pd[i];
    __syncthreads();
    if (blk + (int)gridDim.x < G.nblocks) load(blk + gridDim.x);
#pragma unroll
    for (int s = 0; s < kGVox / 32; ++s) {
      bf16x8 b = *reinterpret_cast<const bf16x8 *>(
          fl + ((s >> 1) * kHE + (s & 1) * 4) * kE);
      if (!real) b = fixed;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const bf16x8 a = voxels_operand(dl + s * (4 * kE) * kC + 16 * m, 4 * kC);
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[m], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co = 16 * m + 4 * kg + i;
      if (real)
        atomicAdd(&dW[((size_t)tap * kC + co) * kC + c], acc[m][i]);
      else if (n == 2 * kTaps)
        atomicAdd(&db[co], acc[m][i]);
    }
}

// The last layer (1 output channel): the taps are the MFMA's rows, dW[tap][ci]
// = sum_u dz[u - tap] x[u][ci], with the output gradient dz (one value per
// voxel) staged in shifted planes.  Bound by reading x once (28 us for 2^20
// voxels).  (The bias gradient, the sum of dz, comes with the loss.)
template <bool kPack>
__global__ void __launch_bounds__(kGThreads) wgrad_last_kernel(
    BlockGeo G, const uint16_t *__restrict__ dz, const __bf16 *__restrict__ x,
    float *__restrict__ grad, size_t stride, size_t off_w, int NOUT) {
  float *const dW = grad_copy(grad, stride) + off_w;
  constexpr int kPlane = (kGZ + 2) * kHE * kE;
  __shared__ __align__(16) __bf16 xs[kGVox * kC];
  __shared__ __align__(16) uint16_t pl[3 * kPlane];
  constexpr int kFL = (kGHalo + kGThreads - 1) / kGThreads, kDL = 4 * kGVox / kGThreads;
  uint16_t pz[kFL];
  bf16x8 px[kDL];
  auto load = [&](int blk) {
    const Block k = block_of<kGZ, kPack>(G, blk);
#pragma unroll
    for (int i = 0; i < kFL; ++i) {
      const int v = (int)threadIdx.x + i * kGThreads;
      const long long g = v < kGHalo ? halo_voxel<kPack>(G, k, v) : -1;
      pz[i] = g >= 0 ? dz[g] : (uint16_t)0;
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i) {
      const int p = (int)threadIdx.x + i * kGThreads;
      const long long g = inner_voxel<kPack>(G, k, p >> 2);
      px[i] = bf16x8{};
      if (g >= 0) px[i] = *reinterpret_cast<const bf16x8 *>(x + g * kC + 8 * (p & 3));
    }
  };
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ml = lane & 15, kg = lane >> 4, r4 = ml >> 2, c4 = lane & 3;
  const __bf16 *const xl = xs + ((kg * kE + r4) * kC + 4 * c4);
  // the lane's row of either half of the taps: halo offset of u - (tap - 1)
  const uint16_t *zl[2];
  bool real[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int tap = 16 * m + ml;
    real[m] = tap < kTaps;
    const int t = real[m] ? tap : 0;
    zl[m] = pl + (2 - t % 3) * kPlane + ((2 - t / 9) * kHE + 2 - (t / 3) % 3) * kE + kg * kE;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q >> 1][q & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  int blk = blockIdx.x;
  if (blk < G.nblocks) load(blk);
  for (; blk < G.nblocks; blk += gridDim.x) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFL; ++i) {
      const int v = (int)threadIdx.x + i * kGThreads;
      const int hx = v % kHE, row = v / kHE;
      if (v < kGHalo) {
#pragma unroll
        for (int s = 0; s < 3; ++s)
          if ((unsigned)(hx - s) < (unsigned)kE) pl[s * kPlane + row * kE + hx - s] = pz[i];
      }
    }
#pragma unroll
    for (int i = 0; i < kDL; ++i)
      reinterpret_cast<bf16x8 *>(xs)[threadIdx.x + i * kGThreads] = px[i];
    __syncthreads();
    if (blk + (int)gridDim.x < G.nblocks) load(blk + gridDim.x);
    // each wave takes two of the block's eight 32-voxel pieces
#pragma unroll
    for (int h = 0; h < kGVox / 32 / 4; ++h) {
      const int s = wave + 4 * h;
      bf16x8 a[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        a[m] = *reinterpret_cast<const bf16x8 *>(zl[m] + ((s >> 1) * kHE + (s & 1) * 4) * kE);
        if (!real[m]) a[m] = bf16x8{};
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const bf16x8 b = voxels_operand(xl + s * (4 * kE) * kC + 16 * c, 4 * kC);
#pragma unroll
        for (int m = 0; m < 2; ++m)
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b, acc[m][c], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tap = 16 * m + 4 * kg + i;
      if (tap < kTaps) {
        atomicAdd(&dW[(size_t)tap * NOUT * kC + ml], acc[m][0][i]);
        atomicAdd(&dW[(size_t)tap * NOUT * kC + 16 + ml], acc[m][1][i]);
      }
    }
}

// Input gradient of the last layer: dx[v][ci] = sum over taps of dz[v + tap - 1]
// w[tap][ci], masked by the ReLU of the layer below; the taps are the MFMA's K
// (27 of 32), one product per 16 voxels and 16 channels.  Bound by the mask
// read and dx written once: 41 us for 2^20 voxels, 290 through 27 products
// per 16 voxels of a 32-channel dz.
template <bool kPack>
__global__ void __launch_bounds__(kConvThreads) dgrad_last_kernel(
    BlockGeo G, const uint16_t *__restrict__ dz, const __bf16 *__restrict__ wb,
    const __bf16 *__restrict__ mask, __bf16 *__restrict__ dx) {
  constexpr int kHalo = kHE * kHE * kHE;
  __shared__ uint16_t zs[kHalo];
  __shared__ __align__(16) __bf16 out[kE * kE * kE * kC];
  const Block k = block_of<kE, kPack>(G, blockIdx.x);
  if (k.z0 >= k.Ds || k.y0 >= k.Hs || k.x0 >= k.Ws) return;
  constexpr int kLoads = (kHalo + kConvThreads - 1) / kConvThreads;
  uint16_t vals[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int v = (int)threadIdx.x + i * kConvThreads;
    const long long g = v < kHalo ? halo_voxel<kPack>(G, k, v) : -1;
    vals[i] = g >= 0 ? dz[g] : (uint16_t)0;
  }
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int v = (int)threadIdx.x + i * kConvThreads;
    if (v < kHalo) zs[v] = vals[i];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int vl = lane & 15, kg = lane >> 4;
  union Taps {
    uint16_t u[8];
    bf16x8 v;
  };
  Taps b[2];
  int off[8];  // halo voxel of the lane's taps at the first plane
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t = 8 * kg + j;
    off[j] = (2 * wave + (vl >> 3)) * kHE + (vl & 7);
    if (t < kTaps) off[j] += ((t / 9) * kHE + (t / 3) % 3) * kHE + t % 3;
#pragma unroll
    for (int n = 0; n < 2; ++n)
      b[n].u[j] = t < kTaps ? reinterpret_cast<const uint16_t *>(
                                  wb)[((size_t)t * 32 + 16 * n + vl) * kC]
                            : (uint16_t)0;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kE; ++r) {
    Taps a;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      a.u[j] = 8 * kg + j < kTaps ? zs[off[j] + r * kHE * kHE] : (uint16_t)0;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b[n].v, acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vrow = 4 * kg + i;
        out[((r * kE + 2 * wave + (vrow >> 3)) * kE + (vrow & 7)) * kC + 16 * n + vl] =
            f2bf(acc[i]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kE * kE * kE * 4 / kConvThreads; ++i) {
    const int p = (int)threadIdx.x + i * kConvThreads;
    const long long g = inner_voxel<kPack>(G, k, p >> 2);
    if (g < 0) continue;
    bf16x8 o = reinterpret_cast<const bf16x8 *>(out)[p];
    const bf16x8 m = *reinterpret_cast<const bf16x8 *>(mask + g * kC + 8 * (p & 3));
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = bf2f(m[e]) > 0.f ? o[e] : f2bf(0.f);
    *reinterpret_cast<bf16x8 *>(dx + g * kC + 8 * (p & 3)) = o;
  }
}

// Weighted mean squared error on logits: with e = z - t and w = w_pos for
// e > 0 (a prediction more neutral than the target), 1 otherwise,
// loss += sum w e^2 / n; dz[v] = 2 w e / n, and its sum to the bias gradient.
__global__ void __launch_bounds__(256) mse_kernel(
    const float *__restrict__ z, const float *__restrict__ tgt, size_t n, float w_pos,
    __bf16 *__restrict__ dz, float *__restrict__ grad, size_t stride, size_t off_loss,
    size_t off_b) {
  __shared__ float sh[8];
  float s = 0.f, d = 0.f;
  const float inv = 1.f / (float)n;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (size_t)gridDim.x * blockDim.x) {
    const float e = z[v] - tgt[v];
    const float w = e > 0.f ? w_pos : 1.f;
    s += w * e * e;
    const __bf16 g = f2bf(2.f * w * e * inv);
    dz[v] = g;
    d += bf2f(g);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    d += __shfl_xor(d, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[threadIdx.x >> 6] = s;
    sh[4 + (threadIdx.x >> 6)] = d;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float *const g = grad_copy(grad, stride);
    atomicAdd(g + off_loss, (sh[0] + sh[1] + sh[2] + sh[3]) * inv);
    atomicAdd(g + off_b, sh[4] + sh[5] + sh[6] + sh[7]);
  }
}

// Layers of the master vector (FP32, padded to the MFMA shapes): W[27][NOUT]
// [32] (tap, output channel, input channel; entries beyond the real channels
// stay 0: their gradients are 0) then b[NOUT].  Packed BF16 GEMM weights: fwd
// = W as is, and the input-gradient weights bwd[t'][cin][cout] =
// W[26-t'][cout][cin] ([27][32][32], zero for cout >= NOUT).
struct Layers {
  size_t off_w[kLayers], off_b[kLayers];
  int nout[kLayers];
  __bf16 *fwd[kLayers], *bwd[kLayers];
};

__global__ void pack_kernel(const float *__restrict__ p, Layers L) {
  const int n = kTaps * 32 * 32;
  const int l = blockIdx.y, NOUT = L.nout[l];
  const float *const master = p + L.off_w[l];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int tap = i / 1024, o = (i / 32) % 32, k = i % 32;
    if (o < NOUT)
      L.fwd[l][((size_t)tap * NOUT + o) * kC + k] = f2bf(master[((size_t)tap * NOUT + o) * kC + k]);
    const float vb = k < NOUT ? master[((size_t)(kTaps - 1 - tap) * NOUT + k) * kC + o] : 0.f;
    L.bwd[l][((size_t)tap * 32 + o) * kC + k] = f2bf(vb);
  }
}

__device__ __forceinline__ float sum_copies(const float *__restrict__ g, size_t stride,
                                            size_t i) {
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < kCopies; ++c) s += g[c * stride + i];
  return s;
}

// The gradient (n values) and the loss after it, summed over the copies.
__global__ void sum_grad_kernel(const float *__restrict__ g, size_t stride, size_t n,
                                float *__restrict__ out) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i <= n;
       i += (size_t)gridDim.x * blockDim.x)
    out[i] = sum_copies(g, stride, i);
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters; an updated weight
// goes to its place in both packed copies at once.  Value n of the gradient is
// the loss.
__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, size_t stride,
                            float *__restrict__ m, float *__restrict__ v, size_t n,
                            float lr, float b1, float b2, float eps, float c1,
                            float c2, float wd, Layers L, float *__restrict__ loss) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i <= n;
       i += (size_t)gridDim.x * blockDim.x) {
    const float gs = sum_copies(g, stride, i);
    if (i == n) {
      *loss = gs;
      continue;
    }
    const float gi = gs + wd * p[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    int l = kLayers - 1;
    while (i < L.off_w[l]) --l;
    if (i < L.off_b[l]) {
      const int j = (int)(i - L.off_w[l]), NOUT = L.nout[l];
      const int k = j % kC, o = (j / kC) % NOUT, tap = j / (kC * NOUT);
      L.fwd[l][j] = f2bf(pi);
      L.bwd[l][((size_t)(kTaps - 1 - tap) * 32 + k) * kC + o] = f2bf(pi);
    }
  }
}

// Crops of the samples (features log10 n_H, log10 jH; FP32) as the network's
// input, 2 normalised BF16 channels per voxel, and their scaled targets.
constexpr int kMaxCrops = 16;
struct Crops {
  int sample[kMaxCrops], d[kMaxCrops], h[kMaxCrops], w[kMaxCrops];  // and origins
};
__device__ __forceinline__ uint32_t pack_features(float f0, float f1, float m0, float s0,
                                                  float m1, float s1) {
  union {
    __bf16 c[2];
    uint32_t u;
  } o;
  o.c[0] = f2bf((f0 - m0) * s0);
  o.c[1] = f2bf((f1 - m1) * s1);
  return o.u;
}
__global__ void crops_kernel(const float *__restrict__ feat, const float *__restrict__ tgt,
                             int D, int H, int W, Crops C, int S0, int S1, int S2, float m0,
                             float s0, float m1, float s1, float inv_scale,
                             uint32_t *__restrict__ out, float *__restrict__ tgt_out) {
  const size_t n = (size_t)S0 * S1 * S2;
  const int b = blockIdx.y;
  const size_t base = (size_t)C.sample[b] * D * H * W;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (size_t)gridDim.x * blockDim.x) {
    const int z = (int)(v % S2), y = (int)((v / S2) % S1), xx = (int)(v / ((size_t)S1 * S2));
    const size_t src =
        base + (((size_t)(C.d[b] + xx) * H) + (C.h[b] + y)) * W + (C.w[b] + z);
    const float2 f = reinterpret_cast<const float2 *>(feat)[src];
    out[b * n + v] = pack_features(f.x, f.y, m0, s0, m1, s1);
    if (tgt) tgt_out[b * n + v] = tgt[src] * inv_scale;
  }
}

// Lattice cell (gx, gy, gz) of a context -> its device address (subgrids in
// the reference's order (sx * nsub_y + sy) * nsub_z + sz, tile-major inside).
__device__ __forceinline__ size_t lattice_addr(const GridDev &g, int gx, int gy, int gz) {
  const int sx = gx / g.sc[0], sy = gy / g.sc[1], sz = gz / g.sc[2];
  const int sub = (sx * g.nsub[1] + sy) * g.nsub[2] + sz;
  return cell_addr(g, sub, gx - sx * g.sc[0], gy - sy * g.sc[1], gz - sz * g.sc[2]);
}

constexpr double kJHFloor = 1e-12;  // s^-1, added before the logarithm

// logit of x_n clamped to [1e-7, 1 - 1/150]: above that every cell is
// opaque (a 256^3-workload cell of neutral gas has optical depth ~76), and
// the clamp keeps the Monte Carlo noise of near-neutral cells (1 - x ~ 1e-6)
// out of the features and targets
constexpr double kXnHigh = 1. - 1. / 150.;
__device__ __forceinline__ double clamped_logit(double x) {
  x = fmin(fmax(x, 1e-7), kXnHigh);
  return log(x / (1. - x));
}

// Features of a context's cells in lattice order: log10 n_H and, in input
// mode 0, log10(jconv * J + floor) (the photoionization rate of the last
// transport), in mode 1 the logit of the current x_n; normalised BF16 into
// act (channels 0, 1 of 32) and/or raw FP32 into feat ([v][2]).
__global__ void ctx_features_kernel(GridDev g, const double *__restrict__ n,
                                    const double *__restrict__ J,
                                    const double *__restrict__ xn, int mode, int D, int H,
                                    int W, double jconv, float m0, float s0, float m1,
                                    float s1, uint32_t *__restrict__ act,
                                    float *__restrict__ feat) {
  const size_t nv = (size_t)D * H * W;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
       v += (size_t)gridDim.x * blockDim.x) {
    const int gz = (int)(v % W), gy = (int)((v / W) % H), gx = (int)(v / ((size_t)W * H));
    const size_t a = lattice_addr(g, gx, gy, gz);
    const float f0 = (float)log10(n[a]);
    const float f1 = mode == 1 ? (float)clamped_logit(xn[a])
                               : (float)log10(jconv * J[a] + kJHFloor);
    if (feat) {
      feat[2 * v] = f0;
      feat[2 * v + 1] = f1;
    }
    if (act) act[v] = pack_features(f0, f1, m0, s0, m1, s1);
  }
}

// Network outputs (lattice order) -> x_n of the context, J = 0, FP32
// opacity.  Mode 0: the output is the logit of x_n; mode 1: it is added to
// the logit of the current x_n.  A cell whose logit exceeds `cut`
// (predicted neutral) starts at `fallback` instead.
__global__ void ctx_apply_kernel(GridDev g, const float *__restrict__ z, int mode, int D,
                                 int H, int W, float out_scale, float cut, double fallback,
                                 const double *__restrict__ n,
                                 double *__restrict__ xn, double *__restrict__ J,
                                 float *__restrict__ kappa, double kscale) {
  const size_t nv = (size_t)D * H * W;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
       v += (size_t)gridDim.x * blockDim.x) {
    const int gz = (int)(v % W), gy = (int)((v / W) % H), gx = (int)(v / ((size_t)W * H));
    const size_t a = lattice_addr(g, gx, gy, gz);
    const double logit =
        (double)z[v] * (double)out_scale + (mode == 1 ? clamped_logit(xn[a]) : 0.);
    double x = 1. / (1. + exp(-logit));
    x = fmin(fmax(x, 1e-7), 1.);
    if (logit > (double)cut) x = fallback;
    xn[a] = x;
    J[a] = 0.;
    if (kappa) kappa[a] = (float)(kscale * n[a] * x);
  }
}

// Coarse start of the warm start.  restrict: coarse n_H = the mean of each
// f^3 block of fine cells (the mass of the block), coarse x_n = 1e-6, J = 0,
// FP32 opacity of that state.
__global__ void restrict_density_kernel(GridDev gf, const double *__restrict__ nf,
                                        GridDev gc, int f, int Dc, int Hc, int Wc,
                                        double *__restrict__ nc, double *__restrict__ xnc,
                                        double *__restrict__ Jc, float *__restrict__ kappa,
                                        double kscale) {
  const size_t nv = (size_t)Dc * Hc * Wc;
  const double inv = 1. / ((double)f * f * f);
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
       v += (size_t)gridDim.x * blockDim.x) {
    const int cz = (int)(v % Wc), cy = (int)((v / Wc) % Hc), cx = (int)(v / ((size_t)Wc * Hc));
    double s = 0.;
    for (int i = 0; i < f; ++i)
      for (int j = 0; j < f; ++j)
        for (int k = 0; k < f; ++k)
          s += nf[lattice_addr(gf, cx * f + i, cy * f + j, cz * f + k)];
    const size_t a = lattice_addr(gc, cx, cy, cz);
    const double n = s * inv;
    nc[a] = n;
    xnc[a] = 1e-6;
    Jc[a] = 0.;
    if (kappa) kappa[a] = (float)(kscale * n * 1e-6);
  }
}

// prolong: the fine x_n is the coarse field's logit (clamped like the
// features) interpolated trilinearly at the fine cell's centre (coarse cell
// centres at (c + 1/2) f fine cells, the edge cells extended), J = 0, FP32
// opacity refreshed.
__global__ void prolong_xn_kernel(GridDev gc, const double *__restrict__ xnc, int f,
                                  int Dc, int Hc, int Wc, GridDev gf,
                                  const double *__restrict__ nf, double *__restrict__ xnf,
                                  double *__restrict__ Jf, float *__restrict__ kappa,
                                  double kscale) {
  const int Df = Dc * f, Hf = Hc * f, Wf = Wc * f;
  const size_t nv = (size_t)Df * Hf * Wf;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv;
       v += (size_t)gridDim.x * blockDim.x) {
    const int z = (int)(v % Wf), y = (int)((v / Wf) % Hf), x = (int)(v / ((size_t)Wf * Hf));
    int c0[3], c1[3];
    double w[3];
    const int fi[3] = {x, y, z}, nc[3] = {Dc, Hc, Wc};
    for (int a = 0; a < 3; ++a) {
      const double u = ((double)fi[a] + 0.5) / (double)f - 0.5;
      const double fl = floor(u);
      w[a] = u - fl;
      c0[a] = min(max((int)fl, 0), nc[a] - 1);
      c1[a] = min(max((int)fl + 1, 0), nc[a] - 1);
    }
    double l = 0.;
    for (int k = 0; k < 8; ++k) {
      const int ix = (k & 4) ? c1[0] : c0[0], iy = (k & 2) ? c1[1] : c0[1],
                iz = (k & 1) ? c1[2] : c0[2];
      const double wk = ((k & 4) ? w[0] : 1. - w[0]) * ((k & 2) ? w[1] : 1. - w[1]) *
                        ((k & 1) ? w[2] : 1. - w[2]);
      l += wk * clamped_logit(xnc[lattice_addr(gc, ix, iy, iz)]);
    }
    const size_t a = lattice_addr(gf, x, y, z);
    const double xn = 1. / (1. + exp(-l));
    xnf[a] = xn;
    Jf[a] = 0.;
    if (kappa) kappa[a] = (float)(kscale * nf[a] * xn);
  }
}

__global__ void zero_f32_kernel(float *p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0.f;
}

}  // namespace cmi

using namespace cmi;

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct cmi_net {
  int device = 0;
  int num_cus = 0;
  hipStream_t stream = nullptr;
  std::string err;
  size_t nparam = 0;
  size_t off_w[kLayers], off_b[kLayers];  // offsets into the master vector
  float *p = nullptr, *m = nullptr, *v = nullptr;  // FP32
  float *g = nullptr;      // kCopies copies of the gradient and the loss
  size_t grad_stride = 0;  // values from copy to copy
  float *grad_sum = nullptr;  // their sum (loss_and_grad)
  __bf16 *wf[kLayers] = {}, *wb[kLayers] = {};                    // packed
  int step = 0;
  // normalisation of the features and of the target logits
  float mean[2] = {8.f, -10.f}, scale[2] = {1.f, 0.25f};
  float out_scale = 8.f;  // logit = out_scale * network output
  // start rule of the warm start: cells predicted more neutral than logit
  // `cut` start at `fallback` (default: no cut)
  float cut = 3.0e38f;
  double fallback = 1e-6;
  int dil[kLayers] = {1, 1, 1, 1};  // dilation of each layer's 3x3x3 taps
  float w_pos = 1.f;  // loss weight of predictions more neutral than the target
  int mode = 0;       // input mode of the warm start (0: jH, 1: refine x_n)
  int tiled = 1;      // forward convolutions through conv_block_kernel
  // dataset (device): features [S][N][2] FP32, targets [S][N] FP32
  float *ds_feat = nullptr, *ds_tgt = nullptr;
  int ds_n = 0, ds_dim[3] = {0, 0, 0};
  size_t ds_cap = 0;
  // work buffers (sized for the largest batch seen)
  size_t work_vox = 0, grad_vox = 0;
  uint32_t *in = nullptr;     // the input, 2 BF16 channels per voxel
  __bf16 *act[kLayers] = {};  // act[l] = output of layer l-1 (l >= 1)
  __bf16 *dact[2] = {};       // gradient ping-pong (training only)
  __bf16 *dz = nullptr;       // gradient of the output, one value per voxel
  float *z = nullptr, *tgt = nullptr, *loss = nullptr;
  float *feat_tmp = nullptr;
  size_t feat_cap = 0;
};

namespace {

int nfail(cmi_net *n, int code, const std::string &m) {
  if (n) n->err = m;
  return code;
}

#define NET_TRY(n, call)                                                   \
  do {                                                                     \
    hipError_t e_ = (call);                                                \
    if (e_ != hipSuccess)                                                  \
      return nfail(n, CMI_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

int nout_of(int l) { return layer_cout(l) > 16 ? 32 : 16; }

// Work buffers for nvox voxels; the gradient's for training only.
int ensure_work(cmi_net *n, size_t nvox, bool training) {
  if (nvox > n->work_vox) {
    n->work_vox = 0;
    hipFree(n->in);
    n->in = nullptr;
    for (int l = 1; l < kLayers; ++l) {
      hipFree(n->act[l]);
      n->act[l] = nullptr;
    }
    hipFree(n->z);
    hipFree(n->tgt);
    n->z = n->tgt = nullptr;
    NET_TRY(n, hipMalloc(&n->in, nvox * sizeof(uint32_t)));
    for (int l = 1; l < kLayers; ++l)
      NET_TRY(n, hipMalloc(&n->act[l], nvox * kC * sizeof(__bf16)));
    NET_TRY(n, hipMalloc(&n->z, nvox * sizeof(float)));
    NET_TRY(n, hipMalloc(&n->tgt, nvox * sizeof(float)));
    n->work_vox = nvox;
  }
  if (training && nvox > n->grad_vox) {
    n->grad_vox = 0;
    for (int k = 0; k < 2; ++k) {
      hipFree(n->dact[k]);
      n->dact[k] = nullptr;
    }
    hipFree(n->dz);
    n->dz = nullptr;
    for (int k = 0; k < 2; ++k)
      NET_TRY(n, hipMalloc(&n->dact[k], nvox * kC * sizeof(__bf16)));
    NET_TRY(n, hipMalloc(&n->dz, nvox * sizeof(__bf16)));
    n->grad_vox = nvox;
  }
  return CMI_OK;
}

Layers layers_of(const cmi_net *n) {
  Layers L;
  for (int l = 0; l < kLayers; ++l) {
    L.off_w[l] = n->off_w[l];
    L.off_b[l] = n->off_b[l];
    L.nout[l] = nout_of(l);
    L.fwd[l] = n->wf[l];
    L.bwd[l] = n->wb[l];
  }
  return L;
}

int pack(cmi_net *n) {
  hipLaunchKernelGGL(pack_kernel, dim3(27, kLayers), dim3(256), 0, n->stream, n->p,
                     layers_of(n));
  NET_TRY(n, hipGetLastError());
  return CMI_OK;
}

// Blocks of bz x 8 x 8 voxels over B samples of D x H x W at a dilation.
//
// Packed: where blocks of one sub-lattice each are more than the chip takes at a
// time (two to a CU); fewer run side by side, and longer when packed.  Four
// layers of one dilation, not packed and packed: 8 x 128 x 128, dilation 8, 2048
// blocks 0.270 and 0.190 ms; 23 x 64 x 128, 8, 1024 blocks 0.232 and 0.224; 12 x
// 64 x 64, 8, 512 blocks 0.115 and 0.140; 16 x 16 x 64, 8, 512 blocks 0.086 and
// 0.120.
//
// Runs instead of blocks (by_runs): an inference is faster voxel run by voxel run
// (conv3_kernel, a tenth of the code) where the runs are about one to a SIMD (16 x
// 16 x 64, dilation 1, 1024 runs: blocks 0.095, runs 0.088 ms; 12 x 12 x 128, 2,
// 1152 runs 0.100 and 0.095; 9 x 31 x 96, 1, 1674 runs 0.101 and 0.105), and where
// voxels fill few of the blocks' positions: packed 0.22 of them (64 x 64 x 96, dilation 24) 0.70 and
// 0.60 ms, 0.30 (96^3, 36) 1.27 and 1.26, 0.39 (128^3, 43) 2.55 and 2.91; not
// packed, which leaves empty planes out, 0.15 (128^3, 30) 3.40 and 2.99, 0.22
// (96^3, 20) 1.24 and 1.31, 0.25 (64 x 64 x 128, 16) 0.66 and 0.79.  In training,
// where one step follows the other, runs are faster only where the blocks are
// also more than the chip takes at a time (8 steps on a crop of 8 x 8 x 32: blocks
// 1.11, runs forward and back 1.19 ms; 4 steps on two of 64^3 at dilations of 16,
// 4096 blocks: 5.97 and 4.77).
BlockGeo block_geo(const cmi_net *n, int B, int D, int H, int W, int dil, int bz) {
  BlockGeo G;
  G.D = D;
  G.H = H;
  G.W = W;
  G.dil = dil;
  // an axis: its residues (or groups of them), blocks and packing
  auto axis = [&](int extent, int edge, bool pack, int &nr, int &nb, Residues &P) {
    const int sub = (extent + dil - 1) / dil;
    P = Residues{std::min(dil, extent), 1, 0, 0};
    // as many sub-lattices as fit with an empty position between neighbours
    const int fit = std::min((edge + 1) / (sub + 1), P.res);
    if (pack && fit > 1) {
      P = Residues{P.res, fit, sub + 1, 256 / (sub + 1) + 1};
      G.packed = true;
    }
    nr = (P.res + P.per_block - 1) / P.per_block;
    nb = (sub + edge - 1) / edge;
  };
  auto blocks = [&](bool pack) {
    G.packed = false;
    axis(D, bz, pack, G.nrz, G.nbz, G.pz);
    axis(H, kE, pack, G.nry, G.nby, G.py);
    axis(W, kE, pack, G.nrx, G.nbx, G.px);
    G.nblocks = B * G.nrz * G.nry * G.nrx * G.nbz * G.nby * G.nbx;
  };
  blocks(false);
  if (G.nblocks > 2 * n->num_cus) blocks(true);
  const double voxels = (double)B * D * H * W;
  G.sparse = voxels < (G.packed ? 0.3 : 0.2) * G.nblocks * bz * kE * kE;
  G.few_runs = voxels <= 16. * 5. * n->num_cus;
  G.one_wave = G.nblocks <= 2 * n->num_cus;
  return G;
}

// Whether a 32-channel convolution goes run by run (block_geo).
bool by_runs(const BlockGeo &G, bool training) {
  return training ? G.sparse && !G.one_wave : G.sparse || G.few_runs;
}

unsigned grid_for(size_t items, unsigned per_block, unsigned cap = 65535) {
  size_t g = (items + per_block - 1) / per_block;
  if (g == 0) g = 1;
  return (unsigned)(g < cap ? g : cap);
}

// The network's input from the features of B whole volumes.
void input_features(cmi_net *n, const float *feat, int B, const int dim[3]) {
  const size_t nv = (size_t)dim[0] * dim[1] * dim[2];
  for (int b0 = 0; b0 < B; b0 += kMaxCrops) {
    const int nb = std::min(kMaxCrops, B - b0);
    Crops C{};
    for (int b = 0; b < nb; ++b) C.sample[b] = b0 + b;
    hipLaunchKernelGGL(crops_kernel, dim3(grid_for(nv, 256, 8192), nb), dim3(256), 0, n->stream,
                       feat, (const float *)nullptr, dim[0], dim[1], dim[2], C, dim[0], dim[1],
                       dim[2], n->mean[0], n->scale[0], n->mean[1], n->scale[1], 1.f,
                       n->in + (size_t)b0 * nv, (float *)nullptr);
  }
}

// forward over n->in (B samples of D x H x W) -> zout; training: a backward
// pass follows
int forward(cmi_net *n, int B, int D, int H, int W, float *zout, bool training) {
  if ((size_t)B * D * H * W == 0) return CMI_OK;  // nothing to compute, no empty grids
  const int nrun = B * D * H * (W / 16);
  const unsigned runs = grid_for((size_t)nrun, 4, 1u << 30);  // one wave per run
  for (int l = 0; l < kLayers; ++l) {
    const float *bias = n->p + n->off_b[l];
    const int dil = n->dil[l], relu = l < kLayers - 1;
    const __bf16 *const x = l == 0 ? reinterpret_cast<const __bf16 *>(n->in) : n->act[l];
    __bf16 *const y = relu ? n->act[l + 1] : nullptr;
    float *const yf = relu ? nullptr : zout;
    const BlockGeo G = block_geo(n, B, D, H, W, dil, kE);
    if (n->tiled && !by_runs(G, training)) {
      const bool pk = G.packed;
      auto *conv = pk ? conv_block_kernel<2, false, true> : conv_block_kernel<2, false, false>;
      if (l == 0)
        conv = pk ? conv_block_kernel<2, true, true> : conv_block_kernel<2, true, false>;
      else if (l == kLayers - 1)
        conv = pk ? conv_block_kernel<1, false, true> : conv_block_kernel<1, false, false>;
      hipLaunchKernelGGL(conv, dim3(G.nblocks), dim3(kConvThreads), 0, n->stream, G, x,
                         n->wf[l], bias, y, yf, (const __bf16 *)nullptr, relu);
      continue;
    }
    auto *run = conv3_kernel<2, false>;
    if (l == 0)
      run = conv3_kernel<2, true>;
    else if (l == kLayers - 1)
      run = conv3_kernel<1, false>;
    hipLaunchKernelGGL(run, dim3(runs), dim3(256), 0, n->stream, x, n->wf[l], bias, nrun, D, H,
                       W, dil, y, yf, (const __bf16 *)nullptr, relu);
  }
  NET_TRY(n, hipGetLastError());
  return CMI_OK;
}

void zero_grad(cmi_net *n) {
  hipLaunchKernelGGL(zero_f32_kernel, dim3(1024), dim3(256), 0, n->stream, n->g,
                     kCopies * n->grad_stride);
}

// Workgroups of a weight gradient: two per CU, the blocks shared out evenly.
unsigned grad_grid(const cmi_net *n, const BlockGeo &G) {
  const int most = 2 * n->num_cus;
  const int each = (G.nblocks + most - 1) / most;
  return (unsigned)((G.nblocks + each - 1) / each);
}

// backward from the MSE loss on z vs tgt; the loss and the gradients add into
// the copies in n->g
int backward(cmi_net *n, int B, int D, int H, int W) {
  static_assert(kLayers >= 3, "a first, a last and layers between");
  const size_t nvox = (size_t)B * D * H * W;
  const uint16_t *const dz = reinterpret_cast<const uint16_t *>(n->dz);
  const int last = kLayers - 1;
  const int nrun = B * D * H * (W / 16);
  const unsigned runs = grid_for((size_t)nrun, 4, 1u << 30);  // one wave per run
  hipLaunchKernelGGL(mse_kernel, dim3(grid_for(nvox, 1024, 512)), dim3(256), 0, n->stream,
                     n->z, n->tgt, nvox, n->w_pos, n->dz, n->g, n->grad_stride, n->nparam,
                     n->off_b[last]);
  __bf16 *dy = n->dact[0], *dx = n->dact[1];
  // without voxels the mean loss is NaN and the gradients stay 0
  for (int l = nvox ? last : -1; l >= 0; --l) {
    const BlockGeo Gw = block_geo(n, B, D, H, W, n->dil[l], kGZ);
    const BlockGeo Gx = block_geo(n, B, D, H, W, n->dil[l], kE);
    const unsigned wg = grad_grid(n, Gw);
    if (l == last) {
      auto *wgrad = Gw.packed ? wgrad_last_kernel<true> : wgrad_last_kernel<false>;
      hipLaunchKernelGGL(wgrad, dim3(wg), dim3(kGThreads), 0, n->stream, Gw, dz, n->act[l],
                         n->g, n->grad_stride, n->off_w[l], nout_of(l));
      auto *dgrad = Gx.packed ? dgrad_last_kernel<true> : dgrad_last_kernel<false>;
      hipLaunchKernelGGL(dgrad, dim3(Gx.nblocks), dim3(kConvThreads), 0, n->stream, Gx, dz,
                         n->wb[l], n->act[l], dy);
      continue;
    }
    if (l == 0) {
      auto *wgrad = Gw.packed ? wgrad_first_kernel<true> : wgrad_first_kernel<false>;
      hipLaunchKernelGGL(wgrad, dim3(wg), dim3(kGThreads), 0, n->stream, Gw, dy, n->in, n->g,
                         n->grad_stride, n->off_w[l], n->off_b[l]);
      continue;
    }
    auto *wgrad = Gw.packed ? wgrad_block_kernel<true> : wgrad_block_kernel<false>;
    hipLaunchKernelGGL(wgrad, dim3(wg), dim3(kGThreads), 0, n->stream, Gw, dy, n->act[l], n->g,
                       n->grad_stride, n->off_w[l], n->off_b[l]);
    // dx = conv(dy, flipped transposed W), masked by the ReLU of layer l-1
    if (by_runs(Gx, true)) {
      hipLaunchKernelGGL((conv3_kernel<2, false>), dim3(runs), dim3(256), 0, n->stream, dy,
                         n->wb[l], (const float *)nullptr, nrun, D, H, W, n->dil[l], dx,
                         (float *)nullptr, n->act[l], 0);
    } else {
      auto *conv =
          Gx.packed ? conv_block_kernel<2, false, true> : conv_block_kernel<2, false, false>;
      hipLaunchKernelGGL(conv, dim3(Gx.nblocks), dim3(kConvThreads), 0, n->stream, Gx, dy,
                         n->wb[l], (const float *)nullptr, dx, (float *)nullptr, n->act[l], 0);
    }
    std::swap(dy, dx);
  }
  NET_TRY(n, hipGetLastError());
  return CMI_OK;
}

}  // namespace

extern "C" {

int cmi_net_create(uint64_t seed, cmi_net **out) {
  if (!out) return CMI_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return CMI_ERR_NODEVICE;
  cmi_net *n = new cmi_net();
  (void)hipGetDevice(&n->device);
  if (hipDeviceGetAttribute(&n->num_cus, hipDeviceAttributeMultiprocessorCount, n->device) !=
      hipSuccess) {
    delete n;
    return CMI_ERR_HIP;
  }
  size_t off = 0;
  for (int l = 0; l < kLayers; ++l) {
    n->off_w[l] = off;
    off += (size_t)kTaps * nout_of(l) * kC;
    n->off_b[l] = off;
    off += nout_of(l);
  }
  n->nparam = off;
  hipError_t e = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc(&n->p, off * sizeof(float));
  n->grad_stride = (off + 1 + 63) / 64 * 64;
  if (e == hipSuccess) e = hipMalloc(&n->g, kCopies * n->grad_stride * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&n->grad_sum, n->grad_stride * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&n->m, off * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&n->v, off * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&n->loss, 65536 * sizeof(float));
  for (int l = 0; l < kLayers && e == hipSuccess; ++l) {
    e = hipMalloc(&n->wf[l], (size_t)kTaps * nout_of(l) * kC * sizeof(__bf16));
    if (e == hipSuccess) e = hipMalloc(&n->wb[l], (size_t)kTaps * 32 * kC * sizeof(__bf16));
  }
  if (e != hipSuccess) {
    cmi_net_destroy(n);
    return CMI_ERR_ALLOC;
  }
  // He-uniform initial weights over the real fan-in, zero biases, from a
  // Philox stream
  std::vector<float> h(off, 0.f);
  uint64_t ctr = 0;
  for (int l = 0; l < kLayers; ++l) {
    const float bound = sqrtf(6.f / (kTaps * layer_cin(l))) * (l == kLayers - 1 ? 0.5f : 1.f);
    const int NOUT = nout_of(l);
    for (int tap = 0; tap < kTaps; ++tap)
      for (int o = 0; o < layer_cout(l); ++o)
        for (int k = 0; k < layer_cin(l); ++k) {
          const u32x4 r = philox4x32_10(u32x4{(uint32_t)ctr, (uint32_t)(ctr >> 32), 0xC0u, 0u},
                                        (uint32_t)seed, (uint32_t)(seed >> 32));
          ++ctr;
          const double u = uniform_open(r.x, r.y);
          h[n->off_w[l] + ((size_t)tap * NOUT + o) * kC + k] = (float)((2. * u - 1.) * bound);
        }
  }
  e = hipMemcpy(n->p, h.data(), off * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(n->m, 0, off * sizeof(float));
  if (e == hipSuccess) e = hipMemset(n->v, 0, off * sizeof(float));
  if (e != hipSuccess || pack(n) != CMI_OK || hipStreamSynchronize(n->stream) != hipSuccess) {
    cmi_net_destroy(n);
    return CMI_ERR_HIP;
  }
  *out = n;
  return CMI_OK;
}

void cmi_net_destroy(cmi_net *n) {
  if (!n) return;
  (void)hipSetDevice(n->device);
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  hipFree(n->p);
  hipFree(n->g);
  hipFree(n->grad_sum);
  hipFree(n->m);
  hipFree(n->v);
  hipFree(n->loss);
  for (int l = 0; l < kLayers; ++l) {
    hipFree(n->wf[l]);
    hipFree(n->wb[l]);
    hipFree(n->act[l]);
  }
  hipFree(n->in);
  for (int k = 0; k < 2; ++k) hipFree(n->dact[k]);
  hipFree(n->dz);
  hipFree(n->z);
  hipFree(n->tgt);
  hipFree(n->ds_feat);
  hipFree(n->ds_tgt);
  hipFree(n->feat_tmp);
  if (n->stream) (void)hipStreamDestroy(n->stream);
  delete n;
}

const char *cmi_net_last_error(const cmi_net *n) { return n ? n->err.c_str() : "null net"; }

size_t cmi_net_param_count(const cmi_net *n) { return n ? n->nparam : 0; }

int cmi_net_get_params(cmi_net *n, float *out) {
  if (!n || !out) return CMI_ERR_ARG;
  (void)hipSetDevice(n->device);
  NET_TRY(n, hipStreamSynchronize(n->stream));
  NET_TRY(n, hipMemcpy(out, n->p, n->nparam * sizeof(float), hipMemcpyDeviceToHost));
  return CMI_OK;
}

int cmi_net_set_params(cmi_net *n, const float *in) {
  if (!n || !in) return CMI_ERR_ARG;
  (void)hipSetDevice(n->device);
  NET_TRY(n, hipStreamSynchronize(n->stream));  // null-stream copies below
  NET_TRY(n, hipMemcpy(n->p, in, n->nparam * sizeof(float), hipMemcpyHostToDevice));
  NET_TRY(n, hipMemset(n->m, 0, n->nparam * sizeof(float)));
  NET_TRY(n, hipMemset(n->v, 0, n->nparam * sizeof(float)));
  n->step = 0;
  const int rc = pack(n);
  if (rc != CMI_OK) return rc;
  NET_TRY(n, hipStreamSynchronize(n->stream));
  return CMI_OK;
}

int cmi_net_set_normalisation(cmi_net *n, const float mean[2], const float scale[2],
                              float logit_scale) {
  if (!n || !mean || !scale || !(logit_scale > 0.f)) return CMI_ERR_ARG;
  n->out_scale = logit_scale;
  for (int c = 0; c < 2; ++c) {
    n->mean[c] = mean[c];
    n->scale[c] = scale[c];
  }
  return CMI_OK;
}

int cmi_net_add_samples(cmi_net *n, const float *feat, const float *target, int nsamples,
                        const int dim[3]) {
  if (!n || !feat || !target || nsamples <= 0 || !dim) return CMI_ERR_ARG;
  (void)hipSetDevice(n->device);
  NET_TRY(n, hipStreamSynchronize(n->stream));  // null-stream copies below
  if (n->ds_n > 0 && (dim[0] != n->ds_dim[0] || dim[1] != n->ds_dim[1] || dim[2] != n->ds_dim[2]))
    return nfail(n, CMI_ERR_ARG, "all samples must have the same shape");
  const size_t nv = (size_t)dim[0] * dim[1] * dim[2];
  const size_t need = (size_t)(n->ds_n + nsamples);
  if (need > n->ds_cap) {
    size_t cap = std::max(need, 2 * n->ds_cap);
    float *f2 = nullptr, *t2 = nullptr;
    NET_TRY(n, hipMalloc(&f2, cap * nv * 2 * sizeof(float)));
    NET_TRY(n, hipMalloc(&t2, cap * nv * sizeof(float)));
    if (n->ds_n) {
      NET_TRY(n, hipMemcpy(f2, n->ds_feat, (size_t)n->ds_n * nv * 2 * sizeof(float),
                           hipMemcpyDeviceToDevice));
      NET_TRY(n, hipMemcpy(t2, n->ds_tgt, (size_t)n->ds_n * nv * sizeof(float),
                           hipMemcpyDeviceToDevice));
    }
    hipFree(n->ds_feat);
    hipFree(n->ds_tgt);
    n->ds_feat = f2;
    n->ds_tgt = t2;
    n->ds_cap = cap;
  }
  NET_TRY(n, hipMemcpy(n->ds_feat + (size_t)n->ds_n * nv * 2, feat,
                       (size_t)nsamples * nv * 2 * sizeof(float), hipMemcpyHostToDevice));
  NET_TRY(n, hipMemcpy(n->ds_tgt + (size_t)n->ds_n * nv, target,
                       (size_t)nsamples * nv * sizeof(float), hipMemcpyHostToDevice));
  for (int a = 0; a < 3; ++a) n->ds_dim[a] = dim[a];
  n->ds_n += nsamples;
  return CMI_OK;
}

int cmi_net_sample_count(const cmi_net *n) { return n ? n->ds_n : 0; }

int cmi_net_set_dilation(cmi_net *n, const int dilation[4]) {
  if (!n || !dilation) return CMI_ERR_ARG;
  for (int l = 0; l < kLayers; ++l)
    if (dilation[l] < 1 || dilation[l] > 64) return nfail(n, CMI_ERR_ARG, "dilation must be 1..64");
  for (int l = 0; l < kLayers; ++l) n->dil[l] = dilation[l];
  return CMI_OK;
}

int cmi_net_set_input_mode(cmi_net *n, int mode) {
  if (!n || (mode != 0 && mode != 1)) return CMI_ERR_ARG;
  n->mode = mode;
  return CMI_OK;
}

int cmi_net_get_input_mode(const cmi_net *n) { return n ? n->mode : -1; }

int cmi_net_set_tiled(cmi_net *n, int on) {
  if (!n) return CMI_ERR_ARG;
  n->tiled = on ? 1 : 0;
  return CMI_OK;
}

int cmi_net_set_loss_weight(cmi_net *n, float w_too_neutral) {
  if (!n || !(w_too_neutral > 0.f)) return CMI_ERR_ARG;
  n->w_pos = w_too_neutral;
  return CMI_OK;
}

int cmi_net_set_start_rule(cmi_net *n, float logit_cut, double fallback_xn) {
  if (!n || !(fallback_xn > 0. && fallback_xn <= 1.) || logit_cut != logit_cut)
    return CMI_ERR_ARG;
  n->cut = logit_cut;
  n->fallback = fallback_xn;
  return CMI_OK;
}

int cmi_net_get_start_rule(const cmi_net *n, float *logit_cut, double *fallback_xn) {
  if (!n || !logit_cut || !fallback_xn) return CMI_ERR_ARG;
  *logit_cut = n->cut;
  *fallback_xn = n->fallback;
  return CMI_OK;
}

int cmi_net_get_dilation(const cmi_net *n, int dilation[4]) {
  if (!n || !dilation) return CMI_ERR_ARG;
  for (int l = 0; l < kLayers; ++l) dilation[l] = n->dil[l];
  return CMI_OK;
}

int cmi_net_train(cmi_net *n, int steps, int batch, const int crop[3], float lr,
                  uint64_t seed, float *losses) {
  if (!n || steps <= 0 || steps > 65536 || batch <= 0 || !crop || !(lr > 0.f))
    return nfail(n, CMI_ERR_ARG, "bad training arguments");
  if (n->ds_n == 0) return nfail(n, CMI_ERR_STATE, "no samples");
  for (int a = 0; a < 3; ++a)
    if (crop[a] <= 0 || crop[a] > n->ds_dim[a]) return nfail(n, CMI_ERR_ARG, "crop larger than samples");
  if (crop[2] % 32 != 0) return nfail(n, CMI_ERR_ARG, "crop: last extent must be a multiple of 32");
  (void)hipSetDevice(n->device);
  const size_t cv = (size_t)crop[0] * crop[1] * crop[2];
  int rc = ensure_work(n, cv * batch, true);
  if (rc != CMI_OK) return rc;
  const float b1 = 0.9f, b2 = 0.999f;
  for (int s = 0; s < steps; ++s) {
    for (int b0 = 0; b0 < batch; b0 += kMaxCrops) {
      const int nb = std::min(kMaxCrops, batch - b0);
      Crops C{};
      for (int b = 0; b < nb; ++b) {
        const u32x4 r =
            philox4x32_10(u32x4{(uint32_t)s, (uint32_t)(b0 + b), (uint32_t)n->step, 0x7A1Eu},
                          (uint32_t)seed, (uint32_t)(seed >> 32));
        C.sample[b] = (int)(r.x % (uint32_t)n->ds_n);
        C.d[b] = (int)(r.y % (uint32_t)(n->ds_dim[0] - crop[0] + 1));
        C.h[b] = (int)(r.z % (uint32_t)(n->ds_dim[1] - crop[1] + 1));
        C.w[b] = (int)(r.w % (uint32_t)(n->ds_dim[2] - crop[2] + 1));
      }
      hipLaunchKernelGGL(crops_kernel, dim3(grid_for(cv, 256, 4096), nb), dim3(256), 0,
                         n->stream, n->ds_feat, n->ds_tgt, n->ds_dim[0], n->ds_dim[1],
                         n->ds_dim[2], C, crop[0], crop[1], crop[2], n->mean[0], n->scale[0],
                         n->mean[1], n->scale[1], 1.f / n->out_scale, n->in + (size_t)b0 * cv,
                         n->tgt + (size_t)b0 * cv);
    }
    zero_grad(n);
    rc = forward(n, batch, crop[0], crop[1], crop[2], n->z, true);
    if (rc != CMI_OK) return rc;
    rc = backward(n, batch, crop[0], crop[1], crop[2]);
    if (rc != CMI_OK) return rc;
    ++n->step;
    const float c1 = 1.f - powf(b1, (float)n->step), c2 = 1.f - powf(b2, (float)n->step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid_for(n->nparam, 256, 1024)), dim3(256), 0,
                       n->stream, n->p, n->g, n->grad_stride, n->m, n->v, n->nparam, lr, b1, b2,
                       1e-8f, c1, c2, 0.f, layers_of(n), n->loss + s);
  }
  NET_TRY(n, hipGetLastError());
  if (losses)
    NET_TRY(n, hipMemcpyAsync(losses, n->loss, steps * sizeof(float), hipMemcpyDeviceToHost,
                              n->stream));
  NET_TRY(n, hipStreamSynchronize(n->stream));
  return CMI_OK;
}

// One forward + backward on the given batch (features [B][D][H][W][2]
// log10 n_H, log10 jH; targets [B][D][H][W] logits): the loss and the FP32
// gradient of every master parameter, no update.
int cmi_net_loss_and_grad(cmi_net *n, const float *feat, const float *target, int B,
                          const int dim[3], float *loss, float *grad) {
  if (!n || !feat || !target || B <= 0 || !dim) return CMI_ERR_ARG;
  if (dim[0] < 0 || dim[1] < 0 || dim[2] < 0) return nfail(n, CMI_ERR_ARG, "negative extent");
  if (dim[2] % 32 != 0) return nfail(n, CMI_ERR_ARG, "last extent must be a multiple of 32");
  (void)hipSetDevice(n->device);
  NET_TRY(n, hipStreamSynchronize(n->stream));  // null-stream copies below
  const size_t nv = (size_t)dim[0] * dim[1] * dim[2];
  int rc = ensure_work(n, nv * B, true);
  if (rc != CMI_OK) return rc;
  std::vector<float> ts(target, target + nv * B);
  for (float &t : ts) t /= n->out_scale;
  float *df = nullptr;
  NET_TRY(n, hipMalloc(&df, nv * B * 2 * sizeof(float)));
  hipError_t e = hipMemcpy(df, feat, nv * B * 2 * sizeof(float), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(n->tgt, ts.data(), nv * B * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    hipFree(df);
    return nfail(n, CMI_ERR_HIP, "loss_and_grad: copy failed");
  }
  input_features(n, df, B, dim);
  zero_grad(n);
  rc = forward(n, B, dim[0], dim[1], dim[2], n->z, true);
  if (rc == CMI_OK) rc = backward(n, B, dim[0], dim[1], dim[2]);
  if (rc == CMI_OK) {
    hipLaunchKernelGGL(sum_grad_kernel, dim3(grid_for(n->nparam, 256, 1024)), dim3(256), 0,
                       n->stream, n->g, n->grad_stride, n->nparam, n->grad_sum);
    e = hipMemcpyAsync(grad, n->grad_sum, n->nparam * sizeof(float), hipMemcpyDeviceToHost,
                       n->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(loss, n->grad_sum + n->nparam, sizeof(float), hipMemcpyDeviceToHost,
                         n->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    if (e != hipSuccess) rc = nfail(n, CMI_ERR_HIP, "loss_and_grad failed");
  }
  hipFree(df);
  return rc;
}

// Logits of x_n for one grid (features [D][H][W][2]).
int cmi_net_predict(cmi_net *n, const float *feat, const int dim[3], float *logits) {
  if (!n || !feat || !dim || !logits) return CMI_ERR_ARG;
  if (dim[0] < 0 || dim[1] < 0 || dim[2] < 0) return nfail(n, CMI_ERR_ARG, "negative extent");
  if (dim[2] % 32 != 0) return nfail(n, CMI_ERR_ARG, "last extent must be a multiple of 32");
  (void)hipSetDevice(n->device);
  NET_TRY(n, hipStreamSynchronize(n->stream));  // null-stream copies below
  const size_t nv = (size_t)dim[0] * dim[1] * dim[2];
  int rc = ensure_work(n, nv, false);
  if (rc != CMI_OK) return rc;
  if (n->feat_cap < nv) {
    hipFree(n->feat_tmp);
    n->feat_tmp = nullptr;
    n->feat_cap = 0;
    NET_TRY(n, hipMalloc(&n->feat_tmp, nv * 2 * sizeof(float)));
    n->feat_cap = nv;
  }
  NET_TRY(n, hipMemcpy(n->feat_tmp, feat, nv * 2 * sizeof(float), hipMemcpyHostToDevice));
  input_features(n, n->feat_tmp, 1, dim);
  rc = forward(n, 1, dim[0], dim[1], dim[2], n->z, false);
  if (rc != CMI_OK) return rc;
  NET_TRY(n, hipMemcpyAsync(logits, n->z, nv * sizeof(float), hipMemcpyDeviceToHost, n->stream));
  NET_TRY(n, hipStreamSynchronize(n->stream));
  for (size_t v = 0; v < nv; ++v) logits[v] *= n->out_scale;
  return CMI_OK;
}

namespace {

// jH = jconv * J of a context's stored intensity (J is kept in units of
// sigma * Delta_0 in FP32 contexts)
double context_jconv(const cmi_ctx *c, double luminosity, uint64_t npackets) {
  double j = luminosity / (double)npackets * c->g.inv_cell_size[0] * c->g.inv_cell_size[1] *
             c->g.inv_cell_size[2];
  if (c->precision != CMI_PREC_FP64) j *= c->sigma * c->g.cell_size[0];
  return j;
}

int check_context(cmi_net *n, const cmi_ctx *c, double luminosity, uint64_t npackets) {
  if (!c || npackets == 0 || !(luminosity > 0.))
    return nfail(n, CMI_ERR_ARG, "bad warm-start arguments");
  if (c->device != n->device) return nfail(n, CMI_ERR_ARG, "context on another device");
  return CMI_OK;
}

}  // namespace

int cmi_net_warm_start(cmi_net *n, cmi_ctx *c, double luminosity, uint64_t npackets) {
  if (!n) return CMI_ERR_ARG;
  int rc = check_context(n, c, luminosity, npackets);
  if (rc != CMI_OK) return rc;
  const int D = c->ncell[0], H = c->ncell[1], W = c->ncell[2];
  if (W % 16 != 0) return nfail(n, CMI_ERR_ARG, "ncell[2] must be a multiple of 16");
  (void)hipSetDevice(n->device);
  const size_t nv = (size_t)D * H * W;
  rc = ensure_work(n, nv, false);
  if (rc != CMI_OK) return rc;
  NET_TRY(n, hipStreamSynchronize(c->stream));  // the first pass has finished
  hipLaunchKernelGGL(ctx_features_kernel, dim3(grid_for(nv, 256, 8192)), dim3(256), 0,
                     n->stream, c->g, (const double *)c->f.n, (const double *)c->f.J,
                     (const double *)c->f.xn, n->mode, D, H, W,
                     context_jconv(c, luminosity, npackets), n->mean[0], n->scale[0],
                     n->mean[1], n->scale[1], n->in, (float *)nullptr);
  rc = forward(n, 1, D, H, W, n->z, false);
  if (rc != CMI_OK) return rc;
  const bool fp32 = c->precision == CMI_PREC_FP32;
  hipLaunchKernelGGL(ctx_apply_kernel, dim3(grid_for(nv, 256, 8192)), dim3(256), 0, n->stream,
                     c->g, (const float *)n->z, n->mode, D, H, W, n->out_scale, n->cut,
                     n->fallback,
                     (const double *)c->f.n,
                     c->f.xn, c->f.J, fp32 ? c->f.kappa : (float *)nullptr,
                     c->sigma * c->g.cell_size[0]);
  NET_TRY(n, hipGetLastError());
  NET_TRY(n, hipStreamSynchronize(n->stream));
  return CMI_OK;
}

// A coarse context of the same box with ncell f times smaller per axis
// (f >= 2), on the same device; returns f or 0.
static int coarse_factor(const cmi_ctx *fine, const cmi_ctx *coarse) {
  if (!fine || !coarse || fine->device != coarse->device) return 0;
  const int f = fine->ncell[0] / coarse->ncell[0];
  if (f < 2) return 0;
  for (int a = 0; a < 3; ++a) {
    if (coarse->ncell[a] * f != fine->ncell[a]) return 0;
    if (fine->box[a] != coarse->box[a] || fine->box[3 + a] != coarse->box[3 + a]) return 0;
  }
  return f;
}

// What is queued on `reader`'s stream reads `source`'s fields: work that
// `source` gets from here on waits for it.
static hipError_t hold_fields(cmi_ctx *source, cmi_ctx *reader) {
  hipError_t e = hipSuccess;
  if (!reader->ev_read) e = hipEventCreateWithFlags(&reader->ev_read, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventRecord(reader->ev_read, reader->stream);
  if (e == hipSuccess) e = hipStreamWaitEvent(source->stream, reader->ev_read, 0);
  return e;
}

int cmi_restrict_density(cmi_ctx *fine, cmi_ctx *coarse) {
  const int f = coarse_factor(fine, coarse);
  if (!f)
    return coarse ? fail(coarse, CMI_ERR_ARG,
                         "restrict: the coarse grid must be the fine one's box with "
                         "ncell an integer factor >= 2 smaller per axis, on its device")
                  : CMI_ERR_ARG;
  (void)hipSetDevice(coarse->device);
  // the fine context's stream has written its fields
  CMI_TRY_HIP(fine, hipStreamSynchronize(fine->stream));
  const size_t nv = (size_t)coarse->ncell[0] * coarse->ncell[1] * coarse->ncell[2];
  const bool fp32 = coarse->precision == CMI_PREC_FP32;
  hipLaunchKernelGGL(restrict_density_kernel, dim3(grid_for(nv, 256, 8192)), dim3(256), 0,
                     coarse->stream, fine->g, (const double *)fine->f.n, coarse->g, f,
                     coarse->ncell[0], coarse->ncell[1], coarse->ncell[2], coarse->f.n,
                     coarse->f.xn, coarse->f.J, fp32 ? coarse->f.kappa : (float *)nullptr,
                     coarse->sigma * coarse->g.cell_size[0]);
  CMI_TRY_HIP(coarse, hipGetLastError());
  CMI_TRY_HIP(coarse, hold_fields(fine, coarse));
  return CMI_OK;
}

int cmi_prolong_neutral_fraction(cmi_ctx *coarse, cmi_ctx *fine) {
  const int f = coarse_factor(fine, coarse);
  if (!f)
    return fine ? fail(fine, CMI_ERR_ARG,
                       "prolong: the coarse grid must be the fine one's box with "
                       "ncell an integer factor >= 2 smaller per axis, on its device")
                : CMI_ERR_ARG;
  (void)hipSetDevice(fine->device);
  CMI_TRY_HIP(coarse, hipStreamSynchronize(coarse->stream));
  const size_t nv = (size_t)fine->ncell[0] * fine->ncell[1] * fine->ncell[2];
  const bool fp32 = fine->precision == CMI_PREC_FP32;
  hipLaunchKernelGGL(prolong_xn_kernel, dim3(grid_for(nv, 256, 8192)), dim3(256), 0,
                     fine->stream, coarse->g, (const double *)coarse->f.xn, f,
                     coarse->ncell[0], coarse->ncell[1], coarse->ncell[2], fine->g,
                     (const double *)fine->f.n, fine->f.xn, fine->f.J,
                     fp32 ? fine->f.kappa : (float *)nullptr,
                     fine->sigma * fine->g.cell_size[0]);
  CMI_TRY_HIP(fine, hipGetLastError());
  CMI_TRY_HIP(fine, hold_fields(coarse, fine));
  return CMI_OK;
}

int cmi_net_context_features(cmi_net *n, cmi_ctx *c, double luminosity, uint64_t npackets,
                             float *features) {
  if (!n || !features) return CMI_ERR_ARG;
  int rc = check_context(n, c, luminosity, npackets);
  if (rc != CMI_OK) return rc;
  (void)hipSetDevice(n->device);
  const int D = c->ncell[0], H = c->ncell[1], W = c->ncell[2];
  const size_t nv = (size_t)D * H * W;
  float *d = nullptr;
  NET_TRY(n, hipStreamSynchronize(c->stream));
  NET_TRY(n, hipMalloc(&d, nv * 2 * sizeof(float)));
  hipLaunchKernelGGL(ctx_features_kernel, dim3(grid_for(nv, 256, 8192)), dim3(256), 0,
                     n->stream, c->g, (const double *)c->f.n, (const double *)c->f.J,
                     (const double *)c->f.xn, n->mode, D, H, W,
                     context_jconv(c, luminosity, npackets), 0.f, 1.f, 0.f, 1.f,
                     (uint32_t *)nullptr, d);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(features, d, nv * 2 * sizeof(float), hipMemcpyDeviceToHost, n->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
  hipFree(d);
  if (e != hipSuccess) return nfail(n, CMI_ERR_HIP, std::string("context features: ") + hipGetErrorString(e));
  return CMI_OK;
}

}  // extern "C"
