// The initial-guess network of the learned solve (no reference counterpart).
//
// Six 3 x 3 x 3 convolutions, 3 -> 32 -> 32 -> 32 -> 32 -> 32 -> 1 channels,
// GELU after the first five, bias on every layer; fields are periodic in x
// and y and zero beyond the walls in z, like the pressure operator.  Every
// layer's forward runs as an implicit GEMM on the bf16 matrix cores
// (v_mfma_f32_32x32x16_bf16, FP32 accumulation) over an input brick staged
// in LDS (k_brick); weights and activations are bf16, the network's input is
// rounded to bf16 on staging.  The backward pass reuses the 32 -> 32 kernel
// for the input gradient (transposed, tap-flipped weights) and has its own
// MFMA kernels for the weight gradients (GEMMs over the voxels, split into
// groups of bricks whose partial sums are added in a fixed order; FP32 MFMA
// in the first and last layers); the last layer's input gradient runs on the
// vector units from the FP32 master weights.
//
// Layout: activations are channels-last [voxel][channel] with voxel =
// i + nx (j + ny k); parameters are one FP32 vector, layer by layer W[27][cout][cin]
// then b[cout], tap t = (dx + 1) + 3 (dy + 1) + 9 (dz + 1) weighing the input
// at (i + dx, j + dy, k + dz).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "pcf_internal.hpp"
#include "solver_common.hpp"

namespace pcf {

namespace {

typedef __bf16 bf16;
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kC = 32;        // hidden channels
constexpr int kLayers = 6;
constexpr int kCin[kLayers] = {3, 32, 32, 32, 32, 32};
constexpr int kCout[kLayers] = {32, 32, 32, 32, 32, 1};

__host__ __device__ constexpr int layer_size(int l) { return 27 * kCout[l] * kCin[l] + kCout[l]; }
__host__ __device__ constexpr int layer_offset(int l) {
  int o = 0;
  for (int q = 0; q < l; ++q) o += layer_size(q);
  return o;
}
constexpr int kParams = layer_offset(kLayers);

struct Dims {
  int nx, ny, nz;
  size_t n;
};

// Voxel index of the neighbour at tap t of voxel (i, j, k); -1 beyond the walls.
__device__ __forceinline__ long long neighbour(const Dims& d, int i, int j, int k, int t) {
  const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
  const int kk = k + dz;
  if (kk < 0 || kk >= d.nz) return -1;
  int ii = i + dx, jj = j + dy;
  ii = ii < 0 ? ii + d.nx : (ii >= d.nx ? ii - d.nx : ii);
  jj = jj < 0 ? jj + d.ny : (jj >= d.ny ? jj - d.ny : jj);
  return (long long)ii + (long long)d.nx * (jj + (long long)d.ny * kk);
}

// (i, j, k) of voxel p in 32-bit arithmetic: pcf_net_create admits at most
// 2^31 - 1 voxels
__device__ __forceinline__ void coords(const Dims& d, size_t p, int& i, int& j, int& k) {
  const unsigned q = (unsigned)p, nx = (unsigned)d.nx, ny = (unsigned)d.ny;
  const unsigned r = q / nx;
  i = (int)(q - r * nx);
  j = (int)(r % ny);
  k = (int)(r / ny);
}

// GELU x Phi(x) = x (1 + erf(x / sqrt 2)) / 2 with 1 + erf(z) from the
// rational approximation of Abramowitz and Stegun 7.1.26 (|error of erf| <=
// 1.5e-7): for z >= 0, 1 + erf(z) = 2 - q, for z < 0 it is q itself, with
// q = t (a1 + t (a2 + ...)) exp(-z^2), t = 1 / (1 + p |z|), so the negative
// side has no cancellation.  Branch-free, about a dozen instructions; the
// activations are rounded to bf16 (relative 3.9e-3) right after, far above
// its 6.2e-7 absolute error (measured against erf on [-12, 12]).
__device__ __forceinline__ float gelu(float x) {
  const float z = x * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * fabsf(z));
  float p = 1.061405429f;
  p = fmaf(p, t, -1.453152027f);
  p = fmaf(p, t, 1.421413741f);
  p = fmaf(p, t, -0.284496736f);
  p = fmaf(p, t, 0.254829592f);
  const float q = p * t * __builtin_amdgcn_exp2f(-(z * z) * 1.4426950408889634f);
  return 0.5f * x * (z >= 0.0f ? 2.0f - q : q);
}
__device__ __forceinline__ float gelu_grad(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * expf(-0.5f * x * x) * 0.39894228040143268f;
}

// ---- the convolutions on the matrix cores (v_mfma_f32_32x32x16_bf16, FP32
// accumulation).  Operand layout: lane l holds A[l % 32][8 (l / 32) + e] and
// B[8 (l / 32) + e][l % 32], e = 0..7, and D[8 (q / 4) + 4 (l / 32) + q % 4][l % 32],
// q = 0..15.  A row is the output channel, a column one of 32 voxels
// consecutive in x (nx is a multiple of 32), K runs over input channels (and,
// for the first layer, taps).
//
// A workgroup of 4 wavefronts computes a block of 32 (x) x 4 (y) x 4 (z)
// voxels.  Its input brick, the block with a one-voxel halo (34 x 6 x 6
// voxels, periodic in x and y, zero beyond the walls in z), is staged in LDS
// once as bf16; each wavefront computes 2 (y) x 2 (z) rows of 32 voxels, so
// one B operand read from LDS (the input row at one (y, z), shifted by dx)
// feeds the MFMAs of every output row of the wavefront whose 3 x 3 x 3
// neighbourhood holds that row (up to four).  The A operands of one (dx,
// channel half) -- nine taps -- stay in registers over the 16 input rows.
// Blocks are numbered so that each XCD (blocks are dealt to the 8 XCDs in
// turn) gets a contiguous range of neighbouring blocks, whose halos its L2
// then shares.
//
// KIND_FIRST: 3 -> 32, K = 27 taps x 3 channels padded to 96; the brick holds
//   the FP32 input rounded to bf16, 4 channels (8 B) per voxel.
// KIND_MID:   32 -> 32 (FWD: W x + bias -> z (FP32, may be null), gelu -> a
//   (bf16); DATA: W x -> g (FP32), the input gradient with transposed,
//   tap-flipped W).
// KIND_LAST:  32 -> 1, the 32 x 32 MFMA with only row 0 of A nonzero; out (FP32).
enum { KIND_FIRST = 0, KIND_MID = 1, KIND_LAST = 2 };
enum { MID_FWD = 0, MID_DATA = 1 };
constexpr int kBX = 34, kBY = 6, kBZ = 6, kBrickVox = kBX * kBY * kBZ;  // 1224 voxels
constexpr int kK1 = 96;  // padded K of the first layer

struct BrickGrid {
  int tiles_x, tiles_y, tiles_z;
};

// 16-byte chunk c (0..3) of brick voxel v, XOR-swizzled over neighbouring
// voxels so that 8 lanes reading one chunk of consecutive voxels hit distinct banks
__device__ __forceinline__ int brick_chunk(int v, int c) { return 4 * v + (c ^ ((v >> 1) & 3)); }

__device__ __forceinline__ int wrap(int q, int n) {
  q %= n;
  return q < 0 ? q + n : q;
}

__device__ __forceinline__ bf8 as_bf8(uint4 u) {
  bf8 r;
  __builtin_memcpy(&r, &u, sizeof(r));
  return r;
}

__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  bf16 h[4] = {(bf16)a, (bf16)b, (bf16)c, (bf16)d};
  uint2 r;
  __builtin_memcpy(&r, h, sizeof(r));
  return r;
}

template <int KIND, int MODE>
__global__ void __launch_bounds__(256, 2) k_brick(Dims d, BrickGrid bg, const void* __restrict__ in_,
                                                  const bf16* __restrict__ W, const float* __restrict__ bias,
                                                  float* zout, bf16* aout, float* gout) {
  __shared__ uint4 brick[KIND == KIND_FIRST ? kBrickVox / 2 : kBrickVox * 4];
  const int nb = (int)gridDim.x;
  int b = (int)blockIdx.x;
  if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
  const int tx = b % bg.tiles_x, tyz = b / bg.tiles_x, ty = tyz % bg.tiles_y, tz = tyz / bg.tiles_y;
  const int x0 = 32 * tx, y0 = 4 * ty, z0 = 4 * tz;

  // ---- stage the input brick
  if (KIND == KIND_FIRST) {
    const float* in = static_cast<const float*>(in_);
    uint2* br = reinterpret_cast<uint2*>(brick);
    for (int v = threadIdx.x; v < kBrickVox; v += 256) {
      const int bx = v % kBX, byz = v / kBX, by = byz % kBY, bz = byz / kBY;
      const int gz = z0 + bz - 1;
      float x0v = 0.0f, x1v = 0.0f, x2v = 0.0f;
      if (gz >= 0 && gz < d.nz) {
        const size_t q = (size_t)wrap(x0 + bx - 1, d.nx) + (size_t)d.nx * (wrap(y0 + by - 1, d.ny) + (size_t)d.ny * gz);
        x0v = in[3 * q];
        x1v = in[3 * q + 1];
        x2v = in[3 * q + 2];
      }
      br[v] = pack4(x0v, x1v, x2v, 0.0f);
    }
  } else {
    const bf16* in = static_cast<const bf16*>(in_);
    constexpr int kChunks = kBrickVox * 4, kPer = (kChunks + 255) / 256;
    uint4 buf[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = threadIdx.x + 256 * u;
      buf[u] = uint4{0u, 0u, 0u, 0u};
      if (e < kChunks) {
        const int v = e >> 2, c = e & 3;
        const int bx = v % kBX, byz = v / kBX, by = byz % kBY, bz = byz / kBY;
        const int gz = z0 + bz - 1;
        if (gz >= 0 && gz < d.nz) {
          const size_t q =
              (size_t)wrap(x0 + bx - 1, d.nx) + (size_t)d.nx * (wrap(y0 + by - 1, d.ny) + (size_t)d.ny * gz);
          buf[u] = *reinterpret_cast<const uint4*>(in + q * kC + 8 * c);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int e = threadIdx.x + 256 * u;
      if (e < kChunks) brick[brick_chunk(e >> 2, e & 3)] = buf[u];
    }
  }
  __syncthreads();

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int wy = 2 * (wv & 1), wz = 2 * (wv >> 1);  // the wavefront's first output row in the block
  f16v acc[2][2];
#pragma unroll
  for (int oy = 0; oy < 2; ++oy)
#pragma unroll
    for (int oz = 0; oz < 2; ++oz) acc[oy][oz] = f16v{};

  if (KIND == KIND_FIRST) {
    // K index k = 3 t + ci; lane (col, half) of k-block kb holds k = 16 kb + 8 half + e
    const uint16_t* br = reinterpret_cast<const uint16_t*>(brick);
    bf8 wa[6];
#pragma unroll
    for (int kb = 0; kb < 6; ++kb) wa[kb] = *reinterpret_cast<const bf8*>(W + (size_t)col * kK1 + 16 * kb + 8 * half);
#pragma unroll
    for (int oy = 0; oy < 2; ++oy)
#pragma unroll
      for (int oz = 0; oz < 2; ++oz) {
        // brick voxel of the output voxel (col, wy + oy, wz + oz) at tap (0, 0, 0)
        const int vc = (col + 1) + kBX * ((wy + oy + 1) + kBY * (wz + oz + 1));
#pragma unroll
        for (int kb = 0; kb < 6; ++kb) {
          bf8 bv;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int k0 = 16 * kb + e, k1 = k0 + 8;  // half 0 / half 1
            const int t0 = k0 / 3, c0 = k0 % 3, t1 = k1 / 3, c1 = k1 % 3;
            const int o0 = (t0 % 3 - 1) + kBX * ((t0 / 3) % 3 - 1) + kBX * kBY * (t0 / 9 - 1);
            const int o1 = (t1 % 3 - 1) + kBX * ((t1 / 3) % 3 - 1) + kBX * kBY * (t1 / 9 - 1);
            const bool z0k = k0 >= 81, z1k = k1 >= 81;
            const int off = half ? 4 * (vc + o1) + c1 : 4 * (vc + o0) + c0;
            const bool zero = half ? z1k : z0k;
            const uint16_t raw = br[zero ? 0 : off];
            bv[e] = zero ? (bf16)0.0f : __builtin_bit_cast(bf16, raw);
          }
          acc[oy][oz] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[kb], bv, acc[oy][oz], 0, 0, 0);
        }
      }
  } else {
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const int c = 2 * kc + half;  // the lane's 8 channels 8c..8c+7
        bf8 wa[3][3];                 // [dy + 1][dz + 1]
#pragma unroll
        for (int ty2 = 0; ty2 < 3; ++ty2)
#pragma unroll
          for (int tz2 = 0; tz2 < 3; ++tz2) {
            const int t = dx + 3 * ty2 + 9 * tz2;
            if (KIND == KIND_LAST) {
              if (col == 0) {
                wa[ty2][tz2] = *reinterpret_cast<const bf8*>(W + (size_t)t * kC + 8 * c);
              } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) wa[ty2][tz2][e] = (bf16)0.0f;
              }
            } else {
              wa[ty2][tz2] = *reinterpret_cast<const bf8*>(W + ((size_t)t * kC + col) * kC + 8 * c);
            }
          }
#pragma unroll
        for (int iy = 0; iy < 4; ++iy)
#pragma unroll
          for (int iz = 0; iz < 4; ++iz) {
            const int v = (col + dx) + kBX * ((wy + iy) + kBY * (wz + iz));
            const bf8 bv = as_bf8(brick[brick_chunk(v, c)]);
#pragma unroll
            for (int oy = 0; oy < 2; ++oy)
#pragma unroll
              for (int oz = 0; oz < 2; ++oz) {
                const int ty2 = iy - oy, tz2 = iz - oz;
                if (ty2 >= 0 && ty2 <= 2 && tz2 >= 0 && tz2 <= 2)
                  acc[oy][oz] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[ty2][tz2], bv, acc[oy][oz], 0, 0, 0);
              }
          }
      }
    }
  }

  // ---- epilogue
#pragma unroll
  for (int oy = 0; oy < 2; ++oy)
#pragma unroll
    for (int oz = 0; oz < 2; ++oz) {
      const int y = y0 + wy + oy, z = z0 + wz + oz;
      if (y >= d.ny || z >= d.nz) continue;
      const size_t p = (size_t)(x0 + col) + (size_t)d.nx * (y + (size_t)d.ny * z);
      if (KIND == KIND_LAST) {
        if (half == 0) zout[p] = acc[oy][oz][0] + bias[0];
        continue;
      }
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int co = 8 * gq + 4 * half;
        float v0 = acc[oy][oz][4 * gq], v1 = acc[oy][oz][4 * gq + 1], v2 = acc[oy][oz][4 * gq + 2],
              v3 = acc[oy][oz][4 * gq + 3];
        if (KIND == KIND_MID && MODE == MID_DATA) {
          *reinterpret_cast<float4*>(gout + p * kC + co) = float4{v0, v1, v2, v3};
          continue;
        }
        v0 += bias[co];
        v1 += bias[co + 1];
        v2 += bias[co + 2];
        v3 += bias[co + 3];
        if (zout) *reinterpret_cast<float4*>(zout + p * kC + co) = float4{v0, v1, v2, v3};
        *reinterpret_cast<uint2*>(aout + p * kC + co) = pack4(gelu(v0), gelu(v1), gelu(v2), gelu(v3));
      }
    }
}

// ---- loss: dout = 2 (out - target) / n; partial sums of (out - target)^2 per block
__global__ void k_loss(Dims d, const float* out, const float* target, float* dout, double* partials) {
  __shared__ double red[4];
  double s = 0.0;
  for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < d.n; p += (size_t)gridDim.x * blockDim.x) {
    const float e = out[p] - target[p];
    dout[p] = 2.0f * e / (float)d.n;
    s += (double)e * e;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ---- layer 6 backward: input gradient g[p][c] = sum_t W[t][c] dout(p - tap_t)
__global__ void k_last_data(Dims d, const float* dout, const float* W, float* g) {
  const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (p >= d.n) return;
  int i, j, k;
  coords(d, p, i, j, k);
  float acc[kC];
#pragma unroll
  for (int c = 0; c < kC; ++c) acc[c] = 0.0f;
  for (int t = 0; t < 27; ++t) {
    const long long q = neighbour(d, i, j, k, 26 - t);  // p - tap_t
    if (q < 0) continue;
    const float dv = dout[q];
    const float* w = W + t * kC;
#pragma unroll
    for (int c = 0; c < kC; ++c) acc[c] += w[c] * dv;
  }
#pragma unroll
  for (int c = 0; c < kC; ++c) g[p * kC + c] = acc[c];
}

// ---- weight gradients, over the bricks of the forward pass.  A workgroup
// takes `per` consecutive bricks of 32 x 4 x 4 voxels, stages each with its
// halo in LDS once for all 27 taps, and keeps its sums in the matrix cores'
// accumulators; its partial sums are added in a fixed order afterwards
// (sum_chunks).  The first and last layers' sums have FP32 factors and run on
// v_mfma_f32_32x32x2_f32 (FP32 products and sums): lane l holds A[l % 32][l / 32]
// and B[l / 32][l % 32], two voxels a step.  Before, these sums walked chunks
// of 4096 voxels one voxel at a time on the vector units, or one tap per
// wavefront: at 128 x 128 x 64 the first, a middle and the last layer took
// 639, 327 and 1598 us, now 102, 83 and 56.
constexpr int kBricksPer = 8;  // most bricks per workgroup

// Brick coordinates and LDS staging shared by the first and last layers:
// NC floats per voxel of the brick with its halo (zero beyond the walls).
template <int NC>
__device__ __forceinline__ void stage_brick(const Dims& d, const float* __restrict__ src, int x0, int y0, int z0,
                                            float* brick) {
  for (int v = threadIdx.x; v < kBrickVox; v += 256) {
    const int bx = v % kBX, byz = v / kBX, by = byz % kBY, bz = byz / kBY;
    const int gz = z0 + bz - 1;
    float x[NC] = {};
    if (gz >= 0 && gz < d.nz) {
      const size_t q = (size_t)wrap(x0 + bx - 1, d.nx) + (size_t)d.nx * (wrap(y0 + by - 1, d.ny) + (size_t)d.ny * gz);
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c] = src[NC * q + c];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) brick[NC * v + c] = x[c];
  }
}
// brick voxel offset of tap t
__device__ __forceinline__ int tap_offset(int t) { return (t % 3 - 1) + kBX * ((t / 3) % 3 - 1) + kBX * kBY * (t / 9 - 1); }

// ---- layer 6: W[t][c] = sum_q in(q)[c] dout(q - tap_t), b = sum dout.  A: the
// 32 channels of two voxels, B: their 27 shifted dout.  Wavefront w takes
// the rows (y, z) = 4 w ... 4 w + 3 of each brick and has its own partial sums.
__global__ void __launch_bounds__(256) k_last_weights(Dims d, BrickGrid bg, int per, const float* __restrict__ dout,
                                                      const bf16* __restrict__ in, float* partials) {
  __shared__ float brick[kBrickVox];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 31, half = lane >> 5;
  const int off = col < 27 ? -tap_offset(col) : 0;
  const int bricks = bg.tiles_x * bg.tiles_y * bg.tiles_z;
  f16v acc = {};
  float bias = 0.0f;
  for (int b = blockIdx.x * per; b < min(bricks, ((int)blockIdx.x + 1) * per); ++b) {
    const int tx = b % bg.tiles_x, tyz = b / bg.tiles_x;
    const int x0 = 32 * tx, y0 = 4 * (tyz % bg.tiles_y), z0 = 4 * (tyz / bg.tiles_y);
    __syncthreads();  // the previous brick's readers
    stage_brick<1>(d, dout, x0, y0, z0, brick);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = y0 + r, z = z0 + wv;
      if (y >= d.ny || z >= d.nz) continue;  // uniform over the wavefront
      const bf16* row = in + ((size_t)x0 + (size_t)d.nx * (y + (size_t)d.ny * z)) * kC + col;
      const int v0 = 1 + kBX * ((r + 1) + kBY * (wv + 1));
      float a[16];
#pragma unroll
      for (int s = 0; s < 16; ++s) a[s] = (float)row[(2 * s + half) * kC];
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const float x = brick[v0 + 2 * s + half + off];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], col < 27 ? x : 0.0f, acc, 0, 0, 0);
      }
      if (half == 0) bias += brick[v0 + col];
    }
  }
  float* out = partials + (size_t)(4 * blockIdx.x + wv) * (27 * kC + 1);
  if (col < 27) {
#pragma unroll
    for (int q = 0; q < 16; ++q) out[col * kC + 8 * (q / 4) + 4 * half + q % 4] = acc[q];
  }
  for (int o = 32; o > 0; o >>= 1) bias += __shfl_down(bias, o, 64);
  if (lane == 0) out[27 * kC] = bias;
}

// ---- GELU backward: dz = g * gelu'(z) (bf16 for the matrix cores), and per
// block of kGeluChunk voxels partial sums of dz per channel (the bias
// gradient, FP32); four channels per thread.  300 -> 66 us at 128 x 128 x 64
// (335 MB), where blocks of 4096 voxels left one workgroup per CU.
constexpr int kGeluChunk = 512;
__global__ void __launch_bounds__(256) k_gelu_back(Dims d, const float* __restrict__ g, const float* __restrict__ z,
                                                   bf16* __restrict__ dz, float* bias_partials) {
  __shared__ float red[32][kC];
  const size_t p0 = (size_t)blockIdx.x * kGeluChunk;
  const int c = 4 * (threadIdx.x & 7), v = threadIdx.x >> 3;  // 32 voxels of 8 quads
  float s[4] = {};
#pragma unroll 4
  for (int u = 0; u < kGeluChunk / 32; ++u) {
    const size_t p = p0 + v + 32 * u;
    if (p < d.n) {
      const float4 gv = *(const float4*)(g + p * kC + c), zv = *(const float4*)(z + p * kC + c);
      const float x[4] = {gv.x * gelu_grad(zv.x), gv.y * gelu_grad(zv.y), gv.z * gelu_grad(zv.z),
                          gv.w * gelu_grad(zv.w)};
      *(uint2*)(dz + p * kC + c) = pack4(x[0], x[1], x[2], x[3]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += x[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[v][c + e] = s[e];
  __syncthreads();
  if (threadIdx.x < kC) {
    float t = 0.0f;
    for (int q = 0; q < 32; ++q) t += red[q][threadIdx.x];
    bias_partials[(size_t)blockIdx.x * kC + threadIdx.x] = t;
  }
}

// ---- 32 -> 32 layers: dW[t] (32 co x 32 ci) = sum_p dz(p)[co] in(p + tap_t)[ci]
// on v_mfma_f32_32x32x16_bf16, K = 16 voxels consecutive in x.  Nine
// wavefronts, one per (dy, dz), each with the accumulators of its three dx.
// The brick is stored channel by channel, so that a lane reads its channel's
// 8 consecutive voxels in one access and the window of 10 serves the three
// dx by shifts; channel strides of 2896 and 1040 bytes put the lanes of an
// access on distinct banks.  The next brick's loads are in flight during the
// current brick's MFMAs.  327 -> 83 us per layer at 128 x 128 x 64.
constexpr int kWThreads = 576;
constexpr int kInRow = 40, kInChan = 36 * kInRow + 8;  // elements per row of 34 voxels, per channel
constexpr int kDzChan = 16 * 32 + 8;
constexpr int kInItems = 36 * 17 * 4, kDzItems = 16 * 16 * 4;  // (row, voxel pair, 8 channels)
constexpr int kInPer = (kInItems + kWThreads - 1) / kWThreads, kDzPer = (kDzItems + kWThreads - 1) / kWThreads;

__global__ void __launch_bounds__(kWThreads) k_mid_weights(Dims d, BrickGrid bg, int per, const bf16* __restrict__ dz,
                                                           const bf16* __restrict__ in, float* partials) {
  extern __shared__ uint4 wlds[];
  uint16_t* li = (uint16_t*)wlds;
  uint16_t* ld = li + kC * kInChan;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 31, half = lane >> 5;
  const int ty = wv % 3, tz = wv / 3;  // dy + 1, dz + 1
  const int bricks = bg.tiles_x * bg.tiles_y * bg.tiles_z;
  const int b0 = (int)blockIdx.x * per, b1 = min(bricks, b0 + per);
  uint4 iv[kInPer][2], dv[kDzPer][2];
  auto load = [&](int b) {
    const int tx = b % bg.tiles_x, tyz = b / bg.tiles_x;
    const int x0 = 32 * tx, y0 = 4 * (tyz % bg.tiles_y), z0 = 4 * (tyz / bg.tiles_y);
#pragma unroll
    for (int u = 0; u < kInPer; ++u) {
      const int e = threadIdx.x + kWThreads * u;
      iv[u][0] = iv[u][1] = uint4{0u, 0u, 0u, 0u};
      const int c = e & 3, pr = (e >> 2) % 17, row = (e >> 2) / 17;
      const int gz = z0 + row / kBY - 1;
      if (e < kInItems && gz >= 0 && gz < d.nz) {
        const size_t r = (size_t)d.nx * (wrap(y0 + row % kBY - 1, d.ny) + (size_t)d.ny * gz);
#pragma unroll
        for (int h = 0; h < 2; ++h)
          iv[u][h] = *(const uint4*)(in + (r + wrap(x0 + 2 * pr + h - 1, d.nx)) * kC + 8 * c);
      }
    }
#pragma unroll
    for (int u = 0; u < kDzPer; ++u) {
      const int e = threadIdx.x + kWThreads * u;
      dv[u][0] = dv[u][1] = uint4{0u, 0u, 0u, 0u};
      const int c = e & 3, pr = (e >> 2) & 15, row = e >> 6;
      const int y = y0 + (row & 3), z = z0 + (row >> 2);
      if (e < kDzItems && y < d.ny && z < d.nz) {
        const size_t p = (size_t)(x0 + 2 * pr) + (size_t)d.nx * (y + (size_t)d.ny * z);
#pragma unroll
        for (int h = 0; h < 2; ++h) dv[u][h] = *(const uint4*)(dz + (p + h) * kC + 8 * c);
      }
    }
  };
  // two voxels' 8 channels -> one 4-byte store per channel
  auto put = [&](uint16_t* base, int stride, const uint4 (&v)[2]) {
    const unsigned a[4] = {v[0].x, v[0].y, v[0].z, v[0].w}, b[4] = {v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      *(unsigned*)(base + (2 * q) * stride) = (a[q] & 0xffffu) | (b[q] << 16);
      *(unsigned*)(base + (2 * q + 1) * stride) = (a[q] >> 16) | (b[q] & 0xffff0000u);
    }
  };
  f16v acc[3] = {};
  if (b0 < b1) load(b0);
  for (int b = b0; b < b1; ++b) {
    __syncthreads();  // the previous brick's readers
#pragma unroll
    for (int u = 0; u < kInPer; ++u) {
      const int e = threadIdx.x + kWThreads * u;
      const int c = e & 3, pr = (e >> 2) % 17, row = (e >> 2) / 17;
      if (e < kInItems) put(li + 8 * c * kInChan + row * kInRow + 2 * pr, kInChan, iv[u]);
    }
#pragma unroll
    for (int u = 0; u < kDzPer; ++u) {
      const int e = threadIdx.x + kWThreads * u;
      const int c = e & 3, pr = (e >> 2) & 15, row = e >> 6;
      if (e < kDzItems) put(ld + 8 * c * kDzChan + row * 32 + 2 * pr, kDzChan, dv[u]);
    }
    __syncthreads();
    if (b + 1 < b1) load(b + 1);
#pragma unroll 4
    for (int row = 0; row < 16; ++row) {
      const uint16_t* ir = li + col * kInChan + ((row & 3) + ty + kBY * ((row >> 2) + tz)) * kInRow;
      const uint16_t* dr = ld + col * kDzChan + row * 32;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint4 A = *(const uint4*)(dr + 16 * s + 8 * half);
        const uint4 w = *(const uint4*)(ir + 16 * s + 8 * half);
        const unsigned w4 = *(const unsigned*)(ir + 16 * s + 8 * half + 8);
        const uint4 w1{__builtin_amdgcn_alignbit(w.y, w.x, 16), __builtin_amdgcn_alignbit(w.z, w.y, 16),
                       __builtin_amdgcn_alignbit(w.w, w.z, 16), __builtin_amdgcn_alignbit(w4, w.w, 16)};
        const uint4 w2{w.y, w.z, w.w, w4};
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(A), as_bf8(w), acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(A), as_bf8(w1), acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(A), as_bf8(w2), acc[2], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) {
    float* out = partials + ((size_t)blockIdx.x * 27 + dx + 3 * ty + 9 * tz) * kC * kC;
#pragma unroll
    for (int q = 0; q < 16; ++q) out[(8 * (q / 4) + 4 * half + q % 4) * kC + col] = acc[dx][q];
  }
}
constexpr unsigned kMidWeightsLds = (unsigned)((kC * kInChan + kC * kDzChan) * sizeof(uint16_t));

// ---- layer 1: W[t][co][ci] = sum_p dz(p)[co] x(p + tap_t)[ci].  A: the 32
// output channels of two voxels, B: three groups of 32 of their 27 x 3 inputs.
__global__ void __launch_bounds__(256) k_first_weights(Dims d, BrickGrid bg, int per, const bf16* __restrict__ dz,
                                                       const float* __restrict__ x, float* partials) {
  __shared__ float brick[3 * kBrickVox];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, col = lane & 31, half = lane >> 5;
  int off[3];  // of column n = 32 m + col: tap n / 3, channel n % 3
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int n = 32 * m + col;
    off[m] = n < 81 ? 3 * tap_offset(n / 3) + n % 3 : 0;
  }
  const int bricks = bg.tiles_x * bg.tiles_y * bg.tiles_z;
  f16v acc[3] = {};
  for (int b = blockIdx.x * per; b < min(bricks, ((int)blockIdx.x + 1) * per); ++b) {
    const int tx = b % bg.tiles_x, tyz = b / bg.tiles_x;
    const int x0 = 32 * tx, y0 = 4 * (tyz % bg.tiles_y), z0 = 4 * (tyz / bg.tiles_y);
    __syncthreads();  // the previous brick's readers
    stage_brick<3>(d, x, x0, y0, z0, brick);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = y0 + r, z = z0 + wv;
      if (y >= d.ny || z >= d.nz) continue;  // uniform over the wavefront
      const bf16* row = dz + ((size_t)x0 + (size_t)d.nx * (y + (size_t)d.ny * z)) * kC + col;
      const int v0 = 1 + kBX * ((r + 1) + kBY * (wv + 1));
      float a[16];
#pragma unroll
      for (int s = 0; s < 16; ++s) a[s] = (float)row[(2 * s + half) * kC];
#pragma unroll
      for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const float v = brick[3 * (v0 + 2 * s + half) + off[m]];
          acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], 32 * m + col < 81 ? v : 0.0f, acc[m], 0, 0, 0);
        }
    }
  }
  float* out = partials + (size_t)(4 * blockIdx.x + wv) * (27 * kC * 3);
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int n = 32 * m + col;
    if (n >= 81) continue;
#pragma unroll
    for (int q = 0; q < 16; ++q) out[((n / 3) * kC + 8 * (q / 4) + 4 * half + q % 4) * 3 + n % 3] = acc[m][q];
  }
}

// sum over chunks in a fixed order, in two levels: groups of kSumGroup
// consecutive chunks (blockIdx.y) into group sums, then the group sums in
// group order (k_sum_groups): out[s] = sum_g sum_{c in g} partials[c][s]
constexpr int kSumGroup = 64;
__global__ void k_sum_chunks(const float* partials, int nchunks, int size, float* groups) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= size) return;
  const int c0 = blockIdx.y * kSumGroup, c1 = c0 + kSumGroup < nchunks ? c0 + kSumGroup : nchunks;
  float acc = 0.0f;
  for (int c = c0; c < c1; ++c) acc += partials[(size_t)c * size + s];
  groups[(size_t)blockIdx.y * size + s] = acc;
}
__global__ void k_sum_groups(const float* groups, int ngroups, int size, float* out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= size) return;
  float acc = 0.0f;
  for (int c = 0; c < ngroups; ++c) acc += groups[(size_t)c * size + s];
  out[s] = acc;
}

// bf16 copies of the 32 -> 32 weights: W16[t][co][ci] and the transposed,
// tap-flipped WT16[t][ci][co] = W[26 - t][co][ci] of the input gradient
__global__ void k_pack(const float* params, bf16* w16, bf16* wt16) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;  // within one layer
  const int l = 1 + blockIdx.y;
  if (s >= 27 * kC * kC) return;
  const float* W = params + layer_offset(l);
  const int t = s / (kC * kC), co = (s / kC) % kC, ci = s % kC;
  const size_t base = (size_t)(l - 1) * 27 * kC * kC;
  w16[base + s] = (bf16)W[s];
  wt16[base + ((size_t)(26 - t) * kC + ci) * kC + co] = (bf16)W[s];
}

// bf16 copies of the first layer's weights as the A operand wants them,
// wf16[co][3 t + ci] padded with zeros to kK1 columns, and of the last
// layer's, wl16[t][ci]
__global__ void k_pack_ends(const float* params, bf16* wf16, bf16* wl16) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < kC * kK1) {
    const int co = s / kK1, k = s % kK1;
    const float* W = params + layer_offset(0);
    wf16[s] = k < 81 ? (bf16)W[((k / 3) * kC + co) * 3 + k % 3] : (bf16)0.0f;
  }
  if (s < 27 * kC) wl16[s] = (bf16)params[layer_offset(5) + s];
}

// input channels of the learned guess: b / |b|, c_prev prev / |b| (prev may
// be null: 0) and jac - 1, channels-last FP32
__global__ void k_guess_input(pcf::Geo g, const double* b, const double* prev, const double* jac, float* in,
                              double inv_bnorm, double prev_scale) {
  const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (p >= g.nv()) return;
  const int i = (int)(p % g.nx), j = (int)((p / g.nx) % g.ny), k = (int)(p / ((size_t)g.nx * g.ny));
  in[3 * p] = (float)(b[p] * inv_bnorm);
  in[3 * p + 1] = prev ? (float)(prev[p] * prev_scale * inv_bnorm) : 0.0f;
  in[3 * p + 2] = (float)(jac[g.h(g.i0 + i, g.j0 + j, g.k0 + k)] - 1.0);
}

// x = c prev + |b| out: the network corrects the rescaled previous solution
// (prev may be null: the first step of a run)
__global__ void k_guess_output(const float* out, double* x, size_t n, double bnorm, const double* prev, double c) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    x[q] = (prev ? c * prev[q] : 0.0) + bnorm * (double)out[q];
}

// ---- the learned preconditioning stage and the residual training
constexpr int kStageGrid = 2048;  // blocks of the sum-of-squares partials

__global__ void k_sumsq(const double* v, size_t n, double* partials) {
  double val[1] = {0.0};
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    val[0] += v[q] * v[q];
  block_partials<1>(val, partials, blockIdx.x);
}

// *out = sqrt(sum of the partials / n), the RMS norm
__global__ void k_rms_final(const double* partials, int nparts, double* out, double n) {
  const double s = finalize_sum(partials, 0, nparts);
  if (threadIdx.x == 0) *out = sqrt(s / n);
}

// the stage's input channels v / |v|, y / |v| and J - 1 with |v| on the device
__global__ void k_stage_input(pcf::Geo g, const double* v, const double* y, const double* jac, float* in,
                              const double* nrm, const SolverScalars* sc) {
  if (sc && sc->done) return;
  const size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (p >= g.nv()) return;
  const int i = (int)(p % g.nx), j = (int)((p / g.nx) % g.ny), k = (int)(p / ((size_t)g.nx * g.ny));
  const double inv = *nrm > 0.0 ? 1.0 / *nrm : 0.0;
  in[3 * p] = (float)(v[p] * inv);
  in[3 * p + 1] = (float)(y[p] * inv);
  in[3 * p + 2] = (float)(jac[g.h(g.i0 + i, g.j0 + j, g.k0 + k)] - 1.0);
}

// y += |v| out
__global__ void k_stage_output(const float* out, double* y, size_t n, const double* nrm, const SolverScalars* sc) {
  if (sc && sc->done) return;
  const double s = *nrm;
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    y[q] += s * (double)out[q];
}

// x = base + c out (base may be null: 0)
__global__ void k_compose(const float* out, const double* base, double* x, size_t n, double c) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    x[q] = (base ? base[q] : 0.0) + c * (double)out[q];
}

// r = a - b
__global__ void k_sub(const double* a, const double* b, double* r, size_t n) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    r[q] = a[q] - b[q];
}

// the output gradient of the residual loss, c A^T r, in FP32
__global__ void k_dout(const double* atr, float* dout, size_t n, double c) {
  for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
    dout[q] = (float)(c * atr[q]);
}

// Adam (Kingma & Ba 2015) on the FP32 parameters
__global__ void k_adam(float* p, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const float gq = g[q];
  const float mq = b1 * m[q] + (1.0f - b1) * gq;
  const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
  m[q] = mq;
  v[q] = vq;
  p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

}  // namespace
}  // namespace pcf

using pcf::bf16;
struct pcf_net;

struct pcf_net {
  pcf::Dims d;
  bool training = false;
  hipStream_t stream = nullptr;
  int device = 0;
  float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
  bf16 *w16 = nullptr, *wt16 = nullptr;
  bf16 *w16_first = nullptr, *w16_last = nullptr;  // the first and last layers' weights in bf16
  float* z[5] = {};        // pre-activations of layers 1..5 (training)
  bf16* a[5] = {};         // activations of layers 1..5 (inference: a[0], a[1] alternate)
  float* out = nullptr;    // network output
  float *dout = nullptr, *g = nullptr;
  bf16* dzb = nullptr;
  float* partials = nullptr;
  float* groups = nullptr;  // group sums of the chunk partials
  double* loss_partials = nullptr;
  double* loss_host = nullptr;
  int step = 0;
  std::vector<void*> allocations;
};

namespace pcf {
namespace {

int net_alloc(pcf_net* net, void** p, size_t bytes) {
  PCF_HIP(hipMalloc(p, bytes));
  net->allocations.push_back(*p);
  return PCF_OK;
}

// blocks of the k_brick launches
BrickGrid brick_grid(const Dims& d) {
  return BrickGrid{d.nx / 32, (d.ny + 3) / 4, (d.nz + 3) / 4};
}
unsigned brick_blocks(const BrickGrid& bg) { return (unsigned)(bg.tiles_x * bg.tiles_y * bg.tiles_z); }
// The weight gradients' bricks per workgroup: enough workgroups for the 256
// CUs, then up to kBricksPer bricks each, which keeps the partial sums (108
// KB per workgroup of a middle layer) small against the activations read.
int weight_per(const BrickGrid& bg) {
  return std::min(kBricksPer, std::max(1, (int)brick_blocks(bg) / 256));
}
int weight_blocks(const BrickGrid& bg) { return ((int)brick_blocks(bg) + weight_per(bg) - 1) / weight_per(bg); }
int gelu_blocks(const Dims& d) { return (int)((d.n + kGeluChunk - 1) / kGeluChunk); }

// out[0..size) = sum over the nc chunk partials (fixed order, two levels)
void sum_chunks(pcf_net* net, int nc, int size, float* out) {
  const unsigned ng = (unsigned)((nc + kSumGroup - 1) / kSumGroup);
  const unsigned blocks = (unsigned)((size + 255) / 256);
  hipLaunchKernelGGL(k_sum_chunks, dim3(blocks, ng), dim3(256), 0, net->stream, net->partials, nc, size, net->groups);
  hipLaunchKernelGGL(k_sum_groups, dim3(blocks), dim3(256), 0, net->stream, net->groups, (int)ng, size, out);
}

// forward pass over the FP32 input (n x 3); output in net->out
int net_forward(pcf_net* net, const float* input, hipStream_t s) {
  const Dims& d = net->d;
  const BrickGrid bg = brick_grid(d);
  const unsigned nb = brick_blocks(bg);
  const float* P = net->params;
  bf16* cur = net->a[0];
  hipLaunchKernelGGL((k_brick<KIND_FIRST, MID_FWD>), dim3(nb), dim3(256), 0, s, d, bg, (const void*)input,
                     net->w16_first, P + layer_offset(0) + 27 * kC * 3, net->training ? net->z[0] : nullptr, cur,
                     nullptr);
  for (int l = 1; l <= 4; ++l) {
    bf16* nxt = net->training ? net->a[l] : net->a[l & 1];
    hipLaunchKernelGGL((k_brick<KIND_MID, MID_FWD>), dim3(nb), dim3(256), 0, s, d, bg, (const void*)cur,
                       net->w16 + (size_t)(l - 1) * 27 * kC * kC, P + layer_offset(l) + 27 * kC * kC,
                       net->training ? net->z[l] : nullptr, nxt, nullptr);
    cur = nxt;
  }
  hipLaunchKernelGGL((k_brick<KIND_LAST, MID_FWD>), dim3(nb), dim3(256), 0, s, d, bg, (const void*)cur,
                     net->w16_last, P + layer_offset(5) + 27 * kC, net->out, nullptr, nullptr);
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

// backward pass from the output gradient in net->dout; gradients in net->grads
int net_backward_dout(pcf_net* net, const float* input) {
  const Dims& d = net->d;
  hipStream_t s = net->stream;
  const unsigned vb = 256, vg = (unsigned)((d.n + vb - 1) / vb);
  const BrickGrid bg = brick_grid(d);
  const int per = weight_per(bg), wb = weight_blocks(bg), gb = gelu_blocks(d);
  const float* P = net->params;
  float* G = net->grads;
  // layer 6
  hipLaunchKernelGGL(k_last_weights, dim3(wb), dim3(256), 0, s, d, bg, per, net->dout, net->a[4], net->partials);
  sum_chunks(net, 4 * wb, 27 * kC + 1, G + layer_offset(5));
  hipLaunchKernelGGL(k_last_data, dim3(vg), dim3(vb), 0, s, d, net->dout, P + layer_offset(5), net->g);
  // layers 5..2
  for (int l = 4; l >= 1; --l) {
    hipLaunchKernelGGL(k_gelu_back, dim3(gb), dim3(256), 0, s, d, net->g, net->z[l], net->dzb, net->partials);
    sum_chunks(net, gb, kC, G + layer_offset(l) + 27 * kC * kC);
    hipLaunchKernelGGL(k_mid_weights, dim3(wb), dim3(kWThreads), kMidWeightsLds, s, d, bg, per, net->dzb, net->a[l - 1],
                       net->partials);
    sum_chunks(net, wb, 27 * kC * kC, G + layer_offset(l));
    hipLaunchKernelGGL((k_brick<KIND_MID, MID_DATA>), dim3(brick_blocks(bg)), dim3(256), 0, s, d, bg,
                       (const void*)net->dzb, net->wt16 + (size_t)(l - 1) * 27 * kC * kC, nullptr, nullptr, nullptr,
                       net->g);
  }
  // layer 1
  hipLaunchKernelGGL(k_gelu_back, dim3(gb), dim3(256), 0, s, d, net->g, net->z[0], net->dzb, net->partials);
  sum_chunks(net, gb, kC, G + layer_offset(0) + 27 * kC * 3);
  hipLaunchKernelGGL(k_first_weights, dim3(wb), dim3(256), 0, s, d, bg, per, net->dzb, input, net->partials);
  sum_chunks(net, 4 * wb, 27 * kC * 3, G + layer_offset(0));
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

// backward pass for the mean squared error against target; loss on the host
int net_backward(pcf_net* net, const float* input, const float* target, double* loss) {
  const Dims& d = net->d;
  hipStream_t s = net->stream;
  const unsigned lg = 1024;
  hipLaunchKernelGGL(k_loss, dim3(lg), dim3(256), 0, s, d, net->out, target, net->dout, net->loss_partials);
  int rc = net_backward_dout(net, input);
  if (rc) return rc;
  std::vector<double> lp(lg);
  PCF_HIP(hipMemcpyAsync(lp.data(), net->loss_partials, lg * sizeof(double), hipMemcpyDeviceToHost, s));
  PCF_HIP(hipStreamSynchronize(s));
  double sum = 0.0;
  for (double v : lp) sum += v;
  if (loss) *loss = sum / (double)d.n;
  return PCF_OK;
}

// input channels for b (and prev scaled by prev_scale) and the RMS norm of b
int guess_input(pcf_state* st, const double* b, const double* prev, double prev_scale, float* input,
                double* bnorm) {
  double bb = 0.0;
  int rc = dot(st, b, b, &bb);
  if (rc) return rc;
  const double nrm = std::sqrt(bb / (double)st->g.nv());
  *bnorm = nrm;
  const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
  hipLaunchKernelGGL(k_guess_input, dim3((unsigned)((st->g.nv() + 255) / 256)), dim3(256), 0, st->stream, st->g, b,
                     prev, st->jac, input, inv, prev_scale);
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

int net_pack(pcf_net* net) {
  hipLaunchKernelGGL(k_pack, dim3((27 * kC * kC + 255) / 256, 4), dim3(256), 0, net->stream, net->params, net->w16,
                     net->wt16);
  hipLaunchKernelGGL(k_pack_ends, dim3((kC * kK1 + 255) / 256), dim3(256), 0, net->stream, net->params,
                     net->w16_first, net->w16_last);
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

}  // namespace

// The learned initial guess of the mixed solve (apply_bicgstab_mixed): x0 in
// st->guess_x, the stage's previous solution rescaled to this dt plus the
// network's correction from the right-hand side, that rescaled solution and
// the Jacobian.
int learned_guess(pcf_state* st, double dt, const double* prev, const double** x0) {
  pcf_net* net = st->guess_net;
  if (!net) {
    set_error("initial_guess = learned needs a network (pcf_set_guess_network)");
    return PCF_E_CONFIG;
  }
  double bnorm = 0.0;
  int rc = guess_input(st, st->rhs, prev, dt, st->guess_in, &bnorm);
  if (rc) return rc;
  ProfScope prof(st, PCF_K_NET);
  if ((rc = net_forward(net, st->guess_in, st->stream))) return rc;
  hipLaunchKernelGGL(k_guess_output, dim3(2048), dim3(256), 0, st->stream, net->out, st->guess_x, st->g.nv(), bnorm,
                     prev, dt);
  PCF_HIP(hipGetLastError());
  *x0 = st->guess_x;
  return PCF_OK;
}

int learned_stage(pcf_state* st, const double* v, double* y, const SolverScalars* sc) {
  pcf_net* net = st->stage_net;
  const Geo& g = st->g;
  const size_t N = g.nv();
  ProfScope prof(st, PCF_K_NET);
  // the fourth dot slot of the partials: the solver's own dot products use
  // slots 0-2 between a kernel that writes them and the one that reads them
  double* part = st->partials + (size_t)3 * kPartialStride;
  hipLaunchKernelGGL(k_sumsq, dim3(kStageGrid), dim3(kReduceBlock), 0, st->stream, v, N, part);
  hipLaunchKernelGGL(k_rms_final, dim3(1), dim3(1024), 0, st->stream, part, kStageGrid, st->stage_norm, (double)N);
  hipLaunchKernelGGL(k_stage_input, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st->stream, g, v, y, st->jac,
                     st->stage_in, st->stage_norm, sc);
  int rc = net_forward(net, st->stage_in, st->stream);
  if (rc) return rc;
  hipLaunchKernelGGL(k_stage_output, dim3(2048), dim3(256), 0, st->stream, net->out, y, N, st->stage_norm, sc);
  PCF_HIP(hipGetLastError());
  return PCF_OK;
}

}  // namespace pcf

extern "C" {

int pcf_guess_input(pcf_state* st, const double* d_b, const double* d_prev, float* d_input, double* b_norm) {
  if (!st || !d_b || !d_input) return PCF_E_ARG;
  double nrm = 0.0;
  int rc = pcf::guess_input(st, d_b, d_prev, 1.0, d_input, &nrm);
  if (rc) return rc;
  PCF_HIP(hipStreamSynchronize(st->stream));
  if (b_norm) *b_norm = nrm;
  return PCF_OK;
}

int pcf_guess_fallbacks(const pcf_state* st, int32_t* count) {
  if (!st || !count) return PCF_E_ARG;
  *count = st->guess_fallbacks;
  return PCF_OK;
}

int pcf_set_guess_network(pcf_state* st, pcf_net* net) {
  using namespace pcf;
  if (!st) return PCF_E_ARG;
  if (net && ((size_t)net->d.nx != (size_t)st->g.nx || net->d.ny != st->g.ny || net->d.nz != st->g.nz)) {
    set_error("pcf_set_guess_network: the network's grid differs from the state's");
    return PCF_E_ARG;
  }
  if (net && !st->guess_in) {
    const size_t N = st->g.nv();
    int rc = device_alloc(st, &st->guess_in, 3 * N);
    if (rc == PCF_OK) rc = device_alloc(st, &st->guess_x, N);
    if (rc) return rc;
  }
  st->guess_net = net;
  return PCF_OK;
}


int pcf_set_stage_network(pcf_state* st, pcf_net* net, int32_t iterations) {
  using namespace pcf;
  if (!st || iterations < 0) return PCF_E_ARG;
  if (net && ((size_t)net->d.nx != (size_t)st->g.nx || net->d.ny != st->g.ny || net->d.nz != st->g.nz)) {
    set_error("pcf_set_stage_network: the network's grid differs from the state's");
    return PCF_E_ARG;
  }
  if (net && (st->cfg.precision != PCF_PRECISION_MIXED || !st->cfg.preconditioner)) {
    set_error("pcf_set_stage_network: the learned stage needs precision = mixed and a preconditioner "
              "(a nonlinear stage needs the flexible form of the solution update)");
    return PCF_E_CONFIG;
  }
  if (net && !st->stage_in) {
    int rc = device_alloc(st, &st->stage_in, 3 * st->g.nv());
    if (rc == PCF_OK) rc = device_alloc(st, &st->stage_norm, 1);
    if (rc) return rc;
  }
  st->stage_net = net;
  st->stage_iterations = net ? iterations : 0;
  return PCF_OK;
}

int pcf_stage_fallbacks(const pcf_state* st, int32_t* count) {
  if (!st || !count) return PCF_E_ARG;
  *count = st->stage_fallbacks;
  return PCF_OK;
}

int pcf_net_param_count(void) { return pcf::kParams; }

int pcf_net_create(int32_t nx, int32_t ny, int32_t nz, int32_t training, pcf_net** out) {
  using namespace pcf;
  if (!out || nx < 32 || nx % 32 != 0 || ny < 1 || nz < 1) {
    set_error("pcf_net_create: nx must be a positive multiple of 32");
    return PCF_E_ARG;
  }
  if ((long long)nx * ny * nz > 0x7fffffffLL) {
    set_error("pcf_net_create: at most 2^31 - 1 voxels");
    return PCF_E_ARG;
  }
  pcf_net* net = new pcf_net();
  net->d = Dims{nx, ny, nz, (size_t)nx * ny * nz};
  net->training = training != 0;
  auto fail = [&](int rc) {
    for (void* p : net->allocations) (void)hipFree(p);
    if (net->stream) (void)hipStreamDestroy(net->stream);
    delete net;
    return rc;
  };
  if (hipGetDevice(&net->device) != hipSuccess) return fail(PCF_E_HIP);
  if (hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking) != hipSuccess) return fail(PCF_E_HIP);
  const size_t N = net->d.n;
  int rc;
  if ((rc = net_alloc(net, (void**)&net->params, kParams * sizeof(float)))) return fail(rc);
  if ((rc = net_alloc(net, (void**)&net->w16, 4 * 27 * kC * kC * sizeof(bf16)))) return fail(rc);
  if ((rc = net_alloc(net, (void**)&net->wt16, 4 * 27 * kC * kC * sizeof(bf16)))) return fail(rc);
  if ((rc = net_alloc(net, (void**)&net->w16_first, kC * kK1 * sizeof(bf16)))) return fail(rc);
  if ((rc = net_alloc(net, (void**)&net->w16_last, 27 * kC * sizeof(bf16)))) return fail(rc);
  if ((rc = net_alloc(net, (void**)&net->out, N * sizeof(float)))) return fail(rc);
  const int na = net->training ? 5 : 2;
  for (int l = 0; l < na; ++l)
    if ((rc = net_alloc(net, (void**)&net->a[l], N * kC * sizeof(bf16)))) return fail(rc);
  if (net->training) {
    for (int l = 0; l < 5; ++l)
      if ((rc = net_alloc(net, (void**)&net->z[l], N * kC * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->grads, kParams * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->adam_m, kParams * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->adam_v, kParams * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->dout, N * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->g, N * kC * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->dzb, N * kC * sizeof(bf16)))) return fail(rc);
    // the partial sums of each use (sum_chunks: chunks, values per chunk)
    const size_t wb = (size_t)weight_blocks(brick_grid(net->d)), gb = (size_t)gelu_blocks(net->d);
    const size_t uses[4][2] = {{wb, 27 * kC * kC}, {4 * wb, 27 * kC * 3}, {4 * wb, 27 * kC + 1}, {gb, kC}};
    size_t part = 0, groups = 0;
    for (const auto& u : uses) {
      part = std::max(part, u[0] * u[1]);
      groups = std::max(groups, (u[0] + kSumGroup - 1) / kSumGroup * u[1]);
    }
    if ((rc = net_alloc(net, (void**)&net->partials, part * sizeof(float)))) return fail(rc);
    if ((rc = net_alloc(net, (void**)&net->groups, groups * sizeof(float)))) return fail(rc);
    if (hipFuncSetAttribute((const void*)k_mid_weights, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)kMidWeightsLds) != hipSuccess)
      return fail(PCF_E_HIP);
    if ((rc = net_alloc(net, (void**)&net->loss_partials, 1024 * sizeof(double)))) return fail(rc);
    if (hipMemsetAsync(net->adam_m, 0, kParams * sizeof(float), net->stream) != hipSuccess) return fail(PCF_E_HIP);
    if (hipMemsetAsync(net->adam_v, 0, kParams * sizeof(float), net->stream) != hipSuccess) return fail(PCF_E_HIP);
  }
  if (hipMemsetAsync(net->params, 0, kParams * sizeof(float), net->stream) != hipSuccess) return fail(PCF_E_HIP);
  if (hipStreamSynchronize(net->stream) != hipSuccess) return fail(PCF_E_HIP);
  *out = net;
  return PCF_OK;
}

int pcf_net_destroy(pcf_net* net) {
  if (!net) return PCF_E_ARG;
  (void)hipStreamSynchronize(net->stream);
  for (void* p : net->allocations) (void)hipFree(p);
  (void)hipStreamDestroy(net->stream);
  delete net;
  return PCF_OK;
}

int pcf_net_set_params(pcf_net* net, const float* host) {
  using namespace pcf;
  if (!net || !host) return PCF_E_ARG;
  PCF_HIP(hipMemcpyAsync(net->params, host, kParams * sizeof(float), hipMemcpyHostToDevice, net->stream));
  int rc = net_pack(net);
  if (rc) return rc;
  PCF_HIP(hipStreamSynchronize(net->stream));
  return PCF_OK;
}

int pcf_net_get_params(pcf_net* net, float* host) {
  using namespace pcf;
  if (!net || !host) return PCF_E_ARG;
  PCF_HIP(hipMemcpyAsync(host, net->params, kParams * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  PCF_HIP(hipStreamSynchronize(net->stream));
  return PCF_OK;
}

int pcf_net_forward(pcf_net* net, const float* d_input, float* d_output) {
  using namespace pcf;
  if (!net || !d_input || !d_output) return PCF_E_ARG;
  int rc = net_forward(net, d_input, net->stream);
  if (rc) return rc;
  PCF_HIP(hipMemcpyAsync(d_output, net->out, net->d.n * sizeof(float), hipMemcpyDeviceToDevice, net->stream));
  PCF_HIP(hipStreamSynchronize(net->stream));
  return PCF_OK;
}

int pcf_net_gradients(pcf_net* net, const float* d_input, const float* d_target, float* host_grads, double* loss) {
  using namespace pcf;
  if (!net || !d_input || !d_target || !net->training) return PCF_E_ARG;
  int rc = net_forward(net, d_input, net->stream);
  if (rc) return rc;
  if ((rc = net_backward(net, d_input, d_target, loss))) return rc;
  if (host_grads) {
    PCF_HIP(hipMemcpyAsync(host_grads, net->grads, kParams * sizeof(float), hipMemcpyDeviceToHost, net->stream));
    PCF_HIP(hipStreamSynchronize(net->stream));
  }
  return PCF_OK;
}

// one Adam step on the gradients in net->grads
static int adam_step(pcf_net* net, float lr) {
  using namespace pcf;
  net->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - std::pow(b1, (float)net->step), c2 = 1.0f - std::pow(b2, (float)net->step);
  hipLaunchKernelGGL(k_adam, dim3((kParams + 255) / 256), dim3(256), 0, net->stream, net->params, net->grads,
                     net->adam_m, net->adam_v, kParams, lr, b1, b2, 1e-8f, c1, c2);
  int rc = net_pack(net);
  if (rc) return rc;
  PCF_HIP(hipStreamSynchronize(net->stream));
  return PCF_OK;
}

int pcf_net_train_step(pcf_net* net, const float* d_input, const float* d_target, float lr, double* loss) {
  using namespace pcf;
  int rc = pcf_net_gradients(net, d_input, d_target, nullptr, loss);
  if (rc) return rc;
  return adam_step(net, lr);
}

// L = |A x - v|^2 / |v|^2 for x = base + |v| out, out the network's output
// (x in st->train_buf[0]); the residual stays in train_buf[1]
static int residual_loss(pcf_state* st, pcf_net* net, const double* v, const double* base, double vnorm, double vv,
                         double* loss) {
  using namespace pcf;
  const size_t N = st->g.nv();
  double *x = st->train_buf[0], *r = st->train_buf[1];
  int rc = net_forward(net, st->guess_in, st->stream);
  if (rc) return rc;
  hipLaunchKernelGGL(k_compose, dim3(2048), dim3(256), 0, st->stream, net->out, base, x, N, vnorm);
  PCF_HIP(hipGetLastError());
  if ((rc = apply_operator(st, x, r, true))) return rc;
  hipLaunchKernelGGL(k_sub, dim3(2048), dim3(256), 0, st->stream, r, v, r, N);
  PCF_HIP(hipGetLastError());
  double rr = 0.0;
  if ((rc = dot(st, r, r, &rr))) return rc;
  *loss = rr / vv;
  return PCF_OK;
}

int pcf_net_train_residual(pcf_state* st, pcf_net* net, const double* d_v, const double* d_base, int32_t objective,
                           int32_t inner, float lr, double* loss_base, double* loss_net) {
  using namespace pcf;
  if (!st || !net || !d_v || inner < 0 || (inner > 0 && !net->training)) return PCF_E_ARG;
  if (objective != PCF_OBJECTIVE_RESIDUAL && objective != PCF_OBJECTIVE_ENERGY) {
    set_error("pcf_net_train_residual: unknown objective");
    return PCF_E_OPTION;
  }
  if ((size_t)net->d.nx != (size_t)st->g.nx || net->d.ny != st->g.ny || net->d.nz != st->g.nz) {
    set_error("pcf_net_train_residual: the network's grid differs from the state's");
    return PCF_E_ARG;
  }
  const size_t N = st->g.nv();
  int rc;
  if (!st->guess_in && (rc = device_alloc(st, &st->guess_in, 3 * N))) return rc;
  for (double*& b : st->train_buf)
    if (!b && (rc = device_alloc(st, &b, N))) return rc;
  double vnorm = 0.0;
  if ((rc = guess_input(st, d_v, d_base, 1.0, st->guess_in, &vnorm))) return rc;
  const double vv = vnorm * vnorm * (double)N;
  if (!(vv > 0.0)) {
    set_error("pcf_net_train_residual: v is zero");
    return PCF_E_ARG;
  }
  double* r = st->train_buf[1];
  double* atr = st->train_buf[2];
  if (loss_base) {  // the residual of base alone
    double rr = vv;
    if (d_base) {
      if ((rc = apply_operator(st, d_base, r, true))) return rc;
      hipLaunchKernelGGL(k_sub, dim3(2048), dim3(256), 0, st->stream, r, d_v, r, N);
      PCF_HIP(hipGetLastError());
      if ((rc = dot(st, r, r, &rr))) return rc;
    }
    *loss_base = rr / vv;
  }
  double loss = 0.0;
  for (int it = 0; it < inner; ++it) {
    if ((rc = residual_loss(st, net, d_v, d_base, vnorm, vv, &loss))) return rc;
    if (objective == PCF_OBJECTIVE_RESIDUAL) {
      if ((rc = apply_operator_transpose(st, r, atr))) return rc;
      hipLaunchKernelGGL(k_dout, dim3(2048), dim3(256), 0, st->stream, atr, net->dout, N, 2.0 * vnorm / vv);
    } else {  // the energy norm of the error under -A: its gradient in x is -(A x - v)
      hipLaunchKernelGGL(k_dout, dim3(2048), dim3(256), 0, st->stream, r, net->dout, N, -2.0 * vnorm / vv);
    }
    PCF_HIP(hipGetLastError());
    PCF_HIP(hipStreamSynchronize(st->stream));  // the backward pass runs on the network's stream
    if ((rc = net_backward_dout(net, st->guess_in))) return rc;
    if ((rc = adam_step(net, lr))) return rc;
  }
  if (loss_net) {
    if ((rc = residual_loss(st, net, d_v, d_base, vnorm, vv, &loss))) return rc;
    *loss_net = loss;
  }
  PCF_HIP(hipStreamSynchronize(st->stream));
  return PCF_OK;
}

int pcf_net_train_step_dout(pcf_net* net, const float* d_input, const float* d_dout, float lr) {
  using namespace pcf;
  if (!net || !d_input || !d_dout || !net->training) return PCF_E_ARG;
  int rc = net_forward(net, d_input, net->stream);
  if (rc) return rc;
  PCF_HIP(hipMemcpyAsync(net->dout, d_dout, net->d.n * sizeof(float), hipMemcpyDeviceToDevice, net->stream));
  if ((rc = net_backward_dout(net, d_input))) return rc;
  return adam_step(net, lr);
}

}  // extern "C"
