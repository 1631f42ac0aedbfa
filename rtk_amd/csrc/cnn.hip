// 3D residual CNN for learned CG warm starts (no counterpart in the reference).
//
// Network (fixed): six 3x3x3 convolutions, 32 channels, ReLU after the first five,
// residual output:  y = x + conv6(relu(conv5(...relu(conv1(s x))...))) / s
// where s is a fixed input scale.  Convolutions are cross-correlations with zero
// padding ("same" size): out[v][co] = b[co] + sum_t sum_ci W[t][co][ci] in[v + d(t)][ci],
// tap t = (dz*3 + dy)*3 + dx, d(t) = (dx-1, dy-1, dz-1).
//
// Storage: activations BF16 channels-last [b][z][y][x][32]; master parameters FP32,
// packed: W1[27][32], b1[32], then for layers 2..5 W[27][32 co][32 ci], b[32], then
// W6[27][32 ci], b6[1].
//
// Kernels (gfx950):
//  * 32->32 layers (forward and data gradient) are implicit GEMMs on
//    v_mfma_f32_16x16x32_bf16: M = 16 output channels, N = 16 voxels along x,
//    K = 32 input channels per tap, 27 taps accumulated in FP32, from an LDS block of the
//    input with its halo.  Bias, ReLU and the ReLU-derivative mask of the data gradient
//    are fused into the epilogue.
//  * The 32->32 weight gradients are GEMMs over the voxels on the same instruction,
//    their operands transposed by the LDS reads.
//  * The 32->1 layer is a GEMM with its FP32 weights as three BF16 terms; the 1->32 layer
//    and the weight gradients of both run on the VALU in FP32.
#include "common.h"

#include <cfloat>
#include <cmath>
#include <vector>

typedef __bf16 bf16_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

namespace rtkhip
{
namespace cnn
{

constexpr int C = 32;
constexpr int T = 27;
constexpr int kL1W = 0, kL1B = kL1W + T * C;
constexpr int kMidBase = kL1B + C;
constexpr int kMidSize = T * C * C + C;
constexpr int kL6W = kMidBase + 4 * kMidSize, kL6B = kL6W + T * C;
constexpr int kNumParams = kL6B + 1;

__device__ __forceinline__ int
TapOffset(int t, int X, int Y, int & dx, int & dy, int & dz)
{
  dx = t % 3 - 1;
  dy = (t / 3) % 3 - 1;
  dz = t / 9 - 1;
  return (dz * Y + dy) * X + dx;
}

// A lane's voxel in the kernels of a thread per voxel: a workgroup is 256 voxels of one (x, y)
// plane (planes of all volumes in a row, `chunks` workgroups each), so that the only division
// by lane is one of 32 bits.  Layer 1 at 256^3: 0.76 ms with the voxel's index in the batch
// divided in 64 bits -> 0.68 (its 864 FMAs a voxel alone 0.38).
struct PlaneVoxel
{
  long v;       // index in the batch
  int  i, j, k; // position in the volume
  bool in;
};
__device__ __forceinline__ PlaneVoxel
VoxelOf(unsigned chunks, int X, int Y, int Z)
{
  const unsigned plane = blockIdx.x / chunks, r = blockIdx.x % chunks * 256u + threadIdx.x;
  const unsigned j = r / unsigned(X), size = unsigned(X) * unsigned(Y);
  return PlaneVoxel{ long(plane) * size + r, int(r - j * unsigned(X)), int(j), int(plane % unsigned(Z)), r < size };
}

// ------------------------------------------------------------------ layer 1
// A1[v][co] = relu(b1[co] + sum_t W1[t][co] * s * x[v + d(t)])
__global__ __launch_bounds__(256) void conv_in_kernel(const float * __restrict__ x, const float * __restrict__ p,
                                                       bf16_t * __restrict__ a1, unsigned chunks, int X, int Y, int Z,
                                                       float scale)
{
  const auto [v, i, j, k, inside] = VoxelOf(chunks, X, Y, Z);
  if (!inside)
    return;
  float xin[T];
#pragma unroll
  for (int t = 0; t < T; t++)
  {
    int       dx, dy, dz;
    const int off = TapOffset(t, X, Y, dx, dy, dz);
    const bool in = i + dx >= 0 && i + dx < X && j + dy >= 0 && j + dy < Y && k + dz >= 0 && k + dz < Z;
    xin[t] = in ? scale * x[v + off] : 0.f;
  }
  bf16x8 out[4];
#pragma unroll
  for (int co = 0; co < C; co++)
  {
    float acc = p[kL1B + co];
#pragma unroll
    for (int t = 0; t < T; t++)
      acc += p[kL1W + t * C + co] * xin[t];
    out[co / 8][co % 8] = bf16_t(fmaxf(acc, 0.f));
  }
  bf16x8 * dst = reinterpret_cast<bf16x8 *>(a1 + v * C);
#pragma unroll
  for (int q = 0; q < 4; q++)
    dst[q] = out[q];
}

// --------------------------------------------------------- 32->32 on MFMA
// out[v][co] = epilogue(b[co] + sum_t sum_ci W[t][co][ci] in[v + d(t)][ci])
// epilogue: optional ReLU; optional mask (out *= mask[v][co] > 0).
// w layout [27][32 co][32 ci] BF16.
//
// A workgroup is 16 (x) x kRowsY (y) x 4 (z) voxels, a wavefront one z plane.  The block's
// input with a one-voxel halo is staged in LDS once (zero outside the volume).  A wavefront
// reads each input row of its three planes once, as three fragments (dx = -1, 0, 1), and
// multiplies it for the up to three output rows it feeds (dy), against the nine taps of the
// plane held in registers: 90 LDS fragments for 432 matrix instructions instead of one for
// every two.  Per output the taps still come in the order (dz, dy, dx), so sums are the same
// as tap by tap.  Products are W (co) x voxels, so a lane ends with four channels of a voxel
// and stores 8 bytes.  256^3 layer: 1.87 ms (497 TFLOP/s; a fragment per tap and output row,
// LDS-bound) -> 1.08 ms (860 TFLOP/s; the matrix units alone need 0.37, the rest is staging,
// which one other workgroup per CU overlaps).
// Rows 8 / 4, a whole inference: 256^3 4.8 ms / 5.6 (where blocks fill the chip; by 128^3 .63 /
// .71 and 64^3 .112 / .137), 48^3 .081 / .080, 32^3 (64 workgroups of 8) .070 / .057.
constexpr int kRowsY = 8;

template <bool RELU, bool MASK>
__global__ __launch_bounds__(256, 2) void conv32_mfma_kernel(const bf16_t * __restrict__ in,
                                                           const bf16_t * __restrict__ w,
                                                           const float * __restrict__ bias,
                                                           const bf16_t * __restrict__ mask, bf16_t * __restrict__ out,
                                                           int X, int Y, int Z, int tilesX, int tilesY, int tilesZ)
{
  constexpr int HX = 18, HY = kRowsY + 2, HZ = 6, NCHUNK = HX * HY * HZ * 4;
  __shared__ bf16x8 halo[NCHUNK];
  const int  lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned   blk = blockIdx.x;
  const int  tx = int(blk % unsigned(tilesX));
  blk /= unsigned(tilesX);
  const int  ty = int(blk % unsigned(tilesY));
  blk /= unsigned(tilesY);
  const int  tz = int(blk % unsigned(tilesZ));
  const int  b = int(blk / unsigned(tilesZ));
  const int  z = tz * 4 + wave;
  const int  y0 = ty * kRowsY;
  const int  xl = lane & 15;  // voxel of this lane's column (x offset in the block)
  const int  kg = lane >> 4;  // channel group: ci = 8 kg .. 8 kg + 7
  const long volBase = long(b) * Z * Y * X;

  const bf16x8 zero8 = bf16x8{ bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f),
                               bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f) };
  // every load of the block is in flight before the first is stored
  constexpr int PER = (NCHUNK + 255) / 256;
  bf16x8        reg[PER];
#pragma unroll
  for (int q = 0; q < PER; q++)
  {
    const int c = int(threadIdx.x) + 256 * q, vi = c >> 2;
    const int xs = tx * 16 - 1 + vi % HX, ys = y0 - 1 + (vi / HX) % HY, zs = tz * 4 - 1 + vi / (HX * HY);
    reg[q] = zero8;
    if (c < NCHUNK && unsigned(xs) < unsigned(X) && unsigned(ys) < unsigned(Y) && unsigned(zs) < unsigned(Z))
      reg[q] = *reinterpret_cast<const bf16x8 *>(in + ((volBase + (long(zs) * Y + ys) * X + xs) * C + 8 * (c & 3)));
  }
#pragma unroll
  for (int q = 0; q < PER; q++)
    if (int(threadIdx.x) + 256 * q < NCHUNK)
      halo[threadIdx.x + 256 * q] = reg[q];

  floatx4 acc[kRowsY][2];
#pragma unroll
  for (int r = 0; r < kRowsY; r++)
    for (int nn = 0; nn < 2; nn++)
      acc[r][nn] = floatx4{ 0.f, 0.f, 0.f, 0.f };
  // the plane's nine taps, both halves of the output channels
  bf16x8 wt[9][2];
  auto   taps = [&](int dz) {
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int nn = 0; nn < 2; nn++)
        wt[t][nn] = *reinterpret_cast<const bf16x8 *>(w + (long(9 * dz + t) * C + 16 * nn + xl) * C + 8 * kg);
  };
  taps(0);
  __syncthreads();
#pragma unroll 1
  for (int dz = 0; dz < 3; dz++)
  {
    const bf16x8 * plane = halo + ((wave + dz) * HY * HX + xl) * 4 + kg;
#pragma unroll
    for (int i = 0; i < HY; i++)
    {
      bf16x8 a[3];
#pragma unroll
      for (int dx = 0; dx < 3; dx++)
        a[dx] = plane[(i * HX + dx) * 4];
#pragma unroll
      for (int dy = 0; dy < 3; dy++)
      {
        const int r = i - dy;
        if (r < 0 || r >= kRowsY)
          continue;
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int nn = 0; nn < 2; nn++)
            acc[r][nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[3 * dy + dx][nn], a[dx], acc[r][nn], 0, 0, 0);
      }
    }
    if (dz < 2)
      taps(dz + 1);
  }
  const int x = tx * 16 + xl;
  if (z >= Z || x >= X)
    return;
  // D layout: lane holds rows (channels) 4 * (lane / 16) + q of column (voxel) lane % 16
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int nn = 0; nn < 2; nn++)
  {
    const int co = 16 * nn + 4 * kg;
    float     bb[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
      bb[q] = bias ? bias[co + q] : 0.f;
#pragma unroll
    for (int r = 0; r < kRowsY; r++)
    {
      const int y = y0 + r;
      if (y >= Y)
        continue;
      const long o = (volBase + (long(z) * Y + y) * X + x) * C + co;
      bf16x4     m, res;
      if (MASK)
        m = *reinterpret_cast<const bf16x4 *>(mask + o);
#pragma unroll
      for (int q = 0; q < 4; q++)
      {
        float v = acc[r][nn][q] + bb[q];
        if (RELU)
          v = fmaxf(v, 0.f);
        if (MASK)
          v = (float(m[q]) > 0.f) ? v : 0.f;
        res[q] = bf16_t(v);
      }
      *reinterpret_cast<bf16x4 *>(out + o) = res;
    }
  }
}

// ------------------------------------------------------------------ layer 6

// Whether one of eight activations (ReLU outputs: the order of the values is that of their
// bits) is infinite; a negative zero counts as one.
__device__ __forceinline__ bool
HasInf(const bf16x8 & v)
{
  typedef unsigned short ushort8v __attribute__((ext_vector_type(8)));
  typedef unsigned short ushort2v __attribute__((ext_vector_type(2)));
  const ushort8v  b = __builtin_bit_cast(ushort8v, v);
  const ushort2v  m = __builtin_elementwise_max(__builtin_elementwise_max(b.lo.lo, b.lo.hi),
                                               __builtin_elementwise_max(b.hi.lo, b.hi.hi));
  return max(m.x, m.y) >= 0x7f80;
}

// y[v] = x[v] + (b6 + sum_t sum_ci W6[t][ci] a5[v + d(t)][ci]) / s
// As a GEMM per voxel u of the input, P[t][u] = sum_ci W6[t][ci] a5[u][ci] (M = 27 taps in two
// halves of 16, N = 16 voxels, K = 32 channels), and the sum y[v] += P[t][v + d(t)].  The FP32
// weights enter as three BF16 terms whose sum is the weight exactly (24 bits in three times
// 8), so every product is exact and the sums are FP32; with fewer sequential additions y's
// error against 64 bits is a quarter of the tap-by-tap loop's (1.2e-7 of the range, 4.8e-7
// before).  Infinite activations meet the weights' first terms alone: a lower term may be 0 or
// of the other sign.  A workgroup is a 16 x 16 (x, y) column marching along z: per plane its
// wavefronts write P of the 18 x 18 halo to LDS, then each thread adds 9 values to each of the
// three outputs the plane feeds, which it keeps in registers; the next plane's activations are
// loaded meanwhile.  Every activation is read 1.3 times instead of 27.
// 256^3: 1.65 ms (864 VALU FMAs and 108 cached 16-byte loads a voxel) -> 0.28 ms.
constexpr int kOutX = 16, kOutHX = kOutX + 2, kOutVox = kOutHX * kOutHX; // halo plane
constexpr int kOutGroups = (kOutVox + 15) / 16;
constexpr int kOutStride = 340; // floats of a tap's plane: 4 taps further is 16 LDS banks on

__global__ __launch_bounds__(256) void conv_out_kernel(const bf16_t * __restrict__ a5, const float * __restrict__ x,
                                                        const float * __restrict__ p, float * __restrict__ y, int X,
                                                        int Y, int Z, int tilesX, int tilesY, int zrun, int runs,
                                                        float inv_scale)
{
  __shared__ float P[T * kOutStride];
  constexpr int PER = (kOutGroups + 3) / 4;
  const int     lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned      blk = blockIdx.x;
  const int     x0 = int(blk % unsigned(tilesX)) * kOutX;
  blk /= unsigned(tilesX);
  const int     y0 = int(blk % unsigned(tilesY)) * kOutX;
  blk /= unsigned(tilesY);
  const int     z0 = int(blk % unsigned(runs)) * zrun, z1 = min(z0 + zrun, Z);
  const long    vol = long(blk / unsigned(runs)) * X * Y * Z;
  const int     col = lane & 15, kg = lane >> 4;
  const bf16x8  zero8 = bf16x8{ bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f),
                               bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f) };
  // weights of tap 16 h + col, channels 8 kg .. + 7, as hi + mid + lo
  bf16x8 wt[2][3];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int e = 0; e < 8; e++)
    {
      const int    t = 16 * h + col;
      const float  w = t < T ? p[kL6W + t * C + 8 * kg + e] : 0.f;
      const bf16_t hi = bf16_t(w), mid = bf16_t(w - float(hi));
      const bool   fin = fabsf(float(hi)) < INFINITY; // an infinite or NaN weight stays one term
      wt[h][0][e] = hi;
      wt[h][1][e] = fin ? mid : bf16_t(0.f);
      wt[h][2][e] = fin ? bf16_t(w - float(hi) - float(mid)) : bf16_t(0.f);
    }
  // this wavefront's groups of 16 halo voxels: group wave + 4 g, voxel 16 group + col
  bf16x8 act[PER];
  auto   load = [&](int z) {
#pragma unroll
    for (int g = 0; g < PER; g++)
    {
      const int v = 16 * (wave + 4 * g) + col, xs = x0 - 1 + v % kOutHX, ys = y0 - 1 + v / kOutHX;
      act[g] = zero8;
      if (v < kOutVox && unsigned(xs) < unsigned(X) && unsigned(ys) < unsigned(Y) && unsigned(z) < unsigned(Z))
        act[g] = *reinterpret_cast<const bf16x8 *>(a5 + ((vol + (long(z) * Y + ys) * X + xs) * C + 8 * kg));
    }
  };
  const int   xo = threadIdx.x & 15, yo = threadIdx.x >> 4;
  const bool  live = x0 + xo < X && y0 + yo < Y;
  const float bias = p[kL6B];
  float       prev = 0.f, cur = 0.f; // sums of outputs z - 1 and z before plane z
  load(z0 - 1);
  for (int z = z0 - 1; z <= z1; z++)
  {
#pragma unroll
    for (int g = 0; g < PER; g++)
    {
      const int v = 16 * (wave + 4 * g) + col;
      if (16 * (wave + 4 * g) >= kOutVox)
        continue; // uniform
      bf16x8 low = act[g]; // for the weights' lower terms
      if (__any(HasInf(low)))
#pragma unroll
        for (int e = 0; e < 8; e++)
          low[e] = fabsf(float(low[e])) < INFINITY ? low[e] : bf16_t(0.f);
#pragma unroll
      for (int h = 0; h < 2; h++)
      {
        floatx4 acc = floatx4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int k = 2; k >= 0; k--)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[h][k], k ? low : act[g], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (16 * h + 4 * kg + q < T)
            P[(16 * h + 4 * kg + q) * kOutStride + v] = acc[q];
      }
    }
    if (z < z1)
      load(z + 1);
    __syncthreads();
    auto plane = [&](int dz) {
      float s = 0.f;
#pragma unroll
      for (int t = 0; t < 9; t++)
        s += P[(9 * dz + t) * kOutStride + (yo + t / 3) * kOutHX + xo + t % 3];
      return s;
    };
    // plane z is at d(t) = -1, 0, 1 of the outputs z + 1, z, z - 1
    const float sum = prev + plane(2);
    if (live && z - 1 >= z0)
    {
      const long o = vol + (long(z - 1) * Y + y0 + yo) * X + x0 + xo;
      y[o] = x[o] + (bias + sum) * inv_scale;
    }
    prev = cur + plane(1);
    cur = plane(0);
    __syncthreads();
  }
}

// dZ5[u][ci] = (sum_t W6[t][ci] g[u - d(t)]) * (a5[u][ci] > 0), g = dy * (1/s)
__global__ __launch_bounds__(256) void conv_out_bwd_data_kernel(const float * __restrict__ dy,
                                                                 const float * __restrict__ p,
                                                                 const bf16_t * __restrict__ a5,
                                                                 bf16_t * __restrict__ dz5, unsigned chunks, int X,
                                                                 int Y, int Z, float inv_scale)
{
  const auto [u, i, j, k, inside] = VoxelOf(chunks, X, Y, Z);
  if (!inside)
    return;
  float g[T];
#pragma unroll
  for (int t = 0; t < T; t++)
  {
    int       dx, dy_, dz;
    const int off = TapOffset(t, X, Y, dx, dy_, dz);
    // v = u - d(t) must be inside
    const bool in = i - dx >= 0 && i - dx < X && j - dy_ >= 0 && j - dy_ < Y && k - dz >= 0 && k - dz < Z;
    g[t] = in ? dy[u - off] * inv_scale : 0.f;
  }
  const bf16x8 * msk = reinterpret_cast<const bf16x8 *>(a5 + u * C);
  bf16x8 *       dst = reinterpret_cast<bf16x8 *>(dz5 + u * C);
#pragma unroll
  for (int q = 0; q < 4; q++)
  {
    const bf16x8 m = msk[q];
    bf16x8       o;
#pragma unroll
    for (int e = 0; e < 8; e++)
    {
      const int ci = 8 * q + e;
      float     acc = 0.f;
#pragma unroll
      for (int t = 0; t < T; t++)
        acc += p[kL6W + t * C + ci] * g[t];
      o[e] = bf16_t(float(m[e]) > 0.f ? acc : 0.f);
    }
    dst[q] = o;
  }
}

// --------------------------------------------------------- weight gradients
// Persistent workgroups: each walks every gridDim.x-th tile of 16 (x) x 4 (y) x 4 (z)
// voxels with its sums in registers and writes them once, to its own slice of `part`;
// wgrad_reduce_kernel adds the slices in a fixed order, so the gradients are the same
// from run to run (per-workgroup atomics on the 27.7k sums of a layer were not).

// Tile `tile` of the batch: its voxel origin and the base of its volume.
struct WgTile
{
  int  x0, y0, z0;
  long vol;
};
__device__ __forceinline__ WgTile
WgTileOf(int tile, int X, int Y, int Z, int tilesX, int tilesY, int tilesZ)
{
  WgTile r;
  r.x0 = (tile % tilesX) * 16;
  tile /= tilesX;
  r.y0 = (tile % tilesY) * 4;
  tile /= tilesY;
  r.z0 = (tile % tilesZ) * 4;
  r.vol = long(tile / tilesZ) * X * Y * Z;
  return r;
}

typedef short    short4v __attribute__((ext_vector_type(4)));
typedef short    short8v __attribute__((ext_vector_type(8)));
using LdsShort4 = __attribute__((address_space(3))) short4v;

// Four 16-bit channels of four voxels, transposed by the LDS read: in each group of 16
// lanes, lane i points at 8 bytes, channels 4 (i % 4) .. + 3 of voxel i / 4, and receives
// channel i of the voxels 0..3 (ds_read_b64_tr_b16).
__device__ __forceinline__ short4v
LdsTranspose(const short * p)
{
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4 *)(p));
}

// dW[t][co][ci] = sum_v dz[v][co] a[v + d(t)][ci];  db[co] = sum_v dz[v][co].
// A GEMM per tap with the voxels as the contracted index: M = co, N = ci, K = 32 voxels
// (two x rows of the tile) per v_mfma_f32_16x16x32_bf16.  Activations are channels-last,
// so both operands are wanted transposed (eight voxels of one channel per lane); the
// transposing LDS read delivers them from the tile as it lies in memory, for every tap
// shift alike (a shift moves the voxel rows, never the alignment).  Both operands take
// the same voxel order inside K, which is all the product needs.
// The tile's a with a one-voxel halo (41.5 KB) and its dz (16 KB) are staged in LDS: two
// workgroups per CU, one loading while the other multiplies.  Wave w takes the taps
// w, w + 4, ..: 7 x 2 x 2 accumulators of 4 FP32 registers; wave 3, with six taps, also
// sums dz (a product with ones).  Voxels outside the volume are zeros in both operands.
// Bound by the LDS reads (a 2 KB operand per 4 matrix instructions) and the staging.
// 4 x 64^3 voxels, one layer: 11.1 ms (one FMA per voxel, tap and channel pair on the
// VALU, every operand from global memory) -> 0.11 ms, and 0.02 ms for the slices.
constexpr int kWgSums = T * C * C + C; // sums of a 32 -> 32 layer

__global__ __launch_bounds__(256) void wgrad32_mfma_kernel(const bf16_t * __restrict__ a,
                                                            const bf16_t * __restrict__ dz, float * __restrict__ part,
                                                            int X, int Y, int Z, int tilesX, int tilesY, int tilesZ,
                                                            int ntiles)
{
  constexpr int HX = 18, HY = 6, HZ = 6, NCHUNK = HX * HY * HZ * 4;
  __shared__ bf16x8 halo[NCHUNK];
  __shared__ bf16x8 dzt[256 * 4];
  const short * hs = reinterpret_cast<const short *>(halo);
  const short * ds = reinterpret_cast<const short *>(dzt);
  const int     lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // this lane's source address inside an x row of voxels: voxel, first channel
  const int     src = (4 * (lane >> 4) + ((lane & 15) >> 2)) * C + 4 * (lane & 3);
  const bf16x8  zero8 = bf16x8{ bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f),
                               bf16_t(0.f), bf16_t(0.f), bf16_t(0.f), bf16_t(0.f) };
  const bf16x8  one8 = bf16x8{ bf16_t(1.f), bf16_t(1.f), bf16_t(1.f), bf16_t(1.f),
                              bf16_t(1.f), bf16_t(1.f), bf16_t(1.f), bf16_t(1.f) };
  floatx4       acc[7][2][2];
#pragma unroll
  for (int i = 0; i < 7; i++)
#pragma unroll
    for (int m = 0; m < 4; m++)
      acc[i][m >> 1][m & 1] = floatx4{ 0.f, 0.f, 0.f, 0.f };

  // K = 32 voxels: x rows y and y + 1 of plane z; `row` is the offset of the first
  auto frag = [&](const short * base, int row, int rowStep, int half) {
    const short4v lo = LdsTranspose(base + row + src + 16 * half);
    const short4v hi = LdsTranspose(base + row + rowStep + src + 16 * half);
    const short8v v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  };
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
  {
    const WgTile w = WgTileOf(tile, X, Y, Z, tilesX, tilesY, tilesZ);
    __syncthreads(); // the previous tile's reads are done
    for (int c = threadIdx.x; c < NCHUNK; c += 256)
    {
      const int part8 = c & 3, vi = c >> 2;
      const int xs = w.x0 - 1 + vi % HX, ys = w.y0 - 1 + (vi / HX) % HY, zs = w.z0 - 1 + vi / (HX * HY);
      bf16x8    v = zero8;
      if (xs >= 0 && xs < X && ys >= 0 && ys < Y && zs >= 0 && zs < Z)
        v = *reinterpret_cast<const bf16x8 *>(a + ((w.vol + (long(zs) * Y + ys) * X + xs) * C + 8 * part8));
      halo[c] = v;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
    {
      const int c = threadIdx.x + 256 * q, part8 = c & 3, vi = c >> 2;
      const int xs = w.x0 + (vi & 15), ys = w.y0 + ((vi >> 4) & 3), zs = w.z0 + (vi >> 6);
      bf16x8    v = zero8;
      if (xs < X && ys < Y && zs < Z)
        v = *reinterpret_cast<const bf16x8 *>(dz + ((w.vol + (long(zs) * Y + ys) * X + xs) * C + 8 * part8));
      dzt[c] = v;
    }
    __syncthreads();
#pragma unroll 1
    for (int s = 0; s < 8; s++)
    {
      const int    z = s >> 1, y = 2 * (s & 1);
      const bf16x8 a0 = frag(ds, (z * 4 + y) * 16 * C, 16 * C, 0), a1 = frag(ds, (z * 4 + y) * 16 * C, 16 * C, 1);
#pragma unroll
      for (int i = 0; i < 7; i++)
      {
        const int t = wave + 4 * i; // uniform; t = 27 (wave 3 only): the sum of dz
        bf16x8    b0 = one8, b1 = one8;
        if (t < T)
        {
          const int row = (((z + t / 9) * HY + y + (t / 3) % 3) * HX + t % 3) * C;
          b0 = frag(hs, row, HX * C, 0);
          b1 = frag(hs, row, HX * C, 1);
        }
        acc[i][0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[i][0][0], 0, 0, 0);
        acc[i][0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b1, acc[i][0][1], 0, 0, 0);
        acc[i][1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b0, acc[i][1][0], 0, 0, 0);
        acc[i][1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[i][1][1], 0, 0, 0);
      }
    }
  }
  // D layout: rows (co) 4 (lane / 16) + q, column (ci) lane % 16
  float * dst = part + size_t(blockIdx.x) * kWgSums;
#pragma unroll
  for (int i = 0; i < 7; i++)
  {
    const int t = wave + 4 * i;
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int q = 0; q < 4; q++)
      {
        const int   co = 16 * (m >> 1) + 4 * (lane >> 4) + q, ci = 16 * (m & 1) + (lane & 15);
        const float v = acc[i][m >> 1][m & 1][q];
        if (t < T)
          dst[(t * C + co) * C + ci] = v;
        else if (ci == 0) // every column holds the sum of dz
          dst[T * C * C + co] = v;
      }
  }
}

// The layers with one channel on one side, as sums over voxels of a 32-channel BF16 field
// m and an FP32 scalar field f:  S[t][c] = sum_v m[v][c] f[v + d(t)].
//   layer 1: dW1[t][c] = s S[t][c] with m = dz1, f = x;  db1[c] = sum_v m[v][c]
//   layer 6: dW6[t][c] = S[26 - t][c] / s with m = a5, f = dy;  db6 = sum_v f[v] / s
// (v + d(t) = u  <=>  u + d(26 - t) = v).
// FP32 on the VALU: a thread is one channel, a half-wave the 32 channels of one voxel, 8
// half-waves the tile's 16 x rows, two each.  f with its halo is staged in LDS and read
// as broadcast rows of 18 values: 5 LDS reads feed 48 FMAs.  VALU-bound (27 FMAs per
// voxel and channel).  4 x 64^3 voxels: 1.21 / 1.24 ms (layers 1 / 6; operands from
// global memory, one voxel a workgroup step) -> 0.09 ms.
constexpr int kWgIoSums = T * C + C + 1; // S, sum of m per channel, sum of f

__global__ __launch_bounds__(256) void wgrad_io_kernel(const float * __restrict__ f, const bf16_t * __restrict__ m,
                                                        float * __restrict__ part, int X, int Y, int Z, int tilesX,
                                                        int tilesY, int tilesZ, int ntiles)
{
  constexpr int HX = 20, HY = 6, HZ = 6; // rows padded from 18 to 20 floats: 16-byte reads
  __shared__ __align__(16) float fh[HX * HY * HZ];
  __shared__ float               red[8][T + 2][C];
  const int c = threadIdx.x & 31, grp = threadIdx.x >> 5;
  float     acc[T], accm = 0.f, accf = 0.f;
#pragma unroll
  for (int t = 0; t < T; t++)
    acc[t] = 0.f;
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
  {
    const WgTile w = WgTileOf(tile, X, Y, Z, tilesX, tilesY, tilesZ);
    __syncthreads();
    for (int q = threadIdx.x; q < HX * HY * HZ; q += 256)
    {
      const int xs = w.x0 - 1 + q % HX, ys = w.y0 - 1 + (q / HX) % HY, zs = w.z0 - 1 + q / (HX * HY);
      fh[q] = (q % HX < 18 && xs >= 0 && xs < X && ys >= 0 && ys < Y && zs >= 0 && zs < Z)
                ? f[w.vol + (long(zs) * Y + ys) * X + xs]
                : 0.f;
    }
    __syncthreads();
#pragma unroll 1
    for (int r = grp; r < 16; r += 8)
    {
      const int y = r & 3, z = r >> 2;
      if (w.y0 + y >= Y || w.z0 + z >= Z)
        continue;
      const bf16_t * src = m + (w.vol + (long(w.z0 + z) * Y + w.y0 + y) * X + w.x0) * C + c;
      float          mv[16];
#pragma unroll
      for (int x = 0; x < 16; x++)
        mv[x] = w.x0 + x < X ? float(src[x * C]) : 0.f;
#pragma unroll
      for (int x = 0; x < 16; x++)
        accm += mv[x];
#pragma unroll
      for (int l = 0; l < 9; l++)
      {
        const float4 * row = reinterpret_cast<const float4 *>(fh + ((z + l / 3) * HY + y + l % 3) * HX);
        float          fv[20];
#pragma unroll
        for (int q = 0; q < 5; q++)
        {
          const float4 v = row[q];
          fv[4 * q] = v.x;
          fv[4 * q + 1] = v.y;
          fv[4 * q + 2] = v.z;
          fv[4 * q + 3] = v.w;
        }
#pragma unroll
        for (int x = 0; x < 16; x++)
#pragma unroll
          for (int d = 0; d < 3; d++)
            acc[3 * l + d] = fmaf(mv[x], fv[x + d], acc[3 * l + d]);
        if (l == 4) // the row itself: its values lie inside the volume or are zero
#pragma unroll
          for (int x = 0; x < 16; x++)
            accf += fv[x + 1];
      }
    }
  }
#pragma unroll
  for (int t = 0; t < T; t++)
    red[grp][t][c] = acc[t];
  red[grp][T][c] = accm;
  red[grp][T + 1][c] = accf; // the same on every channel
  __syncthreads();
  float * dst = part + size_t(blockIdx.x) * kWgIoSums;
  for (int q = threadIdx.x; q < kWgIoSums; q += 256)
  {
    float v = 0.f;
#pragma unroll
    for (int g = 0; g < 8; g++)
      v += red[g][q / C][q % C];
    dst[q] = v;
  }
}

// dst(slot) = sum over the workgroups' slices, in a fixed order: a workgroup takes 16
// slots (64-byte reads), its 16 rows of threads every 16th slice each.  `where` maps a slot
// to its place and factor.
template <class F>
__device__ __forceinline__ void
WgReduce(const float * __restrict__ part, int nslots, int nslices, F && where)
{
  __shared__ float red[16][17];
  const int slot = blockIdx.x * 16 + (threadIdx.x & 15), row = threadIdx.x >> 4;
  float     v = 0.f;
  if (slot < nslots)
#pragma unroll 8
    for (int b = row; b < nslices; b += 16)
      v += part[size_t(b) * nslots + slot];
  red[row][threadIdx.x & 15] = v;
  __syncthreads();
  if (row == 0 && slot < nslots)
  {
    float s = red[0][threadIdx.x];
#pragma unroll
    for (int r = 1; r < 16; r++)
      s += red[r][threadIdx.x];
    where(slot, s);
  }
}

// 32 -> 32 layer: W and b lie together, in the order of the slots.
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const float * __restrict__ part, int nslices,
                                                            float * __restrict__ g)
{
  WgReduce(part, kWgSums, nslices, [&](int slot, float v) { g[slot] = v; });
}

__global__ __launch_bounds__(256) void wgrad_io_reduce_kernel(const float * __restrict__ part, int nslices,
                                                               float * __restrict__ g, float factor, int last)
{
  WgReduce(part, kWgIoSums, nslices, [&](int slot, float v) {
    const int t = slot / C, c = slot % C;
    if (t < T)
      g[last ? (T - 1 - t) * C + c : slot] = factor * v;
    else if (last ? slot == kWgIoSums - 1 : t == T)
      g[T * C + c] = last ? factor * v : v; // db6 (one value), db1 (per channel)
  });
}

// ------------------------------------------------------------ loss, Adam, packing
// dy = 2 s^2 (y - t) / N; partial sums of s^2 (y - t)^2 (FP64, fixed order).
__global__ __launch_bounds__(256) void mse_kernel(const float * __restrict__ y, const float * __restrict__ t,
                                                   float * __restrict__ dy, long n, float scale2, double * partial)
{
  __shared__ double sh[4];
  double            acc = 0.;
  for (long i = long(blockIdx.x) * 256 + threadIdx.x; i < n; i += long(gridDim.x) * 256)
  {
    const float d = y[i] - t[i];
    dy[i] = 2.f * scale2 * d / float(n);
    acc += double(scale2) * double(d) * double(d);
  }
  for (int o = 32; o > 0; o >>= 1)
    acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0)
    sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0)
    partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ void adam_kernel(float * __restrict__ p, const float * __restrict__ g, float * __restrict__ m,
                            float * __restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n)
    return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 copies of the four 32->32 layers: forward [t][co][ci] and data-gradient
// [t'][ci][co] = W[26 - t'][co][ci] (flipped taps, swapped channel roles).
__global__ void pack_kernel(const float * __restrict__ p, bf16_t * __restrict__ wf, bf16_t * __restrict__ wb)
{
  const int idx = blockIdx.x * 256 + threadIdx.x; // over 4 * 27 * 32 * 32
  if (idx >= 4 * T * C * C)
    return;
  const int l = idx / (T * C * C), r = idx % (T * C * C);
  const int t = r / (C * C), co = (r / C) % C, ci = r % C;
  const float wv = p[kMidBase + l * kMidSize + r];
  wf[idx] = bf16_t(wv);
  wb[l * T * C * C + ((T - 1 - t) * C + ci) * C + co] = bf16_t(wv);
}

} // namespace cnn
} // namespace rtkhip

// ------------------------------------------------------------------ handle
struct rtkhip_cnn
{
  rtkhip::DeviceBuffer<float>   params, grads, m, v, dy, out;
  rtkhip::DeviceBuffer<float>   wpart; // per-workgroup sums of the weight gradients (57 MB)
  rtkhip::DeviceBuffer<bf16_t>  wf, wb, act, dz0, dz1;
  rtkhip::DeviceBuffer<double>  partial;
  long                          nvox = 0; // voxels of the activations kept for backward
  int                           dims[4] = { 0, 0, 0, 0 };
  float                         scale = 1.f;
  const float *                 lastIn = nullptr;
};

namespace rtkhip
{
namespace cnn
{
namespace
{

void
Reserve(rtkhip_cnn & net, long nvox)
{
  net.act.Resize(size_t(5) * nvox * C); // A1..A5
  net.out.Resize(size_t(nvox));
}

void
ForwardImpl(rtkhip_cnn & net, int B, const int d[3], const float * in, float * out, float scale, hipStream_t s)
{
  const int  X = d[0], Y = d[1], Z = d[2];
  const long n = long(B) * X * Y * Z;
  Reserve(net, n);
  bf16_t *  A = net.act.get();
  const long     plane = long(X) * Y, chunks = (plane + 255) / 256; // of the kernels of a thread per voxel
  RTKHIP_REQUIRE(plane < (1L << 32) - 256 && chunks * Z * B < (1L << 31), RTKHIP_ERR_UNSUPPORTED, "cnn: volume too large");
  hipLaunchKernelGGL(conv_in_kernel, dim3(unsigned(chunks * Z * B)), dim3(256), 0, s, in, net.params.get(), A,
                     unsigned(chunks), X, Y, Z, scale);
  RTKHIP_CHECK_LAUNCH();
  const int tilesX = (X + 15) / 16, tilesY = (Y + kRowsY - 1) / kRowsY, tilesZ = (Z + 3) / 4;
  const long nb = long(B) * tilesX * tilesY * tilesZ;
  RTKHIP_REQUIRE(nb < (1L << 31), RTKHIP_ERR_UNSUPPORTED, "cnn: volume too large");
  for (int l = 0; l < 4; l++)
  {
    const bf16_t * ain = A + size_t(l) * n * C;
    bf16_t *       aout = A + size_t(l + 1) * n * C;
    hipLaunchKernelGGL((conv32_mfma_kernel<true, false>), dim3(unsigned(nb)), dim3(256), 0, s, ain,
                       net.wf.get() + size_t(l) * T * C * C, net.params.get() + kMidBase + l * kMidSize + T * C * C,
                       nullptr, aout, X, Y, Z, tilesX, tilesY, tilesZ);
    RTKHIP_CHECK_LAUNCH();
  }
  // z planes a workgroup marches through: two more are read, so long runs, but at least
  // four workgroups per CU where the volume has them
  const int  outX = (X + kOutX - 1) / kOutX, outY = (Y + kOutX - 1) / kOutX;
  const long cols = long(B) * outX * outY;
  const int  zrun = int(std::max<long>(4, std::min<long>(64, long(Z) * cols / 1024)));
  const int  runs = (Z + zrun - 1) / zrun;
  RTKHIP_REQUIRE(cols * runs < (1L << 31), RTKHIP_ERR_UNSUPPORTED, "cnn: volume too large");
  hipLaunchKernelGGL(conv_out_kernel, dim3(unsigned(cols * runs)), dim3(256), 0, s, A + size_t(4) * n * C, in,
                     net.params.get(), out, X, Y, Z, outX, outY, zrun, runs, 1.f / scale);
  RTKHIP_CHECK_LAUNCH();
  net.nvox = n;
  net.dims[0] = B;
  net.dims[1] = X;
  net.dims[2] = Y;
  net.dims[3] = Z;
  net.scale = scale;
  net.lastIn = in;
}

// Workgroups of the weight-gradient kernels: two per CU (their LDS), or one a tile.
constexpr int kWgGroups = 512;

} // namespace
} // namespace cnn
} // namespace rtkhip

using namespace rtkhip;
using namespace rtkhip::cnn;

extern "C" int
rtkhip_cnn_num_params(void)
{
  return kNumParams;
}

extern "C" rtkhip_cnn *
rtkhip_cnn_create(void)
{
  rtkhip_cnn * net = nullptr;
  int          rc = Guard([&] {
    RequireDevice();
    net = new rtkhip_cnn();
    net->params.Resize(kNumParams);
    net->grads.Resize(kNumParams);
    net->m.Resize(kNumParams);
    net->v.Resize(kNumParams);
    net->wf.Resize(size_t(4) * T * C * C);
    net->wb.Resize(size_t(4) * T * C * C);
    net->partial.Resize(2048);
    RTKHIP_CHECK(hipMemset(net->params.get(), 0, sizeof(float) * kNumParams));
    RTKHIP_CHECK(hipMemset(net->m.get(), 0, sizeof(float) * kNumParams));
    RTKHIP_CHECK(hipMemset(net->v.get(), 0, sizeof(float) * kNumParams));
  });
  if (rc != RTKHIP_OK)
  {
    delete net;
    return nullptr;
  }
  return net;
}

extern "C" void
rtkhip_cnn_destroy(rtkhip_cnn * net)
{
  delete net;
}

extern "C" int
rtkhip_cnn_set_params(rtkhip_cnn * net, const float * host_params, void * stream)
{
  return Guard([&] {
    RTKHIP_REQUIRE(net && host_params, RTKHIP_ERR_INVALID_ARGUMENT, "cnn_set_params: null argument");
    hipStream_t s = Stream(stream);
    RTKHIP_CHECK(hipMemcpyAsync(net->params.get(), host_params, sizeof(float) * kNumParams, hipMemcpyHostToDevice, s));
    RTKHIP_CHECK(hipMemsetAsync(net->m.get(), 0, sizeof(float) * kNumParams, s));
    RTKHIP_CHECK(hipMemsetAsync(net->v.get(), 0, sizeof(float) * kNumParams, s));
    hipLaunchKernelGGL(pack_kernel, dim3((4 * T * C * C + 255) / 256), dim3(256), 0, s, net->params.get(),
                       net->wf.get(), net->wb.get());
    RTKHIP_CHECK_LAUNCH();
    RTKHIP_CHECK(hipStreamSynchronize(s));
  });
}

extern "C" int
rtkhip_cnn_get_params(rtkhip_cnn * net, float * host_params, float * host_grads, void * stream)
{
  return Guard([&] {
    RTKHIP_REQUIRE(net, RTKHIP_ERR_INVALID_ARGUMENT, "cnn_get_params: null network");
    hipStream_t s = Stream(stream);
    if (host_params)
      RTKHIP_CHECK(
        hipMemcpyAsync(host_params, net->params.get(), sizeof(float) * kNumParams, hipMemcpyDeviceToHost, s));
    if (host_grads)
      RTKHIP_CHECK(
        hipMemcpyAsync(host_grads, net->grads.get(), sizeof(float) * kNumParams, hipMemcpyDeviceToHost, s));
    RTKHIP_CHECK(hipStreamSynchronize(s));
  });
}

extern "C" int
rtkhip_cnn_forward(rtkhip_cnn * net, int batch, const int dim[3], const float * dev_in, float * dev_out, float scale,
                   void * stream)
{
  return Guard([&] {
    RTKHIP_REQUIRE(net && dim && dev_in && dev_out && batch > 0 && scale > 0.f, RTKHIP_ERR_INVALID_ARGUMENT,
                   "cnn_forward: bad argument");
    RTKHIP_REQUIRE(dim[0] > 0 && dim[1] > 0 && dim[2] > 0, RTKHIP_ERR_INVALID_ARGUMENT, "cnn_forward: bad size");
    RTKHIP_REQUIRE(dev_in != dev_out, RTKHIP_ERR_INVALID_ARGUMENT, "cnn_forward: in-place is not supported");
    ForwardImpl(*net, batch, dim, dev_in, dev_out, scale, Stream(stream));
  });
}

extern "C" int
rtkhip_cnn_backward(rtkhip_cnn * net, const float * dev_out, const float * dev_target, double * loss, void * stream)
{
  return Guard([&] {
    RTKHIP_REQUIRE(net && dev_out && dev_target && net->nvox > 0 && net->lastIn, RTKHIP_ERR_INVALID_ARGUMENT,
                   "cnn_backward: call rtkhip_cnn_forward first");
    hipStream_t s = Stream(stream);
    const int   B = net->dims[0], X = net->dims[1], Y = net->dims[2], Z = net->dims[3];
    const long  n = net->nvox;
    const float sc = net->scale;
    net->dy.Resize(size_t(n));
    net->dz0.Resize(size_t(n) * C);
    net->dz1.Resize(size_t(n) * C);
    float *  P = net->params.get();
    float *  G = net->grads.get();
    bf16_t * A = net->act.get();
    // loss and dL/dy
    const int gl = int(std::min<long>((n + 255) / 256, 2048));
    hipLaunchKernelGGL(mse_kernel, dim3(gl), dim3(256), 0, s, dev_out, dev_target, net->dy.get(), n, sc * sc,
                       net->partial.get());
    RTKHIP_CHECK_LAUNCH();
    const int  tilesX = (X + 15) / 16, tilesY = (Y + 3) / 4, tilesZ = (Z + 3) / 4; // of the weight gradients
    const int  convY = (Y + kRowsY - 1) / kRowsY;                                  // of the data gradients
    const long nb = long(B) * tilesX * tilesY * tilesZ, nconv = long(B) * tilesX * convY * tilesZ;
    RTKHIP_REQUIRE(nb < (1L << 31), RTKHIP_ERR_UNSUPPORTED, "cnn: volume too large");
    const int  ng = int(std::min<long>(nb, kWgGroups));
    net->wpart.Resize(size_t(ng) * kWgSums);
    float * part = net->wpart.get();
    auto    wgradIo = [&](const float * f, const bf16_t * m, float * g, float factor, int last) {
      hipLaunchKernelGGL(wgrad_io_kernel, dim3(ng), dim3(256), 0, s, f, m, part, X, Y, Z, tilesX, tilesY, tilesZ,
                         int(nb));
      RTKHIP_CHECK_LAUNCH();
      hipLaunchKernelGGL(wgrad_io_reduce_kernel, dim3((kWgIoSums + 15) / 16), dim3(256), 0, s, part, ng, g, factor,
                         last);
      RTKHIP_CHECK_LAUNCH();
    };
    // layer 6
    wgradIo(net->dy.get(), A + size_t(4) * n * C, G + kL6W, 1.f / sc, 1);
    const long chunks = (long(X) * Y + 255) / 256; // checked by the forward pass
    hipLaunchKernelGGL(conv_out_bwd_data_kernel, dim3(unsigned(chunks * Z * B)), dim3(256), 0, s, net->dy.get(), P,
                       A + size_t(4) * n * C, net->dz0.get(), unsigned(chunks), X, Y, Z, 1.f / sc);
    RTKHIP_CHECK_LAUNCH();
    // layers 5..2: dZ_l in dz_cur; weight grads from A_{l-1}; data grad masked by A_{l-1}
    bf16_t * cur = net->dz0.get();
    bf16_t * nxt = net->dz1.get();
    for (int l = 3; l >= 0; l--) // mid layer index l = layer (l + 2)
    {
      const bf16_t * aprev = A + size_t(l) * n * C; // A_{layer-1} = A[l]
      hipLaunchKernelGGL(wgrad32_mfma_kernel, dim3(ng), dim3(256), 0, s, aprev, cur, part, X, Y, Z, tilesX, tilesY,
                         tilesZ, int(nb));
      RTKHIP_CHECK_LAUNCH();
      hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((kWgSums + 15) / 16), dim3(256), 0, s, part, ng,
                         G + kMidBase + l * kMidSize);
      RTKHIP_CHECK_LAUNCH();
      hipLaunchKernelGGL((conv32_mfma_kernel<false, true>), dim3(unsigned(nconv)), dim3(256), 0, s, cur,
                         net->wb.get() + size_t(l) * T * C * C, nullptr, aprev, nxt, X, Y, Z, tilesX, convY,
                         tilesZ);
      RTKHIP_CHECK_LAUNCH();
      std::swap(cur, nxt);
    }
    // layer 1 (cur = dZ1)
    wgradIo(net->lastIn, cur, G + kL1W, sc, 0);
    if (loss)
    {
      std::vector<double> h(gl);
      RTKHIP_CHECK(hipMemcpyAsync(h.data(), net->partial.get(), sizeof(double) * gl, hipMemcpyDeviceToHost, s));
      RTKHIP_CHECK(hipStreamSynchronize(s));
      double sum = 0.;
      for (double x : h)
        sum += x;
      *loss = sum / double(n);
    }
  });
}

extern "C" int
rtkhip_cnn_adam_step(rtkhip_cnn * net, float lr, float beta1, float beta2, float eps, int step, void * stream)
{
  return Guard([&] {
    RTKHIP_REQUIRE(net && step >= 1, RTKHIP_ERR_INVALID_ARGUMENT, "cnn_adam_step: bad argument");
    hipStream_t s = Stream(stream);
    const float c1 = 1.f - std::pow(beta1, float(step)), c2 = 1.f - std::pow(beta2, float(step));
    hipLaunchKernelGGL(adam_kernel, dim3((kNumParams + 255) / 256), dim3(256), 0, s, net->params.get(),
                       net->grads.get(), net->m.get(), net->v.get(), kNumParams, lr, beta1, beta2, eps, c1, c2);
    RTKHIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(pack_kernel, dim3((4 * T * C * C + 255) / 256), dim3(256), 0, s, net->params.get(),
                       net->wf.get(), net->wb.get());
    RTKHIP_CHECK_LAUNCH();
  });
}
