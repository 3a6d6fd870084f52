// MI355X (gfx950) kernels of the learned interface closure: a 3x3x3, 32
// channel 3D CNN in BF16 with FP32 accumulation on the matrix cores, its
// backward pass (data and weight gradients), a weighted squared-error loss,
// Adam, and the feature / gain maps that connect it to the 3D solver's heat
// exchange.
//
// Convolution as an implicit GEMM on v_mfma_f32_16x16x32_bf16: the GEMM row
// is the output cell, the column the output channel and the reduction runs
// over (tap, input channel) in chunks of 32 input channels, one tap per MFMA.
// Channels-last activations make each lane's A operand one 16-byte load
// (8 channels of one neighbour cell).  Operand lane layout (16x16x32):
//   A (16 x 32): lane l holds row l % 16, reduction elements 8 * (l / 16) + e;
//   B (32 x 16): lane l holds column l % 16, the same reduction elements;
//   D (16 x 16): lane l holds rows 4 * (l / 16) + r, column l % 16.
// A and B use the same reduction index map, so the product does not depend
// on how the hardware orders the reduction elements within a lane.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "icyclosure.h"

namespace icyc {

constexpr int kC = ICYC_CHANNELS;
constexpr int kTaps = ICYC_TAPS;
constexpr int kLayer = ICYC_LAYER_PARAMS;
constexpr int kWeights = kTaps * kC * kC;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);                      // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ floatx4 mfma(bf16x8 a, bf16x8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ------------------------------------------------------------ convolution
// One wave: 8 row tiles of 16 consecutive cells x 32 output channels.
constexpr int kConvThreads = 256;
constexpr int kRowTiles = 8;
constexpr int kCellsPerWave = 16 * kRowTiles;
constexpr int kCellsPerBlock = kCellsPerWave * (kConvThreads / 64);

template <int Epi>
__global__ void __launch_bounds__(kConvThreads)
    k_conv3d(int nx, int ny, int nz, const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
             const float* __restrict__ bias, const uint16_t* __restrict__ mask, uint16_t* __restrict__ out,
             float* __restrict__ out_f32) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long N = (long)nx * ny * nz;
  const long base = (long)blockIdx.x * kCellsPerBlock + (long)wave * kCellsPerWave;
  const int row = lane & 15, group = lane >> 4;
  int ci[kRowTiles], cj[kRowTiles], ck[kRowTiles];
#pragma unroll
  for (int mt = 0; mt < kRowTiles; ++mt) {
    const long m = base + mt * 16 + row;
    ck[mt] = (int)(m % nz);
    cj[mt] = (int)((m / nz) % ny);
    ci[mt] = m < N ? (int)(m / ((long)nz * ny)) : -1000;  // past the end: never inside
  }
  floatx4 acc[kRowTiles][2];
#pragma unroll
  for (int mt = 0; mt < kRowTiles; ++mt) acc[mt][0] = acc[mt][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int t = 0; t < kTaps; ++t) {
    const int di = t / 9 - 1, dj = (t / 3) % 3 - 1, dk = t % 3 - 1;
    const uint4* wt = reinterpret_cast<const uint4*>(w + (long)t * kC * kC);
    const bf16x8 b0 = as_bf16x8(wt[(row * kC + group * 8) / 8]);
    const bf16x8 b1 = as_bf16x8(wt[((16 + row) * kC + group * 8) / 8]);
#pragma unroll
    for (int mt = 0; mt < kRowTiles; ++mt) {
      const int i = ci[mt] + di, j = cj[mt] + dj, k = ck[mt] + dk;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz)
        v = *reinterpret_cast<const uint4*>(in + (((long)i * ny + j) * nz + k) * kC + group * 8);
      const bf16x8 a = as_bf16x8(v);
      acc[mt][0] = mfma(a, b0, acc[mt][0]);
      acc[mt][1] = mfma(a, b1, acc[mt][1]);
    }
  }
#pragma unroll
  for (int mt = 0; mt < kRowTiles; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int co = nt * 16 + row;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long cell = base + mt * 16 + group * 4 + r;
        if (cell >= N) continue;
        const float x = acc[mt][nt][r];
        if (Epi == ICYC_RELU_BF16) {
          out[cell * kC + co] = f2bf(fmaxf(0.0f, x + bias[co]));
        } else if (Epi == ICYC_LINEAR_F32) {
          if (co == 0) out_f32[cell] = x + bias[0];
        } else {
          out[cell * kC + co] = bf2f(mask[cell * kC + co]) > 0.0f ? f2bf(x) : (uint16_t)0;
        }
      }
    }
}

// The form for z-columns of 16, 32, 48 or 64 cells.  A product of 16 cells x
// 16 output channels over one tap's 32 input channels is one
// v_mfma_f32_16x16x32_bf16, 16 cycles of a SIMD's matrix core, and needs 1 KB
// an operand: with both operands read from LDS four SIMDs ask for four times
// what it delivers.  So a wave keeps its 16 channels' weights of all 27 taps
// in registers (108), and the block sweeps along x with three output slabs in
// accumulators: a cell operand read once from LDS (own slab s, shift dj, dk)
// feeds the outputs of slabs s - 1, s and s + 1.  The next slab travels from
// memory to registers meanwhile and into the second LDS buffer after; one
// barrier a slab.
//   - The weights are operand A (rows: output channels) and the cells operand
//     B, so a lane ends up with 4 consecutive channels of one cell (8 bytes).
//   - Eight waves: two halves of the channels times four groups of T tiles of
//     16 cells, over kSweepCols columns of y and `per` slabs of x.
//   - LDS holds 16-byte pieces (8 channels); piece c of cell m sits at
//     c ^ (m / 4 % 4), so that 16 consecutive cells' pieces cover all banks.
// A wave with all 32 channels (v_mfma_f32_32x32x16, 216 weight registers, one
// wave a SIMD) left the compiler no registers to read ahead: 67 us at
// 128x64x64 against 35 us here, and 79 us for 2 x 2 staged columns a block
// with the weights read from memory for every tap (masked form: 101 to 40 us).
//
// Two floats as packed BF16, rounded to nearest even.
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}
// `value` where the packed BF16 pair `m` is positive, else zero.
__device__ __forceinline__ uint32_t keep_positive(uint32_t value, uint32_t m) {
  const uint32_t lo = ((m & 0xffffu) - 1u) < 0x7f80u ? 0xffffu : 0u;
  const uint32_t hi = ((m >> 16) - 1u) < 0x7f80u ? 0xffff0000u : 0u;
  return value & (lo | hi);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxColumn = 64;
constexpr int kSweepThreads = 512, kSweepCols = 4;
constexpr int kSweepColumn = (kMaxColumn + 2) * 4, kSweepSlab = (kSweepCols + 2) * kSweepColumn;
template <int Epi, int T>
__global__ void __launch_bounds__(kSweepThreads, 2)
    k_conv3d_sweep(int nx, int ny, int per, const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                   const float* __restrict__ bias, const uint16_t* __restrict__ mask, uint16_t* __restrict__ out) {
  constexpr int nz = 16 * T;  // four columns of nz cells are 4 T tiles, T a wave
  constexpr int kPieces = (kSweepCols + 2) * nz * 4;
  constexpr int kFetch = (kPieces + kSweepThreads - 1) / kSweepThreads;  // 16-byte pieces a thread stages
  __shared__ u32x4 xs[2][kSweepSlab];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & 15, group = lane >> 4;
  const int channels = (wave & 1) * 16, tile0 = (wave >> 1) * T;
  const int tiles_j = (ny + kSweepCols - 1) / kSweepCols;
  const int j0 = (int)(blockIdx.x % tiles_j) * kSweepCols, x0 = (int)(blockIdx.x / tiles_j) * per;
  const int x1 = min(nx, x0 + per);
  for (int e = threadIdx.x; e < 2 * kSweepSlab; e += kSweepThreads) (&xs[0][0])[e] = u32x4{0u, 0u, 0u, 0u};
  bf16x8 wr[kTaps];
#pragma unroll
  for (int t = 0; t < kTaps; ++t)
    wr[t] = *reinterpret_cast<const bf16x8*>(w + ((long)t * kC + channels + row) * kC + 8 * group);
  float bias_r[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) bias_r[r] = Epi == ICYC_RELU_BF16 ? bias[channels + 4 * group + r] : 0.0f;
  // Staging: piece e % 4 of cell e / 4 of the slab's columns; a thread
  // without a piece reads the slab's first and stores none.
  long src[kFetch];
  int dst[kFetch];
#pragma unroll
  for (int f = 0; f < kFetch; ++f) {
    const int e = threadIdx.x + f * kSweepThreads, col = e / (nz * 4), k = e / 4 % nz, c = e % 4, j = j0 - 1 + col;
    const bool mine = e < kPieces && j >= 0 && j < ny;
    src[f] = mine ? (long)(j * nz + k) * 4 + c : 0;
    dst[f] = mine ? col * kSweepColumn + (k + 1) * 4 + (c ^ (((k + 1) >> 2) & 3)) : -1;
  }
  u32x4 fetched[kFetch];
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const u32x4* slab = reinterpret_cast<const u32x4*>(in) + (long)s * ny * nz * 4;
#pragma unroll
    for (int f = 0; f < kFetch; ++f) fetched[f] = slab[src[f]];
  };
  auto stage = [&](u32x4* buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < kFetch; ++f)
      if (dst[f] >= 0) buffer[dst[f]] = fetched[f];
  };
  // This lane's cell of each tile, and where its operand pieces start.
  int at[T][3], cell_j[T], cell_k[T];
#pragma unroll
  for (int tl = 0; tl < T; ++tl) {
    const int m = tile0 + tl;
    cell_j[tl] = m / T;
    cell_k[tl] = m % T * 16 + row;
#pragma unroll
    for (int dk = 0; dk < 3; ++dk) {
      const int cell = cell_k[tl] + dk;
      at[tl][dk] = cell_j[tl] * kSweepColumn + cell * 4 + (group ^ ((cell >> 2) & 3));
    }
  }
  __syncthreads();
  if (x0 > 0) {
    fetch(x0 - 1);
    stage(xs[0]);
  }
  int current = 0;
  floatx4 acc[3][T];
  // Slab s into the outputs of slabs s - 1 (accumulators P), s (C) and s + 1
  // (N, cleared here); then the finished outputs of slab s - 1.
  auto step = [&](int s, floatx4(&P)[T], floatx4(&C)[T], floatx4(&N)[T]) __attribute__((always_inline)) {
    __syncthreads();
    const bool more = s + 1 <= x1 && s + 1 < nx;
    if (more) fetch(s + 1);
#pragma unroll
    for (int tl = 0; tl < T; ++tl) N[tl] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const bool do_p = s - 1 >= x0, do_c = s >= x0 && s < x1, do_n = s + 1 < x1;
    if (s >= 0 && s < nx) {
      const u32x4* buffer = xs[current];
      if (do_p && do_c && do_n) {
#pragma unroll
        for (int dj = 0; dj < 3; ++dj)
#pragma unroll
          for (int dk = 0; dk < 3; ++dk) {
            bf16x8 b[T];
#pragma unroll
            for (int tl = 0; tl < T; ++tl)
              b[tl] = __builtin_bit_cast(bf16x8, buffer[at[tl][dk] + dj * kSweepColumn]);
#pragma unroll
            for (int tl = 0; tl < T; ++tl) {
              P[tl] = mfma(wr[18 + 3 * dj + dk], b[tl], P[tl]);
              C[tl] = mfma(wr[9 + 3 * dj + dk], b[tl], C[tl]);
              N[tl] = mfma(wr[3 * dj + dk], b[tl], N[tl]);
            }
          }
      } else {  // the first and last slabs: one or two of the three
        auto plane = [&](int first, floatx4(&A)[T]) __attribute__((always_inline)) {
#pragma unroll
          for (int e = 0; e < 9; ++e)
#pragma unroll
            for (int tl = 0; tl < T; ++tl)
              A[tl] = mfma(wr[first + e],
                           __builtin_bit_cast(bf16x8, buffer[at[tl][e % 3] + e / 3 * kSweepColumn]), A[tl]);
        };
        if (do_p) plane(18, P);
        if (do_c) plane(9, C);
        if (do_n) plane(0, N);
      }
    }
    if (do_p) {
#pragma unroll
      for (int tl = 0; tl < T; ++tl) {
        const int j = j0 + cell_j[tl];
        if (j >= ny) continue;
        const long cell = ((long)(s - 1) * ny + j) * nz + cell_k[tl];
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = Epi == ICYC_RELU_BF16 ? fmaxf(0.0f, P[tl][r] + bias_r[r]) : P[tl][r];
        uint2 packed = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
        const long at_c = cell * kC + channels + 4 * group;
        if (Epi == ICYC_MASKED_BF16) {
          const uint2 m = *reinterpret_cast<const uint2*>(mask + at_c);
          packed = make_uint2(keep_positive(packed.x, m.x), keep_positive(packed.y, m.y));
        }
        *reinterpret_cast<uint2*>(out + at_c) = packed;
      }
    }
    current ^= 1;
    if (more) stage(xs[current]);
  };
  for (int s = x0 - 1;;) {
    step(s, acc[0], acc[1], acc[2]);
    if (++s > x1) break;
    step(s, acc[1], acc[2], acc[0]);
    if (++s > x1) break;
    step(s, acc[2], acc[0], acc[1]);
    if (++s > x1) break;
  }
}

// The first layer's form: its input has 8 real channels (the features), so
// one v_mfma_f32_16x16x32_bf16 takes four taps' 8 channels as its reduction
// (lane group g: tap 4 m + g), 7 products for 16 cells x 16 channels.  Bound
// by memory (64 bytes a cell in, of which 16 count but a line comes whole, 64
// out).  The sweep of k_conv3d_sweep with one output slab: the last slabs'
// pieces stay in a ring of four.  2 x 2 columns a block, staged with all their
// neighbours and stored a channel at a time, took 33 us at 128x64x64,
// this 20.
template <int Epi, int T>
__global__ void __launch_bounds__(kSweepThreads)
    k_conv3d_first(int nx, int ny, int per, const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                   const float* __restrict__ bias, uint16_t* __restrict__ out, float* __restrict__ out_f32) {
  constexpr int nz = 16 * T, kCells = (kSweepCols + 2) * nz, kFetch = (kCells + kSweepThreads - 1) / kSweepThreads;
  constexpr int kColumn = kMaxColumn + 2, kSlab = (kSweepCols + 2) * kColumn, kGroups = (kTaps + 3) / 4;
  __shared__ u32x4 ring[4][kSlab];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & 15, group = lane >> 4;
  const int channels = (wave & 1) * 16, tile0 = (wave >> 1) * T;
  const int tiles_j = (ny + kSweepCols - 1) / kSweepCols;
  const int j0 = (int)(blockIdx.x % tiles_j) * kSweepCols, x0 = (int)(blockIdx.x / tiles_j) * per;
  const int x1 = min(nx, x0 + per);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int e = threadIdx.x; e < 4 * kSlab; e += kSweepThreads) (&ring[0][0])[e] = zero;
  bf16x8 wr[kGroups];
  int di[kGroups], at[kGroups];  // of this lane's tap in each product: slab shift, offset in a slab
#pragma unroll
  for (int m = 0; m < kGroups; ++m) {
    const int t = min(4 * m + group, kTaps - 1);
    wr[m] = __builtin_bit_cast(bf16x8, zero);
    if (4 * m + group < kTaps) wr[m] = *reinterpret_cast<const bf16x8*>(w + ((long)t * kC + channels + row) * kC);
    di[m] = t / 9;
    at[m] = t / 3 % 3 * kColumn + t % 3;
  }
  long src[kFetch];
  int dst[kFetch];
#pragma unroll
  for (int f = 0; f < kFetch; ++f) {
    const int e = threadIdx.x + f * kSweepThreads, col = e / nz, k = e % nz, j = j0 - 1 + col;
    const bool mine = e < kCells && j >= 0 && j < ny;
    src[f] = mine ? (long)(j * nz + k) * 4 : 0;
    dst[f] = mine ? col * kColumn + k + 1 : -1;
  }
  u32x4 fetched[kFetch];
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const u32x4* slab = reinterpret_cast<const u32x4*>(in) + (long)min(max(s, 0), nx - 1) * ny * nz * 4;
#pragma unroll
    for (int f = 0; f < kFetch; ++f) fetched[f] = slab[src[f]];
  };
  auto stage = [&](int s) __attribute__((always_inline)) {
    const bool real = s >= 0 && s < nx;
#pragma unroll
    for (int f = 0; f < kFetch; ++f)
      if (dst[f] >= 0) ring[s & 3][dst[f]] = real ? fetched[f] : zero;
  };
  __syncthreads();
  fetch(x0 - 1);
  stage(x0 - 1);
  fetch(x0);
  stage(x0);
  fetch(x0 + 1);
  for (int i = x0; i < x1; ++i) {
    stage(i + 1);  // the slot of slab i - 3, which no wave reads any more
    __syncthreads();
    if (i + 1 < x1) fetch(i + 2);
    floatx4 acc[T];
#pragma unroll
    for (int tl = 0; tl < T; ++tl) acc[tl] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < kGroups; ++m) {
      const u32x4* slab = &ring[0][0] + ((i - 1 + di[m]) & 3) * kSlab + at[m];
#pragma unroll
      for (int tl = 0; tl < T; ++tl) {
        const int f = (tile0 + tl) * 16 + row;
        u32x4 x = slab[f / nz * kColumn + f % nz];
        if (4 * m + 3 >= kTaps && 4 * m + group >= kTaps) x = zero;
        acc[tl] = mfma(wr[m], __builtin_bit_cast(bf16x8, x), acc[tl]);
      }
    }
#pragma unroll
    for (int tl = 0; tl < T; ++tl) {
      const int f = (tile0 + tl) * 16 + row, j = j0 + f / nz;
      if (j >= ny) continue;
      const long cell = ((long)i * ny + j) * nz + f % nz;
      if (Epi == ICYC_LINEAR_F32) {
        if (channels + group == 0) out_f32[cell] = acc[tl][0] + bias[0];
      } else {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaxf(0.0f, acc[tl][r] + bias[channels + 4 * group + r]);
        *reinterpret_cast<uint2*>(out + cell * kC + channels + 4 * group) =
            make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
      }
    }
  }
}

// ------------------------------------------------------- the scalar layer
// The last layer has one output, so its convolution and both gradients are
// narrow: 27 taps by 32 channels.  The taps become a matrix dimension.
typedef float floatx16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ floatx16 mfma32(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
constexpr int kScalarCols = 8;
// Forward: Y[t][x] = sum over ci of w[t][0][ci] in[x][ci] (two products of 32
// taps x 32 cells, operands straight from memory: every line is read whole),
// then out[x] = bias + sum over t of Y[t][x + off(t)] from LDS, three output
// slabs in a thread's registers.  Bound by reading the input once; as one of
// 16 channels of the general form 30 us at 128x64x64, 14 here.
constexpr int kTapThreads = 512, kTapColumn = kMaxColumn + 2, kTapRow = (kScalarCols + 2) * kTapColumn + 4;
template <int T>
__global__ void __launch_bounds__(kTapThreads)
    k_conv3d_taps(int nx, int ny, int per, const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                  const float* __restrict__ bias, float* __restrict__ out) {
  constexpr int nz = 16 * T, kTiles = ((kScalarCols + 2) * nz + 31) / 32;
  constexpr int kPerWave = (kTiles + kTapThreads / 64 - 1) / (kTapThreads / 64);
  __shared__ float y[kTaps][kTapRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5;
  const int tiles_j = (ny + kScalarCols - 1) / kScalarCols;
  const int j0 = (int)(blockIdx.x % tiles_j) * kScalarCols, x0 = (int)(blockIdx.x / tiles_j) * per;
  const int x1 = min(nx, x0 + per);
  for (int e = threadIdx.x; e < kTaps * kTapRow; e += kTapThreads) (&y[0][0])[e] = 0.0f;
  bf16x8 wr[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    wr[h] = as_bf16x8(make_uint4(0u, 0u, 0u, 0u));
    if ((lane & 31) < kTaps)
      wr[h] = *reinterpret_cast<const bf16x8*>(w + (long)(lane & 31) * kC * kC + 16 * h + 8 * half);
  }
  // This lane's cell of the wave's tiles (none: -1) and its place in a row of y.
  long src[kPerWave];
  int dst[kPerWave];
#pragma unroll
  for (int p = 0; p < kPerWave; ++p) {
    const int f = (wave + p * (kTapThreads / 64)) * 32 + (lane & 31), col = f / nz, k = f % nz, j = j0 - 1 + col;
    const bool mine = f < (kScalarCols + 2) * nz && j >= 0 && j < ny;
    src[p] = mine ? (long)(j * nz + k) * 4 + half : -1;
    dst[p] = col * kTapColumn + k + 1;
  }
  u32x4 fetched[kPerWave][2];
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const u32x4* slab = reinterpret_cast<const u32x4*>(in) + (long)s * ny * nz * 4;
#pragma unroll
    for (int p = 0; p < kPerWave; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h) fetched[p][h] = slab[max(src[p], 0L) + 2 * h];
  };
  const int own_j = threadIdx.x / nz, own_k = threadIdx.x % nz;
  const bool owned = (int)threadIdx.x < kScalarCols * nz && j0 + own_j < ny;
  const int own = own_j * kTapColumn + own_k;
  float before = 0.0f, here = 0.0f;  // the sums of slabs s - 1 and s so far
  if (x0 > 0) fetch(x0 - 1);
  for (int s = x0 - 1; s <= x1; ++s) {
    float after = 0.0f;
    __syncthreads();  // the last slab's y has been read
    if (s >= 0 && s < nx) {
#pragma unroll
      for (int p = 0; p < kPerWave; ++p) {
        floatx16 d;
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h) d = mfma32(wr[h], __builtin_bit_cast(bf16x8, fetched[p][h]), d);
        if (src[p] >= 0)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int t = 8 * (r / 4) + 4 * half + r % 4;
            if (t < kTaps) y[t][dst[p]] = d[r];
          }
      }
    }
    if (s + 1 <= x1 && s + 1 < nx) fetch(s + 1);
    __syncthreads();
    if (owned && s >= 0 && s < nx) {
#pragma unroll
      for (int e = 0; e < 9; ++e) {
        const int o = own + e / 3 * kTapColumn + e % 3;
        after += y[e][o];
        here += y[9 + e][o];
        before += y[18 + e][o];
      }
    }
    if (owned && s > x0) out[((long)(s - 1) * ny + j0 + own_j) * nz + own_k] = before + bias[0];
    before = here;
    here = after;
  }
}
// Data gradient: out[x][ci] = sum over t of wb[t][ci][0] g[x + off(t)] where
// the activation is positive, else 0: one product of 32 channels x 32 cells
// with the taps as its reduction (two of depth 16), the gradient plane's
// values gathered from LDS.  Bound by the mask read and the gradient written;
// 40 us at 128x64x64 through the general form, 19 here.
__device__ __forceinline__ void channel_pieces(const floatx16& v, uint4 (&piece)[2]) {
  // Lane l holds channels 8 q + 4 (l / 32) + e of its cell in v[4 q + e]; on
  // return piece[0], piece[1] are its cell's 16-byte pieces 2 (l / 32) + {0, 1}.
  uint32_t p[4][2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[q][0] = pack2(v[4 * q], v[4 * q + 1]);
    p[q][1] = pack2(v[4 * q + 2], v[4 * q + 3]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const auto swapped = __builtin_amdgcn_permlane32_swap(p[q][d], p[q + 2][d], false, false);
      p[q][d] = swapped[0];
      p[q + 2][d] = swapped[1];
    }
    piece[q] = make_uint4(p[q][0], p[q][1], p[q + 2][0], p[q + 2][1]);
  }
}
constexpr int kSpreadThreads = 256, kSpreadSlab = (kScalarCols + 2) * kTapColumn;
template <int T>
__global__ void __launch_bounds__(kSpreadThreads)
    k_conv3d_spread(int nx, int ny, const uint16_t* __restrict__ g, const uint16_t* __restrict__ wb,
                    const uint16_t* __restrict__ mask, uint16_t* __restrict__ out) {
  constexpr int nz = 16 * T;
  __shared__ uint16_t gs[3 * kSpreadSlab];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, half = lane >> 5;
  const int tiles_j = (ny + kScalarCols - 1) / kScalarCols;
  const int j0 = (int)(blockIdx.x % tiles_j) * kScalarCols, i = (int)(blockIdx.x / tiles_j);
  for (int e = threadIdx.x; e < 3 * kSpreadSlab; e += kSpreadThreads) {
    const int s = i - 1 + e / kSpreadSlab, j = j0 - 1 + e % kSpreadSlab / kTapColumn, k = e % kTapColumn - 1;
    gs[e] = s >= 0 && s < nx && j >= 0 && j < ny && k >= 0 && k < nz ? g[((long)s * ny + j) * nz + k] : (uint16_t)0;
  }
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  bf16x8 wr[2];
  int at[2][8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    u16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = 16 * h + 8 * half + e;
      v[e] = t < kTaps ? wb[((long)t * kC + (lane & 31)) * kC] : (uint16_t)0;
      at[h][e] = t < kTaps ? t / 9 * kSpreadSlab + t / 3 % 3 * kTapColumn + t % 3 : -1;
    }
    wr[h] = __builtin_bit_cast(bf16x8, v);
  }
  __syncthreads();
  for (int tile = wave; tile * 32 < kScalarCols * nz; tile += kSpreadThreads / 64) {
    const int f = tile * 32 + (lane & 31), jl = f / nz, k = f % nz, j = j0 + jl;
    const uint16_t* cell_g = gs + jl * kTapColumn + k;
    floatx16 d;
#pragma unroll
    for (int r = 0; r < 16; ++r) d[r] = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u16x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = at[h][e] >= 0 ? cell_g[at[h][e]] : (uint16_t)0;
      d = mfma32(wr[h], __builtin_bit_cast(bf16x8, v), d);
    }
    uint4 piece[2];
    channel_pieces(d, piece);
    if (j >= ny) continue;
    const long at_c = (((long)i * ny + j) * nz + k) * kC + 16 * half;
    const uint4* positive = reinterpret_cast<const uint4*>(mask + at_c);
    uint4* line = reinterpret_cast<uint4*>(out + at_c);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint4 m = positive[q];
      line[q] = make_uint4(keep_positive(piece[q].x, m.x), keep_positive(piece[q].y, m.y),
                           keep_positive(piece[q].z, m.z), keep_positive(piece[q].w, m.w));
    }
  }
}

// ----------------------------------------------------------- weight grad
// dW[t][co][ci] = sum over cells of dout[x][co] in[x + off(t)][ci]: 27
// products with the cells as the reduction, so both operands need 8
// consecutive cells of one channel in a lane.  ds_read_b64_tr_b16 reads them
// so from channels-last rows: in a group of 16 lanes lane l points at row
// l / 4, channels 4 (l % 4), and gets 4 rows of channel l.  Nothing is
// transposed or shifted on the way into LDS.
//   - A block sweeps along x over two columns of y (one for each half of its
//     eight waves).  An input operand (slab s, shift dj, dk) is read once and
//     multiplied with the output gradient's rows s - 1, s and s + 1, whose
//     operands stay in registers from slab to slab: 13 KB read from LDS for
//     27 products of 32 cycles (v_mfma_f32_32x32x16_bf16), where one read a
//     product and operand would ask for twice what LDS delivers.
//   - A wave holds the sums of the 9 taps of three (dj, dk) pairs (144
//     registers).  Nine pairs over four waves: two each, and the ninth pair's
//     16-cell chunks spread over the waves.
//   - At the end the two halves add up through LDS, so 256 blocks write one
//     partial each (28 MB at 128x64x64, half of one a column group).  A block
//     takes several (columns, slabs) items where a grid has more than
//     kMaxGradBlocks of them, as wide ones do.
// A block that staged each column's nine neighbours transposed, element by
// element, took 109 us a layer at 128x64x64; 40 us now, and the fold of half as
// many partials 7 us instead of 12.
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4* lds_shortx4;
// 16 rows (cells) of 32 channels from `rows`, as the operand of one product:
// lane l gets channel l % 32 of rows 8 (l / 32) + 0..7.
__device__ __forceinline__ bf16x8 column_operand(const char* rows, int lane_offset) {
  typedef short shortx8 __attribute__((ext_vector_type(8)));
  char* at = const_cast<char*>(rows) + lane_offset;
  const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4)at);
  const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4)(at + 4 * kC * 2));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
constexpr int kGradThreads = 512, kGradCols = 2;
constexpr int kGradRow = kC * 2, kGradColumn = (kMaxColumn + 2) * kGradRow;  // bytes; one cell of halo at each end
constexpr int kGradBuffer = (kGradCols + 2 + kGradCols) * kGradColumn;       // input columns, then gradient columns
constexpr int kGradTaps = 24;  // taps of the eight pairs that one wave of each half holds alone
constexpr int kGradShared = kGradTaps * kC * kC * 4;
static_assert(2 * kGradBuffer <= kGradShared && 8 * 3 * kC * kC * 4 <= kGradShared, "shared buffer too small");

template <int T>
__global__ void __launch_bounds__(kGradThreads, 2)
    k_conv3d_wgrad(int nx, int ny, int per, int items, const uint16_t* __restrict__ in,
                   const uint16_t* __restrict__ dout, float* __restrict__ partials) {
  constexpr int nz = 16 * T;
  constexpr int kIn = (kGradCols + 2) * nz * 4, kOut = kGradCols * nz * 4;  // 16-byte pieces of a slab and of a row
  constexpr int kFetch = (kIn + kGradThreads - 1) / kGradThreads;
  static_assert(kOut <= kGradThreads, "one gradient piece a thread");
  __shared__ __attribute__((aligned(16))) char shared[kGradShared];
  __shared__ float bias_part[kGradThreads / 64][kC];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = wave >> 2, part = wave & 3;
  const int tiles_j = (ny + kGradCols - 1) / kGradCols;
  int j0, x0, x1;  // of the item in hand: its first column and its slabs
  // Staging: pieces as in the sweep (a thread without one reads the first
  // piece of the slab and stores none).
  long src[kFetch], out_src;
  int dst[kFetch], out_dst;
  auto begin = [&](int item) __attribute__((always_inline)) {
    j0 = item % tiles_j * kGradCols;
    x0 = item / tiles_j * per;
    x1 = min(nx, x0 + per);
    for (int e = tid; e < 2 * kGradBuffer / 16; e += kGradThreads)
      reinterpret_cast<u32x4*>(shared)[e] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int f = 0; f < kFetch; ++f) {
      const int e = tid + f * kGradThreads, col = e / (nz * 4), k = e / 4 % nz, c = e % 4, j = j0 - 1 + col;
      const bool mine = e < kIn && j >= 0 && j < ny;
      src[f] = mine ? (long)(j * nz + k) * 4 + c : 0;
      dst[f] = mine ? col * kGradColumn + (k + 1) * kGradRow + c * 16 : -1;
    }
    const int col = tid / (nz * 4), k = tid / 4 % nz, c = tid % 4, j = j0 + col;
    const bool mine = tid < kOut && j < ny;
    out_src = mine ? (long)(j * nz + k) * 4 + c : 0;
    out_dst = mine ? (kGradCols + 2 + col) * kGradColumn + (k + 1) * kGradRow + c * 16 : -1;
  };
  u32x4 fetched[kFetch], fetched_out;
  // Slab s of the input and row s + 1 of the output gradient.
  auto fetch = [&](int s) __attribute__((always_inline)) {
    if (s >= 0 && s < nx) {
      const u32x4* slab = reinterpret_cast<const u32x4*>(in) + (long)s * ny * nz * 4;
#pragma unroll
      for (int f = 0; f < kFetch; ++f) fetched[f] = slab[src[f]];
    }
    if (s + 1 < x1) fetched_out = (reinterpret_cast<const u32x4*>(dout) + (long)(s + 1) * ny * nz * 4)[out_src];
  };
  float bias_acc[8] = {};
  auto stage = [&](int s, char* buffer) __attribute__((always_inline)) {
    if (s >= 0 && s < nx) {
#pragma unroll
      for (int f = 0; f < kFetch; ++f)
        if (dst[f] >= 0) *reinterpret_cast<u32x4*>(buffer + dst[f]) = fetched[f];
    }
    if (s + 1 < x1 && out_dst >= 0) {
      *reinterpret_cast<u32x4*>(buffer + out_dst) = fetched_out;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bias_acc[2 * e] += __uint_as_float(fetched_out[e] << 16);
        bias_acc[2 * e + 1] += __uint_as_float(fetched_out[e] & 0xffff0000u);
      }
    }
  };
  const int lane_offset = (8 * (lane >> 5) + ((lane & 15) >> 2)) * kGradRow + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int out_column = (kGradCols + 2 + half) * kGradColumn + kGradRow;
  int pair_at[3], pair[3] = {2 * part, 2 * part + 1, 8};
#pragma unroll
  for (int q = 0; q < 3; ++q) pair_at[q] = (half + pair[q] / 3) * kGradColumn + pair[q] % 3 * kGradRow;
  floatx16 acc[3][3];  // [pair][di]
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[q][d][r] = 0.0f;
  int current = 0;
  bf16x8 rows[3][T];
  // Input slab s with the gradient's rows s - 1 (A), s (B) and s + 1 (C, read here).
  auto step = [&](int s, bf16x8(&A)[T], bf16x8(&B)[T], bf16x8(&C)[T]) __attribute__((always_inline)) {
    __syncthreads();
    const char* buffer = shared + current * kGradBuffer;
    if (s < x1) fetch(s + 1);
    const bool has_a = s - 1 >= x0 && s <= x1, has_b = s >= x0 && s < x1, has_c = s + 1 < x1;
    if (has_c) {
#pragma unroll
      for (int c = 0; c < T; ++c) C[c] = column_operand(buffer + out_column + c * 16 * kGradRow, lane_offset);
    }
    if (s >= 0 && s < nx && s <= x1) {
#pragma unroll
      for (int c = 0; c < T; ++c)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          if (q == 2 && c != part) continue;
          const bf16x8 x = column_operand(buffer + pair_at[q] + c * 16 * kGradRow, lane_offset);
          if (has_c) acc[q][0] = mfma32(C[c], x, acc[q][0]);
          if (has_b) acc[q][1] = mfma32(B[c], x, acc[q][1]);
          if (has_a) acc[q][2] = mfma32(A[c], x, acc[q][2]);
        }
    }
    current ^= 1;
    if (s < x1) stage(s + 1, shared + current * kGradBuffer);
  };
  for (int item = (int)blockIdx.x; item < items; item += (int)gridDim.x) {
    if (item != (int)blockIdx.x) __syncthreads();  // the last item's slabs have been read
    begin(item);
    __syncthreads();
    fetch(x0 - 1);
    stage(x0 - 1, shared);
    current = 0;
    for (int s = x0 - 1; s <= x1; s += 3) {  // beyond x1 a step does nothing
      step(s, rows[0], rows[1], rows[2]);
      step(s + 1, rows[1], rows[2], rows[0]);
      step(s + 2, rows[2], rows[0], rows[1]);
    }
  }
  float* result = partials + (long)blockIdx.x * kLayer;
  float* red = reinterpret_cast<float*>(shared);
  // Lane l's sums: input channel l % 32, output channels 8 (r / 4) + 4 (l / 32) + r % 4.
  auto element = [&](int r) { return (8 * (r / 4) + 4 * (lane >> 5) + r % 4) * kC + (lane & 31); };
  __syncthreads();
  if (half == 1)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[(d * 8 + pair[q]) * kC * kC + element(r)] = acc[q][d][r];
  __syncthreads();
  if (half == 0)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          result[(d * 9 + pair[q]) * kC * kC + element(r)] =
              acc[q][d][r] + red[(d * 8 + pair[q]) * kC * kC + element(r)];
  __syncthreads();
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[(wave * 3 + d) * kC * kC + element(r)] = acc[2][d][r];
  // Bias: lanes of equal l % 4 hold the same 8 channels.
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    for (int off = 4; off < 64; off <<= 1) bias_acc[e] += __shfl_xor(bias_acc[e], off);
    if (lane < 4) bias_part[wave][lane * 8 + e] = bias_acc[e];
  }
  __syncthreads();
  for (int e = tid; e < 3 * kC * kC; e += kGradThreads) {
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < 8; ++v) sum += red[v * 3 * kC * kC + e];
    result[(e / (kC * kC) * 9 + 8) * kC * kC + e % (kC * kC)] = sum;
  }
  if (tid < kC) {
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < 8; ++v) sum += bias_part[v][tid];
    result[kWeights + tid] = sum;
  }
}

// The scalar layer's weight gradient: dW[t][0][ci] = sum over x of
// g[x - off(t)] in[x][ci], one product of 32 taps x 32 channels for 16 cells
// (the taps' shifts are in the gathered gradient values, so the input is read
// without a halo).  Bound by reading the input; 40 us at 128x64x64 through the
// general form, 10 here.  A partial row: 27 x 32 sums, then the bias.
constexpr int kScalarGradCols = 4, kScalarGradRow = kTaps * kC + 8, kScalarGradSlab = (kScalarGradCols + 2) * kTapColumn;
template <int T>
__global__ void __launch_bounds__(kGradThreads)
    k_scalar_wgrad(int nx, int ny, int per, int items, const uint16_t* __restrict__ in,
                   const uint16_t* __restrict__ g, float* __restrict__ partials) {
  constexpr int nz = 16 * T, kPieces = kScalarGradCols * nz * 4, kFetch = (kPieces + kGradThreads - 1) / kGradThreads;
  __shared__ __attribute__((aligned(16))) char xs[2][kScalarGradCols * kMaxColumn * kGradRow];
  __shared__ uint16_t gs[2][3 * kScalarGradSlab];
  __shared__ float red[kGradThreads / 64][kC * kC];
  __shared__ float bias_part[kGradThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
  const int tiles_j = (ny + kScalarGradCols - 1) / kScalarGradCols;
  int j0, x0, x1;  // of the item in hand: its first column and its slabs
  u32x4 fetched[kFetch];
  bool mine[kFetch];
  long src[kFetch];
  auto begin = [&](int item) __attribute__((always_inline)) {
    j0 = item % tiles_j * kScalarGradCols;
    x0 = item / tiles_j * per;
    x1 = min(nx, x0 + per);
#pragma unroll
    for (int f = 0; f < kFetch; ++f) {
      const int e = tid + f * kGradThreads, col = e / (nz * 4), j = j0 + col;
      mine[f] = e < kPieces && j < ny;
      src[f] = mine[f] ? (long)j * nz * 4 + e % (nz * 4) : 0;
    }
  };
  float bias_acc = 0.0f;
  constexpr int kGather = (3 * kScalarGradSlab + kGradThreads - 1) / kGradThreads;
  uint16_t gathered[kGather];
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const u32x4* slab = reinterpret_cast<const u32x4*>(in) + (long)s * ny * nz * 4;
#pragma unroll
    for (int f = 0; f < kFetch; ++f) fetched[f] = slab[src[f]];
#pragma unroll
    for (int f = 0; f < kGather; ++f) {
      const int e = tid + f * kGradThreads;
      const int i = s - 1 + e / kScalarGradSlab, j = j0 - 1 + e % kScalarGradSlab / kTapColumn, k = e % kTapColumn - 1;
      const bool real = e < 3 * kScalarGradSlab && i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz;
      gathered[f] = real ? g[((long)i * ny + j) * nz + k] : (uint16_t)0;
    }
  };
  auto stage = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < kFetch; ++f) {
      const int e = tid + f * kGradThreads;
      if (e < kPieces)
        *reinterpret_cast<u32x4*>(xs[buffer] + (e / (nz * 4) * kMaxColumn * 4 + e % (nz * 4)) * 16) =
            mine[f] ? fetched[f] : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int f = 0; f < kGather; ++f) {
      const int e = tid + f * kGradThreads;
      if (e < 3 * kScalarGradSlab) gs[buffer][e] = gathered[f];
      // the slab's own gradient, each cell by the block that owns it
      const int col = e % kScalarGradSlab / kTapColumn;
      if (e / kScalarGradSlab == 1 && col >= 1 && col <= kScalarGradCols) bias_acc += bf2f(gathered[f]);
    }
  };
  const int t = lane & 31;
  const bool tap = t < kTaps;
  const int tap_at = tap ? (2 - t / 9) * kScalarGradSlab + (2 - t / 3 % 3) * kTapColumn + 2 - t % 3 + 8 * half : 0;
  const int lane_offset = (8 * half + ((lane & 15) >> 2)) * kGradRow + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  for (int item = (int)blockIdx.x; item < items; item += (int)gridDim.x) {
    if (item != (int)blockIdx.x) __syncthreads();  // the last item's slabs have been read
    begin(item);
    fetch(x0);
    stage(0);
    for (int s = x0; s < x1; ++s) {
      const int buffer = (s - x0) & 1;
      __syncthreads();
      if (s + 1 < x1) fetch(s + 1);
      for (int unit = wave; unit < kScalarGradCols * T; unit += kGradThreads / 64) {
        const int col = unit / T, k0 = unit % T * 16;
        typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
        u16x8 v;
        const uint16_t* cell_g = gs[buffer] + col * kTapColumn + k0 + tap_at;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tap ? cell_g[e] : (uint16_t)0;
        const bf16x8 x = column_operand(xs[buffer] + (col * kMaxColumn + k0) * kGradRow, lane_offset);
        acc = mfma32(__builtin_bit_cast(bf16x8, v), x, acc);
      }
      if (s + 1 < x1) stage(buffer ^ 1);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) red[wave][(8 * (r / 4) + 4 * half + r % 4) * kC + t] = acc[r];
  for (int off = 1; off < 64; off <<= 1) bias_acc += __shfl_xor(bias_acc, off);
  if (lane == 0) bias_part[wave] = bias_acc;
  __syncthreads();
  float* result = partials + (long)blockIdx.x * kScalarGradRow;
  for (int e = tid; e < kTaps * kC; e += kGradThreads) {
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < kGradThreads / 64; ++v) sum += red[v][e];
    result[e] = sum;
  }
  if (tid == 0) {
    float sum = 0.0f;
    for (int v = 0; v < kGradThreads / 64; ++v) sum += bias_part[v];
    result[kTaps * kC] = sum;
  }
}
// The layer's gradient from the partial rows, in block order; zero for the
// output channels that the layer does not have.  64 loads in flight: a row is
// a serial step of the sum.
__global__ void __launch_bounds__(64) k_fold_scalar(const float* __restrict__ partials, int blocks,
                                                    float* __restrict__ grad) {
  const int p = blockIdx.x * 64 + threadIdx.x;
  if (p >= kLayer) return;
  const int channel = p < kWeights ? p / kC % kC : p - kWeights;
  const int at = p < kWeights ? p / (kC * kC) * kC + p % kC : kTaps * kC;
  float s = 0.0f;
  if (channel == 0) {
    int b = 0;
    for (; b + 64 <= blocks; b += 64) {
      float v[64];
#pragma unroll
      for (int e = 0; e < 64; ++e) v[e] = partials[(long)(b + e) * kScalarGradRow + at];
#pragma unroll
      for (int e = 0; e < 64; ++e) s += v[e];
    }
    for (; b < blocks; ++b) s += partials[(long)b * kScalarGradRow + at];
  }
  grad[p] = s;
}

// grad[p] = sum over blocks of partials[b][p], in block order.  Bound by
// reading the partials (28 MB for 256 blocks): one thread a parameter, the
// adds in order, but kFoldBatch loads in flight and 64-thread blocks so that
// every CU has some.  One load at a time in 256-thread blocks left 108 blocks
// waiting on memory: 144 us for 512 rows at 128x64x64, 12 us this way.
constexpr int kFoldThreads = 64, kFoldBatch = 32;
__global__ void __launch_bounds__(kFoldThreads)
    k_fold(const float* __restrict__ partials, int blocks, int count, float* __restrict__ out) {
  const int p = blockIdx.x * kFoldThreads + threadIdx.x;
  if (p >= count) return;
  float s = 0.0f;
  int b = 0;
  for (; b + kFoldBatch <= blocks; b += kFoldBatch) {
    float v[kFoldBatch];
#pragma unroll
    for (int e = 0; e < kFoldBatch; ++e) v[e] = partials[(long)(b + e) * count + p];
#pragma unroll
    for (int e = 0; e < kFoldBatch; ++e) s += v[e];
  }
  for (; b < blocks; ++b) s += partials[(long)b * count + p];
  out[p] = s;
}

// ------------------------------------------------------------------ loss
constexpr int kLossThreads = 256;
// Plane: dout is one value a cell; otherwise channel 0 of 32, the rest zero.
template <bool Plane>
__global__ void __launch_bounds__(kLossThreads)
    k_weighted_mse(long cells, const float* __restrict__ pred, const float* __restrict__ target,
                   const float* __restrict__ weight, uint16_t* __restrict__ dout, float* __restrict__ partials) {
  __shared__ float part[kLossThreads / 64];
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  float loss = 0.0f;
  if (n < cells) {
    const float d = pred[n] - target[n], w = weight[n];
    loss = w * d * d;
    const uint16_t g = f2bf(2.0f * w * d);
    if (Plane) {
      dout[n] = g;
    } else {
      uint4* o = reinterpret_cast<uint4*>(dout + n * kC);
      o[0] = make_uint4(g, 0u, 0u, 0u);
      o[1] = o[2] = o[3] = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = loss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.0f;
    for (int w = 0; w < kLossThreads / 64; ++w) s += part[w];
    partials[blockIdx.x] = s;
  }
}
// The loss from the block sums: one block, strided shares, then a fixed tree
// (a single thread over the 2048 sums of 128x64x64 took 30 us).
constexpr int kLossFoldThreads = 512;
__global__ void __launch_bounds__(kLossFoldThreads)
    k_fold_loss(const float* __restrict__ partials, int blocks, float* __restrict__ loss) {
  __shared__ float part[kLossFoldThreads];
  float s = 0.0f;
  for (int b = threadIdx.x; b < blocks; b += kLossFoldThreads) s += partials[b];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int width = kLossFoldThreads / 2; width > 0; width >>= 1) {
    if ((int)threadIdx.x < width) part[threadIdx.x] += part[threadIdx.x + width];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = part[0];
}

// ------------------------------------------------------------------ Adam
__device__ __forceinline__ void store_weight(int layer, int p, float value, uint16_t* wf, uint16_t* wb) {
  if (p >= kWeights) return;
  const int t = p / (kC * kC), co = (p / kC) % kC, ci = p % kC;
  const uint16_t b = f2bf(value);
  wf[(long)layer * kWeights + p] = b;
  wb[(long)layer * kWeights + ((kTaps - 1 - t) * kC + ci) * kC + co] = b;
}
__global__ void k_adam(int layers, float* __restrict__ master, float* __restrict__ m, float* __restrict__ v,
                       const float* __restrict__ grad, float lr, float beta1, float beta2, float eps, float c1,
                       float c2, uint16_t* __restrict__ wf, uint16_t* __restrict__ wb) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long)layers * kLayer) return;
  const float g = grad[q];
  const float mq = beta1 * m[q] + (1.0f - beta1) * g;
  const float vq = beta2 * v[q] + (1.0f - beta2) * g * g;
  m[q] = mq;
  v[q] = vq;
  const float w = master[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
  master[q] = w;
  store_weight((int)(q / kLayer), (int)(q % kLayer), w, wf, wb);
}
__global__ void k_pack(int layers, const float* __restrict__ master, uint16_t* __restrict__ wf,
                       uint16_t* __restrict__ wb) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long)layers * kLayer) return;
  store_weight((int)(q / kLayer), (int)(q % kLayer), master[q], wf, wb);
}

// ------------------------------------------------- solver state interface
__device__ __forceinline__ bool touches_ice(int nx, int ny, int nz, int i, int j, int k, const float* coverage,
                                            const int8_t* cov_id) {
  const int offs[7][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}, {0, 0, 0}};
#pragma unroll
  for (int f = 0; f < 7; ++f) {
    const int a = i + offs[f][0], b = j + offs[f][1], c = k + offs[f][2];
    if (a < 0 || a >= nx || b < 0 || b >= ny || c < 0 || c >= nz) continue;
    const long m = ((long)a * ny + b) * nz + c;
    if (cov_id[m] >= 0 && coverage[m] > 1e-8f) return true;
  }
  return false;
}
__global__ void k_features(int nx, int ny, int nz, const float* __restrict__ phi, const float* __restrict__ volume,
                           const float* __restrict__ energy, const float* __restrict__ u,
                           const float* __restrict__ coverage, const int8_t* __restrict__ cov_id, float cell_volume,
                           float rho_cp, float tm, uint16_t* __restrict__ features) {
  const long N = (long)nx * ny * nz;
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int k = (int)(n % nz), j = (int)((n / nz) % ny), i = (int)(n / ((long)nz * ny));
  const float v = volume[n];
  const bool wet = v > 1e-30f * cell_volume;
  const float temperature = wet ? tm + energy[n] / (rho_cp * v) : 0.0f;
  float f[8] = {phi[n], 0.01f * temperature, 10.0f * u[n], 10.0f * u[N + n], 10.0f * u[2 * N + n],
                cov_id[n] >= 0 ? coverage[n] : 0.0f, wet ? 1.0f : 0.0f,
                touches_ice(nx, ny, nz, i, j, k, coverage, cov_id) ? 1.0f : 0.0f};
  uint32_t packed[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) packed[e] = (uint32_t)f2bf(f[2 * e]) | ((uint32_t)f2bf(f[2 * e + 1]) << 16);
  uint4* o = reinterpret_cast<uint4*>(features + n * kC);
  o[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
  o[1] = o[2] = o[3] = make_uint4(0u, 0u, 0u, 0u);
}
__global__ void k_gain(int nx, int ny, int nz, const float* __restrict__ pred, const float* __restrict__ coverage,
                       const int8_t* __restrict__ cov_id, float max_gain, float* __restrict__ gain) {
  const long N = (long)nx * ny * nz;
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int k = (int)(n % nz), j = (int)((n / nz) % ny), i = (int)(n / ((long)nz * ny));
  float g = 1.0f;
  if (touches_ice(nx, ny, nz, i, j, k, coverage, cov_id)) g = fminf(max_gain, fmaxf(0.0f, 1.0f + pred[n]));
  gain[n] = g;
}

int status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}
bool valid_grid(int nx, int ny, int nz) { return nx > 0 && ny > 0 && nz > 0 && (long)nx * ny * nz < (1L << 31); }
unsigned blocks_of(long count, int threads) { return (unsigned)((count + threads - 1) / threads); }
// Slabs a sweep block owns: as many as leave one block for each of the 256
// CUs (a block fills a CU: its waves hold 512 registers), at least one.
int sweep_slabs(int nx, int tiles_j) {
  const int chunks = tiles_j >= 256 ? 1 : 256 / tiles_j;
  return (nx + chunks - 1) / chunks;
}
template <int Epi>
void launch_sweep(int nx, int ny, int nz, const uint16_t* in, const uint16_t* w, const float* bias,
                  const uint16_t* mask, uint16_t* out, hipStream_t s) {
  const int tiles_j = (ny + kSweepCols - 1) / kSweepCols, per = sweep_slabs(nx, tiles_j);
  const unsigned blocks = (unsigned)(tiles_j * ((nx + per - 1) / per));
  auto kernel = nz == 16   ? k_conv3d_sweep<Epi, 1>
                : nz == 32 ? k_conv3d_sweep<Epi, 2>
                : nz == 48 ? k_conv3d_sweep<Epi, 3>
                           : k_conv3d_sweep<Epi, 4>;
  kernel<<<blocks, kSweepThreads, 0, s>>>(nx, ny, per, in, w, bias, mask, out);
}
void launch_taps(int nx, int ny, int nz, const uint16_t* in, const uint16_t* w, const float* bias, float* out,
                 hipStream_t s) {
  const int tiles_j = (ny + kScalarCols - 1) / kScalarCols, per = sweep_slabs(nx, tiles_j);
  const unsigned blocks = (unsigned)(tiles_j * ((nx + per - 1) / per));
  auto kernel = nz == 16 ? k_conv3d_taps<1> : nz == 32 ? k_conv3d_taps<2> : nz == 48 ? k_conv3d_taps<3> : k_conv3d_taps<4>;
  kernel<<<blocks, kTapThreads, 0, s>>>(nx, ny, per, in, w, bias, out);
}
// Weight-gradient items: groups of `cols` columns times chunks of slabs, one
// for each of the 256 CUs where the grid has as many, but four slabs a chunk at
// least: a chunk reads two slabs more than it owns, and each block writes 110
// KB of sums that the fold reads again.  With at least 1, 2, 4 and 8 slabs the
// gradient and its fold take 27, 20, 20 and 22 us at 24x17x16, 28, 22, 24 and
// 28 at 24x17x64, 28, 28, 27 and 30 at 40x33x48 and 12, 15, 14 and 15 at
// 8x8x16 (the scalar layer's 18, 18, 13 and 11, 19, 19, 14 and 14, 20, 20, 14
// and 21, 8, 7, 7 and 8); larger grids have four slabs or more by themselves.
// At most kMaxGradBlocks blocks share the items: the 32768 of 1x65536x16, a
// block each, would leave 3.6 GB of sums and take 1961 us; 251 this way.
constexpr int kMaxGradBlocks = 512;
struct GradPlan {
  int per, items, blocks;
};
GradPlan wgrad_plan(int nx, int ny, int cols) {
  const int tiles_j = (ny + cols - 1) / cols, slabs = sweep_slabs(nx, tiles_j), per = slabs < 4 ? 4 : slabs;
  const int items = tiles_j * ((nx + per - 1) / per);
  return {per, items, items < kMaxGradBlocks ? items : kMaxGradBlocks};
}

}  // namespace icyc

using namespace icyc;

extern "C" {

int icyc_conv3d(int32_t nx, int32_t ny, int32_t nz, const uint16_t* in, const uint16_t* weights, const float* bias,
                int32_t epilogue, const uint16_t* mask_act, uint16_t* out_bf16, float* out_f32, void* stream) {
  if (!valid_grid(nx, ny, nz) || !in || !weights) return ICYC_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  if (nz % 16 == 0 && nz <= kMaxColumn) {
    switch (epilogue) {
      case ICYC_RELU_BF16:
        if (!bias || !out_bf16) return ICYC_ERR_ARGUMENT;
        launch_sweep<ICYC_RELU_BF16>(nx, ny, nz, in, weights, bias, nullptr, out_bf16, s);
        break;
      case ICYC_LINEAR_F32:
        if (!bias || !out_f32) return ICYC_ERR_ARGUMENT;
        launch_taps(nx, ny, nz, in, weights, bias, out_f32, s);
        break;
      case ICYC_MASKED_BF16:
        if (!mask_act || !out_bf16) return ICYC_ERR_ARGUMENT;
        launch_sweep<ICYC_MASKED_BF16>(nx, ny, nz, in, weights, nullptr, mask_act, out_bf16, s);
        break;
      default:
        return ICYC_ERR_ARGUMENT;
    }
    return status();
  }
  const unsigned blocks = blocks_of((long)nx * ny * nz, kCellsPerBlock);
  switch (epilogue) {
    case ICYC_RELU_BF16:
      if (!bias || !out_bf16) return ICYC_ERR_ARGUMENT;
      k_conv3d<ICYC_RELU_BF16><<<blocks, kConvThreads, 0, s>>>(nx, ny, nz, in, weights, bias, nullptr, out_bf16,
                                                              nullptr);
      break;
    case ICYC_LINEAR_F32:
      if (!bias || !out_f32) return ICYC_ERR_ARGUMENT;
      k_conv3d<ICYC_LINEAR_F32><<<blocks, kConvThreads, 0, s>>>(nx, ny, nz, in, weights, bias, nullptr, nullptr,
                                                               out_f32);
      break;
    case ICYC_MASKED_BF16:
      if (!mask_act || !out_bf16) return ICYC_ERR_ARGUMENT;
      k_conv3d<ICYC_MASKED_BF16><<<blocks, kConvThreads, 0, s>>>(nx, ny, nz, in, weights, nullptr, mask_act,
                                                                out_bf16, nullptr);
      break;
    default:
      return ICYC_ERR_ARGUMENT;
  }
  return status();
}

int icyc_conv3d_k8(int32_t nx, int32_t ny, int32_t nz, const uint16_t* in, const uint16_t* weights,
                   const float* bias, int32_t epilogue, uint16_t* out_bf16, float* out_f32, void* stream) {
  if (!valid_grid(nx, ny, nz) || !in || !weights || !bias || nz % 16 != 0 || nz > kMaxColumn)
    return ICYC_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const int tiles_j = (ny + kSweepCols - 1) / kSweepCols, per = sweep_slabs(nx, tiles_j);
  const unsigned blocks = (unsigned)(tiles_j * ((nx + per - 1) / per));
  if (epilogue == ICYC_RELU_BF16 && out_bf16) {
    auto kernel = nz == 16   ? k_conv3d_first<ICYC_RELU_BF16, 1>
                  : nz == 32 ? k_conv3d_first<ICYC_RELU_BF16, 2>
                  : nz == 48 ? k_conv3d_first<ICYC_RELU_BF16, 3>
                             : k_conv3d_first<ICYC_RELU_BF16, 4>;
    kernel<<<blocks, kSweepThreads, 0, s>>>(nx, ny, per, in, weights, bias, out_bf16, nullptr);
  } else if (epilogue == ICYC_LINEAR_F32 && out_f32) {
    auto kernel = nz == 16   ? k_conv3d_first<ICYC_LINEAR_F32, 1>
                  : nz == 32 ? k_conv3d_first<ICYC_LINEAR_F32, 2>
                  : nz == 48 ? k_conv3d_first<ICYC_LINEAR_F32, 3>
                             : k_conv3d_first<ICYC_LINEAR_F32, 4>;
    kernel<<<blocks, kSweepThreads, 0, s>>>(nx, ny, per, in, weights, bias, nullptr, out_f32);
  } else {
    return ICYC_ERR_ARGUMENT;
  }
  return status();
}

int64_t icyc_wgrad_partials_size(int32_t nx, int32_t ny, int32_t nz) {
  if (!valid_grid(nx, ny, nz)) return 0;
  return (int64_t)wgrad_plan(nx, ny, kGradCols).blocks * kLayer;
}

int icyc_conv3d_wgrad(int32_t nx, int32_t ny, int32_t nz, const uint16_t* in, const uint16_t* dout,
                      float* partials, float* grad, void* stream) {
  if (!valid_grid(nx, ny, nz) || nz % 16 != 0 || nz > kMaxColumn || !in || !dout || !partials || !grad)
    return ICYC_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const GradPlan plan = wgrad_plan(nx, ny, kGradCols);
  auto kernel = nz == 16   ? k_conv3d_wgrad<1>
                : nz == 32 ? k_conv3d_wgrad<2>
                : nz == 48 ? k_conv3d_wgrad<3>
                           : k_conv3d_wgrad<4>;
  kernel<<<plan.blocks, kGradThreads, 0, s>>>(nx, ny, plan.per, plan.items, in, dout, partials);
  if (int rc = status()) return rc;
  k_fold<<<blocks_of(kLayer, kFoldThreads), kFoldThreads, 0, s>>>(partials, plan.blocks, kLayer, grad);
  return status();
}

int icyc_conv3d_scalar_data(int32_t nx, int32_t ny, int32_t nz, const uint16_t* dout, const uint16_t* weights,
                            const uint16_t* mask_act, uint16_t* out_bf16, void* stream) {
  if (!valid_grid(nx, ny, nz) || nz % 16 != 0 || nz > kMaxColumn || !dout || !weights || !mask_act || !out_bf16)
    return ICYC_ERR_ARGUMENT;
  const unsigned blocks = (unsigned)(nx * ((ny + kScalarCols - 1) / kScalarCols));
  auto kernel = nz == 16   ? k_conv3d_spread<1>
                : nz == 32 ? k_conv3d_spread<2>
                : nz == 48 ? k_conv3d_spread<3>
                           : k_conv3d_spread<4>;
  kernel<<<blocks, kSpreadThreads, 0, (hipStream_t)stream>>>(nx, ny, dout, weights, mask_act, out_bf16);
  return status();
}

int icyc_conv3d_scalar_wgrad(int32_t nx, int32_t ny, int32_t nz, const uint16_t* in, const uint16_t* dout,
                             float* partials, float* grad, void* stream) {
  if (!valid_grid(nx, ny, nz) || nz % 16 != 0 || nz > kMaxColumn || !in || !dout || !partials || !grad)
    return ICYC_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const GradPlan plan = wgrad_plan(nx, ny, kScalarGradCols);
  auto kernel = nz == 16   ? k_scalar_wgrad<1>
                : nz == 32 ? k_scalar_wgrad<2>
                : nz == 48 ? k_scalar_wgrad<3>
                           : k_scalar_wgrad<4>;
  kernel<<<plan.blocks, kGradThreads, 0, s>>>(nx, ny, plan.per, plan.items, in, dout, partials);
  if (int rc = status()) return rc;
  k_fold_scalar<<<blocks_of(kLayer, 64), 64, 0, s>>>(partials, plan.blocks, grad);
  return status();
}

int64_t icyc_loss_partials_size(int64_t cells) { return cells > 0 ? (int64_t)blocks_of(cells, kLossThreads) : 0; }

static int weighted_mse(bool plane, int64_t cells, const float* pred, const float* target, const float* weight,
                        uint16_t* dout, float* partials, float* loss, void* stream) {
  if (cells <= 0 || !pred || !target || !weight || !dout || !partials || !loss) return ICYC_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = blocks_of(cells, kLossThreads);
  auto kernel = plane ? k_weighted_mse<true> : k_weighted_mse<false>;
  kernel<<<blocks, kLossThreads, 0, s>>>(cells, pred, target, weight, dout, partials);
  if (int rc = status()) return rc;
  k_fold_loss<<<1, kLossFoldThreads, 0, s>>>(partials, (int)blocks, loss);
  return status();
}
int icyc_weighted_mse(int64_t cells, const float* pred, const float* target, const float* weight, uint16_t* dout,
                      float* partials, float* loss, void* stream) {
  return weighted_mse(false, cells, pred, target, weight, dout, partials, loss, stream);
}
int icyc_weighted_mse_plane(int64_t cells, const float* pred, const float* target, const float* weight,
                            uint16_t* dout, float* partials, float* loss, void* stream) {
  return weighted_mse(true, cells, pred, target, weight, dout, partials, loss, stream);
}

int icyc_adam(int32_t layers, float* master, float* m, float* v, const float* grad, float lr, float beta1,
              float beta2, float eps, int32_t step, uint16_t* wf, uint16_t* wb, void* stream) {
  if (layers <= 0 || step <= 0 || !master || !m || !v || !grad || !wf || !wb) return ICYC_ERR_ARGUMENT;
  const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
  k_adam<<<blocks_of((long)layers * kLayer, 256), 256, 0, (hipStream_t)stream>>>(layers, master, m, v, grad, lr, beta1,
                                                                                beta2, eps, c1, c2, wf, wb);
  return status();
}

int icyc_pack_weights(int32_t layers, const float* master, uint16_t* wf, uint16_t* wb, void* stream) {
  if (layers <= 0 || !master || !wf || !wb) return ICYC_ERR_ARGUMENT;
  k_pack<<<blocks_of((long)layers * kLayer, 256), 256, 0, (hipStream_t)stream>>>(layers, master, wf, wb);
  return status();
}

int icyc_features(int32_t nx, int32_t ny, int32_t nz, const float* phi, const float* water_volume,
                  const float* water_energy, const float* u, const float* coverage, const int8_t* cov_id,
                  float cell_volume, float rho_cp, float tm, uint16_t* features, void* stream) {
  if (!valid_grid(nx, ny, nz) || !phi || !water_volume || !water_energy || !u || !coverage || !cov_id || !features)
    return ICYC_ERR_ARGUMENT;
  k_features<<<blocks_of((long)nx * ny * nz, 256), 256, 0, (hipStream_t)stream>>>(
      nx, ny, nz, phi, water_volume, water_energy, u, coverage, cov_id, cell_volume, rho_cp, tm, features);
  return status();
}

int icyc_gain(int32_t nx, int32_t ny, int32_t nz, const float* pred, const float* coverage, const int8_t* cov_id,
              float max_gain, float* gain, void* stream) {
  if (!valid_grid(nx, ny, nz) || !pred || !coverage || !cov_id || !gain) return ICYC_ERR_ARGUMENT;
  k_gain<<<blocks_of((long)nx * ny * nz, 256), 256, 0, (hipStream_t)stream>>>(nx, ny, nz, pred, coverage, cov_id,
                                                                             max_gain, gain);
  return status();
}

}  // extern "C"

#ifndef ICY_SOURCE_HASH
#define ICY_SOURCE_HASH "unrecorded"
#endif
extern "C" const char* icyc_source_hash(void) { return ICY_SOURCE_HASH; }
