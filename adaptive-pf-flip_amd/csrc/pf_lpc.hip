// pf_lpc.hip -- the learned preconditioner's network: a 3-layer 3x3x3 convolutional
// network over 16^3 tiles with a 1-cell input halo, run on MFMA in BF16 with FP32
// accumulation, and its hand-written backward pass for training on the GPU.
// (No reference counterpart: the reference preconditions with Jacobi only,
// src/driver/sparse_ops3d_tp.cpp:322-327.)  pf_lpc_cw.hip feeds it the features of
// the multigrid cycle's aggregates and turns its output into correction weights.
//
// Network (weights W*[tap][ci][co], tap = dx + 3 dy + 9 dz, no biases):
//   X[18^3][4]                     four input channels (pf_lpc_cw.hip)
//   h1 = relu(conv(X, W1))        4 -> 16  (X carries the halo)
//   h2 = relu(conv(pad0 h1, W2)) 16 -> 32  (zero padding at the tile boundary)
//   h3 = relu(conv(pad0 h2, W3)) 32 -> 16
//   o  = h3 . Wh                  16 -> 1
// Activations are stored in BF16, channels last: [tile][cell][channel] with
// cell = x + 16 (y + 16 z); the input X is [tile][18^3][4] with the halo.
//
// Convolution as an implicit GEMM on v_mfma_f32_16x16x32_bf16: one MFMA row block is
// 16 cells along x (M), the K dimension is (tap, ci) in tap-major order, N is 16
// output channels.  Lane l of a wavefront supplies A[m = l % 16][k = 8 (l / 16) + i]
// and B[k = 8 (l / 16) + i][n = l % 16], i = 0..7, and receives
// D[m = 4 (l / 16) + i][n = l % 16], i = 0..3.  A workgroup (4 waves) computes a
// z-plane of one tile, a wave kConvRows rows of 16 cells.  The layer's weights sit in
// LDS as WT[n][k] (k contiguous); the A fragments come straight from global memory:
// for CIN >= 8 each lane loads 8 consecutive channels of one tap (16 bytes), and the
// 16 lanes of a group read 16 neighbouring cells.
//
// The backward pass through a convolution is the same kernel on the zero-padded
// output gradient with the weights tap-flipped and transposed
// (W'[26 - tap][co][ci] = W[tap][ci][co]), followed by the ReLU mask of the
// layer below.  Weight gradients (a reduction over all cells) run on the matrix cores
// from LDS-staged planes, with per-workgroup partial sums reduced in a fixed order, so
// training is deterministic.
#include "pf_internal.h"

namespace pf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 16, kHalo = 18, kTileVol = 4096, kHaloVol = 5832;
constexpr int kC0 = 4;
constexpr int kNW1 = 27 * 4 * 16, kNW2 = 27 * 16 * 32, kNW3 = 27 * 32 * 16, kNWH = 16;
constexpr int kNW = kNW1 + kNW2 + kNW3 + kNWH;   // 29,392 weights
constexpr int kOffW1 = 0, kOffW2 = kNW1, kOffW3 = kNW1 + kNW2, kOffWH = kNW1 + kNW2 + kNW3;

__host__ __device__ constexpr int kpad(int cin) { return ((27 * cin + 31) / 32) * 32; }

enum { EPI_RELU = 0, EPI_HEAD = 1, EPI_MASK = 2 };

struct ConvArgs {
  const __bf16* in;      // [tile][vol][CIN], vol = 18^3 (padded input) or 16^3
  const __bf16* wt;      // [COUT][KP] (k = tap * CIN + ci)
  __bf16* out;           // EPI_RELU / EPI_MASK: [tile][4096][COUT]; EPI_HEAD: h3 (may be null)
  const __bf16* mask;    // EPI_MASK: [tile][4096][COUT], the layer-below activation (> 0 passes)
  const __bf16* wh;      // EPI_HEAD: head weights (16)
  float* o;              // EPI_HEAD: [tile][4096]
  long long ntiles;
  const int* done;       // optional: skip when *done (solver paused / finished)
};

// one wave: kConvRows output rows of plane z of tile t; K chunks outer.  Bound by the
// latency of the A fragments' loads: a workgroup per plane gives 27 tiles (48^3
// aggregates) 432 workgroups, 25 us for <32, 16>, where a wave per plane had 108 and
// took 73 us.
constexpr int kConvRows = 4;
template <int CIN, int COUT, bool PADDED, int EPI>
__global__ void __launch_bounds__(256) k_lpc_conv(ConvArgs a) {
  constexpr int KP = kpad(CIN);
  constexpr int NCH = KP / 32;
  constexpr int NB = COUT / 16;
  __shared__ __attribute__((aligned(16))) __bf16 s_w[COUT * (KP + 8)];   // rows 8 apart: the 16 rows of a read on distinct banks
  if (a.done && *a.done) return;
  const long long t = blockIdx.x >> 4;
  if (t >= a.ntiles) return;
  for (int q = threadIdx.x; q < COUT * KP / 8; q += 256)
    reinterpret_cast<bf16x8*>(s_w)[q + q / (KP / 8)] = reinterpret_cast<const bf16x8*>(a.wt)[q];
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int z = blockIdx.x & 15, y0 = wave * kConvRows;
  const int m = lane & 15, g = lane >> 4;
  const long long in_base = t * (long long)(PADDED ? kHaloVol : kTileVol) * CIN;

  f32x4 acc[kConvRows][NB];
#pragma unroll
  for (int y = 0; y < kConvRows; ++y)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[y][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int c = 0; c < NCH; ++c) {
    bf16x8 bw[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      bw[nb] = *reinterpret_cast<const bf16x8*>(&s_w[(nb * 16 + m) * (KP + 8) + c * 32 + g * 8]);
    const int k0 = c * 32 + g * 8;
#pragma unroll
    for (int y = 0; y < kConvRows; ++y) {
      bf16x8 av;
      if constexpr (CIN >= 8) {
        const int tap = k0 / CIN, ci0 = k0 % CIN;
        const int dx = tap % 3, dy = (tap / 3) % 3, dz = tap / 9;
        const int xi = m + dx - 1, yi = y0 + y + dy - 1, zi = z + dz - 1;
        bool ok = tap < 27;
        long long pos;
        if constexpr (PADDED) {
          pos = ((long long)(zi + 1) * kHalo + (yi + 1)) * kHalo + (xi + 1);
        } else {
          ok = ok && xi >= 0 && xi < kTile && yi >= 0 && yi < kTile && zi >= 0 && zi < kTile;
          pos = ((long long)zi * kTile + yi) * kTile + xi;
        }
        if (ok) {
          av = *reinterpret_cast<const bf16x8*>(a.in + in_base + pos * CIN + ci0);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) av[i] = (__bf16)0.f;
        }
      } else {
        // CIN == 4: the 8 k values are two taps of 4 channels
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int tap = k0 / 4 + h;
          const int dx = tap % 3, dy = (tap / 3) % 3, dz = tap / 9;
          const int xi = m + dx - 1, yi = y0 + y + dy - 1, zi = z + dz - 1;
          bf16x4 v4;
          if (tap < 27) {
            long long pos;
            if constexpr (PADDED) {
              pos = ((long long)(zi + 1) * kHalo + (yi + 1)) * kHalo + (xi + 1);
              v4 = *reinterpret_cast<const bf16x4*>(a.in + in_base + pos * 4);
            } else {
              if (xi >= 0 && xi < kTile && yi >= 0 && yi < kTile && zi >= 0 && zi < kTile) {
                pos = ((long long)zi * kTile + yi) * kTile + xi;
                v4 = *reinterpret_cast<const bf16x4*>(a.in + in_base + pos * 4);
              } else {
                for (int i = 0; i < 4; ++i) v4[i] = (__bf16)0.f;
              }
            }
          } else {
            for (int i = 0; i < 4; ++i) v4[i] = (__bf16)0.f;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) av[h * 4 + i] = v4[i];
        }
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[y][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bw[nb], acc[y][nb], 0, 0, 0);
    }
  }

  // epilogue: lane holds channel nb*16 + m of cells x = 4g + i, i = 0..3
  const long long out_base = t * (long long)kTileVol;
#pragma unroll
  for (int y = 0; y < kConvRows; ++y) {
    if constexpr (EPI == EPI_HEAD) {
      const float wh = (float)a.wh[m];
      float part[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const __bf16 h = (__bf16)fmaxf(acc[y][0][i], 0.f);
        const long long cell = ((long long)z * kTile + y0 + y) * kTile + 4 * g + i;
        if (a.out) a.out[(out_base + cell) * 16 + m] = h;
        part[i] = (float)h * wh;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) part[i] += __shfl_xor(part[i], o, 64);
      }
      if (m < 4) {
        const long long cell = ((long long)z * kTile + y0 + y) * kTile + 4 * g + m;
        float v = m == 0 ? part[0] : (m == 1 ? part[1] : (m == 2 ? part[2] : part[3]));
        a.o[out_base + cell] = v;
      }
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const long long cell = ((long long)z * kTile + y0 + y) * kTile + 4 * g + i;
          const long long idx = (out_base + cell) * COUT + nb * 16 + m;
          float v = acc[y][nb][i];
          if constexpr (EPI == EPI_RELU) v = fmaxf(v, 0.f);
          if constexpr (EPI == EPI_MASK) v = (float)a.mask[idx] > 0.f ? v : 0.f;
          a.out[idx] = (__bf16)v;
        }
    }
  }
}

// Weight gradient of one layer: gw[tap][ci][co] = sum_cells in[cell + off(tap)][ci] * g[cell][co],
// a contraction over cells: A = in^T (16 ci x 32 cells), B = g (32 cells x 16 co) on the
// matrix cores with FP32 accumulation (the BF16 products are exact).  Workgroup
// (w, dz) stages one plane of g and the plane dz of in, transposed to [channel][cell]
// in LDS; its wave dy holds the three dx taps, whose A fragments are one 16-byte LDS
// read shifted by a cell in registers.  No wave shares an output, so nothing is reduced
// inside a workgroup; it walks units (tile, 2 planes) w, w + W, ... and stores its sums
// to part[w][27*CIN*COUT].  What bounds it is latency (loads and transposing stores of
// a plane): 15 us for <32, 16> at 27 tiles, where FP32 outer products on the vector ALU
// took 284 us.
// Long FP32 chains on the matrix cores err more than the vector ALU's: chains of 4 (128
// products) are added by two-sums and the partials are FP64.  Error of the 32 -> 16
// layer's gradient against FP64, 1 / 27 / 64 tiles: 2.50e-8 / 2.64e-8 / 2.62e-8
// (rounding the result alone: 2.38e-8 / 2.56e-8 / 2.50e-8), the vector ALU's 2.72e-8 /
// 2.81e-8 / 3.41e-8; chains of 8 give 2.69e-8 / 2.79e-8 / 2.91e-8 in 14 us.
// Channel strides of 148 and 132 dwords put the 16 channels of a fragment read on
// distinct banks.
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWgradChain = 4;
template <int CIN, int COUT, bool PADDED>
__global__ void __launch_bounds__(192) k_lpc_wgrad(const __bf16* __restrict__ in, const __bf16* __restrict__ gr,
                                                   long long ntiles, double* __restrict__ part) {
  static_assert(PADDED ? CIN == 4 : CIN % 16 == 0, "channel layout");
  constexpr int MT = CIN >= 16 ? CIN / 16 : 1;   // 16-row tiles of ci (CIN 4: 3 dx x 4 ci in one)
  constexpr int DX = CIN >= 16 ? 3 : 1;
  constexpr int NB = COUT / 16;
  constexpr int RW = PADDED ? 12 : 8;            // dwords a row: 8 pairs of cells (and the halo pair)
  constexpr int CS = 18 * RW + 4, GS = 132;      // dwords a channel
  __shared__ __attribute__((aligned(16))) uint32_t s_in[CIN * CS];
  __shared__ __attribute__((aligned(16))) uint32_t s_g[COUT * GS];
  const int dz = (int)(blockIdx.x % 3);
  const long long w = blockIdx.x / 3, W = gridDim.x / 3;
  const int lane = threadIdx.x & 63, dy = threadIdx.x >> 6;
  const int m = lane & 15, q = lane >> 4, half = q & 1;
  f32x4 acc[MT][DX][NB], sum[MT][DX][NB], low[MT][DX][NB];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < DX; ++b)
#pragma unroll
      for (int c = 0; c < NB; ++c) acc[a][b][c] = sum[a][b][c] = low[a][b][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (!PADDED) {
    // rows y = -1 and 16 stay zero
    for (int k = threadIdx.x; k < CIN * 2 * RW; k += 192)
      s_in[(k / (2 * RW)) * CS + (k % (2 * RW) < RW ? 0 : 16 * RW) + k % (2 * RW)] = 0u;
  }
  for (long long u = w * 2; u < ntiles * 16; u += (u & 1) ? 2 * W - 1 : 1) {
    const long long t = u >> 4;
    const int z = (int)(u & 15);
    const int zi = z + dz - 1;
    if (!PADDED && (zi < 0 || zi >= kTile)) continue;
    __syncthreads();
    if constexpr (PADDED) {
      const u16x4* src = reinterpret_cast<const u16x4*>(in) + t * kHaloVol + (long long)(z + dz) * (kHalo * kHalo);
      for (int k = threadIdx.x; k < kHalo * 9; k += 192) {
        const int row = k / 9, e = k % 9;
        const u16x4 lo = src[row * kHalo + (e < 8 ? 1 + 2 * e : 17)], hi = src[row * kHalo + (e < 8 ? 2 + 2 * e : 0)];
#pragma unroll
        for (int j = 0; j < 4; ++j) s_in[j * CS + row * RW + e] = (uint32_t)lo[j] | ((uint32_t)hi[j] << 16);
      }
    } else {
      constexpr int CG = CIN / 8;
      const u16x8* src = reinterpret_cast<const u16x8*>(in) + (t * kTileVol + (long long)zi * 256) * CG;
      for (int k = threadIdx.x; k < 128 * CG; k += 192) {
        const int cg = k % CG, pr = k / CG;
        const u16x8 lo = src[2 * pr * CG + cg], hi = src[(2 * pr + 1) * CG + cg];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          s_in[(cg * 8 + j) * CS + RW + pr] = (uint32_t)lo[j] | ((uint32_t)hi[j] << 16);
      }
    }
    {
      constexpr int CG = COUT / 8;
      const u16x8* src = reinterpret_cast<const u16x8*>(gr) + (t * kTileVol + (long long)z * 256) * CG;
      for (int k = threadIdx.x; k < 128 * CG; k += 192) {
        const int cg = k % CG, pr = k / CG;
        const u16x8 lo = src[2 * pr * CG + cg], hi = src[(2 * pr + 1) * CG + cg];
#pragma unroll
        for (int j = 0; j < 8; ++j) s_g[(cg * 8 + j) * GS + pr] = (uint32_t)lo[j] | ((uint32_t)hi[j] << 16);
      }
    }
    __syncthreads();
#pragma unroll kWgradChain
    for (int ks = 0; ks < 8; ++ks) {   // 32 cells = 2 rows: quarter-wave q has half a row
      bf16x8 bv[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        bv[nb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&s_g[(nb * 16 + m) * GS + ks * 16 + q * 4]));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int ci = CIN >= 16 ? mt * 16 + m : (m & 3);
        const uint32_t* row = &s_in[ci * CS + (2 * ks + (q >> 1) + dy) * RW];
        const u32x4 d = *reinterpret_cast<const u32x4*>(row + half * 4);
        uint32_t prev, next;
        if constexpr (PADDED) {
          prev = row[half ? 3 : 8];
          next = row[half ? 8 : 4];
        } else {
          const uint32_t nbr = row[half ? 3 : 4];
          prev = half ? nbr : 0u;
          next = half ? 0u : nbr;
        }
        const u32x4 dm = {__builtin_amdgcn_alignbyte(d[0], prev, 2), __builtin_amdgcn_alignbyte(d[1], d[0], 2),
                          __builtin_amdgcn_alignbyte(d[2], d[1], 2), __builtin_amdgcn_alignbyte(d[3], d[2], 2)};
        const u32x4 dp = {dm[1], dm[2], dm[3], __builtin_amdgcn_alignbyte(next, d[3], 2)};
        if constexpr (CIN >= 16) {
          const u32x4 av[3] = {dm, d, dp};
#pragma unroll
          for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[mt][dx][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[dx]), bv[nb],
                                                                        acc[mt][dx][nb], 0, 0, 0);
        } else {
          const int dx = m >> 2;
          const u32x4 av = dx == 0 ? dm : (dx == 1 ? d : (dx == 2 ? dp : u32x4{0u, 0u, 0u, 0u}));
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[0][0][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), bv[nb],
                                                                    acc[0][0][nb], 0, 0, 0);
        }
      }
      if (ks % kWgradChain == kWgradChain - 1) {
        // two-sum (Knuth): sum + low holds the chains' total
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
          for (int b = 0; b < DX; ++b)
#pragma unroll
            for (int c = 0; c < NB; ++c) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float x = sum[a][b][c][i], y = acc[a][b][c][i], r = x + y, v = r - x;
                low[a][b][c][i] += (x - (r - v)) + (y - v);
                sum[a][b][c][i] = r;
              }
              acc[a][b][c] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
      }
    }
  }
  double* dst = part + w * (27 * CIN * COUT) + (9 * dz + 3 * dy) * (CIN * COUT);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int dx = 0; dx < DX; ++dx)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tap = CIN >= 16 ? dx : q, ci = CIN >= 16 ? mt * 16 + 4 * q + i : i;
          // (past FP32's range the two-sum's rest is NaN: the sum stands alone)
          const double hi = sum[mt][dx][nb][i], rest = isfinite(hi) ? low[mt][dx][nb][i] : 0.f;
          if (tap < 3) dst[(tap * CIN + ci) * COUT + nb * 16 + m] = hi + rest;
        }
}

// head gradient: dh3 = bf16(go * Wh ⊙ (h3 > 0)); partial gWh[co] = sum_cells h3 * go
__global__ void __launch_bounds__(256) k_lpc_head_bwd(const __bf16* __restrict__ h3, const float* __restrict__ go,
                                                      const __bf16* __restrict__ wh, long long ncells,
                                                      __bf16* __restrict__ dh3, double* __restrict__ part) {
  __shared__ float s[16][17];
  float acc = 0.f;
  const int co = threadIdx.x & 15;
  const float w = (float)wh[co];
  for (long long q = (long long)blockIdx.x * 16 + (threadIdx.x >> 4); q < ncells; q += (long long)gridDim.x * 16) {
    const float h = (float)h3[q * 16 + co];
    const float gv = go[q];
    acc = fmaf(h, gv, acc);
    dh3[q * 16 + co] = (__bf16)(h > 0.f ? gv * w : 0.f);
  }
  s[threadIdx.x >> 4][co] = acc;
  __syncthreads();
  if (threadIdx.x < 16) {
    float r = 0.f;
    for (int k = 0; k < 16; ++k) r += s[k][threadIdx.x];
    part[(long long)blockIdx.x * 16 + threadIdx.x] = r;
  }
}

// grad = the FP64 sums of every layer's partials part[w][n], n contiguous outputs a
// layer: 16 threads an output, thread k takes w = k, k + 16, ... in order, the 16 sums
// are added in order (deterministic).  One launch for all layers, latency bound: about 9 us
// for 216 partials, where a thread per output and a launch per layer took 456 us.
struct LpcParts {
  const double* part[4];
  int nparts[4], off[5];
};

__global__ void __launch_bounds__(256) k_lpc_sum_parts(LpcParts p, float* __restrict__ grad) {
  __shared__ double s[16][17];
  const int k = threadIdx.x >> 4, lo = threadIdx.x & 15;
  const int i = blockIdx.x * 16 + lo;   // the layers' sizes are multiples of 16
  int l = 0;
  while (l < 3 && (int)blockIdx.x * 16 >= p.off[l + 1]) ++l;
  const int n = p.off[l + 1] - p.off[l], np = p.nparts[l];
  const double* src = p.part[l] + (i - p.off[l]);
  double a = 0.0;
#pragma unroll 8
  for (int w = k; w < np; w += 16) a += src[(long long)w * n];
  s[k][lo] = a;
  __syncthreads();
  if (threadIdx.x < 16) {
    double r = 0.0;
    for (int q = 0; q < 16; ++q) r += s[q][threadIdx.x];
    grad[i] = (float)r;
  }
}

// FP32 master weights -> BF16 layer matrices: forward WT[co][tap*CIN + ci] and the
// backward-data (tap-flipped, transposed) WB[ci][tap*COUT + co]; K padding is zero
template <int CIN, int COUT>
__device__ inline void prep_layer(const float* w, __bf16* wt, __bf16* wb, int idx) {
  constexpr int KPF = kpad(CIN), KPB = kpad(COUT);
  if (idx < COUT * KPF) {
    const int co = idx / KPF, k = idx % KPF;
    float v = 0.f;
    if (k < 27 * CIN) {
      const int tap = k / CIN, ci = k % CIN;
      v = w[(tap * CIN + ci) * COUT + co];
    }
    wt[idx] = (__bf16)v;
  }
  if (idx < CIN * KPB) {
    const int ci = idx / KPB, k = idx % KPB;
    float v = 0.f;
    if (k < 27 * COUT) {
      const int tapf = k / COUT, co = k % COUT;
      v = w[((26 - tapf) * CIN + ci) * COUT + co];
    }
    wb[idx] = (__bf16)v;
  }
}

struct LpcW {
  __bf16 *w1f, *w1b, *w2f, *w2b, *w3f, *w3b, *wh;
};

__global__ void __launch_bounds__(256) k_lpc_prep(const float* __restrict__ w, LpcW o) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  prep_layer<4, 16>(w + kOffW1, o.w1f, o.w1b, idx);
  prep_layer<16, 32>(w + kOffW2, o.w2f, o.w2b, idx);
  prep_layer<32, 16>(w + kOffW3, o.w3f, o.w3b, idx);
  if (idx < kNWH) o.wh[idx] = (__bf16)w[kOffWH + idx];
}

// Adam (Kingma and Ba, 2015) on the FP32 master weights
__global__ void __launch_bounds__(256) k_lpc_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                                                  const float* __restrict__ g, int n, float lr, float b1, float b2,
                                                  float eps, float bc1, float bc2) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

__global__ void __launch_bounds__(256) k_f32_to_bf16(const float* __restrict__ in, __bf16* __restrict__ out,
                                                     long long n) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    out[i] = (__bf16)in[i];
}

// ---------------------------------------------------------------- solver coupling
// (the network's inputs and outputs in the solver are built in pf_lpc_cw.hip)

// y = A x over the list (conductance form, FP32); optional q = r - y with partial
// sums q.q and r.r (slots 0, 1)
__global__ void __launch_bounds__(256) k_lpc_apply_a(VecArgs a, const float* __restrict__ x, const float* __restrict__ r,
                                                     float* __restrict__ y, const float* __restrict__ cd,
                                                     const float* __restrict__ cx, const float* __restrict__ cy,
                                                     const float* __restrict__ cz, float scale_out) {
  const int lane = threadIdx.x & 63;
  double qq = 0.0, rr = 0.0;
  FOR_LIST_BLOCKS(a, b, lane) {
    long long c = b * kBlockVol + lane;
    CellNbr n = neighbours(a.dc, b, lane);
    const float xc = x[c];
    float ax = cd[c] * xc;
    ax = fmaf(cx[c], xc - x[n.xp], ax);
    ax = fmaf(cx[n.xm], xc - x[n.xm], ax);
    ax = fmaf(cy[c], xc - x[n.yp], ax);
    ax = fmaf(cy[n.ym], xc - x[n.ym], ax);
    ax = fmaf(cz[c], xc - x[n.zp], ax);
    ax = fmaf(cz[n.zm], xc - x[n.zm], ax);
    if (r) {
      const float q = r[c] - ax;
      y[c] = q;
      qq += (double)q * (double)q;
      rr += (double)r[c] * (double)r[c];
    } else {
      y[c] = scale_out * ax;
    }
  }
  double v[2] = {qq, rr};
  const bool mx[2] = {false, false};
  block_reduce_store<2>(v, mx, a.part, kMaxPartials);
}

}  // namespace pf
