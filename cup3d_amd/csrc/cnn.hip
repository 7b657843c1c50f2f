// Learned warm start: network, inference and training kernels.
//
// Network (per 8^3 block, one-cell halo), in the increment form of the
// pressure solve (PressureProjection.cpp:368-385 solves for p - p_old with
// rhs b - A p_old):
//   input  2 x 10^3      ch0 = res / (h_b s_r), ch1 = p_prev / s_p,
//                        res = b - A p_prev, s_r = RMS(res / h_b), s_p = RMS(p_prev)
//   conv 3^3 valid  2 -> 16, GELU
//   conv 3^3 same  16 -> 16, GELU      (zero padding inside the block)
//   conv 3^3 same  16 -> 1
//   p_net = p_prev + s_r * out
// res / h_b has the units of the 7-point stencil applied to the increment
// (A = h^3 lap), so the input is commensurate on every AMR level. Halo: a face
// halo cell takes the adjacent cell of the same-level neighbour block; every
// other halo cell (wall, coarse/fine face, edge, corner) repeats the nearest
// cell of the block.
//
// Inference (k_cnn_infer): one workgroup per block, activations in LDS as
// FP16 channel-last cells with a shared zero ring, the
// input as the [10][10][10] patch, each layer an implicit
// GEMM on v_mfma_f32_16x16x32_f16 (M = 16 cells, N = 16 output channels,
// K = 27 offsets x input channels; the 8 consecutive K of a lane are 8
// channels of one offset: one 16-byte LDS read), FP32 accumulation, bias and
// GELU in FP32.
// Training (k_cnn_train_item + k_cnn_adam): FP32 on v_mfma_f32_16x16x4_f32, one
// workgroup per (sample, block) item, forward and backward in LDS, per-item
// gradients summed in a fixed order (deterministic), Adam.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>

#include "cnn.h"
#include "device_common.h"
#include "kernels.h"

namespace cup3d {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// GELU of two values as FP16, x in the lower half: the last product is rounded
// once, from its exact value, and lands in its half of the word.
__device__ __forceinline__ unsigned gelu_pair(float x, float y) {
  const float hx = 0.5f * x, ex = 1.0f + erff(x * 0.70710678118654752f);
  const float hy = 0.5f * y, ey = 1.0f + erff(y * 0.70710678118654752f);
  unsigned r;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,0,0]" : "=v"(r) : "v"(hx), "v"(ex));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel_hi:[0,0,0]" : "+v"(r) : "v"(hy), "v"(ey));
  return r;
}

// Index into a field of the cell that padded position (pz, py, px) in 0..9
// of block b takes its value from (the halo rule above).
__device__ __forceinline__ size_t halo_index(const int* __restrict__ nbr, int b, int pz, int py,
                                             int px) {
  int c[3] = {px - 1, py - 1, pz - 1};
  int out = 0, dim = -1;
  for (int d = 0; d < 3; ++d)
    if (c[d] < 0 || c[d] > 7) {
      ++out;
      dim = d;
    }
  int blk = b;
  if (out == 1) {
    const int face = 2 * dim + (c[dim] > 7 ? 1 : 0);
    const int nb = nbr[b * 6 + face];
    if (nb >= 0) {
      blk = nb;
      c[dim] = c[dim] > 7 ? 0 : 7;
    }
  }
  for (int d = 0; d < 3; ++d) c[d] = c[d] < 0 ? 0 : (c[d] > 7 ? 7 : c[d]);
  return (size_t)blk * BLEN + c[2] * 64 + c[1] * 8 + c[0];
}

// ---------------------------------------------------------------------------
// scal[slot] = RMS(f / h_b) (h = nullptr: RMS(f)); deterministic two-pass sum
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(WG_THREADS) void k_cnn_rms(long long n, const double* __restrict__ f,
                                                        const double* __restrict__ h,
                                                        double* part) {
  double v[1] = {0.0};
  const long long base = (long long)blockIdx.x * (4 * BLEN);
  for (int e = threadIdx.x; e < 4 * BLEN; e += WG_THREADS) {
    const long long i = base + e;
    if (i < n) {
      const double x = h ? f[i] / h[i / BLEN] : f[i];
      v[0] += x * x;
    }
  }
  grid_store_partial<1>(v, part);
}

__global__ __launch_bounds__(WG_THREADS) void k_cnn_rms_fin(long long n, double* scal, int slot,
                                                            const double* part, int nparts) {
  double tot[1];
  grid_sum_partials<1>(part, nparts, tot);
  if (threadIdx.x == 0) {
    const double s = sqrt(tot[0] / (double)n);
    scal[slot] = s > 0 ? s : 1.0;
  }
}

// scal[0] = RMS(res / h_b), scal[1] = RMS(p_prev) from the sums of SPMV_NET
__global__ __launch_bounds__(WG_THREADS) void k_cnn_scales_fin(long long n, double* scal,
                                                               const double* part, int nparts) {
  double tot[2];
  grid_sum_partials<2>(part, nparts, tot);
  if (threadIdx.x < 2) {
    const double s = sqrt(tot[threadIdx.x] / (double)n);
    scal[threadIdx.x] = s > 0 ? s : 1.0;
  }
}

// scal[2] = volume-weighted mean of p - p_prev: sum h^3 (p - p_prev) / sum h^3
__global__ __launch_bounds__(WG_THREADS) void k_cnn_dmean(long long n, const double* __restrict__ p,
                                                          const double* __restrict__ prev,
                                                          const double* __restrict__ h,
                                                          double* part) {
  double v[2] = {0.0, 0.0};
  const long long base = (long long)blockIdx.x * (4 * BLEN);
  for (int e = threadIdx.x; e < 4 * BLEN; e += WG_THREADS) {
    const long long i = base + e;
    if (i < n) {
      const double hb = h[i / BLEN], h3 = hb * hb * hb;
      v[0] += h3 * (p[i] - prev[i]);
      v[1] += h3;
    }
  }
  grid_store_partial<2>(v, part);
}

__global__ __launch_bounds__(WG_THREADS) void k_cnn_dmean_fin(double* scal, const double* part,
                                                              int nparts) {
  double tot[2];
  grid_sum_partials<2>(part, nparts, tot);
  if (threadIdx.x == 0) scal[2] = tot[1] > 0 ? tot[0] / tot[1] : 0.0;
}

// ---------------------------------------------------------------------------
// FP16 weight packing for the implicit-GEMM inference.
// Fragment kt, lane l (n = l % 16 output channel, g = l / 16), element e:
//   layer 1: offset o = 4 kt + g, channel c = e (c < 2 real)
//   layers 2, 3: offset o = 2 kt + g / 2, channel c = 8 (g % 2) + e
// (o = dz*9 + dy*3 + dx; o >= 27 and missing channels are zero; layer 3 has
// a single real output channel n = 0).
// ---------------------------------------------------------------------------
__global__ void k_cnn_pack(const float* __restrict__ w, _Float16* __restrict__ pk) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= CNN_PK) return;
  const int e = idx & 7, l = (idx >> 3) & 63, frag = idx >> 9;
  const int n = l & 15, g = l >> 4;
  float v = 0.f;
  if (frag < CNN_KT1) {
    const int o = 4 * frag + g, c = e;
    if (o < 27 && c < 2) v = w[(n * 2 + c) * 27 + o];
  } else if (frag < CNN_KT1 + CNN_KT2) {
    const int kt = frag - CNN_KT1, o = 2 * kt + g / 2, c = 8 * (g % 2) + e;
    if (o < 27) v = w[CNN_OW2 + (n * CNN_C + c) * 27 + o];
  } else {
    const int kt = frag - CNN_KT1 - CNN_KT2, o = 2 * kt + g / 2, c = 8 * (g % 2) + e;
    if (o < 27 && n == 0) v = w[CNN_OW3 + c * 27 + o];
  }
  pk[idx] = (_Float16)v;
}

// ---------------------------------------------------------------------------
// Inference: one workgroup (4 waves) per block.
// ---------------------------------------------------------------------------
constexpr int PADC = 1000;  // 10^3 padded cells

__device__ __forceinline__ int padded(int m) {  // cell 0..511 -> padded index
  return (((m >> 6) + 1) * 10 + ((m >> 3) & 7) + 1) * 10 + (m & 7) + 1;
}

// Activations in LDS: cells of CNN_C halfs, rows of 8 cells behind one zero
// cell, planes of 8 rows behind one zero row, one zero plane in front and one
// behind. The zero cell in front of a row is also the one behind the row
// before it (and so for rows and planes), so the "same" padding costs 820
// cells against 1000, and three workgroups fit a CU.
// The two 16-byte halves of a cell (channels 0-7 and 8-15) change places in the
// padded rows 4 to 7. A tile is the rows y and y + 4 of a plane: the sixteen
// cells that lanes 0-15 read are then in sixteen different 16-byte slots of the
// 64 banks (in the input patch too, whose rows are 40 cells apart), and a read
// takes 6 cycles; with the rows y and y + 1, or the halves in place, 9.4.
constexpr int AROW = 9, APLANE = 81, ACELLS = 9 * APLANE + 9 * AROW + AROW + 1;
__device__ __forceinline__ constexpr int atap(int o) {  // tap o from the (-1, -1, -1) corner
  return (o / 9) * APLANE + ((o / 3) % 3) * AROW + o % 3;
}

// A wavefront owns two planes, eight tiles: tile 4 p + j is the rows j and j + 4
// of plane p. Products are taken with the weights as the first operand, so that
// register q of lane l holds channel 4 (l / 16) + q of cell l % 16 of the tile:
// four channels of a cell are one 8-byte store.

// Layer 1 (valid) on the 10^3 input patch, 8 halfs a cell: 4 taps a k-step,
// tap 4 kt + g in the lanes of group g. The lane's tap offsets are registers
// made once, a tile's offset is added to one base.
template <typename F>
__device__ __forceinline__ void conv_first(const _Float16* __restrict__ in,
                                           const half8_t* __restrict__ wfrag, int w, int l,
                                           F&& f) {
  const int lr = l & 15, g = l >> 4;
  half8_t bq[CNN_KT1];
#pragma unroll
  for (int kt = 0; kt < CNN_KT1; ++kt) bq[kt] = wfrag[kt * 64 + l];
  int po[CNN_KT1];  // halfs
#pragma unroll
  for (int kt = 0; kt < CNN_KT1; ++kt) {
    const int o = 4 * kt + g;
    po[kt] = o < 27 ? ((o / 9) * 100 + ((o / 3) % 3) * 10 + o % 3) * 8 : 0;
  }
  const int base = (2 * w * 100 + (lr >> 3) * 40 + (lr & 7)) * 8;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const _Float16* p = in + base + ((t >> 2) * 100 + (t & 3) * 10) * 8;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < CNN_KT1; ++kt) {
      half8_t a = *reinterpret_cast<const half8_t*>(p + po[kt]);
      if (kt == CNN_KT1 - 1 && g == 3) {  // there is no tap 27
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = (_Float16)0.f;
      }
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(bq[kt], a, acc, 0, 0, 0);
    }
    f(t, acc);
  }
}

// Layers 2 and 3 (same): 2 taps a k-step, taps 2 kt and 2 kt + 1 in the lower
// and upper lanes, 1, 7 or 61 cells apart. The operand of padded rows r and
// r + 4 of a padded plane from column dx serves every output tile that meets it
// with a tap pair of the same distance (rows r - dy, plane z - dz): it is read
// once for all of them, 78 reads for the 112 products. Planes, rows and columns
// are walked in ascending order, so a tile's k-steps come in ascending order.
// Every address is one of seven bases and an immediate offset.
template <typename F>
__device__ __forceinline__ void conv_same(const _Float16* __restrict__ in,
                                          const half8_t* __restrict__ wfrag, int w, int l, F&& f) {
  constexpr int KT = CNN_KT2;
  static_assert(CNN_KT2 == CNN_KT3 && CNN_C == 16, "two taps of 16 channels a k-step");
  const int lr = l & 15, g = l >> 4, hi = g >> 1, rr = lr >> 3;
  half8_t bq[KT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) bq[kt] = wfrag[kt * 64 + l];
  // a base per distance and place of the halves (lower lanes' row, upper lanes'
  // row at or past 4: fl, fu)
  const int c0 = (2 * w * APLANE + rr * 4 * AROW + (lr & 7)) * CNN_C, s = (g & 1) ^ rr;
  auto base = [&](int d, int fl, int fu) {
    return in + c0 + hi * d * CNN_C + 8 * (s ^ (hi ? fu : fl));
  };
  const _Float16* const p1[2] = {base(1, 0, 0), base(1, 1, 1)};
  const _Float16* const p7[3] = {base(7, 0, 0), base(7, 0, 1), base(7, 1, 1)};
  const _Float16* const p61[2] = {base(61, 0, 0), base(61, 1, 0)};
  float4_t acc[2][4];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[p][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int z = 0; z < 4; ++z) {
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const int at = (z * APLANE + r * AROW + dx) * CNN_C;
        // one operand per distance: 1 (dx 0 and 1), 7, 61, or the last tap alone
#pragma unroll
        for (int cls = 0; cls < 4; ++cls) {
          bool used = false;
          half8_t a;
#pragma unroll
          for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
              const int o = 9 * dz + 3 * dy + dx, p = z - dz, j = r - dy;
              const int c = dx < 2 ? 0 : (o == 26 ? 3 : (o == 8 ? 2 : 1));
              if (o % 2 || c != cls || p < 0 || p > 1 || j < 0 || j > 3) continue;
              if (!used) {
                const _Float16* q = cls == 0   ? p1[r >= 4]
                                    : cls == 1 ? p7[(r >= 3) + (r >= 4)]
                                    : cls == 2 ? p61[r >= 4]
                                               : p1[r >= 4];
                // there is no tap 27: the upper lanes read the ring's first (zero) cell
                if (cls == 3) q = hi ? in - at : q;
                a = *reinterpret_cast<const half8_t*>(q + at);
                used = true;
              }
              acc[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bq[o / 2], a, acc[p][j], 0, 0, 0);
            }
        }
      }
    if (z >= 2) {  // the last plane that output plane z - 2 reads
#pragma unroll
      for (int j = 0; j < 4; ++j) f(4 * (z - 2) + j, acc[z - 2][j]);
    }
  }
}

// Zero the ring of an activation buffer (the 512 cells are written by a layer):
// the planes in front and behind, then each plane's first row and the first
// cell of its other rows.
constexpr int ARING = ACELLS - BLEN;
__device__ __forceinline__ void zero_ring(_Float16* buf, int tid) {
  half8_t zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (_Float16)0.f;
  constexpr int ENDS = ARING - BS * (AROW + BS);
#pragma unroll
  for (int i = tid; i < ARING; i += WG_THREADS) {
    const int k = i - ENDS, z = k / (AROW + BS), m = k - z * (AROW + BS);
    const int c = i < APLANE ? i
                  : i < ENDS ? 9 * APLANE + i - APLANE
                             : (z + 1) * APLANE + (m < AROW ? m : (m - BS) * AROW);
    half8_t* p = reinterpret_cast<half8_t*>(&buf[c * CNN_C]);
    p[0] = zero;
    p[1] = zero;
  }
}

// LDS of the inference: the input patch (1000 cells x 8 halfs), later the
// second layer's activations, and the first layer's: 52 KiB per workgroup,
// three workgroups per CU. The vector ALUs bound it, mostly by the exact GELU of
// 16 384 values a block (about 36 instructions each, 120 us of 8192 blocks); the
// LDS reads and the products (60 us) run beside them. A predict of 8192 blocks, of
// which this kernel is all but 35 us (210 us under the profiler): 396 us with the
// zero padding selected per operand (20 instructions a read), 264 us with it built
// into the layout, 221 us with conflict-free reads shared by the tiles, four
// channels a store and the halo positions by face.
constexpr int CNN_IN_HALFS = PADC * 8 > ACELLS * CNN_C ? PADC * 8 : ACELLS * CNN_C;

__global__ __launch_bounds__(WG_THREADS) void k_cnn_infer(int nb, const int* __restrict__ nbr,
                                                          const double* __restrict__ h,
                                                          const double* __restrict__ res,
                                                          const double* __restrict__ prev,
                                                          const double* __restrict__ scal,
                                                          const _Float16* __restrict__ wpk,
                                                          const float* __restrict__ w,
                                                          double* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) _Float16 bufIn[CNN_IN_HALFS];     // input, then act2
  __shared__ __attribute__((aligned(16))) _Float16 bufA[ACELLS * CNN_C];  // act1, then the output
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  if (b >= nb) return;
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, g = l >> 4;
  const double s_r = scal[0];
  const float inv_sp = (float)(1.0 / scal[1]);
  const float inv_hs = (float)(1.0 / (h[b] * s_r));
  // input: 8-channel cells (2 real); the indices of a thread's (up to 4)
  // positions first, then all 8 loads, so the gather costs two memory round
  // trips, not one per position. Positions: two cells of the block, then the
  // halo, a face per wavefront (so its axis is a scalar), edges and corners.
  constexpr int NP = 4, HALO = PADC - BLEN;
  static_assert(WG_THREADS == 256 && HALO <= 2 * WG_THREADS, "two cells and two halo positions");
  size_t gi[NP];
  int pi[NP];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = tid + j * WG_THREADS;
    gi[j] = (size_t)b * BLEN + m;
    pi[j] = padded(m);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = tid + j * WG_THREADS;
    const int face = __builtin_amdgcn_readfirstlane(i >> 6);
    int src = b, c, p;
    if (face < 6) {
      const int d = face >> 1, side = face & 1, u = l & 7, v = l >> 3;
      const int sd = d == 0 ? 1 : (d == 1 ? 8 : 64), pd = d == 0 ? 1 : (d == 1 ? 10 : 100);
      const int s1 = d == 0 ? 8 : 1, s2 = d == 2 ? 8 : 64;
      const int p1 = d == 0 ? 10 : 1, p2 = d == 2 ? 10 : 100;
      const int nbf = nbr[b * 6 + face];
      if (nbf >= 0) src = nbf;
      c = ((side != 0) == (nbf < 0) ? 7 : 0) * sd + u * s1 + v * s2;
      p = (side ? 9 : 0) * pd + (u + 1) * p1 + (v + 1) * p2;
    } else {  // the nearest cell: 12 edges of 8, then 8 corners
      const int e = i - 384, ed = e >> 3, t = e & 7;
      int q[3];  // padded position
      if (e < 96) {
        const int d = ed >> 2, lo = ed & 1 ? 9 : 0, hi = ed & 2 ? 9 : 0;
        q[0] = d == 0 ? t + 1 : lo;
        q[1] = d == 1 ? t + 1 : (d == 0 ? lo : hi);
        q[2] = d == 2 ? t + 1 : hi;
      } else {
        q[0] = e & 1 ? 9 : 0;
        q[1] = e & 2 ? 9 : 0;
        q[2] = e & 4 ? 9 : 0;
      }
      auto near = [](int x) { return min(max(x - 1, 0), 7); };
      c = near(q[0]) + 8 * near(q[1]) + 64 * near(q[2]);
      p = i < HALO ? q[0] + 10 * q[1] + 100 * q[2] : -1;
    }
    gi[2 + j] = (size_t)src * BLEN + c;
    pi[2 + j] = p;
  }
  double rv[NP], pv[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    rv[j] = res[gi[j]];
    pv[j] = prev[gi[j]];
  }
  zero_ring(bufA, tid);
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    if (pi[j] >= 0) {
      half8_t v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (_Float16)0.f;
      v[0] = (_Float16)((float)rv[j] * inv_hs);
      v[1] = (_Float16)((float)pv[j] * inv_sp);
      *reinterpret_cast<half8_t*>(&bufIn[pi[j] * 8]) = v;
    }
  }
  __syncthreads();
  const half8_t* wf = reinterpret_cast<const half8_t*>(wpk);
  // this lane's cell in tile 0, its four channels 4 g .. 4 g + 3 (rows j = 3 and 7
  // are the padded rows 4 and 8, where the halves' places change)
  const int rr = lr >> 3;
  const int ocell = ((2 * wv + 1) * APLANE + (4 * rr + 1) * AROW + (lr & 7) + 1) * CNN_C + 4 * (g & 1);
  const int oh[2] = {ocell + 8 * ((g >> 1) ^ rr), ocell + 8 * ((g >> 1) ^ rr ^ 1)};
  auto store = [&](_Float16* buf, const float (&bias)[4], int t, const float4_t& acc) {
    typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
    const uint2_t v = {gelu_pair(acc[0] + bias[0], acc[1] + bias[1]),
                       gelu_pair(acc[2] + bias[2], acc[3] + bias[3])};
    *reinterpret_cast<uint2_t*>(
        &buf[oh[(t & 3) == 3] + ((t >> 2) * APLANE + (t & 3) * AROW) * CNN_C]) = v;
  };
  float b1[4], b2[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    b1[q] = w[CNN_OB1 + 4 * g + q];
    b2[q] = w[CNN_OB2 + 4 * g + q];
  }
  const float b3 = w[CNN_OB3];
  conv_first(bufIn, wf, wv, l, [&](int t, const float4_t& acc) { store(bufA, b1, t, acc); });
  __syncthreads();
  zero_ring(bufIn, tid);
  conv_same(bufA, wf + CNN_KT1 * 64, wv, l,
            [&](int t, const float4_t& acc) { store(bufIn, b2, t, acc); });
  __syncthreads();
  float* po = reinterpret_cast<float*>(bufA);
  const int ocol = 128 * wv + 32 * rr + (lr & 7);
  conv_same(bufIn, wf + (CNN_KT1 + CNN_KT2) * 64, wv, l, [&](int t, const float4_t& acc) {
    if (g == 0) po[ocol + 64 * (t >> 2) + 8 * (t & 3)] = acc[0];
  });
  __syncthreads();
  const size_t off = (size_t)b * BLEN;
#pragma unroll
  for (int m = tid; m < BLEN; m += WG_THREADS)
    out[off + m] = prev[off + m] + s_r * (double)(po[m] + b3);
}

// ---------------------------------------------------------------------------
// Training (FP32)
// ---------------------------------------------------------------------------
struct SampleRef {
  const float* res_h;
  const float* prev;
  const float* target;
  float s_r;
  float s_p;
};

// ---------------------------------------------------------------------------
// One (sample, block) item per workgroup of 8 wavefronts, forward and backward
// with everything in LDS and registers: every contraction is an implicit GEMM
// on v_mfma_f32_16x16x4_f32 (FP32 inputs and accumulation). Wavefront w owns
// the z plane w of the block: four tiles of 16 cells (two x rows), so the 16
// channels x 16 cells accumulators of the forward layers, of their
// pre-activations and of the backward layers are the same registers.
//   layer 1, 2      M = 16 cells, N = 16 channels, K = (offset, channel)
//   layer 3         M = 16 cells, N = offset, K = channel: the products of
//                   every cell with the 27 taps, then 27 shifted adds
//   dZ2, dZ1        the same convolutions with the taps mirrored
//   dW              M, N = channels (or N = taps), K = the 512 cells: offsets
//                   or tap tiles are split over the wavefronts
// Bound by the FP32 matrix cores: 12 064 MFMAs of 32 cycles an item over 4
// SIMDs, 40 us at 2.4 GHz; a batch of 256 items gives every CU one. With
// scalar FP32 loops through a global scratch buffer (200 KB an item) a step of
// 256 items took 2156 us; now 80 us.
//
// LDS (floats): the input patch, act1 on the zero-padded 10^3 patch, then act2
// and the tap products (later dZ2 on its padded patch), dL/dout padded, the
// prediction with the target's halo, the local residual. A channel stride of
// 1010 (18 mod 32 banks) keeps the 16 channels x 2 cells a half-wave reads for
// the weight gradients in different banks.
// ---------------------------------------------------------------------------
constexpr int TR_T = 512;               // threads per item
constexpr int TR_CS = PADC + 10;        // channel stride of the padded patches
constexpr int TR_HS = BLEN + 20;        // of the unpadded ones (16-byte rows)
constexpr int TR_X = 0;                 // [2][1000]
constexpr int TR_H1 = TR_X + 2 * PADC;  // [16][TR_CS]; later dZ1 [16][TR_HS]
constexpr int TR_H2 = TR_H1 + CNN_C * TR_CS;   // [16][TR_HS]; later dZ2 [16][TR_CS]
constexpr int TR_P = TR_H2 + CNN_C * TR_HS;    // [16][TR_HS] tap products, reductions
constexpr int TR_D = TR_P + CNN_C * TR_HS;     // [1000]
constexpr int TR_OP = TR_D + PADC;             // [1000]
constexpr int TR_RHO = TR_OP + PADC;           // [512]
constexpr int TR_RED = TR_RHO + BLEN;          // [8][16] per-wavefront sums
constexpr int TR_LDS = TR_RED + 8 * 16;
static_assert(TR_X % 4 == 0 && TR_H1 % 4 == 0 && TR_H2 % 4 == 0 && TR_P % 4 == 0 && TR_HS % 4 == 0,
              "16-byte rows");
static_assert(TR_P + CNN_C * TR_HS - TR_H2 >= CNN_C * TR_CS, "dZ2 fits over act2 and the products");
static_assert(TR_LDS * 4 <= 160 * 1024, "LDS of one CU");

// offset of tap off (dz, dy, dx) in the padded 10^3 patch
__device__ __forceinline__ constexpr int tap(int off) {
  return (off / 9) * 100 + ((off / 3) % 3) * 10 + off % 3;
}

// FP32 weight fragments (B operands), 64 values each: value of lane l = k 16 + n
// of k-step s. Mirrored taps (26 - off) turn the transposed convolutions of the
// backward pass into the forward ones.
//   F1  (14): off = 2 s + k / 2, c = k % 2, n = output channel
//   F2 (108): off = s / 4, c = 4 (s % 4) + k, n = output channel
//   T2 (108): off = 26 - s / 4, k = output channel 4 (s % 4) + k, n = input channel
//   F3   (8): tile s / 4 of taps n, c = 4 (s % 4) + k
//   T3   (7): off = 26 - (4 s + k), n = channel
constexpr int FR_F1 = 0, FR_F2 = 14, FR_T2 = FR_F2 + 108, FR_F3 = FR_T2 + 108, FR_T3 = FR_F3 + 8;
static_assert((FR_T3 + 7) * 64 == CNN_FRAG, "fragment buffer");

// Weight j into the fragments that hold it (the missing taps stay zero).
__device__ __forceinline__ void frag_store(float* __restrict__ fr, int j, float v) {
  if (j < CNN_NW1) {
    const int o = j / 54, c = (j / 27) % 2, off = j % 27;
    fr[(FR_F1 + off / 2) * 64 + ((off % 2) * 2 + c) * 16 + o] = v;
  } else if (j >= CNN_OW2 && j < CNN_OW2 + CNN_NW2) {
    const int i = j - CNN_OW2, o = i / (CNN_C * 27), c = (i / 27) % CNN_C, off = i % 27;
    fr[(FR_F2 + off * 4 + c / 4) * 64 + (c % 4) * 16 + o] = v;
    fr[(FR_T2 + (26 - off) * 4 + o / 4) * 64 + (o % 4) * 16 + c] = v;
  } else if (j >= CNN_OW3 && j < CNN_OW3 + CNN_NW3) {
    const int i = j - CNN_OW3, c = i / 27, off = i % 27, r = 26 - off;
    fr[(FR_F3 + (off / 16) * 4 + c / 4) * 64 + (c % 4) * 16 + off % 16] = v;
    fr[(FR_T3 + r / 4) * 64 + (r % 4) * 16 + c] = v;
  }
}

__global__ void k_cnn_frag(const float* __restrict__ w, float* __restrict__ fr) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < CNN_NW) frag_store(fr, j, w[j]);
}

// Position of weight j's gradient in an item's gradient: W2 as [off][o][c], the
// order its accumulators are stored in; everything else as the weights.
__device__ __forceinline__ int grad_index(int j) {
  if (j < CNN_OW2 || j >= CNN_OW2 + CNN_NW2) return j;
  const int i = j - CNN_OW2, o = i / (CNN_C * 27), c = (i / 27) % CNN_C, off = i % 27;
  return CNN_OW2 + off * (CNN_C * CNN_C) + o * CNN_C + c;
}
__device__ __forceinline__ int weight_index(int e) {  // its inverse
  if (e < CNN_OW2 || e >= CNN_OW2 + CNN_NW2) return e;
  const int i = e - CNN_OW2, off = i / (CNN_C * CNN_C), o = (i / CNN_C) % CNN_C, c = i % CNN_C;
  return CNN_OW2 + (o * CNN_C + c) * 27 + off;
}

__device__ __forceinline__ float4_t mfma32(float a, float b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc[t] += the 16 -> 16 channel convolution of the padded patches `in` at the
// four cell tiles of this wavefront; base = k TR_CS + the lane's cell of tile 0.
// The fragments of the next three taps are loaded while these are multiplied.
__device__ __forceinline__ void conv16(const float* in, const float* __restrict__ fr, int base,
                                       int l, float4_t (&acc)[4]) {
  float bq[12], bn[12];
#pragma unroll
  for (int s = 0; s < 12; ++s) bq[s] = fr[s * 64 + l];
#pragma unroll 1
  for (int r = 0; r < 9; ++r) {
    const float* nf = fr + (r < 8 ? r + 1 : r) * 12 * 64;
#pragma unroll
    for (int s = 0; s < 12; ++s) bn[s] = nf[s * 64 + l];
    const float* row = in + base + (r / 3) * 100 + (r % 3) * 10;
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
      for (int cg = 0; cg < 4; ++cg)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t] = mfma32(row[4 * cg * TR_CS + 20 * t + dx], bq[dx * 4 + cg], acc[t]);
#pragma unroll
    for (int s = 0; s < 12; ++s) bq[s] = bn[s];
  }
}

// Sum over the 16 lanes-groups of a channel (lane l % 16) within the wavefront.
__device__ __forceinline__ float channel_sum(const float4_t (&v)[4]) {
  float s = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) s += (v[t][0] + v[t][1]) + (v[t][2] + v[t][3]);
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  return s;
}

__device__ __forceinline__ float wave_sum32(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Forward (and, unless EVAL, backward) of one (sample, block) item.
template <bool EVAL>
__global__ __launch_bounds__(TR_T) void k_cnn_train_item(
    int nitems, const int* __restrict__ items, const SampleRef* __restrict__ samples,
    const int* __restrict__ nbr, const float* __restrict__ wg, const float* __restrict__ fr,
    float* __restrict__ gbuf, float* __restrict__ lossbuf, float inv_ntot, float lam) {
  __shared__ __attribute__((aligned(16))) float S[TR_LDS];
  const int it = blockIdx.x;
  if (it >= nitems) return;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int li = l & 15, k = l >> 4;  // MFMA row or column, and k of the A and B operands
  const int b = items[2 * it + 1];
  const SampleRef smp = samples[items[2 * it]];
  float *X = S + TR_X, *H1 = S + TR_H1, *H2 = S + TR_H2, *P = S + TR_P, *D = S + TR_D,
        *OP = S + TR_OP, *RHO = S + TR_RHO, *RED = S + TR_RED;
  const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  // the input patches and the target with its halo; zero rings
  {
    const float inv_sr = 1.0f / smp.s_r, inv_sp = 1.0f / smp.s_p;
    float v[2][3];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = tid + j * TR_T;
      const size_t gi =
          p < PADC ? halo_index(nbr, b, p / 100, (p / 10) % 10, p % 10) : (size_t)b * BLEN;
      v[j][0] = smp.res_h[gi];
      v[j][1] = smp.prev[gi];
      v[j][2] = smp.target[gi];
    }
    for (int i = tid; i < CNN_C * TR_CS / 4; i += TR_T) reinterpret_cast<float4_t*>(H1)[i] = zero4;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = tid + j * TR_T;
      if (p < PADC) {
        X[p] = v[j][0] * inv_sr;
        X[PADC + p] = v[j][1] * inv_sp;
        OP[p] = v[j][2];
        D[p] = 0.f;
      }
    }
  }
  __syncthreads();
  const int cell0 = w * 100 + (li >> 3) * 10 + (li & 7);  // tile 0, padded origin
  // the accumulator rows of this lane: cells 4 k + q of a tile (q consecutive in x)
  const int out0 = (w + 1) * 100 + ((k >> 1) + 1) * 10 + 4 * (k & 1) + 1;  // padded, tile 0
  const int m0 = 64 * w + 4 * k;                                           // unpadded, tile 0
  float4_t z1[4], c1[4], z2[4], c2[4];  // pre-activations and their normal CDF
  // layer 1 (valid)
  {
    const float bias = wg[CNN_OB1 + li];
#pragma unroll
    for (int t = 0; t < 4; ++t) z1[t] = (float4_t){bias, bias, bias, bias};
    const float* x = X + (k & 1) * PADC + cell0;
#pragma unroll
    for (int s = 0; s < 14; ++s) {
      const float bf = fr[(FR_F1 + s) * 64 + l];
      const int o = k >> 1 ? (2 * s + 1 < 27 ? tap(2 * s + 1) : 0) : tap(2 * s);
#pragma unroll
      for (int t = 0; t < 4; ++t) z1[t] = mfma32(x[o + 20 * t], bf, z1[t]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        c1[t][q] = 0.5f * (1.0f + erff(z1[t][q] * 0.70710678118654752f));
        H1[li * TR_CS + out0 + 20 * t + q] = z1[t][q] * c1[t][q];
      }
  }
  __syncthreads();
  // layer 2 (same)
  {
    const float bias = wg[CNN_OB2 + li];
#pragma unroll
    for (int t = 0; t < 4; ++t) z2[t] = (float4_t){bias, bias, bias, bias};
    conv16(H1, fr + FR_F2 * 64, k * TR_CS + cell0, l, z2);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float4_t h;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        c2[t][q] = 0.5f * (1.0f + erff(z2[t][q] * 0.70710678118654752f));
        h[q] = z2[t][q] * c2[t][q];
      }
      *reinterpret_cast<float4_t*>(&H2[li * TR_HS + m0 + 16 * t]) = h;
    }
  }
  __syncthreads();
  // layer 3 (same): tap products, 16 taps at a time, then the shifted sum
  const int z = tid >> 6, y = (tid >> 3) & 7, x = tid & 7, pm = padded(tid);
  float out = wg[CNN_OB3];
#pragma unroll 1
  for (int n2 = 0; n2 < 2; ++n2) {
    float4_t acc[4] = {zero4, zero4, zero4, zero4};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float bf = fr[(FR_F3 + n2 * 4 + s) * 64 + l];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc[t] = mfma32(H2[(4 * s + k) * TR_HS + 64 * w + 16 * t + li], bf, acc[t]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
      *reinterpret_cast<float4_t*>(&P[li * TR_HS + m0 + 16 * t]) = acc[t];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      const int off = 16 * n2 + n;
      if (off >= 27) break;
      const int zz = z + off / 9 - 1, yy = y + (off / 3) % 3 - 1, xx = x + off % 3 - 1;
      if ((unsigned)zz < 8u && (unsigned)yy < 8u && (unsigned)xx < 8u)
        out += P[n * TR_HS + (zz * 8 + yy) * 8 + xx];
    }
    __syncthreads();
  }
  // the loss and its gradient
  const float d = out - OP[pm];
  float lsum = d * d;
  float dout = d * inv_ntot;
  OP[pm] = out;
  __syncthreads();
  if (lam != 0.f) {
    // rho = lap7(out) - q, the stencil closed by the target halo outside
    // the block; its gradient adds lam * (in-block L^T rho) / N to dL/dout
    const float r = ((OP[pm - 1] + OP[pm + 1]) + (OP[pm - 10] + OP[pm + 10]) +
                     (OP[pm - 100] + OP[pm + 100])) - 6.f * OP[pm] - X[pm];
    RHO[tid] = r;
    lsum += lam * r * r;
    __syncthreads();
    float gsum = -6.f * r;
    if (x > 0) gsum += RHO[tid - 1];
    if (x < 7) gsum += RHO[tid + 1];
    if (y > 0) gsum += RHO[tid - 8];
    if (y < 7) gsum += RHO[tid + 8];
    if (z > 0) gsum += RHO[tid - 64];
    if (z < 7) gsum += RHO[tid + 64];
    dout += lam * gsum * inv_ntot;
  }
  D[pm] = dout;
  {
    const float ls = wave_sum32(lsum), ds = wave_sum32(dout);
    if (l == 0) {
      RED[w] = ls;
      RED[16 + w] = ds;
    }
  }
  __syncthreads();  // D and RED complete
  float* G = gbuf + (size_t)it * CNN_NW;
  if (tid < 2 && !(EVAL && tid == 1)) {
    float s = 0.f;
    for (int i = 0; i < 8; ++i) s += RED[16 * tid + i];
    if (tid == 0) lossbuf[it] = s;
    else G[CNN_OB3] = s;
  }
  if (EVAL) return;
  // dW3: taps n of tile w % 2 over the cells of z planes 2 (w / 2), + 1
  float4_t a3 = zero4;
  {
    const int off = 16 * (w & 1) + li;
    const float* dp = D + (off < 27 ? tap(26 - off) : 0) + k;
    const float* hp = H2 + li * TR_HS + k;
#pragma unroll 4
    for (int s = 0; s < 32; ++s) {  // four cells of a row
      const int row = 16 * (w >> 1) + (s >> 1), xh = 4 * (s & 1);
      a3 = mfma32(hp[row * 8 + xh], dp[(row >> 3) * 100 + (row & 7) * 10 + xh], a3);
    }
    *reinterpret_cast<float4_t*>(&P[w * 256 + 4 * l]) = a3;
  }
  // dZ2 = (W3^T * D) . gelu'(Z2)
  float4_t g2[4] = {zero4, zero4, zero4, zero4};
#pragma unroll
  for (int s = 0; s < 7; ++s) {
    const int off = 4 * s + k;
    const float bf = fr[(FR_T3 + s) * 64 + l];
    const float* dp = D + cell0 + (off < 27 ? tap(off) : 0);
#pragma unroll
    for (int t = 0; t < 4; ++t) g2[t] = mfma32(dp[20 * t], bf, g2[t]);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v = z2[t][q];
      g2[t][q] *= c2[t][q] + v * expf(-0.5f * v * v) * 0.3989422804014327f;
    }
  const float s2 = channel_sum(g2);
  __syncthreads();  // the dW3 partials; H2 and RED read by all
  {
    // partial sums of dW3 in the order of the z planes
    const int n2 = tid >> 8, e = tid & 255, c = 4 * (e >> 6) + (e & 3), off = 16 * n2 + ((e >> 2) & 15);
    const float v = ((P[n2 * 256 + e] + P[(n2 + 2) * 256 + e]) + P[(n2 + 4) * 256 + e]) +
                    P[(n2 + 6) * 256 + e];
    if (off < 27) G[CNN_OW3 + c * 27 + off] = v;
    if (l < 16) RED[w * 16 + l] = s2;
  }
  __syncthreads();  // P and H2 free
  float* Z = H2;  // dZ2 on the padded patch
  for (int i = tid; i < CNN_C * TR_CS / 4; i += TR_T) reinterpret_cast<float4_t*>(Z)[i] = zero4;
  if (tid < CNN_C) {
    float s = 0.f;
    for (int i = 0; i < 8; ++i) s += RED[i * 16 + tid];
    G[CNN_OB2 + tid] = s;
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) Z[li * TR_CS + out0 + 20 * t + q] = g2[t][q];
  __syncthreads();
  // dW2: taps w, w + 8, w + 16 (and 24 + w for w < 3), all cells
  {
    float4_t acc[4] = {zero4, zero4, zero4, zero4};
    const float* zp = Z + li * TR_CS + 111 + k;
    const float* hp = H1 + li * TR_CS + k;
    const int o0 = tap(w), o1 = tap(w + 8), o2 = tap(w + 16), o3 = tap(w < 3 ? w + 24 : w);
#pragma unroll 2
    for (int row = 0; row < 64; ++row) {
      const int r = (row >> 3) * 100 + (row & 7) * 10;
#pragma unroll
      for (int xh = 0; xh < 8; xh += 4) {
        const float a = zp[r + xh];
        acc[0] = mfma32(a, hp[r + xh + o0], acc[0]);
        acc[1] = mfma32(a, hp[r + xh + o1], acc[1]);
        acc[2] = mfma32(a, hp[r + xh + o2], acc[2]);
        if (w < 3) acc[3] = mfma32(a, hp[r + xh + o3], acc[3]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < 3 || w < 3)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          G[CNN_OW2 + (w + 8 * j) * 256 + (4 * k + q) * 16 + li] = acc[j][q];
  }
  // dZ1 = (W2^T * dZ2) . gelu'(Z1)
  float4_t g1[4] = {zero4, zero4, zero4, zero4};
  conv16(Z, fr + FR_T2 * 64, k * TR_CS + cell0, l, g1);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v = z1[t][q];
      g1[t][q] *= c1[t][q] + v * expf(-0.5f * v * v) * 0.3989422804014327f;
    }
  const float s1 = channel_sum(g1);
  __syncthreads();  // H1, Z and RED read by all
#pragma unroll
  for (int t = 0; t < 4; ++t) *reinterpret_cast<float4_t*>(&H1[li * TR_HS + m0 + 16 * t]) = g1[t];
  if (l < 16) RED[w * 16 + l] = s1;
  __syncthreads();
  if (tid < CNN_C) {
    float s = 0.f;
    for (int i = 0; i < 8; ++i) s += RED[i * 16 + tid];
    G[CNN_OB1 + tid] = s;
  }
  // dW1: (channel, tap) pairs n of tile w % 4 over z planes 4 (w / 4) .. + 3
  {
    const int pr = 16 * (w & 3) + li;
    const float* xp = X + (pr < 54 ? (pr / 27) * PADC + tap(pr % 27) : 0) + k;
    const float* hp = H1 + li * TR_HS + k;
    float4_t acc = zero4;
#pragma unroll 4
    for (int s = 0; s < 64; ++s) {
      const int row = 32 * (w >> 2) + (s >> 1), xh = 4 * (s & 1);
      acc = mfma32(hp[row * 8 + xh], xp[(row >> 3) * 100 + (row & 7) * 10 + xh], acc);
    }
    *reinterpret_cast<float4_t*>(&Z[w * 256 + 4 * l]) = acc;
  }
  __syncthreads();
  for (int i = tid; i < 1024; i += TR_T) {
    const int n4 = i >> 8, e = i & 255, o = 4 * (e >> 6) + (e & 3), pr = 16 * n4 + ((e >> 2) & 15);
    if (pr < 54) G[o * 54 + pr] = Z[n4 * 256 + e] + Z[(n4 + 4) * 256 + e];
  }
}

// Sum the per-item gradients and take one Adam step (Kingma & Ba 2015; beta1 =
// 0.9, beta2 = 0.999, eps = 1e-8). 64 weights a workgroup, the items split in
// AD_G contiguous groups that are added in order: the sum reads nitems x 33 KB
// once, with enough loads in flight (256 items: 4.8 us against 64 us for one
// thread per weight over all items).
constexpr int AD_G = 16;
__global__ __launch_bounds__(64 * AD_G) void k_cnn_adam(int nitems, const float* __restrict__ gbuf,
                                                        float* __restrict__ w,
                                                        float* __restrict__ fr,
                                                        float* __restrict__ mv, float lr,
                                                        float bc1, float bc2) {
  __shared__ float part[AD_G][64];
  const int e = blockIdx.x * 64 + (threadIdx.x & 63), grp = threadIdx.x >> 6;
  const int per = (nitems + AD_G - 1) / AD_G;
  const int i0 = grp * per, i1 = min(nitems, i0 + per);
  float s = 0.f;
  if (e < CNN_NW) {
#pragma unroll 8
    for (int i = i0; i < i1; ++i) s += gbuf[(size_t)i * CNN_NW + e];
  }
  part[grp][threadIdx.x & 63] = s;
  __syncthreads();
  if (grp != 0 || e >= CNN_NW) return;
  float g = 0.f;
#pragma unroll
  for (int i = 0; i < AD_G; ++i) g += part[i][threadIdx.x];
  const int j = weight_index(e);
  float m = mv[j], v = mv[CNN_NW + j];
  m = 0.9f * m + 0.1f * g;
  v = 0.999f * v + 0.001f * g * g;
  mv[j] = m;
  mv[CNN_NW + j] = v;
  const float wj = w[j] - lr * (m / bc1) / (sqrtf(v / bc2) + 1e-8f);
  w[j] = wj;
  frag_store(fr, j, wj);
}

// Training-set entry: res / h_b, p_prev and (p - p_prev - m) / s_r in FP32,
// m the volume-weighted mean of p - p_prev (scal[2]): a constant shift of the
// pressure is invisible to the operator and to the inputs, so it is not a
// target.
__global__ void k_cnn_sample(long long n, const double* __restrict__ res,
                             const double* __restrict__ prev, const double* __restrict__ p,
                             const double* __restrict__ h, const double* __restrict__ scal,
                             float* __restrict__ rh, float* __restrict__ pv,
                             float* __restrict__ tg) {
  const double inv_s = 1.0 / scal[0], m = scal[2];
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    rh[i] = (float)(res[i] / h[i / BLEN]);
    pv[i] = (float)prev[i];
    tg[i] = (float)((p[i] - prev[i] - m) * inv_s);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
#define CCHECK(expr)                                            \
  do {                                                          \
    hipError_t e_ = (expr);                                     \
    if (e_ != hipSuccess) {                                     \
      err = std::string(#expr) + ": " + hipGetErrorString(e_);  \
      return -1;                                                \
    }                                                           \
  } while (0)

int cnn_num_weights() { return CNN_NW; }

int cnn_init(CnnState& C, std::string& err) {
  CCHECK(hipMalloc(&C.d_w, CNN_NW * sizeof(float)));
  CCHECK(hipMalloc(&C.d_adam, 2 * CNN_NW * sizeof(float)));
  CCHECK(hipMalloc(&C.d_wpk, CNN_PK * sizeof(_Float16)));
  CCHECK(hipMalloc(&C.d_frag, CNN_FRAG * sizeof(float)));
  CCHECK(hipMalloc(&C.d_scal, 8 * sizeof(double)));
  CCHECK(hipMemset(C.d_w, 0, CNN_NW * sizeof(float)));
  CCHECK(hipMemset(C.d_adam, 0, 2 * CNN_NW * sizeof(float)));
  CCHECK(hipMemset(C.d_frag, 0, CNN_FRAG * sizeof(float)));  // the missing taps stay zero
  return 0;
}

int cnn_set_topology(CnnState& C, int nb, const int* d_nbr, const double* d_h, std::string& err) {
  cnn_clear_samples(C);
  C.nb = nb;
  C.n = (long long)nb * BLEN;
  C.d_nbr = d_nbr;
  C.d_h = d_h;
  if (nb <= C.cap_nb && C.d_part && C.d_pred) return 0;  // the buffers grow only
  if (C.d_part) (void)hipFree(C.d_part);
  if (C.d_pred) (void)hipFree(C.d_pred);
  C.d_part = nullptr;
  C.d_pred = nullptr;
  C.cap_nb = 0;
  // partial sums: up to 2 per workgroup of 4 blocks
  CCHECK(hipMalloc(&C.d_part, (2 * ((nb + 3) / 4) + 16) * sizeof(double)));
  CCHECK(hipMalloc(&C.d_pred, C.n * sizeof(double)));
  C.cap_nb = nb;
  return 0;
}

static int repack(CnnState& C, hipStream_t s, std::string& err) {
  k_cnn_pack<<<(CNN_PK + 255) / 256, 256, 0, s>>>(C.d_w, static_cast<_Float16*>(C.d_wpk));
  CCHECK(hipGetLastError());
  return 0;
}

int cnn_set_weights(CnnState& C, const float* w, int nw, std::string& err) {
  if (nw != CNN_NW || !w) {
    err = "cnn_set_weights: expected " + std::to_string(CNN_NW) + " weights";
    return -1;
  }
  CCHECK(hipMemcpy(C.d_w, w, CNN_NW * sizeof(float), hipMemcpyHostToDevice));
  CCHECK(hipMemset(C.d_adam, 0, 2 * CNN_NW * sizeof(float)));
  C.adam_t = 0;
  if (repack(C, nullptr, err)) return -1;
  k_cnn_frag<<<(CNN_NW + 255) / 256, 256>>>(C.d_w, C.d_frag);
  CCHECK(hipGetLastError());
  CCHECK(hipDeviceSynchronize());
  C.have_weights = true;
  return 0;
}

int cnn_get_weights(CnnState& C, float* w, int nw, std::string& err) {
  if (nw != CNN_NW || !w) {
    err = "cnn_get_weights: expected " + std::to_string(CNN_NW) + " weights";
    return -1;
  }
  CCHECK(hipDeviceSynchronize());
  CCHECK(hipMemcpy(w, C.d_w, CNN_NW * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

// scal[0] = s_r = RMS(res / h_b), scal[1] = s_p = RMS(p_prev)
static int scales(CnnState& C, hipStream_t s, const double* res, const double* prev,
                  std::string& err) {
  const int nwg = (int)((C.n + 4 * BLEN - 1) / (4 * BLEN));
  k_cnn_rms<<<nwg, WG_THREADS, 0, s>>>(C.n, res, C.d_h, C.d_part);
  k_cnn_rms_fin<<<1, WG_THREADS, 0, s>>>(C.n, C.d_scal, 0, C.d_part, nwg);
  k_cnn_rms<<<nwg, WG_THREADS, 0, s>>>(C.n, prev, nullptr, C.d_part);
  k_cnn_rms_fin<<<1, WG_THREADS, 0, s>>>(C.n, C.d_scal, 1, C.d_part, nwg);
  CCHECK(hipGetLastError());
  return 0;
}

int cnn_predict(CnnState& C, hipStream_t s, const double* d_res, const double* d_prev,
                double* d_out, std::string& err, const double* sums) {
  if (!C.have_weights) {
    err = "cnn_predict: no weights (set or train them first)";
    return -1;
  }
  if (sums) k_cnn_scales_fin<<<1, WG_THREADS, 0, s>>>(C.n, C.d_scal, sums, (C.nb + 3) / 4);
  else if (scales(C, s, d_res, d_prev, err)) return -1;
  k_cnn_infer<<<C.nb, WG_THREADS, 0, s>>>(C.nb, C.d_nbr, C.d_h, d_res, d_prev, C.d_scal,
                                          static_cast<const _Float16*>(C.d_wpk), C.d_w, d_out);
  CCHECK(hipGetLastError());
  CCHECK(hipStreamSynchronize(s));
  return 0;
}

int cnn_add_sample(CnnState& C, hipStream_t s, const double* d_res, const double* d_prev,
                   const double* d_p, std::string& err) {
  if (C.nb <= 0) {
    err = "cnn_add_sample: no topology";
    return -1;
  }
  CnnSample S;
  CCHECK(hipMalloc(&S.res_h, 3 * C.n * sizeof(float)));
  S.prev = S.res_h + C.n;
  S.target = S.prev + C.n;
  if (scales(C, s, d_res, d_prev, err)) return -1;
  const int nwg = (int)((C.n + 4 * BLEN - 1) / (4 * BLEN));
  k_cnn_dmean<<<nwg, WG_THREADS, 0, s>>>(C.n, d_p, d_prev, C.d_h, C.d_part);
  k_cnn_dmean_fin<<<1, WG_THREADS, 0, s>>>(C.d_scal, C.d_part, nwg);
  k_cnn_sample<<<4096, 256, 0, s>>>(C.n, d_res, d_prev, d_p, C.d_h, C.d_scal, S.res_h, S.prev,
                                    S.target);
  CCHECK(hipGetLastError());
  double sc[2] = {1.0, 1.0};
  CCHECK(hipMemcpyAsync(sc, C.d_scal, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
  CCHECK(hipStreamSynchronize(s));
  S.s_r = (float)sc[0];
  S.s_p = (float)sc[1];
  C.samples.push_back(S);
  return 0;
}

void cnn_clear_samples(CnnState& C) {
  for (auto& S : C.samples) (void)hipFree(S.res_h);
  C.samples.clear();
}

// Gradients and losses of nitems items (losses twice: a call's first and its
// latest step), and nlist entries of the item list; the buffers grow only.
static int ensure_train_buffers(CnnState& C, int nitems, int nlist, std::string& err) {
  const long long need = (long long)nitems * (CNN_NW + 2);
  if (need > C.scratch_cap) {
    if (C.d_scratch) (void)hipFree(C.d_scratch);
    C.d_scratch = nullptr;
    C.scratch_cap = 0;
    CCHECK(hipMalloc(&C.d_scratch, need * sizeof(float)));
    C.scratch_cap = need;
  }
  if (nlist > C.items_cap) {
    if (C.d_items) (void)hipFree(C.d_items);
    C.d_items = nullptr;
    C.items_cap = 0;
    CCHECK(hipMalloc(&C.d_items, 2 * (size_t)nlist * sizeof(int)));
    C.items_cap = nlist;
  }
  return 0;
}

static int upload_samples(CnnState& C, std::string& err) {
  std::vector<SampleRef> refs(C.samples.size());
  for (size_t k = 0; k < C.samples.size(); ++k)
    refs[k] = {C.samples[k].res_h, C.samples[k].prev, C.samples[k].target, C.samples[k].s_r,
               C.samples[k].s_p};
  if (refs.size() > C.refs_cap) {
    if (C.d_refs) (void)hipFree(C.d_refs);
    C.d_refs = nullptr;
    C.refs_cap = 0;
    CCHECK(hipMalloc(&C.d_refs, refs.size() * sizeof(SampleRef)));
    C.refs_cap = refs.size();
  }
  CCHECK(hipMemcpy(C.d_refs, refs.data(), refs.size() * sizeof(SampleRef), hipMemcpyHostToDevice));
  return 0;
}

int cnn_train(CnnState& C, hipStream_t s, int steps, int batch, float lr, float res_weight,
              uint64_t seed, double* loss, std::string& err) {
  if (C.samples.empty()) {
    err = "cnn_train: empty training set";
    return -1;
  }
  if (steps <= 0 || batch <= 0 || batch > 65536 || !(res_weight >= 0.f)) {
    err = "cnn_train: bad steps/batch/res_weight";
    return -1;
  }
  C.res_weight = res_weight;
  if (!C.have_weights) {  // He-style initialisation from the seed
    std::mt19937_64 R(seed ^ 0x5eedULL);
    std::vector<float> w(CNN_NW, 0.f);
    auto fill = [&](int off, int n, int fan_in) {
      const double sd = std::sqrt(2.0 / fan_in);
      for (int i = 0; i < n; ++i) {
        const double u1 = (double((R() >> 11) + 1)) * (1.0 / 9007199254740993.0);
        const double u2 = double(R() >> 11) * (1.0 / 9007199254740992.0);
        w[off + i] = (float)(sd * std::sqrt(-2.0 * std::log(u1)) * std::cos(2 * M_PI * u2));
      }
    };
    fill(0, CNN_NW1, 2 * 27);
    fill(CNN_OW2, CNN_NW2, CNN_C * 27);
    fill(CNN_OW3, CNN_NW3, CNN_C * 27);
    for (int i = CNN_OW3; i < CNN_OW3 + CNN_NW3; ++i) w[i] *= 0.1f;  // start near p_prev
    if (cnn_set_weights(C, w.data(), CNN_NW, err)) return -1;
  }
  // the items of up to TRAIN_LIST / batch steps are drawn and uploaded at a time
  constexpr int TRAIN_LIST = 1 << 14;
  const int chunk = std::min(steps, std::max(1, TRAIN_LIST / batch));
  if (ensure_train_buffers(C, batch, chunk * batch, err)) return -1;
  if (upload_samples(C, err)) return -1;
  const SampleRef* refs = static_cast<const SampleRef*>(C.d_refs);
  float* gbuf = C.d_scratch;
  float* lbuf = gbuf + (size_t)batch * CNN_NW;  // [0, batch): first step, then the others
  std::vector<int> items(2 * (size_t)chunk * batch);
  std::mt19937_64 R(seed);
  const int ns = (int)C.samples.size();
  const float inv_ntot = 1.0f / (float)((double)batch * BLEN);
  for (int step = 0; step < steps; ++step) {
    if (step % chunk == 0) {
      if (step > 0) CCHECK(hipStreamSynchronize(s));  // the list's last upload is done
      const int m = std::min(chunk, steps - step) * batch;
      for (int i = 0; i < m; ++i) {
        items[2 * i] = (int)(R() % (uint64_t)ns);
        items[2 * i + 1] = (int)(R() % (uint64_t)C.nb);
      }
      CCHECK(hipMemcpyAsync(C.d_items, items.data(), 2 * (size_t)m * sizeof(int),
                            hipMemcpyHostToDevice, s));
    }
    k_cnn_train_item<false><<<batch, TR_T, 0, s>>>(
        batch, C.d_items + 2 * (size_t)(step % chunk) * batch, refs, C.d_nbr, C.d_w, C.d_frag,
        gbuf, lbuf + (step > 0 ? batch : 0), inv_ntot, C.res_weight);
    C.adam_t += 1;
    const float bc1 = 1.0f - std::pow(0.9f, (float)C.adam_t);
    const float bc2 = 1.0f - std::pow(0.999f, (float)C.adam_t);
    k_cnn_adam<<<(CNN_NW + 63) / 64, 64 * AD_G, 0, s>>>(batch, gbuf, C.d_w, C.d_frag, C.d_adam, lr,
                                                        bc1, bc2);
  }
  CCHECK(hipGetLastError());
  if (repack(C, s, err)) return -1;
  std::vector<float> lh(2 * (size_t)batch);
  CCHECK(hipMemcpyAsync(lh.data(), lbuf, lh.size() * sizeof(float), hipMemcpyDeviceToHost, s));
  CCHECK(hipStreamSynchronize(s));
  if (loss) {
    for (int k = 0; k < 2; ++k) {
      const float* f = lh.data() + (k && steps > 1 ? batch : 0);
      double L = 0;
      for (int i = 0; i < batch; ++i) L += f[i];
      loss[k] = L * (0.5 / ((double)batch * BLEN));
    }
  }
  return 0;
}

int cnn_eval(CnnState& C, hipStream_t s, int k, double* loss, std::string& err) {
  if (k < 0 || k >= (int)C.samples.size()) {
    err = "cnn_eval: no such sample";
    return -1;
  }
  const int chunk = std::min(C.nb, 2048);
  if (ensure_train_buffers(C, chunk, chunk, err)) return -1;
  if (upload_samples(C, err)) return -1;
  const SampleRef* refs = static_cast<const SampleRef*>(C.d_refs);
  float* gbuf = C.d_scratch;
  float* lbuf = gbuf + (size_t)chunk * CNN_NW;
  std::vector<int> items(2 * chunk);
  std::vector<float> lh(chunk);
  double L = 0;
  for (int b0 = 0; b0 < C.nb; b0 += chunk) {
    const int m = std::min(chunk, C.nb - b0);
    for (int i = 0; i < m; ++i) {
      items[2 * i] = k;
      items[2 * i + 1] = b0 + i;
    }
    CCHECK(hipMemcpyAsync(C.d_items, items.data(), 2 * m * sizeof(int), hipMemcpyHostToDevice, s));
    k_cnn_train_item<true><<<m, TR_T, 0, s>>>(m, C.d_items, refs, C.d_nbr, C.d_w, C.d_frag, gbuf,
                                              lbuf, 0.f, C.res_weight);
    CCHECK(hipGetLastError());
    CCHECK(hipMemcpyAsync(lh.data(), lbuf, m * sizeof(float), hipMemcpyDeviceToHost, s));
    CCHECK(hipStreamSynchronize(s));
    for (int i = 0; i < m; ++i) L += lh[i];
  }
  *loss = 0.5 * L / ((double)C.nb * BLEN);
  return 0;
}

__global__ void k_cnn_sum_grads(int nitems, const float* __restrict__ gbuf, float* __restrict__ g) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= CNN_NW) return;
  float a = 0.f;
  for (int i = 0; i < nitems; ++i) a += gbuf[(size_t)i * CNN_NW + grad_index(j)];
  g[j] = a;
}

int cnn_gradient(CnnState& C, hipStream_t s, int k, float res_weight, float* grad, double* loss,
                 std::string& err) {
  if (k < 0 || k >= (int)C.samples.size()) {
    err = "cnn_gradient: no such sample";
    return -1;
  }
  if (!C.have_weights) {
    err = "cnn_gradient: no weights";
    return -1;
  }
  if (C.nb > 4096) {
    err = "cnn_gradient: grid too large for a full-batch gradient";
    return -1;
  }
  const int m = C.nb;
  if (ensure_train_buffers(C, m + 1, m, err)) return -1;
  if (upload_samples(C, err)) return -1;
  float* gbuf = C.d_scratch;
  float* gsum = gbuf + (size_t)m * CNN_NW;
  float* lbuf = gsum + CNN_NW;
  std::vector<int> items(2 * m);
  for (int i = 0; i < m; ++i) {
    items[2 * i] = k;
    items[2 * i + 1] = i;
  }
  CCHECK(hipMemcpyAsync(C.d_items, items.data(), 2 * m * sizeof(int), hipMemcpyHostToDevice, s));
  k_cnn_train_item<false><<<m, TR_T, 0, s>>>(m, C.d_items,
                                             static_cast<const SampleRef*>(C.d_refs), C.d_nbr,
                                             C.d_w, C.d_frag, gbuf, lbuf,
                                             1.0f / ((float)m * BLEN), res_weight);
  k_cnn_sum_grads<<<(CNN_NW + 255) / 256, 256, 0, s>>>(m, gbuf, gsum);
  std::vector<float> lh(m);
  CCHECK(hipMemcpyAsync(grad, gsum, CNN_NW * sizeof(float), hipMemcpyDeviceToHost, s));
  CCHECK(hipMemcpyAsync(lh.data(), lbuf, m * sizeof(float), hipMemcpyDeviceToHost, s));
  CCHECK(hipGetLastError());
  CCHECK(hipStreamSynchronize(s));
  double L = 0;
  for (float v : lh) L += v;
  *loss = 0.5 * L / ((double)m * BLEN);
  return 0;
}

void cnn_free(CnnState& C) {
  cnn_clear_samples(C);
  (void)hipFree(C.d_w);
  (void)hipFree(C.d_adam);
  (void)hipFree(C.d_wpk);
  (void)hipFree(C.d_scal);
  if (C.d_part) (void)hipFree(C.d_part);
  if (C.d_pred) (void)hipFree(C.d_pred);
  if (C.d_scratch) (void)hipFree(C.d_scratch);
  if (C.d_items) (void)hipFree(C.d_items);
  if (C.d_refs) (void)hipFree(C.d_refs);
  (void)hipFree(C.d_frag);
  C = CnnState();
}

}  // namespace cup3d
