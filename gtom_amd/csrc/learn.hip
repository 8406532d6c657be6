// The learned orientation-proposal network: a small 3D CNN over 32^3 tiles of
// a tomogram block that scores 500 coarse directions (the Fibonacci-sphere
// directions of the search's orientation set) and one "no peak" class, trained
// on the exhaustive search's own argmax labels. The search then runs only the
// shortlisted directions' orientations on each tile (pick.hip, tile masks).
// There is no counterpart in the reference; its labels are the argmax
// orientation of UpdateCorrelationKernel (src/Correlation/SubTomograms.cu:138-158)
// divided by the 18 in-plane steps of a direction.
//
// Network (channels-last bf16 activations, bf16 weights, fp32 accumulation):
//   x (32^3 x 1) -> conv1 3^3 (1->16) + ReLU -> avgpool 2 -> conv2 (16->16) + ReLU
//   -> avgpool 2 -> conv3 (16->16) + ReLU -> conv4 (16->16) + ReLU -> avgpool 2
//   -> 1024 features (4^3 x 16) -> linear 1024 -> 501 logits.
// Every convolution, its data gradient and its weight gradient is an implicit
// GEMM on the matrix cores (v_mfma_f32_16x16x32_bf16): forward and data
// gradient with M = 16 voxels, N = 16 output channels, K = 2 taps x 16 input
// channels per instruction (14 instructions for the 27 taps, the last half
// zero); weight gradient with M = 16 output channels, N = 16 input channels (or
// 16 taps for the one-channel input), K = 32 voxels. The head is a generic
// strided bf16 GEMM on the same instruction. Parameters are fp32 masters with
// bf16 working copies refreshed after every Adam step.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "runtime.hpp"

namespace gx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

constexpr int PT = 32;    // tile side
constexpr int PC = 16;    // channels
constexpr int NDIR = 500;
constexpr int NCLS = 501; // + "no peak"
constexpr int CPAD = 512; // padded class count
constexpr int NFEAT = 1024;
constexpr int NTAP = 27;

// Parameter layout of the fp32 master array (and of the gradients).
constexpr int OFF_W1 = 0;                        // [16 co][27 taps]
constexpr int OFF_B1 = OFF_W1 + PC * NTAP;       // [16]
constexpr int OFF_W2 = OFF_B1 + PC;              // [27 taps][16 co][16 ci]
constexpr int OFF_B2 = OFF_W2 + NTAP * PC * PC;
constexpr int OFF_W3 = OFF_B2 + PC;
constexpr int OFF_B3 = OFF_W3 + NTAP * PC * PC;
constexpr int OFF_W4 = OFF_B3 + PC;
constexpr int OFF_B4 = OFF_W4 + NTAP * PC * PC;
constexpr int OFF_WF = OFF_B4 + PC;              // [501][1024]
constexpr int OFF_BF = OFF_WF + NCLS * NFEAT;    // [501]
constexpr int NPARAM = OFF_BF + NCLS;

__device__ __forceinline__ u16 f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
  return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((unsigned)h << 16); }
__device__ __forceinline__ bool bf_pos(u16 h) { return (h & 0x8000u) == 0 && (h & 0x7fffu) != 0; }

__device__ __forceinline__ f32x4 mfma(u16x8 a, u16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
__device__ __forceinline__ u16x8 load8(const u16* p) { return *reinterpret_cast<const u16x8*>(p); }

// Tap t in [0, 27): offset (t/9 - 1, (t/3)%3 - 1, t%3 - 1) in (z, y, x); tap 26 - t is its negation.
__device__ __forceinline__ bool tap_src(int t, int S, int z, int y, int x, int& v) {
  const int zz = z + t / 9 - 1, yy = y + (t / 3) % 3 - 1, xx = x + t % 3 - 1;
  v = (zz * S + yy) * S + xx;
  return (unsigned)zz < (unsigned)S && (unsigned)yy < (unsigned)S && (unsigned)xx < (unsigned)S;
}

// ---------------------------------------------------------------------------
// The first layer (1 -> 16 channels at 32^3) never keeps its activation, which is
// 16 times its input and was most of a training pass's traffic (268 MB of the 256
// tiles, written once and read three times): the forward pass pools it in the
// kernel that makes it and leaves one bit per value, whether it is positive
// (16 bits per voxel), and the weight gradient expands the pooled gradient from
// those bits as it goes. 256 tiles: convolution 191 + pooling 56 us, expansion
// 304 + gradient 331 us as separate passes.
//
// A workgroup stages input planes with a zero halo in LDS: rows of HX values, the
// voxel (z, y, x) of the slab's first plane z0 at ((z - z0 + 1) * HY + y + 1) * HX + x + 1.
// ---------------------------------------------------------------------------
constexpr int HY = PT + 2, HX = PT + 2;

__device__ __forceinline__ void stage_slab(const u16* __restrict__ tin, int z0, int planes, u16* slab) {
  // planes z0 - 1 .. z0 + planes; two values at a time (rows of 32 start at odd places: 16-bit stores)
  for (int k = threadIdx.x; k < (planes + 2) * HY * HX; k += 256) {
    const int x = k % HX - 1, y = (k / HX) % HY - 1, z = z0 - 1 + k / (HY * HX);
    const bool in = (unsigned)x < (unsigned)PT && (unsigned)y < (unsigned)PT && (unsigned)z < (unsigned)PT;
    slab[k] = in ? tin[(z * PT + y) * PT + x] : (u16)0;
  }
}

// conv1 + bias + ReLU (rounded to bf16), its positive bits, and the 2^3 average of
// the rounded values. One workgroup per (tile, pooled plane); one wave per 16
// voxels of the four rows under 8 pooled ones, which lie in one lane: D's rows are
// 4 consecutive voxels.
__global__ __launch_bounds__(256) void k_conv1_pool(const u16* __restrict__ in, const u16* __restrict__ wb,
                                                    const float* __restrict__ bias, u16* __restrict__ bits,
                                                    u16* __restrict__ out) {
  constexpr int H = PT / 2, V = PT * PT * PT;
  __shared__ u16 slab[4 * HY * HX];
  const int tile = blockIdx.x / H, zp = blockIdx.x % H;
  stage_slab(in + (size_t)tile * V, 2 * zp, 2, slab);
  __syncthreads();
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const u16x8 w = load8(wb + i * 32 + 8 * g);
  const float bb = bias[i];
  int off[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int t = 8 * g + e, tt = t < NTAP ? t : 0;  // taps past 26 have zero weights
    off[e] = (tt / 9 * HY + (tt / 3) % 3) * HX + tt % 3;
  }
  for (int k = threadIdx.x >> 6; k < 2 * H; k += 4) {
    const int yp = k >> 1, x0 = 16 * (k & 1);
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int dz = r >> 1, y = 2 * yp + (r & 1);
      const u16* src = slab + (dz * HY + y) * HX + x0 + i;
      u16x8 a;
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = src[off[e]];
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = mfma(a, w, acc);
      u16 mine = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const u16 q = f2bf(fmaxf(acc[e] + bb, 0.f));
        sum[e >> 1] += bf2f(q);
        const unsigned long long pos = __ballot(bf_pos(q));
        if (i == e) mine = (u16)(pos >> (16 * g));
      }
      if (i < 4) bits[(size_t)tile * V + ((2 * zp + dz) * PT + y) * PT + x0 + 4 * g + i] = mine;
    }
    const size_t o = (((size_t)tile * H + zp) * H + yp) * H + x0 / 2 + 2 * g;
    out[o * PC + i] = f2bf(sum[0] * 0.125f);
    out[(o + 1) * PC + i] = f2bf(sum[1] * 0.125f);
  }
}

// ---------------------------------------------------------------------------
// Convolution (3^3, zero padding) of 16 channels, forward or data gradient. One
// wave: VG groups of 16 consecutive voxels of one tile x 16 output channels, with
// each tap pair's weights loaded once for all. out = (acc + bias), ReLU if relu,
// zeroed where mask (a post-ReLU activation) is not positive.
// wb: [27][16 out][16 in] bf16.
// ---------------------------------------------------------------------------
constexpr int VG = 4;

template <int S>
__global__ __launch_bounds__(256) void k_conv(const u16* __restrict__ in, const u16* __restrict__ wb,
                                              const float* __restrict__ bias, const u16* __restrict__ mask,
                                              u16* __restrict__ out, int ntiles, int relu) {
  constexpr int V = S * S * S, WPT = V / (16 * VG);
  const int lane = threadIdx.x & 63;
  const long wave = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wave >= (long)ntiles * WPT) return;
  const int tile = (int)(wave / WPT), v0 = (int)(wave % WPT) * 16 * VG;
  const int i = lane & 15, g = lane >> 4;
  const u16* tin = in + (size_t)tile * V * PC;
  const int ci0 = 8 * (g & 1);
  f32x4 acc[VG];
#pragma unroll
  for (int q = 0; q < VG; ++q) acc[q] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < 14; ++p) {
    const int t = 2 * p + (g >> 1);
    u16x8 b = {0, 0, 0, 0, 0, 0, 0, 0};
    if (t < NTAP) b = load8(wb + (t * PC + i) * PC + ci0);
#pragma unroll
    for (int q = 0; q < VG; ++q) {
      const int v = v0 + 16 * q + i, x = v % S, y = (v / S) % S, z = v / (S * S);
      u16x8 a = {0, 0, 0, 0, 0, 0, 0, 0};
      int src;
      if (t < NTAP && tap_src(t, S, z, y, x, src)) a = load8(tin + (size_t)src * PC + ci0);
      acc[q] = mfma(a, b, acc[q]);
    }
  }
  const int co = i;
  const float bb = bias ? bias[co] : 0.f;
#pragma unroll
  for (int q = 0; q < VG; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const size_t o = ((size_t)tile * V + v0 + 16 * q + 4 * g + e) * PC + co;
      float val = acc[q][e] + bb;
      if (relu) val = fmaxf(val, 0.f);
      if (mask && !bf_pos(mask[o])) val = 0.f;
      out[o] = f2bf(val);
    }
}

// ---------------------------------------------------------------------------
// Weight gradients: dW[t][co][ci] = sum_v dz[v][co] * in[v + off_t][ci], and the
// bias gradient sum_v dz[v][co]; M = co, N = ci (or taps), K = 32 voxels. A
// workgroup sums its waves' results and writes one set of partials (27 * 256
// weights, or [16 co][27], then 16 biases), which k_reduce_parts adds.
// ---------------------------------------------------------------------------
template <int CIN> constexpr int dw_part_len() { return CIN == 1 ? PC * NTAP + PC : NTAP * PC * PC + PC; }

// The input of a 16-channel weight gradient, channels first with a zero halo:
// xt[tile][ci][S+2][S+2][S+2]. B's operand is 8 voxels along x of one channel at
// each of 27 shifts: with this layout one 16-byte load without bounds checks, where
// the channels-last one takes 8 checked 2-byte loads (571 us of 256 tiles at 16^3).
template <int S>
__global__ __launch_bounds__(256) void k_halo_channels(const u16* __restrict__ in, u16* __restrict__ xt, int ntiles) {
  constexpr int P = S + 2, VP = P * P * P, V = S * S * S;
  const long total = (long)ntiles * VP;
  for (long id = blockIdx.x * 256L + threadIdx.x; id < total; id += (long)gridDim.x * 256) {
    const int tile = (int)(id / VP), r = (int)(id % VP);
    const int x = r % P - 1, y = (r / P) % P - 1, z = r / (P * P) - 1;
    u16x8 lo = {0, 0, 0, 0, 0, 0, 0, 0}, hi = lo;
    if ((unsigned)x < (unsigned)S && (unsigned)y < (unsigned)S && (unsigned)z < (unsigned)S) {
      const u16* p = in + ((size_t)tile * V + (z * S + y) * S + x) * PC;
      lo = load8(p);
      hi = load8(p + 8);
    }
    u16* o = xt + (size_t)tile * PC * VP + r;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      o[(size_t)c * VP] = lo[c];
      o[(size_t)(c + 8) * VP] = hi[c];
    }
  }
}

// 8 values at any 2-byte place.
__device__ __forceinline__ u16x8 load8_any(const u16* p) {
  u16x8 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

template <int S>
__global__ __launch_bounds__(256) void k_conv_dw(const u16* __restrict__ xt, const u16* __restrict__ dz,
                                                 float* __restrict__ part, int ntiles) {
  constexpr int V = S * S * S, P = S + 2, VP = P * P * P, SPT = V / 32;  // steps of 32 voxels per tile
  constexpr int LEN = dw_part_len<PC>();
  __shared__ float sum[LEN];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  f32x4 acc[NTAP];
#pragma unroll
  for (int t = 0; t < NTAP; ++t) acc[t] = {0.f, 0.f, 0.f, 0.f};
  float bsum = 0.f;
  const long steps = (long)ntiles * SPT, waves = (long)gridDim.x * 4, me = (long)blockIdx.x * 4 + w;
  for (long st = steps * me / waves; st < steps * (me + 1) / waves; ++st) {
    const int tile = (int)(st / SPT), v = (int)(st % SPT) * 32 + 8 * g;  // 8 voxels of one row
    const int x = v % S, y = (v / S) % S, z = v / (S * S);
    const u16* d = dz + ((size_t)tile * V + v) * PC + i;
    u16x8 a;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a[e] = d[e * PC];
      bsum += bf2f(a[e]);
    }
    const u16* src = xt + ((size_t)tile * PC + i) * VP + (z * P + y) * P + x;
#pragma unroll
    for (int t = 0; t < NTAP; ++t)
      acc[t] = mfma(a, load8_any(src + (t / 9 * P + (t / 3) % 3) * P + t % 3), acc[t]);
  }
  bsum += __shfl_xor(bsum, 16);
  bsum += __shfl_xor(bsum, 32);
  // D: column = lane & 15 (ci), rows co = 4g + e; the waves add in turn
  for (int k = 0; k < 4; ++k) {
    if (w == k) {
#pragma unroll
      for (int t = 0; t < NTAP; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int q = (t * PC + 4 * g + e) * PC + i;
          sum[q] = k == 0 ? acc[t][e] : sum[q] + acc[t][e];
        }
      if (g == 0) sum[LEN - PC + i] = k == 0 ? bsum : sum[LEN - PC + i] + bsum;
    }
    __syncthreads();
  }
  float* pw = part + (size_t)blockIdx.x * LEN;
  for (int k = threadIdx.x; k < LEN; k += 256) pw[k] = sum[k];
}

// The first layer's: dz[v][co] = the pooled gradient of v's parent / 8 where the
// activation's bit is set. Items are slabs of 4 planes of a tile.
__global__ __launch_bounds__(256) void k_conv1_dw(const u16* __restrict__ in, const u16* __restrict__ bits,
                                                  const u16* __restrict__ dp, float* __restrict__ part, int ntiles) {
  constexpr int H = PT / 2, V = PT * PT * PT, ZS = 4, SLABS = PT / ZS;
  constexpr int LEN = dw_part_len<1>();
  __shared__ u16 slab[(ZS + 2) * HY * HX];
  __shared__ float sum[LEN];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  float bsum = 0.f;
  int off[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int t = 16 * nb + i < NTAP ? 16 * nb + i : 0;  // columns past tap 26 are not kept
    off[nb] = (t / 9 * HY + (t / 3) % 3) * HX + t % 3;
  }
  for (int item = blockIdx.x; item < ntiles * SLABS; item += gridDim.x) {
    const int tile = item / SLABS, z0 = (item % SLABS) * ZS;
    __syncthreads();
    stage_slab(in + (size_t)tile * V, z0, ZS, slab);
    __syncthreads();
    for (int row = w; row < ZS * PT; row += 4) {  // one row of 32 voxels per step
      const int dz = row / PT, y = row % PT, z = z0 + dz;
      const size_t v = (size_t)tile * V + (z * PT + y) * PT + 8 * g;
      const u16x8 m = load8(bits + v);
      const u16* d = dp + ((((size_t)tile * H + z / 2) * H + y / 2) * H + 4 * g) * PC + i;
      u16x8 a;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const u16 q = f2bf(bf2f(d[(e >> 1) * PC]) * 0.125f);
        a[e] = (m[e] >> i) & 1 ? q : (u16)0;
        bsum += bf2f(a[e]);
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const u16* src = slab + (dz * HY + y) * HX + 8 * g + off[nb];
        u16x8 b;
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = src[e];
        acc[nb] = mfma(a, b, acc[nb]);
      }
    }
  }
  bsum += __shfl_xor(bsum, 16);
  bsum += __shfl_xor(bsum, 32);
  __syncthreads();
  // D: column = lane & 15 (tap), rows co = 4g + e
  for (int k = 0; k < 4; ++k) {
    if (w == k) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 16 * nb + i, q = (4 * g + e) * NTAP + t;
          if (t < NTAP) sum[q] = k == 0 ? acc[nb][e] : sum[q] + acc[nb][e];
        }
      if (g == 0) sum[LEN - PC + i] = k == 0 ? bsum : sum[LEN - PC + i] + bsum;
    }
    __syncthreads();
  }
  float* pw = part + (size_t)blockIdx.x * LEN;
  for (int k = threadIdx.x; k < LEN; k += 256) pw[k] = sum[k];
}

// grad[k] = sum over p of part[p][k], k < len: a workgroup takes 16 values of k,
// 16 threads each (the partials of a set are contiguous: 64-byte reads).
__global__ __launch_bounds__(256) void k_reduce_parts(const float* __restrict__ part, int len, int nparts,
                                                      float* __restrict__ grad) {
  __shared__ float red[256];
  const int t = threadIdx.x, k = blockIdx.x * 16 + (t & 15);
  float s = 0.f;
  if (k < len)
    for (int p = t >> 4; p < nparts; p += 16) s += part[(size_t)p * len + k];
  red[t] = s;
  __syncthreads();
  for (int h = 128; h >= 16; h >>= 1) {
    if (t < h) red[t] += red[t + h];
    __syncthreads();
  }
  if (t < 16 && k < len) grad[k] = red[t];
}

// ---------------------------------------------------------------------------
// Average pooling by 2 (channels-last) and its gradient with the ReLU mask of
// the pooled activation. pool: out rows [ntiles, nrows) are zeroed (they pad
// the head's GEMM). unpool: din = dout(parent) / 8 where a > 0.
// ---------------------------------------------------------------------------
template <int S>
__global__ __launch_bounds__(256) void k_pool(const u16* __restrict__ in, u16* __restrict__ out, int ntiles,
                                              int nrows) {
  constexpr int H = S / 2, VO = H * H * H;
  const long total = (long)nrows * VO * PC;
  for (long id = blockIdx.x * (long)blockDim.x + threadIdx.x; id < total; id += (long)gridDim.x * blockDim.x) {
    const int c = (int)(id % PC);
    const long vo = id / PC;
    const int tile = (int)(vo / VO), r = (int)(vo % VO);
    if (tile >= ntiles) {
      out[id] = 0;
      continue;
    }
    const int x = r % H, y = (r / H) % H, z = r / (H * H);
    float s = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const int vi = ((2 * z + (d >> 2)) * S + 2 * y + ((d >> 1) & 1)) * S + 2 * x + (d & 1);
      s += bf2f(in[((size_t)tile * S * S * S + vi) * PC + c]);
    }
    out[id] = f2bf(s * 0.125f);
  }
}

template <int S, class T>
__global__ __launch_bounds__(256) void k_unpool(const T* __restrict__ dout, const u16* __restrict__ act,
                                                u16* __restrict__ din, int ntiles) {
  constexpr int H = S / 2, V = S * S * S;
  const long total = (long)ntiles * V * PC;
  for (long id = blockIdx.x * (long)blockDim.x + threadIdx.x; id < total; id += (long)gridDim.x * blockDim.x) {
    const int c = (int)(id % PC);
    const long vi = id / PC;
    const int tile = (int)(vi / V), r = (int)(vi % V);
    const int x = r % S, y = (r / S) % S, z = r / (S * S);
    const size_t po = ((size_t)tile * H * H * H + ((z / 2) * H + y / 2) * H + x / 2) * PC + c;
    float d;
    if constexpr (sizeof(T) == 4)
      d = dout[po];
    else
      d = bf2f(dout[po]);
    din[id] = bf_pos(act[id]) ? f2bf(d * 0.125f) : (u16)0;
  }
}

// ---------------------------------------------------------------------------
// C[m][n] = sum_k A(m, k) B(k, n) (+ bias[n]) with A(m, k) = A[m*sam + k*sak],
// B(k, n) = B[k*sbk + n*sbn] (bf16) and C fp32 at C[m*scm + n]; one wave per
// 16 x 16 block of C; rows m >= M and columns n >= N are not stored, operand
// entries past M, N or K read as zero.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_gemm(const u16* __restrict__ A, long sam, long sak, const u16* __restrict__ B,
                                              long sbk, long sbn, float* __restrict__ C, long scm, int M, int N,
                                              int K, const float* __restrict__ bias) {
  const int lane = threadIdx.x & 63;
  const int nbn = (N + 15) / 16;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int mb = wave / nbn, nb = wave % nbn;
  if (mb * 16 >= M) return;
  const int i = lane & 15, g = lane >> 4;
  const int m = mb * 16 + i, n = nb * 16 + i;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // an operand whose k runs contiguously at 16-byte places is loaded 8 values at a time
  const bool va = sak == 1 && sam % 8 == 0 && K % 32 == 0 && ((size_t)A & 15) == 0;
  const bool vb = sbk == 1 && sbn % 8 == 0 && K % 32 == 0 && ((size_t)B & 15) == 0;
  for (int k0 = 0; k0 < K; k0 += 32) {
    u16x8 a = {0, 0, 0, 0, 0, 0, 0, 0}, b = a;
    const int kk = k0 + 8 * g;
    if (va) {
      if (m < M) a = load8(A + m * sam + kk);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = (m < M && kk + e < K) ? A[m * sam + (kk + e) * sak] : (u16)0;
    }
    if (vb) {
      if (n < N) b = load8(B + n * sbn + kk);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = (n < N && kk + e < K) ? B[(kk + e) * sbk + n * sbn] : (u16)0;
    }
    acc = mfma(a, b, acc);
  }
  const int col = nb * 16 + i;
  if (col >= N) return;
  const float bb = bias ? bias[col] : 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = mb * 16 + 4 * g + e;
    if (row < M) C[row * scm + col] = acc[e] + bb;
  }
}

// ---------------------------------------------------------------------------
// Softmax cross-entropy over the 501 classes, one wave per row. Rows < n:
// dlog = (softmax - onehot(label)) / n (fp32 and bf16), loss[r]; rows in
// [n, nrows): zeros.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_softmax_ce(const float* __restrict__ logits, const int* __restrict__ labels,
                                                    int n, int nrows, float* __restrict__ dlog,
                                                    u16* __restrict__ dlogb, float* __restrict__ loss) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= nrows) return;
  float* dr = dlog + (size_t)r * CPAD;
  u16* db = dlogb + (size_t)r * CPAD;
  if (r >= n) {
    for (int k = lane; k < CPAD; k += 64) {
      dr[k] = 0.f;
      db[k] = 0;
    }
    return;
  }
  const float* lr = logits + (size_t)r * CPAD;
  float mx = -INFINITY;
  for (int k = lane; k < NCLS; k += 64) mx = fmaxf(mx, lr[k]);
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  float s = 0.f;
  for (int k = lane; k < NCLS; k += 64) s += expf(lr[k] - mx);
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  const float lse = mx + logf(s);
  const int lab = min(max(labels[r], 0), NCLS - 1);  // labels outside [0, 501) are clamped
  const float inv = 1.f / (float)n;
  for (int k = lane; k < CPAD; k += 64) {
    float d = 0.f;
    if (k < NCLS) d = (expf(lr[k] - lse) - (k == lab ? 1.f : 0.f)) * inv;
    dr[k] = d;
    db[k] = f2bf(d);
  }
  if (lane == 0) loss[r] = lse - lr[lab];
}

// out[k] = sum over rows of in[r*ld + k], k < len (one workgroup per k).
__global__ __launch_bounds__(256) void k_colsum(const float* __restrict__ in, int rows, int ld, float* __restrict__ out) {
  __shared__ float red[256];
  const int k = blockIdx.x;
  float s = 0.f;
  for (int r = threadIdx.x; r < rows; r += 256) s += in[(size_t)r * ld + k];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[k] = red[0];
}

// ---------------------------------------------------------------------------
// Proposals: softmax top-1 probability and class over the 501 classes, the
// top-k of the 500 direction logits (larger logit first, ties to the lower
// index), the summed probability of those k directions (mass) and the
// probability of "no peak" (pnp). One wave per row.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_propose(const float* __restrict__ logits, int n, int topk,
                                                 int* __restrict__ dirs, float* __restrict__ top1,
                                                 int* __restrict__ cls, float* __restrict__ mass,
                                                 float* __restrict__ pnp) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  const float* lr = logits + (size_t)r * CPAD;
  float v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int k = lane + 64 * q;
    v[q] = k < NCLS ? lr[k] : -INFINITY;
  }
  float mx = -INFINITY;
  int mk = 0x7fffffff;
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (v[q] > mx) {
      mx = v[q];
      mk = lane + 64 * q;
    }
  for (int o = 32; o > 0; o >>= 1) {
    const float om = __shfl_xor(mx, o);
    const int ok = __shfl_xor(mk, o);
    if (om > mx || (om == mx && ok < mk)) {
      mx = om;
      mk = ok;
    }
  }
  float s = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) s += expf(v[q] - mx);
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) {
    top1[r] = 1.f / s;
    cls[r] = mk;
    if (pnp) pnp[r] = expf(lr[NDIR] - mx) / s;
  }
  // the background class takes no part in the direction ranking
  for (int q = 0; q < 8; ++q)
    if (lane + 64 * q >= NDIR) v[q] = -INFINITY;
  float msum = 0.f;
  for (int t = 0; t < topk; ++t) {
    float bm = -INFINITY;
    int bk = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (v[q] > bm) {
        bm = v[q];
        bk = lane + 64 * q;
      }
    for (int o = 32; o > 0; o >>= 1) {
      const float om = __shfl_xor(bm, o);
      const int ok = __shfl_xor(bk, o);
      if (om > bm || (om == bm && ok < bk)) {
        bm = om;
        bk = ok;
      }
    }
    if (lane == 0) dirs[(size_t)r * topk + t] = bk < NDIR ? bk : -1;
    if (bk < NDIR) msum += expf(bm - mx) / s;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (lane + 64 * q == bk) v[q] = -INFINITY;
  }
  if (lane == 0 && mass) mass[r] = msum;
}

// ---------------------------------------------------------------------------
// Adam on the fp32 masters, then the bf16 working copies.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ gr,
                                              float* __restrict__ m, float* __restrict__ v, int n, float lr,
                                              float b1, float b2, float eps, float c1, float c2, float wd) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float gi = gr[i] + wd * p[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  }
}

// Working copies: w1b [16][32]; wNb [27][16 co][16 ci]; wNt [27][16 ci][16 co]
// with wNt[t][a][b] = W[26 - t][b][a] (the data-gradient convolution); wfb
// [512][1024] with rows past 501 zero.
__global__ __launch_bounds__(256) void k_refresh(const float* __restrict__ p, u16* __restrict__ w1b,
                                                 u16* __restrict__ wcb, u16* __restrict__ wct,
                                                 u16* __restrict__ wfb) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  const int nconv = 3 * NTAP * PC * PC;
  if (id < PC * 32) {
    const int co = id / 32, t = id % 32;
    w1b[id] = t < NTAP ? f2bf(p[OFF_W1 + co * NTAP + t]) : (u16)0;
  }
  if (id < nconv) {
    const int l = id / (NTAP * PC * PC), r = id % (NTAP * PC * PC);
    const int t = r / (PC * PC), a = (r / PC) % PC, b = r % PC;
    const float* W = p + (l == 0 ? OFF_W2 : l == 1 ? OFF_W3 : OFF_W4);
    wcb[id] = f2bf(W[r]);
    wct[id] = f2bf(W[((NTAP - 1 - t) * PC + b) * PC + a]);
  }
  if (id < CPAD * NFEAT) {
    const int c = id / NFEAT;
    wfb[id] = c < NCLS ? f2bf(p[OFF_WF + id]) : (u16)0;
  }
}

// ---------------------------------------------------------------------------
// Tiles of an n^3 volume (n a multiple of 32), standardised by the volume's
// mean and standard deviation (double sums) and rounded to bf16:
// tiles[(tz*nt + ty)*nt + tx][z][y][x].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_moments(const float* __restrict__ vol, size_t n, double* __restrict__ part) {
  __shared__ double r1[256], r2[256];
  double s1 = 0, s2 = 0;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const double x = vol[i];
    s1 += x;
    s2 += x * x;
  }
  r1[threadIdx.x] = s1;
  r2[threadIdx.x] = s2;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      r1[threadIdx.x] += r1[threadIdx.x + h];
      r2[threadIdx.x] += r2[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r1[0];
    part[2 * blockIdx.x + 1] = r2[0];
  }
}

__global__ __launch_bounds__(256) void k_tiles(const float* __restrict__ vol, int n, const double* __restrict__ part,
                                               int nparts, u16* __restrict__ tiles) {
  __shared__ float stat[2];
  if (threadIdx.x == 0) {
    double s1 = 0, s2 = 0;
    for (int k = 0; k < nparts; ++k) {
      s1 += part[2 * k];
      s2 += part[2 * k + 1];
    }
    const double N = (double)n * n * n, mean = s1 / N;
    const double var = fmax(s2 / N - mean * mean, 0.0);
    stat[0] = (float)mean;
    stat[1] = var > 0 ? (float)(1.0 / sqrt(var)) : 0.f;
  }
  __syncthreads();
  const int nt = n / PT;
  const size_t total = (size_t)n * n * n;
  for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < total; id += (size_t)gridDim.x * blockDim.x) {
    const int x = (int)(id % n), y = (int)((id / n) % n), z = (int)(id / ((size_t)n * n));
    const size_t tile = ((size_t)(z / PT) * nt + y / PT) * nt + x / PT;
    const size_t o = tile * PT * PT * PT + ((size_t)(z % PT) * PT + y % PT) * PT + x % PT;
    tiles[o] = f2bf((vol[id] - stat[0]) * stat[1]);
  }
}

__global__ __launch_bounds__(256) void k_f32_to_bf16(const float* __restrict__ in, u16* __restrict__ out, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = f2bf(in[i]);
}

unsigned grid_of(size_t n, unsigned cap = 65535) { return (unsigned)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, cap)); }

}  // namespace
}  // namespace gx

using namespace gx;

// ---------------------------------------------------------------------------
// Network state
// ---------------------------------------------------------------------------
struct gtomx_pnet {
  int device = 0;
  unsigned cap = 0;   // tiles per pass
  unsigned rows = 0;  // cap rounded up to 16 (head GEMM rows)
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // NPARAM each
  long step = 0;
  u16 *w1b = nullptr, *wcb = nullptr, *wct = nullptr, *wfb = nullptr;
  u16* xt = nullptr;  // input of a 16-channel weight gradient, channels first with a halo (16^3 the largest)
  u16 *x = nullptr, *bits1 = nullptr, *p1 = nullptr, *a2 = nullptr, *p2 = nullptr, *a3 = nullptr, *a4 = nullptr,
      *feat = nullptr;
  float* logits = nullptr;
  float* dlog = nullptr;
  u16* dlogb = nullptr;
  float* dfeat = nullptr;
  float* loss = nullptr;
  u16 *dz4 = nullptr, *dz3 = nullptr, *dp2 = nullptr, *dz2 = nullptr, *dp1 = nullptr;
  float* part = nullptr;
  double* mom = nullptr;  // moments partials of k_moments
  unsigned nlast = 0;     // tiles of the last forward pass
  size_t device_bytes = 0;
  StreamFence fence;
};

namespace gx {
namespace {

constexpr int MOM_BLOCKS = 512;

void pnet_release(gtomx_pnet* nt) {
  if (!nt) return;
  nt->fence.release();
  for (void* q : {(void*)nt->p, (void*)nt->g, (void*)nt->m, (void*)nt->v, (void*)nt->w1b, (void*)nt->wcb,
                  (void*)nt->wct, (void*)nt->wfb, (void*)nt->x, (void*)nt->xt, (void*)nt->bits1, (void*)nt->p1, (void*)nt->a2,
                  (void*)nt->p2, (void*)nt->a3, (void*)nt->a4, (void*)nt->feat, (void*)nt->logits, (void*)nt->dlog,
                  (void*)nt->dlogb, (void*)nt->dfeat, (void*)nt->loss, (void*)nt->dz4, (void*)nt->dz3,
                  (void*)nt->dp2, (void*)nt->dz2, (void*)nt->dp1, (void*)nt->part, (void*)nt->mom})
    dev_free(q);
  delete nt;
}

int pnet_check(const gtomx_pnet* nt) {
  if (!nt) return fail(GTOMX_ERR_INVALID_ARGUMENT, "network is NULL");
  int dev = 0;
  GX_HIP(hipGetDevice(&dev));
  if (dev != nt->device) return fail(GTOMX_ERR_INVALID_ARGUMENT, "network was created on another device");
  return GTOMX_OK;
}

int refresh(gtomx_pnet* nt, hipStream_t s) {
  hipLaunchKernelGGL(k_refresh, dim3(grid_of(CPAD * NFEAT)), dim3(256), 0, s, nt->p, nt->w1b, nt->wcb, nt->wct,
                     nt->wfb);
  GX_LAUNCHED("k_refresh");
  return GTOMX_OK;
}

template <int S>
int conv(const u16* in, const u16* wb, const float* bias, const u16* mask, u16* out, unsigned n, int relu,
         hipStream_t s) {
  const long waves = (long)n * (S * S * S / (16 * VG));
  hipLaunchKernelGGL((k_conv<S>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, in, wb, bias, mask, out, (int)n,
                     relu);
  GX_LAUNCHED("k_conv");
  return GTOMX_OK;
}

constexpr int DW_PARTS = 512;  // workgroups (and sets of partials) of a weight gradient: two per CU

int reduce_parts(gtomx_pnet* nt, int len, int nparts, float* grad, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce_parts, dim3((len + 15) / 16), dim3(256), 0, s, nt->part, len, nparts, grad);
  GX_LAUNCHED("k_reduce_parts");
  return GTOMX_OK;
}

// Weight and bias gradient of a 16-channel convolution into grad (weights, then bias).
template <int S> int conv_dw(gtomx_pnet* nt, const u16* in, const u16* dz, unsigned n, float* grad, hipStream_t s) {
  constexpr int VP = (S + 2) * (S + 2) * (S + 2);
  hipLaunchKernelGGL((k_halo_channels<S>), dim3(grid_of((size_t)n * VP)), dim3(256), 0, s, in, nt->xt, (int)n);
  GX_LAUNCHED("k_halo_channels");
  const int nparts = (int)std::min<long>(DW_PARTS, ((long)n * (S * S * S / 32) + 3) / 4);
  hipLaunchKernelGGL((k_conv_dw<S>), dim3(nparts), dim3(256), 0, s, nt->xt, dz, nt->part, (int)n);
  GX_LAUNCHED("k_conv_dw");
  return reduce_parts(nt, dw_part_len<PC>(), nparts, grad, s);
}

// The first layer's, from the pooled gradient.
int conv1_dw(gtomx_pnet* nt, unsigned n, float* grad, hipStream_t s) {
  const int nparts = (int)std::min<long>(2 * DW_PARTS, (long)n * 8);
  hipLaunchKernelGGL(k_conv1_dw, dim3(nparts), dim3(256), 0, s, nt->x, nt->bits1, nt->dp1, nt->part, (int)n);
  GX_LAUNCHED("k_conv1_dw");
  return reduce_parts(nt, dw_part_len<1>(), nparts, grad, s);
}

int gemm(const u16* A, long sam, long sak, const u16* B, long sbk, long sbn, float* C, long scm, int M, int N, int K,
         const float* bias, hipStream_t s) {
  const int waves = ((M + 15) / 16) * ((N + 15) / 16);
  hipLaunchKernelGGL(k_gemm, dim3((waves + 3) / 4), dim3(256), 0, s, A, sam, sak, B, sbk, sbn, C, scm, M, N, K, bias);
  GX_LAUNCHED("k_gemm");
  return GTOMX_OK;
}

template <int S, class T> int unpool(const T* dout, const u16* act, u16* din, unsigned n, hipStream_t s) {
  hipLaunchKernelGGL((k_unpool<S, T>), dim3(grid_of((size_t)n * S * S * S * PC)), dim3(256), 0, s, dout, act, din,
                     (int)n);
  GX_LAUNCHED("k_unpool");
  return GTOMX_OK;
}

template <int S> int pool(const u16* in, u16* out, unsigned n, unsigned rows, hipStream_t s) {
  hipLaunchKernelGGL((k_pool<S>), dim3(grid_of((size_t)rows * (S / 2) * (S / 2) * (S / 2) * PC)), dim3(256), 0, s,
                     in, out, (int)n, (int)rows);
  GX_LAUNCHED("k_pool");
  return GTOMX_OK;
}

unsigned rows_of(unsigned n) { return (n + 15) / 16 * 16; }

// Forward pass over n tiles already in nt->x.
int forward(gtomx_pnet* nt, unsigned n, hipStream_t s) {
  const unsigned rows = rows_of(n);
  hipLaunchKernelGGL(k_conv1_pool, dim3(n * (PT / 2)), dim3(256), 0, s, nt->x, nt->w1b, nt->p + OFF_B1, nt->bits1,
                     nt->p1);
  GX_LAUNCHED("k_conv1_pool");
  GX_TRY((conv<16>(nt->p1, nt->wcb, nt->p + OFF_B2, nullptr, nt->a2, n, 1, s)));
  GX_TRY(pool<16>(nt->a2, nt->p2, n, n, s));
  GX_TRY((conv<8>(nt->p2, nt->wcb + NTAP * PC * PC, nt->p + OFF_B3, nullptr, nt->a3, n, 1, s)));
  GX_TRY((conv<8>(nt->a3, nt->wcb + 2 * NTAP * PC * PC, nt->p + OFF_B4, nullptr, nt->a4, n, 1, s)));
  GX_TRY(pool<8>(nt->a4, nt->feat, n, rows, s));
  // logits[r][c] = feat[r] . Wf[c] + bf[c] for the 501 classes (columns 501..511 stay zero)
  GX_TRY(gemm(nt->feat, NFEAT, 1, nt->wfb, 1, NFEAT, nt->logits, CPAD, (int)rows, NCLS, NFEAT, nt->p + OFF_BF, s));
  nt->nlast = n;
  return GTOMX_OK;
}

// Backward pass from the labels (after forward over the same n tiles); the
// gradients land in nt->g, the per-tile losses in nt->loss.
int backward(gtomx_pnet* nt, const int* d_labels, unsigned n, hipStream_t s) {
  const unsigned rows = rows_of(n);
  hipLaunchKernelGGL(k_softmax_ce, dim3((rows + 3) / 4), dim3(256), 0, s, nt->logits, d_labels, (int)n, (int)rows,
                     nt->dlog, nt->dlogb, nt->loss);
  GX_LAUNCHED("k_softmax_ce");
  hipLaunchKernelGGL(k_colsum, dim3(NCLS), dim3(256), 0, s, nt->dlog, (int)rows, CPAD, nt->g + OFF_BF);
  GX_LAUNCHED("k_colsum");
  // dWf[c][f] = sum_r dlog[r][c] feat[r][f]
  GX_TRY(gemm(nt->dlogb, 1, CPAD, nt->feat, NFEAT, 1, nt->g + OFF_WF, NFEAT, NCLS, NFEAT, (int)rows, nullptr, s));
  // dfeat[r][f] = sum_c dlog[r][c] Wf[c][f]
  GX_TRY(gemm(nt->dlogb, CPAD, 1, nt->wfb, NFEAT, 1, nt->dfeat, NFEAT, (int)rows, NFEAT, CPAD, nullptr, s));
  GX_TRY((unpool<8, float>(nt->dfeat, nt->a4, nt->dz4, n, s)));
  GX_TRY(conv_dw<8>(nt, nt->a3, nt->dz4, n, nt->g + OFF_W4, s));
  GX_TRY((conv<8>(nt->dz4, nt->wct + 2 * NTAP * PC * PC, nullptr, nt->a3, nt->dz3, n, 0, s)));
  GX_TRY(conv_dw<8>(nt, nt->p2, nt->dz3, n, nt->g + OFF_W3, s));
  GX_TRY((conv<8>(nt->dz3, nt->wct + NTAP * PC * PC, nullptr, nullptr, nt->dp2, n, 0, s)));
  GX_TRY((unpool<16, u16>(nt->dp2, nt->a2, nt->dz2, n, s)));
  GX_TRY(conv_dw<16>(nt, nt->p1, nt->dz2, n, nt->g + OFF_W2, s));
  GX_TRY((conv<16>(nt->dz2, nt->wct, nullptr, nullptr, nt->dp1, n, 0, s)));
  return conv1_dw(nt, n, nt->g + OFF_W1, s);
}

}  // namespace
}  // namespace gx

extern "C" {

int gtomx_pnet_param_count(void) { return NPARAM; }

int gtomx_pnet_create(gtomx_pnet** out, unsigned max_tiles) {
  if (!out) return fail(GTOMX_ERR_INVALID_ARGUMENT, "network pointer is NULL");
  *out = nullptr;
  if (max_tiles == 0 || max_tiles > 65536) return fail(GTOMX_ERR_INVALID_ARGUMENT, "max_tiles must be in [1, 65536]");
  auto* nt = new gtomx_pnet();
  nt->cap = max_tiles;
  nt->rows = rows_of(max_tiles);
  hipError_t he = hipGetDevice(&nt->device);
  if (he != hipSuccess) {
    pnet_release(nt);
    return hip_fail(he, "hipGetDevice");
  }
  int st = GTOMX_OK;
  auto alloc = [&](auto** dst, size_t bytes) {
    if (st != GTOMX_OK) return;
    void* d = nullptr;
    st = dev_alloc(&d, bytes);
    if (st == GTOMX_OK) {
      *dst = static_cast<std::remove_reference_t<decltype(*dst)>>(d);
      nt->device_bytes += bytes;
    }
  };
  const size_t R = nt->rows, C = nt->cap;
  const size_t V1 = 32 * 32 * 32, V2 = 16 * 16 * 16, V3 = 8 * 8 * 8;
  for (float** q : {&nt->p, &nt->g, &nt->m, &nt->v}) alloc(q, NPARAM * sizeof(float));
  alloc(&nt->w1b, PC * 32 * 2);
  alloc(&nt->wcb, 3 * NTAP * PC * PC * 2);
  alloc(&nt->wct, 3 * NTAP * PC * PC * 2);
  alloc(&nt->wfb, (size_t)CPAD * NFEAT * 2);
  alloc(&nt->x, C * V1 * 2);
  alloc(&nt->xt, C * PC * 18 * 18 * 18 * 2);
  alloc(&nt->bits1, C * V1 * 2);
  alloc(&nt->p1, C * V2 * PC * 2);
  alloc(&nt->a2, C * V2 * PC * 2);
  alloc(&nt->p2, C * V3 * PC * 2);
  alloc(&nt->a3, C * V3 * PC * 2);
  alloc(&nt->a4, C * V3 * PC * 2);
  alloc(&nt->feat, R * NFEAT * 2);
  alloc(&nt->logits, R * CPAD * 4);
  alloc(&nt->dlog, R * CPAD * 4);
  alloc(&nt->dlogb, R * CPAD * 2);
  alloc(&nt->dfeat, R * NFEAT * 4);
  alloc(&nt->loss, R * 4);
  alloc(&nt->dz4, C * V3 * PC * 2);
  alloc(&nt->dz3, C * V3 * PC * 2);
  alloc(&nt->dp2, C * V3 * PC * 2);
  alloc(&nt->dz2, C * V2 * PC * 2);
  alloc(&nt->dp1, C * V2 * PC * 2);
  static_assert(2 * dw_part_len<1>() <= dw_part_len<PC>(), "the first layer's partials fit the others' scratch");
  alloc(&nt->part, (size_t)DW_PARTS * dw_part_len<PC>() * 4);
  alloc(&nt->mom, (size_t)MOM_BLOCKS * 2 * sizeof(double));
  if (st != GTOMX_OK) {
    std::string msg = gtomx_last_error();
    pnet_release(nt);
    return fail(st, msg);
  }
  // zero parameters and optimiser state until gtomx_pnet_set_params
  for (float* q : {nt->p, nt->g, nt->m, nt->v}) he = he == hipSuccess ? hipMemset(q, 0, NPARAM * sizeof(float)) : he;
  if (he == hipSuccess) he = hipMemset(nt->logits, 0, R * CPAD * 4);
  if (he == hipSuccess) he = hipStreamSynchronize(nullptr);  // the clears ran on the null stream
  if (he != hipSuccess) {
    pnet_release(nt);
    return hip_fail(he, "network set-up");
  }
  *out = nt;
  return GTOMX_OK;
}

int gtomx_pnet_destroy(gtomx_pnet* net) {
  pnet_release(net);
  return GTOMX_OK;
}

int gtomx_pnet_set_params(gtomx_pnet* nt, const float* h_params, size_t count, void* stream) {
  GX_TRY(pnet_check(nt));
  if (!h_params || count != (size_t)NPARAM) return fail(GTOMX_ERR_INVALID_ARGUMENT, "expected all parameters");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  GX_HIP(hipMemcpyAsync(nt->p, h_params, NPARAM * sizeof(float), hipMemcpyHostToDevice, s));
  GX_HIP(hipMemsetAsync(nt->m, 0, NPARAM * sizeof(float), s));
  GX_HIP(hipMemsetAsync(nt->v, 0, NPARAM * sizeof(float), s));
  nt->step = 0;
  GX_TRY(refresh(nt, s));
  GX_TRY(nt->fence.leave(s));
  GX_HIP(hipStreamSynchronize(s));  // the host array may go away on return
  return GTOMX_OK;
}

int gtomx_pnet_get_params(gtomx_pnet* nt, float* h_params, size_t count, void* stream) {
  GX_TRY(pnet_check(nt));
  if (!h_params || count != (size_t)NPARAM) return fail(GTOMX_ERR_INVALID_ARGUMENT, "expected all parameters");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  GX_HIP(hipMemcpyAsync(h_params, nt->p, NPARAM * sizeof(float), hipMemcpyDeviceToHost, s));
  GX_TRY(nt->fence.leave(s));
  GX_HIP(hipStreamSynchronize(s));
  return GTOMX_OK;
}

// The network's input from n tiles of 32^3 floats (already standardised), rounded to bf16.
int gtomx_pnet_load_tiles(gtomx_pnet* nt, const float* d_tiles, unsigned n, void* stream) {
  GX_TRY(pnet_check(nt));
  if (!d_tiles || n == 0 || n > nt->cap) return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL tiles or n out of range");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  const size_t cnt = (size_t)n * PT * PT * PT;
  hipLaunchKernelGGL(k_f32_to_bf16, dim3(grid_of(cnt)), dim3(256), 0, s, d_tiles, nt->x, cnt);
  GX_LAUNCHED("k_f32_to_bf16");
  return nt->fence.leave(s);
}

// The network's input from every 32^3 tile of an n^3 volume (n a multiple of 32, (n/32)^3 <= max_tiles),
// standardised by the volume's mean and standard deviation; tile (tz*nt + ty)*nt + tx.
int gtomx_pnet_load_volume(gtomx_pnet* nt, const float* d_volume, gtomx_int3 dims, void* stream) {
  GX_TRY(pnet_check(nt));
  if (!d_volume) return fail(GTOMX_ERR_INVALID_ARGUMENT, "d_volume is NULL");
  if (dims.x != dims.y || dims.x != dims.z || dims.x % PT || dims.x < PT)
    return fail(GTOMX_ERR_UNSUPPORTED, "the volume must be a cube whose side is a multiple of 32");
  const size_t ntl = (size_t)(dims.x / PT) * (dims.x / PT) * (dims.x / PT);
  if (ntl > nt->cap) return fail(GTOMX_ERR_INVALID_ARGUMENT, "more tiles than the network's max_tiles");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  const size_t V = elements(dims);
  hipLaunchKernelGGL(k_moments, dim3(MOM_BLOCKS), dim3(256), 0, s, d_volume, V, nt->mom);
  GX_LAUNCHED("k_moments");
  hipLaunchKernelGGL(k_tiles, dim3(grid_of(V)), dim3(256), 0, s, d_volume, dims.x, nt->mom, MOM_BLOCKS, nt->x);
  GX_LAUNCHED("k_tiles");
  return nt->fence.leave(s);
}

// Forward pass over the first n loaded tiles: d_logits (optional) receives n x 512 floats (501 used).
int gtomx_pnet_forward(gtomx_pnet* nt, unsigned n, float* d_logits, void* stream) {
  GX_TRY(pnet_check(nt));
  if (n == 0 || n > nt->cap) return fail(GTOMX_ERR_INVALID_ARGUMENT, "n out of range");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  GX_TRY(forward(nt, n, s));
  if (d_logits) GX_HIP(hipMemcpyAsync(d_logits, nt->logits, (size_t)n * CPAD * 4, hipMemcpyDeviceToDevice, s));
  return nt->fence.leave(s);
}

// Loss and gradients of the loaded tiles against labels (class per tile): d_grads (optional) receives
// the NPARAM gradients, d_loss (optional) the n per-tile losses.
int gtomx_pnet_gradients(gtomx_pnet* nt, const int32_t* d_labels, unsigned n, float* d_grads, float* d_loss,
                         void* stream) {
  GX_TRY(pnet_check(nt));
  if (!d_labels || n == 0 || n > nt->cap) return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL labels or n out of range");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  GX_TRY(forward(nt, n, s));
  GX_TRY(backward(nt, d_labels, n, s));
  if (d_grads) GX_HIP(hipMemcpyAsync(d_grads, nt->g, NPARAM * 4, hipMemcpyDeviceToDevice, s));
  if (d_loss) GX_HIP(hipMemcpyAsync(d_loss, nt->loss, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
  return nt->fence.leave(s);
}

// One Adam step (beta 0.9 / 0.999, eps 1e-8, decoupled-free L2 weight decay wd) on the loaded tiles.
int gtomx_pnet_train_step(gtomx_pnet* nt, const int32_t* d_labels, unsigned n, float lr, float wd, float* d_loss,
                          void* stream) {
  GX_TRY(pnet_check(nt));
  if (!d_labels || n == 0 || n > nt->cap) return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL labels or n out of range");
  if (!(lr >= 0.f) || !std::isfinite(lr)) return fail(GTOMX_ERR_INVALID_ARGUMENT, "lr must be finite, >= 0");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  GX_TRY(forward(nt, n, s));
  GX_TRY(backward(nt, d_labels, n, s));
  nt->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = (float)(1.0 / (1.0 - std::pow((double)b1, (double)nt->step)));
  const float c2 = (float)(1.0 / (1.0 - std::pow((double)b2, (double)nt->step)));
  hipLaunchKernelGGL(k_adam, dim3(grid_of(NPARAM, 2048)), dim3(256), 0, s, nt->p, nt->g, nt->m, nt->v, NPARAM, lr, b1,
                     b2, 1e-8f, c1, c2, wd);
  GX_LAUNCHED("k_adam");
  GX_TRY(refresh(nt, s));
  if (d_loss) GX_HIP(hipMemcpyAsync(d_loss, nt->loss, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
  return nt->fence.leave(s);
}

// Proposals from the last forward pass: per tile the top-k directions (d_dirs, n x topk), the softmax
// probability of the top class (d_top1) and that class (d_class; 500 = no peak), and optionally the
// summed probability of the k directions (d_mass) and the probability of "no peak" (d_nopeak).
int gtomx_pnet_propose(gtomx_pnet* nt, unsigned topk, int32_t* d_dirs, float* d_top1, int32_t* d_class,
                       float* d_mass, float* d_nopeak, void* stream) {
  GX_TRY(pnet_check(nt));
  if (nt->nlast == 0) return fail(GTOMX_ERR_INVALID_ARGUMENT, "no forward pass has run");
  if (topk == 0 || topk > (unsigned)NDIR) return fail(GTOMX_ERR_INVALID_ARGUMENT, "topk must be in [1, 500]");
  if (!d_dirs || !d_top1 || !d_class) return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL output buffer");
  hipStream_t s = as_stream(stream);
  GX_TRY(nt->fence.enter(s));
  hipLaunchKernelGGL(k_propose, dim3((nt->nlast + 3) / 4), dim3(256), 0, s, nt->logits, (int)nt->nlast, (int)topk,
                     d_dirs, d_top1, d_class, d_mass, d_nopeak);
  GX_LAUNCHED("k_propose");
  return nt->fence.leave(s);
}

// The head's GEMM on its own (bf16 operands from float inputs, fp32 result), for tests of the
// matrix-core operand layout: C (M x N, row stride N) = A (M x K) . B (K x N), both row-major.
int gtomx_pnet_debug_gemm(const float* d_a, const float* d_b, float* d_c, int M, int N, int K, void* stream) {
  if (!d_a || !d_b || !d_c || M <= 0 || N <= 0 || K <= 0) return fail(GTOMX_ERR_INVALID_ARGUMENT, "bad GEMM");
  hipStream_t s = as_stream(stream);
  DevBuf ab, bb;
  GX_TRY(ab.alloc((size_t)M * K * 2));
  GX_TRY(bb.alloc((size_t)K * N * 2));
  hipLaunchKernelGGL(k_f32_to_bf16, dim3(grid_of((size_t)M * K)), dim3(256), 0, s, d_a, ab.as<u16>(), (size_t)M * K);
  GX_LAUNCHED("k_f32_to_bf16");
  hipLaunchKernelGGL(k_f32_to_bf16, dim3(grid_of((size_t)K * N)), dim3(256), 0, s, d_b, bb.as<u16>(), (size_t)K * N);
  GX_LAUNCHED("k_f32_to_bf16");
  GX_TRY(gemm(ab.as<u16>(), K, 1, bb.as<u16>(), N, 1, d_c, N, M, N, K, nullptr, s));
  GX_HIP(hipStreamSynchronize(s));
  return GTOMX_OK;
}

}  // extern "C"
