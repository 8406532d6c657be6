// Chirp-z (Bluestein) lines of up to 512 points inside one kernel: the shapes,
// the tables a workgroup stages and the convolution itself, shared by the
// transforms (fft.hip) and the generic search's pass 1 (pick.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dev_fft.hpp"
#include "runtime.hpp"

namespace gx {

template <int M> struct BlueShape;
template <> struct BlueShape<16>   { static constexpr int R1 = 4,  R2 = 4,  TX = 64; };
template <> struct BlueShape<24>   { static constexpr int R1 = 12, R2 = 2,  TX = 64; };
template <> struct BlueShape<32>   { static constexpr int R1 = 8,  R2 = 4,  TX = 64; };
template <> struct BlueShape<48>   { static constexpr int R1 = 12, R2 = 4,  TX = 64; };
template <> struct BlueShape<64>   { static constexpr int R1 = 8,  R2 = 8,  TX = 32; };
template <> struct BlueShape<96>   { static constexpr int R1 = 24, R2 = 4,  TX = 32; };
template <> struct BlueShape<128>  { static constexpr int R1 = 16, R2 = 8,  TX = 32; };
template <> struct BlueShape<192>  { static constexpr int R1 = 24, R2 = 8,  TX = 16; };
template <> struct BlueShape<256>  { static constexpr int R1 = 16, R2 = 16, TX = 16; };
template <> struct BlueShape<512>  { static constexpr int R1 = 32, R2 = 16, TX = 16; };
template <> struct BlueShape<1024> { static constexpr int R1 = 32, R2 = 32, TX = 16; };
#define GX_FOR_BLUE(X) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(512) X(1024)
constexpr int BLUE_FUSED_MAX = 512;  // longest L of the fused form

// The circular convolution of one line with the kernel whose spectrum is B (LDS,
// M values with the 1/M in them), or with CONJ conj(B): the kernels of the two
// directions are conjugate and even, so their spectra are conjugate too. v[m] in
// and out: point j + R2 m, zero for m >= R1/2 on entry, meaningful for m < R1/2 on
// exit. Bound by its instructions: 3.9e8 vector instructions per pass of 200^3 x 32
// orientations are 0.65 ms of issue in passes of 0.8 to 1.2 ms.
template <int M, bool CONJ = false, class Xch, class Sync>
__device__ __forceinline__ void blue_convolve(float2 (&v)[BlueShape<M>::R1], int j, const float2* twl,
                                              const float2* B, Xch xch, Sync sync) {
  constexpr int R1 = BlueShape<M>::R1, R2 = BlueShape<M>::R2;
  dft<R1, -1>(v);
#pragma unroll
  for (int k1 = 1; k1 < R1; ++k1) v[k1] = cmul(v[k1], twl[k1 * (R2 + 1) + j]);
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) *xch(k1, j) = v[k1];
  sync();
#pragma unroll
  for (int u = 0; u < R1 / R2; ++u) {
    __builtin_amdgcn_sched_barrier(0);  // one k1's values at a time in registers
    const int k1 = u * R2 + j;
    float2 z[R2];
#pragma unroll
    for (int jj = 0; jj < R2; ++jj) z[jj] = *xch(k1, jj);
    dft<R2, -1>(z);
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) z[k2] = CONJ ? cmulc(z[k2], B[k1 + R1 * k2]) : cmul(z[k2], B[k1 + R1 * k2]);
    dft<R2, 1>(z);
#pragma unroll
    for (int jj = 0; jj < R2; ++jj) *xch(k1, jj) = jj == 0 ? z[jj] : cmulc(z[jj], twl[k1 * (R2 + 1) + jj]);
  }
  sync();
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) v[k1] = *xch(k1, j);
  dft<R1, 1>(v);
}

// The tables of a workgroup: the twiddles W_M^{j k1} at k1 (R2 + 1) + j, the kernel
// spectrum, the chirp as the direction multiplies by it. (A table of W_M^i read at
// i = j k1 puts the 16 lanes of a row on up to 16 addresses of one bank; by k1 and
// j, with one value of padding, both transforms read it without conflicts: rows of
// 200^3 x 32 orientations 1.17 ms, 1.23 before.)
template <int M> constexpr int blue_tw_len() { return BlueShape<M>::R1 * (BlueShape<M>::R2 + 1); }
template <int M, int DIR>
__device__ __forceinline__ void blue_stage(int t, int nt, int L, const float2* __restrict__ tw,
                                           const float2* __restrict__ B, const float2* __restrict__ chirp, float2* twl,
                                           float2* bl, float2* cl) {
  constexpr int R2 = BlueShape<M>::R2;
  for (int i = t; i < M; i += nt) {
    const int k1 = i / R2, j = i % R2;
    twl[k1 * (R2 + 1) + j] = twiddle<-1, M>(tw, j * k1 % M);
    bl[i] = B[i];
  }
  for (int i = t; i < M / 2; i += nt) {
    const float2 c = i < L ? chirp[i] : make_float2(0.f, 0.f);
    cl[i] = DIR < 0 ? c : cconj(c);
  }
}

// Chirp and kernel spectra of one length (fft.hip): chirp[j] = exp(-i pi (j^2 mod
// 2L) / L), bf / bi the M-point DFTs of the forward / inverse kernels over M.
struct BlueTables {
  int M = 0;
  float2* chirp = nullptr;
  float2* bf = nullptr;
  float2* bi = nullptr;
};
int blue_tables(int L, BlueTables* out);
// The fused form's convolution length for lines of L points.
int blue_fused_len(int L);

// f(integral_constant M) for the fused form's length M.
template <class F> int with_blue_len(int M, F f) {
  switch (M) {
#define GX_CASE(N) \
  case N:          \
    return f(std::integral_constant<int, N>{});
    GX_FOR_BLUE(GX_CASE)
#undef GX_CASE
    default: return fail(GTOMX_ERR_INTERNAL, "chirp-z length not instantiated");
  }
}

}  // namespace gx
