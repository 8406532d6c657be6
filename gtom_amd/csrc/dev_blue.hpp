// Lines of up to 512 points inside one kernel, for lengths without a native
// transform: as mixed-radix transforms where the length has small factors, by the
// chirp-z form otherwise. Shapes, the tables a workgroup stages and the transforms
// themselves, shared by the transforms (fft.hip) and the generic search's pass 1
// (pick.hip).
//
// Both are a "line" type LN of the kernels: LN::lanes threads hold a line, thread j
// the points j + lanes * m, m < LN::PTS, in natural order before and after
// LN::run (LN::WHOLE: all of them below the line's length). A workgroup stages LN::tables values, then has LN::col_area (strided
// axes: lanes over adjacent columns) or LN::row_area (contiguous rows: a line's
// threads are lanes of one wave) values of exchange per line.
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
// exit. Bound by its instructions: 3.8e8 vector instructions in pass 1 and 3.9e8 in the row
// pass of 197^3 x 32 orientations are 0.62 ms of issue each, in 0.87 and 1.19 ms.
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

// What the kernels of a line need to know; t0 / t1 / tw are device tables.
struct LineArgs {
  int L = 0;
  int M = 0;               // chirp-z: the convolution's length, or 0
  int RL = 0;              // mixed radix: points per thread
  int lanes = 0, txlog = 0;
  int r1 = 0, r2 = 0;      // lanes = r1 * r2 (r2 = 1: one stage)
  int inv1 = 0, inv2 = 0;  // 65536 / (lanes / r1) + 1, 65536 / r1 + 1: division by a multiply
  const float2 *t0 = nullptr, *t1 = nullptr, *tw = nullptr;
};

// Chirp-z. Tables: the twiddles W_M^{j k1} at k1 (R2 + 1) + j, the kernel spectrum,
// the chirp. (A table of W_M^i read at i = j k1 puts the 16 lanes of a row on up to 16
// addresses of one bank; by k1 and j, with one value of padding, both transforms read
// it without conflicts: the row pass of a 200^3 search took 1.17 ms per 32 orientations in
// this form, which that side had then, 1.23 before.)
template <int M> struct BlueLine {
  using S = BlueShape<M>;
  static constexpr int R1 = S::R1, R2 = S::R2, PTS = R1 / 2, REGS = R1;
  static constexpr bool WHOLE = false;
  static constexpr int COL_THREADS = S::TX * R2, ROW_WAVES = M <= 512 ? 2 : 1;
  static constexpr int TWL = R1 * (R2 + 1), TABLES = TWL + M + M / 2;
  // LDS of a workgroup, in float2; a constant here, so that it is a static array
  static constexpr int COL_LDS = TABLES + S::TX * M, ROW_LDS = TABLES + 256 / R2 * (M + R1);
  __host__ __device__ static int lanes(const LineArgs&) { return R2; }
  __host__ __device__ static int txlog(const LineArgs&) {
    return S::TX == 64 ? 6 : S::TX == 32 ? 5 : 4;
  }
  __host__ __device__ static int tables(const LineArgs&) { return TABLES; }
  __host__ __device__ static int row_pitch(const LineArgs&) { return R2 + 1; }
  __host__ __device__ static int row_area(const LineArgs&) { return M + R1; }
  __device__ static void stage(float2* lds, int t, int nt, const LineArgs& A) {
    for (int i = t; i < M; i += nt) {
      const int k1 = i / R2, j = i % R2;
      lds[k1 * (R2 + 1) + j] = twiddle<-1, M>(A.tw, j * k1 % M);
      lds[TWL + i] = A.t1[i];
    }
    for (int i = t; i < M / 2; i += nt) lds[TWL + M + i] = i < A.L ? A.t0[i] : make_float2(0.f, 0.f);
  }
  template <int DIR, class Xch, class Sync>
  __device__ __forceinline__ static void run(float2 (&v)[REGS], int j, const LineArgs&, const float2* lds, Xch xch,
                                             Sync sync) {
    const float2* cl = lds + TWL + M;
#pragma unroll
    for (int m = 0; m < PTS; ++m) v[m] = DIR < 0 ? cmul(v[m], cl[j + R2 * m]) : cmulc(v[m], cl[j + R2 * m]);
#pragma unroll
    for (int m = PTS; m < R1; ++m) v[m] = make_float2(0.f, 0.f);
    blue_convolve<M, (DIR > 0)>(v, j, lds, lds + TWL, xch, sync);
#pragma unroll
    for (int m = 0; m < PTS; ++m) v[m] = DIR < 0 ? cmul(v[m], cl[j + R2 * m]) : cmulc(v[m], cl[j + R2 * m]);
  }
};

// Mixed radix: L = RL * lanes, lanes = r1 or r1 * r2. The first stage is a DFT-RL over
// the points a thread holds; its output k0 of thread j, times W_L^{j k0}, goes to
// exchange place (k0, j), where DFTs of `lanes` points along j follow in place, of
// radix r1 then r2, the radices known at run time (a wave-uniform switch): output
// k0 + RL (k1 + r1 k2) ends at (k0, r2 k1 + k2). A fifth of the arithmetic of the
// chirp-z form, whose transforms are at least twice as long and run twice.
// Tables: W_L^{j k0} at k0 lanes + j, W_lanes^{b k1} at k1 r2 + b.
template <int RL_> struct SmoothLine {
  static constexpr int RL = RL_, PTS = RL, REGS = RL;
  static constexpr bool WHOLE = true;
  static constexpr int COL_THREADS = 512, ROW_WAVES = 2;
  static constexpr int COL_LDS = 0, ROW_LDS = 0;  // sized by the length: dynamic
  __host__ __device__ static int lanes(const LineArgs& A) { return A.lanes; }
  __host__ __device__ static int txlog(const LineArgs& A) { return A.txlog; }
  __host__ __device__ static int tables(const LineArgs& A) { return A.L + A.lanes; }
  __host__ __device__ static int row_pitch(const LineArgs& A) { return A.lanes | 1; }
  __host__ __device__ static int row_area(const LineArgs& A) { return RL * (A.lanes | 1); }
  __device__ static void stage(float2* lds, int t, int nt, const LineArgs& A) {
    for (int i = t; i < A.L + A.lanes; i += nt) lds[i] = A.t0[i];
  }
  // The DFT-Rs of one stage, n = lanes / R of them to a k0.
  template <int R, int DIR, bool LAST, class Xch>
  __device__ __forceinline__ static void radix(int j, int lanes, int n, int inv, const float2* tq, Xch xch) {
    for (int i = j; i < RL * n; i += lanes) {
      const int k0 = i * inv >> 16, b = i - k0 * n;
      const int at = LAST ? b * R : b, step = LAST ? 1 : n;
      float2 z[R];
#pragma unroll
      for (int m = 0; m < R; ++m) z[m] = *xch(k0, at + step * m);
      dft<R, DIR>(z);
#pragma unroll
      for (int m = 0; m < R; ++m) {
        if (!LAST && m > 0) z[m] = DIR < 0 ? cmul(z[m], tq[m * n + b]) : cmulc(z[m], tq[m * n + b]);
        *xch(k0, at + step * m) = z[m];
      }
    }
  }
  template <int DIR, class Xch, class Sync>
  __device__ __forceinline__ static void run(float2 (&v)[REGS], int j, const LineArgs& A, const float2* lds, Xch xch,
                                             Sync sync) {
    const int Q = A.lanes;
    dft<RL, DIR>(v);
    *xch(0, j) = v[0];
#pragma unroll
    for (int k = 1; k < RL; ++k) *xch(k, j) = DIR < 0 ? cmul(v[k], lds[k * Q + j]) : cmulc(v[k], lds[k * Q + j]);
    sync();
    int last = A.r1, n = 1, inv = A.inv1;
    if (A.r2 > 1) {
      const float2* tq = lds + A.L;
      switch (A.r1) {
        case 2: radix<2, DIR, false>(j, Q, A.r2, A.inv1, tq, xch); break;
        case 3: radix<3, DIR, false>(j, Q, A.r2, A.inv1, tq, xch); break;
        case 4: radix<4, DIR, false>(j, Q, A.r2, A.inv1, tq, xch); break;
        case 5: radix<5, DIR, false>(j, Q, A.r2, A.inv1, tq, xch); break;
      }
      sync();
      last = A.r2;
      n = A.r1;
      inv = A.inv2;
    }
    switch (last) {
#define GX_CASE(R) \
  case R: radix<R, DIR, true>(j, Q, n, inv, nullptr, xch); break;
      GX_CASE(3) GX_CASE(4) GX_CASE(5) GX_CASE(6) GX_CASE(7) GX_CASE(8) GX_CASE(9) GX_CASE(10)
#undef GX_CASE
    }
    sync();
#pragma unroll
    for (int m = 0; m < RL; ++m) {
      const int p = j + Q * m, k0 = p % RL, k = p / RL;
      const int k2 = A.r2 > 1 ? k * A.inv2 >> 16 : 0, k1 = k - k2 * A.r1;
      v[m] = *xch(k0, k1 * A.r2 + k2);
    }
  }
};
#define GX_FOR_SMOOTH(X) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(15) X(16) X(20)

// Chirp and kernel spectra of one length L and convolution length M (fft.hip): chirp[j] = exp(-i pi (j^2 mod
// 2L) / L), bf / bi the M-point DFTs of the forward / inverse kernels over M.
struct BlueTables {
  int M = 0;
  float2* chirp = nullptr;
  float2* bf = nullptr;
  float2* bi = nullptr;
};
int blue_tables(int L, int M, BlueTables* out);
// The form of lines of L points, 2 <= L <= BLUE_FUSED_MAX, without and with its device tables.
// Rows and columns may be split differently.
LineArgs line_shape(int L, bool rows);
int line_args(int L, bool rows, LineArgs* out);

// f(SmoothLine or BlueLine of A).
template <class F> int with_line(const LineArgs& A, F f) {
  switch (A.RL) {
#define GX_CASE(R) \
  case R:          \
    return f(SmoothLine<R>{});
    GX_FOR_SMOOTH(GX_CASE)
#undef GX_CASE
    default: break;
  }
  switch (A.M) {
#define GX_CASE(N) \
  case N:          \
    return f(BlueLine<N>{});
    GX_FOR_BLUE(GX_CASE)
#undef GX_CASE
    default: return fail(GTOMX_ERR_INTERNAL, "line length not instantiated");
  }
}

// Threads and bytes of dynamic LDS of a workgroup.
template <class LN> unsigned col_threads(const LineArgs& A) { return (unsigned)(LN::lanes(A) << LN::txlog(A)); }
template <class LN> unsigned col_lds(const LineArgs& A) {
  return LN::COL_LDS ? 0 : (unsigned)((LN::tables(A) + (A.L << LN::txlog(A))) * sizeof(float2));
}
// Row pairs of a workgroup of 256 threads.
template <class LN> __host__ __device__ inline int row_pairs(const LineArgs& A) { return 4 * (64 / LN::lanes(A)); }
template <class LN> unsigned row_lds(const LineArgs& A) {
  return LN::ROW_LDS ? 0 : (unsigned)((LN::tables(A) + row_pairs<LN>(A) * LN::row_area(A)) * sizeof(float2));
}
// The workgroup's LDS: FIXED values, or what the launch asked for.
template <int FIXED> __device__ __forceinline__ float2* line_lds() {
  if constexpr (FIXED > 0) {
    __shared__ float2 fixed[FIXED];
    return fixed;
  } else {
    extern __shared__ float2 sized[];
    return sized;
  }
}
// A thread's place in a row kernel: its pair in the workgroup, or -1 for the lanes a
// wave has left over, and j.
template <class LN> __device__ __forceinline__ int row_slot(int t, const LineArgs& A, int* j) {
  const int lane = t % 64, q = lane / LN::lanes(A), per = 64 / LN::lanes(A);
  *j = lane - q * LN::lanes(A);
  return q < per ? t / 64 * per + q : -1;
}

}  // namespace gx
