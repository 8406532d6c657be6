// d_PickSubTomogramsDiff2 (src/Correlation/SubTomograms.cu:165-209, kernel
// PickSubTomogramsDiff2Kernel :211-313): for every voxel of the relevant box
// (shift d = index - r/2 around the volume origin) and every orientation a,
//   score = sum over the half-spectrum bins k of |R_a(k) ctf(k) e^{-2 pi i k.d/n} - E(k)|^2,
// and the smallest score with its orientation (strict '<', first wins).
//
// The reference evaluates one sincos per (voxel, bin, orientation). Here the
// sum is expanded,
//   score = sum|R_a ctf|^2 + sum|E|^2 - 2 Re X_a(d),  X_a(d) = sum_k Q_a(k) e^{-2 pi i k.d/n},
// Q_a = R_a ctf conj(E), and X_a is separable along the three axes: z over the
// columns of Q, then y, then x, each over the relevant shifts only. Along an axis
// the frequencies +-k and the shifts +-d share their products: with e = Q(k) + Q(-k)
// and o = Q(k) - Q(-k),
//   X(+-d) = sum_k e cos(2 pi k d / n) -+ i sum_k o sin(2 pi k d / n),
// a quarter of the multiply-adds of the plain sum. The two norms are accumulated in
// double, the score is formed in double and stored as float.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "dev_project.hpp"
#include "runtime.hpp"

namespace gx {
namespace {

constexpr int NBLK = 128;  // reduction blocks per orientation

__device__ double block_sum_d(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
  __syncthreads();
  double s = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < 4; ++w) s += red[w];
  __syncthreads();
  return s;
}

// |E|^2 of each volume (parts[v * NBLK + block]). 0 * ctf takes a CTF that is not
// finite into every score, also where no projection reaches.
__global__ __launch_bounds__(256) void k_diff2_norm(const float2* __restrict__ E, const float* __restrict__ ctf,
                                                    size_t h, double* __restrict__ parts) {
  __shared__ double red[4];
  E += blockIdx.y * h;
  ctf += blockIdx.y * h;
  double acc = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < h; i += (size_t)gridDim.x * 256) {
    const float2 e = E[i];
    acc += (double)e.x * e.x + (double)e.y * e.y + (double)(0.f * ctf[i]);
  }
  const double t = block_sum_d(acc, red);
  if (threadIdx.x == 0) parts[blockIdx.y * NBLK + blockIdx.x] = t;
}

// sums[i] = sum of parts[i*np .. (i+1)*np)
__global__ __launch_bounds__(256) void k_diff2_sum(const double* __restrict__ parts, int np,
                                                   double* __restrict__ sums) {
  __shared__ double red[4];
  double acc = 0;
  for (int i = threadIdx.x; i < np; i += 256) acc += parts[(size_t)blockIdx.x * np + i];
  const double t = block_sum_d(acc, red);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

// The sums of PD shift pairs d = d0 + 1 .. d0 + PD, and of shift 0.
template <int PD> struct ShiftSums {
  float2 c0 = {0.f, 0.f}, ec[PD] = {}, os[PD] = {};
  // frequencies +-k (qm = 0 where they are one bin); w[d] = (cos, sin), wave-uniform
  __device__ __forceinline__ void add(float2 qp, float2 qm, const float2* __restrict__ w) {
    const float2 e = make_float2(qp.x + qm.x, qp.y + qm.y), o = make_float2(qp.x - qm.x, qp.y - qm.y);
    c0.x += e.x;
    c0.y += e.y;
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      ec[d].x = fmaf(e.x, w[d].x, ec[d].x);
      ec[d].y = fmaf(e.y, w[d].x, ec[d].y);
      os[d].x = fmaf(o.x, w[d].y, os[d].x);
      os[d].y = fmaf(o.y, w[d].y, os[d].y);
    }
  }
  // shift j - r/2 to out[j * stride]
  __device__ __forceinline__ void store(float2* __restrict__ out, size_t stride, int r, int d0) const {
    const int h = r / 2;
    if (d0 == 0) out[h * stride] = c0;
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      const int s = d0 + d + 1;
      if (h + s < r) out[(h + s) * stride] = make_float2(ec[d].x + os[d].y, ec[d].y - os[d].x);
      if (h - s >= 0) out[(h - s) * stride] = make_float2(ec[d].x - os[d].y, ec[d].y + os[d].x);
    }
  }
};

// T[(v nb + a) rz + dz][c] = sum over kz of Q_a, and the partial sums of |R_a ctf|^2
// per (v, a) and wave. A lane is one column c = ky nh + kx; a wave runs to the largest
// |kz| inside the sphere of radius n/2 on any of its columns (R is zero beyond, half
// of the half spectrum). Bound by its loads from the caches, 20 bytes per bin,
// orientation and volume, and the waves in flight to hide them: several orientations
// to a lane share E and ctf but cost registers (64^3 x 8 volumes x 250 orientations,
// the whole search: 0.73 ms with one, 0.89 with two, 1.06 with four). Grid: x = waves
// / 4, y = volume x chunk of PD shift pairs, z = orientation, so that the volumes
// read the same R one after the other.
template <int PD>
__global__ __launch_bounds__(256) void k_diff2_z(const float2* __restrict__ R, const float2* __restrict__ E,
                                                    const float* __restrict__ ctf, const float2* __restrict__ W,
                                                    int wd, int chunks, int n, int r, int nb,
                                                    float2* __restrict__ T, double* __restrict__ parts) {
  const int nh = n / 2 + 1;
  const size_t C = (size_t)n * nh, h = C * n;
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + threadIdx.x / 64);
  const int nwaves = gridDim.x * 4;
  const int v = blockIdx.y / chunks, d0 = (blockIdx.y % chunks) * PD, a = blockIdx.z;
  const size_t col = (size_t)wave * 64 + threadIdx.x % 64;
  const bool ok = col < C;
  const size_t c = ok ? col : C - 1;
  const int kx = (int)(c % nh), iy = (int)(c / nh), ky = iy < n - iy ? iy : n - iy;
  const int q = n / 2 * (n / 2) - kx * kx - ky * ky;
  int zl = -1;
  if (ok && q >= 0) {
    zl = (int)sqrtf((float)q);
    if (zl * zl > q) --zl;
    if ((zl + 1) * (zl + 1) <= q) ++zl;
  }
  for (int o = 32; o > 0; o >>= 1) zl = max(zl, __shfl_xor(zl, o));
  const int zmax = __builtin_amdgcn_readfirstlane(zl);
  E += v * h;
  ctf += v * h;
  R += a * h;
  ShiftSums<PD> S;
  double norm = 0;
  auto product = [&](float2 x, float ct, float2 e) {
    const float2 y = make_float2(x.x * ct, x.y * ct);
    norm += (double)y.x * y.x + (double)y.y * y.y;
    return make_float2(y.x * e.x + y.y * e.y, y.y * e.x - y.x * e.y);
  };
  const float2 zero = make_float2(0.f, 0.f);
  auto single = [&](int k) {  // kz = 0 and, on the column (0, 0) only, kz = n/2
    const size_t p = k * C + c;
    S.add(product(R[p], ctf[p], E[p]), zero, W + (size_t)k * wd + d0);
  };
  if (zmax >= 0) single(0);
  const int zpair = min(zmax, n / 2 - 1);
  for (int k = 1; k <= zpair; ++k) {
    const size_t p = k * C + c, m = (n - k) * C + c;
    const float2 qp = product(R[p], ctf[p], E[p]), qm = product(R[m], ctf[m], E[m]);
    S.add(qp, qm, W + (size_t)k * wd + d0);
  }
  if (zmax == n / 2) single(n / 2);
  double t = ok ? norm : 0.0;
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o);
  if (d0 == 0 && threadIdx.x % 64 == 0) parts[((size_t)v * nb + a) * nwaves + wave] = t;
  if (ok) S.store(T + ((size_t)v * nb + a) * r * C + c, C, r, d0);
}

// out[item][j][kx] = sum over ky of in[item][ky][kx], the columns of all items in a
// row over the lanes (a half spectrum's row seldom fills whole waves). Grid: y =
// chunk of PD shift pairs.
template <int PD>
__global__ __launch_bounds__(256) void k_diff2_y(const float2* __restrict__ in, float2* __restrict__ out,
                                                 const float2* __restrict__ W, int wd, int n, int r, size_t items) {
  const int nh = n / 2 + 1;
  const size_t col = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (col >= items * nh) return;
  const size_t item = col / nh;
  const int kx = (int)(col % nh), d0 = blockIdx.y * PD;
  const float2* src = in + item * n * nh + kx;
  ShiftSums<PD> S;
  const float2 zero = make_float2(0.f, 0.f);
  S.add(src[0], zero, W + d0);
#pragma unroll 4
  for (int k = 1; k < n / 2; ++k)
    S.add(src[(size_t)k * nh], src[(size_t)(n - k) * nh], W + (size_t)k * wd + d0);
  S.add(src[(size_t)(n / 2) * nh], zero, W + (size_t)(n / 2) * wd + d0);
  S.store(out + item * r * nh + kx, nh, r, d0);
}

// The x axis, real part only, and the running minimum over the nb orientations of
// this batch (strict '<', the first wins). A block is one row (dz, dy) of one volume:
// 32 orientations x 8 shift pairs at a time. best / angle are [dz][dy][dx].
__global__ __launch_bounds__(256) void k_diff2_x_min(const float2* __restrict__ T, const float2* __restrict__ W,
                                                     int wd, int n, int rx, int ryz, int nb, int angle0,
                                                     const double* __restrict__ A, const double* __restrict__ Ee,
                                                     float* __restrict__ best, float* __restrict__ angle) {
  __shared__ double sb[2][4][8];
  __shared__ int sk[2][4][8];
  const int nh = n / 2 + 1, row = blockIdx.x, v = blockIdx.y;
  const int slot = threadIdx.x % 8, al = threadIdx.x / 8;
  const size_t base = (size_t)v * nb;
  const double e2 = Ee[v];
  for (int d0 = 0; d0 <= rx / 2; d0 += 8) {
    const int d = d0 + slot;
    double b[2] = {1e300, 1e300};
    int k[2] = {0x7fffffff, 0x7fffffff};
    for (int a = al; a < nb; a += 32) {
      const float2* t = T + ((base + a) * ryz + row) * nh;
      float ec = 0.f, os = 0.f;
#pragma unroll 4
      for (int kx = 0; kx < nh; ++kx) {
        const float2 w = W[(size_t)kx * wd + d], x = t[kx];
        ec = fmaf(x.x, w.x, ec);
        os = fmaf(x.y, w.y, os);
      }
      const double n2 = A[base + a] + e2;
      const double s[2] = {n2 - 2.0 * (double)(ec + os), n2 - 2.0 * (double)(ec - os)};
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (s[i] < b[i]) {
          b[i] = s[i];
          k[i] = a;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      for (int o = 8; o < 64; o <<= 1) {
        const double ob = __shfl_xor(b[i], o);
        const int ok = __shfl_xor(k[i], o);
        if (ob < b[i] || (ob == b[i] && ok < k[i])) {
          b[i] = ob;
          k[i] = ok;
        }
      }
      if (threadIdx.x % 64 < 8) {
        sb[i][threadIdx.x / 64][slot] = b[i];
        sk[i][threadIdx.x / 64][slot] = k[i];
      }
    }
    __syncthreads();
    if (threadIdx.x < 16) {
      const int i = threadIdx.x / 8, s = d0 + slot, j = i == 0 ? rx / 2 + s : rx / 2 - s;
      double bb = sb[i][0][slot];
      int kk = sk[i][0][slot];
      for (int w = 1; w < 4; ++w)
        if (sb[i][w][slot] < bb || (sb[i][w][slot] == bb && sk[i][w][slot] < kk)) {
          bb = sb[i][w][slot];
          kk = sk[i][w][slot];
        }
      const size_t o = ((size_t)v * ryz + row) * rx + j;
      if (j >= 0 && j < rx && !(i == 1 && s == 0) && (float)bb < best[o]) {
        best[o] = (float)bb;
        angle[o] = (float)(angle0 + kk);
      }
    }
    __syncthreads();
  }
}

// W[k * wd + d] = (cos, sin)(2 pi k d / n) for k <= n/2 and d < wd. d = 0 comes first:
// the kernels of z and y are given W + 1.
std::vector<float2> shift_phases(int n, int wd) {
  std::vector<float2> base(n), w((size_t)(n / 2 + 1) * wd);
  const long double two_pi = 6.283185307179586476925286766559005768L;
  for (int m = 0; m < n; ++m)
    base[m] = make_float2((float)std::cos(two_pi * m / n), (float)std::sin(two_pi * m / n));
  base[n / 2].y = 0.f;
  for (int k = 0; k <= n / 2; ++k)
    for (int d = 0; d < wd; ++d) w[(size_t)k * wd + d] = base[(size_t)k * d % n];
  return w;
}

// f(integral_constant PD): the pairs of r shifts in one chunk where they fit.
template <class F> int with_pairs(int r, F f) {
  const int d = r / 2;
  if (d <= 2) return f(std::integral_constant<int, 2>{});
  if (d <= 4) return f(std::integral_constant<int, 4>{});
  if (d <= 6) return f(std::integral_constant<int, 6>{});
  return f(std::integral_constant<int, 8>{});
}

}  // namespace
}  // namespace gx

using namespace gx;

extern "C" int gtomx_pick_subtomograms_diff2(const gtomx_complex* d_projectorft, float oversample,
                                             gtomx_int3 dimsprojector, const gtomx_complex* d_expft,
                                             const float* d_ctf, gtomx_int3 dimsvolume, unsigned nvolumes,
                                             gtomx_int3 dimsrelevant, const gtomx_float3* h_angles, unsigned nangles,
                                             float* d_bestdiff2, float* d_bestangle, void* stream) {
  if (!d_projectorft || !d_expft || !d_ctf || !d_bestdiff2 || !d_bestangle)
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL device buffer");
  if (nangles > 0 && !h_angles) return fail(GTOMX_ERR_INVALID_ARGUMENT, "h_angles is NULL");
  const int n = dimsvolume.x, p = dimsprojector.x;
  if (dimsvolume.y != n || dimsvolume.z != n || n < 2 || n % 2 || n > 1024)
    return fail(GTOMX_ERR_UNSUPPORTED, "volumes must be even cubes of side <= 1024");
  if (dimsprojector.y != p || dimsprojector.z != p || p < 2 || p % 2 || p > 512)
    return fail(GTOMX_ERR_UNSUPPORTED, "projector must be an even cube of side <= 512");
  const int rx = dimsrelevant.x, ry = dimsrelevant.y, rz = dimsrelevant.z;
  if (rx < 1 || ry < 1 || rz < 1 || rx > n || ry > n || rz > n)
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "dimsrelevant must lie within the volume");
  if (nvolumes == 0) return fail(GTOMX_ERR_INVALID_ARGUMENT, "nvolumes must be positive");
  if (!(oversample > 0.f) || !std::isfinite(oversample))
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "projectoroversample must be positive");
  hipStream_t s = as_stream(stream);
  const int nh = n / 2 + 1;
  const size_t H = (size_t)nh * n * n;
  const size_t Vr = (size_t)rx * ry * rz;
  // d_ValueFill(best, 1e30), angle 0 (src/Correlation/SubTomograms.cu:182-183)
  GX_TRY(fill_f32(d_bestdiff2, Vr * nvolumes, 1e30f, s));
  GX_TRY(fill_f32(d_bestangle, Vr * nvolumes, 0.f, s));
  if (nangles == 0) return GTOMX_OK;

  // Orientations per batch: 32, and for small volumes as many as keep the projections
  // within 128 MB, which every volume reads again; volumes per launch while their
  // T stays within 256 MB (and their chunks of shifts within a grid's y).
  const size_t C = (size_t)nh * n;
  const unsigned most = (unsigned)std::min<size_t>(256, std::max<size_t>(32, ((size_t)128 << 20) / (H * 8)));
  const unsigned batches = (nangles + most - 1) / most, B = (nangles + batches - 1) / batches;
  const unsigned VG = (unsigned)std::min<size_t>(
      {(size_t)nvolumes, (size_t)1000, std::max<size_t>(1, ((size_t)256 << 20) / ((size_t)B * rz * C * 8))});
  const unsigned gz = (unsigned)((C + 255) / 256);  // workgroups over the columns
  const int wd = 1 + (std::max({rx, ry, rz}) / 2 + 7) / 8 * 8 + 7;

  std::vector<float> h_mats(9 * (size_t)nangles);
  GX_TRY(gtomx_projector_matrices(h_angles, nangles, oversample, h_mats.data()));
  const std::vector<float2> w = shift_phases(n, wd);
  StreamScratch mats, W, R, T1, T2, sums;
  GX_TRY(mats.take((h_mats.size() + 1) / 2, s, true));
  GX_TRY(W.take(w.size(), s, true));
  GX_TRY(R.take((size_t)B * H, s, true));
  GX_TRY(T1.take((size_t)VG * B * rz * C, s, true));
  GX_TRY(T2.take((size_t)VG * B * rz * ry * nh, s, true));
  // doubles: |R ctf|^2 per (volume, orientation) and its parts, |E|^2 and its parts
  const size_t nparts = std::max((size_t)VG * B * gz * 4, (size_t)nvolumes * NBLK);
  GX_TRY(sums.take((size_t)VG * B + nvolumes + nparts, s, true));
  double *asum = reinterpret_cast<double*>(sums.p), *esum = asum + (size_t)VG * B, *parts = esum + nvolumes;
  float* d_mats = reinterpret_cast<float*>(mats.p);
  GX_HIP(hipMemcpyAsync(d_mats, h_mats.data(), h_mats.size() * sizeof(float), hipMemcpyHostToDevice, s));
  GX_HIP(hipMemcpyAsync(W.p, w.data(), w.size() * sizeof(float2), hipMemcpyHostToDevice, s));
  const float2* E = reinterpret_cast<const float2*>(d_expft);
  for (unsigned v0 = 0; v0 < nvolumes; v0 += 32768) {
    const unsigned nv = std::min(32768u, nvolumes - v0);
    hipLaunchKernelGGL(k_diff2_norm, dim3(NBLK, nv), dim3(256), 0, s, E + v0 * H, d_ctf + v0 * H, H,
                       parts + (size_t)v0 * NBLK);
    GX_LAUNCHED("k_diff2_norm");
  }
  hipLaunchKernelGGL(k_diff2_sum, dim3(nvolumes), dim3(256), 0, s, parts, NBLK, esum);
  GX_LAUNCHED("k_diff2_sum");

  for (unsigned b0 = 0; b0 < nangles; b0 += B) {
    const unsigned nb = std::min(B, nangles - b0);
    // R_a: the projections at the volume size (d_rlnProject, :195), rmax = n/2, for all volumes
    GX_TRY(project_launch(reinterpret_cast<const float2*>(d_projectorft), p, R.p, n, (unsigned)(n / 2),
                          d_mats + 9 * (size_t)b0, nb, s));
    for (unsigned v0 = 0; v0 < nvolumes; v0 += VG) {
      const unsigned nv = std::min(VG, nvolumes - v0);
      // one CTF per volume (src/Correlation/SubTomograms.cu:199)
      const float2* Ev = E + (size_t)v0 * H;
      const float* cv = d_ctf + (size_t)v0 * H;
      GX_TRY(with_pairs(rz, [&](auto pd) {
        constexpr int PD = decltype(pd)::value;
        const unsigned chunks = (unsigned)std::max(1, (rz / 2 + PD - 1) / PD);
        hipLaunchKernelGGL((k_diff2_z<PD>), dim3(gz, nv * chunks, nb), dim3(256), 0, s, R.p, Ev, cv, W.p + 1, wd,
                           (int)chunks, n, rz, (int)nb, T1.p, parts);
        GX_LAUNCHED("k_diff2_z");
        return (int)GTOMX_OK;
      }));
      hipLaunchKernelGGL(k_diff2_sum, dim3(nv * nb), dim3(256), 0, s, parts, (int)gz * 4, asum);
      GX_LAUNCHED("k_diff2_sum");
      GX_TRY(with_pairs(ry, [&](auto pd) {
        constexpr int PD = decltype(pd)::value;
        const size_t items = (size_t)nv * nb * rz, blocks = (items * nh + 255) / 256;
        hipLaunchKernelGGL((k_diff2_y<PD>), dim3((unsigned)blocks, (unsigned)std::max(1, (ry / 2 + PD - 1) / PD)),
                           dim3(256), 0, s, T1.p, T2.p, W.p + 1, wd, n, ry, items);
        GX_LAUNCHED("k_diff2_y");
        return (int)GTOMX_OK;
      }));
      hipLaunchKernelGGL(k_diff2_x_min, dim3((unsigned)(ry * rz), nv), dim3(256), 0, s, T2.p, W.p, wd, n, rx, ry * rz,
                         (int)nb, (int)b0, asum, esum + v0, d_bestdiff2 + (size_t)v0 * Vr, d_bestangle + (size_t)v0 * Vr);
      GX_LAUNCHED("k_diff2_x_min");
    }
  }
  GX_HIP(hipStreamSynchronize(s));  // the results are ready on return
  return GTOMX_OK;
}
