// History correction of the zreion field: bubble mean free paths from random
// skewers (GetBubbleMFP, c++/src/bubblehistory_d2z.C:82-242) and the remap of
// every cell through the corrected history (zreioncorrect and CorrectHistory,
// c++/src/bubblehistory_d2z.C:270-343).
//
//   skewers  one lane per (skewer, ionized fraction) draws start cells from
//            Philox4x32-10 (counter (skewer, fraction, draw, 0), key (seed lo,
//            seed hi)) until zreion > zcur with j, k < N - 2, a bounded number
//            of draws; the wave then walks its 64 skewers in turn, 64 cells at a
//            time, along +y (on a copy with y contiguous) and +z (periodic) to the
//            first cell with zreion < zcur or back to the start; distance
//            log-uniform in [m - 1, m] cells ([1/2, 1] for m = 1) from counter
//            (skewer, fraction, 0xffffffff, 0); distances and their logs in FP64
//   zvz      one thread per history bin, the corrected-history table in LDS,
//            first bracketing interval as the reference's linear search (by
//            bisection where the table does not decrease)
//   remap    zreion <- zvz[bin(zreion)], bin = (int)((z - 49.9)/dzhistory)
//            clamped to the table (the reference indexes out of bounds for
//            z < 0.01 and z > 49.9)
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "d2z_device.h"
#include "d2z_kernels.h"

namespace prc {
namespace {

constexpr int kSkewerThreads = 256;

__device__ __forceinline__ float u24(uint32_t w) { return (float)(w >> 8) * 0x1p-24f; }

// (int)(u N) with the reference's wrap (bubblehistory_d2z.C:140-150)
__device__ __forceinline__ int cell_of(float u, int n) {
  int c = (int)(u * (float)n);
  if (c >= n) c -= n;
  if (c < 0) c += n;
  return c;
}

// lg[m] = log m for 1 <= m <= N and lg[0] = log 1/2: the ends of the distance
// intervals of skewer_distance
__global__ void __launch_bounds__(256) k_skewer_logs(double* __restrict__ lg, int n) {
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m <= n) lg[m] = m > 0 ? log((double)m) : log(0.5);
}

// zt[x][z][y] = z[x][y][z], one 32 x 32 tile per block through LDS
__global__ void __launch_bounds__(256) k_swap_yz(const float* __restrict__ z, float* __restrict__ zt, int N) {
  __shared__ float s[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int z0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
  const long long plane = (long long)blockIdx.z * N * N;
  for (int r = ty; r < 32; r += 8)
    if (y0 + r < N && z0 + tx < N) s[r][tx] = z[plane + (long long)(y0 + r) * N + z0 + tx];
  __syncthreads();
  for (int r = ty; r < 32; r += 8)
    if (z0 + r < N && y0 + tx < N) zt[plane + (long long)(z0 + r) * N + y0 + tx] = s[tx][r];
}

// exp(clow + (chigh - clow) frac) cells, clow = log(m - 1) (log 1/2 for m = 1),
// chigh = log m (bubblehistory_d2z.C:185-189,223-227), in FP64 without contraction
// so that the host restatement rounds identically
__device__ double skewer_distance(int m, float frac, double cell, const double* __restrict__ lg) {
#pragma clang fp contract(off)
  const double clow = lg[m - 1];
  const double chigh = lg[m];
  return exp(clow + (chigh - clow) * (double)frac) * cell;
}

// Steps from cell c0 of a periodic row of n cells to the first one below zc, at
// most n (back at the start), found by the whole wave: lane l looks at step
// m0 + l + 1.  Wave-uniform arguments and result.
__device__ __forceinline__ int walk_row(const float* __restrict__ row, int c0, int n, float zc, int m0, int lane) {
  for (;; m0 += 64) {
    const int m = min(m0 + lane + 1, n);
    int c = c0 + m;
    c = c >= n ? c - n : c;
    const unsigned long long hit = __ballot(m == n || row[c] < zc);
    if (hit) return min(m0 + __ffsll(hit), n);
  }
}

// A lane walking its own skewer waits for one load per step, and its wave for the
// longest of its 64 walks: 18.2 ms at 256^3 (20000 skewers, 1000 fractions), with
// the memory and the ALUs nearly idle.  A wave that looks at 64 cells of one
// skewer at a time ends nearly every walk with one load; the first looks of
// kWalks skewers, in both directions, are in flight together.
constexpr int kWalks = 4;

__global__ void __launch_bounds__(kSkewerThreads)
    k_skewers(const float* __restrict__ zre, const float* __restrict__ zyz, const double* __restrict__ lg,
              const float* __restrict__ zcur, SkewerParams p, double* __restrict__ sums,
              unsigned int* __restrict__ counts, int* __restrict__ fail) {
#pragma clang fp contract(off)
  __shared__ unsigned int h[kNMfp];
  __shared__ double ws[kSkewerThreads / 64];
  const int t = threadIdx.x, ix = blockIdx.y, lane = t & 63;
  for (int b = t; b < kNMfp; b += kSkewerThreads) h[b] = 0u;
  __syncthreads();
  const int s = blockIdx.x * kSkewerThreads + t;
  const int N = p.N;
  const long long NN = (long long)N * N;
  const float zc = zcur[ix];
  const uint2 key = make_uint2(p.seed_lo, p.seed_hi);
  int i0 = 0, j0 = 0, k0 = 0;
  bool found = false;
  if (s < p.nskewers) {
    // draw a; the first one alone, then kWalks at a time (their cells are read
    // together, the first that serves is taken)
    auto draw = [&](uint32_t a, int& i, int& j, int& k) {
      const uint4 w = philox4x32_10(make_uint4((uint32_t)s, (uint32_t)ix, a, 0u), key);
      i = cell_of(u24(w.x), N);
      j = cell_of(u24(w.y), N);
      k = cell_of(u24(w.z), N);
      return zre[i * NN + (long long)j * N + k];
    };
    found = draw(0u, i0, j0, k0) > zc && j0 < N - 2 && k0 < N - 2;
    for (uint32_t a = 1; a < (uint32_t)kMaxStartDraws && !found; a += kWalks) {
      // another skewer already ran out of draws: the call fails, stop early
      if ((a & 255u) == 253u && __hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      int i[kWalks], j[kWalks], k[kWalks];
      float z[kWalks];
#pragma unroll
      for (int u = 0; u < kWalks; ++u) z[u] = draw(a + u, i[u], j[u], k[u]);
#pragma unroll
      for (int u = kWalks - 1; u >= 0; --u)
        if (a + u < (uint32_t)kMaxStartDraws && z[u] > zc && j[u] < N - 2 && k[u] < N - 2) {
          found = true;
          i0 = i[u];
          j0 = j[u];
          k0 = k[u];
        }
    }
    if (!found) atomicOr(fail, 1);
  }
  // +y (bubblehistory_d2z.C:159-183) and +z (:196-221): at most N steps each
  int my = 1, mz = 1;
  const unsigned long long todo = __ballot(found);
  for (int s0 = 0; s0 < 64; s0 += kWalks) {
    if (!((todo >> s0) & ((1ull << kWalks) - 1))) continue;
    const float *ry[kWalks], *rz[kWalks];
    int cy[kWalks], cz[kWalks];
    unsigned long long hy[kWalks], hz[kWalks];
    const int m = min(lane + 1, N);
    float vy[kWalks], vz[kWalks];
#pragma unroll
    for (int u = 0; u < kWalks; ++u) {  // lanes without a start cell hold cell (0, 0, 0) or their last draw: in range
      const int ii = __builtin_amdgcn_readlane(i0, s0 + u);
      cy[u] = __builtin_amdgcn_readlane(j0, s0 + u);
      cz[u] = __builtin_amdgcn_readlane(k0, s0 + u);
      ry[u] = zyz + ii * NN + (long long)cz[u] * N;
      rz[u] = zre + ii * NN + (long long)cy[u] * N;
      const int y = cy[u] + m, z = cz[u] + m;
      vy[u] = ry[u][y >= N ? y - N : y];
      vz[u] = rz[u][z >= N ? z - N : z];
    }
#pragma unroll
    for (int u = 0; u < kWalks; ++u) {
      hy[u] = __ballot(m == N || vy[u] < zc);
      hz[u] = __ballot(m == N || vz[u] < zc);
    }
#pragma unroll
    for (int u = 0; u < kWalks; ++u) {
      if (!((todo >> (s0 + u)) & 1)) continue;
      const int ny = hy[u] ? min(__ffsll(hy[u]), N) : walk_row(ry[u], cy[u], N, zc, 64, lane);
      const int nz = hz[u] ? min(__ffsll(hz[u]), N) : walk_row(rz[u], cz[u], N, zc, 64, lane);
      if (lane == s0 + u) {
        my = ny;
        mz = nz;
      }
    }
  }
  double dsum = 0.0;
  if (found) {
    const uint4 wf = philox4x32_10(make_uint4((uint32_t)s, (uint32_t)ix, 0xffffffffu, 0u), key);
    const double dy = skewer_distance(my, u24(wf.x), p.cell, lg);
    const double dz = skewer_distance(mz, u24(wf.y), p.cell, lg);
    dsum = dy + dz;
    // bins of log distance (bubblehistory_d2z.C:191-194,229-232)
    const double ld[2] = {log(dy), log(dz)};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int b = (int)((ld[q] - (double)p.lmin) / (double)p.dmfp);
      if (b >= 0 && b < kNMfp && ld[q] < (double)p.lmax && ld[q] > (double)p.lmin) atomicAdd(&h[b], 1u);
    }
  }
  const double wsum = wave_sum(dsum);
  if (lane == 0) ws[t >> 6] = wsum;
  __syncthreads();
  if (t == 0) {
    double tot = 0.0;
    for (int w = 0; w < kSkewerThreads / 64; ++w) tot += ws[w];
    if (tot != 0.0) atomicAdd(&sums[ix], tot);
  }
  for (int b = t; b < kNMfp; b += kSkewerThreads)
    if (h[b]) atomicAdd(&counts[ix * kNMfp + b], h[b]);
}

// zreioncorrect (bubblehistory_d2z.C:270-299) for every history bin; -1 where
// the bin is 0 or its ionized fraction is 0 (CorrectHistory, :305-314); NaN
// where no interval brackets x (the reference exits there).  rising: chist does
// not decrease anywhere, so the first interval with chist[q] <= x <= chist[q + 1]
// ends at the first entry >= x, found by bisection (14 steps instead of up to
// 10000: 1.1 ms -> about 10 us).
__global__ void __launch_bounds__(256)
    k_zvz(const float* __restrict__ history, const float* __restrict__ chist, float dzch, int rising,
          float* __restrict__ zvz) {
#pragma clang fp contract(off)
  __shared__ float c[kNCHistory];
  for (int q = threadIdx.x; q < kNCHistory; q += 256) c[q] = chist[q];
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kNHistory) return;
  const float x = history[i];
  float out = -1.0f;
  if (i > 0 && x != 0.0f) {
    if (x < c[0]) {
      out = 49.9f;
    } else if (x > c[kNCHistory - 1]) {
      out = 0.01f;
    } else {
      out = __builtin_nanf("");
      int q0 = 0;
      if (rising) {
        int lo = 0, hi = kNCHistory - 1;  // chist[hi] >= x
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (c[mid] >= x) hi = mid;
          else lo = mid + 1;
        }
        q0 = max(hi - 1, 0);
      }
      for (int q = q0; q < kNCHistory - 1; ++q) {
        if (x >= c[q] && x <= c[q + 1]) {
          const float f = (x - c[q]) / (c[q + 1] - c[q]);
          const double z0 = 49.9 + (double)((float)q * dzch);
          const double z1 = 49.9 + (double)((float)(q + 1) * dzch);
          out = (float)((double)(1.0f - f) * z0 + (double)f * z1);
          break;
        }
      }
    }
  }
  zvz[i] = out;
}

__device__ __forceinline__ float remap_one(float z, const float* __restrict__ zvz, double dz, double rdz) {
  const double q = history_q(z, dz, rdz);
  const int b = q >= (double)kNHistory ? kNHistory - 1 : (q > 0.0 ? (int)q : 0);
  return zvz[b];
}

__global__ void __launch_bounds__(256)
    k_remap(float* __restrict__ zre, long long n, const float* __restrict__ zvz, double dz, double rdz) {
  const long long n4 = n >> 2;
  float4* z4 = reinterpret_cast<float4*>(zre);
  const long long stride = (long long)gridDim.x * 256;
  for (long long id = (long long)blockIdx.x * 256 + threadIdx.x; id < n4; id += stride) {
    float4 v = z4[id];
    v.x = remap_one(v.x, zvz, dz, rdz);
    v.y = remap_one(v.y, zvz, dz, rdz);
    v.z = remap_one(v.z, zvz, dz, rdz);
    v.w = remap_one(v.w, zvz, dz, rdz);
    z4[id] = v;
  }
  for (long long id = 4 * n4 + (long long)blockIdx.x * 256 + threadIdx.x; id < n; id += stride)
    zre[id] = remap_one(zre[id], zvz, dz, rdz);
}

}  // namespace

hipError_t launch_skewers(const float* zre, const float* zcur, const SkewerParams& p, void* scratch, double* sums,
                          unsigned int* counts, int* fail, hipStream_t s) {
  if (p.N < 3 || p.nskewers < 1 || !scratch) return hipErrorInvalidValue;
  float* zyz = static_cast<float*>(scratch);
  double* lg = reinterpret_cast<double*>(zyz + (long long)p.N * p.N * p.N);
  const unsigned nt = (unsigned)((p.N + 31) / 32);
  hipLaunchKernelGGL(k_skewer_logs, dim3((unsigned)(p.N / 256 + 1)), dim3(256), 0, s, lg, p.N);
  hipLaunchKernelGGL(k_swap_yz, dim3(nt, nt, (unsigned)p.N), dim3(256), 0, s, zre, zyz, p.N);
  const dim3 grid((unsigned)((p.nskewers + kSkewerThreads - 1) / kSkewerThreads), kNXMfp);
  hipLaunchKernelGGL(k_skewers, grid, dim3(kSkewerThreads), 0, s, zre, zyz, lg, zcur, p, sums, counts, fail);
  return hipGetLastError();
}

hipError_t launch_zvz(const float* history, const float* chist, float dzch, bool rising, float* zvz, hipStream_t s) {
  hipLaunchKernelGGL(k_zvz, dim3((kNHistory + 255) / 256), dim3(256), 0, s, history, chist, dzch, (int)rising, zvz);
  return hipGetLastError();
}

hipError_t launch_remap(float* zre, long long n, const float* zvz, double dz, hipStream_t s) {
  long long g = (n / 4 + 255) / 256;
  if (g > 8192) g = 8192;
  if (g < 1) g = 1;
  hipLaunchKernelGGL(k_remap, dim3((unsigned)g), dim3(256), 0, s, zre, n, zvz, dz, 1.0 / dz);
  return hipGetLastError();
}

}  // namespace prc
