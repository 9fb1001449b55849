// History correction of the zreion field: bubble mean free paths from random
// skewers (GetBubbleMFP, c++/src/bubblehistory_d2z.C:82-242) and the remap of
// every cell through the corrected history (zreioncorrect and CorrectHistory,
// c++/src/bubblehistory_d2z.C:270-343).
//
//   skewers  one lane per (skewer, ionized fraction) draws start cells from
//            Philox4x32-10 (counter (skewer, fraction, draw, 0), key (seed lo,
//            seed hi)) until zreion > zcur with j, k < N - 2, a bounded number
//            of draws; the wave then walks its 64 skewers in turn, 64 cells at a
//            time, along +y (on a copy with y contiguous, if the walks are many)
//            and +z (periodic) to the first cell with zreion < zcur or back to the
//            start; distance log-uniform in [m - 1, m] cells ([1/2, 1] for m = 1)
//            from counter (skewer, fraction, 0xffffffff, 0); distances and their
//            logs in FP64
//   zvz      one thread per history bin, the corrected-history table in LDS,
//            first bracketing interval as the reference's linear search (by
//            bisection where the table does not decrease)
//   remap    zreion <- zvz[bin(zreion)], bin = (int)((z - 49.9)/dzhistory)
//            clamped to the table (the reference indexes out of bounds for
//            z < 0.01 and z > 49.9)
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

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
// intervals of skewer_distance, for launches with many walks
__global__ void __launch_bounds__(256) k_skewer_logs(double* __restrict__ lg, int n) {
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m <= n) lg[m] = m > 0 ? log((double)m) : log(0.5);
}

// zt[x][z][y] = z[x][y][z], one 64 x 64 tile per block through LDS (N a multiple of 16)
__global__ void __launch_bounds__(256) k_swap_yz(const float* __restrict__ z, float* __restrict__ zt, int N) {
  __shared__ float s[64][65];
  const int c = (threadIdx.x & 15) * 4, r0 = threadIdx.x >> 4;
  const int z0 = blockIdx.x * 64, y0 = blockIdx.y * 64;
  const long long plane = (long long)blockIdx.z * N * N;
#pragma unroll
  for (int r = r0; r < 64; r += 16)
    if (y0 + r < N && z0 + c < N) {
      const float4 v = *reinterpret_cast<const float4*>(z + plane + (long long)(y0 + r) * N + z0 + c);
      s[r][c] = v.x;
      s[r][c + 1] = v.y;
      s[r][c + 2] = v.z;
      s[r][c + 3] = v.w;
    }
  __syncthreads();
#pragma unroll
  for (int r = r0; r < 64; r += 16)
    if (z0 + r < N && y0 + c < N)
      *reinterpret_cast<float4*>(zt + plane + (long long)(z0 + r) * N + y0 + c) =
          make_float4(s[c][r], s[c + 1][r], s[c + 2][r], s[c + 3][r]);
}

// exp(clow + (chigh - clow) frac) cells, clow = log(m - 1) (log 1/2 for m = 1),
// chigh = log m (bubblehistory_d2z.C:185-189,223-227), in FP64 without contraction
// so that the host restatement rounds identically.  lg: k_skewer_logs's table
// (the same bits) or nullptr
__device__ __forceinline__ double skewer_distance(int m, float frac, double cell, const double* __restrict__ lg) {
#pragma clang fp contract(off)
  const double clow = lg ? lg[m - 1] : (m > 1 ? log((double)m - 1.0) : log(0.5));
  const double chigh = lg ? lg[m] : log((double)m);
  return exp(clow + (chigh - clow) * (double)frac) * cell;
}

// Steps from cell c0 of a periodic row of n cells, `step` floats apart, to the first
// one below zc, at most n (back at the start), found by the whole wave: lane l looks
// at step m0 + l + 1.  Wave-uniform arguments and result.
__device__ __forceinline__ int walk_row(const float* __restrict__ row, long long step, int c0, int n, float zc, int m0,
                                        int lane) {
  for (;; m0 += 64) {
    const int m = min(m0 + lane + 1, n);
    int c = c0 + m;
    c = c >= n ? c - n : c;
    const unsigned long long hit = __ballot(m == n || row[c * step] < zc);
    if (hit) return min(m0 + __ffsll(hit), n);
  }
}

// Steps of each lane's walk (lanes that are on; row: its row's offset in f) to the
// first cell below zc, at most n >= 16.  A lane walking alone waits for one load per
// step, and its wave for the longest of 64 walks (256^3, 20000 skewers: 18.2 ms).
// Here 16 lanes look at a walk's first 16 cells, 32 walks in flight; those that go
// on are taken by the whole wave, 64 cells a look and kWalks walks in flight.  Rows of
// fewer than ALONE cells are short enough for lanes alone: 16^3 x 20000 2.30 -> 2.08
// ms, 32^3 x 16 143 -> 119 us (but 32^3 x 20000, with the copy, 1.95 -> 2.35 ms).
constexpr int kWalks = 4;
template <int ALONE>
__device__ __forceinline__ int walks(const float* __restrict__ f, long long row, long long step, int c0, int n, float zc,
                                     bool on, int lane) {
  if (n < ALONE) {
    int k = 0, c = c0;
    if (on) do {
        c = c + 1 == n ? 0 : c + 1;
        ++k;
      } while (k < n && !(f[row + c * step] < zc));
    return k;
  }
  const unsigned long long todo = __ballot(on);
  const int m = (lane & 15) + 1;
  int r = 0;
#pragma unroll 1
  for (int s0 = 0; s0 < 64; s0 += 32) {
    if (!(unsigned)(todo >> s0)) continue;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // lanes that are not on hold a row in range too
      const int src = s0 + 4 * u + (lane >> 4), c = __shfl(c0, src) + m;
      v[u] = f[__shfl(row, src) + (c >= n ? c - n : c) * step];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const unsigned long long hit = __ballot(m == n || v[u] < zc);
      if (lane >> 2 == (s0 >> 2) + u) r = __ffs((int)(hit >> (16 * (lane & 3))) & 0xffff);
    }
  }
  unsigned long long more = __ballot(on && r == 0);
  while (more) {
    int L[kWalks], c[kWalks];
    const float* p[kWalks];
    float v[kWalks];
    const int mm = min(lane + 17, n);
#pragma unroll
    for (int u = 0; u < kWalks; ++u) {
      L[u] = more ? __ffsll(more) - 1 : L[0];
      more &= more - 1;
      c[u] = __builtin_amdgcn_readlane(c0, L[u]);
      p[u] = f + (((long long)__builtin_amdgcn_readlane((int)(row >> 32), L[u]) << 32) |
                  (unsigned)__builtin_amdgcn_readlane((int)row, L[u]));
      v[u] = p[u][(c[u] + mm >= n ? c[u] + mm - n : c[u] + mm) * step];
    }
#pragma unroll
    for (int u = 0; u < kWalks; ++u) {
      const unsigned long long hit = __ballot(mm == n || v[u] < zc);
      const int k = hit ? min(16 + __ffsll(hit), n) : walk_row(p[u], step, c[u], n, zc, 80, lane);
      if (lane == L[u]) r = k;
    }
  }
  return r;
}

// YZ: zyz holds k_swap_yz's copy, which a walk along y reads as whole lines, and lg
// the logarithms; otherwise the walk reads zre, a line per cell (launch_skewers)
template <bool YZ>
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
    // together; the first that serves is drawn again, as keeping three indices of
    // each cost more)
    auto cell = [&](uint32_t a, int& i, int& j, int& k) {
      const uint4 w = philox4x32_10(make_uint4((uint32_t)s, (uint32_t)ix, a, 0u), key);
      i = cell_of(u24(w.x), N);
      j = cell_of(u24(w.y), N);
      k = cell_of(u24(w.z), N);
      return i * NN + (long long)j * N + k;
    };
    found = zre[cell(0u, i0, j0, k0)] > zc && j0 < N - 2 && k0 < N - 2;
    uint32_t at = 0u;
    for (uint32_t a = 1; a < (uint32_t)kMaxStartDraws && !found; a += kWalks) {
      // another skewer already ran out of draws: the call fails, stop early
      if ((a & 255u) == 253u && __hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      float z[kWalks];
      bool in[kWalks];
#pragma unroll
      for (int u = 0; u < kWalks; ++u) {
        int i, j, k;
        z[u] = zre[cell(a + u, i, j, k)];
        in[u] = max(j, k) < N - 2;
      }
#pragma unroll
      for (int u = kWalks - 1; u >= 0; --u)
        if (a + u < (uint32_t)kMaxStartDraws && in[u] && z[u] > zc) at = a + u;
      found = at > 0u;
    }
    if (at > 0u) cell(at, i0, j0, k0);
    if (!found) atomicOr(fail, 1);
  }
  // +y (bubblehistory_d2z.C:159-183) and +z (:196-221): at most N steps each
  constexpr int kAlone = YZ ? 32 : 64;
  const int my = YZ ? walks<kAlone>(zyz, i0 * NN + (long long)k0 * N, 1, j0, N, zc, found, lane)
                    : walks<kAlone>(zre, i0 * NN + k0, N, j0, N, zc, found, lane);
  const int mz = walks<kAlone>(zre, i0 * NN + (long long)j0 * N, 1, k0, N, zc, found, lane);
  double dsum = 0.0;
  if (found) {
    const uint4 wf = philox4x32_10(make_uint4((uint32_t)s, (uint32_t)ix, 0xffffffffu, 0u), key);
    const double dy = skewer_distance(my, u24(wf.x), p.cell, YZ ? lg : nullptr);
    const double dz = skewer_distance(mz, u24(wf.y), p.cell, YZ ? lg : nullptr);
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
      auto at = [&](int q) {
        const float f = (x - c[q]) / (c[q + 1] - c[q]);
        const double z0 = 49.9 + (double)((float)q * dzch);
        const double z1 = 49.9 + (double)((float)(q + 1) * dzch);
        return (float)((double)(1.0f - f) * z0 + (double)f * z1);
      };
      if (rising) {
        int lo = 0, hi = kNCHistory - 1;  // chist[hi] >= x
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (c[mid] >= x) hi = mid;
          else lo = mid + 1;
        }
        const int q = max(hi - 1, 0);
        if (x >= c[q] && x <= c[q + 1]) out = at(q);
      } else {
        for (int q = 0; q < kNCHistory - 1; ++q)
          if (x >= c[q] && x <= c[q + 1]) {
            out = at(q);
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

// Whether the walks pay for k_swap_yz's copy (and k_skewer_logs).  Kernel times with
// / without it: 64^3 x 256 skewers 251 / 277 us, 256^3 x 64 189 / 184, x 256 217 /
// 374, x 20000 4.2 / 22.8 ms; 512^3 x 64 596 / 452 us, x 256 647 / 730; 1024^3 x 1
// 1693 / 83, x 256 2507 / 1358, x 1000 2707 / 2967 us.
static bool many_walks(const SkewerParams& p) { return p.nskewers >= std::max(64, p.N * p.N / 1200); }

hipError_t launch_skewers(const float* zre, const float* zcur, const SkewerParams& p, void* scratch, double* sums,
                          unsigned int* counts, int* fail, hipStream_t s) {
  if (p.N < 16 || p.nskewers < 1 || !scratch) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((p.nskewers + kSkewerThreads - 1) / kSkewerThreads), kNXMfp);
  if (!many_walks(p)) {
    hipLaunchKernelGGL(k_skewers<false>, grid, dim3(kSkewerThreads), 0, s, zre, nullptr, nullptr, zcur, p, sums, counts,
                       fail);
    return hipGetLastError();
  }
  float* zyz = static_cast<float*>(scratch);
  double* lg = reinterpret_cast<double*>(zyz + (long long)p.N * p.N * p.N);
  const unsigned nt = (unsigned)((p.N + 63) / 64);
  hipLaunchKernelGGL(k_skewer_logs, dim3((unsigned)(p.N / 256 + 1)), dim3(256), 0, s, lg, p.N);
  hipLaunchKernelGGL(k_swap_yz, dim3(nt, nt, (unsigned)p.N), dim3(256), 0, s, zre, zyz, p.N);
  hipLaunchKernelGGL(k_skewers<true>, grid, dim3(kSkewerThreads), 0, s, zre, zyz, lg, zcur, p, sums, counts, fail);
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
