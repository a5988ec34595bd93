// USFFT Radon transform R / RT for gfx950 (src/holotomocupy/tomo.py:12-116,
// gridding kernel src/holotomocupy/cuda_kernels.py:3-76).
//
//   R(obj)  = c1d IFFT1(c1d gather(c2d FFT2(c2d embed(obj phi))) / n) / 4   (1/n applied with the 1/4, rounded once)
//   RT(d)   = crop(c2d IFFT2(c2d scatter(c1d FFT1(c1d d)))) phi
//
// c1d[k] = (-1)^(k+1), c2d[i,j] = (-1)^(i+j) on the 2n x 2n grid.  The 2-D
// transforms run as two LDS FFT passes (rows, then columns; only the n
// non-zero rows of the embedded slice are transformed along x), with the sign
// modulations, zero-embedding, cropping and deapodisation folded into the
// loads and stores.  The 9x9 Gaussian gridding taps of every polar sample are
// built once per plan in FP64 (stored FP32).  Between the grid and the line
// spectra (slices fastest) both directions are matrix products over all
// slices: the forward over groups of samples whose windows share a patch of the
// grid, the adjoint over 4x4 tiles of the grid and the samples that touch them
// -- the reference's atomic scatter in a fixed summation order.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/htamd.h"
#include "fft_any.hpp"
#include "fft_lds.hpp"
#include "htamd_bspline.hpp"
#include "htamd_internal.hpp"

namespace htamd {

constexpr int kWRow = 16;  // a sample's weights along an axis: 3 zeros, 9 taps, 4 zeros

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));  // an odd slice count leaves rows 8-byte aligned

struct TomoArgs {
  int n = 0, nz = 0, ntheta = 0;
  const float* phi = nullptr;      // [n, n] deapodisation (mask and scale included)
  const float2* tw2 = nullptr;     // twiddles of length 2n
  const float2* tw1 = nullptr;     // twiddles of length n
  // gridding taps of polar sample s = theta n + t, built in FP64 on the host:
  // weights along x at wt[2 kWRow s + 3 + i] and along y at wt[2 kWRow s +
  // kWRow + 3 + i], tap i < 9, zero elsewhere
  const float* wt = nullptr;
  // the samples by tile of 4x4 grid points: entries [tp[t], tp[t + 1]) of tile
  // t = row n / 2 + column touch it, each (sample, oy << 8 | ox) with ox the
  // index in the sample's x weights of the tile's first column (oy of its row)
  const int* tp = nullptr;
  const int2* te = nullptr;
  // the samples for the forward gather: groups of up to 16 whose first taps lie
  // in one cell of 4 rows x 8 columns, ge[16 g + i] = (sample or -1, oy << 8 |
  // ox) with (oy, ox) the first tap's place in the cell; gc[g] = the cell's
  // place in its region (row << 8 | column); work item = (column, row of the
  // kRG x kRG region, first group, groups)
  const int4* items = nullptr;
  const int2* ge = nullptr;
  const int* gc = nullptr;
  int nitems = 0;
  int sparse = 0;                  // the groups are of regions, one to a work item
  float2* W = nullptr;             // [nz, n, 2n]
  float2* G = nullptr;             // [nz, 2n, 2n]
  float2* Sh = nullptr;            // [ntheta n, nz] line spectra, slices fastest
  const int* heavy = nullptr;      // tiles with more than kHeavyTile entries, longest first
  int nheavy = 0;
  int parts = 0;                   // sums that a heavy list is cut into (4 or 16)
  // per-bin factor of the adjoint's line transform (NULL = none): the
  // detector filter of filtered back-projection, shifted by n/2 to the bins
  // of the c1d-modulated transform and scaled by sqrt(n / ntheta)
  const float* filt = nullptr;
};

__device__ __forceinline__ float sgnf(int k) { return (k & 1) ? -1.0f : 1.0f; }

template <typename T> __device__ __forceinline__ float2 ld_c(const T* p, int64_t i);
template <> __device__ __forceinline__ float2 ld_c<float>(const float* p, int64_t i) { return make_float2(p[i], 0.f); }
template <> __device__ __forceinline__ float2 ld_c<float2>(const float2* p, int64_t i) { return p[i]; }
template <typename T> __device__ __forceinline__ void st_c(T* p, int64_t i, float2 v);
template <> __device__ __forceinline__ void st_c<float>(float* p, int64_t i, float2 v) { p[i] = v.x; }
template <> __device__ __forceinline__ void st_c<float2>(float2* p, int64_t i, float2 v) { p[i] = v; }

// ---- forward pass A: rows of the embedded slice (length 2n) ----------------
template <int N2, int E, typename TI>
__global__ __launch_bounds__(256) void tomo_rows_fwd_k(TomoArgs a, const TI* __restrict__ obj) {
  constexpr int T = N2 / E, ROWS = 256 / T;
  __shared__ float2 lds[ROWS * fft_buf<N2>()];
  const int n = N2 / 2, h = N2 / 4;
  const int r = threadIdx.x / T, t = threadIdx.x % T;
  const int64_t row = (int64_t)blockIdx.x * ROWS + r;  // (z, i'), i' < n
  const bool valid = row < (int64_t)a.nz * n;
  const int64_t z = valid ? row / n : 0;
  const int ip = valid ? (int)(row % n) : 0;
  float2* s = lds + r * fft_buf<N2>();
  FftTw<N2, E> twr;
  fft_load_twiddles<N2, E>(twr, t, a.tw2);
  const TI* src = obj + (z * n + ip) * (int64_t)n;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + e * T;
    float2 v = make_float2(0.f, 0.f);
    if (p >= h && p < h + n) {
      const int jp = p - h;
      v = cscale(ld_c<TI>(src, jp), a.phi[ip * n + jp] * sgnf(ip + h + p));
    }
    s[fpad(p)] = v;
  }
  lds_sync<wave_private<N2, E>()>();
  fft_lds<N2, E, false, kMaxRadix, wave_private<N2, E>()>(s, t, twr);
  if (valid) {
    float2* dst = a.W + (z * n + ip) * (int64_t)N2;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = t + e * T;
      dst[k] = cscale(s[fpad(k)], sgnf(k));
    }
  }
}

// ---- forward pass B: columns (n non-zero rows embedded in 2n) ---------------
template <int N2, int E, int C>
__global__ __launch_bounds__(C*(N2 / E)) void tomo_cols_fwd_k(TomoArgs a) {
  constexpr int T = N2 / E, NT = C * T, LS = col_stride<N2, C>();
  __shared__ float2 lds[C * LS];
  const int n = N2 / 2, h = N2 / 4;
  const int tiles = N2 / C;
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t z = tile / tiles;
  const int k0 = (int)(tile % tiles) * C;
  const int cc = threadIdx.x / T, t = threadIdx.x % T;
  FftTw<N2, E> twr;
  fft_load_twiddles<N2, E>(twr, t, a.tw2);
  const float2* src = a.W + z * (int64_t)n * N2 + k0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int idx = threadIdx.x + e * NT;
    const int c = idx % C, i = idx / C;
    lds[c * LS + fpad(i)] = (i >= h && i < h + n) ? src[(i - h) * N2 + c] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft_lds<N2, E, false, kMaxRadix, wave_private<N2, E>()>(lds + cc * LS, t, twr);
  if constexpr (wave_private<N2, E>()) __syncthreads();  // the store crosses columns
  float2* dst = a.G + z * (int64_t)N2 * N2 + k0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int idx = threadIdx.x + e * NT;
    const int c = idx % C, k = idx / C;
    dst[k * N2 + c] = cscale(lds[c * LS + fpad(k)], sgnf(k));
  }
}

// ---- forward pass C: the grid at the samples ---------------------------------
// Sh[s][z] = c1d sum over the 9x9 window of sample s of wy wx G[z][g], as the
// adjoint (see tomo_grid_k) in FP32 matrix products.  Up to 16 samples whose
// windows start in one cell of 4x8 points have their windows inside 12 rows of
// 16 points: a row is a product of 16 slices x 16 points with the 16 x 16
// matrix of x weights, and its result is added with the lane's sample's y
// weight, as the sum per sample would.
// 81 of the patch's 192 points count for a sample, and far from the centre a
// cell holds about 8 samples at 256^2, 384 angles: 4x4 cells take a third more
// products, 8x8 cells as many more at that density (fewer at sparser ones).
// A workgroup stages a region of kRG x kRG first taps with the margin of the
// windows, wrapped on the 2n grid, for Z slices (slices fastest, a point's
// row padded to Z + 1: the lanes of a read are the slices of 4 neighbouring
// points, the lanes of a staging write 12 pairs of points of one slice), and
// its wavefronts take the groups in turn.
// The 16 rows of a product are 16 slices (re and im in two products), 8 slices
// x (re, im), or 4 slices x (re, im) x two patch rows; a sample's sum runs in the
// same order in all three, and few slices pay neither for staging nor for
// products of slices that are not there (one slice of 512^2, 451 angles: R takes
// 99 us in sixteens, 47 us in fours; 8 slices of 512^2, 128 angles 102 and 74).
// Each sample's two weight rows are read once per group; lane l holds sample
// l % 16 and the points 4 j + l / 16 of a row.
// Few angles leave a cell one or two samples: then a group is 16 samples of a
// region (SPARSE), a workgroup takes one group, and its wavefronts share the
// rows of the region's patch.  The plan takes the form of fewer steps, whatever
// the slab, so that slices keep their bits (in sixteens, R at 8 slices of 512^2,
// 64 angles: 111 us with cells, 92 with regions; 100 slices of 256^2, 100
// angles: 272 and 316).
// 256 slices of 256^2, 384 angles: 974 us with a thread per sample and four
// slices -> 450 us (the products are 177 us).
constexpr int kTL = 9;                        // taps along an axis
constexpr int kRG = 16, kRP = kRG + kTL - 1;  // region and its staged edge
constexpr int kCellY = 4, kCellX = 8;
constexpr int kItemGroups = 16;               // groups of a work item
constexpr int kGatherWaves = 8;
constexpr int kStageSteps = 96;               // a region's staging, in steps of products (see the plan)

// The patch of points a group's windows lie in: that of one cell, or (SPARSE)
// of the whole region.
template <bool SPARSE>
struct GatherShape {
  static constexpr int NY = SPARSE ? kRP : kCellY + kTL - 1;                 // rows
  static constexpr int NX = (SPARSE ? kRP : kCellX + kTL - 1) / 4;           // steps of a row
  static constexpr int NR = SPARSE ? kRP / kGatherWaves : NY;                // rows of a wavefront
};

template <bool SPARSE, int Z>
__global__ __launch_bounds__(64 * kGatherWaves) __attribute__((amdgpu_waves_per_eu(Z < 16 ? 6 : 4))) void tomo_gather_k(
    TomoArgs a, int zper) {
  using S = GatherShape<SPARSE>;
  static_assert(Z == 16 || Z == 8 || Z == 4, "rows of a product: slices, slices x (re, im), two patch rows of these");
  constexpr int ZP = Z + 1;                  // pitch of a staged point
  constexpr int NA = 1 + Z / 16;             // products of a step: re and im, or both in one
  constexpr int P = Z == 4 ? 2 : 1;          // patch rows in a product: r and r + NS
  constexpr int NS = (S::NR + P - 1) / P;
  __shared__ float2 tile[kRP * kRP * ZP];
  const int4 it = a.items[xcd_tile(blockIdx.x, gridDim.x)];
  const int z0 = blockIdx.y * zper, nzb = min(zper, a.nz - z0);
  const int n2 = 2 * a.n;
  const int64_t plane = (int64_t)n2 * n2;
  const int gy0 = it.y * kRG, gx0 = it.x * kRG;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int q = lane & 15, kk = lane >> 4;
  // the lane's sample of a group and its weights
  int s = 0, cell = 0;
  float wx[S::NX], wy[S::NR];
  auto group = [&](int g) {
    const int2 en = a.ge[16 * g + q];
    cell = a.gc[g];
    s = en.x;
    const int ox = en.y & 0xff, oy = en.y >> 8;
    const float* w = a.wt + (int64_t)max(s, 0) * (2 * kWRow);
#pragma unroll
    for (int j = 0; j < S::NX; ++j) {
      const int i = 4 * j + kk - ox;  // tap
      wx[j] = s >= 0 && i >= 0 && i < kTL ? w[3 + i] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < S::NR; ++r) {
      const int i = (SPARSE ? wv + r * kGatherWaves : r) - oy;
      wy[r] = !SPARSE || (i >= 0 && i < kTL) ? w[kWRow + 3 + i] : 0.f;
    }
  };
  if constexpr (SPARSE) group(it.z);  // in flight with the staging
  constexpr int PP = kRP / 2;  // pairs of points of a row (2n is even: the wrap splits none)
  constexpr int NT = 64 * kGatherWaves, NP = Z * kRP * PP, NL = (NP + NT - 1) / NT;
  f32x4 v[NL];
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int idx = threadIdx.x + k * NT, zr = idx / PP, x = (idx - zr * PP) * 2;
    const int z = zr / kRP, r = zr - z * kRP;
    int gr = gy0 + r, gx = gx0 + x;
    gr -= gr >= n2 ? n2 : 0;
    gx -= gx >= n2 ? n2 : 0;
    if constexpr (Z == 16) v[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (z < nzb) v[k] = *reinterpret_cast<const f32x4u*>(a.G + (z0 + z) * plane + (int64_t)gr * n2 + gx);
  }
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int idx = threadIdx.x + k * NT, zr = idx / PP, x = (idx - zr * PP) * 2;
    const int z = zr / kRP, r = zr - z * kRP;
    float2* t = tile + (r * kRP + x) * ZP + z;
    if (Z < 16 && z >= nzb) continue;  // rows of the product that no slice has stay as they are
    t[0] = make_float2(v[k].x, v[k].y);
    t[ZP] = make_float2(v[k].z, v[k].w);
  }
  __syncthreads();
  // SPARSE: one group, whose rows the wavefronts share (wv, wv + 8, wv + 16)
  for (int g = SPARSE ? it.z : it.z + wv; g < it.z + it.w; g += SPARSE ? 1 : kGatherWaves) {
    if constexpr (!SPARSE) group(g);
    constexpr int RS = SPARSE ? kGatherWaves : 1;  // from one of the wavefront's rows to the next
    const int at = (((cell >> 8) * kCellY + (SPARSE ? wv : 0)) * kRP + (cell & 0xff) * kCellX + kk) * ZP;
    // the lane's float of a point (Z < 16); of a second patch row that is not
    // there the first is read again, and not added
    const int lf = P == 1 ? q : (q & 7) + (q >> 3) * 2 * NS * RS * kRP * ZP;
    const int lf1 = S::NR % P == 0 ? lf : q & 7;  // in the last step
    f32x4 sum[NA], acc[NS][NA];
#pragma unroll
    for (int c = 0; c < NA; ++c) sum[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < NS; ++r) {
#pragma unroll
      for (int c = 0; c < NA; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < S::NX; ++j) {
        const float2* t = tile + at + (r * RS * kRP + 4 * j) * ZP;
        if constexpr (Z == 16) {
          const float2 b = t[q];
          acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.x, wx[j], acc[r][0], 0, 0, 0);
          acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.y, wx[j], acc[r][1], 0, 0, 0);
        } else {
          const float b = reinterpret_cast<const float*>(t)[r + 1 < NS ? lf : lf1];
          acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, wx[j], acc[r][0], 0, 0, 0);
        }
      }
#pragma unroll
      for (int c = 0; c < NA; ++c) sum[c] += wy[r] * acc[r][c];
    }
    if constexpr (P == 2) {  // the upper lanes hold rows NS and on, which follow the others in the sum
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[0][i] = __shfl(sum[0][i], lane & 31, 64);
#pragma unroll
      for (int r = NS; r < S::NR; ++r) sum[0] += wy[r] * acc[r - NS][0];
    }
    // rows 4 (l / 16) + i of the products are slices (below 16 re and im of two
    // of them), columns q samples; c1d[t] = -(-1)^t, and t has the parity of s (n
    // is even)
    constexpr int ZL = P * Z / 4;  // slices of a lane
    auto store = [&](int i, float2 o) {
      const int z = ZL * (P == 1 ? kk : kk & 1) + i;
      if (s >= 0 && z < nzb && (P == 1 || kk >= 2)) a.Sh[(int64_t)s * a.nz + z0 + z] = (s & 1) ? o : make_float2(-o.x, -o.y);
    };
    if constexpr (SPARSE) {
      __syncthreads();  // every wavefront has read the tile
      f32x4* part = reinterpret_cast<f32x4*>(tile);
#pragma unroll
      for (int c = 0; c < NA; ++c) part[(NA * wv + c) * 64 + lane] = sum[c];
      __syncthreads();
      if (wv >= ZL) return;
      const float* p = reinterpret_cast<const float*>(tile) + 4 * lane + (Z == 16 ? wv : 2 * wv);
      float2 o = make_float2(0.f, 0.f);
#pragma unroll
      for (int k = 0; k < kGatherWaves; ++k)
        o = cadd(o, make_float2(p[NA * k * 256], Z == 16 ? p[(NA * k + 1) * 256] : p[NA * k * 256 + 1]));
      store(wv, o);
      return;
    } else {
#pragma unroll
      for (int i = 0; i < ZL; ++i)
        store(i, Z == 16 ? make_float2(sum[0][i], sum[NA - 1][i]) : make_float2(sum[0][2 * i], sum[0][2 * i + 1]));
    }
  }
}

static hipError_t launch_gather(const TomoArgs& a, hipStream_t st) {
  // eights where an odd number of them holds the slab (20 slices of 512^2, 200
  // angles: 223 us in two sixteens, 196 in three eights)
  const int Z = a.nz <= 4 ? 4 : ((a.nz + 7) / 8) & 1 ? 8 : 16;
  const int zblocks = (a.nz + Z - 1) / Z, zper = (a.nz + zblocks - 1) / zblocks;
  const dim3 grid((unsigned)a.nitems, (unsigned)zblocks), block(64 * kGatherWaves);
#define HTAMD_GATHER(SPARSE, Z) hipLaunchKernelGGL((tomo_gather_k<SPARSE, Z>), grid, block, 0, st, a, zper)
  if (a.sparse) {
    if (Z == 4) HTAMD_GATHER(true, 4);
    if (Z == 8) HTAMD_GATHER(true, 8);
    if (Z == 16) HTAMD_GATHER(true, 16);
  } else {
    if (Z == 4) HTAMD_GATHER(false, 4);
    if (Z == 8) HTAMD_GATHER(false, 8);
    if (Z == 16) HTAMD_GATHER(false, 16);
  }
#undef HTAMD_GATHER
  return hipGetLastError();
}

// Line passes: a workgroup takes C consecutive lines theta nz + z, which
// mostly are C slices of one angle, so that the slices-fastest spectra are read
// and written C x 8 bytes at a time (the lanes of a tile access run over the
// lines), the sinogram along the lines.  C = 16 where 1024 threads and 70 KiB
// of LDS hold it, 4 below kLineFew lines (one slice of 512^2, 16 angles: 8.5 us
// with one workgroup of 16 lines).
template <int N>
constexpr int line_c() {
  return N <= 512 ? 16 : 8;
}
constexpr int64_t kLineFew = 2048;

// index of (line, t) in the spectra; lines past the end repeat the last
struct LineIdx {
  int64_t base;
  int nz;
  __device__ __forceinline__ LineIdx(const TomoArgs& a, int64_t line) : nz(a.nz) {
    const int64_t last = (int64_t)a.ntheta * a.nz - 1;
    line = line < last ? line : last;
    const int64_t th = line / a.nz;
    base = th * a.n * a.nz + (line - th * a.nz);
  }
  __device__ __forceinline__ int64_t at(int t) const { return base + (int64_t)t * nz; }
};

// ---- forward pass D: line IFFT of the gathered spectra ----------------------
template <int N, int E, int C, typename TO>
__global__ __launch_bounds__(C*(N / E)) void tomo_line_ifft_k(TomoArgs a, TO* __restrict__ out) {
  constexpr int T = N / E, LS = col_stride<N, C>();
  __shared__ float2 lds[C * LS];
  const int cc = threadIdx.x / T, t = threadIdx.x % T;
  const int64_t l0 = (int64_t)blockIdx.x * C;
  FftTw<N, E> twr;
  fft_load_twiddles<N, E>(twr, t, a.tw1);
  {
    const int c = threadIdx.x % C, p0 = threadIdx.x / C;
    const LineIdx li(a, l0 + c);
#pragma unroll
    for (int e = 0; e < E; ++e) lds[c * LS + fpad(p0 + e * T)] = a.Sh[li.at(p0 + e * T)];
  }
  __syncthreads();
  float2* s = lds + cc * LS;
  fft_lds<N, E, true, kMaxRadix, wave_private<N, E>()>(s, t, twr);
  if (l0 + cc < (int64_t)a.ntheta * a.nz) {
    TO* dst = out + (l0 + cc) * N;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int tt = t + e * T;
      st_c<TO>(dst, tt, cscale(s[fpad(tt)], -sgnf(tt) * (float)(0.25 / ((double)N * N))));
    }
  }
}

// ---- adjoint pass C': line FFT into the slices-fastest spectra --------------
template <int N, int E, int C, typename TI>
__global__ __launch_bounds__(C*(N / E)) void tomo_linefft_k(TomoArgs a, const TI* __restrict__ data) {
  constexpr int T = N / E, LS = col_stride<N, C>();
  __shared__ float2 lds[C * LS];
  const int cc = threadIdx.x / T, t = threadIdx.x % T;
  const int64_t l0 = (int64_t)blockIdx.x * C, lines = (int64_t)a.ntheta * a.nz;
  const bool valid = l0 + cc < lines;
  float2* s = lds + cc * LS;
  FftTw<N, E> twr;
  fft_load_twiddles<N, E>(twr, t, a.tw1);
  const TI* src = data + (valid ? l0 + cc : 0) * N;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int tt = t + e * T;
    s[fpad(tt)] = valid ? cscale(ld_c<TI>(src, tt), -sgnf(tt)) : make_float2(0.f, 0.f);
  }
  lds_sync<wave_private<N, E>()>();
  fft_lds<N, E, false, kMaxRadix, wave_private<N, E>()>(s, t, twr);
  if constexpr (wave_private<N, E>()) __syncthreads();  // the store crosses lines
  const int c = threadIdx.x % C, p0 = threadIdx.x / C;
  if (l0 + c >= lines) return;
  const LineIdx li(a, l0 + c);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int tt = p0 + e * T;
    const float sc = a.filt ? -sgnf(tt) * a.filt[tt] : -sgnf(tt);
    a.Sh[li.at(tt)] = cscale(lds[c * LS + fpad(tt)], sc);
  }
}

// ---- detector filter alone (Tomo._filter_sino): IFFT(h FFT(line)) -----------
// h already holds the 1/N of the inverse transform.  in may equal out.
template <int N, int E, typename TIO>
__global__ __launch_bounds__(256) void tomo_filter_k(const TIO* in, TIO* out, int64_t lines,
                                                     const float2* __restrict__ tw, const float* __restrict__ h) {
  constexpr int T = N / E, ROWS = 256 / T;
  __shared__ float2 lds[ROWS * fft_buf<N>()];
  const int r = threadIdx.x / T, t = threadIdx.x % T;
  const int64_t line = (int64_t)blockIdx.x * ROWS + r;
  const bool valid = line < lines;
  float2* s = lds + r * fft_buf<N>();
  FftTw<N, E> twr;
  fft_load_twiddles<N, E>(twr, t, tw);
  const TIO* src = in + (valid ? line : 0) * N;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = t + e * T;
    s[fpad(k)] = valid ? ld_c<TIO>(src, k) : make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft_lds<N, E, false>(s, t, twr);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = t + e * T;
    s[fpad(k)] = cscale(s[fpad(k)], h[k]);
  }
  __syncthreads();
  fft_lds<N, E, true>(s, t, twr);
  if (valid) {
    TIO* dst = out + line * N;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = t + e * T;
      st_c<TIO>(dst, k, s[fpad(k)]);
    }
  }
}

// ---- adjoint pass C'': samples onto the grid --------------------------------
// G[g][z] = sum over the samples s whose 9x9 window covers grid point g of
// wy(s, g) wx(s, g) Sh[s][z]: for one tile of 4x4 points the product of a
// 16 x K matrix of weights (K samples touch the tile, about 9/4 of their
// weights are not zero) with K rows of slices, which is what the matrix
// instructions do: v_mfma_f32_16x16x4_f32 takes four samples at a time, the
// tile's points as rows and 16 floats of slices as columns, FP32 throughout.
// Against a sum per point, a sample's slices are read by the 9 tiles it
// touches instead of by 81 points; those reads (from L2) bounded the gather.
// A wavefront owns one tile and 16 VEC U slices.  Lane l holds sample l / 16
// of the four, reads its VEC slices at q = l % 16 (their re and im columns are
// separate products, so 2 VEC U accumulators) and forms the weight of point
// l % 16 from the sample's two zero-padded weight rows (built in FP64).  The
// order of each sum is the list's, whatever runs when; no atomics.
// The NW wavefronts of a workgroup take NW tiles of a row, which share most
// of their samples and make whole cache lines of the result.  Every line crosses
// the centre, so the lists there are long (2500 samples at 256^2, 384 angles,
// against a mean of 54): the tiles with more than kHeavyTile entries (listed
// longest first, at the front of the launch) take a whole workgroup each.  The
// plan cuts these lists into parts, 16 where the longest has more than kLongTile
// entries and else 4, whose sums are added four by four and the quarters in
// order; a wavefront takes SUBS parts, and with four of them adds a quarter
// itself.  So the order of a sum, and with it every bit of a slice's result, does
// not depend on the slab that the slice comes in.
// 256 slices of 256^2, 384 angles: 1555 us with a sum per point -> 390 us (1.2 GB
// through the L2 misses, a third of it the grid; the products themselves are 104 us);
// 45 real slices of 512^2, 451 angles (filtered back-projection): 1645 -> 275 us.
constexpr int kHeavyTile = 128;
constexpr int kLongTile = 512;  // from here more wavefronts share a long list (few slices)
constexpr int kParts = 16, kQuarters = 4;
constexpr int kBatch = 4;  // steps of four samples taken together
// A grid of more than this, half the Infinity Cache, is not kept in the L2: the
// samples' slices, which the next tiles read, are (RT of 256 slices of 256^2, 384
// angles 787 -> 736 us; 100 slices, 64 angles 174 -> 162).  A smaller one is, for
// the column pass (16 slices of 512^2, 16 angles 105 -> 92 us).
constexpr int64_t kKeepGrid = 128 << 20;

template <int VEC, int U, int NW, int SUBS, bool KEEP>
__global__ __launch_bounds__(64 * NW) void tomo_grid_k(TomoArgs a, int zper) {
  constexpr int NA = 2 * VEC * U;  // accumulators: float columns of 16 slices
  constexpr int PX = 4 * NW;       // points of a workgroup's row
  constexpr int ZS = 4 * PX + 2;   // float2 slots of a slice's 4 rows, padded off its bank
  constexpr int SL = NW == kQuarters ? kQuarters : kParts;  // sums that the wavefronts hand over
  static_assert(SL == (SUBS == 4 ? NW : NW * SUBS), "a quarter or a part in each slot");
  constexpr int kOut = 16 * VEC * U * ZS / 2, kPart = SL * NA * 64;
  __shared__ f32x4 lds[kOut > kPart ? kOut : kPart];
  __shared__ int skipped[NW];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int q = lane & 15, kk = lane >> 4;
  const int nt = a.n / 2, n2 = 2 * a.n;
  const bool heavy = (int)blockIdx.x < a.nheavy;
  bool skip = false;  // nothing of this wavefront's is stored
  int tile, beg, end, stop = 0;  // stop: where the part in hand ends (SUBS > 1)
  // part i of a heavy list begins here: whole batches to a part
  int first = 0, last = 0;
  auto part_at = [&](int i) {
    constexpr int B = 4 * kBatch;
    return min(first + (int)((int64_t)((last - first + B - 1) / B) * i / (NW * SUBS)) * B, last);
  };
  if (heavy) {
    tile = a.heavy[blockIdx.x];
    first = a.tp[tile];
    last = a.tp[tile + 1];
    beg = part_at(wv * SUBS);
    end = part_at((wv + 1) * SUBS);
    stop = part_at(wv * SUBS + 1);
  } else {
    const int nb = (nt + NW - 1) / NW;
    const int bid = (int)xcd_tile(blockIdx.x - a.nheavy, gridDim.x - a.nheavy);
    const int tx = bid % nb * NW + wv;
    tile = bid / nb * nt + min(tx, nt - 1);
    beg = a.tp[tile];
    end = a.tp[tile + 1];
    skip = tx >= nt || end - beg > kHeavyTile;
    if (skip) end = beg;
    if constexpr (SUBS > 1) stop = end;
  }
  const int z0 = blockIdx.y * zper, z1 = min(z0 + zper, a.nz);
  int zc[U];
#pragma unroll
  for (int u = 0; u < U; ++u) zc[u] = min(z0 + (u * 16 + q) * VEC, a.nz - VEC);
  const float* wt = a.wt + (q & 3);
  const float* wty = a.wt + kWRow + (q >> 2);
  // the running sum rounds at every step: sums of kBatch steps, added up, keep
  // the error of the longest lists at that of the shortest (RT at 256^2 and 720
  // angles against FP64: 8.2e-7 in one sum, 2.3e-7 so, 2.4e-7 with a sum per
  // point)
  f32x4 tot[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) tot[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a batch's entries are loaded a batch ahead, one per lane, and its samples'
  // slices and weights all at once; entries past the end repeat the last with
  // zero weight (as the lists' padding to whole steps has)
  int2 next = make_int2(0, 0);
  auto entries = [&](int e) { next = a.te[min(e + (lane & (4 * kBatch - 1)), end - 1)]; };
  auto load = [&](int e, float (&w)[kBatch], float (&v)[kBatch][U][2 * VEC]) {
    const int2 cur = next;
    entries(e + 4 * kBatch);
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int s = __shfl(cur.x, 4 * i + kk, 64), o = __shfl(cur.y, 4 * i + kk, 64);
      const int64_t ws = (int64_t)s * (2 * kWRow);
      w[i] = e + 4 * i < end ? wt[ws + (o & 0xff)] * wty[ws + (o >> 8)] : 0.f;
      const float2* src = a.Sh + (int64_t)s * a.nz;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (VEC == 2) {
          const f32x4u t = *reinterpret_cast<const f32x4u*>(src + zc[u]);
          v[i][u][0] = t.x; v[i][u][1] = t.y; v[i][u][2] = t.z; v[i][u][3] = t.w;
        } else {
          const float2 t = src[zc[u]];
          v[i][u][0] = t.x; v[i][u][1] = t.y;
        }
      }
    }
  };
  auto mul = [&](const float (&w)[kBatch], const float (&v)[kBatch][U][2 * VEC]) {
    f32x4 acc[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < 2 * VEC; ++c)
          acc[u * 2 * VEC + c] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], v[i][u][c], acc[u * 2 * VEC + c], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NA; ++i) tot[i] += acc[i];
  };
  // a wavefront of several parts keeps the sum of those before the one in hand
  // in the lane's own slot (of four parts all, of two the first)
  f32x4(*slot)[NA][64] = reinterpret_cast<f32x4(*)[NA][64]>(lds);
  const int own = wv * SL / NW;
  int sub = wv * SUBS + 1;
  auto cut = [&](int e) {  // e: one past the last entry taken
    if constexpr (SUBS > 1) {
      if (__builtin_expect(e < stop || stop >= end, 1)) return;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        slot[own][i][lane] = SUBS == 2 ? tot[i] : slot[own][i][lane] + tot[i];
        tot[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      while (stop <= e && stop < end) stop = part_at(++sub);
    }
  };
  if constexpr (SUBS > 1) {
    if (heavy) {
#pragma unroll
      for (int i = 0; i < NA; ++i) slot[own][i][lane] = f32x4{0.f, 0.f, 0.f, 0.f};
      while (stop <= beg && stop < end) stop = part_at(++sub);
    }
  }
  if (beg < end) {
    float w0[kBatch], v0[kBatch][U][2 * VEC];
    entries(beg);
    if constexpr (NA <= 4) {
      // few slices: a wavefront's chain of loads is what counts, so two batches
      // take turns, one loading while the other is multiplied (with more
      // slices the second set of registers costs more wavefronts than it gains)
      float w1[kBatch], v1[kBatch][U][2 * VEC];
      load(beg, w0, v0);
#pragma unroll 1
      for (int e = beg;; e += 8 * kBatch) {
        const bool more1 = e + 4 * kBatch < end, more2 = e + 8 * kBatch < end;
        if (more1) load(e + 4 * kBatch, w1, v1);
        mul(w0, v0);
        if (!more1) break;
        cut(e + 4 * kBatch);
        if (more2) load(e + 8 * kBatch, w0, v0);
        mul(w1, v1);
        if (!more2) break;
        cut(e + 8 * kBatch);
      }
    } else {
#pragma unroll 1
      for (int e = beg; e < end; e += 4 * kBatch) {
        load(e, w0, v0);
        mul(w0, v0);
        cut(e + 4 * kBatch);
      }
    }
  }
  const int64_t plane = (int64_t)n2 * n2;
  if (heavy) {
    auto put = [&](int u, int c, f32x4 re, f32x4 im) {
      const int zs = z0 + (u * 16 + q) * VEC;
      if (zs >= z1) return;
      float2* d = a.G + (int64_t)(tile / nt * 4 + kk) * n2 + tile % nt * 4 + (min(zs, a.nz - VEC) + c) * plane;
      *reinterpret_cast<f32x4u*>(d) = f32x4{re.x, im.x, re.y, im.y};
      *reinterpret_cast<f32x4u*>(d + 2) = f32x4{re.z, im.z, re.w, im.w};
    };
    if constexpr (SUBS == 4) {
#pragma unroll
      for (int i = 0; i < NA; ++i) tot[i] = slot[own][i][lane] + tot[i];
    }
    if (SL == kParts || wv) {
#pragma unroll
      for (int i = 0; i < NA; ++i) slot[own + (SUBS == 2)][i][lane] = tot[i];
    }
    __syncthreads();
    if constexpr (SL == kParts) {  // wavefront w the columns of slices (u, c) = w
      if (wv >= U * VEC) return;
      f32x4 sum[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int k = 0; k < SL; k += 4) {
          f32x4 quarter = slot[k][2 * wv + i][lane];
#pragma unroll
          for (int l = 1; l < 4; ++l) quarter += slot[k + l][2 * wv + i][lane];
          sum[i] = k ? sum[i] + quarter : quarter;
        }
      put(wv / VEC, wv % VEC, sum[0], sum[1]);
    } else {
      if (wv) return;
#pragma unroll
      for (int k = 1; k < SL; ++k)
#pragma unroll
        for (int i = 0; i < NA; ++i) tot[i] += slot[k][i][lane];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < VEC; ++c) put(u, c, tot[(u * VEC + c) * 2], tot[(u * VEC + c) * 2 + 1]);
    }
    return;
  }
  // result rows 4 (l / 16) + r are the points (y = l / 16, x = r), columns q
  // the slices: through LDS, so that a slice's row is stored as whole lines
  float2* out = reinterpret_cast<float2*>(lds);
  if (lane == 0) skipped[wv] = skip;
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const f32x4 re = tot[(u * VEC + c) * 2], im = tot[(u * VEC + c) * 2 + 1];
      const int slot = zc[u] + c - z0;  // lanes past the last slice repeat it
      if (slot < 0) continue;
      f32x4* d = reinterpret_cast<f32x4*>(out + slot * ZS + kk * PX + wv * 4);
      d[0] = f32x4{re.x, im.x, re.y, im.y};
      d[1] = f32x4{re.z, im.z, re.w, im.w};
    }
  __syncthreads();
  const int tx0 = tile % nt / NW * NW, gy = tile / nt * 4;  // the workgroup's first tile (tile is clamped to its row)
  constexpr int TR = PX / 2;                                 // threads of a row, 2 points each
  const int t = threadIdx.x % TR;
  if (skipped[t >> 1]) return;
  for (int r = threadIdx.x / TR; r < 4 * (z1 - z0); r += 64 * NW / TR) {
    const int zl = r >> 2, y = r & 3;
    const f32x4u v = *reinterpret_cast<const f32x4u*>(out + zl * ZS + y * PX + t * 2);
    auto* d = reinterpret_cast<f32x4u*>(a.G + (z0 + zl) * plane + (int64_t)(gy + y) * n2 + tx0 * 4 + t * 2);
    if constexpr (KEEP)
      *d = v;
    else
      __builtin_nontemporal_store(v, d);
  }
}

// Slices a wavefront takes: the smallest of 16, 32, 48 and 64 that holds an
// even share of the slab (a share ends anywhere: a lane past the end repeats
// the last slices).
static hipError_t launch_grid_gather(const TomoArgs& a, hipStream_t st) {
  const int nt = a.n / 2;
  // Blocks of 64 slices, or of 16 where long lists have fewer workgroups than the
  // chip has CUs (RT of 40 slices of 32^2, 1200 angles 250 -> 96 us).
  const bool parts = a.parts == kParts;
  const int64_t blocks64 = (a.nz + 63) / 64;
  const int zmax = parts && nt * nt * blocks64 <= kNumCu ? 16 : 64;
  const int zblocks = (a.nz + zmax - 1) / zmax, zper = ((a.nz + zblocks - 1) / zblocks + 1) / 2 * 2;
  auto grid = [&](int nw) { return dim3((unsigned)(a.nheavy + (nt + nw - 1) / nw * nt), (unsigned)zblocks); };
  const bool keep = (int64_t)a.nz * 4 * a.n * a.n * (int64_t)sizeof(float2) <= kKeepGrid;
#define HTAMD_GRID(VEC, U, NW, SUBS)                                                                             \
  do {                                                                                                           \
    if (keep)                                                                                                    \
      hipLaunchKernelGGL((tomo_grid_k<VEC, U, NW, SUBS, true>), grid(NW), dim3(64 * NW), 0, st, a, zper);        \
    else                                                                                                         \
      hipLaunchKernelGGL((tomo_grid_k<VEC, U, NW, SUBS, false>), grid(NW), dim3(64 * NW), 0, st, a, zper);       \
  } while (0)
  if (zper <= 16 && parts)
    HTAMD_GRID(1, 1, 16, 1);
  else if (zper <= 16)
    HTAMD_GRID(1, 1, 4, 1);
  else if (zper <= 32 && parts)
    HTAMD_GRID(2, 1, 8, 2);
  else if (zper <= 32)
    HTAMD_GRID(2, 1, 4, 1);
  else if (zper <= 48 && parts)
    HTAMD_GRID(1, 3, 4, 4);
  else if (zper <= 48)
    HTAMD_GRID(1, 3, 4, 1);
  else if (parts)
    HTAMD_GRID(2, 2, 4, 4);
  else
    HTAMD_GRID(2, 2, 4, 1);
#undef HTAMD_GRID
  return hipGetLastError();
}

// ---- adjoint pass B': columns of the grid, keep the n central rows ----------
template <int N2, int E, int C>
__global__ __launch_bounds__(C*(N2 / E)) void tomo_cols_adj_k(TomoArgs a) {
  constexpr int T = N2 / E, NT = C * T, LS = col_stride<N2, C>();
  __shared__ float2 lds[C * LS];
  const int n = N2 / 2, h = N2 / 4;
  const int tiles = N2 / C;
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t z = tile / tiles;
  const int k0 = (int)(tile % tiles) * C;
  const int cc = threadIdx.x / T, t = threadIdx.x % T;
  FftTw<N2, E> twr;
  fft_load_twiddles<N2, E>(twr, t, a.tw2);
  const float2* src = a.G + z * (int64_t)N2 * N2 + k0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int idx = threadIdx.x + e * NT;
    const int c = idx % C, k = idx / C;
    lds[c * LS + fpad(k)] = cscale(src[k * N2 + c], sgnf(k + k0 + c));
  }
  __syncthreads();
  fft_lds<N2, E, true, kMaxRadix, wave_private<N2, E>()>(lds + cc * LS, t, twr);
  if constexpr (wave_private<N2, E>()) __syncthreads();  // the store crosses columns
  float2* dst = a.W + z * (int64_t)n * N2 + k0;
  const float sc = 1.0f / N2;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int idx = threadIdx.x + e * NT;
    const int c = idx % C, i = idx / C;
    if (i >= h && i < h + n) dst[(i - h) * N2 + c] = cscale(lds[c * LS + fpad(i)], sc * sgnf(i));
  }
}

// ---- adjoint pass A': rows, crop and deapodise -------------------------------
template <int N2, int E, typename TO>
__global__ __launch_bounds__(256) void tomo_rows_adj_k(TomoArgs a, TO* __restrict__ out) {
  constexpr int T = N2 / E, ROWS = 256 / T;
  __shared__ float2 lds[ROWS * fft_buf<N2>()];
  const int n = N2 / 2, h = N2 / 4;
  const int r = threadIdx.x / T, t = threadIdx.x % T;
  const int64_t row = (int64_t)blockIdx.x * ROWS + r;
  const bool valid = row < (int64_t)a.nz * n;
  const int64_t z = valid ? row / n : 0;
  const int ip = valid ? (int)(row % n) : 0;
  float2* s = lds + r * fft_buf<N2>();
  FftTw<N2, E> twr;
  fft_load_twiddles<N2, E>(twr, t, a.tw2);
  const float2* src = a.W + (z * n + ip) * (int64_t)N2;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = t + e * T;
    s[fpad(k)] = src[k];
  }
  lds_sync<wave_private<N2, E>()>();
  fft_lds<N2, E, true, kMaxRadix, wave_private<N2, E>()>(s, t, twr);
  if (valid) {
    TO* dst = out + (z * n + ip) * (int64_t)n;
    const float sc = 1.0f / N2;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = t + e * T;
      if (p >= h && p < h + n) {
        const int jp = p - h;
        st_c<TO>(dst, jp, cscale(s[fpad(p)], sc * sgnf(p) * a.phi[ip * n + jp]));
      }
    }
  }
}

// ---- any even n: the same passes on the run-time mixed-radix FFT --------------
// (fft_any.hpp; rows of the embedded slice and lines are one unit each,
// columns of the 2n grid C per unit).  Loads and stores apply the same sign
// modulations, embedding, cropping and deapodisation as the kernels above.
template <typename TI>
struct TomoRowsFwdAny {  // line = z n + i' of the n non-zero rows, length 2n
  static constexpr bool kInv = false, kTwo = false;
  TomoArgs a;
  const TI* obj;
  __device__ float2 load(int64_t line, int, int p) const {
    const int n = a.n, h = n / 2;
    if (p < h || p >= h + n) return make_float2(0.f, 0.f);
    const int ip = (int)(line % n), jp = p - h;
    return cscale(ld_c<TI>(obj + line * (int64_t)n, jp), a.phi[ip * n + jp] * sgnf(ip + h + p));
  }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t line, int, int k, float2 v) const {
    a.W[line * (int64_t)(2 * a.n) + k] = cscale(v, sgnf(k));
  }
};

struct TomoColsFwdAny {  // unit = z groups + column group
  static constexpr bool kInv = false, kTwo = false;
  TomoArgs a;
  int C, groups;
  __device__ float2 load(int64_t unit, int c, int i) const {
    const int n = a.n, h = n / 2, N2 = 2 * n;
    const int col = (int)(unit % groups) * C + c;
    if (col >= N2 || i < h || i >= h + n) return make_float2(0.f, 0.f);
    return a.W[(unit / groups) * (int64_t)n * N2 + (int64_t)(i - h) * N2 + col];
  }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t unit, int c, int k, float2 v) const {
    const int N2 = 2 * a.n;
    const int col = (int)(unit % groups) * C + c;
    if (col < N2) a.G[(unit / groups) * (int64_t)N2 * N2 + (int64_t)k * N2 + col] = cscale(v, sgnf(k));
  }
};

template <typename TO>
struct TomoLineIfftAny {  // line = theta nz + z, length n
  static constexpr bool kInv = true, kTwo = false;
  TomoArgs a;
  TO* out;
  __device__ float2 load(int64_t line, int, int t) const { return a.Sh[LineIdx(a, line).at(t)]; }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t line, int, int t, float2 v) const {
    st_c<TO>(out + line * a.n, t, cscale(v, -sgnf(t) * (float)(0.25 / ((double)a.n * a.n))));
  }
};

template <typename TI>
struct TomoLineFftAny {  // line = theta nz + z, length n; slices-fastest output
  static constexpr bool kInv = false, kTwo = false;
  TomoArgs a;
  const TI* data;
  __device__ float2 load(int64_t line, int, int t) const {
    return cscale(ld_c<TI>(data + line * a.n, t), -sgnf(t));
  }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t line, int, int t, float2 v) const {
    const float sc = a.filt ? -sgnf(t) * a.filt[t] : -sgnf(t);
    a.Sh[LineIdx(a, line).at(t)] = cscale(v, sc);
  }
};

struct TomoColsAdjAny {  // unit = z groups + column group; keeps the n central rows
  static constexpr bool kInv = true, kTwo = false;
  TomoArgs a;
  int C, groups;
  __device__ float2 load(int64_t unit, int c, int k) const {
    const int N2 = 2 * a.n;
    const int col = (int)(unit % groups) * C + c;
    if (col >= N2) return make_float2(0.f, 0.f);
    return cscale(a.G[(unit / groups) * (int64_t)N2 * N2 + (int64_t)k * N2 + col], sgnf(k + col));
  }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t unit, int c, int i, float2 v) const {
    const int n = a.n, h = n / 2, N2 = 2 * n;
    const int col = (int)(unit % groups) * C + c;
    if (col < N2 && i >= h && i < h + n)
      a.W[(unit / groups) * (int64_t)n * N2 + (int64_t)(i - h) * N2 + col] = cscale(v, sgnf(i) / (float)N2);
  }
};

template <typename TO>
struct TomoRowsAdjAny {  // line = z n + i', length 2n; crop and deapodise
  static constexpr bool kInv = true, kTwo = false;
  TomoArgs a;
  TO* out;
  __device__ float2 load(int64_t line, int, int k) const { return a.W[line * (int64_t)(2 * a.n) + k]; }
  __device__ void mid(float2*, int64_t, int, int, int) const {}
  __device__ void store(int64_t line, int, int p, float2 v) const {
    const int n = a.n, h = n / 2;
    if (p < h || p >= h + n) return;
    const int ip = (int)(line % n), jp = p - h;
    st_c<TO>(out + line * (int64_t)n, jp, cscale(v, sgnf(p) / (float)(2 * n) * a.phi[ip * n + jp]));
  }
};

template <typename TIO>
struct TomoFilterAny {  // IFFT(h FFT(line)), h with the 1/n of the inverse
  static constexpr bool kInv = false, kTwo = true;
  const TIO* in;
  TIO* out;
  int n;
  const float* h;
  __device__ float2 load(int64_t line, int, int k) const { return ld_c<TIO>(in + line * n, k); }
  __device__ void mid(float2* s, int64_t, int, int tid, int nthr) const {
    for (int k = tid; k < n; k += nthr) s[k] = cscale(s[k], h[k]);
  }
  __device__ void store(int64_t line, int, int k, float2 v) const { st_c<TIO>(out + line * n, k, v); }
};

static bool tomo_any_ffts(const TomoArgs& a, AnyFft* f2, AnyFft* f1) {
  if (!any_fft_factor(2 * (int64_t)a.n, f2) || !any_fft_factor(a.n, f1)) return false;
  f2->tw = a.tw2;
  f1->tw = a.tw1;
  return true;
}

template <typename TIO>
static hipError_t tomo_fwd_any(const TomoArgs& a, const TIO* obj, TIO* out, hipStream_t st) {
  AnyFft f2, f1;
  if (!tomo_any_ffts(a, &f2, &f1)) return hipErrorInvalidValue;
  const int N2 = 2 * a.n;
  hipError_t e = any_launch_rows(TomoRowsFwdAny<TIO>{a, obj}, f2, (int64_t)a.nz * a.n, st);
  if (e != hipSuccess) return e;
  const int C = any_cols_c(N2, any_max_lds()), groups = (N2 + C - 1) / C;
  if ((e = any_launch_cols(TomoColsFwdAny{a, C, groups}, f2, C, (int64_t)a.nz * groups, st)) != hipSuccess) return e;
  if ((e = launch_gather(a, st)) != hipSuccess) return e;
  return any_launch_rows(TomoLineIfftAny<TIO>{a, out}, f1, (int64_t)a.ntheta * a.nz, st);
}

template <typename TIO>
static hipError_t tomo_adj_any(const TomoArgs& a, const TIO* data, TIO* out, hipStream_t st) {
  AnyFft f2, f1;
  if (!tomo_any_ffts(a, &f2, &f1)) return hipErrorInvalidValue;
  const int N2 = 2 * a.n;
  hipError_t e = any_launch_rows(TomoLineFftAny<TIO>{a, data}, f1, (int64_t)a.ntheta * a.nz, st);
  if (e != hipSuccess) return e;
  if ((e = launch_grid_gather(a, st)) != hipSuccess) return e;
  const int C = any_cols_c(N2, any_max_lds()), groups = (N2 + C - 1) / C;
  if ((e = any_launch_cols(TomoColsAdjAny{a, C, groups}, f2, C, (int64_t)a.nz * groups, st)) != hipSuccess) return e;
  return any_launch_rows(TomoRowsAdjAny<TIO>{a, out}, f2, (int64_t)a.nz * a.n, st);
}

static bool tomo_pow2(int64_t n) { return n >= 8 && n <= 1024 && (n & (n - 1)) == 0; }

// ---- host dispatch -----------------------------------------------------------
// columns per workgroup of the column passes: at most 16, at most about 70 KiB
// of LDS (8192 / N2 padded columns) and at most 1024 threads
template <int N2>
constexpr int tomo_cols_c() {
  constexpr int T = N2 / 8;
  constexpr int CT = 1024 / T;
  constexpr int CL = 8192 / N2 > 0 ? 8192 / N2 : 1;
  constexpr int C0 = CT < CL ? CT : CL;
  return C0 > 16 ? 16 : C0;
}

template <int N2, typename TIO>
static hipError_t tomo_fwd_n(const TomoArgs& a, const TIO* obj, TIO* out, hipStream_t st) {
  constexpr int E = 8, N = N2 / 2;
  constexpr int C = tomo_cols_c<N2>();
  const int64_t rows = (int64_t)a.nz * N;
  hipLaunchKernelGGL((tomo_rows_fwd_k<N2, E, TIO>), dim3((unsigned)((rows + 256 / (N2 / E) - 1) / (256 / (N2 / E)))),
                     dim3(256), 0, st, a, obj);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((tomo_cols_fwd_k<N2, E, C>), dim3((unsigned)(a.nz * (N2 / C))), dim3(C * (N2 / E)), 0, st, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = launch_gather(a, st)) != hipSuccess) return e;
  constexpr int EL = N >= 8 ? 8 : N, CL = line_c<N>();
  const int64_t lines = (int64_t)a.ntheta * a.nz;
  if (lines < kLineFew)
    hipLaunchKernelGGL((tomo_line_ifft_k<N, EL, 4, TIO>), dim3((unsigned)((lines + 3) / 4)), dim3(4 * (N / EL)), 0,
                       st, a, out);
  else
    hipLaunchKernelGGL((tomo_line_ifft_k<N, EL, CL, TIO>), dim3((unsigned)((lines + CL - 1) / CL)),
                       dim3(CL * (N / EL)), 0, st, a, out);
  return hipGetLastError();
}

template <int N2, typename TIO>
static hipError_t tomo_adj_n(const TomoArgs& a, const TIO* data, TIO* out, hipStream_t st) {
  constexpr int E = 8, N = N2 / 2;
  constexpr int C = tomo_cols_c<N2>();
  constexpr int EL = N >= 8 ? 8 : N, CL = line_c<N>();
  const int64_t lines = (int64_t)a.ntheta * a.nz;
  if (lines < kLineFew)
    hipLaunchKernelGGL((tomo_linefft_k<N, EL, 4, TIO>), dim3((unsigned)((lines + 3) / 4)), dim3(4 * (N / EL)), 0, st,
                       a, data);
  else
    hipLaunchKernelGGL((tomo_linefft_k<N, EL, CL, TIO>), dim3((unsigned)((lines + CL - 1) / CL)),
                       dim3(CL * (N / EL)), 0, st, a, data);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if ((e = launch_grid_gather(a, st)) != hipSuccess) return e;
  hipLaunchKernelGGL((tomo_cols_adj_k<N2, E, C>), dim3((unsigned)(a.nz * (N2 / C))), dim3(C * (N2 / E)), 0, st, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const int64_t rows = (int64_t)a.nz * N;
  hipLaunchKernelGGL((tomo_rows_adj_k<N2, E, TIO>), dim3((unsigned)((rows + 256 / (N2 / E) - 1) / (256 / (N2 / E)))),
                     dim3(256), 0, st, a, out);
  return hipGetLastError();
}

template <int N, typename TIO>
static hipError_t tomo_filter_n(const TIO* in, TIO* out, int64_t lines, const float2* tw, const float* h,
                                hipStream_t st) {
  constexpr int E = N >= 8 ? 8 : N;
  constexpr int RL = 256 / (N / E);
  if (lines == 0) return hipSuccess;
  hipLaunchKernelGGL((tomo_filter_k<N, E, TIO>), dim3((unsigned)((lines + RL - 1) / RL)), dim3(256), 0, st, in, out,
                     lines, tw, h);
  return hipGetLastError();
}

template <typename TIO>
static hipError_t tomo_filter_dispatch(int n, const void* in, void* out, int64_t lines, const float2* tw,
                                       const float* h, hipStream_t st) {
  if (!tomo_pow2(n)) {
    AnyFft f;
    if (!any_fft_factor(n, &f)) return hipErrorInvalidValue;
    f.tw = tw;
    return any_launch_rows(TomoFilterAny<TIO>{(const TIO*)in, (TIO*)out, n, h}, f, lines, st);
  }
#define HTAMD_TFILT_CASE(NN) \
  case NN: return tomo_filter_n<NN, TIO>((const TIO*)in, (TIO*)out, lines, tw, h, st);
  switch (n) {
    HTAMD_TFILT_CASE(8) HTAMD_TFILT_CASE(16) HTAMD_TFILT_CASE(32) HTAMD_TFILT_CASE(64) HTAMD_TFILT_CASE(128)
    HTAMD_TFILT_CASE(256) HTAMD_TFILT_CASE(512) HTAMD_TFILT_CASE(1024)
    default: return hipErrorInvalidValue;
  }
#undef HTAMD_TFILT_CASE
}

template <typename TIO>
static hipError_t tomo_dispatch(bool adjoint, const TomoArgs& a, const void* in, void* out, hipStream_t st) {
  if (!tomo_pow2(a.n))
    return adjoint ? tomo_adj_any<TIO>(a, (const TIO*)in, (TIO*)out, st)
                   : tomo_fwd_any<TIO>(a, (const TIO*)in, (TIO*)out, st);
#define HTAMD_TOMO_CASE(NN)                                                               \
  case NN:                                                                                \
    return adjoint ? tomo_adj_n<2 * NN, TIO>(a, (const TIO*)in, (TIO*)out, st)            \
                   : tomo_fwd_n<2 * NN, TIO>(a, (const TIO*)in, (TIO*)out, st);
  switch (a.n) {
    HTAMD_TOMO_CASE(8) HTAMD_TOMO_CASE(16) HTAMD_TOMO_CASE(32) HTAMD_TOMO_CASE(64) HTAMD_TOMO_CASE(128)
    HTAMD_TOMO_CASE(256) HTAMD_TOMO_CASE(512) HTAMD_TOMO_CASE(1024)
    default: return hipErrorInvalidValue;
  }
#undef HTAMD_TOMO_CASE
}

}  // namespace htamd

using namespace htamd;

struct htamd_tomo_plan {
  int64_t n = 0, ntheta = 0;
  int device = -1;
  float* phi = nullptr;
  float2* tw2 = nullptr;
  float2* tw1 = nullptr;
  float* wt = nullptr;
  int* tp = nullptr;
  int2* te = nullptr;
  int4* items = nullptr;
  int2* ge = nullptr;
  int* gc = nullptr;
  int* heavy = nullptr;
  int nitems = 0, nheavy = 0, parts = 0, sparse = 0;
  // detector filters (ramp, Shepp-Logan, Parzen): [3][n] with the 1/n of the
  // inverse transform for htamd_tomo_filter, and [3][n] shifted by n/2 and
  // scaled by sqrt(n / ntheta) for htamd_tomo_fbp
  float* filt = nullptr;
  float* filt_fbp = nullptr;
};

namespace htamd {

constexpr int kTomoFilters = 3;
// largest slice width: the 2n-point lines of the oversampled grid (two LDS
// buffers of 2n complex values) fit the 160 KiB of LDS up to n = 4096
constexpr int64_t kTomoAnyMax = 4096;

// h[k] on fftfreq(n) (src/holotomocupy/tomo.py:131-155), FP64:
// ramp 4n|f|, Shepp-Logan 4n|f| sinc(f), Parzen 4n|f| w(u), u = 2 (4n|f|),
// w = 1 - 6u^2 + 6u^3 (u <= 1/2) else 2 (1 - u)^3 -- the reference's u.
static double tomo_filter_h(int kind, int64_t k, int64_t n) {
  const double f = (double)(k < (n + 1) / 2 ? k : k - n) / (double)n;
  const double af = std::fabs(f) * 4.0 * (double)n;
  if (kind == 0) return af;
  if (kind == 1) return f == 0.0 ? af : af * std::sin(M_PI * f) / (M_PI * f);
  const double u = 2.0 * af;
  return af * (u <= 0.5 ? 1.0 - 6.0 * u * u + 6.0 * u * u * u : 2.0 * (1.0 - u) * (1.0 - u) * (1.0 - u));
}

}  // namespace htamd

extern "C" {

int htamd_tomo_plan_create(int64_t n, int64_t ntheta, const double* theta, const double* mask,
                           htamd_tomo_plan** plan) {
  if (!plan || !theta) return fail(HTAMD_ERR_ARG, "tomo_plan_create: NULL argument");
  *plan = nullptr;
  {
    AnyFft f2, f1;
    const bool any_ok = n % 2 == 0 && n >= 8 && n <= kTomoAnyMax && any_fft_factor(2 * n, &f2) &&
                        any_fft_factor(n, &f1);
    if (!tomo_pow2(n) && !any_ok)
      return fail(HTAMD_ERR_UNSUPPORTED, "tomo_plan_create: n must be even in [8, " + std::to_string(kTomoAnyMax) +
                                             "] (powers of two up to 1024 on the fastest kernels), got " +
                                             std::to_string(n));
  }
  if (ntheta < 1) return fail(HTAMD_ERR_ARG, "tomo_plan_create: need ntheta >= 1");
  auto* p = new htamd_tomo_plan();
  p->n = n;
  p->ntheta = ntheta;
  // eps, mu, m (tomo.py:14-16)
  const double eps = 1e-3;
  const double mu = -std::log(eps) / (2.0 * (double)n * (double)n);
  const int m = (int)std::ceil(2.0 * n / M_PI * std::sqrt(-mu * std::log(eps) + (mu * n) * (mu * n) / 4.0));
  if (2 * m + 1 != kTL) {  // 4 for every n: the kernels are built for 9x9 windows
    delete p;
    return fail(HTAMD_ERR_UNSUPPORTED, "tomo_plan_create: gridding half-width is not 4");
  }
  const int L = 2 * m + 1;
  const int64_t S = ntheta * n, n2 = 2 * n;
  if (S * L * L > (int64_t)INT32_MAX) {
    delete p;
    return fail(HTAMD_ERR_UNSUPPORTED, "tomo_plan_create: too many gridding taps (ntheta n (2m+1)^2 >= 2^31)");
  }
  hipError_t e = hipGetDevice(&p->device);
  // Gridding taps of every polar sample s = k n + t (cuda_kernels.py:17-51) in
  // FP64: angles rounded to float32 as the reference stores them,
  // x0 = (t - n/2) cos / n, y0 = -(t - n/2) sin / n, first tap floor(2n x0) - m,
  // weights exp(-pi^2/mu d^2) (x) and pi/mu exp(-pi^2/mu d^2) (y).
  std::vector<int2> tb((size_t)S);
  std::vector<float> wt((size_t)(2 * kWRow * S), 0.0f);
  const double cy = M_PI / mu, cx = -M_PI * M_PI / mu, inv2n = 1.0 / (double)n2;
  for (int64_t k = 0; k < ntheta; ++k) {
    const double th = (double)(float)theta[k];
    const double c = std::cos(th), sn = std::sin(th);
    for (int64_t t = 0; t < n; ++t) {
      const int64_t si = k * n + t;
      const double x0 = (double)(t - n / 2) / (double)n * c;
      const double y0 = -(double)(t - n / 2) / (double)n * sn;
      const int bx = (int)std::floor((double)n2 * x0) - m;
      const int by = (int)std::floor((double)n2 * y0) - m;
      tb[(size_t)si] = make_int2(bx, by);
      float* w = &wt[(size_t)(2 * kWRow * si)];
      for (int i = 0; i < L; ++i) {
        const double dx = (bx + i) * inv2n - x0, dy = (by + i) * inv2n - y0;
        w[3 + i] = (float)std::exp(cx * dx * dx);
        w[kWRow + 3 + i] = (float)(cy * std::exp(cx * dy * dy));
      }
    }
  }
  auto wrap = [&](int64_t v) { return (int)((n + v + n2) % n2); };
  // The samples by 4x4 tile, for the adjoint (counting sort; within a tile the
  // samples appear in increasing order): a window of 9 taps touches 3 tiles
  // along each axis, the wrapped first tap's and the next two.  Each list is
  // padded to a multiple of four with entries whose weights are the zeros at
  // the rows' ends.
  const int nt = (int)(n / 2);
  std::vector<int> tp((size_t)nt * nt + 1, 0);
  auto tiles3 = [&](int64_t si, auto&& f) {
    const int wx0 = wrap(tb[(size_t)si].x), wy0 = wrap(tb[(size_t)si].y);
    for (int jy = 0; jy < 3; ++jy)
      for (int jx = 0; jx < 3; ++jx)
        f((wy0 / 4 + jy) % nt * nt + (wx0 / 4 + jx) % nt, 4 * jx - wx0 % 4 + 3, 4 * jy - wy0 % 4 + 3);
  };
  for (int64_t si = 0; si < S; ++si) tiles3(si, [&](int t, int, int) { ++tp[(size_t)t + 1]; });
  std::vector<int> tcnt(tp.begin() + 1, tp.end());
  for (int t = 0; t < nt * nt; ++t) tp[(size_t)t + 1] = tp[(size_t)t] + (tcnt[(size_t)t] + 3) / 4 * 4;
  std::vector<int2> te((size_t)std::max(1, tp.back()), make_int2(0, 12 << 8 | 12));
  {
    std::vector<int> fill(tp.begin(), tp.end() - 1);
    for (int64_t si = 0; si < S; ++si)
      tiles3(si, [&](int t, int ox, int oy) { te[(size_t)fill[(size_t)t]++] = make_int2((int)si, oy << 8 | ox); });
  }
  std::vector<int> heavy;
  for (int t = 0; t < nt * nt; ++t)
    if (tp[(size_t)t + 1] - tp[(size_t)t] > kHeavyTile) heavy.push_back(t);
  std::stable_sort(heavy.begin(), heavy.end(), [&](int x, int y) {
    return tp[(size_t)x + 1] - tp[(size_t)x] > tp[(size_t)y + 1] - tp[(size_t)y];
  });
  // The samples by region and cell of the window's first tap (wrapped), for the
  // forward gather (counting sort, samples in increasing order within a cell),
  // each cell's cut into groups of 16 and each region's groups into work items.
  const int nr = (int)((n2 + kRG - 1) / kRG);  // the last region is partial when kRG does not divide 2n
  constexpr int kCX = kRG / kCellX, kCells = kCX * (kRG / kCellY);
  auto cell_of = [&](int64_t si) {
    const int wx0 = wrap(tb[(size_t)si].x), wy0 = wrap(tb[(size_t)si].y);
    return ((wy0 / kRG) * nr + wx0 / kRG) * kCells + wy0 % kRG / kCellY * kCX + wx0 % kRG / kCellX;
  };
  std::vector<int> ccount((size_t)nr * nr * kCells, 0);
  for (int64_t si = 0; si < S; ++si) ++ccount[(size_t)cell_of(si)];
  // steps of four points of either form, staging a region counted as kStageSteps
  int64_t dense = 0, sparse = 0;
  for (int rg = 0; rg < nr * nr; ++rg) {
    int sum = 0, groups = 0;
    for (int c = 0; c < kCells; ++c) {
      const int k = ccount[(size_t)(rg * kCells + c)];
      groups += (k + 15) / 16;
      sum += k;
    }
    using D = GatherShape<false>;
    using P = GatherShape<true>;
    dense += groups * D::NY * D::NX + (groups + kItemGroups - 1) / kItemGroups * kStageSteps;
    sparse += (sum + 15) / 16 * (P::NY * P::NX + kStageSteps);
  }
  p->sparse = sparse < dense;
  std::vector<int> cfill(ccount.size());
  std::vector<int> gc;
  std::vector<int4> items;
  for (int rg = 0; rg < nr * nr; ++rg) {
    const int first = (int)gc.size();
    for (int c = 0, fill = 0; c < kCells; ++c) {
      const int k = ccount[(size_t)(rg * kCells + c)];
      if (p->sparse) {
        cfill[(size_t)(rg * kCells + c)] = 16 * first + fill;
        fill += k;
        while (16 * ((int)gc.size() - first) < fill) gc.push_back(0);
      } else {
        cfill[(size_t)(rg * kCells + c)] = 16 * (int)gc.size();
        for (int i = 0; i < k; i += 16) gc.push_back(c / kCX << 8 | c % kCX);
      }
    }
    const int step = p->sparse ? 1 : kItemGroups;
    for (int b = first; b < (int)gc.size(); b += step)
      items.push_back(make_int4(rg % nr, rg / nr, b, std::min(step, (int)gc.size() - b)));
  }
  std::vector<int2> ge(16 * gc.size(), make_int2(-1, 0));
  const int py = p->sparse ? kRG : kCellY, px = p->sparse ? kRG : kCellX;
  for (int64_t si = 0; si < S; ++si)
    ge[(size_t)cfill[(size_t)cell_of(si)]++] =
        make_int2((int)si, wrap(tb[(size_t)si].y) % kRG % py << 8 | wrap(tb[(size_t)si].x) % kRG % px);
  p->nitems = (int)items.size();
  p->nheavy = (int)heavy.size();
  p->parts = !heavy.empty() && tp[(size_t)heavy[0] + 1] - tp[(size_t)heavy[0]] > kLongTile ? kParts : kQuarters;
  // deapodiser phi (tomo.py:19-21, 46-47) with the mask folded in
  std::vector<float> phi((size_t)(n * n));
  for (int64_t i = 0; i < n; ++i) {
    const double dy = -0.5 + (double)i / (double)n;
    for (int64_t j = 0; j < n; ++j) {
      const double dx = -0.5 + (double)j / (double)n;
      double v = std::exp(mu * (double)(n * n) * (dx * dx + dy * dy)) * (double)(1 - n % 4);
      v *= (mask ? mask[i * n + j] : 1.0) / ((double)n * std::sqrt((double)n * (double)ntheta));
      phi[(size_t)(i * n + j)] = (float)v;
    }
  }
  std::vector<float> filt((size_t)(kTomoFilters * n)), filt_fbp((size_t)(kTomoFilters * n));
  const double norm_const = std::sqrt((double)n / (double)ntheta);
  for (int kind = 0; kind < kTomoFilters; ++kind)
    for (int64_t k = 0; k < n; ++k) {
      filt[(size_t)(kind * n + k)] = (float)(tomo_filter_h(kind, k, n) / (double)n);
      // FFT(c1d d)[k] picks up h at bin (k - n/2) mod n
      filt_fbp[(size_t)(kind * n + k)] = (float)(tomo_filter_h(kind, (k + n / 2) % n, n) * norm_const);
    }
  auto twid = [](int64_t N) {
    std::vector<float2> t((size_t)N);
    for (int64_t k = 0; k < N; ++k) {
      const double a = -2.0 * M_PI * (double)k / (double)N;
      t[(size_t)k] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    return t;
  };
  auto up = [&](auto** dst, const auto& src) {
    hipError_t r = hipMalloc((void**)dst, src.size() * sizeof(src[0]));
    if (r == hipSuccess) r = hipMemcpy(*dst, src.data(), src.size() * sizeof(src[0]), hipMemcpyHostToDevice);
    return r;
  };
  if (e != hipSuccess || (e = up(&p->phi, phi)) != hipSuccess || (e = up(&p->tw2, twid(2 * n))) != hipSuccess ||
      (e = up(&p->tw1, twid(n))) != hipSuccess || (e = up(&p->wt, wt)) != hipSuccess ||
      (e = up(&p->tp, tp)) != hipSuccess || (e = up(&p->te, te)) != hipSuccess ||
      (e = up(&p->items, items)) != hipSuccess ||
      (!heavy.empty() && (e = up(&p->heavy, heavy)) != hipSuccess) ||
      (e = up(&p->ge, ge)) != hipSuccess || (e = up(&p->gc, gc)) != hipSuccess ||
      (e = up(&p->filt, filt)) != hipSuccess || (e = up(&p->filt_fbp, filt_fbp)) != hipSuccess) {
    htamd_tomo_plan_destroy(p);
    return hip_fail(e, "tomo_plan_create");
  }
  *plan = p;
  return HTAMD_OK;
}

int htamd_tomo_plan_destroy(htamd_tomo_plan* p) {
  if (!p) return HTAMD_OK;
  (void)hipFree(p->phi);
  (void)hipFree(p->tw2);
  (void)hipFree(p->tw1);
  (void)hipFree(p->wt);
  (void)hipFree(p->tp);
  (void)hipFree(p->te);
  (void)hipFree(p->items);
  (void)hipFree(p->ge);
  (void)hipFree(p->gc);
  (void)hipFree(p->heavy);
  (void)hipFree(p->filt);
  (void)hipFree(p->filt_fbp);
  delete p;
  return HTAMD_OK;
}

int htamd_tomo_workspace_size(const htamd_tomo_plan* p, int64_t nz, int64_t* bytes) {
  if (!p || !bytes || nz < 0) return fail(HTAMD_ERR_ARG, "tomo_workspace_size: bad arguments");
  *bytes = nz * (p->n * 2 * p->n + 4 * p->n * p->n) * 8 + p->ntheta * p->n * nz * 8;
  return HTAMD_OK;
}

static int tomo_run(const htamd_tomo_plan* p, bool adjoint, const void* in, int is_complex, void* out,
                    int64_t nz, void* ws, int64_t ws_bytes, void* stream, const char* what, int filter = -1) {
  if (!p) return fail(HTAMD_ERR_ARG, std::string(what) + ": plan is NULL");
  if (nz < 0) return fail(HTAMD_ERR_ARG, std::string(what) + ": negative slice count");
  if (nz == 0) return HTAMD_OK;
  if (!in || !out) return fail(HTAMD_ERR_ARG, std::string(what) + ": NULL buffer");
  int64_t need = 0;
  htamd_tomo_workspace_size(p, nz, &need);
  if (!ws || ws_bytes < need)
    return fail(HTAMD_ERR_ARG, std::string(what) + ": workspace of " + std::to_string(need) + " bytes required");
  int dev = -1;
  (void)hipGetDevice(&dev);
  if (dev != p->device) return fail(HTAMD_ERR_ARG, std::string(what) + ": plan belongs to another device");
  TomoArgs a;
  a.n = (int)p->n;
  a.nz = (int)nz;
  a.ntheta = (int)p->ntheta;
  a.phi = p->phi;
  a.wt = p->wt;
  a.tp = p->tp;
  a.te = p->te;
  a.tw2 = p->tw2;
  a.tw1 = p->tw1;
  a.items = p->items;
  a.ge = p->ge;
  a.gc = p->gc;
  a.nitems = p->nitems;
  a.sparse = p->sparse;
  a.heavy = p->heavy;
  a.nheavy = p->nheavy;
  a.parts = p->parts;
  a.W = (float2*)ws;
  a.G = (float2*)ws + nz * p->n * 2 * p->n;
  a.Sh = a.G + nz * 4 * p->n * p->n;
  if (filter >= 0) a.filt = p->filt_fbp + (int64_t)filter * p->n;
  hipError_t e = is_complex ? tomo_dispatch<float2>(adjoint, a, in, out, (hipStream_t)stream)
                            : tomo_dispatch<float>(adjoint, a, in, out, (hipStream_t)stream);
  return e == hipSuccess ? HTAMD_OK : hip_fail(e, what);
}

int htamd_tomo_R(const htamd_tomo_plan* p, const void* obj, int is_complex, void* out, int64_t nz,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  return tomo_run(p, false, obj, is_complex, out, nz, workspace, workspace_bytes, stream, "tomo_R");
}

int htamd_tomo_RT(const htamd_tomo_plan* p, const void* data, int is_complex, void* out, int64_t nz,
                  void* workspace, int64_t workspace_bytes, void* stream) {
  return tomo_run(p, true, data, is_complex, out, nz, workspace, workspace_bytes, stream, "tomo_RT");
}

int htamd_tomo_fbp(const htamd_tomo_plan* p, const void* data, int is_complex, int filter, void* out, int64_t nz,
                   void* workspace, int64_t workspace_bytes, void* stream) {
  if (filter < 0 || filter >= kTomoFilters)
    return fail(HTAMD_ERR_ARG, "tomo_fbp: filter must be 0 (ramp), 1 (shepp) or 2 (parzen)");
  return tomo_run(p, true, data, is_complex, out, nz, workspace, workspace_bytes, stream, "tomo_fbp", filter);
}

int htamd_tomo_filter(const htamd_tomo_plan* p, const void* data, int is_complex, int filter, void* out, int64_t nz,
                      void* stream) {
  if (!p) return fail(HTAMD_ERR_ARG, "tomo_filter: plan is NULL");
  if (filter < 0 || filter >= kTomoFilters)
    return fail(HTAMD_ERR_ARG, "tomo_filter: filter must be 0 (ramp), 1 (shepp) or 2 (parzen)");
  if (nz < 0) return fail(HTAMD_ERR_ARG, "tomo_filter: negative slice count");
  if (nz == 0) return HTAMD_OK;
  if (!data || !out) return fail(HTAMD_ERR_ARG, "tomo_filter: NULL buffer");
  int dev = -1;
  (void)hipGetDevice(&dev);
  if (dev != p->device) return fail(HTAMD_ERR_ARG, "tomo_filter: plan belongs to another device");
  const float* h = p->filt + (int64_t)filter * p->n;
  const int64_t lines = p->ntheta * nz;
  hipError_t e = is_complex ? tomo_filter_dispatch<float2>((int)p->n, data, out, lines, p->tw1, h, (hipStream_t)stream)
                            : tomo_filter_dispatch<float>((int)p->n, data, out, lines, p->tw1, h, (hipStream_t)stream);
  return e == hipSuccess ? HTAMD_OK : hip_fail(e, "tomo_filter");
}

}  // extern "C"
