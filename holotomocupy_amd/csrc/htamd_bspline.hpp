// Shared device helpers and launch interface of the cubic B-spline kernels.
#pragma once
#include "htamd_common.hpp"

namespace htamd {

// ---- value helpers for real (float) and complex (float2) data --------------
template <typename T> __device__ __forceinline__ T vzero();
template <> __device__ __forceinline__ float vzero<float>() { return 0.0f; }
template <> __device__ __forceinline__ float2 vzero<float2>() { return make_float2(0.0f, 0.0f); }

__device__ __forceinline__ float vfma(float w, float v, float acc) { return fmaf(w, v, acc); }
__device__ __forceinline__ float2 vfma(float w, float2 v, float2 acc) {
  return make_float2(fmaf(w, v.x, acc.x), fmaf(w, v.y, acc.y));
}
// Re(a conj(b)) = Re a Re b + Im a Im b
__device__ __forceinline__ float vredot(float a, float b) { return a * b; }
__device__ __forceinline__ float vredot(float2 a, float2 b) { return a.x * b.x + a.y * b.y; }

// ---- cubic B-spline tap weights ---------------------------------------------
// phi = 6 * beta3 (phi(0) = 4, phi(+-1) = 1).  For a fractional offset d in
// [0, 1) the four taps j = -1, 0, 1, 2 sit at t = d - j, each on a fixed
// polynomial piece of phi; w[j + 1] = phi(d - j), dw = phi', d2w = phi''.
__device__ __forceinline__ void bs_w(float d, float* w) {
  const float u = 1.0f - d;
  w[0] = u * u * u;
  w[1] = 4.0f - 6.0f * d * d + 3.0f * d * d * d;
  w[2] = 4.0f - 6.0f * u * u + 3.0f * u * u * u;
  w[3] = d * d * d;
}
__device__ __forceinline__ void bs_dw(float d, float* w) {
  const float u = 1.0f - d;
  w[0] = -3.0f * u * u;
  w[1] = -12.0f * d + 9.0f * d * d;
  w[2] = 12.0f * u - 9.0f * u * u;
  w[3] = 3.0f * d * d;
}
__device__ __forceinline__ void bs_d2w(float d, float* w) {
  const float u = 1.0f - d;
  w[0] = 6.0f * u;
  w[1] = -12.0f + 18.0f * d;
  w[2] = -12.0f + 18.0f * u;
  w[3] = 6.0f * d;
}

// Sampling coordinate of detector index t (cuda_kernels.py:174-177), in FP32
// with the reference's operation order: used only to bracket candidate taps
// (every caller keeps a one-pixel margin).
__device__ __forceinline__ float bs_coord(int t, int npix, int npsi, float m, float r) {
  const float half = (m - 1.0f) / 2.0f;
  return (m * (float)(t - npix / 2) - r + half) + (float)(npsi / 2);
}

// The same coordinate split into its integer part and fractional offset, which
// is what the taps use: x = m (t - npix/2) - r + (m - 1)/2 + npsi/2 is formed in
// FP64 (exact for these operands), so the offset d in [0, 1) carries FP32
// precision.  An FP32 coordinate near 1000 is only good to 6e-5 of a pixel,
// the dominant error of S against FP64 at 2048^2 detectors.  Every tap weight
// (S, its derivatives and the gather adjoints) comes from this one function, so
// the adjoint pairs use identical weights.
struct BsPos {
  int i;    // floor(x)
  float d;  // x - floor(x)
};
__device__ __forceinline__ BsPos bs_pos(int t, int npix, int npsi, float m, float r) {
  const float half = (m - 1.0f) / 2.0f;
  const double x = (double)m * (double)(t - npix / 2) - (double)r + (double)half + (double)(npsi / 2);
  const double fx = floor(x);
  return BsPos{(int)fx, (float)(x - fx)};
}

// Sadj as a gather: candidate detector pixels [lo, hi] whose taps can reach
// coefficient index i, bracketed analytically with a one-pixel margin (each is
// then re-evaluated with the forward's exact float expression).
__device__ __forceinline__ void bs_candidates(int i, int npix, int npsi, float mb, float rr, int& lo,
                                              int& hi) {
  const float off = bs_coord(0, npix, npsi, mb, rr) + mb * (float)(npix / 2);
  const float a = ((float)i - 2.0f - off) / mb + (float)(npix / 2);
  const float bnd = ((float)i + 2.0f - off) / mb + (float)(npix / 2);
  lo = (int)floorf(fminf(a, bnd)) - 1;
  hi = (int)ceilf(fmaxf(a, bnd)) + 1;
  lo = lo < 0 ? 0 : lo;
  hi = hi > npix - 1 ? npix - 1 : hi;
}

// weight with which sampling position p reaches coefficient index i (0 if none)
__device__ __forceinline__ float bs_reach(BsPos p, int i) {
  const int j = i - p.i;  // tap offset, valid in [-1, 2]
  if (j < -1 || j > 2) return 0.0f;
  float w[4];
  bs_w(p.d, w);
  return w[j + 1];
}

// Block-wide sum of a float2 (fixed order: wave shuffles, then LDS).
template <int NT>
__device__ __forceinline__ float2 block_sum2(float2 v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v.x += __shfl_xor(v.x, off, 64);
    v.y += __shfl_xor(v.y, off, 64);
  }
  constexpr int NW = NT / 64;
  __shared__ float2 red[NW];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float2 s = make_float2(0.0f, 0.0f);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      s.x += red[i].x;
      s.y += red[i].y;
    }
  }
  return s;
}

// ---- Sadj of one tile of coefficients, magnification >= 1 ------------------------
// acc[rr] += sum over detector rows ty, then columns tx, of wy wx g[ty][tx] for
// the coefficients (iy0 + wave kAtR + rr, ix0 + lane) of a 64 x kAtY tile (a
// workgroup of 256 threads).  The detector pixels that reach the tile are
// staged in LDS once; each detector row's x sums are formed once and serve all
// coefficient rows that weigh them, so an output costs about 5 reads for x and
// 4 for y, all from LDS.  Walking the candidates per output row group read each
// pixel some 28 times through the L1, eight predicated loads to a row, and waited
// for each row; here all loads of a tile are in flight together.
// The larger the magnification, the fewer pixels reach a tile and the more the
// weights cost (candidates are tried in FP64): they are formed once for a tile,
// rows by one wavefront and columns by another, and a tile that no pixel reaches
// ends at once.  384 planes of 256^2: walking the candidates 271 us at
// magnification 1, 149 at 1.5, 121 at 1.92, 81 at 4; tiles with the column
// weights formed by every wavefront and all 44 x 76 pixels asked for 136, 125,
// 119 and 108; so 124, 99, 94 and 80.
// Magnification >= 1 leaves at most 4 pixels with a weight along each axis,
// consecutive ones within the first 8 of the bracket; taps that are not there
// read a zeroed slot, so nothing else enters the sums, which run in the order of
// the walk (ascending rows, ascending columns).
constexpr int kAtX = 64, kAtR = 8, kAtY = 4 * kAtR;
constexpr int kAtNX = kAtX + 12, kAtNY = kAtY + 12;  // brackets: (tile + 3) / m + 4 and the margins

template <typename TO>
struct AdjTile {
  TO g[kAtNY][kAtNX + 1];    // the last column of each row stays zero
  TO tmp[kAtNY + 1][kAtX];   // x sums; the last row stays zero
  float wy[kAtY][4], wx[kAtX][4];
  int fy[kAtY], fx[kAtX];
};

// 4 consecutive weights w with which index i collects pixels f .. f + 3 (f = -1: none)
__device__ __forceinline__ int bs_adj_taps(int i, int npix, int npsi, float mb, float r, float (&w)[4]) {
  int lo, hi, f = -1;
  bs_candidates(i, npix, npsi, mb, r, lo, hi);
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = 0.0f;
  hi = min(hi, lo + 7);
#pragma unroll 2
  for (int p = lo; p <= hi; ++p) {
    const float v = bs_reach(bs_pos(p, npix, npsi, mb, r), i);
    if (f < 0 && v != 0.0f) f = p;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (f >= 0 && p == f + j) w[j] = v;
  }
  return f;
}

// Once per kernel, before the first adj_tile_add (which begins with a barrier).
template <typename TO>
__device__ __forceinline__ void adj_tile_init(AdjTile<TO>& s) {
  if (threadIdx.x < kAtNY) s.g[threadIdx.x][kAtNX] = vzero<TO>();
  if (threadIdx.x < kAtX) s.tmp[kAtNY][threadIdx.x] = vzero<TO>();
}

template <typename TO, typename LOAD>
__device__ __forceinline__ void adj_tile_add(AdjTile<TO>& s, int ix0, int iy0, int n, int nz, int npsi, int nzpsi,
                                             float mb, float rx, float ry, const LOAD& load, TO (&acc)[kAtR]) {
  const int t = threadIdx.x, c = t & 63, wv = t >> 6;
  // detector pixels whose taps can reach the tile
  int xlo, xhi, ylo, yhi, unused;
  bs_candidates(ix0, n, npsi, mb, rx, xlo, unused);
  bs_candidates(min(ix0 + kAtX, npsi) - 1, n, npsi, mb, rx, unused, xhi);
  bs_candidates(iy0, nz, nzpsi, mb, ry, ylo, unused);
  bs_candidates(min(iy0 + kAtY, nzpsi) - 1, nz, nzpsi, mb, ry, unused, yhi);
  const int ncol = min(xhi - xlo + 1, kAtNX), nrow = min(yhi - ylo + 1, kAtNY);
  if (ncol <= 0 || nrow <= 0) return;  // the whole workgroup: nothing reaches the tile
  __syncthreads();                     // the last tile's sums have been read
  // (a position that is not finite gives a bracket anywhere: only pixels that
  // exist are read, and those with a weight do).  All loads are issued before
  // the first is stored.
  constexpr int NE = kAtNX - 64, NR = kAtNY / 4, NL = (kAtNY * NE + 255) / 256;
  TO v[NR + NL];
  auto at = [&](int r, int k) {
    const unsigned ty = (unsigned)ylo + r, tx = (unsigned)xlo + k;
    return r < nrow && k < ncol && tx < (unsigned)n && ty < (unsigned)nz ? load((int)ty, (int)tx) : vzero<TO>();
  };
  // rows beyond the first 24 and columns beyond 64 are there at magnifications
  // below about 1.9 and 1.1
  constexpr int NH = 6;
  const bool tall = nrow > 4 * NH, wide = ncol > 64;
#pragma unroll
  for (int i = 0; i < NH; ++i) v[i] = at(wv + 4 * i, c);
  if (tall) {
#pragma unroll
    for (int i = NH; i < NR; ++i) v[i] = at(wv + 4 * i, c);
  }
  if (wide) {
#pragma unroll
    for (int i = 0; i < NL; ++i) v[NR + i] = at((t + 256 * i) / NE, 64 + (t + 256 * i) % NE);
  }
  // the tile's weights, once: rows by the first wavefront, columns by the second
  if (t < kAtX + kAtX && (wv || t < kAtY)) {
    const int i = wv ? ix0 + c : iy0 + t;
    const bool in = i < (wv ? npsi : nzpsi);
    float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int f = -1;
    if (in) f = wv ? bs_adj_taps(i, n, npsi, mb, rx, w) : bs_adj_taps(i, nz, nzpsi, mb, ry, w);
    float* dst = wv ? s.wx[c] : s.wy[t];
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[j] = w[j];
    (wv ? s.fx[c] : s.fy[t]) = f;
  }
#pragma unroll
  for (int i = 0; i < NH; ++i) s.g[wv + 4 * i][c] = v[i];
  if (tall) {
#pragma unroll
    for (int i = NH; i < NR; ++i) s.g[wv + 4 * i][c] = v[i];
  }
  if (wide) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      if (t + 256 * i < kAtNY * NE) s.g[(t + 256 * i) / NE][64 + (t + 256 * i) % NE] = v[NR + i];
  }
  __syncthreads();
  float wx[4];
  int ox[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    wx[j] = s.wx[c][j];
    ox[j] = wx[j] != 0.0f ? s.fx[c] - xlo + j : kAtNX;
  }
  for (int r = wv; r < nrow; r += 4) {
    TO sum = vzero<TO>();
#pragma unroll
    for (int j = 0; j < 4; ++j) sum = vfma(wx[j], s.g[r][ox[j]], sum);
    s.tmp[r][c] = sum;
  }
  __syncthreads();
#pragma unroll
  for (int rr = 0; rr < kAtR; ++rr) {
    const int row = wv * kAtR + rr, f = s.fy[row];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float w = s.wy[row][j];
      acc[rr] = vfma(w, s.tmp[w != 0.0f ? f - ylo + j : kAtNY][c], acc[rr]);
    }
  }
}

// ---- launch interface ------------------------------------------------------
template <typename T>
struct BsArgs {
  const T* c = nullptr;   // coefficients [B, nzpsi, npsi] (adjoint: input g [B, nz, n])
  const T* c1 = nullptr;
  const T* c2 = nullptr;
  const float* r = nullptr;    // shifts, (y, x) at r[b*rs + 0/1]
  const float* m = nullptr;    // magnification at m[b*ms]
  const float* dr1 = nullptr;  // differential shifts
  const float* dr2 = nullptr;
  T* out = nullptr;
  int64_t rs = 2, ms = 1, d1s = 2, d2s = 2;
  int64_t batch = 0;
  int n = 0, nz = 0, npsi = 0, nzpsi = 0;
  int tiles_x = 0, tiles_y = 0;
};

constexpr int kPfH = 12;  // prefilter taps |d| <= kPfH
struct PrefilterTaps {
  float wx[2 * kPfH + 1];
  float wy[2 * kPfH + 1];
};

template <typename T> hipError_t bs_launch_forward(BsArgs<T> a, int mode, hipStream_t st);
template <typename T> hipError_t bs_launch_adjoint(BsArgs<T> a, hipStream_t st);
template <typename T> int64_t bs_dadj_partials(const BsArgs<T>& a);
template <typename T>
hipError_t bs_launch_dadj_reduce(BsArgs<T> a, const T* g, float2* partial, float* out2, hipStream_t st);
// Optional per-plane addresses of the prefilter's input and output (device
// arrays of batch pointers); a NULL table means plane b at in / out + b * plane.
template <typename T>
struct PlaneTab {
  const T* const* in = nullptr;
  T* const* out = nullptr;
};
template <typename T>
hipError_t bs_launch_prefilter(const T* in, T* out, int64_t batch, int nzpsi, int npsi,
                               const PrefilterTaps& taps, hipStream_t st, PlaneTab<T> tab = PlaneTab<T>());

}  // namespace htamd
