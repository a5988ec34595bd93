// Pieces shared by the fused BH passes (gradient and bilinear form): value
// conversions between the object type and complex, the staged-row LDS span,
// the plan that binds a propagator and a shift plan, and the stage-timing hook.
#pragma once
#include "../../include/htamd.h"
#include "fresnel_core.hpp"
#include "htamd_bspline.hpp"
#include "htamd_internal.hpp"

namespace htamd {

template <typename TO> __device__ __forceinline__ float2 to_c(TO v);
template <> __device__ __forceinline__ float2 to_c<float>(float v) { return make_float2(v, 0.f); }
template <> __device__ __forceinline__ float2 to_c<float2>(float2 v) { return v; }
template <typename TO> __device__ __forceinline__ TO from_c(float2 v);
template <> __device__ __forceinline__ float from_c<float>(float2 v) { return v.x; }
template <> __device__ __forceinline__ float2 from_c<float2>(float2 v) { return v; }

// Row-staged gathers.  All pixels of a detector row sample the same four
// object rows (iy .. iy+3), so those rows are combined along y once per
// (angle, row) into LDS with coalesced reads of the coefficients, and each
// pixel then reads 4 LDS values instead of 16 scattered global ones.
__device__ __forceinline__ unsigned char* dyn_lds() {
  extern __shared__ __align__(16) unsigned char htamd_dyn_lds[];
  return htamd_dyn_lds;
}

template <int N>
__device__ __forceinline__ void row_span(int npsi, float mb, float rx, int& lo, int& hi) {
  // the sampling position is monotone in the pixel index, so the row's taps
  // lie within [floor(x(0)) - 1, floor(x(N-1)) + 2] (the floors of bs_pos, which
  // every gather uses)
  const int i0 = bs_pos(0, N, npsi, mb, rx).i, i1 = bs_pos(N - 1, N, npsi, mb, rx).i;
  lo = max(min(i0, i1) - 1, 0);
  hi = min(max(i0, i1) + 3, npsi);
}

// Optional timing hook: events[2k] / events[2k+1] are recorded before / after
// stage k (0 prefilter, 1 rows forward, 2 columns, 3 rows adjoint, 4 Sadj,
// 5 prefilter of the gradient, 6 reductions) on the launch stream.
struct StageEvents {
  hipEvent_t* ev = nullptr;
  int count = 0;
  void mark(int idx, hipStream_t st) const {
    if (ev && idx < count && ev[idx]) (void)hipEventRecord(ev[idx], st);
  }
};

// Workgroup -> row units of the row passes.  Contiguous bands put the XCDs
// ndist nz n bytes apart, which with one to three distances costs up to 9%
// against chunks of 16 workgroups in turn (gradient at 2048^2, 16 angles: 1
// distance 2706 -> 2462 us, 2 distances 8 angles 2493 -> 2299 us; 1024^2, 2
// distances 2334 -> 2160 us).  From four distances on the bands are distances
// whose rows sample the same object rows at the same time, and are better (4
// distances: 8264 against 8327 us; bilinear pair at 1024^2 4422 against 4515).
__device__ __forceinline__ int64_t row_tile(int64_t bid, int64_t nblocks, int ndist) {
  return ndist >= 4 ? xcd_tile(bid, nblocks) : xcd_chunks<16>(bid, nblocks);
}

// With at least this many groups of angles each XCD takes whole groups instead
// (gradient at 256^2, 2 distances, 48 angles: 417 -> 407 us; equal form at
// 256^2, 3 distances, 64 angles 637 -> 618 us).
constexpr int kXcdGroups = 8;

constexpr int64_t kCuLds = 160 * 1024;

// Whether `blocks` workgroups, of which a CU holds per_cu (at most waves_cu
// by their registers, and what their LDS leaves room for), run in whole
// rounds of the chip, or nearly so, and in at most `most` of them.
inline bool whole_rounds(int64_t blocks, int64_t waves_cu, int64_t lds, int64_t most) {
  const int64_t by_lds = lds > 0 ? kCuLds / lds : waves_cu;
  const int64_t per_round = kNumCu * (by_lds < 1 ? 1 : by_lds < waves_cu ? by_lds : waves_cu);
  const int64_t rounds = (blocks + per_round - 1) / per_round;
  return rounds <= most && 10 * blocks >= 9 * rounds * per_round;
}

inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

}  // namespace htamd

struct htamd_bh_plan {
  // binds the plans of one geometry; the fused passes take their tables from them
  const htamd_prop_plan* prop = nullptr;
  const htamd_shift_plan* shift = nullptr;
  htamd::StageEvents events;
};

