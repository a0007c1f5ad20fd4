// Object-increment gather of the DM iterations: sum over the frames that cover an object pixel of
// the (optionally phase-clamped) increments s_O conj(P) psi_new, in ascending frame order, FP64.
#pragma once
#include "ptyk_device.h"
#include "ptyk_internal.h"

namespace ptyk {

constexpr bool dm_may_share(int m) { return m < 512; }  // see dm_share_lists

// A column of an object row is one thread's, or SPLIT threads' of different waves (SHARE).  The frames
// come from the list of the tile of PTYK_DM_TR rows x dm_tile_width(M) columns around it, so few of them
// miss the row and none the columns altogether.  Each of the SPLIT parts takes a share of the list, U
// frames at a time, all their loads issued before the in-order accumulation; the parts add up in order.
// Bound by the reads of psi_new, and on small frames by the chain of a long list over few workgroups, so
// the row is cut finer there and the list shared out: 400 frames of 128^2 44 -> 19 us, 512 of 256^2 (among
// other scans) 105 -> 60, against one list per object row, 256 columns a workgroup and 4 frames at a time.
// Returns the sum to the threads that have(): one per column.
template <int M, bool SHARE>
struct ObjRow {
  static constexpr int TC = dm_tile_width(M), SPLIT = SHARE ? PTYK_NT / TC : 1;
  static constexpr int COLS = PTYK_NT / SPLIT;  // columns of a workgroup
  static_assert(PTYK_NT % TC == 0, "one column and part per thread");
  // column of this thread, its tile's offset in a row of tiles, and its part of the list; tile and part
  // are the same for a whole wave: said so, its list and ROI reads are scalar (as vector reads they made
  // the 512^2 gather twice as long)
  int c, tile, part;
  __device__ __forceinline__ ObjRow() {
    const int seg = __builtin_amdgcn_readfirstlane(threadIdx.x / TC);
    part = SHARE ? seg : 0;
    c = blockIdx.y * COLS + threadIdx.x % COLS;
    tile = blockIdx.y * (COLS / TC) + (SHARE ? 0 : seg);
  }
  __device__ __forceinline__ bool have(int obj_cols) const { return part == 0 && c < obj_cols; }
  // the list of the tile around row p; empty past the last tile
  __device__ __forceinline__ void list(const int* __restrict__ tile_ptr, int p, int obj_cols, int* k0, int* k1) const {
    const int tiles = (obj_cols + TC - 1) / TC;
    *k0 = *k1 = 0;
    if (tile < tiles) {
      const int t = p / PTYK_DM_TR * tiles + tile;
      *k0 = tile_ptr[t];
      *k1 = tile_ptr[t + 1];
    }
  }
};
template <int M, bool SHARE>
__device__ __forceinline__ double2 obj_row_sum(const ObjRow<M, SHARE>& at, int p, const float2* __restrict__ psi,
                                               const float2* __restrict__ probe, const int2* __restrict__ roi,
                                               const int* __restrict__ frames, int k0, int k1, float so,
                                               int phase_constraint) {
  constexpr int TC = dm_tile_width(M), SPLIT = ObjRow<M, SHARE>::SPLIT, U = 8;
  const int part = at.part, c = at.c;
  const int lo = k0 + (int)((long)(k1 - k0) * part / SPLIT), hi = k0 + (int)((long)(k1 - k0) * (part + 1) / SPLIT);
  double ax = 0.0, ay = 0.0;
  for (int kb = lo; kb < hi; kb += U) {
    float2 pv[U], sv[U];
    bool act[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = frames[min(kb + u, hi - 1)];
      const int2 r = roi[j];
      const int q = p - r.x, cc = c - r.y;
      act[u] = kb + u < hi && cc >= 0 && cc < M && q >= 0 && q < M;
      if (act[u]) {
        pv[u] = probe[q * M + cc];
        sv[u] = psi[((long)j * M + q) * M + cc];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!act[u]) continue;
      float2 t = cscale(cmulcj(pv[u], sv[u]), so);
      if (phase_constraint) t = clamp_phase(t);
      ax += t.x;
      ay += t.y;
    }
  }
  if constexpr (SPLIT > 1) {
    __shared__ double2 parts[(SPLIT - 1) * TC];
    if (part) parts[threadIdx.x - TC] = make_double2(ax, ay);
    __syncthreads();
    if (part == 0) {
#pragma unroll
      for (int i = 0; i < SPLIT - 1; ++i) {
        const double2 t = parts[i * TC + threadIdx.x];
        ax += t.x;
        ay += t.y;
      }
    }
  }
  return make_double2(ax, ay);
}

// Lists are shared out where whole columns leave too few workgroups (rows x 256 columns) for the lists'
// length, which grows with the frame; past that, four times the workgroups with a quarter of the columns
// cost more than they gain.  us an iteration, whole and shared: 64^2, 400 frames on 164^2 152 and 102,
// 314^2 100 and 87, 600^2 (1800 workgroups) 88 and 96, 4000^2 203 and 528; 128^2, 400 frames on 228^2 230
// and 145, 600^2 (1800) 136 and 131, 1000^2 (4000) 143 and 153; 256^2, 1000 frames on 406^2 1115 and 984,
// 1200^2 998 and 977, 200 frames on 2000^2 259 and 280.  At 512^2 the reads bind: 900 frames on 1036^2 3319
// and 3310, 100 on 612^2 390 and 403.
inline bool dm_share_lists(int m, long rows, int obj_cols) {
  return dm_may_share(m) && rows * ((obj_cols + PTYK_NT - 1) / PTYK_NT) < 24L * m;
}

}  // namespace ptyk
