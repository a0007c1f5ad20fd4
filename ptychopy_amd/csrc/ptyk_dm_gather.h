// Object-increment gather of the DM iterations: sum over the frames that cover an object pixel of
// the (optionally phase-clamped) increments s_O conj(P) psi_new, in ascending frame order, FP64.
#pragma once
#include "ptyk_device.h"
#include "ptyk_internal.h"

namespace ptyk {

// A workgroup owns dm_tile_width(M) columns of one object row; the frames come from the list of the
// tile of PTYK_DM_TR rows around it, so few of them miss the row and none the columns altogether.
// Each of its SPLIT parts takes a share of the list, U frames at a time, all their loads issued before
// the in-order accumulation; the parts add up in order.  Bound by the reads of psi_new, and on small
// frames by the chain of a long list over few workgroups, so the row is cut finer there and the list
// shared out: 400 frames of 128^2 44 -> 19 us, 512 of 256^2 (among other scans) 105 -> 60, 64 of 512^2
// 35 -> 31, against one list per object row, 256 columns a workgroup and 4 frames at a time.
// Returns the sum to the threads of part 0 (threadIdx.x < dm_tile_width(M)).
template <int M>
__device__ __forceinline__ double2 obj_row_sum(int p, int c, const float2* __restrict__ psi,
                                               const float2* __restrict__ probe, const int2* __restrict__ roi,
                                               const int* __restrict__ frames, int k0, int k1, float so,
                                               int phase_constraint) {
  constexpr int TC = dm_tile_width(M), SPLIT = PTYK_NT / TC, U = 8;
  static_assert(SPLIT * TC == PTYK_NT, "one column and part per thread");
  // the part is the same for a whole wave: said so, its list and ROI reads are scalar (as vector reads
  // they made the 512^2 gather twice as long)
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / TC);
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

}  // namespace ptyk
