// ePIE iteration on gfx950 (replaces ePIE.cpp:65-129 and the kernels it drives:
// d_extractObjectArray (SampleKernels.cu:167-178), d_complexMultiply, the cuFFT pair of
// applyModulusConstraint (utilities.cpp:138-154) with d_adjustFFT / d_adjustModalFFT
// (utilitiesKernels.cu:633-682), d_updateObjectArray(M) (SampleKernels.cu:244-294),
// d_updateProbe(M) (ProbeKernels.cu:425-458), the thrust maxima behind
// Sample/Probe::updateMaxIntensity and d_calculateER (utilitiesKernels.cu:684-712)).
//
// ePIE is a chain of dependent position updates, so one launch walks every position of an
// iteration in the given order, with no host round trip per position.  Frames of 64^2 and more
// are shared by a team of 16 to 128 workgroups (k_epie_team); smaller ones go to one workgroup that
// keeps the exit waves in an L2-resident scratch and stages each 2D transform through LDS in row
// and column chunks (k_epie).
#include "../../include/ptyk.h"
#include "ptyk_device.h"
#include "ptyk_internal.h"
#include "ptyk_team.h"

#include <algorithm>

namespace ptyk {

#define PTYK_EPIE_NT 1024

template <int M, int NT>
struct WgFft {
  static constexpr int RNB = plan_min_batch<M, NT>();
  static constexpr int CNB = (plan_min_batch<M, NT>() + 15) / 16 * 16;
  static constexpr int LDS = (RNB > CNB ? RNB : CNB) * M;  // float2 elements
};

// In-place 2D transform of one M x M frame held in global memory by one workgroup.
template <int M, bool INV, int NT>
__device__ void wg_fft2(float2* __restrict__ g, float2* lds, const float2* __restrict__ tw) {
  constexpr int RNB = WgFft<M, NT>::RNB;
  constexpr int CNB = WgFft<M, NT>::CNB;
  const int tid = threadIdx.x;
  for (int r0 = 0; r0 < M; r0 += RNB) {
    for (int e = tid; e < RNB * M; e += NT) {
      const int row = r0 + e / M;
      lds[e] = row < M ? g[row * M + (e % M)] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft_lds<M, INV, RNB, NT, RowLayout<M, M>, false, false>(lds, tw, tid);
    for (int e = tid; e < RNB * M; e += NT) {
      const int row = r0 + e / M;
      if (row < M) g[row * M + (e % M)] = lds[e];
    }
    __syncthreads();
  }
  for (int c0 = 0; c0 < M; c0 += CNB) {
    for (int e = tid; e < CNB * M; e += NT) {
      const int col = c0 + e % CNB;
      lds[e] = col < M ? g[(e / CNB) * M + col] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft_lds<M, INV, CNB, NT, ColLayout<CNB>, true, false>(lds, tw, tid);
    for (int e = tid; e < CNB * M; e += NT) {
      const int col = c0 + e % CNB;
      if (col < M) g[(e / CNB) * M + col] = lds[e];
    }
    __syncthreads();
  }
}

// Bilinear sample with clamp addressing, matching a linear-filtered, unnormalised texture
// fetch at (u, v) = (col + offY + 0.5, row + offX + 0.5) (SampleKernels.cu:167-178, 493-508).
// quantize: round the weights to 1/256 (8 fractional bits, as texture units store them).
// The sample in steps (tap position and weights; clamped tap indices; the four gathers; the
// weighted sum), so that callers can issue the gathers of several samples before combining any,
// or take the taps from a staged copy of the object.
struct TapPos {
  int i0, j0;  // column and row of the first tap, before clamping
  float al, be;
};
template <bool QUANT>
__device__ __forceinline__ TapPos tap_pos(float u, float v) {
  const float xb = u - 0.5f, yb = v - 0.5f;
  const float fx = floorf(xb), fy = floorf(yb);
  TapPos p;
  p.al = xb - fx;
  p.be = yb - fy;
  if (QUANT) {
    p.al = rintf(p.al * 256.f) * (1.f / 256.f);
    p.be = rintf(p.be * 256.f) * (1.f / 256.f);
  }
  p.i0 = (int)fx;
  p.j0 = (int)fy;
  return p;
}
__device__ __forceinline__ float2 bilinear_sum(float al, float be, float2 t00, float2 t01, float2 t10, float2 t11) {
  const float w00 = (1.f - al) * (1.f - be), w01 = al * (1.f - be), w10 = (1.f - al) * be, w11 = al * be;
  return make_float2(w00 * t00.x + w01 * t01.x + w10 * t10.x + w11 * t11.x,
                     w00 * t00.y + w01 * t01.y + w10 * t10.y + w11 * t11.y);
}
template <bool QUANT>
__device__ __forceinline__ float2 bilinear_t(const float2* __restrict__ o, int rows, int cols, float u, float v) {
  const TapPos p = tap_pos<QUANT>(u, v);
  const int i0 = min(max(p.i0, 0), cols - 1), i1 = min(max(p.i0 + 1, 0), cols - 1);
  const int j0 = min(max(p.j0, 0), rows - 1), j1 = min(max(p.j0 + 1, 0), rows - 1);
  return bilinear_sum(p.al, p.be, o[(long)j0 * cols + i0], o[(long)j0 * cols + i1], o[(long)j1 * cols + i0],
                      o[(long)j1 * cols + i1]);
}
__device__ __forceinline__ float2 bilinear(const float2* __restrict__ o, int rows, int cols, float u, float v,
                                           int quantize) {
  return quantize ? bilinear_t<true>(o, rows, cols, u, v) : bilinear_t<false>(o, rows, cols, u, v);
}

template <int M>
__global__ __launch_bounds__(PTYK_EPIE_NT) void k_epie(EpieArgs a) {
  extern __shared__ float2 lds[];
  __shared__ float redf[PTYK_EPIE_NT / 64];
  __shared__ double redd[PTYK_EPIE_NT / 64];
  constexpr int NT = PTYK_EPIE_NT;
  constexpr int MM = M * M;
  const int tid = threadIdx.x;
  const int ku = a.k_use;
  // The reference keeps these maxima as float (real_t); factors are 1.0/max rounded to float.
  float obj_max = (float)a.scal[0];
  float probe_max = (float)a.scal[1];
  double err = 0.0;
  const long canvas = (long)a.obj_rows * a.obj_cols;

  for (int s = 0; s < a.n_pos; ++s) {
    const int fi = a.order[s];
    const float2 pos = a.pos[fi];
    const float ascale = a.amp_scale[fi];
    const __half* amp = a.amp + (long)fi * MM;

    // psi_old_k = ROI * P_k  (bilinear ROI at the fractional position)
    for (int px = tid; px < MM; px += NT) {
      const int ii = px / M, jj = px % M;
      const float2 roi = bilinear(a.obj, a.obj_rows, a.obj_cols, (float)jj + pos.y + 0.5f, (float)ii + pos.x + 0.5f,
                                  a.tex_quantize);
      for (int k = 0; k < ku; ++k) {
        const float2 v = cmul(roi, a.probe[(long)k * MM + px]);
        a.psi_old[(long)k * MM + px] = v;
        a.psi[(long)k * MM + px] = v;
      }
    }
    __syncthreads();
    for (int k = 0; k < ku; ++k) wg_fft2<M, false, NT>(a.psi + (long)k * MM, lds, a.tw);

    // Fourier modulus constraint (d_adjustFFT / d_adjustModalFFT)
    const float nrm = 1.f / (float)MM;
    for (int px = tid; px < MM; px += NT) {
      const float A = load_amp(amp, px, ascale);
      if (ku == 1) {
        a.psi[px] = modulus_phase(a.psi[px], A, nrm);
      } else {
        float ms = 0.f;
        for (int k = 0; k < ku; ++k) ms += cabs2(a.psi[(long)k * MM + px]);
        const float f = A * rsqrtf(ms) * nrm;
        for (int k = 0; k < ku; ++k) a.psi[(long)k * MM + px] = cscale(a.psi[(long)k * MM + px], f);
      }
    }
    __syncthreads();
    for (int k = 0; k < ku; ++k) wg_fft2<M, true, NT>(a.psi + (long)k * MM, lds, a.tw);

    // Object update at the rounded position (d_updateObjectArray(M))
    const int rx = (int)roundf(pos.x), ry = (int)roundf(pos.y);
    const float co = (float)(1.0 / (double)probe_max);
    for (int px = tid; px < MM; px += NT) {
      const int ii = px / M, jj = px % M;
      float2 u = make_float2(0.f, 0.f);
      for (int k = 0; k < ku; ++k) {
        const long q = (long)k * MM + px;
        u = cadd(u, cmulcj(a.probe[q], csub(a.psi[q], a.psi_old[q])));
      }
      const long oi = (long)(rx + ii) * a.obj_cols + (ry + jj);
      float2 o = cadd(a.obj[oi], cscale(u, co));
      const float mag = sqrtf(o.x * o.x + o.y * o.y);
      if (a.phase_constraint) o = clamp_phase(o);
      a.obj[oi] = o;
      a.obj_int[oi] = mag * mag;
    }
    __syncthreads();
    {
      float mx = 0.f;
      for (long q = tid; q < canvas; q += NT) mx = fmaxf(mx, a.obj_int[q]);
      obj_max = block_max<NT>(mx, redf);
    }

    // Probe update with the updated object (d_updateProbe(M)); Probe::updateMaxIntensity
    if (a.update_probe) {
      const float cp = (float)(1.0 / (double)obj_max);
      for (int px = tid; px < MM; px += NT) {
        const int ii = px / M, jj = px % M;
        const float2 oc = a.obj[(long)(rx + ii) * a.obj_cols + (ry + jj)];
        for (int k = 0; k < ku; ++k) {
          const long q = (long)k * MM + px;
          float2 p = cadd(cscale(cmulcj(oc, csub(a.psi[q], a.psi_old[q])), cp), a.probe[q]);
          a.probe[q] = p;
          const float ia = sqrtf(p.x * p.x + p.y * p.y);
          a.probe_int[q] = ia * ia;
        }
      }
      __syncthreads();
      float mx = 0.f;
      if (a.modal) {
        for (int px = tid; px < MM; px += NT) {
          float sm = 0.f;
          for (int k = 0; k < a.k_total; ++k) sm += a.probe_int[(long)k * MM + px];
          mx = fmaxf(mx, sm);
        }
      } else {
        for (long q = tid; q < (long)a.k_total * MM; q += NT) mx = fmaxf(mx, a.probe_int[q]);
      }
      probe_max = block_max<NT>(mx, redf);
    }

    // Optional Fourier error (PhaserUtil::calculateER; ePIE.cpp:124-125)
    if (a.rms) {
      for (int k = 0; k < ku; ++k) wg_fft2<M, false, NT>(a.psi_old + (long)k * MM, lds, a.tw);
      double acc = 0.0;
      for (int px = tid; px < MM; px += NT) {
        float2 sm = make_float2(0.f, 0.f);
        for (int k = 0; k < ku; ++k) sm = cadd(sm, a.psi_old[(long)k * MM + px]);
        acc += fabs((double)load_amp(amp, px, ascale) - sqrt((double)sm.x * sm.x + (double)sm.y * sm.y));
      }
      acc = block_sum<NT>(acc, redd);
      err += acc / ku / (double)a.amp_sum[fi];
    }
    __syncthreads();
  }
  if (tid == 0) {
    a.scal[0] = obj_max;
    a.scal[1] = probe_max;
    a.scal[2] = err;
  }
}

// ---------------------------------------------------------------- team form (M >= 64)
// A position's work is spread over a team of W workgroups that stay on the chip for the whole
// iteration.  Workgroup w owns R = M / W rows of the frame (and of the probe) and, between the two
// transform directions, C = R of its columns:
//   rows    : ROI (bilinear) x P_k, row transform                     -> exchange buffer
//   columns : column transform, modulus difference, inverse transform -> exchange buffer
//   rows    : inverse row transform = psi - psi_old, object update, then the probe update
// with a team barrier after each step (the last one also publishes the object for the next
// position's ROI), so three barriers a position.  psi - psi_old comes out directly, since the
// column step transforms Psi' - Psi / M^2 (the transform is linear); the Fourier error is of
// psi_old's spectrum, which is Psi itself, and is summed there too.
//
// What bounds it: the chain of three exchanges through the cache shared by the XCDs, not bytes or
// arithmetic.  So every value another workgroup reads (exchange buffer, object, |O|^2, maxima) is
// written and read with device-scope accesses, which go to that cache by themselves, and a barrier
// is a wait for the stores to be acknowledged, one flag store and a poll: no cache is written back
// or invalidated (an agent-scope release here writes back a whole L2).  A thread holds 4 values, so a
// transform is 3 or 4 short stages between two LDS tiles with one workgroup barrier each, its twiddles
// kept in registers for the whole iteration.
//
// Team sizes: 4 rows a workgroup.  More rows mean fewer flags to wait for but more instructions per
// thread in every step of the chain (64^2 in 8 workgroups of 8 rows: 14.0 us a position, in 16 of 4:
// 10.7; 128^2 in 16: 15.0, in 32: 12.0; 256^2 with three modes in 32: 42.6, in 64: 28.6; 512^2 in 64:
// 33, in 128: 27; all with the copies to the host; the iteration alone is now 10.1, 10.9, 24.4 and 16.6).
// One workgroup on one CU took 14.7, 44, 1120 and 1730.  The radix order of 128
// is the one of the least error (median 1.5e-6 of the object over an iteration of the 12 x 12
// benchmark scan; 2.0e-6 for 4 4 4 2).
template <int M> struct TeamCfg;
template <> struct TeamCfg<64>  { static constexpr int W = 16,  NT = 64,  S = 3, R0 = 4, R1 = 4, R2 = 4, R3 = 1; };
template <> struct TeamCfg<128> { static constexpr int W = 32,  NT = 128, S = 4, R0 = 4, R1 = 4, R2 = 2, R3 = 4; };
template <> struct TeamCfg<256> { static constexpr int W = 64,  NT = 256, S = 4, R0 = 4, R1 = 4, R2 = 4, R3 = 4; };
template <> struct TeamCfg<512> { static constexpr int W = 128, NT = 512, S = 3, R0 = 8, R1 = 8, R2 = 8, R3 = 1; };

template <int M>
struct Team : TeamCfg<M> {
  using T = TeamCfg<M>;
  static constexpr int R = M / T::W;         // rows (and columns) of a workgroup
  static constexpr int P = M + 8;            // pitch of a sequence in an LDS tile
  static constexpr int TILE = R * P;         // float2 elements
  static constexpr int PPT = R * M / T::NT;  // values per thread
  static constexpr int WR = R + 2, WC = M + 2, WIN = WR * WC;  // object window behind the rows' ROI
  static constexpr int WU = (WIN + T::NT - 1) / T::NT;
  static constexpr int TILE_B = TILE > WIN ? TILE : WIN;  // the second tile also stages the window
  static constexpr int TPR = T::NT / R;      // threads per row of the scan beside the ROI
  static constexpr int NB = (2 * (PTYK_EPIE_SEG - 1) + TPR - 1) / TPR;  // pixels of it per thread
  static constexpr int CELLS = M / PTYK_EPIE_SEG + 1;                   // segments an ROI row may touch
  static_assert(T::R0 * T::R1 * T::R2 * T::R3 == M && (T::S == 3 || T::S == 4), "radices");
  static_assert(PPT <= R && R % PPT == 0, "a thread's amplitudes lie in the workgroup's columns of one row");
  static_assert(TPR % 8 == 0, "threads beside the ROI: whole groups of 8 lanes per row");
  static_assert(M % PTYK_EPIE_SEG == 0 && PTYK_EPIE_SEG == 64 && R * CELLS <= 64, "a wave's pixels meet two segments");
  static_assert(R * M % T::NT == 0 && M % 64 == 0 && T::W <= PTYK_EPIE_TEAM_MAX, "tile shape");
};

// Device-scope relaxed accesses: coherent between workgroups on different XCDs by themselves.
__device__ __forceinline__ float2 ld_dev(const float2* p) {
  const unsigned long long u =
      __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((unsigned)u), __uint_as_float((unsigned)(u >> 32)));
}
__device__ __forceinline__ void st_dev(float2* p, float2 v) {
  const unsigned long long u = __float_as_uint(v.x) | ((unsigned long long)__float_as_uint(v.y) << 32);
  __hip_atomic_store((unsigned long long*)p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Team barrier in two halves, so that work which needs nothing from the others can stand between.
// arrive: this workgroup's stores have reached the coherence point (a store leaves vmcnt when it is
// acknowledged there), then its flag: the epoch and a value of the workgroup (read by thread 0 from
// LDS, in *value; a non-negative float).  wait: one wave polls all W flags, one per lane, and leaves
// the largest of the values in *most.  Why a slow reader cannot meet a later barrier's value: see
// team_word (ptyk_team.h).  The wait is bounded (limit ticks of the 100 MHz clock; 0: one
// look): the host admits no more workgroups than the device can hold at once, but other processes may
// have theirs there.  Who passes the second barrier, behind which the object is written, knows that
// all have passed the first, so that all are there; if nobody does, nothing has changed and one workgroup
// can take the iteration instead.
__device__ __forceinline__ void team_arrive(unsigned long long* flags, int w, unsigned epoch, const unsigned* value) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + team_word(w, epoch), team_flag(epoch, *value), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float wave_max_pos(float v);
template <int W>
__device__ __forceinline__ bool team_wait(const unsigned long long* flags, unsigned epoch, long long limit, int* gone,
                                          float* most) {
  if (threadIdx.x < 64) {
    const int l = threadIdx.x;
    bool ok = false;
    long long t0 = 0;
    unsigned v = 0;
    for (int i = 0;; ++i) {
      bool here = true;
      v = 0;
#pragma unroll
      for (int q = 0; q < (W + 63) / 64; ++q)
        if (W >= 64 || l < W) {
          const unsigned long long f =
              __hip_atomic_load(flags + team_word(l + q * 64, epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          here = here && team_here(f, epoch);
          v = max(v, team_value(f));  // values are non-negative floats: ordered as integers
        }
      ok = __all(here);
      if (ok || limit == 0) break;
      if (i == 1024) t0 = wall_clock64();
      if (i > 1024 && (i & 255) == 0 && wall_clock64() - t0 > limit) break;
    }
    const float m = wave_max_pos(__uint_as_float(v));
    if (l == 0) {
      *most = m;
      if (!ok) *gone = 1;
    }
  }
  __syncthreads();
  return *gone == 0;
}

// Maximum over a wave of non-negative values: in each row of 16 lanes by DPP moves, then the four
// rows' values through scalar registers (about 40 cycles; six dependent LDS permutes took 0.3 us).
template <int CTRL>
__device__ __forceinline__ float max_dpp(float v) {
  const int o = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true);
  return fmaxf(v, __int_as_float(o));
}
__device__ __forceinline__ float row16_max(float v) {
  v = max_dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  v = max_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  v = max_dpp<0x141>(v);  // row_half_mirror
  return max_dpp<0x140>(v);  // row_mirror
}
__device__ __forceinline__ float wave_max_pos(float v) {
  v = row16_max(v);
  const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// max |O|^2 of every 64 columns of every canvas row, and of every row: a wave per row, 8 segments' loads
// in flight, over the whole chip ahead of the team.  (64^2, 36 positions on 4000 x 4000, whole iteration:
// 0.41 ms; with the team's 16 waves reading the canvas first and rows to their ends per position 4.6.)
__global__ __launch_bounds__(256) void k_canvas_maxima(const float* __restrict__ obj_int, int rows, int cols,
                                                       float* __restrict__ segmax, float* __restrict__ rowmax) {
  const int lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int nseg = epie_segments(cols);
  const float* row = obj_int + (long)r * cols;
  float m = 0.f;
  for (int s0 = 0; s0 < nseg; s0 += 8) {
    float v[8], mine = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = (s0 + u) * PTYK_EPIE_SEG + lane;
      v[u] = c < cols ? fmaxf(row[c], 0.f) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float x = wave_max_pos(v[u]);
      if (lane == u) mine = x;
      m = fmaxf(m, x);
    }
    if (lane < 8 && s0 + lane < nseg) segmax[(long)r * nseg + s0 + lane] = mine;
  }
  if (lane == 0) rowmax[r] = m;
}

// One radix-RX Stockham stage of R sequences from one tile to the other.
template <int M, int RX>
struct TeamStage {
  using T = Team<M>;
  static constexpr int NB = T::R * (M / RX);                 // butterflies
  static constexpr int BPT = (NB + T::NT - 1) / T::NT;       // per thread
  static constexpr bool ALL = NB % T::NT == 0;               // every thread has BPT of them
  static constexpr int NW = RX > 1 ? BPT * (RX - 1) : 1;     // twiddles per thread
};
template <int M, int RX, int NS, bool INV>
__device__ __forceinline__ void team_stage(const float2* src, float2* dst, const float2* w, int tid) {
  using T = Team<M>;
  using G = TeamStage<M, RX>;
#pragma unroll
  for (int q = 0; q < G::BPT; ++q) {
    const int t = tid + q * T::NT, b = t / (M / RX), j = t % (M / RX);
    if (G::ALL || t < G::NB) {
      float2 v[RX];
#pragma unroll
      for (int r = 0; r < RX; ++r) v[r] = src[b * T::P + j + r * (M / RX)];
      if (NS > 1) {
#pragma unroll
        for (int r = 1; r < RX; ++r)
          v[r] = cmul(v[r], INV ? cconj(w[q * (RX - 1) + r - 1]) : w[q * (RX - 1) + r - 1]);
      }
      Dft<RX, INV>::run(v);
      const int idx = (j / NS) * NS * RX + (j % NS);
#pragma unroll
      for (int r = 0; r < RX; ++r) dst[b * T::P + idx + r * NS] = v[r];
    }
  }
  __syncthreads();
}
template <int M, int RX, int NS>
__device__ __forceinline__ void team_twiddles(float2* w, const float2* __restrict__ tw, int tid) {
  using T = Team<M>;
#pragma unroll
  for (int q = 0; q < TeamStage<M, RX>::BPT; ++q) {
    const int j = (tid + q * T::NT) % (M / RX);
#pragma unroll
    for (int r = 1; r < RX; ++r) w[q * (RX - 1) + r - 1] = tw[((j % NS) * r * (PTYK_TWN / (NS * RX))) & (PTYK_TWN - 1)];
  }
}
// Twiddles of stages 1.. of this thread (the same for rows and columns, conjugated for the inverse).
template <int M>
struct TeamTw {
  using T = Team<M>;
  float2 a[TeamStage<M, T::R1>::NW], b[TeamStage<M, T::R2>::NW], c[TeamStage<M, T::R3>::NW];
  __device__ __forceinline__ void load(const float2* __restrict__ tw, int tid) {
    team_twiddles<M, T::R1, T::R0>(a, tw, tid);
    team_twiddles<M, T::R2, T::R0 * T::R1>(b, tw, tid);
    if constexpr (T::S > 3) team_twiddles<M, T::R3, T::R0 * T::R1 * T::R2>(c, tw, tid);
  }
};
// R sequences from tile t0, with t1 as the other tile; returns the tile that holds the result (t0
// where the number of stages is even).
template <int M, bool INV>
__device__ __forceinline__ float2* team_fft(float2* t0, float2* t1, const TeamTw<M>& w, int tid) {
  using T = Team<M>;
  __syncthreads();
  team_stage<M, T::R0, 1, INV>(t0, t1, nullptr, tid);
  team_stage<M, T::R1, T::R0, INV>(t1, t0, w.a, tid);
  team_stage<M, T::R2, T::R0 * T::R1, INV>(t0, t1, w.b, tid);
  if constexpr (T::S > 3) {
    team_stage<M, T::R3, T::R0 * T::R1 * T::R2, INV>(t1, t0, w.c, tid);
    return t0;
  }
  return t1;
}

// Psi' - Psi / M^2 of one mode: f (A / |f| - 1) nrm, parallel to f whatever the rounding of its factor;
// outside the range in which |f|^2 is safe in 32 bits (zero, infinities and NaN among it) the phase
// form of the projection decides.
__device__ __forceinline__ float2 modulus_delta(float2 f, float a, float nrm) {
  const float s = fmaxf(fabsf(f.x), fabsf(f.y));
  if (!(s > 1e-18f && s < 1e18f)) return csub(modulus_phase(f, a, nrm), cscale(f, nrm));
  return cscale(f, (a * rsqrtf(f.x * f.x + f.y * f.y) - 1.f) * nrm);
}

// MULTI: k_use modes, one after another in each step; the first k_res of them keep their spectra in
// LDS tiles of their own through the column step, the others in the exchange buffer, and all keep
// psi - psi_old in a.psi_old until the probe update.  Otherwise one mode, whose probe rows and
// psi - psi_old stay in registers.
template <int M, bool MULTI>
__global__ __launch_bounds__(TeamCfg<M>::NT) void k_epie_team(EpieArgs a) {
  using T = Team<M>;
  constexpr int W = T::W, NT = T::NT, R = T::R, P = T::P, PPT = T::PPT, MM = M * M, CR = R * R;
  constexpr bool ODD = T::S % 2 == 1;  // a transform ends in the other tile
  extern __shared__ float2 lds[];
  float2* const t0 = lds;
  float2* const t1 = lds + T::TILE;              // also stages the object window
  float2* const res = lds + T::TILE + T::TILE_B;  // k_res tiles
  __shared__ double redd[NT / 64];
  // max |O|^2 of the rows' segments that the ROI touches, and of the others; values sent with the three
  // barriers
  __shared__ unsigned cell[R * T::CELLS], rowm[R], value[3];
  __shared__ float most[3];               // largest values received with them
  __shared__ int gone;
  const int tid = threadIdx.x, w = blockIdx.x, lane = tid & 63;
  const int ku = MULTI ? a.k_use : 1;
  const int px0 = w * R * M;  // first frame pixel of this workgroup's rows
  const float nrm = 1.f / (float)MM;
  unsigned long long* const flags = a.team_flags;
  unsigned epoch = a.team_epoch;
  if (tid < 3) value[tid] = 0u;
  if (tid == 0) gone = 0;

  TeamTw<M> tw;
  tw.load(a.tw, tid);
  float obj_max = (float)a.scal[0];
  float probe_max = (float)a.scal[1];
  float2 pv[PPT];
#pragma unroll
  for (int j = 0; j < PPT; ++j) pv[j] = a.probe[px0 + tid + j * NT];
  // modes that take no part keep their intensities, which count in the probe maximum
  float rest = 0.f;
  if (a.update_probe && !a.modal)
    for (int k = ku; k < a.k_total; ++k)
#pragma unroll
      for (int j = 0; j < PPT; ++j) rest = fmaxf(rest, a.probe_int[(long)k * MM + px0 + tid + j * NT]);
  double err = 0.0;

  // The probe update needs max |O|^2 of the canvas after every position.  Of what the position does not
  // write, the maxima of 64-column segments and of rows are kept (k_canvas_maxima starts them), so that
  // only the pixels that share a segment with the ROI are read again: a position costs about the same on
  // every canvas (64^2, 400 positions: 9.2 us on 104 x 104, 10.0 on 200 x 8000, 10.1 on 4000 x 4000; with
  // the rows read to their ends 9.4, 30.4 and 31.5; on one workgroup that rescanned the canvas where it
  // had to 13.1, 13.2 and 19.6).
  const int nseg = epie_segments(a.obj_cols), brow = tid / T::TPR, bcol = tid % T::TPR;
  // [first pixel's segment, segments touched, pixels of those left of the ROI, and on both sides]
  struct Beside { int s0, n, left, both; };
  auto beside_of = [&](int ry) __attribute__((always_inline)) {
    Beside b;
    b.s0 = ry / PTYK_EPIE_SEG;
    b.n = (ry + M - 1) / PTYK_EPIE_SEG - b.s0 + 1;
    b.left = ry - b.s0 * PTYK_EPIE_SEG;
    b.both = b.left + min((b.s0 + b.n) * PTYK_EPIE_SEG, a.obj_cols) - (ry + M);
    return b;
  };

  // What a position needs as soon as the one before has left the object: the window behind the rows' ROI.
  float2 win[T::WU];
  auto load_object = [&](float2 pos) __attribute__((always_inline)) {
    const int ib = (int)floorf(pos.x) + w * R, jb = (int)floorf(pos.y);
#pragma unroll
    for (int u = 0; u < T::WU; ++u) {
      const int e = min(tid + u * NT, T::WIN - 1);
      const int r = min(max(ib + e / T::WC, 0), a.obj_rows - 1), c = min(max(jb + e % T::WC, 0), a.obj_cols - 1);
      win[u] = ld_dev(a.obj + (long)r * a.obj_cols + c);
    }
  };
  // amplitudes of the column step: PPT consecutive columns of one frame row, loaded a position ahead
  const int crow = tid / (R / PPT), ccol = tid % (R / PPT) * PPT;
  struct alignas(2 * PPT) Halves { __half h[PPT]; };
  auto load_amps = [&](int f) __attribute__((always_inline)) {
    return *reinterpret_cast<const Halves*>(a.amp + (long)f * MM + (long)crow * M + w * R + ccol);
  };
  int fi = a.order[0];
  float2 pos = a.pos[fi];
  load_object(pos);
  Halves ah = load_amps(fi);

  const int thread = tid;
  for (int s = 0; s < a.n_pos; ++s) {
    int tid = thread;
    // addresses made anew per position: kept for all of them they filled the registers of the 512^2 form
    // (256 and 42 spilled; now 217; three modes 40 -> 36 us a position)
    if (MULTI && M == 512) asm volatile("" : "+v"(tid));
    const float ascale = a.amp_scale[fi];
    const int rx = (int)roundf(pos.x), ry = (int)roundf(pos.y);
    const Beside bs = beside_of(ry);
    if (tid < R * T::CELLS) cell[tid] = 0u;
    if (tid < R) rowm[tid] = 0u;
    // ---- rows: ROI x P_k, row transform
#pragma unroll
    for (int u = 0; u < T::WU; ++u) {
      const int e = tid + u * NT;
      if (e < T::WIN) t1[e] = win[u];
    }
    __syncthreads();
    float2 roi[PPT], oo[PPT];  // bilinear ROI; object at the rounded position
    {
      const int ib = (int)floorf(pos.x), jb = (int)floorf(pos.y);
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int e = tid + j * NT, lr = e / M, c = e % M, row = w * R + lr;
        const float u = (float)c + pos.y + 0.5f, v = (float)row + pos.x + 0.5f;
        const TapPos q = a.tex_quantize ? tap_pos<true>(u, v) : tap_pos<false>(u, v);
        const int wr = min(max(q.j0 - ib - w * R, 0), R), wc = min(max(q.i0 - jb, 0), M);
        const float2* x = t1 + wr * T::WC + wc;
        roi[j] = bilinear_sum(q.al, q.be, x[0], x[1], x[T::WC], x[T::WC + 1]);
        oo[j] = t1[(lr + rx - ib) * T::WC + c + ry - jb];
      }
    }
    for (int k = 0; k < ku; ++k) {
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int e = tid + j * NT;
        t0[e / M * P + e % M] = cmul(pv[j], roi[j]);
      }
      if (MULTI) {  // the next mode's rows (the first one's again after the last)
        const float2* p = a.probe + (long)(k + 1 < ku ? k + 1 : 0) * MM + px0;
#pragma unroll
        for (int j = 0; j < PPT; ++j) pv[j] = p[tid + j * NT];
      }
      const float2* f = team_fft<M, false>(t0, t1, tw, tid);
      float2* x = a.psi + (long)k * MM;
#pragma unroll
      for (int j = 0; j < PPT; ++j) {  // blocks of R columns x R rows, one per owner of the columns
        const int e = tid + j * NT, v = e / CR, c = e / R % R, r = e % R;
        st_dev(x + (v * W + w) * CR + e % CR, f[r * P + v * R + c]);
      }
      if (MULTI) __syncthreads();
    }
    team_arrive(flags, w, ++epoch, value);
    // |O|^2 that this position does not write, for max |O|^2 after its update: the pixels beside the ROI
    // in this workgroup's rows, and (behind the barrier) the row's segments and a share of the rows apart
    // from the ROI, one load a thread to 1024 columns and rows at 64^2, the rest in rounds of four.  With
    // several modes all of it waits for the end of the column step: kept through the modes' transforms the
    // values cost registers there (128^2, three modes: 23.2 us a position; at the end 21.9).
    float beside[T::NB], segs = 0.f, rows = 0.f;
    auto load_beside = [&]() __attribute__((always_inline)) {
      const float* row = a.obj_int + (long)(rx + w * R + brow) * a.obj_cols;
#pragma unroll
      for (int u = 0; u < T::NB; ++u) {
        const int i = min(bcol + u * T::TPR, bs.both - 1);
        beside[u] = bs.both > 0 ? ld_dev(row + (i < bs.left ? bs.s0 * PTYK_EPIE_SEG + i : ry + M + i - bs.left)) : 0.f;
      }
    };
    auto load_apart = [&]() __attribute__((always_inline)) {
      const float* seg = a.team_segmax + (long)(rx + w * R + brow) * nseg;
      const int nrest = nseg - bs.n, nrow = a.obj_rows - M;
      auto seg_at = [&](int i) __attribute__((always_inline)) {
        i = min(i, nrest - 1);
        return ld_dev(seg + (i < bs.s0 ? i : i + bs.n));
      };
      auto row_at = [&](int i) __attribute__((always_inline)) {
        i = min(i, nrow - 1);
        return ld_dev(a.team_rowmax + (i < rx ? i : i + M));
      };
      const int r0 = w + W * lane;
      if (nrest > 0) segs = seg_at(bcol);
      if (nrow > 0) rows = row_at(r0);
      auto rounds = [&](int i, int step, int n, auto&& at) __attribute__((always_inline)) {
        float m = 0.f;
        for (; i < n; i += 4 * step) {
          const float v[4] = {at(i), at(i + step), at(i + 2 * step), at(i + 3 * step)};
          m = fmaxf(m, fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
        }
        return m;
      };
      if (nrest > T::TPR) segs = fmaxf(segs, rounds(bcol + T::TPR, T::TPR, nrest, seg_at));
      if (nrow > W * 64) rows = fmaxf(rows, rounds(r0 + W * 64, W * 64, nrow, row_at));
    };
    if (a.update_probe && !MULTI) load_beside();
    if (!team_wait<W>(flags, epoch, s ? a.team_limit : a.team_first, &gone, &most[0])) return;
    if (a.update_probe && s > 0) probe_max = most[0];

    // ---- columns
    float ms[PPT];
    float2 sm[PPT];
    if (MULTI) {
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        ms[j] = 0.f;
        sm[j] = make_float2(0.f, 0.f);
      }
    }
    float2* const xc = a.psi + (long)w * R * M;  // this workgroup's columns (mode 0)
    float2 g[PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j) g[j] = ld_dev(xc + tid + j * NT);
    if (a.update_probe && !MULTI) load_apart();
    for (int k = 0; k < ku; ++k) {
      float2* x = xc + (long)k * MM;
      // a resident mode's spectrum has to end in its own tile
      float2* const own = MULTI && k < a.k_res ? res + k * T::TILE : (ODD ? t1 : t0);
      float2* const in = ODD ? t0 : own;
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int e = tid + j * NT;
        in[e / R % R * P + e / CR * R + e % R] = g[j];
      }
      if (MULTI && k + 1 < ku) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) g[j] = ld_dev(x + MM + tid + j * NT);
      }
      float2* f = team_fft<M, false>(in, ODD ? own : t1, tw, tid);
      if (MULTI) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          const float2 v = f[(ccol + j) * P + crow];
          ms[j] += cabs2(v);
          sm[j] = cadd(sm[j], v);
          if (k >= a.k_res) st_dev(x + tid + j * NT, v);  // its own slots: only this thread reads them back
        }
        __syncthreads();
      } else {
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          float2* v = f + (ccol + j) * P + crow;
          const float A = __half2float(ah.h[j]) * ascale;
          if (a.rms) acc += fabs((double)A - sqrt((double)v->x * v->x + (double)v->y * v->y));
          *v = modulus_delta(*v, A, nrm);
        }
        if (a.rms) err += acc / (double)a.amp_sum[fi];
        f = team_fft<M, true>(f, f == t0 ? t1 : t0, tw, tid);
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          const int e = tid + j * NT;
          st_dev(x + e, f[e / R % R * P + e / CR * R + e % R]);
        }
      }
    }
    if (MULTI) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const float A = __half2float(ah.h[j]) * ascale;
        if (a.rms) acc += fabs((double)A - sqrt((double)sm[j].x * sm[j].x + (double)sm[j].y * sm[j].y));
        ms[j] = A * rsqrtf(ms[j]) * nrm - nrm;
      }
      if (a.rms) err += acc / ku / (double)a.amp_sum[fi];
      for (int k = 0; k < ku; ++k) {
        float2* x = xc + (long)k * MM;
        float2* const in = k < a.k_res ? res + k * T::TILE : t0;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          float2* v = in + (ccol + j) * P + crow;
          *v = cscale(k < a.k_res ? *v : ld_dev(x + tid + j * NT), ms[j]);
        }
        const float2* f = team_fft<M, true>(in, t1, tw, tid);
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          const int e = tid + j * NT;
          st_dev(x + e, f[e / R % R * P + e / CR * R + e % R]);
        }
        __syncthreads();
      }
    }
    if (a.update_probe && MULTI) {
      load_beside();
      load_apart();
    }
    team_arrive(flags, w, ++epoch, value + 1);
    const float co = (float)(1.0 / (double)probe_max);
    // next position
    const int fn = s + 1 < a.n_pos ? a.order[s + 1] : fi;
    const float2 posn = a.pos[fn];
    ah = load_amps(fn);
    if (a.update_probe) {
      float m = segs, ml = 0.f, mr = 0.f;
#pragma unroll
      for (int u = 0; u < T::NB; ++u) {
        const bool l = min(bcol + u * T::TPR, bs.both - 1) < bs.left;
        ml = fmaxf(ml, l ? beside[u] : 0.f);
        mr = fmaxf(mr, l ? 0.f : beside[u]);
      }
      // over 8 lanes, of one row
      m = max_dpp<0x141>(max_dpp<0x4E>(max_dpp<0xB1>(m)));
      ml = max_dpp<0x141>(max_dpp<0x4E>(max_dpp<0xB1>(ml)));
      mr = max_dpp<0x141>(max_dpp<0x4E>(max_dpp<0xB1>(mr)));
      if (tid % 8 == 0) {
        atomicMax(&rowm[brow], __float_as_uint(m));
        atomicMax(&cell[brow * T::CELLS], __float_as_uint(ml));
        atomicMax(&cell[brow * T::CELLS + bs.n - 1], __float_as_uint(mr));
      }
      const float o = wave_max_pos(fmaxf(fmaxf(rows, m), fmaxf(ml, mr)));
      if (lane == 0) atomicMax(&value[2], __float_as_uint(o));
    }
    if (!team_wait<W>(flags, epoch, a.team_limit, &gone, &most[1])) return;
    if (s == 0 && tid == 0) st_dev(a.scal + PTYK_EPIE_MARK, -(double)a.team_epoch);  // from here on the state changes

    // ---- rows: psi - psi_old, object update at the rounded position (d_updateObjectArray(M))
    float2 d[PPT], up[PPT];
    const float2* const xr = a.psi + w * CR;
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      const int e = tid + j * NT;
      g[j] = ld_dev(xr + e / CR * W * CR + e % CR);
    }
    for (int k = 0; k < ku; ++k) {
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int e = tid + j * NT;
        t0[e % R * P + e / CR * R + e / R % R] = g[j];
      }
      if (MULTI && k + 1 < ku) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          const int e = tid + j * NT;
          g[j] = ld_dev(xr + (long)(k + 1) * MM + e / CR * W * CR + e % CR);
        }
      }
      const float2* f = team_fft<M, true>(t0, t1, tw, tid);
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int e = tid + j * NT;
        d[j] = f[e / M * P + e % M];
        const float2 t = cconj(cmulcj(d[j], pv[j]));
        up[j] = MULTI && k ? cadd(up[j], t) : t;
        if (MULTI) {
          a.psi_old[(long)k * MM + px0 + e] = d[j];
          pv[j] = a.probe[(long)(k + 1 < ku ? k + 1 : 0) * MM + px0 + e];
        }
      }
      if (MULTI) __syncthreads();
    }
    float2 on[PPT];
    float imax = 0.f;
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      const int e = tid + j * NT, lr = e / M;
      const long oi = (long)(rx + w * R + lr) * a.obj_cols + (ry + e % M);
      float2 o = cadd(oo[j], cscale(up[j], co));
      const float mag = sqrtf(o.x * o.x + o.y * o.y);
      if (a.phase_constraint) o = clamp_phase(o);
      st_dev(a.obj + oi, o);
      st_dev(a.obj_int + oi, mag * mag);
      on[j] = o;
      if (a.update_probe) {  // a wave's 64 pixels lie in one row and in two of its segments
        const bool second = bs.left + lane >= PTYK_EPIE_SEG;
        const float q = fmaxf(mag * mag, 0.f);
        const float m0 = row16_max(second ? 0.f : q), m1 = row16_max(second ? q : 0.f);
        if (lane % 16 == 0) {
          unsigned* x = cell + lr * T::CELLS + e % M / 64;
          atomicMax(x, __float_as_uint(m0));
          atomicMax(x + 1, __float_as_uint(m1));
        }
        imax = fmaxf(imax, fmaxf(m0, m1));
      }
    }
    if (a.update_probe && lane % 16 == 0) atomicMax(&value[2], __float_as_uint(imax));
    team_arrive(flags, w, ++epoch, value + 2);
    // the rows' and their segments' maxima, for the others from the next barrier on
    if (a.update_probe) {
      if (tid < R * T::CELLS && tid % T::CELLS < bs.n)
        st_dev(a.team_segmax + (long)(rx + w * R + tid / T::CELLS) * nseg + bs.s0 + tid % T::CELLS,
               __uint_as_float(cell[tid]));
      if (tid < R) {
        unsigned m = rowm[tid];
#pragma unroll
        for (int c = 0; c < T::CELLS; ++c) m = max(m, cell[tid * T::CELLS + c]);
        st_dev(a.team_rowmax + rx + w * R + tid, __uint_as_float(m));
      }
    }
    if (!team_wait<W>(flags, epoch, a.team_limit, &gone, &most[2])) return;
    load_object(posn);

    // ---- probe update with the updated object (d_updateProbe(M)), own rows
    if (a.update_probe) {
      obj_max = most[2];
      if (tid == 0) value[0] = value[2] = 0u;  // both sent; set again after the barriers below
      const float cp = (float)(1.0 / (double)obj_max);
      float pm = rest, im[PPT];
      for (int k = 0; k < ku; ++k) {
        const long q = (long)k * MM + px0 + tid;
        // all loads before the stores, which the compiler takes to alias them (256^2, three modes: 26.5 us a
        // position with loads and stores by turns, 24.4 so)
        float2 dk[PPT], pk[PPT];
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          dk[j] = MULTI ? a.psi_old[q + j * NT] : d[j];
          pk[j] = MULTI ? a.probe[q + j * NT] : pv[j];
        }
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
          const float2 p = cadd(cscale(cmulcj(on[j], dk[j]), cp), pk[j]);
          if (MULTI) a.probe[q + j * NT] = p;
          if (!MULTI || k == 0) pv[j] = p;
          const float ia = sqrtf(p.x * p.x + p.y * p.y);
          im[j] = MULTI && k ? im[j] + ia * ia : ia * ia;
        }
      }
#pragma unroll
      for (int j = 0; j < PPT; ++j) pm = fmaxf(pm, im[j]);
      pm = wave_max_pos(pm);
      __syncthreads();  // value[0] is cleared
      if (lane == 0) atomicMax(&value[0], __float_as_uint(pm));
    }
    fi = fn;
    pos = posn;
  }

  // ---- state: probe, its intensities, maxima, error
  if (a.update_probe) {
    for (int k = 0; k < ku; ++k)
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const long q = (long)k * MM + px0 + tid + j * NT;
        const float2 p = MULTI ? a.probe[q] : pv[j];
        if (!MULTI) a.probe[q] = p;
        const float ia = sqrtf(p.x * p.x + p.y * p.y);
        a.probe_int[q] = ia * ia;
      }
  } else {
    // 8 loads of two values in flight (64^2, 36 positions on 4000 x 4000: 0.78 ms an iteration; one load of
    // one value at a time 4.1, and one workgroup 1.7)
    const long canvas = (long)a.obj_rows * a.obj_cols, pairs = canvas / 2, step = (long)W * NT;
    const float2* const o2 = reinterpret_cast<const float2*>(a.obj_int);
    float m = canvas % 2 ? ld_dev(a.obj_int + canvas - 1) : 0.f;
    for (long q0 = (long)w * NT + tid; q0 < pairs; q0 += 8 * step) {
      float2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = ld_dev(o2 + min(q0 + u * step, pairs - 1));
#pragma unroll
      for (int u = 0; u < 8; ++u) m = fmaxf(m, fmaxf(v[u].x, v[u].y));
    }
    m = fmaxf(m, 0.f);
    m = wave_max_pos(m);
    if (lane == 0) atomicMax(&value[0], __float_as_uint(m));
  }
  err = block_sum<NT>(err, redd);
  if (tid == 0) st_dev(a.team_err + w, err);
  team_arrive(flags, w, ++epoch, value);
  if (w != 0) return;
  if (!team_wait<W>(flags, epoch, a.team_limit, &gone, &most[0])) return;
  if (tid == 0) {
    double e = 0.0;
    for (int i = 0; i < W; ++i) e += __hip_atomic_load(a.team_err + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    a.scal[0] = a.update_probe ? obj_max : most[0];
    a.scal[1] = a.update_probe ? most[0] : probe_max;
    a.scal[2] = e;
    st_dev(a.scal + PTYK_EPIE_MARK, (double)a.team_epoch);  // the whole chain ran
  }
}

template <int M>
static hipError_t epie_impl(const EpieArgs& a, hipStream_t s) {
  const size_t lds = (size_t)WgFft<M, PTYK_EPIE_NT>::LDS * sizeof(float2);
  hipError_t e = hipFuncSetAttribute((const void*)k_epie<M>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_epie<M>), dim3(1), dim3(PTYK_EPIE_NT), lds, s, a);
  return hipGetLastError();
}

template <int M>
struct TeamLds {
  using T = Team<M>;
  static constexpr size_t base = (size_t)(T::TILE + T::TILE_B) * sizeof(float2), tile = (size_t)T::TILE * sizeof(float2);
  static constexpr int room = (int)((128 * 1024 - base) / tile);  // modes; of the CU's 160 KiB, beside the static arrays
  static int resident(int k_use, int most) {
    return k_use > 1 ? std::min({k_use, room, most > 0 ? most : room}) : 0;
  }
};
template <int M, bool MULTI>
static hipError_t epie_team_launch(EpieArgs a, hipStream_t s) {
  using T = Team<M>;
  a.k_res = TeamLds<M>::resident(a.k_use, a.k_res);
  const size_t lds = TeamLds<M>::base + a.k_res * TeamLds<M>::tile;
  hipError_t e = hipFuncSetAttribute((const void*)k_epie_team<M, MULTI>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds);
  if (e != hipSuccess) return e;
  if (a.update_probe)
    hipLaunchKernelGGL(k_canvas_maxima, dim3((unsigned)((a.obj_rows + 3) / 4)), dim3(256), 0, s, a.obj_int, a.obj_rows,
                       a.obj_cols, a.team_segmax, a.team_rowmax);
  // with no wait at all, one workgroup stays out: the others find it missing and end (what becomes of a
  // team that does not come together, for tests)
  hipLaunchKernelGGL((k_epie_team<M, MULTI>), dim3(a.team_first ? T::W : T::W - 1), dim3(T::NT), lds, s, a);
  return hipGetLastError();
}
template <int M>
static hipError_t epie_team_impl(const EpieArgs& a, hipStream_t s) {
  if (a.team_size == 0) return epie_impl<M>(a, s);
  return a.k_use > 1 ? epie_team_launch<M, true>(a, s) : epie_team_launch<M, false>(a, s);
}

// 0 where one workgroup takes the frame: below 64^2, and where the device (a partition of the part)
// has fewer CUs than the team has workgroups.
int epie_team_size(int m, int cus) {
  const int w = m == 64 ? Team<64>::W : m == 128 ? Team<128>::W : m == 256 ? Team<256>::W : m == 512 ? Team<512>::W : 0;
  return w <= cus ? w : 0;
}
int epie_team_resident(int m, int k_use, int most) {
  switch (m) {
    case 64: return TeamLds<64>::resident(k_use, most);
    case 128: return TeamLds<128>::resident(k_use, most);
    case 256: return TeamLds<256>::resident(k_use, most);
    case 512: return TeamLds<512>::resident(k_use, most);
    default: return 0;
  }
}
unsigned epie_team_barriers(int n_pos) { return 3u * (unsigned)n_pos + 1u; }

hipError_t epie_iteration(const EpieArgs& a, hipStream_t s) {
  switch (a.m) {
    case 16: return epie_impl<16>(a, s);
    case 32: return epie_impl<32>(a, s);
    case 64: return epie_team_impl<64>(a, s);
    case 128: return epie_team_impl<128>(a, s);
    case 256: return epie_team_impl<256>(a, s);
    case 512: return epie_team_impl<512>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ptyk
