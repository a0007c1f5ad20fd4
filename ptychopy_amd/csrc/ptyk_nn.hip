// Learned warm start: a four-level convolutional encoder-decoder (U-Net form, channel widths
// c, 2c, 4c, 8c with c = 32 by default) mapping a log-scaled diffraction amplitude (1 x S x S)
// to the object patch's amplitude and phase (2 x S x S).  No reference counterpart.
//
// Tensors are pixel-major (NHWC) with the channels padded to a multiple of 8 by zeros, so that the
// 8 channels a lane feeds to a matrix instruction are 16 contiguous bytes; the products run over chunks
// of 32 channels, of which those past a tensor's last are zeros in LDS and never stored (a network of 8
// channels would else hold twice its tensors' bytes).  Every 3 x 3 convolution
// between them is an implicit GEMM on v_mfma_f32_32x32x16_bf16 (BF16 operands, FP32 accumulation;
// no im2col buffer): k_conv3 for the forward pass and the data gradient, k_wgrad3 for the weight
// gradient (split over pixels into partial tiles summed in a fixed order).  The first layer (one
// input channel) and the last (1 x 1 to two channels) are bound by memory and run on the vector
// units.  Activations are BF16, gradients FP32 (rounded to BF16 where they enter a product), master
// weights FP32 with Adam.  Skip concatenations and nearest upsampling are never stored: a layer's
// input is up to two tensors, one of which may be read at half resolution.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/ptyk.h"
#include "ptyk_device.h"
#include "ptyk_draw.h"
#include "ptyk_internal.h"

namespace ptyk {

typedef __bf16 bf16;
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

namespace {

constexpr int CT = 256;      // threads of the convolution kernels (4 waves)
constexpr int NN_LAYERS = 15;
inline int pad32(int c) { return (c + 31) / 32 * 32; }
inline int pad8(int c) { return (c + 7) / 8 * 8; }

__device__ __forceinline__ bf16 to_bf(float v) { return (bf16)v; }
__device__ __forceinline__ unsigned bf_bits(float v) { return __builtin_bit_cast(u16, to_bf(v)); }
__device__ __forceinline__ float bf_val(unsigned bits16) { return __uint_as_float(bits16 << 16); }
__device__ __forceinline__ unsigned bf_pair(float a, float b) { return bf_bits(a) | (bf_bits(b) << 16); }

// A layer's input: p0's channels, then p1's, both NHWC with cp0 and cp1 stored channels, each in chunks
// of 32; up0: p0 has half the resolution (nearest upsampling).
struct Src {
  const void* p0;
  const void* p1;
  int cp0, cp1, up0;
};

// The tensor behind chunk ch: its stored channels, the chunk's first among them, and whether it is upsampled.
__device__ __forceinline__ const void* src_base(const Src& s, int ch, int* cp, int* coff, int* up) {
  const bool first = ch * 32 < s.cp0;
  *cp = first ? s.cp0 : s.cp1;
  *coff = (first ? ch : ch - (s.cp0 + 31) / 32) * 32;
  *up = first ? s.up0 : 0;
  return first ? s.p0 : s.p1;
}

// Where a tile of 32 output channels goes (cp of them in all are stored).  Forward: bias, ReLU, BF16.  Data gradient: FP32, zeroed
// where the BF16 activation mask is not positive (the ReLU of the layer that made it; NULL: no ReLU);
// sum4: the 2 x 2 sums go to a half-resolution tensor (the gradient of the upsampling).
struct Dst {
  void* p;
  const bf16* mask;
  int cp, sum4;
};

struct ConvArgs {
  Src in;               // forward: BF16; data gradient: FP32
  const bf16* w;        // fragments: [output tile of 32][input chunk of 32][tap][2][lane][8]
  const float* bias;    // forward: cout values
  Dst out0, out1;       // output tiles below out0_tiles, and the others
  int out0_tiles, cout; // cout: real output channels (forward)
  int batch, h, w_px, chunks, tiles_x, tiles_y, groups, relu;
};

// 3 x 3 convolution, zero edges.  A workgroup makes a tile of 4 ROWS x 32 pixels of NCO x 32 output
// channels; wave v its rows v ROWS .. v ROWS + ROWS - 1.  Per chunk of 32 input channels, the tile
// with its one-pixel border and the chunk's weights go to LDS once and serve all nine taps.  The
// matrix instruction takes weights as its rows and 32 pixels of an image row as its columns, so a
// lane ends with groups of 4 adjacent channels of one pixel.  For one horizontal shift the ROWS + 2
// pixel operands of a wave serve its three vertical shifts from registers: (ROWS + 2 + 3 NCO) LDS
// reads of 16 bytes a lane for 3 ROWS NCO instructions, which keeps the LDS (128 B a clock) below
// the matrix cores' time.  Pixels are 64 bytes apart in LDS; the 16-byte quarter q of column c is
// stored at q ^ ((c >> 1) & 3), so that 8 adjacent lanes' reads spread over all banks.
// GRAD: the data gradient (input FP32, rounded to BF16 on the way to LDS; weights with their taps
// reversed and their channels exchanged).
// AHEAD: the next chunk's loads are in flight during a chunk's products (as long as the registers for
// them are there).
// PART: some tensor's channels do not fill its last chunk (the tests for it cost 4 % of a training step of
// 32 channels, where all do).
template <int NCO, int ROWS, bool GRAD, bool PART>
__global__ __launch_bounds__(CT, 2) void k_conv3(ConvArgs a) {
  constexpr bool AHEAD = NCO * ROWS <= 4;
  constexpr int TR = 4 * ROWS + 2, TC = 34, XN = TR * TC * 4, WF = 9 * 2 * 64, WN = NCO * WF;  // 16-byte pieces
  extern __shared__ u32x4 conv_lds[];
  u32x4* const xs = conv_lds;
  u32x4* const ws = conv_lds + XN;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // blocks go round the 8 XCDs: the output groups of one pixel tile follow each other on one XCD,
  // whose L2 then holds the tile's input
  const int bid = blockIdx.x, tile = (bid / 8 / a.groups) * 8 + bid % 8, grp = bid / 8 % a.groups;
  if (tile >= a.batch * a.tiles_x * a.tiles_y) return;
  const int tx = tile % a.tiles_x, ty = tile / a.tiles_x % a.tiles_y, b = tile / (a.tiles_x * a.tiles_y);
  const int x0 = tx * 32, y0 = ty * 4 * ROWS;
  v16f acc[NCO][ROWS];
#pragma unroll
  for (int t = 0; t < NCO; ++t)
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][r][i] = 0.f;
  constexpr int XU = (XN + CT - 1) / CT, WU = (WN + CT - 1) / CT;
  const u32x4* const w0 = reinterpret_cast<const u32x4*>(a.w) + (long)grp * NCO * a.chunks * WF;
  u32x4 xv[AHEAD ? XU : 1], wr[AHEAD ? WU : 1];
  f32x4 gv[AHEAD && GRAD ? XU : 1][2];
  // one 16-byte piece of a chunk's input tile: FP32 rounded to BF16 for GRAD
  auto pack = [](f32x4 u, f32x4 w) __attribute__((always_inline)) {
    return u32x4{bf_pair(u[0], u[1]), bf_pair(u[2], u[3]), bf_pair(w[0], w[1]), bf_pair(w[2], w[3])};
  };
#define PTYK_CONV_PIECE(i)                                                                              \
  const int e = tid + (i)*CT, q = e & 3, pc = e >> 2, r = pc / TC, c = pc - r * TC;                     \
  const int y = y0 + r - 1, x = x0 + c - 1;                                                             \
  const bool in = e < XN && y >= 0 && y < rows && x >= 0 && x < a.w_px;                                  \
  const long off = in ? (img + (y >> up) * sw + (x >> up)) * cp + coff + q * 8 : 0
#define PTYK_CONV_CHUNK(ch)                                                                             \
  int cp, coff, up;                                                                                     \
  const void* const base = src_base(a.in, ch, &cp, &coff, &up);                                         \
  const int rows = !PART || coff + (tid & 3) * 8 < cp ? a.h : 0; /* of this thread's channels, if any */ \
  const int sw = a.w_px >> up;                                                                          \
  const long img = (long)b * (a.h >> up) * sw
#define PTYK_CONV_LOAD(ch)                                                                              \
  {                                                                                                     \
    PTYK_CONV_CHUNK(ch);                                                                                \
    _Pragma("unroll") for (int i = 0; i < XU; ++i) {                                                    \
      PTYK_CONV_PIECE(i);                                                                               \
      if constexpr (GRAD) {                                                                             \
        const f32x4* g = reinterpret_cast<const f32x4*>((const float*)base + off);                      \
        gv[i][0] = in ? g[0] : f32x4{0.f, 0.f, 0.f, 0.f};                                               \
        gv[i][1] = in ? g[1] : f32x4{0.f, 0.f, 0.f, 0.f};                                               \
      } else {                                                                                          \
        xv[i] = in ? *reinterpret_cast<const u32x4*>((const bf16*)base + off) : u32x4{0u, 0u, 0u, 0u};  \
      }                                                                                                 \
    }                                                                                                   \
    _Pragma("unroll") for (int i = 0; i < WU; ++i) {                                                    \
      const int e = min(tid + i * CT, WN - 1);                                                          \
      wr[i] = w0[((long)(e / WF) * a.chunks + (ch)) * WF + e % WF];                                     \
    }                                                                                                   \
  }
  if constexpr (AHEAD) PTYK_CONV_LOAD(0)
  for (int ch = 0; ch < a.chunks; ++ch) {
    if (ch) __syncthreads();
    if constexpr (AHEAD) {
#pragma unroll
      for (int i = 0; i < XU; ++i) {
        const int e = tid + i * CT, q = e & 3, pc = e >> 2, c = pc % TC;
        if (e < XN) xs[pc * 4 + (q ^ ((c >> 1) & 3))] = GRAD ? pack(gv[GRAD ? i : 0][0], gv[GRAD ? i : 0][1]) : xv[i];
      }
#pragma unroll
      for (int i = 0; i < WU; ++i)
        if (tid + i * CT < WN) ws[tid + i * CT] = wr[i];
    } else {
      PTYK_CONV_CHUNK(ch);
#pragma unroll
      for (int i = 0; i < XU; ++i) {
        PTYK_CONV_PIECE(i);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (in) {
          if constexpr (GRAD) {
            const f32x4* g = reinterpret_cast<const f32x4*>((const float*)base + off);
            v = pack(g[0], g[1]);
          } else {
            v = *reinterpret_cast<const u32x4*>((const bf16*)base + off);
          }
        }
        if (e < XN) xs[pc * 4 + (q ^ ((c >> 1) & 3))] = v;
      }
#pragma unroll
      for (int t = 0; t < NCO; ++t)
        for (int i = tid; i < WF; i += CT) ws[t * WF + i] = w0[((long)t * a.chunks + ch) * WF + i];
    }
    __syncthreads();
    if constexpr (AHEAD)
      if (ch + 1 < a.chunks) PTYK_CONV_LOAD(ch + 1)
#pragma unroll
    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int c = (lane & 31) + dx, q = ks * 2 + (lane >> 5), qs = q ^ ((c >> 1) & 3);
        v8bf x[ROWS + 2];
#pragma unroll
        for (int r = 0; r < ROWS + 2; ++r)
          x[r] = __builtin_bit_cast(v8bf, xs[((wv * ROWS + r) * TC + c) * 4 + qs]);
#pragma unroll
        for (int t = 0; t < NCO; ++t)
#pragma unroll
          for (int dy = 0; dy < 3; ++dy) {
            const v8bf w = __builtin_bit_cast(v8bf, ws[((t * 9 + dy * 3 + dx) * 2 + ks) * 64 + lane]);
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
              acc[t][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x[r + dy], acc[t][r], 0, 0, 0);
          }
      }
  }
  // lane holds pixel x0 + lane % 32, channels 8 g + 4 (lane / 32) + 0..3 in registers 4 g + 0..3
  const int x = x0 + (lane & 31), half = lane >> 5;
#pragma unroll
  for (int t = 0; t < NCO; ++t) {
    const int ot = grp * NCO + t;
    const Dst d = ot < a.out0_tiles ? a.out0 : a.out1;
    const int c0 = (ot < a.out0_tiles ? ot : ot - a.out0_tiles) * 32;
    bool kept[4];  // groups of 8 channels
#pragma unroll
    for (int g = 0; g < 4; ++g) kept[g] = !PART || c0 + 8 * g < d.cp;
    if (!GRAD) {
      float bias[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int co = ot * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
        bias[i] = co < a.cout ? a.bias[co] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int y = y0 + wv * ROWS + r;
        if (y >= a.h || x >= a.w_px) continue;
        bf16* o = (bf16*)d.p + (((long)b * a.h + y) * a.w_px + x) * d.cp + c0 + 4 * half;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] = acc[t][r][4 * g + i] + bias[4 * g + i];
            if (a.relu) v[i] = fmaxf(v[i], 0.f);
          }
          if (kept[g]) *reinterpret_cast<uint2*>(o + 8 * g) = make_uint2(bf_pair(v[0], v[1]), bf_pair(v[2], v[3]));
        }
      }
    } else if (d.sum4) {  // image sizes are even here: whole 2 x 2 blocks, rows in pairs, columns in lane pairs
      if (ROWS % 2 == 0) {
#pragma unroll
        for (int r = 0; r + 1 < ROWS; r += 2) {
          const int y = y0 + wv * ROWS + r;
          const long px = ((long)b * (a.h >> 1) + (y >> 1)) * (a.w_px >> 1) + (x >> 1);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float s = acc[t][r][4 * g + i], u = acc[t][r + 1][4 * g + i];
              const float sx = __shfl_xor(s, 1, 64), ux = __shfl_xor(u, 1, 64);
              v[i] = s + sx + u + ux;
            }
            if (y < a.h && x < a.w_px && !(lane & 1) && kept[g]) {
              const long o = px * d.cp + c0 + 8 * g + 4 * half;
              const uint2 m = *reinterpret_cast<const uint2*>(d.mask + o);
              const unsigned mm[4] = {m.x & 0xffffu, m.x >> 16, m.y & 0xffffu, m.y >> 16};
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (!(bf_val(mm[i]) > 0.f)) v[i] = 0.f;
              *reinterpret_cast<float4*>((float*)d.p + o) = make_float4(v[0], v[1], v[2], v[3]);
            }
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int y = y0 + wv * ROWS + r;
        if (y >= a.h || x >= a.w_px) continue;
        const long o0 = (((long)b * a.h + y) * a.w_px + x) * d.cp + c0 + 4 * half;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (!kept[g]) continue;
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = acc[t][r][4 * g + i];
          if (d.mask) {
            const uint2 m = *reinterpret_cast<const uint2*>(d.mask + o0 + 8 * g);
            const unsigned mm[4] = {m.x & 0xffffu, m.x >> 16, m.y & 0xffffu, m.y >> 16};
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (!(bf_val(mm[i]) > 0.f)) v[i] = 0.f;
          }
          *reinterpret_cast<float4*>((float*)d.p + o0 + 8 * g) = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    }
  }
}

#undef PTYK_CONV_LOAD
#undef PTYK_CONV_PIECE
#undef PTYK_CONV_CHUNK

struct WgradArgs {
  Src x;              // BF16 input of the layer
  const float* dz;    // FP32 gradient of its pre-activation output, NHWC with cz channels
  float* part;        // [chunk][output tile][input tile][tap][32][32] (output, input channel)
  double* bpart;      // [chunk][cpo]: bias gradient
  int batch, h, w_px, cz, cpo, tiles_o, tiles_i, tiles_x, tiles_y, chunks;
};

// Weight gradient: D[co][ci] per tap = sum over pixels of dZ[p][co] x[p + tap][ci], a GEMM whose
// contraction runs over pixels.  A workgroup owns one 32 x 32 channel tile of all nine taps and a
// share of the 8 x 32-pixel tiles; its four waves take two rows each and add up at the end.  The
// matrix instruction wants 8 adjacent pixels of one channel per lane, so tiles are transposed on
// their way to LDS ([channel][pixel]); x is kept three times, shifted by -1, 0 and 1 pixels, so that
// every operand is one aligned 16-byte read.  Per wave and 16 pixels: 2 + 12 reads for 18
// instructions.  Channel pitches of 528 and 656 bytes spread 8 lanes over the banks.
constexpr int WG_R = 8, WG_ZP = WG_R * 64 + 16, WG_XP = (WG_R + 2) * 64 + 16;  // bytes per channel
template <bool PART>  // as for k_conv3
__global__ __launch_bounds__(CT, 2) void k_wgrad3(WgradArgs a) {
  extern __shared__ __align__(16) unsigned char wg_lds[];
  unsigned char* const zs = wg_lds;                // 32 x WG_ZP
  unsigned char* const xs = wg_lds + 32 * WG_ZP;   // 3 x 32 x WG_XP
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int pairs = a.tiles_o * a.tiles_i, pr = blockIdx.x % pairs, chunk = blockIdx.x / pairs;
  const int ot = pr / a.tiles_i, it = pr % a.tiles_i;
  int cp, coff, up;
  const void* base = src_base(a.x, it, &cp, &coff, &up);
  const int sw = a.w_px >> up, sh = a.h >> up;
  const int cpair = tid & 15, slot = tid >> 4;  // 2 channels, one of 16 pixel groups of 8
  // rows of this thread's channels: none where they are not stored
  const int zh = !PART || ot * 32 + cpair * 2 < a.cz ? a.h : 0, xh = !PART || coff + cpair * 2 < cp ? a.h : 0;
  v16f acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  double bs0 = 0.0, bs1 = 0.0;
  const int tiles = a.batch * a.tiles_x * a.tiles_y;
  const int lo = (int)((long)tiles * chunk / a.chunks), hi = (int)((long)tiles * (chunk + 1) / a.chunks);
  for (int tile = lo; tile < hi; ++tile) {
    const int tx = tile % a.tiles_x, ty = tile / a.tiles_x % a.tiles_y, b = tile / (a.tiles_x * a.tiles_y);
    const int x0 = tx * 32, y0 = ty * WG_R;
    if (tile != lo) __syncthreads();
    // dZ: 8 rows x 4 groups of 8 pixels x 16 channel pairs
#pragma unroll
    for (int i = 0; i < WG_R * 4 / 16; ++i) {
      const int g = slot + i * 16, r = g >> 2, xg = (g & 3) * 8, y = y0 + r;
      float2 v[8];
      const int left = y < zh ? a.w_px - (x0 + xg) : 0;  // pixels from here to the row's end
      const float* zp = a.dz + (((long)b * a.h + min(y, a.h - 1)) * a.w_px + x0 + xg) * a.cz + ot * 32 + cpair * 2;
#pragma unroll
      for (int p = 0; p < 8; ++p)
        v[p] = p < left ? *reinterpret_cast<const float2*>(zp + p * a.cz) : make_float2(0.f, 0.f);
      if (it == 0) {
#pragma unroll
        for (int p = 0; p < 8; ++p) {
          bs0 += v[p].x;
          bs1 += v[p].y;
        }
      }
      unsigned char* z = zs + (cpair * 2) * WG_ZP + r * 64 + xg * 2;
      *reinterpret_cast<uint4*>(z) = make_uint4(bf_pair(v[0].x, v[1].x), bf_pair(v[2].x, v[3].x),
                                                bf_pair(v[4].x, v[5].x), bf_pair(v[6].x, v[7].x));
      *reinterpret_cast<uint4*>(z + WG_ZP) = make_uint4(bf_pair(v[0].y, v[1].y), bf_pair(v[2].y, v[3].y),
                                                        bf_pair(v[4].y, v[5].y), bf_pair(v[6].y, v[7].y));
    }
    // x: 10 rows, each group with its neighbours on both sides
#pragma unroll
    for (int i = 0; i < ((WG_R + 2) * 4 + 15) / 16; ++i) {
      const int g = slot + i * 16, r = g >> 2, xg = (g & 3) * 8, y = y0 + r - 1;
      if (g >= (WG_R + 2) * 4) break;
      unsigned v[10];  // two channels of pixels xg - 1 .. xg + 8
      const int left = y >= 0 && y < xh ? a.w_px - (x0 + xg - 1) : 0;
      const bf16* xp = (const bf16*)base + ((long)b * sh + (max(y, 0) >> up)) * sw * cp + coff + cpair * 2;
#pragma unroll
      for (int p = 0; p < 10; ++p)
        v[p] = p < left && (p > 0 || x0 + xg > 0)
                   ? *reinterpret_cast<const unsigned*>(xp + ((x0 + xg + p - 1) >> up) * cp)
                   : 0u;
      unsigned char* d = xs + (cpair * 2) * WG_XP + r * 64 + xg * 2;
#pragma unroll
      for (int s = 0; s < 3; ++s) {  // copy s holds x[p + s - 1]
        unsigned lo4[4], hi4[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          lo4[k] = (v[s + 2 * k] & 0xffffu) | (v[s + 2 * k + 1] << 16);
          hi4[k] = (v[s + 2 * k] >> 16) | (v[s + 2 * k + 1] & 0xffff0000u);
        }
        *reinterpret_cast<uint4*>(d + s * 32 * WG_XP) = make_uint4(lo4[0], lo4[1], lo4[2], lo4[3]);
        *reinterpret_cast<uint4*>(d + s * 32 * WG_XP + WG_XP) = make_uint4(hi4[0], hi4[1], hi4[2], hi4[3]);
      }
    }
    __syncthreads();
    const int ch = lane & 31, half = lane >> 5;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int po = ks * 32 + half * 16;  // bytes: 8 pixels
      v8bf z[2];
#pragma unroll
      for (int r = 0; r < 2; ++r)
        z[r] = *reinterpret_cast<const v8bf*>(zs + ch * WG_ZP + (wv * 2 + r) * 64 + po);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        v8bf x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          x[r] = *reinterpret_cast<const v8bf*>(xs + (s * 32 + ch) * WG_XP + (wv * 2 + r) * 64 + po);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            acc[dy * 3 + s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(z[r], x[r + dy], acc[dy * 3 + s], 0, 0, 0);
      }
    }
  }
  // waves add up through LDS, 3 taps at a time, in wave order; wave 0 writes
  float* red = reinterpret_cast<float*>(wg_lds);  // 3 waves x 3 taps x 1024 floats
  float* out = a.part + ((long)chunk * pairs + pr) * (9 * 1024);
#pragma unroll
  for (int t3 = 0; t3 < 3; ++t3) {
    __syncthreads();
    if (wv > 0)
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) red[(((wv - 1) * 3 + t) * 16 + i) * 64 + lane] = acc[t3 * 3 + t][i];
    __syncthreads();
    if (wv == 0)
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float s = acc[t3 * 3 + t][i];
#pragma unroll
          for (int u = 0; u < 3; ++u) s += red[((u * 3 + t) * 16 + i) * 64 + lane];
          out[(t3 * 3 + t) * 1024 + (8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * 32 + (lane & 31)] = s;
        }
  }
  if (it == 0) {  // bias: 16 pixel slots per channel pair
    double* rb = reinterpret_cast<double*>(wg_lds);
    __syncthreads();
    rb[tid * 2] = bs0;
    rb[tid * 2 + 1] = bs1;
    __syncthreads();
    if (tid < 32) {
      double s = 0.0;
      for (int k = 0; k < 16; ++k) s += rb[(k * 16 + (tid >> 1)) * 2 + (tid & 1)];
      a.bpart[(long)chunk * a.cpo + ot * 32 + tid] = s;
    }
  }
}

// Position of an input channel among the padded channels of a layer's (up to) two input tensors.
struct LayerMap {
  long woff, boff, foff, goff;  // parameters; forward and data-gradient fragments
  int cin, cout, ks, c0;        // c0: real channels of the first input tensor (cin when there is one)
  int cp0, cpi, cpo;            // in chunks of 32: first input tensor, all inputs, outputs
};
struct LayerTable {
  LayerMap l[NN_LAYERS];
};
__device__ __forceinline__ int pad_channel(const LayerMap& m, int ci) { return ci < m.c0 ? ci : m.cp0 + (ci - m.c0); }

// Chunk sums (fixed order) of the weight and bias gradients, scattered to the parameter order.  A
// block makes 32 values (adjacent input channels of one partial tile's row: 128-byte reads), its 8
// lanes of 32 threads taking every eighth chunk; the biases follow behind the weights' blocks.
__global__ __launch_bounds__(256) void k_wgrad_sum(LayerMap m, const float* __restrict__ part,
                                                   const double* __restrict__ bpart, int chunks, float* __restrict__ g) {
  __shared__ double red[8][32];
  const int k = threadIdx.x & 31, ln = threadIdx.x >> 5;
  const int rows = m.cpo / 32 * (m.cpi / 32) * 9 * 32;  // partial tiles' rows: (pair, tap, output channel)
  const bool weight = (int)blockIdx.x < rows;
  double s = 0.0;
  if (weight) {
    const float* p = part + (long)blockIdx.x * 32 + k;
    const long stride = (long)rows * 32;
    float f = 0.f;
    for (int c = ln; c < chunks; c += 8) f += p[c * stride];
    s = f;
  } else {
    const int co = (blockIdx.x - rows) * 32 + k;
    for (int c = ln; c < chunks; c += 8) s += bpart[(long)c * m.cpo + co];
  }
  red[ln][k] = s;
  __syncthreads();
  if (ln) return;
  s = red[0][k];
#pragma unroll
  for (int i = 1; i < 8; ++i) s += red[i][k];
  if (!weight) {
    const int co = (blockIdx.x - rows) * 32 + k;
    if (co < m.cout) g[m.boff + co] = (float)s;
    return;
  }
  const int pair = blockIdx.x / (9 * 32), tap = blockIdx.x / 32 % 9;
  const int co = pair / (m.cpi / 32) * 32 + blockIdx.x % 32, cc = pair % (m.cpi / 32) * 32 + k;
  const int ci = cc < m.cp0 ? cc : m.c0 + (cc - m.cp0);  // the channel behind a padded position
  if (co < m.cout && (cc < m.cp0 ? cc < m.c0 : ci < m.cin)) g[m.woff + ((long)co * m.cin + ci) * 9 + tap] = (float)s;
}

// The BF16 copies of parameter i: plain (first and last layer), and its places among the forward and
// data-gradient fragments ([output tile][input chunk][tap][2][lane][8]).
__device__ __forceinline__ void store_weight(const LayerTable& tb, long i, float v, bf16* __restrict__ wb,
                                             bf16* __restrict__ wf, bf16* __restrict__ wg) {
  const bf16 h = to_bf(v);
  wb[i] = h;
  int l = 0;
  while (l + 1 < NN_LAYERS && i >= tb.l[l + 1].woff) ++l;
  const LayerMap& m = tb.l[l];
  if (i >= m.boff || m.ks != 3 || l == 0) return;
  const int k = (int)(i - m.woff), t = k % 9, ci = pad_channel(m, k / 9 % m.cin), co = k / (9 * m.cin);
  auto frag = [](int o, int chunks, int c, int tap) {
    return ((((long)(o >> 5) * chunks + (c >> 5)) * 9 + tap) * 2 + (c >> 4 & 1)) * 512 + ((o & 31) + 32 * (c >> 3 & 1)) * 8 +
           (c & 7);
  };
  wf[m.foff + frag(co, m.cpi / 32, ci, t)] = h;
  wg[m.goff + frag(ci, m.cpo / 32, co, 8 - t)] = h;
}

__global__ void k_pack(LayerTable tb, const float* __restrict__ w, long n, bf16* __restrict__ wb, bf16* __restrict__ wf,
                       bf16* __restrict__ wg) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) store_weight(tb, i, w[i], wb, wf, wg);
}

// Adam on FP32 master weights; refreshes the BF16 copies
__global__ void k_adam(LayerTable tb, float* __restrict__ w, float* __restrict__ mo, float* __restrict__ ve,
                       const float* __restrict__ g, bf16* __restrict__ wb, bf16* __restrict__ wf, bf16* __restrict__ wg,
                       long n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float m = b1 * mo[i] + (1.f - b1) * gi;
  const float v = b2 * ve[i] + (1.f - b2) * gi * gi;
  mo[i] = m;
  ve[i] = v;
  const float wn = w[i] - lr * (m / c1) / (sqrtf(v / c2) + eps);
  w[i] = wn;
  store_weight(tb, i, wn, wb, wf, wg);
}

// First layer: one input channel, 3 x 3, ReLU.  A thread keeps the weights of 8 channels and makes
// them for one pixel after another (bound by the output's bytes).
__global__ __launch_bounds__(256) void k_first_fwd(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                   const float* __restrict__ bias, bf16* __restrict__ out, int cout,
                                                   int cp, int cg0, long npx, int sh, int s) {
  const int groups = min(cp / 8 - cg0, 32), lanes = 256 / groups;
  const int g = (cg0 + threadIdx.x % groups) * 8, pl = threadIdx.x / groups;
  if (pl >= lanes) return;
  float wv[8][9], bv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    bv[i] = g + i < cout ? bias[g + i] : 0.f;
#pragma unroll
    for (int t = 0; t < 9; ++t) wv[i][t] = g + i < cout ? (float)w[(g + i) * 9 + t] : 0.f;
  }
  for (long px = (long)blockIdx.x * lanes + pl; px < npx; px += (long)gridDim.x * lanes) {
    const int xx = (int)(px & (s - 1)), yy = (int)(px >> sh) & (s - 1);
    float v[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int y = yy + t / 3 - 1, c = xx + t % 3 - 1;
      v[t] = y >= 0 && y < s && c >= 0 && c < s ? (float)x[px + (long)(t / 3 - 1) * s + t % 3 - 1] : 0.f;
    }
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float acc = 0.f;
#pragma unroll
      for (int t = 0; t < 9; ++t) acc = fmaf(wv[i][t], v[t], acc);
      o[i] = fmaxf(acc + bv[i], 0.f);
    }
    *reinterpret_cast<uint4*>(out + px * cp + g) =
        make_uint4(bf_pair(o[0], o[1]), bf_pair(o[2], o[3]), bf_pair(o[4], o[5]), bf_pair(o[6], o[7]));
  }
}

// Its weight and bias gradient: thread = one of 32 channels (blockIdx.y) x one of 8 lanes, which take
// segments of up to 16 pixels of a row and slide the 3 x 3 window along them; the block's sums go to
// part[block][tap][channel] and bpart[block][channel], the channels in whole 32s.
// Four waves a SIMD hide its loads: 65 us for 16 samples of 256 x 256, and 101 with the two registers more
// that leave three.
__global__ __launch_bounds__(256, 4) void k_first_wgrad(const bf16* __restrict__ x, const float* __restrict__ dz, int cp,
                                                     long npx, int sh, int s, float* __restrict__ part,
                                                     double* __restrict__ bpart) {
  __shared__ float red[8][9][32];
  __shared__ double redb[8][32];
  constexpr int SEG = 16;
  const int c = threadIdx.x & 31, pl = threadIdx.x >> 5, co = blockIdx.y * 32 + c, pp = gridDim.y * 32;
  const int len = min(SEG, s), cz = min(co, cp - 1);  // sums of channels past the stored ones are not read
  float acc[9] = {};
  double bs = 0.0;
  for (long sg = (long)blockIdx.x * 8 + pl; sg < npx / len; sg += (long)gridDim.x * 8) {
    const long px = sg * len;
    const int xx = (int)(px & (s - 1)), yy = (int)(px >> sh) & (s - 1);
    const bool up = yy > 0, dn = yy + 1 < s;
    float d[SEG], v[3][SEG + 2];
#pragma unroll
    for (int i = 0; i < SEG; ++i) d[i] = i < len ? dz[(px + i) * cp + cz] : 0.f;
#pragma unroll
    for (int i = 0; i < SEG + 2; ++i) {
      const int cx = xx + i - 1;
      const bool in = cx >= 0 && cx < s && i < len + 2;
      v[0][i] = in && up ? (float)x[px + i - 1 - s] : 0.f;
      v[1][i] = in ? (float)x[px + i - 1] : 0.f;
      v[2][i] = in && dn ? (float)x[px + i - 1 + s] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < SEG; ++i) {
      bs += d[i];
      const float dr = (float)to_bf(d[i]);
#pragma unroll
      for (int t = 0; t < 9; ++t) acc[t] = fmaf(dr, v[t / 3][i + t % 3], acc[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < 9; ++t) red[pl][t][c] = acc[t];
  redb[pl][c] = bs;
  __syncthreads();
  for (int i = threadIdx.x; i < 9 * 32; i += 256) {
    float v = 0.f;
    for (int p = 0; p < 8; ++p) v += red[p][i / 32][i % 32];
    part[((long)blockIdx.x * 9 + i / 32) * pp + blockIdx.y * 32 + i % 32] = v;
  }
  if (threadIdx.x < 32) {
    double v = 0.0;
    for (int p = 0; p < 8; ++p) v += redb[p][c];
    bpart[(long)blockIdx.x * pp + co] = v;
  }
}
// g[co][t] and the bias from the blocks' sums, one wave per value
__global__ __launch_bounds__(64) void k_first_sum(const float* __restrict__ part, const double* __restrict__ bpart,
                                                  int blocks, int cp, float* __restrict__ gw, float* __restrict__ gb) {
  const int co = blockIdx.x, t = blockIdx.y;
  double s = 0.0;
  for (int b = threadIdx.x; b < blocks; b += 64)
    s += t < 9 ? (double)part[((long)b * 9 + t) * cp + co] : bpart[(long)b * cp + co];
  s = wave_sum(s);
  if (threadIdx.x == 0) {
    if (t < 9) gw[co * 9 + t] = (float)s;
    else gb[co] = (float)s;
  }
}

// Last layer: 1 x 1 to two channels (NCHW, FP32 out), one pixel per thread.
__global__ __launch_bounds__(256) void k_last_fwd(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                  const float* __restrict__ bias, float* __restrict__ out, int cin, int cp,
                                                  long npx, long ss) {
  for (long px = (long)blockIdx.x * 256 + threadIdx.x; px < npx; px += (long)gridDim.x * 256) {
    float a0 = 0.f, a1 = 0.f;
    for (int g = 0; g < cin; g += 8) {
      const uint4 v = *reinterpret_cast<const uint4*>(x + px * cp + g);
      const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (g + i >= cin) break;
        const float f = bf_val(i & 1 ? u[i >> 1] >> 16 : u[i >> 1] & 0xffffu);
        a0 = fmaf((float)w[g + i], f, a0);
        a1 = fmaf((float)w[cin + g + i], f, a1);
      }
    }
    const long b = px / ss, p = px - b * ss;
    out[(b * 2) * ss + p] = a0 + bias[0];
    out[(b * 2 + 1) * ss + p] = a1 + bias[1];
  }
}

// Its backward pass: the gradient of the input (masked by the input's ReLU) and the block's sums of
// the weight gradient, part[block][2][cp], and of the bias gradient, bpart[block][2].  A thread keeps
// 8 channels and strides over pixels; blockDim = 256 threads = 256 / (cp / 8) pixels at a time.
__global__ __launch_bounds__(256) void k_last_bwd(const float* __restrict__ gout, const bf16* __restrict__ x,
                                                  const bf16* __restrict__ w, float* __restrict__ gx, int cin, int cp,
                                                  int cg0, long npx, long ss, float* __restrict__ part,
                                                  double* __restrict__ bpart) {
  __shared__ float red[256][17];
  __shared__ double redb[256][2];
  const int groups = min(cp / 8 - cg0, 32), lanes = 256 / groups;
  const int g = threadIdx.x % groups, pl = threadIdx.x / groups, c0 = (cg0 + g) * 8;
  float w0[8], w1[8], s0[8] = {}, s1[8] = {};
  double b0 = 0.0, b1 = 0.0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    w0[i] = c0 + i < cin ? (float)w[c0 + i] : 0.f;
    w1[i] = c0 + i < cin ? (float)w[cin + c0 + i] : 0.f;
  }
  if (pl < lanes)
    for (long px = (long)blockIdx.x * lanes + pl; px < npx; px += (long)gridDim.x * lanes) {
      const long b = px / ss, p = px - b * ss;
      const float d0 = gout[(b * 2) * ss + p], d1 = gout[(b * 2 + 1) * ss + p];
      const float r0 = (float)to_bf(d0), r1 = (float)to_bf(d1);
      b0 += d0;
      b1 += d1;
      const uint4 v = *reinterpret_cast<const uint4*>(x + px * cp + c0);
      const unsigned u[4] = {v.x, v.y, v.z, v.w};
      float o[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float f = bf_val(i & 1 ? u[i >> 1] >> 16 : u[i >> 1] & 0xffffu);
        s0[i] = fmaf(r0, f, s0[i]);
        s1[i] = fmaf(r1, f, s1[i]);
        o[i] = f > 0.f ? fmaf(r1, w1[i], r0 * w0[i]) : 0.f;
      }
      float4* q = reinterpret_cast<float4*>(gx + px * cp + c0);
      q[0] = make_float4(o[0], o[1], o[2], o[3]);
      q[1] = make_float4(o[4], o[5], o[6], o[7]);
    }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    red[threadIdx.x][i] = s0[i];
    red[threadIdx.x][8 + i] = s1[i];
  }
  redb[threadIdx.x][0] = b0;
  redb[threadIdx.x][1] = b1;
  __syncthreads();
  for (int i = threadIdx.x; i < groups * 16; i += 256) {
    const int gg = i / 16, k = i % 16;
    float v = 0.f;
    for (int p = 0; p < lanes; ++p) v += red[p * groups + gg][k];
    part[((long)blockIdx.x * 2 + k / 8) * cp + (cg0 + gg) * 8 + k % 8] = v;
  }
  if (cg0 == 0 && threadIdx.x < 2) {
    double v = 0.0;
    for (int p = 0; p < lanes; ++p) v += redb[p * groups][threadIdx.x];
    bpart[blockIdx.x * 2 + threadIdx.x] = v;
  }
}
__global__ __launch_bounds__(64) void k_last_sum(const float* __restrict__ part, const double* __restrict__ bpart,
                                                 int blocks, int cin, int cp, float* __restrict__ gw,
                                                 float* __restrict__ gb) {
  const int ci = blockIdx.x, o = blockIdx.y;
  double s = 0.0;
  for (int b = threadIdx.x; b < blocks; b += 64)
    s += ci < cin ? (double)part[((long)b * 2 + o) * cp + ci] : bpart[b * 2 + o];
  s = wave_sum(s);
  if (threadIdx.x == 0) {
    if (ci < cin) gw[o * cin + ci] = (float)s;
    else gb[o] = (float)s;
  }
}

// 2 x 2 max pooling, 8 channels of one output pixel per thread; arg holds the winning offsets (0..3)
// for the backward pass, the first of equal ones
__global__ __launch_bounds__(256) void k_pool_fwd(const bf16* __restrict__ in, bf16* __restrict__ out,
                                                  uint8_t* __restrict__ arg, int cp, long total, int osh, int ow) {
  const int groups = cp / 8;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const long px = e / groups;
    const int g = (int)(e - px * groups) * 8, x = (int)(px & (ow - 1));
    const long row = px >> osh;  // (b, y)
    uint4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = *reinterpret_cast<const uint4*>(in + ((2 * row + (q >> 1)) * (2 * ow) + 2 * x + (q & 1)) * cp + g);
    unsigned o[4], am[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float best = -INFINITY;
      unsigned bits = 0xff80u, bi = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const unsigned u = i < 2 ? v[q].x : i < 4 ? v[q].y : i < 6 ? v[q].z : v[q].w;
        const unsigned h = i & 1 ? u >> 16 : u & 0xffffu;
        if (bf_val(h) > best) {
          best = bf_val(h);
          bits = h;
          bi = q;
        }
      }
      o[i >> 1] = i & 1 ? o[i >> 1] | (bits << 16) : bits;
      am[i >> 2] |= bi << (8 * (i & 3));
    }
    *reinterpret_cast<uint4*>(out + px * cp + g) = make_uint4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<uint2*>(arg + px * cp + g) = make_uint2(am[0], am[1]);
  }
}

// Gradient of the pooled tensor's input: the skip gradient already in gin plus gout at the winning
// offsets, zeroed where the activation is not positive (its ReLU).  8 channels of one pooled pixel
// (4 input pixels) per thread.
__global__ __launch_bounds__(256) void k_pool_bwd(const float* __restrict__ gout, float* __restrict__ gin,
                                                  const bf16* __restrict__ act, const uint8_t* __restrict__ arg, int cp,
                                                  long total, int osh, int ow) {
  const int groups = cp / 8;
  for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const long px = e / groups;
    const int g = (int)(e - px * groups) * 8, x = (int)(px & (ow - 1));
    const long row = px >> osh;
    const float4 ga = *reinterpret_cast<const float4*>(gout + px * cp + g);
    const float4 gb = *reinterpret_cast<const float4*>(gout + px * cp + g + 4);
    const float gv[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
    const uint2 am = *reinterpret_cast<const uint2*>(arg + px * cp + g);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long o = ((2 * row + (q >> 1)) * (2 * ow) + 2 * x + (q & 1)) * cp + g;
      float4* p = reinterpret_cast<float4*>(gin + o);
      const float4 u = p[0], w = p[1];
      const uint4 a = *reinterpret_cast<const uint4*>(act + o);
      const unsigned au[4] = {a.x, a.y, a.z, a.w};
      float r[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned bi = ((i < 4 ? am.x : am.y) >> (8 * (i & 3))) & 0xffu;
        if ((int)bi == q) r[i] += gv[i];
        if (!(bf_val(i & 1 ? au[i >> 1] >> 16 : au[i >> 1] & 0xffffu) > 0.f)) r[i] = 0.f;
      }
      p[0] = make_float4(r[0], r[1], r[2], r[3]);
      p[1] = make_float4(r[4], r[5], r[6], r[7]);
    }
  }
}

// weighted mean squared error: sum w(p) (y - t)^2 over all outputs, w an s x s map shared by the
// channels and samples (NULL: 1); g = 2 w (y - t) / norm with norm = batch * 2 * sum_p w(p);
// per-block FP64 partial sums of w (y - t)^2
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ y, const bf16* __restrict__ t, long count,
                                             const float* __restrict__ w, long ss, double norm,
                                             float* __restrict__ g, double* __restrict__ part) {
  __shared__ double red[4];
  double s = 0.0;
  const float sc = (float)(2.0 / norm);
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long)gridDim.x * 256) {
    const float d = y[i] - (float)t[i];
    const float wi = w ? w[i % ss] : 1.f;
    s += (double)wi * d * d;
    if (g) g[i] = sc * wi * d;
  }
  s = block_sum<256>(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_to_bf(const float* __restrict__ s, bf16* __restrict__ d, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = to_bf(s[i]);
}

inline int ilog2(int v) {
  int r = 0;
  while ((1 << r) < v) ++r;
  return r;
}
inline dim3 grid_of(long n) { return dim3((unsigned)std::min<long>((n + 255) / 256, 65535L * 4)); }
// enough blocks of an element loop to fill the GPU, no more
inline unsigned loop_blocks(long n) { return (unsigned)std::max<long>(1, std::min<long>((n + 255) / 256, 8192)); }

}  // namespace

// ---------------------------------------------------------------- host side
struct NnLayer {
  int cin, cout, ks, relu;
  long woff, boff;  // offsets in the parameter vector
};

constexpr int NN_CHUNKS = 512;       // workgroups that share a layer's weight gradient, about
constexpr int PREP_PARTS = 32;         // blocks per sample of the input's preparation
constexpr int NN_FIRST_BLOCKS = 1024;  // blocks of the first and last layer's gradients

struct NnNet {
  int s = 256, c = 32, batch = 8;
  std::vector<NnLayer> layers;
  LayerTable table{};
  long nparam = 0, nfwd = 0, ngrad = 0;  // parameters; elements of the fragment arrays
  float *w = nullptr, *mo = nullptr, *ve = nullptr, *g = nullptr;
  bf16 *wb = nullptr, *wf = nullptr, *wg = nullptr;  // BF16 copies: plain, forward and data-gradient fragments
  float* partial = nullptr;   // weight-gradient partial tiles
  double* bpart = nullptr;    // bias-gradient partial sums
  double* lpart = nullptr;
  long step = 0;
  struct Buf {
    int cp = 0, h = 0;   // stored channels, pixels a side
    bf16* a = nullptr;   // activation
    float* g = nullptr;  // its gradient
  };
  std::vector<Buf> bufs;
  uint8_t* arg[3] = {nullptr, nullptr, nullptr};
  float* out = nullptr;   // batch x 2 x s x s
  float* gout = nullptr;
  float* lw = nullptr;    // s x s loss weight (NULL: uniform)
  double lw_sum = 0.0;    // sum of the weight (s^2 when uniform)
  bf16* x = nullptr;      // batch x s x s
  bf16* target = nullptr; // batch x 2 x s x s (staging)
  hipStream_t stream = nullptr;
};

// Activations: A = first convolution of a level, E = encoder output, P = pooled, BN = bottleneck,
// D = decoder output of a level.
enum { B_A0, B_E0, B_P0, B_A1, B_E1, B_P1, B_A2, B_E2, B_P2, B_A3, B_BN, B_A4, B_D2, B_A5, B_D1, B_A6, B_D0, B_COUNT };
// The 13 convolutions between them: layer, inputs (in1 < 0: one; else in0 is upsampled), output, level.
struct ConvStep {
  int layer, in0, in1, out, level;
};
static const ConvStep kSteps[13] = {{1, B_A0, -1, B_E0, 0},  {2, B_P0, -1, B_A1, 1},   {3, B_A1, -1, B_E1, 1},
                                    {4, B_P1, -1, B_A2, 2},  {5, B_A2, -1, B_E2, 2},   {6, B_P2, -1, B_A3, 3},
                                    {7, B_A3, -1, B_BN, 3},  {8, B_BN, B_E2, B_A4, 2}, {9, B_A4, -1, B_D2, 2},
                                    {10, B_D2, B_E1, B_A5, 1}, {11, B_A5, -1, B_D1, 1}, {12, B_D1, B_E0, B_A6, 0},
                                    {13, B_A6, -1, B_D0, 0}};

int nn_layer_table(int c, std::vector<NnLayer>* out, long* nparam) {
  const int tab[NN_LAYERS][4] = {{1, c, 3, 1},          {c, c, 3, 1},          {c, 2 * c, 3, 1},     {2 * c, 2 * c, 3, 1},
                                 {2 * c, 4 * c, 3, 1},  {4 * c, 4 * c, 3, 1},  {4 * c, 8 * c, 3, 1}, {8 * c, 8 * c, 3, 1},
                                 {12 * c, 4 * c, 3, 1}, {4 * c, 4 * c, 3, 1},  {6 * c, 2 * c, 3, 1}, {2 * c, 2 * c, 3, 1},
                                 {3 * c, c, 3, 1},      {c, c, 3, 1},          {c, 2, 1, 0}};
  out->clear();
  long off = 0;
  for (auto& t : tab) {
    NnLayer l{t[0], t[1], t[2], t[3], 0, 0};
    l.woff = off;
    off += (long)l.cout * l.cin * l.ks * l.ks;
    l.boff = off;
    off += l.cout;
    out->push_back(l);
  }
  *nparam = off;
  return NN_LAYERS;
}

template <int NCO, int ROWS, bool GRAD>
static long conv3_blocks(const ConvArgs& a, int out_tiles) {
  const long tiles = (long)a.batch * ((a.w_px + 31) / 32) * ((a.h + 4 * ROWS - 1) / (4 * ROWS));
  return (tiles + 7) / 8 * 8 * (out_tiles / NCO);
}
template <int NCO, int ROWS, bool GRAD, bool PART>
static hipError_t conv3_launch(ConvArgs a, int out_tiles, hipStream_t st) {
  constexpr size_t lds = (size_t)((4 * ROWS + 2) * 34 * 4 + NCO * 9 * 2 * 64) * sizeof(uint4);
  static_assert(lds <= 80 * 1024, "two workgroups per CU");
  const hipError_t e = hipFuncSetAttribute((const void*)k_conv3<NCO, ROWS, GRAD, PART>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  a.tiles_x = (a.w_px + 31) / 32;
  a.tiles_y = (a.h + 4 * ROWS - 1) / (4 * ROWS);
  a.groups = out_tiles / NCO;
  const long blocks = conv3_blocks<NCO, ROWS, GRAD>(a, out_tiles);
  if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_conv3<NCO, ROWS, GRAD, PART>), dim3((unsigned)blocks), dim3(CT), lds, st, a);
  return hipGetLastError();
}
// The largest tile that still gives the 256 CUs two workgroups each: two output tiles of 32 channels
// halve the input reads, 16 rows halve the border; the small levels (32 x 32 and 64 x 64 pixels of 8
// samples) run on finer tiles instead of on a quarter of the chip.
template <bool GRAD, bool PART>
static hipError_t conv3_tiled(const ConvArgs& a, int out_tiles, hipStream_t st) {
  constexpr long FULL = 512;
  if (out_tiles % 2 == 0 && a.h > 8 && conv3_blocks<2, 4, GRAD>(a, out_tiles) >= FULL)
    return conv3_launch<2, 4, GRAD, PART>(a, out_tiles, st);
  if (out_tiles % 2 == 0 && conv3_blocks<2, 2, GRAD>(a, out_tiles) >= FULL)
    return conv3_launch<2, 2, GRAD, PART>(a, out_tiles, st);
  if (a.h > 8 && conv3_blocks<1, 4, GRAD>(a, out_tiles) >= FULL) return conv3_launch<1, 4, GRAD, PART>(a, out_tiles, st);
  return conv3_launch<1, 2, GRAD, PART>(a, out_tiles, st);
}
template <bool GRAD>
static hipError_t conv3(const ConvArgs& a, int out_tiles, hipStream_t st) {
  const bool part = (a.in.cp0 | a.in.cp1 | a.out0.cp | a.out1.cp) % 32 != 0;
  return part ? conv3_tiled<GRAD, true>(a, out_tiles, st) : conv3_tiled<GRAD, false>(a, out_tiles, st);
}

static Src conv_src(const NnNet& n, const ConvStep& s) {
  const auto& b0 = n.bufs[s.in0];
  if (s.in1 < 0) return Src{b0.a, nullptr, b0.cp, 0, 0};
  const auto& b1 = n.bufs[s.in1];
  return Src{b0.a, b1.a, b0.cp, b1.cp, 1};
}

static hipError_t conv_fwd(NnNet& n, const ConvStep& s) {
  const LayerMap& m = n.table.l[s.layer];
  ConvArgs a{};
  a.in = conv_src(n, s);
  a.w = n.wf + m.foff;
  a.bias = n.w + m.boff;
  a.out0 = Dst{n.bufs[s.out].a, nullptr, n.bufs[s.out].cp, 0};
  a.out0_tiles = m.cpo / 32;
  a.cout = m.cout;
  a.batch = n.batch;
  a.h = a.w_px = n.s >> s.level;
  a.chunks = m.cpi / 32;
  a.relu = n.layers[s.layer].relu;
  return conv3<false>(a, m.cpo / 32, n.stream);
}

// The share of a layer's 8 x 32-pixel tiles: about NN_CHUNKS workgroups in all.
static int wgrad_chunks(const LayerMap& m, int batch, int hw) {
  const long tiles = (long)batch * ((hw + WG_R - 1) / WG_R) * ((hw + 31) / 32);
  const int pairs = (m.cpo / 32) * (m.cpi / 32);
  return (int)std::max<long>(1, std::min<long>(tiles, (NN_CHUNKS + pairs - 1) / pairs));
}

// n.bufs[s.out].g holds the gradient of the layer's pre-activation output; makes the parameters'
// gradient and the inputs' (masked by their ReLU, where no pooling gradient is still to be added).
static hipError_t conv_bwd(NnNet& n, const ConvStep& s) {
  const LayerMap& m = n.table.l[s.layer];
  const int hw = n.s >> s.level;
  const float* dz = n.bufs[s.out].g;
  {
    WgradArgs a{};
    a.x = conv_src(n, s);
    a.dz = dz;
    a.part = n.partial;
    a.bpart = n.bpart;
    a.batch = n.batch;
    a.h = a.w_px = hw;
    a.cz = n.bufs[s.out].cp;
    a.cpo = m.cpo;
    a.tiles_o = m.cpo / 32;
    a.tiles_i = m.cpi / 32;
    a.tiles_x = (hw + 31) / 32;
    a.tiles_y = (hw + WG_R - 1) / WG_R;
    a.chunks = wgrad_chunks(m, n.batch, hw);
    constexpr size_t lds = 32 * WG_ZP + 3 * 32 * WG_XP;
    static_assert(lds >= 9 * 1024 * sizeof(float) && lds <= 80 * 1024, "reduction scratch; two workgroups per CU");
    const auto kernel = (a.x.cp0 | a.x.cp1 | a.cz) % 32 ? k_wgrad3<true> : k_wgrad3<false>;
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles_o * a.tiles_i * a.chunks)), dim3(CT), lds, n.stream, a);
    hipLaunchKernelGGL(k_wgrad_sum, dim3((unsigned)(a.tiles_o * a.tiles_i * 9 * 32 + a.tiles_o)), dim3(256), 0, n.stream, m,
                       n.partial, n.bpart, a.chunks, n.g);
  }
  ConvArgs a{};
  a.in = Src{dz, nullptr, n.bufs[s.out].cp, 0, 0};
  a.w = n.wg + m.goff;
  const auto& b0 = n.bufs[s.in0];
  const bool pooled = s.in0 == B_P0 || s.in0 == B_P1 || s.in0 == B_P2;
  a.out0 = Dst{b0.g, pooled ? nullptr : b0.a, b0.cp, s.in1 >= 0 ? 1 : 0};
  a.out0_tiles = m.cp0 / 32;
  if (s.in1 >= 0) a.out1 = Dst{n.bufs[s.in1].g, nullptr, n.bufs[s.in1].cp, 0};
  a.batch = n.batch;
  a.h = a.w_px = hw;
  a.chunks = m.cpo / 32;
  return conv3<true>(a, m.cpi / 32, n.stream);
}

static void pool_fwd(NnNet& n, int in, int out, int lv) {
  const auto& o = n.bufs[out];
  const long total = (long)n.batch * o.h * o.h * (o.cp / 8);
  hipLaunchKernelGGL(k_pool_fwd, dim3(loop_blocks(total)), dim3(256), 0, n.stream, n.bufs[in].a, o.a, n.arg[lv], o.cp,
                     total, ilog2(o.h), o.h);
}
static void pool_bwd(NnNet& n, int in, int out, int lv) {
  const auto& o = n.bufs[out];
  const long total = (long)n.batch * o.h * o.h * (o.cp / 8);
  hipLaunchKernelGGL(k_pool_bwd, dim3(loop_blocks(total)), dim3(256), 0, n.stream, o.g, n.bufs[in].g, n.bufs[in].a,
                     n.arg[lv], o.cp, total, ilog2(o.h), o.h);
}

hipError_t nn_forward(NnNet& n) {
  const LayerMap &f = n.table.l[0], &l = n.table.l[14];
  const long npx = (long)n.batch * n.s * n.s;
  const int cf = n.bufs[B_A0].cp, cl = n.bufs[B_D0].cp;
  for (int cg = 0; cg < cf / 8; cg += 32)
    hipLaunchKernelGGL(k_first_fwd, dim3((unsigned)std::max<long>(1, std::min<long>(2048, npx / 64))), dim3(256), 0,
                       n.stream, n.x, n.wb + f.woff, n.w + f.boff, n.bufs[B_A0].a, f.cout, cf, cg, npx, ilog2(n.s), n.s);
  for (const ConvStep& s : kSteps) {
    const hipError_t e = conv_fwd(n, s);
    if (e != hipSuccess) return e;
    if (s.out == B_E0) pool_fwd(n, B_E0, B_P0, 0);
    if (s.out == B_E1) pool_fwd(n, B_E1, B_P1, 1);
    if (s.out == B_E2) pool_fwd(n, B_E2, B_P2, 2);
  }
  hipLaunchKernelGGL(k_last_fwd, dim3(loop_blocks(npx)), dim3(256), 0, n.stream, n.bufs[B_D0].a, n.wb + l.woff,
                     n.w + l.boff, n.out, l.cin, cl, npx, (long)n.s * n.s);
  return hipGetLastError();
}

// loss over the batch (returned via lpart partials, count = batch*2*s*s); with_grad: backward
hipError_t nn_loss(NnNet& n, bool with_grad, int* nparts) {
  const long count = (long)n.batch * 2 * n.s * n.s;
  const int nb = (int)std::min<long>((count + 255) / 256, 1024);
  const double norm = (double)n.batch * 2 * n.lw_sum;
  hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, n.stream, n.out, n.target, count, n.lw, (long)n.s * n.s, norm,
                     with_grad ? n.gout : nullptr, n.lpart);
  *nparts = nb;
  return hipGetLastError();
}

hipError_t nn_backward(NnNet& n) {
  const LayerMap &f = n.table.l[0], &l = n.table.l[14];
  const long ss = (long)n.s * n.s, npx = n.batch * ss;
  {
    const unsigned nb = (unsigned)std::max<long>(1, std::min<long>(NN_FIRST_BLOCKS, npx / 64));
    const int cl = n.bufs[B_D0].cp;
    for (int cg = 0; cg < cl / 8; cg += 32)
      hipLaunchKernelGGL(k_last_bwd, dim3(nb), dim3(256), 0, n.stream, n.gout, n.bufs[B_D0].a, n.wb + l.woff,
                         n.bufs[B_D0].g, l.cin, cl, cg, npx, ss, n.partial, n.bpart);
    hipLaunchKernelGGL(k_last_sum, dim3(l.cin + 1, 2), dim3(64), 0, n.stream, n.partial, n.bpart, (int)nb, l.cin, cl,
                       n.g + l.woff, n.g + l.boff);
  }
  for (int i = 12; i >= 0; --i) {
    const ConvStep& s = kSteps[i];
    // the encoder outputs' gradients are whole once their pooled tensor's is there
    if (s.out == B_E0) pool_bwd(n, B_E0, B_P0, 0);
    if (s.out == B_E1) pool_bwd(n, B_E1, B_P1, 1);
    if (s.out == B_E2) pool_bwd(n, B_E2, B_P2, 2);
    const hipError_t e = conv_bwd(n, s);
    if (e != hipSuccess) return e;
  }
  const unsigned nb = (unsigned)std::max<long>(1, std::min<long>(NN_FIRST_BLOCKS, npx / 64));
  hipLaunchKernelGGL(k_first_wgrad, dim3(nb, f.cpo / 32), dim3(256), 0, n.stream, n.x, n.bufs[B_A0].g, n.bufs[B_A0].cp, npx,
                     ilog2(n.s), n.s, n.partial, n.bpart);
  hipLaunchKernelGGL(k_first_sum, dim3(f.cout, 10), dim3(64), 0, n.stream, n.partial, n.bpart, (int)nb, f.cpo,
                     n.g + f.woff, n.g + f.boff);
  return hipGetLastError();
}

hipError_t nn_adam(NnNet& n, float lr) {
  n.step += 1;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = (float)(1.0 - std::pow(0.9, (double)n.step)), c2 = (float)(1.0 - std::pow(0.999, (double)n.step));
  hipLaunchKernelGGL(k_adam, dim3((unsigned)((n.nparam + 255) / 256)), dim3(256), 0, n.stream, n.table, n.w, n.mo, n.ve,
                     n.g, n.wb, n.wf, n.wg, n.nparam, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t nn_refresh_bf16(NnNet& n) {
  hipLaunchKernelGGL(k_pack, dim3((unsigned)((n.nparam + 255) / 256)), dim3(256), 0, n.stream, n.table, n.w, n.nparam,
                     n.wb, n.wf, n.wg);
  return hipGetLastError();
}

static hipError_t nn_alloc1(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes ? bytes : 8);
  if (e == hipSuccess) e = hipMemset(*p, 0, bytes ? bytes : 8);
  return e;
}

hipError_t nn_create(NnNet& n, int s, int c, int batch) {
  n.s = s;
  n.c = c;
  n.batch = batch;
  n.lw_sum = (double)s * s;
  nn_layer_table(c, &n.layers, &n.nparam);
  const int ch[B_COUNT] = {c, c, c, 2 * c, 2 * c, 2 * c, 4 * c, 4 * c, 4 * c, 8 * c, 8 * c, 4 * c, 4 * c, 2 * c, 2 * c, c, c};
  const int lv[B_COUNT] = {0, 0, 1, 1, 1, 2, 2, 2, 3, 3, 3, 2, 2, 1, 1, 0, 0};
  for (int i = 0; i < NN_LAYERS; ++i) {
    const NnLayer& L = n.layers[i];
    LayerMap& m = n.table.l[i];
    m = LayerMap{L.woff, L.boff, 0, 0, L.cin, L.cout, L.ks, L.cin, pad32(L.cin), pad32(L.cin), pad32(L.cout)};
  }
  for (const ConvStep& st : kSteps) {
    LayerMap& m = n.table.l[st.layer];
    m.c0 = ch[st.in0];
    m.cp0 = pad32(m.c0);
    m.cpi = m.cp0 + (st.in1 >= 0 ? pad32(ch[st.in1]) : 0);
    m.foff = n.nfwd;
    m.goff = n.ngrad;
    n.nfwd += (long)m.cpo * m.cpi * 9;
    n.ngrad += (long)m.cpo * m.cpi * 9;
  }
  n.bufs.resize(B_COUNT);
  hipError_t e = hipSuccess;
  for (int i = 0; i < B_COUNT && e == hipSuccess; ++i) {
    n.bufs[i].cp = pad8(ch[i]);
    n.bufs[i].h = s >> lv[i];
    const size_t cnt = (size_t)batch * n.bufs[i].cp * n.bufs[i].h * n.bufs[i].h;
    e = nn_alloc1((void**)&n.bufs[i].a, cnt * sizeof(bf16));
    if (e == hipSuccess) e = nn_alloc1((void**)&n.bufs[i].g, cnt * sizeof(float));
  }
  for (int l = 0; l < 3 && e == hipSuccess; ++l)
    e = nn_alloc1((void**)&n.arg[l], (size_t)batch * pad8(c << l) * (s >> (l + 1)) * (s >> (l + 1)));
  const size_t outc = (size_t)batch * 2 * s * s;
  if (e == hipSuccess) e = nn_alloc1((void**)&n.x, outc / 2 * sizeof(bf16));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.out, outc * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.gout, outc * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.target, outc * sizeof(bf16));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.w, n.nparam * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.mo, n.nparam * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.ve, n.nparam * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.g, n.nparam * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.wb, n.nparam * sizeof(bf16));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.wf, n.nfwd * sizeof(bf16));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.wg, n.ngrad * sizeof(bf16));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.lpart, 1024 * sizeof(double));
  // partial sums of the gradients: the most any layer needs
  const LayerMap &f = n.table.l[0], &l = n.table.l[14];
  size_t part = std::max<size_t>((size_t)NN_FIRST_BLOCKS * std::max(9 * f.cpo, 2 * l.cpi), (size_t)batch * PREP_PARTS), bias = (size_t)NN_FIRST_BLOCKS * std::max(f.cpo, 2);
  for (const ConvStep& st : kSteps) {
    const LayerMap& m = n.table.l[st.layer];
    const size_t chunks = wgrad_chunks(m, batch, s >> st.level);
    part = std::max(part, chunks * m.cpo * m.cpi * 9);
    bias = std::max(bias, chunks * m.cpo);
  }
  if (e == hipSuccess) e = nn_alloc1((void**)&n.partial, part * sizeof(float));
  if (e == hipSuccess) e = nn_alloc1((void**)&n.bpart, bias * sizeof(double));
  if (e == hipSuccess) e = hipDeviceSynchronize();
  return e;
}

void nn_free(NnNet& n) {
  for (auto& b : n.bufs) {
    if (b.a) hipFree(b.a);
    if (b.g) hipFree(b.g);
  }
  n.bufs.clear();
  for (auto& p : n.arg)
    if (p) hipFree(p);
  for (void* p : {(void*)n.x, (void*)n.out, (void*)n.gout, (void*)n.target, (void*)n.w, (void*)n.mo, (void*)n.ve, (void*)n.g,
                  (void*)n.wb, (void*)n.wf, (void*)n.wg, (void*)n.bpart, (void*)n.lpart, (void*)n.partial, (void*)n.lw})
    if (p) hipFree(p);
}


__global__ void k_gather_rows(const bf16* __restrict__ src, const int64_t* __restrict__ idx, long row, int count,
                              bf16* __restrict__ dst) {
  const long total = (long)count * row;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long r = i / row, q = i - r * row;
    dst[i] = src[idx[r] * row + q];
  }
}

// Network input from raw amplitudes: x = log(1 + max(A, 0)) / max over the sample (a sample whose
// maximum is 0 maps to 0), in two passes of PREP_PARTS blocks per sample: the parts' maxima, then the
// values.  (One block per sample ran on as many CUs as there are samples: 243 us for 8 of 256 x 256.)
__global__ __launch_bounds__(256) void k_prep_max(const float* __restrict__ amp, long ss, float* __restrict__ part) {
  __shared__ float red[4];
  const float* a = amp + blockIdx.y * ss;
  float mx = 0.f;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < ss; i += PREP_PARTS * 256)
    mx = fmaxf(mx, log1pf(fmaxf(a[i], 0.f)));
  mx = block_max<256>(mx, red);
  if (threadIdx.x == 0) part[blockIdx.y * PREP_PARTS + blockIdx.x] = mx;
}
__global__ __launch_bounds__(256) void k_prep_amplitudes(const float* __restrict__ amp, long ss,
                                                         const float* __restrict__ part, bf16* __restrict__ x) {
  const float* a = amp + blockIdx.y * ss;
  bf16* o = x + blockIdx.y * ss;
  const float mx = wave_max(part[blockIdx.y * PREP_PARTS + (threadIdx.x & (PREP_PARTS - 1))]);
  const float inv = mx > 0.f ? 1.f / mx : 0.f;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < ss; i += PREP_PARTS * 256)
    o[i] = to_bf(log1pf(fmaxf(a[i], 0.f)) * inv);
}

}  // namespace ptyk

// ---------------------------------------------------------------- C ABI
using namespace ptyk;

struct ptyk_net {
  NnNet n;
  int device = 0;
  std::string err;
  bf16* data_x = nullptr;
  bf16* data_y = nullptr;
  int64_t ndata = 0;     // samples [0, ndata) hold data
  int64_t data_cap = 0;  // samples the device buffers hold room for
  int64_t* idx = nullptr;
  int64_t idx_cap = 0;
  hipStream_t copy = nullptr;  // the predictions' copies to and from the host; made by the first one
  float* io = nullptr;         // `held` batches of samples and of results
  int64_t held = 0;
};

static thread_local std::string g_net_err;

#define NCHK(h, call)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) {                                                            \
      (h)->err = std::string(#call) + ": " + hipGetErrorString(e_);                    \
      return e_ == hipErrorOutOfMemory ? PTYK_ENOMEM : PTYK_EDEVICE;                   \
    }                                                                                  \
  } while (0)

extern "C" {

int ptyk_net_create(int32_t device, int32_t size, int32_t base_channels, int32_t batch, uint64_t seed,
                    ptyk_net** out) {
  if (!out || size < 8 || (size & (size - 1)) || base_channels < 1 || batch < 1) {
    g_net_err = "size must be a power of two >= 8; channels and batch >= 1";
    return PTYK_EINVAL;
  }
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
    g_net_err = "no such HIP device";
    return PTYK_EDEVICE;
  }
  hipSetDevice(device);
  ptyk_net* h = new ptyk_net();
  h->device = device;
  hipError_t e = hipStreamCreateWithFlags(&h->n.stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = nn_create(h->n, size, base_channels, batch);
  if (e != hipSuccess) {
    g_net_err = std::string("network allocation: ") + hipGetErrorString(e);
    nn_free(h->n);
    if (h->n.stream) hipStreamDestroy(h->n.stream);
    delete h;
    return e == hipErrorOutOfMemory ? PTYK_ENOMEM : PTYK_EDEVICE;
  }
  // He-normal weights (seeded), zero biases
  std::vector<float> w(h->n.nparam, 0.f);
  NormalDraw nd(seed);
  for (const auto& L : h->n.layers) {
    const double sd = std::sqrt(2.0 / (L.cin * L.ks * L.ks));
    for (long i = 0; i < (long)L.cout * L.cin * L.ks * L.ks; ++i) w[L.woff + i] = (float)(sd * nd());
  }
  int r = ptyk_net_set_params(h, w.data());
  if (r) {
    g_net_err = h->err;
    ptyk_net_destroy(h);
    return r;
  }
  *out = h;
  return PTYK_OK;
}

void ptyk_net_destroy(ptyk_net* h) {
  if (!h) return;
  hipSetDevice(h->device);
  if (h->n.stream) hipStreamSynchronize(h->n.stream);
  nn_free(h->n);
  for (void* p : {(void*)h->data_x, (void*)h->data_y, (void*)h->idx, (void*)h->io})
    if (p) hipFree(p);
  for (hipStream_t st : {h->n.stream, h->copy})
    if (st) hipStreamDestroy(st);
  delete h;
}

const char* ptyk_net_last_error(const ptyk_net* h) { return h ? h->err.c_str() : g_net_err.c_str(); }

int64_t ptyk_net_num_params(const ptyk_net* h) { return h ? h->n.nparam : -1; }

int ptyk_net_get_params(ptyk_net* h, float* out) {
  if (!h || !out) return PTYK_EINVAL;
  hipSetDevice(h->device);
  NCHK(h, hipMemcpyAsync(out, h->n.w, h->n.nparam * sizeof(float), hipMemcpyDeviceToHost, h->n.stream));
  NCHK(h, hipStreamSynchronize(h->n.stream));
  return PTYK_OK;
}

int ptyk_net_set_params(ptyk_net* h, const float* in) {
  if (!h || !in) return PTYK_EINVAL;
  hipSetDevice(h->device);
  NCHK(h, hipMemcpyAsync(h->n.w, in, h->n.nparam * sizeof(float), hipMemcpyHostToDevice, h->n.stream));
  NCHK(h, nn_refresh_bf16(h->n));
  NCHK(h, hipMemsetAsync(h->n.mo, 0, h->n.nparam * sizeof(float), h->n.stream));
  NCHK(h, hipMemsetAsync(h->n.ve, 0, h->n.nparam * sizeof(float), h->n.stream));
  NCHK(h, hipStreamSynchronize(h->n.stream));
  h->n.step = 0;
  return PTYK_OK;
}

// Per-pixel loss weight (s x s, non-negative, not all zero), shared by both output channels and
// every sample; NULL restores the uniform weight.
int ptyk_net_set_loss_weight(ptyk_net* h, const float* weight) {
  if (!h) return PTYK_EINVAL;
  hipSetDevice(h->device);
  const long ss = (long)h->n.s * h->n.s;
  if (!weight) {
    NCHK(h, hipStreamSynchronize(h->n.stream));
    if (h->n.lw) hipFree(h->n.lw);
    h->n.lw = nullptr;
    h->n.lw_sum = (double)ss;
    return PTYK_OK;
  }
  double sum = 0.0;
  for (long i = 0; i < ss; ++i) {
    if (!(weight[i] >= 0.f) || !std::isfinite(weight[i])) {
      h->err = "loss weights must be finite and non-negative";
      return PTYK_EINVAL;
    }
    sum += weight[i];
  }
  if (!(sum > 0.0)) {
    h->err = "loss weights are all zero";
    return PTYK_EINVAL;
  }
  if (!h->n.lw) NCHK(h, hipMalloc((void**)&h->n.lw, ss * sizeof(float)));
  NCHK(h, hipMemcpyAsync(h->n.lw, weight, ss * sizeof(float), hipMemcpyHostToDevice, h->n.stream));
  NCHK(h, hipStreamSynchronize(h->n.stream));
  h->n.lw_sum = sum;
  return PTYK_OK;
}

// Device room for n samples (BF16); previous samples are dropped.
int ptyk_net_reserve_data(ptyk_net* h, int64_t n) {
  if (!h || n <= 0) return PTYK_EINVAL;
  hipSetDevice(h->device);
  const long ss = (long)h->n.s * h->n.s;
  NCHK(h, hipStreamSynchronize(h->n.stream));
  if (h->data_x) hipFree(h->data_x);
  if (h->data_y) hipFree(h->data_y);
  h->data_x = h->data_y = nullptr;
  h->ndata = h->data_cap = 0;
  NCHK(h, hipMalloc((void**)&h->data_x, (size_t)n * ss * sizeof(bf16)));
  NCHK(h, hipMalloc((void**)&h->data_y, (size_t)n * 2 * ss * sizeof(bf16)));
  h->data_cap = n;
  return PTYK_OK;
}

// BF16 device copy of samples [offset, offset + count): inputs count x s x s, targets
// count x 2 x s x s (float, host); samples up to offset + count become usable.
int ptyk_net_put_data(ptyk_net* h, int64_t offset, const float* inputs, const float* targets, int64_t count) {
  if (!h || !inputs || !targets || offset < 0 || count <= 0) return PTYK_EINVAL;
  if (offset + count > h->data_cap) {
    h->err = "samples beyond the reserved room";
    return PTYK_EINVAL;
  }
  hipSetDevice(h->device);
  const long ss = (long)h->n.s * h->n.s;
  const int64_t slice = 256;
  float* stage = nullptr;
  NCHK(h, hipMalloc((void**)&stage, (size_t)std::min(slice, count) * 2 * ss * sizeof(float)));
  hipError_t e = hipSuccess;
  for (int64_t b = 0; b < count && e == hipSuccess; b += slice) {
    const int64_t cnt = std::min(slice, count - b);
    bf16* dx = h->data_x + (offset + b) * ss;
    bf16* dy = h->data_y + (offset + b) * 2 * ss;
    e = hipMemcpyAsync(stage, inputs + b * ss, (size_t)cnt * ss * sizeof(float), hipMemcpyHostToDevice, h->n.stream);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((cnt * ss + 255) / 256)), dim3(256), 0, h->n.stream, stage, dx,
                         (long)(cnt * ss));
      e = hipMemcpyAsync(stage, targets + b * 2 * ss, (size_t)cnt * 2 * ss * sizeof(float), hipMemcpyHostToDevice,
                         h->n.stream);
    }
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((cnt * 2 * ss + 255) / 256)), dim3(256), 0, h->n.stream, stage, dy,
                         (long)(cnt * 2 * ss));
      e = hipStreamSynchronize(h->n.stream);  // the staging buffer is refilled next slice
    }
  }
  hipFree(stage);
  NCHK(h, e);
  h->ndata = std::max(h->ndata, offset + count);
  return PTYK_OK;
}

int ptyk_net_set_data(ptyk_net* h, const float* inputs, const float* targets, int64_t n) {
  if (!h || !inputs || !targets || n <= 0) return PTYK_EINVAL;
  int r = ptyk_net_reserve_data(h, n);
  return r ? r : ptyk_net_put_data(h, 0, inputs, targets, n);
}

static int net_load_batch(ptyk_net* h, const int64_t* order, int64_t off) {
  const long ss = (long)h->n.s * h->n.s;
  const int B = h->n.batch;
  if (h->idx_cap < B) {
    if (h->idx) hipFree(h->idx);
    NCHK(h, hipMalloc((void**)&h->idx, B * sizeof(int64_t)));
    h->idx_cap = B;
  }
  NCHK(h, hipMemcpyAsync(h->idx, order + off, B * sizeof(int64_t), hipMemcpyHostToDevice, h->n.stream));
  hipLaunchKernelGGL(k_gather_rows, grid_of((long)B * ss), dim3(256), 0, h->n.stream, h->data_x, h->idx, ss, B,
                     h->n.x);
  hipLaunchKernelGGL(k_gather_rows, grid_of((long)B * 2 * ss), dim3(256), 0, h->n.stream, h->data_y, h->idx, 2 * ss,
                     B, h->n.target);
  NCHK(h, hipStreamSynchronize(h->n.stream));  // the order slice is host memory of the caller
  return PTYK_OK;
}

static int net_loss_value(ptyk_net* h, int nparts, double* loss) {
  std::vector<double> p(nparts);
  NCHK(h, hipMemcpyAsync(p.data(), h->n.lpart, nparts * sizeof(double), hipMemcpyDeviceToHost, h->n.stream));
  NCHK(h, hipStreamSynchronize(h->n.stream));
  double s = 0;
  for (double v : p) s += v;
  *loss = s / ((double)h->n.batch * 2 * h->n.lw_sum);
  return PTYK_OK;
}

// Adam steps over the stored samples order[0..count) in batches (count a multiple of batch).
int ptyk_net_train(ptyk_net* h, const int64_t* order, int64_t count, float lr, double* mean_loss) {
  if (!h || !order || count <= 0 || count % h->n.batch) {
    if (h) h->err = "count must be a positive multiple of the batch";
    return PTYK_EINVAL;
  }
  for (int64_t i = 0; i < count; ++i)
    if (order[i] < 0 || order[i] >= h->ndata) {
      h->err = "sample index out of range";
      return PTYK_EINVAL;
    }
  hipSetDevice(h->device);
  double tot = 0;
  for (int64_t off = 0; off < count; off += h->n.batch) {
    int r = net_load_batch(h, order, off);
    if (r) return r;
    NCHK(h, nn_forward(h->n));
    int np = 0;
    NCHK(h, nn_loss(h->n, true, &np));
    NCHK(h, nn_backward(h->n));
    NCHK(h, nn_adam(h->n, lr));
    double l = 0;
    r = net_loss_value(h, np, &l);
    if (r) return r;
    tot += l;
  }
  if (mean_loss) *mean_loss = tot / (count / h->n.batch);
  return PTYK_OK;
}

int ptyk_net_evaluate(ptyk_net* h, const int64_t* order, int64_t count, double* mean_loss) {
  if (!h || !order || count <= 0 || count % h->n.batch || !mean_loss) return PTYK_EINVAL;
  for (int64_t i = 0; i < count; ++i)
    if (order[i] < 0 || order[i] >= h->ndata) {
      h->err = "sample index out of range";
      return PTYK_EINVAL;
    }
  hipSetDevice(h->device);
  double tot = 0;
  for (int64_t off = 0; off < count; off += h->n.batch) {
    int r = net_load_batch(h, order, off);
    if (r) return r;
    NCHK(h, nn_forward(h->n));
    int np = 0;
    NCHK(h, nn_loss(h->n, false, &np));
    double l = 0;
    r = net_loss_value(h, np, &l);
    if (r) return r;
    tot += l;
  }
  *mean_loss = tot / (count / h->n.batch);
  return PTYK_OK;
}

// Forward pass on host inputs (n x s x s float) -> outputs (n x 2 x s x s float); raw: the
// inputs are diffraction amplitudes, preprocessed on the device.
//
// The batches of a block run one after the other with no wait between them: the samples after the first
// batch's come in while that is computed, and results leave as their batch ends.  60 frames of 256^2 in
// batches of 8 took 6.0 ms, half of it copies and allocations with the device idle; now 3.5, the kernels 3.0.
static int net_predict(ptyk_net* h, const float* inputs, int64_t n, float* outputs, bool raw) {
  if (!h || !inputs || !outputs || n <= 0) return PTYK_EINVAL;
  hipSetDevice(h->device);
  const long ss = (long)h->n.s * h->n.s;
  const int B = h->n.batch;
  if (!h->copy) NCHK(h, hipStreamCreateWithFlags(&h->copy, hipStreamNonBlocking));
  const hipStream_t s = h->n.stream, cs = h->copy;
  const size_t batch_bytes = (size_t)B * 3 * ss * sizeof(float);
  // batches held at once: 32, and 64 MiB of samples and results
  int64_t hold = std::max<int64_t>(1, std::min<int64_t>({(n + B - 1) / B, 32, (int64_t)((64u << 20) / batch_bytes)}));
  if (h->held < hold) {
    hipFree(h->io);
    h->io = nullptr;
    h->held = 0;
    hipError_t e = hipMalloc((void**)&h->io, hold * batch_bytes);
    if (e != hipSuccess && hold > 1) {
      (void)hipGetLastError();
      hold = 1;
      e = hipMalloc((void**)&h->io, batch_bytes);
    }
    NCHK(h, e);
    h->held = hold;
  }
  float *const in = h->io, *const res = in + hold * B * ss, *const own = h->n.out;
  hipEvent_t came[2] = {}, done[32] = {};
  hipError_t e = hipSuccess;
  for (auto* ev : {&came[0], &came[1]})
    if (e == hipSuccess) e = hipEventCreateWithFlags(ev, hipEventDisableTiming);
  for (int64_t k = 0; k < hold && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&done[k], hipEventDisableTiming);
  for (int64_t off = 0; off < n && e == hipSuccess; off += hold * B) {
    const int64_t frames = std::min<int64_t>(hold * B, n - off), batches = (frames + B - 1) / B;
    for (int64_t k = 0; k < batches && e == hipSuccess; ++k) {
      float* x = in + k * B * ss;
      if (k < 2) {
        const int64_t cnt = k ? frames - B : std::min<int64_t>(B, frames);
        e = hipMemcpyAsync(x, inputs + (off + k * B) * ss, (size_t)cnt * ss * sizeof(float), hipMemcpyHostToDevice, cs);
        if (e == hipSuccess && k == (batches > 1) && frames < batches * B)
          e = hipMemsetAsync(in + frames * ss, 0, (size_t)(batches * B - frames) * ss * sizeof(float), cs);
        if (e == hipSuccess) e = hipEventRecord(came[k], cs);
        if (e == hipSuccess) e = hipStreamWaitEvent(s, came[k], 0);
        if (e != hipSuccess) break;
      }
      if (raw) {
        float* part = h->n.partial;  // scratch of the gradients
        hipLaunchKernelGGL(k_prep_max, dim3(PREP_PARTS, B), dim3(256), 0, s, x, ss, part);
        hipLaunchKernelGGL(k_prep_amplitudes, dim3(PREP_PARTS, B), dim3(256), 0, s, x, ss, part, h->n.x);
      } else
        hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((B * ss + 255) / 256)), dim3(256), 0, s, x, h->n.x, (long)(B * ss));
      h->n.out = res + k * B * 2 * ss;
      e = nn_forward(h->n);
      h->n.out = own;
      if (e == hipSuccess) e = hipEventRecord(done[k], s);
    }
    if (e == hipSuccess)
      e = copy_to_host(outputs + off * 2 * ss, res, (size_t)frames * 2 * ss * sizeof(float), h->device, cs, done,
                       (size_t)B * 2 * ss * sizeof(float));
  }
  hipStreamSynchronize(s);
  hipStreamSynchronize(cs);
  for (hipEvent_t ev : came)
    if (ev) hipEventDestroy(ev);
  for (hipEvent_t ev : done)
    if (ev) hipEventDestroy(ev);
  NCHK(h, e);
  return PTYK_OK;
}

int ptyk_net_predict(ptyk_net* h, const float* inputs, int64_t n, float* outputs) {
  return net_predict(h, inputs, n, outputs, false);
}

int ptyk_net_predict_amplitudes(ptyk_net* h, const float* amplitudes, int64_t n, float* outputs) {
  return net_predict(h, amplitudes, n, outputs, true);
}

// Loss and parameter gradient of one batch (host inputs batch x s x s, targets batch x 2 x s x s);
// for gradient checks.
int ptyk_net_gradient(ptyk_net* h, const float* inputs, const float* targets, double* loss, float* grad) {
  if (!h || !inputs || !targets || !loss || !grad) return PTYK_EINVAL;
  hipSetDevice(h->device);
  const long ss = (long)h->n.s * h->n.s;
  const int B = h->n.batch;
  float* stage = nullptr;
  NCHK(h, hipMalloc((void**)&stage, (size_t)B * 2 * ss * sizeof(float)));
  hipError_t e = hipMemcpyAsync(stage, inputs, (size_t)B * ss * sizeof(float), hipMemcpyHostToDevice, h->n.stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((B * ss + 255) / 256)), dim3(256), 0, h->n.stream, stage,
                       h->n.x, (long)(B * ss));
    e = hipStreamSynchronize(h->n.stream);
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(stage, targets, (size_t)B * 2 * ss * sizeof(float), hipMemcpyHostToDevice, h->n.stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_to_bf, dim3((unsigned)((B * 2 * ss + 255) / 256)), dim3(256), 0, h->n.stream, stage,
                       h->n.target, (long)(B * 2 * ss));
    e = nn_forward(h->n);
  }
  int np = 0;
  if (e == hipSuccess) e = nn_loss(h->n, true, &np);
  if (e == hipSuccess) e = nn_backward(h->n);
  if (e == hipSuccess) e = hipStreamSynchronize(h->n.stream);
  hipFree(stage);
  NCHK(h, e);
  int r = net_loss_value(h, np, loss);
  if (r) return r;
  NCHK(h, hipMemcpyAsync(grad, h->n.g, h->n.nparam * sizeof(float), hipMemcpyDeviceToHost, h->n.stream));
  NCHK(h, hipStreamSynchronize(h->n.stream));
  return PTYK_OK;
}

}  // extern "C"
