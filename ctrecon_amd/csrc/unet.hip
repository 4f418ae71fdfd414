// Kernels of the learned warm-start network: a 3-level 3-D U-Net with BF16
// activations and weights, FP32 accumulation on the matrix cores (MFMA), FP32 master
// weights and Adam.
//
// Tensors are channels-last over the volume grid (Y, X, Z), z fastest, the layout of
// the reconstruction volume: element (v, c) of a tensor with channel stride cs is at
// v * cs + c, v = (y * X + x) * Z + z.  A channel slice of a wider tensor (the skip
// half of a concatenation) is addressed by offsetting the base pointer.
//
// 3x3x3 convolution ("same", zero padding) as an implicit GEMM:
//   out[v][co] = sum_{tap, ci} in[v + off(tap)][ci] * W[tap][co][ci] + bias[co]
// M = voxels, N = output channels, K = 27 * Cin flattened as k = tap * Cin + ci.
// One wave computes 32 voxels x Cout with v_mfma_f32_16x16x32_bf16.  Operand layout of
// that instruction (lane l, j < 8, r < 4): A[l % 16][8 (l / 16) + j],
// B[8 (l / 16) + j][l % 16], D[4 (l / 16) + r][l % 16].
// The backward-data pass is the same convolution of the output gradient with the
// flipped, channel-transposed weights Wb[tap][ci][co] = W[26 - tap][co][ci].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device_common.hpp"
#include "unet_internal.hpp"

namespace ctr {
namespace unet {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 zero8() {
  return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
}

__device__ __forceinline__ float bf(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Block-wide FP64 sum of one value per thread into out[blockIdx.x].
__device__ __forceinline__ void block_sum(double a, double* out) {
  __shared__ double red[4];
  for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ---------------------------------------------------------------------------
// Convolution forward (and backward-data) with its input staged in LDS.
//
// A workgroup of WY x WX waves computes a box of output voxels, each wave 2 x LX lines (y, x)
// of 16 voxels along z and 16 NB output channels (blockIdx.y: the channel block); the box's
// input halo, one voxel wider on every side with zeros outside the grid, is staged CC
// channels at a time (CC = 16; 8 for the network's input), 2 CC bytes per voxel without
// padding, so that a wave's 16-byte reads of 16 neighbouring voxels are one contiguous run.
// K runs over the channel chunks, and within a chunk over k = tap * CC + c, 32 to an MFMA:
// the taps of a step differ by one of three fixed offsets, so all LDS reads of a chunk are
// immediate offsets from three addresses.  Weights are the first MFMA operand: a lane then
// holds four consecutive channels of one voxel and stores them as 8 bytes.
// Every K step adds the same 32 products in the same order whatever the box, so results do
// not depend on the configuration.
//
// Inputs: channels [0, ca) from a BF16 tensor, the rest read from the half-resolution tensor
// `up` (the decoder's nearest upsampling, never written out); or (CC = 8) the two FP32
// volumes of the network's input, scaled and rounded here.  Epilogues: bias and ReLU; also
// the 2x2x2 mean; only the 1x1x1 head; or the ReLU mask of a backward pass.
//
// 512 x 512 x 256: the ten layers take 10.5 ms (gathers of 16-byte operands from memory with
// separate pooling, upsampling, concatenation and head passes: 27.4 ms).  Full-resolution
// layers move 3 to 5 TB/s through HBM (16 -> 16 channels and pooling: 1.55 ms, 6 GB), with the
// matrix units busy 0.2 to 0.42 of the time and the texture unit returning data 0.85 to 0.93.
// ---------------------------------------------------------------------------
constexpr int kTZ = 16, kHZ = kTZ + 2;

enum Epi { kStore = 0, kPool = 1, kHead = 2, kGate = 3 };

struct ConvK {
  ConvIn in;
  const uint16_t* W;
  const float* bias;
  int Cin, Cout;
  ConvOut out;
  Grid3 g;
  int tiles_x, tiles_z, zrun;  // zrun: boxes along z per workgroup
};

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): constant indices keep
// register arrays in registers.
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// Where a convolution reads its input: one BF16 tensor; a tensor and the upsampled coarser
// one; or two FP32 volumes.
enum Src { kOne = 0, kUp = 1, kPair = 2 };

// One workgroup's share of a box's halo: thread t holds 16-byte unit t % (18 U) of lines
// t / (18 U), + LPP, ...; the units of the next stage (channel chunk or box along z) load into
// registers while the current one is in use.  Offsets are bytes from one voxel before the
// tensor's line (y0 - 1, 0), fixed for the workgroup (a stage adds a uniform offset); voxels
// outside the grid have an offset that the buffer's range check rejects, which reads zeros.
// FAR: the box's lines span 2 GiB or more, and the addresses are computed per load in 64 bits.
template <int CC, int NT, int HY, int HX, int SRC, bool FAR>
struct HaloLoad {
  static constexpr int U = CC / 8, kUnits = kHZ * U, LPP = NT / kUnits;
  static constexpr int kIt = (HY * HX + LPP - 1) / LPP;
  const void *pa, *pb;  // uniform bases
  uint32_t off[kIt], offb[SRC == kUp ? kIt : 1];
  uint4 v[kIt];
  int hz, y0, x0;

  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, 0x7fffffff,
                                             0x00020000);
  }
  __device__ __forceinline__ HaloLoad(const ConvIn& in, const Grid3& g, int y0_, int x0_)
      : y0(y0_), x0(x0_) {
    const int l0 = threadIdx.x / kUnits, u = threadIdx.x - l0 * kUnits;
    hz = u / U;
    if constexpr (FAR) return;
    const int c = 8 * (u - hz * U);
    const long long line = (long long)(y0 - 1) * g.X;
    const int yh = (y0 - 1) >> 1, Xh = g.X >> 1, Zh = g.Z >> 1;
    if constexpr (SRC == kPair) {
      pa = in.fx + (line * g.Z - 1);
      pb = in.fd + (line * g.Z - 1);
    } else {
      pa = in.a + (line * g.Z - 1) * in.cs_a;
      if constexpr (SRC == kUp) pb = in.up + ((long long)yh * Xh * Zh - 1) * in.cs_up;
    }
    static_for<kIt>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const int l = l0 + i * LPP, hy = l / HX, hx = l - hy * HX;
      const int yy = y0 - 1 + hy, xx = x0 - 1 + hx;
      const bool ok = l0 < LPP && l < HY * HX && (unsigned)yy < (unsigned)g.Y &&
                      (unsigned)xx < (unsigned)g.X;
      // z relative to one voxel before the box: hz; its coarse voxel (hz - 1) >> 1
      const int e = (hy * g.X + xx) * g.Z + hz;
      if constexpr (SRC == kPair) off[i] = ok ? (uint32_t)e * 4u : ~0u;
      else off[i] = ok ? (uint32_t)(e * in.cs_a + c) * 2u : ~0u;
      if constexpr (SRC == kUp) {
        const int eb = (((yy >> 1) - yh) * Xh + (xx >> 1)) * Zh + ((hz + 1) >> 1);
        offb[i] = ok ? (uint32_t)(eb * in.cs_up + c) * 2u : ~0u;
      }
    });
  }
  __device__ __forceinline__ void load(const ConvIn& in, const Grid3& g, int z0, int c0) {
    const bool zok = (unsigned)(z0 - 1 + hz) < (unsigned)g.Z;
    const bool up = SRC == kUp && c0 >= in.ca;
    if constexpr (FAR) {
      const int l0 = threadIdx.x / kUnits, c = 8 * (threadIdx.x % U), zz = z0 - 1 + hz;
      static_for<kIt>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int l = l0 + i * LPP, yy = y0 - 1 + l / HX, xx = x0 - 1 + l % HX;
        v[i] = make_uint4(0, 0, 0, 0);
        if (l0 < LPP && l < HY * HX && (unsigned)yy < (unsigned)g.Y &&
            (unsigned)xx < (unsigned)g.X && zok) {
          const long long e = ((long long)yy * g.X + xx) * g.Z + zz;
          const long long eh =
              ((long long)(yy >> 1) * (g.X >> 1) + (xx >> 1)) * (g.Z >> 1) + (zz >> 1);
          if constexpr (SRC == kPair)
            v[i] = make_uint4(__float_as_uint(in.fx[e]), __float_as_uint(in.fd[e]), 0, 0);
          else
            v[i] = *(const uint4*)(up ? in.up + eh * in.cs_up + c0 - in.ca + c
                                      : in.a + e * in.cs_a + c0 + c);
        }
      });
      return;
    }
    const int so = SRC == kPair ? z0 * 4
                   : up         ? ((z0 >> 1) * in.cs_up + c0 - in.ca) * 2
                                : (z0 * in.cs_a + c0) * 2;
    const __amdgpu_buffer_rsrc_t r = buf(up ? pb : pa);
    if constexpr (SRC == kPair) {
      const __amdgpu_buffer_rsrc_t r2 = buf(pb);
      static_for<kIt>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const uint32_t o = zok ? off[i] : ~0u;
        v[i] = make_uint4(__builtin_amdgcn_raw_buffer_load_b32(r, o, so, 0),
                          __builtin_amdgcn_raw_buffer_load_b32(r2, o, so, 0), 0, 0);
      });
    } else {
      static_for<kIt>([&](auto I) {
        constexpr int i = decltype(I)::value;
        uint32_t o = off[i];
        if constexpr (SRC == kUp) {
          const uint32_t ob = offb[i];  // (a value: choosing between the arrays' elements by
          o = up ? ob : o;              //  address would put both in scratch)
        }
        v[i] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(r, zok ? o : ~0u, so, 0));
      });
    }
  }
  __device__ __forceinline__ void store(char* halo, const ConvIn& in) {
    if (threadIdx.x >= LPP * kUnits) return;
    char* p = halo + threadIdx.x * 16;
    static_for<kIt>([&](auto I) {
      constexpr int i = decltype(I)::value;
      uint4 o = v[i];
      if constexpr (SRC == kPair)
        o = make_uint4((uint32_t)to_bf16(__uint_as_float(o.x) * in.s0) |
                           (uint32_t)to_bf16(__uint_as_float(o.y) * in.s1) << 16,
                       0, 0, 0);
      if (i + 1 < kIt || threadIdx.x + i * (LPP * kUnits) < HY * HX * kUnits)
        *(uint4*)(p + i * (LPP * kUnits * 16)) = o;
    });
  }
};

// The value of the neighbouring lane (lane ^ 1).
__device__ __forceinline__ uint32_t lane_xor1(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
}

template <int NB, int CC, int WY, int WX, int LX, int SRC, int EPI, bool FAR>
__global__ __launch_bounds__(64 * WY * WX, NB == 1 ? 4 : 2) void conv3_kernel(ConvK P) {
  constexpr int NT = 64 * WY * WX, LY = 2;
  constexpr int TY = WY * LY, TX = WX * LX, HY = TY + 2, HX = TX + 2;
  constexpr int VB = 2 * CC;  // bytes per staged voxel
  constexpr int KS = (27 * CC + 31) / 32;
  __shared__ __align__(16) char halo[HY * HX * kHZ * VB];
  const Grid3 g = P.g;
  const int lane = threadIdx.x & 63, row = lane & 15, grp = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int t = xcd_logical_block(blockIdx.x, gridDim.x);
  const int nzr = (P.tiles_z + P.zrun - 1) / P.zrun;
  const int tz0 = (t % nzr) * P.zrun, tz1 = min(tz0 + P.zrun, P.tiles_z);
  t /= nzr;
  const int tx = t % P.tiles_x, ty = t / P.tiles_x;
  const int y0 = ty * TY, x0 = tx * TX;
  const int co0 = blockIdx.y * 16 * NB;  // first output channel
  const int wy = (wv / WX) * LY, wx = (wv % WX) * LX;
  f32x4 acc[LY][LX][NB];
  const char* hw = halo + ((wy * HX + wx) * kHZ + row) * VB;  // tap 0 of the wave's first line
  // weights: the lane's channel row and K offset (in bytes)
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(P.W), (short)0, 27 * P.Cin * P.Cout * 2, 0x00020000);
  const uint32_t wlane =
      CC == 16 ? (uint32_t)((((grp >> 1) * P.Cout + co0 + row) * P.Cin + (grp & 1) * 8) * 2)
               : (uint32_t)((grp * P.Cout + co0 + row) * P.Cin * 2);
  HaloLoad<CC, NT, HY, HX, SRC, FAR> next(P.in, g, y0, x0);
  next.load(P.in, g, tz0 * kTZ, 0);
  for (int tz = tz0; tz < tz1; ++tz) {
    const int z0 = tz * kTZ;
#pragma unroll
    for (int a = 0; a < LY; ++a)
#pragma unroll
      for (int b = 0; b < LX; ++b)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[a][b][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < P.Cin; c0 += CC) {
      __syncthreads();
      next.store(halo, P.in);
      __syncthreads();
      if (c0 + CC < P.Cin) next.load(P.in, g, z0, c0 + CC);
      else if (tz + 1 < tz1) next.load(P.in, g, z0 + kTZ, 0);
      // voxel offset of a tap in the halo
      auto tap_off = [](int tap) constexpr {
        return ((tap / 9) * HX + (tap / 3) % 3) * kHZ + tap % 3;
      };
      // weights of step i: a step ahead of their use, and no further (the scheduler would
      // otherwise hold all steps' weights in registers)
      auto weights = [&](int i, bf16x8(&w)[NB]) {
        // CC = 16: lanes 0-31 the even tap, lanes 32-63 the odd one; CC = 8: a tap per group
        const int tap = CC == 16 ? 2 * i : 4 * i;
        const bool last = i == KS - 1;
        const bool pad = last && (CC == 16 ? grp >> 1 : grp == 3);  // no such tap: zeros
        const int so = (tap * P.Cout * P.Cin + c0) * 2;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const uint4 q = __builtin_bit_cast(
              uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, last && pad ? ~0u : wlane,
                                                           so + nb * 32 * P.Cin, 0));
          w[nb] = __builtin_bit_cast(bf16x8, q);
        }
      };
      // the wave's lines at an LDS address; a padding tap's values are zeros too
      auto step = [&](const char* h, const bf16x8(&w)[NB], bool last, bool pad) {
#pragma unroll
        for (int a = 0; a < LY; ++a)
#pragma unroll
          for (int b = 0; b < LX; ++b) {
            bf16x8 v = __builtin_bit_cast(bf16x8, *(const uint4*)(h + (a * HX + b) * kHZ * VB));
            if (last) v = pad ? zero8() : v;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[a][b][nb] = mfma(w[nb], v, acc[a][b][nb]);
          }
      };
      bf16x8 wt[2][NB];
      weights(0, wt[0]);
      // CC = 16: the odd tap of a step lies one voxel, one line less two voxels, or two lines
      // less two voxels further on
      const int odd = grp >> 1;
      const char* hc = hw + (CC == 16 ? (grp & 1) * 16 : 0);
      const char* ha = hc + odd * VB;
      const char* hb = hc + odd * (kHZ - 2) * VB;
      const char* hd = hc + odd * ((HX - 2) * kHZ - 2) * VB;
      static_for<KS>([&](auto I) {
        constexpr int i = decltype(I)::value;
        constexpr bool last = i == KS - 1;
        if constexpr (!last) weights(i + 1, wt[(i + 1) & 1]);
        if constexpr (CC == 16) {
          constexpr int te = 2 * i;
          const int d = last ? 0 : tap_off(te + 1) - tap_off(te);
          const char* h = last ? hc : (d == 1 ? ha : (d == kHZ - 2 ? hb : hd));
          step(h + tap_off(te) * VB, wt[i & 1], last, last && odd);
        } else {
          step(hw + tap_off(min(4 * i + grp, 26)) * VB, wt[i & 1], last, last && grp == 3);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    const int zz = z0 + row;
    const bool zok = zz < g.Z;
    // bias, ReLU and rounding: four channels of one voxel per lane
    uint2 o[LY][LX][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int co = co0 + 16 * nb + 4 * grp;
      float b4[4] = {0.f, 0.f, 0.f, 0.f};
      if (P.bias) {
#pragma unroll
        for (int r = 0; r < 4; ++r) b4[r] = P.bias[co + r];
      }
#pragma unroll
      for (int a = 0; a < LY; ++a)
#pragma unroll
        for (int b = 0; b < LX; ++b) {
          uint32_t h[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float val = acc[a][b][nb][r] + b4[r];
            if (P.out.relu) val = fmaxf(val, 0.f);
            h[r] = to_bf16(val);
          }
          o[a][b][nb] = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
        }
    }
    if constexpr (EPI == kHead) {
      // h = sum_c w[c] d[c] + b in channel order, 16 channels: the chain passes through the four
      // lane groups of a voxel
      const float* hwt = P.out.head;
      const float w0 = hwt[4 * grp], w1 = hwt[4 * grp + 1], w2 = hwt[4 * grp + 2],
                  w3 = hwt[4 * grp + 3], hb = hwt[16];
#pragma unroll
      for (int a = 0; a < LY; ++a)
#pragma unroll
        for (int b = 0; b < LX; ++b) {
          const uint2 q = o[a][b][0];
          const float c0 = bf((uint16_t)q.x), c1 = bf((uint16_t)(q.x >> 16)),
                      c2 = bf((uint16_t)q.y), c3 = bf((uint16_t)(q.y >> 16));
          float sum = hb;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float in = k == 0 ? hb : __shfl_up(sum, 16, 64);
            sum = fmaf(w3, c3, fmaf(w2, c2, fmaf(w1, c1, fmaf(w0, c0, in))));
          }
          const int yy = y0 + wy + a, xx = x0 + wx + b;
          if (grp == 3 && zok && yy < g.Y && xx < g.X)
            P.out.h[((long long)yy * g.X + xx) * g.Z + zz] = sum * P.out.hscale;
        }
      continue;
    }
#pragma unroll
    for (int a = 0; a < LY; ++a)
#pragma unroll
      for (int b = 0; b < LX; ++b) {
        const int yy = y0 + wy + a, xx = x0 + wx + b;
        if (!zok || yy >= g.Y || xx >= g.X) continue;
        const long long v = ((long long)yy * g.X + xx) * g.Z + zz;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int co = co0 + 16 * nb + 4 * grp;
          uint2 q = o[a][b][nb];
          if constexpr (EPI == kGate) {
            // ReLU backward: the gradient where the forward output is positive
            const uint2 y = *(const uint2*)(P.out.gate + v * P.out.cs_gate + co);
            auto keep = [](uint32_t y2, uint32_t q2) {
              const uint32_t lo = bf((uint16_t)y2) > 0.f ? q2 & 0xffffu : 0u;
              const uint32_t hi = bf((uint16_t)(y2 >> 16)) > 0.f ? q2 & 0xffff0000u : 0u;
              return lo | hi;
            };
            q = make_uint2(keep(y.x, q.x), keep(y.y, q.y));
          }
          *(uint2*)(P.out.out + v * P.out.cs_out + co) = q;
        }
      }
    if constexpr (EPI == kPool) {
      // mean of the 2x2x2 children in their order (y, x, z): lines of this wave, z neighbours
      // in the neighbouring lane
      const int zp = zz >> 1;
#pragma unroll
      for (int b = 0; b < LX; b += 2)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint2 q = o[k >> 1][b + (k & 1)][nb];
            const uint2 n = make_uint2(lane_xor1(q.x), lane_xor1(q.y));
            const uint32_t own[2] = {q.x, q.y}, nxt[2] = {n.x, n.y};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              sum[r] += bf((uint16_t)(own[r >> 1] >> (16 * (r & 1))));
              sum[r] += bf((uint16_t)(nxt[r >> 1] >> (16 * (r & 1))));
            }
          }
          const int yy = y0 + wy, xx = x0 + wx + b;
          if ((row & 1) == 0 && zok && yy < g.Y && xx < g.X) {
            const long long vp =
                ((long long)(yy >> 1) * (g.X >> 1) + (xx >> 1)) * (g.Z >> 1) + zp;
            uint32_t h[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = to_bf16(0.125f * sum[r]);
            *(uint2*)(P.out.pool + vp * P.out.cs_pool + co0 + 16 * nb + 4 * grp) =
                make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
          }
        }
    }
  }
}

// ---------------------------------------------------------------------------
// Weight gradient: part[s][tap][co][ci] = sum over the voxels of workgroup s of
// dY[v][co] * X[v + off(tap)][ci], for 16 NBO output and 16 input channels (blockIdx.y), and
// for the first input channels bpart[s][co] = sum dY[v][co].
//
// MFMA with rows co, columns ci and K = 32 voxels, two z lines of 16.  A workgroup walks
// boxes of 4 x 4 x 16 voxels: the gradient and the input's halo are staged channels-last in
// LDS, once for all 27 taps, and read as K fragments by transposing LDS reads (each group of
// 16 lanes reads four voxels' 16 channels, and lane c receives channel c of the four); the
// four waves take seven taps each (the last slot of the fourth the sum of dY).  One partial
// sum per workgroup, added in fixed order by reduce_splits_kernel.
// 128 x 128 x 64, 16 x 16 channels: a gather of 16-bit values per tap from memory took
// 590 us; this form 50 us (MFMA time 6 us): every tap reads its fragments from LDS again.
// ---------------------------------------------------------------------------
struct WgradK {
  ConvIn X;
  int Cin;
  const uint16_t* dY;
  int cs_dy, Cout;
  Grid3 g;
  int tiles_x, tiles_z, boxes;
  float *part, *bpart;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
// Two transposing reads: channel (lane % 16) of the eight voxels of 32-byte rows at `p`,
// p being the lane's own address (row lane % 16 / 4, 8-byte unit lane % 4).
__device__ __forceinline__ bf16x8 load8_tr(const char* p) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * 32));
  return __builtin_bit_cast(bf16x8,
                            __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int NBO>
__global__ __launch_bounds__(256) void wgrad_kernel(WgradK P) {
  constexpr int HY = 6, HX = 6, kTaps = 7;
  __shared__ __align__(16) char halo[HY * HX * kHZ * 32];
  __shared__ __align__(16) char grad[NBO][16 * kTZ * 32];
  const Grid3 g = P.g;
  const int lane = threadIdx.x & 63, row = lane & 15, grp = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nci = (P.Cin + 15) / 16;
  const int ci0 = ((int)blockIdx.y % nci) * 16, co0 = ((int)blockIdx.y / nci) * 16 * NBO;
  const int uin = P.Cin == 8 ? 1 : 2;  // 16-byte units of a staged voxel that hold channels
  f32x4 acc[kTaps][NBO], accb[NBO];
#pragma unroll
  for (int i = 0; i < NBO; ++i) {
    accb[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kTaps; ++t) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the lane's part of a transposing read: line (grp / 2) of the pair, z half grp % 2
  const int zr = (grp & 1) * 8 + (row >> 2), unit = (row & 3) * 8;
  const char* ga = grad[0] + ((grp >> 1) * kTZ + zr) * 32 + unit;
  const char* hx[kTaps];
#pragma unroll
  for (int t = 0; t < kTaps; ++t) {
    const int tap = min(wv * kTaps + t, 26);
    hx[t] = halo + (((tap / 9) * HX + (tap / 3) % 3 + (grp >> 1)) * kHZ + tap % 3 + zr) * 32 + unit;
  }
  const bf16x8 ones = __builtin_bit_cast(
      bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
  for (int box = blockIdx.x; box < P.boxes; box += gridDim.x) {
    int t = box;
    const int tz = t % P.tiles_z;
    t /= P.tiles_z;
    const int x0 = (t % P.tiles_x) * 4, y0 = (t / P.tiles_x) * 4, z0 = tz * kTZ;
    __syncthreads();
    for (int i = threadIdx.x; i < HY * HX * kHZ * 2; i += 256) {
      const int hv = i >> 1, u = i & 1;
      const int line = hv / kHZ, hz = hv - line * kHZ;
      const int hy = line / HX, hxx = line - hy * HX;
      const int yy = y0 - 1 + hy, xx = x0 - 1 + hxx, zz = z0 - 1 + hz;
      uint4 val = make_uint4(0, 0, 0, 0);
      if (u < uin && yy >= 0 && yy < g.Y && xx >= 0 && xx < g.X && zz >= 0 && zz < g.Z) {
        if (ci0 < P.X.ca) {
          const long long v = ((long long)yy * g.X + xx) * g.Z + zz;
          val = *(const uint4*)(P.X.a + v * P.X.cs_a + ci0 + 8 * u);
        } else {
          const long long vc =
              ((long long)(yy >> 1) * (g.X >> 1) + (xx >> 1)) * (g.Z >> 1) + (zz >> 1);
          val = *(const uint4*)(P.X.up + vc * P.X.cs_up + (ci0 - P.X.ca) + 8 * u);
        }
      }
      *(uint4*)(halo + i * 16) = val;
    }
#pragma unroll
    for (int nb = 0; nb < NBO; ++nb)
      for (int i = threadIdx.x; i < 16 * kTZ * 2; i += 256) {
        const int v = i >> 1, u = i & 1, line = v >> 4;
        const int yy = y0 + (line >> 2), xx = x0 + (line & 3), zz = z0 + (v & 15);
        uint4 val = make_uint4(0, 0, 0, 0);
        if (yy < g.Y && xx < g.X && zz < g.Z)
          val = *(const uint4*)(P.dY + (((long long)yy * g.X + xx) * g.Z + zz) * P.cs_dy + co0 +
                                16 * nb + 8 * u);
        *(uint4*)(grad[nb] + i * 16) = val;
      }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) {  // lines 2 s and 2 s + 1 of the box
      bf16x8 a[NBO];
#pragma unroll
      for (int i = 0; i < NBO; ++i)
        a[i] = load8_tr(ga + i * (16 * kTZ * 32) + s * (2 * kTZ * 32));
#pragma unroll
      for (int t = 0; t < kTaps; ++t) {
        const bf16x8 b = load8_tr(hx[t] + ((s >> 1) * HX + (s & 1) * 2) * kHZ * 32);
#pragma unroll
        for (int i = 0; i < NBO; ++i) acc[t][i] = mfma(a[i], b, acc[t][i]);
      }
      if (wv == 3) {
#pragma unroll
        for (int i = 0; i < NBO; ++i) accb[i] = mfma(a[i], ones, accb[i]);
      }
    }
  }
  const int ci = ci0 + row;
#pragma unroll
  for (int t = 0; t < kTaps; ++t) {
    const int tap = wv * kTaps + t;
    if (tap >= 27 || ci >= P.Cin) continue;
    float* o = P.part + ((size_t)blockIdx.x * 27 + tap) * P.Cout * P.Cin;
#pragma unroll
    for (int i = 0; i < NBO; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[(size_t)(co0 + 16 * i + 4 * grp + r) * P.Cin + ci] = acc[t][i][r];
  }
  if (wv == 3 && ci0 == 0 && row == 0) {
#pragma unroll
    for (int i = 0; i < NBO; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        P.bpart[(size_t)blockIdx.x * P.Cout + co0 + 16 * i + 4 * grp + r] = accb[i][r];
  }
}

// out[i] = sum_s part[s * n + i], then the same for the second array (fixed order): 32
// elements to a workgroup, eight threads each over every eighth split.
__global__ __launch_bounds__(256) void reduce_splits_kernel(const float* __restrict__ part,
                                                            size_t n, float* __restrict__ out,
                                                            const float* __restrict__ part2,
                                                            size_t n2, float* __restrict__ out2,
                                                            int nsplit) {
  __shared__ float red[8][32];
  const int e = threadIdx.x & 31, l = threadIdx.x >> 5;
  const size_t nb = (n + 31) / 32;
  const bool second = blockIdx.x >= nb;
  const float* p = second ? part2 : part;
  const size_t m = second ? n2 : n;
  const size_t i = (second ? blockIdx.x - nb : blockIdx.x) * 32 + e;
  float a = 0.f;
  if (i < m) {
#pragma unroll 8
    for (int s = l; s < nsplit; s += 8) a += p[(size_t)s * m + i];
  }
  red[l][e] = a;
  __syncthreads();
  if (l == 0 && i < m) {
    float t = red[0][e];
#pragma unroll
    for (int k = 1; k < 8; ++k) t += red[k][e];
    (second ? out2 : out)[i] = t;
  }
}

// Master weights [27][Cout][Cin] (FP32) -> forward BF16 copy (same layout) and the
// backward-data copy Wb[tap][ci][co] = W[26 - tap][co][ci].
__global__ void convert_weights_kernel(const float* __restrict__ Wm, int Cin, int Cout,
                                       uint16_t* __restrict__ Wf, uint16_t* __restrict__ Wb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 27 * Cin * Cout) return;
  const int tap = i / (Cin * Cout), rem = i - tap * Cin * Cout;
  const int co = rem / Cin, ci = rem - co * Cin;
  const uint16_t h = to_bf16(Wm[i]);
  Wf[i] = h;
  Wb[((size_t)(26 - tap) * Cin + ci) * Cout + co] = h;
}

// Network input: channels (x * s0, d * s1, 0 ...) of an 8-channel tensor.
__global__ void pack_input_kernel(const float* __restrict__ x, const float* __restrict__ d,
                                  float s0, float s1, long long V, uint16_t* __restrict__ out) {
  for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < V;
       v += (long long)gridDim.x * blockDim.x) {
    uint16_t h[8] = {to_bf16(x[v] * s0), to_bf16(d[v] * s1), 0, 0, 0, 0, 0, 0};
    *(uint4*)(out + v * 8) = __builtin_bit_cast(uint4, h);
  }
}

// Backward passes of the pooling and the upsampling with the ReLU mask that follows them,
// eight channels (16 bytes) per thread, a workgroup per (y, x) line of the grid written.
__device__ __forceinline__ uint4 gate8(const uint4& y, const uint4& v) {
  auto keep = [](uint32_t a, uint32_t b) {
    return (bf((uint16_t)a) > 0.f ? b & 0xffffu : 0u) |
           (bf((uint16_t)(a >> 16)) > 0.f ? b & 0xffff0000u : 0u);
  };
  return make_uint4(keep(y.x, v.x), keep(y.y, v.y), keep(y.z, v.z), keep(y.w, v.w));
}

// din[child][c] = (gate > 0) ? din[child][c] + dout[p][c] / 8 : 0 (gf: the fine grid).
__global__ __launch_bounds__(256) void pool_bwd_kernel(const uint16_t* __restrict__ dout,
                                                       int cs_out, int C, Grid3 gf,
                                                       uint16_t* __restrict__ din, int cs_in,
                                                       const uint16_t* __restrict__ gate,
                                                       int cs_gate) {
  const int U = C / 8;
  for (int line = blockIdx.x; line < gf.Y * gf.X; line += gridDim.x) {
    const int y = line / gf.X, x = line - y * gf.X;
    const long long pl = (long long)(y >> 1) * (gf.X >> 1) + (x >> 1);
    for (int i = threadIdx.x; i < gf.Z * U; i += 256) {
      const int z = i / U, c = (i - z * U) * 8;
      const long long v = (long long)line * gf.Z + z, p = pl * (gf.Z >> 1) + (z >> 1);
      uint16_t a[8], b[8];
      *(uint4*)a = *(const uint4*)(din + v * cs_in + c);
      *(uint4*)b = *(const uint4*)(dout + p * cs_out + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = to_bf16(bf(a[j]) + 0.125f * bf(b[j]));
      *(uint4*)(din + v * cs_in + c) =
          gate8(*(const uint4*)(gate + v * cs_gate + c), *(const uint4*)a);
    }
  }
}

// din[p][c] = (gate > 0) ? sum of dout over the 8 children : 0 (gf: the fine grid).
__global__ __launch_bounds__(256) void upsample_bwd_kernel(const uint16_t* __restrict__ dout,
                                                           int cs_out, int C, Grid3 gf,
                                                           uint16_t* __restrict__ din, int cs_in,
                                                           const uint16_t* __restrict__ gate,
                                                           int cs_gate) {
  const int Xc = gf.X / 2, Zc = gf.Z / 2, U = C / 8;
  for (int line = blockIdx.x; line < (gf.Y / 2) * Xc; line += gridDim.x) {
    const int y = line / Xc, x = line - y * Xc;
    for (int i = threadIdx.x; i < Zc * U; i += 256) {
      const int z = i / U, c = (i - z * U) * 8;
      const long long p = (long long)line * Zc + z;
      float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int o = 0; o < 8; ++o) {
        const long long vf =
            ((long long)(2 * y + (o >> 2)) * gf.X + 2 * x + ((o >> 1) & 1)) * gf.Z + 2 * z +
            (o & 1);
        uint16_t b[8];
        *(uint4*)b = *(const uint4*)(dout + vf * cs_out + c);
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] += bf(b[j]);
      }
      uint16_t a[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = to_bf16(s[j]);
      *(uint4*)(din + p * cs_in + c) =
          gate8(*(const uint4*)(gate + p * cs_gate + c), *(const uint4*)a);
    }
  }
}

// Head: h[v] = sum_c w[c] a[v][c] + b (FP32 output), 16 channels.
__global__ void head_kernel(const uint16_t* __restrict__ a, const float* __restrict__ wb,
                            long long V, float scale, float* __restrict__ h) {
  for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < V;
       v += (long long)gridDim.x * blockDim.x) {
    const uint4 q0 = *(const uint4*)(a + v * 16), q1 = *(const uint4*)(a + v * 16 + 8);
    const uint16_t* e0 = (const uint16_t*)&q0;
    const uint16_t* e1 = (const uint16_t*)&q1;
    float s = wb[16];
#pragma unroll
    for (int c = 0; c < 8; ++c) s = fmaf(wb[c], bf(e0[c]), s);
#pragma unroll
    for (int c = 0; c < 8; ++c) s = fmaf(wb[8 + c], bf(e1[c]), s);
    h[v] = s * scale;
  }
}

// Loss L = sum_v e_v^2 / (2 V) with e = h - t * tscale: dh = e / V, and part[block]
// the block's partial sum of e^2 (FP64).
__global__ __launch_bounds__(256) void mse_kernel(const float* __restrict__ h,
                                                  const float* __restrict__ t, float tscale,
                                                  long long V, float* __restrict__ dh,
                                                  double* __restrict__ part) {
  double s = 0.0;
  const float invV = 1.0f / (float)V;
  for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < V;
       v += (long long)gridDim.x * blockDim.x) {
    const float e = h[v] - t[v] * tscale;
    dh[v] = e * invV;
    s += (double)e * (double)e;
  }
  block_sum(s, part);
}

// Head backward with the ReLU of its input: da[v][c] = (a > 0) ? dh[v] w[c] : 0, and
// per-block partials of dw[c] = sum dh a[v][c] (c < 16) and db = sum dh.
__global__ __launch_bounds__(256) void head_bwd_kernel(const uint16_t* __restrict__ a,
                                                       const float* __restrict__ wb,
                                                       const float* __restrict__ dh, long long V,
                                                       uint16_t* __restrict__ da,
                                                       double* __restrict__ part) {
  double acc[17];
#pragma unroll
  for (int c = 0; c < 17; ++c) acc[c] = 0.0;
  for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < V;
       v += (long long)gridDim.x * blockDim.x) {
    const float g = dh[v];
    uint16_t out[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const float av = bf(a[v * 16 + c]);
      acc[c] += (double)g * av;
      out[c] = av > 0.f ? to_bf16(g * wb[c]) : (uint16_t)0;
    }
    acc[16] += g;
    uint16_t o0[8], o1[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      o0[c] = out[c];
      o1[c] = out[8 + c];
    }
    *(uint4*)(da + v * 16) = __builtin_bit_cast(uint4, o0);
    *(uint4*)(da + v * 16 + 8) = __builtin_bit_cast(uint4, o1);
  }
  __shared__ double red[17][4];
#pragma unroll
  for (int c = 0; c < 17; ++c) {
    double x = acc[c];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    if ((threadIdx.x & 63) == 0) red[c][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 17) {
    const int c = threadIdx.x;
    part[(size_t)blockIdx.x * 17 + c] = red[c][0] + red[c][1] + red[c][2] + red[c][3];
  }
}

// out[i] = sum over blocks b of part[b * n + i] (FP64 sum in fixed order, FP32 result), one
// workgroup per i.
__global__ __launch_bounds__(256) void reduce_dpart_kernel(const double* __restrict__ part,
                                                           int nb, int n,
                                                           float* __restrict__ out) {
  __shared__ double red[4];
  double s = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) s += part[(size_t)b * n + blockIdx.x];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (float)(red[0] + red[1] + red[2] + red[3]);
}

// Adam on FP32 master parameters.
__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, size_t n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

int grid1(long long n) {
  long long g = (n + 255) / 256;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

constexpr int kMaxLines = 1 << 20;  // workgroups of the line kernels

int check(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(CTR_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return CTR_OK;
}

}  // namespace

namespace {
template <int NB, int CC, int WY, int WX, int LX, bool FAR = false>
int conv3_launch(ConvK P, hipStream_t st) {
  constexpr int TY = 2 * WY, TX = LX * WX;
  P.tiles_x = (P.g.X + TX - 1) / TX;
  P.tiles_z = (P.g.Z + kTZ - 1) / kTZ;
  const long long lines = (long long)((P.g.Y + TY - 1) / TY) * P.tiles_x;
  // runs of up to four boxes along z (the next box loads while one is computed) while two
  // workgroups per CU remain for four rounds (512 x 512 x 256: 10.6 ms, 10.9 ms without runs)
  const int gy = P.Cout / (16 * NB);
  P.zrun = 1;
  while (P.zrun < 4 && lines * ((P.tiles_z + 2 * P.zrun - 1) / (2 * P.zrun)) * gy >= 2048)
    P.zrun *= 2;
  const long long tiles = lines * ((P.tiles_z + P.zrun - 1) / P.zrun);
  const dim3 grid((unsigned)tiles, (unsigned)gy), block(64 * WY * WX);
#define CV(SRC, EPI)                                                                       \
  do {                                                                                     \
    hipLaunchKernelGGL((conv3_kernel<NB, CC, WY, WX, LX, SRC, EPI, FAR>), grid, block, 0, st, \
                       P);                                                                 \
    return check("conv3_kernel");                                                          \
  } while (0)
  const ConvIn& in = P.in;
  const ConvOut& o = P.out;
  if constexpr (CC == 8) {
    if (!o.head && !o.pool && !o.gate && !in.up) {
      if (in.fx) CV(kPair, kStore);
      CV(kOne, kStore);
    }
  } else if (in.fx) {
    return fail(CTR_ERR_ARG, "conv3: the FP32 input has 8 channels");
  } else if (in.up) {
    if (!o.head && !o.pool && !o.gate) CV(kUp, kStore);
  } else if (o.head) {
    if constexpr (NB == 1) {
      if (P.Cout == 16) CV(kOne, kHead);
    }
  } else if (o.pool) {
    CV(kOne, kPool);
  } else if (o.gate) {
    CV(kOne, kGate);
  } else {
    CV(kOne, kStore);
  }
#undef CV
  return fail(CTR_ERR_UNSUPPORTED, "conv3: combination of input and output not instantiated");
}

template <int CC>
int conv3_shape(const ConvK& P, hipStream_t st) {
  const int NB = P.Cout / 16;
  // 32-bit byte offsets reach over a box's ten lines y
  if ((long long)P.g.X * P.g.Z * std::max({P.in.cs_a, P.in.cs_up, 2}) * 20 >= 0x7fffffffLL)
    return conv3_launch<1, CC, 2, 2, 2, true>(P, st);
  // boxes of 8 x 8 lines, 8 waves (1.8 halo voxels staged per output; 2.5 with 4 x 4 lines),
  // where they fill the chip twice; else boxes of 4 x 4 lines, one block of channels each.
  // 512 x 512 x 256, whole pass: 10.6 ms, 13.0 ms with 4 x 4 lines throughout; loss and gradient
  // at 128 x 128 x 64: 1.33 ms, 1.38 ms with 8 x 8 lines from 64 boxes on.
  const long long big = (long long)((P.g.Y + 7) / 8) * ((P.g.X + 7) / 8) * ((P.g.Z + 15) / 16);
  if (big * ((NB + 1) / 2) >= 512) {
    if constexpr (CC == 16) {
      if (NB % 2 == 0) return conv3_launch<2, CC, 4, 2, 4>(P, st);
    }
    return conv3_launch<1, CC, 4, 2, 4>(P, st);
  }
  return conv3_launch<1, CC, 2, 2, 2>(P, st);
}
}  // namespace

int conv3(const ConvIn& in, int Cin, const uint16_t* W, const float* bias, int Cout,
          const ConvOut& out, Grid3 g, hipStream_t st) {
  if (!(Cin == 8 || Cin % 16 == 0) || Cout % 16)
    return fail(CTR_ERR_ARG, "conv3: channel counts must be 8 or multiples of 16");
  if ((in.a && in.cs_a % 8) || (in.up && (in.cs_up % 8 || in.ca % 16)) ||
      (out.out && out.cs_out % 4) || (out.pool && out.cs_pool % 4) ||
      (out.gate && out.cs_gate % 4))
    return fail(CTR_ERR_ARG, "conv3: channel strides must be multiples of 8");
  ConvK P{in, W, bias, Cin, Cout, out, g, 0, 0, 1};
  return Cin == 8 ? conv3_shape<8>(P, st) : conv3_shape<16>(P, st);
}

int wgrad(const ConvIn& X, int Cin, const uint16_t* dY, int cs_dy, int Cout, Grid3 g,
          float* part, float* bpart, float* dW, float* db, hipStream_t st) {
  if (!(Cin == 8 || Cin % 16 == 0) || Cout % 16)
    return fail(CTR_ERR_ARG, "wgrad: channel counts must be 8 or multiples of 16");
  WgradK P{X, Cin, dY, cs_dy, Cout, g, 0, 0, 0, part, bpart};
  P.tiles_x = (g.X + 3) / 4;
  P.tiles_z = (g.Z + kTZ - 1) / kTZ;
  const long long boxes = (long long)((g.Y + 3) / 4) * P.tiles_x * P.tiles_z;
  if (boxes > 0x7fffffffLL) return fail(CTR_ERR_ARG, "wgrad: grid too large");
  P.boxes = (int)boxes;
  const int nbo = Cout % 32 == 0 ? 2 : 1;
  const int gy = ((Cin + 15) / 16) * (Cout / (16 * nbo));
  // about four workgroups per CU over all channel blocks (128 x 128 x 64, whole gradient:
  // 1.25 ms, 1.32 ms with two, whose staging then stands uncovered)
  const int ns = (int)std::max<long long>(1, std::min<long long>(boxes, kWgradBlocks / gy));
  const dim3 grid(ns, gy);
  if (nbo == 2) hipLaunchKernelGGL(wgrad_kernel<2>, grid, dim3(256), 0, st, P);
  else hipLaunchKernelGGL(wgrad_kernel<1>, grid, dim3(256), 0, st, P);
  int rc = check("wgrad_kernel");
  if (rc) return rc;
  const size_t n = (size_t)27 * Cout * Cin;
  hipLaunchKernelGGL(reduce_splits_kernel, dim3((unsigned)((n + 31) / 32 + (Cout + 31) / 32)),
                     dim3(256), 0, st, part, n, dW, bpart, (size_t)Cout, db, ns);
  return check("reduce_splits_kernel");
}

int convert_weights(const float* Wm, int Cin, int Cout, uint16_t* Wf, uint16_t* Wb,
                    hipStream_t st) {
  const int n = 27 * Cin * Cout;
  hipLaunchKernelGGL(convert_weights_kernel, dim3((n + 255) / 256), dim3(256), 0, st, Wm, Cin,
                     Cout, Wf, Wb);
  return check("convert_weights_kernel");
}

int pack_input(const float* x, const float* d, float s0, float s1, long long V, uint16_t* out,
               hipStream_t st) {
  hipLaunchKernelGGL(pack_input_kernel, dim3(grid1(V)), dim3(256), 0, st, x, d, s0, s1, V, out);
  return check("pack_input_kernel");
}

int pool_bwd(const uint16_t* dout, int cs_out, int C, Grid3 gf, uint16_t* din, int cs_in,
             const uint16_t* gate, int cs_gate, hipStream_t st) {
  hipLaunchKernelGGL(pool_bwd_kernel, dim3(std::min(gf.Y * gf.X, kMaxLines)), dim3(256), 0, st,
                     dout, cs_out, C, gf, din, cs_in, gate, cs_gate);
  return check("pool_bwd_kernel");
}

int upsample_bwd(const uint16_t* dout, int cs_out, int C, Grid3 gf, uint16_t* din, int cs_in,
                 const uint16_t* gate, int cs_gate, hipStream_t st) {
  hipLaunchKernelGGL(upsample_bwd_kernel, dim3(std::min((gf.Y / 2) * (gf.X / 2), kMaxLines)),
                     dim3(256), 0, st, dout, cs_out, C, gf, din, cs_in, gate, cs_gate);
  return check("upsample_bwd_kernel");
}

int head(const uint16_t* a, const float* wb, long long V, float scale, float* h, hipStream_t st) {
  hipLaunchKernelGGL(head_kernel, dim3(grid1(V)), dim3(256), 0, st, a, wb, V, scale, h);
  return check("head_kernel");
}

int mse(const float* h, const float* t, float tscale, long long V, float* dh, double* part,
        int nblocks, hipStream_t st) {
  hipLaunchKernelGGL(mse_kernel, dim3(nblocks), dim3(256), 0, st, h, t, tscale, V, dh, part);
  return check("mse_kernel");
}

int head_bwd(const uint16_t* a, const float* wb, const float* dh, long long V, uint16_t* da,
             double* part, int nblocks, float* dwb, hipStream_t st) {
  hipLaunchKernelGGL(head_bwd_kernel, dim3(nblocks), dim3(256), 0, st, a, wb, dh, V, da, part);
  int rc = check("head_bwd_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(reduce_dpart_kernel, dim3(17), dim3(256), 0, st, part, nblocks, 17, dwb);
  return check("reduce_dpart_kernel");
}

int adam(float* p, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2,
         float eps, int step, hipStream_t st) {
  const float c1 = 1.f / (1.f - powf(b1, (float)step));
  const float c2 = 1.f / (1.f - powf(b2, (float)step));
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, g, m, v,
                     n, lr, b1, b2, eps, c1, c2);
  return check("adam_kernel");
}

}  // namespace unet
}  // namespace ctr
