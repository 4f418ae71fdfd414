// Internal interface of the warm-start network kernels (unet.hip) used by the host
// driver (unet.cpp).  BF16 tensors are uint16_t arrays; see unet.hip for layouts.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "ctr_internal.hpp"

namespace ctr {
namespace unet {

struct Grid3 {
  int Y, X, Z;
};

// Input of a convolution: channels [0, ca) of the BF16 tensor a (channel stride cs_a), the
// rest from the half-resolution tensor up, upsampled to the nearest voxel; or, with Cin = 8,
// the channels (fx s0, fd s1, 0 ...) of two FP32 volumes.
struct ConvIn {
  const uint16_t* a = nullptr;
  int cs_a = 0, ca = 0;
  const uint16_t* up = nullptr;
  int cs_up = 0;
  const float *fx = nullptr, *fd = nullptr;
  float s0 = 0.f, s1 = 0.f;
};
inline ConvIn conv_in(const uint16_t* a, int cs) { return ConvIn{a, cs, 1 << 30}; }

// Output: out (channel stride cs_out) after an optional ReLU, masked by gate > 0 when set
// (ReLU backward); also its 2x2x2 means when pool is set; with head set, only
// h = hscale (sum_c head[c] out[c] + head[16]).
struct ConvOut {
  uint16_t* out = nullptr;
  int cs_out = 0, relu = 0;
  const uint16_t* gate = nullptr;
  int cs_gate = 0;
  uint16_t* pool = nullptr;
  int cs_pool = 0;
  const float* head = nullptr;
  float hscale = 1.f;
  float* h = nullptr;
};

int conv3(const ConvIn& in, int Cin, const uint16_t* W, const float* bias, int Cout,
          const ConvOut& out, Grid3 g, hipStream_t st);
// part: kWgradBlocks * 27 * 16 * 32 floats and bpart: kWgradBlocks * 64 floats of scratch
constexpr int kWgradBlocks = 1024;
int wgrad(const ConvIn& X, int Cin, const uint16_t* dY, int cs_dy, int Cout, Grid3 g,
          float* part, float* bpart, float* dW, float* db, hipStream_t st);
int convert_weights(const float* Wm, int Cin, int Cout, uint16_t* Wf, uint16_t* Wb,
                    hipStream_t st);
int pack_input(const float* x, const float* d, float s0, float s1, long long V, uint16_t* out,
               hipStream_t st);
// C a multiple of 8, strides multiples of 8; gate: ReLU mask of the tensor written
int pool_bwd(const uint16_t* dout, int cs_out, int C, Grid3 gf, uint16_t* din, int cs_in,
             const uint16_t* gate, int cs_gate, hipStream_t st);
int upsample_bwd(const uint16_t* dout, int cs_out, int C, Grid3 gf, uint16_t* din, int cs_in,
                 const uint16_t* gate, int cs_gate, hipStream_t st);
int head(const uint16_t* a, const float* wb, long long V, float scale, float* h, hipStream_t st);
int mse(const float* h, const float* t, float tscale, long long V, float* dh, double* part,
        int nblocks, hipStream_t st);
int head_bwd(const uint16_t* a, const float* wb, const float* dh, long long V, uint16_t* da,
             double* part, int nblocks, float* dwb, hipStream_t st);
int adam(float* p, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2,
         float eps, int step, hipStream_t st);

}  // namespace unet
}  // namespace ctr
