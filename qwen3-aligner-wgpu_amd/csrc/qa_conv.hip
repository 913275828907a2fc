// qa_conv.hip -- the first conv level of the audio tower's stem as a direct
// convolution: 3x3, stride 2, pad 1 over a single-channel input (the mel
// chunk), bias and erf GELU, one rounding per output (CpuConvStem::conv_block,
// src/audio_encoder.rs:376-447, c_in = 1; the GPU tower's im2col + gemm_conv +
// bias_gelu, src/audio_encoder_gpu.rs:1165-1201,1714-1794).  With one input
// channel the im2col row of an output pixel is 9 scattered values, which the
// implicit GEMM's 16-byte channel chunks cannot fetch.  The 9-tap dot
// products run on the matrix cores as a K = 16 product (taps 9..15 zero), with
// the bias as the accumulator's start: a wave multiplies 32 output pixels by
// the weights of 32 output channels per v_mfma_f32_32x32x16, every product of
// two 16-bit values exact in f32.  What is left on the VALU per output is the
// erf GELU (16 issue slots) and the rounding, and that bounds the kernel: over
// the 300-chunk stem (461 M outputs) about 0.2 ms of the 256 CUs' VALU issue
// at 2.2 GHz, more than the 922 MB it writes.
//
// A block takes 128 output pixels (32 per wave) x a group of channel tiles;
// each lane holds one pixel's taps as the MFMA's B fragment and, per channel
// tile, 16 of that pixel's outputs, which leave as two 16-byte stores after a
// swap between the two halves of the wave.  The weights come straight from
// global memory in the A fragment's layout (15 KB at 480 channels: a channel's
// 16 taps are one 32-byte row), one tile ahead; staging them in LDS as 9
// two-byte loads per channel cost every block ~8 us.
#include "qa_internal.h"

namespace qa {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <int DT>
__device__ __forceinline__ float widen(uint16_t h) {
  if constexpr (DT == QA_F16) return (float)__builtin_bit_cast(_Float16, h);
  else return __uint_as_float((uint32_t)h << 16);
}
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {  // RNE
  if constexpr (DT == QA_F16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

constexpr int kMaxCout = 1024;
constexpr int kPix = 128;  // output pixels per block

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int DT>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (DT == QA_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// MFMA lane layout (v_mfma_f32_32x32x16, A = 32 channels x 16 taps, B = 16
// taps x 32 pixels): lane (r, h) = (lane % 32, lane / 32) supplies taps
// 8h .. 8h + 7 of channel r (A) and of pixel r (B), and receives pixel r's
// outputs for channels 8g + 4h + {0..3}, g = 0..3.
template <int DT, bool GELU>
__global__ void __launch_bounds__(256) conv1_kernel(const Conv1Params p, int group_tiles) {
  __shared__ __attribute__((aligned(16))) float bs[kMaxCout];
  const int ct0 = (int)blockIdx.y * group_tiles;
  const int ct1 = min((p.c_out + 31) / 32, ct0 + group_tiles);
  for (int i = ct0 * 32 + threadIdx.x; i < ct1 * 32; i += 256)
    bs[i] = p.bias && i < p.c_out ? widen<DT>(p.bias[i]) : 0.f;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  // channel ct * 32 + r's taps 8h .. 8h + 7 (only tap 8 of the upper eight;
  // channels past the last repeat it, their outputs are not stored)
  auto weights = [&](int ct) {
    const int c = min(ct * 32 + r, p.c_out - 1);
    const u32x4 w = *reinterpret_cast<const u32x4*>(p.w + (int64_t)c * p.ldw + 8 * h);
    return h == 0 ? w : u32x4{w.x & 0xffffu, 0, 0, 0};
  };
  u32x4 aop = weights(ct0);
  const int64_t m = (int64_t)blockIdx.x * kPix + (threadIdx.x >> 6) * 32 + r;
  // this lane's taps 8h .. 8h + 7 of pixel m (zeros past tap 8, in the
  // padding and past the last pixel)
  uint32_t tv[4] = {0, 0, 0, 0};
  if (m < p.M) {
    const int plane = p.ho * p.wo;
    const int64_t b = m / plane;
    const int q = (int)(m - b * plane);
    const int ho = p.tmajor ? q % p.ho : q / p.wo;
    const int wo = p.tmajor ? q / p.ho : q % p.wo;
    const uint16_t* x = p.x + b * p.h * p.w_in;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = 8 * h + e;
      if (t < 9) {
        const int kh = t / 3, kw = t % 3;
        const int ih = 2 * ho + kh - 1, iw = 2 * wo + kw - 1;
        if (ih >= 0 && ih < p.h && iw >= 0 && iw < p.w_in)
          tv[e >> 1] |= (uint32_t)x[ih * p.w_in + iw] << (16 * (e & 1));
      }
    }
  }
  const u32x4 bop = {tv[0], tv[1], tv[2], tv[3]};
  __syncthreads();
  uint16_t* y = p.y + m * p.c_out;
  for (int ct = ct0; ct < ct1; ++ct) {
    f32x16 acc;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 b4 = *reinterpret_cast<const f32x4*>(bs + ct * 32 + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[4 * g + e] = b4[e];
    }
    acc = mfma<DT>(aop, bop, acc);
    if (ct + 1 < ct1) aop = weights(ct + 1);
    // GELU and rounding of the lane's 16 outputs, with no branch between them
    // so their instruction chains interleave
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = acc[2 * i], b = acc[2 * i + 1];
      o[i] = GELU ? pack2<DT>(gelu_erf(a), gelu_erf(b)) : pack2<DT>(a, b);
    }
    // runs 2k and 2k + 1 (channels 16 k + 4 h .. and 16 k + 8 + 4 h ..): swapping
    // the upper half's first run with the lower half's second leaves lane h
    // with channels 16 k + 8 h .. + 7
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const auto x = __builtin_amdgcn_permlane32_swap(o[4 * k], o[4 * k + 2], false, false);
      const auto z = __builtin_amdgcn_permlane32_swap(o[4 * k + 1], o[4 * k + 3], false, false);
      const int c = ct * 32 + 16 * k + 8 * h;  // c_out % 8 == 0: all in or all out
      if (m < p.M && c < p.c_out) *reinterpret_cast<u32x4*>(y + c) = u32x4{x[0], z[0], x[1], z[1]};
    }
  }
}

}  // namespace

hipError_t launch_conv1(int dtype, const Conv1Params& p, hipStream_t s) {
  if (p.c_out > kMaxCout) return hipErrorInvalidValue;  // rejected by validation
  const unsigned blocks = (unsigned)((p.M + kPix - 1) / kPix);
  // Groups of five tiles (160 channels) per block, so that a short clip's last
  // round is not mostly idle; all of a pixel's channels in one block for the
  // longest clips, whose rows are then written whole.  480 channels, f16, groups of 5 against one of 15, us by pixel blocks:
  // 375 18.9 / 24.0, 1000 38.5 / 38.4, 2050 73 / 74, 3000 111 / 118, 3750 141 / 171,
  // 5000 186 / 221, 6250 294 / 263, 7500 384 / 308, 10000 555 / 398.  (Groups of two
  // are 14-31% faster up to 125 and 6-12% slower from 500 on.)
  const int tiles = (p.c_out + 31) / 32, group = blocks >= 5632 ? tiles : 5;
  const dim3 g(blocks, (unsigned)((tiles + group - 1) / group)), t(256);
  if (dtype == QA_BF16) {
    if (p.gelu) hipLaunchKernelGGL((conv1_kernel<QA_BF16, true>), g, t, 0, s, p, group);
    else hipLaunchKernelGGL((conv1_kernel<QA_BF16, false>), g, t, 0, s, p, group);
  } else {
    if (p.gelu) hipLaunchKernelGGL((conv1_kernel<QA_F16, true>), g, t, 0, s, p, group);
    else hipLaunchKernelGGL((conv1_kernel<QA_F16, false>), g, t, 0, s, p, group);
  }
  return hipGetLastError();
}

}  // namespace qa
