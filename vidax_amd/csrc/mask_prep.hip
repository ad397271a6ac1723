// Mask preparation of the flash kernels for gfx950: the caller's masks, in
// whatever strides and widths they come, to the forms the attention kernels
// stage, one launch each. As chains of six to eight elementwise and reduction
// launches they took more time than the attention itself: one launch instead
// took masked self-attention B=2 H=24 S=256 from 56.6 to 29.0 us a call, a full
// bias with a padding mask B=2 H=8 S=512 D=64 from 63.5 to 34.2 us, a key bias
// H=24 S=8192 from 686 to 677 us.
#include "vx_gfx950.hpp"
#include "vx_kernels.h"

#include <algorithm>

namespace vx {
namespace {

constexpr uint32_t kNegInfBits = 0xff800000u;
constexpr uint32_t kQuietNanBits = 0x7fc00000u;

// ---- key masks: one workgroup per batch item, 16 keys per thread and pass.
// Validity bytes and fp32 biases of the keys go to rows padded to whole
// 64-key tiles (padding invalid, -inf), and the index of the last key that is
// valid and whose bias is above -inf, plus one, to kv_len. Latency-bound (a
// row is a few KiB to 0.5 MiB): the loads of a pass are independent 16-byte
// ones where base and key stride allow, and a row needs no second launch.
constexpr int kKeyThreads = 1024;
constexpr int kKeysPerThread = 16;

__global__ __launch_bounds__(kKeyThreads) void key_mask_kernel(const KeyMaskArgs a) {
  __shared__ int wave_last[kKeyThreads / 64];
  const int b = blockIdx.x;
  const uint32_t Sk = (uint32_t)a.Sk, width = (Sk + 63) & ~63u;  // (unsigned counters: seq_k goes up to 2^31 - 1)
  const uint8_t* vp = a.valid != nullptr ? a.valid + b * a.valid_strides[0] : nullptr;
  const float* bp = a.bias != nullptr ? a.bias + b * a.bias_strides[0] : nullptr;
  uint8_t* vo = a.valid_rows != nullptr ? a.valid_rows + b * a.row_stride : nullptr;
  float* bo = a.bias_rows != nullptr ? a.bias_rows + b * a.row_stride : nullptr;
  const bool v16 = a.valid_strides[1] == 1 && ((uintptr_t)vp & 15) == 0;
  const bool b16 = a.bias_strides[1] == 1 && ((uintptr_t)bp & 15) == 0;
  int last = 0;
  for (uint32_t k0 = threadIdx.x * kKeysPerThread; k0 < width; k0 += kKeyThreads * kKeysPerThread) {
    const bool whole = k0 + kKeysPerThread <= Sk;
    uint32_t vw[4] = {0, 0, 0, 0};  // validity, one byte (0 or 1) per key
    uint32_t bw[16];                // bias bits
    if (vp != nullptr) {
      if (v16 && whole) {
        const u32x4 x = *(const u32x4*)(vp + k0);
#pragma unroll
        for (int i = 0; i < 16; ++i) vw[i >> 2] |= (((x[i >> 2] >> (8 * (i & 3))) & 0xffu) != 0 ? 1u : 0u) << (8 * (i & 3));
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (k0 + i < Sk) vw[i >> 2] |= (vp[(k0 + i) * a.valid_strides[1]] != 0 ? 1u : 0u) << (8 * (i & 3));
      }
    }
    if (bp != nullptr) {
      if (b16 && whole) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u32x4 x = *(const u32x4*)(bp + k0 + 4 * i);
#pragma unroll
          for (int e = 0; e < 4; ++e) bw[4 * i + e] = x[e];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          bw[i] = k0 + i < Sk ? ((const uint32_t*)bp)[(k0 + i) * a.bias_strides[1]] : kNegInfBits;
      }
    }
    if (vo != nullptr) *(u32x4*)(vo + k0) = u32x4{vw[0], vw[1], vw[2], vw[3]};
    if (bo != nullptr) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *(u32x4*)(bo + k0 + 4 * i) = u32x4{bw[4 * i], bw[4 * i + 1], bw[4 * i + 2], bw[4 * i + 3]};
    }
    if (a.kv_len != nullptr) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        bool ok = k0 + i < Sk;
        if (vp != nullptr) ok = ok && ((vw[i >> 2] >> (8 * (i & 3))) & 0xffu) != 0;
        // above -inf: neither -inf nor NaN (tested on the bits)
        if (bp != nullptr) ok = ok && bw[i] != kNegInfBits && (bw[i] & 0x7fffffffu) <= 0x7f800000u;
        if (ok) last = (int)(k0 + i + 1);
      }
    }
  }
  if (a.kv_len == nullptr) return;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
  if ((threadIdx.x & 63) == 0) wave_last[threadIdx.x >> 6] = last;
  __syncthreads();
  if (threadIdx.x == 0) {
    int m = 0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) m = max(m, wave_last[w]);
    a.kv_len[b] = m;
  }
}

// ---- full bias: rows of round_up(Sk, 64) fp32 values, one per (batch item,
// head, query) of the broadcast extents, each bias + (mask ? 0 : -inf), the
// padding 0 (no score there is used). One wave per kBiasSeg keys of a row, 4
// keys per lane and pass; bound by the row stores (4 bytes per score), so
// nothing is gained by wider loads of a mask byte.
constexpr int kBiasWaves = 4;
constexpr int kBiasSeg = 4096;

// bits of x + -inf: -inf, or NaN where x is NaN or +inf
__device__ __forceinline__ uint32_t masked_bits(uint32_t x) {
  return (x & 0x7fffffffu) > 0x7f800000u || x == 0x7f800000u ? kQuietNanBits : kNegInfBits;
}

__global__ __launch_bounds__(kBiasWaves * 64) void full_bias_kernel(const FullBiasArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t Sk = (uint32_t)a.Sk, width = (Sk + 63) & ~63u;
  const uint32_t n_seg = (width + kBiasSeg - 1) / kBiasSeg;
  const int64_t items = (int64_t)a.n[0] * a.n[1] * a.n[2] * n_seg;
  for (int64_t w = (int64_t)blockIdx.x * kBiasWaves + wave; w < items; w += (int64_t)gridDim.x * kBiasWaves) {
    const int64_t r = w / n_seg;
    const uint32_t k_lo = (uint32_t)(w - r * n_seg) * kBiasSeg, k_hi = min(k_lo + kBiasSeg, width);
    const int64_t bh = r / a.n[2];
    const int q = (int)(r - bh * a.n[2]);
    const int b = (int)(bh / a.n[1]), h = (int)(bh - (int64_t)b * a.n[1]);
    const uint32_t* bp = a.bias != nullptr ? (const uint32_t*)a.bias + b * a.bias_strides[0] + h * a.bias_strides[1] +
                                                 q * a.bias_strides[2]
                                           : nullptr;
    const uint8_t* mp =
        a.mask != nullptr ? a.mask + b * a.mask_strides[0] + h * a.mask_strides[1] + q * a.mask_strides[2] : nullptr;
    uint32_t* orow = (uint32_t*)a.out + r * width;
    for (uint32_t k0 = k_lo + lane * 4; k0 < k_hi; k0 += 256) {
      u32x4 o = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t k = k0 + e;
        if (k < Sk) {
          if (bp != nullptr) o[e] = bp[k * a.bias_strides[3]];
          if (mp != nullptr && mp[k * a.mask_strides[3]] == 0) o[e] = masked_bits(o[e]);
        }
      }
      *(u32x4*)(orow + k0) = o;
    }
  }
}

// The same for inputs whose queries lie closer together than their keys (a
// transposed bias): 64 x 64 tiles through LDS, read along the queries and
// written along the keys, so that both sides are whole lines (a wave per row
// read 64 lines for 64 values: a call with 4 heads of 4095 x 4095 768 us, in
// tiles 248; 8 of 2000 x 2000 299 and 117). One tile per workgroup and pass.
constexpr int kBiasTile = 64;

__global__ __launch_bounds__(256) void full_bias_transposed_kernel(const FullBiasArgs a) {
  __shared__ uint32_t tile[kBiasTile][kBiasTile + 1];  // [key][query]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t width = ((int64_t)a.Sk + 63) & ~(int64_t)63;
  const int64_t n_kt = width / kBiasTile, n_qt = ((int64_t)a.n[2] + kBiasTile - 1) / kBiasTile;
  const int64_t items = (int64_t)a.n[0] * a.n[1] * n_qt * n_kt;
  for (int64_t w = blockIdx.x; w < items; w += gridDim.x) {  // (uniform: every thread passes the barriers)
    const int64_t bhq = w / n_kt, k0 = (w - bhq * n_kt) * kBiasTile;
    const int64_t bh = bhq / n_qt, q0 = (bhq - bh * n_qt) * kBiasTile;
    const int b = (int)(bh / a.n[1]), h = (int)(bh - (int64_t)b * a.n[1]);
    const int64_t q = q0 + lane;
    const uint32_t* bp = a.bias != nullptr ? (const uint32_t*)a.bias + b * a.bias_strides[0] + h * a.bias_strides[1] +
                                                 q * a.bias_strides[2]
                                           : nullptr;
    const uint8_t* mp =
        a.mask != nullptr ? a.mask + b * a.mask_strides[0] + h * a.mask_strides[1] + q * a.mask_strides[2] : nullptr;
#pragma unroll
    for (int i = 0; i < kBiasTile / 4; ++i) {
      const int64_t k = k0 + 4 * i + wave;
      uint32_t o = 0;
      if (q < a.n[2] && k < a.Sk) {
        if (bp != nullptr) o = bp[k * a.bias_strides[3]];
        if (mp != nullptr && mp[k * a.mask_strides[3]] == 0) o = masked_bits(o);
      }
      tile[4 * i + wave][lane] = o;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kBiasTile / 4; ++i) {
      const int64_t row = q0 + 4 * i + wave;
      if (row < a.n[2]) ((uint32_t*)a.out)[(bh * a.n[2] + row) * width + k0 + lane] = tile[lane][4 * i + wave];
    }
    __syncthreads();
  }
}

}  // namespace

int launch_key_masks(const KeyMaskArgs& a, void* stream, const char** launched) {
  const int64_t need = ((int64_t)a.Sk + kKeysPerThread - 1) / kKeysPerThread;
  const int threads = (int)std::min<int64_t>(kKeyThreads, (need + 63) / 64 * 64);
  hipLaunchKernelGGL(key_mask_kernel, dim3(a.B), dim3(threads), 0, (hipStream_t)stream, a);
  *launched = "key_mask_kernel";
  return (int)hipGetLastError();
}

int launch_full_bias(const FullBiasArgs& a, void* stream, const char** launched) {
  // Tiles for transposed inputs, by the bias (four times the mask's bytes) if
  // both are given; heads of fewer scores stay in the CU's cache, and a wave
  // per row starts more of them at once (64 x 128 x 12 heads of 128 x 128 22 us
  // a call, in tiles 26; 2 x 256 x 24 of 256 x 256 25 either way).
  const int64_t* s = a.bias != nullptr ? a.bias_strides : a.mask_strides;
  if (s[2] > 0 && s[2] < s[3] && (int64_t)a.n[2] * a.Sk >= 256 * 256) {
    const int64_t tiles = (int64_t)a.n[0] * a.n[1] * (((int64_t)a.n[2] + kBiasTile - 1) / kBiasTile) *
                          (((int64_t)a.Sk + kBiasTile - 1) / kBiasTile);
    hipLaunchKernelGGL(full_bias_transposed_kernel, dim3((unsigned)std::min<int64_t>(tiles, 8192)), dim3(256), 0,
                       (hipStream_t)stream, a);
    *launched = "full_bias_transposed_kernel";
    return (int)hipGetLastError();
  }
  const int64_t n_seg = ((int64_t)a.Sk + kBiasSeg - 1) / kBiasSeg;
  const int64_t items = (int64_t)a.n[0] * a.n[1] * a.n[2] * n_seg;
  const int64_t groups = std::min<int64_t>((items + kBiasWaves - 1) / kBiasWaves, 8192);
  hipLaunchKernelGGL(full_bias_kernel, dim3((unsigned)groups), dim3(kBiasWaves * 64), 0, (hipStream_t)stream, a);
  *launched = "full_bias_kernel";
  return (int)hipGetLastError();
}

}  // namespace vx
