// Format kernels (affine quantize / dequantize) and the HBM stream
// calibrator.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace rmoe {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Bound by the stream of w.  Sixteen lanes hold a 64-value group, four
// values each, so a load instruction reads whole lines; a wave takes 16
// groups (each row of 16 lanes four neighbouring ones), all requested before
// the first is used.  One thread per group read 16 bytes of 64 lines with
// every load: 134 M values at 8 | 4 bits took 164 | 130 us (4.1 | 4.7 TB/s, in
// and out), now 116 | 107 (5.9 | 5.7).
// Arithmetic is plain IEEE fp32 (correctly rounded division, round-half-even
// rint), so the result is reproducible on the host bit for bit.
constexpr int kQuantGroups = 16;  // groups per wave

// The value of lane u of each four.
__device__ __forceinline__ float quad_bcast(float v, int u) {
  const int i = __float_as_int(v);
  int r;
  switch (u) {  // the control must be a compile-time constant
    case 0: r = __builtin_amdgcn_update_dpp(0, i, 0x00, 0xF, 0xF, false); break;
    case 1: r = __builtin_amdgcn_update_dpp(0, i, 0x55, 0xF, 0xF, false); break;
    case 2: r = __builtin_amdgcn_update_dpp(0, i, 0xAA, 0xF, 0xF, false); break;
    default: r = __builtin_amdgcn_update_dpp(0, i, 0xFF, 0xF, 0xF, false); break;
  }
  return __int_as_float(r);
}

template <int BITS>
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ w,
                                                       const int64_t groups,
                                                       uint32_t* __restrict__ wq,
                                                       uint16_t* __restrict__ s_out,
                                                       uint16_t* __restrict__ b_out) {
  constexpr int U = kQuantGroups / 4;
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15;
  const int64_t g0 =
      ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kQuantGroups + (lane >> 4) * U;
  f32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t g = g0 + u < groups ? g0 + u : groups - 1;
    v[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + g * 64) + l16);
  }
  const float n_bins = (float)((1 << BITS) - 1);
  // extremes of the groups: lane l16 keeps those of group l16 & 3 and works
  // out that one's scale and bias (every lane those of all four, three
  // divisions each, took 138 | 141 us)
  const int mine = l16 & 3;
  float w_max = 0.0f, w_min = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float hi = fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w));
    float lo = fminf(fminf(v[u].x, v[u].y), fminf(v[u].z, v[u].w));
    hi = fmaxf(hi, dpp_f(hi, 0xB1));
    lo = fminf(lo, dpp_f(lo, 0xB1));
    hi = fmaxf(hi, dpp_f(hi, 0x4E));
    lo = fminf(lo, dpp_f(lo, 0x4E));
    hi = fmaxf(hi, dpp_f(hi, 0x141));
    lo = fminf(lo, dpp_f(lo, 0x141));
    hi = fmaxf(hi, dpp_f(hi, 0x140));
    lo = fminf(lo, dpp_f(lo, 0x140));
    w_max = mine == u ? hi : w_max;
    w_min = mine == u ? lo : w_min;
  }
  // a NaN only counts as its group's first value (the sequential "larger
  // than" scan from value 0 that defines the format)
  bool nan = false;
#pragma unroll
  for (int u = 0; u < U; ++u) nan = nan || v[u].x != v[u].x;
  if (__any(nan && l16 == 0)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float first = __shfl(v[u].x, lane & 48, 64);
      if (mine == u && first != first) w_max = w_min = first;
    }
  }
  const bool mask = fabsf(w_min) > fabsf(w_max);
  float scale = (w_max - w_min) / n_bins;
  scale = scale > 1e-7f ? scale : 1e-7f;
  scale = mask ? scale : -scale;
  const float edge = mask ? w_min : w_max;
  const float q0 = rintf(edge / scale);
  if (q0 != 0.0f) scale = edge / q0;
  const uint32_t sb = f32_to_bf16(scale);
  const uint32_t bb = f32_to_bf16(q0 == 0.0f ? 0.0f : edge);
  const float s_own = bf16_to_f32(sb);
  const float b_own = bf16_to_f32(bb);
  // Codes: rint of the correctly rounded quotient.  The product with the
  // rounded reciprocal is within 3 x 2^-24 |t| of that quotient: under 4.7e-5
  // for |t| < 260, and beyond that both clamp alike.  So unless t lies within
  // 1e-4 of a half-integer (or is not finite, or the reciprocal is near the
  // ends of its range: NaN here) the two round to the same whole number; the
  // others divide.  (A division per value took 162 us at 8 bits.)
  const bool plain = fabsf(s_own) > 0x1p-100f && fabsf(s_own) < 0x1p100f;
  const float r_own = plain ? 1.0f / s_own : __builtin_nanf("");
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float s = quad_bcast(s_own, u);
    const float b = quad_bcast(b_own, u);
    const float r = quad_bcast(r_own, u);
    float q4[4];
    bool all = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float t = (v[u][j] - b) * r;
      q4[j] = rintf(t);
      all = all && fabsf(t - q4[j]) < 0.4999f;
    }
    if (!all) {
#pragma unroll
      for (int j = 0; j < 4; ++j) q4[j] = rintf((v[u][j] - b) / s);
    }
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float q = q4[j];
      q = q < 0.0f ? 0.0f : (q > n_bins ? n_bins : q);
      word |= ((uint32_t)q) << (BITS * j);
    }
    const bool live = g0 + u < groups;
    if constexpr (BITS == 8) {
      if (live) wq[(g0 + u) * 16 + l16] = word;
    } else {
      // two lanes make a word
      word |= dpp_u(word, 0xB1) << 16;
      if (live && !(l16 & 1)) wq[(g0 + u) * 8 + (l16 >> 1)] = word;
    }
  }
  if (l16 < U && g0 + l16 < groups) {
    s_out[g0 + l16] = (uint16_t)sb;
    b_out[g0 + l16] = (uint16_t)bb;
  }
}

hipError_t launch_quantize(const float* w, int64_t rows, int cols, int bits,
                           uint32_t* wq, uint16_t* s, uint16_t* b, hipStream_t st) {
  const int64_t groups = rows * (cols / 64);
  if (groups == 0) return hipSuccess;
  constexpr int kPerBlock = 4 * kQuantGroups;
  const unsigned blocks = (unsigned)((groups + kPerBlock - 1) / kPerBlock);
  if (bits == 8)
    hipLaunchKernelGGL(quantize_kernel<8>, dim3(blocks), dim3(256), 0, st, w,
                       groups, wq, s, b);
  else
    hipLaunchKernelGGL(quantize_kernel<4>, dim3(blocks), dim3(256), 0, st, w,
                       groups, wq, s, b);
  return hipGetLastError();
}

// fl32(q * s + b) with q * s exact, i.e. a single rounding, and optionally
// bf16 (round-to-nearest-even) of it.  Bound by the output stream: a thread
// writes 8 values per step in 16-byte pieces (V: the outputs are 16-byte
// aligned) and has STEPS steps' loads in flight.  Rows are whole groups, so
// words, groups and outputs are all linear in the value index.
// One packed word per thread with 2-byte stores took 138 us for 134 M values
// at 8 bits to bf16 (3.0 TB/s, in and out), now 71 (5.8).
template <int BITS, bool V, int STEPS>
__global__ __launch_bounds__(256) void dequantize_kernel(const QW q, const int64_t value0,
                                                         const int64_t chunks,
                                                         float* __restrict__ out_f32,
                                                         uint16_t* __restrict__ out_bf16) {
  constexpr int WPC = BITS / 4;  // words per 8 values
  const int64_t c0 = (int64_t)blockIdx.x * (256 * STEPS) + threadIdx.x;
  uint32_t word[STEPS][WPC];
  uint32_t sv[STEPS], bv[STEPS];
#pragma unroll
  for (int k = 0; k < STEPS; ++k) {
    const int64_t c = c0 + 256 * k < chunks ? c0 + 256 * k : chunks - 1;
    const int64_t at = (value0 >> 3) + c;
    __builtin_memcpy(word[k], __builtin_assume_aligned(q.w + at * WPC, 4 * WPC), 4 * WPC);
    sv[k] = q.s[at >> 3];
    bv[k] = q.b[at >> 3];
  }
#pragma unroll
  for (int k = 0; k < STEPS; ++k) {
    const int64_t c = c0 + 256 * k;
    if (c >= chunks) return;
    const float s = bf16_to_f32(sv[k]);
    const float b = bf16_to_f32(bv[k]);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t code = (word[k][j * BITS / 32] >> (BITS * j % 32)) & ((1u << BITS) - 1u);
      v[j] = fmaf((float)code, s, b);
    }
    if (out_f32) {
      float* o = out_f32 + c * 8;
      if constexpr (V) {
        reinterpret_cast<float4*>(o)[0] = make_float4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<float4*>(o)[1] = make_float4(v[4], v[5], v[6], v[7]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = v[j];
      }
    }
    if (out_bf16) {
      uint32_t h[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) h[j] = f32_to_bf16(v[j]);
      uint16_t* o = out_bf16 + c * 8;
      if constexpr (V) {
        *reinterpret_cast<uint4*>(o) = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16,
                                                  h[4] | h[5] << 16, h[6] | h[7] << 16);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (uint16_t)h[j];
      }
    }
  }
}

hipError_t launch_dequantize(const QW& q, int cols, int bits, int64_t row_begin,
                             int64_t rows, float* out_f32, uint16_t* out_bf16,
                             hipStream_t st) {
  const int64_t chunks = rows * (cols / 8);
  if (chunks == 0) return hipSuccess;
  const bool vec = (((uintptr_t)out_f32 | (uintptr_t)out_bf16) & 15) == 0;
  // Four steps a thread for bf16 alone from 2^24 values on (134 M at 8 | 4
  // bits: 77 | 79 us with one, 71 | 63 with four; 16 M, read once, 12.7 | 12.5
  // and 12.7 | 11.6; also where one would not fit a launch).  Fewer values
  // leave the device idle with four (65536 at 8 bits: 1.9 and 2.5), and
  // fp32's wider stores want the threads (134 M at 8 bits: 121 and 165).
  const bool four = (!out_f32 && chunks >= 1 << 21) || chunks >= 1ll << 31;
  const int per = four ? 1024 : 256;
  const unsigned blocks = (unsigned)((chunks + per - 1) / per);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, st, q, row_begin * (int64_t)cols, chunks,
                       out_f32, out_bf16);
  };
  auto steps = [&](auto bits_c, auto vec_c) {
    constexpr int B = decltype(bits_c)::value;
    constexpr bool V = decltype(vec_c)::value;
    if (four) go(dequantize_kernel<B, V, 4>);
    else go(dequantize_kernel<B, V, 1>);
  };
  using B8 = std::integral_constant<int, 8>;
  using B4 = std::integral_constant<int, 4>;
  if (bits == 8) {
    if (vec) steps(B8{}, std::true_type{});
    else steps(B8{}, std::false_type{});
  } else {
    if (vec) steps(B4{}, std::true_type{});
    else steps(B4{}, std::false_type{});
  }
  return hipGetLastError();
}

// Grid-stride read of 16-byte vectors, 4 loads in flight per lane; each
// workgroup folds what it read into partials[blockIdx.x].
__global__ __launch_bounds__(256) void stream_read_kernel(const u32x4* __restrict__ buf,
                                                          const int64_t n,
                                                          uint32_t* __restrict__ partials) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t acc = 0;
  for (; i + 3 * stride < n; i += 4 * stride) {
    const u32x4 a = __builtin_nontemporal_load(buf + i);
    const u32x4 b = __builtin_nontemporal_load(buf + i + stride);
    const u32x4 c = __builtin_nontemporal_load(buf + i + 2 * stride);
    const u32x4 d = __builtin_nontemporal_load(buf + i + 3 * stride);
    acc += (a.x ^ a.y ^ a.z ^ a.w) + (b.x ^ b.y ^ b.z ^ b.w) +
           (c.x ^ c.y ^ c.z ^ c.w) + (d.x ^ d.y ^ d.z ^ d.w);
  }
  for (; i < n; i += stride) {
    const u32x4 a = __builtin_nontemporal_load(buf + i);
    acc += a.x ^ a.y ^ a.z ^ a.w;
  }
  __shared__ uint32_t red[4];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partials[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

hipError_t launch_stream_read(const void* buf, size_t bytes, uint32_t* partials,
                              int blocks, hipStream_t st) {
  hipLaunchKernelGGL(stream_read_kernel, dim3(blocks), dim3(256), 0, st,
                     reinterpret_cast<const u32x4*>(buf), (int64_t)(bytes / 16),
                     partials);
  return hipGetLastError();
}

}  // namespace rmoe
