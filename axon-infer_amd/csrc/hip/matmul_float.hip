// Float-activation matmuls of the hip table: F32 / F16 / BF16 weights
// (trickymind1324/axon-infer src/kernels/ref/matmul.cpp:12-68) and Q8_0 / Q4_0 / Q4_1 weights
// against float activations (src/kernels/ref/quant.cpp:15-40, 147-159), single-row and rows.
//
// These entries serve float weight files and the exact-activations option. Every output is one
// chain over its weight row, left to right in float, which reproduces the scalar table's sum bit for
// bit, including the interleaved low/high nibble order of the Q4 formats.
//
// matmul_float_kernel (F32 / F16 / BF16 weights): a workgroup takes 16 outputs x 16 activation rows, a
// thread one of each. A chunk of kChunk elements of the 16 weight rows and the activation rows is
// loaded coalesced, two chunks ahead (one chunk's chains take less than a load's way from memory),
// widened to float once and laid in LDS; the chains read four elements per 16-byte read, the rows
// padded so that 16 of them cover the banks. One lane walking its row in memory, as before, was bound
// by its own uncoalesced loads on a few CUs: F16 2048 x 2048 at 16 rows 252 -> 30 us, at one row
// 237 -> 27, 2048 x 8192 at 64 rows 1899 -> 127. Now the chains and their LDS reads bound it.
//
// matmul_blocks_kernel (Q8_0 / Q4_0 / Q4_1): one lane per output, whose short rows of blocks the L1
// holds (2048 x 2048 at 16 rows 35-47 us); staged as above it ran 34-36 us at 16 rows, and slower
// from 17 on.
#include "common.h"
#include "matmul_float.h"

namespace axon_hip {

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kOut = 16, kRows = 16;  // outputs and activation rows per workgroup
constexpr uint32_t kChunk = 256;           // elements per chunk
constexpr uint32_t kPitch = kChunk + 4;    // floats per row in LDS

template <int T>
__device__ __forceinline__ float weight_value(uint32_t bits) {
  if constexpr (T == F32) return __uint_as_float(bits);
  else if constexpr (T == F16) return half_bits_to_float(bits);
  else return bf16_bits_to_float(bits);
}

template <int T>
__global__ __launch_bounds__(kThreads) void matmul_float_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                                float* __restrict__ y, uint32_t n_rows, uint32_t n_out,
                                                                uint32_t n_in, uint32_t y_stride, size_t row_bytes) {
  __shared__ __attribute__((aligned(16))) float ws[kOut * kPitch];
  __shared__ __attribute__((aligned(16))) float xs[kRows * kPitch];
  const uint32_t tid = threadIdx.x;
  const uint32_t o0 = blockIdx.x * kOut, m0 = blockIdx.y * kRows;
  const uint32_t oo = min(kOut, n_out - o0), mm = min(kRows, n_rows - m0);

  // A thread's loads of a chunk: element tid of every row. Rows and elements past the ends count as
  // zero, and a zero product leaves a chain as it is.
  static_assert(kChunk == kThreads, "a thread holds one element of each row");
  struct Raw {
    float x[kRows];
    uint32_t w[kOut];
  };
  auto load = [&](uint32_t k0, Raw& r) {
    const bool in = k0 + tid < n_in;
#pragma unroll
    for (uint32_t m = 0; m < kRows; ++m) r.x[m] = in && m < mm ? x[static_cast<size_t>(m0 + m) * n_in + k0 + tid] : 0.0f;
#pragma unroll
    for (uint32_t o = 0; o < kOut; ++o) {
      r.w[o] = 0;
      if (in && o < oo) {
        const uint8_t* p = w + (o0 + o) * row_bytes;
        if constexpr (T == F32) r.w[o] = reinterpret_cast<const uint32_t*>(p)[k0 + tid];
        else r.w[o] = reinterpret_cast<const uint16_t*>(p)[k0 + tid];
      }
    }
  };
  const uint32_t o = tid % kOut, m = tid / kOut;
  const float* wp = ws + o * kPitch;
  const float* xp = xs + m * kPitch;
  float acc = 0.0f;
  auto chunk = [&](uint32_t k0, Raw& r) {
    __syncthreads();  // the previous chunk has been read
#pragma unroll
    for (uint32_t i = 0; i < kRows; ++i) xs[i * kPitch + tid] = r.x[i];
#pragma unroll
    for (uint32_t i = 0; i < kOut; ++i) ws[i * kPitch + tid] = weight_value<T>(r.w[i]);
    __syncthreads();
    if (k0 + 2 * kChunk < n_in) load(k0 + 2 * kChunk, r);
    if (m >= mm) return;
    const uint32_t n = (min(kChunk, n_in - k0) + 3) / 4;
#pragma unroll 8
    for (uint32_t q = 0; q < n; ++q) {
      const float4 a = *reinterpret_cast<const float4*>(wp + 4 * q);
      const float4 b = *reinterpret_cast<const float4*>(xp + 4 * q);
      acc += a.x * b.x;
      acc += a.y * b.y;
      acc += a.z * b.z;
      acc += a.w * b.w;
    }
  };
  Raw ra, rb;
  load(0, ra);
  load(kChunk, rb);
  for (uint32_t k0 = 0; k0 < n_in; k0 += 2 * kChunk) {
    chunk(k0, ra);
    if (k0 + kChunk < n_in) chunk(k0 + kChunk, rb);
  }
  if (o < oo && m < mm) y[static_cast<size_t>(m0 + m) * y_stride + o0 + o] = acc;
}

template <int T>
__device__ float row_dot(const uint8_t* w, const float* x, uint32_t n_in) {
  float acc = 0.0f;
  if constexpr (T == Q8_0) {
    for (uint32_t b = 0; b < n_in / kQK; ++b) {
      const uint8_t* blk = w + b * kBytesQ8_0;
      const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(blk));
      const float* xb = x + b * kQK;
      for (int i = 0; i < kQK; ++i) acc += static_cast<float>(static_cast<int8_t>(blk[2 + i])) * d * xb[i];
    }
  } else if constexpr (T == Q4_0) {
    for (uint32_t b = 0; b < n_in / kQK; ++b) {
      const uint8_t* blk = w + b * kBytesQ4_0;
      const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(blk));
      const float* xb = x + b * kQK;
      for (int i = 0; i < 16; ++i) {
        const uint8_t q = blk[2 + i];
        acc += static_cast<float>(static_cast<int>(q & 0x0f) - 8) * d * xb[i];
        acc += static_cast<float>(static_cast<int>(q >> 4) - 8) * d * xb[i + 16];
      }
    }
  } else {
    for (uint32_t b = 0; b < n_in / kQK; ++b) {
      const uint8_t* blk = w + b * kBytesQ4_1;
      const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(blk));
      const float m = half_bits_to_float(*reinterpret_cast<const uint16_t*>(blk + 2));
      const float* xb = x + b * kQK;
      for (int i = 0; i < 16; ++i) {
        const uint8_t q = blk[4 + i];
        acc += (static_cast<float>(q & 0x0f) * d + m) * xb[i];
        acc += (static_cast<float>(q >> 4) * d + m) * xb[i + 16];
      }
    }
  }
  return acc;
}

template <int T>
__global__ __launch_bounds__(256) void matmul_blocks_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                           float* __restrict__ y, uint32_t n_rows, uint32_t n_out,
                                                           uint32_t n_in, uint32_t y_stride, size_t row_bytes) {
  const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t r = blockIdx.y;
  if (o >= n_out || r >= n_rows) return;
  y[static_cast<size_t>(r) * y_stride + o] = row_dot<T>(w + o * row_bytes, x + static_cast<size_t>(r) * n_in, n_in);
}

}  // namespace

int matmul_float_launch(int type, const void* w, const float* x, float* y, uint32_t n_rows, uint32_t n_out,
                        uint32_t n_in, uint32_t y_stride) {
  if (n_rows == 0 || n_out == 0) return kOk;
  size_t row_bytes = 0;
  switch (type) {
  case F32: row_bytes = 4ull * n_in; break;
  case F16: case BF16: row_bytes = 2ull * n_in; break;
  case Q8_0: row_bytes = n_in / kQK * kBytesQ8_0; break;
  case Q4_0: row_bytes = n_in / kQK * kBytesQ4_0; break;
  case Q4_1: row_bytes = n_in / kQK * kBytesQ4_1; break;
  default: return fail(kUnsupported, "matmul: weight type %d", type);
  }
  if ((type == Q8_0 || type == Q4_0 || type == Q4_1) && n_in % kQK != 0)
    return fail(kInvalidArgument, "quantized matmul: n_in %u is not a multiple of 32", n_in);
  const dim3 grid(static_cast<uint32_t>(ceil_div(n_out, 256)), n_rows);
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  const dim3 tiles(static_cast<uint32_t>(ceil_div(n_out, kOut)), static_cast<uint32_t>(ceil_div(n_rows, kRows)));
  switch (type) {
  case F32: hipLaunchKernelGGL(matmul_float_kernel<F32>, tiles, dim3(kThreads), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  case F16: hipLaunchKernelGGL(matmul_float_kernel<F16>, tiles, dim3(kThreads), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  case BF16: hipLaunchKernelGGL(matmul_float_kernel<BF16>, tiles, dim3(kThreads), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  case Q8_0: hipLaunchKernelGGL(matmul_blocks_kernel<Q8_0>, grid, dim3(256), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  case Q4_0: hipLaunchKernelGGL(matmul_blocks_kernel<Q4_0>, grid, dim3(256), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  default: hipLaunchKernelGGL(matmul_blocks_kernel<Q4_1>, grid, dim3(256), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes); break;
  }
  return check_launch("matmul_float");
}

}  // namespace axon_hip
