// Float-activation matmuls of the hip table: F32 / F16 / BF16 weights
// (trickymind1324/axon-infer src/kernels/ref/matmul.cpp:12-68) and Q8_0 / Q4_0 / Q4_1 weights
// against float activations (src/kernels/ref/quant.cpp:15-40, 147-159), single-row and rows.
//
// These entries serve float weight files and the exact-activations option. Every output is one
// chain over its weight row, left to right in float, which reproduces the scalar table's sum bit for
// bit, including the interleaved low/high nibble order of the Q4 formats.
//
// matmul_float_kernel (F32 / F16 / BF16 weights): a workgroup takes 16 outputs x 16 or 32 activation
// rows; a lane owns one output of one row, the lanes of a row of 16 the same activation row. A chunk of
// kChunk elements of the 16 weight rows is loaded coalesced, two chunks ahead (one chunk's chains take
// less than a load's way from memory), widened to float once and laid in one of two LDS buffers, rows
// padded so that 16 of them cover the banks; a lane reads four elements at a time. The activations stay
// in registers, 16 elements of a row across its lanes, and reach the multiply by its own DPP
// broadcast, so LDS holds and serves the weights only. A wave is mostly alone on its SIMD: what
// bounds it is the in-order chain at an instruction about every 5 cycles (a multiply and an add per
// element, 4.5 ns), then the chunk's barrier and loads. So products are formed four elements ahead
// of their adds, LDS reads 24 ahead, in an order the compiler keeps, and whole chunks of whole tiles
// load without a look at the ends (24 -> 18 us). Two activation rows per lane were slower at every size.
// F16, us: one lane walking its row in memory -> both operands in LDS, a thread one output of one
// row -> now: 2048 x 2048 at 16 rows 252 -> 29 -> 16.5, at one row 237 -> 27 -> 15.8.
//
// matmul_lane_kernel: one lane per output, for Q8_0 / Q4_0 / Q4_1, whose short rows of blocks the L1
// holds (2048 x 2048 at 16 rows 35-47 us; staged as above it ran 34-36 us at 16 rows, and slower from 17
// on), and for float weights in very short rows, of which a workgroup above holds 16 in a chunk of 256
// elements. Where the line lies, us, a lane per output / tiles: F16 at 300 rows, 30000 outputs, 14 elements
// 105 / 103, 16 246 / 102 (F32: 9 elements 88 / 117, 12 152 / 100); at 8 rows, 40000 outputs, 26 elements 15.8 /
// 15.7, 32 21.2 / 15.7 (12000 outputs 8.6 / 6.6); at one row, 9000 outputs, 49 elements 6.1 / 7.0, 56 9.0 / 6.4,
// 32000 outputs, 64 elements 11.0 / 13.2, 110000 outputs, 16 elements 5.3 / 36.6.
#include "common.h"
#include "matmul_float.h"

namespace axon_hip {

namespace {

constexpr uint32_t kOut = 16;              // outputs per workgroup, one per lane of a row of 16
constexpr uint32_t kChunk = 256;           // elements per chunk
constexpr uint32_t kPitch = kChunk + 4;    // floats per row in LDS

template <int T>
__device__ __forceinline__ float weight_value(uint32_t bits) {
  if constexpr (T == F32) return __uint_as_float(bits);
  else if constexpr (T == F16) return half_bits_to_float(bits);
  else return bf16_bits_to_float(bits);
}

// W waves of 4 activation rows. PAIR: the weight rows' elements can be loaded two at a time.
template <int T, uint32_t W, bool PAIR>
__global__ __launch_bounds__(64 * W) void matmul_float_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                              float* __restrict__ y, uint32_t n_rows, uint32_t n_out,
                                                              uint32_t n_in, uint32_t y_stride, size_t row_bytes) {
  constexpr uint32_t kPairs = kChunk / 2, kItems = kOut * kPairs / (64 * W), kSteps = kChunk / 16;
  static_assert(64 * W % kPairs == 0, "a thread's pair has the same place in every row it loads");
  __shared__ __attribute__((aligned(16))) float ws[2][kOut * kPitch];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t o0 = blockIdx.x * kOut, m0 = blockIdx.y * (4 * W) + wave * 4;
  const uint32_t oo = min(kOut, n_out - o0);
  const uint32_t l16 = lane % 16, pair = tid % kPairs, irow = tid / kPairs;

  // A thread's weights of a chunk: one pair of kItems rows. Rows and elements past the ends count as
  // zero, and a zero product leaves a chain as it is.
  struct Raw {
    uint32_t v[kItems][T == F32 || !PAIR ? 2 : 1];
  };
  auto load_w = [&](uint32_t k0, Raw& r) {
    constexpr size_t es = T == F32 ? 4 : 2;
    if (oo == kOut && k0 + kChunk <= n_in) {
      // A whole chunk of whole tiles: no element needs a look at the ends.
      const uint8_t* mine = w + (o0 + irow) * row_bytes + 2 * pair * es;
#pragma unroll
      for (uint32_t i = 0; i < kItems; ++i) {
        const uint8_t* p = mine + (i * (64 * W / kPairs) * row_bytes + k0 * es);
        if constexpr (PAIR && T == F32) {
          const uint2 u = *reinterpret_cast<const uint2*>(p);
          r.v[i][0] = u.x;
          r.v[i][1] = u.y;
        } else if constexpr (PAIR) {
          r.v[i][0] = *reinterpret_cast<const uint32_t*>(p);
        } else {
#pragma unroll
          for (uint32_t e = 0; e < 2; ++e) {
            if constexpr (T == F32) r.v[i][e] = reinterpret_cast<const uint32_t*>(p)[e];
            else r.v[i][e] = reinterpret_cast<const uint16_t*>(p)[e];
          }
        }
      }
      return;
    }
    const uint32_t k = k0 + 2 * pair;
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i) {
      const uint32_t row = i * (64 * W / kPairs) + irow;
      const uint8_t* p = w + (o0 + row) * row_bytes;
      if constexpr (PAIR) {  // (n_in is even)
        if constexpr (T == F32) {
          const uint2 u = row < oo && k < n_in ? *reinterpret_cast<const uint2*>(p + static_cast<size_t>(k) * 4) : make_uint2(0, 0);
          r.v[i][0] = u.x;
          r.v[i][1] = u.y;
        } else {
          r.v[i][0] = row < oo && k < n_in ? *reinterpret_cast<const uint32_t*>(p + static_cast<size_t>(k) * 2) : 0;
        }
      } else {
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e) {
          r.v[i][e] = 0;
          if (row < oo && k + e < n_in) {
            if constexpr (T == F32) r.v[i][e] = reinterpret_cast<const uint32_t*>(p)[k + e];
            else r.v[i][e] = reinterpret_cast<const uint16_t*>(p)[k + e];
          }
        }
      }
    }
  };
  auto store_w = [&](const Raw& r, float* dst) {
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i) {
      float2 f;
      if constexpr (T == F32 || !PAIR) {
        f = make_float2(weight_value<T>(r.v[i][0]), weight_value<T>(r.v[i][1]));
      } else {
        f = make_float2(weight_value<T>(r.v[i][0] & 0xffffu), weight_value<T>(r.v[i][0] >> 16));
      }
      *reinterpret_cast<float2*>(dst + (i * (64 * W / kPairs) + irow) * kPitch + 2 * pair) = f;
    }
  };
  // The wave's activations of a chunk: lane l of a row of 16 holds elements 16 q + l of that row's own
  // activation row, and the multiplies take them by a broadcast within it.
  struct Acts {
    float v[kSteps];
  };
  const uint32_t m = m0 + lane / 16;
  const float* xrow = x + static_cast<size_t>(min(m, n_rows - 1)) * n_in;
  auto load_x = [&](uint32_t k0, Acts& a) {
    if (k0 + kChunk <= n_in) {
      const float* p = xrow + k0 + l16;
#pragma unroll
      for (uint32_t q = 0; q < kSteps; ++q) a.v[q] = p[16 * q];
      return;
    }
#pragma unroll
    for (uint32_t q = 0; q < kSteps; ++q) {
      const uint32_t k = k0 + 16 * q + l16;
      a.v[q] = k < n_in ? xrow[k] : 0.0f;
    }
  };

  float acc = 0.0f;
  auto chunk = [&](uint32_t k0, uint32_t buf, Raw& r, Acts& a) {
    store_w(r, ws[buf]);
    __syncthreads();  // the chunk is in LDS; the other buffer, of the chunk before, has been read
    if (k0 + 2 * kChunk < n_in) load_w(k0 + 2 * kChunk, r);
    if (m0 >= n_rows) return;
    const float4* row = reinterpret_cast<const float4*>(ws[buf] + l16 * kPitch);
    auto step = [&]<int Q>() {
      float v[16];
#pragma unroll
      for (uint32_t c = 0; c < 4; ++c) {
        const float4 u = row[4 * Q + c];
        v[4 * c] = u.x;
        v[4 * c + 1] = u.y;
        v[4 * c + 2] = u.z;
        v[4 * c + 3] = u.w;
      }
      for_each_index<0, 16>([&]<int E>() {
        acc += row_lane<E>(a.v[Q]) * v[E];
      });
    };
    if (k0 + kChunk <= n_in) {
      // Quad T's adds beside quad T + 1's products, in an order that the compiler keeps, and its LDS
      // reads kAhead quads before.
      constexpr int kQuads = kChunk / 4, kAhead = 6;
      float4 v[8];
      float p[2][4];
      auto product = [&]<int T4, int E>() {
        const float4 u = v[T4 % 8];
        const float ve = E == 0 ? u.x : E == 1 ? u.y : E == 2 ? u.z : u.w;
        p[T4 % 2][E] = row_lane<(4 * T4 + E) % 16>(a.v[T4 / 4]) * ve;
      };
#pragma unroll
      for (int t = 0; t < kAhead; ++t) v[t] = row[t];
      for_each_index<0, 4>([&]<int E>() { product.template operator()<0, E>(); });
      for_each_index<0, kQuads>([&]<int T4>() {
        if constexpr (T4 + kAhead < kQuads) v[(T4 + kAhead) % 8] = row[T4 + kAhead];
        for_each_index<0, 4>([&]<int E>() {
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (T4 + 1 < kQuads) product.template operator()<T4 + 1, E>();
          acc += p[T4 % 2][E];
        });
      });
    } else {
      const uint32_t n = (n_in - k0 + 15) / 16;
      for_each_index<0, kSteps>([&]<int Q>() {
        if (Q < static_cast<int>(n)) step.template operator()<Q>();
      });
    }
    if (k0 + 2 * kChunk < n_in) load_x(k0 + 2 * kChunk, a);
  };
  Raw ra, rb;
  Acts xa, xb;
  load_w(0, ra);
  load_x(0, xa);
  load_w(kChunk, rb);
  load_x(kChunk, xb);
  for (uint32_t k0 = 0; k0 < n_in; k0 += 2 * kChunk) {
    chunk(k0, 0, ra, xa);
    if (k0 + kChunk < n_in) chunk(k0 + kChunk, 1, rb, xb);
  }
  if (l16 < oo && m < n_rows) y[static_cast<size_t>(m) * y_stride + o0 + l16] = acc;
}

template <int T>
int matmul_float_tiles(const uint8_t* w, const float* x, float* y, uint32_t n_rows, uint32_t n_out, uint32_t n_in,
                       uint32_t y_stride, size_t row_bytes) {
  const uint32_t cols = static_cast<uint32_t>(ceil_div(n_out, kOut));
  const bool pair = n_in % 2 == 0 && reinterpret_cast<uintptr_t>(w) % (T == F32 ? 8 : 4) == 0;
  // Eight waves (32 rows) share a chunk's loads where that leaves a workgroup per CU, and up to 16 rows,
  // where the waves without rows only load; else four. F16, us with eight / four: 2048 x 2048 at 16 rows
  // 16.5 / 18.1, 8192 x 2048 at 16 rows 23.4 / 25.4, 2048 x 2048 at 64 rows 22.6 / 24.4 (256 workgroups
  // of eight), 1024 x 8192 at 64 rows 83.8 / 65.2 (128).
  const bool eight = n_rows <= 16 || static_cast<uint64_t>(cols) * ceil_div(n_rows, 32) >= 256;
  auto go = [&](auto kernel, uint32_t waves) {
    const dim3 grid(cols, static_cast<uint32_t>(ceil_div(n_rows, 4 * waves)));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, stream(), w, x, y, n_rows, n_out, n_in, y_stride, row_bytes);
  };
  if (pair && eight) go(matmul_float_kernel<T, 8, true>, 8);
  else if (pair) go(matmul_float_kernel<T, 4, true>, 4);
  else if (eight) go(matmul_float_kernel<T, 8, false>, 8);
  else go(matmul_float_kernel<T, 4, false>, 4);
  return check_launch("matmul_float");
}

template <int T>
__device__ float row_dot(const uint8_t* w, const float* x, uint32_t n_in) {
  float acc = 0.0f;
  if constexpr (T == F32 || T == F16 || T == BF16) {
    for (uint32_t i = 0; i < n_in; ++i) {
      if constexpr (T == F32) acc += reinterpret_cast<const float*>(w)[i] * x[i];
      else acc += weight_value<T>(reinterpret_cast<const uint16_t*>(w)[i]) * x[i];
    }
  } else if constexpr (T == Q8_0) {
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
__global__ __launch_bounds__(256) void matmul_lane_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
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
  // (Rows of 32 bytes apart fall on few channels: 246 us where rows of 30 take 122.)
  const bool short_rows =
      n_rows <= 65535 && ((row_bytes <= (type == F32 ? 36 : 28) && row_bytes != 32) || (row_bytes <= 80 && n_rows * row_bytes <= 416) ||
                          (n_rows == 1 && ((row_bytes <= 100 && n_out >= 8192) || (row_bytes <= 128 && n_out >= 32000))));
  auto by_lanes = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream(), wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes);
    return check_launch("matmul_float");
  };
  switch (type) {
  case F32:
    if (short_rows) return by_lanes(matmul_lane_kernel<F32>);
    return matmul_float_tiles<F32>(wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes);
  case F16:
    if (short_rows) return by_lanes(matmul_lane_kernel<F16>);
    return matmul_float_tiles<F16>(wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes);
  case BF16:
    if (short_rows) return by_lanes(matmul_lane_kernel<BF16>);
    return matmul_float_tiles<BF16>(wb, x, y, n_rows, n_out, n_in, y_stride, row_bytes);
  case Q8_0: return by_lanes(matmul_lane_kernel<Q8_0>);
  case Q4_0: return by_lanes(matmul_lane_kernel<Q4_0>);
  default: return by_lanes(matmul_lane_kernel<Q4_1>);
  }
}

}  // namespace axon_hip
