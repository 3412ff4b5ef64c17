// General projections and the standalone activation: the FfnAgent operator cases that the
// tuned kernels of gemm.hip do not take.
//
// Reference behaviour (CrossPool checkout):
//  * Gemm.run_into (src/xpool/runtime/ffnagent/operators/linear.py:163-257) with the
//    projection epilogue of operators/activation.py:112-173 and the IEEE kernels of
//    operators/simt.py:13-80: value = fp32 sum of x . w + the fp32 bias; with a fused
//    activation the value is first rounded to the payload dtype (projection_round_dtype,
//    linear.py:56-60), then activated in fp32 (gated: Gate/Up INTERLEAVED, Gate clipped above
//    at the limit, Up clamped to +-limit, plus up_offset); the store rounds to the output
//    dtype.
//  * activation_kernel / Activation.apply_into (operators/activation.py:55-84, 175-207):
//    the same activation over already-projected values, gated (INTERLEAVED or CONCATENATED)
//    or not; an ungated activation may run in place.  ReLU keeps NaN payloads and maps
//    every other non-positive value to +0 (activation.py:19-27).
//
// Payloads are bf16, fp16 or fp32 (activations: bf16 or fp16), any K and N, rows of any
// alignment.  16-bit projections of whole 16-byte rows leave this file where gemm.hip serves them:
// without a bias or activation the Dense projection kernels, from 65 rows with a bias or a gated
// activation the tile kernels' EXTENDED epilogue when it is modelled as faster (and
// projection_reduce_kernel for its K ranges); a gated activation evaluates as here on every route.
// The Router's FP32 and FP32_LOGITS projections, and its odd geometries, run here too.

#include "xp_kernels.hpp"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace xp {
namespace {

__device__ __forceinline__ float load_value(const void *base, int64_t index, int dtype) {
  switch (dtype) {
    case kDtypeF16:
      return __half2float(reinterpret_cast<const __half *>(base)[index]);
    case kDtypeF32:
      return reinterpret_cast<const float *>(base)[index];
    default:
      return bf16_to_float(reinterpret_cast<const uint16_t *>(base)[index]);
  }
}

// Nearest-even rounding to the payload dtype, back in fp32.
__device__ __forceinline__ float round_to(float value, int dtype) {
  switch (dtype) {
    case kDtypeF16:
      return __half2float(__float2half_rn(f32_rounding_point(value)));
    case kDtypeF32:
      return value;
    default:
      return round_bf16(value);
  }
}

__device__ __forceinline__ void store_value(void *base, int64_t index, float value, int dtype) {
  switch (dtype) {
    case kDtypeF16:
      reinterpret_cast<__half *>(base)[index] = __float2half_rn(f32_rounding_point(value));
      break;
    case kDtypeF32:
      reinterpret_cast<float *>(base)[index] = value;
      break;
    default:
      reinterpret_cast<uint16_t *>(base)[index] = static_cast<uint16_t>(float_to_bf16(value));
      break;
  }
}

// ReLU that keeps NaN payloads: x for x > 0 or NaN, +0 otherwise.
__device__ __forceinline__ float relu_keep_nan(float value) { return (value > 0.0f || value != value) ? value : 0.0f; }

__device__ __forceinline__ float apply_function(float value, const ActivationArgs &act) {
  switch (act.function) {
    case kActivationRelu:
      return relu_keep_nan(value);
    case kActivationGelu:
      if (act.approximate_tanh) {
        const float inner = 0.7978845608028654f * (value + 0.044715f * value * value * value);
        return 0.5f * value * (1.0f + tanhf(inner));
      }
      return 0.5f * value * (1.0f + erff(value * 0.7071067811865476f));
    default:  // SiLU: v / (1 + exp(-alpha v)), IEEE divide
      return value / (1.0f + expf(-act.alpha * value));
  }
}

__device__ __forceinline__ float apply_gated(float gate, float up, const ActivationArgs &act) {
  if (act.has_limit) {
    gate = fminf(gate, act.limit);
    up = fminf(fmaxf(up, -act.limit), act.limit);
  }
  return apply_function(gate, act) * (up + act.up_offset);
}

// ------------------------------------------------------------------ general projection
// out = x . w^T on the matrix cores for any K, N, row alignment and payload: BN weight rows
// (the MFMA's M operand) x BM token rows per 4-wave workgroup, K in slabs of 128 bytes per
// row.  Element type T is the weights' (fp32: v_mfma_f32_32x32x2, fp32 products and sums);
// XT is the tokens', widened while staging when T is fp32 (the Router's FP32 precision).
//
// Rows may start at any element (K = 2053 in bf16 leaves them 2-byte aligned), so slabs go
// through registers instead of direct buffer-to-LDS loads: 16-byte global loads (the
// hardware takes any alignment), one slab ahead, into the other of two LDS buffers, one
// barrier per slab.  LDS rows hold eight 16-byte chunks, chunk c of row r at c ^ (r / 2 % 8)
// as in the tile kernel.  Rows past the end read the last row (their products are not
// stored); columns past K, in the last slab only, are zero in both operands.
//
// A small grid is split over K (grid z): each range's fp32 sums go to `partials` and
// projection_reduce_kernel adds them in range order, so results are deterministic.
//
// Bound by the latency of a workgroup's slab chain below about 128 rows, by the rate of LDS
// staging above (bf16 1024 x 12288 x 2048: 570 TFLOP/s; fp32 2000 x 2002 x 2001: 108 TFLOP/s).
// The element-wise kernel this replaced (4 x 4 sums per thread on the vector pipes) took 1059
// us for bf16 130 x 2048 x 6144 (16.7 now), 362 us for 130 x 12288 x 2048 (27.0) and 496 us
// for fp32 257 x 1030 x 2053 (23.4).
constexpr int kSlabBytes = 128;

// The fp32 element type beside Bf16Payload / F16Payload: a 16-byte chunk holds 4 columns, and
// its MFMA step covers 8 (lane half h multiplies columns 4 h + j of both operands at step j).
struct F32Payload {
  __device__ static __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[j]), __uint_as_float(b[j]), c, 0, 0, 0);
    }
    return c;
  }
};

template <class T>
constexpr int kElementBytes = std::is_same_v<T, F32Payload> ? 4 : 2;
template <class T>
constexpr int kDtypeOf = std::is_same_v<T, F32Payload> ? kDtypeF32 : std::is_same_v<T, F16Payload> ? kDtypeF16 : kDtypeBf16;

// 16 (or 8) bytes from an address aligned to an element only.
__device__ __forceinline__ u32x4 load16_any(const unsigned char *address) {
  u32x4 value;
  __builtin_memcpy(&value, address, 16);
  return value;
}
__device__ __forceinline__ u32x2 load8_any(const unsigned char *address) {
  u32x2 value;
  __builtin_memcpy(&value, address, 8);
  return value;
}

// One LDS chunk (16 bytes of T) of a row at `source` (XT elements).
template <class XT, class T>
__device__ __forceinline__ u32x4 load_chunk(const unsigned char *source) {
  if constexpr (kElementBytes<XT> == kElementBytes<T>) {
    return load16_any(source);
  } else {
    const u32x2 packed = load8_any(source);
    return u32x4{__float_as_uint(XT::widen(packed[0] & 0xffffu)), __float_as_uint(XT::widen(packed[0] >> 16)),
                 __float_as_uint(XT::widen(packed[1] & 0xffffu)), __float_as_uint(XT::widen(packed[1] >> 16))};
  }
}

// The same where only `valid` (fewer than a chunk's) columns are left: zeros past them.
template <class XT, class T>
__device__ __forceinline__ u32x4 load_chunk_tail(const unsigned char *source, int64_t valid) {
  u32x4 chunk = {0u, 0u, 0u, 0u};
  if constexpr (kElementBytes<T> == 4) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < valid) {
        chunk[j] = kElementBytes<XT> == 4 ? reinterpret_cast<const uint32_t *>(source)[j]
                                          : __float_as_uint(load_value(source, j, kDtypeOf<XT>));
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < valid) {
        chunk[j / 2] |= static_cast<uint32_t>(reinterpret_cast<const uint16_t *>(source)[j]) << (16 * (j % 2));
      }
    }
  }
  return chunk;
}

// Bias, rounding point and activation of four consecutive weight rows' sums, and the store:
// n is a multiple of 4, `out` the token's output row.
template <class T>
__device__ __forceinline__ void store_outputs(const ProjectionArgs &a, f32x4 sum, int64_t n, int64_t token) {
  constexpr int dtype = kDtypeOf<T>;
  const int valid = a.n - n < 4 ? static_cast<int>(a.n - n) : 4;
  float value[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    value[j] = sum[j] + (a.bias != nullptr && j < valid ? a.bias[n + j] : 0.0f);
  }
  if (a.act.gated) {
    // N is even: a Gate/Up pair is whole or absent.
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      value[j / 2] = apply_gated(round_to(value[j], dtype), round_to(value[j + 1], dtype), a.act);
    }
  } else if (a.act.function != kActivationNone) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      value[j] = apply_function(round_to(value[j], dtype), a.act);
    }
  }
  const int64_t first = a.act.gated ? token * (a.n / 2) + n / 2 : token * a.n + n;
  const int count = a.act.gated ? valid / 2 : valid;
  if constexpr (kElementBytes<T> == 4) {
    float *out = static_cast<float *>(a.out) + first;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < count) {
        out[j] = value[j];
      }
    }
  } else {
    uint16_t *out = static_cast<uint16_t *>(a.out) + first;
    const u32x2 packed = {T::pack2(value[0], value[1]), T::pack2(value[2], value[3])};
    if (count == 4) {
      __builtin_memcpy(out, &packed, 8);
    } else if (count == 2) {
      __builtin_memcpy(out, &packed, 4);
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if (j < count) {
          out[j] = static_cast<uint16_t>(packed[j / 2] >> (16 * (j % 2)));
        }
      }
    }
  }
}

template <class XT, class T, int BM, int BN>
__global__ __launch_bounds__(256) void projection_kernel(ProjectionArgs a) {
  constexpr int XS = kElementBytes<XT>;
  constexpr int WS = kElementBytes<T>;
  constexpr int BK = kSlabBytes / WS;    // columns per slab
  constexpr int CHUNK = 16 / WS;         // columns per chunk
  constexpr int MT = BM / 64;            // 32-token tiles per wave
  constexpr int NT = BN / 64;            // 32-weight-row tiles per wave
  constexpr int X_LOADS = BM / 32;       // chunks per thread and slab
  constexpr int W_LOADS = BN / 32;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][(BM + BN) * kSlabBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wn = wave & 1;
  const int wm = wave >> 1;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * BN;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * BM;
  if (m0 >= a.rows) {
    return;  // a grid sized for more rows than are live
  }
  const int64_t k_begin = static_cast<int64_t>(blockIdx.z) * a.k_slice;
  const int64_t k_end = a.k - k_begin < a.k_slice ? a.k : k_begin + a.k_slice;
  const int slabs = static_cast<int>((k_end - k_begin + BK - 1) / BK);

  // Thread t stages chunk t % 8 of rows t / 8, t / 8 + 32, ... of both tiles.
  const int chunk = threadIdx.x & 7;
  const int row0 = threadIdx.x >> 3;
  const unsigned char *x_source[X_LOADS];
  const unsigned char *w_source[W_LOADS];
  int x_slot[X_LOADS];
  int w_slot[W_LOADS];
#pragma unroll
  for (int q = 0; q < X_LOADS; ++q) {
    const int row = row0 + 32 * q;
    const int64_t token = m0 + row < a.rows ? m0 + row : a.rows - 1;
    x_source[q] = static_cast<const unsigned char *>(a.x) + (token * a.k + k_begin + chunk * CHUNK) * XS;
    x_slot[q] = (BN + row) * kSlabBytes + ((chunk ^ ((row >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int q = 0; q < W_LOADS; ++q) {
    const int row = row0 + 32 * q;
    const int64_t weight = n0 + row < a.n ? n0 + row : a.n - 1;
    w_source[q] = static_cast<const unsigned char *>(a.w) + (weight * a.k + k_begin + chunk * CHUNK) * WS;
    w_slot[q] = row * kSlabBytes + ((chunk ^ ((row >> 1) & 7)) << 4);
  }
  u32x4 x_next[X_LOADS];
  u32x4 w_next[W_LOADS];
  auto fetch = [&](int slab) __attribute__((always_inline)) {
    const int64_t column = static_cast<int64_t>(slab) * BK;
    if (k_begin + column + BK <= k_end) {
#pragma unroll
      for (int q = 0; q < W_LOADS; ++q) {
        w_next[q] = load_chunk<T, T>(w_source[q] + column * WS);
      }
#pragma unroll
      for (int q = 0; q < X_LOADS; ++q) {
        x_next[q] = load_chunk<XT, T>(x_source[q] + column * XS);
      }
    } else {
      const int64_t valid = k_end - k_begin - column - chunk * CHUNK;
#pragma unroll
      for (int q = 0; q < W_LOADS; ++q) {
        w_next[q] = valid >= CHUNK ? load_chunk<T, T>(w_source[q] + column * WS)
                                   : load_chunk_tail<T, T>(w_source[q] + column * WS, valid);
      }
#pragma unroll
      for (int q = 0; q < X_LOADS; ++q) {
        x_next[q] = valid >= CHUNK ? load_chunk<XT, T>(x_source[q] + column * XS)
                                   : load_chunk_tail<XT, T>(x_source[q] + column * XS, valid);
      }
    }
  };
  auto stage = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < W_LOADS; ++q) {
      *reinterpret_cast<u32x4 *>(lds[buffer] + w_slot[q]) = w_next[q];
    }
#pragma unroll
    for (int q = 0; q < X_LOADS; ++q) {
      *reinterpret_cast<u32x4 *>(lds[buffer] + x_slot[q]) = x_next[q];
    }
  };

  f32x16 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[nt][mt][r] = 0.0f;
      }
    }
  }
  const int frag_row = lane & 31;
  const int frag_half = lane >> 5;
  const int swizzle = (frag_row >> 1) & 7;  // unchanged by the multiples of 32 added below
  const int w_frag = (wn * (BN / 2) + frag_row) * kSlabBytes;
  const int x_frag = (BN + wm * (BM / 2) + frag_row) * kSlabBytes;
  auto compute = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int place = ((2 * ks + frag_half) ^ swizzle) << 4;
      u32x4 w_chunk[NT];
      u32x4 x_chunk[MT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        w_chunk[nt] = *reinterpret_cast<const u32x4 *>(lds[buffer] + w_frag + nt * 32 * kSlabBytes + place);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        x_chunk[mt] = *reinterpret_cast<const u32x4 *>(lds[buffer] + x_frag + mt * 32 * kSlabBytes + place);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[nt][mt] = T::mfma32(w_chunk[nt], x_chunk[mt], acc[nt][mt]);
        }
      }
    }
  };

  fetch(0);
  stage(0);
  __syncthreads();
  for (int slab = 0; slab < slabs; ++slab) {
    const bool more = slab + 1 < slabs;
    if (more) {
      fetch(slab + 1);
    }
    compute(slab & 1);
    if (more) {
      stage((slab + 1) & 1);  // last read two slabs ago, before the previous barrier
    }
    __syncthreads();
  }

  // Lane holds D[8 (r / 4) + 4 (lane / 32) + r % 4][lane % 32]: four consecutive weight rows
  // of one token per r / 4.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int64_t token = m0 + wm * (BM / 2) + mt * 32 + frag_row;
    if (token >= a.rows) {
      continue;
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int quad = 0; quad < 4; ++quad) {
        const int64_t n = n0 + wn * (BN / 2) + nt * 32 + 8 * quad + 4 * frag_half;
        if (n >= a.n) {
          continue;
        }
        const f32x4 sum = {acc[nt][mt][4 * quad], acc[nt][mt][4 * quad + 1], acc[nt][mt][4 * quad + 2],
                           acc[nt][mt][4 * quad + 3]};
        if (a.partials != nullptr) {
          float *plane = a.partials + (static_cast<int64_t>(blockIdx.z) * a.rows + token) * a.n + n;
          if (n + 4 <= a.n) {
            __builtin_memcpy(plane, &sum, 16);
          } else {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              if (n + j < a.n) {
                plane[j] = sum[j];
              }
            }
          }
        } else {
          store_outputs<T>(a, sum, n, token);
        }
      }
    }
  }
}

// Sums of the K ranges' partials [ranges, rows, n] in range order, then the epilogue: one
// thread per four consecutive weight rows of one token.
template <class T>
__global__ __launch_bounds__(256) void projection_reduce_kernel(ProjectionArgs a) {
  const int64_t quads = (a.n + 3) / 4;
  const int64_t index = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t token = index / quads;
  if (token >= a.rows) {
    return;
  }
  const int64_t n = (index - token * quads) * 4;
  const int64_t ranges = (a.k + a.k_slice - 1) / a.k_slice;
  const int64_t plane = a.rows * a.n;
  const float *source = a.partials + token * a.n + n;
  const bool whole = n + 4 <= a.n;
  auto partial = [&](int64_t range) {
    f32x4 value = {0.0f, 0.0f, 0.0f, 0.0f};
    const float *address = source + range * plane;
    if (whole) {
      __builtin_memcpy(&value, address, 16);
    } else {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        value[j] = n + j < a.n ? address[j] : 0.0f;
      }
    }
    return value;
  };
  // Four ranges' loads are issued together; the additions keep range order.
  f32x4 sum = partial(0);
  int64_t range = 1;
  for (; range + 4 <= ranges; range += 4) {
    const f32x4 p0 = partial(range), p1 = partial(range + 1), p2 = partial(range + 2), p3 = partial(range + 3);
    sum += p0;
    sum += p1;
    sum += p2;
    sum += p3;
  }
  for (; range < ranges; ++range) {
    sum += partial(range);
  }
  store_outputs<T>(a, sum, n, token);
}

// ------------------------------------------------------------------ standalone activation
// One thread per output element (grid-stride): gated reads Gate and Up from the layout the
// order names; ungated ReLU works on the raw 16-bit patterns (bit-exact, in place allowed).
__global__ __launch_bounds__(256) void activation_kernel(ActivationLaunchArgs a) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t index = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; index < a.elements;
       index += stride) {
    if (!a.act.gated) {
      if (a.act.function == kActivationRelu) {
        const uint16_t bits = reinterpret_cast<const uint16_t *>(a.inputs)[index];
        const float value = load_value(a.inputs, index, a.dtype);
        reinterpret_cast<uint16_t *>(a.output)[index] = (value > 0.0f || value != value) ? bits : uint16_t{0};
      } else {
        store_value(a.output, index, apply_function(load_value(a.inputs, index, a.dtype), a.act), a.dtype);
      }
      continue;
    }
    const int64_t row = index / a.width;
    const int64_t column = index - row * a.width;
    const int64_t gate_at = a.interleaved ? row * 2 * a.width + 2 * column : row * 2 * a.width + column;
    const int64_t up_at = a.interleaved ? gate_at + 1 : gate_at + a.width;
    const float gate = load_value(a.inputs, gate_at, a.dtype);
    const float up = load_value(a.inputs, up_at, a.dtype);
    store_value(a.output, index, apply_gated(gate, up, a.act), a.dtype);
  }
}

}  // namespace

// Tile and K ranges of a projection from a cost model in microseconds.  A workgroup's slabs
// follow one another at no less than the slab latency, and a CU's workgroups share its
// throughput; a K split adds the reduction launch and its sums' traffic.  Measured on MI355X
// (weights rotated over three copies), least time over forced tiles and ranges against the
// time of this choice: bf16 1 x 12288 x 2048 13.1 / 13.1 us (4 ranges; 16 ranges 16.9),
// 130 x 2048 x 6144 16.7 / 16.7 us (8; unsplit 51), 130 x 12288 x 2048 27.0 / 27.0 us
// (unsplit; 3 ranges 29.1), 1024 x 2048 x 6144 46.7 / 46.7 us (128 x 128 tiles, 4 ranges; 64 x
// 64 unsplit 58.7), a Router's 2048 x 128 x 2048 11.1 / 11.1 us (4; 16 ranges 17.5); fp32
// 257 x 1030 x 2053 23.4 / 23.4 us (6; unsplit 51.9), 2000 x 2002 x 2001 148.5 / 148.5 us.
struct ProjectionCost {
  int tile;
  double latency;     // us per slab of one workgroup on an idle CU
  double throughput;  // us per slab of a CU with several workgroups
};
constexpr ProjectionCost kProjectionCosts16[] = {{64, 0.33, 0.27}, {128, 1.37, 0.885}};
constexpr ProjectionCost kProjectionCosts32[] = {{64, 0.72, 0.59}, {128, 2.5, 2.2}};
constexpr double kProjectionLaunchUs = 4.7;
constexpr double kProjectionReduceUs = 2.5;
constexpr double kProjectionPartialBytesPerUs = 16e6;
constexpr double kProjectionCus = 256.0;
constexpr int64_t kProjectionMaxRanges = 16;
constexpr int64_t kProjectionMinSlabs = 2;  // per range

ProjectionPlan plan_projection(int64_t rows, int64_t n, int64_t k, int element_bytes, size_t scratch_bytes) {
  const int64_t slab = kSlabBytes / element_bytes;
  const int64_t slabs = (k + slab - 1) / slab;
  const int64_t plane_bytes = rows * n * 4;
  // Priced at whole 64-row tiles: the choice then changes only with their number, which makes
  // projection_scratch_bytes exact.
  const int64_t whole_plane_bytes = (rows + 63) / 64 * 64 * n * 4;
  ProjectionPlan best{64, 1, k, 0.0};
  double best_us = -1.0;
  for (const ProjectionCost &cost : element_bytes == 4 ? kProjectionCosts32 : kProjectionCosts16) {
    const int64_t tiles = ((rows + cost.tile - 1) / cost.tile) * ((n + cost.tile - 1) / cost.tile);
    for (int64_t ranges = 1; ranges <= kProjectionMaxRanges; ++ranges) {
      const int64_t per_range = (slabs + ranges - 1) / ranges;
      if (ranges > 1 && (per_range < kProjectionMinSlabs || (ranges - 1) * per_range >= slabs ||
                         static_cast<uint64_t>(ranges * plane_bytes) > scratch_bytes)) {
        continue;
      }
      // 64 x 64 workgroups run in whole rounds of the chip; a CU holds few 128 x 128 ones.
      const double per_cu = static_cast<double>(tiles * ranges) / kProjectionCus;
      const double rounds = cost.tile == 64 ? std::ceil(per_cu) : per_cu;
      double us = static_cast<double>(per_range) * std::max(cost.latency, rounds * cost.throughput);
      if (ranges > 1) {
        us += kProjectionReduceUs + 2.0 * static_cast<double>(ranges * whole_plane_bytes) / kProjectionPartialBytesPerUs;
      }
      if (best_us < 0.0 || us < best_us) {
        best = {cost.tile, ranges, ranges > 1 ? per_range * slab : k, kProjectionLaunchUs + us};
        best_us = us;
      }
    }
  }
  return best;
}

size_t projection_scratch_bytes(int64_t capacity, int64_t n, int64_t k, int element_bytes) {
  size_t most = 0;
  for (int64_t rows = 64; rows < capacity + 64; rows += 64) {
    const int64_t live = std::min(rows, capacity);
    const ProjectionPlan plan = plan_projection(live, n, k, element_bytes, static_cast<size_t>(INT64_MAX));
    if (plan.ranges > 1) {
      most = std::max(most, static_cast<size_t>(plan.ranges * live * n) * sizeof(float));
    }
  }
  return most;
}

template <class XT, class T>
const void *projection_kernel_for(int tile) {
  return tile == 128 ? reinterpret_cast<const void *>(&projection_kernel<XT, T, 128, 128>)
                     : reinterpret_cast<const void *>(&projection_kernel<XT, T, 64, 64>);
}

ProjectionLaunch make_projection(const ProjectionArgs &args, const ProjectionPlan &plan, int64_t capacity, int x_dtype) {
  ProjectionLaunch launches;
  ProjectionArgs record = args;
  record.k_slice = plan.k_slice;
  launches.main.func = args.dtype == kDtypeF32
                           ? (x_dtype == kDtypeF32   ? projection_kernel_for<F32Payload, F32Payload>(plan.tile)
                              : x_dtype == kDtypeF16 ? projection_kernel_for<F16Payload, F32Payload>(plan.tile)
                                                     : projection_kernel_for<Bf16Payload, F32Payload>(plan.tile))
                       : args.dtype == kDtypeF16 ? projection_kernel_for<F16Payload, F16Payload>(plan.tile)
                                                 : projection_kernel_for<Bf16Payload, Bf16Payload>(plan.tile);
  launches.main.grid = dim3(static_cast<unsigned>((args.n + plan.tile - 1) / plan.tile),
                            static_cast<unsigned>((capacity + plan.tile - 1) / plan.tile),
                            static_cast<unsigned>(plan.ranges));
  launches.main.block = dim3(256, 1, 1);
  launches.main.set_args(record);
  if (plan.ranges > 1) {
    launches.reduce = make_projection_reduce(record, capacity);
  }
  return launches;
}

KernelLaunch make_projection_reduce(const ProjectionArgs &args, int64_t capacity) {
  KernelLaunch reduce;
  reduce.func = args.dtype == kDtypeF32   ? reinterpret_cast<const void *>(&projection_reduce_kernel<F32Payload>)
                : args.dtype == kDtypeF16 ? reinterpret_cast<const void *>(&projection_reduce_kernel<F16Payload>)
                                          : reinterpret_cast<const void *>(&projection_reduce_kernel<Bf16Payload>);
  reduce.grid = dim3(static_cast<unsigned>((capacity * ((args.n + 3) / 4) + 255) / 256), 1, 1);
  reduce.block = dim3(256, 1, 1);
  reduce.set_args(args);
  return reduce;
}

KernelLaunch make_activation(const ActivationLaunchArgs &args) {
  KernelLaunch kernel;
  kernel.func = reinterpret_cast<const void *>(&activation_kernel);
  const int64_t blocks = (args.elements + 255) / 256;
  kernel.grid = dim3(static_cast<unsigned>(blocks < 4096 ? (blocks > 0 ? blocks : 1) : 4096), 1, 1);
  kernel.block = dim3(256, 1, 1);
  kernel.set_args(args);
  return kernel;
}

}  // namespace xp
