// Elementwise (pointwise) maps for gfx950, f32 and bf16 storage.
//
// Reference arithmetic: tiler-reference/src/evaluate.rs:448-485 `binary`
// (operand/result conformance around canon(op(l, r)), rank-0 operands
// broadcast); the emitted forms are tiler-metal's goldens
// pointwise_scale_bias{,_bf16}.metal:41-58 (one statement per operation, NaN
// canonicalized per result) and elementary_silu_activation.metal:41-62.
//
// bf16 storage computes each operation in binary32 on exactly widened operands
// and narrows the one result (ADR 0091 decision 2).  For a single add or
// multiply that equals the exact-rational bf16 result of
// tiler-reference/src/bf16.rs: binary32 carries 24 >= 2*8+2 bits, so the
// double rounding is innocuous; scale-bias is two operations and narrows after
// each, as the bf16 golden does.
//
// Ops: 0 scale-bias y = x*a + b (two roundings), 1 SiLU, 2 add, 3 multiply.
// `x2` is the second operand of add/multiply; x2_stride 0 broadcasts a rank-0
// operand, 1 reads it elementwise.
#include "common.h"

using tiler::canon;

namespace {

__device__ __forceinline__ float map_op(uint32_t op, float x, float x2, float a, float b) {
  switch (op) {
    case 0: {
      float t = canon(x * a);
      return canon(t + b);
    }
    case 1:
      return canon(tiler::silu_f32(x));
    case 2:
      return canon(x + x2);
    default:
      return canon(x * x2);
  }
}

__device__ __forceinline__ float map_op_bf16(uint32_t op, float x, float x2, float a, float b) {
  switch (op) {
    case 0: {
      float t = tiler::bf16_widen(tiler::bf16_narrow(x * a));
      return t + b;
    }
    case 1:
      return tiler::silu_f32(x);
    case 2:
      return x + x2;
    default:
      return x * x2;
  }
}

// The same operations under the declared subnormal modes, at every site as
// evaluate.rs:448-485 `binary` applies them (apply_to_result(canon(op(
// apply_to_operand(l), apply_to_operand(r))))), and the SiLU as
// silu.rs:511-533 silu_f32_under.
__device__ __forceinline__ float map_op_modes(uint32_t op, float x, float x2, float a, float b, uint32_t im,
                                              uint32_t rm) {
  using tiler::subnormal;
  switch (op) {
    case 0: {
      const float t = canon(subnormal(rm, subnormal(im, x) * subnormal(im, a)));
      return canon(subnormal(rm, subnormal(im, t) + subnormal(im, b)));
    }
    case 1: {
      if (x != x) return canon(x);
      if (x == __builtin_huge_valf()) return x;
      if (x == -__builtin_huge_valf()) return __uint_as_float(TILER_CANONICAL_F32_NAN);
      const float v = subnormal(im, x);
      const float e = subnormal(rm, tiler::exp_f32_cr(subnormal(im, -v)));
      const float divisor = subnormal(rm, 1.0f + subnormal(im, e));
      return canon(subnormal(rm, subnormal(im, v) / subnormal(im, divisor)));
    }
    case 2:
      return canon(subnormal(rm, subnormal(im, x) + subnormal(im, x2)));
    default:
      return canon(subnormal(rm, subnormal(im, x) * subnormal(im, x2)));
  }
}

// bf16 under the modes (bf16.rs:517-533): the input dimension replaces a
// subnormal operand encoding before it is read, the result dimension a
// subnormal rounded result; each operation rounds once to bf16.
__device__ __forceinline__ float bf16_commit(float r, uint32_t rm) {
  return tiler::subnormal(rm, tiler::bf16_widen(tiler::bf16_narrow(r)));
}
__device__ __forceinline__ float map_op_bf16_modes(uint32_t op, float x, float x2, float a, float b, uint32_t im,
                                                   uint32_t rm) {
  using tiler::subnormal;
  switch (op) {
    case 0: {
      const float t = bf16_commit(subnormal(im, x) * subnormal(im, a), rm);
      return bf16_commit(subnormal(im, t) + subnormal(im, b), rm);
    }
    case 2:
      return bf16_commit(subnormal(im, x) + subnormal(im, x2), rm);
    default:
      return bf16_commit(subnormal(im, x) * subnormal(im, x2), rm);
  }
}

}  // namespace

// Scalar forms under the declared subnormal modes (a flushing contract).
extern "C" __global__ void __launch_bounds__(256)
tiler_map_f32_m(const float* __restrict__ x, const float* __restrict__ x2, uint64_t x2_stride, uint64_t n,
                uint32_t op, float a, float b, float* __restrict__ y, uint32_t in_mode, uint32_t out_mode) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float s2 = x2 ? x2[i * x2_stride] : 0.0f;
    y[i] = map_op_modes(op, x[i], s2, a, b, in_mode, out_mode);
  }
}

extern "C" __global__ void __launch_bounds__(256)
tiler_map_bf16_m(const uint16_t* __restrict__ x, const uint16_t* __restrict__ x2, uint64_t x2_stride, uint64_t n,
                 uint32_t op, float a, float b, uint16_t* __restrict__ y, uint32_t in_mode, uint32_t out_mode) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float s2 = x2 ? tiler::bf16_widen(x2[i * x2_stride]) : 0.0f;
    y[i] = (uint16_t)tiler::bf16_narrow(
        map_op_bf16_modes(op, tiler::bf16_widen(x[i]), s2, a, b, in_mode, out_mode));
  }
}

extern "C" __global__ void __launch_bounds__(256)
tiler_map_f32(const float* __restrict__ x, const float* __restrict__ x2, uint64_t x2_stride,
              uint64_t n, uint32_t op, float a, float b, float* __restrict__ y) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float s2 = x2 ? x2[i * x2_stride] : 0.0f;
    y[i] = map_op(op, x[i], s2, a, b);
  }
}

extern "C" __global__ void __launch_bounds__(256)
tiler_map_bf16(const uint16_t* __restrict__ x, const uint16_t* __restrict__ x2,
               uint64_t x2_stride, uint64_t n, uint32_t op, float a, float b,
               uint16_t* __restrict__ y) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    float s2 = x2 ? tiler::bf16_widen(x2[i * x2_stride]) : 0.0f;
    y[i] = (uint16_t)tiler::bf16_narrow(map_op_bf16(op, tiler::bf16_widen(x[i]), s2, a, b));
  }
}

// Vectorized maps: 16 bytes per lane per step (4 f32 or 8 bf16 elements),
// non-temporal loads and stores (f32 results of 48 to 128 MiB: ordinary stores,
// tiler::keep_in_cache), the op and the rank-0 broadcast of x2 fixed at compile
// time.  Every element sees exactly the scalar kernels' arithmetic.
// The host uses them on 16-byte-aligned operands for the whole 16-byte chunks
// and the scalar kernels for the tail.
template <uint32_t OP, bool BCAST, bool kKeep>
__device__ __forceinline__ void map_f32_v4_body(const f32x4* __restrict__ x, const float* __restrict__ x2,
                                                uint64_t n4, float a, float b, f32x4* __restrict__ y) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const float s2b = (OP >= 2 && BCAST) ? x2[0] : 0.0f;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
    const f32x4 v = __builtin_nontemporal_load(&x[i]);
    f32x4 s2 = {s2b, s2b, s2b, s2b};
    if (OP >= 2 && !BCAST) s2 = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x2) + i);
    const f32x4 o = {map_op(OP, v.x, s2.x, a, b), map_op(OP, v.y, s2.y, a, b),
                     map_op(OP, v.z, s2.z, a, b), map_op(OP, v.w, s2.w, a, b)};
    tiler::store_result<kKeep>(o, &y[i]);
  }
}

template <uint32_t OP, bool BCAST>
__device__ __forceinline__ void map_bf16_v8_body(const u32x4* __restrict__ x, const uint16_t* __restrict__ x2,
                                                 uint64_t n8, float a, float b, u32x4* __restrict__ y) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const float s2b = (OP >= 2 && BCAST) ? tiler::bf16_widen(x2[0]) : 0.0f;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += stride) {
    const u32x4 v = __builtin_nontemporal_load(&x[i]);
    u32x4 w = {0, 0, 0, 0};
    if (OP >= 2 && !BCAST) w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x2) + i);
    u32x4 o;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const float x0 = tiler::bf16_widen(v[h] & 0xffffu), x1 = tiler::bf16_widen(v[h] >> 16);
      const float w0 = (OP >= 2 && !BCAST) ? tiler::bf16_widen(w[h] & 0xffffu) : s2b;
      const float w1 = (OP >= 2 && !BCAST) ? tiler::bf16_widen(w[h] >> 16) : s2b;
      o[h] = tiler::bf16_narrow(map_op_bf16(OP, x0, w0, a, b)) |
             (tiler::bf16_narrow(map_op_bf16(OP, x1, w1, a, b)) << 16);
    }
    __builtin_nontemporal_store(o, &y[i]);
  }
}

#define TILER_MAP_VEC(OP, BC, SFX)                                                                 \
  extern "C" __global__ void __launch_bounds__(256) tiler_map_f32_v4_op##OP##SFX(                    \
      const f32x4* __restrict__ x, const float* __restrict__ x2, uint64_t n4, float a, float b,      \
      f32x4* __restrict__ y) {                                                                       \
    if (tiler::keep_in_cache(n4 * 16u)) map_f32_v4_body<OP, BC, true>(x, x2, n4, a, b, y);            \
    else map_f32_v4_body<OP, BC, false>(x, x2, n4, a, b, y);                                         \
  }                                                                                                  \
  extern "C" __global__ void __launch_bounds__(256) tiler_map_bf16_v8_op##OP##SFX(                   \
      const u32x4* __restrict__ x, const uint16_t* __restrict__ x2, uint64_t n8, float a, float b,   \
      u32x4* __restrict__ y) {                                                                       \
    map_bf16_v8_body<OP, BC>(x, x2, n8, a, b, y);                                                    \
  }
TILER_MAP_VEC(0, false, )
TILER_MAP_VEC(1, false, )
TILER_MAP_VEC(2, false, )
TILER_MAP_VEC(2, true, _b)
TILER_MAP_VEC(3, false, )
TILER_MAP_VEC(3, true, _b)

// Broadcast / reindex (tiler-reference/src/structural.rs:75-108): a pure move.
// out element o (row-major over out_dims) reads source offset
// base + sum_d coord_d(o) * src_stride_d; a broadcast axis has stride 0, a
// reversed axis a negative stride (two's complement: the sum wraps modulo
// 2^64 to the in-range offset the host proved, as the mirrored reindex
// golden's `1 - i%2` does).  Rank <= 8.
struct BroadcastGeometry {
  uint64_t out_dims[8];
  uint64_t src_strides[8];
  uint32_t rank;
  uint64_t base;
};

template <typename T>
__device__ __forceinline__ void broadcast_body(const T* __restrict__ src, T* __restrict__ out,
                                               uint64_t n, const BroadcastGeometry& g) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint64_t rem = i, off = g.base;
    for (int d = (int)g.rank - 1; d >= 0; --d) {
      uint64_t c = rem % g.out_dims[d];
      rem /= g.out_dims[d];
      off += c * g.src_strides[d];
    }
    out[i] = src[off];
  }
}

// Row mode (innermost out dimension >= 256): each workgroup step takes one
// out row, decodes its source row offset once, and copies the row -- in
// 16-byte vectors when the row is contiguous in the source and both rows are
// 16-byte aligned, as a replicated fill when the inner axis broadcasts (stride
// 0), element by element otherwise.
template <typename T>
__device__ __forceinline__ void broadcast_rows_body(const T* __restrict__ src, T* __restrict__ out,
                                                    uint64_t rows, const BroadcastGeometry& g) {
  constexpr uint32_t kPer = 16 / sizeof(T);
  const uint64_t inner = g.out_dims[g.rank - 1], sin = g.src_strides[g.rank - 1];
  for (uint64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    uint64_t rem = r, base = g.base;
    for (int d = (int)g.rank - 2; d >= 0; --d) {
      const uint64_t c = rem % g.out_dims[d];
      rem /= g.out_dims[d];
      base += c * g.src_strides[d];
    }
    const T* s = src + base;
    T* o = out + r * inner;
    const bool vec = ((uintptr_t)o & 15u) == 0 && inner % kPer == 0 &&
                     (sin == 0 || (sin == 1 && ((uintptr_t)s & 15u) == 0));
    if (vec) {
      const uint64_t chunks = inner / kPer;
      if (sin == 0) {
        const T v = s[0];
        T lanes[kPer];
#pragma unroll
        for (uint32_t e = 0; e < kPer; ++e) lanes[e] = v;
        u32x4 fill;
        __builtin_memcpy(&fill, lanes, 16);
        for (uint64_t q = threadIdx.x; q < chunks; q += blockDim.x)
          __builtin_nontemporal_store(fill, reinterpret_cast<u32x4*>(o) + q);
      } else {
        for (uint64_t q = threadIdx.x; q < chunks; q += blockDim.x)
          __builtin_nontemporal_store(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(s) + q),
                                      reinterpret_cast<u32x4*>(o) + q);
      }
    } else {
      for (uint64_t j = threadIdx.x; j < inner; j += blockDim.x) o[j] = s[j * sin];
    }
  }
}

extern "C" __global__ void __launch_bounds__(256)
tiler_broadcast_rows_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ out, uint64_t rows,
                         BroadcastGeometry g) {
  broadcast_rows_body<uint32_t>(src, out, rows, g);
}
extern "C" __global__ void __launch_bounds__(256)
tiler_broadcast_rows_u16(const uint16_t* __restrict__ src, uint16_t* __restrict__ out, uint64_t rows,
                         BroadcastGeometry g) {
  broadcast_rows_body<uint16_t>(src, out, rows, g);
}

extern "C" __global__ void __launch_bounds__(256)
tiler_broadcast_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ out, uint64_t n,
                    BroadcastGeometry g) {
  broadcast_body<uint32_t>(src, out, n, g);
}
extern "C" __global__ void __launch_bounds__(256)
tiler_broadcast_u16(const uint16_t* __restrict__ src, uint16_t* __restrict__ out, uint64_t n,
                    BroadcastGeometry g) {
  broadcast_body<uint16_t>(src, out, n, g);
}

// Fill: dst[i] = value for i < words.  A kernel rather than a memset so that a
// captured graph holds kernel nodes only.
extern "C" __global__ void __launch_bounds__(256)
tiler_fill_u32(uint32_t* __restrict__ dst, uint32_t value, uint64_t words) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += stride)
    dst[i] = value;
}

// Subnormal probe: the f32 subnormal handling this code object delivers on
// the live device, measured rather than assumed.  in[] holds the operands, so
// nothing folds at compile time:
//   out[0] = in[0] * in[1]: -2^-149 (a subnormal input) times 2^30, whose
//            exact product -2^-119 is normal -- the input side;
//   out[1] = in[2] * in[3]: 2^-120 times -2^-10, whose exact product -2^-130
//            is subnormal -- the result side.
extern "C" __global__ void __launch_bounds__(64)
tiler_probe_subnormals(const float* __restrict__ in, uint32_t* __restrict__ out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    out[0] = __float_as_uint(in[0] * in[1]);
    out[1] = __float_as_uint(in[2] * in[3]);
  }
}
