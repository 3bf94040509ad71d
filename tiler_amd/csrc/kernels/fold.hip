// Serial folds over any reduced-axis set, one invocation per output -- the
// emitted form of tiler-ir's emit_reduction / emit_maximum_reduction
// (tiler-ir/src/kernel/lower.rs:1236-1305, 2485-2500; tiler-metal goldens
// reduction_single_axis, reduction_multi_axis, reduction_fused_multiply_add):
//   StrictSerialSum               acc = canon(acc + x)
//   SquaredSerialSum              acc = canon(acc + canon(x * x))
//   FusedMultiplyAddSerialSum     acc = canon(acc + canon(canon(x * scale) + bias))
//                                 (contraction is permitted, never required:
//                                 the unfused form is what every contract admits)
//   StrictSerialMaximum           acc = maximum(acc, x), NaN-propagating,
//                                 -0 < +0 (tiler-reference/src/softmax.rs:168-186)
// over the contributors in lexicographic order of the reduced coordinates
// (tiler-reference/src/evaluate.rs:548-585), seeded at the first contributor.
// Seeding a sum at -0.0 and adding every (canonical) contributor value is the
// same bits: -0.0 is the exact additive identity, and each combine is
// canonicalized; a maximum seeded at -inf likewise (-inf is its two-sided
// identity, model.rs:889-900).  The sums' result is canonicalized; an empty
// sum commits the identity bits.  An optional one-input epilogue program
// (SquaredSerialSumThenEpilogue, model.rs:815-830) transforms the folded value.
//
// Where the reduced axes are adjacent the tensor is [outer, reduced, inner]
// and three further forms give the same bits (plan_fold chooses):
//   tiler_fold_*_f32_lanes  inner > 1, many outputs: a lane per output, its
//                           loads a batch ahead of its chain;
//   tiler_fold_*_f32_cols   inner > 1, fewer outputs: a workgroup per 16
//                           columns, the rows staged through LDS;
//   tiler_fold_maximum_f32_rows  inner == 1, a wave or a workgroup per row
//                           (the sums over rows are the staged sum kernels).
#include "common.h"

namespace {

// Kept axes first (output order), then reduced axes (contributor order); each
// with its dense input stride in elements.
struct FoldGeometry {
  uint64_t dims[8];
  uint64_t strides[8];
  uint32_t kept_rank, red_rank;
};

enum : uint32_t { kFoldSum = 0, kFoldSquared = 1, kFoldFma = 2, kFoldMaximum = 3 };

template <uint32_t OP>
__device__ __forceinline__ void fold_body(const float* __restrict__ x, float* __restrict__ out,
                                          uint64_t outputs, uint64_t contributors, const FoldGeometry& g,
                                          float scale, float bias, uint32_t empty_bits,
                                          const ExprInstr* __restrict__ epi, uint32_t epi_count,
                                          uint32_t epi_result) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t id = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; id < outputs; id += stride) {
    uint64_t rem = id, base = 0;
    for (int d = (int)g.kept_rank - 1; d >= 0; --d) {
      const uint64_t c = rem % g.dims[d];
      rem /= g.dims[d];
      base += c * g.strides[d];
    }
    float acc = OP == kFoldMaximum ? -__builtin_huge_valf() : -0.0f;
    uint64_t coord[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    uint64_t off = base;
    const uint32_t r0 = g.kept_rank, rn = g.kept_rank + g.red_rank;
    for (uint64_t p = 0; p < contributors; ++p) {
      const float v = x[off];
      if (OP == kFoldMaximum) {
        acc = tiler::maximum_f32(acc, v);
      } else {
        float t = v;
        if (OP == kFoldSquared) t = tiler::canon(v * v);
        if (OP == kFoldFma) t = tiler::canon(tiler::canon(v * scale) + bias);
        acc = tiler::canon(acc + t);
      }
      // odometer over the reduced axes, last axis fastest
      for (int d = (int)rn - 1; d >= (int)r0; --d) {
        off += g.strides[d];
        if (++coord[d] < g.dims[d]) break;
        off -= g.strides[d] * g.dims[d];
        coord[d] = 0;
      }
    }
    float total = contributors == 0 ? __uint_as_float(empty_bits) : tiler::canon(acc);
    if (epi) total = expr_epilogue_f32(epi, epi_count, epi_result, total);
    out[id] = total;
  }
}

// The sums under a FoldRule: its prologue and the declared subnormal modes at
// every arithmetic site, seeded at the first contributor (the form a flushing
// contract realizes as; the maximum compares and takes no mode).
__device__ __forceinline__ void fold_rule_body(const float* __restrict__ x, float* __restrict__ out,
                                               uint64_t outputs, uint64_t contributors, const FoldGeometry& g,
                                               const tiler::FoldRule& rule, uint32_t empty_bits) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t id = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; id < outputs; id += stride) {
    uint64_t rem = id, base = 0;
    for (int d = (int)g.kept_rank - 1; d >= 0; --d) {
      const uint64_t c = rem % g.dims[d];
      rem /= g.dims[d];
      base += c * g.strides[d];
    }
    float acc = 0.0f;
    uint64_t coord[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    uint64_t off = base;
    const uint32_t r0 = g.kept_rank, rn = g.kept_rank + g.red_rank;
    for (uint64_t p = 0; p < contributors; ++p) {
      const float t = tiler::fold_contributor(rule, x[off]);
      acc = p == 0 ? t : tiler::fold_combine(rule, acc, t);
      for (int d = (int)rn - 1; d >= (int)r0; --d) {
        off += g.strides[d];
        if (++coord[d] < g.dims[d]) break;
        off -= g.strides[d] * g.dims[d];
        coord[d] = 0;
      }
    }
    out[id] = contributors == 0 ? __uint_as_float(empty_bits) : tiler::canon(acc);
  }
}

}  // namespace

extern "C" __global__ void __launch_bounds__(256)
tiler_fold_f32_m(const float* __restrict__ x, float* __restrict__ out, uint64_t outputs, uint64_t contributors,
                 FoldGeometry g, tiler::FoldRule rule, uint32_t empty_bits) {
  fold_rule_body(x, out, outputs, contributors, g, rule, empty_bits);
}

#define TILER_FOLD(NAME, OP)                                                                         \
  extern "C" __global__ void __launch_bounds__(256) NAME(                                            \
      const float* __restrict__ x, float* __restrict__ out, uint64_t outputs, uint64_t contributors, \
      FoldGeometry g, float scale, float bias, uint32_t empty_bits, const ExprInstr* __restrict__ epi, \
      uint32_t epi_count, uint32_t epi_result) {                                                     \
    fold_body<OP>(x, out, outputs, contributors, g, scale, bias, empty_bits, epi, epi_count, epi_result); \
  }
TILER_FOLD(tiler_fold_sum_f32, kFoldSum)
TILER_FOLD(tiler_fold_squared_f32, kFoldSquared)
TILER_FOLD(tiler_fold_fma_f32, kFoldFma)
TILER_FOLD(tiler_fold_maximum_f32, kFoldMaximum)

// ---------------------------------------------------------------------------
// Adjacent reduced axes: out[o * inner + i] folds x[(o * reduced + r) * inner
// + i] over ascending r.
namespace {

template <uint32_t OP>
__device__ __forceinline__ float fold_term(float v, float scale, float bias) {
  if (OP == kFoldSquared) return tiler::canon(v * v);
  if (OP == kFoldFma) return tiler::canon(tiler::canon(v * scale) + bias);
  return v;
}

// A lane per output.  A wave's loads are contiguous runs of the inner axis,
// but a lane that loads, adds and loads again waits a memory latency per
// contributor; batches of 16 loads are issued one batch ahead of the adds, so
// the loads in flight (4 KiB a wave) cover it once the outputs fill the chip:
// 64 x 64 x 4096 (67 MB) takes 11.8 us, 5.7 TB/s, bound by memory.
template <uint32_t OP>
__device__ __forceinline__ void fold_lanes_body(const float* __restrict__ x, float* __restrict__ out,
                                                uint64_t outputs, uint64_t reduced, uint64_t inner, float scale,
                                                float bias) {
  constexpr uint32_t kBatch = 16;
  const uint64_t id = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (id >= outputs) return;
  const uint64_t o = id / inner;
  const float* p = x + (o * reduced * inner + (id - o * inner));
  float acc = OP == kFoldMaximum ? -__builtin_huge_valf() : -0.0f;
  auto take = [&](float v) {
    if (OP == kFoldMaximum) acc = tiler::maximum_f32(acc, v);
    else acc = acc + fold_term<OP>(v, scale, bias);
  };
  const uint64_t batches = reduced / kBatch;
  float cur[kBatch], nxt[kBatch];
  if (batches) {
#pragma unroll
    for (uint32_t j = 0; j < kBatch; ++j) cur[j] = p[j * inner];
    for (uint64_t b = 1; b < batches; ++b) {
      p += kBatch * inner;
#pragma unroll
      for (uint32_t j = 0; j < kBatch; ++j) nxt[j] = p[j * inner];
#pragma unroll
      for (uint32_t j = 0; j < kBatch; ++j) take(cur[j]);
#pragma unroll
      for (uint32_t j = 0; j < kBatch; ++j) cur[j] = nxt[j];
    }
    p += kBatch * inner;
  }
  // the remainder's loads are in flight while the last batch is folded
  const uint32_t rest = (uint32_t)(reduced - batches * kBatch);
#pragma unroll
  for (uint32_t j = 0; j < kBatch; ++j)
    if (j < rest) nxt[j] = p[j * inner];
  if (batches) {
#pragma unroll
    for (uint32_t j = 0; j < kBatch; ++j) take(cur[j]);
  }
#pragma unroll
  for (uint32_t j = 0; j < kBatch; ++j)
    if (j < rest) take(nxt[j]);
  out[id] = tiler::canon(acc);
}

// A workgroup of nine waves per 16 columns of one outer index.  With fewer
// outputs than the chip needs loads in flight, a lane per output is bound by
// its own latency; here eight waves load (a thread takes four consecutive rows
// of column t % 16, four times), two stages ahead in registers, and store the
// contributor values column-major to one of two LDS buffers; the ninth folds.
// The fold is a relay (tiler::relay_fold's idea, four lanes to a column and a
// column to each lane of a 16-lane row): row g of lanes holds rows 32 g ..
// 32 g + 31 of a 128-row pass in registers, the running sum enters in the
// lanes of g = 0 and moves on after each 32 adds, so every dependent add reads
// registers and one wave instruction advances 16 columns.  The lane rows take
// the segments in the order 0, 1, 3, 2, which v_permlane16_swap and
// v_permlane32_swap walk in one instruction a hop.  Rows past the end are
// staged as -0.0, which leaves every sum unchanged.  Columns lie 4 floats
// apart modulo the 64 banks: the 16-byte stores and reads of a 16-lane row
// touch each bank once.  Adjacent 16-column tiles share 128-byte lines: blocks
// r and r + 8 of each 16 (the same XCD, so the same L2) take neighbours.
// Bound by the chain of adds, then memory: 1 x 4096 x 4096 (67 MB) takes
// 17.6 us, 3.8 TB/s, where one lane per output with a load per step took
// 1018 us; 4 byte reads of the stage (one per add and lane) took 46 us.
constexpr uint32_t kColTile = 16, kColStage = 512, kColLoaders = 512, kColPer = kColStage * kColTile / kColLoaders;
constexpr uint32_t kColStride = kColStage + 4;

__device__ __forceinline__ uint64_t column_group(uint64_t groups) {
  const uint64_t b = blockIdx.x, q = b & ~15ull, r = b & 15u;
  return q + 16 <= groups ? q + 2 * (r & 7u) + (r >> 3) : b;
}

// The hops of the relay across the 16-lane rows: 0 -> 1, 1 -> 3, 3 -> 2 and
// back 2 -> 0 (the other rows' values are never read).
template <int kHop>
__device__ __forceinline__ float row_hop(float v) {
  const uint32_t u = __float_as_uint(v);
  if constexpr (kHop == 0) return __uint_as_float(__builtin_amdgcn_permlane16_swap(u, u, false, false)[0]);
  if constexpr (kHop == 1) return __uint_as_float(__builtin_amdgcn_permlane32_swap(u, u, false, false)[0]);
  if constexpr (kHop == 2) return __uint_as_float(__builtin_amdgcn_permlane16_swap(u, u, false, false)[1]);
  return __uint_as_float(__builtin_amdgcn_permlane32_swap(u, u, false, false)[1]);
}

template <uint32_t OP>
__device__ __forceinline__ void fold_cols_body(const float* __restrict__ x, float* __restrict__ out,
                                               uint64_t groups, uint64_t reduced, uint64_t inner, float scale,
                                               float bias) {
  __shared__ __align__(16) float stage[2][kColTile * kColStride];
  const uint32_t t = threadIdx.x, col = t & (kColTile - 1), row0 = t / kColTile * 4;
  const uint64_t tiles = (inner + kColTile - 1) / kColTile;
  const uint64_t group = column_group(groups), o = group / tiles, c0 = (group - o * tiles) * kColTile;
  // A load is a uniform row base plus this thread's 32-bit byte offset (the
  // planner keeps a stage's rows below 2^32 bytes).  Columns past the last
  // read column 0 and rows past the last read the last: neither is folded.
  const uint32_t pitch = (uint32_t)inner * 4u, coff = c0 + col < inner ? col * 4u : 0u, voff = row0 * pitch + coff;
  const float* base = x + o * reduced * inner + c0;
  const uint64_t stages = (reduced + kColStage - 1) / kColStage;
  // element 4 i + j of a thread's share of a stage: row row0 + 128 i + j
  auto at = [](const float* p, uint32_t bytes) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes);
  };
  auto load = [&](float (&r)[kColPer], uint64_t s) {
    if (s >= stages) return;
    const float* p = base + s * kColStage * inner;
    const uint64_t left = reduced - s * kColStage;  // rows from the stage's first on
    if (left >= kColStage) {
#pragma unroll
      for (uint32_t e = 0; e < kColPer; ++e) r[e] = at(p + (uint64_t)(128 * (e / 4) + e % 4) * inner, voff);
    } else {
      const uint32_t last = (uint32_t)left - 1u;
#pragma unroll
      for (uint32_t e = 0; e < kColPer; ++e) {
        const uint32_t row = row0 + 128 * (e / 4) + e % 4;
        r[e] = at(p, (row < last ? row : last) * pitch + coff);
      }
    }
  };
  auto store = [&](const float (&r)[kColPer], uint64_t s) {
    const uint64_t left = reduced - s * kColStage;
    f32x4* d = reinterpret_cast<f32x4*>(stage[s & 1] + col * kColStride + row0);
#pragma unroll
    for (uint32_t i = 0; i < kColPer / 4; ++i) {
      f32x4 v;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j)
        v[j] = row0 + 128 * i + j < left ? fold_term<OP>(r[4 * i + j], scale, bias) : -0.0f;
      d[32 * i] = v;
    }
  };
  float acc = -0.0f;
  const uint32_t fc = t & 15u, fg = ((t >> 4) & 3u) ^ ((t >> 5) & 1u);  // lane rows 0, 1, 3, 2
  auto fold = [&](uint64_t s) {
    const uint64_t left = reduced - s * kColStage;
    const uint32_t passes = left >= kColStage ? kColStage / 128 : (uint32_t)((left + 127) / 128);
    const f32x4* src = reinterpret_cast<const f32x4*>(stage[s & 1] + fc * kColStride + 32 * fg);
    f32x4 a[8], b[8];  // this pass's segment and the next one's, by turns
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) a[k] = src[k];
    auto pass = [&](auto ps) -> bool {
      constexpr uint32_t p = decltype(ps)::value;
      if (p >= passes) return false;
      f32x4(&cur)[8] = (p & 1) ? b : a;
      f32x4(&nxt)[8] = (p & 1) ? a : b;
      const f32x4* next = src + (p + 1 < passes ? p + 1 : p) * 32;
#pragma unroll
      for (uint32_t k = 0; k < 8; ++k) nxt[k] = next[k];
      auto add = [&] {
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
          acc = acc + cur[k].x;
          acc = acc + cur[k].y;
          acc = acc + cur[k].z;
          acc = acc + cur[k].w;
        }
      };
      add();
      acc = row_hop<0>(acc);
      add();
      acc = row_hop<1>(acc);
      add();
      acc = row_hop<2>(acc);
      add();
      acc = row_hop<3>(acc);
      __builtin_amdgcn_sched_barrier(0);  // keep one pass's reads ahead, not every pass's
      return true;
    };
    tiler::unrolled_while<0, kColStage / 128>(pass);
  };
  // One barrier per stage on both sides: the folding wave is through stage
  // s - 2 when it reaches barrier s - 1, so the loaders' store of stage s
  // after that barrier finds the buffer free.  The loaders' barrier waits for
  // LDS only (a full fence would drain the loads ahead).
  if (t < kColLoaders) {
    float ra[kColPer], rb[kColPer];
    load(ra, 0);
    load(rb, 1);
    for (uint64_t s = 0; s < stages; s += 2) {
      store(ra, s);
      load(ra, s + 2);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + 1 == stages) break;
      store(rb, s + 1);
      load(rb, s + 3);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    return;
  }
  for (uint64_t s = 0; s < stages; ++s) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fold(s);
  }
  if (t - kColLoaders < 16u && c0 + fc < inner) out[o * inner + c0 + fc] = tiler::canon(acc);
}

// The maximum takes its contributors in any order (it is associative and
// commutative, bit for bit), so every thread folds the rows it loads and one
// LDS pass combines the 32 threads of each column.
__device__ __forceinline__ void fold_cols_maximum_body(const float* __restrict__ x, float* __restrict__ out,
                                                       uint64_t groups, uint64_t reduced, uint64_t inner) {
  __shared__ float part[32][kColTile + 1];
  const uint32_t t = threadIdx.x, col = t & (kColTile - 1), row0 = t / kColTile;
  const uint64_t tiles = (inner + kColTile - 1) / kColTile;
  const uint64_t group = column_group(groups), o = group / tiles, c0 = (group - o * tiles) * kColTile;
  const bool live = c0 + col < inner;
  const float* p = x + o * reduced * inner + c0 + col;
  float acc = -__builtin_huge_valf();
  for (uint64_t r0 = row0; r0 < reduced; r0 += kColStage) {
    float v[kColPer];
#pragma unroll
    for (uint32_t i = 0; i < kColPer; ++i) {
      v[i] = -__builtin_huge_valf();
      if (live && r0 + 32 * i < reduced) v[i] = p[(r0 + 32 * i) * inner];
    }
#pragma unroll
    for (uint32_t i = 0; i < kColPer; ++i) acc = tiler::maximum_f32(acc, v[i]);
  }
  part[row0][col] = acc;
  __syncthreads();
  if (t < kColTile && live) {
    float m = part[0][t];
#pragma unroll
    for (uint32_t r = 1; r < 32; ++r) m = tiler::maximum_f32(m, part[r][t]);
    out[o * inner + c0 + t] = m;
  }
}

}  // namespace

#define TILER_FOLD_ADJACENT(NAME, OP)                                                                  \
  extern "C" __global__ void __launch_bounds__(256) NAME##_lanes(                                      \
      const float* __restrict__ x, float* __restrict__ out, uint64_t outputs, uint64_t reduced,        \
      uint64_t inner, float scale, float bias) {                                                       \
    fold_lanes_body<OP>(x, out, outputs, reduced, inner, scale, bias);                                 \
  }                                                                                                    \
  extern "C" __global__ void __launch_bounds__(OP == kFoldMaximum ? 512 : 576) NAME##_cols(            \
      const float* __restrict__ x, float* __restrict__ out, uint64_t groups, uint64_t reduced,         \
      uint64_t inner, float scale, float bias) {                                                       \
    if constexpr (OP == kFoldMaximum) fold_cols_maximum_body(x, out, groups, reduced, inner);          \
    else fold_cols_body<OP>(x, out, groups, reduced, inner, scale, bias);                              \
  }
TILER_FOLD_ADJACENT(tiler_fold_sum_f32, kFoldSum)
TILER_FOLD_ADJACENT(tiler_fold_squared_f32, kFoldSquared)
TILER_FOLD_ADJACENT(tiler_fold_fma_f32, kFoldFma)
TILER_FOLD_ADJACENT(tiler_fold_maximum_f32, kFoldMaximum)

// The maximum of contiguous rows: `lanes` (16, 64 or all 256) threads of the
// workgroup to a row, eight loads in flight per thread.  Short rows are bound
// by the combining steps, not by their loads: with 16 lanes a wave combines
// four rows in four steps where 64 lanes take six for one.
extern "C" __global__ void __launch_bounds__(256)
tiler_fold_maximum_f32_rows(const float* __restrict__ x, float* __restrict__ out, uint64_t rows, uint64_t reduced,
                            uint32_t lanes) {
  __shared__ float part[4];
  const uint32_t lane = threadIdx.x & (lanes - 1u);
  const uint64_t row = (uint64_t)blockIdx.x * (256u / lanes) + threadIdx.x / lanes;
  float acc = -__builtin_huge_valf();
  if (row < rows) {
    const float* p = x + row * reduced;
    for (uint64_t e = lane; e < reduced; e += 8ull * lanes) {
      float v[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {
        v[i] = -__builtin_huge_valf();
        if (e + (uint64_t)i * lanes < reduced) v[i] = p[e + (uint64_t)i * lanes];
      }
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) acc = tiler::maximum_f32(acc, v[i]);
    }
  }
  for (uint32_t o = lanes < 64u ? lanes / 2 : 32u; o >= 1; o >>= 1)
    acc = tiler::maximum_f32(acc, __shfl_xor(acc, (int)o, 64));
  if (lanes <= 64) {
    if (lane == 0 && row < rows) out[row] = acc;
    return;
  }
  if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0)
    out[row] = tiler::maximum_f32(tiler::maximum_f32(part[0], part[1]), tiler::maximum_f32(part[2], part[3]));
}
