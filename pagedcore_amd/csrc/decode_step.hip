// Elementwise kernels of the batched decode step around paged attention: RoPE fused with the
// KV append, residual add fused with RMSNorm, and SiLU fused with the up-projection product.
// The first two also take their projection input as fp32 split-K partial sums (the output of
// pc_gemm_m128's partials epilogue), added in split order and rounded to fp16 once: the
// value the reference's fp16 GEMM output holds, up to the order of fp32 accumulation.
//
// Each one reproduces the fp16 rounding points of the reference's torch expressions
// (src/pagedcore/dense.py:17-21, 33-61, 102-104): every torch op on fp16 tensors computes
// in fp32 and rounds its result to fp16 once, so a kernel rounds exactly where the
// reference expression materialises an fp16 tensor and nowhere else. Contraction of a
// multiply into a following add is switched off wherever that would skip a rounding.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "pagedcore_hip.h"
#include "pc_internal.h"
#include "rope_device.h"

namespace {

using namespace rope_device;
using pc_internal::aligned;
using pc_internal::check_launch;
using pc_internal::ok;
using pc_internal::set_error;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

constexpr int kRopeTasks = 160;                        // 128 of q, 16 of k, 16 of v
constexpr int kRopeThreads = 192;
constexpr int kNormThreads = 256;
constexpr int kNormMaxChunks = 4;                      // rows of up to 4 * 256 * 8 = 8192
constexpr int kSiluThreads = 256;

__device__ __forceinline__ _Float16 round_h(float x) { return static_cast<_Float16>(x); }

typedef float float4_t __attribute__((ext_vector_type(4)));

// What bounds the two kernels below at decode sizes is the number of dependent memory round
// trips (each about 0.6-1 us: their inputs were just written on other XCDs), so every load that
// does not depend on another is issued before the first wait. The split count is a template
// argument for the counts a decode step uses: 2 splits then load 2 parts (a form unrolled to 8
// that reloaded split 0 for the missing ones took the L1 four times as long).

constexpr int kFp16Input = 0;     // the projection is an fp16 row
constexpr int kAnySplits = -1;    // a split count without its own instance

// 8 consecutive columns of a projection: the fp16 values, or the parts that make them.
template <int SPLITS>
struct Chunk8 {
  float4_t lo[SPLITS > 0 ? SPLITS : 1], hi[SPLITS > 0 ? SPLITS : 1];
  half8_t value;
};

// Issues the chunk's loads: SPLITS fp32 parts at `offset` + s * stride of `input`, or its fp16 chunk.
template <int SPLITS>
__device__ __forceinline__ Chunk8<SPLITS> load8(const void* input, int64_t offset, int64_t stride) {
  Chunk8<SPLITS> c;
  if constexpr (SPLITS == kFp16Input) {
    c.value = *reinterpret_cast<const half8_t*>(static_cast<const _Float16*>(input) + offset);
  } else {
    const float* parts = static_cast<const float*>(input);
#pragma unroll
    for (int s = 0; s < (SPLITS > 0 ? SPLITS : 1); ++s) {
      c.lo[s] = *reinterpret_cast<const float4_t*>(parts + s * stride + offset);
      c.hi[s] = *reinterpret_cast<const float4_t*>(parts + s * stride + offset + 4);
    }
  }
  return c;
}

// fp16(sum of the parts), added in split order.
template <int SPLITS>
__device__ __forceinline__ half8_t value8(const Chunk8<SPLITS>& c, const void* input, int64_t offset, int64_t stride,
                                          int splits) {
  if constexpr (SPLITS == kFp16Input) {
    return c.value;
  } else {
    float4_t lo = c.lo[0], hi = c.hi[0];
    if constexpr (SPLITS == kAnySplits) {
      const float* parts = static_cast<const float*>(input);
#pragma unroll 4
      for (int s = 1; s < splits; ++s) {
        lo += *reinterpret_cast<const float4_t*>(parts + s * stride + offset);
        hi += *reinterpret_cast<const float4_t*>(parts + s * stride + offset + 4);
      }
    } else {
#pragma unroll
      for (int s = 1; s < SPLITS; ++s) {
        lo += c.lo[s];
        hi += c.hi[s];
      }
    }
    half8_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[i] = round_h(lo[i]);
      out[i + 4] = round_h(hi[i]);
    }
    return out;
  }
}

// Calls f(integral_constant) with the instance for a split count (kFp16Input: no parts).
template <typename F>
void with_splits(bool fp16, int32_t splits, F&& f) {
  if (fp16) f(std::integral_constant<int, kFp16Input>{});
  else if (splits == 1) f(std::integral_constant<int, 1>{});
  else if (splits == 2) f(std::integral_constant<int, 2>{});
  else if (splits == 4) f(std::integral_constant<int, 4>{});
  else if (splits == 8) f(std::integral_constant<int, 8>{});
  else f(std::integral_constant<int, kAnySplits>{});
}

// ---------------------------------------------------------------------------------------
// RoPE + KV append.
//
// One workgroup per token row t. Every thread owns a task of two 16 B chunks 32 dims apart:
//   threads   0..127  q head tid / 4, dims [8c, 8c + 8) with their partners
//   threads 128..143  k head (tid - 128) / 4, the same dims
//   threads 144..159  v head (tid - 144) / 4, the same dims, not rotated
// (threads 160..191 repeat the last task and store nothing). Two memory round trips: position,
// slot and the projections together, then the table row of the position; six, one after the
// other, took 5.2 us a launch at 37 rows and 4.8 at one (22 layers of rope and q|k|v at 37 rows
// 419 -> 338 us).
// ---------------------------------------------------------------------------------------

// qkv: fp16 rows of stride qkv_stride (SPLITS kFp16Input), or fp32 parts [splits][T][2560] of
// split stride qkv_stride. Scalar parameters, those the first loads need leading (the compiler
// preloads the leading 64 bytes into SGPRs at wave launch: no kernel-argument round trip
// before them).
template <int SPLITS>
__global__ __launch_bounds__(kRopeThreads) void rope_kv_append_kernel(
    const int64_t* positions, const int64_t* slot_mapping, const void* qkv, int64_t qkv_stride, const _Float16* rope,
    _Float16* query_out, int32_t splits, int32_t rope_positions, _Float16* layer_pool, int64_t kind_elems,
    _Float16* key_out, _Float16* value_out) {
  const int64_t t = blockIdx.x;
  const int tid = threadIdx.x;
  const int task = min(tid, kRopeTasks - 1);
  const bool is_q = task < 128, is_v = task >= 144;
  const int index = is_q ? task : is_v ? task - 144 : task - 128;  // within its part
  const int offset = (index >> 2) * kHeadDim + 8 * (index & 3);    // head and dims in its part
  const int col = offset + (is_q ? 0 : is_v ? kQElems + static_cast<int>(kRowElems) : kQElems);
  const int64_t at = SPLITS == kFp16Input ? t * qkv_stride + col : t * kQkvElems + col;
  const Chunk8<SPLITS> first = load8<SPLITS>(qkv, at, qkv_stride);
  const Chunk8<SPLITS> second = load8<SPLITS>(qkv, at + kHalfDim, qkv_stride);
  const int64_t position = positions[t];
  int64_t slot = (slot_mapping != nullptr ? slot_mapping : positions)[t];
  // Position, slot and the remaining arguments are scalar loads: all at once here, instead of
  // each where it is used.
  asm volatile("" ::"s"(position), "s"(slot), "s"(layer_pool), "s"(kind_elems), "s"(key_out), "s"(value_out));
  if (slot_mapping == nullptr || slot >= kind_elems / kRowElems) slot = -1;  // outside the pool: never written
  const bool valid_position = position >= 0 && position < rope_positions;
  const _Float16* table = rope + (valid_position ? position : 0) * kHeadDim + 8 * (index & 3);
  const half8_t cs = *reinterpret_cast<const half8_t*>(table);
  const half8_t sn = *reinterpret_cast<const half8_t*>(table + kHalfDim);

  half8_t lo = value8<SPLITS>(first, qkv, at, qkv_stride, splits);
  half8_t hi = value8<SPLITS>(second, qkv, at + kHalfDim, qkv_stride, splits);
  half8_t rotated_lo = lo, rotated_hi = hi;
  rotate_pair<8>(rotated_lo, rotated_hi, cs, sn);  // in every lane, so that the table is not read under a branch
  // A bad position is never reached through the host API (positions are checked there); it
  // yields NaN rows instead of a read outside the table.
  const half8_t nan = static_cast<half8_t>(__builtin_nanf16(""));
  lo = is_v ? lo : valid_position ? rotated_lo : nan;
  hi = is_v ? hi : valid_position ? rotated_hi : nan;
  if (tid >= kRopeTasks) return;
  if (is_q) {
    _Float16* dst = query_out + t * kQElems + offset;
    *reinterpret_cast<half8_t*>(dst) = lo;
    *reinterpret_cast<half8_t*>(dst + kHalfDim) = hi;
    return;
  }
  _Float16* out = is_v ? value_out : key_out;
  if (out != nullptr) {
    *reinterpret_cast<half8_t*>(out + t * kRowElems + offset) = lo;
    *reinterpret_cast<half8_t*>(out + t * kRowElems + offset + kHalfDim) = hi;
  }
  if (slot >= 0 && valid_position) {
    _Float16* dst = layer_pool + (is_v ? kind_elems : 0) + slot * kRowElems + offset;
    *reinterpret_cast<half8_t*>(dst) = lo;
    *reinterpret_cast<half8_t*>(dst + kHalfDim) = hi;
  }
}

// ---------------------------------------------------------------------------------------
// Residual add + RMSNorm (dense.py:17-21 after the residual sum of decoder.py:191-192).
//
// One workgroup per row; thread i owns 16 B chunks i, i + 256, ... of the row.
//   h   = fp16(hidden + delta)                     (only when delta is given; stored back)
//   r   = 1 / sqrt(sum(h * h) / width + eps)       (fp32)
//   out = fp16(weight * fp16(h * r))
// Weight, residual and every part are loaded before the first sum: one memory round trip (22 layers of
// a 7-row MLP 435 -> 414 us, of a 128-row one 731 -> 708), or one per chunk where the parts of all
// chunks would take too many registers. Only the last chunk can end inside the row, and threads past
// it load nothing: with every thread loading four chunks, the row's last one over again, and one
// part of each at a time, wide rows were slower than with a branch per chunk (us, 8 splits: 37 rows of 2056
// 5.6, now 3.3, 4.5 with a branch; of 4096 5.6, now 3.4, 4.7; 2048 rows of 2056 35, now 26, 26).
// ---------------------------------------------------------------------------------------

template <int CTRL>
__device__ __forceinline__ float add_dpp(float x) {
  const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false);
  return x + __int_as_float(moved);
}

// Sum over the wave in every lane: halves, 16-lane groups, then rotations by 8, 4, 2 and 1 within
// each group (the additions of an xor butterfly, without its LDS round trips).
__device__ __forceinline__ float wave_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(q[0]) + __uint_as_float(q[1]);
  x = add_dpp<0x128>(x);  // row_ror 8, 4, 2, 1
  x = add_dpp<0x124>(x);
  x = add_dpp<0x122>(x);
  return add_dpp<0x121>(x);
}

// delta, when given (HAS_DELTA), is fp16 [rows][width] (SPLITS kFp16Input) or fp32 partial sums
// [splits][rows][width], rounded to fp16 before the add. CHUNKS chunks per thread, all but the last
// within the row for every thread. CLAMP: a thread past the row loads its last chunk again instead of
// branching round the loads (for rows that fill the workgroup, where it never does: a one-row
// decode step of 44 norms 784 us, 789 with the branch). All the parameters fit the 64 bytes that are
// preloaded into SGPRs.
template <int CHUNKS, bool CLAMP, bool HAS_DELTA, int SPLITS>
__global__ __launch_bounds__(kNormThreads) void add_rms_norm_kernel(_Float16* hidden, const void* delta,
                                                                    int64_t parts_stride, const _Float16* weight,
                                                                    _Float16* out, int32_t splits, int32_t width,
                                                                    float eps) {
#pragma clang fp contract(off)
  // Every chunk's loads at once, or one chunk's at a time where they would take too many registers.
  constexpr bool kTogether = !HAS_DELTA || CHUNKS * (SPLITS > 0 ? SPLITS : 1) <= 8;
  __shared__ float wave_sums[kNormThreads / 64];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * width;
  const int tid = threadIdx.x;
  half8_t wt[CHUNKS], h[CHUNKS];
  Chunk8<SPLITS> d[CHUNKS];
  const int chunks = width / 8;
  auto mine = [&](int k) { return k + 1 < CHUNKS || tid + k * kNormThreads < chunks; };
  auto column = [&](int k) {
    const int chunk = tid + k * kNormThreads;
    return 8 * (CLAMP && chunk >= chunks ? chunks - 1 : chunk);
  };
  auto at = [&](int k) { return base + column(k); };
  float squares = 0.0f;
  auto load = [&](int k) {
    if constexpr (HAS_DELTA) d[k] = load8<SPLITS>(delta, at(k), parts_stride);
    h[k] = *reinterpret_cast<const half8_t*>(hidden + at(k));
    wt[k] = *reinterpret_cast<const half8_t*>(weight + column(k));
  };
  auto add = [&](int k) {
    if constexpr (HAS_DELTA) {
      const half8_t v = value8<SPLITS>(d[k], delta, at(k), parts_stride, splits);
#pragma unroll
      for (int i = 0; i < 8; ++i) h[k][i] = round_h(static_cast<float>(h[k][i]) + static_cast<float>(v[i]));
    }
    if (!CLAMP || mine(k)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = static_cast<float>(h[k][i]);
        squares += x * x;
      }
    }
  };
#pragma unroll
  for (int k = 0; k < CHUNKS; ++k) {
    if (CLAMP || mine(k)) load(k);
    if constexpr (!kTogether) {
      if (CLAMP || mine(k)) add(k);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (kTogether) {
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k) {
      if (CLAMP || mine(k)) add(k);
    }
  }
  squares = wave_sum(squares);
  if ((tid & 63) == 0) wave_sums[tid >> 6] = squares;
  // The barrier also orders every thread's residual loads before the first store (CLAMP: a chunk may be
  // loaded by more threads than the one that stores it).
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int w = 0; w < kNormThreads / 64; ++w) total += wave_sums[w];
  const float scale = 1.0f / sqrtf(total / static_cast<float>(width) + eps);
#pragma unroll
  for (int k = 0; k < CHUNKS; ++k) {
    if (mine(k)) {
      half8_t o;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float normalized = static_cast<float>(round_h(static_cast<float>(h[k][i]) * scale));
        o[i] = round_h(static_cast<float>(wt[k][i]) * normalized);
      }
      if constexpr (HAS_DELTA) *reinterpret_cast<half8_t*>(hidden + at(k)) = h[k];
      *reinterpret_cast<half8_t*>(out + at(k)) = o;
    }
  }
}

// ---------------------------------------------------------------------------------------
// SwiGLU activation (dense.py:102-104): out = fp16(fp16(silu(gate)) * up), where
// gate_up row r is [gate (width) | up (width)], silu(x) = x / (1 + exp(-x)) in fp32.
// ---------------------------------------------------------------------------------------

__global__ __launch_bounds__(kSiluThreads) void silu_mul_kernel(_Float16* __restrict__ out,
                                                                const _Float16* __restrict__ gate_up,
                                                                int64_t rows, int32_t width) {
#pragma clang fp contract(off)
  const int64_t chunks_per_row = width / 8;
  const int64_t chunk = static_cast<int64_t>(blockIdx.x) * kSiluThreads + threadIdx.x;
  if (chunk >= rows * chunks_per_row) return;
  const int64_t r = chunk / chunks_per_row;
  const int64_t c = chunk % chunks_per_row;
  const _Float16* src = gate_up + r * 2 * width + 8 * c;
  const half8_t g = *reinterpret_cast<const half8_t*>(src);
  const half8_t u = *reinterpret_cast<const half8_t*>(src + width);
  half8_t o;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = static_cast<float>(g[i]);
    const float activated = static_cast<float>(round_h(x / (1.0f + expf(-x))));
    o[i] = round_h(activated * static_cast<float>(u[i]));
  }
  *reinterpret_cast<half8_t*>(out + r * width + 8 * c) = o;
}

// Shared by both RoPE entry points: exactly one of qkv / qkv_parts is given (checked by the
// callers), with qkv_stride its row stride or split stride.
int rope_kv_append(void* query_out, void* key_out, void* value_out, const void* qkv, const float* qkv_parts,
                   int32_t splits, int64_t qkv_stride, const int64_t* positions, const void* rope_table,
                   int32_t rope_positions, void* pool, int64_t num_blocks, int32_t layer,
                   const int64_t* slot_mapping, int64_t num_tokens, void* stream) {
  if (!query_out || !positions || !rope_table) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (rope_positions < 1) return set_error(PC_ERR_ARGUMENT, "rope_positions must be positive");
  if ((pool == nullptr) != (slot_mapping == nullptr))
    return set_error(PC_ERR_ARGUMENT, "pool and slot_mapping must both be given or both be null");
  if (pool != nullptr) {
    if (num_blocks < 1 || num_blocks > INT32_MAX)
      return set_error(PC_ERR_ARGUMENT, "num_blocks %lld out of range", static_cast<long long>(num_blocks));
    if (layer < 0 || layer >= kLayers) return set_error(PC_ERR_ARGUMENT, "layer %d outside [0, 22)", layer);
  }
  if (!aligned(query_out, 16) || !aligned(qkv, 16) || !aligned(qkv_parts, 16) || !aligned(rope_table, 16) ||
      !aligned(pool, 16) || !aligned(key_out, 16) || !aligned(value_out, 16))
    return set_error(PC_ERR_ARGUMENT, "buffers must be 16-byte aligned");
  const int64_t kind_elems = pool ? num_blocks * kSlots * kRowElems : 0;
  _Float16* layer_pool = pool ? static_cast<_Float16*>(pool) + static_cast<int64_t>(layer) * 2 * kind_elems : nullptr;
  with_splits(qkv_parts == nullptr, splits, [&](auto instance) {
    hipLaunchKernelGGL(rope_kv_append_kernel<decltype(instance)::value>, dim3(static_cast<uint32_t>(num_tokens)),
                       dim3(kRopeThreads), 0, static_cast<hipStream_t>(stream), positions, slot_mapping,
                       qkv_parts ? static_cast<const void*>(qkv_parts) : qkv, qkv_stride,
                       static_cast<const _Float16*>(rope_table), static_cast<_Float16*>(query_out), splits, rope_positions,
                       layer_pool, kind_elems, static_cast<_Float16*>(key_out), static_cast<_Float16*>(value_out));
  });
  return check_launch("rope_kv_append");
}

int add_rms_norm(void* out, void* hidden, const void* delta, const float* delta_parts, int32_t splits,
                 const void* weight, int64_t rows, int32_t width, float eps, void* stream) {
  if (rows < 0 || rows > INT32_MAX) return set_error(PC_ERR_ARGUMENT, "rows %lld out of range", static_cast<long long>(rows));
  if (width < 8 || width % 8 != 0 || width > kNormThreads * kNormMaxChunks * 8)
    return set_error(PC_ERR_ARGUMENT, "width %d must be a multiple of 8 in [8, %d]", width,
                     kNormThreads * kNormMaxChunks * 8);
  if (rows == 0) return ok();  // nothing to read or write (empty buffers may be null)
  if (!out || !hidden || !weight) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (!(eps >= 0.0f)) return set_error(PC_ERR_ARGUMENT, "eps must be non-negative");
  if (!aligned(out, 16) || !aligned(hidden, 16) || !aligned(delta, 16) || !aligned(delta_parts, 16) ||
      !aligned(weight, 16))
    return set_error(PC_ERR_ARGUMENT, "buffers must be 16-byte aligned");
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(rows)), dim3(kNormThreads), 0, static_cast<hipStream_t>(stream),
                       static_cast<_Float16*>(hidden), delta_parts ? static_cast<const void*>(delta_parts) : delta,
                       rows * width, static_cast<const _Float16*>(weight), static_cast<_Float16*>(out), splits, width, eps);
  };
  auto launch_row = [&](auto has_delta, auto instance) {
    constexpr bool D = decltype(has_delta)::value;
    constexpr int S = decltype(instance)::value;
    static_assert(kNormMaxChunks == 4, "one instance per chunk count");
    switch ((width / 8 - 1) / kNormThreads) {
      case 0:
        return width == 8 * kNormThreads ? launch(add_rms_norm_kernel<1, true, D, S>) : launch(add_rms_norm_kernel<1, false, D, S>);
      case 1: return launch(add_rms_norm_kernel<2, false, D, S>);
      case 2: return launch(add_rms_norm_kernel<3, false, D, S>);
      default: return launch(add_rms_norm_kernel<4, false, D, S>);
    }
  };
  if (delta == nullptr && delta_parts == nullptr) {
    launch_row(std::false_type{}, std::integral_constant<int, kFp16Input>{});
  } else {
    with_splits(delta_parts == nullptr, splits, [&](auto instance) { launch_row(std::true_type{}, instance); });
  }
  return check_launch("add_rms_norm");
}

}  // namespace

extern "C" {

int pc_rope_kv_append(void* query_out, void* key_out, void* value_out, const void* qkv, int64_t qkv_stride,
                      const int64_t* positions, const void* rope_table, int32_t rope_positions, void* pool,
                      int64_t num_blocks, int32_t layer, const int64_t* slot_mapping, int64_t num_tokens,
                      void* stream) {
  if (num_tokens < 0) return set_error(PC_ERR_ARGUMENT, "negative token count");
  if (num_tokens > INT32_MAX) return set_error(PC_ERR_ARGUMENT, "too many tokens");
  if (num_tokens == 0) return ok();  // nothing to read or write (empty buffers may be null)
  if (!qkv) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (qkv_stride < kQkvElems || qkv_stride % 8 != 0)
    return set_error(PC_ERR_ARGUMENT, "qkv_stride %lld must be >= %d and a multiple of 8",
                     static_cast<long long>(qkv_stride), kQkvElems);
  return rope_kv_append(query_out, key_out, value_out, qkv, nullptr, 1, qkv_stride, positions, rope_table,
                        rope_positions, pool, num_blocks, layer, slot_mapping, num_tokens, stream);
}

int pc_rope_kv_append_parts(void* query_out, void* key_out, void* value_out, const float* qkv_parts, int32_t splits,
                            const int64_t* positions, const void* rope_table, int32_t rope_positions, void* pool,
                            int64_t num_blocks, int32_t layer, const int64_t* slot_mapping, int64_t num_tokens,
                            void* stream) {
  if (num_tokens < 0) return set_error(PC_ERR_ARGUMENT, "negative token count");
  if (num_tokens > INT32_MAX / kQkvElems) return set_error(PC_ERR_ARGUMENT, "too many tokens");
  if (num_tokens == 0) return ok();
  if (!qkv_parts) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (splits < 1 || splits > 64) return set_error(PC_ERR_ARGUMENT, "splits %d outside [1, 64]", splits);
  return rope_kv_append(query_out, key_out, value_out, nullptr, qkv_parts, splits, num_tokens * kQkvElems, positions,
                        rope_table, rope_positions, pool, num_blocks, layer, slot_mapping, num_tokens, stream);
}

int pc_add_rms_norm(void* out, void* hidden, const void* delta, const void* weight, int64_t rows, int32_t width,
                    float eps, void* stream) {
  return add_rms_norm(out, hidden, delta, nullptr, 1, weight, rows, width, eps, stream);
}

int pc_add_rms_norm_parts(void* out, void* hidden, const float* delta_parts, int32_t splits, const void* weight,
                          int64_t rows, int32_t width, float eps, void* stream) {
  if (rows > 0 && !delta_parts) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (splits < 1 || splits > 64) return set_error(PC_ERR_ARGUMENT, "splits %d outside [1, 64]", splits);
  if (rows > INT32_MAX / 8192) return set_error(PC_ERR_ARGUMENT, "rows %lld out of range", static_cast<long long>(rows));
  return add_rms_norm(out, hidden, nullptr, delta_parts, splits, weight, rows, width, eps, stream);
}

int pc_silu_mul(void* out, const void* gate_up, int64_t rows, int32_t width, void* stream) {
  if (rows < 0) return set_error(PC_ERR_ARGUMENT, "negative row count");
  if (width < 8 || width % 8 != 0) return set_error(PC_ERR_ARGUMENT, "width %d must be a positive multiple of 8", width);
  if (rows == 0) return ok();  // nothing to read or write (empty buffers may be null)
  if (!out || !gate_up) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (!aligned(out, 16) || !aligned(gate_up, 16)) return set_error(PC_ERR_ARGUMENT, "buffers must be 16-byte aligned");
  const int64_t chunks = rows * (width / 8);
  const int64_t blocks = (chunks + kSiluThreads - 1) / kSiluThreads;
  if (blocks > INT32_MAX) return set_error(PC_ERR_ARGUMENT, "silu_mul too large");
  hipLaunchKernelGGL(silu_mul_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kSiluThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<_Float16*>(out),
                     static_cast<const _Float16*>(gate_up), rows, width);
  return check_launch("silu_mul");
}

}  // extern "C"
