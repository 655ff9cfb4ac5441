// Device helpers of RoPE and the KV write, shared by the kernels that end with them (not part
// of the C ABI): the decoder's head layout, the rotation, and where rotated columns go.
#ifndef PAGEDCORE_ROPE_DEVICE_H
#define PAGEDCORE_ROPE_DEVICE_H

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace rope_device {

constexpr int kLayers = 22;
constexpr int kSlots = 16;
constexpr int kKVHeads = 4;
constexpr int kQHeads = 32;
constexpr int kHeadDim = 64;
constexpr int kHalfDim = kHeadDim / 2;               // 32 rotation frequencies
constexpr int64_t kRowElems = kKVHeads * kHeadDim;   // 256 fp16 per pool token row
constexpr int kQElems = kQHeads * kHeadDim;          // 2048
constexpr int kQkvElems = kQElems + 2 * kRowElems;   // 2560: q | k | v of one token

// The reference rotation (dense.py:56-59) is x * cos + cat(-x2, x1) * sin with cos/sin the
// fp16 tables of the position; for d < 32 that is x[d] * c[d] + (-x[d + 32]) * s[d], for
// d >= 32 x[d] * c[d - 32] + x[d - 32] * s[d - 32], each product and the sum rounded to fp16.
// lo, hi: N columns d and their partners d + 32.
template <int N, typename V>
__device__ __forceinline__ void rotate_pair(V& lo, V& hi, const V c, const V s) {
#pragma clang fp contract(off)
  const auto round = [](float x) { return static_cast<_Float16>(x); };
  V out_lo, out_hi;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float x1 = static_cast<float>(lo[i]);
    const float x2 = static_cast<float>(hi[i]);
    const float cf = static_cast<float>(c[i]);
    const float sf = static_cast<float>(s[i]);
    const float a1 = static_cast<float>(round(x1 * cf));
    // fp16(-a * b) == -fp16(a * b): round-to-nearest-even is symmetric.
    const float b1 = static_cast<float>(-round(x2 * sf));
    const float a2 = static_cast<float>(round(x2 * cf));
    const float b2 = static_cast<float>(round(x1 * sf));
    out_lo[i] = round(a1 + b1);
    out_hi[i] = round(a2 + b2);
  }
  lo = out_lo;
  hi = out_hi;
}

// Where a projection with the RoPE epilogue writes (the outputs of pc_rope_kv_append).
struct RopeOut {
  const _Float16* table;  // [positions][2][32]: cos, then sin
  int64_t table_positions;
  _Float16* query;
  _Float16* layer_pool;  // null: no pool
  int64_t kind_elems;    // elements of the layer's K (V follows)
  _Float16* key;         // null: not kept
  _Float16* value;
};

// The weight rows of a q|k|v projection in pairs: pair p is row 64 (p / 32) + p % 32 (column d < 32
// of a head) and the row 32 below it. 32 q heads, 4 k heads and 4 v heads, 1280 pairs.
constexpr int kPairs = kQkvElems / 2;
__device__ __forceinline__ int pair_row(int p) { return kHeadDim * (p / kHalfDim) + p % kHalfDim; }

// One token's position and pool slot, and the table row of the position.
struct RopeRow {
  int64_t slot;  // -1: not written to the pool
  bool valid;    // the position lies in the table
  const _Float16* table;
};

__device__ __forceinline__ RopeRow rope_row(const RopeOut& out, int64_t position, int64_t slot, bool has_slot) {
  RopeRow r;
  r.valid = position >= 0 && position < out.table_positions;
  r.table = out.table + (r.valid ? position : 0) * kHeadDim;
  r.slot = has_slot && r.valid && slot >= 0 && slot < out.kind_elems / kRowElems ? slot : -1;
  return r;
}

// Rotates and stores pairs p .. p + 3 (of one head) of token t: lo, hi the fp16 projections, c, s
// the table values of p % 32 ... A bad position is never reached through the host API
// (positions are checked there); it yields NaN rows instead of a read outside the table.
template <typename V>
__device__ __forceinline__ void store_pairs(const RopeOut& out, const RopeRow& r, int64_t t, int p, V lo, V hi, const V c,
                                            const V s) {
  const int head = p / kHalfDim, d = p % kHalfDim;
  const bool is_v = head >= kQHeads + kKVHeads;
  if (!is_v) {
    rotate_pair<4>(lo, hi, c, s);
  }
  const V nan = static_cast<V>(__builtin_nanf16(""));
  if (!r.valid && !is_v) lo = hi = nan;
  if (head < kQHeads) {
    _Float16* dst = out.query + t * kQElems + head * kHeadDim + d;
    *reinterpret_cast<V*>(dst) = lo;
    *reinterpret_cast<V*>(dst + kHalfDim) = hi;
    return;
  }
  const int offset = (head - (is_v ? kQHeads + kKVHeads : kQHeads)) * kHeadDim + d;
  _Float16* kept = is_v ? out.value : out.key;
  if (kept != nullptr) {
    *reinterpret_cast<V*>(kept + t * kRowElems + offset) = lo;
    *reinterpret_cast<V*>(kept + t * kRowElems + offset + kHalfDim) = hi;
  }
  if (r.slot >= 0) {
    _Float16* dst = out.layer_pool + (is_v ? out.kind_elems : 0) + r.slot * kRowElems + offset;
    *reinterpret_cast<V*>(dst) = lo;
    *reinterpret_cast<V*>(dst + kHalfDim) = hi;
  }
}

}  // namespace rope_device

#endif  // PAGEDCORE_ROPE_DEVICE_H
