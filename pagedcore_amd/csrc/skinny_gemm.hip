// Projection GEMMs of the batched decode step at up to 128 rows: Y = X W^T with X fp16
// [m <= 128][k] (the step's activations) and W fp16 [n][k] (a weight, row-major as stored),
// fp32 accumulation. The reference computes these with torch.nn.functional.linear on fp16
// tensors (src/pagedcore/dense.py:91-104 via decoder.py:156-199): fp32 accumulation and one
// rounding to fp16 per output element. Here the rounding stays where the reference has it:
// the split-K consumers (pc_rope_kv_append_parts, pc_add_rms_norm_parts) add the fp32
// partial sums in split order and round once.
//
// Design for decode shapes (m = batch, n and k in the thousands): the weight is read once
// from HBM and is the only large stream, so one workgroup computes ALL m rows of an NT-row
// slice of W over a range of K (split-K when n alone gives too few workgroups to fill the
// 256 CUs). X and W chunks stream through a ring of LDS stages filled by LDS DMA
// (global_load_lds_dwordx4, 16 B per lane, rows swizzled so that the MFMA operand reads are
// bank-conflict free); the waves read 16x32 operand fragments from LDS and issue
// v_mfma_f32_16x16x32_f16 with W as the A operand (16 weight rows) and X as the B operand
// (16 activation rows), so each lane ends with 4 consecutive output columns of one row.
//
// pc_qkv_rope_append is here too: the q|k|v projection whose epilogue rotates q and k and writes
// them and v where pc_rope_kv_append does (pairs of a head's columns d and d + 32 in one tile, no
// split-K, so that a workgroup holds final sums). A launch, a round trip of the partials and
// a kernel of a few kilobytes per row less in every layer.
//
// The form above (gemm_m128_kernel) is for many rows: its X ring has 128 rows whatever m is. Up to
// 64 rows, and where it leaves CUs idle, gemm_stream_kernel takes over (see there).
//
// Epilogues: fp32 partials [splits][m][n]; fp16 [m][n] (one split); or SwiGLU (one split):
// a tile's W rows are 32 gate_proj rows and the 32 matching up_proj rows of the stacked
// [gate | up] weight, and the tile writes fp16(fp16(silu(fp16 gate)) * fp16 up) for its 32
// columns (dense.py:102-104 with the roundings of silu_mul_kernel).

#include "gemm_device.h"

namespace {

using namespace gemm_device;
using namespace rope_device;
using pc_internal::aligned;
using pc_internal::check_launch;
using pc_internal::set_error;

constexpr int kMaxRows = 128;
constexpr int kMaxQkvK = 1 << 18;  // 2560 rows of W within 32-bit offsets
constexpr int kMaxStreamK = 1 << 24;  // gemm_stream_kernel: 64 rows within 32-bit offsets
constexpr int kSwiGLUHalf = 32;  // gate (and up) rows per SwiGLU tile

struct GemmArgs {
  const _Float16* x;
  const _Float16* w;
  int m, n, k, ksplit;  // ksplit: K range of one split
  int tiles;            // workgroups per split
  int half_rows;        // SwiGLU: rows of gate_proj (up_proj starts there)
  void* out;
};

template <int NT, int KC, int STAGES, int WAVES>
struct Shape {
  static constexpr int CH = KC / 8;        // 16-byte chunks per LDS row
  static constexpr int XB = kMaxRows * KC * 2;
  static constexpr int WB = NT * KC * 2;
  static constexpr int SB = XB + WB;       // bytes per ring stage
  static constexpr int XI = XB / 1024;     // 1 KiB DMA instructions per stage
  static constexpr int WI = WB / 1024;
  static_assert(XI % WAVES == 0 && WI % WAVES == 0, "each wave issues the same number of DMA instructions");
  static constexpr int PER = (XI + WI) / WAVES;
  static constexpr int MT = kMaxRows / 16 / WAVES;  // 16-row X tiles per wave
  static constexpr int NTL = NT / 16;               // 16-row W tiles
  static constexpr int LDS = STAGES * SB;
  static_assert(LDS <= 160 * 1024, "ring fits the CU's LDS");
};

// Position of 16-byte chunk c of LDS row r (an involution): the 16 rows one operand read
// touches at one chunk land on distinct banks.
template <int CH>
__device__ __forceinline__ int swizzle(int r, int c) {
  if constexpr (CH == 16) {
    return c ^ (r & 15);
  } else {
    static_assert(CH == 8, "KC of 64 or 128");
    return c ^ ((r >> 1) & 7);
  }
}

// Weight row held in LDS row r of tile `tile`.
template <int NT, Epilogue E>
__device__ __forceinline__ int weight_row(const GemmArgs& a, int tile, int r) {
  if constexpr (E == kSwiGLU) {
    return (r < kSwiGLUHalf ? 0 : a.half_rows - kSwiGLUHalf) + tile * kSwiGLUHalf + r;
  } else {
    return tile * NT + r;
  }
}

// DMA of one ring stage: X rows 0..127 (rows past m repeat row m - 1) and the tile's W rows,
// K columns [kbase, kbase + KC).
template <int NT, int KC, int STAGES, int WAVES, Epilogue E>
__device__ __forceinline__ void issue_stage(char* stage, const GemmArgs& a, int tile, int kbase, int wave, int lane) {
  using S = Shape<NT, KC, STAGES, WAVES>;
#pragma unroll
  for (int i = 0; i < S::XI / WAVES; ++i) {
    const int j = i * WAVES + wave;
    const int p = j * 64 + lane;
    const int r = p / S::CH;
    const int c = swizzle<S::CH>(r, p % S::CH);
    const int xr = r < a.m ? r : a.m - 1;
    const _Float16* src = a.x + static_cast<int64_t>(xr) * a.k + kbase + 8 * c;
    __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), lds_ptr(stage + j * 1024), 16, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < S::WI / WAVES; ++i) {
    const int j = i * WAVES + wave;
    const int p = j * 64 + lane;
    const int r = p / S::CH;
    const int c = swizzle<S::CH>(r, p % S::CH);
    const _Float16* src = a.w + static_cast<int64_t>(weight_row<NT, E>(a, tile, r)) * a.k + kbase + 8 * c;
    __builtin_amdgcn_global_load_lds(static_cast<const void*>(src), lds_ptr(stage + S::XB + j * 1024), 16, 0, 0);
  }
}

// Scalar parameters in the order of GemmArgs: all of them are preloaded into SGPRs at wave
// launch (no kernel-argument round trip before the first DMA).
template <int NT, int KC, int STAGES, int WAVES, Epilogue E>
__global__ __launch_bounds__(64 * WAVES) void gemm_m128_kernel(const _Float16* x, const _Float16* w, int m, int n, int k,
                                                               int ksplit, int tiles, int half_rows, void* out) {
  const GemmArgs a{x, w, m, n, k, ksplit, tiles, half_rows, out};
  using S = Shape<NT, KC, STAGES, WAVES>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tile = blockIdx.x % a.tiles;
  const int split = blockIdx.x / a.tiles;
  const int k0 = split * a.ksplit;
  const int steps = a.ksplit / KC;
  float4_t acc[S::NTL][S::MT];
#pragma unroll
  for (int i = 0; i < S::NTL; ++i)
#pragma unroll
    for (int j = 0; j < S::MT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) {
    if (t < steps) issue_stage<NT, KC, STAGES, WAVES, E>(smem + t * S::SB, a, tile, k0 + t * KC, wave, lane);
  }

  const uint32_t lds0 = lds_offset(smem);
  const int r16 = lane & 15, g = lane >> 4;
  for (int t = 0; t < steps; ++t) {
    // This wave's DMA of stage t has landed once at most the later stages already issued
    // (min(STAGES - 2, steps - 1 - t) of them, PER instructions each) are outstanding.
    if constexpr (STAGES == 4) {
      if (t + 2 < steps) wait_vm<2 * S::PER>();
      else if (t + 1 < steps) wait_vm<S::PER>();
      else wait_vm<0>();
    } else {
      static_assert(STAGES == 3, "three or four stages");
      if (t + 1 < steps) wait_vm<S::PER>();
      else wait_vm<0>();
    }
    // Every wave's DMA of stage t has landed, and every wave has finished reading stage
    // t - 1 (its LDS reads were consumed by its MFMAs), which the next DMA overwrites. A
    // bare barrier: a fence here would wait for the DMAs still in flight.
    stage_barrier();
    if (t + STAGES - 1 < steps) {
      issue_stage<NT, KC, STAGES, WAVES, E>(smem + ((t + STAGES - 1) % STAGES) * S::SB, a, tile,
                                            k0 + (t + STAGES - 1) * KC, wave, lane);
    }
    const uint32_t xs = lds0 + (t % STAGES) * S::SB;
    const uint32_t ws = xs + S::XB;
#pragma unroll
    for (int ks = 0; ks < KC / 32; ++ks) {
      // Lane (r16, g) supplies row r16 of each 16-row tile at K columns 32 ks + 8 g .. + 7.
      const int chunk = 4 * ks + g;
      half8_t wf[S::NTL], xf[S::MT];
#pragma unroll
      for (int i = 0; i < S::NTL; ++i) {
        const int r = 16 * i + r16;
        wf[i] = lds_read(ws + (r * S::CH + swizzle<S::CH>(r, chunk)) * 16);
      }
#pragma unroll
      for (int j = 0; j < S::MT; ++j) {
        const int r = 16 * (wave * S::MT + j) + r16;
        xf[j] = lds_read(xs + (r * S::CH + swizzle<S::CH>(r, chunk)) * 16);
      }
#pragma unroll
      for (int i = 0; i < S::NTL; ++i)
#pragma unroll
        for (int j = 0; j < S::MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
  }

  // acc[i][j], lane (r16, g), element e: output row m = 16 (wave MT + j) + r16, column
  // (LDS W row) 16 i + 4 g + e of the tile.
#pragma unroll
  for (int j = 0; j < S::MT; ++j) {
    const int m = 16 * (wave * S::MT + j) + r16;
    if (m >= a.m) continue;
    if constexpr (E == kSwiGLU) {
      const int width = a.half_rows;
#pragma unroll
      for (int i = 0; i < kSwiGLUHalf / 16; ++i) {
        half4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = swiglu(acc[i][j][e], acc[i + kSwiGLUHalf / 16][j][e]);
        const int col = tile * kSwiGLUHalf + 16 * i + 4 * g;
        *reinterpret_cast<half4_t*>(static_cast<_Float16*>(a.out) + static_cast<int64_t>(m) * width + col) = o;
      }
    } else {
#pragma unroll
      for (int i = 0; i < S::NTL; ++i) {
        const int col = tile * NT + 16 * i + 4 * g;
        if constexpr (E == kHalf) {
          half4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = round_h(acc[i][j][e]);
          *reinterpret_cast<half4_t*>(static_cast<_Float16*>(a.out) + static_cast<int64_t>(m) * a.n + col) = o;
        } else {
          float* y = static_cast<float*>(a.out) + (static_cast<int64_t>(split) * a.m + m) * a.n;
          *reinterpret_cast<float4_t*>(y + col) = acc[i][j];
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Wave-private streaming form, for few rows.
//
// One workgroup computes 16 MT rows of X times 16 NT rows of W; its waves split K: wave v
// takes the 64-column units v, v + WAVES, ... of the split's K range, so every byte of the
// tile's X and W is fetched by exactly one wave. Each wave streams its units through a ring
// of D slots of its own by LDS DMA (8 rows x 128 bytes per instruction, whole cache lines)
// and waits only on its own counter: the main loop has no barrier, and up to D units of each
// wave are in flight. The waves' accumulators are added in wave order through LDS at the end.
//
// What bounds it: bytes in flight. The weight stream needs about 50 KB outstanding per CU to
// reach the HBM rate; gemm_m128_kernel's ring holds 128 rows of X for every 64 (or 32) of W,
// whatever m is, which left 24 KB of W in flight. Operand fragments loaded straight to
// registers (16 rows x 64 bytes per instruction) run at 38 bytes/ns per CU against 120-140
// for whole lines, so W goes through LDS as well although only one wave reads it.
// ---------------------------------------------------------------------------------------

template <int MT, int NT, int WAVES, int D>
struct StreamShape {
  static constexpr int XB = MT * 2048;      // X part of a unit: 16 MT rows of 128 bytes
  static constexpr int UB = XB + NT * 2048; // one unit
  static constexpr int PER = 2 * (MT + NT); // DMA instructions per unit
  static constexpr int RING = WAVES * D * UB;
  static constexpr int SUMS = WAVES * MT * NT * 1024;
  static constexpr int LDS = RING > SUMS ? RING : SUMS;
  static_assert(LDS <= 160 * 1024, "ring and accumulator exchange fit the CU's LDS");
  static_assert((D - 1) * PER < 64 && D >= 2 && D <= 4, "vmcnt counts the later units");
};

template <int MT, int NT, int WAVES, int D, Epilogue E>
__global__ __launch_bounds__(64 * WAVES) void gemm_stream_kernel(const _Float16* x, const _Float16* w, int m, int n,
                                                                 int k, int ksplit, int tiles, int mtiles,
                                                                 const int64_t* positions, const int64_t* slots,
                                                                 typename OutOf<E>::type out) {
  using S = StreamShape<MT, NT, WAVES, D>;
  constexpr int kRowsX = 16 * MT, kXBytes = 2048 * MT;
  constexpr int kCols = paired(E) ? 8 * NT : 16 * NT;  // output columns per tile (pairs of them)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15, g = lane >> 4;
  // Workgroups of one W tile (one per X tile) are 8 apart, on one XCD: W comes from HBM once.
  int id = blockIdx.x, mtile = 0;
  if (mtiles > 1) {
    const int q = id >> 3;
    mtile = q % mtiles;
    id = (q / mtiles) * 8 + (id & 7);
  }
  const int tile = id % tiles, split = id / tiles;
  if (split * ksplit >= k) return;  // the grid is rounded up to 8 tiles
  const int limit = paired(E) ? n / 2 : n;
  const int units = ksplit / 64;
  const int mine = (units - wave + WAVES - 1) / WAVES;

  // DMA instruction i of a part covers rows 8 i .. 8 i + 7: lane L takes row 8 i + L / 8 and the
  // chunk stored at position L % 8 (chunk c of row r at c ^ (r & 7)). Rows past the matrix
  // repeat its last row.
  const int row8 = lane >> 3;
  const uint32_t chunk = 16 * ((lane & 7) ^ row8);
  const uint32_t line = 2 * static_cast<uint32_t>(k);
  uint32_t xoff[2 * MT], woff[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) xoff[i] = min(8 * i + row8, m - 1 - kRowsX * mtile) * line + chunk;
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) {
    const int r = 8 * i + row8;
    if constexpr (E == kSwiGLU) {
      const int last = limit - 1 - kCols * tile;
      woff[i] = (r < kCols ? min(r, last) : limit + min(r - kCols, last)) * line + chunk;
    } else if constexpr (E == kRope) {
      const int first = pair_row(kCols * tile);  // a tile's pairs are consecutive rows of one head
      woff[i] = (first + (r < kCols ? r : kHalfDim + r - kCols)) * line + chunk;
    } else {
      woff[i] = min(r, limit - 1 - kCols * tile) * line + chunk;
    }
  }
  // RoPE: thread e ends with quad e % Q of row e / Q of the tile (one each at most). Its position
  // and slot are loaded before the stream's first unit and the table values behind it, so that
  // the stream hides both round trips (loads return in order: an older one in flight only
  // makes the waits below longer).
  constexpr int Q = kCols / 4;  // groups of four output columns
  static_assert(E != kRope || (kHalfDim % kCols == 0 && Q * kRowsX <= 64 * WAVES), "one quad of one head per thread");
  int64_t position = 0, slot = 0;
  if constexpr (E == kRope) {
    const int row = min(kRowsX * mtile + static_cast<int>(threadIdx.x) / Q, m - 1);
    position = positions[row];
    slot = (slots != nullptr ? slots : positions)[row];
  }
  const int64_t k0 = static_cast<int64_t>(split) * ksplit + 64 * wave;
  const char* xbase = reinterpret_cast<const char*>(x + static_cast<int64_t>(kRowsX) * mtile * k + k0);
  const char* wbase = reinterpret_cast<const char*>(w + (E == kRope ? 0 : static_cast<int64_t>(kCols) * tile * k) + k0);
  char* const ring = smem + wave * D * S::UB;
  auto issue = [&](char* slot) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(wbase + woff[i]), lds_ptr(slot + kXBytes + i * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(xbase + xoff[i]), lds_ptr(slot + i * 1024), 16, 0, 0);
    asm volatile("" ::: "memory");
    wbase += 128 * WAVES;
    xbase += 128 * WAVES;
  };

  float4_t acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < D; ++t) {
    if (t < mine) issue(ring + t * S::UB);
  }
  [[maybe_unused]] RopeRow rope{};
  [[maybe_unused]] half4_t cs{}, sn{};
  if constexpr (E == kRope) {
    rope = rope_row(out, position, slot, slots != nullptr);
    const _Float16* table = rope.table + (kCols * tile + 4 * (static_cast<int>(threadIdx.x) % Q)) % kHalfDim;
    cs = *reinterpret_cast<const half4_t*>(table);
    sn = *reinterpret_cast<const half4_t*>(table + kHalfDim);
  }

  const uint32_t ring0 = lds_offset(ring);
  const uint32_t a0 = r16 * 128 + ((g ^ (r16 & 7)) * 16), a1 = r16 * 128 + (((4 + g) ^ (r16 & 7)) * 16);
  // Unit t in slot d: its DMA has landed once at most `later` units issued after it are
  // outstanding.
  auto unit = [&](int d) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t base = ring0 + d * S::UB + (s ? a1 : a0);
      half8_t wf[NT], xf[MT];
#pragma unroll
      for (int i = 0; i < NT; ++i) wf[i] = lds_read(base + S::XB + i * 2048);
#pragma unroll
      for (int j = 0; j < MT; ++j) xf[j] = lds_read(base + j * 2048);
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
  };
  int t = 0;
  // Steady state: D units per pass, each refilled as soon as its LDS reads are done.
#pragma nounroll
  for (; t + 2 * D <= mine; t += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      wait_vm<(D - 1) * S::PER>();
      unit(d);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(ring + d * S::UB);
    }
  }
  // The last up to 2 D - 1 units (slot t % D, as t is a multiple of D here).
#pragma unroll
  for (int e = 0; e < 2 * D - 1; ++e) {
    if (t + e < mine) {
      const int later = mine - 1 - t - e;
      if (D > 3 && later >= 3) wait_vm<3 * S::PER>();
      else if (D > 2 && later >= 2) wait_vm<2 * S::PER>();
      else if (later >= 1) wait_vm<S::PER>();
      else wait_vm<0>();
      unit(e % D);
      if (e + D < 2 * D - 1 && t + e + D < mine) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(ring + (e % D) * S::UB);
      }
    }
  }

  // Accumulators to LDS (over the rings, once every wave is done with its own), then added in
  // wave order: acc[i][j] of lane (r16, g) holds X row 16 j + r16, W rows 16 i + 4 g .. + 3.
  __syncthreads();
  float4_t* sums = reinterpret_cast<float4_t*>(smem);
  constexpr int T = MT * NT;
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) sums[(wave * T + i * MT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int e = threadIdx.x; e < Q * kRowsX; e += 64 * WAVES) {
    const int q = e % Q, r = e / Q;
    const int row = kRowsX * mtile + r, col = kCols * tile + 4 * q;
    auto total = [&](int quad) {
      const float4_t* p = sums + ((quad >> 2) * MT + (r >> 4)) * 64 + 16 * (quad & 3) + (r & 15);
      float4_t v = p[0];
#pragma unroll
      for (int u = 1; u < WAVES; ++u) v += p[u * T * 64];
      return v;
    };
    if (row >= m || col >= limit) continue;
    if constexpr (E == kSwiGLU) {
      const float4_t gate = total(q), up = total(Q + q);
      half4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = swiglu(gate[i], up[i]);
      *reinterpret_cast<half4_t*>(static_cast<_Float16*>(out) + static_cast<int64_t>(row) * limit + col) = o;
    } else if constexpr (E == kRope) {
      const float4_t low = total(q), high = total(Q + q);
      half4_t lo, hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = round_h(low[i]);
        hi[i] = round_h(high[i]);
      }
      store_pairs(out, rope, row, col, lo, hi, cs, sn);
    } else {
      const float4_t v = total(q);
      if constexpr (E == kHalf) {
        half4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = round_h(v[i]);
        *reinterpret_cast<half4_t*>(static_cast<_Float16*>(out) + static_cast<int64_t>(row) * n + col) = o;
      } else {
        float* y = static_cast<float*>(out) + (static_cast<int64_t>(split) * m + row) * n + col;
        *reinterpret_cast<float4_t*>(y) = v;
      }
    }
  }
}

template <int NT, int KC, int STAGES, int WAVES, Epilogue E>
int launch(GemmArgs a, int splits, hipStream_t s) {
  using S = Shape<NT, KC, STAGES, WAVES>;
  if (a.ksplit % KC != 0) {
    return set_error(PC_ERR_ARGUMENT, "k per split (%d) must be a multiple of %d", a.ksplit, KC);
  }
  auto kernel = gemm_m128_kernel<NT, KC, STAGES, WAVES, E>;
  static std::atomic<uint64_t> raised{0};
  if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), S::LDS, raised)) return rc;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.tiles * splits)), dim3(64 * WAVES), S::LDS, s, a.x, a.w, a.m,
                     a.n, a.k, a.ksplit, a.tiles, a.half_rows, a.out);
  return check_launch("gemm_m128");
}

template <int MT, int NT, int WAVES, int D, Epilogue E>
int launch_stream(const GemmArgs& a, int splits, const int64_t* positions, const int64_t* slots,
                  typename OutOf<E>::type out, hipStream_t s) {
  using S = StreamShape<MT, NT, WAVES, D>;
  if (a.ksplit % 64 != 0) return set_error(PC_ERR_ARGUMENT, "k per split (%d) must be a multiple of 64", a.ksplit);
  auto kernel = gemm_stream_kernel<MT, NT, WAVES, D, E>;
  static std::atomic<uint64_t> raised{0};
  if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), S::LDS, raised)) return rc;
  constexpr int cols = paired(E) ? 8 * NT : 16 * NT;
  const int tiles = ((paired(E) ? a.n / 2 : a.n) + cols - 1) / cols;
  const int mtiles = (a.m + 16 * MT - 1) / (16 * MT);
  int64_t grid = static_cast<int64_t>(tiles) * splits;
  if (mtiles > 1) grid = (grid + 7) / 8 * 8 * mtiles;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * WAVES), S::LDS, s, a.x, a.w, a.m, a.n, a.k,
                     a.ksplit, tiles, mtiles, positions, slots, out);
  return check_launch("gemm_stream");
}

template <int MT, int NT, int WAVES, int D, Epilogue E>
int launch_stream(const GemmArgs& a, int splits, hipStream_t s) {
  return launch_stream<MT, NT, WAVES, D, E>(a, splits, nullptr, nullptr, a.out, s);
}

constexpr int kCUs = 256;

// X tile (in 16 rows) of a launch with `wtiles` W tiles: the fewest rows per workgroup that give each
// CU at most one workgroup, up to 64; beyond that 48 rows, of which two workgroups fit a CU.
int x_tile(int m, int wtiles) {
  const int places = wtiles < kCUs ? kCUs / wtiles : 1;
  const int mt = (m + 16 * places - 1) / (16 * places);
  return mt <= 4 ? mt : 3;
}

// A form of gemm_stream_kernel: 16 mt rows of X times 16 nt rows of W per workgroup.
struct StreamTile {
  int mt, nt;
};
constexpr StreamTile kStreamTiles[] = {{1, 2}, {2, 2}, {3, 2}, {4, 2}, {2, 3}, {3, 3}, {4, 3}};

template <Epilogue E>
int launch_stream_tile(const GemmArgs& a, StreamTile t, int splits, hipStream_t s) {
  switch (t.mt + (t.nt == 3 ? 10 : 0)) {
    case 1: return launch_stream<1, 2, 4, 2, E>(a, splits, s);
    case 2: return launch_stream<2, 2, 4, 2, E>(a, splits, s);
    case 3: return launch_stream<3, 2, 4, 2, E>(a, splits, s);
    case 4: return launch_stream<4, 2, 4, 2, E>(a, splits, s);
    case 12: return launch_stream<2, 3, 4, 2, E>(a, splits, s);
    case 13: return launch_stream<3, 3, 4, 2, E>(a, splits, s);
    default: return launch_stream<4, 3, 4, 2, E>(a, splits, s);
  }
}

int64_t rounds(int64_t workgroups) { return (workgroups + kCUs - 1) / kCUs; }

// 64-row W tiles of gemm_m128_kernel: with eight waves when they alone fill the GPU's workgroup
// slots; with four waves (2 x 4 register tiles per wave) when they give 160 to 175 workgroups,
// where 32-row tiles would need more workgroups than one round on the CUs (q|k|v at 4
// splits: 7.5 vs 8.3 us); else 32-row tiles with four waves.
enum M128Tile { k32x4, k64x4, k64x8 };
M128Tile m128_tile(int n, int splits) {
  const int64_t tiles64 = n % 64 == 0 ? static_cast<int64_t>(n / 64) * splits : 0;
  if (tiles64 >= 176) return k64x8;
  return tiles64 >= 160 && static_cast<int64_t>(n / 32) * splits > kCUs ? k64x4 : k32x4;
}

// Which form takes a call, from an estimate of its time (us; a constant common to all is left out):
// rounds of workgroups on the CUs times a round's setup and the bytes it moves into a CU. A later
// round overlaps an earlier one where workgroups share a CU (two of up to 80 KB of LDS; three of 48 KB,
// while a K range is short enough for the L2 to hold what they share). The constants are fitted to
// the times of every form at 23000 calls (m 1 to 128, n 32 to 37000, k 64 to 16000, 1 to 16
// splits, weights from HBM): the form taken is 2 % off the fastest on average; it is more than 5 %
// slower than gemm_m128_kernel alone at 0.4 % of them (17 % at most) and 35 % faster on average. A
// rule on the number of W tiles was more than 5 % slower at 15 % of them, by up to 2.2 times (SwiGLU of n
// 14336 at 64 rows 20.7 / 15.0, 299 tiles of 48 rows; n 7136, k 256 at 111 rows 5.8 / 4.1).
float stream_time(const GemmArgs& a, int splits, StreamTile t) {
  const int64_t workgroups =
      static_cast<int64_t>((a.n + 16 * t.nt - 1) / (16 * t.nt)) * splits * ((a.m + 16 * t.mt - 1) / (16 * t.mt));
  const int lds_kb = 16 * (t.mt + t.nt), units = a.ksplit / 64;
  const int64_t r = rounds(workgroups);
  const float overlap = r == 1 || lds_kb > 80 ? 1.0f : lds_kb > 48 || units > 16 ? 0.88f : 0.75f;
  const float round = (lds_kb > 80 ? 0.7f : 0.22f) + 0.074f * (t.mt + t.nt) * ((units + 3) / 4);  // units per wave
  return overlap * r * round + 0.066e-6f * a.n * static_cast<float>(a.k);
}

float m128_time(const GemmArgs& a, int splits, M128Tile t) {
  const int nt = t == k32x4 ? 2 : 4;
  const int64_t r = rounds(static_cast<int64_t>(a.n / (16 * nt)) * splits);
  const float overlap = r == 1 || t != k32x4 ? 1.0f : 0.8f;
  return 0.15f + overlap * r * (0.055f + 0.022f * (8 + nt) * (a.ksplit / 64));
}

// The fastest stream form, of those with 48-row W tiles alone if `wide`, and its time.
StreamTile stream_tile(const GemmArgs& a, int splits, bool wide, float& time) {
  StreamTile best{1, 2};
  time = INFINITY;
  for (const StreamTile t : kStreamTiles) {
    if (16 * (t.mt - 1) >= a.m || (wide && t.nt != 3)) continue;
    const float estimate = stream_time(a, splits, t);
    if (estimate < time) time = estimate, best = t;
  }
  return best;
}

constexpr int kMaxStreamQkv = 288;  // rows of the last form below

// RoPE epilogue, 80 tiles of 16 column pairs: the fewest rows per workgroup that still give each
// CU at most one (us with weights from HBM, against the partials of pc_gemm_m128 at 2 splits and
// pc_rope_kv_append_parts: 1 row 5.5 / 6.4, 16 rows 5.8 / 7.0, 37 rows 6.3 / 7.8, 48 rows 6.7 / 8.1,
// 64 rows 7.7 / 9.2, 96 rows 7.7 / 10.4, 128 rows 8.4 / 10.2, 160 rows 8.9 / 11.6; at 48 rows 32
// of them per workgroup 7.2, at 64 rows 16 per workgroup 8.9). One 16-row tile alone leaves
// CUs idle: 160 tiles of 8 pairs (16 rows 5.8, 80 tiles 6.7). Above that 48 rows, two workgroups
// per CU (256 rows 11.6 / 13.9, the best tile of launch_qkv_rows 12.3).
int launch_qkv_stream(const QkvArgs& q, hipStream_t s) {
  const GemmArgs a{q.x, q.w, q.m, kQkvElems, q.k, q.k, 0, 0, nullptr};
  if (q.m <= 16) return launch_stream<1, 1, 4, 3, kRope>(a, 1, q.positions, q.slots, q.out, s);
  switch (x_tile(q.m, kQkvElems / 32)) {
    case 1: return launch_stream<1, 2, 4, 3, kRope>(a, 1, q.positions, q.slots, q.out, s);
    case 2: return launch_stream<2, 2, 4, 2, kRope>(a, 1, q.positions, q.slots, q.out, s);
    case 4: return launch_stream<4, 2, 4, 2, kRope>(a, 1, q.positions, q.slots, q.out, s);
    default: return launch_stream<3, 2, 4, 2, kRope>(a, 1, q.positions, q.slots, q.out, s);
  }
}

}  // namespace

namespace gemm_device {

// The rows and columns of the q|k|v projection above, so that an unsplit product of 2560 columns has
// pc_qkv_rope_append's bits at every row count (from 289 rows both are on tiles, which all add in one
// order; k from 256, where every wave has a unit). It and narrower products are also faster here than on 64 x 64 tiles (us: n 2560 at 160
// rows 6.9 / 10.5, at 288 9.5 / 10.6; n 2048 at 256 rows 7.0 / 10.4; n 512 4.9 / 10.3), wider ones
// hardly or not (n 5632 at 160 rows 14.6 / 14.9, at 96 12.2 / 11.5).
bool rows_stream(int m, int n, int k) { return m <= kMaxStreamQkv && n <= kQkvElems && k >= 256 && k <= kMaxStreamK; }

int launch_rows_stream(void* out, const _Float16* x, const _Float16* w, int m, int n, int k, Epilogue epilogue,
                       hipStream_t s) {
  const GemmArgs a{x, w, m, n, k, k, 0, 0, out};
  const int mt = x_tile(m, n / 32);
  if (epilogue == kHalf) return launch_stream_tile<kHalf>(a, {mt, 2}, 1, s);
  if (epilogue == kPartials) return launch_stream_tile<kPartials>(a, {mt, 2}, 1, s);
  switch (mt) {
    case 1: return launch_stream<1, 1, 4, 3, kSwiGLU>(a, 1, s);
    case 2: return launch_stream<2, 3, 4, 2, kSwiGLU>(a, 1, s);
    case 3: return launch_stream<3, 3, 4, 2, kSwiGLU>(a, 1, s);
    default: return launch_stream<4, 3, 4, 2, kSwiGLU>(a, 1, s);
  }
}

}  // namespace gemm_device

namespace {

// Whether a call of pc_gemm_m128 runs on gemm_stream_kernel: by m, n, k and splits alone, not by
// epilogue (an unsplit product only if every epilogue gains), and always with four waves, so that one
// product has the same bits under every epilogue, and under two row counts that are sent to
// the same kernel (each projection of the decoder from 1 to 64 rows, and from 65 to 128).
constexpr float kMargin = 1.1f;  // where the estimates are close, gemm_m128_kernel
bool stream_form(const GemmArgs& a, int splits) {
  if (a.ksplit % 64 != 0 || a.k > kMaxStreamK) return false;
  if (splits == 1 && rows_stream(a.m, a.n, a.k)) return true;
  // A K range of fewer units than waves leaves waves idle (n 1024, k 128 per split, 48 rows: 3.5
  // us / 3.1; k 64, n 15488, SwiGLU at 12 rows 4.2 / 3.2).
  const int units = a.ksplit / 64;
  if (units < 4 && a.m > 16 * units) return false;
  if (units == 1 && splits == 1 && a.n > 48 * kCUs) return false;
  if (a.m <= 16) return true;
  float time;
  if (splits == 1 && a.n % 64 == 0) {  // SwiGLU, which has tiles of its own
    stream_tile(a, 1, true, time);
    if (kMargin * time >= m128_time(a, 1, k64x8)) return false;
  }
  stream_tile(a, splits, false, time);
  return kMargin * time < m128_time(a, splits, m128_tile(a.n, splits));
}

}  // namespace

extern "C" {

int pc_qkv_rope_append(void* query_out, void* key_out, void* value_out, const void* x, const void* w, int32_t m, int32_t k,
                       const int64_t* positions, const void* rope_table, int32_t rope_positions, void* pool,
                       int64_t num_blocks, int32_t layer, const int64_t* slot_mapping, void* stream) {
  if (!query_out || !x || !w || !positions || !rope_table) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (m < 1 || m > (1 << 16)) return set_error(PC_ERR_ARGUMENT, "m = %d outside [1, 65536]", m);
  if (k < 64 || k % 64 != 0 || k > kMaxQkvK || static_cast<int64_t>(m) * k > (int64_t{1} << 31)) {
    return set_error(PC_ERR_ARGUMENT, "k = %d must be a multiple of 64 up to %d, m * k up to 2^31", k, kMaxQkvK);
  }
  if (rope_positions < 1) return set_error(PC_ERR_ARGUMENT, "rope_positions must be positive");
  if ((pool == nullptr) != (slot_mapping == nullptr)) {
    return set_error(PC_ERR_ARGUMENT, "pool and slot_mapping must both be given or both be null");
  }
  if (pool != nullptr) {
    if (num_blocks < 1 || num_blocks > INT32_MAX) {
      return set_error(PC_ERR_ARGUMENT, "num_blocks %lld out of range", static_cast<long long>(num_blocks));
    }
    if (layer < 0 || layer >= kLayers) return set_error(PC_ERR_ARGUMENT, "layer %d outside [0, 22)", layer);
  }
  if (!aligned(query_out, 16) || !aligned(x, 16) || !aligned(w, 16) || !aligned(rope_table, 16) || !aligned(pool, 16) ||
      !aligned(key_out, 16) || !aligned(value_out, 16)) {
    return set_error(PC_ERR_ARGUMENT, "buffers must be 16-byte aligned");
  }
  QkvArgs a;
  a.x = static_cast<const _Float16*>(x);
  a.w = static_cast<const _Float16*>(w);
  a.m = m;
  a.k = k;
  a.positions = positions;
  a.slots = slot_mapping;
  a.out.table = static_cast<const _Float16*>(rope_table);
  a.out.table_positions = rope_positions;
  a.out.query = static_cast<_Float16*>(query_out);
  a.out.kind_elems = pool ? num_blocks * kSlots * kRowElems : 0;
  a.out.layer_pool = pool ? static_cast<_Float16*>(pool) + static_cast<int64_t>(layer) * 2 * a.out.kind_elems : nullptr;
  a.out.key = static_cast<_Float16*>(key_out);
  a.out.value = static_cast<_Float16*>(value_out);
  (void)hipGetLastError();
  return m <= kMaxStreamQkv ? launch_qkv_stream(a, static_cast<hipStream_t>(stream))
                       : launch_qkv_rows(a, static_cast<hipStream_t>(stream));
}

int pc_gemm_m128(void* out, const void* x, const void* w, int32_t m, int32_t n, int32_t k, int32_t splits,
                 int32_t epilogue, void* stream) {
  if (!out || !x || !w) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (m < 1 || m > kMaxRows) return set_error(PC_ERR_ARGUMENT, "m = %d outside [1, %d]", m, kMaxRows);
  if (n < 1 || k < 1 || splits < 1) return set_error(PC_ERR_ARGUMENT, "n, k and splits must be positive");
  if (k % splits != 0) return set_error(PC_ERR_ARGUMENT, "k = %d not divisible into %d splits", k, splits);
  if (static_cast<int64_t>(n) * k > (int64_t{1} << 31) || static_cast<int64_t>(splits) * m * n > (int64_t{1} << 31)) {
    return set_error(PC_ERR_ARGUMENT, "GEMM of %d x %d x %d with %d splits too large", m, n, k, splits);
  }
  if (!aligned(out, 16) || !aligned(x, 16) || !aligned(w, 16)) {
    return set_error(PC_ERR_ARGUMENT, "out, x and w must be 16-byte aligned");
  }
  GemmArgs a;
  a.x = static_cast<const _Float16*>(x);
  a.w = static_cast<const _Float16*>(w);
  a.out = out;
  a.m = m;
  a.n = n;
  a.k = k;
  a.ksplit = k / splits;
  a.half_rows = 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  switch (epilogue) {
    case kPartials:
    case kHalf:
      if (epilogue == kHalf && splits != 1) return set_error(PC_ERR_ARGUMENT, "fp16 output needs one split");
      if (n % 32 != 0) return set_error(PC_ERR_ARGUMENT, "n = %d must be a multiple of 32", n);
      if (splits == 1 && rows_stream(m, n, k)) return launch_rows_stream(out, a.x, a.w, m, n, k, static_cast<Epilogue>(epilogue), s);
      if (stream_form(a, splits)) {
        float time;
        const StreamTile t = stream_tile(a, splits, false, time);
        return epilogue == kHalf ? launch_stream_tile<kHalf>(a, t, splits, s) : launch_stream_tile<kPartials>(a, t, splits, s);
      }
      switch (m128_tile(n, splits)) {
        case k64x8:
          a.tiles = n / 64;
          return epilogue == kHalf ? launch<64, 64, 4, 8, kHalf>(a, splits, s) : launch<64, 64, 4, 8, kPartials>(a, splits, s);
        case k64x4:
          a.tiles = n / 64;
          return epilogue == kHalf ? launch<64, 64, 4, 4, kHalf>(a, splits, s) : launch<64, 64, 4, 4, kPartials>(a, splits, s);
        default:
          a.tiles = n / 32;
          return epilogue == kHalf ? launch<32, 64, 4, 4, kHalf>(a, splits, s) : launch<32, 64, 4, 4, kPartials>(a, splits, s);
      }
    case kSwiGLU:
      if (splits != 1) return set_error(PC_ERR_ARGUMENT, "the SwiGLU epilogue needs one split");
      if (n % (2 * kSwiGLUHalf) != 0) return set_error(PC_ERR_ARGUMENT, "n = %d must be a multiple of 64", n);
      if (rows_stream(m, n, k)) return launch_rows_stream(out, a.x, a.w, m, n, k, kSwiGLU, s);
      // One tile per 8 NT gate rows: 704 small tiles at one X tile (11.0 us at 16 rows, 235
      // tiles of 24 gate rows the same), 235 above it (14.6 -> 11.5 us at 32 rows).
      if (stream_form(a, splits)) {
        if (m <= 16) return launch_stream<1, 1, 4, 3, kSwiGLU>(a, splits, s);
        float time;
        switch (stream_tile(a, splits, true, time).mt) {
          case 2: return launch_stream<2, 3, 4, 2, kSwiGLU>(a, splits, s);
          case 3: return launch_stream<3, 3, 4, 2, kSwiGLU>(a, splits, s);
          default: return launch_stream<4, 3, 4, 2, kSwiGLU>(a, splits, s);
        }
      }
      if (k % 64 == 0 && swiglu_short_tiles(m, n, k)) return launch_swiglu_short(out, a.x, a.w, m, n, k, s);
      a.half_rows = n / 2;
      a.tiles = n / (2 * kSwiGLUHalf);
      return launch<64, 64, 4, 8, kSwiGLU>(a, splits, s);
    default:
      return set_error(PC_ERR_ARGUMENT, "unknown epilogue %d", epilogue);
  }
}

}  // extern "C"
