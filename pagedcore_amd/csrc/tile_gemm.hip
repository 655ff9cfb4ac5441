// Projection GEMM for more rows than a decode step has (a prompt's forward): Y = X W^T with X
// fp16 [m][k] and W fp16 [n][k], fp32 accumulation, and the epilogues of pc_gemm_m128 (fp32
// split-K partials, fp16, SwiGLU). It takes the place of torch.nn.functional.linear on a
// prompt's activations (reference src/pagedcore/dense.py:91-104 via decoder.py:113-135).
//
// One workgroup computes a BM x BN tile over one split's K range; its WM x WN waves own
// (BM / WM) x (BN / WN) of it. X and W stream through a ring of ST stages of 64 columns
// (LDS DMA, whole 128-byte lines, chunks swizzled so that the operand reads are free of bank
// conflicts), one barrier per stage. The second half's operand fragments are read before the
// first half's MFMAs, and the next stage's first half before the second half's, so LDS latency
// and the barrier hide behind matrix work.
//
// What bounds it at a prompt's sizes: bytes into each CU (an L2 that misses to the memory side
// delivers about 50 bytes/ns to each of 256 CUs, 115 where all hits) and, from about 1000
// rows, power: MFMA with LDS reads beside it runs at 1.7 GHz instead of 2.4. So tiles are as
// large as still give every CU one, K is split where the tiles alone are too few, and each
// XCD works on a compact block of tiles, which cuts what its L2 has to fetch (gate|up at 2048
// rows 98.9 -> 95.6 us, down at 1024 rows 31.7 -> 29.8 against rows of tiles dealt round).

#include "gemm_device.h"

namespace {

using namespace gemm_device;
using namespace rope_device;
using pc_internal::aligned;
using pc_internal::check_launch;
using pc_internal::set_error;

constexpr int kMaxRows = 1 << 16;
constexpr int kMaxK = 1 << 22;  // tile-relative byte offsets fit 32 bits
constexpr int kCUs = 256;
constexpr int kXCDs = 8;
constexpr int kTileGroup = 8;  // X tiles that one XCD walks together

struct TileArgs {
  const _Float16* x;
  const _Float16* w;
  int m, n, k, ksplit;
  void* out;
};

template <int BM, int BN, int WM, int WN, int ST, Epilogue E>
__global__ __launch_bounds__(64 * WM * WN) void gemm_tile_kernel(const _Float16* x, const _Float16* w, int m, int n,
                                                                 int k, int ksplit, int ntiles, int mtiles,
                                                                 const int64_t* positions, const int64_t* slots,
                                                                 typename OutOf<E>::type out) {
  constexpr int kWaves = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN, MT = TM / 16, NT = TN / 16;
  constexpr int kXBytes = BM * 128, kStage = (BM + BN) * 128;      // one stage: X rows, then W rows, 128 bytes each
  constexpr int XI = BM / 8 / kWaves, WI = BN / 8 / kWaves;        // DMA instructions per wave and stage
  constexpr int kPer = XI + WI;
  constexpr int kCols = paired(E) ? BN / 2 : BN;                   // output columns (or pairs) per tile
  static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0 && TN % 32 == 0, "waves share the tile evenly");
  static_assert((ST - 1) * kPer < 64 && ST >= 2 && ST <= 4, "vmcnt counts the later stages");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;

  // XCD j takes the j-th eighth of the tiles (the hardware deals workgroups to XCDs in turn):
  // splits slowest, then groups of kTileGroup X tiles, W tiles, and X tiles fastest.
  const int tiles = ntiles * mtiles;
  const int total = tiles * (k / ksplit);
  const int share = (total + kXCDs - 1) / kXCDs;
  int u = (blockIdx.x % kXCDs) * share + blockIdx.x / kXCDs;
  if (u >= total) return;  // the grid is rounded up to whole shares
  const int split = u / tiles;
  u -= split * tiles;
  const int group = u / (kTileGroup * ntiles);
  const int in_group = min(kTileGroup, mtiles - kTileGroup * group);
  u -= group * kTileGroup * ntiles;
  const int tile = u / in_group, mtile = kTileGroup * group + u % in_group;

  const int limit = paired(E) ? n / 2 : n;
  // DMA instruction i of a part covers rows 8 i .. 8 i + 7: lane L takes row 8 i + L / 8 and the
  // chunk stored at position L % 8 (chunk c of row r at c ^ (r & 7)). Rows past the matrix
  // repeat its last row. SwiGLU: each wave's W rows are TN / 2 gate rows, then their up rows; RoPE:
  // TN / 2 columns d < 32 of the heads, then their partners d + 32.
  const int row8 = lane >> 3;
  const uint32_t chunk = 16 * ((lane & 7) ^ row8);
  const uint32_t line = 2 * static_cast<uint32_t>(k);
  uint32_t xoff[XI], woff[WI];
#pragma unroll
  for (int i = 0; i < XI; ++i) xoff[i] = min(8 * (i * kWaves + wave) + row8, m - 1 - BM * mtile) * line + chunk;
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = 8 * (i * kWaves + wave) + row8;
    const int last = limit - 1 - kCols * tile;
    if constexpr (E == kRope) {
      const int base = (r / TN) * (TN / 2), in = r % TN, upper = in >= TN / 2;
      const int pair = kCols * tile + min(base + in - upper * (TN / 2), last);
      woff[i] = (pair_row(pair) + upper * kHalfDim) * line + chunk;
    } else if constexpr (E == kSwiGLU) {
      const int base = (r / TN) * (TN / 2), in = r % TN;
      woff[i] = (in < TN / 2 ? min(base + in, last) : limit + min(base + in - TN / 2, last)) * line + chunk;
    } else {
      woff[i] = min(r, last) * line + chunk;
    }
  }
  const int64_t k0 = static_cast<int64_t>(split) * ksplit;
  const char* xbase = reinterpret_cast<const char*>(x + static_cast<int64_t>(BM) * mtile * k + k0);
  const char* wbase = reinterpret_cast<const char*>(w + (E == kRope ? 0 : static_cast<int64_t>(kCols) * tile * k) + k0);
  // RoPE: the positions and slots of the wave's rows, before the stream (see the end).
  [[maybe_unused]] int64_t position[MT], token_slot[MT];
  if constexpr (E == kRope) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int row = min(BM * mtile + wm * TM + 16 * j + r16, m - 1);
      position[j] = positions[row];
      token_slot[j] = (slots != nullptr ? slots : positions)[row];
    }
  }
  auto issue = [&](char* stage) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < WI; ++i)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(wbase + woff[i]),
                                       lds_ptr(stage + kXBytes + (i * kWaves + wave) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < XI; ++i)
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(xbase + xoff[i]),
                                       lds_ptr(stage + (i * kWaves + wave) * 1024), 16, 0, 0);
    asm volatile("" ::: "memory");
    wbase += 128;
    xbase += 128;
  };
  float4_t acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int steps = ksplit / 64;
#pragma unroll
  for (int t = 0; t < ST; ++t) {
    if (t < steps) issue(smem + t * kStage);
  }

  const uint32_t lds0 = lds_offset(smem);
  const uint32_t a0 = lds0 + r16 * 128 + ((g ^ (r16 & 7)) * 16), a1 = lds0 + r16 * 128 + (((4 + g) ^ (r16 & 7)) * 16);
  half8_t wfa[NT], xfa[MT], wfb[NT], xfb[MT];  // fragments of a stage's columns 0-31 and 32-63
  auto read = [&](half8_t(&wf)[NT], half8_t(&xf)[MT], uint32_t base) {
#pragma unroll
    for (int i = 0; i < NT; ++i) wf[i] = lds_read(base + kXBytes + (wn * TN + 16 * i) * 128);
#pragma unroll
    for (int j = 0; j < MT; ++j) xf[j] = lds_read(base + (wm * TM + 16 * j) * 128);
  };
  auto multiply = [&](half8_t(&wf)[NT], half8_t(&xf)[MT]) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[i], xf[j], acc[i][j], 0, 0, 0);
  };
  // A stage has landed for every wave: at most `later` stages issued after it are outstanding
  // in this one, and the barrier holds until the others say the same.
  auto landed = [&](int later) {
    if (ST > 3 && later == 3) wait_vm<3 * kPer>();
    else if (ST > 2 && later == 2) wait_vm<2 * kPer>();
    else if (later == 1) wait_vm<kPer>();
    else wait_vm<0>();
    stage_barrier();
  };
  landed(min(ST - 1, steps - 1));
  read(wfa, xfa, a0);
  int slot = 0;
#pragma nounroll
  for (int t = 0; t < steps; ++t) {
    read(wfb, xfb, a1 + slot * kStage);
    __builtin_amdgcn_sched_barrier(0);
    multiply(wfa, xfa);
    __builtin_amdgcn_sched_barrier(0);
    // This wave has read all of stage t; once every wave has (the barrier below), its slot is
    // refilled with stage t + ST.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int next = slot + 1 == ST ? 0 : slot + 1;
    if (t + 1 < steps) {
      landed(min(ST - 2, steps - 2 - t));
      if (t + ST < steps) issue(smem + slot * kStage);
      read(wfa, xfa, a0 + next * kStage);
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(wfb, xfb);
    __builtin_amdgcn_sched_barrier(0);
    slot = next;
  }

  // acc[i][j] of lane (r16, g), element e: X row wm TM + 16 j + r16, W row wn TN + 16 i + 4 g + e
  // of the tile.
  [[maybe_unused]] RopeRow rope[MT];
  [[maybe_unused]] half4_t cs[NT / 2][MT], sn[NT / 2][MT];
  if constexpr (E == kRope) {  // every table value the wave needs in one round trip
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      rope[j] = rope_row(out, position[j], token_slot[j], slots != nullptr);
#pragma unroll
      for (int i = 0; i < NT / 2; ++i) {
        const _Float16* table = rope[j].table + (kCols * tile + wn * (TN / 2) + 16 * i + 4 * g) % kHalfDim;
        cs[i][j] = *reinterpret_cast<const half4_t*>(table);
        sn[i][j] = *reinterpret_cast<const half4_t*>(table + kHalfDim);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int row = BM * mtile + wm * TM + 16 * j + r16;
    if (row >= m) continue;
    if constexpr (E == kRope) {
#pragma unroll
      for (int i = 0; i < NT / 2; ++i) {
        const int pair = kCols * tile + wn * (TN / 2) + 16 * i + 4 * g;
        half4_t lo, hi;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          lo[e] = round_h(acc[i][j][e]);
          hi[e] = round_h(acc[i + NT / 2][j][e]);
        }
        if (pair < limit) store_pairs(out, rope[j], row, pair, lo, hi, cs[i][j], sn[i][j]);
      }
    } else if constexpr (E == kSwiGLU) {
#pragma unroll
      for (int i = 0; i < NT / 2; ++i) {
        const int col = kCols * tile + wn * (TN / 2) + 16 * i + 4 * g;
        half4_t o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = swiglu(acc[i][j][e], acc[i + NT / 2][j][e]);
        if (col < limit) *reinterpret_cast<half4_t*>(static_cast<_Float16*>(out) + static_cast<int64_t>(row) * limit + col) = o;
      }
    } else {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int col = kCols * tile + wn * TN + 16 * i + 4 * g;
        if (col >= limit) continue;
        if constexpr (E == kHalf) {
          half4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = round_h(acc[i][j][e]);
          *reinterpret_cast<half4_t*>(static_cast<_Float16*>(out) + static_cast<int64_t>(row) * n + col) = o;
        } else {
          *reinterpret_cast<float4_t*>(static_cast<float*>(out) + (static_cast<int64_t>(split) * m + row) * n + col) = acc[i][j];
        }
      }
    }
  }
}

int64_t tile_count(const TileArgs& a, int bm, int cols, int width) {
  return static_cast<int64_t>((a.m + bm - 1) / bm) * ((width + cols - 1) / cols) * (a.k / a.ksplit);
}

template <int BM, int BN, int WM, int WN, int ST, Epilogue E>
int launch(const TileArgs& a, const int64_t* positions, const int64_t* slots, typename OutOf<E>::type out, hipStream_t s) {
  constexpr int lds = ST * (BM + BN) * 128;
  static_assert(lds <= 160 * 1024, "ring fits the CU's LDS");
  auto kernel = gemm_tile_kernel<BM, BN, WM, WN, ST, E>;
  static std::atomic<uint64_t> raised{0};
  if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, raised)) return rc;
  constexpr int cols = paired(E) ? BN / 2 : BN;
  const int width = paired(E) ? a.n / 2 : a.n;
  const int ntiles = (width + cols - 1) / cols, mtiles = (a.m + BM - 1) / BM;
  const int64_t total = tile_count(a, BM, cols, width);
  const int64_t grid = (total + kXCDs - 1) / kXCDs * kXCDs;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * WM * WN), lds, s, a.x, a.w, a.m, a.n, a.k,
                     a.ksplit, ntiles, mtiles, positions, slots, out);
  return check_launch("gemm_tile");
}

template <int BM, int BN, int WM, int WN, int ST, Epilogue E>
int launch(const TileArgs& a, hipStream_t s) {
  return launch<BM, BN, WM, WN, ST, E>(a, nullptr, nullptr, a.out, s);
}

// The smallest tile of which every CU gets at most one, with a fourth stage where it fits (us with
// weights from HBM and the norm that consumes the output, against three stages): 64 x 64 (o_proj at
// 256 rows and 2 splits 11.3 / 12.3, at 512 rows unsplit 15.5), 128 x 64 (down at
// 160 rows and 4 splits 16.2 / 16.4, at 256 rows 17.7 / 18.1; 64 x 128 17.3 and 19.0), 128 x 128 (down
// at 512 rows and 4 splits 25.2, four stages 25.1), 128 x 192 (down at 640 rows
// and 4 splits 29.5). A second round of workgroups costs more than larger tiles.
template <Epilogue E>
int launch_plain(const TileArgs& a, hipStream_t s) {
  if (tile_count(a, 64, 64, a.n) <= kCUs) return launch<64, 64, 2, 2, 4, E>(a, s);
  if (tile_count(a, 128, 64, a.n) <= kCUs) return launch<128, 64, 4, 2, 4, E>(a, s);
  if (tile_count(a, 128, 128, a.n) <= kCUs) return launch<128, 128, 4, 2, 3, E>(a, s);
  return launch<128, 192, 4, 2, 3, E>(a, s);
}

// SwiGLU (no splits): the same rule over 128-row tiles of 48, 96 and 128 output columns (gate|up
// at 256 rows 22.6 us against 31.0 for hipBLASLt and pc_silu_mul, at 160 rows 20.8 (64 columns,
// eight waves: 23.1); at 512 rows 30.8 / 37.5, at 640 rows 37.4 / 40.9); where none fits one round,
// 96 columns with two stages, two workgroups per CU (1024 rows 50.9 / 58.0, 2048 rows 95.6 / 101.7).
int launch_swiglu(const TileArgs& a, hipStream_t s) {
  const int width = a.n / 2;
  if (tile_count(a, 128, 48, width) <= kCUs) return launch<128, 96, 4, 1, 3, kSwiGLU>(a, s);
  if (tile_count(a, 128, 96, width) <= kCUs) return launch<128, 192, 4, 2, 3, kSwiGLU>(a, s);
  if (tile_count(a, 128, 128, width) <= kCUs) return launch<128, 256, 2, 4, 3, kSwiGLU>(a, s);
  return launch<128, 192, 4, 2, 2, kSwiGLU>(a, s);
}

}  // namespace

namespace gemm_device {

// RoPE epilogue: the smallest tile of which every CU gets at most one, as above, with a stage
// more where it fits (us, against this file's partials or hipBLASLt and pc_rope_kv_append: 64 x 64
// at 384 rows 12.5 / 14.5, three stages 14.5; 128 x 64 at 512 rows 17.0 / 18.0, at 768 17.4 / 20.3;
// 128 x 128 at 1024 rows 25.1 / 26.5, at 1536 25.5 / 28.6). Larger than that it ties (33.6 / 33.2 at
// 2048 rows), and the decoder leaves it to hipBLASLt: 128 x 192 serves direct calls.
int launch_qkv_rows(const QkvArgs& q, hipStream_t s) {
  const TileArgs a{q.x, q.w, q.m, kQkvElems, q.k, q.k, nullptr};
  if (tile_count(a, 64, 64, a.n) <= kCUs) return launch<64, 64, 2, 2, 4, kRope>(a, q.positions, q.slots, q.out, s);
  if (tile_count(a, 128, 64, a.n) <= kCUs) return launch<128, 64, 4, 2, 4, kRope>(a, q.positions, q.slots, q.out, s);
  if (tile_count(a, 128, 128, a.n) <= kCUs) return launch<128, 128, 4, 2, 3, kRope>(a, q.positions, q.slots, q.out, s);
  return launch<128, 192, 4, 2, 3, kRope>(a, q.positions, q.slots, q.out, s);
}

// 64 x 96 tiles (48 output columns) for 81 to 128 rows, one workgroup per CU: gate|up moves 655 KB
// into each of 236 CUs, where gemm_m128_kernel moves 768 KB into each of 176 (128 rows 16.5 us /
// 17.7, 96 rows 15.5 / 16.4, 80 rows 15.9 / 15.7; five to seven stages 17.0 to 17.8). A short K does not
// repay the setup (at k 64 and 128 8 to 12 % slower, from 1024 level, from 2048 2 % faster and more).
bool swiglu_short_tiles(int m, int n, int k) {
  return m > 80 && m <= 128 && k >= 1024 && k <= kMaxK && 2 * ((n / 2 + 47) / 48) <= kCUs;
}

int launch_swiglu_short(void* out, const _Float16* x, const _Float16* w, int m, int n, int k, hipStream_t s) {
  return launch<64, 96, 4, 1, 4, kSwiGLU>(TileArgs{x, w, m, n, k, k, out}, s);
}

}  // namespace gemm_device

extern "C" int pc_gemm_rows(void* out, const void* x, const void* w, int32_t m, int32_t n, int32_t k, int32_t splits,
                            int32_t epilogue, void* stream) {
  if (!out || !x || !w) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (m < 1 || m > kMaxRows) return set_error(PC_ERR_ARGUMENT, "m = %d outside [1, %d]", m, kMaxRows);
  if (n < 1 || k < 1 || splits < 1) return set_error(PC_ERR_ARGUMENT, "n, k and splits must be positive");
  if (k % splits != 0) return set_error(PC_ERR_ARGUMENT, "k = %d not divisible into %d splits", k, splits);
  if (k / splits % 64 != 0) {
    return set_error(PC_ERR_ARGUMENT, "k per split (%d) must be a multiple of 64", k / splits);
  }
  if (k > kMaxK || static_cast<int64_t>(n) * k > (int64_t{1} << 31) || static_cast<int64_t>(m) * k > (int64_t{1} << 31) ||
      static_cast<int64_t>(splits) * m * n > (int64_t{1} << 31)) {
    return set_error(PC_ERR_ARGUMENT, "GEMM of %d x %d x %d with %d splits too large", m, n, k, splits);
  }
  if (!aligned(out, 16) || !aligned(x, 16) || !aligned(w, 16)) {
    return set_error(PC_ERR_ARGUMENT, "out, x and w must be 16-byte aligned");
  }
  const TileArgs a{static_cast<const _Float16*>(x), static_cast<const _Float16*>(w), m, n, k, k / splits, out};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (epilogue != kPartials && epilogue != kHalf && epilogue != kSwiGLU) {
    return set_error(PC_ERR_ARGUMENT, "unknown epilogue %d", epilogue);
  }
  if (epilogue != kPartials && splits != 1) return set_error(PC_ERR_ARGUMENT, "fp16 output needs one split");
  if (n % (epilogue == kSwiGLU ? 64 : 32) != 0) {
    return set_error(PC_ERR_ARGUMENT, "n = %d must be a multiple of %d", n, epilogue == kSwiGLU ? 64 : 32);
  }
  (void)hipGetLastError();
  if (splits == 1 && rows_stream(m, n, k)) return launch_rows_stream(out, a.x, a.w, m, n, k, static_cast<Epilogue>(epilogue), s);
  if (epilogue == kSwiGLU) return launch_swiglu(a, s);
  return epilogue == kHalf ? launch_plain<kHalf>(a, s) : launch_plain<kPartials>(a, s);
}
