// Causal prompt attention over contiguous K/V (the prefill of one sequence).
//
// o[t][h] = softmax_{j <= t}(q[t][h] . k[j][h / 8] / 8) . v[j][h / 8] for a prompt of T tokens,
// with q [T][32][64], k and v [T][4][64] (the rotated keys and the values that
// pc_rope_kv_append wrote), o [T][32][64], all fp16.
//
// Work split: one workgroup per (16-query block, four query heads), one wave per head; two
// workgroups share a kv head. The workgroup stages 64 keys of K and V at a time in LDS (LDS
// DMA, two stages, one barrier per step) and every wave reads them. With KG = 2 a second set of
// four waves takes every other step, and the two sets' results meet in LDS at the end. A wave
// walks key blocks 0 .. its query block with an online softmax in fp32:
//   S^T = K_blk . Q^T   on v_mfma_f32_16x16x32_f16 (lane (c, g): keys 4g..4g+3 of position c)
//   O^T += V^T . P^T    on v_mfma_f32_16x16x32_f16 over pairs of blocks, V^T from the decode
//                       kernel's transposing LDS reads, P^T straight from the S^T registers
//   l   += 1 . P^T      one more MFMA with an all-ones A operand: the softmax denominator of
//                       every position, summed on the matrix core
// so every per-position quantity (running max, sum, rescale) stays in the lane that owns
// the position. Only the diagonal block needs the causal mask. Probabilities enter the PV
// product as fp16 (relative error 2^-11) and the denominator sums those same fp16 weights;
// everything else is fp32 with one final fp16 rounding.
//
// What bounds it: a step of 64 keys is a chain (barrier, K from LDS, MFMA, max, exp, MFMA) of
// about 1400 cycles for a wave alone on its SIMD, 440 of them VALU issue and 290 matrix work.
// Short prompts run that chain with the chip half empty, so they get the two key sets (half
// the chain) and small workgroups; long ones need every SIMD kept full to the end, so heavy and
// light query blocks are paired on a CU (kSnake). All K fragments of a step, and all V fragments,
// are read in one block each: two exposed LDS latencies per step instead of six. Measured, us
// per layer, against eight waves per workgroup without these (same outputs bit for bit for
// KG = 1): 64 tokens 3.8 -> 3.1, 333 7.3 -> 5.7, 512 9.0 -> 6.9, 1024 14.8 -> 10.6, 2048 31.1 ->
// 26.5. Slower: three stages (28.7 at 2048, 6.7 at 333), 32 queries per wave (34.2), packed
// fp16 conversion (29.8 against 28.6).
//
// Prompts beyond that keep every SIMD busy whatever the order, and the time is that of the work on a
// CU: there a workgroup has all eight heads of a kv head (half the staging) and reads K and V two key
// blocks at a time, which takes 78 registers instead of 96 (24 waves on a CU, not 16 to 20).

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "pagedcore_hip.h"
#include "pc_device.h"
#include "pc_internal.h"

namespace {

using namespace pc_device;
using pc_internal::aligned;
using pc_internal::check_launch;
using pc_internal::ok;
using pc_internal::set_error;

constexpr int kKVHeads = 4;
constexpr int kQHeads = 32;
constexpr int kHeadDim = 64;
constexpr int kHeadsPerKV = kQHeads / kKVHeads;
constexpr int kSnake = 256;                  // one workgroup per CU
constexpr int kBlock = 16;                   // positions per query block and keys per key block
constexpr int kTileBytes = kBlock * kHeadDim * 2;  // 16 rows of one kv head: 2 KiB
constexpr int kBufBytes = 2 * kTileBytes;           // one key block: K tile, then V tile
constexpr int kStepBlocks = 4;                      // key blocks per step
constexpr int kStageBytes = kStepBlocks * kBufBytes;
constexpr int kMaxTokens = 1 << 16;
constexpr float kFloatMax = 3.402823466e38f;
constexpr float kLazyLog2 = 8.0f;            // headroom (log2 of p) before the running max is raised

// f(integral_constant<int, p>) for every pair p of key blocks of a step, in order.
template <typename F, int... P>
__device__ __forceinline__ void for_pairs_impl(F&& f, std::integer_sequence<int, P...>) {
  (f(std::integral_constant<int, P>{}), ...);
}
template <typename F>
__device__ __forceinline__ void for_pairs(F&& f) {
  for_pairs_impl(f, std::make_integer_sequence<int, kStepBlocks / 2>{});
}

// Two 16-key tiles as one 32-key MFMA operand (first tile's keys first).
__device__ __forceinline__ half8_t join(short4_t x, short4_t y) {
  const half4_t a = __builtin_bit_cast(half4_t, x), b = __builtin_bit_cast(half4_t, y);
  return half8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

struct PrefillArgs {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  int tokens;
  _Float16* out;
};

// KG key sets of HEADS waves (query heads of one kv head) each. Scalar parameters in the order of
// PrefillArgs: all are preloaded into SGPRs at wave launch.
template <int KG, int HEADS>
__global__ __launch_bounds__(64 * HEADS * KG) void prefill_attention_kernel(const _Float16* q, const _Float16* k,
                                                                             const _Float16* v, int tokens,
                                                                             _Float16* out) {
  constexpr int kPerKV = kHeadsPerKV / HEADS;   // workgroups per kv head and query block
  constexpr int kPerBlock = kKVHeads * kPerKV;  // workgroups per query block
  constexpr int kStagers = HEADS / 4;           // waves that stage the same rows of different key blocks
  constexpr bool kPairReads = HEADS == 8;       // LDS reads of two key blocks at a time (see the top)
  const PrefillArgs a{q, k, v, tokens, out};
  // Per key set two stages of kStepBlocks key blocks each: stage s, block b: K tile at
  // s * kStageBytes + b * kBufBytes, its V tile kTileBytes after it.
  __shared__ __attribute__((aligned(16))) char smem[KG * 2 * kStageBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wave % HEADS, kg = wave / HEADS;
  char* const lds = smem + kg * 2 * kStageBytes;
  const int lane = threadIdx.x & 63;
  const int c = lane & 15;
  const int g = lane >> 4;
  const int qblocks = (a.tokens + kBlock - 1) / kBlock;
  // Latest (longest) query blocks first, in chunks of one workgroup per CU whose order turns
  // round from chunk to chunk: the hardware deals a chunk to the CUs in turn, so a CU that got
  // one of the longest of one chunk gets one of the shortest of the next (2048 tokens: a CU's
  // blocks sum to 127 instead of 64 to 190; 31.1 -> 28.6 us).
  int id = blockIdx.x;
  const int chunk = id / kSnake, base = chunk * kSnake;
  if (chunk & 1) {
    const int in = id - base, blocks = min(kSnake, static_cast<int>(gridDim.x) - base) / kPerBlock;
    id = base + (blocks - 1 - in / kPerBlock) * kPerBlock + in % kPerBlock;
  }
  const int h = id % kPerBlock / kPerKV;
  const int qb = qblocks - 1 - id / kPerBlock;
  const int head = kHeadsPerKV * h + HEADS * (id % kPerKV) + w;
  const int pos = kBlock * qb + c;  // this lane's query position (column of S^T)
  const int last = a.tokens - 1;

  const _Float16* qrow = a.q + (static_cast<int64_t>(min(pos, last)) * kQHeads + head) * kHeadDim + 8 * g;
  half8_t qa = *reinterpret_cast<const half8_t*>(qrow);
  half8_t qc = *reinterpret_cast<const half8_t*>(qrow + 32);

  // Staging: wave w of a key set issues kStepBlocks / kStagers LDS DMA instructions per stage (each 64
  // lanes x 16 B = rows srow .. srow + 7 of one tile): of blocks w / 4, w / 4 + kStagers, ..., the K
  // (w & 2 = 0) or V tile, rows 8 (w & 1) .. 8 (w & 1) + 7. K piece p of row r sits at position p ^ (r & 7) (the
  // A-operand reads of 16 rows then hit 8 different 16 B bank groups); V uses the decode
  // kernel's 32 B-group swizzle for its transposing reads.
  const bool stage_v = (w & 2) != 0;
  const int qs = lane & 7;
  const int srow = 8 * (w & 1) + (lane >> 3);
  const int piece = stage_v ? 2 * ((qs >> 1) ^ row_sel(srow)) + (qs & 1) : qs ^ (srow & 7);
  const _Float16* ssrc = (stage_v ? a.v : a.k) + h * kHeadDim + 8 * piece;
  const int sdst = (stage_v ? kTileBytes : 0) + 1024 * (w & 1);
  const uint32_t lds0 = lds_offset(lds);
  // K reads: lane (c, g) takes row c, pieces g and 4 + g
  const uint32_t kaddr0 = lds0 + c * 128 + 16 * (g ^ (c & 7));
  const uint32_t kaddr1 = lds0 + c * 128 + 16 * ((4 + g) ^ (c & 7));
  // V transposing reads: lane (c, g) supplies row 4g + c/4, 8 B piece c % 4
  const int rr = 4 * g + (c >> 2);
  const uint32_t vbase = lds0 + kTileBytes + rr * 128 + 8 * (c & 3);
  const uint32_t tsel = row_sel(rr);
  const uint32_t va[4] = {vbase + 32 * (0 ^ tsel), vbase + 32 * (1 ^ tsel), vbase + 32 * (2 ^ tsel), vbase + 32 * (3 ^ tsel)};

  // Key blocks kStepBlocks * j .. + kStepBlocks - 1 into stage `buf` (rows past the prompt
  // repeat its last row; their scores are masked).
  auto stage = [&](int j, int buf) {
#pragma unroll
    for (int i = 0; i < kStepBlocks / kStagers; ++i) {
      const int b = w / 4 + kStagers * i;
      const int row = min(kBlock * (kStepBlocks * j + b) + srow, last);
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(ssrc + static_cast<int64_t>(row) * kKVHeads * kHeadDim),
                                       lds_ptr(lds + buf * kStageBytes + sdst + b * kBufBytes), 16, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  const half8_t ones = {1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16};
  float m = 0.f, mc = 0.f;
  float4_t acc[4], lacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 4; ++u) acc[u] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int steps = (qb + kStepBlocks) / kStepBlocks;  // causal: key blocks 0 .. qb

  const int rounds = (steps + KG - 1) / KG;

  // Round J: each key set's step j = KG J + kg, staged in stage B (a compile-time constant, so
  // every LDS address below is a fixed base plus an immediate offset).
  auto step = [&](int J, auto stage_index) {
    constexpr int B = decltype(stage_index)::value;
    constexpr uint32_t so = B * kStageBytes;
    const int j = KG * J + kg;
    // This wave's staging of step j (and, before the first step, Q) has landed; after the
    // barrier every wave's has, and every wave has finished reading the other stage (its
    // reads of the round before waited for lgkmcnt(0)), which the next staging refills. Q is
    // named so that the compiler does not add a wait of its own for it, which would also wait
    // for the staging issued below.
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(qa), "+v"(qc) : : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (j + KG < steps) stage(j + KG, B ^ 1);
    if (KG > 1 && j >= steps) return;  // the last round of a set with no step left in it
    // sc[4 b + e]: key 4g + e of block kStepBlocks * j + b
    float sc[4 * kStepBlocks];
    if constexpr (kPairReads) {
      for_pairs([&](auto pair) {
        constexpr int b = 2 * decltype(pair)::value;
        half8_t k00, k01, k10, k11;
        asm volatile(
            "ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\tds_read_b128 %2, %4 offset:%7\n\t"
            "ds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(k00), "=&v"(k01), "=&v"(k10), "=&v"(k11)
            : "v"(kaddr0), "v"(kaddr1), "i"(so + b * kBufBytes), "i"(so + (b + 1) * kBufBytes)
            : "memory");
        float4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k00, qa, s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k10, qa, s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k01, qc, s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(k11, qc, s1, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[4 * b + e] = s0[e];
          sc[4 * b + 4 + e] = s1[e];
        }
      });
    } else     {
      half8_t kf[8];
      asm volatile(
          "ds_read_b128 %0, %8 offset:%10\n\tds_read_b128 %1, %9 offset:%10\n\t"
          "ds_read_b128 %2, %8 offset:%11\n\tds_read_b128 %3, %9 offset:%11\n\t"
          "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\t"
          "ds_read_b128 %6, %8 offset:%13\n\tds_read_b128 %7, %9 offset:%13\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(kf[0]), "=&v"(kf[1]), "=&v"(kf[2]), "=&v"(kf[3]), "=&v"(kf[4]), "=&v"(kf[5]), "=&v"(kf[6]),
            "=&v"(kf[7])
          : "v"(kaddr0), "v"(kaddr1), "i"(so), "i"(so + kBufBytes), "i"(so + 2 * kBufBytes), "i"(so + 3 * kBufBytes)
          : "memory");
      float4_t s[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        s[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[2 * b], qa, float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[2 * b + 1], qc, s[b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[4 * b + e] = s[b][e];
    }
    if (kStepBlocks * j + kStepBlocks - 1 >= qb) {  // the diagonal step: keys after the position, or past the prompt, are masked
#pragma unroll
      for (int e = 0; e < 4 * kStepBlocks; ++e) {
        const int key = kBlock * (kStepBlocks * j + (e >> 2)) + 4 * g + (e & 3);
        sc[e] = (key <= pos && key <= last) ? sc[e] : -INFINITY;
      }
    }
    float bm = sc[0];
#pragma unroll
    for (int e = 1; e < 4 * kStepBlocks; ++e) bm = fmaxf(bm, sc[e]);
    if (J == 0) {
      // A step's first key is visible to every position; the bound keeps the max finite where
      // infinite inputs make all 64 scores -inf (their weights are then 0, not NaN).
      m = fmaxf(max_over_groups(bm), -kFloatMax);
      mc = m * kScoreToLog2;
    } else if (__builtin_amdgcn_ballot_w64(bm * kScoreToLog2 > mc + kLazyLog2) != 0) {
      const float mn = fmaxf(m, max_over_groups(bm));
      const float alpha = exp2_fast((m - mn) * kScoreToLog2);
      lacc *= alpha;
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] *= alpha;
      m = mn;
      mc = m * kScoreToLog2;
    }
    __builtin_amdgcn_sched_barrier(0);
    // Per pair of blocks, P^T as one 32-key B operand: element e is key 4g + (e & 3) of
    // the pair's block e / 4; the V^T A operands concatenate the two blocks in the same
    // order.
    auto weights = [&](int b) {
      half8_t pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[e] = static_cast<_Float16>(exp2_fast(fmaf(sc[4 * b + e], kScoreToLog2, -mc)));
      return pb;
    };
    auto accumulate = [&](const half8_t pb, const short4_t* v0, const short4_t* v1) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(join(v0[u], v1[u]), pb, acc[u], 0, 0, 0);
      lacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pb, lacc, 0, 0, 0);
    };
    if constexpr (kPairReads) {
      for_pairs([&](auto pair) {
        constexpr int b = 2 * decltype(pair)::value;
        const half8_t pb = weights(b);
        short4_t v0[4], v1[4];
        read_v_tiles<so + b * kBufBytes>(vbase, tsel, v0[0], v0[1], v0[2], v0[3]);
        read_v_tiles<so + (b + 1) * kBufBytes>(vbase, tsel, v1[0], v1[1], v1[2], v1[3]);
        accumulate(pb, v0, v1);
      });
    } else {
      short4_t vt[16];  // vt[4 b + u]: block b, dims 16 u .. 16 u + 15
      asm volatile(
          "ds_read_b64_tr_b16 %0, %16 offset:%20\n\tds_read_b64_tr_b16 %1, %17 offset:%20\n\t"
          "ds_read_b64_tr_b16 %2, %18 offset:%20\n\tds_read_b64_tr_b16 %3, %19 offset:%20\n\t"
          "ds_read_b64_tr_b16 %4, %16 offset:%21\n\tds_read_b64_tr_b16 %5, %17 offset:%21\n\t"
          "ds_read_b64_tr_b16 %6, %18 offset:%21\n\tds_read_b64_tr_b16 %7, %19 offset:%21\n\t"
          "ds_read_b64_tr_b16 %8, %16 offset:%22\n\tds_read_b64_tr_b16 %9, %17 offset:%22\n\t"
          "ds_read_b64_tr_b16 %10, %18 offset:%22\n\tds_read_b64_tr_b16 %11, %19 offset:%22\n\t"
          "ds_read_b64_tr_b16 %12, %16 offset:%23\n\tds_read_b64_tr_b16 %13, %17 offset:%23\n\t"
          "ds_read_b64_tr_b16 %14, %18 offset:%23\n\tds_read_b64_tr_b16 %15, %19 offset:%23\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(vt[0]), "=&v"(vt[1]), "=&v"(vt[2]), "=&v"(vt[3]), "=&v"(vt[4]), "=&v"(vt[5]), "=&v"(vt[6]),
            "=&v"(vt[7]), "=&v"(vt[8]), "=&v"(vt[9]), "=&v"(vt[10]), "=&v"(vt[11]), "=&v"(vt[12]), "=&v"(vt[13]),
            "=&v"(vt[14]), "=&v"(vt[15])
          : "v"(va[0]), "v"(va[1]), "v"(va[2]), "v"(va[3]), "i"(so), "i"(so + kBufBytes), "i"(so + 2 * kBufBytes),
            "i"(so + 3 * kBufBytes)
          : "memory");
      for_pairs([&](auto pair) {
        constexpr int b = 2 * decltype(pair)::value;
        accumulate(weights(b), vt + 4 * b, vt + 4 * b + 4);
      });
    }
  };

  if (kg < steps) stage(kg, 0);
  for (int J = 0; J < rounds; J += 2) {
    step(J, std::integral_constant<int, 0>{});
    if (J + 1 < rounds) step(J + 1, std::integral_constant<int, 1>{});
  }

  if constexpr (KG == 2) {
    // The second set leaves its accumulators, max and sum in LDS (over the stages, once every
    // wave is done with them); the first folds them into its own. A set that had no step
    // contributes with weight 0.
    constexpr int kValues = 18;
    __syncthreads();
    float* other = reinterpret_cast<float*>(smem) + 64 * kValues * w + lane;
    if (kg == 1) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) other[64 * (4 * u + e)] = acc[u][e];
      other[64 * 16] = kg < steps ? m : -INFINITY;
      other[64 * 17] = lacc[0];
    }
    __syncthreads();
    if (kg == 1) return;
    const float mo = other[64 * 16], mn = fmaxf(m, mo);
    const float a0 = exp2_fast((m - mn) * kScoreToLog2), a1 = exp2_fast((mo - mn) * kScoreToLog2);
    lacc[0] = fmaf(other[64 * 17], a1, lacc[0] * a0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[u][e] = fmaf(other[64 * (4 * u + e)], a1, acc[u][e] * a0);
  }

  // lane (c, g) of tile u holds O^T[dims 16u + 4g .. + 3][position c]; every row of lacc
  // holds the denominator of position c
  const float inv = 1.0f / lacc[0];
  if (pos <= last) {
    _Float16* dst = a.out + (static_cast<int64_t>(pos) * kQHeads + head) * kHeadDim + 4 * g;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      half4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = static_cast<_Float16>(acc[u][e] * inv);
      *reinterpret_cast<half4_t*>(dst + 16 * u) = o;
    }
  }
}

}  // namespace

extern "C" int pc_prefill_attention(void* out, const void* query, const void* key, const void* value, int32_t tokens,
                                    void* stream) {
  if (tokens < 0 || tokens > kMaxTokens) return set_error(PC_ERR_ARGUMENT, "tokens %d outside [0, %d]", tokens, kMaxTokens);
  if (tokens == 0) return ok();
  if (!out || !query || !key || !value) return set_error(PC_ERR_ARGUMENT, "null pointer");
  if (!aligned(out, 16) || !aligned(query, 16) || !aligned(key, 16) || !aligned(value, 16))
    return set_error(PC_ERR_ARGUMENT, "buffers must be 16-byte aligned");
  // Two key sets while their workgroups (64 KiB of LDS, two per CU) run at once, above the 128
  // tokens (two steps) where the merge costs more than the shorter chain saves: 3.8 against
  // 4.1 us at 128 tokens, 5.1 / 5.1 at 256, 6.1 / 5.7 at 333, 12.3 / 10.6 at 1024, 26.5 / 29.6
  // at 2048. Eight heads per workgroup from the sixth round of half-size ones on, where what counts is
  // the waves on a CU and the bytes staged, no longer how evenly the CUs end (us against four heads):
  // 33.4 / 31.4 at 2300 tokens, 40.2 / 41.1 at 2600, 49.6 / 52.6 at 3000, 89.7 / 93.3 at 4096, 323 / 352 at 8192.
  const unsigned blocks = static_cast<unsigned>((tokens + kBlock - 1) / kBlock);
  auto launch = [&](auto kernel, unsigned per_block, int waves) {
    hipLaunchKernelGGL(kernel, dim3(blocks * per_block), dim3(64 * waves), 0, static_cast<hipStream_t>(stream),
                       static_cast<const _Float16*>(query), static_cast<const _Float16*>(key),
                       static_cast<const _Float16*>(value), static_cast<int>(tokens), static_cast<_Float16*>(out));
  };
  if (8 * blocks > 5 * kSnake) launch(prefill_attention_kernel<1, 8>, 4, 8);
  else if (tokens > 128 && 8 * blocks <= 2 * kSnake) launch(prefill_attention_kernel<2, 4>, 8, 8);
  else launch(prefill_attention_kernel<1, 4>, 8, 4);
  return check_launch("prefill_attention");
}
