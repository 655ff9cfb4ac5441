// Device helpers shared by the GEMM kernels (not part of the C ABI): operand types, LDS
// addressing, the explicit waits of the LDS DMA rings, and the SwiGLU epilogue.
#ifndef PAGEDCORE_GEMM_DEVICE_H
#define PAGEDCORE_GEMM_DEVICE_H

#include <hip/hip_runtime.h>

#include <atomic>

#include <math.h>
#include <stdint.h>

#include "pagedcore_hip.h"
#include "pc_internal.h"
#include "rope_device.h"

namespace gemm_device {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// kRope: the q|k|v projection rotated and written where pc_rope_kv_append writes it.
enum Epilogue : int32_t { kPartials = PC_GEMM_PARTIALS, kHalf = PC_GEMM_HALF, kSwiGLU = PC_GEMM_SWIGLU, kRope = 3 };
// The epilogues whose tiles hold pairs of W rows: gate and up, or a head's d and d + 32.
constexpr bool paired(Epilogue e) { return e == kSwiGLU || e == kRope; }
template <Epilogue E>
struct OutOf { typedef void* type; };
template <>
struct OutOf<kRope> { typedef rope_device::RopeOut type; };

__device__ __forceinline__ __attribute__((address_space(3))) void* lds_ptr(char* p) {
  return (__attribute__((address_space(3))) void*)(p);
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)p));
}
__device__ __forceinline__ half8_t lds_read(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) half8_t*>(static_cast<uintptr_t>(addr));
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
// Workgroup barrier without a memory fence (a fence would wait for every DMA in flight);
// the empty asm statements keep the compiler from moving LDS accesses across it.
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ _Float16 round_h(float x) { return static_cast<_Float16>(x); }

// fp16(fp16(silu(fp16 gate)) * fp16 up), silu(x) = x / (1 + exp(-x)) in fp32.
__device__ __forceinline__ _Float16 swiglu(float gate, float up) {
#pragma clang fp contract(off)
  const float x = static_cast<float>(round_h(gate));
  const float activated = static_cast<float>(round_h(x / (1.0f + expf(-x))));
  return round_h(activated * static_cast<float>(round_h(up)));
}

constexpr int kMaxDevices = 64;

// Raises a kernel's dynamic LDS limit once per device (on the current one), remembering
// the devices done in `done` (one bit each).
inline int raise_lds_limit(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) {
    return pc_internal::set_error(PC_ERR_LAUNCH, "cannot determine the current device");
  }
  const uint64_t bit = uint64_t{1} << device;
  if (done.load(std::memory_order_acquire) & bit) return PC_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
    return pc_internal::set_error(PC_ERR_LAUNCH, "cannot raise the GEMM's LDS limit to %d bytes", bytes);
  }
  done.fetch_or(bit, std::memory_order_acq_rel);
  return PC_OK;
}

// A q|k|v projection with the RoPE epilogue (x [m][k], w [2560][k]).
struct QkvArgs {
  const _Float16* x;
  const _Float16* w;
  int m, k;
  const int64_t* positions;
  const int64_t* slots;  // null: no pool
  rope_device::RopeOut out;
};
int launch_qkv_rows(const QkvArgs& a, hipStream_t s);  // the tiles of a prompt's rows
// SwiGLU at most of a decode step's rows on those tiles: where they are faster, and the launch
// (k a multiple of 64, n of 64).
bool swiglu_short_tiles(int m, int n, int k);
int launch_swiglu_short(void* out, const _Float16* x, const _Float16* w, int m, int n, int k, hipStream_t s);
// An unsplit product of a prompt's rows on the streams of a decode step: where, and the launch (k a
// multiple of 64, n of 32, for SwiGLU of 64).
bool rows_stream(int m, int n, int k);
int launch_rows_stream(void* out, const _Float16* x, const _Float16* w, int m, int n, int k, Epilogue epilogue, hipStream_t s);

}  // namespace gemm_device

#endif  // PAGEDCORE_GEMM_DEVICE_H
