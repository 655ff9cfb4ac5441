// Reading the attention workspace's fault word without a stream synchronization: a one-lane
// kernel behind the attention launch writes the word, with the caller's ticket, into pinned host
// memory that the host polls. What bounds a call of paged_attention is the time from its launch to
// the host knowing that it is done: the word is there about as soon as the attention is, where a
// copy waits for the runtime's completion signal (a call over 128 cached tokens 27.8 us with the
// copy, 20.6 polled; about 1.5 us of it is one look-up of the batch less).

#include <hip/hip_runtime.h>

#include <chrono>

#include <stdint.h>

#include "pagedcore_hip.h"
#include "pc_internal.h"

namespace {

using pc_internal::aligned;
using pc_internal::check_launch;
using pc_internal::set_error;

// {fault word, ticket} in one 8-byte store: the host sees both or neither.
__global__ void publish_faults_kernel(const int32_t* word, uint64_t* host, uint32_t ticket) {
  const uint32_t faults = static_cast<uint32_t>(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  __hip_atomic_store(host, static_cast<uint64_t>(ticket) << 32 | faults, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Longer waits are left to the runtime's own synchronization.
constexpr std::chrono::microseconds kPollTime{200};
constexpr int kPollsPerClock = 32;

}  // namespace

extern "C" int64_t pc_attn_read_faults(const void* workspace, void* host, uint32_t ticket, void* stream) {
  if (!workspace || !host) return -set_error(PC_ERR_ARGUMENT, "null pointer");
  if (!aligned(workspace, 256) || !aligned(host, 8)) {
    return -set_error(PC_ERR_ARGUMENT, "workspace must be 256-byte, the host word 8-byte aligned");
  }
  (void)hipGetLastError();
  hipLaunchKernelGGL(publish_faults_kernel, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream),
                     static_cast<const int32_t*>(workspace), static_cast<uint64_t*>(host), ticket);
  if (int rc = check_launch("publish_faults")) return -static_cast<int64_t>(rc);
  const auto end = std::chrono::steady_clock::now() + kPollTime;
  do {
    for (int i = 0; i < kPollsPerClock; ++i) {
      const uint64_t seen = __atomic_load_n(static_cast<const uint64_t*>(host), __ATOMIC_ACQUIRE);
      if (static_cast<uint32_t>(seen >> 32) == ticket) return static_cast<int64_t>(seen & 0xffffffffu);
      __builtin_ia32_pause();
    }
  } while (std::chrono::steady_clock::now() < end);
  return PC_ATTN_FAULTS_PENDING;
}
