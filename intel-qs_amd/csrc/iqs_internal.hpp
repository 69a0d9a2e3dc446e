// Library-internal helpers shared by the C-ABI translation units of libiqs_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

#include "../../include/iqs_hip.h"

// A register: 2^n interleaved complex amplitudes in device memory.
struct iqsh_state {
  unsigned n = 0;
  int dtype = IQSH_C128;
  void* d = nullptr;        // amplitudes
  bool owned = true;
  void* spare = nullptr;    // second buffer for out-of-place permutation
  std::atomic<uint64_t> touched{0};  // iqsi::cached_pass
  std::atomic<bool> cold{false};
  uint64_t size() const { return uint64_t(1) << n; }
  size_t esz() const { return dtype == IQSH_C128 ? 16 : 8; }
};

namespace iqsk {
struct CutSpec;
}

namespace iqsi {

// Record a failure for iqsh_last_error() and return `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// The library stream (iqsh_set_stream).
hipStream_t stream();
// Whether the library stream is being captured into a graph.
bool capturing();
// The kernel of dense blocks of three and more positions (iqsh_set_block_mfma).
int block_kernel();
// Compute units of the current device.
int device_cus();
// Results that workgroups of a reduction kernel write one by one into pinned host memory: the
// host marks the slots before the launch and polls them, for up to 100 us before it waits for
// the stream.  (A kernel, a copy of its result and a stream synchronization take 15.1 us, a
// kernel that writes to the host and the synchronization 11.5, with the polling 6.6; 2048
// workgroups writing to the host take 1.4 us more than writing to the device.)  Only for kernels
// that write nothing else: their other stores could still be on the way.  The mark is a signaling
// NaN, which no arithmetic returns.
constexpr uint64_t kPending = 0x7ff4dead0000beefull;
inline void mark_pending(double* p, uint64_t count)
{
  for (uint64_t i = 0; i < count; ++i) __atomic_store_n(reinterpret_cast<uint64_t*>(p) + i, kPending, __ATOMIC_RELAXED);
}
int await_results(const double* p, uint64_t count);
// Whether amplitudes of `bytes` in all, gone over again by call after call, stay in the 256 MiB
// last-level cache if the kernels use ordinary accesses (non-temporal ones stream past it).
// Measured with one kernel after another on the same register: dense 1q complex128 21
// qubits (32 MiB) 11.0 -> 7.5 us, 22 qubits 22 -> 19.5, 24 qubits (256 MiB) 85 -> 72.5; QAOA
// layer 24 qubits 298 -> 241.  Above 256 MiB non-temporal accesses stream faster (25 qubits 167
// against 177 us, layer at 26 qubits 1188 against 1236); below 32 MiB stores that stay in the
// L2s cost more when the kernel ends and writes them back (20 qubits 4.6 against 5.3 us, layer 21
// against 30).
constexpr uint64_t kCacheBytes = uint64_t(256) << 20;
inline bool cache_set(uint64_t bytes) { return bytes >= (uint64_t(32) << 20) && bytes <= kCacheBytes; }
// The same for a pass over `bytes` of h that starts now: not if h is used in turn with other
// registers, that is if before this pass and before the last one over h, passes over others have
// put more through the cache than it holds beside h (gates on 4 registers of 23 complex128 qubits in
// turn: 52 us with ordinary accesses, 47 with non-temporal ones).  A first pass after others
// brings h back into the cache for those that follow it.
bool cached_pass(iqsh_handle h, uint64_t bytes);
// Edge-parity tables and phase table of a MaxCut cost for register h (at most 64 edges):
// the phase exp(-i gamma cut) per amplitude.
int build_cut_spec(iqsh_handle h, unsigned ne, const unsigned* u, const unsigned* v, const double* w, double gamma,
                   iqsk::CutSpec* cs);
// lam := C psi with cost_blocks(psi) partial sums of cut |psi|^2 (iqsh_qaoa_cost_apply without
// the sum).
unsigned cost_blocks(iqsh_handle psi);
int launch_cost(iqsh_handle psi, iqsh_handle lam, const iqsk::CutSpec& cs, double* partial);

}  // namespace iqsi

#define IQSI_TRY(expr)                                                                        \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess) return iqsi::fail(IQSH_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)
