// How results that a kernel does not read again go to memory.
//
// Through: straight through the L2 (which keeps the line) to the memory-side cache.  A plain
// store leaves its line dirty in the L2, and a kernel's end waits for all of those to be written
// back; going through, that happens while the kernel runs.  N32 C128 28x28 R16 (12.8 MB written)
// 10.6 -> 9.3 us, N12 C256 56x56 R32 (38 MB) 23.4 -> 21.1, one call after the other; where the
// next call reads what this one wrote 22.4 -> 20.2.
// Streamed: past the memory-side cache (256 MB) as well, for results too large to be still there
// when somebody reads them: N32 C256 56x56 R32 (103 MB read, 103 written) on rotating buffers 57 us
// plain, 60 through, 51.6 streamed, each call reading what the one before wrote 59, 61 and 51; but N24
// (77 and 77 MB) in the same order 48, 47 and 40 on rotating buffers, 31, 29 and 41 reading what was
// written.
// Behind a layer's activation results from 96 to 128 MB are stored plainly: N32 C256 56x56 R32's training
// step 217 us with a streamed y, 215 with one that goes through, 211.
// A result that the next launch reads again is streamed from 128 MB on if that is another pass of the
// layer (R128, us, through / streamed: N32 C256 56x56 155 / 171, N44 237 / 231, N52 293 / 285; R96 N36 145 /
// 182, N48 263 / 249), never if it is the bias / activation kernel (R64: N32 100 / 116, N44 149 / 156, N50
// 156 / 170).
// Plain where planes start inside a cache line and the result is not small: parts of lines then
// go to memory one by one (N8 C64 130x130, 35 MB, rotating buffers: 28 us, through 35; N8 C64 66x70,
// 9 MB, 11.1 and 10.3).
#ifndef CP4_STORE_POLICY_H
#define CP4_STORE_POLICY_H

#include <cstdint>

#include <hip/hip_runtime.h>

namespace cp4 {

enum StorePolicy { kStorePlain, kStoreThrough, kStoreStreamed };

// Bytes of a result from which it is streamed: one that a training step reads soon after (behind a
// layer's activation), and others; and up to which it goes through although its planes start
// inside cache lines.
constexpr size_t kStreamBytesLayer = (size_t)128 << 20, kStreamBytes = (size_t)96 << 20;
constexpr size_t kThroughOffLine = (size_t)16 << 20;
// ... where another pass of the layer follows; and bytes up to which a result goes through.
constexpr size_t kStreamBytesPass = (size_t)128 << 20, kNeverStreamed = ~(size_t)0;
constexpr size_t kThroughBytes = kStreamBytes;

// For planes of `plane` bytes, `bytes` in all.
inline int store_policy(const void* dst, size_t plane, size_t bytes, size_t stream_from,
                        size_t through_to = kThroughBytes) {
  const bool lines = plane % 128 == 0 && (reinterpret_cast<uintptr_t>(dst) & 127) == 0;
  if (!lines) return bytes <= kThroughOffLine ? kStoreThrough : kStorePlain;
  return bytes >= stream_from ? kStoreStreamed : bytes <= through_to ? kStoreThrough : kStorePlain;
}

template <class T>
__device__ __forceinline__ void store_through(T* p, T v) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "a dword or two");
  if constexpr (sizeof(T) == 4)
    __hip_atomic_store(reinterpret_cast<unsigned*>(p), __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  else
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p),
                       __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void store_streamed(T* p, T v) {
  if constexpr (sizeof(T) == 4)
    __builtin_nontemporal_store(__builtin_bit_cast(unsigned, v), reinterpret_cast<unsigned*>(p));
  else
    __builtin_nontemporal_store(__builtin_bit_cast(unsigned long long, v),
                                reinterpret_cast<unsigned long long*>(p));
}

template <int STORE, class T>
__device__ __forceinline__ void store_as(T* p, T v) {
  if constexpr (STORE == kStoreThrough) store_through(p, v);
  else if constexpr (STORE == kStoreStreamed) store_streamed(p, v);
  else *p = v;
}

// The last argument of the raw buffer stores.
constexpr int buffer_policy(int store) { return store == kStoreThrough ? 16 : store == kStoreStreamed ? 2 : 0; }

}  // namespace cp4
#endif
