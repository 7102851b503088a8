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
// written.  The same line behind a layer's activation, where a training step's backward reads y next
// (forward with bias and ReLU alone and the whole step on rotating buffers, us, plain / streamed: N32 C256
// 56x56 R32 59 / 50 and 211 / 213, N36 59 / 54 and 235 / 232, N40 74 / 67 and 266 / 259, N16 C128 112x112
// R16 53 / 44 and 203 / 204, N18 54 / 49 and 225 / 219).
// A result that the next launch reads again is streamed from 128 MB on if that is another pass of the
// layer (R128, us, through / streamed: N32 C256 56x56 155 / 171, N44 237 / 231, N52 293 / 285; R96 N36 145 /
// 182, N48 263 / 249), never if it is the bias / activation kernel (R64: N32 100 / 116, N44 149 / 156, N50
// 156 / 170).
// Plain where planes start inside a cache line and the result is not small: parts of lines then
// go to memory one by one (N8 C64 130x130, 35 MB, rotating buffers: 28 us, through 35; N8 C64 66x70,
// 9 MB, 11.1 and 10.3).  The strip kernels' fp32 results: also where strips start inside a line and the
// result is not found in the memory-side cache any more (rotating buffers, plain / through: N12 C256 56x56
// R32, three rows, 37 MB, 31.1 / 29.5 us; N20, five rows, 61 MB, 42.4 / 48.3), and from 76 MB on (N18,
// 55 MB, 38.6 / 36.3; N22 45.1 / 43.8; N24, 74 MB, 49.1 / 47.4; N26, 80 MB, 53.7 / 56.6; N28 55.1 / 57.9; N30
// 56.5 / 59.0).
#ifndef CP4_STORE_POLICY_H
#define CP4_STORE_POLICY_H

#include <cstdint>

#include <hip/hip_runtime.h>

namespace cp4 {

enum StorePolicy { kStorePlain, kStoreThrough, kStoreStreamed };

// Bytes of a result from which it is streamed: in general; where another pass follows; with few
// channels (fwd_few.hip) behind a layer's activation, where little else goes through the cache before the
// backward reads y (training step of N9 C3 K64 224x224 R16, 110 MB: through 87.6 us, streamed 94.2, plain 93.3).
constexpr size_t kStreamBytes = (size_t)96 << 20, kStreamBytesPass = (size_t)128 << 20,
                 kStreamBytesFewLayer = (size_t)128 << 20;
constexpr size_t kNeverStreamed = ~(size_t)0;
// Bytes up to which a result goes through: although its planes start inside cache lines; of the strip
// kernels, although strips do; of the strip kernels at all; of any other.
constexpr size_t kThroughOffLine = (size_t)16 << 20, kThroughOffStrip = (size_t)48 << 20,
                 kThroughStrips = (size_t)76 << 20, kThroughBytes = kStreamBytes;

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
