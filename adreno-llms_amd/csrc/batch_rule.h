// Which calls of a batch may share a launch: calls that cannot observe one another's results, whatever order
// their blocks run in.  Host code without HIP.
#pragma once
#include <cstddef>
#include <cstdint>

namespace mi {

// True when [a, a+na) and [b, b+nb) share a byte.
inline bool overlaps(const void* a, size_t na, const void* b, size_t nb) {
    const auto pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa < pb + nb && pb < pa + na;
}

// The memory of one call out = x W^T: what it reads (scale: null, 0 bytes for fp16 weights) and what it writes.
struct CallMemory {
    const void *x, *W, *scale, *out;
    size_t x_bytes, w_bytes, scale_bytes, out_bytes;
};

// kind: a WeightKind (0 fp16, 4 block-32 Q4, 8 int8)
inline CallMemory call_memory(int kind, int M, int N, int K, const void* x, const void* W, const void* scale, const void* out) {
    const size_t m = static_cast<size_t>(M), n = static_cast<size_t>(N), k = static_cast<size_t>(K);
    CallMemory c{x, W, scale, out, m * k * 2, n * k * 2, 0, m * n * 2};
    if (kind == 8) { c.w_bytes = n * k; c.scale_bytes = n * 2; }
    if (kind == 4) { c.w_bytes = n * k / 2; c.scale_bytes = n * (k / 32) * 2; }
    return c;
}

// What `w` writes, `r` reads: x, the weights or their scales.
inline bool writes_what_reads(const CallMemory& w, const CallMemory& r) {
    return overlaps(w.out, w.out_bytes, r.x, r.x_bytes) || overlaps(w.out, w.out_bytes, r.W, r.w_bytes) ||
           overlaps(w.out, w.out_bytes, r.scale, r.scale_bytes);
}

// Neither call reads or writes what the other one writes.
inline bool independent(const CallMemory& a, const CallMemory& b) {
    return !writes_what_reads(a, b) && !writes_what_reads(b, a) && !overlaps(a.out, a.out_bytes, b.out, b.out_bytes);
}

}  // namespace mi
