// Entries of the tables of kept COUNT values, which every wave of a launch
// reads and writes without waiting for the others.
//
// An entry of a KEEP_POOL table serves many keys in turn, so a value is good
// only together with the key it was written for: both halves must come from
// one access. Plain loads and stores of the pair promise nothing of the kind
// (one whose halves are used in different branches is compiled to two 4-byte
// loads); an 8-byte atomic is one access by definition, and the word is private
// so that no other access can be written. The order of accesses does not matter (an
// entry tells by itself whom it serves, and a stale one is computed again), so
// they are relaxed and of workgroup scope, the widest that leaves the L1 cache
// in use.
#pragma once
#include <hip/hip_runtime.h>

namespace gatk {

class KeptEntry {
    unsigned long long word;  // tag | value << 32 | epoch << 56

  public:
    struct Read {
        unsigned tag, rest;
        __device__ __forceinline__ bool serves(unsigned key_tag, unsigned epoch) const {
            return tag == key_tag && rest >> 24 == epoch;
        }
        __device__ __forceinline__ int value() const { return (int)(rest & 0xffffffu); }
    };
    __device__ __forceinline__ Read read() const {
        const unsigned long long w = __hip_atomic_load(&word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return {(unsigned)w, (unsigned)(w >> 32)};
    }
    __device__ __forceinline__ void write(unsigned tag, int value, unsigned epoch) {
        __hip_atomic_store(&word, tag | (unsigned long long)((unsigned)value | epoch << 24) << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};
static_assert(sizeof(KeptEntry) == 8 && alignof(KeptEntry) == 8, "one aligned 8-byte access");

// The value of an edge table's entry, or -1. Its four bytes hold nothing else,
// so that they cannot disagree; the accesses are relaxed atomics because other
// waves write the same value at the same time.
class KeptEdge {
    int value;

  public:
    __device__ __forceinline__ int read() const {
        return __hip_atomic_load(&value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void write(int v) {
        __hip_atomic_store(&value, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};
static_assert(sizeof(KeptEdge) == 4 && alignof(KeptEdge) == 4, "one aligned 4-byte access");

}  // namespace gatk
