// factor_source.hpp -- whether a tree build may read a caller's factor where it
// is.  A copy takes memory that a kernel cannot read: another GPU's without peer
// access, pageable host memory, a range that ends inside the factor (which the
// runtime refuses).  Plain host code, without the HIP headers.
#pragma once

#include <cstddef>
#include <cstdint>

namespace ftl {

// What the runtime reports of the memory at an address.
struct FactorMemory {
    bool device_memory;   // allocated on a GPU, not managed or host memory
    int owner;            // that GPU
    uint64_t base, size;  // the allocation
};

// `bytes` of FP64 entries at `address`, read by a kernel on GPU `device`.
inline bool factor_in_place(const FactorMemory& m, int device, uint64_t address, uint64_t bytes) {
    return m.device_memory && m.owner == device && address % sizeof(double) == 0 && address >= m.base &&
           address - m.base <= m.size && bytes <= m.size - (address - m.base);
}

}  // namespace ftl
