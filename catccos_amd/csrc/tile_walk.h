// Which slabs the persistent kernels ask memory for: whole numbers only, for the device and for a host that checks them.
#pragma once

#include <cstdint>

namespace cmx {

// K of an operand row in slabs: `real` ones in memory, `walked` by the kernel.  INT8 takes any number of at least two and fills an odd one up
// with a slab of zeros (loads of a buffer of no bytes); the other formats come in whole blocks of slabs.
struct KSlabs {
    uint32_t real, walked;
};
constexpr KSlabs k_slabs(uint32_t kbytes, uint32_t slab_bytes, bool fill_to_even) {
    const uint32_t real = kbytes / slab_bytes;
    return {real, fill_to_even ? (real + 1) & ~1u : real};
}
// tile loads past the end repeat the last slab
constexpr uint32_t load_slab(uint32_t slab, const KSlabs& k) { return slab < k.walked ? slab : k.walked - 1; }
// whether the tile loads of that slab find operands; if not, the buffer that they go through has no bytes
constexpr bool slab_in_memory(uint32_t slab, const KSlabs& k) { return slab < k.real; }
// Prefetches past the end repeat the last slab, too, but the last one in memory: they run ahead of the tile loads, through the buffer of those.
constexpr uint32_t prefetch_slab(uint32_t slab, const KSlabs& k) { return slab < k.real ? slab : k.real - 1; }

}  // namespace cmx
