// Which tiles the persistent kernels walk and which slabs they ask memory for: whole numbers only, for the device and for a host that checks
// them.
#pragma once

#include <cstdint>

namespace cmx {

constexpr int kXcds = 8;

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

// Persistent kernels that walk in fixed strides (no tile counter), with at least one full round of tiles: instead of
// owning a contiguous run, the XCDs take turns at blocks of (workgroups per XCD) consecutive tiles, workgroup j of XCD x
// walking tiles x * per + j, + grid, + 2 * grid, ...  The whole chip then works on one stretch of `grid` consecutive
// tiles at a time -- two bands of m-tiles across all their weight tiles -- so an activation panel is wanted by four XCDs
// and a weight panel by two at about the same time (the memory-side cache can serve the repeats), and every block of 32
// tiles starts on a multiple of 32, where the contiguous runs cut across the bands.  Zipf-routed 16-expert problem: 16 %
// fewer L2 misses, 1.7-3.3 % less time.  Problems of less than a round keep the contiguous runs, which spread few tiles
// over all eight L2s.
constexpr void interleave_xcd_walk(uint32_t total_tiles, uint32_t wg, uint32_t grid, uint32_t& tile_id, uint32_t& stride, uint32_t& end) {
    if (total_tiles < grid) return;
    tile_id = (wg % kXcds) * (grid / kXcds) + wg / kXcds;
    stride = grid;
    end = total_tiles;
}
// The tile after tile_id of such a walk, or `end`.  In the last, partly filled round the XCDs take fewer tiles each, in whole bands of 8: in
// blocks of 32 they would all lie on the first XCDs, and the L2s and links of the others would have nothing to do.  320 tiles on 256
// workgroups (us): SwiGLU 8 x 1280 rows, K = 4096, N = 2048 124.5 -> 112.6, FP4 125.7 -> 117.2, dense 8192 x 5120 x 7168 (640 tiles) 281 -> 264; 384
// tiles 128 -> 117.  In contiguous runs of any length, which cut across the bands, 65536 rows on 32 groups (17 rounds) lose 1.6 %.
constexpr uint32_t kSpreadRounds = 6;              // (five rounds 337 -> 333; at eight the workgroups have drifted apart and the order makes no difference)
constexpr uint32_t next_of_walk(uint32_t tile_id, uint32_t stride, uint32_t end, uint32_t wg, uint32_t grid) {
    const uint32_t next = tile_id + stride;
    if (stride != grid || end >= kSpreadRounds * stride || next < end / stride * stride) return next;
    const uint32_t full = end / stride * stride, bands = ((end - full + kXcds - 1) / kXcds + 7) / 8 * 8, j = wg / kXcds;
    const uint32_t per = bands < grid / kXcds ? bands : grid / kXcds;         // (no more than there are workgroups of an XCD, which may be no whole bands)
    const uint32_t last = full + wg % kXcds * per + j;
    return tile_id < full && j < per && last < end ? last : end;
}

}  // namespace cmx
