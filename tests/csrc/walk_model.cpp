// A host's walk through the index arithmetic of the persistent kernels.  Prints what is wrong; exit status 1 if anything is.
#include <cstdio>
#include <vector>

#include "../../catccos_amd/csrc/tile_walk.h"

using namespace cmx;

namespace {

int faults = 0;

// Slabs that a workgroup's loads ask for in a sequence of tiles, as mx_gemm_pipe_kernel (2 x 2 wavefronts) issues them: two slabs and the
// prefetch of a third before the loop, then in each of its bodies a slab two ahead of the multiplied one and a prefetch two further on.
void check_slabs(uint32_t real, bool fill_to_even) {
    constexpr uint32_t kSlab = 128, kAhead = 2;
    const KSlabs k = k_slabs(real * kSlab, kSlab, fill_to_even);
    const auto expect = [&](bool ok, const char* what, uint32_t sq) {
        if (ok) return;
        ++faults;
        std::printf("%u slabs: %s, load stream at slab %u\n", real, what, sq);
    };
    expect(k.walked % 2 == 0 && k.walked >= real && k.walked <= real + 1, "slabs walked", 0);
    expect(load_slab(0, k) == 0 && load_slab(1, k) == 1 && slab_in_memory(1, k), "first two slabs", 0);
    expect(prefetch_slab(1 + kAhead, k) < real, "first prefetch past K", 1);
    for (uint32_t tile = 0; tile < 3; ++tile) {
        const bool last = tile == 2;
        // slabs sm and sm + 1 are multiplied; the stream enters the next tile where this one's last two are
        for (uint32_t sm = 0; sm < k.walked; sm += 2) {
            uint32_t sq = sm + 2;
            if (sq == k.walked && !last) sq = 0;
            for (uint32_t s = sq; s < sq + 2; ++s) {
                const bool unlimited = slab_in_memory(load_slab(s, k), k);
                expect(s >= k.walked || load_slab(s, k) == s, "a slab left out", s);
                expect(!unlimited || load_slab(s, k) < real, "tile load past K", s);
                expect(!unlimited || prefetch_slab(s + kAhead, k) < real, "prefetch past K", s);
            }
        }
    }
}

// Every tile of `total` goes to one workgroup of `grid`, in the walk of at least a round of tiles.
void check_tiles(uint32_t grid, uint32_t total) {
    std::vector<int> visits(total);
    bool outside = false;
    for (uint32_t wg = 0; wg < grid; ++wg) {
        uint32_t tile = total, stride = 0, end = 0;
        interleave_xcd_walk(total, wg, grid, tile, stride, end);
        for (uint32_t turn = 0; tile < end && turn <= total; tile = next_of_walk(tile, stride, end, wg, grid), ++turn) {
            if (tile < total) ++visits[tile];
            else outside = true;
        }
    }
    uint32_t lost = 0, twice = 0;
    for (int v : visits) lost += v == 0, twice += v > 1;
    if (lost == 0 && twice == 0 && !outside) return;
    ++faults;
    std::printf("%u tiles on %u workgroups: %u with nobody, %u more than once%s\n", total, grid, lost, twice, outside ? ", some that do not exist" : "");
}

}  // namespace

int main() {
    // (launches take a multiple of eight workgroups)
    for (uint32_t grid = 8; grid <= 304; grid += 8)
        for (uint32_t total = grid; total <= (kSpreadRounds + 1) * grid; ++total) check_tiles(grid, total);
    for (uint32_t real = 2; real <= 64; ++real) {
        check_slabs(real, true);
        if (real % 4 == 0) check_slabs(real, false);
    }
    std::printf("%d wrong\n", faults);
    return faults != 0;
}
