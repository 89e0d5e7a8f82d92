// Host interface of the split-K matmul kernels (mx_gemm_ksplit.hip).
#pragma once

#include "mx_gemm_common.h"

namespace cmx {

// Tile of a split-K launch: 16 * fw weight rows x 16 * fm activation rows by `waves` wavefronts; fw == 0: none.
struct KsplitTile {
    int fw, fm, waves;
};

// LDS bytes the kernel needs for a tile of a problem (scale rows of the whole tile and the exchange buffers, or the partial
// sums), and the most it may ask for.
constexpr size_t kKsplitMaxLds = 160 * 1024;
size_t ksplit_lds_bytes(const KsplitTile& t, int fmt, uint32_t kblocks, int layout = 0);

// How the weights are read.  kStreamed: non-temporal, for weights with one reader, which leaves the L2 to the activation rows (32
// experts x 4 / 16 / 32 rows, K = 7168, N = 4096: 142 / 145 / 152 us with it, 160 / 162 / 172 without).  kCached: for weights that the
// next m-tile reads again.  kByGroup: each group as its size asks for (32 experts, 1024 rows on one of them: streamed 76, by group 55; 256
// experts x 8 rows, where all are streamed either way, pre-tiled 1101 and 1112: twice the code).
enum class KsplitWeights { kCached, kStreamed, kByGroup };

// p as for the other kernels, with w_tiles counted in tiles of 16 * t.fw weight rows (8 * t.fw output columns for epilogues
// that pair gate and up) and, for grouped problems, group tables made for m-tiles of 16 * t.fm rows.  Dense problems read their
// weights cached; `loads` is for grouped ones.
int launch_ksplit(const GemmParams& p, const KsplitTile& t, int fmt, int epi, uint32_t max_m_tiles, KsplitWeights loads, hipStream_t s);


// Weights stored [K][ldw] with scales [K / 64][n][2] at a pitch of ld_ws bytes (dense, 8-bit formats, K whole slabs, n a multiple of 4
// and at least 16, p.w dword-aligned, K * ldw below 2^32): tiles of 64 columns with the wavefronts, and so the bits, of the tile that
// the same problem gets on K-contiguous weights.  Turns *t into such a tile; false where its scales do not fit the LDS.
bool ksplit_k_slow_tile(KsplitTile* t, uint32_t m, uint32_t n, int fmt, uint32_t kblocks, int cus);
int launch_ksplit_k_slow(const GemmParams& p, const KsplitTile& t, int fmt, uint32_t max_m_tiles, hipStream_t s);

}  // namespace cmx
