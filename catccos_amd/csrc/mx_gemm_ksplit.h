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
size_t ksplit_lds_bytes(const KsplitTile& t, int fmt, uint32_t kblocks, bool tiled);

// p as for the other kernels, with w_tiles counted in tiles of 16 * t.fw weight rows (8 * t.fw output columns for epilogues
// that pair gate and up) and, for grouped problems, group tables made for m-tiles of 16 * t.fm rows.
// stream: load the weights non-temporal (grouped problems whose groups mostly fit one m-tile: each weight byte has one reader,
// and the hint keeps the activation rows in the L2.  32 experts x 4 / 16 rows, K = 7168, N = 4096: 142 / 145 us with it, 160 /
// 162 us without; 64 rows, where a second m-tile reads the weights again, 244 against 242 us).
int launch_ksplit(const GemmParams& p, const KsplitTile& t, int fmt, int epi, uint32_t max_m_tiles, bool stream, hipStream_t s);

}  // namespace cmx
