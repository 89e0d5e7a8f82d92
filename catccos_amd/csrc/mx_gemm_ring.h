// Host interface of the ring matmul kernels (mx_gemm_ring.hip).
#pragma once

#include "mx_gemm_common.h"

namespace cmx {

// Tile of a ring launch, weight rows x activation rows: 128 x 128, 128 x 256, 256 x 128 (not k_slow), 128 x 192 (8-bit formats, plain store).
struct RingTile {
    int tw, tm;
};

// p as for the other kernels, with w_tiles counted in tiles of t.tw weight rows (t.tw / 2 output columns for epilogues that pair gate and
// up) and, for grouped problems, group tables made for m-tiles of t.tm rows; MX formats (scale rows of any alignment and pitch) and INT8, K whole
// 128-byte slabs.
// k_slow: p.w is [K][ldw] and p.w_scale [K / 64][n][2] at a pitch of ld_ws bytes; dense, n a multiple of 4 and at least 16, p.w dword-aligned,
// K * ldw below 2^32.
int launch_ring(const GemmParams& p, const RingTile& t, int fmt, int epi, bool k_slow, uint32_t max_m_tiles, hipStream_t s);

// cmx_mx_gemm on weights stored [k, n] with scales [k / 64, n, 2] (a: [m, k], scales [m, k / 32]; k a multiple of 64) where a kernel reads
// them as they lie; *taken = false, and nothing launched, where none does.
int gemm_k_slow(const uint8_t* a, const uint8_t* a_scale, const uint8_t* b, const uint8_t* b_scale, void* c, uint32_t ldc, uint32_t m,
                uint32_t n, uint32_t k, int fmt, int out_type, hipStream_t s, bool* taken);

}  // namespace cmx
