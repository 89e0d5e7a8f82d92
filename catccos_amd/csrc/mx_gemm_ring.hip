// Block-scaled and INT8 matmul for problems of one round of tiles and for short groups: TW weight rows x TM activation rows (128 x 128 to 256 x 128) per
// workgroup of four wavefronts.
//
// What bounds it: a CU moves some 87 bytes per nanosecond from the L2 into its LDS (1.3-1.5 ns for a 128-byte line), whatever
// waits for them, so a tile costs what its rows cost: 64 x 64 tiles of the split-K kernel pull a byte of operands for 64 flop,
// 128 x 128 ones for 128, and 256 x 256 ones for 256, but of those a problem of 1024 x 4096 has only 64.  Measured there at K = 7168:
// split-K 50.4 us, 256 x 256 64, this kernel 36.4, of which its loads alone would take 28, its MFMAs alone 26 (the chip lowers its
// clock under them: 32 workgroups alone 20) and start, prologue and epilogue 7.
//   * Slabs of 128 bytes of K travel by LDS-DMA into a ring of three slots; one barrier per slab says both that slab s has been read and
//     that slab s + 1 has arrived.  A fourth slot changes nothing (38.4 against 36.6); only INT8 at 128 x 128, which has no scales, has one.
//   * One wavefront per SIMD issues in order, so the matrix pipe is busy only if LDS reads and loads stand between the MFMAs; the
//     compiler puts the MFMAs of a slab together behind them (48 us at 64 rows, where the order below takes 30).  So each step of
//     the loop is pinned (sched_barrier): an MFMA, its share of the fragment reads of the step after, its share of the loads.  The loads
//     of a slab are spread over both steps (all of them in one: 37).
//   * Tile loads without branches: past the last slab they go on from a buffer of no bytes.  (The one branch of the loop asks for the next
//     block of scales.)
//   * Scales are a byte per 32 elements in rows of their own.  A dword per row and slab touches as many lines as the tile itself
//     (320 lines a slab instead of 256: 4.5 us), so they come SPAN dwords of a row at a time into one of two halves of an area behind the
//     ring.  SPAN is what the LDS has left: 32 dwords at 128 x 128, 16 at 128 x 192, 4 at 128 x 256 and 256 x 128.  A slab takes one of them, of
//     FP4 (256 elements) two.  INT8 has none: its scales are the epilogue's.
//   * Weights stored [K, N] (KSLOW) are fetched as they lie, 128 columns of 128 K positions, and turned on the way from the LDS into
//     the registers by ds_read_b64_tr_b8: 1024 x 4096 x 7168 38.9 us, where the pass that rewrites them takes 15 and a launch.
// The K order of the sums is that of the 256-row kernels (one chain, the same instruction), and so are the bits.
#include "mx_gemm_ring_tile.h"
#include "mx_launch.h"

namespace cmx {

namespace {

template <int FMT, int TW, int TM, int WW, int WM, int NSLOT, int SPAN, int EPI, bool KSLOW>
__global__ __launch_bounds__(64 * WW * WM) void mx_gemm_ring_kernel(const GemmParams p) {
    Tile tc;
    if (!locate_tile<TM, Locate::kAny>(p, tc)) return;
    ring_tile<FMT, TW, TM, WW, WM, NSLOT, SPAN, EPI, KSLOW>(p, tc);
}

template <int FMT, int TW, int TM, int WW, int WM, int NSLOT, int SPAN, int EPI, bool KSLOW>
int launch_one(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    constexpr auto kfn = mx_gemm_ring_kernel<FMT, TW, TM, WW, WM, NSLOT, SPAN, EPI, KSLOW>;
    constexpr size_t smem = ring_lds_bytes(TW, TM, NSLOT, SPAN);
    static_assert(smem <= 160 * 1024, "LDS");
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    hipLaunchKernelGGL(kfn, dim3((uint32_t)tiles), dim3(64 * WW * WM), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

template <int FMT, int EPI, bool KSLOW>
int launch_shape(const GemmParams& p, const RingTile& t, uint32_t max_m_tiles, hipStream_t s) {
    if (t.tw == 128 && t.tm == 128) return launch_one<FMT, 128, 128, 2, 2, 3, 32, EPI, KSLOW>(p, max_m_tiles, s);
    if (t.tw == 128 && t.tm == 256) return launch_one<FMT, 128, 256, 2, 2, 3, 4, EPI, KSLOW>(p, max_m_tiles, s);
    if constexpr (EPI == kEpiStore && FMT != CMX_FMT_E2M1) {
        if (t.tw == 128 && t.tm == 192) return launch_one<FMT, 128, 192, 2, 2, 3, 16, EPI, KSLOW>(p, max_m_tiles, s);
    }
    if constexpr (!KSLOW) {
        if (t.tw == 256 && t.tm == 128) return launch_one<FMT, 256, 128, 2, 2, 3, 4, EPI, KSLOW>(p, max_m_tiles, s);
    }
    set_error("unsupported ring tile");
    return CMX_EINVAL;
}

}  // namespace

int launch_ring(const GemmParams& params, const RingTile& t, int fmt, int epi, bool k_slow, uint32_t max_m_tiles, hipStream_t s) {
    GemmParams p = params;
    // The split-K kernels, which share the dense sizes with this one, take scale rows of any pitch.
    if (!k_slow && ((uint64_t)p.n * p.ld_ws >= (1ull << 32) || (uint64_t)p.ld_as * t.tm >= (1ull << 32))) p.scale_vec = 0;
    if (fmt == CMX_FMT_E4M3 && epi == kEpiStore)
        return k_slow ? launch_shape<CMX_FMT_E4M3, kEpiStore, true>(p, t, max_m_tiles, s) : launch_shape<CMX_FMT_E4M3, kEpiStore, false>(p, t, max_m_tiles, s);
    if (fmt == CMX_FMT_E5M2 && epi == kEpiStore)
        return k_slow ? launch_shape<CMX_FMT_E5M2, kEpiStore, true>(p, t, max_m_tiles, s) : launch_shape<CMX_FMT_E5M2, kEpiStore, false>(p, t, max_m_tiles, s);
    if (fmt == CMX_FMT_E4M3 && epi == kEpiSwigluQuant && !k_slow) return launch_shape<CMX_FMT_E4M3, kEpiSwigluQuant, false>(p, t, max_m_tiles, s);
    if (fmt == CMX_FMT_E4M3 && epi == kEpiSwigluQuantAct && !k_slow) return launch_shape<CMX_FMT_E4M3, kEpiSwigluQuantAct, false>(p, t, max_m_tiles, s);
    if (fmt == CMX_FMT_E2M1 && epi == kEpiStore && !k_slow) return launch_shape<CMX_FMT_E2M1, kEpiStore, false>(p, t, max_m_tiles, s);
    if (fmt == kFmtI8 && epi == kEpiI8DequantSwiglu && !k_slow) {
        if (t.tw == 128 && t.tm == 128) return launch_one<kFmtI8, 128, 128, 2, 2, 4, 0, kEpiI8DequantSwiglu, false>(p, max_m_tiles, s);
        if (t.tw == 128 && t.tm == 256) return launch_one<kFmtI8, 128, 256, 2, 2, 3, 0, kEpiI8DequantSwiglu, false>(p, max_m_tiles, s);
        if (t.tw == 256 && t.tm == 128) return launch_one<kFmtI8, 256, 128, 2, 2, 3, 0, kEpiI8DequantSwiglu, false>(p, max_m_tiles, s);
    }
    set_error("unsupported ring problem");
    return CMX_EINVAL;
}

}  // namespace cmx
