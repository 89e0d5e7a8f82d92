// What the block-scaled matmul kernels of all translation units share: the parameter block, the epilogue kinds, the mapping
// of tile numbers to (group, m-tile, weight tile) and of workgroups to tile numbers.
#pragma once

#include "mx_common.h"
#include "tile_walk.h"

namespace cmx {

#if defined(__HIPCC__)

constexpr int kSlabBytes = 128;     // K bytes per LDS slab and row
constexpr int kChunks = kSlabBytes / 16;

// kEpiStoreBf16 / kEpiStoreFp16: 16-bit output whose rows and row pitch are multiples of eight elements (16-byte
// stores, no per-element edge handling): small enough to sit inside a persistent kernel's tile loop.  Two epilogues, not one with a run-time switch: a second copy of the store loop inside the kernel costs
// registers, and values spilled because of it are reloaded inside the scheduled loop, where the waits that the
// compiler puts behind such reloads drain the operand loads in flight.
// kEpiSwigluQuantAct: kEpiSwigluQuant that also writes the bf16 SwiGLU output (what the tests check the requantised
// codes against).  A kernel of its own for the same reason: the extra output path costs the SwiGLU kernels
// 30 registers, all of them spilled at the tile boundaries, 3 % of a launch, whether the output is asked for or not.
enum Epilogue { kEpiStore = 0, kEpiSwigluQuant = 1, kEpiStoreBf16 = 2, kEpiI8DequantSwiglu = 3, kEpiStoreFp16 = 4, kEpiSwigluQuantAct = 5 };
constexpr bool epi_is_lean_store(int epi) { return epi == kEpiStoreBf16 || epi == kEpiStoreFp16; }
constexpr bool epi_is_swiglu_quant(int epi) { return epi == kEpiSwigluQuant || epi == kEpiSwigluQuantAct; }
// epilogues whose weight tile pairs gate rows (first half of N) with their up partners (second half)
constexpr bool epi_pairs_gate_up(int epi) { return epi_is_swiglu_quant(epi) || epi == kEpiI8DequantSwiglu; }
// element "format" of the INT8 path inside the kernel templates (the public format codes are the MX ones)
constexpr int kFmtI8 = 8;

// Groups of a grouped problem that a launch takes: all; those of 1 .. small_rows rows (one m-tile each); those of more.
enum GroupClass { kAllGroups = 0, kSmallGroups = 1, kLargeGroups = 2 };
constexpr uint32_t kInlineGroups = 256;

struct GemmParams {
    const uint8_t* a;        // activations codes
    const uint8_t* a_scale;
    const uint8_t* w;        // weights codes [groups][n][ldw]
    const uint8_t* w_scale;  // [groups][n][ld_ws]
    void* c;
    uint8_t* act_codes;
    uint8_t* act_scales;
    uint16_t* act_bf16;
    const int32_t* row_off;     // [groups+1] (grouped) or null (dense)
    const int32_t* tile_pref;   // [groups+1] prefix of m-tiles (grouped) or null
    int32_t* tile_ctr;          // [8] per-XCD tile counters, zeroed before the launch (persistent grouped 4 x 1 kernels) or null
    uint32_t lda, ld_as, ldw, ld_ws, ldc, ld_act, ld_acts;
    uint32_t m, n, kbytes, kblocks;   // kblocks = K/32
    uint32_t groups, w_tiles;
    int out_type;
    int scale_vec;   // scale rows are 4-byte aligned: one dword load per row and slab
    int scale_vec16; // scale rows are 16-byte aligned: one 16-byte load per row fetches the scales of four slabs
    int w_pretiled;  // w holds the weights in the tiled order of cmx_mx_pretile_weights (the weights-to-registers kernel)
    // (the last members: in front of the others they move the kernel arguments that the scheduled kernels keep in registers, and
    // the weights-to-registers kernel of 256 rows then reloads a spilled value, and waits for all its loads, in every tile)
    const int32_t* sizes;       // [groups] rows of the groups, in the place of row_off and tile_pref (at most kInlineGroups), or null
    uint32_t small_rows;        // with `sizes`: the limit between ...
    int group_class;            // ... the groups that this launch takes (GroupClass)
    const int32_t* short_tiles; // INT8, 128- or 256-row tiles chosen on the device (choice_cus != 0): the choice, where tables have been filled
    uint32_t choice_cus;        // ... and the workgroups that run at a time
};

__device__ __forceinline__ uint32_t swz(uint32_t row, uint32_t chunk) {
    return chunk ^ ((row & 7u) ^ ((row >> 3) & 1u));
}

__device__ __forceinline__ v4f to_v4(const v16f& v, int q) {
    v4f r = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    return r;
}

// g / (1 + exp(-g)) * u with the hardware exponential and reciprocal (about 1 ulp each; the result is rounded
// to bf16 right after)
__device__ __forceinline__ float silu_mul(float g, float u) {
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-g));
    return (g * s) * u;
}

// v as the fp32 value it is written as.  (_Float16)(a * b) becomes one v_fma_mixlo_f16, which rounds the product to fp16
// once, also where the product is written __fmul_rn: a whole fp16 step away from the two roundings where the fp32 product is
// a tie between two fp16 values.  The empty asm makes the product a register of its own.
__device__ __forceinline__ float as_f32(float v) {
    asm("" : "+v"(v));
    return v;
}

// INT8 path: fp16(fp32(sum) * channel scale), the two roundings of the reference's arithmetic
// (examples/utils/gen_data_dispatch_gmm_dequant_swiglu.py:291-320), as fp32
__device__ __forceinline__ float i8_dequant(int32_t sum, float channel_scale) {
    return (float)(_Float16)as_f32(__fmul_rn((float)sum, channel_scale));
}

struct Tile {
    uint32_t g, mt, wt, row0, rows_valid;
    uint32_t rows_left;      // rows of the group (or problem) from row0 on
    uint32_t group_tiles;    // m-tiles of the group (or problem)
};

// The group tables (row offsets, m-tile prefix) are written by gmm_prepare_kernel before the matmul kernel starts and
// never change under it: reading them through the constant address space lets a wavefront-uniform lookup use scalar
// loads, which wait on lgkmcnt and so do not drain the LDS-DMA loads a persistent kernel has in flight (a vector load
// would: its s_waitcnt vmcnt covers everything issued before it).
__device__ __forceinline__ int32_t table_at(const int32_t* t, uint32_t i) {
    return ((const __attribute__((address_space(4))) int32_t*)t)[i];
}

// Tiles are numbered linearly: within a group m-tiles run fastest so that neighbours share a weight panel;
// dense problems walk bands of four m-tiles across a run of weight tiles.
template <int TM>
__device__ __forceinline__ uint32_t count_m_tiles(const GemmParams& p) {
    return p.row_off != nullptr ? (uint32_t)table_at(p.tile_pref, p.groups) : (p.m + TM - 1) / TM;
}

// Tile L of an XCD-aware order: linear ids congruent mod 8 run on one XCD; each XCD gets a contiguous run.
// Returns the first tile of XCD x and the number of tiles it owns.
__device__ __forceinline__ uint32_t xcd_run(uint32_t total_tiles, uint32_t x, uint32_t& count) {
    const uint32_t base = total_tiles / kXcds, rem = total_tiles % kXcds;
    count = base + (x < rem ? 1u : 0u);
    return x * base + (x < rem ? x : rem);
}

// One tile per workgroup (blockIdx.x < total_tiles).  Workgroups start in the order of their ids, ids congruent mod 8 on one
// XCD.  Whole chunks of 256 tiles: the XCDs take blocks of 32 consecutive tiles of the chunk in turn, for the reason given
// at interleave_xcd_walk (the INT8 operator on the 16-expert problem, when it ran on the streaming kernel: 973-982 -> 942-945 us); the rest: a
// contiguous run per XCD.
__device__ __forceinline__ uint32_t tile_of_workgroup(uint32_t total_tiles, uint32_t bid = blockIdx.x) {
    constexpr uint32_t kChunk = 32 * kXcds;
    const uint32_t full = total_tiles / kChunk * kChunk;
    if (bid < full) return bid / kChunk * kChunk + (bid % kXcds) * 32 + (bid % kChunk) / kXcds;
    uint32_t count;
    const uint32_t k = bid - full;
    return full + xcd_run(total_tiles - full, k % kXcds, count) + k / kXcds;
}

// Tile L of group g, whose m-tiles are tp .. tp1 - 1 and whose rows r_begin .. r_end - 1.  Bands of 8 m-tiles share a run of weight tiles
// (m fastest inside a band): the 32 tiles that an XCD works on at a time then touch 8 + 4 operand panels instead of mtg + 32/mtg
// SHORT: groups of one m-tile, which is what short groups are, without a division
template <int TM, bool SHORT = false>
__device__ __forceinline__ void place_in_group(const GemmParams& p, uint32_t g, uint32_t tp, uint32_t tp1, uint32_t r_begin, uint32_t r_end,
                                               uint32_t L, Tile& t) {
    t.g = g;
    const uint32_t mtg = tp1 - tp;
    t.group_tiles = mtg;
    const uint32_t local = L - tp * p.w_tiles;
    if (SHORT && mtg == 1) {
        t.mt = 0;
        t.wt = local;
        t.row0 = r_begin;
        t.rows_left = r_end - r_begin;
        t.rows_valid = t.rows_left < (uint32_t)TM ? t.rows_left : (uint32_t)TM;
        return;
    }
    const uint32_t band = 8;
    const uint32_t per_band = band * p.w_tiles;
    const uint32_t b = local / per_band, within = local % per_band;
    const uint32_t band_rows = (mtg - b * band) < band ? (mtg - b * band) : band;
    t.mt = b * band + within % band_rows;
    t.wt = within / band_rows;
    t.row0 = r_begin + t.mt * TM;
    t.rows_left = r_end - t.row0;
    t.rows_valid = t.rows_left < (uint32_t)TM ? t.rows_left : (uint32_t)TM;
}

// Tile L of a dense problem: bands of 4 m-tiles share a run of weight tiles
template <int TM>
__device__ __forceinline__ void place_dense(const GemmParams& p, uint32_t m_tiles_all, uint32_t L, Tile& t) {
    const uint32_t band = 4;
    const uint32_t per_band = band * p.w_tiles;
    const uint32_t b = L / per_band, within = L % per_band;
    const uint32_t band_rows = (m_tiles_all - b * band) < band ? (m_tiles_all - b * band) : band;
    t.g = 0;
    t.group_tiles = m_tiles_all;
    t.mt = b * band + within % band_rows;
    t.wt = within / band_rows;
    t.row0 = t.mt * TM;
    t.rows_left = p.m - t.row0;
    t.rows_valid = t.rows_left < (uint32_t)TM ? t.rows_left : (uint32_t)TM;
}

// g_from: a group at or before the tile's (0, or the group of an earlier tile of an increasing sequence)
template <int TM>
__device__ __forceinline__ void decode_tile(const GemmParams& p, uint32_t m_tiles_all, uint32_t L, Tile& t, uint32_t g_from = 0) {
    if (p.row_off != nullptr) {
        // find g with tile_pref[g]*w_tiles <= L < tile_pref[g+1]*w_tiles.  A workgroup's next tile mostly lies in the
        // same group or one of the next two: three independent loads settle that before the bisection's
        // chain of dependent ones
        const uint32_t G = p.groups;
        uint32_t lo = g_from, hi = G;
        const uint32_t i2 = lo + 2 < G ? lo + 2 : G, i3 = lo + 3 < G ? lo + 3 : G;
        const uint32_t t1 = (uint32_t)table_at(p.tile_pref, lo + 1) * p.w_tiles, t2 = (uint32_t)table_at(p.tile_pref, i2) * p.w_tiles,
                       t3 = (uint32_t)table_at(p.tile_pref, i3) * p.w_tiles;
        if (t1 > L) hi = lo + 1;
        else if (t2 > L) { lo += 1; hi = lo + 1; }
        else if (t3 > L) { lo += 2; hi = lo + 1; }
        else lo += 3;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if ((uint32_t)table_at(p.tile_pref, mid) * p.w_tiles <= L) lo = mid; else hi = mid;
        }
        place_in_group<TM>(p, lo, (uint32_t)table_at(p.tile_pref, lo), (uint32_t)table_at(p.tile_pref, lo + 1), (uint32_t)table_at(p.row_off, lo),
                           (uint32_t)table_at(p.row_off, lo + 1), L, t);
    } else {
        place_dense<TM>(p, m_tiles_all, L, t);
    }
}

// op (neutral element 0) over lanes 0 .. l of the wavefront, in lane l
template <class Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, Op op) {
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false));       // row_shr:1
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));       // row_bcast:15
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));       // row_bcast:31
    return v;
}

// The tile of this workgroup from the group sizes themselves: every wavefront scans them (four groups per lane), so that no launch has to
// write tables first (5 us) and no chain of dependent table reads follows the start of every workgroup.  Sizes are clipped as in
// fill_group_tables: negative ones count as zero, rows past m_total (p.m) do not exist (a sum that stops at m_total is associative).
constexpr int kGroupsPerLane = kInlineGroups / 64;
// off[0 .. kGroupsPerLane]: where the rows of the lane's groups begin, and where the last of them ends
__device__ __forceinline__ void scan_group_rows(const GemmParams& p, uint32_t (&off)[kGroupsPerLane + 1]) {
    const uint32_t lane = threadIdx.x & 63u, m = p.m;
    const auto sat = [m](uint32_t a, uint32_t b) -> uint32_t { return min(a + b, m); };          // a, b <= m < 2^31
    uint32_t c[kGroupsPerLane], sum = 0;
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) {
        const uint32_t i = kGroupsPerLane * lane + j;
        const int32_t v = i < p.groups ? p.sizes[i] : 0;
        c[j] = v > 0 ? min((uint32_t)v, m) : 0u;
        sum = sat(sum, c[j]);
    }
    const uint32_t to = wave_scan(sum, sat);
    off[0] = (uint32_t)__shfl_up((int)to, 1);
    if (lane == 0) off[0] = 0;
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) off[j + 1] = sat(off[j], c[j]);
}
// m-tiles of tm rows that the launch makes of a group
__device__ __forceinline__ uint32_t tiles_of_group(const GemmParams& p, uint32_t rows, uint32_t tm) {
    const uint32_t small = rows <= p.small_rows ? 1u : 0u, whole = (rows + tm - 1) / tm;
    return p.group_class == kAllGroups ? whole : (p.group_class == kSmallGroups ? (rows != 0 ? small : 0u) : (small ? 0u : whole));
}

// The two scans are independent of each other where the sizes add up to no more than the rows that there are; otherwise (a sum that stops one
// past them says so) the rows are clipped first.  It stands in front of the first load of every workgroup (FP4, 32 groups x 16 rows: 1.4 us of
// 17; with one scan behind the other, a trip through the LDS between them and divisions for groups of one m-tile 1.7).
template <int TM>
__device__ __forceinline__ bool locate_tile_by_sizes(const GemmParams& p, Tile& t, uint32_t bid) {
    constexpr int kPer = kGroupsPerLane;
    static_assert(kPer == 4, "a 16-byte load");
    const uint32_t lane = threadIdx.x & 63u, m = p.m;
    const auto add = [](uint32_t a, uint32_t b) -> uint32_t { return a + b; };
    const auto sat = [m](uint32_t a, uint32_t b) -> uint32_t { return min(__builtin_elementwise_add_sat(a, b), m + 1); };      // (two sums of 2^31 do not wrap)
    int32_t v[kPer] = {0, 0, 0, 0};
    if (kPer * lane + kPer <= p.groups) {
        __builtin_memcpy(v, p.sizes + kPer * lane, sizeof v);
    } else {
#pragma unroll
        for (int j = 0; j < kPer - 1; ++j)
            if (kPer * lane + j < p.groups) v[j] = p.sizes[kPer * lane + j];
    }
    uint32_t off[kPer + 1], tiles[kPer], all = 0, rows = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t c = v[j] > 0 ? min((uint32_t)v[j], m) : 0u;
        off[j] = rows;
        rows = sat(rows, c);
        tiles[j] = tiles_of_group(p, c, TM);
        all += tiles[j];
    }
    off[kPer] = rows;
    uint32_t pref = all;
    const uint32_t to = wave_scan(rows, sat);
    pref = wave_scan(pref, add);
    if ((uint32_t)__builtin_amdgcn_readlane((int)to, 63) <= m) {
#pragma unroll
        for (int j = 0; j <= kPer; ++j) off[j] += to - rows;
    } else {
        scan_group_rows(p, off);
        all = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            tiles[j] = tiles_of_group(p, off[j + 1] - off[j], TM);
            all += tiles[j];
        }
        pref = wave_scan(all, add);
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)pref, 63) * p.w_tiles;
    if (bid >= total) return false;
    const uint32_t L = tile_of_workgroup(total, bid);
    const int at = (int)__builtin_ctzll(__ballot(pref * p.w_tiles > L));                         // lane of the tile's group
    uint32_t tp = (uint32_t)__builtin_amdgcn_readlane((int)(pref - all), at), g = kPer * at;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)tiles[j], at);
        const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)off[j], at), r1 = (uint32_t)__builtin_amdgcn_readlane((int)off[j + 1], at);
        if (L >= tp * p.w_tiles && L < (tp + n) * p.w_tiles) place_in_group<TM, true>(p, g + j, tp, tp + n, r0, r1, L, t);
        tp += n;
    }
    return true;
}

// The same for persistent kernels: the groups are scanned once and stay in registers, so that the way to a further tile touches no memory.
struct GroupScan {
    uint32_t rows[kGroupsPerLane], row0, tile0;      // of the lane's groups: rows of each; first row and first m-tile of the first
};
// returns the m-tiles of all groups
template <int TM>
__device__ __forceinline__ uint32_t scan_groups(const GemmParams& p, GroupScan& gs) {
    uint32_t off[kGroupsPerLane + 1], all = 0;
    scan_group_rows(p, off);
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) {
        gs.rows[j] = off[j + 1] - off[j];
        all += tiles_of_group(p, gs.rows[j], TM);
    }
    const uint32_t pref = wave_scan(all, [](uint32_t a, uint32_t b) -> uint32_t { return a + b; });
    gs.row0 = off[0];
    gs.tile0 = pref - all;
    return (uint32_t)__builtin_amdgcn_readlane((int)pref, 63);
}
// tile L, which exists
template <int TM>
__device__ __forceinline__ void decode_scanned_tile(const GemmParams& p, const GroupScan& gs, uint32_t L, Tile& t) {
    uint32_t end = gs.tile0;
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) end += tiles_of_group(p, gs.rows[j], TM);
    const int at = (int)__builtin_ctzll(__ballot(end * p.w_tiles > L));                          // lane of the tile's group
    uint32_t tp = (uint32_t)__builtin_amdgcn_readlane((int)gs.tile0, at), r0 = (uint32_t)__builtin_amdgcn_readlane((int)gs.row0, at);
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) {
        const uint32_t rows = (uint32_t)__builtin_amdgcn_readlane((int)gs.rows[j], at), n = tiles_of_group(p, rows, TM);
        if (L >= tp * p.w_tiles && L < (tp + n) * p.w_tiles) place_in_group<TM>(p, kGroupsPerLane * at + j, tp, tp + n, r0, r0 + rows, L, t);
        tp += n;
        r0 += rows;
    }
}

// How a kernel finds its tiles: without a look for groups, in their tables (or none), by their sizes, or as the parameters say.  What a kernel
// never does is left out of it.  The 500 to 1000 instructions that look for groups stand between the start of a small kernel and its first
// load (dense split-K, us, without -> with: 48 x 2048 x 512 4.8 -> 5.1, 1 x 4096 x 7168 8.6 -> 9.1), and two ways in one kernel cost
// each of its workgroups 0.07 us, of which a launch for few rows in many groups has ten thousand (200 groups, 400 rows on four of them,
// K = 640, N = 3584: 15.9 against 14.1).
enum class Locate { kDense, kTables, kSizes, kAny };

// Maps the id of a workgroup (of one that goes on with further tiles: of the workgroup that would take this one if each took one) to
// (group, m-tile, weight tile).  Returns false for ids past the last tile.
template <int TM, Locate HOW>
__device__ __forceinline__ bool locate_tile(const GemmParams& p, Tile& t, uint32_t bid = blockIdx.x) {
    if constexpr (HOW == Locate::kDense) {
        const uint32_t m_tiles = (p.m + TM - 1) / TM, total_tiles = m_tiles * p.w_tiles;
        if (bid >= total_tiles) return false;
        place_dense<TM>(p, m_tiles, tile_of_workgroup(total_tiles, bid), t);
        return true;
    }
    if constexpr (HOW == Locate::kSizes) return locate_tile_by_sizes<TM>(p, t, bid);
    if constexpr (HOW == Locate::kAny)
        if (p.sizes != nullptr) return locate_tile_by_sizes<TM>(p, t, bid);
    const uint32_t m_tiles_all = count_m_tiles<TM>(p);
    const uint32_t total_tiles = m_tiles_all * p.w_tiles;
    if (bid >= total_tiles) return false;
    decode_tile<TM>(p, m_tiles_all, tile_of_workgroup(total_tiles, bid), t);
    return true;
}

#endif  // __HIPCC__

}  // namespace cmx
