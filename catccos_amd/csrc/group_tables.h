// The tables that a grouped matmul schedules its tiles by, written on the device from the group sizes, and what of them other
// launches of a chain can fill on the side.
#pragma once

#include <type_traits>

#include "mx_gemm_common.h"

namespace cmx {

struct GroupTablesJob {
    const int32_t* sizes;                                  // [groups]
    uint32_t groups, tile_m, m_total, small_rows;
    int32_t *row_off, *tile_pref, *small_pref;             // [groups + 1] each
    int32_t* tile_ctr;                                     // [kXcds], zeroed
};

#if defined(__HIPCC__)

// Row offsets and m-tile prefix of the groups (one workgroup of 256 threads): each thread owns a contiguous run of
// groups; the 256 partial sums are scanned in LDS, first for the rows, then for the m-tiles.
// Group sizes live on the device, so the host cannot check them: negative sizes count as zero and rows past
// m_total (the rows the caller's buffers hold) are cut off here, so that no tile ever points outside them.
// small_rows != 0: groups of 1 .. small_rows rows are one m-tile each of small_pref and none of tile_pref.
// With pick, the tables are for m-tiles of tile_m or of alt_tile_m rows: pick(m-tiles of the first height, of the second) says whether the
// first, to every thread alike.
struct NoPick {};
template <class Pick = NoPick>
__device__ __forceinline__ void fill_group_tables(const GroupTablesJob& j, uint32_t alt_tile_m = 0, Pick pick = {}) {
    constexpr bool kPick = !std::is_same<Pick, NoPick>::value;
    __shared__ unsigned long long part_r[256];
    __shared__ int32_t part_t[256], part_s[256], part_a[kPick ? 256 : 1];
    if (threadIdx.x < kXcds) j.tile_ctr[threadIdx.x] = 0;
    const uint32_t per = (j.groups + 255) / 256;
    const uint32_t lo = threadIdx.x * per < j.groups ? threadIdx.x * per : j.groups;
    const uint32_t hi = lo + per < j.groups ? lo + per : j.groups;
    auto size_of = [&](uint32_t i) -> unsigned long long {
        const int32_t c = j.sizes[i];
        return c > 0 ? (unsigned long long)c : 0ull;
    };
    // inclusive scan of part[0..255] in place: within each wavefront by lane shuffles, then the three wavefront totals
    // before it added to every element (two barriers instead of sixteen)
    auto scan256 = [&](auto* part) {
        auto v = part[threadIdx.x];
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const auto u = __shfl_up(v, d);
            if (lane >= (uint32_t)d) v += u;
        }
        part[threadIdx.x] = v;
        __syncthreads();
        decltype(v) before = 0;
        for (uint32_t w = 0; w < wave; ++w) before += part[64 * w + 63];
        __syncthreads();
        part[threadIdx.x] = v + before;
        __syncthreads();
    };
    unsigned long long r = 0;
    for (uint32_t i = lo; i < hi; ++i) r += size_of(i);
    part_r[threadIdx.x] = r;
    __syncthreads();
    scan256(part_r);
    const unsigned long long r_base = threadIdx.x ? part_r[threadIdx.x - 1] : 0ull;
    // rows of group i that fit below j.m_total, given the rows before it
    auto clipped = [&](unsigned long long before, unsigned long long c) -> uint32_t {
        const unsigned long long b = before < j.m_total ? before : j.m_total;
        const unsigned long long e = before + c < j.m_total ? before + c : j.m_total;
        return (uint32_t)(e - b);
    };
    auto is_small = [&](uint32_t rows) -> bool { return rows != 0 && rows <= j.small_rows; };
    r = r_base;
    int32_t t = 0, sm = 0, ta = 0;
    for (uint32_t i = lo; i < hi; ++i) {
        const unsigned long long c = size_of(i);
        const uint32_t rows = clipped(r, c);
        if (is_small(rows)) ++sm;
        else t += (int32_t)((rows + j.tile_m - 1) / j.tile_m);
        if constexpr (kPick)
            if (!is_small(rows)) ta += (int32_t)((rows + alt_tile_m - 1) / alt_tile_m);
        r += c;
    }
    part_t[threadIdx.x] = t;
    part_s[threadIdx.x] = sm;
    if constexpr (kPick) part_a[threadIdx.x] = ta;
    __syncthreads();
    scan256(part_t);
    if (j.small_rows != 0) scan256(part_s);
    const int32_t* tiles = part_t;
    uint32_t tile_m = j.tile_m;
    if constexpr (kPick) {
        scan256(part_a);
        if (!pick((uint32_t)part_t[255], (uint32_t)part_a[255])) {
            tiles = part_a;
            tile_m = alt_tile_m;
        }
    }
    r = r_base;
    t = threadIdx.x ? tiles[threadIdx.x - 1] : 0;
    sm = threadIdx.x ? part_s[threadIdx.x - 1] : 0;
    for (uint32_t i = lo; i < hi; ++i) {
        const unsigned long long c = size_of(i);
        const uint32_t rows = clipped(r, c);
        j.row_off[i] = (int32_t)(r < j.m_total ? r : j.m_total);
        j.tile_pref[i] = t;
        if (j.small_rows != 0) j.small_pref[i] = sm;
        if (is_small(rows)) ++sm;
        else t += (int32_t)((rows + tile_m - 1) / tile_m);
        r += c;
    }
    if (threadIdx.x == 255) {
        const unsigned long long all = part_r[255];
        j.row_off[j.groups] = (int32_t)(all < j.m_total ? all : j.m_total);
        j.tile_pref[j.groups] = tiles[255];
        if (j.small_rows != 0) j.small_pref[j.groups] = part_s[255];
    }
}

#endif  // __HIPCC__

// ---- a chain that fills the tables of its grouped matmuls in an earlier launch --------------------------------------------------------
// What a grouped matmul on these sizes will ask of its tables (in `workspace`, as for the call itself), and the two matmuls of the
// FFN with their tables filled.
int plan_group_tables(GroupTablesJob* job, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, int fmt,
                      bool swiglu, bool pretiled, void* workspace);
int gmm_swiglu_quant_prepared(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b, const uint8_t* b_scale,
                              uint8_t* act_codes, uint32_t ld_act, uint8_t* act_scales, uint32_t ld_acts, const int32_t* group_sizes,
                              uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, void* workspace, bool pretiled, hipStream_t s);
int gmm_prepared(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b, const uint8_t* b_scale, void* c,
                 uint32_t ldc, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, int fmt, int out_type,
                 void* workspace, bool pretiled, hipStream_t s);
// cmx_quant_scatter that also fills `jobs` (up to two) tables
constexpr int kMaxTableJobs = 2;
int quant_scatter_with_tables(const void* x, uint32_t ld_x, const int32_t* src2sorted, uint8_t* out_codes, uint32_t ld_out, uint8_t* out_scales,
                              uint32_t ld_outs, uint32_t tokens, uint32_t k, uint32_t top_k, const GroupTablesJob* job, int jobs, hipStream_t s);
int launch_group_tables(const GroupTablesJob& job, hipStream_t s);

}  // namespace cmx
