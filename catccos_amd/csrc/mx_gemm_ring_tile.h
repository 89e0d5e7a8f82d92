// The tile of the ring matmul (mx_gemm_ring.hip says what it is).
#pragma once

#include <type_traits>

#include "mx_gemm_ring.h"
#include "mx_gemm_store.h"

namespace cmx {

namespace {

// SPAN: scale dwords of a row that one half of the scale area holds
// (0: no scales, the INT8 kernels)
constexpr int ring_scale_bytes(int tw, int tm, int span) { return 2 * (tw + tm) * 4 * span; }
constexpr int ring_sum_bytes(int tw, int tm) { return tm * (tw + 4) * 4; }
constexpr size_t ring_lds_bytes(int tw, int tm, int nslot, int span) {
    const int loop = nslot * (tw + tm) * kSlabBytes + ring_scale_bytes(tw, tm, span), sums = ring_sum_bytes(tw, tm);
    return loop > sums ? loop : sums;
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// LDS-DMA of 16 (or 4) bytes per lane to lds_dst + 16 * lane (4 * lane); lds_dst and soff wavefront-uniform
__device__ __forceinline__ void ring_dma16(uint32_t lds_dst, uint32_t voff, v4i rsrc, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(uniform(lds_dst)), "v"(voff), "s"(rsrc), "s"(uniform(soff)) : "memory");
}
__device__ __forceinline__ void ring_dma4(uint32_t lds_dst, uint32_t voff, v4i rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 ::"s"(uniform(lds_dst)), "v"(voff), "s"(rsrc) : "memory");
}
// all but the youngest N vector memory accesses of this wavefront and all its LDS accesses are done; then everyone's
template <int N>
__device__ __forceinline__ void ring_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// MFMA j of a 64-byte step h: 8-bit formats one of 64 deep; FP4 two of 64 deep on the halves of the fragment registers, each with two scale
// bytes of dword h; INT8 two of 32 deep (a sum of whole numbers does not care which lane holds which K position)
constexpr int ring_subs(int fmt) { return fmt == CMX_FMT_E2M1 || fmt == kFmtI8 ? 2 : 1; }
constexpr int ring_scale_dwords(int fmt) { return fmt == CMX_FMT_E2M1 ? 2 : 1; }             // per row and slab
template <int FMT, int H, int J, int SD>
__device__ __forceinline__ v16f ring_mfma(const v8i& w, const v8i& a, const v16f& c, const uint32_t (&sw)[SD], const uint32_t (&sa)[SD]) {
    const v4i w4 = {w[4 * J], w[4 * J + 1], w[4 * J + 2], w[4 * J + 3]}, a4 = {a[4 * J], a[4 * J + 1], a[4 * J + 2], a[4 * J + 3]};
    if constexpr (FMT == kFmtI8) {
        typedef int v16i __attribute__((ext_vector_type(16)));
        return __builtin_bit_cast(v16f, __builtin_amdgcn_mfma_i32_32x32x32_i8(w4, a4, __builtin_bit_cast(v16i, c), 0, 0, 0));
    } else if constexpr (FMT == CMX_FMT_E2M1) {
        const v8i w8 = {w4[0], w4[1], w4[2], w4[3], 0, 0, 0, 0}, a8 = {a4[0], a4[1], a4[2], a4[3], 0, 0, 0, 0};
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8, a8, c, 4, 4, 2 * J, (int)sw[H], 2 * J, (int)sa[H]);
    } else {
        constexpr int kF = FMT == CMX_FMT_E5M2 ? 1 : 0;
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, kF, kF, 2 * H, (int)sw[0], 2 * H, (int)sa[0]);
    }
}

// One tile, by the first 64 WW WM threads of a workgroup
template <int FMT, int TW, int TM, int WW, int WM, int NSLOT, int SPAN, int EPI, bool KSLOW>
__device__ __forceinline__ void ring_tile(const GemmParams& p, Tile tc) {
    constexpr int NW = WW * WM, NT = 64 * NW, FW = TW / WW / 32, FM = TM / WM / 32;
    constexpr int kRows = TW + TM, kSlotBytes = kRows * kSlabBytes;
    constexpr int kTileLoads = kRows / (8 * NW), kWTileLoads = TW / (8 * NW);
    constexpr int kScaleBase = NSLOT * kSlotBytes, kScaleHalf = kRows * 4 * SPAN;
    constexpr bool kScales = FMT != kFmtI8;
    constexpr int kSD = ring_scale_dwords(FMT), kSpanSlabs = kScales ? SPAN / kSD : 1;
    constexpr int kPieces = SPAN / 4, kAllPieces = kRows * kPieces;     // 16-byte pieces of a row in a half; of all rows
    constexpr int kScaleLoads = (kAllPieces + NT - 1) / NT;
    constexpr int kEarly = kTileLoads / 2;                              // loads of a slab in the second step of the slab before, the rest in the first
    constexpr int kM = FW * FM, kSteps = kM * ring_subs(FMT), kFrags = FW + FM;                       // MFMAs and fragments per step
    static_assert(TW % (8 * NW) == 0 && TM % (8 * NW) == 0 && TW % 64 == 0 && TM % 64 == 0 && FW >= 1 && FM >= 1, "tile shape");
    static_assert(!KSLOW || TW % 128 == 0, "whole 128-byte lines along n");
    static_assert(!epi_pairs_gate_up(EPI) || (!KSLOW && TW % 64 == 0), "gate and up rows");
    static_assert((NSLOT - 1) * kTileLoads < 64, "loads");
    static_assert(kScales ? TW * kPieces % 64 == 0 && TM * kPieces % 64 == 0 && (SPAN & (SPAN - 1)) == 0 && SPAN >= 4 && SPAN <= 32 && kSpanSlabs >= 2 && (!KSLOW || kSD == 1) : SPAN == 0 && !KSLOW, "scales");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = uniform(tid >> 6);
    const uint32_t ww = wave % WW, wm = wave / WW;
    const uint32_t l32 = lane & 31u, lh = lane >> 5;

    tc.g = uniform(tc.g); tc.wt = uniform(tc.wt); tc.row0 = uniform(tc.row0); tc.rows_valid = uniform(tc.rows_valid);
    const uint32_t half = p.n >> 1;

    auto wrow_of = [&](uint32_t t) -> uint32_t {                        // rows past the matrix repeat the last one
        if (epi_pairs_gate_up(EPI)) {
            uint32_t rr = tc.wt * (TW / 2) + (t < TW / 2 ? t : t - TW / 2);
            rr = rr < half ? rr : half - 1;
            return t < TW / 2 ? rr : half + rr;
        }
        const uint32_t gr = tc.wt * TW + t;
        return gr < p.n ? gr : p.n - 1;
    };
    auto arow_of = [&](uint32_t t) -> uint32_t { return t < tc.rows_valid ? t : tc.rows_valid - 1; };
    // K-slow: first column of the tile's 16-column chunk c; one that the matrix ends inside of is moved back to end with it
    // (its first columns are computed twice), one past the end repeats the last
    auto wcol_of = [&](uint32_t c) -> uint32_t {
        const uint32_t col = tc.wt * TW + 16 * c;
        return col + 16 <= p.n ? col : p.n - 16;
    };

    auto make_rsrc = [](const uint8_t* q) -> v4i {
        const uint64_t v = reinterpret_cast<uint64_t>(q);
        return (v4i){(int)uniform((uint32_t)v), (int)uniform((uint32_t)(v >> 32)), -1, 0x00020000};
    };
    // the same buffer, or, past the last slab, one of no bytes: its loads put zeros into the LDS without going to memory, so that
    // every slab counts the same loads and the loop has no branch
    auto live_rsrc = [](const v4i& r, bool live) -> v4i { return (v4i){r[0], r[1], (int)uniform(live ? ~0u : 0u), r[3]}; };
    const v4i w_rs = make_rsrc(KSLOW ? p.w : p.w + (size_t)tc.g * p.n * p.ldw);
    // (INT8: the scales are the epilogue's)
    const uint8_t* const w_scales = KSLOW ? p.w_scale : p.w_scale + (size_t)tc.g * p.n * p.ld_ws;
    const uint8_t* const a_scales = p.a_scale + (size_t)tc.row0 * p.ld_as;
    const v4i ws_rs = make_rsrc(w_scales);
    const v4i a_rs = make_rsrc(p.a + (size_t)tc.row0 * p.lda);
    const v4i as_rs = make_rsrc(a_scales);

    // load i of this wavefront fills combined tile rows (NW * i + wave) * 8 .. + 8; lane -> row lane / 8, LDS chunk lane % 8.
    // K-slow weights: "row" 128 h + k of the tile is K position k of the columns 128 h .. 128 h + 127.
    uint32_t goff[kTileLoads];
#pragma unroll
    for (int i = 0; i < kTileLoads; ++i) {
        const uint32_t cr = (NW * i + wave) * 8 + (lane >> 3), chunk = swz(cr, lane & 7u);
        if (i >= kWTileLoads) goff[i] = arow_of(cr - TW) * p.lda + chunk * 16;
        else if (KSLOW) goff[i] = (cr & 127u) * p.ldw + wcol_of((cr >> 7) * 8 + chunk);
        else goff[i] = wrow_of(cr) * p.ldw + chunk * 16;
    }
    const uint32_t nslab = p.kbytes / kSlabBytes, ndw = p.kblocks / 4;
    const uint32_t w_step = KSLOW ? kSlabBytes * p.ldw : kSlabBytes;

    // load i of slab s into ring slot `slot`
    auto issue_one = [&](uint32_t s, uint32_t slot, int i) {
        const bool live = s < nslab;
        const uint32_t dst = lds0 + slot * kSlotBytes + wave * 1024 + i * (NW * 1024);
        if (i < kWTileLoads) ring_dma16(dst, goff[i], live_rsrc(w_rs, live), s * w_step);
        else ring_dma16(dst, goff[i], live_rsrc(a_rs, live), s * kSlabBytes);
    };
    // Scales of block b (dwords SPAN b .. SPAN b + SPAN - 1 of a row, one a slab, FP4 two) into half b % 2 of the scale area, in pieces of four dwords.
    // K-contiguous rows: the pieces of a row change places by XOR so that the 32 rows of a fragment lie in different banks two by
    // two; a last piece in part is fetched from the row's last 16 bytes.  K-slow weights: [K / 64 within the block][column] pairs.
    const bool whole_pieces = p.scale_vec && ndw >= 4;
    const uint32_t last_dw = whole_pieces ? ndw - 4 : ndw - 1;
    auto load_scales = [&](uint32_t b) {
        if constexpr (kScales) {
            const uint32_t half_at = kScaleBase + (b & 1u) * kScaleHalf;
            // in bytes, as a T: 32 bits do where the pieces are whole (launch_ring)
            auto address = [&](auto as, uint32_t piece, uint32_t d, bool of_w) {
                using T = decltype(as);
                const uint32_t row = piece / kPieces;
                if (KSLOW && of_w) {
                    const uint32_t k64 = 2 * SPAN * b + piece / (TW / 8), col = piece % (TW / 8) * 8 + 2 * d;
                    return (T)(k64 < 2 * nslab ? k64 : 2 * nslab - 1) * p.ld_ws + 2 * (wcol_of(col / 16) + col % 16);
                }
                const uint32_t dw = SPAN * b + 4 * ((piece ^ (row / (64 / SPAN))) & (kPieces - 1)) + d;
                const uint32_t at = 4 * (dw < last_dw ? dw : last_dw);               // past K: never used
                return of_w ? (T)wrow_of(row) * p.ld_ws + at : (T)arow_of(row - TW) * p.ld_as + at;
            };
            constexpr uint32_t kWPieces = TW * kPieces;                              // the weights' come first; a load has one kind
            if (whole_pieces) {
#pragma unroll
                for (int i = 0; i < kScaleLoads; ++i) {
                    const uint32_t p0 = min((uint32_t)(NW * i + wave) * 64, (uint32_t)kAllPieces - 64);          // (a duplicate at most)
                    const bool of_w = p0 < kWPieces;
                    ring_dma16(lds0 + half_at + p0 * 16, address(uint32_t{}, p0 + lane, 0, of_w), of_w ? ws_rs : as_rs, 0);
                }
            } else {
                // rows at any byte, of less than a piece, or further apart than 32 bits reach: through registers (the waits for them drain the ring, once in SPAN slabs)
#pragma unroll 2
                for (int i = 0; i < 4 * kScaleLoads; ++i) {
                    const uint32_t p0 = min((uint32_t)(NW * i + wave) * 16, (uint32_t)kAllPieces - 16);
                    const bool of_w = p0 < kWPieces;
                    uint32_t v;
                    __builtin_memcpy(&v, (of_w ? w_scales : a_scales) + address(size_t{}, p0 + lane / 4, lane & 3u, of_w), 4);
                    *reinterpret_cast<uint32_t*>(smem + half_at + p0 * 16 + lane * 4) = v;
                }
            }
        }
    };

    // ---- fragments -------------------------------------------------------------------------------------------------------
    auto wfrag_row = [&](int f) -> uint32_t {
        if (epi_pairs_gate_up(EPI))
            return f < FW / 2 ? ww * (TW / 2 / WW) + f * 32 : TW / 2 + ww * (TW / 2 / WW) + (f - FW / 2) * 32;
        return ww * (TW / WW) + f * 32;
    };
    auto read_frag = [&](const uint8_t* tile, uint32_t r, int h) -> v8i {
        const uint8_t* rp = tile + r * kSlabBytes;
        const v4i lo = *reinterpret_cast<const v4i*>(rp + swz(r, h * 4 + lh) * 16);
        const v4i hi = *reinterpret_cast<const v4i*>(rp + swz(r, h * 4 + lh + 2) * 16);
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    // K-slow: four transposing reads; lanes 16 i .. 16 i + 15 read eight K rows x 16 columns, two lanes to a row, and lane j of
    // them gets the eight K values of column j
    typedef __attribute__((address_space(3))) v2i* lds_v2i;
    auto read_frag_t = [&](uint32_t slot_lds, uint32_t col, int h) -> v8i {
        const uint32_t c = col + (lane & 16u), half_base = (c >> 7) * (128 * kSlabBytes), chunk = (c & 127u) >> 4;
        v8i r;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t k = 64 * h + 32 * (j >> 1) + 16 * lh + 8 * (j & 1) + ((lane & 15u) >> 1);
            const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(uintptr_t)(slot_lds + half_base + k * kSlabBytes + swz(k, chunk) * 16 + (lane & 1u) * 8));
            r[2 * j] = v[0];
            r[2 * j + 1] = v[1];
        }
        return r;
    };

    v16f acc[FW][FM];
#pragma unroll
    for (int i = 0; i < FW; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    v8i wf[2][FW], af[2][FM];
    uint32_t sw[FW][kSD] = {}, sa[FM][kSD] = {}, swn[FW][kSD] = {}, san[FM][kSD] = {};

    const uint32_t a_row = wm * (TM / WM) + l32;                         // activation row of fragment 0
    // fragment `pos` in the order of first use by the MFMAs (weights outside, activations inside): W0 A0 A1 .. W1 W2 ..
    auto read_one = [&](uint32_t slot, int h, int buf, int pos) {
        const uint8_t* st = smem + slot * kSlotBytes;
        const bool is_w = pos == 0 || pos > FM;
        const int f = pos == 0 ? 0 : (is_w ? pos - FM : pos - 1);
        if (!is_w) af[buf][f] = read_frag(st + TW * kSlabBytes, a_row + f * 32, h);
        else wf[buf][f] = KSLOW ? read_frag_t(lds0 + slot * kSlotBytes, wfrag_row(f), h) : read_frag(st, wfrag_row(f) + l32, h);
    };
    // scale dwords of slab s of fragment `pos` (0 .. FW - 1 weights, then activations), the lane's byte of MFMA j (FP4) or step h at bits 16
    const uint32_t sc_x = l32 * SPAN / 64 & (kPieces - 1);
    auto read_scale = [&](uint32_t s, int pos) {
        if constexpr (kScales) {
            const uint32_t d = kSD * s;
            const uint8_t* at = smem + kScaleBase + (s / kSpanSlabs & 1u) * kScaleHalf;
            const uint32_t in_piece = whole_pieces && d >= (ndw & ~3u) ? d - last_dw : d % 4;
            const uint32_t in_row = ((d % SPAN / 4) ^ sc_x) * 16 + in_piece * 4;
            if constexpr (KSLOW) {
                if (pos < FW) {
                    const uint8_t* q = at + s % SPAN * (4 * TW) + (wfrag_row(pos) + l32) * 2 + lh;
                    swn[pos][0] = q[0] | ((uint32_t)q[2 * TW] << 16);
                    return;
                }
            }
#pragma unroll
            for (int j = 0; j < kSD; ++j) {
                if (pos >= FW) san[pos - FW][j] = *reinterpret_cast<const uint32_t*>(at + TW * 4 * SPAN + in_row + 4 * j + (a_row + (pos - FW) * 32) * (4 * SPAN));
                else swn[pos][j] = *reinterpret_cast<const uint32_t*>(at + in_row + 4 * j + (wfrag_row(pos) + l32) * (4 * SPAN));
            }
        }
    };
    auto take_scales = [&]() {
#pragma unroll
        for (int j = 0; j < kSD; ++j) {
#pragma unroll
            for (int f = 0; f < FW; ++f) sw[f][j] = KSLOW ? swn[f][j] : swn[f][j] >> (8 * lh);
#pragma unroll
            for (int f = 0; f < FM; ++f) sa[f][j] = san[f][j] >> (8 * lh);
        }
    };

    // ---- K loop ----------------------------------------------------------------------------------------------------------
#pragma unroll
    for (int d = 0; d < NSLOT; ++d) {
#pragma unroll
        for (int i = 0; i < (d + 1 < NSLOT ? kTileLoads : kEarly); ++i) issue_one(d, d, i);
        if (d == 0) load_scales(0);
    }
    ring_wait_barrier<(NSLOT - 2) * kTileLoads + kEarly>();
#pragma unroll
    for (int i = 0; i < kFrags; ++i) {
        read_one(0, 0, 0, i);
        read_scale(0, i);
    }
    take_scales();
    // One MFMA, then its share of what the step has to issue: with one or two wavefronts per SIMD the matrix pipe stays busy only
    // if the LDS reads and the loads stand between the MFMAs, where the compiler by itself puts all of them in front.
    auto step = [&](auto hc, auto&& items, auto n_items) {
        constexpr int h = decltype(hc)::value, n = decltype(n_items)::value;
#pragma unroll
        for (int x = 0; x < kSteps; ++x) {
            const int i = x % kM / FM, j = x % FM;
            if (x < kM) acc[i][j] = ring_mfma<FMT, h, 0>(wf[h][i], af[h][j], acc[i][j], sw[i], sa[j]);
            else acc[i][j] = ring_mfma<FMT, h, 1>(wf[h][i], af[h][j], acc[i][j], sw[i], sa[j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int it = x * n / kSteps; it < (x + 1) * n / kSteps; ++it) items(it);
            __builtin_amdgcn_sched_barrier(0);
        }
        // (the sums are used here: otherwise the MFMAs sink below the barrier that follows)
#pragma unroll
        for (int x = 0; x < kM; ++x) asm volatile("" ::"a"(acc[x / FM][x % FM]));
    };
    using c0 = std::integral_constant<int, 0>;
    using c1 = std::integral_constant<int, 1>;
    uint32_t slot = 0, prev = NSLOT - 1;
    for (uint32_t s = 0; s < nslab; ++s) {
        step(c0{}, [&](int it) {
            if (it < kFrags) read_one(slot, 1, 1, it);
            else issue_one(s + NSLOT - 1, prev, kEarly + it - kFrags);
        }, std::integral_constant<int, kFrags + kTileLoads - kEarly>{});
        // every fragment of slab s has been read (by all) and slab s + 1 has arrived (for all): its slot takes slab s + NSLOT
        ring_wait_barrier<(NSLOT - 2) * kTileLoads>();
        __builtin_amdgcn_sched_barrier(0);
        // block 1 of the scales behind the first slab; block b + 2 behind the last slab of block b, whose scales were read a slab
        // ago by all
        if constexpr (kScales)
            if ((s == 0 && nslab > kSpanSlabs) || (s % kSpanSlabs == kSpanSlabs - 1 && s + kSpanSlabs + 1 < nslab)) load_scales(s == 0 ? 1 : s / kSpanSlabs + 2);
        const uint32_t next = slot + 1 < NSLOT ? slot + 1 : 0;
        step(c1{}, [&](int it) {
            if (it < kFrags) { read_one(next, 0, 0, it); read_scale(s + 1, it); }
            else issue_one(s + NSLOT, slot, it - kFrags);
        }, std::integral_constant<int, kFrags + kEarly>{});
        take_scales();
        prev = slot;
        slot = next;
    }
    ring_wait_barrier<0>();                                              // the loads past the end, before the LDS changes hands

    // ---- epilogue: sums through the LDS, whole rows to memory ----------------------------------------------------------------
    constexpr uint32_t kPitch = TW + 4;
    float* const sums = reinterpret_cast<float*>(smem);
    constexpr uint32_t kQuads = epi_pairs_gate_up(EPI) ? TW / 8 : TW / 4;
    // INT8: a thread keeps its columns from row to row, so their scales and those of its rows are requested once and up front.  Between
    // the stores, which the compiler cannot tell from them, every row would wait for nine loads of its own (256 x 128 tiles, us: 32 groups x 90
    // rows, K = 128, N = 1024, one round, 16.6 -> 10.3; 256 x 48, four rounds, 43.2 -> 31.8, at K = 1024 81.1 -> 70.6).
    constexpr int kTurns = EPI == kEpiI8DequantSwiglu ? TM * kQuads / NT : 1;
    static_assert(NT % kQuads == 0 && TM * kQuads % NT == 0, "whole rows a turn");
    v4f i8_g, i8_u;
    float i8_t[kTurns];
    if constexpr (EPI == kEpiI8DequantSwiglu) {
        const uint32_t ncol = tc.wt * (TW / 2) + 4 * (tid % kQuads);
        load_channel_scales(p, tc.g, ncol < half ? ncol : half - 4, i8_g, i8_u);
#pragma unroll
        for (int i = 0; i < kTurns; ++i) i8_t[i] = reinterpret_cast<const float*>(p.a_scale)[tc.row0 + arow_of((i * NT + tid) / kQuads)];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int i = 0; i < FW; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<v4f*>(sums + (wm * (TM / WM) + j * 32 + l32) * kPitch + wfrag_row(i) + 8 * q + 4 * lh) = to_v4(acc[i][j], q);
    __syncthreads();
    if constexpr (EPI == kEpiI8DequantSwiglu) {
        const uint32_t q = tid % kQuads, ncol = tc.wt * (TW / 2) + 4 * q;
#pragma unroll
        for (int i = 0; i < kTurns; ++i) {
            const uint32_t m = (i * NT + tid) / kQuads;
            if (m >= tc.rows_valid || ncol >= half) continue;
            store_i8_quad(p, (size_t)(tc.row0 + m), ncol, *reinterpret_cast<const v4f*>(sums + m * kPitch + 4 * q),
                          *reinterpret_cast<const v4f*>(sums + m * kPitch + TW / 2 + 4 * q), i8_g, i8_u, i8_t[i]);
        }
        return;
    }
    if constexpr (EPI == kEpiStore) {
        if (stores_pieces(p)) {
            // A thread keeps its eight columns from row to row, so that a piece costs two LDS reads, four conversions and a store: with one
            // wavefront per SIMD the general loop below is bound by its instructions (1024 x 4096, 2.5 us of it;
            // at K = 1024, quantizer and matmul 14.5 -> 12.8 us).
            constexpr uint32_t kPieces8 = TW / 8, kTurn = NT / kPieces8;
            static_assert(NT % kPieces8 == 0 && TM % kTurn == 0, "whole rows a turn");
            const uint32_t q = tid % kPieces8, m0 = tid / kPieces8;
            uint32_t ncol = tc.wt * TW + 8 * q;
            if constexpr (KSLOW) ncol = ncol / 16 * 16 < p.n ? wcol_of(q / 2) + 8 * (q % 2) : p.n;
            if (ncol >= p.n) return;
            auto store_rows = [&](auto out_c) {
                uint16_t* o = reinterpret_cast<uint16_t*>(p.c) + (size_t)(tc.row0 + m0) * p.ldc + ncol;
#pragma unroll
                for (uint32_t i = 0; i < TM / kTurn; ++i) {
                    const float* const s = sums + (m0 + i * kTurn) * kPitch + 8 * q;
                    const uint4 v = pack_piece<decltype(out_c)::value>(*reinterpret_cast<const v4f*>(s), *reinterpret_cast<const v4f*>(s + 4));
                    if (m0 + i * kTurn < tc.rows_valid) *reinterpret_cast<uint4*>(o) = v;
                    o += (size_t)kTurn * p.ldc;
                }
            };
            if (p.out_type == CMX_OUT_BF16) store_rows(std::integral_constant<int, CMX_OUT_BF16>{});
            else store_rows(std::integral_constant<int, CMX_OUT_FP16>{});
            return;
        }
    }
    if constexpr (epi_is_swiglu_quant(EPI)) {
        // The same: eight activation columns of a thread, its rows one after the other.
        constexpr uint32_t kPieces8 = TW / 16, kTurn = NT / kPieces8;
        static_assert(NT % kPieces8 == 0 && TM % kTurn == 0, "whole rows a turn");
        const uint32_t q = tid % kPieces8, m0 = tid / kPieces8;
        const uint32_t ncol = tc.wt * (TW / 2) + 8 * q, blk = ncol / 32, blocks = half / 32;
        const bool aligned8 = p.ld_act % 8 == 0 && (reinterpret_cast<uintptr_t>(p.act_codes) & 7u) == 0;
#pragma unroll 2
        for (uint32_t i = 0; i < TM / kTurn; ++i) {
            const uint32_t m = m0 + i * kTurn;
            const float* const s = sums + m * kPitch + 8 * q;
            const v4f g[2] = {*reinterpret_cast<const v4f*>(s), *reinterpret_cast<const v4f*>(s + 4)};
            const v4f u[2] = {*reinterpret_cast<const v4f*>(s + TW / 2), *reinterpret_cast<const v4f*>(s + TW / 2 + 4)};
            uint32_t pk[4];
            uint2 codes;
            const int e = swiglu_quant_piece(g, u, pk, codes);                       // (all lanes: they hold the blocks together)
            if (m >= tc.rows_valid || ncol >= half) continue;                        // n is a multiple of 64: a block is in or out as a whole
            const size_t mrow = tc.row0 + m;
            if constexpr (EPI == kEpiSwigluQuantAct) {
                if (p.act_bf16) {
                    uint16_t* const o = p.act_bf16 + mrow * half + ncol;
#pragma unroll
                    for (int j = 0; j < 8; ++j) o[j] = (uint16_t)(pk[j >> 1] >> (16 * (j & 1)));
                }
            }
            uint8_t* const o = p.act_codes + mrow * p.ld_act + ncol;
            if (aligned8) {
                *reinterpret_cast<uint2*>(o) = codes;
            } else {
                *reinterpret_cast<uint32_t*>(o) = codes.x;
                *reinterpret_cast<uint32_t*>(o + 4) = codes.y;
            }
            if (q % 4 == 0) {
                uint8_t* const srow = p.act_scales + mrow * p.ld_acts;
                srow[blk] = (uint8_t)(e + 127);
                if (blk == blocks - 1 && (blocks & 1u)) srow[blocks] = 127;
            }
        }
        return;
    }
#pragma unroll 4
    for (uint32_t it = tid; it < TM * kQuads; it += NT) {
        const uint32_t m = it / kQuads, q = it % kQuads;
        if (m >= tc.rows_valid) continue;
        const v4f v = *reinterpret_cast<const v4f*>(sums + m * kPitch + 4 * q), u = v;
        uint32_t ncol = tc.wt * TW + 4 * q;
        if constexpr (KSLOW) {
            const uint32_t col = tc.wt * TW + 16 * (q / 4);
            ncol = col < p.n ? wcol_of(q / 4) + 4 * (q % 4) : p.n;
        }
        store_quad<EPI>(p, tc, m, ncol, v, u);
    }
}

}  // namespace

}  // namespace cmx
