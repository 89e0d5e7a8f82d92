// Block-scaled (and INT8) matmul for problems with few activation rows or few tiles: split over K inside the workgroup.
//
// A problem of a few rows reads every weight byte once and multiplies it a handful of times: what counts is how many
// bytes are in flight on how many CUs, and tiles of 256 weight rows leave most of the chip without work (16 x 4096 x 7168:
// sixteen workgroups).  Here a workgroup owns a small tile, 16 FW weight rows x 16 FM activation rows, and its NW wavefronts
// split K between them: wavefront w multiplies the 128-byte K slabs w, w + NW, w + 2 NW, ... of the WHOLE tile, so
//   * every operand byte of the tile is needed by exactly one wavefront: both operands go straight from memory into that
//     wavefront's registers (buffer_load_dwordx4) through a ring of PD slabs (eight for a tile of 16 x 16, one for a full 64 x
//     64: what the registers hold), with no barrier and no wait for another wavefront in the K loop;
//   * v_mfma_scale_f32_16x16x128_f8f6f4 takes, per lane group g = lane / 16, the bytes 16 g .. 16 g + 15 of a slab's first
//     64 bytes in registers 0-3 and of its second 64 bytes in registers 4-7 (and the scale of the 32-block g), for the
//     row lane % 16.  Loading row-major operands in that order costs the vector cache a visit per lane quad and row, a third
//     more time than whole 128-byte lines (16 x 4096 x 7168, operands in the memory-side cache: 9.7 against 7.2 us), so the lanes
//     fetch whole lines, eight to a row, and a fragment changes places through 2 KiB of LDS that belong to the wavefront alone
//     (its LDS accesses execute in order: nothing to wait for).  Pre-tiled weights are stored in the fragment order and need none of it;
//   * weights stored [K, N] (kKSlow) are fetched as they lie, 64 columns of 128 K positions a slab, and turned on the way out of the
//     exchange by ds_read_b64_tr_b8.  A K row of the tile is half a line, so the vector cache serves 128 + 16 FM visits a slab instead
//     of 64 + 16 FM and bounds the kernel (16 x 4096 x 7168: 64 workgroups, 19 us, where K-contiguous weights take 9.3 on 256); a pass that
//     rewrites the weights first brings that to 26;
//   * the block scales of the tile, which are a byte per 32 elements in rows of their own, are fetched once, coalesced, for
//     the whole of K into the LDS and read from there a byte per lane and fragment.
// The NW partial sums meet in the LDS at the end and are added in the order of the wavefronts, so the result does not
// depend on timing; it does depend on NW, and where the fp32 additions round it differs in the last bits from that of the
// kernels that walk K in one chain.  (The error against 64-bit sums is the same on both: 6.3e-5 to 6.7e-5 of the 2-norm at K = 512 to
// 7168, E4M3, normal data with outliers; it comes from the matrix cores, which keep 2^-13 of the largest of eight products.)
// Every tile shape with the same NW gives the same bits, and so do row-major and pre-tiled weights.
#include <type_traits>

#include "mx_gemm_ksplit.h"
#include "mx_gemm_store.h"
#include "mx_launch.h"

namespace cmx {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// how the weights lie in memory: rows of K; tiled by cmx_mx_pretile_weights; rows of N (K the slow axis)
enum WeightLayout { kRowMajor = 0, kTiled = 1, kKSlow = 2 };

constexpr int ks_scale_steps(int fmt) { return fmt == kFmtI8 ? 0 : (fmt == CMX_FMT_E2M1 ? 2 : 1); }   // scale dwords per row and slab
// slabs in the register ring: what fits beside the accumulators, a slab on its way through the exchange, their scales and
// addresses in 256 registers (two wavefronts per SIMD).  (Fragments change places in the registers that they have, but rings that count on all
// of that room spill 30 registers: FP4, 32 experts x 16 rows 90 -> 104 us.)  The scale pieces in flight before the K loop (sreg, treg: up to 32
// registers at 8 wavefronts) are not counted; by the compiler's report they cost 16 x 16 tiles 3-4 spilled registers and 16 x 32
// tiles 7 (FP4 12), stored and reloaded before the loop, and no other tile more than one.
constexpr int ks_ring(int fmt, int fw, int fm) {
    const int room = 256 - 40 - 4 * fw * fm - (fw + fm) * (10 + 2 * ks_scale_steps(fmt));
    const int n = room / ((fw + fm) * 8), most = fw + fm == 2 ? 8 : (fw + fm == 3 ? 5 : 4);
    return n < 1 ? 1 : (n > most ? most : n);
}
// activation rows whose partial sums go through the LDS at a time: all of them where the workgroup is alone on its CU (eight
// wavefronts) or where two still fit (1000 x 1000 x 960: four passes of 16 rows, half of the threads idle, took 2.7 us, one 2.5)
constexpr int ks_pass_frags(int fw, int fm, int nw) {
    int n = fm;
    while (n > 1 && nw * n * 16 * (16 * fw + 4) * 4 > (nw == 8 ? 140 : 70) * 1024) n /= 2;
    return n;
}
// exchange buffers of a wavefront (2 KiB, one fragment): four, used in turn; K-slow weights change places a whole slab at a time, in
// four more, and leave two to the activations
constexpr int ks_exchange_bufs(int fw, int fm, int layout) {
    if (layout == kKSlow) return fw + (fm < 2 ? fm : 2);
    const int n = (layout == kTiled ? 0 : fw) + fm;
    return n < 4 ? n : 4;
}
constexpr size_t ks_sum_bytes(int fw, int fm, int nw) { return (size_t)nw * ks_pass_frags(fw, fm, nw) * 16 * (16 * fw + 4) * 4; }
// dwords of a scale row in the LDS: whole slabs, an odd count so that the sixteen rows of a fragment lie in different banks
__host__ __device__ inline uint32_t ks_scale_pitch(int fmt, uint32_t kblocks) {
    const uint32_t per = fmt == CMX_FMT_E2M1 ? 8 : 4;
    return ((kblocks + per - 1) / per * per / 4) | 1u;
}

// acc += W-fragment x A-fragment over one 128-byte slab
template <int FMT>
__device__ __forceinline__ v4f ks_mfma(const v4i (&w)[2], const v4i (&a)[2], v4f c, const uint32_t (&sw)[2], const uint32_t (&sa)[2]) {
    if constexpr (FMT == kFmtI8) {
        v4i acc = __builtin_bit_cast(v4i, c);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[0], a[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[1], a[1], acc, 0, 0, 0);
        return __builtin_bit_cast(v4f, acc);
    } else if constexpr (FMT == CMX_FMT_E2M1) {
        const v8i w0 = {w[0][0], w[0][1], w[0][2], w[0][3], 0, 0, 0, 0}, w1 = {w[1][0], w[1][1], w[1][2], w[1][3], 0, 0, 0, 0};
        const v8i a0 = {a[0][0], a[0][1], a[0][2], a[0][3], 0, 0, 0, 0}, a1 = {a[1][0], a[1][1], a[1][2], a[1][3], 0, 0, 0, 0};
        c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w0, a0, c, 4, 4, 0, (int)sw[0], 0, (int)sa[0]);
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w1, a1, c, 4, 4, 0, (int)sw[1], 0, (int)sa[1]);
    } else {
        constexpr int kF = FMT == CMX_FMT_E5M2 ? 1 : 0;
        const v8i w8 = {w[0][0], w[0][1], w[0][2], w[0][3], w[1][0], w[1][1], w[1][2], w[1][3]};
        const v8i a8 = {a[0][0], a[0][1], a[0][2], a[0][3], a[1][0], a[1][1], a[1][2], a[1][3]};
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w8, a8, c, kF, kF, 0, (int)sw[0], 0, (int)sa[0]);
    }
}

// STREAM: weights are loaded non-temporal (KsplitWeights); PD: slabs in the ring
template <int FMT, int FW, int FM, int NW, int EPI, int LAYOUT, bool STREAM, int PD = ks_ring(FMT, FW, FM)>
__device__ __forceinline__ void ks_tile(const GemmParams& p, const Tile& tc, uint8_t* smem) {
    constexpr int NT = 64 * NW, TW = 16 * FW;
    constexpr int kS = ks_scale_steps(FMT);
    constexpr int kSA = kS ? kS : 1;
    constexpr bool TILED = LAYOUT == kTiled, KSLOW = LAYOUT == kKSlow;
    constexpr int kScaleW = KSLOW ? 0 : TW, kRows = kScaleW + 16 * FM;            // rows of scales: weights (unless K-slow), activations
    static_assert(!KSLOW || (FW == 4 && kS == 1 && EPI == kEpiStore), "K-slow weights: 64 columns, 8-bit formats");
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;
    const uint32_t half = p.n >> 1;
    static_assert(!epi_is_swiglu_quant(EPI) || TW / 2 % 32 == 0, "whole MX blocks in a tile");

    // global weight row of tile row t (rows past the matrix repeat the last one; masked at the store)
    auto wrow_of = [&](uint32_t t) -> uint32_t {
        if (epi_pairs_gate_up(EPI)) {
            uint32_t rr = tc.wt * (TW / 2) + (t < TW / 2 ? t : t - TW / 2);
            rr = rr < half ? rr : half - 1;
            return t < TW / 2 ? rr : half + rr;
        }
        const uint32_t gr = tc.wt * TW + t;
        return gr < p.n ? gr : p.n - 1;
    };
    auto arow_of = [&](uint32_t t) -> uint32_t { return t < tc.rows_valid ? t : tc.rows_valid - 1; };

    // K-slow: first column of the tile's 16-column chunk c; one that the matrix ends inside of is moved back to end with it, one past
    // the end repeats the last
    auto wcol_of = [&](uint32_t c) -> uint32_t {
        const uint32_t col = tc.wt * TW + 16 * c;
        return col + 16 <= p.n ? col : p.n - 16;
    };

    // ---- scales of the tile: request -----------------------------------------------------------------------------------
    const uint32_t pitch = ks_scale_pitch(FMT, p.kblocks);
    uint32_t* const s_sc = reinterpret_cast<uint32_t*>(smem);
    auto scale_row = [&](uint32_t t) -> const uint8_t* {
        return t < (uint32_t)kScaleW ? p.w_scale + ((size_t)tc.g * p.n + wrow_of(t)) * p.ld_ws
                                     : p.a_scale + (size_t)(tc.row0 + arow_of(t - kScaleW)) * p.ld_as;
    };
    // Whole 16-byte pieces, numbered with the next power of two of pieces per row (no division), and behind them the up to
    // 15 bytes of a row that is no whole number of pieces as four dwords (none reaches past the row: the last is read from its
    // last four bytes and shifted; a last slab in part is filled up with 1.0).  Rows start at any byte (the pitch of 30 scales is 30): the pieces are read by unaligned loads.  All of it is
    // requested before the operands and deposited behind their requests: one trip to memory.  (A dword at a time, each
    // waited for, it was most of the kernel where K is no multiple of 512: see the rule's comment in mx_gemm.hip.)
    constexpr int kBatch = 2048 / NT;                  // pieces per thread in flight together: 32 KiB per workgroup
    constexpr int kTail = (kRows * 4 + NT - 1) / NT;
    const uint32_t pieces = p.kblocks / 16, shift = pieces > 1 ? 32 - __builtin_clz(pieces - 1) : 0;
    const uint32_t total16 = kRows << shift;
    const bool ragged = p.kblocks % 16 != 0;
    u32x4 sreg[kBatch];
    uint32_t treg[kTail];
    auto request16 = [&](uint32_t i0) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const uint32_t i = i0 + b * NT + tid, t = i >> shift, q = i & ((1u << shift) - 1);
            if (i < total16 && q < pieces) __builtin_memcpy(&sreg[b], scale_row(t) + q * 16, 16);
        }
    };
    auto deposit16 = [&](uint32_t i0) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const uint32_t i = i0 + b * NT + tid, t = i >> shift, q = i & ((1u << shift) - 1);
            if (i < total16 && q < pieces) {
                uint32_t* d = s_sc + t * pitch + q * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = sreg[b][e];
            }
        }
    };
    // K-slow weights: pairs of scales [K / 64][64 columns] behind the rows, in pieces of eight columns
    uint8_t* const s_pairs = smem + kRows * pitch * 4 + ((0u - kRows * pitch * 4) & 15u);
    const uint32_t pair_pieces = KSLOW ? p.kblocks / 2 * 8 : 0;
    constexpr int kPairBatch = KSLOW ? 1024 / NT : 1;          // K = 8192 in flight together
    u32x4 preg[kPairBatch];
    auto request_pairs = [&](uint32_t i0) {
#pragma unroll
        for (int b = 0; b < kPairBatch; ++b) {
            const uint32_t i = i0 + b * NT + tid;
            if (i < pair_pieces) __builtin_memcpy(&preg[b], p.w_scale + (size_t)(i / 8) * p.ld_ws + 2 * (wcol_of(i % 8 / 2) + i % 2 * 8), 16);
        }
    };
    auto deposit_pairs = [&](uint32_t i0) {
#pragma unroll
        for (int b = 0; b < kPairBatch; ++b) {
            const uint32_t i = i0 + b * NT + tid;
            if (i < pair_pieces) *reinterpret_cast<u32x4*>(s_pairs + i * 16) = preg[b];
        }
    };
    if constexpr (KSLOW) request_pairs(0);
    if constexpr (kS != 0) {
        request16(0);
        if (ragged && p.kblocks >= 4) {
#pragma unroll
            for (int b = 0; b < kTail; ++b) {
                const uint32_t i = b * NT + tid, at = 16 * pieces + 4 * (i & 3u);
                if (i < kRows * 4) __builtin_memcpy(&treg[b], scale_row(i >> 2) + min(at, p.kblocks - 4), 4);
            }
        }
    }

    // ---- operand streams ---------------------------------------------------------------------------------------------
    constexpr int kRsrcFlags = 0x00020000;
    auto uniform_ptr = [](const uint8_t* q) -> uint8_t* {
        const uint64_t v = reinterpret_cast<uint64_t>(q);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return reinterpret_cast<uint8_t*>(((uint64_t)hi << 32) | lo);
    };
    const uint8_t* wbase;
    // row-major: load h of a fragment covers its rows 8 h .. 8 h + 7, lane -> row lane / 8, 16-byte chunk lane % 8
    const uint32_t x_row = lane >> 3, x_chunk = lane & 7u;
    uint32_t woff[FW][2], aoff[FM][2];
    if constexpr (TILED) {
        // [256-row tile][slab][wavefront block][step 0/1][fragment][half][lane half][32 rows][16 bytes]: the bytes
        // 64 j + 16 g of a row's slab lie in step j, half g / 2, lane half g % 2
        constexpr bool kPair = epi_pairs_gate_up(EPI);
        const uint32_t row0 = kPair ? tc.wt * (TW / 2) : tc.wt * TW;
        const uint32_t big = kPair ? row0 / 128 : row0 / 256;
        const uint32_t w256 = kPair ? (half + 127) / 128 : (p.n + 255) / 256;
        wbase = p.w + ((size_t)tc.g * w256 + big) * ((size_t)p.kbytes * 256);
#pragma unroll
        for (int f = 0; f < FW; ++f) {
            uint32_t blk, frag, row;
            if (kPair) {
                const uint32_t q = (row0 + (f < FW / 2 ? f : f - FW / 2) * 16 + r) % 128;
                blk = q / 32; frag = f < FW / 2 ? 0 : 1; row = q % 32;
            } else {
                const uint32_t q = (row0 + f * 16 + r) % 256;
                blk = q / 64; frag = q / 32 % 2; row = q % 32;
            }
            woff[f][0] = blk * 8192 + frag * 2048 + (g >> 1) * 1024 + (g & 1u) * 512 + row * 16;
            woff[f][1] = woff[f][0] + 4096;
        }
    } else if constexpr (KSLOW) {
        // load 2 f + h: 16 K rows of 64 bytes, lane -> row lane / 4, columns 16 (lane % 4) ..
        wbase = p.w;
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h) woff[f][h] = (32 * f + 16 * h + (lane >> 2)) * p.ldw + wcol_of(lane & 3u);
    } else {
        wbase = p.w + (size_t)tc.g * p.n * p.ldw;
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h) woff[f][h] = wrow_of(f * 16 + 8 * h + x_row) * p.ldw + x_chunk * 16;
    }
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int h = 0; h < 2; ++h) aoff[f][h] = arow_of(f * 16 + 8 * h + x_row) * p.lda + x_chunk * 16;
    const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(wbase), 0, -1, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t a_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p.a + (size_t)tc.row0 * p.lda), 0, -1, kRsrcFlags);
    const uint32_t kWSlab = TILED ? 256 * kSlabBytes : (KSLOW ? kSlabBytes * p.ldw : kSlabBytes);
    constexpr int kWAux = STREAM ? 2 : 0;              // 2: non-temporal

    v4i wf[PD][FW][2], af[PD][FM][2];
    // Slab s of this wavefront into ring slot d; past the last slab every lane re-reads the operand's first bytes (one line,
    // never used), so that the number of loads in flight does not depend on the length of K.
    const uint32_t nslab = p.kbytes / kSlabBytes;
    auto load_slot = [&](int d, uint32_t s) {
        const bool in = s < nslab;
        const uint32_t mask = in ? ~0u : 0u, sw = in ? s * kWSlab : 0u, sa = in ? s * kSlabBytes : 0u;
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                wf[d][f][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w_rs, (int)(woff[f][h] & mask), (int)sw, kWAux));
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                af[d][f][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(a_rs, (int)(aoff[f][h] & mask), (int)sa, 0));
    };
#pragma unroll
    for (int d = 0; d < PD; ++d) load_slot(d, wave + NW * d);

    // ---- scales of the tile: deposit -----------------------------------------------------------------------------------
    if constexpr (KSLOW) {
        deposit_pairs(0);
        for (uint32_t i0 = kPairBatch * NT; i0 < pair_pieces; i0 += kPairBatch * NT) {
            request_pairs(i0);
            deposit_pairs(i0);
        }
    }
    if constexpr (kS != 0) {
        deposit16(0);
        if (ragged) {
#pragma unroll
            for (int b = 0; b < kTail; ++b) {
                const uint32_t i = b * NT + tid, q = 4 * pieces + (i & 3u);
                if (i >= kRows * 4 || q >= pitch) continue;
                uint32_t v = 0x7F7F7F7Fu;
                if (p.kblocks >= 4) {
                    const uint32_t past = 4 * q - min(4 * q, p.kblocks - 4);          // bytes of the dword past the row
                    if (past == 0) v = treg[b];
                    else if (past < 4) v = (treg[b] >> (8 * past)) | (v << (32 - 8 * past));
                } else {
                    const uint8_t* row = scale_row(i >> 2);
                    for (uint32_t e = 0; 4 * q + e < p.kblocks; ++e) v = (v & ~(0xFFu << (8 * e))) | ((uint32_t)row[e] << (8 * e));
                }
                s_sc[(i >> 2) * pitch + q] = v;
            }
        }
        for (uint32_t i0 = kBatch * NT; i0 < total16; i0 += kBatch * NT) {
            request16(i0);
            deposit16(i0);
        }
    }
    const uint8_t* const sw_row = smem + r * pitch * 4 + g;
    const uint8_t* const sa_row = smem + (kScaleW + r) * pitch * 4 + g;
    const uint8_t* const sp_col = s_pairs + (g >> 1) * 128 + r * 2 + (g & 1u);

    v4f acc[FW][FM];
#pragma unroll
    for (int i = 0; i < FW; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

    // a fragment from the order of the loads (rows 8 h + lane / 8, chunk lane % 8) to that of the MFMA (row lane % 16, chunks
    // lane / 16 and 4 + lane / 16); chunks XOR-swizzled by row: neither side meets bank conflicts
    constexpr int kBufs = ks_exchange_bufs(FW, FM, LAYOUT), kWBufs = KSLOW ? FW : 0;
    uint8_t* const xbuf = (kS ? s_pairs : smem) + pair_pieces * 16 + wave * (kBufs * 2048);
    uint32_t xw[2], xr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        xw[h] = (8 * h + x_row) * 128 + swz(8 * h + x_row, x_chunk) * 16;
        xr[h] = r * 128 + swz(r, 4 * h + g) * 16;
        // A lane loads what other lanes stored.  The LDS executes a wavefront's accesses in order; that the compiler issues them in
        // order rests on a store and a load that may be to one address, and the empty asm keeps it from ever knowing better.
        // (A fence of wavefront scope orders the operand loads as well: 256 experts x 8 rows, E4M3, 1080 -> 1139 us.  The asm costs
        // nothing, and without expressions to rebuild the offsets from the compiler spills less: FP4, 32 experts x 16 rows 98 -> 87.)
        asm("" : "+v"(xw[h]), "+v"(xr[h]));
    }
    auto exchange = [&](int buf, const v4i (&in)[2], v4i (&out)[2]) {
        uint8_t* const b = xbuf + (kWBufs + buf % (kBufs - kWBufs)) * 2048;
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<v4i*>(b + xw[h]) = in[h];
#pragma unroll
        for (int h = 0; h < 2; ++h) out[h] = *reinterpret_cast<const v4i*>(b + xr[h]);
    };
    // K-slow: a slab as [128 K][64 columns], the 16-column pieces of a row XOR-swizzled; a fragment (column lane % 16, K 16 (lane / 16) ..
    // and 64 + 16 (lane / 16) ..) by four transposing reads: lanes 16 i .. 16 i + 15 read eight K rows x 16 columns, two lanes to a row,
    // and each gets the eight K values of its column.  Neither side meets bank conflicts.
    auto kslow_piece = [](uint32_t k, uint32_t c) -> uint32_t { return k * 64 + (c ^ ((k >> 2 & 1u) | (k >> 3 & 2u))) * 16; };
    uint32_t kw = kslow_piece(lane >> 2, lane & 3u), kr[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) kr[j] = kslow_piece(16 * g + 8 * j + (r >> 1), 0) + (r & 1u) * 8;
    asm("" : "+v"(kw), "+v"(kr[0]), "+v"(kr[1]));                                // as for xw and xr
    typedef __attribute__((address_space(3))) v2i* lds_v2i;
    auto exchange_kslow = [&](const v4i (&in)[FW][2], v4i (&out)[FW][2]) {
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                // (rows 16 apart from load to load: the swizzle's second bit changes with h)
                *reinterpret_cast<v4i*>(xbuf + (2 * f + h) * 1024 + (kw ^ (h ? 32u : 0u))) = in[f][h];
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint8_t* at = xbuf + 4096 * h + (kr[j] ^ (16u * f));
                    const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)at);
                    out[f][h][2 * j] = v[0];
                    out[f][h][2 * j + 1] = v[1];
                }
    };
    // a slab from the order of the loads to that of the MFMA, in the registers that it has
    auto arrange = [&](v4i (&w)[FW][2], v4i (&a)[FM][2]) {
#pragma unroll
        for (int f = 0; f < FM; ++f) exchange(f, a[f], a[f]);
        if constexpr (KSLOW) exchange_kslow(w, w);
#pragma unroll
        for (int f = 0; f < FW && !KSLOW && !TILED; ++f) exchange(FM + f, w[f], w[f]);
    };
    auto multiply = [&](const v4i (&w)[FW][2], const v4i (&a)[FM][2], uint32_t s) {
        uint32_t sw[FW][2] = {}, sa[FM][2] = {};
#pragma unroll
        for (int j = 0; j < kS; ++j) {
#pragma unroll
            for (int f = 0; f < FW; ++f) sw[f][j] = KSLOW ? sp_col[s * 256 + f * 32] : sw_row[f * 16 * pitch * 4 + s * (4 * kSA) + 4 * j];
#pragma unroll
            for (int f = 0; f < FM; ++f) sa[f][j] = sa_row[f * 16 * pitch * 4 + s * (4 * kSA) + 4 * j];
        }
#pragma unroll
        for (int i = 0; i < FW; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = ks_mfma<FMT>(w[i], a[j], acc[i][j], sw[i], sa[j]);
    };

    // ---- K loop --------------------------------------------------------------------------------------------------------
    const uint32_t mine = nslab > wave ? (nslab - wave + NW - 1) / NW : 0u;          // slabs of this wavefront
    // Eight wavefronts, which are alone on their CU, arrange the slabs of the first turn while the scales are on their way: with the scales
    // in front, the exchange of all slabs (16 x 4096 x 7168: 1.5 us of LDS time) stood between the arrival of the last operands and the
    // first MFMA.  Quantizer included, us: 16 x 4096 x 7168 10.2 -> 9.3, 200 x 2048 x 4096 13.4 -> 12.4, 512 x 512 x 4096 11.5 -> 10.7, [K, N] 64 x
    // 4096 x 4096 15.0 -> 13.5.  Beside a second workgroup of four wavefronts nothing is gained (32 experts x 60 rows 87.1 against 88.3).
    constexpr bool kFirst = NW == 8;
#pragma unroll
    for (int d = 0; d < PD && kFirst; ++d)
        if ((uint32_t)d < mine) arrange(wf[d], af[d]);
    if constexpr (kS != 0) __syncthreads();
    uint32_t i = 0;
    for (; i + PD < mine; i += PD) {
#pragma unroll
        for (int d = 0; d < PD; ++d) {
            if (!kFirst || i != 0) arrange(wf[d], af[d]);
            multiply(wf[d], af[d], wave + NW * (i + d));
            load_slot(d, wave + NW * (i + PD + d));
        }
    }
#pragma unroll
    for (int d = 0; d < PD; ++d)
        if (i + d < mine) {
            if (!kFirst || i != 0) arrange(wf[d], af[d]);
            multiply(wf[d], af[d], wave + NW * (i + d));
        }
    // K not a whole number of slabs: the rest, zeros past K
    if constexpr (FMT != kFmtI8 && LAYOUT == kRowMajor) {
        if (p.kbytes % kSlabBytes != 0 && nslab % NW == wave) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool in = nslab * kSlabBytes + x_chunk * 16 < p.kbytes;        // K is whole 16-byte pieces
                const int kb = (int)(nslab * kSlabBytes);
#pragma unroll
                for (int f = 0; f < FW; ++f) {
                    wf[0][f][h] = (v4i){0, 0, 0, 0};
                    if (in) wf[0][f][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w_rs, (int)woff[f][h], kb, 0));
                }
#pragma unroll
                for (int f = 0; f < FM; ++f) {
                    af[0][f][h] = (v4i){0, 0, 0, 0};
                    if (in) af[0][f][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(a_rs, (int)aoff[f][h], kb, 0));
                }
            }
            arrange(wf[0], af[0]);
            multiply(wf[0], af[0], nslab);
        }
    }

    // ---- sum over the wavefronts, epilogue ------------------------------------------------------------------------------
    // partial sums as [wavefront][row][column] with four floats between the rows
    constexpr int kPass = ks_pass_frags(FW, FM, NW);
    constexpr uint32_t kRowPitch = TW + 4, kPart = kPass * 16 * kRowPitch;
    float* const sums = reinterpret_cast<float*>(smem);
    constexpr uint32_t kQuads = epi_pairs_gate_up(EPI) ? TW / 8 : TW / 4;            // columns are written in fours
#pragma unroll
    for (int f0 = 0; f0 < FM; f0 += kPass) {
        __syncthreads();                                                             // the scales (or the last pass's sums) have been read
#pragma unroll
        for (int j = 0; j < kPass; ++j)
#pragma unroll
            for (int f = 0; f < FW; ++f)
                *reinterpret_cast<v4f*>(sums + wave * kPart + (j * 16 + r) * kRowPitch + f * 16 + 4 * g) = acc[f][f0 + j];
        __syncthreads();
        for (uint32_t it = tid; it < kPass * 16 * kQuads; it += NT) {
            const uint32_t m = it / kQuads, q = it % kQuads;
            auto total = [&](uint32_t col) -> v4f {
                const float* s = sums + m * kRowPitch + col;
                v4f v = *reinterpret_cast<const v4f*>(s);
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    const v4f o = *reinterpret_cast<const v4f*>(s + w * kPart);
                    if constexpr (FMT == kFmtI8) v = __builtin_bit_cast(v4f, __builtin_bit_cast(v4i, v) + __builtin_bit_cast(v4i, o));
                    else v += o;
                }
                return v;
            };
            const v4f v = total(4 * q);
            v4f u = v;
            if constexpr (epi_pairs_gate_up(EPI)) u = total(TW / 2 + 4 * q);
            uint32_t ncol = tc.wt * (epi_pairs_gate_up(EPI) ? TW / 2 : TW) + 4 * q;
            if constexpr (KSLOW) ncol = ncol / 16 * 16 < p.n ? wcol_of(q / 4) + q % 4 * 4 : p.n;
            store_quad<EPI>(p, tc, f0 * 16 + m, ncol, v, u);
        }
    }
}

// a ragged tile does the work of the rows it has
template <int FMT, int FW, int FM, int NW, int EPI, int LAYOUT, bool STREAM>
__device__ __forceinline__ void ks_rows(const GemmParams& p, const Tile& tc, uint8_t* smem) {
    if constexpr (FM >= 4) {
        if (tc.rows_valid <= 16 * FM / 4) return ks_tile<FMT, FW, FM / 4, NW, EPI, LAYOUT, STREAM>(p, tc, smem);
    }
    if constexpr (FM >= 2) {
        if (tc.rows_valid <= 16 * FM / 2) return ks_tile<FMT, FW, FM / 2, NW, EPI, LAYOUT, STREAM>(p, tc, smem);
    }
    // A slot without a slab costs the vector cache its loads all the same, so a short K gets a short ring (us, quantizer included: 30 x 1000 x
    // 512, five slots for one slab 7.1 -> 5.7; 5 x 4096 x 2048 7.5 -> 6.1; 1 x 4096 x 4096, eight for four 7.7 -> 6.9).
    if constexpr (NW == 8 && ks_ring(FMT, FW, FM) >= 4) {
        if (p.kbytes <= 2 * NW * kSlabBytes) return ks_tile<FMT, FW, FM, NW, EPI, LAYOUT, STREAM, 2>(p, tc, smem);
        if constexpr (ks_ring(FMT, FW, FM) > 4)
            if (p.kbytes <= 4 * NW * kSlabBytes) return ks_tile<FMT, FW, FM, NW, EPI, LAYOUT, STREAM, 4>(p, tc, smem);
    }
    ks_tile<FMT, FW, FM, NW, EPI, LAYOUT, STREAM>(p, tc, smem);
}

template <int FMT, int FW, int FM, int NW, int EPI, int LAYOUT, KsplitWeights LOADS, Locate HOW>
__global__ __launch_bounds__(64 * NW, 2) void mx_gemm_ksplit_kernel(const GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    Tile tc;
    if (!locate_tile<16 * FM, HOW>(p, tc)) return;
    tc.g = __builtin_amdgcn_readfirstlane(tc.g);
    tc.wt = __builtin_amdgcn_readfirstlane(tc.wt);
    tc.row0 = __builtin_amdgcn_readfirstlane(tc.row0);
    tc.rows_valid = __builtin_amdgcn_readfirstlane(tc.rows_valid);
    if constexpr (LOADS == KsplitWeights::kByGroup) {
        if (__builtin_amdgcn_readfirstlane(tc.mt != 0 || tc.rows_left > 16u * FM))
            return ks_rows<FMT, FW, FM, NW, EPI, LAYOUT, false>(p, tc, smem);
    }
    ks_rows<FMT, FW, FM, NW, EPI, LAYOUT, LOADS != KsplitWeights::kCached>(p, tc, smem);
}

template <int FMT, int FW, int FM, int NW, int EPI, int LAYOUT, KsplitWeights LOADS, Locate HOW>
int launch_one(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    constexpr auto kfn = mx_gemm_ksplit_kernel<FMT, FW, FM, NW, EPI, LAYOUT, LOADS, HOW>;
    if (int rc = allow_dynamic_lds<kfn, kKsplitMaxLds>(); rc != CMX_OK) return rc;
    const size_t smem = ksplit_lds_bytes({FW, FM, NW}, FMT, p.kblocks, LAYOUT);
    CMX_REQUIRE(smem <= kKsplitMaxLds, "split-K tile exceeds the LDS");
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    hipLaunchKernelGGL(kfn, dim3((uint32_t)tiles), dim3(64 * NW), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

// the tile shapes that exist for an element format and epilogue: one for grouped problems, all for dense ones
template <int FMT, int EPI, int LAYOUT>
int launch_shape(const GemmParams& p, const KsplitTile& t, uint32_t max_m_tiles, KsplitWeights loads, hipStream_t s) {
#define CMX_KS(FW_, FM_, NW_) if (t.fw == FW_ && t.fm == FM_ && t.waves == NW_) return launch_one<FMT, FW_, FM_, NW_, EPI, LAYOUT, KsplitWeights::kCached, Locate::kDense>(p, max_m_tiles, s)
    const bool grouped = p.row_off != nullptr || p.sizes != nullptr;             // (kCached kernels know no groups)
    constexpr KsplitWeights kS = KsplitWeights::kStreamed, kG = KsplitWeights::kByGroup;
    if constexpr (LAYOUT != kKSlow) if (t.fw == 4 && t.fm == 4 && t.waves == 4 && grouped) {
        if (p.sizes != nullptr)
            return loads == kS ? launch_one<FMT, 4, 4, 4, EPI, LAYOUT, kS, Locate::kSizes>(p, max_m_tiles, s) : launch_one<FMT, 4, 4, 4, EPI, LAYOUT, kG, Locate::kSizes>(p, max_m_tiles, s);
        return loads == kS ? launch_one<FMT, 4, 4, 4, EPI, LAYOUT, kS, Locate::kTables>(p, max_m_tiles, s) : launch_one<FMT, 4, 4, 4, EPI, LAYOUT, kG, Locate::kTables>(p, max_m_tiles, s);
    }
    CMX_REQUIRE(!grouped, "split-K tile of a grouped problem: 64 x 64 only");
    if constexpr (LAYOUT == kKSlow) {
        CMX_KS(4, 4, 4);
        CMX_KS(4, 1, 8);
        CMX_KS(4, 2, 8);
        CMX_KS(4, 4, 8);
    }
    if constexpr (EPI == kEpiStore && LAYOUT == kRowMajor) {
        CMX_KS(4, 4, 4);
        CMX_KS(1, 1, 8);
        CMX_KS(1, 2, 8);
        CMX_KS(2, 1, 8);
        CMX_KS(2, 2, 8);
        CMX_KS(2, 4, 8);
        CMX_KS(4, 1, 8);
        CMX_KS(4, 2, 8);
        CMX_KS(4, 4, 8);
    }
#undef CMX_KS
    set_error("unsupported split-K tile");
    return CMX_EINVAL;
}

}  // namespace

size_t ksplit_lds_bytes(const KsplitTile& t, int fmt, uint32_t kblocks, int layout) {
    const size_t rows = layout == kKSlow ? 16 * t.fm : 16 * (t.fw + t.fm);
    const size_t scales = ks_scale_steps(fmt) ? round_up_sz(rows * ks_scale_pitch(fmt, kblocks) * 4, 16) : 0;
    const size_t pairs = layout == kKSlow ? (size_t)kblocks / 2 * 128 : 0;
    const size_t loop = scales + pairs + (size_t)t.waves * ks_exchange_bufs(t.fw, t.fm, layout) * 2048;
    const size_t sums = ks_sum_bytes(t.fw, t.fm, t.waves);
    return loop > sums ? loop : sums;
}

bool ksplit_k_slow_tile(KsplitTile* t, uint32_t m, uint32_t n, int fmt, uint32_t kblocks, int cus) {
    if (fmt == CMX_FMT_E2M1 || kblocks % 4 != 0) return false;
    KsplitTile out = {4, 4, t->waves};
    if (t->waves == 8) {
        const auto tiles = [&](int fm) { return (uint64_t)ceil_div(n, 64) * ceil_div(m, 16 * fm); };
        out.fm = tiles(1) <= (uint64_t)cus ? 1 : (tiles(2) <= (uint64_t)cus ? 2 : 4);
    }
    if (ksplit_lds_bytes(out, fmt, kblocks, kKSlow) > kKsplitMaxLds) return false;
    *t = out;
    return true;
}

int launch_ksplit_k_slow(const GemmParams& p, const KsplitTile& t, int fmt, uint32_t max_m_tiles, hipStream_t s) {
    if (fmt == CMX_FMT_E5M2) return launch_shape<CMX_FMT_E5M2, kEpiStore, kKSlow>(p, t, max_m_tiles, KsplitWeights::kCached, s);
    return launch_shape<CMX_FMT_E4M3, kEpiStore, kKSlow>(p, t, max_m_tiles, KsplitWeights::kCached, s);
}

int launch_ksplit(const GemmParams& p, const KsplitTile& t, int fmt, int epi, uint32_t max_m_tiles, KsplitWeights loads, hipStream_t s) {
    if (fmt == CMX_FMT_E4M3) {
        if (epi == kEpiStore)
            return p.w_pretiled ? launch_shape<CMX_FMT_E4M3, kEpiStore, kTiled>(p, t, max_m_tiles, loads, s) : launch_shape<CMX_FMT_E4M3, kEpiStore, kRowMajor>(p, t, max_m_tiles, loads, s);
        if (epi == kEpiSwigluQuant)
            return p.w_pretiled ? launch_shape<CMX_FMT_E4M3, kEpiSwigluQuant, kTiled>(p, t, max_m_tiles, loads, s)
                                : launch_shape<CMX_FMT_E4M3, kEpiSwigluQuant, kRowMajor>(p, t, max_m_tiles, loads, s);
        if (epi == kEpiSwigluQuantAct && !p.w_pretiled) return launch_shape<CMX_FMT_E4M3, kEpiSwigluQuantAct, kRowMajor>(p, t, max_m_tiles, loads, s);
    }
    if (fmt == CMX_FMT_E5M2 && epi == kEpiStore)
        return p.w_pretiled ? launch_shape<CMX_FMT_E5M2, kEpiStore, kTiled>(p, t, max_m_tiles, loads, s) : launch_shape<CMX_FMT_E5M2, kEpiStore, kRowMajor>(p, t, max_m_tiles, loads, s);
    if (fmt == CMX_FMT_E2M1 && epi == kEpiStore) return launch_shape<CMX_FMT_E2M1, kEpiStore, kRowMajor>(p, t, max_m_tiles, loads, s);
    if (fmt == kFmtI8 && epi == kEpiI8DequantSwiglu) return launch_shape<kFmtI8, kEpiI8DequantSwiglu, kRowMajor>(p, t, max_m_tiles, loads, s);
    set_error("unsupported split-K problem");
    return CMX_EINVAL;
}

}  // namespace cmx
