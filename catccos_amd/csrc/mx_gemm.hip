// Block-scaled MX matmul for gfx950 on v_mfma_scale_f32_32x32x64_f8f6f4.
//
//   C[m, n] = sum_k deq(A)[m, k] * deq(W)[n, k]        A = activations, W = transposed weights
//
// Both operands are K-contiguous, which is what the scaled MFMA wants: per step a lane feeds two
// 16-byte runs of one row (FP4: one run = a whole 32-block) plus that row's E8M0 byte for the
// 32-block its half-wave owns.  The weights
// are the MFMA's first operand and the activations the second, so an accumulator register quad
// holds four consecutive n for one m: stores are 8-byte vectors and the SwiGLU/requant epilogue
// finds a whole 32-wide MX block of one activation row in two lanes (l and l^32).
//
// One workgroup (256 threads = 4 wavefronts) owns a TW x TM tile (weight rows x activation rows)
// and walks K in 128-byte slabs through a two-stage LDS ring: while the MFMAs consume slab i
// the global loads of slab i+1 are in flight in registers.  A/W tiles are stored with a 16-byte
// chunk XOR swizzle so both the 16-byte row-strided MFMA operand reads and the staging writes are
// bank-conflict free; the per-row scale dwords of the slab ride along in LDS.
//
// Ragged expert groups: a tiny prologue kernel turns the device-resident group sizes into row
// offsets and a prefix of m-tiles; each workgroup binary-searches its (group, n-tile, m-tile) from
// that prefix, so no host synchronisation is needed and empty groups cost nothing.  Workgroup ids
// are remapped so that each XCD (ids congruent mod 8) walks a contiguous run of tiles that share
// weight panels in its own L2.
#include <type_traits>

#include "group_tables.h"
#include "mx_gemm_common.h"
#include "mx_gemm_ksplit.h"
#include "mx_gemm_ring_tile.h"
#include "mx_launch.h"

namespace cmx {

namespace {

template <int FMT>
__device__ __forceinline__ v16f mfma(v8i w, v8i a, v16f c, int opsel_tag, int sw, int sa);

// opsel picks which byte of the lane's scale register feeds the MFMA (same byte for both operands here)
#define CMX_MFMA_CASE(fmtcode, sel) \
    __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, fmtcode, fmtcode, sel, sw, sel, sa)

template <>
__device__ __forceinline__ v16f mfma<CMX_FMT_E4M3>(v8i w, v8i a, v16f c, int sel, int sw, int sa) {
    switch (sel) {
        case 0: return CMX_MFMA_CASE(0, 0);
        case 1: return CMX_MFMA_CASE(0, 1);
        case 2: return CMX_MFMA_CASE(0, 2);
        default: return CMX_MFMA_CASE(0, 3);
    }
}
template <>
__device__ __forceinline__ v16f mfma<CMX_FMT_E5M2>(v8i w, v8i a, v16f c, int sel, int sw, int sa) {
    switch (sel) {
        case 0: return CMX_MFMA_CASE(1, 0);
        case 1: return CMX_MFMA_CASE(1, 1);
        case 2: return CMX_MFMA_CASE(1, 2);
        default: return CMX_MFMA_CASE(1, 3);
    }
}
template <>
__device__ __forceinline__ v16f mfma<CMX_FMT_E2M1>(v8i w, v8i a, v16f c, int sel, int sw, int sa) {
    switch (sel) {
        case 0: return CMX_MFMA_CASE(4, 0);
        case 1: return CMX_MFMA_CASE(4, 1);
        case 2: return CMX_MFMA_CASE(4, 2);
        default: return CMX_MFMA_CASE(4, 3);
    }
}

// INT8: one 64-deep K step is two v_mfma_i32_32x32x32_i8, fed by the two halves of the same fragment registers
// (any fixed assignment of the 32 K positions to lanes and registers gives the same integer sum, as long as both
// operands use the same one); the INT32 accumulators travel in the fp32 accumulator type bit for bit.
template <>
__device__ __forceinline__ v16f mfma<kFmtI8>(v8i w, v8i a, v16f c, int, int, int) {
    typedef int v16i __attribute__((ext_vector_type(16)));
    v16i acc = __builtin_bit_cast(v16i, c);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8((v4i){w[0], w[1], w[2], w[3]}, (v4i){a[0], a[1], a[2], a[3]}, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8((v4i){w[4], w[5], w[6], w[7]}, (v4i){a[4], a[5], a[6], a[7]}, acc, 0, 0, 0);
    return __builtin_bit_cast(v16f, acc);
}

// LDS/tile row of a wavefront's weight fragment f (gate fragments first, their up partners second)
template <int TW, int WW, int EPI, int FW>
__device__ __forceinline__ uint32_t wfrag_row_of(uint32_t ww, int f) {
    if (epi_pairs_gate_up(EPI))
        return f < FW / 2 ? ww * (TW / 2 / WW) + f * 32 : TW / 2 + ww * (TW / 2 / WW) + (f - FW / 2) * 32;
    return ww * (TW / WW) + f * 32;
}

template <int TW, int TM, int WW, int WM, int EPI, int FW, int FM>
__device__ __forceinline__ void epilogue(const GemmParams& p, const Tile& tc, v16f (&acc)[FW][FM], uint32_t ww,
                                         uint32_t wm, uint32_t lane) {
    const uint32_t l32 = lane & 31u, lh = lane >> 5;
    const uint32_t wt = tc.wt, row0 = tc.row0, rows_valid = tc.rows_valid;
    auto wfrag_row = [&](int f) -> uint32_t { return wfrag_row_of<TW, WW, EPI, FW>(ww, f); };
    if constexpr (epi_is_lean_store(EPI)) {
        uint16_t* const c = reinterpret_cast<uint16_t*>(p.c);
        auto pack = [](float a, float b) -> uint32_t {
            if constexpr (EPI == kEpiStoreFp16) {
                typedef _Float16 v2h __attribute__((ext_vector_type(2)));
                return __builtin_bit_cast(uint32_t, (v2h){(_Float16)a, (_Float16)b});
            } else {
                return cvt_pk_bf16(a, b);
            }
        };
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            const uint32_t mloc = wm * (TM / WM) + fm * 32 + l32;
            const bool mvalid = mloc < rows_valid;
            uint16_t* const crow = c + (size_t)(row0 + (mvalid ? mloc : 0)) * p.ldc;
#pragma unroll
            for (int fw = 0; fw < FW; ++fw) {
                // A lane holds columns 8q + 4 lh + {0..3} of its row for q = 0..3, its partner in the other half-wave
                // (same row) the four next to them.  Swapping register halves between the two gives either lane eight
                // consecutive columns: one 16-byte store instead of two 8-byte ones.
#pragma unroll
                for (int qp = 0; qp < 2; ++qp) {
                    const int q = 2 * qp;
                    const uint32_t a0 = pack(acc[fw][fm][4 * q], acc[fw][fm][4 * q + 1]);
                    const uint32_t a1 = pack(acc[fw][fm][4 * q + 2], acc[fw][fm][4 * q + 3]);
                    const uint32_t b0 = pack(acc[fw][fm][4 * q + 4], acc[fw][fm][4 * q + 5]);
                    const uint32_t b1 = pack(acc[fw][fm][4 * q + 6], acc[fw][fm][4 * q + 7]);
                    // upper half of a <-> lower half of b: lower lanes end up with columns 8q .. 8q+7 in (a, b), upper
                    // lanes with 8(q+1) .. 8(q+1)+7
                    const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
                    const uint32_t ncol = wt * TW + wfrag_row(fw) + 8 * (q + lh);
                    if (mvalid && ncol < p.n) *reinterpret_cast<uint4*>(crow + ncol) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
                }
            }
        }
    } else if constexpr (EPI == kEpiStore) {
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            const uint32_t mloc = wm * (TM / WM) + fm * 32 + l32;
            if (mloc >= rows_valid) continue;
            const size_t mrow = (size_t)(row0 + mloc);
#pragma unroll
            for (int fw = 0; fw < FW; ++fw) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t ncol = wt * TW + wfrag_row(fw) + 8 * q + 4 * lh;
                    if (ncol >= p.n) continue;
                    const v4f v = to_v4(acc[fw][fm], q);
                    const bool full = ncol + 4 <= p.n;
                    if (p.out_type == CMX_OUT_BF16) {
                        uint16_t* o = reinterpret_cast<uint16_t*>(p.c) + mrow * p.ldc + ncol;
                        uint32_t b0 = f32_to_bf16(v[0]), b1 = f32_to_bf16(v[1]), b2 = f32_to_bf16(v[2]),
                                 b3 = f32_to_bf16(v[3]);
                        if (full && (p.ldc % 4 == 0)) {
                            *reinterpret_cast<uint2*>(o) = make_uint2(b0 | (b1 << 16), b2 | (b3 << 16));
                        } else {
                            uint32_t bb[4] = {b0, b1, b2, b3};
                            for (uint32_t i = 0; i < 4 && ncol + i < p.n; ++i) o[i] = (uint16_t)bb[i];
                        }
                    } else if (p.out_type == CMX_OUT_FP16) {
                        _Float16* o = reinterpret_cast<_Float16*>(p.c) + mrow * p.ldc + ncol;
                        for (uint32_t i = 0; i < 4 && ncol + i < p.n; ++i) o[i] = (_Float16)v[i];
                    } else {
                        float* o = reinterpret_cast<float*>(p.c) + mrow * p.ldc + ncol;
                        for (uint32_t i = 0; i < 4 && ncol + i < p.n; ++i) o[i] = v[i];
                    }
                }
            }
        }
    } else if constexpr (EPI == kEpiI8DequantSwiglu) {
        // INT32 sums -> fp32 * per-channel scale -> fp16 -> fp32 * per-token scale -> x0 * sigmoid(x0) * gate, fp32 out.
        // w_scale holds the fp32 channel scales of all groups ([groups * n], element stride ld_ws), a_scale the fp32
        // per-row scales.
        typedef int v16i __attribute__((ext_vector_type(16)));
        const uint32_t half = p.n >> 1;
        const float* ch = reinterpret_cast<const float*>(p.w_scale) + (size_t)tc.g * p.n * p.ld_ws;
        const float* ts = reinterpret_cast<const float*>(p.a_scale);
        float* const out = reinterpret_cast<float*>(p.c);
        const bool vec = p.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0;
#pragma unroll
        for (int f = 0; f < FW / 2; ++f) {
            const uint32_t ncol0 = wt * (TW / 2) + ww * (TW / 2 / WW) + f * 32;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // the four columns 8 q + 4 lh + {0..3} of this fragment: their channel scales serve every row block
                const uint32_t ncol = ncol0 + 8 * q + 4 * lh;
                float cg[4], cu[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t nc = ncol + i < half ? ncol + i : half - 1;
                    cg[i] = ch[(size_t)nc * p.ld_ws];
                    cu[i] = ch[(size_t)(half + nc) * p.ld_ws];
                }
                const bool whole = vec && ncol + 4 <= half;
#pragma unroll
                for (int fm = 0; fm < FM; ++fm) {
                    const uint32_t mloc = wm * (TM / WM) + fm * 32 + l32;
                    if (mloc >= rows_valid) continue;
                    const size_t mrow = (size_t)(row0 + mloc);
                    const float tsv = ts[mrow];
                    const v16i ig = __builtin_bit_cast(v16i, acc[f][fm]), iu = __builtin_bit_cast(v16i, acc[f + FW / 2][fm]);
                    float y[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = 4 * q + i;
                        const float x0 = __fmul_rn(i8_dequant(ig[r], cg[i]), tsv);
                        const float gate = __fmul_rn(i8_dequant(iu[r], cu[i]), tsv);
                        y[i] = __fmul_rn(__fmul_rn(x0, __builtin_amdgcn_rcpf(1.0f + __expf(-x0))), gate);
                    }
                    if (p.out_type == CMX_OUT_FP32) {
                        float* o = out + mrow * p.ldc + ncol;
                        if (whole) {
                            *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
                        } else {
                            for (uint32_t i = 0; i < 4 && ncol + i < half; ++i) o[i] = y[i];
                        }
                    } else {
                        uint16_t h[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            h[i] = p.out_type == CMX_OUT_FP16 ? __builtin_bit_cast(uint16_t, (_Float16)as_f32(y[i])) : (uint16_t)f32_to_bf16(y[i]);
                        uint16_t* o = reinterpret_cast<uint16_t*>(p.c) + mrow * p.ldc + ncol;
                        if (whole) {
                            *reinterpret_cast<uint2*>(o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                        } else {
                            for (uint32_t i = 0; i < 4 && ncol + i < half; ++i) o[i] = h[i];
                        }
                    }
                }
            }
        }
    } else {
        const uint32_t half = p.n >> 1;
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            const uint32_t mloc = wm * (TM / WM) + fm * 32 + l32;
            const bool mvalid = mloc < rows_valid;
            const size_t mrow = (size_t)(row0 + (mvalid ? mloc : 0));
#pragma unroll
            for (int f = 0; f < FW / 2; ++f) {
                // activation column of this fragment's 32-wide MX block
                const uint32_t ncol0 = wt * (TW / 2) + ww * (TW / 2 / WW) + f * 32;
                // GMM1 output rounded to bf16, SwiGLU in fp32, rounded to bf16 again: all on packed pairs with the
                // hardware bf16 conversion; pk[j] holds activation values 2j, 2j+1 of this lane
                uint32_t pk[8];
                uint32_t m = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t g2 = cvt_pk_bf16(acc[f][fm][2 * j], acc[f][fm][2 * j + 1]);
                    const uint32_t u2 = cvt_pk_bf16(acc[f + FW / 2][fm][2 * j], acc[f + FW / 2][fm][2 * j + 1]);
                    const float a0 = silu_mul(__uint_as_float(g2 << 16), __uint_as_float(u2 << 16));
                    const float a1 = silu_mul(__uint_as_float(g2 & 0xFFFF0000u), __uint_as_float(u2 & 0xFFFF0000u));
                    pk[j] = cvt_pk_bf16(a0, a1);
                    m = pk_max_u16(m, pk[j] & 0x7FFF7FFFu);
                }
                if constexpr (EPI == kEpiSwigluQuantAct) {
                    if (p.act_bf16 && mvalid) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const uint32_t ncol = ncol0 + 8 * (r >> 2) + 4 * lh + (r & 3);
                            if (ncol < half) p.act_bf16[mrow * half + ncol] = (uint16_t)(pk[r >> 1] >> (16 * (r & 1)));
                        }
                    }
                }
                uint32_t amax = max(m & 0xFFFFu, m >> 16);
                // the other half of the block's columns sits in lane l ^ 32: swap the half-waves of two copies in the
                // register file (no trip through the LDS crossbar, no lgkmcnt wait between the blocks)
                const auto both = __builtin_amdgcn_permlane32_swap(amax, amax, false, false);
                amax = max(both[0], both[1]);
                const int e = block_exp_from_bf16_amax(amax, kEmaxE4M3);
                if (!mvalid || ncol0 >= half) continue;
                // clamp the magnitudes to 448 * 2^e on the bit patterns, divide by 2^e and cast in one instruction
                const uint32_t lim = (((uint32_t)(e + kEmaxE4M3 + 127) << 7) | 0x60u) * 0x10001u;
                const float scale = __uint_as_float((uint32_t)(e + 127) << 23);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t c0 = pk_min_u16(pk[2 * q] & 0x7FFF7FFFu, lim) | (pk[2 * q] & 0x80008000u);
                    const uint32_t c1 = pk_min_u16(pk[2 * q + 1] & 0x7FFF7FFFu, lim) | (pk[2 * q + 1] & 0x80008000u);
                    *reinterpret_cast<uint32_t*>(p.act_codes + mrow * p.ld_act + ncol0 + 8 * q + 4 * lh) =
                        cvt_scaled_pk4<CMX_FMT_E4M3>(c0, c1, scale);
                }
                if (lh == 0) {
                    uint8_t* srow = p.act_scales + mrow * p.ld_acts;
                    const uint32_t blk = ncol0 >> 5;
                    srow[blk] = (uint8_t)(e + 127);
                    const uint32_t nblk = half >> 5;
                    if (blk == nblk - 1 && (nblk & 1u)) srow[nblk] = 127;
                }
            }
        }
    }
}

// The lean 16-bit store in whole cache lines, for the persistent two-slot kernels.  Straight from the accumulator layout
// (epilogue above) a store instruction writes 32 bytes to each of 32 rows and a 128-byte line is complete only after four
// such instructions.  Here the 32 rows x 128 bytes that two neighbouring weight fragments hold for one activation fragment go
// through a 4 KiB staging area in the LDS (16-byte pieces, XOR-swizzled by row: neither the writes nor the reads conflict)
// and come back with eight lanes on a row, so that a store instruction writes eight whole lines, non-temporal (the kernel
// does not read its output again).  `stage` is the wavefront's own 4 KiB; a wavefront reads only what it wrote itself.
template <int TW, int TM, int WW, int WM, int EPI, int FW, int FM>
__device__ __forceinline__ void lean_store_lines(const GemmParams& p, const Tile& tc, v16f (&acc)[FW][FM], uint32_t ww, uint32_t wm,
                                                 uint32_t lane, uint32_t stage) {
    static_assert(epi_is_lean_store(EPI) && FW % 2 == 0, "16-bit store epilogues, weight fragments in pairs");
    const uint32_t l32 = lane & 31u, lh = lane >> 5;
    auto pack = [](float a, float b) -> uint32_t {
        if constexpr (EPI == kEpiStoreFp16) {
            typedef _Float16 v2h __attribute__((ext_vector_type(2)));
            return __builtin_bit_cast(uint32_t, (v2h){(_Float16)a, (_Float16)b});
        } else {
            return cvt_pk_bf16(a, b);
        }
    };
    // write side: row l32 of the fragment, piece (f2, qp, lh) = columns 32 f2 + 16 qp + 8 lh .. + 8 of the pair's 64
    const uint32_t wr_row = stage + l32 * 128;
    // read side: instruction j covers rows 8 j .. 8 j + 7, lane i row 8 j + i / 8, piece i % 8
    const uint32_t rd_r = lane >> 3, rd_p = lane & 7u;
    uint16_t* const c = reinterpret_cast<uint16_t*>(p.c);
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
#pragma unroll
        for (int pr = 0; pr < FW / 2; ++pr) {
#pragma unroll
            for (int f2 = 0; f2 < 2; ++f2) {
                const int fw = 2 * pr + f2;
#pragma unroll
                for (int qp = 0; qp < 2; ++qp) {
                    const int q = 2 * qp;
                    const uint32_t a0 = pack(acc[fw][fm][4 * q], acc[fw][fm][4 * q + 1]);
                    const uint32_t a1 = pack(acc[fw][fm][4 * q + 2], acc[fw][fm][4 * q + 3]);
                    const uint32_t b0 = pack(acc[fw][fm][4 * q + 4], acc[fw][fm][4 * q + 5]);
                    const uint32_t b1 = pack(acc[fw][fm][4 * q + 6], acc[fw][fm][4 * q + 7]);
                    // upper half of a <-> lower half of b: either lane ends up with eight consecutive columns of its row
                    const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
                    const uint32_t piece = 4 * f2 + 2 * qp + lh;
                    const uint32_t addr = wr_row + ((piece ^ (l32 & 7u)) << 4);
                    asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"((v4i){(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]}) : "memory");
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            v4i v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t r = 8 * j + rd_r;
                asm volatile("ds_read_b128 %0, %1" : "=v"(v[j]) : "v"(stage + r * 128 + ((rd_p ^ (r & 7u)) << 4)) : "memory");
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // also: the area is free for the next pair's pieces
            const uint32_t col = tc.wt * TW + ww * (TW / WW) + pr * 64 + rd_p * 8;      // first of the lane's eight output columns
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t mloc = wm * (TM / WM) + fm * 32 + 8 * j + rd_r;
                if (mloc < tc.rows_valid && col < p.n)                   // n is a multiple of 8: a piece is in or out as a whole
                    __builtin_nontemporal_store(v[j], reinterpret_cast<v4i*>(c + (size_t)(tc.row0 + mloc) * p.ldc + col));
            }
        }
    }
}

// INT8 dequant + SwiGLU of the persistent two-slot kernel, stored in whole lines like lean_store_lines: the 32 rows x 128 bytes that a
// gate and an up fragment (16-bit outputs: two of each) give for one activation fragment go through `stage`.  The scales of the tile lie
// in the LDS at `scales` ([256 channels][256 tokens] fp32, in the order of the tile's rows): a load from memory would wait, in order, for
// the two slabs of operands in flight.
template <int TW, int TM, int WW, int WM, int FW, int FM>
__device__ __forceinline__ void i8_store_lines(const GemmParams& p, const Tile& tc, v16f (&acc)[FW][FM], uint32_t ww, uint32_t wm, uint32_t lane,
                                               uint32_t stage, uint32_t scales) {
    typedef int v16i __attribute__((ext_vector_type(16)));
    static_assert(FW == 4, "two gate fragments and their up partners");
    typedef const __attribute__((address_space(3))) v4f* lds_v4f;
    typedef const __attribute__((address_space(3))) float* lds_float;
    const uint32_t l32 = lane & 31u, lh = lane >> 5, half = p.n >> 1;
    const uint32_t wr_row = stage + l32 * 128, x = l32 & 7u;
    const uint32_t rd_r = lane >> 3, rd_p = lane & 7u;
    // 16-bit values are made in both types and picked by a mask: with one wavefront per SIMD a branch on the type for each of a thread's 128
    // values, and five instructions for the conversion to bf16, stood for 5 us a tile (bf16 output, times those of the streaming kernel, with
    // branches -> so: 8 x 2048 rows, K = 384, N = 2048 1.12 -> 0.90; K = 1152, N = 4096 1.08 -> 0.92; 8 x 1000, 7168, 2048 0.97 -> 0.92).
    const bool wide = p.out_type == CMX_OUT_FP32;
    uint32_t fp16 = p.out_type == CMX_OUT_FP16 ? ~0u : 0u;
    asm("" : "+v"(fp16));
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
        const float tsv = *(lds_float)(uintptr_t)(scales + (TW + wm * (TM / WM) + fm * 32 + l32) * 4);
#pragma unroll
        for (int f = 0; f < FW / 2; ++f) {
            const v16i ig = __builtin_bit_cast(v16i, acc[f][fm]), iu = __builtin_bit_cast(v16i, acc[f + FW / 2][fm]);
            const uint32_t ch = scales + (ww * (TW / 2 / WW) + f * 32 + 4 * lh) * 4;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4f cg = *(lds_v4f)(uintptr_t)(ch + 32 * q), cu = *(lds_v4f)(uintptr_t)(ch + 32 * q + TW / 2 * 4);
                float y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x0 = __fmul_rn(i8_dequant(ig[4 * q + i], cg[i]), tsv);
                    const float gate = __fmul_rn(i8_dequant(iu[4 * q + i], cu[i]), tsv);
                    y[i] = __fmul_rn(__fmul_rn(x0, __builtin_amdgcn_rcpf(1.0f + __expf(-x0))), gate);
                }
                if (wide) {
                    asm volatile("ds_write_b128 %0, %1" ::"v"(wr_row + (((2 * q + lh) ^ x) << 4)), "v"((v4f){y[0], y[1], y[2], y[3]}) : "memory");
                } else {
                    v2i h;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint32_t lo = __builtin_bit_cast(uint16_t, (_Float16)as_f32(y[2 * j])), hi = __builtin_bit_cast(uint16_t, (_Float16)as_f32(y[2 * j + 1]));
                        h[j] = (int)(((lo | hi << 16) & fp16) | (cvt_pk_bf16(y[2 * j], y[2 * j + 1]) & ~fp16));
                    }
                    asm volatile("ds_write_b64 %0, %1" ::"v"(wr_row + (((4 * f + q) ^ x) << 4) + 8 * lh), "v"(h) : "memory");
                }
            }
            if (!wide && f == 0) continue;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            v4i v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t r = 8 * j + rd_r;
                asm volatile("ds_read_b128 %0, %1" : "=v"(v[j]) : "v"(stage + r * 128 + ((rd_p ^ (r & 7u)) << 4)) : "memory");
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // also: the area is free for the next pieces
            const uint32_t col = tc.wt * (TW / 2) + ww * (TW / 2 / WW) + (wide ? f * 32 + rd_p * 4 : rd_p * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t mloc = wm * (TM / WM) + fm * 32 + 8 * j + rd_r;
                if (mloc < tc.rows_valid && col < half)                // n / 2 is a multiple of 32: a piece is in or out as a whole
                    __builtin_nontemporal_store(v[j], reinterpret_cast<v4i*>(static_cast<uint8_t*>(p.c) + ((size_t)(tc.row0 + mloc) * p.ldc + col) * (wide ? 4 : 2)));
            }
        }
    }
}

// TW/TM: tile rows (weights / activations); WW x WM wavefront grid over the tile (4 or 8 wavefronts).
// FAST: K is a whole number of slabs and scale rows are dword aligned, so the main loop carries no
// bounds checks at all.
template <int FMT, int TW, int TM, int WW, int WM, int EPI, bool FAST>
__global__ __launch_bounds__(64 * WW * WM) void mx_gemm_kernel(const GemmParams p) {
    constexpr int NT = 64 * WW * WM;
    static_assert(NT == 256 || NT == 512, "four or eight wavefronts per workgroup");
    constexpr bool kFp4 = FMT == CMX_FMT_E2M1;
    constexpr int kSub = kFp4 ? 4 : 2;                 // MFMA steps (64 K elements each) per slab
    constexpr int kScaleDw = kFp4 ? 2 : 1;             // scale dwords per row per slab
    constexpr int FW = TW / WW / 32;                   // 32-row fragments per wavefront, weights
    constexpr int FM = TM / WM / 32;                   // activations
    constexpr int kRowsPerPass = NT / kChunks;         // tile rows covered by one 16-byte load per thread
    constexpr int kWLoads = TW / kRowsPerPass;         // 16-byte chunks per thread per slab
    constexpr int kALoads = TM / kRowsPerPass;
    static_assert(FW >= 1 && FM >= 1 && kWLoads >= 1 && kALoads >= 1, "tile too small for the wavefront grid");
    static_assert(!epi_pairs_gate_up(EPI) || (FW % 2 == 0), "gate/up fragments come in pairs");
    static_assert(TW <= NT && TM <= NT, "one scale row per thread");
    constexpr int kStageBytes = (TW + TM) * kSlabBytes + (TW + TM) * 4 * kScaleDw;

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = tid >> 6;
    const uint32_t ww = wave % WW, wm = wave / WW;

    Tile tc;
    if (!locate_tile<TM, Locate::kTables>(p, tc)) return;
    const uint32_t g = tc.g, wt = tc.wt, row0 = tc.row0, rows_valid = tc.rows_valid;

    // ---- global -> LDS staging assignments -----------------------------------------------------
    const uint32_t ld_chunk = tid & 7u;                // 16-byte chunk inside the slab
    const uint32_t ld_row = tid >> 3;                  // + kRowsPerPass*j
    const uint8_t* wg = p.w + (size_t)g * p.n * p.ldw;             // uniform bases, 32-bit lane offsets
    const uint8_t* wsg = p.w_scale + (size_t)g * p.n * p.ld_ws;
    const uint8_t* ag = p.a + (size_t)row0 * p.lda;
    const uint8_t* asg = p.a_scale + (size_t)row0 * p.ld_as;

    // global weight row of LDS tile row r (rows past the matrix repeat the last one; masked at the store)
    auto wrow_of = [&](uint32_t r) -> uint32_t {
        uint32_t gr;
        if (epi_pairs_gate_up(EPI)) {
            const uint32_t half = p.n >> 1;
            uint32_t rr = r < TW / 2 ? wt * (TW / 2) + r : wt * (TW / 2) + (r - TW / 2);
            rr = rr < half ? rr : half - 1;
            gr = r < TW / 2 ? rr : half + rr;
        } else {
            gr = wt * TW + r;
            gr = gr < p.n ? gr : p.n - 1;
        }
        return gr;
    };
    auto arow_of = [&](uint32_t r) -> uint32_t { return r < rows_valid ? r : rows_valid - 1; };

    uint32_t woff[kWLoads], aoff[kALoads];
#pragma unroll
    for (int j = 0; j < kWLoads; ++j) woff[j] = wrow_of(ld_row + kRowsPerPass * j) * p.ldw + ld_chunk * 16;
#pragma unroll
    for (int j = 0; j < kALoads; ++j) aoff[j] = arow_of(ld_row + kRowsPerPass * j) * p.lda + ld_chunk * 16;
    // scale rows: thread t serves weight row t (t < TW) and activation row t (t < TM)
    const uint32_t wsoff = wrow_of(tid < TW ? tid : 0) * p.ld_ws;
    const uint32_t asoff = arow_of(tid < TM ? tid : 0) * p.ld_as;

    const uint32_t nslab = (p.kbytes + kSlabBytes - 1) / kSlabBytes;
    constexpr uint32_t blocks_per_slab = 4 * kScaleDw;

    uint4 wreg[kWLoads], areg[kALoads];
    uint32_t wsreg[kScaleDw], asreg[kScaleDw];

    auto load_scale_dw = [&](const uint8_t* rowp, uint32_t blk0) -> uint32_t {
        // four consecutive scale bytes starting at block blk0; beyond K the scale is 1.0
        if (FAST || (p.scale_vec && blk0 + 4 <= p.kblocks)) return *reinterpret_cast<const uint32_t*>(rowp + blk0);
        uint32_t v = 0x7F7F7F7Fu;
        for (uint32_t i = 0; i < 4; ++i)
            if (blk0 + i < p.kblocks) v = (v & ~(0xFFu << (8 * i))) | ((uint32_t)rowp[blk0 + i] << (8 * i));
        return v;
    };
    auto load_global = [&](uint32_t slab) {
        const uint8_t* wslab = wg + (size_t)slab * kSlabBytes;
        const uint8_t* aslab = ag + (size_t)slab * kSlabBytes;
        const bool in = FAST || (slab * kSlabBytes + ld_chunk * 16 < p.kbytes);
#pragma unroll
        for (int j = 0; j < kWLoads; ++j)
            wreg[j] = in ? *reinterpret_cast<const uint4*>(wslab + woff[j]) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < kALoads; ++j)
            areg[j] = in ? *reinterpret_cast<const uint4*>(aslab + aoff[j]) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int d = 0; d < kScaleDw; ++d) {
            const uint32_t blk0 = slab * blocks_per_slab + 4 * d;
            if (tid < TW) wsreg[d] = load_scale_dw(wsg + wsoff, blk0);
            if (tid < TM) asreg[d] = load_scale_dw(asg + asoff, blk0);
        }
    };
    auto store_lds = [&](uint32_t stage) {
        uint8_t* sW = smem + stage * kStageBytes;
        uint8_t* sA = sW + TW * kSlabBytes;
        uint32_t* sWs = reinterpret_cast<uint32_t*>(sA + TM * kSlabBytes);
        uint32_t* sAs = sWs + TW * kScaleDw;
#pragma unroll
        for (int j = 0; j < kWLoads; ++j) {
            const uint32_t r = ld_row + kRowsPerPass * j;
            *reinterpret_cast<uint4*>(sW + r * kSlabBytes + swz(r, ld_chunk) * 16) = wreg[j];
        }
#pragma unroll
        for (int j = 0; j < kALoads; ++j) {
            const uint32_t r = ld_row + kRowsPerPass * j;
            *reinterpret_cast<uint4*>(sA + r * kSlabBytes + swz(r, ld_chunk) * 16) = areg[j];
        }
#pragma unroll
        for (int d = 0; d < kScaleDw; ++d) {
            if (tid < TW) sWs[tid * kScaleDw + d] = wsreg[d];
            if (tid < TM) sAs[tid * kScaleDw + d] = asreg[d];
        }
    };

    // ---- accumulators --------------------------------------------------------------------------
    v16f acc[FW][FM];
#pragma unroll
    for (int i = 0; i < FW; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    auto wfrag_row = [&](int f) -> uint32_t { return wfrag_row_of<TW, WW, EPI, FW>(ww, f); };
    const uint32_t l32 = lane & 31u, lh = lane >> 5;

    // byte offsets (within a stage's W / A tile) of the lane's two 16-byte runs for step 0; the runs
    // of step h sit at chunk index + 4h (8-bit) or + 2h (FP4), i.e. the XOR swizzle is re-applied
    auto frag_addr = [&](uint32_t r, uint32_t c) -> uint32_t { return r * kSlabBytes + swz(r, c) * 16; };

    auto read_frag = [&](const uint8_t* tile, uint32_t r, int h) -> v8i {
        if (kFp4) {
            v4i lo = *reinterpret_cast<const v4i*>(tile + frag_addr(r, h * 2 + lh));
            return (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
        }
        // 8-bit operands: registers 0-3 carry k = 16*lh + [0,16) of the step's first 32-block,
        // registers 4-7 the same slice of its second 32-block
        v4i lo = *reinterpret_cast<const v4i*>(tile + frag_addr(r, h * 4 + lh));
        v4i hi = *reinterpret_cast<const v4i*>(tile + frag_addr(r, h * 4 + lh + 2));
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    auto compute = [&](uint32_t stage) {
        const uint8_t* sW = smem + stage * kStageBytes;
        const uint8_t* sA = sW + TW * kSlabBytes;
        const uint32_t* sWs = reinterpret_cast<const uint32_t*>(sA + TM * kSlabBytes);
        const uint32_t* sAs = sWs + TW * kScaleDw;
        // operand fragments are double buffered in registers: the LDS reads of step h+1 are issued
        // before the MFMAs of step h
        v8i af[2][FM], wf[2][FW];
#pragma unroll
        for (int f = 0; f < FM; ++f) af[0][f] = read_frag(sA, wm * (TM / WM) + f * 32 + l32, 0);
#pragma unroll
        for (int f = 0; f < FW; ++f) wf[0][f] = read_frag(sW, wfrag_row(f) + l32, 0);
        // lane's scale registers: byte 2*h' (after the lh shift) belongs to MFMA step h' of the dword
        uint32_t sw[FW][kScaleDw], sa[FM][kScaleDw];
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int d = 0; d < kScaleDw; ++d) sw[f][d] = sWs[(wfrag_row(f) + l32) * kScaleDw + d] >> (8 * lh);
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int d = 0; d < kScaleDw; ++d)
                sa[f][d] = sAs[(wm * (TM / WM) + f * 32 + l32) * kScaleDw + d] >> (8 * lh);

#pragma unroll
        for (int h = 0; h < kSub; ++h) {
            const int cur = h & 1, nxt = cur ^ 1;
            if (h + 1 < kSub) {
#pragma unroll
                for (int f = 0; f < FM; ++f) af[nxt][f] = read_frag(sA, wm * (TM / WM) + f * 32 + l32, h + 1);
#pragma unroll
                for (int f = 0; f < FW; ++f) wf[nxt][f] = read_frag(sW, wfrag_row(f) + l32, h + 1);
            }
#pragma unroll
            for (int fw = 0; fw < FW; ++fw) {
#pragma unroll
                for (int fm = 0; fm < FM; ++fm) {
                    // step h uses scale dword h/2, byte 2*(h%2) of the shifted register
                    acc[fw][fm] = mfma<FMT>(wf[cur][fw], af[cur][fm], acc[fw][fm], (h & 1) * 2, (int)sw[fw][h >> 1],
                                            (int)sa[fm][h >> 1]);
                }
            }
        }
    };

    // ---- main loop -------------------------------------------------------------------------------
    load_global(0);
    store_lds(0);
    __syncthreads();
    // steady state is branch free: prefetch slab s+1, consume slab s, refill the other stage
    for (uint32_t s = 0; s + 1 < nslab; ++s) {
        load_global(s + 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(s & 1u);
        // Keep the LDS refill (which waits for the global loads) behind the MFMAs of this slab: without
        // a use of the accumulators here the compiler sinks the MFMAs below the refill and the barrier,
        // which exposes the whole global-load latency every iteration.
#pragma unroll
        for (int i = 0; i < FW; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) asm volatile("" ::"a"(acc[i][j][0]) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        store_lds((s + 1) & 1u);
        __syncthreads();
    }
    compute((nslab - 1) & 1u);

    epilogue<TW, TM, WW, WM, EPI, FW, FM>(p, tc, acc, ww, wm, lane);
}

// ------------------------------------------------------------------------------------------------
// Streaming kernel: operand tiles go global -> LDS directly (LDS-DMA loads, no staging registers and
// no ds_write) into a two-slot ring of 128-byte-deep K slabs; whole 128-byte lines per row keep every
// fetched cache line fully used.  Operand fragments are prefetched into a spare register set one MFMA
// step ahead, so a slot is drained one step before its slab's MFMAs end; at that point
//   wait (own reads of slot s and own loads of slab s+1 done) -> barrier (everyone's) ->
//   refill slot s with slab s+2 -> read the first fragments of slab s+1 -> last MFMA step of slab s.
// One barrier per slab; every load has a full slab of MFMA time to land.
// A load instruction of one wavefront fills 1 KiB of LDS linearly (lane p -> 16 bytes at 16p), i.e.
// 8 tile rows x 8 chunks; the XOR swizzle that keeps the row-strided fragment reads conflict-free is
// applied on the global side (which 16 bytes of the row a lane fetches).  Scale dwords (4 blocks each)
// ride in their own two-slot ring.
#define CMX_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x0F70)
#define CMX_WAIT_ALL() __builtin_amdgcn_s_waitcnt(0x0070)   // vmcnt(0) lgkmcnt(0)

typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef const __attribute__((address_space(1))) void* global_void_ptr;

template <int FMT, int TW, int TM, int WW, int WM, int EPI>
__device__ __forceinline__ void dl_tile(const GemmParams& p, const Tile& tc) {
    constexpr int NW = WW * WM;                        // wavefronts: 4 (one per SIMD) or 8 (two per SIMD)
    static_assert(NW == 4 || NW == 8, "four or eight wavefronts per workgroup");
    constexpr bool kFp4 = FMT == CMX_FMT_E2M1;
    constexpr bool kI8 = FMT == kFmtI8;                // INT8: no block scales at all
    constexpr int kSub = kFp4 ? 4 : 2;                 // MFMA steps (64 K elements each) per slab
    constexpr int kScaleDw = kI8 ? 0 : (kFp4 ? 2 : 1); // scale dwords per row per slab
    constexpr int kScaleDwA = kScaleDw ? kScaleDw : 1; // array extent
    constexpr int FW = TW / WW / 32, FM = TM / WM / 32;
    constexpr int kRows = TW + TM;                     // W tile rows then A tile rows
    constexpr int kTileLoads = kRows / (8 * NW);       // direct loads per thread and slab (8 rows per wavefront-load)
    constexpr int kWTileLoads = TW / (8 * NW);
    constexpr int kSlotBytes = kRows * kSlabBytes;
    constexpr int kScaleSlot = kRows * kScaleDw;       // dwords
    constexpr int kScaleWaveLoads = kRows / 64;        // wavefront-loads that cover one scale dword of every row
    constexpr int kScalePerWave = (kScaleWaveLoads + NW - 1) / NW;
    constexpr int kLoadsPerSlab = kTileLoads + kScalePerWave * kScaleDw;
    static_assert(TW % (8 * NW) == 0 && TM % (8 * NW) == 0 && TW % 64 == 0 && TM % 64 == 0, "tile shape");
    static_assert(FW >= 1 && FM >= 1, "tile too small for the wavefront grid");
    static_assert(!epi_pairs_gate_up(EPI) || (FW % 2 == 0), "gate/up fragments come in pairs");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint32_t* const sScale = reinterpret_cast<uint32_t*>(smem + 2 * kSlotBytes);

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ww = wave % WW, wm = wave / WW;
    const uint32_t l32 = lane & 31u, lh = lane >> 5;

    const uint32_t g = __builtin_amdgcn_readfirstlane(tc.g), wt = __builtin_amdgcn_readfirstlane(tc.wt);
    const uint32_t row0 = __builtin_amdgcn_readfirstlane(tc.row0);
    const uint32_t rows_valid = __builtin_amdgcn_readfirstlane(tc.rows_valid);

    const uint8_t* wg = p.w + (size_t)g * p.n * p.ldw;
    const uint8_t* wsg = p.w_scale + (size_t)g * p.n * p.ld_ws;
    const uint8_t* ag = p.a + (size_t)row0 * p.lda;
    const uint8_t* asg = p.a_scale + (size_t)row0 * p.ld_as;

    auto wrow_of = [&](uint32_t r) -> uint32_t {
        uint32_t gr;
        if (epi_pairs_gate_up(EPI)) {
            const uint32_t half = p.n >> 1;
            uint32_t rr = r < TW / 2 ? wt * (TW / 2) + r : wt * (TW / 2) + (r - TW / 2);
            rr = rr < half ? rr : half - 1;
            gr = r < TW / 2 ? rr : half + rr;
        } else {
            gr = wt * TW + r;
            gr = gr < p.n ? gr : p.n - 1;
        }
        return gr;
    };
    auto arow_of = [&](uint32_t r) -> uint32_t { return r < rows_valid ? r : rows_valid - 1; };

    // ---- per-lane offsets of the direct loads --------------------------------------------------
    // load i of this wavefront fills combined tile rows (NW*i + wave)*8 .. +8; lane p -> row +p/8, LDS chunk p%8
    uint32_t goff[kTileLoads];
#pragma unroll
    for (int i = 0; i < kTileLoads; ++i) {
        const uint32_t cr = (NW * i + wave) * 8 + (lane >> 3);
        const uint32_t logical = swz(cr, lane & 7u);
        goff[i] = (i < kWTileLoads ? wrow_of(cr) * p.ldw : arow_of(cr - TW) * p.lda) + logical * 16;
    }
    // scale dwords: one wavefront-load covers 64 rows; wavefront-load j serves W rows 64j.. (j < TW/64) or A rows
    uint32_t soff_[kScalePerWave], sdst_[kScalePerWave];
    bool s_is_w[kScalePerWave];
#pragma unroll
    for (int t = 0; t < kScalePerWave; ++t) {
        const uint32_t j = wave + NW * t;
        s_is_w[t] = j < TW / 64;
        const uint32_t aj = (j - TW / 64) % (TM / 64);
        soff_[t] = s_is_w[t] ? wrow_of(64 * j + lane) * p.ld_ws : arow_of(64 * aj + lane) * p.ld_as;
        sdst_[t] = s_is_w[t] ? 64 * j : TW + 64 * aj;
    }

    const uint32_t nslab = p.kbytes / kSlabBytes;

    // Buffer addressing: per-lane byte offsets stay constant over the whole K loop and the slab
    // position is a scalar offset, so a load costs no vector ALU work at all.
    constexpr int kRsrcFlags = 0x00020000;
    auto uniform_ptr = [](const uint8_t* q) -> uint8_t* {
        const uint64_t v = reinterpret_cast<uint64_t>(q);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return reinterpret_cast<uint8_t*>(((uint64_t)hi << 32) | lo);
    };
    const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(wg), 0, -1, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t a_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(ag), 0, -1, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t ws_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(wsg), 0, -1, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t as_rs = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(asg), 0, -1, kRsrcFlags);

    auto issue_slab = [&](uint32_t slab) {
        const uint32_t k = slab < nslab ? slab : nslab - 1;              // past the end: harmless reload
        uint8_t* dst = smem + (slab & 1u) * kSlotBytes + wave * 1024;
        const int koff = (int)(k * kSlabBytes);
#pragma unroll
        for (int i = 0; i < kTileLoads; ++i) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(i < kWTileLoads ? w_rs : a_rs, (lds_void_ptr)(dst + i * (NW * 1024)), 16,
                                                     (int)goff[i], koff, 0, 0);
        }
        uint32_t* sdst = sScale + (slab & 1u) * kScaleSlot;
#pragma unroll
        for (int d = 0; d < kScaleDw; ++d) {
            const int soff = (int)((k * kScaleDw + d) * 4);
#pragma unroll
            for (int t = 0; t < kScalePerWave; ++t) {
                if (s_is_w[t])
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(ws_rs, (lds_void_ptr)(sdst + d * kRows + sdst_[t]), 4, (int)soff_[t], soff, 0, 0);
                else
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(as_rs, (lds_void_ptr)(sdst + d * kRows + sdst_[t]), 4, (int)soff_[t], soff, 0, 0);
            }
        }
    };

    // ---- fragment reads ------------------------------------------------------------------------
    auto wfrag_row = [&](int f) -> uint32_t { return wfrag_row_of<TW, WW, EPI, FW>(ww, f); };
    auto read_frag = [&](const uint8_t* tile, uint32_t r, int h) -> v8i {
        const uint8_t* rp = tile + r * kSlabBytes;
        if (kFp4) {
            v4i lo = *reinterpret_cast<const v4i*>(rp + swz(r, h * 2 + lh) * 16);
            return (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
        }
        // 8-bit operands: registers 0-3 carry k = 16*lh + [0,16) of the step's first 32-block,
        // registers 4-7 the same slice of its second 32-block
        v4i lo = *reinterpret_cast<const v4i*>(rp + swz(r, h * 4 + lh) * 16);
        v4i hi = *reinterpret_cast<const v4i*>(rp + swz(r, h * 4 + lh + 2) * 16);
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    v16f acc[FW][FM];
#pragma unroll
    for (int i = 0; i < FW; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    v8i wf[2][FW], af[2][FM];
    uint32_t sw[kScaleDwA][FW] = {}, sa[kScaleDwA][FM] = {}, swn[kScaleDwA][FW] = {}, san[kScaleDwA][FM] = {};

    auto read_frags = [&](uint32_t slab, int h, int buf) {
        const uint8_t* st = smem + (slab & 1u) * kSlotBytes;
#pragma unroll
        for (int f = 0; f < FM; ++f) af[buf][f] = read_frag(st + TW * kSlabBytes, wm * (TM / WM) + f * 32 + l32, h);
#pragma unroll
        for (int f = 0; f < FW; ++f) wf[buf][f] = read_frag(st, wfrag_row(f) + l32, h);
    };
    auto read_scales = [&](uint32_t slab, uint32_t (&w_)[kScaleDwA][FW], uint32_t (&a_)[kScaleDwA][FM]) {
        const uint32_t* sc = sScale + (slab & 1u) * kScaleSlot;
#pragma unroll
        for (int d = 0; d < kScaleDw; ++d) {
#pragma unroll
            for (int f = 0; f < FW; ++f) w_[d][f] = sc[d * kRows + wfrag_row(f) + l32] >> (8 * lh);
#pragma unroll
            for (int f = 0; f < FM; ++f) a_[d][f] = sc[d * kRows + TW + wm * (TM / WM) + f * 32 + l32] >> (8 * lh);
        }
    };

    // ---- prologue -----------------------------------------------------------------------------------
    issue_slab(0);
    issue_slab(1);
    CMX_WAIT_VMCNT(kLoadsPerSlab);      // slab 0 has landed (slab 1 may still be in flight)
    __syncthreads();
    read_frags(0, 0, 0);
    read_scales(0, sw, sa);

    for (uint32_t s = 0; s < nslab; ++s) {
#pragma unroll
        for (int h = 0; h < kSub; ++h) {
            if (h + 1 < kSub) {
                read_frags(s, h + 1, (h + 1) & 1);
            } else {
                // slot s&1 is drained by this wavefront one step early: refill point
                CMX_WAIT_ALL();                 // own fragment reads of slab s and own loads of slab s+1 are done
                __syncthreads();                // ... and everyone else's
                issue_slab(s + 2);
                read_frags(s + 1, 0, 0);
                read_scales(s + 1, swn, san);
            }
            // One wavefront per SIMD issues in order, so the MFMA pipe idles whenever more than one
            // MFMA time of other instructions sits between two MFMAs: spread the LDS reads and the
            // LDS-DMA loads of this step evenly behind the MFMAs instead of clustering them.
            {
                constexpr int kMfmas = FW * FM * (kI8 ? 2 : 1);
                constexpr int kFragReads = (FW + FM) * (kFp4 ? 1 : 2);
                constexpr int kDs = kFragReads + (FW + FM) * kScaleDw;     // refill step also reads the scales
                constexpr int kDsPer = (kDs + kMfmas - 1) / kMfmas;
                constexpr int kVmPer = (kLoadsPerSlab + kMfmas - 1) / kMfmas;
#pragma unroll
                for (int i = 0; i < kMfmas; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);          // one MFMA
                    if (h + 1 == kSub) __builtin_amdgcn_sched_group_barrier(0x020, kVmPer, 0);   // VMEM reads
                    __builtin_amdgcn_sched_group_barrier(0x100, kDsPer, 0);     // DS reads
                }
            }
#pragma unroll
            for (int fw = 0; fw < FW; ++fw)
#pragma unroll
                for (int fm = 0; fm < FM; ++fm)
                    acc[fw][fm] = mfma<FMT>(wf[h & 1][fw], af[h & 1][fm], acc[fw][fm], (h & 1) * 2, (int)sw[h >> 1][fw],
                                            (int)sa[h >> 1][fm]);
            // ... and this step's MFMAs must be issued before the next step's wait/barrier
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int d = 0; d < kScaleDw; ++d) {
#pragma unroll
            for (int f = 0; f < FW; ++f) sw[d][f] = swn[d][f];
#pragma unroll
            for (int f = 0; f < FM; ++f) sa[d][f] = san[d][f];
        }
    }
    CMX_WAIT_VMCNT(0);      // the two reloads issued past the end must land before the LDS is released

    epilogue<TW, TM, WW, WM, EPI, FW, FM>(p, tc, acc, ww, wm, lane);
}

template <int FMT, int TW, int TM, int WW, int WM, int EPI>
__global__ __launch_bounds__(64 * WW * WM) void mx_gemm_dl_kernel(const GemmParams p) {
    Tile tc;
    if (!locate_tile<TM, FMT == kFmtI8 ? Locate::kAny : Locate::kTables>(p, tc)) return;
    dl_tile<FMT, TW, TM, WW, WM, EPI>(p, tc);
}

// INT8 groups of up to 128 rows on average (but one round of 128 x 128 tiles): 256 x 128 tiles of the ring kernel, or 256 x 256 ones.
// What decides is the number of rounds, of a workgroup per CU, that each takes, and with it how the rows lie, which the host does not
// know: a round of the ring's tiles takes 0.7 of one of the others, but where groups are a little longer than 128 rows,
// or few of them hold all rows, there are up to twice as many.  So the device counts both from the sizes: in every workgroup up to two
// rounds, in the launch that fills the tables beyond (a count costs each tile 1 us).  A kernel for each side, the one that the choice
// leaves out finding nothing to do (2 us): both in one kernel share its registers, and the ring's loop comes out slower by a quarter
// (8 groups x 76 rows u, 7168, 3072 58.8 against 41.5).  Below K = 512 the launches cost more than is won (64 x 128 u, 128, 3072 42 -> 51).
// Measured (us, fp32 output, 256 x 256 alone / 256 x 128 alone / the choice; u: routes drawn uniformly, z: Zipf, c: all rows on four groups):
//   K, N, groups x rows      u               z               c
//   7168, 3072, 64 x 100     318 279 286     395 327 338     182 164 169
//   7168, 3072, 32 x 90      200 154 161     195 183 190      81  99  87
//   7168, 3072, 64 x 125     321 354 334     393 335 344     188 215 193
//   2048, 3072, 32 x 90       65  48  52      67  60  66      32  40  38
//   2048, 1024, 256 x 48     154 126 129     183 127 132      36  43  42
//   1024, 3072, 64 x 100      71  58  62      91  70  77      47  47  52
//    512, 3072, 128 x 70      99  77  79     113  90  89      37  52  42
// tiles of 128 and of 256 rows that a problem has; cus: workgroups that run at a time
__device__ __forceinline__ bool short_tiles_pay(uint32_t t128, uint32_t t256, uint32_t cus, uint32_t kblocks) {
    const uint32_t r128 = (t128 + cus - 1) / cus, r256 = (t256 + cus - 1) / cus;
    return kblocks >= 64 ? 5 * r128 <= 8 * r256 : 8 * r128 <= 11 * r256;
}
__device__ __forceinline__ bool short_tiles_pay_by_sizes(const GemmParams& p, uint32_t cus) {
    uint32_t off[kGroupsPerLane + 1], n128 = 0, n256 = 0;
    scan_group_rows(p, off);
#pragma unroll
    for (int j = 0; j < kGroupsPerLane; ++j) {
        n128 += tiles_of_group(p, off[j + 1] - off[j], 128);
        n256 += tiles_of_group(p, off[j + 1] - off[j], 256);
    }
    const auto add = [](uint32_t a, uint32_t b) -> uint32_t { return a + b; };
    return short_tiles_pay((uint32_t)__builtin_amdgcn_readlane((int)wave_scan(n128, add), 63) * p.w_tiles,
                           (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(n256, add), 63) * p.w_tiles, cus, p.kblocks);
}

#include "mx_gemm_pipe.h"
#include "mx_gemm_wreg.h"
#include "mx_gemm_pipe_fp4.h"

// The side of the 128-row tiles, which is left at once where the choice falls on the other (mx_gemm_pipe_kernel).  A workgroup goes on with
// further tiles, so that there are no more of them than run at a time: leaving takes each 0.3 us (256 groups x 48 rows c, 512, 1024, a
// workgroup for each tile 33.9, so 26.3).
__global__ __launch_bounds__(256) void mx_gemm_i8_short_kernel(const GemmParams p) {
    const bool pay = p.sizes != nullptr ? short_tiles_pay_by_sizes(p, p.choice_cus) : table_at(p.short_tiles, 0) != 0;
    if (__builtin_amdgcn_readfirstlane((int)pay) == 0) return;
    Tile tc;
    for (uint32_t id = blockIdx.x; locate_tile<128, Locate::kAny>(p, tc, id); id += gridDim.x) {
        if (id != blockIdx.x) __syncthreads();                 // the LDS of the tile before has been read
        ring_tile<kFmtI8, 256, 128, 2, 2, 3, 0, kEpiI8DequantSwiglu, false>(p, tc);
    }
}
__global__ __launch_bounds__(256) void i8_choice_prepare_kernel(const GroupTablesJob job, uint32_t w_tiles, uint32_t cus, uint32_t kblocks,
                                                                int32_t* const short_tiles) {
    fill_group_tables(job, 256, [=](uint32_t n128, uint32_t n256) -> bool {
        const bool pay = short_tiles_pay(n128 * w_tiles, n256 * w_tiles, cus, kblocks);
        if (threadIdx.x == 0) *short_tiles = pay ? 1 : 0;
        return pay;
    });
}

__global__ __launch_bounds__(256) void gmm_prepare_kernel(const GroupTablesJob job) { fill_group_tables(job); }

template <int FMT, int TW, int TM, int WW, int WM, int EPI, bool FAST>
int launch_gemm_impl(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    constexpr int kScaleDw = FMT == CMX_FMT_E2M1 ? 2 : 1;
    constexpr size_t smem = 2 * ((TW + TM) * kSlabBytes + (TW + TM) * 4 * kScaleDw);
    constexpr auto kfn = mx_gemm_kernel<FMT, TW, TM, WW, WM, EPI, FAST>;
    CMX_REQUIRE(p.sizes == nullptr, "groups by their sizes: not this kernel");
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    hipLaunchKernelGGL(kfn, dim3((uint32_t)tiles), dim3(64 * WW * WM), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

template <int FMT, int TW, int TM, int WW, int WM, int EPI>
int launch_gemm_dl(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    constexpr int kScaleDw = FMT == CMX_FMT_E2M1 ? 2 : 1;
    constexpr size_t smem = 2 * (TW + TM) * kSlabBytes + 2 * (TW + TM) * kScaleDw * 4;
    constexpr auto kfn = mx_gemm_dl_kernel<FMT, TW, TM, WW, WM, EPI>;
    CMX_REQUIRE(FMT == kFmtI8 || p.sizes == nullptr, "groups by their sizes: not this kernel");
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    hipLaunchKernelGGL(kfn, dim3((uint32_t)tiles), dim3(64 * WW * WM), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

// tables of the chosen m-tiles and the choice itself (small groups have no tables of their own then: short_tiles lies in the place of those)
int launch_i8_choice_tables(const GroupTablesJob& job, const GemmParams& p, int32_t* short_tiles, hipStream_t s) {
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    CMX_REQUIRE(job.small_rows == 0 && job.tile_m == 128, "tables of a choice: all groups, 128 rows first");
    hipLaunchKernelGGL(i8_choice_prepare_kernel, dim3(1), dim3(256), 0, s, job, p.w_tiles, (uint32_t)cus, p.kblocks, short_tiles);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

template <int FMT, int EPI, int TM, int WW, int WM, int NSLOT, bool SCAN = FMT == kFmtI8>
int launch_gemm_pipe(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    // tile ring, scale ring (two-slot kernels: two blocks of 16 bytes per row), next-tile mailbox, 256-byte sink of the L2 prefetch loads
    // (+ the 16 KiB staging area of the whole-line stores, which overlays the last 512 bytes)
    // (INT8: the scales of two tiles instead of the scale ring, and a staging area of its own)
    constexpr size_t smem = NSLOT * (256 + TM) * kSlabBytes + (FMT == kFmtI8 ? 2 * (256 + TM) * 4 + 16384 : NSLOT == 2 ? 2 * (256 + TM) * 16 : NSLOT * (256 + TM) * 4) +
                            (pipe_stages_stores(NSLOT, EPI, WW, WM) ? 16384 : 512);
    constexpr auto kfn = mx_gemm_pipe_kernel<FMT, EPI, TM, WW, WM, NSLOT, SCAN>;
    CMX_REQUIRE(SCAN || p.sizes == nullptr, "groups by their sizes: not this kernel");
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    uint32_t grid = (uint32_t)tiles;
    if (pipe_is_persistent(NSLOT, EPI)) {
        // persistent: one workgroup per CU (the LDS footprint admits no second one), a multiple of the XCD count
        int cus = 0;
        if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
        grid = (uint32_t)(cus / kXcds * kXcds);
        if (grid < (uint32_t)kXcds) grid = kXcds;
    }
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(256), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

// tiles128, tiles256: the most m-tiles that either side can have
int launch_i8_choice(const GemmParams& p, uint32_t tiles128, uint32_t tiles256, hipStream_t s) {
    constexpr size_t smem = ring_lds_bytes(256, 128, 3, 0);
    constexpr auto kfn = mx_gemm_i8_short_kernel;
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)tiles128 * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    hipLaunchKernelGGL(kfn, dim3((uint32_t)std::min<uint64_t>(tiles, p.choice_cus)), dim3(256), smem, s, p);
    CMX_LAUNCH_CHECK();
    return launch_gemm_pipe<kFmtI8, kEpiI8DequantSwiglu, 256, 2, 2, 2>(p, tiles256, s);
}

template <int FMT, int EPI, int TM>
int launch_gemm_wreg(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    constexpr auto kfn = mx_gemm_wreg_kernel<FMT, EPI, TM>;
    constexpr size_t kWregLdsBytes = wreg_lds_bytes(TM);
    if (int rc = allow_dynamic_lds<kfn, kWregLdsBytes>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    // persistent: one workgroup per CU, a multiple of the XCD count
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    uint32_t grid = (uint32_t)(cus / kXcds * kXcds);
    if (grid < (uint32_t)kXcds) grid = kXcds;
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(256), kWregLdsBytes, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

template <int EPI, int WW, int WM, bool SCAN = false>
int launch_gemm_pipe_fp4(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    // tile ring, ring of two scale blocks, next-tile mailbox and sink of the L2 prefetch loads (or the 16 KiB staging area of the
    // whole-line stores, which overlays those 512 bytes)
    constexpr size_t smem = 2 * 512 * kSlabBytes + 2 * 512 * 16 + (pipe_stages_stores(2, EPI, WW, WM) ? 16384 : 512);
    constexpr auto kfn = mx_gemm_pipe_fp4_kernel<EPI, WW, WM, SCAN>;
    CMX_REQUIRE(SCAN || p.sizes == nullptr, "groups by their sizes: not this kernel");
    if (int rc = allow_dynamic_lds<kfn, smem>(); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)max_m_tiles * p.w_tiles;
    CMX_REQUIRE(tiles > 0 && tiles < (1ull << 31), "tile count out of range");
    uint32_t grid = (uint32_t)tiles;
    if (pipe_is_persistent(2, EPI)) {
        // persistent: one workgroup per CU (the LDS footprint admits no second one), a multiple of the XCD count
        int cus = 0;
        if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
        grid = (uint32_t)(cus / kXcds * kXcds);
        if (grid < (uint32_t)kXcds) grid = kXcds;
    }
    hipLaunchKernelGGL(kfn, dim3(grid), dim3(256), smem, s, p);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

// The test build of this file (CMX_TEST_HOOKS, linked into the test library only) can force the register-staged
// kernels and pin the tile shape, so that tests reach every compiled instantiation; the product has neither switch.
#ifdef CMX_TEST_HOOKS
bool g_disable_dl = false;
#else
constexpr bool g_disable_dl = false;
#endif

template <int FMT, int TW, int TM, int WW, int WM, int EPI>
int launch_gemm(const GemmParams& p, uint32_t max_m_tiles, hipStream_t s) {
    // streaming kernel: whole 128-element scale groups, dword-aligned scale rows, four wavefronts
    if constexpr (TW % (8 * WW * WM) == 0 && TM % (8 * WW * WM) == 0 && TW % 64 == 0 && TM % 64 == 0) {
        if (!g_disable_dl && p.scale_vec && p.kbytes % kSlabBytes == 0)
            return launch_gemm_dl<FMT, TW, TM, WW, WM, EPI>(p, max_m_tiles, s);
    }
    const bool fast = p.scale_vec && (p.kbytes % kSlabBytes == 0);
    if (fast) return launch_gemm_impl<FMT, TW, TM, WW, WM, EPI, true>(p, max_m_tiles, s);
    return launch_gemm_impl<FMT, TW, TM, WW, WM, EPI, false>(p, max_m_tiles, s);
}

struct TileChoice {
    int tw, tm, waves;
};
constexpr int kRing = 6;               // `waves` of a tile of the ring kernel

#ifdef CMX_TEST_HOOKS
TileChoice g_force_tile = {0, 0, 0};   // tw == 0 -> heuristic
int g_pretiled_tile_rows = 0;          // 0 -> heuristic
#else
constexpr TileChoice g_force_tile = {0, 0, 0};
constexpr int g_pretiled_tile_rows = 0;
#endif

#ifdef CMX_TEST_HOOKS
KsplitTile g_force_ksplit = {0, 0, 0};   // fw == 0 -> heuristic, fw < 0 -> never
#else
constexpr KsplitTile g_force_ksplit = {0, 0, 0};
#endif
// whether the test build takes the choice of a split-K tile away from the heuristic, and with what
bool ksplit_is_forced(KsplitTile* out) {
    *out = g_force_ksplit.fw > 0 ? g_force_ksplit : KsplitTile{0, 0, 0};
    return g_force_ksplit.fw != 0 || g_force_tile.tw != 0 || g_disable_dl;
}

// Dense 8-bit problems that 128 x 128 tiles of four wavefronts (mx_gemm_dl_kernel) take: K of 128, 256 or 384, too many 64 x 64 tiles
// for the split-K kernel to run in two rounds of a workgroup per CU, few enough 128 x 128 tiles for one.  From K = 512 on it is the ring
// kernel that takes these sizes (a row of scales shorter than 16 bytes goes to its LDS through registers: 1024 x 4096 x 256 9.0
// here, 13.6 there).
// The alignment of the scale rows does not enter, because it must not change the sums.
bool takes_128_tile(uint32_t m, uint32_t n, int fmt, uint32_t kblocks, int cus) {
    if (fmt == CMX_FMT_E2M1 || kblocks % 4 != 0 || kblocks >= 16) return false;
    const uint64_t t64 = (uint64_t)ceil_div(n, 64) * ceil_div(m, 64), t128 = (uint64_t)ceil_div(n, 128) * ceil_div(m, 128);
    return t128 <= (uint64_t)cus && t64 > 2 * (uint64_t)cus;
}

// Dense 8-bit problems that the ring kernel (mx_gemm_ring.hip) takes, and the height of its tile (0: none): more 64 x 64 tiles than
// the split-K kernel runs in two rounds of a workgroup per CU, and few enough tiles of 128 x 128, 192 or 256 for one round of
// the ring kernel's.  Its sums are the 256-row kernels' (one chain over K), so the limit to those is a matter of time only; the limit
// to split-K (whose sums differ in the last bits) goes by sizes alone.
// Measured (us, E4M3, bf16 out, operands of three calls in turn; split-K 64 x 64 or 256-row kernels -> ring; on weights stored [K, N] the
// other kernels need a pass of 4 (K = 512) to 9 (K = 4096) before them):
//   n = 4096:      K = 512         1024            2048            4096
//   m = 512    7.0 against 7.1  8.6    8.6     11.8   12.0     17.6   18.7       split-K stays
//   768       10.1 ->  7.4     12.8 ->  9.2    17.2 -> 12.7    25.4 -> 19.9       128
//   1024      11.8 ->  7.8     15.4 ->  9.6    20.4 -> 13.2    31.5 -> 21.4       128
//   1280      12.1 ->  9.0     15.9 -> 10.9    23.4 -> 15.4    38.9 -> 25.1       192
//   1536      12.1 ->  9.4     15.9 -> 11.3    23.5 -> 16.2    38.7 -> 26.8       192
//   2048      12.5 -> 11.0     16.6 -> 13.8    24.3 -> 20.6    39.7 -> 34.4       256
// On weights stored [K, N], the 256-row kernels with their pass / split-K 64 x 64 in place / ring:
//   n = 4096:      K = 512             1024                2048                4096                7168
//   m = 768    16.6 11.5  7.7    21.9 15.1  9.7    33.0 20.9 13.3    54.1 32.8 21.0     90.7  50.5 32.4
//   1024       16.7 13.2  8.0    22.1 17.4 10.5    33.0 24.6 14.0    53.7 39.5 21.8     90.6  63.6 34.5
//   1536       17.1 18.3  9.4    23.5 24.0 12.2    34.6 34.0 17.1    54.6 55.8 27.4     89.3  94.6 44.2
//   2048       17.1 22.9 11.2    23.2 30.4 14.3    34.1 43.2 20.9    54.2 69.6 33.2     88.8 121.7 54.4
// Past one round the 256-row kernels are the faster ones (2560 x 4096, ring in two rounds: K = 1024 24.8 against 16.6, 4096 57.4 against 43.2).
int ring_rows(uint32_t m, uint32_t n, int fmt, uint32_t kblocks, int cus) {
    if (fmt == CMX_FMT_E2M1 || kblocks % 4 != 0 || kblocks < 16) return 0;
    if ((uint64_t)ceil_div(n, 64) * ceil_div(m, 64) <= 2 * (uint64_t)cus) return 0;
    const auto one_round = [&](uint32_t tm) { return (uint64_t)ceil_div(n, 128) * ceil_div(m, tm) <= (uint64_t)cus; };
    return one_round(128) ? 128 : (one_round(192) ? 192 : (one_round(256) ? 256 : 0));
}

// Whether a problem goes to the split-K kernels (mx_gemm_ksplit.hip), and with which tile; fw == 0: no.  The choice depends
// on sizes, element format and the number of CUs only, so that every layout, pitch and output type of a problem gets the same sums.
// Dense: the smallest tile that still leaves every CU at most one workgroup (time goes with the bytes a workgroup pulls
// through its vector cache, and a second round costs as much as the first); past that 64 x 64 tiles, two workgroups of
// four wavefronts on a CU, up to 1024 tiles.  Measured (us, E4M3, before = 256-row tiles): 16 x 4096 x 7168 44.7 -> 9.0,
// 64 x 4096 x 7168 49.2 -> 10.8, 256 x 4096 x 7168 62.5 -> 18.0, 512 x 4096 x 7168 62.5 -> 28.1, 640 x 4096 x 4096 (640
// tiles) 38.7 -> 28.4, 2048 x 4096 x 7168 (2048 tiles) 63.4 against 99.3; 1000 x 1000 x 960 37.6 -> 7.7.  Scale rows that are no
// whole 16-byte pieces or not aligned to them cost next to nothing (700 x 3000 x 1984, 62 scales a row: 36.0 with a dword
// of scales at a time, 19.8 with pieces).
// 8-bit problems whose K is no whole number of slabs are left to the register-staged 256-row kernel, slower by two to four
// times than the streaming ones, so they stay here up to 2048 tiles (us, 256-row -> here): 2048 x 4096 x 6976 240 -> 117, 1536 x
// 4096 x 3040 75 -> 47; 3000 x 5000 x 4064 (3713 tiles) 97 against 138, 8192 x 4096 x 7136 300 against 463.
int choose_ksplit(uint32_t m, uint32_t n, int fmt, uint32_t kblocks, KsplitTile* out) {
    if (ksplit_is_forced(out)) return CMX_OK;
    const auto fits = [&](const KsplitTile& t) { return ksplit_lds_bytes(t, fmt, kblocks) <= kKsplitMaxLds; };
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    const auto tiles = [&](const KsplitTile& t) { return (uint64_t)ceil_div(n, 16 * t.fw) * ceil_div(m, 16 * t.fm); };
    for (const KsplitTile& t : {KsplitTile{1, 1, 8}, KsplitTile{1, 2, 8}, KsplitTile{2, 1, 8}, KsplitTile{2, 2, 8}, KsplitTile{4, 1, 8},
                                KsplitTile{2, 4, 8}, KsplitTile{4, 2, 8}, KsplitTile{4, 4, 8}})
        if (tiles(t) <= (uint64_t)cus && fits(t)) {
            *out = t;
            return CMX_OK;
        }
    const KsplitTile t = {4, 4, 4};
    const uint64_t per_cu = fmt != CMX_FMT_E2M1 && kblocks % 4 != 0 ? 8 : 4;
    if (tiles(t) <= per_cu * cus && !takes_128_tile(m, n, fmt, kblocks, cus) && ring_rows(m, n, fmt, kblocks, cus) == 0 && fits(t)) *out = t;
    return CMX_OK;
}

// Grouped problems on the split-K kernels: their tile (fw == 0: none of the groups), and the largest group that they take
// (0: groups of any size).
struct GroupedKsplit {
    KsplitTile tile;
    uint32_t small_rows;
    KsplitWeights weights;
};
constexpr uint32_t kSmallGroupRows = 64;               // one m-tile of the 64 x 64 tile

// Groups that average few rows stream their weights once whatever the tile; 64 x 64 tiles of four wavefronts keep more of
// the stream in flight than the 256-row tiles.  An average says little about the groups, though, and a group of many
// m-tiles of 64 rows reads its weights as many times.  So beyond four 64 x 64 tiles per CU (up to there the split-K kernel is the
// faster one also where all rows are one group's) the groups are told apart on the device: those of one m-tile go to the
// split-K kernel, the others, in a second launch, to the 256-row kernel that the average selects.
// Measured (us, K = 7168, N = 4096, 256 experts unless noted; 256-row kernels alone / split-K alone, weights streamed where the average
// is at most 32 / this rule):
//   rows per expert               E4M3 SwiGLU         pre-tiled           INT8
//   8 each                        1402  1082  1081    1251  1102  1105    1728  1104  1106
//   40 each                       1464  1413  1265    1316  1329  1180    1762  1427  1398
//   32 on average, random         1448  1220  1207    1281  1140  1145    1723  1317  1299
//   32 on average, Zipf           1535  1505  1355    1369  1409  1210    1795  1520  1274
//   8192 rows on 8 experts         305   565   314     206   530   210     223   561   227
//   2048 rows on 2 experts          73   144    76      90   128    95      83   140    89
//   32 experts, 512 rows on 1       57    42    40      84    37    36      77    40    39
//   32 experts, 1024 rows on 4      59    82    55      85    78    50      75    79    54
//   32 experts, 1280 rows on 4      56    69    59      91    60    92      78    66    81
// (256-row kernel: the three-slot 256 x 128 kernel for E4M3 SwiGLU, 256 x 256 tiles for INT8.  Since ring_groups has put the ring's tiles in their
// place the rule's column reads, E4M3 SwiGLU and INT8: 32 on average, Zipf 1315 and 1326; 8192 rows on 8 experts 256 and 242 on a box where the
// 256-row kernel takes 242 too, 2048 on 2 69 and 81; 32 experts, 512 rows on 1 37 and 36, 1024 on 4 53 and 52, 1280 on 4 53 and 63.)
// The empty one of the two launches costs 2-6 us.  A limit of 32 or 40 rows instead of 64: 1360 or 1308 against 1214 (random), 1349 or
// 1298 against 1352 (Zipf).  8-bit problems whose K is no whole number of slabs go by size only past the 2048 tiles up to which the
// split-K kernel beats the register-staged one (choose_ksplit).  Row-major and pre-tiled weights go by one rule, because they
// promise the same bits.
// The averages up to which this pays (32 experts, rows each; 256-row -> split-K): 36 rows E4M3 190 -> 164, pre-tiled 177 -> 162, INT8 220 ->
// 178; 40 rows 191 -> 165, 178 -> 165, 221 -> 186; with cached weights 48 rows 193 -> 181, 176 against 181, 241 -> 184; 64 rows 197 ->
// 195, 177 against 191, 234 -> 194: from there on it is the pre-tiled kernel that would lose.
// FP4: split-K alone is the faster side at every one of these distributions (8192 rows on 8 experts 358 -> 257, Zipf 1063 -> 802, 32
// experts at 64 rows 129 -> 107, at 128 rows 202 against 200), so it takes all groups in one launch.
// Weights are streamed without a look at the group where all groups are one m-tile, and in small problems of few rows on
// average, where the look would cost more (32 tokens of 256 experts 1101 -> 1110) than the rare larger group loses.
int choose_grouped_ksplit(uint32_t m_total, uint32_t groups, uint32_t n, int fmt, uint32_t kblocks, GroupedKsplit* out) {
    out->small_rows = 0;
    out->weights = KsplitWeights::kByGroup;
    if (ksplit_is_forced(&out->tile) || g_pretiled_tile_rows != 0) return CMX_OK;
    const KsplitTile t = {4, 4, 4};
    if (ceil_div(m_total, groups) > (fmt == CMX_FMT_E2M1 ? 64u : 40u) || ksplit_lds_bytes(t, fmt, kblocks) > kKsplitMaxLds) return CMX_OK;
    out->tile = t;
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    const uint64_t tiles = (uint64_t)ceil_div(n, 64) * ceil_div(m_total, 64), per_cu = kblocks % 4 != 0 ? 8 : 4;
    if (fmt != CMX_FMT_E2M1 && tiles > per_cu * cus && m_total > kSmallGroupRows) out->small_rows = kSmallGroupRows;
    if (out->small_rows != 0 || (tiles <= 2 * (uint64_t)cus && ceil_div(m_total, groups) <= 32)) out->weights = KsplitWeights::kStreamed;
    return CMX_OK;
}

// waves: at 256 x 256 "4" and "5" select the hand-scheduled kernel in its 2 x 2 and 4 x 1 wavefront layouts
// when the problem is eligible for it (8-bit elements, whole 512-byte K blocks).  2 x 2 reads a fifth less
// from the LDS per slab and is the faster one on full tiles; grouped problems whose groups average less
// than two tiles of rows take 4 x 1, where every wavefront shares in whatever rows a ragged tile has
// (measured: 16 groups of ~2048 rows 891 vs 918 us in favour of 2 x 2, 256 groups of ~256 rows 4.33 vs
// 4.38 ms in favour of 4 x 1).  FP4 has its own hand-scheduled kernel in the same two layouts (K a multiple of 512
// elements; 16 groups of ~2048 rows at K = 7168, N = 4096: 2 x 2 persistent 565 us, one tile per workgroup 2 x 2
// 635 us and 4 x 1 700 us, the eight-wavefront streaming kernel, which takes every other FP4 problem, 750 us).
TileChoice choose_tile(uint32_t m_hint, uint32_t n, int fmt, bool grouped) {
    if (g_force_tile.tw) return g_force_tile;
    // short problems stream their weights once: the three-slot 256 x 128 kernel keeps two slabs in flight
    if (m_hint <= 128 && fmt != CMX_FMT_E2M1) return {256, 128, 5};
    // (FP4, and of that what the split-K kernels leave: dense problems of more than 1024 of their tiles, rows of scales beyond the LDS)
    if (m_hint <= 64) return {256, 64, 4};
    if (m_hint <= 128) return {256, 128, 8};
    return {256, 256, grouped && m_hint < 512 ? 5 : 4};
}

// 16-bit output whose rows start at whole 16-byte pieces takes the lean store epilogue, and with it the persistent kernels
bool lean_store(const GemmParams& p) {
    return p.out_type != CMX_OUT_FP32 && p.n % 8 == 0 && p.ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0;
}
// Whether launch_tile takes a grouped problem to a persistent kernel that scans the group sizes by itself.
bool scans_groups(const GemmParams& p, const TileChoice& t, int fmt, bool swiglu) {
    if (g_disable_dl || p.w_pretiled || t.tw != 256 || t.tm != 256 || t.waves != 4 || !p.scale_vec16) return false;
    if (swiglu) return p.act_bf16 == nullptr && p.kbytes % (4 * kSlabBytes) == 0;
    return fmt == CMX_FMT_E2M1 && lean_store(p) && p.kbytes % (2 * kSlabBytes) == 0;
}

// Eight-wavefront shapes exist only as streaming kernels; when a problem is not eligible for
// streaming (ragged K, unaligned scale rows) the four-wavefront register-staged kernel of the same
// tile takes over.
template <int FMT, int TW, int TM, int EPI>
int launch_tile(const GemmParams& p, int waves, uint32_t max_m_tiles, hipStream_t s) {
    const bool stream_ok = !g_disable_dl && p.scale_vec && p.kbytes % kSlabBytes == 0;
    if constexpr (TW == 256 && TM == 256 && FMT != CMX_FMT_E2M1) {
        // whole four-slab scale blocks, fetched 16 bytes per row: K a multiple of 512 bytes, 16-byte aligned scale rows
        if ((waves == 4 || waves == 5) && stream_ok && p.scale_vec16 && p.kbytes % (4 * kSlabBytes) == 0) {
            // plain 16-bit output with 8-element-aligned rows takes the lean store epilogue and with it the persistent kernel
            constexpr int kLeanBf16 = EPI == kEpiStore ? kEpiStoreBf16 : EPI, kLeanFp16 = EPI == kEpiStore ? kEpiStoreFp16 : EPI;
            const bool lean = EPI == kEpiStore && lean_store(p);
            // (the 4 x 1 layout with the lean store epilogue does not fit the register file without spilling
            // inside the loop, so the persistent store kernel is always 2 x 2)
            if (lean && p.out_type == CMX_OUT_BF16) return launch_gemm_pipe<FMT, kLeanBf16, 256, 2, 2, 2>(p, max_m_tiles, s);
            if (lean) return launch_gemm_pipe<FMT, kLeanFp16, 256, 2, 2, 2>(p, max_m_tiles, s);
            if constexpr (EPI == kEpiSwigluQuant)
                if (waves == 4 && p.sizes != nullptr) return launch_gemm_pipe<FMT, EPI, 256, 2, 2, 2, true>(p, max_m_tiles, s);
            if (waves == 4) return launch_gemm_pipe<FMT, EPI, 256, 2, 2, 2>(p, max_m_tiles, s);
            return launch_gemm_pipe<FMT, EPI, 256, 4, 1, 2>(p, max_m_tiles, s);
        }
    }
    if constexpr (TW == 256 && TM == 256 && FMT == CMX_FMT_E2M1) {
        // hand-scheduled FP4 kernel: whole two-slab scale blocks (K a multiple of 512 elements), 16-byte aligned scale rows
        if ((waves == 4 || waves == 5) && stream_ok && p.scale_vec16 && p.kbytes % (2 * kSlabBytes) == 0) {
            if constexpr (EPI == kEpiStore) {
                // plain 16-bit output with 8-element-aligned rows: lean store epilogue, persistent kernel
                const bool lean = lean_store(p);
                // (unlike the 8-bit kernel, whose fragments take twice the registers, the 4 x 1 layout fits here too)
                if (lean && waves == 4 && p.sizes != nullptr)
                    return p.out_type == CMX_OUT_BF16 ? launch_gemm_pipe_fp4<kEpiStoreBf16, 2, 2, true>(p, max_m_tiles, s) : launch_gemm_pipe_fp4<kEpiStoreFp16, 2, 2, true>(p, max_m_tiles, s);
                if (lean && waves == 4 && p.out_type == CMX_OUT_BF16) return launch_gemm_pipe_fp4<kEpiStoreBf16, 2, 2>(p, max_m_tiles, s);
                if (lean && waves == 4) return launch_gemm_pipe_fp4<kEpiStoreFp16, 2, 2>(p, max_m_tiles, s);
                if (lean && p.out_type == CMX_OUT_BF16) return launch_gemm_pipe_fp4<kEpiStoreBf16, 4, 1>(p, max_m_tiles, s);
                if (lean) return launch_gemm_pipe_fp4<kEpiStoreFp16, 4, 1>(p, max_m_tiles, s);
                if (waves == 4) return launch_gemm_pipe_fp4<EPI, 2, 2>(p, max_m_tiles, s);
                return launch_gemm_pipe_fp4<EPI, 4, 1>(p, max_m_tiles, s);
            }
        }
    }
    if constexpr (TW == 256 && TM == 128 && FMT != CMX_FMT_E2M1) {
        if (waves == 5 && stream_ok) return launch_gemm_pipe<FMT, EPI, 128, 4, 1, 3>(p, max_m_tiles, s);
    }
    if constexpr (TM >= 128) {
        // the four-wavefront streaming kernel of the 256 x 256 tile runs out of registers: eight there
        if ((waves == 8 || (TW == 256 && TM == 256)) && stream_ok) return launch_gemm_dl<FMT, TW, TM, 2, 4, EPI>(p, max_m_tiles, s);
    }
    constexpr int WW = TM >= 128 ? 2 : 4, WM = TM >= 128 ? 2 : 1;
    return launch_gemm<FMT, TW, TM, WW, WM, EPI>(p, max_m_tiles, s);
}

template <int FMT, int EPI>
int dispatch_tile(const GemmParams& p, TileChoice t, uint32_t max_m_tiles, hipStream_t s) {
    if (t.tw == 256 && t.tm == 256) return launch_tile<FMT, 256, 256, EPI>(p, t.waves, max_m_tiles, s);
    if (t.tw == 256 && t.tm == 128) return launch_tile<FMT, 256, 128, EPI>(p, t.waves, max_m_tiles, s);
    if (t.tw == 256 && t.tm == 64) return launch_tile<FMT, 256, 64, EPI>(p, t.waves, max_m_tiles, s);
    if (t.tw == 128 && t.tm == 128) return launch_tile<FMT, 128, 128, EPI>(p, t.waves, max_m_tiles, s);
    set_error("unsupported tile shape");
    return CMX_EINVAL;
}

// Pre-tiled weights (cmx_mx_pretile_weights): only the weights-to-registers kernel reads that order, so a problem it
// cannot take is an error, not a reason to fall back.
int check_pretiled(const GemmParams& p, int fmt, bool swiglu) {
    CMX_REQUIRE(fmt == CMX_FMT_E4M3 || fmt == CMX_FMT_E5M2, "pre-tiled weights: 8-bit element formats only");
    CMX_REQUIRE(p.kbytes % (4 * kSlabBytes) == 0, "pre-tiled weights: k must be a multiple of 512");
    CMX_REQUIRE(p.scale_vec16, "pre-tiled weights: scale rows of both operands must be 16-byte aligned");
    // (with the bf16 activation output on top, the SwiGLU epilogue no longer fits the register file beside the weight ring)
    CMX_REQUIRE(!swiglu || p.act_bf16 == nullptr, "pre-tiled weights: no bf16 activation output (act_bf16 must be NULL)");
    CMX_REQUIRE(swiglu || (p.out_type != CMX_OUT_FP32 && p.n % 8 == 0 && p.ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0),
                "pre-tiled weights: 16-bit output, n and ldc multiples of 8, c 16-byte aligned");
    return CMX_OK;
}

template <int TM>
int launch_pretiled(const GemmParams& p, int fmt, bool swiglu, uint32_t max_m_tiles, hipStream_t s) {
    if (swiglu) return launch_gemm_wreg<CMX_FMT_E4M3, kEpiSwigluQuant, TM>(p, max_m_tiles, s);
    if (fmt == CMX_FMT_E4M3) {
        if (p.out_type == CMX_OUT_BF16) return launch_gemm_wreg<CMX_FMT_E4M3, kEpiStoreBf16, TM>(p, max_m_tiles, s);
        return launch_gemm_wreg<CMX_FMT_E4M3, kEpiStoreFp16, TM>(p, max_m_tiles, s);
    }
    if (p.out_type == CMX_OUT_BF16) return launch_gemm_wreg<CMX_FMT_E5M2, kEpiStoreBf16, TM>(p, max_m_tiles, s);
    return launch_gemm_wreg<CMX_FMT_E5M2, kEpiStoreFp16, TM>(p, max_m_tiles, s);
}

int check_operands(const void* a, uint32_t lda, const void* as, uint32_t ld_as, const void* w, uint32_t ldw,
                   const void* ws, uint32_t ld_ws, uint32_t k, int fmt) {
    CMX_REQUIRE(a && as && w && ws, "null pointer");
    CMX_REQUIRE(fmt == CMX_FMT_E4M3 || fmt == CMX_FMT_E5M2 || fmt == CMX_FMT_E2M1, "unknown element format");
    CMX_REQUIRE(k > 0 && k % 32 == 0, "k must be a positive multiple of 32");
    const uint32_t kbytes = fmt == CMX_FMT_E2M1 ? k / 2 : k;
    CMX_REQUIRE(lda >= kbytes && ldw >= kbytes, "operand row pitch smaller than a row");
    CMX_REQUIRE(lda % 16 == 0 && ldw % 16 == 0 && aligned16(a) && aligned16(w), "operand rows must be 16-byte aligned");
    CMX_REQUIRE(ld_as >= k / 32 && ld_ws >= k / 32, "scale row pitch smaller than a row");
    return CMX_OK;
}

bool scales_aligned16(const void* as, uint32_t ld_as, const void* ws, uint32_t ld_ws) {
    return ld_as % 16 == 0 && ld_ws % 16 == 0 && (reinterpret_cast<uintptr_t>(as) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(ws) & 15u) == 0;
}

bool scales_dword_aligned(const void* as, uint32_t ld_as, const void* ws, uint32_t ld_ws) {
    return ld_as % 4 == 0 && ld_ws % 4 == 0 && (reinterpret_cast<uintptr_t>(as) & 3u) == 0 &&
           (reinterpret_cast<uintptr_t>(ws) & 3u) == 0;
}

}  // namespace

}  // namespace cmx

#ifdef CMX_TEST_HOOKS
extern "C" int cmx_debug_disable_streaming(int off) {
    cmx::g_disable_dl = off != 0;
    return CMX_OK;
}

// pin the tile height (256 or 288 rows) of every later matmul call on pre-tiled weights (0 restores the heuristic)
extern "C" int cmx_debug_pretiled_tile_rows(int rows) {
    cmx::g_pretiled_tile_rows = rows == 256 || rows == 288 ? rows : 0;
    return CMX_OK;
}

// pin the split-K tile of every later matmul call (fw = 0 restores the heuristic, fw < 0 keeps every problem off those kernels)
extern "C" int cmx_debug_force_ksplit(int fw, int fm, int waves) {
    cmx::g_force_ksplit = {fw, fm, waves};
    return CMX_OK;
}

// pin the tile shape and wavefront count of every later matmul call (tw = 0 restores the heuristic)
extern "C" int cmx_debug_force_tile(int tw, int tm, int waves) {
    cmx::g_force_tile = (tw > 0 && tm > 0) ? cmx::TileChoice{tw, tm, waves > 0 ? waves : 4} : cmx::TileChoice{0, 0, 0};
    return CMX_OK;
}
#endif

namespace cmx {
namespace {
int ring_gemm(GemmParams& p, const RingTile& t, int fmt, bool k_slow, hipStream_t s) {
    p.w_tiles = ceil_div(p.n, t.tw);
    return launch_ring(p, t, fmt, kEpiStore, k_slow, ceil_div(p.m, t.tm), s);
}
}  // namespace
}  // namespace cmx

extern "C" int cmx_mx_gemm(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b,
                           uint32_t ldb, const uint8_t* b_scale, uint32_t ld_bs, void* c, uint32_t ldc, uint32_t m,
                           uint32_t n, uint32_t k, int fmt, int out_type, cmx_stream_t stream) {
    using namespace cmx;
    if (m == 0 || n == 0) return CMX_OK;
    int rc = check_operands(a, lda, a_scale, ld_as, b, ldb, b_scale, ld_bs, k, fmt);
    if (rc != CMX_OK) return rc;
    CMX_REQUIRE(c && ldc >= n, "bad output");
    CMX_REQUIRE(out_type == CMX_OUT_BF16 || out_type == CMX_OUT_FP16 || out_type == CMX_OUT_FP32, "unknown output type");
    GemmParams p{};
    p.a = a; p.a_scale = a_scale; p.w = b; p.w_scale = b_scale; p.c = c;
    p.lda = lda; p.ld_as = ld_as; p.ldw = ldb; p.ld_ws = ld_bs; p.ldc = ldc;
    p.m = m; p.n = n; p.kbytes = fmt == CMX_FMT_E2M1 ? k / 2 : k; p.kblocks = k / 32;
    p.groups = 1; p.out_type = out_type;
    p.scale_vec = scales_dword_aligned(a_scale, ld_as, b_scale, ld_bs);
    p.scale_vec16 = scales_aligned16(a_scale, ld_as, b_scale, ld_bs);
    CMX_REQUIRE((uint64_t)n * ldb < (1ull << 32) && (uint64_t)lda * 256 < (1ull << 32), "operand tile exceeds 32-bit offsets");
    hipStream_t s = static_cast<hipStream_t>(stream);
    KsplitTile ks;
    if (rc = choose_ksplit(m, n, fmt, p.kblocks, &ks); rc != CMX_OK) return rc;
    if (ks.fw != 0) {
        p.w_tiles = ceil_div(n, 16 * ks.fw);
        return launch_ksplit(p, ks, fmt, kEpiStore, ceil_div(m, 16 * ks.fm), KsplitWeights::kCached, s);
    }
    int cus = 0;
    if (rc = cu_count(&cus); rc != CMX_OK) return rc;
    TileChoice t = choose_tile(m, n, fmt, false);
    if (!g_force_tile.tw && !g_disable_dl) {
        if (const int tm = ring_rows(m, n, fmt, p.kblocks, cus)) return ring_gemm(p, {128, tm}, fmt, false, s);
        if (takes_128_tile(m, n, fmt, p.kblocks, cus)) t = {128, 128, 4};
    }
    if (t.waves == kRing) return ring_gemm(p, {t.tw, t.tm}, fmt, false, s);
    p.w_tiles = ceil_div(n, t.tw);
    const uint32_t m_tiles = ceil_div(m, t.tm);
    switch (fmt) {
        case CMX_FMT_E4M3: return dispatch_tile<CMX_FMT_E4M3, kEpiStore>(p, t, m_tiles, s);
        case CMX_FMT_E5M2: return dispatch_tile<CMX_FMT_E5M2, kEpiStore>(p, t, m_tiles, s);
        default: return dispatch_tile<CMX_FMT_E2M1, kEpiStore>(p, t, m_tiles, s);
    }
}

namespace cmx {
namespace {
// Split-K problems on weights stored [k, n]: a tile of 64 columns takes half a line from each of its K rows, 128 a slab where K-contiguous
// rows take 64 lines, and its time goes with K; the pass that rewrites the weights costs a launch and goes with k * n.  Measured (us,
// with the pass -> as they lie): 16 x 4096 x 7168 26.3 -> 19.2, 64 28.5 -> 18.3, 256 36.1 -> 23.5, 512 46.7 -> 33.9; 16 x 8192 x 512 9.6 -> 5.1;
// 16 x 7168 x 2048 16.4 -> 9.3; 64 x 2052 x 2048 13.1 -> 8.4; 64 x 512 x 4096 11.1 -> 8.3; 64 x 2048 x 8192 22.0 -> 16.3; but 64 x 1024 x 8192 13.0
// against 17.3, 64 x 512 x 8192 13.4 against 17.3, 700 x 1536 x 8192 37 against 46.
// `ks`: the tile on K-contiguous weights.  Two lines inside of that: tiles of 16 columns x 32 rows that fill three quarters of the CUs are hard to beat
// behind a short pass (100 x 1024 at K = 3584 10.1 against 11.2, 4096 10.4 against 12.9, but 100 x 768 x 4096, 192 tiles, 11.9 -> 11.5), and past
// K = 7168 the scales of a 64 x 64 tile leave room for one workgroup per CU instead of two (K = 8192, 700 x 2048 41.1 against 41.7,
// 400 x 2560 40.8 against 45.4, 700 x 2816 45.5 -> 43.3, 700 x 4096 66 -> 39).
bool k_slow_pays(uint32_t m, uint32_t n, uint32_t k, const KsplitTile& ks, int cus) {
    KsplitTile t;
    if (ksplit_is_forced(&t)) return true;
    if (k <= 4096) return !(k > 3328 && ks.fw == 1 && ks.fm == 2 && (uint64_t)ceil_div(n, 16) * ceil_div(m, 32) * 4 > 3 * (uint64_t)cus);
    return (uint64_t)n * k >= (k > 7168 && ks.waves == 4 ? 22u << 20 : 16u << 20);
}
}  // namespace
}  // namespace cmx

// cmx_mx_gemm on weights stored [k, n] with scales [k / 64, n, 2], where a kernel reads them as they lie: `taken` says whether
// one does (the caller has them rewritten otherwise).  The sums are those of the same problem on K-contiguous weights.
int cmx::gemm_k_slow(const uint8_t* a, const uint8_t* a_scale, const uint8_t* b, const uint8_t* b_scale, void* c, uint32_t ldc, uint32_t m,
                     uint32_t n, uint32_t k, int fmt, int out_type, hipStream_t s, bool* taken) {
    *taken = false;
    if (!(fmt == CMX_FMT_E4M3 || fmt == CMX_FMT_E5M2) || k % kSlabBytes != 0) return CMX_OK;
    // 16-byte pieces of a row start at any dword; the matrix ends in a piece of its own
    if (n % 4 != 0 || n < 16 || (reinterpret_cast<uintptr_t>(b) & 3u) != 0 || (uint64_t)k * n >= (1ull << 32)) return CMX_OK;
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    // the kernel that the same problem gets on K-contiguous weights: split-K, or one whose sums the ring kernel gives
    KsplitTile ks;
    if (int rc = choose_ksplit(m, n, fmt, k / 32, &ks); rc != CMX_OK) return rc;
    int tm = 0;
    if (ks.fw != 0) {
        if (!k_slow_pays(m, n, k, ks, cus) || !ksplit_k_slow_tile(&ks, m, n, fmt, k / 32, cus)) return CMX_OK;
    } else {
        tm = g_force_tile.waves == kRing ? g_force_tile.tm : (g_force_tile.tw || g_disable_dl ? 0 : ring_rows(m, n, fmt, k / 32, cus));
        if (tm == 0) return CMX_OK;
    }
    CMX_REQUIRE(a && a_scale && b && b_scale && aligned16(a), "operand rows must be 16-byte aligned");
    CMX_REQUIRE(c && ldc >= n, "bad output");
    CMX_REQUIRE(out_type == CMX_OUT_BF16 || out_type == CMX_OUT_FP16 || out_type == CMX_OUT_FP32, "unknown output type");
    CMX_REQUIRE((uint64_t)k * 256 < (1ull << 32), "operand tile exceeds 32-bit offsets");
    GemmParams p{};
    p.a = a; p.a_scale = a_scale; p.w = b; p.w_scale = b_scale; p.c = c;
    p.lda = k; p.ld_as = k / 32; p.ldw = n; p.ld_ws = 2 * n; p.ldc = ldc;
    p.m = m; p.n = n; p.kbytes = k; p.kblocks = k / 32;
    p.groups = 1; p.out_type = out_type;
    p.scale_vec = scales_dword_aligned(a_scale, p.ld_as, b_scale, p.ld_ws);
    *taken = true;
    if (tm != 0) return ring_gemm(p, {128, tm}, fmt, true, s);
    p.w_tiles = ceil_div(n, 64);
    return launch_ksplit_k_slow(p, ks, fmt, ceil_div(m, 16 * ks.fm), s);
}

extern "C" size_t cmx_mx_gmm_workspace_bytes(uint32_t groups) {
    // row offsets, m-tile prefixes of the larger and of the small groups, per-XCD tile counters
    return cmx::round_up_sz((3 * (size_t)(groups + 1) + 8) * sizeof(int32_t), 256);
}

namespace cmx {
namespace {
// The schedule metadata of a grouped problem in its workspace.
struct GroupTables {
    int32_t *row_off, *tile_pref, *small_pref, *tile_ctr;
    GroupTables(void* workspace, uint32_t groups)
        : row_off(static_cast<int32_t*>(workspace)), tile_pref(row_off + (groups + 1)), small_pref(tile_pref + (groups + 1)),
          tile_ctr(small_pref + (groups + 1)) {}
};

GroupTablesJob tables_job(const GroupTables& g, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t tile_m, uint32_t small_rows) {
    return {group_sizes, groups, tile_m, m_total, small_rows, g.row_off, g.tile_pref, g.small_pref, g.tile_ctr};
}

// Sets the parameters that say where the groups lie: their sizes, where all kernels of the call locate their tiles by them, or the
// tables for m-tiles of tile_m rows (of the groups past small_rows), filled here unless an earlier launch has.
int prepare_groups(GemmParams& p, const GroupTablesJob& job, bool by_sizes, bool filled, hipStream_t s) {
    p.small_rows = job.small_rows;
    p.group_class = job.small_rows != 0 ? kLargeGroups : kAllGroups;
    p.groups = job.groups;
    if (by_sizes) {
        p.sizes = job.sizes;
        return CMX_OK;
    }
    if (!filled)
        if (int rc = launch_group_tables(job, s); rc != CMX_OK) return rc;
    p.row_off = job.row_off;
    p.tile_pref = job.tile_pref;
    p.tile_ctr = job.tile_ctr;
    return CMX_OK;
}

// The split-K launch of a grouped problem: all groups, or those of at most ks.small_rows rows, which are one m-tile each and
// read their weights once.
int launch_grouped_ksplit(GemmParams p, const GroupTables& g, const GroupedKsplit& ks, int fmt, int epi, uint32_t m_total, hipStream_t s) {
    p.w_tiles = epi_pairs_gate_up(epi) ? ceil_div(p.n / 2, 8 * ks.tile.fw) : ceil_div(p.n, 16 * ks.tile.fw);
    if (ks.small_rows == 0)
        return launch_ksplit(p, ks.tile, fmt, epi, m_total / (16 * ks.tile.fm) + p.groups, ks.weights, s);
    p.tile_pref = g.small_pref;
    p.group_class = kSmallGroups;
    return launch_ksplit(p, ks.tile, fmt, epi, p.groups < m_total ? p.groups : m_total, ks.weights, s);
}

// most m-tiles of tile_m rows that groups of more than small_rows rows can have
uint32_t max_group_tiles(uint32_t m_total, uint32_t groups, uint32_t tile_m, uint32_t small_rows) {
    const uint32_t n = m_total / (small_rows + 1);
    return m_total / tile_m + (n < groups ? n : groups);
}

// Grouped problems on row-major weights that the ring kernel takes from the 256-row kernels of choose_tile (same sums, so the line is a
// matter of time).  128 x 128 where its tiles are one round of a workgroup per CU whatever the rows' distribution (a second round costs as
// much as the first: 16 experts x 64 rows, Zipf, K = 2048, N = 2048, 320 tiles, 30 against 23); else 256 x 128 in the place of the three-slot
// kernel of short groups, which pulls a dword of scales per row and slab; else 128 x 256 in one round.
// Measured (us, before -> ring; SwiGLU + requant / 16-bit store; u: routes drawn uniformly, z: Zipf):
//   128 x 128    8 experts x 64 rows u, K = 1024, N = 1024   14.6 -> 13.9 / 18.3 -> 13.7    x 200 z   22.1 -> 14.3 / 19.7 -> 14.5
//                8 x 100 u, 4096, 2048                       35.7 -> 25.0 / 40.1 -> 25.4    16 x 64 z, 7168, 1024   56.8 -> 36.8 / 61.5 -> 36.7
//   256 x 128    32 x 100 u, 7168, 4096                      206 -> 190 / 221 -> 204        32 x 128 z   320 -> 279 / 327 -> 284
//                SwiGLU 32 x 100 u, K = 1024, N = 2048 21.5 -> 18.5, 4096 36.9 -> 35.8; 2048, 4096 61.2 -> 54.8; 64 x 90 z, 2048, 2048 71.9 -> 66.9; below K = 1536
//                only up to eight rounds: 64 x 110 u, 1024, 4096 83.6 -> 82.5, but 128 x 70, 1024, 4096 u 138.7 against 141.1, z 165.2 against 171.0; 256 x 50 u, 1024,
//                2048 136.8 against 140.7; 128 x 90 z, 1152, 4096 199.8 against 206.8 (K = 1536, 128 x 70 u 190.8 and 191.5).  Between two and eight rounds
//                it is within -3 and +4 % there (K = 1024: 32 x 70 z 42.3 and 42.7, 64 x 60 z, 2048 42.9 and 41.7, 64 x 70 u 66.3 and 69.1); below K = 1024 not measured
//   128 x 256    8 x 200 u, 4096, 2048                       45.9 -> 34.5 / 43.1 -> 35.7    16 x 300 u, 7168, 1024   74 -> 57 / 69 -> 62
//                8 x 500 u, 1024, 1024                       22.6 -> 18.6 / 19.4 -> 12.9; store 8 x 200 u, 512, 2048 15.3 -> 9.6, 16 x 300 u, 512, 1024 16.5 -> 11.3
// Where n is at most 128, half of a 256-row tile would be empty: 128 x 128 for 256 x 128 (SwiGLU 256 x 68 z, 3072, 64 45 -> 34 where 256 x 128 takes
// 48; FP4 256 x 128 u, 512, 64 20 -> 16, 23).
// Problems of more tiles stay on the persistent kernels (32 x 194 rows, 7168, 4096: 287 against 311 with 128 x 256).
// INT8, whose other kernels have 256 x 256 tiles (us, fp32 output; the faster of the persistent and the streaming one -> ring):
//   128 x 128    8 x 44 u, 4096, 2048 43.4 -> 17.6     16 x 100 z, 7168, 1024 70.2 -> 30.4
//   256 x 128    32 x 44 u, 7168, 4096 223 -> 174       32 x 100 z 284 -> 213      32 x 100 z, 1152, 2048 41.7 -> 30.4: from K = 512 on, and where the device
//                chooses it (mx_gemm_i8_short_kernel)
//   128 x 256    16 x 200 u, 7168, 1024 70.7 -> 42.7    8 x 200 u, 4096, 2048 45.6 -> 28.5    8 x 500 u, 1024, 1024 20.3 -> 15.5    16 x 300 u, 512, 1024 16.5 -> 13.9;
//                of more than a round 32 x 200 u, 7168, 4096 281 against 247, 16 x 2048 1062 against 889
// FP4, whose other kernels past the split-K sizes have tiles of 256 x 128 and 256 x 256 (us, bf16 output):
//   128 x 128    8 x 70 u, 4096, 2048 31.6 -> 15.9     8 x 200 u 36.0 -> 18.4     16 x 100 z, 7168, 1024 46.9 -> 24.1     8 x 70 u, 7168, 4096 49 -> 26
//   256 x 128    32 x 70 u, 7168, 4096 144 -> 111       32 x 100 z 196 -> 141      32 x 100 z, 1280, 2048 29.9 -> 26.9
//   128 x 256    8 x 200 u, 7168, 4096 56.7 -> 40.6; of more than a round 32 x 200 u, 7168, 4096 180 against 148
int ring_groups(TileChoice* t, uint32_t m_total, uint32_t groups, uint32_t n, int fmt, uint32_t kblocks, bool swiglu) {
    if (kblocks % (fmt == CMX_FMT_E2M1 ? 8 : 4) != 0 || (fmt != kFmtI8 && kblocks < 16)) return CMX_OK;
    const bool eight_bit = fmt == CMX_FMT_E4M3 || fmt == CMX_FMT_E5M2;
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    const uint64_t w128 = ceil_div(n, 128);
    const bool short_k = eight_bit && swiglu && kblocks < 48, many = (uint64_t)ceil_div(n, 256) * (m_total / 128 + groups) > 8 * (uint64_t)cus;
    const uint32_t k_min = eight_bit && swiglu ? 32 : 16;
    if (w128 * (m_total / 128 + groups) <= (uint64_t)cus) *t = {128, 128, kRing};
    else if (t->tm <= 128 && kblocks >= k_min && !(short_k && many)) *t = {w128 == 1 ? 128 : 256, 128, kRing};
    else if (t->tm == 256 && w128 * (m_total / 256 + groups * 3 / 4) <= (uint64_t)cus) *t = {128, 256, kRing};
    return CMX_OK;
}

// Which kernels a grouped problem goes to, and the rows of their m-tiles.
struct GroupPlan {
    GroupedKsplit ks;
    TileChoice t;
    bool all_ksplit() const { return ks.tile.fw != 0 && ks.small_rows == 0; }
    uint32_t tile_m() const { return all_ksplit() ? 16 * ks.tile.fm : t.tm; }
};

// Whether kernels that take one tile per workgroup locate it by the sizes themselves.  A launch that fills tables first costs 5 us; a scan at
// the start of a workgroup some 0.3 us more than the table reads, once for each round of workgroups: 32 experts x 16 rows of FP4, five
// rounds of two workgroups per CU, 93.4 us with tables and 92.4 without; INT8 of 2144 tiles, eight rounds of one per CU, no difference; FFN of
// 32 tokens, 256 experts, where the tables cost no launch, 1119 with and 1053 against 1039 of another box without.  So up to six rounds.
int tiles_by_sizes(bool* out, uint32_t groups, uint64_t max_tiles, uint32_t per_cu) {
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    *out = groups <= kInlineGroups && max_tiles <= 6 * (uint64_t)per_cu * cus;
    return CMX_OK;
}
int plan_groups(GroupPlan* plan, uint32_t m_total, uint32_t groups, uint32_t n, int fmt, uint32_t kblocks, bool swiglu, bool pretiled) {
    if (int rc = choose_grouped_ksplit(m_total, groups, n, fmt, kblocks, &plan->ks); rc != CMX_OK) return rc;
    // average rows per group steers the tile height
    plan->t = choose_tile(ceil_div(m_total, groups), n, fmt, true);
    if (!pretiled && !g_force_tile.tw && !g_disable_dl)
        if (int rc = ring_groups(&plan->t, m_total, groups, n, fmt, kblocks, swiglu); rc != CMX_OK) return rc;
    // the weights-to-registers kernel, tiles drawn from the counters: 256 x 288 when the groups average less than four
    // tiles of rows (a group of 257 to 288 rows then takes one pass over its weights instead of two), else 256 x 256
    if (pretiled) plan->t = {256, g_pretiled_tile_rows ? g_pretiled_tile_rows : (ceil_div(m_total, groups) < 1024 ? 288 : 256), 5};
    return CMX_OK;
}

int gmm_common(GemmParams& p, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, void* workspace, int fmt,
               bool swiglu, bool tables_filled, hipStream_t s) {
    CMX_REQUIRE(group_sizes && workspace, "null pointer");
    CMX_REQUIRE(groups > 0 && groups <= 65536, "bad group count");
    CMX_REQUIRE(m_total < (1u << 31), "too many rows");
    CMX_REQUIRE((uint64_t)p.n * p.ldw < (1ull << 32) && (uint64_t)p.lda * 256 < (1ull << 32),
                "operand tile exceeds 32-bit offsets");
    CMX_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 3u) == 0, "workspace must be 4-byte aligned");
    if (p.w_pretiled)
        if (int rc = check_pretiled(p, fmt, swiglu); rc != CMX_OK) return rc;
    GroupPlan plan;
    if (int rc = plan_groups(&plan, m_total, groups, p.n, fmt, p.kblocks, swiglu, p.w_pretiled); rc != CMX_OK) return rc;
    const GroupedKsplit& ks = plan.ks;
    const TileChoice& t = plan.t;
    const bool all_ksplit = plan.all_ksplit();
    const GroupTables tables(workspace, groups);
    bool by_sizes = false;
    // (the other persistent kernels walk from tile to tile through tables)
    if (!tables_filled && (all_ksplit || t.waves == kRing || (ks.small_rows == 0 && scans_groups(p, t, fmt, swiglu)))) {
        const uint64_t tiles = all_ksplit ? (uint64_t)(m_total / 64 + groups) * ceil_div(p.n, 64) : (uint64_t)(m_total / t.tm + groups) * ceil_div(p.n, t.tw);
        if (int rc = tiles_by_sizes(&by_sizes, groups, tiles, all_ksplit ? 2 : 1); rc != CMX_OK) return rc;
    }
    if (int rc = prepare_groups(p, tables_job(tables, group_sizes, groups, m_total, plan.tile_m(), ks.small_rows), by_sizes, tables_filled, s); rc != CMX_OK) return rc;
    if (ks.tile.fw != 0) {
        const int epi = !swiglu ? kEpiStore : (p.act_bf16 != nullptr ? kEpiSwigluQuantAct : kEpiSwigluQuant);
        if (int rc = launch_grouped_ksplit(p, tables, ks, fmt, epi, m_total, s); rc != CMX_OK || all_ksplit) return rc;
    }
    // The persistent kernels draw their next tile from a per-XCD counter when tiles differ in cost (4 x 1 wavefronts skip
    // the MFMAs of absent rows).  With 2 x 2 wavefronts every tile costs the same, so those kernels walk their XCD's run in
    // fixed strides instead: no atomic whose result has to be waited for with everything else in flight.  (8-bit stores have 2 x 2 wavefronts
    // whatever `waves` says: 16 groups x 300 rows, K = 512, N = 2048 18.6 -> 16.8 us, 4096 28.4 -> 25.9; behind the FFN's first matmul, where the
    // counters cost no launch, they are the better walk by half a per cent of the chain.)
    if (t.waves == 4 || (!swiglu && fmt != CMX_FMT_E2M1 && !p.w_pretiled && !tables_filled)) p.tile_ctr = nullptr;
    p.w_tiles = swiglu ? ceil_div(p.n / 2, t.tw / 2) : ceil_div(p.n, t.tw);
    const uint32_t max_m_tiles = max_group_tiles(m_total, groups, t.tm, ks.small_rows);
    if (p.w_pretiled) return t.tm == 288 ? launch_pretiled<288>(p, fmt, swiglu, max_m_tiles, s) : launch_pretiled<256>(p, fmt, swiglu, max_m_tiles, s);
    if (t.waves == kRing)
        return launch_ring(p, {t.tw, t.tm}, fmt, !swiglu ? kEpiStore : (p.act_bf16 != nullptr ? kEpiSwigluQuantAct : kEpiSwigluQuant), false, max_m_tiles, s);
    if (swiglu && p.act_bf16 != nullptr) return dispatch_tile<CMX_FMT_E4M3, kEpiSwigluQuantAct>(p, t, max_m_tiles, s);
    if (swiglu) return dispatch_tile<CMX_FMT_E4M3, kEpiSwigluQuant>(p, t, max_m_tiles, s);
    switch (fmt) {
        case CMX_FMT_E4M3: return dispatch_tile<CMX_FMT_E4M3, kEpiStore>(p, t, max_m_tiles, s);
        case CMX_FMT_E5M2: return dispatch_tile<CMX_FMT_E5M2, kEpiStore>(p, t, max_m_tiles, s);
        default: return dispatch_tile<CMX_FMT_E2M1, kEpiStore>(p, t, max_m_tiles, s);
    }
}
}  // namespace
}  // namespace cmx

namespace cmx {
namespace {
int gmm_store(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b, const uint8_t* b_scale,
              void* c, uint32_t ldc, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k,
              int fmt, int out_type, void* workspace, bool pretiled, cmx_stream_t stream, bool tables_filled = false) {
    if (m_total == 0 || n == 0) return CMX_OK;
    const uint32_t kbytes = fmt == CMX_FMT_E2M1 ? k / 2 : k;
    // weight scale rows are as every producer writes them: padded to an even count (the quantizer, the
    // reference generator's transposed even-padded matrix, the host operators' ScaleCols(k))
    const uint32_t ld_ws = scale_cols(k);
    int rc = check_operands(a, lda, a_scale, ld_as, b, kbytes, b_scale, ld_ws, k, fmt);
    if (rc != CMX_OK) return rc;
    CMX_REQUIRE(c && ldc >= n, "bad output");
    CMX_REQUIRE(out_type == CMX_OUT_BF16 || out_type == CMX_OUT_FP16 || out_type == CMX_OUT_FP32, "unknown output type");
    GemmParams p{};
    p.a = a; p.a_scale = a_scale; p.w = b; p.w_scale = b_scale; p.c = c;
    p.lda = lda; p.ld_as = ld_as; p.ldw = kbytes; p.ld_ws = ld_ws; p.ldc = ldc;
    p.m = m_total; p.n = n; p.kbytes = kbytes; p.kblocks = k / 32; p.out_type = out_type;
    p.scale_vec = scales_dword_aligned(a_scale, ld_as, b_scale, ld_ws);
    p.scale_vec16 = scales_aligned16(a_scale, ld_as, b_scale, ld_ws);
    p.w_pretiled = pretiled ? 1 : 0;
    return gmm_common(p, group_sizes, groups, m_total, workspace, fmt, false, tables_filled, static_cast<hipStream_t>(stream));
}
}  // namespace
}  // namespace cmx

extern "C" int cmx_mx_gmm(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b,
                          const uint8_t* b_scale, void* c, uint32_t ldc, const int32_t* group_sizes, uint32_t groups,
                          uint32_t m_total, uint32_t n, uint32_t k, int fmt, int out_type, void* workspace,
                          cmx_stream_t stream) {
    return cmx::gmm_store(a, lda, a_scale, ld_as, b, b_scale, c, ldc, group_sizes, groups, m_total, n, k, fmt, out_type,
                          workspace, false, stream);
}

extern "C" int cmx_mx_gmm_pretiled(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as,
                                   const uint8_t* b_tiled, const uint8_t* b_scale, void* c, uint32_t ldc,
                                   const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k,
                                   int fmt, int out_type, void* workspace, cmx_stream_t stream) {
    return cmx::gmm_store(a, lda, a_scale, ld_as, b_tiled, b_scale, c, ldc, group_sizes, groups, m_total, n, k, fmt,
                          out_type, workspace, true, stream);
}

extern "C" size_t cmx_int8_gmm_workspace_bytes(uint32_t groups, uint32_t n, uint32_t k, int trans_b) {
    const size_t meta = cmx::round_up_sz(cmx_mx_gmm_workspace_bytes(groups), 256);
    return meta + (trans_b ? 0 : cmx::round_up_sz((size_t)groups * n * k, 256));
}

namespace cmx {
namespace {
// Takes fp32 outputs of up to two rounds of 256 x 256 tiles and short K from the persistent kernel (*pipe) where it is slower than the streaming
// one.  With an odd number of slabs it walks one more, a microsecond a round (K below 2048); where groups average 256 rows or less, the tiles of
// a second round are few and its longer start shows (K up to 1536; K = 256: up to 512 rows).  With 16-bit outputs it is the faster one throughout.
// Measured (us, streaming against persistent; u: routes drawn uniformly, z: Zipf; N = 2048):
//   groups x rows   K = 256         384           512           640           1152          1536          1920          2048          3072
//   16 x 300 u      16.3  17.8   18.1  19.7   19.8  20.1   21.8  22.3   28.2  29.0   32.5  32.1   36.9  37.4   38.7  37.6   50.2  48.6
//   32 x 140 z      26.4  28.6   29.8  32.8   32.2  34.5   34.9  38.9   44.1  47.9   51.1  53.0   58.8  62.4   61.0  62.4   81.6  82.1
//   24 x 150 z      16.0  17.4   17.9  19.3   19.7  20.0                27.8  29.0   32.3  32.2   36.6  37.4   38.8  37.6   49.0  48.4
//   8 x 1000 u      29.6  29.4   32.6  33.6   34.7  33.9   37.8  38.7   47.3  48.3   54.8  53.7   63.0  63.5   65.2  63.3   86.6  83.4
//   16 x 700 z      31.7  30.1   35.3  35.3   37.2  36.1   40.6  41.5   51.3  52.2   59.5  58.4   68.5  69.2   70.8  69.2   93.5  91.6
//   8 x 1900 u (past two rounds)  45.2  38.3                54.0  45.2   62.7  56.0
int i8_streams(bool* pipe, uint64_t most_tiles, uint32_t mean_rows, uint32_t nslab) {
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    const bool slower = nslab % 2 != 0 ? nslab < 16 : nslab <= 12 && mean_rows <= (nslab == 2 ? 512u : 256u);
    if (slower && most_tiles <= 2 * (uint64_t)cus) *pipe = false;
    return CMX_OK;
}
}  // namespace
}  // namespace cmx

extern "C" int cmx_int8_gmm_dequant_swiglu(const int8_t* a, uint32_t lda, const float* token_scale, const int8_t* b,
                                           const float* channel_scale, uint32_t channel_scale_stride, void* out,
                                           uint32_t ld_out, int out_type, const int32_t* group_sizes, uint32_t groups,
                                           uint32_t m_total, uint32_t n, uint32_t k, int trans_b, void* workspace,
                                           cmx_stream_t stream) {
    using namespace cmx;
    if (m_total == 0 || n == 0) return CMX_OK;
    CMX_REQUIRE(a && token_scale && b && channel_scale && out && group_sizes && workspace, "null pointer");
    CMX_REQUIRE(groups > 0 && groups <= 65536 && m_total < (1u << 31), "bad group count or too many rows");
    CMX_REQUIRE(k > 0 && k % kSlabBytes == 0 && k < (1u << 17), "k must be a multiple of 128 below 131072 (INT32 accumulation)");
    CMX_REQUIRE(n % 64 == 0, "n must be a multiple of 64 (32-wide gate and up fragments)");
    CMX_REQUIRE(lda >= k && lda % 16 == 0 && aligned16(a) && aligned16(b), "operand rows must be 16-byte aligned");
    CMX_REQUIRE(ld_out >= n / 2 && channel_scale_stride >= 1, "bad output pitch or scale stride");
    CMX_REQUIRE(out_type == CMX_OUT_BF16 || out_type == CMX_OUT_FP16 || out_type == CMX_OUT_FP32, "unknown output type");
    CMX_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255u) == 0, "workspace must be 256-byte aligned");
    CMX_REQUIRE((uint64_t)n * k < (1ull << 32) && (uint64_t)lda * 256 < (1ull << 32), "operand tile exceeds 32-bit offsets");
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const uint8_t* w = reinterpret_cast<const uint8_t*>(b);
    if (!trans_b) {
        // weights stored [groups, k, n]: rewrite them K-contiguous behind the schedule metadata
        uint8_t* wt = ws + round_up_sz(cmx_mx_gmm_workspace_bytes(groups), 256);
        int rc = cmx_bytes_to_k_major(w, n, wt, k, k, n, groups, stream);
        if (rc != CMX_OK) return rc;
        w = wt;
    }
    GemmParams p{};
    p.a = reinterpret_cast<const uint8_t*>(a);
    p.a_scale = reinterpret_cast<const uint8_t*>(token_scale);
    p.w = w;
    p.w_scale = reinterpret_cast<const uint8_t*>(channel_scale);
    p.c = out;
    p.lda = lda; p.ld_as = 0; p.ldw = k; p.ld_ws = channel_scale_stride; p.ldc = ld_out;
    p.m = m_total; p.n = n; p.kbytes = k; p.kblocks = k / 32; p.out_type = out_type;
    p.scale_vec = 1;
    GroupedKsplit ks;
    if (int rc = choose_grouped_ksplit(m_total, groups, n, kFmtI8, p.kblocks, &ks); rc != CMX_OK) return rc;
    const bool all_ksplit = ks.tile.fw != 0 && ks.small_rows == 0;
    TileChoice t = {256, ceil_div(m_total, groups) <= 128 ? 128 : 256, 8};
    // The persistent kernel of 256 x 256 tiles stores 16 bytes at a time and has the scales' offsets in 32 bits; the streaming kernel takes the rest.
    bool pipe = (!g_force_tile.tw || g_force_tile.waves == 4) && !g_disable_dl && k >= 2 * kSlabBytes && (uint64_t)ld_out * (out_type == CMX_OUT_FP32 ? 4 : 2) % 16 == 0 &&
                aligned16(out) && (uint64_t)n * channel_scale_stride * 4 < (1ull << 32);
    // 128- or 256-row tiles: the device chooses by the sizes.  Not for outputs that the persistent kernel cannot store: against the streaming kernel
    // the ring's tiles alone win wherever the rows lie (rows at 4 bytes, us, ring / choice: 64 x 100, 7168, 3072 u 317 325, z 338 349, on four groups
    // 157 164; 32 x 90, 2048, 3072 45 51, 62 67, 40 47; 64 x 128, 4096, 3072 232 266, 232 236, 133 147; only 32 x 90, 7168, 3072 on four 95 91).
    bool choice = false;
    if (g_force_tile.waves == kRing) t = g_force_tile;
    else if (!g_force_tile.tw && !g_disable_dl) {
        if (int rc = ring_groups(&t, m_total, groups, n, kFmtI8, p.kblocks, true); rc != CMX_OK) return rc;
        choice = !all_ksplit && t.waves == kRing && t.tw == 256 && pipe;
    }
    if (t.waves != kRing) t.tm = 256;
    const uint64_t most_tiles = (uint64_t)max_group_tiles(m_total, groups, 256, ks.small_rows) * ceil_div(n, 256);
    if (t.waves != kRing && !g_force_tile.tw && out_type == CMX_OUT_FP32)
        if (int rc = i8_streams(&pipe, most_tiles, ceil_div(m_total, groups), k / kSlabBytes); rc != CMX_OK) return rc;
    // Kernels of one tile per workgroup find it by the sizes up to some rounds; past those the launch that fills the tables makes the
    // choice.  Where it would fill them for small groups as well, those that are left to the large tiles are large for
    // their average (256 x 32, 7168, 4096, on eight groups 227 against 277).  The persistent kernel scans the sizes once,
    // in any number of rounds (scan / tables, us: 16 x 2048, K = 512, N = 4096, 8 rounds 150 155; 32 x 2048, 1024, 17 rounds 384 386; 32 x 4096, 33 rounds 741 739).
    bool by_sizes = false;
    if (pipe && !all_ksplit && t.waves != kRing && ks.small_rows == 0) {
        by_sizes = groups <= kInlineGroups;
    } else {
        const uint64_t most = all_ksplit ? (uint64_t)(m_total / 64 + groups) * ceil_div(n, 64) : (uint64_t)(m_total / t.tm + groups) * ceil_div(n, t.tw);
        // (a choice by the sizes is a second scan for every tile)
        if (int rc = tiles_by_sizes(&by_sizes, groups, choice && ks.small_rows == 0 ? 3 * most : most, all_ksplit ? 2 : 1); rc != CMX_OK) return rc;
    }
    if (choice && !by_sizes && ks.small_rows != 0) {
        choice = false;
        t = {256, 256, 8};
    }
    const GroupTables tables(ws, groups);
    const GroupTablesJob job = tables_job(tables, group_sizes, groups, m_total, all_ksplit ? 16 * ks.tile.fm : t.tm, ks.small_rows);
    if (choice) {
        int cus = 0;
        if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
        p.choice_cus = (uint32_t)cus;
        p.short_tiles = tables.small_pref;
    }
    p.w_tiles = ceil_div(n / 2, t.tw / 2);
    if (choice && !by_sizes)
        if (int rc = launch_i8_choice_tables(job, p, tables.small_pref, s); rc != CMX_OK) return rc;
    if (int rc = prepare_groups(p, job, by_sizes, choice, s); rc != CMX_OK) return rc;
    if (ks.tile.fw != 0)
        if (int rc = launch_grouped_ksplit(p, tables, ks, kFmtI8, kEpiI8DequantSwiglu, m_total, s); rc != CMX_OK || all_ksplit) return rc;
    const uint32_t max_m_tiles = max_group_tiles(m_total, groups, t.tm, ks.small_rows);
    p.tile_ctr = nullptr;                                      // tiles of one cost: fixed strides
    if (choice) return launch_i8_choice(p, max_m_tiles, max_group_tiles(m_total, groups, 256, ks.small_rows), s);
    if (t.waves == kRing) return launch_ring(p, {t.tw, t.tm}, kFmtI8, kEpiI8DequantSwiglu, false, max_m_tiles, s);
    if (pipe) return launch_gemm_pipe<kFmtI8, kEpiI8DequantSwiglu, 256, 2, 2, 2>(p, max_m_tiles, s);
    return launch_gemm_dl<kFmtI8, 256, 256, 2, 4, kEpiI8DequantSwiglu>(p, max_m_tiles, s);
}

namespace cmx {
namespace {
int gmm_swiglu_quant(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b,
                     const uint8_t* b_scale, uint8_t* act_codes, uint32_t ld_act, uint8_t* act_scales, uint32_t ld_acts,
                     void* act_bf16, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k,
                     void* workspace, bool pretiled, cmx_stream_t stream, bool tables_filled = false) {
    const uint32_t ld_ws = scale_cols(k);      // even-padded weight scale rows, as in cmx_mx_gmm
    int rc = check_operands(a, lda, a_scale, ld_as, b, k, b_scale, ld_ws, k, CMX_FMT_E4M3);
    if (rc != CMX_OK) return rc;
    CMX_REQUIRE(n % 64 == 0, "n must be a multiple of 64 (gate|up halves of whole MX blocks)");
    CMX_REQUIRE(act_codes && act_scales, "null pointer");
    CMX_REQUIRE(ld_act >= n / 2 && ld_act % 4 == 0 && (reinterpret_cast<uintptr_t>(act_codes) & 3u) == 0,
                "activation code rows must be 4-byte aligned and hold n/2 bytes");
    CMX_REQUIRE(ld_acts >= scale_cols(n / 2), "activation scale pitch too small");
    GemmParams p{};
    p.a = a; p.a_scale = a_scale; p.w = b; p.w_scale = b_scale;
    p.act_codes = act_codes; p.act_scales = act_scales; p.act_bf16 = static_cast<uint16_t*>(act_bf16);
    p.ld_act = ld_act; p.ld_acts = ld_acts;
    p.lda = lda; p.ld_as = ld_as; p.ldw = k; p.ld_ws = ld_ws;
    p.m = m_total; p.n = n; p.kbytes = k; p.kblocks = k / 32; p.out_type = CMX_OUT_BF16;
    p.scale_vec = scales_dword_aligned(a_scale, ld_as, b_scale, ld_ws);
    p.scale_vec16 = scales_aligned16(a_scale, ld_as, b_scale, ld_ws);
    p.w_pretiled = pretiled ? 1 : 0;
    return gmm_common(p, group_sizes, groups, m_total, workspace, CMX_FMT_E4M3, true, tables_filled, static_cast<hipStream_t>(stream));
}

// Schedule metadata of the allocation-free entry point (row offsets, m-tile prefixes, per-XCD tile counters of up to
// kStaticGroups groups): a fixed array in device memory instead of a caller's workspace.  Every device that runs
// the library holds its own copy; its address on a device comes from hipGetSymbolAddress with that device current
// (the array's name is only a host-side handle).
constexpr uint32_t kStaticGroups = 4096;
constexpr size_t kStaticScratchBytes = (3 * ((size_t)kStaticGroups + 1) + 8) * sizeof(int32_t);
static __device__ __align__(256) unsigned char scratch[(kStaticScratchBytes + 255) / 256 * 256];

int static_scratch(void** out) {
    static std::atomic<void*> ptrs[kMaxDevices];
    int dev = 0;
    int rc = current_device_slot(&dev);
    if (rc != CMX_OK) return rc;
    void* q = ptrs[dev].load(std::memory_order_acquire);
    if (q == nullptr) {
        CMX_HIP(hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)));
        CMX_REQUIRE(q != nullptr, "no device address for the static scratch array");
        ptrs[dev].store(q, std::memory_order_release);
    }
    *out = q;
    return CMX_OK;
}
}  // namespace
}  // namespace cmx

extern "C" int cmx_mx_gmm_swiglu_quant(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as,
                                       const uint8_t* b, const uint8_t* b_scale, uint8_t* act_codes, uint32_t ld_act,
                                       uint8_t* act_scales, uint32_t ld_acts, void* act_bf16,
                                       const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n,
                                       uint32_t k, void* workspace, cmx_stream_t stream) {
    if (m_total == 0 || n == 0) return CMX_OK;
    return cmx::gmm_swiglu_quant(a, lda, a_scale, ld_as, b, b_scale, act_codes, ld_act, act_scales, ld_acts, act_bf16,
                                 group_sizes, groups, m_total, n, k, workspace, false, stream);
}

extern "C" int cmx_mx_gmm_swiglu_quant_pretiled(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as,
                                                const uint8_t* b_tiled, const uint8_t* b_scale, uint8_t* act_codes,
                                                uint32_t ld_act, uint8_t* act_scales, uint32_t ld_acts, void* act_bf16,
                                                const int32_t* group_sizes, uint32_t groups, uint32_t m_total,
                                                uint32_t n, uint32_t k, void* workspace, cmx_stream_t stream) {
    if (m_total == 0 || n == 0) return CMX_OK;
    return cmx::gmm_swiglu_quant(a, lda, a_scale, ld_as, b_tiled, b_scale, act_codes, ld_act, act_scales, ld_acts,
                                 act_bf16, group_sizes, groups, m_total, n, k, workspace, true, stream);
}

int cmx::launch_group_tables(const GroupTablesJob& job, hipStream_t s) {
    hipLaunchKernelGGL(gmm_prepare_kernel, dim3(1), dim3(256), 0, s, job);
    CMX_LAUNCH_CHECK();
    return CMX_OK;
}

int cmx::plan_group_tables(GroupTablesJob* job, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, int fmt,
                           bool swiglu, bool pretiled, void* workspace) {
    GroupPlan plan;
    if (int rc = plan_groups(&plan, m_total, groups, n, fmt, k / 32, swiglu, pretiled); rc != CMX_OK) return rc;
    *job = tables_job(GroupTables(workspace, groups), group_sizes, groups, m_total, plan.tile_m(), plan.ks.small_rows);
    return CMX_OK;
}

int cmx::gmm_swiglu_quant_prepared(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b,
                                   const uint8_t* b_scale, uint8_t* act_codes, uint32_t ld_act, uint8_t* act_scales, uint32_t ld_acts,
                                   const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, void* workspace,
                                   bool pretiled, hipStream_t s) {
    return gmm_swiglu_quant(a, lda, a_scale, ld_as, b, b_scale, act_codes, ld_act, act_scales, ld_acts, nullptr, group_sizes, groups, m_total, n,
                            k, workspace, pretiled, s, true);
}

int cmx::gmm_prepared(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as, const uint8_t* b, const uint8_t* b_scale, void* c,
                      uint32_t ldc, const int32_t* group_sizes, uint32_t groups, uint32_t m_total, uint32_t n, uint32_t k, int fmt, int out_type,
                      void* workspace, bool pretiled, hipStream_t s) {
    return gmm_store(a, lda, a_scale, ld_as, b, b_scale, c, ldc, group_sizes, groups, m_total, n, k, fmt, out_type, workspace, pretiled, s, true);
}

extern "C" uint32_t cmx_mx_gmm_noalloc_max_groups(void) { return cmx::kStaticGroups; }

extern "C" int cmx_mx_gmm_swiglu_quant_noalloc(const uint8_t* a, uint32_t lda, const uint8_t* a_scale, uint32_t ld_as,
                                               const uint8_t* b, const uint8_t* b_scale, uint8_t* act_codes,
                                               uint32_t ld_act, uint8_t* act_scales, uint32_t ld_acts, void* act_bf16,
                                               const int32_t* group_sizes, uint32_t groups, uint32_t m_total,
                                               uint32_t n, uint32_t k, cmx_stream_t stream) {
    using namespace cmx;
    if (m_total == 0 || n == 0) return CMX_OK;
    CMX_REQUIRE(groups <= kStaticGroups, "at most 4096 groups fit the static schedule array: use cmx_mx_gmm_swiglu_quant with a workspace");
    void* meta = nullptr;
    if (int rc = static_scratch(&meta); rc != CMX_OK) return rc;
    // gmm_prepare_kernel rewrites every word of the metadata that the matmul kernel reads (and zeroes the tile
    // counters), so nothing of an earlier call survives into this one
    return gmm_swiglu_quant(a, lda, a_scale, ld_as, b, b_scale, act_codes, ld_act, act_scales, ld_acts, act_bf16,
                            group_sizes, groups, m_total, n, k, meta, false, stream);
}

// One-time set-up on the current device: raises the dynamic-LDS limit of every matmul kernel, has the runtime load the
// code object of every translation unit, reads the CU count and resolves the static schedule array, so that no later
// call has to (none of this is allowed, or wise, inside a stream capture).  Optional: every entry point still does
// what it needs on first use.
extern "C" int cmx_init(void) {
    using namespace cmx;
    for (const LdsKernel& k : lds_registry())
        if (int rc = allow_dynamic_lds(k.fn, k.bytes, *k.flag); rc != CMX_OK) return rc;
    // the matmul kernels without an LDS limit to raise (and with them this unit's code object), then the other units
    hipFuncAttributes attr;
    CMX_HIP(hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(gmm_prepare_kernel)));
    if (int rc = preload_routing_kernels(); rc != CMX_OK) return rc;
    if (int rc = preload_layout_kernels(); rc != CMX_OK) return rc;
    if (int rc = preload_quant_kernels(); rc != CMX_OK) return rc;
    int cus = 0;
    if (int rc = cu_count(&cus); rc != CMX_OK) return rc;
    void* meta = nullptr;
    return static_scratch(&meta);
}
