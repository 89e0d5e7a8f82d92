// Epilogue of the matmul kernels whose sums pass through the LDS (split-K and ring kernels): four columns of a row at a time.
#pragma once

#include "mx_gemm_common.h"

namespace cmx {

#if defined(__HIPCC__)

// channel scales of four gate columns from ncol on and of their up partners (ncol + 4 <= n / 2)
__device__ __forceinline__ void load_channel_scales(const GemmParams& p, uint32_t g, uint32_t ncol, v4f& cg, v4f& cu) {
    const float* ch = reinterpret_cast<const float*>(p.w_scale) + (size_t)g * p.n * p.ld_ws;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        cg[i] = ch[(size_t)(ncol + i) * p.ld_ws];
        cu[i] = ch[(size_t)((p.n >> 1) + ncol + i) * p.ld_ws];
    }
}

// INT32 sums of four gate and up columns -> fp32 * per-channel scale -> fp16 -> fp32 * per-token scale -> x0 * sigmoid(x0) * gate
__device__ __forceinline__ void store_i8_quad(const GemmParams& p, size_t mrow, uint32_t ncol, const v4f& v, const v4f& u, const v4f& cg,
                                              const v4f& cu, float tsv) {
    const v4i ig = __builtin_bit_cast(v4i, v), iu = __builtin_bit_cast(v4i, u);
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x0 = __fmul_rn(i8_dequant(ig[i], cg[i]), tsv);
        const float gate = __fmul_rn(i8_dequant(iu[i], cu[i]), tsv);
        y[i] = __fmul_rn(__fmul_rn(x0, __builtin_amdgcn_rcpf(1.0f + __expf(-x0))), gate);
    }
    if (p.out_type == CMX_OUT_FP32) {
        float* o = reinterpret_cast<float*>(p.c) + mrow * p.ldc + ncol;
        if ((reinterpret_cast<uintptr_t>(o) & 15u) == 0) {
            *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
        } else {
            for (uint32_t i = 0; i < 4; ++i) o[i] = y[i];
        }
    } else {
        uint16_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            h[i] = p.out_type == CMX_OUT_FP16 ? __builtin_bit_cast(uint16_t, (_Float16)as_f32(y[i])) : (uint16_t)f32_to_bf16(y[i]);
        uint16_t* o = reinterpret_cast<uint16_t*>(p.c) + mrow * p.ldc + ncol;
        if ((reinterpret_cast<uintptr_t>(o) & 7u) == 0) {
            *reinterpret_cast<uint2*>(o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
        } else {
            for (uint32_t i = 0; i < 4; ++i) o[i] = h[i];
        }
    }
}

// Whether rows of 16-bit output are whole 16-byte pieces, so that eight columns from a multiple of eight on are in or out together.
__device__ __forceinline__ bool stores_pieces(const GemmParams& p) {
    return p.out_type != CMX_OUT_FP32 && p.n % 8 == 0 && p.ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15u) == 0;
}
// eight sums as such a piece
template <int OUT>
__device__ __forceinline__ uint4 pack_piece(const v4f& lo, const v4f& hi) {
    if constexpr (OUT == CMX_OUT_BF16) {
        return make_uint4(cvt_pk_bf16(lo[0], lo[1]), cvt_pk_bf16(lo[2], lo[3]), cvt_pk_bf16(hi[0], hi[1]), cvt_pk_bf16(hi[2], hi[3]));
    } else {
        typedef _Float16 v8h __attribute__((ext_vector_type(8)));
        return __builtin_bit_cast(uint4, (v8h){(_Float16)lo[0], (_Float16)lo[1], (_Float16)lo[2], (_Float16)lo[3],
                                               (_Float16)hi[0], (_Float16)hi[1], (_Float16)hi[2], (_Float16)hi[3]});
    }
}

// Sums of one output row, four consecutive columns from ncol on (SwiGLU kinds: four gate columns and their up partners, ncol the
// activation column), to memory.  SwiGLU + requant: eight neighbouring lanes hold the 32 columns of an MX block.
template <int EPI>
__device__ __forceinline__ void store_quad(const GemmParams& p, const Tile& tc, uint32_t mloc, uint32_t ncol, const v4f& v, const v4f& u) {
    const bool mvalid = mloc < tc.rows_valid;
    const size_t mrow = (size_t)(tc.row0 + (mvalid ? mloc : 0));
    if constexpr (EPI == kEpiStore) {
        if (!mvalid || ncol >= p.n) return;
        const bool full = ncol + 4 <= p.n;
        if (p.out_type == CMX_OUT_FP32) {
            float* o = reinterpret_cast<float*>(p.c) + mrow * p.ldc + ncol;
            if (full && (reinterpret_cast<uintptr_t>(o) & 15u) == 0) {
                *reinterpret_cast<v4f*>(o) = v;
            } else {
                for (uint32_t i = 0; i < 4 && ncol + i < p.n; ++i) o[i] = v[i];
            }
        } else {
            uint32_t h0, h1;
            if (p.out_type == CMX_OUT_BF16) {
                h0 = cvt_pk_bf16(v[0], v[1]);
                h1 = cvt_pk_bf16(v[2], v[3]);
            } else {
                typedef _Float16 v2h __attribute__((ext_vector_type(2)));
                h0 = __builtin_bit_cast(uint32_t, (v2h){(_Float16)v[0], (_Float16)v[1]});
                h1 = __builtin_bit_cast(uint32_t, (v2h){(_Float16)v[2], (_Float16)v[3]});
            }
            uint16_t* o = reinterpret_cast<uint16_t*>(p.c) + mrow * p.ldc + ncol;
            if (full && (reinterpret_cast<uintptr_t>(o) & 7u) == 0) {
                *reinterpret_cast<uint2*>(o) = make_uint2(h0, h1);
            } else {
                const uint32_t h[2] = {h0, h1};
                for (uint32_t i = 0; i < 4 && ncol + i < p.n; ++i) o[i] = (uint16_t)(h[i >> 1] >> (16 * (i & 1)));
            }
        }
    } else if constexpr (EPI == kEpiI8DequantSwiglu) {
        const uint32_t half = p.n >> 1;
        if (!mvalid || ncol >= half) return;                      // n is a multiple of 64: four columns are in or out together
        v4f cg, cu;
        load_channel_scales(p, tc.g, ncol, cg, cu);
        store_i8_quad(p, mrow, ncol, v, u, cg, cu, reinterpret_cast<const float*>(p.a_scale)[mrow]);
    } else {
        // SwiGLU on the bf16-rounded sums, bf16 again, then the MX block of 32 columns: eight neighbouring lanes hold it
        const uint32_t half = p.n >> 1;
        uint32_t pk[2], m = 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t g2 = cvt_pk_bf16(v[2 * j], v[2 * j + 1]), u2 = cvt_pk_bf16(u[2 * j], u[2 * j + 1]);
            pk[j] = cvt_pk_bf16(silu_mul(__uint_as_float(g2 << 16), __uint_as_float(u2 << 16)),
                                silu_mul(__uint_as_float(g2 & 0xFFFF0000u), __uint_as_float(u2 & 0xFFFF0000u)));
            m = pk_max_u16(m, pk[j] & 0x7FFF7FFFu);
        }
        m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xF, 0xF, true));     // lane ^ 1
        m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xF, 0xF, true));     // lane ^ 2
        m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xF, 0xF, true));    // the other quad of eight
        const uint32_t amax = max(m & 0xFFFFu, m >> 16);
        const int e = block_exp_from_bf16_amax(amax, kEmaxE4M3);
        if (!mvalid || ncol >= half) return;
        if constexpr (EPI == kEpiSwigluQuantAct) {
            if (p.act_bf16) {
                uint16_t* o = p.act_bf16 + mrow * half + ncol;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (uint16_t)(pk[i >> 1] >> (16 * (i & 1)));
            }
        }
        const uint32_t lim = (((uint32_t)(e + kEmaxE4M3 + 127) << 7) | 0x60u) * 0x10001u;
        const float scale = __uint_as_float((uint32_t)(e + 127) << 23);
        const uint32_t c0 = pk_min_u16(pk[0] & 0x7FFF7FFFu, lim) | (pk[0] & 0x80008000u);
        const uint32_t c1 = pk_min_u16(pk[1] & 0x7FFF7FFFu, lim) | (pk[1] & 0x80008000u);
        *reinterpret_cast<uint32_t*>(p.act_codes + mrow * p.ld_act + ncol) = cvt_scaled_pk4<CMX_FMT_E4M3>(c0, c1, scale);
        if ((ncol & 31u) == 0) {
            uint8_t* srow = p.act_scales + mrow * p.ld_acts;
            const uint32_t blk = ncol >> 5, nblk = half >> 5;
            srow[blk] = (uint8_t)(e + 127);
            if (blk == nblk - 1 && (nblk & 1u)) srow[nblk] = 127;
        }
    }
}

// SwiGLU on the bf16-rounded sums of eight gate and up columns of one row, bf16 again, then the MX block of 32 columns, which four neighbouring
// lanes hold: its scale exponent, and the lane's eight codes (pk: the bf16 values, in pairs)
__device__ __forceinline__ int swiglu_quant_piece(const v4f (&g)[2], const v4f (&u)[2], uint32_t (&pk)[4], uint2& codes) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t g2 = cvt_pk_bf16(g[j / 2][j % 2 * 2], g[j / 2][j % 2 * 2 + 1]), u2 = cvt_pk_bf16(u[j / 2][j % 2 * 2], u[j / 2][j % 2 * 2 + 1]);
        pk[j] = cvt_pk_bf16(silu_mul(__uint_as_float(g2 << 16), __uint_as_float(u2 << 16)),
                            silu_mul(__uint_as_float(g2 & 0xFFFF0000u), __uint_as_float(u2 & 0xFFFF0000u)));
        m = pk_max_u16(m, pk[j] & 0x7FFF7FFFu);
    }
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xF, 0xF, true));     // lane ^ 1
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xF, 0xF, true));     // lane ^ 2
    const int e = block_exp_from_bf16_amax(max(m & 0xFFFFu, m >> 16), kEmaxE4M3);
    const uint32_t lim = (((uint32_t)(e + kEmaxE4M3 + 127) << 7) | 0x60u) * 0x10001u;
    const float scale = __uint_as_float((uint32_t)(e + 127) << 23);
    uint32_t c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = pk_min_u16(pk[j] & 0x7FFF7FFFu, lim) | (pk[j] & 0x80008000u);
    codes = make_uint2(cvt_scaled_pk4<CMX_FMT_E4M3>(c[0], c[1], scale), cvt_scaled_pk4<CMX_FMT_E4M3>(c[2], c[3], scale));
    return e;
}

#endif  // __HIPCC__

}  // namespace cmx
