// Epilogue pieces shared by the GEMM kernels: one 16-byte chunk of bf16
// results to the output, plain or added to the residual rows in place.
#pragma once

#include "common.hpp"
#include "gemm.hpp"

namespace ssa {

// v: the 8 bf16 results of row `o / ns`, columns col .. col + 7 (element offset
// o); vec: the chunk is inside the row and 16-byte aligned, else `left` of its
// columns exist and go one by one.
template <int EPI>
__device__ __forceinline__ void gemm_store_chunk(void* outp, int64_t o, const u32x4_v& v, bool vec, int left) {
    float y[8];
    unpack8<bf16_t>(v, y);
    if (vec) {
        if constexpr (EPI == kGemmStore) {
            *reinterpret_cast<u32x4_v*>(static_cast<uint16_t*>(outp) + o) = v;
        } else if constexpr (EPI == kGemmResidualBf16) {
            uint16_t* h = static_cast<uint16_t*>(outp) + o;
            float hv[8];
            unpack8<bf16_t>(*reinterpret_cast<const u32x4_v*>(h), hv);
            u32x4_v w;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = f32_to_bf16_bits(hv[2 * i] + y[2 * i]) | (f32_to_bf16_bits(hv[2 * i + 1] + y[2 * i + 1]) << 16);
            *reinterpret_cast<u32x4_v*>(h) = w;
        } else {
            float* h = static_cast<float*>(outp) + o;
            f32x4_v h0 = *reinterpret_cast<const f32x4_v*>(h), h1 = *reinterpret_cast<const f32x4_v*>(h + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h0[i] = bf16_round(h0[i] + y[i]);
                h1[i] = bf16_round(h1[i] + y[4 + i]);
            }
            *reinterpret_cast<f32x4_v*>(h) = h0;
            *reinterpret_cast<f32x4_v*>(h + 4) = h1;
        }
    } else {
        for (int i = 0; i < 8 && i < left; ++i) {
            if constexpr (EPI == kGemmStore) {
                static_cast<uint16_t*>(outp)[o + i] = static_cast<uint16_t>(f32_to_bf16_bits(y[i]));
            } else if constexpr (EPI == kGemmResidualBf16) {
                uint16_t* h = static_cast<uint16_t*>(outp);
                h[o + i] = static_cast<uint16_t>(f32_to_bf16_bits(bf16_bits_to_f32(h[o + i]) + y[i]));
            } else {
                float* h = static_cast<float*>(outp);
                h[o + i] = bf16_round(h[o + i] + y[i]);
            }
        }
    }
}

}  // namespace ssa
