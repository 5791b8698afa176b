// What the GEMM translation units share: exact dequantization of resident quantized weights
// (layouts at struct QWeight) and the operand DMA into LDS.
#pragma once
#include "internal.h"

namespace tlhip {

// Residency buffers of a quantized weight (layout at struct QWeight).
struct QView {
    const uint8_t* qs;
    const __half* d;
    const uint8_t* hdr;
    const uint8_t* qh;
    const int8_t* sc;
};

// Q4_K sub-block j's d * scale and dmin * min from its resident super-block header
// (q4k_hdr_sm; QTensor::get_scale_min_k4, quantized.rs:405-415); both products are exact in f32.
__device__ __forceinline__ void q4k_scale_min(const uint4& hd, int j, float* d1, float* m1) {
    uint32_t sc, mn;
    q4k_hdr_sm(hd, j, &sc, &mn);
    *d1 = __half2float(__ushort_as_half((uint16_t)(hd.x & 0xFFFF))) * (float)sc;
    *m1 = __half2float(__ushort_as_half((uint16_t)(hd.x >> 16))) * (float)mn;
}

// Dequantise the 32 weights of unit blk into v[32] (f32, bit-identical to the reference's
// dequantizers: Q4_0 d * (q - 8), Q8_0 d * q, Q4_K (d sc) q - dmin m, Q6_K (d sc) (q - 32)).
template <int QT>
__device__ __forceinline__ void dequant_block(const QView& qv, int64_t blk, float* v) {
    if constexpr (QT == TL_HIP_GGML_Q4_0) {
        const float d = __half2float(qv.d[blk]);
        uint4 w = *reinterpret_cast<const uint4*>(qv.qs + blk * 16);
        const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t byte = (q[c] >> (8 * i)) & 0xFF;
                v[4 * c + i] = d * (float)((int)(byte & 0xF) - 8);
                v[16 + 4 * c + i] = d * (float)((int)(byte >> 4) - 8);
            }
    } else if constexpr (QT == TL_HIP_GGML_Q8_0) {
        const float d = __half2float(qv.d[blk]);
        const uint4* p = reinterpret_cast<const uint4*>(qv.qs + blk * 32);
        uint4 w0 = p[0], w1 = p[1];
        const uint32_t q[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[4 * c + i] = d * (float)(int8_t)((q[c] >> (8 * i)) & 0xFF);
    } else if constexpr (QT == TL_HIP_GGML_Q4_K) {
        float d1, m1;
        q4k_scale_min(reinterpret_cast<const uint4*>(qv.hdr)[blk >> 3], (int)(blk & 7), &d1, &m1);
        uint4 w = *reinterpret_cast<const uint4*>(qv.qs + blk * 16);
        const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t byte = (q[c] >> (8 * i)) & 0xFF;
                v[4 * c + i] = d1 * (float)(byte & 0xF) - m1;
                v[16 + 4 * c + i] = d1 * (float)(byte >> 4) - m1;
            }
    } else {
        const float d = __half2float(qv.d[blk >> 3]);
        const float e0 = d * (float)qv.sc[2 * blk], e1 = d * (float)qv.sc[2 * blk + 1];
        uint4 w = *reinterpret_cast<const uint4*>(qv.qs + blk * 16);
        const uint2 h = reinterpret_cast<const uint2*>(qv.qh)[blk];
        const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t byte = (q[c] >> (8 * i)) & 0xFF;
                const uint32_t h0 = (h.x >> (8 * i + 2 * c)) & 3, h1 = (h.y >> (8 * i + 2 * c)) & 3;
                v[4 * c + i] = e0 * (float)((int)((byte & 0xF) | (h0 << 4)) - 32);
                v[16 + 4 * c + i] = e1 * (float)((int)((byte >> 4) | (h1 << 4)) - 32);
            }
    }
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Operand DMA: buffer loads straight into LDS through a raw (stride 0) buffer resource over
// [p, p + bytes).  A lane's SIZE bytes at voff + soff land at lds + lane * SIZE (one 64-lane
// instruction writes 64 consecutive elements).  The per-lane offset is fixed for the whole K
// loop and the iteration's advance is a scalar, so the loop spends no vector instruction on
// addresses (with flat global_load_lds each load cost two 64-bit vector adds).
__device__ __forceinline__ void buf_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void buf_dma4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, void* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, voff, soff, 0, 0);
}

}  // namespace tlhip
