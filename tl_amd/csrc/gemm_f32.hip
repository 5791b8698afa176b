// The quantized GEMM of the f32 path (tl_qtensor_matmul past four rows): Y = X . W^T with W's
// values exact, every entry of X within 2^-23 of itself and f32 sums; max-rel-err 1e-4 class
// against tl_cpu.
//
//  * k_qgemm_x2   matrix cores: X split into two f16 planes of a row-scaled value (k_x_split),
//                 W's whole numbers as f16, one f32 sum per 32-weight unit scaled in f32.
//  * k_qgemm_f32  plain f32 FMAs over dequantized tiles; needs no workspace.
//
// k_qgemm_x2 with one plane (X rounded to f16) is also the f16 path's GEMM for Q6_K weights.
#include "gemm_common.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace tlhip {

// ------------------------------------------------------------ f32 quantized GEMM ----
// The form without a workspace: the allocation-free entry, calls under stream capture, and
// calls the other form has no memory or no 32-bit offsets for.
// Tile 64 (x rows) x 64 (weight rows) x 32 (one quant block); 256 threads, 4x4 outputs
// per thread.  LDS holds the k-major tiles Xs[32][64] and Ws[32][64].
constexpr int F_BM = 64, F_BN = 64, F_BK = 32;

template <int QT>
__global__ __launch_bounds__(256) void k_qgemm_f32(QView qv, const float* __restrict__ x,
                                                   float* y, const float* res, int64_t m, int64_t n,
                                                   int64_t k, int64_t nb) {
    __shared__ __attribute__((aligned(16))) float Xs[F_BK][F_BM + 4];
    __shared__ __attribute__((aligned(16))) float Ws[F_BK][F_BN + 4];
    const int t = threadIdx.x;
    const int tx = t & 15, ty = t >> 4;
    const int64_t m0 = (int64_t)blockIdx.y * F_BM, n0 = (int64_t)blockIdx.x * F_BN;
    float acc[4][4] = {};
    for (int64_t kb = 0; kb < nb; kb++) {
        // X tile: 64 rows x 32 floats -> 512 float4, 2 per thread
#pragma unroll
        for (int i = 0; i < 2; i++) {
            int idx = t + i * 256;
            int r = idx >> 3, c4 = idx & 7;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (m0 + r < m) v = *reinterpret_cast<const float4*>(x + (m0 + r) * k + kb * 32 + c4 * 4);
            Xs[c4 * 4 + 0][r] = v.x;
            Xs[c4 * 4 + 1][r] = v.y;
            Xs[c4 * 4 + 2][r] = v.z;
            Xs[c4 * 4 + 3][r] = v.w;
        }
        // W tile: 64 rows x one block, threads 0..63 dequantise a row each
        if (t < 64) {
            float v[32];
            int64_t row = n0 + t < n ? n0 + t : n - 1;
            dequant_block<QT>(qv, row * nb + kb, v);
#pragma unroll
            for (int j = 0; j < 32; j++) Ws[j][t] = v[j];
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < F_BK; kk++) {
            float4 a = *reinterpret_cast<const float4*>(&Xs[kk][ty * 4]);
            float4 b = *reinterpret_cast<const float4*>(&Ws[kk][tx * 4]);
            const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int64_t r = m0 + ty * 4 + i;
        if (r >= m) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            int64_t c = n0 + tx * 4 + j;
            if (c < n) y[r * n + c] = res ? res[r * n + c] + acc[i][j] : acc[i][j];
        }
    }
}

// ------------------------------------------------ f32 products on the matrix cores ----
// A quantized weight is (whole number) x (scale of its 32- or 16-weight unit), and the whole
// numbers (-8 .. 7, -128 .. 127, -32 .. 31) are exact in f16.  X, scaled per row by a power of
// two so that the row's largest magnitude lies in [2^14, 2^15), is the sum of two f16 values
// hi + 2^-12 lo; lo meets the whole numbers times 2^-12, exact in f16 too.  An entry down to
// 2^-28 of the row's largest is within 2^-23 of itself that way.  Smaller ones, which matter where
// the weights under the large ones are zero, are not left short: up to X2_REST of a row keep
// what the planes miss in a list that the epilogue adds (rest_dot), a row with more of them is
// formed from X itself (plain_block).  So
// each unit's sum q . x is two MFMAs with f32 accumulation over exact products, and y gathers
// d * (q . x) in f32: as many roundings per output as units, where an f32 FMA chain has one
// per weight.  Relative error against 64-bit sums over N(0, 1) inputs, k 256 .. 11008:
// 0.8e-7 .. 2.2e-7 (the FMA chain of k_qgemm_f32: 1.3e-7 .. 1.9e-6).
//
// What bounds it: the matrix cores and the VALU work between them (11008 x 4096, m = 512: 92
// GFLOP of MFMA in 127 us = 725 TFLOP/s where a large f16 product by the vendor's library
// reaches 1160), the weight stream and launch latencies at short inputs.  us per call,
// k_qgemm_f32 before -> this form: Q4_0 11008 x 4096 m 512 724 -> 132; Q8_0 4096 x 11008 m 16
// 733 -> 19.2; Q4_K 2048 x 2048 m 128 117 -> 17.  The lo plane's own scale costs four packed
// multiplications per weight operand (without it, 2^-14 of the row's largest would be the limit);
// the 64-row tiles therefore take wavefront grids that share an operand among as many row tiles
// as they have (Q4_K 5632 x 2048 m 128: 34 -> 29 us of 4 x 2 against 2 x 4 wavefronts; m 512 71 ->
// 60 of 2 x 4 against 1 x 8).

struct XRest {
    int32_t at;  // element of the row
    float rest;  // its value less what the planes hold
};
constexpr int X2_REST = 16;
constexpr float X2_LO = 4096.0f;  // lo plane: 2^12 times what hi leaves, at most 2^15

// X f32 [m, k] -> planes [m][unit of 32][8 words of 8 halves]: words 0-3 hi, 4-7 lo, in the k
// order of the MFMA operands (NAT: word t = elements 8t .. 8t+7, Q8_0; else elements 4t .. 4t+3
// and 16+4t .. 16+4t+3, the nibble order).  sh[row]: the exponent that scales a sum back (low 16
// bits) and the number of entries in rest[row] (from bit 16), or INT_MIN for a row that plain_block
// forms: one with an infinity or NaN (zeros here) or with more than X2_REST such entries.  sx (Q4_K):
// the scaled unit sums [unit][mp].  One workgroup per row: the row is read once for its
// largest magnitude and kept in registers (k <= 12288) for the split.  SRC (XSource): X is the
// RMSNorm of the row, or SwiGLU of its interleaved gate / up pairs, formed here with the f32
// operations of k_rmsnorm and k_swiglu_rows: no launch and no pass through memory for X itself
// (512 x 2048 norm + split 10.4 -> 6.7 us, 512 x 5632 SwiGLU + split 13.2 -> 8.0); only a row
// left to plain_block is written to src.rows.
template <bool NAT, int SRC>
__global__ __launch_bounds__(512) void k_x_split(const XSource src, half8* __restrict__ xp,
                                                 int32_t* __restrict__ sh, float* __restrict__ sx,
                                                 XRest* __restrict__ rest, int64_t k, int64_t mp) {
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x, units = k >> 3;
    const float4* xr = reinterpret_cast<const float4*>(src.x + row * k * (SRC == XSource::SWIGLU ? 2 : 1));
    const float4* nw = reinterpret_cast<const float4*>(src.norm);
    __shared__ uint32_t red[8];
    __shared__ float redf[8];
    __shared__ int s_rests;
    __shared__ XRest s_rest[X2_REST];
    if (tid == 0) s_rests = 0;
    float rms = 1.f;
    auto read = [&](int64_t i) {  // four elements of X (RMSNorm: of the row it normalizes)
        if constexpr (SRC == XSource::SWIGLU) {
            const float4 a = xr[2 * i], b = xr[2 * i + 1];
            auto f = [](float g, float u) { return (g * (1.0f / (1.0f + expf(-g)))) * u; };
            return make_float4(f(a.x, a.y), f(a.z, a.w), f(b.x, b.y), f(b.z, b.w));
        } else {
            return xr[i];
        }
    };
    auto normed = [&](float4 a, const float4& w) {
        if constexpr (SRC == XSource::RMSNORM)
            a = make_float4(a.x / rms * w.x, a.y / rms * w.y, a.z / rms * w.z, a.w / rms * w.w);
        return a;
    };
    auto value = [&](int64_t i) { return SRC == XSource::RMSNORM ? normed(xr[i], nw[i]) : read(i); };
    auto at = [&](int64_t u, int h) {  // float4 index of half h of unit u = block * 4 + word
        return NAT ? 2 * u + h : (u >> 2) * 8 + (u & 3) + 4 * h;
    };
    constexpr int R = 3;  // 8-element words per thread held in registers
    float4 v[R][2];
    uint32_t mx = 0;
    auto amax = [&](const float4& a) {
        mx = max(max(mx, __float_as_uint(a.x) & 0x7FFFFFFFu), __float_as_uint(a.y) & 0x7FFFFFFFu);
        mx = max(max(mx, __float_as_uint(a.z) & 0x7FFFFFFFu), __float_as_uint(a.w) & 0x7FFFFFFFu);
    };
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int64_t u = tid + 512 * i;
        const bool on = u < units;
#pragma unroll
        for (int h = 0; h < 2; h++) v[i][h] = on ? read(at(u, h)) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if constexpr (SRC == XSource::RMSNORM) {
        float4 wv[R][2];
        float ss = 0.f;
        auto add = [&](const float4& a) { ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w; };
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int64_t u = tid + 512 * i;
#pragma unroll
            for (int h = 0; h < 2; h++) wv[i][h] = u < units ? nw[at(u, h)] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int i = 0; i < R; i++) {
            add(v[i][0]);
            add(v[i][1]);
        }
        for (int64_t u = tid + 512 * R; u < units; u += 512) {
            add(xr[2 * u]);
            add(xr[2 * u + 1]);
        }
        ss = wave_allsum(ss);
        if ((tid & 63) == 0) redf[tid >> 6] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) ss += redf[i];
        rms = sqrtf(ss / (float)k + src.eps);
#pragma unroll
        for (int i = 0; i < R; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) v[i][h] = normed(v[i][h], wv[i][h]);
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
        amax(v[i][0]);
        amax(v[i][1]);
    }
    for (int64_t u = tid + 512 * R; u < units; u += 512) {
        amax(value(2 * u));
        amax(value(2 * u + 1));
    }
    mx = max(mx, lane_pair_dpp<1>(mx));
    mx = max(mx, lane_pair_dpp<2>(mx));
    mx = max(mx, lane_pair_dpp<4>(mx));
    mx = max(mx, lane_pair_dpp<8>(mx));
    mx = max(mx, lane_xor_u32<16>(mx));
    mx = max(mx, lane_xor_u32<32>(mx));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) mx = max(mx, red[i]);
    const bool bad = mx >= 0x7F800000u;
    // exponent of the largest magnitude (a subnormal's from its leading bit)
    const int e = mx >= 0x00800000u ? (int)(mx >> 23) - 127 : mx ? -118 - __clz(mx) : 14;
    const int s = bad ? 0 : 14 - e;
    half8* o = xp + row * units * 2;
    auto put = [&](int64_t u, const float4& a, const float4& b) {
        const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        half8 hi, lo;
        float sum = 0.f, least = 1.f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float y = bad ? 0.f : ldexpf(f[j], s);
            hi[j] = (_Float16)y;
            lo[j] = (_Float16)((y - (float)hi[j]) * X2_LO);
            sum += y;
            least = fminf(least, fabsf(y));
        }
        // (from 2^-14 on hi is a normal f16, and what it leaves is lo's to 2^-23 of the entry)
        if (least < 0x1p-14f && !bad) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float left = f[j] - ldexpf(fmaf((float)lo[j], 1.0f / X2_LO, (float)hi[j]), -s);
                if (fabsf(left) > 0x1p-23f * fabsf(f[j])) {
                    const int i = atomicAdd(&s_rests, 1);
                    if (i < X2_REST) s_rest[i] = XRest{(int32_t)(at(u, j >> 2) * 4 + (j & 3)), left};
                    sum -= ldexpf(left, s);  // rest_dot takes the whole weight
                }
            }
        }
        half8* p = o + (u >> 2) * 8 + (u & 3);
        p[0] = hi;
        p[4] = lo;
        if (sx) {  // the unit of 32's sum: its four words sit in four neighbouring lanes
            sum += dpp_f<0xB1>(sum);
            sum += dpp_f<0x4E>(sum);
            if ((u & 3) == 0) sx[(u >> 2) * mp + row] = sum;
        }
    };
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int64_t u = tid + 512 * i;
        if (u < units) put(u, v[i][0], v[i][1]);
    }
    for (int64_t u = tid + 512 * R; u < units; u += 512) put(u, value(at(u, 0)), value(at(u, 1)));
    __syncthreads();
    const int rests = s_rests;
    const bool plain = bad || rests > X2_REST;
    if (tid == 0) sh[row] = plain ? INT_MIN : (rests << 16) | (-s & 0xFFFF);
    if (!plain && tid < rests) {  // in element order, whatever order they came in
        int before = 0;
        for (int i = 0; i < rests; i++) before += s_rest[i].at < s_rest[tid].at;
        rest[row * X2_REST + before] = s_rest[tid];
    }
    if (SRC != XSource::ROWS && plain) {
        float4* to = reinterpret_cast<float4*>(src.rows + row * k);
        auto keep = [&](int64_t u, const float4& a, const float4& b) {
            to[at(u, 0)] = a;
            to[at(u, 1)] = b;
        };
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int64_t u = tid + 512 * i;
            if (u < units) keep(u, v[i][0], v[i][1]);
        }
        for (int64_t u = tid + 512 * R; u < units; u += 512) keep(u, value(at(u, 0)), value(at(u, 1)));
    }
}

// whole-number operand of a unit: word g (4-bit types, nibble + off) or bytes 8g .. 8g + 7 (Q8_0)
__device__ __forceinline__ half8 int_operand_q4(uint32_t w, float o) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    const half2v off = {(_Float16)o, (_Float16)o};
    const half2v p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, false) + off;
    const half2v p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, true) + off;
    const half2v p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, false) + off;
    const half2v p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, true) + off;
    return half8{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}
// bytes b of w0, w1 -> b + off - 1024 (the f16 of 0x6400 | b is 1024 + b)
__device__ __forceinline__ half8 int_operand_bytes(uint32_t w0, uint32_t w1, float off) {
    const half2v o = {(_Float16)(off - 1024.0f), (_Float16)(off - 1024.0f)};
    half8 r;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint32_t bits = __builtin_amdgcn_perm(0x64646464u, h ? w1 : w0, p ? 0x04030402u : 0x04010400u);
            const half2v v = __builtin_bit_cast(half2v, bits) + o;
            r[4 * h + 2 * p] = v.x;
            r[4 * h + 2 * p + 1] = v.y;
        }
    return r;
}

// word c of a unit as dequant_block forms it: elements 4c .. 4c + 3 and 16 + 4c .. 16 + 4c + 3
template <int QT>
__device__ __forceinline__ void dequant_word(const QView& qv, int64_t blk, int c, float* v) {
    if constexpr (QT == TL_HIP_GGML_Q8_0) {
        const float d = __half2float(qv.d[blk]);
        const uint32_t* p = reinterpret_cast<const uint32_t*>(qv.qs + blk * 32);
        const uint32_t w0 = p[c], w1 = p[4 + c];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = d * (float)(int8_t)((w0 >> (8 * i)) & 0xFF);
            v[4 + i] = d * (float)(int8_t)((w1 >> (8 * i)) & 0xFF);
        }
    } else {
        const uint32_t w = reinterpret_cast<const uint32_t*>(qv.qs + blk * 16)[c];
        const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
        float d0, d1, m = 0.f;
        uint2 h = {0u, 0u};
        int o = 8;
        if constexpr (QT == TL_HIP_GGML_Q4_0) {
            d0 = d1 = __half2float(qv.d[blk]);
        } else if constexpr (QT == TL_HIP_GGML_Q4_K) {
            q4k_scale_min(reinterpret_cast<const uint4*>(qv.hdr)[blk >> 3], (int)(blk & 7), &d0, &m);
            d1 = d0;
            o = 0;
        } else {
            const float d = __half2float(qv.d[blk >> 3]);
            d0 = d * (float)qv.sc[2 * blk];
            d1 = d * (float)qv.sc[2 * blk + 1];
            h = reinterpret_cast<const uint2*>(qv.qh)[blk];
            h = uint2{((h.x >> (2 * c)) & 0x03030303u) << 4, ((h.y >> (2 * c)) & 0x03030303u) << 4};
            o = 32;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = d0 * (float)((int)(((lo | h.x) >> (8 * i)) & 0xFF) - o) - m;
            v[4 + i] = d1 * (float)((int)(((hi | h.y) >> (8 * i)) & 0xFF) - o) - m;
        }
    }
}

// The 16 x 16 outputs of a wavefront's row block that the planes do not hold, from X and the weights
// in f32 (lane (col, g): row col of X, weight row col, elements 4 g + e of the halves of a unit).
// Every lane takes part; a row's result comes from its own entries alone.  11008 x 4096, m = 512,
// all rows 1490 us, one 373, none 133 (k_qgemm_f32: 724; a dot product per lane 5500 and 344);
// 4096 x 11008, m = 16, all rows 60 (186).
template <int QT>
__device__ __attribute__((noinline)) floatx4 plain_block(const QView qv, const float* x, int64_t u0, int nblk, int g) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    const floatx4* xr = reinterpret_cast<const floatx4*>(x);
#pragma unroll 4
    for (int b = 0; b < nblk; b++) {
        const floatx4 x0 = xr[8 * b + g], x1 = xr[8 * b + 4 + g];
        float v[8];
        dequant_word<QT>(qv, u0 + b, g, v);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x0[e], v[e], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[e], v[4 + e], acc, 0, 0, 0);
    }
    return acc;
}

// what the planes of a row miss of one output: its entries in units u0 .. u0 + nblk of the weight row
template <int QT>
__device__ __attribute__((noinline)) float rest_dot(const QView qv, const XRest* r, int n, int64_t wu, int u0, int nblk) {
    float acc = 0.f;
    for (int i = 0; i < n; i++) {
        const int b = r[i].at >> 5, at = r[i].at & 31;
        if (b < u0 || b >= u0 + nblk) continue;
        float v[32], w = 0.f;
        dequant_block<QT>(qv, wu + b, v);
#pragma unroll
        for (int j = 0; j < 32; j++) w = at == j ? v[j] : w;
        acc = fmaf(r[i].rest, w, acc);
    }
    return acc;
}

// One-launch split K: an arrival counter per tile, zero at load and returned to zero by the
// tile's last-arriving split
constexpr int X2_ARRIVE_MAX = 1024, X2_FUSE_NSP = 16;
__device__ uint32_t g_x2_arrive[X2_ARRIVE_MAX];

// Workgroup tile BM (x rows) x BN (weight rows), eight wavefronts in a WM x WN grid; an
// iteration covers KB units, double-buffered in LDS by DMA (X planes, quants and scales), so
// that the loop's loads write no VGPR.  Where an iteration holds 4 units, neighbouring lanes of a
// DMA instruction take a row's neighbouring chunks (RM), which the L1 fetches as one request (one
// chunk of 64 rows per instruction made as many requests as lanes: Q8_0 4096 x 11008 at m = 16
// 26 -> 20 us), swizzled by row in LDS so that the fragment reads of 16 rows cover all banks.
// The 2-unit tiles, bound by issue, keep one chunk of 64 rows per instruction: rows of 2 chunks
// gain little in requests, and the prompt of 512 through 22 layers took 4.8 ms against 4.65.  Q6_K has a scale per 16 weights: two MFMAs per plane,
// each with half of the unit's weights zeroed.  Q4_K's value d q - m is formed as
// d (q - o) + (d o - m), the second part times the unit's sum of X (sx), with o the whole number
// in 0 .. 15 nearest to m / d: each part is then at most twice the weight itself (the second at
// most d / 2, or of the first's sign where o is 0 or 15), so that a weight near zero leaves no
// large parts to cancel.
// PL planes of X: 2, or 1 for the f16 path (Q6_K): a weight's exact value is then rounded to f16 in
// registers, as k_dequant_f16q rounds it, and the MFMAs gather the output themselves.
// blockIdx.x is dealt to the 8 XCDs in turn: each takes a contiguous run of tiles, x tiles of a
// weight tile next to each other, so a weight tile is fetched by one L2.
template <int QT, int PL, int BM, int BN, int KB, int WM, int WN, int OCC>
__global__ __launch_bounds__(512, OCC) void k_qgemm_x2(const QView qv, const half8* __restrict__ xp,
                                                       const int32_t* __restrict__ sh, const float* __restrict__ sx,
                                                       const float* __restrict__ x, float* y, const float* res, int m,
                                                       int64_t n, int nb, int mt, int tiles, int mp,
                                                       float* __restrict__ part, int64_t stride, int fuse,
                                                       const RopeKvEpi rk, const XRest* __restrict__ rest) {
    static_assert(WM * WN == 8, "eight wavefronts");
    constexpr bool Q8 = QT == TL_HIP_GGML_Q8_0, K4 = QT == TL_HIP_GGML_Q4_K, K6 = QT == TL_HIP_GGML_Q6_K;
    constexpr int TM = BM / (16 * WM), TN = BN / (16 * WN), QC = Q8 ? 2 : 1;
    // DMA instructions (64 lanes each) of an iteration
    constexpr int XC = 4 * PL, XJ = KB * BM * XC / 64, QJ = KB * QC * BN / 64, HJ = K6 ? KB / 2 * BN / 64 : 0;
    constexpr int DW = K4 ? 4 : KB / 2 + 1;  // scale words per row (Q4_0 / Q8_0: the aligned words around KB halves)
    constexpr int QR = KB * QC, HR = K6 ? KB / 2 : 1;  // 16-byte chunks of a row
    constexpr bool RM = KB >= 4;
    constexpr int DJ = K4 ? BN / 64 : DW * BN / 64, SJ = K4 && PL == 2 ? (KB * BM + 63) / 64 : 0;
    constexpr int XU = (XJ + 7) / 8, QU = (QJ + 7) / 8, HU = (HJ + 7) / 8, DU = (DJ + 7) / 8;
    static_assert(SJ <= 8, "tile");
    struct Stage {
        half8 X[XJ * 64];                       // [unit][row][XC chunks], chunk c of row r at xpos(c, r)
        uint4 Wq[QJ * 64];                      // RM: [row][QR], chunk c at c ^ wsw(row, QR); else [chunk][row]
        uint4 Wh[K6 ? HJ * 64 : 1];             // Q6_K high bits, laid out alike
        uint32_t Wd[DW * BN];                   // scales, RM: [row][word], else [word][row] (Q4_K: [row] super-block headers)
        float S[SJ ? SJ * 64 : 1];              // Q4_K: sums of X over the unit, [unit][row]
    };
    static_assert(OCC < 4 || 4 * sizeof(Stage) + 64 <= 160 * 1024, "two workgroups per CU");
    __shared__ __attribute__((aligned(16))) Stage S0, S1;
    auto xpos = [](int c, int r) { return PL == 2 ? c ^ (r & 7) : c ^ ((r >> 2) & 3); };  // a bijection of c
    auto wsw = [](int r, int n) { return n > 1 ? (r / (16 / n)) & (n - 1) : 0; };  // 16 rows over all banks
    auto qpos = [wsw](int c, int r, int n) { return RM ? r * n + (c ^ wsw(r, n)) : c * BN + r; };
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, col = lane & 15, g = lane >> 4;
    const int per = (int)gridDim.x >> 3, tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (tile >= tiles) return;
    // (tiles past the last leave before any barrier, the workgroup as a whole)
    const int64_t m0 = (int64_t)(tile % mt) * BM, n0 = (int64_t)(tile / mt) * BN;

    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(xp, (uint32_t)((int64_t)m * nb * 64 * PL));
    const __amdgpu_buffer_rsrc_t rq = buf_rsrc(qv.qs, (uint32_t)(n * nb * 16 * QC));
    const __amdgpu_buffer_rsrc_t rh = buf_rsrc(qv.qh, (uint32_t)(K6 ? n * nb * 8 : 0));
    const __amdgpu_buffer_rsrc_t rd =
        K4 ? buf_rsrc(qv.hdr, (uint32_t)(n * nb * 2)) : buf_rsrc(qv.d, (uint32_t)(K6 ? n * (nb >> 3) * 2 + 4 : n * nb * 2 + 4));
    const __amdgpu_buffer_rsrc_t rc = buf_rsrc(qv.sc, (uint32_t)(K6 ? n * nb * 2 : 0));
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sx, (uint32_t)(K4 ? (int64_t)nb * mp * 4 : 0));
    auto wrow = [&](int r) { return n0 + r < n ? n0 + r : n - 1; };  // rows past n feed no output
    uint32_t xo[XU], qo[QU], ho[HU ? HU : 1], dof[DU], so = 0;
#pragma unroll
    for (int u = 0; u < XU; u++) {
        const int slot = (wave + 8 * u) * 64 + lane, b = slot / (BM * XC), r = slot / XC % BM, c = xpos(slot % XC, r);
        const int64_t row = m0 + r < m ? m0 + r : m - 1;
        xo[u] = (uint32_t)((row * nb + b) * 64 * PL + c * 16);
    }
#pragma unroll
    for (int u = 0; u < QU; u++) {
        const int slot = (wave + 8 * u) * 64 + lane, r = RM ? slot / QR % BN : slot % BN, c = RM ? slot % QR ^ wsw(r, QR) : slot / BN;
        qo[u] = (uint32_t)(wrow(r) * nb * 16 * QC + c * 16);
    }
#pragma unroll
    for (int u = 0; u < HU; u++) {
        const int slot = (wave + 8 * u) * 64 + lane, r = RM ? slot / HR % BN : slot % BN, c = RM ? slot % HR ^ wsw(r, HR) : slot / BN;
        ho[u] = (uint32_t)(wrow(r) * nb * 8 + c * 16);
    }
#pragma unroll
    for (int u = 0; u < DU; u++) {  // the scale DMA starts at the last wavefront
        const int slot = (7 - wave + 8 * u) * 64 + lane;
        if (K4) dof[u] = (uint32_t)(wrow(slot % BN) * (nb >> 3) * 16);
        else if (K6) dof[u] = (uint32_t)(slot < KB / 2 * BN ? wrow(slot / (KB / 2)) * nb * 2 + 4 * (slot % (KB / 2))
                                                            : wrow(slot % BN) * (nb >> 3));  // the last words' is an index
        else dof[u] = (uint32_t)(((wrow(RM ? slot / DW % BN : slot % BN) * nb) >> 1) * 4 + (RM ? slot % DW : slot / BN) * 4);
    }
    if (K4) {
        const int slot = wave * 64 + lane, b = slot / BM, r = slot % BM;
        so = (uint32_t)(((int64_t)(b < KB ? b : 0) * mp + m0 + r) * 4);
    }
    auto issue = [&](int kb, Stage& st) {
#pragma unroll
        for (int u = 0; u < XU; u++)
            if (XJ % 8 == 0 || wave + 8 * u < XJ) buf_dma16(rx, xo[u], (uint32_t)kb * 64 * PL, &st.X[(wave + 8 * u) * 64]);
#pragma unroll
        for (int u = 0; u < QU; u++)
            if (QJ % 8 == 0 || wave + 8 * u < QJ) buf_dma16(rq, qo[u], (uint32_t)kb * 16 * QC, &st.Wq[(wave + 8 * u) * 64]);
        #pragma unroll
        for (int u = 0; u < HU; u++)
            if (HJ % 8 == 0 || wave + 8 * u < HJ) buf_dma16(rh, ho[u], (uint32_t)kb * 8, &st.Wh[(wave + 8 * u) * 64]);
#pragma unroll
        for (int u = 0; u < DU; u++) {
            const int dj = 7 - wave + 8 * u;
            if (DJ % 8 != 0 && dj >= DJ) continue;
            if constexpr (K4) {
                buf_dma16(rd, dof[u], (uint32_t)(kb >> 3) * 16, &st.Wd[dj * 256]);
            } else if constexpr (K6) {
                if (dj < KB / 2 * BN / 64) buf_dma4(rc, dof[u], (uint32_t)kb * 2, &st.Wd[dj * 64]);
                else buf_dma4(rd, ((dof[u] + (uint32_t)(kb >> 3)) >> 1) * 4, 0, &st.Wd[dj * 64]);
            } else {
                buf_dma4(rd, dof[u], (uint32_t)kb * 2, &st.Wd[dj * 64]);
            }
        }
        if (SJ && wave < SJ) buf_dma4(rs, so, (uint32_t)kb * (uint32_t)mp * 4, &st.S[wave * 64]);
    };

    // Where registers allow, even and odd units gather in sums of their own: half as many roundings
    // in a chain (4096 x 11008 at m = 301, one K range: 1.6e-7 of the 64-bit sums against 2.1e-7).
    constexpr int AC = PL == 2 && TM * TN <= 4 ? 2 : 1;
    floatx4 acc2[AC][TM][TN];
    auto& acc = acc2[0];
#pragma unroll
    for (int a = 0; a < AC; a++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc2[a][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](const Stage& st, int kb) {
#pragma unroll
        for (int b = 0; b < KB; b++) {
            half8 ah[TM], al[TM];
            floatx4 s4[TM];
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int r = (wm * TM + i) * 16 + col;
                ah[i] = st.X[(b * BM + r) * XC + xpos(g, r)];
                if constexpr (PL == 2) al[i] = st.X[(b * BM + r) * XC + xpos(4 + g, r)];
                if constexpr (K4 && PL == 2) s4[i] = *reinterpret_cast<const floatx4*>(&st.S[b * BM + (wm * TM + i) * 16 + 4 * g]);
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int r = (wn * TN + j) * 16 + col;
                half8 w;
                float d0, d1 = 0.f, off = -8.0f;
                if constexpr (K4) {
                    float mn;
                    q4k_scale_min(*reinterpret_cast<const uint4*>(&st.Wd[4 * r]), (kb + b) & 7, &d0, &mn);
                    off = -__builtin_amdgcn_fmed3f(rintf(mn * __builtin_amdgcn_rcpf(d0)), 0.f, 15.0f);  // 0 where d0 = mn = 0 (NaN)
                    d1 = -fmaf(off, d0, mn);
                }
                if constexpr (Q8) {
                    const uint2 q = reinterpret_cast<const uint2*>(&st.Wq[qpos(2 * b + (g >> 1), r, QR)])[g & 1];
                    w = int_operand_bytes(q.x ^ 0x80808080u, q.y ^ 0x80808080u, -128.0f);
                } else {
                    const uint32_t q = reinterpret_cast<const uint32_t*>(&st.Wq[qpos(b, r, QR)])[g];
                    if constexpr (K6) {
                        const uint2 h = reinterpret_cast<const uint2*>(&st.Wh[qpos(b / 2, r, HR)])[b & 1];
                        w = int_operand_bytes((q & 0x0F0F0F0Fu) | (((h.x >> (2 * g)) & 0x03030303u) << 4),
                                              ((q >> 4) & 0x0F0F0F0Fu) | (((h.y >> (2 * g)) & 0x03030303u) << 4), -32.0f);
                    } else {
                        w = int_operand_q4(q, off);
                    }
                }
                if constexpr (K6) {
                    const uint32_t scw = st.Wd[r * (KB / 2) + b / 2] >> (16 * (b & 1)), par = (uint32_t)((wrow(r) * (nb >> 3) + (kb >> 3)) & 1) * 16;
                    const float d = __half2float(__ushort_as_half((uint16_t)(st.Wd[KB / 2 * BN + r] >> par)));
                    d0 = d * (float)(int8_t)(scw & 0xFF);
                    d1 = d * (float)(int8_t)((scw >> 8) & 0xFF);
                } else if constexpr (!K4) {
                    const int h = (int)((wrow(r) * nb) & 1) + b;  // half of the row's words (kb is even)
                    d0 = __half2float(RM ? reinterpret_cast<const __half*>(&st.Wd[r * DW])[h]
                                         : __ushort_as_half((uint16_t)(st.Wd[(h >> 1) * BN + r] >> (16 * (h & 1)))));
                    if (b > 0 && kb + b >= nb) d0 = 0.f;  // a unit past the row's last (X's planes are finite)
                }
                if constexpr (PL == 1) {
                    // f16 path: the exact value (one scale per half of the word) rounded once to f16
                    static_assert(PL == 2 || K6, "one plane: Q6_K");
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int e = 0; e < 4; e++) w[4 * h + e] = (_Float16)((h ? d1 : d0) * (float)w[4 * h + e]);
#pragma unroll
                    for (int i = 0; i < TM; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], w, acc[i][j], 0, 0, 0);
                    continue;
                }
                const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
                const half8 wl = w * (_Float16)(1.0f / X2_LO);
                auto& au = acc2[b % AC];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    if constexpr (K6) {
                        const _Float16 z = (_Float16)0.0f;
                        const half8 w0 = {w[0], w[1], w[2], w[3], z, z, z, z}, w1 = {z, z, z, z, w[4], w[5], w[6], w[7]};
                        const half8 wl0 = {wl[0], wl[1], wl[2], wl[3], z, z, z, z}, wl1 = {z, z, z, z, wl[4], wl[5], wl[6], wl[7]};
                        floatx4 c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], w0, zero, 0, 0, 0);
                        floatx4 c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], w1, zero, 0, 0, 0);
                        c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], wl0, c0, 0, 0, 0);
                        c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], wl1, c1, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; e++) au[i][j][e] = fmaf(d1, c1[e], fmaf(d0, c0[e], au[i][j][e]));
                    } else {
                        floatx4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], w, zero, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], wl, c, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            au[i][j][e] = fmaf(d0, c[e], au[i][j][e]);
                            if constexpr (K4) au[i][j][e] = fmaf(d1, s4[i][e], au[i][j][e]);
                        }
                    }
                }
            }
        }
    };

    const int iters = (nb + KB - 1) / KB, itp = (iters + (int)gridDim.y - 1) / (int)gridDim.y;
    const int it0 = (int)blockIdx.y * itp, it1 = min(it0 + itp, iters);
    auto step = [&](int it, const Stage& cur, Stage& next) {
        __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0): this iteration's DMA has landed
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (it + 1 < it1) issue((it + 1) * KB, next);
        __builtin_amdgcn_sched_barrier(0);
        compute(cur, it * KB);
    };
    if (it0 < it1) issue(it0 * KB, S0);
    for (int it = it0; it < it1; it += 2) {
        step(it, S0, S1);
        if (it + 1 < it1) step(it + 1, S1, S0);
    }
    if constexpr (AC == 2)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] += acc2[1][i][j];
    // Split K: this range's sums go to its slice of part (stride floats apart), which k_x2_sum
    // adds in a launch of its own or, with fuse, the tile's last-arriving split does: slices
    // are then written through to the agent's point of coherence and read there.
    const bool split = gridDim.y > 1;
    float* const pb = part + (int64_t)blockIdx.y * stride;
    const int u0 = it0 * KB, un = min(it1 * KB, nb) - u0;
    const bool rope = PL == 1 && rk.q;  // RoPE and the KV append of a [q | k | v] projection instead of y
    const int64_t rpos = rope ? (int64_t)*rk.pos : 0;
    if (rope && !split) {
        // the pair (2i, 2i + 1) of a row sits in lanes col, col ^ 1
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                float v4[4], u4[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v4[e] = acc[i][j][e];
                    u4[e] = dpp_f<0xB1>(v4[e]);
                }
                const int64_t c = n0 + (wn * TN + j) * 16 + col, rb = m0 + (wm * TM + i) * 16 + 4 * g;
                if (c >= n) continue;
                const RopeCol cl = rope_col(rk, c);
                const bool odd = (col & 1) != 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int64_t r = rb + e;
                    if (r >= m) break;
                    float cs = 0.f, sn = 0.f;
                    if (cl.kind != 2) {
                        const int64_t ti = rope_tab(rk, cl, r, rpos);
                        cs = rk.ct[ti];
                        sn = rk.st[ti];
                    }
                    rope_kv_put(rk, cl, r, rpos, odd ? u4[e] : v4[e], odd ? v4[e] : u4[e], v4[e], cs, sn);
                }
            }
        return;
    }
    int scale[TM][4];  // a row's entry of sh, all requested at once (one by one: Q8_0 4096 x 11008 at m = 16 20.1 us, now 19.2)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t r = m0 + (wm * TM + i) * 16 + 4 * g + e;
            scale[i][e] = PL == 2 && r < m ? sh[r] : 0;
        }
    if constexpr (PL == 2)
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (!__ballot((scale[i][0] | scale[i][1] | scale[i][2] | scale[i][3]) < 0)) continue;  // uniform
            const int64_t r = m0 + (wm * TM + i) * 16 + col;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const floatx4 d = plain_block<QT>(qv, x + ((r < m ? r : m - 1) * nb + u0) * 32,
                                                  wrow((wn * TN + j) * 16 + col) * nb + u0, un, g);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[i][j][e] = scale[i][e] < 0 ? d[e] : acc[i][j][e];
            }
        }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int64_t r = m0 + (wm * TM + i) * 16 + 4 * g + e;
            if (r >= m) continue;
            const int s = scale[i][e];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int64_t c = n0 + (wn * TN + j) * 16 + col;
                if (c >= n) continue;
                float v = acc[i][j][e];
                if constexpr (PL == 2) {
                    if (s >= 0) {
                        v = ldexpf(v, (int16_t)s);
                        if (s >> 16) v += rest_dot<QT>(qv, rest + r * X2_REST, s >> 16, c * nb, u0, un);
                    }
                }
                if (!split) y[r * n + c] = res ? res[r * n + c] + v : v;
                else if (!fuse) pb[r * n + c] = v;
                else
                    __hip_atomic_store(reinterpret_cast<uint32_t*>(pb + r * n + c), __float_as_uint(v), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    if (!split || !fuse) return;
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's slice stores have completed
    __syncthreads();
    const int nsp = (int)gridDim.y;
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(g_x2_arrive + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = old == (uint32_t)(nsp - 1);
        if (last) __hip_atomic_store(g_x2_arrive + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last;
    }
    __syncthreads();
    if (!s_last) return;  // uniform per workgroup
    const __amdgpu_buffer_rsrc_t rp = buf_rsrc(part, (uint32_t)(nsp * stride * 4));
    constexpr int UPR = BN / 4;  // 4-column units per tile row
    for (int u = tid; u < BM * UPR; u += 512) {
        const int64_t r = m0 + u / UPR, c = n0 + 4 * (u % UPR);
        if (r >= m || c >= n) continue;
        // every slice's 16 bytes requested at once (past nsp the offset is the resource's size,
        // never more: those read 0 and the selects keep them out of the sum)
        u32x4 t[X2_FUSE_NSP];
#pragma unroll
        for (int p = 0; p < X2_FUSE_NSP; p++)
            t[p] = __builtin_amdgcn_raw_buffer_load_b128(rp, (uint32_t)((r * n + c) * 4), (int)(min(p, nsp) * stride * 4), CPOL_SC1);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int p = 0; p < X2_FUSE_NSP; p++) {
            const bool on = p < nsp;
            v.x = on ? v.x + __uint_as_float(t[p].x) : v.x;
            v.y = on ? v.y + __uint_as_float(t[p].y) : v.y;
            v.z = on ? v.z + __uint_as_float(t[p].z) : v.z;
            v.w = on ? v.w + __uint_as_float(t[p].w) : v.w;
        }
        if (rope) {  // a unit holds two whole pairs
            rope_kv_store4(rk, r, c, rpos, v);
            continue;
        }
        if (res) {
            const float4 q = *reinterpret_cast<const float4*>(res + r * n + c);
            v = make_float4(q.x + v.x, q.y + v.y, q.z + v.z, q.w + v.w);
        }
        *reinterpret_cast<float4*>(y + r * n + c) = v;
    }
}

// y = [res +] the nsp slices added in slice order (slices 16-byte aligned, stride floats apart)
__global__ __launch_bounds__(256) void k_x2_sum(const float* __restrict__ part, float* y, const float* res, int64_t mn,
                                                int64_t stride, int nsp, int vec) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= mn) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p = 0; p < nsp; p++) {
        const float4 t = *reinterpret_cast<const float4*>(part + p * stride + i);
        v = make_float4(v.x + t.x, v.y + t.y, v.z + t.z, v.w + t.w);
    }
    if (vec && i + 4 <= mn) {
        if (res) {
            const float4 q = *reinterpret_cast<const float4*>(res + i);
            v = make_float4(q.x + v.x, q.y + v.y, q.z + v.z, q.w + v.w);
        }
        *reinterpret_cast<float4*>(y + i) = v;
        return;
    }
    const float o[4] = {v.x, v.y, v.z, v.w};
    for (int j = 0; j < 4 && i + j < mn; j++) y[i + j] = res ? res[i + j] + o[j] : o[j];
}

// Tile and K split.  Tiles by input rows: up to 16 and 32 rows take tiles of those heights
// with 4 units per iteration (a short tile's iteration is bound by the DMA's latency); longer
// inputs take 64 x 128, 64 x 64 (small outputs, and one x tile) or, Q4_0 and Q8_0, 128 x 192 (where
// its fewer, larger tiles fill the CUs once: 11264 x 2048 at m = 512 74 us against 87 of 64 x
// 128; the K-quants' loop does not fit the registers there: Q6_K 4096 x 11008 at m = 512 508
// against 214).  Up to 64 rows 64 x 64 with 4 units and 32 x 64 come in too (the former's stages
// are too large for two workgroups per CU in Q8_0: 4096 x 11008 at m = 64 43 against 36 with 2 units).
// 128 x 192 tiles have registers for one sum per output only and take K ranges of up to 64 units,
// whose sum is as near to 64 bits as the two sums of 128 units in the others (11008 x 4096 at m =
// 512, one range: 2.1e-7 in 126 us against 1.5e-7 in 135 of 64 x 128).  The estimate (rounds of one
// workgroup per CU x iterations x time per iteration, us; a CU with a single workgroup hides
// less latency, hence `single`; a split pays for writing and reading its slices) was fitted to
// sweeps of 4 types, m 8 .. 512, 7 shapes and every split: the plan it picks is within 1 % of the
// sweep's fastest on average and 10 % at most (one table for all types: 4 to 6 % on average past 32
// rows, up to 36 %, and the K-quants on 128 x 192 up to 2.6 times).
struct X2Tile {
    int bm, bn, kb;
    double us, single;  // per iteration (0: no such tile); factor of a lone workgroup
    int most = 1 << 30;  // units of a K range
};
struct X2Plan {
    int cfg, bm, bn;
    int64_t mt, tiles, nsp;
};
struct X2Fit {
    double wg, split, each, sum;  // us per round, split and slice; slice bytes per us
};
static X2Plan plan_x2(const QWeight* w, int64_t m, const X2Tile* T, int lo, int hi, const X2Fit& f) {
    const int cus = state() ? state()->num_cus : 256;
    X2Plan best{};
    double least = 1e30;
    for (int c = lo; c <= hi; c++) {
        if (T[c].us == 0) continue;
        const int64_t mt = cdiv(m, T[c].bm), tiles = mt * cdiv(w->n, T[c].bn), iters = cdiv(w->nb, T[c].kb);
        for (int64_t ns = 1; ns <= std::min<int64_t>(iters, X2_FUSE_NSP); ns++) {
            const int64_t per = cdiv(iters, ns);
            if (per * T[c].kb > T[c].most || cdiv(iters, per) != ns || (ns > 1 && tiles * ns > 4 * cus)) continue;  // every range non-empty
            double us = (double)cdiv(tiles * ns, cus) * (per * T[c].us * (tiles * ns <= cus ? T[c].single : 1.0) + f.wg);
            if (ns > 1) us += f.split + f.each * ns + (double)ns * m * w->n * 4 / f.sum;
            if (us < least) {
                least = us;
                best = X2Plan{c, T[c].bm, T[c].bn, mt, tiles, ns};
            }
        }
    }
    return best;
}
static X2Plan plan_f32(const QWeight* w, int64_t m) {
    static const X2Tile LONG[4][3] = {
        {{128, 192, 2, 1.83, 0.91, 64}, {64, 128, 2, 0.605, 1.46}, {64, 64, 2, 0.37, 1.50}},    // Q4_0
        {{128, 192, 2, 1.80, 0.91, 64}, {64, 128, 2, 0.55, 1.46}, {64, 64, 2, 0.367, 1.50}},    // Q8_0
        {{128, 192, 2, 0, 0}, {64, 128, 2, 0.73, 1.46}, {64, 64, 2, 0.52, 1.50}},           // Q4_K
        {{128, 192, 2, 0, 0}, {64, 128, 2, 0.845, 1.46}, {64, 64, 2, 0.51, 1.50}}};         // Q6_K
    static const X2Tile MID[4][3] = {
        {{64, 64, 2, 0.317, 1.69}, {64, 64, 4, 0.71, 1.38}, {32, 64, 4, 0.542, 1.18}},
        {{64, 64, 2, 0.394, 1.69}, {64, 64, 4, 0, 0}, {32, 64, 4, 0.541, 1.18}},
        {{64, 64, 2, 0.475, 1.69}, {64, 64, 4, 0.944, 1.38}, {32, 64, 4, 0.653, 1.18}},
        {{64, 64, 2, 0.51, 1.69}, {64, 64, 4, 1.015, 1.38}, {32, 64, 4, 0.707, 1.18}}};
    static const X2Tile SHORT[2] = {{32, 64, 4, 0.448, 1.467}, {16, 128, 4, 0.506, 1.467}};
    const int t = w->ggml_type == TL_HIP_GGML_Q4_0 ? 0 : w->ggml_type == TL_HIP_GGML_Q8_0 ? 1
                : w->ggml_type == TL_HIP_GGML_Q4_K ? 2 : 3;
    X2Plan pl;
    if (m > 64) {
        pl = plan_x2(w, m, LONG[t], 0, 2, X2Fit{0.001, 0.32, 0.275, 1.685e6});
    } else if (m > 32) {
        pl = plan_x2(w, m, MID[t], 0, 2, X2Fit{0.0, 4.33, 0.102, 1.77e6});
        pl.cfg += 2;
    } else {
        pl = plan_x2(w, m, SHORT, m <= 16, m <= 16, X2Fit{0.2, 1.66, 0.08, 1.4e6});
        pl.cfg += 4;
    }
    return pl;
}
// Q6_K on the f16 path (m 16 .. 512, 8 shapes: within 3 % of the sweep's fastest on average)
static X2Plan plan_q6(const QWeight* w, int64_t m) {
    static const X2Tile T[7] = {{128, 128, 2, 0.72, 1.7}, {128, 64, 2, 0.40, 1.7}, {64, 128, 2, 0.41, 1.7}, {64, 64, 4, 0.66, 1.7},
                                {32, 64, 4, 0.49, 1.7}, {32, 128, 4, 0.54, 1.7}, {16, 128, 4, 0.60, 1.7}};
    return plan_x2(w, m, T, m <= 16 ? 6 : m <= 32 ? 4 : 0, m <= 16 ? 6 : m <= 32 ? 5 : 3, X2Fit{0.8, 3.4, 0.0, 8.7e5});
}
// One launch when no other stream can run a call that shares the arrival counters; past 64
// rows the slices are large and a launch of its own adds them faster (2048 x 5632, m 512:
// 44.2 against 45.5 us; m 16: 14.9 against 13.0 us).
static bool x2_fuse(const X2Plan& pl, const QWeight* w, int64_t m, size_t part_bytes, bool vec) {
    return pl.nsp > 1 && m <= 64 && pl.tiles <= X2_ARRIVE_MAX && w->n % 4 == 0 && vec && part_bytes < (1ull << 31) &&
           single_stream() && one_launch_merge();
}

// Returns -1 without launching when there is no memory for the workspace.
template <int QT>
static int launch_x2(const QWeight* w, const float* x, float* y, const float* res, int64_t m, hipStream_t s,
                     const XSource& src) {
    const X2Plan pl = plan_f32(w, m);
    const int64_t mp = cdiv(m, 128) * 128, mn = m * w->n, stride = cdiv(mn, 4) * 4;
    const size_t xb = ((size_t)m * w->k * 4 + 255) & ~size_t(255), shb = ((size_t)m * 4 + 255) & ~size_t(255);
    const size_t rb = (size_t)m * X2_REST * sizeof(XRest);
    const size_t sb = QT == TL_HIP_GGML_Q4_K ? (size_t)w->nb * mp * 4 : 0;
    const size_t pb = pl.nsp > 1 ? (size_t)pl.nsp * stride * 4 : 0;
    const int vec = ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(res)) & 15) == 0;
    const int fuse = x2_fuse(pl, w, m, pb, vec);
    uint8_t* ws = static_cast<uint8_t*>(dev_alloc_on(xb + shb + rb + sb + pb, s));
    if (!ws) {
        clear_error();
        return -1;
    }
    half8* xp = reinterpret_cast<half8*>(ws);
    int32_t* sh = reinterpret_cast<int32_t*>(ws + xb);
    XRest* rest = reinterpret_cast<XRest*>(ws + xb + shb);
    float* sx = sb ? reinterpret_cast<float*>(ws + xb + shb + rb) : nullptr;
    float* part = reinterpret_cast<float*>(ws + xb + shb + rb + sb);
    constexpr bool NAT = QT == TL_HIP_GGML_Q8_0;
    switch (src.kind) {
        case XSource::RMSNORM: k_x_split<NAT, XSource::RMSNORM><<<(unsigned)m, 512, 0, s>>>(src, xp, sh, sx, rest, w->k, mp); break;
        case XSource::SWIGLU: k_x_split<NAT, XSource::SWIGLU><<<(unsigned)m, 512, 0, s>>>(src, xp, sh, sx, rest, w->k, mp); break;
        default: k_x_split<NAT, XSource::ROWS><<<(unsigned)m, 512, 0, s>>>(src, xp, sh, sx, rest, w->k, mp); break;
    }
    const QView qv{w->qs, w->d, w->hdr, w->qh, w->sc};
    const dim3 grid((unsigned)(cdiv(pl.tiles, 8) * 8), (unsigned)pl.nsp);
#define TLH_X2(BM, BN, KB, WM, WN, OCC)                                                                              \
    k_qgemm_x2<QT, 2, BM, BN, KB, WM, WN, OCC><<<grid, 512, 0, s>>>(qv, xp, sh, sx, x, y, res, (int)m, w->n, (int)w->nb, \
                                                                 (int)pl.mt, (int)pl.tiles, (int)mp, part, stride, fuse, \
                                                                 RopeKvEpi{}, rest)
    // (tiles that the type's table leaves out are not built)
    constexpr bool Q4 = QT == TL_HIP_GGML_Q4_0, Q8 = QT == TL_HIP_GGML_Q8_0;
    switch (pl.cfg) {
        case 0:
            if constexpr (Q4 || Q8) TLH_X2(128, 192, 2, 2, 4, 2);
            break;
        case 1: TLH_X2(64, 128, 2, 1, 8, 4); break;
        case 2: TLH_X2(64, 64, 2, 2, 4, 4); break;
        case 3:
            if constexpr (!Q8) TLH_X2(64, 64, 4, 2, 4, 4);
            break;
        case 4: TLH_X2(32, 64, 4, 2, 4, 4); break;
        default: TLH_X2(16, 128, 4, 1, 8, 4); break;
    }
#undef TLH_X2
    if (pl.nsp > 1 && !fuse)
        k_x2_sum<<<(unsigned)cdiv(stride / 4, 256), 256, 0, s>>>(part, y, res, mn, stride, (int)pl.nsp, vec);
    dev_free_on(ws, s);  // freed on s: reused at once only by later work on s
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TL_HIP_OK : hip_fail(e, "quant gemm launch");
}

// y = [res +] x16 . W^T, or the RoPE / KV epilogue of ep, on the f16 path, x16 [m, k] in the nibble operand order.  The weights went
// through an f16 copy per call before (2048 x 5632, m 301: 42 -> 33.9 us; 32000 x 2048, m 16: 78 ->
// 23); what bounds it now is the dequantization in registers (26 VALU instructions per eight
// weights, shared by the tile's rows) beside the matrix cores.
int launch_gemm_q6_f16(const QWeight* w, const _Float16* x16, float* y, int64_t m, const GemmEpi& ep, hipStream_t s,
                       int plan[3]) {
    const float* res = ep.mode == GEMM_RES ? ep.res : nullptr;
    const bool rope = ep.mode == GEMM_ROPE_KV;
    const RopeKvEpi rk = rope ? ep.rk : RopeKvEpi{};
    const X2Plan pl = plan_q6(w, m);
    const int64_t mn = m * w->n, stride = cdiv(mn, 4) * 4;
    const size_t pb = pl.nsp > 1 ? (size_t)pl.nsp * stride * 4 : 0;
    const int vec = rope || ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(res)) & 15) == 0;
    const int fuse = x2_fuse(pl, w, m, pb, vec);
    float* part = pb ? static_cast<float*>(dev_alloc_on(pb, s)) : nullptr;
    if (pb && !part) return TL_HIP_ERR_ALLOC;
    plan[0] = pl.bm, plan[1] = pl.bn, plan[2] = (int)pl.nsp;
    const half8* xp = reinterpret_cast<const half8*>(x16);
    const QView qv{w->qs, w->d, w->hdr, w->qh, w->sc};
    const dim3 grid((unsigned)(cdiv(pl.tiles, 8) * 8), (unsigned)pl.nsp);
#define TLH_Q6(BM, BN, KB, WM, WN)                                                                                     \
    k_qgemm_x2<TL_HIP_GGML_Q6_K, 1, BM, BN, KB, WM, WN, 4><<<grid, 512, 0, s>>>(                                       \
        qv, xp, nullptr, nullptr, nullptr, y, res, (int)m, w->n, (int)w->nb, (int)pl.mt, (int)pl.tiles, 0, part, stride,         \
        fuse, rk, nullptr)
    switch (pl.cfg) {
        case 0: TLH_Q6(128, 128, 2, 2, 4); break;
        case 1: TLH_Q6(128, 64, 2, 2, 4); break;
        case 2: TLH_Q6(64, 128, 2, 1, 8); break;
        case 3: TLH_Q6(64, 64, 4, 2, 4); break;
        case 4: TLH_Q6(32, 64, 4, 2, 4); break;
        case 5: TLH_Q6(32, 128, 4, 1, 8); break;
        default: TLH_Q6(16, 128, 4, 1, 8); break;
    }
#undef TLH_Q6
    if (pl.nsp > 1 && !fuse) {
        if (rope) launch_splitk_sum_rope(part, m, w->n, (int)pl.nsp, rk, s);
        else k_x2_sum<<<(unsigned)cdiv(stride / 4, 256), 256, 0, s>>>(part, y, res, mn, stride, (int)pl.nsp, vec);
    }
    if (part) dev_free_on(part, s);  // freed on s: reused at once only by later work on s
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TL_HIP_OK : hip_fail(e, "quant gemm launch");
}

// res: y = res + X . W^T (res may be y).
int launch_quant_gemm_f32(const QWeight* w, const float* x, float* y, int64_t m, hipStream_t s, const float* res,
                          bool workspace, const XSource* from) {
    const XSource src = from ? *from : XSource{XSource::ROWS, x, nullptr, 0.f, nullptr};
    if (from) x = from->rows;
    // k_qgemm_x2's buffer offsets are 32-bit, and grids (512 threads a row of X and a tile, 64 x 64 past
    // 64 rows) have fewer than 2^32 threads; a call under capture takes no workspace, which the graph's
    // replays would find in other hands
    const int64_t lim = 1ll << 31, mp = cdiv(m, 128) * 128;
    if (workspace && m * w->k * 4 < lim && w->n * w->k < lim && w->nb * mp * 4 < lim &&
        m < (1 << 23) && cdiv(m, 64) * cdiv(w->n, 64) < (1 << 23) - 8) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) {
            int rc;
            switch (w->ggml_type) {
                case TL_HIP_GGML_Q4_0: rc = launch_x2<TL_HIP_GGML_Q4_0>(w, x, y, res, m, s, src); break;
                case TL_HIP_GGML_Q8_0: rc = launch_x2<TL_HIP_GGML_Q8_0>(w, x, y, res, m, s, src); break;
                case TL_HIP_GGML_Q4_K: rc = launch_x2<TL_HIP_GGML_Q4_K>(w, x, y, res, m, s, src); break;
                default: rc = launch_x2<TL_HIP_GGML_Q6_K>(w, x, y, res, m, s, src); break;
            }
            if (rc != -1) return rc;
        }
    }
    if (from) {
        const int rc = src.kind == XSource::RMSNORM
                           ? launch_rmsnorm(src.x, nullptr, src.norm, from->rows, m, w->k, src.eps, 0, s)
                           : launch_swiglu_rows(src.x, from->rows, m, w->k, s);
        if (rc) return rc;
    }
    dim3 grid((unsigned)cdiv(w->n, F_BN), (unsigned)cdiv(m, F_BM));
    const QView qv{w->qs, w->d, w->hdr, w->qh, w->sc};
    switch (w->ggml_type) {
        case TL_HIP_GGML_Q4_0: k_qgemm_f32<TL_HIP_GGML_Q4_0><<<grid, 256, 0, s>>>(qv, x, y, res, m, w->n, w->k, w->nb); break;
        case TL_HIP_GGML_Q8_0: k_qgemm_f32<TL_HIP_GGML_Q8_0><<<grid, 256, 0, s>>>(qv, x, y, res, m, w->n, w->k, w->nb); break;
        case TL_HIP_GGML_Q4_K: k_qgemm_f32<TL_HIP_GGML_Q4_K><<<grid, 256, 0, s>>>(qv, x, y, res, m, w->n, w->k, w->nb); break;
        default: k_qgemm_f32<TL_HIP_GGML_Q6_K><<<grid, 256, 0, s>>>(qv, x, y, res, m, w->n, w->k, w->nb); break;
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TL_HIP_OK : hip_fail(e, "quant gemm launch");
}

}  // namespace tlhip
