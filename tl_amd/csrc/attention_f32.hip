// f32 attention over many query rows: the scaled-dot-product-attention operator and the f32
// path's prefill.  One pass over the keys with an online softmax, products on the f32 matrix
// instruction (v_mfma_f32_16x16x4_f32: f32 operands, f32 sums).
//
// Rows are (query, head) pairs that share a slice's keys and values; a workgroup of RW x PW
// wavefronts takes 16 RW of them, wavefront (rw, pw) 16 rows and every PW-th part of each tile of
// TP positions.  S^T = K Q^T leaves lane (col, g) the scores of row col at positions 4g .. 4g+3
// of each 16, so the mask, the running maximum and the sum need two cross-lane exchanges a tile,
// and those registers are the P operand of O^T = V^T P^T as they stand (the k slots of an MFMA
// are positions 4g + e of the four lane groups).  K and V tiles reach LDS by DMA, the next tile
// under this one's MFMAs; 16-byte chunks are swizzled so that the fragment reads (K: 16 or 8
// bytes per lane of 16 rows; V: one element of 16 columns in four rows) spread over the banks.
//
// What bounds it: the f32 matrix instructions and the VALU work between them, which share one
// pipe (2 x 1.07 GFLOP of MFMA take 14 us at the f32 rate and the softmax about as long again,
// whatever the number of wavefronts); at short inputs, launch and the chain of tiles.  us per
// call before (one workgroup per query row, which re-read the slice's keys and values) -> now:
// [32, 512, 64] with a mask 899 -> 30, [32, 512, 128] 1351 -> 44, 1 query over 700 keys of 32
// heads 114 -> 14; a 512-token prompt, 32 heads over 4 KV heads of 64, f32 cache 163 -> 23.
// Relative error against 64 bits 1.5e-7 / 2.7e-7 at the first two (2.0e-7 / 4.3e-7 before).

#include "gemm_common.h"

#include <type_traits>

namespace tlhip {

struct AttnF32Args {
    const float* q;
    const void* k;
    const void* v;
    const float* mask;  // [mask_len] flat over (query, key), or null
    float* out;
    const int32_t* pos_dev;  // CAUSAL: query i attends keys 0 .. pos + i
    int64_t mask_len;
    int64_t q_gs, q_is, q_hs, o_gs, o_is, o_hs, k_gs, v_gs;  // strides in elements: slice, query, head
    int rows, G, n, dk, dv, sk;                              // rows = n G per slice
    float scale;
};

template <typename KVT, int DP, int RW, int PW, int TP, bool CAUSAL>
__global__ __launch_bounds__(64 * RW * PW) void k_attn_f32(const AttnF32Args a) {
    constexpr bool H16 = std::is_same_v<KVT, __half>;
    constexpr int W = RW * PW, NT = TP / 16 / PW, EB = sizeof(KVT), CH = 16 / EB, CK = DP / CH;
    constexpr int U = TP * CK / (64 * W);  // DMA instructions per wavefront for K, and for V
    static_assert(NT >= 1 && U >= 1 && U * 64 * W == TP * CK, "tile");
    struct Stage {
        uint4 K[TP * CK], V[TP * CK];
    };
    constexpr int RS = DP / 4 + 2;  // words per lane that a part of a row leaves for the merge
    struct Merge {
        float w[RW * (PW - 1) * RS * 64 + 1];
    };
    union First {
        Stage st;
        Merge mg;
    };
    __shared__ __attribute__((aligned(16))) First F0;
    __shared__ __attribute__((aligned(16))) Stage S1;
    Stage& S0 = F0.st;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave / PW, pw = wave % PW, col = lane & 15, g = lane >> 4;
    const int64_t grp = blockIdx.x;
    const int r0 = (CAUSAL ? (int)(gridDim.y - 1 - blockIdx.y) : (int)blockIdx.y) * 16 * RW;  // the longest rows first
    const int pos0 = CAUSAL ? *a.pos_dev : 0;
    const int row = min(r0 + rw * 16 + col, a.rows - 1), qi = row / a.G, qh = row - qi * a.G;
    const int limit = CAUSAL ? pos0 + a.n : a.sk;  // keys that exist
    // keys that this row, this wavefront's rows and the workgroup's rows reach
    const int mine = CAUSAL ? pos0 + qi + 1 : a.sk;
    const int wlast = CAUSAL ? pos0 + min(r0 + rw * 16 + 15, a.rows - 1) / a.G + 1 : a.sk;
    const int last = CAUSAL ? pos0 + min(r0 + 16 * RW - 1, a.rows - 1) / a.G + 1 : a.sk;

    // Rows past the limit and columns past the head size lie outside the resources and read 0.
    const uint32_t kb = (uint32_t)a.dk * EB, vb = (uint32_t)a.dv * EB;
    const __amdgpu_buffer_rsrc_t rk = buf_rsrc(static_cast<const KVT*>(a.k) + grp * a.k_gs, (uint32_t)limit * kb);
    const __amdgpu_buffer_rsrc_t rv = buf_rsrc(static_cast<const KVT*>(a.v) + grp * a.v_gs, (uint32_t)limit * vb);
    uint32_t ko[U], vo[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int slot = (wave * U + u) * 64 + lane, r = slot / CK, c = slot % CK;
        const uint32_t ck = (uint32_t)(c ^ (H16 ? r & 7 : r & 15)) * 16;
        const uint32_t cv = (uint32_t)(c ^ (((r >> 2) & 3) << (H16 ? 1 : 2))) * 16;
        ko[u] = ck < kb ? (uint32_t)r * kb + ck : 0x7FFFFFF0u;
        vo[u] = cv < vb ? (uint32_t)r * vb + cv : 0x7FFFFFF0u;
    }
    auto issue = [&](int j0, Stage& st) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++)
            buf_dma16(rk, ko[u], (uint32_t)j0 * kb, &st.K[(wave * U + u) * 64]);
#pragma unroll
        for (int u = 0; u < U; u++)
            buf_dma16(rv, vo[u], (uint32_t)j0 * vb, &st.V[(wave * U + u) * 64]);
    };
    issue(0, S0);

    floatx4 qf[DP / 16];
    const float* qp = a.q + grp * a.q_gs + qi * a.q_is + qh * a.q_hs;
#pragma unroll
    for (int s = 0; s < DP / 16; s++)
        qf[s] = 16 * s + 4 * g < a.dk ? *reinterpret_cast<const floatx4*>(qp + 16 * s + 4 * g) : floatx4{0.f, 0.f, 0.f, 0.f};

    // e^x: 2^y of y = x log2(e) rounded, times 1 + ln(2) (x log2(e) - y), which takes the rounding
    // of y (2^-24 of its magnitude, an error of e^x that grows with x) out again
    auto expx = [](float x) {
        constexpr float L2E = 1.44269504088896340736f, L2E_LO = 1.92596299112661746887e-8f, LN2 = 0.69314718055994530942f;
        const float y = x * L2E, r = fmaf(x, L2E_LO, fmaf(x, L2E, -y)), p = __builtin_amdgcn_exp2f(y);
        return x < -100.0f ? p : fmaf(p, r * LN2, p);
    };
    float m = -INFINITY, l = 0.f;
    floatx4 acc[DP / 16];
#pragma unroll
    for (int d = 0; d < DP / 16; d++) acc[d] = floatx4{0.f, 0.f, 0.f, 0.f};

    // this tile's mask entries, four keys at a time where rows are whole float4s
    float mk[NT][4];
    auto load_mask = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int j = j0 + (pw * NT + t) * 16 + 4 * g;
            const int64_t mi = (int64_t)qi * a.sk + j;
            if ((a.sk & 3) == 0 && j < a.sk && mi + 4 <= a.mask_len) {
                const float4 v = *reinterpret_cast<const float4*>(a.mask + mi);
                mk[t][0] = v.x, mk[t][1] = v.y, mk[t][2] = v.z, mk[t][3] = v.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) mk[t][e] = j + e < a.sk && mi + e < a.mask_len ? a.mask[mi + e] : 1.0f;
            }
        }
    };
    auto compute = [&](const Stage& st, int j0) __attribute__((always_inline)) {
        if (CAUSAL && j0 + pw * NT * 16 >= wlast) return;  // nothing of this wavefront's part is attended
        floatx4 s[NT], sp[NT][4];  // four sums per score, added at the end: shorter chains, fewer roundings in each
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) sp[t][e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DP / 16; c++)
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int r = (pw * NT + t) * 16 + col;
                floatx4 kf;
                if constexpr (H16) {
                    typedef _Float16 half4v __attribute__((ext_vector_type(4)));
                    const half4v h = reinterpret_cast<const half4v*>(&st.K[r * CK + ((2 * c + (g >> 1)) ^ (r & 7))])[g & 1];
                    kf = floatx4{(float)h.x, (float)h.y, (float)h.z, (float)h.w};
                } else {
                    kf = *reinterpret_cast<const floatx4*>(&st.K[r * CK + ((4 * c + g) ^ (r & 15))]);
                }
#pragma unroll
                for (int e = 0; e < 4; e++) sp[t][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[c][e], sp[t][e], 0, 0, 0);
            }
#pragma unroll
        for (int t = 0; t < NT; t++) s[t] = (sp[t][0] + sp[t][1]) + (sp[t][2] + sp[t][3]);
        float mt = -INFINITY;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int j = j0 + (pw * NT + t) * 16 + 4 * g + e;
                float x = s[t][e] * a.scale;
                if (!CAUSAL && a.mask && mk[t][e] == 0.0f) x = -1e9f;
                if (j >= mine) x = -INFINITY;
                s[t][e] = x;
                mt = fmaxf(mt, x);
            }
        mt = lane_pair_max<16>(mt);
        mt = lane_pair_max<32>(mt);
        const float mn = fmaxf(m, mt), ms = mn == -INFINITY ? 0.f : mn;  // no key yet: every weight 0
        const float al = expx(m - ms);
        m = mn;
        float ps = 0.f;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                s[t][e] = expx(s[t][e] - ms);
                ps += s[t][e];
            }
        l = l * al + ps;  // this lane's positions; the four lane groups' sums are added at the end
#pragma unroll
        for (int d = 0; d < DP / 16; d++) acc[d] *= al;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = (pw * NT + t) * 16 + 4 * g + e;
#pragma unroll
                for (int d = 0; d < DP / 16; d++) {
                    float vf;
                    if constexpr (H16)
                        vf = (float)reinterpret_cast<const _Float16*>(&st.V[r * CK + ((2 * d + (col >> 3)) ^ (g << 1))])[col & 7];
                    else
                        vf = reinterpret_cast<const float*>(&st.V[r * CK + ((4 * d + (col >> 2)) ^ (g << 2))])[col & 3];
                    acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf, s[t][e], acc[d], 0, 0, 0);
                }
            }
    };
    auto step = [&](int j0, const Stage& cur, Stage& next, auto live) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0): this tile's DMA has landed
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (!CAUSAL && live && a.mask) load_mask(j0);  // before the DMA: a wait for these loads leaves it in flight
        if (j0 + TP < last) issue(j0 + TP, next);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(live)::value) compute(cur, j0);
    };
    auto tiles = [&](auto live) __attribute__((always_inline)) {
        for (int j0 = 0; j0 < last; j0 += 2 * TP) {
            step(j0, S0, S1, live);
            if (j0 + TP < last) step(j0 + TP, S1, S0, live);
        }
    };
    if (RW == 1 || r0 + rw * 16 < a.rows) tiles(std::true_type{});
    else tiles(std::false_type{});  // no rows in this wavefront's block: its share of the DMA, and the barriers
    l = lane_pair_sum<16>(l);
    l = lane_pair_sum<32>(l);
    if constexpr (PW > 1) {  // the parts of a row are added by its first wavefront
        __syncthreads();
        float* red = F0.mg.w;
        float* w = red + rw * (PW - 1) * RS * 64 + lane;  // parts 1 .. PW - 1 of this row block
        if (pw > 0) {
            float* o = w + (pw - 1) * RS * 64;
            o[0] = m;
            o[64] = l;
#pragma unroll
            for (int d = 0; d < DP / 16; d++)
#pragma unroll
                for (int e = 0; e < 4; e++) o[(2 + 4 * d + e) * 64] = acc[d][e];
        }
        __syncthreads();
        if (pw > 0) return;
        float mx = m;
#pragma unroll
        for (int p = 0; p < PW - 1; p++) mx = fmaxf(mx, w[p * RS * 64]);
        const float ms = mx == -INFINITY ? 0.f : mx, f0 = expx(m - ms);
        m = mx;
        l *= f0;
#pragma unroll
        for (int d = 0; d < DP / 16; d++) acc[d] *= f0;
#pragma unroll
        for (int p = 0; p < PW - 1; p++) {
            const float f = expx(w[p * RS * 64] - ms);
            l = fmaf(w[(p * RS + 1) * 64], f, l);
#pragma unroll
            for (int d = 0; d < DP / 16; d++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[d][e] = fmaf(w[(p * RS + 2 + 4 * d + e) * 64], f, acc[d][e]);
        }
    }
    if (r0 + rw * 16 + col >= a.rows) return;
    if constexpr (CAUSAL) {
        // A tile's products give a key past the row the weight 0, which an infinite or NaN value
        // there does not respect: such a row takes its own keys one by one instead.
        bool off = false;
#pragma unroll
        for (int d = 0; d < DP / 16; d++)
#pragma unroll
            for (int e = 0; e < 4; e++) off |= (__float_as_uint(acc[d][e]) & 0x7F800000u) == 0x7F800000u;
        if (off) {
#pragma unroll
            for (int d = 0; d < DP / 16; d++) acc[d] = floatx4{0.f, 0.f, 0.f, 0.f};
            const KVT* kr = static_cast<const KVT*>(a.k) + grp * a.k_gs;
            const KVT* vr = static_cast<const KVT*>(a.v) + grp * a.v_gs;
#pragma unroll 1
            for (int j = 0; j < mine; j++, kr += a.dk, vr += a.dv) {
                float x = 0.f;
#pragma unroll 4
                for (int i = 0; i < a.dk; i++) x = fmaf(qp[i], (float)kr[i], x);
                const float p = expx(x * a.scale - m);
#pragma unroll
                for (int d = 0; d < DP / 16; d++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (16 * d + 4 * g < a.dv) acc[d][e] = fmaf(p, (float)vr[16 * d + 4 * g + e], acc[d][e]);
            }
        }
    }
    const float inv = 1.0f / l;
    float* op = a.out + grp * a.o_gs + qi * a.o_is + qh * a.o_hs;
#pragma unroll
    for (int d = 0; d < DP / 16; d++)
        if (16 * d + 4 * g < a.dv) *reinterpret_cast<floatx4*>(op + 16 * d + 4 * g) = acc[d] * inv;
}

// Workgroup shape (us, 512 keys): where two row blocks per workgroup give every CU one, K and V
// tiles are fetched for 32 rows and four (head size 64) wavefronts share each block's positions
// ([32, 512, 64] with a mask: 29.9 against 39.1 of 16-row workgroups); head size 128 takes 64
// rows by two wavefronts each where that still fills the CUs ([32, 512, 128]: 44.4 against 48.6;
// causal rows differ in length and stay on the smaller ones).  Slices alone may make up the
// count: wavefronts whose block holds no rows then skip the tile's work (1 query, 512 keys: 1024
// slices of 64 61 -> 44, 256 of 128 52 -> 33 us), and at head size 128 up to 32 rows of two or more
// slices per CU take the 32-row form, of which two fit a CU (1024 slices of 128: 121 against 139;
// 256: 43 against 33).  Shorter inputs take 16 rows by
// four wavefronts ([32, 128, 64]: 6.6 against 7.6), a single block of rows eight and longer tiles
// (1 query over 700 keys: 13.9 against 17.0).
template <typename KVT, bool CAUSAL>
static int attn_f32_launch(const AttnF32Args& a, int64_t groups, hipStream_t s) {
    const int64_t r16 = cdiv(a.rows, 16), cus = state() ? state()->num_cus : 256;
    const bool two = cdiv(r16, 2) * groups >= cus;
#define TLH_AF(DP, RW, PW, TP) \
    k_attn_f32<KVT, DP, RW, PW, TP, CAUSAL><<<dim3((unsigned)groups, (unsigned)cdiv(r16, RW)), 64 * RW * PW, 0, s>>>(a)
    if (a.dk <= 64 && a.dv <= 64) {
        if (two) TLH_AF(64, 2, 4, 64);
        else if (r16 > 1) TLH_AF(64, 1, 4, 64);
        else TLH_AF(64, 1, 8, 128);
    } else if (!CAUSAL && cdiv(r16, 4) * groups >= cus && (r16 > 2 || groups < 2 * cus)) {
        if constexpr (!CAUSAL) TLH_AF(128, 4, 2, 64);
    } else if (two) {
        constexpr int TP = std::is_same_v<KVT, __half> ? 64 : 32;  // two workgroups' stages per CU
        TLH_AF(128, 2, 2, TP);
    } else {
        TLH_AF(128, 1, 4, 64);
    }
#undef TLH_AF
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TL_HIP_OK : hip_fail(e, "attention launch");
}

// 16-byte rows (f32: head sizes in steps of 4), head sizes up to 128, 32-bit offsets within a
// slice's keys and values, and a grid of fewer than 2^32 threads per dimension (at most 512 per slice).
bool sdpa_f32_supported(int64_t slices, int64_t sq, int64_t sk, int64_t dk, int64_t dv) {
    return dk % 4 == 0 && dv % 4 == 0 && dk >= 4 && dv >= 4 && dk <= 128 && dv <= 128 && sq >= 1 && sk >= 1 &&
           sk < (1 << 20) && cdiv(sq, 16) <= 65535 && slices < (1 << 23);
}

int launch_sdpa_f32(const float* q, const float* k, const float* v, const float* mask, int64_t mask_len, float* out,
                    int64_t slices, int64_t sq, int64_t sk, int64_t dk, int64_t dv, float scale, hipStream_t s) {
    AttnF32Args a{};
    a.q = q, a.k = k, a.v = v, a.mask = mask, a.mask_len = mask_len, a.out = out;
    a.q_gs = sq * dk, a.q_is = dk, a.o_gs = sq * dv, a.o_is = dv, a.k_gs = sk * dk, a.v_gs = sk * dv;
    a.rows = (int)sq, a.G = 1, a.n = (int)sq, a.dk = (int)dk, a.dv = (int)dv, a.sk = (int)sk, a.scale = scale;
    return attn_f32_launch<float, false>(a, slices, s);
}

// The shapes of the split forms (attention.hip), which take the decode steps that follow.
bool attention_prefill_f32_supported(int hq, int hkv, int D, int64_t n, int64_t lmax) {
    const int G = hkv > 0 && hq % hkv == 0 ? hq / hkv : 0;
    return (D == 64 || D == 128) && (G == 1 || G == 2 || G == 4 || G == 8) && lmax < (1 << 20) && cdiv(n * G, 16) <= 65535;
}

int launch_attention_prefill_f32(const float* q, const void* k, const void* v, int kv_dtype, float* out, int n, int hq,
                                 int hkv, int D, int64_t lmax, const int32_t* pos_dev, float scale, hipStream_t s) {
    AttnF32Args a{};
    a.q = q, a.k = k, a.v = v, a.out = out, a.pos_dev = pos_dev;
    a.G = hq / hkv;
    a.q_gs = a.o_gs = (int64_t)a.G * D, a.q_is = a.o_is = (int64_t)hq * D, a.q_hs = a.o_hs = D;
    a.k_gs = a.v_gs = lmax * D;
    a.rows = n * a.G, a.n = n, a.dk = a.dv = D, a.scale = scale;
    return kv_dtype == TL_HIP_F16 ? attn_f32_launch<__half, true>(a, hkv, s) : attn_f32_launch<float, true>(a, hkv, s);
}

}  // namespace tlhip
