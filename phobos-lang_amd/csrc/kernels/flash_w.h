// Flash attention for launches too small for flash_block (included by
// flash.hip, whose softmax and operand layouts they share): a workgroup's
// waves split the keys of its queries into groups and merge their sums in LDS.
//
// What bounds them: flash_block walks the keys with all its waves in step, at
// about 1 us (f16) or 4.3 us (f32) per 64 keys whether the GPU is full or not,
// and fills few CUs unless the keys are cut into many chunks whose partial
// results a second kernel merges.  With 4 or 8 key groups in the workgroup
// the chain per wave is 4 or 8 times shorter, and most launches need no
// second kernel.  What is left is 5 us of launch, first loads and merge, and
// per step 1.1-1.4 us (f16: dependent softmax chain, and with 32 queries per
// workgroup the K and V bytes, 60 KB/us per CU) or 2.1 us per 32 keys (f32:
// 1.7 of MFMA).
// Measured on MI355X (us, HIP events, one box, against the regular kernel in
// the chunks its rule takes): f16 one head of 4096^2 14.6 against 23.2, 16
// heads of 1000^2 10.5 against 20.4, 8 heads of 512^2 7.1 against 13.2; f32 4
// heads of 1000 x 4133 42.6 against 51.0, 16 heads of 200 x 300 11.3 against
// 20.2, one head of 1024^2 10.9 against 19.5.
#pragma once

#define FW_PITCH 68  // floats per query in the merge
// A key group's running max before its first block, and the least it takes
// there: finite, so that a block of -inf scores only weighs 0 and not
// exp2(-inf + inf).  M_INIT will not do: a group may start on a block whose
// scores all lie below it (keys a caller pads with a large negative value), and
// 2^(M_INIT - max) then overflows.
#define FW_M0 (-3.402823466e38f)

// Merges the key groups' sums of a workgroup of QW x KG waves (wave = grp * QW
// + query tile): O = sum_g 2^(m_g - M) acc_g / sum_g 2^(m_g - M) l_g.  The first
// half of the waves' accumulators go to st0 as [query][64], the others' to
// st1, m and l behind the first ones.
template <int QW, int KG, bool PART>
__device__ __forceinline__ void fw_merge(const phx_f16v (&acc)[2], float m2, float lh, T *O, int64_t ldo, uint32_t Nq, uint32_t q0,
                                          char *st0, char *st1, float *pacc, float *pml) {
    constexpr uint32_t NW = QW * KG, NQ = 32 * QW;
    constexpr uint32_t WB = 32 * FW_PITCH * 4;  // bytes of one wave's sums
    const uint32_t tid = threadIdx.x, lane = tid & 63, lq = lane & 31, g = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *const ml = (float *)(st0 + NW / 2 * WB);  // [wave][query of the wave]{m, l}
    const float lw = xor32_add(lh);
    {
        float *dst = (float *)((wave < NW / 2 ? st0 : st1) + wave % (NW / 2) * WB) + lq * FW_PITCH;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                *(phx_f4 *)(dst + 32 * dt + 8 * b + 4 * g) =
                    (phx_f4){acc[dt][4 * b], acc[dt][4 * b + 1], acc[dt][4 * b + 2],
                             acc[dt][4 * b + 3]};
        if (g == 0) *(float2 *)(ml + (wave * 32 + lq) * 2) = make_float2(m2, lw);
    }
    __syncthreads();
    constexpr uint32_t TPQ = 64 * NW / NQ, NV = 64 / TPQ / 4;  // threads per query, float4s each
    const uint32_t qt = tid / TPQ, d0 = (tid % TPQ) * (4 * NV), q = q0 + qt;
    const uint32_t ql = qt % 32, w0 = qt / 32;  // the query's place in waves w0, w0 + QW, ...
    // from the groups' own maxima: a group without a block carries FW_M0 and l = 0
    float mw[KG], M = FW_M0, l = 0.0f;
#pragma unroll
    for (int x = 0; x < KG; ++x) {
        mw[x] = ml[((w0 + x * QW) * 32 + ql) * 2];
        M = fmaxf(M, mw[x]);
    }
    phx_f4 o[NV];
#pragma unroll
    for (int x = 0; x < (int)NV; ++x) o[x] = (phx_f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int x = 0; x < KG; ++x) {
        const uint32_t w = w0 + x * QW;
        const float e = __builtin_amdgcn_exp2f(mw[x] - M);
        const float *src =
            (const float *)((w < NW / 2 ? st0 : st1) + w % (NW / 2) * WB) + ql * FW_PITCH + d0;
        l = l + e * ml[(w * 32 + ql) * 2 + 1];
#pragma unroll
        for (int y = 0; y < (int)NV; ++y) o[y] = o[y] + e * *(const phx_f4 *)(src + 4 * y);
    }
    if (q >= Nq) return;
    if (PART && d0 == 0) *(float2 *)(pml + 2 * (int64_t)q) = make_float2(M, l);
#pragma unroll
    for (int x = 0; x < (int)NV; ++x) {
        if (PART)
            *(phx_f4 *)(pacc + (int64_t)q * D + d0 + 4 * x) = o[x];
        else
#ifdef PHX_FLASH_F16
            *(phx_h4 *)(O + (int64_t)q * ldo + d0 + 4 * x) =
                (phx_h4){(_Float16)(o[x][0] / l), (_Float16)(o[x][1] / l), (_Float16)(o[x][2] / l),
                         (_Float16)(o[x][3] / l)};
#else
            *(phx_f4 *)(O + (int64_t)q * ldo + d0 + 4 * x) = o[x] / l;
#endif
    }
}

#define FLASH_W(NAME, FN, QW, KG, STB)                                                       \
    extern "C" __global__ __launch_bounds__(64 * QW * KG, 2) void NAME(                        \
        const T *Qb, const T *Kb, const T *Vb, T *Ob, float *W, int64_t BH, int64_t Nq,        \
        int64_t Nk, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int64_t hq,            \
        int64_t hk, int64_t hv, int64_t ho, int64_t kchunk, int32_t nsplit, float scale) {     \
        /* each stage its own array, so that the compiler's LDS-DMA tracking tells */          \
        /* the copies in flight from the stage being read */                                   \
        __shared__ __attribute__((aligned(16))) char st0[KG * STB], st1[KG * STB];             \
        static_assert(QW * KG / 2 * 32 * FW_PITCH * 4 + QW * KG * 32 * 8 <= KG * STB,         \
                      "the merge fits in the stages");                                         \
        const uint32_t nrb = (uint32_t)((Nq + 32 * QW - 1) / (32 * QW));                       \
        const int64_t k0 = (int64_t)blockIdx.y * kchunk;                                       \
        if (blockDim.x != 64 * QW * KG || blockIdx.x >= nrb * (uint32_t)BH || k0 >= Nk ||      \
            kchunk % BC)                                                                       \
            return;                                                                            \
        const uint32_t ws = phx_xcd_swizzle_any(blockIdx.x, gridDim.x);                        \
        const uint32_t h = ws / nrb, q0 = ws % nrb * (32 * QW);                                \
        const uint32_t nk = (uint32_t)(Nk - k0 < kchunk ? Nk - k0 : kchunk);                   \
        const T *Q = Qb + h * hq, *K = Kb + h * hk + k0 * ldk, *V = Vb + h * hv + k0 * ldv;    \
        if (nsplit > 1) {                                                                      \
            const int64_t plane = ((int64_t)blockIdx.y * BH + h) * Nq;                         \
            FN<KG, true>(Q, K, V, nullptr, ldq, ldk, ldv, 0, (uint32_t)Nq, nk, q0, scale, st0, \
                         st1, W + plane * D, W + (int64_t)nsplit * BH * Nq * D + plane * 2);   \
        } else {                                                                               \
            FN<KG, false>(Q, K, V, Ob + h * ho, ldq, ldk, ldv, ldo, (uint32_t)Nq, nk, q0,      \
                          scale, st0, st1, nullptr, nullptr);                                  \
        }                                                                                      \
    }
#ifdef PHX_FLASH_F16
#include "flash_w16.h"
#else
#include "flash_w32.h"
#endif
