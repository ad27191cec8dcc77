// The f32 small-launch kernels (flash_w4, flash_w8: 32 queries, 4 or 8 key
// groups of one wave): every wave by itself, K and V straight from global
// memory into its MFMA operands (32 lanes of a V load are 32 consecutive d of
// one key), no LDS and no barrier in the loop.  The loads of the next step's
// K go out when its registers' last MFMA has, V's likewise, so each has the
// other product's 32 MFMAs to land in.
#pragma once

// One step of 32 keys, i*32 ..; a lane's score register r holds key 8(r/4) +
// 4g + r%4 of query lq.
struct W32 {
    phx_f16v acc[2];  // [d tile]: d = 32dt + 8(r/4) + 4g + r%4, query lq
    float m2, l;      // l: this lane's half of the keys
    phx_f4 qf[8];
    phx_f4 k[8];      // K row lq, d 8qq + 4g .. +3
    float v[4][2][4]; // V rows 8b + 4g + s, d 32dt + lq
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t w32_rsrc(const T *P, int64_t ld, uint32_t Nk,
                                                           uint32_t i) {
    const uint32_t in = 0u - (uint32_t)(i * 32 < Nk), r0 = (i * 32) & in;
    return phx_rsrc(P + (int64_t)r0 * ld, (uint32_t)(((Nk - 1 - r0) * ld + D) * 4) & in);
}
__device__ __forceinline__ void w32_load_k(W32 &w, const T *Kp, int64_t ldk, uint32_t Nk,
                                           uint32_t i, uint32_t vk) {
    const __amdgpu_buffer_rsrc_t rk = w32_rsrc(Kp, ldk, Nk, i);
#pragma unroll
    for (int qq = 0; qq < 8; ++qq)
        w.k[qq] = __builtin_bit_cast(
            phx_f4, __builtin_amdgcn_raw_buffer_load_b128(rk, (int)(vk + 32 * qq), 0, 0));
}
__device__ __forceinline__ void w32_load_v(W32 &w, const T *Vp, int64_t ldv, uint32_t Nk,
                                           uint32_t i, uint32_t vv) {
    const __amdgpu_buffer_rsrc_t rv = w32_rsrc(Vp, ldv, Nk, i);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
                w.v[b][dt][s] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               rv, (int)(vv + 128 * dt), (int)((uint32_t)((8 * b + s) * ldv) * 4), 0));
}

template <int KG>
__device__ __forceinline__ void w32_step(W32 &w, const T *Kp, const T *Vp, int64_t ldk, int64_t ldv,
                                         uint32_t Nk, uint32_t i, bool first, float c2, uint32_t vk,
                                         uint32_t vv, uint32_t g) {
    // two chains, over the even and the odd d groups: an MFMA that adds to
    // the one before it waits about 15 cycles more than its 64
    phx_f16v sc[2];
    sc[0] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    sc[1] = sc[0];
#pragma unroll
    for (int qq = 0; qq < 8; qq += 2)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int x = 0; x < 2; ++x)
                sc[x] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.k[qq + x][s], w.qf[qq + x][s], sc[x],
                                                             0, 0, 0);
    w32_load_k(w, Kp, ldk, Nk, i + KG, vk);
    phx_f16v p = sc[0] + sc[1];
    const uint32_t kv = Nk - i * 32;
    if (kv < 32) {  // partial last step (uniform)
        int32_t lim = (int32_t)kv - 4 * (int32_t)g;
        asm volatile("" : "+v"(lim));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float x = p[r];
            p[r] = 8 * (r >> 2) + (r & 3) < lim ? x : -__builtin_inff();
        }
    }
    float mx = p[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, p[r]);
    mx = xor32_max(mx) * c2;
    const bool raise = first || mx > w.m2 + RESCALE_SLACK;
    const float m2n = raise ? fmaxf(mx, FW_M0) : w.m2;
    float part[4];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(p[r], c2, -m2n));
        part[r & 3] = r < 4 ? e : part[r & 3] + e;
        p[r] = e;
    }
    if (__ballot(raise)) {  // wave-uniform
        const float corr = __builtin_amdgcn_exp2f(w.m2 - m2n);  // 1 where not raised
        w.l = w.l * corr;
        w.acc[0] = w.acc[0] * corr;
        w.acc[1] = w.acc[1] * corr;
    }
    w.l += (part[0] + part[1]) + (part[2] + part[3]);
    w.m2 = m2n;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
                w.acc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.v[b][dt][s], p[4 * b + s],
                                                                 w.acc[dt], 0, 0, 0);
    w32_load_v(w, Vp, ldv, Nk, i + KG, vv);
}

template <int KG, bool PART>
__device__ __forceinline__ void w32_block(const T *Q, const T *Kp, const T *Vp, T *O, int64_t ldq,
                                          int64_t ldk, int64_t ldv, int64_t ldo, uint32_t Nq,
                                          uint32_t Nk, uint32_t q0, float scale, char *st0,
                                          char *st1, float *pacc, float *pml) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lq = lane & 31, g = lane >> 5;
    const float c2 = softmax_c2(scale);
    const uint32_t n32 = (Nk + 31) / 32;
    const uint32_t vk = (uint32_t)((lq * ldk + 4 * g) * 4), vv = (uint32_t)((4 * g * ldv + lq) * 4);
    W32 w;
    const __amdgpu_buffer_rsrc_t rq = phx_rsrc(Q, (uint32_t)(((Nq - 1) * ldq + D) * 4));
    const float qsign = scale < 0.0f ? -1.0f : 1.0f;  // exact
    w32_load_k(w, Kp, ldk, Nk, wave, vk);
#pragma unroll
    for (int qq = 0; qq < 8; ++qq)
        w.qf[qq] = qsign * __builtin_bit_cast(
                               phx_f4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rq, (int)(((q0 + lq) * ldq + 8 * qq + 4 * g) * 4), 0, 0));
    w32_load_v(w, Vp, ldv, Nk, wave, vv);
    w.acc[0] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    w.acc[1] = w.acc[0];
    w.m2 = FW_M0;
    w.l = 0.0f;
    // this wave's steps: wave, wave + KG, ...
    for (uint32_t i = wave; i < n32; i += KG)
        w32_step<KG>(w, Kp, Vp, ldk, ldv, Nk, i, i == wave, c2, vk, vv, g);
    fw_merge<1, KG, PART>(w.acc, w.m2, w.l, O, ldo, Nq, q0, st0, st1, pacc, pml);
}

FLASH_W(flash_w4, w32_block, 1, 4, 5120)
FLASH_W(flash_w8, w32_block, 1, 8, 5120)
