// The f16 small-launch kernels.
//   flash_w4    32 queries, 4 waves, each its own key group: K goes straight
//               to the MFMA operands, V through the wave's own LDS ring (its
//               operand needs the transposing read), no barrier in the loop.
//   flash_w2x4  64 queries, 4 key groups of 2 waves that share K and V in LDS:
//               half the bytes per query, which is what bounds flash_w4 once
//               every CU has a workgroup (one head of 4096^2: 14.6 us in 4
//               chunks against 16.8 in 2).
// 8 key groups of one wave, and 64 queries per wave, measured slower than
// either (8 heads of 512^2 8.3 and 10.5 us against 7.1).
#pragma once

// K operands of one key block, straight from global memory: K row 32t + lq, d
// 16s + 8g .. +7.
struct KFrag {
    phx_h8 k[2][4];
};
__device__ __forceinline__ void w16_load_k(KFrag &f, const T *Kp, int64_t ldk, uint32_t Nk,
                                           uint32_t blk, uint32_t vo) {
    const __amdgpu_buffer_rsrc_t rk = kv_rsrc(Kp, ldk, Nk, blk);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            f.k[t][s] = __builtin_bit_cast(
                phx_h8, __builtin_amdgcn_raw_buffer_load_b128(
                            rk, (int)(vo + 32 * s), (int)((uint32_t)(32 * t * ldk) * 2), 0));
}
// V rows of key block blk into this wave's part of a stage.
__device__ __forceinline__ void w16_copy_v(char *dst, const T *Vp, int64_t ldv, uint32_t Nk,
                                           uint32_t blk, uint32_t vv) {
    const __amdgpu_buffer_rsrc_t rv = kv_rsrc(Vp, ldv, Nk, blk);
#pragma unroll
    for (int c = 0; c < 8; ++c)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (phx_lds_vp)(dst + c * 8 * KV_ROW), 16, vv,
                                                 (int)((uint32_t)(c * 8 * ldv) * 2), 0, 0);
}

// One key block of one wave: KG key groups (waves) per workgroup, this one's
// blocks are i, i + KG, ...; a partial block is masked.
template <int KG, bool FIRST>
__device__ __forceinline__ void w16_step(Flash16 &fs, KFrag &kf, char *Vs, const T *Kp,
                                         const T *Vp, int64_t ldk, int64_t ldv, uint32_t Nk,
                                         uint32_t i, float c2, uint32_t vk, uint32_t vv,
                                         uint32_t lane) {
    phx_f16v sc[2];
    const uint32_t kv = Nk - i * BC;
    if (kv < BC)
        key_bias(sc, kv, lane >> 5);
    else
        sc[0] = sc[1] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
            sc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf.k[t][s], fs.qf[s], sc[t], 0, 0, 0);
    w16_load_k(kf, Kp, ldk, Nk, i + 2 * KG, vk);  // into the operands just used
    phx_h8 pf[4];
    float ps = 0.0f;
    bool slow = FIRST;
    if (!FIRST) {
        ps = softmax_p(pf, sc, c2, fs.m2);
        slow = __ballot(!(ps <= FAST_SUM_LIMIT));  // wave-uniform; NaN too
    }
    if (slow) {
        const float mx = row_max(sc) * c2;  // log2 units
        const float m2n = FIRST                            ? fmaxf(mx, FW_M0)
                          : mx > fs.m2 + RESCALE_SLACK ? mx
                                                       : fs.m2;
        ps = softmax_p(pf, sc, c2, m2n);
        if (!FIRST) {
            const float corr = __builtin_amdgcn_exp2f(fs.m2 - m2n);  // 1 where not raised
            fs.l = fs.l * corr;
            fs.acc[0] = fs.acc[0] * corr;
            fs.acc[1] = fs.acc[1] * corr;
        }
        fs.m2 = m2n;
    }
    fs.l += ps;
    // V of block i landed.  Issued after it: K and V of the group's next block,
    // 16, and except in its last step (whose K loads nothing reads, so they
    // are not there) K of the block after that; with those in flight, the wait
    // for 16 is also one for the next block's K.
    __builtin_amdgcn_sched_barrier(0);
    PHX_WAIT_VMCNT(16);
    pv(fs.acc, Vs, pf, lane);
    w16_copy_v(Vs, Vp, ldv, Nk, i + 2 * KG, vv);  // into the stage just read
    __builtin_amdgcn_sched_barrier(0);            // the wait above counts on this order
}

template <int KG, bool PART>
__device__ __forceinline__ void w16_block(const T *Q, const T *Kp, const T *Vp, T *O, int64_t ldq,
                                          int64_t ldk, int64_t ldv, int64_t ldo, uint32_t Nq,
                                          uint32_t Nk, uint32_t q0, float scale, char *st0,
                                          char *st1, float *pacc, float *pml) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lq = lane & 31, g = lane >> 5;
    char *const S0 = st0 + wave * KV_TILE, *const S1 = st1 + wave * KV_TILE;
    const float c2 = softmax_c2(scale);
    const uint32_t nkb = (Nk + BC - 1) / BC;
    const uint32_t vk = (uint32_t)((lq * ldk + 8 * g) * 2);
    const uint32_t vv =
        (uint32_t)(((lane >> 3) * ldv + 8 * ((lane & 7) ^ (((lane >> 4) & 1) << 2))) * 2);

    Flash16 fs;
    const __amdgpu_buffer_rsrc_t rq = phx_rsrc(Q, (uint32_t)(((Nq - 1) * ldq + D) * 2));
#pragma unroll
    for (int s = 0; s < 4; ++s)
        fs.qf[s] = __builtin_bit_cast(
            phx_h8, __builtin_amdgcn_raw_buffer_load_b128(
                        rq, (int)(((q0 + lq) * ldq + 16 * s + 8 * g) * 2), 0, 0));
    // this wave's key blocks: wave, wave + KG, ...
    KFrag k0, k1;
    w16_load_k(k0, Kp, ldk, Nk, wave, vk);
    w16_copy_v(S0, Vp, ldv, Nk, wave, vv);
    __builtin_amdgcn_sched_barrier(0);
    w16_load_k(k1, Kp, ldk, Nk, wave + KG, vk);
    w16_copy_v(S1, Vp, ldv, Nk, wave + KG, vv);
    if (scale < 0.0f) {  // wave-uniform
#pragma unroll
        for (int s = 0; s < 4; ++s) fs.qf[s] = -fs.qf[s];
    }
    fs.acc[0] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    fs.acc[1] = fs.acc[0];
    fs.m2 = FW_M0;  // replaced by the first block's row max, if the group has one
    fs.l = 0.0f;
#define W16S(F, S, KF, I) w16_step<KG, F>(fs, KF, S, Kp, Vp, ldk, ldv, Nk, I, c2, vk, vv, lane)
    uint32_t i = wave;
    if (i < nkb) {
        W16S(true, S0, k0, i);
        i += KG;
        for (; i + KG < nkb; i += 2 * KG) {
            W16S(false, S1, k1, i);
            W16S(false, S0, k0, i + KG);
        }
        if (i < nkb) W16S(false, S1, k1, i);
    }
#undef W16S
    PHX_WAIT_VMCNT(0);
    __syncthreads();

    fw_merge<1, KG, PART>(fs.acc, fs.m2, fs.l, O, ldo, Nq, q0, st0, st1, pacc, pml);
}

// One key block of a group of two waves of 32 queries, K and V from LDS; the
// copies of the group's next block go out after the barrier that ends the
// last one's reads.
template <int KG, bool FIRST>
__device__ __forceinline__ void w2_step(Flash16 &fs, const char *cur, char *fill, const T *Kp,
                                        const T *Vp, int64_t ldk, int64_t ldv, uint32_t Nk,
                                        uint32_t i, float c2, const uint32_t (&vk)[2], uint32_t vv,
                                        uint32_t w2, uint32_t lane) {
    const uint32_t lq = lane & 31, g = lane >> 5;
    PHX_WAIT_VM_LGKM0(0);  // own copies of block i landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    {
        const __amdgpu_buffer_rsrc_t rk = kv_rsrc(Kp, ldk, Nk, i + KG);
        const __amdgpu_buffer_rsrc_t rv = kv_rsrc(Vp, ldv, Nk, i + KG);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t row = w2 * 32 + c * 8;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (phx_lds_vp)(fill + row * KV_ROW), 16,
                                                     vk[c & 1], (int)((uint32_t)(row * ldk) * 2), 0,
                                                     0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv,
                                                     (phx_lds_vp)(fill + KV_TILE + row * KV_ROW),
                                                     16, vv, (int)((uint32_t)(row * ldv) * 2), 0, 0);
        }
    }
    if (i * BC >= Nk) return;  // no block left for this group (uniform)
    phx_f16v sc[2];
    const uint32_t kv = Nk - i * BC;
    if (kv < BC) {
        key_bias(sc, kv, g);
        scores<true>(sc, cur, fs, lq, g);
    } else {
        scores(sc, cur, fs, lq, g);
    }
    phx_h8 pf[4];
    float ps = 0.0f;
    bool slow = FIRST;
    if (!FIRST) {
        ps = softmax_p(pf, sc, c2, fs.m2);
        slow = __ballot(!(ps <= FAST_SUM_LIMIT));  // wave-uniform; NaN too
    }
    if (slow) {
        const float mx = row_max(sc) * c2;  // log2 units
        const float m2n = FIRST                            ? fmaxf(mx, FW_M0)
                          : mx > fs.m2 + RESCALE_SLACK ? mx
                                                       : fs.m2;
        ps = softmax_p(pf, sc, c2, m2n);
        if (!FIRST) {
            const float corr = __builtin_amdgcn_exp2f(fs.m2 - m2n);  // 1 where not raised
            fs.l = fs.l * corr;
            fs.acc[0] = fs.acc[0] * corr;
            fs.acc[1] = fs.acc[1] * corr;
        }
        fs.m2 = m2n;
    }
    fs.l += ps;
    pv(fs.acc, cur + KV_TILE, pf, lane);
}

template <int KG, bool PART>
__device__ __forceinline__ void w2_block(const T *Q, const T *Kp, const T *Vp, T *O, int64_t ldq,
                                         int64_t ldk, int64_t ldv, int64_t ldo, uint32_t Nq,
                                         uint32_t Nk, uint32_t q0, float scale, char *st0,
                                         char *st1, float *pacc, float *pml) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t w2 = wave & 1, grp = wave >> 1;
    const uint32_t lq = lane & 31, g = lane >> 5;
    char *const S0 = st0 + grp * STAGE_BYTES, *const S1 = st1 + grp * STAGE_BYTES;
    const float c2 = softmax_c2(scale);
    const uint32_t nkb = (Nk + BC - 1) / BC;
    // copy c fills rows 8c + lane/8; the K swizzle (row >> 1) & 7 has the
    // parity of c in its top bit
    const uint32_t vk[2] = {
        (uint32_t)(((lane >> 3) * ldk + 8 * ((lane & 7) ^ ((lane >> 4) & 3))) * 2),
        (uint32_t)(((lane >> 3) * ldk + 8 * ((lane & 7) ^ (4 + ((lane >> 4) & 3)))) * 2)};
    const uint32_t vv =
        (uint32_t)(((lane >> 3) * ldv + 8 * ((lane & 7) ^ (((lane >> 4) & 1) << 2))) * 2);
    Flash16 fs;
    const __amdgpu_buffer_rsrc_t rq = phx_rsrc(Q, (uint32_t)(((Nq - 1) * ldq + D) * 2));
#pragma unroll
    for (int s = 0; s < 4; ++s)
        fs.qf[s] = __builtin_bit_cast(
            phx_h8, __builtin_amdgcn_raw_buffer_load_b128(
                        rq, (int)(((q0 + 32 * w2 + lq) * ldq + 16 * s + 8 * g) * 2), 0, 0));
    {
        const __amdgpu_buffer_rsrc_t rk = kv_rsrc(Kp, ldk, Nk, grp);
        const __amdgpu_buffer_rsrc_t rv = kv_rsrc(Vp, ldv, Nk, grp);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t row = w2 * 32 + c * 8;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (phx_lds_vp)(S0 + row * KV_ROW), 16,
                                                     vk[c & 1], (int)((uint32_t)(row * ldk) * 2), 0,
                                                     0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (phx_lds_vp)(S0 + KV_TILE + row * KV_ROW),
                                                     16, vv, (int)((uint32_t)(row * ldv) * 2), 0, 0);
        }
    }
    if (scale < 0.0f) {  // wave-uniform
#pragma unroll
        for (int s = 0; s < 4; ++s) fs.qf[s] = -fs.qf[s];
    }
    fs.acc[0] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    fs.acc[1] = fs.acc[0];
    fs.m2 = FW_M0;  // replaced by the first block's row max, if the group has one
    fs.l = 0.0f;
    // the groups take blocks grp, grp + KG, ... in step, so every wave meets
    // every barrier; a group past its last block skips the work
#define W2S(F, A, B, I) w2_step<KG, F>(fs, A, B, Kp, Vp, ldk, ldv, Nk, (I) + grp, c2, vk, vv, w2, lane)
    W2S(true, S0, S1, 0);
    uint32_t i = KG;
    for (; i + KG < nkb; i += 2 * KG) {
        W2S(false, S1, S0, i);
        W2S(false, S0, S1, i + KG);
    }
    if (i < nkb) W2S(false, S1, S0, i);
#undef W2S
    PHX_WAIT_VMCNT(0);
    __syncthreads();
    fw_merge<2, KG, PART>(fs.acc, fs.m2, fs.l, O, ldo, Nq, q0, st0, st1, pacc, pml);
}

FLASH_W(flash_w4, w16_block, 1, 4, KV_TILE)
FLASH_W(flash_w2x4, w2_block, 2, 4, STAGE_BYTES)
