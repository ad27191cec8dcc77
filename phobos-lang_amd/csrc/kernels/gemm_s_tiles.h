// The small output tiles of the f32 GEMMs (included by gemm_s.hip, whose
// masking and arithmetic they share): 64 x 64, 64 x 32 and 32 x 32, for
// gemm_fp32 (with split-K forms) and the cluster step leaf.
//
// What bounds them: the f32 MFMA (64 cycles per 32 x 32 x 2), so a launch is
// as fast as its CUs are evenly loaded.  The earlier 64 x 64 x 16 tiling
// spent about 15 cycles more on every MFMA, each adding to the sum of the one
// before it (two accumulators in turn remove that, and halve the f32 error),
// and left CUs idle where its tiles are no multiple of 256: smaller tiles,
// whose four waves share a tile's K steps, split the same work finer.  A
// launch of more workgroups than fit at once (three per CU) clumped its last
// ones on the CUs that came free first (2048^3: 148 us); it now runs 768
// workgroups that walk the tiles (121 us).  The host picks the tile by the
// MFMA time of the fullest CU (s_tile_plan in phx_runtime.cpp).
// Measured on MI355X (us, HIP events, one box, against the earlier plan):
// 512^3 5.3 (32 x 32) against 12.4, 768^3 12.7 (32 x 32) against 17.3, 1024^3
// 18.7 (64 x 64) against 22.2, 1536^3 60.4 (32 x 32) against 76.2, 1200 x 2000
// x 1000 42.8 (64 x 32) against 52, 2048^3 121 (64 x 64) against 131; f32
// matrix peak 13.7 at 1024^3, 109 at 2048^3.
#pragma once

// A TM x TN output tile per workgroup of 4 waves: WR x WC MFMA tiles of 32 x
// 32, each of which KW = 4 / (WR WC) waves share, taking TK / KW of every K
// step.  TK / KW = 16 or 32: 2 or 4 k-groups of 8 per wave and step.  NA
// accumulators in turn: two, since an MFMA that adds to the one before it waits
// about 15 cycles more than its 64; four (gemm_s32a4) where the tile stands in
// for a split of many chunks, whose chains of sums are that short (400 x 96 x
// 376 against f64: 1.22e-7 in 12 chunks, 1.34e-7 with two, 1.06e-7 with four;
// 512^3 runs in 5.41 us with four, 5.33 with two).
template <int WR_, int WC_, int TK_, int NA_ = 2>
struct STile {
    static constexpr int NA = NA_;
    static constexpr int WR = WR_, WC = WC_, KW = 4 / (WR * WC), TK = TK_;
    static constexpr int TM = 32 * WR, TN = 32 * WC;
    static constexpr int AROW = TK * 4, BROW = TN * 4;      // LDS row bytes
    static constexpr int CPA = AROW / 16, CPB = BROW / 16;  // 16-byte chunks per row
    static constexpr int ABYTES = TM * AROW, BBYTES = TK * BROW;
    static constexpr int STAGE = ABYTES + BBYTES;
    static constexpr int AC = ABYTES / 4096, BC = BBYTES / 4096;  // copies per wave and step
    static constexpr int NG = TK / 8 / KW;                        // k-groups per wave and step
    static_assert(NG % 2 == 0, "the next step's group 0 lands in f[0]");
    static_assert(STAGE >= 8192, "two waves' sums fit in one stage");
    static_assert((CPA == 8 || CPA == 16) && (CPB == 8 || CPB == 16), "the swizzles below");
};

// LDS serves 256 bytes per clock.  A: the 16 rows of one ds_read_b128 group
// at one logical chunk land in 16 distinct slots.  B: the two k rows of an
// operand read are 4 apart and must fall in different halves of 256 bytes.
template <class T>
__device__ __forceinline__ uint32_t sa_off(uint32_t row, uint32_t chunk) {
    return row * T::AROW + ((chunk ^ (T::CPA == 16 ? row & 15 : (row >> 1) & 7)) << 4);
}
template <class T>
__device__ __forceinline__ uint32_t sb_off(uint32_t row, uint32_t chunk) {
    const uint32_t x = (row >> 2) & 1;
    return T::CPB == 16 ? row * T::BROW + ((chunk ^ (x << 3)) << 4)
                        : (row ^ x) * T::BROW + (chunk << 4);
}

// Operands of k-group q (k = 8q .. 8q+7), as in gemm_s.hip: MFMA s of lane
// group g uses k = 8q + 4g + s.
struct SFrags {
    phx_f4 a;
    float b[4];
};
template <class T>
__device__ __forceinline__ void s_read(SFrags &f, const char *stage, uint32_t q, uint32_t wm,
                                       uint32_t wn, uint32_t lane, int r) {
    const uint32_t lrow = lane & 31, g = lane >> 5;
    if (r == 0) {
        f.a = *(const phx_f4 *)(stage + sa_off<T>(wm + lrow, 2 * q + g));
    } else {
        const uint32_t col = wn + lrow;
        f.b[r - 1] = *(const float *)(stage + T::ABYTES +
                                      sb_off<T>(8 * q + 4 * g + r - 1, col >> 2) + 4 * (col & 3));
    }
}

// Tiles t0, t0 + tstride, ... of C = alpha*A@B + beta*C (C not read when beta
// == 0; the cluster step leaf passes beta = 1, which multiplies exactly).
template <class T>
__device__ __forceinline__ void s_body(const float *A, int64_t lda, const float *B, int64_t ldb,
                                       float *C, int64_t ldc, int64_t M, int64_t N, int64_t K,
                                       float alpha, float beta, uint32_t t0, uint32_t tstride) {
    // each stage its own array, so that the compiler's LDS-DMA tracking tells
    // the copies in flight from the stage being read
    __shared__ __attribute__((aligned(16))) char st0[T::STAGE], st1[T::STAGE], st2[T::STAGE];
    char *const S[3] = {st0, st1, st2};
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t sp = wave / T::KW, kw = wave % T::KW;  // MFMA tile, share of the K step
    const uint32_t wm = (sp / T::WC) * 32, wn = (sp % T::WC) * 32;
    const uint32_t tiles_n = (uint32_t)((N + T::TN - 1) / T::TN);
    const uint32_t tiles_m = (uint32_t)((M + T::TM - 1) / T::TM);
    const uint32_t ntiles = tiles_m * tiles_n;
    const uint32_t Ku = (uint32_t)K, nk = (Ku + T::TK - 1) / T::TK, kwl = Ku % T::TK;

    uint32_t va[T::AC], vt[T::AC], vb[T::BC];  // lane offsets; vt: the partial last step
#pragma unroll
    for (int i = 0; i < T::AC; ++i) {
        const uint32_t s = (wave * T::AC + i) * 64 + lane, row = s / T::CPA;
        const uint32_t lc = (sa_off<T>(row, s % T::CPA) - row * T::AROW) >> 4;
        va[i] = (row * (uint32_t)lda + lc * 4) * 4;
        vt[i] = kwl == 0 || lc * 4 < kwl ? va[i] : 0x80000000u;
    }
#pragma unroll
    for (int i = 0; i < T::BC; ++i) {
        const uint32_t s = (wave * T::BC + i) * 64 + lane;
        const uint32_t off = sb_off<T>(s / T::CPB, s % T::CPB);  // an involution of the slot
        vb[i] = (off / T::BROW * (uint32_t)ldb + (off % T::BROW) / 4) * 4;
    }

    for (uint32_t t = t0; t < ntiles; t += tstride) {
        // t % 8 is the block's XCD in every round when the stride keeps it
        const uint32_t ts =
            tstride == ntiles || tstride % 8 == 0 ? phx_xcd_swizzle_any(t, ntiles) : t;
        const uint32_t gsz = GROUP_M * tiles_n;
        const uint32_t g0 = (ts / gsz) * GROUP_M;
        const uint32_t gm = (tiles_m - g0) < GROUP_M ? (tiles_m - g0) : GROUP_M;
        const uint32_t m0 = (g0 + (ts % gsz) % gm) * T::TM, n0 = ((ts % gsz) / gm) * T::TN;
        const uint32_t ml = (uint32_t)M - m0, nl = (uint32_t)N - n0;
        const uint32_t mr = ml < T::TM ? ml : T::TM, nc = nl < T::TN ? nl : T::TN;

        // copy c of K step k into stage dst (steps past K: zeros, through an
        // empty resource, so every wait count stays a constant)
        auto copy = [&](uint32_t k, char *dst, int c) {
            const uint32_t k0 = k * T::TK, kl = Ku - k0;
            const uint32_t kx = kl < T::TK ? kl : T::TK, in = 0u - (uint32_t)(k0 < Ku);
            if (c < T::AC)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    phx_rsrc(A + (int64_t)m0 * lda + k0, (((mr - 1) * (uint32_t)lda + kx) * 4) & in),
                    (phx_lds_vp)(dst + (wave * T::AC + c) * 1024), 16,
                    k0 + T::TK <= Ku ? va[c] : vt[c], 0, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    phx_rsrc(B + (int64_t)k0 * ldb + n0, (((kx - 1) * (uint32_t)ldb + nc) * 4) & in),
                    (phx_lds_vp)(dst + T::ABYTES + (wave * T::BC + c - T::AC) * 1024), 16,
                    vb[c - T::AC], 0, 0, 0);
        };
        constexpr int DMA = T::AC + T::BC, NM = 4 * T::NG;
        phx_f16v acc[T::NA];
#pragma unroll
        for (int x = 0; x < T::NA; ++x)
            acc[x] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
#pragma unroll
            for (int c = 0; c < DMA; ++c) copy(p, S[p], c);
            __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
        }
        PHX_WAIT_VMCNT(DMA);
        __builtin_amdgcn_s_barrier();
        SFrags f[2];
#pragma unroll
        for (int r = 0; r < 5; ++r) s_read<T>(f[0], st0, kw * T::NG, wm, wn, lane, r);
        // One K step: each k-group's MFMAs run with the next group's operand
        // reads and an even share of the copies of step k + 2 between them;
        // before the last group the barrier that publishes step k + 1
        auto step = [&](uint32_t k, int u) {
#pragma unroll
            for (int g = 0; g < T::NG; ++g) {
                const bool last = g == T::NG - 1;
                if (last) {  // own copies of step k+1 landed; most of k+2's may be in flight
                    PHX_WAIT_VM_LGKM0(DMA * (T::NG - 1) / T::NG);
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int m = 4 * g + s;
                    phx_f16v &c = acc[s % T::NA];
                    c = __builtin_amdgcn_mfma_f32_32x32x2f32(f[g & 1].a[s], f[g & 1].b[s], c, 0, 0,
                                                             0);
#pragma unroll
                    for (int r = s * 5 / 4; r < (s + 1) * 5 / 4; ++r)
                        s_read<T>(f[(g + 1) & 1], last ? S[(u + 1) % 3] : S[u],
                                  kw * T::NG + (last ? 0 : g + 1), wm, wn, lane, r);
#pragma unroll
                    for (int c = m * DMA / NM; c < (m + 1) * DMA / NM; ++c)
                        copy(k + 2, S[(u + 2) % 3], c);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        uint32_t kt = 0;
        for (; kt + 3 <= nk; kt += 3) {
#pragma unroll
            for (int u = 0; u < 3; ++u) step(kt + u, u);
        }
        if (kt < nk) step(kt, 0);
        if (kt + 1 < nk) step(kt + 1, 1);
#pragma unroll
        for (int h = T::NA / 2; h > 0; h /= 2)  // pairwise
#pragma unroll
            for (int x = 0; x < h; ++x) acc[x] = acc[x] + acc[x + h];

        // Epilogue: the waves' sums to LDS as [wave][register][lane]; then the
        // KW waves of an MFMA tile take 32 / KW of its rows each, 8 lanes a
        // row, 4 columns a lane, adding the shares in order.
        const uint32_t pitch = (uint32_t)ldc * 4;
        const __amdgpu_buffer_rsrc_t rc = phx_rsrc(C + (int64_t)m0 * ldc, mr * pitch);
        const uint32_t col = n0 + wn + (lane & 7) * 4;
        const uint32_t voff = (wm + (lane >> 3)) * pitch +
                              (col < (uint32_t)N ? col * 4 : 0x80000000u);
        constexpr int NP = 4 / T::KW;
        phx_f4 old[NP];
        if (beta != 0.0f) {
#pragma unroll
            for (int x = 0; x < NP; ++x)
                old[x] = __builtin_bit_cast(
                    phx_f4, __builtin_amdgcn_raw_buffer_load_b128(
                                rc, (int)voff, (int)((kw * NP + x) * 8 * pitch), 0));
        }
        PHX_WAIT_VMCNT(0);
        __syncthreads();
        auto sums = [&](uint32_t w) { return (float *)(w & 2 ? st1 : st0) + (w & 1) * 1024; };
#pragma unroll
        for (int r = 0; r < 16; ++r) sums(wave)[r * 64 + lane] = acc[0][r];
        __syncthreads();
#pragma unroll
        for (int x = 0; x < NP; ++x) {
            const uint32_t row = (kw * NP + x) * 8 + (lane >> 3);
            // row's register and the lane of its first column (see MFMA layout)
            const uint32_t at = (4 * (row >> 3) + (row & 3)) * 64 + 32 * ((row >> 2) & 1) +
                                (lane & 7) * 4;
            phx_f4 v = *(const phx_f4 *)(sums(sp * T::KW) + at);
#pragma unroll
            for (int w = 1; w < T::KW; ++w)
                v = v + *(const phx_f4 *)(sums(sp * T::KW + w) + at);
            phx_f4 o = alpha * v;
            if (beta != 0.0f) o = o + beta * old[x];
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(phx_u4, o), rc, (int)voff,
                                                   (int)((kw * NP + x) * 8 * pitch), 0);
        }
        __syncthreads();
    }
}
