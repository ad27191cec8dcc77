// The smaller output tiles of the f16-operand GEMMs (included by gemm_h.hip,
// whose arithmetic, operand layouts and masking they share): gemm_m64 (64 x
// 64), gemm_m128x64 and gemm_m128 (128 x 128), and their split-K forms.
//
// What bounds them: with the 256 x 256 tile a launch below about 2300^2
// outputs leaves most CUs idle, or is cut over K and pays a second kernel
// and its partial planes.  A 64 x 64 tile gives 1024^2 outputs one workgroup
// per CU without a split; what a CU then takes is its operand bytes,
// (TM + TN) K, through a load path that delivers 66-85 KB/us to one CU
// whatever the tile or schedule (an all-L2-hit probe was only 5-10% faster,
// and one wave per SIMD, two, or a K slice per wave group all measured the
// same), so each K doubles at half the bytes with the next larger tile, until
// that tile leaves CUs idle.  The host picks the tile by that model
// (gemm_tile_plan in phx_runtime.cpp), for gemm_fp16tc among the tiles whose
// sums are no less exact than those of the split they replace.
// Measured on MI355X (us, HIP events, one box, against the 256 x 256 tile
// with its best split): gemm_fp16 512^3 4.8 (64 x 64) against 14.0, 1024^3
// 7.0 (64 x 64) against 22.8, 1280^3 10.6 (128 x 64) against 22.4, 2048^3
// 21.7 (128 x 128) against 36.3, 2560^3 44.3 (128 x 128) against 53.1;
// gemm_fp16tc_fp32acc 512^3 6.0 against 14.5, 1024^3 10.1 against 20.9,
// 2048^3 30.0 against 39.8.  At 3072^3 the 256 x 256 tile is the faster one
// (64.4 against 75.9).
//
// Design: 4 waves in a 2 x 2 arrangement; v_mfma_f32_32x32x16_f16; each k
// slice's MFMAs run with the next slice's operand reads and an even share of
// the step's operand moves between them, one barrier per K step, before its
// last slice, so the next step's first operands are read while the last
// slice multiplies.  gemm_fp16 copies global -> LDS into 4 stages, three
// steps ahead; gemm_fp16tc converts step k + 2 into a 3-stage ring from
// registers loaded one step before.  The k slices add into AS accumulator
// sets in turn, summed pairwise at the end: the f32 rounding of a short chain
// without a split (gemm_fp16tc at 1024^3, against f64: 1.0e-7 with four sets
// on the 64 x 64 tile, 1.8e-7 with one, 1.1e-7 for the 4-way split it
// replaces), within 3% of the time of one set.  gemm_fp16, whose result
// rounds to f16, keeps one set where registers are short.
#pragma once
#include <type_traits>

// A TM x TN output tile per workgroup, K steps of TK.
template <int TM_, int TN_, int TK_, int AS_, int OCC_>
struct MTile {
    static constexpr int TM = TM_, TN = TN_, TK = TK_;
    static constexpr int AS = AS_;    // accumulator sets: k slice s adds into set s % AS
    static constexpr int OCC = OCC_;  // waves per SIMD the registers must allow
    static constexpr int WMT = TM / 2, WNT = TN / 2;
    static constexpr int MI = WMT / 32, NJ = WNT / 32;
    static constexpr int AROW = TK * 2, BROW = TN * 2;
    static constexpr int CPA = AROW / 16, CPB = BROW / 16;  // 16-byte chunks per row
    static constexpr int ABYTES = TM * AROW, BBYTES = TK * BROW;
    static constexpr int STAGE = ABYTES + BBYTES;
    static constexpr int AC = ABYTES / 4096, BC = BBYTES / 4096;  // chunks per thread
    static constexpr int SL = TK / 16;                            // k slices per step
    static constexpr int EPP = WNT + 8;                           // epilogue pitch (floats)
    static_assert(SL % AS == 0 && (AS & (AS - 1)) == 0, "every step uses the sets alike");
    static_assert(SL % 2 == 0, "the next step's slice 0 lands in f[0]");
    static_assert(4 * 8 * EPP * 4 <= STAGE, "the epilogue's rows fit in one stage");
    static_assert((CPA == 4 || CPA == 8) && (CPB == 8 || CPB == 16), "the swizzles below");
};

// LDS serves 256 bytes per clock: the 16 rows one ds_read_b128 group reads
// at one logical chunk, and the 4 rows x 64 bytes of a transposing read's
// 32-lane group, land in distinct banks.
template <class T>
__device__ __forceinline__ uint32_t ma_off(uint32_t row, uint32_t chunk) {
    return row * T::AROW + ((chunk ^ (T::CPA == 8 ? (row >> 1) & 7 : (row >> 2) & 3)) << 4);
}
template <class T>
__device__ __forceinline__ uint32_t mb_off(uint32_t row, uint32_t chunk) {
    return row * T::BROW + ((chunk ^ (T::TN >= 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2)) << 4);
}

template <class T>
struct MFrags {
    phx_h8 a[T::MI];
    phx_h8 b[T::NJ];
};

// Operand read r of a slice: r < MI the A fragments, then the B fragments.
template <class T>
__device__ __forceinline__ void m_read(MFrags<T> &f, const char *stage, uint32_t s, uint32_t wm,
                                       uint32_t wn, uint32_t lane, int r) {
    if (r < T::MI) {
        f.a[r] = *(const phx_h8 *)(stage + ma_off<T>(wm + r * 32 + (lane & 31), 2 * s + (lane >> 5)));
        return;
    }
    const int j = r - T::MI;
    const char *Bs = stage + T::ABYTES;
    const uint32_t q = lane >> 4, sl = lane & 15;
    const uint32_t col = wn + j * 32 + 16 * (q & 1) + 4 * (sl & 3);
    phx_fp16x4 h[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t row = 16 * s + 8 * (q >> 1) + 4 * t + (sl >> 2);
        h[t] = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
            (phx_lds_h4p)((__attribute__((address_space(3))) char *)(
                Bs + mb_off<T>(row, col >> 3) + ((col & 7) << 1))));
    }
    const phx_h4 lo = __builtin_bit_cast(phx_h4, h[0]);
    const phx_h4 hi = __builtin_bit_cast(phx_h4, h[1]);
    f.b[j] = (phx_h8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// One K step: each slice's MFMAs run with the next slice's operand reads and
// an even share of the step's NC operand moves (move(c)) between them; sync()
// before the last slice, whose reads are of the next step's slice 0.  f[0]
// holds slice 0 on entry and the next step's on exit.
template <class T, int NC, class MV, class SY>
__device__ __forceinline__ void m_step(phx_f16v (&acc)[T::AS][T::MI][T::NJ], MFrags<T> (&f)[2],
                                       const char *cur, const char *nxt, uint32_t wm, uint32_t wn,
                                       uint32_t lane, MV move, SY sync) {
    constexpr int NM = T::MI * T::NJ, RD = T::MI + T::NJ;
#pragma unroll
    for (int s = 0; s < T::SL; ++s) {
        const bool last = s == T::SL - 1;
        if (last) {
            sync();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            phx_f16v &c = acc[s % T::AS][m / T::NJ][m % T::NJ];
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[s & 1].a[m / T::NJ], f[s & 1].b[m % T::NJ],
                                                       c, 0, 0, 0);
#pragma unroll
            for (int r = m * RD / NM; r < (m + 1) * RD / NM; ++r)
                m_read<T>(f[(s + 1) & 1], last ? nxt : cur, last ? 0 : s + 1, wm, wn, lane, r);
#pragma unroll
            for (int x = (s * NM + m) * NC / (T::SL * NM); x < (s * NM + m + 1) * NC / (T::SL * NM); ++x)
                move(x);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Buffer resources of one K step, as a_rsrc<true> and b_rsrc<true> above.
template <class T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ma_rsrc(const TIn *A, uint32_t lda, uint32_t M,
                                                          uint32_t K, uint32_t m0, uint32_t k0) {
    const uint32_t kl = K - k0, ml = M - m0;
    const uint32_t kw = kl < T::TK ? kl : T::TK, mr = ml < T::TM ? ml : T::TM;
    const uint32_t in = 0u - (uint32_t)(k0 < K);
    return phx_rsrc(A + (int64_t)m0 * lda + k0, ((mr - 1) * lda + kw) * (uint32_t)sizeof(TIn) & in);
}
template <class T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mb_rsrc(const TIn *B, uint32_t ldb, uint32_t N,
                                                          uint32_t K, uint32_t n0, uint32_t k0) {
    const uint32_t kl = K - k0, nl = N - n0;
    const uint32_t kw = kl < T::TK ? kl : T::TK, nc = nl < T::TN ? nl : T::TN;
    const uint32_t in = 0u - (uint32_t)(k0 < K);
    return phx_rsrc(B + (int64_t)k0 * ldb + n0, ((kw - 1) * ldb + nc) * (uint32_t)sizeof(TIn) & in);
}

template <class T, bool BETA, typename TO>
__device__ __forceinline__ void m_epilogue(const phx_f16v (&acc)[T::MI][T::NJ], float *ep_all,
                                           TO *C, int64_t ldc, int64_t M, int64_t N, uint32_t m0,
                                           uint32_t n0, uint32_t wm, uint32_t wn, float alpha,
                                           float beta, uint32_t wave, uint32_t lane) {
    const uint32_t lrow = lane & 31, lgrp = lane >> 5;
    float *ep = ep_all + wave * (8 * T::EPP);
    const uint32_t ml = (uint32_t)M - m0;
    const uint32_t rows = ml < T::TM ? ml : T::TM;
    const uint32_t pitch = (uint32_t)ldc * (uint32_t)sizeof(TO);
    const __amdgpu_buffer_rsrc_t rc = phx_rsrc(C + (int64_t)m0 * ldc, rows * pitch);
    constexpr int LPR = T::WNT / 4, RPI = 64 / LPR;  // lanes per row, rows per store
    const uint32_t c4 = (lane % LPR) * 4, er = lane / LPR;
    const uint32_t col = n0 + wn + c4;
    const uint32_t voff = (wm + er) * pitch +
                          (col < (uint32_t)N ? col * (uint32_t)sizeof(TO) : 0x80000000u);
    constexpr int NST = T::WMT / RPI;  // stores per lane
    // all of the old C is read up front, one latency for the whole tile
    typedef std::conditional_t<sizeof(TO) == 4, phx_f4, phx_h4> vec;
    vec old[BETA ? NST : 1];
    if constexpr (BETA) {
#pragma unroll
        for (int x = 0; x < NST; ++x) {
            const int so = (int)(x * RPI * pitch);
            if constexpr (sizeof(TO) == 4)
                old[x] = __builtin_bit_cast(
                    vec, __builtin_amdgcn_raw_buffer_load_b128(rc, (int)voff, so, 0));
            else
                old[x] = __builtin_bit_cast(
                    vec, __builtin_amdgcn_raw_buffer_load_b64(rc, (int)voff, so, 0));
        }
    }
#pragma unroll
    for (int p = 0; p < T::WMT / 8; ++p) {
        const int i = p / 4, r0 = (p % 4) * 4;
#pragma unroll
        for (int j = 0; j < T::NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                ep[(4 * lgrp + r) * T::EPP + 32 * j + lrow] = alpha * acc[i][j][r0 + r];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int rr = 0; rr < 8 / RPI; ++rr) {
            phx_f4 o = *(const phx_f4 *)(ep + (rr * RPI + er) * T::EPP + c4);
            const int x = p * (8 / RPI) + rr, so = (int)(x * RPI * pitch);
            if constexpr (BETA) {
                const vec c = old[x];
                o = o + beta * (phx_f4){(float)c[0], (float)c[1], (float)c[2], (float)c[3]};
            }
            if constexpr (sizeof(TO) == 4) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(phx_u4, o), rc,
                                                       (int)voff, so, 0);
            } else {
                const phx_h4 h = {(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]};
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(phx_u2, h), rc,
                                                      (int)voff, so, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

#ifdef PHX_GEMM_TC
template <class T>
struct MRegs {
    Chunk a[T::AC];
    Chunk b[T::BC];
};
#endif

template <class T, typename TO>
__device__ __forceinline__ void m_body(const TIn *A, const TIn *B, TO *C, uint32_t lda,
                                       uint32_t ldb, int64_t ldc, int64_t M, int64_t N, int64_t K,
                                       float alpha, float beta, uint32_t t0, uint32_t tstride) {
#ifdef PHX_GEMM_TC
    __shared__ __attribute__((aligned(16))) char lds[3 * T::STAGE];
    float *const EP = (float *)lds;
#else
    // each stage its own array, so that the compiler's LDS-DMA tracking tells
    // the copies in flight from the stage being read
    __shared__ __attribute__((aligned(16))) char st0[T::STAGE], st1[T::STAGE], st2[T::STAGE],
        st3[T::STAGE];
    char *const S[4] = {st0, st1, st2, st3};
    float *const EP = (float *)st0;
#endif
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = (wave >> 1) * T::WMT, wn = (wave & 1) * T::WNT;
    const uint32_t tiles_n = (uint32_t)((N + T::TN - 1) / T::TN);
    const uint32_t tiles_m = (uint32_t)((M + T::TM - 1) / T::TM);
    const uint32_t ntiles = tiles_m * tiles_n;
    const uint32_t Ku = (uint32_t)K, nk = (Ku + T::TK - 1) / T::TK;
    const uint32_t kwl = Ku % T::TK;  // columns of a partial last step, or 0

    for (uint32_t t = t0; t < ntiles; t += tstride) {
        const uint32_t ts = tstride == ntiles ? phx_xcd_swizzle_any(t, ntiles) : t;
        const uint32_t gsz = GROUP_M * tiles_n;
        const uint32_t g0 = (ts / gsz) * GROUP_M;
        const uint32_t gm = (tiles_m - g0) < GROUP_M ? (tiles_m - g0) : GROUP_M;
        const uint32_t m0 = (g0 + (ts % gsz) % gm) * T::TM, n0 = ((ts % gsz) / gm) * T::TN;
        phx_f16v acc[T::AS][T::MI][T::NJ];
#pragma unroll
        for (int x = 0; x < T::AS; ++x)
#pragma unroll
            for (int i = 0; i < T::MI; ++i)
#pragma unroll
                for (int j = 0; j < T::NJ; ++j)
                    acc[x][i][j] = (phx_f16v){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

#ifdef PHX_GEMM_TC
        const uint32_t kc = (tid % T::CPA) * 8;
        const uint32_t voa = ((tid / T::CPA) * lda + kc) * ESZ;
        const uint32_t voa_t = kwl == 0 || kc < kwl ? voa : 0x80000000u;
        const uint32_t vob = ((tid / T::CPB) * ldb + (tid % T::CPB) * 8) * ESZ;
        auto load_a = [&](Chunk &c, uint32_t k, int i) {
            const uint32_t k0 = k * T::TK;
            c = load_chunk(ma_rsrc<T>(A, lda, (uint32_t)M, Ku, m0, k0), k0 + T::TK <= Ku ? voa : voa_t,
                           (int)((uint32_t)(i * (NT / T::CPA) * lda) * ESZ));
        };
        auto load_b = [&](Chunk &c, uint32_t k, int i) {
            c = load_chunk(mb_rsrc<T>(B, ldb, (uint32_t)N, Ku, n0, k * T::TK), vob,
                           (int)((uint32_t)(i * (NT / T::CPB) * ldb) * ESZ));
        };
        auto store_a = [&](const Chunk &c, char *st, int i) {
            *(phx_u4 *)(st + ma_off<T>(i * (NT / T::CPA) + tid / T::CPA, tid % T::CPA)) = pack(c);
        };
        auto store_b = [&](const Chunk &c, char *st, int i) {
            *(phx_u4 *)(st + T::ABYTES +
                        mb_off<T>(i * (NT / T::CPB) + tid / T::CPB, tid % T::CPB)) = pack(c);
        };
        MRegs<T> R;
        {
            MRegs<T> P[2];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                MRegs<T> &d = p < 2 ? P[p] : R;
#pragma unroll
                for (int i = 0; i < T::AC; ++i) load_a(d.a[i], p, i);
#pragma unroll
                for (int i = 0; i < T::BC; ++i) load_b(d.b[i], p, i);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
#pragma unroll
                for (int i = 0; i < T::AC; ++i) store_a(P[p].a[i], lds + p * T::STAGE, i);
#pragma unroll
                for (int i = 0; i < T::BC; ++i) store_b(P[p].b[i], lds + p * T::STAGE, i);
            }
        }
        PHX_WAIT_VM_LGKM0(63);
        __builtin_amdgcn_s_barrier();
        MFrags<T> f[2];
#pragma unroll
        for (int r = 0; r < T::MI + T::NJ; ++r) m_read<T>(f[0], lds, 0, wm, wn, lane, r);
        // step k = u mod 3: its data in stage u, step k+1's in the next; step
        // k+2's is converted into the third, which every wave has left since
        // step k-1's barrier.  Whole rings, so that every stage's address is
        // an immediate (a rotating base cost the 128 x 128 tile 8%).
        auto step = [&](uint32_t k, int u) {
            char *const fill = lds + (u + 2) % 3 * T::STAGE;
            m_step<T, T::AC + T::BC>(
                acc, f, lds + u * T::STAGE, lds + (u + 1) % 3 * T::STAGE, wm, wn, lane,
                [&](int c) {
                    if (c < T::AC) {
                        store_a(R.a[c], fill, c);
                        load_a(R.a[c], k + 3, c);
                    } else {
                        store_b(R.b[c - T::AC], fill, c - T::AC);
                        load_b(R.b[c - T::AC], k + 3, c - T::AC);
                    }
                },
                [&] {
                    PHX_WAIT_VM_LGKM0(63);
                    __builtin_amdgcn_s_barrier();
                });
        };
        uint32_t kt = 0;
        for (; kt + 3 <= nk; kt += 3) {
#pragma unroll
            for (int u = 0; u < 3; ++u) step(kt + u, u);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (kt + u < nk) step(kt + u, u);
        PHX_WAIT_VMCNT(0);
        __syncthreads();
#else
        uint32_t va[T::AC], vt[T::AC], vb[T::BC];
#pragma unroll
        for (int i = 0; i < T::AC; ++i) {
            const uint32_t s = (wave * T::AC + i) * 64 + lane, row = s / T::CPA;
            const uint32_t lc = (ma_off<T>(row, s % T::CPA) - row * T::AROW) >> 4;
            va[i] = (row * lda + lc * 8) * 2;
            vt[i] = kwl == 0 || lc * 8 < kwl ? va[i] : 0x80000000u;
        }
#pragma unroll
        for (int i = 0; i < T::BC; ++i) {
            const uint32_t s = (wave * T::BC + i) * 64 + lane, row = s / T::CPB;
            const uint32_t lc = (mb_off<T>(row, s % T::CPB) - row * T::BROW) >> 4;
            vb[i] = (row * ldb + lc * 8) * 2;
        }
        // copy c of K step k into stage dst (steps past K: zeros, through an
        // empty resource, so every wait count stays a constant)
        auto copy = [&](uint32_t k, char *dst, int c) {
            const uint32_t k0 = k * T::TK;
            if (c < T::AC)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    ma_rsrc<T>(A, lda, (uint32_t)M, Ku, m0, k0),
                    (phx_lds_vp)(dst + (wave * T::AC + c) * 1024), 16,
                    k0 + T::TK <= Ku ? va[c] : vt[c], 0, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    mb_rsrc<T>(B, ldb, (uint32_t)N, Ku, n0, k0),
                    (phx_lds_vp)(dst + T::ABYTES + (wave * T::BC + c - T::AC) * 1024), 16,
                    vb[c - T::AC], 0, 0, 0);
        };
        constexpr int DMA = T::AC + T::BC;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int c = 0; c < DMA; ++c) copy(p, S[p], c);
            __builtin_amdgcn_sched_barrier(0);  // the waits count on this order
        }
        PHX_WAIT_VMCNT(2 * DMA);
        __builtin_amdgcn_s_barrier();
        MFrags<T> f[2];
#pragma unroll
        for (int r = 0; r < T::MI + T::NJ; ++r) m_read<T>(f[0], st0, 0, wm, wn, lane, r);
        auto step = [&](uint32_t k, int u) {
            m_step<T, DMA>(
                acc, f, S[u], S[(u + 1) & 3], wm, wn, lane,
                [&](int c) { copy(k + 3, S[(u + 3) & 3], c); },
                [&] {  // step k+1 landed; k+2's and most of k+3's copies may be in flight
                    PHX_WAIT_VM_LGKM0(DMA + DMA * (T::SL - 1) / T::SL);
                    __builtin_amdgcn_s_barrier();
                });
        };
        uint32_t kt = 0;
        for (; kt + 4 <= nk; kt += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) step(kt + u, u);
        }
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (kt + u < nk) step(kt + u, u);
        PHX_WAIT_VMCNT(0);
        __syncthreads();
#endif
#pragma unroll
        for (int h = T::AS / 2; h > 0; h /= 2)  // the sets' sums, pairwise
#pragma unroll
            for (int x = 0; x < h; ++x)
#pragma unroll
                for (int i = 0; i < T::MI; ++i)
#pragma unroll
                    for (int j = 0; j < T::NJ; ++j) acc[x][i][j] = acc[x][i][j] + acc[x + h][i][j];
        if (beta != 0.0f)
            m_epilogue<T, true, TO>(acc[0], EP, C, ldc, M, N, m0, n0, wm, wn, alpha, beta, wave, lane);
        else
            m_epilogue<T, false, TO>(acc[0], EP, C, ldc, M, N, m0, n0, wm, wn, alpha, beta, wave, lane);
        __syncthreads();
    }
}

#ifdef PHX_GEMM_TC
#define M_NMULT PHX_TC_N_MULT
#define M_KMULT PHX_TC_K_MULT
#else
#define M_NMULT PHX_H16_NK_MULT
#define M_KMULT PHX_H16_NK_MULT
#endif

#define GEMM_M(NAME, T)                                                                        \
    extern "C" __global__ __launch_bounds__(NT, T::OCC) void gemm_##NAME(                      \
        PHX_MEMREF2(TIn, a, int64_t), PHX_MEMREF2(TIn, b, int64_t),                            \
        PHX_MEMREF2(TOut, c, int64_t), float alpha, float beta) {                              \
        const int64_t M = a_s0, K = a_s1, N = b_s1;                                            \
        if (blockDim.x != NT || N % M_NMULT || K % M_KMULT || M <= 0 || N <= 0 || K <= 0 ||    \
            b_s0 != K || c_s0 != M || c_s1 != N || a_st1 != 1 || b_st1 != 1 || c_st1 != 1 ||   \
            a_st0 % M_KMULT || (b_st0 | c_st0) % M_NMULT || M > INT32_MAX || a_st0 < K ||      \
            b_st0 < N || c_st0 < N ||                                                          \
            (BM + 1) * (a_st0 > b_st0 ? a_st0 : b_st0) * (int64_t)sizeof(TIn) > INT32_MAX ||   \
            (BM + 1) * c_st0 * (int64_t)sizeof(TOut) > INT32_MAX ||                            \
            ((uintptr_t)(a_ptr + a_off) | (uintptr_t)(b_ptr + b_off) |                         \
             (uintptr_t)(c_ptr + c_off)) & 15)                                                 \
            return;                                                                            \
        m_body<T, TOut>(a_ptr + a_off, b_ptr + b_off, c_ptr + c_off, (uint32_t)a_st0,          \
                        (uint32_t)b_st0, c_st0, M, N, K, alpha, beta, phx_block_linear(),      \
                        phx_block_count());                                                    \
    }                                                                                          \
    extern "C" __global__ __launch_bounds__(NT, T::OCC) void gemm_##NAME##_splitk(             \
        const TIn *A, const TIn *B, float *W, int64_t lda, int64_t ldb, int64_t M, int64_t N,  \
        int64_t K, int64_t kchunk) {                                                           \
        const int64_t k0 = (int64_t)blockIdx.y * kchunk;                                       \
        if (blockDim.x != NT || k0 >= K || kchunk % BK) return;                                \
        const int64_t kc = K - k0 < kchunk ? K - k0 : kchunk;                                  \
        m_body<T, float>(A + k0, B + k0 * ldb, W + (int64_t)blockIdx.y * M * N, (uint32_t)lda, \
                         (uint32_t)ldb, N, M, N, kc, 1.0f, 0.0f, blockIdx.x, gridDim.x);  \
    }
