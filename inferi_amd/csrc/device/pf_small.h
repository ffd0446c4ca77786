// Prefill GEMM for products with too few 256 x 256 tiles to fill the chip:
// 32 x 32, 64 x 64 and 128 x 128 tiles (m x n) of the same product
// (device/pf_gemm.h has the large form, the argument conventions and the
// epilogues), split by role as the large Q4_K form is.
//
// A workgroup has (BM / 32 MI) (BN / 32 NJ) MFMA waves, which read both
// operands from LDS and run the products, and four staging waves.  X comes in
// by direct global-to-LDS loads, two K steps ahead through three buffers,
// issued by a wave of its own (by the MFMA waves in the 128 x 128 form, where
// they are few per wave).  The staging waves only dequantize: each of their 256
// threads owns half of one weight row's 64-element run per K step, loads its
// GGUF bytes D steps ahead into registers (the loads are the compiler's, and
// nothing else is in these waves' load queue, so its own waits leave the
// later ones in flight) and stores the f16 values into the other of two
// buffers.  One barrier per step for all waves.  16 KB of X and of W per step
// in every form: 80 KB of LDS, two workgroups per CU.
//
// Why: a prompt of tens or hundreds of tokens leaves the 128 x 128 form that
// was here before (every wave loading, dequantizing and multiplying in turn,
// two barriers per 64-wide step, one step of loads ahead) with 8 to 200
// workgroups whose steps each cost a memory round trip.  The sum over K of an
// output stays one MFMA chain in k order, the same products in the same order
// as in every other form, so that results do not depend on the form; K can
// therefore not be split over workgroups, and a small product is bound by its
// chain (36 cycles per 16 of K: 17 us at K 14336 with nothing else) and, a
// little each, by its operand reads, the staged stores, X and the weights.
// Measured, us per product before and now: Q4_K, N 4096, K 14336, 61 tokens
// 300, 37 (196 TFLOP/s); N 28672, K 4096, 61 tokens 83, 39; Q6_K, N 3072, K
// 8192, 1021 tokens 304, 117; N 1024, K 3072, 1021 tokens 108, 24.  (The
// staging split over eight waves that take turns and operands read a step
// ahead, one workgroup per CU for their LDS: no faster, 36 and 44 us.)
#pragma once
#include "pf_gemm.h"

namespace ifr {

// The workgroup's tile: m fastest, so that neighbours share their weight
// rows, and a contiguous run of tiles for each XCD (workgroup b runs on XCD
// b % 8), so that those rows come from memory once and stay in one L2.
template <int BM, int BN>
IFR_DEV void pg_tile_small(const PfGemmArgs &a, uint32_t &m0, uint32_t &n0) {
    const uint32_t tm = a.tiles_m, tiles = tm * a.tiles_n, b = blockIdx.x;
    const uint32_t x = b & 7u, per = tiles >> 3, rem = tiles & 7u;
    const uint32_t t = x * per + min(x, rem) + (b >> 3);
    m0 = (t % tm) * BM;
    n0 = (t / tm) * BN;
}

// The products of sub-tile u are read and stored with chunk index c ^
// pg_sub_swz(u): the 16 lanes of a store's pass cover several sub-tiles (whose
// rows lie on the same banks), and this puts them on distinct ones.  The two
// parts of a row write chunks that differ in bit 1 (K-quants) or bit 2.
template <int FMT, int NS>
IFR_DEV uint32_t pg_sub_swz(uint32_t u) {
    constexpr bool KQ = FMT == Q4_K || FMT == Q5_K || FMT == Q6_K;
    if constexpr (NS == 1) return 0;
    else if constexpr (NS == 2) return KQ ? u << 2 : u << 1;
    else return KQ ? (u & 1u) | (u & 2u) << 1 : u;
}

// XW: a wave of its own for the X loads.  P: operand reads run P 16-wide
// groups ahead of the products.  D: steps of weight bytes ahead.
template <int FMT, int EPI, int BM, int BN, int BK, int MI, int NJ, int D, bool XW, int P>
__device__ __attribute__((always_inline)) void pf_gemm_small_body(const PfGemmArgs &a) {
    constexpr int NS = BK / 64;                          // 64-wide sub-tiles of a step
    constexpr int T = 4 * NS;                            // 16-wide groups of a step
    constexpr int WM = BM / (32 * MI), WN = BN / (32 * NJ);
    constexpr int NMW = WM * WN;                         // MFMA waves
    constexpr int XS = NS * BM * 64, WS = NS * BN * 64;  // halves per buffer
    constexpr int NXL = XS / 512 / (XW ? 1 : NMW);       // 1 KB direct loads per loading wave and step
    static_assert(BN * NS * 2 == 256, "one half run per staging thread");
    static_assert(XS / 512 % NMW == 0 && 2 * NXL < 64, "direct loads");
    __shared__ __attribute__((aligned(1024))) _Float16 xs[3 * XS];
    __shared__ __attribute__((aligned(1024))) _Float16 ws[2 * WS];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t K = a.K, nk = (K + BK - 1) / BK;
    uint32_t m0, n0;
    pg_tile_small<BM, BN>(a, m0, n0);

    if (wave < NMW + (XW ? 1 : 0)) {
        // direct load j of this wave: 8 rows (lane / 8) of one sub-tile; the
        // offset of this lane's 16 bytes from the tile's first row (32 bits:
        // the host splits a launch whose tiles' offsets would not fit)
        const bool loads = !XW || wave == NMW;
        const uint32_t c0 = XW ? 0 : wave * NXL;
        const uint64_t xa = (uint64_t)(const _Float16 *)a.x + (uint64_t)m0 * a.ldx * 2;
        const void *x = (const void *)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(xa >> 32)) << 32 |
                                       (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)xa));
        uint32_t xoff[NXL];
#pragma unroll
        for (int j = 0; j < NXL; j++) {
            const uint32_t row = 8 * ((c0 + (uint32_t)j) % (BM / 8)) + (lane >> 3);
            xoff[j] = 2 * (min(row, a.M - 1 - m0) * a.ldx + 8 * ((lane & 7u) ^ pg_swz_of(row)));
        }
        const uint32_t xbase = lds_addr(xs);
        // X of step s into buffer b (a sub-tile past K reads the last one;
        // its products are not run)
        auto load_x = [&](uint32_t s, uint32_t b) {
            const uint32_t dst = xbase + b * (2 * XS);
#pragma unroll
            for (int j = 0; j < NXL; j++) {
                const uint32_t c = c0 + (uint32_t)j, k = min(s * BK + 64 * (c / (BM / 8)), K - 64);
                lds_dma16(x, xoff[j] + 2 * k, __builtin_amdgcn_readfirstlane(dst + 1024 * c));
            }
        };
        if (loads) {
            load_x(0, 0);
            load_x(1, 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NXL) : "memory");
        }
        asm volatile("s_barrier" ::: "memory");
        if (XW && loads) {
            uint32_t b = 2; // (s + 2) % 3: the buffer read in step s - 1
            for (uint32_t s = 0; s < nk; s++) {
                load_x(s + 2, b);
                // X of step s + 1 has landed; this step's loads may stay in flight
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NXL) : "memory");
                b = b == 2 ? 0 : b + 1;
            }
            // the loads past the end land before the workgroup's LDS is
            // given up
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            return;
        }
        const uint32_t wm = 32 * MI * (wave % WM), wn = 32 * NJ * (wave / WM);
        const uint32_t li = lane & 31u, hi = lane >> 5;
        float16v acc[MI][NJ];
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;
        // 16-wide group q (sub-tile q / 4) of the step in xb, wb
        auto product = [&](const _Float16 *xb, const _Float16 *wb, uint32_t q) {
            half8v av[MI], bv[NJ];
            const uint32_t u = q >> 2, c = 2 * (q & 3u) + hi;
            const _Float16 *xu = xb + u * (BM * 64), *wu = wb + u * (BN * 64);
#pragma unroll
            for (int i = 0; i < MI; i++) av[i] = *(const half8v *)(xu + pg_swz(wm + 32 * i + li, c));
#pragma unroll
            for (int j = 0; j < NJ; j++) bv[j] = *(const half8v *)(wu + pg_swz(wn + 32 * j + li, c ^ pg_sub_swz<FMT, NS>(u)));
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i], bv[j], acc[i][j], 0, 0, 0);
        };
        auto end_step = [&]() {
            // this step's operands are read (and X of step s + 1 has landed,
            // this step's loads may stay in flight)
            if constexpr (XW) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NXL) : "memory");
        };
        // whole steps, then (K no multiple of BK) the rest, apart from them so
        // that the accumulators stay where they are
        const uint32_t nf = K / BK;
        uint32_t b = 0; // s % 3
        for (uint32_t s = 0; s < nf; s++) {
            if constexpr (!XW) load_x(s + 2, b == 0 ? 2 : b - 1);
            const _Float16 *xb = xs + b * XS, *wb = ws + (s & 1u) * WS;
#pragma unroll
            for (uint32_t q = 0; q < T; q++) product(xb, wb, q);
            // reads P groups ahead (0x100 LDS reads, 0x008 MFMAs)
            __builtin_amdgcn_sched_group_barrier(0x100, P * (MI + NJ), 0);
#pragma unroll
            for (int q = 0; q < T - P; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, MI + NJ, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, P * MI * NJ, 0);
            end_step();
            b = b == 2 ? 0 : b + 1;
        }
        if (nf < nk) {
            const uint32_t nq = (K - nf * BK) / 16;
            for (uint32_t q = 0; q < nq; q++) product(xs + b * XS, ws + (nf & 1u) * WS, q);
            end_step();
        }
        if constexpr (!XW) asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // as above
        if (EPI == PG_STORE && a.rope)
            pg_epilogue_rope<MI, NJ>(a, acc, lane, wm, wn, m0, n0);
        else
            pg_epilogue<EPI, MI, NJ>(a, acc, lane, wm, wn, m0, n0);
        return;
    }

    // staging: thread t owns part p of sub-tile u of tile row r
    const uint32_t t = tid - 64u * (NMW + (XW ? 1 : 0)), p = t & 1u, u = (t >> 1) % NS, r = t / (2 * NS);
    const uint32_t x = pg_sub_swz<FMT, NS>(u);
    const uint8_t *wrow = pg_wrow<EPI>(a, n0, r);
    _Float16 *const tile = ws + u * (BN * 64);
    auto kof = [&](uint32_t s) { return min(s * BK + 64 * u, K - 64); };
    PgRun<FMT> st[D];
    auto put = [&](PgRun<FMT> &w, uint32_t s) {
        w.pin();
        w.template store<0>(kof(s), p, tile + (s & 1u) * WS, r, x);
        w.template store<1>(kof(s), p, tile + (s & 1u) * WS, r, x);
    };
#pragma unroll
    for (int i = 0; i < D; i++) st[i].load(wrow, kof((uint32_t)i), p);
    put(st[0], 0);
    st[0].load(wrow, kof(D), p);
    lds_barrier();
    // step s: the weights of step s + 1 into the other buffer, and their
    // registers refilled with step s + 1 + D (steps past the end repeat the
    // last run, into a buffer nobody reads)
    uint32_t s = 0;
    for (; s + D <= nk; s += D) {
#pragma unroll
        for (int i = 0; i < D; i++) {
            put(st[(i + 1) % D], s + (uint32_t)i + 1);
            st[(i + 1) % D].load(wrow, kof(s + (uint32_t)i + 1 + D), p);
            lds_barrier();
        }
    }
#pragma unroll
    for (int i = 0; i < D - 1; i++) {
        if (s + (uint32_t)i >= nk) break;
        put(st[(i + 1) % D], s + (uint32_t)i + 1);
        lds_barrier();
    }
    // the last loads land here (vmcnt 0, said so that the compiler's own
    // count knows it: it would otherwise wait for them in the MFMA waves'
    // loop, which its control flow places behind this)
    __builtin_amdgcn_s_waitcnt(0x0F70);
}

// Steps of weight bytes a staging thread holds, as many as its registers
// take (the 128 x 128 form keeps to 128 registers for its two workgroups per
// CU).
template <int FMT>
constexpr int pg_small_ahead(int bm) {
    return FMT == F32 || bm == 128 ? 2 : 4;
}
template <int FMT, int EPI>
IFR_DEV void pf_gemm_t32_body(const PfGemmArgs &a) {
    pf_gemm_small_body<FMT, EPI, 32, 32, 256, 1, 1, pg_small_ahead<FMT>(32), true, 4>(a);
}
template <int FMT, int EPI>
IFR_DEV void pf_gemm_t64_body(const PfGemmArgs &a) {
    pf_gemm_small_body<FMT, EPI, 64, 64, 128, 1, 2, pg_small_ahead<FMT>(64), true, 3>(a);
}
template <int FMT, int EPI>
IFR_DEV void pf_gemm_t128_body(const PfGemmArgs &a) {
    pf_gemm_small_body<FMT, EPI, 128, 128, 64, 2, 2, pg_small_ahead<FMT>(128), false, 2>(a);
}
constexpr int PG_T32_THREADS = 6 * 64, PG_T64_THREADS = 7 * 64, PG_T128_THREADS = 8 * 64;

} // namespace ifr
