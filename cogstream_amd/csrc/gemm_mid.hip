// Mid-size GEMM (bf16):  C[M,N] = epilogue( A[M,K] . W[N,K]^T ), same sums in the same order as the kernels of gemm.hip.
//
// For products whose 256-wide tiles would leave most of the chip idle. One tile per workgroup, tiles from 32x64 to 128x256; the
// K slabs (64 elements: one whole 128-byte line a row) go by LDS-DMA into a ring of S slots, S - 1 of them in flight ahead of the
// slab being multiplied, one barrier and one counted vmcnt per slab. A slab's second half is read while the first half is multiplied,
// the next slab's first half while the second is, so that LDS latency hides behind the wave's own matrix instructions; the small
// tiles leave room for two workgroups per CU, which hide each other's barriers.
//
// What bounds it: a CU takes in about 60 bytes a nanosecond of operand lines that miss its XCD's L2, whatever the tile, the ring
// depth or the row stride (16 KiB slab 0.26 us, 32 KiB 0.53, 48 KiB 0.82), so a launch costs rounds x (TM + TN) x K x 2 / 60 ns and a
// few us around it: the choice of a tile (gemm.hip) trades bytes per CU against CUs that have none. Products split over K would
// need fewer bytes, and give other bits. Measured against the 128x128 / 256x128 tiles that were here before, one slab ahead or with
// 256 rows per workgroup (weights from HBM): 256 x 1152 x 4352 80 -> 18 us, 256 x 3456 x 1152 24 -> 8.3, 1024 x 1152 x 4352 64 -> 31,
// 621 x 3584 x 18944 250 -> 157, 160 x 3584 x 18944 306 -> 75, 400 x 2048 x 8192 127 -> 30, 4096 x 2048 x 5632 105 -> 83.
//
// K is walked in order by one accumulator per output: a row's bits do not depend on which tile size, or which kernel of gemm.hip,
// computed it (frame ranges, prompts behind a kept prefix and whole prompts are compared bit for bit).
#include "common.h"
#include "kernels.h"
#include "gemm_epilogue.h"
#include "debug.h"

namespace {

struct MidArgs {
    const char* A; long lda;   // bytes per row
    const char* W; long ldw;
    int M, N, KT;              // KT: 64-wide K slabs
    int nbm, nbn;
    const float* ln_part; int ln_tiles; float ln_inv_h, ln_eps;     // EPI_LNFOLD: row statistics still in partial sums (or null)
    EpiArgs epi;
};

constexpr int ROW_BYTES = 128;

__device__ __forceinline__ void glds16(const char* g, char* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

// at most n slabs' pieces (P each) of this wave may stay in flight, n <= MAX
template <int P, int MAX>
__device__ __forceinline__ void wait_slabs(int n) {
    static_assert(MAX <= 6 && MAX * P < 64, "vmcnt is a 6-bit immediate");
    if (n <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (n == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P) : "memory");
    else if (n == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 2 ? 2 * P : 0) : "memory");
    else if (n == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 3 ? 3 * P : 0) : "memory");
    else if (n == 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 4 ? 4 * P : 0) : "memory");
    else if (n == 5) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 5 ? 5 * P : 0) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 6 ? 6 * P : 0) : "memory");
}

// WM x WN waves of 16 MI x 16 NI outputs, S ring slots
template <int EPI, int MI, int NI, int WM, int WN, int S, int WPE>
__global__ __launch_bounds__(64 * WM * WN, WPE) void gemm_mid_kernel(MidArgs p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int TM = 16 * MI * WM, TN = 16 * NI * WN, WAVES = WM * WN;
    constexpr int SLAB = (TM + TN) * ROW_BYTES, P = SLAB / 1024 / WAVES;
    static_assert(SLAB % (1024 * WAVES) == 0, "every wave stages the same number of pieces");
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid / WN, wn = wid % WN;
    const int KT = p.KT;

    // block -> tile: XCD-aware, then groups of 8 row tiles with the rows running fastest, so that the row tiles that share a
    // panel of weights run on one XCD
    int m0, n0;
    {
        const int nb = p.nbm * p.nbn, xcd = blockIdx.x & 7, q = nb >> 3, r = nb & 7;
        const int bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (blockIdx.x >> 3);
        const int per_group = 8 * p.nbn, first_m = bid / per_group * 8, gsz = min(p.nbm - first_m, 8);
        m0 = (first_m + (bid % per_group) % gsz) * TM;
        n0 = ((bid % per_group) / gsz) * TN;
    }
    // piece pc of a slab: tile rows 8 pc .. +7 (A's rows, then W's); lane -> row + (lane >> 3), 16-byte chunk lane & 7, swizzled
    const char* src[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int r = (wid * P + i) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ (r & 7);
        src[i] = r < TM ? p.A + (long)min(m0 + r, p.M - 1) * p.lda + c * 16 : p.W + (long)min(n0 + r - TM, p.N - 1) * p.ldw + c * 16;
    }
    char* const lds_wave = smem + wid * P * 1024;
    auto stage = [&](int slot) {                 // the next slab of the stream
        char* dst = lds_wave + slot * SLAB;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            glds16(src[i], dst + i * 1024);
            src[i] += ROW_BYTES;
        }
    };
    int foff[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) foff[s] = (lane & 15) * ROW_BYTES + ((((s << 2) + (lane >> 4)) ^ (lane & 7)) << 4);
    const int a_off = wm * 16 * MI * ROW_BYTES, w_off = (TM + wn * 16 * NI) * ROW_BYTES;

    f32x4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Frags { u32x4 a[2][MI], w[2][NI]; } f0, f1;       // the halves of a slab
    auto load_frags = [&](Frags& f, int slot) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const char* As = smem + slot * SLAB + a_off + foff[s];
            const char* Ws = smem + slot * SLAB + w_off + foff[s];
#pragma unroll
            for (int i = 0; i < MI; ++i) f.a[s][i] = *reinterpret_cast<const u32x4*>(As + i * 16 * ROW_BYTES);
#pragma unroll
            for (int i = 0; i < NI; ++i) f.w[s][i] = *reinterpret_cast<const u32x4*>(Ws + i * 16 * ROW_BYTES);
        }
    };
    auto mma = [&](Frags& f) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.w[s][ni]),
                                                                          __builtin_bit_cast(bf16x8, f.a[s][mi]), acc[mi][ni], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };
    // the wait for the fragments stands here, in front of newer LDS reads
    auto touch = [&](Frags& f) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < MI; ++i) asm volatile("" : "+v"(f.a[s][i]));
#pragma unroll
            for (int i = 0; i < NI; ++i) asm volatile("" : "+v"(f.w[s][i]));
        }
    };

    // what the epilogue reads, in front of the product where the registers are there to hold it (NI = 4 has none to spare):
    // M = 256 of the vision encoder, N x K = 1152 x 4304 / 1152 with residual 13.5 -> 13.0 us, 4304 x 1152 14.6 -> 14.2; M = 1024
    // 28.1 -> 27.0
    const int mb = m0 + wm * 16 * MI, nb = n0 + wn * 16 * NI;
    constexpr bool EARLY = NI == 2 && (EPI & EPI_GENERIC) == 0;
    EpiOperands<bf16_t, EPI, MI, NI> early;
    if constexpr (EARLY) early.load(p.epi, mb, nb, p.M, p.N, lane);
    for (int i = 0; i < S && i < KT; ++i) stage(i);
    // EPI_LNFOLD: the factors of this wave's rows while the ring fills; lane l has row l of its 16 MI
    float factor = 0.f;
    if constexpr ((EPI & EPI_LNFOLD) != 0) {
        const long r = min(m0 + wm * 16 * MI + (lane & (16 * MI - 1)), p.M - 1);
        factor = p.ln_part ? ln_row_factors(reinterpret_cast<const f32x2*>(p.ln_part) + r * p.ln_tiles, p.ln_tiles, p.ln_inv_h, p.ln_eps)[0]
                           : p.epi.ln_ab[2 * r];
    }
    wait_slabs<P, S - 1>(min(S, KT) - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_frags(f0, 0);
    int slot = 0, kt = 0;
    // slab kt is in the fragments `cur`: once every wave has it there, its slot takes slab kt + S, and slab kt + 1 is read into the
    // other set while this one is multiplied
    auto steady = [&](Frags& cur, Frags& nxt) {
        const int next = slot == S - 1 ? 0 : slot + 1;
        touch(cur);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * P) : "memory");       // slab kt + 1 has landed
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        stage(slot);
        load_frags(nxt, next);
        mma(cur);
        slot = next;
    };
    for (; kt + 1 + S < KT; kt += 2) {
        steady(f0, f1);
        steady(f1, f0);
    }
    auto tail = [&](Frags& cur, Frags& nxt) {
        const int next = slot == S - 1 ? 0 : slot + 1;
        touch(cur);
        if (kt + 1 < KT) {
            wait_slabs<P, S - 1>(min(S - 2, KT - kt - 2));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (kt + S < KT) stage(slot);
            load_frags(nxt, next);
        }
        mma(cur);
        slot = next;
        ++kt;
    };
    while (kt < KT) {
        tail(f0, f1);
        if (kt < KT) tail(f1, f0);
    }

    const auto* operands = EARLY ? &early : nullptr;
    if constexpr ((EPI & EPI_LNFOLD) != 0) {
        float rs[MI];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) rs[mi] = __shfl(factor, 16 * mi + (lane & 15));
        epilogue_tile<bf16_t, EPI, MI, NI>(p.epi, mb, nb, p.M, p.N, lane, acc, nullptr, rs, operands);
    } else if constexpr (MI == 4 && NI == 4) {
        epilogue_wave<bf16_t, EPI>(p.epi, mb, nb, p.M, p.N, lane, acc);
    } else if constexpr ((EPI & EPI_ROWSTAT) != 0 && NI == 2) {
        // a 64-column block's sums come from two waves; the pair is added lane by lane in the order of one 64-column wave, then
        // over the lanes, so the statistics have the same bits
        f32x2 st[MI];
        epilogue_tile<bf16_t, EPI, MI, NI>(p.epi, mb, nb, p.M, p.N, lane, acc, st, nullptr, operands);
        __syncthreads();                         // the ring is free
        f32x2* xch = reinterpret_cast<f32x2*>(smem) + (wid & ~1) * MI * 64 + lane;
        static_assert(WN % 2 == 0, "the two halves of a 64-column block are neighbouring waves");
        if (wn & 1) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) xch[mi * 64] = st[mi];
        }
        __syncthreads();
        if ((wn & 1) == 0 && nb < p.N) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
                const f32x2 o = xch[mi * 64];
                const float s1 = rowgroup_sum(st[mi][0] + o[0]), s2 = rowgroup_sum(st[mi][1] + o[1]);
                const int m = mb + 16 * mi + (lane & 15);
                if ((lane >> 4) == 0 && m < p.M)
                    *reinterpret_cast<f32x2*>(p.epi.stat_part + ((long)m * p.epi.stat_tiles + (nb >> 6)) * 2) = f32x2{s1, s2};
            }
        }
    } else {
        epilogue_tile<bf16_t, EPI, MI, NI>(p.epi, mb, nb, p.M, p.N, lane, acc, nullptr, nullptr, operands);
    }
}

template <int EPI, int MI, int NI, int WM, int WN, int S, int WPE>
void launch(hipStream_t st, MidArgs& p) {
    constexpr int TM = 16 * MI * WM, TN = 16 * NI * WN, lds = S * (TM + TN) * ROW_BYTES;
    static std::atomic<uint64_t> attr_done{0};
    cogs_ensure_dyn_lds((const void*)gemm_mid_kernel<EPI, MI, NI, WM, WN, S, WPE>, lds, attr_done);
    p.nbm = (p.M + TM - 1) / TM;
    p.nbn = (p.N + TN - 1) / TN;
    hipLaunchKernelGGL((gemm_mid_kernel<EPI, MI, NI, WM, WN, S, WPE>), dim3(p.nbm * p.nbn), dim3(64 * WM * WN), lds, st, p);
}

template <int EPI>
void dispatch_tile(hipStream_t st, MidArgs& p, int tile) {
    switch (tile) {
        case 1: launch<EPI, 2, 2, 1, 2, 6, 1>(st, p); break;          // 32 x 64
        case 2: launch<EPI, 2, 2, 2, 2, 5, 2>(st, p); break;          // 64 x 64
        case 3: launch<EPI, 2, 2, 4, 2, 3, 4>(st, p); break;          // 128 x 64
        case 4: launch<EPI, 4, 2, 2, 4, 5, 2>(st, p); break;          // 128 x 128
        default: launch<EPI, 4, 4, 2, 4, 3, 2>(st, p); break;         // 128 x 256
    }
}

}  // namespace

int cogs_k_gemm_mid(hipStream_t st, const CogsGemm& g, int tile) {
    MidArgs p;
    const int rc = cogs_fill_epi(g, &p.epi);
    if (rc != COGS_OK) return rc;
    p.A = (const char*)g.A; p.lda = g.lda * 2;
    p.W = (const char*)g.W; p.ldw = g.ldw * 2;
    p.M = g.M; p.N = g.N; p.KT = g.K / 64;
    p.ln_part = g.ln_part; p.ln_tiles = g.K / 64; p.ln_inv_h = 1.0f / (float)g.K; p.ln_eps = g.ln_eps;
#define COGS_MID_CASE(E) case E: dispatch_tile<E>(st, p, tile); break;
    switch (cogs_epi_mask(g)) {
        COGS_MID_CASE(0)
        COGS_MID_CASE(EPI_BIAS)
        COGS_MID_CASE(EPI_RES)
        COGS_MID_CASE(EPI_BIAS | EPI_RES)
        COGS_MID_CASE(EPI_BIAS | EPI_ROPE)
        COGS_MID_CASE(EPI_BIAS | EPI_GELU_TANH)
        COGS_MID_CASE(EPI_BIAS | EPI_GELU_ERF)
        COGS_MID_CASE(EPI_BIAS | EPI_ROWSTAT)
        COGS_MID_CASE(EPI_BIAS | EPI_RES | EPI_ROWSTAT)
        COGS_MID_CASE(EPI_BIAS | EPI_LNFOLD)
        COGS_MID_CASE(EPI_BIAS | EPI_ROPE | EPI_LNFOLD)
        COGS_MID_CASE(EPI_BIAS | EPI_GELU_TANH | EPI_LNFOLD)
        COGS_MID_CASE(EPI_BIAS | EPI_ROPE | EPI_HM)
        COGS_MID_CASE(EPI_BIAS | EPI_ROPE | EPI_LNFOLD | EPI_HM)
        COGS_MID_CASE(EPI_ROPE)
        COGS_MID_CASE(EPI_SWIGLU)
        COGS_MID_CASE(EPI_SWIGLU | EPI_BIAS)
        COGS_MID_CASE(EPI_GELU_ERF)
        COGS_MID_CASE(EPI_F32OUT)
        default: dispatch_tile<EPI_GENERIC>(st, p, tile); break;
    }
#undef COGS_MID_CASE
    return COGS_LAUNCH_CHECK();
}
