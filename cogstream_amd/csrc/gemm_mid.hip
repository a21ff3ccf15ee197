// Mid-size GEMM (bf16):  C[M,N] = epilogue( A[M,K] . W[N,K]^T ), same sums in the same order as the kernels of gemm.hip.
//
// For products whose 256-wide tiles would leave most of the chip idle, and for what whole rounds of those leave of a product (rows0, cols0).
// One tile per workgroup, tiles from 32x64 to 160x256, which size by what the chip makes of their number (gemm.hip); the
// K slabs (64 elements: one whole 128-byte line a row; KS of them at a time) go by LDS-DMA into a ring of S slots, S - 1 of them in
// flight ahead of the slabs being multiplied, one barrier and one counted vmcnt per KS slabs. While a slab is multiplied, the next
// one's fragments are read and its slot is filled again.
//
// What bounds it, and what each part is there for (us per launch, weights from HBM, 27 of them in turn; before -> after):
//   * A CU has about 60 KB of missing lines under way whatever the ring's depth, so weights that come from HBM arrive at 55 to 60 B/ns
//     a CU, and at 105 to 115 B/ns from its XCD's L2. Where CUs are left over, workgroups behind the tiles' (prefetch_weights) ask
//     for one dword of every weight line of their XCD's tiles, far ahead of the ring, on CUs whose own misses are free:
//     256 x 1152 x 4352 13.6 -> 11.9, 1024 x 1152 x 4352 27.2 -> 23.8, 621 x 3584 x 18944 157 -> 137. (The tiles' own workgroups asking
//     ahead gained a third of that: the same lines under way. A's lines asked for as well: no better, and worse for M = 1024.)
//   * A slab of a small tile is multiplied faster than a barrier and the LDS round trip: two slabs per barrier where LDS is there for it
//     (32x64: 13.6 -> 11.9 with the weights in L2; 128x64: 24.9 -> 23.8).
//   * A wave issues in order, so fragment reads and DMA in front of the matrix instructions leave the matrix pipe idle meanwhile: they
//     stand between them, one behind each (621 x 3584 x 18944 at 160x64: 121 -> 109; 4096 x 2048 x 5632 at 128x256: 87.5 -> 84.2).
//     128x64 with two workgroups a CU has sixteen waves to fill the gaps, and is the slower for it (24.7 -> 26.1): not there.
//   * 32x64 is four waves of 16x32 (two of 32x32: 13.7 instead of 11.9): every SIMD has one. 128x256 is eight of 64x64: four of 64x128 read a
//     quarter less LDS and are slower, a wave alone on its SIMD waits for each DMA and read it issues (4096 x 2048 x 8192 139 us, 110;
//     160x128 as four of 80x64 49 against 41). Where eight waves cannot share a slab's pieces evenly one of them fetches a few twice (2 to 9 %
//     more DMA): 160x128, 160x256. 192x256 has no room for a third slot and spills.
// Products split over K would need fewer bytes per CU, and give other bits.
//
// K is walked in order by one accumulator per output: a row's bits do not depend on which tile size, or which kernel of gemm.hip,
// computed it (frame ranges, prompts behind a kept prefix and whole prompts are compared bit for bit).
#include "common.h"
#include "kernels.h"
#include "gemm_epilogue.h"
#include "weights_ahead.h"
#include "debug.h"

namespace {

struct MidArgs {
    const char* A; long lda;   // bytes per row
    const char* W; long ldw;
    int M, N, KT;              // KT: 64-wide K slabs
    int rows0, cols0;          // the rectangle at the origin that is computed elsewhere (0, 0: none)
    int nbm, nbn;              // tiles of the rows from rows0 on
    int nbm0, nbn0;            // ... and of the columns from cols0 on of the rows in front of them; workgroups past both are prefetch_weights
    int group, group0;         // row tiles that share a panel of weights
    const float* ln_part; int ln_tiles; float ln_inv_h, ln_eps;     // EPI_LNFOLD: row statistics still in partial sums (or null)
    int ln_staged;             // a tile's fit a ring slot
    CogsWeightsAhead next;     // the next product's
    bool hot;                  // the launches in front have read this one's
    char* kv_k; char* kv_v; int kv_col, kv_dim;      // EPI_ROPE, K and V columns into cache rows of kv_dim (or null)
    EpiArgs epi;
};

constexpr int ROW_BYTES = 128, MID_CUS = 256, MAX_GROUP = 12;

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

// columns whose weights `of` workgroups can ask for in the time of a tile (below)
constexpr int read_ahead_cols(int TM, int TN, int of) { return of * (TM + TN) * 9 / 16; }

// workgroups (a multiple of 8: as many on each XCD) behind those of the tiles: one dword of every weight line that the tiles of this
// XCD read, slabs in order, so that the tiles' DMA finds them in L2. Nothing waits for them and nothing is kept.
__device__ __forceinline__ void prefetch_weights(const MidArgs& p, char* smem, int TM, int TN, int waves, int wid, int lane) {
    const int nb = p.nbm * p.nbn, xcd = blockIdx.x & 7, q = nb >> 3, r = nb & 7;
    const int x0 = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q, x1 = x0 + q + (xcd < r);
    const int of = ((int)gridDim.x - nb) >> 3, me = ((int)blockIdx.x - nb) >> 3;
    const int per_group = p.group * p.nbn;
    auto columns = [&](int& t, int& lo, int& hi) {               // of the next group of row tiles (usually there is one)
        const int g0 = t / per_group * per_group, gsz = min(p.nbm - g0 / p.nbn, p.group), e = min(x1, g0 + gsz * p.nbn);
        lo = (t - g0) / gsz * TN;
        hi = min(((e - 1 - g0) / gsz + 1) * TN, p.N);
        t = e;
    };
    int cols = 0, lo, hi;
    for (int t = x0; t < x1;) {
        columns(t, lo, hi);
        cols += hi - lo;
    }
    // A CU asks for missing lines at 55 to 60 B/ns and a tile takes in TM + TN rows of a slab at up to 110: where these workgroups have
    // more columns than they can ask for in the tiles' time the launch would wait for them, so they take evenly spaced slabs, and none
    // if that were less than half of them. 37 888 x 3584, M = 128 (a fifth): every slab 145 us, the fifth 75, none 68; 6176 x 2048,
    // M = 1152 110 -> 32.5; 4608 x 3584, M = 1152 95 -> 46; where all can be had (3584 x 18 944, M = 621) 108, none 134.
    const int slabs = (int)min((long)p.KT, (long)p.KT * read_ahead_cols(TM, TN, of) / max(cols, 1));
    if (2 * slabs < p.KT) return;
    for (int j = me * waves + wid; j < slabs; j += of * waves) {
        const int k = (int)((long)j * p.KT / slabs);
        for (int t = x0; t < x1;) {
            columns(t, lo, hi);
            for (int n = lo; n < hi; n += 64)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p.W + (long)min(n + lane, hi - 1) * p.ldw + (long)k * ROW_BYTES),
                                                 (__attribute__((address_space(3))) void*)smem, 4, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// WM x WN waves of 16 MI x 16 NI outputs, S ring slots of KS slabs; IL: reads and DMA between the matrix instructions
template <int EPI, int MI, int NI, int WM, int WN, int S, int WPE, int KS, bool IL>
__global__ __launch_bounds__(64 * WM * WN, WPE) void gemm_mid_kernel(MidArgs p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int TM = 16 * MI * WM, TN = 16 * NI * WN, WAVES = WM * WN;
    constexpr int SUB = (TM + TN) * ROW_BYTES, SLAB = SUB * KS, PIECES = SUB / 1024, P1 = (PIECES + WAVES - 1) / WAVES, P = P1 * KS;      // P: a wave's pieces per slot
    static_assert(SUB % 1024 == 0, "");
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid / WN, wn = wid % WN;
    const int rest_tiles = p.nbm * p.nbn, tiles = rest_tiles + p.nbm0 * p.nbn0;
    if ((int)blockIdx.x >= tiles) {
        if (p.next.W) read_weights_ahead(p.next, CogsWeightsAhead{}, blockIdx.x & 7, (((int)blockIdx.x - tiles) >> 3) * WAVES + wid, (((int)gridDim.x - tiles) >> 3) * WAVES, lane);
        else prefetch_weights(p, smem, TM, TN, WAVES, wid, lane);
        return;
    }
    const int KT = (p.KT + KS - 1) / KS;                         // slots' worth
    const bool odd = KS == 2 && (p.KT & 1);                      // the last one holds one slab

    // block -> tile: XCD-aware, then groups of up to 12 row tiles with the rows running fastest, so that the row tiles that share a
    // panel of weights run on one XCD
    int m0, n0;
    {
        const int xcd = blockIdx.x & 7, q = tiles >> 3, r = tiles & 7;
        int bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (blockIdx.x >> 3);
        const bool front = bid >= rest_tiles;                    // of the rows in front of rows0
        if (front) bid -= rest_tiles;
        const int group = front ? p.group0 : p.group, nbm = front ? p.nbm0 : p.nbm, per_group = group * (front ? p.nbn0 : p.nbn);
        const int first_m = bid / per_group * group, gsz = min(nbm - first_m, group);
        m0 = (first_m + (bid % per_group) % gsz) * TM + (front ? 0 : p.rows0);
        n0 = ((bid % per_group) / gsz) * TN + (front ? p.cols0 : 0);
        if (front) p.M = p.rows0;
    }
    // piece pc of a slab: tile rows 8 pc .. +7 (A's rows, then W's); lane -> row + (lane >> 3), 16-byte chunk lane & 7, swizzled. Every wave
    // stages P1 of them (its waits count them); where they do not divide, the last wave writes some of its neighbour's again, the same bytes
    const int first_piece = min(wid * P1, PIECES - P1);
    const char* src[P1];
#pragma unroll
    for (int i = 0; i < P1; ++i) {
        const int r = (first_piece + i) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ (r & 7);
        src[i] = r < TM ? p.A + (long)min(m0 + r, p.M - 1) * p.lda + c * 16 : p.W + (long)min(n0 + r - TM, p.N - 1) * p.ldw + c * 16;
    }
    char* const lds_wave = smem + first_piece * 1024;
    auto stage_piece = [&](int slot, int i, int u, int step) {
        glds16(src[i] + u * step, lds_wave + slot * SLAB + u * SUB + i * 1024);
    };
    auto advance = [&]() {
#pragma unroll
        for (int i = 0; i < P1; ++i) src[i] += ROW_BYTES * KS;
    };
    // the next KS slabs of the stream; alone: K ends behind the first (which then stands in for the second, not multiplied)
    auto stage = [&](int slot, bool alone) {
        const int step = KS == 2 && alone ? 0 : ROW_BYTES;
#pragma unroll
        for (int u = 0; u < KS; ++u)
#pragma unroll
            for (int i = 0; i < P1; ++i) stage_piece(slot, i, u, step);
        advance();
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
    struct Frags { u32x4 a[2 * KS][MI], w[2 * KS][NI]; } f0, f1;       // half slabs
    auto load_frag = [&](Frags& f, int slot, int s, int i) {           // half slab s: its NI weight fragments, then its MI others
        const char* r = smem + slot * SLAB + (s >> 1) * SUB + foff[s & 1];
        if (i < NI) f.w[s][i] = *reinterpret_cast<const u32x4*>(r + w_off + i * 16 * ROW_BYTES);
        else f.a[s][i - NI] = *reinterpret_cast<const u32x4*>(r + a_off + (i - NI) * 16 * ROW_BYTES);
    };
    auto load_frags = [&](Frags& f, int slot) {
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s)
#pragma unroll
            for (int i = 0; i < MI + NI; ++i) load_frag(f, slot, s, i);
    };
    auto mma1 = [&](Frags& f, int s, int mi, int ni) {
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.w[s][ni]), __builtin_bit_cast(bf16x8, f.a[s][mi]),
                                                              acc[mi][ni], 0, 0, 0);
    };
    auto mma = [&](Frags& f, int s0, int s1) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = s0; s < s1; ++s)
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) mma1(f, s, mi, ni);
        __builtin_amdgcn_s_setprio(0);
    };
    // the wait for the fragments stands here, in front of newer LDS reads
    auto touch = [&](Frags& f) {
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s) {
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
    // K and V of a prompt: straight into the cache (28 copies of 4.8 us in a prompt of 621 tokens)
    if constexpr (EPI == EPI_ROPE || EPI == (EPI_BIAS | EPI_ROPE)) {
        if (p.kv_k && nb >= p.kv_col) {
            const bool v = nb >= p.kv_col + p.kv_dim;
            p.epi.C = (v ? p.kv_v : p.kv_k) - (long)(v ? p.kv_col + p.kv_dim : p.kv_col) * 2;
            p.epi.ldc = p.kv_dim;
        }
    }
    constexpr bool EARLY = NI == 2 && (EPI & EPI_GENERIC) == 0;
    EpiOperands<bf16_t, EPI, MI, NI> early;
    if constexpr (EARLY) early.load(p.epi, mb, nb, p.M, p.N, lane);
    // EPI_LNFOLD: the factors of this wave's rows while the ring fills; lane l has rows l and l + 64 of its 16 MI. Their partial sums, one run of memory
    // for the tile's rows, come through the ring's last slot, ahead of the slabs: a lane reading its row's from memory is 64 lines a
    // load, 18 loads a wave, in front of the loop (M = 256 of the vision encoder: fc1 13.8 -> 12.5 us, QKV 11.2 -> 10.3)
    constexpr int FACTORS = MI > 4 ? 2 : 1;
    float factor[FACTORS];
    int filled = 0;
    auto fill = [&](int upto) {
        for (; filled < upto && filled < KT; ++filled) stage(filled, odd && filled == KT - 1);
    };
    if constexpr ((EPI & EPI_LNFOLD) != 0) {
        auto in_tile = [&](int f) { return wm * 16 * MI + min(64 * f + lane, 16 * MI - 1); };
        if (p.ln_part && p.ln_staged) {
            char* const lds = smem + (S - 1) * SLAB;
            const long first = (long)m0 * p.ln_tiles * 8, last = (long)p.M * p.ln_tiles * 8 - 16;
            for (int i = wid * 1024; i < TM * p.ln_tiles * 8; i += WAVES * 1024)
                glds16(reinterpret_cast<const char*>(p.ln_part) + min(first + i + lane * 16, last), lds + i);
            fill(S - 1);
            wait_slabs<P, S - 1>(filled);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int f = 0; f < FACTORS; ++f) {
                factor[f] = ln_row_factors(reinterpret_cast<const f32x2*>(lds) + min(in_tile(f), p.M - 1 - m0) * p.ln_tiles, p.ln_tiles, p.ln_inv_h, p.ln_eps)[0];
                asm volatile("" : "+v"(factor[f]));
            }
            __builtin_amdgcn_s_barrier();                        // every wave has read it
            asm volatile("" ::: "memory");
        } else {
            fill(S);
#pragma unroll
            for (int f = 0; f < FACTORS; ++f) {
                const long r = min(m0 + in_tile(f), p.M - 1);
                factor[f] = p.ln_part ? ln_row_factors(reinterpret_cast<const f32x2*>(p.ln_part) + r * p.ln_tiles, p.ln_tiles, p.ln_inv_h, p.ln_eps)[0] : p.epi.ln_ab[2 * r];
            }
        }
    }
    fill(S);
    wait_slabs<P, S - 1>(min(S, KT) - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_frags(f0, 0);
    int slot = 0, kt = 0;
    // slot kt is in the fragments `cur`: once every wave has it there, its place takes slot kt + S, and slot kt + 1 is read into the
    // other set while this one is multiplied
    auto steady = [&](Frags& cur, Frags& nxt) {
        const int next = slot == S - 1 ? 0 : slot + 1;
        touch(cur);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * P) : "memory");       // slot kt + 1 has landed
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (!IL) {
            stage(slot, false);
            load_frags(nxt, next);
            mma(cur, 0, 2 * KS);
        } else {
            constexpr int READS = 2 * KS * (MI + NI), OPS = READS + P, MMAS = 2 * KS * MI * NI;
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int m = 0; m < MMAS; ++m) {
                mma1(cur, m / (MI * NI), m / NI % MI, m % NI);
#pragma unroll
                for (int o = 0; o < OPS; ++o) {                  // one behind each; what is left behind the last
                    if (o < m || (o > m && m < MMAS - 1)) continue;
                    if (o < READS) load_frag(nxt, next, o / (MI + NI), o % (MI + NI));
                    else stage_piece(slot, (o - READS) % P1, (o - READS) / P1, ROW_BYTES);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            advance();
        }
        slot = next;
    };
    for (; kt + S + KS < KT; kt += 2) {
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
            load_frags(nxt, next);
            if (kt + S < KT) stage(slot, odd && kt + S == KT - 1);
        }
        mma(cur, 0, 2);
        if (KS == 2 && !(odd && kt == KT - 1)) mma(cur, 2, 2 * KS);
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
        for (int mi = 0; mi < MI; ++mi) rs[mi] = __shfl(factor[mi >> 2], 16 * (mi & 3) + (lane & 15));
        epilogue_tile<bf16_t, EPI, MI, NI>(p.epi, mb, nb, p.M, p.N, lane, acc, nullptr, rs, operands);
    } else if constexpr (MI == 5 && NI == 4) {
        f32x4 top[4][4], low[1][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) top[i][j] = acc[i][j];
            low[0][j] = acc[4][j];
        }
        epilogue_wave<bf16_t, EPI>(p.epi, mb, nb, p.M, p.N, lane, top);
        epilogue_tile<bf16_t, EPI, 1, 4>(p.epi, mb + 64, nb, p.M, p.N, lane, low);
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

// CUs without a tile: up to four workgroups an XCD prefetch (one image, encoded over and over: 1561 us without, 1494 with two an XCD, 1371 with four,
// 1374 with eight). The next product's weights are read on all of them: with 32, 64, 112 of the 112 CUs that 256 x 1152 x 4352 leaves 1424, 1335, 1313 us
int read_ahead_workgroups(int tiles) { return tiles >= MID_CUS ? 0 : tiles > MID_CUS - 32 ? (MID_CUS - tiles) / 8 * 8 : 32; }

template <int EPI, int MI, int NI, int WM, int WN, int S, int WPE, int KS, bool IL>
void launch(hipStream_t st, MidArgs& p, bool alone) {
    constexpr int TM = 16 * MI * WM, TN = 16 * NI * WN, lds = S * KS * (TM + TN) * ROW_BYTES;
    static_assert(lds <= 160 * 1024, "");
    static std::atomic<uint64_t> attr_done{0};
    cogs_ensure_dyn_lds((const void*)gemm_mid_kernel<EPI, MI, NI, WM, WN, S, WPE, KS, IL>, lds, attr_done);
    p.nbm = (p.M - p.rows0 + TM - 1) / TM;
    p.nbn = (p.N + TN - 1) / TN;
    p.nbm0 = (p.rows0 + TM - 1) / TM;
    p.nbn0 = (p.N - p.cols0 + TN - 1) / TN;
    // groups of row tiles as equal as they come: one row tile left over read every weight for itself, 9 row tiles of 1152 x 3456 x 1152
    // 69.6 us (with its XCD's prefetch, below) against 14.1 in one group
    auto group_of = [](int nbm) {
        const int groups = (nbm + MAX_GROUP - 1) / MAX_GROUP;
        return groups ? (nbm + groups - 1) / groups : 1;
    };
    p.group = group_of(p.nbm);
    p.group0 = group_of(p.nbm0);
    p.ln_staged = (long)TM * p.ln_tiles * 8 <= KS * (TM + TN) * ROW_BYTES && ((long)p.M * p.ln_tiles) % 2 == 0;
    const int tiles = p.nbm * p.nbn + p.nbm0 * p.nbn0;
    const int free = max(MID_CUS - tiles, 0) / 8 * 8;
    if (ahead_bytes(p.next) > free * WEIGHTS_AHEAD_BYTES) p.next.W = nullptr;
    const int extra = !alone || p.rows0 != 0 ? 0 : p.next.W ? free : p.hot ? 0 : read_ahead_workgroups(tiles);
    if (extra == 0) p.next.W = nullptr;
    hipLaunchKernelGGL((gemm_mid_kernel<EPI, MI, NI, WM, WN, S, WPE, KS, IL>), dim3(tiles + extra), dim3(64 * WM * WN), lds, st, p);
}

// 64x64 tiles, four ring slots or five: the fifth hides latency where the weights come from HBM -- the launch is slow for its lines, not
// for its matrix instructions, and most of all where the last row tile is nearly empty: 200 x 3584 x 3584 17.0 -> 15.0 us, 129 x 4096 x 2048
// 11.1 -> 10.1, 129 x 3584 x 1152 7.5 -> 7.1, whole row tiles 256 x 3584 x 3584 18.2 -> 17.4. It costs a slab's time in front of a short loop
// (1024 x 1152 x 512 6.5 -> 6.9, 256 x 3584 x 768 level; up to twice as long a one with two workgroups on a CU, which hide each other's
// latency: 1024 x 1152 x 1536 13.0 -> 13.5) and 1 to 4 % where every weight is read ahead into L2 (256 x 1152 x 1152 6.6 -> 6.8,
// 256 x 1152 x 2560 10.3 -> 10.6).
bool four_slots(const MidArgs& p, bool alone) {
    const int nbm = (p.M + 63) / 64, tiles = nbm * ((p.N + 63) / 64), cols = ((tiles + 7) / 8 + nbm - 1) / nbm * 64;      // of an XCD
    return p.KT <= (tiles > MID_CUS ? 24 : 12) || cols <= read_ahead_cols(64, 64, (alone ? read_ahead_workgroups(tiles) : 0) / 8);
}

template <int EPI>
void dispatch_tile(hipStream_t st, MidArgs& p, int tile, bool alone) {
    switch (tile) {
        case 1: launch<EPI, 1, 2, 2, 2, 4, 2, 2, true>(st, p, alone); break;          // 32 x 64
        case 2:                                                                       // 64 x 64, two a CU
            if (four_slots(p, alone)) launch<EPI, 2, 2, 2, 2, 4, 2, 1, true>(st, p, alone);
            else launch<EPI, 2, 2, 2, 2, 5, 2, 1, true>(st, p, alone);
            break;
        case 3: launch<EPI, 2, 2, 4, 2, 3, 4, 1, false>(st, p, alone); break;         // 128 x 64, two a CU
        case 4: launch<EPI, 4, 2, 2, 4, 4, 2, 1, true>(st, p, alone); break;          // 128 x 128
        case 5: launch<EPI, 4, 4, 2, 4, 3, 2, 1, true>(st, p, alone); break;          // 128 x 256
        case 6: launch<EPI, 2, 2, 4, 2, 3, 2, 2, true>(st, p, alone); break;          // 128 x 64, two slabs at a time
        case 7: launch<EPI, 5, 2, 2, 2, 5, 2, 1, true>(st, p, alone); break;          // 160 x 64
        case 8: launch<EPI, 3, 2, 2, 2, 5, 2, 1, true>(st, p, alone); break;          // 96 x 64
        case 9: launch<EPI, 5, 2, 2, 4, 4, 2, 1, true>(st, p, alone); break;          // 160 x 128
        case 10: launch<EPI, 3, 4, 4, 2, 4, 2, 1, true>(st, p, alone); break;         // 192 x 128
        default: launch<EPI, 5, 4, 2, 4, 3, 2, 1, true>(st, p, alone); break;         // 160 x 256
    }
}

}  // namespace

int cogs_k_gemm_mid(hipStream_t st, const CogsGemm& g, int tile, bool alone, int rows0, int cols0) {
    MidArgs p;
    const int rc = cogs_fill_epi(g, &p.epi);
    if (rc != COGS_OK) return rc;
    p.A = (const char*)g.A; p.lda = g.lda * 2;
    p.W = (const char*)g.W; p.ldw = g.ldw * 2;
    p.M = g.M; p.N = g.N; p.KT = g.K / 64; p.rows0 = rows0; p.cols0 = cols0;
    p.next = g.next; p.hot = g.weights_read;
    p.kv_k = (char*)g.kv_k; p.kv_v = (char*)g.kv_v; p.kv_col = g.kv_col0; p.kv_dim = g.kv_dim;
    if (g.kv_k && (g.kv_col0 % 64 || g.kv_dim % 64)) p.kv_k = nullptr;      // (copied by the caller)
    p.ln_part = g.ln_part; p.ln_tiles = g.K / 64; p.ln_inv_h = 1.0f / (float)g.K; p.ln_eps = g.ln_eps;
#define COGS_MID_CASE(E) case E: dispatch_tile<E>(st, p, tile, alone); break;
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
        default: dispatch_tile<EPI_GENERIC>(st, p, tile, alone); break;
    }
#undef COGS_MID_CASE
    if (g.next_read) *g.next_read = p.next.W != nullptr;
    g_cogs_debug.weights_ahead_read += p.next.W != nullptr;
    g_cogs_debug.weights_ahead_counted_on += g.weights_read;
    return COGS_LAUNCH_CHECK();
}
