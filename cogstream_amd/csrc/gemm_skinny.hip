// Few-row GEMM for batched decode:  C[M,N] = epilogue( A[M,K] . W[N,K]^T ),  1 <= M <= 64, bf16.
//
// HBM-bound like the single-row GEMV (gemv.hip): every weight byte is read once. A workgroup owns 16 NT output columns; its NW waves
// take alternate 64-element slices of K, the batch rows are the columns of v_mfma_f32_16x16x32_bf16 (MT groups of 16), and the
// waves' partial tiles are summed through LDS in a fixed order. (How many waves and partial sums there are depends on M as well as on N
// and K: a row's bits may differ between steps of other numbers of rows.)
//
// Each wave streams its slices through a ring of its own, D slices of whole 128-byte lines by LDS-DMA: no barrier in the loop, the
// wave waits for its own loads alone. Matrix fragments straight from memory put sixteen rows of 16 bytes into every quarter of a load: the
// vector-memory path then took in 39 B/ns a CU whatever was in flight, also of weights that sat in L2 (8 x 8192 x 2048: 7.4 us from
// L2, 9.8 from HBM); whole lines come at 110 (4.6 and 8.0). The weights are read with the streaming hint: nothing reads them again before
// the next step, and 5 to 10 % less time (11 264 x 2048, 16 rows: 11.6 -> 10.9). Columns are taken 64, 48 or 32 at a time where that still
// makes 160 workgroups: the batch rows come from L2 once per workgroup, as many bytes as the weights with NT = 1 and M = 16. Fragments
// from memory -> ring, weights from HBM (us):
//      rows    6176 x 2048    8192 x 2048    11 264 x 2048    32 768 x 2048    2048 x 8192    2048 x 5632    4096 x 11 008
//       16     9.9 -> 7.2     11.1 -> 8.6     14.8 -> 11.0     32.0 -> 26.6     9.5 -> 8.0     8.3 -> 6.4     21.9 -> 17.7
//       64    14.7 -> 10.3    15.6 -> 11.6    20.5 -> 14.9     41.6 -> 35.0    13.2 -> 10.8   10.8 -> 9.1     27.9 -> 22.4
//
// A sublayer's last product has few columns and a long K: 2048 columns are 128 workgroups of 16, each a quarter of what the chip
// could have in flight. Where the caller takes partial sums (cogs_k_stream_norm adds them up as it reads them), K is cut over
// gridDim.y workgroups that each store an fp32 partial.
#include "common.h"
#include "kernels.h"
#include "gemm_epilogue.h"
#include "mla_latent.h"
#include "debug.h"

namespace {

struct SkinnyArgs {
    const bf16_t* A; long lda;
    const bf16_t* W; long ldw;
    int M, N, K;
    float* part;               // gridDim.y > 1: partial sums [gridDim.y][M][N], the bias in the first
    EpiArgs epi;
};

// at most n slices' pieces (P each) of this wave may stay in flight, n <= MAX
template <int P, int MAX>
__device__ __forceinline__ void wait_slices(int n) {
    static_assert(MAX <= 3 && MAX * P < 64, "vmcnt is a 6-bit immediate");
    if (n <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (n == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P) : "memory");
    else if (n == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 2 ? 2 * P : 0) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MAX >= 3 ? 3 * P : 0) : "memory");
}

// a piece: 8 rows x 128 bytes, 1 KiB of LDS; HINT: cache policy bits of the load (2: streaming)
template <int HINT>
__device__ __forceinline__ void piece16(const bf16_t* g, char* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g, (__attribute__((address_space(3))) void*)l, 16, 0, HINT);
}

// AP: pieces of batch rows a slice has (rows past M repeat the last), D: slices in a wave's ring
template <int MT, int AP, int NT, int NW, int D>
__global__ __launch_bounds__(64 * NW) void gemm_skinny_kernel(SkinnyArgs p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int P = 2 * NT + AP, RING = D * P * 1024;
    static_assert(MT * NT * 1024 <= RING, "a wave's partial tile takes its ring's place");
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * (16 * NT);
    char* const ring = smem + wid * RING;
    const int all = p.K >> 6, end = all * (blockIdx.y + 1) / gridDim.y, first = all * blockIdx.y / gridDim.y + wid;
    const int n = first < end ? (end - first + NW - 1) / NW : 0;                // this wave's slices
    // lane -> row lane >> 3 of a piece, 16-byte chunk lane & 7, swizzled
    const int r = lane >> 3, c = (lane & 7) ^ r;
    const bf16_t *w[2 * NT], *a[AP];
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) w[i] = p.W + (long)min(n0 + 8 * i + r, p.N - 1) * p.ldw + 64 * first + 8 * c;
#pragma unroll
    for (int i = 0; i < AP; ++i) a[i] = p.A + (long)min(8 * i + r, p.M - 1) * p.lda + 64 * first + 8 * c;
    auto stage = [&](int slot) {                 // the next slice of the stream
        char* d = ring + slot * (P * 1024);
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i) { piece16<2>(w[i], d + i * 1024); w[i] += NW * 64; }
#pragma unroll
        for (int i = 0; i < AP; ++i) { piece16<0>(a[i], d + (2 * NT + i) * 1024); a[i] += NW * 64; }
    };
    for (int i = 0; i < D && i < n; ++i) stage(i);
    f32x4 acc[MT * NT];
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int off[2];                                  // row li of a 16-row group, 16-byte chunk 4 h + g
#pragma unroll
    for (int h = 0; h < 2; ++h) off[h] = (li & 7) * 128 + (((4 * h + g) ^ (li & 7)) << 4);
    int slot = 0;
    for (int i = 0; i < n; ++i) {
        wait_slices<P, D - 1>(min(D - 1, n - 1 - i));
        const char* d = ring + slot * (P * 1024);
        u32x4 wf[NT][2], af[MT][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t][h] = *reinterpret_cast<const u32x4*>(d + (2 * t + (li >> 3)) * 1024 + off[h]);
#pragma unroll
            for (int t = 0; t < MT; ++t) af[t][h] = *reinterpret_cast<const u32x4*>(d + (2 * NT + min(2 * t + (li >> 3), AP - 1)) * 1024 + off[h]);
        }
        // the wait for the fragments stands here, in front of the DMA into their slot
#pragma unroll
        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(wf[t][0]), "+v"(wf[t][1]));
#pragma unroll
        for (int t = 0; t < MT; ++t) asm volatile("" : "+v"(af[t][0]), "+v"(af[t][1]));
        asm volatile("" ::: "memory");
        if (i + D < n) stage(slot);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[t * NT + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[q][h]),
                                                                              __builtin_bit_cast(bf16x8, af[t][h]), acc[t * NT + q], 0, 0, 0);
        slot = slot == D - 1 ? 0 : slot + 1;
    }
    // (every load into the ring has been waited for)
    auto red = [&](int wave, int t) { return reinterpret_cast<f32x4*>(smem + wave * RING) + t * 64 + lane; };
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) *red(wid, t) = acc[t];
    __syncthreads();
    for (int t = wid; t < MT * NT; t += NW) {
        f32x4 v = *red(0, t);
#pragma unroll
        for (int s = 1; s < NW; ++s) v += *red(s, t);
        const int m = 16 * (t / NT) + li, nn = n0 + 16 * (t % NT) + 4 * g;
        if (m >= p.M || nn >= p.N) continue;
        if (gridDim.y == 1) {
            epilogue4<bf16_t>(p.epi, m, nn, v);
        } else {
            if (p.epi.bias && blockIdx.y == 0) v += ld4_f<bf16_t>(reinterpret_cast<const bf16_t*>(p.epi.bias) + nn);
            *reinterpret_cast<f32x4*>(p.part + ((long)blockIdx.y * p.M + m) * p.N + nn) = v;
        }
    }
}

// The query product of latent attention, up to 16 rows: A is the normed query latent, formed by every workgroup itself from the fused projection's fp32 rows
// while its first weights are on their way (50 to 100 KB from L2 a workgroup), and kept in LDS; the workgroups behind the columns' norm and rotate a row's
// key and value latent into its cache. A launch of 16 workgroups in front of this one cost 4.7 us of latency, and this one 2.7 more: 16 rows of 3072 x 768
// 4.7 + 4.2 -> 6.9, a token of 16 requests 694 -> 684, of 3 553 -> 536. The norms have the bits of mla_latent_kernel (four waves share K, also of 32 columns).
template <int AP, int J, int NT, int D>
__global__ __launch_bounds__(256) void gemm_skinny_latent_kernel(SkinnyArgs p, CogsMlaLatent l) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ __attribute__((aligned(16))) float red[16][4];
    constexpr int NW = 4, P = 2 * NT, RING = D * P * 1024;
    static_assert(NT * 1024 <= RING, "a wave's partial tile takes its ring's place");
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = (p.N + 16 * NT - 1) / (16 * NT);
    if ((int)blockIdx.x >= tiles) {
        latent_row<bf16_t, false>(l, blockIdx.x - tiles, tid, &red[0][0]);
        return;
    }
    const int n0 = blockIdx.x * (16 * NT);
    char* const ring = smem + wid * RING;
    char* const rows = smem + NW * RING;                         // [slice][AP pieces], as a ring slot would hold them
    const int all = p.K >> 6, n = wid < all ? (all - wid + NW - 1) / NW : 0;
    const int r = lane >> 3, c = (lane & 7) ^ r;
    const bf16_t* w[2 * NT];
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) w[i] = p.W + (long)min(n0 + 8 * i + r, p.N - 1) * p.ldw + 8 * c;
    auto stage = [&](int slot, int i) {                          // slice i of this wave (past its last: K's last once more)
        const int k = 64 * min(wid + NW * i, all - 1);
#pragma unroll
        for (int q = 0; q < 2 * NT; ++q) piece16<2>(w[q] + k, ring + (slot * P + q) * 1024);
    };
    {
        constexpr int R = 8 * AP;                                // a thread has four columns of every 1024 of each row
        f32x4 v[R][J];
#pragma unroll
        for (int m = 0; m < R; ++m)
#pragma unroll
            for (int j = 0; j < J; ++j) v[m][j] = *reinterpret_cast<const f32x4*>(l.t + (long)min(m, p.M - 1) * l.ldt + min(tid * 4 + 1024 * j, p.K - 4));
        f32x4 norm[J];
#pragma unroll
        for (int j = 0; j < J; ++j) norm[j] = *reinterpret_cast<const f32x4*>(l.q_norm + min(tid * 4 + 1024 * j, p.K - 4));
#pragma unroll
        for (int i = 0; i < D; ++i) stage(i, i);                 // (behind the rows' loads, and as many on every way here: those are waited for alone)
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (tid * 4 + 1024 * j >= p.K)
#pragma unroll
                for (int m = 0; m < R; ++m) v[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < R; ++m) {
            float sq = 0.f;
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) sq = fmaf(v[m][j][e], v[m][j][e], sq);      // (written out: left to the compiler, the first two swap places here)
            sq = wave_sum(sq);
            if (lane == 0) red[m][wid] = sq;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // a row's factor by one lane each
        const f32x4 sums = *reinterpret_cast<const f32x4*>(red[min(li, R - 1)]);
        const float factor = 1.f / sqrtf(((sums[0] + sums[1]) + (sums[2] + sums[3])) / (float)l.qr + l.eps);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int col = tid * 4 + 1024 * j;
            if (col >= p.K) continue;
#pragma unroll
            for (int m = 0; m < R; ++m) {
                const float rq = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(factor), m));
                u32x2 b;
                b[0] = pack_bf2(v[m][j][0] * rq * norm[j][0], v[m][j][1] * rq * norm[j][1]);
                b[1] = pack_bf2(v[m][j][2] * rq * norm[j][2], v[m][j][3] * rq * norm[j][3]);
                *reinterpret_cast<u32x2*>(rows + ((col >> 6) * AP + (m >> 3)) * 1024 + (m & 7) * 128 + ((((col >> 3) & 7) ^ (m & 7)) << 4) + (col & 4) * 2) = b;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) off[h] = (li & 7) * 128 + (((4 * h + g) ^ (li & 7)) << 4);
    int slot = 0;
    for (int i = 0; i < n; ++i) {
        wait_slices<P, D - 1>(min(D - 1, max(n, D) - 1 - i));
        const char* d = ring + slot * (P * 1024);
        const char* a = rows + ((wid + NW * i) * AP + min(li >> 3, AP - 1)) * 1024;
        u32x4 wf[NT][2], af[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t][h] = *reinterpret_cast<const u32x4*>(d + (2 * t + (li >> 3)) * 1024 + off[h]);
            af[h] = *reinterpret_cast<const u32x4*>(a + off[h]);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(wf[t][0]), "+v"(wf[t][1]));
        asm volatile("" ::: "memory");
        if (i + D < n) stage(slot, i + D);
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[q][h]), __builtin_bit_cast(bf16x8, af[h]), acc[q], 0, 0, 0);
        slot = slot == D - 1 ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // (slices past the last)
    auto part = [&](int wave, int t) { return reinterpret_cast<f32x4*>(smem + wave * RING) + t * 64 + lane; };
#pragma unroll
    for (int t = 0; t < NT; ++t) *part(wid, t) = acc[t];
    __syncthreads();
    for (int t = wid; t < NT; t += NW) {
        f32x4 v = *part(0, t);
#pragma unroll
        for (int s = 1; s < NW; ++s) v += *part(s, t);
        const int nn = n0 + 16 * t + 4 * g;
        if (li < p.M && nn < p.N) epilogue4<bf16_t>(p.epi, li, nn, v);
    }
}

template <int AP, int J, int NT, int D>
void launch_latent(hipStream_t st, const SkinnyArgs& p, const CogsMlaLatent& l, int extra) {
    static std::atomic<uint64_t> attr_done{0};
    cogs_ensure_dyn_lds((const void*)gemm_skinny_latent_kernel<AP, J, NT, D>, 152 * 1024, attr_done);
    const size_t lds = (size_t)4 * D * 2 * NT * 1024 + (size_t)(p.K / 64) * AP * 1024;
    hipLaunchKernelGGL((gemm_skinny_latent_kernel<AP, J, NT, D>), dim3((p.N + 16 * NT - 1) / (16 * NT) + extra), dim3(256), lds, st, p, l);
}
template <int AP, int J>
void launch_latent_cols(hipStream_t st, const SkinnyArgs& p, const CogsMlaLatent& l, int cols, int extra) {
    if (cols >= 48) launch_latent<AP, J, 4, 2>(st, p, l, extra);
    else if (cols == 32) launch_latent<AP, J, 2, 3>(st, p, l, extra);
    else launch_latent<AP, J, 1, 3>(st, p, l, extra);
}

template <int MT, int AP, int NT, int NW, int D>
void launch1(hipStream_t st, const SkinnyArgs& p, int splits) {
    constexpr int lds = NW * D * (2 * NT + AP) * 1024;
    static_assert(lds <= 160 * 1024, "");
    static std::atomic<uint64_t> attr_done{0};
    cogs_ensure_dyn_lds((const void*)gemm_skinny_kernel<MT, AP, NT, NW, D>, lds, attr_done);
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, AP, NT, NW, D>), dim3((p.N + 16 * NT - 1) / (16 * NT), splits), dim3(64 * NW), lds, st, p);
}
template <int MT, int NT, int NW, int D>
void launch(hipStream_t st, const SkinnyArgs& p, int splits) {
    if constexpr (MT == 1)
        if (p.M <= 8) return launch1<MT, 1, NT, NW, D>(st, p, splits);
    launch1<MT, 2 * MT, NT, NW, D>(st, p, splits);
}
// columns at a time; the ring takes 48 (up to eight rows, 16 columns) to 144 KB, two workgroups a CU for the most used sizes
template <int MT>
void launch_cols(hipStream_t st, const SkinnyArgs& p, int cols, int splits) {
    if (cols == 64) launch<MT, 4, 4, 2>(st, p, splits);
    else if (cols == 48 && MT == 1) launch<1, 3, 4, 2>(st, p, splits);
    else if (cols == 32) launch<MT, 2, MT == 1 ? 8 : 4, 3>(st, p, splits);
    else launch<MT, 1, 4, MT == 1 ? 4 : MT == 2 ? 3 : 2>(st, p, splits);
}

// columns per workgroup of a product without partial sums. 48 instead of 64 where the CU with most workgroups then takes fewer columns in (with the 16
// batch rows of each): 16 rows, us, 64 / 48 columns, 11 264 x 2048 10.7 / 10.3, 22 016 x 4096 36.8 / 30.3, 10 808 x 3584 15.7 / 14.1, and by the rule
// with 64: 12 320 x 4096 19.3 / 24.3, 16 384 x 4096 25.6 / 27.4, 28 416 x 3584 32.9 / 36.3, 37 888 x 3584 46.5 / 47.5
int whole_cols(int M, int N) {
    if (N < 64 * 160) return N >= 32 * 160 ? 32 : 16;
    auto taken = [N](int cols) { return ((N + cols - 1) / cols + 255) / 256 * (cols + 16); };
    return M <= 16 && taken(48) < taken(64) ? 48 : 64;
}

}  // namespace

bool cogs_k_gemm_skinny_fits(const CogsGemm& g) {
    return g.dtype == COGS_DT_BF16 && g.M >= 1 && g.M <= 64 && g.K % 64 == 0 && g.N % 4 == 0 && g.lda % 8 == 0 && g.ldw % 8 == 0 &&
           !g.rms_gamma && !g.row_stats && !g.ln_ab && !g.kv_k && g.hm_rows == 0;
}

// One row, without partial sums: here where the columns come to whole rounds of workgroups, else by the GEMV, whose waves take four columns at a time
// (GEMV / here, us: 32 768 x 2048 31.6 / 24.3, 22 016 x 4096 33.4 / 30.1, 28 416 x 3584 33.4 / 31.8, 10 808 x 3584 15.2 / 13.2, 16 384 x 4096 26.1 / 26.0;
// not full 37 888 x 3584 42.5 / 45.2, 6144 x 4096 10.5 / 11.9, 1344 x 2048 3.9 / 4.5). With three quarters of the CUs busy a short K is still the
// faster here, where latency counts: 3072 x 2048 5.4 / 4.7, 6176 x 2048 6.9 / 6.4, 5376 x 3584 9.4 / 8.3. Partial sums are always: 2048 x 2048 5.0 / 3.8,
// 2048 x 5632 7.2 / 6.1, 3584 x 28 416 35.7 / 31.4.
bool cogs_k_gemm_skinny_one_row(int N, int K) {
    const int cols = whole_cols(1, N), wgs = (N + cols - 1) / cols, rounds = (wgs + 255) / 256;
    return wgs * 5 >= rounds * 256 * 4 || (rounds == 1 && wgs >= 128 && K < 4096);
}

// how many partial sums a product of this size is stored as when its caller takes them (1: none). K shorter than 64 slices: two
// (M <= 16) or four; else eight or four, so that the 64-column groups come to 256 workgroups.
int cogs_k_gemm_skinny_parts(int M, int N, int K) {
    if (N > 4096 || K < 1024) return 1;
    if (K < 4096) return M <= 16 ? 2 : 4;
    return N <= 2048 ? 8 : 4;
}

// how much of the next product's weights a mix of 4 us reads on idle CUs: what HBM gives meanwhile, or the mix takes the longer. Widths of 2048, 3 rows
// stepped 24 times: none 11.57 ms, 5 MB 11.04, 8 MB 11.00, 12 MB 11.05, 18 MB 11.20, 40 MB 12.19; 8 rows 12.43 -> 12.06 with 8 MB; width
// 3584, 16 rows, 12 steps 8.51 -> 8.36. (Norms of one stream are shorter and gained nothing.)
constexpr long AHEAD_BYTES = 8000000;

CogsAhead cogs_k_gemm_skinny_ahead(const void* W, long ldw, int M, int N, int K) {
    CogsAhead a;
    CogsGemm g;
    g.dtype = COGS_DT_BF16; g.M = M; g.N = N; g.K = K; g.lda = K; g.ldw = ldw;
    if (!W || g_cogs_debug.gemm_skinny == 0 || !cogs_k_gemm_skinny_fits(g) || (M == 1 && !cogs_k_gemm_skinny_one_row(N, K))) return a;
    const long lines = AHEAD_BYTES / (128L * N);
    a.W = (const char*)W; a.ldw = ldw * 2; a.N = N; a.cols = whole_cols(M, N); a.groups = (N + a.cols - 1) / a.cols;
    a.lines = (int)(lines < K / 64 ? lines : K / 64);
    return a;
}

int cogs_k_gemm_skinny(hipStream_t st, const CogsGemm& g, float* part) {
    if (!cogs_k_gemm_skinny_fits(g)) return COGS_E_UNSUPPORTED;
    SkinnyArgs p;
    const int rc = cogs_fill_epi(g, &p.epi);
    if (rc != COGS_OK) return rc;
    p.A = (const bf16_t*)g.A; p.lda = g.lda; p.W = (const bf16_t*)g.W; p.ldw = g.ldw;
    p.M = g.M; p.N = g.N; p.K = g.K; p.part = part;
    g_cogs_debug.gemm_last_body = 7;
    const int parts = part ? cogs_k_gemm_skinny_parts(g.M, g.N, g.K) : 1;
    if (part && (g.act != COGS_ACT_NONE || g.residual || g.rope_cos || g.out_f32 || parts < 2)) return COGS_E_UNSUPPORTED;
    const int cols = parts > 1 ? (g.K >= 4096 ? 64 : g.M <= 16 ? 16 : 32) : whole_cols(g.M, g.N);
    if (g.M <= 16) launch_cols<1>(st, p, cols, parts);
    else if (g.M <= 32) launch_cols<2>(st, p, cols, parts);
    else launch_cols<4>(st, p, cols, parts);
    return COGS_LAUNCH_CHECK();
}

// (one row too: one token of one request, by the GEMV and a launch for its norms in front 567 us, 550 so; of width 4096 669, 661, of 3584 738, 730)
bool cogs_k_gemm_skinny_latent_fits(const CogsGemm& g) { return cogs_k_gemm_skinny_fits(g) && g.M <= 16 && g.K <= 2048 && g_cogs_debug.gemm_skinny != 0; }

// g's rows are l's normed query latents (g.A is not read); l's key and value latents and gates go where cogs_k_mla_latent puts them
int cogs_k_gemm_skinny_latent(hipStream_t st, const CogsGemm& g, const CogsMlaLatent& l) {
    if (!cogs_k_gemm_skinny_latent_fits(g) || g.K != l.qrp || l.kvp % 4 || l.krc % 2 || l.ldt % 4 || l.dr % 2) return COGS_E_UNSUPPORTED;
    SkinnyArgs p;
    const int rc = cogs_fill_epi(g, &p.epi);
    if (rc != COGS_OK) return rc;
    p.A = nullptr; p.lda = 0; p.W = (const bf16_t*)g.W; p.ldw = g.ldw;
    p.M = g.M; p.N = g.N; p.K = g.K; p.part = nullptr;
    g_cogs_debug.gemm_last_body = 7;
    const int extra = l.own_kv || l.gate_col >= 0 ? g.M : 0, cols = whole_cols(g.M, g.N);
    if (g.M <= 8) g.K <= 1024 ? launch_latent_cols<1, 1>(st, p, l, cols, extra) : launch_latent_cols<1, 2>(st, p, l, cols, extra);
    else g.K <= 1024 ? launch_latent_cols<2, 1>(st, p, l, cols, extra) : launch_latent_cols<2, 2>(st, p, l, cols, extra);
    return COGS_LAUNCH_CHECK();
}
