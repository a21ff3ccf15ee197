// Few-row GEMM for batched decode:  C[M,N] = epilogue( A[M,K] . W[N,K]^T ),  2 <= M <= 64, bf16.
//
// HBM-bound like the single-row GEMV (gemv.hip): every weight byte is read once, straight into MFMA A fragments. A workgroup owns
// 16 NT output columns; its NW waves take alternate 64-element slices of K (a row's slice is one whole 128-byte line), the batch rows
// are the columns of v_mfma_f32_16x16x32_bf16 (MT groups of 16), and the waves' partial tiles are summed through LDS in a fixed
// order. (How many waves and partial sums there are depends on M as well as on N and K: a row's bits may differ between steps of
// other numbers of rows.) The batch rows come from L2 once per workgroup -- as many bytes as the weights with NT = 1 and M = 16 -- so columns are
// taken 64 or 32 at a time where that still makes 160 workgroups.
//
// A sublayer's last product has few columns and a long K: 2048 columns are 128 workgroups of 16, each a quarter of what the chip
// could have in flight. Where the caller takes partial sums (cogs_k_stream_norm adds them up as it reads them), K is cut over
// gridDim.y workgroups that each store an fp32 partial. 16 rows, weights from HBM: 2048 x 5632 15.1 -> 7.9 us (2.9 TB/s),
// 2048 x 8192 18.6 -> 9.1, 2048 x 2048 6.6 -> 4.6, 4096 x 11008 30.1 -> 20.0 (4.5 TB/s); unsplit, 64 columns at a time and without the
// streaming hint on the weight loads, 11264 x 2048 16.5 -> 12.9, 22016 x 4096 50.4 -> 43.
#include "common.h"
#include "kernels.h"
#include "gemm_epilogue.h"
#include "debug.h"

namespace {

struct SkinnyArgs {
    const bf16_t* A; long lda;
    const bf16_t* W; long ldw;
    int M, N, K;
    float* part;               // gridDim.y > 1: partial sums [gridDim.y][M][N], the bias in the first
    EpiArgs epi;
};

// U slices in flight per wave
template <int MT, int NT, int NW, int U>
__global__ __launch_bounds__(64 * NW) void gemm_skinny_kernel(SkinnyArgs p) {
    __shared__ __attribute__((aligned(16))) f32x4 red[NW][MT * NT][64];
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * (16 * NT);
    const bf16_t *w[NT], *a[MT];
    f32x4 acc[MT * NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t] = p.W + (long)min(n0 + 16 * t + li, p.N - 1) * p.ldw + 8 * g;
#pragma unroll
    for (int t = 0; t < MT; ++t) a[t] = p.A + (long)min(16 * t + li, p.M - 1) * p.lda + 8 * g;
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int all = p.K >> 6, ns = all * (blockIdx.y + 1) / gridDim.y;
    for (int sl = all * blockIdx.y / gridDim.y + wid; sl < ns; sl += NW * U) {
        u32x4 wf[U][NT][2], af[U][MT][2];
        // (slices past the end repeat the last one and are not multiplied: every load of a batch goes out at once)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 64 * min(sl + NW * u, ns - 1);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) wf[u][t][hf] = *reinterpret_cast<const u32x4*>(w[t] + k + 32 * hf);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 64 * min(sl + NW * u, ns - 1);
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) af[u][t][hf] = *reinterpret_cast<const u32x4*>(a[t] + k + 32 * hf);
        }
        __builtin_amdgcn_sched_barrier(0);          // (hipcc otherwise sinks the loads to their uses to save registers)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (sl + NW * u >= ns) break;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int q = 0; q < NT; ++q)
#pragma unroll
                    for (int hf = 0; hf < 2; ++hf)
                        acc[t * NT + q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[u][q][hf]),
                                                                                  __builtin_bit_cast(bf16x8, af[u][t][hf]), acc[t * NT + q], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) red[wid][t][lane] = acc[t];
    __syncthreads();
    for (int t = wid; t < MT * NT; t += NW) {
        f32x4 v = red[0][t][lane];
#pragma unroll
        for (int s = 1; s < NW; ++s) v += red[s][t][lane];
        const int m = 16 * (t / NT) + li, n = n0 + 16 * (t % NT) + 4 * g;
        if (m >= p.M || n >= p.N) continue;
        if (gridDim.y == 1) {
            epilogue4<bf16_t>(p.epi, m, n, v);
        } else {
            if (p.epi.bias && blockIdx.y == 0) v += ld4_f<bf16_t>(reinterpret_cast<const bf16_t*>(p.epi.bias) + n);
            *reinterpret_cast<f32x4*>(p.part + ((long)blockIdx.y * p.M + m) * p.N + n) = v;
        }
    }
}

template <int MT, int NT, int NW, int U>
void launch(hipStream_t st, const SkinnyArgs& p, int splits) {
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, NW, U>), dim3((p.N + 16 * NT - 1) / (16 * NT), splits), dim3(64 * NW), 0, st, p);
}

}  // namespace

bool cogs_k_gemm_skinny_fits(const CogsGemm& g) {
    return g.dtype == COGS_DT_BF16 && g.M >= 2 && g.M <= 64 && g.K % 64 == 0 && g.N % 4 == 0 && g.lda % 8 == 0 && g.ldw % 8 == 0 &&
           !g.rms_gamma && !g.row_stats && !g.ln_ab && !g.kv_k && g.hm_rows == 0;
}

// how many partial sums a product of this size is stored as when its caller takes them (1: none). K shorter than 64 slices: two
// (M <= 16) or four; else eight or four, so that the 64-column groups come to 256 workgroups.
int cogs_k_gemm_skinny_parts(int M, int N, int K) {
    if (N > 4096 || K < 1024) return 1;
    if (M <= 32 && K < 4096) return M <= 16 ? 2 : 4;
    return N <= 2048 ? 8 : 4;
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
    if (parts > 1) {
        const bool long_k = g.K >= 4096;
        if (g.M <= 16) { if (long_k) launch<1, 4, 4, 2>(st, p, parts); else launch<1, 1, 4, 4>(st, p, parts); }
        else if (g.M <= 32) { if (long_k) launch<2, 4, 4, 2>(st, p, parts); else launch<2, 2, 4, 2>(st, p, parts); }
        else launch<4, 4, 4, 1>(st, p, parts);
        return COGS_LAUNCH_CHECK();
    }
    const bool deep = g.K >= 1024;                  // else too few slices for eight waves
    const int cols = g.N >= 64 * 160 ? 64 : g.N >= 32 * 160 ? 32 : 16;
    if (g.M <= 16) {
        if (!deep) launch<1, 1, 4, 4>(st, p, 1);
        else if (cols == 64) launch<1, 4, 4, 2>(st, p, 1);
        else if (cols == 32) launch<1, 2, 8, 2>(st, p, 1);
        else launch<1, 1, 8, 4>(st, p, 1);
    } else if (g.M <= 32) {
        if (!deep) launch<2, 1, 4, 4>(st, p, 1);
        else if (cols == 64) launch<2, 4, 8, 1>(st, p, 1);
        else if (cols == 32) launch<2, 2, 8, 2>(st, p, 1);
        else launch<2, 1, 8, 2>(st, p, 1);
    } else {
        if (!deep) launch<4, 1, 4, 2>(st, p, 1);
        else if (cols > 16) launch<4, 2, 8, 1>(st, p, 1);
        else launch<4, 1, 8, 2>(st, p, 1);
    }
    return COGS_LAUNCH_CHECK();
}
