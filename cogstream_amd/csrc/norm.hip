// Row normalisations: LayerNorm (ViT), RMSNorm (Qwen2), and post-LayerNorm fused with the
// 2x2 token merge.
//
// Replaces: nn.LayerNorm(1152, eps=1e-6) x(2*27+1) (model/modeling_videollama3_encoder.py:382-384,
// :475), post_layernorm + un-permute + F.interpolate(bilinear, 1/2) (:482-501; with the
// merge-window-major row order every 4 consecutive rows are one 2x2 window, so the bilinear
// half-size resample is their mean), and transformers' Qwen2RMSNorm (fp32 variance,
// x*rsqrt(var+eps) cast back, then * weight).
//
// HBM-bound: one wave per row, the row lives in registers (16-byte loads, 8 elements per
// lane per chunk), statistics by 64-lane butterfly, one read + one write per element.
#include "common.h"
#include "kernels.h"

namespace {

template <typename T, int CPL, bool RMS>
__global__ __launch_bounds__(256) void norm_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                   const T* __restrict__ gamma, const T* __restrict__ beta,
                                                   int rows, int H, float eps) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int nch = H >> 3;
    const T* xr = x + (long)row * H;
    // the row and its gain are asked for as a whole, chunks past the end as the last one again: under a test of the chunk every load was
    // waited for before the next went out (621 rows of 3584: 7.2 -> 5.1 us)
    constexpr int V = sizeof(T) * 8 / 16;                // 16-byte loads of a chunk
    u32x4 raw[CPL][V], graw[CPL][V];
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int i = 0; i < V; ++i) raw[c][i] = *(reinterpret_cast<const u32x4*>(xr + min(lane + 64 * c, nch - 1) * 8) + i);
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int i = 0; i < V; ++i) graw[c][i] = *(reinterpret_cast<const u32x4*>(gamma + min(lane + 64 * c, nch - 1) * 8) + i);
    float v[CPL][8];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        ld8_f<T>(reinterpret_cast<const T*>(raw[c]), v[c]);
        if (lane + 64 * c < nch) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += RMS ? v[c][e] * v[c][e] : v[c][e];
        }
    }
    sum = wave_sum(sum);
    float mean = 0.f, rstd;
    if (RMS) {
        rstd = rsqrtf(sum / (float)H + eps);
    } else {
        mean = sum / (float)H;
        float sq = 0.f;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int ch = lane + 64 * c;
            if (ch < nch) {
#pragma unroll
                for (int e = 0; e < 8; ++e) { const float d = v[c][e] - mean; sq += d * d; }
            }
        }
        sq = wave_sum(sq);
        rstd = rsqrtf(sq / (float)H + eps);
    }
    T* yr = y + (long)row * H;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = lane + 64 * c;
        if (ch < nch) {
            float gm[8], o[8];
            ld8_f<T>(reinterpret_cast<const T*>(graw[c]), gm);
            if (RMS) {
                // Qwen2RMSNorm: weight * (x*rstd).to(input_dtype)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float n = v[c][e] * rstd;
                    if (sizeof(T) == 2) n = bf2f(f2bf(n));
                    o[e] = gm[e] * n;
                }
            } else {
                float bt[8];
                ld8_f<T>(beta + ch * 8, bt);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (v[c][e] - mean) * rstd * gm[e] + bt[e];
            }
            st8_f<T>(yr + ch * 8, o);
        }
    }
}

template <typename T, int CPL>
__global__ __launch_bounds__(256) void ln_merge_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                       const T* __restrict__ gamma, const T* __restrict__ beta,
                                                       int out_rows, int group, int H, float eps) {
    const int lane = threadIdx.x & 63;
    const int orow = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (orow >= out_rows) return;
    const int nch = H >> 3;
    // (loads as in norm_kernel, the next row of the group ahead of this one's sums)
    constexpr int V = sizeof(T) * 8 / 16;
    u32x4 raw[CPL][V], graw[CPL][V], braw[CPL][V];
    auto load = [&](u32x4 (&to)[CPL][V], const T* from) {
#pragma unroll
        for (int c = 0; c < CPL; ++c)
#pragma unroll
            for (int i = 0; i < V; ++i) to[c][i] = *(reinterpret_cast<const u32x4*>(from + min(lane + 64 * c, nch - 1) * 8) + i);
    };
    const T* xr = x + (long)orow * group * H;
    load(raw, xr);
    load(graw, gamma);
    load(braw, beta);
    float acc[CPL][8];
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[c][e] = 0.f;
    for (int gidx = 0; gidx < group; ++gidx) {
        float v[CPL][8];
        float sum = 0.f;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            ld8_f<T>(reinterpret_cast<const T*>(raw[c]), v[c]);
            if (lane + 64 * c < nch) {
#pragma unroll
                for (int e = 0; e < 8; ++e) sum += v[c][e];
            }
        }
        if (gidx + 1 < group) load(raw, xr + (long)(gidx + 1) * H);
        sum = wave_sum(sum);
        const float mean = sum / (float)H;
        float sq = 0.f;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (lane + 64 * c < nch) {
#pragma unroll
                for (int e = 0; e < 8; ++e) { const float d = v[c][e] - mean; sq += d * d; }
            }
        }
        sq = wave_sum(sq);
        const float rstd = rsqrtf(sq / (float)H + eps);
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (lane + 64 * c < nch) {
                float gm[8], bt[8];
                ld8_f<T>(reinterpret_cast<const T*>(graw[c]), gm);
                ld8_f<T>(reinterpret_cast<const T*>(braw[c]), bt);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float n = (v[c][e] - mean) * rstd * gm[e] + bt[e];
                    if (sizeof(T) == 2) n = bf2f(f2bf(n));  // post_layernorm output is stored in T
                    acc[c][e] += n;
                }
            }
        }
    }
    const float invg = 1.0f / (float)group;
    T* yr = y + (long)orow * H;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = lane + 64 * c;
        if (ch < nch) {
            float o[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = acc[c][e] * invg;
            st8_f<T>(yr + ch * 8, o);
        }
    }
}

template <typename T, bool RMS>
int launch_norm(hipStream_t st, const void* x, void* y, const void* g, const void* b, int rows, int H, float eps) {
    const int cpl = (H / 8 + 63) / 64;
    dim3 grid((rows + 3) / 4), blk(256);
#define COGS_NORM_CASE(C)                                                                             \
    hipLaunchKernelGGL((norm_kernel<T, C, RMS>), grid, blk, 0, st, (const T*)x, (T*)y, (const T*)g, \
                       (const T*)b, rows, H, eps)
    if (cpl <= 1) COGS_NORM_CASE(1);
    else if (cpl <= 2) COGS_NORM_CASE(2);
    else if (cpl <= 3) COGS_NORM_CASE(3);
    else if (cpl <= 4) COGS_NORM_CASE(4);
    else if (cpl <= 8) COGS_NORM_CASE(8);
    else return COGS_E_UNSUPPORTED;
#undef COGS_NORM_CASE
    return COGS_LAUNCH_CHECK();
}

template <typename T>
int launch_ln_merge(hipStream_t st, const void* x, void* y, const void* g, const void* b, int out_rows, int group,
                    int H, float eps) {
    const int cpl = (H / 8 + 63) / 64;
    dim3 grid((out_rows + 3) / 4), blk(256);
#define COGS_LNM_CASE(C)                                                                            \
    hipLaunchKernelGGL((ln_merge_kernel<T, C>), grid, blk, 0, st, (const T*)x, (T*)y, (const T*)g, \
                       (const T*)b, out_rows, group, H, eps)
    if (cpl <= 1) COGS_LNM_CASE(1);
    else if (cpl <= 2) COGS_LNM_CASE(2);
    else if (cpl <= 3) COGS_LNM_CASE(3);
    else if (cpl <= 4) COGS_LNM_CASE(4);
    else if (cpl <= 8) COGS_LNM_CASE(8);
    else return COGS_E_UNSUPPORTED;
#undef COGS_LNM_CASE
    return COGS_LAUNCH_CHECK();
}

// (a, b) = (rstd, -rstd * mean) of every row from the per-tile partial sums the producing GEMM's epilogue wrote
// (EPI_ROWSTAT). One wave a workgroup: latency, so the rows of a short clip are spread over as many CUs as there are.
__global__ __launch_bounds__(64) void ln_finalize_kernel(const float* __restrict__ part, int rows, int tiles, float inv_h,
                                                          float eps, float* __restrict__ ab) {
    const int r = blockIdx.x * 64 + threadIdx.x;
    if (r >= rows) return;
    *reinterpret_cast<f32x2*>(ab + 2 * (long)r) = ln_row_factors(reinterpret_cast<const f32x2*>(part) + (long)r * tiles, tiles, inv_h, eps);
}

// the sum of NP partial arrays at q, `step` apart: all loads out before the first addition
template <int NP>
__device__ __forceinline__ f32x4 sum_parts(const float* q, long step) {
    f32x4 part[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) part[s] = *reinterpret_cast<const f32x4*>(q + s * step);
#pragma unroll
    for (int s = 1; s < NP; ++s) part[0] += part[s];
    return part[0];
}
// four columns of a sublayer's output; PARTS: in partial sums
template <typename T, bool PARTS>
__device__ __forceinline__ f32x4 stream_y(const CogsStreamNorm& p, long row, int i) {
    if constexpr (!PARTS) return ld4_f<T>(reinterpret_cast<const T*>(p.y) + row * p.Hp + i);
    const float* q = reinterpret_cast<const float*>(p.y) + row * p.Hp + i;
    const long step = (long)p.rows * p.Hp;
    return p.y_parts == 2 ? sum_parts<2>(q, step) : p.y_parts == 4 ? sum_parts<4>(q, step) : sum_parts<8>(q, step);
}

// fp32 residual stream around a sublayer (kernels.h, CogsStreamNorm): one workgroup of TPB threads per row, the row in
// registers (C chunks of four columns per thread). Norms entirely in fp32, one rounding of the normed row.
template <typename T, int C, int TPB, bool PARTS>
__global__ __launch_bounds__(TPB) void stream_norm_kernel(CogsStreamNorm p) {
    constexpr int NW = TPB / 64;
    __shared__ float red[2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const long row = p.pick ? p.pick[blockIdx.x] : blockIdx.x;
    float* x = p.x + row * p.Hp;
    auto row_rstd = [&](float ss, int which) {
        ss = wave_sum(ss);
        if (lane == 0) red[which][wid] = ss;
        __syncthreads();
        ss = red[which][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) ss += red[which][w];
        return 1.f / sqrtf(ss / (float)p.H + p.eps);
    };
    f32x4 v[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = (tid + TPB * c) * 4;
        v[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (i < p.Hp) v[c] = p.embeds ? ld4_f<T>(reinterpret_cast<const T*>(p.embeds) + row * p.Hp + i) : *reinterpret_cast<const f32x4*>(x + i);
    }
    if (p.y) {
        f32x4 y[C];
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = (tid + TPB * c) * 4;
            y[c] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (i < p.Hp) y[c] = stream_y<T, PARTS>(p, row, i);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += y[c][e] * y[c][e];
        }
        if (p.y_gamma) {
            const float rs = row_rstd(ss, 0);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int i = (tid + TPB * c) * 4;
                if (i >= p.Hp) continue;
                const f32x4 g = *reinterpret_cast<const f32x4*>(p.y_gamma + i);
#pragma unroll
                for (int e = 0; e < 4; ++e) y[c][e] = y[c][e] * rs * g[e];
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) v[c] += y[c];
    }
    if (p.y || p.embeds) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = (tid + TPB * c) * 4;
            if (i < p.Hp) *reinterpret_cast<f32x4*>(x + i) = v[c];
        }
    }
    if (!p.out) return;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += v[c][e] * v[c][e];
    const float rs = row_rstd(ss, 1);
    T* o = reinterpret_cast<T*>(p.out) + (long)blockIdx.x * p.Hp;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = (tid + TPB * c) * 4;
        if (i >= p.Hp) continue;
        const f32x4 g = *reinterpret_cast<const f32x4*>(p.out_gamma + i);
        st4_f<T>(o + i, f32x4{v[c][0] * rs * g[0], v[c][1] * rs * g[1], v[c][2] * rs * g[2], v[c][3] * rs * g[3]});
    }
}

// Workgroups behind those of a mix of few rows: lines of the next product's weights into the L2 caches (kernels.h, CogsAhead). Such a mix is 4 us
// of latency on as many CUs as it has rows while HBM, which bounds the few-row product behind it (8 x 8192 x 2048: 8.0 us, 4.6 from L2), is
// idle. Workgroup i runs on XCD i % 8, here and there, so each reads the lines of the column groups that its own XCD will want. How many:
// cogs_k_gemm_skinny_ahead.
constexpr int AHEAD_CUS = 256;

int ahead_workgroups(const CogsAhead& p, int rows) { return p.lines > 0 && rows < AHEAD_CUS ? (AHEAD_CUS - rows) / 8 * 8 : 0; }

__device__ __forceinline__ void read_ahead(const CogsAhead& p, int rows) {
    const int xcd = blockIdx.x & 7, me = ((int)blockIdx.x - rows) >> 3, of = ((int)gridDim.x - rows) >> 3;
    const int total = ((p.groups - xcd + 7) >> 3) * p.cols * p.lines, step = of * (int)blockDim.x;
    for (int t = me * (int)blockDim.x + (int)threadIdx.x; t < total; t += step) {
        const int row = t / p.lines, n = ((row / p.cols) * 8 + xcd) * p.cols + row % p.cols;
        if (n >= p.N) continue;
        const int v = *reinterpret_cast<const int*>(p.W + n * p.ldw + (long)(t - row * p.lines) * 128);
        asm volatile("" ::"v"(v));
    }
}

// the same with a scaled embedding and a position table at the start and hyper-connected streams (x [row][stream][Hp]). NS: streams
// rounded up; a chunk's old streams are in registers together, only the combination that is normed stays there for the row.
template <typename T, int C, int TPB, int NS, bool PARTS>
__global__ __launch_bounds__(TPB) void stream_mix_kernel(CogsStreamNorm p) {
    if constexpr (TPB == 1024) {
        if ((int)blockIdx.x >= p.rows) {
            read_ahead(p.ahead, p.rows);
            return;
        }
    }
    constexpr int NW = TPB / 64;
    __shared__ float red[2][NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const long row = p.pick ? p.pick[blockIdx.x] : blockIdx.x;
    const int ns = p.streams > 0 ? p.streams : 1;
    float* x = p.x + row * ns * p.Hp;
    auto row_rstd = [&](float ss, int which) {
        ss = wave_sum(ss);
        if (lane == 0) red[which][wid] = ss;
        __syncthreads();
        ss = red[which][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) ss += red[which][w];
        return 1.f / sqrtf(ss / (float)p.H + p.eps);
    };
    f32x4 y[C], u[C];
    float rs = 1.f;
    // one chunk a thread (few rows): latency counts, so the streams, their weights and the gain are asked for in front of the sublayer's
    // output, whose partial sums would otherwise be waited for first (8 rows of 4 x 2048, eight partial sums: 5.2 -> 4.4 us)
    constexpr bool EARLY = C == 1, WEIGHTS = EARLY && NS <= 4;
    f32x4 early[EARLY ? NS : 1], gain = {0.f, 0.f, 0.f, 0.f};
    float mixw[WEIGHTS ? NS * NS : 1], outw[WEIGHTS ? NS : 1], inw[WEIGHTS ? NS : 1];
    auto read_stream = [&](int s, int i) { return *reinterpret_cast<const f32x4*>(x + (long)s * p.Hp + i); };
    if constexpr (EARLY) {
        const int i = tid * 4;
        if (i < p.Hp) {
            if (!p.embeds)
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    if (s < ns) early[s] = read_stream(s, i);
            if (p.out) gain = *reinterpret_cast<const f32x4*>(p.out_gamma + i);
        }
        if constexpr (WEIGHTS)
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s >= ns) continue;
                inw[s] = p.in_w ? p.in_w[s] : 1.f;
                if (!p.mix) continue;
                outw[s] = p.out_w[s];
#pragma unroll
                for (int t = 0; t < NS; ++t)
                    if (t < ns) mixw[s * NS + t] = p.mix[s * ns + t];
            }
    }
    auto mix_of = [&](int s, int t) { if constexpr (WEIGHTS) return mixw[s * NS + t]; else return p.mix[s * ns + t]; };
    auto out_of = [&](int t) { if constexpr (WEIGHTS) return outw[t]; else return p.out_w[t]; };
    auto in_of = [&](int s) { if constexpr (WEIGHTS) return inw[s]; else return p.in_w[s]; };
    if (p.y) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = (tid + TPB * c) * 4;
            y[c] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (i < p.Hp) y[c] = stream_y<T, PARTS>(p, row, i);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += y[c][e] * y[c][e];
        }
        if (p.y_gamma) rs = row_rstd(ss, 0);
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = (tid + TPB * c) * 4;
        u[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (i >= p.Hp) continue;
        f32x4 v[NS];
        if (p.embeds) {
            f32x4 e = ld4_f<T>(reinterpret_cast<const T*>(p.embeds) + row * p.Hp + i) * p.embed_scale;
            if (p.pos) e += ld4_f<T>(reinterpret_cast<const T*>(p.pos) + (long)p.rowpos[row] * p.Hp + i);
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = e;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (s < ns) v[s] = EARLY ? early[EARLY ? s : 0] : read_stream(s, i);
        }
        if (p.y) {
            f32x4 yv = y[c];
            if (p.y_gamma) yv *= rs * *reinterpret_cast<const f32x4*>(p.y_gamma + i);
            if (p.mix) {
                f32x4 w[NS];
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    if (t >= ns) continue;
                    w[t] = yv * out_of(t);
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        if (s < ns) w[t] += v[s] * mix_of(s, t);
                }
#pragma unroll
                for (int t = 0; t < NS; ++t)
                    if (t < ns) v[t] = w[t];
            } else {
                v[0] += yv;
            }
        }
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s >= ns) continue;
            if (p.y || p.embeds) *reinterpret_cast<f32x4*>(x + (long)s * p.Hp + i) = v[s];
            sum += v[s];
            u[c] += p.in_w ? v[s] * in_of(s) : v[s];
        }
        if (p.sum) *reinterpret_cast<f32x4*>(p.sum + row * p.Hp + i) = sum;
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += u[c][e] * u[c][e];
    }
    if (!p.out) return;
    rs = row_rstd(ss, 1);
    T* o = reinterpret_cast<T*>(p.out) + (long)blockIdx.x * p.Hp;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = (tid + TPB * c) * 4;
        if (i >= p.Hp) continue;
        st4_f<T>(o + i, u[c] * rs * (EARLY ? gain : *reinterpret_cast<const f32x4*>(p.out_gamma + i)));
    }
}

// Many rows: HBM. A mix reads and writes every stream (4 x fp32) for one sublayer output of 16 bits, so it need not be done at once: what the next
// sublayer reads is formed from the streams as they were and the outputs since, each mix in its turn with the arithmetic and the order of
// stream_mix_kernel (the same bits), and only the COGS_CHAIN-th output has the streams written. The first ones start from the embeddings, one
// 16-bit row for all streams, and the last ones are mixed for the rows that are asked for alone. 4096 rows of 4 x 2048, us (stream_mix_kernel
// 66 each): 26, 27, 36, 53 from the embeddings, then 38, 37, 42, 61 in turn; 1109 -> 634 in a prompt of 16 sublayers. (A number of streams that is
// not the template's made it 760, predicates and scalar loads one by one; rows walked by fewer workgroups 907. Longer chains cost what they save:
// 20 multiplications an element and output.) Up to 64 wanted rows of more than 1024 columns are latency: 1024 threads each as in stream_mix_kernel, so
// that a row's sum is that of a row mixed at once, and beside them the head's weights are read ahead.
template <typename T, int C, int NS, int TPB>
__global__ __launch_bounds__(TPB) void stream_chain_kernel(CogsStreamChain p) {
    if constexpr (TPB == 1024) {
        if ((int)blockIdx.x >= p.rows) {
            read_ahead(p.ahead, p.rows);
            return;
        }
    }
    typedef T raw_t __attribute__((ext_vector_type(4)));
    __shared__ float red[TPB / 64];
    const int tid = threadIdx.x;
    const long row = p.pick ? p.pick[blockIdx.x] : blockIdx.x;
    float* x = p.x + row * NS * p.Hp;
    int at[C];
#pragma unroll
    for (int c = 0; c < C; ++c) at[c] = min((tid + TPB * c) * 4, p.Hp - 4);
    f32x4 v[C][NS];
    raw_t y[COGS_CHAIN][C];
    if (p.embeds) {
        const T* pos = p.pos ? reinterpret_cast<const T*>(p.pos) + (long)p.rowpos[row] * p.Hp : nullptr;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            f32x4 e = ld4_f<T>(reinterpret_cast<const T*>(p.embeds) + row * p.Hp + at[c]) * p.embed_scale;
            if (pos) e += ld4_f<T>(pos + at[c]);
#pragma unroll
            for (int s = 0; s < NS; ++s) v[c][s] = e;
        }
    } else {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int s = 0; s < NS; ++s) v[c][s] = *reinterpret_cast<const f32x4*>(x + (long)s * p.Hp + at[c]);
    }
#pragma unroll
    for (int q = 0; q < COGS_CHAIN; ++q)
        if (q < p.n)
#pragma unroll
            for (int c = 0; c < C; ++c) y[q][c] = *reinterpret_cast<const raw_t*>(reinterpret_cast<const T*>(p.outs[q].y) + row * p.Hp + at[c]);
#pragma unroll
    for (int q = 0; q < COGS_CHAIN; ++q) {
        if (q >= p.n) continue;
        float mix[NS * NS], out_w[NS];
#pragma unroll
        for (int s = 0; s < NS * NS; ++s) mix[s] = p.outs[q].mix[s];
#pragma unroll
        for (int s = 0; s < NS; ++s) out_w[s] = p.outs[q].out_w[s];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const f32x4 yv = ld4_f<T>(reinterpret_cast<const T*>(&y[q][c]));
            f32x4 w[NS];
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                w[t] = yv * out_w[t];
#pragma unroll
                for (int s = 0; s < NS; ++s) w[t] += v[c][s] * mix[s * NS + t];
            }
#pragma unroll
            for (int t = 0; t < NS; ++t) v[c][t] = w[t];
        }
    }
    f32x4 u[C];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        u[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if ((tid + TPB * c) * 4 >= p.Hp) continue;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (p.store) *reinterpret_cast<f32x4*>(x + (long)s * p.Hp + at[c]) = v[c][s];
            u[c] += p.in_w ? v[c][s] * p.in_w[s] : v[c][s];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += u[c][e] * u[c][e];
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = red[0];
#pragma unroll
    for (int w = 1; w < TPB / 64; ++w) ss += red[w];
    const float rs = 1.f / sqrtf(ss / (float)p.H + p.eps);
    T* o = reinterpret_cast<T*>(p.out) + (long)blockIdx.x * p.Hp;
#pragma unroll
    for (int c = 0; c < C; ++c)
        if ((tid + TPB * c) * 4 < p.Hp) st4_f<T>(o + at[c], u[c] * rs * *reinterpret_cast<const f32x4*>(p.out_gamma + at[c]));
}

template <typename T>
int launch_stream_chain(hipStream_t st, const CogsStreamChain& a) {
    const bool few = a.rows <= 64 && a.Hp > 1024;
    const int more = few ? ahead_workgroups(a.ahead, a.rows) : 0;
#define COGS_CHAIN_CASE(C, NS, TPB) hipLaunchKernelGGL((stream_chain_kernel<T, C, NS, TPB>), dim3(a.rows + more), dim3(TPB), 0, st, a)
#define COGS_CHAIN_STREAMS(NS)                      \
    case NS:                                        \
        if (few) COGS_CHAIN_CASE(1, NS, 1024);      \
        else if (a.Hp <= 2048) COGS_CHAIN_CASE(2, NS, 256); \
        else COGS_CHAIN_CASE(4, NS, 256);           \
        break;
    switch (a.streams) {
        COGS_CHAIN_STREAMS(2)
        COGS_CHAIN_STREAMS(3)
        COGS_CHAIN_STREAMS(4)
    }
#undef COGS_CHAIN_STREAMS
#undef COGS_CHAIN_CASE
    return COGS_LAUNCH_CHECK();
}

template <typename T, int NS>
int launch_stream_mix(hipStream_t st, const CogsStreamNorm& a) {
    const int rows = a.rows, more = ahead_workgroups(a.ahead, rows);
#define COGS_STREAM(C, TPB) hipLaunchKernelGGL((stream_mix_kernel<T, C, TPB, NS, false>), dim3(rows + (TPB == 1024 ? more : 0)), dim3(TPB), 0, st, a)
// (partial sums come of products of at most 64 rows)
#define COGS_STREAM_FEW(C, TPB)                                                                                                     \
    do {                                                                                                                            \
        if (a.y_parts > 0) hipLaunchKernelGGL((stream_mix_kernel<T, C, TPB, NS, true>), dim3(rows + (TPB == 1024 ? more : 0)), dim3(TPB), 0, st, a); \
        else COGS_STREAM(C, TPB);                                                                                                   \
    } while (0)
    if (a.rows <= 64 && a.Hp > 1024) {
        if (a.Hp <= 4096) COGS_STREAM_FEW(1, 1024);
        else if (a.Hp <= 16384) COGS_STREAM_FEW(4, 1024);
        else return COGS_E_UNSUPPORTED;
    } else if (a.Hp <= 1024) COGS_STREAM_FEW(1, 256);
    else if (a.y_parts > 0) return COGS_E_UNSUPPORTED;
    else if (a.Hp <= 4096) COGS_STREAM(4, 256);
    else if (a.Hp <= 16384) COGS_STREAM(16, 256);
    else return COGS_E_UNSUPPORTED;
#undef COGS_STREAM_FEW
#undef COGS_STREAM
    return COGS_LAUNCH_CHECK();
}

template <typename T>
int launch_stream_norm(hipStream_t st, const CogsStreamNorm& a) {
    if (a.streams > 0 || a.pos || a.embed_scale != 1.f || a.sum) {
        if (a.streams <= 1) return launch_stream_mix<T, 1>(st, a);
        if (a.streams <= 2) return launch_stream_mix<T, 2>(st, a);
        if (a.streams <= 4) return launch_stream_mix<T, 4>(st, a);
        if (a.streams <= 8) return launch_stream_mix<T, 8>(st, a);
        if (a.streams <= 16) return launch_stream_mix<T, 16>(st, a);
        return COGS_E_UNSUPPORTED;
    }
    const dim3 grid(a.rows);
#define COGS_STREAM(C, TPB) hipLaunchKernelGGL((stream_norm_kernel<T, C, TPB, false>), grid, dim3(TPB), 0, st, a)
#define COGS_STREAM_FEW(C, TPB)                                                                                                     \
    do {                                                                                                                            \
        if (a.y_parts > 0) hipLaunchKernelGGL((stream_norm_kernel<T, C, TPB, true>), grid, dim3(TPB), 0, st, a);                    \
        else COGS_STREAM(C, TPB);                                                                                                   \
    } while (0)
    if (a.rows <= 64 && a.Hp > 1024) {           // few rows: latency, not bandwidth -- more threads on each
        if (a.Hp <= 4096) COGS_STREAM_FEW(1, 1024);
        else if (a.Hp <= 8192) COGS_STREAM_FEW(2, 1024);
        else if (a.Hp <= 16384) COGS_STREAM_FEW(4, 1024);
        else return COGS_E_UNSUPPORTED;
    } else if (a.Hp <= 1024) COGS_STREAM_FEW(1, 256);
    else if (a.y_parts > 0) return COGS_E_UNSUPPORTED;
    else if (a.Hp <= 2048) COGS_STREAM(2, 256);
    else if (a.Hp <= 4096) COGS_STREAM(4, 256);
    else if (a.Hp <= 8192) COGS_STREAM(8, 256);
    else if (a.Hp <= 16384) COGS_STREAM(16, 256);
    else return COGS_E_UNSUPPORTED;
#undef COGS_STREAM_FEW
#undef COGS_STREAM
    return COGS_LAUNCH_CHECK();
}

}  // namespace

int cogs_k_stream_norm(hipStream_t st, int dtype, const CogsStreamNorm& a) {
    if (a.rows <= 0) return COGS_OK;
    if ((a.pos && !a.rowpos) || (a.y && a.streams > 0 && (!a.mix || !a.out_w)) || (a.streams <= 0 && (a.mix || a.in_w))) return COGS_E_INVALID;
    if (a.y_parts != 0 && a.y_parts != 2 && a.y_parts != 4 && a.y_parts != 8) return COGS_E_INVALID;
    if (!a.x || a.Hp % 4 || a.H <= 0 || a.H > a.Hp || (a.out && !a.out_gamma) || (a.pick && (!a.out || a.y || a.embeds))) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_stream_norm<bf16_t>(st, a) : launch_stream_norm<float>(st, a);
}

// more than 64 rows: fewer are latency (their own kernel, which reads weights ahead). The row is in the registers of 256 or 1024 threads: up to 4096 columns
bool cogs_k_stream_chain_fits(int streams, int Hp, int rows) { return streams >= 2 && streams <= 4 && Hp <= 4096 && rows > 64; }

int cogs_k_stream_chain(hipStream_t st, int dtype, const CogsStreamChain& a) {
    if (a.rows <= 0) return COGS_OK;
    if (a.streams < 2 || a.streams > 4 || a.Hp > 4096 || a.Hp % 4 || a.H <= 0 || a.H > a.Hp || a.n < 0 || a.n > COGS_CHAIN) return COGS_E_INVALID;
    if (!a.x || !a.out || !a.out_gamma || (a.pos && !a.rowpos) || (a.pick && a.store) || a.y || a.sum) return COGS_E_INVALID;
    for (int q = 0; q < a.n; ++q)
        if (!a.outs[q].y || !a.outs[q].mix || !a.outs[q].out_w) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_stream_chain<bf16_t>(st, a) : launch_stream_chain<float>(st, a);
}

int cogs_k_layernorm(hipStream_t st, int dtype, const void* x, void* y, const void* gamma, const void* beta,
                     int rows, int H, float eps) {
    if (rows <= 0) return COGS_OK;
    if (H % 8) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_norm<bf16_t, false>(st, x, y, gamma, beta, rows, H, eps)
                                 : launch_norm<float, false>(st, x, y, gamma, beta, rows, H, eps);
}

int cogs_k_rmsnorm(hipStream_t st, int dtype, const void* x, void* y, const void* gamma, int rows, int H, float eps) {
    if (rows <= 0) return COGS_OK;
    if (H % 8) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_norm<bf16_t, true>(st, x, y, gamma, nullptr, rows, H, eps)
                                 : launch_norm<float, true>(st, x, y, gamma, nullptr, rows, H, eps);
}

int cogs_k_ln_merge(hipStream_t st, int dtype, const void* x, void* y, const void* gamma, const void* beta,
                    int out_rows, int group, int H, float eps) {
    if (out_rows <= 0) return COGS_OK;
    if (H % 8 || group <= 0) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_ln_merge<bf16_t>(st, x, y, gamma, beta, out_rows, group, H, eps)
                                 : launch_ln_merge<float>(st, x, y, gamma, beta, out_rows, group, H, eps);
}

int cogs_k_ln_finalize(hipStream_t st, const float* stat_part, int rows, int tiles, int H, float eps, float* ab) {
    if (rows <= 0 || tiles <= 0 || H <= 0) return COGS_E_INVALID;
    hipLaunchKernelGGL(ln_finalize_kernel, dim3((rows + 63) / 64), dim3(64), 0, st, stat_part, rows, tiles, 1.0f / (float)H,
                       eps, ab);
    return COGS_LAUNCH_CHECK();
}
