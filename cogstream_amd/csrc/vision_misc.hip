// Small HBM-bound helpers around the ViT encoder: patch-row packing and rotary tables.
//
//   pack_rows     pixel_values [N,588] (fp32 or bf16) -> compute dtype, K padded to a multiple of
//                 the GEMM slab (640) so that patch-embed (nn.Conv2d k=s=14,
//                 model/modeling_videollama3_encoder.py:194-210) is a plain row-major GEMM.
//   vit_rope      cos/sin of the 2-D rotary angles in merge-window row order
//                 (rot_pos_emb, model/modeling_videollama3_encoder.py:405-434; VisionRotaryEmbedding
//                 :173-183): row r of a frame -> window r/ms^2, (dy,dx) inside it; angles are
//                 [h*inv_freq[0..n), w*inv_freq[0..n)].
//   llm_rope_table cos/sin(pos * inv_freq) for Qwen2 (theta 1e6, rotate_half pairs d, d+hd/2).
#include "common.h"
#include "kernels.h"

namespace {

template <typename TI, typename TO>
__device__ __forceinline__ void pack_rows(const TI* __restrict__ in, long ld_in, TO* __restrict__ out, long ld_out, int rows, int cols_in, int cols_out,
                                          int block, int blocks) {
    const int cpr = cols_out >> 2;  // 4-element groups per output row
    const long total = (long)rows * cpr;
    for (long i = (long)block * 256 + threadIdx.x; i < total; i += (long)blocks * 256) {
        const long r = i / cpr;
        const int c = (int)(i % cpr) * 4;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (c + 3 < cols_in) {
            v = ld4_f<TI>(in + r * ld_in + c);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < cols_in) v[e] = ld_f<TI>(in + r * ld_in + c + e);
        }
        st4_f<TO>(out + r * ld_out + c, v);
    }
}
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void pack_rows_kernel(const TI* __restrict__ in, long ld_in, TO* __restrict__ out,
                                                        long ld_out, int rows, int cols_in, int cols_out) {
    pack_rows<TI, TO>(in, ld_in, out, ld_out, rows, cols_in, cols_out, blockIdx.x, gridDim.x);
}

__device__ __forceinline__ void vit_rope(float* cos_t, float* sin_t, int row0, int t, int gh, int gw, int ms, const float* inv_freq, int nf,
                                         int block, int blocks) {
    const int per_frame = gh * gw;
    const long total = (long)t * per_frame * 2 * nf;
    const int wpr = gw / ms;  // merge windows per row
    for (long i = (long)block * 256 + threadIdx.x; i < total; i += (long)blocks * 256) {
        const int f = (int)(i % (2 * nf));
        const long row = i / (2 * nf);
        const int r = (int)(row % per_frame);
        const int win = r / (ms * ms), in = r % (ms * ms);
        const int hpos = (win / wpr) * ms + in / ms;
        const int wpos = (win % wpr) * ms + in % ms;
        const float ang = (f < nf) ? (float)hpos * inv_freq[f] : (float)wpos * inv_freq[f - nf];
        const long o = ((long)row0 + row) * (2 * nf) + f;
        if (sin_t) { cos_t[o] = cosf(ang); sin_t[o] = sinf(ang); }
        else { cos_t[2 * o] = cosf(ang); cos_t[2 * o + 1] = sinf(ang); }   // interleaved (cos, sin)
    }
}

// (cos, sin) of pos * inv_freq[f] for pos < maxpos: lut[pos][f][2]; the SAME expression as vit_rope, so a
// GEMM tile that reads the LUT and one that reads the per-row table see bit-identical factors
__device__ __forceinline__ void vit_rope_lut(float* lut, int maxpos, const float* inv_freq, int nf, int block, int blocks) {
    const int total = maxpos * nf;
    for (int i = block * 256 + threadIdx.x; i < total; i += blocks * 256) {
        const int f = i % nf, pos = i / nf;
        const float ang = (float)pos * inv_freq[f];
        lut[2 * i] = cosf(ang);
        lut[2 * i + 1] = sinf(ang);
    }
}

__global__ __launch_bounds__(256) void llm_rope_kernel(float* cos_t, float* sin_t, const int* pos, int pos0, int rows,
                                                       const float* inv_freq, int nf) {
    const long total = (long)rows * nf;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const int f = (int)(i % nf);
        const int r = (int)(i / nf);
        const int pp = pos ? pos[r] : pos0 + r;
        const float ang = (float)pp * inv_freq[f];
        if (sin_t) { cos_t[i] = cosf(ang); sin_t[i] = sinf(ang); }
        else { cos_t[2 * i] = cosf(ang); cos_t[2 * i + 1] = sinf(ang); }   // interleaved (cos, sin)
    }
}

// cu_seqlens (modeling_videollama3_encoder.py:439-440) of one video, frame f of which has rows [row0 + f*per, row0 + (f+1)*per), and for
// every row its position (h | w << 16) in the order of vit_rope, or its frame's rows (eager-global mode)
__device__ __forceinline__ void vit_rows(const CogsVitTables& p, int block, int blocks) {
    const int per = p.gh * p.gw, wpr = p.gw / p.ms;
    const long total = (long)p.t * per, i0 = (long)block * 256 + threadIdx.x, stride = (long)blocks * 256;
    for (long i = i0; i <= p.t; i += stride)
        if (i > 0 || p.frame0 == 0) p.cu[p.frame0 + i] = p.row0 + (int)i * per;
    for (long i = i0; i < total; i += stride) {
        const int f = (int)(i / per);
        if (p.rowpos) {
            const int r = (int)(i - (long)f * per), win = r / (p.ms * p.ms), in = r % (p.ms * p.ms);
            p.rowpos[p.row0 + i] = ((win / wpr) * p.ms + in / p.ms) | (((win % wpr) * p.ms + in % p.ms) << 16);
        }
        if (p.lo) {
            p.lo[p.row0 + i] = p.row0 + f * per;
            p.hi[p.row0 + i] = p.row0 + (f + 1) * per;
        }
    }
}

// All that an encode needs of a video's grid, and the patches' rows: none of it waits for anything else of it. As five launches of 1.4 to 5 us, one
// behind the other, they were 13 us of an encode's start: one image of 224 x 224 1317 -> 1310 us, 8 frames 2995 -> 2987
struct VitSetup { int rows, lut, rope; long pack_ld_in, pack_ld_out; int pack_rows, cols_in, cols_out; };      // workgroups of each; the rest pack
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void vit_setup_kernel(CogsVitTables p, VitSetup g, const TI* __restrict__ in, TO* __restrict__ out) {
    int b = blockIdx.x;
    if (b < g.rope) return vit_rope(p.cos_t, p.sin_t, p.row0, p.t, p.gh, p.gw, p.ms, p.inv_freq, p.nf, b, g.rope);
    b -= g.rope;
    if (b < g.rows) return vit_rows(p, b, g.rows);
    b -= g.rows;
    if (b < g.lut) return vit_rope_lut(p.lut, p.maxpos, p.inv_freq, p.nf, b, g.lut);
    pack_rows<TI, TO>(in, g.pack_ld_in, out, g.pack_ld_out, g.pack_rows, g.cols_in, g.cols_out, b - g.lut, gridDim.x - g.rope - g.rows - g.lut);
}

// positions restart at every segment: pos[i] = i - cu[s] for cu[s] <= i < cu[s+1]; one workgroup per segment
__global__ __launch_bounds__(256) void seg_positions_kernel(const int* __restrict__ cu, int* __restrict__ pos) {
    const int b = cu[blockIdx.x], e = cu[blockIdx.x + 1];
    for (int i = b + threadIdx.x; i < e; i += 256) pos[i] = i - b;
}

inline int grid_for(long total) {
    long g = (total + 255) / 256;
    return (int)(g < 1 ? 1 : (g > 4096 ? 4096 : g));
}

}  // namespace

int cogs_k_pack_rows(hipStream_t st, int in_dtype, int out_dtype, const void* in, long ld_in, void* out, long ld_out,
                     int rows, int cols_in, int cols_out) {
    if (rows <= 0) return COGS_OK;
    if (cols_out % 4 || cols_in > cols_out || ld_in % 4 || ld_out % 4) return COGS_E_INVALID;
    const int g = grid_for((long)rows * (cols_out / 4));
    if (in_dtype == COGS_DT_F32 && out_dtype == COGS_DT_BF16)
        hipLaunchKernelGGL((pack_rows_kernel<float, bf16_t>), dim3(g), dim3(256), 0, st, (const float*)in, ld_in,
                           (bf16_t*)out, ld_out, rows, cols_in, cols_out);
    else if (in_dtype == COGS_DT_BF16 && out_dtype == COGS_DT_BF16)
        hipLaunchKernelGGL((pack_rows_kernel<bf16_t, bf16_t>), dim3(g), dim3(256), 0, st, (const bf16_t*)in, ld_in,
                           (bf16_t*)out, ld_out, rows, cols_in, cols_out);
    else if (in_dtype == COGS_DT_F32 && out_dtype == COGS_DT_F32)
        hipLaunchKernelGGL((pack_rows_kernel<float, float>), dim3(g), dim3(256), 0, st, (const float*)in, ld_in,
                           (float*)out, ld_out, rows, cols_in, cols_out);
    else if (in_dtype == COGS_DT_BF16 && out_dtype == COGS_DT_F32)
        hipLaunchKernelGGL((pack_rows_kernel<bf16_t, float>), dim3(g), dim3(256), 0, st, (const bf16_t*)in, ld_in,
                           (float*)out, ld_out, rows, cols_in, cols_out);
    else
        return COGS_E_INVALID;
    return COGS_LAUNCH_CHECK();
}

// ... rows > 0: the patches of all videos are packed beside the tables of this one
int cogs_k_vit_setup(hipStream_t st, const CogsVitTables& p, int in_dtype, int out_dtype, const void* in, long ld_in, void* out, long ld_out, int rows,
                     int cols_in, int cols_out) {
    if (p.t <= 0 || p.gh <= 0 || p.gw <= 0 || p.ms <= 0 || p.gh % p.ms || p.gw % p.ms || !p.cu) return COGS_E_INVALID;
    if (rows > 0 && (cols_out % 4 || cols_in > cols_out || ld_in % 4 || ld_out % 4)) return COGS_E_INVALID;
    const long n = (long)p.t * p.gh * p.gw;
    VitSetup g{};
    g.rope = grid_for(n * 2 * p.nf);
    g.rows = p.rowpos || p.lo ? grid_for(n) : grid_for(p.t + 1);
    g.lut = p.lut ? grid_for((long)p.maxpos * p.nf) : 0;
    g.pack_ld_in = ld_in; g.pack_ld_out = ld_out; g.pack_rows = rows; g.cols_in = cols_in; g.cols_out = cols_out;
    const dim3 grid(g.rope + g.rows + g.lut + (rows > 0 ? grid_for((long)rows * (cols_out / 4)) : 0));
    const bool fi = in_dtype == COGS_DT_F32, fo = out_dtype == COGS_DT_F32;
    if ((!fi && in_dtype != COGS_DT_BF16) || (!fo && out_dtype != COGS_DT_BF16)) return COGS_E_INVALID;
#define COGS_SETUP(TI, TO) hipLaunchKernelGGL((vit_setup_kernel<TI, TO>), grid, dim3(256), 0, st, p, g, (const TI*)in, (TO*)out)
    if (fi && fo) COGS_SETUP(float, float);
    else if (fi) COGS_SETUP(float, bf16_t);
    else if (fo) COGS_SETUP(bf16_t, float);
    else COGS_SETUP(bf16_t, bf16_t);
#undef COGS_SETUP
    return COGS_LAUNCH_CHECK();
}

int cogs_k_seg_positions(hipStream_t st, const int* cu, int nseg, int* pos) {
    if (nseg <= 0) return COGS_OK;
    hipLaunchKernelGGL(seg_positions_kernel, dim3(nseg), dim3(256), 0, st, cu, pos);
    return COGS_LAUNCH_CHECK();
}

int cogs_k_llm_rope_table(hipStream_t st, float* cos_t, float* sin_t, const int* pos, int pos0, int rows,
                          const float* inv_freq, int n_freq) {
    if (rows <= 0) return COGS_OK;
    hipLaunchKernelGGL(llm_rope_kernel, dim3(grid_for((long)rows * n_freq)), dim3(256), 0, st, cos_t, sin_t, pos, pos0,
                       rows, inv_freq, n_freq);
    return COGS_LAUNCH_CHECK();
}
