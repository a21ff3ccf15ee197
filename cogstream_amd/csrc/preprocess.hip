// GPU pre-processing: uint8 frames -> Pillow-exact bicubic resize -> x/255,
// (x-0.5)/0.5 -> merge-window-major [N,588] patch rows, written straight in the encoder's input dtype.
//
// Replaces Videollama3ImageProcessor._preprocess (model/image_processing_videollama3.py:235-347): PIL
// Image.resize(BICUBIC) + rescale + normalize + the reshape/transpose patchify (:326-345). The resample is
// Pillow's fixed-point algorithm restated exactly (two passes, horizontal first, 22-bit integer coefficients
// built on the host by cogstream_amd.processing.resample_coeffs, uint8 rounding after each pass), so the uint8
// image -- and, through the [3,256] value table (processing.pixel_value_table), pixel_values -- is bit-identical to the reference's host path.
// One kernel does both passes tile by tile; the two-pass kernels remain for shrinking by so much that a tile's intermediate rows
// do not fit the LDS, and for outputs that are not aligned to a pair of elements.
#include "common.h"
#include "kernels.h"

namespace {

constexpr int PBITS = 22;

__device__ __forceinline__ int clip8(int v) { return v < 0 ? 0 : (v > 255 ? 255 : v); }

// horizontal pass: one thread per (image row, output column), 3 channels
__global__ __launch_bounds__(256) void resize_h_kernel(const uint8_t* __restrict__ in, uint8_t* __restrict__ tmp,
                                                       long rows, int W, int TW, const int* __restrict__ bounds,
                                                       const int* __restrict__ kk, int ksize) {
    const long total = rows * TW;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long row = i / TW;
        const int xx = (int)(i % TW);
        const int x0 = bounds[2 * xx], n = bounds[2 * xx + 1];
        const uint8_t* p = in + (row * W + x0) * 3;
        const int* k = kk + (long)xx * ksize;
        int s0 = 1 << (PBITS - 1), s1 = s0, s2 = s0;
        for (int x = 0; x < n; ++x) {
            const int c = k[x];
            s0 += p[3 * x] * c;
            s1 += p[3 * x + 1] * c;
            s2 += p[3 * x + 2] * c;
        }
        uint8_t* o = tmp + i * 3;
        o[0] = (uint8_t)clip8(s0 >> PBITS);
        o[1] = (uint8_t)clip8(s1 >> PBITS);
        o[2] = (uint8_t)clip8(s2 >> PBITS);
    }
}

// vertical pass + rescale/normalise + patchify: one thread per output element (element index fastest)
template <typename TO>
__global__ __launch_bounds__(256) void resize_v_patchify_kernel(const uint8_t* __restrict__ tmp, TO* __restrict__ out,
                                                                int T, int H, int TW, int gh, int gw, int ms,
                                                                const int* __restrict__ bounds,
                                                                const int* __restrict__ kk, int ksize,
                                                                const float* __restrict__ table) {
    const int per_frame = gh * gw;
    const long total = (long)T * per_frame * 588;
    const int wpr = gw / ms;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long r = i / 588;
        const int e = (int)(i % 588);
        const int c = e / 196, py = (e % 196) / 14, px = e % 14;
        const int f = (int)(r / per_frame), rr = (int)(r % per_frame);
        const int win = rr / (ms * ms), inw = rr % (ms * ms);
        const int prow = (win / wpr) * ms + inw / ms, pcol = (win % wpr) * ms + inw % ms;
        const int y = prow * 14 + py, x = pcol * 14 + px;
        const int y0 = bounds[2 * y], n = bounds[2 * y + 1];
        const uint8_t* p = tmp + (((long)f * H + y0) * TW + x) * 3 + c;
        const int* k = kk + (long)y * ksize;
        int s = 1 << (PBITS - 1);
        for (int j = 0; j < n; ++j) s += p[(long)j * TW * 3] * k[j];
        // rescale + normalise through the host-built per-channel byte table (reference arithmetic, exact)
        st_f<TO>(out + i, table[c * 256 + clip8(s >> PBITS)]);
    }
}

// ---- both passes of one tile: a band of 14 or 28 output rows by up to TILE_P patches of 14 columns ---------------------------
// The horizontal pass leaves the tile's intermediate rows in LDS, one plane per channel; the vertical pass reads them from there
// and writes pixel_values, so the frames are read once (a tenth more for the bands' and tiles' overlap) and nothing else goes
// through memory. Horizontal: a thread keeps one output column, its taps in registers, and walks the rows; the 12 bytes of four
// taps are one unaligned load. Vertical: a lane owns two neighbouring columns of a patch row -- the order of the output, so that
// 98 lanes write 392 contiguous bytes -- and takes the three channels together, one tap at a time.
// Bound by integer arithmetic (two instructions a product; the 22-bit taps leave no packed form) and byte traffic in LDS:
// 64 frames 480 x 854 -> 308 x 588 in 102 us (1.5 TB/s of
// frames and pixel_values); the two-pass kernels, a byte load per product, took 447.
constexpr int TILE_P = 6, TILE_C = 14 * TILE_P;
struct Bytes12 { unsigned w[3]; };

// NG groups of four taps in registers (taps past ksize are zero)
template <typename TO, int NG>
__global__ __launch_bounds__(256) void resize_patchify_kernel(const uint8_t* __restrict__ in, TO* __restrict__ out, int T, int H, int W, int gh, int gw,
                                                              int ms, int band_p, int max_rows, const int* __restrict__ bx, const int* __restrict__ kx,
                                                              int ksx, const int* __restrict__ by, const int* __restrict__ ky, int ksy,
                                                              const float* __restrict__ table) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int band = 14 * band_p, cols_pad = TILE_C;
    float* const lut = reinterpret_cast<float*>(smem);                           // [3][256]
    int* const rows_lo = reinterpret_cast<int*>(smem) + 768;                     // [band][2]: first row, taps
    int* const rows_k = rows_lo + 2 * band;                                      // [band][ksy]
    uint8_t* const mid = reinterpret_cast<uint8_t*>(rows_k + band * ksy);        // [3][max_rows][TILE_C]
    const int tid = threadIdx.x;
    const int tiles_x = (gw + TILE_P - 1) / TILE_P, bands = gh / band_p;
    const int tx = blockIdx.x % tiles_x, bd = blockIdx.x / tiles_x % bands, f = blockIdx.x / tiles_x / bands;
    const int p0 = tx * TILE_P, np = min(TILE_P, gw - p0), cols = 14 * np, y_first = bd * band;
    for (int i = tid; i < 768; i += 256) lut[i] = table[i];
    for (int i = tid; i < 2 * band; i += 256) rows_lo[i] = by[2 * y_first + i];
    for (int i = tid; i < band * ksy; i += 256) rows_k[i] = ky[(long)y_first * ksy + i];
    const int r0 = by[2 * y_first], last = y_first + band - 1;
    const int nrows = min(by[2 * last] + by[2 * last + 1] - r0, max_rows);

    const int plane = max_rows * cols_pad;
    const int col = tid % cols, group = tid / cols, groups = 256 / cols;
    if (group < groups) {
        const int xx = p0 * 14 + col, x0 = bx[2 * xx];
        int k[4 * NG];
#pragma unroll
        for (int t = 0; t < 4 * NG; ++t) k[t] = t < ksx ? kx[(long)xx * ksx + t] : 0;
        const uint8_t* const end = in + (long)T * H * W * 3;
        const uint8_t* p = in + (((long)f * H + r0 + group) * W + x0) * 3;
        uint8_t* o = mid + group * cols_pad + col;
        for (int r = group; r < nrows; r += groups, p += (long)groups * W * 3, o += groups * cols_pad) {
            Bytes12 b[NG];
            if (p + 12 * NG <= end) {
#pragma unroll
                for (int g = 0; g < NG; ++g) __builtin_memcpy(&b[g], p + 12 * g, 12);
            } else {                                                            // the clip's last bytes: no load past them
#pragma unroll
                for (int g = 0; g < NG; ++g)
#pragma unroll
                    for (int w = 0; w < 3; ++w) {
                        unsigned v = 0;
                        for (int e = 0; e < 4; ++e) v |= (p + 12 * g + 4 * w + e < end ? (unsigned)p[12 * g + 4 * w + e] : 0u) << (8 * e);
                        b[g].w[w] = v;
                    }
            }
            int s[3] = {1 << (PBITS - 1), 1 << (PBITS - 1), 1 << (PBITS - 1)};
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int e = 0; e < 12; ++e) s[e % 3] += __mul24((int)((b[g].w[e / 4] >> (8 * (e % 4))) & 255u), k[4 * g + e / 3]);
#pragma unroll
            for (int c = 0; c < 3; ++c) o[c * plane] = (uint8_t)clip8(s[c] >> PBITS);
        }
    }
    __syncthreads();

    const int per_patch = 14 * 7, wpr = gw / ms;
    for (int i = tid; i < band_p * np * per_patch; i += 256) {
        const int patch = i / per_patch, e = i % per_patch, py = e / 7, px = 2 * (e % 7);
        const int pr = patch / np, pc = patch % np, y = pr * 14 + py;
        const int n = rows_lo[2 * y + 1], from = rows_lo[2 * y] - r0;
        const uint8_t* q = mid + from * cols_pad + pc * 14 + px;
        const int* k = rows_k + y * ksy;
        int s[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) s[c] = 1 << (PBITS - 1);
        for (int j = 0; j < n && from + j < max_rows; ++j, q += cols_pad) {
            const int kj = k[j];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const unsigned two = *reinterpret_cast<const uint16_t*>(q + c * plane);
                s[2 * c] += __mul24((int)(two & 255u), kj);
                s[2 * c + 1] += __mul24((int)(two >> 8), kj);
            }
        }
        const int prow = bd * band_p + pr, pcol = p0 + pc;
        const long row = (long)f * gh * gw + ((prow / ms) * wpr + pcol / ms) * (ms * ms) + (prow % ms) * ms + pcol % ms;
        TO* const o = out + row * 588 + py * 14 + px;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            // rescale + normalise through the host-built per-channel byte table (reference arithmetic, exact)
            const float a = lut[c * 256 + clip8(s[2 * c] >> PBITS)], b = lut[c * 256 + clip8(s[2 * c + 1] >> PBITS)];
            if constexpr (sizeof(TO) == 2) *reinterpret_cast<unsigned*>(o + c * 196) = pack_bf2(a, b);
            else *reinterpret_cast<f32x2*>(o + c * 196) = f32x2{a, b};
        }
    }
}

template <typename TO, int NG>
void launch_fused(hipStream_t st, size_t lds, int grid, const uint8_t* frames, TO* out, int T, int H, int W, int gh, int gw, int ms, int band_p, int max_rows,
                  const int* bx, const int* kx, int ksx, const int* by, const int* ky, int ksy, const float* table) {
    hipLaunchKernelGGL((resize_patchify_kernel<TO, NG>), dim3(grid), dim3(256), lds, st, frames, out, T, H, W, gh, gw, ms, band_p, max_rows, bx, kx, ksx,
                       by, ky, ksy, table);
}
template <typename TO>
void dispatch_fused(hipStream_t st, size_t lds, int grid, const uint8_t* frames, TO* out, int T, int H, int W, int gh, int gw, int ms, int band_p,
                    int max_rows, const int* bx, const int* kx, int ksx, const int* by, const int* ky, int ksy, const float* table) {
#define COGS_PRE(NG) launch_fused<TO, NG>(st, lds, grid, frames, out, T, H, W, gh, gw, ms, band_p, max_rows, bx, kx, ksx, by, ky, ksy, table)
    if (ksx <= 8) COGS_PRE(2);
    else if (ksx <= 12) COGS_PRE(3);
    else if (ksx <= 16) COGS_PRE(4);
    else COGS_PRE(6);
#undef COGS_PRE
}

inline int grid_for(long total) {
    long g = (total + 255) / 256;
    return (int)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

}  // namespace

int cogs_k_preprocess(hipStream_t st, const uint8_t* frames, int T, int H, int W, int th, int tw, int ms,
                      const int* bx, const int* kx, int ksx, const int* by, const int* ky, int ksy, void* out,
                      int out_dtype, const float* table, uint8_t* tmp) {
    if (T <= 0 || th % (14 * ms) || tw % (14 * ms)) return COGS_E_INVALID;
    {
        // rows a band reads: its centres' span and a kernel's support (2 source rows, scaled when shrinking) on either side
        const int gh1 = th / 14, gw1 = tw / 14, band_p = gh1 % 2 == 0 ? 2 : 1;
        const double scale = (double)H / th, wide = scale > 1.0 ? scale : 1.0;
        const double span = (14 * band_p - 1) * scale + 4 * wide + 3;
        const int max_rows = (int)(span < H ? span : H);
        const size_t lds = 768 * 4 + (size_t)14 * band_p * (2 + ksy) * 4 + (size_t)3 * max_rows * TILE_C;
        const long grid = (long)T * (gh1 / band_p) * ((gw1 + TILE_P - 1) / TILE_P);
        const size_t pair = out_dtype == COGS_DT_BF16 ? 4 : 8;
        if (lds <= 64 * 1024 && ksx <= 24 && (reinterpret_cast<size_t>(out) & (pair - 1)) == 0 && grid < 0x7fffffff) {
            if (out_dtype == COGS_DT_BF16)
                dispatch_fused<bf16_t>(st, lds, (int)grid, frames, (bf16_t*)out, T, H, W, gh1, gw1, ms, band_p, max_rows, bx, kx, ksx, by, ky, ksy, table);
            else
                dispatch_fused<float>(st, lds, (int)grid, frames, (float*)out, T, H, W, gh1, gw1, ms, band_p, max_rows, bx, kx, ksx, by, ky, ksy, table);
            return COGS_LAUNCH_CHECK();
        }
    }
    const long rows = (long)T * H;
    hipLaunchKernelGGL(resize_h_kernel, dim3(grid_for(rows * tw)), dim3(256), 0, st, frames, tmp, rows, W, tw, bx, kx, ksx);
    const int gh = th / 14, gw = tw / 14;
    const long total = (long)T * gh * gw * 588;
    if (out_dtype == COGS_DT_BF16)
        hipLaunchKernelGGL(resize_v_patchify_kernel<bf16_t>, dim3(grid_for(total)), dim3(256), 0, st, tmp, (bf16_t*)out, T,
                           H, tw, gh, gw, ms, by, ky, ksy, table);
    else
        hipLaunchKernelGGL(resize_v_patchify_kernel<float>, dim3(grid_for(total)), dim3(256), 0, st, tmp, (float*)out, T,
                           H, tw, gh, gw, ms, by, ky, ksy, table);
    return COGS_LAUNCH_CHECK();
}
