// GPU pre-processing: uint8 frames -> Pillow-exact bicubic resize -> x/255,
// (x-0.5)/0.5 -> merge-window-major [N,588] patch rows, written straight in the encoder's input dtype.
//
// Replaces Videollama3ImageProcessor._preprocess (model/image_processing_videollama3.py:235-347): PIL
// Image.resize(BICUBIC) + rescale + normalize + the reshape/transpose patchify (:326-345). The resample is
// Pillow's fixed-point algorithm restated exactly (two passes, horizontal first, 22-bit integer coefficients
// built on the host by cogstream_amd.processing.resample_coeffs, uint8 rounding after each pass), so the uint8
// image -- and, through the [3,256] value table (processing.pixel_value_table), pixel_values -- is bit-identical to the reference's host path.
// resize_mfma_kernel does both passes as integer matrix products; resize_patchify_kernel does them with vector instructions where a patch's
// taps span more than 48 source pixels or a band's more than 64 rows (shrinking by more than about 2.6), a row has fewer pixels than the
// products take, or large images come one or a few at a time (vector_is_faster); the two-pass kernels remain for shrinking by so much that a tile's intermediate rows do not fit the LDS, and for outputs
// that are not aligned to a pair of elements.
#include "common.h"
#include "kernels.h"
#include "debug.h"
#include <algorithm>

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

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
// Bound by loads off a word boundary, integer arithmetic (two instructions a product) and byte traffic in LDS: 64 frames 480 x 854 -> 308 x
// 588 in 102 us; the two-pass kernels, a byte load per product, took 447.
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

// ---- both passes as integer matrix products ----------------------------------------------------------------------------------
// A resize is a banded matrix product, and the 22-bit taps are three signed bytes, so that v_mfma_i32_16x16x64_i8 computes it exactly:
//   sum p k = sum (p - 128) k0 + 2^8 sum (p - 128) k1 + 2^16 sum (p - 128) k2 + 128 sum k,   k = k0 + 2^8 k1 + 2^16 k2  (|k| < 1.99 * 2^22).
// A wave owns one patch column (14 output columns) of a band of one or two patch rows and walks over frames. Horizontal: 16 source rows
// are the product's rows, the patch's columns its columns, and K is the interleaved source bytes as they lie in memory, 12 (four
// pixels) to a lane's 16 -- a channel's taps are zero at the other channels' bytes. The result lies as four neighbouring rows of one column
// in a lane: one dword of the wave's transposed [channel][column][64 rows] in LDS, which is the vertical product's operand; that product
// leaves four neighbouring columns of one output row in a lane, the order of pixel_values. The taps of both passes are in registers in the
// order of the lanes, built once per wave from the tables.
// 64 frames 480 x 854 -> 308 x 588: 61 us (the vector form above: 109) with the frames in the Infinity Cache, 111 (142) on frames that are not; 149 MB
// of frames and pixel_values take 30. 8 of them 32 -> 22 us, 64 x 720 x 1280 192 -> 108. What is left: some 700 vector and 90 matrix instructions a frame and wave.
constexpr int MM_ROWS = 64, MM_STRIDE = MM_ROWS + 16, MM_WAVES = 4, MM_RESIDENT = 2048;      // source rows of a band; bytes of a column of them in LDS

// digits of a tap, each in the low byte
__device__ __forceinline__ void tap_digits(int k, unsigned (&d)[3]) {
    const int d0 = (int)(signed char)k, k1 = (k - d0) >> 8, d1 = (int)(signed char)k1;
    d[0] = (unsigned)d0 & 255u;
    d[1] = (unsigned)d1 & 255u;
    d[2] = (unsigned)((k1 - d1) >> 8) & 255u;
}
__device__ __forceinline__ int join_digits(int d0, int d1, int d2) { return (((d2 << 8) + d1) << 8) + d0; }
// four sums -> their bytes clip8(sum >> PBITS). v_ashr_pk_u8_i32 writes two and leaves the destination's upper half as it was, which hipcc
// (7.2) takes for zero when it forms the instruction from shifts and ORs by itself: here only the lower halves are looked at
__device__ __forceinline__ unsigned four_bytes(const i32x4 (&d)[3]) {
    const unsigned lo = __builtin_amdgcn_ashr_pk_u8_i32(join_digits(d[0][0], d[1][0], d[2][0]), join_digits(d[0][1], d[1][1], d[2][1]), PBITS);
    const unsigned hi = __builtin_amdgcn_ashr_pk_u8_i32(join_digits(d[0][2], d[1][2], d[2][2]), join_digits(d[0][3], d[1][3], d[2][3]), PBITS);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// sum over the lanes {r, r + 16, r + 32, r + 48}, in all four
__device__ __forceinline__ int sum_groups(int v) {
    const auto a = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    const unsigned w = a[0] + a[1];
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return (int)(b[0] + b[1]);
}

// KS: 64-byte steps of K (16 pixels each); BP: patch rows of a band; RT: 16-row tiles of its source rows. The loop over the frames has no
// branch: the next frame's loads are in flight while this one is worked on, and its stores are not waited for.
template <typename TO, int KS, int BP, int RT>
__global__ __launch_bounds__(64 * MM_WAVES, KS == 3 && RT == 4 ? 1 : 2) void resize_mfma_kernel(const uint8_t* __restrict__ in, TO* __restrict__ out, int T, int H, int W, int gh, int gw,
                                                                       int ms, int frames, const int* __restrict__ bx, const int* __restrict__ kx, int ksx,
                                                                       const int* __restrict__ by, const int* __restrict__ ky, int ksy,
                                                                       const float* __restrict__ table) {
    __shared__ float lut[768];
    __shared__ __attribute__((aligned(16))) char mids[MM_WAVES][3 * 16 * MM_STRIDE];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = tid; i < 768; i += 64 * MM_WAVES) lut[i] = table[i];
    __syncthreads();
    // neighbouring workgroups on one XCD: the lines that two patch columns share are in its L2
    const int nwg = gridDim.x, xcd = blockIdx.x & 7, q8 = nwg >> 3, r8 = nwg & 7;
    const int wg = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + ((int)blockIdx.x >> 3);
    const int bands = gh / BP, unit = wg * MM_WAVES + wid, pcol = unit % gw, bd = unit / gw % bands, f0 = unit / gw / bands * frames;
    if (f0 >= T) return;
    const int fend = min(f0 + frames, T);
    char* const mid = mids[wid];
    const int li14 = min(li, 13);                                   // (rows and columns 14 and 15 of the products repeat the last)

    // horizontal: lane = column li of the patch, unit 4 s + g of K = the four pixels from base + 4 (4 s + g) on: the 16 bytes from the word
    // that the first one starts in, shifted down to twelve (the fourth word has no taps). Loads off a word boundary are many times
    // slower: with them a frame took 7 us a wave. The clip's last row is read byte by byte where a word behind it would be touched
    const int x = pcol * 14 + li14, x0 = bx[2 * x], base = min(bx[2 * pcol * 14], W - 16 * KS);
    const int y_first = bd * BP * 14, r0 = by[2 * y_first];
    const bool at_end = fend == T && base + 16 * KS >= W - 1 && r0 + 16 * RT >= H;      // (one more pixel behind is three bytes)
    long src_at[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) src_at[t] = (((long)f0 * H + min(r0 + 16 * t + li, H - 1)) * W + base + 4 * g) * 3;
    const long words = (long)(reinterpret_cast<size_t>(in) & 3);     // (frames may start off a word)
    const uint8_t* const in_w = in - words;
    u32x4 src[RT][KS];
    unsigned shift[RT];
    auto load = [&](bool slow) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const long at = src_at[t] + words;
            shift[t] = (unsigned)at & 3u;
            if (slow) {
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int w = 0; w < 3; ++w) {
                        const uint8_t* q = in + src_at[t] + 48 * s + 4 * w;
                        src[t][s][w] = q[0] | q[1] << 8 | q[2] << 16 | (unsigned)q[3] << 24;
                    }
                shift[t] = 0;
            } else {
#pragma unroll
                for (int s = 0; s < KS; ++s) src[t][s] = *reinterpret_cast<const u32x4_a4*>(in_w + (at - shift[t]) + 48 * s);
            }
            src_at[t] += (long)H * W * 3;
        }
    };
    load(at_end && f0 == T - 1);
    u32x4 tx[KS][3][3];                                             // [step][channel][digit]
    int sum_x = 0;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int d = 0; d < 3; ++d) tx[s][c][d] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = base + 4 * (4 * s + g) + j - x0, k = t >= 0 && t < ksx ? kx[(long)x * ksx + t] : 0;
            unsigned d[3];
            sum_x += k;
            tap_digits(k, d);
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int e = 0; e < 3; ++e) tx[s][c][e][(3 * j + c) >> 2] |= d[e] << (8 * ((3 * j + c) & 3));
        }
    }
    // vertical: lane = row li of the patch, source rows r0 + 16 g .. + 15
    u32x4 ty[BP][3];
    int start_y[BP];
#pragma unroll
    for (int pr = 0; pr < BP; ++pr) {
        const int y = y_first + 14 * pr + li14, y0 = by[2 * y], n = by[2 * y + 1];
        int sum = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) ty[pr][d] = u32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = r0 + 16 * g + j - y0, k = t >= 0 && t < n ? ky[(long)y * ksy + t] : 0;
            unsigned d[3];
            sum += k;
            tap_digits(k, d);
#pragma unroll
            for (int e = 0; e < 3; ++e) ty[pr][e][j >> 2] |= d[e] << (8 * (j & 3));
        }
        start_y[pr] = 128 * sum_groups(sum) + (1 << (PBITS - 1));
    }
    const int start_x = 128 * sum_groups(sum_x) + (1 << (PBITS - 1));

    // The vertical product's rows are columns 0 .. 11 of the patch and 10 .. 13: a lane's four are neighbours in memory
    const int wpr = gw / ms, px = g < 3 ? 4 * g : 10, xa = li < 12 ? li : li - 2;
    const long frame = (long)gh * gw * 588;
    TO* o[BP];
#pragma unroll
    for (int pr = 0; pr < BP; ++pr) {
        const int prow = bd * BP + pr;
        o[pr] = out + f0 * frame + (((prow / ms) * wpr + pcol / ms) * (ms * ms) + (prow % ms) * ms + pcol % ms) * 588l + li14 * 14 + px;
    }
    for (int f = f0; f < fend; ++f) {
        u32x4 cur[RT][KS];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int s = 0; s < KS; ++s) {
#pragma unroll
                for (int w = 0; w < 3; ++w) cur[t][s][w] = __builtin_amdgcn_alignbyte(src[t][s][w + 1], src[t][s][w], shift[t]) ^ 0x80808080u;
                cur[t][s][3] = 0;
            }
        if (f + 1 < fend) load(at_end && f + 1 == T - 1);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                i32x4 acc[3] = {{start_x, start_x, start_x, start_x}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int d = 0; d < 3; ++d)
                        acc[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, cur[t][s]), __builtin_bit_cast(i32x4, tx[s][c][d]), acc[d], 0, 0, 0);
                *reinterpret_cast<unsigned*>(mid + (c * 16 + li) * MM_STRIDE + 16 * t + 4 * g) = four_bytes(acc) ^ 0x80808080u;
            }
        }
        asm volatile("" ::: "memory");                             // (a wave's own LDS operations are in order)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const u32x4 a = *reinterpret_cast<const u32x4*>(mid + (c * 16 + xa) * MM_STRIDE + 16 * g);
#pragma unroll
            for (int pr = 0; pr < BP; ++pr) {
                i32x4 acc[3] = {{start_y[pr], start_y[pr], start_y[pr], start_y[pr]}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    acc[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, ty[pr][d]), acc[d], 0, 0, 0);
                // rescale + normalise through the host-built per-channel byte table (reference arithmetic, exact)
                const unsigned b = four_bytes(acc);
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = lut[c * 256 + (b >> (8 * r) & 255u)];
                if constexpr (sizeof(TO) == 2) {
                    const u32x2 w = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
                    __builtin_memcpy(o[pr] + c * 196, &w, 8);
                } else {
                    __builtin_memcpy(o[pr] + c * 196, v, 16);
                }
            }
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int pr = 0; pr < BP; ++pr) o[pr] += frame;
    }
}

// pixels that a patch column's taps span (centres and a kernel's support, as for the bands' rows), rows that a band's do
inline double tap_span(int in_size, int out_size, int outputs) {
    const double scale = (double)in_size / out_size, wide = scale > 1.0 ? scale : 1.0;
    return (outputs - 1) * scale + 4 * wide + 3;
}
// A wave's prologue, the taps in the order of its lanes, costs one and a half frames, and the waves of a large image by itself are more than the
// chip holds: with few frames a wave and few taps an output the vector form is the faster. Times in ns a patch, the prologue over its frames
// here, the taps' growth with the scale there, and 1.7 us more for a launch of that one. Vector / products, us: 1 x 1080 x 1920 -> 1078 x 1918
// 19.8 / 33.6, two frames 33.2 / 43.8, three 44.5 / 53.9; 1 x 720 x 1280 -> 546 x 966 10.0 / 11.7, two 15.7 / 15.0; bands of two patches, 1 x
// 1440 x 2560 -> 1428 x 2548 32.4 / 39.6, -> 1008 x 1792 23.9 / 21.7; 2 x 2160 x 3840 -> 2156 x 3836 91 / 102, 4 x 720 x 1280 -> 728 x 1288
// 31.8 / 28.5. The other form taken costs 6 % at the most over 200 such launches, scales 0.8 to 1.5, one to three frames.
bool vector_is_faster(long waves, int frames, int bp, double scale) {
    const double patches = 1e-3 * waves * frames * bp;
    return waves > MM_RESIDENT && (bp == 1 ? 0.92 : 0.65) * (1 + 1.5 / frames) * patches > ((scale > 1 ? scale : 1) + 0.05) * patches + 1.7;
}
// false: sizes this kernel does not take (columns above 48 source pixels or more than the row has, bands above 64 source rows) or is slower for
template <typename TO>
bool launch_mfma(hipStream_t st, const uint8_t* frames, TO* out, int T, int H, int W, int th, int tw, int ms, const int* bx, const int* kx, int ksx,
                 const int* by, const int* ky, int ksy, const float* table) {
    const int gh = th / 14, gw = tw / 14;
    const double px = tap_span(W, tw, 14);
    const int steps = px <= 32 ? 2 : 3;
    const int bp = steps == 2 && gh % 2 == 0 && tap_span(H, th, 28) <= MM_ROWS ? 2 : 1;       // (three steps leave no registers for two)
    if (px > 48 || W < 16 * steps || tap_span(H, th, 14 * bp) > MM_ROWS) return false;
    // frames in as many groups as give the shortest rounds of waves (two a SIMD); a wave's prologue costs one and a half frames
    const long columns = (long)(gh / bp) * gw;
    int each = T;
    double best = 0;
    for (int groups = 1; groups <= T && groups <= 64; ++groups) {
        const int n = (T + groups - 1) / groups;
        const double cost = (double)((columns * ((T + n - 1) / n) + MM_RESIDENT - 1) / MM_RESIDENT) * (n + 1.5);
        if (groups == 1 || cost < best) { best = cost; each = n; }
    }
    const long units = columns * ((T + each - 1) / each), grid = (units + MM_WAVES - 1) / MM_WAVES;
    if (grid > 0x7fffffff) return false;
    if (steps == 2 && ksx <= 7 && ksy <= 7 && vector_is_faster(units, each, bp, std::max((double)W / tw, (double)H / th))) return false;
    const int tiles = (int)((tap_span(H, th, 14 * bp) + 15) / 16);
#define COGS_MM(KS, BP, RT) hipLaunchKernelGGL((resize_mfma_kernel<TO, KS, BP, RT>), dim3((unsigned)grid), dim3(64 * MM_WAVES), 0, st, frames, out, T, H, W, gh, gw, ms, each, bx, kx, ksx, by, ky, ksy, table)
    if (bp == 2) { if (tiles <= 3) COGS_MM(2, 2, 3); else COGS_MM(2, 2, 4); }
    else if (steps == 2) { if (tiles <= 3) COGS_MM(2, 1, 3); else COGS_MM(2, 1, 4); }
    else if (tiles <= 3) COGS_MM(3, 1, 3);
    else COGS_MM(3, 1, 4);
#undef COGS_MM
    g_cogs_debug.preprocess_last_kernel = 100 * steps + 10 * bp + (tiles <= 3 ? 3 : 4);
    return true;
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
        if ((reinterpret_cast<size_t>(out) & (pair - 1)) == 0 &&
            (out_dtype == COGS_DT_BF16 ? launch_mfma<bf16_t>(st, frames, (bf16_t*)out, T, H, W, th, tw, ms, bx, kx, ksx, by, ky, ksy, table)
                                       : launch_mfma<float>(st, frames, (float*)out, T, H, W, th, tw, ms, bx, kx, ksx, by, ky, ksy, table)))
            return COGS_LAUNCH_CHECK();
        g_cogs_debug.preprocess_last_kernel = 2;
        if (lds <= 64 * 1024 && ksx <= 24 && (reinterpret_cast<size_t>(out) & (pair - 1)) == 0 && grid < 0x7fffffff) {
            if (out_dtype == COGS_DT_BF16)
                dispatch_fused<bf16_t>(st, lds, (int)grid, frames, (bf16_t*)out, T, H, W, gh1, gw1, ms, band_p, max_rows, bx, kx, ksx, by, ky, ksy, table);
            else
                dispatch_fused<float>(st, lds, (int)grid, frames, (float*)out, T, H, W, gh1, gw1, ms, band_p, max_rows, bx, kx, ksx, by, ky, ksy, table);
            return COGS_LAUNCH_CHECK();
        }
    }
    g_cogs_debug.preprocess_last_kernel = 1;
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
