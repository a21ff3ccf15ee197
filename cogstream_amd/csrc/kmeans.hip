// Time-aware k-means device steps (model/kmeans_with_time.py:4-137). The host keeps the reference's RNG draws
// (random.randint / torch.multinomial on the CPU generator); everything that touches the features runs here.
//
//   sqdist        partial[t][slice][k] = sum over the slice's 512 columns of (x[t,j]-c[k,j])^2   (:48,:73  torch.cdist)
//   reduce+assign dist2 = sum of the slice partials (fp64), per-row min-max of feature/time distances,
//                 sqrt(nf^2 + alpha nt^2), argmin                                                   (:76-104)
//   members       member lists per cluster, empty clusters -> reseed rows from the host-drawn pool    (:107-120)
//   update        per-cluster means (or the reseed row), centre shift                                (:107-125)
//
// HBM-bound by design: the features [T, P*D] (bf16 or fp32, 92/183 MB at T = 256) are read exactly once by sqdist and
// once by update per Lloyd iteration, once per k-means++ step. The kernels are built around that bound (rocprofv3
// at [256, 179 200] bf16, K = 18: sqdist 349 -> 76 us; the first version reduced every (row, centre) pair
// across the wave on its own -- 12 cross-lane steps per pair -- and walked member lists one load at a time):
//   * sqdist keeps one accumulator per centre in registers and reduces all of them across the wave in ONE
//     transposing butterfly per row (v_permlane32_swap / v_permlane16_swap on register pairs, then DPP row sums):
//     2.5 instructions per centre instead of 12; the centre slice sits in LDS in a lane-major order that makes the
//     two ds_read_b128 per centre conflict free; rows are taken four at a time so four 16-byte loads per lane are in
//     flight.
//   * the slice partials are summed in fp64 by lanes that own a centre each (coalesced reads), in a fixed order, and
//     the assignment of the row is computed by the same workgroup (one launch instead of two plus a host round trip).
//   * update runs one workgroup per (column block, cluster) -- K times the parallelism -- with four member rows in
//     flight per thread.
// All sums run in a fixed order (reproducible run to run). Distances are DIRECT sums of (x - c)^2, fp32 within a
// 512-column slice, fp64 across slices: |x|^2 + |c|^2 - 2 x.c cancels (|x|^2 is 200 times the nearest distances here, an ulp of it 1e-5 of them), and
// more than a quarter of the rows whose two nearest centres lie within 1e-4 of one another were assigned by its rounding.
#include "common.h"
#include "kernels.h"
#include "debug.h"
#include <stdlib.h>

namespace {

// control words of the in-library Lloyd loop (device ints, in the workspace). The host queues SEVERAL iterations between
// two reads; every kernel of an iteration returns at once when the loop has ended (converged / pool exhausted), so the
// speculatively queued ones change nothing.
enum { CTL_USED = 0,      // reseed-pool entries consumed so far
       CTL_ABORT = 1,     // an iteration wanted more reseeds than the pool holds: it was not committed, the loop stops
       CTL_EMPTY = 2,     // empty clusters of the last iteration
       CTL_SHIFT = 3,     // centre shift of the last committed iteration (float bits)
       CTL_DONE = 4,      // shift <= tol: converged
       CTL_ITERS = 5,     // iterations committed
       CTL_MARGIN = 6,    // bits(+inf) - bits(min over rows and iterations of the decision margin) (reduce_assign_kernel)
       CTL_NEAR = 7,      // rows (summed over iterations) whose margin is below NEAR_TIE
       CTL_WORDS = 8 };
// ... and of the seeding (in the same place)
constexpr int KPP_C = 4;      // rows a pass measures at most
enum { KPP_DONE_ROWS = 0,     // rows measured so far (workgroups that have finished)
       KPP_M = 1,             // centres drawn
       KPP_END = 2,           // all of them
       KPP_N = 3,             // rows of the next pass: the newest centre, then the guesses (the rest of them repeat the newest centre)
       KPP_ROWS = 4 };        // ... KPP_ROWS + KPP_C words in all
static_assert(KPP_ROWS + KPP_C <= CTL_WORDS, "");
constexpr float NEAR_TIE = 1e-3f;   // below this the reference's own sgemm rounding decides a row

constexpr int SL = 512;       // columns per slice
constexpr int KMAX = 32;      // centres per sqdist launch (K itself is unbounded: 18 for 256 frames, 40 for 600)
constexpr int UB = 2048;      // columns per update workgroup (256 threads x 8)

__device__ __forceinline__ float swap32_sum(float a, float b) {
    // lanes 0..31: a[i] + a[i+32]; lanes 32..63: b[i-32] + b[i]
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float swap16_sum(float a, float b) {
    // 16-lane rows 0, 2: a's row pair summed; rows 1, 3: b's row pair summed
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// sum over each 16-lane row, result in every lane of the row: four DPP adds (quad swaps, then the two mirrors). The
// __shfl_xor form compiles to four DEPENDENT ds_bpermute round trips -- ~400 exposed cycles per call, more than the
// arithmetic of the unit it closes (a pass of K = 18 took 102 us with it).
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_mov<0xB1>(v);      // quad_perm [1,0,3,2]: lane ^ 1
    v += dpp_mov<0x4E>(v);      // quad_perm [2,3,0,1]: lane ^ 2
    v += dpp_mov<0x141>(v);     // row_half_mirror: the other quad of the 8-lane half
    v += dpp_mov<0x140>(v);     // row_mirror: the other half of the 16-lane row
    return v;
}

// grid = (slices, row groups); 4 waves; LDS holds the centre slice as [k][half][lane][4] fp32 (half h, lane l = columns
// 8l+4h..+3) for this launch's K <= KMAX centres, padded with zero centres to a multiple of 4 (never stored).
// centre_row >= 0: the single centre is feature row `centre_row` (k-means++ step), else centre_rows / centres.
template <typename T>
__global__ __launch_bounds__(256, 4) void sqdist_kernel(const T* __restrict__ x, int Tn, long PD,
                                                        const float* __restrict__ centres,
                                                        const int* __restrict__ centre_rows, int centre_row, int K, int k0,
                                                        int Ktot, float* __restrict__ partial, const int* __restrict__ ctl, const int* __restrict__ keep) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* cs = reinterpret_cast<float*>(smem_raw);
    if (ctl && (centre_rows ? ctl[KPP_END] : ctl[CTL_ABORT] | ctl[CTL_DONE])) return;   // queued behind the last iteration, or the last draw
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long j = (long)blockIdx.x * SL + lane * 8;
    const bool in = j < PD;
    // the centres that have moved since their distances were last summed (keep null: all of them), their list in a register of every wave: lane i has
    // the i-th. (In LDS its 160 bytes took a workgroup's place on the CU, which the centres fill: launch_sqdist. 256 rows, us, in LDS / here: 18
    // centres of 168, 301, 350, 448 slices 48.4 / 39.6, 82.1 / 68.2, 78.8 / 76.2, 110.7 / 89.7; 13 to 16 and more than 20 centres 3 to 6 % less)
    const bool mine = lane < K && !(keep && keep[k0 + lane]);
    const unsigned long long some = __ballot(mine);
    const bool all = __popcll(some) == K;
    K = __popcll(some);
    if (K == 0) return;
    const int before = __popcll(some & ((1ull << lane) - 1ull));
    const int moved = __builtin_amdgcn_ds_permute(4 * (mine ? before : K + lane - before), lane);
    const int KB = (K + 3) & ~3;
    for (int i = wid; i < KB; i += 4) {
        const int k = k0 + __builtin_amdgcn_readlane(moved, i);
        float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (i < K && in) {
            if (centre_row >= 0) ld8_f<T>(x + (long)centre_row * PD + j, v);
            else if (centre_rows) ld8_f<T>(x + (long)centre_rows[k] * PD + j, v);
            else ld8_f<float>(centres + (long)k * PD + j, v);
        }
        *reinterpret_cast<f32x4*>(cs + i * SL + lane * 4) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>(cs + i * SL + 256 + lane * 4) = f32x4{v[4], v[5], v[6], v[7]};
    }
    __syncthreads();
    // Two rows per wave and step (rows t, t + 4: a centre's two LDS reads serve both), the NEXT step's global loads issued
    // before this step's arithmetic, and the centres taken FOUR at a time in a real loop: four accumulators per row are
    // exactly one unit of the transposing butterfly below, so nothing outlives a trip and the kernel needs ~80 VGPRs
    // (four workgroups per CU). History: one wave reduction per (row, centre) pair -- 12 cross-lane steps each -- 349 us
    // per pass at [256, 179 200] bf16, K = 18; all centres unrolled with one accumulator each: 147 us, and every
    // attempt to share the LDS reads between rows in that form made hipcc issue all the centre reads first (96-160
    // registers, 150 spilled or one wave per SIMD: 257 us).
    // grid.y row groups (a slice alone is 350 workgroups at cfg3 -- too few to hide the load latency on 256 CUs):
    // this workgroup takes rows [r_lo, r_hi)
    const int rows_per = (Tn + (int)gridDim.y - 1) / (int)gridDim.y;
    const int r_lo = (int)blockIdx.y * rows_per, r_hi = min(Tn, r_lo + rows_per);
    const int row = lane >> 4;
    const int kperm = ((row & 1) << 1) + (row >> 1);       // 16-lane row -> centre of a unit: 0, 2, 1, 3
    const bool writer = (lane & 15) == 0;
    const float* cl = cs + lane * 4;
    float xn[2][8];
    auto load_rows = [&](int t) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
#pragma unroll
            for (int e = 0; e < 8; ++e) xn[r][e] = 0.f;
            if (in && t + 4 * r < r_hi) ld8_f<T>(x + (long)(t + 4 * r) * PD + j, xn[r]);
        }
    };
    load_rows(r_lo + wid);
    for (int t = r_lo + wid; t < r_hi; t += 8) {
        f32x2 xab[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) xab[e] = f32x2{xn[0][e], xn[1][e]};
        if (t + 8 < r_hi) load_rows(t + 8);
        const bool live_b = t + 4 < r_hi;
        float* pa = partial + ((long)t * gridDim.x + blockIdx.x) * Ktot + k0;
        float* pb = pa + 4 * (long)gridDim.x * Ktot;
        unsigned k = (unsigned)kperm;
#pragma unroll 1
        for (int m = 0; m < KB; m += 4, k += 4) {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 c0 = *reinterpret_cast<const f32x4*>(cl + (m + q) * SL);
                const f32x4 c1 = *reinterpret_cast<const f32x4*>(cl + (m + q) * SL + 256);
                // the two rows ride in the two halves of a register pair. Every accumulator still sees its own products in the same
                // order (column e of the first half, then of the second), so the sums are bit-identical to the scalar form
                f32x2 s = {0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x2 d0 = xab[e] - f32x2{c0[e], c0[e]};
                    const f32x2 d1 = xab[4 + e] - f32x2{c1[e], c1[e]};
                    s = __builtin_elementwise_fma(d0, d0, s);
                    s = __builtin_elementwise_fma(d1, d1, s);
                }
                a[q] = s[0];
                b[q] = s[1];
            }
            // transposing butterfly of one unit: 4 values x 64 lanes -> every 16-lane row holds the wave total of ONE
            // centre: row 0 -> m, row 1 -> m + 2, row 2 -> m + 1, row 3 -> m + 3
            const float ua = row16_sum(swap16_sum(swap32_sum(a[0], a[1]), swap32_sum(a[2], a[3])));
            const float ub = row16_sum(swap16_sum(swap32_sum(b[0], b[1]), swap32_sum(b[2], b[3])));
            if (!all) k = (unsigned)__shfl(moved, m + kperm);
            if (writer && m + kperm < K) {
                pa[k] = ua;
                if (live_b) pb[k] = ub;
            }
        }
    }
}

// fp64 sum over the slices of partial[t][slice][k] for row t (one run of memory), by the lanes of one workgroup: lane (g, k) owns centre k
// and slice group g; groups are combined in a fixed order. Result in d2s[k] (LDS, fp32 like torch.cdist's output).
// keep[k] (keep nullable): the centre has not moved, kept[t][k] has its sum
__device__ __forceinline__ void reduce_row(const float* __restrict__ partial, int nslices, int K, int t,
                                           float* d2s, double* scratch /* [groups][kp]: 256 doubles */, const int* __restrict__ keep, const float* kept) {
    const int tid = threadIdx.x;
    for (int kc = 0; kc < K; kc += 64) {
        const int Kc = min(64, K - kc);
        int kp = 1;
        while (kp < Kc) kp <<= 1;                 // lanes per slice group (power of two <= 64)
        const int G = 256 / kp;                   // slice groups in the workgroup
        const int k = tid & (kp - 1), g = tid / kp;
        double s = 0.0;
        const bool moved = k < Kc && !(keep && keep[kc + k]);
        if (moved) {
            const float* pp = partial + (long)t * nslices * K + kc + k;
            const long stride = K;
            int sl = g;
            for (; sl + 7 * G < nslices; sl += 8 * G) {       // eight loads in flight, added in slice order
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = pp[(long)(sl + u * G) * stride];
#pragma unroll
                for (int u = 0; u < 8; ++u) s += (double)v[u];
            }
            for (; sl < nslices; sl += G) s += (double)pp[(long)sl * stride];
        }
        if (k < Kc) scratch[g * kp + k] = s;
        __syncthreads();
        if (tid < Kc) {
            double tot = 0.0;
            for (int gg = 0; gg < G; ++gg) tot += scratch[gg * kp + tid];
            d2s[kc + tid] = keep && keep[kc + tid] ? kept[(long)t * K + kc + tid] : (float)tot;
        }
        __syncthreads();
    }
}

// one workgroup per row t: slice reduction + the row's assignment (kmeans_with_time.py:76-104). dist2_out nullable.
// The arithmetic is torch's, operation by operation in fp32 (no contraction): sqrt, |.|, per-row min/max over the
// clusters, (d - min) / (max - min) or 0, sqrt(nf*nf + alpha*(nt*nt)), first minimum wins.
__global__ __launch_bounds__(256) void reduce_assign_kernel(const float* __restrict__ partial, int nslices, int Tn, int K,
                                                            const float* __restrict__ ts, const float* __restrict__ cts,
                                                            float alpha, float* dist2_out,
                                                            int64_t* __restrict__ assign, int* __restrict__ ctl, const int* __restrict__ keep) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    double* scratch = reinterpret_cast<double*>(smem_raw);           // 256 doubles
    if (ctl && (ctl[CTL_ABORT] | ctl[CTL_DONE])) return;
    float* d2s = reinterpret_cast<float*>(scratch + 256);            // [K]
    const int t = blockIdx.x;
    reduce_row(partial, nslices, K, t, d2s, scratch, keep, dist2_out);
    const int tid = threadIdx.x;
    if (dist2_out)
        for (int k = tid; k < K; k += 256) dist2_out[(long)t * K + k] = d2s[k];
    if (!assign) return;
    if (tid >= 64) return;                        // one wave finishes the row
    const int lane = tid;
    const float tt = ts[t];
    float fmin_ = INFINITY, fmax_ = -INFINITY, tmin_ = INFINITY, tmax_ = -INFINITY;
    for (int k = lane; k < K; k += 64) {
        const float df = sqrtf(d2s[k]);
        const float dt = fabsf(tt - cts[k]);
        fmin_ = fminf(fmin_, df); fmax_ = fmaxf(fmax_, df);
        tmin_ = fminf(tmin_, dt); tmax_ = fmaxf(tmax_, dt);
    }
    fmin_ = wave_min(fmin_); fmax_ = wave_max(fmax_);
    tmin_ = wave_min(tmin_); tmax_ = wave_max(tmax_);
    float best = INFINITY, second = INFINITY;
    int bk = 0x7fffffff, sk = 0x7fffffff;
    auto final_dist = [&](int k, float& df, float& nf) {
        df = sqrtf(d2s[k]);
        const float dt = fabsf(tt - cts[k]);
        nf = fmax_ > fmin_ ? __fdiv_rn(__fsub_rn(df, fmin_), __fsub_rn(fmax_, fmin_)) : 0.f;
        const float nt = tmax_ > tmin_ ? __fdiv_rn(__fsub_rn(dt, tmin_), __fsub_rn(tmax_, tmin_)) : 0.f;
        return sqrtf(__fadd_rn(__fmul_rn(nf, nf), __fmul_rn(alpha, __fmul_rn(nt, nt))));
    };
    for (int k = lane; k < K; k += 64) {
        float df, nf;
        const float fd = final_dist(k, df, nf);
        if (fd < best) { second = best; sk = bk; best = fd; bk = k; }     // ascending k per lane: the lane keeps its FIRST minimum
        else if (fd < second) { second = fd; sk = k; }
    }
    const float wbest = wave_min(best);
    // first minimum overall = smallest k among the lanes that hold the minimum value
    int cand = (best == wbest) ? bk : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    if (lane == 0) assign[t] = cand == 0x7fffffff ? 0 : cand;        // all-NaN row: cluster 0, like a serial first-minimum scan
    if (ctl && K > 1 && cand != 0x7fffffff) {
        // How close was the decision? Runner-up = the smallest final distance of any OTHER cluster. The margin is
        // expressed in the unit the near-tie study (tests/golden/kmeans_tie_study.py) uses: the RELATIVE change of the feature
        // distances that would flip the order. A relative change e of d_k moves nf_k by d_k e / R (R = max - min of
        // the row) and the final distance sqrt(nf^2 + alpha nt^2) by (nf_k / fd_k) d_k e / R; with the winner moving up
        // and the runner-up down the gap closes at e* = gap / (s_1 + s_2); reported as 2 e*, which for a pure feature
        // decision (all time terms equal) is (d_2 - d_1) / mean(d_1, d_2), the study's margin. A decision the feature
        // distances cannot flip (s_1 = s_2 = 0) reports +inf.
        const float oval = bk == cand ? second : best;
        const int okk = bk == cand ? sk : bk;
        const float wsecond = wave_min(oval);
        int cand2 = (oval == wsecond) ? okk : 0x7fffffff;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) cand2 = min(cand2, __shfl_xor(cand2, o, 64));
        if (lane == 0 && cand2 != 0x7fffffff) {
            float d1, n1, d2, n2;
            const float f1 = final_dist(cand, d1, n1), f2 = final_dist(cand2, d2, n2);
            const float R = fmax_ - fmin_;
            float m = INFINITY;
            if (R > 0.f) {
                const float s1 = (f1 > 0.f ? n1 / f1 : 1.f) * d1 / R, s2 = (f2 > 0.f ? n2 / f2 : 1.f) * d2 / R;
                if (s1 + s2 > 0.f) m = 2.f * (f2 - f1) / (s1 + s2);
            }
            if (!(m == m) || m < 0.f) m = 0.f;
            // non-negative floats order like their bits; kept as the MAXIMUM of (bits(+inf) - bits(m)) so that the
            // all-zero control block the loop starts from means "margin = +inf"
            atomicMax(reinterpret_cast<unsigned*>(ctl + CTL_MARGIN), 0x7f800000u - __float_as_uint(m));
            if (m < NEAR_TIE) atomicAdd(ctl + CTL_NEAR, 1);
        }
    }
}

// The whole seeding, several centres a pass. A draw needs the distances to every centre in front of it, but which row it falls on can mostly be told
// without the last of them: nearest2 only shrinks, and a new centre shrinks it for the rows of its own scene alone. So a pass over the features measures
// the newest centre and, beside it, the rows that the next draws would fall on if nearest2 stayed as it is; the workgroup that finishes last draws
// centres for as long as the newest one is among those measured, and leaves the next pass's rows. What is drawn, from which distances and in which
// order is what a pass per centre draws: a guess that does not come true has been measured in vain. Passes queued behind the last draw return at once.
// 256 frames of some twenty scenes, 18 centres: 5.4 passes of 4 rows on the average instead of 17.
struct KppArgs {
    int Tn, K;
    float* nearest2; const float* q; int* idx; int* zero_flag;
    int* state;
    float* d2; int ldd2;            // the pass's distances [Tn][ldd2]
    float* dist2;                   // nullable [Tn][K]
};

// sum or maximum over a wave in every lane, lanes 32, 16, 8, .. 1 apart (a register move each; through LDS a draw was 0.6 us longer)
template <typename F>
__device__ __forceinline__ void wave_join(F&& join) {
    join([](unsigned v) { const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false); return (threadIdx.x & 32) ? (unsigned)r[0] : (unsigned)r[1]; });
    join([](unsigned v) { const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false); return (threadIdx.x & 16) ? (unsigned)r[0] : (unsigned)r[1]; });
    join([](unsigned v) { return __float_as_uint(lane_xor_dpp<8>(__uint_as_float(v))); });
    join([](unsigned v) { return __float_as_uint(lane_xor_dpp<4>(__uint_as_float(v))); });
    join([](unsigned v) { return __float_as_uint(lane_xor_dpp<2>(__uint_as_float(v))); });
    join([](unsigned v) { return __float_as_uint(lane_xor_dpp<1>(__uint_as_float(v))); });
}
__device__ __forceinline__ double wave_sum_f64(double s) {
    wave_join([&](auto&& other) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, s);
        s += __builtin_bit_cast(double, (unsigned long long)other((unsigned)(b >> 32)) << 32 | other((unsigned)b));
    });
    return s;
}
// a ratio and its row as one number: larger ratio first, NaN before all others like in torch.argmax, then the lower row; 0 is no row
__device__ __forceinline__ unsigned long long ranked(float r, int t) {
    const unsigned b = __float_as_uint(r + 0.f), up = r != r ? 0xffffffffu : b & 0x80000000u ? ~b : b | 0x80000000u;
    return (unsigned long long)up << 32 | ~(unsigned)t;
}
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
    wave_join([&](auto&& other) {
        const unsigned long long o = (unsigned long long)other((unsigned)(v >> 32)) << 32 | other((unsigned)v);
        v = v > o ? v : o;
    });
    return v;
}
__device__ __forceinline__ int ranked_row(unsigned long long v, int none) { return v == 0 ? none : (int)~(unsigned)v; }

// the rows that the draws behind centre m would fall on, a wave each (guess(t): what is known of row t's nearest2)
template <typename F>
__device__ __forceinline__ void kpp_guess(const KppArgs& p, int m, int newest, int tid, int waves, F&& guess) {
    const int lane = tid & 63, wid = tid >> 6, n = max(1, min(min(KPP_C, p.ldd2), p.K - m));      // (the last centre's distances are not needed)
    for (int j = wid; j < KPP_C; j += waves) {
        unsigned long long best = 0;
        if (j > 0 && j < n) {
            const float* q = p.q + (long)(m + j - 2) * p.Tn;
            for (int t = lane; t < p.Tn; t += 64) {
                const float r = guess(t) / q[t];
                if (t != newest && r > 0.f) best = max(best, ranked(r, t));
            }
            best = wave_max_u64(best);
        }
        if (lane == 0) p.state[KPP_ROWS + j] = ranked_row(best, newest);
    }
    if (tid == 0) p.state[KPP_N] = n;
}

// k-means++ draws (:53-60) on the device: probs = (sqrt(nearest2))^2 as the reference computes them from cdist's distances,
// normalised by their sum; torch.multinomial(probs, 1) on the CPU IS argmax(probs / q), q ~ Exponential(1) one draw per
// element from the CPU generator (ATen multinomial, n_sample == 1) -- the host hands those draws over. A zero sum (every
// row coincides with a chosen centre) is the reference's random.randint branch: flagged, the host then takes the step-wise
// path. The sum runs in fp64 in a fixed order (torch's own fp32 summation order is not reproduced: the sum
// is a common divisor of all ratios and only moves the argmax between ratios closer than a few ulps).
// Run by the workgroup that measured the last row (others wrote d2: read past the caches), the rows by its first 256 threads. It is all latency: what a
// thread's first two rows need for the draws of a pass is loaded at once (in turn, with the waves' sums through LDS: 3.7 us a draw).
template <int THREADS>
__device__ __forceinline__ void kpp_draw(const KppArgs& p) {
    __shared__ double red[4];
    __shared__ unsigned long long rv[4];
    constexpr int R = 2;
    __shared__ float near_s[256 * R], d2_s[KPP_C][256 * R], q_s[KPP_C][256 * R];        // (of rows that are all one thread's but in kpp_guess)
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const bool on = tid < 256;
    int m = p.state[KPP_M], newest = p.state[KPP_ROWS], rows[KPP_C], c = 0;
    const int n = p.state[KPP_N], m0 = m;
#pragma unroll
    for (int j = 0; j < KPP_C; ++j) rows[j] = p.state[KPP_ROWS + j];
    auto load_d2 = [&](int t, int j) { return __hip_atomic_load(p.d2 + (long)t * p.ldd2 + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    if (on) {
        float d2[R][KPP_C], q[R][KPP_C], near[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int t = min(tid + 256 * r, p.Tn - 1);          // (rows and draws past the end repeat the last one and are not used)
#pragma unroll
            for (int j = 0; j < KPP_C; ++j) {
                d2[r][j] = load_d2(t, min(j, n - 1));
                q[r][j] = p.q[(long)min(m - 1 + j, p.K - 2) * p.Tn + t];
            }
            near[r] = m == 1 ? 0.f : p.nearest2[t];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int j = 0; j < KPP_C; ++j) {
                d2_s[j][tid + 256 * r] = d2[r][j];
                q_s[j][tid + 256 * r] = q[r][j];
            }
            near_s[tid + 256 * r] = near[r];
        }
    }
    auto d2_of = [&](int t) { return t < 256 * R ? d2_s[c][t] : load_d2(t, c); };
    auto q_of = [&](int t) { return t < 256 * R ? q_s[m - m0][t] : p.q[(long)(m - 1) * p.Tn + t]; };
    auto near_of = [&](int t) -> float& { return t < 256 * R ? near_s[t] : p.nearest2[t]; };
    bool end = false;
    for (;;) {
        double sum = 0.0;
        for (int t = on ? tid : p.Tn; t < p.Tn; t += 256) {
            const float d2 = d2_of(t), near = m > 1 ? fminf(near_of(t), d2) : d2;
            near_of(t) = near;
            if (p.dist2) p.dist2[(long)t * p.K + m - 1] = d2;
            const float d = sqrtf(near);
            sum += (double)__fmul_rn(d, d);
        }
        sum = wave_sum_f64(sum);
        if (on && lane == 0) red[wid] = sum;
        __syncthreads();
        const float total = (float)((red[0] + red[1]) + (red[2] + red[3]));
        if (total == 0.f) {                                      // nothing is drawn from here on
            if (tid == 0) *p.zero_flag = 1;
            for (int k = m + tid; k < p.K; k += THREADS) p.idx[k] = 0;
            if (p.dist2)
                for (int t = tid; t < p.Tn; t += THREADS)
                    for (int k = m; k < p.K - 1; ++k) p.dist2[(long)t * p.K + k] = 0.f;
            end = true;
            break;
        }
        unsigned long long best = 0;
        for (int t = on ? tid : p.Tn; t < p.Tn; t += 256) {
            const float d = sqrtf(near_of(t));
            best = max(best, ranked(__fdiv_rn(__fdiv_rn(__fmul_rn(d, d), total), q_of(t)), t));
        }
        best = wave_max_u64(best);
        if (on && lane == 0) rv[wid] = best;
        __syncthreads();
        newest = ranked_row(max(max(rv[0], rv[1]), max(rv[2], rv[3])), 0);
        if (tid == 0) p.idx[m] = newest;
        if (++m == p.K) { end = true; break; }
        c = -1;
#pragma unroll
        for (int j = KPP_C - 1; j >= 0; --j)
            if (j < n && rows[j] == newest) c = j;
        if (c < 0 || m - m0 == KPP_C) break;
    }
    if (tid == 0) {
        p.state[KPP_M] = m;
        p.state[KPP_END] = end;
        p.state[KPP_DONE_ROWS] = 0;                              // for the next pass
    }
    if (end) return;
    for (int t = tid; on && t < min(256 * R, p.Tn); t += 256) p.nearest2[t] = near_s[t];
    __threadfence_block();                                       // (further rows of nearest2 were written by other threads of the workgroup)
    __syncthreads();
    kpp_guess(p, m, newest, tid, THREADS / 64, near_of);
}

// the first pass's rows: no distance is known yet.
__global__ __launch_bounds__(256) void kpp_start_kernel(KppArgs p, int first_row) {
    if (threadIdx.x == 0) {
        p.state[KPP_DONE_ROWS] = 0;
        p.state[KPP_M] = 1;
        p.state[KPP_END] = p.K < 2;
        *p.zero_flag = 0;
        p.idx[0] = first_row;
    }
    kpp_guess(p, 1, first_row, threadIdx.x, 4, [](int) { return 1.f; });
}

// One pass (:46-60) with a row per workgroup: workgroup t measures row t against up to KPP_C others, a slice of 512 columns per wave at a time. The sums
// are those of sqdist_kernel and kpp_reduce_kernel, value by value: fp32 within a slice (lanes 32, 16, then 1, 2, 4, 8 apart), the
// slices in fp64 by one wave's lanes. Bound by what a CU takes in (its row and the others', which its XCD's L2 has) and by the products' sums.
constexpr int KPP_T = 1024;
template <typename T, int C>
__device__ __forceinline__ void kpp_measure(const T* __restrict__ x, const KppArgs& p, long PD, int nslices, float* sums) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NW = KPP_T / 64, U = C == 1 ? 4 : sizeof(T) == 2 ? 3 : 1;
    const T* xr = x + (long)blockIdx.x * PD + lane * 8;
    const T* cr[C];
#pragma unroll
    for (int j = 0; j < C; ++j) cr[j] = x + (long)__builtin_amdgcn_readfirstlane(p.state[KPP_ROWS + j]) * PD + lane * 8;
    const int row = lane >> 4, mine = ((row & 1) << 1) + (row >> 1);          // 16-lane row -> its row's sum: 0, 2, 1, 3
    // a row is a whole number of memory interleaves away from the next as often as not: every workgroup starts at another slice
    const int turn = (int)((unsigned)blockIdx.x * 61u % (unsigned)nslices);
    auto slice = [&](int i) { const int sl = i + turn; return sl < nslices ? sl : sl - nslices; };
    for (int s0 = wid; s0 < nslices; s0 += NW * U) {
        float a[U][8], c[U][C][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {                            // (slices and columns past the end repeat what is there and are not used)
            const long j = (long)slice(min(s0 + NW * u, nslices - 1)) * SL;
            const long at = j + lane * 8 < PD ? j : PD - 8 - lane * 8;
            ld8_f<T>(xr + at, a[u]);
#pragma unroll
            for (int k = 0; k < C; ++k) ld8_f<T>(cr[k] + at, c[u][k]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s0 + NW * u >= nslices) break;
            const int sl = slice(s0 + NW * u);
            float s[C];
#pragma unroll
            for (int k = 0; k < C; ++k) {
                s[k] = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float d0 = a[u][e] - c[u][k][e], d1 = a[u][4 + e] - c[u][k][4 + e];
                    s[k] = fmaf(d0, d0, s[k]);
                    s[k] = fmaf(d1, d1, s[k]);
                }
                if ((long)sl * SL + lane * 8 >= PD) s[k] = 0.f;
            }
            if constexpr (C == 1) {
                float v = swap32_sum(s[0], s[0]);
                v = row16_sum(swap16_sum(v, v));
                if (lane == 0) sums[sl] = v;
            } else {
                const float v = row16_sum(swap16_sum(swap32_sum(s[0], s[1]), swap32_sum(s[2], s[3])));
                if ((lane & 15) == 0) sums[mine * nslices + sl] = v;
            }
        }
    }
    __syncthreads();
    if (wid < C) {
        double d = 0.0;
        for (int sl = lane; sl < nslices; sl += 64) d += (double)sums[wid * nslices + sl];
        d = wave_sum_f64(d);
        if (lane == 0) __hip_atomic_store(p.d2 + (long)blockIdx.x * p.ldd2 + wid, (float)d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// true in every thread of the workgroup that calls it last; d2 of all of them is there then
__device__ __forceinline__ bool kpp_last(const KppArgs& p) {
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // every wave's own stores (past the caches) have arrived
    __syncthreads();
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(p.state + KPP_DONE_ROWS, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == p.Tn - 1;
    __syncthreads();
    return last;
}

template <typename T>
__global__ __launch_bounds__(KPP_T) void kpp_pass_kernel(const T* __restrict__ x, KppArgs p, long PD, int nslices) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* const sums = reinterpret_cast<float*>(smem_raw);                                                     // [KPP_C][nslices]
    if (p.state[KPP_END]) return;
    if (p.state[KPP_N] == 1) kpp_measure<T, 1>(x, p, PD, nslices, sums);
    else kpp_measure<T, KPP_C>(x, p, PD, nslices, sums);
    if (kpp_last(p)) kpp_draw<KPP_T>(p);
}

// ... of a pass that sqdist_kernel has measured by slices, partial [row][slice][ldd2]: a workgroup per row, a wave per measured row, lanes over slices
__global__ __launch_bounds__(256) void kpp_reduce_kernel(const float* __restrict__ partial, KppArgs p, int nslices) {
    if (p.state[KPP_END]) return;
    constexpr int U = 8;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (wid < p.ldd2) {
        double s = 0.0;
        for (int s0 = lane; s0 < nslices; s0 += 64 * U) {        // U loads in flight, added in slice order
            float v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = s0 + 64 * u < nslices ? partial[((long)blockIdx.x * nslices + s0 + 64 * u) * p.ldd2 + wid] : 0.f;
#pragma unroll
            for (int u = 0; u < U; ++u) s += (double)v[u];
        }
        s = wave_sum_f64(s);
        if (lane == 0) __hip_atomic_store(p.d2 + (long)blockIdx.x * p.ldd2 + wid, (float)s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (kpp_last(p)) kpp_draw<256>(p);
}

// k-means++ step (:46-60): nearest2[t] = min(nearest2[t], dist2 to the newest centre) (first: plain store)
__global__ __launch_bounds__(256) void reduce_min_kernel(const float* __restrict__ partial, int nslices, int Tn, int first,
                                                         float* __restrict__ nearest2) {
    // one wave per row: lanes over slices, fp64 butterfly
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= Tn) return;
    double s = 0.0;
    for (int sl = lane; sl < nslices; sl += 64) s += (double)partial[(long)t * nslices + sl];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) {
        const float d2 = (float)s;
        nearest2[t] = first ? d2 : fminf(nearest2[t], d2);
    }
}

// ctl words (device ints): [0] reseeds used so far, [1] abort (pool exhausted), [2] empty clusters of this iteration
// One workgroup. Member lists (rows of every cluster in ascending order): offs [K+1], members [T]. Empty cluster k gets
// reseed_rows[k] = pool[used + (empty clusters below k)] -- the reference draws one random row per empty cluster in
// ascending k (:116-120) -- unless `reseed_in` is given (host-chosen rows, the step-wise API). Tn <= MEMB_T rows of
// assignments are staged in LDS.
constexpr int MEMB_T = 16384;
__global__ __launch_bounds__(1024) void members_kernel(const int64_t* __restrict__ assign, int Tn, int K,
                                                       int* __restrict__ offs, int* __restrict__ members,
                                                       const int* __restrict__ pool, int pool_len,
                                                       const int* __restrict__ reseed_in, int* __restrict__ reseed_rows,
                                                       int* __restrict__ ctl, int* __restrict__ before, int* __restrict__ keep, const float* __restrict__ shift) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    int* a = reinterpret_cast<int*>(smem_raw);        // [Tn]
    int* cnt = a + Tn;                                // [K + 1]
    const int tid = threadIdx.x, nt = blockDim.x;
    if (ctl && (ctl[CTL_ABORT] | ctl[CTL_DONE])) return;
    // a cluster that no row has joined or left since the last committed iteration of this call keeps its centre, the mean of the same rows in the
    // same order -- if that is finite (its last shift was), so that what is not a number goes on moving
    const bool again = ctl && keep && ctl[CTL_ITERS] > 0;
    for (int k = tid; k <= K; k += nt) cnt[k] = 0;
    if (keep)
        for (int k = tid; k < K; k += nt) keep[k] = again && shift[k] < INFINITY;
    __syncthreads();
    for (int t = tid; t < Tn; t += nt) {
        int c = (int)assign[t];
        c = c < 0 ? 0 : (c >= K ? K - 1 : c);       // a foreign assignment vector must not index outside the tables
        a[t] = c;
        atomicAdd(&cnt[c], 1);
        if (!keep) continue;
        if (again && before[t] != c) keep[before[t]] = keep[c] = 0;
        before[t] = c;
    }
    __syncthreads();
    // one wave: where every cluster's rows begin, and the empty clusters in ascending order, 64 clusters at a time
    if (tid < 64) {
        int o = 0, ne = 0;
        const int used = ctl ? ctl[CTL_USED] : 0;
        for (int k0 = 0; k0 < K; k0 += 64) {
            const int k = k0 + tid, n = k < K ? cnt[k] : 0;
            int upto = n;                                        // rows of the clusters up to this one
#pragma unroll
            for (int d = 1; d < 64; d *= 2) {
                const int v = __shfl_up(upto, d, 64);
                if (tid >= d) upto += v;
            }
            const unsigned long long none = __ballot(k < K && n == 0);
            if (k < K) {
                if (n == 0) {
                    const int e = used + ne + __popcll(none & ((1ull << tid) - 1ull));
                    reseed_rows[k] = reseed_in ? reseed_in[k] : pool && e < pool_len ? pool[e] : 0;
                    if (keep) keep[k] = 0;
                }
                cnt[k] = o + upto - n;                           // becomes the cluster's write cursor base
                offs[k + 1] = o + upto;
            }
            o += __shfl(upto, 63, 64);
            ne += __popcll(none);
        }
        if (tid == 0) offs[0] = 0;
        if (tid == 0 && ctl) {
            ctl[CTL_EMPTY] = ne;
            if (!reseed_in && ne > 0) {
                if (!pool || used + ne > pool_len) ctl[CTL_ABORT] = 1;      // abort: this iteration must not commit
                else ctl[CTL_USED] = used + ne;
            }
        }
    }
    __syncthreads();
    // rank of row t inside its cluster = rows t' < t of the same cluster (LDS broadcast reads)
    for (int t = tid; t < Tn; t += nt) {
        const int c = a[t];
        int r = 0;
#pragma unroll 8
        for (int u = 0; u < t; ++u) r += (a[u] == c) ? 1 : 0;
        members[cnt[c] + r] = t;
    }
}

// fallback for Tn > MEMB_T (no LDS staging): thread k walks the assignment vector
__global__ __launch_bounds__(256) void members_slow_kernel(const int64_t* __restrict__ assign, int Tn, int K,
                                                           int* __restrict__ offs, int* __restrict__ members) {
    for (int k = threadIdx.x; k < K; k += 256) {
        int n = 0;
        for (int t = 0; t < Tn; ++t) n += ((int)assign[t] == k) ? 1 : 0;
        offs[k + 1] = n;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int o = 0;
        offs[0] = 0;
        for (int k = 0; k < K; ++k) { const int n = offs[k + 1]; offs[k + 1] = o + n; o += n; }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += 256) {
        int o = offs[k];
        for (int t = 0; t < Tn; ++t)
            if ((int)assign[t] == k) members[o++] = t;
    }
}

// grid (column blocks, K): the mean of cluster k over this block's 2048 columns (members walked in ascending order, four
// loads in flight, summed in order), or the reseed row when the cluster is empty; squared shift of the block
template <typename T>
__global__ __launch_bounds__(256) void update_kernel(const T* __restrict__ x, long PD, int K,
                                                     const int* __restrict__ offs, const int* __restrict__ members,
                                                     const int* __restrict__ reseed_rows, const int* __restrict__ ctl,
                                                     float* __restrict__ centres, float* __restrict__ shift_partial, const int* __restrict__ keep) {
    __shared__ float red[4];
    if (ctl && (ctl[CTL_ABORT] | ctl[CTL_DONE])) return;   // pool exhausted: nothing of this iteration is committed; or the loop has ended
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int k = blockIdx.y;
    if (keep && keep[k]) {
        if (tid == 0) shift_partial[(long)blockIdx.x * K + k] = 0.f;
        return;
    }
    const long col = ((long)blockIdx.x * 256 + tid) * 8;
    const bool in = col < PD;
    float sh = 0.f;
    if (in) {
        const int b = offs[k], e = offs[k + 1];
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (e > b) {
            int i = b;
            for (; i + 4 <= e; i += 4) {
                float v[4][8];
#pragma unroll
                for (int u = 0; u < 4; ++u) ld8_f<T>(x + (long)members[i + u] * PD + col, v[u]);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < 8; ++c) acc[c] += v[u][c];
            }
            for (; i < e; ++i) {
                float v[8];
                ld8_f<T>(x + (long)members[i] * PD + col, v);
#pragma unroll
                for (int c = 0; c < 8; ++c) acc[c] += v[c];
            }
            const float n = (float)(e - b);
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[c] = acc[c] / n;
        } else {
            ld8_f<T>(x + (long)reseed_rows[k] * PD + col, acc);
        }
        float* cp = centres + (long)k * PD + col;
        float old[8];
        ld8_f<float>(cp, old);
#pragma unroll
        for (int c = 0; c < 8; ++c) { const float d = acc[c] - old[c]; sh = fmaf(d, d, sh); }
        st8_f<float>(cp, acc);
    }
    sh = wave_sum(sh);
    if (lane == 0) red[wid] = sh;
    __syncthreads();
    if (tid == 0) shift_partial[(long)blockIdx.x * K + k] = (red[0] + red[1]) + (red[2] + red[3]);
}

// one workgroup: centre times, shift norms (scratch [2K]: feature-shift norm, squared time shift), total movement.
// status (nullable, host-mapped): {shift, reseeds used, abort, empty clusters} for the Lloyd loop's one read per iteration
constexpr int UF_T = 1024, UF_K = 128;
__global__ __launch_bounds__(UF_T) void update_final_kernel(const float* __restrict__ ts, int K,
                                                           const int* __restrict__ offs, const int* __restrict__ members,
                                                           const int* __restrict__ reseed_rows, int* __restrict__ ctl,
                                                           float* __restrict__ cts,
                                                           const float* __restrict__ shift_partial, int nblk,
                                                           float* __restrict__ scratch, float* __restrict__ shift_out,
                                                           volatile int* __restrict__ status, int Tn_lds, float tol, const int* __restrict__ watch) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* mts = reinterpret_cast<float*>(smem_raw);      // [Tn] time stamps in member order (0 floats when Tn_lds == 0)
    __shared__ float moved[2 * UF_K];                     // as scratch, of the first UF_K clusters: what thread 0 adds up at the end, one after the other
    if (ctl && ctl[CTL_DONE]) return;                     // a speculatively queued iteration behind the converged one
    const bool aborted = ctl && ctl[CTL_ABORT];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (!aborted) {
        if (Tn_lds > 0) {
            for (int i = threadIdx.x; i < Tn_lds; i += UF_T) mts[i] = ts[members[i]];     // one dependent pair per thread, in parallel
            __syncthreads();
        }
        for (int k = wid; k < K; k += UF_T / 64) {          // shift: one wave per cluster
            double s = 0.0;
            for (int b = lane; b < nblk; b += 64) s += (double)shift_partial[(long)b * K + k];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
            if (lane == 0) {
                const float v = scratch[k] = sqrtf((float)s);
                if (k < UF_K) moved[k] = v;
            }
        }
        for (int k = UF_T - 1 - (int)threadIdx.x; k < K; k += UF_T) {      // times: one thread per cluster, its members in order (the last waves first: they
            float tsum = 0.f;                                                       // have the fewest shifts to sum)
            const int b0 = offs[k], e0 = offs[k + 1];
            if (Tn_lds > 0) { for (int i = b0; i < e0; ++i) tsum += mts[i]; }
            else { for (int i = b0; i < e0; ++i) tsum += ts[members[i]]; }
            const float nt = e0 > b0 ? tsum / (float)(e0 - b0) : ts[reseed_rows[k]];
            const float d = nt - cts[k];
            scratch[K + k] = d * d;
            if (k < UF_K) moved[UF_K + k] = d * d;
            cts[k] = nt;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        if (!aborted) {
            float f = 0.f, tt = 0.f;
            for (int i = 0; i < K; ++i) { f += i < UF_K ? moved[i] : scratch[i]; tt += i < UF_K ? moved[UF_K + i] : scratch[K + i]; }
            total = f + sqrtf(tt);
            shift_out[0] = total;
        }
        if (ctl && !aborted) {
            ctl[CTL_SHIFT] = __builtin_bit_cast(int, total);
            ctl[CTL_ITERS] += 1;
            if (total <= tol) ctl[CTL_DONE] = 1;
        }
        if (status) {      // host-mapped copy of the control words (one read per batch of iterations)
#pragma unroll
            for (int i = 0; i < CTL_WORDS; ++i) status[i] = ctl ? ctl[i] : 0;
            status[CTL_WORDS] = watch ? *watch : 0;
            __threadfence_system();
        }
    }
}

// what a loop starts from: zeros at ctl, ones and zeros at keep. One launch: memsets of a few words are one to three of 1 to
// 5 us and a gap (256 frames of 50 tokens: 28 us in front of the Lloyd loop, 5 so)
__global__ __launch_bounds__(256) void start_kernel(int* ctl, int* keep, int K, int known) {
    if (threadIdx.x < CTL_WORDS) ctl[threadIdx.x] = 0;
    for (int k = threadIdx.x; k < K; k += 256) keep[k] = k < known;
}

// one thread per row t from dist2 (the step-wise API, cogs_kmeans_assign); counts must be zero on entry
__global__ __launch_bounds__(256) void assign_kernel(const float* __restrict__ dist2, const float* __restrict__ ts,
                                                     const float* __restrict__ cts, int Tn, int K, float alpha,
                                                     int64_t* __restrict__ assign, int* __restrict__ counts) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= Tn) return;
    const float* d2 = dist2 + (long)t * K;
    float fmin_ = INFINITY, fmax_ = -INFINITY, tmin_ = INFINITY, tmax_ = -INFINITY;
    for (int k = 0; k < K; ++k) {
        const float df = sqrtf(d2[k]);
        const float dt = fabsf(ts[t] - cts[k]);
        fmin_ = fminf(fmin_, df); fmax_ = fmaxf(fmax_, df);
        tmin_ = fminf(tmin_, dt); tmax_ = fmaxf(tmax_, dt);
    }
    float best = INFINITY;
    int bk = 0;
    for (int k = 0; k < K; ++k) {
        const float df = sqrtf(d2[k]);
        const float dt = fabsf(ts[t] - cts[k]);
        const float nf = fmax_ > fmin_ ? __fdiv_rn(__fsub_rn(df, fmin_), __fsub_rn(fmax_, fmin_)) : 0.f;
        const float nt = tmax_ > tmin_ ? __fdiv_rn(__fsub_rn(dt, tmin_), __fsub_rn(tmax_, tmin_)) : 0.f;
        const float fd = sqrtf(__fadd_rn(__fmul_rn(nf, nf), __fmul_rn(alpha, __fmul_rn(nt, nt))));
        if (fd < best) { best = fd; bk = k; }
    }
    assign[t] = bk;
    atomicAdd(&counts[bk], 1);
}

// select_additional_frames (model/cogreasoner_chat.py:50-64): per cluster, all members if there are at most n, else the n
// members nearest to the centroid (smallest dist2, ties to the lower row; torch.topk(largest=False) order = ascending
// distance). One wave per cluster; picks [K][n] int64 (-1 padded), counts [K] int32. n <= 8.
__global__ __launch_bounds__(64) void select_near_kernel(const float* __restrict__ dist2, const int64_t* __restrict__ assign,
                                                         int Tn, int K, int n, int64_t* __restrict__ picks,
                                                         int* __restrict__ counts) {
    const int k = blockIdx.x, lane = threadIdx.x;
    // the lane's own candidates: its n best (distance, row) pairs, ascending
    float bd[8];
    int bi[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { bd[j] = INFINITY; bi[j] = 0x7fffffff; }
    int cnt = 0;
    for (int t = lane; t < Tn; t += 64) {
        if ((int)assign[t] != k) continue;
        ++cnt;
        float d = dist2[(long)t * K + k];
        int id = t;
#pragma unroll
        for (int j = 0; j < 8; ++j) {              // insertion into the sorted list (rows arrive in ascending order per lane)
            if (j < n && (d < bd[j] || (d == bd[j] && id < bi[j]))) {
                const float td = bd[j]; const int ti = bi[j];
                bd[j] = d; bi[j] = id; d = td; id = ti;
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
    if (lane == 0) counts[k] = cnt < n ? cnt : n;
    if (cnt <= n) {
        // all members, ascending row: rank of each member = members before it
        if (lane == 0)
            for (int j = cnt; j < n; ++j) picks[(long)k * n + j] = -1;        // the unused slots (never written below)
        for (int base = 0, rank = 0; base < Tn; base += 64) {
            const int t = base + lane;
            const bool mine = t < Tn && (int)assign[t] == k;
            const unsigned long long m = __ballot(mine);
            if (mine) picks[(long)k * n + rank + __popcll(m & ((1ull << lane) - 1ull))] = t;
            rank += __popcll(m);
        }
        return;
    }
    // n rounds: the wave's best head-of-list wins and is popped from its lane
    for (int r = 0; r < n; ++r) {
        float d = bd[0];
        int id = bi[0];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float od = __shfl_xor(d, o, 64);
            const int oi = __shfl_xor(id, o, 64);
            if (od < d || (od == d && oi < id)) { d = od; id = oi; }
        }
        if (lane == 0) picks[(long)k * n + r] = id;
        if (bi[0] == id) {                          // pop (rows are unique: exactly one lane holds the winner)
#pragma unroll
            for (int j = 0; j < 7; ++j) { bd[j] = bd[j + 1]; bi[j] = bi[j + 1]; }
            bd[7] = INFINITY; bi[7] = 0x7fffffff;
        }
    }
}

}  // namespace

int cogs_k_select_near(hipStream_t st, const float* dist2, const int64_t* assign, int T, int K, int n, int64_t* picks,
                       int* counts) {
    if (T <= 0 || K <= 0 || n <= 0 || n > 8) return COGS_E_INVALID;
    hipLaunchKernelGGL(select_near_kernel, dim3(K), dim3(64), 0, st, dist2, assign, T, K, n, picks, counts);
    return COGS_LAUNCH_CHECK();
}

// ---- workspace: [A] max(sqdist slice partials [T][ns][K], update shift partials [nblk][K]) floats, then the member
// lists (offs [K+1], members [T]), the update scratch [2K], and the Lloyd loop's own state: dist2 [T][K] floats,
// reseed rows [K], ctl [CTL_WORDS], reseed pool [POOL_MAX], the last assignments [T], centres that have not moved [K] ints
constexpr int POOL_MAX = 4096;
static size_t ws_floats(int T, long PD, int K, int ns) {
    const size_t a = (size_t)ns * T * K;
    const size_t b = (size_t)cogs_k_kmeans_update_blocks(PD) * K;
    return a > b ? a : b;
}
size_t cogs_k_kmeans_ws(int T, long PD, int K, int* nslices) {
    const int ns = (int)((PD + SL - 1) / SL);
    if (nslices) *nslices = ns;
    return (ws_floats(T, PD, K, ns) + (size_t)(K + 1) + (size_t)T + 2 * (size_t)K + (size_t)T * K + (size_t)K + CTL_WORDS + POOL_MAX + (size_t)T + (size_t)K) * 4;
}
namespace {
struct KmWs {
    float* partial; int* offs; int* members; float* scratch; float* dist2; int* reseed; int* ctl; int* pool; int* before; int* keep;
};
KmWs carve(float* ws, int T, long PD, int K) {
    int ns = 0;
    (void)cogs_k_kmeans_ws(T, PD, K, &ns);
    KmWs w;
    w.partial = ws;
    w.offs = (int*)(ws + ws_floats(T, PD, K, ns));
    w.members = w.offs + K + 1;
    w.scratch = (float*)(w.members + T);
    w.dist2 = w.scratch + 2 * K;
    w.reseed = (int*)(w.dist2 + (size_t)T * K);
    w.ctl = w.reseed + K;
    w.pool = w.ctl + CTL_WORDS;
    w.before = w.pool + POOL_MAX;
    w.keep = w.before + T;
    return w;
}

template <typename T>
void launch_sqdist(hipStream_t st, const void* feats, int Tn, long PD, const float* centres, const int* centre_rows,
                   int centre_row, int kb, int k0, int K, float* partial, int nslices, const int* ctl, const int* keep) {
    static std::atomic<uint64_t> done{0};
    cogs_ensure_dyn_lds((const void*)sqdist_kernel<T>, KMAX * SL * 4, done);
    const int kp = (kb + 3) & ~3;
    // row groups on grid.y: as many as keep the whole grid RESIDENT at once (LDS: 2 KiB per centre and workgroup, at most
    // 8 workgroups per CU) -- a grid a few workgroups over that runs a second, nearly empty round (measured at K = 18:
    // 700 workgroups 84 us, 1 050 -> 103 us, 1 400 -> 80 us) -- with at least 16 rows each
    const int per_cu = 80 / kp < 1 ? 1 : (80 / kp > 8 ? 8 : 80 / kp);
    int rg = 256 * per_cu / nslices;
    const int env_rg = (int)g_cogs_debug.km_row_groups;     // experiments
    if (env_rg > 0) rg = env_rg;
    rg = rg < 1 ? 1 : (rg > 8 ? 8 : rg);
    while (rg > 1 && (Tn + rg - 1) / rg < 16) --rg;
    hipLaunchKernelGGL((sqdist_kernel<T>), dim3(nslices, rg), dim3(256), (size_t)kp * SL * 4, st, (const T*)feats, Tn, PD,
                       centres, centre_rows, centre_row, kb, k0, K, partial, ctl, keep);
}
int sqdist_partials(hipStream_t st, int dtype, const void* feats, int T, long PD, const float* centres,
                    const int* centre_rows, int centre_row, int K, float* partial, int nslices, const int* ctl = nullptr, const int* keep = nullptr) {
    if (K <= 0 || T <= 0 || PD % 8) return COGS_E_INVALID;
    if (nslices != (int)((PD + SL - 1) / SL)) return COGS_E_WORKSPACE;
    for (int k0 = 0; k0 < K; k0 += KMAX) {          // the LDS centre slice holds KMAX clusters at a time
        const int kb = K - k0 < KMAX ? K - k0 : KMAX;
        if (dtype == COGS_DT_BF16) launch_sqdist<bf16_t>(st, feats, T, PD, centres, centre_rows, centre_row, kb, k0, K, partial, nslices, ctl, keep);
        else launch_sqdist<float>(st, feats, T, PD, centres, centre_rows, centre_row, kb, k0, K, partial, nslices, ctl, keep);
    }
    return COGS_LAUNCH_CHECK();
}
int launch_reduce_assign(hipStream_t st, const float* partial, int nslices, int T, int K, const float* ts, const float* cts,
                         float alpha, float* dist2, int64_t* assign, int* ctl = nullptr, const int* keep = nullptr) {
    if (K > 4096) return COGS_E_UNSUPPORTED;
    hipLaunchKernelGGL(reduce_assign_kernel, dim3(T), dim3(256), (size_t)256 * 8 + (size_t)K * 4, st, partial, nslices, T, K, ts, cts, alpha, dist2, assign, ctl, keep);
    return COGS_LAUNCH_CHECK();
}
int launch_members(hipStream_t st, const int64_t* assign, int T, int K, const KmWs& w, const int* pool, int pool_len,
                   const int* reseed_in, int* ctl) {
    if (T <= MEMB_T && (size_t)(T + K + 1) * 4 <= 64 * 1024) {
        const int nt = T >= 1024 ? 1024 : ((T + 63) / 64) * 64;
        hipLaunchKernelGGL(members_kernel, dim3(1), dim3(nt < 64 ? 64 : nt), (size_t)(T + K + 1) * 4, st, assign, T, K, w.offs,
                           w.members, pool, pool_len, reseed_in, w.reseed, ctl, w.before, ctl ? w.keep : nullptr, w.scratch);
    } else {
        if (!reseed_in) return COGS_E_UNSUPPORTED;     // the Lloyd loop needs the LDS path (T <= 16 384 rows)
        hipLaunchKernelGGL(members_slow_kernel, dim3(1), dim3(256), 0, st, assign, T, K, w.offs, w.members);
        if (hipMemcpyAsync(w.reseed, reseed_in, (size_t)K * 4, hipMemcpyDeviceToDevice, st) != hipSuccess) return COGS_E_HIP;
    }
    return COGS_LAUNCH_CHECK();
}
int launch_update(hipStream_t st, int dtype, const void* feats, const float* ts, int T, long PD, int K, const KmWs& w,
                  int* ctl, float* centres, float* centre_ts, float* shift_out, volatile int* status, float tol = -1.f, const int* watch = nullptr) {
    const int nblk = cogs_k_kmeans_update_blocks(PD);
    if (dtype == COGS_DT_BF16)
        hipLaunchKernelGGL(update_kernel<bf16_t>, dim3(nblk, K), dim3(256), 0, st, (const bf16_t*)feats, PD, K, w.offs, w.members,
                           w.reseed, ctl, centres, w.partial, ctl ? w.keep : nullptr);
    else
        hipLaunchKernelGGL(update_kernel<float>, dim3(nblk, K), dim3(256), 0, st, (const float*)feats, PD, K, w.offs, w.members,
                           w.reseed, ctl, centres, w.partial, ctl ? w.keep : nullptr);
    const int t_lds = T <= MEMB_T ? T : 0;       // member-ordered time stamps staged in LDS: up to 64 KiB, and 1 KiB of the kernel's own beside them
    static std::atomic<uint64_t> attr_done{0};
    cogs_ensure_dyn_lds((const void*)update_final_kernel, MEMB_T * 4, attr_done);
    hipLaunchKernelGGL(update_final_kernel, dim3(1), dim3(UF_T), (size_t)t_lds * 4, st, ts, K, w.offs, w.members, w.reseed, ctl,
                       centre_ts, w.partial, nblk, w.scratch, shift_out, status, t_lds, tol, watch);
    return COGS_LAUNCH_CHECK();
}
}  // namespace

int cogs_k_kmeans_update_blocks(long PD) { return (int)((PD + UB - 1) / UB); }

int cogs_k_kmeans_sqdist(hipStream_t st, int dtype, const void* feats, int T, long PD, const float* centres,
                         const int* centre_rows, int K, float* ws, int nslices, float* dist2) {
    const KmWs w = carve(ws, T, PD, K);
    const int rc = sqdist_partials(st, dtype, feats, T, PD, centres, centre_rows, -1, K, w.partial, nslices);
    if (rc != COGS_OK) return rc;
    return launch_reduce_assign(st, w.partial, nslices, T, K, nullptr, nullptr, 0.f, dist2, nullptr);
}

int cogs_k_kmeans_assign(hipStream_t st, const float* dist2, const float* ts, const float* centre_ts, int T, int K,
                         float alpha, int64_t* assign, int* counts) {
    if (T <= 0 || K <= 0) return COGS_E_INVALID;
    if (hipMemsetAsync(counts, 0, (size_t)K * sizeof(int), st) != hipSuccess) return COGS_E_HIP;
    hipLaunchKernelGGL(assign_kernel, dim3((T + 255) / 256), dim3(256), 0, st, dist2, ts, centre_ts, T, K, alpha, assign, counts);
    return COGS_LAUNCH_CHECK();
}

int cogs_k_kmeans_update(hipStream_t st, int dtype, const void* feats, const float* ts, int T, long PD, int K,
                         const int64_t* assign, const int* reseed_rows, float* centres, float* centre_ts,
                         float* ws, int nblk, float* shift_out) {
    if (T <= 0 || K <= 0 || PD % 8) return COGS_E_INVALID;
    if (nblk != cogs_k_kmeans_update_blocks(PD)) return COGS_E_WORKSPACE;
    const KmWs w = carve(ws, T, PD, K);
    const int rc = launch_members(st, assign, T, K, w, nullptr, 0, reseed_rows, nullptr);
    if (rc != COGS_OK) return rc;
    return launch_update(st, dtype, feats, ts, T, PD, K, w, nullptr, centres, centre_ts, shift_out, nullptr);
}

// one k-means++ step: distance^2 of every row to feature row `row`, folded into nearest2 (device [T]); the updated
// nearest2 is copied to probs_host (pinned host memory, nullable) and the stream is synchronised when it is given
int cogs_k_kmeans_pp_step(hipStream_t st, int dtype, const void* feats, int T, long PD, int row, int first,
                          float* nearest2, float* probs_host, float* ws, int nslices) {
    if (row < 0 || row >= T) return COGS_E_INVALID;
    const KmWs w = carve(ws, T, PD, 1);
    const int rc = sqdist_partials(st, dtype, feats, T, PD, nullptr, nullptr, row, 1, w.partial, nslices);
    if (rc != COGS_OK) return rc;
    hipLaunchKernelGGL(reduce_min_kernel, dim3((T + 3) / 4), dim3(256), 0, st, w.partial, nslices, T, first, nearest2);
    if (COGS_LAUNCH_CHECK() != COGS_OK) return COGS_E_HIP;
    if (probs_host) {
        if (hipMemcpyAsync(probs_host, nearest2, (size_t)T * 4, hipMemcpyDeviceToHost, st) != hipSuccess) return COGS_E_HIP;
        if (hipStreamSynchronize(st) != hipSuccess) return COGS_E_HIP;
    }
    return COGS_OK;
}

// Which form the passes of the whole seeding take. One launch has a workgroup, and so a CU's intake, per row: it wins where rows are
// about as many as CUs, or short. Fewer long rows leave CUs idle, and long ones are read from L2 with up to four others by every workgroup, where
// sqdist keeps those in LDS: [256, 179 200] bf16 35 to 39 us a pass, 21 and 15 in two launches; behind the last draw a pass is 2 us, or two of them.
// Time of a seeding by slices over one by rows (18 centres of some scenes of twelve rows each, 6 up to 48 rows):        (MI355X)
//                     T = 24    48    80   120   160   200   256   257   300
//   bf16,  28 KB         1.32  1.24  1.28  1.35  1.38  1.40  1.40  1.35  1.32
//   bf16,  84 KB         1.11  1.04  1.09  1.21  1.19  1.27  1.32  1.10  1.10
//   bf16, 128 KB         0.94  1.00  0.99  1.08  1.11  1.14  1.20  0.99  0.99
//   bf16, 168 KB         0.85  0.88  0.99  1.02  1.06  1.18  1.23  0.91  0.97
//   bf16, 350 KB         0.62  0.68  0.76  0.86  0.94  1.00  1.05  0.73  0.82
//   bf16, 896 KB         0.50  0.44  0.56  0.65  0.70  0.76  0.78  0.52  0.50
//   fp32, 128 KB         1.07  1.03  1.06  1.08  1.01  1.07  1.12  1.02  0.99
//   fp32, 350 KB         0.68  0.72  0.67  0.90  0.97  1.00  1.10  0.76  0.85
// and of nearly as many rows as CUs (fp32 rows are half as many values):
//                     T = 193   200   224   240   256
//   bf16, 400 KB         1.00  1.00  1.06  1.03  1.10
//   bf16, 448 KB         0.94  0.97  1.01  1.03  1.07
//   bf16, 512 KB         0.96  0.97  1.02  1.05  1.06
//   bf16, 640 KB         0.92  0.94  0.98  0.98  1.03
//   fp32, 350 KB         1.03  1.04  1.12  1.12  1.13
//   fp32, 416 KB         0.93  0.94  1.00  0.99  1.03
//   fp32, 448 KB         0.91  0.91  0.96  0.96  0.99
//   fp32, 512 KB         0.90  0.91  0.94  0.96  0.99
static bool kpp_in_one_launch(int dtype, int T, long PD) {
    const long kb = PD * (dtype == COGS_DT_BF16 ? 2 : 4) >> 10;
    const bool bf = dtype == COGS_DT_BF16;
    return kb <= 100 ? T <= 300 : T <= 256 && kb <= (T < 100 ? 128 : T <= 192 ? 224 : T < 224 ? (bf ? 400 : 352) : bf ? 512 : 416);
}

// The whole k-means++ seeding (kmeans_with_time.py:41-62) in one call, no host round trip per centre: up to K - 1 passes measure
// every row against the newest centre and guesses of the next ones (rows read from device memory), fold it into nearest2 and draw centre m
// as argmax(probs / q[m-1]) (kpp_draw). 256 frames of 179 200 bf16, 18 centres: 17 launches of 23 us were 388 us, now 205 (17 too, 12 of which return
// at once). q: device fp32 [K-1][T], the Exponential(1) draws the reference's K-1
// torch.multinomial calls would make on the CPU generator, made ahead by the host. idx: device int32 [K], idx[0] given.
// dist2 (nullable) [T][K]: column m - 1 receives the squared distances to centre m - 1, the last column nothing.
// *zero_flag (device int, zeroed here) is set when a step found all probabilities zero -- the reference's
// random.randint branch; the indices from that step on are then meaningless and the caller redoes the seeding step by step.
int cogs_k_kmeans_pp(hipStream_t st, int dtype, const void* feats, int T, long PD, int K, int first_row, const float* q, int* idx,
                     int* zero_flag, float* nearest2, float* dist2, float* ws, size_t ws_bytes, int nslices) {
    if (T <= 0 || K <= 0 || PD % 8 || !q || !idx || !zero_flag || !nearest2 || first_row < 0 || first_row >= T) return COGS_E_INVALID;
    if (nslices != (int)((PD + SL - 1) / SL)) return COGS_E_WORKSPACE;
    const int form = (int)g_cogs_debug.km_pp_form;
    const bool one = form > 0 ? form == 1 && T <= 300 : kpp_in_one_launch(dtype, T, PD);
    // rows a pass measures: what the workspace has room for (one centre's is accepted)
    int C = KPP_C < K ? KPP_C : K;
    while (C > 1 && cogs_k_kmeans_ws(T, PD, C, nullptr) > ws_bytes) --C;
    const KmWs w = carve(ws, T, PD, one ? 1 : C);
    static_assert(KPP_C * 300 <= POOL_MAX, "a row per workgroup: up to 300 rows, their distances in the pool's place");
    if (one) C = KPP_C;
    const KppArgs p{T, K, nearest2, q, idx, zero_flag, w.ctl, one ? (float*)w.pool : w.dist2, C, dist2};
    hipLaunchKernelGGL(kpp_start_kernel, dim3(1), dim3(256), 0, st, p, first_row);
    g_cogs_debug.km_pp_last_launches = one ? 1 : 3;
    const size_t lds = (size_t)nslices * KPP_C * 4;
    for (int m = 1; m < K; ++m) {
        if (!one) {
            const int rc = sqdist_partials(st, dtype, feats, T, PD, nullptr, w.ctl + KPP_ROWS, -1, C, w.partial, nslices, w.ctl);
            if (rc != COGS_OK) return rc;
            hipLaunchKernelGGL(kpp_reduce_kernel, dim3(T), dim3(256), 0, st, w.partial, p, nslices);
        } else if (dtype == COGS_DT_BF16)
            hipLaunchKernelGGL(kpp_pass_kernel<bf16_t>, dim3(T), dim3(KPP_T), lds, st, (const bf16_t*)feats, p, PD, nslices);
        else
            hipLaunchKernelGGL(kpp_pass_kernel<float>, dim3(T), dim3(KPP_T), lds, st, (const float*)feats, p, PD, nslices);
    }
    return COGS_LAUNCH_CHECK();
}

// The Lloyd loop (kmeans_with_time.py:71-131). Centres that have not moved keep their distances (dist2) and means: a cluster that no row has joined
// or left, and in the first iteration the `known` leading centres whose columns of dist2 the caller brings from the seeding (the same fp32 slice sums,
// added up in another fp64 order). 256 frames of 179 200 bf16, 18 centres, two iterations that move and one that does not: distances 3 x 76 us ->
// 23 + 78 + 24, means 3 x 21 -> 20 + 8 + 5; with one launch and one read instead of several the whole clustering 948 -> 843.
// The host queues up to LLOYD_BATCH iterations between two reads of the
// control words (update_final copies them into host-mapped memory): every kernel of an iteration returns at once when an
// earlier one has converged or run the reseed pool dry, so the iterations queued behind the last one change nothing.
// Empty clusters take their rows from `pool`, the host's pre-drawn random.randint values, in the reference's order; if an
// iteration needs more than the pool holds it is not committed and the call returns with *exhausted = 1 (the caller
// draws more and calls again with the remaining budget).
constexpr int LLOYD_BATCH = 4;
namespace {
// host-mapped: [0, 64) the control words as update_final leaves them, [64, 64 + 4 * POOL_MAX) the reseed pool -- the
// device reads the pool in place (only when a cluster runs empty), so a call uploads nothing and frees the caller's
// array the moment it returns
struct StatusBlock { volatile int* h = nullptr; int* d = nullptr; int dev = -1; };
constexpr size_t STATUS_BYTES = 64 + (size_t)POOL_MAX * 4;
// one host-mapped block per calling thread; replaced (and the old one freed) when the thread's device changes
bool status_block(StatusBlock& b) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (b.h && b.dev == dev) return true;
    if (b.h) { (void)hipHostFree((void*)b.h); b.h = nullptr; b.d = nullptr; }
    void* hp = nullptr;
    if (hipHostMalloc(&hp, STATUS_BYTES, hipHostMallocMapped) != hipSuccess) return false;
    void* dp = nullptr;
    if (hipHostGetDevicePointer(&dp, hp, 0) != hipSuccess) { (void)hipHostFree(hp); return false; }
    b.h = (volatile int*)hp; b.d = (int*)dp; b.dev = dev;
    return true;
}
}  // namespace

int cogs_k_kmeans_lloyd(hipStream_t st, int dtype, const void* feats, const float* ts, int T, long PD, int K, float alpha,
                        int max_iter, float tol, const int* pool_host, int pool_len, float* centres, float* centre_ts,
                        int64_t* assign, int* iterations, int* reseeds_used, int* exhausted, float* dist2, int known, const int* watch, CogsKmReport* report, float* ws, int nslices) {
    if (T <= 0 || K <= 0 || PD % 8 || known < 0 || known > K || (known > 0 && !dist2) || max_iter < 0 || pool_len < 0 || pool_len > POOL_MAX) return COGS_E_INVALID;
    if (T > MEMB_T || (size_t)(T + K + 1) * 4 > 64 * 1024 || K > 4096) return COGS_E_UNSUPPORTED;   // T + K + 1 <= 16 384
    static thread_local StatusBlock sb;
    if (!status_block(sb)) return COGS_E_HIP;
    if (iterations) *iterations = 0;
    if (reseeds_used) *reseeds_used = 0;
    if (exhausted) *exhausted = 0;
    if (report) *report = CogsKmReport{INFINITY, 0, 0, 0};
    if (max_iter == 0) return COGS_OK;             // nothing to do
    const KmWs w = carve(ws, T, PD, K);
    if (!dist2) dist2 = w.dist2;
    int* pool_d = sb.d + 16;
    for (int i = 0; i < pool_len; ++i) sb.h[16 + i] = pool_host[i];        // plain host stores into the mapped block
    for (int i = 0; i <= CTL_WORDS; ++i) sb.h[i] = 0;
    hipLaunchKernelGGL(start_kernel, dim3(1), dim3(256), 0, st, w.ctl, w.keep, K, known);     // margin word 0 = +inf
    int queued = 0, it = 0, used = 0, ex = 0;
    int rc = COGS_OK;
    while (queued < max_iter) {
        const int batch = max_iter - queued < LLOYD_BATCH ? max_iter - queued : LLOYD_BATCH;
        for (int b = 0; b < batch && rc == COGS_OK; ++b) {
            rc = sqdist_partials(st, dtype, feats, T, PD, centres, nullptr, -1, K, w.partial, nslices, w.ctl, w.keep);
            if (rc == COGS_OK) rc = launch_reduce_assign(st, w.partial, nslices, T, K, ts, centre_ts, alpha, dist2, assign, w.ctl, w.keep);
            if (rc == COGS_OK) rc = launch_members(st, assign, T, K, w, pool_d, pool_len, nullptr, w.ctl);
            if (rc == COGS_OK) rc = launch_update(st, dtype, feats, ts, T, PD, K, w, w.ctl, centres, centre_ts, (float*)(w.ctl + CTL_SHIFT),
                                                  (volatile int*)sb.d, tol, watch);
        }
        queued += batch;
        if (hipStreamSynchronize(st) != hipSuccess) return COGS_E_HIP;
        if (rc != COGS_OK) return rc;
        it = sb.h[CTL_ITERS];
        used = sb.h[CTL_USED];
        if (sb.h[CTL_ABORT]) { ex = 1; break; }      // the aborted iteration was not committed
        if (sb.h[CTL_DONE]) break;
    }
    if (iterations) *iterations = it;
    if (reseeds_used) *reseeds_used = used;
    if (exhausted) *exhausted = ex;
    if (report) *report = CogsKmReport{__builtin_bit_cast(float, 0x7f800000 - sb.h[CTL_MARGIN]), sb.h[CTL_NEAR], sb.h[CTL_WORDS], 1};
    return COGS_OK;
}

// how close the assignments of the last cogs_k_kmeans_lloyd call on this workspace were: the smallest relative margin
// (second-best - best) / best of the final distance over all rows and iterations, and the number of (row, iteration)
// pairs below 1e-3 -- below that the reference's own cdist rounding decides the row
int cogs_k_kmeans_margins(hipStream_t st, int T, long PD, int K, float* ws, float* min_margin, int* rows_below) {
    const KmWs w = carve(ws, T, PD, K);
    int h[CTL_WORDS];
    if (hipMemcpyAsync(h, w.ctl, sizeof(h), hipMemcpyDeviceToHost, st) != hipSuccess) return COGS_E_HIP;
    if (hipStreamSynchronize(st) != hipSuccess) return COGS_E_HIP;
    if (min_margin) *min_margin = __builtin_bit_cast(float, 0x7f800000 - h[CTL_MARGIN]);
    if (rows_below) *rows_below = h[CTL_NEAR];
    return COGS_OK;
}
