// Gated delta rule (cogs_delta_mixer): per head a matrix S [dk][dv] carried from token to token,
//
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q.
//
// Everything here is fp32, whatever the model's dtype: the fused projection's output t, the convolution's memory, S, and all products.
//   prompts   delta_inputs (convolution, silu, unit vectors, beta, ln g) -> delta_chunk + delta_scan (32 tokens at a time on the fp32
//             matrix instructions; workgroups behind the scan's keep the convolution's last inputs) -> delta_out (norm and gate)
//   decode    delta_step: one launch per layer does all of it
// A token-by-token kernel (delta_recur) serves the sizes the chunked pair has no instance for.
//
// Chunks. With G_i = sum of ln g over the chunk's tokens 0 .. i and S0 the state in front of it,
//   u_i = beta_i (v_i - e^{G_i} S0^T k_i - sum_{j<i} e^{G_i - G_j} (k_i . k_j) u_j),  i.e.  U = T diag(beta) (V - diag(e^G) K S0)
//   with T = (I + L)^-1, L_ij = beta_i e^{G_i - G_j} k_i . k_j (j < i);   O = diag(e^G) Q S0 + P U with P_ij = e^{G_i - G_j} q_i . k_j (j <= i);
//   S = e^{G_last} S0 + K^T diag(e^{G_last - G_j}) U.
// Only exponentials of differences of later minus earlier sums appear (<= 1); the sums themselves are fp64. T diag(beta), P and the
// exponentials do not depend on S: delta_chunk forms them for all chunks at once, T by forward substitution. delta_scan walks a
// sequence's chunks: a workgroup owns 16 columns of S, its four waves the 16-row tiles of S in turn.
// The scan's chunks follow one another, so what counts is the length of one: K S, a sum over the waves, the product with T, the new
// state. Operands in the order of the lanes and buffer loads without address arithmetic took it from 2.1 to 1.4 us a chunk, 3400 cycles. 63 matrix
// instructions are 2000 of them, the loads 300 (a chunk over and over in registers: 3100); the rest are some hundred vector instructions, which do not run
// beside fp32 matrix instructions, and the exchange through LDS.
// MFMA layout: a 16x16 accumulator holds rows 4 g + r in register r of lane group g, which is the B operand of the r-th of four
// 4-deep steps if k is taken in the order 4 g + r -- so S, V - diag(e^G) K S and U go from product to product in their registers, and A operands are
// 16-byte loads of four neighbouring k.
#include "common.h"
#include "kernels.h"
#include "debug.h"

namespace {

constexpr int CH = 32;                        // tokens of a chunk
constexpr int TILE = 256;                     // floats of a 16x16 tile, row-major
constexpr int EXPS = 6 * TILE;                // per chunk and head: P tiles (0,0) (1,0) (1,1) | T beta tiles | e^G | e^{G_last - G} | e^{G_last}, ..;
constexpr int REC = EXPS + 3 * CH;            // P as A operands [4 steps][64 lanes], T beta as [64 lanes][4 steps]

// Chunks have q, k and v as the operands of the scan's 16x16 tiles, [chunk][16 tokens a][16 columns t][64 lanes][4 floats]: q and k with a token per lane
// (lane 16 g + li: token li, columns 4 g ..), k once more and v with a column per lane (column li, tokens 4 g ..). A sequence starts on a chunk of
// its own; tokens past its end are zeros, or read as such (p.pad, cogs_k_delta_prompt). An operand is one load of 1 KiB in a row, 25 of them a wave and chunk; as rows it was sixteen lines of 64 bytes, and those
// with a column per lane four loads of 4 bytes a lane, 43 in all. 4096 rows, 16 heads of 128: scan 206 -> 198 us, 32 heads 242 -> 227 and the chunks
// 57 -> 49; the inputs 31 -> 36 (k is written twice). Prompts of 4096 rows, width 2048 5021 -> 4963 us, of 700 1450 -> 1428, of 300, width 4096
// 2101 -> 2081. (T, v and the exponentials, which all four waves read, through LDS instead of into each one's registers: 206 again.)
__device__ __forceinline__ int token_major(int tiles, int a, int row, int c) {      // first of four columns c ..
    return (a * tiles + (c >> 4)) * TILE + (((c & 15) >> 2) * 16 + row) * 4 + (c & 3);
}
__device__ __forceinline__ int column_major(int tiles, int a, int row, int c) {     // first of four rows
    return (a * tiles + (c >> 4)) * TILE + ((row >> 2) * 16 + (c & 15)) * 4 + (row & 3);
}
// floats in front of a chunk of a head of n columns (a later sequence starts behind the chunks of an earlier one)
__device__ __forceinline__ long chunk_at(const CogsDelta& p, const CogsSeq& s, int seq, int chunk, int head, int n) {
    return ((long)head * p.slots + s.row0 / CH + seq + chunk) * CH * n;
}
// four lanes' four values each, transposed
__device__ __forceinline__ void quad_transpose(f32x4& v, int lane) {
#pragma unroll
    for (int b = 1; b <= 2; b *= 2) {
        const bool up = lane & b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i & b) continue;
            const float lo = v[i], hi = v[i + b], give = up ? lo : hi;
            const float got = b == 1 ? lane_xor_dpp<1>(give) : lane_xor_dpp<2>(give);
            v[i] = up ? got : lo;
            v[i + b] = up ? hi : got;
        }
    }
}

__device__ __forceinline__ float unit_scale(float ss) { return 1.f / sqrtf(ss + 1e-6f); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// convolution + silu of channel c at position pos; `back` input rows (stride ldt) lie in front of x, older ones in the ring
__device__ __forceinline__ float conv_silu(const CogsDelta& p, const float* x, const float* ring, int c, int pos, int back) {
    float y = p.conv[(long)(p.taps - 1) * p.channels + c] * x[c];
    for (int j = 1; j < p.taps; ++j) {
        if (j > pos) break;
        const float v = j <= back ? x[c - (long)j * p.ldt] : ring[(long)((pos - j) % p.taps) * p.channels + c];
        y = fmaf(p.conv[(long)(p.taps - 1 - j) * p.channels + c], v, y);
    }
    return y / (1.f + expf(-y));
}

// quick silu: the activation behind a short convolution
__device__ __forceinline__ float silu_q(float y) { return y * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * y)); }

// RUN consecutive rows of a sequence at a time: a wave walks one q / k head, or 64 E channels of v, or the heads' beta and ln g, with
// the convolution's window in registers and the whole run's inputs requested ahead. E: 64-channel steps of a head; TAPS: taps, rounded up
template <int E, int TAPS, int RUN>
__global__ __launch_bounds__(256) void delta_inputs_kernel(CogsDelta p) {
    const int seq = blockIdx.z;
    const CogsSeq s = p.seqs[seq];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i0 = blockIdx.x * RUN, n = min(RUN, s.len - i0);
    if (n <= 0 && (!p.pad || i0 >= (s.len + CH - 1) / CH * CH)) return;      // (runs of zeros behind the end belong to its chunk)
    const int stored = p.pad ? RUN : n;                        // tokens
    const int nqk = 2 * p.kv_heads, nv = p.heads * p.dvp, units = nqk + (nv + 64 * E - 1) / (64 * E);
    const int unit = blockIdx.y * 4 + wid, v0 = nqk * p.dkp;
    const long row0 = s.row0 + i0;
    const float* x = p.t + row0 * p.ldt;
    if (unit > units) return;
    if (unit == units) {
        const float *tb = x + v0 + 2 * nv, *ta = tb + p.headsp;
        for (int i = lane; i < n * p.heads; i += 64) {
            const int r = i / p.heads, h = i - r * p.heads;
            p.bg[(row0 * p.heads + i) * 2] = sigmoid_f(tb[(long)r * p.ldt + h]);
            p.bg[(row0 * p.heads + i) * 2 + 1] = p.neg_a[h] * softplus_f(ta[(long)r * p.ldt + h] + p.dt_bias[h]);
        }
        return;
    }
    const bool is_v = unit >= nqk;
    const int c0 = is_v ? v0 + (unit - nqk) * 64 * E : unit * p.dkp, size = is_v ? min(64 * E, v0 + nv - c0) : p.dkp;
    const float* ring = s.state + p.state_off + (long)p.heads * p.dkp * p.dvp;
    float w[TAPS][E], in[TAPS - 1 + RUN][E];          // in[TAPS - 1 + r]: row i0 + r
    int ch[E];
#pragma unroll
    for (int e = 0; e < E; ++e) ch[e] = c0 + min(lane + 64 * e, size - 1);
#pragma unroll
    for (int r = 0; r < RUN; ++r)
#pragma unroll
        for (int e = 0; e < E; ++e) in[TAPS - 1 + r][e] = x[(long)min(r, n - 1) * p.ldt + ch[e]];      // (n <= 0: the sequence's last row)
#pragma unroll
    for (int j = 1; j < TAPS; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = i0 - j, pos = s.pos0 + i;
            float v = 0.f;
            if (j < p.taps && pos >= 0 && n > 0) v = i >= 0 ? x[ch[e] - (long)j * p.ldt] : ring[(long)(pos % p.taps) * p.channels + ch[e]];
            in[TAPS - 1 - j][e] = v;
        }
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) w[j][e] = j < p.taps ? p.conv[(long)(p.taps - 1 - j) * p.channels + ch[e]] : 0.f;
    const float scale = unit < p.kv_heads ? p.q_scale : 1.f;
    f32x4 y[RUN / 4][E];
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float a = w[0][e] * in[TAPS - 1 + r][e];
#pragma unroll
            for (int j = 1; j < TAPS; ++j) a = fmaf(w[j][e], in[TAPS - 1 + r - j][e], a);
            const float v = lane + 64 * e < size ? silu_q(a) : 0.f;
            ss = fmaf(v, v, ss);
            y[r >> 2][e][r & 3] = v;
        }
        const float f = is_v ? 1.f : unit_scale(wave_sum(ss)) * scale;
#pragma unroll
        for (int e = 0; e < E; ++e) y[r >> 2][e][r & 3] = r < n ? y[r >> 2][e][r & 3] * f : 0.f;
    }
    const int a = (i0 >> 4) & 1, first = i0 & 15;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool mine = lane + 64 * e < size;
        const int c = ch[e] - (is_v ? v0 : c0), width = is_v ? p.dvp : p.dkp, head = is_v ? c / width : unit % p.kv_heads, col = is_v ? c - head * width : c;
        const long at = chunk_at(p, s, seq, i0 / CH, head, width);      // (v's pieces may cross heads)
        float* const by_column = is_v ? p.v : p.kt;
#pragma unroll
        for (int q = 0; q < RUN / 4; ++q) {
            f32x4 v = y[q][e];
            if (mine && 4 * q < stored && unit >= p.kv_heads) *reinterpret_cast<f32x4*>(by_column + at + column_major(width >> 4, a, first + 4 * q, col)) = v;
            if (is_v) continue;
            quad_transpose(v, lane);
            if (mine && 4 * q + (lane & 3) < stored) *reinterpret_cast<f32x4*>((unit < p.kv_heads ? p.q : p.k) + at + token_major(width >> 4, a, first + 4 * q + (lane & 3), col & ~3)) = v;
        }
    }
}

// the same for any size: one workgroup per new row; a wave per q / k head
template <bool TILES>
__global__ __launch_bounds__(256) void delta_inputs_any_kernel(CogsDelta p) {
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int sq = p.rowseq[row], pos = p.rowpos[row];
    const CogsSeq s = p.seqs[sq];
    const int i = row - s.row0, chunk = i / CH;
    const int after = TILES && i == s.len - 1 ? (p.pad ? (i / CH + 1) * CH - s.len : 3 - (i & 3)) : 0;       // rows of zeros that this one is followed by
    const float* x = p.t + (long)row * p.ldt;
    const float* ring = s.state + p.state_off + (long)p.heads * p.dkp * p.dvp;
    const int back = row - s.row0;
    for (int j = wid; j < 2 * p.kv_heads; j += 4) {
        float v[8], ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int d = lane + 64 * e;
            v[e] = d < p.dkp ? conv_silu(p, x, ring, j * p.dkp + d, pos, back) : 0.f;
            ss += v[e] * v[e];
        }
        float f = unit_scale(wave_sum(ss));
        if (j < p.kv_heads) f *= p.q_scale;
        float* o = j < p.kv_heads ? p.q : p.k;
        const int head = j % p.kv_heads;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int d = lane + 64 * e;
            if (d >= p.dkp) continue;
            if constexpr (TILES) {
                const long at = chunk_at(p, s, sq, chunk, head, p.dkp);
                for (int z = 0; z <= after; ++z) {
                    const int r = i + z, b = (r >> 4) & 1;
                    const float y = z ? 0.f : v[e] * f;
                    if (z == 0 || p.pad) o[at + token_major(p.dkp >> 4, b, r & 15, d)] = y;
                    if (j >= p.kv_heads) p.kt[at + column_major(p.dkp >> 4, b, r & 15, d)] = y;
                }
            } else o[((long)head * p.rows + row) * p.dkp + d] = v[e] * f;
        }
    }
    const int v0 = 2 * p.kv_heads * p.dkp, nv = p.heads * p.dvp;
    for (int c = tid; c < nv; c += 256) {
        const float y = conv_silu(p, x, ring, v0 + c, pos, back);
        const int head = c / p.dvp, d = c - head * p.dvp;
        if constexpr (TILES) {
            const long at = chunk_at(p, s, sq, chunk, head, p.dvp);
            for (int z = 0; z <= after; ++z) p.v[at + column_major(p.dvp >> 4, ((i + z) >> 4) & 1, (i + z) & 15, d)] = z ? 0.f : y;
        } else p.v[((long)head * p.rows + row) * p.dvp + d] = y;
    }
    const float *tb = x + v0 + 2 * nv, *ta = tb + p.headsp;
    for (int h = tid; h < p.heads; h += 256) {
        p.bg[((long)row * p.heads + h) * 2] = sigmoid_f(tb[h]);
        p.bg[((long)row * p.heads + h) * 2 + 1] = p.neg_a[h] * softplus_f(ta[h] + p.dt_bias[h]);
    }
}

// the last inputs of the convolution into the ring (behind every reader of the old ones)
__device__ __forceinline__ void conv_tail(const CogsDelta& p, const CogsSeq& s, int block, int blocks) {
    float* ring = s.state + p.state_off + (long)p.heads * p.dkp * p.dvp;
    const int n = min(s.len, p.taps);
    for (int i = block * 256 + threadIdx.x; i < n * p.channels; i += blocks * 256) {
        const int r = s.len - n + i / p.channels, c = i % p.channels;
        ring[(long)((s.pos0 + r) % p.taps) * p.channels + c] = p.t[(long)(s.row0 + r) * p.ldt + c];
    }
}

__global__ __launch_bounds__(256) void delta_tail_kernel(CogsDelta p) { conv_tail(p, p.seqs[blockIdx.y], blockIdx.x, gridDim.x); }

// token by token, a thread per column of S, S in memory
__global__ __launch_bounds__(64) void delta_recur_kernel(CogsDelta p) {
    const int h = blockIdx.y, col = blockIdx.x * 64 + threadIdx.x;
    const CogsSeq s = p.seqs[blockIdx.z];
    if (col >= p.dvp) return;
    float* S = s.state + p.state_off + (long)h * p.dkp * p.dvp + col;
    const int kh = h / (p.heads / p.kv_heads);
    for (int i = 0; i < s.len; ++i) {
        const long row = s.row0 + i;
        const bool fresh = s.pos0 + i == 0;
        const float *q = p.q + ((long)kh * p.rows + row) * p.dkp, *k = p.k + ((long)kh * p.rows + row) * p.dkp;
        const float beta = p.bg[(row * p.heads + h) * 2], g = expf(p.bg[(row * p.heads + h) * 2 + 1]);
        float a = 0.f;
        if (!fresh)
            for (int d = 0; d < p.dkp; ++d) a = fmaf(S[(long)d * p.dvp] * g, k[d], a);
        const float u = beta * (p.v[((long)h * p.rows + row) * p.dvp + col] - a);
        float o = 0.f;
        for (int d = 0; d < p.dkp; ++d) {
            const float v = fmaf(k[d], u, fresh ? 0.f : S[(long)d * p.dvp] * g);
            S[(long)d * p.dvp] = v;
            o = fmaf(v, q[d], o);
        }
        p.o[((long)h * p.rows + row) * p.dvp + col] = o;
    }
}

// A or B operands of four 4-deep steps: 16 rows (stride ld) of 16 columns
__device__ __forceinline__ f32x4 frag(const float* m, long ld, int li, int g) { return *reinterpret_cast<const f32x4*>(m + li * ld + 4 * g); }

__device__ __forceinline__ f32x4 mfma4(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
    return c;
}

__device__ __forceinline__ float* chunk_rec(const CogsDelta& p, const CogsSeq& s, int seq, int chunk, int h) {
    return p.rec + ((long)(s.row0 / CH + seq + chunk) * p.heads + h) * REC;      // (a later sequence starts behind the chunks of an earlier one)
}

// What a chunk needs besides S and V: P, T diag(beta) and the exponentials. Three waves take a tile (0,0), (1,0), (1,1) each of the
// 32 x 32 matrices.
__global__ __launch_bounds__(256) void delta_chunk_kernel(CogsDelta p) {
    __shared__ double cum[CH];
    __shared__ __attribute__((aligned(16))) float beta_s[CH], eg_s[CH];
    __shared__ __attribute__((aligned(16))) float L10[16][20], Ts[3][16][20];
    const int chunk = blockIdx.x, h = blockIdx.y, seq = blockIdx.z;
    const CogsSeq s = p.seqs[seq];
    const int n = min(CH, s.len - chunk * CH);
    if (n <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
    // the waves' roles go round from workgroup to workgroup: the k-th waves of all of a compute unit's workgroups share a SIMD
    const int turn = (blockIdx.y * gridDim.x + blockIdx.x) >> 8;
    const int wid = (__builtin_amdgcn_readfirstlane(tid >> 6) + turn + blockIdx.x) & 3;
    const long row0 = s.row0 + chunk * CH;
    const int kh = h / (p.heads / p.kv_heads);
    const float* K = p.k + chunk_at(p, s, seq, chunk, kh, p.dkp);
    const float* Q = p.q + chunk_at(p, s, seq, chunk, kh, p.dkp);
    float* rec = chunk_rec(p, s, seq, chunk, h);
    const int ta = wid > 0 ? 1 : 0, tb = wid == 2 ? 1 : 0;
    if (wid == 3 && lane < CH) {
        const int r = min(lane, n - 1);
        const float* bg = p.bg + ((row0 + r) * p.heads + h) * 2;
        beta_s[lane] = bg[0];
        double sum = lane < n ? (double)bg[1] : 0.0;
#pragma unroll
        for (int o = 1; o < CH; o *= 2) {
            const double before = __shfl_up(sum, o, CH);
            if (lane >= o) sum += before;
        }
        cum[lane] = sum;
        eg_s[lane] = expf((float)sum);
    }
    f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
    if (wid < 3) {
        const int da = 16 * p.dkp * ta + 4 * lane, db = 16 * p.dkp * tb + 4 * lane;
        for (int d = 0; d < p.dkp; d += 64) {          // four 16-wide steps in flight; steps past the end are not multiplied
            f32x4 a[4], b[4], q[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = 16 * min(d + 16 * e, p.dkp - 16);
                a[e] = *reinterpret_cast<const f32x4*>(K + da + o);
                b[e] = *reinterpret_cast<const f32x4*>(K + db + o);
                q[e] = *reinterpret_cast<const f32x4*>(Q + da + o);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (d + 16 * e >= p.dkp) break;
                kk = mfma4(a[e], b[e], kk);
                qk = mfma4(q[e], b[e], qk);
            }
        }
    }
    __syncthreads();
    if (wid < 3) {
        const int j = 16 * tb + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ta + 4 * g + r;
            const float e = j <= i ? expf((float)(cum[i] - cum[j])) : 0.f;
            const bool in = i < n && j < n;
            kk[r] = in && j < i ? beta_s[i] * e * kk[r] : 0.f;                   // L
            rec[wid * TILE + (li & 3) * 64 + (li >> 2) * 16 + 4 * g + r] = in && j <= i ? e * qk[r] : 0.f;      // [step][lane] of the scan's A operands
        }
    } else if (lane < CH) {
        rec[EXPS + lane] = eg_s[lane];
        rec[EXPS + CH + lane] = lane < n ? expf((float)(cum[CH - 1] - cum[lane])) : 0.f;
        if (lane == 0) rec[EXPS + 2 * CH] = eg_s[CH - 1];
    }
    if (wid == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) L10[4 * g + r][li] = kk[r];
    } else if (wid < 3) {                              // inverse of a diagonal block: a lane per column, L from its registers
        float z[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] = i == li ? 1.f : 0.f;
#pragma unroll
        for (int m = 0; m < 15; ++m)
#pragma unroll
            for (int i = m + 1; i < 16; ++i)
                z[i] = fmaf(-__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(kk[i & 3]), (i >> 2) * 16 + m)), z[m], z[i]);
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; ++i) Ts[wid][i][lane] = z[i];
    }
    __syncthreads();
    // T(1,0) = -T(1,1) L(1,0) T(0,0)
    if (wid == 0) {
        f32x4 b, m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r] = Ts[0][4 * g + r][li];
        m = mfma4(frag(&L10[0][0], 20, li, g), b, m);
        f32x4 t = mfma4(frag(&Ts[2][0][0], 20, li, g), m, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int r = 0; r < 4; ++r) Ts[1][4 * g + r][li] = -t[r];
    }
    __syncthreads();
    if (wid < 3) {                                     // T diag(beta): row li, tokens 4 g + r
        const int i = 16 * ta + li, j = 16 * tb + 4 * g;
        f32x4 t = frag(&Ts[wid][0][0], 20, li, g) * *reinterpret_cast<const f32x4*>(beta_s + j);
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = i < n && j + r < n ? t[r] : 0.f;
        *reinterpret_cast<f32x4*>(rec + (3 + wid) * TILE + 4 * lane) = t;
    }
}

// what a wave needs of one chunk
template <int NK>
struct ScanIn {
    f32x4 k[2][NK], q[2][NK], kt[2][NK], eg[2], ec[2], tm[3], v[2];
    float pm[3], gl;
};

// NK: 16-row tiles of S per wave. A chunk: K S in partial sums over the waves' rows of S that meet in LDS (one barrier); while they do,
// Q S; then R = V - diag(e^G) K S and U = T diag(beta) R, which every wave forms whole, the new state and, beside it, a quarter of P U per
// wave into the partial read-outs. Those ride on the next chunk's barrier, and every wave finishes a quarter of them behind it. One wave per
// SIMD issues in order, so everything else -- the next chunk's loads, scaling, sums -- stands between matrix instructions that do not
// need it (sched_barrier keeps it there). R comes first and is multiplied then: where keys recur the state already predicts V, R is small
// against both, and so is what rounding T and the product add. (As T diag(beta) V + W S, with W = -T diag(beta) diag(e^G) K ahead of the
// scan, 54 instead of 63 matrix instructions, two terms of V's size were rounded and cancelled: read-outs of 8 recurring pairs were off
// by 1.2e-7 of them instead of 8.2e-8, values read back from the state by 1.2e-7 instead of 3.5e-8.) K S and Q S are two chains each, and
// P U and the state's growth sums of their own: chained to what they are added to, they were rounded at its size.
// MASK: tokens past a sequence's end are not there, but for zeros up to the next fourth one (a lane's own); their lanes read behind the buffers' sizes.
// The workgroups from `scan` on keep the convolution's last inputs, which nothing here reads: a launch for them alone, between the inputs and
// the chunks, was 4.9 us a layer (prompts of 100 rows, width 2048 815 -> 793 us, of 4096 5048 -> 5022).
template <int NK, bool MASK>
__global__ __launch_bounds__(256, NK > 2 ? 1 : 2) void delta_scan_kernel(CogsDelta p, int scan) {
    __shared__ __attribute__((aligned(16))) f32x4 red[2][4][4][64];
    const int seq = blockIdx.z;
    const CogsSeq s = p.seqs[seq];
    if ((int)blockIdx.x >= scan) { conv_tail(p, s, blockIdx.x - scan, gridDim.x - scan); return; }
    // workgroups go round the XCDs: the columns of a head stay on one, whose L2 then serves its K and Q once
    const int ng = p.dvp >> 4, place = blockIdx.x >> 3, h = (blockIdx.x & 7) + 8 * (place / ng), col0 = (place % ng) * 16;
    if (h >= p.heads) return;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), half = wid & 1, fin = wid >> 1;
    const int kh = h / (p.heads / p.kv_heads);
    const int ld = p.dkp, ldv = p.dvp;
    float* O = p.o + ((long)h * p.rows + s.row0) * ldv + col0;
    float* S = s.state + p.state_off + (long)h * p.dkp * p.dvp + col0 + li;
    const int tiles = p.dkp >> 4;
    f32x4 st[NK];
    int tn[NK];                                  // tiles past the end repeat the last one, and their S stays zero
#pragma unroll
    for (int n = 0; n < NK; ++n) {
        st[n] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int t = wid + 4 * n;
        tn[n] = min(t, tiles - 1);
        if (t < tiles && s.pos0 > 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) st[n][r] = S[(long)(16 * t + 4 * g + r) * p.dvp];
    }
    const int nc = (s.len + CH - 1) / CH;
    // a lane's places in a chunk's tiles and read-outs (bytes)
    int oo[2];
    const int tmo = lane * 16, po = lane * 4 + wid * 256, ego = 16 * g;
    int tok[2] = {tmo, tmo}, col[2] = {tmo, tmo};      // ... of tiles with a token, and with a column per lane
    auto mask = [&](int rows) {
        if constexpr (MASK)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                tok[a] = 16 * a + li < rows ? tmo : 1 << 30;
                col[a] = 16 * a + 4 * g < rows ? tmo : 1 << 30;
            }
    };
    mask(s.len);
    int zo = 0;
    asm("" : "+v"(zo));                          // (a scalar load would share its counter with LDS)
#pragma unroll
    for (int r = 0; r < 2; ++r) oo[r] = ((16 * fin + 4 * g + 2 * half + r) * ldv + li) * 4;
    // buffer loads: a scalar base per array and chunk, a lane's place, a scalar piece -- no address arithmetic per load; K's columns of a tile
    // past S's end lie behind the buffer's size and read as zero
    struct From { float *k, *q, *kt, *v, *rec; };
    const long qk0 = chunk_at(p, s, seq, 0, kh, ld);
    const From f0{p.k + qk0, p.q + qk0, p.kt + qk0, p.v + chunk_at(p, s, seq, 0, h, ldv) + col0 * 16, chunk_rec(p, s, seq, 0, h)};
    From f = f0;
    constexpr int bytes_rec = REC * 4;
    const int bytes_q = CH * ld * 4, bytes_v = CH * ldv * 4 - col0 * 64;
    int bytes_k[NK];
#pragma unroll
    for (int n = 0; n < NK; ++n) bytes_k[n] = wid + 4 * n < tiles ? bytes_q : 0;
    auto at4 = [](float* base, int size, int lane_off, int off) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(__builtin_amdgcn_make_buffer_rsrc(base, 0, size, 0x00020000), lane_off, off, 0));
    };
    auto at1 = [](float* base, int size, int lane_off, int off) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(__builtin_amdgcn_make_buffer_rsrc(base, 0, size, 0x00020000), lane_off, off, 0));
    };
    const long step_k = (long)CH * ld, step_v = (long)CH * ldv, step_rec = (long)p.heads * REC;
    int at = 0;                                                // the chunk f points to
    auto advance = [&] {                                       // (the last chunk is loaded again rather than nothing)
        at = min(at + 1, nc - 1);
        f = From{f0.k + at * step_k, f0.q + at * step_k, f0.kt + at * step_k, f0.v + at * step_v, f0.rec + at * step_rec};
        mask(s.len - at * CH);
    };
    // load i of a chunk, in the order of their use, the 16-byte ones first
    constexpr int L_Q = 2 * NK, L_E = L_Q + 2 * NK, L_T = L_E + 4, L_V = L_T + 3, L_KT = L_V + 2, L_G = L_KT + 2 * NK, L_PM = L_G + 1, L_ALL = L_PM + 3;
    auto load = [&](ScanIn<NK>& in, int i) __attribute__((always_inline)) {
        auto tile = [&](int j) { return (j / NK * tiles + tn[j % NK]) * TILE * 4; };
        if (i < L_Q) in.k[i / NK][i % NK] = at4(f.k, bytes_q, tok[i / NK], tile(i));
        else if (i < L_E) { const int j = i - L_Q; in.q[j / NK][j % NK] = at4(f.q, bytes_q, tok[j / NK], tile(j)); }
        else if (i < L_T) { const int j = i - L_E; (j & 2 ? in.ec : in.eg)[j & 1] = at4(f.rec, bytes_rec, ego, (EXPS + (j & 2 ? CH : 0) + 16 * (j & 1)) * 4); }
        else if (i < L_V) in.tm[i - L_T] = at4(f.rec, bytes_rec, tmo, (3 + i - L_T) * TILE * 4);
        else if (i < L_KT) { const int j = i - L_V; in.v[j] = at4(f.v, bytes_v, col[j], j * ldv * 64); }
        else if (i < L_G) { const int j = i - L_KT; in.kt[j / NK][j % NK] = at4(f.kt, bytes_k[j % NK], col[j / NK], tile(j)); }
        else if (i < L_PM) in.gl = at1(f.rec, bytes_rec, zo, (EXPS + 2 * CH) * 4);
        else if (i < L_ALL) in.pm[i - L_PM] = at1(f.rec, bytes_rec, po, (i - L_PM) * TILE * 4);
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 y[2] = {zero, zero};                                 // the previous chunk's read-outs, this wave's part of the sums
    auto gather = [&](f32x2 (&o)[4], f32x4 (*rd)[4][64]) {
#pragma unroll
        for (int w = 0; w < 4; ++w) o[w] = *(reinterpret_cast<const f32x2*>(&rd[w][2 + fin][lane]) + half);
    };
    auto finish = [&](int c, const f32x2 (&o)[4], bool ragged) {
        float* oc = O + (long)c * CH * ldv;
        const f32x2 t = (o[0] + o[1]) + (o[2] + o[3]);
#pragma unroll
        for (int r = 0; r < 2; ++r)
            if (!ragged || c * CH + 16 * fin + 4 * g + 2 * half + r < s.len) *reinterpret_cast<float*>(reinterpret_cast<char*>(oc) + oo[r]) = t[r];
    };
    auto meet = [&] {                                          // (loads of later chunks stay in flight)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto mfma = [](float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
    auto mine = [&](const f32x4& v) { return wid < 2 ? (wid == 0 ? v[0] : v[1]) : (wid == 2 ? v[2] : v[3]); };
    auto pin = [](f32x4 (&v)[4]) { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])); };      // (used from here on, no earlier)
    // chunk c from `in`, the next one into nx
    auto chunk = [&](int c, const ScanIn<NK>& in, ScanIn<NK>& nx) __attribute__((always_inline)) {
        constexpr int STEPS = 24 * NK + 12;                    // matrix instructions that bring loads with them
        constexpr int LONG = L_G, WORK = L_ALL + LONG;         // the four waves' 16-byte loads take the time of two matrix instructions, the others half
        static_assert(WORK <= 2 * STEPS);
        int step = 0, next = 0;
        auto due = [&] { return next < L_ALL && (next + min(next, LONG)) * STEPS < (step + 1) * WORK; };
        auto feed = [&] {
            if (due()) load(nx, next++);
            if (due()) load(nx, next++);
            ++step;
            __builtin_amdgcn_sched_barrier(0);
        };
        f32x4 (*rd)[4][64] = red[c & 1];
        f32x4 x[2], o[2], odd;
        auto qs = [&](int a, int i) {
            f32x4& t = i & 1 ? odd : o[a];
            t = mfma(in.q[a][i >> 2][i & 3], st[i >> 2][i & 3], i < 2 ? zero : t);
            if (i == 4 * NK - 1) o[a] += odd;
            feed();
        };
#pragma unroll
        for (int a = 0; a < 2; ++a) {                          // (one 16 rows after the other: the first ones' sums travel meanwhile)
#pragma unroll
            for (int i = 0; i < 4 * NK; ++i) {
                f32x4& t = i & 1 ? odd : x[a];
                t = mfma(in.k[a][i >> 2][i & 3], st[i >> 2][i & 3], i < 2 ? zero : t);
                if (i == 0 && a == 0) advance();
                if (i == 1) rd[wid][a == 0 ? 2 : 3][lane] = y[a];
                if (i == 2 && a == 1) rd[wid][0][lane] = x[0];
                feed();
            }
            x[a] += odd;
        }
        qs(0, 0);
        rd[wid][1][lane] = x[1];
        qs(0, 1);
        qs(0, 2);
        meet();
        f32x4 part[2][4], rr[2], u[2], u10, ue[2], grow[NK];
        f32x2 fo[4];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int w = 0; w < 4; ++w) part[a][w] = rd[w][a][lane];
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 3; i < 8 * NK; ++i) {
            qs(i / (4 * NK), i % (4 * NK));
            if (i == 8 * NK - 3) { pin(part[0]); rr[0] = in.v[0] - in.eg[0] * ((part[0][0] + part[0][1]) + (part[0][2] + part[0][3])); }
            if (i == 8 * NK - 2) { pin(part[1]); rr[1] = in.v[1] - in.eg[1] * ((part[1][0] + part[1][1]) + (part[1][2] + part[1][3])); }
            if (i == 8 * NK - 1) gather(fo, rd);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) { u[0] = mfma(in.tm[0][r], rr[0][r], r < 1 ? zero : u[0]); feed(); }
#pragma unroll
        for (int r = 0; r < 4; ++r) { u10 = mfma(in.tm[1][r], rr[0][r], r < 1 ? zero : u10); feed(); }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            u[1] = mfma(in.tm[2][r], rr[1][r], r < 1 ? zero : u[1]);
            if (r == 0) ue[0] = u[0] * in.ec[0];
            feed();
        }
#pragma unroll
        for (int i = 0; i < 8 * NK; ++i) {
            // rows of the chunk's first half before the second's, so that U's second half has time
            const int n = (i >> 2) % NK, a = (i >> 2) / NK, r = i & 3;
            if (i == 1) u[1] += u10;
            if (i == 2) ue[1] = u[1] * in.ec[1];
            grow[n] = mfma(in.kt[a][n][r], ue[a][r], a == 0 && r == 0 ? zero : grow[n]);
            if (a == 1 && n > 0 && r == 1) st[n - 1] = st[n - 1] * in.gl + grow[n - 1];        // (summed by itself: one rounding of S per chunk)
            if (i == 3) { const float m = mine(u[0]); y[0] = mfma(in.pm[0], m, zero); y[1] = mfma(in.pm[1], m, zero); }
            if (i == 4) y[1] = mfma(in.pm[2], mine(u[1]), y[1]);
            if (i == 5) y[0] += o[0] * in.eg[0];
            if (i == 6) y[1] += o[1] * in.eg[1];
            if (i == 6 && c > 0) finish(c - 1, fo, false);
            feed();
        }
        st[NK - 1] = st[NK - 1] * in.gl + grow[NK - 1];
    };
    ScanIn<NK> in0, in1;
#pragma unroll
    for (int i = 0; i < L_ALL; ++i) {
        load(in0, i);
        __builtin_amdgcn_sched_barrier(0);                     // (in this order: the waits count on it)
    }
    // the first chunk in front of the loop, and no exit in the loop's middle: the loads then stand in the same order on every way to a
    // wait, and none waits for all of them
    chunk(0, in0, in1);
    int c = 1;
    for (; c + 1 < nc; c += 2) {
        chunk(c, in1, in0);
        chunk(c + 1, in0, in1);
    }
    if (c < nc) chunk(c, in1, in0);
    {
        f32x4 (*rd)[4][64] = red[nc & 1];
        f32x2 fo[4];
#pragma unroll
        for (int a = 0; a < 2; ++a) rd[wid][2 + a][lane] = y[a];
        meet();
        gather(fo, rd);
        finish(nc - 1, fo, true);
    }
#pragma unroll
    for (int n = 0; n < NK; ++n) {
        const int t = wid + 4 * n;
        if (t < tiles)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[(long)(16 * t + 4 * g + r) * p.dvp] = st[n][r];
    }
}

// read-outs -> the output product's operand: RMS norm over the head, weight, silu of the gate; half a wave (HALF) or a wave per head. The squares
// are written as fused operations, one after the other: left to the compiler, an unrolled sum rounds its second square by itself and
// fuses the first one into it, and the two forms' bits differ
template <typename T, bool HALF>
__global__ __launch_bounds__(256) void delta_out_kernel(CogsDelta p) {
    const int row = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const long nv = (long)p.heads * p.dvp;
    const float* gate = p.t + (long)row * p.ldt + 2L * p.kv_heads * p.dkp + nv;
    // heads of up to 128 columns: half a wave has one in its registers, all of its loads out together, two heads of each half at a time (a wave a
    // head left half the lanes idle and read the row twice: 4096 rows of 16 heads of 128 27.5 us, 17.0; 84 MB)
    if constexpr (HALF) {
        constexpr int U = 2;
        const int d = min((lane & 31) * 4, p.dvp - 4);
        const bool in = (lane & 31) * 4 < p.dvp;
        const f32x4 w = *reinterpret_cast<const f32x4*>(p.norm + d);
        for (int h0 = 2 * wid + (lane >> 5); h0 - (lane >> 5) < p.heads; h0 += 8 * U) {
            f32x4 v[U], z[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int h = min(h0 + 8 * u, p.heads - 1);
                v[u] = *reinterpret_cast<const f32x4*>(p.o + ((long)h * p.rows + row) * p.dvp + d);
                z[u] = *reinterpret_cast<const f32x4*>(gate + (long)h * p.dvp + d);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int h = h0 + 8 * u;
                float ss = 0.f;
                if (in)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss = fmaf(v[u][e], v[u][e], ss);
                const float f = 1.f / sqrtf(half_wave_sum(ss) / (float)p.vdim + p.eps);
                f32x4 r;
#pragma unroll
                for (int e = 0; e < 4; ++e) r[e] = v[u][e] * f * w[e] * (z[u][e] / (1.f + expf(-z[u][e])));
                if (in && h < p.heads) st4_f<T>(reinterpret_cast<T*>(p.att) + (long)row * p.ldo + (long)h * p.dvp + d, r);
            }
        }
        return;
    }
    for (int h = wid; h < p.heads; h += 4) {
        const float* o = p.o + ((long)h * p.rows + row) * p.dvp;
        float ss = 0.f;
        for (int d = lane * 4; d < p.dvp; d += 256) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(o + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(v[e], v[e], ss);
        }
        const float f = 1.f / sqrtf(wave_sum(ss) / (float)p.vdim + p.eps);
        T* y = reinterpret_cast<T*>(p.att) + (long)row * p.ldo + (long)h * p.dvp;
        for (int d = lane * 4; d < p.dvp; d += 256) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(o + d), z = *reinterpret_cast<const f32x4*>(gate + (long)h * p.dvp + d),
                        w = *reinterpret_cast<const f32x4*>(p.norm + d);
            f32x4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = v[e] * f * w[e] * (z[e] / (1.f + expf(-z[e])));
            st4_f<T>(y + d, r);
        }
    }
}

// One new token per sequence: a workgroup per (head, sequence), a wave per 16 columns of S: lane = (row group of 16, four columns), PER rows
// a lane, so that both products with S close inside the wave and only the read-out's norm needs the others. S passes through registers
// once; it is asked for behind the convolution's inputs (loads return in order) and arrives while they are worked on.
// What is there besides the state is latency: a thread per column group with the row groups' sums in LDS had five barriers and sums of 16
// in a row (8 sequences, 16 heads of 128: 10.6 us; this one 9.9, of which 33.6 MB of state in and out take 6.8).
template <typename T, int PER, int TAPS>
__global__ __launch_bounds__(1024) void delta_step_kernel(CogsDelta p) {
    __shared__ __attribute__((aligned(16))) float z[3 * 256];           // q | k | v of this head behind the convolution
    __shared__ float red[16];
    const int h = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, threads = blockDim.x;
    const int rep = p.heads / p.kv_heads, kh = h / rep, v0 = 2 * p.kv_heads * p.dkp, rg = lane >> 2, col = 16 * wid + 4 * (lane & 3);
    const float* x = p.t + (long)row * p.ldt;
    const float* gate = x + v0 + (long)p.heads * p.dvp + (long)h * p.dvp;
    const float* tb = x + v0 + 2 * p.heads * p.dvp;
    const CogsSeq s = p.seqs[row];
    const int pos = s.pos0, at = pos % p.taps, n = 2 * p.dkp + p.dvp;
    float* S = s.state + p.state_off + (long)h * p.dkp * p.dvp;
    float* ring = s.state + p.state_off + (long)p.heads * p.dkp * p.dvp;
    // channel of z[i]; its inputs, latest first, and their taps (zeros past the sequence's start)
    auto channel = [&](int i) { return i < p.dkp ? kh * p.dkp + i : i < 2 * p.dkp ? (p.kv_heads + kh) * p.dkp + i - p.dkp : v0 + h * p.dvp + i - 2 * p.dkp; };
    float in[TAPS], tap[TAPS];
    auto request = [&](int i) {
        const int c = channel(i);
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            const bool there = j < p.taps && j <= pos;
            tap[j] = there ? p.conv[(long)(p.taps - 1 - j) * p.channels + c] : 0.f;
            in[j] = j == 0 ? x[c] : there ? ring[(long)(at - j + (j > at ? p.taps : 0)) * p.channels + c] : 0.f;
        }
    };
    auto finish = [&](int i) {
        float y = tap[0] * in[0];
#pragma unroll
        for (int j = 1; j < TAPS; ++j) y = fmaf(tap[j], in[j], y);
        z[(i < p.dkp ? 0 : i < 2 * p.dkp ? 256 - p.dkp : 512 - 2 * p.dkp) + i] = y / (1.f + expf(-y));
        // the new input takes the oldest one's place, which no position reads any more
        if (i >= 2 * p.dkp || h % rep == 0) ring[(long)at * p.channels + channel(i)] = in[0];
    };
    if (tid < n) request(tid);
    const f32x4 zg = *reinterpret_cast<const f32x4*>(gate + col), wn = *reinterpret_cast<const f32x4*>(p.norm + col);
    const float beta = sigmoid_f(tb[h]), g = expf(p.neg_a[h] * softplus_f(tb[p.headsp + h] + p.dt_bias[h]));
    f32x4 sr[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i)
        sr[i] = pos > 0 && 16 * i < p.dkp ? *reinterpret_cast<const f32x4*>(S + (long)(16 * i + rg) * p.dvp + col) : f32x4{0.f, 0.f, 0.f, 0.f};
    if (tid < n) finish(tid);
    for (int i = tid + threads; i < n; i += threads) { request(i); finish(i); }
    __syncthreads();
    float sq = 0.f, sk = 0.f;
    for (int d = lane; d < p.dkp; d += 64) { sq += z[d] * z[d]; sk += z[256 + d] * z[256 + d]; }
    const float fq = unit_scale(wave_sum(sq)) * p.q_scale, fk = unit_scale(wave_sum(sk));
    // the sum over the 16 row groups, in every lane
    auto close = [](f32x4 a) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = a[e];
            v += lane_xor_dpp<4>(v);
            v += lane_xor_dpp<8>(v);
            const unsigned b = __builtin_bit_cast(unsigned, v);
            const auto m = __builtin_amdgcn_permlane16_swap(b, b, false, false);
            v = __builtin_bit_cast(float, (unsigned)m[0]) + __builtin_bit_cast(float, (unsigned)m[1]);
            const unsigned c = __builtin_bit_cast(unsigned, v);
            const auto o = __builtin_amdgcn_permlane32_swap(c, c, false, false);
            a[e] = __builtin_bit_cast(float, (unsigned)o[0]) + __builtin_bit_cast(float, (unsigned)o[1]);
        }
        return a;
    };
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (16 * i >= p.dkp) continue;
        sr[i] *= g;
        a += sr[i] * (z[256 + 16 * i + rg] * fk);
    }
    a = close(a);
    const f32x4 u = beta * (*reinterpret_cast<const f32x4*>(z + 512 + col) - a);
    a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (16 * i >= p.dkp) continue;
        sr[i] += u * (z[256 + 16 * i + rg] * fk);
        *reinterpret_cast<f32x4*>(S + (long)(16 * i + rg) * p.dvp + col) = sr[i];
        a += sr[i] * (z[16 * i + rg] * fq);
    }
    a = close(a);
    // read-out's norm and gate
    float ss = (a[0] * a[0] + a[1] * a[1]) + (a[2] * a[2] + a[3] * a[3]);
    ss += lane_xor_dpp<1>(ss);
    ss += lane_xor_dpp<2>(ss);
    if (lane == 0) red[wid] = ss;
    __syncthreads();
    ss = 0.f;
    for (int w = 0; w < threads >> 6; ++w) ss += red[w];
    const float f = 1.f / sqrtf(ss / (float)p.vdim + p.eps);
    if (lane < 4) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = a[e] * f * wn[e] * (zg[e] / (1.f + expf(-zg[e])));
        st4_f<T>(reinterpret_cast<T*>(p.att) + (long)row * p.ldo + (long)h * p.dvp + col, y);
    }
}

// The same for heads of more than 256 rows or columns. S passes through registers once (NPER chunks of four columns per
// thread; 0: read twice from memory): thread = (row group, four columns), the row groups' partial sums meet in LDS.
constexpr int STEP_T = 512;
template <typename T, int NPER>
__global__ __launch_bounds__(STEP_T) void delta_step_wide_kernel(CogsDelta p) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int row = blockIdx.y;
    const CogsSeq s = p.seqs[row];
    const int pos = s.pos0, rep = p.heads / p.kv_heads, kh = h / rep;
    const float* x = p.t + (long)row * p.ldt;
    float* S = s.state + p.state_off + (long)h * p.dkp * p.dvp;
    float* ring = s.state + p.state_off + (long)p.heads * p.dkp * p.dvp;
    const int nc = p.dvp >> 2, groups = STEP_T / nc, rg = tid / nc, c4 = tid - rg * nc;
    float *q = sm, *k = q + p.dkp, *v = k + p.dkp, *red8 = v + p.dvp, *u = red8 + 16;
    f32x4* part = reinterpret_cast<f32x4*>(u + p.dvp);             // [groups][nc]
    const bool active = rg < groups;

    f32x4 sr[NPER > 0 ? NPER : 1];
    auto load = [&](int i) {
        const int d = rg + groups * i;
        return active && d < p.dkp && pos > 0 ? *reinterpret_cast<const f32x4*>(S + (long)d * p.dvp + 4 * c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    if constexpr (NPER > 0) {
#pragma unroll
        for (int i = 0; i < NPER; ++i) sr[i] = load(i);
    }
    // convolution + silu of this head's q, k and v channels; the new inputs into the ring (rows other positions read stay as they are)
    const int v0 = 2 * p.kv_heads * p.dkp;
    for (int i = tid; i < 2 * p.dkp + p.dvp; i += STEP_T) {
        const int c = i < p.dkp ? kh * p.dkp + i : i < 2 * p.dkp ? (p.kv_heads + kh) * p.dkp + i - p.dkp : v0 + h * p.dvp + i - 2 * p.dkp;
        sm[i] = conv_silu(p, x, ring, c, pos, 0);
        if (i >= 2 * p.dkp || h % rep == 0) ring[(long)(pos % p.taps) * p.channels + c] = x[c];
    }
    __syncthreads();
    if (wid < 2) {
        float* z = wid ? k : q;
        float ss = 0.f;
        for (int d = lane; d < p.dkp; d += 64) ss += z[d] * z[d];
        const float f = unit_scale(wave_sum(ss)) * (wid ? 1.f : p.q_scale);
        for (int d = lane; d < p.dkp; d += 64) z[d] *= f;
    }
    const float *tb = x + v0 + 2 * p.heads * p.dvp;
    const float beta = sigmoid_f(tb[h]), g = expf(p.neg_a[h] * softplus_f(tb[p.headsp + h] + p.dt_bias[h]));
    __syncthreads();
    const int iters = NPER > 0 ? NPER : (p.dkp + groups - 1) / groups;
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < iters; ++i) {
        const int d = rg + groups * i;
        if (active && d < p.dkp) {
            f32x4 w;
            if constexpr (NPER > 0) { sr[i] *= g; w = sr[i]; } else w = load(i) * g;
            a += w * k[d];
        }
    }
    if (active) part[rg * nc + c4] = a;
    __syncthreads();
    for (int j = tid; j < p.dvp; j += STEP_T) {
        const float* pf = reinterpret_cast<const float*>(part);
        float t = 0.f;
        for (int r = 0; r < groups; ++r) t += pf[r * p.dvp + j];
        u[j] = beta * (v[j] - t);
    }
    __syncthreads();
    const f32x4 uv = active ? *reinterpret_cast<const f32x4*>(u + 4 * c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < iters; ++i) {
        const int d = rg + groups * i;
        if (active && d < p.dkp) {
            f32x4 w;
            if constexpr (NPER > 0) w = sr[i]; else w = load(i) * g;
            w += uv * k[d];
            *reinterpret_cast<f32x4*>(S + (long)d * p.dvp + 4 * c4) = w;
            a += w * q[d];
        }
    }
    if (active) part[rg * nc + c4] = a;
    __syncthreads();
    // read-out, its norm and gate (v's place takes the read-out)
    float ss = 0.f;
    for (int j = tid; j < p.dvp; j += STEP_T) {
        const float* pf = reinterpret_cast<const float*>(part);
        float t = 0.f;
        for (int r = 0; r < groups; ++r) t += pf[r * p.dvp + j];
        v[j] = t;
        ss += t * t;
    }
    ss = wave_sum(ss);
    if (lane == 0) red8[wid] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < STEP_T / 64; ++w) ss += red8[w];
    const float f = 1.f / sqrtf(ss / (float)p.vdim + p.eps);
    T* y = reinterpret_cast<T*>(p.att) + (long)row * p.ldo + (long)h * p.dvp;
    const float* gate = x + v0 + (long)p.heads * p.dvp + (long)h * p.dvp;
    for (int j = tid; j < p.dvp; j += STEP_T) st_f<T>(y + j, v[j] * f * p.norm[j] * (gate[j] / (1.f + expf(-gate[j]))));
}

template <typename T>
int launch_step(hipStream_t st, const CogsDelta& p, int nseq) {
    const dim3 grid(p.heads, nseq);
    if (p.dkp <= 256 && p.dvp <= 256 && p.taps <= 8) {
#define COGS_STEP(N, TAPS) hipLaunchKernelGGL((delta_step_kernel<T, N, TAPS>), grid, dim3(4 * p.dvp), 0, st, p)
        if (p.dkp <= 128) { if (p.taps <= 4) COGS_STEP(8, 4); else COGS_STEP(8, 8); }
        else if (p.taps <= 4) COGS_STEP(16, 4);
        else COGS_STEP(16, 8);
#undef COGS_STEP
        return COGS_LAUNCH_CHECK();
    }
    const int nc = p.dvp / 4, groups = STEP_T / nc, nper = (p.dkp + groups - 1) / groups;
    const size_t lds = (size_t)(2 * p.dkp + 2 * p.dvp + 16) * 4 + (size_t)groups * nc * 16;
#define COGS_STEP(N) hipLaunchKernelGGL((delta_step_wide_kernel<T, N>), grid, dim3(STEP_T), lds, st, p)
    if (nper <= 8) COGS_STEP(8);
    else if (nper <= 32) COGS_STEP(32);
    else COGS_STEP(0);
#undef COGS_STEP
    return COGS_LAUNCH_CHECK();
}

void launch_inputs(hipStream_t st, const CogsDelta& a, int rows, int nseq, int max_new) {
    const int nv = a.heads * a.dvp;
    const auto grid = [&](int e, int run) { return dim3((max_new + CH - 1) / CH * (CH / run), (2 * a.kv_heads + (nv + 64 * e - 1) / (64 * e) + 1 + 3) / 4, nseq); };
    if (a.taps <= 4 && a.dkp <= 64) hipLaunchKernelGGL((delta_inputs_kernel<1, 4, 16>), grid(1, 16), dim3(256), 0, st, a);
    else if (a.taps <= 4 && a.dkp <= 128) hipLaunchKernelGGL((delta_inputs_kernel<2, 4, 16>), grid(2, 16), dim3(256), 0, st, a);
    else if (a.taps <= 8 && a.dkp <= 256) hipLaunchKernelGGL((delta_inputs_kernel<4, 8, 8>), grid(4, 8), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(delta_inputs_any_kernel<true>, dim3(rows), dim3(256), 0, st, a);
}

template <int NK>
void launch_scan(hipStream_t st, const CogsDelta& a, dim3 grid, int scan) {
    if (a.pad) hipLaunchKernelGGL((delta_scan_kernel<NK, false>), grid, dim3(256), 0, st, a, scan);
    else hipLaunchKernelGGL((delta_scan_kernel<NK, true>), grid, dim3(256), 0, st, a, scan);
}

bool sizes_ok(const CogsDelta& a) {
    return a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.taps > 0 && a.dkp % 16 == 0 && a.dvp % 16 == 0 && a.dkp <= 512 &&
           a.dvp <= 2048 && a.vdim > 0 && a.vdim <= a.dvp && a.channels == 2 * a.kv_heads * a.dkp + a.heads * a.dvp && a.ldt % 4 == 0 && a.ldo % 4 == 0;
}

}  // namespace

int cogs_k_delta_slots(int rows, int nseq) { return rows / CH + nseq; }
size_t cogs_k_delta_rec_floats(int rows, int nseq, int heads) { return (size_t)cogs_k_delta_slots(rows, nseq) * heads * REC; }

// Short sequences: zeros for whole chunks would be up to 32 times their bytes. Without them the scan masks its loads, 0.3 to 0.8 % of a long prompt's
// time: 4 to 8 ns a chunk, and the zeros 0.08 us a sequence. Widths 2048, 4096, us, zeros / masks: 128 prompts of 2 tokens 2021 / 1992, 4323 / 4112; 300
// rows that join 16 requests 1315 / 1276, 2578 / 2550, 32 requests 1511 / 1477, 3010 / 2955; one prompt of 4096 4948 / 4987, 12 147 / 12 190
static bool zeros_to_the_end(int nseq, int max_new) {
    if (g_cogs_debug.delta_zeros > 0) return g_cogs_debug.delta_zeros == 1;
    return nseq == 1 || nseq * 512L <= max_new;
}

int cogs_k_delta_prompt(hipStream_t st, int dtype, const CogsDelta& delta, int rows, int nseq, int max_new) {
    CogsDelta a = delta;
    a.pad = zeros_to_the_end(nseq, max_new);
    if (!sizes_ok(a) || rows <= 0 || nseq <= 0 || nseq > 65535 || a.heads > 65535) return COGS_E_INVALID;
    if (a.slots != cogs_k_delta_slots(rows, nseq)) return COGS_E_INVALID;
    const int keep = (max_new < a.taps ? max_new : a.taps) * a.channels, tail = (keep + 1023) / 1024;
    if (a.dkp <= 256 && g_cogs_debug.delta_chunk != 0) {
        launch_inputs(st, a, rows, nseq, max_new);
        hipLaunchKernelGGL(delta_chunk_kernel, dim3((max_new + CH - 1) / CH, a.heads, nseq), dim3(256), 0, st, a);
        const int scan = (a.heads + 7) / 8 * 8 * (a.dvp / 16);
        const dim3 grid(scan + (tail + 7) / 8 * 8, 1, nseq);      // (a multiple of 8: the heads of every sequence keep their XCDs)
        if (a.dkp <= 64) launch_scan<1>(st, a, grid, scan);
        else if (a.dkp <= 128) launch_scan<2>(st, a, grid, scan);
        else launch_scan<4>(st, a, grid, scan);
    } else {
        hipLaunchKernelGGL(delta_inputs_any_kernel<false>, dim3(rows), dim3(256), 0, st, a);
        hipLaunchKernelGGL(delta_tail_kernel, dim3(tail, nseq), dim3(256), 0, st, a);
        hipLaunchKernelGGL(delta_recur_kernel, dim3((a.dvp + 63) / 64, a.heads, nseq), dim3(64), 0, st, a);
    }
    const bool half = a.dvp <= 128 && g_cogs_debug.delta_out_wave == 0;
    if (dtype == COGS_DT_BF16) {
        if (half) hipLaunchKernelGGL((delta_out_kernel<bf16_t, true>), dim3(rows), dim3(256), 0, st, a);
        else hipLaunchKernelGGL((delta_out_kernel<bf16_t, false>), dim3(rows), dim3(256), 0, st, a);
    } else {
        if (half) hipLaunchKernelGGL((delta_out_kernel<float, true>), dim3(rows), dim3(256), 0, st, a);
        else hipLaunchKernelGGL((delta_out_kernel<float, false>), dim3(rows), dim3(256), 0, st, a);
    }
    return COGS_LAUNCH_CHECK();
}

int cogs_k_delta_step(hipStream_t st, int dtype, const CogsDelta& a, int nseq) {
    if (!sizes_ok(a) || nseq <= 0 || nseq > 65535) return COGS_E_INVALID;
    return dtype == COGS_DT_BF16 ? launch_step<bf16_t>(st, a, nseq) : launch_step<float>(st, a, nseq);
}
