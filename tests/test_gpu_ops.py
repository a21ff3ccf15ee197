"""Operator-level parity: every HIP kernel, called through the C ABI, against a plain torch fp32
restatement of the same op on the same seeded inputs. Tolerances are stated per test:
bf16 storage => ~2^-8 relative per rounding; fp32 parity mode => 1e-4 or tighter."""
import math

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _ops():
    from cogstream_amd import ops
    return ops


def _L():
    from cogstream_amd import _lib
    return _lib


@pytest.fixture(params=[1, 0], ids=["dispatched", "unsplit"])
def gemm_split(request):
    """products as the dispatch takes them, and (0) wholly by the ping-pong kernel from 256 rows on where N pads to 256 by at most 12 %"""
    with _L().debug_switch("gemm_split", request.param):
        yield request.param


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1.2e-2), (torch.float32, 2e-5)])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (300, 256, 192), (1, 512, 256), (77, 132, 128), (1024, 1152, 1152),
                                   (515, 132, 64), (777, 384, 704)])
def test_gemm_bias_residual(dev, dtype, tol, M, N, K):
    ops = _ops()
    torch.manual_seed(M * 7 + N)
    a = torch.randn(M, K).to(dtype)
    w = (torch.randn(N, K) / math.sqrt(K)).to(dtype)
    b = torch.randn(N).to(dtype)
    r = torch.randn(M, N).to(dtype)
    ref = a.float() @ w.float().t() + b.float() + r.float()
    out = ops.gemm(a.to(dev), w.to(dev), b.to(dev), residual=r.to(dev))
    assert out.dtype == dtype
    assert rel_err(out.float(), ref) < tol


def test_gemm_integer_exact(dev):
    """MFMA fragment/layout check with exactly representable data and an asymmetric W"""
    run_gemm_integer_exact(dev, 256, 256, 128)
    run_gemm_integer_exact(dev, 1024 + 40, 384, 448)   # fp32: 256x128 ring-buffered variant, ragged M


def run_gemm_integer_exact(dev, M, N, K):
    ops = _ops()
    a = torch.randint(-3, 4, (M, K)).float()
    w = (torch.arange(N)[:, None] % 5 - 2).float() * torch.randint(0, 2, (N, K)).float() + (torch.arange(K)[None, :] % 3).float()
    ref = a @ w.t()
    out = ops.gemm(a.to(dev).bfloat16(), w.to(dev).bfloat16(), out_f32=True)
    assert torch.equal(out.cpu(), ref)
    out32 = ops.gemm(a.to(dev), w.to(dev))
    assert torch.equal(out32.cpu(), ref)


@pytest.mark.parametrize("act", ["tanh", "erf"])
def test_gemm_gelu(dev, act):
    ops, L = _ops(), _L()
    torch.manual_seed(1)
    a = torch.randn(200, 128).bfloat16()
    w = (torch.randn(256, 128) / 11).bfloat16()
    b = torch.randn(256).bfloat16()
    pre = a.float() @ w.float().t() + b.float()
    ref = F.gelu(pre, approximate="tanh") if act == "tanh" else F.gelu(pre)
    out = ops.gemm(a.to(dev), w.to(dev), b.to(dev), act=L.ACT_GELU_TANH if act == "tanh" else L.ACT_GELU_ERF)
    assert rel_err(out.float(), ref) < 1.2e-2


@pytest.mark.parametrize("M", [1, 130])
def test_gemm_swiglu(dev, M):
    ops, L = _ops(), _L()
    torch.manual_seed(2)
    H, I = 128, 192
    x = torch.randn(M, H).bfloat16()
    wg = (torch.randn(I, H) / 11).bfloat16()
    wu = (torch.randn(I, H) / 11).bfloat16()
    ref = F.silu(x.float() @ wg.float().t()) * (x.float() @ wu.float().t())
    gu = torch.stack([wg, wu], dim=1).reshape(2 * I, H).contiguous()
    out = ops.gemm(x.to(dev), gu.to(dev), act=L.ACT_SWIGLU)
    assert out.shape == (M, I)
    assert rel_err(out.float(), ref) < 1.2e-2


@pytest.mark.parametrize("M,heads,interleaved", [(1, 2, False), (96, 2, False), (96, 2, True), (1300, 2, True),
                                                 (1300, 7, True), (1300, 7, False)])
def test_gemm_rope_epilogue(dev, gemm_split, M, heads, interleaved):
    """columns [0, rope_cols) rotated as rotate_half pairs after the (d, d+hd/2) row interleave; both table
    formats; M = 1300 reaches the mid-size (heads 2, and 7 as dispatched) and ping-pong (heads 7) kernels, whose interior wave tiles
    take the lean epilogue while the tile straddling rope_cols and the ragged last row block take the general one"""
    ops = _ops()
    torch.manual_seed(3)
    hd, K = 72, 128
    N = 3 * heads * hd  # q | k | v, v not rotated
    x = torch.randn(M, K).bfloat16()
    w = (torch.randn(N, K) / 11).bfloat16()
    b = torch.randn(N).bfloat16()
    ang = torch.rand(M, hd // 2) * 6.0
    y = (x.float() @ w.float().t() + b.float()).view(M, 3 * heads, hd)
    cos = torch.cat([ang.cos(), ang.cos()], -1)[:, None, :]
    sin = torch.cat([ang.sin(), ang.sin()], -1)[:, None, :]
    rot = torch.cat([-y[..., hd // 2:], y[..., :hd // 2]], -1)
    ref = y.clone()
    ref[:, :2 * heads] = (y * cos + rot * sin)[:, :2 * heads]
    # pack: within each q/k head, new row 2i <- d=i, 2i+1 <- d=i+hd/2
    perm = torch.arange(hd).view(2, hd // 2).t().reshape(-1)
    wp = w.view(3 * heads, hd, K).clone()
    bp = b.view(3 * heads, hd).clone()
    wp[:2 * heads] = wp[:2 * heads][:, perm]
    bp[:2 * heads] = bp[:2 * heads][:, perm]
    out = ops.gemm(x.to(dev), wp.reshape(N, K).contiguous().to(dev), bp.reshape(N).contiguous().to(dev),
                   rope_cos=(torch.stack([ang.cos(), ang.sin()], -1) if interleaved else ang.cos()).contiguous().to(dev),
                   rope_sin=None if interleaved else ang.sin().contiguous().to(dev),
                   rope_cols=2 * heads * hd, head_dim=hd)
    refp = ref.clone()
    refp[:, :2 * heads] = ref[:, :2 * heads][:, :, perm]
    assert rel_err(out.float().view(M, 3 * heads, hd), refp) < 1.2e-2


def test_gemm_rope_position_lut_equals_row_table(dev, gemm_split):
    """the ping-pong GEMM's LDS position LUT (2-D rotary: first half of a head's pairs uses the row's h, second half
    its w) must give bit-identical outputs to the per-row (cos, sin) table built from the same angles -- and both
    must match the plain reference"""
    ops = _ops()
    torch.manual_seed(17)
    hd, heads, K, M = 72, 7, 128, 1500            # N = 1512: unsplit, the ping-pong kernel; ragged last row block; rope straddle
    nf, maxpos = hd // 4, 45
    N = 3 * heads * hd
    x = torch.randn(M, K).bfloat16()
    w = (torch.randn(N, K) / 11).bfloat16()
    b = torch.randn(N).bfloat16()
    hpos, wpos = torch.randint(0, 23, (M,)), torch.randint(0, maxpos, (M,))
    inv_freq = 1.0 / (10000.0 ** (torch.arange(nf, dtype=torch.float32) / nf))
    lut_ang = torch.arange(maxpos, dtype=torch.float32)[:, None] * inv_freq[None, :]            # [maxpos, nf]
    lut = torch.stack([lut_ang.cos(), lut_ang.sin()], -1).contiguous()                          # [maxpos, nf, 2]
    ang = torch.cat([hpos[:, None].float() * inv_freq[None, :], wpos[:, None].float() * inv_freq[None, :]], 1)   # [M, hd/2]
    table = torch.cat([lut[hpos], lut[wpos]], 1).contiguous()                                   # [M, hd/2, 2] same values
    assert torch.equal(table[..., 0], torch.cat([lut_ang[hpos], lut_ang[wpos]], 1).cos())
    rowpos = (hpos | (wpos << 16)).to(torch.int32)
    perm = torch.arange(hd).view(2, hd // 2).t().reshape(-1)
    wp = w.view(3 * heads, hd, K).clone()
    bp = b.view(3 * heads, hd).clone()
    wp[:2 * heads] = wp[:2 * heads][:, perm]
    bp[:2 * heads] = bp[:2 * heads][:, perm]
    args = dict(rope_cos=table.to(dev), rope_sin=None, rope_cols=2 * heads * hd, head_dim=hd)
    xa, wa, ba = x.to(dev), wp.reshape(N, K).contiguous().to(dev), bp.reshape(N).contiguous().to(dev)
    out_tab = ops.gemm(xa, wa, ba, **args)
    out_lut = ops.gemm(xa, wa, ba, rope_lut=lut.to(dev), rope_rowpos=rowpos.to(dev), **args)
    assert torch.equal(out_lut, out_tab)
    y = (x.float() @ w.float().t() + b.float()).view(M, 3 * heads, hd)
    cos = torch.cat([ang.cos(), ang.cos()], -1)[:, None, :]
    sin = torch.cat([ang.sin(), ang.sin()], -1)[:, None, :]
    rot = torch.cat([-y[..., hd // 2:], y[..., :hd // 2]], -1)
    ref = y.clone()
    ref[:, :2 * heads] = (y * cos + rot * sin)[:, :2 * heads]
    ref[:, :2 * heads] = ref[:, :2 * heads][:, :, perm]
    assert rel_err(out_lut.float().view(M, 3 * heads, hd), ref) < 1.2e-2


def _attn_ref(q, k, v, hq, hkv, hd, cu=None, causal=False, q_pos0=0, row_lo=None, row_hi=None, bias=0.0, scale=None):
    Lq, Lk = q.shape[0], k.shape[0]
    q = q.float().view(Lq, hq, hd).transpose(0, 1)
    k = k.float().view(Lk, hkv, hd).transpose(0, 1).repeat_interleave(hq // hkv, 0)
    v = v.float().view(Lk, hkv, hd).transpose(0, 1).repeat_interleave(hq // hkv, 0)
    s = q @ k.transpose(1, 2) * (1.0 / math.sqrt(hd) if scale is None else scale)
    qi, kj = torch.arange(Lq)[:, None], torch.arange(Lk)[None, :]
    allow = torch.ones(Lq, Lk, dtype=torch.bool)
    if cu is not None:
        seg_q = torch.bucketize(qi, cu[1:], right=True)
        seg_k = torch.bucketize(kj, cu[1:], right=True)
        allow &= seg_q == seg_k
    if causal:
        allow &= kj <= qi + q_pos0
    if row_lo is not None:
        s = s + ((kj >= row_lo[:, None]) & (kj < row_hi[:, None])).float() * bias
    s = s.masked_fill(~allow, float("-inf"))
    return (F.softmax(s, -1) @ v).transpose(0, 1).reshape(Lq, hq * hd)


@pytest.mark.parametrize("hd,heads,lens", [(72, 2, [256, 256]), (72, 3, [200, 200, 200]), (72, 2, [924]), (72, 1, [37, 130])])
def test_attention_block_diag_bf16(dev, hd, heads, lens):
    ops = _ops()
    torch.manual_seed(sum(lens))
    n = sum(lens)
    qkv = torch.randn(n, 3 * heads * hd).bfloat16()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    H = heads * hd
    ref = _attn_ref(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], heads, heads, hd, cu=cu.long())
    g = qkv.to(dev)
    out = ops.attention(g[:, :H], g[:, H:2 * H], g[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd,
                        cu_seqlens=cu.to(dev), max_seqlen=max(lens))
    assert rel_err(out.float(), ref) < 1.5e-2


LOG2E = 1.4426950408889634


@pytest.mark.parametrize("hd,heads,lens", [(72, 2, [256, 256]), (72, 2, [924]), (72, 1, [37, 130]), (128, 2, [300, 64])])
def test_attention_prescaled_q_block_diag(dev, hd, heads, lens):
    """q_prescaled: Q carries scale*log2(e) (rounded to bf16 once, as the QKV GEMM epilogue does) and the kernel
    runs the deferred-max softmax; the reference is the plain softmax of the same rounded Q with scale ln 2"""
    ops = _ops()
    torch.manual_seed(sum(lens) + hd)
    n = sum(lens)
    H = heads * hd
    qkv = torch.randn(n, 3 * H)
    qkv[:, :H] *= LOG2E / math.sqrt(hd)
    # rows whose scores move by tens of log2 units from tile to tile exercise the rebase path
    qkv[5, :H] *= 6.0
    qkv = qkv.bfloat16()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    ref = _attn_ref(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], heads, heads, hd, cu=cu.long(), scale=math.log(2.0))
    g = qkv.to(dev)
    out = ops.attention(g[:, :H], g[:, H:2 * H], g[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd,
                        cu_seqlens=cu.to(dev), max_seqlen=max(lens), q_prescaled=True)
    assert rel_err(out.float(), ref) < 1.5e-2


@pytest.mark.parametrize("heads,lens", [
    (1, [1]), (1, [31]), (2, [32, 33]), (1, [63, 64, 65]), (2, [96, 127, 128, 129]), (1, [160, 191, 192, 193]),
    (8, [200] * 5), (2, [255, 256, 257]), (1, [320, 384, 449]), (8, [924, 924]), (3, [1024, 70, 1000]), (16, [130] * 4)])
@pytest.mark.parametrize("data", ["random", "ramp"])
def test_attention_vit_pipeline_edges(dev, heads, lens, data):
    """The encoder's production attention kernel (csrc/attn_vit.hip: hd 72, per-frame segments, pre-scaled Q,
    software-pipelined at 32-key blocks with a 4-slot LDS-DMA ring) over every seam of its control flow: segments
    shorter than a block / a tile / the three-tile prologue, ragged and exactly-full last blocks and tiles, ragged and
    empty query blocks (waves that only stage), both workgroup orders (frames x heads a multiple of 8 or not).
    "ramp": the scores of every row GROW along the keys by ~2 log2 units per key block, so the deferred maximum is
    moved (O rescaled, the block's scores recomputed) again and again in steady state, and one row sits far below
    zero. Checked row by row against the fp32 softmax of the same bf16 inputs."""
    ops = _ops()
    hd, H = 72, heads * 72
    n = sum(lens)
    g = torch.Generator().manual_seed(1000 * heads + n + (data == "ramp"))
    qkv = torch.randn(n, 3 * H, generator=g)
    qkv[:, :H] *= LOG2E / math.sqrt(hd)
    if data == "ramp":
        # q = a common direction u (scaled), k = u * (position in the segment / 16): score ~ 1.5 * pos / 16 log2 units
        u = torch.randn(hd, generator=g)
        u /= u.norm()
        pos = torch.cat([torch.arange(L, dtype=torch.float32) for L in lens])
        for hh in range(heads):
            qkv[:, hh * hd:(hh + 1) * hd] += 1.5 * u
            qkv[:, H + hh * hd:H + (hh + 1) * hd] += u * (pos[:, None] / 16.0)
        qkv[n // 2, :H] = -3.0 * u.repeat(heads)          # a row whose scores fall with the key index
    qkv = qkv.bfloat16()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    ref = _attn_ref(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], heads, heads, hd, cu=cu.long(), scale=math.log(2.0))
    gq = qkv.to(dev)
    out = ops.attention(gq[:, :H], gq[:, H:2 * H], gq[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd,
                        cu_seqlens=cu.to(dev), max_seqlen=max(lens), q_prescaled=True).float().cpu()
    assert torch.isfinite(out).all()
    # per row: error against the row's own largest output (a dropped or doubled block shows up at 1e-1 .. 1)
    err = (out - ref).abs().view(n, heads, hd).amax(2) / ref.abs().view(n, heads, hd).amax(2).clamp_min(1e-3)
    assert float(err.max()) < 3e-2, (float(err.max()), int(err.argmax()) // heads)
    # convexity: every output lies inside the range its segment's V spans
    v = qkv[:, 2 * H:].float()
    for i, L in enumerate(lens):
        a, b = int(cu[i]), int(cu[i + 1])
        assert (out[a:b] <= v[a:b].amax(0) + 2e-2).all() and (out[a:b] >= v[a:b].amin(0) - 2e-2).all()


@pytest.mark.parametrize("seg", [129, 132, 160, 161, 176, 192, 193, 200, 240, 256, 257, 264, 308, 320, 336, 360, 384, 396, 440, 448,
                                 500, 512, 576, 924, 1024])
@pytest.mark.parametrize("layout", ["token", "head"])
def test_attention_vit_compile_time_end_equals_run_time_end_bit_for_bit(dev, seg, layout):
    """One video = every segment the same length: the pipelined ViT kernel is launched as the instantiation whose ragged end
    (tiles behind the four-tile loop R = 4..7, 32-key blocks of the last tile 1 / 2) has that length's shape as template
    parameters (csrc/attn_vit.hip, round 6). Lengths for all eight (R, blocks) pairs, last blocks of 1, 8, 31, 32 keys, exactly
    full last tiles, the loop running 0 / 1 / 3 trips, both K/V layouts, growing scores on half the heads. The launch with the
    hint must equal the launch without it (run-time end) bit for bit, and both the fp32 softmax."""
    ops = _ops()
    from cogstream_amd import _lib as L
    heads, nseg, hd = 4, 5, 72
    H, n = heads * hd, nseg * seg
    g = torch.Generator().manual_seed(seg)
    qkv = torch.randn(n, 3 * H, generator=g)
    qkv[:, :H] *= LOG2E / math.sqrt(hd)
    u = torch.randn(hd, generator=g)
    u /= u.norm()
    pos = torch.arange(seg, dtype=torch.float32).repeat(nseg)
    for hh in range(0, heads, 2):
        qkv[:, hh * hd:(hh + 1) * hd] += 1.5 * u
        qkv[:, H + hh * hd:H + (hh + 1) * hd] += u * (pos[:, None] / 16.0)
    qkv = qkv.bfloat16()
    cu = torch.arange(nseg + 1, dtype=torch.int32) * seg
    ref = _attn_ref(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], heads, heads, hd, cu=cu.long(), scale=math.log(2.0))
    if layout == "head":
        hm = qkv.view(n, 3, heads, hd).permute(1, 2, 0, 3).contiguous().to(dev)        # [which][head][row][hd]
        run = lambda: ops.attention(hm[0], hm[1], hm[2], hq=heads, hkv=heads, head_dim=hd, cu_seqlens=cu.to(dev),
                                    max_seqlen=seg, q_prescaled=True, head_major=True)
    else:
        gq = qkv.to(dev)
        run = lambda: ops.attention(gq[:, :H], gq[:, H:2 * H], gq[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd,
                                    cu_seqlens=cu.to(dev), max_seqlen=seg, q_prescaled=True)
    plain = run()
    assert L.debug_get("attn_vit_last_end") == 0
    with L.debug_switch("attn_uniform_hint", seg):
        hinted = run()
        nt = (seg + 63) // 64
        want = 10 * (4 + ((nt - 4) & 3)) + (2 if seg - 64 * (nt - 1) > 32 else 1) if nt >= 4 else 0
        assert L.debug_get("attn_vit_last_end") == want
        with L.debug_switch("attn_vit_len", 0):
            hinted_rt = run()
            assert L.debug_get("attn_vit_last_end") == 0
    assert torch.equal(plain, hinted) and torch.equal(plain, hinted_rt)
    out = hinted.float().cpu()
    err = (out - ref).abs().view(n, heads, hd).amax(2) / ref.abs().view(n, heads, hd).amax(2).clamp_min(1e-3)
    assert float(err.max()) < 3e-2, (float(err.max()), int(err.argmax()) // heads)


@pytest.mark.parametrize("S,pos0", [(200, 0), (130, 77), (1, 300), (1, 5000)])
def test_attention_prescaled_q_causal_gqa(dev, S, pos0):
    ops = _ops()
    torch.manual_seed(S + 1)
    hd, hq, hkv = 128, 4, 2
    ctx = pos0 + S
    q = (torch.randn(S, hq * hd) * (LOG2E / math.sqrt(hd))).bfloat16()
    k = torch.randn(ctx, hkv * hd).bfloat16()
    v = torch.randn(ctx, hkv * hd).bfloat16()
    ref = _attn_ref(q, k, v, hq, hkv, hd, causal=True, q_pos0=pos0, scale=math.log(2.0))
    out = ops.attention(q.to(dev), k.to(dev), v.to(dev), hq=hq, hkv=hkv, head_dim=hd, causal=True, q_pos0=pos0,
                        q_prescaled=True)
    assert rel_err(out.float(), ref) < 1.5e-2
    if S == 1:
        out2 = ops.attention(q.to(dev), k.to(dev), v.to(dev), hq=hq, hkv=hkv, head_dim=hd, causal=True, q_pos0=pos0,
                             nsplit=3 if pos0 < 1000 else 20, q_prescaled=True)
        assert rel_err(out2.float(), ref) < 1.5e-2


@pytest.mark.parametrize("hq,hkv", [(28, 4), (16, 1), (4, 4), (6, 2)])
@pytest.mark.parametrize("ctx,nsplit", [(1, 2), (63, 2), (64, 3), (65, 2), (255, 4), (256, 4), (257, 5), (1000, 8), (1000, 33),
                                        (4100, 17)])
def test_decode_attention_kernel_edges(dev, hq, hkv, ctx, nsplit):
    """The generated tokens' attention (csrc/attn_decode.hip: one query row, every wave owns whole 64-key tiles, four
    waves merged in LDS, partials combined by attn_combine_kernel): contexts around every tile boundary, splits with a
    ragged last tile, with fewer tiles than waves and with no tile at all (nsplit > tiles), 1 / 2 / 7 / 16 query heads
    per key/value head. Checked per head against the fp32 softmax of the same bf16 inputs."""
    ops = _ops()
    hd = 128
    g = torch.Generator().manual_seed(ctx * 131 + nsplit * 7 + hq)
    q = (torch.randn(1, hq * hd, generator=g) * (LOG2E / math.sqrt(hd))).bfloat16()
    k = torch.randn(ctx, hkv * hd, generator=g).bfloat16()
    v = torch.randn(ctx, hkv * hd, generator=g).bfloat16()
    if ctx > 4:
        k[ctx // 2] *= 4.0                       # one dominant key in the middle: the running maximum moves inside a split
    ref = _attn_ref(q, k, v, hq, hkv, hd, causal=True, q_pos0=ctx - 1, scale=math.log(2.0))
    out = ops.attention(q.to(dev), k.to(dev), v.to(dev), hq=hq, hkv=hkv, head_dim=hd, causal=True, q_pos0=ctx - 1,
                        nsplit=nsplit, q_prescaled=True).float().cpu()
    assert torch.isfinite(out).all()
    err = (out - ref).abs().view(hq, hd).amax(1) / ref.abs().view(hq, hd).amax(1).clamp_min(1e-3)
    assert float(err.max()) < 2e-2, (float(err.max()), int(err.argmax()))


def test_attention_integer_exact(dev):
    """layout check: one-hot attention (huge scale) must copy integer V rows exactly"""
    ops = _ops()
    hd, n = 128, 192
    torch.manual_seed(0)
    tgt = torch.randperm(n)
    # unique two-hot keys: q = 256*k[tgt] scores 512 on its target and <= 256 elsewhere (others underflow to 0)
    k = torch.zeros(n, hd)
    k[torch.arange(n), torch.arange(n) % 120] = 1.0
    k[torch.arange(n), 120 + torch.arange(n) // 120] = 1.0
    q = k[tgt] * 256.0
    v = torch.randint(-8, 9, (n, hd)).float()
    out = ops.attention(q.bfloat16().to(dev), k.bfloat16().to(dev), v.bfloat16().to(dev), hq=1, hkv=1, head_dim=hd,
                        scale=1.0)
    assert torch.equal(out.float().cpu(), v[tgt])


@pytest.mark.parametrize("S,pos0", [(200, 0), (130, 77), (1, 300)])
def test_attention_causal_gqa_bf16(dev, S, pos0):
    ops = _ops()
    torch.manual_seed(S)
    hd, hq, hkv = 128, 4, 2
    ctx = pos0 + S
    q = torch.randn(S, hq * hd).bfloat16()
    k = torch.randn(ctx, hkv * hd).bfloat16()
    v = torch.randn(ctx, hkv * hd).bfloat16()
    ref = _attn_ref(q, k, v, hq, hkv, hd, causal=True, q_pos0=pos0)
    out = ops.attention(q.to(dev), k.to(dev), v.to(dev), hq=hq, hkv=hkv, head_dim=hd, causal=True, q_pos0=pos0)
    assert rel_err(out.float(), ref) < 1.5e-2
    if S == 1:
        out2 = ops.attention(q.to(dev), k.to(dev), v.to(dev), hq=hq, hkv=hkv, head_dim=hd, causal=True, q_pos0=pos0,
                             nsplit=3)
        assert rel_err(out2.float(), ref) < 1.5e-2


@pytest.mark.parametrize("dtype,tol,rowwise", [(torch.bfloat16, 1.5e-2, False), (torch.float32, 1e-5, True)])
def test_attention_eager_global_bias(dev, dtype, tol, rowwise):
    ops = _ops()
    torch.manual_seed(5)
    hd, heads, lens = 72, 2, [64, 64, 64]
    n = sum(lens)
    H = heads * hd
    qkv = torch.randn(n, 3 * H).to(dtype)
    lo = torch.tensor([64 * (i // 64) for i in range(n)], dtype=torch.int32)
    hi = lo + 64
    ref = _attn_ref(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], heads, heads, hd, row_lo=lo.long(), row_hi=hi.long(), bias=1.0)
    g = qkv.to(dev)
    out = ops.attention(g[:, :H], g[:, H:2 * H], g[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd, row_lo=lo.to(dev),
                        row_hi=hi.to(dev), bias=1.0, force_rowwise=rowwise)
    assert rel_err(out.float(), ref) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float32, 1e-5)])
@pytest.mark.parametrize("H", [144, 1152, 3584])
def test_norms(dev, dtype, tol, H):
    ops = _ops()
    torch.manual_seed(H)
    x = (torch.randn(37, H) * 2 + 0.3).to(dtype)
    g = (1 + 0.1 * torch.randn(H)).to(dtype)
    b = (0.1 * torch.randn(H)).to(dtype)
    ref = F.layer_norm(x.float(), (H,), g.float(), b.float(), 1e-6)
    assert rel_err(ops.layernorm(x.to(dev), g.to(dev), b.to(dev)).float(), ref) < tol
    xf = x.float()
    ref = g.float() * (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6))
    assert rel_err(ops.rmsnorm(x.to(dev), g.to(dev)).float(), ref) < tol
    xm = x[:36]
    ref = F.layer_norm(xm.float(), (H,), g.float(), b.float(), 1e-6).view(9, 4, H).mean(1)
    assert rel_err(ops.ln_merge(xm.contiguous().to(dev), g.to(dev), b.to(dev), 4).float(), ref) < tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_pixdiff_mask_matches_torch_semantics(dev, dtype):
    """bit-exact against the torch expression of cogreasoner_chat.py:407-414 run in the same dtype"""
    ops = _ops()
    torch.manual_seed(11)
    t, P, E = 6, 20, 2352
    base = torch.rand(1, P, E) * 2 - 1
    pix = base.repeat(t, 1, 1)
    pix[1] += 0.002 * torch.randn(P, E)           # tiny change: mostly below threshold
    pix[2, :5] += 0.5 * torch.randn(5, E)         # big change on 5 tokens
    pix[4] = pix[3]                               # identical frame -> min_tokens kicks in
    pix = pix.to(dtype)
    diff = torch.abs(pix[1:] - pix[:-1]).mean(dim=-1) * 255
    diff = torch.cat([torch.full_like(diff[0:1], 1.1), diff], dim=0)
    m = diff > 0.1
    pad = torch.nonzero(m.sum(dim=1) < 1)[:, 0]
    m[pad, :1] = 1
    minor = torch.zeros(t, dtype=torch.uint8)
    minor[5] = 1
    m[5, 0] = True
    m[5, 1:] = False
    out = ops.pixdiff_mask(pix.reshape(-1, 588).contiguous().to(dev), t, P, minor=minor.to(dev))
    assert torch.equal(out.cpu().bool(), m.flatten())
    assert 0 < int(m.sum()) < m.numel()


def test_frame_mean_gather_mean_cosine(dev):
    ops = _ops()
    torch.manual_seed(12)
    P, D, T = 7, 256, 5
    f = torch.randn(T * P, D).bfloat16()
    ref = f.view(T, P, D).clone()
    for i in (1, 3):
        ref[i, 0] = ref[i].mean(dim=0)
    g = f.to(dev).clone()
    ops.frame_mean_to_slot0(g, P, torch.tensor([1, 3], dtype=torch.int32, device=dev))
    assert rel_err(g.float().cpu(), ref.view(-1, D).float()) < 8e-3
    ta, tb = torch.randn(50, D).bfloat16(), torch.randn(9, D).bfloat16()
    idx = torch.tensor([3, -1, 49, -9, 0, -4], dtype=torch.int64)
    out = ops.gather_rows(ta.to(dev), tb.to(dev), idx.to(dev))
    ref = torch.stack([ta[i] if i >= 0 else tb[-i - 1] for i in idx.tolist()])
    assert torch.equal(out.cpu(), ref)
    x = torch.randn(333, D).bfloat16()
    assert rel_err(ops.mean_rows(x.to(dev)), x.float().mean(0)) < 1e-5
    a, b = torch.randn(D), torch.randn(6, D)
    assert rel_err(ops.cosine(a.to(dev), b.to(dev)), F.cosine_similarity(a[None], b, dim=1)) < 1e-5


def test_logits_ops(dev):
    ops = _ops()
    torch.manual_seed(13)
    n = 152064
    lg = torch.randn(n)
    lg[777] = lg.max() + 1
    assert int(ops.argmax(lg.to(dev))) == 777
    prev = torch.tensor([5, 777, 5, 42], dtype=torch.int64)
    ref = lg.clone()
    g = ref[prev]
    ref[prev] = torch.where(g < 0, g * 1.05, g / 1.05)
    ref = ref / 0.7
    x = lg.to(dev).clone()
    ops.logits_process(x, prev.to(dev), 1.05, None, 0.7)
    assert torch.allclose(x.cpu(), ref, rtol=1e-6, atol=0)
    allowed = torch.tensor([11, 15, 16, 58, 60, 151645], dtype=torch.int32)
    x = lg.to(dev).clone()
    ops.logits_process(x, None, 1.0, allowed.to(dev), 1.0)
    refm = torch.full_like(lg, float("-inf"))
    refm[allowed.long()] = lg[allowed.long()]
    assert torch.equal(x.cpu(), refm)
    val, idx = ops.topk(lg.to(dev), 20)
    rv, ri = torch.topk(lg, 20)
    assert torch.equal(val.cpu(), rv) and torch.equal(idx.cpu().long(), ri)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_kmeans_steps(dev, dtype):
    ops = _ops()
    torch.manual_seed(14)
    T, PD, K = 40, 2 * 1024 + 512 + 8, 5
    cent = torch.randn(K, PD) * 3
    lab = torch.randint(0, K, (T,))
    x = (cent[lab] + 0.3 * torch.randn(T, PD)).to(dtype)
    ts = torch.arange(T).float()
    ws = ops.kmeans_workspace(T, PD, K, dev)
    rows = torch.tensor([0, 7, 13, 21, 30], dtype=torch.int32)
    xg = x.to(dev)
    d2 = ops.kmeans_sqdist(xg, None, rows.to(dev), K, ws)
    ref = torch.cdist(x.double(), x[rows.long()].double()) ** 2
    assert rel_err(d2, ref) < 1e-5
    cf = x[rows.long()].float().contiguous()
    ct = ts[rows.long()].contiguous()
    d2b = ops.kmeans_sqdist(xg, cf.to(dev), None, K, ws)
    assert rel_err(d2b, ref) < 1e-5
    assign, counts = ops.kmeans_assign(d2b, ts.to(dev), ct.to(dev), 2.0)
    df = ref.float().sqrt()
    dtm = (ts[:, None] - ct[None]).abs()
    nf = (df - df.min(1, keepdim=True).values) / (df.max(1, keepdim=True).values - df.min(1, keepdim=True).values)
    nt = (dtm - dtm.min(1, keepdim=True).values) / (dtm.max(1, keepdim=True).values - dtm.min(1, keepdim=True).values)
    ra = torch.sqrt(nf ** 2 + 2 * nt ** 2).argmin(1)
    assert torch.equal(assign.cpu(), ra)
    assert torch.equal(counts.cpu().long(), torch.bincount(ra, minlength=K))
    # force an empty cluster to exercise the reseed path
    a2 = ra.clone()
    a2[a2 == 4] = 0
    reseed = torch.tensor([0, 0, 0, 0, 17], dtype=torch.int32)
    cg, ctg = cf.to(dev).clone(), ct.to(dev).clone()
    shift = ops.kmeans_update(xg, ts.to(dev), a2.to(dev), reseed.to(dev), cg, ctg, ws)
    ncf, nct = torch.zeros_like(cf), torch.zeros_like(ct)
    for i in range(K):
        m = a2 == i
        if m.any():
            ncf[i] = x.float()[m].mean(0)
            nct[i] = ts[m].mean()
        else:
            ncf[i] = x.float()[17]
            nct[i] = ts[17]
    rs = torch.norm(ncf - cf, dim=1).sum() + torch.norm(nct - ct)
    assert rel_err(cg, ncf) < 1e-5 and rel_err(ctg, nct) < 1e-6
    assert abs(float(shift) - float(rs)) / float(rs) < 1e-5


@pytest.mark.parametrize("shape", [(3, 120, 214), (2, 56, 84), (4, 480, 854)])
def test_gpu_preprocessing_bit_exact_vs_pil_path(dev, shape):
    """uint8 frames -> pixel_values on the GPU == the PIL host path (fp32 bit-identical, bf16 = one rounding)"""
    from cogstream_amd import processing as pr
    from cogstream_amd.preprocess_gpu import preprocess_videos_gpu
    t, h, w = shape
    frames, _ = pr.synthetic_clip(t, h, w, kind="drift", clip_idx=3)
    ref = pr.preprocess_videos([frames])
    got = preprocess_videos_gpu([torch.from_numpy(frames).to(dev)], out_dtype=torch.float32)
    assert got["grid_sizes"].tolist() == ref["grid_sizes"].tolist()
    assert torch.equal(got["pixel_values"].cpu(), torch.from_numpy(ref["pixel_values"]))
    got16 = preprocess_videos_gpu([torch.from_numpy(frames).to(dev)], out_dtype=torch.bfloat16)
    assert torch.equal(got16["pixel_values"].cpu(), torch.from_numpy(ref["pixel_values"]).bfloat16())


def test_pair_epilogue_and_relaxed_vmcnt_equal_the_generic_build_bit_for_bit(dev):
    """The ping-pong GEMM's lean pair epilogue lets the next tile's first K-tile waits leave its stores in flight
    (`s_waitcnt vmcnt(8 + ops)`, csrc/gemm.hip). libcogs_hip_nopair.so is the same source built with
    -DCOGS_EPI_NOPAIR: generic epilogue, conservative waits. On the cfg2 ViT shapes (plain, bias, bias+residual,
    bias+GELU, bias+rotary table, bias+rotary LUT) and a Qwen2-prefill shape the two builds must agree bit for bit:
    a wait that lets a wave read a ring slot before its LDS-DMA pieces landed would show up here."""
    import ctypes as C
    from cogstream_amd import _lib as L2
    from cogstream_amd.build import LIB_NOPAIR
    ops = _ops()
    assert LIB_NOPAIR.exists(), "build it with `python -m cogstream_amd.build --nopair` (__graft_entry__.build does)"
    alt = C.CDLL(str(LIB_NOPAIR))
    stamp = LIB_NOPAIR.parent / "csrc" / "build" / "gemm.epi_check.txt"
    assert stamp.read_text().startswith("ok:"), stamp.read_text()      # the build's disassembly check passed
    torch.manual_seed(5)
    M = 59136 // 4                                     # a quarter of cfg2's patches: 58 row blocks, several rounds
    hd, heads = 72, 16
    H, I = 1152, 4352
    g = torch.Generator(device=dev).manual_seed(1)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    x, big = rnd(M, H), rnd(M, I)
    nf, maxpos = hd // 4, 42
    hpos = torch.randint(0, 22, (M,), generator=g, device=dev)
    wpos = torch.randint(0, maxpos, (M,), generator=g, device=dev)
    inv_freq = 1.0 / (10000.0 ** (torch.arange(nf, dtype=torch.float32, device=dev) / nf))
    lut_ang = torch.arange(maxpos, dtype=torch.float32, device=dev)[:, None] * inv_freq[None, :]
    lut = torch.stack([lut_ang.cos(), lut_ang.sin()], -1).contiguous()
    rowpos = (hpos | (wpos << 16)).to(torch.int32)
    ang = torch.cat([hpos[:, None].float() * inv_freq, wpos[:, None].float() * inv_freq], 1)
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    cases = [
        ("qkv+rope table", dict(a=x, w=rnd(3 * H, H), bias=rnd(3 * H), rope_cos=table, rope_cols=2 * H, head_dim=hd)),
        ("qkv+rope lut", dict(a=x, w=rnd(3 * H, H), bias=rnd(3 * H), rope_cos=table, rope_cols=2 * H, head_dim=hd,
                              rope_lut=lut, rope_rowpos=rowpos)),
        ("out-proj+res", dict(a=x, w=rnd(H, H), bias=rnd(H), residual=rnd(M, H))),
        ("fc1+gelu", dict(a=x, w=rnd(I, H), bias=rnd(I), act=L2.ACT_GELU_TANH)),
        ("fc2+res", dict(a=big, w=rnd(H, I), bias=rnd(H), residual=rnd(M, H))),
        ("plain", dict(a=x, w=rnd(3584, H))),
        ("proj gelu-erf", dict(a=x, w=rnd(3584, H), bias=rnd(3584), act=L2.ACT_GELU_ERF)),
        # round 6: the SwiGLU pair epilogue (lane transpose, 16-byte stores) against the generic one's two 2-byte stores
        ("gate/up swiglu", dict(a=x, w=rnd(2 * 2048, H), act=L2.ACT_SWIGLU)),
        ("gate/up swiglu, ragged N", dict(a=x, w=rnd(2 * 2000, H), act=L2.ACT_SWIGLU)),
    ]
    for name, kw in cases:
        for rep in range(2):
            a = ops.gemm(**kw)
            b = ops.gemm(**kw, lib=alt)
            torch.cuda.synchronize()
            assert torch.equal(a, b), (name, rep, float((a.float() - b.float()).abs().max()))


def test_whole_line_gemm_equals_the_k_tile_gemm_bit_for_bit(dev):
    """gemm_tn_pp64_kernel (round 4: 64-wide slabs of whole 128-byte lines in a five-unit ring, three kinds of slab, the
    two wave groups' epilogues in one interval) must produce the bits of gemm_tn_pp_kernel (32-wide K-tiles): same tile,
    same MFMA order, same epilogues. The second kernel is reached through the debug switch gemm_pp64 = 0 (the dispatch
    is asked which body ran), as the dispatch takes them -- where it sends a shape, or a split's remainder, to the mid-size kernel both
    sides have that part in common -- and with gemm_split = 0, where all of the product is theirs. Shapes: the cfg2 ViT GEMMs at a quarter of the clip (several rounds of the persistent grid,
    ragged last row block), a frame-sharded share (few tiles), the Qwen2 gate/up and down projections at 2 100 rows
    (SwiGLU epilogue; K = 18 944: 296 slabs per tile)."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(11)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()

    class _KTile:
        """stands in for the second library of the round-4 form of this test: gemm(..., lib=alt) = the K-tile body"""
    alt = _KTile()
    _gemm = ops.gemm

    def gemm_ab(**kw):
        if kw.pop("lib", None) is None:
            out = _gemm(**kw)
            assert L2.debug_get("gemm_last_body") in (2, 4, 5), L2.debug_get("gemm_last_body")
            return out
        with L2.debug_switch("gemm_pp64", 0):
            out = _gemm(**kw)
            assert L2.debug_get("gemm_last_body") in (2, 3, 5), L2.debug_get("gemm_last_body")
        return out

    def both_whole(tag, **kw):
        with L2.debug_switch("gemm_split", 0):
            a = _gemm(**kw)
            assert L2.debug_get("gemm_last_body") == 4, tag
            with L2.debug_switch("gemm_pp64", 0):
                b = _gemm(**kw)
                assert L2.debug_get("gemm_last_body") == 3, tag
        assert torch.equal(a, b), tag

    class _Ops:
        gemm = staticmethod(gemm_ab)
    ops = _Ops()
    hd, H, I = 72, 1152, 4352
    for M in (59136 // 4 + 40, 6400):
        x, big = rnd(M, H), rnd(M, I)
        nf = hd // 4
        hpos = torch.randint(0, 22, (M,), generator=g, device=dev)
        wpos = torch.randint(0, 42, (M,), generator=g, device=dev)
        inv_freq = 1.0 / (10000.0 ** (torch.arange(nf, dtype=torch.float32, device=dev) / nf))
        ang = torch.cat([hpos[:, None].float() * inv_freq, wpos[:, None].float() * inv_freq], 1)
        table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
        cases = [
            ("qkv+rope table", dict(a=x, w=rnd(3 * H, H), bias=rnd(3 * H), rope_cos=table, rope_cols=2 * H, head_dim=hd)),
            ("out-proj+res", dict(a=x, w=rnd(H, H), bias=rnd(H), residual=rnd(M, H))),
            ("fc1+gelu", dict(a=x, w=rnd(I, H), bias=rnd(I), act=L2.ACT_GELU_TANH)),
            ("fc2+res", dict(a=big, w=rnd(H, I), bias=rnd(H), residual=rnd(M, H))),
            ("plain", dict(a=x, w=rnd(3584, H))),
            ("K = 128 (two slabs)", dict(a=rnd(M, 128), w=rnd(H, 128))),
        ]
        for name, kw in cases:
            for rep in range(2):
                a = ops.gemm(**kw)
                b = ops.gemm(**kw, lib=alt)
                torch.cuda.synchronize()
                assert torch.equal(a, b), (M, name, rep, float((a.float() - b.float()).abs().max()))
            both_whole((M, name), **kw)
    xq, inter = rnd(2100, 3584), rnd(2100, 18944)
    for name, kw in (("gate/up swiglu", dict(a=xq, w=rnd(2 * 18944, 3584), act=L2.ACT_SWIGLU)),
                     ("down+res", dict(a=inter, w=rnd(3584, 18944), residual=rnd(2100, 3584)))):
        a = ops.gemm(**kw)
        b = ops.gemm(**kw, lib=alt)
        torch.cuda.synchronize()
        assert torch.equal(a, b), (name, float((a.float() - b.float()).abs().max()))
        both_whole(name, **kw)


def test_tall_ragged_column_tiles_equal_padded_tiles_bit_for_bit(dev):
    """Round 6: gemm_tn_pp64_kernel walks a ragged column block of <= 128 columns (N = 1152: 4.5 blocks of 256, N = 3456:
    13.5) as tiles of 384 rows x 128 columns through the same LDS ring (csrc/gemm.hip, TALL4) instead of a half-empty 256 x 256
    tile. Every output element keeps its MFMAs and its K order, so the results must be the bits of the padded walk (debug switch
    gemm_tall = 0). Shapes: row counts that are / are not multiples of 384 and of 256, fewer rows than one tall tile's second
    and third row group, a ragged block narrower than 128 columns (generic epilogue in its second column group), every fused
    ViT epilogue of an N = 1152 / 3456 GEMM (bias + residual + row statistics, rotary + head-major), walk groups forced to
    3 / 6 / 9 row blocks, and the few-tile split choices of a frame-sharded share. The dispatch sends most of these shapes, or part of
    them, to the mid-size kernel: with gemm_split = 0 every shape that pads to whole column blocks by at most 12 % is all theirs."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(17)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    hd, H, I = 72, 1152, 4352

    def both(tag, **kw):
        outs = []
        for tall in (1, 0):
            with L2.debug_switch("gemm_tall", tall):
                rs = kw.get("row_stats")
                if rs is not None:
                    rs.fill_(-7.0)
                o = ops.gemm(**kw).clone()
                body = L2.debug_get("gemm_last_body")
                outs.append((o, None if rs is None else rs.clone(), body))
        torch.cuda.synchronize()
        (a, sa, ba), (b, sb, bb) = outs
        assert torch.equal(a, b), (tag, ba, bb, float((a.float() - b.float()).abs().max()))
        if sa is not None:
            assert torch.equal(sa, sb), (tag, "row statistics")
        return ba

    bodies = set()
    for M in (59136 // 4, 59136 // 4 + 40, 7392, 6400, 1024, 1280 + 8, 1536, 3 * 384 + 130, 2049):
        x, big = rnd(M, H), rnd(M, I)
        nf = hd // 4
        hpos = torch.randint(0, 22, (M,), generator=g, device=dev)
        wpos = torch.randint(0, 42, (M,), generator=g, device=dev)
        inv_freq = 1.0 / (10000.0 ** (torch.arange(nf, dtype=torch.float32, device=dev) / nf))
        ang = torch.cat([hpos[:, None].float() * inv_freq, wpos[:, None].float() * inv_freq], 1)
        table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
        stats = torch.empty(M, H // 64, 2, device=dev, dtype=torch.float32)
        ln_ab = torch.rand(M, 2, generator=g, device=dev) + 0.5
        col_c = torch.randn(3 * H, generator=g, device=dev)
        cases = [
            ("out-proj + residual + statistics", dict(a=x, w=rnd(H, H), bias=rnd(H), residual=rnd(M, H), row_stats=stats)),
            ("fc2 + residual + statistics", dict(a=big, w=rnd(H, I), bias=rnd(H), residual=rnd(M, H), row_stats=stats)),
            ("qkv + rotary, head-major, LN fold", dict(a=x, w=rnd(3 * H, H), rope_cos=table, rope_cols=2 * H, head_dim=hd,
                                                       ln_ab=ln_ab, col_c=col_c, hm_cols=H)),
            ("qkv + rotary, row-major", dict(a=x, w=rnd(3 * H, H), bias=rnd(3 * H), rope_cos=table, rope_cols=2 * H, head_dim=hd)),
            ("plain, 1.5 column blocks", dict(a=x, w=rnd(384, H))),
            ("plain, ragged block of 76 columns", dict(a=x, w=rnd(1100, H), bias=rnd(1100))),
            ("K = 128 (two slabs)", dict(a=rnd(M, 128), w=rnd(H, 128))),
        ]
        for name, kw in cases:
            bodies.add(both((M, name), **kw))
            with L2.debug_switch("gemm_split", 0):
                n = kw["w"].shape[0]
                assert both((M, name, "unsplit"), **kw) == (4 if -(-n // 256) * 256 * 100 <= n * 112 else 2)
        for gm in (3, 4, 9):
            with L2.debug_switch("gemm_group_m", gm), L2.debug_switch("gemm_split", 0):
                bodies.add(both((M, "group_m", gm), **cases[0][1]))
    assert 4 in bodies, bodies          # the whole-line kernel (and with it the tall walk) did run


@pytest.mark.parametrize("variant", ["deep", "round4", "general", "general hd72"])
def test_prescaled_attention_survives_a_key_far_above_the_running_reference(dev, variant):
    """The deferred-maximum softmax of the pre-scaled kernels evaluates P = exp2(score - reference) against the reference it had
    BEFORE the tile and rescales (O, l) afterwards; a key more than ~127 log2 units above everything a row has seen made P
    infinite and the deferred factor turned it into inf * 0 = NaN. Such a tile now moves the
    reference in front of its exponentials (PRE_FAR, csrc/attn.hip). One key in the middle of the sequence is scaled until
    its scores reach +-400 log2 units: the output must be finite and as close to the fp32 softmax as without that key."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    hd = 72 if variant.endswith("hd72") else 128
    hq, hkv = (4, 4) if hd == 72 else (28, 4)
    S, far = 1100, 733
    g = torch.Generator().manual_seed(S + hd)
    q = (torch.randn(S, hq * hd, generator=g) * (LOG2E / math.sqrt(hd))).bfloat16()
    k = torch.randn(S, hkv * hd, generator=g).bfloat16()
    v = torch.randn(S, hkv * hd, generator=g).bfloat16()
    k[far] *= 300.0
    big = (q.float().view(S, hq, hd)[far:, :, :] * k.float().view(S, hkv, hd)[far].repeat_interleave(hq // hkv, 0)).sum(-1)
    assert float(big.max()) > 160 and float(big.min()) < -160        # both signs, far beyond fp32's exponent range for exp2
    sw = {"deep": {"attn_prefill_deep": 1}, "round4": {"attn_prefill_deep": 0}, "general": {"attn_prefill_dma": 0},
          "general hd72": {}}[variant]
    causal = hd == 128
    import contextlib
    with contextlib.ExitStack() as st:
        for name, val in sw.items():
            st.enter_context(L2.debug_switch(name, val))
        if hd == 72:
            st.enter_context(L2.debug_switch("attn_vit", 0))
        kw = dict(hq=hq, hkv=hkv, head_dim=hd, causal=causal, q_prescaled=True)
        if hd == 72:
            kw.update(cu_seqlens=torch.tensor([0, S], dtype=torch.int32, device=dev), max_seqlen=S)
        out = ops.attention(q.to(dev), k.to(dev), v.to(dev), **kw)
        want = {"deep": 5, "round4": 5, "general": 1, "general hd72": 1}[variant]
        assert L2.debug_get("attn_last_kernel") == want, L2.debug_get("attn_last_kernel")
    assert torch.isfinite(out.float()).all(), "NaN / inf rows: %d" % int((~torch.isfinite(out.float())).any(1).sum())
    ref = _attn_ref(q, k, v, hq, hkv, hd, causal=causal, scale=math.log(2.0))
    assert rel_err(out.float(), ref) < 1.5e-2, rel_err(out.float(), ref)


def test_round5_prompt_attention_kernel_is_as_close_to_fp32_as_the_round4_kernel(dev):
    """attn_prefill_dma_kernel<1> (round 5, the default) re-orders attn_prefill_dma_kernel<0> (round 4): fragment reads ahead
    of their MFMAs, and the running reference only moves when a score exceeds it by 2^6 (P <= 64 instead of <= 1 before the
    bf16 rounding), so the two outputs differ like two bf16 roundings do; what must hold is that the new kernel is as close to
    the fp32 softmax as the old one. Whole prompts, ragged lengths, two- and three-tile prompts, one-tile sequences in the
    var-len form, prefix-KV continuation (also with fewer than 128 new rows), a late dominant key (the rescale path)."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(5)
    hq, hkv, hd = 28, 4, 128
    mk = lambda n, h, sc=0.5: (torch.randn(n, h * hd, generator=g, device=dev) * sc).bfloat16()

    def both(*a, **kw):
        with L2.debug_switch("attn_prefill_deep", 1):
            x = ops.attention(*a, **kw)
            assert L2.debug_get("attn_last_kernel") == 5
        with L2.debug_switch("attn_prefill_deep", 0):
            y = ops.attention(*a, **kw)
            assert L2.debug_get("attn_last_kernel") == 5
        torch.cuda.synchronize()
        assert torch.isfinite(x.float()).all()
        cu = kw.get("cu_seqlens")
        ref = _attn_ref(a[0].cpu(), a[1].cpu(), a[2].cpu(), hq, hkv, hd, cu=None if cu is None else cu.cpu().long(), causal=True,
                        q_pos0=kw.get("q_pos0", 0), scale=math.log(2.0))
        e_new, e_old = rel_err(x.float(), ref), rel_err(y.float(), ref)
        assert e_new < 1.2e-2 and e_new <= 1.5 * e_old + 1e-3, (e_new, e_old)
    for S, pos0 in ((4096, 0), (2100, 0), (2433, 0), (300, 0), (128, 0), (129, 0), (191, 0), (192, 0), (193, 0), (1000, 1500), (130, 700), (127, 173), (5, 40), (64, 0), (63, 0), (2, 0)):
        q, kk, v = mk(S, hq), mk(S + pos0, hkv), mk(S + pos0, hkv, 1.0)
        if S > 2000:
            kk[S - 700] *= 6.0                                                   # the maximum moves late, by a lot
        both(q, kk, v, hq=hq, hkv=hkv, head_dim=hd, causal=True, q_prescaled=True, q_pos0=pos0)
    lens = [300, 1, 64, 129, 1000, 63, 512]
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev)
    S = sum(lens)
    q, kk, v = mk(S, hq), mk(S, hkv), mk(S, hkv, 1.0)
    both(q, kk, v, hq=hq, hkv=hkv, head_dim=hd, causal=True, q_prescaled=True, cu_seqlens=cu, max_seqlen=max(lens))


@pytest.mark.parametrize("M", [300, 1300, 4096])
def test_gemm_row_stats_and_ln_fold(dev, gemm_split, M):
    """LayerNorm fused around the GEMMs: (1) a residual-stream GEMM (N = hidden) also writes per-row partial sums,
    cogs_ln_finalize turns them into (rstd, -rstd * mean); (2) the consuming GEMM reads x itself with W * diag(gamma)
    (rows centred) and applies rstd_r * acc + c_n -- together LN(x) W^T + bias of nn.LayerNorm + nn.Linear
    (model/modeling_videollama3_encoder.py:382-391). The mid-size kernel (as dispatched) and the ping-pong kernel with
    ragged last row blocks."""
    ops = _ops()
    torch.manual_seed(M)
    H, N2, eps = 1152, 1472, 1e-6
    a0 = torch.randn(M, 256).bfloat16()
    w0 = (torch.randn(H, 256) / 16).bfloat16()
    b0 = torch.randn(H).bfloat16()
    res = (torch.randn(M, H) * 2 + 0.7).bfloat16()                       # rows with a clearly non-zero mean
    res[::7] += 16.0                                                     # and some with |mean / std| ~ 8
    res[3::11] += 200.0                                                  # and ~ 100 (rows dominated by their mean)
    y32 = a0.float() @ w0.float().t() + b0.float() + res.float()
    part = torch.zeros(M, H // 64, 2, device=dev)
    x = ops.gemm(a0.to(dev), w0.to(dev), b0.to(dev), residual=res.to(dev), row_stats=part)
    assert rel_err(x.float(), y32) < 1.2e-2
    xs = x.float().cpu()                                                 # the statistics are those of the STORED rows
    want = torch.stack([xs.view(M, H // 64, 64).sum(-1), (xs ** 2).view(M, H // 64, 64).sum(-1)], -1)
    assert rel_err(part, want) < 1e-5
    ab = ops.ln_finalize(part, H, eps)
    mean, var = xs.double().mean(1).float(), xs.double().var(1, unbiased=False).float()
    rstd = (var + eps).rsqrt()
    # rows dominated by their mean (|mean / std| ~ 100) lose (mean/std)^2 of the fp32 partial sums' precision in
    # E[x^2] - mean^2: 1e-3 there, 1e-4 everywhere else -- both far below the bf16 rounding of the consumer's output
    huge_rows = torch.zeros(M, dtype=torch.bool)
    huge_rows[3::11] = True
    abc = ab.cpu()
    for rows, tol in ((~huge_rows, 1e-4), (huge_rows, 1e-3)):
        assert rel_err(abc[rows, 0], rstd[rows]) < tol and rel_err(abc[rows, 1], (-rstd * mean)[rows]) < tol
    # consumer: fc1-like (GELU) and plain
    gamma, beta = (1 + 0.3 * torch.randn(H)).bfloat16(), (0.2 * torch.randn(H)).bfloat16()
    w1 = (torch.randn(N2, H) / 30).bfloat16()
    b1 = torch.randn(N2).bfloat16()
    from cogstream_amd.weights import fold_layernorm
    wf, col_s, col_c = fold_layernorm(w1, b1, gamma, beta)               # W * gamma, rows centred AND zero-sum after rounding
    # the stored bf16 rows sum to zero up to one step of their smallest entries (plain rounding leaves ~1e-2 of |w|_1 / K)
    assert float(col_s.abs().max()) < 1e-5 * float(wf.float().abs().sum(1).mean())
    xr = x.float().cpu()
    ln = F.layer_norm(xr, (H,), gamma.float(), beta.float(), eps)
    for act, fn in ((L_ACT_NONE(), lambda t: t), (L_ACT_GELU(), lambda t: F.gelu(t, approximate="tanh"))):
        ref = fn(ln @ w1.float().t() + b1.float())
        out = ops.gemm(x, wf.to(dev), None, act=act, ln_ab=ab, col_c=col_c.to(dev))
        unfused = ops.gemm(ln.bfloat16().to(dev), w1.to(dev), b1.to(dev), act=act)
        # every row class -- ordinary mean, |mean / std| ~ 8 and ~ 100 -- is as accurate as the unfused bf16 path: with
        # zero-sum weight rows the product on x equals the product on x - mean, whatever the mean (round 2 allowed the
        # |mean / std| ~ 8 rows 9x the error: the bf16 rounding of the centred rows left a row sum that the mean multiplied)
        big = torch.zeros(M, dtype=torch.bool)
        big[::7] = True
        huge = torch.zeros(M, dtype=torch.bool)
        huge[3::11] = True
        for rows in (~(big | huge), big & ~huge, huge):
            e_f, e_u = rel_err(out.float().cpu()[rows], ref[rows]), rel_err(unfused.float().cpu()[rows], ref[rows])
            assert e_f < 2.0 * e_u + 2e-3, (act, e_f, e_u)


def test_ln_fold_through_the_c_abi_as_the_header_states_it(dev):
    """cogs_gemm with ln_ab, called through ctypes with operands built by hand from the text of include/cogs.h
    (cogs_gemm_desc.ln_ab): W = rows of W0 * diag(gamma) minus their mean over k, col_c = bias0 + W0 . beta, bias NULL,
    ln_ab[r] = (rstd_r, anything) -- equals nn.Linear(nn.LayerNorm(x)). The second component of ln_ab is filled with
    garbage: the header says it is not read. Unsupported combinations return COGS_E_UNSUPPORTED instead of silently
    dropping the LayerNorm (M == 1 -> GEMV; ln_ab + residual -> no specialised epilogue)."""
    import ctypes as C
    from cogstream_amd import _lib as L
    torch.manual_seed(5)
    M, H, N, eps = 1500, 1152, 640, 1e-6
    x = (torch.randn(M, H) * 1.5 + 0.4).bfloat16()
    gamma, beta = (1 + 0.2 * torch.randn(H)).bfloat16(), (0.1 * torch.randn(H)).bfloat16()
    w0, b0 = (torch.randn(N, H) / 30).bfloat16(), torch.randn(N).bfloat16()
    wg = w0.double() * gamma.double()[None, :]
    w = (wg - wg.mean(dim=1, keepdim=True)).to(torch.bfloat16).contiguous()          # the header's W, rounded once
    col_c = (b0.double() + w0.double() @ beta.double()).float()
    xf = x.float()
    rstd = (xf.var(1, unbiased=False) + eps).rsqrt()
    ln_ab = torch.stack([rstd, torch.full_like(rstd, 1e30)], 1).contiguous()         # [r][1] must not be read
    ref = F.layer_norm(xf, (H,), gamma.float(), beta.float(), eps) @ w0.float().t() + b0.float()
    xd, wd_, cd, abd = x.to(dev), w.to(dev), col_c.to(dev), ln_ab.to(dev)
    out = torch.empty(M, N, device=dev, dtype=torch.bfloat16)

    def desc(m, **kw):
        d = L.GemmDesc()
        d.dtype = L.DT_BF16
        d.A, d.lda, d.W, d.ldw, d.C, d.ldc = xd.data_ptr(), H, wd_.data_ptr(), H, out.data_ptr(), N
        d.M, d.N, d.K = m, N, H
        d.ln_ab, d.col_c = abd.data_ptr(), cd.data_ptr()
        for k, v in kw.items():
            setattr(d, k, v)
        return d

    assert L.lib.cogs_gemm(L.current_stream(), C.byref(desc(M))) == L.OK
    torch.cuda.synchronize()
    assert rel_err(out.float().cpu(), ref) < 1e-2
    assert L.lib.cogs_gemm(L.current_stream(), C.byref(desc(1))) == L.E_UNSUPPORTED
    assert L.lib.cogs_gemm(L.current_stream(), C.byref(desc(M, residual=xd.data_ptr(), ldr=H))) == L.E_UNSUPPORTED
    stats = torch.zeros(M, N // 64, 2, device=dev)
    d = desc(M, act=L.ACT_GELU_ERF)
    d.ln_ab, d.col_c, d.row_stats = None, None, stats.data_ptr()
    assert L.lib.cogs_gemm(L.current_stream(), C.byref(d)) == L.E_UNSUPPORTED        # row_stats + GELU(erf): no such epilogue


@pytest.mark.parametrize("n", [1, 2, 3, 8])
def test_select_near_centroid_vs_torch(dev, n):
    """cogs_select_near_centroid against the reference's per-cluster logic (model/cogreasoner_chat.py:50-64: members if at
    most n, else members[topk(dist, n, largest=False)]) on random distances: clusters with 0, fewer than n, exactly n and
    many members; T beyond one 64-row sweep; exact ties go to the lower row."""
    ops = _ops()
    torch.manual_seed(70 + n)
    T, K = 333, 11
    d2 = torch.rand(T, K)
    d2[5::40] = d2[6::40][: d2[5::40].shape[0]]                                # some exactly equal rows (ties)
    assign = torch.randint(0, K - 3, (T,))
    assign[:2] = K - 3                                                        # a cluster with 2 members
    assign[2:2 + n] = K - 2                                                   # a cluster with exactly n members (cluster K-1: none)
    picks, counts = ops.select_near_centroid(d2.to(dev), assign.to(dev), n)
    picks, counts = picks.cpu(), counts.cpu()
    for k in range(K):
        members = torch.nonzero(assign == k, as_tuple=True)[0]
        if members.numel() <= n:
            want = members
        else:
            dk = d2[members, k]
            order = sorted(range(members.numel()), key=lambda i: (float(dk[i]), int(members[i])))[:n]
            want = members[torch.tensor(order)]
        assert int(counts[k]) == want.numel()
        assert picks[k, :want.numel()].tolist() == want.tolist()
        assert (picks[k, want.numel():] == -1).all()


def L_ACT_NONE():
    from cogstream_amd import _lib as L
    return L.ACT_NONE


def L_ACT_GELU():
    from cogstream_amd import _lib as L
    return L.ACT_GELU_TANH


@pytest.mark.parametrize("M,heads,fold", [(96, 2, False), (1300, 2, True), (1300, 7, True), (2048 + 40, 16, True), (6400, 16, False),
                                          (14824, 16, True)])
def test_gemm_head_major_output_equals_row_major_bit_for_bit(dev, gemm_split, M, heads, fold):
    """cogs_gemm_desc.hm_rows (round 5: the encoder's QKV GEMM stores q | k | v as [block][head][row][hd] so that the
    attention kernel streams whole 128-byte lines): the same epilogue arithmetic, only the store address changes -- the
    head-major result must be the row-major result re-arranged, bit for bit. heads = 2 / 7: hm_cols is not a multiple of
    64, so a wave tile straddles q / k / v and every tile takes the general epilogue; heads = 16 (the production width):
    interior tiles take the lean paired epilogue; M covers the mid-size and ping-pong kernels, a ragged last
    row block, and the round-aligned split (6 400 rows as dispatched)."""
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M + heads)
    hd, K = 72, 1152 if heads == 16 else 128
    Hc = heads * hd
    N = 3 * Hc
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    x = rnd(M, K) + 0.25
    ang = torch.rand(M, hd // 2, generator=g, device=dev) * 6.0
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    kw = dict(rope_cos=table, rope_sin=None, rope_cols=2 * Hc, head_dim=hd)
    if fold:
        from cogstream_amd.weights import fold_layernorm
        wf, _, col_c = fold_layernorm(rnd(N, K).cpu(), rnd(N).cpu(), (1 + 0.3 * torch.randn(K)).bfloat16(), (0.2 * torch.randn(K)).bfloat16())
        xs = x.float()
        rstd = (xs.var(1, unbiased=False) + 1e-6).rsqrt()
        ab = torch.stack([rstd, -rstd * xs.mean(1)], 1).contiguous()
        args = dict(a=x, w=wf.to(dev), bias=None, ln_ab=ab, col_c=col_c.to(dev), **kw)
    else:
        args = dict(a=x, w=rnd(N, K), bias=rnd(N), **kw)
    row = ops.gemm(**args)
    hm = ops.gemm(**args, hm_cols=Hc)
    torch.cuda.synchronize()
    assert hm.shape == (3, heads, M, hd)
    want = row.view(M, 3, heads, hd).permute(1, 2, 0, 3)
    assert torch.equal(hm, want), float((hm.float() - want.float()).abs().max())


@pytest.mark.parametrize("heads,lens", [(1, [1]), (2, [32, 33]), (1, [63, 64, 65]), (8, [200] * 5), (2, [255, 256, 257]),
                                        (16, [924, 924]), (3, [1024, 70, 1000]), (16, [130] * 4)])
@pytest.mark.parametrize("variant", [2, 1])
def test_attention_head_major_inputs_equal_token_major_bit_for_bit(dev, heads, lens, variant):
    """cogs_attn_desc.head_stride: the encoder's attention kernels (pipelined LDS-DMA kernel = debug switch attn_vit 2,
    unpipelined = 1) reading q, k, v as [head][row][72] -- contiguous key tiles, whole-line LDS-DMA pieces -- must give the
    bits they give on the token-major fused buffer: only the source addresses differ. Ragged last tiles (rows past a
    segment's end are re-read from its last row, never from the next frame or head), one-row segments, both grid orders."""
    from cogstream_amd import _lib as L
    ops = _ops()
    hd, H = 72, heads * 72
    n = sum(lens)
    g = torch.Generator(device=dev).manual_seed(n + heads)
    qkv = torch.randn(n, 3 * H, generator=g, device=dev)
    qkv[:, :H] *= LOG2E / math.sqrt(hd)
    qkv = qkv.bfloat16()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev)
    with L.debug_switch("attn_vit", variant):
        tok = ops.attention(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], hq=heads, hkv=heads, head_dim=hd, cu_seqlens=cu,
                            max_seqlen=max(lens), q_prescaled=True)
        assert L.debug_get("attn_last_kernel") == (3 if variant == 2 else 2)
        hm3 = qkv.view(n, 3, heads, hd).permute(1, 2, 0, 3).contiguous()           # [3][heads][n][hd], one buffer
        out = ops.attention(hm3[0], hm3[1], hm3[2], hq=heads, hkv=heads, head_dim=hd, cu_seqlens=cu, max_seqlen=max(lens),
                            q_prescaled=True, head_major=True)
        assert L.debug_get("attn_last_kernel") == (8 if variant == 2 else 2)
        # the same with GUARD rows behind every head's rows (head stride = (n + 70) rows): a ragged last tile must repeat the
        # segment's last row, never read on into what follows the head. The guards hold a huge FINITE value (the kernel file is
        # built with -fno-honor-nans, so a NaN is no reliable tracer): one of them taken for a key would own its softmax row,
        # one taken for a value would blow the output up
        G = 70
        guarded = torch.full((3, heads, n + G, hd), 3.0e38, device=dev, dtype=torch.bfloat16)
        guarded[:, :, :n] = hm3
        outg = ops.attention(guarded[0][:, :n], guarded[1][:, :n], guarded[2][:, :n], hq=heads, hkv=heads, head_dim=hd,
                             cu_seqlens=cu, max_seqlen=max(lens), q_prescaled=True, head_major=True)
        assert L.debug_get("attn_last_kernel") == (8 if variant == 2 else 2)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    assert torch.equal(out, tok), float((out.float() - tok.float()).abs().max())
    assert torch.equal(outg, tok), "guard rows behind a head's rows were read: %g" % float((outg.float() - tok.float()).abs().max())


@pytest.mark.parametrize("lens,hq,hkv,pos0", [((1,), 4, 2, 3), ((63,), 28, 4, 0), ((65,), 28, 4, 64), ((127,), 4, 4, 1), ((129,), 28, 4, 500), ((320,), 8, 1, 0),
                                              ((621,), 28, 4, 0), ((1, 64, 130, 7), 4, 2, 0)])
def test_prompt_attention_of_64_row_workgroups(dev, lens, hq, hkv, pos0):
    """attn.hip, prompt kernel: query tiles of 64 rows (few of them) and of 128 (attn_prio 1 keeps to those) give the same bits, at the edges of
    both and of key tiles, behind kept keys, and in segments; and the float64 result within the weights' and the output's bf16 rounding
    (2^-8 each, of values up to the largest |v|)"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(sum(lens) + pos0)
    n = sum(lens)
    q = torch.randn(n, hq * 128, generator=g, device=dev).bfloat16() * 0.2
    k, v = (torch.randn(n + pos0, hkv * 128, generator=g, device=dev).bfloat16() for _ in range(2))
    kw = dict(hq=hq, hkv=hkv, head_dim=128, causal=True, q_prescaled=True, q_pos0=pos0)
    if len(lens) > 1:
        kw["cu_seqlens"] = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=dev)
        kw["max_seqlen"] = max(lens)
    got = ops.attention(q, k, v, **kw)
    with L2.debug_switch("attn_prio", 1):
        assert torch.equal(got, ops.attention(q, k, v, **kw))
    at = 0
    for m in lens:
        K, V = (t[at:at + m + pos0].double().view(m + pos0, hkv, 128).repeat_interleave(hq // hkv, 1) for t in (k, v))
        s = (q[at:at + m].double().view(m, hq, 128).transpose(0, 1) @ K.permute(1, 2, 0).contiguous()) * math.log(2.0)
        s = s.masked_fill(torch.arange(m + pos0, device=dev)[None, None] > torch.arange(m, device=dev)[None, :, None] + pos0, -math.inf)
        want = (s.softmax(-1) @ V.transpose(0, 1).contiguous()).transpose(0, 1).reshape(m, hq * 128)
        assert float((got[at:at + m].double() - want).abs().max()) <= float(V.abs().max()) * 2.0 ** -7
        at += m


@pytest.mark.parametrize("hq,hkv,rows,pos0,want", [(28, 4, 1280, 0, 64), (28, 4, 1280, 1281, 128), (28, 4, 1152, 9000, 64), (28, 4, 1500, 0, 128),
                                                   (64, 8, 621, 4000, 128), (64, 8, 512, 4000, 64)])
def test_prompt_attention_rows_behind_kept_keys(dev, hq, hkv, rows, pos0, want):
    """query tiles of 64 rows are for prompts whose tiles of 128 leave CUs idle, and, up to 320 of those, for prompts that are not mostly
    kept keys; the same bits either way"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(rows + pos0)
    q = torch.randn(rows, hq * 128, generator=g, device=dev).bfloat16() * 0.2
    k, v = (torch.randn(rows + pos0, hkv * 128, generator=g, device=dev).bfloat16() for _ in range(2))
    kw = dict(hq=hq, hkv=hkv, head_dim=128, causal=True, q_prescaled=True, q_pos0=pos0)
    got = ops.attention(q, k, v, **kw)
    assert L2.debug_get("attn_last_rows") == want
    with L2.debug_switch("attn_prio", 1):
        assert torch.equal(got, ops.attention(q, k, v, **kw))
        assert L2.debug_get("attn_last_rows") == 128


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("M,N,K", [(1147, 328, 192), (1537, 1544, 128), (100, 9000, 640)])
def test_mid_size_gemm_groups_of_row_tiles(dev, tile, M, N, K):
    """gemm_mid.hip: row tiles in groups of up to twelve, as equal as they come (9, 10 and 13 tiles of 128 rows, 8 to 49 of the other
    heights, a shorter last group), with all, some and none of the weights fetched ahead by the workgroups behind the tiles'. Against
    float64: half a bf16 step of the value and 2^-20 of the sum of |a||w| for fp32 sums of up to 640 products."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M + tile)
    a, w = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, K), (N, K)))
    with L2.debug_switch("gemm_mid", tile):
        got = ops.gemm(a, w).double()
    want, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    assert bool(((got - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -20).all())


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
def test_mid_size_gemm_tiles_equal_each_other_and_fp64(dev, tile):
    """gemm_mid.hip: every tile size, forced, at the edges of its tiles (rows and columns one short of and past a tile, a ragged
    last one, fewer slabs than the ring has slots, odd slab counts), with each fused epilogue. Against float64 products of the same bf16
    operands: the output's rounding is half a bf16 step (8 significant bits: spacing 2^-7 in [1, 2), half of it 2^-8 of the value at the
    most), the fp32 sums of up to 1152 products add at most 2^-20 of the sum of |a||w|; fp32 outputs only have the latter; behind an
    activation (slope 1.13 at the most) the sums' part grows by that and its exponential and reciprocal add 2^-18 of the value; the
    statistics are sums of the stored values. And bit for bit against the tile that the dispatch picks and, from 256 rows on and where N
    pads to 256 by at most 12 %, the ping-pong kernel: a row's bits must not depend on either."""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(tile)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    for M, N, K in ((2, 4, 64), (31, 60, 128), (33, 64, 192), (63, 132, 320), (65, 128, 384), (127, 260, 448), (129, 384, 512), (300, 700, 1152), (640, 1152, 640)):
        a, w, b, r = rnd(M, K), rnd(N, K), rnd(N), rnd(M, N)
        cases = [("plain", {}), ("bias", dict(bias=b)), ("residual", dict(bias=b, residual=r)), ("fp32", dict(out_f32=True)),
                 ("gelu", dict(bias=b, act=L2.ACT_GELU_TANH)), ("swiglu", dict(act=L2.ACT_SWIGLU))]
        if N % 64 == 0:
            cases.append(("statistics", dict(bias=b, residual=r, row_stats=torch.empty(M, N // 64, 2, device=dev))))
            table = torch.randn(M, 32, 2, generator=g, device=dev)
            fold = dict(ln_ab=torch.rand(M, 2, generator=g, device=dev) + 0.5, col_c=torch.randn(N, generator=g, device=dev))
            cases += [("rotary", dict(bias=b, rope_cos=table, rope_cols=64, head_dim=64)), ("folded norm", fold),
                      ("rotary, head-major, folded norm", dict(rope_cos=table, rope_cols=64, head_dim=64, hm_cols=N, **fold))]
        for name, kw in cases:
            outs = []
            for t, split in ((tile, 1), (0, 1)) + (((0, 0),) if M >= 256 and -(-N // 256) * 256 * 100 <= N * 112 else ()):
                with L2.debug_switch("gemm_mid", t), L2.debug_switch("gemm_split", split):
                    stats = kw.get("row_stats")
                    if stats is not None:
                        stats.fill_(-7.0)
                    outs.append((ops.gemm(a, w, **kw).clone(), None if stats is None else stats.clone()))
                    assert split or L2.debug_get("gemm_last_body") == 4
            x, sx = outs[0]
            for y, sy in outs[1:]:
                assert torch.equal(x, y), (M, N, K, name)
                assert sx is None or torch.equal(sx, sy), (M, N, K, name)
            ref = a.double() @ w.double().t()
            size = a.double().abs() @ w.double().abs().t()
            if sx is not None:
                blocks = x.double().view(M, N // 64, 64)
                for got, terms in ((sx[..., 0], blocks), (sx[..., 1], blocks ** 2)):
                    assert bool(((got.double() - terms.sum(-1)).abs() <= terms.abs().sum(-1) * 2.0 ** -18).all()), (M, N, K, name)
            if name == "gelu":
                z = ref + b.double()
                want = F.gelu(z, approximate="tanh")
                bound = size * 1.13 * 2.0 ** -20 + z.abs() * 2.0 ** -18 + want.abs() * 2.0 ** -8 + 1e-30
                assert bool(((x.double() - want).abs() <= bound * 1.01).all()), (M, N, K, name)
            if name == "swiglu":
                gate, up, eg, eu = ref[:, 0::2], ref[:, 1::2], size[:, 0::2] * 2.0 ** -20, size[:, 1::2] * 2.0 ** -20
                want = F.silu(gate) * up
                bound = 1.13 * up.abs() * eg + F.silu(gate).abs() * eu + 1.13 * eg * eu + (gate * up).abs() * 2.0 ** -18 + want.abs() * 2.0 ** -8 + 1e-30
                assert bool(((x.double() - want).abs() <= bound * 1.01).all()), (M, N, K, name)
            if name == "folded norm":
                ab, cc = kw["ln_ab"].double()[:, :1], kw["col_c"].double()
                want = ab * ref + cc
                bound = ab * size * 2.0 ** -20 + (want.abs() + cc.abs()) * 2.0 ** -22 + want.abs() * 2.0 ** -8
                assert bool(((x.double() - want).abs() <= bound * 1.01).all()), (M, N, K, name)
            if name in ("plain", "bias", "residual", "fp32"):
                if "bias" in kw:
                    ref += b.double()
                if "residual" in kw:
                    ref += r.double()
                bound = size * 2.0 ** -20 + (0 if name == "fp32" else ref.abs() * 2.0 ** -8 + 1e-30)
                assert bool(((x.double() - ref).abs() <= bound * 1.01).all()), (M, N, K, name)


@pytest.mark.parametrize("M,N,K", [(600, 3584, 3584), (600, 3584, 18944), (2048, 1152, 4352)])
def test_tiles_that_want_every_cu_are_not_chosen_beside_another_stream(dev, M, N, K):
    """160x64 is for a product that has the chip to itself; the bits do not depend on it"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M + K)
    a, w = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, K), (N, K)))
    alone = ops.gemm(a, w)
    assert L2.debug_get("gemm_last_tile") == 7
    with L2.debug_switch("gemm_co_streams", 2):
        beside = ops.gemm(a, w)
        assert L2.debug_get("gemm_last_tile") in (4, 5)
    assert torch.equal(alone, beside)


@pytest.mark.parametrize("M,want", [(129, 4), (160, 4), (320, 7)])
def test_one_row_of_160_row_tiles_is_not_chosen(dev, M, want):
    """it would read every weight for itself, 64 columns a workgroup"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M)
    N = 11264 if M <= 160 else 6176
    a, w = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in ((M, 2048), (N, 2048)))
    got = ops.gemm(a, w)
    assert L2.debug_get("gemm_last_tile") == want
    with L2.debug_switch("gemm_mid", 11 - want):
        assert torch.equal(got, ops.gemm(a, w))


@pytest.mark.parametrize("tile", [6, 7])
def test_mid_size_gemm_tiles_of_two_slabs_and_of_160_rows(dev, tile):
    """the same edges for 128x64 with two slabs a slot and 160x64 (five row blocks a wave)"""
    test_mid_size_gemm_tiles_equal_each_other_and_fp64(dev, tile)


@pytest.mark.parametrize("tile", [8, 9, 10, 11])
def test_mid_size_gemm_tiles_of_96_160_and_192_rows(dev, tile):
    """the same edges for 96x64, 160x128, 192x128 and 160x256: pieces of a slab that the waves do not share evenly, three and five row
    blocks a wave (a folded norm's factors: fewer rows than lanes, more than lanes); and their groups of row tiles"""
    test_mid_size_gemm_tiles_equal_each_other_and_fp64(dev, tile)
    test_mid_size_gemm_groups_of_row_tiles(dev, tile, 1537, 1544, 128)


@pytest.mark.parametrize("M,N,K", [(700, 25600, 512), (4096, 6176, 512), (1030, 16640, 512), (2100, 9000, 512)])
def test_whole_rounds_and_an_l_shaped_rest_equal_one_launch(dev, M, N, K):
    """gemm.hip: whole rounds of ping-pong tiles over some row and column blocks and the rest of the product in one mid-size launch
    (a strip of columns; columns and rows; ragged in either) give the bits of the ping-pong kernel alone: with a residual that
    is overwritten (a tile that two launches computed would add it twice), statistics, rotation, a folded norm, SwiGLU"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    a, w, b, r = rnd(M, K), rnd(N, K), rnd(N), rnd(M, N)
    cases = [("bias", dict(bias=b)), ("residual", dict(residual=r)), ("swiglu", dict(act=L2.ACT_SWIGLU)), ("fp32", dict(out_f32=True))]
    if N % 64 == 0:
        fold = dict(ln_ab=torch.rand(M, 2, generator=g, device=dev) + 0.5, col_c=torch.randn(N, generator=g, device=dev))
        cases += [("statistics", dict(bias=b, residual=r, row_stats=torch.empty(M, N // 64, 2, device=dev))), ("folded norm", fold),
                  ("rotary", dict(rope_cos=torch.randn(M, 32, 2, generator=g, device=dev), rope_cols=128, head_dim=64, bias=b))]
    for name, kw in cases:
        outs = []
        for split in (1, 0):
            with L2.debug_switch("gemm_split", split):
                stats, out = kw.get("row_stats"), None
                if stats is not None:
                    stats.fill_(-7.0)
                if name == "residual":
                    kw = dict(residual=r.clone())
                    out = kw["residual"]
                y = ops.gemm(a, w, out=out, **kw)
                assert L2.debug_get("gemm_last_body") == (5 if split else 4), (name, split)
                outs.append((y.clone(), None if stats is None else stats.clone()))
        assert torch.equal(outs[0][0], outs[1][0]), name
        assert outs[0][1] is None or torch.equal(outs[0][1], outs[1][1]), name


@pytest.mark.parametrize("M,N,K,tile", [(300, 4352, 1152, 6), (400, 3456, 1152, 6), (560, 3072, 768, 6), (300, 4096, 1024, 8), (700, 2048, 2048, 8), (384, 4096, 1024, 6)])
def test_choice_between_tiles_of_64_columns(dev, M, N, K, tile):
    """gemm.hip: 128x64 with one slab a slot is not taken where it has a CU to itself (two slabs are 4 to 10 % faster there), 96x64 on every CU only where
    its last row tile is far from full"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M)
    a, w = (torch.randn(n, K, generator=g, device=dev).bfloat16() for n in (M, N))
    y = ops.gemm(a, w)
    assert L2.debug_get("gemm_last_tile") == tile
    with L2.debug_switch("gemm_mid", 2):
        assert torch.equal(y, ops.gemm(a, w))


@pytest.mark.parametrize("M,N,K,split", [(4707, 3584, 18944, True), (6117, 8256, 8256, True), (1514, 21888, 9728, False), (2242, 21824, 9472, False)])
def test_rows_left_over_large_weights(dev, M, N, K, split):
    """gemm.hip, REST_AGAIN and REST_ROWS: weights that half the last-level cache does not hold are read again for left-over rows only of products
    whose rows do not stay there either; up to four rounds nothing else splits them. The bits of one launch"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M)
    a, w = (torch.randn(n, K, generator=g, device=dev).bfloat16() for n in (M, N))
    outs = []
    for on in (1, 0):
        with L2.debug_switch("gemm_split", on):
            outs.append(ops.gemm(a, w))
            assert L2.debug_get("gemm_last_body") == (5 if split and on else 4)
    assert torch.equal(*outs)


@pytest.mark.parametrize("t,h,w,merge,max_tokens,offset", [
    (1, 28, 28, 2, 16384, 0),        # one window, enlarged: the smallest
    (1, 45, 61, 1, 16384, 1),        # odd source sizes, frames that start off a word
    (2, 120, 214, 2, 16384, 2),      # a last tile of fewer than six patches
    (3, 333, 517, 2, 300, 3),        # shrunk by less than 2 (9 taps) and the clip's last bytes read one by one
    (2, 480, 854, 2, 120, 0),        # shrunk by about 3 (16 taps)
    (1, 700, 640, 2, 40, 1),         # by about 4 (24 taps)
    (1, 1024, 1500, 2, 16, 0),       # by about 10: the two-pass kernels
])
def test_fused_resize_equals_the_host_path(dev, t, h, w, merge, max_tokens, offset):
    """csrc/preprocess.hip: the one-kernel resize and patchify, and the two-pass kernels behind it, give the bytes of the host
    path (Pillow's arithmetic) through the value table: fp32 equal, bf16 that rounded once"""
    from cogstream_amd import processing as pr
    from cogstream_amd.preprocess_gpu import preprocess_videos_gpu
    rng = np.random.default_rng(h)
    frames = rng.integers(0, 256, (t, h, w, 3), dtype=np.uint8)
    ref = pr.preprocess_videos([frames], merge_size=merge, max_tokens=max_tokens)
    room = torch.empty(frames.size + offset, dtype=torch.uint8, device=dev)
    room[offset:].copy_(torch.from_numpy(frames).reshape(-1))
    clip = room[offset:].view(t, h, w, 3)
    for dtype in (torch.float32, torch.bfloat16):
        got = preprocess_videos_gpu([clip], merge_size=merge, max_tokens=max_tokens, out_dtype=dtype)
        assert got["grid_sizes"].tolist() == ref["grid_sizes"].tolist()
        assert torch.equal(got["pixel_values"].cpu(), torch.from_numpy(ref["pixel_values"]).to(dtype))


@pytest.mark.parametrize("t,h,w,merge,max_tokens,offset,want", [
    (3, 70, 32, 1, 16384, 1, 223),       # a row of exactly two steps of source bytes: the clip's last row is read byte by byte
    (2, 57, 33, 1, 16384, 3, 223),       # one pixel behind them
    (2, 64, 34, 1, 16384, 2, 223),       # two: whole words to the end
    (3, 200, 300, 1, 90, 0, 2),          # shrunk by 3.6: more than three steps, the vector form
    (70, 90, 120, 2, 2000, 1, 223),      # frames in groups of several, the last one shorter
    (1, 260, 90, 1, 40, 2, 313),         # shrunk by 2.1 across, by 1.9 down: three steps, bands of one patch
    (2, 180, 320, 1, 228, 3, 224),       # by 1.6: a band's rows are four tiles
    (2, 75, 90, 1, 16384, 3, 213),       # an odd number of patch rows: bands of one patch
    (1, 44, 1000, 1, 88, 1, 214),        # one patch row from 44 source rows, by 1.6 across: four tiles of one patch's rows
    (1, 48, 700, 1, 43, 2, 314),         # the same from 48, by 2 across: three steps
])
def test_resize_as_matrix_products_equals_the_host_path(dev, t, h, w, merge, max_tokens, offset, want):
    """the sizes at which the matrix form's loads, steps, bands, row tiles and groups of frames change, every instance of the kernel: the
    bytes of the host path"""
    from cogstream_amd import _lib as L2
    test_fused_resize_equals_the_host_path(dev, t, h, w, merge, max_tokens, offset)
    assert L2.debug_get("preprocess_last_kernel") == want


@pytest.mark.parametrize("t,h,w,merge,max_tokens,want", [
    (1, 602, 798, 1, 16384, 2),          # a large image by itself: more waves than the chip holds, a prologue each
    (1, 728, 1288, 2, 16384, 2),         # bands of two patches
    (1, 480, 640, 1, 16384, 223),        # as many waves as it holds
    (3, 336, 518, 1, 16384, 223),        # several frames a wave
    (4, 728, 1288, 2, 16384, 223),
])
def test_resize_of_large_images_takes_the_faster_form(dev, t, h, w, merge, max_tokens, want):
    """matrix products or vector instructions, the bytes of the host path either way"""
    from cogstream_amd import _lib as L2
    test_fused_resize_equals_the_host_path(dev, t, h, w, merge, max_tokens, 1)
    assert L2.debug_get("preprocess_last_kernel") == want


def test_tap_tables_outlive_their_place_in_the_cache(dev):
    """a resize queued on a side stream, and tables that leave the cache before it runs: their memory, asked for again on the stream that
    made them, is not theirs until the resize is done. (Zeros in it would be tables of no taps: a black clip, no read out of place)"""
    from cogstream_amd import preprocess_gpu as pg
    frames = torch.randint(1, 256, (1, 300, 400, 3), device=dev, dtype=torch.uint8)
    want = pg.preprocess_videos_gpu([frames])["pixel_values"].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)
        got = pg.preprocess_videos_gpu([frames])["pixel_values"]
    tables = [(t.data_ptr(), t.numel() * 4) for key in ((400, 392), (300, 308)) for t in pg._tables(*key, 0)[:2]] + [(pg._value_table(0)[0].data_ptr(), 3072)]
    pg._tables.cache_clear()
    pg._value_table.cache_clear()
    reused = [torch.zeros(1 << 14, device=dev, dtype=torch.int32) for _ in range(64)]      # more than the small blocks' segments hold
    assert not side.query(), "the resize must still be queued here"
    for x in reused:
        assert not any(p < x.data_ptr() + x.numel() * 4 and x.data_ptr() < p + n for p, n in tables)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_preprocessing_is_not_captured(dev):
    """also when the size's tables are there already: they are the cache's, not the graph's"""
    from cogstream_amd import _lib as L2
    from cogstream_amd.preprocess_gpu import preprocess_videos_gpu
    frames = torch.randint(0, 256, (1, 56, 84, 3), device=dev, dtype=torch.uint8)
    want = preprocess_videos_gpu([frames])["pixel_values"].clone()
    with pytest.raises(L2.CogsError), torch.cuda.graph(torch.cuda.CUDAGraph()):
        preprocess_videos_gpu([frames])
    assert torch.equal(preprocess_videos_gpu([frames])["pixel_values"], want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,PD,K", [(2, 8, 2), (5, 520, 4), (257, 1000, 9), (300, 4096, 12), (3, 6_300_000, 3), (130, 179_200, 4), (24, 179_200, 4),
                                    (256, 65_536, 3), (257, 65_536, 3), (160, 65_544, 3), (161, 65_536, 3)])
def test_whole_seeding_equals_the_steps(dev, T, PD, K, dtype):
    """cogs_kmeans_pp draws the rows that distances of cogs_kmeans_pp_step and the same exponentials give on the host, by passes with a row per workgroup (form 1) and
    by slices (form 3): one slice and fewer, a ragged last slice, more rows than a workgroup's threads draw from at once; rows that all coincide raise the flag"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(T)
    x = torch.randn(T, PD, generator=g, device=dev).to(dtype)
    q = torch.empty(K - 1, T).exponential_(1)
    first = T // 2
    ws = ops.kmeans_workspace(T, PD, K, x.device)
    idx, flag = ops.kmeans_pp(x, first, K, q.to(dev), ws)
    kb = PD * x.element_size() >> 10
    if T > 400 or kb > 1024 or (T < 100 and kb > 256) or (T > 256 and kb > 100):     # few long rows, more rows than CUs: the slower form of 0.5 to 0.9
        assert L2.debug_get("km_pp_last_launches") == 3
    elif T <= 160 and kb <= 128:
        assert L2.debug_get("km_pp_last_launches") == 1
    want, near = [first], torch.empty(T, device=dev)
    probs = torch.empty(T).pin_memory()
    for m in range(K - 1):
        ops.kmeans_pp_step(x, want[-1], m == 0, near, probs, ws)
        p = probs.sqrt() ** 2
        want.append(int((p / p.double().sum().float() / q[m]).argmax()))
    assert idx.tolist() == want and int(flag) == 0
    same = x[:1].expand(T, PD).contiguous()
    _, flag = ops.kmeans_pp(same, first, K, q.to(dev), ws)
    assert int(flag) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,kb,bf16,fp32", [(300, 100, 1, 1), (301, 100, 3, 3), (256, 101, 1, 1), (257, 101, 3, 3), (99, 128, 1, 1), (99, 129, 3, 3), (100, 129, 1, 1), (100, 224, 1, 1),
                                            (100, 225, 3, 3), (192, 224, 1, 1), (192, 225, 3, 3), (193, 225, 1, 1), (193, 352, 1, 1), (193, 353, 1, 3), (223, 400, 1, 3),
                                            (223, 401, 3, 3), (224, 401, 1, 1), (224, 416, 1, 1), (224, 417, 1, 3), (256, 512, 1, 3), (256, 513, 3, 3), (257, 512, 3, 3)])
def test_forms_of_the_seeding_on_both_sides_of_their_lines(dev, T, kb, bf16, fp32, dtype):
    """the form that rows and bytes a row choose, and the rows and distances it draws by: those of the other form, and of a step per centre"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    K, PD, form = 4, kb * 1024 // dtype.itemsize, bf16 if dtype == torch.bfloat16 else fp32
    g = torch.Generator(device=dev).manual_seed(T + kb)
    x = (torch.randn(5, PD, generator=g, device=dev)[torch.arange(T, device=dev) * 5 // T] + 0.2 * torch.randn(T, PD, generator=g, device=dev)).to(dtype)
    q = torch.empty(K - 1, T).exponential_(1, generator=torch.Generator().manual_seed(T))
    ws = ops.kmeans_workspace(T, PD, K, x.device)
    got = []
    for forced in (0, 1, 3):
        d2 = torch.full((T, K), -1.0, device=dev)
        with L2.debug_switch("km_pp_form", forced):
            idx, flag = ops.kmeans_pp(x, T // 2, K, q.to(dev), ws, d2)
        assert L2.debug_get("km_pp_last_launches") == (form if forced == 0 else 3 if T > 300 else forced)
        got.append((idx.tolist(), int(flag), d2))
    near, probs, want = torch.empty(T, device=dev), torch.empty(T).pin_memory(), [T // 2]
    for m in range(K - 1):
        ops.kmeans_pp_step(x, want[-1], m == 0, near, probs, ws)
        p = probs.sqrt() ** 2
        want.append(int((p / p.double().sum().float() / q[m]).argmax()))
    for rows, zero, d2 in got:
        assert rows == want and zero == 0 and torch.equal(d2, got[0][2])


@pytest.mark.parametrize("form", [1, 3])
@pytest.mark.parametrize("T,PD,K,scenes", [(5, 8, 2, 2), (9, 520, 3, 3), (40, 1032, 39, 4), (255, 2048, 18, 21), (300, 512, 60, 1), (700, 1032, 30, 11)])
def test_seeding_draws_several_centres_a_pass(dev, T, PD, K, scenes, form):
    """a pass measures rows that the next draws are likely to fall on and draws while they do: the rows and distances of a pass per centre, where
    guesses come true (rows of scenes), where most do not (more centres than scenes), for the last centres (fewer guesses), for more rows than
    a workgroup keeps in LDS, and with a workspace of one centre"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(T + K)
    x = (torch.randn(scenes, PD, generator=g, device=dev)[torch.arange(T, device=dev) * scenes // T] + 0.2 * torch.randn(T, PD, generator=g, device=dev)).bfloat16()
    q = torch.empty(K - 1, T).exponential_(1, generator=torch.Generator().manual_seed(K))
    ws = ops.kmeans_workspace(T, PD, K, x.device)
    want, near, cols = [T // 3], torch.empty(T, device=dev), []
    probs = torch.empty(T).pin_memory()
    for m in range(K - 1):
        ops.kmeans_pp_step(x, want[-1], m == 0, near, probs, ws)
        one = torch.empty(T, device=dev)
        ops.kmeans_pp_step(x, want[-1], True, one, None, ws)
        cols.append(one)
        p = probs.sqrt() ** 2
        want.append(int((p / p.double().sum().float() / q[m]).argmax()))
    for space in (ws, ops.kmeans_workspace(T, PD, 1, x.device)):
        d2 = torch.full((T, K), -1.0, device=dev)
        with L2.debug_switch("km_pp_form", form):
            idx, flag = ops.kmeans_pp(x, T // 3, K, q.to(dev), space, d2)
        assert idx.tolist() == want and int(flag) == 0
        assert torch.equal(d2[:, :K - 1], torch.stack(cols, 1)) and bool((d2[:, K - 1] == -1).all())


@pytest.mark.parametrize("M,N,K,form", [
    (4609, 3456, 1152, "rotary, head-major, folded norm"), (3841, 4352, 1152, "folded norm, gelu"), (13825, 1152, 1152, "residual, statistics"),
    (13825, 1152, 4352, "residual, statistics"), (3585, 4608, 3584, "rotary"), (4609, 3584, 3584, "residual"), (2049, 8192, 2048, "plain"),
    (1281, 11264, 2048, "swiglu"), (2049, 8192, 2048, "fp32")])
def test_a_split_product_whose_remainder_is_one_row(dev, M, N, K, form):
    """a product cut into whole rounds of 256x256 tiles and one more row: that row gets its fused epilogue and the bits of the unsplit
    launch, like every other"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(M)
    rnd = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.5).bfloat16()
    a, w = rnd(M, K), rnd(N, K)
    table = lambda: torch.randn(M, 36, 2, generator=g, device=dev)
    fold = lambda: dict(ln_ab=torch.rand(M, 2, generator=g, device=dev) + 0.5, col_c=torch.randn(N, generator=g, device=dev))
    kw = {"rotary, head-major, folded norm": lambda: dict(rope_cos=table(), rope_cols=2304, head_dim=72, hm_cols=1152, **fold()),
          "folded norm, gelu": lambda: dict(act=L2.ACT_GELU_TANH, **fold()),
          "residual, statistics": lambda: dict(bias=rnd(N), residual=rnd(M, N), row_stats=torch.empty(M, N // 64, 2, device=dev)),
          "rotary": lambda: dict(bias=rnd(N), rope_cos=torch.randn(M, 64, 2, generator=g, device=dev), rope_cols=4096, head_dim=128),
          "residual": lambda: dict(residual=rnd(M, N)), "plain": dict, "swiglu": lambda: dict(act=L2.ACT_SWIGLU),
          "fp32": lambda: dict(out_f32=True)}[form]()
    outs = []
    for split, body in ((1, 5), (0, 4)):
        stats = kw.get("row_stats")
        if stats is not None:
            stats.fill_(-7.0)
        with L2.debug_switch("gemm_split", split):
            out = ops.gemm(a, w, **kw)
        assert L2.debug_get("gemm_last_body") == body
        outs.append((out, None if stats is None else stats.clone()))
    (x, sx), (y, sy) = outs
    assert torch.equal(x, y) and (sx is None or torch.equal(sx, sy))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,K,PD,kind", [(40, 5, 520, "plain"), (150, 33, 1032, "plain"), (200, 70, 512, "plain"), (64, 6, 1024, "empty"),
                                         (48, 4, 1024, "infinite"), (3, 2, 8, "plain"), (60, 7, 1032, "far"), (150, 33, 520, "far"), (90, 12, 1024, "dry")])
def test_centres_that_stay_keep_their_distances_and_means(dev, T, K, PD, kind, dtype):
    """csrc/kmeans.hip: the Lloyd loop sums distances and means only for centres whose rows have changed, and not those the seeding
    has summed. Every iteration bit for bit against the same steps called one by one, which sum everything: more centres than one distance
    launch holds, or than a wave, with clusters that run empty (duplicated centres; every other centre too late for any row, from the seeding's
    distances; both reseeded), a pool that runs dry in a call that starts from those and is called again, and a row of infinities"""
    ops = _ops()
    g = torch.Generator(device=dev).manual_seed(T + K)
    x = (torch.randn(max(2, K // 2), PD, generator=g, device=dev).repeat(T, 1)[:T] + 0.3 * torch.randn(T, PD, generator=g, device=dev)).to(dtype)
    if kind == "infinite":
        x[5, 3] = float("inf")
    ts = torch.arange(T, device=dev, dtype=torch.float32)
    ws = ops.kmeans_workspace(T, PD, K, dev)
    q = torch.rand(K - 1, T, generator=g, device=dev) + 0.01
    d2 = torch.full((T, K), -1.0, device=dev)
    rows, flag = ops.kmeans_pp(x, 2, K, q, ws, d2)
    known = K - 1 if kind in ("plain", "far", "dry") and int(flag) == 0 else 0
    assert known or kind in ("empty", "infinite")
    rows = rows.long()
    if kind == "empty":
        rows = torch.full((K,), 7, device=dev)
        rows[0] = 11
    pool = [int(v) for v in torch.randint(0, T, (400,), generator=torch.Generator().manual_seed(1))]
    c0, t0 = x[rows].float().contiguous(), ts[rows].contiguous()
    if kind in ("far", "dry"):
        t0[1::2] = 10.0 * T
    if known:                                  # the seeding's sums are those of the distance pass (fp64 over slices: the last place at most)
        whole = ops.kmeans_sqdist(x, c0, None, K, ws)
        assert bool(((d2[:, :known] - whole[:, :known]).abs() <= whole[:, :known] * 2.0 ** -23).all())
    for iters in (1, 2, 3, 5, 9):
        c, ct, used, done = c0.clone(), t0.clone(), 0, 0
        for _ in range(iters):
            a, _ = ops.kmeans_assign(ops.kmeans_sqdist(x, c, None, K, ws), ts, ct, 2.0)
            empty = torch.bincount(a, minlength=K) == 0
            reseed = torch.zeros(K, dtype=torch.int32, device=dev)
            n = int(empty.sum())
            reseed[empty] = torch.tensor(pool[used:used + n], dtype=torch.int32, device=dev)
            used, done = used + n, done + 1
            if float(ops.kmeans_update(x, ts, a, reseed, c, ct, ws)) <= 1e-4:
                break
        gc, gt, ga = c0.clone(), t0.clone(), torch.empty(T, dtype=torch.int64, device=dev)
        mine, left = d2.clone() if known else None, known
        if kind == "dry":
            assert ops.kmeans_lloyd(x, ts, gc, gt, ga, 2.0, iters, 1e-4, pool[:K // 2 - 1], ws, mine, left) == (0, 0, True)
            left = 0
        got = ops.kmeans_lloyd(x, ts, gc, gt, ga, 2.0, iters, 1e-4, pool, ws, mine, left)
        assert got == (done, used, False), (iters, got, done, used)
        assert used >= K // 2 or kind not in ("far", "dry")
        assert torch.equal(ga, a) and torch.equal(gt, ct) and torch.equal(gc.view(torch.int32), c.view(torch.int32)), iters


def test_token_ids_reach_the_device_as_they_were_at_the_call(dev):
    """ops.token_ids: host ids behind work that is still running, their tensor rewritten as soon as the call returns; pinned ids, other types and shapes,
    none at all; and a capture, which cannot hold a copy from the caller's memory, still refuses"""
    ops = _ops()
    d = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator().manual_seed(3)
    for n in (0, 1, 7, 4096):
        for make in (lambda t: t, lambda t: t.int(), lambda t: t.pin_memory() if n else t, lambda t: t.reshape(1, -1), lambda t: t.to(dev)):
            want = torch.randint(0, 1000, (n,), generator=g)
            ids = make(want.clone())
            torch.cuda._sleep(2_000_000)
            got = ops.token_ids(ids, d)
            if not ids.is_cuda:
                ids.fill_(-1)
            assert got.is_cuda and got.dtype == torch.int64 and torch.equal(got.cpu(), want)
    with pytest.raises(RuntimeError), torch.cuda.graph(torch.cuda.CUDAGraph()):
        ops.token_ids(torch.arange(8), d)
    torch.cuda.synchronize()
    assert ops.token_ids(torch.arange(8), d).tolist() == list(range(8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 127, 128, 129])
def test_rows_of_few_tokens(dev, n, dtype):
    """ops.embed_rows: up to 128 host ids as the launch's arguments, read before the call returns; more, pinned ones and those on the device as before;
    a capture still refuses ids of the host"""
    ops = _ops()
    g = torch.Generator().manual_seed(n)
    table = torch.randn(1000, 264, generator=g).to(dtype).to(dev)
    for make in (lambda t: t, lambda t: t.int().reshape(1, -1), lambda t: t.repeat_interleave(2)[::2], lambda t: t.pin_memory() if n else t, lambda t: t.to(dev)):
        want = torch.randint(0, 1000, (n,), generator=g)
        want[-1:] = 999
        ids = make(want.clone())
        torch.cuda._sleep(1_000_000)
        got = ops.embed_rows(table, ids)
        if not ids.is_cuda:
            ids.fill_(1)
        assert torch.equal(got, table[want.to(dev)])
    if n:
        with pytest.raises(RuntimeError), torch.cuda.graph(torch.cuda.CUDAGraph()):
            ops.embed_rows(table, want)
        torch.cuda.synchronize()


@pytest.mark.parametrize("grid", [(1, 2, 2), (1, 12, 11), (1, 16, 16), (1, 16, 24), (2, 12, 23), (1, 24, 24), (1, 1, 577), (3, 14, 16)])
def test_weights_read_ahead_change_nothing(dev, grid):
    """the encoder's launches of up to 576 patches read the next products' weights on idle CUs: first and last layer, fewer columns than tiles, and sizes on both
    sides of the line, bit for bit against launches that read none (as beside another stream)"""
    from cogstream_amd import _lib as L2
    from cogstream_amd.vision import VisionEncoder
    from cogstream_amd.weights import VisionConfig, random_vit_state
    cfg = VisionConfig(num_hidden_layers=3)
    enc = VisionEncoder(random_vit_state(cfg, seed=1, device=dev, dtype=torch.bfloat16), cfg)
    n = grid[0] * grid[1] * grid[2]
    pix = (torch.rand(n, cfg.patch_dim, generator=torch.Generator(device=dev).manual_seed(n), device=dev) * 2 - 1).bfloat16()
    run = lambda: enc(pix, torch.tensor([grid]), torch.tensor([1]))
    got = run()
    with L2.debug_switch("gemm_co_streams", 2):
        want = run()
    assert torch.isfinite(got.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("grid,heads,mode", [((1, 12, 12), 16, {}), ((1, 16, 16), 16, {}), ((1, 16, 24), 16, {}), ((16, 6, 6), 16, {}), ((9, 8, 8), 16, {}), ((2, 4, 4), 8, {}), ((1, 16, 16), 9, {}), ((1, 24, 24), 16, {}),
                                             ((1, 16, 16), 16, {"attn_vit": 1}), ((1, 16, 16), 16, {"attn_vit": 0}), ((1, 16, 16), 16, {"gemm_mid": 3})])
def test_read_ahead_is_counted_on_only_where_it_was(dev, grid, heads, mode):
    """a product leaves out its own read-ahead of weights only where a launch in front has really read them: not behind an attention of many short frames, of heads whose number or size
    its kernel has no such workgroups for, or of another kernel, nor where few workgroups would have too many bytes each. Never more products than were read ahead; of one image with
    16 heads of 72 all four of a layer, of one of 16 x 24 patches (40 CUs beside the output product) the attention's alone"""
    import contextlib
    from cogstream_amd import _lib as L2
    from cogstream_amd.vision import VisionEncoder
    from cogstream_amd.weights import VisionConfig, random_vit_state
    layers = 3
    cfg = VisionConfig(num_hidden_layers=layers, num_attention_heads=heads)
    enc = VisionEncoder(random_vit_state(cfg, seed=1, device=dev, dtype=torch.bfloat16), cfg)
    n = grid[0] * grid[1] * grid[2]
    pix = (torch.rand(n, cfg.patch_dim, generator=torch.Generator(device=dev).manual_seed(n), device=dev) * 2 - 1).bfloat16()
    with contextlib.ExitStack() as switches:
        for name, value in mode.items():
            switches.enter_context(L2.debug_switch(name, value))
        before = [L2.debug_get(k) for k in ("weights_ahead_read", "weights_ahead_counted_on")]
        out = enc(pix, torch.tensor([grid]), torch.tensor([1]))
        read, counted = (L2.debug_get(k) - b for k, b in zip(("weights_ahead_read", "weights_ahead_counted_on"), before))
    assert torch.isfinite(out.float()).all()
    assert counted <= read
    if heads == 16 and not mode:          # (the first layer's first weights are its own product's to read, and that one reads none ahead)
        want = {(1, 12, 12): 4 * layers - 2, (1, 16, 16): 4 * layers - 2, (1, 16, 24): layers}
        assert grid not in want or counted == read == want[grid]


@pytest.mark.parametrize("K", [2, 130])
@pytest.mark.parametrize("T", [16127, 16128, 16129, 16251, 16381, 16384])
def test_means_of_as_many_rows_as_the_loop_takes(dev, T, K):
    """up to the documented limits (T + K + 1 <= 16 384 in the loop, no more than 16 384 staged time stamps in a step), where the last kernel of an update has 64 KiB of LDS and
    more: centres of whole numbers, so that every sum is exact"""
    from cogstream_amd import _lib as L2
    ops = _ops()
    a = torch.arange(T, device=dev) * 7 % K
    x = (a[:, None] * 64 + torch.arange(8, device=dev)).float()
    ts = (torch.arange(T, device=dev) % 13).float()
    sums = torch.zeros(K, dtype=torch.float64, device=dev).index_add_(0, a, ts.double())
    mean = sums.float() / torch.bincount(a, minlength=K).float()
    start = lambda: (x[:K].clone().index_copy_(0, a[:K], x[:K]) + 1, torch.full((K,), 6.0, device=dev))
    ws = ops.kmeans_workspace(T, 8, K, x.device)
    c, ct = start()
    ops.kmeans_update(x, ts, a, torch.zeros(K, dtype=torch.int32, device=dev), c, ct, ws)
    assert torch.equal(ct, mean) and torch.equal(c, torch.arange(K, device=dev)[:, None] * 64 + torch.arange(8, device=dev).float())
    c, ct = start()
    got = torch.empty(T, dtype=torch.int64, device=dev)
    if T + K + 1 > 16384:
        with pytest.raises(L2.CogsError):
            ops.kmeans_lloyd(x, ts, c, ct, got, 0.0, 4, 1e-4, [], ws)
        return
    assert ops.kmeans_lloyd(x, ts, c, ct, got, 0.0, 4, 1e-4, [], ws) == (2, 0, False)
    assert torch.equal(got, a) and torch.equal(ct, mean) and torch.equal(c, torch.arange(K, device=dev)[:, None] * 64 + torch.arange(8, device=dev).float())


@pytest.mark.parametrize("K,passes", [(2, 1), (5, 1), (6, 2), (18, 5)])
def test_passes_of_a_seeding_are_not_overstated(dev, K, passes):
    """last_stats counts the passes a seeding in one call takes at least (up to four centres each), and every one of a seeding step by step"""
    from cogstream_amd import kmeans
    x = torch.randn(40, 1, 64, generator=torch.Generator(device=dev).manual_seed(K), device=dev)
    kmeans.kmeans_with_time_min_max(x, torch.arange(40.0), K)
    assert kmeans.last_stats["kpp_path"] == "one call" and kmeans.last_stats["kpp_passes"] == passes
    kmeans.kmeans_with_time_min_max(x[:1].expand(40, 1, 64).contiguous(), torch.arange(40.0), K)
    assert kmeans.last_stats["kpp_path"].startswith("step by step") and kmeans.last_stats["kpp_passes"] == K - 1
