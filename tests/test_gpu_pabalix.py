"""Pabalix on the GPU against its oracle (oracle/pabalix.py): every mechanism, prompts against token-by-token decoding, prompts
in portions, unequal batches, caches that grow, are freed and used again, keys at every place of interest, first tokens, long
decoding, other sizes, and generation through the framework's entry points. float32 pins the arithmetic, bfloat16 the kernels."""
import json
import os
import subprocess
import sys

import pytest
import torch

from oracle import pabalix as po
from pabalix_models import A, B, CONFIGS, G, YARN, config, double, mixer, rms_err, state, tokens

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# largest row error of the logits. bfloat16: about twice what rounding the operands of the matrix products does to these models
TOL = {torch.float32: 2e-5, torch.bfloat16: 3e-2}
TINY = 2.5        # the eight-wide model has nothing to average rounding errors over
DTYPES = [torch.float32, torch.bfloat16]
_cache = {}


def engine(cfg, st, dtype):
    from cogstream_amd.llm import DecoderEngine
    from cogstream_amd.pabalix import parse_config
    return DecoderEngine(st, parse_config(cfg), dtype=dtype, device="cuda:0")


def named(name, dtype, dev, n=0):
    """(config, weights, engine, tokens, oracle logits, oracle streams) of a shared model, made once"""
    key = (name, dtype)
    if key not in _cache:
        cfg = CONFIGS[name]
        st = state(cfg)
        _cache[key] = (cfg, st, engine(cfg, st, dtype))
    cfg, st, e = _cache[key]
    if (name, n) not in _cache:
        t = tokens(cfg, n)
        _cache[(name, n)] = (t,) + po.forward(cfg, double(st), t)
    return (cfg, st, e) + _cache[(name, n)]


def sequences(e, reserve=64):
    from cogstream_amd.llm import Sequences
    return Sequences(e, reserve)


def run(e, toks, cuts=(), reserve=64):
    """logits of every token, the prompt cut at `cuts`"""
    s = sequences(e, reserve)
    edges = [0, *cuts, len(toks)]
    return torch.cat([s.step([("r", toks[a:b], list(range(b - a)))]) for a, b in zip(edges, edges[1:])])


# ------------------------------------------------------------------------------------------------ mechanisms
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_prompt_against_the_oracle_layer_by_layer(dev, name, dtype):
    """logits and the residual stream behind every layer, all sizes (also ranks and heads above the MFMA kernels' instances)"""
    n = 70 if name in ("wide", "large_rank") else 150
    cfg, st, e, toks, lg, streams = named(name, dtype, dev, n)
    W, tol = cfg["width"], TOL[dtype] * (TINY if name == "one" else 1)
    buf = torch.empty(len(cfg["layers"]), n, e.packed.width_p, device=dev)
    got = e.forward_batch(e.embed_tokens(torch.tensor(toks)), [n], [e.new_cache(n)], list(range(n)), streams=buf)
    assert got.shape == (n, cfg["vocab"])
    for i, want in enumerate(streams):
        assert rms_err(buf[i, :, :W], want) < tol, (name, i)
        assert not buf[i, :, W:].any()
    assert rms_err(got, lg) < tol


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_decoding_against_the_oracle(dev, name, dtype):
    """the absorbed form, from the first token on"""
    n = 70 if name in ("wide", "large_rank") else 150
    cfg, st, e, toks, lg, _ = named(name, dtype, dev, n)
    got = run(e, toks, range(1, n))
    assert rms_err(got, lg) < TOL[dtype] * (TINY if name == "one" else 1)


@pytest.mark.parametrize("kind", [A, B, G])
@pytest.mark.parametrize("dtype", DTYPES)
def test_rotation_far_from_the_start(dev, kind, dtype):
    """one layer, peaked scores, positions in the thousands: prompt and decoded"""
    n = 2100
    cfg = config([dict(mixer(kind, heads=2, dim=8, rot=32, vdim=16, gain=2.0, base=30.0, scaling=None if kind == B else YARN), ff=None)], width=64, vocab=64)
    st = state(cfg, seed=5)
    toks, w = tokens(cfg, n), double(state(cfg, seed=5))
    lg = po.forward(cfg, w, toks)[0]
    e = engine(cfg, st, dtype)
    assert rms_err(run(e, toks), lg) < TOL[dtype]
    assert rms_err(run(e, toks, range(n - 40, n))[-40:], lg[-40:]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
def test_sink_and_gate_at_their_extremes(dev, dtype):
    """a sink far above every score, one far below, and saturated gates, for prompts and decoding"""
    cfg = config([mixer(G, heads=4, scaling=YARN)])
    st = state(cfg, seed=2)
    st["l0.mix.sink"] = torch.tensor([40.0, -40.0, 3.0, 0.0])
    st["l0.mix.g"] = st["l0.mix.g"] * torch.tensor([8.0, -8.0, 0.0, 1.0])[:, None]
    toks = tokens(cfg, 60)
    lg = po.forward(cfg, double(st), toks)[0]
    e = engine(cfg, st, dtype)
    assert rms_err(run(e, toks), lg) < TOL[dtype] and rms_err(run(e, toks, range(1, 60)), lg) < TOL[dtype]


# ------------------------------------------------------------------------------------------------ one key among many
def needle_model(kind, dtype_seed=7):
    """token 1 asks for token 2: one score is far above all others, so whether exactly that key is seen shows in the logits"""
    cfg = config([dict(mixer(kind, heads=2, dim=16, rot=4, vdim=32, q_rank=64, kv_rank=64, scale=1.0, base=1e6, scaling=None if kind == B else (1.0, 64, 32.0, 1.0)), ff=None)],
                 width=64, vocab=64)
    st = state(cfg, seed=dtype_seed)
    if kind == G:
        st["l0.mix.sink"] = torch.tensor([0.5, 1.0])
    w, eps = double(st), cfg["norm"]["eps"]
    h = po.rms(w["embed"], w["l0.norm1"], eps)
    cq = po.rms(h @ w["l0.mix.dq"].T, w["l0.mix.dq.norm"], eps)[1]
    c = po.rms((h @ w["l0.mix.dkv"].T)[:, :64], w["l0.mix.dkv.norm"], eps)[2]
    for hd in range(2):
        st["l0.mix.uq"][hd * 20] = (5 * cq / (cq @ cq)).float()
        st["l0.mix.uk"][hd * 16] = (5 * c / (c @ c)).float()
    st = {k: v.to(torch.bfloat16).float() for k, v in st.items()}
    return cfg, st


@pytest.mark.parametrize("kind", [A, B, G])
@pytest.mark.parametrize("dtype", DTYPES)
def test_a_single_key_at_every_place_of_interest(dev, kind, dtype):
    """the asked-for key first, last, at tile and split borders, itself, and one past the query (which must not be seen)"""
    cfg, st = needle_model(kind)
    e, w = engine(cfg, st, dtype), double(st)
    n = 330
    base = [t if t > 2 else 3 + t for t in tokens(cfg, n)]
    ask = n - 1
    without = None
    for at in (None, 0, 1, 15, 16, 31, 32, 63, 64, 65, 127, 128, 255, 256, 319, 320, n - 2):
        toks = list(base)
        toks[ask] = 1
        if at is not None:
            toks[at] = 2
        lg = po.forward(cfg, w, toks)[0]
        if at is None:
            without = lg[ask]
        else:
            assert rms_err(lg[ask:], without[None]) > 0.3            # the oracle's answer depends on that key
        got = run(e, toks)
        assert rms_err(got[ask:], lg[ask:]) < TOL[dtype], ("prompt", at)
        assert rms_err(run(e, toks, [ask])[ask:], lg[ask:]) < TOL[dtype], ("decoded", at)
        assert rms_err(run(e, toks, [ask - 70])[ask:], lg[ask:]) < TOL[dtype], ("second portion", at)
    # the key right behind the query: invisible, also when it shares the query's tile
    for ask in (0, 15, 62, 63, 64, 126, 127, 128, 200):
        toks = list(base)
        toks[ask], toks[ask + 1] = 1, 2
        lg = po.forward(cfg, w, toks[:ask + 2])[0]
        assert rms_err(run(e, toks[:ask + 2]), lg) < TOL[dtype], ask


# ------------------------------------------------------------------------------------------------ schedules
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_portions_of_a_prompt(dev, name, dtype):
    cfg, st, e, toks, lg, _ = named(name, dtype, dev, 150)
    for cuts in ([2], [1, 3], [64], [63, 65], [128], [149], [148], [50, 52, 54, 118], list(range(2, 150, 2)), list(range(7, 150, 29))):
        assert rms_err(run(e, toks, cuts), lg) < TOL[dtype], cuts


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 63, 64, 65, 129])
@pytest.mark.parametrize("dtype", DTYPES)
def test_short_sequences_and_first_tokens(dev, n, dtype):
    cfg, st, e, toks, lg, _ = named("peaked", dtype, dev, 150)
    assert rms_err(run(e, toks[:n]), lg[:n]) < TOL[dtype]
    assert rms_err(run(e, toks[:n] + toks[n:n + 2], [n, n + 1]), lg[:n + 2]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_unequal_batch_against_each_alone(dev, name, dtype):
    """prompts of 1 .. 140 tokens in one step, then decoded together, shorter requests ending earlier; and steps that mix whole
    prompts with single tokens"""
    cfg, st, e, _, _, _ = named(name, dtype, dev, 150)
    w = double(st)
    lens = [1, 140, 2, 65, 64, 33, 17, 90]
    full = [tokens(cfg, n + 3 + i, seed=i) for i, n in enumerate(lens)]
    want = [po.forward(cfg, w, t)[0] for t in full]
    s = sequences(e, 16)
    out = s.step([(i, full[i][:n], list(range(n))) for i, n in enumerate(lens)])
    at = 0
    for i, n in enumerate(lens):
        assert rms_err(out[at:at + n], want[i][:n]) < TOL[dtype], i
        at += n
    pos = list(lens)
    while True:
        live = [i for i in range(len(lens)) if pos[i] < len(full[i])]
        if not live:
            break
        order = live[::-1] if len(live) % 2 else live          # the order in a batch is nothing a request sees
        out = s.step([(i, [full[i][pos[i]]], [0]) for i in order])
        for r, i in enumerate(order):
            assert rms_err(out[r:r + 1], want[i][pos[i]:pos[i] + 1]) < TOL[dtype], (i, pos[i])
            pos[i] += 1
        for i in live:
            if pos[i] == len(full[i]):
                s.release(i)
    assert not s.caches
    s = sequences(e)
    s.step([("a", full[1][:100], []), ("b", full[3][:1], [])])
    out = s.step([("b", full[3][1:2], [0]), ("c", full[7], [len(full[7]) - 1]), ("a", full[1][100:], [0, 40])])
    assert rms_err(out, torch.stack([want[3][1], want[7][-1], want[1][100], want[1][140]])) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
def test_large_batch_decoding(dev, dtype):
    """more sequences than one MFMA column tile, and more rows than the few-row GEMM takes"""
    cfg, st, e, toks, lg, _ = named("peaked", dtype, dev, 150)
    for count in (2, 16, 17, 40, 70):
        s = sequences(e)
        s.step([(i, toks[:1 + i], []) for i in range(count)])
        out = s.step([(i, [toks[1 + i]], [0]) for i in range(count)])
        assert rms_err(out, lg[1:1 + count]) < TOL[dtype], count


@pytest.mark.parametrize("dtype", DTYPES)
def test_memory_that_is_freed_and_used_again(dev, dtype):
    """caches and workspaces that hold another request's rows, or NaN, change nothing"""
    cfg, st, e, toks, lg, _ = named("mixed", dtype, dev, 150)
    s = sequences(e, 16)
    for r in range(6):
        n = [90, 20, 130, 60, 7, 150][r]
        size = sum(e.packed.cache_widths) * (-(-n // 16) * 16)
        poison = torch.full((size,), float("nan"), device=dev, dtype=dtype)
        del poison
        e.handle._ws["decoder"].view(torch.int16).fill_(0x7fc0)          # NaN in either type
        other = [t ^ 1 if (t ^ 1) < cfg["vocab"] else t for t in toks]
        s.step([("junk", other[:n], [])])
        s.release("junk")
        out = s.step([("x", toks[:n - 2], list(range(n - 2)))])
        assert rms_err(out, lg[:n - 2]) < TOL[dtype], r
        for k in (n - 2, n - 1):
            assert rms_err(s.step([("x", [toks[k]], [0])]), lg[k:k + 1]) < TOL[dtype], r
        s.release("x")


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding_through_a_growing_cache(dev, dtype):
    cfg, st, e, toks, lg, _ = named("peaked", dtype, dev, 400)
    got = run(e, toks, range(5, 400), reserve=8)
    assert rms_err(got, lg) < TOL[dtype]


def test_forms_and_kernels_agree(dev):
    """bfloat16: absorbed against expanded single tokens, MFMA against row-wise attention, few-row against general GEMM, and any
    number of key splits: all inside the tolerance of the oracle"""
    from cogstream_amd import _lib as L
    cfg, st, e, toks, lg, _ = named("peaked", torch.bfloat16, dev, 400)
    for name, value in (("mla_absorb", 0), ("mla_rowwise", 1), ("gemm_skinny", 0), ("mla_split_keys", 16), ("mla_split_keys", 100), ("mla_split_keys", 4096)):
        with L.debug_switch(name, value):
            assert rms_err(run(e, toks, [20, 380, *range(381, 400)]), lg) < TOL[torch.bfloat16], (name, value)


@pytest.mark.parametrize("heads,q_rank", [(3, 40), (3, 64), (5, 1000), (3, 1024), (80, 1100), (3, 2048), (160, 300), (3, 2100)])
@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17])
def test_query_products_that_norm_their_rows(dev, heads, q_rank, rows):
    """one token of up to 16 sequences: the query product forms its rows' norms itself (up to 2048 columns of query latent; 17 rows and 2100 columns take the
    launch in front), 16, 32 and 64 columns a workgroup, fewer slices of K than its waves have in flight and more; a layer with gates and one that borrows
    its rows and has none, so that no workgroup is left for rows. Logits and the rows that went into the caches against the oracle and the launch of their own"""
    from cogstream_amd import _lib as L
    cfg = config([dict(mixer(G, heads=heads, q_rank=q_rank, dim=24, rot=16, vdim=16), ff=None), dict(mixer(A, heads=3, q_rank=q_rank, dim=24, rot=16), ff=None),
                  dict(mixer(A, heads=3, q_rank=q_rank, dim=24, rot=16, kv_from=1), ff=None)], width=64, vocab=96)
    st = state(cfg)
    e = engine(cfg, st, torch.bfloat16)
    toks = [tokens(cfg, 4 + i % 3, seed=i) for i in range(rows)]
    s = sequences(e)
    s.step([(i, t[:-1], []) for i, t in enumerate(toks)])
    got = s.step([(i, t[-1:], [0]) for i, t in enumerate(toks)])
    want = torch.cat([po.forward(cfg, double(st), t)[0][-1:] for t in toks])
    assert rms_err(got, want) < TOL[torch.bfloat16]
    other = sequences(e)
    with L.debug_switch("gemm_skinny", 0):
        other.step([(i, t[:-1], []) for i, t in enumerate(toks)])
        other.step([(i, t[-1:], [0]) for i, t in enumerate(toks)])
    for i, t in enumerate(toks):
        for a, b in zip(s.caches[i]._blocks(), other.caches[i]._blocks()):
            a, b = a[..., :len(t), :].float(), b[..., :len(t), :].float()
            assert bool((a - b).abs().max() <= TOL[torch.bfloat16] * b.abs().max())


@pytest.mark.parametrize("heads,q_rank", [(3, 40), (5, 1000), (3, 1024), (80, 1100), (3, 2048), (3, 2100)])
def test_the_query_product_of_one_row_norms_it(dev, heads, q_rank):
    """... one sequence (the sizes of the test above)"""
    test_query_products_that_norm_their_rows(dev, heads, q_rank, 1)


@pytest.mark.parametrize("rows,q_rank", [(16, 768), (8, 2048), (16, 2048), (3, 1024)])
def test_query_norms_have_the_same_bits_by_either_kernel(dev, rows, q_rank):
    """the query latents' norms formed inside the query product and by the launch in front, bit for bit. Every product's rows of weights have one entry of 1 or -1 (those
    of the query latents a second one of 1/64, for values of more bits than a square in fp32 holds), so that no order of sums and no store of a partial one rounds: the norms
    are all that could differ. A norm whose last bit is off moves one of some 65 000 of its bf16 values, so it takes thousands of rows to show"""
    from cogstream_amd import _lib as L
    cfg = config([dict(mixer(A, heads=q_rank // 32, q_rank=q_rank, dim=24, rot=16, vdim=8), ff=None)] * 2, width=256, vocab=1024)
    st = state(cfg)
    g = torch.Generator().manual_seed(rows)
    for k, w in st.items():
        if w.dim() == 2 and k.rsplit(".", 1)[-1] not in ("embed", "uk", "uv"):
            st[k] = torch.zeros_like(w).scatter_(1, torch.randint(0, w.shape[1], (w.shape[0], 1), generator=g), torch.randint(0, 2, (w.shape[0], 1), generator=g) * 2.0 - 1)
            if k.endswith(".dq"):
                st[k] += torch.zeros_like(w).scatter_(1, torch.randint(0, w.shape[1], (w.shape[0], 1), generator=g), 2.0 ** -6)
    e = engine(cfg, st, torch.bfloat16)
    steps = 6000 // (2 * rows)
    toks = [tokens(cfg, 4 + steps, seed=i) for i in range(rows)]

    def logits():
        s = sequences(e, 1024)
        s.step([(i, t[:4], []) for i, t in enumerate(toks)])
        return torch.stack([s.step([(i, [t[4 + n]], [0]) for i, t in enumerate(toks)]) for n in range(steps)])
    got = logits()
    with L.debug_switch("gemm_skinny", 0):
        want = logits()
    assert torch.equal(got, want)


@pytest.mark.parametrize("dim,rot", [(128, 64), (96, 64), (64, 32), (32, 64)])
def test_columns_that_are_not_rotated(dev, dim, rot):
    """the query product reads no factors for blocks of columns in front of a head's rotated part (64 columns a wave, 32 in the small tiles; heads where such
    blocks cross into the rotated part or the next head): a prompt against the oracle, and the same bits with every tile size and with the ping-pong kernel"""
    from cogstream_amd import _lib as L
    cfg = config([mixer(B, heads=4, dim=dim, rot=rot, vdim=32, q_rank=128, kv_rank=64, gain=1.5), mixer(A, heads=4, dim=dim, rot=rot, vdim=32, q_rank=192, kv_rank=64, scaling=YARN)],
                 width=128, ff=128)
    st = state(cfg)
    e = engine(cfg, st, torch.bfloat16)
    toks = tokens(cfg, 300)
    whole = lambda: run(e, toks)
    first = whole()
    assert rms_err(first, po.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]
    for tile in range(1, 12):
        with L.debug_switch("gemm_mid", tile):
            assert torch.equal(whole(), first), tile
    with L.debug_switch("gemm_split", 0):                # (what the ping-pong kernel can take is all its)
        assert torch.equal(whole(), first)


@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17])
def test_few_rows_by_48_and_64_columns(dev, rows):
    """few-row products whose columns go 48 to a workgroup (10 240 to 12 288 of up to 16 rows: here the feed-forward's and the head's, the last group
    ragged in both; 17 rows take 64): every row's logits against the oracle"""
    cfg = config([mixer(A)], width=256, vocab=10811, ff=5632)
    st = state(cfg)
    e = engine(cfg, st, torch.bfloat16)
    toks = [tokens(cfg, 4, seed=i) for i in range(rows)]
    s = sequences(e)
    s.step([(i, t[:3], []) for i, t in enumerate(toks)])
    got = s.step([(i, t[3:], [0]) for i, t in enumerate(toks)])
    want = torch.cat([po.forward(cfg, double(st), t)[0][3:] for t in toks])
    assert rms_err(got, want) < TOL[torch.bfloat16]


@pytest.mark.parametrize("keys", [16384, 16385, 16600, 40000])
def test_a_context_of_more_splits_than_are_combined(dev, keys):
    """one sequence of up to 256 splits of two tiles (16 384 keys with the new one) and of more, which get longer ones, alone and between short ones.
    Even weights, and cached rows that are zero but for one key tile (the first, the last and ones between): the logits show whether its
    split was read once. Against the row-by-row kernel on the same rows"""
    from cogstream_amd import _lib as L
    cfg = config([dict(mixer(A, heads=20, dim=16, rot=32, vdim=32, kv_rank=64, scale=1e-7), ff=None)], width=64, vocab=96)
    e = engine(cfg, state(cfg), torch.bfloat16)
    g = torch.Generator(device=dev).manual_seed(keys)
    for contexts in ([keys - 1], [37, keys - 1, 900]):
        caches = [e.new_cache(n + 1) for n in contexts]
        rows = caches[len(contexts) // 2]._blocks()[0]

        def step(name, value):
            for c, n in zip(caches, contexts):
                c.reset(n)
            with L.debug_switch(name, value):
                return e.forward_batch(e.embed_tokens(torch.arange(len(contexts))), [1] * len(contexts), caches, list(range(len(contexts)))).cpu()

        for c in caches:
            c.k.zero_()
        empty = step("mla_rowwise", 1)
        for first in (0, 32 * 191, 32 * 192, keys // 2 // 32 * 32, (keys - 33) // 32 * 32, (keys - 1) // 32 * 32):
            for c in caches:
                c.k.zero_()
            tile = rows[first:min(first + 32, keys - 1)]
            if len(tile):
                tile.copy_(torch.randn(64 + 32, generator=g, device=dev) * keys / len(tile))
            want = step("mla_rowwise", 1)
            assert not len(tile) or rms_err(empty, want) > 10 * TOL[torch.bfloat16], first
            for keys_a_split in (0, 64):
                assert rms_err(step("mla_split_keys", keys_a_split), want) < TOL[torch.bfloat16], (contexts, first, keys_a_split)


@pytest.mark.parametrize("kv_rank,heads,n", [(56, 32, 63), (56, 32, 64), (200, 16, 33)])
def test_splits_combined_by_four_waves_or_by_one(dev, kv_rank, heads, n):
    """one token of many sequences: 2016 workgroups of the combine (four waves each) and 2048 or more (a wave each), latents of 64 and of 208 columns, with
    and without a sink, one split to more than 64, against the oracle"""
    from cogstream_amd import _lib as L
    cfg = config([mixer(k, heads=heads, dim=16, rot=16, vdim=16, q_rank=40, kv_rank=kv_rank) for k in (G, B)], width=96, vocab=64)
    st = state(cfg)
    e = engine(cfg, st, torch.bfloat16)
    toks = tokens(cfg, 2100)
    lg = po.forward(cfg, double(st), toks)[0]
    lens = ([2099, 1, 2, 31, 32, 33, 63, 64, 65, 300, 511, 513] * 6)[:n]
    lens = [m if i < 12 else min(m, 513) for i, m in enumerate(lens)]
    s = sequences(e)
    for i, m in enumerate(lens):
        s.step([(i, toks[:m], [])])
    for keys_a_split in (32, 0):
        with L.debug_switch("mla_split_keys", keys_a_split):
            got = s.step([(i, [toks[m]], [0]) for i, m in enumerate(lens)])
        assert rms_err(got, lg[lens]) < TOL[torch.bfloat16], keys_a_split
        for i, m in enumerate(lens):
            s.caches[i].reset(m)


@pytest.mark.parametrize("rows", [2, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("width,ff", [(70, 4100), (1100, 1030), (3140, 4100)])
def test_sublayer_outputs_in_partial_sums(dev, rows, width, ff):
    """up to 64 rows: the products into the residual stream are stored as 2, 4 or 8 partial sums (a bias in the first) that the
    stream's norm adds up; odd widths, K on both sides of the line between two ways to cut it, against the oracle"""
    cfg = config([mixer(G, heads=8, dim=32, rot=16, vdim=130)], width=width, ff=ff, vocab=97)
    st = state(cfg)
    toks = tokens(cfg, rows)
    got = run(engine(cfg, st, torch.bfloat16), toks)
    assert rms_err(got, po.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("width,ff", [(70, 4100), (1100, 1030), (3140, 4100)])
def test_one_row_in_partial_sums(dev, width, ff):
    """... of a single row, which the same kernel takes"""
    test_sublayer_outputs_in_partial_sums(dev, 1, width, ff)


@pytest.mark.parametrize("width,ff,vocab", [(64, 1000, 2032), (64, 2048, 4096), (200, 5200, 10496), (200, 2600, 13000), (64, 9000, 33000)])
def test_one_row_by_the_few_row_product_or_the_gemv(dev, width, ff, vocab):
    """products of one row, N on both sides of 128 workgroups, of four fifths of a round, of one and of two rounds: the logits of single tokens against the
    oracle"""
    cfg = config([mixer(G, heads=2, dim=16, rot=16, vdim=16), mixer(A, heads=3)], width=width, ff=ff, vocab=vocab)
    st = state(cfg)
    toks = tokens(cfg, 6)
    got = run(engine(cfg, st, torch.bfloat16), toks, range(1, 6))
    assert rms_err(got, po.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_a_query_tile_by_one_wave_or_by_two(dev, name):
    """many prompts at once (each query tile's keys are one wave's) and few (every second key tile is another wave's): prompts that end
    at the edges of the 64-key tiles and of the 128-row tiles, from nothing and behind cached tokens, against the oracle"""
    cfg, st, e, toks, lg, _ = named(name, torch.bfloat16, dev, 400)
    lens = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 257]
    for times in (1, 20):
        for cut in (0, 30):
            s = sequences(e)
            jobs = [(i, n) for i, n in enumerate(lens * times) if n > cut]
            if cut:
                s.step([(i, toks[:cut], []) for i, _ in jobs])
            out = s.step([(i, toks[cut:n], [n - 1 - cut]) for i, n in jobs])
            assert rms_err(out, lg[[n - 1 for _, n in jobs]]) < TOL[torch.bfloat16], (times, cut)


@pytest.mark.parametrize("name", ["peaked", "mixed"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 127, 129, 191, 193, 300])
def test_query_tiles_of_64_rows(dev, name, n):
    """one prompt, few query tiles: they have 64 rows, one group of 16 a wave, whose second half of the keys another wave hands over; the edges of both
    kinds of tiles, from nothing and behind cached tokens, against the oracle"""
    cfg, st, e, toks, lg, _ = named(name, torch.bfloat16, dev, 400)
    for cut in (0, 1, 70):
        s = sequences(e)
        if cut:
            s.step([(0, toks[:cut], [])])
        out = s.step([(0, toks[cut:cut + n], list(range(n)))])
        assert rms_err(out, lg[cut:cut + n]) < TOL[torch.bfloat16], cut


def test_short_prompts_beside_a_long_one(dev):
    """a prompt of many key tiles by itself has each query tile's keys shared by two waves; short ones beside it, most of whose query tiles are
    empty, take that away (every workgroup would wait for a whole CU) and none of the result"""
    from cogstream_amd import _lib as L
    cfg, st, e, toks, _, _ = named("peaked", torch.bfloat16, dev, 150)
    toks = tokens(cfg, 1100, seed=3)
    lens = [1100] + [64] * 15
    alone = [sequences(e).step([("r", toks[:n], [n - 1])]).cpu() for n in (64, 1100)]
    assert L.debug_get("mla_last_waves") == 8
    out = sequences(e).step([(i, toks[:n], [n - 1]) for i, n in enumerate(lens)])
    assert L.debug_get("mla_last_waves") == 4
    for i, n in enumerate(lens):
        assert rms_err(out[i:i + 1], alone[n == 1100]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_workspace_serves_every_smaller_step(dev, dtype):
    """of one sequence, from two rows on: few rows need partial sums of their own, and no more memory for them than more rows do"""
    import ctypes as C
    from cogstream_amd import _lib as L
    cfg, st, e, toks, _, _ = named("mixed", dtype, dev, 150)
    e._activate()
    sizes = []
    for rows in range(2, 140):
        n = C.c_size_t()
        L.check(L.lib.cogs_decoder_workspace_bytes(e.handle.h, rows, 1, 200, 1, C.byref(n)))
        sizes.append(n.value)
    assert sizes == sorted(sizes)


def test_unsupported_calls_are_refused(dev):
    from cogstream_amd import _lib as L
    cfg, st, e, toks, _, _ = named("peaked", torch.bfloat16, dev, 150)
    emb = e.embed_tokens(torch.tensor(toks[:4]))
    c = e.new_cache(8)
    for args in (([3], [e.new_cache(2)], []), ([1, 2], [c, c], []), ([3], [c], [3]), ([3], [c], [-1])):
        with pytest.raises(L.CogsError):
            e.forward_batch(emb[:3], *args)
    assert c.len == 0


# ------------------------------------------------------------------------------------------------ fused GEMM epilogues
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M", [1, 5, 200, 700, 2048])
def test_gemm_swiglu_with_bias_and_rotation_without(dev, dtype, M):
    """biases inside the gated activation (rows and biases interleaved) and rotary columns without a bias, in every GEMM body"""
    from cogstream_amd import _lib as L
    from cogstream_amd import ops
    g = torch.Generator().manual_seed(M)
    K, N = 320, 768
    a = torch.randn(M, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    b = torch.randn(N, generator=g).to(dtype)
    lin = a.double() @ w.double().T
    v = lin + b.double()
    want = torch.nn.functional.silu(v[:, 0::2]) * v[:, 1::2]
    got = ops.gemm(a.to(dev), w.to(dev), b.to(dev), act=L.ACT_SWIGLU)
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
    assert float((got.cpu().double() - want).abs().max() / want.abs().max()) < tol
    for hd in (96, 192):
        ang = torch.rand(M, hd // 2, generator=g) * 6
        c, s = ang.cos(), ang.sin()
        x = lin.view(M, N // hd, hd // 2, 2)
        want = torch.stack([x[..., 0] * c[:, None] - x[..., 1] * s[:, None], x[..., 1] * c[:, None] + x[..., 0] * s[:, None]], -1).view(M, N)
        got = ops.gemm(a.to(dev), w.to(dev), rope_cos=torch.stack([c, s], -1).to(dev).contiguous(), rope_cols=N, head_dim=hd)
        assert float((got.cpu().double() - want).abs().max() / want.abs().max()) < tol


# ------------------------------------------------------------------------------------------------ the framework's entry points
def _checkpoint(tmp_path, name):
    from cogstream_amd import checkpoint as ck
    cfg = CONFIGS[name]
    st = state(cfg)
    ck.save_decoder(str(tmp_path), cfg, st)
    return cfg, st


def test_greedy_generation_through_the_registry(dev, tmp_path):
    """AutoModelForCausalLM -> generate: one prompt, several unequal prompts in one batch, in groups, with an end token, and the
    single-sequence loop with its prefix cache, against the oracle's greedy continuation"""
    from cogstream_amd.auto import AutoModelForCausalLM
    from cogstream_amd.llm import PrefixKV
    cfg, st = _checkpoint(tmp_path, "peaked")
    m = AutoModelForCausalLM.from_pretrained(str(tmp_path), torch_dtype=torch.float32)
    prompts = [tokens(cfg, n, seed=n) for n in (9, 1, 30, 66)]
    want = [po.greedy(cfg, double(st), p, 8) for p in prompts]
    assert m.generate(prompts[0], max_new_tokens=8) == [want[0]]
    assert m.generate(torch.tensor(prompts[2]), max_new_tokens=8) == [want[2]]
    assert m.generate(prompts, max_new_tokens=8) == want
    assert m.generate(prompts, max_new_tokens=8, max_batch=3) == want
    stop = want[3][2]
    cut = [w[:w.index(stop) + 1] if stop in w else w for w in want]
    assert m.generate(prompts, max_new_tokens=8, eos_token_id=[stop]) == cut
    assert m.generate(prompts, max_new_tokens=8, eos_token_id=stop) == cut
    e = m.llm
    emb = e.embed_tokens(torch.tensor(prompts[3]))
    assert e.generate(emb, max_new_tokens=8) == want[3]
    pre = PrefixKV(e)
    assert e.generate(emb, max_new_tokens=8, prefix=pre) == want[3]
    longer = prompts[3] + tokens(cfg, 40, seed=5)
    assert e.generate(e.embed_tokens(torch.tensor(longer)), max_new_tokens=4, prefix=pre) == po.greedy(cfg, double(st), longer, 4)
    assert pre.reused == 66
    # sampling: a request's draws do not depend on its batch; top_k = 1 is greedy
    a = m.generate(prompts, max_new_tokens=6, do_sample=True, temperature=0.8, top_k=20, top_p=0.9, seed=3)
    assert a == m.generate(prompts, max_new_tokens=6, do_sample=True, temperature=0.8, top_k=20, top_p=0.9, seed=3)
    assert a[0] == m.generate(prompts[0], max_new_tokens=6, do_sample=True, temperature=0.8, top_k=20, top_p=0.9, seed=3)[0]
    assert m.generate(prompts, max_new_tokens=8, do_sample=True, top_k=1) == want


def test_two_models_share_a_handle(dev):
    """the handle keeps one decoder; engines re-activate themselves, also in turns and in either type"""
    a, b = named("peaked", torch.float32, dev, 150), named("mixed", torch.bfloat16, dev, 150)
    sa, sb = sequences(a[2]), sequences(b[2])
    for lo, hi in ((0, 60), (60, 61), (61, 90)):
        ra = sa.step([("r", a[3][lo:hi], list(range(hi - lo)))])
        rb = sb.step([("r", b[3][lo:hi], list(range(hi - lo)))])
        assert rms_err(ra, a[4][lo:hi]) < TOL[torch.float32] and rms_err(rb, b[4][lo:hi]) < TOL[torch.bfloat16]


def test_models_of_the_same_rotations_take_turns(dev):
    """engines whose tables on the device are the same, whose rotations differ in a number or in their frequencies, and one without any, in turn on a handle:
    each against its own oracle"""
    models = []
    for i, cfg in enumerate((CONFIGS["peaked"], CONFIGS["peaked"], config([mixer(G, heads=4), mixer(B, heads=4)], width=192, ff=128),
                             config([mixer(G, heads=4, base=500.0), mixer(B, heads=4, base=500.0)], width=192, ff=128))):
        st = state(cfg, seed=10 + i)
        toks = tokens(cfg, 40, seed=i)
        e = engine(cfg, st, torch.bfloat16)
        models.append((e, toks, po.forward(cfg, double(st), toks)[0], sequences(e)))
    for lo, hi in ((0, 20), (20, 21), (21, 40)):
        for order in ((0, 1, 2, 3), (3, 1, 0, 2)):
            for m in order:
                e, toks, lg, s = models[m]
                if order[0] == 3:
                    s.caches["r"].reset(lo)
                got = s.step([("r", toks[lo:hi], list(range(hi - lo)))])
                assert rms_err(got, lg[lo:hi]) < TOL[torch.bfloat16], (m, lo)


def test_command_lines(dev, tmp_path):
    """python -m cogstream_amd.generate and bin/trace_run in processes of their own"""
    cfg, st = _checkpoint(tmp_path, "peaked")
    w = double(st)
    prompts = [tokens(cfg, n, seed=n) for n in (9, 30)]
    r = subprocess.run([sys.executable, "-m", "cogstream_amd.generate", "--model_path", str(tmp_path), "--dtype", "float32", "--max_new_tokens", "6",
                        "--greedy"] + [x for p in prompts for x in ("--prompt", ",".join(map(str, p)))], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [json.loads(x)["tokens"] for x in r.stdout.splitlines()] == [po.greedy(cfg, w, p, 6) for p in prompts]
    out = tmp_path / "out"
    out.mkdir()
    a, b = tokens(cfg, 40, seed=1), tokens(cfg, 25, seed=2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:37], "want": [0, 36]}, {"id": "b", "tokens": b[:24], "want": [23]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[37:38], "want": []}, {"id": "b", "tokens": b[24:], "want": []}], "end": ["b"]},
             {"step": 7, "entries": [{"id": "a", "tokens": a[38:39], "want": [0]}], "end": ["a"]},
             {"step": 8, "entries": [{"id": "a", "tokens": b, "want": [24]}], "end": []}]
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", "float32", "--out", str(out), "--max-tokens", "64"],
                       input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, cwd=str(tmp_path), timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [x for x in r.stdout.splitlines() if x.startswith("done")] == ["done 0", "done 1", "done 7", "done 8"]
    assert sorted(os.listdir(out)) == ["0.f32", "7.f32", "8.f32"]
    la, lb = po.forward(cfg, w, a)[0], po.forward(cfg, w, b)[0]
    load = lambda n: torch.frombuffer(bytearray((out / f"{n}.f32").read_bytes()), dtype=torch.float32).view(-1, cfg["vocab"])
    assert rms_err(load(0), torch.stack([la[0], la[36], lb[23]])) < TOL[torch.float32]
    assert rms_err(load(7), la[38:39]) < TOL[torch.float32] and rms_err(load(8), lb[24:25]) < TOL[torch.float32]


def test_qwen2_engine_takes_the_same_batches(dev):
    """Sequences and generate_batch over the Qwen2 engine: its logits are its own single-sequence ones"""
    from cogstream_amd.llm import Qwen2Engine
    from cogstream_amd.weights import LlmConfig, random_llm_state
    cfg = LlmConfig(hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=2, num_key_value_heads=1,
                    vocab_size=512, image_token_index=500, eos_token_id=499)
    e = Qwen2Engine(random_llm_state(cfg, seed=7, std=0.05), cfg, dtype=torch.float32, device=dev)
    prompts = [list(range(3, 40)), [5, 6, 7], [9]]
    s = sequences(e, 8)
    out = s.step([(i, p, [len(p) - 1]) for i, p in enumerate(prompts)])
    for i, p in enumerate(prompts):
        want = e.forward(e.embed_tokens(torch.tensor(p)), e.new_cache(64))["logits"]
        assert torch.equal(out[i], want)
    got = e.generate_batch(prompts, max_new_tokens=5)
    assert got == [e.generate(e.embed_tokens(torch.tensor(p)), max_new_tokens=5) for p in prompts]
