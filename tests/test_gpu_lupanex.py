"""Lupanex on the GPU against its oracle (oracle/lupanex.py): every mechanism alone, prompts against token-by-token decoding, prompts
in portions, unequal batches, caches and states that grow, are freed and used again, keys at every place of interest, the edges of
the distance buckets, memories over hundreds of tokens, first tokens, long decoding, other sizes, and generation through the
framework's entry points. float32 pins the arithmetic, bfloat16 the kernels."""
import json
import os
import subprocess
import sys

import pytest
import torch

from lupanex_models import CONFIGS, attention, config, delta, double, parse, public, rms_err, state, tokens
from oracle import lupanex as lo

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# largest row error of the logits. bfloat16: about twice what rounding the operands of the matrix products does to these models
TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}
TINY = 2.5        # the eight-wide models have nothing to average rounding errors over
DTYPES = [torch.float32, torch.bfloat16]
LONG = {"wide": 100, "large": 100}
_cache = {}


def tol(name, dtype):
    return TOL[dtype] * (TINY if name.startswith("one") else 1)


def engine(cfg, st, dtype):
    from cogstream_amd.llm import DecoderEngine
    return DecoderEngine(st, parse(cfg), dtype=dtype, device="cuda:0")


def named(name, dtype, n=150):
    """(config, weights, engine, tokens, oracle logits, oracle streams) of a shared model, made once"""
    if (name, dtype) not in _cache:
        cfg = CONFIGS[name]
        st = state(cfg)
        _cache[(name, dtype)] = (cfg, st, engine(cfg, st, dtype))
    cfg, st, e = _cache[(name, dtype)]
    if (name, n) not in _cache:
        t = tokens(cfg, n)
        _cache[(name, n)] = (t,) + lo.forward(cfg, double(st), t)
    return (cfg, st, e) + _cache[(name, n)]


def sequences(e, reserve=64):
    from cogstream_amd.llm import Sequences
    return Sequences(e, reserve)


def run(e, toks, cuts=(), reserve=64):
    """logits of every token, the prompt cut at `cuts`"""
    s = sequences(e, reserve)
    edges = [0, *cuts, len(toks)]
    return torch.cat([s.step([("r", toks[a:b], list(range(b - a)))]) for a, b in zip(edges, edges[1:])])


def both_ways(cfg, st, dtype, n, seed=0, cuts=(37, 90), limit=None):
    """a model whole, in portions and token by token against its oracle"""
    toks = tokens(cfg, n, seed=seed)
    lg = lo.forward(cfg, double(st), toks)[0]
    e = engine(cfg, st, dtype)
    for c in ((), [x for x in cuts if x < n], range(1, n)):
        assert rms_err(run(e, toks, c), lg) < (limit or TOL[dtype]), c
    return e, toks, lg


# ------------------------------------------------------------------------------------------------ mechanisms
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_prompt_against_the_oracle_layer_by_layer(dev, name, dtype):
    """logits and the residual stream behind every layer run, all sizes (also those above the matrix kernels' instances)"""
    n = LONG.get(name, 150)
    cfg, st, e, toks, lg, streams = named(name, dtype, n)
    W = cfg["width"]
    buf = torch.empty(len(streams), n, e.packed.width_p, device=dev)
    got = e.forward_batch(e.embed_tokens(torch.tensor(toks)), [n], [e.new_cache(n)], list(range(n)), streams=buf)
    assert got.shape == (n, cfg["vocab"])
    for i, want in enumerate(streams):
        assert rms_err(buf[i, :, :W], want) < tol(name, dtype), (name, i)
        assert not buf[i, :, W:].any()
    assert rms_err(got, lg) < tol(name, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_decoding_against_the_oracle(dev, name, dtype):
    """from the first token on"""
    n = LONG.get(name, 150)
    cfg, st, e, toks, lg, _ = named(name, dtype, n)
    assert rms_err(run(e, toks, range(1, n)), lg) < tol(name, dtype)


def alone(mech):
    """one layer in which one mechanism decides"""
    st = None
    if mech == "bias":                     # no content scores at all: the weights are the bias table's
        cfg = config([attention(heads=4, kv_heads=2, rows=10, far=80, temp=None, ff=None)], width=128)
        st = state(cfg)
        st["l0.mix.q"] *= 0
    elif mech == "temperature":            # every position its own temperature, and a steep one
        cfg = config([attention(heads=3, dim=32, rows=4, far=9, temp=(1.5, 1), ff=None)], width=128)
    elif mech == "temperature_fraction":   # a period that is no whole number of tokens
        cfg = config([attention(heads=2, temp=(0.7, 6.5), ff=None)], width=64)
    elif mech == "qk_norm":                # queries and keys of very unlike sizes
        cfg = config([attention(heads=2, dim=40, ff=None)], width=64, eps=1e-2)
        st = state(cfg)
        st["l0.mix.q"] *= 0.05
        st["l0.mix.k"] *= torch.logspace(-2, 1, st["l0.mix.k"].shape[0])[:, None]
    elif mech == "groups":
        cfg = config([attention(heads=12, kv_heads=3, dim=16, vdim=16, ff=None)], width=128)
    elif mech == "delta":
        cfg = config([delta(ff=None)], width=128)
    elif mech == "delta_fast":             # decays from nearly nothing kept to everything kept, heads unlike
        cfg = config([delta(heads=4, kv_heads=1, dim=32, vdim=16, ff=None)], width=128)
        st = state(cfg)
        st["l0.mix.A_log"], st["l0.mix.dt_bias"] = torch.tensor([4.0, 1.0, -3.0, -9.0]), torch.tensor([6.0, 0.0, -1.0, -8.0])
    elif mech == "delta_hard":             # beta near 0 and near 1, keys often alike
        cfg = config([delta(heads=4, kv_heads=2, dim=8, vdim=16, ff=None)], width=128, vocab=6)
        st = state(cfg)
        st["l0.mix.b"] *= 8
    elif mech == "delta_zero":             # unit vectors of nothing: the first query and key channels see silu(0)
        cfg = config([delta(heads=2, kv_heads=2, conv=4, ff=None)], width=64)
        st = state(cfg)
        st["l0.mix.q"][:20] *= 0
        st["l0.mix.k"][:20] *= 1e-4
    elif mech in ("conv1", "conv2", "conv7", "conv12"):
        cfg = config([delta(heads=2, conv=int(mech[4:]), ff=None)], width=64)
    elif mech == "hyper":                  # the sublayers do nothing: the streams only mix
        cfg = config([delta(heads=2, kv_heads=1), attention(heads=2)], width=64, streams=6, loop=(0, 2, 2))
        st = state(cfg)
        for k in st:
            if k.endswith(("mix.o", "mlp.down")):
                st[k] = st[k] * 0
    elif mech == "hyper1":                 # a single stream with weights of its own
        cfg = config([attention(heads=2), delta(heads=2, kv_heads=1)], width=64, streams=1)
    elif mech == "loop":
        cfg = config([delta(heads=2, kv_heads=2), attention(heads=2)], width=64, loop=(0, 1, 4))
    elif mech == "feed_forward":
        cfg = config([delta(heads=1, kv_heads=1, dim=4, vdim=4, ff=200)], width=64)
        st = state(cfg)
        st["l0.mix.o"] *= 0
        st["l0.mlp.up"] *= 2
    elif mech == "positions":              # one word over and over
        cfg = config([attention(heads=2, ff=None)], width=64)
        st = state(cfg)
        st["embed"][:] = st["embed"][0]
    st = state(cfg) if st is None else st
    return cfg, {k: v.to(torch.bfloat16).float() for k, v in st.items()}


@pytest.mark.parametrize("mech", ["bias", "temperature", "temperature_fraction", "qk_norm", "groups", "delta", "delta_fast", "delta_hard", "delta_zero", "conv1", "conv2",
                                  "conv7", "conv12", "hyper", "hyper1", "loop", "feed_forward", "positions"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_mechanism_alone(dev, mech, dtype):
    cfg, st = alone(mech)
    both_ways(cfg, st, dtype, 110)


@pytest.mark.parametrize("rows,far", [(2, 3), (6, 40), (16, 128), (32, 64), (8, 2000)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_edges_of_the_distance_buckets(dev, rows, far, dtype):
    """each head's table has one bucket far above the others, so the output is the mean of exactly that bucket's values: every
    first and last distance of every bucket, in prompts, portions and decoding"""
    n = 330
    cfg = config([attention(heads=rows, kv_heads=1, dim=8, vdim=32, rows=rows, far=far, temp=None, ff=None)], width=64, vocab=128)
    st = state(cfg, seed=rows)
    st["l0.mix.q"] *= 0
    st["l0.mix.rel"] = 16 * torch.eye(rows) - 3
    toks = tokens(cfg, n)
    lg = lo.forward(cfg, double(st), toks)[0]
    e = engine(cfg, st, dtype)
    assert rms_err(run(e, toks), lg) < TOL[dtype]
    assert rms_err(run(e, toks, [200, 203, *range(230, n)]), lg) < TOL[dtype]


# ------------------------------------------------------------------------------------------------ one key among many
def needle_model(heads=2, kv_heads=2, dim=32, scale=0.7, seed=7):
    """token 1 asks for token 2: one score is far above all others, so whether exactly that key is seen shows in the logits"""
    cfg = config([attention(heads=heads, kv_heads=kv_heads, dim=dim, vdim=32, rows=12, far=100, scale=scale, temp=(0.1, 50), ff=None)], width=64, vocab=64, streams=2)
    st = state(cfg, seed=seed)
    st["pos"] *= 0.02
    st["l0.mix.rel"] *= 0.3
    w = double(st)
    x = w["embed"] * cfg["embedding"]["scale"]
    h = lo.rms(sum(w["l0.hc1.in"][s] * x for s in range(2)), cfg["norm"]["eps"]) * w["l0.norm1"]
    for i in range(heads):
        g = i // (heads // kv_heads)
        q, k = w["l0.mix.q"][i * dim:(i + 1) * dim], w["l0.mix.k"][g * dim:(g + 1) * dim]
        st["l0.mix.q"][i * dim:(i + 1) * dim] = (q + torch.outer(k @ h[2] - q @ h[1], h[1]) / (h[1] @ h[1])).float()
    return cfg, {k: v.to(torch.bfloat16).float() for k, v in st.items()}


@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (6, 2)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_a_single_key_at_every_place_of_interest(dev, heads, kv_heads, dtype):
    """the asked-for key first, last, at tile and split borders, itself, and one past the query (which must not be seen)"""
    cfg, st = needle_model(heads, kv_heads)
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
        lg = lo.forward(cfg, w, toks)[0]
        if at is None:
            without = lg[ask]
        else:
            assert rms_err(lg[ask:], without[None]) > 0.3            # the oracle's answer depends on that key
        assert rms_err(run(e, toks)[ask:], lg[ask:]) < TOL[dtype], ("prompt", at)
        assert rms_err(run(e, toks, [ask])[ask:], lg[ask:]) < TOL[dtype], ("decoded", at)
        assert rms_err(run(e, toks, [ask - 70])[ask:], lg[ask:]) < TOL[dtype], ("second portion", at)
    # the key right behind the query: invisible, also when it shares the query's tile
    for ask in (0, 15, 62, 63, 64, 126, 127, 128, 200):
        toks = list(base)
        toks[ask], toks[ask + 1] = 1, 2
        lg = lo.forward(cfg, w, toks[:ask + 2])[0]
        assert rms_err(run(e, toks[:ask + 2]), lg) < TOL[dtype], ask


def memory_model(dim=48):
    """a delta layer that keeps everything and writes only on token 2, whose key token 1 reads back"""
    cfg = config([delta(heads=2, kv_heads=1, dim=dim, vdim=32, conv=2, ff=None)], width=64, vocab=40, streams=1)
    st = state(cfg, seed=4)
    st["pos"] *= 0
    w = double(st)
    h = lo.rms(w["l0.hc1.in"][0] * w["embed"] * cfg["embedding"]["scale"], cfg["norm"]["eps"]) * w["l0.norm1"]
    for n in "qkv":
        st[f"l0.mix.{n}.conv"] = torch.tensor([0.0, 1.0]).repeat(len(st[f"l0.mix.{n}.conv"]), 1)
    want = torch.full((40, 2), -12.0, dtype=torch.float64)
    want[2] = 6
    st["l0.mix.b"] = (torch.linalg.pinv(h) @ want).T.float()
    st["l0.mix.dt_bias"] = torch.full((2,), -20.0)
    q, k = w["l0.mix.q"], w["l0.mix.k"]
    st["l0.mix.q"] = (q + torch.outer(k @ h[2] - q @ h[1], h[1]) / (h[1] @ h[1])).float()
    return cfg, {k: v.to(torch.bfloat16).float() for k, v in st.items()}


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_write_is_read_back_from_any_distance(dev, dtype):
    """a single write at chunk borders, the first token, the query's neighbour, read hundreds of tokens later: in one prompt, decoded, and
    with portions of every kind between write and read"""
    cfg, st = memory_model()
    e, w = engine(cfg, st, dtype), double(st)
    n = 330
    base = [t if t > 2 else 3 + t for t in tokens(cfg, n)]
    ask, without = n - 1, None
    for at in (None, 0, 1, 15, 16, 30, 31, 32, 33, 63, 64, 160, 319, 320, n - 2):
        toks = list(base)
        toks[ask] = 1
        if at is not None:
            toks[at] = 2
        lg = lo.forward(cfg, w, toks)[0]
        if at is None:
            without = lg[ask]
        else:
            assert rms_err(lg[ask:], without[None]) > 0.2
        for cuts in ((), [ask], [32, 64, 97], [2, 3, ask - 2], [max(at or 1, 1), (at or 1) + 1] if (at or 1) + 1 < n else [at]):
            assert rms_err(run(e, toks, cuts)[ask:], lg[ask:]) < TOL[dtype], (at, cuts)


# ------------------------------------------------------------------------------------------------ schedules
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_portions_of_a_prompt(dev, name, dtype):
    cfg, st, e, toks, lg, _ = named(name, dtype)
    for cuts in ([2], [1, 3], [31], [32], [33], [64], [63, 65], [128], [149], [148], [50, 52, 54, 118], list(range(2, 150, 2)), list(range(3, 150, 3)), list(range(7, 150, 29))):
        assert rms_err(run(e, toks, cuts), lg) < TOL[dtype], cuts


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129])
@pytest.mark.parametrize("dtype", DTYPES)
def test_short_sequences_and_first_tokens(dev, n, dtype):
    cfg, st, e, toks, lg, _ = named("peaked", dtype)
    assert rms_err(run(e, toks[:n]), lg[:n]) < TOL[dtype]
    assert rms_err(run(e, toks[:n] + toks[n:n + 2], [n, n + 1]), lg[:n + 2]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_unequal_batch_against_each_alone(dev, name, dtype):
    """prompts of 1 .. 140 tokens in one step, then decoded together, shorter requests ending earlier; and steps that mix whole
    prompts with single tokens"""
    cfg, st, e, _, _, _ = named(name, dtype)
    w = double(st)
    lens = [1, 140, 2, 65, 64, 33, 17, 90]
    full = [tokens(cfg, n + 3 + i, seed=i) for i, n in enumerate(lens)]
    want = [lo.forward(cfg, w, t)[0] for t in full]
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
    cfg, st, e, toks, lg, _ = named("peaked", dtype)
    for count in (2, 16, 17, 40, 70):
        s = sequences(e)
        s.step([(i, toks[:1 + i], []) for i in range(count)])
        out = s.step([(i, [toks[1 + i]], [0]) for i in range(count)])
        assert rms_err(out, lg[1:1 + count]) < TOL[dtype], count


@pytest.mark.parametrize("dtype", DTYPES)
def test_memory_that_is_freed_and_used_again(dev, dtype):
    """caches, states and workspaces that hold another request's rows, or NaN, change nothing"""
    cfg, st, e, toks, lg, _ = named("mixed", dtype)
    s = sequences(e, 16)
    for r in range(6):
        n = [90, 20, 130, 60, 7, 150][r]
        poison = [torch.full((sum(e.packed.cache_widths) * (-(-n // 16) * 16),), float("nan"), device=dev, dtype=dtype),
                  torch.full((e.packed.state_floats,), float("nan"), device=dev)]
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
    # a cache with everything NaN, from the first token on, by either kernel of the delta rule
    for cuts in ((), range(1, 12)):
        c = e.new_cache(64)
        c.k.fill_(float("nan"))
        c.state.fill_(float("nan"))
        edges = [0, *cuts, 12]
        for a, b in zip(edges, edges[1:]):
            out = e.forward_batch(e.embed_tokens(torch.tensor(toks[a:b])), [b - a], [c], [b - a - 1])
            assert rms_err(out, lg[b - 1:b]) < TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding_through_a_growing_cache(dev, dtype):
    cfg, st, e, toks, lg, _ = named("peaked", dtype, 400)
    assert rms_err(run(e, toks, range(5, 400), reserve=8), lg) < TOL[dtype]


def test_forms_and_kernels_agree(dev):
    """bfloat16: chunked against token-by-token delta rule, MFMA against row-wise attention, few-row against general GEMM, and any
    number of key splits: all inside the tolerance of the oracle"""
    from cogstream_amd import _lib as L
    cfg, st, e, toks, lg, _ = named("peaked", torch.bfloat16, 400)
    for name, value in (("delta_chunk", 0), ("mla_rowwise", 1), ("gemm_skinny", 0), ("mla_split_keys", 16), ("mla_split_keys", 100), ("mla_split_keys", 4096)):
        with L.debug_switch(name, value):
            assert rms_err(run(e, toks, [20, 380, *range(381, 400)]), lg) < TOL[torch.bfloat16], (name, value)


@pytest.mark.parametrize("rows", [3, 16, 31, 64])
@pytest.mark.parametrize("width,ff", [(70, 4100), (1100, 1030), (2120, 4100)])
def test_sublayer_outputs_in_partial_sums(dev, rows, width, ff):
    """as in test_gpu_pabalix.py, through the hyper-connected streams"""
    cfg = config([attention(heads=8, kv_heads=2, dim=32, vdim=130), delta(heads=8, kv_heads=4, dim=16, vdim=130)], width=width, ff=ff, vocab=97)
    st = state(cfg)
    toks = tokens(cfg, rows)
    got = run(engine(cfg, st, torch.bfloat16), toks)
    assert rms_err(got, lo.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("rows", [2, 8, 9, 17, 33])
@pytest.mark.parametrize("width,ff", [(70, 10300), (1344, 5200)])
def test_few_row_products_at_the_edges_of_their_rings(dev, rows, width, ff):
    """rows at the edges of 8-row pieces and 16-row groups; waves with no, one and more slices than their ring holds (K = 128, 192, 1344,
    5248, 10 304); 16, 32 and 64 columns at a time, ragged at the end; partial sums"""
    cfg = config([attention(heads=4, kv_heads=2, dim=32, vdim=40)], width=width, ff=ff, vocab=97)
    st = state(cfg)
    toks = tokens(cfg, rows)
    got = run(engine(cfg, st, torch.bfloat16), toks)
    assert rms_err(got, lo.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("width,ff", [(70, 10300), (1344, 5200)])
def test_one_row_products_at_the_edges_of_their_rings(dev, width, ff):
    """... a single row"""
    test_few_row_products_at_the_edges_of_their_rings(dev, 1, width, ff)


@pytest.mark.parametrize("dim,vdim,conv", [(16, 16, 1), (64, 256, 4), (256, 48, 5), (128, 128, 4), (130, 256, 8), (272, 16, 3), (16, 272, 9)])
def test_one_token_delta_rule_at_the_edges_of_its_kernels(dev, dim, vdim, conv):
    """one to sixteen waves of 16 columns, whole and ragged rows a lane, more channels than threads, windows of one to nine taps that start
    empty and wrap around, shared q / k heads; above 256 rows or columns, or eight taps, the wide form: within the tolerance of the oracle"""
    cfg = config([delta(heads=4, kv_heads=2, dim=dim, vdim=vdim, conv=conv, ff=None)], width=64)
    st = state(cfg)
    toks = tokens(cfg, 24)
    lg = lo.forward(cfg, double(st), toks)[0]
    for dtype in DTYPES:
        e = engine(cfg, st, dtype)
        for first in (1, 5):
            assert rms_err(run(e, toks, range(first, 24), reserve=8), lg) < TOL[dtype], (dtype, first)


@pytest.mark.parametrize("rows", [2, 7, 64])
@pytest.mark.parametrize("width,ff,vocab", [(1100, 200, 61), (1408, 10300, 40003)])
def test_weights_read_beside_a_mix_of_streams(dev, rows, width, ff, vocab):
    """all lines of the next product's rows and some of them (one of 22 of the head's); fewer column groups than XCDs, and numbers of them that
    8 does not divide"""
    cfg = config([attention(heads=4, kv_heads=2, dim=32, vdim=40)], width=width, ff=ff, vocab=vocab, streams=4)
    st = state(cfg)
    toks = tokens(cfg, rows)
    got = run(engine(cfg, st, torch.bfloat16), toks)
    assert rms_err(got, lo.forward(cfg, double(st), toks)[0]) < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("streams,width,loop", [(2, 60, None), (3, 1028, (0, 1, 2)), (4, 2050, None), (4, 320, (0, 2, 2))])
def test_streams_that_wait_for_several_outputs(dev, streams, width, loop, dtype):
    """norm.hip: prompts of more than 64 rows mix the streams of up to four sublayers together and the last ones for the wanted rows
    alone. The bits are those of mixes done at once (asked for by wanting every layer's streams): two to four streams, rows of one to three
    chunks of 1024 columns, chains that end anywhere (3 to 8 outputs), wanted rows anywhere, as few as a row has 1024 threads for and more,
    two sequences, against the oracle too"""
    kw = dict(width=width, streams=streams, ff=128)
    if loop:
        kw["loop"] = loop
    cfg = config([attention(heads=2, kv_heads=1, dim=32, vdim=32), delta(heads=2, kv_heads=1, dim=32, vdim=32, ff=None)], **kw)
    st = state(cfg)
    e = engine(cfg, st, dtype)
    toks = tokens(cfg, 131)
    lens = [66, 65]
    embeds = e.embed_tokens(torch.tensor(toks))
    runs = len(e.cfg.layers) if not loop else len(e.cfg.layers) + (loop[1] - loop[0]) * (loop[2] - 1)
    each = torch.empty(runs, 131, e.packed.width_p, device=dev)
    for want in (list(range(131)), list(range(65)), list(range(20, 84)), list(range(67, 131)), [0, 64, 65, 66, 130]):
        at_once = e.forward_batch(embeds, lens, [e.new_cache(n) for n in lens], want, streams=each)
        got = e.forward_batch(embeds, lens, [e.new_cache(n) for n in lens], want)
        assert torch.equal(got, at_once), len(want)
    assert e.forward_batch(embeds[:65], [65], [e.new_cache(65)], []) is None
    for r, lg in ((slice(0, 3), lo.forward(cfg, double(st), toks[:66])[0][[0, 64, 65]]), (slice(3, 5), lo.forward(cfg, double(st), toks[66:])[0][[0, 64]])):
        assert rms_err(got[r], lg) < TOL[dtype]


@pytest.mark.parametrize("past,n,heads", [(0, 257, 4), (0, 321, 4), (90, 320, 4), (3, 449, 4), (40, 449, 40), (0, 449, 80)])
@pytest.mark.parametrize("name", ["latent", "latent, nothing fed forward", "attention", "delta"])
def test_rows_of_the_last_layer_that_nothing_reads(dev, name, past, n, heads):
    """decoder.hip: a prompt of one sequence goes on behind its last layer's keys, values and state with the query tiles from the first row
    whose logits are asked for. Caches and states bit for bit those of a prompt that wants every row, logits bit for bit those of one that goes
    on with every row (asked for by wanting every layer's streams), wherever the wanted rows lie and whichever form of the attention
    the whole prompt's query tiles have: tiles of 64 rows, of 128 rows in halves, of 128 rows (12 to 16, 160 and 320 tiles, and fewer of the rest)"""
    if name.startswith("latent"):
        import pabalix_models as pm
        from cogstream_amd.llm import DecoderEngine
        layers = [pm.mixer(pm.A, heads=3), pm.mixer(pm.G, heads=heads, kv_rank=56)]
        if "nothing" in name:
            layers[1] = dict(layers[1], ff=None)
        cfg = pm.config(layers, width=136)
        e = DecoderEngine(pm.state(cfg), pm.parse_config(cfg), dtype=torch.bfloat16, device="cuda:0")
    else:
        last = attention(heads=heads, kv_heads=2, dim=64, vdim=32) if name == "attention" else delta(heads=2, kv_heads=1, dim=32, vdim=32)
        cfg = config([delta(heads=2, kv_heads=1, dim=32, vdim=32), last], width=200, streams=4)
        e = engine(cfg, state(cfg), torch.bfloat16)
    toks = torch.tensor([(7 * i * i + 3 * i) % cfg["vocab"] for i in range(past + n + 1)])

    def prompt(want, streams=None):
        c = e.new_cache(past + n + 1)
        if past:
            e.forward_batch(e.embed_tokens(toks[:past]), [past], [c], [])
        got = e.forward_batch(e.embed_tokens(toks[past:past + n]), [n], [c], want, streams=streams)
        return got, c.k.clone(), None if c.state is None else c.state.clone(), e.forward_batch(e.embed_tokens(toks[-1:]), [1], [c], [0])

    every = prompt(list(range(n)))
    for want in ([n - 1], [n - 66, n - 1], [n - 65, n - 2], [n - 1, 128], [127, n - 1], [129], []):
        got, k, st, after = prompt(want)
        at = 0
        for w in e.packed.cache_widths:
            size = w * (past + n + 1)
            assert torch.equal(k[at:at + size].view(-1, w)[:past + n], every[1][at:at + size].view(-1, w)[:past + n]), want
            at += size
        assert st is None or torch.equal(st, every[2]), want
        assert torch.equal(after, every[3]), want
        if want:
            assert rms_err(got, every[0][want].double().cpu()) < TOL[torch.bfloat16], want
            assert torch.equal(got, prompt(want, torch.empty(2, n, e.packed.width_p, device=dev))[0]), want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,vdim", [(1, 16), (2, 128), (3, 96), (7, 112), (17, 32), (33, 128), (9, 144)])
def test_read_outs_of_one_head_or_two_a_wave(dev, heads, vdim, dtype):
    """delta.hip, delta_out_kernel: fewer heads than a workgroup takes at a time, more, numbers that it does not divide, and heads wider than
    half a wave's columns, against the oracle; and, over more rows, the bits of a wave per head"""
    from cogstream_amd import _lib as L
    cfg = config([delta(heads=heads, kv_heads=1, dim=16, vdim=vdim, ff=None)], width=192, streams=2)
    st = state(cfg)
    toks = tokens(cfg, 70)
    e = engine(cfg, st, dtype)
    assert rms_err(run(e, toks), lo.forward(cfg, double(st), toks)[0]) < TOL[dtype]
    embeds = e.embed_tokens(torch.tensor(tokens(cfg, 500)))
    logits = []
    for wave in (0, 1):
        with L.debug_switch("delta_out_wave", wave):
            logits.append(e.forward_batch(embeds, [500], [e.new_cache(500)], list(range(500))))
    assert torch.equal(*logits)


@pytest.mark.parametrize("dim,vdim", [(16, 16), (64, 48), (80, 16), (128, 128), (144, 32), (256, 16)])
def test_chunked_delta_rule_at_the_edges_of_its_tiles(dev, dim, vdim):
    """every number of row tiles per wave, whole and ragged; chunks of one token, whole and ragged ones, one to four of them, from nothing
    and from a state, unequal prompts together: within the tolerance of the oracle, and as close to it as the token-by-token form (both
    sum in fp32, in another order: a quarter more at most, of errors that vary by a tenth from one sequence of words to the next)"""
    from cogstream_amd import _lib as L
    cfg = config([delta(heads=4, kv_heads=2, dim=dim, vdim=vdim, conv=4, ff=None)], width=64)
    st = state(cfg)
    toks = tokens(cfg, 130)
    lg = lo.forward(cfg, double(st), toks)[0]
    e = engine(cfg, st, torch.float32)
    for cuts in ((), [1, 33, 64], [31], [32, 65, 97], [96], [128, 129]):
        got = rms_err(run(e, toks, cuts), lg)
        with L.debug_switch("delta_chunk", 0):
            want = rms_err(run(e, toks, cuts), lg)
        assert got < TOL[torch.float32] and got < 1.25 * want + 1e-7, (cuts, got, want)
    s = sequences(e)
    lens = [1, 33, 96, 130, 32]
    out = s.step([(i, toks[:n], [n - 1]) for i, n in enumerate(lens)])
    assert rms_err(out, lg[[n - 1 for n in lens]]) < TOL[torch.float32]


@pytest.mark.parametrize("dim,vdim,conv", [(32, 80, 1), (128, 48, 3), (64, 16, 6), (256, 32, 8), (48, 130, 9), (144, 32, 11)])
def test_tiles_of_chunks_from_every_convolution(dev, dim, vdim, conv):
    """the kernels that form q, k and v as the scan's tiles (short and long convolutions, runs of 16 and 8 rows, a row at a time): prompts that end
    at the edges of runs, of 16-row tiles and of chunks, together and behind cached tokens, against the oracle (fp32 sums in another order)"""
    cfg = config([delta(heads=4, kv_heads=2, dim=dim, vdim=vdim, conv=conv, ff=None)], width=64)
    st = state(cfg)
    toks = tokens(cfg, 131)
    lg = lo.forward(cfg, double(st), toks)[0]
    e = engine(cfg, st, torch.float32)
    lens = [2, 7, 8, 15, 16, 17, 31, 32, 33, 47, 49, 64, 65, 130]
    s = sequences(e)
    out = s.step([(i, toks[:n], [n - 1]) for i, n in enumerate(lens)])
    assert rms_err(out, lg[[n - 1 for n in lens]]) < TOL[torch.float32]
    out = s.step([(i, toks[n:131], [130 - n]) for i, n in enumerate(lens)])
    assert rms_err(out, lg[[130] * len(lens)]) < TOL[torch.float32]


@pytest.mark.parametrize("dim,vdim,conv", [(32, 80, 1), (128, 48, 3), (64, 16, 6), (256, 32, 8), (48, 130, 9), (144, 32, 11), (128, 128, 4)])
def test_tokens_past_the_end_as_zeros_or_masked(dev, dim, vdim, conv):
    """what lies past a sequence's end in its last chunk, stored as zeros (few or long sequences) or not stored and masked (many short ones): the same bits in logits and
    states, whatever was in the workspace. Ends at every token of a lane's four, on both sides of 16 and of 32; together, one by itself, behind cached tokens"""
    from cogstream_amd import _lib as L
    cfg = config([delta(heads=4, kv_heads=2, dim=dim, vdim=vdim, conv=conv, ff=None)], width=64)
    e = engine(cfg, state(cfg), torch.float32)
    toks = tokens(cfg, 200)
    lens = [1, 2, 3, 4, 5, 7, 8, 9, 13, 15, 16, 17, 18, 21, 30, 31, 32, 33, 36, 48, 49, 63, 64, 65, 130]

    def results(poison):
        out = []
        for batch in (lens, [3], [65], [1, 64]):
            s = sequences(e)
            for parts in ((0, 1), (1, 2), (2, 3)):
                cut = [[0, n, n + 1 + n % 7, 150][k] for n in batch for k in range(4)]
                if poison:
                    e.handle.workspace("decoder", 1).fill_(255)
                out.append(s.step([(i, toks[cut[4 * i + parts[0]]:cut[4 * i + parts[1]]], [0]) for i in range(len(batch))]))
            out += [s.caches[i].state for i in range(len(batch))]
        return out
    want = results(False)
    assert all(torch.isfinite(x).all() for x in want)
    for form in (0, 1, 2):
        with L.debug_switch("delta_zeros", form):
            for poison in (False, True):
                assert all(torch.equal(a, b) for a, b in zip(results(poison), want)), (form, poison)


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_the_chunked_delta_rule_keeps_what_recurs(dev, dim):
    """a few (key, value) pairs that come again and again: the state already predicts every value, so what a chunk writes is the rounding of
    its own sums. Read back at the stored keys, against 64-bit arithmetic on the very same inputs, the chunked form must be as exact as the
    token-by-token one, and off by no more than its last write is: an entry of S is rounded by at most 2^-24 of itself, V - K S by at most
    half of that of V (measured 3.4e-8 to 6.8e-8; two terms of V's size that cancel 1.2e-7 to 1.9e-7). The inputs are exact: one-hot
    tokens, whole values (silu returns them as they are), beta and g equal to one; the keys come out of one-token states, in the column
    whose value is a power of two"""
    from cogstream_amd import _lib as L
    H, P, width, vdim = 4, 4, 64, 64
    cfg = config([delta(heads=H, kv_heads=2, dim=dim, vdim=vdim, conv=1, ff=None)], width=width, vocab=P, scale=1.0, streams=None, eps=1e-30)
    st = state(cfg)
    g = torch.Generator().manual_seed(dim)
    st["embed"].copy_(torch.eye(P, width))               # normed: 8 in one column
    st["pos"].zero_()
    st["l0.norm1"].fill_(1.0)
    for n in "qkv":
        st[f"l0.mix.{n}.conv"].fill_(1.0)
    st["l0.mix.k"].normal_(generator=g)
    values = torch.randint(18, 64, (H, vdim, P), generator=g).float()
    values[:, 0] = 32.0
    st["l0.mix.v"].zero_()[:, :P] = values.view(H * vdim, P) / 8
    st["l0.mix.b"].fill_(25.0)                           # sigmoid(200)
    st["l0.mix.A_log"].fill_(-100.0)
    e = engine(cfg, st, torch.float32)

    def state_of(toks):
        s = sequences(e)
        s.step([("r", toks, [])])
        return s.caches["r"].state[:H * dim * vdim].view(H, dim, vdim).cpu()

    keys = []
    for t in range(P):
        one = state_of([t])
        keys.append(one[:, :, 0] / 32)
        assert torch.equal(one, keys[-1][:, :, None] * values[:, None, :, t])
    toks = torch.randint(0, P, (500,), generator=g).tolist()
    exact = torch.zeros(H, dim, vdim, dtype=torch.float64)
    for t in toks:
        k, v = keys[t].double()[:, :, None], values[:, :, t].double()[:, None]
        exact += k * (v - (k * exact).sum(1, keepdim=True))
    at = torch.stack(keys, 1).double()
    want = at @ exact
    err = []
    for chunked in (1, 0):
        with L.debug_switch("delta_chunk", chunked):
            got = at @ state_of(toks).double()
        err.append(float((got - want).norm() / want.norm()))
    assert err[0] < err[1] and err[0] < 1.5 * 2.0 ** -24, err


@pytest.mark.parametrize("name", ["peaked", "mixed"])
def test_a_query_tile_by_one_wave_or_by_two(dev, name):
    """many prompts at once (each query tile's keys are one wave's) and few (every second key tile is another wave's): prompts that end
    at the edges of the 64-key tiles and of the 128-row tiles, from nothing and behind cached tokens, against the oracle"""
    cfg, st, e, toks, lg, _ = named(name, torch.bfloat16, 400)
    lens = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 257]
    for times in (1, 20):
        for cut in (0, 30):
            s = sequences(e)
            jobs = [(i, n) for i, n in enumerate(lens * times) if n > cut]
            if cut:
                s.step([(i, toks[:cut], []) for i, _ in jobs])
            out = s.step([(i, toks[cut:n], [n - 1 - cut]) for i, n in jobs])
            assert rms_err(out, lg[[n - 1 for _, n in jobs]]) < TOL[torch.bfloat16], (times, cut)


def test_unsupported_calls_are_refused(dev):
    from cogstream_amd import _lib as L
    cfg, st, e, toks, _, _ = named("peaked", torch.bfloat16)
    emb = e.embed_tokens(torch.tensor(toks[:4]))
    c = e.new_cache(8)
    for args in (([3], [e.new_cache(2)], []), ([1, 2], [c, c], []), ([3], [c], [3]), ([3], [c], [-1])):
        with pytest.raises(L.CogsError):
            e.forward_batch(emb[:3], *args)
    assert c.len == 0
    e.forward_batch(emb, [4], [c], [])
    c.reset(2)                                           # the state is that of four tokens
    with pytest.raises(L.CogsError):
        e.forward_batch(emb[:1], [1], [c], [])
    short = config([attention(heads=2), delta(heads=2)], width=64, positions=20)
    s = sequences(engine(short, state(short), torch.bfloat16))
    s.step([("r", tokens(short, 20), [])])
    with pytest.raises(L.CogsError):
        s.step([("r", [1], [0])])


# ------------------------------------------------------------------------------------------------ the framework's entry points
def _checkpoint(tmp_path, name):
    from cogstream_amd import checkpoint as ck
    cfg = CONFIGS[name]
    st = state(cfg)
    ck.save_decoder(str(tmp_path), public(cfg), st)
    return cfg, st


def test_greedy_generation_through_the_registry(dev, tmp_path):
    """AutoModelForCausalLM -> generate: one prompt, several unequal prompts in one batch, in groups, with an end token, and the
    single-sequence loop with its prefix cache, against the oracle's greedy continuation"""
    from cogstream_amd.auto import AutoModelForCausalLM
    from cogstream_amd.llm import PrefixKV
    cfg, st = _checkpoint(tmp_path, "peaked")
    m = AutoModelForCausalLM.from_pretrained(str(tmp_path), torch_dtype=torch.float32)
    assert type(m).__name__ == "LupanexForCausalLM"
    w = double(st)
    prompts = [tokens(cfg, n, seed=n) for n in (9, 1, 30, 66)]
    want = [lo.greedy(cfg, w, p, 8) for p in prompts]
    assert m.generate(prompts[0], max_new_tokens=8) == [want[0]]
    assert m.generate(torch.tensor(prompts[2]), max_new_tokens=8) == [want[2]]
    assert m.generate(prompts, max_new_tokens=8) == want
    assert m.generate(prompts, max_new_tokens=8, max_batch=3) == want
    stop = want[3][2]
    cut = [w[:w.index(stop) + 1] if stop in w else w for w in want]
    assert m.generate(prompts, max_new_tokens=8, eos_token_id=[stop]) == cut
    e = m.llm
    emb = e.embed_tokens(torch.tensor(prompts[3]))
    assert e.generate(emb, max_new_tokens=8) == want[3]
    # a state can stand behind the whole previous prompt, or start again
    pre = PrefixKV(e)
    assert e.generate(emb, max_new_tokens=8, prefix=pre) == want[3]
    longer = prompts[3] + tokens(cfg, 40, seed=5)
    assert e.generate(e.embed_tokens(torch.tensor(longer)), max_new_tokens=4, prefix=pre) == lo.greedy(cfg, w, longer, 4)
    assert pre.reused == 66
    other = longer[:80] + prompts[2]
    assert e.generate(e.embed_tokens(torch.tensor(other)), max_new_tokens=4, prefix=pre) == lo.greedy(cfg, w, other, 4)
    assert pre.reused == 66
    a = m.generate(prompts, max_new_tokens=6, do_sample=True, temperature=0.8, top_k=20, top_p=0.9, seed=3)
    assert a == m.generate(prompts, max_new_tokens=6, do_sample=True, temperature=0.8, top_k=20, top_p=0.9, seed=3)
    assert m.generate(prompts, max_new_tokens=8, do_sample=True, top_k=1) == want


def test_two_designs_share_a_handle(dev):
    """the handle keeps one decoder; engines of either design re-activate themselves, in turns and in either type"""
    import pabalix_models as pm
    from cogstream_amd.llm import DecoderEngine
    from cogstream_amd.pabalix import parse_config
    from oracle import pabalix as po
    a = named("peaked", torch.bfloat16)
    pc = pm.CONFIGS["plain"]
    pst = pm.state(pc)
    ptoks = pm.tokens(pc, 90)
    plg = po.forward(pc, double(pst), ptoks)[0]
    sa, sb = sequences(a[2]), sequences(DecoderEngine(pst, parse_config(pc), dtype=torch.float32, device="cuda:0"))
    for x, y in ((0, 60), (60, 61), (61, 90)):
        ra = sa.step([("r", a[3][x:y], list(range(y - x)))])
        rb = sb.step([("r", ptoks[x:y], list(range(y - x)))])
        assert rms_err(ra, a[4][x:y]) < TOL[torch.bfloat16] and rms_err(rb, plg[x:y]) < TOL[torch.float32]


def test_command_lines(dev, tmp_path):
    """python -m cogstream_amd.generate and bin/trace_run in processes of their own"""
    cfg, st = _checkpoint(tmp_path, "mixed")
    w = double(st)
    prompts = [tokens(cfg, n, seed=n) for n in (9, 30)]
    r = subprocess.run([sys.executable, "-m", "cogstream_amd.generate", "--model_path", str(tmp_path), "--dtype", "float32", "--max_new_tokens", "6",
                        "--greedy"] + [x for p in prompts for x in ("--prompt", ",".join(map(str, p)))], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [json.loads(x)["tokens"] for x in r.stdout.splitlines()] == [lo.greedy(cfg, w, p, 6) for p in prompts]
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
    la, lb = lo.forward(cfg, w, a)[0], lo.forward(cfg, w, b)[0]
    load = lambda n: torch.frombuffer(bytearray((out / f"{n}.f32").read_bytes()), dtype=torch.float32).view(-1, cfg["vocab"])
    assert rms_err(load(0), torch.stack([la[0], la[36], lb[23]])) < TOL[torch.float32]
    assert rms_err(load(7), la[38:39]) < TOL[torch.float32] and rms_err(load(8), lb[24:25]) < TOL[torch.float32]
