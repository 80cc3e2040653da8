"""The recurrences in blocks of 32 tokens (option rec.min) against the plain oracles and against the token by token scan: wkv and the delta rule (Vitudra), the delta rule with a decay
per channel (Keronex), at the edges of blocks, of the matrix cores' tiles and of the state's tiles; portions that continue a state; several requests of unequal length in one step; decays
of zero and products of decays that underflow inside a block; and without scratch.  fp32 storage, 1e-4 of the largest logit, as for these designs' other forms."""
import numpy as np
import pytest

import test_hip_keronex as tk
import test_hip_vitudra as tv

pytestmark = pytest.mark.gpu
HEADS = [(4, 5), (12, 16), (64, 17), (68, 64), (128, 33)]      # key and value channels
WIDE = [(128, 144), (128, 256), (64, 208)]                      # more columns than the preparation has threads: a second pass over them


def model(kind, dim, vdim, over=None, **kw):
    """(engine, tokens -> wanted logits, config) of two layers of the recurrence around a plain one"""
    if kind == "cdelta":
        cfg = tk.config([tk.cd(tk.dense(), dim=dim, vdim=vdim), tk.ret(), tk.cd(dim=dim, vdim=vdim, heads=2, kv_heads=2)])
        eng, w = tk.engine(cfg, "fp32", 3, over, **kw)
        return eng, lambda t: tk.want_of(cfg, w, t), cfg
    layers = ([tv.wkv(tv.ff(), heads=3, dim=dim), tv.attn(tv.ff()), tv.wkv(heads=2, dim=dim)] if kind == "wkv" else
              [tv.par(tv.ff(), right=dict(dim=dim, vdim=vdim)), tv.attn(tv.ff()), tv.par(right=dict(dim=dim, vdim=vdim, heads=2, kv_heads=1))])
    cfg = tv.config(layers)
    eng, w = tv.engine(cfg, "fp32", 3, over, **kw)
    return eng, lambda t: tv.want_of(cfg, w, t), cfg


def close(got, want, what=""):
    err = np.abs(got - want).max() / np.abs(want).max()
    assert err < 1e-4, f"{what}: {err:.3e}"


def by_portions(eng, rid, toks, sizes):
    got, at = [], 0
    for n in sizes:
        got.append(eng.step([(rid, toks[at:at + n], list(range(n)))]))
        at += n
    return np.concatenate(got)


@pytest.mark.parametrize("kind,dim,vdim", [(k, *h) for k in ("wkv", "delta", "cdelta") for h in HEADS + (WIDE if k != "wkv" else [])])
def test_blocks_equal_the_oracle_and_the_scan(kind, dim, vdim):
    """one portion over a few blocks, and the same tokens in portions that end in, on and behind a block's edge (a state that goes on, blocks of one token, tails of a block)"""
    eng, want_of, cfg = model(kind, dim, vdim)
    toks = tk.tokens(cfg, 131, seed=dim)
    want = want_of(toks)
    eng.model.set_option("rec.min", 0)
    scan = by_portions(eng, "a", toks, [131])
    eng.model.set_option("rec.min", 1)
    blocks = by_portions(eng, "b", toks, [131])
    close(scan, want, "scan")
    close(blocks, want, "blocks")
    assert not np.array_equal(scan, blocks)      # (another order of sums: both forms ran)
    close(by_portions(eng, "c", toks, [33, 31, 1, 2, 63, 1]), want, "portions")
    eng.close()


@pytest.mark.parametrize("kind", ["wkv", "delta", "cdelta"])
def test_requests_of_unequal_length_in_one_step(kind):
    eng, want_of, cfg = model(kind, 64, 64)
    eng.model.set_option("rec.min", 1)
    sizes = [1, 97, 32, 45]
    seqs = [tk.tokens(cfg, n + 40, seed=n) for n in sizes]
    first = eng.step([("r%d" % i, s[:n], list(range(n))) for i, (s, n) in enumerate(zip(seqs, sizes))])
    second = eng.step([("r%d" % i, s[n:], list(range(40))) for i, (s, n) in enumerate(zip(seqs, sizes))])
    at = 0
    for i, (s, n) in enumerate(zip(seqs, sizes)):
        want = want_of(s)
        close(first[at:at + n], want[:n], "first %d" % n)
        close(second[40 * i:40 * i + 40], want[n:], "second %d" % n)
        at += n
    eng.close()


@pytest.mark.parametrize("kind,dim,vdim", [("wkv", 132, 132), ("delta", 132, 16), ("delta", 64, 260), ("cdelta", 132, 16), ("cdelta", 64, 260), ("delta", 6, 16)])
def test_heads_beyond_the_blocks_take_the_scan(kind, dim, vdim):
    eng, want_of, cfg = model(kind, dim, vdim)
    toks = tk.tokens(cfg, 70, seed=5)
    got = []
    for least in (0, 1):
        eng.model.set_option("rec.min", least)
        got.append(by_portions(eng, "r%d" % least, toks, [70]))
    close(got[1], want_of(toks))
    assert np.array_equal(got[0], got[1])
    eng.close()


@pytest.mark.parametrize("kind,heads,dim,vdim", [("wkv", 17, 64, 64), ("wkv", 9, 128, 128), ("delta", 16, 64, 72), ("delta", 16, 128, 72), ("cdelta", 16, 64, 72), ("cdelta", 16, 128, 72)])
def test_more_workgroups_than_compute_units(kind, heads, dim, vdim):
    """four requests of one to ten blocks, odd and even counts, whose heads and columns are 272 to 320 workgroups, then all of them a second time from the states that they left"""
    if kind == "cdelta":
        cfg = tk.config([tk.cd(dim=dim, vdim=vdim, heads=heads, kv_heads=heads // 2)])
        eng, w = tk.engine(cfg, "fp32", 3)
        want_of = tk.want_of
    else:
        cfg = tv.config([tv.wkv(heads=heads, dim=dim) if kind == "wkv" else tv.par(right=dict(dim=dim, vdim=vdim, heads=heads, kv_heads=heads // 2))])
        eng, w = tv.engine(cfg, "fp32", 3)
        want_of = tv.want_of
    eng.model.set_option("rec.min", 1)
    sizes = [257, 64, 33, 320]
    seqs = [tk.tokens(cfg, 2 * n, seed=n) for n in sizes]
    halves = [eng.step([("r%d" % i, s[k * n:(k + 1) * n], list(range(n))) for i, (s, n) in enumerate(zip(seqs, sizes))]) for k in (0, 1)]
    at = 0
    for s, n in zip(seqs, sizes):
        close(np.concatenate([h[at:at + n] for h in halves]), want_of(cfg, w, s), "%d" % n)
        at += n
    eng.close()


@pytest.mark.parametrize("kind,heads,dim,sizes,blocks", [
    ("wkv", 16, 32, [96], False), ("wkv", 16, 32, [512], True), ("wkv", 16, 32, [130] * 8, False), ("wkv", 64, 32, [300] * 4, False), ("wkv", 8, 128, [300] * 2, True),
    ("delta", 16, 32, [512], True), ("delta", 32, 32, [300] * 8, False), ("delta", 16, 64, [192] * 8, False), ("delta", 4, 64, [300] * 4, True),
    ("cdelta", 16, 32, [200] * 16, False), ("cdelta", 8, 128, [512], True), ("cdelta", 8, 128, [200] * 16, False), ("cdelta", 8, 128, [700] + [3] * 7, True)])
def test_the_form_follows_the_step(kind, heads, dim, sizes, blocks):
    """steps of which one form takes at least a tenth less than the other: by themselves they take that one (its bits)"""
    kw = dict(max_seqs=16, max_ctx=1024, budget_tokens=8192)
    if kind == "cdelta":
        cfg = tk.config([tk.cd(dim=dim, vdim=dim, heads=heads, kv_heads=heads)])
        eng, _ = tk.engine(cfg, "fp32", 3, **kw)
    else:
        cfg = tv.config([tv.wkv(heads=heads, dim=dim) if kind == "wkv" else tv.par(right=dict(dim=dim, vdim=dim, heads=heads, kv_heads=heads // 2))])
        eng, _ = tv.engine(cfg, "fp32", 3, **kw)
    got = {}
    for least in (-1, 0, 1):
        eng.model.set_option("rec.min", least)
        got[least] = eng.step([(i, tk.tokens(cfg, n, i), [n // 2, n - 1]) for i, n in enumerate(sizes)], range(len(sizes)))
    eng.close()
    assert not np.array_equal(got[0], got[1])
    assert np.array_equal(got[-1], got[1 if blocks else 0])


@pytest.mark.parametrize("strength", [1.5, 3.0, 6.0])      # decays of 1e-2, 2e-9 (a block's product underflows) and zero a token
@pytest.mark.parametrize("kind", ["wkv", "delta", "cdelta"])
def test_strong_decays(kind, strength):
    names = {"wkv": ("l0.mix.w0",), "delta": ("l0.mix.right.A_log",), "cdelta": ("l0.mix.A_log",)}[kind]
    import keronex_oracle as ko
    import vitudra_oracle as vo
    eng, _, cfg = model(kind, 64, 32)
    w0 = (ko.random_tensors(cfg, 3, None, 5, 7) if kind == "cdelta" else vo.random_tensors(cfg, 3))
    eng.close()
    over = {}
    for n in names:
        v = w0[n].copy()
        v.reshape(-1)[::2] = strength      # every other channel or head keeps its own
        over[n] = v
    eng, want_of, cfg = model(kind, 64, 32, over)
    eng.model.set_option("rec.min", 1)
    toks = tk.tokens(cfg, 100, seed=9)
    close(by_portions(eng, "r", toks, [70, 30]), want_of(toks))
    eng.close()


@pytest.mark.parametrize("kind", ["wkv", "delta", "cdelta"])
def test_without_scratch_the_scan_takes_over(kind):
    eng, want_of, cfg = model(kind, 64, 64)
    toks = tk.tokens(cfg, 100, seed=2)
    eng.model.set_option("ssd.min", 0)      # (the retention between takes scratch of its own)
    eng.model.set_option("rec.min", 0)
    scan = by_portions(eng, "a", toks, [100])
    eng.model.set_option("stack.ws_max", 1)
    eng.model.set_option("rec.min", 1)
    assert np.array_equal(by_portions(eng, "b", toks, [100]), scan)
    eng.close()


@pytest.mark.parametrize("kind,dim,vdim", [("wkv", 64, 64), ("delta", 64, 64), ("delta", 128, 64), ("cdelta", 64, 64), ("cdelta", 128, 64)])
def test_blocks_round_no_more_than_the_scan(kind, dim, vdim):
    """the error against 64 bits of a model that is little else than the recurrence, over eight seeds of 300 tokens: no larger in blocks than token by token.  (The two forms' errors are
    sums over the same 160000 logits, and a seed's ratio lies within 0.03 of the mean: 0.97 to 1.00; with a pair's sum, the decays' products and the system's right-hand sides rounded at
    every step the delta rules' means were 1.02 to 1.04.)"""
    err = {0: 0.0, 1: 0.0}
    for seed in range(8):
        if kind == "cdelta":
            cfg = tk.config([tk.cd(dim=dim, vdim=vdim, heads=2, kv_heads=2)], streams=1, bigram=None, embed=0.1)
            eng, w = tk.engine(cfg, "fp32", seed)
            want_of = tk.want_of
        else:
            cfg = tv.config([tv.wkv(heads=2, dim=dim)] if kind == "wkv" else [tv.par(right=dict(dim=dim, vdim=vdim, heads=2, kv_heads=1), left_scale=0.0, right_scale=1.0)], mult=8.0)
            eng, w = tv.engine(cfg, "fp32", seed)
            want_of = tv.want_of
        toks = tk.tokens(cfg, 300, seed)
        want = want_of(cfg, w, toks)
        for blocks in (0, 1):
            eng.model.set_option("rec.min", blocks)
            got = eng.step([("r%d" % blocks, toks, list(range(300)))])
            err[blocks] += np.linalg.norm(got - want) / np.linalg.norm(want)
        eng.close()
    assert err[1] <= 1.01 * err[0], err
