"""The matrix products of layered models at the sizes where their forms change and their tiles end: rows of a step (one and two on the vector kernel, up to 64 on the
few-row kernel, beyond on the tiles), contraction lengths that are no multiple of a step of 64, column counts that are no multiple of sixteen, grouped expert
products with few and with many pairs.  fp32 storage against the plain oracle: nothing is rounded, so what remains is fp32 summation over at most 264 terms per
product through two layers (measured 1e-6; bound 2e-5 of the largest logit).  16-bit storage against the same sequences stepped one at a time: the cached latents may
round to the other neighbour (2^-9 for bf16, 2^-12 for fp16) where two sums of the same terms differ in their last bit; the bound is that of one such step,
and holds against the oracle as well (0.15 of it measured)."""
import numpy as np
import pytest

import modepel_oracle as mo
import stack_oracle as so
import test_hip_modepel as tm
import test_hip_vitudra as tv
import test_hip_zaluvik as tz
from tinygpt_amd.desc import LayerDesc, StackDesc
from tinygpt_amd.serving import SlotEngine

pytestmark = pytest.mark.gpu


def desc(width, dtype, slots, ff, vdim=5):
    layers = [LayerDesc(heads=3, dim=8, vdim=vdim, kv_rank=24, scale=0.35, mlp="moe", experts=5, top=2, ff=ff, limit=1.5),
              LayerDesc(heads=2, dim=16, vdim=16, kv_rank=16, scale=0.25, mlp="moe", experts=3, top=2, ff=ff + 16, limit=2.0)]
    return StackDesc(width=width, vocab=101, canon_taps=3, norm_groups=2, norm_eps=1e-6, logit_scale=0.5, max_seqs=slots, max_ctx=64, budget_tokens=64 * slots,
                     compute_dtype=dtype, layers=layers)


def both(d, tensors, seqs):
    """the sequences stepped together: first tokens, then a decoded token each; logits [seqs][2][vocab]"""
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in tensors.items()})
    got = [eng.step([(i, [s[t]], [0]) for i, s in enumerate(seqs)]) for t in range(2)]
    eng.close()
    return np.stack(got, 1)


# (width 72 and 264: a step of 64 and eight more; vdim 5 sends three layers' products to the tiles whose loads take any alignment)
@pytest.mark.parametrize("width,ff,vdim", [(72, 24, 8), (264, 40, 8), (128, 64, 8), (72, 24, 5)])
@pytest.mark.parametrize("slots", [1, 2, 3, 16, 17, 32, 33, 64, 65])
def test_rows_of_a_step(slots, width, ff, vdim):
    d = desc(width, "fp32", slots, ff, vdim)
    t = so.random_tensors(d, slots)
    rng = np.random.default_rng(slots)
    seqs = rng.integers(0, d.vocab, (slots, 2))
    got = both(d, t, seqs)
    for i in range(0, slots, max(1, slots // 9)):
        want = so.forward(d, t, seqs[i].tolist())
        assert np.abs(got[i] - want).max() / np.abs(want).max() < 2e-5, (slots, width, i)


# (where the few-row kernel brings another four rows of a tile; the bound above)
@pytest.mark.parametrize("width,ff", [(72, 24), (264, 40), (1024, 64)])
@pytest.mark.parametrize("slots", [4, 5, 7, 8, 9, 12])
def test_rows_of_a_tile(slots, width, ff):
    d = desc(width, "fp32", slots, ff, 8)
    t = so.random_tensors(d, slots)
    seqs = np.random.default_rng(slots).integers(0, d.vocab, (slots, 2))
    got = both(d, t, seqs)
    for i in range(slots):
        want = so.forward(d, t, seqs[i].tolist())
        assert np.abs(got[i] - want).max() / np.abs(want).max() < 2e-5, (slots, width, i)


@pytest.mark.parametrize("dtype,bound", [("bf16", 2.0 ** -8), ("fp16", 2.0 ** -11)])
@pytest.mark.parametrize("slots", [2, 3, 16, 33, 64, 65])
def test_rows_of_a_step_in_half_storage(slots, dtype, bound):
    d = desc(264, dtype, slots, 40, 8)
    t = so.random_tensors(d, 7 + slots)
    seqs = np.random.default_rng(slots).integers(0, d.vocab, (slots, 2))
    got = both(d, t, seqs)
    one = desc(264, dtype, 1, 40, 8)
    for i in range(0, slots, max(1, slots // 5)):
        want = both(one, t, seqs[i:i + 1])[0]
        assert np.abs(got[i] - want).max() / np.abs(want).max() < bound, (slots, dtype, i)
        want = so.forward(d, t, seqs[i].tolist())
        assert np.abs(got[i] - want).max() / np.abs(want).max() < bound, (slots, dtype, i)


# The few-row kernel's sums are as exact as the vector kernel's: sixteen rows together against one at a time, fp32 storage, a model that caches nothing, geometric means of the
# errors' ratio over ten models.  1.41 (standard error 0.05) with one chain over a wave's share of K, 1.05 (0.12) with a chain a level; the bound lies between.
def test_few_rows_are_as_exact_as_one():
    import vitudra_oracle as vo
    W, ff, rows, ratios = 1024, 512, 16, []
    for seed in range(10):
        cfg = dict(width=W, vocab=101, norm=dict(eps=1e-5), residual_mult=0.5, layers=[dict(type="wkv", mixer=dict(heads=W // 64, dim=64), mlp=dict(kind="dense", ff=ff))])
        t = vo.random_tensors(cfg, seed, decay_rank=64)
        d = StackDesc(family="vitudra", width=W, vocab=101, compute_dtype="fp32", max_seqs=rows, max_ctx=64, budget_tokens=64 * rows, norm_eps=1e-5, residual_mult=0.5,
                      layers=[LayerDesc(mixer="wkv", heads=W // 64, kv_heads=W // 64, dim=64, vdim=64, decay_rank=64, mlp="dense", ff=ff)])
        eng = SlotEngine(desc=d, tensors={k: np.asarray(v, np.float32) for k, v in t.items()})
        ids = np.random.default_rng(seed).permutation(101)[:rows]
        want = np.stack([vo.forward(cfg, t, [int(i)])[0] for i in ids])
        many = eng.step([(i, [x], [0]) for i, x in enumerate(ids)], range(rows))
        one = np.concatenate([eng.step([(0, [x], [0])], [0]) for x in ids])
        eng.close()
        ratios.append(np.linalg.norm(many - want) / np.linalg.norm(one - want))
    assert np.exp(np.log(ratios).mean()) < 1.25, ratios


# ---- prompts: the line kernels against the register-staged tiles ---------------------------------------------------------------------------
# Both forms multiply the same two 16-bit terms of an activation by the same stored weights; only the order of fp32 sums differs (5e-7 measured per product, 1e-4 allowed
# through two layers and a recurrence).  The wkv model caches nothing, so nothing rounds on the way; the expert model's cached latents may round to the other neighbour.
def wkv_model(W, ff, dtype, T):
    layers = [LayerDesc(mixer="wkv", heads=W // 64, kv_heads=W // 64, dim=64, vdim=64, decay_rank=64, mlp="dense", ff=ff) for _ in range(2)]
    return StackDesc(family="vitudra", width=W, vocab=101, compute_dtype=dtype, max_seqs=1, max_ctx=T, budget_tokens=T, norm_eps=1e-5, residual_mult=0.5, layers=layers)


# What the second terms are worth: without them (act.round16) a row of logits moves by 1.5e-4 (wkv; experts 3e-5) in fp16 and ten times that in bf16 at least.  With them the two
# forms differ by fp32 sums and by second terms that round to the other neighbour, 2^-17 of an activation in bf16 and 2^-23 in fp16: a median row by 2.5e-6 and 2.8e-7 at most
# (measured), 2^-16 and 2^-20 allowed.  Single terms round the same inputs, which differ in their last bits, so their roundings part from layer to layer and only the distance that
# they bring can be compared: that of one form's median row against the other's (0.92 to 1.07 measured), two thirds to three halves.
MEDIAN = {"bf16": 2.0 ** -16, "fp16": 2.0 ** -20}


def on_and_off(eng, ids, want, dtype):
    """a prompt's logits by the line kernels and by the tiles, both terms of an activation; single terms are compared on the way"""
    out = {}
    for one in (0, 1):
        eng.model.set_option("act.round16", one)
        for line in (1, 0):
            eng.model.set_option("stack.line", line)
            out[line, one] = eng.step([("p", ids, want)], ["p"]).astype(np.float64)
    eng.close()
    assert all(np.isfinite(x).all() for x in out.values())
    away = lambda x, y: np.median(np.abs(out[x] - out[y]).max(1) / np.abs(out[y]).max())      # noqa: E731
    assert 0 < away((1, 0), (0, 0)) < MEDIAN[dtype], away((1, 0), (0, 0))
    ratio = away((1, 1), (1, 0)) / away((0, 1), (0, 0))
    assert 2 / 3 < ratio < 3 / 2, ratio
    return out[1, 0], out[0, 0]


# (T 2177: 18 row tiles of 128, the last of one row; 4161: 256-row tiles, the last of 65; ff 1088 = 17 x 64: column tiles that end inside; width 320: five steps of K)
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("W,ff,T", [(320, 1088, 2177), (320, 1088, 4161), (256, 1024, 2048), (320, 64, 8200)])
def test_prompt_products_of_a_model_that_caches_nothing(W, ff, T, dtype):
    import vitudra_oracle as vo
    d = wkv_model(W, ff, dtype, T)
    rng = np.random.default_rng(T)
    cfg = dict(width=W, vocab=101, layers=[dict(type="wkv", mixer=dict(heads=W // 64, dim=64), mlp=dict(ff=ff))] * 2)
    t = vo.random_tensors(cfg, 3, decay_rank=64)
    want = sorted({0, 1, 63, 64, 127, 128, 255, 256, T // 2, T - 66, T - 2, T - 1})
    eng = SlotEngine(desc=d, tensors={k: np.asarray(v, np.float32) for k, v in t.items()})
    on, off = on_and_off(eng, rng.integers(0, d.vocab, T), want, dtype)
    assert np.abs(on - off).max() / np.abs(off).max() < 1e-4, (W, ff, T, dtype)


# a near tie of the router may send a token to another expert, and a cached latent may round to the other neighbour: one row in sixteen may go beyond the bound of such a step
@pytest.mark.parametrize("dtype,bound", [("bf16", 2.0 ** -7), ("fp16", 2.0 ** -10)])
@pytest.mark.parametrize("T,experts,top,ff,kv_rank", [(2100, 5, 2, 192, 128), (4000, 3, 3, 1024, 128), (1537, 9, 4, 320, 128), (2100, 5, 2, 192, 256), (4100, 3, 2, 512, 320)])
def test_prompt_products_of_experts(T, experts, top, ff, kv_rank, dtype, bound):
    """kv_rank from 256 on: the gated products of every head's latents take the line kernels too"""
    layers = [LayerDesc(heads=4, dim=64, vdim=64, kv_rank=kv_rank, scale=0.125, mlp="moe", experts=experts, top=top, ff=ff, limit=7.0) for _ in range(2)]
    d = StackDesc(width=256, vocab=101, canon_taps=3, norm_groups=2, norm_eps=1e-6, max_seqs=1, max_ctx=T, budget_tokens=T, compute_dtype=dtype, layers=layers)
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in so.random_tensors(d, T).items()})
    on, off = on_and_off(eng, np.random.default_rng(T).integers(0, d.vocab, T), sorted({*range(0, T, 33), 127, 128, T // 2, T - 1}), dtype)
    rows = np.abs(on - off).max(1) / np.abs(off).max()
    assert np.quantile(rows, 15 / 16) < bound, (T, dtype, rows)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("T,experts,top,ff,shared", [(1100, 4, 2, 512, 512), (2100, 9, 3, 320, 64), (1500, 3, 1, 1024, 0)])
def test_prompt_products_of_experts_weighted_at_their_input(T, experts, top, ff, shared, dtype):
    """gathered products with a weight a row and an activation in the epilogue; retention caches nothing, so only a router's near tie goes beyond 1e-4"""
    import test_hip_keronex as tk
    layer = tk.ret(tk.moe(experts, top, ff, shared), heads=4, dim=32, vdim=64, decay=[0.875, 0.99, 0.5, 0.9])
    cfg = tk.config([layer, layer], width=256)
    eng, _ = tk.engine(cfg, dtype, max_seqs=1, max_ctx=T, budget_tokens=T + 64)
    on, off = on_and_off(eng, np.array(tk.tokens(cfg, T)), sorted({*range(0, T, 17), 127, 128, T - 1}), dtype)
    rows = np.abs(on - off).max(1) / np.abs(off).max()
    assert np.quantile(rows, 15 / 16) < 1e-4, (T, dtype, rows)


# The steps of a stage keep sums of their own on the 128 x 128 tiles too (tests/test_hip_prefill.py has the same of the flat families' kernel): every token the same row of one value, the
# head's rows a large number in step 0 of a stage, its negative in step 2, small ones in steps 1 and 3
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_steps_of_a_stage_keep_their_own_sums(dtype):
    W, V, T = 1024, 4096, 300
    rng = np.random.default_rng(4)
    d = wkv_model(W, 64, dtype, T)
    d.vocab = V
    w = {n: np.zeros(s, np.float32) for n, s in d.tensor_shapes().items()}
    w["embed"][:] = 1
    head = rng.integers(-8, 9, (V, W)) / 8
    k = np.arange(W) % 64
    head[:, (k < 16) | ((k >= 32) & (k < 48))] = 0
    head[:, k == 0], head[:, k == 32] = 2.0 ** 15, -2.0 ** 15
    w["head"][:] = head
    eng = SlotEngine(desc=d, tensors=w)
    got = eng.step([("p", rng.integers(0, V, T), list(range(T)))], ["p"])
    eng.close()
    want = head.sum(1) / np.sqrt(1 + 1e-5)
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-5


# Tiles of a last, at most half full round as two halves of K (line_plan.h): width 1024, 6208 hidden values and 1700 tokens halve 87 tiles of 256 x 256 (16 steps of K; rows that end
# inside) and 112 of 128 x 128 (97 steps: uneven halves).  Against whole tiles only the order of fp32 sums differs
# (1e-4 as above); a pass repeats itself bit for bit, whichever half comes first.
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("T", [1700, 1537])
def test_halved_tiles(T, dtype):
    import vitudra_oracle as vo
    W, ff = 1024, 6208
    cfg = dict(width=W, vocab=101, layers=[dict(type="wkv", mixer=dict(heads=W // 64, dim=64), mlp=dict(ff=ff))] * 2)
    eng = SlotEngine(desc=wkv_model(W, ff, dtype, T), tensors={k: np.asarray(v, np.float32) for k, v in vo.random_tensors(cfg, 3, decay_rank=64).items()})
    ids, want = np.random.default_rng(T).integers(0, 101, T), [0, 127, 128, 255, 256, T - 2, T - 1]
    halved = [eng.step([("p", ids, want)], ["p"]) for _ in range(3)]
    eng.model.set_option("stack.line_share", 0)
    whole = eng.step([("p", ids, want)], ["p"])
    eng.model.set_option("stack.line_share", 1)
    eng.model.set_option("stack.ws_max", 32 * 1024)      # (enough for the rows' terms and for halves of 128 x 128, not for halves of 256 x 256)
    some = [eng.step([("p", ids, want)], ["p"]) for _ in range(2)]
    eng.model.set_option("stack.line", 0)
    plain = eng.step([("p", ids, want)], ["p"])
    eng.close()
    assert (some[0] == some[1]).all() and not (some[0] == whole).all() and not (some[0] == halved[0]).all()
    assert np.abs(some[0] - whole).max() / np.abs(whole).max() < 1e-4, (T, dtype)
    assert (halved[0] == halved[1]).all() and (halved[0] == halved[2]).all() and not (halved[0] == whole).all()
    for other in (whole, plain):
        assert np.abs(halved[0] - other).max() / np.abs(other).max() < 1e-4, (T, dtype)


def test_memory_of_halved_tiles():
    """taken once, in front of a context's first step of more than 64 rows and of the size that its steps can come to need; where it is not to be had every tile is whole, and the next step asks
    again"""
    import vitudra_oracle as vo
    W, ff, T = 1024, 6208, 1700
    cfg = dict(width=W, vocab=101, layers=[dict(type="wkv", mixer=dict(heads=W // 64, dim=64), mlp=dict(ff=ff))] * 2)
    w = {k: np.asarray(v, np.float32) for k, v in vo.random_tensors(cfg, 3, decay_rank=64).items()}
    ids, want = np.random.default_rng(T).integers(0, 101, T), [0, 255, T - 1]

    def engine(**options):
        eng = SlotEngine(desc=wkv_model(W, ff, "bf16", T), tensors=w)
        for k, v in options.items():
            eng.model.set_option("stack." + k, v)
        return eng

    eng = engine()
    held = lambda: eng.model.get_option("stack.line_share_kib")      # noqa: E731
    eng.step([("p", ids[:64], [63])], ["p"])
    assert held() == 0
    halved = eng.step([("p", ids, want)], ["p"])
    kib, grown = held(), eng.model.get_option("stack.ws_grown")
    assert kib % 128 <= 1 and kib >= 128 * 200      # (128 KiB and a number a compute unit)
    assert (eng.step([("p", ids, want)], ["p"]) == halved).all() and (held(), eng.model.get_option("stack.ws_grown")) == (kib, grown)
    eng.close()
    got = []
    for line_share in (0, 1):
        eng = engine(line_share=line_share, ws_max=8 * 1024 - 1)      # (neither tile's halves fit; the rows' terms do not either, so that products go through the staged tiles)
        got.append(eng.step([("p", ids, want)], ["p"]))
        assert held() == 0
        if line_share:
            eng.model.set_option("stack.ws_max", -1)
            assert (eng.step([("p", ids, want)], ["p"]) == halved).all() and held() == kib
        eng.close()
    assert (got[0] == got[1]).all()
    eng = engine(ws_max=32 * 1024)      # (halves of 128 x 128 alone)
    some = eng.step([("p", ids, want)], ["p"])
    assert 0 < held() < kib and not (some == halved).all()
    eng.model.set_option("stack.ws_max", -1)
    assert (eng.step([("p", ids, want)], ["p"]) == halved).all() and held() == kib
    eng.close()


# ... and experts' tiles stay whole: their rows stand in any order (the plan takes them as they come), so that a row that is summed in halves in one pass would be summed whole in the next
@pytest.mark.parametrize("T,experts,top", [(2100, 5, 2), (700, 3, 1)])
def test_experts_tiles_stay_whole(T, experts, top):
    import test_hip_keronex as tk
    layer = tk.ret(tk.moe(experts, top, 2112, 2112), heads=4, dim=32, vdim=64, decay=[0.875, 0.99, 0.5, 0.9])
    cfg = tk.config([layer, layer], width=1024)
    eng, _ = tk.engine(cfg, "bf16", max_seqs=1, max_ctx=T, budget_tokens=T + 64)
    ids, want = np.array(tk.tokens(cfg, T)), sorted({*range(0, T, 17), 127, 128, T - 1})
    passes = [eng.step([("p", ids, want)], ["p"]) for _ in range(3)]
    eng.model.set_option("stack.line_share", 0)
    whole = eng.step([("p", ids, want)], ["p"])
    eng.close()
    assert all((p == whole).all() for p in passes)


@pytest.mark.parametrize("vocab", [53, 96, 1028, 1030])
def test_wanted_logits_reach_their_slots(vocab):
    """a step's last wanted logits are its slots' current logits (bit for bit) and their argmax is what the greedy pick starts from; slots whose last place is not wanted keep theirs"""
    d = StackDesc(width=72, vocab=vocab, canon_taps=2, norm_groups=2, norm_eps=1e-6, max_seqs=5, max_ctx=64, budget_tokens=320, compute_dtype="fp32",
                  layers=[LayerDesc(heads=2, dim=8, vdim=8, kv_rank=8, scale=0.35, mlp=None)])
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in so.random_tensors(d, vocab).items()})
    ids = np.random.default_rng(vocab).integers(0, vocab, 64)
    first = eng.step([(i, ids[5 * i:5 * i + 3 + i], [2 + i]) for i in range(4)])
    slot = [eng.slot_of[i] for i in range(4)]
    assert (eng.model.logits(rounded=False)[slot] == first).all()
    assert [eng.model.sample_row(s) for s in slot] == first.argmax(1).tolist()
    second = eng.step([(2, ids[:3], [0, 2]), (0, ids[3:5], [0]), (3, ids[5:6], [0])])      # request 0's last place is not wanted
    now = eng.model.logits(rounded=False)
    assert (now[slot[2]] == second[1]).all() and (now[slot[3]] == second[3]).all() and (now[slot[0]] == first[0]).all() and (now[slot[1]] == first[1]).all()
    assert eng.model.sample_row(slot[2]) == int(second[1].argmax()) and eng.model.sample_row(slot[3]) == int(second[3].argmax())
    eng.close()


# ---- the recurrences' scan: sixteen row groups (few workgroups, rows in vectors of four), eight, and rows of any length number by number; 64 rows a group and their
# remainders.  fp32 storage against the plain oracle: fp32 sums over at most 196 rows and 64 steps; 1e-4 of the largest logit as in the design's own tests.
@pytest.mark.parametrize("dim", [4, 12, 36, 60, 64, 68, 100, 128, 132, 196, 6, 70, 129])
@pytest.mark.parametrize("entries", [1, 40])
def test_scan_of_the_recurrences(dim, entries):
    cfg = tv.config([tv.wkv(heads=2, dim=dim), tv.par(right={"heads": 4, "kv_heads": 2, "dim": dim, "vdim": 36})], width=20)
    eng, w = tv.engine(cfg, seed=dim, max_seqs=entries, max_ctx=128, budget_tokens=64 * entries)
    seqs = [tv.tokens(cfg, 64 - i, seed=i) for i in range(entries)]
    got = [eng.step([(i, s[:24], [23]) for i, s in enumerate(seqs)]), eng.step([(i, s[24:], [len(s) - 25]) for i, s in enumerate(seqs)])]
    eng.close()
    for i in {0, entries // 2}:
        want = tv.want_of(cfg, w, seqs[i])
        for at, part in ((23, got[0]), (-1, got[1])):
            assert np.abs(part[i] - want[at]).max() / np.abs(want).max() < 1e-4, (dim, entries, i, at)


# ---- matrix memories in blocks (portions from 64 tokens): remainders of a block, of a portion of the gate scan (1024 tokens), of the state's and the values' tiles; then a
# second portion and single tokens that carry both states on.  fp32 storage against the plain oracle: fp32 sums over at most 256 channels and 64 tokens, an order of
# magnitude below the 1e-4 of the largest logit that the design's own tests allow.
@pytest.mark.parametrize("dim,vdim", [(4, 8), (32, 33), (36, 32), (132, 6), (256, 40)])
@pytest.mark.parametrize("n", [64, 65, 127, 192, 1023, 1025, 2050])
def test_matrix_memory_in_blocks(n, dim, vdim):
    cfg = tm.config([tm.rec(heads=3, dim=dim, vdim=vdim), tm.rec(heads=2, dim=dim, vdim=vdim, gate_cap=4.0)], width=20)
    eng, w = tm.engine(cfg, seed=n, max_seqs=2, max_ctx=4096, budget_tokens=8192)
    tok = [np.random.default_rng(n + i).integers(0, cfg["vocab"], n + 70).tolist() for i in range(2)]
    at = sorted({0, 63, n // 2, n - 1})
    got = [eng.step([(0, tok[0][:n], at), (1, tok[1][:3], [2])]), eng.step([(1, tok[1][3:n], [n - 4]), (0, tok[0][n:n + 68], [67])]),
           eng.step([(0, tok[0][n + 68:n + 69], [0]), (1, tok[1][n:n + 1], [0])])]
    eng.close()
    want = [mo.forward(cfg, w, t[:n + 69])[0] for t in tok]
    for i, rows, pos in ((0, got[0][:len(at)], at), (1, got[0][len(at):], [2]), (1, got[1][:1], [n - 1]), (0, got[1][1:], [n + 67]), (0, got[2][:1], [n + 68]), (1, got[2][1:], [n])):
        assert np.abs(rows - want[i][pos]).max() / np.abs(want[i]).max() < 1e-4, (n, dim, vdim, i, pos)


# The blocks' error against 64 bits is no larger than the scan's.  Geometric means over 16 models, fp32 storage: with one sum over a row's channels in the blocks' key products it
# was 1.02 times (128 channels) and 1.06 times (256) the scan's, with eight sums 0.96 (standard errors 0.005 and 0.013).
@pytest.mark.parametrize("heads,dim,vdim,n", [(2, 128, 64, 700), (1, 256, 256, 500)])
def test_matrix_memory_in_blocks_is_as_exact_as_the_scan(heads, dim, vdim, n):
    cfg = tm.config([tm.rec(heads=heads, dim=dim, vdim=vdim), tm.rec(heads=heads, dim=dim, vdim=vdim)], width=64)
    ratios = []
    for seed in range(16):
        eng, w = tm.engine(cfg, seed=seed, max_ctx=4096, budget_tokens=4096)
        ids = np.random.default_rng(seed).integers(0, cfg["vocab"], n).tolist()
        want = mo.forward(cfg, w, ids)[0]
        err = []
        for least in (64, 0):
            eng.model.set_option("ssd.min", least)
            err.append(np.linalg.norm(eng.step([("p", ids, list(range(n)))], ["p"]) - want))
        eng.close()
        ratios.append(err[0] / err[1])
    assert np.exp(np.log(ratios).mean()) <= 1.0, ratios


# ---- seams and norms: rows of one, two and four vectors a thread, widths that are no multiple of four, and widths past the registers; taps by number and by name.
# fp32 storage against the plain oracles of the designs: fp32 sums over at most 4100 channels, 1e-4 of the largest logit as in the designs' own tests.
@pytest.mark.parametrize("width", [1024, 1028, 1030, 2044, 2052, 4096, 4100])
@pytest.mark.parametrize("design", ["modepel", "zaluvik", "vitudra"])
def test_seams_of_wide_rows(design, width):
    t, layers = {"modepel": (tm, [tm.rec(tm.moe()), tm.attn(tm.dense())]), "zaluvik": (tz, [tz.attn(tz.moe()), tz.lat(tz.dense())]), "vitudra": (tv, [tv.wkv(tv.ff()), tv.attn()])}[design]
    cfg = t.config(layers, width=width)
    eng, w = t.engine(cfg, seed=width)
    toks = t.tokens(cfg, 5, seed=width)
    got = t.run_whole(eng, "a", toks)
    eng.close()
    t.check(got, t.want_of(cfg, w, toks), "fp32", f"{design} {width}")


@pytest.mark.parametrize("width,groups", [(1024, 2), (1032, 6), (1036, 7), (1030, 5)])
@pytest.mark.parametrize("taps", [1, 2, 4, 5, 8])
def test_norm_and_convolution_of_wide_rows(taps, width, groups):
    layers = [LayerDesc(heads=3, dim=8, vdim=8, kv_rank=24, scale=0.35, mlp="moe", experts=5, top=2, ff=24, limit=1.5)]
    d = StackDesc(width=width, vocab=53, canon_taps=taps, norm_groups=groups, norm_eps=1e-6, max_seqs=2, max_ctx=64, budget_tokens=128, compute_dtype="fp32", layers=layers)
    t = so.random_tensors(d, taps)
    toks = np.random.default_rng(taps).integers(0, 53, 14).tolist()
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    got = np.concatenate([eng.step([("a", toks[lo:hi], list(range(hi - lo)))]) for lo, hi in ((0, 2), (2, 3), (3, 12), (12, 14))])
    eng.close()
    want = so.forward(d, t, toks)
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-4, (taps, width)


# ---- layers whose mixer and feed-forward share a decode step's launches (one and two rows, whole slices of eight): against the plain oracle, fp32 sums over at most 320
# channels (1e-4 of the largest logit as in the design's own tests), and against the same step with each product launched by itself.
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("width,ffn,dim", [(64, 40, 8), (72, 1096, 24), (520, 24, 16)])
@pytest.mark.parametrize("rows", [1, 2, 3])
def test_merged_products_of_a_step(rows, width, ffn, dim, dtype):
    layers = [tv.wkv(tv.ff(ffn), heads=4, dim=dim), tv.par(tv.ff(ffn), left={"heads": 4, "kv_heads": 2, "dim": dim, "vdim": dim + 8, "rot": {"base": 300.0, "dims": 4}}, right={"heads": 4, "kv_heads": 2, "dim": dim, "vdim": 8}),
              tv.attn(tv.ff(ffn), heads=4, kv_heads=2, dim=dim, vdim=dim), tv.attn(), tv.wkv()]
    cfg = tv.config(layers, width=width)
    eng, w = tv.engine(cfg, dtype, seed=width)
    toks = [tv.tokens(cfg, 6, seed=i) for i in range(rows)]
    out = []
    for on in (1, 0):
        eng.model.set_option("stack.gemv", on)
        out.append(np.stack([eng.step([((on, i), [toks[i][t]], [0]) for i in range(rows)], [(on, i) for i in range(rows)] if t == 5 else []) for t in range(6)], 1))
    eng.close()
    for i in range(rows):
        want = tv.want_of(cfg, w, toks[i])
        tv.check(out[0][i], want, "fp32" if dtype == "fp32" else "bf16", f"{rows} rows, row {i}")
        tv.check(out[1][i], want, "fp32" if dtype == "fp32" else "bf16", f"{rows} rows, row {i}, apart")


# ---- choice kernels that take the router's products themselves (up to 64 rows and 64 products): widths around a wave's 256 channels a load, expert counts around the four
# of a wave's pass, beside the step of one row more that takes the general products.  fp32 storage against the plain oracles: 1e-4 of the largest logit as above.
@pytest.mark.parametrize("width", [8, 252, 260, 1028])
@pytest.mark.parametrize("experts,identity", [(3, 1), (13, 2), (62, 2), (63, 3)])
@pytest.mark.parametrize("rows", [1, 64, 65])
def test_router_products_in_the_choice(rows, experts, identity, width):
    cfg = tm.config([tm.attn(tm.moe(experts=experts, identity=identity, top=3, count=1, keep=1))], width=width)
    eng, w = tm.engine(cfg, seed=experts + width)
    toks = tm.tokens(cfg, rows, seed=rows)
    got = tm.run_whole(eng, "a", toks)
    eng.close()
    tm.check(got, tm.want_of(cfg, w, toks), "fp32", f"{rows} rows")


@pytest.mark.parametrize("experts", [2, 5, 16, 17, 64, 65])
@pytest.mark.parametrize("rows", [1, 63, 64, 65])
def test_router_products_in_the_biased_choice(rows, experts):
    layers = [LayerDesc(heads=3, dim=8, vdim=8, kv_rank=24, scale=0.35, mlp="moe", experts=experts, top=2, ff=24, limit=1.5)]
    d = StackDesc(width=76, vocab=53, canon_taps=2, norm_groups=2, norm_eps=1e-6, max_seqs=2, max_ctx=128, budget_tokens=256, compute_dtype="fp32", layers=layers)
    t = so.random_tensors(d, experts)
    toks = np.random.default_rng(rows).integers(0, 53, rows).tolist()
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    got = eng.step([("a", toks, list(range(rows)))])
    eng.close()
    want = so.forward(d, t, toks)
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-4, (rows, experts)


# ---- products over a step's (token, expert) pairs (up to 128): fewer pairs than experts and more, experts of one to 64 rows (tiles of four and eight), contraction lengths around
# the chunk of 128 and below it, column counts that end inside a workgroup's; more than six rows an expert on average take a plan and tiles of sixteen rows, one pair more than 128
# the other planned tiles.  fp32 storage against the plain oracle: fp32 sums over
# at most 1032 terms, 1e-4 of the largest logit as above.
@pytest.mark.parametrize("width,ff", [(8, 24), (136, 8), (1032, 520), (264, 1032)])
@pytest.mark.parametrize("rows,experts,top", [(1, 12, 3), (1, 2, 2), (9, 40, 2), (64, 3, 2), (25, 5, 5), (65, 3, 2), (33, 2, 1), (24, 8, 2), (25, 8, 2), (64, 11, 1), (64, 22, 2), (65, 22, 2)])
def test_products_of_pairs(rows, experts, top, width, ff):
    layers = [LayerDesc(heads=3, dim=8, vdim=8, kv_rank=24, scale=0.35, mlp="moe", experts=experts, top=top, ff=ff, limit=1.5) for _ in range(2)]
    d = StackDesc(width=width, vocab=53, canon_taps=2, norm_groups=2, norm_eps=1e-6, max_seqs=2, max_ctx=128, budget_tokens=256, compute_dtype="fp32", layers=layers)
    t = so.random_tensors(d, experts)
    toks = np.random.default_rng(rows).integers(0, 53, rows).tolist()
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    got = eng.step([("a", toks, list(range(rows)))])
    eng.close()
    want = so.forward(d, t, toks)
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-4, (rows, experts, width)


# ---- norms that write the next products' terms themselves: the same two terms as the split in front of each product, so the same bits.  A limit on scratch that holds every product's
# own terms and hidden rows, but not a norm's lines beside them, leaves the split.  (T 4161: 33 row tiles, the last of one row; widths of one line, five and sixteen)
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("width", [64, 320, 1024])
@pytest.mark.parametrize("design", ["vitudra", "nusovik"])
def test_terms_of_a_norm(design, width, dtype):
    import test_hip_nusovik as tn
    T, ff = 4161, 1344
    heads = dict(heads=8, kv_heads=4, dim=32, vdim=32)
    half = dict(heads=4, kv_heads=2, dim=32, vdim=32)
    t, layers = {"vitudra": (tv, [tv.par(tv.ff(ff), left=heads, right=half), tv.wkv(tv.ff(ff), heads=2, dim=32), tv.attn(tv.ff(ff), **heads), tv.attn()]),
                 "nusovik": (tn, [tn.mamba(tn.ff(ff), inner=256), tn.par(tn.ff(ff), left=heads, right=dict(heads=4, state=32, vdim=32)), tn.par(left=heads), tn.mamba(inner=256)])}[design]
    cfg = t.config(layers, width=width)
    eng, _ = t.engine(cfg, dtype, max_seqs=1, max_ctx=T, budget_tokens=T + 64)
    ids, want, got = np.array(t.tokens(cfg, T)), [0, 63, 64, 127, 128, 2000, T - 2, T - 1], []
    for limit in (T * 4 * (max(ff, 4 * width) + width // 2) // 1024, -1):
        eng.model.set_option("stack.ws_max", limit)
        got.append(eng.step([("p", ids, want)], ["p"]))
    eng.close()
    assert np.isfinite(got[0]).all() and (got[0] == got[1]).all()


@pytest.mark.parametrize("dim,vdim", [(16, 16), (128, 40), (136, 33)])      # one and two tiles of state rows, ragged columns
@pytest.mark.parametrize("sizes", [[384, 5], [385, 193, 64, 1], [700, 320], [320, 129]])      # portions of two blocks and more: whole and ragged ones, an entry of one portion, none at all
@pytest.mark.parametrize("design", ["modepel", "keronex"])
def test_scalar_decay_in_portions(design, sizes, dim, vdim):
    """long entries' blocks in portions that run side by side, from the start of a sequence and from a state that it left, against the recurrence token by token (fp32 both)"""
    if design == "modepel":
        t, cfg = tm, tm.config([tm.rec(heads=2, dim=dim, vdim=vdim)], width=64)
    else:
        import test_hip_keronex as tk
        t, cfg = tk, tk.config([tk.ret(heads=2, dim=dim, vdim=vdim, decay=[0.9, 0.99], rot=None)], width=64)
    got = {}
    for least in (64, 0):
        eng, w = t.engine(cfg, seed=3, max_seqs=len(sizes), max_ctx=2048, budget_tokens=4096)
        eng.model.set_option("ssd.min", least)
        out = []
        for step in range(2):      # (the second in reverse: the longest entry is not the first)
            ids = list(range(len(sizes)))[::-1 if step else 1]
            out.append(eng.step([("s%d" % i, t.tokens(cfg, sizes[i], 10 * step + i), [0, sizes[i] // 2, sizes[i] - 1]) for i in ids]))
        out.append(eng.step([("s%d" % i, t.tokens(cfg, 1, i), [0]) for i in range(len(sizes))]))
        got[least] = np.concatenate(out)
        eng.close()
    assert np.abs(got[64] - got[0]).max() / np.abs(got[0]).max() < 1e-4


@pytest.mark.parametrize("heads,vdim,sizes", [(8, 256, [400] * 4), (8, 320, [500, 70]), (8, 320, [448, 70]), (40, 128, [500]), (40, 128, [448])])      # room for two portions, and for three or four
def test_portions_only_where_they_pay(heads, vdim, sizes):
    """entries whose portions would be too few, and as many as are enough, against the recurrence token by token (fp32 both)"""
    import test_hip_keronex as tk
    cfg = tk.config([tk.ret(heads=heads, dim=128, vdim=vdim, decay=[0.9, 0.99] * (heads // 2), rot=None)], width=64)
    got = {}
    for least in (64, 0):
        eng, w = tk.engine(cfg, seed=3, max_seqs=len(sizes), max_ctx=2048, budget_tokens=4096)
        eng.model.set_option("ssd.min", least)
        out = [eng.step([("s%d" % i, tk.tokens(cfg, n, 10 * step + i), [0, n // 2, n - 1]) for i, n in enumerate(sizes)]) for step in range(2)]
        got[least] = np.concatenate(out)
        eng.close()
    assert np.abs(got[64] - got[0]).max() / np.abs(got[0]).max() < 1e-4


@pytest.mark.parametrize("slots", [64, 65])
def test_order_of_many_entries(slots):
    """blocks that more than fill the chip (576 workgroups) take up to 64 entries longest first and more as they stand: entries of equal and unequal length, every request's outputs and the state it leaves, against the scan"""
    import test_hip_keronex as tk
    cfg = tk.config([tk.ret(heads=9, dim=16, vdim=16, decay=[0.9, 0.99, 0.8] * 3, rot=None)], width=64)
    got = {}
    for least in (1, 0):
        eng, w = tk.engine(cfg, seed=3, max_seqs=slots, max_ctx=256, budget_tokens=256 * slots)
        eng.model.set_option("ssd.min", least)
        out = []
        for step in range(2):
            sizes = [[5, 70, 5, 64, 129, 1, 70][(i + step) % 7] for i in range(slots)]
            out.append(eng.step([("s%d" % i, tk.tokens(cfg, n, 100 * step + i), [0, n // 2, n - 1]) for i, n in enumerate(sizes)]))
        out.append(eng.step([("s%d" % i, tk.tokens(cfg, 1, i), [0]) for i in range(slots)]))
        got[least] = np.concatenate(out)
        eng.close()
    assert np.abs(got[1] - got[0]).max() / np.abs(got[0]).max() < 1e-4
    assert not np.array_equal(got[1], got[0])      # (both forms ran)


# The scan's, the filter's, the attention's and the part norms' rows as terms that the product behind them reads, against the same step with fp32 rows and the other products (stack.line 0).
# Both multiply weights of 16 bits by two 16-bit terms (2^-16 of an input, or 2^-22), layer by layer: 2^-12 of the largest logit holds what four layers make of it.
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("inner,rank,left,right", [(192, 160, 16, 16), (256, 168, 32, 16), (200, 160, 16, 12)])      # rows of whole lines, and (the last) none that are
def test_rows_as_terms_of_the_product_behind(inner, rank, left, right, dtype):
    import test_hip_nusovik as tn
    mamba = tn.mamba(tn.ff(64), inner=inner, dt_rank=rank, state=16)
    cfg = tn.config([mamba, tn.par(tn.ff(64), left=dict(heads=4, kv_heads=2, dim=left, mask={"size": 65}), right=dict(vdim=right))] * 2, width=320)
    sizes = [3001, 1160]
    got = []
    for line in (1, 0):
        eng, w = tn.engine(cfg, dtype, max_seqs=2, max_ctx=4096, budget_tokens=8192, options={"stack.line": line, "stack.conv_tiles": 1})
        got.append(eng.step([("s%d" % i, tn.tokens(cfg, n, i), [0, 64, n // 2, n - 1]) for i, n in enumerate(sizes)]))
        got[-1] = np.concatenate([got[-1], eng.step([("s%d" % i, tn.tokens(cfg, 1, i), [0]) for i in range(2)])])
        eng.close()
    assert np.abs(got[0] - got[1]).max() / np.abs(got[1]).max() < 2.0 ** -12
    assert not (got[0] == got[1]).all()
