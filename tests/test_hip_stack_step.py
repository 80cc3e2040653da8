"""Single tokens through a mixer's one launch (kernels/stack_step.h): recurrences whose heads fill, exceed and fall short of the columns and row groups of a workgroup,
convolutions of one tap to the most that the kernel takes and one more, attention over one key up to the most that it takes and past that, masks, caps, slopes, rotations and
groups of one to eight query heads.  fp32 storage against the plain oracles of the designs: fp32 sums over at most 256 channels and keys, 1e-4 of the largest logit as in the
designs' own tests; and against the same steps in the launches that it stands for, whose sums meet in another order (1e-5: a thousand roundings of 2^-24)."""
import numpy as np
import pytest

import test_hip_keronex as tk
import test_hip_modepel as tm
import test_hip_nusovik as tn
import test_hip_vitudra as tv
from tinygpt_amd.ffi import GREEDY, SamplerCfg

pytestmark = pytest.mark.gpu


def stepped(t, cfg, n, seed, first=2, **kw):
    """three sequences: a portion of `first` tokens each, then single tokens of all of them; the last logits by the step kernels and by the launches of their own, and the oracle's"""
    out, toks = [], [t.tokens(cfg, n, seed + i) for i in range(3)]
    for on in (1, 0):
        eng, w = t.engine(cfg, seed=seed, **kw)
        eng.model.set_option("stack.rec_step", on)
        got = [eng.step([(i, s[:first], [first - 1]) for i, s in enumerate(toks)])]
        got += [eng.step([(i, s[j:j + 1], [0]) for i, s in enumerate(toks)]) for j in range(first, n)]
        eng.close()
        out.append(np.stack(got, 1))
    assert np.abs(out[0] - out[1]).max() / np.abs(out[1]).max() < 1e-5
    for i, s in enumerate(toks):
        want = t.want_of(cfg, w, s)
        assert np.abs(out[0][i] - want[first - 1:n]).max() / np.abs(want).max() < 1e-4, i


@pytest.mark.parametrize("dim,vdim", [(4, 1), (6, 5), (8, 32), (36, 33), (64, 64), (128, 128), (132, 130), (256, 128), (40, 256), (24, 260)])
def test_delta_rule(dim, vdim):
    cfg = tv.config([tv.par(right=dict(dim=dim, vdim=vdim, heads=4, kv_heads=2)), tv.par(tv.ff(16), right=dict(dim=dim, vdim=vdim, heads=2, kv_heads=2, conv=2))], width=24)
    stepped(tv, cfg, 7, dim)


@pytest.mark.parametrize("taps", [1, 2, 3, 5, 8, 9])
@pytest.mark.parametrize("first", [1, 2, 9])
def test_convolution_tails(taps, first):
    cfg = tv.config([tv.par(right=dict(conv=taps)), tv.par(right=dict(conv=taps))], width=24)
    stepped(tv, cfg, first + 11, taps, first)


@pytest.mark.parametrize("dim,rank", [(4, 5), (6, 16), (33, 17), (64, 64), (128, 1), (160, 40), (256, 64)])
def test_wkv_with_its_decays(dim, rank):
    cfg = tv.config([tv.wkv(heads=2, dim=dim), tv.wkv(tv.ff(16), heads=3, dim=dim)], width=24)
    stepped(tv, cfg, 7, dim, decay_rank=rank)


@pytest.mark.parametrize("dim,vdim,rot", [(8, 12, 6), (64, 64, 64), (128, 256, 128), (10, 3, 2), (20, 130, None)])
def test_retention(dim, vdim, rot):
    cfg = tk.config([tk.ret(dim=dim, vdim=vdim, rot={"base": 10000.0, "dims": rot} if rot else None), tk.ret(dim=dim, vdim=vdim)], width=24)
    stepped(tk, cfg, 7, dim)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_blocks_of_single_tokens_where_they_are_asked_for(dtype):
    """ssd.min 1 sends single tokens of retention layers through the blocked recurrence whatever stack.rec_step says: the same bits, and others than the step kernel's"""
    cfg = tk.config([tk.ret(dim=64, vdim=128), tk.ret(dim=32, vdim=32)], width=32)
    out, toks = {}, tk.tokens(cfg, 9, 3)
    for ssd_min, on in ((1, 1), (1, 0), (64, 1)):
        eng, _ = tk.engine(cfg, dtype, 5, options={"ssd.min": ssd_min, "stack.rec_step": on})
        out[ssd_min, on] = np.concatenate([eng.step([("r", toks[:3], [2])])] + [eng.step([("r", toks[i:i + 1], [0])]) for i in range(3, 9)])
        eng.close()
    np.testing.assert_array_equal(out[1, 1], out[1, 0])
    assert (out[1, 1] != out[64, 1]).any()


@pytest.mark.parametrize("dim,vdim", [(8, 6), (64, 32), (128, 128), (100, 65), (4, 200)])
def test_channel_decays(dim, vdim):
    cfg = tk.config([tk.cd(dim=dim, vdim=vdim), tk.cd(tk.dense(16), dim=dim, vdim=vdim, conv=1)], width=24)
    stepped(tk, cfg, 7, dim)


@pytest.mark.parametrize("n", [1, 2, 62, 63, 64, 127, 128, 255, 256, 257])
@pytest.mark.parametrize("shape", [dict(heads=4, kv_heads=1, dim=8, vdim=6), dict(heads=2, kv_heads=2, dim=64, vdim=64), dict(heads=3, kv_heads=1, dim=136, vdim=128), dict(heads=8, kv_heads=2, dim=256, vdim=100), dict(heads=5, kv_heads=1, dim=16, vdim=24),
                                   dict(heads=16, kv_heads=2, dim=64, vdim=64)])
def test_attention_of_so_many_keys(n, shape):
    layers = [tv.attn(mask=None, **shape), tv.attn(tv.ff(16), kv_from=0, mask=None, **shape), tv.par(tv.ff(16), left=dict(shape, mask=None, softcap=3.0, rot={"base": 300.0, "dims": 8}))]
    cfg = tv.config(layers, width=24)
    stepped(tv, cfg, n + 2, n, max(1, n - 1))


# as many entries as give a workgroup a query head (256 compute units), and one more: four heads of a key / value head a workgroup from there on, the last of a group fewer (9 on 1: four, four,
# one), a layer that reads another's pool, caps, rotations, slopes, values mixed with the first layer's; keys from one to the most that the kernels take
@pytest.mark.parametrize("t", [tv, tm])
@pytest.mark.parametrize("shape", [dict(heads=8, kv_heads=2, dim=128, vdim=128), dict(heads=9, kv_heads=3, dim=16, vdim=24), dict(heads=9, kv_heads=1, dim=8, vdim=6), dict(heads=8, kv_heads=4, dim=136, vdim=100),
                                   dict(heads=16, kv_heads=1, dim=64, vdim=72)])
@pytest.mark.parametrize("more", [0, 1])
def test_attention_of_many_entries(t, shape, more):
    if t is tv:
        cfg = tv.config([tv.attn(mask=None, **shape), tv.attn(tv.ff(16), kv_from=0, mask=None, **shape), tv.par(tv.ff(16), left=dict(shape, mask=None, softcap=3.0, rot={"base": 300.0, "dims": 8}))], width=24)
    else:
        cfg = tm.config([tm.attn(tm.dense(), **shape), tm.attn(tm.dense(), **shape), tm.attn(v_mix=False, **shape)], width=24)
    n = 256 // shape["heads"] + more
    lens = [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 252]
    toks = [t.tokens(cfg, lens[i % len(lens)] + 3, i) for i in range(n)]
    out = []
    for on in (1, 0):
        eng, w = t.engine(cfg, seed=shape["dim"], max_seqs=n, max_ctx=256, budget_tokens=256 * n)
        eng.model.set_option("stack.rec_step", on)
        got = [eng.step([(i, s[:-3], [len(s) - 4]) for i, s in enumerate(toks)])]
        got += [eng.step([(i, s[len(s) - j:len(s) - j + 1], [0]) for i, s in enumerate(toks)]) for j in (3, 2, 1)]
        eng.close()
        out.append(np.stack(got, 1))
    assert np.abs(out[0] - out[1]).max() / np.abs(out[1]).max() < 1e-5
    for i in (*range(min(n, len(lens))), n - 1):
        want = t.want_of(cfg, w, toks[i])
        assert np.abs(out[0][i] - want[-4:]).max() / np.abs(want).max() < 1e-4, i


@pytest.mark.parametrize("mask", [{"size": 1}, {"size": 64}, {"size": 200}, {"size": 256}, {"size": 300}])
def test_attention_behind_masks(mask):
    cfg = tv.config([tv.attn(mask=mask), tv.par(tv.ff(16), left=dict(mask=mask))], width=24)
    stepped(tv, cfg, 330, mask["size"], 326)


# ---- sigmoid attention of single tokens over divided keys (kernels/stack_loop.h sigmoid_mix_step_kernel): value slices that divide 256 threads evenly and not, one to four query
# heads a key / value head, one to three of those, head counts up to sixteen, tiles of 32 keys that end inside; and shapes past its limits
@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 2, 8, 8), (3, 3, 16, 24), (8, 2, 128, 128), (16, 4, 64, 40), (4, 1, 120, 256), (6, 3, 24, 104), (17, 17, 8, 8), (5, 1, 8, 8), (2, 1, 12, 8)])
@pytest.mark.parametrize("n,mask", [(130, None), (163, {"size": 100}), (300, {"size": 257})])
def test_sigmoid_attention_of_divided_keys(heads, kv, dim, vdim, n, mask):
    import test_hip_zaluvik as tz
    kw = dict(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, mask=mask)
    cfg = tz.config([tz.attn(**kw), tz.attn(tz.dense(), **kw)], width=24)
    toks = tz.tokens(cfg, n, seed=dim)
    eng, w = tz.engine(cfg, seed=heads)
    got = [eng.step([("a", toks[:n - 3], [n - 4])])] + [eng.step([("a", toks[j:j + 1], [0])]) for j in range(n - 3, n)]
    eng.close()
    want = tz.want_of(cfg, w, toks)
    assert np.abs(np.concatenate(got) - want[n - 4:]).max() / np.abs(want).max() < 1e-4


# ---- the scan over portions: blocks of sixteen and eight tokens, one and two turns of eight, sixteen and thirty-two row groups, odd ends of each; then single tokens carry on
@pytest.mark.parametrize("dim,vdim,entries", [(128, 36, 1), (100, 20, 1), (64, 17, 1), (192, 24, 1), (32, 40, 24), (128, 64, 24), (30, 6, 2)])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 15, 16, 17, 24, 33])
def test_scan_over_portions(dim, vdim, entries, n):
    cfg = tv.config([tv.par(right=dict(dim=dim, vdim=vdim, heads=4, kv_heads=2)), tv.wkv(heads=2, dim=dim)], width=20)
    eng, w = tv.engine(cfg, seed=dim, max_seqs=entries, max_ctx=128, budget_tokens=64 * entries)
    toks = [tv.tokens(cfg, n + 3, seed=i) for i in range(entries)]
    got = [eng.step([(i, s[:max(1, n - i % 3)], [max(1, n - i % 3) - 1]) for i, s in enumerate(toks)])]
    got.append(eng.step([(i, s[max(1, n - i % 3):], [len(s) - max(1, n - i % 3) - 1]) for i, s in enumerate(toks)]))
    eng.close()
    for i in {0, entries // 2}:
        want = tv.want_of(cfg, w, toks[i])
        for at, part in ((max(1, n - i % 3) - 1, got[0]), (n + 2, got[1])):
            assert np.abs(part[i] - want[at]).max() / np.abs(want).max() < 1e-4, (n, i, at)


# ---- sigmoid attention of prompts over divided keys (two to four shares while the tiles leave half of the chip idle), against the undivided lane kernels: the same bf16 weights and
# cached rows, bound of the design's own comparison of the two
@pytest.mark.parametrize("shape", [dict(heads=4, kv_heads=2, dim=32, vdim=64), dict(heads=2, kv_heads=1, dim=16, vdim=32)])
@pytest.mark.parametrize("size", [None, 513, 770, 1100])
def test_sigmoid_attention_of_prompts_over_divided_keys(shape, size):
    import test_hip_zaluvik as tz
    mask = {"size": size} if size else None
    cfg = tz.config([tz.attn(tz.dense(), mask=mask, scale=2.0, **shape), tz.attn(mask=mask, scale=2.0, **shape)], width=64, loop=None)
    toks = [tz.tokens(cfg, n, seed=n) for n in (1201, 530)]
    out = []
    for on in (1, 0):
        eng, _ = tz.engine(cfg, "bf16", seed=3, max_ctx=2048, budget_tokens=4096)
        eng.model.set_option("attn.mfma", on)
        o = [eng.step([("a", toks[0][:640], [0, 511, 512, 639]), ("b", toks[1], [0, 31, 32, 529])])]
        o.append(eng.step([("a", toks[0][640:], [0, 31, 300, 560])]))
        eng.close()
        out.append(np.concatenate(o))
    assert np.abs(out[0] - out[1]).max() / np.abs(out[1]).max() < 1e-3


# ---- products in one launch beside what does not need them: a channel-delta layer's low-rank pair (equal inner lengths; outputs of equal and of different widths; unequal lengths
# stand apart) and a latent layer's append beside its queries, rows around the sixteen, 32 and 64 of an operand and past the last
@pytest.mark.parametrize("ranks", [(8, 8), (72, 72), (16, 8)])
@pytest.mark.parametrize("dim,vdim", [(16, 16), (8, 24), (40, 8)])
@pytest.mark.parametrize("rows", [3, 16, 17, 33, 64, 65])
def test_low_rank_pair(rows, dim, vdim, ranks):
    cfg = tk.config([tk.cd(dim=dim, vdim=vdim)], width=24)
    eng, w = tk.engine(cfg, seed=rows, ranks=ranks)
    toks = tk.tokens(cfg, rows, seed=dim)
    got = tk.run_whole(eng, "a", toks)
    eng.close()
    tk.check(got, tk.want_of(cfg, w, toks), "fp32", f"{rows} rows")


@pytest.mark.parametrize("kv_rank,dim,heads", [(24, 8, 3), (72, 16, 2), (16, 40, 5)])
@pytest.mark.parametrize("slots", [2, 3, 16, 17])
def test_latents_beside_their_queries(slots, kv_rank, dim, heads):
    import stack_oracle as so
    from tinygpt_amd.desc import LayerDesc, StackDesc
    from tinygpt_amd.serving import SlotEngine
    layers = [LayerDesc(heads=heads, dim=dim, vdim=8, kv_rank=kv_rank, scale=0.35, mlp="moe", experts=5, top=2, ff=24, limit=1.5) for _ in range(3)]
    d = StackDesc(width=72, vocab=53, canon_taps=4, norm_groups=2, norm_eps=1e-6, max_seqs=slots, max_ctx=64, budget_tokens=64 * slots, compute_dtype="fp32", layers=layers)
    t = so.random_tensors(d, slots)
    seqs = np.random.default_rng(slots).integers(0, 53, (slots, 5))
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    got = np.stack([eng.step([(i, [s[j]], [0]) for i, s in enumerate(seqs)]) for j in range(5)], 1)
    eng.close()
    for i in {0, slots // 2, slots - 1}:
        want = so.forward(d, t, seqs[i].tolist())
        assert np.abs(got[i] - want).max() / np.abs(want).max() < 1e-4, (slots, i)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("width", [24, 1016, 1032, 2056])      # one lane's slices, eight waves with a remainder, four waves, two passes and a remainder
@pytest.mark.parametrize("rows", [1, 2])
def test_norms_inside_the_products_of_one_and_two_rows(width, rows, dtype):
    """the norms in front of a layer and of the output head in the products behind them, against the oracle and against the norms' own launches (stack.gemv 0): one row, two rows of one
    sequence (the shift's row before is one of the step's) and two sequences of one row"""
    cfg = tv.config([tv.wkv(tv.ff(16)), tv.par(tv.ff(16)), tv.attn(tv.ff(16))], width=width, vocab=4104)
    tol = 1e-4 if dtype == "fp32" else 3e-2
    eng, w = tv.engine(cfg, dtype, seed=4)
    toks = [tv.tokens(cfg, 8, i) for i in range(2)]
    want = [tv.want_of(cfg, w, t) for t in toks]
    for one in (True, False):
        got = {}
        for on in (1, 0):
            eng.model.set_option("stack.gemv", on)
            out = []
            for at in range(0, 8, rows if one else 1):
                e = [("a", toks[0][at:at + rows], list(range(rows)))] if one else [(i, toks[i][at:at + 1], [0]) for i in range(rows)]
                out.append(eng.step(e))
            for r in (["a"] if one else range(rows)):
                eng.release(r)
            got[on] = np.concatenate(out)
        ref = want[0] if one else np.stack(want[:rows], 1).reshape(-1, want[0].shape[1])
        scale = np.abs(ref).max()
        assert np.abs(got[1] - ref).max() / scale < tol
        if dtype == "fp32":
            assert np.abs(got[1] - got[0]).max() / scale < 1e-5
    eng.close()


@pytest.mark.parametrize("rank,vdim,heads", [(64, 8, 3), (128, 33, 2), (320, 70, 2), (512, 16, 1), (72, 8, 2)])      # (72: merge and product apart)
@pytest.mark.parametrize("keys,dtype", [(700, "fp32"), (1130, "bf16")])      # two or three records a token; eighteen
def test_values_from_the_records_of_divided_keys(rank, vdim, heads, keys, dtype):
    """a latent attention's merge and value product in one launch: one and three tokens over divided keys, against the oracle, and in fp32 against the two launches (act.round16, which
    rounds nothing there, keeps them)"""
    import stack_oracle as so
    from tinygpt_amd.desc import LayerDesc, StackDesc
    from tinygpt_amd.serving import SlotEngine
    layers = [LayerDesc(heads=heads, dim=16, vdim=vdim, kv_rank=rank, scale=0.35, mlp=None) for _ in range(2)]
    d = StackDesc(width=32, vocab=53, canon_taps=4, norm_groups=2, norm_eps=1e-6, max_seqs=3, max_ctx=1280, budget_tokens=3840, compute_dtype=dtype, layers=layers)
    t = so.random_tensors(d, rank)
    seqs = [np.random.default_rng(rank + i).integers(0, 53, keys - 9 * i) for i in range(3)]
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    eng.model.set_option("attn.split_min", 64)
    got = {}
    for apart in (0, 1):
        eng.model.set_option("act.round16", apart if dtype == "fp32" else 0)
        eng.step([(i, s[:-4], []) for i, s in enumerate(seqs)])
        rows = [eng.step([(0, seqs[0][-4:-3], [0])])]
        rows += [eng.step([(i, s[len(s) - 4 + j + (i == 0):len(s) - 3 + j + (i == 0)], [0]) for i, s in enumerate(seqs)]) for j in range(3)]
        got[apart] = np.concatenate(rows)
        for i in range(3):
            eng.release(i)
    eng.close()
    want = [so.forward(d, t, s.tolist()) for s in seqs]
    ref = np.concatenate([want[0][-4:-3]] + [np.stack([want[i][len(seqs[i]) - 4 + j + (i == 0)] for i in range(3)]) for j in range(3)])
    scale = np.abs(ref).max()
    assert np.abs(got[0] - ref).max() / scale < (1e-4 if dtype == "fp32" else 3e-2)
    if dtype == "fp32":
        assert np.abs(got[0] - got[1]).max() / scale < 1e-5


def choice_margin(scores, top, groups, keep, group_score):
    """the least difference of choice scores, over all tokens, that sends one to another group or another expert"""
    least = np.inf
    for c in scores:
        g = c.reshape(groups, -1)
        gs = np.array([group_score(v) for v in g])
        order = np.argsort(-gs)
        if keep < groups:
            least = min(least, gs[order[keep - 1]] - gs[order[keep]])
        c = np.sort(g[order[:keep]].reshape(-1))[::-1]
        if top < len(c):
            least = min(least, c[top - 1] - c[top])
    return least


@pytest.mark.parametrize("design", ["zaluvik", "modepel", "modepel_plain"])
@pytest.mark.parametrize("tokens", [1, 2, 3, 16, 21, 40, 43, 90])      # pairs with the shared choice: up to 128 ride, of one to many rows an expert, more do not
def test_shared_experts_among_the_routed_ones(design, tokens, monkeypatch):
    """a shared expert of the routed ones' size as one more choice (Modepel: between the experts and the identity outputs, weighted by its gate) against the oracle, and against its own
    launches (a width of the experts that keeps the forms of few pairs away has none to compare: stack.gemv 0).  The first weights and prompt whose choices are no close calls, so that every row counts"""
    import modepel_oracle as mo
    import test_hip_modepel as tm
    import test_hip_zaluvik as tz
    import zaluvik_oracle as zo
    least = []
    if design == "zaluvik":
        t, cfg = tz, tz.config([tz.attn(tz.moe(ff=16, shared=16)), tz.lat(tz.moe(ff=16, shared=16, groups=None))], loop=None)

        def watch(h, f, wr, route=zo.route):
            grp = f["router"].get("groups") or {"count": 1, "keep": 1}
            least.append(choice_margin(zo.sigmoid(h @ wr.T), f["router"]["top"], grp["count"], grp["keep"], lambda v: np.sort(v)[-2:].sum()))
            return route(h, f, wr)
        monkeypatch.setattr(zo, "route", watch)
    else:
        identity = 2 if design == "modepel" else 0
        t, cfg = tm, tm.config([tm.attn(tm.moe(ff=16, shared=16, identity=identity)), tm.rec(tm.moe(ff=16, shared=16, identity=identity, experts=8 - identity, top=3, keep=2))])

        def watch(h, wr, correction, r, route=mo.route):
            z = np.exp(h @ wr.T)
            least.append(choice_margin(z / z.sum(-1, keepdims=True) + correction, r["top"], r["groups"]["count"], r["groups"]["keep"], np.max))
            return route(h, wr, correction, r)
        monkeypatch.setattr(mo, "route", watch)
    for seed in range(11, 31):
        w = (zo if design == "zaluvik" else mo).random_tensors(cfg, seed)
        toks = t.tokens(cfg, tokens, tokens + seed)
        least.clear()
        want = t.want_of(cfg, w, toks)
        assert len(least) == 2
        if min(least) > 1e-4:
            break
    else:
        raise AssertionError("no prompt without close calls")
    eng, _ = t.engine(cfg, "fp32", seed)
    got = {}
    for on in (1, 0):
        eng.model.set_option("stack.gemv", on)
        got[on] = t.run_whole(eng, "r%d" % on, toks)
    eng.close()
    assert np.abs(got[1] - got[0]).max() / np.abs(got[0]).max() < 1e-4
    assert np.abs(got[1] - want).max() / np.abs(want).max() < 1e-4


@pytest.mark.parametrize("kv_rank,dim,rot_dim", [(16, 8, 8), (1032, 40, 16), (24, 136, 0)])
@pytest.mark.parametrize("slots", [1, 2, 3, 16, 17])
def test_rotated_latents_beside_their_queries(slots, kv_rank, dim, rot_dim):
    """a rotated latent layer's append beside the queries' products into latent space (the vector kernel's up to two rows, the matrix cores' up to 16), token by token against the oracle"""
    import test_hip_zaluvik as tz
    cfg = tz.config([tz.lat(tz.dense(), heads=3, dim=dim, rot_dim=rot_dim, vdim=8, kv_rank=kv_rank, mask={"size": 4})], loop=None)
    eng, w = tz.engine(cfg, "fp32", 2, max_seqs=slots, max_ctx=64, budget_tokens=64 * slots)
    toks = [tz.tokens(cfg, 6, i) for i in range(slots)]
    got = np.stack([eng.step([("s%d" % i, [s[j]], [0]) for i, s in enumerate(toks)]) for j in range(6)], 1)
    eng.close()
    for i in {0, slots // 2, slots - 1}:
        want = tz.want_of(cfg, w, toks[i])
        assert np.abs(got[i] - want).max() / np.abs(want).max() < 1e-4, (slots, i)


@pytest.mark.parametrize("slots,heads,kv_rank,rot_dim,vdim", [(3, 9, 64, 64, 8), (3, 10, 64, 64, 8), (4, 4, 64, 64, 8), (5, 4, 64, 64, 8), (16, 8, 64, 0, 256), (16, 8, 64, 0, 264)])
def test_latent_steps_of_many_heads_and_tokens(slots, heads, kv_rank, rot_dim, vdim):
    """both sides of where a latent layer's append and queries (rotated parts of 640 elements, four workgroups) and its merge and values (1024 workgroups) share a launch, against the oracle"""
    import test_hip_zaluvik as tz
    cfg = tz.config([tz.lat(tz.dense(), heads=heads, dim=16, rot_dim=rot_dim, vdim=vdim, kv_rank=kv_rank, mask=None) for _ in range(2)], loop=None)
    eng, w = tz.engine(cfg, "fp32", 2, max_seqs=slots, max_ctx=384, budget_tokens=384 * slots)
    eng.model.set_option("attn.split_min", 32)
    toks = [tz.tokens(cfg, 134, i) for i in range(slots)]
    for i, s in enumerate(toks): eng.step([(i, s[:130], [])])
    got = np.stack([eng.step([(i, s[130 + j:131 + j], [0]) for i, s in enumerate(toks)]) for j in range(4)], 1)
    eng.close()
    for i in {0, slots // 2, slots - 1}:
        want = tz.want_of(cfg, w, toks[i])
        assert np.abs(got[i] - want[130:]).max() / np.abs(want).max() < 1e-4, (slots, i)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("kv_heads,dim,vdim,size", [(1, 8, 8, None), (2, 24, 40, 128), (4, 128, 512, 160), (4, 64, 16, 128)])
def test_sigmoid_attention_appends_in_its_step(kv_heads, dim, vdim, size, dtype):
    """single tokens whose keys are divided between workgroups: the last share stores the token's own row (one of its own, the last and the first of a tile and of a page), against the oracle"""
    import test_hip_zaluvik as tz
    cfg = tz.config([tz.attn(tz.dense(), heads=4, kv_heads=kv_heads, dim=dim, vdim=vdim, mask={"size": size} if size else None) for _ in range(2)], loop=None)
    eng, w = tz.engine(cfg, dtype, 6)
    toks = [tz.tokens(cfg, 200, i) for i in range(2)]
    starts = [126, 188]      # keys that the steps see: 127 .. 131 and 189 .. 193, around a tile's and a page's first
    got = [[], []]
    eng.step([("s%d" % i, toks[i][:starts[i]], [0]) for i in range(2)])
    for j in range(5):
        step = eng.step([("s%d" % i, [toks[i][starts[i] + j]], [0]) for i in range(2)])
        for i in range(2): got[i].append(step[i])
    eng.close()
    for i in range(2):
        tz.check(np.stack(got[i]), tz.want_of(cfg, w, toks[i][:starts[i] + 5])[starts[i]:], dtype, f"sequence {i}")


# The launch between two greedy steps (kernels/stack_next.h): heads of one column, of fewer and of more than there are partials; a slot that was given back, and one that was never taken, ride
# along.  The same kernels run in steps that are fed those tokens, so that the logits are the same numbers.
@pytest.mark.parametrize("t,vocab", [(tv, 1), (tv, 67), (tv, 4100), (tv, 32772), (tv, 65536), (tv, 65540), (tm, 67), (tn, 131)])
def test_between_greedy_steps(t, vocab):
    cfg = t.config(vocab=vocab)
    first = [t.tokens(cfg, 3 + i, i) for i in range(3)]
    eng, _ = t.engine(cfg, seed=5)
    m = eng.model
    eng.step([(i, s, [len(s) - 1]) for i, s in enumerate(first)])
    eng.release(1)
    start = m.sample(GREEDY)
    toks = np.concatenate([m.decode(5, GREEDY), m.decode(1, GREEDY)])
    last, again = m.logits(rounded=False), m.sample(GREEDY)
    drawn = m.sample(SamplerCfg(temperature=0.7, top_k=1), seed=3)      # the sampler's maximum comes from the partials that the launch left
    eng.close()
    eng, _ = t.engine(cfg, seed=5)
    want = eng.step([(i, s, [len(s) - 1]) for i, s in enumerate(first)])
    eng.release(1)
    live, fed = [0, 2], start
    assert (np.argmax(want, 1)[live] == start[live]).all()
    for row in toks:
        want = eng.step([(i, [int(fed[i])], [0]) for i in live])
        assert (np.argmax(want, 1) == row[live]).all()
        fed = row
    assert np.array_equal(last[live], want) and (again[live] == toks[-1][live]).all()
    assert (drawn[live] == toks[-1][live]).all()
    eng.close()


# a dense feed-forward's PolyNorm: rows of fours up to 8192 channels stay in registers, others pass through memory; prompts and single tokens.  fp32 sums over the row: 1e-4 as in the design's tests
@pytest.mark.parametrize("ff", [1, 3, 4, 1020, 1022, 1024, 1028, 8188, 8192, 8196])
def test_poly_norm_rows(ff):
    cfg = tm.config([tm.rec(tm.dense(ff)), tm.rec(tm.dense(ff))])
    eng, w = tm.engine(cfg, seed=ff)
    toks = tm.tokens(cfg, 6, ff)
    got = np.concatenate([eng.step([(0, toks[:4], [0, 1, 2, 3])])] + [eng.step([(0, toks[i:i + 1], [0])]) for i in (4, 5)])
    want = tm.want_of(cfg, w, toks)
    eng.close()
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-4
