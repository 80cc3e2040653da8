"""The filters in front of the recurrences in tiles of eight tokens (option stack.conv_tiles) against the form of a channel a thread and against the oracles: entries that begin, end and
change inside a tile, shorter than a tile and than the filter, that go on from a slot's tails; widths of one tile and a remainder; every filter length that has tiles; heads of every size
that has tiles.  All sums run in the same order, those of a delta rule's unit vectors too, so the two forms answer with the same bits.  fp32 storage, 1e-4 of the largest logit against the oracle."""
import numpy as np
import pytest

import test_hip_keronex as tk
import test_hip_nusovik as tn
import test_hip_vitudra as tv

pytestmark = pytest.mark.gpu


def model(kind, taps, **kw):
    if kind == "mamba1":      # 260 channels: a tile and four
        cfg = tn.config([tn.mamba(tn.ff(), inner=260, conv=taps), tn.mamba(inner=28, conv=taps)])
        eng, w = tn.engine(cfg, "fp32", 3, **kw)
        return eng, lambda t: tn.want_of(cfg, w, t), cfg
    if kind == "ssd":
        cfg = tn.config([tn.par(tn.ff(), right=dict(conv=taps, heads=8, vdim=32, state=16)), tn.mamba()])
        eng, w = tn.engine(cfg, "fp32", 3, **kw)
        return eng, lambda t: tn.want_of(cfg, w, t), cfg
    dim = int(kind.rstrip("+").split("-")[1])      # key channels of a head; +: q and k alone are more than a tile's 256 channels
    if kind.startswith("delta"):
        cfg = tv.config([tv.par(tv.ff(), right=dict(conv=taps, dim=dim, heads=4, kv_heads=2, vdim=36)), tv.par(right=dict(conv=taps, dim=dim, heads=2, kv_heads=1, vdim=8))])
        eng, w = tv.engine(cfg, "fp32", 3, **kw)
        return eng, lambda t: tv.want_of(cfg, w, t), cfg
    heads = 3 if kind.endswith("+") else 2
    cfg = tk.config([tk.cd(tk.dense(), conv=taps, dim=dim, heads=heads, kv_heads=heads, vdim=20), tk.cd(conv=taps, dim=dim, vdim=4)])
    eng, w = tk.engine(cfg, "fp32", 3, **kw)
    return eng, lambda t: tk.want_of(cfg, w, t), cfg


@pytest.mark.parametrize("taps", [2, 3, 4, 5])      # (five: no tiles)
@pytest.mark.parametrize("kind", ["mamba1", "ssd", "delta-32", "delta-64", "delta-128", "cdelta-32", "cdelta-64", "cdelta-128+"])
def test_tiles_equal_the_plain_form(kind, taps):
    eng, want_of, cfg = model(kind, taps)
    sizes = [[9, 1, 16, 33], [2, 7, 8, 3], [1, 1, 31, 5]]      # three steps of four entries: 59, 20 and 38 tokens
    seqs = [tk.tokens(cfg, sum(s[i] for s in sizes), seed=i) for i in range(4)]
    want = [want_of(s) for s in seqs]
    got = {}
    for tiles in (0, 1):
        eng.model.set_option("stack.conv_tiles", tiles)
        at, rows = [0] * 4, [[] for _ in range(4)]
        for step in sizes:
            out = eng.step([("%d/%d" % (tiles, i), seqs[i][at[i]:at[i] + n], list(range(n))) for i, n in enumerate(step)])
            k = 0
            for i, n in enumerate(step):
                rows[i].append(out[k:k + n])
                at[i] += n; k += n
        got[tiles] = [np.concatenate(r) for r in rows]
        for i in range(4):
            eng.release("%d/%d" % (tiles, i))
    for i in range(4):
        scale = np.abs(want[i]).max()
        assert np.abs(got[1][i] - want[i]).max() / scale < 1e-4
        assert np.array_equal(got[0][i], got[1][i])
    eng.close()
