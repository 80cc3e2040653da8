"""The matrix products of layered models at the sizes where their forms change and their tiles end: rows of a step (one and two on the vector kernel, up to 64 on the
few-row kernel, beyond on the tiles), contraction lengths that are no multiple of a step of 64, column counts that are no multiple of sixteen, grouped expert
products with few and with many pairs.  fp32 storage against the plain oracle: nothing is rounded, so what remains is fp32 summation over at most 264 terms per
product through two layers (measured 1e-6; bound 2e-5 of the largest logit).  16-bit storage against the same sequences stepped one at a time: the cached latents may
round to the other neighbour (2^-9 for bf16, 2^-12 for fp16) where two sums of the same terms differ in their last bit; the bound is that of one such step."""
import numpy as np
import pytest

import stack_oracle as so
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
