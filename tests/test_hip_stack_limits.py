"""Layered models where something runs out: a step that cannot issue one of its kernels."""
import numpy as np
import pytest

import stack_oracle as so
from test_hip_stack_products import desc
from tinygpt_amd.ffi import TgxError
from tinygpt_amd.serving import SlotEngine

pytestmark = pytest.mark.gpu


# The refused product is one of the few-row kernel (four requests), and its outputs are then those of the step before: finite numbers, so nothing is addressed by garbage.
@pytest.mark.parametrize("how", ["decode", "step", "async"])
@pytest.mark.parametrize("nth", [1, 4])
def test_a_step_that_cannot_issue_a_kernel_fails_and_a_reset_goes_on(how, nth):
    d = desc(264, "bf16", 4, 40, 8)
    t = so.random_tensors(d, 3)
    eng = SlotEngine(desc=d, tensors={k: v.astype(np.float32) for k, v in t.items()})
    m = eng.model
    ids = np.random.default_rng(5).integers(0, d.vocab, (4, 6))

    def begin():
        first = eng.step([(i, ids[i, :5], [4]) for i in range(4)])
        m.sample()
        return first, m.decode(3)

    whole = begin()
    for i in range(4):
        eng.release(i)
    eng.step([(i, ids[i, :5], [4]) for i in range(4)])
    m.sample()
    m.set_option("debug.refuse_lds", nth)
    with pytest.raises(TgxError, match="refused"):
        if how == "decode":
            m.decode(3)
        elif how == "async":
            m.step_async()
        else:
            eng.step([(i, ids[i, 5:], [0]) for i in range(4)])
    for call in (lambda: m.decode(1), lambda: eng.step([(0, ids[0, 5:], [0])]), lambda: m.forward_row(0, ids[0]), lambda: eng.release(0)):      # nothing goes on from half a step
        with pytest.raises(TgxError, match="half-way"):
            call()
    m.reset_cache()
    eng.slot_of, eng.free = {}, list(range(3, -1, -1))
    again = begin()
    eng.close()
    assert (again[0] == whole[0]).all() and (again[1] == whole[1]).all()
