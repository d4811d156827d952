"""A launch's plan follows its own shape, scale group, options and pins, whatever ran before it in the same context."""
import numpy as np
import pytest

from llm170_amd import ops

pytestmark = pytest.mark.gpu


class _Program:
    def __init__(self):
        self.dec = ops.W4a16Dec()
        self.cc = self.dec.cc
        self.bufs = [self.cc.to_device(np.zeros((600, 5120), np.uint16)), self.cc.alloc(600 * 5120 * 4)]

    def upload(self, name, n, k, group):
        self.dec.upload_lin_synth(name, n, k, group, 3, 5)

    def run(self, call):
        call(*self.bufs)
        return self.cc.last_launch_symbol()

    def close(self):
        for b in self.bufs:
            self.cc.free(b)
        self.cc.close()


@pytest.fixture
def prog():
    p = _Program()
    yield p
    p.close()


@pytest.mark.parametrize("order", [(128, 32), (32, 128)])
def test_groups_of_one_shape_plan_on_their_own(prog, order):
    """5120 x 5120 at 200 rows: k groups at group 128, slices of k at group 32."""
    n, k, t = 5120, 5120, 200
    want = {128: "w4a16_prefill_g128_f16_m64_n2k4", 32: "w4a16_prefill_splitk_sum"}
    for g in order:
        prog.upload("g%d" % g, n, k, g)
    for g in order + order:
        assert prog.run(lambda x, y: prog.dec.lin_forward("g%d" % g, x, y, t)) == want[g], (g, order)


@pytest.mark.parametrize("pinned_first", [False, True])
def test_pinned_slices_and_whole_k_options_plan_on_their_own(prog, pinned_first):
    """A gated launch with an input factor keeps k whole by itself and may use k groups; a caller's pin of one slice names the
    256-column tiles."""
    n, k, t = 4096, 1024, 200
    prog.upload("glu", n, k, 128)

    def automatic():
        return prog.run(lambda x, y: prog.dec.lin_forward_glu_deferred_norm("glu", x, t, y, in_exp=1, out_exp=0))

    def pinned():
        prog.dec.set_prefill_ksplit(-1)
        try:
            return prog.run(lambda x, y: prog.dec.lin_forward_glu("glu", x, y, t))
        finally:
            prog.dec.set_prefill_ksplit(0)

    got = {}
    for f in ([pinned, automatic] if pinned_first else [automatic, pinned]) * 2:
        got.setdefault(f.__name__, set()).add(f())
    assert got == {"automatic": {"w4a16_prefill_g128_f16_m64_n2k4_glu"}, "pinned": {"w4a16_prefill_g128_f16_m64_glu"}}
