"""The MFMA-tiled grouped kernels at the edges of their block tiles: runs that end just before and after 32 and 64 slots, empty
and single experts, more segments than one per XCD and fewer, XCD shares that end inside a segment, column tiles that are half empty."""
import numpy as np
import pytest

from llm170_amd import gen, ops

from .test_gpu_moe import _check_ffn, _run_ffn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    d.set_moe_tiled(1)
    yield d
    d.cc.close()


@pytest.mark.parametrize("group", [32, 128])
@pytest.mark.parametrize("h,n_ff,runs", [
    (128, 384, [1, 0, 32, 33, 0, 64, 65, 96, 97, 128, 129, 31]), (384, 128, [700]), (256, 256, [0, 0, 5]),
    (640, 128, [63, 1, 64, 32] * 5), (640, 384, [64] * 9)])
def test_tiled_runs_of_every_length(dec, orc, group, h, n_ff, runs):
    """top_k = 1, so that run lengths are what the list says; the slots of a run are scattered over the tokens.  silu only: the
    gelu's 1 + tanhf(..) cancels for gates below about -3, an error of up to 0.5 |g u| 2^-23 that the one-step envelope of the
    check does not hold (3 of 89600 values at 700 slots, in any kernel), and the activation has nothing to do with tile edges."""
    print("tiled runs", group, h, n_ff, runs, flush=True)
    E, t = len(runs), sum(runs)
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, group, seed=gen.GATE_SEED + 17)
    dec.upload_experts("edge", q13, s13, q2, s2, E, h, n_ff, group, False)
    idx = np.random.default_rng(5).permutation(np.repeat(np.arange(E), runs)).astype(np.int32)[:, None]
    wt = (0.25 + np.random.default_rng(6).random((t, 1))).astype(np.float32)
    x = gen.normal_f16(79, (t, h))
    y, act, c2, blk = _run_ffn(dec, "edge", x, idx, wt, t, 1, h)
    assert blk == 64
    _check_ffn(orc, y, act, c2, x, idx, wt, q13, s13, q2, s2, h, n_ff, group, False, "tiled runs")
    assert np.array_equal(y, c2.view(np.float16).astype(np.float32))  # one expert per token: its f16 row
