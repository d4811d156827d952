"""Routing and slot alignment at the edges of the sizes their kernels are built for: 2, 4 or 16 experts per lane of the
routing wave, one workgroup or several for the alignment."""
import numpy as np
import pytest

from llm170_amd import gen, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    yield d
    d.cc.close()


@pytest.mark.parametrize("n,k,t", [(1, 1, 3), (2, 2, 1), (64, 8, 5), (65, 8, 4), (128, 64, 2), (129, 8, 7), (256, 8, 1),
                                   (257, 3, 2), (1000, 64, 3), (1024, 8, 9)])
def test_route_edges(dec, n, k, t):
    print("route", n, k, t, flush=True)
    lg = gen.normal_f32(n * 31 + t, (t, n))
    lg[0, : n // 2] = lg[0, n // 2]  # ties: the lower index first
    if t > 1:
        lg[1, : n - k] = -200.0      # probabilities that underflow to zero are still chosen in index order
    cc = dec.cc
    pl, pi, pw = cc.to_device(lg), cc.alloc(t * k * 4), cc.alloc(t * k * 4)
    dec.moe_route(pl, t, n, k, pi, pw)
    idx, w = cc.d2h(pi, (t, k), np.int32), cc.d2h(pw, (t, k), np.float32)
    for p in (pl, pi, pw):
        cc.free(p)
    want_i, want_w = ops.moe_topk(lg, k)
    assert np.array_equal(idx, want_i)
    # exp and the softmax sum in another order than on the host: 16 f32 roundings at most along either
    assert np.max(np.abs(w - want_w) / np.maximum(want_w, 1e-30)) < 16 * 2.0**-23
