"""The order in which the tiled GEMM's workgroups walk the block tiles of an output: every tile of every k slice is computed, whatever
the numbers of tile rows, columns and slices (tiles that do not divide by the panels and bands, fewer tiles than XCDs, more than the
chip holds), against the bit-exact device twin of the oracle's lane order."""
import numpy as np
import pytest

from llm170_amd import gen, ops, parity

pytestmark = pytest.mark.gpu

GUARD = 0x7F5A5A5A  # a NaN no kernel here writes


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    yield d
    d.cc.close()


def _check(dec, n, k, t, group, what):
    q, s, x = gen.make_linear(n, k, group, t, seed=95)
    dec.upload_lin_g("walk", q, s, n, k, group, False)
    cc = dec.cc
    xd, yd, wd = cc.to_device(x), cc.to_device(np.full(t * n + 64, GUARD, np.uint32)), cc.alloc(t * n * 4)
    try:
        dec.lin_forward("walk", xd, yd, t, path=ops.PATH_PREFILL)
        dec.lin_forward("walk", xd, wd, t, path=ops.PATH_LANE)
        y, want = cc.d2h(yd, (t * n + 64,), np.uint32), cc.d2h(wd, (t, n), np.float32)
    finally:
        for b in (xd, yd, wd):
            cc.free(b)
    assert np.all(y[t * n:] == GUARD) and not np.any(y[:t * n] == GUARD)
    parity.assert_close(y[:t * n].view(np.float32).reshape(t, n), want, what)


@pytest.mark.parametrize("tile", [64, 96, 128])
@pytest.mark.parametrize("slices", [-1, 2, 5, 7, 8])
@pytest.mark.parametrize("n,t", [(2600, 650), (20, 65), (3600, 70), (260, 1500), (9000, 290)])
def test_every_tile_of_every_slice(dec, n, t, slices, tile):
    print("walk", n, t, slices, tile, flush=True)
    dec.set_prefill_tile(tile)
    dec.set_prefill_ksplit(slices)
    try:
        _check(dec, n, 4096, t, 128, "walk n%d t%d tile%d slices%d" % (n, t, tile, slices))
    finally:
        dec.set_prefill_tile(0)
        dec.set_prefill_ksplit(0)


@pytest.mark.parametrize("n,t,cols", [(848, 2982, 192), (576, 2022, 128), (2016, 966, 128), (128, 65, 128), (4096, 281, 128)])
def test_every_tile_of_the_k_group_builds(dec, n, t, cols):
    print("walk k groups", n, t, cols, flush=True)
    p = ops.plan_prefill_launch(t, n, 1280)
    assert (p["k_groups"], p["tile_cols"]) == (4, cols), p
    _check(dec, n, 1280, t, 128, "walk n%d t%d k groups" % (n, t))
