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
    live = max(1, k // 2)
    if t > 1:
        lg[1, : n - live] = -200.0  # fewer live experts than rounds: the others' probabilities underflow to zero
    cc = dec.cc
    pl, pi, pw = cc.to_device(lg), cc.alloc(t * k * 4), cc.alloc(t * k * 4)
    dec.moe_route(pl, t, n, k, pi, pw)
    idx, w = cc.d2h(pi, (t, k), np.int32), cc.d2h(pw, (t, k), np.float32)
    for p in (pl, pi, pw):
        cc.free(p)
    want_i, want_w = ops.moe_topk(lg, k)
    assert np.array_equal(idx, want_i)
    if t > 1:  # and are still chosen, each once, the lower index first
        assert np.array_equal(idx[1, live:], np.arange(k - live)) and np.all(w[1, live:] == 0) and np.all(w[1, :live] > 0)
    # Per weight, in units of 2^-24 and on both sides: exp 2 and the division by the softmax sum 1, for the weight and for
    # the sum it is divided by; k - 1 additions of that sum; the last division 1.  The softmax sum itself cancels.
    bound = 2 * (2 * 3 + (k - 1) + 1) * 2.0**-24
    assert np.all(np.abs(w - want_w) <= bound * want_w)


@pytest.mark.parametrize("bits", [0x7FC00000, 0xFFFFFFFF])
def test_route_nan_row(dec, bits):
    """A row with a NaN logit (also one of all ones, the largest bit pattern) still names k different experts."""
    n, k, t = 128, 8, 2
    lg = gen.normal_f32(5, (t, n))
    lg.view(np.uint32)[0, :] = bits
    lg.view(np.uint32)[1, 77] = bits
    cc = dec.cc
    pl, pi, pw = cc.to_device(lg), cc.alloc(t * k * 4), cc.alloc(t * k * 4)
    dec.moe_route(pl, t, n, k, pi, pw)
    idx, w = cc.d2h(pi, (t, k), np.int32), cc.d2h(pw, (t, k), np.float32)
    for p in (pl, pi, pw):
        cc.free(p)
    assert np.all(np.isnan(w))
    for row in idx:
        assert np.unique(row).size == k and row.min() >= 0 and row.max() < n


@pytest.mark.parametrize("ns,n_exp,block", [(2048, 128, 32), (2049, 128, 32), (4097, 128, 48), (32769, 128, 64),
                                            (70000, 8, 64), (2500, 1024, 16)])
@pytest.mark.parametrize("kind", ["random", "one expert", "dropped"])
def test_align_edges(dec, ns, n_exp, block, kind):
    print("align", ns, n_exp, block, kind, flush=True)
    idx = np.random.default_rng(ns).integers(0, n_exp, ns).astype(np.int32)
    if kind == "one expert":
        idx[:] = n_exp - 1
    if kind == "dropped":
        idx[::3] = -1
        idx[1::7] = n_exp
    cc = dec.cc
    cap_s, cap_e = ns + n_exp * block, ns // block + n_exp + 1
    pi, ps, pe, pn = cc.to_device(idx), cc.alloc(cap_s * 4), cc.alloc(cap_e * 4), cc.alloc(8)
    dec.moe_align(pi, ns, n_exp, block, ps, pe, pn)
    n_post, hit = cc.d2h(pn, (2,), np.int32)
    s, e = cc.d2h(ps, (cap_s,), np.int32), cc.d2h(pe, (cap_e,), np.int32)
    for p in (pi, ps, pe, pn):
        cc.free(p)
    want_s, want_e = [], []
    for x in range(n_exp):
        run = np.flatnonzero(idx == x)
        segs = -(-run.size // block)
        want_s.append(np.concatenate([run, np.full(segs * block - run.size, ns)]))
        want_e.append(np.full(segs, x))
    want_s, want_e = np.concatenate(want_s), np.concatenate(want_e)
    assert n_post == want_s.size and hit == np.unique(want_e).size
    assert np.array_equal(s[:n_post], want_s) and np.array_equal(e[: want_e.size], want_e)
