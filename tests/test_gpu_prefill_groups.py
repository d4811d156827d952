"""The k-group builds of the MFMA-tiled kernel (kernels/prefill.hip, _n2k4 / _n3k4): every build at the edges of its tiles,
plain, gated and with the options of a deferred normalisation, against the bit-exact device twin of the oracle's lane order."""
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


def _upload(dec, n, k, group, bf16, t):
    q, s, x = gen.make_linear(n, k, group, t, seed=91)
    if bf16:
        s = (gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16)
    dec.upload_lin_g("pg", q, s, n, k, group, bf16)
    return x


def _run(dec, x, words, call):
    """Result words of one call on a buffer with guard words behind it, which must stay."""
    cc = dec.cc
    xd, yd = cc.to_device(x), cc.to_device(np.full(words + 64, GUARD, np.uint32))
    try:
        call(xd, yd)
        y, sym = cc.d2h(yd, (words + 64,), np.uint32), cc.last_launch_symbol()
    finally:
        cc.free(xd)
        cc.free(yd)
    assert np.all(y[words:] == GUARD)
    return y[:words], sym


def _name(group, bf16, cols):
    return "w4a16_prefill_g%d_%s_m64_n%dk4" % (group, "bf16" if bf16 else "f16", cols)


# n with rows past a multiple of 16, 32, 64 and of the block tile; 1, 3 and 9 k tiles (groups that stay empty, shorter last
# ones); t on both sides of a multiple of 64 and of 32
SHAPES = [(200, 128, 65, 2), (1000, 640, 97, 2), (1152, 384, 129, 2), (4104, 1152, 127, 2), (4104, 1152, 320, 2), (8232, 1152, 193, 3),
          (8200, 640, 256, 3), (12296, 1152, 129, 3)]
TYPES = [(128, False), (128, True), (32, False), (32, True)]


@pytest.mark.parametrize("group,bf16", TYPES)
@pytest.mark.parametrize("n,k,t,cols", SHAPES)
def test_builds_match_the_lane_twin(dec, n, k, t, cols, group, bf16):
    print("groups", n, k, t, group, bf16, flush=True)
    x = _upload(dec, n, k, group, bf16, t)
    want, _ = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t, path=ops.PATH_LANE))
    got, sym = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t))
    assert sym == _name(group, bf16, cols)
    parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "groups t%d" % t)
    again, _ = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t))
    assert np.array_equal(got, again)
    h, _ = _run(dec, x, (t * n + 1) // 2, lambda xd, yd: dec.lin_forward("pg", xd, yd, t, out_f16=True))
    assert np.array_equal(h.view(np.uint16)[:t * n], gen.f32_to_f16_bits(got.view(np.float32)).reshape(-1))


@pytest.mark.parametrize("group,bf16", TYPES)
@pytest.mark.parametrize("n,k,t,cols", [(224, 128, 65, 2), (4128, 1152, 127, 2), (8224, 1152, 193, 3)])
def test_gated_builds_give_the_bits_of_the_pair(dec, n, k, t, cols, group, bf16):
    """The gated launch against the plain one followed by the element-wise kernel: same tile, same k groups."""
    x = _upload(dec, n, k, group, bf16, t)
    cc = dec.cc
    f, _ = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t))
    fd, od = cc.to_device(f), cc.alloc(t * n)
    try:
        for gelu in (False, True):
            dec.act_mul_f16(fd, n // 2, t, od, gelu=gelu)
            want = cc.d2h(od, (t * n // 4,), np.uint32)
            got, sym = _run(dec, x, t * n // 4, lambda xd, yd: dec.lin_forward_glu("pg", xd, yd, t, gelu=gelu))
            assert sym == _name(group, bf16, cols) + "_glu"
            assert np.array_equal(got, want)
    finally:
        cc.free(fd)
        cc.free(od)


@pytest.mark.parametrize("n,k,t,cols", [(2120, 640, 97, 2), (8232, 640, 193, 3)])
def test_options_of_a_deferred_norm(dec, n, k, t, cols):
    """Row factor, residual stream, statistics per 64 columns, norm weight and hand-over factors, applied by the group that
    finishes the row, each against the same arithmetic on the plain launch's sums.  The factor is s_in * 2^3 rounded once (two
    roundings apart from the f64 value, 2 ulp of f32 each way: 4 * 2^-23 of the factored sum); the rest is exact on what the
    launch leaves in the residual stream."""
    ldx, in_cols, n_in, stat_rows = k + 128, 777, 37, n - 100
    x = _upload(dec, n, k, 128, False, t)
    plain, _ = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t))
    plain = plain.view(np.float32).reshape(t, n)
    xw = np.zeros((t, ldx), np.uint16)
    xw[:, :k] = x.view(np.uint16).reshape(t, k)
    rng = np.random.default_rng(t)
    ld = (t + 3) // 4 * 4
    prev = np.zeros((n_in, ld), np.float32)
    prev[:, :t] = (rng.standard_normal((n_in, t)) ** 2 * 100).astype(np.float32)
    total = np.zeros(ld, np.float32)
    for e in range(n_in):
        total += prev[e]  # f32, in the order of the entries
    fac = 8.0 / np.sqrt(total.astype(np.float64)[:t] * np.float64(np.float32(1.0 / in_cols)) + 1e-6)
    resid0 = (rng.standard_normal((t, n)) * 0.5).astype(np.float32)
    nw = (1.0 + 0.3 * rng.standard_normal(n)).astype(np.float32)
    cc = dec.cc
    entries = (n + 63) // 64
    px, pp, py, ps = cc.to_device(xw), cc.to_device(prev), cc.alloc(t * n * 2), cc.alloc(entries * ld * 4)
    pr, pw = cc.to_device(resid0), cc.to_device(nw)
    try:
        n_out = dec.lin_forward_deferred_norm("pg", px, t, py, out_f16=True, ldx=ldx, stats_in=pp, n_stats_in=n_in, in_cols=in_cols,
                                              stats_out=ps, stat_rows=stat_rows, resid=pr, nw=pw, in_exp=3, out_exp=2)
        assert cc.last_launch_symbol() == _name(128, False, cols) and n_out == (stat_rows + 63) // 64
        v = cc.d2h(pr, (t, n), np.float32)
        scaled = fac[:, None] * plain.astype(np.float64)
        bound = 4 * 2.0 ** -23 * np.abs(scaled) + 2.0 ** -23 * (np.abs(resid0) + np.abs(scaled))  # factored sum, then the addition
        assert np.all(np.abs(v - (resid0 + scaled)) <= bound)
        y = cc.d2h(py, (t, n), np.uint16)
        assert np.array_equal(y, gen.f32_to_f16_bits((v * nw[None, :]).astype(np.float32) * np.float32(0.25)))
        st = cc.d2h(ps, (n_out, ld), np.float32)[:, :t].astype(np.float64)
        for e in range(n_out):  # 64 squares added in f32: 64 roundings at most
            want = (v[:, e * 64:min(e * 64 + 64, stat_rows)].astype(np.float64) ** 2).sum(1)
            assert np.all(np.abs(st[e] - want) <= 64 * 2.0 ** -24 * want)
    finally:
        for p in (px, pp, py, ps, pr, pw):
            cc.free(p)


@pytest.mark.parametrize("group,bf16", [(128, False), (32, True)])
@pytest.mark.parametrize("n,k,t,cols", [(1, 640, 65, 2), (67, 384, 100, 2), (1001, 640, 97, 2), (4103, 1152, 129, 2), (8234, 1152, 193, 3)])
def test_widths_that_are_no_multiple_of_four(dec, n, k, t, cols, group, bf16):
    print("odd width", n, k, t, group, bf16, flush=True)
    x = _upload(dec, n, k, group, bf16, t)
    want, _ = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t, path=ops.PATH_LANE))
    got, sym = _run(dec, x, t * n, lambda xd, yd: dec.lin_forward("pg", xd, yd, t))
    assert sym == _name(group, bf16, cols)
    parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "odd width %d" % n)
    h, _ = _run(dec, x, (t * n + 1) // 2, lambda xd, yd: dec.lin_forward("pg", xd, yd, t, out_f16=True))
    h = h.view(np.uint16)
    assert np.array_equal(h[:t * n], gen.f32_to_f16_bits(got.view(np.float32)).reshape(-1))
    assert t * n % 2 == 0 or h[t * n] == GUARD >> 16  # the half word behind the last element
