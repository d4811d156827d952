"""Dense linears at 17..64 rows (kernels/mid.hip): every build of the kernel at the edges of its tiles, against the bit-exact
device twin of the oracle's lane order, and the guarantee that launch shapes agree bit for bit."""
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


def _upload(dec, n, k, group, bf16, seed=83):
    q, s, x = gen.make_linear(n, k, group, 130, seed=seed)
    if bf16:
        s = (gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16)
    dec.upload_lin_g("mid", q, s, n, k, group, bf16)
    return x


def _run(dec, x, n, t, words, call):
    """Result words of one call on a buffer with a row of guard words behind it, which must stay."""
    cc = dec.cc
    xd, yd = cc.to_device(np.ascontiguousarray(x[:t])), cc.to_device(np.full(words + 64, GUARD, np.uint32))
    try:
        call(xd, yd)
        y = cc.d2h(yd, (words + 64,), np.uint32)
    finally:
        cc.free(xd)
        cc.free(yd)
    assert np.all(y[words:] == GUARD)
    return y[:words], cc.last_launch_symbol()


# n, k: one build of (waves along n, waves along k) each; odd numbers of row blocks and rows past a multiple of 16 among
# them, k tiles that do not divide by the four parts (5: parts of 2, 2, 1 and 0 tiles; 1: one part only)
SHAPES = [(4104, 128, "n1k4"), (424, 640, "n1k4"), (8232, 640, "n2k4"), (17000, 384, "n3k4"), (27016, 256, "n4k2"), (33008, 640, "n5k2"),
          (4104, 8448, "n4k1"), (2120, 5120, "n1k4"), (200, 16384, "n1k4")]  # the last three are split over k


FORMS = [(128, False, t) for t in (17, 32, 33, 48, 49, 64)] + [(32, True, t) for t in (17, 32, 33, 48, 49, 64)] + [
    (group, bf16, t) for group, bf16 in ((128, True), (32, False)) for t in (33, 64)]


@pytest.mark.parametrize("group,bf16,t", FORMS)
@pytest.mark.parametrize("n,k,build", SHAPES)
def test_builds_match_the_lane_twin(dec, n, k, build, group, bf16, t):
    print("mid", n, k, build, group, bf16, t, flush=True)
    x = _upload(dec, n, k, group, bf16)
    want, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_LANE))
    got, sym = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t))
    assert sym == "w4a16_mid_g%d_%s_t%d_%s" % (group, "bf16" if bf16 else "f16", 2 if t <= 32 else 3 if t <= 48 else 4, build)
    parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "mid %s t%d" % (build, t))
    h, _ = _run(dec, x, n, t, (t * n + 1) // 2, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, out_f16=True))
    assert np.array_equal(h.view(np.uint16)[:t * n], gen.f32_to_f16_bits(got.view(np.float32)).reshape(-1))


@pytest.mark.parametrize("t", [65, 130])
def test_rows_beyond_a_segment(dec, t):
    """PATH_STREAM at any number of rows: segments of 64, a ragged last one, also split over k."""
    for n, k in [(424, 640), (2120, 5120), (4104, 8448)]:
        x = _upload(dec, n, k, 128, False)
        want, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_LANE))
        got, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_STREAM))
        parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "segments t%d" % t)
        # k whole, or in a given number of slices (which follows the size of the grid), a row's sums do not depend on the rows around it
        try:
            for nks in (-1, 4):
                dec.set_decode_ksplit(nks)
                got, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_STREAM))
                parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "segments t%d" % t)
                one, _ = _run(dec, x, n, 64, 64 * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, 64, path=ops.PATH_STREAM))
                assert np.array_equal(one, got[:64 * n])
        finally:
            dec.set_decode_ksplit(0)


def test_many_segments_stay_whole_along_k(dec):
    """Slices of k are for a grid that does not fill the chip: ten segments do, and need no workspace."""
    n, k, t = 4104, 8448, 640
    q, s, x = gen.make_linear(n, k, 128, t, seed=86)
    dec.upload_lin_g("mid", q, s, n, k, 128, False)
    want, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_LANE))
    got, sym = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_STREAM))
    assert sym.endswith("_t4_n3k4")
    parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "ten segments")


@pytest.mark.parametrize("n,k,group,build", [(64, 384, 32, "n1k4"), (16448, 640, 128, "n3k4"), (8256, 1408, 128, "n2k4"),
                                             (26688, 384, 32, "n4k2"), (33024, 1152, 128, "n5k2")])
@pytest.mark.parametrize("t", [20, 45, 64])
def test_gated_builds_give_the_bits_of_the_pair(dec, n, k, group, build, t):
    """The gated launch against the plain one with k unsplit, whatever shapes the two take, and the element-wise kernel."""
    x = _upload(dec, n, k, group, group == 32)
    cc = dec.cc
    dec.set_decode_ksplit(-1)
    try:
        f, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t))
    finally:
        dec.set_decode_ksplit(0)
    fd, od = cc.to_device(f), cc.alloc(t * n)
    words = t * n // 4
    for gelu in (False, True):
        dec.act_mul_f16(fd, n // 2, t, od, gelu=gelu)
        want = cc.d2h(od, (words,), np.uint32)
        got, sym = _run(dec, x, n, t, words, lambda xd, yd: dec.lin_forward_glu("mid", xd, yd, t, gelu=gelu))
        assert sym.endswith("_%s_glu" % build)
        assert np.array_equal(got, want)
    cc.free(fd)
    cc.free(od)


def test_pinned_slices_agree_with_slice_launches(dec):
    """Slices of a split launch hold the same runs of k tiles as launches of their own, in the build that keeps its finished
    parts in LDS (n4k1) as in the one that spreads them over waves."""
    n, k, t, nks = 6160, 2560, 40, 4
    q, s, x = gen.make_linear(n, k, 128, t, seed=84)
    dec.upload_lin_g("mid", q, s, n, k, 128, False)
    dec.set_decode_ksplit(nks)
    try:
        got, sym = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t))
        assert sym.endswith("_n4k1")
        dec.set_decode_ksplit(-1)
        want = None
        for i in range(nks):
            lo, hi = i * 5, (i + 1) * 5
            dec.upload_lin_g("slice", np.ascontiguousarray(q[:, lo * 16:hi * 16]), np.ascontiguousarray(s[:, lo:hi]), n, 640, 128, False)
            part, sym = _run(dec, x[:, lo * 128:hi * 128], n, t, t * n, lambda xd, yd: dec.lin_forward("slice", xd, yd, t))
            assert sym.endswith("_n1k4")
            p = part.view(np.float32)
            want = p if want is None else (want + p).astype(np.float32)
    finally:
        dec.set_decode_ksplit(0)
    assert np.array_equal(got, want.view(np.uint32))


def test_weights_between_2_and_4_gib(dec):
    """Offsets into the tiled weights are unsigned 32-bit: rows on both sides of 2 GiB, and the last, against float64.
    Bound: f32 sums of k terms err by less than k * 2^-24 of the sum of the terms' magnitudes, far more than they do."""
    n, k, t, rng = 131088, 33024, 20, np.random.default_rng(85)
    q = np.tile(rng.integers(0, 2**32, (n // 16, k // 8), dtype=np.uint32), (16, 1))
    q[::16, 0] = np.arange(n // 16, dtype=np.uint32)  # rows of the copies differ
    s = np.tile(rng.uniform(0.002, 0.02, (n // 16, k // 128)).astype(np.float16), (16, 1)).view(np.uint16)
    x = rng.standard_normal((t, k)).astype(np.float16)
    dec.upload_lin_g("mid2g", q, s, n, k, 128, False)
    mark = 2**31 // (k // 2)
    rows = np.r_[0:16, mark - 32:mark + 32, n - 48:n]
    w = ((q[rows][:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(len(rows), k).astype(np.float64) - 8
    w *= np.repeat(s[rows].view(np.float16).astype(np.float64), 128, axis=1)
    got, sym = _run(dec, x.view(np.uint16), n, t, t * n, lambda xd, yd: dec.lin_forward("mid2g", xd, yd, t))
    dec.upload_lin_g("mid2g", q[:16], s[:16], 16, k, 128, False)  # the big copy is freed
    assert sym.startswith("w4a16_mid_g128_f16_t2_")
    y = got.view(np.float32).reshape(t, n)[:, rows]
    bound = k * 2.0**-24 * (np.abs(x.astype(np.float64)) @ np.abs(w).T)
    assert np.all(np.abs(y - x.astype(np.float64) @ w.T) <= bound)
    assert np.all(y != 0)


@pytest.mark.parametrize("group,bf16", [(128, False), (32, True)])
@pytest.mark.parametrize("t", [20, 45, 64])
def test_very_wide_outputs_walk_k_alone(dec, group, bf16, t):
    """Workgroups of four waves along n whose waves walk the whole of k (one group, finished parts kept in LDS), plain and
    gated: the last workgroup has surplus waves, k tiles (3) leave a part empty."""
    n, k, cc = 65504, 384, dec.cc
    x = _upload(dec, n, k, group, bf16)
    want, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_LANE))
    f, sym = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t))
    assert sym.endswith("_n4k1")
    parity.assert_close(f.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "wide t%d" % t)
    fd, od = cc.to_device(f), cc.alloc(t * n)
    dec.act_mul_f16(fd, n // 2, t, od)
    want = cc.d2h(od, (t * n // 4,), np.uint32)
    got, sym = _run(dec, x, n, t, t * n // 4, lambda xd, yd: dec.lin_forward_glu("mid", xd, yd, t))
    cc.free(fd)
    cc.free(od)
    assert sym.endswith("_n4k1_glu")
    assert np.array_equal(got, want)


@pytest.mark.parametrize("group,bf16", [(128, False), (32, True)])
@pytest.mark.parametrize("n,k,build", [(1, 640, "n1k4"), (19, 5120, "n1k4"), (423, 640, "n1k4"), (4097, 8448, "n4k1"), (8233, 640, "n2k4"),
                                       (17002, 384, "n3k4"), (33009, 256, "n5k2")])
def test_widths_that_are_no_multiple_of_four(dec, n, k, build, group, bf16):
    """Rows of y start at any element: the four-column stores are unaligned and the last columns go out one by one; whole
    and in k slices, f32 and f16."""
    for t in (18, 33, 64):
        print("odd width", n, k, t, group, bf16, flush=True)
        x = _upload(dec, n, k, group, bf16)
        want, _ = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, path=ops.PATH_LANE))
        got, sym = _run(dec, x, n, t, t * n, lambda xd, yd: dec.lin_forward("mid", xd, yd, t))
        assert sym.endswith("_" + build)
        parity.assert_close(got.view(np.float32).reshape(t, n), want.view(np.float32).reshape(t, n), "odd width %d t%d" % (n, t))
        h, _ = _run(dec, x, n, t, (t * n + 1) // 2, lambda xd, yd: dec.lin_forward("mid", xd, yd, t, out_f16=True))
        h = h.view(np.uint16)
        assert np.array_equal(h[:t * n], gen.f32_to_f16_bits(got.view(np.float32)).reshape(-1))
        assert t * n % 2 == 0 or h[t * n] == GUARD >> 16  # the half word behind the last element
