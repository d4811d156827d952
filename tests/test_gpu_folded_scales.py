"""Group 32 with bf16 scales: (nibble - 8) * scale as an f16 weight.  The builds that fold the scale and those that scale group sums,
against float64 sums of the dequantised weights, at the edges of the tiles and of the scales' range."""
import numpy as np
import pytest

from llm170_amd import gen, ops

pytestmark = pytest.mark.gpu

LO, HI, WIDE = 0x3880, 0x45FF, 0x4600  # 2^-14; 8160, the last bf16 below 2^13; 2^13


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    yield d
    d.cc.close()


def _linear(n, k, t, wide, seed=91):
    q, s, x = gen.make_linear(n, k, 32, t, seed=seed)
    s = (gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16)
    s[0, :], s[1 % n, 0], s[n - 1, -1] = LO, WIDE if wide else HI, LO  # every nibble meets the smallest, some the largest
    return q, s, x


def _weights(q, s, k):
    return gen.unpack_nibbles(q, k).astype(np.float64) * np.repeat((s.astype(np.uint32) << 16).view(np.float32).astype(np.float64), 32, axis=-1)


def _bound(x, w):
    """Sums in f32 in any order: every one of the k products is exact, and every addition rounds by at most 2^-24 of a partial sum,
    itself at most the sum of the magnitudes; the chain of additions of one output is no longer than k / 8 (an MFMA adds its
    products in a tree of at least eight) plus the 64 that scaled groups, parts and slices can add."""
    return (w.shape[1] / 8 + 64) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


def _check(dec, n, k, t, wide, call, glu=False):
    q, s, x = _linear(n, k, t, wide)
    dec.upload_lin_g("fold", q, s, n, k, 32, True)
    xd, yd = dec.cc.to_device(x), dec.cc.to_device(np.zeros((t, n), np.float32))
    try:
        call(xd, yd)
        y = dec.cc.d2h(yd, (t, n // 2) if glu else (t, n), np.uint16 if glu else np.float32)
    finally:
        dec.cc.free(xd)
        dec.cc.free(yd)
    cols = np.unique(np.concatenate([np.arange(min(n, 20)), np.random.default_rng(n).integers(0, n, 400), np.arange(max(0, n - 20), n)]))
    if glu:
        cols = np.unique(cols % (n // 2))
        y, cols = y[:, cols], np.concatenate([cols, cols + n // 2])
    else:
        y = y[:, cols]
    n, q, s = len(cols), q[cols], s[cols]
    xf, w = gen.f16_bits_to_f32(x).astype(np.float64), _weights(q, s, k)
    ref, bound = xf @ w.T, _bound(xf, w)
    if not glu:
        assert np.all(np.abs(y - ref) <= bound), float(np.max(np.abs(y - ref) / bound))
        return
    g, u, bg, bu = ref[:, :n // 2], ref[:, n // 2:], bound[:, :n // 2], bound[:, n // 2:]
    with np.errstate(over="ignore"):
        act = g / (1.0 + np.exp(-g))
    # |d silu / d g| <= 1.1; expf and the division of the activation: a few f32 units; then one rounding to f16
    err = 1.1 * bg * np.abs(u) + np.abs(act) * bu + 1.1 * bg * bu + 2.0 ** -20 * np.abs(act * u)
    ok = np.abs(act * u) + err < 65504.0
    err += np.maximum(2.0 ** -11 * (np.abs(act * u) + err), 2.0 ** -25)
    assert np.all(np.abs(gen.f16_bits_to_f32(y) - act * u)[ok] <= err[ok])


# a build of each number of waves; row blocks and rows past a multiple of 16; k tiles that do not divide by the four parts; the last
# three: one k tile fewer than a slice needs to fold, k in slices that fold, k in slices that do not
SHAPES = [(40, 3072), (4104, 3200), (8232, 3072), (17000, 3328), (27016, 3072), (33008, 3072), (4104, 2944), (2048, 17408), (512, 8192)]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("t", [17, 33, 64])
def test_streaming_rows(dec, n, k, t, wide):
    print("fold mid", n, k, t, wide, flush=True)
    _check(dec, n, k, t, wide, lambda xd, yd: dec.lin_forward("fold", xd, yd, t))
    folds = not wide and k // 128 >= 24 * ops.plan_stream(n, k, t)["k_slices"]
    assert dec.cc.last_launch_symbol().startswith("w4a16_mid_g32_%s_t" % ("bf16x" if folds else "bf16"))


@pytest.mark.parametrize("n,k", [(4104, 3200), (17000, 3328), (27016, 3072), (33008, 3072), (2048, 17408)])
@pytest.mark.parametrize("t", [17, 64])
def test_streaming_sums_no_further_from_64_bits(dec, n, k, t):
    """The distance that decides where linears fold, on the rows of ordinary scales: over the rms of the sums, of the builds left to the
    library and of those a single scale that does not fold selects.  4 k / 128 additions of group sums, each rounding a partial sum that
    grows as a random walk by 2^-24 / sqrt 3 at most, are sqrt(2 k / 128) of them; the two distances are equal to the spread of an rms
    over 400 columns x 17 rows (1 %) where few k tiles are folded, a tenth is allowed."""
    print("fold distance", n, k, t, flush=True)
    far = []
    for wide in (False, True):
        q, s, x = _linear(n, k, t, wide)
        dec.upload_lin_g("far", q, s, n, k, 32, True)
        xd, yd = dec.cc.to_device(x), dec.cc.alloc(t * n * 4)
        try:
            dec.lin_forward("far", xd, yd, t)
            y = dec.cc.d2h(yd, (t, n), np.float32)
        finally:
            dec.cc.free(xd)
            dec.cc.free(yd)
        cols = np.unique(np.random.default_rng(n).integers(2, n - 1, 400))
        ref = gen.f16_bits_to_f32(x).astype(np.float64) @ _weights(q[cols], s[cols], k).T
        far.append(float(np.sqrt(np.mean((y[:, cols] - ref) ** 2) / np.mean(ref ** 2))))
    print("distance: %.3g, scaled sums %.3g" % tuple(far), flush=True)
    assert max(far) <= np.sqrt(2.0 * k / 128) * 2.0 ** -24 / np.sqrt(3.0)
    assert far[0] <= 1.1 * far[1]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("t", [17, 40, 64])
def test_gated(dec, t, wide):
    print("fold glu", t, wide, flush=True)
    _check(dec, 544, 3200, t, wide, lambda xd, yd: dec.lin_forward_glu("fold", xd, yd, t), glu=True)
    assert dec.cc.last_launch_symbol().startswith("w4a16_mid_g32_%s_t" % ("bf16" if wide else "bf16x"))


def test_fused_parts_fold_only_together(dec):
    """A linear fused of one part that folds and one that does not runs the builds that take any scale."""
    n, k, t = 4096, 3072, 20
    for name, wide in (("a", False), ("b", True)):
        q, s, x = _linear(n, k, t, wide)
        dec.upload_lin_g(name, q, s, n, k, 32, True)
    xd, yd = dec.cc.to_device(x), dec.cc.alloc(t * 2 * n * 4)
    for parts in (["a", "b"], ["b", "a"]):
        dec.lin_fuse("ab", parts)
        dec.lin_forward("ab", xd, yd, t)
        assert dec.cc.last_launch_symbol().startswith("w4a16_mid_g32_bf16_")
    dec.lin_forward("a", xd, yd, t)
    assert dec.cc.last_launch_symbol().startswith("w4a16_mid_g32_bf16x_")
    dec.cc.free(xd)
    dec.cc.free(yd)


@pytest.mark.parametrize("block,runs", [(32, [1, 16, 17, 32, 33, 0, 5]), (32, [9, 7, 8, 8]), (32, [7, 9, 8, 7]), (48, [48, 47, 31, 1, 49, 33]), (64, [64, 65, 63, 49, 17, 16]),
                                        (0, [70, 1, 33, 64, 0, 97])])
@pytest.mark.parametrize("wide", [False, True])
def test_experts(dec, block, runs, wide):
    """Runs that end at and around 16-slot blocks and segments; block 0: the MFMA-tiled kernels.  top_k = 1, weight 1: y is a slot's
    f16 row.  The activation is compared first, then the down projection of the activation the device wrote."""
    print("fold experts", block, runs, wide, flush=True)
    E, t, h, n_ff = len(runs), sum(runs), 384, 256
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, 32, seed=gen.GATE_SEED + 23)
    s13, s2 = ((gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16) for s in (s13, s2))
    s13[:, 0, :] = s2[:, 1, :] = LO
    if wide:
        s13[0, 5, 1] = 0x3800  # 2^-15: no f16 normal
    dec.upload_experts("fold", q13, s13, q2, s2, E, h, n_ff, 32, True)
    idx = np.random.default_rng(5).permutation(np.repeat(np.arange(E), runs)).astype(np.int32)[:, None]
    x = gen.normal_f16(80, (t, h))
    cc = dec.cc
    bufs = [cc.to_device(x), cc.to_device(idx), cc.to_device(np.ones((t, 1), np.float32)), cc.to_device(np.zeros((t, h), np.float32))]
    dec.set_moe_shape(block, 0)
    dec.set_moe_tiled(0 if block else 1)
    try:
        dec.moe_ffn("fold", *bufs[:3], t, 1, bufs[3])
        y, act = cc.d2h(bufs[3], (t, h), np.float32), dec.moe_scratch(3, np.uint16)[0].reshape(t, n_ff)
    finally:
        dec.set_moe_shape(0, 0)
        dec.set_moe_tiled(0)
        for b in bufs:
            cc.free(b)
    xf, af = gen.f16_bits_to_f32(x).astype(np.float64), gen.f16_bits_to_f32(act).astype(np.float64)
    for e in range(E):
        rows = np.nonzero(idx[:, 0] == e)[0]
        w13, w2 = _weights(q13[e], s13[e], h), _weights(q2[e], s2[e], n_ff)
        gu, bgu = xf[rows] @ w13.T, _bound(xf[rows], w13)
        bgu = bgu + 2.0 ** -11 * (np.abs(gu) + bgu) + 2.0 ** -25  # gate and up are rounded to f16
        g, u, bg, bu = gu[:, :n_ff], gu[:, n_ff:], bgu[:, :n_ff], bgu[:, n_ff:]
        silu = g / (1.0 + np.exp(-g))
        err = 1.1 * bg * np.abs(u) + np.abs(silu) * bu + 1.1 * bg * bu + 2.0 ** -20 * np.abs(silu * u)
        err += 2.0 ** -11 * (np.abs(silu * u) + err) + 2.0 ** -25
        assert np.all(np.abs(af[rows] - silu * u) <= err), (e, "act")
        down, bd = af[rows] @ w2.T, _bound(af[rows], w2)
        assert np.all(np.abs(y[rows] - down) <= bd + 2.0 ** -11 * (np.abs(down) + bd) + 2.0 ** -25), (e, "down")


def _misrounded(dec, name, x, idx, h, n_ff, w2):
    """Number of f16 rows' values that are not the nearest f16 to the 64-bit sum of the device's activation and w2 (values of at least
    half the rms).  A sum that is off by err lands on the wrong side of a rounding boundary with a chance of err / ulp, so the number
    grows in proportion to the mean distance of the f32 sums from 64-bit ones."""
    t, cc = len(idx), dec.cc
    bufs = [cc.to_device(x), cc.to_device(idx), cc.to_device(np.ones((t, 1), np.float32)), cc.to_device(np.zeros((t, h), np.float32))]
    try:
        dec.moe_ffn(name, *bufs[:3], t, 1, bufs[3])
        y, act = cc.d2h(bufs[3], (t, h), np.float32), dec.moe_scratch(3, np.uint16)[0].reshape(t, n_ff)
    finally:
        for b in bufs:
            cc.free(b)
    count = 0
    for e in np.unique(idx):
        rows = np.nonzero(idx[:, 0] == e)[0]
        ref = gen.f16_bits_to_f32(act[rows]).astype(np.float64) @ w2(e).T
        wrong = y[rows] != ref.astype(np.float16).astype(np.float32)
        count += int(np.count_nonzero(wrong & (np.abs(ref) > 0.5 * np.sqrt(np.mean(ref * ref)))))
    return count


@pytest.mark.parametrize("block", [32, 48, 64, 0])
@pytest.mark.parametrize("n_ff", [768, 1024, 3584])
def test_expert_sums_no_further_from_64_bits(dec, n_ff, block):
    """Experts whose scales fold against the same experts next to one that has a negative scale and no token, which run the builds that
    do not fold.  Misrounded values are independent rare events: five standard deviations of the difference of two equal counts.
    Block 0: the MFMA-tiled kernels."""
    print("fold sums", n_ff, block, flush=True)
    E, t, h = 3, 1024, 4096
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, 32, seed=gen.GATE_SEED + 31)
    s13, s2 = ((gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16) for s in (s13, s2))
    x, idx = gen.normal_f16(81, (t, h)), (np.arange(t, dtype=np.int32) % 2)[:, None].copy()
    counts = []
    for negative in (False, True):
        s13[2, 0, 0] = (s13[2, 0, 0] & 0x7FFF) | (0x8000 if negative else 0)
        dec.upload_experts("sums", q13, s13, q2, s2, E, h, n_ff, 32, True)
        dec.set_moe_shape(block, 0)
        dec.set_moe_tiled(0 if block else 1)
        try:
            counts.append(_misrounded(dec, "sums", x, idx, h, n_ff, lambda e: _weights(q2[e], s2[e], n_ff)))
        finally:
            dec.set_moe_shape(0, 0)
            dec.set_moe_tiled(0)
    fold, scaled = counts
    print("misrounded: folded %d, scaled %d" % (fold, scaled), flush=True)
    assert fold <= scaled + 5.0 * np.sqrt(2.0 * scaled)


@pytest.mark.parametrize("bf16,run", [(True, 50), (False, 64), (False, 67)])
def test_expert_route_of_medium_runs_keeps_the_sums(dec, bf16, run):
    """Mean runs of 40 to 67 slots, as many block tiles as any rule asks for: left to the library the sums are no further from 64 bits
    than those of the streaming kernels (64-slot segments pinned).  Bounds as above."""
    print("medium runs", bf16, run, flush=True)
    E, h, n_ff = 32, 1024, 2048
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, 32, seed=gen.GATE_SEED + 37)
    if bf16:
        s13, s2 = ((gen.f16_bits_to_f32(s).view(np.uint32) >> 16).astype(np.uint16) for s in (s13, s2))
    value = (lambda s: (s.astype(np.uint32) << 16).view(np.float32)) if bf16 else gen.f16_bits_to_f32
    w2 = lambda e: gen.unpack_nibbles(q2[e], n_ff).astype(np.float64) * np.repeat(value(s2[e]).astype(np.float64), 32, axis=-1)
    x, idx = gen.normal_f16(82, (E * run, h)), (np.arange(E * run, dtype=np.int32) % E)[:, None].copy()
    dec.upload_experts("medium", q13, s13, q2, s2, E, h, n_ff, 32, bf16)
    counts = []
    for block in (0, 64):
        dec.set_moe_shape(block, 0)
        try:
            counts.append(_misrounded(dec, "medium", x, idx, h, n_ff, w2))
        finally:
            dec.set_moe_shape(0, 0)
    print("misrounded: automatic %d, streaming %d" % tuple(counts), flush=True)
    assert counts[0] <= counts[1] + 5.0 * np.sqrt(2.0 * counts[1])
