"""How the decode kernels take x from five rows on: whole rows re-ordered through LDS, or direct loads in operand order."""
import numpy as np
import pytest

from llm170_amd import gen, ops, parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    yield d
    d.cc.close()


@pytest.mark.parametrize("group,k,t", [(32, 128 * 1152, 7), (32, 128 * 1152, 16), (128, 128 * 4608, 16)])
def test_pinned_shape_without_room_for_staged_x(dec, orc, group, k, t):
    """Eight waves over an unsplit k whose staged scales (144 KiB) leave room for the partial tiles, not for staged x."""
    print("no room", group, k, t, flush=True)
    n = 16
    q, s, x = gen.make_linear(n, k, group, t, seed=k + t)
    dec.upload_lin_g("long", q, s, n, k, group, False)
    try:
        dec.set_decode_shape(16, 8)
        dec.set_decode_ksplit(-1)
        got = dec.gemv_host("long", x, t=t, path=ops.PATH_DECODE)
        assert dec.cc.last_launch_symbol().endswith("_rb1_x%dd" % (2 if t <= 8 else 4))
    finally:
        dec.set_decode_shape(0, 0)
        dec.set_decode_ksplit(0)
    parity.assert_close(got, orc.gemm_lane(x, t, q, s, n, k, group), "k%d g%d t%d" % (k, group, t))


def test_pinned_gated_shape_without_room_for_staged_x(dec):
    """The gated kernel likewise (128 KiB of scales), against the plain launch of the same shape and the activation."""
    n, k, group, t = 32, 128 * 512, 32, 16
    print("no room, gated", n, k, group, t, flush=True)
    q, s, x = gen.make_linear(n, k, group, t, seed=3)
    dec.upload_lin_g("longglu", q, s, n, k, group, False)
    cc = dec.cc
    xd, gu, a, b = cc.to_device(x), cc.alloc(t * n * 4), cc.alloc(t * n), cc.alloc(t * n)
    try:
        dec.set_decode_shape(32, 8)
        dec.set_decode_ksplit(-1)
        dec.lin_forward_glu("longglu", xd, a, t)
        assert cc.last_launch_symbol().endswith("_glu_x4d")
        dec.lin_forward("longglu", xd, gu, t, path=ops.PATH_DECODE)
        assert cc.last_launch_symbol().endswith("_rb2_x4d")
        dec.silu_mul_f16(gu, n // 2, t, b)
        got, want = cc.d2h(a, (t, n // 2), np.uint16), cc.d2h(b, (t, n // 2), np.uint16)
    finally:
        dec.set_decode_shape(0, 0)
        dec.set_decode_ksplit(0)
        for p in (xd, gu, a, b):
            cc.free(p)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("group,rows,waves,t,direct", [
    (128, 16, 4, 5, True), (128, 32, 4, 8, True), (128, 32, 4, 9, True), (128, 32, 4, 11, True), (128, 32, 4, 12, False),
    (32, 16, 4, 8, True), (32, 32, 4, 8, False), (32, 32, 4, 14, True), (32, 32, 4, 15, False),
    (128, 64, 4, 13, True), (128, 64, 4, 14, False),
    (128, 32, 8, 8, True), (32, 32, 8, 8, False), (128, 16, 8, 8, False), (32, 64, 8, 8, True), (128, 64, 8, 9, False),
])
def test_short_launches_take_x_directly_with_the_same_bits(dec, group, rows, waves, t, direct):
    """One workgroup per CU at most and few k tiles per wave: the rule's edges, and every row's bits as in the 16-row
    launch (x through LDS), whose sums run in the same order."""
    print("short", group, rows, waves, t, flush=True)
    n, k = 200, 1280  # a partial row block; ten k tiles on four or eight waves
    q, s, x = gen.make_linear(n, k, group, 16, seed=group + rows + t)
    dec.upload_lin_g("few", q, s, n, k, group, False)
    try:
        dec.set_decode_shape(rows, waves)
        want = dec.gemv_host("few", x, t=16, path=ops.PATH_DECODE)
        assert dec.cc.last_launch_symbol().endswith("_rb%d_x4" % (rows // 16))
        got = dec.gemv_host("few", np.ascontiguousarray(x[:t]), t=t, path=ops.PATH_DECODE)
        assert dec.cc.last_launch_symbol().endswith("d") == direct
    finally:
        dec.set_decode_shape(0, 0)
    assert np.array_equal(got.view(np.uint32), want[:t].view(np.uint32))
