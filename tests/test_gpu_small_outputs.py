"""Decode launches of outputs with at most one 16-row block per CU: one row block per wave, up to eight waves; a long k in
slices, over one, two or four row blocks per wave; x rows re-ordered through LDS or loaded directly (five to sixteen
rows).  The edges of those ranges against the lane-order oracle."""
import numpy as np
import pytest

from llm170_amd import gen, ops, parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,group,t", [
    (4096, 512, 128, 1), (4096, 512, 128, 16),   # the last size with one row block per workgroup
    (4112, 512, 128, 9),                         # one row block more: two per wave
    (17, 1024, 32, 5), (1, 128, 128, 8),         # a partial row block; fewer k tiles than waves
    (272, 4096, 128, 13), (272, 4096, 32, 6),    # eight waves of four k tiles: the load ring and staged x go round
    (96, 8192, 128, 6), (96, 8192, 128, 7),      # a long k: one row block per wave up to six rows, two from seven
    (96, 8192, 32, 16), (80, 8320, 128, 13),     # 65 k tiles in four slices: the last one short
    (16, 17408, 128, 4), (144, 17408, 32, 3),    # one row block; two per wave in eight slices
    (528, 9472, 128, 2), (528, 9472, 32, 6),     # 74 k tiles in four slices of four and of eight waves
    (1040, 9728, 128, 5), (2064, 10240, 128, 9), # two and four row blocks per wave, a partial last group
])
def test_small_outputs(orc, n, k, group, t):
    print("small outputs", n, k, group, t, flush=True)
    dec = ops.W4a16Dec()
    try:
        q, s, x = gen.make_linear(n, k, group, t, seed=n + k + t)
        dec.upload_lin_g("s", q, s, n, k, group, False)
        want = orc.gemm_lane(x, t, q, s, n, k, group)
        for _ in range(2):  # the tickets of a split launch are left at zero
            got = dec.gemv_host("s", x, t=t, path=ops.PATH_DECODE)
            parity.assert_close(got, want, "n%d k%d g%d t%d" % (n, k, group, t))
        got16 = dec.gemv_host("s", x, t=t, out_f16=True, path=ops.PATH_DECODE)
        assert np.array_equal(got16, gen.f32_to_f16_bits(got))
    finally:
        dec.cc.close()


@pytest.mark.parametrize("t", [1, 8])
def test_pinned_rows_keep_their_slices(t):
    """32 rows per wave pinned, and the launch with one output per part (built for 32): a long k over few workgroups
    runs in eight slices of four waves, at any row count, whatever the automatic row count would do."""
    print("pinned rows", t, flush=True)
    n, k = 512, 16384
    dec = ops.W4a16Dec()
    cc = dec.cc
    try:
        q, s, x = gen.make_linear(n, k, 128, t, seed=t)
        dec.upload_lin_g("a", np.ascontiguousarray(q[:256]), np.ascontiguousarray(s[:256]), 256, k, 128, False)
        dec.upload_lin_g("b", np.ascontiguousarray(q[256:]), np.ascontiguousarray(s[256:]), 256, k, 128, False)
        dec.lin_fuse("ab", ["a", "b"])
        xd, ya, yb = cc.to_device(x), cc.alloc(t * 256 * 4), cc.alloc(t * 256 * 4)
        dec.lin_forward_multi("ab", xd, [ya, yb], t)
        multi = np.concatenate([cc.d2h(ya, (t, 256), np.uint32), cc.d2h(yb, (t, 256), np.uint32)], axis=1)
        dec.set_decode_shape(32, 0)
        auto = dec.gemv_host("ab", x, t=t, path=ops.PATH_DECODE).view(np.uint32)
        dec.set_decode_shape(32, 4)
        sliced = {}
        for slices in (4, 8):
            dec.set_decode_ksplit(slices)
            sliced[slices] = dec.gemv_host("ab", x, t=t, path=ops.PATH_DECODE).view(np.uint32)
    finally:
        dec.cc.close()
    assert not np.array_equal(sliced[4], sliced[8])  # another order of the same sums
    assert np.array_equal(auto, sliced[8]) and np.array_equal(multi, sliced[8])
