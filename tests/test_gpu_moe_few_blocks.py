"""Expert FFNs at group 128 whose launches have few workgroups: the LDS-staged kernel with two k tiles per stage, at every
remainder of the k tiles by the two stages in flight, against the oracle and, bit for bit, against one tile per stage (64-slot
segments have no other build and add up in the same order)."""
import numpy as np
import pytest

from llm170_amd import gen, ops

from .test_gpu_moe import _bf16_scales, _check_ffn, _run_ffn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dec():
    d = ops.W4a16Dec()
    yield d
    d.cc.close()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("h,n_ff", [(128, 256), (384, 512), (640, 768), (1152, 896)])
@pytest.mark.parametrize("runs,block", [([1, 16, 17, 0, 31, 32, 33, 5], 32), ([48, 16, 0, 33, 32, 47], 48)])
def test_two_k_tiles_per_stage(dec, orc, h, n_ff, runs, block, bf16):
    print("few blocks", h, n_ff, runs, bf16, flush=True)
    E, t = len(runs), sum(runs)
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, 128, seed=gen.GATE_SEED + 23)
    if bf16:
        s13, s2 = _bf16_scales(s13), _bf16_scales(s2)
        s13[0, 0, 0] = s2[0, 0, 0] = (127 - 20) << 7  # 2^-20: no normal f16 number, the arenas stay bf16
    dec.upload_experts("few", q13, s13, q2, s2, E, h, n_ff, 128, bf16)
    idx = np.random.default_rng(7).permutation(np.repeat(np.arange(E), runs)).astype(np.int32)[:, None]
    wt = (0.25 + np.random.default_rng(8).random((t, 1))).astype(np.float32)
    x = gen.normal_f16(83, (t, h))
    y, act, c2, blk = _run_ffn(dec, "few", x, idx, wt, t, 1, h)
    assert blk == block
    _check_ffn(orc, y, act, c2, x, idx, wt, q13, s13, q2, s2, h, n_ff, 128, bf16, "few blocks")
    dec.set_moe_shape(64, 0)
    try:
        y64, act64, c64, blk = _run_ffn(dec, "few", x, idx, wt, t, 1, h)
    finally:
        dec.set_moe_shape(0, 0)
    assert blk == 64
    assert np.array_equal(y, y64) and np.array_equal(act, act64) and np.array_equal(c2, c64)


@pytest.mark.parametrize("fold", [False, True])
@pytest.mark.parametrize("h,n_ff", [(128, 256), (384, 512), (640, 768), (1152, 896), (256, 2176)])
@pytest.mark.parametrize("runs,block", [([1, 16, 17, 0, 31, 32, 33, 5], 32), ([48, 16, 0, 33, 32, 47], 48), ([1, 2, 3, 0, 17, 5, 1, 2], 32)])
def test_two_k_tiles_per_stage_group_32(dec, h, n_ff, runs, block, fold):
    """Bit for bit against one tile per stage, which 64-slot segments have; n_ff 2176: more than one workgroup per CU."""
    print("few blocks, group 32", h, n_ff, runs, fold, flush=True)
    E, t = len(runs), sum(runs)
    q13, s13, q2, s2 = gen.make_experts(E, h, n_ff, 32, seed=gen.GATE_SEED + 29)
    if fold:
        s13, s2 = _bf16_scales(s13), _bf16_scales(s2)
    dec.upload_experts("few32", q13, s13, q2, s2, E, h, n_ff, 32, fold)
    idx = np.random.default_rng(9).permutation(np.repeat(np.arange(E), runs)).astype(np.int32)[:, None]
    wt = (0.25 + np.random.default_rng(10).random((t, 1))).astype(np.float32)
    x = gen.normal_f16(84, (t, h))
    got = []
    for b in (block, 64):
        dec.set_moe_shape(b, 0)
        try:
            *out, blk = _run_ffn(dec, "few32", x, idx, wt, t, 1, h)
        finally:
            dec.set_moe_shape(0, 0)
        assert blk == b and all(np.all(np.isfinite(o.view(np.float16) if o.dtype == np.uint16 else o)) for o in out)
        got.append(out)
    assert all(np.array_equal(a, b) for a, b in zip(*got))
