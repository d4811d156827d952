"""Launch plans of the decode, streaming and prefill paths as pure functions (w4a16_plan_*): no GPU.

The prefill planner is a price model with constants fitted to measurements; the table of those measurements that is
kept under profiles/ names, per layer shape, the (tile, k slices) that measured fastest.  This test feeds the planner
the same shapes and requires its choice to be that winner or a row the table shows within 3 % of it (the same plan's
time moves by 2-3 % between boxes, so closer rows trade places from one sweep to the next), so that a change to the
kernel or the constants that moves a plan shows up here."""
import os
import re

import pytest

from llm170_amd import ffi, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SWEEP = os.path.join(ROOT, "profiles", "prefill_plan_sweep.md")


def sweep_rows():
    """Rows `| n | k | t | tile | slices | us | note |` of the committed sweep table."""
    rows = []
    for ln in open(SWEEP):
        m = re.match(r"^\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*(\d+)\s*\|\s*([0-9.]+)\s*\|(.*)\|", ln)
        if m:
            rows.append(tuple(int(m.group(i)) for i in range(1, 6)) + (float(m.group(6)), m.group(7)))
    return rows


def test_prefill_plan_is_the_sweeps_winner_at_the_layer_shapes():
    rows = sweep_rows()
    shapes = sorted(set(r[:3] for r in rows))
    assert {(34816, 5120, 512), (34816, 5120, 1024), (34816, 5120, 4096), (5120, 17408, 512), (5120, 17408, 1024),
            (5120, 17408, 4096)} <= set(shapes)
    for (n, k, t) in shapes:
        cand = {(r[3], r[4]): r[5] for r in rows if r[:3] == (n, k, t)}
        best = min(cand.values())
        marked = [r[3:5] for r in rows if r[:3] == (n, k, t) and "plan" in r[6]]
        p = ops.plan_prefill(t, n, k, cu_count=256)
        pick = (p["tile_rows"], p["k_slices"])
        assert pick in cand, ("the sweep has no row for the planner's choice", n, k, t, pick)
        assert cand[pick] <= 1.03 * best, (n, k, t, pick, cand[pick], best)
        assert marked == [pick], ("the sweep marks another plan", n, k, t, marked, pick)


def visited(tiles_m, tiles_n, slices, sup_m, sup_n, bands):
    """(tile row, tile column, slice) of every workgroup, XCD by XCD, as kernels/prefill.hip numbers them (prefill_body)."""
    work, out = tiles_m * tiles_n * slices, []
    for xcd in range(8):
        run = []
        for b in range(-(-work // 8)):
            at = work * xcd // 8 + b
            if at >= work * (xcd + 1) // 8:
                continue
            r, sl = divmod(at, slices)
            so, si, to, ti = (sup_m, sup_n, tiles_m, tiles_n) if bands else (sup_n, sup_m, tiles_n, tiles_m)
            o, in_o = divmod(r, ti * so)
            wide = min(so, to - o * so)
            sup, in_super = divmod(in_o, si * wide)
            deep = min(si, ti - sup * si)
            i_n, i_m = divmod(in_super, wide if bands else deep)
            run.append(((o * so if bands else sup * si) + i_m, (sup * si if bands else o * so) + i_n, sl))
        out.append(run)
    return out


def check_walk(p, t, n, glu=False):
    cols = p.get("tile_cols", 256)
    tiles_m, tiles_n = -(-t // p["tile_rows"]), -(-(n // 2) // (cols // 2)) if glu else -(-n // cols)
    runs = visited(tiles_m, tiles_n, p["k_slices"], p["super_m"], p["super_n"], p["bands"])
    seen = [v for run in runs for v in run]
    assert len(set(seen)) == len(seen) == tiles_m * tiles_n * p["k_slices"], (t, n, p)
    assert all(0 <= m < tiles_m and 0 <= c < tiles_n for m, c, _ in seen), (t, n, p)
    assert max(map(len, runs)) - min(map(len, runs)) <= 1 and p["super_m"] < 2**15, (t, n, p)


def test_prefill_plan_walks_every_tile_and_pins_are_honoured():
    for (t, n, k) in [(4096, 34816, 5120), (1280, 5120, 17408), (100, 7168, 5120), (65, 256, 512), (2982, 848, 2048), (40000, 16, 512)]:
        p = ops.plan_prefill(t, n, k)
        check_walk(p, t, n)
        assert p["k_slices"] == 1 or p["k_slices"] <= (k // 128) // 4
    assert ops.plan_prefill(4096, 34816, 5120, tile_rows=64)["tile_rows"] == 64
    assert ops.plan_prefill(4096, 34816, 5120, tile_rows=96)["tile_rows"] == 96
    assert ops.plan_prefill(4096, 34816, 5120, k_slices=-1)["k_slices"] == 1
    assert ops.plan_prefill(512, 5120, 17408, k_slices=4)["k_slices"] == 4
    with pytest.raises(ops.W4a16Error):
        ops.plan_prefill(512, 5120, 17408, tile_rows=100)


def test_decode_plan_at_the_layer_shapes():
    """The shapes the launch-shape sweeps settled on (27B dense layer, group 128, 256 CUs)."""
    gate_up, down, qkv, o = (34816, 5120), (5120, 17408), (7168, 5120), (5120, 5120)
    want = {  # (n, k, t) -> (rows per wave, waves, k slices)
        gate_up + (1,): (16, 4, 1), gate_up + (4,): (32, 4, 1), gate_up + (16,): (64, 4, 1),
        down + (1,): (32, 4, 8), down + (4,): (32, 4, 8), down + (8,): (64, 4, 8), down + (16,): (64, 4, 8),
        qkv + (4,): (32, 8, 1), o + (4,): (32, 8, 1),
    }
    for (n, k, t), (rows, waves, nks) in want.items():
        p = ops.plan_decode(n, k, 128, t)
        assert (p["rows_per_wave"], p["waves_per_block"], p["k_slices"]) == (rows, waves, nks), (n, k, t, p)
        assert p["lds_bytes"] <= 160 * 1024


def test_decode_plan_of_small_outputs():
    """At most one row block per CU (256): the edges of the rule for k slices.  A narrow output with a long k is split,
    so that it does not stream its whole k from a few workgroups."""
    want = {  # (n, k tiles, t) -> (rows per wave, waves, k slices)
        (4096, 32, 1): (16, 8, 1), (4096, 32, 16): (16, 8, 1), (4112, 32, 1): (32, 8, 1),  # a row block more than CUs
        (4096, 63, 16): (16, 8, 1), (4096, 64, 16): (32, 4, 4),                            # a long k from 64 tiles
        (4096, 136, 6): (16, 8, 1), (4096, 136, 7): (32, 4, 4), (4096, 136, 9): (64, 4, 4), (4096, 128, 7): (64, 4, 4),
        (16, 136, 1): (16, 4, 8), (16, 136, 16): (16, 4, 8), (16, 63, 1): (16, 8, 1),      # one row block
        (128, 136, 4): (16, 4, 8), (144, 136, 4): (32, 4, 8), (336, 136, 4): (16, 4, 4),
        (512, 71, 4): (16, 8, 1), (512, 72, 4): (16, 4, 4), (1024, 87, 1): (16, 8, 1), (1024, 88, 1): (16, 4, 4),
        (2048, 103, 4): (16, 8, 1), (2048, 104, 4): (16, 4, 4), (2064, 136, 4): (16, 8, 1),
        (1024, 64, 5): (16, 8, 4), (1040, 75, 6): (16, 8, 1), (1040, 76, 6): (32, 4, 4), (2304, 112, 5): (32, 4, 7),
        (2064, 128, 5): (16, 8, 1), (2064, 136, 5): (32, 4, 8), (3088, 136, 5): (16, 8, 1),
        (1024, 136, 8): (32, 4, 8), (1040, 136, 8): (32, 4, 4), (2304, 112, 16): (64, 4, 7), (2304, 79, 16): (32, 4, 4),
    }
    for (n, kt, t), (rows, waves, nks) in want.items():
        p = ops.plan_decode(n, 128 * kt, 128, t)
        assert (p["rows_per_wave"], p["waves_per_block"], p["k_slices"]) == (rows, waves, nks), (n, kt, t, p)
    # no shape streams a long k from fewer waves than the 16-tile slices of four waves would bring, two row blocks each
    for n in range(16, 1025, 16):
        for kt in (104, 120, 136):
            for t in range(1, 17):
                p = ops.plan_decode(n, 128 * kt, 128, t)
                blocks = -(-n // p["rows_per_wave"])
                assert blocks * p["waves_per_block"] * p["k_slices"] >= -(-n // 64) * 4 * (kt // 16), (n, kt, t, p)


def test_decode_plan_takes_x_directly_where_few_waves_run():
    """At most four waves per CU: a wave's LDS holds its partial tiles (2 KiB at two row blocks) and scales, not staged
    x (4.25 KiB), up to the row count where staging wins; 5120 x 5120 is 160 workgroups of four waves."""
    scales = {128: 4 * 1024, 32: 4 * 3 * 1024}  # 2 row blocks x 10 k tiles x (1 or 4) groups x 32 B, in whole KiB
    for group, last in [(128, 11), (32, 14)]:
        for t in (9, last, last + 1, 16):
            p = ops.plan_decode(5120, 5120, group, t)
            assert (p["rows_per_wave"], p["waves_per_block"], p["k_slices"]) == (32, 4, 1)
            assert p["lds_bytes"] == 4 * (2048 if t <= last else 17 * 256) + scales[group], (group, t, p)
    # eight waves, five and six rows: staged x needs 2.25 KiB per wave; rows + k tiles per wave decide at group 128
    for kt, t, group, direct in [(40, 5, 128, True), (48, 5, 128, False), (32, 6, 128, True), (40, 6, 128, False), (32, 5, 32, False)]:
        p = ops.plan_decode(5120, 128 * kt, group, t)
        assert (p["rows_per_wave"], p["waves_per_block"]) == (32, 8)
        scales_w = -(-2 * (kt // 8) * (128 // group) * 32 // 1024) * 1024
        assert p["lds_bytes"] == 8 * ((2048 if direct else 9 * 256) + scales_w), (kt, t, group, p)
    # twice the row blocks: two workgroups per CU, staged from nine rows on
    p = ops.plan_decode(10240, 5120, 128, 9)
    assert p["lds_bytes"] == 4 * 17 * 256 + scales[128], p


def test_decode_plan_shrinks_to_fit_the_lds():
    """Group 32 with a long unsplit k: the staged scales of four row blocks per wave would pass 160 KiB (n = 16384,
    k = 53248, t = 8: 4 waves x 104 k tiles x 4 groups x 4 row blocks x 32 B = 213 KiB).  The plan halves the rows per
    wave instead of refusing the shape; the gated kernel (two row blocks by construction) cuts k into slices."""
    p = ops.plan_decode(16384, 53248, 32, 8)
    assert p["lds_bytes"] <= 160 * 1024 and p["rows_per_wave"] in (16, 32), p
    p = ops.plan_decode(16384, 53248, 128, 8)
    assert p["rows_per_wave"] == 64, "group 128 needs a quarter of that and keeps four row blocks"
    p = ops.plan_decode(16384, 106496, 32, 8, glu=True)
    assert p["lds_bytes"] <= 160 * 1024 and p["k_slices"] >= 2, p
    # staged x (4.25 KiB per wave from nine rows on) takes no shape away: it gives way to direct loads first
    p = ops.plan_decode(16, 128 * 9216, 32, 16)
    assert p["lds_bytes"] <= 160 * 1024 and p["k_slices"] == 8, p
    # nothing fits: a k range that even one row block per wave and eight slices cannot stage
    with pytest.raises(ops.W4a16Error) as e:
        ops.plan_decode(64, 128 * 20000, 32, 1)
    assert e.value.code == ffi.ERR_SHAPE and "LDS" in str(e.value)
    for bad in [(0, 128, 128, 1), (64, 100, 128, 1), (64, 128, 64, 1), (64, 128, 128, 17)]:
        with pytest.raises(ops.W4a16Error):
            ops.plan_decode(*bad)


def test_stream_plan_follows_the_sweep():
    """17..64 rows, the shape that measured fastest (or within 4 % of it) at widths and k on both sides of the rule's lines,
    among them those that a rule read from fewer widths gave a slower launch than the kernel before this one."""
    want = {  # (n, k tiles, t) -> (waves along n, waves along k, k slices)
        (13824, 136, 40): (4, 1, 4), (13824, 104, 64): (4, 1, 4), (13824, 40, 24): (2, 4, 1),  # 432 units: eight slices not resident
        (12288, 160, 48): (4, 1, 8), (12288, 120, 56): (4, 1, 4),                              # 384: eight are, at three token blocks
        (9216, 72, 24): (4, 1, 8), (9216, 86, 40): (4, 1, 8), (9216, 104, 64): (4, 1, 4), (9216, 40, 64): (2, 4, 1),
        (11008, 104, 32): (4, 1, 8), (17408, 136, 40): (4, 1, 4), (17408, 136, 64): (3, 4, 1), (28672, 160, 56): (4, 1, 2),
        (4096, 136, 24): (1, 4, 2), (3072, 136, 24): (1, 4, 2), (2560, 72, 24): (1, 4, 2), (2560, 33, 24): (1, 4, 1),
        (5120, 40, 64): (1, 4, 1), (5120, 136, 64): (4, 1, 8), (8192, 64, 64): (1, 4, 1), (8192, 136, 24): (4, 1, 8),
        (2048, 136, 24): (1, 4, 4), (2048, 16, 64): (1, 4, 1), (512, 136, 40): (1, 4, 8), (512, 16, 40): (1, 4, 1),
    }
    for (n, kt, t), shape in want.items():
        p = ops.plan_stream(n, 128 * kt, t)
        assert (p["waves_n"], p["waves_k"], p["k_slices"]) == shape, (n, kt, t, p)
    for (n, shape) in [(8192, (1, 4, 1)), (8224, (2, 4, 1)), (22016, (3, 4, 1)), (28672, (4, 2, 1)), (34816, (5, 2, 1)), (65536, (4, 1, 1))]:
        p = ops.plan_stream(n, 17408, 64, glu=True)  # the gated launch never splits
        assert (p["waves_n"], p["waves_k"], p["k_slices"]) == shape, (n, p)


def test_stream_plan_is_one_the_kernel_has():
    """Every launch shape is built, its slices hold two k tiles or more and are resident at once where four units share a
    workgroup, and a split launch needs less than 128 MiB of partial tiles, whatever the rows."""
    built = {(1, 4), (2, 4), (3, 4), (4, 1), (4, 2), (5, 2)}
    for n in list(range(16, 2100, 208)) + list(range(2100, 45000, 1337)) + [8224, 22016, 34816]:
        for kt in (1, 2, 7, 18, 31, 64, 90, 136, 300):
            for t in (1, 17, 33, 64, 65, 200, 1000):
                p = ops.plan_stream(n, 128 * kt, t)
                wn, wk, nks = p["waves_n"], p["waves_k"], p["k_slices"]
                assert (wn, wk) in built and nks in (1, 2, 4, 8), p
                assert nks == 1 or kt >= 2 * nks, p
                tt = 2 if t <= 32 else 3 if t <= 48 else 4
                groups = -(-((-(-n // 16) + 1) // 2) // wn) * -(-t // (16 * tt))
                if (wn, wk) == (4, 1) and nks > 1:
                    assert groups * nks <= 256 * (10 // tt), (n, kt, t, p)
                assert nks == 1 or groups * wn * 2 * tt * 1024 * nks < 2**27, (n, kt, t, p)
                if n % 32 == 0:
                    p = ops.plan_stream(n, 128 * kt, t, glu=True)
                    assert p["k_slices"] == 1 and (p["waves_n"], p["waves_k"]) in built, (n, kt, t, p)
    for bad in [(0, 128, 17), (64, 100, 17), (64, 128, 0)]:
        with pytest.raises(ops.W4a16Error):
            ops.plan_stream(*bad)


def test_prefill_plans_that_an_earlier_fit_lost():
    """Launches that a fit to fewer shapes made 7 to 17 % slower than the plans before it: the build that measured fastest of all (us, it
    / the one that fit chose)."""
    want = {  # (t, n, k, group, glu) -> (rows, columns, k groups, k slices)
        (105, 6336, 2176, 32, True): (64, 128, 4, 1),     # 17.0 / 19.8, 64 x 256 in four slices
        (193, 4096, 4096, 128, False): (64, 128, 4, 1),   # 18.8 / 21.8, 64 x 256 in four slices
        (122, 4160, 3072, 128, True): (64, 128, 4, 1),    # 15.6 / 17.4, 64 x 256 in six slices
        (319, 2816, 2688, 32, True): (64, 128, 4, 1),     # 19.5 / 21.8, 64 x 256 in four slices
        (542, 22016, 4096, 128, True): (128, 256, 1, 1),  # 103.6 / 118.8, 64 rows
        (553, 22016, 4096, 32, False): (128, 256, 1, 1),  # 135.5 / 151.3, 64 rows
        (644, 36048, 1280, 128, False): (96, 256, 1, 1),  # 67.4 / 76.9, 64 rows
        (83, 34816, 5120, 128, False): (96, 256, 1, 3),   # 45.9 / 50.9, five slices
        (409, 7168, 5120, 32, False): (64, 256, 1, 2),    # 57.7 / 62.8, four slices
    }
    for (t, n, k, g, glu), shape in want.items():
        p = ops.plan_prefill_launch(t, n, k, group=g, glu=glu)
        assert (p["tile_rows"], p["tile_cols"], p["k_groups"], p["k_slices"]) == shape, (t, n, k, g, glu, p)


def test_prefill_walk_where_an_xcds_eighth_is_resident():
    """The chip's own size decides what is resident at once: 3 x 256 blocks of the 64-row tile on 256 CUs, 3 x 128 on 128."""
    walk = lambda cus: {f: ops.plan_prefill(640, 12288, 512, cu_count=cus, tile_rows=64, k_slices=-1)[f] for f in ("super_m", "super_n", "bands")}
    assert walk(256) == {"super_m": 10, "super_n": 8, "bands": 1}  # 10 x 48 tiles, all rows in one band
    assert walk(128)["super_m"] == 8                               # 60 per XCD, 48 resident: super-tiles


def test_prefill_launch_plan():
    """What is launched with nothing pinned: k-group builds of 128 or 192 columns where the grid is at most one block tile per
    CU and they are priced below the 256-column tiles, which are otherwise those of plan_prefill.  The scale group decides too."""
    want = {  # (t, n, k, group) -> (columns, k groups, k slices)
        (300, 5120, 5120, 128): (128, 4, 1), (300, 7168, 5120, 128): (192, 4, 1), (300, 4096, 2048, 128): (128, 4, 1),
        (100, 1024, 640, 128): (128, 4, 1), (300, 5120, 2048, 32): (128, 4, 1), (65, 256, 512, 128): (128, 4, 1),
        (200, 5120, 5120, 128): (128, 4, 1), (200, 5120, 5120, 32): (256, 1, 6),
        (100, 5120, 2048, 128): (128, 4, 1), (100, 5120, 2048, 32): (128, 4, 1), (128, 592, 2560, 128): (256, 1, 4), (80, 1768, 1920, 32): (256, 1, 3),
        (128, 5120, 17408, 128): (256, 1, 6),  # 36.8 us; eight slices 38.5
        (512, 34816, 5120, 128): (256, 1, 1), (4096, 5120, 17408, 128): (256, 1, 1),
    }
    for (t, n, k, g), shape in want.items():
        p = ops.plan_prefill_launch(t, n, k, group=g)
        assert (p["tile_cols"], p["k_groups"], p["k_slices"]) == shape, (t, n, k, g, p)
    for t in (65, 100, 200, 300, 449, 640, 957, 1000):
        for n in (256, 1000, 1928, 4096, 5120, 7168, 12288, 34816):
            for k in (128, 640, 2048, 5120, 17408):
                for g in (128, 32):
                    for glu in (False, True):
                        if glu and n % 32:
                            continue
                        p = ops.plan_prefill_launch(t, n, k, group=g, glu=glu)
                        tiles_m, tiles_n = -(-t // p["tile_rows"]), -(-n // p["tile_cols"])
                        if p["k_groups"] == 4:
                            assert p["tile_rows"] == 64 and p["k_slices"] == 1 and tiles_m * tiles_n <= 256, p
                            assert p["bands"] == 1, p  # an XCD's eighth is resident: one band
                        elif not glu:
                            q = ops.plan_prefill(t, n, k, group=g)
                            assert p["tile_cols"] == 256 and all(p[f] == q[f] for f in q), (p, q)
                        check_walk(p, t, n, glu)
                        assert ops.plan_prefill_launch(t, n, k, group=g, glu=glu, whole_k=True)["k_slices"] == 1
    # a block tile per CU, and one more: 64 rows x 128 columns
    assert ops.plan_prefill_launch(64 * 16, 128 * 16, 640)["k_groups"] == 4
    assert ops.plan_prefill_launch(64 * 16 + 1, 128 * 16, 640)["tile_cols"] != 128
    with pytest.raises(ops.W4a16Error):
        ops.plan_prefill_launch(100, 1000, 640, glu=True)


def test_expert_plan_segments_and_tiled_line():
    """Mean runs on both sides of 24, 40 and 68 slots per expert, whatever the scales; the direct mode up to 15 tokens of top-8."""
    for scales, fam in ((0, "f16"), (1, "bf16"), (2, "f16x")):
        for t, seg in [(15, 1), (16, 32), (383, 32), (384, 48), (639, 48), (640, 64), (1087, 64), (1088, 64)]:
            p = ops.plan_moe(t, 8, 128, 2048, 768, 32, scales)
            assert p["segment"] == seg, (t, scales, p)
            tiled = t >= 1088
            if tiled:
                assert (p["gate_up"], p["down"]) == ("w4a16_moe_g32_%s_pf_glu" % fam, "w4a16_moe_g32_%s_pf_lin" % fam), p
            elif seg > 1:
                assert "_mm_glu_t%d" % (seg // 16) in p["gate_up"] and "_mm_lin_t%d" % (seg // 16) in p["down"], p
    assert ops.plan_moe(8, 9, 32, 2048, 768)["segment"] == 16 and ops.plan_moe(4, 9, 32, 2048, 768)["segment"] == 4
    for bad in [(0, 1, 4, 128, 128), (4, 5, 4, 128, 128), (4, 1, 4, 100, 128)]:
        with pytest.raises(ops.W4a16Error):
            ops.plan_moe(*bad)
    with pytest.raises(ops.W4a16Error):
        ops.plan_moe(100, 1, 4, 128, 128, 128, 2)


def test_expert_plan_folds_from_eight_k_tiles_and_eight_slots():
    def folds(t, n_exp, h, n_ff, top_k=8):
        p = ops.plan_moe(t, top_k, n_exp, h, n_ff, 32, 2)
        return "_f16x_" in p["gate_up"], "_f16x_" in p["down"]

    assert folds(517, 128, 2048, 768) == (True, False)                              # down: six k tiles
    assert folds(517, 128, 896, 1024) == (False, True)                              # gate|up: seven
    assert folds(517, 128, 1024, 896) == (True, False)
    assert folds(31, 32, 2048, 1024) == (False, False) and folds(32, 32, 2048, 1024) == (True, True)  # 248 and 256 slots
    # 32-slot segments: 20 waves per CU from one segment per expert, 5120 waves (units of 32 rows; 40 experts of 128 waves)
    assert folds(100, 40, 4096, 2048) == (True, True) and folds(100, 41, 4096, 2048) == (False, False)
    assert folds(240, 41, 4096, 2048) == (True, True)                               # 48-slot segments: however many
    for scales in (0, 1):
        p = ops.plan_moe(517, 8, 128, 2048, 1024, 32, scales)
        assert "f16x" not in p["gate_up"] + p["down"], p


def test_expert_plan_two_k_tiles_per_stage():
    def two(t, n_exp, h, n_ff, group, scales, top_k):
        p = ops.plan_moe(t, top_k, n_exp, h, n_ff, group, scales)
        return p["gate_up"].endswith("_k2"), p["down"].endswith("_k2")

    # group 32: one segment per expert at most one workgroup of four waves per CU (256 of them; n_ff 4096: 64 per expert, h 4096: 32)
    for scales in (0, 2):
        assert two(24, 4, 4096, 4096, 32, scales, 2) == (True, True)
        assert two(24, 5, 4096, 4096, 32, scales, 2) == (False, True)
        assert two(24, 8, 4096, 2048, 32, scales, 2) == (True, True) and two(24, 9, 4096, 2048, 32, scales, 2) == (False, False)
    assert two(24, 4, 4096, 4096, 32, 1, 2) == (False, False)                       # bf16 arenas: never
    # runs of 32 slots on: one tile
    assert two(127, 8, 4096, 2048, 32, 0, 2) == (True, True) and two(128, 8, 4096, 2048, 32, 0, 2) == (False, False)
    # group 128: at most three workgroups per CU, segments counted (768; 24 and 25 of them at n_ff 2048 and h 4096: 32 per segment)
    for scales in (0, 1):
        assert two(88, 19, 4096, 2048, 128, scales, 2) == (True, True)              # 176 slots: 5 + 19 segments
        assert two(96, 19, 4096, 2048, 128, scales, 2) == (False, False)            # 192: 6 + 19
