"""Sizes of the built tiled kernels: what a launch of ten microseconds fetches cold.  A gated launch has one epilogue, or stores partial sums: its code is no longer than that of the
plain kernel of the same tile, which has more.  The arguments fill two lines of 64 bytes."""
import os
import re
import struct
import subprocess

import pytest

from llm170_amd import build


def _code_bytes(path):
    """Function symbols of an ELF64 code object: name -> bytes."""
    blob = open(path, "rb").read()
    assert blob[:5] == b"\x7fELF\x02"
    sec_at, = struct.unpack_from("<Q", blob, 0x28)
    size, count = struct.unpack_from("<HH", blob, 0x3A)
    secs = [struct.unpack_from("<IIQQQQIIQQ", blob, sec_at + i * size) for i in range(count)]
    out = {}
    for _, kind, _, _, at, length, link, _, _, each in secs:
        if kind != 2:  # SHT_SYMTAB
            continue
        names = secs[link][4]
        for i in range(0, length, each):
            name, info, _, _, _, nbytes = struct.unpack_from("<IBBHQQ", blob, at + i)
            if info & 15 == 2:  # STT_FUNC
                end = blob.index(b"\0", names + name)
                out[blob[names + name:end].decode()] = nbytes
    return out


@pytest.mark.parametrize("asset", ["prefill", "prefill_g128"])
def test_gated_kernels_are_no_longer_than_plain_ones(asset):
    sizes = _code_bytes(os.path.join(build.ASSET_DIR, asset + ".hsaco"))
    pairs = [(n, n + "_glu") for n in sizes if n.startswith("w4a16_prefill_g") and n + "_glu" in sizes]
    assert len(pairs) >= 10, sizes
    for plain, gated in pairs:
        assert sizes[gated] <= sizes[plain], (plain, sizes[plain], sizes[gated])


@pytest.mark.parametrize("asset", ["prefill", "prefill_g128"])
def test_arguments_fill_two_lines(asset):
    notes = subprocess.run([os.path.join(build.ROCM, "llvm", "bin", "llvm-readelf"), "--notes", os.path.join(build.ASSET_DIR, asset + ".hsaco")],
                           capture_output=True, text=True, check=True).stdout
    found = []
    for kernel in re.split(r"- \.agpr_count", notes)[1:]:
        name = re.search(r"\.symbol:\s*(\w+)\.kd", kernel).group(1)
        if name.startswith("w4a16_prefill_g"):
            found.append((name, int(re.search(r"\.kernarg_segment_size:\s*(\d+)", kernel).group(1))))
    assert len(found) == 20, found
    assert all(size <= 128 for _, size in found), found
