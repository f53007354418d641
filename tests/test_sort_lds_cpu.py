"""The LDS of the radix sort's scatter kernel, as the compiler allocates it.

The instances that add up the tiles' digit counts themselves keep two sums of
256 words for each of 4 waves while the waves' own counts (4 x 256 words), the
digits' offsets (256 words) and the scan's sums exist: an allocation smaller
than their total means that some of them share storage they must not share.
"""
import os
import re
import subprocess

import pytest

from illcrawl_amd import build as hipbuild

SUMS, WAVE_COUNTS, OFFSETS, SCAN = 2 * 4 * 256 * 4, 4 * 256 * 4, 256 * 4, 4 * 4


@pytest.fixture(scope="module")
def lds(tmp_path_factory):
    """{(items, carries a second value, adds up the counts): LDS bytes}"""
    out = tmp_path_factory.mktemp("lds") / "grid.o"
    cmd = [hipbuild.hipcc(), "-O3", "-std=c++17", f"--offload-arch={hipbuild.ARCH}",
           "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage",
           "-I", os.path.join(hipbuild.ROOT, "include"), "-I", hipbuild.CSRC, "-x", "hip", "-c",
           os.path.join(hipbuild.CSRC, "grid.hip"), "-o", str(out)] + hipbuild.DEVICE_FLAGS
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    got = {}
    for name, size in re.findall(r"Function Name: (\S+).*?LDS Size \[bytes/block\]: (\d+)",
                                 r.stderr, re.S):
        m = re.search(r"k_radix_scatterILi(\d+)ELb([01])ELb([01])E", name)
        if m:
            got[int(m[1]), m[2] == "1", m[3] == "1"] = int(size)
    assert len(got) == 6, sorted(got)
    return got


@pytest.mark.parametrize("items,second,small", [
    (4, False, True), (4, True, True), (16, False, True), (16, True, True), (16, False, False),
    (16, True, False)])
def test_scatter_holds_its_arrays(lds, items, second, small):
    tile = 256 * items * 4
    need = max(tile, SUMS if small else 0) + WAVE_COUNTS + OFFSETS + SCAN
    assert lds[items, second, small] >= need
