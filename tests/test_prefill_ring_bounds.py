"""Every activation read of the prefill gate/up ring lies within its stage, and within the LDS: block b of token tile
u + j is read at 1 KB x (4 (u + j) + b) + 16 lane past the stage's activations (mx_ring.h, as the kernel computes it)."""

import ctypes as C
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "vesper_amd" / "libmxmoe_hostcheck.so"


@pytest.mark.parametrize("live", range(1, 9))
def test_reads_stay_within_the_live_tiles(live):
    assert LIB.exists(), "build first: python -m vesper_amd.build"
    lib = C.CDLL(str(LIB))
    read = set()
    for u in range(0, live, 4):
        out = (C.c_int32 * 5)()
        lib.mxh_prefill_ring(live, u, out)
        stage, stages, lds, acts, count = out
        assert stage == acts + 4096 * live and 2 <= stages <= 4 and stages * stage <= lds <= 160 * 1024
        for j in range(count):
            read.add(u + j)
            last = 1024 * (4 * (u + j) + 3) + 16 * 63 + 16
            assert acts + last <= stage and (stages - 1) * stage + acts + last <= lds
    assert read == set(range(live))   # and every live tile is read
