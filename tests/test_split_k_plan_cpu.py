"""CPU checks of the split-K plan (``split_plan`` in csrc/split_k.h, through
the probe library; no GPU call): over row counts, widths and depths of any
alignment, a plan that splits gives every K range work, starts no more
workgroups than the CUs, and wants a workspace of exactly its fp32 sums,
bounded by one largest tile per CU; decode rows and wide outputs never split;
sizes beyond any launch are answered, not divided by."""
import ctypes
import subprocess
import sys
from pathlib import Path

import pytest

PROBE = Path(__file__).resolve().parents[1] / "llm-inference-optimizer_amd" / "libmi355_probe.so"
ROWS = (1, 16, 17, 24, 32, 33, 48, 64, 65, 100, 128, 129, 333, 512, 1000, 1537, 4096, 100000)
KS = (8, 64, 200, 896, 1536, 3584, 4096, 4864, 8960, 18944, 18952, 65536)
NS = (1, 3, 37, 896, 1536, 3584, 5120, 13824, 18944, 151936)


@pytest.fixture(scope="module")
def plan():
    if not PROBE.exists():
        pytest.skip("probe library not built")
    f = ctypes.CDLL(str(PROBE)).mi355_probe_split_plan
    f.argtypes, f.restype = [ctypes.c_longlong] * 3 + [ctypes.c_int] * 2 + [ctypes.POINTER(ctypes.c_int)], ctypes.c_longlong

    def call(rows, k, n, wb, cus):
        out = (ctypes.c_int * 4)()
        return f(rows, k, n, wb, cus, out), *out
    return call


@pytest.mark.parametrize("wb", [1, 2])
@pytest.mark.parametrize("cus", [64, 256, 304])
def test_split_plan_is_launchable(plan, wb, cus):
    tiles_seen = set()
    for rows in ROWS:
        for k in KS:
            for n in NS:
                nbytes, tile, splits, bm, bn = plan(rows, k, n, wb, cus)
                if tile < 0:
                    assert nbytes == 0
                    continue
                tiles_seen.add(tile)
                assert rows > 16
                steps, tiles = -(-k // 64), -(-rows // bm) * -(-n // bn)
                per = -(-steps // splits)
                assert 2 <= splits <= 32 and tiles * splits <= cus
                assert per >= 4 and (splits - 1) * per < steps, "every range has work"
                assert nbytes == 4 * splits * rows * n <= 4 * cus * 256 * 256
    if cus == 256:
        assert tiles_seen == set(range(5)), tiles_seen


@pytest.mark.parametrize("wb", [1, 2])
def test_sizes_beyond_a_launch_want_no_workspace(wb):
    # Tile counts that are multiples of 2^32, or wrap to a few: the size query
    # takes any rows, k, n below 2^31.  In a child process, which a division
    # by zero would end.
    if not PROBE.exists():
        pytest.skip("probe library not built")
    code = f"""
import ctypes
f = ctypes.CDLL({str(PROBE)!r}).mi355_probe_split_plan
f.argtypes, f.restype = [ctypes.c_longlong] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p], ctypes.c_longlong
out = (ctypes.c_int * 4)()
near = [v for e in range(8, 32) for v in (2 ** e - 1, 2 ** e, 2 ** e + 1) if v < 2 ** 31]
for rows in near:
    for n in near:
        if rows * n > 2 ** 34:
            for k in (64, 4096, 2 ** 31 - 1):
                assert f(rows, k, n, {wb}, 256, out) == 0 and out[0] < 0, (rows, k, n)
"""
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert res.returncode == 0, (res.returncode, res.stderr)
