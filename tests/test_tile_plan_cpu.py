"""CPU checks of the unsplit tile plans (``plan_tiles`` in csrc/tiled_plan.h,
through the probe library; no GPU call): a plan's launches stay below the
runtime's 2^32 threads wherever one of the table's tiles does."""
import ctypes
from pathlib import Path

import pytest

PROBE = Path(__file__).resolve().parents[1] / "llm-inference-optimizer_amd" / "libmi355_probe.so"
LINEAR16, W8, GATE_UP16, GATE_UP8 = range(4)


def tile_plan(table, rows, k, n, cus=256):
    """(predicted us, shape, lead, tail, (bm, bn, threads) of the first and of the second launch)"""
    f = ctypes.CDLL(str(PROBE)).mi355_probe_tile_plan
    f.argtypes = [ctypes.c_int] + [ctypes.c_longlong] * 3 + [ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    f.restype = ctypes.c_double
    out = (ctypes.c_int * 9)()
    us = f(table, rows, k, n, cus, out)
    return us, out[0], out[1], out[2], tuple(out[3:6]), tuple(out[6:9])


def split_plan(rows, k, n, wb, cus=256):
    """(tile (< 0: not split), K ranges, the tile's rows, its columns)"""
    f = ctypes.CDLL(str(PROBE)).mi355_probe_split_plan
    f.argtypes = [ctypes.c_longlong] * 3 + [ctypes.c_int] * 2 + [ctypes.POINTER(ctypes.c_int)]
    f.restype = ctypes.c_longlong
    out = (ctypes.c_int * 4)()
    f(rows, k, n, wb, cus, out)
    return tuple(out)


def _threads(rows, cols, shape):
    bm, bn, threads = shape
    return -(-rows // bm) * -(-cols // bn) * threads


@pytest.mark.parametrize("rows", [33, 64, 65, 128, 129, 256, 512])
def test_gate_up_launches_hold_their_threads(rows):
    """The 16-bit gate/up takes any n below 2^31: 256 x 128 tiles of 512
    threads hold 256 rows of 2^30 columns (128 x 128 ones 128 rows)."""
    if not PROBE.exists():
        pytest.skip("probe library not built")
    for k in (8, 64, 208, 1536):
        for n in (2 ** 26 + 1, 2 ** 27, 2 ** 28 - 64, 2 ** 28, 2 ** 28 + 200, 2 ** 29, 2 ** 30 - 128):
            _, _, lead, _, first, second = tile_plan(GATE_UP16, rows, k, n)
            if _threads(rows, n, (256, 128, 512)) >= 2 ** 32:
                continue
            assert _threads(rows, lead or n, first) < 2 ** 32, (k, n, first)
            if lead:
                assert 0 < lead < n and lead % first[1] == 0
                assert _threads(rows, n - lead, second) < 2 ** 32, (k, n, second)
