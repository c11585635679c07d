"""CPU checks of the unsplit tile plans (``plan_tiles`` in csrc/tiled_plan.h,
through the probe library; no GPU call): a plan's launches stay below the
runtime's 2^32 threads wherever one of the table's tiles does, and the GPU
tests' sizes take the tiles they name, every tile of every table among them
(256 CUs)."""
import ctypes
from pathlib import Path

import pytest

import test_tiled_shapes as shapes
import test_tiled_stores as stores

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


def _w8_skinny(rows, n):
    """65 - 256 rows that leave the int8 linear 32-row tiles of its own."""
    return rows <= 256 and (-(-n // 64) * -(-rows // 64) < 32 or (rows <= 128 and n < 2048))


def _unsplit_tile(table, rows, k, n):
    """The tile an eager call takes, by the launchers' rules beyond 64 rows."""
    assert rows > (32 if table == GATE_UP16 else 64)
    if table in (LINEAR16, W8):
        assert split_plan(rows, k, n, 2 if table == LINEAR16 else 1)[0] < 0, "must not split K"
    if table in (W8, GATE_UP8):
        assert k % 16 == 0 and not _w8_skinny(rows, n)
    _, shape, lead, tail, _, _ = tile_plan(table, rows, k, n)
    return shape, lead, tail


def test_every_tile_has_its_gpu_cases():
    if not PROBE.exists():
        pytest.skip("probe library not built")
    seen = {}
    for table, tile, rows, k, n in shapes.SHAPE_CASES:
        assert _unsplit_tile(table, rows, k, n)[:2] == (tile, 0), (table, tile, rows, k, n)
        bm, bn, _ = tile_plan(table, rows, k, n)[4]
        assert rows % bm and n % bn and k % 64, "ragged in every direction"
        seen.setdefault((table, tile), []).append(k)
    assert set(seen) == {(table, i) for table, count in enumerate((7, 5, 6, 7)) for i in range(count)}
    assert all(max(ks) >= 64 * 29 for ks in seen.values()), "the main loop of every tile"
    for first, second, rows, k, n in shapes.SPLIT_CASES:
        shape, lead, tail = _unsplit_tile(GATE_UP16, rows, k, n)
        assert lead > 0 and (shape, tail) == (first, second), (rows, k, n)
        assert n % 64


def test_store_cases_take_the_tiles_they_name():
    """Several 32 x 32 blocks per wave and waves in the second LDS stage among them."""
    if not PROBE.exists():
        pytest.skip("probe library not built")
    for int8, tile, rows, n, k in stores.TILE_CASES:
        table = W8 if int8 else LINEAR16
        assert _unsplit_tile(table, rows, k, n)[1] == 0
        assert tile_plan(table, rows, k, n)[4][:2] == tile, (rows, k, n)
    assert {t for int8, t, *_ in stores.TILE_CASES if int8} == {(32, 64), (64, 128), (128, 128), (192, 128)}
    assert {t for int8, t, *_ in stores.TILE_CASES if not int8} == {(128, 64), (64, 128), (128, 128), (256, 128), (256, 256)}


@pytest.mark.parametrize("rows,k,n", [(3500, 13824, 5120), (3400, 13824, 5120), (4352, 18944, 4096)])
def test_linear16_takes_no_thin_round_of_its_largest_tile(rows, k, n):
    """256 x 256 tiles that leave a last round of a few (280, 280 and 272 on 256
    CUs) cost a whole tile's chain: smaller ones measured faster."""
    if not PROBE.exists():
        pytest.skip("probe library not built")
    assert 256 < -(-rows // 256) * -(-n // 256) < 300
    assert tile_plan(LINEAR16, rows, k, n)[4][:2] != (256, 256)
