"""CPU checks of the quantiser's launch rule (``quant_plan`` in
csrc/quantize_plan.h, through the probe library; no GPU call): every row and
every packet of a row has a lane, and a launch stays below 2^32 threads (the
runtime's limit) for every row count that a wave per row would still hold."""
import ctypes
from pathlib import Path

import pytest

PROBE = Path(__file__).resolve().parents[1] / "llm-inference-optimizer_amd" / "libmi355_probe.so"
MOST_ROWS = 4 * ((2 ** 32 - 1) // 256)  # 4 rows per workgroup of 256 threads


@pytest.fixture(scope="module")
def plan():
    if not PROBE.exists():
        pytest.skip("probe library not built")
    f = ctypes.CDLL(str(PROBE)).mi355_probe_quant_plan
    f.argtypes, f.restype = [ctypes.c_longlong] * 2 + [ctypes.POINTER(ctypes.c_int)], ctypes.c_longlong

    def call(n, packets):
        out = (ctypes.c_int * 4)()
        return f(n, packets, out), *out[:3]
    return call


@pytest.mark.parametrize("n", [1, 3, 4, 5, 18944, 2 ** 22, 4194303, 4194304, 22369621, 22369622, MOST_ROWS])
def test_launches_hold_their_rows(plan, n):
    for packets in (0, 1, 64, 65, 448, 512, 513, 514, 768, 769, 2048, 4096, 4097, 8191, 8192, 8193, 2 ** 28):
        grid, vpl, block, threads = plan(n, packets)
        assert grid * threads < 2 ** 32, packets
        assert threads % 64 == 0 and 64 <= threads <= 1024
        assert grid * (1 if block else 4) >= n and (block or threads == 256)
        if vpl:
            assert 1 <= vpl <= 8 and vpl * (threads if block else 64) >= packets >= 1
        if packets in range(1, 513) or (packets in range(513, 8193) and n <= 4194303):
            assert vpl, "rows in registers wherever a launch holds them"
