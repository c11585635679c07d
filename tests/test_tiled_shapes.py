"""The tiled kernels over the plans of csrc/tiled_plan.h: the 16-bit and int8
gate/up + SiLU-and-mul and the two single-matrix linears against fp64 GEMMs on
the GPU, within one output ulp plus the worst-case fp32 summation error; the
16-bit output is the fp32 output rounded once.

Shapes are picked by size alone.  A grid runs over the row counts and widths
at which the plans change over, with K of a few steps and a partial last one
(fewer steps than LDS stages included).  Beside it SHAPE_CASES holds sizes for
each tile of each table and for the gate/up's two-launch column splits, on
ragged rows and columns, with K of 3 steps and a part (fewer than the ring's
unrolled steps) where the plan takes the tile there and of 29 and a part or
56 and a part (its main loop, and a remainder);
test_tile_plan_cpu.py checks that each of them takes the tile it names and
that no tile is left out."""
import importlib

import pytest
import torch

from parity_utils import act_error_bound, gen, ulp16

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
ROWS = (33, 65, 96, 129, 191, 257, 385, 520)
KS = (16, 80, 208, 336, 1104)
NS = (66, 1030, 5000, 19000)

LINEAR16, W8, GATE_UP16, GATE_UP8 = range(4)
# (table, its tile, rows, k, n); in SPLIT_CASES (tile of the leading columns,
# tile of the rest, rows, k, n) of the 16-bit gate/up in two launches
SHAPE_CASES = [
    (LINEAR16, 0, 67, 208, 330), (LINEAR16, 0, 3353, 1872, 35),
    (LINEAR16, 1, 3465, 208, 4622), (LINEAR16, 1, 67, 1872, 12099), (LINEAR16, 1, 129, 3600, 7499),
    (LINEAR16, 2, 133, 400, 5537), (LINEAR16, 2, 66, 1872, 8237),
    (LINEAR16, 3, 193, 208, 12622), (LINEAR16, 3, 67, 1872, 16450),
    (LINEAR16, 4, 195, 208, 16534), (LINEAR16, 4, 259, 1872, 13189),
    (LINEAR16, 5, 130, 1872, 16429), (LINEAR16, 5, 131, 3600, 16763),
    (LINEAR16, 6, 388, 1872, 16429), (LINEAR16, 6, 391, 3600, 16652),
    (W8, 0, 3495, 208, 385), (W8, 0, 4209, 1872, 65),
    (W8, 1, 98, 208, 12415), (W8, 1, 67, 1872, 11003),
    (W8, 2, 321, 208, 19113), (W8, 2, 69, 1872, 16447),
    (W8, 3, 520, 208, 20027), (W8, 3, 259, 1872, 13071),
    (W8, 4, 259, 208, 1030), (W8, 4, 69, 1872, 2185),
    (GATE_UP16, 0, 34, 208, 77), (GATE_UP16, 0, 67, 1872, 70),
    (GATE_UP16, 1, 35, 1872, 12475), (GATE_UP16, 1, 67, 3600, 7133),
    (GATE_UP16, 2, 35, 1872, 16977), (GATE_UP16, 2, 34, 3600, 16425),
    (GATE_UP16, 3, 132, 1872, 16491), (GATE_UP16, 3, 131, 3600, 16045),
    (GATE_UP16, 4, 203, 1872, 16465), (GATE_UP16, 4, 198, 3600, 16631),
    (GATE_UP16, 5, 129, 1872, 11029), (GATE_UP16, 5, 130, 3600, 10917),
    (GATE_UP8, 0, 262, 208, 9818), (GATE_UP8, 0, 67, 1872, 16451),
    (GATE_UP8, 1, 131, 208, 8276), (GATE_UP8, 1, 260, 1872, 67),
    (GATE_UP8, 2, 69, 208, 16695), (GATE_UP8, 2, 4116, 1872, 195),
    (GATE_UP8, 3, 326, 1872, 16683), (GATE_UP8, 3, 67, 3600, 8199),
    (GATE_UP8, 4, 261, 208, 19657), (GATE_UP8, 4, 132, 1872, 16497),
    (GATE_UP8, 5, 396, 208, 12469), (GATE_UP8, 5, 387, 1872, 12437),
    (GATE_UP8, 6, 261, 208, 75), (GATE_UP8, 6, 67, 1872, 8309),
]
SPLIT_CASES = [(2, 5, 2838, 1872, 2702), (3, 0, 262, 1872, 16435), (3, 1, 257, 1872, 19677), (3, 2, 580, 1872, 14309),
               (3, 5, 792, 1872, 9431), (4, 0, 386, 1872, 16527), (4, 1, 391, 1872, 19069), (4, 2, 590, 1872, 16465),
               (4, 3, 772, 1872, 14147), (4, 5, 972, 1872, 10257), (5, 1, 3457, 1872, 1679)]


def _inputs(rows, k, n, dt, int8, mats, cuda):
    x = torch.randn(rows, k, generator=gen(rows + k)).to(dt).to(cuda)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    ws = []
    for _ in range(mats):
        if int8:
            w = torch.randint(-127, 128, (n, k), generator=g, device=cuda, dtype=torch.int8)
            s = (torch.rand(n, generator=g, device=cuda) + 0.5) / (74 * k ** 0.5)
            ws.append((w, s, w.double() * s.double()[:, None]))
        else:
            w = (torch.randn(n, k, generator=g, device=cuda) * k ** -0.5).to(dt)
            ws.append((w, None, w.double()))
    return x, ws


def _gamma(k):
    return k * 2.0 ** -24 / (1 - k * 2.0 ** -24)


def _check_single(pkg, cuda, rows, k, n, dt, int8, bias=False):
    x, [(w, s, w64)] = _inputs(rows, k, n, dt, int8, 1, cuda)
    b = torch.randn(n, generator=gen(n)).to(cuda) if bias else None
    call = (lambda **kw: pkg.w8a16_linear(x, w, s, b, **kw)) if int8 else (lambda **kw: pkg.linear16(x, w, b, **kw))
    got16, got32 = call(), call(out_dtype=F32).double()
    exact, mag = x.double() @ w64.T, x.double().abs() @ w64.abs().T
    if bias:
        exact, mag = exact + b.double(), mag + b.double().abs()
    bound = _gamma(k) * mag + 2.0 ** -22 * exact.abs() + 1e-30
    ulp = torch.from_numpy(ulp16(exact.cpu().numpy(), dt)).to(cuda)
    assert float(((got32 - exact).abs() - bound).max()) <= 0, (k, n)
    assert float(((got16.double() - exact).abs() - (ulp + bound)).max()) <= 0, (k, n)
    assert torch.equal(got16, got32.to(dt)), (k, n)


def _check_gate_up(pkg, cuda, rows, k, n, dt, int8):
    x, [(wg, sg, g64), (wu, su, u64)] = _inputs(rows, k, n, dt, int8, 2, cuda)
    if int8:
        def call(**kw):
            return pkg.fused_gate_up_silu_w8a16(x, wg, sg, wu, su, **kw)
    else:
        def call(**kw):
            return pkg.fused_gate_up_silu(x, wg, wu, **kw)
    got16, got32 = call(), call(out_dtype=F32).double()
    x64 = x.double()
    g, u = x64 @ g64.T, x64 @ u64.T
    exact = torch.nn.functional.silu(g) * u
    bound = torch.from_numpy(act_error_bound(*(t.cpu().numpy() for t in (g, u, x64.abs() @ g64.abs().T,
                                                                          x64.abs() @ u64.abs().T)), k)).to(cuda)
    bound = bound + 2.0 ** -21 * exact.abs() + 1e-30
    ulp = torch.from_numpy(ulp16(exact.cpu().numpy(), dt)).to(cuda)
    assert float(((got32 - exact).abs() - bound).max()) <= 0, (k, n)
    assert float(((got16.double() - exact).abs() - (ulp + bound)).max()) <= 0, (k, n)
    assert torch.equal(got16, got32.to(dt)), (k, n)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("rows", ROWS)
def test_single(pkg, cuda, rows, dt, int8):
    for i, k in enumerate(KS):
        _check_single(pkg, cuda, rows, k, NS[(i + rows) % len(NS)], dt, int8)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("rows", ROWS)
def test_gate_up(pkg, cuda, rows, dt, int8):
    for i, k in enumerate(KS):
        _check_gate_up(pkg, cuda, rows, k, NS[(i + rows // 2) % len(NS)], dt, int8)


@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("table,tile,rows,k,n", SHAPE_CASES)
def test_each_tile(pkg, cuda, table, tile, rows, k, n, dt):
    if table in (LINEAR16, W8):
        _check_single(pkg, cuda, rows, k, n, dt, table == W8, bias=True)
    else:
        _check_gate_up(pkg, cuda, rows, k, n, dt, table == GATE_UP8)


@pytest.mark.parametrize("lead,tail,rows,k,n", SPLIT_CASES)
def test_column_splits(pkg, cuda, lead, tail, rows, k, n):
    """Two launches on column ranges, ragged in rows and columns; the same
    values in a row-strided output whose gap stays untouched."""
    dt = BF16 if (lead + tail) % 2 else F16
    _check_gate_up(pkg, cuda, rows, k, n, dt, False)
    x, [(wg, _, _), (wu, _, _)] = _inputs(rows, k, n, dt, False, 2, cuda)
    L = importlib.import_module("llm-inference-optimizer_amd._lib")
    for gap in (7, 16 - n % 8):  # rows of any alignment, and of whole 16-byte packets
        out = torch.full((rows, n + gap), 7.0, dtype=dt, device=cuda)
        code = L.DTYPE_CODE[dt]
        L.gate_up_silu_fwd(x.data_ptr(), wg.data_ptr(), wu.data_ptr(), out.data_ptr(), rows, k, n, k, k, n + gap,
                           code, code, L.stream_handle(cuda))
        assert torch.equal(out[:, :n], pkg.fused_gate_up_silu(x, wg, wu))
        assert bool((out[:, n:] == 7.0).all())
