"""Every tile shape the unsplit plans choose from (csrc/tiled_plan.h), at row
counts one short of, on and past its tile, K of a few steps with a partial
last one (fewer steps than LDS stages included) and ragged columns: the 16-bit
and int8 gate/up + SiLU-and-mul and the two single-matrix linears against fp64
GEMMs on the GPU, within one output ulp plus the worst-case fp32 summation
error; the 16-bit output is the fp32 output rounded once.  The shapes are
picked by size alone, so the grid runs over the row counts and widths at which
the plans change over."""
import pytest
import torch

from parity_utils import act_error_bound, gen, ulp16

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
ROWS = (33, 65, 96, 129, 191, 257, 385, 520)
KS = (16, 80, 208, 336, 1104)
NS = (66, 1030, 5000, 19000)


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


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("rows", ROWS)
def test_single(pkg, cuda, rows, dt, int8):
    for i, k in enumerate(KS):
        n = NS[(i + rows) % len(NS)]
        x, [(w, s, w64)] = _inputs(rows, k, n, dt, int8, 1, cuda)
        call = (lambda **kw: pkg.w8a16_linear(x, w, s, **kw)) if int8 else (lambda **kw: pkg.linear16(x, w, **kw))
        got16, got32 = call(), call(out_dtype=F32).double()
        exact = x.double() @ w64.T
        bound = _gamma(k) * (x.double().abs() @ w64.abs().T) + 2.0 ** -22 * exact.abs() + 1e-30
        ulp = torch.from_numpy(ulp16(exact.cpu().numpy(), dt)).to(cuda)
        assert float(((got32 - exact).abs() - bound).max()) <= 0, (k, n)
        assert float(((got16.double() - exact).abs() - (ulp + bound)).max()) <= 0, (k, n)
        assert torch.equal(got16, got32.to(dt)), (k, n)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("rows", ROWS)
def test_gate_up(pkg, cuda, rows, dt, int8):
    for i, k in enumerate(KS):
        n = NS[(i + rows // 2) % len(NS)]
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
