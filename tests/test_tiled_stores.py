"""The tiled kernels' output stores (csrc/tiled_gemm.h): 64-byte row segments
through LDS where the output's row stride and address allow 16-byte stores,
8-byte stores or single elements otherwise, ragged last segments and rows in
each.  The same call into outputs of those four kinds through the C ABI gives
the same values (equal bits: one kernel, one summation order), and nothing
outside the output's columns is written.  The small sizes run 64 x 64 tiles
(int8 also 32 x 64); TILE_CASES names a size for every other tile of the two
linears (test_tile_plan_cpu.py checks that it takes it)."""
import importlib

import pytest
import torch

from parity_utils import gen

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
CODE = {F32: 0, F16: 1, BF16: 2}


def _call(lib, int8, x, w, scale, bias, out, os, n):
    rows, k = x.shape
    p = lambda t: 0 if t is None else t.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    if int8:
        return lib.mi355_w8a16_linear_fwd(p(x), p(w), p(scale), p(bias), p(out), rows, k, n, k, k, os, CODE[x.dtype],
                                          CODE[scale.dtype], 0 if bias is None else CODE[bias.dtype], CODE[out.dtype],
                                          stream)
    return lib.mi355_linear16_fwd(p(x), p(w), p(bias), p(out), rows, k, n, k, k, os, CODE[x.dtype],
                                  0 if bias is None else CODE[bias.dtype], CODE[out.dtype], stream)


# (int8 weights, tile, rows, n, k)
TILE_CASES = [(False, (128, 64), 67, 12099, 1872), (False, (64, 128), 66, 8237, 1872),
              (False, (128, 128), 67, 16450, 1872), (False, (256, 128), 130, 16429, 1872),
              (False, (256, 256), 388, 16429, 1872), (True, (32, 64), 259, 1030, 208), (True, (64, 128), 98, 12415, 208),
              (True, (128, 128), 69, 16447, 1872), (True, (192, 128), 259, 13071, 1872)]


@pytest.mark.parametrize("out_dt", ["half", "fp32"])
@pytest.mark.parametrize("int8,tile,rows,n,k", TILE_CASES)
def test_output_layouts_of_each_tile(pkg, cuda, int8, tile, rows, n, k, out_dt):
    _check_layouts(cuda, rows, n, k, out_dt, int8)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("out_dt", ["half", "fp32"])
@pytest.mark.parametrize("rows,n", [(130, 1032), (259, 1026), (300, 1029), (700, 3001), (1100, 9004)])
def test_output_layouts(pkg, cuda, rows, n, out_dt, int8):
    _check_layouts(cuda, rows, n, 208, out_dt, int8)


def _check_layouts(cuda, rows, n, k, out_dt, int8):
    lib = importlib.import_module("llm-inference-optimizer_amd._lib").load()
    dt = F16 if n % 2 else BF16
    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x = torch.randn(rows, k, generator=gen(n)).to(dt).to(cuda)
    if int8:
        w = torch.randint(-127, 128, (n, k), generator=g, device=cuda, dtype=torch.int8)
        scale = (torch.rand(n, generator=g, device=cuda) + 0.5).to(dt if n % 4 else F32) / 64
    else:
        w, scale = torch.randn(n, k, generator=g, device=cuda).to(dt), None
    bias = torch.randn(n, generator=g, device=cuda).to(F32 if n % 2 else dt)
    odt = dt if out_dt == "half" else F32
    wide = (n + 23) // 8 * 8  # a row stride of whole 16-byte packets, at least 16 columns of guard
    got = []
    for os, off in ((wide, 0), (wide, 1), (n + 17, 0), (wide + 4, 0)):
        buf = torch.full((rows * os + 64,), 77.0, device=cuda, dtype=odt)
        view = buf[off:off + rows * os].view(rows, os)
        assert _call(lib, int8, x, w, scale, bias, view, os, n) == 0
        assert bool((view[:, n:] == 77.0).all()) and bool((buf[off + rows * os:] == 77.0).all())
        assert bool((buf[:off] == 77.0).all())
        got.append(view[:, :n].clone())
    w64 = w.double() * scale.double()[:, None] if int8 else w.double()
    exact = x.double() @ w64.T + bias.double()
    mag = x.double().abs() @ w64.abs().T + bias.double().abs()
    # fp32 sums of k terms and two more roundings, then one rounding to 16 bits
    eps = 2.0 ** -24 * (k + 4) + (0 if odt == F32 else 2.0 ** (-11 if dt == F16 else -8))
    assert float(((got[0].double() - exact).abs() - eps * mag).max()) <= 0
    assert all(torch.equal(got[0], other) for other in got[1:])
