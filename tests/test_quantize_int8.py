"""The int8 quantiser (csrc/quantize_int8.hip) against the reference's torch
expression in fp32, bit for bit, at the edges of its row shapes (packets per
lane, waves per row, the scalar kernel beyond) and on rows whose quotients lie
at and next to half-integers, where its reciprocal arithmetic must fall back
to the division; rows with NaN and infinities keep the plain formula."""
import pytest
import torch

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def _reference(w):
    w = w.float().cpu()  # on the CPU torch divides by 127; on a GPU it multiplies by 1 / 127
    amax = torch.where(w.isnan(), torch.zeros_like(w), w.abs()).amax(1)  # fmaxf skips NaN
    scale = torch.clamp(amax / 127.0, min=1e-8)
    v = torch.round(w / scale[:, None])
    v = torch.where(v.isnan(), torch.full_like(v, -127.0), v)  # fmaxf(NaN, -127)
    return torch.clamp(v, -127, 127).to(torch.int8), scale


def _check(pkg, w):
    q, s = pkg.quantize_int8_weight(w)
    rq, rs = _reference(w)
    assert torch.equal(s.cpu(), rs)
    assert torch.equal(q.cpu(), rq), f"{int((q.cpu() != rq).sum())} codes differ"


@pytest.mark.parametrize("dt", [F16, BF16, F32])
@pytest.mark.parametrize("n,k", [(1, 8), (5, 504), (7, 512), (9, 520), (130, 3584), (3, 4096), (6, 4104), (4, 18944),
                                 (2, 32768), (3, 32776), (2, 65536), (2, 65544), (11, 1001), (8, 4)])
def test_matches_torch(pkg, cuda, dt, n, k):
    g = torch.Generator(device="cuda").manual_seed(n * k)
    _check(pkg, (torch.randn(n, k, generator=g, device=cuda) * 0.02).to(dt))


@pytest.mark.parametrize("k", [2048, 8192])
def test_half_integers(pkg, cuda, k):
    """Every representable w next to (i + 1/2) * scale, for random scales."""
    g = torch.Generator(device="cuda").manual_seed(k)
    amax = (torch.rand(256, 1, generator=g, device=cuda) + 0.5) * 2.0 ** torch.randint(-20, 20, (256, 1), generator=g,
                                                                                       device=cuda)
    half = torch.randint(-127, 127, (256, k), generator=g, device=cuda) + 0.5
    w = half * (amax / 127.0)
    step = torch.randint(-3, 4, w.shape, generator=g, device=cuda, dtype=torch.int32)
    w = (w.view(torch.int32) + step).view(F32)
    w[:, :1] = amax
    _check(pkg, w)
    exact = torch.cat([(torch.arange(-127, 127, device=cuda) + 0.5).repeat(4) * 2.0 ** -7,
                       torch.full((8,), 127.0 * 2.0 ** -7, device=cuda)])
    for dt in (F16, BF16, F32):
        _check(pkg, exact.to(dt).repeat(3, 1))


@pytest.mark.parametrize("dt", [F16, BF16, F32])
@pytest.mark.parametrize("k", [64, 3584, 18944])
def test_special_rows(pkg, cuda, dt, k):
    g = torch.Generator(device="cuda").manual_seed(k)
    w = torch.randn(8, k, generator=g, device=cuda).to(dt)
    w[0] = 0
    w[1, k // 2] = float("nan")
    w[2, 3] = float("inf")
    w[3, 5], w[3, 6] = float("-inf"), float("nan")
    w[4] = float("nan")
    w[5] *= 1e-6 if dt == F16 else 1e-30
    w[6, :] = torch.finfo(dt).max
    _check(pkg, w)
    strided = torch.zeros(8, k + 8, dtype=dt, device=cuda)[:, :k].copy_(w)
    _check(pkg, strided)
