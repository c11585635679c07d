"""The split-K kernels (csrc/split_k.h) behind ``linear16`` and
``w8a16_linear``: every tile of the plan at ragged rows, K tails and columns
(n not a multiple of 4 takes the scalar second pass), against fp64 GEMMs on
the GPU -- within one output ulp plus the worst-case fp32 summation error,
the fp32 output within that bound, the 16-bit output equal to the fp32 output
rounded once -- and against the unsplit kernels the C ABI runs without a
workspace.  Also under graph replay and with row-strided inputs."""
import gc
import importlib

import pytest
import torch

from parity_utils import gen, ulp16

pytestmark = pytest.mark.gpu

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
# rows, k, n: the 32 x 128, 64 x 64, 64 x 128, 128 x 128 and 256 x 256 tiles at
# the edges of their rows, k with a partial last step, n odd or not of 4
SHAPES16 = [(31, 12008, 2050), (65, 2008, 130), (129, 4000, 131), (17, 9016, 5121), (65, 12008, 1536), (128, 6000, 3582),
            (400, 9008, 5122), (1001, 12008, 2049)]
SHAPES8 = [(200, 2032, 500), (32, 18960, 3584), (65, 4016, 130), (64, 9008, 1537), (33, 6000, 3584), (129, 6000, 5122),
           (65, 18960, 1538), (1001, 9008, 5122)]


@pytest.fixture(scope="module")
def lib():
    return importlib.import_module("llm-inference-optimizer_amd._lib")


def _check(got16, got32, exact, absum, k, dt):
    gam = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    bound = gam * absum + 2.0 ** -22 * exact.abs() + 1e-30
    ulp = torch.from_numpy(ulp16(exact.cpu().numpy(), dt)).to(exact.device)
    assert float(((got32.double() - exact).abs() - bound).max()) <= 0
    assert float(((got16.double() - exact).abs() - (ulp + bound)).max()) <= 0
    assert torch.equal(got16, got32.to(dt)), "the 16-bit output must be the fp32 output rounded once"


def _case(shape, dt, cuda, int8, bias):
    rows, k, n = shape
    x = torch.randn(rows, k, generator=gen(rows)).to(dt).to(cuda)
    b = torch.randn(n, generator=gen(n)).to(cuda) if bias else None
    if int8:
        g = torch.Generator(device="cuda").manual_seed(k)
        w = torch.randint(-127, 128, (n, k), generator=g, device=cuda, dtype=torch.int8)
        s = (torch.rand(n, generator=gen(3)) + 0.5).to(cuda) / 74 / k ** 0.5
        w64 = w.double() * s.double()[:, None]
    else:
        w, s = (torch.randn(n, k, generator=gen(k)) * k ** -0.5).to(dt).to(cuda), None
        w64 = w.double()
    x64 = x.double()
    exact, absum = x64 @ w64.T, x64.abs() @ w64.abs().T
    if bias:
        exact, absum = exact + b.double(), absum + b.double().abs()
    return x, w, s, b, exact, absum


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("shape", SHAPES16)
def test_linear16_split(pkg, cuda, lib, shape, dt, bias):
    assert lib.load().mi355_linear16_workspace(*shape) > 0, "the shape must take the split path"
    x, w, _, b, exact, absum = _case(shape, dt, cuda, False, bias)
    _check(pkg.linear16(x, w, b), pkg.linear16(x, w, b, out_dtype=F32), exact, absum, shape[1], dt)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dt", [F16, BF16])
@pytest.mark.parametrize("shape", SHAPES8)
def test_w8a16_split(pkg, cuda, lib, shape, dt, bias):
    assert lib.load().mi355_w8a16_linear_workspace(*shape) > 0, "the shape must take the split path"
    x, q, s, b, exact, absum = _case(shape, dt, cuda, True, bias)
    _check(pkg.w8a16_linear(x, q, s, b), pkg.w8a16_linear(x, q, s, b, out_dtype=F32), exact, absum, shape[1], dt)


@pytest.mark.parametrize("int8", [False, True])
def test_split_against_unsplit_and_strided_and_graph(pkg, cuda, lib, int8):
    """Row-strided x and weights, the ABI without a workspace (the unsplit
    kernels), and graph replays between eager calls."""
    rows, k, n = 77, 6000, 1540
    x, w, s, _, exact, absum = _case((rows, k, n), F16, cuda, int8, False)
    xs = torch.zeros(rows, k + 16, dtype=F16, device=cuda)[:, :k].copy_(x)
    ws = torch.zeros(n, k + 32, dtype=w.dtype, device=cuda)[:, :k].copy_(w)
    call = (lambda a, b: pkg.w8a16_linear(a, b, s)) if int8 else pkg.linear16
    want = call(x, w)
    assert torch.equal(call(xs, ws), want), "strides do not change the sums"
    _check(want, pkg.w8a16_linear(x, w, s, out_dtype=F32) if int8 else pkg.linear16(x, w, out_dtype=F32), exact, absum,
           k, F16)
    unsplit = torch.empty_like(want)
    stream = torch.cuda.current_stream().cuda_stream
    if int8:
        lib.w8a16_linear_fwd(x.data_ptr(), w.data_ptr(), s.data_ptr(), None, unsplit.data_ptr(), rows, k, n, k, k, n,
                             lib.F16, lib.F32, 0, lib.F16, stream)
    else:
        lib.linear16_fwd(x.data_ptr(), w.data_ptr(), None, unsplit.data_ptr(), rows, k, n, k, k, n, lib.F16, 0, lib.F16,
                         stream)
    ulp = torch.from_numpy(ulp16(exact.cpu().numpy(), F16)).to(cuda)
    gam = k * 2.0 ** -24
    assert float(((unsplit.double() - want.double()).abs() - (ulp + 2 * gam * absum)).max()) <= 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want)
        assert torch.equal(call(x, w), want)


def _linear(pkg, cuda, int8, rows, k, n):
    x, w, s, _, _, _ = _case((rows, k, n), F16, cuda, int8, False)
    return x, w, s, (lambda: pkg.w8a16_linear(x, w, s)) if int8 else (lambda: pkg.linear16(x, w))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("rows,k,n,offset", [(200, 4001, 500, 0), (200, 4008, 500, 1)])
def test_no_workspace_where_split_k_cannot_run(pkg, cuda, int8, rows, k, n, offset):
    """Rows that are no whole 16-byte packets run the generic kernel: such a
    call allocates its output and nothing else."""
    x = torch.randn(rows * k + offset, generator=gen(3)).to(F16).to(cuda)[offset:].view(rows, k)
    if int8:
        w, s = torch.randint(-127, 128, (n, k), device=cuda, dtype=torch.int8), torch.rand(n, device=cuda)
        call = lambda: pkg.w8a16_linear(x, w, s)
    else:
        w = torch.randn(n, k, generator=gen(4)).to(F16).to(cuda)
        call = lambda: pkg.linear16(x, w)
    call()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = call()
    assert torch.cuda.max_memory_allocated() - before <= out.numel() * 2 + 512


@pytest.mark.parametrize("int8", [False, True])
def test_without_memory_for_the_workspace(pkg, cuda, lib, int8):
    """A call whose output fits but whose workspace does not runs the unsplit
    kernels, as one through the C ABI without a workspace does."""
    rows, k, n = 700, 18944, 3584
    x, w, s, call = _linear(pkg, cuda, int8, rows, k, n)
    want = torch.empty(rows, n, dtype=F16, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    if int8:
        nbytes = lib.load().mi355_w8a16_linear_workspace(rows, k, n)
        lib.w8a16_linear_fwd(x.data_ptr(), w.data_ptr(), s.data_ptr(), None, want.data_ptr(), rows, k, n, k, k, n,
                             lib.F16, lib.F32, 0, lib.F16, stream)
    else:
        nbytes = lib.load().mi355_linear16_workspace(rows, k, n)
        lib.linear16_fwd(x.data_ptr(), w.data_ptr(), None, want.data_ptr(), rows, k, n, k, k, n, lib.F16, 0, lib.F16,
                         stream)
    assert nbytes > 20 << 20, "more than a segment that the allocator makes for the output"
    torch.cuda.synchronize()
    room, fill = torch.empty_like(want), []
    gc.collect()
    try:
        torch.cuda.set_per_process_memory_fraction(
            torch.cuda.memory_reserved() / torch.cuda.get_device_properties(cuda).total_memory)
        # what other tests left free, down to gaps and a remainder that hold no output
        for size in (nbytes, want.numel() * 2):
            with pytest.raises(torch.OutOfMemoryError):
                while True:
                    fill.append(torch.empty(size, dtype=torch.uint8, device=cuda))
        del room  # the one block for the output, between blocks in use
        got = call()
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(nbytes, dtype=torch.uint8, device=cuda)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)
