#!/usr/bin/env python3
"""Benchmark of the fused RMSNorm + SiLU-and-mul path on one MI355X.

One *step* is one pass of the hot path over one batch of synthetic input at
the Qwen2.5-1.5B prefill shape (BASELINE configs 1 and 2): RMSNorm over
x [2048, 1536] fp16 followed by SiLU-and-mul over gate/up [2048, 8960] fp16.
Every step runs on the next of several buffer sets whose total footprint is
above 1 GiB (4x the 256 MB Infinity Cache), so each step reads cold HBM.

`value` is the whole job's algorithmic bandwidth over the timed steps:
K * (RMSNorm bytes + SiLU-and-mul bytes) / elapsed, in GB/s, with the inputs
already resident in HBM.  Algorithmic bytes: RMSNorm (2*M*N + N) * 2,
SiLU-and-mul 3 * M * I * 2.

Also reported on the same JSON line:
  roofline      dominant kernel (SiLU-and-mul, C2): bytes / average launch
                duration from HIP events on the launch stream, vs 8 TB/s;
                traffic = FETCH_SIZE + WRITE_SIZE per launch from the
                committed rocprofv3 PMC summary (profiles/), when present;
  cpu_baseline  the reference's naive PyTorch path (restated in the oracle),
                timed on the host cores on a bounded sample of the workload;
  kernels       per-kernel durations and GB/s (C1, C2, C4), cold and warm;
  decode        C3 latency per call (host-inclusive and device-only) and
                inside a hipGraph of 28 x (RMSNorm, SiLU-and-mul, RMSNorm);
  gate_up_silu  the fused gate/up projections + SiLU-and-mul at decode rows
                vs the reference's two-GEMM + SiLU-and-mul chain;
  gate_up_silu_prefill  the same at prefill rows (tiled MFMA GEMM), same baseline;
  w8a16         the weight-only int8 linear vs fp16 torch.matmul (hipBLASLt);
  gate_up_silu_w8a16  int8 gate/up + SiLU-and-mul vs two W8A16 linears + SiLU-and-mul;
  linear16_down the MLP's down projection on the HIP 16-bit linear vs torch's
                linear (hipBLASLt) at decode rows;
  copy_ceiling  a plain 16-byte streaming copy on the same device;
  ceilings      the same probe (and a two-input, one-output variant) at each
                kernel's own byte count and access mix, cold, and each
                kernel's time as a fraction of it.

    python bench.py [--gpus 1] [--steps K] [--warmup W]
"""
from __future__ import annotations

import argparse
import ctypes
import importlib
import json
import os
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
PKG = "llm-inference-optimizer_amd"
PEAK_GBS = 8000.0  # MI355X HBM3E, published
METRIC = "achieved HBM GB/s (% of 8 TB/s peak) for RMSNorm+SwiGLU; decode-row latency µs"
MALL_BYTES = 256 * 2**20
MIN_FOOTPRINT = 1 << 30


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def parse_args():
    p = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=2000)
    p.add_argument("--warmup", type=int, default=50)
    p.add_argument("--cpu-seconds", type=float, default=12.0,
                   help="wall-clock budget of the CPU-baseline sample")
    p.add_argument("--skip-cpu", action="store_true")
    p.add_argument("--skip-extras", action="store_true", help="headline only (no C4 / decode / copy)")
    p.add_argument("--skip-e2e", action="store_true", help="no end-to-end before/after leg")
    p.add_argument("--only", choices=["c2-silu", "c1-rms", "c1-add-rms", "c4-silu", "c4-rms", "c1-decomp", "copy", "ceilings", "decode", "linear16", "linear16-table", "gate-up",
                                      "gate-up-prefill", "gate-up-w8", "gate-up-w8-decode", "w8a16", "w8a16-decode", "decode-wide-rows",
                                      "w8a16-prefill", "w8a16-prefill-1.5b", "prefill-core",
                                      "gate-up-w8-prefill", "w8a16-prefill-wide", "w8a16-prefill-narrow",
                                      "gate-up-prefill-sweep", "tile-plans", "w8a16-prefill-ragged", "w8-decomp", "w8-layouts", "w8-layouts8", "w8-stream-sweep", "gu16-stream-sweep", "stream-sweep16", "stream-sweep16-wide", "stream-sweep-r8", "stream-sweep-m4", "stream-sweep16-k", "stream-sweep-dualn", "stream-sweep-dual32", "stream-sweep-3b14b", "stream-sweep-bal", "stream-sweep-few16", "stream-sweep-dual4", "stream-sweep-14b-wide", "stream-sweep-smallm", "l16-stream-sweep", "stream-sweep32", "stream-sweep64", "stage3",
                                      "e2e-compact", "e2e-int8-compact"],
                   default=None,
                   help="run one kernel loop only (for profiler runs)")
    p.add_argument("--e2e-int8", action="store_true",
                   help="fp16 vs int8-weight (W8A16) decode end to end, after the reference's run_stage7_e2e.py")
    p.add_argument("--e2e", action="store_true",
                   help="instead of the kernel bench: TTFT and decode tok/s of a random-init Qwen2-1.5B "
                        "architecture before and after patch_model_with_fused_kernels (the reference's "
                        "benchmarks/run_stage3_e2e.py method)")
    p.add_argument("--seq-lens", type=int, nargs="+", default=[128, 512, 1024, 2048])
    p.add_argument("--gen-len", type=int, default=32)
    p.add_argument("--trials", type=int, default=5)
    p.add_argument("--full-json", default=None, metavar="PATH",
                   help="also write the full result (every leg) to PATH; stdout carries the compact line")
    p.add_argument("--rocprof-summary", nargs="+", metavar="DIR", default=None,
                   help="summarise rocprofv3 output directories (kernel trace and/or PMC) and exit; "
                        "no GPU needed")
    return p.parse_args()


class Ctx:
    """Bound C-ABI entry points.  Launch closures read `self.stream` at call
    time, so a graph capture can redirect them to the capturing stream."""

    def __init__(self):
        import torch

        sys.path.insert(0, str(ROOT))
        self.torch = torch
        self.pkg = importlib.import_module(PKG)
        self.L = importlib.import_module(PKG + "._lib")
        self.lib = self.L.load()
        self.dev = torch.device("cuda:0")
        torch.cuda.set_device(self.dev)
        self.stream = torch.cuda.current_stream(self.dev).cuda_stream
        self._scratch = None
        probe_path = ROOT / PKG / "libmi355_probe.so"
        self.probe = ctypes.CDLL(str(probe_path)) if probe_path.exists() else None
        if self.probe is not None:
            self.probe.mi355_probe_copy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64,
                                                    ctypes.c_int, ctypes.c_void_p]
            self.probe.mi355_probe_copy.restype = ctypes.c_int
            self.probe.mi355_probe_add2.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                                    ctypes.c_int64, ctypes.c_void_p]
            self.probe.mi355_probe_add2.restype = ctypes.c_int
            self.probe.mi355_probe_empty.argtypes = [ctypes.c_void_p]
            self.probe.mi355_probe_empty.restype = ctypes.c_int
            self.probe.mi355_probe_read.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p,
                                                    ctypes.c_void_p]
            self.probe.mi355_probe_read.restype = ctypes.c_int
            i32 = ctypes.c_int
            self.probe.mi355_probe_w8_stream.argtypes = [ctypes.c_void_p, i32, i32, ctypes.c_int64, ctypes.c_void_p,
                                                         i32, ctypes.c_int64, i32, i32, i32, i32, i32, i32, i32,
                                                         ctypes.c_void_p, ctypes.c_void_p]
            self.probe.mi355_probe_w8_stream.restype = ctypes.c_int
            vp = ctypes.c_void_p
            self.probe.mi355_probe_w8a16_stream.argtypes = [vp, vp, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32,
                                                            i32, vp]
            self.probe.mi355_probe_w8a16_stream.restype = ctypes.c_int
            self.probe.mi355_probe_w8a16_stream_plan.argtypes = [i32, i32, i32, i32, i32, ctypes.POINTER(i32)]
            self.probe.mi355_probe_linear16_stream_plan.argtypes = [i32, i32, i32, i32, ctypes.POINTER(i32)]
            self.probe.mi355_probe_gate_up16_stream_plan.argtypes = [i32, i32, i32, i32, ctypes.POINTER(i32)]
            self.probe.mi355_probe_w8a16_stream_plan.restype = None
            self.probe.mi355_probe_w8a16_stream_loads.argtypes = [vp, vp, i32, i32, i32, i32, i32, i32, i32, i32,
                                                                  vp, vp]
            self.probe.mi355_probe_w8a16_stream_loads.restype = ctypes.c_int
            self.probe.mi355_probe_gate_up16_stream.argtypes = [vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32, vp]
            self.probe.mi355_probe_gate_up16_stream.restype = ctypes.c_int
            self.probe.mi355_probe_linear16_stream.argtypes = [vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32, vp]
            self.probe.mi355_probe_linear16_stream.restype = ctypes.c_int

    def check(self, fn, st):
        if st:
            msg = self.lib.mi355_last_error().decode(errors="replace")
            raise self.L.KernelError(fn, st, msg)

    def rms_call(self, x, w, y, eps=1e-6):
        M, N = x.shape
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_rmsnorm_fwd
        args = (x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, N, N, ctypes.c_float(eps), code,
                self.L.DTYPE_CODE[w.dtype], code)

        def call():
            st = f(*args, self.stream)
            if st:
                self.check("mi355_rmsnorm_fwd", st)
        return call

    def add_rms_call(self, x, r, w, y, h, eps=1e-6):
        M, N = x.shape
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_add_rmsnorm_fwd
        args = (x.data_ptr(), r.data_ptr(), w.data_ptr(), y.data_ptr(), h.data_ptr(), M, N, N, N, N, N,
                ctypes.c_float(eps), code, self.L.DTYPE_CODE[w.dtype], code)

        def call():
            st = f(*args, self.stream)
            if st:
                self.check("mi355_add_rmsnorm_fwd", st)
        return call

    def silu_call(self, g, u, o):
        code = self.L.DTYPE_CODE[g.dtype]
        f = self.lib.mi355_silu_mul_fwd
        args = (g.data_ptr(), u.data_ptr(), o.data_ptr(), g.numel(), code, code)

        def call():
            st = f(*args, self.stream)
            if st:
                self.check("mi355_silu_mul_fwd", st)
        return call

    def gate_up_call(self, x, wg, wu, o):
        M, K = x.shape
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_gate_up_silu_fwd
        args = (x.data_ptr(), wg.data_ptr(), wu.data_ptr(), o.data_ptr(), M, K, wg.shape[0], K, K, wg.shape[0],
                code, code)

        def call():
            st = f(*args, self.stream)
            if st:
                self.check("mi355_gate_up_silu_fwd", st)
        return call

    def gate_up_w8_call(self, x, qg, sg, qu, su, o):
        M, K = x.shape
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_gate_up_silu_w8a16_fwd
        args = (x.data_ptr(), qg.data_ptr(), qu.data_ptr(), sg.data_ptr(), su.data_ptr(), o.data_ptr(), M, K,
                qg.shape[0], K, K, qg.shape[0], code, self.L.DTYPE_CODE[sg.dtype], code)

        def call():
            st = f(*args, self.stream)
            if st:
                self.check("mi355_gate_up_silu_w8a16_fwd", st)
        return call

    def scratch(self, nbytes):
        """`nbytes` of device scratch for the linears' split K, shared by every
        call on the stream (their kernels run in order): (tensor, address)."""
        if nbytes <= 0:
            return None, None
        if self._scratch is None or self._scratch.numel() < nbytes:
            self._scratch = self.torch.empty(nbytes, dtype=self.torch.uint8, device=self.dev)
        return self._scratch, self._scratch.data_ptr()

    def w8a16_call(self, x, q, scale, out, bias=None, split=True):
        """The int8 linear as the package calls it, with the workspace its
        split-K kernels ask for; split=False: its unsplit kernels."""
        M, K = x.shape
        N = q.shape[0]
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_w8a16_linear_ws_fwd
        nbytes = self.lib.mi355_w8a16_linear_workspace(M, K, N) if split else 0
        work, wp = self.scratch(nbytes)
        args = (x.data_ptr(), q.data_ptr(), scale.data_ptr(), bias.data_ptr() if bias is not None else None,
                out.data_ptr(), M, K, N, K, K, N, code, self.L.DTYPE_CODE[scale.dtype],
                self.L.DTYPE_CODE[bias.dtype] if bias is not None else 0, code, wp, nbytes)

        def call(keep=work):
            st = f(*args, self.stream)
            if st:
                self.check("mi355_w8a16_linear_fwd", st)
        return call

    def linear16_call(self, x, w, out, bias=None, split=True):
        """The 16-bit linear, with the workspace rule of w8a16_call."""
        M, K = x.shape
        N = w.shape[0]
        code = self.L.DTYPE_CODE[x.dtype]
        f = self.lib.mi355_linear16_ws_fwd
        nbytes = self.lib.mi355_linear16_workspace(M, K, N) if split else 0
        work, wp = self.scratch(nbytes)
        args = (x.data_ptr(), w.data_ptr(), bias.data_ptr() if bias is not None else None, out.data_ptr(),
                M, K, N, K, K, N, code, self.L.DTYPE_CODE[bias.dtype] if bias is not None else 0, code, wp, nbytes)

        def call(keep=work):
            st = f(*args, self.stream)
            if st:
                self.check("mi355_linear16_fwd", st)
        return call

    def copy_call(self, src, dst):
        f = self.probe.mi355_probe_copy
        args = (src.data_ptr(), dst.data_ptr(), src.numel() * src.element_size(), 0)

        def call():
            if f(*args, self.stream):
                raise RuntimeError("probe copy failed")
        return call

    def empty_call(self):
        f = self.probe.mi355_probe_empty

        def call():
            if f(self.stream):
                raise RuntimeError("probe empty kernel failed")
        return call

    def read_call(self, src, sink):
        f = self.probe.mi355_probe_read
        args = (src.data_ptr(), src.numel() * src.element_size(), sink.data_ptr())

        def call():
            if f(*args, self.stream):
                raise RuntimeError("probe read failed")
        return call

    def w8_stream_call(self, q, sink, rpw, waves, g, u, layout=0, x=None, xl=1, stagger=0):
        """The int8 weight stream of a decode kernel's launch shape, without
        its MFMAs, reduction and epilogue (csrc/probe/w8_stream.hip)."""
        n, k = q.shape
        f = self.probe.mi355_probe_w8_stream
        args = (q.data_ptr(), n, k, k, x.data_ptr() if x is not None else None, x.shape[0] if x is not None else 0,
                x.shape[1] if x is not None else 0, rpw, waves, g, u, layout, xl, stagger, sink.data_ptr())

        def call():
            if f(*args, self.stream):
                raise RuntimeError(f"probe w8 stream failed for {args[5:12]}")
        return call

    def w8_stream_plan(self, rows, k, n, dual, cus):
        """The W8A16 decode kernel's launch plan (rpw, r4, waves, u), from the
        same source the library compiles."""
        out4 = (ctypes.c_int * 4)()
        self.probe.mi355_probe_w8a16_stream_plan(rows, k, n, int(dual), cus, out4)
        return tuple(out4)

    def gu16_stream_plan(self, rows, k, n, cus):
        """The 16-bit gate/up + SiLU-and-mul's stream launch plan."""
        out4 = (ctypes.c_int * 4)()
        self.probe.mi355_probe_gate_up16_stream_plan(rows, k, n, cus, out4)
        return tuple(out4)

    def l16_stream_plan(self, rows, k, n, cus):
        """The 16-bit linear's stream launch plan (rpw, r4, waves, u)."""
        out4 = (ctypes.c_int * 4)()
        self.probe.mi355_probe_linear16_stream_plan(rows, k, n, cus, out4)
        return tuple(out4)

    def w8_stream_loads_call(self, x, q, sink, rpw, r4, waves, u, with_x):
        """The W8A16 decode kernel's loads alone at a launch shape."""
        M, K = x.shape
        N = q.shape[0]
        f = self.probe.mi355_probe_w8a16_stream_loads
        args = (x.data_ptr(), q.data_ptr(), M, K, N, rpw, r4, waves, u, int(with_x), sink.data_ptr())

        def call():
            if f(*args, self.stream):
                raise RuntimeError(f"probe w8a16 stream loads failed for {args[2:10]}")
        return call

    def w8_stream_plan_call(self, x, q, scale, out, rpw, r4, waves, u, q2=None, scale2=None):
        """The W8A16 decode kernel with a forced launch shape (fp16 x and out,
        fp32 scales; csrc/probe/w8_stream_plan.hip)."""
        M, K = x.shape
        N = q.shape[0]
        f = self.probe.mi355_probe_w8a16_stream
        args = (x.data_ptr(), q.data_ptr(), scale.data_ptr(), q2.data_ptr() if q2 is not None else None,
                scale2.data_ptr() if scale2 is not None else None, out.data_ptr(), M, K, N, rpw, r4, waves, u)

        def call():
            if f(*args, self.stream):
                raise RuntimeError(f"probe w8a16 stream failed for {args[6:]}")
        return call

    def gate_up16_stream_call(self, x, wg, wu, out, rpw, r4, waves, u):
        """The 16-bit gate/up + SiLU-and-mul through the weight-streaming
        kernel at a forced launch shape (fp16; csrc/probe/w8_stream_plan.hip)."""
        M, K = x.shape
        N = wg.shape[0]
        f = self.probe.mi355_probe_gate_up16_stream
        args = (x.data_ptr(), wg.data_ptr(), wu.data_ptr(), out.data_ptr(), M, K, N, rpw, r4, waves, u)

        def call():
            if f(*args, self.stream):
                raise RuntimeError(f"probe gate_up16 stream failed for {args[4:]}")
        return call

    def linear16_stream_call(self, x, w, out, rpw, r4, waves, u, bias=None):
        """The 16-bit linear through the weight-streaming kernel at a forced
        launch shape (fp16, bias fp16 or none; csrc/probe/w8_stream_plan.hip)."""
        M, K = x.shape
        N = w.shape[0]
        f = self.probe.mi355_probe_linear16_stream
        args = (x.data_ptr(), w.data_ptr(), bias.data_ptr() if bias is not None else None, out.data_ptr(), M, K, N,
                rpw, r4, waves, u)

        def call():
            if f(*args, self.stream):
                raise RuntimeError(f"probe linear16 stream failed for {args[4:]}")
        return call

    def add2_call(self, a, b, dst):
        f = self.probe.mi355_probe_add2
        args = (a.data_ptr(), b.data_ptr(), dst.data_ptr(), a.numel() * a.element_size())

        def call():
            if f(*args, self.stream):
                raise RuntimeError("probe add2 failed")
        return call


def rand(ctx, shape, seed, dtype, mean=0.0, std=1.0):
    torch = ctx.torch
    g = torch.Generator(device=ctx.dev)
    g.manual_seed(seed)
    t = torch.randn(*shape, generator=g, device=ctx.dev, dtype=torch.float32)
    if mean != 0.0 or std != 1.0:
        t = t.mul_(std).add_(mean)
    return t.to(dtype)


def n_sets(bytes_per_set: int) -> int:
    return max(1, -(-MIN_FOOTPRINT // bytes_per_set))


def spin_up(ctx, calls, ms=30.0):
    """Launches `calls` (cycled) for about `ms` of device time, untimed: the
    first launches after host-side setup run below full clocks, and a pass
    over freshly generated buffers pays for their write-backs."""
    torch = ctx.torch
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    n = 0
    while True:
        for c in calls:
            c()
        n += len(calls)
        end.record()
        end.synchronize()
        if start.elapsed_time(end) >= ms or n > 100000:
            return


def time_loop(ctx, calls, iters, warmup=5):
    """Average device time per iteration of `calls` (list cycled), from HIP
    events recorded on the launch stream around `iters` back-to-back launches."""
    torch = ctx.torch
    for i in range(warmup):
        calls[i % len(calls)]()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for i in range(iters):
        calls[i % len(calls)]()
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) * 1e3 / iters  # us


def time_graph(ctx, calls, iters, replays=5):
    """Average device time per launch with `iters` launches captured in one
    hipGraph (no host launch cost between kernels)."""
    torch = ctx.torch
    s = torch.cuda.Stream(device=ctx.dev)
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    old = ctx.stream
    try:
        with torch.cuda.stream(s):
            ctx.stream = s.cuda_stream  # the closures now launch on the capture stream
            for c in calls:
                c()
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=s):
                for i in range(iters):
                    calls[i % len(calls)]()
    finally:
        ctx.stream = old
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(replays):
        graph.replay()
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) * 1e3 / (replays * iters)


def kernel_entry(name, nbytes, us, extra=None):
    d = {"kernel": name, "bytes": nbytes, "us": round(us, 3), "GBps": round(nbytes / us / 1e3, 1),
         "frac_of_peak": round(nbytes / us / 1e3 / PEAK_GBS, 4)}
    if extra:
        d.update(extra)
    return d


def read_traffic(label: str):
    """HBM bytes per launch (calibrated FETCH_SIZE + WRITE_SIZE) recorded from
    rocprofv3 PMC runs in profiles/traffic.json, if that summary exists."""
    p = ROOT / "profiles" / "traffic.json"
    if not p.exists():
        return None
    try:
        d = json.loads(p.read_text()).get(label)
        return None if d is None else d.get("traffic_bytes")
    except Exception:
        return None


def cpu_baseline(M, N, I, budget_s):
    """The reference's naive PyTorch path (oracle restatement) on the host
    cores: RMSNorm [M,N] + SiLU-and-mul [M,I] fp16, repeated for ~budget_s."""
    import torch

    sys.path.insert(0, str(ROOT))
    from oracle import oracle as orc

    cores = len(os.sched_getaffinity(0))
    env_threads = os.environ.get("OMP_NUM_THREADS")
    if env_threads and env_threads.isdigit():
        cores = min(cores, int(env_threads))
    torch.set_num_threads(cores)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(M, N, generator=g).to(torch.float16)
    w = (1 + 0.1 * torch.randn(N, generator=g)).to(torch.float16)
    gate = torch.randn(M, I, generator=g).to(torch.float16)
    up = torch.randn(M, I, generator=g).to(torch.float16)
    orc.naive_rmsnorm_torch(x, w)
    orc.naive_silu_mul_torch(gate, up)
    times = []
    t_end = time.perf_counter() + budget_s
    while time.perf_counter() < t_end or len(times) < 3:
        t0 = time.perf_counter()
        orc.naive_rmsnorm_torch(x, w)
        orc.naive_silu_mul_torch(gate, up)
        times.append(time.perf_counter() - t0)
        if len(times) >= 20000:
            break
    step = statistics.median(times)
    nbytes = (2 * M * N + N) * 2 + 3 * M * I * 2
    try:
        model = next(line.split(":", 1)[1].strip() for line in open("/proc/cpuinfo") if line.startswith("model name"))
    except Exception:
        model = "unknown"
    return {"value": round(nbytes / step / 1e9, 3), "unit": "GB/s", "cores": torch.get_num_threads(),
            "kind": "port", "ms_per_step": round(step * 1e3, 3), "steps_timed": len(times),
            "cpu_model": model,
            "sample": f"naive torch RMSNorm [{M},{N}] + SiLU-and-mul [{M},{I}] fp16 on host tensors, "
                      f"median of {len(times)} steps in ~{budget_s:.0f}s"}


# --------------------------------------------------------- rocprof summaries

# Algorithmic bytes per launch, keyed by (kernel-name fragment, grid size X):
# used to turn rocprofv3 durations into GB/s and to set PMC traffic against
# the ideal.  Grid sizes are in threads, as rocprofv3 reports them.
KNOWN_LAUNCHES = {
    ("silu_mul_chunks<mi355::F16, mi355::F16, 512, 2>", 1146880): ("C2 SiLU-and-mul [2048,8960] fp16",
                                                                   3 * 2048 * 8960 * 2),
    ("rmsnorm_wave_rows<mi355::F16, mi355::F16, mi355::F16, 3, 1, false>", 131072): (
        "C1 RMSNorm [2048,1536] fp16", (2 * 2048 * 1536 + 1536) * 2),
    ("rmsnorm_wave_rows<mi355::F16, mi355::F16, mi355::F16, 3, 2, true>", 65536): (
        "C1 residual add + RMSNorm [2048,1536] fp16", (4 * 2048 * 1536 + 1536) * 2),
    ("silu_mul_chunks<mi355::BF16, mi355::BF16, 256, 4>", 9699328): (
        "C4 SiLU-and-mul [16384,18944] bf16", 3 * 16384 * 18944 * 2),
    ("rmsnorm_block_rows<mi355::BF16, mi355::BF16, mi355::BF16, 2, 1, false>", 4194304): (
        "C4 RMSNorm [16384,3584] bf16", (2 * 16384 * 3584 + 3584) * 2),
    ("stream_copy", 67108864): ("copy probe, 1 GiB", 2 << 30),
    ("w8a16_stream<mi355::F16, mi355::F16, 1, 2, 2, true, 2>", 8960 // 4 * 64 * 2): (
        "gate/up + SiLU-and-mul, 8 rows, [8960,1536] weights, fp16",
        2 * 8960 * 1536 * 2 + 8 * 1536 * 2 + 8 * 8960 * 2),
    # W8A16 decode (w8a16_stream) at its launch plan, 8 rows: grid = workgroups x 64 x waves
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 2, 1, false, 1>", 1120 * 64 * 2): (
        "W8A16 1.5B gate/up, 8 rows, [8960,1536] int8, fp16", 8960 * 1536 + 4 * 8960 + 8 * 1536 * 2 + 8 * 8960 * 2),
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 2, 1, false, 1>", 256 * 64 * 12): (
        "W8A16 1.5B down, 8 rows, [1536,8960] int8, fp16", 1536 * 8960 + 4 * 1536 + 8 * 8960 * 2 + 8 * 1536 * 2),
    ("w8a16_stream<mi355::BF16, mi355::BF16, 4, 2, 1, false, 1>", 1184 * 64 * 2): (
        "W8A16 7B gate/up, 8 rows, [18944,3584] int8, bf16",
        18944 * 3584 + 4 * 18944 + 8 * 3584 * 2 + 8 * 18944 * 2),
    ("w8a16_stream<mi355::BF16, mi355::BF16, 4, 2, 1, false, 1>", 224 * 64 * 8): (
        "W8A16 7B down, 8 rows, [3584,18944] int8, bf16",
        3584 * 18944 + 4 * 3584 + 8 * 18944 * 2 + 8 * 3584 * 2),
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 2, 1, true, 1>", 1120 * 64 * 2): (
        "int8 gate/up + SiLU-and-mul 1.5B, 8 rows, 2 x [8960,1536] int8, fp16",
        2 * 8960 * 1536 + 8 * 8960 + 8 * 1536 * 2 + 8 * 8960 * 2),
    ("w8a16_stream<mi355::BF16, mi355::BF16, 4, 2, 1, true, 1>", 1184 * 64 * 1): (
        "int8 gate/up + SiLU-and-mul 7B, 8 rows, 2 x [18944,3584] int8, bf16",
        2 * 18944 * 3584 + 8 * 18944 + 8 * 3584 * 2 + 8 * 18944 * 2),
    # 32 - 64 rows (bench.py --only decode-wide-rows): the stream kernel at 32 rows of the 1.5B
    # down projection, split K (first pass; then split_k_reduce) for the 7B one
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 8, 1, false, 1>", 256 * 64 * 8): (
        "W8A16 1.5B down, 32 rows, [1536,8960] int8, fp16", 1536 * 8960 + 4 * 1536 + 32 * 8960 * 2 + 32 * 1536 * 2),
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 8, 1, false, 2>", 256 * 64 * 8): (
        "16-bit linear, 32 rows, [1536,8960] weights, fp16 (1.5B down)",
        1536 * 8960 * 2 + 32 * 8960 * 2 + 32 * 1536 * 2),
    ("w8a16_stream<mi355::F16, mi355::F16, 2, 2, 2, false, 2>", 256 * 64 * 8): (
        "16-bit linear, 8 rows, [1536,8960] weights, fp16 (1.5B down)", 1536 * 8960 * 2 + 8 * 8960 * 2 + 8 * 1536 * 2),
    ("w8a16_stream<mi355::BF16, mi355::BF16, 4, 2, 1, false, 2>", 224 * 64 * 8): (
        "16-bit linear, 8 rows, [3584,18944] weights, bf16 (7B down)", 3584 * 18944 * 2 + 8 * 18944 * 2 + 8 * 3584 * 2),
    # tiled GEMMs: (label, algorithmic bytes, flops).  The first passes of split K write fp32
    # sums of 9 K ranges (64 x 128 tiles) or 2 (128 x 128 tiles)
    ("tiled_gemm<mi355::BF16, 1, mi355::F32, 1, 4, 2, 1, 4, 4, 1, 0, 4>", 28 * 9 * 256): (
        "W8A16 7B down, 48 rows, [3584,18944] int8, bf16 (split K, first pass)",
        3584 * 18944 + 48 * 18944 * 2 + 9 * 48 * 3584 * 4, 2 * 48 * 18944 * 3584),
    ("tiled_gemm<mi355::BF16, 0, mi355::F32, 1, 4, 2, 1, 4, 4, 1, 0, 4>", 28 * 9 * 256): (
        "16-bit linear, 64 rows, [3584,18944] weights, bf16 (7B down; split K, first pass)",
        3584 * 18944 * 2 + 64 * 18944 * 2 + 9 * 64 * 3584 * 4, 2 * 64 * 18944 * 3584),
    ("tiled_gemm<mi355::F16, 1, mi355::F32, 2, 4, 2, 1, 4, 3, 1, 0, 3>", 96 * 2 * 512): (
        "W8A16 prefill down, 1024 rows, [1536,8960] int8, fp16 (split K, first pass)",
        1536 * 8960 + 1024 * 8960 * 2 + 2 * 1024 * 1536 * 4, 2 * 1024 * 8960 * 1536),
    # the 1.5B gate/up at 1024 and 4096 rows runs as a column split: whole rounds of 256 x 128
    # tiles over the first 8192 columns, then 768 columns in 64 x 64 or 256 x 64 tiles
    ("tiled_gemm<mi355::F16, 0, mi355::F16, 2, 4, 4, 1, 1, 2, 1, 0, 3>", 256 * 512): (
        "gate/up + SiLU-and-mul prefill, 1024 rows, first 8192 of 8960 columns, fp16",
        2 * 8192 * 1536 * 2 + 1024 * 1536 * 2 + 1024 * 8192 * 2, 4 * 1024 * 1536 * 8192),
    ("tiled_gemm<mi355::F16, 0, mi355::F16, 2, 2, 1, 1, 1, 3, 1, 0, 3>", 192 * 256): (
        "gate/up + SiLU-and-mul prefill, 1024 rows, last 768 of 8960 columns, fp16",
        2 * 768 * 1536 * 2 + 1024 * 1536 * 2 + 1024 * 768 * 2, 4 * 1024 * 1536 * 768),
    ("tiled_gemm<mi355::F16, 0, mi355::F16, 2, 4, 4, 1, 1, 2, 1, 0, 3>", 1024 * 512): (
        "gate/up + SiLU-and-mul prefill, 4096 rows, first 8192 of 8960 columns, fp16",
        2 * 8192 * 1536 * 2 + 4096 * 1536 * 2 + 4096 * 8192 * 2, 4 * 4096 * 1536 * 8192),
    ("tiled_gemm<mi355::F16, 0, mi355::F16, 4, 2, 2, 1, 1, 3, 0, 0, 3>", 192 * 512): (
        "gate/up + SiLU-and-mul prefill, 4096 rows, last 768 of 8960 columns, fp16",
        2 * 768 * 1536 * 2 + 4096 * 1536 * 2 + 4096 * 768 * 2, 4 * 4096 * 1536 * 768),
    # one int8 matrix, unsplit, by the tile plan
    ("tiled_gemm<mi355::F16, 1, mi355::F16, 1, 2, 1, 1, 0, 4, 0, 0, 4>", 768 * 128): (
        "W8A16 prefill q/o, 1024 rows, [1536,1536] int8, fp16 (32x64 tiles)",
        1536 * 1536 + 4 * 1536 + 1024 * 1536 * 2 + 1024 * 1536 * 2, 2 * 1024 * 1536 * 1536),
    ("tiled_gemm<mi355::F16, 1, mi355::F16, 2, 4, 3, 1, 0, 2, 1, 4, 2>", 420 * 512): (
        "W8A16 prefill gate/up, 1024 rows, [8960,1536] int8, fp16 (192x128 tiles)",
        8960 * 1536 + 4 * 8960 + 1024 * 1536 * 2 + 1024 * 8960 * 2, 2 * 1024 * 1536 * 8960),
    ("tiled_gemm<mi355::F16, 1, mi355::F16, 2, 4, 2, 1, 0, 3, 1, 0, 3>", 2240 * 512): (
        "W8A16 prefill gate/up, 4096 rows, [8960,1536] int8, fp16 (128x128 tiles)",
        8960 * 1536 + 4 * 8960 + 4096 * 1536 * 2 + 4096 * 8960 * 2, 2 * 4096 * 1536 * 8960),
}
COPY_READ_KIB = COPY_WRITE_KIB = (1 << 30) / 1024


def _match_launch(name: str, grid: int):
    for (frag, g), v in KNOWN_LAUNCHES.items():
        if frag in name and g == grid:
            return frag, v
    return None, None


def rocprof_summary(dirs):
    """Markdown summary of rocprofv3 CSV output: per (kernel, grid) average
    duration and GB/s from *_kernel_trace.csv; per-dispatch FETCH_SIZE /
    WRITE_SIZE from *_counter_collection.csv, scaled by the factor that makes
    the copy probe read and write exactly 1 GiB."""
    import csv
    import glob

    out = []
    pmc = {}  # (kernel fragment, grid, counter) -> per-dispatch values, over all dirs
    pmc_all = {}  # the same for every kernel, by shortened name
    for d in dirs:
        for f in sorted(glob.glob(os.path.join(d, "*kernel_stats.csv"))):
            # rocprofv3 --stats: every kernel of the run, whatever its grid
            out.append(f"### kernel stats: {f}\n")
            out.append("| kernel | calls | avg us | min us | max us | % of GPU time |")
            out.append("|---|---|---|---|---|---|")
            for r in csv.DictReader(open(f)):
                out.append(f"| {r['Name'][:160]} | {r['Calls']} | {float(r['AverageNs']) / 1e3:.3f} | "
                           f"{float(r['MinNs']) / 1e3:.3f} | {float(r['MaxNs']) / 1e3:.3f} | "
                           f"{float(r['Percentage']):.2f} |")
            out.append("")
        for f in sorted(glob.glob(os.path.join(d, "*kernel_trace.csv"))):
            out.append(f"### kernel trace: {f}\n")
            out.append("| kernel | grid (threads) | launches | avg us | median us | algorithmic bytes | GB/s (avg) | "
                       "% of 8 TB/s | TFLOP/s (avg) | % of 2.5 PFLOP/s |")
            out.append("|---|---|---|---|---|---|---|---|---|---|")
            groups = {}
            for r in csv.DictReader(open(f)):
                grid = int(r["Grid_Size_X"]) * int(r["Grid_Size_Y"]) * int(r["Grid_Size_Z"])  # threads
                frag, known = _match_launch(r["Kernel_Name"], grid)
                if known is None:
                    continue
                groups.setdefault((frag, grid), []).append(int(r["End_Timestamp"]) - int(r["Start_Timestamp"]))
            for (frag, grid), v in groups.items():
                label, nbytes = KNOWN_LAUNCHES[(frag, grid)][:2]
                flops = KNOWN_LAUNCHES[(frag, grid)][2] if len(KNOWN_LAUNCHES[(frag, grid)]) > 2 else None
                v.sort()
                avg = sum(v) / len(v) / 1e3
                gbs = nbytes / avg / 1e3
                tf = f"{flops / avg / 1e6:.1f} | {100 * flops / avg / 1e6 / MFMA_PEAK_TFLOPS:.1f}" if flops else "- | -"
                out.append(f"| {frag} ({label}) | {grid} | {len(v)} | {avg:.3f} | {v[len(v) // 2] / 1e3:.3f} | "
                           f"{nbytes} | {gbs:.0f} | {100 * gbs / PEAK_GBS:.1f} | {tf} |")
            out.append("")
        for f in sorted(glob.glob(os.path.join(d, "*counter_collection.csv"))):
            for r in csv.DictReader(open(f)):
                name = _short_name(r["Kernel_Name"])
                pmc_all.setdefault((name, int(r["Grid_Size"]), r["Counter_Name"]), []).append(float(r["Counter_Value"]))
                frag, known = _match_launch(r["Kernel_Name"], int(r["Grid_Size"]))
                if known is None:
                    continue
                pmc.setdefault((frag, int(r["Grid_Size"]), r["Counter_Name"]), []).append(float(r["Counter_Value"]))
    traffic = {}
    if pmc:
        cf = pmc.get(("stream_copy", 67108864, "FETCH_SIZE"))
        cw = pmc.get(("stream_copy", 67108864, "WRITE_SIZE"))
        fscale = COPY_READ_KIB / (sum(cf) / len(cf)) if cf else None
        wscale = COPY_WRITE_KIB / (sum(cw) / len(cw)) if cw else None
        out.append("### PMC traffic (KiB per dispatch, then scaled)\n")
        out.append(f"Calibration: the copy probe reads and writes exactly 1 GiB per launch; "
                   f"FETCH_SIZE scale = {fscale if fscale is None else round(fscale, 5)}, "
                   f"WRITE_SIZE scale = {wscale if wscale is None else round(wscale, 5)}.\n")
        out.append("| kernel | dispatches | FETCH_SIZE KiB | WRITE_SIZE KiB | scaled HBM bytes | algorithmic bytes | ratio |")
        out.append("|---|---|---|---|---|---|---|")
        keys = sorted({(k[0], k[1]) for k in pmc})
        for frag, grid in keys:
            fv = pmc.get((frag, grid, "FETCH_SIZE"))
            wv = pmc.get((frag, grid, "WRITE_SIZE"))
            if not fv or not wv or fscale is None or wscale is None:
                continue
            fk = sum(fv) / len(fv)
            wk = sum(wv) / len(wv)
            tb = (fk * fscale + wk * wscale) * 1024
            label, nbytes = KNOWN_LAUNCHES[(frag, grid)][:2]
            out.append(f"| {frag} ({label}) | {len(fv)} | {fk:.1f} | {wk:.1f} | {tb:.0f} | {nbytes} | {tb / nbytes:.4f} |")
            traffic[label] = {"traffic_bytes": round(tb), "algorithmic_bytes": nbytes,
                              "fetch_kib": round(fk, 1), "write_kib": round(wk, 1)}
        out.append("")
        occ_names = tuple(sorted({k[2] for k in pmc} - {"FETCH_SIZE", "WRITE_SIZE"}))
        occ_keys = sorted({(k[0], k[1]) for k in pmc if k[2] in occ_names})
        if occ_keys:
            out.append("### Other counters and derived metrics (per dispatch, averaged over dispatches)\n")
            out.append("| kernel | dispatches | " + " | ".join(occ_names) + " |")
            out.append("|---|---|" + "---|" * len(occ_names))
            for frag, grid in occ_keys:
                cells = []
                for c in occ_names:
                    v = pmc.get((frag, grid, c))
                    cells.append(f"{sum(v) / len(v):.2f}" if v else "-")
                nd = max(len(pmc.get((frag, grid, c), [])) for c in occ_names)
                label = KNOWN_LAUNCHES[(frag, grid)][0]
                out.append(f"| {frag} ({label}) | {nd} | " + " | ".join(cells) + " |")
            out.append("")
    derived = sorted({k[2] for k in pmc_all} - {"FETCH_SIZE", "WRITE_SIZE"})
    if derived:
        keys = sorted({(k[0], k[1]) for k in pmc_all if k[2] in derived})
        out.append("### Counters of every kernel (per dispatch, averaged; grid in threads)\n")
        out.append("| kernel | grid | dispatches | " + " | ".join(derived) + " |")
        out.append("|---|---|---|" + "---|" * len(derived))
        for name, grid in keys:
            cells = []
            for c in derived:
                v = pmc_all.get((name, grid, c))
                cells.append(f"{sum(v) / len(v):.2f}" if v else "-")
            nd = max(len(pmc_all.get((name, grid, c), [])) for c in derived)
            out.append(f"| {name} | {grid} | {nd} | " + " | ".join(cells) + " |")
        out.append("")
    return "\n".join(out), traffic


def _short_name(name: str) -> str:
    """A kernel's name without its parameter list, namespaces or `void `."""
    n = name.split("(")[0] if not name.startswith("(") else name
    for pre in ("void ", "mi355::", "(anonymous namespace)::", "tiled::"):
        n = n.replace(pre, "")
    return n[:110]


def main():
    args = parse_args()
    if args.rocprof_summary:
        text, traffic = rocprof_summary(args.rocprof_summary)
        print(text)
        if traffic:
            print("\n```json\n" + json.dumps(traffic, indent=1) + "\n```")
        return
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py: this build measures one GPU only (the fused RMSNorm/SwiGLU path is row-parallel "
              "and needs no cross-GPU exchange); run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    if args.e2e:
        bench_e2e(args)
        return
    if args.e2e_int8:
        bench_e2e_int8(args)
        return

    ctx = Ctx()
    torch = ctx.torch
    props = torch.cuda.get_device_properties(ctx.dev)
    log(f"device: {props.name} ({getattr(props, 'gcnArchName', '?')}), CUs={props.multi_processor_count}")

    F16 = torch.float16
    M, N, I = 2048, 1536, 8960
    rms_bytes = (2 * M * N + N) * 2
    silu_bytes = 3 * M * I * 2
    step_bytes = rms_bytes + silu_bytes
    nset = n_sets(step_bytes)

    w = rand(ctx, (N,), 1, F16, 1.0, 0.1)
    sets = []
    for s in range(nset):
        x = rand(ctx, (M, N), 100 + s, F16)
        gate = rand(ctx, (M, I), 200 + s, F16)
        up = rand(ctx, (M, I), 300 + s, F16)
        y = torch.empty_like(x)
        out = torch.empty_like(gate)
        sets.append((ctx.rms_call(x, w, y), ctx.silu_call(gate, up, out), (x, y, gate, up, out)))
    torch.cuda.synchronize()
    log(f"headline: {nset} buffer sets, footprint {nset * step_bytes / 2**30:.2f} GiB")
    # one untimed pass over every set: the generator's freshly written inputs
    # are written back from the caches to HBM here, not inside the timed region
    spin_up(ctx, [c for r, s_, _ in sets for c in (r, s_)], ms=5.0)

    if args.only:
        run_only(ctx, args, sets)
        return

    # ---- timed region: K steps, each RMSNorm C1 + SiLU-and-mul C2 on the next set
    for i in range(args.warmup):
        r, s_, _ = sets[i % nset]
        r()
        s_()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for i in range(args.steps):
        r, s_, _ = sets[i % nset]
        r()
        s_()
    end.record()
    torch.cuda.synchronize()
    elapsed_s = start.elapsed_time(end) / 1e3
    value = args.steps * step_bytes / elapsed_s / 1e9
    log(f"headline: {args.steps} steps in {elapsed_s * 1e3:.2f} ms -> {value:.1f} GB/s "
        f"({value / PEAK_GBS:.1%} of 8 TB/s)")

    # ---- per-kernel average launch durations (cold HBM, rotating sets)
    iters = max(200, args.steps)
    silu_us = time_loop(ctx, [s[1] for s in sets], iters)
    rms_us = time_loop(ctx, [s[0] for s in sets], iters)
    rms_graph_us = time_graph(ctx, [s[0] for s in sets], 200)
    silu_graph_us = time_graph(ctx, [s[1] for s in sets], 200)
    # the same launches through the product API (fused_rmsnorm: the C++
    # launcher extension, which also allocates the output) and an empty
    # kernel through the C ABI, eager back to back: the host's share of C1
    pkg = ctx.pkg
    rms_api_us = time_loop(ctx, [(lambda x=t[0]: pkg.fused_rmsnorm(x, w, 1e-6)) for _, _, t in sets], iters)
    empty_us = time_loop(ctx, [ctx.empty_call()], iters)
    silu_warm_us = time_loop(ctx, [sets[0][1]], iters)
    rms_warm_graph_us = time_graph(ctx, [sets[0][0]], 200)
    kernels = {
        "c2_silu_mul_f16_2048x8960": kernel_entry("silu_mul_chunks", silu_bytes, silu_us,
                                                  {"timing": "events over back-to-back launches, cold"}),
        "c1_rmsnorm_f16_2048x1536": kernel_entry("rmsnorm_wave_rows", rms_bytes, rms_us,
                                                 {"timing": "events over back-to-back launches, cold"}),
        "c1_rmsnorm_f16_2048x1536_graph": kernel_entry("rmsnorm_wave_rows", rms_bytes,
                                                       rms_graph_us, {"timing": "hipGraph of 200 launches, cold"}),
        "c2_silu_mul_f16_2048x8960_graph": kernel_entry("silu_mul_chunks", silu_bytes,
                                                        silu_graph_us, {"timing": "hipGraph of 200 launches, cold"}),
        "c1_rmsnorm_f16_2048x1536_api": kernel_entry("rmsnorm_wave_rows", rms_bytes, rms_api_us,
                                                     {"timing": "fused_rmsnorm (product API), events over "
                                                                "back-to-back calls, cold"}),
        "empty_kernel_eager_us": round(empty_us, 3),
        "c2_silu_mul_f16_2048x8960_warm": kernel_entry("silu_mul_chunks", silu_bytes, silu_warm_us,
                                                       {"timing": "same buffers every launch (MALL-warm)"}),
        "c1_rmsnorm_f16_2048x1536_warm_graph": kernel_entry("rmsnorm_wave_rows", rms_bytes, rms_warm_graph_us,
                                                            {"timing": "hipGraph, same buffers (MALL-warm)"}),
    }
    for k, v in kernels.items():
        if isinstance(v, dict):
            log(f"  {k}: {v['us']:.2f} us, {v['GBps']:.0f} GB/s ({v['frac_of_peak']:.1%})")

    result = {
        "metric": METRIC, "value": round(value, 2), "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(elapsed_s * 1e3 / args.steps, 5),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic (seeded N(0,1) gate/up/x, N(1,0.1) weight, fp16 storage)",
        "config": {"workload": "qwen2.5-1.5b-prefill-2048: RMSNorm x[2048,1536] + SiLU-and-mul gate/up[2048,8960]",
                   "storage_dtype": "f16", "math_dtype": "f32", "eps": 1e-6, "buffer_sets": nset,
                   "footprint_GiB": round(nset * step_bytes / 2**30, 3), "step_bytes": step_bytes},
        "roofline": {"bound": "hbm", "kernel": "silu_mul_chunks (C2 SiLU-and-mul [2048,8960] fp16)",
                     "achieved": round(silu_bytes / silu_us / 1e3, 1), "peak": PEAK_GBS, "unit": "GB/s",
                     "frac": round(silu_bytes / silu_us / 1e3 / PEAK_GBS, 4),
                     "traffic": read_traffic("C2 SiLU-and-mul [2048,8960] fp16"), "algorithmic_bytes": silu_bytes,
                     "avg_launch_us": round(silu_us, 3)},
    }
    full = {"kernels": kernels}

    if not args.skip_extras:
        del sets
        torch.cuda.empty_cache()
        full["add_rmsnorm"] = bench_add_rms(ctx, iters)
        full["c4"] = bench_c4(ctx, iters=60)
        full["decode"] = bench_decode(ctx)
        full["copy_ceiling"] = bench_copy(ctx)
        full["ceilings"] = bench_ceilings(ctx)
        full["gate_up_silu"] = bench_gate_up(ctx)
        full["gate_up_silu_prefill"] = bench_gate_up_prefill(ctx)
        full["w8a16"] = bench_w8a16(ctx)
        full["gate_up_silu_w8a16"] = bench_gate_up_w8(ctx)
        full["linear16_down"] = bench_linear16(ctx)
        full["stage3"] = bench_stage3_table(ctx)
        result["stage3_kernels"] = full["stage3"]
        result["w8a16_decode"] = w8a16_decode_block(full["w8a16"])
        if not args.skip_e2e:
            full["e2e"] = bench_e2e_compact(ctx)
            result["e2e_stage3"] = full["e2e"]
            full["e2e_int8"] = bench_e2e_int8_compact(ctx)
            result["e2e_stage7_int8"] = full["e2e_int8"]
        result["roofline"]["per_config"] = per_config(full)

    if not args.skip_cpu:
        log("cpu baseline ...")
        result["cpu_baseline"] = cpu_baseline(M, N, I, args.cpu_seconds)
        log(f"  cpu: {result['cpu_baseline']['value']} GB/s on {result['cpu_baseline']['cores']} threads")
    else:
        result["cpu_baseline"] = None
    if args.full_json:
        Path(args.full_json).parent.mkdir(parents=True, exist_ok=True)
        Path(args.full_json).write_text(json.dumps({**result, "full": full}, indent=1))
    log("full: " + json.dumps(full))
    print(json.dumps(result), flush=True)


def w8a16_decode_block(w8):
    """The W8A16 linear at decode rows (<= 32), compact: graph-node us, GB/s
    and fraction of 8 TB/s, and the speedup over fp16 hipBLASLt."""
    out = {}
    for key, e in w8.items():
        if e["M"] <= 32:
            out[key] = {"us": e["us"], "GBps": e["GBps"], "frac": e["frac_of_peak"],
                        "vs_fp16_matmul": e.get("speedup_vs_fp16_matmul")}
    return out


def per_config(full):
    """The compact per-config block of the stdout line: each BASELINE config's
    kernel time, rate and fraction of 8 TB/s (cold), the same-size probe's
    time, and the decode-row latencies (C3) -- a few hundred bytes the driver
    keeps whole inside `roofline`."""
    k, c4, dec, ceil = full["kernels"], full["c4"], full["decode"], full.get("ceilings") or {}

    def entry(d, rows, probe_label=None, graph=None):
        e = {"us": d["us"], "GBps": d["GBps"], "frac": d["frac_of_peak"], "rows_per_s": round(rows / d["us"] * 1e6)}
        if graph is not None:
            e["graph_us"] = graph["us"]
            e["graph_frac"] = graph["frac_of_peak"]
        if probe_label and probe_label in ceil:
            e["probe_us"] = ceil[probe_label]["us"]
        return e

    pc = {
        "C1_rmsnorm_f16_2048x1536": entry(k["c1_rmsnorm_f16_2048x1536"], 2048, "C1 RMSNorm [2048,1536] fp16",
                                          k["c1_rmsnorm_f16_2048x1536_graph"]),
        "C2_silu_mul_f16_2048x8960": entry(k["c2_silu_mul_f16_2048x8960"], 2048,
                                           "C2 SiLU-and-mul [2048,8960] fp16",
                                           k.get("c2_silu_mul_f16_2048x8960_graph")),
        "C4_rmsnorm_bf16_16384x3584": entry(c4["c4_rmsnorm_bf16_16384x3584"], 16384,
                                            "C4 RMSNorm [16384,3584] bf16"),
        "C4_silu_mul_bf16_16384x18944": entry(c4["c4_silu_mul_bf16_16384x18944"], 16384,
                                              "C4 SiLU-and-mul [16384,18944] bf16"),
    }
    if "c1_rmsnorm_f16_2048x1536_api" in k:
        pc["C1_rmsnorm_f16_2048x1536"]["api_us"] = k["c1_rmsnorm_f16_2048x1536_api"]["us"]
        pc["C1_rmsnorm_f16_2048x1536"]["empty_kernel_eager_us"] = k["empty_kernel_eager_us"]
    c3 = {}
    for m, d in dec.items():
        if not m.startswith("M="):
            continue
        rows = int(m[2:])
        c3["M" + m[2:]] = {"rms_api_us": d["rmsnorm_api_us"], "silu_api_us": d["silu_mul_api_us"],
                           "rms_call_us": d.get("rmsnorm_call_us"), "silu_call_us": d.get("silu_mul_call_us"),
                           "rms_dev_us": d["rmsnorm_device_us"], "silu_dev_us": d["silu_mul_device_us"],
                           "graph_node_us": d["graph_per_kernel_us"], "graph_28_layers_us": d["graph_replay_us"],
                           "rms_rows_per_s": round(rows / d["rmsnorm_device_us"] * 1e6),
                           "silu_rows_per_s": round(rows / d["silu_mul_device_us"] * 1e6)}
    pc["C3_decode_f16_latency"] = c3
    if "floor" in dec:
        pc["C3_floor"] = {"empty_graph_node_us": dec["floor"]["empty_kernel_graph_node_us"],
                          "row_copy_graph_node_us": dec["floor"]["row_copy_graph_node_us"]}
    if full.get("copy_ceiling"):
        pc["copy_1GiB_frac"] = full["copy_ceiling"]["frac_of_peak"]
    return pc


def run_only(ctx, args, sets):
    """One kernel loop only, so a profiler run sees exactly one kernel name."""
    torch = ctx.torch
    iters = max(200, args.steps)
    if args.only == "c2-silu":
        us = time_loop(ctx, [s[1] for s in sets], iters)
        log(f"c2-silu avg {us:.3f} us")
    elif args.only == "c1-rms":
        us = time_loop(ctx, [s[0] for s in sets], iters)
        log(f"c1-rms avg {us:.3f} us")
    elif args.only == "c1-add-rms":
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_add_rms(ctx, iters)))
    elif args.only in ("c4-silu", "c4-rms"):
        del sets
        torch.cuda.empty_cache()
        d = bench_c4(ctx, iters=60, which=args.only)
        log(json.dumps(d))
    elif args.only == "c1-decomp":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"c1_decomposition": c1_decomposition(ctx)}), flush=True)
    elif args.only == "copy":
        log(json.dumps(bench_copy(ctx)))
    elif args.only == "decode":
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_decode(ctx)))
    elif args.only == "ceilings":
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_ceilings(ctx)))
    elif args.only == "gate-up":
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up(ctx, shapes=GATE_UP_SHAPES[1:2], iters=iters, baselines=False)))
    elif args.only == "gate-up-w8":
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up_w8(ctx)))
    elif args.only == "gate-up-w8-prefill":  # prefill rows of the 1.5B and 7B MLPs, kernel only
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up_w8(ctx, shapes=GATE_UP_W8_PREFILL_SHAPES, iters=100, baselines=False)))
    elif args.only == "gate-up-w8-decode":  # the two 8-row shapes profiled under profiles/, no baseline
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up_w8(ctx, shapes=[s for s in GATE_UP_W8_SHAPES if s[0] == 8], iters=iters,
                                        baselines=False)))
    elif args.only == "linear16-table":  # every decode row count of the down projection, with torch's linear
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"linear16_down": bench_linear16(ctx)}), flush=True)
    elif args.only == "linear16":  # kernel only, the 1.5B down projection at 8 rows and the 7B one at 8 rows
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_linear16(ctx, shapes=[s for s in LINEAR16_SHAPES if s[0] == 8], iters=iters,
                                      baselines=False)))
    elif args.only == "gate-up-prefill":  # kernel only, the 1.5B MLP at 1024 and 4096 rows
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up_prefill(ctx, shapes=GATE_UP_PREFILL_SHAPES[1:3], baselines=False)))
    elif args.only == "gate-up-prefill-sweep":  # every prefill row count of the MLP table, with the unfused chain
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_gate_up_prefill(ctx, shapes=GATE_UP_PREFILL_SWEEP_SHAPES)))
    elif args.only in ("w8a16-prefill-wide", "w8a16-prefill-narrow", "w8a16-prefill-ragged"):  # kernel only
        del sets
        torch.cuda.empty_cache()
        shapes = {"wide": W8A16_WIDE_PREFILL_SHAPES, "narrow": W8A16_NARROW_PREFILL_SHAPES,
                  "ragged": W8A16_RAGGED_PREFILL_SHAPES}[args.only.rsplit("-", 1)[1]]
        # (the ragged row counts also time fp16 hipBLASLt on the same shapes)
        log(json.dumps(bench_w8a16(ctx, shapes=shapes, iters=100, baselines=args.only.endswith("ragged"))))
    elif args.only in ("w8a16", "w8a16-decode", "w8a16-prefill", "w8a16-prefill-1.5b"):
        del sets
        torch.cuda.empty_cache()
        if args.only == "w8a16":
            log(json.dumps(bench_w8a16(ctx)))
        elif args.only == "w8a16-prefill-1.5b":  # the 1.5B gate/up and down projections at 1024 and 4096 rows,
            # each against fp16 hipBLASLt on the same shape
            log(json.dumps(bench_w8a16(ctx, shapes=[s for s in W8A16_SHAPES if s[0] in (1024, 4096)
                                                    and s[3] == "f16" and s[4] in ("gate/up proj", "down proj")])))
        elif args.only == "w8a16-prefill":  # kernel only, the 1.5B gate/up and down projections at 1024 rows
            log(json.dumps(bench_w8a16(ctx, shapes=[s for s in W8A16_SHAPES if s[0] == 1024 and s[2] in (8960, 1536)
                                                    and s[1] in (1536, 8960)][-2:], iters=iters, baselines=False)))
        else:  # the 8-row gate/up and down projections of 1.5B and 7B, kernel only
            log(json.dumps(bench_w8a16(ctx, shapes=[s for s in W8A16_SHAPES if s[0] == 8 and s[4] in
                                                    ("gate/up proj", "down proj", "7b gate/up proj", "7b down proj")],
                                       iters=iters, baselines=False)))
    elif args.only == "decode-wide-rows":  # kernels only: down projections at 32 - 64 rows (for PMC runs)
        del sets
        torch.cuda.empty_cache()
        log(json.dumps(bench_w8a16(ctx, shapes=[(32, 8960, 1536, "f16", "down proj"),
                                                (48, 18944, 3584, "bf16", "7b down proj")],
                                   iters=iters, baselines=False)))
        log(json.dumps(bench_linear16(ctx, shapes=[(32, 8960, 1536, "f16", "qwen2.5-1.5b down"),
                                                   (64, 18944, 3584, "bf16", "qwen2.5-7b down")],
                                      iters=iters, baselines=False)))
    elif args.only == "prefill-core":
        print(json.dumps(bench_prefill_core(ctx)), flush=True)
    elif args.only == "stage3":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"stage3_kernels": bench_stage3_table(ctx)}), flush=True)
    elif args.only == "e2e-compact":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"e2e_stage3": bench_e2e_compact(ctx)}), flush=True)
    elif args.only == "e2e-int8-compact":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"e2e_stage7_int8": bench_e2e_int8_compact(ctx)}), flush=True)
    elif args.only == "gu16-stream-sweep":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"gate_up16_stream_sweep": gu16_stream_sweep(ctx)}), flush=True)
    elif args.only == "tile-plans":  # the plans' predicted times against measured ones
        del sets
        torch.cuda.empty_cache()
        print(tile_plan_table(ctx), flush=True)
    elif args.only == "stream-sweep32":  # 17 - 32 rows: all three forms of the decode kernel
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP32_SHAPES, True),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP32_SHAPES),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP32_SHAPES, True)}), flush=True)
    elif args.only == "stream-sweep64":  # 33 - 64 rows of the narrow projections
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP64_SHAPES, True),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP64_SHAPES)}), flush=True)
    elif args.only == "l16-stream-sweep":  # the 16-bit linear on the weight-streaming kernel
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"linear16_stream_sweep": l16_stream_sweep(ctx)}), flush=True)
    elif args.only == "stream-sweep16-k":  # 9 - 16 rows, k < 3072, with 16-row workgroups too
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP16_K_SHAPES, True),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP16_K_SHAPES, True)}),
              flush=True)
    elif args.only == "stream-sweep-dualn":  # the dual kernels by workgroups per CU
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_DUALN_SHAPES, True),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_DUALN_SHAPES, True)}),
              flush=True)
    elif args.only == "stream-sweep-dual32":  # 17 - 32 rows of the gate/up kernels vs the small tiles
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_DUAL32_SHAPES, True),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_DUAL32_SHAPES, True)}),
              flush=True)
    elif args.only == "stream-sweep-3b14b":  # the 3B and 14B shapes
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_3B14B_SHAPES, True),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP_3B14B_SHAPES),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_3B14B_SHAPES, True)}),
              flush=True)
    elif args.only == "stream-sweep-bal":  # rows per workgroup that balance the CUs
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_BAL_SHAPES, True,
                                                                rpws=STREAM_BAL_RPWS),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP_BAL_SHAPES, rpws=STREAM_BAL_RPWS),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_BAL_SHAPES, True,
                                                                      rpws=STREAM_BAL_RPWS)}), flush=True)
    elif args.only == "stream-sweep-few16":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_FEW16_SHAPES, True,
                                                                rpws=(8, 12, 14, 15, 16))}), flush=True)
    elif args.only == "stream-sweep-dual4":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_DUAL4_SHAPES, True,
                                                                rpws=(4, 8, 12, 14, 16)),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_DUAL4_SHAPES, True,
                                                                      rpws=(4, 8, 12, 14, 15, 16))}), flush=True)
    elif args.only == "stream-sweep-14b-wide":
        del sets
        torch.cuda.empty_cache()
        rp = (4, 6, 8, 10, 12, 14, 16)
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_14B_WIDE_SHAPES, True, rpws=rp),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP_14B_WIDE_SHAPES, rpws=rp),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_14B_WIDE_SHAPES, True,
                                                                      rpws=rp)}), flush=True)
    elif args.only == "stream-sweep-smallm":  # the 3B and 14B shapes at 1 - 4 rows
        del sets
        torch.cuda.empty_cache()
        rp = (4, 6, 8, 10, 12, 14, 16)
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_SMALLM_SHAPES, True, rpws=rp),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP_SMALLM_SHAPES, rpws=rp),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_SMALLM_SHAPES, True,
                                                                      rpws=rp)}), flush=True)
    elif args.only == "stream-sweep-m4":  # 1 - 4 rows on the deep projections that are not narrow
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_M4_SHAPES, rpws=(8, 12, 16)),
                          "linear16_stream_sweep": l16_stream_sweep(ctx, L16_SWEEP_M4_SHAPES),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_M4_SHAPES)}), flush=True)
    elif args.only == "stream-sweep-r8":  # wide outputs with 17 - 32 weight rows per workgroup too
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP_R8_SHAPES, rpws=STREAM_R8_RPWS),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP_R8_SHAPES,
                                                                      rpws=STREAM_R8_RPWS)}), flush=True)
    elif args.only == "stream-sweep16-wide":  # 12 / 16 rows with 16-row workgroups too
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP16_WIDE_SHAPES, True),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP16_WIDE_SHAPES, True)}),
              flush=True)
    elif args.only == "stream-sweep16":  # 9 - 16 rows: both decode sweeps
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx, W8_STREAM_SWEEP16_SHAPES),
                          "gate_up16_stream_sweep": gu16_stream_sweep(ctx, GU16_SWEEP16_SHAPES)}), flush=True)
    elif args.only == "w8-stream-sweep":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_stream_sweep": w8_stream_sweep(ctx)}), flush=True)
    elif args.only == "w8-layouts8":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8_stream_layouts8": w8_layout8_sweep(ctx)}), flush=True)
    elif args.only == "w8-layouts":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8_stream_layouts": w8_layout_sweep(ctx)}), flush=True)
    elif args.only == "w8-decomp":
        del sets
        torch.cuda.empty_cache()
        print(json.dumps({"w8a16_decode_decomposition": w8_decode_decomposition(ctx)}), flush=True)


def c1_decomposition(ctx):
    """Where C1's time goes, from the floor up (cold buffers unless noted):
    an empty kernel and the copy of one 3 KiB row (one HBM round trip), back
    to back and as nodes of a hipGraph; a one-row RMSNorm; the probe copy of
    C1's own bytes; the C1 kernel back to back, in a graph, and MALL-warm in a
    graph."""
    torch = ctx.torch
    F16 = torch.float16
    M, N = 2048, 1536
    nbytes = (2 * M * N + N) * 2
    out = {"bytes": nbytes}
    empty = [ctx.empty_call()]
    src = torch.empty(N * 2, dtype=torch.uint8, device=ctx.dev)
    dst = torch.empty_like(src)
    row = [ctx.copy_call(src, dst)]
    out["empty_kernel_eager_us"] = time_loop(ctx, empty, 2000)
    out["empty_kernel_graph_node_us"] = time_graph(ctx, empty, 200, replays=20)
    out["row_copy_eager_us"] = time_loop(ctx, row, 2000)
    out["row_copy_graph_node_us"] = time_graph(ctx, row, 200, replays=20)
    w = rand(ctx, (N,), 1, F16, 1.0, 0.1)
    x1 = rand(ctx, (1, N), 5, F16)
    y1 = torch.empty_like(x1)
    one = [ctx.rms_call(x1, w, y1)]
    out["one_row_rmsnorm_eager_us"] = time_loop(ctx, one, 2000)
    out["one_row_rmsnorm_graph_node_us"] = time_graph(ctx, one, 200, replays=20)
    half = M * N * 2
    bufs = [(torch.empty(half, dtype=torch.uint8, device=ctx.dev).random_(0, 255),
             torch.empty(half, dtype=torch.uint8, device=ctx.dev)) for _ in range(n_sets(2 * half))]
    copies = [ctx.copy_call(a, b) for a, b in bufs]
    spin_up(ctx, copies)
    out["same_size_copy_eager_us"] = time_loop(ctx, copies, 2000)
    out["same_size_copy_graph_us"] = time_graph(ctx, copies, 200, replays=20)
    del bufs, copies
    sets = []
    for s_ in range(n_sets(nbytes)):
        x = rand(ctx, (M, N), 100 + s_, F16)
        sets.append((x, torch.empty_like(x)))
    rms = [ctx.rms_call(x, w, y) for x, y in sets]
    spin_up(ctx, rms)
    out["c1_eager_us"] = time_loop(ctx, rms, 2000)
    out["c1_graph_us"] = time_graph(ctx, rms, 200, replays=20)
    out["c1_warm_graph_us"] = time_graph(ctx, rms[:1], 200, replays=20)
    for k in list(out):
        if k.endswith("_us"):
            out[k] = round(out[k], 3)
    out["c1_graph_frac"] = round(nbytes / out["c1_graph_us"] / 1e3 / PEAK_GBS, 4)
    out["c1_eager_frac"] = round(nbytes / out["c1_eager_us"] / 1e3 / PEAK_GBS, 4)
    out["us_for_80pct"] = round(nbytes / (0.8 * PEAK_GBS) / 1e3, 3)
    del sets, rms
    torch.cuda.empty_cache()
    return out


STAGE3_ROWS = (64, 256, 1024, 8192, 32768)


def _time_per_call(torch, fn, trials=20, warmup=5):
    """Mean device time of one call including its launch, timed as the
    reference's benchmarks/run_stage3_kernels.py:34-49 times it: synchronize,
    record an event, call, record, synchronize, per trial."""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    ts = []
    for _ in range(trials):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record()
        fn()
        b.record()
        torch.cuda.synchronize()
        ts.append(a.elapsed_time(b))
    return statistics.mean(ts) * 1e3  # us


def bench_stage3_table(ctx, rows=STAGE3_ROWS, hidden=1536, inter=8960, trials=20):
    """The reference's Stage 3 kernel table (benchmarks/run_stage3_kernels.py:
    52-121, results in benchmarks/results/stage3_kernels.json:4-93) on this
    device: for each row count, the package's naive path (the unfused torch
    ops of naive_rmsnorm_reference / naive_silu_mul_reference) against the
    fused HIP kernel through the package's drop-in API (fused_rmsnorm /
    fused_silu_mul: the C++ launcher allocates the output and launches), fp16,
    per call including the launch, the same buffers every call (as the
    reference), mean of `trials`.  `cold_us` is the fused kernel's device time
    alone (C ABI, hipGraph nodes over buffer sets rotating over up to 1 GiB,
    at most 512 sets).  GB/s and rows/s are from the per-call time; the
    algorithmic bytes are RMSNorm (2 M N + N) * 2, SiLU-and-mul 3 M I * 2."""
    torch = ctx.torch
    pkg = ctx.pkg
    F16 = torch.float16
    out = {"rmsnorm_N1536": {}, "silu_mul_I8960": {}}
    for M in rows:
        x = rand(ctx, (M, hidden), 0, F16)
        w = rand(ctx, (hidden,), 1, F16)
        naive = _time_per_call(torch, lambda: pkg.naive_rmsnorm_reference(x, w), trials)
        fused = _time_per_call(torch, lambda: pkg.fused_rmsnorm(x, w), trials)
        nbytes = (2 * M * hidden + hidden) * 2
        sets = min(512, n_sets(nbytes))
        bufs = [(rand(ctx, (M, hidden), 10 + i, F16), torch.empty((M, hidden), dtype=F16, device=ctx.dev))
                for i in range(sets)]
        calls = [ctx.rms_call(a, w, b) for a, b in bufs]
        spin_up(ctx, calls, ms=5.0)
        cold = time_graph(ctx, calls, max(sets, 64))
        del bufs, calls
        out["rmsnorm_N1536"][str(M)] = {
            "naive_us": round(naive, 2), "fused_us": round(fused, 2), "speedup": round(naive / fused, 2),
            "GBps": round(nbytes / fused / 1e3, 1), "rows_per_s": round(M / fused * 1e6),
            "cold_us": round(cold, 2), "cold_GBps": round(nbytes / cold / 1e3, 1)}
        del x
        gate = rand(ctx, (M, inter), 2, F16)
        up = rand(ctx, (M, inter), 3, F16)
        naive = _time_per_call(torch, lambda: pkg.naive_silu_mul_reference(gate, up), trials)
        fused = _time_per_call(torch, lambda: pkg.fused_silu_mul(gate, up), trials)
        nbytes = 3 * M * inter * 2
        sets = min(512, n_sets(nbytes))
        bufs = [(rand(ctx, (M, inter), 20 + i, F16), rand(ctx, (M, inter), 30 + i, F16),
                 torch.empty((M, inter), dtype=F16, device=ctx.dev)) for i in range(sets)]
        calls = [ctx.silu_call(g_, u_, o_) for g_, u_, o_ in bufs]
        spin_up(ctx, calls, ms=5.0)
        cold = time_graph(ctx, calls, max(sets, 64))
        del bufs, calls, gate, up
        torch.cuda.empty_cache()
        out["silu_mul_I8960"][str(M)] = {
            "naive_us": round(naive, 2), "fused_us": round(fused, 2), "speedup": round(naive / fused, 2),
            "GBps": round(nbytes / fused / 1e3, 1), "rows_per_s": round(M / fused * 1e6),
            "cold_us": round(cold, 2), "cold_GBps": round(nbytes / cold / 1e3, 1)}
        log(f"  stage3 M={M}: rmsnorm {json.dumps(out['rmsnorm_N1536'][str(M)])}; "
            f"silu_mul {json.dumps(out['silu_mul_I8960'][str(M)])}")
    return out


# The decomposed decode shapes: (label, rows, k, n) of the Qwen2.5-1.5B down
# and gate/up projections.
W8_DECOMP_SHAPES = [("down_M1", 1, 8960, 1536), ("down_M8", 8, 8960, 1536),
                    ("gateup_M1", 1, 1536, 8960), ("gateup_M8", 8, 1536, 8960),
                    ("7b_down_M8", 8, 18944, 3584), ("7b_gateup_M8", 8, 3584, 18944)]


def w8_decode_decomposition(ctx):
    """Where the W8A16 decode kernel's time goes, at the Qwen2.5-1.5B down
    (k 8960, n 1536) and gate/up (k 1536, n 8960) projections with 1 and 8
    rows of fp16 x and the Qwen2.5-7B ones (k 18944, n 3584; k 3584, n 18944)
    with 8 rows, every figure a hipGraph node over cold weights (sets
    rotating over >= 1 GiB): an empty kernel; the read floor (the weights'
    bytes read by the copy probe's shape) and a copy moving the same bytes;
    the kernel's own loads alone at its launch plan (csrc/probe/
    w8_stream_plan.hip: the same descriptors, offsets and chunk split, no
    MFMA, reduction or epilogue), the weights only and the weights with x;
    and the kernel itself (through the C ABI)."""
    torch = ctx.torch
    F16 = torch.float16
    cus = torch.cuda.get_device_properties(ctx.dev).multi_processor_count
    out = {"empty_graph_node_us": round(time_graph(ctx, [ctx.empty_call()], 200, replays=20), 3)}
    sink = torch.zeros(1024, dtype=torch.int32, device=ctx.dev)
    for label, M, K, N in W8_DECOMP_SHAPES:
        wbytes = N * K
        sets = n_sets(wbytes)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(2100 + K)
        qs = [torch.randint(-127, 128, (N, K), generator=g, device=ctx.dev, dtype=torch.int8) for _ in range(sets)]
        scales = [(torch.rand(N, generator=g, device=ctx.dev) * 1e-3 + 1e-4) for _ in range(sets)]
        x = rand(ctx, (M, K), 2200 + M, F16)
        o = torch.empty((M, N), dtype=F16, device=ctx.dev)
        nodes = max(2 * sets, 64)

        def graph_us(calls):
            spin_up(ctx, calls, ms=5.0)
            return round(time_graph(ctx, calls, nodes, replays=5), 3)

        rpw, r4, waves, u = ctx.w8_stream_plan(M, K, N, False, cus)
        d = {"M": M, "K": K, "N": N, "weight_bytes": wbytes, "weight_sets": sets,
             "plan": {"rows_per_wg": rpw, "waves": waves, "chunks_in_flight": u, "workgroups": -(-N // rpw)}}
        d["read_floor_us"] = graph_us([ctx.read_call(q, sink) for q in qs])
        half = wbytes // 2 // 16 * 16
        cbufs = [(q.view(-1)[:half], q.view(-1)[half:2 * half]) for q in qs]
        d["same_size_copy_us"] = graph_us([ctx.copy_call(a, b) for a, b in cbufs])
        del cbufs
        d["weight_loads_us"] = graph_us([ctx.w8_stream_loads_call(x, q, sink, rpw, r4, waves, u, False) for q in qs])
        d["weight_and_x_loads_us"] = graph_us([ctx.w8_stream_loads_call(x, q, sink, rpw, r4, waves, u, True)
                                               for q in qs])
        d["kernel_us"] = graph_us([ctx.w8a16_call(x, q, sc, o) for q, sc in zip(qs, scales)])
        d["read_floor_GBps"] = round(wbytes / d["read_floor_us"] / 1e3, 1)
        d["kernel_GBps"] = round((wbytes + 4 * N + 2 * M * (K + N)) / d["kernel_us"] / 1e3, 1)
        d["kernel_over_weight_loads"] = round(d["kernel_us"] / d["weight_loads_us"], 3)
        d["kernel_over_read_floor"] = round(d["kernel_us"] / d["read_floor_us"], 3)
        out[label] = d
        log(f"  w8 decomp {label}: " + json.dumps(d))
        del qs, scales
        torch.cuda.empty_cache()
    return out


# Load-layout sampling of the weight-stream probe at 8 rows of x: launch
# shapes (rpw, waves, G, U) per projection, crossed with the weight lane
# layouts WL, the x lane layouts XL (0 = no x) and the per-workgroup stagger.
W8_LAYOUT_SHAPES = {
    1536: [(6, 16, 1, 8), (8, 16, 1, 8)],
    8960: [(8, 3, 1, 4), (16, 3, 2, 4), (32, 6, 4, 2)],
}


def w8_layout_sweep(ctx):
    """The weight-stream probe (csrc/probe/w8_stream.hip) at the Qwen2.5-1.5B
    down and gate/up projections with 8 rows of fp16 x, over its weight and x
    lane layouts and the stagger: graph-node us, cold weights."""
    torch = ctx.torch
    sink = torch.zeros(1024, dtype=torch.int32, device=ctx.dev)
    out = {}
    for label, K, N in (("down", 8960, 1536), ("gateup", 1536, 8960)):
        sets = n_sets(N * K)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(2300 + K)
        qs = [torch.randint(-127, 128, (N, K), generator=g, device=ctx.dev, dtype=torch.int8) for _ in range(sets)]
        x = rand(ctx, (8, K), 2400, torch.float16)
        nodes = max(2 * sets, 64)
        res = {}
        for rpw, wv, gg, uu in W8_LAYOUT_SHAPES[N]:
            for wl in (0, 2, 3):
                for xl in (0, 1, 2, 3):
                    for st in (0, 1):
                        calls = [ctx.w8_stream_call(q, sink, rpw, wv, gg, uu, layout=wl, x=x if xl else None,
                                                    xl=xl or 1, stagger=st) for q in qs]
                        spin_up(ctx, calls, ms=3.0)
                        res[f"rpw{rpw}_w{wv}_G{gg}_U{uu}_WL{wl}_XL{xl}_S{st}"] = round(
                            time_graph(ctx, calls, nodes, replays=5), 3)
        out[label] = res
        log(f"  w8 layouts {label}: {json.dumps(res)}")
        del qs
        torch.cuda.empty_cache()
    return out


# The weight-stream probe at the decode kernel's 8-row launch plans (rpw,
# waves, G 8-row groups, U blocks in flight: one 256-byte chunk of each 4-row
# set): its lane layout (WL 3 with the kernel's x loads, XL 5) against 8 rows x
# 128 bytes with pairs of lanes on 32 bytes (WL 4, x to match: XL 4)
W8_LAYOUT8_SHAPES = [("down", 8960, 1536, (6, 12, 1, 2)), ("gateup", 1536, 8960, (8, 2, 1, 2)),
                     ("down7b", 18944, 3584, (16, 8, 2, 2)), ("gateup7b", 3584, 18944, (16, 2, 2, 2))]


def w8_layout8_sweep(ctx):
    """WL 3 / XL 5 (the decode kernel's loads) against WL 4 / XL 4 in the
    weight-stream probe (csrc/probe/w8_stream.hip), weights alone and with 8
    rows of fp16 x, at the kernel's 8-row launch plans: graph-node us, cold
    weights."""
    torch = ctx.torch
    sink = torch.zeros(1024, dtype=torch.int32, device=ctx.dev)
    out = {}
    for label, K, N, (rpw, wv, gg, uu) in W8_LAYOUT8_SHAPES:
        sets = n_sets(N * K)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(2700 + K)
        qs = [torch.randint(-127, 128, (N, K), generator=g, device=ctx.dev, dtype=torch.int8) for _ in range(sets)]
        x = rand(ctx, (8, K), 2800, torch.float16)
        nodes = max(2 * sets, 64)
        res = {}
        for wl, xl in ((3, 0), (4, 0), (3, 5), (4, 4)):
            calls = [ctx.w8_stream_call(q, sink, rpw, wv, gg, uu, layout=wl, x=x if xl else None, xl=xl or 1)
                     for q in qs]
            spin_up(ctx, calls, ms=3.0)
            res[f"WL{wl}_XL{xl}"] = round(time_graph(ctx, calls, nodes, replays=5), 3)
        out[label] = res
        log(f"  w8 layouts (8 rows) {label} rpw{rpw} w{wv} G{gg} U{uu}: {json.dumps(res)}")
        del qs
        torch.cuda.empty_cache()
    return out


def stream_max_waves(r4, mt4, u, dual, wb=1):
    """Most waves per workgroup of the decode stream kernel's instantiation
    (stream_max_threads of csrc/w8a16_stream.h / 64): 16, or 8 where its
    estimated live registers (stream_regs) reach 112, 0 above 224."""
    nq = 2 if dual else 1
    est = 4 * nq * r4 * mt4 + u * (4 * nq * r4 + (8 if wb == 1 else 4) * mt4) + r4 + mt4
    return 0 if est > 224 else (8 if est >= 112 else 16)


def stream_x_sets(rows):
    """4-row x sets of the decode stream kernel (stream_x_sets of
    csrc/w8a16_stream.h): ceil(rows / 4) up to 16 rows, then 6, 8, 12 or 16."""
    if rows <= 16:
        return -(-rows // 4)
    return 6 if rows <= 24 else (8 if rows <= 32 else (12 if rows <= 48 else 16))


def _w8_stream_shapes(nchunk, dual, mt4, wide16=False, wb=1, rpws=(4, 6, 8, 12, 16)):
    """Launch shapes (rpw, r4, waves, u) of the W8A16 decode kernel sampled by
    w8_stream_sweep: rows per workgroup `rpws` (4-16 by default; 17-32 take
    eight 4-row weight sets, up to 8 rows of x), 1-16 waves (at most
    stream_max_waves), 1 or 2 chunks in flight; 16-row workgroups with more
    than 8 rows of x only when `wide16`."""
    out = []
    for rpw in rpws:
        r4 = 1 if rpw <= 4 else (2 if rpw <= 8 else (4 if rpw <= 16 else 8))
        if r4 == 8 and mt4 > 2:
            continue
        if mt4 > 2 and r4 == 4 and not wide16:
            continue
        for waves in (1, 2, 3, 4, 6, 8, 12, 16):
            if waves > nchunk:
                continue
            per_wave = -(-nchunk // waves)
            for u in (1, 2):
                if u > 1 and (u > per_wave or mt4 > 2):
                    continue
                if waves > stream_max_waves(r4, mt4, u, dual, wb):
                    continue
                out.append((rpw, r4, waves, u))
    return out


# (label, rows, k, n, dual) of the decode sweep: the Qwen2.5-1.5B projections
# and MLP, then the 7B, 0.5B and small 1.5B projections.
W8_STREAM_SWEEP_SHAPES = [
    ("down_M1", 1, 8960, 1536, False), ("down_M8", 8, 8960, 1536, False),
    ("gateup_M1", 1, 1536, 8960, False), ("gateup_M8", 8, 1536, 8960, False),
    ("dual_gateup_M1", 1, 1536, 8960, True), ("dual_gateup_M8", 8, 1536, 8960, True),
    ("down7b_M1", 1, 18944, 3584, False), ("down7b_M8", 8, 18944, 3584, False),
    ("gateup7b_M1", 1, 3584, 18944, False), ("gateup7b_M8", 8, 3584, 18944, False),
    ("o7b_M8", 8, 3584, 3584, False), ("down0.5b_M8", 8, 4864, 896, False),
    ("o1.5b_M8", 8, 1536, 1536, False), ("kv1.5b_M8", 8, 1536, 256, False), ("o1.5b_M4", 4, 1536, 1536, False),
    ("dual7b_M1", 1, 3584, 18944, True), ("dual7b_M8", 8, 3584, 18944, True), ("dual0.5b_M8", 8, 896, 4864, True),
]


# 9 - 16 rows of x (four 4-row x sets at most): the Qwen2.5-0.5B, 1.5B and 7B
# projections and MLPs at 12 and 16 rows
# the wide, deep 7B gate/up projection at 12 and 16 rows, with 12- and
# 16-row workgroups too (the single kernel: a few registers spill at 16 rows)
W8_STREAM_SWEEP16_WIDE_SHAPES = [("gateup7b_M9", 9, 3584, 18944, False), ("gateup7b_M12", 12, 3584, 18944, False),
                                 ("gateup7b_M16", 16, 3584, 18944, False), ("down7b_M12", 12, 18944, 3584, False),
                                 ("down7b_M16", 16, 18944, 3584, False), ("down_M16", 16, 8960, 1536, False),
                                 ("dual7b_M8", 8, 3584, 18944, True), ("dual7b_M12", 12, 3584, 18944, True),
                                 ("dual7b_M16", 16, 3584, 18944, True), ("dual_gateup_M16", 16, 1536, 8960, True)]
# 17 - 32 rows (6 and 8 x sets): the Qwen2.5-1.5B and 7B projections and MLPs
W8_STREAM_SWEEP32_SHAPES = [("down_M24", 24, 8960, 1536, False), ("down_M32", 32, 8960, 1536, False),
                            ("gateup_M32", 32, 1536, 8960, False), ("o1.5b_M32", 32, 1536, 1536, False),
                            ("down7b_M32", 32, 18944, 3584, False), ("gateup7b_M32", 32, 3584, 18944, False),
                            ("dual_gateup_M32", 32, 1536, 8960, True), ("dual7b_M32", 32, 3584, 18944, True),
                            ("gateup0.5b_M32", 32, 896, 4864, False), ("down0.5b_M32", 32, 4864, 896, False),
                            ("dual0.5b_M32", 32, 896, 4864, True), ("o7b_M32", 32, 3584, 3584, False),
                            ("down_M20", 20, 8960, 1536, False)]
# 33 - 64 rows (12 and 16 x sets) of the narrow projections
W8_STREAM_SWEEP64_SHAPES = [("down_M48", 48, 8960, 1536, False), ("down_M64", 64, 8960, 1536, False),
                            ("down7b_M64", 64, 18944, 3584, False), ("o1.5b_M64", 64, 1536, 1536, False),
                            ("down0.5b_M64", 64, 4864, 896, False), ("down7b_M48", 48, 18944, 3584, False),
                            ("o7b_M48", 48, 3584, 3584, False), ("down_M40", 40, 8960, 1536, False),
                            ("down0.5b_M48", 48, 4864, 896, False), ("dual0.5b_M48", 48, 896, 4864, True)]
L16_SWEEP64_SHAPES = [("down1.5b_M64", 64, 8960, 1536), ("down7b_M48", 48, 18944, 3584),
                      ("down7b_M64", 64, 18944, 3584), ("o7b_M64", 64, 3584, 3584), ("down1.5b_M48", 48, 8960, 1536),
                      ("down0.5b_M64", 64, 4864, 896), ("o1.5b_M64", 64, 1536, 1536)]
GU16_SWEEP32_SHAPES = [("gu1.5b_M32", 32, 1536, 8960), ("gu7b_M32", 32, 3584, 18944), ("gu0.5b_M32", 32, 896, 4864)]
L16_SWEEP32_SHAPES = [("down1.5b_M24", 24, 8960, 1536), ("down1.5b_M32", 32, 8960, 1536),
                      ("down7b_M32", 32, 18944, 3584), ("down0.5b_M32", 32, 4864, 896), ("o7b_M32", 32, 3584, 3584)]
# wide outputs at up to 8 rows of x with 17 - 32 weight rows per workgroup
# (eight 4-row weight sets) beside 12 - 16: fewer workgroups re-read x
STREAM_R8_RPWS = (8, 12, 14, 16, 20, 24, 28, 32)
W8_STREAM_SWEEP_R8_SHAPES = [("gateup_M4", 4, 1536, 8960, False), ("gateup_M8", 8, 1536, 8960, False),
                             ("gateup7b_M1", 1, 3584, 18944, False), ("gateup7b_M4", 4, 3584, 18944, False),
                             ("gateup7b_M8", 8, 3584, 18944, False), ("down7b_M8", 8, 18944, 3584, False),
                             ("o7b_M8", 8, 3584, 3584, False), ("dual_gateup_M8", 8, 1536, 8960, True),
                             ("dual7b_M4", 4, 3584, 18944, True), ("dual7b_M8", 8, 3584, 18944, True)]
# 9 - 16 rows on the shallower wide projections (k < 3072), with 16-row
# workgroups too: each 8-row workgroup re-reads x worth 2 - 4 times its weights
W8_STREAM_SWEEP16_K_SHAPES = [("gateup_M12", 12, 1536, 8960, False), ("gateup_M16", 16, 1536, 8960, False),
                              ("gateup0.5b_M16", 16, 896, 4864, False), ("gateup_M10", 10, 1536, 8960, False),
                              ("dual_gateup_M12", 12, 1536, 8960, True), ("dual0.5b_M16", 16, 896, 4864, True)]
GU16_SWEEP16_K_SHAPES = [("gu1.5b_M12", 12, 1536, 8960), ("gu0.5b_M16", 16, 896, 4864)]
# the dual kernels where 8-row workgroups number few per CU (0.5B MLP: 608)
# against more (1.5B: 1120, 3B: 1376), 5 - 32 rows
W8_STREAM_SWEEP_DUALN_SHAPES = [("dual0.5b_M6", 6, 896, 4864, True), ("dual0.5b_M12", 12, 896, 4864, True),
                                ("dual0.5b_M24", 24, 896, 4864, True), ("dual3b_M8", 8, 2048, 11008, True),
                                ("dual3b_M16", 16, 2048, 11008, True), ("dual_gateup_M16", 16, 1536, 8960, True),
                                ("dual_gateup_M24", 24, 1536, 8960, True)]
GU16_SWEEP_DUALN_SHAPES = [("gu0.5b_M10", 10, 896, 4864), ("gu0.5b_M12", 12, 896, 4864),
                           ("gu3b_M16", 16, 2048, 11008), ("gu0.5b_M24", 24, 896, 4864)]
# 17 - 32 rows of the gate/up + SiLU-and-mul kernels on the MLPs where the
# launchers take the small tiled shapes (>= 128 tile columns)
W8_STREAM_SWEEP_DUAL32_SHAPES = [("dual_gateup_M18", 18, 1536, 8960, True), ("dual_gateup_M20", 20, 1536, 8960, True),
                                 ("dual_gateup_M24", 24, 1536, 8960, True), ("dual_gateup_M28", 28, 1536, 8960, True),
                                 ("dual_gateup_M32", 32, 1536, 8960, True), ("dual3b_M24", 24, 2048, 11008, True),
                                 ("dual3b_M32", 32, 2048, 11008, True), ("dual7b_M20", 20, 3584, 18944, True)]
GU16_SWEEP_DUAL32_SHAPES = [("gu1.5b_M20", 20, 1536, 8960), ("gu1.5b_M24", 24, 1536, 8960),
                            ("gu3b_M24", 24, 2048, 11008)]
# Qwen2.5-3B (hidden 2048, MLP 11008) and 14B (hidden 5120, MLP 13824)
# projections and MLPs, which the fitted sweeps did not sample
W8_STREAM_SWEEP_3B14B_SHAPES = [("gateup3b_M8", 8, 2048, 11008, False), ("gateup3b_M24", 24, 2048, 11008, False),
                                ("down3b_M8", 8, 11008, 2048, False), ("down3b_M32", 32, 11008, 2048, False),
                                ("o3b_M8", 8, 2048, 2048, False), ("gateup14b_M8", 8, 5120, 13824, False),
                                ("down14b_M8", 8, 13824, 5120, False), ("down14b_M32", 32, 13824, 5120, False),
                                ("o14b_M8", 8, 5120, 5120, False), ("dual14b_M8", 8, 5120, 13824, True),
                                ("dual14b_M16", 16, 5120, 13824, True), ("dual3b_M4", 4, 2048, 11008, True)]
L16_SWEEP_3B14B_SHAPES = [("down3b_M8", 8, 11008, 2048), ("down3b_M32", 32, 11008, 2048),
                          ("down14b_M8", 8, 13824, 5120), ("down14b_M16", 16, 13824, 5120)]
GU16_SWEEP_3B14B_SHAPES = [("gu3b_M8", 8, 2048, 11008), ("gu14b_M8", 8, 5120, 13824), ("gu14b_M16", 16, 5120, 13824)]
# rows per workgroup that spread the weight rows evenly over the CUs (10 at
# n 5120, 14 at n 3584, 15 at n 18944) beside 8, 12 and 16
STREAM_BAL_RPWS = (8, 10, 12, 14, 15, 16)
W8_STREAM_SWEEP_BAL_SHAPES = [("down14b_M8", 8, 13824, 5120, False), ("down14b_M32", 32, 13824, 5120, False),
                              ("o14b_M8", 8, 5120, 5120, False), ("gateup14b_M8", 8, 5120, 13824, False),
                              ("down7b_M8", 8, 18944, 3584, False), ("o7b_M8", 8, 3584, 3584, False),
                              ("gateup7b_M8", 8, 3584, 18944, False), ("down7b_M4", 4, 18944, 3584, False),
                              ("dual14b_M8", 8, 5120, 13824, True), ("gateup3b_M24", 24, 2048, 11008, False)]
L16_SWEEP_BAL_SHAPES = [("down14b_M8", 8, 13824, 5120), ("down7b_M8", 8, 18944, 3584)]
GU16_SWEEP_BAL_SHAPES = [("gu14b_M8", 8, 5120, 13824)]
# the dual kernel at 5 - 16 rows where 16-row workgroups number under 4 per
# CU (14B MLP) against the 7B MLP, and the 3B gate/up at 17 - 32 rows
W8_STREAM_SWEEP_FEW16_SHAPES = [("dual14b_M5", 5, 5120, 13824, True), ("dual14b_M8", 8, 5120, 13824, True),
                                ("dual14b_M12", 12, 5120, 13824, True), ("dual14b_M16", 16, 5120, 13824, True),
                                ("dual7b_M8", 8, 3584, 18944, True), ("dual7b_M16", 16, 3584, 18944, True),
                                ("gateup3b_M17", 17, 2048, 11008, False), ("gateup3b_M20", 20, 2048, 11008, False),
                                ("gateup3b_M28", 28, 2048, 11008, False), ("gateup3b_M32", 32, 2048, 11008, False)]
# the gate/up + SiLU-and-mul kernels at 2 - 4 rows below k = 3072
W8_STREAM_SWEEP_DUAL4_SHAPES = [("dual_gateup_M2", 2, 1536, 8960, True), ("dual_gateup_M3", 3, 1536, 8960, True),
                                ("dual_gateup_M4", 4, 1536, 8960, True), ("dual3b_M2", 2, 2048, 11008, True),
                                ("dual3b_M3", 3, 2048, 11008, True), ("dual3b_M4", 4, 2048, 11008, True),
                                ("dual0.5b_M4", 4, 896, 4864, True), ("dual14b_M4", 4, 5120, 13824, True)]
GU16_SWEEP_DUAL4_SHAPES = [("gu1.5b_M4", 4, 1536, 8960), ("gu3b_M4", 4, 2048, 11008), ("gu3b_M8", 8, 2048, 11008),
                           ("gu14b_M16", 16, 5120, 13824), ("gu14b_M12", 12, 5120, 13824)]
# the 14B projections and MLP beyond 16 rows
W8_STREAM_SWEEP_14B_WIDE_SHAPES = [("down14b_M48", 48, 13824, 5120, False), ("o14b_M32", 32, 5120, 5120, False),
                                   ("o14b_M48", 48, 5120, 5120, False), ("dual14b_M24", 24, 5120, 13824, True),
                                   ("dual14b_M32", 32, 5120, 13824, True), ("gateup14b_M24", 24, 5120, 13824, False)]
L16_SWEEP_14B_WIDE_SHAPES = [("down14b_M32", 32, 13824, 5120), ("down14b_M64", 64, 13824, 5120),
                             ("o14b_M32", 32, 5120, 5120)]
GU16_SWEEP_14B_WIDE_SHAPES = [("gu14b_M24", 24, 5120, 13824), ("gu14b_M32", 32, 5120, 13824)]
# the 3B and 14B shapes at 1 - 4 rows
W8_STREAM_SWEEP_SMALLM_SHAPES = [("down14b_M1", 1, 13824, 5120, False), ("down14b_M4", 4, 13824, 5120, False),
                                 ("o14b_M1", 1, 5120, 5120, False), ("o14b_M4", 4, 5120, 5120, False),
                                 ("gateup14b_M1", 1, 5120, 13824, False), ("gateup14b_M4", 4, 5120, 13824, False),
                                 ("dual14b_M1", 1, 5120, 13824, True), ("dual14b_M2", 2, 5120, 13824, True),
                                 ("down3b_M1", 1, 11008, 2048, False), ("gateup3b_M1", 1, 2048, 11008, False),
                                 ("dual3b_M1", 1, 2048, 11008, True)]
L16_SWEEP_SMALLM_SHAPES = [("down14b_M1", 1, 13824, 5120), ("down14b_M4", 4, 13824, 5120),
                           ("down3b_M1", 1, 11008, 2048), ("down3b_M4", 4, 11008, 2048)]
GU16_SWEEP_SMALLM_SHAPES = [("gu14b_M1", 1, 5120, 13824), ("gu14b_M4", 4, 5120, 13824), ("gu3b_M1", 1, 2048, 11008)]
# 1 - 4 rows of x (one x set) on the deep projections that are not narrow
# (k >= 3072, more 8-row workgroups than CUs): 8- against 16-row workgroups
W8_STREAM_SWEEP_M4_SHAPES = [("gateup7b_M1", 1, 3584, 18944, False), ("dual7b_M1", 1, 3584, 18944, True),
                             ("gateup7b_M2", 2, 3584, 18944, False), ("gateup7b_M3", 3, 3584, 18944, False),
                             ("gateup7b_M4", 4, 3584, 18944, False), ("down7b_M1", 1, 18944, 3584, False),
                             ("down7b_M2", 2, 18944, 3584, False), ("down7b_M4", 4, 18944, 3584, False),
                             ("down7b_M3", 3, 18944, 3584, False), ("o7b_M1", 1, 3584, 3584, False),
                             ("o7b_M2", 2, 3584, 3584, False), ("o7b_M3", 3, 3584, 3584, False),
                             ("o7b_M4", 4, 3584, 3584, False),
                             ("dual7b_M2", 2, 3584, 18944, True), ("dual7b_M3", 3, 3584, 18944, True),
                             ("dual7b_M4", 4, 3584, 18944, True)]
L16_SWEEP_M4_SHAPES = [("down7b_M2", 2, 18944, 3584), ("down7b_M4", 4, 18944, 3584), ("o7b_M4", 4, 3584, 3584)]
GU16_SWEEP_M4_SHAPES = [("gu7b_M2", 2, 3584, 18944), ("gu7b_M3", 3, 3584, 18944)]
GU16_SWEEP_R8_SHAPES = [("gu1.5b_M8", 8, 1536, 8960), ("gu7b_M4", 4, 3584, 18944), ("gu7b_M8", 8, 3584, 18944)]
GU16_SWEEP16_WIDE_SHAPES = [("gu7b_M12", 12, 3584, 18944), ("gu7b_M16", 16, 3584, 18944),
                            ("gu1.5b_M16", 16, 1536, 8960)]
W8_STREAM_SWEEP16_SHAPES = [
    ("down_M12", 12, 8960, 1536, False), ("down_M16", 16, 8960, 1536, False),
    ("gateup_M12", 12, 1536, 8960, False), ("gateup_M16", 16, 1536, 8960, False),
    ("dual_gateup_M16", 16, 1536, 8960, True), ("down7b_M16", 16, 18944, 3584, False),
    ("gateup7b_M16", 16, 3584, 18944, False), ("o1.5b_M16", 16, 1536, 1536, False),
    ("down0.5b_M16", 16, 4864, 896, False), ("dual7b_M16", 16, 3584, 18944, True),
]


def _stream_sweep_shape(ctx, tag, label, M, nchunk, dual, wb, wide16, o, ref, lib_calls, make_calls, plan=None,
                        rpws=(4, 6, 8, 12, 16)):
    """The body the decode-kernel sweeps share, for one (rows, k, n): every
    launch shape _w8_stream_shapes samples (make_calls(rpw, r4, waves, u)
    builds its calls over the rotating weight sets, writing `o`), checked
    against `ref` (the library's output, within 2e-3 of its largest value:
    the fp32 summation order differs with the split of K) and timed as
    graph nodes, then the library's own calls; `plan` (rpw, r4, waves, u) is
    the launcher's plan, reported with its time."""
    torch = ctx.torch
    nodes = max(2 * len(lib_calls), 64)
    tol = 2e-3 * ref.float().abs().max().item()
    res, bad = {}, []
    for rpw, r4, waves, u in _w8_stream_shapes(nchunk, dual, stream_x_sets(M), wide16, wb, rpws):
        calls = make_calls(rpw, r4, waves, u)
        calls[0]()
        torch.cuda.synchronize()
        err = (o.float() - ref.float()).abs().max().item()
        if not err <= tol:
            bad.append((rpw, r4, waves, u, err))
        spin_up(ctx, calls, ms=3.0)
        res[f"rpw{rpw}_w{waves}_u{u}"] = round(time_graph(ctx, calls, nodes, replays=5), 3)
    # the library's own launch (unsplit, as the shapes) last, on a device already warm from the
    # shapes (timed first it read 3-10% high: clocks still ramping)
    spin_up(ctx, lib_calls, ms=5.0)
    res["library_us"] = round(time_graph(ctx, lib_calls, nodes, replays=5), 3)
    best = min((k for k in res if k != "library_us"), key=lambda k: res[k])
    rec = {"best": best, "best_us": res[best]}
    plan_msg = ""
    if plan is not None:
        key = f"rpw{plan[0]}_w{plan[2]}_u{plan[3]}"
        rec.update(plan=key, plan_us=res.get(key))
        plan_msg = f", plan {key} {res.get(key)} us"
    rec.update(library_us=res["library_us"], mismatches=bad, shapes=res)
    log(f"  {tag} stream sweep {label}: library {res['library_us']} us{plan_msg}, best {best} {res[best]} us, "
        f"{len(bad)} mismatches {bad[:3]}")
    return rec


def w8_stream_sweep(ctx, shapes=W8_STREAM_SWEEP_SHAPES, wide16=False, rpws=(4, 6, 8, 12, 16)):
    """The W8A16 decode kernel (w8a16_stream) over launch shapes, through the
    probe library's forced-shape entry point, at the Qwen2.5-1.5B down and
    gate/up projections and the int8 gate/up + SiLU-and-mul MLP, 1 and 8 rows
    of fp16 x: graph-node us over cold weights, each shape's output checked
    against the library's (within 2e-3 of the largest output: the fp32
    summation order differs with the split of K)."""
    torch = ctx.torch
    F16 = torch.float16
    cus = torch.cuda.get_device_properties(ctx.dev).multi_processor_count
    out = {}
    for label, M, K, N, dual in shapes:
        nq = 2 if dual else 1
        sets = n_sets(nq * N * K)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(2500 + K + M)
        qs = [torch.randint(-127, 128, (nq, N, K), generator=g, device=ctx.dev, dtype=torch.int8)
              for _ in range(sets)]
        scs = [(torch.rand(nq, N, generator=g, device=ctx.dev) * 1e-3 + 1e-4) for _ in range(sets)]
        x = rand(ctx, (M, K), 2600 + M, F16)
        o = torch.empty((M, N), dtype=F16, device=ctx.dev)
        ref = torch.empty_like(o)
        if dual:
            lib_calls = [ctx.gate_up_w8_call(x, q[0], sc[0], q[1], sc[1], o) for q, sc in zip(qs, scs)]
            ctx.gate_up_w8_call(x, qs[0][0], scs[0][0], qs[0][1], scs[0][1], ref)()
        else:
            lib_calls = [ctx.w8a16_call(x, q[0], sc[0], o, split=False) for q, sc in zip(qs, scs)]
            ctx.w8a16_call(x, qs[0][0], scs[0][0], ref, split=False)()
        torch.cuda.synchronize()

        def make_calls(rpw, r4, waves, u, x=x, qs=qs, scs=scs, o=o, dual=dual):
            if dual:
                return [ctx.w8_stream_plan_call(x, q[0], sc[0], o, rpw, r4, waves, u, q[1], sc[1])
                        for q, sc in zip(qs, scs)]
            return [ctx.w8_stream_plan_call(x, q[0], sc[0], o, rpw, r4, waves, u) for q, sc in zip(qs, scs)]
        out[label] = _stream_sweep_shape(ctx, "w8", label, M, -(-K // 256), dual, 1, wide16, o, ref, lib_calls,
                                         make_calls, plan=ctx.w8_stream_plan(M, K, N, dual, cus), rpws=rpws)
        del qs, scs, make_calls, lib_calls
        torch.cuda.empty_cache()
    return out


# (label, rows, k, n) of the 16-bit gate/up + SiLU-and-mul decode sweep: the
# Qwen2.5-0.5B, 1.5B and 7B MLPs at 1, 4 and 8 rows
GU16_SWEEP_SHAPES = [("gu1.5b_M1", 1, 1536, 8960), ("gu1.5b_M4", 4, 1536, 8960), ("gu1.5b_M8", 8, 1536, 8960),
                     ("gu0.5b_M1", 1, 896, 4864), ("gu0.5b_M8", 8, 896, 4864),
                     ("gu7b_M1", 1, 3584, 18944), ("gu7b_M8", 8, 3584, 18944)]
GU16_SWEEP16_SHAPES = [("gu1.5b_M12", 12, 1536, 8960), ("gu1.5b_M16", 16, 1536, 8960),
                       ("gu0.5b_M16", 16, 896, 4864), ("gu7b_M16", 16, 3584, 18944)]


# (label, rows, k, n) of the 16-bit linear sweep: the MLP down projections
# of Qwen2.5-0.5B, 1.5B and 7B at decode rows
L16_SWEEP_SHAPES = [("down1.5b_M1", 1, 8960, 1536), ("down1.5b_M8", 8, 8960, 1536), ("down1.5b_M16", 16, 8960, 1536),
                    ("down7b_M1", 1, 18944, 3584), ("down7b_M8", 8, 18944, 3584), ("down7b_M16", 16, 18944, 3584),
                    ("down0.5b_M8", 8, 4864, 896), ("down1.5b_M4", 4, 8960, 1536)]


def l16_stream_sweep(ctx, shapes=L16_SWEEP_SHAPES, rpws=(4, 6, 8, 12, 16)):
    """The 16-bit linear at decode rows: the library's launch
    (mi355_linear16_fwd) against the weight-streaming kernel of
    w8a16_stream.h with one 16-bit matrix over launch shapes (rows per
    workgroup 4-16 x waves 1-16 x chunks in flight 1-2), graph-node us over
    cold weights, fp16; each shape's output checked against the library's
    (within 2e-3 of the largest output)."""
    torch = ctx.torch
    F16 = torch.float16
    cus = torch.cuda.get_device_properties(ctx.dev).multi_processor_count
    out = {}
    for label, M, K, N in shapes:
        sets = n_sets(N * K * 2)
        ws = [rand(ctx, (N, K), 3300 + i, F16, std=K ** -0.5) for i in range(sets)]
        x = rand(ctx, (M, K), 3200 + M, F16)
        o = torch.empty((M, N), dtype=F16, device=ctx.dev)
        ref = torch.empty_like(o)
        lib_calls = [ctx.linear16_call(x, w, o, split=False) for w in ws]
        ctx.linear16_call(x, ws[0], ref, split=False)()
        torch.cuda.synchronize()
        out[label] = _stream_sweep_shape(
            ctx, "l16", label, M, -(-K // 128), False, 2, True, o, ref, lib_calls,
            lambda rpw, r4, waves, u, x=x, ws=ws, o=o: [ctx.linear16_stream_call(x, w, o, rpw, r4, waves, u)
                                                         for w in ws],
            plan=ctx.l16_stream_plan(M, K, N, cus), rpws=rpws)
        del ws
        torch.cuda.empty_cache()
    return out


def gu16_stream_sweep(ctx, shapes=GU16_SWEEP_SHAPES, wide16=False, rpws=(4, 6, 8, 12, 16)):
    """The 16-bit gate/up + SiLU-and-mul at decode rows: the library's
    launch (mi355_gate_up_silu_fwd) against the weight-streaming kernel of
    w8a16_stream.h with 16-bit weights over launch shapes (rows per
    workgroup 4-16 x waves 1-16 x chunks in flight 1-2), graph-node us over
    cold weights, fp16; each shape's output checked against the library's
    (within 2e-3 of the largest output)."""
    torch = ctx.torch
    F16 = torch.float16
    cus = torch.cuda.get_device_properties(ctx.dev).multi_processor_count
    out = {}
    for label, M, K, N in shapes:
        sets = n_sets(2 * N * K * 2)
        ws = [(rand(ctx, (N, K), 3100 + 2 * i, F16, std=2.0 * K ** -0.5), rand(ctx, (N, K), 3101 + 2 * i, F16,
                                                                                std=K ** -0.5))
              for i in range(sets)]
        x = rand(ctx, (M, K), 3000 + M, F16)
        o = torch.empty((M, N), dtype=F16, device=ctx.dev)
        ref = torch.empty_like(o)
        lib_calls = [ctx.gate_up_call(x, wg, wu, o) for wg, wu in ws]
        ctx.gate_up_call(x, ws[0][0], ws[0][1], ref)()
        torch.cuda.synchronize()
        out[label] = _stream_sweep_shape(
            ctx, "gu16", label, M, -(-K // 128), True, 2, wide16, o, ref, lib_calls,
            lambda rpw, r4, waves, u, x=x, ws=ws, o=o: [ctx.gate_up16_stream_call(x, wg, wu, o, rpw, r4, waves, u)
                                                         for wg, wu in ws],
            plan=ctx.gu16_stream_plan(M, K, N, cus), rpws=rpws)
        del ws
        torch.cuda.empty_cache()
    return out


def bench_add_rms(ctx, iters):
    """Residual add + RMSNorm at the C1 shape (beyond the reference): the fused
    kernel vs the unfused pair (torch's add, then the RMSNorm kernel), cold."""
    torch = ctx.torch
    F16 = torch.float16
    M, N = 2048, 1536
    fused_bytes = (4 * M * N + N) * 2
    w = rand(ctx, (N,), 1, F16, 1.0, 0.1)
    sets = []
    for s in range(n_sets(fused_bytes)):
        x, r = rand(ctx, (M, N), 700 + s, F16), rand(ctx, (M, N), 800 + s, F16)
        sets.append((x, r, torch.empty_like(x), torch.empty_like(x)))
    fused = [ctx.add_rms_call(x, r, w, y, h) for x, r, y, h in sets]
    rms = [ctx.rms_call(h, w, y) for x, r, y, h in sets]

    def unfused_call(i):
        x, r, y, h = sets[i]
        return lambda: (torch.add(r, x, out=h), rms[i]())

    fused_us = time_loop(ctx, fused, iters)
    unfused_us = time_loop(ctx, [unfused_call(i) for i in range(len(sets))], iters)
    out = {"c1_add_rmsnorm_f16_2048x1536": kernel_entry("rmsnorm_wave_rows (add)", fused_bytes,
                                                        fused_us, {"buffer_sets": len(sets)}),
           "c1_add_then_rmsnorm_unfused_us": round(unfused_us, 3),
           "fused_speedup": round(unfused_us / fused_us, 3)}
    log(f"  add+rmsnorm C1: fused {fused_us:.2f} us ({out['c1_add_rmsnorm_f16_2048x1536']['GBps']:.0f} GB/s), "
        f"unfused {unfused_us:.2f} us")
    del sets
    torch.cuda.empty_cache()
    return out


def bench_c4(ctx, iters=60, which=None):
    torch = ctx.torch
    BF16 = torch.bfloat16
    out = {}
    if which in (None, "c4-rms"):
        M, N = 16384, 3584
        nbytes = (2 * M * N + N) * 2
        w = rand(ctx, (N,), 1, BF16, 1.0, 0.1)
        calls, keep = [], []
        for s in range(n_sets(nbytes)):
            x = rand(ctx, (M, N), 400 + s, BF16)
            y = torch.empty_like(x)
            keep.append((x, y))
            calls.append(ctx.rms_call(x, w, y))
        spin_up(ctx, calls)
        us = time_loop(ctx, calls, iters)
        out["c4_rmsnorm_bf16_16384x3584"] = kernel_entry("rmsnorm_block_rows", nbytes, us,
                                                         {"buffer_sets": len(calls)})
        del keep, calls
        torch.cuda.empty_cache()
    if which in (None, "c4-silu"):
        M, I = 16384, 18944
        nbytes = 3 * M * I * 2
        gate = rand(ctx, (M, I), 500, BF16)
        up = rand(ctx, (M, I), 501, BF16)
        o = torch.empty_like(gate)
        spin_up(ctx, [ctx.silu_call(gate, up, o)])
        us = time_loop(ctx, [ctx.silu_call(gate, up, o)], iters)
        out["c4_silu_mul_bf16_16384x18944"] = kernel_entry("silu_mul_chunks", nbytes, us,
                                                           {"buffer_sets": 1, "footprint_GiB": round(nbytes / 2**30, 2)})
        del gate, up, o
        torch.cuda.empty_cache()
    for k, v in out.items():
        log(f"  {k}: {v['us']:.2f} us, {v['GBps']:.0f} GB/s ({v['frac_of_peak']:.1%})")
    return out


def bench_decode(ctx, layers=28):
    """C3: decode shapes.  Per call through the Python API, two ways: the
    host's wall clock around the call and a synchronize (`*_api_us`, median),
    and events around the call as the reference's _time_cuda records them
    (`*_call_us`, mean; benchmarks/run_stage3_kernels.py:34-49); device-only
    from events over back-to-back ABI launches; and inside a hipGraph of
    `layers` x (RMSNorm, SiLU-and-mul, RMSNorm) on per-layer buffers."""
    torch = ctx.torch
    F16 = torch.float16
    N, I = 1536, 8960
    res = {}
    for M in (1, 2, 4, 8, 32):
        w = rand(ctx, (N,), 1, F16, 1.0, 0.1)
        x = rand(ctx, (M, N), 600 + M, F16)
        g = rand(ctx, (M, I), 700 + M, F16)
        u = rand(ctx, (M, I), 800 + M, F16)

        def api_us(fn, n=200):
            for _ in range(10):
                fn()
            ts = []
            for _ in range(n):
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                fn()
                torch.cuda.synchronize()
                ts.append((time.perf_counter() - t0) * 1e6)
            return statistics.median(ts)

        rms_api = api_us(lambda: ctx.pkg.fused_rmsnorm(x, w))
        silu_api = api_us(lambda: ctx.pkg.fused_silu_mul(g, u))
        rms_call = _time_per_call(torch, lambda: ctx.pkg.fused_rmsnorm(x, w), 200)
        silu_call = _time_per_call(torch, lambda: ctx.pkg.fused_silu_mul(g, u), 200)
        y = torch.empty_like(x)
        o = torch.empty_like(g)
        rms_dev = time_loop(ctx, [ctx.rms_call(x, w, y)], 2000)
        silu_dev = time_loop(ctx, [ctx.silu_call(g, u, o)], 2000)

        # 28-layer graph on per-layer buffers
        xs = [rand(ctx, (M, N), 900 + l, F16) for l in range(layers)]
        ys = [torch.empty_like(t) for t in xs]
        gs = [rand(ctx, (M, I), 1000 + l, F16) for l in range(layers)]
        us_ = [rand(ctx, (M, I), 1100 + l, F16) for l in range(layers)]
        os_ = [torch.empty_like(t) for t in gs]
        ws = [rand(ctx, (N,), 1200 + l, F16, 1.0, 0.1) for l in range(2 * layers)]
        zs = [torch.empty_like(t) for t in xs]
        calls = []
        for l in range(layers):
            calls += [ctx.rms_call(xs[l], ws[2 * l], ys[l]), ctx.silu_call(gs[l], us_[l], os_[l]),
                      ctx.rms_call(ys[l], ws[2 * l + 1], zs[l])]
        per_kernel = time_graph(ctx, calls, len(calls), replays=50)
        replay_us = per_kernel * len(calls)
        res[f"M={M}"] = {
            "rmsnorm_api_us": round(rms_api, 2), "silu_mul_api_us": round(silu_api, 2),
            "rmsnorm_call_us": round(rms_call, 2), "silu_mul_call_us": round(silu_call, 2),
            "rmsnorm_device_us": round(rms_dev, 3), "silu_mul_device_us": round(silu_dev, 3),
            "graph_replay_us": round(replay_us, 2), "graph_per_layer_us": round(replay_us / layers, 3),
            "graph_per_kernel_us": round(per_kernel, 3),
            "rows_per_s_rmsnorm": round(M / (rms_dev * 1e-6)),
        }
        log(f"  decode M={M}: {res[f'M={M}']}")
    if ctx.probe is not None:
        # the floor under every decode figure: an empty kernel, and the probe
        # copy of one 1536-wide fp16 row (one HBM round trip), back to back and
        # as nodes of a hipGraph of the same length as the 28-layer graph
        empty = [ctx.empty_call()]
        src = torch.empty(1536 * 2, dtype=torch.uint8, device=ctx.dev)
        dst = torch.empty_like(src)
        row = [ctx.copy_call(src, dst)]
        res["floor"] = {
            "empty_kernel_eager_us": round(time_loop(ctx, empty, 2000), 3),
            "empty_kernel_graph_node_us": round(time_graph(ctx, empty, 3 * layers, replays=50), 3),
            "row_copy_eager_us": round(time_loop(ctx, row, 2000), 3),
            "row_copy_graph_node_us": round(time_graph(ctx, row, 3 * layers, replays=50), 3),
        }
        log(f"  decode floor: {res['floor']}")
    return res


# (rows, k, n_out, dtype name, label): decode steps of Qwen2.5-1.5B and -7B MLPs
GATE_UP_SHAPES = [(1, 1536, 8960, "f16", "qwen2.5-1.5b"), (8, 1536, 8960, "f16", "qwen2.5-1.5b"),
                  (32, 1536, 8960, "f16", "qwen2.5-1.5b"), (8, 3584, 18944, "bf16", "qwen2.5-7b")]


def bench_gate_up(ctx, shapes=GATE_UP_SHAPES, iters=400, baselines=True):
    """Gate/up projections + SiLU-and-mul at decode rows (beyond the
    reference): the fused kernel against the reference's FusedMLP chain (two
    GEMMs through torch / hipBLASLt, then the SiLU-and-mul kernel), on
    per-layer weight sets whose footprint exceeds 1 GiB, so every call
    streams its weights from HBM as a decode step walking the layers does.
    Algorithmic bytes: both weight matrices + x + out.  Timed over
    back-to-back launches and inside a hipGraph (no launch gaps)."""
    torch = ctx.torch
    dts = {"f16": torch.float16, "bf16": torch.bfloat16}
    res = {}
    for M, K, I, dname, label in shapes:
        dt = dts[dname]
        wbytes = 2 * I * K * 2
        nbytes = wbytes + M * K * 2 + M * I * 2
        layers = n_sets(wbytes)
        x = rand(ctx, (M, K), 1400 + M, dt)
        ws = [(rand(ctx, (I, K), 1500 + 2 * l, dt, std=2.0 * K ** -0.5),
               rand(ctx, (I, K), 1501 + 2 * l, dt, std=K ** -0.5)) for l in range(layers)]
        outs = [torch.empty((M, I), dtype=dt, device=ctx.dev) for _ in range(layers)]
        fused = [ctx.gate_up_call(x, wg, wu, o) for (wg, wu), o in zip(ws, outs)]
        us = time_loop(ctx, fused, iters)
        us_graph = time_graph(ctx, fused, 4 * layers)
        key = f"{label}_M{M}_{dname}"
        kname = "w8a16_stream (16-bit weights)" if M <= 8 else ("gate_up_silu_skinny" if M <= 16 else
                                                                  "gate_up_silu_skinny or tiled_gemm")
        entry = kernel_entry(kname, nbytes, us,
                             {"weight_sets": layers, "graph_us": round(us_graph, 3),
                              "graph_GBps": round(nbytes / us_graph / 1e3, 1)})
        if baselines:
            silu = ctx.pkg.fused_silu_mul

            def chain(wg, wu):
                return lambda: silu(torch.matmul(x, wg.T), torch.matmul(x, wu.T))

            chains = [chain(wg, wu) for wg, wu in ws]
            c_us = time_loop(ctx, chains, iters)
            c_graph = time_graph(ctx, chains, 4 * layers)
            entry.update({"unfused_chain_us": round(c_us, 3), "unfused_chain_graph_us": round(c_graph, 3),
                          "speedup_graph": round(c_graph / us_graph, 3)})
        res[key] = entry
        log(f"  gate_up {key}: {entry}")
        del ws, outs, fused
        torch.cuda.empty_cache()
    return res


# (rows, k, n_out, dtype name, label): prefill batches of Qwen2.5-1.5B and -7B MLPs
GATE_UP_PREFILL_SHAPES = [(128, 1536, 8960, "f16", "qwen2.5-1.5b"), (1024, 1536, 8960, "f16", "qwen2.5-1.5b"),
                          (4096, 1536, 8960, "f16", "qwen2.5-1.5b"), (4096, 3584, 18944, "bf16", "qwen2.5-7b")]
# the Qwen2.5-0.5B, 1.5B and 7B MLPs over prefill row counts (--only gate-up-prefill-sweep)
GATE_UP_PREFILL_SWEEP_SHAPES = (
    [(m, 1536, 8960, "f16", "qwen2.5-1.5b") for m in (64, 128, 256, 384, 512, 768, 1024, 1400, 1536, 2048, 2900, 3072,
                                                       4096)]
    + [(m, 3584, 18944, "bf16", "qwen2.5-7b") for m in (256, 512, 1024, 1100, 1536, 1792, 2048, 4096)]
    + [(m, 896, 4864, "bf16", "qwen2.5-0.5b") for m in (256, 1024, 4096)])


def bench_gate_up_prefill(ctx, shapes=GATE_UP_PREFILL_SHAPES, iters=60, baselines=True):
    """Gate/up projections + SiLU-and-mul at prefill rows (the tiled MFMA
    GEMM with the activation in its epilogue) against the reference's FusedMLP
    chain on the same weights: two torch.matmul GEMMs (hipBLASLt), each
    rounded to x's dtype, then the SiLU-and-mul kernel.  MFMA-bound: flops
    2 * 2 * rows * k * n_out per call; weight sets rotate as in the decode leg."""
    torch = ctx.torch
    dts = {"f16": torch.float16, "bf16": torch.bfloat16}
    res = {}
    for M, K, I, dname, label in shapes:
        dt = dts[dname]
        flops = 4.0 * M * K * I
        layers = min(8, n_sets(2 * I * K * 2))
        x = rand(ctx, (M, K), 2400 + M, dt)
        ws = [(rand(ctx, (I, K), 2500 + 2 * l, dt, std=2.0 * K ** -0.5),
               rand(ctx, (I, K), 2501 + 2 * l, dt, std=K ** -0.5)) for l in range(layers)]
        outs = [torch.empty((M, I), dtype=dt, device=ctx.dev) for _ in range(2)]
        fused = [ctx.gate_up_call(x, wg, wu, outs[l % 2]) for l, (wg, wu) in enumerate(ws)]
        spin_up(ctx, fused)
        us = time_loop(ctx, fused, iters)
        tf = flops / us / 1e6
        entry = {"kernel": "tiled_gemm<2 x 16-bit B, SiLU-and-mul epilogue>", "rows": M, "k": K, "n_out": I,
                 "dtype": dname, "us": round(us, 3), "TFLOPs": round(tf, 1),
                 "frac_of_mfma_peak": round(tf / MFMA_PEAK_TFLOPS, 4), "weight_sets": layers}
        if baselines:
            silu = ctx.pkg.fused_silu_mul

            def chain(wg, wu):
                return lambda: silu(torch.matmul(x, wg.T), torch.matmul(x, wu.T))

            chains = [chain(wg, wu) for wg, wu in ws]
            spin_up(ctx, chains)
            c_us = time_loop(ctx, chains, iters)
            entry.update({"unfused_chain_us": round(c_us, 3), "unfused_chain_TFLOPs": round(flops / c_us / 1e6, 1),
                          "speedup": round(c_us / us, 3)})
            del chains
        res[f"{label}_M{M}_{dname}"] = entry
        log(f"  gate_up prefill {label} M={M}: {entry}")
        del ws, outs, fused
        torch.cuda.empty_cache()
    return res


# (rows, k, n_out, dtype name, label): int8 gate/up + SiLU-and-mul, decode and prefill rows
GATE_UP_W8_SHAPES = [(1, 1536, 8960, "f16", "qwen2.5-1.5b"), (8, 1536, 8960, "f16", "qwen2.5-1.5b"),
                     (32, 1536, 8960, "f16", "qwen2.5-1.5b"), (8, 3584, 18944, "bf16", "qwen2.5-7b"),
                     (1024, 1536, 8960, "f16", "qwen2.5-1.5b")]
GATE_UP_W8_PREFILL_SHAPES = [(1024, 1536, 8960, "f16", "qwen2.5-1.5b"), (4096, 1536, 8960, "f16", "qwen2.5-1.5b"),
                             (1024, 3584, 18944, "bf16", "qwen2.5-7b"), (4096, 3584, 18944, "bf16", "qwen2.5-7b"),
                             # row counts whose tile counts are not multiples of 8
                             (1400, 1536, 8960, "f16", "qwen2.5-1.5b"), (2900, 1536, 8960, "f16", "qwen2.5-1.5b"),
                             (1100, 3584, 18944, "bf16", "qwen2.5-7b")]


def bench_gate_up_w8(ctx, shapes=GATE_UP_W8_SHAPES, iters=300, baselines=True):
    """Int8 gate/up projections + SiLU-and-mul (one kernel, through its C ABI
    entry point) against
    the quantised model's chain: two W8A16 linears (this build's kernel, each
    rounded to x's dtype) and the SiLU-and-mul kernel.  Per-layer int8
    weight sets with a footprint above 1 GiB; eager back-to-back and hipGraph
    timing (min).  Algorithmic bytes: both int8 matrices + both fp32 scales +
    x + out."""
    torch = ctx.torch
    pkg = ctx.pkg
    dts = {"f16": torch.float16, "bf16": torch.bfloat16}
    res = {}
    for M, K, I, dname, label in shapes:
        dt = dts[dname]
        nbytes = 2 * I * K + 2 * 4 * I + M * K * 2 + M * I * 2
        flops = 4.0 * M * K * I
        sets = min(128, n_sets(2 * I * K))
        x = rand(ctx, (M, K), 2600 + M, dt)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(2700 + K + I)
        ws = [(torch.randint(-127, 128, (I, K), generator=g, device=ctx.dev, dtype=torch.int8),
               torch.rand(I, generator=g, device=ctx.dev) * 2e-3 + 1e-4,
               torch.randint(-127, 128, (I, K), generator=g, device=ctx.dev, dtype=torch.int8),
               torch.rand(I, generator=g, device=ctx.dev) * 1e-3 + 1e-4) for _ in range(sets)]
        outs = [torch.empty((M, I), dtype=dt, device=ctx.dev) for _ in range(4)]
        fused = [ctx.gate_up_w8_call(x, w[0], w[1], w[2], w[3], outs[i % 4]) for i, w in enumerate(ws)]
        spin_up(ctx, fused)
        us = min(time_loop(ctx, fused, iters), time_graph(ctx, fused, max(2 * sets, 64)))
        entry = kernel_entry("w8a16 dual (gate/up + SiLU-and-mul)", nbytes, us,
                             {"rows": M, "k": K, "n_out": I, "dtype": dname, "weight_sets": sets,
                              "TFLOPs": round(flops / us / 1e6, 1)})
        if baselines:
            chains = [lambda w=w: pkg.fused_silu_mul(pkg.w8a16_linear(x, w[0], w[1]),
                                                     pkg.w8a16_linear(x, w[2], w[3])) for w in ws]
            spin_up(ctx, chains)
            c_us = min(time_loop(ctx, chains, iters), time_graph(ctx, chains, max(2 * sets, 64)))
            entry.update({"w8a16_chain_us": round(c_us, 3), "speedup": round(c_us / us, 3)})
            del chains
        res[f"{label}_M{M}_{dname}"] = entry
        log(f"  int8 gate_up {label} M={M}: {entry}")
        del ws, fused, outs
        torch.cuda.empty_cache()
    return res


# (M, K, N, dtype name, label): the reference's stage-7 kernel benchmark shapes
# (benchmarks/run_stage7_kernel.py:33-39, Qwen2.5-1.5B projections, M in
# {1, 8, 128, 1024}) plus Qwen2.5-7B MLP decode shapes in bf16.
W8A16_SHAPES = [(M, K, N, "f16", lab) for K, N, lab in ((1536, 1536, "q/o proj"), (1536, 256, "k/v proj"),
                                                         (1536, 8960, "gate/up proj"), (8960, 1536, "down proj"))
                for M in (1, 8, 128, 1024)] + [(8, 3584, 18944, "bf16", "7b gate/up proj"),
                                               (8, 18944, 3584, "bf16", "7b down proj"),
                                               (4096, 1536, 8960, "f16", "gate/up proj"),
                                               (4096, 8960, 1536, "f16", "down proj")]


# (rows, k, n, dtype name, label): W8A16 single GEMMs with wide outputs at prefill rows
W8A16_WIDE_PREFILL_SHAPES = [(1024, 1536, 8960, "f16", "gate/up proj"), (4096, 1536, 8960, "f16", "gate/up proj"),
                             (1024, 3584, 18944, "bf16", "7b gate/up proj"),
                             (4096, 3584, 18944, "bf16", "7b gate/up proj"), (1024, 1536, 4736, "f16", "n 4736"),
                             (1024, 18944, 3584, "bf16", "7b down proj"), (4096, 18944, 3584, "bf16", "7b down proj"),
                             (1024, 3584, 3584, "bf16", "7b o proj"), (1280, 1536, 8960, "f16", "gate/up proj"),
                             (1024, 1536, 8960, "bf16", "gate/up proj"), (2048, 1536, 4736, "f16", "n 4736")]
# W8A16 single GEMMs with narrow (1536-wide) outputs at prefill rows: the 1.5B down and q/o projections
W8A16_NARROW_PREFILL_SHAPES = [(1024, 8960, 1536, "f16", "down proj"), (4096, 8960, 1536, "f16", "down proj"),
                               (2048, 8960, 1536, "f16", "down proj"), (1024, 1536, 1536, "f16", "q/o proj"),
                               (4096, 1536, 1536, "f16", "q/o proj"), (512, 8960, 1536, "f16", "down proj"),
                               (768, 8960, 1536, "f16", "down proj"), (1280, 8960, 1536, "f16", "down proj"),
                               (512, 1536, 1536, "f16", "q/o proj"), (1024, 1536, 2048, "f16", "n 2048"),
                               (1024, 1536, 1024, "f16", "n 1024")]

# W8A16 single GEMMs at prefill row counts whose tile counts are not multiples of 8
W8A16_RAGGED_PREFILL_SHAPES = [(1400, 1536, 8960, "f16", "gate/up proj"), (2900, 1536, 8960, "f16", "gate/up proj"),
                               (1100, 3584, 18944, "bf16", "7b gate/up proj"), (700, 1536, 8960, "f16", "gate/up proj"),
                               (1300, 8960, 1536, "f16", "down proj"), (1900, 8960, 1536, "f16", "down proj"),
                               (1100, 18944, 3584, "bf16", "7b down proj")]

# (rows, k, n, dtype name, label): the MLP down projections of Qwen2.5-1.5B and -7B at decode rows
LINEAR16_SHAPES = [(1, 8960, 1536, "f16", "qwen2.5-1.5b down"), (8, 8960, 1536, "f16", "qwen2.5-1.5b down"),
                   (16, 8960, 1536, "f16", "qwen2.5-1.5b down"), (32, 8960, 1536, "f16", "qwen2.5-1.5b down"),
                   (1, 18944, 3584, "bf16", "qwen2.5-7b down"), (8, 18944, 3584, "bf16", "qwen2.5-7b down"),
                   (16, 18944, 3584, "bf16", "qwen2.5-7b down")]


def bench_linear16(ctx, shapes=LINEAR16_SHAPES, iters=300, baselines=True):
    """The MLP's down projection at decode rows on the HIP 16-bit linear
    (mi355_linear16_ws_fwd: weight streaming on MFMA, from 17 rows split K)
    against torch's linear
    (hipBLASLt), the call FusedMLP makes otherwise, on per-layer weight sets
    whose footprint exceeds 1 GiB (cold HBM, as a decode step walking the
    layers).  Algorithmic bytes: weights + x + out.  Timed over back-to-back
    launches and inside a hipGraph."""
    torch = ctx.torch
    dts = {"f16": torch.float16, "bf16": torch.bfloat16}
    res = {}
    for M, K, N, dname, label in shapes:
        dt = dts[dname]
        wbytes = N * K * 2
        nbytes = wbytes + M * K * 2 + M * N * 2
        layers = n_sets(wbytes)
        x = rand(ctx, (M, K), 1700 + M, dt)
        ws = [rand(ctx, (N, K), 1800 + l, dt, std=K ** -0.5) for l in range(layers)]
        outs = [torch.empty((M, N), dtype=dt, device=ctx.dev) for _ in range(layers)]
        calls = [ctx.linear16_call(x, w, o) for w, o in zip(ws, outs)]
        spin_up(ctx, calls)
        us = time_loop(ctx, calls, iters)
        us_graph = time_graph(ctx, calls, 4 * layers)
        best = min(us, us_graph)
        key = f"{label}_M{M}_{dname}"
        small_tiles = 16 < M <= 64 and -(-N // (128 if (M <= 32 and N > 10000) else 64)) >= 128
        kname = "w8a16_stream (16-bit weights)" if M <= 64 and not small_tiles else "linear16 tiled"
        if ctx.lib.mi355_linear16_workspace(M, K, N) > 0:
            kname = "linear16 tiled (split K) + split_k_reduce"
        entry = kernel_entry(kname, nbytes, best,
                             {"rows": M, "k": K, "n": N, "weight_sets": layers, "eager_us": round(us, 3),
                              "graph_us": round(us_graph, 3)})
        if (M, K, N, dname) == (8, 8960, 1536, "f16"):
            entry["traffic"] = read_traffic("16-bit linear, 8 rows, [1536,8960] weights, fp16 (1.5B down)")
        if baselines:
            tcalls = [(lambda w=w: torch.nn.functional.linear(x, w)) for w in ws]
            t_us = time_loop(ctx, tcalls, iters)
            t_graph = time_graph(ctx, tcalls, 4 * layers)
            tb = min(t_us, t_graph)
            entry.update({"torch_linear_us": round(tb, 3), "torch_linear_GBps": round(nbytes / tb / 1e3, 1),
                          "speedup": round(tb / best, 3)})
        res[key] = entry
        log(f"  linear16 {key}: {entry}")
        del ws, outs, calls
        torch.cuda.empty_cache()
    return res


# (hidden, intermediate) of the Qwen2.5 sizes the tile plans were fitted on, and prompt-sized row counts
TILE_PLAN_DIMS = ((896, 4864), (1536, 8960), (2048, 11008), (3584, 18944), (5120, 13824))
TILE_PLAN_ROWS = (72, 100, 160, 256, 333, 512, 700, 1000, 1536, 2048, 3000, 4096)


def tile_plan_table(ctx, dims=TILE_PLAN_DIMS, rows=TILE_PLAN_ROWS):
    """The time that the tile and split-K plans predict for the launch they
    choose against that launch measured (hipGraph, weights rotated through
    HBM, fp16), over the Qwen2.5 projections at more than 64 rows: a markdown
    table per kernel, with the mean error and bias.  (Calls that leave the
    tiled kernels are not listed.)"""
    torch = ctx.torch
    F16, ll, i32 = torch.float16, ctypes.c_longlong, ctypes.c_int
    tile = ctx.probe.mi355_probe_tile_plan
    tile.argtypes, tile.restype = [i32, ll, ll, ll, i32, ctypes.POINTER(i32)], ctypes.c_double
    split = ctx.probe.mi355_probe_split_plan
    split.argtypes, split.restype = [ll, ll, ll, i32, i32, ctypes.POINTER(i32)], ll
    cost = ctx.probe.mi355_probe_split_cost
    cost.argtypes, cost.restype = [ll, ll, ll, i32, i32, ctypes.POINTER(ctypes.c_double)], None
    cus = torch.cuda.get_device_properties(ctx.dev).multi_processor_count
    t9, s4, c2 = (i32 * 9)(), (i32 * 4)(), (ctypes.c_double * 2)()
    g = torch.Generator(device=ctx.dev)
    g.manual_seed(7)
    out = []
    for table, name, wb, mats in ((0, "16-bit linear", 2, 1), (1, "int8 linear", 1, 1), (2, "16-bit gate/up", 2, 2),
                                  (3, "int8 gate/up", 1, 2)):
        lines, err = [], {"unsplit": [], "split K": []}
        shapes = [(h, i) for h, i in dims]
        if mats == 1:
            shapes = [s for h, i in dims for s in ((h, h), (i, h), (h, i))]
        for k, n in shapes:
            sets = min(40, max(2, n_sets(mats * n * k * wb)))
            if wb == 1:
                ws = [(torch.randint(-127, 128, (mats, n, k), generator=g, device=ctx.dev, dtype=torch.int8),
                       torch.rand(mats, n, generator=g, device=ctx.dev) * 1e-3) for _ in range(sets)]
            else:
                ws = [(rand(ctx, (mats, n, k), 40 + i, F16, std=k ** -0.5), None) for i in range(sets)]
            for m in rows:
                x, o = rand(ctx, (m, k), m, F16), torch.empty((m, n), dtype=F16, device=ctx.dev)
                tiles64 = -(-n // 64) * -(-m // 64)
                if wb == 1 and m <= 256 and (tiles64 < 32 or (m <= 128 and n < 2048)):
                    continue  # 32-row tiles of the W8A16 kernels' own
                us, kind = tile(table, m, k, n, cus, t9), "unsplit"
                plan = f"{t9[3]} x {t9[4]}"
                if t9[1]:
                    plan += f" over {t9[1]} columns, then {t9[6]} x {t9[7]}"
                if mats == 1 and split(m, k, n, wb, cus, s4) > 0:
                    cost(m, k, n, wb, cus, c2)
                    us, kind, plan = c2[0], "split K", f"{s4[2]} x {s4[3]}, {s4[1]} ranges"
                if mats == 2:
                    calls = [ctx.gate_up_w8_call(x, w[0], s[0], w[1], s[1], o) if wb == 1 else
                             ctx.gate_up_call(x, w[0], w[1], o) for w, s in ws]
                else:
                    calls = [ctx.w8a16_call(x, w[0], s[0], o) if wb == 1 else ctx.linear16_call(x, w[0], o)
                             for w, s in ws]
                spin_up(ctx, calls, ms=4.0)
                got = time_graph(ctx, calls, max(sets, 20), replays=3)
                err[kind].append(us / got - 1)
                lines.append(f"| {m} | {k} | {n} | {plan} | {us:.1f} | {got:.1f} | {us / got - 1:+.0%} |")
            del ws
            torch.cuda.empty_cache()
        out.append(f"## {name}\n")
        for kind, e in err.items():
            if e:
                out.append(f"{kind}: {len(e)} sizes, mean error {statistics.mean(map(abs, e)):.1%}, bias "
                           f"{statistics.mean(e):+.1%}, from {min(e):+.0%} to {max(e):+.0%}.")
        out += ["", "| rows | k | n | launch | predicted us | measured us | error |", "|---|---|---|---|---|---|---|",
                *lines, ""]
        log(f"  tile plans, {name}: {len(lines)} sizes")
    return "\n".join(out)


def w8a16_kernel_name(M, N, K=0, workspace=0):
    """The kernel mi355_w8a16_linear_ws_fwd runs for this shape (aligned
    inputs, descriptors that fit), given the workspace bytes it asks for: split
    K where it asks for any; the weight-streaming kernel up to 48 rows (64 for
    at most 8 MB of weights), but for wide outputs with 2048 < k < 3072 beyond
    8 rows (the skinny kernel) and where the small tiled shapes pay (17 - 64
    rows, >= 128 tile columns); the skinny kernel for small grids, the tiled
    MFMA GEMM otherwise."""
    if workspace > 0:
        return "tiled_gemm<int8 B> (split K) + split_k_reduce"
    bn = 128 if (M <= 32 and N > 10000) else 64
    if 16 < M <= 64 and -(-N // bn) >= 128:
        return "tiled_gemm<int8 B> (small tiles)"
    if M <= 8 or ((M <= 48 or (M <= 64 and N * K <= 8 << 20)) and not (N > 10000 and 2048 < K < 3072)):
        return "w8a16_stream"
    if M <= 32:
        return "w8a16_skinny"
    tiles64 = ((N + 63) // 64) * ((M + 63) // 64)
    skinny = M <= 256 and (tiles64 < 32 or (M <= 128 and N < 2048))
    return "w8a16_skinny" if skinny else "tiled_gemm<int8 B>"


MFMA_PEAK_TFLOPS = 2500.0  # MI355X dense fp16 / bf16


def bench_w8a16(ctx, shapes=W8A16_SHAPES, iters=300, baselines=True):
    """Weight-only int8 linear (the reference's stage-7 path): the W8A16
    kernel against an fp16/bf16 torch.matmul (hipBLASLt) on the same shape,
    as the reference's run_stage7_kernel.py compares against cuBLAS.  Both
    rotate per-layer weight sets with a footprint above 1 GiB (cold HBM).
    Algorithmic bytes: int8 weights + fp32 scales + x + out; flops 2*M*N*K."""
    torch = ctx.torch
    dts = {"f16": torch.float16, "bf16": torch.bfloat16}
    res = {}
    for M, K, N, dname, label in shapes:
        dt = dts[dname]
        nbytes = N * K + 4 * N + M * K * 2 + M * N * 2
        flops = 2.0 * M * N * K
        sets = min(512, n_sets(N * K))
        x = rand(ctx, (M, K), 1700 + M, dt)
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(1800 + K + N)
        qs = [torch.randint(-127, 128, (N, K), generator=g, device=ctx.dev, dtype=torch.int8) for _ in range(sets)]
        scales = [(torch.rand(N, generator=g, device=ctx.dev) * 1e-3 + 1e-4) for _ in range(sets)]
        outs = [torch.empty((M, N), dtype=dt, device=ctx.dev) for _ in range(min(sets, 8))]
        calls = [ctx.w8a16_call(x, q, sc, outs[i % len(outs)]) for i, (q, sc) in enumerate(zip(qs, scales))]
        spin_up(ctx, calls)
        us = time_loop(ctx, calls, iters)
        us_graph = time_graph(ctx, calls, max(2 * sets, 64) if sets <= 256 else sets)
        kname = w8a16_kernel_name(M, N, K, ctx.lib.mi355_w8a16_linear_workspace(M, K, N))
        entry = kernel_entry(kname, nbytes, min(us, us_graph),
                             {"layer": label, "M": M, "K": K, "N": N, "dtype": dname, "weight_sets": sets,
                              "eager_us": round(us, 3), "graph_us": round(us_graph, 3),
                              "TFLOPs": round(flops / min(us, us_graph) / 1e6, 2)})
        entry["frac_of_mfma_peak"] = round(entry["TFLOPs"] / MFMA_PEAK_TFLOPS, 4)
        del qs, scales, calls
        torch.cuda.empty_cache()
        if baselines:
            bsets = min(512, n_sets(N * K * 2))
            ws = [rand(ctx, (N, K), 1900 + i, dt, std=0.02) for i in range(bsets)]

            def mm(w, o):
                return lambda: torch.matmul(x, w.T, out=o)

            base = [mm(w, outs[i % len(outs)]) for i, w in enumerate(ws)]
            spin_up(ctx, base)
            b_us = time_loop(ctx, base, iters)
            b_graph = time_graph(ctx, base, max(2 * bsets, 64) if bsets <= 256 else bsets)
            b = min(b_us, b_graph)
            entry.update({"fp16_matmul_us": round(b, 3), "speedup_vs_fp16_matmul": round(b / entry["us"], 3)})
            del ws, base
        res[f"{label.replace(' ', '_').replace('/', '')}_M{M}_{dname}"] = entry
        log(f"  w8a16 {label} M={M} K={K} N={N} {dname}: {entry['us']:.2f} us, {entry['GBps']:.0f} GB/s "
            f"({entry['frac_of_peak']:.1%}), {entry['TFLOPs']:.1f} TFLOP/s; fp16 matmul "
            f"{entry.get('fp16_matmul_us', float('nan')):.2f} us")
        del outs
        torch.cuda.empty_cache()
    return res


def bench_prefill_core(ctx, shapes=((1024, 1536, 8960), (1024, 8960, 1536), (4096, 1536, 8960),
                                      (4096, 8960, 1536)), iters=200):
    """The tiled GEMM core at prefill rows with each kind of B operand, next
    to hipBLASLt: the 1.5B gate/up and down projections (fp16 x) through
    mi355_linear16_ws_fwd (16-bit weights), mi355_w8a16_linear_ws_fwd (int8 weights,
    widened after each LDS read) and torch.matmul on the 16-bit weights.  If
    widening the int8 weights were what held the W8A16 GEMM back, the 16-bit
    path of the same core would be the faster one.  Cold weights (rotating
    sets), min of eager and hipGraph timing, us."""
    torch = ctx.torch
    F16 = torch.float16
    res = {}
    for M, K, N in shapes:
        x = rand(ctx, (M, K), 3, F16)
        outs = [torch.empty((M, N), dtype=F16, device=ctx.dev) for _ in range(4)]
        sets = min(64, n_sets(N * K * 2))
        ws = [rand(ctx, (N, K), 10 + i, F16, std=0.02) for i in range(sets)]
        entry = {}
        for name, calls in (("linear16_us", [ctx.linear16_call(x, w, outs[i % 4]) for i, w in enumerate(ws)]),
                            ("hipblaslt_fp16_us", [(lambda w=w, o=outs[i % 4]: torch.matmul(x, w.T, out=o))
                                                   for i, w in enumerate(ws)])):
            spin_up(ctx, calls)
            entry[name] = round(min(time_loop(ctx, calls, iters), time_graph(ctx, calls, 2 * sets)), 3)
        del ws
        torch.cuda.empty_cache()
        g = torch.Generator(device=ctx.dev)
        g.manual_seed(1)
        sets8 = min(128, n_sets(N * K))
        qs = [torch.randint(-127, 128, (N, K), generator=g, device=ctx.dev, dtype=torch.int8) for _ in range(sets8)]
        sc = [(torch.rand(N, generator=g, device=ctx.dev) * 1e-3 + 1e-4) for _ in range(sets8)]
        calls = [ctx.w8a16_call(x, q, s_, outs[i % 4]) for i, (q, s_) in enumerate(zip(qs, sc))]
        spin_up(ctx, calls)
        entry["w8a16_us"] = round(min(time_loop(ctx, calls, iters), time_graph(ctx, calls, 2 * sets8)), 3)
        for k_ in ("linear16_us", "w8a16_us"):
            entry[k_.replace("_us", "_vs_hipblaslt")] = round(entry["hipblaslt_fp16_us"] / entry[k_], 3)
        res[f"M{M}_K{K}_N{N}"] = entry
        log(f"  prefill core M={M} K={K} N={N}: {entry}")
        del qs, sc, calls, outs
        torch.cuda.empty_cache()
    return res


def bench_copy(ctx, nbytes=1 << 30, iters=30):
    """Plain 16-byte streaming copy of 1 GiB (2 GiB of traffic per launch)."""
    if ctx.probe is None:
        return None
    torch = ctx.torch
    src = torch.empty(nbytes, dtype=torch.uint8, device=ctx.dev).random_(0, 255)
    dst = torch.empty_like(src)
    us = time_loop(ctx, [ctx.copy_call(src, dst)], iters)
    d = kernel_entry("stream_copy", 2 * nbytes, us)
    del src, dst
    torch.cuda.empty_cache()
    log(f"  copy ceiling: {d['GBps']:.0f} GB/s ({d['frac_of_peak']:.1%})")
    return d


# (label, streams read, bytes per stream) of each benchmarked kernel's access
# mix: RMSNorm reads one row stream and writes one (its weight row is an L2
# hit), SiLU-and-mul reads two and writes one.
CEILING_SHAPES = [
    ("C1 RMSNorm [2048,1536] fp16", 1, 2048 * 1536 * 2),
    ("C2 SiLU-and-mul [2048,8960] fp16", 2, 2048 * 8960 * 2),
    ("C4 RMSNorm [16384,3584] bf16", 1, 16384 * 3584 * 2),
    ("C4 SiLU-and-mul [16384,18944] bf16", 2, 16384 * 18944 * 2),
    ("1 GiB per stream", 1, 1 << 30),
    ("512 MiB per stream", 2, 1 << 29),
]


def bench_ceilings(ctx, iters=200):
    """Achievable HBM bandwidth at each kernel's own byte count and access mix:
    the probe copy (one read stream, one write stream) or add2 (two read
    streams, one write stream), cold (rotating buffer sets of >= 1 GiB), the
    same timing as the kernels.  A kernel's time over its ceiling's time is
    the fraction of what this device moves at that size that it reaches."""
    if ctx.probe is None:
        return None
    torch = ctx.torch
    out = {}
    for label, nread, nbytes in CEILING_SHAPES:
        traffic = (nread + 1) * nbytes
        nset = n_sets(traffic)
        bufs, calls = [], []
        for _ in range(nset):
            ins = [torch.empty(nbytes, dtype=torch.uint8, device=ctx.dev).random_(0, 255) for _ in range(nread)]
            dst = torch.empty(nbytes, dtype=torch.uint8, device=ctx.dev)
            bufs.append((ins, dst))
            calls.append(ctx.copy_call(ins[0], dst) if nread == 1 else ctx.add2_call(ins[0], ins[1], dst))
        torch.cuda.synchronize()
        spin_up(ctx, calls)
        n = iters if traffic < (1 << 30) else max(20, iters // 10)
        us = time_loop(ctx, calls, n)
        d = kernel_entry("stream_copy" if nread == 1 else "stream_add2", traffic, us, {"buffer_sets": nset})
        out[label] = d
        log(f"  ceiling {label}: {us:.2f} us, {d['GBps']:.0f} GB/s ({d['frac_of_peak']:.1%})")
        del bufs, calls
        torch.cuda.empty_cache()
    return out


def _e2e_model(torch, dev):
    """A random-init Qwen2 with Qwen2.5-1.5B's architecture (28 layers, hidden
    1536, intermediate 8960, 12 / 2 heads, vocab 151936) in fp16 on `dev`,
    sdpa attention: the reference's e2e model without Hub access."""
    from transformers import Qwen2Config, Qwen2ForCausalLM

    cfg = Qwen2Config(vocab_size=151936, hidden_size=1536, intermediate_size=8960, num_hidden_layers=28,
                      num_attention_heads=12, num_key_value_heads=2, max_position_embeddings=32768,
                      rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=True, attn_implementation="sdpa")
    torch.manual_seed(0)
    with torch.device(dev):
        model = Qwen2ForCausalLM(cfg)
    return model.half().eval()


def _e2e_run(torch, model, ids, gen_len):
    """One prefill (TTFT, ms, event-timed) and gen_len - 1 greedy decode steps
    over HF's KV cache (tokens/s), as the reference's profiler times them
    (src/engine/profiler.py:72-204)."""
    with torch.inference_mode():
        torch.cuda.synchronize()
        s0, s1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s0.record()
        out = model(input_ids=ids, use_cache=True)
        past = out.past_key_values
        tok = out.logits[:, -1].argmax(-1, keepdim=True)
        s1.record()
        torch.cuda.synchronize()
        d0, d1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        d0.record()
        for _ in range(gen_len - 1):
            out = model(input_ids=tok, past_key_values=past, use_cache=True)
            past = out.past_key_values
            tok = out.logits[:, -1].argmax(-1, keepdim=True)
        d1.record()
        torch.cuda.synchronize()
        return s0.elapsed_time(s1), (gen_len - 1) / (d0.elapsed_time(d1) / 1e3)


def _e2e_prompt(torch, model, S, dev):
    g = torch.Generator()
    g.manual_seed(S)
    return torch.randint(0, model.config.vocab_size, (1, S), generator=g).to(dev)


def _e2e_measure(torch, model, seq_lens, gen_len, trials, dev, tag, warmup=2):
    """{S: (mean TTFT ms, mean decode tok/s)} over `trials` runs after `warmup`."""
    res = {}
    for S in seq_lens:
        ids = _e2e_prompt(torch, model, S, dev)
        for _ in range(warmup):
            _e2e_run(torch, model, ids, gen_len)
        t = [_e2e_run(torch, model, ids, gen_len) for _ in range(trials)]
        res[S] = (statistics.mean(x[0] for x in t), statistics.mean(x[1] for x in t))
        log(f"  {tag} seq {S}: TTFT {res[S][0]:.2f} ms, decode {res[S][1]:.1f} tok/s")
    return res


def bench_e2e_compact(ctx, seq_lens=(128, 512, 1024, 2048), gen_len=32, trials=3):
    """The reference's Stage 3 end-to-end table (benchmarks/run_stage3_e2e.py:
    33-108, results in benchmarks/results/stage3_e2e.json:9-39) in the
    default bench run: TTFT and decode tokens/s at batch 1, 32 generated
    tokens, before and after patch_model_with_fused_kernels (57 RMSNorm, 28
    MLP replacements) on the same model instance, mean of `trials` runs after
    2 warm-up runs per sequence length."""
    torch = ctx.torch
    model = _e2e_model(torch, ctx.dev)
    for S in seq_lens:
        _e2e_run(torch, model, _e2e_prompt(torch, model, S, ctx.dev), 4)
    before = _e2e_measure(torch, model, seq_lens, gen_len, trials, ctx.dev, "e2e before")
    counts = ctx.pkg.patch_model_with_fused_kernels(model)
    after = _e2e_measure(torch, model, seq_lens, gen_len, trials, ctx.dev, "e2e after")
    del model
    torch.cuda.empty_cache()
    return {"model": "random-init Qwen2 (Qwen2.5-1.5B architecture), fp16, sdpa, batch 1", "gen_len": gen_len,
            "trials": trials, "patched": counts, "seq_len": list(seq_lens),
            "ttft_ms_before": [round(before[S][0], 2) for S in seq_lens],
            "ttft_ms_after": [round(after[S][0], 2) for S in seq_lens],
            "ttft_speedup": [round(before[S][0] / after[S][0], 3) for S in seq_lens],
            "decode_tok_s_before": [round(before[S][1], 1) for S in seq_lens],
            "decode_tok_s_after": [round(after[S][1], 1) for S in seq_lens],
            "decode_speedup": [round(after[S][1] / before[S][1], 3) for S in seq_lens]}


def bench_e2e(args):
    """TTFT and decode throughput before/after the module replacement, as the
    reference measures them (benchmarks/run_stage3_e2e.py:33-108 with
    src/engine/profiler.py:72-204): batch 1, uniform random prompts, event-
    timed prefill, event-timed greedy decode over HF's KV cache, mean of
    `trials` after `warmup` runs.  The model is a random-init Qwen2 with
    Qwen2.5-1.5B's architecture in fp16 (no Hub access here), sdpa attention."""
    import torch

    sys.path.insert(0, str(ROOT))
    pkg = importlib.import_module(PKG)
    dev = torch.device("cuda:0")
    model = _e2e_model(torch, dev)
    cfg = model.config

    def run(ids, gen_len):
        return _e2e_run(torch, model, ids, gen_len)

    def prompt(S):
        return _e2e_prompt(torch, model, S, dev)

    def measure(tag):
        return _e2e_measure(torch, model, args.seq_lens, args.gen_len, args.trials, dev, tag)

    def graphed_decode_tok_s(S=512, new=64, B=1):
        """Decode tokens/s (B per step) with the whole decode step replayed as
        one HIP graph (GraphedGreedyDecoder over a StaticCache)."""
        g = torch.Generator()
        g.manual_seed(4)
        ids = torch.randint(0, cfg.vocab_size, (B, S), generator=g).to(dev)
        dec = pkg.GraphedGreedyDecoder(model, B, S + new + 8)
        dec.generate(ids, new)  # capture
        times = []
        for _ in range(args.trials):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            dec.generate(ids, 2)
            torch.cuda.synchronize()
            t1 = time.perf_counter()
            dec.generate(ids, new)
            torch.cuda.synchronize()
            t2 = time.perf_counter()
            times.append(((t2 - t1) - (t1 - t0)) / (new - 2))  # subtract prefill + first step
        del dec
        torch.cuda.empty_cache()
        return B / statistics.median(times)

    def graphed(tag):
        r = {"b1": graphed_decode_tok_s(), "b8": graphed_decode_tok_s(B=8), "b32": graphed_decode_tok_s(B=32)}
        log(f"  {tag}, graphed decode (seq 512): batch 1 {r['b1']:.1f} tok/s, batch 8 {r['b8']:.1f} tok/s, "
            f"batch 32 {r['b32']:.1f} tok/s")
        return {k: round(v, 1) for k, v in r.items()}

    # warm every shape once before timing anything
    for S in args.seq_lens:
        run(prompt(S), 4)
    before = measure("before")
    graph_before = graphed("before")
    counts = pkg.patch_model_with_fused_kernels(model)
    log(f"patched {counts}")
    after = measure("after")
    graph_after = graphed("after")
    counts_fr = pkg.patch_model_with_fused_kernels(model, fuse_residual=True)
    log(f"fused residual {counts_fr}")
    fused_res = measure("after+fuse_residual")
    graph_fr = graphed("after+fuse_residual")
    # the same model with each FusedMLP's gate/up projections fused as well
    n_gu = 0
    for m in model.modules():
        if isinstance(m, pkg.FusedMLP) and m.gate_up_fusable():
            m.fuse_gate_up = True
            n_gu += 1
    log(f"fused gate/up in {n_gu} MLPs")
    fused_gu = measure("after+fuse_residual+fuse_gate_up")
    graph_gu = graphed("after+fuse_residual+fuse_gate_up")
    # ... and each FusedMLP's down projection on the HIP 16-bit linear for decode rows
    n_down = 0
    for m in model.modules():
        if isinstance(m, pkg.FusedMLP) and m.down_hip_capable():
            m.hip_down = True
            n_down += 1
    log(f"HIP down projection in {n_down} MLPs")
    hip_down = measure("after+fuse_residual+fuse_gate_up+hip_down")
    graph_hd = graphed("after+fuse_residual+fuse_gate_up+hip_down")
    rows = []
    for S in args.seq_lens:
        rows.append({"seq_len": S, "before_ttft_ms": round(before[S][0], 3), "after_ttft_ms": round(after[S][0], 3),
                     "ttft_speedup": round(before[S][0] / after[S][0], 4),
                     "before_decode_tok_s": round(before[S][1], 2), "after_decode_tok_s": round(after[S][1], 2),
                     "decode_speedup": round(after[S][1] / before[S][1], 4)})
    for row in rows:
        S = row["seq_len"]
        row["fuse_residual_ttft_ms"] = round(fused_res[S][0], 3)
        row["fuse_residual_decode_tok_s"] = round(fused_res[S][1], 2)
        row["fuse_gate_up_ttft_ms"] = round(fused_gu[S][0], 3)
        row["fuse_gate_up_decode_tok_s"] = round(fused_gu[S][1], 2)
        row["hip_down_ttft_ms"] = round(hip_down[S][0], 3)
        row["hip_down_decode_tok_s"] = round(hip_down[S][1], 2)
    print(json.dumps({"metric": "e2e TTFT / decode tok/s speedup from patch_model_with_fused_kernels",
                      "model": "random-init Qwen2 (Qwen2.5-1.5B architecture), fp16, sdpa, batch 1",
                      "gen_len": args.gen_len, "trials": args.trials, "patched": counts, "results": rows,
                      "fuse_gate_up_mlps": n_gu, "hip_down_mlps": n_down,
                      "graphed_decode_tok_s": {"seq_len": 512, "unpatched": graph_before, "patched": graph_after,
                                               "patched_fuse_residual": graph_fr,
                                               "patched_fuse_residual_fuse_gate_up": graph_gu,
                                               "patched_fuse_residual_fuse_gate_up_hip_down": graph_hd}}),
          flush=True)


def _int8_phases(torch, pkg, dev, S, GEN, TRIALS, batches, full):
    """fp16 vs int8 weights end to end on one model instance, after the
    reference's benchmarks/run_stage7_e2e.py: the model is measured in fp16,
    quantised in place with quantize_model_int8 (196 linears -> W8A16 HIP
    kernels) and measured again (with `full`, then also patched with the
    fused RMSNorm / SiLU-and-mul kernels, then with the int8 gate/up +
    SiLU-and-mul fused).  Per phase: transformer-layer weight MB; the HF path
    (eager decode over HF's KV cache) per batch -- TTFT, decode tok/s, peak
    memory -- for prompts of S tokens and GEN generated; and decode tok/s with
    the whole step replayed as one HIP graph (GraphedGreedyDecoder).
    Random-init Qwen2 with Qwen2.5-1.5B's architecture, fp16, sdpa."""
    model = _e2e_model(torch, dev)
    cfg = model.config

    def layer_weight_mb():
        total = 0
        for m in model.model.layers.modules():
            for t in list(m.parameters(recurse=False)) + list(m.buffers(recurse=False)):
                total += t.numel() * t.element_size()
        return total / 2**20

    def ids_for(B, seed):
        g = torch.Generator()
        g.manual_seed(seed)
        return torch.randint(0, cfg.vocab_size, (B, S), generator=g).to(dev)

    def hf_run(ids):
        with torch.inference_mode():
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats(dev)
            s0, s1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            d0, d1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s0.record()
            out = model(input_ids=ids, use_cache=True)
            past = out.past_key_values
            tok = out.logits[:, -1].argmax(-1, keepdim=True)
            s1.record()
            d0.record()
            for _ in range(GEN - 1):
                out = model(input_ids=tok, past_key_values=past, use_cache=True)
                past = out.past_key_values
                tok = out.logits[:, -1].argmax(-1, keepdim=True)
            d1.record()
            torch.cuda.synchronize()
            return (s0.elapsed_time(s1), ids.shape[0] * (GEN - 1) / (d0.elapsed_time(d1) / 1e3),
                    torch.cuda.max_memory_allocated(dev) / 2**20)

    def graphed_tok_s(B):
        ids = ids_for(B, 7)
        dec = pkg.GraphedGreedyDecoder(model, B, S + GEN + 8)
        dec.generate(ids, GEN)  # capture
        times = []
        for _ in range(TRIALS):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            dec.generate(ids, 2)
            torch.cuda.synchronize()
            t1 = time.perf_counter()
            dec.generate(ids, GEN)
            torch.cuda.synchronize()
            t2 = time.perf_counter()
            times.append(((t2 - t1) - (t1 - t0)) / (GEN - 2))
        del dec
        torch.cuda.empty_cache()
        return B / statistics.median(times)

    def phase(label):
        r = {"layer_weight_mb": round(layer_weight_mb(), 1), "hf": {}, "graphed_decode_tok_s": {}}
        for B in batches:
            ids = ids_for(B, 5)
            for _ in range(2):
                hf_run(ids)
            t = [hf_run(ids) for _ in range(TRIALS)]
            r["hf"][B] = {"ttft_ms": round(statistics.mean(x[0] for x in t), 3),
                          "decode_tok_s": round(statistics.mean(x[1] for x in t), 1),
                          "peak_mb": round(max(x[2] for x in t), 1)}
            r["graphed_decode_tok_s"][B] = round(graphed_tok_s(B), 1)
            log(f"  {label} batch {B}: TTFT {r['hf'][B]['ttft_ms']:.2f} ms, HF decode {r['hf'][B]['decode_tok_s']:.1f} "
                f"tok/s, peak {r['hf'][B]['peak_mb']:.0f} MB; graphed decode {r['graphed_decode_tok_s'][B]:.1f} tok/s")
        return r

    res = {"fp16": phase("fp16")}
    res["quantize_stats"] = pkg.quantize_model_int8(model)
    log(f"quantized {res['quantize_stats']}")
    res["int8"] = phase("int8")
    if full:
        res["patched"] = pkg.patch_model_with_fused_kernels(model, fuse_residual=True)
        log(f"patched {res['patched']}")
        res["int8_fused_kernels"] = phase("int8+fused")
        n_gu = 0
        for m in model.modules():
            if isinstance(m, pkg.FusedMLP) and m.gate_up_kind() == "int8":
                m.fuse_gate_up = True
                n_gu += 1
        log(f"int8 gate/up + SiLU-and-mul fused in {n_gu} MLPs")
        res["int8_fused_kernels_int8_gate_up"] = phase("int8+fused+int8_gate_up")
        res["int8_gate_up_mlps"] = n_gu
    del model
    torch.cuda.empty_cache()
    return res


def bench_e2e_int8(args):
    """fp16 vs int8 weights end to end (bench.py --e2e-int8): every phase of
    _int8_phases at batch 1 and 8, prompts of 128 tokens, 64 generated."""
    import torch

    sys.path.insert(0, str(ROOT))
    pkg = importlib.import_module(PKG)
    S, GEN = 128, 64
    res = _int8_phases(torch, pkg, torch.device("cuda:0"), S, GEN, args.trials, (1, 8), True)
    print(json.dumps({"metric": "fp16 vs int8-weight (W8A16) decode tok/s, after run_stage7_e2e.py",
                      "model": "random-init Qwen2 (Qwen2.5-1.5B architecture), fp16 activations, sdpa",
                      "seq_len": S, "gen_len": GEN, "trials": args.trials, **res}), flush=True)


def bench_e2e_int8_compact(ctx, S=128, GEN=32, trials=3):
    """The reference's Stage 7 end-to-end comparison (benchmarks/
    run_stage7_e2e.py, results in benchmarks/results/stage7_e2e.json) in the
    default bench run, compact: fp16 against int8 weights (W8A16 kernels) at
    batch 1 and 8 -- layer weight MB, TTFT, eager HF decode tok/s and
    hipGraph decode tok/s -- on one model instance."""
    r = _int8_phases(ctx.torch, ctx.pkg, ctx.dev, S, GEN, trials, (1, 8), False)
    out = {"model": "random-init Qwen2 (Qwen2.5-1.5B architecture), fp16 activations, sdpa", "seq_len": S,
           "gen_len": GEN, "trials": trials, "batch": [1, 8],
           "linears_quantized": r["quantize_stats"].get("layers_quantized")}
    for ph in ("fp16", "int8"):
        d = r[ph]
        out[ph] = {"layer_weight_mb": d["layer_weight_mb"],
                   "ttft_ms": [d["hf"][B]["ttft_ms"] for B in (1, 8)],
                   "decode_tok_s": [d["hf"][B]["decode_tok_s"] for B in (1, 8)],
                   "graphed_decode_tok_s": [d["graphed_decode_tok_s"][B] for B in (1, 8)],
                   "peak_mb": [d["hf"][B]["peak_mb"] for B in (1, 8)]}
    out["int8_over_fp16_graphed_decode"] = [round(out["int8"]["graphed_decode_tok_s"][i] /
                                                  out["fp16"]["graphed_decode_tok_s"][i], 3) for i in range(2)]
    return out

if __name__ == "__main__":
    main()
