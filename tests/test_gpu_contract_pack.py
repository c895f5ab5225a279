"""Contractions whose operands are copied K-contiguous before the kernel runs
(the planner's choice for large operands that it would otherwise gather
element by element): odd extents, conflicting K orders, batches, touch
kernels, several streams, and stream capture (which reads them in place).

Checker: torch.einsum in 64 bits on the same values.  Bars: fp32 1e-5 and
bf16 2e-3 relative Frobenius (fp32 sums of exact products), fp64 1e-12.
"""
import ctypes
import threading

import pytest

import einsum_ir_amd as eir
from tests.helpers import TOL_BF16, TOL_FP32, TOL_FP64

pytestmark = pytest.mark.gpu

EIR = {"float32": eir.FP32, "bfloat16": eir.BF16, "float64": eir.FP64}
TOL = {"float32": TOL_FP32, "bfloat16": TOL_BF16, "float64": TOL_FP64}


def _operands(torch, expr, sizes, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    ins, out = expr.split("->")
    shape = lambda t: [sizes[d] for d in t]  # noqa: E731
    a, b = ((torch.rand(shape(t), device="cuda", generator=g) * 2 - 1).to(getattr(torch, dtype))
            for t in ins.split(","))
    return a, b, shape(out)


def _plan(expr, sizes, dtype, **kw):
    lp = eir.binary_loops(expr, sizes)
    dt = EIR[dtype]
    comp = eir.FP64 if dtype == "float64" else eir.FP32
    return eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                               lp["strides_out"], dtype_left=dt, dtype_right=dt, dtype_comp=comp, dtype_out=comp,
                               **kw)


def _error(ref, got):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("expr,sizes", [
    ("mk,nk->mn", dict(m=767, n=769, k=773)),                       # padded to 776 a row
    ("km,kn->mn", dict(m=1021, n=767, k=769)),
    ("km,nk->nm", dict(m=767, n=1023, k=1025)),                     # roles swapped, one past a vector
    ("zakm,zbkn->zabmn", dict(z=3, a=31, m=21, b=23, n=37, k=517)),  # batch, split rows
    ("kzml,nlzk->zmn", dict(z=2, m=901, n=703, k=37, l=29)),        # two K dims, opposite orders
    ("aecf,bfde->abcd", dict(a=50, b=50, c=26, d=26, e=24, f=28)),  # K orders conflict
])
def test_packed(torch_cuda, expr, sizes, dtype):
    torch = torch_cuda
    a, b, shape = _operands(torch, expr, sizes, dtype, 7)
    out = torch.full(shape, float("nan"), device="cuda")
    plan = _plan(expr, sizes, dtype)
    assert "packed" in plan.describe(), plan.describe()
    for _ in range(2):
        plan.execute(a, b, out, stream=torch.cuda.current_stream())
    assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL[dtype]
    plan.close()


@pytest.mark.parametrize("expr,sizes,dtype", [
    ("mk,nk->mn", dict(m=767, n=769, k=773), "bfloat16"),               # 776 = 8 x 97
    ("mk,nk->mn", dict(m=1021, n=1023, k=1041), "bfloat16"),            # 1048 = 8 x 131
    ("eafd,fbec->abcd", dict(a=10, d=9, c=75, b=64, f=39, e=61), "bfloat16"),   # 2384 = 16 x 149
    ("abkl,cdkl->abcd", dict(a=31, b=8, d=13, c=24, k=92, l=61), "float32"),
])
def test_packed_kernels_load_vectors(torch_cuda, expr, sizes, dtype):
    """Where K of the copies is split, the parts keep the vector loads that the
    copies are made for."""
    torch = torch_cuda
    a, b, shape = _operands(torch, expr, sizes, dtype, 17)
    out = torch.full(shape, float("nan"), device="cuda")
    plan = _plan(expr, sizes, dtype)
    desc = plan.describe()
    assert " | packed" not in desc or "scalar" not in desc.split(" | packed")[1], desc
    plan.execute(a, b, out, stream=torch.cuda.current_stream())
    assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL[dtype]
    plan.close()


def test_packed_fp64_and_unaligned(torch_cuda):
    """fp64 with conflicting K orders; operands one element off alignment."""
    torch = torch_cuda
    expr, sizes = "aecf,bfde->abcd", dict(a=48, b=48, c=24, d=24, e=24, f=25)
    a, b, shape = _operands(torch, expr, sizes, "float64", 8)
    out = torch.full(shape, float("nan"), device="cuda", dtype=torch.float64)
    plan = _plan(expr, sizes, "float64")
    assert "packed" in plan.describe(), plan.describe()
    off = [torch.empty(x.numel() + 1, device="cuda", dtype=x.dtype)[1:].view_as(x).copy_(x) for x in (a, b)]
    plan.execute(off[0], off[1], out, stream=torch.cuda.current_stream())
    assert _error(torch.einsum(expr, a, b), out) <= TOL_FP64
    plan.close()


def test_packed_touch_kernels(torch_cuda):
    """First touch ADD (out + aux + sum), last touch RELU."""
    torch = torch_cuda
    expr, sizes = "km,kn->mn", dict(m=767, n=769, k=773)
    a, b, shape = _operands(torch, expr, sizes, "float32", 9)
    out0, aux = torch.randn(shape, device="cuda"), torch.randn(shape, device="cuda")
    out = out0.clone()
    plan = _plan(expr, sizes, "float32", ktype_first_touch=eir.ADD, ktype_last_touch=eir.RELU)
    assert "packed" in plan.describe(), plan.describe()
    plan.execute(a, b, out, aux=aux, stream=torch.cuda.current_stream())
    ref = torch.relu(torch.einsum(expr, a.double(), b.double()) + out0.double() + aux.double())
    assert _error(ref, out) <= TOL_FP32
    plan.close()


def test_packed_on_several_streams(torch_cuda):
    """One plan, other inputs on each of three streams in turn, nothing waited
    for in between: each execution has the copies to itself."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=1023, n=1021, k=1019)
    plan = _plan(expr, sizes, "float32")
    assert "packed" in plan.describe(), plan.describe()
    sets = [_operands(torch, expr, sizes, "float32", 20 + i) for i in range(6)]
    outs = [torch.full(s[2], float("nan"), device="cuda") for s in sets]
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for i, (a, b, _) in enumerate(sets):
        plan.execute(a, b, outs[i], stream=streams[i % 3])
    torch.cuda.synchronize()
    for (a, b, _), out in zip(sets, outs):
        assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL_FP32
    plan.close()


def test_packed_padding_is_cleared_before_the_first_execution(torch_cuda):
    """Rows padded from 1019 to 1020: the first execution, on a stream that does
    not wait for the null stream, follows the plan's creation with nothing
    waited for in between, in memory that held NaN before."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=1023, n=1021, k=1019)
    lib = eir.hip_lib()
    a, b, shape = _operands(torch, expr, sizes, "float32", 40)
    ref = torch.einsum(expr, a.double(), b.double())
    outs = [torch.full(shape, float("nan"), device="cuda") for _ in range(4)]
    stream = ctypes.c_void_p()
    eir.check(lib.etir_hip_stream_create(ctypes.byref(stream)))
    for out in outs:
        # the workspace is likely to be this block again
        block = ctypes.c_void_p()
        eir.check(lib.etir_hip_malloc(ctypes.byref(block), 4 * 1020 * (1023 + 1021)))
        eir.check(lib.etir_hip_memset(block, 0xff, 4 * 1020 * (1023 + 1021)))
        torch.cuda.synchronize()
        eir.check(lib.etir_hip_free(block))
        plan = _plan(expr, sizes, "float32")
        plan.execute(a, b, out, stream=stream.value)
        assert "packed" in plan.describe(), plan.describe()
        eir.synchronize(stream.value)
        plan.close()
    eir.check(lib.etir_hip_stream_destroy(stream))
    for out in outs:
        assert _error(ref, out) <= TOL_FP32


def test_copies_leave_memory_free(torch_cuda):
    """With 512 MB of device memory left, 134 MB of copies are not taken."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=4095, n=4093, k=4091)
    lib = eir.hip_lib()
    _plan("mk,nk->mn", dict(m=16, n=16, k=16), "float32").close()
    torch.cuda.empty_cache()
    blocks = []
    try:
        while (take := torch.cuda.mem_get_info()[0] - (512 << 20)) >= 4 << 20:
            block = ctypes.c_void_p()
            eir.check(lib.etir_hip_malloc(ctypes.byref(block), min(take, 32 << 30)))
            blocks.append(block)
        full = _plan(expr, sizes, "float32")
        left = torch.cuda.mem_get_info()[0]
    finally:
        for block in blocks:
            eir.check(lib.etir_hip_free(block))
    assert "packed" not in full.describe(), full.describe()
    assert left >= 500 << 20, left
    full.close()
    plan = _plan(expr, sizes, "float32")
    assert "packed" in plan.describe(), plan.describe()
    plan.close()


@pytest.mark.parametrize("own_streams", [False, True])
def test_packed_from_several_threads(torch_cuda, own_streams):
    """Three host threads on one plan, on the null stream or on streams of
    their own: the copies and the kernel of an execution stay together."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=1023, n=1021, k=1019)
    plan = _plan(expr, sizes, "float32")
    assert "packed" in plan.describe(), plan.describe()
    sets = [[_operands(torch, expr, sizes, "float32", 60 + 10 * t + i) for i in range(3)] for t in range(3)]
    outs = [[torch.full(s[2], float("nan"), device="cuda") for s in x] for x in sets]
    streams = [torch.cuda.Stream() if own_streams else None for _ in range(3)]
    torch.cuda.synchronize()

    def work(t):
        for (a, b, _), out in zip(sets[t], outs[t]):
            plan.execute(a, b, out, stream=streams[t])

    threads = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for x, y in zip(sets, outs):
        for (a, b, _), out in zip(x, y):
            assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL_FP32
    plan.close()


def test_packed_on_a_recycled_stream(torch_cuda):
    """A stream destroyed with an execution in flight; the next one may get its
    handle and still waits for that execution."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=2047, n=2045, k=2043)
    lib = eir.hip_lib()
    plan = _plan(expr, sizes, "float32")
    assert "packed" in plan.describe(), plan.describe()
    sets = [_operands(torch, expr, sizes, "float32", 50 + i) for i in range(4)]
    outs = [torch.full(s[2], float("nan"), device="cuda") for s in sets]
    torch.cuda.synchronize()
    for (a, b, _), out in zip(sets, outs):
        stream = ctypes.c_void_p()
        eir.check(lib.etir_hip_stream_create(ctypes.byref(stream)))
        plan.execute(a, b, out, stream=stream.value)
        eir.check(lib.etir_hip_stream_destroy(stream))
    torch.cuda.synchronize()
    for (a, b, _), out in zip(sets, outs):
        assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL_FP32
    plan.close()


def test_packed_plan_under_capture(torch_cuda):
    """A captured execution reads its operands in place: replays, with eager
    executions of the same plan on another stream between them, stay right."""
    torch = torch_cuda
    expr, sizes = "mk,nk->mn", dict(m=767, n=769, k=773)
    plan = _plan(expr, sizes, "float32")
    assert "packed" in plan.describe(), plan.describe()
    a, b, shape = _operands(torch, expr, sizes, "float32", 30)
    c, d, _ = _operands(torch, expr, sizes, "float32", 31)
    out, other = torch.empty(shape, device="cuda"), torch.empty(shape, device="cuda")
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        plan.execute(a, b, out, stream=side)
    for i in range(3):
        a.mul_(-0.5)
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        plan.execute(c, d, other, stream=side)
        torch.cuda.synchronize()
        assert _error(torch.einsum(expr, a.double(), b.double()), out) <= TOL_FP32
        assert _error(torch.einsum(expr, c.double(), d.double()), other) <= TOL_FP32
    plan.close()
