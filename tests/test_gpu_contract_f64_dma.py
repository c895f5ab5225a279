"""The fp64 direct-to-LDS kernel (both operands K-contiguous, 128 x 128 tiles):
edge tiles, k steps cut short, batches, every touch kernel, operands off
alignment (register-staged fallback), and packed operands that reach it.

Checker: torch.einsum in float64, whose sums differ in order only; bar 1e-12.
"""
import pytest

import einsum_ir_amd as eir
from tests.helpers import TOL_FP64

pytestmark = pytest.mark.gpu


def _case(torch, expr, sizes, first=eir.ZERO, last=eir.UNDEFINED_KTYPE, offset=0):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes.values()))
    ins, out = expr.split("->")
    rand = lambda t: torch.rand([sizes[d] for d in t], device="cuda", generator=g, dtype=torch.float64) * 2 - 1  # noqa: E731
    a, b = (rand(t) for t in ins.split(","))
    c, aux = rand(out), rand(out)
    lp = eir.binary_loops(expr, sizes)
    plan = eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                               lp["strides_out"], dtype_left=eir.FP64, dtype_right=eir.FP64, dtype_comp=eir.FP64,
                               dtype_out=eir.FP64, ktype_first_touch=first, ktype_last_touch=last)
    ref = torch.einsum(expr, a, b)
    if first in (eir.ADD, eir.UNDEFINED_KTYPE):
        ref = ref + c
    if first in (eir.ADD, eir.COPY):
        ref = ref + aux
    if last == eir.RELU:
        ref = torch.relu(ref)
    elif last == eir.ADD:
        ref = ref + aux
    if first in (eir.ZERO, eir.COPY):
        c.fill_(float("nan"))
    if offset:
        a = torch.empty(a.numel() + offset, device="cuda", dtype=a.dtype)[offset:].view_as(a).copy_(a)
    plan.execute(a, b, c, aux=aux, stream=torch.cuda.current_stream())
    desc = plan.describe()
    plan.close()
    return float((c - ref).norm() / ref.norm()), desc


@pytest.mark.parametrize("expr,sizes", [
    ("mk,nk->mn", dict(m=2047, n=2033, k=34)),       # a row short of 16 tiles, 2 k in the last step
    ("mk,nk->mn", dict(m=2048, n=2048, k=2)),        # one step, nearly empty
    ("mk,nk->mn", dict(m=2040, n=2048, k=48)),
    ("zmk,znk->zmn", dict(z=5, m=1000, n=1020, k=22)),
    ("nk,mk->mn", dict(m=2040, n=2044, k=30)),       # roles swapped
    ("amk,nk->amn", dict(a=3, m=701, n=2047, k=18)),
])
def test_f64_dma(torch_cuda, expr, sizes):
    err, desc = _case(torch_cuda, expr, sizes)
    assert "f64_dma_128x128x16" in desc, desc
    assert err <= TOL_FP64


@pytest.mark.parametrize("m,n,k,taken", [
    (2544, 1539, 66, False),     # 2 rounds of 128 x 128 tiles against 4 of 64 x 64
    (2544, 1539, 64, True),
    (2047, 2033, 66, True),      # 1 against 4
    (3000, 2590, 98, True),      # 2 (504 tiles) against 8
    (3000, 2689, 98, False),     # 3 (528) against 8
])
def test_f64_tile_rounds(torch_cuda, m, n, k, taken):
    err, desc = _case(torch_cuda, "mk,nk->mn", dict(m=m, n=n, k=k))
    assert ("f64_dma_128x128x16" in desc) == taken, desc
    assert err <= TOL_FP64


@pytest.mark.parametrize("first,last", [(eir.COPY, eir.UNDEFINED_KTYPE), (eir.ADD, eir.RELU),
                                        (eir.UNDEFINED_KTYPE, eir.ADD), (eir.ZERO, eir.RELU)])
def test_f64_dma_touch_kernels(torch_cuda, first, last):
    err, desc = _case(torch_cuda, "mk,nk->mn", dict(m=2047, n=2033, k=34), first=first, last=last)
    assert "f64_dma_128x128x16" in desc, desc
    assert err <= TOL_FP64


def test_f64_unaligned_operand(torch_cuda):
    err, _ = _case(torch_cuda, "mk,nk->mn", dict(m=2047, n=2033, k=34), offset=1)
    assert err <= TOL_FP64


def test_f64_packed(torch_cuda):
    """Conflicting K orders: both operands copied, rows padded to 16 bytes."""
    err, desc = _case(torch_cuda, "aecf,bfde->abcd", dict(a=48, b=46, c=43, d=44, e=41, f=39))
    assert "packed" in desc and "f64_dma" in desc, desc
    assert err <= TOL_FP64
