"""The 128 x 128 direct-to-LDS bf16 tile (two workgroups per CU) and the
16-byte bf16 stores: every pairing of the vector modes, edge tiles, k steps
cut short, touch kernels, and values a rounding could lose.

Checker: torch in 64 bits on the same values.  Bars: fp32 results 1e-5, bf16
results 2^-8 (half a unit in the last place of 8 bits is 2^-9) relative
Frobenius.
"""
import pytest

import einsum_ir_amd as eir

pytestmark = pytest.mark.gpu


def _run(torch, expr, sizes, out_dtype, a=None, offset=0, **kw):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes.values()))
    ins, out = expr.split("->")
    left, right = ins.split(",")
    shape = lambda t: [sizes[d] for d in t]  # noqa: E731
    if a is None:
        a = (torch.rand(shape(left), device="cuda", generator=g) * 2 - 1).bfloat16()
    b = (torch.rand(shape(right), device="cuda", generator=g) * 2 - 1).bfloat16()
    lp = eir.binary_loops(expr, sizes)
    plan = eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                               lp["strides_out"], dtype_left=eir.BF16, dtype_right=eir.BF16,
                               dtype_out=eir.BF16 if out_dtype == torch.bfloat16 else eir.FP32, **kw)
    n = 1
    for d in out:
        n *= sizes[d]
    c = torch.full((n + offset,), float("nan"), device="cuda", dtype=out_dtype)[offset:].view(shape(out))
    plan.execute(a, b, c, stream=torch.cuda.current_stream())
    desc = plan.describe()
    plan.close()
    return torch.einsum(expr, a.double(), b.double()), c, desc


def _error(ref, got):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("bf16_out", [False, True])
@pytest.mark.parametrize("expr,sizes", [
    ("mk,nk->mn", dict(m=2049, n=2056, k=72)),     # one row past a tile, a k step of 8
    ("mk,kn->mn", dict(m=1921, n=2176, k=64)),     # one k step
    ("km,kn->mn", dict(m=2040, n=2184, k=200)),
    ("km,nk->mn", dict(m=2056, n=2043, k=136)),    # an odd number of columns: no 16-byte stores
    ("zakm,zbkn->zabmn", dict(z=3, a=32, b=40, m=40, n=32, k=56)),  # batch, 32-column runs, k below one step
    ("zmk,znk->zmn", dict(z=5, m=900, n=904, k=104)),
])
def test_dma_128x128(torch_cuda, expr, sizes, bf16_out):
    torch = torch_cuda
    ref, got, desc = _run(torch, expr, sizes, torch.bfloat16 if bf16_out else torch.float32)
    assert "bf16_dma_128x128" in desc, desc
    assert _error(ref, got) <= (2 ** -8 if bf16_out else 1e-5)


@pytest.mark.parametrize("sizes,bf16_out,kw", [
    (dict(m=4072, n=4088, k=8192), False, {}),     # one ragged tile per CU
    (dict(m=4096, n=4064, k=8200), True, {}),      # a last k step of 8
    (dict(m=4096, n=4096, k=8192), False, dict(ktype_last_touch=eir.RELU)),
    (dict(m=8184, n=4096, k=4096), True, {}),      # two rounds from a K of 4096 on
])
def test_dma_256x256_long_k(torch_cuda, sizes, bf16_out, kw):
    """Row-contiguous operands with a long K that the persistent loop does not take."""
    torch = torch_cuda
    ref, got, desc = _run(torch, "km,kn->mn", sizes, torch.bfloat16 if bf16_out else torch.float32, **kw)
    assert "bf16_dma_256x256" in desc and "persistent" not in desc, desc
    ref = torch.relu(ref) if kw else ref
    assert _error(ref, got) <= (2 ** -8 if bf16_out else 1e-5)


def test_bf16_stores_relu_and_unaligned(torch_cuda):
    """ReLU in the 16-byte stores, and an output one element off alignment
    (element stores)."""
    torch = torch_cuda
    sizes = dict(m=2049, n=2056, k=72)
    ref, got, _ = _run(torch, "mk,nk->mn", sizes, torch.bfloat16, ktype_last_touch=eir.RELU)
    assert _error(torch.relu(ref), got) <= 2 ** -8
    ref, off, _ = _run(torch, "mk,nk->mn", sizes, torch.bfloat16, offset=1)
    assert _error(ref, off) <= 2 ** -8


def test_bf16_stores_of_special_values(torch_cuda):
    """Rows of infinities, NaN, values that round up to infinity and results
    below bf16's normal range come out as torch rounds the fp32 results."""
    torch = torch_cuda
    sizes = dict(m=2048, n=2048, k=64)
    a = torch.zeros(2048, 64, device="cuda")
    a[0::5, 0] = float("inf")
    a[1::5, 0] = float("nan")
    a[2::5, 0] = 3.38e38
    a[3::5, 0] = 1e-39
    a[4::5, 0] = 1.0
    b = torch.zeros(2048, 64, device="cuda").bfloat16()
    b[:, 0] = torch.linspace(0.5, 1.5, 2048, device="cuda").bfloat16()
    outs = []
    for dt in (torch.float32, torch.bfloat16):
        lp = eir.binary_loops("mk,nk->mn", sizes)
        plan = eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                                   lp["strides_out"], dtype_left=eir.BF16, dtype_right=eir.BF16,
                                   dtype_out=eir.BF16 if dt == torch.bfloat16 else eir.FP32)
        c = torch.empty(2048, 2048, device="cuda", dtype=dt)
        plan.execute(a.bfloat16(), b, c, stream=torch.cuda.current_stream())
        outs.append(c)
        plan.close()
    assert torch.equal(torch.nan_to_num(outs[0].bfloat16().float(), nan=7.0), torch.nan_to_num(outs[1].float(), nan=7.0))
