"""The one-step form of the fp32 direct-to-LDS kernel (K up to 32, plain
output): every pairing of the vector modes, edge tiles, k past the last
fragment, ReLU, an output off alignment, and outputs of short unit-stride
runs written by whole runs (read in place or from packed copies).

Checker: torch.einsum in 64 bits; fp32 bar 1e-5 relative Frobenius.
"""
import pytest

import einsum_ir_amd as eir
from tests.helpers import TOL_FP32

pytestmark = pytest.mark.gpu


def _run(torch, expr, sizes, offset=0, **kw):
    g = torch.Generator(device="cuda").manual_seed(sum(sizes.values()))
    ins, out = expr.split("->")
    shape = lambda t: [sizes[d] for d in t]  # noqa: E731
    a, b = (torch.rand(shape(t), device="cuda", generator=g) * 2 - 1 for t in ins.split(","))
    lp = eir.binary_loops(expr, sizes)
    plan = eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                               lp["strides_out"], **kw)
    ref = torch.einsum(expr, a.double(), b.double())
    c = torch.full((ref.numel() + offset + 1024,), float("nan"), device="cuda")
    plan.execute(a, b, c[offset:], stream=torch.cuda.current_stream())
    desc = plan.describe()
    plan.close()
    got = c[offset:offset + ref.numel()].view(ref.shape)
    assert bool(c[:offset].isnan().all()) and bool(c[offset + ref.numel():].isnan().all()), "written past the output"
    return ref, got, desc


def _error(ref, got):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("expr,sizes", [
    ("mk,nk->mn", dict(m=2040, n=2048, k=32)),
    ("km,kn->mn", dict(m=2044, n=2016, k=9)),
    ("km,nk->mn", dict(m=2044, n=2272, k=20)),
    ("mk,kn->mn", dict(m=2303, n=1920, k=4)),
    ("zmk,zkn->zmn", dict(z=5, m=1020, n=1024, k=24)),
])
@pytest.mark.parametrize("relu", [False, True])
def test_one_step(torch_cuda, expr, sizes, relu):
    kw = dict(ktype_last_touch=eir.RELU) if relu else {}
    ref, got, desc = _run(torch_cuda, expr, sizes, **kw)
    assert "one_step" in desc, desc
    assert _error(torch_cuda.relu(ref) if relu else ref, got) <= TOL_FP32


@pytest.mark.parametrize("expr,sizes,run", [
    # rows (m, e), columns (n, f): [m][n][e][f], f the run; row-contiguous left, K-contiguous right
    ("kme,nfk->mnef", dict(m=16, e=127, n=102, f=20, k=24), 20),   # rows past a tile in one m, 128 - 8 columns a tile
    ("kme,nfk->mnef", dict(m=12, e=160, n=130, f=28, k=32), 28),   # 112 columns a tile, a part tile of columns
    ("kme,nfk->mnef", dict(m=8, e=255, n=255, f=8, k=8), 8),       # 128 columns a tile
    ("kme,nfk->mnef", dict(m=10, e=200, n=180, f=12, k=28), 12),
])
@pytest.mark.parametrize("offset", [0, 1])
def test_runs(torch_cuda, expr, sizes, run, offset):
    ref, got, desc = _run(torch_cuda, expr, sizes, offset=offset)
    assert ("one_step runs=%d" % run) in desc, desc
    assert _error(ref, got) <= TOL_FP32


def test_runs_of_packed_operands(torch_cuda):
    """Six free modes, both operands copied: rows (a, d, e), columns (b, c, f)."""
    sizes = dict(a=24, b=20, c=20, d=24, e=20, f=20, g=24)
    ref, got, desc = _run(torch_cuda, "dega,gfbc->abcdef", sizes, ktype_last_touch=eir.RELU)
    assert "packed" in desc and "runs=20" in desc, desc
    assert _error(torch_cuda.relu(ref), got) <= TOL_FP32
