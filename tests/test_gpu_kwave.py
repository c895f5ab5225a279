"""GPU parity of the fp32 contraction that splits K over the waves of one
workgroup (tile f32_kwave_32x32): few output tiles, both operands
K-contiguous.  Ragged tile edges, C dims, a non-affine row table, K over
several register batches, every touch kernel.  Checker: the CPU oracle (fp64
accumulation), relative Frobenius error <= 1e-5."""
import numpy as np
import pytest

import einsum_ir_amd as eir
from tests.test_gpu_contract import run_case

pytestmark = pytest.mark.gpu

KWAVE_SHAPES = [
    ("mk,nk->mn", dict(m=390, n=356, k=512)),          # ragged edges, BASELINE-1-like K
    ("cmk,cnk->cmn", dict(c=3, m=224, n=200, k=256)),   # C dims
    ("abk,nk->ban", dict(a=12, b=24, n=480, k=256)),    # kernel rows (b, a): non-affine A row table
    ("mk,nk->mn", dict(m=400, n=360, k=4096)),          # four register batches per wave
    ("abkl,cdkl->abcd", dict(a=32, b=16, c=32, d=16, k=32, l=16)),
]


@pytest.mark.parametrize("expr,sizes", KWAVE_SHAPES)
def test_kwave_layouts(torch_cuda, oracle, expr, sizes):
    _, desc = run_case(torch_cuda, oracle, expr, sizes, seed=31)
    assert "f32_kwave_32x32" in desc, desc


@pytest.mark.parametrize("first,last", [(eir.COPY, eir.UNDEFINED_KTYPE), (eir.ADD, eir.UNDEFINED_KTYPE),
                                        (eir.UNDEFINED_KTYPE, eir.UNDEFINED_KTYPE), (eir.ZERO, eir.RELU),
                                        (eir.COPY, eir.RELU), (eir.ZERO, eir.ADD)])
def test_kwave_touch_kernels(torch_cuda, oracle, first, last):
    _, desc = run_case(torch_cuda, oracle, "mk,nk->mn", dict(m=390, n=356, k=256), first=first, last=last,
                       seed=37)
    assert "f32_kwave_32x32" in desc, desc


def test_kwave_matches_split_k(torch_cuda, oracle, monkeypatch):
    """The same contraction through the workgroup K split and through split K."""
    got_w, desc_w = run_case(torch_cuda, oracle, "mk,nk->mn", dict(m=256, n=512, k=1024), seed=41)
    monkeypatch.setenv("ETIR_NO_KWAVE", "1")
    got_s, desc_s = run_case(torch_cuda, oracle, "mk,nk->mn", dict(m=256, n=512, k=1024), seed=41)
    assert "kwave" in desc_w and "kwave" not in desc_s, (desc_w, desc_s)
    assert np.linalg.norm(got_w - got_s) / np.linalg.norm(got_s) <= 1e-5


@pytest.mark.parametrize("m,n,k", [(64, 64, 96), (128, 100, 112), (33, 47, 240), (256, 256, 256), (1, 33, 304),
                                   (100, 100, 496), (128, 128, 512)])
def test_kwave_few_tiles(torch_cuda, oracle, m, n, k):
    """Few tiles and a K of 96 to 512: waves whose K range is short or empty."""
    _, desc = run_case(torch_cuda, oracle, "mk,nk->mn", dict(m=m, n=n, k=k), seed=k)
    assert m == 1 or "f32_kwave_32x32" in desc, desc


@pytest.mark.parametrize("n,k,taken", [(512, 96, True), (544, 96, False), (544, 112, True)])
def test_kwave_short_k_takes_one_round(torch_cuda, oracle, n, k, taken):
    """256 and 272 tiles: with a K of 96 no second workgroup per CU."""
    _, desc = run_case(torch_cuda, oracle, "mk,nk->mn", dict(m=512, n=n, k=k), seed=k)
    assert ("f32_kwave_32x32" in desc) == taken, desc
