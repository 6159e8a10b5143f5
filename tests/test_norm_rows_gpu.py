"""Norms whose rows stay in registers (norm.hip): row lengths around what a thread holds and
past it, in place and not, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hidden", [8, 1024, 1032, 2040, 2048, 2056, 4096, 4104, 8192, 8200])
@pytest.mark.parametrize("rows", [1, 65])
def test_rows(dtype, hidden, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(hidden + rows)
    x, r = (torch.randn((rows, hidden), generator=g, device="cuda").to(dtype) for _ in "xr")
    w = torch.randn(hidden, generator=g, device="cuda").to(dtype)

    def check(got, value):
        want = value.double() * torch.rsqrt(value.double().square().mean(-1, keepdim=True) + 1e-5)
        want = want * w.double()
        # one rounding of the result, float32 arithmetic before it
        unit = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 2 ** -20}[dtype]
        assert ((got.double() - want).abs() <= unit * want.abs() + 1e-7).all()

    check(ops.rms_norm(x, w, 1e-5), x)
    summed = (x.float() + r.float()).to(dtype)
    normed, residual = ops.fused_add_rms_norm(x.clone(), r.clone(), w, 1e-5)
    assert torch.equal(residual, summed)
    check(normed, summed)


# more rows, without a sum, have two or four vectors a thread
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hidden", [1024, 1032, 2056, 4096, 4104, 8192])
@pytest.mark.parametrize("rows", [768, 769])
def test_many_rows(dtype, hidden, rows):
    test_rows(dtype, hidden, rows)
