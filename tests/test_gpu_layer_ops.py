"""Residual add + RMSNorm and the SwiGLU product against float64: results
within one rounding of the dtype (silu's product two), the residual sum bit-exact."""
import pytest
import torch

from nanopd_amd import paged_kernels as pk

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # unit roundoff


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 1536), (37, 2048), (527, 4096), (5, 2056),
                                        (2, 8192), (4, 8200), (3, 100)])
@pytest.mark.parametrize("add", [False, True])
def test_add_rms_norm(device, dtype, rows, width, add):
    """One to four chunks per thread, a part-full last one; 8200 and 100
    columns take the torch operations."""
    print(f"add_rms_norm {rows}x{width} {dtype} add={add}", flush=True)
    g = torch.Generator(device=device).manual_seed(width + rows)
    x = (torch.randn(rows, width, generator=g, device=device) * 3).to(dtype)
    d = torch.randn(rows, width, generator=g, device=device).to(dtype) if add else None
    w = (1 + 0.2 * torch.randn(width, generator=g, device=device)).to(dtype)
    want_x = x + d if add else x.clone()
    got = pk.add_rms_norm(x, d, w, 1e-6)
    assert torch.equal(x, want_x)
    xd = want_x.double()
    want = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    # one rounding to nearest, on top of a few fp32 ones
    assert ((got.double() - want).abs() <= (U[dtype] * 1.01) * want.abs() + 1e-7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 8960), (77, 328), (527, 12288), (2, 12)])
def test_silu_mul(device, dtype, rows, width):
    print(f"silu_mul {rows}x{width} {dtype}", flush=True)
    g = torch.Generator(device=device).manual_seed(width)
    gu = (torch.randn(rows, 2 * width, generator=g, device=device) * 4).to(dtype)
    gu[0, :4] = torch.tensor([0.0, -60.0, 60.0, float("inf")], device=device).to(dtype)
    gu[0, width:width + 4] = 1.0
    got = pk.silu_mul(gu)
    gate, up = gu[:, :width].double(), gu[:, width:].double()
    want = gate * torch.sigmoid(gate) * up
    assert torch.isinf(got[0, 3]) and got[0, 3] > 0
    fin = torch.isfinite(want)
    # silu is rounded before the product: two roundings, each of relative error
    # u or, below the normal range (fp16 from 2^-14 down), half the subnormal
    # spacing -- the first one times |up|
    half = 2.0 ** -25 if dtype == torch.float16 else 2.0 ** -134
    err = (got.double() - want).abs()[fin]
    assert (err <= U[dtype] * 2.01 * want.abs()[fin] + half * 1.01 * (up.abs()[fin] + 1)).all()
    nan = torch.full((1, 16), float("nan"), dtype=dtype, device=device)
    assert pk.silu_mul(nan).isnan().all()


def test_silu_of_far_negative_gates(device):
    """Gates down to -88.5, where 1 / (1 + e^88) is no normal fp32 number but
    silu(-88) = -5.3e-37 is a bf16 one: two roundings, as above."""
    g = torch.arange(-88.5, -80.0, 0.5, device=device)[:16].to(torch.bfloat16)
    gu = torch.cat([g, torch.ones_like(g)]).view(1, 32)
    got = pk.silu_mul(gu)[0].double()
    want = g.double() * torch.sigmoid(g.double())
    assert (got != 0).all()
    # (and fp32's exponential of 128 log2 units: 128 * 2^-24 * ln 2 of the value)
    assert ((got - want).abs() <= (U[torch.bfloat16] * 2.01 + 1e-5) * want.abs()).all()
