"""Which layer_ops calls reach a launch, without a GPU: CPU tensors that report
themselves as CUDA ones, and a recorder in the place of the library call. A call
that a launch would take out of a tensor's bounds has to go to the torch
operations, which refuse it."""
import pytest
import torch

from nanopd_amd import paged_kernels as pk


class OnGpu(torch.Tensor):
    """A CPU tensor that says it is on GPU `gpu`."""
    gpu = 0
    is_cuda = property(lambda self: True)

    def get_device(self):
        return self.gpu


def on_gpu(*shape, dtype=torch.bfloat16, gpu=0):
    t = torch.ones(*shape, dtype=dtype).as_subclass(OnGpu)
    t.gpu = gpu
    return t


@pytest.fixture
def launches(monkeypatch):
    calls = []
    monkeypatch.setattr(pk._lib, "call", lambda name, *args: calls.append((name, args)))
    monkeypatch.setattr(pk, "_stream", lambda dev: 0)
    return calls


def test_add_rms_norm_launches_what_fits(launches):
    x, d, w = on_gpu(2, 4096), on_gpu(2, 4096), on_gpu(4096)
    pk.add_rms_norm(x, d, w, 1e-6)
    pk.add_rms_norm(x, None, w, 1e-6)
    assert [c[0] for c in launches] == ["npd_add_rms_norm"] * 2


@pytest.mark.parametrize("shape", [(2048,), (8192,), (1, 4096), (4096, 1), (8,)])
def test_add_rms_norm_refuses_a_weight_of_another_shape(launches, shape):
    """The kernel reads x.size(1) weights: 4096 from a tensor of 2048 are 4 KB
    past its end."""
    with pytest.raises(RuntimeError):
        pk.add_rms_norm(on_gpu(2, 4096), None, on_gpu(*shape), 1e-6)
    assert not launches


@pytest.mark.parametrize("which", ["weight", "delta"])
def test_add_rms_norm_launches_nothing_across_gpus(launches, which):
    x = on_gpu(2, 64)
    w, d = on_gpu(64, gpu=which == "weight"), on_gpu(2, 64, gpu=which == "delta")
    pk.add_rms_norm(x, d, w, 1e-6)   # (the torch operations refuse real tensors of two GPUs)
    assert not launches


def test_no_launch_records_a_gradient_or_takes_nothing(launches):
    w = on_gpu(64).requires_grad_()
    assert pk.add_rms_norm(on_gpu(2, 64), None, w, 1e-6).requires_grad
    with torch.no_grad():
        assert not launches
        pk.add_rms_norm(on_gpu(2, 64), None, w, 1e-6)
    assert len(launches) == 1
    assert pk.add_rms_norm(on_gpu(0, 64), None, w, 1e-6).shape == (0, 64)
    assert len(launches) == 1
    with torch.enable_grad():
        assert pk.silu_mul(on_gpu(2, 64).requires_grad_()).requires_grad
    assert pk.silu_mul(on_gpu(3, 0)).shape == (3, 0)
    assert len(launches) == 1


@pytest.mark.parametrize("shape", [(32,), (2, 32), (2, 1, 32), (3, 2, 5, 16), (2, 6)])
def test_silu_mul_takes_the_halves_of_the_last_dim(shape):
    gu = torch.randn(*shape, generator=torch.Generator().manual_seed(1))
    n = shape[-1] // 2
    gate, up = gu.split(n, dim=-1)
    got = pk.silu_mul(gu)
    assert got.shape == shape[:-1] + (n,)
    assert torch.equal(got, torch.nn.functional.silu(gate) * up)


@pytest.mark.parametrize("shape", [(2, 3), (2, 17), (1, 2, 5)])
def test_silu_mul_refuses_halves_of_two_widths(shape):
    with pytest.raises(RuntimeError):
        pk.silu_mul(torch.ones(*shape))
