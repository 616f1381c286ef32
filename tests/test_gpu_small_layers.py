"""Layers with fewer neurons than the chip has row waves, by the kernels of small layers, which take them, and by the single-pass kernel:
there shares of 4 to 24 neurons a workgroup, the last one short, some row waves without a neuron, some with a second one."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["small", "single pass"])
def kernels(request):
    from cats_amd import capi

    capi.set_tuning(gate_variant=0 if request.param == "small" else -1)  # any other than 0 keeps whole calls off the small layers' kernels
    yield request.param
    capi.set_tuning()


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("I", [1, 3, 4, 5, 7, 13, 1023, 1025, 1535, 1536, 1537, 2049, 3071, 3073, 6145])
def test_small_layers(I, B, kernels):
    import flash_gemv

    H, t = 132, 0.2
    g = torch.Generator(device="cuda").manual_seed(I)
    x = torch.randn(B, 1, H, generator=g, device="cuda")
    wg, wu, wd = (torch.randn(I, H, generator=g, device="cuda") * H ** -0.5 for _ in range(3))
    X = x.double().reshape(B, H)
    near = ((F.silu(X @ wg.double().t()).abs() - t).abs() < 1e-5).any(0)
    wg[near] = 0  # no activation within the error of a sum from the threshold
    a = F.silu(X @ wg.double().t())
    kept = a * (a.abs() > t)
    want = (kept * (X @ wu.double().t())) @ wd.double()
    tol = 2e-6 * float(want.norm()) + 1e-12  # fp32 sums of at most 6145 products: see their error in the 2-norm, 3e-7, times seven
    y, flag, fetched = flash_gemv.cats_mlp_stats(x, wg, wu, wd, t)
    assert torch.equal(flag.reshape(B, I).bool(), kept != 0) and int(fetched) == int((kept != 0).any(0).sum())
    out = torch.ones(B, H, device="cuda")
    flash_gemv.flag_gemv_gemv_atomic(x, wg, wu, wd, out, t)
    act = F.silu((X @ wg.double().t()).float()).reshape(B, 1, I)
    for got in (y, flash_gemv.cats_mlp(x, wg, wu, wd, t), flash_gemv.gemv_gemv_triton(x, act, wu, wd, t), out - 1):
        assert float((got.double().reshape(B, H) - want).norm()) <= tol + (1e-6 if got is not y else 0)
