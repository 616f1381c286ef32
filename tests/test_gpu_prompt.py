"""The kernel between the matrix products of a prompt, and the module routes that lead to it and past it."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2048, 2049, 100003])
def test_silu_mask_mul(n, dtype):
    import flash_gemv  # noqa: F401

    g = torch.Generator(device="cuda").manual_seed(n)
    gate, up = (2 * torch.randn(n, generator=g, device="cuda")).to(dtype), torch.randn(n, generator=g, device="cuda").to(dtype)
    for k, v in enumerate((float("nan"), float("inf"), -float("inf"), 0.0)):
        if n > 100:
            gate[10 * k], up[10 * k + 5] = v, v
    for t in (-1.0, 0.0, 0.3, float("inf")):
        a = F.silu(gate)
        a[a.abs() <= t] = 0
        got, want = torch.ops.flash_gemv.cats_silu_mask_mul(gate, up, t), a * up
        # the same operations with the same roundings; exp may differ in its last bit, which moves a by one step at most
        torch.testing.assert_close(got, want, rtol={torch.float16: 2e-3, torch.bfloat16: 1.6e-2, torch.float32: 1e-6}[dtype], atol=0, equal_nan=True)
        assert torch.equal(got == 0, want == 0)


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("method", [0, 2, 3])
def test_module_routes_agree(method, rows):
    """With and without a hook on the activation, which keeps the module on torch's operations."""
    from cats_amd.mlp import CatsMLP

    with torch.no_grad():
        torch.manual_seed(0)
        m = CatsMLP(256, 515, dead_threshold=0.05, dtype=torch.float16, device="cuda").eval()
        for p in m.parameters():
            p.normal_(0, 0.05)
        m.prepare_decode(method)
        x = torch.randn(3, rows, 256, device="cuda").half()
        a = m(x)
        handle = m.act_fn.register_forward_hook(lambda *args: None)
        b = m(x)
        handle.remove()
    torch.testing.assert_close(a, b, rtol=1e-2, atol=2e-3)
    y = m(x)                                       # gradients are asked for: torch's operations
    if rows > 1 or method == 0:
        assert y.requires_grad
        torch.testing.assert_close(y, b, rtol=0, atol=0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(3, 1, 256), (1, 7, 256), (1, 600, 256)])
def test_sp_method_0_is_torch_bit_for_bit(shape, dtype):
    from cats_amd.mlp import CatsMLP

    with torch.no_grad():
        torch.manual_seed(1)
        m = CatsMLP(256, 515, dead_threshold=0.05, dtype=dtype, device="cuda").eval()
        for p in m.parameters():
            p.normal_(0, 0.05)
        m.is_profile, m.sp_method = True, 0
        x = torch.randn(shape, device="cuda").to(dtype)
        a = F.silu(F.linear(x, m.gate_proj.weight))
        a[a.abs() <= 0.05] = 0
        assert torch.equal(m(x), F.linear(a * F.linear(x, m.up_proj.weight), m.down_proj.weight))
