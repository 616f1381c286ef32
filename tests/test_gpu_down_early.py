"""The matrix-core down pass asks for the first 64 neurons of every range before their flags are there, and cuts rows into slabs of equal
width: whole-MLP calls at the edges of both, against 64-bit sums over the kernel's own activations."""
import pytest
import torch

from cats_amd import capi

pytestmark = pytest.mark.gpu

CASES = [
    # H, I, B, dtype
    (2056, 2100, 3, torch.float16),    # ranges of 48 neurons: shorter than what is asked for early
    (4096, 2060, 16, torch.bfloat16),  # ranges of 72: eight neurons behind the early ones; the last one of 44 ends inside a step
    (3080, 4095, 3, torch.bfloat16),   # seven slabs of 56 vectors, the last one of 49
    (4168, 1500, 5, torch.float16),    # nine slabs of 64, the last one of 9
    (4096, 17000, 16, torch.float16),  # more z values than a thread asks for at once
    (8192, 33001, 3, torch.float16),   # ranges of 2064 neurons, whose rows wait for the flags
    (2048, 8100, 3, torch.float16),    # ranges of 128, 512 KiB apart, whose rows wait too; the next one's do not
    (2048, 7169, 3, torch.float16),
]


@pytest.mark.parametrize("H,I,B,dtype", CASES)
@pytest.mark.parametrize("sparsity", [0.0, 0.9])
def test_early_rows_and_slabs(H, I, B, dtype, sparsity):
    g = torch.Generator(device="cuda").manual_seed(H + I + B)
    wg, wu, wdt = ((torch.randn(I, H, generator=g, device="cuda") * 0.02).to(dtype) for _ in range(3))
    x = torch.randn(B, H, generator=g, device="cuda").to(dtype)
    t = -1.0
    if sparsity:
        a = capi.gate_flag(x, wg, -1.0)[0]
        t = float(torch.kthvalue(a.float().abs().flatten(), int(sparsity * a.numel())).values)
    a, flag = capi.gate_flag(x, wg, t)
    dead = ~flag.bool().view(B, I).any(dim=0)
    assert bool(dead.any()) == (sparsity > 0)
    wdt[dead] = float("inf")  # asked for early or read as padding, never used
    print(f"[case] early rows H={H} I={I} B={B} {dtype} sparsity={sparsity}", flush=True)
    ws = capi.Workspace(B, H, I)
    y = capi.mlp(x, wg, wu, wdt, t, ws).view(B, H)
    again = capi.mlp(x, wg, wu, wdt, t, ws).view(B, H)
    assert torch.equal(y, again)
    u = (x.double() @ wu.double().t()).to(dtype)
    z = torch.where(flag.bool().view(B, I), (a.view(B, I).float() * u.float()).to(dtype), torch.zeros_like(u)).double()
    want = z @ torch.where(dead[:, None], torch.zeros_like(wdt), wdt).double()
    # y is rounded once (half a unit in the last place, 2^-11 or 2^-8 relative, at most), and a product u or z that fp32 sums put on
    # the other side of a rounding boundary moves by one unit: together below two of the half units
    eps = 2.0 ** (-10 if dtype is torch.float16 else -7)
    assert torch.isfinite(y).all()
    assert float((y.double() - want).norm() / want.norm()) < eps
