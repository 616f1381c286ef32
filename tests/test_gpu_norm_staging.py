"""The norm in front of the MLP where the kernels take it from registers, and the rounding to bf16 by the hardware's conversion."""
import pytest
import torch

import cats_amd.capi as capi
from tests.test_gpu_parity import close
from tests.util import dev, make_mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,B,dtype", [
    (1000, 6000, 1, torch.float16), (8192, 3000, 1, torch.bfloat16), (3080, 4500, 2, torch.bfloat16),          # single-pass kernel, one to two rounds of x
    (1288, 5000, 3, torch.bfloat16), (4096, 3000, 8, torch.float16), (6152, 2100, 5, torch.bfloat16),           # matrix-core pass, with and without phases, two register sets
    (8160, 2100, 4, torch.bfloat16), (8192, 2100, 8, torch.float16), (9208, 900, 3, torch.bfloat16), (4096, 1500, 6, torch.float32),             # the longest of these
    (2568, 3500, 9, torch.float16), (4096, 3000, 16, torch.bfloat16), (2056, 2500, 7, torch.float32),
    (2056, 3000, 2, torch.float32), (4100, 1500, 3, torch.float32), (8192, 601, 4, torch.float32), (12288, 300, 2, torch.float32),               # wave per row
    (384, 777, 4, torch.bfloat16), (264, 500, 11, torch.float16), (1288, 300, 2, torch.float16), (520, 300, 4, torch.float32)])  # small layers
def test_norm_from_registers(oracle, H, I, B, dtype):
    m = make_mlp(H, I, B, dtype, seed=H + 3 * I + B)
    h = (m["x"].float() * 1.9 - 0.2).to(dtype)
    h[-1] = 0  # a row without squares: the norm leaves zeros
    nw = (1.0 + 0.2 * torch.randn(H, generator=torch.Generator().manual_seed(H))).to(dtype)
    x = oracle.torch_rms_norm(h, nw, 1e-5)
    t = float(torch.quantile(oracle.c_gate(x, m["wg"], -1.0)[0].float().abs().flatten()[:1 << 20], 0.5))
    d = dev(m)
    out = capi.mlp_norm_residual(h.cuda(), nw.cuda(), 1e-5, d["wg"], d["wu"], d["wdt"], t, capi.Workspace(B, H, I))
    a, flag = capi.gate_flag(x.cuda(), d["wg"], t)
    torch.cuda.synchronize()
    want = h.float() + oracle.c_mlp(x, m["wg"], m["wu"], m["wd"], t, a_in=a.cpu(), flag_in=flag.cpu())["y"].float()
    close(out.cpu(), want, dtype)
    assert not out[-1].any()


@pytest.mark.parametrize("B", [1, 4])
def test_bf16_rounding(B):
    """A sum of two bf16 numbers that fp32 holds exactly leaves as torch rounds it: ties, the carry into the exponent, subnormal results,
    the step to infinity, infinities and NaN.  (The sign of a zero sum is not looked at: it depends on what the sum starts from.)"""
    import flash_gemv  # noqa: F401

    pairs = [(1.0, 2.0 ** -8), (1.0 + 2.0 ** -7, 2.0 ** -8), (1.0, -(2.0 ** -9)), (1.0, 2.0 ** -8 + 2.0 ** -14), (2.0 - 2.0 ** -7, 2.0 ** -8),
             (2.0 ** -126, -(2.0 ** -127) + 2.0 ** -133), (2.0 ** -133, 0.0), (3 * 2.0 ** -133, -(2.0 ** -133)),
             (3.3895313892515355e38, 2.0 ** 119), (3.3895313892515355e38, -(2.0 ** 119)), (-3.3895313892515355e38, -(2.0 ** 119)),
             (float("inf"), 1.0), (float("inf"), float("-inf")), (float("nan"), 0.0)]
    w = torch.zeros(16, 64, dtype=torch.bfloat16)
    w[:len(pairs), :2] = torch.tensor(pairs).to(torch.bfloat16)
    x = torch.zeros(B, 64, dtype=torch.bfloat16)
    x[:, :2] = 1.0
    out = torch.ops.flash_gemv.cats_linear(x.cuda(), None, 1e-5, w.cuda()).cpu()
    want = (w[:, 0].float() + w[:, 1].float()).to(torch.bfloat16)
    keep = torch.isfinite(w[:, :2].float()).all(1)
    for b in range(B):
        assert torch.equal(out[b][keep].abs(), want[keep].abs()) and torch.equal(out[b][keep] < 0, want[keep] < 0)
        assert torch.equal(torch.isnan(out[b]), torch.isnan(want)) and torch.equal(torch.isinf(out[b]), torch.isinf(want))


def test_bf16_rounding_of_any_float():
    """Floats of random bits, a third of them ties and as many a last bit beside one, as sums of three bf16 numbers of their own bits: every partial
    sum is exact, whatever the order, so what is stored is the float rounded once."""
    import flash_gemv  # noqa: F401

    n = 1 << 18
    g = torch.Generator().manual_seed(3)
    bits = torch.randint(0, 1 << 31, (n,), generator=g) | (torch.randint(0, 2, (n,), generator=g) << 31)
    low = torch.tensor([0x8000, 0x7FFF, 0x8001])
    kind = torch.arange(n) % 9
    bits = torch.where(kind < 3, (bits & ~0xFFFF) | 0x8000, torch.where(kind < 6, (bits & ~0xFFFF) | low[1 + kind % 2], bits))
    exponent = (bits >> 23) & 0xFF
    bits = (bits & ~(0xFF << 23)) | (exponent.clamp(60, 250) << 23)  # parts of normal size
    f = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32).view(torch.float32)
    part = lambda v: (v.view(torch.int32) & ~0xFFFF).view(torch.float32)  # the leading eight bits of it, towards zero
    hi = part(f)
    mid = part(f - hi)
    w = torch.zeros(n, 64, dtype=torch.bfloat16)
    for k, v in enumerate((hi, mid, f - hi - mid)):
        w[:, 7 * k] = v.to(torch.bfloat16)
        assert torch.equal(w[:, 7 * k].float(), v)
    out = torch.ops.flash_gemv.cats_linear(torch.ones(1, 64, dtype=torch.bfloat16, device="cuda"), None, 1e-5, w.cuda()).cpu().flatten()
    assert torch.equal(out.view(torch.int16), f.to(torch.bfloat16).view(torch.int16))
