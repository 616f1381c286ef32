"""The one-trip kernels of small layers (cats_small.h): workgroups with fewer than sixteen neurons, or none; rows of one vector up to the longest;
every batch size's kernel; rows that start off the cache lines; and both reductions of the layer tail."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

UNIT = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def reference(x, wg, wu, wd, t, dtype):
    """The call's roundings with 64-bit sums.  Gate rows with an activation near the threshold are zeroed in place first: no order of the sums
    may decide a flag."""
    r = lambda v: v.to(dtype).double()
    gate = lambda: F.silu(r(x.double() @ wg.double().t()))
    wg[((gate().abs() - t).abs() < 8 * UNIT[dtype]).any(0)] = 0
    a = r(gate())
    flag = a.abs() > t
    z = torch.where(flag, r(a * r(x.double() @ wu.double().t())), torch.zeros_like(a))
    return z @ wd.double(), flag


def layer(H, I, B, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    return rn(B, H).to(dtype), (rn(I, H) * H ** -0.5).to(dtype), (rn(I, H) * H ** -0.5).to(dtype), (rn(I, H) * 0.1).to(dtype)


# rounded products and outputs: one unit of the type for each of z's three roundings and for y's, in the 2-norm; fp32 sums come on top
def tolerance(want, dtype):
    return (4 * UNIT[dtype] + 1e-6) * float(want.norm()) + 1e-12


CASES = [(8, 1, 1), (8, 17, 3), (256, 15, 2), (512, 16, 9), (520, 1000, 4), (1024, 129, 16), (1032, 777, 5), (1536, 272, 1), (1544, 2049, 3),
         (2040, 300, 8), (2048, 512, 2), (2048, 31, 12), (512, 4097, 1), (512, 4113, 3), (1024, 5000, 2),
         # both sides of the lines to the other kernels, a workgroup a CU, two, and more than one without place for two
         (2048, 4096, 3), (2048, 4096, 4), (1024, 5000, 4), (1024, 5000, 6), (1000, 4200, 3), (1000, 4200, 4), (520, 4500, 12), (640, 4500, 11)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,I,B", CASES)
def test_whole_mlp(H, I, B, dtype):
    import flash_gemv

    if dtype == torch.float32:
        H //= 2
    x, wg, wu, wd = layer(H, I, B, dtype, H + I + B)
    t = 0.2
    want, flag = reference(x, wg, wu, wd, t, dtype)
    dead = ~flag.any(0)
    wd[dead] = float("inf")  # a neuron that no row keeps is read but must not count
    wu[dead] = float("nan")
    y, flags, count = flash_gemv.cats_mlp_stats(x, wg, wu, wd, t)
    out = torch.ones(B, H, device="cuda")
    flash_gemv.flag_gemv_gemv_atomic(x, wg, wu, wd, out, t)
    assert torch.equal(flags.reshape(B, I).bool(), flag) and int(count) == int(flag.any(0).sum())
    assert torch.equal(y, flash_gemv.cats_mlp(x, wg, wu, wd, t))
    assert float((y.double() - want).norm()) <= tolerance(want, dtype)
    assert float((out.double() - 1 - want).norm()) <= tolerance(want, dtype) + 1e-6 * out.numel() ** 0.5


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,I,B", [(256, 33, 1), (512, 1024, 2), (992, 1025, 4), (1024, 500, 11), (2016, 700, 3), (1024, 2000, 16)])
def test_layer_tail(H, I, B, dtype):
    import flash_gemv

    if dtype == torch.float32:
        H = H // 64 * 32
    h, wg, wu, wd = layer(H, I, B, dtype, H + I + B)
    n1, n2 = torch.linspace(0.5, 1.5, H, device="cuda").to(dtype), torch.linspace(1.2, 0.8, H, device="cuda").to(dtype)
    r = lambda v: v.to(dtype).double()
    x = (n1.double() * r(h.double() * (h.double().square().mean(1, keepdim=True) + 1e-5).rsqrt())).to(dtype)
    t = -1.0  # every neuron is kept: x is rounded from fp32 sums, so a flag at the threshold would hang on their order
    want, _ = reference(x, wg, wu, wd, t, dtype)
    out, nxt = flash_gemv.cats_mlp_norm_residual_norm(h, n1, 1e-5, wg, wu, wd, t, n2, 1e-6)
    assert torch.equal(out, flash_gemv.cats_mlp_norm_residual(h, n1, 1e-5, wg, wu, wd, t))
    # a last bit of x (its scale is an fp32 sum) moves the products by at most a unit of the type each
    assert float((out.double() - h.double() - want).norm()) <= tolerance(want, dtype) + 2 * UNIT[dtype] * float(want.norm() + h.double().norm())
    o = out.double()
    scale = (o.square().mean(1, keepdim=True) + 1e-6).rsqrt()
    assert float((nxt.double() - n2.double() * o * scale).norm()) <= 2.5 * UNIT[dtype] * float((n2.double() * o * scale).norm()) + 1e-12


@pytest.mark.parametrize("H,I,B", [(512, 1000, 1), (1024, 2731, 2), (1024, 500, 4), (512, 300, 16)])
def test_two_streams_add_into_one_buffer(H, I, B):
    """The fp32-accumulate calls of two streams, a workspace each, add into one buffer without losing any: 1 and 2 rows in one and
    two launches, and batches."""
    from cats_amd import capi

    n = 150
    layers = [layer(H, I, B, torch.float16, seed) for seed in (1, 2)]
    spaces = [capi.Workspace(B, H, I) for _ in layers]
    once = []
    for (x, wg, wu, wd), ws in zip(layers, spaces):
        v = torch.zeros(B, H, device="cuda")
        capi.mlp(x, wg, wu, wd, 0.2, ws, y_f32=v)
        once.append(v.double())
    out, streams = torch.zeros(B, H, device="cuda"), [torch.cuda.Stream() for _ in layers]
    torch.cuda.synchronize()
    for _ in range(n):
        for (x, wg, wu, wd), ws, s in zip(layers, spaces, streams):
            with torch.cuda.stream(s):
                capi.mlp(x, wg, wu, wd, 0.2, ws, y_f32=out)
    torch.cuda.synchronize()
    # a call's totals have a fixed order, so each adds the same value every time; 2 n fp32 additions round by half a unit of a running
    # sum of at most n (|a| + |b|) each.  One addition lost is a whole |a| or |b|, hundreds of times as much.
    a, b = once
    bound = 2 * n * 2.0 ** -24 * n * (a.abs() + b.abs())
    assert bool(((out.double() - n * (a + b)).abs() <= bound + 1e-30).all())
