"""fp32 batches of 5..16 rows: the matrix-core passes (x whole in LDS up to 4580 elements at 8 rows and 2180 at 16, and rows of whole
128-byte lines up to 4608 and 2240), the two dense products and their join beyond that, and the dense down product over rows of any length."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# (4, 4): every matrix is half a cache line, and what a lane without work re-reads has to lie in it;
# H around the limits of one and two groups of x in LDS; I odd, below a tile, over 8192 (two launches of a product)
SIZES = [(256, 613, 5), (36, 9, 16), (1024, 515, 9), (2304, 1000, 16), (2308, 1001, 16), (4608, 515, 8), (4612, 777, 5), (4612, 777, 11),
         (260, 8200, 7), (5120, 8204, 8), (64, 4, 12),
         (4, 4, 5), (4, 4, 16), (2180, 301, 16), (2184, 301, 16), (2240, 300, 16), (2244, 300, 16), (4580, 201, 7), (4584, 201, 7)]


def _data(H, I, B):
    g = torch.Generator(device="cuda").manual_seed(H + I + B)
    x = torch.randn(B, 1, H, generator=g, device="cuda")
    wg, wu, wd = (torch.randn(I, H, generator=g, device="cuda") * H ** -0.5 for _ in range(3))
    X = x.double().reshape(B, H)
    a = F.silu(X @ wg.double().t())
    # no activation within the error of a sum from the threshold: every order of summation keeps the same neurons
    t = 0.2
    near = ((a.abs() - t).abs() < 1e-5).any(0)
    wg[near] = 0
    a = F.silu(X @ wg.double().t())
    a[a.abs() <= t] = 0
    return x, wg, wu, wd, t, a, a * (X @ wu.double().t())


def _close(got, want):
    # fp32 sums over at most 8204 products in chains of K / 64 and a short tree: about sqrt(K / 64) * 2^-24 of the result's norm, three times
    assert float((got.double().reshape(want.shape) - want).norm()) <= 2e-6 * float(want.norm()) + 1e-12


@pytest.mark.parametrize("H,I,B", SIZES)
def test_fp32_rows(H, I, B):
    import flash_gemv

    x, wg, wu, wd, t, a, z = _data(H, I, B)
    want = z @ wd.double()
    _close(flash_gemv.cats_mlp(x, wg, wu, wd, t), want)
    out = torch.ones(B, H, device="cuda")
    flash_gemv.flag_gemv_gemv_atomic(x, wg, wu, wd, out, t)
    _close(out, want + 1)
    y, flag, fetched = flash_gemv.cats_mlp_stats(x, wg, wu, wd, t)
    _close(y, want)
    assert int(fetched) == int((a != 0).any(0).sum())
    if I % 4 == 0:
        _close(flash_gemv.flag_gemv_gemv_inner_fp32(x, wg, wu, wd.t().contiguous(), t), want)


def test_what_is_not_kept_does_not_count():
    """An infinite up weight of a neuron that no row keeps, and of one that only some rows keep."""
    import flash_gemv

    for H in (256, 4612):
        x, wg, wu, wd, t, a, z = _data(H, 404, 6)
        wg[3], wu[3, 0] = 0, float("inf")
        a[:, 3] = 0
        some = int((a != 0).any(0).logical_and((a == 0).any(0)).nonzero()[0])
        wu[some, 0] = float("inf")
        y = flash_gemv.cats_mlp(x, wg, wu, wd, t).reshape(6, H)
        keeps = a[:, some] != 0
        assert not y[keeps].isfinite().any() and y[~keeps].isfinite().all()


@pytest.mark.parametrize("H,I,B", [(256, 613, 5), (4608, 515, 8), (4612, 777, 5), (4612, 777, 11), (2240, 300, 16), (2244, 515, 9), (2308, 1001, 16),
                                   (5120, 8204, 8), (4096, 1000, 16)])
def test_gate_call_and_fused_calls_share_their_activations(H, I, B):
    """With a threshold that is one of the gate call's own activations, bit for bit, every call flags exactly what it flags: a sum in another
    order moves some activation across it."""
    from cats_amd import capi

    x, wg, wu, wd, _, a64, _ = _data(H, I, B)
    x[:, 0, 0] = 1
    wu.zero_()
    wu[:, 0] = 1                                     # the up sum is 1: z is the activation
    X, ws = x.reshape(B, H), capi.Workspace(B, H, I)
    a, flag = capi.gate_flag(X, wg, 0.2)
    # fp32 sums over H products of unit variance in chains of K / 64: see _close; single values up to six of their deviations
    assert float((a.double() - F.silu(X.double() @ wg.double().t())).abs().max()) < 6 * 2e-6
    for k in range(0, a.numel(), max(1, a.numel() // 40)):
        t = float(a.flatten()[k].abs())
        _, flag = capi.gate_flag(X, wg, t, want_a=False)
        assert torch.equal(flag, a.abs() > t)
        z, flag_up = capi.gate_up(X, wg, wu, t)
        assert torch.equal(flag_up, flag) and torch.equal(z, torch.where(flag, a, torch.zeros_like(a)))
        _, flag_mlp, _ = capi.mlp(X, wg, wu, wd, t, ws, want_flag=True, want_count=True)
        assert torch.equal(flag_mlp, flag)


@pytest.mark.parametrize("H,B,steps,joined", [
    (2180, 9, (0, 7, 33), False), (2184, 9, (0, 7, 33), True), (2240, 16, (0, 7, 33), False), (2244, 16, (0, 7, 33), True),
    (4580, 8, (0, 17, 115), False), (4584, 8, (0, 17, 115), True), (4608, 5, (0, 17, 115), False), (4612, 5, (0, 17, 115), True)])
def test_where_the_one_launch_kernel_ends(H, B, steps, joined):
    """Which kernel it is, told by the order of its sums: 1 and twice t, t below half a unit in the last place of 1 and 2t above it, in three
    steps of 32 elements.  The one-launch kernel gives a wave consecutive steps, so one wave adds both t first: 1 + 2^-23.  The joined
    products deal the steps of a chunk to all waves: each t meets the 1, or a wave with nothing, by itself: 1."""
    from cats_amd import capi

    t = 0.75 * 2.0 ** -24
    w, x = torch.zeros(64, H, device="cuda"), torch.ones(B, H, device="cuda")
    for step, v in zip(steps, (t, t, 1.0)):
        w[0, 32 * step] = v
    a, _ = capi.gate_flag(x, w, -1.0)
    one, more = (F.silu(torch.tensor([v], dtype=torch.float64)).item() for v in (1.0, 1.0 + 2.0 ** -23))
    a = a[:, 0].double()
    assert bool(((a - (one if joined else more)).abs() < (a - (more if joined else one)).abs()).all())
