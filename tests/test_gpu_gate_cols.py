"""The one-row MLP over an (H, I) gate weight, at the sizes where its cut of the columns and rows changes."""
import pytest
import torch

from tests.test_gpu_parity import close
from tests.util import dev, make_mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,dtype", [
    (8, 8, torch.float16),          # one vector, one lane
    (16, 9, torch.bfloat16),        # a second lane moved back by all but one column; one row per wave
    (256, 511, torch.float16), (264, 513, torch.bfloat16),   # around one slab of columns, rows off the vector
    (4096, 1536, torch.float16), (4096, 11008, torch.float16),
    (1000, 3001, torch.bfloat16),
    (8200, 640, torch.float16),     # more than 64 rows to a wave, ranges of rows that do not divide
    (17000, 120, torch.bfloat16),   # rows too long for the single-pass kernel
    (4, 4, torch.float32), (516, 257, torch.float32), (4096, 1000, torch.float32),
    (4100, 333, torch.float32)])    # the same in fp32
def test_gate_cols(oracle, H, I, dtype):
    import flash_gemv as fg

    m = make_mlp(H, I, 1, dtype, seed=H + I)
    a, _ = oracle.c_gate(m["x"], m["wg"], -1.0)
    d = dev(m)
    wg_t = d["wg"].t().contiguous()
    for q in (0.0, 0.6, 1.0):
        # in the widest gap near the quantile, so that no order of summation decides a flag
        mags = a.float().abs().flatten().sort().values
        i = min(int(q * (I - 1)), I - 1)
        lo, hi = max(0, i - 8), min(I - 1, i + 8)
        j = lo + int((mags[lo + 1:hi + 1] - mags[lo:hi]).argmax()) if hi > lo else 0
        t = -1.0 if q == 0.0 else float("inf") if q == 1.0 else float(mags[j:j + 2].mean())
        want = oracle.c_mlp(m["x"], m["wg"], m["wu"], m["wd"], t)["y"]
        got = fg.flag_gemv_gemv_dejavu(d["x"], wg_t, d["wu"], d["wdt"], t)
        assert got.shape == (1, H) and got.dtype == dtype
        close(got.cpu(), want, dtype)
        same = fg.flag_gemv_gemv_triton(d["x"].view(1, 1, H), wg_t, d["wu"], d["wdt"], t)
        assert torch.equal(same.view(1, H), got)


def test_gate_cols_reads_nothing_past_the_weight():
    """The weight at the end of its buffer, at an odd element, with infinities before and behind it."""
    import flash_gemv as fg

    H, I = 264, 515
    m = make_mlp(H, I, 1, torch.float16, seed=3)
    d = dev(m)
    wg_t = d["wg"].t().contiguous()
    buf = torch.full((H * I + 6,), float("inf"), dtype=torch.float16, device="cuda")
    view = buf[3:3 + H * I].view(H, I)
    view.copy_(wg_t)
    want = fg.flag_gemv_gemv_dejavu(d["x"], wg_t, d["wu"], d["wdt"], 0.05)
    assert torch.equal(fg.flag_gemv_gemv_dejavu(d["x"], view, d["wu"], d["wdt"], 0.05), want)


def test_what_the_kernels_do_not_take_keeps_the_composite():
    import flash_gemv as fg

    H, I = 256, 512
    d = dev(make_mlp(H, I, 1, torch.float16, seed=4))
    wg_t = d["wg"].t().contiguous()
    args = (d["x"], wg_t, d["wu"], d["wdt"])
    assert fg._takes_gate_cols(*args, 0.05)
    assert not fg._takes_gate_cols(d["x"], d["wg"].t(), d["wu"], d["wdt"], 0.05)          # a view of the (I, H) weight
    assert not fg._takes_gate_cols(*args, torch.tensor(0.05))
    assert not fg._takes_gate_cols(d["x"].expand(2, H).contiguous(), *args[1:], 0.05)
    with torch.autocast("cuda"):
        assert not fg._takes_gate_cols(*args, 0.05)
    y = fg.flag_gemv_gemv_dejavu(d["x"], d["wg"].t(), d["wu"], d["wdt"], 0.05)
    torch.testing.assert_close(y, fg.flag_gemv_gemv_dejavu(*args, 0.05), rtol=1e-2, atol=2e-3)


def test_watched_calls_keep_the_composite():
    """A trace made at one row is of the operations and takes other rows later; a dispatch mode sees the gate's product."""
    import flash_gemv as fg
    from torch.utils._python_dispatch import TorchDispatchMode

    H, I = 256, 512
    d = dev(make_mlp(H, I, 2, torch.float16, seed=5))
    wg_t, x = d["wg"].t().contiguous(), d["x"].view(2, 1, H)
    traced = torch.jit.trace(lambda x: fg.flag_gemv_gemv_triton(x, wg_t, d["wu"], d["wdt"], 0.05), (x[:1].clone(),))
    assert torch.equal(traced(x), fg.flag_gemv_gemv_triton(x, wg_t, d["wu"], d["wdt"], 0.05))

    class Names(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    with Names() as names:
        fg.flag_gemv_gemv_dejavu(x[0], wg_t, d["wu"], d["wdt"], 0.05)
    assert "nonzero" in names.seen and "silu" in names.seen

    class Sub(torch.Tensor):
        pass

    assert not fg._takes_gate_cols(x[:1].as_subclass(Sub), wg_t, d["wu"], d["wdt"], 0.05)
    assert fg._takes_gate_cols(x[:1], torch.nn.Parameter(wg_t), d["wu"], d["wdt"], 0.05)
