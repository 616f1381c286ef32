"""The matrix-core gate / gate+up / up kernels at the row lengths where their split of a row changes: rows of one vector, rows that
end inside a 64-element step, pitches that are no multiple of a cache line (rows eight apart share a workgroup), the last
length of one register set per tile and the first of two, the longest row that fits on chip."""
import pytest
import torch

from tests.test_gpu_parity import check_mlp_case, close
from tests.util import dev, make_mlp

pytestmark = pytest.mark.gpu

capi = None


@pytest.fixture(scope="module", autouse=True)
def _load():
    import tests.test_gpu_parity as parity
    from cats_amd import capi as _capi

    global capi
    _capi.lib()
    capi = parity.capi = _capi


ROWS = [
    # H, I, B, dtype
    (8, 9, 3, torch.float16),         # one vector: seven of the eight waves have no step
    (64, 200, 5, torch.bfloat16),     # exactly one step
    (72, 64, 8, torch.float16),       # pitch 144 bytes: two phases of 16-byte vectors in every step
    (520, 333, 16, torch.bfloat16),   # nine or ten steps with the phase
    (1000, 777, 11, torch.float16),
    (3080, 1000, 3, torch.bfloat16),
    (4088, 515, 16, torch.float16),   # 64 steps plus the phase: nine per wave, two groups of batch rows
    (4104, 260, 4, torch.bfloat16),   # 65 steps or 66
    (4672, 130, 8, torch.float16),    # 73 steps: the first length of two register sets per tile
    (5128, 263, 7, torch.bfloat16),   # 81 or 82 steps: eleven per wave, rounded up to twelve
    (8184, 200, 5, torch.float16),    # 128 steps or 129
    (8192, 520, 8, torch.float16),
    (9152, 64, 4, torch.bfloat16),
    (9216, 64, 3, torch.float16),     # whole lines, no phase: the longest row whose eight x operands fit in LDS
    (9160, 65, 5, torch.float16),     # the longest one with phases
    (9168, 65, 5, torch.float16),     # its operands do not fit any more: the wave-per-row kernel's
    (9224, 64, 8, torch.bfloat16),    # more steps than the register sets hold
    (4360, 65, 16, torch.float16),    # two groups of operands: the longest row with phases
    (4368, 65, 16, torch.bfloat16),   # two passes of eight
    (4480, 64, 16, torch.bfloat16),   # the longest row of whole lines
    (4488, 64, 16, torch.float16),
    (1024, 256 * 8 + 1, 6, torch.float16),   # nine rows per workgroup: a full tile and one row of the next
]


@pytest.mark.parametrize("H,I,B,dtype", ROWS)
def test_row_lengths(oracle, H, I, B, dtype):
    m = make_mlp(H, I, B, dtype, seed=H + 5 * I + B, corr=0.5)
    a, _ = oracle.c_gate(m["x"], m["wg"], -1.0)
    mags = a.float().abs().flatten()
    ws = capi.Workspace(B, H, I)
    d = dev(m)
    for q in (0.0, 0.6):
        t = -1.0 if q == 0.0 else float(torch.quantile(mags, q))
        check_mlp_case(oracle, m, t, tag=f"row-length-q{q}", ws=ws)
        flag = torch.abs(a) > t
        y = capi.up_down(d["x"], a.cuda(), d["wu"], d["wdt"], t, ws)
        close(y.cpu(), oracle.c_mlp(m["x"], m["wg"], m["wu"], m["wd"], t, a_in=a, flag_in=flag)["y"], dtype)


@pytest.mark.parametrize("H,I,B,dtype", [(72, 64, 8, torch.float16), (3080, 300, 3, torch.bfloat16), (5128, 70, 4, torch.float16), (4088, 96, 12, torch.bfloat16)])
def test_padding_lanes_do_not_reach_the_sums(H, I, B, dtype):
    """A lane in front of a row or behind it re-reads the first vector of the matrix, and the last vector of a row has the next
    row's weights behind it: infinities in row 0 and in every odd row must not change one bit of the other rows' activations."""
    m = make_mlp(H, I, B, dtype, seed=H + I)
    d = dev(m)
    a, flag = capi.gate_flag(d["x"], d["wg"], 0.05)
    bad = d["wg"].clone()
    bad[0] = float("inf")
    bad[1::2] = float("inf")
    a2, flag2 = capi.gate_flag(d["x"], bad, 0.05)
    torch.cuda.synchronize()
    assert torch.equal(a2[:, 2::2], a[:, 2::2]) and torch.equal(flag2[:, 2::2], flag[:, 2::2])
    assert bool(torch.isfinite(a2[:, 2::2].float()).all())


@pytest.mark.parametrize("H,I,B,dtype", [(520, 200, 5, torch.float16), (4104, 96, 8, torch.bfloat16), (1000, 128, 16, torch.float16)])
def test_weights_off_a_cache_line(oracle, H, I, B, dtype):
    """16-byte alignment is all the entry points ask for: gate and up matrices that start at different places of a cache line."""
    m = make_mlp(H, I, B, dtype, seed=H + I + B, corr=0.5)
    t = float(torch.quantile(oracle.c_gate(m["x"], m["wg"], -1.0)[0].float().abs().flatten(), 0.5))
    d = dev(m)
    for name, vecs in (("wg", 3), ("wu", 6), ("wdt", 1)):
        buf = torch.zeros(d[name].numel() + 128, dtype=dtype, device="cuda")
        view = buf[vecs * 8:vecs * 8 + d[name].numel()].view_as(d[name])
        view.copy_(d[name])
        d[name] = view
    ws = capi.Workspace(B, H, I)
    a, flag = capi.gate_flag(d["x"], d["wg"], t)
    y = capi.mlp(d["x"], d["wg"], d["wu"], d["wdt"], t, ws)
    y = y[0] if isinstance(y, tuple) else y
    torch.cuda.synchronize()
    assert torch.equal(flag.cpu(), torch.abs(a.cpu()) > t)
    close(y.cpu(), oracle.c_mlp(m["x"], m["wg"], m["wu"], m["wd"], t, a_in=a.cpu(), flag_in=flag.cpu())["y"], dtype)


@pytest.mark.parametrize("H,I,B,dtype", [(520, 200, 5, torch.float16), (3104, 96, 8, torch.bfloat16), (8192, 64, 4, torch.float16), (1000, 128, 16, torch.float16),
                                           (520, 200, 5, torch.float32), (4096, 64, 8, torch.float32), (2180, 96, 16, torch.float32), (2184, 96, 12, torch.float32)])
def test_norm_while_staging(oracle, H, I, B, dtype):
    """h + MLP(norm(h)): the norm works on the staged operands, padding steps included."""
    m = make_mlp(H, I, B, dtype, seed=H + 3 * I)
    h = (m["x"].float() * 2.5 + 0.3).to(dtype)
    nw = (1.0 + 0.2 * torch.randn(H, generator=torch.Generator().manual_seed(H))).to(dtype)
    x = oracle.torch_rms_norm(h, nw, 1e-5)
    t = float(torch.quantile(oracle.c_gate(x, m["wg"], -1.0)[0].float().abs().flatten(), 0.5))
    d = dev(m)
    out = capi.mlp_norm_residual(h.cuda(), nw.cuda(), 1e-5, d["wg"], d["wu"], d["wdt"], t, capi.Workspace(B, H, I))
    a, flag = capi.gate_flag(x.cuda(), d["wg"], t)
    torch.cuda.synchronize()
    want = h.float() + oracle.c_mlp(x, m["wg"], m["wu"], m["wd"], t, a_in=a.cpu(), flag_in=flag.cpu())["y"].float()
    close(out.cpu(), want, dtype)


@pytest.mark.parametrize("H,I,B,dtype,variant", [(5128, 263, 16, torch.float16, 0), (4488, 200, 9, torch.bfloat16, 0), (4612, 777, 13, torch.float32, -1)])
def test_count_of_a_call_in_two_passes(H, I, B, dtype, variant):
    """Rows that no one-pass kernel takes: the count without flags, whose bytes wait in the workspace while the second pass runs, is
    that of the flags."""
    m = make_mlp(H, I, B, dtype, seed=H + B)
    d = dev(m)
    ws = capi.Workspace(B, H, I)
    L = capi.lib()
    t = float(capi.gate_flag(d["x"], d["wg"], -1.0)[0].float().abs().flatten().quantile(0.95))
    count, y2 = torch.full((1,), -1, dtype=torch.int32, device="cuda"), torch.empty(B, H, dtype=dtype, device="cuda")
    L.cats_set_tuning(variant, 0, 0, 0)
    try:
        y, flag, with_flags = capi.mlp(d["x"], d["wg"], d["wu"], d["wdt"], t, ws, want_flag=True, want_count=True)
        assert L.cats_mlp(capi._p(d["x"]), capi._p(d["wg"]), capi._p(d["wu"]), capi._p(d["wdt"]), capi._p(y2), None, None, capi._p(count), B, H, I,
                          capi.DTYPE_CODE[dtype], t, capi._p(ws.buf), ws.nbytes, capi._stream(d["x"])) == 0
        torch.cuda.synchronize()
    finally:
        L.cats_set_tuning(0, 0, 0, 0)
    want = int(flag.any(dim=0).sum())
    assert 0 < want < I and int(count) == want and int(with_flags) == want and torch.equal(y.view_as(y2), y2)


@pytest.mark.parametrize("H,B,dtype,matrix_cores", [
    (9160, 5, torch.float16, True), (9168, 5, torch.float16, False), (9216, 3, torch.bfloat16, True), (9224, 3, torch.bfloat16, False),
    (4360, 9, torch.bfloat16, True), (4368, 9, torch.bfloat16, False), (4480, 9, torch.float16, True), (4488, 9, torch.float16, False),
    (9216, 2, torch.float16, False)])
def test_where_the_matrix_cores_end(H, B, dtype, matrix_cores):
    """Which kernel took the last batch row, told by the order of its sums: the products of a row cancel in pairs, so what is left of a sum
    is its rounding errors.  With the tuning knob the row goes to the wave-per-row kernel, which adds in one order whatever B is.  Of nine
    rows the last is a pass of its own unless all go in one."""
    g = torch.Generator(device="cuda").manual_seed(H)
    half = torch.randn(96, H // 2, generator=g, device="cuda").to(dtype)
    w = torch.cat((half, -half), 1)
    x1 = torch.randn(B, H // 2, generator=g, device="cuda").to(dtype)
    x = torch.cat((x1, x1), 1)
    a, _ = capi.gate_flag(x, w, -1.0)
    capi.set_tuning(-1, 0, 0, 0)
    try:
        b, _ = capi.gate_flag(x, w, -1.0)
    finally:
        capi.set_tuning(0, 0, 0, 0)
    assert torch.equal(a[-1], b[-1]) != matrix_cores
