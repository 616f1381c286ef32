"""The two matrix products of a prompt on the matrix cores, against the same roundings with 64-bit sums, at the edges of the tiles
(32, 64, 128 and 256 tokens; 16-row fragments; steps of 64 and 128 elements) and at row pitches of any element."""
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

SIZES = [  # tokens, H, I
    (1, 8, 8), (2, 8, 9), (3, 72, 17), (22, 304, 569), (31, 128, 130), (32, 136, 127), (33, 200, 1041), (64, 1024, 515), (65, 264, 2731),
    (128, 520, 1000), (129, 1288, 333), (257, 512, 4099), (300, 2048, 5461), (256, 4096, 11008), (511, 4096, 11003), (1030, 77, 91),
    # a long K over few columns: the second product in ranges of K, whose sums have a pitch of whole quads of columns
    (33, 77, 2731), (5, 201, 5461), (200, 333, 4099), (64, 78, 3001), (65, 9, 2731),
]


def _draw(M, H, I, dtype):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + H * 3 + I)
    x = torch.randn(M, H, generator=g, device="cuda").to(dtype)
    ws = [(torch.randn(s, generator=g, device="cuda") * (1.3 / math.sqrt(H))).to(dtype) for s in ((I, H), (I, H), (H, I))]
    return x, *ws


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,H,I", SIZES)
def test_prompt_mlp(M, H, I, dtype):
    import flash_gemv  # noqa: F401

    x, wg, wu, wd = _draw(M, H, I, dtype)
    t = 0.1
    y = torch.ops.flash_gemv.cats_prompt_mlp(x, wg, wu, wd, t)
    gate, up = (x.double() @ wg.double().t()).to(dtype), (x.double() @ wu.double().t()).to(dtype)
    a = F.silu(gate)
    a[a.abs() <= torch.tensor(t).to(dtype)] = 0
    want = (a * up).double() @ wd.double().t()
    # z carries the roundings of gate, a, up and z, y one more: below three steps of the type in the 2-norm; and a neuron whose gate sum
    # lies a rounding away from the threshold is kept by one order of summation and dropped by the other: |a| is near t there, a
    # twentieth of the kept ones' size at most
    step = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    kept = int((a != 0).sum())
    rel = float((y.double() - want).norm() / want.norm().clamp_min(1e-30))
    assert kept == 0 or rel < 3 * step + 0.1 / math.sqrt(kept), rel


@pytest.mark.parametrize("M,H,I", [(2, 640, 515), (32, 641, 1000), (9, 773, 515), (48, 905, 900), (64, 1283, 515), (100, 384, 700), (128, 393, 1041), (200, 520, 2731)])
def test_small_tiles(M, H, I):
    """Half tiles of 32 tokens and 32 rows, one or two blocks of tokens, and launches of at most one workgroup a CU with too few steps
    for two ahead; odd and even numbers of steps, K ending inside and on a step."""
    test_prompt_mlp(M, H, I, torch.float16)


AHEAD = [  # product, tokens, H, I, its tile, its steps
    (1, 128, 1279, 130, 0, 10), (1, 70, 1536, 130, 0, 12), (1, 128, 1409, 130, 0, 12), (1, 100, 1408, 130, 0, 11), (1, 70, 1283, 131, 0, 11),
    (1, 200, 640, 4099, 2, 10), (1, 160, 630, 5461, 2, 10), (1, 200, 832, 4099, 2, 13), (1, 200, 772, 4099, 2, 13), (1, 192, 2048, 5461, 2, 32),
    (2, 256, 1400, 1300, 0, 11), (2, 256, 1408, 1408, 0, 11), (2, 130, 3072, 3001, 2, 10), (2, 130, 3072, 3200, 2, 10), (2, 200, 772, 5461, 2, 11),
    (2, 200, 770, 5632, 2, 11),
]


@pytest.mark.parametrize("product,M,H,I,tile,steps", AHEAD)
def test_two_steps_ahead(product, M, H, I, tile, steps):
    """Launches of at most one workgroup a CU and ten steps and more, whose loads are two steps ahead: both tiles that have this, in either
    product, odd and even numbers of steps, K ending inside and on a step, the second product also in ranges of K."""
    from cats_amd import capi

    plan = capi.prompt_plan(product, M, H, I)
    assert (plan[0], plan[3], plan[5]) == (tile, steps, 2), plan
    test_prompt_mlp(M, H, I, torch.float16)


@pytest.mark.parametrize("M,H,I", [(5, 64, 9), (40, 304, 569), (130, 136, 1041)])
def test_what_lies_outside_a_row_stays_outside(M, H, I):
    """Infinities and NaN in one token or one weight row: reached by the columns torch reaches, whatever vector they share with others."""
    import flash_gemv  # noqa: F401

    x, wg, wu, wd = _draw(M, H, I, torch.float16)
    wd[1, 0], wd[2, I - 1], x[1, 0], x[2, H - 1] = float("inf"), float("nan"), float("nan"), float("inf")
    y = torch.ops.flash_gemv.cats_prompt_mlp(x, wg, wu, wd, 0.1)
    a = F.silu((x.double() @ wg.double().t()).half())
    a[a.abs() <= torch.tensor(0.1).half()] = 0
    want = (a * (x.double() @ wu.double().t()).half()).double() @ wd.double().t()
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())


def test_module_takes_it_and_leaves_it():
    from cats_amd.mlp import CatsMLP

    with torch.no_grad():
        torch.manual_seed(0)
        m = CatsMLP(264, 515, dead_threshold=0.05, dtype=torch.bfloat16, device="cuda").eval()
        for p in m.parameters():
            p.normal_(0, 0.05)
        m.prepare_decode(3)
        x = torch.randn(3, 21, 264, device="cuda").bfloat16()
        assert m._prompt_weights(x) is not None
        a = m(x)
        for other in (x.transpose(0, 1), x.float(), x[..., :256], x[..., :256].contiguous(), x[:0], x.repeat(1, 4000, 1)):
            assert m._prompt_weights(other) is None
        handle = m.up_proj.register_forward_hook(lambda *args: None)
        assert m._prompt_weights(x) is None
        b = m(x)
        handle.remove()
        # captured and replayed between eager work: the same values
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(x)
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                out = m(x)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, a)
            x.copy_(torch.randn_like(x))
            a = m(x)
    assert m._prompt_weights(x) is None  # gradients
    assert a.shape == x.shape and b.shape == x.shape


@pytest.mark.parametrize("M,H,I", [(33, 77, 2731), (5, 201, 5461), (64, 78, 3001), (65, 9, 2731), (40, 13, 21)])
def test_nothing_is_written_behind_y(M, H, I):
    """Columns that are no whole quad: y and the scratch end where the call says they end."""
    from cats_amd import capi

    x, wg, wu, wd = _draw(M, H, I, torch.bfloat16)
    want = torch.ops.flash_gemv.cats_prompt_mlp(x, wg, wu, wd, 0.1)
    L = capi.lib()
    size = L.cats_prompt_scratch_bytes(M, H, I)
    y, scratch = torch.full((M * H + 512,), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((size + 4096,), 7, dtype=torch.uint8, device="cuda")
    assert L.cats_prompt_mlp(*(capi._p(t) for t in (x, wg, wu, wd, y)), M, H, I, capi.BF16, 0.1, capi._p(scratch), size, capi._stream(x)) == 0
    assert torch.equal(y[:M * H].view(M, H), want) and bool((y[M * H:] == 7).all()) and bool((scratch[size:] == 7).all())
