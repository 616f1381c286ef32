"""The projection and attention kernels of a decode step against the torch operations they stand for, in float64 on the CPU."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2 ** -11, torch.bfloat16: 2 ** -8, torch.float32: 2 ** -24}


def _randn(g, *shape, dtype, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def _check(got, want, dtype, terms):
    """Rounding of the stored value, and fp32 sums of `terms` products of the size of the result's own scale."""
    tol = (2 * EPS[dtype] + terms * 2 ** -24) * (want.abs() + want.std() + 1e-3)
    assert bool((got.cpu().double() - want).abs().le(tol).all()), float(((got.cpu().double() - want).abs() / tol).max())


@pytest.mark.parametrize("B,K,N,dtype", [
    (1, 8, 1, torch.float16), (1, 4096, 4096, torch.float16), (1, 4096, 1001, torch.bfloat16), (2, 264, 33, torch.float16),
    (3, 1000, 77, torch.bfloat16), (4, 4096, 515, torch.float16), (8, 3080, 130, torch.bfloat16), (1, 8200, 19, torch.float16),
    (1, 516, 40, torch.float32), (4, 4096, 64, torch.float32), (8, 1028, 9, torch.float32)])
@pytest.mark.parametrize("norm", [False, True])
def test_linear(B, K, N, dtype, norm):
    import flash_gemv  # noqa: F401

    g = torch.Generator().manual_seed(B + K + N)
    x, w, nw = _randn(g, B, 1, K, dtype=dtype, scale=2.0), _randn(g, N, K, dtype=dtype, scale=0.02), (1 + 0.1 * torch.randn(K, generator=g)).to(dtype)
    out = torch.ops.flash_gemv.cats_linear(x.cuda(), nw.cuda() if norm else None, 1e-5, w.cuda())
    xr = x.double()
    if norm:
        xr = (nw.double() * (xr * torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + 1e-5)).to(dtype).double()).to(dtype).double()
    want = xr @ w.double().t()
    if norm:  # a normed value that sits on a rounding tie may go either way: half a step of each term, added as random signs
        tie = 4 * EPS[dtype] * (xr.pow(2) @ w.double().pow(2).t()).sqrt()
        assert bool(((out.cpu().double() - want).abs() <= tie + (2 * EPS[dtype] + K * 2 ** -24) * (want.abs() + want.std() + 1e-3 if N > 1 else 1)).all())
    else:
        _check(out, want, dtype, K) if N > 1 else torch.testing.assert_close(out.cpu().double(), want, rtol=4 * EPS[dtype], atol=1e-3)


@pytest.mark.parametrize("B,K,N,dtype", [
    (3, 64, 8, torch.float16), (5, 64, 2000, torch.bfloat16), (4, 512, 4099, torch.float16), (8, 576, 7, torch.bfloat16), (3, 1024, 6001, torch.float16),
    (7, 1088, 2500, torch.bfloat16), (3, 2048, 4105, torch.float16), (6, 2112, 300, torch.float16), (8, 4608, 100, torch.bfloat16),
    (4, 4672, 4200, torch.float16), (3, 8192, 520, torch.bfloat16), (8, 8192, 40, torch.float16), (3, 9216, 40, torch.float16), (4, 9280, 24, torch.float16)])
@pytest.mark.parametrize("norm", [False, True])
def test_linear_on_the_matrix_cores(B, K, N, dtype, norm):
    """One to nine steps a wave in one register set and five to nine in two (9280: too long, a wave a row), eight to one tiles a round in up to
    two rounds, a last tile that is not whole, fewer tiles than CUs and several each."""
    test_linear(B, K, N, dtype, norm)


@pytest.mark.parametrize("B,K,N,dtype", [
    (8, 512, 50001, torch.float16), (3, 448, 36000, torch.bfloat16), (5, 1024, 32000, torch.float16), (7, 1024, 24001, torch.bfloat16),
    (4, 2048, 16001, torch.float16), (3, 1536, 14003, torch.bfloat16), (4, 2048, 12001, torch.bfloat16)])
@pytest.mark.parametrize("norm", [False, True])
def test_linear_of_many_rounds(B, K, N, dtype, norm):
    """Output heads on the matrix cores: three and four rounds of eight, four and two tiles, so that registers are refilled with what is used and
    each half of the sums is written again; the last round whole and not."""
    test_linear(B, K, N, dtype, norm)


@pytest.mark.parametrize("B,K,N,dtype", [(6, 512, 45003, torch.float16), (8, 1024, 24001, torch.bfloat16), (3, 2048, 12005, torch.float16),
                                         (4, 4672, 4100, torch.bfloat16), (2, 1024, 4099, torch.float16), (1, 4096, 1001, torch.bfloat16), (3, 1000, 77, torch.float32)])
def test_linear_with_a_residual(B, K, N, dtype):
    """What the product is added to, by the C interface (the operators add to it at square matrices only): many rounds, two register sets, a wave a row."""
    from cats_amd import capi

    g = torch.Generator().manual_seed(B + K + N)
    x, w, r = _randn(g, B, K, dtype=dtype), _randn(g, N, K, dtype=dtype, scale=1 / math.sqrt(K)), _randn(g, B, N, dtype=dtype)
    xd, wd, rd, out = x.cuda(), w.cuda(), r.cuda(), torch.empty(B, N, dtype=dtype, device="cuda")
    at = lambda t: ctypes.c_void_p(t.data_ptr())
    assert capi.lib().cats_linear(at(xd), None, ctypes.c_float(0.0), at(wd), at(rd), at(out), B, K, N, capi.DTYPE_CODE[dtype],
                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    _check(out, r.double() + x.double() @ w.double().t(), dtype, K)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("K,N", [(256, 1000), (1024, 33), (1032, 4099), (2048, 70), (2056, 515)])
@pytest.mark.parametrize("norm", [False, True])
def test_linear_over_short_rows(B, K, N, norm):
    """Blocks of two, four and eight chunks of a row, whole and not, at the rows a wave that goes with them."""
    test_linear(B, K, N, torch.float16, norm)


@pytest.mark.parametrize("offset", [8, 56, 64])
def test_linear_where_the_matrix_starts(offset):
    """A matrix that starts inside a cache line (8, 56 elements behind its start) keeps the wave-per-row kernel; one that starts on the next line does not."""
    import flash_gemv  # noqa: F401

    g = torch.Generator(device="cuda").manual_seed(offset)
    buf = torch.randn(700 * 640 + 64, generator=g, device="cuda").half() * 0.05
    w, x = buf[offset:offset + 700 * 640].view(700, 640), torch.randn(4, 640, generator=g, device="cuda").half()
    _check(torch.ops.flash_gemv.cats_linear(x, None, 1e-5, w), x.cpu().double() @ w.cpu().double().t(), torch.float16, 640)


def _reference(h, x, wq, wk, wv, wo, kc, vc, cos, sin, pos):
    B, heads, _, hd = kc.shape
    shp = (B, heads, hd)
    d = lambda t: t.double()
    q, k, v = (d(x).view(B, -1) @ d(w).t() for w in (wq, wk, wv))
    q, k, v = q.view(shp), k.view(shp), v.view(shp)
    half = lambda t: torch.cat((-t[..., hd // 2:], t[..., : hd // 2]), -1)
    q, k = (t * d(cos)[pos] + half(t) * d(sin)[pos] for t in (q, k))
    kc, vc = kc.clone(), vc.clone()
    kc[:, :, pos], vc[:, :, pos] = k.to(kc.dtype), v.to(vc.dtype)
    att = torch.softmax((d(kc[:, :, : pos + 1]) @ q.unsqueeze(-1)).squeeze(-1) / math.sqrt(hd), -1)
    o = (att.unsqueeze(-2) @ d(vc[:, :, : pos + 1])).reshape(B, -1)
    return d(h).view(B, -1) + o @ d(wo).t(), kc, vc


def _attention_step(B, heads, hd, max_len, pos, dtype, norm=False, inside=None):
    """inside: which of the three matrices starts inside a cache line."""
    import flash_gemv  # noqa: F401

    H = heads * hd
    g = torch.Generator().manual_seed(H + pos)
    h, x = _randn(g, B, 1, H, dtype=dtype, scale=2.0), _randn(g, B, 1, H, dtype=dtype)
    ws = [_randn(g, H, H, dtype=dtype, scale=1 / math.sqrt(H)) for _ in range(4)]
    kc, vc = (_randn(g, B, heads, max_len, hd, dtype=dtype) for _ in range(2))
    kc[:, :, pos:], vc[:, :, pos:] = float("inf"), float("nan")   # what has not been written yet takes no part
    ang = torch.outer(torch.arange(max_len).float(), 1.0 / (10000.0 ** (torch.arange(0, hd, 2).float() / hd)))
    emb = torch.cat((ang, 0.7 * ang + 0.3), -1)  # the two elements that are mixed turn by angles of their own
    cos, sin = emb.cos().to(dtype), emb.sin().to(dtype)
    kd, vd = kc.cuda(), vc.cuda()
    p = torch.tensor([pos], device="cuda")
    nw = (1 + 0.1 * torch.randn(H, generator=g)).to(dtype) if norm else None
    on_gpu = [w.cuda() for w in ws]
    if inside is not None:
        buf = torch.empty(H * H + 64, dtype=dtype, device="cuda")
        on_gpu[inside] = buf[8:8 + H * H].view(H, H).copy_(on_gpu[inside])
    args = (h.cuda(), x.cuda(), nw.cuda() if norm else None, 1e-5, *on_gpu, kd, vd, cos.cuda(), sin.cuda())
    out = torch.ops.flash_gemv.cats_attention_step(*args, p)
    xr = x
    if norm:
        xr = (x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5)).to(dtype)
        xr = (nw.double() * xr.double()).to(dtype)
    want, kw, vw = _reference(h, xr, *ws, kc, vc, cos, sin, pos)
    # attention is rounded once before the output projection: half a step of each of its H terms, added as random signs
    _check(out.view(B, H), want, dtype, 4 * H)
    _check(kd[:, :, pos], kw[:, :, pos].double(), dtype, 2 * H)
    _check(vd[:, :, pos], vw[:, :, pos].double(), dtype, 2 * H)
    assert torch.equal(kd[:, :, :pos].cpu(), kc[:, :, :pos]) and torch.equal(vd[:, :, :pos].cpu(), vc[:, :, :pos])
    assert torch.equal(kd[:, :, pos + 1:].cpu(), kc[:, :, pos + 1:])
    for bad in (-1, max_len):   # a position outside the cache stores nothing
        before = kd.clone()
        out = torch.ops.flash_gemv.cats_attention_step(*args, torch.tensor([bad], device="cuda"))
        assert bool(out.isnan().all()) and torch.equal(kd, before)


@pytest.mark.parametrize("B,heads,hd,max_len,pos,dtype", [
    (1, 2, 16, 4, 0, torch.float16), (1, 3, 32, 40, 39, torch.bfloat16), (2, 4, 64, 512, 63, torch.float16), (1, 2, 128, 300, 255, torch.float16),
    (4, 8, 128, 512, 256, torch.bfloat16), (8, 2, 128, 700, 699, torch.float16), (3, 2, 256, 130, 100, torch.bfloat16),
    (1, 4, 128, 1100, 1030, torch.float32), (2, 3, 8, 33, 32, torch.float32), (1, 32, 128, 512, 480, torch.float16)])
@pytest.mark.parametrize("norm", [False, True])
def test_attention_step(B, heads, hd, max_len, pos, dtype, norm):
    _attention_step(B, heads, hd, max_len, pos, dtype, norm)


@pytest.mark.parametrize("B,heads,hd,dtype", [(3, 6, 16, torch.float16), (4, 4, 16, torch.bfloat16), (5, 3, 64, torch.float16), (3, 20, 128, torch.bfloat16),
                                              (8, 16, 256, torch.float16), (4, 32, 128, torch.float16), (3, 40, 128, torch.bfloat16), (2, 4, 64, torch.bfloat16)])
@pytest.mark.parametrize("norm", [False, True])
def test_attention_step_of_batches(B, heads, hd, dtype, norm):
    """The three projections in tiles of four pairs of a head: one to several tiles a workgroup, of one matrix or of two, rows of 96 elements
    (no whole cache lines) and two rows with a wave a row; 5120 elements in two register sets."""
    _attention_step(B, heads, hd, 50, 33, dtype, norm)


@pytest.mark.parametrize("inside", [0, 1, 2])
def test_attention_step_where_the_matrices_start(inside):
    """One of the three matrices inside a cache line: a wave a row for all three."""
    _attention_step(4, 5, 128, 50, 33, torch.float16, inside=inside)


@pytest.mark.parametrize("B,heads,hd,max_len,pos", [(5, 13, 16, 40, 20), (5, 13, 128, 600, 513), (1, 20, 128, 600, 255), (1, 20, 128, 600, 256),
                                                    (1, 20, 128, 600, 511), (8, 8, 16, 3, 2), (8, 8, 128, 1100, 900), (8, 8, 128, 1100, 1023)])
def test_attention_with_and_without_workgroups_that_fetch_ahead(B, heads, hd, max_len, pos):
    """65 of 256 CUs attending: none fetch the next weights or the slots of a turn ahead; 20 and 64: the rest do, also from a number that is
    no multiple of eight, up to 960 slots of 64 heads of 128; turns of 256 slots, one to five of them, ending on and behind a turn."""
    _attention_step(B, heads, hd, max_len, pos, torch.float16)


@pytest.mark.parametrize("B,mode", [(1, "cats_fused_next"), (4, "cats_fused_next"), (2, "cats_fused"), (3, "cats"), (1, "dense")])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_step_matches_torch_operations(B, mode, dtype):
    """The model's step through the kernels and through the torch operations (a hook on the output head keeps it there)."""
    from cats_amd import decoder as dec

    cfg = dec.DecoderConfig(hidden_size=512, intermediate_size=1000, num_layers=2, num_heads=4, vocab_size=503, max_len=64)
    with torch.no_grad():
        model = dec.LlamaDecoder(cfg, dtype, "cuda", seed=0, init_std=0.05).eval()
        model.embed_tokens.weight.mul_(40)
        model.set_mlp_mode(mode)
        g = torch.Generator(device="cuda").manual_seed(5)
        prompt = torch.randint(0, 503, (B, 9), generator=g, device="cuda")
        tok, pos = prompt[:, :1].contiguous(), torch.full((1,), 9, device="cuda")

        def step(hook):
            model.reset_cache(B)
            model(prompt, torch.arange(9, device="cuda"))
            handle = model.lm_head.register_forward_hook(lambda *a: None) if hook else None
            assert model._takes_step(model.embed_tokens(tok), pos) == (not hook)
            out = model(tok, pos)
            if handle:
                handle.remove()
            return out.double(), model.layers[1].self_attn.k_cache[:, :, 9].double()

        for a, b in zip(step(False), step(True)):
            assert float((a - b).norm() / b.norm()) < 16 * EPS[dtype]  # two layers of roundings, at most eight steps each


def test_step_leaves_watched_calls_to_torch():
    from cats_amd import decoder as dec

    cfg = dec.DecoderConfig(hidden_size=256, intermediate_size=512, num_layers=1, num_heads=4, vocab_size=53, max_len=16)
    model = dec.LlamaDecoder(cfg, torch.float16, "cuda", seed=0).eval()
    model.reset_cache(1)
    h, pos = torch.randn(1, 1, 256, device="cuda").half(), torch.zeros(1, dtype=torch.int64, device="cuda")
    assert not model._takes_step(h, pos)                                       # gradients
    with torch.no_grad():
        assert model._takes_step(h, pos)
        assert not model._takes_step(h.expand(9, 1, 256).contiguous(), pos)    # rows, and a cache of another batch
        assert not model._takes_step(h.expand(2, 1, 256).contiguous(), pos)
        assert not model._takes_step(h, pos.int()) and not model._takes_step(h.expand(1, 2, 256).contiguous(), pos)
        with torch.autocast("cuda"):
            assert not model._takes_step(h, pos)
        handle = model.layers[0].self_attn.q_proj.register_forward_hook(lambda *a: None)
        assert not model._takes_step(h, pos)
        handle.remove()
        model.layers[0].self_attn.q_proj.weight.data = torch.randn(256, 256, device="cuda").half().t()
        assert not model._takes_step(h, pos)
