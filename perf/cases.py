"""What the speed of this framework is measured on: the calls a decode program makes, from the smallest layer to the largest.

A case is one call (or one composite of calls) of the public Python surface -- ``flash_gemv``, ``cats_amd.mlp.CatsMLP``
and ``cats_amd.decoder.LlamaDecoder`` -- at one layer shape, batch, data type and sparsity.  ``listed()`` names twelve of
them, ``draw()`` gives others of the same ranges.

Fields of a case: ``op`` (below), ``H`` hidden and ``I`` intermediate size, ``B`` batch rows (for ``prefill`` the prompt
tokens), ``dtype``, ``sparsity`` (share of the gate activations below the threshold, per row), ``corr`` (pairwise
correlation of the batch rows) and ``heavy`` (gate rows scaled by log-normal(0, 0.5) factors).  ``decode`` has ``layers``,
``heads``, ``vocab`` and ``context`` (prompt tokens in the KV cache) besides.

  mlp      flash_gemv.cats_mlp                           whole sparse MLP, neuron-major down weights (sp_method 3)
  tail     flash_gemv.cats_mlp_norm_residual_norm        the layer tail: norm, MLP, residual, next norm
  atomic   flash_gemv.flag_gemv_gemv_atomic              whole MLP added into a zeroed fp32 buffer
  inner    flash_gemv.flag_gemv_gemv_inner{,_bf16,_fp32} whole MLP with nn.Linear's (H, I) down weight (sp_method 1)
  module2  CatsMLP.forward, sp_method 2                  gate projection, then the sparse up / down call
  list     flash_gemv.flag_gemv_gemv_dejavu              the index-list composite, (H, I) gate weight
  prefill  CatsMLP.forward on a prompt                   the thresholded MLP over many tokens
  decode   LlamaDecoder.forward under a HIP graph        one greedy step of a model, logits out
"""
import functools
import math

import numpy as np
import torch

import flash_gemv
from cats_amd.decoder import DecoderConfig, LlamaDecoder
from cats_amd.mlp import CatsMLP

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}
STD = 0.02  # of every weight; x has unit variance


def listed():
    def case(name, op, H, I, B, dtype, sparsity=0.5, corr=0.5, heavy=False, **more):
        return {"name": name, "op": op, "H": H, "I": I, "B": B, "dtype": dtype, "sparsity": sparsity, "corr": corr, "heavy": heavy, **more}

    return [
        # a toy or test model, one token: launches and the call itself are all there is
        case("small layer", "mlp", 512, 1024, 1, "fp16"),
        # single-stream decoding of a 7B model, the headline layer
        case("7B layer - 1 row", "mlp", 4096, 11008, 1, "fp16"),
        # the same in the layout and the call that need no prepared weights, in a checkpoint's fp32
        case("7B layer - 1 row - fp32 - HF layout", "inner", 4096, 11008, 1, "fp32"),
        # the reference's own decode path (gate by the module, sparse up / down) with a wider, heavy-tailed layer
        case("wide 7B layer - 1 row - module", "module2", 4096, 14336, 1, "bf16", 0.7, heavy=True),
        # the reference's index-list baseline, which its users compare with
        case("7B layer - 1 row - index list", "list", 4096, 11008, 1, "fp16"),
        # a handful of streams or beams: the union of the masks is nearly dense
        case("7B layer - 4 rows", "mlp", 4096, 11008, 4, "fp16"),
        # a small server's batch over weights as they come from a checkpoint
        case("wide 7B layer - 8 rows - HF layout", "inner", 4096, 14336, 8, "bf16", 0.7, heavy=True),
        # the largest batch the path takes
        case("wide 7B layer - 16 rows", "mlp", 4096, 14336, 16, "bf16"),
        # sizes no kernel was shaped for: a row that is no whole number of blocks, an odd number of neurons, odd batch
        case("ragged layer - 3 rows", "mlp", 3080, 8191, 3, "bf16", 0.6),
        # a 70B layer, a server's batch: the largest matrices
        case("70B layer - 8 rows", "mlp", 8192, 28672, 8, "fp16", 0.7),
        # the prompt of a 7B model goes through the same module before decoding starts
        case("7B layer - prompt", "prefill", 4096, 11008, 512, "fp16"),
        # one token of a 7B-architecture model, four of its layers with attention, norms and the output head around them
        case("7B model step", "decode", 4096, 11008, 1, "fp16", layers=4, heads=32, vocab=32000, context=256),
    ]


MOST_WEIGHTS = 8192 * 28672 * 2  # bytes of one matrix of the largest listed layer


def draw(rng):
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    op = rng.choice(["mlp", "mlp", "mlp", "mlp", "tail", "tail", "atomic", "inner", "inner", "module2", "list", "prefill", "decode"])
    dtype = rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"])
    H = 8 * round(log_uniform(256, 8192) / 8)
    if rng.random() < 0.5:  # half of all models have round sizes
        H = max(256, 256 * round(H / 256))
    I = round(H * rng.uniform(1.5, 4.0))
    B = rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 8, 11, 16])
    more = {}
    if op == "tail":
        H = 32 * round(H / 32)
        B = min(B, 4) if dtype == "fp32" else B  # the call keeps the normed rows of a pass on chip: 128 KiB
    if op == "inner":
        I = 8 * round(I / 8)
    if op in ("list", "module2"):
        B = 1
    if op in ("prefill", "decode"):
        dtype = rng.choice(["fp16", "bf16"])
    if op == "prefill":
        H, I, B = min(H, 4096), min(I, 11008), round(log_uniform(2, 512))
    if op == "decode":
        H = 128 * max(2, round(min(H, 4096) / 128))
        I = min(round(H * rng.uniform(2.0, 3.5)), 11008)
        B = rng.choice([1, 1, 2, 4])
        more = {"layers": rng.randint(1, 4), "heads": H // 128, "vocab": rng.choice([8000, 32000]), "context": round(log_uniform(16, 480))}
    I = min(I, MOST_WEIGHTS // (H * BYTES[dtype]) // 8 * 8)
    return {"op": op, "H": H, "I": I, "B": B, "dtype": dtype, "sparsity": round(rng.uniform(0.3, 0.9), 2), "corr": rng.choice([0.0, 0.5]),
            "heavy": op != "decode" and rng.random() < 0.3, **more}


# ---- inputs ----------------------------------------------------------------------------------------------------------


def _rows(g, B, H, corr):
    """B rows of unit variance with pairwise correlation `corr`: streams that continue similar texts."""
    return math.sqrt(corr) * torch.randn(1, H, generator=g, device="cuda") + math.sqrt(1 - corr) * torch.randn(B, H, generator=g, device="cuda")


def _weights(g, shape, dtype):
    return (torch.randn(shape, generator=g, device="cuda") * STD).to(dtype)


def _gate_weight(g, case, dtype):
    w = torch.randn(case["I"], case["H"], generator=g, device="cuda") * STD
    if case["heavy"]:
        w *= torch.exp(0.5 * torch.randn(case["I"], 1, generator=g, device="cuda"))
    return w.to(dtype)


def _threshold(g, wg, sparsity):
    """The `sparsity` quantile of |SiLU(gate)| over calibration rows, as a user's calibration run finds it."""
    cal = torch.randn(32, wg.shape[1], generator=g, device="cuda")
    a = torch.nn.functional.silu(cal @ wg.float().t()).abs().flatten()
    return float(torch.kthvalue(a, max(1, round(sparsity * a.numel()))).values)


def _prepare_decode(case, seed, dtype):
    """A model with its prompt in the KV cache and one decode step captured into a HIP graph, as generate_greedy does."""
    cfg = DecoderConfig(hidden_size=case["H"], intermediate_size=case["I"], num_layers=case["layers"], num_heads=case["heads"],
                        vocab_size=case["vocab"], max_len=512)
    with torch.no_grad():
        model = LlamaDecoder(cfg, dtype, "cuda", seed=seed).eval()
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        # In a trained model the hidden state is larger than what one layer adds to it.  At initialisation it is smaller,
        # and then a tie at one threshold decides a visible part of the logits.
        model.embed_tokens.weight.mul_(400)
        for layer in model.layers:  # the gate's inputs are normed rows
            layer.mlp.dead_threshold = _threshold(g, layer.mlp.gate_proj.weight, case["sparsity"])
        model.set_mlp_mode("cats_fused_next")
        B, P = case["B"], case["context"]
        prompt = torch.randint(0, cfg.vocab_size, (B, P), generator=g, device="cuda")
        tok = torch.randint(0, cfg.vocab_size, (B, 1), generator=g, device="cuda")
        pos = torch.full((1,), P, dtype=torch.int64, device="cuda")
        model.reset_cache(B)
        model(prompt, torch.arange(P, device="cuda"))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(tok, pos)
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                logits = model(tok, pos)
        torch.cuda.current_stream().wait_stream(side)
    return {"op": "decode", "model": model, "graph": graph, "inputs": (tok, pos), "logits": logits}


def prepare(case, seed):
    op, H, I, B, dtype = case["op"], case["H"], case["I"], case["B"], DTYPES[case["dtype"]]
    if op == "decode":
        return _prepare_decode(case, seed, dtype)
    g = torch.Generator(device="cuda").manual_seed(seed)
    wg = _gate_weight(g, case, dtype)
    s = {"op": op, "dtype": case["dtype"], "t": _threshold(g, wg, case["sparsity"])}
    if op in ("module2", "prefill"):
        with torch.no_grad():
            m = CatsMLP(H, I, dead_threshold=s["t"], dtype=dtype, device="cuda").eval()
            m.gate_proj.weight.copy_(wg)
            m.up_proj.weight.copy_(_weights(g, (I, H), dtype))
            m.down_proj.weight.copy_(_weights(g, (H, I), dtype))
            s["module"] = m.prepare_decode(2 if op == "module2" else 3)
        s["x"] = (_rows(g, B, H, case["corr"]).to(dtype)).view((B, 1, H) if op == "module2" else (1, B, H))
        return s
    s["wg"] = wg.t().contiguous() if op == "list" else wg
    s["wu"] = _weights(g, (I, H), dtype)
    s["wd"] = _weights(g, (H, I) if op == "inner" else (I, H), dtype)
    x = _rows(g, B, H, case["corr"])
    s["x"] = x.to(dtype) if op == "list" else x.to(dtype).view(B, 1, H)
    if op == "tail":
        s["norms"] = [(1 + 0.1 * torch.randn(H, generator=g, device="cuda")).to(dtype) for _ in range(2)]
    if op == "atomic":
        s["out"] = torch.empty(B, H, dtype=torch.float32, device="cuda")
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------

INNER = {"fp16": flash_gemv.flag_gemv_gemv_inner, "bf16": flash_gemv.flag_gemv_gemv_inner_bf16, "fp32": flash_gemv.flag_gemv_gemv_inner_fp32}


@torch.no_grad()
def run(s):
    op = s["op"]
    if op == "decode":
        s["graph"].replay()
        return s["logits"]
    if op in ("module2", "prefill"):
        return s["module"](s["x"])
    x, wg, wu, wd, t = s["x"], s["wg"], s["wu"], s["wd"], s["t"]
    if op == "mlp":
        return flash_gemv.cats_mlp(x, wg, wu, wd, t)
    if op == "tail":
        return flash_gemv.cats_mlp_norm_residual_norm(x, s["norms"][0], 1e-5, wg, wu, wd, t, s["norms"][1], 1e-5)
    if op == "inner":
        return INNER[s["dtype"]](x, wg, wu, wd, t)
    if op == "list":
        return flash_gemv.flag_gemv_gemv_dejavu(x, wg, wu, wd, t)
    s["out"].zero_()  # the contract of the fp32-accumulate call: it adds into what is there
    flash_gemv.flag_gemv_gemv_atomic(x, wg, wu, wd, s["out"], t)
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _kept(B, sparsity, corr, heavy, H):
    """Share of the neurons that some batch row keeps, by simulation of the inputs' distribution."""
    rng = np.random.RandomState(1)
    n = 20000
    sigma = STD * math.sqrt(H) * (np.exp(0.5 * rng.randn(n, 1)) if heavy else np.ones((n, 1)))

    def silu(g):
        return np.abs(g / (1 + np.exp(-np.clip(g, -80, 80))))

    t = np.quantile(silu(sigma * rng.randn(n, 1)), sparsity)
    g = math.sqrt(corr) * rng.randn(n, 1) + math.sqrt(1 - corr) * rng.randn(n, B)
    return float((silu(sigma * g) > t).any(axis=1).mean())


def work(case):
    op, H, I, B, sz = case["op"], case["H"], case["I"], case["B"], BYTES[case["dtype"]]
    if op == "prefill":  # dense: every matrix once, x and y once; the three products
        return {"bytes": sz * (3 * H * I + 2 * B * H), "flops": 6 * B * H * I}
    kept = _kept(B, case["sparsity"], case["corr"], case["heavy"], H)
    rows = I * (1 + kept + (1 if op == "inner" else kept))  # rows of the three matrices that have to be read
    layer = {"bytes": sz * (rows * H + 2 * B * H), "flops": 2 * B * H * rows}
    if op != "decode":
        return layer
    kv = 2 * B * case["context"] * H * sz
    return {"bytes": case["layers"] * (layer["bytes"] + 4 * H * H * sz + kv) + sz * case["vocab"] * (H + B),
            "flops": case["layers"] * (layer["flops"] + 8 * B * H * H + 4 * B * H * case["context"]) + 2 * B * case["vocab"] * H}


def tolerance(case):
    """Four times the distance from the same arithmetic with its sums in 64 bits (fp16 3.8e-4 to 4.3e-4, bf16 3.0e-3 to
    4.0e-3, fp32 3.6e-7), and one tie: a neuron whose activation the gate sum puts a rounding step above the threshold or
    on it is kept by one order of summation and dropped by another, which moves the output by about half the share of one
    kept neuron.  A decode step meets ties in every layer: measured over 1 to 4 layers against attention in 32 bits,
    up to 6.6e-3 in fp16 and 1.2e-2 in bf16."""
    if case["op"] == "decode":
        return {"rel": {"fp16": 2e-2, "bf16": 3e-2}[case["dtype"]]}
    tie = 0.5 / math.sqrt(case["I"] * (1 - case["sparsity"]) * case["B"])
    return {"rel": {"fp16": 1.6e-3 + tie, "bf16": 1.4e-2 + tie, "fp32": 5e-6}[case["dtype"]]}
