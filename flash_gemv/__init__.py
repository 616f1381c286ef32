"""flash_gemv -- the CATS sparse-MLP decode ops, backed by hand-written gfx950 HIP kernels.

Drop-in for the reference package of the same name (flash_gemv/flash_gemv/__init__.py): the same 14
``torch.ops.flash_gemv.*`` ops, the same Python wrappers and the same four composites.  Importing it loads
``_C.so`` from this directory (as the reference does, __init__.py:29-36) and fails loudly if that library is
missing -- there is no PyTorch fallback.  Triton is not imported.

Layout conventions (they differ between entry points, as in the reference):
  ``flag_gemv_gemv_triton`` / ``flag_gemv_gemv_dejavu`` / ``flag_gemv_gemv_fuse_dejavu`` take ``Wgate`` as
  (H, I) and compute ``x @ Wgate``; every ``torch.ops`` gate op takes (I, H).  ``Wup`` is (I, H) and
  ``Wdownt`` is neuron-major (I, H) everywhere in this file.
"""
import importlib.machinery
import os.path as osp

import torch

library = "_C"
spec = importlib.machinery.PathFinder().find_spec(library, [osp.dirname(__file__)])
if spec is not None:
    torch.ops.load_library(spec.origin)
else:
    raise ImportError(
        f"Could not find module '{library}' in {osp.dirname(__file__)}: build it with `python -m cats_amd.build`"
    )

from .flash_gemv import (  # noqa: E402
    fuse_gemv_cmp,
    fuse_gemv_flag,
    fuse_gemv_flag_gemv,
    fuse_gemv_flag_gemv_gemv,
    fuse_gemv_gemv_gemv,
    fuse_gemv_flag_batch,
    fuse_gemv_flag_local,
    fuse_flag_gemv_local,
    atomic_gemv,
    flag_gemv_gemv_atomic,
    flag_gemv_gemv,
    flag_gemv_gemv_inner,
    flag_gemv_gemv_inner_fp32,
    flag_gemv_gemv_inner_bf16,
)
from .kernels import (  # noqa: E402
    gather_gemv_elemul_flag_3d,
    gather_transposed_gemv_flag_3d,
    mistral_mlp_partial_sparse,
    mistral_mlp_sparse_direct_index_2d,
)

__version__ = "0.0.1"


_PLAIN = {torch.Tensor, torch.nn.Parameter}


def _watched():
    """Whether tracing, a transform, a mode or a module hook is at work that has to see the single torch operations of a composite."""
    c, m = torch._C, torch.nn.modules.module
    return (c._is_tracing() or torch.compiler.is_compiling() or torch.is_autocast_enabled("cuda")
            or c._len_torch_dispatch_stack() or c._len_torch_function_stack()
            or c._functorch.peek_interpreter_stack() is not None or torch.autograd.forward_ad._current_level >= 0
            or m._global_forward_hooks or m._global_forward_pre_hooks)


def _gate_cols_fits(H, I, size):
    """Whether cats_mlp_gate_cols takes a layer of these sizes, whatever is kept: rows of up to 16 KiB go to the single-pass kernel, longer
    ones to a down pass whose groups hold 12288 neurons in LDS, 256 groups over the slabs of 1 KiB of a row.  The list's own groups hold
    the kept neurons only, so a call beyond this may still be one for the list."""
    row = H * size
    return I <= 1 << 18 if row <= 16384 else row <= 128 * 1024 and I <= 12288 * min(64, 256 // -(-row // 1024))


def _takes_gate_cols(x, Wgate, Wup, Wdownt, threshold):
    """Whether one call of the kernels, from the gate on, gives what the composite below gives: one row of a 16-byte aligned x,
    one type, all weights as they lie, a plain number as threshold, nothing that watches the operations.  Everything else keeps
    torch's gate."""
    if not (isinstance(threshold, (int, float)) and {type(x), type(Wgate), type(Wup), type(Wdownt)} <= _PLAIN
            and not _watched() and x.is_cuda and x.numel() == x.shape[-1] and x.is_contiguous() and Wgate.dim() == 2):
        return False
    H, I = shape = Wgate.shape
    d, sz, device = x.dtype, x.element_size(), x.device
    if not (d in (torch.float16, torch.bfloat16, torch.float32) and x.shape[-1] == H and H * sz % 16 == 0 and I * sz >= 16 and _gate_cols_fits(H, I, sz)
            and Wup.shape == shape[::-1] and Wdownt.shape == shape[::-1] and (x.data_ptr() | Wup.data_ptr() | Wdownt.data_ptr()) % 16 == 0):
        return False
    return all(w.dtype == d and w.device == device and w.is_contiguous() for w in (Wgate, Wup, Wdownt))


def flag_gemv_gemv_triton(x, Wgate, Wup, Wdownt, threshold):
    """Gate in torch (``x @ Wgate``, Wgate (H, I)), then sparse up / down (reference __init__.py:38-43).  One row is a
    single call of the kernels, gate included."""
    if x.dim() == 3 and _takes_gate_cols(x, Wgate, Wup, Wdownt, threshold):
        return torch.ops.flash_gemv.cats_mlp_gate_cols(x, Wgate, Wup, Wdownt, threshold)
    act_fn = torch.nn.SiLU()
    x_1 = act_fn(torch.matmul(x, Wgate))
    # flags = |x_1| > threshold, sparse up, sparse down: one call (the flags are derived where x_1 is read)
    return gemv_gemv_triton(x, x_1, Wup, Wdownt, threshold)


def gemv_gemv_triton(x, x_1, Wup, Wdownt, threshold):
    """Sparse up / down given the gate activations x_1 (reference __init__.py:45-48).  The flags |x_1| > threshold are
    derived inside the up kernel (same strict comparison, threshold rounded to x_1's dtype as torch does)."""
    return torch.ops.flash_gemv.cats_up_down(x, x_1.contiguous(), Wup, Wdownt, threshold)


def flag_gemv_gemv_dejavu(x, Wgate, Wup, Wdownt, threshold):
    """Index-list baseline: x (1, H) 2-D (reference __init__.py:50-54).  The list is what this composite is named for and not part of
    its result: one row goes from the gate to the output in the kernels, with the same roundings and no list, and nobody
    waits for its length."""
    if x.dim() == 2 and _takes_gate_cols(x, Wgate, Wup, Wdownt, threshold):
        return torch.ops.flash_gemv.cats_mlp_gate_cols(x, Wgate, Wup, Wdownt, threshold)
    act_fn = torch.nn.SiLU()
    x_1 = act_fn(torch.matmul(x, Wgate))
    (_, idx) = torch.nonzero(torch.abs(x_1) > threshold, as_tuple=True)
    return mistral_mlp_partial_sparse(x, x_1[0][idx], Wup, Wdownt, idx)


def flag_gemv_gemv_fuse_dejavu(x, Wgate, Wup, Wdownt, threshold):
    """Index-list variant with the element-wise multiply fused into up (reference __init__.py:56-60)."""
    act_fn = torch.nn.SiLU()
    x_1 = act_fn(torch.matmul(x, Wgate))
    (_, idx) = torch.nonzero(torch.abs(x_1) > threshold, as_tuple=True)
    return mistral_mlp_sparse_direct_index_2d(x, x_1[0][idx], Wup, Wdownt, idx)


def cats_mlp(x, Wgate, Wup, Wdownt, threshold):
    """Whole CATS MLP in two HIP launches: gate + SiLU + threshold + sparse up, then sparse down.

    x (B, 1, H) or (B, H); Wgate, Wup, Wdownt all (I, H) (Wdownt neuron-major).  No reference counterpart as a
    single call: it is flag_gemv_gemv_triton with the gate GEMV fused in and (I, H) gate weights.
    """
    return torch.ops.flash_gemv.cats_mlp(x, Wgate, Wup, Wdownt, threshold)


def cats_mlp_norm_residual(h, norm_weight, eps, Wgate, Wup, Wdownt, threshold):
    """h + CATS_MLP(norm_weight * rms_norm(h, eps)) in the same two launches as cats_mlp.

    The three module calls at the end of the reference's decoder layer (residual = h; h = post_attention_layernorm(h);
    h = residual + mlp(h), experiments/models/sparse_silu/ugly_utils.py:1036-1057) for decode, batch * seq <= 16.
    """
    return torch.ops.flash_gemv.cats_mlp_norm_residual(h, norm_weight, eps, Wgate, Wup, Wdownt, threshold)


def cats_mlp_norm_residual_norm(h, norm_weight, eps, Wgate, Wup, Wdownt, threshold, next_norm_weight, next_eps):
    """(out, next): out as cats_mlp_norm_residual, next = next_norm_weight * rms_norm(out, next_eps) from the same two
    launches -- the input_layernorm of the following decoder layer (ugly_utils.py:1016-1057), or the final norm."""
    return torch.ops.flash_gemv.cats_mlp_norm_residual_norm(h, norm_weight, eps, Wgate, Wup, Wdownt, threshold, next_norm_weight, next_eps)


def cats_mlp_stats(x, Wgate, Wup, Wdownt, threshold):
    """cats_mlp that also returns the (B, I) bool flags and the number of neurons fetched (int32 tensor)."""
    return torch.ops.flash_gemv.cats_mlp_stats(x, Wgate, Wup, Wdownt, threshold)


__all__ = [
    "fuse_gemv_cmp",
    "fuse_gemv_flag",
    "fuse_gemv_flag_gemv",
    "fuse_gemv_flag_gemv_gemv",
    "fuse_gemv_gemv_gemv",
    "fuse_gemv_flag_batch",
    "fuse_gemv_flag_local",
    "fuse_flag_gemv_local",
    "atomic_gemv",
    "flag_gemv_gemv_atomic",
    "flag_gemv_gemv",
    "flag_gemv_gemv_inner",
    "flag_gemv_gemv_inner_fp32",
    "flag_gemv_gemv_inner_bf16",
    "flag_gemv_gemv_triton",
    "gemv_gemv_triton",
    "flag_gemv_gemv_fuse_dejavu",
    "flag_gemv_gemv_dejavu",
    "gather_gemv_elemul_flag_3d",
    "gather_transposed_gemv_flag_3d",
    "mistral_mlp_partial_sparse",
    "mistral_mlp_sparse_direct_index_2d",
    "cats_mlp",
    "cats_mlp_stats",
    "cats_mlp_norm_residual",
    "cats_mlp_norm_residual_norm",
]
