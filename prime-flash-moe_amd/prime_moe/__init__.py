"""prime_moe for MI355X (gfx950): the fused-MoE forward behind the reference's op surface.

Drop-in for the reference package (prime_moe/__init__.py:1-122 and the op schemas of
prime_moe/csrc/torch_interface.cpp:271-324): the same three ``prime_moe::`` torch-library
ops with the same schemas, the same Python wrappers returning ``out``, ``BLOCK`` and
``pack_scales_blocked``.  The schemas and fake impls are defined here, the implementations in
``_torch_ops.so`` (csrc/torch_ops.cpp), which calls hand-written HIP kernels through the C ABI
of ``libprime_moe_hip.so`` (``include/prime_moe_hip.h``); the PyTorch-ROCm device is dispatch
key ``CUDA``.  Argument checks raise ``RuntimeError`` for the conditions the reference's
``TORCH_CHECK``s reject (torch_interface.cpp:85-87, :132-155, :208-241).

Extras that the reference leaves to its callers: a fake impl for ``moe_align`` (so all
three ops trace), :func:`quantize_mx`, the OCP-MX quantiser in front of the mxfp8 op, and
:func:`route`, the router front-end (top-k + softmax + ``moe_align``) in front of both.
"""
from __future__ import annotations

import torch

BLOCK = 32  # MX scale block size

_LIB = torch.library.Library("prime_moe", "FRAGMENT")
_LIB.define(
    "fused_moe_bf16(Tensor x, Tensor w, Tensor w2, Tensor sorted_token_ids, Tensor expert_ids, "
    "Tensor num_tokens_post_padded, Tensor topk_weights, Tensor(a!) out, int top_k, int block_m, "
    "int block_n, int warp_n, int stages, int bpc, int cpc, bool split=True) -> ()"
)
_LIB.define(
    "fused_moe_mxfp8(Tensor x, Tensor x_scales, Tensor w, Tensor w_scales, Tensor w2, "
    "Tensor w2_scales, Tensor sorted_token_ids, Tensor expert_ids, Tensor num_tokens_post_padded, "
    "Tensor topk_weights, Tensor(a!) out, int top_k, int block_m, int block_n, int warp_n, "
    "int stages, int bpc, bool split=True) -> ()"
)
_LIB.define("moe_align(Tensor topk_ids, int num_experts, int block_m, int bpc) -> (Tensor, Tensor, Tensor)")


try:
    # host side of the ops (csrc/torch_ops.cpp): registers their CUDA-key implementations, does the argument checks
    from . import _torch_ops
except ImportError as _err:
    # Not built, or built against another torch or library: the package still imports (its build module has to), and
    # everything that needs the native code raises.
    class _Unavailable:
        def __init__(self, reason):
            self._reason = reason

        def _raise(self, *args, **kwargs):
            raise RuntimeError(f"prime_moe: _torch_ops.so cannot be loaded ({self._reason}). Build the native code "
                               "first: python prime-flash-moe_amd/prime_moe/build.py (there is no fallback path).")

        def __getattr__(self, name):
            return self._raise

    _torch_ops = _Unavailable(str(_err))
    for _op in ("moe_align", "fused_moe_bf16", "fused_moe_mxfp8"):
        _LIB.impl(_op, _torch_ops._raise, "CUDA")


# ------------------------------------------------------------------------------- moe_align

def align_sizes(n: int, num_experts: int, block_m: int, bpc: int):
    """(pad_to, max_padded, max_blocks) as torch_interface.cpp:88-91 computes them."""
    pad_to = block_m * bpc
    max_padded = (n + num_experts * (pad_to - 1) + pad_to - 1) // pad_to * pad_to
    return pad_to, max_padded, max_padded // block_m


def _validate_align(topk_ids, num_experts, block_m, bpc, placement: bool = True) -> None:
    """Argument checks of the op.  `placement=False` skips the device check (what is left can then be
    exercised with CPU tensors)."""
    _torch_ops.validate_align(topk_ids, num_experts, block_m, bpc, placement)


def _moe_align_fake(topk_ids, num_experts, block_m, bpc):
    _, max_padded, max_blocks = align_sizes(topk_ids.numel(), num_experts, block_m, bpc)
    mk = lambda n: torch.empty((n,), dtype=torch.int32, device=topk_ids.device)
    return mk(max_padded), mk(max_blocks), mk(1)


# ------------------------------------------------------------------------------- fused_moe_bf16

def _validate_bf16(x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights, out,
                   top_k, block_m, block_n, warp_n, stages, bpc, cpc, split, placement: bool = True) -> None:
    """Argument checks of the op.  `placement=False` skips the device and alignment checks."""
    _torch_ops.validate_bf16(x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights, out,
                             top_k, block_m, block_n, warp_n, stages, bpc, cpc, split, placement)


def _fused_moe_bf16_fake(x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights,
                         out, top_k, block_m, block_n, warp_n, stages, bpc, cpc, split=True):
    return None


# ------------------------------------------------------------------------------- fused_moe_mxfp8

def _validate_mxfp8(x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids,
                    num_tokens_post_padded, topk_weights, out, top_k, block_m, block_n, warp_n, stages,
                    bpc, split, placement: bool = True) -> None:
    """Argument checks of the op.  `placement=False` skips the device and alignment checks."""
    _torch_ops.validate_mxfp8(x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids,
                              num_tokens_post_padded, topk_weights, out, top_k, block_m, block_n, warp_n, stages,
                              bpc, split, placement)


def _fused_moe_mxfp8_fake(x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids,
                          num_tokens_post_padded, topk_weights, out, top_k, block_m, block_n, warp_n,
                          stages, bpc, split=True):
    return None


torch.library.register_fake("prime_moe::moe_align", _moe_align_fake, lib=_LIB)
torch.library.register_fake("prime_moe::fused_moe_bf16", _fused_moe_bf16_fake, lib=_LIB)
torch.library.register_fake("prime_moe::fused_moe_mxfp8", _fused_moe_mxfp8_fake, lib=_LIB)


# ------------------------------------------------------------------------------- public wrappers

def fused_moe_bf16(x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights, out,
                   top_k: int, block_m: int, block_n: int, warp_n: int, stages: int, bpc: int = 1,
                   cpc: int = 1, split: bool = True) -> torch.Tensor:
    """Runs ``prime_moe::fused_moe_bf16`` and returns ``out`` (reference __init__.py:27-49)."""
    torch.ops.prime_moe.fused_moe_bf16(
        x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights, out,
        top_k, block_m, block_n, warp_n, stages, bpc, cpc, split)
    return out


def fused_moe_mxfp8(x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids,
                    num_tokens_post_padded, topk_weights, out, top_k: int, block_m: int, block_n: int,
                    warp_n: int, stages: int, bpc: int = 1, split: bool = True) -> torch.Tensor:
    """Runs ``prime_moe::fused_moe_mxfp8`` and returns ``out`` (reference __init__.py:75-100)."""
    torch.ops.prime_moe.fused_moe_mxfp8(
        x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids,
        num_tokens_post_padded, topk_weights, out, top_k, block_m, block_n, warp_n, stages, bpc, split)
    return out


def pack_scales_blocked(scales: torch.Tensor) -> torch.Tensor:
    """Row-major ``(..., MN, K/32)`` e8m0 scales -> the 128x4 blocked tiles the kernels read.

    Layout contract of the reference (__init__.py:106-115): tiles of 128 rows x 4 K-blocks, 512
    bytes each, ordered [row tile][K tile]; inside a tile the scale of (row r, block b) is byte
    ``(r % 32) * 16 + (r % 128 // 32) * 4 + b % 4``, so the four scales of one row over 128
    consecutive K form one aligned 32-bit word.  Load-time work, plain torch.
    """
    u = scales.view(torch.uint8)
    mn, kb = u.shape[-2], u.shape[-1]
    assert mn % 128 == 0, f"MN ({mn}) must be a multiple of 128"
    assert kb % 4 == 0, f"K ({kb * 32}) must be a multiple of 128"
    lead = u.shape[:-2]
    # axes: [lead, row tile, quarter (r%128//32), r%32, K tile, b%4] -> [lead, row tile, K tile, r%32, quarter, b%4]
    tiles = u.reshape(-1, mn // 128, 4, 32, kb // 4, 4).permute(0, 1, 4, 3, 2, 5)
    return tiles.contiguous().reshape(*lead, -1).view(torch.float8_e8m0fnu)


def quantize_mx(t: torch.Tensor):
    """OCP-MX quantisation of the last dimension of a bf16 tensor on the GPU.

    Returns ``(float8_e4m3fn values, float8_e8m0fnu scales)`` with scales of shape
    ``t.shape[:-1] + (K // 32,)`` row major -- the format ``fused_moe_mxfp8`` takes for ``x``
    and, after :func:`pack_scales_blocked`, for the weights (specification: the reference's
    test/test_mxfp8.py:21-38).
    """
    return _torch_ops.quantize_mx(t)


def route(logits: torch.Tensor, top_k: int, block_m: int = 128, bpc: int = 1, bias: torch.Tensor = None):
    """Router front-end: gate logits ``(T, E)`` -> top-k, softmax weights and the ``moe_align`` schedule.

    The step the reference leaves to its callers (README.md:147-149): returns
    ``(topk_ids (T, top_k) int32, topk_weights (T, top_k) fp32, sorted_token_ids, expert_ids,
    num_tokens_post_padded)``; the last three are what ``torch.ops.prime_moe.moe_align(topk_ids, E,
    block_m, bpc)`` returns.  Selection: the ``top_k`` largest of ``logits[t] (+ bias)``, largest first,
    ties to the lower expert index; weights: softmax over the selected values in fp32.  One top-k kernel
    plus the align kernels on the current stream, no host synchronisation.
    """
    return _torch_ops.route(logits, top_k, block_m, bpc, bias)


__all__ = [
    "route",
    "fused_moe_bf16",
    "fused_moe_mxfp8",
    "pack_scales_blocked",
    "quantize_mx",
    "BLOCK",
]
