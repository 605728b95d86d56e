"""Python-level ops over the extension (counterpart of llmquant/cuda/ops.py)."""

from __future__ import annotations

import torch

from llmquant.core.observers import pad_to_group
from llmquant.core.scheme import QuantizationArgs
from llmquant.hip.build import load_extension


def _group_size_for(x: torch.Tensor, args: QuantizationArgs) -> int:
    if args.strategy == "group":
        return args.group_size
    if args.strategy in ("channel", "token"):
        return x.shape[-1]  # a single group spanning the row
    raise ValueError(f"unsupported strategy {args.strategy!r}")


def fake_quantize_hip(x: torch.Tensor, args: QuantizationArgs, return_scale: bool = False):
    """Quant-dequant on the GPU, bit-exact with llmquant.core.quant_ops.fake_quantize.

    Groups run along the last axis. A last axis that is not a whole number of groups gives
    what the PyTorch form's zero padding and trimming give: for groups of a power of two 16-byte
    packets the kernel reads and writes the rows as they lie, others are padded and trimmed.
    """
    group_size = _group_size_for(x, args)
    width = x.shape[-1]
    if width % group_size and x.is_cuda and x.element_size() <= 4:
        packets, rest = divmod(group_size * x.element_size(), 16)
        if rest == 0 and packets <= 64 and packets & (packets - 1) == 0 and width >= 8 and x.numel() < 1 << 30:
            out, scale = load_extension().fake_quant_rows(x, args.num_bits, group_size, return_scale)
            return (out, scale) if return_scale else out
    padded = pad_to_group(x, group_size)
    out, scale = load_extension().fake_quant_group(padded, args.num_bits, group_size, return_scale)
    if padded.shape[-1] != width:
        out = out[..., :width]
    return (out, scale) if return_scale else out


def quantize_activation(x: torch.Tensor, args: QuantizationArgs):
    """(int8 codes [..., K], fp32 scales [..., K / group]) for an activation whose last axis
    is already a whole number of groups -- the dynamic A8 quantizer as one kernel."""
    group_size = _group_size_for(x, args)
    return load_extension().quant_group_codes(x, args.num_bits, group_size, False)


# the reference's name for the same op
fake_quantize_cuda = fake_quantize_hip
