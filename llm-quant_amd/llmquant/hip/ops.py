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


def _rows_in_place(numel: int, width: int, element_size: int, group_size: int) -> bool:
    """Whether ragged rows go to the kernel that takes them as they lie: groups of a power of two 16-byte packets that
    one wave holds, rows of a packet or more, and fewer than 2^31 packets counting each row's zeros up to whole groups
    (narrow rows under wide groups are mostly zeros)."""
    if numel == 0 or width < 8 or width % group_size == 0 or element_size > 4:
        return False
    packets, rest = divmod(group_size * element_size, 16)
    padded_packets = numel // width * -(-width // group_size) * packets
    return rest == 0 and packets <= 64 and packets & (packets - 1) == 0 and padded_packets < 1 << 31


def fake_quantize_hip(x: torch.Tensor, args: QuantizationArgs, return_scale: bool = False):
    """Quant-dequant on the GPU, bit-exact with llmquant.core.quant_ops.fake_quantize.

    Groups run along the last axis. A last axis that is not a whole number of groups gives
    what the PyTorch form's zero padding and trimming give: for groups of a power of two 16-byte
    packets the kernel reads and writes the rows as they lie, others are padded and trimmed.
    """
    group_size = _group_size_for(x, args)
    width = x.shape[-1]
    if x.is_cuda and _rows_in_place(x.numel(), width, x.element_size(), group_size):
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
