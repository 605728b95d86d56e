"""What the compiler made of the kernels whose operands come out of inline assembly or are held at the register limit: the
device code of this repository's own sources, compiled here (no GPU needed), read as text."""

import functools
import pathlib
import re
import shutil
import subprocess

import pytest

PACKAGE = pathlib.Path(__file__).resolve().parent.parent / "llm-quant_amd"
CSRC = PACKAGE / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
needs_hipcc = pytest.mark.skipif(not pathlib.Path(HIPCC).exists(), reason="needs hipcc")


@functools.lru_cache(maxsize=None)
def assembly(source: str) -> str:
    """gfx950 assembly of a source, with the Makefile's flags."""
    flags = subprocess.run(["make", "-s", "-C", str(PACKAGE), "--no-print-directory", "--eval=flags: ; @echo $(HIPFLAGS)", "flags"],
                           check=True, capture_output=True, text=True).stdout.split()
    return subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", str(CSRC / source), "-o", "-"],
                          check=True, capture_output=True, text=True).stdout


def registers(operand: str) -> range:
    one, several = re.fullmatch(r"v(\d+)", operand), re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    if one:
        return range(int(one[1]), int(one[1]) + 1)
    return range(int(several[1]), int(several[2]) + 1) if several else range(0)


def operands_too_soon(text: str, wait_states: int = 2) -> list[str]:
    """Matrix instructions that read a vector register fewer than `wait_states` after a vector instruction wrote it, in the
    order of the listing (an instruction is one state, s_nop N is N + 1)."""
    found, kernel, at, written = [], None, 0, {}
    for line in text.splitlines():
        if label := re.match(r"(_Z\w+):", line):
            kernel, at, written = label[1], 0, {}
        match = re.match(r"\s+((?:v|s|ds|buffer|global|flat|scratch)_\w+)\s*([^;]*)", line)
        if kernel is None or not match:
            continue
        op, operands = match[1], [part.strip() for part in match[2].split(",")]
        if op.startswith("v_mfma"):
            for register in (r for operand in operands[1:4] for r in registers(operand)):
                if register in written and at - written[register][0] - 1 < wait_states:
                    found.append(f"{kernel}: v{register} of {written[register][1]}")
            for register in registers(operands[0]):
                written.pop(register, None)
        elif op.startswith("v_"):
            written.update((register, (at, line.strip())) for register in registers(operands[0]))
        at += int(operands[0], 0) + 1 if op == "s_nop" else 1
    return found


def test_the_listing_is_read():
    listing = "_Zk:\n\tv_and_or_b32 v3, v1, s0, v2\n\ts_nop {}\n\tv_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], 0\n"
    assert len(operands_too_soon(listing.format(0))) == 1 and operands_too_soon(listing.format(1)) == []


@pytest.mark.parametrize("source", sorted(p.name for p in CSRC.rglob("*") if p.suffix in (".hip", ".h")))
def test_inline_assembly_only_waits(source):
    """The compiler does not look into inline assembly for its wait states: what is written there is a wait, or nothing."""
    text = next(CSRC.rglob(source)).read_text()
    bodies = re.findall(r'\basm\b(?:\s+volatile)?\s*\(\s*"([^"]*)"', text)
    assert all(body == "" or body.startswith("s_waitcnt ") for body in bodies), bodies


@needs_hipcc
@pytest.mark.parametrize("source", ["wq_gemm_a16.hip", "wq_gemm_a16_tile.hip", "wq_gemm_experts.hip"])
def test_operands_are_written_two_wait_states_ahead(source):
    text = assembly(source)
    assert text.count("v_mfma") > 100
    assert operands_too_soon(text) == []


@needs_hipcc
@pytest.mark.parametrize("source", ["wq_gemm_experts.hip", "wq_gemm_a16_tile.hip"])
def test_the_tiles_do_not_spill(source):
    """A spilled register's reload waits for every transfer into LDS that was asked for before it."""
    kernels = re.findall(r"\.name:\s+(_Z\S+).*?\.vgpr_spill_count:\s+(\d+)", assembly(source), re.S)
    assert len(kernels) > 10
    assert [name for name, spilled in kernels if int(spilled)] == []
