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
def flags() -> list[str]:
    return subprocess.run(["make", "-s", "-C", str(PACKAGE), "--no-print-directory", "--eval=flags: ; @echo $(HIPFLAGS)", "flags"],
                          check=True, capture_output=True, text=True).stdout.split()


@functools.lru_cache(maxsize=None)
def assembly(source: str) -> str:
    """gfx950 assembly of a source, with the Makefile's flags."""
    return subprocess.run([HIPCC, *flags(), "--cuda-device-only", "-S", str(CSRC / source), "-o", "-"],
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


@needs_hipcc
def test_forms_of_the_gemm_for_a_few_dozen_rows(tmp_path):
    """The lines between the forms, on both sides: the kernel's own rule, at compile time. (They were drawn with an earlier loop;
    what either side takes with the present one stands at the rule.)"""
    lines = [  # bits, rows, outputs, groups, row tiles, scales held
        (4, 17, 16384, 1, 4, False), (4, 32, 128256, 8, 4, False), (4, 32, 16384, 16, 4, False), (4, 17, 24577, 16, 4, True),
        (4, 32, 32000, 18, 4, False), (4, 17, 16384, 19, 4, False), (4, 17, 16384, 20, 4, True), (4, 33, 16384, 64, 4, False),
        (8, 32, 28672, 4, 4, False), (8, 32, 28672, 16, 4, False), (8, 17, 128256, 16, 4, True), (8, 17, 128256, 20, 4, False),
        (8, 17, 12288, 31, 4, False), (8, 17, 15360, 32, 4, True), (8, 17, 16384, 39, 4, False), (8, 17, 16384, 40, 4, True),
        (8, 3, 14336, 32, 4, True), (8, 3, 14337, 32, 2, False), (8, 8, 15360, 39, 2, False), (8, 8, 15360, 40, 4, True),
        (8, 4, 16384, 191, 2, False), (8, 4, 16384, 192, 4, True), (8, 5, 16384, 64, 2, False), (8, 5, 16384, 96, 4, True),
        (8, 9, 16384, 32, 4, False), (8, 9, 14336, 32, 4, True), (8, 9, 16384, 31, 2, False), (4, 3, 16384, 32, 4, True), (4, 3, 16448, 32, 2, False),
        (8, 3, 12288, 255, 4, True), (8, 3, 12288, 256, 4, False), (4, 32, 12288, 256, 4, False),   # what the LDS holds
        (8, 33, 16384, 32, 2, False), (4, 64, 16384, 32, 2, False), (4, 16, 12224, 32, 2, False), (4, 16, 8176, 32, 1, False),
    ]
    checks = [f"static_assert(form_of({b}, {m}, {n}, {g}).row_tiles == {t} && form_of({b}, {m}, {n}, {g}).held == {str(h).lower()});"
              for b, m, n, g, t, h in lines]
    source = tmp_path / "forms.hip"
    source.write_text(f'#include "{CSRC}/wq_gemm_a16.hip"\n' + "\n".join(checks) + "\n")
    ran = subprocess.run([HIPCC, *flags(), "--cuda-host-only", "-fsyntax-only", str(source)], capture_output=True, text=True)
    assert ran.returncode == 0, "\n".join(line for line in ran.stderr.splitlines() if "error" in line or "static_assert" in line)
