"""The streamed products and latent attention's prompts issue their matrix instructions as inline assembly: the compiler does not
know them for matrix instructions and would read a sum right behind one without the wait that takes.  So in the streamed
products no sum may be moved between a kernel's first matrix instruction and the wait behind its last, and in all of them (the
products of few rows whose operands go straight to registers among them) no vector instruction may come too close: read from
the assembly of these sources."""

import functools
import os
import re
import subprocess

import pytest

from synaptix_amd.kernels import build



@functools.lru_cache(maxsize=None)
def assembly_of(source, folder):
    _, defines = build._spec("core")
    flags = [f for f in build.FLAGS if f != "-shared"]
    listing = folder / (source + ".s")
    subprocess.check_call([build.find_hipcc(), "-w", *flags, *defines, "-S", "--cuda-device-only",
                           os.path.join(build.CSRC, source), "-o", str(listing)])
    return listing.read_text().split("\n")


@pytest.fixture(scope="module")
def folder(tmp_path_factory):
    return tmp_path_factory.mktemp("assembly")


def kernels_of(source, kernel, folder):
    lines = assembly_of(source, folder)
    starts = [i for i, l in enumerate(lines) if re.match(rf"_Z\d+{kernel}\w*:", l)]
    assert starts
    for start in starts:
        end = next(i for i in range(start, len(lines)) if lines[i].startswith(".Lfunc_end"))
        yield lines[start], [l.split(";")[0].strip() for l in lines[start:end]]


STREAMED = [("gemm.hip", "gemm_stream_kernel"), ("grouped.hip", "grouped_stream_kernel")]


@pytest.mark.parametrize("source,kernel", STREAMED + [("gemm.hip", "gemm_rows_kernel")])
def test_no_sum_moves_between_matrix_instructions(source, kernel, folder):
    for name, body in kernels_of(source, kernel, folder):
        matrix = [i for i, l in enumerate(body) if "v_mfma" in l]
        behind = next(i for i in range(matrix[-1], len(body)) if "s_nop 15" in body[i])
        moves = [l for l in body[matrix[0]:behind] if "v_accvgpr" in l or "scratch_" in l]
        assert not moves, (name, moves[:4])


def registers(operand):
    m = re.match(r"([va])\[(\d+):(\d+)\]$|([va])(\d+)$", operand.strip())
    if not m:
        return set()
    return {(m[4], int(m[5]))} if m[4] else {(m[1], k) for k in range(int(m[2]), int(m[3]) + 1)}


@pytest.mark.parametrize("source,kernel", STREAMED + [("gemm.hip", "gemm_rows_kernel"), ("latent_attention.hip", "latent_prompt_bf16_kernel")])
def test_vector_instructions_keep_away_from_matrix_instructions(source, kernel, folder):
    """No vector instruction may write what a matrix instruction reads one or two states later, nor touch a result within
    eighteen of its start (latent attention mixes both on every page; the streamed products at the ends of their tiles)."""
    for name, body in kernels_of(source, kernel, folder):
        body = [l for l in body if re.match(r"[a-z]+_", l)]
        for i, line in enumerate(body):
            if not line.startswith("v_"):
                continue
            operands = [registers(o) for o in line.split(None, 1)[1].split(", ")]
            states, matrix = 0, line.startswith("v_mfma")
            for before in reversed(body[max(i - 20, 0):i]):
                if states >= (2 if matrix else 18):
                    break
                if before.startswith("s_nop"):
                    states += int(before.split()[1])
                elif before.startswith("v_"):
                    written = registers(before.split(None, 1)[1].split(", ")[0])
                    if matrix != before.startswith("v_mfma"):
                        touched = set().union(*(operands[1:] if matrix else operands))
                        assert not written & touched, (name, before, line)
                states += 1
