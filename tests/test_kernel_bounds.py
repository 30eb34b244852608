"""Kernel sources in a CPU build (kernel_bounds/): the layer tail's rule, and the
buffer accesses of the kernels that request operands ahead of their use.  The
range check of a buffer resource is specified for the vector offset only, so
every access must be masked by its vector offset alone or lie inside its
resource, scalar offset included."""
import glob
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "compress-zip_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "kernel_bounds")
CLANG = "/opt/rocm/llvm/bin/clang++"
ASM = [('asm("v_sad_u32 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));', "r = a > b ? a - b : b - a;"),
       ('asm volatile("" : "+v"(t));', ""),
       ('asm volatile("" ::"v"(touched[0]), "v"(touched[1]), "v"(touched[2]), "v"(touched[3]));', "")]

# gemms M d F T skinny_rows wide_rows; tail M d F qkv; fused S d F; attention B T H
CASES = [
    # 128 x 256 tiles: partial row blocks and column tiles, odd and even K steps (3, 7, 11, 13 among them)
    "gemms 300 768 3072 100 0 1", "gemms 129 768 192 100 0 1", "gemms 77 704 448 7 0 1", "gemms 1 832 192 1 0 1",
    # few rows; tiled and W-stationary kernels; row kernels
    "gemms 77 896 832 100 1024 4096", "gemms 17 256 4160 5 1024 4096", "gemms 300 512 1024 100 0 100000",
    "gemms 300 384 1024 100 0 100000", "gemms 100 768 3072 100 0 100000", "gemms 1 64 64 1 0 100000",
    # layer tail: fewer column pairs than waves, K steps that are no multiple of those in flight, 16 and 32 rows
    "tail 40 512 1024 1", "tail 40 512 704 1", "tail 40 384 1024 0", "tail 17 256 64 1", "tail 17 256 4096 1", "tail 4100 256 64 1",
    # whole-stream decode: feed-forwards short of its K steps
    "fused 3 384 1024", "fused 3 512 960", "fused 2 384 448", "fused 1 256 64",
    # prefill attention: whole tiles, last tiles short of 64 and of 32 keys
    "attention 9 512 6", "attention 3 64 5", "attention 3 100 4", "attention 2 93 6", "attention 1 1 5",
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("no clang++")
    src = tmp_path_factory.mktemp("bounds")
    for path in glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")):
        with open(path) as f:
            text = f.read()
        for old, new in ASM:
            text = text.replace(old, new)
        with open(src / os.path.basename(path), "w") as f:
            f.write(text)
    exe = str(src / "bounds")
    subprocess.run([CLANG, "-O0", "-std=c++17", "-w", "-x", "c++", "-I", HERE, "-I", str(src), "-I", os.path.join(ROOT, "include"),
                    os.path.join(HERE, "bounds.cpp"), "-o", exe], check=True)
    return exe


def _tail_rounds(M, F, weights, decode, lanes):
    """The layer tail's rule on its rounds, restated from its measurements."""
    mb = weights / (1 << 20)
    if lanes and mb > 2:
        return False
    if F > 2048:  # 16 rows a workgroup: one round, and the fuller half of the second
        return M <= 4096 or 6144 <= M <= 8192
    if M <= 8192 or mb <= 2:
        return True
    half = M >= 12288  # the second round is at least half full
    return half if decode and mb > 3 else decode or (half and mb <= 3)


def test_layer_tail_rounds_rule(program):
    for F, weights in ((512, 1 << 20), (2048, 2 << 20), (2048, (2 << 20) + 1), (1536, 3 << 20), (2048, (3 << 20) + 1), (3072, 1 << 20),
                       (3072, 4 << 20)):
        for M in (600, 4096, 4097, 6143, 6144, 8192, 8193, 12287, 12288, 20480):
            for decode in (0, 1):
                for lanes in (0, decode):
                    r = subprocess.run([program, "tail_rounds", *map(str, (M, F, weights, decode, lanes))], capture_output=True, text=True)
                    assert int(r.stdout) == _tail_rounds(M, F, weights, decode, lanes), (M, F, weights, decode, lanes)


@pytest.mark.parametrize("case", CASES)
def test_buffer_accesses_in_range(program, case):
    r = subprocess.run([program, *case.split()], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    n = int(r.stdout.split(" accesses")[0].split()[-1])
    assert n > 0
