"""The order in which the packed forward's workgroups take its query blocks (``areno_amd/csrc/varlen_blocks.hpp``
compiled by g++ into ``tests/native/varlen_blocks.cpp``): every block once, longest place first."""

import ctypes
import os
import random
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def walk():
    out = os.path.join(tempfile.mkdtemp(prefix="varlen_blocks_"), "libvarlen_blocks.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-o", out,
                    os.path.join(ROOT, "tests", "native", "varlen_blocks.cpp")], check=True)  # fmt: skip
    return ctypes.CDLL(out)


@pytest.mark.parametrize("block", [8, 9, 14, 18, 21, 25, 42, 64, 128])
def test_every_block_is_taken_once_and_the_longest_first(walk, block):
    rng = random.Random(block)
    packs = [[0], [1], [block], [block + 1, 0, block - 1], [0] * 64 + [300, 0, 5], [1] * 1000 + [4096], [24] * 1024]
    packs += [[rng.randint(0, rng.choice([1, 40, 3000])) for _ in range(rng.choice([1, 5, 63, 64, 65, 200]))] for _ in range(40)]
    msg = ctypes.create_string_buffer(256)
    for lens in packs:
        rc = walk.varlen_blocks_check((ctypes.c_int * len(lens))(*lens), len(lens), block, msg, 256)
        assert rc == 0, (msg.value.decode(), lens[:8])


def test_the_division_is_exact_at_its_edges(walk):
    for block in range(8, 129):
        for n in [0, 1, block - 1, block, block + 1] + [x * block + d for x in (1000, 99999, (1 << 30) // block) for d in (-1, 0)]:
            assert walk.varlen_block_division_check(block, min(n, (1 << 30) - 1)) == 0, (block, n)
