"""When one launch may do the packed attention and the cache write (``areno_amd/csrc/page_write.hpp`` compiled by g++ into
``tests/native/page_write.cpp``): never where the pages or the output share a byte with what the launch reads, or with each other."""

import ctypes
import os
import subprocess
import tempfile

import pytest

from areno_amd.accel import cabi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check():
    out = os.path.join(tempfile.mkdtemp(prefix="page_write_"), "libpage_write.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-o", out,
                    os.path.join(ROOT, "tests", "native", "page_write.cpp")], check=True)  # fmt: skip
    return ctypes.CDLL(out).page_write_check


@pytest.mark.parametrize("kv,element,scale,scale_element", [("act", 2, "F32", 0), ("I8", 1, "F16", 2), ("FP8_E4M3", 1, "F32", 4)])
@pytest.mark.parametrize("act", ["BF16", "F16"])
@pytest.mark.parametrize("head_dim", [64, 256])
def test_pages_and_output_apart_from_what_is_read(check, kv, element, scale, scale_element, act, head_dim):
    code = lambda name: getattr(cabi, f"DT_{name}")  # noqa: E731
    msg = ctypes.create_string_buffer(256)
    rc = check(code(act if kv == "act" else kv), code(scale), code(act), head_dim, element, scale_element, msg, 256)
    assert rc == 0, msg.value.decode()
