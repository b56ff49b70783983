"""Launches of a 3x3 convolution's windows for images of any size, without a GPU: a stand-in for the HIP runtime's launch calls writes down what
it is asked to launch."""
import subprocess
import sys

import pytest

from test_adam_launch_host import RECORD

CHILD = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)     # before anything else that brings the HIP runtime in
from pfeife_amd import hip
lib = hip.load()
B, H, W, C = [int(a) for a in sys.argv[2:]]
rc = lib.pf_im2col3x3(1 << 20, 1 << 21, hip.PF_F32, B, H, W, C, 0, None)      # (nothing reads them)
assert rc == 0, lib.pf_last_error()
out = (ctypes.c_longlong * 192)()
at = 0
for i in range(stub.stub_seen(out)):
    first, blocks, threads = out[3 * i:3 * i + 3]      # in order, each piece of 16 bytes once, within what a launch may have
    assert first == at and 0 < blocks and blocks * threads < 1 << 32, (first, blocks, threads)
    at += blocks
assert (at - 1) * 256 < B * H * W * 9 * (C // 4) <= at * 256, at
"""


@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 13, 11, 8), (1, 1 << 16, 1 << 13, 4), (1, 1, 1 << 24, 4), (3, 1 << 14, 1 << 14, 12), (1, 1, 1, 1 << 29)])
def test_every_piece_is_launched_once(shape, tmp_path):
    src, so = tmp_path / "stub.cpp", tmp_path / "libstub.so"
    src.write_text(RECORD)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    res = subprocess.run([sys.executable, "-c", CHILD, str(so), *map(str, shape)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
