"""Launches of the Adam step over groups of any size, without a GPU: a stand-in for the HIP runtime's launch calls writes down what it is asked to
launch."""
import subprocess
import sys

import pytest

from test_launch_host import STUB

RECORD = STUB.replace("int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t lds, void*) {", r"""
static long long seen[64][3];
static int n_seen = 0;
int stub_seen(long long* out) { const int n = n_seen; for (int i = 0; i < 3 * n; ++i) out[i] = seen[0][i]; n_seen = 0; return n; }
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t lds, void*) {
  if (n_seen < 64) { seen[n_seen][0] = *(long long*)args[2]; seen[n_seen][1] = grid.x; seen[n_seen][2] = block.x; ++n_seen; }
""")
CHILD = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)     # before anything else that brings the HIP runtime in
from pfeife_amd import hip
lib = hip.load()
for n in [int(a) for a in sys.argv[2:]]:
    rc = lib.pf_adam_step_chunks(1 << 20, 1 << 21, 3, n, 1e-3, 0.9, 0.999, 1e-8, 0.0, 1, 0, None, None)      # (nothing reads them)
    assert rc == 0, lib.pf_last_error()
    out = (ctypes.c_longlong * 192)()
    seen = [tuple(out[3 * i:3 * i + 3]) for i in range(stub.stub_seen(out))]
    at = 0
    for first, blocks, threads in seen:      # every chunk once, in order, within what a launch may have
        assert first == at and blocks > 0 and blocks * threads < 1 << 32, seen
        at += blocks
    assert at == n, seen
"""


@pytest.mark.parametrize("chunks", [[1, 2, 4097], [(1 << 23) - 1, 1 << 23, (1 << 23) + 1], [(1 << 24) - 1, 1 << 24, (1 << 24) + 5, 3 << 23]])
def test_every_chunk_is_launched_once(chunks, tmp_path):
    src, so = tmp_path / "stub.cpp", tmp_path / "libstub.so"
    src.write_text(RECORD)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    res = subprocess.run([sys.executable, "-c", CHILD, str(so), *map(str, chunks)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
