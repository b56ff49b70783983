"""What the library's launchers do on the host, without a GPU: a stand-in for the HIP runtime's launch calls, loaded
ahead of the library in a child process, checks and counts launches and runs none."""
import subprocess
import sys

import pytest

STUB = r"""
#include <cstddef>
#include <cstdio>
#include <map>
#include <utility>
struct Dim3 { unsigned x, y, z; };
static int device = 0, fail_attribute = 0, launches = 0, last_error = 0;
static std::map<std::pair<const void*, int>, int> allowed;
static struct { Dim3 grid, block; size_t lds; void* stream; } config;
extern "C" {
void stub_device(int d) { device = d; }
void stub_fail_attribute(int on) { fail_attribute = on; }
int stub_launches() { const int n = launches; launches = 0; return n; }
int hipGetDevice(int* d) { *d = device; return 0; }
int hipFuncSetAttribute(const void* f, int, int value) {
  if (fail_attribute) return 1;
  allowed[{f, device}] = value;
  return 0;
}
unsigned __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* s) { config = {g, b, lds, s}; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** s) {
  *g = config.grid; *b = config.block; *lds = config.lds; *s = config.stream; return 0;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t lds, void*) {
  if (lds > 65536 && (size_t)allowed[{f, device}] < lds) return last_error = 1;   // as the runtime refuses it
  ++launches;
  return 0;
}
int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
}
"""

CHILD = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)     # before anything else that brings the HIP runtime in
from pfeife_amd import hip
lib = hip.load(*sys.argv[2:3])

def gemm(M, N, K, at=0, bt=0, dtype=hip.PF_F32, variant=0, **kw):
    d = hip.GemmDesc()
    d.in_dtype, d.c_dtype, d.M, d.N, d.K = dtype, hip.PF_F32, M, N, K
    d.a_trans, d.b_trans, d.variant = at, bt, variant
    d.lda, d.ldb, d.ldc = (M if at else K), (N if bt else K), N
    d.batch1, d.batch2, d.alpha = 1, 1, 1.0
    d.A, d.B, d.C = 1 << 20, 1 << 21, 1 << 22           # (nothing reads them)
    for k, v in kw.items():
        setattr(d, k, v)
    return d

def run(d):
    return lib.pf_gemm(ctypes.byref(d), None), stub.stub_launches()
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    path = tmp_path_factory.mktemp("stub")
    src, so = path / "stub.cpp", path / "libstub.so"
    src.write_text(STUB)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    return str(so)


def child(stub, code):
    res = subprocess.run([sys.executable, "-c", CHILD + code, stub], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr


def test_dynamic_lds_is_allowed_on_every_device_a_kernel_runs_on(stub):
    """Tiles that need more than 64 KB of LDS, on two devices of one process: every launch is allowed its LDS on the
    device it goes to; where that fails the call is an error and nothing is launched."""
    child(stub, r"""
calls = []
for at in (0, 1):
    for bt in (0, 1):
        calls += [gemm(2048, 2048, 64, at, bt), gemm(1024, 384, 64, at, bt), gemm(256, 192, 64, at, bt), gemm(64, 64, 64, at, bt)]
        for dt in (hip.PF_F16, hip.PF_BF16):
            calls += [gemm(512, 512, 128, at, bt, dt, v) for v in (11, 12, 13, 14)]
            if at == bt:
                calls += [gemm(512, 512, 128, at, bt, dt, v) for v in list(range(1, 11)) + [15] if not (at and v in (4, 10))]
stub.stub_fail_attribute(1)
refused = [run(d) for d in calls]
assert all((rc == 0) == (n == 1) for rc, n in refused) and sum(rc != 0 for rc, _ in refused) >= 30, refused
stub.stub_fail_attribute(0)
for device in (0, 1, 0, 5):
    stub.stub_device(device)
    for d in calls:
        got = run(d)
        assert got == (0, 1), (device, d.M, d.N, d.a_trans, d.b_trans, d.in_dtype, d.variant, got, lib.pf_last_error())
group = (hip.GemmDesc * 2)(*[gemm(512, 512, 128, 1, 1, hip.PF_F16, 8, beta=1)] * 2)
for device in (0, 1):
    stub.stub_device(device)
    assert (lib.pf_gemm_grouped(group, 2, None), stub.stub_launches()) == (0, 1), device
""")


def test_transposed_product_with_bias_and_overflow_flag_is_accepted(stub):
    """Both operands transposed, fp32 C stored or accumulated, a bias and `nonfinite_flag`, on every tile with such a
    kernel; the flag stays refused with an activation and where no tile checks what it writes."""
    child(stub, r"""
for dt in (hip.PF_F16, hip.PF_BF16):
    for beta in (0, 1):
        for v in (0, 1, 2, 3, 5, 6, 7, 8, 9, 15):
            d = gemm(512, 512, 128, 1, 1, dt, v, beta=beta, bias=1 << 23, nonfinite_flag=1 << 24)
            assert run(d) == (0, 1), (dt, beta, v, lib.pf_last_error())
    assert run(gemm(512, 512, 128, 1, 1, dt, act=1, aux_out=1 << 23, ld_aux_out=512, nonfinite_flag=1 << 24)) == (-2, 0)
    assert run(gemm(512, 512, 128, 1, 0, dt, nonfinite_flag=1 << 24)) == (-2, 0)
    assert run(gemm(512, 512, 128, 1, 1, dt, 11, nonfinite_flag=1 << 24)) == (-2, 0)
""")


def test_transposed_product_that_rounds_before_it_stores_runs_where_that_is_done(stub):
    """round_mid of a product with both operands transposed: not on the straight-line kernels (no rounding there), and
    not as a member of a grouped launch."""
    child(stub, r"""
name = ctypes.create_string_buffer(128)
for dt in (hip.PF_F16, hip.PF_BF16):
    for beta in (0, 1):
        for v in (0, 1, 2, 3, 5, 6, 7, 8, 9, 15):
            for flag in (None, 1 << 24):
                d = gemm(512, 512, 128, 1, 1, dt, v, beta=beta, round_mid=1, nonfinite_flag=flag)
                assert run(d) == (0, 1), (dt, beta, v, lib.pf_last_error())
                assert lib.pf_gemm_variant(ctypes.byref(d), name, 128) == 0 and name.value.endswith(b", true, true, -1>"), name.value
                group = (hip.GemmDesc * 2)(d, d)
                assert (lib.pf_gemm_grouped(group, 2, None), stub.stub_launches()) == (0, 2)
""")


def test_rows_so_wide_that_a_tiles_last_rows_wrap_a_32_bit_offset_take_the_generic_epilogue(stub):
    """The straight-line epilogues drop rows past M by the range check of a buffer: for every tile, class and operand
    the byte offset of any row of the last tile stays below 2^32, and nothing else changes its class."""
    child(stub, r"""
name = ctypes.create_string_buffer(128)
def straight(M, fits, **kw):
    d = gemm(M, 64, 64, dtype=hip.PF_F16, **kw)
    assert lib.pf_gemm_variant(ctypes.byref(d), name, 128) == 0 and run(d) == (0, 1)
    d.nonfinite_flag = 1 << 24
    plain = d.c_dtype == hip.PF_F32 and not d.residual and fits
    assert (run(d) == (0, 1)) == plain, lib.pf_last_error()      # what took the flag takes it on either epilogue
    return not name.value.endswith(b", -1>")
for variant, bm in ((7, 256), (8, 128), (9, 256), (10, 192), (15, 64), (1, 256), (3, 128), (4, 192), (5, 128)):
    for M in (1, 8, 63, 128, 300):
        rows = (M + bm - 1) // bm * bm
        for ld in (64, 1 << 16, 1 << 20, (1 << 21) - 8, 1 << 21, 1 << 22, 1 << 23, 1 << 24, 1 << 26):
            for kw, size in ((dict(ldc=ld), 4), (dict(ldc=ld, c_dtype=hip.PF_F16), 2), (dict(ldc=ld, beta=1), 4),
                             (dict(residual=1 << 23, ld_res=ld), 4),
                             (dict(c_dtype=hip.PF_F16, act=1, aux_out=1 << 23, ld_aux_out=ld), 2),
                             (dict(c_dtype=hip.PF_F16, dact=1, aux_in=1 << 23, ld_aux_in=ld), 2)):
                fits = M * ld * (4 if "ldc" in kw or "ld_res" in kw else 2) < (1 << 31) - 64
                assert straight(M, fits, variant=variant, **kw) == (fits and rows * ld * size < 1 << 32), (variant, M, ld, kw)
""")


def test_an_issuer_without_a_thread_is_an_error(stub):
    """No room for another thread's stack: pf_issuer_create reports it (an exception that left a C entry point would end
    the process) and works once there is room."""
    child(stub, r"""
import resource
out = ctypes.c_void_p()
size = 1024 * int(next(l for l in open("/proc/self/status") if l.startswith("VmSize")).split()[1])
before = resource.getrlimit(resource.RLIMIT_AS)
resource.setrlimit(resource.RLIMIT_AS, (size + (2 << 20), before[1]))
rc, text = lib.pf_issuer_create(0, ctypes.byref(out)), lib.pf_last_error()
resource.setrlimit(resource.RLIMIT_AS, before)
assert rc != 0 and b"pf_issuer_create" in text and not out.value, (rc, text)
assert lib.pf_issuer_create(0, ctypes.byref(out)) == 0 and out.value
assert lib.pf_issuer_destroy(out) == 0
""")
