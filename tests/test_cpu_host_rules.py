"""What the library decides on the host, without a GPU: a runtime that runs no kernels (cpp/fake_hip.cpp) is preloaded in a
child process, and the calls' return codes, the kernels they would launch and the memory they hold are read off."""
import os
import subprocess
import sys

import pytest

from mgg_osdi23_amd import host

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r'''
import ctypes as C, re
from mgg_osdi23_amd import host
fake = C.CDLL(None)
fake.fake_used.restype = C.c_size_t
fake.fake_launches.restype = C.c_char_p
lib = host.lib()
assert lib.mggx_init(0) == 0
def malloc(n):
    p = C.c_void_p()
    assert lib.mggx_malloc(C.byref(p), C.c_size_t(n)) == 0, lib.mggx_last_error()
    return p.value
def opts(**kw):
    o = host._AggOpts()
    for k, v in kw.items(): setattr(o, k, v)
    return C.byref(o)
def at(p): return C.c_void_p(p)
'''


@pytest.fixture(scope="module")
def without_device(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "fake_hip.cpp"), "-o", so], check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE + code], cwd=ROOT, capture_output=True, text=True,
                           env=dict(os.environ, LD_PRELOAD=so))
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def test_whole_pieces_only_where_they_stay_inside_the_row(without_device):
    """fp32 rows of a width that is not a multiple of 4, in a column window of a wider table: the last 16-byte piece is read
    whole (mode 0) only where the rows start on 16-byte boundaries, so that it cannot reach past the pitch; from any other
    column on the piece starts early (mode 3).  Pitch 48, width 41: at column 7 a whole piece would be columns 47 to 50."""
    out = without_device(r'''
rows, ld, dim = 64, 48, 41
ptr = malloc(4 * (rows + 1)); C.memset(ptr, 0, 4 * (rows + 1))
col, out = malloc(4), malloc(4 * rows * dim)
for dim in (41, 40):
    for left in range(8):
        table = malloc(4 * rows * ld)
        rc = lib.mggx_sag_np_div(at(out), at(table + 4 * left), None, at(ptr), at(col), None, None, 0, rows, dim, rows, 16, 4, 1, opts(ld_in=ld))
        assert rc == 0, lib.mggx_last_error()
        print(dim, left, re.match(r"k_agg<\d+,(\d)", host.last_agg_kernel()).group(1))
''')
    got = {tuple(map(int, l.split()[:2])): int(l.split()[2]) for l in out.splitlines()}
    assert got == {(d, c): (3 if d == 41 and c % 4 else 0) for d in (41, 40) for c in range(8)}
