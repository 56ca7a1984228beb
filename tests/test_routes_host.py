"""Which kernel a call goes to, on the CPU: the library over a stand-in for the HIP runtime (tests/hip_stub) that records the
launches. The lines of the dispatch lie where both sides were measured; a call on the wrong side is right but slow, which
no parity test sees."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

CHILD = r"""
import ctypes as C, json, re, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_record.restype = C.c_char_p
import kernelcore_amd as kc
kc.init()


def launched(f):
    stub.stub_clear()
    f()
    out = []
    for line in stub.stub_record().decode().splitlines():
        name, *grid = line.split()
        m = re.search(r"\d+([a-z][a-z0-9_]*_kernel)(I(?:Li\d+E|Lb\dE)+E)?", name)
        out.append([m.group(1) + "".join("," + v for v in re.findall(r"L[ib](\d+)E", m.group(2) or ""))] + [int(g) for g in grid])
    return out


def matmul(qtype, rows, k, ncols):
    w, x, y = (kc.Buffer(n) for n in (kc.stream_bytes(qtype, rows, k), k // 256 * 340 * ncols, 4 * rows * ncols))
    r = launched(lambda: kc.launch("matmul_%s_q8kx8" % qtype, kc.MatmulKQ8Args(w.ptr, x.ptr, y.ptr, None, rows, k, ncols, 8)))
    for b in (w, x, y):
        b.free()
    return r


def f16(rows, k, ncols):
    w, x, y = kc.Buffer(2 * rows * k), kc.Buffer(4 * k * ncols), kc.Buffer(4 * rows * ncols)
    r = launched(lambda: kc.launch("matmul_f16", kc.MatmulF16Args(w.ptr, x.ptr, y.ptr, None, rows, k, ncols)))
    for b in (w, x, y):
        b.free()
    return r


print(json.dumps([globals()[name](*args) for name, args in json.loads(sys.argv[2])]))
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes([(function, arguments)]): for each call its launches, [kernel, gridx, gridy, gridz, blockx]."""
    import json

    lib = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub", "hip_stub.cpp"), "-o", lib], check=True)

    def run(calls):
        r = subprocess.run([sys.executable, "-c", CHILD, lib, json.dumps(calls)], cwd=os.path.dirname(HERE), text=True,
                           capture_output=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.splitlines()[-1])

    return run


def test_q6k_prefill_column_tile(routes):
    """128 columns per workgroup only where there are more than 64."""
    got = routes([("matmul", ("q6k", rows, 3072, n)) for rows, n in ((128256, 64), (65536, 64), (128256, 65), (16384, 512), (512, 65))])
    assert [g[0][0] for g in got] == ["matmul_i8_kernel,2", "matmul_i8_kernel,2", "matmul_i8_kernel,4", "matmul_i8_kernel,4",
                                      "matmul_i8_kernel,2"]


def test_two_columns_of_a_tall_matrix(routes):
    """The column tiles where they were measured faster (one line of sizes on either side), the short-batch kernel else."""
    cols = [("q6k", 128256, 1024, 2), ("q6k", 128256, 4096, 2), ("q6k", 16384, 4096, 2), ("q6k", 10240, 2048, 2),
            ("q6k", 65536, 1024, 3), ("q4k", 16384, 1024, 2), ("q4k", 49152, 4096, 2), ("q4k", 128256, 2048, 2),
            ("q4k", 32768, 1024, 3)]
    short = [("q6k", 128256, 512, 2), ("q6k", 20480, 4096, 2), ("q6k", 8192, 1024, 2), ("q6k", 10240, 4096, 2),
             ("q6k", 128256, 2048, 3), ("q6k", 128256, 1024, 4), ("q4k", 65536, 4096, 2), ("q4k", 8192, 3072, 2),
             ("q4k", 65536, 1024, 3), ("q4k", 16384, 4096, 2)]
    got = routes([("matmul", c) for c in cols + short])
    names = [g[0][0].split(",")[0] for g in got]
    assert names == ["matmul_cols_kernel"] * len(cols) + ["matmul_short_kernel"] * len(short)
