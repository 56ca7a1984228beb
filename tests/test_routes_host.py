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
import numpy as np
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


def matmul(qtype, rows, k, ncols, no_scratch=0):
    w, x, y = (kc.Buffer(n) for n in (kc.stream_bytes(qtype, rows, k), k // 256 * 340 * ncols, 4 * rows * ncols))
    stub.stub_capturing(no_scratch)
    r = launched(lambda: kc.launch("matmul_%s_q8kx8" % qtype, kc.MatmulKQ8Args(w.ptr, x.ptr, y.ptr, None, rows, k, ncols, 8)))
    stub.stub_capturing(0)
    for b in (w, x, y):
        b.free()
    return r


def f16(rows, k, ncols):
    w, x, y = kc.Buffer(2 * rows * k), kc.Buffer(4 * k * ncols), kc.Buffer(4 * rows * ncols)
    r = launched(lambda: kc.launch("matmul_f16", kc.MatmulF16Args(w.ptr, x.ptr, y.ptr, None, rows, k, ncols)))
    for b in (w, x, y):
        b.free()
    return r


def model(n, types={}, options={}, no_scratch=0, **cfg):
    # a prompt of n tokens on a two-layer driver (the last layer's FFN runs on one token); no_scratch: streams' staging
    # buffers cannot grow (as while a stream captures)
    cfg = dict(dict(n_layer=2, n_embd=1024, n_head=8, n_head_kv=2, head_dim=128, n_ff=2048, n_vocab=512, max_ctx=n,
                    max_batch=n, norm_eps=1e-5, rope_theta=1e4), **cfg)
    m = kc.Model(**cfg)
    for name, t in kc.TENSORS.items():
        if name in ("q_norm", "k_norm", "rope_freqs"):
            continue
        for layer in (-1,) if name in ("token_embd", "output_norm", "output") else (0, 1):
            _, rows, k, nbytes = m.tensor_info(name, layer)
            if name in types:
                m.set_tensor(name, layer, np.zeros(rows * (k // 256) * {"q4k": 144, "q6k": 210}[types[name]], np.uint8), types[name])
            else:
                m.set_tensor(name, layer, np.zeros(nbytes, np.uint8))
    for o, v in options.items():
        kc.set_option(o, v)
    stub.stub_capturing(no_scratch)
    r = launched(lambda: m.forward(np.zeros(n, np.int32)))
    stub.stub_capturing(0)
    for o in options:
        kc.set_option(o, 0)
    m.close()
    return r


print(json.dumps([globals()[name](*args, **kw) for name, args, kw in json.loads(sys.argv[2])]))
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes([(function, arguments[, keywords])]): for each call its launches, [kernel, gridx, gridy, gridz, blockx]."""
    import json

    lib = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub", "hip_stub.cpp"), "-o", lib], check=True)

    def run(calls):
        r = subprocess.run([sys.executable, "-c", CHILD, lib, json.dumps([(*c, {})[:3] for c in calls])], cwd=os.path.dirname(HERE), text=True,
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


def test_unstaged_batches_keep_the_prefill_kernel(routes):
    """64 columns and more that cannot be staged run on the prefill kernel that stages nothing, not on the short-batch one:
    past the fp16 layout's 32-bit offsets (a down projection of 16384 columns of 131072 values), and with no staging buffer."""
    down, groups = routes([("model", [16384], dict(types={"w_down": "q4k"}, n_embd=256, n_head=2, n_head_kv=2, n_ff=131072)),
                           ("model", [80], dict(types={"w_down": "q4k"}, n_embd=512, n_head=4, options={"prefill_act": 1}, no_scratch=1))])
    for got, count in ((down, 1), (groups, 2 * 4 + 2 + 1)):  # (q / k / v and o of two layers, gate / up and down of one)
        names = [g[0].split(",")[0] for g in got if g[0].startswith("matmul_")]
        assert "matmul_short_kernel" not in names and names.count("matmul_kq_mfma8_kernel") == count, names


def test_f16_limits(routes):
    """Past a launch's columns and a tile's offsets matmul_f16 keeps kernels of whole wavefronts, not the one thread per
    output of unaligned rows."""
    got = routes([("f16", (8, 512, n)) for n in (1 << 20, (1 << 20) + 1, (2 << 20) + 70)]
                 + [("f16", (8, k, 9)) for k in ((1 << 25) - 16, 1 << 25)])
    names = [[g[0].split(",")[0] for g in c] for c in got]
    assert names == [["mmf16_mfma_kernel"], ["mmf16_mfma_kernel", "mmf16_vec_kernel"], ["mmf16_mfma_kernel"] * 3,
                     ["mmf16_mfma_kernel"], ["mmf16_vec_kernel"] * 2]


def test_f16_short_rows(routes):
    """Rows short of a K-split chunk, where the workgroups take several rounds: the kernel of one tile per wavefront."""
    tile = [(4096, 128, 512), (4096, 144, 2048), (16384, 16, 9), (16384, 128, 16), (4096, 272, 512), (16384, 176, 1000),
            (20480, 288, 12)]
    split = [(64, 16, 512), (4096, 192, 512), (4096, 96, 64), (4096, 288, 512), (4096, 384, 512), (16384, 256, 1000)]
    got = routes([("f16", c) for c in tile + split])
    assert [g[0][0].split(",")[0] for g in got] == ["mmf16_tile_kernel"] * len(tile) + ["mmf16_mfma_kernel"] * len(split)


def test_int8_prefill_without_staging(routes):
    """A Q6_K batch on the int8 kernel stages no activations: with no staging buffer it keeps that kernel, in one K range."""
    got = routes([("matmul", ("q6k", 16384, 3072, 128), dict(no_scratch=1))]
                 + [("matmul", ("q6k", 1024, 3072, 128), dict(no_scratch=n)) for n in (1, 0)])
    assert [[g[0].split(",")[0] for g in c] for c in got] == [["matmul_i8_kernel"], ["matmul_i8_kernel"],
                                                              ["matmul_i8_kernel", "add_partial_kernel"]]
    assert [c[0][3] for c in got] == [1, 1, 2]
