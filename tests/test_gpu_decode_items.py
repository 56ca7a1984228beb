"""The fused decode matvec (kdecode.hip, dmv) where its work splits at an edge: one item per wavefront (computed slab by slab
from the loads) and several (the loop), partial groups of super-blocks, numbers of terms that are no multiple of four, both
weight types behind the norm and the slot prologue, tiles past the rows; every count of slabs issued before the norm
prologue. Against one launch per node, which sums the same terms in the same order: the same bits."""
import numpy as np
import pytest

import kernelcore_amd as kc
from kernelcore_amd import ggml_graph as gg
from tests.test_gpu_ggml_backend import Layer

pytestmark = pytest.mark.gpu
HEADS = dict(n_head=8, n_head_kv=2, head_dim=64)


@pytest.fixture(scope="module", autouse=True)
def runtime():
    kc.init()
    yield
    kc.synchronize()


def outputs(L, **options):
    for name, value in options.items():
        kc.set_option(name, value)
    try:
        be = kc.GgmlBackend(graphs=0)
        be.compute(L.g.nodes)
        kc.synchronize()
        be.close()
        return {n: L.get(n, np.float32) for n in ("q", "k", "v", "attn", "ffn_inp", "out")}
    finally:
        for name in options:
            kc.set_option(name, 0)


@pytest.mark.parametrize("shape", [
    dict(n_embd=512, n_ff=256),
    dict(n_embd=1280, n_ff=2816, wq="q6k", wv="q4k", wo="q6k", wg="q6k", wu="q6k", wd="q4k"),
    dict(n_embd=3328, n_ff=1280, wk="q6k", wd="q4k"),
    dict(n_embd=1024, n_ff=11008),
], ids=lambda s: f"{s['n_embd']}-{s['n_ff']}")
def test_decode_matvec_items(shape):
    L = Layer(gg.LayerShape(**HEADS, **shape), 1, 70, seed=shape["n_ff"])
    names, _ = kc.ggml_graph_plan(L.g.nodes)
    assert "decode_norm_matvec" in names and "decode_norm_swiglu" in names
    want = outputs(L, ggml_extra_fusions=1)
    for pre in (0, 3, 6, 9, 14):
        got = outputs(L, swiglu_pre=pre) if pre else outputs(L)
        for n in want:
            assert np.array_equal(got[n].view(np.uint32), want[n].view(np.uint32)), (n, pre)
    L.free()
