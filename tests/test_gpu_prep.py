"""GPU parity of the generator, preprocessing and core-matrix kernels at the sizes where they change path."""
import numpy as np
import pytest

import tribit_amd

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("scale", [1, 2, 7, 12, 15])
def test_rmat_generator_scales(gpu_ctx, oracle_mod, scale):
    """Even and odd scales (the last word of an odd scale gives one level): keys equal the oracle's."""
    note(f"rmat keys s{scale}")
    assert np.array_equal(gpu_ctx.gen_rmat_keys(scale, 5, seed=9), oracle_mod.gen_rmat(scale, 5, seed=9))


@pytest.mark.parametrize("core", [65536, 65537, 66001])
def test_core_wider_than_one_window(gpu_ctx, oracle_mod, core):
    """Core rows of one LDS column window, and of two."""
    note(f"core of {core} ids, er 70001")
    keys = oracle_mod.gen_er(70001, 900000, seed=4)
    with gpu_ctx.graph_from_keys(keys, 70001) as g:
        r = g.count("wedge", dense_core=core)
        assert r.dense_core == core
        assert r.triangles == oracle_mod.count_keys(keys, 70001)


@pytest.mark.parametrize("graphs", [1, 8192, 8193])
def test_batch_edge_counts(gpu_ctx, oracle_mod, graphs):
    """Per-graph edge counts at and past the largest batch summed in LDS."""
    note(f"batch of {graphs} small graphs")
    rng = np.random.default_rng(graphs)
    ns = rng.integers(2, 7, graphs)
    keys = []
    for n in ns:
        a, b = rng.integers(0, n, (2, int(rng.integers(0, 9))))
        keys.append(((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64))
    with gpu_ctx.batch_from_keys(keys, ns) as b:
        n, m = b.sizes()
        assert np.array_equal(n, ns.astype(np.uint64))
        assert [int(x) for x in m] == [len(set(k.tolist())) for k in keys]
        c, _ = b.count()
        assert [int(x) for x in c] == [oracle_mod.count_keys(k, int(v)) for k, v in zip(keys, ns)]
