"""The load-time order at the edges of its kernels: node and workgroup sizes,
more waiting small nodes than their list holds, and NaN among the positions
of one small node.  Integer output: bit-exact.
"""
import os

import numpy as np
import pytest

import bvh_scenes as B
import orc

pytestmark = pytest.mark.gpu


def _order(G, m, q, s):
    return G.SceneArrays(m, q, s, np.zeros(len(m), np.float32), np.zeros((len(m), 3), np.float32), 0).bvh_order()


@pytest.mark.parametrize("kind", ["uniform", "clusters", "line"])
@pytest.mark.parametrize("n", [34, 63, 65, 66, 511, 513, 2047, 2048, 2049, 4095, 4097, 8449, 524288, 1050625])
def test_edges(gpu, kind, n):
    m, q, s = B.scene(n, 31 + n, kind)
    print(f"bvh nodes kind={kind} n={n}", flush=True)
    assert np.array_equal(_order(gpu, m, q, s), orc.bvh_order(m, q, s))


@pytest.mark.parametrize("base", [1.5, 2.0])
def test_chain_of_small_nodes(gpu, base):
    # each split cuts a few off the far end: one open node, many small ones
    n = int(np.log(1e24) / np.log(base))
    m, q, s = B.scene(n, 5, "uniform")
    m[:, 0] = (base ** np.arange(n)).astype(np.float32)
    s[:] = 2.0 ** -6
    print(f"bvh chain base={base} n={n}", flush=True)
    assert np.array_equal(_order(gpu, m, q, s), orc.bvh_order(m, q, s))


def nan_scene(n, axis):
    m, q, s = B.scene(n, 900 + n, "uniform")
    m[n // 2, axis] = np.nan
    return m, q, s


@pytest.mark.parametrize("n", [2, 9, 32])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_nan_in_a_small_node(gpu, n, axis):
    # orders recorded from a one-thread form of the same builder
    want = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "bvh_nan_small.npz"))
    print(f"bvh nan n={n} axis={axis}", flush=True)
    assert np.array_equal(_order(gpu, *nan_scene(n, axis)), want[f"{n}_{axis}"])
