"""The candidate search by a group of lanes: the 2D alpha-shape bit for bit
against the CPU oracle on both sides of the rule that chooses between it and
one lane per node, and where it leaves its usual shape: fewer nodes than a
block, lists around and beyond the reference's limit of 250, more pending
entries than its stack holds, and points whose Morton codes differ in their
last bits only (a tree of one long chain)."""
import numpy as np
import pytest

import oracle_lib as ol
from stream_amd import clouds

pytestmark = pytest.mark.gpu


def _cloud(name):
    kind, k = name.split("-")
    k = int(k)
    rng = np.random.default_rng(k)
    if kind == "all":  # every node is everyone's candidate
        return rng.random((k, 2)), 2.0
    if kind == "dense":
        return rng.random((k, 2)), 4.0 / k ** 0.5
    if kind == "chain":  # clusters at 2^-1, 2^-2, ...
        r = 2.0 ** -np.repeat(np.arange(k), 3)
        return r[:, None] * (0.5 + 0.4 * rng.random((3 * k, 2))), 2.0
    return clouds.dam_break_scaled(k, 1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", ["all-3", "all-4", "all-31", "all-33", "all-100", "all-246", "dense-700", "dense-5000",
                                  "chain-8", "chain-18", "dam-3000"])
def test_alphashape2d_matches_oracle(name, dtype):
    _check(*_cloud(name), dtype, name)


@pytest.mark.parametrize("n", [90_112, 90_113])
def test_both_sides_of_the_rule(n):
    pts = ol.glibc_uniform(n, 2, 7)
    _check(pts, np.float32(1.2 / n ** 0.5), np.float32, f"uniform {n}")


def _check(pts, alpha, dtype, label):
    from stream_amd.mesh import AlphaShape2D

    print(f"[fill] {label} {np.dtype(dtype).name}", flush=True)
    pts = np.asarray(pts, dtype)
    al = np.broadcast_to(np.asarray(alpha, dtype), len(pts)).copy()
    o = ol.ashape2d(pts, al, bits=32, dtype=dtype)
    a = AlphaShape2D(dtype=dtype, morton_bits=32)
    a.set_nodes(pts, al)
    a.compute()
    row, neig, eb = a.get_edges()
    assert np.array_equal(a.get_permutation(), o["perm"])
    assert np.array_equal(a.get_elem(), o["elem"])
    assert np.array_equal(row, o["row"]) and np.array_equal(neig, o["neig"])
    assert np.array_equal(eb, o["edge_is_bnd"])
    assert np.array_equal(a.get_boundary_nodes(), o["node_is_bnd"])
