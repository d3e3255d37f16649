"""The 16-lane local Delaunay of the 3D alpha-shape at the edges of its rules,
bit for bit against the CPU oracle: node counts around a wavefront's four
nodes, an XCD's 256 and the 2,048 of all, candidate lists from none to the clamped 124 (nodes that wait for room
in the candidate pool), stars beyond 32 and beyond 64 tetrahedra, cavities
beyond 14 and 32 and walks that the step cap stops, coordinates far from and
close to 1 (FP32 tests that only the FP64 filter decides), and a pair of nodes
that all but coincide beside infinity nodes at hundreds of alpha; the count of the
nodes that needed the exact stage; and nodes that coincide, which are refused."""
import numpy as np
import pytest

import oracle_lib as ol
from stream_amd import clouds

pytestmark = pytest.mark.gpu


def _ball(n, seed):
    """A centre and n points on the unit sphere, radii jittered by 1e-3: the
    centre's star has about 2 n tetrahedra."""
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((n, 3))
    v *= ((1.0 + 1e-3 * rng.random(n)) / np.linalg.norm(v, axis=1))[:, None]
    return np.concatenate([np.zeros((1, 3)), v])


def _cloud(name):
    kind, k = name.split("-")
    k = int(k)
    if kind == "random":  # few points, all candidates of each other
        return np.random.default_rng(k).random((k, 3)), 2.0
    if kind == "sparse":  # 0, 1, 2, ... candidates
        return np.random.default_rng(k).random((k, 3)), 0.35 / k ** (1 / 3)
    if kind == "ball":
        return _ball(k, k), 3.0
    if kind == "twin":  # of the origin, at 2e-23 alpha, in a box of 1,200 alpha
        rng = np.random.default_rng(k)
        pts = rng.uniform(-1, 1, (60, 3))
        pts[30:, 1] = pts[30:, 2] * (1 + 1e-7 * rng.standard_normal(30))  # almost in a plane with the pair
        box = 600.0 * np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)])
        return np.concatenate([[[0.0, 0.0, 0.0], [-1e-23, 1.3e-23, 1.3e-23]], pts, box]), 1.0
    if kind == "cluster":  # as many nodes again within a hundredth of the box: one-sided clamped lists
        rng = np.random.default_rng(k)
        return np.concatenate([rng.random((k, 3)), 0.5 + 0.01 * rng.random((k, 3))]), 1.1 / k ** (1 / 3)
    if kind == "dense":  # alpha well above the spacing: clamped lists
        return np.random.default_rng(k).random((k, 3)), 1.9 / k ** (1 / 3)
    pts, al = clouds.sloshing_tank_scaled(k, 3)
    return pts, 1.08 * al


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name, scale, offset", [
    ("random-4", 1.0, 0.0), ("random-5", 1.0, 0.0), ("random-7", 1.0, 0.0), ("random-33", 1.0, 0.0),
    ("random-124", 1.0, 0.0), ("random-127", 1.0, 0.0), ("sparse-255", 1.0, 0.0), ("sparse-257", 1.0, 0.0),
    ("sparse-2048", 1.0, 0.0), ("sparse-2049", 1.0, 0.0), ("cluster-1500", 1.0, 0.0), ("sparse-301", 1.0, 0.0), ("ball-17", 1.0, 0.0),
    ("ball-34", 1.0, 0.0), ("ball-35", 1.0, 0.0), ("ball-60", 1.0, 0.0), ("ball-123", 1.0, 0.0),
    ("dense-1500", 1.0, 0.0), ("dense-400", 2.0 ** -9, 0.0), ("dense-400", 2.0 ** 20, 0.0),
    ("dense-400", 1.0, 300.0), ("tank-9000", 1.0, 0.0), ("twin-1", 1.0, 0.0), ("twin-5", 1.0, 0.0)])
def test_outputs_match_oracle(name, scale, offset, dtype):
    from stream_amd.mesh import AlphaShape3D

    print(f"[star3] {name} x {scale} + {offset} {np.dtype(dtype).name}", flush=True)
    pts, alpha = _cloud(name)
    pts = ((pts + offset) * scale).astype(dtype)
    al = np.broadcast_to(np.asarray(alpha * scale, dtype), len(pts)).copy()
    o = ol.ashape3d(pts, al, bits=21, dtype=dtype)
    a = AlphaShape3D(dtype=dtype, morton_bits=21)
    a.set_nodes(pts, al)
    a.compute()
    row, neig, eb = a.get_edges()
    assert np.array_equal(a.get_permutation(), o["perm"])
    assert np.array_equal(row, o["row"])
    assert np.array_equal(neig, o["neig"])
    assert np.array_equal(eb, o["edge_is_bnd"])
    assert np.array_equal(a.get_boundary_nodes(), o["node_is_bnd"])
    assert np.array_equal(a.get_elem(), o["elem"])
    if dtype == np.float64 and offset == 0.0:
        # room alone never counts as an exact evaluation
        assert a.get_nexact() <= o["n_exact_calls"]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [70, 90])
def test_exact_nodes_are_counted_whatever_else_they_need(n, dtype):
    """Five cospherical nodes, a centre and four of its sphere on one circle, and
    n more of the sphere in general position: these five need the exact stage,
    the centre's star outgrows 64 tetrahedra as well."""
    from stream_amd.mesh import AlphaShape3D

    four = np.array([[0.25, 0.125, 0.9375], [-0.25, 0.125, 0.9375], [0.25, -0.125, 0.9375], [-0.25, -0.125, 0.9375]])
    rng = np.random.default_rng(n)
    v = rng.standard_normal((40 * n, 3))
    v *= (np.linalg.norm(four[0]) * (1.0 + 1e-3 * rng.random(len(v))) / np.linalg.norm(v, axis=1))[:, None]
    v = v[v[:, 2] < 0.7][:n]  # the circle stays empty
    pts = np.concatenate([np.zeros((1, 3)), four, v]).astype(dtype)
    al = np.full(len(pts), 3.0, dtype)
    print(f"[star3] exact nodes n={n} {np.dtype(dtype).name}", flush=True)
    a = AlphaShape3D(dtype=dtype, morton_bits=21)
    a.set_nodes(pts, al)
    a.compute()
    o = ol.ashape3d(pts, al, bits=21, dtype=dtype)
    assert np.array_equal(a.get_elem(), o["elem"])
    assert o["n_exact_calls"] > 0 and a.get_nexact() == 5


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_coinciding_nodes_are_refused(dtype):
    """A star of coinciding points has no order to break ties by: its cavity's
    boundary does not close, and the node ends there (an id of the open boundary
    must not index anything).  The handle computes the next cloud."""
    from stream_amd import StreamError
    from stream_amd.mesh import AlphaShape3D

    print(f"[star3] coinciding nodes {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(10)
    a = AlphaShape3D(dtype=dtype, morton_bits=21)
    pts = np.repeat(rng.random((40, 3)), 2, axis=0).astype(dtype)
    a.set_nodes(pts, np.full(len(pts), 0.4, dtype))
    with pytest.raises(StreamError, match="capacity"):
        a.compute()
    pts = np.ascontiguousarray(pts[::2])
    al = np.full(len(pts), 0.4, dtype)
    a.set_nodes(pts, al)
    a.compute()
    assert np.array_equal(a.get_elem(), ol.ashape3d(pts, al, bits=21, dtype=dtype)["elem"])
