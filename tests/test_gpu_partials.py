"""The gradient's block partials, against the CPU oracle: node counts whose edge
kernels write 1, 63, 64, 65, 256 and 257 rows of partials (the reduction sums 64
rows side by side, 4 groups in flight), and graphs in which a few nodes carry the
whole gradient, so that a lost row or a lost rest of a block shows.  And their
workspace."""
import numpy as np
import pytest

from oracle import mpnn

pytestmark = pytest.mark.gpu


def _chain_lattice(n):
    """A row of n nodes coupled to the next and the next but one."""
    from scipy import sparse as sp

    rng = np.random.default_rng(n)
    w1, w2 = 0.5 + rng.random(n - 1), 0.2 + 0.3 * rng.random(n - 2)
    off = sp.diags([-w1, -w2], [1, 2], shape=(n, n))
    A = (off + off.T).tocsr()
    A = (A + sp.diags(0.5 - np.asarray(A.sum(1)).ravel())).tocsr()
    A.sort_indices()
    xy = np.stack([np.arange(n) / n, 0.1 * rng.random(n)], 1)
    bnd = np.zeros(n, np.uint8)
    return A.indptr.astype(np.uint32), A.indices.astype(np.uint32), A.data.astype(np.float64), xy, bnd


@pytest.mark.parametrize("n", [4, 32, 33, 252, 256, 257, 1024, 1025, 2049])
def test_gradient_matches_oracle(n):
    from stream_amd.learned import PrecLearned

    print(f"[partials] n={n}", flush=True)
    row, col, val, xy, bnd = _chain_lattice(n)
    w = mpnn.init_params(7)
    rng = np.random.default_rng(1)
    w = np.where(w == 0.0, 0.3 * rng.standard_normal(w.shape), w).astype(np.float32)
    net = PrecLearned(w)
    net.set_system(row, col, val, xy, bnd)
    loss, grad = net.gradient()
    ref_loss, ref = mpnn.backward(mpnn.unflatten(w.astype(np.float64)), mpnn.Graph(row, col, val, xy, bnd))[:2]
    ref = mpnn.flatten(ref)
    # same bf16 operands; activations on a rounding boundary may fall either
    # way (2^-8 of one value in a few tens of thousands)
    assert abs(loss - ref_loss) <= 1e-3 * max(1.0, abs(ref_loss))
    assert np.linalg.norm(grad - ref) <= 1e-2 * np.linalg.norm(ref)


def _live_windows():
    """(n, first live node): four coupled nodes, the rest without neighbours and on
    the boundary, so with no part in the gradient.  Up to 8,192 nodes block k of the edge kernels has nodes 4k
    .. 4k + 3.  41,000 nodes: the weight products take 64 rows per block in two
    stages, 40 in the last."""
    out = [(41_000, 40_996), (41_000, 64 * 100 + 60), (163_841, 163_837)]
    for n in (256, 257, 1020, 1024, 1025, 2049):
        blocks = (n + 3) // 4
        out += [(n, min(4 * k, n - 4)) for k in sorted({0, 63, 64, 191, 192, blocks - 2, blocks - 1}) if k < blocks]
    return out


def _few_live(n, first):
    _, _, val, xy, bnd = _chain_lattice(n)
    m = min(4, n - first)
    live = np.arange(first, first + m)
    col = [np.array([i]) for i in range(n)]
    for i in live:
        col[i] = live
    row = np.concatenate([[0], np.cumsum([len(c) for c in col])]).astype(np.uint32)
    col = np.concatenate(col).astype(np.uint32)
    val = np.ones(len(col))
    rng = np.random.default_rng(first)
    K = -0.2 - 0.3 * rng.random((m, m))
    K = K + K.T
    np.fill_diagonal(K, 0.0)
    np.fill_diagonal(K, 0.5 - K.sum(1))
    val[row[first]:row[first + m]] = K.ravel()
    bnd[:] = 1
    bnd[live] = 0
    return row, col, val, xy, bnd


@pytest.mark.parametrize("n, first", _live_windows())
def test_gradient_of_a_few_live_nodes_matches_oracle(n, first):
    from stream_amd.learned import PrecLearned

    print(f"[partials] n={n} live {first}", flush=True)
    row, col, val, xy, bnd = _few_live(n, first)
    w = mpnn.init_params(7)
    rng = np.random.default_rng(1)
    w = np.where(w == 0.0, 0.3 * rng.standard_normal(w.shape), w).astype(np.float32)
    net = PrecLearned(w)
    net.set_system(row, col, val, xy, bnd)
    loss, grad = net.gradient()
    ref_loss, ref = mpnn.backward(mpnn.unflatten(w.astype(np.float64)), mpnn.Graph(row, col, val, xy, bnd))
    assert abs(loss - ref_loss) <= 1e-3 * max(1.0, abs(ref_loss))
    # as above, by tensor; a lost block takes 0.7 or more of each
    got = mpnn.unflatten(grad.astype(np.float64))
    for name in ref:
        assert np.linalg.norm(got[name] - ref[name]) <= 2e-2 * np.linalg.norm(ref[name]), name


def test_partials_take_the_graph_s_own_blocks():
    """Workspace for the block partials: none without a gradient, then that of the
    graph's own blocks (75 x 12,352 floats for 2,400 nodes)."""
    import gc

    import stream_amd
    from stream_amd.learned import PrecLearned

    n = 2400
    print(f"[partials] workspace n={n}", flush=True)
    row, col, val, xy, bnd = _chain_lattice(n)
    net = PrecLearned(mpnn.init_params(7))
    gc.collect()  # other tests' networks
    net.set_system(row, col, val, xy, bnd)
    net.forward()
    before = stream_amd.device_bytes()["current"]
    net.gradient()
    assert stream_amd.device_bytes()["current"] - before == 4 * 75 * (3 * 64 * 64 + 64)
    # activations and their gradients take 1,856 floats a node
    net2 = PrecLearned(mpnn.init_params(7))
    net2.set_system(row, col, val, xy, bnd)
    before = stream_amd.device_bytes()["current"]
    net2.forward()
    assert stream_amd.device_bytes()["current"] - before < 1.2 * 4 * 1856 * n
