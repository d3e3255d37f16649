"""The gradient's block-partial sums at sizes on both sides of the row
groups the reduction kernel walks (64 rows side by side, 4 groups in
flight): node counts whose edge kernels write 1, 63, 64, 65, 256 and 257
rows of partials, against the CPU oracle."""
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
