"""Training sets larger than what the network keeps on the device (64 MB,
fribo_mlp.hip) train in pieces: the same steps, bit for bit, as one call per
minibatch, within the memory of a piece."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_large_set_trains_in_pieces():
    torch = pytest.importorskip("torch")
    from fribois2d_amd.gpu import Mlp
    ni, no, n, batch = 256, 4, 400000, 5000     # 416 MB; pieces of 60000 samples, the last of 40000
    rng = np.random.default_rng(3)
    X = rng.standard_normal((n, ni), dtype=np.float32) / 16.0
    T = rng.standard_normal((n, no), dtype=np.float32)
    one = Mlp(ni, no, seed=9)
    free = torch.cuda.mem_get_info()[0]
    loss = one.train(X, T, 2, batch, 1e-3)
    kept = free - torch.cuda.mem_get_info()[0]
    each = Mlp(ni, no, seed=9)
    for _ in range(2):
        for s in range(0, n, batch):
            last = each.train(X[s:s + batch], T[s:s + batch], 1, batch, 1e-3)
    assert np.array_equal(one.params(), each.params())
    assert loss == last
    print(f"kept {kept / 2 ** 20:.0f} MiB", flush=True)
    assert kept <= 128 << 20     # a piece, the gradient parts, and the allocator's rounding
    one.close()
    each.close()


@pytest.mark.parametrize("n,batch", [(70000, 70000), (70000, 69000), (70000, 1 << 20)])
def test_a_minibatch_larger_than_a_piece(n, batch):
    """One minibatch is on the device as a whole, whatever its size."""
    pytest.importorskip("torch")
    from fribois2d_amd.gpu import Mlp
    ni, no = 256, 2
    rng = np.random.default_rng(4)
    X = rng.standard_normal((n, ni), dtype=np.float32) / 16.0
    T = rng.standard_normal((n, no), dtype=np.float32)
    one, each = Mlp(ni, no, seed=2), Mlp(ni, no, seed=2)
    loss = one.train(X, T, 2, batch, 1e-3)
    for _ in range(2):
        for s in range(0, n, batch):
            last = each.train(X[s:s + batch], T[s:s + batch], 1, n, 1e-3)
    assert np.array_equal(one.params(), each.params()) and loss == last
    one.close()
    each.close()
