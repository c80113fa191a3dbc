"""Pinned staging memory of the state transfers: one block for all handles
that take turns, one per transfer that runs at the same time, nothing
allocated by the first read-back in a batch, nothing held without handles."""
import gc
import threading

import numpy as np
import pytest

from fribois2d_amd import cases

pytestmark = pytest.mark.gpu
BLOCK = 12 << 20   # three chunks of 4 MB


def _step(n3m, n2m, seed):
    from fribois2d_amd.gpu import FluidStep
    rc, zz = np.linspace(0.0, 6.0, n2m + 1), np.linspace(0.0, 8.0, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=8.0, rext2=6.0, visc=0.02, ibact=False)
    g = FluidStep(p, rc, zz)
    rng = np.random.default_rng(seed)
    st = {k: np.asfortranarray(rng.standard_normal((n2m + 1, n3m + 6))) for k in ("q2", "q3", "pr")}
    st.update({k: np.asfortranarray(rng.standard_normal((n2m + 1, n3m))) for k in ("ru2", "ru3")})
    return g, st


def _round_trip(g, st):
    g.set_state(st)
    back = g.get_state()
    return all(np.array_equal(back[k], st[k]) for k in st)


def test_handles_share_the_staging_memory():
    from fribois2d_amd import gpu
    held = gpu.load().fribo_staging_bytes
    gc.collect()
    before = held()
    # states of 0.03, 0.5, 2.4, 5.5, 11 and 26 MB, large after small and small after large
    sizes = [(32, 24), (131, 97), (300, 200), (450, 300), (600, 460), (900, 720), (131, 97), (600, 460), (32, 24)]
    hs = [_step(n3m, n2m, i) for i, (n3m, n2m) in enumerate(sizes)]
    for g, st in hs:
        assert _round_trip(g, st)
        assert 0 < held() <= max(before, BLOCK)
    small = [g for g, _ in hs[:3]]
    now = held()
    b = gpu.FluidBatch(small)
    for g, st in hs[:3]:
        back = g.get_state()
        assert all(np.array_equal(back[k], st[k]) for k in st)
    assert held() == now
    b.close()
    assert all(_round_trip(g, st) for g, st in hs)
    assert held() == now
    for g, _ in hs:
        g.close()
    if before == 0:
        assert held() == 0


def test_concurrent_transfers_have_blocks_of_their_own():
    from fribois2d_amd import gpu
    held = gpu.load().fribo_staging_bytes
    before = held()
    hs = [_step(300 + 40 * i, 260 + 30 * i, 10 + i) for i in range(4)]
    bad = []

    def work(g, st):
        for _ in range(12):
            if not _round_trip(g, st):
                bad.append(g)

    th = [threading.Thread(target=work, args=h) for h in hs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    assert held() <= max(before, len(hs) * BLOCK)
    for g, _ in hs:
        g.close()


def test_a_read_back_of_nothing_waits_for_the_handle():
    """fribo_get_state without arrays and fribo_fetch_fields without fields
    return when the handle's work is done: a fribo_sync after them has nothing
    left to wait for (the 200 rollbacks take about 2.5 ms; the sync
    itself some microseconds)."""
    import time
    from fribois2d_amd import gpu
    L = gpu.load()
    g, st = _step(1200, 1000, 3)
    g.set_state(st)
    g.save_state()
    for call in (lambda: L.fribo_get_state(g.h, *[None] * 11),
                 lambda: L.fribo_fetch_fields(g.h, 0, 1, 1, *[None] * 5)):
        for _ in range(200):
            g.restore_state()
        t0 = time.perf_counter()
        assert call() == 0
        t1 = time.perf_counter()
        g.sync()
        t2 = time.perf_counter()
        print(f"read-back {1e3 * (t1 - t0):.2f} ms, sync {1e3 * (t2 - t1):.3f} ms", flush=True)
        assert t2 - t1 < 1e-3
    g.close()
