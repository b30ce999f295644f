"""put / get of a field through the pinned chunks: boxes below, at and past
the chunk size (2**20 floats), whole boxes equal."""
import numpy as np
import pytest

from cm1_amd import model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk", [(8, 8, 6), (57, 121, 125), (249, 121, 29), (250, 121, 29), (401, 230, 70)])
def test_put_get_round_trip(require_gpu, ni, nj, nk):
    m = model.Model(model.make_config(ni=ni, nj=nj, nk=nk))
    rng = np.random.default_rng(ni)
    a = rng.standard_normal((m.pz, m.py, ni + 7)).astype(np.float32)
    b = rng.standard_normal((m.pz, m.py, ni + 7)).astype(np.float32)
    for _ in range(2):
        m.put("dum1", a)
        m.put("dum2", b)
        assert np.array_equal(m.get("dum1"), a)
        assert np.array_equal(m.get("dum2"), b)
    m.close()


@pytest.mark.parametrize("ni,nj,nk", [(57, 40, 20), (401, 230, 70)])
def test_fetches_from_several_threads(require_gpu, ni, nj, nk):
    """Fields of one model fetched (and one stored again) by threads side by
    side: every thread gets its own field's bytes."""
    import threading

    m = model.Model(model.make_config(ni=ni, nj=nj, nk=nk))
    rng = np.random.default_rng(ni)
    want = {n: rng.standard_normal((m.pz, m.py, ni + 7)).astype(np.float32) for n in ("dum1", "dum2", "dum3")}
    for n, a in want.items():
        m.put(n, a)
    bad = []

    def work(n, store):
        for q in range(10):
            if not np.array_equal(m.get(n), want[n]):
                bad.append((n, q))
            if store:
                m.put(n, want[n])

    threads = [threading.Thread(target=work, args=(n, n == "dum3")) for n in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    m.close()
    assert not bad, bad


def test_move_with_another_device_current(require_gpu):
    import torch

    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    m = model.Model(model.make_config(ni=57, nj=40, nk=20))
    a = np.random.default_rng(3).standard_normal((m.pz, m.py, 64)).astype(np.float32)
    with torch.cuda.device(1):
        m.put("dum1", a)
        assert np.array_equal(m.get("dum1"), a)
        assert torch.cuda.current_device() == 1
    m.close()
