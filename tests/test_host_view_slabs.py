"""The host views of several systems lie in shared slabs of pinned memory: systems of equal and different
sizes that are made, run and destroyed in any order, also on several threads, read what a system alone
reads."""
import threading

import numpy as np
import pytest

import systems as S

pytestmark = pytest.mark.gpu


def _system(cells, seed):
    from jellyfysh_amd.chain import DeviceChain
    meta, pos = S.lj_system(n_cells=cells, rho=0.8, seed=seed)
    return DeviceChain(S.device_desc(meta), pos)


def _read(c):
    return [c.positions(), c.estimators(), np.array(c.active()), np.array(c.rng_words())]


def _alone(cells, seed, legs):
    c = _system(cells, seed)
    assert c.run(legs, log=False) == legs
    out = _read(c)
    c.close()
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_gpu_systems_made_and_destroyed_in_any_order(device):
    from jellyfysh_amd.chain import run_together
    want = {(cells, seed): _alone(cells, seed, 40) for cells in (2, 3) for seed in range(6)}
    rng = np.random.default_rng(1)
    live = []
    for step in range(60):
        print("step", step, "systems", len(live), flush=True)
        if len(live) < 4 or rng.random() < 0.6:
            key = (int(rng.integers(2, 4)), int(rng.integers(6)))
            live.append((key, _system(*key)))
        else:
            live.pop(int(rng.integers(len(live))))[1].close()
    fresh = [(k, c) for k, c in live]
    legs, _ = run_together([c for _, c in fresh], 40)
    assert (legs == 40).all()
    for key, c in fresh:
        assert _same(_read(c), want[key])
    for _, c in fresh[::2]:
        c.close()
    again = _system(3, 2)
    assert again.run(40, log=False) == 40 and _same(_read(again), want[(3, 2)])
    for key, c in fresh[1::2]:
        assert _same(_read(c), want[key])
        c.close()
    again.close()


def test_gpu_systems_of_several_threads(device):
    want = [_alone(2, seed, 25) for seed in range(4)]
    bad = []

    def work(t):
        try:
            for k in range(6):
                cs = [_system(2, (t + i) % 4) for i in range(1 + (t + k) % 5)]
                for c in cs:
                    c.run(25, log=False)
                if not all(_same(_read(c), want[(t + i) % 4]) for i, c in enumerate(cs)):
                    bad.append((t, k))
                for c in cs:
                    c.close()
        except Exception as e:      # a thread's exception would pass unseen
            bad.append(repr(e))

    print("four threads", flush=True)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
