"""What a launch leaves in host memory for the readers (state, committed legs, positions) is what a
system without resident positions copies back, also after steps that the host drives."""
import os

import numpy as np
import pytest

import systems as S

pytestmark = pytest.mark.gpu


def _chain(seed):
    from jellyfysh_amd.chain import DeviceChain
    meta, pos = S.lj_system(n_cells=3, rho=0.8, seed=seed)
    return DeviceChain(S.device_desc(meta), pos)


def _big():
    """A system whose positions do not fit into LDS, so that all of its launch work on global memory."""
    from jellyfysh_amd.chain import DeviceChain, make_desc
    from jellyfysh_amd import config
    from jellyfysh_amd.config import RunConfig
    from jellyfysh_amd.batch import lattice_positions
    n = 8000
    length = (n / 0.8) ** (1.0 / 3.0)
    cfg = RunConfig.from_file(os.path.join(os.path.dirname(config.__file__), "configs", "lennard_jones_truncated.ini"))
    desc = make_desc(3, n, length, cfg.beta, int(length / 2.5), cfg.taggers, 5, scheduler=cfg.scheduler)
    return DeviceChain(desc, lattice_positions(n, length, 0.01, np.random.default_rng(5)))


def _read(c):
    return [c.positions(), c.estimators(), np.array(c.active()), np.array(c.rng_words())]


def _same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(_read(a), _read(b)))


@pytest.mark.parametrize("legs", [1, 63, 500])
def test_gpu_readers_agree_with_and_without_residency(device, legs):
    from jellyfysh_amd.chain import run_together
    a, b, big = _chain(3), _chain(3), _big()
    assert a.launch_lds()[1] and not big.launch_lds()[1]
    _same(a, b)                                   # before any launch
    print("resident run, then in one launch with a big system", flush=True)
    assert a.run(legs, log=False) == legs
    n, _ = run_together([b, big], legs)
    assert list(n) == [legs, legs]
    _same(a, b)
    assert a.run(legs, log=False) == legs and b.run(legs, log=False) == legs
    _same(a, b)


@pytest.mark.parametrize("together", [False, True])
def test_gpu_reader_on_another_thread_sees_whole_launches(device, together):
    """A reader beside a running launch gets the state before it or after it, never a part of it."""
    import threading
    from jellyfysh_amd.chain import run_together
    legs = 20000
    a, b = _chain(3), _chain(3)
    states = [_read(b)]
    for _ in range(2):
        b.run(legs, log=False)
        states.append(_read(b))
    keys = [[s[0].tobytes() for s in states], [s[1].tobytes() for s in states]]
    done = []

    def work():
        for _ in range(2):
            done.append(run_together([a], legs)[0][0] if together else a.run(legs, log=False))

    t = threading.Thread(target=work)
    print("reading beside two launches", flush=True)
    t.start()
    seen = [[], []]
    for _ in range(20000):
        seen[0].append(keys[0].index(a.positions().tobytes()))
        seen[1].append(keys[1].index(a.estimators().tobytes()))
        if not t.is_alive():
            break
    t.join(60)
    assert done == [legs, legs]
    assert all(s == sorted(s) for s in seen)
    _same(a, b)
