"""Candidates whose inversion ends in the reference's ValueError (an attractive unit passed so closely that
the root's argument rounds below zero): an error where no event of the candidate's set comes before it.
The others do not stop a run, whichever of them the horizon of a leg or its general form takes in."""
import numpy as np
import pytest

import systems as S

FIELDS = ("tagger", "flags", "active", "target", "tq", "tr", "pos", "ncand", "chash")
POWER, PREFACTOR = 5.0, -1.0


def _passes(oracle, nan):
    """Perpendicular separations of a unit ahead whose inversion is NaN (or is not) for every usual draw."""
    perps = [(1e-4 if nan else 1e-2) * (1.0 + k * 1e-2) for k in range(3)]
    for perp in perps:
        sep = np.array([0.3, (0.5 + perp) - 0.5, 0.0])
        dt = oracle.lib().ora_ip_displacement(3, 0, 1.0, oracle._dp(sep), 1.0, 1.0, POWER, PREFACTOR, 0.7, oracle.MATH_CR)
        assert np.isnan(dt) == nan
    return perps


def _wiring(chain_time, sampling=0.0):
    return S.standard_wiring([dict(S.factor_tagger("pull", "inverse_power", [POWER, PREFACTOR]), kind="pair_all")], chain_time,
                             1.0e9, sampling)


@pytest.mark.gpu
def test_gpu_error_that_comes_first_is_reported(device, oracle):
    from jellyfysh_amd.chain import DeviceChain, make_desc
    perp = _passes(oracle, True)[0]
    pos = np.array([[0.1, 0.5, 0.5], [0.4, 0.5 + perp, 0.5]])
    print("first", flush=True)
    chain = DeviceChain(make_desc(3, 2, 1.0, 1.0, 1, _wiring(5.0), 3, scheduler="list"), pos)
    with pytest.raises(RuntimeError, match="math domain"):
        chain.run(10)
    with pytest.raises(RuntimeError, match="math domain"):
        chain.run(10)
    chain.close()
    from jellyfysh_amd import _lib as L
    import ctypes
    step = DeviceChain(make_desc(3, 2, 1.0, 1.0, 1, _wiring(5.0), 3, scheduler="list"), pos)
    assert step.run(1, log=False) == 1                   # the start of run
    L.check(L.lib().ecmc_system_begin_leg(step._h))
    t, q = ctypes.c_int32(), ctypes.c_double()
    assert L.lib().ecmc_system_send_event_time(step._h, 0, ctypes.byref(q), ctypes.byref(q), ctypes.byref(t), ctypes.byref(t)) != 0
    step.close()


@pytest.mark.gpu
@pytest.mark.parametrize("case,legs", [("sampling", 5), ("pair_event", 2)])
def test_gpu_errors_behind_the_event_do_not_stop_a_run(device, oracle, case, legs):
    """The run up to the closest approaches is that of units passed at separations without the error: a
    unit behind pulls before them, or sampling events, which bring in the general form, come first."""
    from jellyfysh_amd.chain import DeviceChain, make_desc
    wiring = _wiring(5.0 if case == "pair_event" else 0.01, 0.003 if case == "sampling" else 0.0)
    logs = []
    for nan in (True, False):
        ahead = 0.15 if case == "pair_event" else 0.4
        pos = np.array([[0.1, 0.5, 0.5], [0.08, 0.55, 0.5]] + [[ahead, 0.5 + p, 0.5] for p in _passes(oracle, nan)])
        if case == "sampling":
            pos[1] = [0.0, 0.95, 0.95]      # an event of the set before the closest approaches
        print(case, "with errors" if nan else "without", flush=True)
        chain = DeviceChain(make_desc(3, len(pos), 1.0, 1.0, 1, wiring, 3, scheduler="list"), pos)
        logs.append(chain.run(legs))
        chain.close()
    assert logs[0]["tagger"][-1] == (0 if case == "pair_event" else len(wiring) - 3)
    for f in FIELDS:
        assert np.array_equal(logs[0][f], logs[1][f]), f
