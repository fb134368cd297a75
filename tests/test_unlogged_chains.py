"""Unlogged chains of four wavefronts whose legs have one barrier each (a single set inverted without
a quick test, the active unit kept by cell boundaries), and chains whose sampling events send the leg
through the general form, end in the state of the logged run, which has barriers of its own between
two legs' exchanges of winners."""
import numpy as np
import pytest

import systems as S

pytestmark = pytest.mark.gpu

LJ = [S.factor_tagger("lj_twelve", "inverse_power", [12.0, 4.0]), S.factor_tagger("lj_six", "inverse_power", [6.0, -4.0])]


@pytest.mark.parametrize("name,factors,sampling", [
    ("lennard_jones", [S.factor_tagger("lj", "lennard_jones", [4.0, 1.0])], 0.0),
    ("hard_sphere", [S.factor_tagger("sphere", "hard_sphere", [0.3])], 0.0),
    ("non_integer_power", [S.factor_tagger("soft", "inverse_power", [7.5, 1.0])], 0.0),
    ("lennard_jones_sampled", [S.factor_tagger("lj", "lennard_jones", [4.0, 1.0])], 0.07),
    ("two_factors_sampled", LJ, 0.07),
])
def test_gpu_unlogged_chain_ends_where_the_logged_one_does(device, name, factors, sampling):
    from jellyfysh_amd.chain import DeviceChain, make_desc
    n, length = 500, (500 / 0.8) ** (1 / 3)
    pos = S.fcc_lattice(5, length / 5, 0.02, np.random.default_rng(8))
    wiring = S.standard_wiring(factors, 0.9, 1.0e9, sampling)
    desc = make_desc(3, n, length, 1 / 1.5, 3, wiring, 31, scheduler="heap")
    logged, plain = DeviceChain(desc, pos), DeviceChain(desc, pos)
    print(name, "logged run", flush=True)
    kinds = np.concatenate([logged.run(700) for _ in range(2)])["tagger"]
    assert (kinds == len(factors)).any()                 # cell boundaries: the active unit stays
    assert not sampling or (kinds == len(factors) + 1).any()
    print(name, "unlogged run", flush=True)
    assert [plain.run(700, log=False) for _ in range(2)] == [700, 700]
    assert plain.active() == logged.active() and plain.rng_words() == logged.rng_words()
    assert np.array_equal(plain.positions(), logged.positions())
    assert np.array_equal(plain.estimators(), logged.estimators())
    logged.close()
    plain.close()
