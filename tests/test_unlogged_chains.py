"""Unlogged chains of four wavefronts whose legs have one barrier each (a single set inverted without
a quick test, the active unit kept by cell boundaries or refused cell vetoes, the random words made
ahead filling the ring), and chains whose sampling events send the leg through the general form, end in
the state of the logged run, which has barriers of its own between two legs' exchanges of winners."""
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


def test_gpu_unlogged_direct_legs_with_a_cell_veto_and_a_full_ring(device):
    from jellyfysh_amd.chain import DeviceChain, make_desc
    from jellyfysh_amd.batch import lattice_positions
    n, legs = 2800, 250
    length = n ** (1 / 3)
    pos = lattice_positions(n, length, 0.02, np.random.default_rng(3))
    charges = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    wiring = S.standard_wiring([dict(S.factor_tagger("lj", "lennard_jones", [1.0, 0.8]), kind="pair_all")], 0.9, 1.0e9)
    pairs = wiring[0]["create"]
    for t in wiring:
        for key in ("create", "trash"):
            if set(pairs) <= set(t[key]):
                t[key] = t[key] + ["veto"]
    wiring.append(dict(tag="veto", kind="cell_veto", potential="merged_image_coulomb", params=[3.45, 6.0, 2.0, 1.0],
                       bounding_params=[1.5, 10, 1.0, float("inf")], charge=True, create=wiring[0]["create"],
                       trash=wiring[0]["trash"], number_event_handlers=1))
    desc = make_desc(3, n, length, 2.0, 5, wiring, 12, scheduler="heap", max_occupants=1)
    logged, plain = DeviceChain(desc, pos, charges), DeviceChain(desc, pos, charges)
    print("logged run", flush=True)
    ev = logged.run(legs)
    veto = ev["tagger"] == len(wiring) - 1
    assert (veto & (ev["flags"] & 1 == 0)).any()         # vetoes that are refused: the active unit stays
    print("unlogged run", flush=True)
    assert plain.run(legs, log=False) == legs
    assert plain.active() == logged.active() and plain.rng_words() == logged.rng_words()
    assert np.array_equal(plain.positions(), logged.positions())
    assert np.array_equal(plain.estimators(), logged.estimators())
    logged.close()
    plain.close()
