"""Two-leaf inverse powers that multiply by the charges, in systems without Coulomb taggers: the quick
test of their candidates takes the charges of both units, so that event logs equal the oracle's for
charges of either sign and any strength, in three and two dimensions, plain and truncated, over cells
and over all units, for one wavefront and four."""
import numpy as np
import pytest

import systems as S

pytestmark = pytest.mark.gpu

FIELDS = ("tagger", "flags", "active", "target", "tq", "tr", "pos", "ncand", "chash")


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("dim,kind,potential,params", [
    (3, "pair_cells", "inverse_power", [6.0, 1.0]),
    (3, "pair_all", "inverse_power", [1.0, 1.0]),
    (3, "pair_cells", "inverse_power_truncated", [6.0, 2.0, 1.5]),
    (2, "pair_cells", "inverse_power", [3.0, 1.0]),
    (2, "pair_all", "inverse_power_truncated", [12.0, 1.0, 1.5]),
])
def test_gpu_charged_inverse_power_matches_oracle(device, oracle, waves, dim, kind, potential, params):
    from jellyfysh_amd.chain import DeviceChain, make_desc
    rng = np.random.default_rng(dim)
    if dim == 3:
        m = 2 if waves == 1 else 4
        n, length = 4 * m ** 3, 1.6 * m + (1.0 if m == 2 else 0.0)
        pos = S.fcc_lattice(m, length / m, 0.02, rng)
    else:
        m = 6 if waves == 1 else 16
        n, length = m * m, 1.1 * m
        pos = S.square_lattice(m, length, 0.05, rng)
    charges = rng.choice([-1.0, 1.0, 0.5, -2.0], n)
    factors = [dict(S.factor_tagger("charged", potential, params, charge=True), kind=kind),
               dict(S.factor_tagger("core", "inverse_power", [12.0, 1.0]), kind=kind)]
    wiring = S.standard_wiring(factors, 0.8, 1.0e9)
    desc = make_desc(dim, n, length, 1.0, 3, wiring, 5, scheduler="heap")
    chain = DeviceChain(desc, pos, charges)
    legs = 600
    print(dim, kind, potential, params, "units", n, flush=True)
    got = np.concatenate([chain.run(legs // 2) for _ in range(2)])
    engine = oracle.Engine(S.oracle_config_from_wiring(dim, n, length, 1.0, 3, wiring, 5, math_mode=oracle.MATH_CR), pos, charges)
    want = engine.run(legs)
    assert (want["tagger"] == 0).sum() > 20 and len(set(charges[want["active"][1:]])) > 2
    for f in FIELDS:
        assert np.array_equal(got[f], want[f]), f
    assert np.array_equal(chain.positions(), engine.positions())
    plain = DeviceChain(desc, pos, charges)
    assert plain.run(legs, log=False) == legs
    assert np.array_equal(plain.positions(), chain.positions()) and plain.rng_words() == chain.rng_words()
    chain.close()
    plain.close()
