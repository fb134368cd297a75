"""The leg loop's FP32 candidate test against full evaluations (the oracle's, of every candidate) over the
forms that it accepts: powers of 1 to 32 and those it does not take, plain and truncated, either sign,
with and without charges, over cells (few, many, one) and over all units, two to four taggers sharing
separations or not, boxes of very small and very large units, speeds and temperatures, sampling, one
wavefront and four.  Attractive powers are 6 and 12 in boxes of small or ordinary numbers, beside a
repulsive core: (k / U) ** (2 / p) of a number below one with 2 / p rounded down does not end in the
reference's ValueError where a unit is passed closely, which other systems do."""
import numpy as np
import pytest

import systems as S

pytestmark = pytest.mark.gpu

FIELDS = ("tagger", "flags", "active", "target", "tq", "tr", "pos", "ncand", "chash")
REPULSIVE = [1.0, 2.0, 3.0, 4.0, 5.0, 7.0, 8.0, 9.0, 12.0, 16.0, 24.0, 31.0, 32.0, 0.5, 2.5, 7.5, 33.0]


def _system(k):
    rng = np.random.default_rng([7, k])
    dim = 2 + k % 2
    m = int(rng.integers(1, 5)) if dim == 3 else int(rng.integers(3, 14))
    n = 4 * m ** 3 if dim == 3 else m * m
    scale = 10.0 ** [0, -3, 0, 3][k % 4]
    length = m * float(rng.uniform(1.4, 1.9) if dim == 3 else rng.uniform(0.9, 1.4)) * scale
    pos = S.fcc_lattice(m, length / m, 0.03 * length / m, rng) if dim == 3 else S.square_lattice(m, length, 0.05, rng)
    pos = np.where(pos >= length, 0.0, pos)
    kinds = ["pair_cells", "pair_all"]
    factors = []
    for f in range(int(rng.integers(1, 4))):
        attractive = scale <= 1.0 and rng.random() < 0.4
        p = float(rng.choice([6.0, 12.0] if attractive else REPULSIVE))
        pref = (-0.2 if attractive else 10.0 ** float(rng.uniform(-2, 0.5))) * scale ** p
        t = S.factor_tagger("f%d" % f, "inverse_power", [p, pref])
        if rng.random() < 0.4:
            t.update(potential="inverse_power_truncated", params=[p, pref, float(rng.uniform(0.2, 0.5)) * length])
        t.update(kind=kinds[int(rng.integers(2))], charge=bool(not attractive and p >= 6.0 and rng.random() < 0.4))
        factors.append(t)
    factors.append(dict(S.factor_tagger("core", "inverse_power", [12.0, scale ** 12]), kind=kinds[int(rng.integers(2))]))
    wiring = S.standard_wiring(factors, float(rng.uniform(0.05, 1.5)) * length, 1.0e9 * scale,
                               [0.0, 0.17][int(rng.integers(2))] * length, speed=float(rng.choice([1.0, 0.5, 3.0])))
    charges = rng.choice([0.3, 1.0, 2.5], n)      # (charges of both signs: test_charged_two_leaf.py)
    return dim, n, length, float(rng.choice([0.1, 1.0, 10.0])), int(rng.integers(1, 6)), wiring, pos, charges


@pytest.mark.parametrize("block", range(8))
def test_gpu_candidate_test_leaves_out_no_event(device, oracle, block):
    from jellyfysh_amd.chain import DeviceChain, make_desc
    for k in range(8 * block, 8 * block + 8):
        dim, n, length, beta, cells, wiring, pos, charges = _system(k)
        print(k, dim, n, "%.3g" % length, cells, [(t["potential"], t["params"][0], t["kind"]) for t in wiring if "potential" in t], flush=True)
        desc = make_desc(dim, n, length, beta, cells, wiring, k, scheduler="list")
        config = S.oracle_config_from_wiring(dim, n, length, beta, cells, wiring, k, scheduler="list", math_mode=oracle.MATH_CR)
        chain, plain = DeviceChain(desc, pos, charges), DeviceChain(desc, pos, charges)
        got, want = chain.run(150), oracle.Engine(config, pos, charges).run(150)
        assert plain.run(150, log=False) == 150
        for f in FIELDS:
            assert np.array_equal(got[f], want[f]), (k, f)
        assert np.array_equal(plain.positions(), chain.positions()) and plain.rng_words() == chain.rng_words()
        chain.close()
        plain.close()
