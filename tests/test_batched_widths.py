"""Replicas run with one wavefront, with the width that few replicas take by themselves and in the mode
that inverts every candidate end in the same state: boxes without cells, with 3, 4 and 5 cells per side
(rows of nearby cells that wrap and that do not), sizes about the limit of the wider form, one factor
and two, and a cutoff small enough that most cells are left out of a leg."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(sizes, cutoff, chain_length, factors, classes, seed=4):
    from jellyfysh_amd.batch import DeviceBatch, lattice_positions
    lengths = (np.array(sizes) / 0.8) ** (1.0 / 3.0)
    pos = [lattice_positions(n, float(v), 0.05, np.random.default_rng([seed, n])) for n, v in zip(sizes, lengths)]
    return DeviceBatch(np.array(sizes, dtype=np.int32), lengths, pos, cutoff=cutoff, chain_length=chain_length, factors=factors,
                       seed=seed, classes=classes)


@pytest.mark.parametrize("cutoff,chain_length,factors", [
    (2.5, 1.0, ((12.0, 4.0), (6.0, -4.0))),
    (2.5, 4.0, ((12.0, 4.0), (6.0, -4.0))),
    (1.6, 0.7, ((12.0, 4.0), (6.0, -4.0))),
    (2.5, 1.0, ((12.0, 1.0),)),
])
@pytest.mark.parametrize("sizes", [[383, 31], [384, 2, 130], [900, 500, 340], [2048, 64]])
def test_gpu_widths_and_modes_agree(device, sizes, cutoff, chain_length, factors):
    wide = (max(sizes) / 0.8) ** (1.0 / 3.0) / min(cutoff, (max(sizes) / 0.8) ** (1.0 / 3.0) / 2) <= 8.99
    assert wide
    legs = 300
    runs = []
    for blocks, mode, classes in ((0, 0, ([16384], [1])), (64, 0, ([16384], [1])), (0, 0, ([16384], [2])), (64, 1, ([16384], [1])),
                                  (0, 2, ([16384], [1]))):
        b = _batch(sizes, cutoff, chain_length, factors, classes)
        b.set_max_blocks(blocks)
        b.set_mode(mode)
        print(sizes, cutoff, chain_length, len(factors), "blocks", blocks, "mode", mode, "width", classes[1][0], flush=True)
        b.run(legs)
        b.run(legs)
        if mode == 2:
            assert b.audit() == 0
        s = b.states()
        runs.append([s["active"], s["direction"], s["chain_left"], s["legs"], s["est"]] + list(b.positions()))
        b.close()
    for other in runs[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(runs[0], other))
