"""A class given with one wavefront per replica is launched with one, whatever the number of replicas;
classes left to the default run wider where the replicas are few and large, but not beyond what the
card holds of all classes at once, and report it.  The events do not depend on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(sizes, classes):
    from jellyfysh_amd.batch import DeviceBatch, lattice_positions
    lengths = (np.array(sizes) / 0.8) ** (1.0 / 3.0)
    pos = [lattice_positions(n, float(v), 0.05, np.random.default_rng([1, i])) for i, (n, v) in enumerate(zip(sizes, lengths))]
    return DeviceBatch(np.array(sizes, dtype=np.int32), lengths, pos, seed=6, classes=classes)


@pytest.mark.parametrize("sizes,expected", [([383, 40], [1]), ([384, 40], [4]), ([2048] * 3, [4]), ([400] * 520, [2]), ([384] * 1040, [1])])
def test_gpu_explicit_width_is_kept_and_automatic_width_reported(device, sizes, expected):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus != 256:
        pytest.skip("widths worked out for 256 CUs")
    one, auto = _batch(sizes, ([16384], [1])), _batch(sizes, None)
    assert one.widths() == [1] and one.classes[1] == [1]
    assert auto.widths() == expected
    two = _batch(sizes, ([16384], [2]))
    assert two.widths() == [2]
    ends = []
    for b in (one, auto, two):
        print(len(sizes), max(sizes), b.widths(), flush=True)
        b.run(60)
        b.run_graph(60, 1)
        s = b.states()
        ends.append([s["active"], s["direction"], s["chain_left"], s["legs"], s["est"], np.concatenate(b.positions())])
    assert all(np.array_equal(x, y) for e in ends[1:] for x, y in zip(ends[0], e))
    auto.set_max_blocks(8)
    assert auto.widths() == [1]
    auto.set_max_blocks(0)
    assert auto.widths() == expected
    auto.set_classes([16384], [1])
    assert auto.widths() == [1]
    for b in (one, auto, two):
        b.close()


def test_gpu_automatic_width_counts_the_replicas_of_all_classes(device):
    import ctypes
    import torch
    from jellyfysh_amd import _lib as L
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("widths worked out for 256 CUs")
    b = _batch([64] * 500 + [500] * 20, ([256, 16384], [1, 1]))
    assert b.widths() == [1, 1]
    L.check(L.lib().ecmc_batch_set_automatic_width(b._h, 1))
    assert b.widths() == [1, 2]            # 520 replicas, though 20 alone would take four
    w = ctypes.c_int32()
    assert L.lib().ecmc_batch_class_width(b._h, 2, ctypes.byref(w)) != 0
    b.close()
