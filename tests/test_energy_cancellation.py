"""Coulomb rows whose pairs in scope are a small part of all charges: the structure factors hold the
whole system, so a row of few or weakly charged partners beside much charge out of scope (or beside a
strong charge of its own) is summed pair by pair, and units out of a row's scope leave nothing in it,
not even a value that is not finite.

The reference sums the pairs in scope in plain FP64 torch on the CPU.  A row's result is a sum of rounded
terms whose magnitudes add up to size = sum_j |c_j| (1 / r_ij + 4 / L) over its partners; the
structure-factor form adds at most as much out of scope.  With at most 1500 partners and 64 x 2^-53 a
term, (64 + 2 x 1500) 2^-53 < 1e-12 of that bounds the error."""
import math

import numpy as np
import pytest

from test_energy_scopes import _configuration, _coulomb

pytestmark = pytest.mark.gpu
PAR = [3.45, 4, 2, 1.3]


def _rows(torch, pos, charges, pairs, length):
    """Per unit: sum_j c_j psi, its gradient times c_i, and size, over the ordered pairs (i, j)."""
    x = torch.tensor(pos, dtype=torch.float64)
    c = torch.tensor(charges, dtype=torch.float64)
    i, j = (torch.tensor(v) for v in pairs)
    s = x[j] - x[i]
    s = (s - length * torch.floor(s / length + 0.5)).requires_grad_(True)
    psi = _coulomb(torch, s, length, PAR)
    (ds,) = torch.autograd.grad(psi.sum(), s)
    n = len(charges)
    add = lambda v: torch.zeros((n,) + v.shape[1:], dtype=torch.float64).index_add_(0, i, v)
    return (PAR[3] * add(c[j] * psi.detach()), -PAR[3] * c[:, None] * add(c[j][:, None] * ds),
            abs(PAR[3]) * add(c[j].abs() * (1.0 / s.detach().norm(dim=-1) + 4.0 / length)))


def _device(torch, pos, charges, molecule, scope, length):
    from jellyfysh_amd.energy import pair_energy
    x = torch.tensor(pos, dtype=torch.float64, device="cuda", requires_grad=True)
    c = torch.tensor(charges, dtype=torch.float64, device="cuda", requires_grad=True)
    u = pair_energy(x, PAR, "merged_image_coulomb", length, charges=c, molecule=torch.tensor(molecule, device="cuda"), scope=scope)
    gx, gc = torch.autograd.grad(u, [x, c])
    return u.item(), gx.cpu(), gc.cpu()


@pytest.mark.parametrize("case", ["large_molecule", "strong_molecule", "strong_unit"])
def test_gpu_weak_rows_keep_their_accuracy(device, case):
    import torch
    n = 200 if case == "strong_unit" else 1500
    length = 1.1 * n ** (1 / 3)
    pos = _configuration(n, length, 5)
    charges = np.where(np.arange(n) % 3 == 0, 1.0, 0.7)
    molecule = np.zeros(n, dtype=np.int32)
    scope = "inter"
    if case == "strong_unit":
        charges[17] = 1.0e9
        scope = "all"
        pairs = np.nonzero(~np.eye(n, dtype=bool))
    else:
        molecule[-2:] = 1
        if case == "strong_molecule":
            charges[:-2] *= 1.0e6
        pairs = np.nonzero(molecule[:, None] != molecule[None, :])
    print(case, n, flush=True)
    want_c, want_x, size = _rows(torch, pos, charges, pairs, length)
    u, got_x, got_c = _device(torch, pos, charges, molecule, scope, length)
    assert bool(((got_c - want_c).abs() <= 1e-12 * size).all())
    # a gradient's terms are below 8 times the value's at separations of at least 0.4
    bound = 1e-12 * 8 * size * torch.tensor(np.abs(charges))
    assert bool(((got_x - want_x).abs().amax(dim=1) <= bound).all())
    total = 0.5 * float((torch.tensor(charges) * want_c).sum())
    assert abs(u - total) <= 1e-12 * float((torch.tensor(np.abs(charges)) * size).sum())


@pytest.mark.parametrize("what", ["position", "position_infinite", "charge", "charge_infinite"])
def test_gpu_units_out_of_scope_that_are_not_finite(device, what):
    import torch
    n = 70
    length = 1.1 * n ** (1 / 3)
    pos = _configuration(n, length, 6)
    charges = np.where(np.arange(n) % 2 == 0, 1.0, -0.8)
    molecule = np.arange(n) // 2
    want_c, want_x, size = _rows(torch, pos, charges, np.nonzero(molecule[:, None] != molecule[None, :]), length)
    bad = float("inf") if what.endswith("infinite") else float("nan")
    if what.startswith("position"):
        pos[0, 1] = bad
    else:
        charges[0] = bad
    print(what, flush=True)
    u, got_x, got_c = _device(torch, pos, charges, molecule, "inter", length)
    # unit 1 shares unit 0's molecule, so none of its pairs holds it
    assert float((got_c[1] - want_c[1]).abs()) <= 1e-12 * float(size[1])
    assert float((got_x[1] - want_x[1]).abs().max()) <= 8e-12 * float(size[1])
    assert not math.isfinite(u) and not bool(torch.isfinite(got_c[2:]).any())
