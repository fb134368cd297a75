"""Pair energies and gradients over the scopes and sizes that take the kernels' different paths: rows of
one to four wavefronts, the Coulomb Fourier part from structure factors (scopes all and inter, the pairs
out of scope taken off) and pair by pair (intra), and the powers with and without inlined forms.

The reference sums the pair functions in plain FP64 torch on the CPU.  Both sides are sums of rounded
terms: with at most 257 partners of relative error below 64 x 2^-53 (the reference's pow, erfc and cos, the
device's powers) and the sums' own n 2^-53, 1e-12 of the sum of magnitudes bounds the difference."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _configuration(n, length, seed):
    rng = np.random.default_rng(seed)
    m = int(math.ceil(n ** (1 / 3)))
    sites = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return np.mod((sites + rng.uniform(0.3, 0.7, (n, 3))) * length / m, length)


def _coulomb(torch, s, length, par):
    alpha, fc, pc, _ = par
    psi = torch.zeros(s.shape[:-1], dtype=torch.float64)
    for i in range(-pc, pc + 1):
        for j in range(-pc, pc + 1):
            for k in range(-pc, pc + 1):
                if i * i + j * j + k * k <= pc * pc:
                    r = (s + length * torch.tensor([i, j, k], dtype=torch.float64)).norm(dim=-1)
                    psi = psi + torch.erfc(alpha / length * r) / r
    for i in range(-fc, fc + 1):
        for j in range(-fc, fc + 1):
            for k in range(-fc, fc + 1):
                n2 = i * i + j * j + k * k
                if 0 < n2 <= fc * fc:
                    phase = 2 * math.pi / length * (i * s[..., 0] + j * s[..., 1] + k * s[..., 2])
                    psi = psi + math.exp(-math.pi ** 2 * n2 / alpha ** 2) / (math.pi * length * n2) * torch.cos(phase)
    return psi - math.pi / (alpha ** 2 * length)


def _pairs(torch, potential, s, length, par, cc):
    r2 = (s * s).sum(-1)
    if potential == "merged_image_coulomb":
        return par[3] * cc * _coulomb(torch, s, length, par)
    if potential == "inverse_power":
        return cc * par[1] * r2 ** (-par[0] / 2)
    if potential == "inverse_power_truncated":
        return torch.where(r2 < par[2] ** 2, cc * par[1] * (r2 ** (-par[0] / 2) - par[2] ** -par[0]), torch.zeros_like(r2))
    if potential == "lennard_jones":
        x6 = (par[1] ** 2 / r2) ** 3
        return par[0] * (x6 * x6 - x6)
    return par[2] * (r2.sqrt() - par[0]) ** int(par[1])


CASES = [("merged_image_coulomb", [3.45, 3, 1, 1.3], True), ("merged_image_coulomb", [3.0, 2, 2, -0.7], False),
         ("inverse_power", [12.0, 1.3], True), ("inverse_power", [9.0, 0.7], False),
         ("inverse_power_truncated", [6.0, -4.0, 1.4], True), ("lennard_jones", [4.0, 0.9], False),
         ("displaced_even_power", [1.0, 4.0, 30.0], False)]


@pytest.mark.parametrize("scope", ["all", "inter", "intra"])
@pytest.mark.parametrize("potential,par,charged", CASES)
@pytest.mark.parametrize("n", [2, 3, 64, 65, 129, 257])
def test_gpu_energy_and_gradients_match_plain_sums(device, n, potential, par, charged, scope):
    import torch
    from jellyfysh_amd.energy import pair_energy
    length = max(3.0, 1.1 * n ** (1 / 3))
    pos = _configuration(n, length, n)
    pos[0] -= length          # a unit outside of the box: its separations take more than one period
    charges = np.where(np.arange(n) % 2 == 0, 1.0, -0.8) if charged else np.ones(n)
    molecule = np.arange(n) // 3

    x = torch.tensor(pos, dtype=torch.float64, requires_grad=True)
    c = torch.tensor(charges, dtype=torch.float64, requires_grad=charged)
    s = x[None, :, :] - x[:, None, :]
    s = s - length * torch.floor(s.detach() / length + 0.5)
    same = torch.tensor(molecule[:, None] == molecule[None, :])
    pick = ~torch.eye(n, dtype=torch.bool)
    if scope != "all":
        pick = pick & (same if scope == "intra" else ~same)
    u = 0.5 * _pairs(torch, potential, s[pick], length, par, (c[:, None] * c[None, :])[pick])
    want = torch.autograd.grad(u.sum() + 0.0 * x.sum() + 0.0 * c.sum(), [x, c] if charged else [x])

    print(potential, scope, n, flush=True)
    xd = torch.tensor(pos, dtype=torch.float64, device="cuda", requires_grad=True)
    cd = torch.tensor(charges, dtype=torch.float64, device="cuda", requires_grad=True) if charged else None
    got_u = pair_energy(xd, par, potential, length, charges=cd, molecule=torch.tensor(molecule, device="cuda"), scope=scope)
    got = torch.autograd.grad(got_u, [xd, cd] if charged else [xd])
    # magnitudes that the sums' roundings scale with (a pair's Coulomb terms are below its 1 / r sum)
    size = float(u.abs().sum()) + 1e-3
    assert abs(got_u.item() - u.sum().item()) <= 1e-12 * size
    for a, b in zip(got, want):
        assert float((a.cpu() - b).abs().max()) <= 1e-12 * (float(b.abs().max()) * 10 + size)
