"""The float64 erfc of the pair kernels at large arguments: one pair at distance 1 with unit charges, the Ewald
parameter being the argument u, so that the energy is erfc(u) itself (every factor 1, no other term).

Tolerance, in units of e = 2^-53: the function may be off by as much as a C library's (3.2e-16, 3 e) and the
reference by another unit in the last place (2 e), the product and the sum by nothing: 5 e."""

import math

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi", [(0.0, 3.6), (3.6, 6.0), (6.0, 10.0), (10.0, 20.0), (20.0, 26.0)])
def test_erfc_at_large_arguments(lo, hi):
    t = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    x, box, one, zero = t([[0.0, 0, 0], [1.0, 0, 0]]), torch.eye(3, dtype=torch.float64).cuda() * 8.0, t([1.0, 1.0]), \
        t([0.0, 0.0])
    pairs = torch.tensor([[1, 0]], device="cuda")
    u = np.random.default_rng(int(10 * lo)).uniform(lo, hi, 400)
    print(f"far erfc {lo} {hi}", flush=True)
    with torch.no_grad():
        e = [torchff.compute_nonbonded_ewald_energy_from_atom_pairs(x, pairs, box, one, zero, one, 1.0, 2.0, float(a))
             for a in u]
    got = torch.stack([v.reshape(()) for v in e]).cpu().numpy()
    ref = np.array([math.erfc(a) for a in u])
    assert np.all(np.abs(got - ref) <= 5 * 2.0 ** -53 * ref)
