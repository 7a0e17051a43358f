"""The float64 erfc, exp and 1/sqrt of the pair kernels, pair by pair against the C library: isolated pairs at known
distances, the charge gradient being coul erfc(a r) / r and the force coul (erfc(a r) / r + 2 a / sqrt(pi)
exp(-(a r)^2)) / r.

Tolerance, in units of e = 2^-53: u = a r is off by at most 2.5 e (square root, two products), which erfc and exp
turn into at most (2 u^2 + 1) 2.5 e; the functions themselves are off by at most 6 e, the products that follow by
6 e and the reference by 3 e.  The gradients are summed as integers of 2^-56 (1.5 steps)."""

import math

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [0.0, 1.0, 3.4, 4.0, 40.0])
def test_pair_functions_against_the_c_library(alpha):
    coul, m = 2.0 ** 20, 4000
    r = np.concatenate([np.linspace(0.09, 1.2, m - 4), [2.0 ** -10, 0.25, 0.5, 1.0]])
    x = np.zeros((2 * m, 3))
    x[1::2, 0] = r
    t = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    xs, q = t(x).requires_grad_(True), t(np.ones(2 * m)).requires_grad_(True)
    zero = t(np.zeros(2 * m))
    pairs = torch.arange(2 * m, device="cuda").reshape(m, 2)
    print(f"pair functions alpha {alpha}", flush=True)
    E = torchff.compute_nonbonded_ewald_energy_from_atom_pairs(xs, pairs, torch.eye(3, dtype=torch.float64,
                                                               device="cuda") * 64.0, zero + 0.1, zero, q, coul,
                                                               1.5, alpha)
    E.sum().backward()
    dq, f = q.grad.cpu().numpy()[1::2], xs.grad.cpu().numpy()[1::2, 0]
    u = alpha * r
    ec = np.array([math.erfc(v) for v in u])
    em = np.array([math.exp(-float(v) * float(v)) for v in u])
    # the reference's own exp(-u u) is off by u^2 e more
    e = 2.0 ** -53
    rel = ((2 * u * u + 1) * 2.5 + 15 + u * u) * e
    step = 1.5 * 2.0 ** -56
    assert np.all(np.abs(dq - coul * ec / r) <= rel * coul * ec / r + step)
    g = coul * (ec / r + 2 * alpha / math.sqrt(math.pi) * em) / r
    assert np.all(np.abs(-f - g) <= rel * g + step)
