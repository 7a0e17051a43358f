"""The energy-only launch of the pair terms (other workgroups and another order of rows than with gradients) against the
call with gradients, at list lengths around its chunks.  Charges of one sign and no Lennard-Jones term, so that the
energy is the sum of the terms' magnitudes: both sides add the same terms in float64, at most 100 additions one after
another (100 x 2^-53 = 1.2e-14; 1e-13), and round to the dtype (float32: 2^-23)."""

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-13), (torch.float32, 2.0 ** -23)])
@pytest.mark.parametrize("rows", [0, 1, 511, 513, 4095, 2 ** 20 + 3, 2 ** 22 + 2049])
def test_energy_only_matches_the_call_with_gradients(rows, dtype, tol):
    n = 4000
    rng = np.random.default_rng(rows)
    t = lambda a: torch.tensor(a, dtype=dtype, device="cuda")
    k = np.arange(n)
    x = t((np.stack([k // 400, k // 20 % 20, k % 20], 1) + 0.3 * rng.random((n, 3))) * 0.1)
    box = torch.diag(t([1.0, 2.0, 2.0]))
    q, s, e = t(rng.uniform(0.1, 0.5, n)), t(np.full(n, 0.1)), t(np.zeros(n))
    p = rng.integers(0, n, (rows, 2))
    p[p[:, 0] == p[:, 1]] = -1
    pairs = torch.tensor(p, device="cuda", dtype=torch.int64).reshape(-1, 2)
    print(f"energy only {rows} {dtype}", flush=True)
    call = lambda c: torchff.compute_nonbonded_energy_from_atom_pairs(c, pairs, box, s, e, q, 138.935456, 0.5, False)
    with torch.no_grad():
        a, again = call(x), call(x)
    b = call(x.clone().requires_grad_(True))
    assert torch.equal(a, again)
    assert abs(float(a) - float(b)) <= tol * float(b)
