"""The LDS-table pair kernel (coordinate and charge gradients) against the general pair kernel, which a call that
also asks for sigma gradients takes, and on lists that its table does not suit: random order (far more atoms per
chunk than slots), one atom in every row, repeated rows, padding rows and lengths around the rows of a chunk
(512 threads x 1 to 4 rows).  Both kernels sum the same float64 contributions as integers, in other groupings of a
run: coordinates 1e-13 of the gradient RMS in float64, 1e-6 in float32 (one rounding of the result)."""

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu


def _list(kind, n, rows, rng):
    if kind == "random":
        p = rng.integers(0, n, (rows, 2))
    elif kind == "hub":  # every row holds atom 7
        p = np.stack([np.full(rows, 7), rng.integers(8, n, rows)], 1)
        p[::2] = p[::2, ::-1]
    elif kind == "runs":  # rows of one atom together, the partners near it
        i = np.sort(rng.integers(16, n, rows))
        p = np.stack([i, i - rng.integers(1, 16, rows)], 1)
    else:  # the same pair over and over, with padding rows between
        p = np.tile([[11, 3]], (rows, 1))
        p[rng.random(rows) < 0.5] = -1
    p[p[:, 0] == p[:, 1]] = -1
    return p


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-13), (torch.float32, 1e-6)])
@pytest.mark.parametrize("kind,rows", [("random", 40000), ("random", 2 ** 21 + 77), ("hub", 9001), ("runs", 511),
                                       ("runs", 100003), ("repeat", 5000), ("runs", 1)])
def test_table_kernel_matches_general_kernel(kind, rows, dtype, tol):
    n = 6000
    rng = np.random.default_rng(rows)
    L = 4.0
    box = torch.eye(3, dtype=dtype, device="cuda") * L
    t = lambda a: torch.tensor(a, dtype=dtype, device="cuda")
    # a jittered lattice keeps the pair terms of one size
    k = np.arange(n)
    x = t((np.stack([k // 400, k // 20 % 20, k % 20], 1) + 0.3 * rng.random((n, 3))) * (L / 20))
    q, s, e = t(rng.normal(0, 0.4, n)), t(rng.uniform(0.1, 0.15, n)), t(rng.uniform(0.1, 0.6, n))
    pairs = torch.tensor(_list(kind, n, rows, rng), device="cuda")
    print(f"pair table {kind} {rows} {dtype}", flush=True)
    got = []
    for sigma_grad in (False, True):
        xs, qs = x.clone().requires_grad_(True), q.clone().requires_grad_(True)
        ss = s.clone().requires_grad_(sigma_grad)
        E = torchff.compute_nonbonded_ewald_energy_from_atom_pairs(xs, pairs, box, ss, e, qs, 138.935456, 1.4, 2.0)
        E.sum().backward()
        got.append((E.detach().double(), xs.grad.double(), qs.grad.double()))
    for a, b in zip(*got):
        scale = b.pow(2).mean().sqrt()
        assert (a - b).abs().max() <= tol * max(float(scale), float(b.abs().max())) + 1e-300
    # the same list again: bitwise the same gradients
    xs = x.clone().requires_grad_(True)
    qs = q.clone().requires_grad_(True)
    torchff.compute_nonbonded_ewald_energy_from_atom_pairs(xs, pairs, box, s, e, qs, 138.935456, 1.4, 2.0).sum().backward()
    assert torch.equal(xs.grad.double(), got[0][1]) and torch.equal(qs.grad.double(), got[0][2])
