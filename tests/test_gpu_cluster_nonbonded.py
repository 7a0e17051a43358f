"""The nonbonded terms on cluster pairs (rows of 16 lanes rotating their columns) against the atom-pair op on the
decoded list: atom counts around the 32 slots of a cluster, both box kinds, each set of requested gradients, rows
with padding.  float64 sums the same terms in another order (1e-12 of the RMS); in float32 each pair term carries a
few ulp (twelve of s^12), which the cancelling force sums raise to at most 2e-5 of the RMS.

The float32 pair predicate is the decoded list's float64 one, also for pairs at the cutoff to within the rounding
of the coordinates and for coordinates several boxes away."""

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu
K = 138.935456
BOXES = {"ortho": np.diag([2.4, 2.6, 2.5]), "tri": np.array([[2.6, 0.0, 0.0], [0.5, 2.5, 0.0], [-0.4, 0.6, 2.4]])}


@pytest.mark.parametrize("want", ["", "x", "q", "xqse", "e"])
@pytest.mark.parametrize("n", [1, 31, 33, 500])
@pytest.mark.parametrize("box", ["ortho", "tri"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_terms_and_requested_gradients(dtype, box, n, want):
    rng = np.random.default_rng(n)
    B = BOXES[box]
    site = rng.permutation(512)[:n]  # a jittered 8^3 lattice, some atoms in other images
    f = (np.stack([site // 64, site // 8 % 8, site % 8], 1) + 0.25 * rng.random((n, 3))) / 8
    t = lambda a: torch.tensor(a, dtype=dtype, device="cuda")
    x, b = t((f + rng.integers(-1, 2, (n, 3))) @ B), t(B)
    par = dict(x=x, q=t(rng.normal(0, 0.5, n)), s=t(rng.uniform(0.15, 0.25, n)), e=t(rng.uniform(0.1, 0.6, n)))
    par["e"][::3] = 0
    excl = torch.tensor(np.stack([np.arange(0, n - 1), np.arange(1, n)]), device="cuda") if n > 1 else None
    print(f"cluster terms {dtype} {box} {n} {want}", flush=True)
    nbl = torchff.build_cluster_pairs(x, b, 0.9, excl, 0.4)
    pairs, _ = torchff.decode_cluster_pairs(x, b, *nbl, 0.9)
    outs = []
    for cluster in (True, False):
        p = {k: v.clone().requires_grad_(k in want) for k, v in par.items()}
        if cluster:
            E = torchff.compute_nonbonded_energy_from_cluster_pairs(p["x"], b, p["s"], p["e"], p["q"], K, 0.9, *nbl, True)
        else:
            E = torchff.compute_nonbonded_energy_from_atom_pairs(p["x"], pairs.long(), b, p["s"], p["e"], p["q"], K,
                                                                 0.9, True)
        if want:
            E.sum().backward()
        outs.append([E.detach().double().reshape(-1)] + [p[k].grad.double() for k in want])
    tol = 1e-12 if dtype == torch.float64 else 2e-5
    for a, r in zip(*outs):
        assert (a - r).pow(2).mean().sqrt() <= tol * r.pow(2).mean().sqrt()


@pytest.mark.parametrize("shift", [0, 2])
def test_float32_predicate_at_the_cutoff(shift):
    rng = np.random.default_rng(shift)
    m, L, rc = 2000, 40.0, 1.0
    k = np.arange(m)
    a = np.stack([k // 256, k // 16 % 16, k % 16], 1) * 2.5
    u = rng.normal(size=(m, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    x = np.empty((2 * m, 3))
    x[::2], x[1::2] = a, a + u * (rc * (1 + 3e-7 * rng.uniform(-1, 1, (m, 1))))
    x += rng.integers(-shift, shift + 1, x.shape) * L
    t = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")
    c, b = t(x), torch.eye(3, device="cuda") * L
    nbl = torchff.build_cluster_pairs(c, b, rc, None, 1.2)
    pairs, _ = torchff.decode_cluster_pairs(c, b, *nbl, rc)
    q = t(np.ones(2 * m)).requires_grad_(True)
    print(f"cluster predicate {shift}", flush=True)
    zero = t(np.zeros(2 * m))
    E = torchff.compute_nonbonded_energy_from_cluster_pairs(c, b, zero + 0.1, zero, q, K, rc, *nbl, False)
    E.sum().backward()
    listed = torch.zeros(2 * m, dtype=torch.bool, device="cuda")
    listed[pairs.long().reshape(-1)] = True
    assert 0.2 * m < int(listed.sum()) / 2 < 0.8 * m
    assert torch.equal(q.grad != 0, listed)
