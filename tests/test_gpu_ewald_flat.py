"""Direct Ewald at 33 to 53 values of m_z, where the lanes of the atom pass stride over all k: the ends of that range and
the first order past it, eight, several and one wave per atom.  float64 sums in another order than the oracle's: 1e-9
relative, as the float64 Ewald tests."""

import numpy as np
import pytest
import torch

import torchff
from oracle import ewald as oe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kmax,n,rank", [(16, 5, 0), (16, 5, 1), (16, 5, 2), (17, 1300, 1), (20, 300, 2), (25, 33, 0),
                                         (25, 33, 1), (25, 33, 2), (26, 33, 2), (16, 8193, 0)])
def test_lanes_striding_over_all_vectors(kmax, n, rank):
    rng = np.random.default_rng(100 * kmax + rank)
    box, alpha = np.array([[1.6, 0.0, 0.0], [0.2, 1.5, 0.0], [-0.1, 0.3, 1.7]]), 3.0
    x, q = rng.uniform(0, 1, (n, 3)) @ box, rng.normal(0, 0.4, n)
    p = rng.normal(0, 0.02, (n, 3)) if rank >= 1 else None
    th = None
    if rank >= 2:
        th = rng.normal(0, 0.01, (n, 3, 3))
        th = 0.5 * (th + th.transpose(0, 2, 1))
        th -= np.trace(th, axis1=1, axis2=2)[:, None, None] * np.eye(3) / 3
    sets = []
    print(f"ewald flat kmax {kmax} n {n} rank {rank}", flush=True)
    for dev in ("cpu", "cuda"):
        t = lambda a: None if a is None else torch.tensor(a, dtype=torch.float64, device=dev, requires_grad=True)
        v = [t(a) for a in (x, q, p, th)]
        b = torch.tensor(box, dtype=torch.float64, device=dev)
        if dev == "cpu":
            E = oe.ewald_recip_energy(v[0], b, v[1], kmax, alpha, p=v[2], th=v[3])
        else:
            E = torchff.Ewald(alpha, kmax, rank, return_fields=False)(v[0], b, *v[1:])
        E.sum().backward()
        sets.append([E.detach().reshape(1).cpu()] + [a.grad.cpu() for a in v if a is not None])
    for r, a in zip(*sets):
        assert (a.reshape(-1) - r.reshape(-1)).norm() <= 1e-9 * r.norm()
