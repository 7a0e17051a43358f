"""Direct Ewald where its lanes are split differently: 21, 4, 2, 1 and 1 atoms (or lines) per wave step, few and many
waves per atom.  Both sides sum the same float64 terms in other orders: 1e-9 relative, as the float64 Ewald tests."""

import numpy as np
import pytest
import torch

import torchff
from oracle import ewald as oe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kmax,n", [(1, 5), (7, 1300), (15, 17), (16, 2), (31, 3)])
@pytest.mark.parametrize("rank", [0, 1, 2])
def test_orders_and_atom_counts(kmax, n, rank):
    rng = np.random.default_rng(kmax)
    box, alpha = np.array([[1.6, 0.0, 0.0], [0.2, 1.5, 0.0], [-0.1, 0.3, 1.7]]), 3.0
    x, q = rng.uniform(0, 1, (n, 3)) @ box, rng.normal(0, 0.4, n)
    p = rng.normal(0, 0.02, (n, 3)) if rank >= 1 else None
    th = None
    if rank >= 2:
        th = rng.normal(0, 0.01, (n, 3, 3))
        th = 0.5 * (th + th.transpose(0, 2, 1))
        th -= np.trace(th, axis1=1, axis2=2)[:, None, None] * np.eye(3) / 3
    sets = []
    print(f"ewald lanes kmax {kmax} n {n} rank {rank}", flush=True)
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
