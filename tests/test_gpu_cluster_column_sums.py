"""The column sums of the cluster-pair terms in float32: a column atom with 32 partners at one point, one of charge 1
and 31 of 2^-25 (half a unit in the last place of 1), in every order that the 32 lanes can meet them and for every
column of a row.  One float32 sum over all partners loses each small term that comes after the large one, up to
15.5 u of the result (u = 2^-24).  Tolerance: the sums are float64 after chains of eight float32 additions (7 u), the
distance, the product and the result round once each (3 u): 10 u."""

import numpy as np
import pytest
import torch

import torchff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lj_gradients", [False, True])
@pytest.mark.parametrize("triclinic", [False, True])
def test_float32_column_sums(triclinic, lj_gradients):
    C = 32  # clusters of partners; cluster C holds the column atoms
    n = 32 * C + C
    x, q = np.zeros((n, 3)), np.full(n, 2.0 ** -25)
    x[32 * C:, 0] = 0.5
    q[32 * C:] = 1.0
    q[33 * np.arange(C)] = 1.0  # cluster c: its slot c
    t = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda")
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")
    box = np.eye(3) * 8.0
    box[1, 0] = 1.0 if triclinic else 0.0
    order = i32(np.arange(n))
    none = i32(np.zeros((2, 0))), i32(np.zeros((0, 32)))
    print(f"cluster column sums {triclinic} {lj_gradients}", flush=True)
    for s in range(32):  # the column's place in its row
        ia = np.full((C, 32), -1)
        ia[:, s] = 32 * C + np.arange(C)
        xs, qs = t(x).requires_grad_(True), t(q).requires_grad_(True)
        sg = torch.full((n,), 0.1, device="cuda", requires_grad=lj_gradients)
        E = torchff.compute_nonbonded_energy_from_cluster_pairs(xs, t(box), sg, torch.zeros(n, device="cuda"), qs, 1.0,
                                                                1.0, order, *none, i32(np.arange(C)), i32(ia), False)
        E.sum().backward()
        tot = 1.0 + 31 * 2.0 ** -25
        dq, dx = qs.grad[32 * C:].double().cpu().numpy(), xs.grad[32 * C:, 0].double().cpu().numpy()
        assert np.all(np.abs(dq / (2.0 * tot) - 1.0) <= 10 * 2.0 ** -24)
        assert np.all(np.abs(dx / (-4.0 * tot) - 1.0) <= 10 * 2.0 ** -24)
