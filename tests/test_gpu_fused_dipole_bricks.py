"""Force-matching gradients in mixed precision on charge grids whose last brick of 8 points is short (its home bricks
are found by interval overlap, and a stencil may reach two bricks back), unequal per axis, at the spline orders that
spread from the home-brick lists.  Reference: the float64 mode, whose backward spreads by another kernel.  The two
modes agree to 1e-4 of a gradient's RMS (the float32 bound of the oracle comparisons); a brick or a stencil point
missed or doubled changes the dipole grid by whole terms.  The backward that rebuilds the lists (another forward
call came in between) gives the bits of the one that reuses them."""

import pytest
import torch

from torchff.fused import FusedNonbondedPME
from torchff.workloads import make_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [4, 5, 6])
@pytest.mark.parametrize("K", [(25, 30, 27), (36, 25, 20), (18, 20, 25)])
def test_gradients_with_short_last_bricks(K, order):
    w = make_workload("water900")
    box = torch.tensor(w["box"], dtype=torch.float64, device="cuda")
    torch.manual_seed(0)
    v = torch.randn(len(w["coords"]), 3, dtype=torch.float64).cuda()
    print(f"dipole bricks {K} {order}", flush=True)

    def grads(precision, rebuild=False):
        m = FusedNonbondedPME(w["natoms"], w["cutoff"], w["alpha"], K, order=order, exclusions=w["exclusions"],
                              precision=precision)
        inp = [torch.tensor(w[k], dtype=torch.float64, device="cuda", requires_grad=True)
               for k in ("coords", "charges", "sigma", "epsilon")]
        _, F, _ = m(inp[0], box, *inp[1:])
        if rebuild:
            m((inp[0] + 0.01).detach().requires_grad_(True), box, *inp[1:])
        (F * v).sum().backward()
        m.check()
        return [x.grad for x in inp]

    mixed = grads("mixed")
    for a, r in zip(mixed, grads("fp64")):
        assert (a - r).pow(2).mean().sqrt() <= 1e-4 * r.pow(2).mean().sqrt()
    for a, r in zip(mixed, grads("mixed", rebuild=True)):
        assert torch.equal(a, r)
