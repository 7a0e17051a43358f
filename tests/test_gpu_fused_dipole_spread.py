"""The force backward's dipole grid for upstream vectors of very different size: contributions below 2^10 are converted to
fixed point by their mantissa, larger ones generally.  Scaling the upstream vectors by a power of two scales every
float32 product exactly, so the gradients scale with them up to the fixed-point steps (2^-40 on the grid, 2^-32 in the
sums, against gradients of 10^4 and more, which times 2^12 still fit the sums' range of 2^31): 1e-6 of the RMS."""

import pytest
import torch

from torchff.fused import for_workload
from torchff.workloads import make_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [2.0 ** 7, 2.0 ** 12])
def test_gradients_scale_with_the_upstream_vectors(scale):
    w = make_workload("water900")
    m = for_workload(w, "mixed")
    t = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda", requires_grad=True)
    box = torch.tensor(w["box"], dtype=torch.float64, device="cuda")
    torch.manual_seed(0)
    v = torch.randn(len(w["coords"]), 3, dtype=torch.float64).cuda()
    print(f"dipole spread scale {scale}", flush=True)
    out = []
    for s in (1.0, scale):
        inp = [t(w[k]) for k in ("coords", "charges", "sigma", "epsilon")]
        _, F, _ = m(inp[0], box, *inp[1:])
        (F * (v * s)).sum().backward()
        m.check()
        out.append([x.grad / s for x in inp[:2]])
    for a, b in zip(*out):
        assert (a - b).pow(2).mean().sqrt() <= 1e-6 * a.pow(2).mean().sqrt()
