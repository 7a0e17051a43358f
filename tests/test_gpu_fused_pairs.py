"""Pair list and pair kernels of the fused path at the edges of their units (GPU): systems of one to a few
hundred atoms (clusters of 32, groups of 8, quads of list entries partly filled), boxes of one or two
columns (every pair by its own minimum image) and longer ones (periodic shifts per entry), and up to 8
exclusion partners per atom spread over several clusters.  A pair missed, doubled or taken at the wrong
image changes its term by all of it, so the bounds follow from the arithmetic of one pair: float32 2e-6
relative (erfc by its polynomial 1.5e-6, the products and powers the rest), float64 1e-11 (library functions,
plus sums rounded to 2^-32), each times the summed magnitude of the pair terms; forces 1e-4 / 1e-9 of the
RMS of the real-space forces plus that of the reciprocal ones (which all but cancel in one molecule)."""

import numpy as np
import pytest
import torch
from scipy.special import erfc

from oracle import composite, pme
from torchff.workloads import COULOMB_KJMOL, ewald_alpha, water_box

pytestmark = pytest.mark.gpu


def _system(n_waters, L, group):
    """n_waters waters on an x-fastest lattice in the box L, every `group` consecutive waters one exclusion set."""
    n_lat = int(np.ceil(n_waters ** (1.0 / 3.0) - 1e-9))
    w = water_box(n_waters, 0.31 * n_lat, n_lat, seed=60 + n_waters)
    w["box"] = np.diag(np.asarray(L, dtype=np.float64))
    atoms = np.arange(3 * n_waters)
    sets = [atoms[k:k + 3 * group] for k in range(0, 3 * n_waters, 3 * group)]
    i, j = (np.concatenate([np.repeat(s, len(s)) for s in sets]), np.concatenate([np.tile(s, len(s)) for s in sets]))
    w["exclusions"] = np.stack([i, j], 1).astype(np.int64)
    w["pairs_excl"] = np.ascontiguousarray(w["exclusions"][i < j])
    w.update(cutoff=0.9, skin=0.0, K=25, order=5, alpha=ewald_alpha(0.9), name=f"water{n_waters}")
    return w


def _pair_magnitudes(w):
    """Summed |Lennard-Jones| and |Coulomb| terms of the pairs within the cutoff (excluded: erfc - 1)."""
    x, L = w["coords"], np.diag(w["box"])
    i, j = np.triu_indices(len(x), 1)
    d = x[i] - x[j]
    r = np.linalg.norm(d - L * np.rint(d / L), axis=1)
    keep = r <= w["cutoff"]
    i, j, r = i[keep], j[keep], r[keep]
    n = w["natoms"]
    excl = np.isin(i * n + j, w["pairs_excl"][:, 0] * n + w["pairs_excl"][:, 1])
    s6 = (0.5 * (w["sigma"][i] + w["sigma"][j]) / r) ** 6
    lj = 4.0 * np.sqrt(w["epsilon"][i] * w["epsilon"][j]) * s6 * (s6 + 1.0) * ~excl
    coul = COULOMB_KJMOL * np.abs(w["charges"][i] * w["charges"][j]) * np.abs(erfc(w["alpha"] * r) - excl) / r
    return lj.sum(), coul.sum()


@pytest.mark.parametrize("n_waters,L,group", [(1, (2.0, 2.0, 2.0), 1), (11, (2.0, 2.1, 2.2), 3),
                                              (43, (2.0, 2.0, 2.0), 3), (130, (4.0, 2.0, 2.2), 3),
                                              (216, (2.0, 2.3, 2.6), 1)])
@pytest.mark.parametrize("precision,te,tf", [("fp64", 1e-11, 1e-9), ("mixed", 2e-6, 1e-4)])
def test_pair_units(n_waters, L, group, precision, te, tf):
    from torchff.fused import for_workload
    w = _system(n_waters, L, group)
    E, F, terms, _ = composite.energy_forces(w)
    m = for_workload(w, precision)
    args = [torch.tensor(w[k], dtype=torch.float64, device="cuda") for k in ("coords", "box", "charges", "sigma",
                                                                              "epsilon")]
    print(f"pair units {n_waters} {L} {precision}", flush=True)
    _, Fd, td = m(*args, check=True)
    td, Fd = td.cpu().numpy(), Fd.cpu().numpy()
    lj, coul = _pair_magnitudes(w)
    assert abs(td[0] - terms["lj"]) <= te * (lj + 1.0)
    assert abs(td[1] - terms["coul_real"]) <= te * (coul + 1.0)
    x = torch.tensor(w["coords"], dtype=torch.float64, requires_grad=True)
    q = torch.tensor(w["charges"], dtype=torch.float64)
    rec = pme.pme_energy(x, torch.tensor(w["box"]), q, w["K"], w["alpha"], w["order"]) * COULOMB_KJMOL
    Fr = -torch.autograd.grad(rec, x)[0].numpy()
    rms = lambda a: np.sqrt(np.mean(a ** 2))
    assert rms(Fd - F) < tf * (rms(Fr) + rms(F - Fr))
    again = m(*args, check=True)  # the list and every sum are built in a fixed order
    assert torch.equal(again[1].cpu(), torch.from_numpy(Fd)) and torch.equal(again[2].cpu(), torch.from_numpy(td))
