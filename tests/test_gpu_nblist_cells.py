"""The cell-list search at the edges of its units, pair set against the oracle's bit for bit: self pairs on the cell path
with and without the float32 prefilter, atoms with more exclusion partners than the kernel keeps (4), cells of more
than 64 atoms (several chunks of home atoms) and of more than 1024 (several batches of the half shell that begin inside
the home cell), orthorhombic and triclinic boxes."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import nblist as onb

pytestmark = pytest.mark.gpu

RC = 0.8
BOXES = {"prefilter": np.diag([4.0, 4.1, 3.9]),  # nine or ten cells an axis
         "exact": np.diag([2.6, 2.5, 2.7]),      # six: a cell pair's shift need not be the minimum image
         "triclinic": np.array([[3.6, 0.0, 0.0], [0.9, 3.5, 0.0], [-0.7, 0.8, 3.4]])}


def _coords(kind, B, rng):
    """300 atoms anywhere, and a clump that one cell (0.4 wide) holds."""
    f = rng.random((300, 3))
    extra = {"spread": 0, "clump of 150": 150, "clump of 1500": 1500}[kind]
    nc = np.floor(2.0 / RC / np.linalg.norm(np.linalg.inv(B), axis=0))  # cells per axis
    clump = (np.array([0, nc[1] - 1, nc[2] // 2]) + 0.5) / nc  # its half shell wraps on two axes
    f = np.concatenate([f, clump + 0.02 * (rng.random((extra, 3)) - 0.5)])
    return f[rng.permutation(len(f))] @ B


@pytest.mark.parametrize("include_self", [False, True])
@pytest.mark.parametrize("kind", ["spread", "clump of 150", "clump of 1500"])
@pytest.mark.parametrize("box", list(BOXES))
def test_cell_list_units(box, kind, include_self):
    import torchff
    from torchff import _lib
    B = BOXES[box]
    rng = np.random.default_rng(len(kind))
    dtype = torch.float32 if kind == "spread" else torch.float64
    x = torch.tensor(_coords(kind, B, rng), dtype=dtype, device="cuda")
    n = len(x)
    # groups of 8 exclude each other (7 partners), groups of 3 of the rest (2)
    sets = [np.arange(k, k + 8) for k in range(0, 160, 8)] + [np.arange(k, min(k + 3, n)) for k in range(160, n, 3)]
    excl = np.concatenate([np.stack(np.triu_indices(len(s), 1), 1) + s[0] for s in sets])
    bh, lib = (ctypes.c_double * 9)(*B.ravel()), _lib.load()
    assert lib.tff_nblist_workspace_bytes(n, bh, RC, 1) > lib.tff_nblist_workspace_bytes(n, bh, RC, 0) + 2000  # cells
    xh = x.double().cpu().numpy()
    ref = onb.neighbor_pairs(xh, B, RC, exclusions=excl, include_self=include_self)
    nl = torchff.NeighborList(n, exclusions=torch.tensor(excl, device="cuda"), include_self=include_self,
                              algorithm="cell_list").to("cuda")
    print(f"cell list {box} {kind} {include_self} {n} {len(ref)}", flush=True)
    pairs, npairs = nl(x, torch.tensor(B, dtype=dtype, device="cuda"), RC, len(ref) + 5, padding=True)
    got, found = pairs.cpu().numpy(), int(npairs.item())
    assert found == len(ref) and np.all(got[found:] == -1)
    np.testing.assert_array_equal(onb.canonicalize(got, found), ref)
