"""Exclusion lists of the cluster-pair build made on the GPU against the host's sort: repeated, self and padding pairs,
both layouts, more pairs than one scan tile covers; what the build refuses.  Whole numbers: equal."""

import numpy as np
import pytest
import torch

import torchff
from torchff import _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["2xE", "Ex2"])
@pytest.mark.parametrize("n,pairs", [(1, 3), (40, 60), (9000, 9001), (20000, 50000)])
def test_lists_match_the_host(n, pairs, layout):
    rng = np.random.default_rng(n)
    i = rng.integers(0, n, pairs)
    coo = np.stack([i, (i + rng.integers(0, 4, pairs)) % n], 1)
    coo[rng.random(pairs) < 0.1] = [-1, 0]
    coo[pairs // 2:][:50] = coo[0]  # repeated
    e = torch.tensor(coo.T.copy() if layout == "2xE" else coo)
    rp, col = (t.tolist() for t in _ops._exclusions_csr(e, n, torch.device("cpu")))
    print(f"exclusion lists {n} {pairs} {layout}", flush=True)
    status = torch.zeros(1, dtype=torch.int64, device="cuda")
    grp, gcol = (t.tolist() for t in _ops._exclusions_csr(e.cuda(), n, torch.device("cuda"), status))
    assert int(status) == 0
    for k in range(n):
        row = [j for j in gcol[grp[k]:grp[k + 1]] if j >= 0]
        assert sorted(row) == col[rp[k]:rp[k + 1]]


def test_refuses():
    x = torch.rand(200, 3, device="cuda") * 2.0
    b = torch.eye(3, device="cuda") * 2.0
    build = lambda pairs: torchff.build_cluster_pairs(x, b, 0.6, torch.tensor(pairs, device="cuda"), 0.4)
    build([[0, k] for k in range(1, 17)] * 3)  # 16 partners, each three times
    with pytest.raises(RuntimeError, match="more than 16"):
        build([[0, k] for k in range(1, 18)])
    with pytest.raises(RuntimeError, match="past the atoms"):
        build([[0, 1], [3, 200]])
