"""The cluster-pair selection's prefix search (select.hip) where it can go wrong: key counts and
channel counts at the edges of its key blocks and channel chunks, many equal probabilities around
the threshold, and rows whose mass is not finite. The oracle is the torch restatement of
select_cluster_connections (peco/clustering.py:140-186)."""
import numpy as np
import pytest
import torch

from oracle import reference_path
from peco_amd import clustering, clustering_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(seed, h, cq, ck, dims):
    g = torch.Generator().manual_seed(seed)
    # The scores' spread is kept near 1.5 for every channel count.
    scale = 1.5 ** 0.5
    qc = torch.randn(1, h, cq, dims, generator=g) * scale
    kc = torch.randn(1, h, ck, dims, generator=g) * scale
    qs = torch.randint(0, 40, (1, h, cq), generator=g, dtype=torch.int32)
    ks = torch.randint(0, 40, (1, h, ck), generator=g, dtype=torch.int32)
    return qc, kc, qs, ks


@pytest.mark.parametrize("dims", [1, 3, 17, 64, 128, 220])
@pytest.mark.parametrize("ck", [1, 63, 64, 65, 129, 511, 512, 513, 1025, 2048])
def test_select_at_block_edges_matches_oracle(ck, dims):
    if 4 * (8 * ((dims + 3) // 4 * 4) + 64 * (dims + 1)) + 8 * ck > 65536:
        pytest.skip("refused shape")
    qc, kc, qs, ks = _case(ck * 7 + dims, 2, 9, ck, dims)
    for p, ratio in ((0.0, 0.3), (0.6, 0.0), (0.95, 0.02), (1.0, 0.0)):
        got = clustering.select_cluster_connections(qc.to(DEV), kc.to(DEV), qs.to(DEV), ks.to(DEV), p, ratio).cpu()
        assert torch.equal(got, reference_path.select_connections(qc, kc, qs, ks, p, ratio)), (p, ratio)


@pytest.mark.parametrize("ck,m", [(130, 129), (500, 300), (700, 640)])
def test_select_ties_across_blocks_match_oracle(ck, m):
    """m equal probabilities fl(1/m) at random keys (exact scores, counts of 1), zeros elsewhere: the
    kept prefix ends inside one group of ties, at the rank the sequential sum gives."""
    g = torch.Generator().manual_seed(m)
    kc = torch.zeros(1, 3, ck, 128)
    for r in range(3):
        kc[0, r, torch.randperm(ck, generator=g)[:m]] = 20.0
    qc = torch.ones(1, 3, 1, 128)
    qs, ks = torch.ones(1, 3, 1, dtype=torch.int32), torch.ones(1, 3, ck, dtype=torch.int32)
    prob = np.float32(1.0) / np.float32(m)
    befores = (np.cumsum(np.full(m, prob, np.float64)).astype(np.float32) - prob).astype(np.float32)
    for i in (1, 2, m // 3, m // 2, m - 2, m - 1):
        for p in (befores[i], np.nextafter(befores[i], np.float32(1)), np.nextafter(befores[i], np.float32(0))):
            got = clustering.select_cluster_connections(qc.to(DEV), kc.to(DEV), qs.to(DEV), ks.to(DEV), float(p), 0.0)
            assert torch.equal(got.cpu(), reference_path.select_connections(qc, kc, qs, ks, float(p), 0.0)), (i, p)


@pytest.mark.parametrize("poison", [float("nan"), float("inf")])
def test_select_non_finite_row_leaves_the_others(poison):
    """A query centroid that is not finite: every other row is the oracle's. Its own row, which takes the
    sequential walk, keeps exactly the minimum when no probability is a number (by index); with an
    infinite centroid the keys of infinite mass have the probability inf / inf, ordered last, and all
    keys of zero mass come before them and are kept."""
    qc, kc, qs, ks = _case(5, 2, 12, 300, 128)
    qs.clamp_(min=1)
    ref = reference_path.select_connections(qc, kc, qs, ks, 0.8, 5 / 300)
    qc[0, 1, 7, 3] = poison
    got, _, _ = clustering_cuda.select_connections(qc.to(DEV), kc.to(DEV), qs.to(DEV), ks.to(DEV), 0.8, 5)
    got = got.cpu()
    rows = [r for r in range(12) if r != 7]
    assert torch.equal(got[:, :1], ref[:, :1]) and torch.equal(got[0, 1, rows], ref[0, 1, rows])
    want = (ks[0, 1] > 0) & (kc[0, 1, :, 3] < 0)
    if poison != poison:
        want = torch.zeros(300, dtype=torch.bool)
        want[(ks[0, 1] > 0).nonzero()[:5, 0]] = True
        assert torch.equal(want, reference_path.select_connections(qc, kc, qs, ks, 0.8, 5 / 300)[0, 1, 7])
    assert want.sum() >= 5 and torch.equal(got[0, 1, 7], want)
