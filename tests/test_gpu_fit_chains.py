"""Fits with enough workgroups for the four-chain layouts (kmeans.hip, km_fit): mixed chains, chains by
problem, odd head counts, one problem. Every head must come out as in a fit of its own, which is one
chain of launches, with and without the packing."""
import pytest
import torch

from peco_amd import clustering_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(g, heads, tokens, clusters, length):
    x = torch.randn(heads, length, 64, generator=g, device=DEV)
    x += 3 * torch.randn(heads, 1, 64, generator=g, device=DEV) * torch.randint(3, (1, length, 1), generator=g, device=DEV)
    x = x.bfloat16()
    at = torch.randint(tokens, (heads, clusters), generator=g, device=DEV)
    return clustering_cuda.KMeansProblem(x[:, :tokens], x.float().gather(1, at[..., None].expand(-1, -1, 64)))


def _head(p, h):
    return clustering_cuda.KMeansProblem(p.x[h:h + 1], p.init[h:h + 1])


@pytest.mark.parametrize("heads,tokens,problems", [(24, 5000, 2), (5, 24001, 2), (41, 6000, 1)])
@pytest.mark.parametrize("pack", [False, True])
def test_chained_fit_equals_each_head_alone(heads, tokens, problems, pack):
    g = torch.Generator(device=DEV)
    g.manual_seed(heads)
    length = tokens + 7
    sets = [_problem(g, heads, tokens, clusters, length) for clusters in (20, 70)[:problems]]
    spec = [(4, length, None)] * problems if pack else None
    outs = clustering_cuda.kmeans_fit(sets, 5, pack=spec, pack_order="original" if pack else "cluster")
    packed = outs[1] if pack else None
    outs = outs[0] if pack else outs
    for i, p in enumerate(sets):
        for h in (0, heads // 4, heads // 2, heads - 1):
            one = clustering_cuda.kmeans_fit([_head(p, h)], 5, pack=spec and spec[:1],
                                             pack_order="original" if pack else "cluster")
            fit = one[0][0] if pack else one[0]
            assert all(torch.equal(a[h], b[0]) for a, b in zip(outs[i], fit))
            if pack:
                assert torch.equal(packed[i][0][h], one[1][0][0][0])
