"""fit_token_clusters with a tolerance (iterations launched ahead, settled entries skipped) against one
kmeans_fit call per iteration with the displacement taken in between: labels, centres, counts and
the iteration count, bit for bit."""
import math

import pytest
import torch

from peco_amd import clustering, clustering_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _stepwise(x, centers, max_iters, tol):
    for i in range(1, max_iters + 1):
        labels, means, counts, _, _ = clustering_cuda.kmeans_fit([clustering_cuda.KMeansProblem(x, centers)], 1)[0]
        shift = torch.linalg.vector_norm(means - centers, dim=-1).max().item()
        centers = means
        if shift <= tol:
            break
    return labels, centers, counts, i


def _equal(got, ref):
    assert got[3] == ref[3]
    assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2])
    assert torch.equal(got[1].view(torch.int32), ref[1].view(torch.int32))


@pytest.mark.parametrize("dtype,dim,heads,tokens,clusters", [
    (torch.float32, 128, 3, 700, 20), (torch.bfloat16, 64, 2, 257, 5), (torch.float16, 128, 1, 1000, 3),
    (torch.bfloat16, 128, 2, 8200, 40), (torch.float32, 64, 5, 64, 64), (torch.bfloat16, 128, 2, 300, 1)])
@pytest.mark.parametrize("max_iters,tol", [(1, 1e-4), (2, 1e-4), (8, 1e-4), (60, 1e-4), (60, 0.05), (9, 1e-30), (30, 1e6)])
def test_fit_with_tolerance_matches_stepwise(dtype, dim, heads, tokens, clusters, max_iters, tol):
    g = torch.Generator().manual_seed(tokens + clusters)
    means = torch.randn(heads, 8, dim, generator=g) * 3
    x = (means[:, torch.randint(8, (tokens,), generator=g)] + torch.randn(heads, tokens, dim, generator=g)).to(dtype)
    init = x[:, torch.randperm(tokens, generator=g)[:clusters]].float()
    x, init = x.to(DEV), init.to(DEV)
    _equal(clustering.fit_token_clusters(x, clusters, max_iters, tol, init), _stepwise(x, init, max_iters, tol))


def test_fit_with_tolerance_from_a_fixed_point_and_a_poisoned_head():
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 500, 64, generator=g).to(DEV)
    _, settled, _, used = clustering.fit_token_clusters(x, 6, 200, 1e-4, x[:, :6].contiguous())
    assert used < 200
    got = clustering.fit_token_clusters(x, 6, 50, 1e-4, settled)
    assert got[3] == 1
    _equal(got, _stepwise(x, settled, 50, 1e-4))
    settled = settled.clone()
    settled[1, 2, 0] = float("nan")  # its displacement is not a number and never passes the tolerance
    got = clustering.fit_token_clusters(x, 6, 11, 1e-4, settled)
    ref = _stepwise(x, settled, 11, 1e-4)
    assert got[3] == ref[3] == 11
    # The poisoned head does not reach the other one.
    assert torch.equal(got[0][0], ref[0][0]) and torch.equal(got[1][0], ref[1][0])
    assert torch.equal(got[1][0], settled[0]) and got[1][1, 2, 0].isnan()


def test_tolerance_is_rounded_down_to_float32():
    for value in (0.1, 1e-4, 1.0, 1e300, 5e-46, math.pi):
        f = clustering_cuda._float32_floor(value)
        assert f <= value and torch.nextafter(torch.tensor(f), torch.tensor(float("inf"))).double().item() > value


@pytest.mark.parametrize("max_iters", [1, 2, 3, 6, 7, 14, 15, 63, 64, 65, 150])
def test_fit_that_never_settles_runs_every_iteration(max_iters):
    """Every length of the last stretch between looks, and more iterations than one block of flags."""
    g = torch.Generator().manual_seed(5)
    x = torch.randn(2, 300, 64, generator=g).to(DEV)
    init = x[:, :4].contiguous()
    init[1, 2, 0] = float("nan")
    got, ref = (f(x, *a) for f, a in ((clustering.fit_token_clusters, (4, max_iters, 1e-4, init)),
                                      (_stepwise, (init, max_iters, 1e-4))))
    assert got[3] == ref[3] == max_iters
    assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2])
    assert torch.equal(got[1].nan_to_num(7.0), ref[1].nan_to_num(7.0))


def test_fit_from_its_fixed_point_launches_little(monkeypatch):
    """A fit that stops at once does not first launch the iterations of a long one."""
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 500, 64, generator=g).to(DEV)
    settled = clustering.fit_token_clusters(x, 6, 200, 1e-4, x[:, :6].contiguous())[1]
    library, launched = clustering_cuda._library(), []

    class Counting:
        def __getattr__(self, name):
            return getattr(library, name)

        def peco_kmeans_iterate(self, *args):
            launched.append(args[15])
            return library.peco_kmeans_iterate(*args)

    monkeypatch.setattr(clustering_cuda, "_library", Counting)
    assert clustering.fit_token_clusters(x, 6, 50, 1e-4, settled)[3] == 1
    assert sum(launched) <= 2
