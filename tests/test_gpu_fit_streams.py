"""A fit of many workgroups runs as four chains of launches, three on library streams forked from and
joined back to the caller's stream: by problem (each problem's heads in halves) or, for two problems
of at most 16384 tokens with at least four heads, mixed (each chain a quarter of both problems'
heads). A fit of few runs as one chain on the caller's stream. Its results must not depend on the
layout, on which stream the caller is on, on calls queued back to back without a
synchronization, or on work the caller queues right after the call on its own stream."""
import pytest
import torch

from peco_amd import clustering_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problems(seed, h=3, n=5000, d=128, kq=16, kk=48):
    g = torch.Generator()
    g.manual_seed(seed)
    out = []
    for k in (kq, kk):
        means = torch.randn(h, 24, d, generator=g) * 3.0
        comp = torch.randint(24, (h, n), generator=g)
        x = (means.gather(1, comp[..., None].expand(-1, -1, d)) + torch.randn(h, n, d, generator=g))
        x = x.to(torch.bfloat16).to(DEV)
        idx = torch.randint(n, (h, k), generator=g).to(DEV)
        init = x.float().gather(1, idx[..., None].expand(-1, -1, d)).contiguous()
        out.append(clustering_cuda.KMeansProblem(x, init))
    return out


def _equal(a, b):
    return all(torch.equal(x, y) for pa, pb in zip(a, b) for x, y in zip(pa, pb))


# (heads, tokens, iterations). A fit is split from 897 assign workgroups (heads * ceil(tokens / 256) of both
# problems) and 4097 over its iterations on. The first three run as one chain; 24 heads of 5000 tokens
# (960 workgroups) as mixed chains; five of 24001 (940), one of them odd, by problem.
LAYOUTS = [(3, 5000, 4), (6, 3000, 4), (4, 17000, 4), (24, 5000, 5), (5, 24001, 5)]


@pytest.mark.parametrize("h,n,iterations", LAYOUTS)
def test_fit_on_a_caller_stream_matches_the_default_stream(announce, h, n, iterations):
    announce(f"two-problem fit on a caller stream, consumer on the same stream, H={h} N={n}")
    problems = _problems(1, h=h, n=n)
    ref = clustering_cuda.kmeans_fit(problems, iterations)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(device=DEV)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        out = clustering_cuda.kmeans_fit(problems, iterations)
        # Consumers queued on the caller's stream right after the call see finished results.
        total = out[1][2].sum() + out[0][2].sum()
        cent = out[1][1].clone()
    s.synchronize()
    assert _equal(ref, out)
    assert total.item() == 2 * h * n  # every token counted once per problem
    assert torch.equal(cent, ref[1][1])


@pytest.mark.parametrize("h,n,iterations", [(*shape[:2], 3) for shape in LAYOUTS[:2]] + LAYOUTS[3:])
def test_layouts_match_one_problem_fits(announce, h, n, iterations):
    """Each problem fitted alone (one chain) equals its part of the two-problem fit."""
    announce(f"two-problem fit against one-problem fits, H={h} N={n}")
    problems = _problems(2, h=h, n=n)
    both = clustering_cuda.kmeans_fit(problems, iterations)
    alone = [clustering_cuda.kmeans_fit([p], iterations)[0] for p in problems]
    torch.cuda.synchronize()
    assert _equal(both, alone)


@pytest.mark.parametrize("h,n,iterations", [(3, 5000, 3), *LAYOUTS[3:]])
def test_fits_queued_back_to_back(announce, h, n, iterations):
    announce(f"five two-problem fits queued without synchronization, H={h} N={n}")
    sets = [_problems(10 + i, h=h, n=n, kq=16 + i) for i in range(5)]
    refs = []
    for p in sets:
        refs.append(clustering_cuda.kmeans_fit(p, iterations))
        torch.cuda.synchronize()
    outs = [clustering_cuda.kmeans_fit(p, iterations) for p in sets]
    torch.cuda.synchronize()
    for r, o in zip(refs, outs):
        assert _equal(r, o)


@pytest.mark.parametrize("h,n,iterations", LAYOUTS[3:])
def test_fits_queued_from_two_streams(announce, h, n, iterations):
    """Calls of two streams share the library's streams and events: each one's consumers see its own
    finished results."""
    announce(f"six two-problem fits queued from two streams, H={h} N={n}")
    sets = [_problems(20 + i, h=h, n=n) for i in range(3)]
    refs = [clustering_cuda.kmeans_fit(p, iterations) for p in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=DEV) for _ in range(2)]
    outs = []
    for i in range(6):
        with torch.cuda.stream(streams[i % 2]):
            out = clustering_cuda.kmeans_fit(sets[i % 3], iterations)
            outs.append([[t.clone() for t in problem] for problem in out])
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        assert _equal(refs[i % 3], out)
