"""The one-launch cluster size check (attention.hip) against the torch expressions it stands for, on
valid and invalid sizes (the flags only; nothing is asserted on the device here)."""
import pytest
import torch

from peco_amd import _native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("bh,cq,ck", [(1, 1, 1), (3, 64, 65), (24, 100, 500), (130, 257, 7)])
def test_size_flags_match_torch(bh, cq, ck):
    g = torch.Generator().manual_seed(bh + cq)
    qs = torch.randint(0, 9, (bh, cq), generator=g, dtype=torch.int32)
    ks = torch.randint(0, 9, (bh, ck), generator=g, dtype=torch.int32)
    qs[:, 0] += 9 * cq - qs.sum(-1).int()
    ks[:, -1] += 9 * ck - ks.sum(-1).int()
    sq, sk = 9 * cq, 9 * ck
    huge = ks.clone()
    huge[-1, 0] = 2**31 - 1  # sums past int32
    off = qs.clone()
    off[bh // 2, cq - 1] += 1
    negative = qs.clone()
    negative[-1, 0] -= 10 + negative[-1, 0]
    for a, b in ((qs, ks), (off, ks), (qs, huge), (negative, ks), (negative, -ks)):
        ok = torch.ones(4, dtype=torch.bool, device=DEV)
        a, b = a.to(DEV), b.to(DEV)
        status = _native.library().peco_check_cluster_sizes(_native.ptr(a), _native.ptr(b), bh, cq, ck, sq, sk,
                                                            _native.ptr(ok), _native.current_stream(a.device))
        assert status == 0
        want = [(a >= 0).all(), (b >= 0).all(), (a.sum(-1) == sq).all(), (b.sum(-1) == sk).all()]
        assert ok.tolist() == [bool(w) for w in want]
