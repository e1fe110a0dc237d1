"""The device-ranged stable argsort of labels (sort.hip) against torch.argsort(stable=True): sizes at
the edges of its chunks and wavefront steps, both forms, one to eight passes, both label types."""
import pytest
import torch

from peco_amd import clustering, clustering_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tokens", [1, 63, 65, 511, 513, 4097, 12288, 12289, 20481])
@pytest.mark.parametrize("low,high,dtype", [
    (0, 1, torch.int32), (0, 512, torch.int32), (0, 2048, torch.int32), (0, 2049, torch.int64),
    (-5000, 70000, torch.int32), (-2**31, 2**31 - 1, torch.int32), (-2**62, 2**62, torch.int64),
    (2**40, 2**40 + 300, torch.int64)])
def test_label_argsort_matches_torch(tokens, low, high, dtype):
    g = torch.Generator().manual_seed(tokens)
    labels = torch.randint(low, high, (3, tokens), generator=g, dtype=torch.int64).to(dtype)
    labels[1, ::3] = labels[1, 0]  # many equal labels, an entry with a range of its own
    labels[2] = labels[2, 0]
    if tokens > 2 and low < 0:
        labels[0, :2] = torch.tensor([torch.iinfo(dtype).min, torch.iinfo(dtype).max], dtype=dtype)
    got = clustering_cuda.label_argsort(labels.to(DEV))
    assert torch.equal(got.cpu().long(), torch.argsort(labels, dim=-1, stable=True))


def test_gather_by_labels_takes_any_label_tensor():
    g = torch.Generator().manual_seed(1)
    x = torch.randn(1, 2, 300, 64, generator=g).to(DEV)
    labels = torch.randint(0, 9, (2, 300), generator=g)
    want = torch.argsort(labels, dim=-1, stable=True)
    for lab in (labels.int(), labels, labels.to(torch.uint8), labels.float(), labels.int().t().contiguous().t()):
        packed, indices = clustering.gather_clustered_tokens(x, lab.to(DEV))
        assert indices.dtype == torch.int32 and torch.equal(indices.cpu().long(), want)
        assert torch.equal(packed.cpu(), x.cpu().gather(2, want[None, ..., None].expand(-1, -1, -1, 64)))
        assert torch.equal(clustering.restore_sequence_order(packed, indices), x)


def test_gather_by_labels_of_very_long_entries_stays_with_torch(monkeypatch):
    """The argsort's time on labels of any value grows with the length of an entry."""
    calls = []
    monkeypatch.setattr(clustering_cuda, "label_argsort", lambda rows: calls.append(rows.shape))
    for tokens, taken in ((131072, True), (131073, False), (1000000, False)):
        x = torch.zeros(1, 1, tokens, 8, dtype=torch.bfloat16, device=DEV)
        labels = torch.arange(tokens, device=DEV).flip(0) * (2**20 + 1)
        calls.clear()
        indices = clustering._prepare_sequence_indices(x, labels, 2, None)
        assert bool(calls) == taken
        if not taken:
            assert indices.dtype == torch.int32 and torch.equal(indices[0], torch.arange(tokens, device=DEV).flip(0).int())
