"""The standalone Base-Offset quantizer and decoder (quant.hip) at the edges of their row passes, with
batches that do and do not spread over the XCDs and both label types, bit for bit against the torch
arithmetic of the reference (peco/quantization.py:97-150) on the CPU."""
import pytest
import torch

from peco_amd import quantization

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _reference(x, labels, centroids, bits):
    c = centroids.gather(1, labels.long()[..., None].expand(-1, -1, x.shape[2]))
    r = x.float() - c
    low = r.amin(-1, keepdim=True)
    scale = (r.amax(-1, keepdim=True) - low) / (2 ** bits - 1)
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    codes = ((r - low) / scale).round().clamp(0, 2 ** bits - 1)
    return codes.to(torch.uint8), low, scale, (c + (low + scale * codes)).to(x.dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("batch,tokens,clusters,dim,bits,label_dtype", [
    (1, 1, 1, 128, 4, torch.int32), (3, 15, 4, 128, 8, torch.int64), (8, 63, 9, 128, 4, torch.int64),
    (8, 64, 9, 64, 8, torch.int32), (16, 65, 2, 128, 4, torch.int32), (5, 129, 30, 64, 4, torch.int64)])
def test_quantizer_rows_match_torch(dtype, batch, tokens, clusters, dim, bits, label_dtype):
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn(batch, tokens, dim, generator=g).to(dtype)
    centroids = torch.randn(batch, clusters, dim, generator=g)
    labels = torch.randint(clusters, (batch, tokens), generator=g).to(label_dtype)
    x[0, 0] = centroids[0, labels[0, 0].long()].to(dtype)  # a row next to its centre
    codes, low, scale, xhat = _reference(x, labels, centroids, bits)
    args = (x.to(DEV), labels.to(DEV), centroids.to(DEV))
    packed = quantization.quantize_base_offset(*args, bits)
    assert packed.labels.dtype == torch.int64 and torch.equal(packed.labels.cpu(), labels.long())
    assert torch.equal(packed.codes.cpu(), codes)
    assert torch.equal(packed.offset_min.cpu(), low) and torch.equal(packed.scale.cpu(), scale)
    assert torch.equal(packed.dequantize().cpu(), xhat)
    assert torch.equal(quantization.fake_quantize_base_offset(*args, bits).cpu(), xhat)
