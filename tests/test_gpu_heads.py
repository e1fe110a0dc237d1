"""The processor prologue's placing kernel (heads.hip) against the torch expression it stands for,
bit for bit, and the processor call with it against the call that takes the torch path."""
import pytest
import torch

from peco_amd import clustering_cuda, processor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tables(rows, dim, g):
    theta = torch.rand(rows, dim // 2, generator=g) * 6.3
    return tuple(t.repeat_interleave(2, -1).to(DEV).contiguous() for t in (theta.cos(), theta.sin()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch,heads,rows,first,length", [
    (1, 1, 1, 0, 1), (1, 7, 15, 3, 20), (2, 8, 16, 0, 16), (1, 9, 17, 5, 40), (1, 24, 333, 0, 400), (3, 2, 33, 7, 40)])
def test_place_heads_matches_torch(dtype, dim, batch, heads, rows, first, length):
    g = torch.Generator().manual_seed(rows * heads + dim)
    x = torch.randn(batch, rows, heads, dim, generator=g).to(dtype).to(DEV)
    x[0, 0, 0, :2] = torch.tensor([float("inf"), -0.0], dtype=dtype)
    wide = torch.zeros(batch, rows, heads, dim + 8, dtype=dtype, device=DEV)  # rows with a gap between heads
    wide[..., :dim] = x
    tables = _tables(rows, dim, g)
    for part in (x.transpose(1, 2), x.transpose(1, 2).contiguous(), wide[..., :dim].transpose(1, 2)):
        for rotary in (None, tables):
            out = torch.full((batch, heads, length, dim), 7.0, dtype=dtype, device=DEV)
            ref = out.clone()
            clustering_cuda.place_heads(part, out, first, rotary)
            ref[:, :, first:first + rows] = part if rotary is None else processor._apply_rotary_emb(part, rotary)
            assert torch.equal(torch.isnan(out), torch.isnan(ref))
            assert torch.equal(out.nan_to_num(3.0), ref.nan_to_num(3.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch,heads,rows,first,length", [
    (1, 1, 1, 0, 1), (1, 7, 15, 3, 20), (2, 8, 16, 0, 16), (1, 9, 17, 5, 40), (1, 24, 333, 0, 400)])
def test_place_heads_rms_norm(dtype, dim, batch, heads, rows, first, length):
    """Bound: the fp32 sum of squares (at most 9 roundings on the way of a term), eps, the inverse root
    (one ulp) and two products are within 20 * 2^-24 of the real value, then one rounding to the dtype
    (2^-8 or 2^-11, and half the smallest fp16 subnormal)."""
    g = torch.Generator().manual_seed(rows * heads + dim)
    x = (torch.randn(batch, rows, heads, dim, generator=g) * 3.0).to(dtype).to(DEV)
    x[0, 0, 0] = 0.0
    weight = (1.0 + torch.rand(dim, generator=g)).to(dtype).to(DEV)
    tables = _tables(rows, dim, g)
    for part in (x.transpose(1, 2), x.transpose(1, 2).contiguous()):
        for w in (weight, None):
            out = torch.full((batch, heads, length, dim), 7.0, dtype=dtype, device=DEV)
            clustering_cuda.place_heads(part, out, first, None, (w, 1e-6))
            wide = part.double()
            ref = wide / (wide.square().mean(-1, keepdim=True) + 1e-6).sqrt() * (1.0 if w is None else w.double())
            placed = out[:, :, first:first + rows]
            unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
            assert ((placed.double() - ref).abs() <= (unit + 20 * 2.0 ** -24) * 1.01 * ref.abs() + 2.0 ** -25).all()
            module = torch.nn.functional.rms_norm(part.transpose(1, 2), (dim,), w, 1e-6).transpose(1, 2)
            assert torch.equal(placed, module)
            assert (out[:, :, :first] == 7.0).all() and (out[:, :, first + rows:] == 7.0).all()
            turned = torch.empty_like(out)
            clustering_cuda.place_heads(part, turned, first, tables, (w, 1e-6))
            assert torch.equal(turned[:, :, first:first + rows], processor._apply_rotary_emb(placed, tables))


class _Block(torch.nn.Module):
    def __init__(self, heads, dim, double):
        super().__init__()
        width = heads * dim
        self.heads = heads
        linear = lambda: torch.nn.Linear(width, width)  # noqa: E731
        self.to_q, self.to_k, self.to_v = linear(), linear(), linear()
        self.norm_q, self.norm_k = torch.nn.RMSNorm(dim, eps=1e-6), torch.nn.RMSNorm(dim, eps=1e-6)
        self.add_q_proj = None
        if double:
            self.add_q_proj, self.add_k_proj, self.add_v_proj = linear(), linear(), linear()
            self.norm_added_q, self.norm_added_k = torch.nn.LayerNorm(dim), None


@pytest.mark.parametrize("double", [False, True])
@pytest.mark.parametrize("text", [0, 40])
def test_call_matches_the_torch_prologue(double, text, monkeypatch):
    heads, dim, video = 3, 64, 500
    torch.manual_seed(5)
    block = _Block(heads, dim, double).to(DEV, torch.bfloat16)
    g = torch.Generator().manual_seed(9)
    hidden = torch.randn(1, video, heads * dim, generator=g).to(DEV, torch.bfloat16)
    enc = torch.randn(1, text, heads * dim, generator=g).to(DEV, torch.bfloat16) if text else None
    freqs = _tables(video, dim, g)
    layer = processor.PecoAttention(0, processor.PecoConfig(), processor.InferenceContext(5, text, text))
    layer.attention = lambda q, k, v: torch.cat((q, k, v), -1)
    got = layer(block, hidden, enc, image_rotary_emb=freqs)
    # A rotary function of the caller's own, and norms with a hook, take the torch operations.
    monkeypatch.setattr(processor, "_rotary_function", lambda: lambda x, f: processor._apply_rotary_emb(x, f))
    monkeypatch.setattr(processor, "_placeable", lambda part, buffer: False)
    for norm in (block.norm_q, block.norm_k):
        norm.register_forward_hook(lambda module, args, out: None)
    ref = layer(block, hidden, enc, image_rotary_emb=freqs)
    assert torch.equal(got[0], ref[0])
    assert (got[1] is None and ref[1] is None) if not text else torch.equal(got[1], ref[1])


@pytest.mark.parametrize("eps,size", [(0.0, 1e-20), (0.0, 3e-19), (1e-40, 1e-20), (2.0 ** -126, 1e-20), (1e-6, 1.0)])
def test_call_with_a_norm_of_tiny_rows(eps, size, monkeypatch):
    """Rows whose mean square is subnormal come out as the block's norm gives them, whatever its eps."""
    monkeypatch.setattr(processor, "_NORM_ELEMENTS", 0)  # the placing launch for any size
    heads, dim, video = 3, 64, 40
    torch.manual_seed(6)
    block = _Block(heads, dim, False).to(DEV, torch.bfloat16)
    for name in ("q", "k"):
        norm, proj = getattr(block, "norm_" + name), getattr(block, "to_" + name)
        norm.eps = eps
        proj.weight.data *= size
        proj.bias.data *= size
    hidden = torch.randn(1, video, heads * dim, device=DEV).bfloat16()
    layer = processor.PecoAttention(0, processor.PecoConfig(), processor.InferenceContext(5, 0, 0))
    layer.attention = lambda q, k, v: torch.cat((q, k), -1)
    got = layer(block, hidden, None)[0].unflatten(2, (heads, -1))
    for at, name in ((0, "q"), (dim, "k")):
        rows = getattr(block, "to_" + name)(hidden).unflatten(2, (heads, -1))
        want = getattr(block, "norm_" + name)(rows)
        assert torch.isfinite(want).all() and torch.equal(got[..., at:at + dim], want)


@pytest.mark.parametrize("rotate", [False, True])
@pytest.mark.parametrize("norm", [None, torch.nn.RMSNorm, torch.nn.LayerNorm])
def test_call_is_the_same_on_both_sides_of_the_size_rules(norm, rotate, monkeypatch):
    """A projection placed by torch operations and by the placing launch: the same bits."""
    heads, dim, video, text = 5, 128, 67, 9
    torch.manual_seed(8)
    block = _Block(heads, dim, False).to(DEV, torch.bfloat16)
    block.norm_q, block.norm_k = (norm(dim, eps=1e-6).to(DEV, torch.bfloat16) if norm else None for _ in range(2))
    g = torch.Generator().manual_seed(3)
    hidden, enc = (torch.randn(2, rows, heads * dim, generator=g).to(DEV, torch.bfloat16) for rows in (video, text))
    freqs = _tables(video, dim, g) if rotate else None
    layer = processor.PecoAttention(0, processor.PecoConfig(), processor.InferenceContext(5, text, text))
    layer.attention = lambda q, k, v: torch.cat((q, k, v), -1)
    placed, outs = [], []
    launch = clustering_cuda.place_heads
    monkeypatch.setattr(clustering_cuda, "place_heads", lambda *a: (placed.append(a), launch(*a)))
    for limit in (0, 1 << 40):
        monkeypatch.setattr(processor, "_COPY_ELEMENTS", limit)
        monkeypatch.setattr(processor, "_NORM_ELEMENTS", limit)
        placed.clear()
        outs.append(layer(block, hidden, enc, image_rotary_emb=freqs))
        assert len(placed) == (6 if limit == 0 else 2 * rotate)
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
