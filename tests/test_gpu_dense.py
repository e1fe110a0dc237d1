"""Dense attention of the warm-up branch (processor.dense_attention) on the sparse kernel: lengths at
the edges of its key tiles, row blocks and items, both item sizes, the persistent grid, layouts,
and the calls that stay with SDPA. The reference is float32 softmax attention per segment; bounds
are those of the attention tests (P and the output are rounded to 16 bits) and, per segment, one on the
error relative to the result, which a single key too many or too few would pass (``_check``)."""
import pytest
import torch

from peco_amd import _native, attention_cuda, processor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _reference(q, k, v, valid):
    out = torch.empty(q.shape, device=q.device)
    for a, b in ((0, valid), (valid, q.shape[2])):
        if a < b:
            for h in range(q.shape[1]):  # head by head: small score matrices
                s = q[:, h, a:b].float() @ k[:, h, a:b].float().transpose(1, 2).contiguous() * q.shape[3] ** -0.5
                out[:, h, a:b] = torch.softmax(s, -1) @ v[:, h, a:b].float()
    return out


def _check(out, ref, valid, dtype):
    """Per segment of n keys the 2-norm of the error is at most 2^-7.5 (bf16) or 2^-10.5 (fp16) of the
    result's. Rounding the weights and the output, each to within u = 2^-8 or 2^-11 of itself, costs an
    element two independent errors of at most u / sqrt(3) of the row's size in the mean, 0.82 u together
    (0.58 u measured); the bound is 1.4 u = 5.5e-3 or 6.9e-4. One key more or less moves a row of normal
    values by 1 / sqrt(n) of its size: 1.1e-2 at the longest 8192 keys here. The smallest fp16 subnormal
    is allowed for beside it."""
    err = (out.float() - ref)
    assert err.abs().max().item() <= 2e-2 and err.abs().mean().item() <= 2e-3
    bound = 2.0 ** -7.5 if dtype == torch.bfloat16 else 2.0 ** -10.5
    for part in (slice(0, valid), slice(valid, ref.shape[2])):
        n = ref[:, :, part].numel()
        assert err[:, :, part].norm().item() <= bound * ref[:, :, part].norm().item() + 2.0 ** -25 * n ** 0.5, part


def _inputs(batch, heads, length, dim, dtype):
    g = torch.Generator(device=DEV)
    g.manual_seed(length + heads)
    return [torch.randn(batch, heads, length, dim, generator=g, device=DEV).to(dtype) for _ in range(3)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,heads,length,dim,valid", [
    (1, 1, 1, 128, 1), (1, 2, 63, 64, 0), (1, 2, 64, 128, 64), (2, 3, 65, 128, 64), (1, 3, 129, 64, 1),
    (1, 2, 257, 128, 128), (1, 2, 1000, 128, 937),
    (1, 64, 2309, 64, 2100),    # paired 64-row items, more than run at once
    (1, 64, 4300, 128, 4250),   # 256-row items on 8-wavefront workgroups, on the persistent grid
    (1, 32, 4300, 128, 4113),   # the same without it
    (1, 2, 4097, 128, 4096),    # 128-row items
    (1, 62, 8193, 64, 8192),    # the same on the persistent grid
    (10, 200, 70, 64, 40),      # 64-row items on the persistent grid
])
def test_dense_attention_matches_reference(dtype, batch, heads, length, dim, valid):
    q, k, v = _inputs(batch, heads, length, dim, dtype)
    assert attention_cuda.dense_supported(q, k, v, valid)
    ref = _reference(q, k, v, valid)
    for _ in range(2):  # the second call finds the workspace as the first left it
        _check(processor.dense_attention(q, k, v, valid), ref, valid, dtype)
    # The bound sees one key of the longer segment moved to the other side of the boundary.
    if length > 64 and 0 < valid < length:
        moved = valid - 1 if valid > length - valid else valid + 1
        wrong = _reference(q[:, :2], k[:, :2], v[:, :2], moved)
        edge = min(valid, moved)
        for part in (slice(0, edge), slice(max(valid, moved), length)):
            if part.stop - part.start > 1:
                assert (wrong[:, :, part] - ref[:, :2, part]).norm() > 2.0 ** -7.5 * ref[:, :2, part].norm()


@pytest.mark.parametrize("heads,length,dim,valid", [
    (64, 448, 128, 383), (64, 449, 64, 320), (128, 192, 64, 129), (3, 1025, 128, 1024), (2, 4097, 64, 65)])
def test_dense_attention_short_items(heads, length, dim, valid):
    """Items of 64 rows, of one row and past a whole tile, few and many per head."""
    q, k, v = _inputs(1, heads, length, dim, torch.bfloat16)
    _check(processor.dense_attention(q, k, v, valid), _reference(q, k, v, valid), valid, torch.bfloat16)


def test_dense_attention_keeps_layout_and_sdpa_calls():
    q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in _inputs(1, 4, 200, 64, torch.bfloat16))
    out = processor.dense_attention(q, k, v, 150)
    assert out.stride() == torch.empty_like(q).stride()
    assert (out.float() - _reference(q, k, v, 150)).abs().max().item() <= 2e-2
    # Gradients, other head dimensions and float32 are SDPA's.
    leaf = q.clone().requires_grad_(True)
    processor.dense_attention(leaf, k, v, 150).float().sum().backward()
    assert leaf.grad is not None and torch.isfinite(leaf.grad).all()
    for dim, dtype in ((32, torch.bfloat16), (64, torch.float32)):
        a, b, c = _inputs(1, 2, 90, dim, dtype)
        assert not attention_cuda.dense_supported(a, b, c, 60)
        assert (processor.dense_attention(a, b, c, 60).float() - _reference(a, b, c, 60)).abs().max().item() <= 2e-2


def test_dense_attention_padding_segment_sees_no_video_value():
    """A non-finite value row is seen by its own segment only, also where a key tile is partial."""
    q, k, v = _inputs(1, 2, 300, 128, torch.bfloat16)
    v[0, 0, 0] = float("inf")
    out = processor.dense_attention(q, k, v, 250)
    assert torch.isfinite(out[0, 0, 250:]).all() and torch.isfinite(out[0, 1]).all()
    assert not torch.isfinite(out[0, 0, :250]).any()


@pytest.mark.parametrize("length,dim,valid", [
    (300, 128, 211), (2100, 128, 1975), (4096, 128, 4000), (4097, 128, 4000), (7006, 128, 6881),
    (7006, 128, 6817), (7006, 128, 6693), (3000, 64, 2900),
    (8192, 64, 8100), (8193, 64, 8100)])
def test_dense_attention_of_a_head_is_the_same_in_any_call(length, dim, valid):
    """A head's output does not depend on how many heads share its call: 24 heads together, as batch
    entries and in shards of one to twelve give the same bits (lengths on both sides of the rules for
    items)."""
    q, k, v = _inputs(1, 24, length, dim, torch.bfloat16)
    out = processor.dense_attention(q, k, v, valid)
    assert torch.equal(out, processor.dense_attention(q, k, v, valid))
    assert torch.equal(out, processor.dense_attention(*(t.view(4, 6, length, dim) for t in (q, k, v)), valid).view_as(out))
    for a, b in ((0, 1), (21, 24), (3, 9), (12, 24)):
        part = processor.dense_attention(*(t[:, a:b].contiguous() for t in (q, k, v)), valid)
        assert torch.equal(part, out[:, a:b]), (a, b)
    wide = [torch.cat((t, t, t, t), 1) for t in (q, k, v)]
    assert torch.equal(processor.dense_attention(*wide, valid)[:, 48:72], out)


def test_dense_attention_leaves_misaligned_tensors_to_sdpa():
    """A contiguous view that does not start on 16 bytes is not taken (the kernel loads 16 bytes at a
    time); a strided one is copied first, wherever it starts. The C entry refuses such a pointer."""
    aligned = _inputs(1, 2, 200, 64, torch.bfloat16)
    ref = _reference(*aligned, 150)
    for i in range(3):
        views = list(aligned)
        flat = torch.empty(views[i].numel() + 1, dtype=torch.bfloat16, device=DEV)
        views[i] = flat[1:].view(views[i].shape).copy_(views[i])
        assert views[i].is_contiguous() and not attention_cuda.dense_supported(*views, 150)
        assert (processor.dense_attention(*views, 150).float() - ref).abs().max().item() <= 2e-2
        wide = torch.empty(1, 2, 200, 65, dtype=torch.bfloat16, device=DEV)
        views[i] = wide[..., 1:].copy_(aligned[i])
        assert attention_cuda.dense_supported(*views, 150)
        assert torch.equal(processor.dense_attention(*views, 150), processor.dense_attention(*aligned, 150))
    library = _native.library()
    ints = library.peco_dense_attention_workspace_size(2, 200)
    workspace = torch.empty(ints, dtype=torch.int32, device=DEV)
    out = torch.empty_like(aligned[0])
    pointers = [t.data_ptr() for t in (*aligned, out)]
    for i in range(4):
        shifted = [p + 2 * (j == i) for j, p in enumerate(pointers)]
        assert library.peco_dense_attention(*shifted, 150, _native.ptr(workspace), ints, 2, 200, 64, 1,
                                            _native.current_stream(out.device, out)) != 0


@pytest.mark.parametrize("length,dim", [(300, 64), (300, 128), (4500, 128)])
def test_dense_attention_with_scores_of_any_size(length, dim):
    """Large scores (on both sides of the point where a row's maximum is subtracted first) and keys with
    scores of -inf give what an ordinary softmax gives. Rows whose two best scores differ by less than
    the products' rounding are left out."""
    valid = length - 50
    plain = _inputs(1, 2, length, dim, torch.bfloat16)
    for a, b in ((60.0, 1e3), (3e2, 4e3), (1e5, 1e5), (1e18, 1e18)):
        q, k, v = plain[0] * a, plain[1] * b, plain[2]
        got = processor.dense_attention(q, k, v, valid).float()
        assert torch.isfinite(got).all()
        for lo, hi in ((0, valid), (valid, length)):
            scores = q[:, :, lo:hi].double() @ k[:, :, lo:hi].double().transpose(2, 3).contiguous() * dim ** -0.5
            ref = torch.softmax(scores, -1) @ v[:, :, lo:hi].double()
            best = scores.topk(2, -1).values
            clear = (best[..., 0] - best[..., 1]) > 1e-5 * scores.abs().amax(-1) + 10
            assert clear.float().mean() > 0.5
            assert ((got[:, :, lo:hi] - ref).abs().amax(-1)[clear] <= 2e-2).all()
    for rows in (32, 64, length):  # the first keys; every key
        q, k, v = plain[0], plain[1].clone(), plain[2]
        k[:, :, :rows, 0] = -float("inf")
        got = processor.dense_attention(q, k, v, length).float()
        none = q[..., 0] < 0  # scores of +inf: not a number
        assert (got.isnan().all(-1) == none).all()
        if rows < length:
            ref = torch.softmax(q.float() @ k[:, :, rows:].float().transpose(2, 3).contiguous() * dim ** -0.5, -1) @ \
                v[:, :, rows:].float()
            assert ((got - ref).abs().amax(-1)[~none] <= 2e-2).all()
        else:
            assert (got[~none] == 0).all()  # no weight at all
