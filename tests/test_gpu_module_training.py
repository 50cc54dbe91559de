"""GPU tests of the module under autograd as a training program calls it: explicit sample lists, tensors that are views
of a layer's projections.  Gradients against torch autograd on the oracle."""
import pytest
import torch

from oracle import hyper_oracle as O

pytestmark = pytest.mark.gpu

from _util import _gen, _randn
from test_gpu_backward import _check, _oracle_grads, ha  # noqa: F401

BLOCK = SAMPLE = 128


def _module(ha, d, dtype, min_seq_len, **kw):
    m = ha.HyperAttention(input_dim=d, block_size=BLOCK, sample_size=SAMPLE, min_seq_len=min_seq_len, rng=_gen(95), **kw)
    return m.to(device="cuda", dtype=dtype)


def _reference(m, q, k, v, do, causal, sampled=None):
    proj = m.lsh.proj_dir[0, 0].cpu()
    expand = lambda x: x.repeat_interleave(q.shape[1] // x.shape[1], dim=1)
    return _oracle_grads(lambda a, b, c: O.hyper_forward(a, expand(b), expand(c), proj, causal=causal, block_size=BLOCK,
                                                         sample_size=SAMPLE, min_seq_len=m.min_seq_len, sampled_idx=sampled,
                                                         detach_lse=True), q, k, v, do)


# ------------------------------------------------------------------------------- explicit sample lists
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("idx_dtype", [torch.int32, torch.int64])
def test_training_with_an_explicit_sample_list(ha, causal, idx_dtype):
    """The gradients are those of the listed rows.  A list that is redrawn in place between forward and backward is an
    error where the backward would read it (int32 on the GPU: taken as it is) and without effect where it was copied."""
    dtype, h, n, d = torch.float16, 2, 1024, 64
    q, k, v, do = (_randn((1, h, n, d), 60 + i, dtype) for i in range(4))
    sampled = torch.randperm(256, generator=_gen(64))[:SAMPLE]
    m = _module(ha, d, dtype, 256, sampled_idx=sampled.to(device="cuda", dtype=idx_dtype))
    ref = _reference(m, q, k, v, do, causal, sampled)
    leaves = [x.cuda().requires_grad_() for x in (q, k, v)]
    out = m(*leaves, causal=causal)
    for got, want, name in zip(torch.autograd.grad(out, leaves, do.cuda(), retain_graph=True), ref, ("dq", "dk", "dv")):
        _check(got, want, name, dtype)
    m.sampled_idx.add_(1)
    if idx_dtype == torch.int32:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(out, leaves, do.cuda())
    else:
        for got, want, name in zip(torch.autograd.grad(out, leaves, do.cuda()), ref, ("dq", "dk", "dv")):
            _check(got, want, name, dtype)


@pytest.mark.parametrize("per_batch", [False, True])
def test_training_without_mask_takes_a_sample_list_per_key_head(ha, per_batch):
    dtype, b, h, hk, n, d = torch.float16, 2, 4, 2, 512, 64
    q, do = (_randn((b, h, n, d), 65 + i, dtype) for i in range(2))
    k, v = (_randn((b, hk, n, d), 67 + i, dtype) for i in range(2))
    lists = torch.stack([torch.randperm(n, generator=_gen(i))[:SAMPLE] for i in range(b * hk)]).view(b, hk, SAMPLE)
    if not per_batch:
        lists = lists[0]
    m = _module(ha, d, dtype, 256, sampled_idx=lists.cuda())
    of_q_heads = lists.expand(b, hk, SAMPLE).repeat_interleave(h // hk, dim=1)
    leaves = [x.cuda().requires_grad_() for x in (q, k, v)]
    grads = torch.autograd.grad(m(*leaves, causal=False), leaves, do.cuda())
    for got, want, name in zip(grads, _reference(m, q, k, v, do, False, of_q_heads), ("dq", "dk", "dv")):
        _check(got, want, name, dtype)
    with pytest.raises(AssertionError):  # the recursion's calls share one list, and so does the one-call forward
        m(*leaves, causal=True)
    with torch.no_grad(), pytest.raises(AssertionError):
        m(*leaves, causal=False)


def test_saved_tensor_hooks_see_the_sample_list(ha):
    dtype, n, d = torch.float16, 512, 64
    q, k, v, do = (_randn((1, 1, n, d), 70 + i, dtype).cuda() for i in range(4))
    m = _module(ha, d, dtype, 256, sampled_idx=torch.arange(SAMPLE, dtype=torch.int32, device="cuda"))
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    want = torch.autograd.grad(m(*leaves, causal=False), leaves, do)
    with torch.autograd.graph.save_on_cpu():
        out = m(*leaves, causal=False)
    for a, b in zip(torch.autograd.grad(out, leaves, do), want):
        _check(a, b, "gradient", dtype)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(x) or x, lambda x: x):
        m(*leaves, causal=False)
    assert any(x.data_ptr() == m.sampled_idx.data_ptr() for x in packed)


def test_the_operator_refuses_a_sample_list_changed_before_its_backward(ha):
    dtype, n, d = torch.float16, 512, 64
    q, k, v, do = (_randn((1, n, 1, d), 80 + i, dtype).cuda() for i in range(4))
    order = torch.randperm(n, generator=_gen(84)).view(1, n, 1).cuda()
    sampled = torch.arange(SAMPLE, device="cuda")
    leaf = q.requires_grad_()
    out, _ = ha.hyper_attn_func(leaf, k, v, order, order, BLOCK, SAMPLE, sampled_idx=sampled)
    sampled.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, leaf, do)


def test_training_without_mask_takes_a_negative_min_seq_len(ha):
    dtype, n, d = torch.float16, 256, 64
    q, k, v, do = (_randn((1, 1, n, d), 90 + i, dtype) for i in range(4))
    m = _module(ha, d, dtype, -1)
    leaves = [x.cuda().requires_grad_() for x in (q, k, v)]
    grads = torch.autograd.grad(m(*leaves, causal=False), leaves, do.cuda())
    for got, want, name in zip(grads, _reference(m, q, k, v, do, False), ("dq", "dk", "dv")):
        _check(got, want, name, dtype)
    with torch.no_grad(), pytest.raises(AssertionError, match="min_seq_len"):
        m(*leaves, causal=False)


# ------------------------------------------------------------------------------- layouts
LAYOUTS = {
    # what a layer has in memory for b batches, h query heads, hk key/value heads, and the views it calls the module with
    "transposed": (lambda b, h, hk, n, d: [(b, n, h, d), (b, n, hk, d), (b, n, hk, d)],
                   lambda t, h, hk: [x.transpose(1, 2) for x in t]),
    "packed": (lambda b, h, hk, n, d: [(b, n, h + 2 * hk, d)],
               lambda t, h, hk: [x.transpose(1, 2) for x in t[0].split((h, hk, hk), dim=2)]),
    "rows_first": (lambda b, h, hk, n, d: [(n, b, h, d), (n, b, hk, d), (n, b, hk, d)],
                   lambda t, h, hk: [x.permute(1, 2, 0, 3) for x in t]),
    "expanded": (lambda b, h, hk, n, d: [(b, h, n, d), (b, 1, n, d), (b, 1, n, d)],
                 lambda t, h, hk: [t[0]] + [x.expand(-1, h, -1, -1) for x in t[1:]]),
}


def _layouts(layout, b, h, hk, n, d, dtype):
    shapes, views = LAYOUTS[layout]
    leaves = [_randn(s, 110 + i, dtype).cuda().requires_grad_() for i, s in enumerate(shapes(b, h, hk, n, d))]
    return leaves, views(leaves, h, hk)


@pytest.mark.parametrize("layout", ["transposed", "packed", "rows_first", "expanded"])
@pytest.mark.parametrize("dtype,d,causal,n", [(torch.float16, 64, True, 511), (torch.bfloat16, 128, True, 512),
                                              (torch.float16, 64, False, 512), (torch.bfloat16, 96, True, 512),
                                              (torch.float16, 64, True, 200)])
@pytest.mark.parametrize("gradient", ["rows", "heads", "broadcast"])
def test_training_on_views(ha, layout, dtype, d, causal, n, gradient):
    """Inputs and output gradients are read where they lie; the gradients are those of the same values laid out plainly."""
    b, h, hk = 2, 4, 2
    m = _module(ha, d, dtype, 256)
    leaves, call = _layouts(layout, b, h, hk, n, d, dtype)
    out = m(*call, causal=causal)
    do = _randn((b, h, n, d), 120, dtype).cuda()
    if gradient == "heads":  # (batch, rows, heads, dim) in memory: what the layer's output projection hands back
        do = do.transpose(1, 2).contiguous().transpose(1, 2)
    elif gradient == "broadcast":
        do = do[:, :, :1, :1].expand(b, h, n, d)
    grads = torch.autograd.grad(out, leaves, do)
    plain = [x.detach().contiguous().requires_grad_() for x in call]
    out_plain = m(*plain, causal=causal)
    assert torch.equal(out.detach(), out_plain.detach())
    want = torch.autograd.grad(out_plain, plain, do.contiguous())
    # back through the views alone
    want = torch.autograd.grad(LAYOUTS[layout][1](leaves, h, hk), leaves, want)
    for got, ref in zip(grads, want):
        # (the sampled keys' sums are added up by atomics, in an order that can differ between runs)
        assert ((got.double() - ref.double()).norm() / ref.double().norm()).item() < (2e-3 if dtype == torch.bfloat16 else 5e-4)


@pytest.mark.parametrize("causal", [True, False])
def test_training_on_packed_rows_against_the_oracle(ha, causal):
    dtype, b, h, hk, n, d = torch.float16, 1, 2, 1, 512, 64
    m = _module(ha, d, dtype, 256)
    (leaf,), call = _layouts("packed", b, h, hk, n, d, dtype)
    do = _randn((b, n, h, d), 121, dtype).transpose(1, 2)
    got = torch.autograd.grad(m(*call, causal=causal), leaf, do.cuda())[0].split((h, hk, hk), dim=2)
    ref = _reference(m, *(x.detach().cpu() for x in call), do, causal)
    for g, r, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g.transpose(1, 2), r, name, dtype)


@pytest.mark.parametrize("wide", ["query", "gradient"])
def test_training_copies_rows_that_lie_too_far_apart_to_be_addressed(ha, wide):
    """Rows 16 MiB apart, 4 GiB in all: past the kernels' limits, so the module works on a copy."""
    dtype, n, d = torch.float16, 256, 64
    q, k, v, do = (_randn((1, 1, n, d), 100 + i, dtype) for i in range(4))
    far = torch.empty((1, 1, n, 1 << 23), dtype=dtype, device="cuda")[..., :d]
    m = _module(ha, d, dtype, 128)
    leaves = [x.cuda().requires_grad_() for x in (q, k, v)]
    if wide == "query":
        leaves[0] = far.copy_(q.cuda()).requires_grad_()
        out, dout = m(*leaves, causal=True), do.cuda()
    else:
        out, dout = m(*leaves, causal=True), far.copy_(do.cuda())
    for got, want, name in zip(torch.autograd.grad(out, leaves, dout), _reference(m, q, k, v, do, True), ("dq", "dk", "dv")):
        _check(got, want, name, dtype)
