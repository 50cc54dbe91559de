"""Training at head dims that the backward is not built for: the forward runs on the rows as they are, the backward in padded
copies.  Gradients against torch autograd on the oracle, and the copies' own kernel against torch."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn
from test_gpu_backward import _check, ha  # noqa: F401
from test_gpu_module_training import _module, _reference


@pytest.mark.parametrize("dtype,d,h,hk,n,causal,layout", [
    (torch.bfloat16, 96, 2, 2, 1024, True, "bhnd"),    # hashed level, leaves of 512
    (torch.float16, 80, 4, 2, 1023, True, "bnhd"),     # an appended row, grouped heads, views
    (torch.float16, 96, 2, 1, 640, False, "bnhd"),     # hashed, without mask
    (torch.bfloat16, 72, 2, 2, 300, True, "bhnd"),     # one exact call
    (torch.float16, 120, 2, 2, 129, False, "bhnd"),
    (torch.float16, 40, 2, 2, 640, True, "bhnd"),      # padded to 64
    (torch.bfloat16, 8, 2, 2, 512, False, "bnhd"),
])
def test_gradients(ha, dtype, d, h, hk, n, causal, layout):  # noqa: F811
    q, do = (_randn((1, h, n, d), 80 + i, dtype) for i in range(2))
    k, v = (_randn((1, hk, n, d), 82 + i, dtype) for i in range(2))
    m = _module(ha, d, dtype, 512)
    on_gpu = lambda x: x.cuda() if layout == "bhnd" else x.transpose(1, 2).contiguous().cuda().transpose(1, 2)
    leaves = [on_gpu(x).requires_grad_() for x in (q, k, v)]
    grads = torch.autograd.grad(m(*leaves, causal=causal), leaves, on_gpu(do))
    for got, want, leaf, name in zip(grads, _reference(m, q, k, v, do, causal), leaves, ("dq", "dk", "dv")):
        assert got.shape == leaf.shape
        _check(got, want, name, dtype)


def test_a_broadcast_gradient_and_large_values_beside_the_padding(ha):  # noqa: F811
    """The gradient of a sum is one expanded number; large outputs meet zeros of the padding only."""
    dtype, d, n = torch.bfloat16, 96, 512
    q, k, v = (_randn((1, 2, n, d), 90 + i, dtype).cuda() for i in range(3))
    v = v * 1e30
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    m = _module(ha, d, dtype, 256)
    (m(*leaves, causal=True).sum() * 1e-30).backward()
    ref = _reference(m, q.cpu(), k.cpu(), v.cpu(), torch.full((1, 2, n, d), 1e-30, dtype=dtype), True)
    assert all(torch.isfinite(x.grad.float()).all() for x in leaves)
    _check(leaves[2].grad * 1e30, ref[2] * 1e30, "dv", dtype)


@pytest.mark.parametrize("src_d,dst_d,n,seqs", [(96, 128, 1, 1), (80, 128, 1000, 3), (128, 80, 257, 2), (8, 64, 64, 5), (64, 64, 100, 70000)])
def test_copy_rows(src_d, dst_d, n, seqs):
    from hyperattention_amd import _lib
    if seqs > 1000:
        n = 2
    src = torch.randn((1, n, seqs, src_d), device="cuda").bfloat16().transpose(1, 2)
    dst = torch.full((1, seqs, n, dst_d), 7., device="cuda").bfloat16()
    guard = torch.full_like(dst, 7.)
    row = lambda a, b: _lib.RowCopy(a.data_ptr(), b.data_ptr(), *a.shape, b.shape[-1], *a.stride()[:3], *b.stride()[:3])
    jobs = (_lib.RowCopy * 2)(row(src, dst), row(src[:, :1], guard[:, :1]))
    assert _lib.lib().ha_copy_rows(jobs, 2, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    want = torch.nn.functional.pad(src, (0, dst_d - src_d)) if dst_d > src_d else src[..., :dst_d]
    assert torch.equal(dst, want)
    assert torch.equal(guard[:, :1], want[:, :1]) and bool((guard[:, 1:] == 7.).all())
    bad = (_lib.RowCopy * 1)(row(src, dst))
    bad[0].src_d = 12
    assert _lib.lib().ha_copy_rows(bad, 1, None) != 0
