"""GPU tests of which gradients a row that is not finite (padding, say) reaches: those of the rows that attend it or are
attended by it, and no others beyond the 64 rows that are worked on together."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn
from test_gpu_backward import ha  # noqa: F401

BAD = float("nan")


def _leaves(shape, seed, dtype):
    return [_randn(shape, seed + i, dtype).cuda().requires_grad_() for i in range(3)]


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 128)])
@pytest.mark.parametrize("heads,kv_heads", [(2, 1), (1024, 512)])  # steps split over waves, and not
@pytest.mark.parametrize("row", [31, 33, 100, 127, 128, 290, 511])
def test_exact_causal_backward(ha, dtype, d, heads, kv_heads, row):
    """A bad key row reaches no query before its 64 rows, a bad query row no key after its 64 rows."""
    n = 512
    q = _randn((1, n, heads, d), 201, dtype).cuda().requires_grad_()
    k, v = (_randn((1, n, kv_heads, d), s, dtype).cuda().requires_grad_() for s in (202, 203))
    do = _randn((1, n, heads, d), 204, dtype).cuda()
    out, _ = ha.flash_attn_func(q, k, v, None, True)
    want = torch.autograd.grad(out, (q, k, v), do, retain_graph=True)
    first, end = row // 64 * 64, row // 64 * 64 + 64

    bad_do = do.clone()
    bad_do[:, row] = BAD
    saved = q.detach()[:, row].clone()
    q.data[:, row] = BAD
    _, dk, dv = torch.autograd.grad(out, (q, k, v), bad_do, retain_graph=True)
    q.data[:, row] = saved
    for got, ref in ((dk, want[1]), (dv, want[2])):
        assert torch.isnan(got[:, row].float()).all()
        assert torch.equal(got[:, end:], ref[:, end:])

    for x in (k, v):
        x.data[:, row] = BAD
    dq = torch.autograd.grad(out, (q, k, v), do)[0]
    assert torch.isnan(dq[:, row].float()).all()
    assert torch.equal(dq[:, :first], want[0][:, :first])


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 128)])
@pytest.mark.parametrize("row", [5, 200, 300, 511])
def test_backward_of_smooth_blocks(ha, dtype, d, row):
    """Two tiles of 128 to a block: a query tile's window starts 64 keys before it, half a key tile."""
    n, block = 512, 256
    q, k, v = _leaves((1, n, 2, d), 211, dtype)
    do = _randn((1, n, 2, d), 214, dtype).cuda()
    order = torch.arange(n, device="cuda").view(1, n, 1).expand(1, n, 2)
    out, _ = ha.hyper_attn_func(q, k, v, order, order, block, 0, None, True)
    want = torch.autograd.grad(out, (q, k, v), do, retain_graph=True)
    bad_do = do.clone()
    bad_do[:, row] = BAD
    q.data[:, row] = BAD
    _, dk, dv = torch.autograd.grad(out, (q, k, v), bad_do)
    start = (row // 128 * 128 - 64) % n
    window = torch.zeros(n, dtype=torch.bool, device="cuda")
    window[(start + torch.arange(block, device="cuda")) % n] = True
    for got, ref in ((dk, want[1]), (dv, want[2])):
        assert torch.isnan(got[:, window].float()).all()
        assert torch.equal(got[:, ~window], ref[:, ~window])
