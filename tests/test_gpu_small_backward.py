"""GPU tests of the backward of exact attention at the edges of its tiles: few heads, where a launch is too small to fill
the chip and the steps of the streamed tiles are split over waves (64 stationary rows per workgroup), and the same or
similar lengths with many heads, where it is not.  Against gradients of the oracle, on the first, a middle and the last
pair of query heads."""
import pytest
import torch

from oracle import hyper_oracle as O

pytestmark = pytest.mark.gpu

from _util import _randn
from test_gpu_backward import _check, _gpu_grads, _oracle_grads, ha  # noqa: F401


# No case has a single key for many queries: its soft-max is constant, so dq and dk are zero and what comes out is D's
# rounding, |dP - D| <= 2^-11 sum |dO O| (fp16: about 3e-3 per query at d = 64), which a relative bound cannot hold.
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("heads,causal,nq,nk", [
    (4, True, 1, 1), (4, True, 63, 63), (4, True, 65, 65), (4, True, 129, 129), (4, True, 321, 321), (4, True, 97, 200),
    (4, False, 1, 33), (4, False, 64, 31), (4, False, 65, 129), (4, False, 257, 700), (4, False, 700, 2),
    (1024, True, 449, 449), (1024, True, 511, 511), (1024, False, 192, 128), (1024, False, 257, 700)])
def test_exact_backward_at_tile_edges(ha, dtype, d, heads, causal, nq, nk):
    q, do = (_randn((1, heads, nq, d), s, dtype) for s in (31, 32))
    k, v = (_randn((1, heads // 2, nk, d), s, dtype) for s in (33, 34))
    grads = _gpu_grads(lambda a, b, c: ha.flash_attn_func(a, b, c, None, causal), q, k, v, do)[2:]
    for kv in sorted({0, heads // 4, heads // 2 - 1}):
        h = slice(2 * kv, 2 * kv + 2)
        expand = lambda x: x.expand(1, 2, nk, d)
        ref = _oracle_grads(lambda a, b, c: O.exact_attention(a, expand(b), expand(c), None, causal),
                            q[:, h], k[:, kv:kv + 1], v[:, kv:kv + 1], do[:, h])
        got = (grads[0][:, h], grads[1][:, kv:kv + 1], grads[2][:, kv:kv + 1])
        for g, r, name in zip(got, ref, ("dq", "dk", "dv")):
            _check(g, r, f"{name} of key head {kv}", dtype)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("heads,n", [(2, 65), (1024, 512)])
def test_fp16_dk_of_large_gradients(ha, d, heads, n):
    """P (dP - D) of the first rows is past 65504 and scale times it is not: dK comes from the latter."""
    sign = torch.where(_randn((1, heads, n, 1), 41, torch.float32) > 0, 1., -1.)
    v = (24 * sign).expand(1, heads, n, d).half()
    do = torch.full((1, heads, n, d), 160.).half()
    q, k = ((_randn((1, heads, n, d), s, torch.float32) * a).half() for s, a in ((42, 0.05), (43, 0.01)))
    h = slice(0, 2)
    ref = _oracle_grads(lambda a, b, c: O.exact_attention(a, b, c, None, True), q[:, h], k[:, h], v[:, h], do[:, h])
    dp = torch.einsum("bhid,bhjd->bhij", do[:, h].double(), v[:, h].double())
    p = torch.softmax((torch.einsum("bhid,bhjd->bhij", q[:, h].double(), k[:, h].double()) * d ** -0.5)
                      .masked_fill(torch.ones(n, n).triu(1).bool(), float("-inf")), dim=-1)
    ds = (p * (dp - (p * dp).sum(-1, keepdim=True))).abs().max()
    assert 65504 < ds and ds * d ** -0.5 < 65504
    _, dk, dv = _gpu_grads(lambda a, b, c: ha.flash_attn_func(a, b, c, None, True), q, k, v, do)[2:]
    _check(dk[:, h], ref[1], "dk", torch.float16)
    _check(dv[:, h], ref[2], "dv", torch.float16)
