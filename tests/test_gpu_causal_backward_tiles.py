"""Backward of exact causal attention, 128 rows per workgroup: one tile per workgroup, longest first, and pairs of tiles
(launches of many workgroups), with odd numbers of tiles and ragged ends, and the second 256 workgroups' reversed order."""
import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_backward import _check, _gpu_grads, _oracle_grads, ha  # noqa: F401 (fixture)
from _util import _randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d,h,hk,n", [
    (torch.bfloat16, 64, 100, 100, 600),   # single tiles from here on: 500 in both passes, the last 244 reversed
    (torch.float16, 64, 130, 130, 270),    # 390 of dq
    (torch.bfloat16, 64, 180, 60, 400),    # 720 of dq; grouped heads
    (torch.float16, 64, 200, 100, 600),    # 1000 of dq, 500 of dk, dv with two query heads each
    (torch.bfloat16, 128, 80, 80, 600),    # 400 of dq
    (torch.float16, 128, 120, 120, 385),   # 480 of dq
    (torch.bfloat16, 64, 48, 48, 600),     # 64 rows and split steps: too few tiles
    (torch.float16, 128, 100, 100, 385),
    (torch.bfloat16, 128, 150, 150, 130),
    (torch.float16, 64, 1160, 1160, 140),  # pairs from here on
    (torch.bfloat16, 64, 600, 600, 300),   # three tiles, the middle one alone
])
def test_causal(ha, dtype, d, h, hk, n):  # noqa: F811
    q, do = (_randn((1, h, n, d), s, dtype) for s in (91, 92))
    k, v = (_randn((1, hk, n, d), s, dtype) for s in (93, 94))
    fn = lambda a, b, c: O.exact_attention(a, *(x.repeat_interleave(h // hk, 1) for x in (b, c)), None, True)  # noqa: E731
    ref = _oracle_grads(fn, q, k, v, do)
    _, _, *got = _gpu_grads(lambda a, b, c: ha.flash_attn_func(a, b, c, None, True), q, k, v, do)
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, want, name, dtype)


@pytest.mark.parametrize("dtype,h,nq,nk", [
    (torch.float16, 248, 300, 200),   # dk, dv in single tiles
    (torch.bfloat16, 600, 800, 500),  # and in pairs
])
def test_more_queries_than_keys(ha, dtype, h, nq, nk):  # noqa: F811
    """Head dim 128, where launches of as many queries as keys are left to the 256-key pass.  Four different heads in turn."""
    q, do = (_randn((1, 4, nq, 128), s, dtype) for s in (95, 96))
    k, v = (_randn((1, 4, nk, 128), s, dtype) for s in (97, 98))
    ref = _oracle_grads(lambda a, b, c: O.exact_attention(a, b, c, None, True), q, k, v, do)
    many = lambda x: x.repeat(1, h // 4, 1, 1)  # noqa: E731
    _, _, *got = _gpu_grads(lambda a, b, c: ha.flash_attn_func(a, b, c, None, True), *(many(x) for x in (q, k, v, do)))
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, many(want), name, dtype)
