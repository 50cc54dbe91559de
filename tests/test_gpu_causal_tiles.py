"""Exact causal attention, 256-query kernel: one query tile per workgroup, longest first, and pairs of tiles (launches of
many workgroups), with odd numbers of tiles and ragged ends, and the second 256 workgroups' reversed order."""
import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_ops import ha  # noqa: F401 (fixture)
from _util import _randn, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d,b,h,hk,n", [
    (torch.bfloat16, 64, 1, 1, 1, 256),    # single tiles from here on: the only one
    (torch.float16, 64, 1, 2, 2, 700),     # three tiles, the last ragged
    (torch.bfloat16, 64, 2, 150, 50, 500), # 600 workgroups: 256, 256 reversed, the rest in order; grouped heads
    (torch.float16, 64, 1, 257, 257, 260), # 514
    (torch.float16, 96, 1, 300, 300, 300),
    (torch.bfloat16, 128, 1, 6, 2, 1030),
    (torch.float16, 64, 1, 930, 930, 300), # pairs from here on: two tiles
    (torch.bfloat16, 64, 1, 460, 460, 600),# three, the middle one alone
    (torch.float16, 128, 2, 520, 260, 270),
])
def test_causal(ha, monkeypatch, dtype, d, b, h, hk, n):  # noqa: F811
    monkeypatch.setenv("HA_SPLIT", "0")
    q = _randn((b, h, n, d), 81, dtype)
    k, v = (_randn((b, hk, n, d), s, dtype) for s in (82, 83))
    o, lse = ha.flash_attn_func(*(x.cuda().transpose(1, 2) for x in (q, k, v)), None, True)
    ro, rl = O.exact_attention(q, *(x.repeat_interleave(h // hk, 1) for x in (k, v)), None, True)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :n], rl, "lse")
