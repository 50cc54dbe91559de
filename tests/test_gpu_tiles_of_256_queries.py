"""Exact attention at head dims above 64 in workgroups of 8 waves, 256 queries: launches that fill the chip's last round with them, at
ragged ends, grouped heads and head dims below the built ones."""
import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_ops import ha  # noqa: F401 (fixture)
from _util import _randn, assert_close, forward_kernels

pytestmark = pytest.mark.gpu


def _check(ha, dtype, d, h, hk, n, causal, form):  # noqa: F811
    q = _randn((1, h, n, d), 74, dtype)
    k, v = (_randn((1, hk, n, d), s, dtype) for s in (75, 76))
    on_gpu = [x.cuda().transpose(1, 2) for x in (q, k, v)]
    call = lambda: ha.flash_attn_func(*on_gpu, None, causal)  # noqa: E731
    assert forward_kernels(call) == [form]
    o, lse = call()
    ro, rl = O.exact_attention(q, *(x.repeat_interleave(h // hk, 1) for x in (k, v)), None, causal)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :n], rl, "lse")


@pytest.mark.parametrize("dtype,d,h,hk,n,form", [
    (torch.bfloat16, 128, 100, 50, 300, "256"),    # the last tile has 44 rows
    (torch.float16, 128, 64, 64, 513, "256"),      # one row
    (torch.bfloat16, 96, 90, 30, 512, "256"),      # whole tiles
    (torch.float16, 72, 256, 64, 129, "256"),      # one tile per sequence, one per CU
    (torch.bfloat16, 104, 128, 128, 387, "256"),
    (torch.float16, 80, 170, 170, 768, "256"),     # two rounds
    (torch.bfloat16, 80, 402, 402, 130, "256"),
    (torch.bfloat16, 128, 85, 85, 300, "128"),     # too few workgroups of 128 for two on every other CU
    (torch.float16, 128, 129, 43, 257, "128"),     # one more of 256 than CUs
    (torch.bfloat16, 128, 200, 200, 512, "128"),   # two rounds of short rows
])
def test_without_mask(ha, dtype, d, h, hk, n, form):  # noqa: F811
    _check(ha, dtype, d, h, hk, n, False, form)


# (heads not a multiple of 8: an instance that follows in the first tile, one tile per workgroup, longest first)
@pytest.mark.parametrize("dtype,d,h,hk,n,form", [
    (torch.bfloat16, 128, 250, 125, 129, "256 follow"),   # one tile per sequence
    (torch.float16, 96, 236, 236, 192, "256 follow"),
    (torch.bfloat16, 80, 110, 110, 385, "256 follow"),    # two, the last of 129 rows
    (torch.float16, 128, 129, 43, 768, "256 follow"),    # whole tiles, more workgroups than CUs
    (torch.bfloat16, 104, 129, 129, 767, "256 follow"),    # a last row less
    (torch.bfloat16, 128, 102, 102, 1000, "256 follow"),
    (torch.float16, 128, 57, 19, 1700, "256 follow"),     # 14 tiles of 128 in 7 of 256
    (torch.bfloat16, 128, 124, 124, 768, "128 follow"),
    (torch.float16, 96, 121, 121, 768, "128 follow"),
    (torch.bfloat16, 128, 200, 200, 129, "128 follow"),   # less than four of five CUs
])
def test_causal(ha, dtype, d, h, hk, n, form):  # noqa: F811
    _check(ha, dtype, d, h, hk, n, True, form)
