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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("data", ["normal", "clusters"])
@pytest.mark.parametrize("d,h,n", [(64, 100, 600), (64, 48, 2048), (128, 60, 700)])
def test_single_tiles_are_as_close_as_split_keys(ha, monkeypatch, dtype, data, d, h, n):  # noqa: F811
    """Launches where single tiles have taken the place of the split kernel: no further from float64 than it is.  The errors are
    sums over some 10^6 roundings, so the ratio repeats to 0.1 % over seeds; with exponents that do not follow the row
    maxima it is 1.01 to 1.024."""
    g = torch.Generator(device="cuda").manual_seed(91)
    q, k, v = (torch.randn((1, n, h, d), generator=g, device="cuda").to(dtype) for _ in range(3))
    if data == "clusters":
        centroids = 4 * torch.nn.functional.normalize(torch.randn((64, d), generator=g, device="cuda"), dim=-1).to(dtype)
        for x in (q, k):
            x.mul_(0.5).add_(centroids[torch.randint(0, 64, x.shape[:3], generator=g, device="cuda")])
    past = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    want = torch.empty((1, n, h, d), dtype=torch.float64, device="cuda")
    for i in range(h):
        a, b, c = (x[0, :, i].double().contiguous() for x in (q, k, v))
        want[0, :, i] = (a @ b.T.contiguous() * d ** -0.5).masked_fill(past, float("-inf")).softmax(-1) @ c
    out, _ = ha.flash_attn_func(q, k, v, None, True)
    monkeypatch.setenv("HA_SPLIT", "1")
    split, _ = ha.flash_attn_func(q, k, v, None, True)
    assert not torch.equal(out, split), "the launch takes the split kernel: nothing is compared"
    err, split_err = (((x.double() - want).norm() / want.norm()).item() for x in (out, split))
    assert err <= 1.003 * split_err, f"{err:.4e}, split {split_err:.4e}"
