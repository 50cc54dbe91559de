"""Gathered attention, 256-query kernel, where the two query tiles of a workgroup see different windows of keys: blocks of an
odd number of tiles and smooth windows, whose second half starts later and whose first half ends earlier; and the plain
instance of the head dims below the built widths."""
import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_ops import _run_hyper, _sorted_inputs, ha  # noqa: F401 (fixture)
from _util import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 96)])
@pytest.mark.parametrize("n,block,sample,smooth", [
    (512, 128, 0, False),    # windows side by side, no samples: nothing in common
    (640, 128, 128, False),  # the last workgroup has one tile
    (1152, 384, 256, False), # a block boundary between the two tiles now and then; a short last block
    (768, 256, 128, True),
    (640, 512, 0, True),     # windows wrap around the sequence
    (256, 512, 128, True),   # a block longer than the sequence
    (1024, 128, 128, True),  # windows of one tile, 64 keys off
    (640, 256, 128, False),  # the plain instance with one tile in the last workgroup
    (128, 512, 0, False),    # and in the only one
])
def test_windows(ha, monkeypatch, dtype, d, n, block, sample, smooth):  # noqa: F811
    monkeypatch.setenv("HA_SPLIT", "0")
    q, k, v, qi, ki = _sorted_inputs(1, 2, n, d, dtype, 60)
    o, lse = _run_hyper(ha, q, k, v, qi, ki, block, sample, None, smooth)
    ro, rl = O.block_sampled_attention(q, k, v, qi, ki, block, sample, None, smooth)
    assert_close(o, ro, "out", dtype)
    assert_close(lse, rl, "lse")


@pytest.mark.parametrize("dtype,d", [(torch.float16, 40), (torch.bfloat16, 96), (torch.float16, 120)])
def test_plain_blocks_of_narrow_heads_resumed(ha, monkeypatch, dtype, d):  # noqa: F811
    monkeypatch.setenv("HA_SPLIT", "0")
    q, k, v, qi, ki = _sorted_inputs(1, 2, 768, d, dtype, 70)
    o0, l0 = O.exact_attention(q, v, v, None, False)
    o0, l0 = o0.to(dtype), l0.float()
    c = lambda t: t.cuda().transpose(1, 2)
    o, lse = ha.hyper_attn_func(c(q), c(k), c(v), c(qi), c(ki), 256, 128, None, False, resume=(c(o0).contiguous(), l0.cuda()))
    ro, rl = O.block_sampled_attention(q, k, v, qi, ki, 256, 128, None, False)
    mo, ml = O.add_self_attentions(o0.double(), l0.double().unsqueeze(-1), ro, rl.unsqueeze(-1))
    assert_close(o.transpose(1, 2), mo, "merged out", dtype)
    assert_close(lse, ml.squeeze(-1), "merged lse")
