"""GPU tests of head dims around 96, up to which the 128-wide forward kernels compute with 96 columns: q/k and value dims
on either side of it, against the oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn, assert_close
from test_gpu_forward import _module, _oracle, ha  # noqa: F401


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,d,dv", [(torch.float16, 72, 96), (torch.bfloat16, 96, 72), (torch.float16, 104, 96),
                                        (torch.bfloat16, 96, 104), (torch.float16, 80, 80)])
def test_head_dims_around_96(ha, monkeypatch, split, causal, dtype, d, dv):
    monkeypatch.setenv("HA_SPLIT", split)
    q, k = (_randn((1, 2, 1280, d), s, dtype) for s in (50, 51))
    v = _randn((1, 2, 1280, dv), 52, dtype)
    m, proj = _module(ha, d, dtype, 53, block_size=256, sample_size=128, min_seq_len=640)
    attn, lse = m(q.cuda(), k.cuda(), v.cuda(), causal=causal, return_lse=True)
    ro, rl = _oracle(q, k, v, proj, m, causal)
    assert_close(attn, ro, "attn", dtype)
    assert_close(lse, rl, "lse")
