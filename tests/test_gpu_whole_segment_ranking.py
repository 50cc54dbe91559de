"""Bucket orders of the one segment of the one hashed level ranked as a whole, at the edges of its lengths and of the number of sequences."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn


@pytest.mark.parametrize("b,h,hk,n,msl,causal", [
    (1, 2, 1, 4224, 1, False), (1, 2, 2, 8192, 1, False), (2, 3, 1, 8320, 1, False), (1, 1, 1, 12288, 1, False),
    (1, 1, 1, 12416, 1, False),                                   # units and their placement
    (1, 2, 2, 2 * 4224, 4200, True), (1, 1, 1, 2 * 12288 - 1, 12000, True), (1, 2, 1, 2 * 12416, 12300, True),
    (2, 64, 64, 4352, 1, False), (2, 65, 65, 4352, 1, False),     # 256 sequences, and more
])
@pytest.mark.parametrize("skewed", [False, True])
def test_whole_segments(b, h, hk, n, msl, causal, skewed):
    from hyperattention_amd import ops
    q, k = (_randn((b, x, n, 64), s, torch.bfloat16).cuda() for x, s in ((h, 310), (hk, 311)))
    if skewed:  # two of three rows in one bucket
        q[:, :, torch.arange(n) % 3 > 0] = 1.
        k[:, :, torch.arange(n) % 3 > 0] = -1.
    proj = _randn((1, 1, 64, 8), 312, torch.bfloat16).cuda()
    q_idx, k_idx = ops.forward_sort(q, k, proj, causal=causal, lsh_num_projs=8, min_seq_len=msl)
    bq, bk = ops.lsh_hash(q, proj), ops.lsh_hash(k, proj)
    if causal and n % 2:  # the appended zero row is in bucket 0
        bq, bk = (torch.cat([x, x.new_zeros((*x.shape[:2], 1))], -1) for x in (bq, bk))
    if causal:
        half = bq.shape[-1] // 2
        bq, bk = bq[..., half:], bk[..., :half]
    assert torch.equal(q_idx[0].long(), bq.sort(dim=-1, stable=True).indices)
    assert torch.equal(k_idx[0].long(), bk.sort(dim=-1, stable=True).indices)
