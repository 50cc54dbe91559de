"""Causal lengths whose deepest level is exact as a whole (its halves are shorter than min_seq_len): its off-diagonal
part and its leaves are one launch over the level's segments."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _gen, _randn, assert_close
from oracle import hyper_oracle as O


@pytest.mark.parametrize("n,heads,kv_heads,d,dtype", [
    (1536, 2, 2, 64, torch.float16),    # one hashed level, two exact segments of 768
    (1535, 2, 1, 64, torch.bfloat16),   # the last segment has 767 rows
    (3071, 4, 2, 96, torch.float16),    # two hashed levels, four segments, the last of 767
    (3072, 2, 2, 128, torch.bfloat16),
    (1023, 3, 3, 128, torch.float16),   # no hashed level: the whole call is one exact launch
    (600, 2, 2, 40, torch.float16),
])
def test_exact_deepest_level_matches_the_oracle(n, heads, kv_heads, d, dtype):
    import hyperattention_amd as ha
    q = _randn((1, heads, n, d), 51, dtype)
    k, v = (_randn((1, kv_heads, n, d), s, dtype) for s in (52, 53))
    m = ha.HyperAttention(input_dim=d, block_size=128, sample_size=128, min_seq_len=512, rng=_gen(54)).to(device="cuda", dtype=dtype)
    attn, lse = m(q.cuda(), k.cuda(), v.cuda(), causal=True, return_lse=True)
    full = [x.repeat_interleave(heads // kv_heads, 1) for x in (k, v)]
    ref, ref_lse = O.hyper_forward(q, *full, m.lsh.proj_dir[0, 0].cpu(), causal=True, block_size=128, sample_size=128,
                                   min_seq_len=512)
    assert_close(attn, ref, "attn", dtype)
    assert_close(lse[:, :, :n].reshape(ref_lse.shape), ref_lse, "lse")
