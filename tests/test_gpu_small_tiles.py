"""Head dim 64 in workgroups of 128 queries: gathered launches with windows of their own, plain ones and exact ones of a
few workgroups per CU, at ragged ends; exponents that follow the row maxima where they take the split kernel's place."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _gen, _randn, assert_close, forward_kernels
from oracle import hyper_oracle as O


def _inputs(h, hk, n, dtype):
    return (_randn((1, h, n, 64), 61, dtype), *(_randn((1, hk, n, 64), s, dtype) for s in (62, 63)))


# (heads, kv_heads, n): launches that the estimates give tiles of 128 queries, a last tile of 1, 60 and 127 rows; rows in a
# sequence's first tile only
@pytest.mark.parametrize("dtype,h,hk,n,causal", [
    (torch.bfloat16, 56, 56, 700, True), (torch.float16, 64, 32, 1025, True), (torch.bfloat16, 96, 96, 639, True),
    (torch.float16, 160, 160, 188, True), (torch.bfloat16, 64, 64, 1300, False), (torch.float16, 96, 48, 769, False),
])
def test_exact_in_tiles_of_128_queries(dtype, h, hk, n, causal):
    import hyperattention_amd as ha
    q, k, v = _inputs(h, hk, n, dtype)
    on_gpu = [x.cuda().transpose(1, 2) for x in (q, k, v)]
    call = lambda: ha.flash_attn_func(*on_gpu, None, causal)  # noqa: E731
    assert forward_kernels(call) == ["128 follow" if causal else "128"]
    o, lse = call()
    ro, rl = O.exact_attention(q, *(x.repeat_interleave(h // hk, 1) for x in (k, v)), None, causal)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :n], rl, "lse")


@pytest.mark.parametrize("dtype,h,hk,n,block,sample,smooth,split", [
    (torch.float16, 12, 12, 2560, 128, 128, False, None),   # in the split kernel's place: follows in 2 chunks
    (torch.bfloat16, 12, 6, 2560, 256, 256, False, None),   # plain, in 4 chunks
    (torch.float16, 16, 16, 2048, 256, 256, True, None),    # smooth, in 4 chunks
    (torch.bfloat16, 48, 48, 2048, 256, 256, False, None),  # plain, by the estimates
    (torch.float16, 2, 1, 1920, 384, 128, False, "0"),      # blocks of three tiles
    (torch.bfloat16, 2, 2, 1152, 512, 0, True, "0"),        # no samples, windows that wrap, a short last block
    (torch.float16, 2, 2, 384, 512, 128, True, "0"),        # a block longer than the sequence
    (torch.bfloat16, 2, 2, 128, 128, 128, False, "0"),      # one tile
])
def test_gathered_in_tiles_of_128_queries(monkeypatch, dtype, h, hk, n, block, sample, smooth, split):
    import hyperattention_amd as ha
    if split is not None:
        monkeypatch.setenv("HA_SPLIT", split)
    q, k, v = _inputs(h, hk, n, dtype)
    m = ha.HyperAttention(input_dim=64, block_size=block, sample_size=sample, min_seq_len=1, smooth_block=smooth,
                          rng=_gen(64)).to(device="cuda", dtype=dtype)
    call = lambda: m(q.cuda(), k.cuda(), v.cuda(), return_lse=True)  # noqa: E731
    assert forward_kernels(call) == ["128 follow" if h in (12, 16) else "128"]
    attn, lse = call()
    full = [x.repeat_interleave(h // hk, 1) for x in (k, v)]
    kw = dict(block_size=block, sample_size=sample, min_seq_len=1, smooth_block=smooth)
    ref, ref_lse = O.hyper_forward(q, *full, m.lsh.proj_dir[0, 0].cpu(), **kw)
    assert_close(attn, ref, "attn", dtype)
    assert_close(lse, ref_lse, "lse")
