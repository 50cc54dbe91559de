"""GPU tests of what runs only at small launches: attention with the keys of a query tile split over waves, at the
edges of its tiles of 64 queries and 32 keys, against the oracle, and beside it the kernels it stands in for."""
import pytest
import torch

from oracle import hyper_oracle as O

pytestmark = pytest.mark.gpu

from _util import _randn, assert_close
from test_gpu_ops import _run_hyper, _sorted_inputs, ha  # noqa: F401


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 96), (torch.bfloat16, 40)])
@pytest.mark.parametrize("causal,nq,nk", [(True, 1, 1), (True, 63, 63), (True, 65, 65), (True, 321, 321), (False, 1, 33),
                                          (False, 64, 31), (False, 65, 129), (False, 257, 700)])
def test_exact_attention_at_tile_edges(ha, monkeypatch, split, dtype, d, causal, nq, nk):
    monkeypatch.setenv("HA_SPLIT", split)
    q = _randn((2, nq, 2, d), 11, dtype)
    k, v = (_randn((2, nk, 1, d), s, dtype) for s in (12, 13))
    o, lse = ha.flash_attn_func(q.cuda(), k.cuda(), v.cuda(), None, causal, None)
    expand = lambda x: x.transpose(1, 2).repeat_interleave(2, dim=1)
    args = (q.transpose(1, 2), expand(k), expand(v), None, causal)
    ro, rl = O.exact_attention(*args)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :nq], rl, "lse")


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("dtype,d,block,sample,smooth", [(torch.float16, 64, 128, 128, False), (torch.bfloat16, 128, 256, 0, False),
                                                         (torch.float16, 96, 384, 128, False), (torch.bfloat16, 64, 256, 128, True)])
def test_gathered_attention_resumed(ha, monkeypatch, split, dtype, d, block, sample, smooth):
    """640 rows (no multiple of the 256-query tile), with an explicit sample list, merged into a previous result."""
    monkeypatch.setenv("HA_SPLIT", split)
    b, h, n = 1, 2, 640
    q, k, v, qi, ki = _sorted_inputs(b, h, n, d, dtype, 40)
    sampled = torch.arange(n - sample, n) if sample else None
    o1, l1 = _run_hyper(ha, q, k, v, qi, ki, block, sample, None, smooth, sampled, torch.int32)
    o0, l0 = O.exact_attention(q, v, v, None, False)
    o0, l0 = o0.to(dtype), l0.float()
    c = lambda t: t.cuda().transpose(1, 2)
    o, lse = ha.hyper_attn_func(c(q), c(k), c(v), c(qi), c(ki), block, sample, None, smooth,
                                sampled_idx=None if sampled is None else sampled.cuda(), resume=(c(o0).contiguous(), l0.cuda()))
    ro, rl = O.block_sampled_attention(q, k, v, qi, ki, block, sample, None, smooth, sampled)
    assert_close(o1, ro, "out", dtype)
    assert_close(l1, rl, "lse")
    mo, ml = O.add_self_attentions(o0.double(), l0.double().unsqueeze(-1), ro, rl.unsqueeze(-1))
    assert_close(o.transpose(1, 2), mo, "merged out", dtype)
    assert_close(lse, ml.squeeze(-1), "merged lse")


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("d,n", [(64, 65), (128, 1), (128, 321), (64, 128)])
def test_padded_log_sum_exp_of_a_top_level_leaf_ends_in_zeros(ha, monkeypatch, split, d, n):
    monkeypatch.setenv("HA_SPLIT", split)
    q, k, v = (_randn((1, 2, n, d), s, torch.float16).cuda() for s in (21, 22, 23))
    m = ha.HyperAttention(input_dim=d).to(device="cuda", dtype=torch.float16)
    filler = torch.full((1, 2, -(-n // 128) * 128), 7.0, device="cuda")  # so that the next allocation holds no zeros
    del filler
    _, lse = m(q, k, v, causal=True, return_lse=True)
    assert lse.shape == (1, 2, -(-n // 128) * 128) and float(lse[..., n:].abs().sum()) == 0


@pytest.mark.parametrize("heads,n", [(3, 130), (700, 257), (1030, 257), (1030, 600)])  # 2, 4, 8 and 16 tiles per wave
def test_hash_at_every_wave_length(ha, heads, n):
    x = _randn((1, heads, n, 64), 31, torch.bfloat16)
    proj = _randn((1, 1, 64, 6), 32, torch.bfloat16)
    assert torch.equal(ha.lsh_hash(x.cuda(), proj.cuda()).cpu(), torch.as_tensor(O.lsh_hash(x, proj[0, 0])).int())


def test_module_without_hashing_takes_a_projection_it_does_not_read(ha):
    m = ha.HyperAttention(input_dim=64, min_seq_len=256)  # projection left in fp32 on the host
    q, k, v = (_randn((1, 2, 200, 64), s, torch.float16).cuda().requires_grad_() for s in (41, 42, 43))
    for causal in (True, False):
        out = m(q, k, v, causal=causal)
        ref, _ = O.exact_attention(*(x.detach().cpu() for x in (q, k, v)), None, causal)
        assert_close(out, ref, "out", torch.float16)
        torch.autograd.grad(out, q, torch.ones_like(out))
    long = [torch.cat([x.detach()] * 2 + [x.detach()[:, :, :112]], dim=2) for x in (q, k, v)]  # 512 rows: hashed
    with pytest.raises(AssertionError):
        m(*long, causal=False)
    m.lsh.proj_dir = m.lsh.proj_dir.half()  # the right type, still on the host
    with pytest.raises(AssertionError):
        m(*long, causal=False)
    with torch.no_grad():
        assert m(q, k, v, causal=True).shape == q.shape
