"""Head dims above 64: workgroups of 128 queries, whose query and output rows are staged in tiles of keys and values.  Tile edges,
ragged ends, pairs of causal tiles (the second tile's rows arrive where the first's were staged) and single ones."""
import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_ops import ha  # noqa: F401 (fixture)
from _util import _gen, _randn, assert_close, forward_kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d,h,hk,n,causal", [
    (torch.bfloat16, 128, 2, 2, 1, False),
    (torch.float16, 128, 2, 1, 127, False),
    (torch.bfloat16, 96, 2, 2, 129, False),
    (torch.bfloat16, 128, 3, 3, 385, False),
    (torch.float16, 80, 2, 2, 640, False),
    (torch.bfloat16, 128, 2, 2, 1, True),          # single tiles
    (torch.float16, 128, 2, 1, 128, True),
    (torch.bfloat16, 128, 2, 2, 257, True),
    (torch.float16, 96, 5, 5, 1025, True),
    (torch.bfloat16, 128, 150, 150, 510, True),    # 600 workgroups: 256, 256 reversed, the rest in order
    (torch.bfloat16, 128, 200, 200, 890, True),    # 1400: single ones in more than one round of pairs
    (torch.float16, 96, 176, 88, 1025, True),      # a last tile of one row
    (torch.bfloat16, 96, 1040, 1040, 130, True),   # pairs of tiles: one pair, the second of 2 rows
    (torch.float16, 128, 520, 260, 500, True),     # two pairs
    (torch.bfloat16, 128, 520, 520, 384, True),    # three tiles, the middle one alone
])
def test_exact(ha, monkeypatch, dtype, d, h, hk, n, causal):  # noqa: F811
    monkeypatch.setenv("HA_SPLIT", "0")
    q = _randn((1, h, n, d), 71, dtype)
    k, v = (_randn((1, hk, n, d), s, dtype) for s in (72, 73))
    o, lse = ha.flash_attn_func(*(x.cuda().transpose(1, 2) for x in (q, k, v)), None, causal)
    ro, rl = O.exact_attention(q, *(x.repeat_interleave(h // hk, 1) for x in (k, v)), None, causal)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :n], rl, "lse")


# more than one round of split workgroups by the launcher's estimates: tiles whose exponents follow the row maxima in the first chunks
@pytest.mark.parametrize("dtype,d,h,hk,n,scale", [
    (torch.bfloat16, 128, 16, 16, 2048, 1.), (torch.float16, 96, 12, 4, 2676, 1.), (torch.bfloat16, 120, 8, 8, 3001, 1.),
    (torch.float16, 128, 16, 8, 2047, 12.),  # maxima that rise by hundreds
])
def test_exact_without_mask_in_rounds(ha, dtype, d, h, hk, n, scale):  # noqa: F811
    q = _randn((1, h, n, d), 74, dtype) * scale
    k, v = (_randn((1, hk, n, d), s, dtype) for s in (75, 76))
    on_gpu = [x.cuda().transpose(1, 2) for x in (q, k, v)]
    call = lambda: ha.flash_attn_func(*on_gpu, None, False)  # noqa: E731
    assert forward_kernels(call) == ["128 follow"]
    o, lse = call()
    ro, rl = O.exact_attention(q, *(x.repeat_interleave(h // hk, 1) for x in (k, v)), None, False)
    assert_close(o.transpose(1, 2), ro, "out", dtype)
    assert_close(lse[:, :, :n], rl, "lse")


@pytest.mark.parametrize("dtype,d,h,hk,n,smooth", [
    (torch.bfloat16, 128, 12, 12, 2688, False), (torch.float16, 96, 12, 4, 2688, False), (torch.bfloat16, 120, 12, 12, 2688, True),
])
def test_gathered_in_rounds(ha, dtype, d, h, hk, n, smooth):  # noqa: F811
    q = _randn((1, h, n, d), 77, dtype)
    k, v = (_randn((1, hk, n, d), s, dtype) for s in (78, 79))
    kw = dict(block_size=512, sample_size=512, min_seq_len=1, smooth_block=smooth)
    m = ha.HyperAttention(input_dim=d, rng=_gen(80), **kw).to(device="cuda", dtype=dtype)
    call = lambda: m(q.cuda(), k.cuda(), v.cuda(), return_lse=True)  # noqa: E731
    assert forward_kernels(call) == ["128 follow"]
    attn, lse = call()
    full = [x.repeat_interleave(h // hk, 1) for x in (k, v)]
    ref, ref_lse = O.hyper_forward(q, *full, m.lsh.proj_dir[0, 0].cpu(), **kw)
    assert_close(attn, ref, "attn", dtype)
    assert_close(lse, ref_lse, "lse")
