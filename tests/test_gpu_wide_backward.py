"""dk, dv with 256 keys and dq with 256 queries per workgroup at head dim 128 (csrc/attn_bwd_wide.hip,
attn_bwd_wide_dq.hip): launches that fill the chip with few rows
per head, at the edges of its tiles of 256 keys and 32 queries.  The shapes are ones that its dispatch rules take, or say so."""
import ctypes

import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_backward import _check, _gpu_grads, _oracle_grads, ha  # noqa: F401 (fixture)
from _util import _gen, _randn

pytestmark = pytest.mark.gpu

D = 128


def _orders(h, n, seed):
    return torch.rand((1, h, n), generator=_gen(seed)).argsort(-1)


def _grouped(fn, group):
    """An oracle with `group` query heads on each key head."""
    return lambda q, k, v: fn(q, k.repeat_interleave(group, 1), v.repeat_interleave(group, 1))


@pytest.mark.parametrize("dtype,h,hk,nq,nk,causal", [
    (torch.bfloat16, 640, 640, 128, 128, True),    # half the waves have no queries; dk, dv stay with the narrow pass
    (torch.float16, 640, 640, 64, 128, True),      # no queries, no keys, keys that nothing attends
    (torch.float16, 640, 640, 40, 33, True),       # two steps of dq, six waves without queries
    (torch.float16, 300, 300, 128, 128, True),     # too few for the wide passes
    (torch.bfloat16, 300, 300, 192, 192, False),
    (torch.float16, 300, 300, 77, 500, False),     # ragged on both sides
    (torch.bfloat16, 200, 200, 1001, 250, False),
    (torch.float16, 400, 200, 300, 300, True),     # two query heads, a last tile with 44 keys
    (torch.bfloat16, 300, 300, 300, 500, True),    # keys that nothing attends
    (torch.float16, 300, 300, 300, 256, True),     # queries after the last key
    (torch.bfloat16, 600, 200, 20, 260, False),    # one step per query head
    (torch.float16, 130, 130, 40, 33, True),       # nor these
])
def test_exact(ha, dtype, h, hk, nq, nk, causal):  # noqa: F811
    q, do = (_randn((1, h, nq, D), s, dtype) for s in (51, 52))
    k, v = (_randn((1, hk, nk, D), s, dtype) for s in (53, 54))
    ref = _oracle_grads(_grouped(lambda a, b, c: O.exact_attention(a, b, c, None, causal), h // hk), q, k, v, do)
    _, _, *got = _gpu_grads(lambda a, b, c: ha.flash_attn_func(a, b, c, None, causal), q, k, v, do)
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, want, name, dtype)


@pytest.mark.parametrize("dtype,h,hk,n,block,sample,idx", [
    (torch.float16, 130, 130, 128, 256, 0, torch.int64),     # half a block
    (torch.bfloat16, 65, 65, 384, 256, 128, torch.int32),    # the last block is half
    (torch.float16, 44, 44, 640, 512, 256, torch.int32),     # two tiles of a block, a short block
    (torch.bfloat16, 132, 44, 640, 256, 0, torch.int64),     # three query heads on each key head
    (torch.float16, 52, 26, 1280, 1024, 0, torch.int32),     # four tiles of a block, two of a short one
    (torch.float16, 44, 22, 1280, 1024, 0, torch.int32),     # too few for the wide pass
])
def test_blocks(ha, dtype, h, hk, n, block, sample, idx):  # noqa: F811
    q, do = (_randn((1, h, n, D), s, dtype) for s in (61, 62))
    k, v = (_randn((1, hk, n, D), s, dtype) for s in (63, 64))
    qi, ki = _orders(h, n, 65), _orders(hk, n, 66)
    group = h // hk
    ref = _oracle_grads(_grouped(lambda a, b, c: O.block_sampled_attention(a, b, c, qi, ki.repeat_interleave(group, 1), block, sample), group),
                        q, k, v, do)
    qi_g, ki_g = (x.cuda().to(idx).transpose(1, 2) for x in (qi, ki))
    _, _, *got = _gpu_grads(lambda a, b, c: ha.hyper_attn_func(a, b, c, qi_g, ki_g, block, sample, None, False), q, k, v, do)
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, want, name, dtype)


@pytest.mark.parametrize("dtype,h,hk,n,sample,smooth", [
    (torch.float16, 130, 130, 384, 256, False),    # one share: the sums themselves
    (torch.bfloat16, 33, 33, 2048, 256, True),     # ranges of a head's queries
    (torch.float16, 44, 11, 1664, 512, False),     # and four heads; two tiles of sampled keys
])
def test_sampled_keys(ha, dtype, h, hk, n, sample, smooth):  # noqa: F811
    """Sums of the sampled keys from shares in the workspace, and, in a workspace without room for them, by atomics; a row
    listed twice."""
    from hyperattention_amd import _lib, ops
    q, do = (_randn((1, n, h, D), s, dtype).cuda() for s in (101, 102))
    k, v = (_randn((1, n, hk, D), s, dtype).cuda() for s in (103, 104))
    qi, ki = _orders(h, n, 105), _orders(hk, n, 106)
    sl = torch.randint(0, n, (sample,), generator=_gen(107))
    sl[sample - 1] = sl[3]
    group = h // hk
    ref = _oracle_grads(_grouped(lambda a, b, c: O.block_sampled_attention(a, b, c, qi, ki.repeat_interleave(group, 1), 256, sample,
                                                                           None, smooth, sampled_idx=sl), group),
                        *(x.transpose(1, 2).cpu() for x in (q, k, v, do)))
    qi_g, ki_g = (x.cuda().int().transpose(1, 2) for x in (qi, ki))
    o, lse = ops.hyper_attn_func(q, k, v, qi_g, ki_g, 256, sample, None, smooth, sampled_idx=sl.cuda())
    a, _keep = ops._block_attn_args(q, k, v, o, lse, qi_g, ki_g, 256, sample, D ** -0.5, smooth, sl.cuda())
    sums = (h * n * 8 + 255) // 256 * 256 + 2 * hk * sample * D * 4  # statistics, one row of dk and dv per slot
    for room in (True, False):
        grads = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        g, ws = ops._attn_grads(a.t, do, *grads, sample_size=sample)
        assert g.workspace_bytes >= sums and (group == 1 or g.workspace_bytes > sums)
        ws.fill_(255)  # NaN: nothing is read that has not been written
        if not room:
            g.workspace_bytes = sums
        _lib.check(_lib.lib().ha_block_attn_bwd(ctypes.byref(a), ctypes.byref(g), ops._stream(q)))
        torch.cuda.synchronize()
        for got, want, name in zip(grads, ref, ("dq", "dk", "dv")):
            _check(got.transpose(1, 2), want, f"{name}, room {room}", dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("exact", [False, True])
def test_adds_to_what_is_there(ha, dtype, exact):  # noqa: F811
    """Gradients added to (bnhd layout): the result is what was there and the plain gradient, up to the rounding of the sum."""
    from hyperattention_amd import _lib, ops
    h, n = (300, 200) if exact else (70, 384)
    q, k, v, do = (_randn((1, n, h, D), s, dtype).cuda() for s in (71, 72, 73, 74))
    qi, ki = _orders(h, n, 75), _orders(h, n, 76)
    back = lambda x: x.transpose(1, 2).cpu()  # noqa: E731
    if exact:
        fn = lambda a, b, c: O.exact_attention(a, b, c, None, False)  # noqa: E731
        o, lse = ops.flash_attn_func(q, k, v)
        t, entry = ops._operands(q, k, v, o, lse, D ** -0.5, layout_bnhd=True, lse_row_stride=lse.shape[-1]), _lib.lib().ha_flash_attn_bwd
    else:
        fn = lambda a, b, c: O.block_sampled_attention(a, b, c, qi, ki, 256)  # noqa: E731
        qi_g, ki_g = (x.cuda().int().transpose(1, 2) for x in (qi, ki))
        o, lse = ops.hyper_attn_func(q, k, v, qi_g, ki_g, 256, 0, None, False)
        a, _keep = ops._block_attn_args(q, k, v, o, lse, qi_g, ki_g, 256, 0, D ** -0.5, False, None)
        t, entry = a.t, _lib.lib().ha_block_attn_bwd
    ref = _oracle_grads(fn, *(back(x) for x in (q, k, v, do)))
    there = [_randn((1, n, h, D), s, dtype).cuda() for s in (77, 78, 79)]
    grads = [x.clone() for x in there]
    g, ws = ops._attn_grads(t, do, *grads, sample_size=0)
    g.accumulate = 1
    if exact:
        _lib.check(entry(ctypes.byref(t), 0, ctypes.byref(g), ops._stream(q)))
    else:
        _lib.check(entry(ctypes.byref(a), ctypes.byref(g), ops._stream(q)))
    torch.cuda.synchronize()
    # the sum is rounded to the type once more: half a unit of its last place, of values of N(0, 1) plus the gradient
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for got, was, want, name in zip(grads, there, ref, ("dq", "dk", "dv")):
        total = back(was).double() + want
        err = (back(got).double() - total).norm() / total.norm()
        assert err <= unit + (3e-3 if dtype == torch.float16 else 8e-3), f"{name}: {err:.2e}"
        assert torch.isfinite(got).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("h,n,causal", [(300, 200, False), (320, 200, True), (4, 200, True)])  # the last not in 256 rows
@pytest.mark.parametrize("dead", ["q", "k"])
def test_a_sum_added_to_what_is_there_is_rounded_once(ha, dtype, h, n, causal, dead):  # noqa: F811
    """Gradients of exact attention added to.  The inputs make every fp32 sum exact and not representable in 16 bits: with
    q or k zero and log-sum-exps of log(256) all weights are 1/256, O is zero (D = 0), v has one column of -1, 0, 1, and dO
    and the other of q and k are whole numbers whose products stay below 2^24.  So the one rounding, of the sum with what
    is there, is known to the bit."""
    from hyperattention_amd import _lib, ops
    gen, top = _gen(81), 1000 if dtype == torch.float16 else 100
    whole = lambda limit: torch.randint(-limit, limit + 1, (1, n, h, D), generator=gen).double()  # noqa: E731
    q, k, do, v = whole(63), whole(63), whole(top), whole(1)
    v[..., 1:] = 0
    (q if dead == "q" else k).zero_()
    heads = lambda x: x.transpose(1, 2)  # noqa: E731
    weight = torch.ones(n, n, dtype=torch.float64) / 256
    if causal:
        weight = weight.tril()
    scale = 0.125
    ds = weight * (heads(do) @ heads(v).transpose(-1, -2).contiguous()) * scale
    sums = [ds @ heads(k), ds.transpose(-1, -2).contiguous() @ heads(q), weight.T.contiguous() @ heads(do)]
    there = [(torch.randn((1, n, h, D), generator=gen) * max(x.std().item(), 1.)).to(dtype) for x in sums]
    q_g, k_g, v_g, do_g = (x.to(dtype).cuda() for x in (q, k, v, do))
    lse = torch.full((1, h, n), 256., device="cuda").log()
    out = torch.zeros_like(q_g)
    t = ops._operands(q_g, k_g, v_g, out, lse, scale, layout_bnhd=True, lse_row_stride=n)
    grads = [x.cuda() for x in there]
    g, ws = ops._attn_grads(t, do_g, *grads, accumulate=True)
    _lib.check(_lib.lib().ha_flash_attn_bwd(ctypes.byref(t), int(causal), ctypes.byref(g), ops._stream(q_g)))
    torch.cuda.synchronize()
    for got, was, want, name in zip(grads, there, sums, ("dq", "dk", "dv")):
        total = (was.float() + heads(want).float()).to(dtype)
        assert torch.equal(got.cpu(), total), f"{name}: {(got.cpu() != total).float().mean().item():.3f} of the elements differ"
