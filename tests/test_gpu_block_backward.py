"""The one-kernel backward of plain blocks of 256 at head dim 64 (csrc/attn_bwd_block.hip) at the edges of what it takes:
one block and many, a last block of half the rows, runs of blocks that do not divide a sequence, phases of sampled keys,
index types and layouts, results added to what is there."""
import ctypes

import pytest
import torch

from oracle import hyper_oracle as O
from test_gpu_backward import _check, _gpu_grads, _oracle_grads, _perms, ha  # noqa: F401 (fixture)
from _util import _gen, _randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,h,n,sample,idx", [
    (torch.float16, 1, 128, 0, torch.int64),       # half a block, nothing else
    (torch.bfloat16, 2, 256, 256, torch.int32),    # one block
    (torch.float16, 1, 384, 256, torch.int32),     # the last block is half
    (torch.bfloat16, 3, 1152, 512, torch.int64),   # two phases of sampled keys
    (torch.float16, 1, 1024, 1024, torch.int32),   # few blocks and many samples: three passes
    (torch.bfloat16, 17, 1024, 1024, torch.int64), # the most samples
    (torch.bfloat16, 1, 1280, 1280, torch.int32),  # three passes above
    (torch.float16, 66, 1152, 768, torch.int32),   # three phases, runs of blocks that end with half of one
    (torch.float16, 5, 16512, 256, torch.int32),   # 65 blocks in runs of two: the last run has one, of half the rows
])
def test_blocks_and_samples(ha, dtype, h, n, sample, idx):  # noqa: F811
    q, k, v, do = (_randn((1, h, n, 64), s, dtype) for s in (31, 32, 33, 34))
    qi, ki = _perms(1, h, n, 35), _perms(1, h, n, 36)
    ref = _oracle_grads(lambda a, b, c: O.block_sampled_attention(a, b, c, qi, ki, 256, sample, None, False), q, k, v, do)
    qi_g, ki_g = (x.cuda().to(idx).transpose(1, 2) for x in (qi, ki))
    _, _, *got = _gpu_grads(lambda a, b, c: ha.hyper_attn_func(a, b, c, qi_g, ki_g, 256, sample, None, False), q, k, v, do)
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, want, f"{name}, {h} x {n}, {sample} samples", dtype)


@pytest.mark.parametrize("dtype,h,n,idx", [
    (torch.float16, 896, 512, torch.int32),   # runs of two
    (torch.bfloat16, 600, 640, torch.int64),  # runs of three: the last block has half the rows
])
def test_two_phases_of_samples(ha, dtype, h, n, idx):  # noqa: F811
    """Many heads, four different ones in turn."""
    q, k, v, do = (_randn((1, 4, n, 64), s, dtype) for s in (31, 32, 33, 34))
    qi, ki = _perms(1, 4, n, 35), _perms(1, 4, n, 36)
    ref = _oracle_grads(lambda a, b, c: O.block_sampled_attention(a, b, c, qi, ki, 256, 512, None, False), q, k, v, do)
    many = lambda x: x.repeat(1, h // 4, *[1] * (x.dim() - 2))  # noqa: E731
    qi_g, ki_g = (many(x).cuda().to(idx).transpose(1, 2) for x in (qi, ki))
    _, _, *got = _gpu_grads(lambda a, b, c: ha.hyper_attn_func(a, b, c, qi_g, ki_g, 256, 512, None, False), *(many(x) for x in (q, k, v, do)))
    for g, want, name in zip(got, ref, ("dq", "dk", "dv")):
        _check(g, many(want), f"{name}, {h} x {n}", dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_adds_to_gradients_in_transposed_layout_and_keeps_an_explicit_list(ha, dtype):  # noqa: F811
    """Gradients added to (bnhd layout, repeated rows in an int64 sample list), a short last block: the result is
    what was there and the plain gradient, up to the rounding of the sum."""
    from hyperattention_amd import _lib, ops
    b, h, n, sample, scale = 2, 2, 896, 256, 0.11
    q, k, v, do = (_randn((b, n, h, 64), s, dtype).cuda() for s in (41, 42, 43, 44))
    qi, ki = (_perms(b, h, n, s).cuda().int().transpose(1, 2) for s in (45, 46))
    sl = torch.randint(0, n, (sample,), generator=_gen(47)).cuda()
    sl[1] = sl[0]
    o, lse = ops.hyper_attn_func(q, k, v, qi, ki, 256, sample, scale, False, sampled_idx=sl)
    ref = _oracle_grads(lambda x, y, z: O.block_sampled_attention(x, y, z, qi.transpose(1, 2).cpu().long(), ki.transpose(1, 2).cpu().long(),
                                                                  256, sample, scale, False, sampled_idx=sl.cpu()),
                        *(x.transpose(1, 2).cpu() for x in (q, k, v, do)))
    there = [_randn((b, n, h, 64), s, dtype).cuda() for s in (48, 49, 50)]
    grads = [x.clone() for x in there]
    a, _keep = ops._block_attn_args(q, k, v, o, lse, qi, ki, 256, sample, scale, False, sl)
    g, ws = ops._attn_grads(a.t, do, *grads, sample_size=sample)
    g.accumulate = 1
    _lib.check(_lib.lib().ha_block_attn_bwd(ctypes.byref(a), ctypes.byref(g), ops._stream(q)))
    torch.cuda.synchronize()
    # the sum is rounded to the type once more: half a unit of its last place, of values of N(0, 1) plus the gradient
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for got, was, want, name in zip(grads, there, ref, ("dq", "dk", "dv")):
        total = was.double().cpu().transpose(1, 2) + want
        err = (got.double().cpu().transpose(1, 2) - total).norm() / total.norm()
        assert err <= unit + (3e-3 if dtype == torch.float16 else 8e-3), f"{name}: {err:.2e}"
        assert torch.isfinite(got).all()


@pytest.mark.parametrize("dtype,h,n,out_d", [(torch.float16, 2, 640, 48), (torch.bfloat16, 3, 1024, 40), (torch.float16, 1, 256, 8)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_short_output_rows(ha, dtype, h, n, out_d, accumulate):  # noqa: F811
    """Head dims below 64 padded for the backward, with the forward's output as it is: bit for bit the gradients of padded output
    rows, from the same kernel (the three passes sum in another order)."""
    from hyperattention_amd import _lib, ops
    pad = lambda x: torch.nn.functional.pad(x, (0, 64 - out_d)).cuda()  # noqa: E731
    q, k, v, do = (pad(_randn((1, n, h, out_d), s, dtype)) for s in (51, 52, 53, 54))
    qi, ki = (_perms(1, h, n, s).cuda().int().transpose(1, 2) for s in (55, 56))
    o, lse = ops.hyper_attn_func(q, k, v, qi, ki, 256, 0, 0.2, False)
    there = [_randn((1, n, h, 64), s, dtype).cuda() for s in (57, 58, 59)]
    results = []
    for out, columns in ((o, 0), (o[..., :out_d].contiguous(), out_d)):
        grads = [x.clone() for x in there]
        a, _keep = ops._block_attn_args(q, k, v, out, lse, qi, ki, 256, 0, 0.2, False, None)
        g, _ws = ops._attn_grads(a.t, do, *grads)
        g.accumulate, g.out_d = int(accumulate), columns
        _lib.check(_lib.lib().ha_block_attn_bwd(ctypes.byref(a), ctypes.byref(g), ops._stream(q)))
        results.append(grads)
    for padded, short, name in zip(*results, ("dq", "dk", "dv")):
        assert torch.equal(padded, short), name


def test_small_workspace_takes_the_passes(ha):  # noqa: F811
    """A workspace without room for the workgroups' shares of the sampled keys' sums, as large as one of the sums alone."""
    from hyperattention_amd import _lib, ops
    h, n, sample = 24, 1024, 256
    q, k, v, do = (_randn((1, n, h, 64), s, torch.float16).cuda() for s in (61, 62, 63, 64))
    qi, ki = (_perms(1, h, n, s).cuda().int().transpose(1, 2) for s in (65, 66))
    o, lse = ops.hyper_attn_func(q, k, v, qi, ki, 256, sample, 0.125, False)
    a, _keep = ops._block_attn_args(q, k, v, o, lse, qi, ki, 256, sample, 0.125, False, None)
    results = []
    for small in (False, True):
        grads = [torch.empty_like(x) for x in (q, k, v)]
        g, ws = ops._attn_grads(a.t, do, *grads, sample_size=sample)
        if small:
            g.workspace_bytes = h * n * 8 + 2 * h * sample * 64 * 4
            assert g.workspace_bytes < ws.numel()
        _lib.check(_lib.lib().ha_block_attn_bwd(ctypes.byref(a), ctypes.byref(g), ops._stream(q)))
        results.append(grads)
    for x, y, name in zip(*results, ("dq", "dk", "dv")):
        # the same sums in another order, each rounded to fp16: half a unit of its last place on either side
        assert (x.double() - y.double()).norm() / y.double().norm() <= 2.0 ** -10, name


def test_runs_of_sixteen_blocks(ha):  # noqa: F811
    """One round of workgroups, each with 16 blocks: the passes' gradients (see above: the sums' order, each rounded to fp16)."""
    from hyperattention_amd import _lib, ops
    h, n, sample = 64, 16384, 256
    g = torch.Generator(device="cuda").manual_seed(71)
    q, k, v, do = (torch.randn((1, n, h, 64), generator=g, device="cuda", dtype=torch.float16) for _ in range(4))
    qi, ki = (torch.rand((1, h, n), generator=g, device="cuda").argsort(-1).int().transpose(1, 2) for _ in range(2))
    o, lse = ops.hyper_attn_func(q, k, v, qi, ki, 256, sample, 0.125, False)
    a, _keep = ops._block_attn_args(q, k, v, o, lse, qi, ki, 256, sample, 0.125, False, None)
    results = []
    for small in (False, True):
        grads = [torch.empty_like(x) for x in (q, k, v)]
        args, _ws = ops._attn_grads(a.t, do, *grads, sample_size=sample)
        if small:
            args.workspace_bytes = h * n * 8 + 2 * h * sample * 64 * 4
        _lib.check(_lib.lib().ha_block_attn_bwd(ctypes.byref(a), ctypes.byref(args), ops._stream(q)))
        results.append(grads)
    for x, y, name in zip(*results, ("dq", "dk", "dv")):
        assert (x.double() - y.double()).norm() / y.double().norm() <= 2.0 ** -10, name
