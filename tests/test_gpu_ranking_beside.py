"""Units hashed and ranked by workgroups of the exact causal launch: the forward pass in one call against the same launches with
the orders of ha_forward_sort (hash, rank and placement launches), and at odd lengths its orders themselves, bit for bit."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn


def _launch_by_launch(q, k, v, proj, projs, block, sample, msl):
    """The leaves, then the hashed levels merged in place, as hyper_forward runs them; even lengths."""
    from hyperattention_amd import _lib, ops
    b, h, n, d = q.shape
    hk = k.shape[1]
    q_idx, k_idx = ops.forward_sort(q, k, proj, causal=True, lsh_num_projs=projs, min_seq_len=msl)
    halves, leaf = ops.causal_plan(n, msl)
    hashed = [j for j, x in enumerate(q_idx) if x is not None]
    out, lse = torch.empty_like(q), torch.empty((b, h, n), device=q.device, dtype=torch.float32)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def operands(segs, rows, stride, q_off):
        t = _lib.AttnOperands()
        t.q, t.k, t.v, t.out, t.lse = (x.data_ptr() for x in (q, k, v, out, lse))
        t.batch, t.heads, t.n_q, t.n_k, t.d, t.dv = b, h, rows, rows, d, d
        for name, x in (("q", q), ("k", k), ("v", v), ("o", out)):
            for i, axis in enumerate("bhn"):
                setattr(t, f"{name}_stride_{axis}", x.stride(i))
        t.lse_stride_b, t.lse_stride_h = h * n, n
        t.segs, t.seg_stride_rows, t.q_seg_offset, t.k_seg_offset = segs, stride, q_off, 0
        t.kv_group, t.scale, t.dtype = h // hk, d ** -0.5, ops._dtype_code(q)
        return t

    levels = len(hashed)  # a deepest level that is not hashed is exact as a whole
    rows = n if not halves else halves[levels - 1]
    _lib.check(_lib.lib().ha_flash_attn_fwd(ctypes.byref(operands(1 << levels, rows, rows, 0)), 1, stream))
    for j in reversed(hashed):
        a = _lib.BlockAttnArgs()
        half = halves[j]
        a.t = operands(1 << j, half, 2 * half, half)
        a.q_idx, a.k_idx = q_idx[j].data_ptr(), k_idx[j].data_ptr()
        a.q_idx_stride_b, a.q_idx_stride_h, a.q_idx_stride_n = h * (half << j), half << j, 1
        a.k_idx_stride_b, a.k_idx_stride_h, a.k_idx_stride_n = hk * (half << j), half << j, 1
        a.block_size, a.sample_size, a.accumulate = block, sample, 1
        _lib.check(_lib.lib().ha_block_attn_fwd(ctypes.byref(a), stream))
    return out, lse


@pytest.mark.parametrize("b,h,hk,n,msl,d,projs,dtype", [
    (1, 2, 2, 256, 128, 64, 8, torch.float16),        # one segment of 128 rows, less than a step per wave
    (1, 3, 1, 1536, 512, 64, 8, torch.bfloat16),      # the deepest level, of 384 rows, is exact
    (1, 24, 24, 4096, 2048, 64, 8, torch.bfloat16),   # in front of the tiles: they take every place
    (2, 4, 2, 8448, 4200, 64, 6, torch.float16),      # a unit of 4224 rows, a whole segment
    (1, 2, 1, 16384, 8192, 64, 8, torch.bfloat16),    # the longest such one
    (1, 2, 1, 16640, 8300, 64, 8, torch.bfloat16),    # three units and their placement
    (1, 8, 8, 15360, 1024, 64, 8, torch.float16),     # four levels, one unit per granule of 1920
    (4, 24, 24, 10240, 2048, 64, 8, torch.float16),   # pairs of tiles
    (1, 2, 2, 9216, 4100, 128, 8, torch.bfloat16),    # two units of 4608 rows in a granule, the second of 512
    (1, 2, 2, 4096, 512, 128, 8, torch.float16),      # the split kernel
    (1, 16, 2, 8192, 2048, 128, 7, torch.bfloat16),
    (1, 35, 35, 4096, 2048, 128, 8, torch.float16),   # eight waves per workgroup
    (1, 4, 2, 4096, 1024, 40, 8, torch.bfloat16),     # rows shorter than their place
    (1, 24, 12, 8192, 2048, 96, 8, torch.float16),
    (2, 8, 8, 4096, 512, 80, 5, torch.bfloat16),
    (1, 4, 4, 2048, 256, 112, 8, torch.float16),
    (64, 32, 32, 2048, 1024, 16, 8, torch.float16),   # so many units that they are hashed ahead of the leaves
])
def test_orders_are_those_of_the_sort(b, h, hk, n, msl, d, projs, dtype):
    from hyperattention_amd import ops
    q, v = (_randn((b, x, n, d), s, dtype).cuda() for x, s in ((h, 610), (hk, 612)))
    k = _randn((b, hk, n, d), 611, dtype).cuda()
    # equal rows tie, and their places in the order show in what they attend to
    q[:, :, torch.arange(n) % 3 > 0] = q[:, :, :1].clone()
    k[:, :, torch.arange(n) % 5 > 2] = k[:, :, :1].clone()
    proj = _randn((1, 1, d, projs), 613, dtype).cuda()
    got = ops.hyper_forward(q, k, v, proj, scale=d ** -0.5, causal=True, lsh_num_projs=projs, block_size=128, sample_size=128,
                            min_seq_len=msl, smooth_block=False)
    want = _launch_by_launch(q, k, v, proj, projs, 128, 128, msl)
    for x, y in zip(got, want):
        assert torch.equal(x, y)


@pytest.mark.parametrize("b,h,hk,n,msl,d,projs,dtype", [
    (1, 2, 2, 256, 128, 64, 8, torch.float16),        # one segment, no placement
    (1, 24, 24, 4096, 2048, 64, 8, torch.bfloat16),
    (1, 3, 1, 3072, 512, 64, 8, torch.bfloat16),      # two hashed levels and an exact one
    (2, 4, 2, 8192, 1024, 128, 7, torch.float16),
    (1, 4, 2, 4096, 1024, 80, 8, torch.bfloat16),
    (1, 2, 2, 2048, 512, 64, 9, torch.float16),       # more buckets than a unit's ranking takes: launches of their own
    (1, 2, 2, 1000, 1024, 64, 8, torch.float16),      # no level at all
])
def test_sort_with_the_leaves(b, h, hk, n, msl, d, projs, dtype):
    """ha_forward_sort_leaves on transposed views: the orders of ha_forward_sort, the leaves of ha_flash_attn_fwd, bit for bit."""
    from hyperattention_amd import _lib, ops
    q, k, v = (_randn((b, n, x, d), s, dtype).cuda().transpose(1, 2) for x, s in ((h, 620), (hk, 621), (hk, 622)))
    k[:, :, torch.arange(n) % 5 > 2] = k[:, :, :1].clone()  # ties
    proj = _randn((1, 1, d, projs), 623, dtype).cuda()
    want_q, want_k = ops.forward_sort(q, k, proj, causal=True, lsh_num_projs=projs, min_seq_len=msl)
    halves, leaf = ops.causal_plan(n, msl)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    t = _lib.AttnOperands()
    t.batch, t.heads, t.n_q, t.n_k, t.d, t.dv = b, h, leaf, leaf, d, d
    t.segs, t.seg_stride_rows, t.kv_group, t.scale, t.dtype = 1 << len(halves), leaf, h // hk, d ** -0.5, ops._dtype_code(q)
    t.lse_stride_b, t.lse_stride_h = h * n, n
    results = []
    for with_sort in (False, True):
        out, lse = torch.zeros((b, h, n, d), device="cuda", dtype=dtype), torch.zeros((b, h, n), device="cuda")
        for name, x in (("q", q), ("k", k), ("v", v), ("o", out)):
            for i, axis in enumerate("bhn"):
                setattr(t, f"{name}_stride_{axis}", x.stride(i))
        t.q, t.k, t.v, t.out, t.lse = (x.data_ptr() for x in (q, k, v, out, lse))
        if with_sort:
            a, keep = ops._forward_args(q, k, None, None, None, proj, scale=1.0, causal=True, lsh_num_projs=projs, block_size=128,
                                        sample_size=0, min_seq_len=msl, smooth_block=False)
            q_at, k_at, levels = (ctypes.c_int64 * 48)(), (ctypes.c_int64 * 48)(), ctypes.c_int(0)
            _lib.check(_lib.lib().ha_forward_sort_leaves(ctypes.byref(a), ctypes.byref(t), q_at, k_at, ctypes.byref(levels), stream))
            assert levels.value == len(want_q)
            for at, want in ((q_at, want_q), (k_at, want_k)):
                for j, w in enumerate(want):
                    assert (at[j] < 0) == (w is None)
                    if w is not None:
                        got = keep[-1][at[j]:at[j] + 4 * w.numel()].view(torch.int32).view(w.shape)
                        assert torch.equal(got, w)
            t.k = t.v  # another tensor than the one that is hashed: refused before any launch
            if want_q and want_q[0] is not None:
                assert _lib.lib().ha_forward_sort_leaves(ctypes.byref(a), ctypes.byref(t), q_at, k_at, ctypes.byref(levels), stream) == -3
        else:
            _lib.check(_lib.lib().ha_flash_attn_fwd(ctypes.byref(t), 1, stream))
        results.append((out, lse))
    for x, y in zip(*results):
        assert torch.equal(x, y)


@pytest.mark.parametrize("b,h,hk,n,msl,d,projs,dtype", [
    (1, 2, 2, 255, 128, 64, 8, torch.float16),        # a unit is a whole segment, its last row the appended one
    (1, 24, 24, 4095, 2048, 64, 8, torch.bfloat16),
    (2, 4, 2, 8447, 4200, 64, 6, torch.float16),
    (1, 2, 1, 16639, 8300, 64, 8, torch.bfloat16),    # three units per granule, the last of 128 rows
    (1, 8, 8, 15359, 1024, 64, 8, torch.float16),     # ragged leaves under three hashed levels
    (1, 4, 2, 4095, 1024, 40, 8, torch.bfloat16),
    (1, 2, 1, 12287, 6000, 96, 8, torch.bfloat16),
    (1, 12, 4, 5119, 1024, 96, 7, torch.float16),
    (1, 2, 2, 9215, 4100, 128, 8, torch.bfloat16),    # units of 4096 and 512 rows
    (1, 16, 2, 8191, 2048, 128, 8, torch.float16),
])
def test_odd_lengths_place_the_appended_row(b, h, hk, n, msl, d, projs, dtype):
    """The orders that ha_forward leaves in its workspace against ha_forward_sort's of the same rows, bit for bit.  Where they lie is
    asked of ha_forward_sort_leaves, for the rows with the zero row that the recursion appends; its orders are the same too."""
    from hyperattention_amd import _lib, ops
    q, k, v = (_randn((b, x, n, d), s, dtype).cuda() for x, s in ((h, 640), (hk, 641), (hk, 642)))
    q[:, :, torch.arange(n) % 4 > 1] = q[:, :, :1].clone()
    k[:, :, torch.arange(n) % 3 > 1] = k[:, :, :1].clone()
    for x in (q, k):  # rows that tie with the appended one, at the end and before
        x[:, :, n - 5:n - 2] = 0
        x[:, :, n // 3] = 0
    proj = _randn((1, 1, d, projs), 643, dtype).cuda()
    want = ops.forward_sort(q, k, proj, causal=True, lsh_num_projs=projs, min_seq_len=msl)
    opts = dict(scale=d ** -0.5, causal=True, lsh_num_projs=projs, block_size=128, sample_size=128, min_seq_len=msl, smooth_block=False)
    lib, stream = _lib.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out, lse = torch.empty_like(q), torch.empty((b, h, n), device="cuda")
    a, keep = ops._forward_args(q, k, v, out, lse, proj, **opts)
    _lib.check(lib.ha_forward(ctypes.byref(a), stream))

    pq, pk, pv = (torch.nn.functional.pad(x, (0, 0, 0, 1)) for x in (q, k, v))
    halves, leaf = ops.causal_plan(n + 1, msl)
    pa, pkeep = ops._forward_args(pq, pk, None, None, None, proj, **opts)
    po, pl = torch.empty_like(pq), torch.empty((b, h, n + 1), device="cuda")
    t = _lib.AttnOperands()
    t.batch, t.heads, t.n_q, t.n_k, t.d, t.dv = b, h, leaf, leaf, d, d
    t.segs, t.seg_stride_rows, t.kv_group, t.scale, t.dtype = 1 << len(halves), leaf, h // hk, d ** -0.5, ops._dtype_code(q)
    t.lse_stride_b, t.lse_stride_h = h * (n + 1), n + 1
    for name, x in (("q", pq), ("k", pk), ("v", pv), ("o", po)):
        for i, axis in enumerate("bhn"):
            setattr(t, f"{name}_stride_{axis}", x.stride(i))
    t.q, t.k, t.v, t.out, t.lse = (x.data_ptr() for x in (pq, pk, pv, po, pl))
    at = (ctypes.c_int64 * 48)(), (ctypes.c_int64 * 48)()
    levels = ctypes.c_int(0)
    _lib.check(lib.ha_forward_sort_leaves(ctypes.byref(pa), ctypes.byref(t), *at, ctypes.byref(levels), stream))
    for side in (0, 1):
        for j, w in enumerate(want[side]):
            assert (at[side][j] < 0) == (w is None)
            if w is not None:
                for ws in (keep[-1], pkeep[-1]):
                    got = ws[at[side][j]:at[side][j] + 4 * w.numel()].view(torch.int32).view(w.shape)
                    assert torch.equal(got, w), (side, j)


@pytest.mark.parametrize("b,n,msl,beside", [
    (24, 512, 256, True),      # 1536 units of 256 rows
    (25, 512, 256, False),     # more of so few rows are hashed in a launch of their own
    (32, 2048, 1024, True),    # 2048 units of 1024 rows
    (33, 2048, 1024, False),
])
def test_many_units_are_hashed_ahead(b, n, msl, beside):
    from torch.profiler import ProfilerActivity, profile
    from hyperattention_amd import ops
    g = torch.Generator(device="cuda").manual_seed(630)
    q, k, v = (torch.randn((b, 32, n, 16), generator=g, device="cuda", dtype=torch.float16) for _ in range(3))
    proj = torch.randn((1, 1, 16, 8), generator=g, device="cuda", dtype=torch.float16)

    def call():
        ops.hyper_forward(q, k, v, proj, scale=0.25, causal=True, lsh_num_projs=8, block_size=128, sample_size=128,
                          min_seq_len=msl, smooth_block=False)
        torch.cuda.synchronize()

    call()
    with profile(activities=[ProfilerActivity.CUDA]) as trace:
        call()
    names = [e.name for e in trace.events()]
    assert any("ha_attn_fwd" in x for x in names), "no attention kernel in the trace"
    assert any("lsh_hash" in x for x in names) == (not beside)
