"""Bucket ids at the edges of the hash kernel's tiles of 16 rows, waves of 1, 2 and 4 tiles, and row widths."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from _util import _randn
from oracle import hyper_oracle as O


@pytest.fixture(scope="module")
def ha():
    import hyperattention_amd
    from hyperattention_amd import _lib
    _lib.lib()
    return hyperattention_amd


# (heads, n): one tile per wave with a remainder of 1 and of 15 rows; two tiles; four tiles (d <= 64) or two
@pytest.mark.parametrize("heads,n", [(2, 1), (3, 17), (2, 159), (700, 257), (1030, 271)])
@pytest.mark.parametrize("d,r", [(64, 8), (72, 6), (96, 8), (128, 8), (128, 16), (16, 9)])
def test_hash_at_tile_edges_and_row_widths(ha, heads, n, d, r):
    dtype = torch.bfloat16 if (heads + d) % 3 else torch.float16
    x = _randn((1, heads, n, d), 41, dtype)
    x[0, -1, -1] = 0                      # no sign: every bit is decided in float64
    if n > 16:
        x[0, 0, 16] = x[0, 0, 15]         # a row and its negative in neighbouring tiles
        x[0, 0, 15] = -x[0, 0, 15]
    if dtype == torch.bfloat16:
        x[0, 0, 0] *= 1e38                # finite values whose float32 sums are not
    proj = _randn((1, 1, d, r), 42, dtype)
    got = ha.lsh_hash(x.cuda(), proj.cuda()).cpu()
    assert torch.equal(got, torch.as_tensor(O.lsh_hash(x, proj[0, 0])).int())
