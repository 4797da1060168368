"""Narrow heads into 64-channel blocks and back on the GPU: the one-launch moves
equal the tensor-op maps bit for bit (they only copy), at partly filled blocks,
odd widths, one head and one channel, both element sizes, with inputs that are
not contiguous, and on rows that do not fill a wave's turn."""

import pytest
import torch

from pararnn_amd import ops
from pararnn_amd.head_blocks import HeadBlocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,dh,rows", [(1, 1, (1, 1)), (8, 24, (1, 67)), (3, 32, (2, 5)),
                                       (5, 20, (3, 33)), (2, 48, (1, 8)), (3, 63, (1, 129)),
                                       (65, 1, (2, 9)), (4, 32, (2, 7)), (2, 64, (1, 3))])
def test_moves_equal_the_tensor_maps(H, dh, rows, dtype):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(H * 100 + dh)
    hb = HeadBlocks(H, dh, dev)
    x = torch.randn(*rows, 3 * H * dh, generator=g).to(dev, dtype)
    h0 = torch.randn(rows[0], H * dh, generator=g).to(dev, dtype)
    y = torch.randn(*rows, 2 * H * dh, generator=g).to(dev, dtype)[..., ::2]
    x[0, 0, 0], y[-1, -1, -1] = float("nan"), float("inf")
    mats = [torch.randn(H, dh, dh, generator=g).to(dev, dtype) for _ in range(3)]
    mats[2] = mats[2].transpose(1, 2)
    chans, blocks = ops._to_blocks(hb, [(x, 3), (None, 1), (h0, 1), (y, 1)], mats)
    want = [hb.to_blocks(x, 3), None, hb.to_blocks(h0), hb.to_blocks(y)]
    for got, ref in zip(chans + blocks, want + [hb.matrices(m) for m in mats]):
        if ref is None:
            assert got is None
            continue
        assert got.shape == ref.shape and got.is_contiguous()
        assert torch.equal(got.nan_to_num(9.0, 8.0), ref.nan_to_num(9.0, 8.0))
    grads = torch.randn(3, hb.n_blocks, 64, 64, generator=g).to(dev)
    (bx, bh), (ga,) = ops._from_blocks(hb, [(chans[0], 3), (chans[2], 1)], [grads])
    assert torch.equal(bx.nan_to_num(9.0), x.nan_to_num(9.0)) and torch.equal(bh, h0)
    assert torch.equal(ga, hb.head_grads(grads))
