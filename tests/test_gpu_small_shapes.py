"""Shapes at the edges of the kernels' dispatch: the smallest launches, remainders of tiles, and the sizes on both sides
of a rule that picks a kernel variant."""
import pytest
import torch

from noise_amd import _lib
from tests._util import log_case

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _dense(x, w, layout, members, T):
    y = torch.empty(members * T, w.shape[0], device=DEV, dtype=torch.bfloat16)
    wp = w
    if layout == _lib.LAYOUT_WTILE:
        wp = torch.empty_like(w)
        _lib.call('noise_weight_tiles', w.data_ptr(), w.shape[0], w.shape[1], wp.data_ptr(), _stream())
    _lib.call('noise_dense_bf16', x.data_ptr(), _lib.LAYOUT_ROWS, w.shape[1], w.shape[0], wp.data_ptr(), layout, members,
              T, y.data_ptr(), _stream())
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize('dout', [256, 512, 1536])
@pytest.mark.parametrize('members,T', [(1, 32), (3, 96), (8, 256)])
def test_weight_resident_product_from_both_weight_layouts(members, T, dout):
    """The weight-resident kernel (512 deep, whole 32-row blocks) holds the same fragments whether the weight comes row
    by row through LDS or from WTILE blocks: equal bits, one block per launch up to several per workgroup, and within
    bf16 rounding (half a step of an 8-bit significand: 2^-8 relative) plus the fp32 sum's 512 2^-24 of the terms of the fp64 product."""
    g = torch.Generator().manual_seed(31)
    log_case(f'weight-resident product members={members} T={T} 512->{dout}')
    x = torch.randn(members * T, 512, generator=g).bfloat16()
    w = (torch.randn(dout, 512, generator=g) / 22).bfloat16()
    rows = _dense(x.to(DEV), w.to(DEV), _lib.LAYOUT_ROWS, members, T)
    tiles = _dense(x.to(DEV), w.to(DEV), _lib.LAYOUT_WTILE, members, T)
    assert torch.equal(rows, tiles)
    xd, wd = x.double(), w.double()
    ref = xd @ wd.t()
    bound = 2 ** -8 * ref.abs() + 512 * 2 ** -24 * (xd.abs() @ wd.abs().t())
    assert ((rows.cpu().double() - ref).abs() <= bound).all()
