"""dh = dl . W_lm over the K split counts the plan picks: one workgroup's share of K down to a
single 64-entry block, sums of partials in one, four and sixteen groups, ragged token, column
and K edges; against fp64."""

import pytest
import torch

from nanospec_amd import ops

from dh_bar import assert_dh_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,d,v", [
    (1, 64, 8), (7, 64, 64), (8, 72, 8200),        # one block of K; many splits of one tile
    (64, 256, 8192), (257, 256, 16392),            # 128 and 128 splits, a token tile of one row
    (224, 1032, 8192), (300, 2048, 4104),          # a partial column tile; 16 splits of 16 tiles
    (520, 5120, 2048), (2048, 264, 4096),
])
def test_dh_against_fp64(gpu_lib, n, d, v):
    g = torch.Generator(device=DEV).manual_seed(n * 7 + d)
    dl = (torch.randn((n, v), generator=g, device=DEV) * torch.rand((n, 1), generator=g, device=DEV)).bfloat16()
    w = (0.02 * torch.randn((v, d), generator=g, device=DEV)).bfloat16()
    got = ops.lm_head_backward(dl, w)
    assert torch.equal(got, ops.lm_head_backward(dl, w))
    want = dl.double() @ w.double()
    assert_dh_rows(got.float().cpu().numpy(), want.float().cpu().numpy())
