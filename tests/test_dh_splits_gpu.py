"""dh = dl . W_lm over the K split counts the plan picks: one workgroup's share of K down to a
single 64-entry block, sums of partials in one, four and sixteen groups, ragged token, column
and K edges; against fp64."""

import pytest
import torch

from nanospec_amd import _lib, ops

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


@pytest.mark.parametrize("n,d,v", [(8, 256, 32000), (64, 1024, 65536), (300, 256, 32000)])
@pytest.mark.parametrize("splits", [16, 17, 40])
def test_dh_in_a_workspace_of_fewer_splits(gpu_lib, n, d, v, splits):
    """Where the plan would take more K splits than the workspace holds, dh takes those that fit; less
    than 16 is refused.  Nothing past the bytes given is written."""
    g = torch.Generator(device=DEV).manual_seed(n + splits)
    dl = (torch.randn((n, v), generator=g, device=DEV) * torch.rand((n, 1), generator=g, device=DEV)).bfloat16()
    w = (0.02 * torch.randn((v, d), generator=g, device=DEV)).bfloat16()
    given = splits * n * d * 4
    assert gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, d) > given
    ws = torch.full((given + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
    dh = torch.empty((n, d), dtype=torch.bfloat16, device=DEV)
    args = (_lib.ptr(dl), v, _lib.ptr(w), d, _lib.ptr(dh), d, n, v, d, _lib.ptr(ws))
    st = _lib.stream(torch.device(DEV))
    _lib.check(gpu_lib.ns_lmhead_bwd(*args, given, st), "ns_lmhead_bwd")
    assert_dh_rows(dh.float().cpu().numpy(), (dl.double() @ w.double()).float().cpu().numpy())
    assert bool((ws[given:] == 0x5a).all())
    with pytest.raises(ValueError, match="workspace"):
        _lib.check(gpu_lib.ns_lmhead_bwd(*args, 16 * n * d * 4 - 256, st), "ns_lmhead_bwd")


@pytest.mark.parametrize("norm", [False, True])
def test_markov_backward_in_a_smaller_workspace(gpu_lib, norm):
    """The factored Markov head's backward with the fewest splits it accepts is its backward with
    all of them, to the sums' order."""
    from nanospec_amd import head, synthetic

    n, d, v, r = 64, 256, 32000, 64
    g = torch.Generator(device=DEV).manual_seed(81)
    dl = (torch.randn((n, v), generator=g, device=DEV) * 1e-2).bfloat16()
    w = (0.02 * torch.randn((v, d), generator=g, device=DEV)).bfloat16()
    mk = head.MarkovFactors(*synthetic.markov_factors(n, v, r, 82, DEV))
    x = torch.randn((n, d), generator=g, device=DEV).bfloat16()
    nw = torch.ones(d, dtype=torch.bfloat16, device=DEV)
    _, saved = ops.rms_norm(x, nw, 1e-6)
    full = int(gpu_lib.ns_lmhead_markov_bwd_workspace_bytes(n, v, d, r))
    splits = int(gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, d)) // (4 * n * d)
    assert splits > 16

    def run(nbytes):
        ws = torch.full((nbytes + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
        g1 = torch.zeros((v, r), dtype=torch.bfloat16, device=DEV)
        g2 = torch.empty((v, r), dtype=torch.bfloat16, device=DEV)
        wg, dh = torch.zeros_like(nw), torch.zeros((n, d), dtype=torch.bfloat16, device=DEV)
        args = keep = None
        if norm:
            args, dh, keep = head._final_norm_args((saved, nw, wg), n, d, torch.device(DEV))
        status = gpu_lib.ns_lmhead_markov_bwd(
            _lib.ptr(dl), v, _lib.ptr(w), d, _lib.ptr(mk.previous), _lib.ptr(mk.w1), r, _lib.ptr(mk.w2), r, r,
            None if norm else _lib.ptr(dh), d, args, _lib.ptr(g1), r, _lib.ptr(g2), r, n, v, d, _lib.ptr(ws), nbytes,
            _lib.stream(torch.device(DEV)))
        _lib.check(status, "ns_lmhead_markov_bwd")
        torch.cuda.synchronize()
        assert bool((ws[nbytes:] == 0x5a).all())
        return dh, g1, g2, wg

    a, b = run(full), run(full - (splits - 16) * n * d * 4)
    assert torch.equal(a[2], b[2])   # dl^T . w1[previous] takes no part of it
    # fp32 sums of 32000 products in another order (2^-24 each, 64 of them in a chain at most),
    # rounded to bf16: a unit in the last place, 2^-8
    for p, q in zip(a, b):
        assert float((p.double() - q.double()).norm()) <= 2.0 ** -8 * float(p.double().norm()) + 1e-30
    with pytest.raises(ValueError, match="workspace"):
        run(full - (splits - 15) * n * d * 4)
