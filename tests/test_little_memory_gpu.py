"""The fused forward on a device without room for a window of kept values: it takes the small
workspace, to the same bits, instead of running out of memory."""

import pytest
import torch

from nanospec_amd import _lib, head, synthetic
from nanospec_amd.config import Objective

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def largest(monkeypatch):
    """largest(bytes): from here on torch.empty refuses, as on a full device, what is larger."""
    empty = torch.empty

    def limit(nbytes):
        def refuse(*size, **kw):
            shape = size[0] if len(size) == 1 and isinstance(size[0], (tuple, list)) else size
            t = empty(shape, **{**kw, "device": "meta"})
            if t.numel() * t.element_size() > nbytes:
                raise torch.OutOfMemoryError("no room")
            return empty(*size, **kw)

        monkeypatch.setattr(torch, "empty", refuse)

    return limit


def _step(inputs, form):
    h, w, markov, u, slots, factors = inputs
    kw = {"factored": {"markov": factors}, "skip": {"markov_logits": markov, "skip_masked_rows": True},
          "dense": {"markov_logits": markov}}[form]
    m, saved = head.lm_head_ce_kl_loss(h, w, u, slots, Objective(block_size=8), **kw)
    stats = saved.row_stats.clone()
    dh, dl = head.lm_head_ce_kl_backward(saved, return_dlogits=True)
    torch.cuda.synchronize()
    return [m.numerator.clone(), m.denominator.clone(), stats[:, :4].clone(), dh, dl]


@pytest.mark.parametrize("form", ["dense", "factored", "skip"])
def test_no_room_for_the_kept_values(gpu_lib, largest, monkeypatch, form):
    n, d, v = 512, 320, 131072   # 268 MB of values, 134 MB of dl
    h, w, markov, u, slots = synthetic.head_inputs(n, d, v, 7700, DEV, ragged=True)
    factors = synthetic.markov_factors(n, v, 64, 7701, DEV)
    want = _step((h, w, markov, u, slots, head.MarkovFactors(*factors)), form)
    kinds, workspace = [], _lib.workspace
    monkeypatch.setattr(_lib, "workspace", lambda kind, *a, **kw: kinds.append(kind) or workspace(kind, *a, **kw))
    # dl and dh's partials fit, the values do not
    assert gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD, n, v, d) > 4 * n * v
    assert max(2 * n * v, gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, d)) < 4 * n * v
    largest(4 * n * v - 1)
    got = _step((h, w, markov, u, slots, head.MarkovFactors(*factors)), form)
    assert _lib.NS_WS_LMHEAD_MIN in kinds
    for a, b in zip(want, got):
        assert torch.equal(a, b)


def test_workspace_without_a_smaller_one_raises(gpu_lib, largest):
    largest(16 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        _lib.workspace(_lib.NS_WS_LMHEAD, 512, 131072, 320, torch.device(DEV))
