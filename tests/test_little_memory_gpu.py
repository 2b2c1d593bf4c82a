"""The fused forward on a device without room for a window of kept values: it takes the small
workspace, to the same bits, instead of running out of memory."""

import pytest
import torch

from nanospec_amd import _lib, head, synthetic
from nanospec_amd.config import Objective

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def room():
    """room(bytes): no more than that may be allocated from here on, until the test ends."""
    total = torch.cuda.get_device_properties(0).total_memory

    def limit(nbytes):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + nbytes) / total, 0)

    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0, 0)


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
def test_no_room_for_the_kept_values(gpu_lib, room, monkeypatch, form):
    n, d, v = 512, 320, 131072   # 268 MB of values, 134 MB of dl
    h, w, markov, u, slots = synthetic.head_inputs(n, d, v, 7700, DEV, ragged=True)
    factors = synthetic.markov_factors(n, v, 64, 7701, DEV)
    want = _step((h, w, markov, u, slots, head.MarkovFactors(*factors)), form)
    # each in memory of its own: nothing larger is left free within what is reserved
    torch.cuda.empty_cache()
    h, w, markov, u, want, factors = [t.clone() if torch.is_tensor(t) else [x.clone() for x in t]
                                      for t in (h, w, markov, u, want, factors)]
    kinds, workspace = [], _lib.workspace
    monkeypatch.setattr(_lib, "workspace", lambda kind, *a, **kw: kinds.append(kind) or workspace(kind, *a, **kw))
    # room for dl of all rows and the compact one, dh's partials and 40 MB of small blocks (the segments
    # of 20 MB that they come in): with the compact dl alone allocated 216 MB are left, not the
    # 268 MB of the values
    assert gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD, n, v, d) > 4 * n * v
    dl, partials = 2 * n * v, gpu_lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_BWD, n, v, d)
    assert dl + partials + (40 << 20) < 4 * n * v
    room((dl + dl * 5 // 8 if form == "skip" else dl) + partials + (40 << 20))
    got = _step((h, w, markov, u, slots, head.MarkovFactors(*factors)), form)
    assert _lib.NS_WS_LMHEAD_MIN in kinds
    for a, b in zip(want, got):
        assert torch.equal(a, b)


def test_workspace_without_a_smaller_one_raises(gpu_lib, room):
    room(16 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        _lib.workspace(_lib.NS_WS_LMHEAD, 512, 131072, 320, torch.device(DEV))
