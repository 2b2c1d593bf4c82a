"""The fused forward's second pass over kept tile values (NS_WS_LMHEAD workspace) against the
second run of the GEMM it replaces (NS_WS_LMHEAD_MIN): metrics, row statistics and dl are the
same bits over every form of the teacher and the Markov head, at the edges of token and vocab
tiles, without dl, and over several windows of rows."""

import ctypes

import pytest
import torch

from nanospec_amd import _lib, synthetic
from nanospec_amd.objective import _slot_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _forward(lib, kind, h, w, u, slots, *, markov=None, factors=None, rows=None, lse=None, want_dl=True):
    n, d = h.shape
    v = w.shape[0]
    wts, y, valid, k = _slot_inputs(slots, n, torch.device(DEV))
    out = [torch.full((6,), float("nan"), device=DEV), torch.full((n, 8), float("nan"), device=DEV),
           torch.full((n, v), float("nan"), dtype=torch.bfloat16, device=DEV) if want_dl else None]
    targs = None
    if rows is not None or lse is not None:
        targs = ctypes.byref(_lib.TeacherArgs(_lib.ptr(rows), u.shape[0] if rows is not None else 0, _lib.ptr(lse)))
    ws = _lib.workspace(kind, n, v, d, torch.device(DEV))
    ws.fill_(0x7f)
    tail = (_lib.ptr(u), _lib.dtype_code(u), v, targs, _lib.ptr(y), _lib.ptr(wts), _lib.ptr(valid), n, d, v, k, 0.1,
            0.9, 0.5, _lib.ptr(out[2]), v, _lib.ptr(out[1]), _lib.ptr(out[0]), _lib.ptr(ws), ws.numel(),
            _lib.stream(torch.device(DEV)))
    if factors is None:
        status = lib.ns_lmhead_ce_kl_fwd(_lib.ptr(h), d, _lib.ptr(w), d, _lib.ptr(markov), v, *tail)
    else:
        prev, w1, w2 = factors
        r = w1.shape[1]
        status = lib.ns_lmhead_markov_ce_kl_fwd(_lib.ptr(h), d, _lib.ptr(w), d, _lib.ptr(prev), _lib.ptr(w1), r,
                                                _lib.ptr(w2), r, r, *tail)
    _lib.check(status, "forward")
    torch.cuda.synchronize()
    return out


def _assert_same(a, b):
    for x, y in zip(a, b):
        if x is not None:   # NaN patterns too
            assert torch.equal(x.view(torch.int16 if x.dtype == torch.bfloat16 else torch.int32),
                               y.view(torch.int16 if y.dtype == torch.bfloat16 else torch.int32))


@pytest.mark.parametrize("n,d,v", [(8, 64, 8), (40, 64, 264), (264, 128, 2056), (512, 192, 65536 + 136),
                                   (136, 320, 65536),
                                   # few rows and a large vocabulary: thin.hip's kernel for pass 1
                                   (8, 320, 8456), (40, 64, 9000), (64, 128, 16384), (128, 192, 131336),
                                   (96, 64, 131080)])
@pytest.mark.parametrize("form", ["rows", "gathered", "lse", "fp32", "fp32_lse", "factored", "no_dl"])
def test_kept_values_give_the_same_bits(gpu_lib, n, d, v, form):
    h, w, markov, u, slots = synthetic.head_inputs(n, d, v, 7000 + n, DEV, ragged=True)
    slots.target_ids[0, 0] = -100
    slots.target_ids[0, 1] = v - 1
    kw = {"markov": markov if n % 16 else None}
    if form.startswith("fp32"):
        u = u.float()
    if form.endswith("lse"):
        kw["lse"] = torch.logsumexp(u.double(), -1).float()
    if form == "gathered":
        u = torch.cat([u, u[: n // 2].flip(0)]).contiguous()
        kw["rows"] = torch.randint(0, u.shape[0], (n,), device=DEV)
        kw["rows"][n // 3] = u.shape[0]       # outside: that row's teacher is NaN
    if form == "factored":
        prev, w1, w2 = synthetic.markov_factors(n, v, 64, 7100 + n, DEV)
        prev[n // 2] = v                      # outside: that row's logits are NaN
        kw = {"factors": (prev, w1, w2)}
    kw["want_dl"] = form != "no_dl"
    lib = gpu_lib
    assert lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD, n, v, d) > lib.ns_workspace_bytes(_lib.NS_WS_LMHEAD_MIN, n, v, d)
    _assert_same(_forward(lib, _lib.NS_WS_LMHEAD, h, w, u, slots, **kw),
                 _forward(lib, _lib.NS_WS_LMHEAD_MIN, h, w, u, slots, **kw))


def test_several_windows_of_rows(gpu_lib):
    """V = 2^21 keeps 256 rows' values in a window: 520 rows are three windows.  The same bits as
    the GEMM run again, and every row's log-normalisers within 1e-5 of fp64's."""
    n, d, v = 520, 320, 1 << 21
    h, w, _, u, slots = synthetic.head_inputs(n, d, v, 7300, DEV, ragged=True)
    a = _forward(gpu_lib, _lib.NS_WS_LMHEAD, h, w, u, slots)
    b = _forward(gpu_lib, _lib.NS_WS_LMHEAD_MIN, h, w, u, slots)
    _assert_same(a, b)
    stats = a[1]
    for r in (0, 255, 256, 511, 512, 519):
        z = torch.cat([h[r].double() @ c.double().t() for c in w.split(1 << 18)])
        lz, lu = torch.logsumexp(z, -1), torch.logsumexp(u[r].double(), -1)
        assert abs(float(stats[r, 0] - lz)) < 1e-5 * abs(float(lz))
        assert abs(float(stats[r, 1] - lu)) < 1e-5 * abs(float(lu))
        p, t = (z - lz).exp(), (u[r].double() - lu).exp()
        assert float(stats[r, 4]) == pytest.approx(float(torch.minimum(p, t).sum()), rel=1e-4)


@pytest.mark.parametrize("kind", [_lib.NS_WS_LMHEAD, _lib.NS_WS_LMHEAD_MIN])
@pytest.mark.parametrize("form", ["dense", "gathered", "lse", "fp32", "fp32_lse", "factored", "no_dl"])
def test_each_window_is_a_call_of_its_rows(gpu_lib, form, kind):
    """Every operand moves on with the window: three windows of 256, 256 and 8 rows (V = 2^21) give the
    row statistics and dl of three calls on those rows, bit for bit."""
    n, d, v, step = 520, 320, 1 << 21, 256
    h, w, markov, u, slots = synthetic.head_inputs(n, d, v, 7350, DEV, ragged=True)
    slots.target_ids[40, 3] = -100
    rows = lse = factors = None
    if form != "dense":
        markov = None
    if form.startswith("fp32"):
        u = u.float()
    if form.endswith("lse"):
        lse = torch.stack([torch.logsumexp(x.double(), -1) for x in u]).float()
    if form == "gathered":
        rows = torch.randint(0, n, (n,), device=DEV)
        rows[300] = n            # outside: that row's teacher is NaN
        rows[515] = -1
    if form == "factored":
        factors = synthetic.markov_factors(n, v, 64, 7351, DEV)
        factors[0][400] = v      # outside: that row's logits are NaN
    _, stats, dl = _forward(gpu_lib, kind, h, w, u, slots, markov=markov, factors=factors, rows=rows, lse=lse,
                            want_dl=form != "no_dl")
    for r0 in range(0, n, step):
        r = slice(r0, min(r0 + step, n))
        b = slice(r0 // 8, r.stop // 8)
        part = synthetic.Slots(slots.weights[b], slots.target_ids[b], slots.valid[b])
        _, s, x = _forward(gpu_lib, kind, h[r], w, u if rows is not None else u[r], part,
                           markov=None if markov is None else markov[r],
                           factors=None if factors is None else (factors[0][r], *factors[1:]),
                           rows=None if rows is None else rows[r], lse=None if lse is None else lse[r],
                           want_dl=form != "no_dl")
        _assert_same([stats[r], None if dl is None else dl[r]], [s, x])


@pytest.mark.parametrize("n", [1, 7, 32, 33, 64, 65, 100, 128])
@pytest.mark.parametrize("v,d", [(8, 64), (8456, 320), (131336, 128)])
def test_few_rows_projection(gpu_lib, n, v, d):
    """The projection of up to 128 rows (thin.hip) is that of the same rows in a larger batch, bit for
    bit, with an addend and with gathered rows (one out of range: NaN); its log-sum-exp that of the
    stored logits."""
    from nanospec_amd import head

    g = torch.Generator(device=DEV).manual_seed(7400 + n)
    x = torch.randn((300, d), generator=g, device=DEV).bfloat16()
    w = (0.05 * torch.randn((v, d), generator=g, device=DEV)).bfloat16()
    add = torch.randn((300, v), generator=g, device=DEV).bfloat16()
    whole = head.lm_head_linear(x, w)
    assert torch.equal(head.lm_head_linear(x[:n], w), whole[:n])
    assert torch.equal(head.lm_head_linear(x[:n], w, add[:n]), head.lm_head_linear(x, w, add)[:n])
    rows = torch.randint(0, 300, (n,), generator=g, device=DEV)
    t = head.teacher_logits(x, w, rows)
    assert torch.equal(t.logits, whole[rows])
    want = torch.logsumexp(t.logits.double(), -1)
    assert float(((t.lse.double() - want) / want).abs().max()) < 2e-6
    rows[n // 2] = 300
    t = head.teacher_logits(x, w, rows)
    assert torch.isnan(t.logits[n // 2]).all() and torch.isnan(t.lse[n // 2])
    keep = torch.arange(n, device=DEV) != n // 2
    assert torch.equal(t.logits[keep], whole[rows[keep]]) and bool(torch.isfinite(t.lse[keep]).all())


@pytest.mark.parametrize("v", [81912, 81920, 84008])   # d = 2048: below, at and past 320 MiB of W
@pytest.mark.parametrize("n", [8, 64])
def test_few_rows_with_workgroups_started_apart(gpu_lib, n, v):
    """Whether the workgroups start apart (W's pitch a multiple of 4 KB, and W larger than the caches)
    changes no bit of the projection."""
    from nanospec_amd import head

    g = torch.Generator(device=DEV).manual_seed(7500 + n)
    x = torch.randn((200, 2048), generator=g, device=DEV).bfloat16()
    w = (0.05 * torch.randn((v, 2048), generator=g, device=DEV)).bfloat16()
    assert torch.equal(head.lm_head_linear(x[:n], w), head.lm_head_linear(x, w)[:n])


def test_windows_only_where_values_are_kept(gpu_lib):
    """Three windows of rows (V = 2^21) at a d whose values pass 2 reads; one launch of each pass where
    they are not kept, and of pass 2 alone."""
    from nanospec_amd import head
    from nanospec_amd.config import Objective

    n, v = 520, 1 << 21
    for d, windows in ((320, 3), (64, 1)):
        h, w, _, u, slots = synthetic.head_inputs(n, d, v, 7600 + d, DEV, ragged=True)
        with _lib.KernelTimer() as t:
            _, saved = head.lm_head_ce_kl_loss(h, w, u, slots, Objective(block_size=8), emit_dlogits=False)
            torch.cuda.synchronize()
        assert t.times["head_stats"][0] == windows and t.times["head_emit"][0] == windows
        with _lib.KernelTimer() as t:
            head._reemit_dlogits(saved, 1)
            torch.cuda.synchronize()
        assert t.times["head_emit"][0] == 1
