"""The forward that leaves its intermediates for the backward (sfm_monarch_fwd_kept, sfm_monarch_attn_with_kv_cache_kept,
sfm_monarch_bwd_kept) against the chain that forms them again: the same kernels on the same numbers, so the same bits.  The
autograd tests of the operators hold this path to the oracle."""
import ctypes as C

import pytest
import torch

import self_forcing_amd as sfa
from gpu_util import randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
mattn, L = sfa.monarch_attn, sfa.lib


def holding(budget):
    return budget.left < 2 << 30


# rows per column just below, at and above whole chunks of 32, one and two key tiles, one to three query tiles, head_dim 64 / 128
@pytest.mark.parametrize("tiling,Fq,Fk,H,D,causal", [
    ((1, 1, 1, 1, 5), 1, 1, 1, 64, 0), ((1, 1, 1, 4, 8), 2, 8, 3, 128, 0), ((1, 1, 1, 31, 1), 1, 1, 2, 64, 0),
    ((1, 1, 1, 11, 52), 3, 3, 2, 128, 0), ((1, 1, 1, 30, 52), 3, 6, 2, 128, 0), ((1, 2, 1, 8, 33), 1, 4, 2, 64, 0),
    ((3, 1, 2, 7, 64), 3, 6, 1, 128, 0), ((3, 1, 1, 13, 20), 3, 3, 2, 64, 0), ((1, 1, 1, 90, 8), 1, 2, 2, 128, 0),
    ((1, 2, 1, 4, 60), 9, 9, 1, 128, 6), ((1, 1, 1, 3, 43), 12, 2, 2, 64, 0),      # 1080 and 516 (a, j) columns
    ((1, 1, 1, 5, 20), 6, 6, 2, 128, 2), ((3, 1, 1, 12, 16), 6, 6, 2, 64, 1),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kept_intermediates_give_the_bits_of_the_recomputed_ones(tiling, Fq, Fk, H, D, causal, dtype):
    f_tied, hr, wr, h, w = tiling
    q, do = (randn((2, Fq * h * w, H, D), 500 + i, dtype).to(DEV) for i in range(2))
    k, v = (randn((2, Fk * h * w, H, D), 502 + i, dtype).to(DEV) for i in range(2))
    sc = D ** -0.5
    out, stats = mattn._monarch_fwd_stats(q, k, v, tiling, sc, 0, causal)
    d = mattn._desc(q, k, v, out, *tiling, sc, 0, causal)
    n = C.c_size_t(0)
    L.check(L.load().sfm_monarch_kept_bytes(C.byref(d), C.byref(n)))
    assert n.value > 0
    kept = torch.full((n.value + 4096,), 0xAB, dtype=torch.uint8, device=DEV)
    out2, stats2 = torch.empty_like(out), torch.empty_like(stats)
    args = (C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), out2.data_ptr(), stats2.data_ptr(), kept.data_ptr())
    assert L.load().sfm_monarch_fwd_kept(*args, n.value - 1, None) == -6
    L.check(L.load().sfm_monarch_fwd_kept(*args, n.value, mattn._stream(q)))
    assert torch.equal(out, out2) and bool((kept[n.value:] == 0xAB).all())
    want = mattn._monarch_bwd(q, k, v, do, tiling, sc, 0, causal, out=out, stats=stats)
    want = (want[0].to(dtype), *want[1:])                      # one rounding of the same sum
    before = kept.clone()
    for _ in range(2):                                        # only read: a second backward finds the same
        got = mattn._monarch_bwd(q, k, v, do, tiling, sc, 0, causal, out=out2, stats=stats2, kept=kept[:n.value])
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert torch.equal(kept, before)


@pytest.mark.parametrize("start", [0, 3])
def test_kept_with_a_new_chunk_and_in_several_passes(start):
    """The cache call keeps what a call on the written cache does; a backward with room for one unit runs in passes."""
    h, w, H, D, dtype = 9, 24, 3, 128, torch.bfloat16
    per, tiling, sc = h * w, (1, 1, 1, 9, 24), 128 ** -0.5
    q, do, nk, nv = (randn((1, 3 * per, H, D), 510 + i, dtype).to(DEV) for i in range(4))
    kc, vc = (randn((1, 6 * per, H, D), 514 + i, dtype).to(DEV) for i in range(2))
    out, stats, kept = mattn._monarch_fwd_kept(q, kc, vc, tiling, sc, 1, 0, new=(nk, nv, start * per, (start + 3) * per))
    assert kept is not None and torch.equal(kc[:, start * per:(start + 3) * per], nk)
    want = mattn._monarch_bwd(q, kc, vc, do, tiling, sc, 1, 0, start, start + 3)
    got = mattn._monarch_bwd(q, kc, vc, do, tiling, sc, 1, 0, start, start + 3, out=out, stats=stats, kept=kept)
    for a, b in zip(got, want):                                # `want` sums the left factor's statistics itself
        torch.testing.assert_close(a.float(), b.float(), atol=2e-2, rtol=2e-2)
    bd = L.MonarchBwdDesc()
    dq, dk, dv = (torch.empty_like(t) for t in got)
    bd.fwd = mattn._desc(q, kc, vc, do, *tiling, sc, 1, 0)
    bd.dq_stride, bd.dkv_stride = L.strides3(dq), L.strides3(dk)
    bd.kv_grad_frame_start, bd.kv_grad_frame_end = start, start + 3
    n = C.c_size_t(0)
    L.check(L.load().sfm_monarch_bwd_kept_workspace_bytes(C.byref(bd), C.byref(n)))
    ws = torch.empty(n.value // 2, dtype=torch.uint8, device=DEV)       # one or two of the three units
    L.check(L.load().sfm_monarch_bwd_kept(C.byref(bd), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), stats.data_ptr(),
                                          kept.data_ptr(), kept.numel(), do.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                          ws.data_ptr(), ws.numel(), mattn._stream(q)))
    assert all(torch.equal(a, b) for a, b in zip((dq, dk, dv), got))


def test_what_is_kept_is_bounded_and_given_back(monkeypatch):
    h, w, H, D, dtype = 6, 20, 2, 64, torch.bfloat16
    q, k, v, do = (randn((1, 3 * h * w, H, D), 520 + i, dtype).to(DEV) for i in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]

    def forward():
        return mattn.monarch_attn(q, k, v, 1, 1, 1, h, w)

    forward()
    budget = mattn._KEPT[torch.cuda.current_device()]
    full = budget.left
    out = forward()
    size = full - budget.left
    assert size > 0
    want = torch.autograd.grad(out, leaves, do)
    assert budget.left == full
    out = forward()
    del out
    assert budget.left == full
    # no room: the backward forms the intermediates again
    monkeypatch.setattr(budget, "left", size - 1)
    got = torch.autograd.grad(forward(), leaves, do)
    assert budget.left == size - 1 and all(torch.equal(a, b) for a, b in zip(got, want))
    monkeypatch.setattr(budget, "left", full)
    # hooks on saved tensors see the small ones only
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.numel()) or t, lambda t: t):
        got = torch.autograd.grad(forward(), leaves, do)
    assert budget.left == full and max(seen) <= q.numel() and all(torch.equal(a, b) for a, b in zip(got, want))
    # another implementation than the forward ran with
    out = forward()
    old = L.load().sfm_set_switches(L.SW_BWD_SIMT)
    try:
        got = torch.autograd.grad(out, leaves, do)
    finally:
        L.load().sfm_set_switches(old)
    for a, b in zip(got, want):
        torch.testing.assert_close(a.float(), b.float(), atol=1e-2, rtol=1e-2)


def test_the_newest_forward_alone_holds_its_intermediates():
    """Layers whose backwards come later hold one buffer between them, not one each: the others' backwards, a second one of a
    retained graph and one whose buffer made room for a larger workspace form the intermediates again, with the same bits."""
    h, w, H, D, dtype = 6, 20, 2, 64, torch.bfloat16
    q, k, v, do = (randn((1, 3 * h * w, H, D), 530 + i, dtype).to(DEV) for i in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]

    def forward(**kw):
        return mattn.monarch_attn(q, k, v, 1, 1, 1, h, w, **kw)

    want = torch.autograd.grad(forward(heads_per_pass=H), leaves, do)
    first = forward()
    budget = mattn._KEPT[torch.cuda.current_device()]
    left = budget.left
    assert holding(budget)
    second = forward()
    assert budget.left == left and holding(budget)
    forward(heads_per_pass=H)                                       # holds none, and leaves the newest that does its own
    assert budget.left == left
    for _ in range(2):
        got = torch.autograd.grad(second, leaves, do, retain_graph=True)
        assert not holding(budget) and all(torch.equal(a, b) for a, b in zip(got, want))
    held = forward()
    assert holding(budget)
    got = torch.autograd.grad(first, leaves, do)                    # its workspace is the larger one
    assert not holding(budget) and all(torch.equal(a, b) for a, b in zip(got, want))
    got = torch.autograd.grad(held, leaves, do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    held = forward()
    key = (torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
    mattn.scratch(mattn._SCRATCH[key].numel() + 1, q.device)
    assert not holding(budget)
    got = torch.autograd.grad(held, leaves, do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    layers = [forward() for _ in range(6)]
    assert holding(budget) or budget.unused > 1
    for o in reversed(layers):
        got = torch.autograd.grad(o, leaves, do)
        assert not holding(budget) and all(torch.equal(a, b) for a, b in zip(got, want))


def test_forward_and_backward_in_turn_take_no_more_memory_than_without_what_is_kept(monkeypatch):
    h, w, H, D, dtype = 30, 52, 4, 128, torch.bfloat16
    q, k, v, do = (randn((1, 3 * h * w, H, D), 540 + i, dtype).to(DEV) for i in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]

    def peak():
        mattn.release_scratch()
        torch.cuda.empty_cache()
        for i in range(3):
            if i == 1:                                              # the first pass allocates the workspace
                torch.cuda.reset_peak_memory_stats()
            out = mattn.monarch_attn(q, k, v, 1, 1, 1, h, w)
            torch.autograd.grad(out, leaves, do)
            del out
        return torch.cuda.max_memory_allocated()

    kept = peak()
    monkeypatch.setattr(mattn, "_kept_buffer", lambda *a: None)
    assert kept <= peak() + (2 << 20)                               # allocations are rounded up to 512 bytes and more


@pytest.mark.parametrize("writer", ["kv_cache_write", "operator", "operator_static", "operator_under_autograd", "dense", "prologue"])
def test_cache_rows_written_before_the_backward_are_what_it_computes_with(writer):
    """The caches are saved by reference: a call that writes rows between forward and backward makes the backward form all of its
    intermediates from the new ones, as one does whose forward held none."""
    h, w, H, D, dtype = 6, 20, 2, 64, torch.bfloat16
    per, tiling = h * w, (1, 1, 1, 6, 20)
    q, do, nk, nv, other_k, other_v = (randn((1, 3 * per, H, D), 550 + i, dtype).to(DEV) for i in range(6))
    caches = [randn((1, 6 * per, H, D), 556 + i, dtype).to(DEV) for i in range(2)]
    leaves = [t.requires_grad_(True) for t in (q, nk, nv)]
    ones, rope = torch.ones(H * D, dtype=dtype, device=DEV), sfa.prologue.rope_table(D, device=DEV)
    flat = [t.detach().reshape(1, 3 * per, H * D) for t in (q, other_k, other_v)]

    def write(kc, vc):
        rows = (other_k, other_v, 3 * per, 6 * per)
        if writer == "operator_under_autograd":
            return mattn.monarch_attn_with_kv_cache(q, kc, vc, *rows, *tiling, heads_per_pass=H)
        with torch.no_grad():
            if writer == "kv_cache_write":
                mattn.kv_cache_write(*rows[:2], kc, vc, *rows[2:], *tiling)
            elif writer == "operator":
                mattn.monarch_attn_with_kv_cache(q, kc, vc, *rows, *tiling)
            elif writer == "operator_static":
                mattn.monarch_attn_with_kv_cache_static(q, kc, vc, *rows, *tiling)
            elif writer == "dense":
                sfa.attention.full_attention_with_kv_cache(q, kc, vc, *rows)
            else:
                sfa.prologue.qk_prologue(*flat, ones, ones, H, (3, h, w), 3, rope, kc, vc, 3 * per)

    def grads(overwrite, **kw):
        kc, vc = (t.clone() for t in caches)
        out = mattn.monarch_attn_with_kv_cache(q, kc, vc, nk, nv, 3 * per, 6 * per, *tiling, grad_only_new_kv=True, **kw)
        if overwrite:
            write(kc, vc)
        return torch.autograd.grad(out, leaves, do)

    plain, want = grads(False), grads(True, heads_per_pass=H)
    assert not torch.equal(plain[0], want[0])
    for got in (grads(True), grads(True)):
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(torch.equal(a, b) for a, b in zip(grads(False), plain))


def test_forwards_that_get_no_backward_stop_leaving_anything():
    h, w, H, D, dtype = 6, 20, 2, 64, torch.bfloat16
    q, k, v, do = (randn((1, 3 * h * w, H, D), 570 + i, dtype).to(DEV) for i in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]

    def forward():
        return mattn.monarch_attn(q, k, v, 1, 1, 1, h, w)

    def backward(out):
        return torch.autograd.grad(out, leaves, do)

    def leaves_something(out):
        return holding(budget)

    want = backward(forward())
    budget = mattn._KEPT[torch.cuda.current_device()]
    backward(forward())
    assert all(leaves_something(forward()) for _ in range(2))       # their graphs die here
    assert not any(leaves_something(forward()) for _ in range(3))
    out = forward()
    assert not leaves_something(out)
    assert all(torch.equal(a, b) for a, b in zip(backward(out), want))      # it would have found its own
    out = forward()
    assert leaves_something(out) and all(torch.equal(a, b) for a, b in zip(backward(out), want))
    layers = [forward() for _ in range(5)]                          # each makes room for the next
    assert not leaves_something(layers)
    backward(layers[0])                                             # would not
    assert not leaves_something(forward())


@pytest.mark.parametrize("tiling,D", [((1, 1, 1, 9, 24), 128), ((3, 1, 1, 12, 16), 64), ((1, 2, 1, 8, 33), 128)])
def test_kept_intermediates_of_strided_tensors(tiling, D):
    """q out of a fused projection, the new chunk too, caches that are some rows and heads of larger ones, a gradient with another
    order: the bits of the path that keeps nothing, and of contiguous tensors."""
    f_tied, hr, wr, h, w = tiling
    per, H, B, dtype = h * w, 3, 2, torch.bfloat16
    qkv = randn((B, 3 * per, 3, H, D), 580, dtype).to(DEV)
    q, nk, nv = qkv.unbind(2)
    big_k, big_v = (randn((B, 11 * per, H + 2, D), 581 + i, dtype).to(DEV) for i in range(2))
    do = randn((B, H, 3 * per, D), 583, dtype).to(DEV).transpose(1, 2)
    grads = []
    for kw in ({}, dict(heads_per_pass=B * H)):
        for dense in (False, True):
            ql, nkl, nvl = (t.detach().clone(memory_format=torch.contiguous_format) if dense else t.detach() for t in (q, nk, nv))
            assert dense or not ql.is_contiguous()
            kc, vc = (t.clone()[:, 2 * per:8 * per, 1:H + 1] for t in (big_k, big_v))
            kc, vc = (t.contiguous() if dense else t for t in (kc, vc))
            leaves = [t.requires_grad_(True) for t in (ql, nkl, nvl)]
            out = mattn.monarch_attn_with_kv_cache(ql, kc, vc, nkl, nvl, 3 * per, 6 * per, *tiling, grad_only_new_kv=True, **kw)
            assert holding(mattn._KEPT[torch.cuda.current_device()]) != bool(kw)
            grads.append((out, *torch.autograd.grad(out, leaves, do)))
    for g in grads[1:]:
        assert all(torch.equal(a, b) for a, b in zip(grads[0], g))
