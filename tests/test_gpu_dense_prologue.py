"""GPU parity of the dense-attention and fused-prologue kernels against the CPU oracle."""
import ctypes as C

import pytest
import torch

import self_forcing_amd as sfa
from gpu_util import assert_close_16bit, max_abs, randn
from oracle import blocks, dense, monarch, prologue

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,Lq,Lk,H,D", [(1, 17, 13, 1, 32), (2, 31, 29, 3, 64), (2, 64, 48, 4, 64), (1, 300, 1000, 2, 128),
                                         (1, 129, 65, 2, 128)])
def test_dense_reference_shapes(dtype, B, Lq, Lk, H, D):
    """attn_patch.py:499-503 shapes plus ragged tiles of the MFMA kernel (128-query / 64-key tiles)."""
    q, k, v = randn((B, Lq, H, D), 1, dtype), randn((B, Lk, H, D), 2, dtype), randn((B, Lk, H, D), 3, dtype)
    ref, lse_ref = dense.attention(q, k, v, dtype=torch.float32, return_lse=True)
    out, lse = sfa.attention.attention(q.to(DEV), k.to(DEV), v.to(DEV), dtype=dtype, return_lse=True)
    if dtype == torch.float32:
        assert max_abs(out, ref) < 1e-5
    else:
        assert_close_16bit(out, ref, dtype)
    assert max_abs(lse, lse_ref) < 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Lq,Lk,H,D", [(1, 4200, 333, 8, 128), (2, 2100, 130, 8, 64), (1, 4680, 512, 12, 128)])
def test_dense_wide_workgroups(dtype, B, Lq, Lk, H, D):
    """Enough query blocks for the 256-query workgroups (8 waves): ragged last query block and last key tile, both head
    dims, and the cross-attention shape (4680 queries against 512 text tokens, 12 heads)."""
    q, k, v = randn((B, Lq, H, D), 21, dtype), randn((B, Lk, H, D), 22, dtype), randn((B, Lk, H, D), 23, dtype)
    ref, lse_ref = dense.attention(q, k, v, dtype=torch.float32, return_lse=True)
    out, lse = sfa.attention.attention(q.to(DEV), k.to(DEV), v.to(DEV), dtype=dtype, return_lse=True)
    assert_close_16bit(out, ref, dtype)
    assert max_abs(lse, lse_ref) < 1e-3


def test_attention_keeps_half_dtypes_and_returns_qs_dtype():
    """attention.py:62-70, 135-138: float16 / bfloat16 inputs are used as they are (not recast to the default
    bfloat16), anything else is computed in `dtype`; the result has q's original dtype."""
    q, k, v = (randn((1, n, 2, 64), 90 + i, torch.float32) for i, n in enumerate((33, 70, 70)))
    ref = dense.attention(q, k, v, dtype=torch.float64)
    o16 = sfa.attention.attention(q.half().to(DEV), k.half().to(DEV), v.half().to(DEV))
    assert o16.dtype == torch.float16
    assert max_abs(o16, dense.attention(q.half(), k.half(), v.half(), dtype=torch.float64)) < 2e-3       # fp16 bar, not bf16's
    o32 = sfa.attention.attention(q.to(DEV), k.to(DEV), v.to(DEV))
    assert o32.dtype == torch.float32 and max_abs(o32, ref) < 2e-2
    o32h = sfa.attention.attention(q.to(DEV), k.to(DEV), v.to(DEV), dtype=torch.float16)
    assert o32h.dtype == torch.float32 and max_abs(o32h, ref) < 2e-3


def test_dense_with_kv_cache_writes_in_token_order():
    dtype = torch.bfloat16
    q = randn((2, 40, 3, 64), 4, dtype)
    kc, vc = randn((2, 96, 3, 64), 5, dtype), randn((2, 96, 3, 64), 6, dtype)
    nk, nv = randn((2, 48, 3, 64), 7, dtype), randn((2, 48, 3, 64), 8, dtype)
    kd, vd = kc.to(DEV), vc.to(DEV)
    out = sfa.attention.full_attention_with_kv_cache(q.to(DEV), kd, vd, nk.to(DEV), nv.to(DEV), 48, 96)
    ref = dense.full_attention_with_kv_cache(q, kc, vc, nk, nv, 48, 96, dtype=torch.float32)
    assert torch.equal(kd.cpu(), kc) and torch.equal(vd.cpu(), vc)
    assert_close_16bit(out, ref, dtype)
    with pytest.raises(ValueError):
        sfa.attention.full_attention_with_kv_cache(q.to(DEV), kd, vd, nk.to(DEV), nv.to(DEV), 60, 108)


def test_dense_chunk_vs_cache_shape_two_heads():
    """One 3-frame chunk against a 6-frame cache at the 30 x 52 grid (2 heads to bound the oracle)."""
    dtype = torch.bfloat16
    q, k, v = randn((1, 4680, 2, 128), 9, dtype), randn((1, 9360, 2, 128), 10, dtype), randn((1, 9360, 2, 128), 11, dtype)
    ref = dense.attention(q, k, v, dtype=torch.float32)
    out = sfa.attention.attention(q.to(DEV), k.to(DEV), v.to(DEV))
    assert_close_16bit(out, ref, dtype)


def _ulp_report(got, ref):
    """(fraction of differing elements, max |diff| / max(|ref|, 1))."""
    g, r = got.float().cpu(), ref.float().cpu()
    diff = (g - r).abs()
    return (diff > 0).float().mean().item(), (diff / r.abs().clamp_min(1.0)).max().item()


@pytest.mark.parametrize("dtype,f_tied,h_reduce,w_reduce,F,h,w,H,D", [
    (torch.bfloat16, 1, 1, 1, 2, 4, 6, 2, 128),
    (torch.float32, 3, 2, 2, 3, 4, 6, 3, 64),
    (torch.float16, 1, 2, 3, 2, 6, 12, 4, 64),
    (torch.bfloat16, 1, 2, 1, 3, 30, 52, 12, 128),      # one 1.3B chunk, reduce2xh tiling
])
def test_prologue_vs_oracle(dtype, f_tied, h_reduce, w_reduce, F, h, w, H, D):
    """Cache placement is exact; V is copied bit for bit; q/k values agree with the oracle up to one
    rounding step of the tensor dtype on a small fraction of elements (the fp32 mean of squares is
    summed in a different order than torch's)."""
    B, S, Cd = 2, F * h * w, H * D
    xq, xk, xv = (randn((B, S, Cd), 20 + i, dtype) for i in range(3))
    wq, wk = (1 + 0.1 * randn((Cd,), 23, torch.float32)).to(dtype), (1 + 0.1 * randn((Cd,), 24, torch.float32)).to(dtype)
    start_frame, pre = 4, f_tied * h * w
    qr, kr, vr = prologue.qk_prologue(xq, xk, xv, wq, wk, H, (F, h, w), start_frame)
    kc = torch.zeros(B, pre + S + pre, H, D, dtype=dtype, device=DEV)
    vc = torch.zeros_like(kc)
    rope = sfa.prologue.rope_table(D, device=DEV)
    qo = sfa.prologue.qk_prologue(xq.to(DEV), xk.to(DEV), xv.to(DEV), wq.to(DEV), wk.to(DEV), H, (F, h, w), start_frame,
                                  rope, kc, vc, pre, f_tied, h_reduce, w_reduce)
    kref = blocks.to_blocks(kr, f_tied, h_reduce, w_reduce, h, w).reshape(B, S, H, D)
    vref = blocks.to_blocks(vr, f_tied, h_reduce, w_reduce, h, w).reshape(B, S, H, D)
    assert torch.equal(vc[:, pre:pre + S].cpu(), vref)
    assert (kc[:, :pre] == 0).all() and (kc[:, pre + S:] == 0).all() and (vc[:, :pre] == 0).all()
    one_step = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10, torch.float32: 2 ** -21}[dtype]
    for got, ref in ((qo, qr), (kc[:, pre:pre + S], kref)):
        frac, rel = _ulp_report(got, ref)
        assert rel <= 2 * one_step, rel
        if dtype != torch.float32:
            assert frac < 1e-3, frac


def test_prologue_then_monarch_c2_pipeline():
    """C2 as specified: activations ~ N(0,1) from seed 0 cast to bf16, RMSNorm (weight 1) + RoPE through the
    fused prologue, cache frames 0-17 filled chunk by chunk, new chunk at start_frame 18 (tokens
    28080..32760), then Monarch attention over the 21-frame cache.  Checked on 2 of 12 heads against the
    oracle chain (oracle prologue -> oracle Monarch), and reported against dense attention."""
    H, D, h, w = 12, 128, 30, 52
    Cd, S = H * D, 4680
    g = torch.Generator().manual_seed(0)
    xq = torch.randn(S, Cd, generator=g).to(torch.bfloat16)
    xk_new = torch.randn(S, Cd, generator=g).to(torch.bfloat16)
    xk_cache = torch.randn(28080, Cd, generator=g).to(torch.bfloat16)
    v_new = torch.randn(S, Cd, generator=g).to(torch.bfloat16)
    v_cache = torch.randn(28080, Cd, generator=g).to(torch.bfloat16)
    ones = torch.ones(Cd, dtype=torch.bfloat16)
    rope = sfa.prologue.rope_table(D, device=DEV)
    kc = torch.zeros(1, 32760, H, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    wd = ones.to(DEV)
    for c in range(6):
        xs = xk_cache[c * S:(c + 1) * S][None].to(DEV)
        vs = v_cache[c * S:(c + 1) * S][None].to(DEV)
        sfa.prologue.qk_prologue(xs, xs, vs, wd, wd, H, (3, h, w), 3 * c, rope, kc, vc, c * S)
    qd = sfa.prologue.qk_prologue(xq[None].to(DEV), xk_new[None].to(DEV), v_new[None].to(DEV), wd, wd, H, (3, h, w), 18,
                                  rope, kc, vc, 28080)
    out = sfa.monarch_attn.monarch_attn(qd, kc, vc, 1, 1, 1, h, w)
    # oracle chain on heads 3 and 8
    heads = [3, 8]
    k_all = torch.cat([xk_cache, xk_new])[None]
    v_all = torch.cat([v_cache, v_new])[None]
    q_o, _, _ = prologue.qk_prologue(xq[None], xq[None], xq[None], ones, ones, H, (3, h, w), 18)
    _, k_o, v_o = prologue.qk_prologue(k_all, k_all, v_all, ones, ones, H, (21, h, w), 0)
    assert (kc.cpu() != k_o).float().mean().item() < 1e-3 and torch.equal(vc.cpu(), v_o)
    ref = monarch.monarch_attn(q_o[:, :, heads], k_o[:, :, heads], v_o[:, :, heads], 1, 1, 1, h, w, dtype=torch.float32)
    assert_close_16bit(out[:, :, heads], ref, torch.bfloat16)
    dn = sfa.attention.attention(qd, kc, vc)
    print(f"C2 monarch vs dense: max-abs {max_abs(out, dn):.3e}")


@pytest.mark.gpu
def test_mfma_probe_reports_a_rate():
    import ctypes as C
    from self_forcing_amd import lib as L
    lib = L.load()
    out = C.c_float(0)
    L.check(lib.sfm_probe_mfma_bf16(2000, None, C.byref(out)))
    assert 10.0 < out.value < 5000.0       # TFLOP/s; the nominal peak is 2500


@pytest.mark.gpu
def test_row_stream_probe_reports_a_duration_and_leaves_the_rows_alone():
    import ctypes as C
    from self_forcing_amd import lib as L
    lib = L.load()
    waves, kb = 37, 19                                         # a workgroup with one wave, a last batch of 3 KB
    ws = torch.randint(0, 256, (2 * waves * kb * 1024,), dtype=torch.uint8, device="cuda")
    before = ws.clone()
    out = C.c_float(0)
    L.check(lib.sfm_probe_row_stream(waves, kb, ws.data_ptr(), ws.numel(), None, C.byref(out)))
    torch.cuda.synchronize()
    assert 0.1 < out.value < 1e5               # microseconds per pass
    assert torch.equal(ws, before)


@pytest.mark.gpu
def test_traffic_probe_moves_the_bytes_and_reports_a_duration():
    import ctypes as C
    from self_forcing_amd import lib as L
    lib = L.load()
    tiles, rows_in, rows_out, row_bytes = 300, 52, 156, 256
    nin = tiles * 2 * rows_in * row_bytes
    nout = tiles * rows_out * row_bytes
    for nt in (0, 1):
        ws = torch.zeros(nin + 2 * nout, dtype=torch.uint8, device="cuda")
        ws[:nin] = torch.randint(0, 256, (nin,), dtype=torch.uint8, device="cuda")
        ws[nin:] = 0xEE
        src = ws[:nin].clone()
        out = C.c_float(0)
        L.check(lib.sfm_probe_tile_traffic(tiles, rows_in, rows_out, row_bytes, nt, ws.data_ptr(), ws.numel(), None, C.byref(out)))
        torch.cuda.synchronize()
        assert 0.1 < out.value < 1e5           # microseconds per pass
        assert torch.equal(ws[:nin], src)      # the input region is only read
        o0 = ws[nin:nin + nout].view(rows_out, tiles, row_bytes // 16, 16)
        o1 = ws[nin + nout:].view(rows_out, tiles, row_bytes // 16, 16)
        assert torch.equal(o0, o1)
        # every 16-byte piece of item t holds the xor of the pieces one thread read: thread x reads pieces x, x + 320, ...
        pieces = src.view(tiles, 2 * rows_in * row_bytes // 16, 16)
        t = 7
        want = torch.zeros(320, 16, dtype=torch.uint8, device="cuda")
        for c0 in range(0, pieces.shape[1], 320):
            blk = pieces[t, c0:c0 + 320]
            want[:blk.shape[0]] ^= blk
        got = o0[:, t].reshape(-1, 16)          # piece c of the item's output comes from thread c % 320
        idx = torch.arange(got.shape[0], device="cuda") % 320
        assert torch.equal(got, want[idx])


# few queries against many keys are split over the keys: 2 to 64 ranges of four tiles or more, ragged last tiles, query blocks of
# one row up to two blocks; 16 heads x 2048 queries run the 256-query kernel in two ranges
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.bfloat16), (128, torch.float16), (64, torch.float16)])
@pytest.mark.parametrize("B,H,nq,nk", [(1, 1, 1, 960), (1, 1, 1, 1600), (1, 2, 129, 2049), (2, 3, 128, 2112), (1, 1, 64, 16384),
                                       (1, 1, 200, 16449), (1, 5, 255, 2500), (1, 16, 2048, 8000), (1, 25, 300, 5000)])
def test_queries_split_over_the_keys(B, H, nq, nk, D, dtype):
    q, k, v = (randn((B, n, H, D), 70 + i, dtype).to(DEV) for i, n in enumerate((nq, nk, nk)))
    lib = sfa.lib.load()
    out, lse = sfa.attention.attention(q, k, v, return_lse=True)
    n = C.c_size_t(0)
    d = sfa.attention._dense_desc(q, k, v, out, D ** -0.5)
    sfa.lib.check(lib.sfm_dense_workspace_bytes(C.byref(d), C.byref(n)))
    assert (n.value > 0) == (nk > 960)
    whole, wlse = torch.empty_like(out), torch.empty_like(lse)
    sfa.lib.check(lib.sfm_dense_fwd(C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), whole.data_ptr(), wlse.data_ptr(),
                                    C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    qd, kd, vd = (t.transpose(1, 2).double() for t in (q, k, v))
    ref, rl = torch.empty_like(qd), []
    for b in range(B):
        for h in range(H):
            z = qd[b, h] @ kd[b, h].T.contiguous() * D ** -0.5
            ref[b, h] = torch.softmax(z, -1) @ vd[b, h]
            rl.append(torch.logsumexp(z, -1))
    ref, rl = ref.transpose(1, 2), torch.stack(rl).reshape(B, H, nq)
    err = lambda x: ((x.double() - ref).norm() / ref.norm()).item()
    # one rounding of P and of the output each (2^-9 for bfloat16, rms about 0.4 of it); no worse than the unsplit kernel, up to four times the
    # spread 1 / sqrt(n) of the ratio of two such errors over n elements
    unit = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -11
    assert err(out) < unit and err(out) < (1.02 + 4 / ref.numel() ** 0.5) * err(whole)
    # float32 sums of nk terms around 1, logits of size about ten: 2^-24 (log2 nk + 10) rounded up
    assert (lse.double() - rl).abs().max() < 1e-5 and (wlse.double() - rl).abs().max() < 1e-5


# tiles of 64 keys with and without a ragged tail, one workgroup over all keys and split over the keys
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nk", [7, 64, 200, 256, 3000, 3072])
def test_logits_at_minus_infinity_and_at_the_lowest_floats(nk, D):
    """softmax as torch takes it: a key at -inf weighs nothing, a row of nothing but such keys is NaN, and a row whose logits are
    all alike is the mean of v however low they are.  Logits are the products with one element of k, exactly."""
    H, nq, ln2 = 2, 3, 0.6931471805599453          # sm_scale = ln 2: the kernel's base-2 factor is 1 and rounds nothing
    q = torch.zeros(1, nq, H, D, dtype=torch.bfloat16, device=DEV)
    q[..., 0] = 1
    k = torch.zeros(1, nk, H, D, dtype=torch.bfloat16, device=DEV)
    v = randn((1, nk, H, D), 81, torch.bfloat16).to(DEV)
    mean = v.double().mean(1, keepdim=True)

    def run(column):
        k[..., 0] = column
        return sfa.attention.attention(q, k, v, softmax_scale=ln2, return_lse=True)

    for low in (-2.0e30, -3.2e38):
        out, _ = run(low)
        assert ((out.double() - mean).abs().max() < 2 ** -8 * v.abs().max()), low
    out, lse = run(float("-inf"))
    assert bool(out.isnan().all()) and bool((lse == float("-inf")).all())
    column = torch.full((1, nk, 1), float("-inf"), device=DEV)
    column[:, nk // 2] = 3.0                          # one key of all has the whole weight, whichever tile or range it is in
    out, lse = run(column)
    assert torch.equal(out, v[:, nk // 2:nk // 2 + 1].expand_as(out))
    assert (lse - 3 * ln2).abs().max() < 1e-6
