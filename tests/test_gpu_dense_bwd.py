"""Backward of the dense attention operators (sfm_dense_bwd through the autograd functions) against torch autograd
through the float64 oracle.  The oracle's dense attention is a plain softmax(q k^T s) v in torch (oracle/dense.py),
pinned by the golden vectors and closed forms of tests/test_oracle_dense_prologue.py; its autograd gradient is the
mathematical one."""
import ctypes as C

import pytest
import torch

import self_forcing_amd as sfa
from gpu_util import randn
from oracle import dense

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _leaf(t, dev=None):
    t = t.clone().detach()
    if dev:
        t = t.to(dev)
    return t.requires_grad_(True)


def _close(got, ref, dtype):
    got, ref = got.detach().float().cpu(), ref.detach().float()
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-3
    # 16-bit gradients are rounded once at the end; accumulation is fp32
    assert torch.allclose(got, ref, atol=tol * max(1.0, ref.abs().max().item()), rtol=tol)


@pytest.mark.parametrize("dtype,B,Lq,Lk,H,D", [
    (torch.bfloat16, 1, 128, 64, 1, 128),          # one workgroup of each kernel, one tile
    (torch.bfloat16, 2, 200, 333, 3, 128),         # ragged in both directions, several tiles
    (torch.float16, 1, 70, 130, 2, 64),
    (torch.bfloat16, 1, 1560, 4680, 2, 128),       # a frame of queries against three frames of keys (480p grid)
])
def test_dense_gradients(dtype, B, Lq, Lk, H, D):
    q0, do = (randn((B, Lq, H, D), 200 + i, dtype) for i in range(2))
    k0, v0 = (randn((B, Lk, H, D), 202 + i, dtype) for i in range(2))
    qr, kr, vr = _leaf(q0.double()), _leaf(k0.double()), _leaf(v0.double())
    dense.attention(qr, kr, vr).backward(do.double())
    qd, kd, vd = _leaf(q0, DEV), _leaf(k0, DEV), _leaf(v0, DEV)
    out = sfa.attention.attention(qd, kd, vd, dtype=dtype)
    out.backward(do.to(DEV))
    _close(qd.grad, qr.grad, dtype)
    _close(kd.grad, kr.grad, dtype)
    _close(vd.grad, vr.grad, dtype)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [1, 32, 33, 64, 65, 97, 128, 161, 192, 257])
def test_dense_gradients_around_the_halves_of_a_tile(Lq, D):
    """The keys' gradients take the queries 32 at a time in a pipeline over tiles of 64: one, two and more tiles, the last of them
    one query, a half, a half and one query, or whole."""
    dtype = torch.bfloat16
    q0, do = (randn((1, Lq, 2, D), 300 + Lq + i, dtype) for i in range(2))
    k0, v0 = (randn((1, 150, 2, D), 302 + Lq + i, dtype) for i in range(2))
    qr, kr, vr = _leaf(q0.double()), _leaf(k0.double()), _leaf(v0.double())
    dense.attention(qr, kr, vr).backward(do.double())
    qd, kd, vd = _leaf(q0, DEV), _leaf(k0, DEV), _leaf(v0, DEV)
    sfa.attention.attention(qd, kd, vd, dtype=dtype).backward(do.to(DEV))
    _close(qd.grad, qr.grad, dtype)
    _close(kd.grad, kr.grad, dtype)
    _close(vd.grad, vr.grad, dtype)


@pytest.mark.parametrize("partial", [False, True])
def test_dense_kv_cache_gradients(partial):
    """q against a cache of 5 x 48 keys of which keys 96..192 arrive with the call; partial = grad_only_new_kv."""
    dtype, H, D = torch.bfloat16, 2, 64
    q0, do = (randn((1, 100, H, D), 210 + i, dtype) for i in range(2))
    k_old, v_old = (randn((1, 240, H, D), 212 + i, dtype) for i in range(2))
    k_new, v_new = (randn((1, 96, H, D), 214 + i, dtype) for i in range(2))
    qr, kor, vor, knr, vnr = (_leaf(t.double()) for t in (q0, k_old, v_old, k_new, v_new))
    kfull = torch.cat([kor[:, :96], knr, kor[:, 192:]], 1)
    vfull = torch.cat([vor[:, :96], vnr, vor[:, 192:]], 1)
    dense.attention(qr, kfull, vfull).backward(do.double())

    qd, knd, vnd = _leaf(q0, DEV), _leaf(k_new, DEV), _leaf(v_new, DEV)
    kc, vc = k_old.to(DEV).clone(), v_old.to(DEV).clone()
    kc.requires_grad_(not partial)
    vc.requires_grad_(not partial)
    out = sfa.attention.full_attention_with_kv_cache(qd, kc, vc, knd, vnd, 96, 192, grad_only_new_kv=partial)
    out.backward(do.to(DEV))
    _close(qd.grad, qr.grad, dtype)
    _close(knd.grad, knr.grad, dtype)
    _close(vnd.grad, vnr.grad, dtype)
    if not partial:
        # rows 96..192 of the cache gradient belong to the keys written by the call
        keep = torch.ones(240, dtype=torch.bool)
        keep[96:192] = False
        _close(kc.grad[:, keep], kor.grad[:, keep], dtype)
        _close(vc.grad[:, keep], vor.grad[:, keep], dtype)
    else:
        assert kc.grad is None and vc.grad is None


def test_dense_backward_argument_checks():
    q = randn((1, 64, 1, 32), 220, torch.bfloat16).to(DEV).requires_grad_(True)      # head_dim 32: forward only
    out = sfa.attention.attention(q, q, q)
    with pytest.raises(Exception):
        out.sum().backward()


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("B,H,Lq,Lk,kv0,grids", [              # grids that are split on 256 compute units
    (1, 1, 1, 64, 0, ""),              # one tile on either side: nothing to split
    (1, 1, 130, 4001, 0, "dq"),        # two query blocks against 63 key tiles; ragged last tile in the last range
    (2, 3, 2001, 100, 0, "dkv"),       # one key block per head against 32 query tiles
    (1, 5, 3000, 6600, 0, "dq dkv"),   # 260 key blocks: one whole round of 256 compute units and four blocks of a second
    (1, 7, 700, 2500, 1801, "dq"),     # gradients of the last keys only, from an odd key on
    (1, 1, 3000, 300, 1, "dkv"),       # the same with those of the keys in ranges
    (1, 2, 500, 900, 900, "dq"),       # dq only
    (1, 40, 1700, 1290, 1290, "dq"),   # dq only: 560 query blocks, 512 in the whole round and 48 in ranges
])
def test_last_round_split_into_ranges(B, H, Lq, Lk, kv0, grids, D, dtype):
    """sfm_dense_bwd with the queried workspace, which lets the last round's workgroups be split, and with the smallest one,
    which does not: the split gradients are as close to float64 as the unsplit ones, and nothing is written behind the
    workspace."""
    q, do = (randn((B, Lq, H, D), 600 + i, dtype).to(DEV) for i in range(2))
    k, v = (randn((B, Lk, H, D), 602 + i, dtype).to(DEV) for i in range(2))
    s = D ** -0.5
    out, lse = sfa.attention.attention(q, k, v, return_lse=True)
    lib, stream = sfa.lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    got = []
    for smallest in (False, True):
        dq = torch.full((B, Lq, H, D), float("nan"), device=DEV)
        dk, dv = (torch.full((B, Lk - kv0, H, D), float("nan"), dtype=dtype, device=DEV) for _ in range(2))
        bd = sfa.lib.DenseBwdDesc()
        bd.fwd = sfa.attention._dense_desc(q, k, v, out, s)
        bd.dq_stride, bd.dkv_stride = sfa.lib.strides3(dq), sfa.lib.strides3(dk)
        bd.kv_grad_start, bd.kv_grad_end = kv0, Lk
        n = C.c_size_t(0)
        sfa.lib.check(lib.sfm_dense_bwd_workspace_bytes(C.byref(bd), C.byref(n)))
        nbytes = 2 * B * H * Lq * 4 if smallest else n.value
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert (n.value > (2 * B * H * Lq * 4 + 255) // 256 * 256) == bool(grids)
        ws = torch.full((nbytes + 1024,), 0x5a, dtype=torch.uint8, device=DEV)
        sfa.lib.check(lib.sfm_dense_bwd(C.byref(bd), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(), do.data_ptr(),
                                        dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), nbytes, stream))
        assert bool((ws[nbytes:] == 0x5a).all())
        got.append((dq, dk, dv))
    f = lambda t, b, h: t[b, :, h].double()
    num, den = torch.zeros(2, 3), torch.zeros(3)
    for b in range(B):
        for h in range(H):
            p = torch.softmax(f(q, b, h) @ f(k, b, h).T.contiguous() * s, -1)
            dp = f(do, b, h) @ f(v, b, h).T.contiguous()
            ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * s
            ref = (ds @ f(k, b, h), (ds.T.contiguous() @ f(q, b, h))[kv0:], (p.T.contiguous() @ f(do, b, h))[kv0:])
            for x, r in enumerate(ref):
                den[x] += r.square().sum().cpu()
                for y in range(2):
                    num[y, x] += (f(got[y][x], b, h) - r).square().sum().cpu()
    # P, dS and a 16-bit gradient are rounded once each, delta comes from a rounded output: two units of the last place
    unit = 2 ** -7 if dtype == torch.bfloat16 else 2 ** -10
    for x in range(3 if Lk > kv0 else 1):
        split, whole = ((num[y, x] / den[x]).sqrt() for y in range(2))
        assert split < unit and split < 1.02 * whole + 1e-6
