"""Decode attention over short contexts (csrc/paged_attention.hip: one workgroup per sequence and kv head) and the stream with more workgroups than the
contexts have stages, against softmax attention in 64 bits."""
import ctypes

import pytest
import torch

from candle_vllm_amd._lib import lib

pytestmark = pytest.mark.gpu
BF16, PAGED = 2, 1


def cache(ctxs, G, D, bs, fp8, seed):
    """pages in random order, NaN wherever no token was written -> (k pages, v pages, block table, [keys, values] per sequence in f64)"""
    torch.manual_seed(seed)
    nb = [max(1, -(-c // bs)) for c in ctxs]
    x = 16 if fp8 else 8
    k = torch.full((sum(nb) + 2, G, D // x, bs, x), float("nan"), device="cuda")
    v = torch.full((sum(nb) + 2, G, D, bs), float("nan"), device="cuda")
    perm, at, kv = torch.randperm(sum(nb) + 2), 0, []
    bt = torch.zeros(len(ctxs), max(nb) + 1, dtype=torch.int32)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    for i, c in enumerate(ctxs):
        keys, vals = torch.randn(c, G, D, device="cuda").to(dt), torch.randn(c, G, D, device="cuda").to(dt)
        bt[i, :nb[i]] = perm[at:at + nb[i]]
        at += nb[i]
        t = torch.arange(c, device="cuda")
        blk = bt[i].cuda().long()[t // bs]
        k[blk, :, :, t % bs] = keys.float().view(c, G, D // x, x)
        v[blk, :, :, t % bs] = vals.float()
        kv.append((keys.double(), vals.double()))
    return k.to(dt), v.to(dt), bt.cuda(), kv


def reference(q, kv, scale, cap):
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for i, (k, v) in enumerate(kv):
        if k.shape[0] == 0:
            continue
        G = k.shape[1]
        s = torch.matmul(q[i].double().view(G, -1, q.shape[2]), k.permute(1, 2, 0).contiguous()) * scale
        if cap:
            s = torch.tanh(s / cap) * cap
        out[i] = torch.matmul(torch.softmax(s, -1), v.permute(1, 0, 2).contiguous()).view(q.shape[1:])
    return out


def attend(q, k, v, bt, ctxs, most, ps, bs, scale, cap, fp8, ks=1.0, vs=1.0):
    B, H, D = q.shape
    G = k.shape[1]
    P = max(1, -(-most // max(ps, 1)))
    out = torch.full((B, H, D), 7.0, dtype=torch.bfloat16, device="cuda")
    tmp, mx, sm = torch.full((B * H * P * D,), float("nan"), device="cuda"), torch.zeros(B * H * P, device="cuda"), torch.zeros(B * H * P, device="cuda")
    cl = torch.tensor(ctxs, dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    lib.mi355_clear_error()
    common = (B, H, G, D, bs, bt.shape[1], most)
    if fp8:
        rc = lib.mi355_paged_attention_fp8(out.data_ptr(), sm.data_ptr(), mx.data_ptr(), tmp.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), bt.data_ptr(), cl.data_ptr(),
                                           *common, ps, scale, cap, ks, vs, st)
    elif ps == 0:
        rc = lib.mi355_paged_attention_v1(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), bt.data_ptr(), cl.data_ptr(), *common, scale, cap, PAGED, BF16, st)
    else:
        rc = lib.mi355_paged_attention_v2(out.data_ptr(), sm.data_ptr(), mx.data_ptr(), tmp.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), bt.data_ptr(), cl.data_ptr(),
                                          *common, ps, scale, cap, PAGED, BF16, st)
    assert rc == 0
    torch.cuda.synchronize()
    return out


# lengths at the edges of a partition and of 4, 8 and 16 of them; groups of 1 to 16 heads (16 waves of 16 heads of 128 do not fit: the general kernel); blocks that
# hold a partition, two, or half of one
@pytest.mark.parametrize("H,G,D,bs", [(8, 8, 128, 64), (6, 2, 128, 16), (14, 2, 128, 32), (16, 2, 64, 16), (16, 1, 128, 64), (24, 8, 64, 48)])
@pytest.mark.parametrize("most", [1, 32, 33, 128, 150, 256, 257, 500, 512])
@pytest.mark.parametrize("fp8", [False, True])
def test_short_contexts(H, G, D, bs, most, fp8):
    ctxs = [most, 0, 1, max(1, most - 1), (most + 1) // 2, min(most, 31), min(most, 32), min(most, 65)]
    k, v, bt, kv = cache(ctxs, G, D, bs, fp8, most + H)
    q = torch.randn(len(ctxs), H, D, device="cuda").bfloat16()
    for ps in (0, 32):
        for cap, scale in ((0.0, D ** -0.5), (20.0, 0.5)):
            got = attend(q, k, v, bt, ctxs, most, ps, bs, scale, cap, fp8).double()
            want = reference(q, kv, scale, cap)
            for i, c in enumerate(ctxs):
                if c == 0 and ps == 0:
                    continue                                          # (nothing to attend to: zeros or untouched)
                # bf16 outputs, 2^-9 of each; where 16 waves do not fit, probabilities of bf16 too
                assert torch.isfinite(got[i]).all() and (got[i] - want[i]).abs().max() <= 2.0 ** -7 * max(want[i].abs().max().item(), 1e-3), (ps, c)


@pytest.mark.parametrize("most", [1, 33, 146, 250, 500])
def test_scores_that_are_no_numbers(most):
    """a key that is NaN makes the heads over it NaN, a query that is infinite its own head, and no other"""
    ctxs = [most, (most + 1) // 2, most]
    k, v, bt, kv = cache(ctxs, 2, 128, 16, False, most)
    q = torch.randn(3, 8, 128, device="cuda").bfloat16()
    k[bt[0].long()[(most - 1) // 16], 0, 3, (most - 1) % 16, 5] = float("nan")
    q[1, 6, 9] = float("inf")
    for ps in (0, 32):
        got, want = attend(q, k, v, bt, ctxs, most, ps, 16, 128 ** -0.5, 0.0, False), reference(q, kv, 128 ** -0.5, 0.0)
        bad = torch.zeros(3, 8, dtype=torch.bool, device="cuda")
        bad[0, :4] = bad[1, 6] = True
        assert got[bad].isnan().all() and torch.isfinite(got[~bad]).all()
        assert (got[~bad].double() - want[~bad]).abs().max() <= 2.0 ** -7 * want[~bad].abs().max()


def test_probabilities_keep_more_than_bf16():
    """against 64 bits the result is off by its own rounding to bf16 (2-norm 2^-9 / sqrt(3) to 2^-8 / sqrt(3)... measured 1.6e-3) and no more"""
    k, v, bt, kv = cache([256, 200, 130, 512], 8, 128, 64, False, 1)
    q = torch.randn(4, 32, 128, device="cuda").bfloat16()
    want = reference(q, kv, 128 ** -0.5, 0.0)
    got = attend(q, k, v, bt, [256, 200, 130, 512], 512, 0, 64, 128 ** -0.5, 0.0, False)
    near = want.bfloat16()
    assert (got != near).double().mean() < 0.01                          # (ties and sums in f32)
    assert ((got.double() - want).norm() / want.norm()).item() < 1.01 * ((near.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("H,G,ctxs", [(28, 4, [584, 600, 3, 64, 65, 128] * 3), (24, 8, [520, 1, 0, 300, 100, 64, 513, 64]), (32, 8, [1] * 9)])
def test_stream_with_more_workgroups_than_stages(H, G, ctxs, fp8):
    f = lib.mi355_internal_pa_plan
    f.restype, f.argtypes = ctypes.c_int32, [ctypes.c_int32] * 8 + [ctypes.POINTER(ctypes.c_int32)]
    ps, most = ctypes.c_int32(32), max(max(ctxs), 513)
    cap = f(len(ctxs), H, G, 128, 64, most, int(fp8), 513, ctypes.byref(ps))
    assert ps.value == 64 and cap == 64 * min(64, (512 if fp8 else 256) // G)
    assert f(len(ctxs), H, G, 128, 64, most, int(fp8), 9, ctypes.byref(ps)) == most              # no room for that many partials
    assert f(len(ctxs), H, G, 128, 64, 300, int(fp8), 513, ctypes.byref(ps)) == 300 and ps.value == 32
    k, v, bt, kv = cache(ctxs, G, 128, 64, fp8, H)
    q = torch.randn(len(ctxs), H, 128, device="cuda").bfloat16()
    got = attend(q, k, v, bt, ctxs, cap, 64, 64, 128 ** -0.5, 0.0, fp8).double()
    want = reference(q, kv, 128 ** -0.5, 0.0)
    for i, c in enumerate(ctxs):
        if c:
            assert (got[i] - want[i]).abs().max() <= 2.0 ** -7 * max(want[i].abs().max().item(), 1e-3), c
