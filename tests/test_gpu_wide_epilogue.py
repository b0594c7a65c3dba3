"""9 .. 32 tokens: the launch that adds the ranges of K and applies the epilogue eight columns a lane, against the general one (which pointers off 16 bytes take): the
same bits, at outputs that end inside a k-block of the next image, odd token counts, with and without norm, bias and a next product."""
import ctypes

import numpy as np
import pytest
import torch

import candle_vllm_amd.ops as cv
from candle_vllm_amd.model import KV_PAGED_FP8
from oracle import kquants as kq
from tests.test_gpu_prompt_tiles import TOL, _desc, blocks, close, product

pytestmark = pytest.mark.gpu
Q4, Q6 = kq.GGML_Q4_K, kq.GGML_Q6_K


def go(d):
    assert cv.lib.mi355_qmatmul_fused(ctypes.byref(d), torch.cuda.current_stream().cuda_stream) == 0


@pytest.mark.parametrize("T", [9, 16, 17, 32])
@pytest.mark.parametrize("epi,N,K,kind,norm,bias", [("store", 264, 512, Q4, True, True), ("store", 4104, 256, Q6, False, False), ("resid", 1000, 4096, Q4, False, True),
                                                    ("resid", 16, 14336, Q6, True, False), ("silu", 520, 1024, Q4, True, False), ("silu", 272, 2048, Q4, False, True)])
def test_same_bits_as_the_general_launch(T, epi, N, K, kind, norm, bias):
    rng = np.random.default_rng(T + N + K)
    ms = [cv.QMatMul(blocks(rng, N, K, kind), kind, "cuda") for _ in range(2 if epi == "silu" else 1)]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    nw = torch.from_numpy(rng.uniform(0.5, 1.5, K).astype(np.float32)).cuda() if norm else None
    b = torch.from_numpy(rng.normal(0, 1, N * len(ms)).astype(np.float32)).cuda() if bias else None
    old = torch.from_numpy(rng.normal(0, 1, (T, N)).astype(np.float32)).cuda()
    got = []
    for shift in (0, 1):
        buf = torch.full((T * N + 8,), float("nan"), device="cuda")
        out = buf[shift:shift + T * N].view(T, N)
        if epi == "resid":
            out.copy_(old)
        d = _desc(x, ms, nw, {"store": cv.EPI_STORE, "resid": cv.EPI_RESID, "silu": cv.EPI_SILU_MUL}[epi], out)
        if bias:
            d.bias = b.data_ptr()
        go(d)
        got.append(out.clone())
        assert torch.isnan(buf[:shift]).all() and torch.isnan(buf[shift + T * N:]).all()
    assert torch.isfinite(got[0]).all() and torch.equal(got[0], got[1])


@pytest.mark.parametrize("T,hid,inter", [(9, 768, 2048), (31, 1024, 2816)])
def test_image_for_the_next_product(T, hid, inter):
    """wo (residual) -> gate/up -> down with the next product's image left by the launch, against the same calls without the hint: the same bits"""
    rng = np.random.default_rng(T)
    shapes = ((hid, 512), (inter, hid), (inter, hid), (hid, inter))
    wo, w1, w3, w2 = (cv.QMatMul(blocks(rng, n, k, Q4, odd=False), Q4, "cuda") for n, k in shapes)
    x = torch.from_numpy(rng.normal(0, 1, (T, 512)).astype(np.float32)).cuda()
    nw = torch.from_numpy(rng.uniform(0.5, 1.5, hid).astype(np.float32)).cuda()
    start, got = torch.from_numpy(rng.normal(0, 1, (T, hid)).astype(np.float32)).cuda(), []
    for chain in (0, 1):
        r, h = start.clone(), torch.empty(T, inter, device="cuda")
        a, b, c = _desc(x, [wo], None, cv.EPI_RESID, r), _desc(r, [w1, w3], nw, cv.EPI_SILU_MUL, h), _desc(h, [w2], None, cv.EPI_RESID, r)
        a.chain_next, a.chain_next_k, a.chain_next_norm = chain, hid, nw.data_ptr()
        b.chain_next, b.chain_next_k = chain, inter
        for d in (a, b, c):
            go(d)
        got += [h, r]
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])


@pytest.mark.parametrize("layout,D,rot,T", [("flash", 128, 64, 9), ("fp8", 128, 128, 32), ("paged", 72, 24, 17), ("fp8", 64, 32, 16), ("paged", 64, 64, 31)])
@pytest.mark.parametrize("bias", [False, True])
def test_qkv(layout, D, rot, T, bias):
    """against the general launch, and against 64 bits: q and what the cache gets, rounded to bf16 (2^-8), for an e4m3 cache once more (2^-4)"""
    H, Hkv, K, block = 6, 2, 1024, 16
    rng = np.random.default_rng(T)
    kinds, heads = (Q4, Q4, Q6), (H, Hkv, Hkv)
    bs = [blocks(rng, n * D, K, t, odd=False) for n, t in zip(heads, kinds)]
    ms = [cv.QMatMul(b, t, "cuda") for b, t in zip(bs, kinds)]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    nw = torch.from_numpy(rng.uniform(0.5, 1.5, K).astype(np.float32)).cuda()
    add = torch.from_numpy(rng.normal(0, 1, (H + 2 * Hkv) * D).astype(np.float32)).cuda()
    pos, slot = torch.from_numpy(rng.integers(0, 500, T)).cuda(), torch.from_numpy(rng.permutation(T + 64)[:T].astype(np.int64)).cuda()
    slot[::7] = -1
    ang = torch.arange(500, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(rot // 2, device="cuda").double() / (rot // 2))
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    n = ((T + 64 + block - 1) // block) * block * Hkv * D
    dt = torch.uint8 if layout == "fp8" else torch.bfloat16
    got = []
    for shift in (0, 1):
        q = torch.zeros(T * H * D + 8, dtype=torch.bfloat16, device="cuda")[shift:shift + T * H * D]
        kc, vc = torch.zeros(n, dtype=dt, device="cuda"), torch.zeros(n, dtype=dt, device="cuda")
        d = _desc(x, ms, nw, cv.EPI_QKV_ROPE_CACHE, q.view(T, -1))
        d.out, d.ldo = None, 0
        d.bias = add.data_ptr() if bias else None
        d.cos_table, d.sin_table, d.positions, d.slot_mapping = (v.data_ptr() for v in (cos, sin, pos, slot))
        d.q_out, d.key_cache, d.value_cache = q.data_ptr(), kc.data_ptr(), vc.data_ptr()
        d.num_heads, d.num_kv_heads, d.head_dim, d.rotary_dim, d.block_size = H, Hkv, D, rot, block
        d.kv_layout = {"flash": cv.KV_FLASH, "paged": cv.KV_PAGED, "fp8": KV_PAGED_FP8}[layout]
        go(d)
        got.append([q.float().clone(), kc, vc])
    assert got[0][0].abs().sum() > 0 and got[0][1].any() and got[0][2].any()
    assert torch.equal(got[0][2], got[1][2])                          # values: not rotated, the same bits
    # a rotation is one product and one multiply-add in either order, so 2^-23 of a product apart: now and then across the middle of two bf16 (2^-7), then e4m3 (2^-3), numbers
    for a, b, step in zip(got[0], got[1], (2.0 ** -7, 2.0 ** -3 if layout == "fp8" else 2.0 ** -7)):
        a, b = ((v.view(torch.float8_e4m3fn) if v.dtype == torch.uint8 else v).float() for v in (a, b))
        assert ((a - b).abs() <= step * torch.maximum(a.abs(), b.abs()) + 2.0 ** -9).all() and (a != b).float().mean() < 1e-2
    xn = (x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 0.3) * nw.double()).float()
    y = [(product(xn, b, t) + (a.double() if bias else 0)).view(T, -1, D) for b, t, a in zip(bs, kinds, add.split([n * D for n in heads]))]
    c, s = ang.cos()[pos][:, None], ang.sin()[pos][:, None]
    turned = [torch.cat([torch.stack([z[..., 0:rot:2] * c - z[..., 1:rot:2] * s, z[..., 0:rot:2] * s + z[..., 1:rot:2] * c], dim=-1).reshape(T, -1, rot), z[..., rot:]], -1) for z in y[:2]]
    q, kc, vc = got[0]
    blk, off, x16 = slot[slot >= 0] // block, slot[slot >= 0] % block, 16 if layout == "fp8" else 8
    if layout == "fp8":
        kc, vc = kc.view(torch.float8_e4m3fn).float(), vc.view(torch.float8_e4m3fn).float()
        assert max(turned[1].abs().max(), y[2].abs().max()).item() < 448  # nothing saturates
    kc = kc.view(-1, block, Hkv, D)[blk, off] if layout == "flash" else kc.view(-1, Hkv, D // x16, block, x16)[blk, :, :, off].reshape(-1, Hkv, D)
    vc = vc.view(-1, block, Hkv, D)[blk, off] if layout == "flash" else vc.view(-1, Hkv, D, block)[blk, :, :, off]
    cache_tol = TOL + 2.0 ** -8 + (2.0 ** -4 if layout == "fp8" else 0)
    for have, want, tol in ((q.view(T, H, D), turned[0], TOL + 2.0 ** -8), (kc, turned[1][slot >= 0], cache_tol), (vc, y[2][slot >= 0], cache_tol)):
        assert close(have, want) < tol


@pytest.mark.parametrize("kind,N,K,silu", [(Q4, 4096, 14336, False), (Q6, 2064, 8192, False), (Q6, 32000, 2048, False), (Q4, 8192, 3072, True), (Q4, 8200, 2816, True)])
def test_ranges_of_k(kind, N, K, silu):
    """launches whose ranges of K fill what they leave idle (long K; a few more workgroups than CUs; little more than half of them), against 64 bits"""
    rng = np.random.default_rng(N + K)
    bs = [blocks(rng, N, K, kind, odd=False) for _ in range(2 if silu else 1)]
    ms = [cv.QMatMul(b, kind, "cuda") for b in bs]
    x = torch.from_numpy(rng.normal(0, 1, (19, K)).astype(np.float32)).cuda()
    out = torch.empty(19, N, device="cuda")
    go(_desc(x, ms, None, cv.EPI_SILU_MUL if silu else cv.EPI_STORE, out))
    want = [product(x, b, kind) for b in bs]
    if silu:                                                          # (the product of two: twice the error of one)
        assert close(out, torch.nn.functional.silu(want[0]) * want[1]) < 2 * TOL
    else:
        assert close(out, want[0]) < TOL


def last_ranges():
    f = cv.lib.mi355_internal_last_qw1_split
    f.restype = ctypes.c_int32
    return f()


# row-tile workgroups (seven tiles each) on 256 CUs: the last number that takes a rule, and the first that does not
@pytest.mark.parametrize("wgs,nkb,T,kind,ranges", [(37, 56, 9, Q4, 6), (42, 32, 32, Q4, 6), (43, 32, 32, Q6, 5), (128, 12, 9, Q4, 2), (129, 12, 32, Q4, 3), (146, 20, 9, Q6, 3), (170, 16, 32, Q4, 3),
                                                   (171, 16, 32, Q4, 1), (150, 11, 9, Q4, 1), (256, 16, 9, Q4, 1), (257, 16, 9, Q4, 3), (341, 16, 32, Q6, 3), (342, 16, 32, Q6, 2), (384, 16, 9, Q4, 2),
                                                   (385, 16, 9, Q4, 1), (511, 12, 32, Q4, 1), (300, 12, 32, Q4, 2), (300, 8, 9, Q4, 2), (300, 8, 32, Q4, 1), (300, 8, 32, Q6, 2), (300, 7, 9, Q6, 1)])
def test_number_of_ranges(wgs, nkb, T, kind, ranges):
    from candle_vllm_amd.model import random_tiles
    N, K = wgs * 7 * 16 - 48, 256 * nkb
    tiles = random_tiles(kind, N, K, "cuda", torch.Generator(device="cuda").manual_seed(wgs))
    x, out = torch.randn(T, K, device="cuda"), torch.full((T, N), float("nan"), device="cuda")
    d = cv.QmmDesc()
    d.nseg, d.w_tiles[0], d.ggml_type[0], d.n_rows[0] = 1, tiles.data_ptr(), kind, N
    d.x, d.x_dtype, d.ldx, d.k, d.num_tokens = x.data_ptr(), cv.DT_F32, K, K, T
    d.epilogue, d.out, d.ldo = cv.EPI_STORE, out.data_ptr(), N
    go(d)
    assert last_ranges() == ranges and torch.isfinite(out).all()


@pytest.mark.parametrize("kind,N,K,T,few,ranges", [(Q4, 4096, 14336, 19, 4, 6), (Q6, 32000, 4096, 32, 1, 3), (Q4, 16384, 3072, 9, 1, 3)])
def test_no_room_for_more_sums(kind, N, K, T, few, ranges):
    """room for the sums of the powers of two and no more: the product goes in those, on a full card and in a capture, where the buffer of an earlier product may not grow"""
    rng = np.random.default_rng(N)
    b = blocks(rng, N, K, kind, odd=False)
    m = cv.QMatMul(b, kind, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    want, tokens = product(x, b, kind), 16 if T <= 16 else 32
    cv.lib.mi355_internal_scratch_limit.argtypes = [ctypes.c_int64]
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        cv.lib.mi355_internal_scratch_limit(max(few * tokens * N * 4, K // 256 * 20480))   # (a k-block of the image: less than 20 KiB)
        try:
            got = m.forward(x)
            assert last_ranges() == few and close(got, want) < TOL
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
                captured = m.forward(x)
        finally:
            cv.lib.mi355_internal_scratch_limit(-1)
        assert last_ranges() == few
        for _ in range(3):
            captured.zero_()
            graph.replay()
            assert torch.equal(captured, got)
        assert close(m.forward(x), want) < TOL and last_ranges() == ranges
