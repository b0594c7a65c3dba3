"""The prompt products that unpack every weight once per workgroup (csrc/qmm_prompt_gemm.inc): each tile of both types, at tiles that end inside
a token block, a row tile or the matrix, with every epilogue, against dequantised weights in 64 bits."""
import ctypes

import numpy as np
import pytest
import torch

import candle_vllm_amd.ops as cv
from candle_vllm_amd.model import KV_PAGED_FP8
from oracle import kquants as kq

pytestmark = pytest.mark.gpu
Q4, Q6 = kq.GGML_Q4_K, kq.GGML_Q6_K
# activations are rounded to f16 once (2^-12 of each, its share of a row's error about 2^-12 / sqrt(3) and, over the largest outputs, three times that)
TOL = 5e-4


def last_tile():
    f = cv.lib.mi355_internal_last_qpw
    f.restype = ctypes.c_int32
    return f()


def blocks(rng, n, k, kind, odd=True):
    """native GGUF blocks of random codes; with `odd`, blocks of d = 0 (with and without a minimum), of a large minimum beside a tiny d, and, Q6_K, of d < 0"""
    size = 144 if kind == Q4 else 210
    b = rng.integers(0, 256, (n, k // 256, size), dtype=np.uint8)
    d = rng.uniform(1e-4, 3e-4, (n, k // 256)).astype(np.float16)
    m = rng.uniform(1e-4, 3e-3, (n, k // 256)).astype(np.float16)
    if odd:
        pick = rng.integers(0, 16, (n, k // 256))
        d[pick == 0] = 0
        m[pick == 0] *= rng.integers(0, 2, (pick == 0).sum()).astype(np.float16)
        d[pick == 1] = 6e-7
        d[pick == 2] = 2e-2 if kind == Q4 else -3e-4

    def put(at, v):
        b[:, :, at:at + 2] = v.view(np.uint8).reshape(n, k // 256, 2)
    put(0 if kind == Q4 else 208, d)
    if kind == Q4:
        put(2, m)
    return b


def product(x, b, kind):
    return x.double() @ torch.from_numpy(kq.dequantize(b, kind)).cuda().double().t()


def close(got, want):
    assert torch.isfinite(got).all()
    return ((got.double() - want).abs().max() / want.abs().max()).item()


@pytest.mark.parametrize("kind,T,N,K,tile", [(Q4, 385, 28628, 1024, 0), (Q4, 700, 16380, 1024, 2), (Q4, 1281, 4096, 2048, 1), (Q4, 1300, 4120, 2048, 1), (Q4, 4097, 2064, 1024, 2),
                                             (Q4, 4001, 4084, 1024, 0), (Q4, 200, 512, 512, -1), (Q6, 1300, 4120, 1024, 11), (Q6, 1153, 4096, 512, 11), (Q6, 100, 2048, 8192, -1)])
def test_store_and_residual(kind, T, N, K, tile):
    rng = np.random.default_rng(T + N)
    b = blocks(rng, N, K, kind)
    m = cv.QMatMul(b, kind, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    x[T // 2] *= 3000.0                                               # a token that the image scales
    want = product(x, b, kind)
    rows = torch.cat([torch.arange(T // 2), torch.arange(T // 2 + 1, T)]).cuda()
    bias = torch.randn(N, device="cuda")
    got = m.forward(x)
    assert last_tile() == tile
    assert close(got[rows], want[rows]) < TOL and close(got[T // 2], want[T // 2]) < TOL
    assert close(m.forward(x, bias)[rows], (want + bias)[rows]) < TOL
    for pad in (0, 3):                                                # whole fours, and rows that are not
        o = torch.randn(T, N + pad, device="cuda")
        keep = o.clone()
        d = cv.QmmDesc()
        d.nseg, d.w_tiles[0], d.ggml_type[0], d.n_rows[0] = 1, m.tiles.data_ptr(), kind, N
        d.x, d.x_dtype, d.ldx, d.k, d.num_tokens = x.data_ptr(), cv.DT_F32, K, K, T
        d.epilogue, d.out, d.ldo, d.residual = cv.EPI_RESID, o.data_ptr(), N + pad, o.data_ptr()
        assert cv.lib.mi355_qmatmul_fused(d, torch.cuda.current_stream().cuda_stream) == 0
        assert close(o[rows, :N], (want + keep[:, :N].double())[rows]) < TOL
        assert torch.equal(o[:, N:], keep[:, N:])


@pytest.mark.parametrize("T,N,K,wide", [(385, 2064, 8192, True), (500, 4096, 3584, True), (1000, 1040, 14336, True), (193, 4096, 2048, False)])
def test_q6k_ranges(T, N, K, wide):
    """ranges of K on the 256 x 128 tiles of Q6_K: tiles that end inside a token block or the matrix, ranges of unequal lengths, store and residual"""
    rng = np.random.default_rng(T + N)
    b = blocks(rng, N, K, Q6)
    m = cv.QMatMul(b, Q6, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    want = product(x, b, Q6)
    keep = torch.randn(T, N, device="cuda")
    for epi in (cv.EPI_STORE, cv.EPI_RESID):
        out = keep.clone()
        d = _desc(x, [m], None, epi, out)
        assert cv.lib.mi355_qmatmul_fused(ctypes.byref(d), torch.cuda.current_stream().cuda_stream) == 0
        assert last_split() > 1 and (last_tile() == 12) == wide
        assert close(out, want + (keep.double() if epi == cv.EPI_RESID else 0)) < TOL


@pytest.mark.parametrize("kind,T,N,K,tile", [(Q4, 1281, 4096, 2048, 1), (Q4, 4097, 2064, 1024, 2), (Q6, 1300, 4096, 1024, 11)])
def test_no_room_for_whole_tiles(kind, T, N, K, tile):
    """room for the image in whole 128 tokens but not in whole tiles: the 64-token kernels take the product -- on a full card, and in a capture, where the buffer of
    an earlier product may not grow"""
    rng = np.random.default_rng(T)
    b = blocks(rng, N, K, kind)
    m = cv.QMatMul(b, kind, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    want, rows = product(x, b, kind), (T + 127) // 128 * 128
    room = rows * (2 * K + K // 256 * 32 + 8) + 4 * T * N + 4096
    cv.lib.mi355_internal_scratch_limit.argtypes = [ctypes.c_int64]
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        cv.lib.mi355_internal_scratch_limit(room)
        try:
            got = m.forward(x)
        finally:
            cv.lib.mi355_internal_scratch_limit(-1)
        assert last_tile() == -1 and close(got, want) < TOL
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
            captured = m.forward(x)
        assert last_tile() == -1
        for _ in range(3):
            captured.zero_()
            graph.replay()
            assert torch.equal(captured, got)
        assert close(m.forward(x), want) < TOL and last_tile() == tile


@pytest.mark.parametrize("T,N,K,tile", [(385, 14314, 1024, 0), (700, 8190, 1024, 2), (1281, 2048, 2048, 1), (1300, 2060, 2048, 1)])
def test_gate_up(T, N, K, tile):
    rng = np.random.default_rng(T + N)
    bg, bu = blocks(rng, N, K, Q4), blocks(rng, N, K, Q4)
    g, u = cv.QMatMul(bg, Q4, "cuda"), cv.QMatMul(bu, Q4, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    nw = 1 + 0.1 * torch.randn(K, device="cuda")
    xn = (x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * nw.double()).float()
    want = torch.nn.functional.silu(product(xn, bg, Q4)) * product(xn, bu, Q4)
    out = torch.empty(T, N, device="cuda")
    cv.qmatmul_fused([g, u], x, epilogue=cv.EPI_SILU_MUL, out=out, norm_weight=nw, norm_eps=1e-5)
    assert last_tile() == tile
    assert close(out, want) < 2 * TOL                                 # two rounded factors


# heads and rotated parts of whole eights (eight columns per lane) and not (a column per lane); values Q4_K and Q6_K; the three cache layouts
@pytest.mark.parametrize("layout,D,rot,v_kind,H,Hkv,T,K", [("paged", 128, 128, Q6, 32, 8, 2049, 1024), ("paged", 64, 32, Q4, 64, 2, 2049, 1024), ("flash", 128, 128, Q4, 32, 4, 2049, 1024),
                                                           ("fp8", 128, 64, Q4, 40, 4, 2049, 1024), ("paged", 80, 20, Q4, 60, 3, 2051, 1024), ("flash", 80, 20, Q6, 60, 3, 2051, 1024)])
def test_qkv(layout, D, rot, v_kind, H, Hkv, T, K):
    rng = np.random.default_rng(T + D)
    kinds, heads = (Q4, Q4, v_kind), (H, Hkv, Hkv)
    bs = [blocks(rng, n * D, K, t, odd=layout != "fp8") for n, t in zip(heads, kinds)]   # (e4m3 ends at 448)
    ms = [cv.QMatMul(b, t, "cuda") for b, t in zip(bs, kinds)]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    block = 16
    pos = torch.from_numpy(rng.integers(0, 5000, T)).cuda()
    slot = torch.from_numpy(rng.permutation(T + 64)[:T].astype(np.int64)).cuda()
    slot[5] = -1                                                      # a token that the cache does not take
    half = rot // 2
    ang = torch.arange(5000, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(half, device="cuda").double() / half)
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    nb = (T + 64 + block - 1) // block
    x16 = 16 if layout == "fp8" else 8
    dt = torch.uint8 if layout == "fp8" else torch.bfloat16
    if layout == "flash":
        kc, vc = (torch.zeros(nb, block, Hkv, D, dtype=dt, device="cuda") for _ in range(2))
    else:
        kc, vc = torch.zeros(nb, Hkv, D // x16, block, x16, dtype=dt, device="cuda"), torch.zeros(nb, Hkv, D, block, dtype=dt, device="cuda")
    q_out = torch.zeros(T, H * D, dtype=torch.bfloat16, device="cuda")
    bias = torch.randn(sum(heads) * D, device="cuda") * 0.1
    d = cv.QmmDesc()
    d.nseg = 3
    for i, (m, n, t) in enumerate(zip(ms, heads, kinds)):
        d.w_tiles[i], d.ggml_type[i], d.n_rows[i] = m.tiles.data_ptr(), t, n * D
    d.x, d.x_dtype, d.ldx, d.k, d.num_tokens = x.data_ptr(), cv.DT_F32, K, K, T
    d.epilogue, d.bias, d.cos_table, d.sin_table, d.positions, d.slot_mapping = cv.EPI_QKV_ROPE_CACHE, bias.data_ptr(), cos.data_ptr(), sin.data_ptr(), pos.data_ptr(), slot.data_ptr()
    d.q_out, d.key_cache, d.value_cache = q_out.data_ptr(), kc.data_ptr(), vc.data_ptr()
    d.num_heads, d.num_kv_heads, d.head_dim, d.rotary_dim, d.block_size = H, Hkv, D, rot, block
    d.kv_layout = {"paged": cv.KV_PAGED, "flash": cv.KV_FLASH, "fp8": 2}[layout]
    assert cv.lib.mi355_qmatmul_fused(d, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert last_tile() >= 0
    parts = torch.split(torch.cat([product(x, b, t) for b, t in zip(bs, kinds)], 1) + bias, [n * D for n in heads], 1)

    def turned(y):
        y = y.view(T, -1, D).clone()
        c, s = cos[pos].double()[:, None], sin[pos].double()[:, None]
        a, b = y[..., 0:rot:2].clone(), y[..., 1:rot:2].clone()
        y[..., 0:rot:2], y[..., 1:rot:2] = a * c - b * s, a * s + b * c
        return y
    tol = TOL + 2.0 ** -8 if layout != "fp8" else TOL + 2.0 ** -3     # bf16's rounding; e4m3's
    assert close(q_out, turned(parts[0]).reshape(T, -1)) < TOL + 2.0 ** -8
    ok = slot >= 0
    blk, off = slot[ok] // block, slot[ok] % block
    if layout == "flash":
        k, v = kc[blk, off], vc[blk, off]
    else:
        k, v = kc[blk, :, :, off].reshape(int(ok.sum()), Hkv, D), vc[blk, :, :, off]
        if layout == "fp8":
            k, v = k.view(torch.float8_e4m3fn).float(), v.contiguous().view(torch.float8_e4m3fn).float()
    assert close(k.float(), turned(parts[1])[ok]) < tol
    assert close(v.float(), parts[2].view(T, Hkv, D)[ok]) < tol
    untouched = torch.ones(nb * block, dtype=torch.bool, device="cuda")
    untouched[slot[ok]] = False
    flat = kc.view(nb * block, -1) if layout == "flash" else kc.permute(0, 3, 1, 2, 4).reshape(nb * block, -1)
    assert (flat[untouched].float() == 0).all()


def last_split():
    f = cv.lib.mi355_internal_last_qpg_split
    f.restype = ctypes.c_int32
    return f()


# K in ranges: a token in a block of its own, one to eight behind whole portions of 32 (they go in a launch of their own), blocks that end inside, rows that fill neither tile nor workgroup, k-blocks that the ranges do not divide
@pytest.mark.parametrize("kind,T,N,K", [(Q4, 41, 2048, 2048), (Q4, 64, 530, 8192), (Q4, 65, 4096, 4096), (Q4, 73, 4096, 4096), (Q4, 129, 3072, 8192), (Q4, 300, 1024, 2816), (Q4, 500, 2048, 8192),
                                        (Q6, 41, 2048, 8192), (Q6, 64, 4100, 2048), (Q6, 72, 2048, 8192), (Q6, 95, 424, 1024), (Q6, 130, 4096, 14336), (Q6, 700, 512, 3328)])
def test_ranges_of_k(kind, T, N, K):
    rng = np.random.default_rng(T + N)
    b = blocks(rng, N, K, kind)
    m = cv.QMatMul(b, kind, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    x[T // 2] *= 3000.0                                               # tokens that the image scales down and up
    x[T // 3] *= 1e-7
    want, bias = product(x, b, kind), torch.randn(N, device="cuda")
    for got, ref in ((m.forward(x), want), (m.forward(x, bias), want + bias)):
        assert last_split() > 1
        for t in (T // 2, T // 3):
            assert close(got[t], ref[t]) < TOL
        rest = [t for t in range(T) if t not in (T // 2, T // 3)]
        assert close(got[rest], ref[rest]) < TOL
    o = torch.randn(T, N + 3, device="cuda")
    keep = o.clone()
    d = cv.QmmDesc()
    d.nseg, d.w_tiles[0], d.ggml_type[0], d.n_rows[0] = 1, m.tiles.data_ptr(), kind, N
    d.x, d.x_dtype, d.ldx, d.k, d.num_tokens = x.data_ptr(), cv.DT_F32, K, K, T
    d.epilogue, d.out, d.ldo, d.residual = cv.EPI_RESID, o.data_ptr(), N + 3, o.data_ptr()
    assert cv.lib.mi355_qmatmul_fused(d, torch.cuda.current_stream().cuda_stream) == 0
    assert close(o[rest, :N], (want + keep[:, :N].double())[rest]) < TOL and torch.equal(o[:, N:], keep[:, N:])


def rms(got, want):
    assert torch.isfinite(got).all()
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("kind", [Q4, Q6])
@pytest.mark.parametrize("T", [33, 40, 41, 65, 72, 73])
def test_last_tokens_of_a_launch(kind, T):
    """the last 1 .. 8 tokens behind whole portions of 32 keep their activations in two bf16 planes: 2^-17 of each at most, and that of every sum, since roundings
    add up as independent values do; 2^-16 with the f32 sums (one plane, as the others have, shows 2^-13 and more).  Store, and gate/up behind a norm"""
    rng = np.random.default_rng(T)
    K, N, tail = 2048, 1024, T % 32 if T % 32 <= 8 else 0
    head = T - tail
    b = blocks(rng, N, K, kind, odd=False)
    m = cv.QMatMul(b, kind, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    want = product(x, b, kind)
    got = m.forward(x)
    assert close(got[:head], want[:head]) < TOL
    assert not tail or rms(got[head:], want[head:]) < 2.0 ** -16
    bu = blocks(rng, N, K, kind, odd=False)
    u, nw, out = cv.QMatMul(bu, kind, "cuda"), 1 + 0.1 * torch.randn(K, device="cuda"), torch.empty(T, N, device="cuda")
    xn = x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * nw.double()
    g, up = product(xn, b, kind), product(xn, bu, kind)
    cv.qmatmul_fused([m, u], x, epilogue=cv.EPI_SILU_MUL, out=out, norm_weight=nw, norm_eps=1e-5)
    want = torch.nn.functional.silu(g) * up
    assert close(out[:head], want[:head]) < 2 * TOL
    assert not tail or rms(out[head:], want[head:]) < 2.0 ** -14      # two rounded factors, and silu's slope of up to 1.1 beside values that may be smaller than they


@pytest.mark.parametrize("T,N,K", [(41, 2048, 2048), (74, 8192, 3072), (90, 500, 4096)])
def test_gate_up_ranges_of_k(T, N, K):
    rng = np.random.default_rng(T + N)
    bg, bu = blocks(rng, N, K, Q4, odd=False), blocks(rng, N, K, Q4, odd=False)
    g, u = cv.QMatMul(bg, Q4, "cuda"), cv.QMatMul(bu, Q4, "cuda")
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    nw = 1 + 0.1 * torch.randn(K, device="cuda")
    xn = (x.double() * torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * nw.double()).float()
    want = torch.nn.functional.silu(product(xn, bg, Q4)) * product(xn, bu, Q4)
    out = torch.empty(T, N, device="cuda")
    cv.qmatmul_fused([g, u], x, epilogue=cv.EPI_SILU_MUL, out=out, norm_weight=nw, norm_eps=1e-5)
    assert last_split() > 1
    assert close(out, want) < 2 * TOL                                 # two rounded factors


@pytest.mark.parametrize("v_kind,T", [(Q4, 41), (Q6, 41), (Q4, 72), (Q6, 66), (Q4, 161), (Q6, 320)])
def test_qkv_ranges_of_k(v_kind, T):
    H, Hkv, D, K, block = 16, 4, 128, 2048, 16
    rng = np.random.default_rng(T)
    kinds, heads = (Q4, Q4, v_kind), (H, Hkv, Hkv)
    bs = [blocks(rng, n * D, K, t) for n, t in zip(heads, kinds)]
    ms = [cv.QMatMul(b, t, "cuda") for b, t in zip(bs, kinds)]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    pos, slot = torch.from_numpy(rng.integers(0, 500, T)).cuda(), torch.from_numpy(rng.permutation(T + 64)[:T].astype(np.int64)).cuda()
    slot[5] = -1
    ang = torch.arange(500, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(D // 2, device="cuda").double() / (D // 2))
    nb = (T + 64 + block - 1) // block
    kc, vc = torch.zeros(nb, Hkv, D // 8, block, 8, dtype=torch.bfloat16, device="cuda"), torch.zeros(nb, Hkv, D, block, dtype=torch.bfloat16, device="cuda")
    q_out = torch.zeros(T, H * D, dtype=torch.bfloat16, device="cuda")
    cv.qmatmul_fused(ms, x, epilogue=cv.EPI_QKV_ROPE_CACHE, rope=dict(cos=ang.cos().float().contiguous(), sin=ang.sin().float().contiguous(), positions=pos, slot_mapping=slot,
                                                                     q_out=q_out, key_cache=kc, value_cache=vc, num_heads=H, num_kv_heads=Hkv, head_dim=D, rotary_dim=D))
    assert last_split() > 1
    y = [product(x, b, t).view(T, -1, D) for b, t in zip(bs, kinds)]
    c, s = ang.cos()[pos][:, None], ang.sin()[pos][:, None]
    turned = [torch.stack([z[..., 0::2] * c - z[..., 1::2] * s, z[..., 0::2] * s + z[..., 1::2] * c], dim=-1).reshape(T, -1, D) for z in y[:2]]
    ok = slot >= 0
    blk, off = slot[ok] // block, slot[ok] % block
    for got, want in ((q_out.view(T, H, D), turned[0]), (kc[blk, :, :, off].reshape(-1, Hkv, D), turned[1][ok]), (vc[blk, :, :, off], y[2][ok])):
        assert close(got.float(), want) < TOL + 2.0 ** -8                 # bf16's rounding


def test_ranges_of_k_without_room():
    """no room for the sums of several ranges: one range from 96 tokens on, the 32-token launches below"""
    rng = np.random.default_rng(3)
    K, N = 4096, 2048
    b = blocks(rng, N, K, Q4)
    m = cv.QMatMul(b, Q4, "cuda")
    cv.lib.mi355_internal_scratch_limit.argtypes = [ctypes.c_int64]
    for T, splits in ((200, 1), (80, 0)):
        x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
        want = product(x, b, Q4)
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            cv.lib.mi355_internal_scratch_limit(4200000)                  # 200 tokens: image 2.2 MB, sums of a range 1.6 MB
            try:
                got = m.forward(x)
                assert last_split() == splits
            finally:
                cv.lib.mi355_internal_scratch_limit(-1)
            assert close(got, want) < TOL
            assert close(m.forward(x), want) < TOL and last_split() > 1


def test_sums_of_ranges_are_bounded():
    """256 MiB of sums at most, and a workspace that grows for them is not doubled beyond those and the image of 1024 tokens"""
    from candle_vllm_amd.model import random_tiles
    K, MiB = 14336, 1 << 20
    tiles = random_tiles(Q4, 57344, K, "cuda", torch.Generator(device="cuda").manual_seed(1))
    x, out = torch.randn(809, K, device="cuda"), torch.empty(809, 57344, device="cuda")

    def run(tokens, rows):
        d = cv.QmmDesc()
        d.nseg, d.w_tiles[0], d.ggml_type[0], d.n_rows[0] = 1, tiles.data_ptr(), Q4, rows
        d.x, d.x_dtype, d.ldx, d.k, d.num_tokens = x.data_ptr(), cv.DT_F32, K, K, tokens
        d.epilogue, d.out, d.ldo = cv.EPI_STORE, out.data_ptr(), rows
        assert cv.lib.mi355_qmatmul_fused(d, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return last_split()
    with torch.cuda.stream(torch.cuda.Stream()):                          # (a workspace of its own)
        assert run(41, 4096) > 1
        before = torch.cuda.mem_get_info()[0]
        ks = run(569, 32768)
        assert ks > 1 and ks * 569 * 32768 * 4 > 128 * MiB               # twice this launch's bytes would be more than the bound
        image = 1024 * (K * 2 + K // 256 * 32 + 8)
        assert before - torch.cuda.mem_get_info()[0] <= image + 256 * MiB + 4 * MiB
        assert run(809, 57344) == 1                                       # two ranges: 353 MiB


class PromptImage(ctypes.Structure):
    """csrc/prompt_image.h"""
    _fields_ = [("buf", ctypes.c_void_p), ("bytes", ctypes.c_size_t), ("valid", ctypes.c_bool), ("live", ctypes.c_int32), ("rows", ctypes.c_int32),
                ("K", ctypes.c_int32), ("half", ctypes.c_int32), ("norm", ctypes.c_void_p), ("x", ctypes.c_void_p), ("eps", ctypes.c_float), ("next", ctypes.c_bool), ("want_parts", ctypes.c_bool),
                ("ks", ctypes.c_int32), ("ldp", ctypes.c_int32), ("parts", ctypes.c_void_p), ("scale", ctypes.c_void_p)]


@pytest.mark.parametrize("T,hid,inter,kinds,staged", [(41, 2048, 8192, (Q4, Q4, Q4), 2), (73, 3072, 8192, (Q6, Q4, Q6), 2), (193, 2048, 4096, (Q4, Q4, Q6), 2),
                                                      (42, 1024, 16640, (Q4, Q4, Q4), 1)])
def test_image_handed_on(T, hid, inter, kinds, staged):
    """wo (residual) -> gate/up -> down as a prompt step runs them, the image handed on (after wo, and after gate/up up to 16384 columns) against every
    product building its own: the same bits (the sums, also that of the squares, have the same order)"""
    rng = np.random.default_rng(T)
    shapes = ((hid, hid, kinds[0]), (inter, hid, kinds[1]), (inter, hid, kinds[1]), (hid, inter, kinds[2]))
    ms = [cv.QMatMul(blocks(rng, n, k, t, odd=False), t, "cuda") for n, k, t in shapes]
    attn = torch.from_numpy(rng.normal(0, 1, (T, hid)).astype(np.float32)).cuda().bfloat16()
    start = torch.from_numpy(rng.normal(0, 1, (T, hid)).astype(np.float32)).cuda()
    norm = 1 + 0.1 * torch.randn(hid, device="cuda")
    fn = cv.lib.mi355_internal_qmatmul_prompt
    fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64], ctypes.c_int
    room = 16384 + (T + 255) // 256 * 256 * (inter * 2 + inter // 256 * 32)
    buf = torch.full((room,), 255, dtype=torch.uint8, device="cuda")              # NaN patterns: what is read has been written
    results = []
    for hand_on in (False, True):
        xs, h = start.clone(), torch.empty(T, inter, device="cuda")
        io = PromptImage(buf.data_ptr(), room, eps=0.3)                          # (an eps that shows)
        seen = []
        for x, ws, nw, epi, out in ((attn, ms[:1], None, cv.EPI_RESID, xs), (xs, ms[1:3], norm, cv.EPI_SILU_MUL, h), (h, ms[3:], None, cv.EPI_RESID, xs)):
            d = _desc(x, ws, nw, epi, out)
            d.chain_next, d.chain_next_k = int(hand_on and x is not h), out.shape[1]
            d.chain_next_norm = norm.data_ptr() if x is attn else None
            assert fn(ctypes.byref(d), ctypes.byref(io), torch.cuda.current_stream().cuda_stream) == 0
            seen.append(bool(io.valid))
            if x is attn:
                first = xs.clone()
        assert seen == [hand_on, hand_on and staged == 2, False]
        results.append((first, h, xs))
    torch.cuda.synchronize()
    (f0, h0, x0), (f1, h1, x1) = results
    assert torch.isfinite(x0).all() and torch.equal(f0, f1) and torch.equal(h0, h1) and torch.equal(x0, x1)


def test_image_of_other_values_is_not_taken():
    """a product whose x is not the output that the image was made of, with the same rows, columns and norm, builds its own"""
    rng = np.random.default_rng(8)
    T, K = 73, 2048
    a, b = (cv.QMatMul(blocks(rng, K, K, Q4, odd=False), Q4, "cuda") for _ in range(2))
    x, other = (torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda() for _ in range(2))
    norm = 1 + 0.1 * torch.randn(K, device="cuda")
    xs, want, got = x.clone(), torch.empty(T, K, device="cuda"), torch.empty(T, K, device="cuda")
    fn, st = cv.lib.mi355_internal_qmatmul_prompt, torch.cuda.current_stream().cuda_stream
    fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64], ctypes.c_int
    room = 16384 + 256 * (K * 2 + K // 256 * 32)
    buf = torch.zeros(room, dtype=torch.uint8, device="cuda")
    io = PromptImage(buf.data_ptr(), room, eps=0.3)
    d = _desc(x, [a], None, cv.EPI_RESID, xs)
    d.chain_next, d.chain_next_k, d.chain_next_norm = 1, K, norm.data_ptr()
    assert fn(ctypes.byref(d), ctypes.byref(io), st) == 0 and io.valid
    assert fn(ctypes.byref(_desc(other, [b], norm, cv.EPI_STORE, got)), ctypes.byref(io), st) == 0 and not io.valid
    assert cv.lib.mi355_qmatmul_fused(ctypes.byref(_desc(other, [b], norm, cv.EPI_STORE, want)), st) == 0
    assert torch.equal(got, want)


def _desc(x, ws, nw, epi, out):
    from candle_vllm_amd._lib import QmmDesc
    d = QmmDesc()
    d.nseg = len(ws)
    for i, w in enumerate(ws):
        d.w_tiles[i], d.ggml_type[i], d.n_rows[i] = w.tiles.data_ptr(), w.ggml_type, w.n
    d.x, d.x_dtype = x.data_ptr(), cv.DT_F32 if x.dtype == torch.float32 else cv.DT_BF16
    d.ldx = d.k = x.shape[1]
    d.num_tokens, d.norm_weight, d.norm_eps = x.shape[0], nw.data_ptr() if nw is not None else None, 0.3 if nw is not None else 0.0
    d.epilogue, d.out, d.ldo, d.residual = epi, out.data_ptr(), out.shape[1], out.data_ptr() if epi == cv.EPI_RESID else None
    return d


@pytest.mark.parametrize("layout,D,rot,T", [("flash", 128, 64, 73), ("fp8", 128, 128, 41), ("paged", 72, 24, 130), ("fp8", 64, 32, 97), ("paged", 64, 64, 41)])
def test_qkv_sums_by_eights(layout, D, rot, T):
    """the launch that adds the ranges up, turns q and k and writes the cache eight columns at a time: every layout, rotated parts that end inside
    a head, heads that are no whole row tiles' multiple, tokens without a slot; one rounding to bf16 (2^-8), for an e4m3 cache one more (2^-4)"""
    H, Hkv, K, block = 8, 2, 2048, 16
    rng = np.random.default_rng(T)
    heads = (H, Hkv, Hkv)
    bs = [blocks(rng, n * D, K, Q4, odd=False) for n in heads]
    ms = [cv.QMatMul(b, Q4, "cuda") for b in bs]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    pos, slot = torch.from_numpy(rng.integers(0, 500, T)).cuda(), torch.from_numpy(rng.permutation(T + 64)[:T].astype(np.int64)).cuda()
    slot[::7] = -1
    ang = torch.arange(500, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(rot // 2, device="cuda").double() / (rot // 2))
    nb = (T + 64 + block - 1) // block
    x16 = 16 if layout == "fp8" else 8
    dt = torch.uint8 if layout == "fp8" else torch.bfloat16
    kc = torch.zeros((nb, block, Hkv, D) if layout == "flash" else (nb, Hkv, D // x16, block, x16), dtype=dt, device="cuda")
    vc = torch.zeros((nb, block, Hkv, D) if layout == "flash" else (nb, Hkv, D, block), dtype=dt, device="cuda")
    q_out = torch.zeros(T, H * D, dtype=torch.bfloat16, device="cuda")
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()
    d = _desc(x, ms, None, cv.EPI_QKV_ROPE_CACHE, q_out)
    d.out, d.ldo = None, 0
    d.cos_table, d.sin_table, d.positions, d.slot_mapping = (v.data_ptr() for v in (cos, sin, pos, slot))
    d.q_out, d.key_cache, d.value_cache = q_out.data_ptr(), kc.data_ptr(), vc.data_ptr()
    d.num_heads, d.num_kv_heads, d.head_dim, d.rotary_dim, d.block_size = H, Hkv, D, rot, block
    d.kv_layout = {"flash": cv.KV_FLASH, "paged": cv.KV_PAGED, "fp8": KV_PAGED_FP8}[layout]
    assert cv.lib.mi355_qmatmul_fused(ctypes.byref(d), torch.cuda.current_stream().cuda_stream) == 0
    assert last_split() > 1
    y = [product(x, b, Q4).view(T, -1, D) for b in bs]
    c, s = ang.cos()[pos][:, None], ang.sin()[pos][:, None]
    turned = [torch.cat([torch.stack([z[..., 0:rot:2] * c - z[..., 1:rot:2] * s, z[..., 0:rot:2] * s + z[..., 1:rot:2] * c], dim=-1).reshape(T, -1, rot), z[..., rot:]], -1) for z in y[:2]]
    ok = slot >= 0
    blk, off = slot[ok] // block, slot[ok] % block
    if layout == "fp8":
        kc, vc = kc.view(torch.float8_e4m3fn).float(), vc.view(torch.float8_e4m3fn).float()
        big = max(turned[1].abs().max(), y[2].abs().max()).item()
        assert big < 448, big                                         # nothing saturates
    gk = kc[blk, off] if layout == "flash" else kc[blk, :, :, off].reshape(-1, Hkv, D)
    gv = vc[blk, off] if layout == "flash" else vc[blk, :, :, off]
    cache_tol = TOL + 2.0 ** -8 + (2.0 ** -4 if layout == "fp8" else 0)
    for got, want, tol in ((q_out.view(T, H, D), turned[0], TOL + 2.0 ** -8), (gk, turned[1][ok], cache_tol), (gv, y[2][ok], cache_tol)):
        assert close(got.float(), want) < tol


@pytest.mark.parametrize("kind,counts", [(Q4, (5, 64, 0, 65)), (Q6, (1, 0, 130, 63)), (Q4, (0, 0, 0, 1))])
def test_down_of_experts_in_ranges_of_k(kind, counts):
    """a mixture's down product over its block table, sums of ranges of K and the launch that adds them into the residual: experts without rows, of one row,
    of whole blocks and of one row more; against dequantised weights in 64 bits, every row of the sums that belongs to a pair"""
    E, K, hid, top = len(counts), 4096, 512, 2
    rng = np.random.default_rng(sum(counts))
    bs = [blocks(rng, hid, K, kind, odd=False) for _ in range(E)]
    ms = [cv.QMatMul(b, kind, "cuda") for b in bs]
    slab = torch.cat([m.tiles.view(torch.uint8).reshape(-1) for m in ms])
    first, table, rows_of = 0, [], []
    for e, c in enumerate(counts):
        nb = -(-c // 64)
        table += [(e, 64 * first + c)] * nb
        rows_of += [(e, 64 * first + i) for i in range(c)]
        first += nb
    table += [(0, 0)] * 3                                             # blocks behind the last expert's: nothing to do
    T = 64 * len(table)
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    out = torch.empty(T, hid, device="cuda")
    tab = torch.tensor(table, dtype=torch.int32, device="cuda")
    d = _desc(x, ms[:1], None, cv.EPI_STORE, out)
    d.w_tiles[0], d.moe_expert_stride[0], d.group_block_table = slab.data_ptr(), slab.numel() // E, tab.data_ptr()
    fn = cv.lib.mi355_internal_qmatmul_prompt
    fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64], ctypes.c_int
    st = torch.cuda.current_stream().cuda_stream
    io = PromptImage(want_parts=True)
    assert fn(ctypes.byref(d), ctypes.byref(io), st) == 0 and io.ks > 1
    order = rng.permutation(len(rows_of))
    pairs = (len(rows_of) // top) * top
    toks = max(1, pairs // top)
    picked = [rows_of[order[i % len(rows_of)]] for i in range(toks * top)]
    inv = torch.tensor([r for _, r in picked], dtype=torch.int32, device="cuda")
    w = torch.from_numpy(rng.uniform(0.1, 1, toks * top).astype(np.float32)).cuda()
    ys0 = torch.from_numpy(rng.normal(0, 1, (toks, hid)).astype(np.float32)).cuda()
    ys = ys0.clone()
    comb = cv.lib.mi355_internal_moe_combine_parts
    vp, i32 = ctypes.c_void_p, ctypes.c_int32
    comb.argtypes, comb.restype = [vp, vp, i32, i32, i32, vp, vp, vp, i32, i32, i32, ctypes.c_int64], ctypes.c_int
    assert comb(ys.data_ptr(), io.parts, io.ks, T, io.ldp, io.scale, w.data_ptr(), inv.data_ptr(), toks, hid, top, st) == 0
    want = ys0.double()
    for p, (e, r) in enumerate(picked):
        want[p // top] += w[p].double() * product(x[r:r + 1], bs[e], kind)[0]
    assert close(ys, want) < TOL
    d2 = _desc(x, ms[:1], None, cv.EPI_STORE, out)                    # the call without the wish: outputs, as before
    d2.w_tiles[0], d2.moe_expert_stride[0], d2.group_block_table = d.w_tiles[0], d.moe_expert_stride[0], d.group_block_table
    assert cv.lib.mi355_qmatmul_fused(ctypes.byref(d2), st) == 0
    for e, r in picked[:8]:
        assert close(out[r], product(x[r:r + 1], bs[e], kind)[0]) < 2 * TOL


@pytest.mark.parametrize("kind,epi,counts,N,K", [(Q4, cv.EPI_SILU_MUL, (256, 1, 0, 129, 128, 300), 1040, 512), (Q4, cv.EPI_STORE, (65, 513, 0), 528, 1024), (Q4, cv.EPI_STORE, (0, 0, 31), 16640, 256),
                                                 (Q6, cv.EPI_STORE, (64, 65, 0, 257, 192, 193), 272, 512), (Q6, cv.EPI_STORE, (1, 320), 4112, 256)])
def test_experts_in_whole_tiles(kind, epi, counts, N, K):
    """a mixture's prompt products whose experts own whole tiles of 256 rows: experts without rows, of one row, whose last tile leaves a part of the waves without rows, and
    of whole tiles; positions and table, every stored row against dequantised weights in 64 bits, no other row touched"""
    E = len(counts)
    rng = np.random.default_rng(sum(counts) + N)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)
    nblk = 4 * (-(-len(ids) // 256) + E)
    tab = torch.full((nblk + 2, 2), -7, dtype=torch.int32, device="cuda")
    pos = torch.empty(len(ids), dtype=torch.int32, device="cuda")
    st, ids_d = torch.cuda.current_stream().cuda_stream, torch.from_numpy(ids).cuda()
    fn = cv.lib.mi355_internal_moe_group_tiles
    vp, i32 = ctypes.c_void_p, ctypes.c_int32
    fn.argtypes, fn.restype = [vp, vp, vp, i32, i32, i32, ctypes.c_int64], ctypes.c_int
    assert fn(pos.data_ptr(), tab.data_ptr(), ids_d.data_ptr(), len(ids), E, nblk + 2, st) == 0
    assert fn(pos.data_ptr(), tab.data_ptr(), ids_d.data_ptr(), len(ids), E, nblk - 1, st) != 0   # table too short
    cv.lib.mi355_clear_error()
    want_tab = np.zeros((nblk + 2, 2), np.int32)
    row_of, at = [np.empty(c, np.int64) for c in counts], 0
    for part in (0, 1):                                               # full tiles, then what is left of every expert
        for e, c in enumerate(counts):
            lo, hi = (0, c // 256 * 256) if part == 0 else (c // 256 * 256, c)
            row_of[e][lo:hi] = at + np.arange(hi - lo)
            want_tab[at // 64:-(-(at + hi - lo) // 256) * 4] = (e, at + hi - lo)
            at += -(-(hi - lo) // 256) * 256
    want_pos = np.empty(len(ids), np.int32)
    for e in range(E):
        want_pos[ids == e] = row_of[e]
    assert np.array_equal(pos.cpu().numpy(), want_pos) and np.array_equal(tab.cpu().numpy(), want_tab)
    T, n_w = 64 * nblk, 2 if epi == cv.EPI_SILU_MUL else 1
    bs = [[blocks(rng, N, K, kind) for _ in range(E)] for _ in range(n_w)]
    ms = [[cv.QMatMul(b, kind, "cuda") for b in w] for w in bs]
    slabs = [torch.cat([m.tiles.view(torch.uint8).reshape(-1) for m in w]) for w in ms]
    x = torch.from_numpy(rng.normal(0, 1, (T, K)).astype(np.float32)).cuda()
    out = torch.full((T, N), float("nan"), device="cuda")
    d = _desc(x, [w[0] for w in ms], None, epi, out)
    for i, s in enumerate(slabs):
        d.w_tiles[i], d.moe_expert_stride[i] = s.data_ptr(), s.numel() // E
    d.group_block_table = tab.data_ptr()
    fn = cv.lib.mi355_internal_qmatmul_prompt
    fn.argtypes, fn.restype = [vp, vp, ctypes.c_int64], ctypes.c_int
    ms[0][0].forward(torch.full((T, K), float("nan"), device="cuda"))      # what the image's rows behind a group's end hold
    io = PromptImage()
    ctypes.c_int16.from_buffer(io, PromptImage.want_parts.offset + 1).value = -1   # tiles: between want_parts and ks
    assert fn(ctypes.byref(d), ctypes.byref(io), st) == 0 and last_tile() == (20 if kind == Q4 else 21)
    live = torch.zeros(T, dtype=torch.bool, device="cuda")
    for e, c in enumerate(counts):
        if c == 0:
            continue
        r = torch.from_numpy(row_of[e]).cuda()
        live[r] = True
        want = [product(x[r], w[e], kind) for w in bs]
        if n_w == 2:                                                  # (the product of two: twice the error of one)
            assert close(out[r], torch.nn.functional.silu(want[0]) * want[1]) < 2 * TOL
        else:
            assert close(out[r], want[0]) < TOL
    assert torch.isnan(out[~live]).all()
