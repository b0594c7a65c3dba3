"""GPU parity tests for the safetensors path (K10, K12-K15): dense 16-bit and GPTQ/AWQ/Marlin 4-bit linears through
the C ABI vs the numpy oracle.  Repack / permutation results are bit-exact; matmul outputs are 16-bit values
compared at 1 ulp of the output dtype (tolerance next to the assert)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import gptq as G               # noqa: E402

TD = {"bf16": torch.bfloat16, "f16": torch.float16}
ULP = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}


@pytest.fixture(scope="module")
def cv(lib):
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X (torch.cuda.is_available() is False)")
    import candle_vllm_amd.ops as ops
    return ops


def dev16(a_f32, dt):
    """f32 numpy values (already exactly representable) -> 16-bit cuda tensor, bit-exact"""
    bits = G.to_bits(a_f32, dt)
    return torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).cuda().view(TD[dt])


def host16(t, dt):
    return G.from_bits(t.detach().view(torch.int16).cpu().numpy().view(np.uint16), dt)


def dev_u32(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


def check_ulp(got, ref, dt, ulps=1.01, what="", mag=None):
    """|got-ref| <= ulps * ulp(mag) elementwise (mag = |ref|, or the largest intermediate of a rounding chain:
    a 1-ulp flip of the matmul result survives a cancelling bias / residual add), plus a small absolute floor for
    cancellation inside the dot product (f32 accumulation order differs from the f64 oracle)."""
    got, ref = np.asarray(got, np.float64), np.asarray(ref, np.float64)
    mag = np.abs(ref) if mag is None else np.maximum(np.abs(ref), np.abs(mag))
    tol = ulps * 2 * ULP[dt] * mag                              # ulp(v) <= 2 * 2^-p * |v|
    floor = 1e-3 * np.abs(ref).max() * (ULP[dt] / ULP["bf16"])
    bad = np.abs(got - ref) > np.maximum(tol, floor)
    assert not bad.any(), f"{what}: {bad.sum()} / {bad.size} off, max abs err {np.abs(got - ref).max()}"


# ------------------------------------------------------------------------------------------------ K10 dense
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K", [(1, 256, 512), (5, 48, 256), (16, 1024, 1024), (17, 64, 768), (33, 128, 512),
                                   (64, 96, 256), (70, 32, 512), (128, 64, 512), (200, 48, 256),
                                   (256, 384, 1024), (300, 200, 576), (97, 130, 64)])   # (64, 96, 256) and more tokens: the MFMA GEMM (ragged T / N tiles, one K step)
def test_linear_matches_oracle(cv, dt, T, N, K):
    rng = np.random.default_rng(T * 1000 + N)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    w = G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
    b = G.round_dt(rng.normal(0, 0.2, N), dt)
    lin = cv.Linear(dev16(w, dt), dev16(b, dt))
    y = host16(lin.forward(dev16(x, dt)), dt)
    check_ulp(y, G.linear16(x, w, b, dt), dt, what="linear+bias", ulps=2.01, mag=G.linear16(x, w, None, dt))
    lin2 = cv.Linear(dev16(w, dt))
    res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
    y2 = host16(lin2.forward(dev16(x, dt), epilogue=cv.EPI_RESID, residual=dev16(res, dt)), dt)
    check_ulp(y2, G.round_dt(G.linear16(x, w, None, dt) + res, dt), dt, what="linear+resid", ulps=2.01,
              mag=G.linear16(x, w, None, dt))


@pytest.mark.parametrize("T,N,K,kind,made", [(5, 16, 8192, 0, True), (8, 1040, 8192, 1, True), (16, 2064, 8192, 1, True), (32, 4096, 8192, 1, True), (20, 8192, 8192, 0, True),
                                             (7, 8208, 8192, 1, False), (8, 2064, 1024, 1, False), (3, 1040, 8192, 1, False),     # too long a row; sums in one range
                                             (5, 1040, 8192, 2, True), (16, 3584, 18944, 2, True), (32, 2064, 8192, 2, True), (16, 2064, 512, 2, False)])
def test_residual_product_with_the_norm_behind_it(cv, T, N, K, kind, made):
    """a residual product that also leaves the RmsNorm of its output: where the split sums' launch makes it, the output equals the plain product's to the bit and the
    norm is the norm launch's of that output, up to the order of one f32 sum (an ulp where a value is on the edge of two)"""
    import ctypes

    from candle_vllm_amd._lib import lib
    dt, st, rng = "bf16", torch.cuda.current_stream().cuda_stream, np.random.default_rng(T + N + kind)
    x, res, nw = dev16(G.round_dt(rng.normal(0, 1, (T, K)), dt), dt), dev16(G.round_dt(rng.normal(0, 1, (T, N)), dt), dt), dev16(G.round_dt(rng.normal(1, 0.1, N), dt), dt)
    want = torch.empty(T, N, dtype=torch.bfloat16, device="cuda")
    sc = None
    if kind == 2:
        q, s = _gptq_case(rng, K, N, 128, dt)
        lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), 128)
        w, sc = lin.qweight, lin.scales
        want = lin.forward(x, epilogue=cv.EPI_RESID, residual=res)
    else:
        w = dev16(G.round_dt(rng.normal(0, 0.02, (N, K)), dt), dt)
        if kind == 1:
            w, flat = torch.empty_like(w), w
            assert lib.mi355_dense_tile_repack(flat.data_ptr(), w.data_ptr(), N, K, K, st) == 0
        assert (lib.mi355_linear_tiled if kind else lib.mi355_linear)(want.data_ptr(), x.data_ptr(), w.data_ptr(), None, res.data_ptr(), T, N, K, 2, 1, st) == 0
    out, normed, done = res.clone(), torch.full((T, N), 7.0, dtype=torch.bfloat16, device="cuda"), ctypes.c_int32(-1)
    fused = lib.mi355_internal_resid_norm_linear
    fused.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int32] * 6 + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float, ctypes.c_void_p, ctypes.c_int64]
    assert fused(out.data_ptr(), x.data_ptr(), w.data_ptr(), sc.data_ptr() if sc is not None else None, out.data_ptr(), T, N, K, 128, kind, 2,
                 normed.data_ptr(), nw.data_ptr(), 1e-5, ctypes.addressof(done), st) == 0
    assert torch.equal(out, want.view(T, N)) and done.value == int(made)
    if not made:
        assert bool((normed == 7).all())
        return
    ref = torch.empty_like(normed)
    assert lib.mi355_rms_norm(ref.data_ptr(), out.data_ptr(), nw.data_ptr(), T, N, 1e-5, 2, 2, st) == 0
    a, b = normed.view(torch.int16).int(), ref.view(torch.int16).int()
    assert int((a - b).abs().max()) <= 1 and float((a != b).float().mean()) < 0.01


@pytest.mark.parametrize("B,V", [(1, 1), (1, 3), (3, 4), (2, 1020), (1, 1024), (5, 1027), (1, 4100), (33, 8192), (9, 32001), (1, 151936), (300, 2052)])
@pytest.mark.parametrize("skew", [0, 1])
def test_argmax_slices(cv, B, V, skew):
    """the first of the largest logits of every row, whatever slice it is in: ties, NaN (never), infinities, rows of nothing else; rows on and off 16 bytes;
    the slots are clear again for the next call, whose logits are all below this one's, the largest of them last"""
    rng = np.random.default_rng(B + V)
    x = np.round(rng.normal(0, 2, (B, V)), 1).astype(np.float32)            # many ties
    x[rng.random((B, V)) < 0.05] = np.nan
    x[0, V // 2] = np.inf
    x[-1, :] = np.nan if V % 2 else -np.inf
    buf = torch.empty(B * V + skew, device="cuda")
    d = buf[skew:].view(B, V)
    d.copy_(torch.from_numpy(x))
    want = np.where(np.isnan(x).all(1), 0, np.argmax(np.where(np.isnan(x), -np.inf, x), 1))
    want = np.where((np.nan_to_num(x, nan=-np.inf) == -np.inf).all(1) & ~np.isnan(x).all(1), np.argmax(~np.isnan(x), 1), want)
    below = torch.linspace(-9e3, -8e3, V, device="cuda").repeat(B, 1)
    for _ in range(2):
        assert np.array_equal(cv.argmax(d).cpu().numpy(), want)
        assert bool((cv.argmax(below) == V - 1).all())


def test_argmax_behind_an_error_of_the_callers(cv):
    """an error that an earlier call of the caller's left behind is reported, and costs neither this call's winners nor the next one's"""
    import ctypes

    from candle_vllm_amd._lib import lib
    hip, st = ctypes.CDLL("libamdhip64.so.7"), torch.cuda.current_stream().cuda_stream
    high, low, out = torch.zeros(3, 5000, device="cuda"), torch.zeros(3, 5000, device="cuda"), torch.full((3,), 7, dtype=torch.int32, device="cuda")
    high[:, 40], low[:, 4000] = 2.0, 1.0
    cv.argmax(low)
    torch.cuda.synchronize()
    assert hip.hipSetDevice(1 << 20) != 0                                   # (a number that no card has: the call is refused, and leaves its error)
    assert lib.mi355_argmax_f32(out.data_ptr(), high.data_ptr(), 3, 5000, st) != 0
    assert out.tolist() == [40] * 3 and cv.argmax(low).tolist() == [4000] * 3


def test_argmax_two_threads_on_one_stream(cv):
    """the winners pass from one launch to the next in the stream's slots: two threads on one stream, each over its own logits, have their own winners"""
    import threading
    xs = [torch.zeros(40, 3000, device="cuda") for _ in range(2)]
    xs[0][:, 2900], xs[1][:, 17] = 1.0, 2.0
    got, go = [[], []], threading.Barrier(2)

    def work(i):
        go.wait()
        got[i] = [cv.argmax(xs[i]) for _ in range(400)]
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    torch.cuda.synchronize()
    for i, at in enumerate((2900, 17)):
        assert len(got[i]) == 400 and all(bool((g == at).all()) for g in got[i])


@pytest.mark.parametrize("T,N,K,epi", [(1153, 4096, 1024, 0), (2100, 2050, 2048, 0), (1344, 4080, 1280, 1), (1345, 4096, 1024, 2)])
def test_linear_prompt_gemm_tall_narrow_tile(cv, T, N, K, epi):
    """the prompt GEMM's 192 x 128 tile: one token into the last tile, ragged tokens and rows, each epilogue; row-major and tiled weights alike bit for bit, and
    the sums within the op's bound of the oracle at the tiles' edges"""
    from candle_vllm_amd._lib import lib
    dt, st = "bf16", torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(T + N)
    x, w, res = G.round_dt(rng.normal(0, 1, (T, K)), dt), G.round_dt(rng.normal(0, 0.05, (N, K)), dt), G.round_dt(rng.normal(0, 1, (T, N)), dt)
    xd, wd, rd = dev16(x, dt), dev16(w, dt), dev16(res, dt)
    images, outs = [(lib.mi355_linear, wd)], []
    if N % 16 == 0 and K % 256 == 0:
        images.append((lib.mi355_linear_tiled, torch.empty_like(wd)))
        assert lib.mi355_dense_tile_repack(wd.data_ptr(), images[1][1].data_ptr(), N, K, K, st) == 0
    for fn, img in images:
        out = torch.full((T, N // 2 if epi == 2 else N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert fn(out.data_ptr(), xd.data_ptr(), img.data_ptr(), None, rd.data_ptr() if epi == 1 else None, T, N, K, 2, epi, st) == 0
        assert lib.mi355_internal_last_gemm() == 501              # 100 tile + K ranges
        outs.append(host16(out, dt))
    assert all(np.array_equal(outs[0], o) for o in outs) and np.isfinite(outs[0]).all()
    rows = np.unique([t for e in range(0, T, 192) for t in (e, e + 1, e + 95, e + 191, T - 1) if t < T])
    y = G.linear16(x[rows], w, None, dt)
    if epi == 2:
        check_ulp(outs[0][rows], G.silu_mul16(y[:, :N // 2], y[:, N // 2:], dt), dt, ulps=3.0, what="silu(gate)*up")
    else:
        check_ulp(outs[0][rows], G.round_dt(y + res[rows], dt) if epi == 1 else y, dt, what="linear", ulps=2.01, mag=y)


@pytest.mark.parametrize("T,N,K,launch", [(33, 288, 2304, 404), (65, 160, 4096, 408),          # 64-token tiles, K in 4 and 8 ranges; one token into the next tile
                                          (130, 96, 8192, 416),                                # K in 16 ranges over three token tiles
                                          (900, 8192, 128, 201),                               # 128 x 128 tiles, exactly two per CU
                                          (1030, 2560, 704, 301),                              # 128 x 128 tiles, one per CU
                                          (1530, 8192, 128, 101),                              # 192 x 256 tiles, exactly one per CU, ragged tokens
                                          (1540, 8208, 128, 1),                                # 256 x 256 tiles, ragged both ways
                                          (162, 4256, 8192, 507),                              # 192 x 128 tiles, K in 7 ranges, where a two-buffered tile's are longer
                                          (185, 6880, 3072, 401), (903, 1152, 7936, 303)])     # ... and never where the tiles of six or four buffers serve
def test_linear_prompt_gemm_every_tile(cv, T, N, K, launch):
    """16-bit prompt GEMM where its dispatch takes each of its tiles and K splits: row-major and tiled weights alike bit for bit, and within the
    op's bound of the oracle (tokens and rows at the tile's edges and at the matrix's)"""
    from candle_vllm_amd._lib import lib
    dt, st = "bf16", torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(T + N + K)
    x, w = G.round_dt(rng.normal(0, 1, (T, K)), dt), G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
    b, res = G.round_dt(rng.normal(0, 0.2, N), dt), G.round_dt(rng.normal(0, 1, (T, N)), dt)
    xd, wd, bd, rd = dev16(x, dt), dev16(w, dt), dev16(b, dt), dev16(res, dt)
    tiled = None
    if K % 256 == 0:
        tiled = torch.empty_like(wd)
        assert lib.mi355_dense_tile_repack(wd.data_ptr(), tiled.data_ptr(), N, K, K, st) == 0
    rows = np.unique(np.concatenate([np.arange(0, T, max(1, T // 40)), [t for e in (63, 64, 127, 128, 191, 192, 255, 256) for t in (e, T - 1 - e) if 0 <= t < T], [T - 1]])).astype(np.int64)
    I = N // 2
    for epi, bias, resid, n_out in ((0, bd, None, N), (1, None, rd, N), (2, None, None, I)):
        outs = []
        for fn, img in ((lib.mi355_linear, wd), (lib.mi355_linear_tiled, tiled)):
            if img is None:
                continue
            out = torch.full((T, n_out), float("nan"), dtype=torch.bfloat16, device="cuda")
            assert fn(out.data_ptr(), xd.data_ptr(), img.data_ptr(), bias.data_ptr() if bias is not None else None,
                      resid.data_ptr() if resid is not None else None, T, N, K, 2, epi, st) == 0
            assert lib.mi355_internal_last_gemm() == launch       # 100 tile + K ranges
            outs.append(host16(out, dt))
        assert len(outs) == 1 or np.array_equal(outs[0], outs[1])
        y = G.linear16(x[rows], w, None, dt)
        if epi == 0:
            check_ulp(outs[0][rows], G.linear16(x[rows], w, b, dt), dt, what="linear+bias", ulps=2.01, mag=y)
        elif epi == 1:
            check_ulp(outs[0][rows], G.round_dt(y + res[rows], dt), dt, what="linear+resid", ulps=2.01, mag=y)
        else:
            check_ulp(outs[0][rows], G.silu_mul16(y[:, :I], y[:, I:], dt), dt, ulps=3.0, what="silu(gate)*up")
        assert np.isfinite(outs[0]).all()


@pytest.mark.parametrize("T", [17, 33, 100])
@pytest.mark.parametrize("off_x,off_w", [(4, 0), (0, 4)])
def test_linear_prompt_operands_off_the_16_byte_grid(cv, T, off_x, off_w):
    """x or w that do not start on 16 bytes stay with the kernels that read them element-aligned: same bound (the GEMM copies 16-byte pieces)"""
    from candle_vllm_amd._lib import lib
    dt, N, K, st = "bf16", 96, 512, torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(T + 8 * off_x + off_w)
    x, w = G.round_dt(rng.normal(0, 1, (T, K)), dt), G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
    xd, wd = (torch.zeros(v.size + 8, dtype=torch.bfloat16, device="cuda") for v in (x, w))
    xd[off_x:off_x + x.size], wd[off_w:off_w + w.size] = dev16(x, dt).flatten(), dev16(w, dt).flatten()
    out = torch.empty((T, N), dtype=torch.bfloat16, device="cuda")
    assert lib.mi355_linear(out.data_ptr(), xd[off_x:].data_ptr(), wd[off_w:].data_ptr(), None, None, T, N, K, 2, 0, st) == 0
    check_ulp(host16(out, dt), G.linear16(x, w, None, dt), dt, what="unaligned operands")


@pytest.mark.parametrize("T,N,K", [(96, 72, 576), (150, 130, 64), (100, 96, 512)])
@pytest.mark.parametrize("off_x,off_w", [(4, 0), (0, 1), (3, 4)])
def test_linear_prompt_operands_off_the_grid_of_any_shape(cv, T, N, K, off_x, off_w):
    """from 96 tokens any rows and any k that is a multiple of 64 are served, also from operands that do not start on 16 bytes"""
    from candle_vllm_amd._lib import lib
    dt, st = "bf16", torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(T + 8 * off_x + off_w)
    x, w, res = G.round_dt(rng.normal(0, 1, (T, K)), dt), G.round_dt(rng.normal(0, 0.05, (N, K)), dt), G.round_dt(rng.normal(0, 1, (T, N)), dt)
    xd, wd = (torch.zeros(v.size + 8, dtype=torch.bfloat16, device="cuda") for v in (x, w))
    xd[off_x:off_x + x.size], wd[off_w:off_w + w.size] = dev16(x, dt).flatten(), dev16(w, dt).flatten()
    out, rd, y = torch.empty((T, N), dtype=torch.bfloat16, device="cuda"), dev16(res, dt), G.linear16(x, w, None, dt)
    assert lib.mi355_linear(out.data_ptr(), xd[off_x:].data_ptr(), wd[off_w:].data_ptr(), None, rd.data_ptr(), T, N, K, 2, 1, st) == 0
    check_ulp(host16(out, dt), G.round_dt(y + res, dt), dt, ulps=2.01, what="unaligned operands", mag=y)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K", [(256, 384, 1024), (300, 200, 576), (97, 130, 64), (700, 128, 256)])
def test_linear_prompt_gemm_tall_tile(cv, dt, T, N, K):
    """the 256 x 256 tile of the 16-bit prompt GEMM (tuning key 30 bits 32 | 64 = wherever the GEMM runs): the same as the 64-token tile these launches
    take by themselves -- bit for bit (K in one range, the same order per output element) -- and within the op's bound of the oracle; plain, residual and
    SiLU * up launches, ragged token / column tiles"""
    from candle_vllm_amd import lib, tuning
    rng = np.random.default_rng(T * 7 + N)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    w = G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
    b = G.round_dt(rng.normal(0, 0.2, N), dt)
    res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
    I = N // 2
    lin, lin2 = cv.Linear(dev16(w, dt), dev16(b, dt)), cv.Linear(dev16(w, dt))

    def run():
        y = host16(lin.forward(dev16(x, dt)), dt)
        y2 = host16(lin2.forward(dev16(x, dt), epilogue=cv.EPI_RESID, residual=dev16(res, dt)), dt)
        y3 = host16(lin2.forward(dev16(x, dt), epilogue=cv.EPI_SILU_MUL), dt)
        return y, y2, y3

    base = run()
    assert lib.mi355_internal_last_gemm() == 401
    with tuning(30, 32 | 64):
        tall = run()
    assert lib.mi355_internal_last_gemm() == 1
    for a_, b_ in zip(base, tall):
        assert np.array_equal(np.asarray(a_), np.asarray(b_))
    check_ulp(tall[0], G.linear16(x, w, b, dt), dt, what="linear+bias", ulps=2.01, mag=G.linear16(x, w, None, dt))
    gu = G.linear16(x, w, None, dt)
    check_ulp(tall[2], G.silu_mul16(gu[:, :I], gu[:, I:], dt), dt, ulps=3.0, what="silu(gate)*up")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T", [1, 8, 32, 40, 130, 257])
def test_linear_gate_up_silu(cv, dt, T):
    rng = np.random.default_rng(T)
    K, I = (512, 192) if T != 257 else (1024, 328)              # 257 tokens: three token tiles, 5.1 column tiles of the prompt GEMM
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    w = G.round_dt(rng.normal(0, 0.06, (2 * I, K)), dt)          # packed [gate; up] (mlp.rs:324-352)
    lin = cv.Linear(dev16(w, dt))
    y = host16(lin.forward(dev16(x, dt), epilogue=cv.EPI_SILU_MUL), dt)
    gu = G.linear16(x, w, None, dt)
    ref = G.silu_mul16(gu[:, :I], gu[:, I:], dt)
    # the 1-ulp differences of gate/up (f32 vs f64 accumulation) propagate through silu*up: 3 ulp
    check_ulp(y, ref, dt, ulps=3.0, what="silu(gate)*up")


# ------------------------------------------------------------------------------------------------ K15 repack
def test_repack_bit_exact(cv):
    rng = np.random.default_rng(3)
    K, N = 512, 128
    q = rng.integers(0, 16, (K, N))
    gq = G.gptq_pack(q)
    tiled = G.gptq_tile(gq)                                       # numpy statement of the library's 16 x 256 tile order
    out = cv.marlin_weight_repack(dev_u32(gq), 4, False)
    assert tuple(out.shape) == (K // 16, 2 * N)                   # gptq.rs:291-297
    assert (out.cpu().numpy().view(np.uint32).reshape(-1) == tiled).all()
    assert (cv.gptq_tile_unpack(out, K, N).cpu().numpy().view(np.uint32) == gq).all()      # and back: a permutation of words
    out2 = cv.marlin_weight_repack(dev_u32(G.awq_pack(q)), 4, True)
    assert tuple(out2.shape) == (K // 16, 2 * N)                  # gptq.rs:285-290
    assert (out2.cpu().numpy().view(np.uint32).reshape(-1) == tiled).all()
    # a shape the marlin arm does not take (k % 256 != 0) keeps the checkpoint layout
    q3 = rng.integers(0, 16, (128, 32))
    out3 = cv.marlin_weight_repack(dev_u32(G.gptq_pack(q3)), 4, False)
    assert (out3.cpu().numpy().view(np.uint32).reshape(16, 32) == G.gptq_pack(q3)).all()
    # columns [0, n) into tiles tile0 .. of a wider image (how the host layer packs gate_proj | up_proj)
    from candle_vllm_amd import lib
    wide = torch.zeros((K // 8) * 2 * N, dtype=torch.int32, device="cuda")
    q4 = rng.integers(0, 16, (K, N))
    parts = [dev_u32(gq), dev_u32(G.gptq_pack(q4))]
    for part, t0 in zip(parts, (0, N // 16)):
        assert lib.mi355_gptq_tile_repack(part.data_ptr(), wide.data_ptr(), K, N, t0, 0) == 0
    torch.cuda.synchronize()
    both = np.concatenate([gq, G.gptq_pack(q4)], axis=1)
    assert (wide.cpu().numpy().view(np.uint32) == G.gptq_tile(both)).all()


# ------------------------------------------------------------------------------------------------ K12 / K13 marlin
def _gptq_case(rng, K, N, gs, dt):
    q = rng.integers(0, 16, (K, N))
    ng = 1 if gs == -1 else K // gs
    s = G.round_dt(rng.uniform(0.005, 0.02, (ng, N)), dt)
    return q, s


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,gs", [(1, 128, 512, 128), (3, 64, 256, 64), (16, 256, 1024, 128), (20, 64, 512, -1),
                                      (33, 128, 512, 32), (64, 64, 768, 256), (7, 192, 512, 64)])
def test_marlin_4bit_matches_oracle(cv, dt, T, N, K, gs):
    rng = np.random.default_rng(K + N + T)
    q, s = _gptq_case(rng, K, N, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    qw = cv.marlin_weight_repack(dev_u32(G.gptq_pack(q)), 4, False)
    sp = G.marlin_permute_scales(s, K, N, gs)                    # what the reference's loader hands over
    ws = torch.zeros(N, dtype=torch.int32, device="cuda")
    y = cv.gptq_matmul(dev16(x, dt).reshape(1, T, K), qw, dev16(sp, dt), None, None, ws, 4, gs, False)
    assert tuple(y.shape) == (1, T, N)
    ref = G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), None, dt)
    check_ulp(host16(y, dt).reshape(T, N), ref, dt, what="marlin_4bit")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,gs", [(1, 128, 512, 128), (9, 64, 256, 64), (32, 192, 512, 128)])
def test_marlin_awq_matches_oracle(cv, dt, T, N, K, gs):
    rng = np.random.default_rng(K + N + T + 1)
    q, s = _gptq_case(rng, K, N, gs, dt)
    z = rng.integers(0, 16, (K // gs, N))
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    qw = cv.marlin_weight_repack(dev_u32(G.awq_pack(q)), 4, True)
    awq_qzeros = G.awq_pack(z)                                   # AWQ checkpoint packing
    mzp = G.awq_to_marlin_zero_points(awq_qzeros, K // gs, N)    # examples/convert_awq_marlin.py
    sp = G.marlin_permute_scales(s, K, N, gs)
    ws = torch.zeros(N, dtype=torch.int32, device="cuda")
    y = cv.gptq_matmul(dev16(x, dt).reshape(1, T, K), qw, dev16(sp, dt), dev_u32(mzp), None, ws, 4, gs, True)
    ref = G.gptq_linear(x, G.gptq_dequant(q, s, z, gs), None, dt)
    check_ulp(host16(y, dt).reshape(T, N), ref, dt, what="marlin_awq_4bit")


# ------------------------------------------------------------------------------------------------ K14 exllama
@pytest.mark.parametrize("T,N,K,gs", [(1, 64, 256, 64), (5, 128, 512, 128), (24, 64, 256, 32), (40, 32, 128, 32)])
def test_exllama_act_order_matches_oracle(cv, T, N, K, gs):
    rng = np.random.default_rng(K + T)
    q, s = _gptq_case(rng, K, N, gs, "f16")
    z = rng.integers(1, 17, (K // gs, N))
    g_idx = (rng.permutation(K) // gs).astype(np.int32)          # desc_act
    x = G.round_dt(rng.normal(0, 1, (T, K)), "f16")
    y = cv.gptq_matmul(dev16(x, "f16").reshape(1, T, K), dev_u32(G.gptq_pack(q)), dev16(s, "f16"),
                       dev_u32(G.gptq_pack_zeros(z)), torch.from_numpy(g_idx).cuda(), None, 4, gs, False)
    w16 = G.gptq_dequant(q, s, z, g_idx=g_idx, round_to="f16")   # half-precision dequant, as the exllama family does
    ref = G.gptq_linear(x, w16, None, "f16")
    check_ulp(host16(y, "f16").reshape(T, N), ref, "f16", what="gemm_half_q_half_alt")
    # and within north_star's 1e-3 of the exact (unrounded-weight) definition
    exact = x.astype(np.float64) @ G.gptq_dequant(q, s, z, g_idx=g_idx)
    assert np.abs(host16(y, "f16").reshape(T, N) - exact).max() <= 2e-3 * np.abs(exact).max()


@pytest.mark.parametrize("T,N,K,gs", [(1, 64, 256, 64), (7, 128, 512, 128), (33, 32, 128, 32)])
def test_exllama_8bit_matches_oracle(cv, T, N, K, gs):
    """bits = 8 on the exllama arm (the reference admits 4 | 8, linear.rs:215-217, and forwards `bits`, gptq.rs:181-194)"""
    rng = np.random.default_rng(K + T + 8)
    q = rng.integers(0, 256, (K, N))
    s = G.round_dt(rng.uniform(0.0005, 0.002, (K // gs, N)), "f16")
    z = rng.integers(1, 257, (K // gs, N))
    g_idx = (rng.permutation(K) // gs).astype(np.int32)
    x = G.round_dt(rng.normal(0, 1, (T, K)), "f16")
    y = cv.gptq_matmul(dev16(x, "f16").reshape(1, T, K), dev_u32(G.gptq_pack8(q)), dev16(s, "f16"),
                       dev_u32(G.gptq_pack_zeros8(z)), torch.from_numpy(g_idx).cuda(), None, 8, gs, False)
    assert tuple(y.shape) == (1, T, N)
    w16 = G.gptq_dequant(q, s, z, g_idx=g_idx, round_to="f16")
    ref = G.gptq_linear(x, w16, None, "f16")
    check_ulp(host16(y, "f16").reshape(T, N), ref, "f16", what="gemm_half_q_half_alt 8-bit")


def test_void_ffi_refuses_loudly(cv):
    """a configuration the library cannot serve must not read as data: NaN-filled output + a recorded error
    (`bits != 4` used to return with `c` untouched)"""
    from candle_vllm_amd import lib
    rng = np.random.default_rng(5)
    T, N, K, gs = 3, 64, 256, 64
    q, s = _gptq_case(rng, K, N, gs, "f16")
    z = rng.integers(1, 17, (K // gs, N))
    x = dev16(G.round_dt(rng.normal(0, 1, (T, K)), "f16"), "f16")
    out = torch.zeros((T, N), dtype=torch.float16, device="cuda")
    lib.mi355_clear_error()
    lib.gemm_half_q_half_alt(x.data_ptr(), dev_u32(G.gptq_pack(q)).data_ptr(), dev_u32(G.gptq_pack_zeros(z)).data_ptr(),
                             dev16(s, "f16").data_ptr(), None, out.data_ptr(), T, N, K, 3, 0)      # 3-bit: not served
    torch.cuda.synchronize()
    assert lib.mi355_last_error() != 0
    assert torch.isnan(out).all()
    lib.mi355_clear_error()
    assert lib.mi355_last_error() == 0
    with pytest.raises(RuntimeError):                             # the Python mirror turns the record into an exception
        cv.gptq_matmul(x.reshape(1, T, K), dev_u32(G.gptq_pack(q)), dev16(s, "f16"), dev_u32(G.gptq_pack_zeros(z)),
                       torch.zeros(K, dtype=torch.int32, device="cuda"), None, 3, gs, False)
    assert lib.mi355_last_error() == 0


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,gs", [(1, 128, 512, 128), (16, 256, 1024, 128), (5, 64, 256, -1)])
def test_marlin_format_checkpoint(cv, dt, T, N, K, gs):
    """`checkpoint_format == "marlin"`: B [k/16, 2n] straight from the file (Marlin tile order) + permuted `s`; the load-time
    un-permute makes it the weight image marlin_4bit_* streams, bit for bit the image gptq_repack makes of the same codes."""
    rng = np.random.default_rng(K + N + T + 77)
    q, s = _gptq_case(rng, K, N, gs, dt)
    B = G.marlin_format_pack(q)
    assert B.shape == (K // 16, 2 * N)                            # linear.rs:226-231 (marlin_format dims)
    qw = cv.marlin_format_repack(dev_u32(B))
    if K % 256 == 0:
        assert (qw.cpu().numpy().view(np.uint32).reshape(-1) == G.gptq_tile(G.gptq_pack(q))).all()
    else:
        assert (qw.cpu().numpy().view(np.uint32).reshape(K // 8, N) == G.gptq_pack(q)).all()
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    sp = G.marlin_permute_scales(s, K, N, gs)
    ws = torch.zeros(N, dtype=torch.int32, device="cuda")
    y = cv.gptq_matmul(dev16(x, dt).reshape(1, T, K), qw, dev16(sp, dt), None, None, ws, 4, gs, False)
    ref = G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), None, dt)
    check_ulp(host16(y, dt).reshape(T, N), ref, dt, what="marlin-format checkpoint")


# ------------------------------------------------------------------------------------------------ fused GPTQ epilogues
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T", [6, 1, 4])
def test_gptq_linear_fused_epilogues(cv, dt, T):
    """T = 6: the 16-token-tile kernel; T = 1, 4: the 1..4-token kernel (activations staged in LDS, weight ring)"""
    rng = np.random.default_rng(11)
    K, I, gs = 512, 128, 128
    q, s = _gptq_case(rng, K, 2 * I, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs)
    y = host16(lin.forward(dev16(x, dt), epilogue=cv.EPI_SILU_MUL), dt)
    gu = G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), None, dt)
    check_ulp(y, G.silu_mul16(gu[:, :I], gu[:, I:], dt), dt, ulps=3.0, what="gptq silu*up")
    z = rng.integers(1, 17, (K // gs, 2 * I))
    lin2 = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs, qzeros=dev_u32(G.gptq_pack_zeros(z)),
                         zero_mode=cv.ZERO_GPTQ_PLUS1)
    res = G.round_dt(rng.normal(0, 1, (T, 2 * I)), dt)
    y2 = host16(lin2.forward(dev16(x, dt), epilogue=cv.EPI_RESID, residual=dev16(res, dt)), dt)
    ref2 = G.round_dt(G.gptq_linear(x, G.gptq_dequant(q, s, z, gs), None, dt) + res, dt)
    check_ulp(y2, ref2, dt, what="gptq asym + resid", ulps=2.01, mag=G.gptq_linear(x, G.gptq_dequant(q, s, z, gs), None, dt))


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("T,N,K,gs", [(1, 256, 3584, 128), (2, 64, 3584, 64), (3, 64, 1792, 32), (1, 48, 18944, 128), (4, 32, 4864, 256)])
def test_small_batch_4bit_kernel_shapes(cv, T, N, K, gs, tiled):
    """the 1..4-token kernel at k-block counts that do not divide by 8 (Qwen2: 14 and 74), every group size, both weight
    layouts, against the oracle -- and against the 16-token-tile kernel (tuning key 31) to the same bound"""
    from candle_vllm_amd import lib
    rng = np.random.default_rng(K + N + T)
    q, s = _gptq_case(rng, K, N, gs, "bf16")
    x = G.round_dt(rng.normal(0, 1, (T, K)), "bf16")
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, "bf16"), gs, tiled=tiled)
    ref = G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), None, "bf16")
    y = host16(lin.forward(dev16(x, "bf16")), "bf16")
    check_ulp(y, ref, "bf16", what="1..4-token kernel")
    from candle_vllm_amd import tuning
    with tuning(30, 1):                                           # key 30 bit 0: the 1..4-token kernel off
        y0 = host16(lin.forward(dev16(x, "bf16")), "bf16")
    check_ulp(y0, ref, "bf16", what="16-token-tile kernel")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,pair", [(16, 12304, 512, False), (9, 12288, 256, False), (13, 12320, 768, False), (6, 12288, 512, False),
                                        (16, 12304, 512, True), (5, 12288, 256, True), (11, 12320, 768, True)])
def test_wide_16bit_kernel_many_row_tiles(cv, dt, T, N, K, pair):
    """5..16 tokens against >= 768 row tiles (gate/up, lm_head shapes): the LDS-shared-activation kernel (one row tile or gate/up
    pair per wave, 2-slot weight ring; a tile count that is not a multiple of 4 leaves surplus waves), against the oracle -- and
    the K-split kernel on the same inputs (tuning key 37) to the same bound"""
    from candle_vllm_amd import lib
    rng = np.random.default_rng(T * 31 + N + K)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    if pair:
        w = G.round_dt(rng.normal(0, 0.06, (2 * N, K)), dt)
        gu = G.linear16(x, w, None, dt)
        ref, mag, ulps = G.silu_mul16(gu[:, :N], gu[:, N:], dt), None, 3.0
    else:
        w = G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
        ref, mag, ulps = G.linear16(x, w, None, dt), None, 1.01
    lin = cv.Linear(dev16(w, dt))
    kw = {"epilogue": cv.EPI_SILU_MUL} if pair else {}
    lib.mi355_internal_last_gemm()
    y = host16(lin.forward(dev16(x, dt), **kw), dt)
    check_ulp(y, ref, dt, ulps=ulps, what="wide 16-bit kernel", mag=mag)
    assert lib.mi355_internal_last_gemm() == -1                   # not the prompt GEMM
    from candle_vllm_amd import tuning
    with tuning(30, 8):                                           # key 30 bit 3: the LDS-shared-activation kernel off
        y0 = host16(lin.forward(dev16(x, dt), **kw), dt)
    check_ulp(y0, ref, dt, ulps=ulps, what="K-split kernel", mag=mag)


def test_dense_tile_repack_bit_exact(cv):
    from candle_vllm_amd import lib
    rng = np.random.default_rng(8)
    N, K = 64, 768
    w = rng.integers(0, 2 ** 16, (N, K), dtype=np.uint16)
    d_in = torch.from_numpy(w.view(np.int16)).cuda()
    d_out = torch.zeros_like(d_in)
    assert lib.mi355_dense_tile_repack(d_in.data_ptr(), d_out.data_ptr(), N, K, K, 0) == 0
    torch.cuda.synchronize()
    assert (d_out.cpu().numpy().view(np.uint16).reshape(-1) == G.dense_tile(w)).all()
    assert lib.mi355_dense_tile_repack(d_in.data_ptr(), d_out.data_ptr(), 40, K, K, 0) != 0      # n % 16
    assert lib.mi355_dense_tile_repack(d_in.data_ptr(), d_out.data_ptr(), N, 128, 128, 0) != 0    # k % 256


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,pair", [(1, 64, 512, False), (8, 128, 256, False), (33, 96, 768, False), (64, 32, 512, False),
                                        (32, 12304, 512, False), (20, 12320, 256, True), (3, 96, 512, True),
                                        (130, 208, 512, False), (257, 336, 1024, True), (97, 144, 256, False)])
def test_linear_over_the_tiled_weight_image(cv, dt, T, N, K, pair):
    """mi355_linear_tiled through the 16-bit kernels (K-split streaming kernel; MFMA GEMM from 33 tokens, at >= 768 row tiles from 17) == the oracle ==
    the row-major result to the same bound"""
    rng = np.random.default_rng(T * 7 + N + K)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    if pair:
        w = G.round_dt(rng.normal(0, 0.06, (2 * N, K)), dt)
        gu = G.linear16(x, w, None, dt)
        ref, ulps, kw = G.silu_mul16(gu[:, :N], gu[:, N:], dt), 3.0, {"epilogue": cv.EPI_SILU_MUL}
    else:
        w = G.round_dt(rng.normal(0, 0.05, (N, K)), dt)
        ref, ulps, kw = G.linear16(x, w, None, dt), 1.01, {}
    for tiled in (True, False):
        lin = cv.Linear(dev16(w, dt), tiled=tiled)
        y = host16(lin.forward(dev16(x, dt), **kw), dt)
        check_ulp(y, ref, dt, ulps=ulps, what=f"linear tiled={tiled}")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,gs,mode", [(96, 64, 256, 64, "sym"), (130, 208, 512, 128, "sym"), (257, 96, 1024, 256, "sym"),
                                           (200, 48, 512, -1, "sym"), (128, 80, 768, 128, "zp"), (161, 144, 512, 128, "silu"),
                                           (97, 32, 256, 128, "resid")])
def test_gptq_prompt_gemm_one_pass(cv, dt, T, N, K, gs, mode):
    """>= 96 tokens over the tiled 4-bit image: the one-pass MFMA GEMM (weights unpacked from LDS, per-group scale / offset with
    the prep launch's group sums of x; ragged token and column tiles, groups of 64 / 128 / 256 / whole K, zero points, the fused
    epilogues) == the oracle == the decode kernel in 64-token chunks (tuning key 39) to the same bound"""
    from candle_vllm_amd import tuning
    rng = np.random.default_rng(T + N + K)
    pair = mode == "silu"
    Nw = 2 * N if pair else N
    q, s = _gptq_case(rng, K, Nw, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    z = rng.integers(1, 17, ((1 if gs == -1 else K // gs), Nw)) if mode == "zp" else None
    kw = {}
    if z is not None:
        kw = {"qzeros": dev_u32(G.gptq_pack_zeros(z)), "zero_mode": cv.ZERO_GPTQ_PLUS1}
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs if gs > 0 else K, **kw)
    assert lin.tiled
    lin_ref = G.gptq_linear(x, G.gptq_dequant(q, s, z, gs), None, dt)
    fkw, ulps, mag = {}, 1.01, None
    if pair:
        ref, fkw, ulps = G.silu_mul16(lin_ref[:, :N], lin_ref[:, N:], dt), {"epilogue": cv.EPI_SILU_MUL}, 3.0
    elif mode == "resid":
        res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
        ref, fkw, ulps, mag = G.round_dt(lin_ref + res, dt), {"epilogue": cv.EPI_RESID, "residual": dev16(res, dt)}, 2.01, lin_ref
    else:
        ref = lin_ref
    y = host16(lin.forward(dev16(x, dt), **fkw), dt)
    check_ulp(y, ref, dt, ulps=ulps, what="gptq prompt GEMM", mag=mag)
    with tuning(30, 16):                                          # key 30 bit 4: the one-pass 4-bit prompt GEMM off
        y0 = host16(lin.forward(dev16(x, dt), **fkw), dt)
    check_ulp(y0, ref, dt, ulps=ulps, what="decode kernel in chunks", mag=mag)


@pytest.mark.parametrize("T,N,K,gs,mode,launch", [(33, 272, 4352, 128, "resid", 207), (65, 48, 2048, 64, "zp", 204),   # 64-token tiles, K in 7 and 4 ranges
                                                  (65, 160, 768, 256, "silu", 201), (300, 4176, 256, 128, "zp", 201),   # ... in one; pairs; one token into the next
                                                  (900, 8192, 256, 128, "store", 1), (1100, 8224, 512, 512, "silu", 101)])   # 128 x 256: exactly one per CU; 128 x 128, ragged
def test_gptq_prompt_gemm_every_tile(cv, T, N, K, gs, mode, launch):
    """the one-pass 4-bit prompt GEMM where its dispatch takes each of its tiles and K ranges, tokens at the tiles' edges, at the oracle's bound"""
    dt = "bf16"
    rng = np.random.default_rng(T + N + K)
    q, s = _gptq_case(rng, K, N, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    z = rng.integers(1, 17, (K // gs, N)) if mode == "zp" else None
    kw = {"qzeros": dev_u32(G.gptq_pack_zeros(z)), "zero_mode": cv.ZERO_GPTQ_PLUS1} if z is not None else {}
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs, **kw)
    rows = np.unique([t for e in range(0, T, 64) for t in (e, e + 1, e + 63, T - 1) if t < T])
    res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
    y = G.gptq_linear(x[rows], G.gptq_dequant(q, s, z, gs), None, dt)
    if mode == "silu":
        got, ref, ulps, mag = lin.forward(dev16(x, dt), epilogue=cv.EPI_SILU_MUL), G.silu_mul16(y[:, :N // 2], y[:, N // 2:], dt), 3.0, None
    elif mode == "resid":
        got, ref, ulps, mag = lin.forward(dev16(x, dt), epilogue=cv.EPI_RESID, residual=dev16(res, dt)), G.round_dt(y + res[rows], dt), 2.01, y
    else:
        got, ref, ulps, mag = lin.forward(dev16(x, dt)), y, 1.01, None
    from candle_vllm_amd import lib
    assert lib.mi355_internal_last_gemm() == launch               # 100 tile + K ranges
    got = host16(got, dt)
    assert np.isfinite(got).all()
    check_ulp(got[rows], ref, dt, ulps=ulps, what="gptq prompt GEMM", mag=mag)


@pytest.mark.parametrize("T,N,K,gemm", [(33, 4096, 1024, False), (48, 2048, 2048, False), (64, 4096, 2048, False), (64, 1024, 1024, False), (33, 8192, 1024, False),
                                        (17, 12288, 512, False), (32, 12304, 1536, False), (33, 1024, 8192, False), (48, 528, 8448, False),  # K in ranges
                                        (48, 48, 8448, True),
                                        (49, 8192, 2048, True), (64, 4096, 3072, True), (41, 4112, 512, True), (33, 512, 256, True), (32, 12288, 2048, True)])
def test_linear_17_to_64_tokens_take_the_faster_kernel(cv, T, N, K, gemm):
    """16-bit products of 17 to 64 tokens: the streaming kernels to the sizes where the prompt GEMM becomes the faster one, both at the op's bound"""
    from candle_vllm_amd import lib
    dt = "bf16"
    rng = np.random.default_rng(T + N + K)
    x, w, b = G.round_dt(rng.normal(0, 1, (T, K)), dt), G.round_dt(rng.normal(0, 0.05, (N, K)), dt), G.round_dt(rng.normal(0, 0.2, N), dt)
    lin = cv.Linear(dev16(w, dt), dev16(b, dt), tiled=True)
    lib.mi355_internal_last_gemm()
    y = host16(lin.forward(dev16(x, dt)), dt)
    assert (lib.mi355_internal_last_gemm() >= 0) == gemm
    check_ulp(y, G.linear16(x, w, b, dt), dt, what="linear+bias", ulps=2.01, mag=G.linear16(x, w, None, dt))


@pytest.mark.parametrize("T,N,K,gs,zp,gemm", [(33, 512, 256, 128, False, False), (64, 1024, 1024, 128, False, False), (48, 4096, 2048, 128, False, False),
                                              (33, 2048, 2048, 64, True, False), (64, 4096, 1536, 128, True, False), (40, 12304, 512, 128, False, False),
                                              (48, 512, 8192, 128, False, False), (33, 2560, 8192, 256, False, False),      # K in ranges, one and two workgroups per CU
                                              (33, 2048, 4096, 128, False, True), (64, 2048, 3072, 128, False, True), (48, 4608, 2048, 128, False, True),
                                              (33, 512, 8192, 64, False, True)])
def test_gptq_33_to_64_tokens_take_the_faster_kernel(cv, T, N, K, gs, zp, gemm):
    """4-bit products of 33 to 64 tokens: the streaming kernels where they are faster than the prompt GEMM with its launch in front, both at the op's bound"""
    from candle_vllm_amd import lib
    dt = "bf16"
    rng = np.random.default_rng(T + N + K)
    q, s = _gptq_case(rng, K, N, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    z = rng.integers(1, 17, (K // gs, N)) if zp else None
    kw = {"qzeros": dev_u32(G.gptq_pack_zeros(z)), "zero_mode": cv.ZERO_GPTQ_PLUS1} if zp else {}
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs, **kw)
    lib.mi355_internal_last_gemm()
    y = host16(lin.forward(dev16(x, dt)), dt)
    assert (lib.mi355_internal_last_gemm() >= 0) == gemm
    check_ulp(y, G.gptq_linear(x, G.gptq_dequant(q, s, z, gs), None, dt), dt, ulps=1.01, what="gptq linear")


@pytest.mark.parametrize("T,ns,K,bits,gemm", [(64, (2048, 512, 512), 512, 16, False), (47, (2048, 2048, 2048), 1024, 16, False), (48, (2048, 2048, 2048), 1024, 16, True),
                                              (33, (2048, 2048, 2048), 512, 16, True), (64, (2048, 2048, 2048), 512, 4, False), (49, (4096, 4096, 4096), 512, 4, True),
                                              (48, (4096, 4096, 4096), 512, 4, False), (49, (2048, 2048, 2048), 1280, 4, True)])
def test_three_products_take_the_faster_kernel(cv, T, ns, K, bits, gemm):
    """q, k and v in one launch, 16-bit and 4-bit: streaming kernel or prompt GEMM by rows, k and tokens; within the op's bound of the products in 64 bits"""
    import ctypes
    from candle_vllm_amd import lib
    gen, st = torch.Generator(device="cuda").manual_seed(T + K), torch.cuda.current_stream().cuda_stream
    x, out, ws, ss, refs = torch.randn(T, K, generator=gen, device="cuda").to(torch.bfloat16), [], [], [], []
    for n in ns:
        out.append(torch.full((T, n), float("nan"), device="cuda", dtype=torch.bfloat16))
        if bits == 16:
            w = (torch.randn(n, K, generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
            img = torch.empty_like(w)
            assert lib.mi355_dense_tile_repack(w.data_ptr(), img.data_ptr(), n, K, K, st) == 0
            wd = w.double().T
        else:
            q = torch.randint(0, 16, (K, n), generator=gen, device="cuda", dtype=torch.int32)
            packed = sum((q.view(K // 8, 8, n)[:, i] << (4 * i)) for i in range(8)).contiguous()
            img = torch.empty_like(packed)
            assert lib.mi355_gptq_tile_repack(packed.data_ptr(), img.data_ptr(), K, n, 0, st) == 0
            ss.append((torch.rand(K // 128, n, generator=gen, device="cuda") * 0.01 + 0.002).to(torch.bfloat16))
            wd = ((q.double() - 8).view(K // 128, 128, n) * ss[-1].double()[:, None]).view(K, n)
        ws.append(img)
        refs.append(x.double() @ wd)
    p3 = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts])
    fn = lib.mi355_internal_linear3
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int32] * 5 + [ctypes.c_void_p, ctypes.c_float, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64]
    lib.mi355_internal_last_gemm()
    assert fn(p3(out), x.data_ptr(), p3(ws), p3(ss) if ss else None, None, (ctypes.c_int32 * 3)(*ns), T, K, 128, 3 if bits == 16 else 2, 2, None, 0.0, None, None, st) == 0
    assert (lib.mi355_internal_last_gemm() >= 0) == gemm
    for o, r in zip(out, refs):
        check_ulp(o.double().cpu().numpy(), r.to(torch.bfloat16).double().cpu().numpy(), "bf16", ulps=1.01, what="one of three", mag=r.abs().cpu().numpy())


def test_gptq_prompt_gemm_in_slabs(cv):
    """more tokens than the permuted copy of x has room for (128 MiB: 3 328 of 18 944): slabs of tokens, rows at their borders against the product in 64
    bits, residual in place; and the memory taken"""
    T, N, K, gs = 8000, 48, 18944, 128
    gen = torch.Generator(device="cuda").manual_seed(2)
    q = torch.randint(0, 16, (K, N), generator=gen, device="cuda", dtype=torch.int32)
    packed = sum((q.view(K // 8, 8, N)[:, i] << (4 * i)) for i in range(8)).contiguous()
    s = (torch.rand(K // gs, N, generator=gen, device="cuda") * 0.004 + 0.002).to(torch.bfloat16)
    x, out = (torch.randn(*sh, generator=gen, device="cuda").to(torch.bfloat16) for sh in ((T, K), (T, N)))
    rows = torch.tensor(sorted({0, 1, 255, 256, 3327, 3328, 3329, 6655, 6656, T - 1}), device="cuda")
    y = x[rows].double() @ ((q.double() - 8).view(K // gs, gs, N) * s.double()[:, None]).view(K, N)
    mag, want = y.abs(), y.to(torch.bfloat16).double() + out[rows].double()
    lin = cv.GPTQLinear(packed, s, gs)

    def taken():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free - torch.cuda.memory_reserved()
    before = taken()
    got = lin.forward(x, epilogue=cv.EPI_RESID, residual=out)
    assert taken() - before <= (256 + 8) << 20                    # with room for partial sums
    check_ulp(got[rows].double().cpu().numpy(), want.cpu().numpy(), "bf16", ulps=2.01, what="slabs", mag=mag.cpu().numpy())


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,gs,mode", [(32, 1184, 3584, 128, "store"), (32, 3584, 3584, 128, "resid"), (9, 224, 2048, 64, "store"),
                                           (48, 512, 4864, 256, "bias"), (17, 2 * 4736, 1792, 128, "silu"), (32, 2 * 608, 3584, 128, "silu"),
                                           (5, 64, 18944, 128, "resid"), (33, 4096, 256, 128, "store")])
def test_gptq_wide_kernel_5_to_48_tokens(cv, dt, T, N, K, gs, mode):
    """csrc/gptq_wide.inc: 5..48 tokens over the tiled 4-bit image with the activations shared through LDS -- many-tile launches
    in one sweep (gate/up as pairs per wave, SiLU * up from the accumulators), few-tile launches split over K with the partial sums added
    by the epilogue launch (Qwen2-7B's wo / down shapes: 14 and 74 k-blocks), a single k-block, ragged last workgroups.  Against the oracle
    at the bound of the 16-token-tile kernel it replaces, and against that kernel itself (tuning key 30 bit 128)."""
    from candle_vllm_amd import tuning
    rng = np.random.default_rng(K + N + T)
    q, s = _gptq_case(rng, K, N, gs, dt)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    bias = G.round_dt(rng.normal(0, 1, N), dt) if mode == "bias" else None
    lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, dt), gs, bias=None if bias is None else dev16(bias, dt))
    assert lin.tiled
    full = G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), bias, dt)
    kw, ulps = {}, 1.0
    if mode == "silu":
        ref = G.silu_mul16(full[:, :N // 2], full[:, N // 2:], dt)
        kw, ulps = dict(epilogue=cv.EPI_SILU_MUL), 3.0
    elif mode == "resid":
        res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
        ref = G.round_dt(full + res, dt)
        kw, ulps = dict(epilogue=cv.EPI_RESID, residual=dev16(res, dt)), 2.01
    else:
        ref = full
        if mode == "bias":
            ulps = 2.01
    magkw = {"mag": full} if mode == "resid" else ({"mag": G.gptq_linear(x, G.gptq_dequant(q, s, None, gs), None, dt)} if mode == "bias" else {})
    from candle_vllm_amd import lib
    lib.mi355_internal_last_gemm()
    with tuning(30, 16):                                           # key 30 bit 16: the prompt GEMM off, which takes 33 tokens and more
        y = host16(lin.forward(dev16(x, dt), **kw), dt)
    check_ulp(y, ref, dt, ulps=ulps, what="gptq wide kernel", **magkw)
    with tuning(30, 16 | 128):                                     # bit 128: the wide kernel off
        y0 = host16(lin.forward(dev16(x, dt), **kw), dt)
    assert lib.mi355_internal_last_gemm() == -1
    check_ulp(y0, ref, dt, ulps=ulps, what="16-token-tile kernel", **magkw)
    assert np.abs(y - y0).max() <= 3 * (2.0 ** -8 if dt == "bf16" else 2.0 ** -11) * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("T,N,K,tiled", [(32, 256, 8192, True), (20, 336, 14336, True), (31, 64, 8448, False), (9, 4096, 8192, True)])
def test_wide_16bit_kernel_few_tiles_long_k_split(cv, dt, T, N, K, tiled):
    """5..32 tokens: few-tile 16-bit launches with a long K (down_proj of a batch-32 step: 256 tiles x 56 k-blocks at Llama-3-8B) take the
    LDS-shared-activation sweep split over K across workgroups; the partial sums meet in the epilogue launch (split order), which applies
    bias / residual and the rounding chain.  Against the oracle at the bound of the kernel it replaces, bias + residual included."""
    rng = np.random.default_rng(T + N + K)
    x = G.round_dt(rng.normal(0, 1, (T, K)), dt)
    w = G.round_dt(rng.normal(0, 0.02, (N, K)), dt)
    b = G.round_dt(rng.normal(0, 0.2, N), dt)
    res = G.round_dt(rng.normal(0, 1, (T, N)), dt)
    lin = cv.Linear(dev16(w, dt), dev16(b, dt), tiled=tiled)
    y = host16(lin.forward(dev16(x, dt), epilogue=cv.EPI_RESID, residual=dev16(res, dt)), dt)
    full = G.linear16(x, w, b, dt)
    check_ulp(y, G.round_dt(full + res, dt), dt, what="split-K wide kernel + bias + residual", ulps=3.01, mag=np.maximum(np.abs(full), np.abs(G.linear16(x, w, None, dt))))
    from candle_vllm_amd import lib
    lib.mi355_internal_last_gemm()
    y2 = host16(cv.Linear(dev16(w, dt), tiled=tiled).forward(dev16(x, dt)), dt)
    check_ulp(y2, G.linear16(x, w, None, dt), dt, what="split-K wide kernel")
    assert lib.mi355_internal_last_gemm() == -1                   # not the prompt GEMM


@pytest.mark.parametrize("kind,T,N,K", [("16-bit", 96, 96, 8192), ("16-bit", 9, 256, 8192), ("4-bit", 100, 64, 8192), ("4-bit", 33, 64, 8192)])
def test_no_room_for_a_workspace(cv, kind, T, N, K):
    """launches that split K or prepare their operands, where the workspace cannot be allocated (a new stream, on which every allocation fails as on a full
    card): another way to the same result at the same bound, and no error behind it"""
    import ctypes
    from candle_vllm_amd._lib import lib
    lib.mi355_internal_scratch_limit.argtypes = [ctypes.c_int64]
    rng = np.random.default_rng(T + N + K)
    x = G.round_dt(rng.normal(0, 1, (T, K)), "bf16")
    if kind == "4-bit":
        q, s = _gptq_case(rng, K, N, 128, "bf16")
        lin, ref = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, "bf16"), 128), G.gptq_linear(x, G.gptq_dequant(q, s, None, 128), None, "bf16")
    else:
        w = G.round_dt(rng.normal(0, 0.02, (N, K)), "bf16")
        lin, ref = cv.Linear(dev16(w, "bf16"), tiled=True), G.linear16(x, w, None, "bf16")
    xd = dev16(x, "bf16")
    torch.cuda.synchronize()
    for limit in (0, -1):
        with torch.cuda.stream(torch.cuda.Stream()):
            lib.mi355_internal_scratch_limit(limit)
            try:
                y = lin.forward(xd)
            finally:
                lib.mi355_internal_scratch_limit(-1)
            torch.cuda.current_stream().synchronize()
            check_ulp(host16(y, "bf16"), ref, "bf16", what=f"{kind}, limit {limit}")


@pytest.mark.parametrize("kind,T,N,K", [("4-bit", 130, 64, 4096), ("16-bit", 96, 96, 4096), ("16-bit", 9, 256, 8192)])
def test_two_threads_on_one_stream(cv, kind, T, N, K):
    """launches that hand a workspace on to each other, from two threads on one stream, each over its own x: every result is the one it has alone, bit for bit"""
    import threading
    rng = np.random.default_rng(T + N)
    if kind == "4-bit":
        q, s = _gptq_case(rng, K, N, 128, "bf16")
        lin = cv.GPTQLinear(dev_u32(G.gptq_pack(q)), dev16(s, "bf16"), 128)
    else:
        lin = cv.Linear(dev16(G.round_dt(rng.normal(0, 0.02, (N, K)), "bf16"), "bf16"), tiled=True)
    xs = [torch.randn(T, K, device="cuda").to(torch.bfloat16) for _ in range(2)]
    alone = [lin.forward(x) for x in xs]
    torch.cuda.synchronize()
    got = [[], []]
    go = threading.Barrier(2)

    def work(i):
        go.wait()
        got[i] = [lin.forward(xs[i]) for _ in range(300)]
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 300 and all(torch.equal(y.view(torch.int16), alone[i].view(torch.int16)) for y in got[i])


# K in ranges: prompts whose tiles leave units idle, in 16 and 4 bits, both cache layouts, biases, heads of 64, 128 and 80, tokens that the cache does not take
@pytest.mark.parametrize("T,H,G_,D,K,bits,flash,bias", [(66, 16, 4, 128, 2048, 16, False, False), (99, 16, 4, 128, 2048, 16, True, True), (359, 16, 4, 64, 4096, 16, False, False),
                                                         (50, 28, 4, 128, 3584, 4, False, True), (133, 28, 4, 128, 3584, 4, True, False), (150, 14, 2, 64, 4096, 4, False, True),
                                                         (70, 8, 2, 80, 2048, 16, False, True)])
def test_three_products_in_ranges_of_k_with_rope_and_cache(cv, T, H, G_, D, K, bits, flash, bias):
    """q, rotated, and the rotated k and v in the cache by the launch that adds the ranges: each within the bf16 steps of its rounding chain (product, bias, rotation) of
    64 bits, the cache's other slots untouched"""
    import ctypes
    from candle_vllm_amd import lib
    gen, st = torch.Generator(device="cuda").manual_seed(T + K), torch.cuda.current_stream().cuda_stream
    ns, bs = (H * D, G_ * D, G_ * D), 32
    x, out, ws, ss, refs, bb = torch.randn(T, K, generator=gen, device="cuda").to(torch.bfloat16), [], [], [], [], []
    for n in ns:
        out.append(torch.full((T, n), float("nan"), device="cuda", dtype=torch.bfloat16))
        bb.append(torch.randn(n, generator=gen, device="cuda").to(torch.bfloat16))
        if bits == 16:
            w = (torch.randn(n, K, generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
            img = torch.empty_like(w)
            assert lib.mi355_dense_tile_repack(w.data_ptr(), img.data_ptr(), n, K, K, st) == 0
            wd = w.double().T
        else:
            q = torch.randint(0, 16, (K, n), generator=gen, device="cuda", dtype=torch.int32)
            packed = sum((q.view(K // 8, 8, n)[:, i] << (4 * i)) for i in range(8)).contiguous()
            img = torch.empty_like(packed)
            assert lib.mi355_gptq_tile_repack(packed.data_ptr(), img.data_ptr(), K, n, 0, st) == 0
            ss.append((torch.rand(K // 128, n, generator=gen, device="cuda") * 0.01 + 0.002).to(torch.bfloat16))
            wd = ((q.double() - 8).view(K // 128, 128, n) * ss[-1].double()[:, None]).view(K, n)
        ws.append(img)
        refs.append(x.double() @ wd + (bb[-1].double() if bias else 0))
    nb = (T + 40) // bs + 1
    shape = (nb, bs, G_, D) if flash else (nb, G_, D // 8, bs, 8)
    kc, vc = torch.full(shape, 7.0, device="cuda", dtype=torch.bfloat16), torch.full(shape if flash else (nb, G_, D, bs), 7.0, device="cuda", dtype=torch.bfloat16)
    pos = torch.randint(0, 500, (T,), generator=gen, device="cuda")
    slot = torch.randperm(nb * bs, device="cuda")[:T]
    slot[3] = -1
    ang = torch.arange(500, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(D // 2, device="cuda").double() / (D // 2))
    cos, sin = ang.cos().float().contiguous(), ang.sin().float().contiguous()

    class Rope(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in ("cos", "sin", "pos", "slots", "kc", "vc")] + [(n, ctypes.c_int32) for n in ("kv", "d", "bs", "flash")]
    rope = Rope(cos.data_ptr(), sin.data_ptr(), pos.data_ptr(), slot.data_ptr(), kc.data_ptr(), vc.data_ptr(), G_, D, bs, int(flash))
    p3 = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts])
    fn = lib.mi355_internal_linear3_prompt
    fn.argtypes = [ctypes.c_void_p] * 6 + [ctypes.c_int32] * 5 + [ctypes.c_void_p, ctypes.c_float] + [ctypes.c_void_p] * 4 + [ctypes.c_int64]
    done = ctypes.c_int32(-1)
    lib.mi355_internal_last_gemm()
    assert fn(p3(out), x.data_ptr(), p3(ws), p3(ss) if ss else None, p3(bb) if bias else None, (ctypes.c_int32 * 3)(*ns), T, K, 128, 3 if bits == 16 else 2, 2, None, 0.0, None, None,
              ctypes.byref(rope), ctypes.byref(done), st) == 0
    assert lib.mi355_internal_last_gemm() % 100 > 1 and done.value == 1
    c, s = ang.cos()[pos][:, None], ang.sin()[pos][:, None]

    def turned(y):
        a, b = y.view(T, -1, D)[..., :D // 2], y.view(T, -1, D)[..., D // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1), torch.cat([a.abs() + b.abs()] * 2, -1)
    flat = (lambda t: t.reshape(nb * bs, G_, D)) if flash else (lambda t: (t.permute(0, 3, 1, 2, 4) if t.dim() == 5 else t.permute(0, 3, 1, 2)).reshape(nb * bs, G_, D))
    ok = slot >= 0
    for got, (want, mag) in ((out[0].view(T, H, D), turned(refs[0])), (flat(kc)[slot[ok]], [v[ok] for v in turned(refs[1])]),
                             (flat(vc)[slot[ok]], (refs[2].view(T, G_, D)[ok], refs[2].view(T, G_, D)[ok].abs()))):
        # product, bias and rotation are rounded to bf16 each: 2^-8 of the largest value in the chain at most (the sums of K products in f32 are far below)
        assert ((got.double() - want).abs() <= 3.0 * 2.0 ** -8 * (mag + (0 if not bias else 8.0)) + 1e-6).all()
    rest = torch.ones(nb * bs, dtype=torch.bool, device="cuda")
    rest[slot[ok]] = False
    assert (flat(kc)[rest] == 7).all() and (flat(vc)[rest] == 7).all()
