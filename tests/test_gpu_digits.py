"""Products of one and two tokens, whose x is staged as four base-256 digits of an integer in units of its 32 columns' largest exponent."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import kquants as kq          # noqa: E402
from oracle import ops as O               # noqa: E402
from tests.test_gpu_ops import bf16_dev, cv, dev          # noqa: E402,F401


def bound(x, blocks, t, products=1):
    """of |got - exact| per (token, row): a unit per column -- the unit is 2^-29 of the largest exponent of the 32 --, times the weight without its minimum
    and offset (at most 2 x the weight's scale times the largest code), and 2^-20 of all that is added for the f32 sums"""
    w = np.abs(kq.dequantize(blocks, t)).astype(np.float64)
    peak = w.reshape(len(w), -1, 32).max(axis=2, keepdims=True) * 2.0
    top = np.abs(x.astype(np.float64)).reshape(len(x), -1, 32).max(axis=2, keepdims=True)
    unit = np.repeat(top, 32, axis=2).reshape(x.shape) * 2.0 ** -29
    coarse = np.repeat(peak, 32, axis=2).reshape(w.shape)
    return unit @ coarse.T + 2.0 ** -20 * np.abs(x.astype(np.float64)) @ coarse.T + 1e-30


@pytest.mark.parametrize("t", [kq.GGML_Q4_K, kq.GGML_Q6_K])
@pytest.mark.parametrize("T,N,K", [(1, 16, 256), (1, 40, 512), (1, 272, 2048), (1, 33, 2304), (1, 48, 14336), (2, 16, 256), (2, 40, 4096), (2, 528, 2304)])
@pytest.mark.parametrize("spread", [0.0, 3.0])
def test_products_within_a_unit(cv, t, T, N, K, spread):
    rng = np.random.default_rng(T + N + K)
    blocks = kq.quantize(rng.normal(0, 0.05, (N, K)).astype(np.float32), t)
    x = (rng.normal(size=(T, K)) * np.exp(spread * rng.normal(size=(T, K)))).astype(np.float32)
    x[0, :32] = 0.0                                                     # 32 columns without an exponent
    x[-1, 32:64] *= np.float32(1e-38)                                   # and of the smallest ones
    got = cv.QMatMul(blocks, t, "cuda").forward(dev(x)).cpu().numpy().astype(np.float64)
    ref = x.astype(np.float64) @ kq.dequantize(blocks, t).astype(np.float64).T
    assert (np.abs(got - ref) <= bound(x, blocks, t)).all(), np.abs(got - ref).max()
    if spread == 0.0:
        e = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert e < (5e-7 if T == 1 or t == kq.GGML_Q4_K else 4e-6)      # 2^-24 for each of a few f32 roundings; two tokens of Q6_K have bf16 pieces: 2.8e-6


@pytest.mark.parametrize("t,T", [(kq.GGML_Q4_K, 1), (kq.GGML_Q4_K, 2), (kq.GGML_Q6_K, 1)])
@pytest.mark.parametrize("times", [10, 30, 100, 1000])
def test_small_columns_beside_large_ones_on_weights_of_zero(cv, t, T, times):
    """one column of 32 is `times` the others and its weights are zero: what is left has to be as exact as two bf16 pieces of each value make it, 2^-18 of it (evenly spread:
    2^-18 / sqrt(3) of the norm), whatever the largest of its 32 columns.  A thousand times, Q4_K: its high nibbles' offset adds 8 x 1000 x 2^-24 in f32 to sub-blocks of about 40"""
    rng = np.random.default_rng(times + T)
    w = np.abs(rng.normal(0, 0.05, (512, 2048))).astype(np.float32)          # (not below zero: Q4_K has no minimum then)
    w[:, ::32] = 0.0
    blocks = kq.quantize(w, t)
    w = kq.dequantize(blocks, t).astype(np.float64)
    assert (w[:, ::32] == 0.0).all()
    x = rng.normal(size=(T, 2048)).astype(np.float32)
    x[:, ::32] *= np.float32(times)
    ref = x.astype(np.float64) @ w.T
    got = cv.QMatMul(blocks, t, "cuda").forward(dev(x)).cpu().numpy().astype(np.float64)
    e = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert e < (1.2e-5 if times == 1000 and t == kq.GGML_Q4_K else 2.2e-6), e


@pytest.mark.parametrize("t", [kq.GGML_Q4_K, kq.GGML_Q6_K])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_that_are_no_numbers_reach_every_row(cv, t, bad):
    rng = np.random.default_rng(3)
    blocks = kq.quantize(rng.normal(0, 0.05, (64, 768)).astype(np.float32), t)
    mm = cv.QMatMul(blocks, t, "cuda")
    for T in (1, 2):
        x = rng.normal(size=(T, 768)).astype(np.float32)
        x[T - 1, 300] = bad
        y = mm.forward(dev(x)).cpu().numpy()
        assert (~np.isfinite(y[T - 1])).all() and np.isfinite(y[:T - 1]).all()


@pytest.mark.parametrize("types", [(12, 12), (14, 14), (12, 14), (14, 12)])
@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("bf16", [False, True])
def test_gate_and_up_of_either_type(cv, types, T, bf16):
    rng = np.random.default_rng(5 + T)
    hid, I = 1280, 208
    w = [kq.quantize(rng.normal(0, 0.05, (I, hid)).astype(np.float32), t) for t in types]
    mats = [cv.QMatMul(b, t, "cuda") for b, t in zip(w, types)]
    x = rng.normal(size=(T, hid)).astype(np.float32)
    xd = dev(x)
    if bf16:
        xb = O.f32_to_bf16_bits(x)
        x, xd = O.bf16_bits_to_f32(xb), bf16_dev(xb)
    h = torch.empty((T, I), dtype=torch.float32, device="cuda")
    cv.qmatmul_fused(mats, xd, epilogue=cv.EPI_SILU_MUL, out=h)
    g, u = (x.astype(np.float64) @ kq.dequantize(b, t).astype(np.float64).T for b, t in zip(w, types))
    ref = g / (1 + np.exp(-g)) * u
    # silu's slope is at most 1.1; f32 exp and division: 2^-20 of the value
    tol = 1.1 * bound(x, w[0], types[0]) * np.abs(u) + bound(x, w[1], types[1]) * np.abs(g) + 2.0 ** -20 * np.abs(ref)
    assert (np.abs(h.cpu().numpy() - ref) <= tol).all()


def test_segments_of_both_types_with_norm(cv):
    """a launch of mixed tiles; the norm's sum of squares comes from the values, not from their integers"""
    rng = np.random.default_rng(9)
    hid, types, rows = 2048, (12, 12, 14), (64, 16, 32)
    w = [kq.quantize(rng.normal(0, 0.05, (n, hid)).astype(np.float32), t) for n, t in zip(rows, types)]
    mats = [cv.QMatMul(b, t, "cuda") for b, t in zip(w, types)]
    x, nw = rng.normal(size=(1, hid)).astype(np.float32), (1 + rng.normal(0, 0.1, hid)).astype(np.float32)
    out = torch.empty((1, sum(rows)), dtype=torch.float32, device="cuda")
    cv.qmatmul_fused(mats, dev(x), epilogue=cv.EPI_STORE, out=out, norm_weight=dev(nw), norm_eps=1e-5)
    xn = x.astype(np.float64) * nw / np.sqrt((x.astype(np.float64) ** 2).mean() + 1e-5)
    ref = np.concatenate([xn @ kq.dequantize(b, t).astype(np.float64).T for b, t in zip(w, types)], axis=1)
    assert np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref) < 2e-6
