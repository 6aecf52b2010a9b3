"""The weights the tiled and decode kernels multiply with, bit for bit: one-hot
rows of X return them, and they have to be affine_dequantize's (the oracle's
RNE of fmaf(s, q, b)) over scales and biases of every exponent: subnormal, zero,
negative and, in bf16, past 2^104 where the subnormal form gives way."""
import numpy as np
import pytest

from cider_press_amd.kernels import qmm as kqmm
from cider_press_amd.kernels import qmv as kqmv
from cider_press_amd.synthetic import from_bits, to_bits

pytestmark = pytest.mark.gpu

WIDTHS = [2, 3, 4, 5, 6, 8]


def _patterns(rng, shape, dtype, top):
    """Random 16-bit floats with a biased exponent below `top`."""
    shift = 7 if dtype == "bf16" else 10
    return ((rng.integers(0, 2, shape) << 15) | (rng.integers(0, top, shape) << shift) |
            rng.integers(0, 1 << shift, shape)).astype(np.uint16)


def _weight(rng, rows, cols, gs, bits, dtype, large=False):
    """Any packed values; s * q + b finite in T."""
    w_q = rng.integers(0, 1 << 32, (rows, cols * bits // 32), dtype=np.uint64).astype(np.uint32)
    tops = (231, 240) if dtype == "bf16" else (22, 27)
    s, b = (_patterns(rng, (rows, cols // gs), dtype, t) for t in tops)
    s[::5, ::3] &= 0x807F if dtype == "bf16" else 0x83FF  # subnormal and zero scales
    b[::7, ::2] &= 0x807F if dtype == "bf16" else 0x83FF
    if large:
        s[rows // 3, 1] = to_bits(np.float32([2.0 ** 104]), "bf16")[0]
        s[rows // 2, 0] = to_bits(np.float32([-1.5 * 2.0 ** 110]), "bf16")[0]
    return w_q, s, b


def _one_hot(ks, k, dtype):
    x = np.zeros((len(ks), k), np.uint16)
    x[np.arange(len(ks)), ks] = to_bits(np.float32([1.0]), dtype)[0]
    return x


def _call(device, library, w_q, s, b, x, m, n, k, gs, bits, dtype, op):
    W, S, B = device.upload(w_q.reshape(-1), "u32"), device.upload(s.reshape(-1), dtype), device.upload(b.reshape(-1), dtype)
    X, Y, cmds = device.upload(x.reshape(-1), dtype), device.alloc_buffer(m * n, dtype), device.commands()
    if op == "n":
        kqmm.affine_qmm_n(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)
    elif m == 1:
        kqmv.affine_qmv(cmds, library, W, S, B, X, Y, k, gs, bits)
    else:
        kqmm.affine_qmm_t(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)
    cmds.commit_and_wait()
    return from_bits(Y.to_numpy().reshape(m, n), dtype)


def _same(y, w_bits, dtype, label):
    w = from_bits(w_bits, dtype)
    assert np.isfinite(w).all()
    bad = np.argwhere(y != w)  # -0 and +0 compare equal: the sum's zero is +0
    assert bad.size == 0, (label, len(bad), bad[:4], y[tuple(bad[0])], w[tuple(bad[0])])


@pytest.mark.parametrize("cfg", [0, 2, 4])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("op", ["t", "n"])
def test_tiles(device, library, oracle, monkeypatch, op, dtype, cfg):
    for name, value in (("CPQ_TILE_CFG", str(cfg)), ("CPQ_QMM_DMA", "0"), ("CPQ_SKINNY_MAX_M", "1"),
                        ("CPQ_SMALL_ROWS", "0"), ("CPQ_SMALL_DENSE", "0")):
        monkeypatch.setenv(name, value)
    rng = np.random.default_rng(cfg + len(dtype))
    for bits in WIDTHS:
        for gs, large in ((32, False), (64, dtype == "bf16")):
            k, n = (352 if gs == 32 else 320), 256
            rows, cols = (n, k) if op == "t" else (k, n)
            w_q, s, b = _weight(rng, rows, cols, gs, bits, dtype, large)
            y = _call(device, library, w_q, s, b, _one_hot(np.arange(k), k, dtype), k, n, k, gs, bits, dtype, op)
            w = oracle.dequantize(w_q, s, b, rows, cols, gs, bits, dtype)
            _same(y, w.T if op == "t" else w, dtype, (bits, gs, large))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", WIDTHS)
@pytest.mark.parametrize("phased", [False, True])
def test_decode(device, library, oracle, monkeypatch, phased, bits, dtype):
    if phased:
        monkeypatch.setenv("CPQ_DECODE_PHASED", "1")
    rng = np.random.default_rng(bits)
    for gs, large in ((32, False), (64, dtype == "bf16"), (128, False)):
        n, k = 96, 3456 if gs == 128 else 3520
        w_q, s, b = _weight(rng, n, k, gs, bits, dtype, large)
        w = oracle.dequantize(w_q, s, b, n, k, gs, bits, dtype)
        ks = rng.permutation(k)
        ks = np.concatenate([[0, k - 1], ks[(ks != 0) & (ks != k - 1)]])[:64].reshape(4, 16)
        for row in ks:
            y = _call(device, library, w_q, s, b, _one_hot(row, k, dtype), 16, n, k, gs, bits, dtype, "t")
            _same(y, w[:, row].T, dtype, (bits, gs, large))


@pytest.mark.parametrize("m,op", [(5, "t"), (70, "t"), (70, "n"), (1, "t")])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [3, 4, 8])
def test_infinite_and_nan_scales(device, library, oracle, monkeypatch, bits, dtype, m, op):
    """A scale of Inf or NaN makes its own columns infinite or NaN and no other."""
    monkeypatch.setenv("CPQ_QMM_DMA", "0")
    monkeypatch.setenv("CPQ_SMALL_ROWS", "0")
    rng = np.random.default_rng(bits + m)
    k, n, gs = 2112, 128, 32
    rows, cols = (n, k) if op == "t" else (k, n)
    w_q, s, b = _weight(rng, rows, cols, gs, bits, dtype)
    top = 120 if dtype == "bf16" else 10
    s = _patterns(rng, s.shape, dtype, top)
    b = _patterns(rng, b.shape, dtype, top)
    inf, nan = (0x7F80, 0x7FC0) if dtype == "bf16" else (0x7C00, 0x7E00)
    hit = np.zeros(n, bool)
    for row, group, value in ((7, 3, inf), (40, 1, nan), (90, 2, inf | 0x8000)):
        s[row, group] = value
        if op == "t":
            hit[row] = True
        else:
            hit[group * gs:(group + 1) * gs] = True
    x = to_bits(rng.standard_normal((m, k)).astype(np.float32), dtype)
    y = _call(device, library, w_q, s, b, x, m, n, k, gs, bits, dtype, op)
    ok = ~hit
    assert np.isfinite(y[:, ok]).all()
    assert not np.isfinite(y[:, hit]).any()
