"""The tiled matmul kernels: every tile size and K split forced, at the edges
of tiles, K stages and groups, every width; scales too large for the
subnormal form of the dequantization."""
import numpy as np
import pytest

from cider_press_amd.kernels import qmm as kqmm
from cider_press_amd.synthetic import from_bits, make_weight, make_x, to_bits

pytestmark = pytest.mark.gpu


def _run_n(device, library, oracle, m, n, k, gs, bits, dtype, edit=None, calls=1):
    """affine_qmm_n and its float64 reference over the oracle's dequantized table."""
    rng = np.random.default_rng(m * 7 + n + k + bits)
    w_q, s, b = make_weight(rng, k, n, gs, bits, dtype)
    if edit:
        edit(s, b)
    x = make_x(rng, m, k, dtype)
    W, S, B = (device.upload(w_q.reshape(-1), "u32"), device.upload(s.reshape(-1), dtype),
               device.upload(b.reshape(-1), dtype))
    X = device.upload(x.reshape(-1), dtype)
    cmds, outs = device.commands(), []
    for _ in range(calls):
        Y = device.alloc_buffer(m * n, dtype)
        kqmm.affine_qmm_n(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)
        cmds.commit_and_wait()
        outs.append(Y.to_numpy().reshape(m, n))
    w = from_bits(oracle.dequantize(w_q, s, b, k, n, gs, bits, dtype), dtype).astype(np.float64)
    return outs, from_bits(x, dtype).astype(np.float64) @ w


def _close(y, ref, dtype):
    """Half an ulp of T for the output's rounding, and fp32 accumulation of K
    products: a few 2^-24 of the terms' magnitude, far below 2e-3 in 2-norm."""
    got = from_bits(y, dtype).astype(np.float64)
    assert np.isfinite(got).all()
    assert np.linalg.norm(got - ref) <= 2e-3 * np.linalg.norm(ref)


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("m,n,k,gs,bits,dtype,split", [
    (1, 32, 8, 32, 6, "bf16", 1),        # one row, one 8-k piece
    (257, 288, 72, 32, 4, "bf16", 1),    # one past a tile, K one piece past a stage
    (65, 128, 264, 64, 8, "f16", 2),     # two parts, the second ends in 8 k
    (33, 416, 640, 32, 3, "bf16", 3),    # stages do not divide into the parts
    (129, 384, 1032, 128, 5, "f16", 5),
    (40, 256, 136, 64, 2, "bf16", 1),
])
def test_tile_n(device, library, oracle, monkeypatch, cfg, m, n, k, gs, bits, dtype, split):
    monkeypatch.setenv("CPQ_TILE_CFG", str(cfg))
    monkeypatch.setenv("CPQ_QMM_SPLIT", str(split))
    outs, ref = _run_n(device, library, oracle, m, n, k, gs, bits, dtype, calls=2)
    _close(outs[0], ref, dtype)
    assert np.array_equal(outs[0], outs[1])  # parts are added in k order whoever finishes last


@pytest.mark.parametrize("split", [1, 2])
def test_tile_n_large_scales(device, library, oracle, monkeypatch, split):
    """A bf16 scale at 2^104 and above overflows the subnormal form: its tile
    is computed again with explicit conversions; the other tiles are not."""
    monkeypatch.setenv("CPQ_QMM_SPLIT", str(split))

    def edit(s, b):
        s[3, 1] = to_bits(np.float32([2.0 ** 104]), "bf16")[0]
        b[3, 1] = to_bits(np.float32([-2.0 ** 107]), "bf16")[0]

    outs, ref = _run_n(device, library, oracle, 70, 512, 256, 64, 4, "bf16", edit)
    _close(outs[0][:, 64:128], ref[:, 64:128], "bf16")
    rest = np.r_[0:64, 128:512]
    _close(outs[0][:, rest], ref[:, rest], "bf16")
