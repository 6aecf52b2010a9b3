"""The tiled matmul kernels: every tile size and K split forced, at the edges
of tiles, K stages and groups, every width; scales too large for the
subnormal form of the dequantization."""
import ctypes
import time

import numpy as np
import pytest

from cider_press_amd import _lib
from cider_press_amd.kernels import _ptr
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


def _close(y, ref, dtype, k=1 << 14):
    """Rounding to T errs by at most u of a value (2^-8 with bf16's 8 significant
    bits, 2^-11 with f16's 11), and evenly up to there over many values: their
    root mean square is at most u / sqrt(3).  fp32 sums of k terms add 2^-24 of
    partial sums as large as the result, k times at random."""
    got = from_bits(y, dtype).astype(np.float64)
    assert np.isfinite(got).all()
    u = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    bound = u / (np.sqrt(3.0) if ref.size >= 256 else 1.0) + 2.0 ** -23 * np.sqrt(k)
    assert np.linalg.norm(got - ref) <= bound * np.linalg.norm(ref)


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


def test_long_k_n_is_split(device, library, oracle):
    """K past the tiles' 31-bit ranges keeps its K split: a column tile
    walking 2^21 of K unsplit take tens of milliseconds, split under one."""
    m, n, k, gs, bits, dtype = 5, 32, (1 << 21) + 8, 32, 4, "bf16"
    outs, ref = _run_n(device, library, oracle, m, n, k, gs, bits, dtype, calls=2)
    _close(outs[0], ref, dtype, k)
    assert np.array_equal(outs[0], outs[1])
    W, S, B = (device.alloc_buffer(c, d) for c, d in ((k * n // 8, "u32"), (k * n // gs, dtype), (k * n // gs, dtype)))
    X, Y, cmds = device.alloc_buffer(m * k, dtype), device.alloc_buffer(m * n, dtype), device.commands()
    took = []
    for _ in range(5):
        cmds.commit_and_wait()
        begin = time.perf_counter()
        kqmm.affine_qmm_n(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)
        cmds.commit_and_wait()
        took.append(time.perf_counter() - begin)
    assert min(took) < 10e-3, took


@pytest.mark.parametrize("cfg", [0, 2, 4])
@pytest.mark.parametrize("k", [72, 104, 136])
def test_tile_n_skips_values_past_k(device, library, oracle, monkeypatch, cfg, k):
    """A stage of X past K holds the next row's first values: an infinity there
    must not reach the row before it."""
    monkeypatch.setenv("CPQ_TILE_CFG", str(cfg))
    m, n, gs = 40, 128, 64
    rng = np.random.default_rng(k)
    w_q, s, b = make_weight(rng, k, n, gs, 4, "bf16")
    x = make_x(rng, m, k, "bf16")
    x[8, :8] = 0x7F80
    W, S, B = (device.upload(t.reshape(-1), d) for t, d in ((w_q, "u32"), (s, "bf16"), (b, "bf16")))
    X, Y, cmds = device.upload(x.reshape(-1), "bf16"), device.alloc_buffer(m * n, "bf16"), device.commands()
    kqmm.affine_qmm_n(cmds, library, W, S, B, X, Y, m, n, k, gs, 4)
    cmds.commit_and_wait()
    y = from_bits(Y.to_numpy().reshape(m, n), "bf16")
    assert not np.isfinite(y[8]).any()
    assert np.isfinite(np.delete(y, 8, axis=0)).all()


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


def _run_t(device, library, oracle, m, n, k, gs, bits, dtype, edit=None, calls=1, skew=0):
    """affine_qmm_t and its float64 reference; `skew` starts the scales and
    biases that many elements into their allocations."""
    rng = np.random.default_rng(m * 5 + n + k + bits)
    w_q, s, b = make_weight(rng, n, k, gs, bits, dtype)
    if edit:
        edit(s, b)
    x = make_x(rng, m, k, dtype)
    W = device.upload(w_q.reshape(-1), "u32")
    pad = np.zeros(skew, np.uint16)
    S, B = (device.upload(np.concatenate([pad, t.reshape(-1)]), dtype) for t in (s, b))
    X = device.upload(x.reshape(-1), dtype)
    cmds, outs = device.commands(), []
    for _ in range(calls):
        Y = device.alloc_buffer(m * n, dtype)
        at = lambda t: ctypes.c_void_p(t.ptr + 2 * skew)  # noqa: E731
        _lib.check(_lib.lib().cpq_affine_qmm_t(
            cmds.handle, _lib.DTYPES[dtype], _ptr(W), len(W), at(S), s.size, at(B), b.size, _ptr(X), len(X), _ptr(Y),
            len(Y), m, n, k, gs, bits))
        cmds.commit_and_wait()
        outs.append(Y.to_numpy().reshape(m, n))
    w = from_bits(oracle.dequantize(w_q, s, b, n, k, gs, bits, dtype), dtype).astype(np.float64)
    return outs, from_bits(x, dtype).astype(np.float64) @ w.T


@pytest.fixture
def tiles(monkeypatch):
    """affine_qmm_t on the tiles at every M."""
    monkeypatch.setenv("CPQ_QMM_DMA", "0")
    monkeypatch.setenv("CPQ_SKINNY_MAX_M", "1")
    monkeypatch.setenv("CPQ_SMALL_ROWS", "0")
    monkeypatch.setenv("CPQ_SMALL_DENSE", "0")
    return monkeypatch


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("m,n,k,gs,bits,dtype,split,skew", [
    (2, 32, 32, 32, 6, "bf16", 1, 0),      # one 32-k stage
    (257, 288, 96, 32, 4, "bf16", 1, 1),   # one past a tile, K half a stage past one, odd table start
    (65, 128, 288, 32, 8, "f16", 2, 1),    # 9 groups a row: rows of 2-byte aligned scales
    (33, 416, 1088, 32, 3, "bf16", 3, 0),  # blocks of 8 groups end inside the parts
    (129, 384, 1024, 128, 5, "f16", 5, 1),
    (40, 256, 704, 64, 2, "bf16", 1, 0),   # 11 groups a row
    (130, 256, 2112, 64, 6, "bf16", 4, 1),
    (70, 160, 1280, 32, 4, "f16", 7, 0),
])
def test_tile_t(device, library, oracle, tiles, cfg, m, n, k, gs, bits, dtype, split, skew):
    tiles.setenv("CPQ_TILE_CFG", str(cfg))
    tiles.setenv("CPQ_QMM_SPLIT", str(split))
    outs, ref = _run_t(device, library, oracle, m, n, k, gs, bits, dtype, calls=2, skew=skew)
    _close(outs[0], ref, dtype)
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("m,n,k,gs,bits,dtype", [
    (3, 32, (1 << 21) + 32, 32, 8, "bf16"),    # one past what 256 rows of X allow
    (2, 32, (1 << 23) + 128, 128, 4, "f16"),   # the smallest tile only
])
def test_tile_t_long_k(device, library, oracle, m, n, k, gs, bits, dtype):
    """K past 2^21 stays on the tiles (those whose rows fit 31-bit ranges), its
    K split with it: the general kernel takes tens of milliseconds."""
    outs, ref = _run_t(device, library, oracle, m, n, k, gs, bits, dtype, calls=2)
    _close(outs[0], ref, dtype, k)
    assert np.array_equal(outs[0], outs[1])
    words, groups = k * n * bits // 32, k * n // gs
    W, S, B = device.alloc_buffer(words, "u32"), device.alloc_buffer(groups, dtype), device.alloc_buffer(groups, dtype)
    X, Y, cmds = device.alloc_buffer(m * k, dtype), device.alloc_buffer(m * n, dtype), device.commands()
    took = []
    for _ in range(5):
        cmds.commit_and_wait()
        begin = time.perf_counter()
        kqmm.affine_qmm_t(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)
        cmds.commit_and_wait()
        took.append(time.perf_counter() - begin)
    assert min(took) < 20e-3, took


def test_tile_t_skips_values_past_k(device, library, oracle, tiles):
    """The half stage past K holds the next row of X: an infinity there must
    not reach the row before it."""
    m, n, k, gs = 40, 64, 96, 32
    rng = np.random.default_rng(3)
    w_q, s, b = make_weight(rng, n, k, gs, 4, "bf16")
    x = make_x(rng, m, k, "bf16")
    x[7, 3] = 0x7F80
    W, S, B = (device.upload(t.reshape(-1), d) for t, d in ((w_q, "u32"), (s, "bf16"), (b, "bf16")))
    X, Y, cmds = device.upload(x.reshape(-1), "bf16"), device.alloc_buffer(m * n, "bf16"), device.commands()
    kqmm.affine_qmm_t(cmds, library, W, S, B, X, Y, m, n, k, gs, 4)
    cmds.commit_and_wait()
    y = from_bits(Y.to_numpy().reshape(m, n), "bf16")
    assert not np.isfinite(y[7]).any()
    assert np.isfinite(np.delete(y, 7, axis=0)).all()


@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("value", [2.0 ** 104, 2.0 ** 120])
def test_tile_t_large_scales(device, library, oracle, tiles, split, value):
    tiles.setenv("CPQ_QMM_SPLIT", str(split))

    def edit(s, b):
        s[70, 2] = to_bits(np.float32([value]), "bf16")[0]
        b[70, 2] = to_bits(np.float32([-2.0 ** 100]), "bf16")[0]

    outs, ref = _run_t(device, library, oracle, 70, 512, 256, 64, 4, "bf16", edit)
    _close(outs[0][:, [70]], ref[:, [70]], "bf16")
    _close(np.delete(outs[0], 70, axis=1), np.delete(ref, 70, axis=1), "bf16")


def _graph_us(device, library, m, n, k, gs, bits, calls=20):
    """us a call of affine_qmm_t: the best of a few replays of a graph of calls."""
    words, groups = n * k * bits // 32, n * k // gs
    W, S, B = (device.alloc_buffer(c, d) for c, d in ((words, "u32"), (groups, "bf16"), (groups, "bf16")))
    X, Y, cmds = device.alloc_buffer(m * k, "bf16"), device.alloc_buffer(m * n, "bf16"), device.commands()

    def encode():
        for _ in range(calls):
            kqmm.affine_qmm_t(cmds, library, W, S, B, X, Y, m, n, k, gs, bits)

    encode()
    cmds.commit_and_wait()
    cmds.begin_capture()
    encode()
    graph = cmds.end_capture()
    took = []
    for _ in range(12):
        begin = time.perf_counter()
        graph.launch(cmds)
        cmds.commit_and_wait()
        took.append(time.perf_counter() - begin)
    graph.close()
    return min(took) / calls * 1e6


@pytest.mark.parametrize("m,n,k,gs,bits,other", [
    (607, 3456, 2048, 32, 4, {"CPQ_QMM_SPLIT": "1"}),     # two-wave kernel, tiles a quarter slower
    (143, 11744, 2048, 32, 4, {"CPQ_QMM_SPLIT": "1"}),
    (3, 24064, 10592, 32, 4, {"CPQ_SMALL_DENSE": "1"}),   # the dense form, tiles half as slow again
    (4, 22880, 4032, 64, 4, {"CPQ_SMALL_DENSE": "1"}),
])
def test_tiles_only_where_they_are_faster(device, library, monkeypatch, m, n, k, gs, bits, other):
    """The routed call takes no longer than the kernel the tiles compete with
    (forced: the two-wave kernel by a split of one, the dense form by its
    hook), with an allowance for timing of half of what the tiles lose; routed
    calls are timed on both sides of the forced ones."""
    routed = _graph_us(device, library, m, n, k, gs, bits)
    with monkeypatch.context() as forcing:
        for name, value in other.items():
            forcing.setenv(name, value)
        forced = _graph_us(device, library, m, n, k, gs, bits)
    routed = min(routed, _graph_us(device, library, m, n, k, gs, bits))
    assert routed <= 1.12 * forced, (routed, forced)
