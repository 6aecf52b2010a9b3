"""The decode kernel for any K (up to 16 rows, every width): edges of columns,
128-k steps, groups and waves; scales too large for the subnormal form."""
import ctypes
import time

import numpy as np
import pytest

from cider_press_amd import _lib
from cider_press_amd.kernels import _ptr
from cider_press_amd.kernels import qmv as kqmv
from cider_press_amd.synthetic import from_bits, make_weight, make_x, to_bits

pytestmark = pytest.mark.gpu


def _run(device, oracle, m, n, k, gs, bits, dtype, edit=None, skew=0):
    rng = np.random.default_rng(m * 3 + n + k + bits)
    w_q, s, b = make_weight(rng, n, k, gs, bits, dtype)
    if edit:
        edit(s, b)
    x = make_x(rng, m, k, dtype)
    W = device.upload(w_q.reshape(-1), "u32")
    pad = np.zeros(skew, np.uint16)
    S, B = (device.upload(np.concatenate([pad, t.reshape(-1)]), dtype) for t in (s, b))
    X, Y = device.upload(x.reshape(-1), dtype), device.alloc_buffer(m * n, dtype)
    at = lambda t: ctypes.c_void_p(t.ptr + 2 * skew)  # noqa: E731
    cmds, L = device.commands(), _lib.lib()
    if m == 1:
        _lib.check(L.cpq_affine_qmv(cmds.handle, _lib.DTYPES[dtype], _ptr(W), len(W), at(S), s.size, at(B), b.size,
                                    _ptr(X), X.alloc_len, _ptr(Y), len(Y), k, gs, bits))
    else:
        _lib.check(L.cpq_affine_qmm_t(cmds.handle, _lib.DTYPES[dtype], _ptr(W), len(W), at(S), s.size, at(B), b.size,
                                      _ptr(X), len(X), _ptr(Y), len(Y), m, n, k, gs, bits))
    cmds.commit_and_wait()
    w = from_bits(oracle.dequantize(w_q, s, b, n, k, gs, bits, dtype), dtype).astype(np.float64)
    return (from_bits(Y.to_numpy().reshape(m, n), dtype).astype(np.float64),
            from_bits(x, dtype).astype(np.float64) @ w.T, dtype)


def _close(y, ref, dtype):
    """Rounding to T errs by at most u of a value (2^-8 with bf16's 8 significant
    bits, 2^-11 with f16's 11), and evenly up to there over many values: their
    root mean square is at most u / sqrt(3).  fp32 sums of K terms add
    2^-24 of partial sums as large as the result at random: under 1e-4 for the
    bf16 cases' K (up to 2^21), 1e-5 for the f16 ones'."""
    assert np.isfinite(y).all()
    u = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    bound = u / (np.sqrt(3.0) if ref.size >= 256 else 1.0) + (1e-5 if dtype == "f16" else 1e-4)
    assert np.linalg.norm(y - ref) <= bound * np.linalg.norm(ref)


@pytest.mark.parametrize("waves", [0, 1, 3, 12, 40])  # out of range: the nearest
@pytest.mark.parametrize("m,n,k,gs,bits,dtype,skew", [
    (1, 1, 32, 32, 6, "bf16", 0),        # one column, a quarter step
    (1, 17, 96, 32, 3, "f16", 1),        # one column past a block, tables on an odd element
    (1, 131, 2080, 32, 5, "bf16", 1),    # 65 groups a row
    (1, 48, 4416, 64, 2, "f16", 0),      # 69 groups, half a step at the end, several batches a wave
    (1, 40, 1152, 64, 4, "bf16", 1),
    (1, 33, 1152, 128, 8, "f16", 0),
    (2, 64, 3520, 64, 4, "bf16", 1),
    (5, 96, 2112, 64, 8, "f16", 1),
    (16, 160, 1376, 32, 6, "bf16", 0),
    (13, 96, 896, 128, 3, "bf16", 0),
])
def test_decode(device, oracle, monkeypatch, waves, m, n, k, gs, bits, dtype, skew):
    monkeypatch.setenv("CPQ_DECODE_WAVES", str(waves))
    _close(*_run(device, oracle, m, n, k, gs, bits, dtype, skew=skew))


@pytest.mark.parametrize("n,k,gs,bits,dtype", [
    (48, 16224, 32, 4, "bf16"),      # x and 16 rows' constants: 159 to 160 KiB, more than the shared-staging kernel gets
    (48, 16256, 32, 4, "bf16"),
    (33, 16288, 32, 8, "f16"),
    (40, 27072, 64, 8, "bf16"),
    (40, 27136, 64, 8, "f16"),
    (17, 40576, 128, 8, "bf16"),
    (5120, 17920, 32, 4, "bf16"),    # past it
    (33, 81920, 64, 4, "bf16"),      # x past a workgroup's LDS
    (20, 98304, 128, 8, "f16"),
    (16, 80064, 64, 6, "bf16"),
    (16, (1 << 21) + 64, 64, 4, "bf16"),
])
def test_one_long_row(device, oracle, n, k, gs, bits, dtype):
    """Decode with K past what the layouts with x and constants in LDS take."""
    _close(*_run(device, oracle, 1, n, k, gs, bits, dtype))


@pytest.mark.parametrize("m", [1, 3])
def test_decode_large_scales(device, oracle, m):
    """bf16 scales of 2^104 and above overflow the subnormal form."""
    def edit(s, b):
        for col, value in ((5, 2.0 ** 104), (40, 2.0 ** 112)):
            s[col, 2] = to_bits(np.float32([value]), "bf16")[0]
            b[col, 2] = to_bits(np.float32([-2.0 ** 100]), "bf16")[0]

    y, ref, dtype = _run(device, oracle, m, 64, 1280, 64, 6, "bf16", edit)
    for cols in ([5], [40], [c for c in range(64) if c not in (5, 40)]):
        _close(y[:, cols], ref[:, cols], dtype)


@pytest.mark.parametrize("n,k,gs,bits,dtype", [
    (200, 7168, 64, 4, "bf16"),      # waves with ranges of different lengths
    (8200, 2816, 64, 4, "f16"),      # the same on 512 column blocks
    (33, 20480, 128, 4, "bf16"),     # every wave whole batches
    (40, 9984, 32, 4, "f16"),
    (48, 9216, 64, 8, "bf16"),
    (8200, 3520, 64, 8, "f16"),
    (17, 20480, 128, 8, "bf16"),
])
def test_shared_staging(device, oracle, n, k, gs, bits, dtype):
    """Decode shapes that stay on the shared-staging kernel."""
    def edit(s, b):
        s[::3, ::5] = 0  # zero scales: its exact form inside one workgroup

    _close(*_run(device, oracle, 1, n, k, gs, bits, dtype, edit))


def test_one_row_costs_as_its_neighbours(device, library):
    """K = 7168 (7 x 1024) on a kernel of its own next to the lean layout's 8192:
    a wave with a second, mostly empty batch made it take 1.8 times as long."""
    def us(n, k, gs=64, calls=20):
        W, S, B = (device.alloc_buffer(c, d) for c, d in ((n * k // 8, "u32"), (n * k // gs, "bf16"),
                                                          (n * k // gs, "bf16")))
        X, Y, cmds = device.alloc_buffer(k, "bf16"), device.alloc_buffer(n, "bf16"), device.commands()

        def encode():
            for _ in range(calls):
                kqmv.affine_qmv(cmds, library, W, S, B, X, Y, k, gs, 4)

        encode()
        cmds.commit_and_wait()
        cmds.begin_capture()
        encode()
        graph, took = cmds.end_capture(), []
        for _ in range(12):
            begin = time.perf_counter()
            graph.launch(cmds)
            cmds.commit_and_wait()
            took.append(time.perf_counter() - begin)
        graph.close()
        return min(took) / calls * 1e6

    odd, even = us(4672, 7168), us(4672, 8192)
    assert odd <= 1.4 * even, (odd, even)


def test_decode_skips_values_past_k(device, oracle):
    """Rows of X follow one another: an infinity at the next row's start must not
    reach the partial last step of the row before it."""
    m, n, k, gs, bits = 3, 32, 1184, 32, 6
    rng = np.random.default_rng(2)
    w_q, s, b = make_weight(rng, n, k, gs, bits, "bf16")
    x = make_x(rng, m, k, "bf16")
    x[1, 0] = 0x7F80
    W, S, B = (device.upload(t.reshape(-1), d) for t, d in ((w_q, "u32"), (s, "bf16"), (b, "bf16")))
    X, Y, cmds = device.upload(x.reshape(-1), "bf16"), device.alloc_buffer(m * n, "bf16"), device.commands()
    _lib.check(_lib.lib().cpq_affine_qmm_t(cmds.handle, _lib.DTYPES["bf16"], _ptr(W), len(W), _ptr(S), len(S), _ptr(B),
                                           len(B), _ptr(X), len(X), _ptr(Y), len(Y), m, n, k, gs, bits))
    cmds.commit_and_wait()
    y = from_bits(Y.to_numpy().reshape(m, n), "bf16")
    assert np.isfinite(y[[0, 2]]).all() and not np.isfinite(y[1]).any()


@pytest.mark.parametrize("m,n,k,gs,bits,dtype,skew", [
    (16, 32, 128, 64, 6, "bf16", 0),      # one step, one wave
    (13, 64, 6496, 32, 3, "f16", 1),      # a partial last step, odd group counts
    (7, 64, 12288, 64, 8, "bf16", 0),     # two phases, whole
    (16, 96, 9632, 32, 5, "bf16", 1),     # 9 waves, a last phase of part of a batch, a last wave with fewer steps
    (12, 2080, 8064, 128, 8, "f16", 0),   # as the route takes it
    (2, 32, 40960, 64, 4, "f16", 1),      # one row block, many batches a phase; more groups than the slab kernel holds
    (16, 32, 30720, 64, 2, "bf16", 0),    # many phases
])
def test_decode_phased(device, oracle, monkeypatch, m, n, k, gs, bits, dtype, skew):
    """Activations staged in phases, where the rows exceed a workgroup's LDS."""
    monkeypatch.setenv("CPQ_DECODE_PHASED", "1")

    def edit(s, b):
        if dtype == "bf16":  # a wave that meets a large scale goes over its phases again
            s[5, -1], b[5, -1] = to_bits(np.float32([2.0 ** 104, -2.0 ** 100]), "bf16")

    y, ref, dtype = _run(device, oracle, m, n, k, gs, bits, dtype, edit, skew)
    for cols in ([5], [c for c in range(n) if c != 5]):
        _close(y[:, cols], ref[:, cols], dtype)


@pytest.mark.parametrize("m,n,k,gs,bits,phased,large", [
    (1, 64, 6112, 32, 6, False, False),
    (16, 64, 2080, 32, 5, False, True),   # rows staged four at a time, the large-scale pass reads them again
    (16, 64, 9632, 32, 3, True, False),   # a wave's lanes refill what other lanes were reading
    (7, 64, 12288, 64, 8, True, True),
])
def test_decode_lanes_read_what_others_staged(device, oracle, monkeypatch, m, n, k, gs, bits, phased, large):
    """Lanes of a wave read activations that other lanes wrote to LDS.  Calls on
    other values in between leave theirs there: whoever read early would see
    them, so every call gives the first one's bits."""
    if phased:
        monkeypatch.setenv("CPQ_DECODE_PHASED", "1")

    def edit(s, b):
        if large:
            s[5, -1], b[5, -1] = to_bits(np.float32([2.0 ** 104, -2.0 ** 100]), "bf16")

    def other(s, b):
        s[:] = to_bits(np.full(s.size, 0.5, np.float32), "bf16").reshape(s.shape)

    y, ref, dtype = _run(device, oracle, m, n, k, gs, bits, "bf16", edit)
    for cols in ([5], [c for c in range(n) if c != 5]):
        _close(y[:, cols], ref[:, cols], dtype)
    for _ in range(3):
        _run(device, oracle, m, n, k, gs, bits, "bf16", other)
        assert np.array_equal(_run(device, oracle, m, n, k, gs, bits, "bf16", edit)[0], y)
