"""Host check of the dequantization through f16 subnormals.

A packed value q left at bit p of a 16-bit half reads as the f16 subnormal
q * 2^(p - 24); the kernels compute fma(s * 2^24 * 2^-p, q * 2^(p - 24), b)
(cider_press_amd/csrc/kernels/subnormal.hpp).  That is fmaf(s, q, b) exactly
when s * 2^24 * 2^-p is a finite fp32 value and its product with the subnormal
is the real number s * q: checked here for every scale pattern below the
header's limit, every value and every place of every width."""
import pathlib
import re

import numpy as np
import pytest

from cider_press_amd.synthetic import from_bits

HEADER = (pathlib.Path(__file__).resolve().parent.parent / "cider_press_amd" / "csrc" / "kernels" / "subnormal.hpp").read_text()
LIMIT = {"bf16": eval(re.search(r"kSubScaleLimit = Sig16<TT>::bf16 \? (\d+)u << (\d+)", HEADER).expand(r"\1 << \2")), "f16": 0x10000}
# Bit places of each width's fields (val<place> in the header).
PLACES = {2: (0, 2, 4, 6), 3: range(8), 4: (0, 4), 5: range(6), 6: (0, 2, 4), 8: (0,)}


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
def test_product_is_exact(bits, dtype):
    q = np.arange(1 << bits)
    pattern = np.arange(0x8000)
    s = from_bits(pattern.astype(np.uint16), dtype)
    below = (pattern < LIMIT[dtype]) & np.isfinite(s)
    with np.errstate(over="ignore", invalid="ignore"):
        s24 = s * np.float32(2.0 ** 24)  # the limit is where this leaves fp32
    assert np.isfinite(s24[below]).all()
    if dtype == "bf16":
        finite = np.isfinite(s)
        assert not np.isfinite(s24[finite & ~below]).any()
    for p in PLACES[bits]:
        assert bits + p <= 10
        h = (q << p).astype(np.uint16).view(np.float16).astype(np.float64)
        assert np.array_equal(h, q * 2.0 ** (p - 24))
        c = (s24[below] * np.float32(2.0 ** -p)).astype(np.float64)
        assert np.array_equal(c, s[below].astype(np.float64) * 2.0 ** (24 - p))  # exact in fp32
        # 24 + 10 significant bits: exact in float64
        assert np.array_equal(c[:, None] * h[None, :], s[below].astype(np.float64)[:, None] * q[None, :])
        # Larger scales: the field scaled to q first.
        assert np.array_equal(h.astype(np.float32) * np.float32(2.0 ** 24 / (1 << p)), q.astype(np.float32))


def test_places_are_the_headers():
    """PLACES holds every place the header uses (per width's branch)."""
    branches = re.split(r"BITS == (\d)\b", HEADER[HEADER.index("u32x4 sub_group"):])
    for bits, text in zip(branches[1::2], branches[2::2]):
        used = {int(p) for p in re.findall(r"val<(\d+)>", text)}
        assert used == set(PLACES[int(bits)]), bits
