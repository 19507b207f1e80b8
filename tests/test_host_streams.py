"""CPU: the host codec's streams (drinkme_amd/csrc/codec.cpp packs and unpacks
eight fields at a time through 64-bit words) at every tier width and at the
remainders of eight fields, a word and a block, against the oracle's bytes; and
the round-trip comparison (op 4), which must see one changed bit anywhere."""

import numpy as np
import pytest

from drinkme_amd import radix_pack as rp
from oracle import radix_oracle as O
from tests.helpers import escape_heavy_bits, finite_bits

WIDTHS = [(w, 8) for w in range(1, 9)] + [(2, 2, 4, 8), (5, 6, 8), (7, 7, 8), (1, 1, 1, 1, 1, 1, 1, 8)]
COLS = [1, 7, 8, 9, 31, 1023, 1024, 1025, 2041, 3078]


@pytest.mark.parametrize("widths", WIDTHS)
@pytest.mark.parametrize("kind", ["spread", "escapes"])
def test_streams_of_every_width_are_the_oracles(widths, kind):
    rng = np.random.default_rng(len(widths) * 100 + widths[0])
    for cols in COLS:
        shape = (5, cols)
        bits = finite_bits(rng, shape, spread=True) if kind == "spread" else escape_heavy_bits(rng, shape, 0.35)
        palette, offsets, data = rp.encode(bits, widths)
        o = O.pack(bits, widths=widths, allow_raw=False)
        assert np.array_equal(palette, o.palette) and np.array_equal(offsets, o.offsets), cols
        assert np.array_equal(data, o.data), cols
        assert np.array_equal(rp.decode(palette, offsets, data, *shape, widths), bits), cols


@pytest.mark.parametrize("widths", [(3, 8), (2, 3, 8), (2, 2, 4, 8)])
def test_the_comparison_sees_one_changed_bit(widths):
    rng = np.random.default_rng(7)
    bits = finite_bits(rng, (300, 1500), spread=True)
    codec = rp.HostCodec(300, 1500, widths)
    tables, offsets, data = codec.compress(bits)
    before = bits.copy()
    assert codec.op(codec.COMPARE, bits, tables, offsets, data, 0, 300) == 1
    assert np.array_equal(bits, before), "the source is only read"
    assert codec.op(codec.COMPARE, bits[100:], tables, offsets, data, 100, 200) == 1
    for r, c, b in ((0, 0, 0), (299, 1499, 15), (150, 1023, 7), (150, 1024, 14)):
        other = bits.copy()
        other[r, c] ^= np.uint16(1 << b)
        assert codec.op(codec.COMPARE, other, tables, offsets, data, 0, 300) == 0, (r, c, b)
    with pytest.raises(ValueError, match="range"):
        codec.op(codec.COMPARE, bits, tables, offsets, data, 200, 101)
