"""The staging blocks of the per-call entry points (host-side call of the C ABI, no device): the
kernel that copies them to the device moves whole 16-byte words, so a block must hold the input
bytes rounded up to them.  A Hermite tensor stages 8 bytes per order of its largest cutoff, so odd
cutoffs above 8190 have inputs past the smallest block that end in half a word."""
import pytest

from thewalrus_amd import _native


@pytest.mark.parametrize("modes", [1, 2, 6])
@pytest.mark.parametrize("cutoff", [1, 2, 8180, 8181, 8187, 8189, 8191, 70001, 70002])
def test_staged_words_fit_the_block(modes, cutoff):
    bytes_ = 16 * modes * modes + 16 * modes + 16 + 8 * cutoff
    assert _native.load().wh_debug_stage_capacity(bytes_) >= (bytes_ + 15) // 16 * 16


def test_capacity_of_every_remainder():
    L = _native.load()
    for b in [0, 1, *range(65520, 65570), *range(10**6, 10**6 + 300)]:
        assert L.wh_debug_stage_capacity(b) >= (b + 15) // 16 * 16 >= b
    assert L.wh_debug_stage_capacity(-1) == -1
