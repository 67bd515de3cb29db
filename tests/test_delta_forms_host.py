"""Which segments of a step the delta rule takes 16 tokens at a time: a rule on lengths, so on the host (256 compute units where no device is in use)."""
import numpy as np
import pytest

from xfastertransformer_amd import capi as xh

WIDE = (16, 128, 128, 4, False)  # 128 tiles of 16 columns a segment


@pytest.mark.parametrize("layer,lens,forms", [
    (WIDE, [16], [1]), (WIDE, [15], [0]), (WIDE, [1500] * 4, [1] * 4),
    (WIDE, [1500, 1, 1], [1] * 3),  # most of the device idle: the short ones go along
    (WIDE, [32] * 16, [1] * 16), (WIDE, [31] * 16, [0] * 16),
    (WIDE, [400] * 16 + [1] * 3, [1] * 19), (WIDE, [400] * 16 + [1] * 4, [1] * 16 + [0] * 4),
    # prompts beside decoding sequences: each by its own length
    (WIDE, [500] + [1] * 50, [1] + [0] * 50), (WIDE, [1] * 20 + [64, 63] + [8] * 9, [0] * 20 + [1, 0] + [0] * 9), (WIDE, [32] + [1] * 200, [0] * 201),
    ((32, 128, 128, 4, True), [500, 128, 127] + [1] * 50, [1, 1, 0] + [0] * 50), ((32, 128, 128, 4, True), [127] * 16, [0] * 16), ((32, 128, 128, 4, True), [128] * 16, [1] * 16),
    ((16, 32, 64, 4, False), [500], [0]), ((16, 128, 128, 1, False), [500], [0]), ((16, 128, 128, 5, False), [500], [0]), ((4, 33, 40, 2, False), [500], [1]),
])
def test_forms(layer, lens, forms):
    assert xh.delta_forms(*layer, lens) == forms


def test_short_segments_stay_out_of_large_steps():
    """A segment of a token or a few costs a whole chunk there: many of them never go, whatever is beside them; and the order of the segments changes nothing."""
    rng = np.random.default_rng(3)
    for _ in range(300):
        layer = (int(rng.choice([8, 16, 64])), int(rng.choice([64, 100, 256])), int(rng.choice([64, 128])), int(rng.integers(2, 5)), bool(rng.integers(2)))
        tiles = layer[0] * layer[2] // 16
        short = -(-512 // tiles) + int(rng.integers(0, 60))
        lens = np.concatenate([rng.integers(1, 9, short), rng.integers(1, 2000, rng.integers(1, 30))])
        if len(lens) * tiles < 1024:
            continue
        forms = np.array(xh.delta_forms(*layer, lens))
        assert not forms[lens < 64].any() and forms[lens >= 128].all()
        order = rng.permutation(len(lens))
        assert (np.array(xh.delta_forms(*layer, lens[order])) == forms[order]).all()


@pytest.mark.parametrize("lens", [[0], [5, -1]])
def test_refused(lens):
    with pytest.raises(xh.XftHipError):
        xh.delta_forms(*WIDE, lens)
