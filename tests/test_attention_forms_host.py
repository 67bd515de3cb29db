"""Which form of the kernels a prompt takes: rules on sizes, so on the host (256 compute units where no device is in use)."""
import pytest

from xfastertransformer_amd import capi as xh


@pytest.mark.parametrize("q,kv,batch,tokens,past,int8,form", [
    (32, 8, 1, 100, 0, False, 0), (32, 8, 1, 100, 0, True, 0), (32, 8, 64, 1, 2000, False, 0),
    (32, 8, 8, 500, 0, False, 1), (32, 8, 4, 800, 0, False, 1), (32, 8, 1, 512, 8000, False, 1), (32, 8, 8, 400, 0, True, 1), (32, 8, 1, 511, 0, True, 1),
    (32, 8, 4, 2000, 0, False, 2), (32, 8, 1, 4000, 0, False, 2), (32, 8, 8, 1000, 0, False, 2), (32, 8, 1, 512, 0, True, 2), (32, 8, 1, 512, 8000, True, 2),
])
def test_contiguous(q, kv, batch, tokens, past, int8, form):
    assert xh.attention_prefill_form(q, kv, batch, tokens, past, int8) == form


@pytest.mark.parametrize("q,kv,lens,forms", [
    (32, 8, [1500, 1400, 1200, 1000, 900, 750], [2] * 6),
    (32, 8, [40, 3000] + [60] * 30, [2] * 32),  # most of the work is the long one's
    # one long sequence beside many short ones, whose columns see few tokens: as a batch of its length alone it would be taken for twice and three times the work
    (32, 8, [1500] + [60] * 60, [1] * 61),
    (32, 8, [64] * 20 + [1200] + [64] * 43, [1] * 64),
    (32, 8, [1000] * 3, [1] * 3),
    (24, 24, [2000, 200, 200], [1, 0, 0]),  # too few workgroups
    (32, 8, [33, 1700, 701], [0, 2, 2]),
    (32, 8, [30], [0]), (32, 8, [4000], [2]),  # alone: as over a contiguous cache
    (16, 4, [20, 30, 1], [0, 0, 0]),
])
def test_paged(q, kv, lens, forms):
    assert xh.paged_attention_prefill_forms(q, kv, lens) == forms


def test_a_call_of_several_launches():
    """64 sequences a launch, the longest first: each launch by its own sequences, forms in the caller's order."""
    lens = [50] * 64 + [2000] * 64
    assert xh.paged_attention_prefill_forms(32, 8, lens) == [1] * 64 + [2] * 64


@pytest.mark.parametrize("lens", [[0, 5], [-3]])
def test_refused(lens):
    with pytest.raises(xh.XftHipError):
        xh.paged_attention_prefill_forms(32, 8, lens)
