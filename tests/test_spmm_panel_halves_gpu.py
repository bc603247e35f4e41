"""Large D over few long panels: the XCDs take the panels in halves (panel_halves): both sides of the rule, odd numbers of
panels, column tiles that do and do not divide by four, panels that keep nothing, rows permuted and not, against exact
integer products."""
import pytest

from tests import spmm_large

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,X,N,per,permuted,residual,first", [
    (128, 33, 12288, 800, True, False, 16),   # halves of 16 and 17 panels, 48 column tiles
    (128, 33, 12352, 800, False, True, 16),   # a last tile of 64 columns; 49 column tiles: ranges that split a column tile
    (128, 33, 32768, 800, True, True, 16),    # C streamed
    (128, 64, 16384, 420, True, False, 32),   # a pitch of 32 KiB, as many panels to a half as an XCD has workgroups
    (128, 64, 16448, 420, False, False, 0),   # another pitch: not halved
    (128, 48, 16384, 200, True, True, 24),    # that pitch, a short A: halved with C and permuted rows only
    (128, 48, 16384, 200, False, True, 0),
    (128, 48, 16384, 200, True, False, 0),
    (128, 81, 16384, 320, False, False, 40),  # more panels to a half than an XCD has workgroups
    (128, 24, 18432, 1100, False, True, 12),  # the fewest panels
    (128, 23, 18432, 1100, True, True, 0),
    (128, 9, 46080, 3300, True, True, 0),
    (128, 41, 12288, 650, True, False, 0),    # more panels than at any pitch
    (64, 33, 24576, 1400, False, False, 0),   # a block height that is not halved
])
def test_panel_halves(torch_gpu, V, X, N, per, permuted, residual, first):
    kept, K = spmm_large.lengths(X, per), 2 * per
    if V == 128:
        assert spmm_large.launch(V, kept, K, N, permuted, residual)[1] == first
    spmm_large.check(torch_gpu, V, kept, K, N, permuted, residual)


@pytest.mark.parametrize("X,N,per,residual,first", [
    (33, 12288, 800, False, 16),
    (64, 16384, 420, True, 32),
])
def test_stages_in_alternating_order(torch_gpu, X, N, per, residual, first):
    kept, K = spmm_large.lengths(X, per), 5400  # rows of B under a column tile: 2.8 MB
    assert spmm_large.launch(128, kept, K, N, True, residual)[1] == first
    spmm_large.check(torch_gpu, 128, kept, K, N, True, residual)


def test_uneven_panels(torch_gpu):
    kept = [1400] * 10 + [500] * 23
    assert spmm_large.launch(128, kept, 2000, 12288, True, False)[1] == 11
    spmm_large.check(torch_gpu, 128, kept, 2000, 12288, True, False)
