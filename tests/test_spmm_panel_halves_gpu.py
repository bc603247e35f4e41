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
    (128, 9, 46080, 3300, True, True, 4),     # fewer panels than workgroups of an XCD
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
