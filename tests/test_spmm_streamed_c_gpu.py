"""C is streamed where B, C and D are twice the Infinity Cache (streams_c), against exact integer products."""
import pytest

from tests import spmm_large

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,X,N,per,permuted,residual,streamed", [
    (128, 33, 32768, 700, True, True, 1),
    (128, 33, 14336, 700, False, True, 0),  # cached
    (64, 33, 61440, 1400, False, True, 1),
    (32, 64, 61440, 150, True, True, 1),
    (16, 64, 122880, 150, True, True, 1),
])
def test_streamed_c(torch_gpu, V, X, N, per, permuted, residual, streamed):
    kept, K = spmm_large.lengths(X, per), 2 * per
    assert spmm_large.launch(V, kept, K, N, permuted, residual)[0] == streamed
    spmm_large.check(torch_gpu, V, kept, K, N, permuted, residual)
