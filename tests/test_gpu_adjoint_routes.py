"""The Cahn-Hilliard adjoint on long thin grids, whose x axis is cut into more
than 64 chunks, against autograd through the float64 oracle."""
import pytest

from tests.test_gpu_adjoint_stream import test_tile_edges as against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["float64", "float32"])
@pytest.mark.parametrize("shape,c,based", [((300, 2, 3), 1, True), ((2001, 9, 5), 2, False), ((4000, 1, 70), 1, True)])
def test_more_than_64_chunks(shape, c, based, precision):
    against_oracle(shape, c, based, precision)
