"""Weight gradients over enough rows to be summed in slices (from 2,048 rows, operands whose rows start at 16
bytes), one row less and odd widths (one sum each), and the training step whose gradient is stored first and
applied by a pass of its own.  The models and bounds are those of the products at tile edges."""
import pytest
import test_gpu_mlp_tiles as tiles

from spock_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


@pytest.mark.parametrize("n_in,hidden,n_out,rows", [(8, 64, 16, 2048), (8, 64, 16, 2047), (16, 136, 8, 4100), (24, 200, 264, 3073),
                                                    (9, 65, 15, 2049)])
def test_gradients_of_many_rows(ctx, n_in, hidden, n_out, rows):
    tiles.test_products_at_tile_edges(ctx, n_in, hidden, n_out, rows)


@pytest.mark.parametrize("hidden,layers,count", [(64, 2, 2048), (65, 2, 2048), (8, 1, 3100)])
def test_training_step_of_many_rows(ctx, problem_dirs, hidden, layers, count):
    tiles.test_predictions_and_training_step(ctx, problem_dirs, "small", hidden, layers, count)
