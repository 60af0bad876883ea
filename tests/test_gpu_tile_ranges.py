"""The four-step kernel's tiles of 16 at two to a CU, between the last grid
that 512 tiles of 12 cover and the first that marches, against one-step
launches: just past the former (552 tiles of 12, 306 of 16) and just within the
latter (506 of 16)."""
import pytest
import torch

from test_gpu_tiles import test_tiles_match_one_step_launches as match_one_step_launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(277, 270), (352, 368)])
@pytest.mark.parametrize("bc", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_sixteen_cells_two_to_a_cu(gpu, dtype, bc, shape):
    def tiles(side):
        return -(-shape[0] // side) * -(-shape[1] // side)

    assert tiles(12) > 512 and 256 < tiles(16) <= 512
    match_one_step_launches(gpu, dtype, bc, shape)
