"""The temporally blocked kernel with from one to 146 steps per launch (the halo takes
7 sites per step of a segment's 2048 or 1024): short chains, where the chain bounds the
halo, single chains, whose run is one launch, and ensembles; against the CPU oracle."""
import pytest

from test_gpu_parity import check_move

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,copies,steps", [(256, 3, 1), (257, 2, 40), (1021, 1, 150), (2100, 1, 146), (5003, 2, 147),
                                            (17000, 1, 75), (17000, 60, 20)])
@pytest.mark.parametrize("model_name", ["DNKG", "Toda"])
def test_tiled_steps(gpu, model_name, n, copies, steps):
    check_move(gpu, model_name, n, copies, steps=steps, dens=0.1, plane=True, kernel=gpu.KERNEL_TILED,
               expect="kernel=tiled")
