"""Toda shapes of 8 to 24 sites per lane, whose bonds are evaluated in runs of
four (wave kernels) or two (workgroup kernels): whole runs and remainders, with
full lanes and with lanes one site short, against the CPU oracle."""
import pytest

from test_gpu_parity import check_move

pytestmark = pytest.mark.gpu

# (n, lanes, sites per lane); 128 lanes and more are the workgroup form
SHAPES = [(8, 1, 8), (11, 1, 11), (24, 1, 24), (64, 8, 8), (128, 16, 8), (137, 16, 9), (144, 16, 9), (175, 16, 11),
          (379, 16, 24), (449, 64, 8), (512, 64, 8), (513, 64, 9), (1025, 64, 17), (1408, 64, 22), (1535, 64, 24),
          (1024, 128, 8), (2048, 128, 16), (1030, 128, 9), (2432, 128, 19), (3000, 128, 24), (3071, 128, 24)]


@pytest.mark.parametrize("n,L,S", SHAPES)
def test_toda_runs(gpu, n, L, S):
    check_move(gpu, "Toda", n, 7, steps=60, dens=0.25, lanes_per_chain=L, sites_per_lane=S)
