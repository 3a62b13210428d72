"""The float64 RBM forward of more than 512 hidden units, one row of W at a time, on both
sides of the line (896) above which every register is loaded: as test_gpu_rbm_forward."""
import numpy as np
import pytest

from .test_gpu_rbm_forward import test_forward as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [575, 576, 577, 833, 895, 896, 897, 960, 961])
def test_partly_filled_registers(M):
    check(M, np.float64)
