"""Smooth dabs on both sides of the rule for their workgroups (about 512 gathered leaves) and
over halo sizes from one local a thread to several, against the separate kernels."""
import numpy as np
import pytest

from test_gpu_chain import _check, _path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,leaf,radii", [(6, 9, (0.15, 0.3, 0.5, 0.9)), (6, 20, (0.3, 0.7)), (5, 128, (0.2, 2.5)),
                                              (4, 300, (0.3, 1.0)), (5, 900, (0.3, 1.0))])
@pytest.mark.parametrize("k", [1, 4, 7])
def test_smooth(sg, level, leaf, radii, k):
    co, tris = sg.noisy_icosphere(level, seed=5, amplitude=0.02)
    _check(sg, co, tris, _path(sg, 6, 6, np.resize(radii, 6), (2, 2, 1), (k,)), leaf=leaf)
