"""GPU PQ encoding through the matrix-core filter (vk_pq_encode): codes must be the oracle's for every sub-vector width
with an instance (2, 3, 4, 6, 8, 12, 16) and others, at sizes around a wave and a block, with near ties (centroids a few
units in the last place apart), exact ties, magnitudes that leave the filter's range, infinities and NaN.
"""
import numpy as np
import pytest

import veckern_amd as vk
from oracle import binding as orc

pytestmark = pytest.mark.gpu


def case(seed, n, m, dsub):
    rng = np.random.default_rng(seed)
    cent = rng.standard_normal((m, 256, dsub)).astype(np.float32)
    return cent, rng.standard_normal((n, m * dsub)).astype(np.float32), rng


@pytest.mark.parametrize("dsub", [1, 2, 3, 4, 5, 6, 8, 12, 16])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 63), (16, 257), (9, 1025), (2, 20_011)])
def test_encode_widths_and_sizes(dsub, m, n):
    cent, x, _ = case(dsub * 100 + n, n, m, dsub)
    assert (vk.pq_encode(cent, x) == orc.pq_encode(cent, x)).all()


@pytest.mark.parametrize("dsub", [2, 8, 16])
def test_encode_near_ties(dsub):
    cent, x, rng = case(7 + dsub, 30_000, 4, dsub)
    half = cent[:, :128]
    cent[:, 128:] = np.nextafter(half, np.where(rng.random(half.shape) < 0.5, -np.inf, np.inf).astype(np.float32))
    x[::2] = cent[:, rng.integers(0, 256, 15_000)].transpose(1, 0, 2).reshape(15_000, -1)  # on a centroid
    assert (vk.pq_encode(cent, x) == orc.pq_encode(cent, x)).all()


@pytest.mark.parametrize("dsub", [2, 4, 8, 12])
def test_encode_special_values(dsub):
    cent, x, rng = case(17 + dsub, 4_000, 3, dsub)
    cent[0, 3] = np.inf
    cent[1, 9, 0] = np.nan
    x[5, 0], x[6, -1] = np.inf, np.nan
    for row, scale in ((10, 1e-30), (11, 1e-20), (12, 1e13), (13, 1e19), (14, 3e38), (15, 0.0)):
        x[row] = np.clip(x[row], -1, 1) * np.float32(scale)
    with np.errstate(all="ignore"):
        assert (vk.pq_encode(cent, x) == orc.pq_encode(cent, x)).all()
    for scale in (1e-30, 1e-12, 1e6, 1e13, 1e25):
        c2, x2, _ = case(27 + dsub, 2_000, 3, dsub)
        c2, x2 = c2 * np.float32(scale), x2 * np.float32(scale)
        assert (vk.pq_encode(c2, x2) == orc.pq_encode(c2, x2)).all(), scale
