"""The packed density product at the edges of its tiles and chunks: 64-wide
tiles, 32 levels a chunk in two halves of 16, against numpy."""
import numpy as np
import pytest

from mopac_gpu_amd import geometry, hamiltonian

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,occupied", [(1, (0, 1, 5, 6)), (11, (1, 15, 16, 17, 31, 32, 33, 66)),
                                             (22, (47, 48, 49, 63, 64, 65, 132)), (43, (1, 172, 257, 258))])
def test_packed_density_matches_numpy(gpu_ctx, waters, occupied):
    s = hamiltonian.build(*geometry.water_cluster(waters, 5))
    n = s.norbs
    gpu_ctx.upload(s)
    c = np.asfortranarray(np.random.default_rng(n).standard_normal((n, n)))
    for k in occupied:
        want = 2.0 * c[:, :k] @ c[:, :k].T
        got = gpu_ctx.density(c, k)
        # sums of k products of order 1, in any order
        assert np.max(np.abs(got - want[np.tril_indices(n)])) <= 4e-15 * max(k, 1) * max(1.0, np.max(np.abs(c)) ** 2)
