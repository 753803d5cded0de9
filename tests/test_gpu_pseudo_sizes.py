"""diag's rotations where their chain of lanes changes: one and several blocks
of 64 virtuals, ragged ones, a single occupied or virtual, steps that end in
a part of a load, and rows that no wave fills."""
import numpy as np
import pytest

from mopac_gpu_amd import geometry, hamiltonian
from oracle import oracle

pytestmark = pytest.mark.gpu


def _check(gpu_ctx, s, nocc):
    n = s.norbs
    rng = np.random.default_rng(n + nocc)
    gpu_ctx.upload(s)
    c = np.asfortranarray(np.linalg.qr(rng.standard_normal((n, n)))[0])
    f = rng.standard_normal(n * (n + 1) // 2)
    eig = np.sort(20.0 * rng.standard_normal(n))
    got, nr = gpu_ctx.diag(f, c, nocc, eig)
    want, nr_ref = oracle.diag(f, c, nocc, eig)
    assert nr == nr_ref and nr > 0
    # every coefficient: up to n rotations, angles from products of n terms
    assert np.max(np.abs(got - want)) < 1e-12 * max(1.0, n / 64)


@pytest.mark.parametrize("waters,occupied", [(1, (1, 5)), (11, (1, 2, 33, 65)), (22, (1, 17, 66, 67, 68, 69, 131)),
                                             (43, (1, 64, 65, 128, 129, 130, 194, 257))])
def test_rotations_match_oracle(gpu_ctx, waters, occupied):
    s = hamiltonian.build(*geometry.water_cluster(waters, 5))
    for nocc in occupied:
        _check(gpu_ctx, s, nocc)


@pytest.mark.parametrize("occupied", (4977, 4978, 5190))
def test_rows_that_fill_the_lds(gpu_ctx, occupied):
    """Over 4 977 occupied levels a row goes through the LDS in parts; one and
    several blocks of 64 virtuals."""
    s = hamiltonian.build(*geometry.water_cluster(870 if occupied == 5190 else 841, 5))
    _check(gpu_ctx, s, occupied)
