"""tidy and check, a wave per LMO: the kept atoms and every coefficient against
the same sums in the same order on the host, for LMOs below and above the 64
atoms and 128 coefficients that a wave takes at once."""
import math

import numpy as np
import pytest

from mopac_gpu_amd import geometry, mozyme

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def grown(gpu_ctx):
    ms = mozyme.MozymeSystem.from_geometry(*geometry.glycine_helix(24, 3))
    ms.upload(gpu_ctx)
    f0 = ms.fock2z(gpu_ctx, ms.diagonal_density())
    s = ms.scf(gpu_ctx, mozyme.lewis_lmos(ms, f0), itrmax=8)["lmos"]
    s.eigs, s.eigv = np.zeros(s.nocc), np.zeros(s.nvir)
    return s


def _sides(s, occupied):
    return (s.ncf, s.nncf, s.ncocc, s.icocc, s.cocc) if occupied else (s.nce, s.nnce, s.ncvir, s.icvir, s.cvir)


@pytest.mark.parametrize("occupied", [1, 0])
@pytest.mark.parametrize("thresh", [1e-13, 1e-5, 1e-2])
def test_tidy_keeps_and_check_scales(gpu_ctx, grown, occupied, thresh):
    nc, nn, no, ic, c = _sides(grown, occupied)
    want = []
    for k in range(len(nc)):
        atoms, coefs, m = [], [], no[k]
        for a in ic[nn[k]:nn[k] + nc[k]]:
            x = [float(v) for v in c[m:m + grown.iorbs[a - 1]]]
            m += len(x)
            total = 0.0
            for v in x:
                total += v * v
            if total > thresh:
                atoms.append(a)
                coefs += x
        want.append((atoms, coefs))
    assert min(nc) < 64 < max(nc) and max(len(w[1]) for w in want) > (128 if thresh < 1e-6 else 0)
    g = mozyme.GpuMozyme(gpu_ctx, grown)
    g.tidy(occupied, thresh)
    gnc, gnn, gno, gic, gc = _sides(g.get(), occupied)
    for k, (atoms, coefs) in enumerate(want):
        assert gic[gnn[k]:gnn[k] + gnc[k]].tolist() == atoms
        assert gc[gno[k]:gno[k] + len(coefs)].tolist() == coefs
    if thresh > 1e-4:
        return  # norms far from 1: check would stop the job
    error = g.check(occupied)
    gc = _sides(g.get(), occupied)[4]
    expected = 0.0
    for k, (_, coefs) in enumerate(want):
        total = 0.0
        for v in coefs:
            total += v * v
        expected += abs(1.0 - total)
        scale = 1.0 / math.sqrt(total)
        assert gc[gno[k]:gno[k] + len(coefs)].tolist() == [v * scale for v in coefs]
    assert error == expected


def test_density_from_per_atom_lists(gpu_ctx, grown):
    """The stored blocks of 2 C C^T from the atoms' lists of LMOs."""
    s = grown
    c = np.zeros((s.norbs, s.nocc))
    first = np.concatenate([[0], np.cumsum(s.iorbs)])
    for k in range(s.nocc):
        m = s.ncocc[k]
        for a in s.icocc[s.nncf[k]:s.nncf[k] + s.ncf[k]]:
            no = s.iorbs[a - 1]
            c[first[a - 1]:first[a - 1] + no, k] = s.cocc[m:m + no]
            m += no
    p = 2.0 * c @ c.T
    got = mozyme.GpuMozyme(gpu_ctx, s).density()
    nij = np.asarray(s.nijbo)
    seen = 0
    for a in range(s.numat):
        for b in range(a + 1):
            if nij[a, b] < 0:
                continue
            block = p[first[a]:first[a + 1], first[b]:first[b + 1]]
            want = block[np.tril_indices(len(block))] if a == b else block.ravel()
            have = got[nij[a, b]:nij[a, b] + want.size]
            # at most nocc products of numbers below 1 a sum
            assert np.max(np.abs(have - want)) < 1e-15 * s.nocc
            seen += want.size
    assert seen > 1000
