"""The batched SCF's two forms at the edges of their ranges: one workgroup for
a molecule up to 64 orbitals, block-Jacobi steps over several above (padded
sizes 128, 192 and 256), and the single-molecule SCF that shares the first."""
import ctypes
import dataclasses

import numpy as np
import pytest

from mopac_gpu_amd import batch as B
from mopac_gpu_amd import geometry, hamiltonian
from mopac_gpu_amd import lib as L
from mopac_gpu_amd.scf import Context
from oracle import oracle

pytestmark = pytest.mark.gpu

# 6 to 254 orbitals, on both sides of and at 32, 64, 128 and 192
MOLS = [("water", 1), ("alkane", 1), ("water", 5), ("alkane", 5), ("water", 6), ("alkane", 10), ("helix", 3),
        ("water", 11), ("alkane", 20), ("alkane", 21), ("water", 22), ("alkane", 31), ("water", 32), ("water", 33),
        ("alkane", 42)]
MAKE = {"water": geometry.water_cluster, "alkane": geometry.alkane, "helix": geometry.glycine_helix}


@pytest.fixture(scope="module")
def systems():
    return [hamiltonian.build(*MAKE[kind](size, 17)) for kind, size in MOLS]


@pytest.fixture(scope="module")
def edge_batch(systems):
    b = B.Batch(systems, scfcrt=1e-6)
    yield b
    b.close()


def test_every_size_matches_the_oracle(systems, edge_batch):
    edge_batch.run()
    escf, niter, conv = edge_batch.results()
    assert conv.all()
    for m, s in enumerate(systems):
        o = oracle.iterate(s, scfcrt=1e-6)
        assert int(niter[m]) == o["niter"], (MOLS[m], niter[m], o["niter"])
        assert abs(escf[m] - o["escf"]) < 1e-6 * max(1.0, abs(o["escf"])), MOLS[m]
        assert np.max(np.abs(edge_batch.density(m) - o["p"])) < 1e-6, MOLS[m]


def test_iteration_limit_stops_both_forms(systems, edge_batch):
    """Three iterations are the same three in either eigensolver form, and a
    second run starts over."""
    edge_batch.run(iters_per_graph=3, max_launches=1)
    e1, n1, c1 = edge_batch.results()
    edge_batch.set_eig_lds(False)
    edge_batch.run(iters_per_graph=1, max_launches=3)
    e2, n2, c2 = edge_batch.results()
    edge_batch.set_eig_lds(True)
    assert not c1.any() and not c2.any()
    assert (n1 == n2).all() and (n1 <= 3).all()
    assert np.max(np.abs(e1 - e2) / np.maximum(1.0, np.abs(e1))) < 1e-9
    edge_batch.run()
    assert edge_batch.results()[2].all()


@pytest.mark.parametrize("m", range(7))
def test_single_molecule_in_one_workgroup_matches_the_general_path(systems, m):
    s = systems[m]
    assert s.norbs <= 64
    kw = dict(scfcrt=1e-6, want=("p", "f", "c", "eig"))
    out = []
    for inner in (0, 16):  # a chosen inner sweep count takes the general path
        ctx = Context(0)
        ctx.lib.mhip_set_tuning(ctx.h, -1, inner, -1.0)
        ctx.upload(s)
        out.append((ctx.iter(**kw), ctx.iter(itrmax=4, **kw)))
        ctx.close()
    (a, few), (b, few_b) = out
    assert a["converged"] and b["converged"] and a["niter"] == b["niter"]
    assert few["niter"] == few_b["niter"] and few["converged"] == few_b["converged"]
    assert abs(a["escf"] - b["escf"]) < 1e-7 * max(1.0, abs(b["escf"]))
    # the in-loop eigensolves stop at residuals of 1e-10, which the densities'
    # differences carry over gaps of tenths of eV and the iterations left
    for k in ("p", "f", "eig"):
        assert np.max(np.abs(a[k] - b[k])) < 1e-7, k
    # the eigenvectors of the exit diagonalization: orthonormal, and F's own
    n = s.norbs
    f = np.zeros((n, n))
    f[np.tril_indices(n)] = a["f"]
    f = f + np.tril(f, -1).T
    assert np.max(np.abs(a["c"].T @ a["c"] - np.eye(n))) < 1e-11
    assert np.max(np.abs(f @ a["c"] - a["c"] * a["eig"])) < 1e-8  # F(i,i) + i*1e-10 is what is diagonalized


def test_eigensolves_out_of_sweeps_do_not_count(systems, edge_batch):
    """Two sweeps do not converge the first diagonalization; the SCF may still
    settle, on levels that are not F's."""
    b = edge_batch
    for lds in (True, False):
        b.set_eig_lds(lds)
        b.lib.mhip_batch_set_eig_sweeps(b.h, 2)
        _, n = b.run()
        assert n == 0 and not b.results()[2].any()
        b.lib.mhip_batch_set_eig_sweeps(b.h, 60)
        _, n = b.run()
        assert n == len(systems) and b.results()[2].all()
    b.set_eig_lds(True)


def test_device_memory_of_the_default_form(systems):
    """Four padded matrices, the rotations and diagonal blocks of two steps and
    the caller's arrays for a molecule above 64 orbitals; the matrices of the
    global-memory form are there once it is chosen."""
    s = systems[13]
    n, npad, count = s.norbs, 256, 256
    assert 192 < n <= npad
    B.Batch([s], scfcrt=1e-6).close()  # the module's code is loaded

    def free():  # the HIP library that this one is linked with
        now, all_of_it = ctypes.c_size_t(), ctypes.c_size_t()
        assert L.load().hipMemGetInfo(ctypes.byref(now), ctypes.byref(all_of_it)) == 0
        return now.value

    before = free()
    b = B.Batch([s] * count, scfcrt=1e-6)
    each = (before - free()) / 8 / count
    caller = len(s.w) + 5 * s.mpack
    # the Fock build's column partials: an atom's 1 or 10 elements by every later atom
    limit = np.where(np.asarray(s.nlast) > np.asarray(s.nfirst), 10, 1)
    columns = int(np.sum(limit * (s.numat - 1 - np.arange(s.numat))))
    # rows, levels and atoms' tables are under 100 numbers an orbital
    assert each < caller + columns + 4 * npad * npad + 192 * npad + 100 * n
    b.set_eig_lds(False)
    assert (before - free()) / 8 / count > each + 2.9 * n * n
    b.close()


def test_split_precision_of_a_small_molecule(gpu_ctx, systems):
    """precision = 1 is the split-BF16 form at any size."""
    gpu_ctx.upload(systems[2])
    plain = gpu_ctx.iter(scfcrt=1e-6)
    split = gpu_ctx.iter(scfcrt=1e-6, precision=1)
    assert split["n_split_iter"] > 0 and plain["n_split_iter"] == 0
    assert abs(split["escf"] - plain["escf"]) < 1e-6


@pytest.mark.parametrize("scale", (1.0, 1e6, 1e20, 1e40))
@pytest.mark.parametrize("mol", [("water", 5), ("water", 11), ("water", 22), ("water", 32), ("water", 33)])
def test_levels_of_any_size(mol, scale):
    """One iteration on an H whose levels are evenly spread over -scale to
    scale: the density is that of H's own lower levels."""
    s = hamiltonian.build(*MAKE[mol[0]](mol[1], 17))
    n = s.norbs
    rng = np.random.default_rng(n)
    v = np.linalg.qr(rng.standard_normal((n, n)))[0]
    h = (v * (scale * np.linspace(-1.0, 1.0, n))) @ v.T
    # no integrals: F is H, and a level shift of the starting diagonal
    s = dataclasses.replace(s, h=h[np.tril_indices(n)], w=np.zeros_like(s.w), pdiag=np.full(n, 2.0 * s.nclose / n))
    b = B.Batch([s], scfcrt=1e-6)
    b.run(iters_per_graph=1, max_launches=1)
    p = b.density(0)
    b.close()
    want = 2.0 * v[:, :s.nclose] @ v[:, :s.nclose].T
    # residuals of 1e-10 of the largest level over the gap of 2 / (n - 1), on up
    # to n elements
    assert np.max(np.abs(p - want[np.tril_indices(n)])) < 1e-10 * n * n
