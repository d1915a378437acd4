"""Observables and system-matrix assembly on the HIP path against the oracle."""

import numpy as np
import pytest
import scipy.sparse as sps
import torch

import oracle.rgf as orgf
from oracle.observables import assemble_system_matrix as o_assemble
from oracle.observables import contact_currents as o_currents
from oracle.observables import density as o_density
from quatrex_amd.datastructures import DSDBCOO
from quatrex_amd.greens_function_solver import RGF, OBCBlocks
from quatrex_amd.observables import SystemMatrixAssembler, contact_currents, density
from tests.conftest import rel_err
from tests.test_gpu_rgf import _oracle_containers, to_gpu
from tests.test_oracle_observables import _btd_mask, _cn, _container
from quatrex_amd.workloads import make_workload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solved():
    w = make_workload(seed=4)
    oa, osl, osg = _oracle_containers(w)
    ref = orgf.RGF(16).selected_solve(oa, osl, osg)
    return w, (oa, osl, osg), ref


@pytest.mark.parametrize("max_batch_size", [16, 5])
def test_fused_density_output(device, solved, max_batch_size):
    w, (oa, osl, osg), (rl, rg) = solved
    n_orb = int(np.sum(w.block_sizes))
    dens = torch.zeros((oa.data.shape[0], n_orb), dtype=torch.float64, device=device)
    xl, xg = RGF(max_batch_size).selected_solve(to_gpu(oa, device), to_gpu(osl, device),
                                                to_gpu(osg, device), density=dens)
    ref = o_density(rl)
    assert rel_err(dens.cpu().numpy(), ref) < 1e-10
    assert rel_err(density(xl).cpu().numpy(), ref) < 1e-10


def test_density_with_overlap(device):
    rng = np.random.default_rng(0)
    bs = [3, 4, 2]
    n = sum(bs)
    g = _cn(rng, (5, n, n))
    x = _container(g, bs)
    s = _cn(rng, (n, n))
    s = np.where(_btd_mask(bs), s + s.conj().T, 0)
    gx = DSDBCOO(torch.as_tensor(x.data, device=device), x.rows, x.cols, x.block_sizes,
                 x.global_stack_shape)
    got = density(gx, sps.csr_matrix(s)).cpu().numpy()
    assert rel_err(got, o_density(x, sps.csr_matrix(s))) < 1e-13


def test_contact_currents(device, solved):
    w, (oa, osl, osg), _ = solved
    ne, b0, bn, nb = oa.data.shape[0], w.block_sizes[0], w.block_sizes[-1], w.n_blocks
    rng = np.random.default_rng(3)
    obc = orgf.OBCBlocks(nb)
    obc.lesser[0] = 0.1j * _cn(rng, (ne, b0, b0))
    obc.greater[0] = -0.1j * _cn(rng, (ne, b0, b0))
    obc.lesser[-1] = 0.2j * _cn(rng, (ne, bn, bn))
    obc.greater[-1] = -0.2j * _cn(rng, (ne, bn, bn))
    xl, xg = orgf.RGF(16).selected_solve(oa, osl, osg, obc_blocks=obc)
    ref = o_currents(xl, xg, obc)
    gobc = OBCBlocks(nb)
    for name in ("lesser", "greater"):
        for j in (0, -1):
            getattr(gobc, name)[j] = torch.as_tensor(getattr(obc, name)[j], device=device)
    gl, gg = to_gpu(xl, device), to_gpu(xg, device)
    got = contact_currents(gl, gg, gobc)
    for r, g in zip(ref, got):
        assert rel_err(g.cpu().numpy(), r) < 1e-12


@pytest.mark.parametrize("with_overlap", [False, True])
def test_system_matrix_assembly(device, with_overlap):
    rng = np.random.default_rng(5)
    bs = [3, 3, 2, 4]
    n, ne = sum(bs), 6
    h = _cn(rng, (n, n))
    h = np.where(_btd_mask(bs), h + h.conj().T, 0)
    sse = np.where(_btd_mask(bs), _cn(rng, (ne, n, n)), 0)
    v = rng.standard_normal(n)
    e = rng.uniform(-1, 1, ne)
    s = np.where(_btd_mask(bs), np.eye(n) + 0.1 * _cn(rng, (n, n)), 0) if with_overlap else None
    a = _container(np.zeros((ne, n, n), complex), bs)
    hc = _container(np.broadcast_to(h, (ne, n, n)).copy(), bs)
    sc = _container(sse, bs)
    ov = sps.csr_matrix(s) if with_overlap else None
    o_assemble(a, e, 1e-3, hc, sc, overlap=ov, potential=v)
    pattern = DSDBCOO(torch.zeros((ne, a.data.shape[-1]), dtype=torch.complex128, device=device),
                      a.rows, a.cols, a.block_sizes, a.global_stack_shape)
    gs = DSDBCOO(torch.as_tensor(sc.data, device=device), sc.rows, sc.cols, sc.block_sizes,
                 sc.global_stack_shape)
    asm = SystemMatrixAssembler(pattern, sps.csr_matrix(h), overlap=ov, potential=v)
    got = asm(e, 1e-3, gs)
    assert rel_err(got.data.cpu().numpy(), a.data) < 1e-14


@pytest.mark.parametrize("batch", [1, 7, 8, 9, 17])
@pytest.mark.parametrize("nnz", [1, 255, 257])
@pytest.mark.parametrize("terms", ["zst", "st", "z", "t"])
def test_assembly_kernel_edges(device, batch, nnz, terms):
    """A = z S + T - Sigma for stacks and patterns around the kernel's groups of
    eight energies and 256 entries, with each of the terms absent; entries
    outside the stack are left alone."""
    from quatrex_amd import _lib

    rng = np.random.default_rng(batch * 1000 + nnz)
    cn = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    z, s, t, sig = cn(batch), cn(nnz), cn(nnz), cn(batch, nnz)
    want = np.zeros((batch, nnz), complex)
    args = {"z": None, "s": None, "t": None, "sig": None}
    if "z" in terms:
        want += z[:, None] * s
        args["z"], args["s"] = z, s
    if "t" in terms:
        want += t
        args["t"] = t
    if "s" in terms:
        want -= sig
        args["sig"] = sig
    dev = {k: None if v is None else torch.as_tensor(v, device=device) for k, v in args.items()}
    out = torch.full((batch + 1, nnz), 7.0, dtype=torch.complex128, device=device)
    ptr = {k: None if v is None else v.data_ptr() for k, v in dev.items()}
    h = _lib.handle(device)
    rc = _lib.load().qx_assemble_system_matrix(h, _lib.stream_ptr(device), batch, nnz, ptr["z"],
                                               ptr["s"], ptr["t"], ptr["sig"], nnz,
                                               out.data_ptr(), nnz)
    _lib.check(rc, h, "assemble")
    got = out.cpu().numpy()
    assert np.allclose(got[:batch], want, rtol=1e-15, atol=4e-15)
    assert np.all(got[batch] == 7.0)


@pytest.mark.parametrize("with_sigma", [True, False])
@pytest.mark.parametrize("batch,nnz", [(3, 29), (1001, 30), (4097, 7), (5, 300), (65537, 1), (9, 2047),
                                       (9, 2048), (9, 2305)])
def test_assembly_small_patterns(device, batch, nnz, with_sigma):
    """Patterns shorter than a workgroup (its threads cover several groups of
    energies) and around the line of the flat grid, with strides above nnz and in place over Sigma; entries outside
    are left alone.  Two roundings a term: 4 eps of the terms' sizes."""
    from quatrex_amd import _lib

    g = torch.Generator(device=device).manual_seed(batch + nnz)
    cn = lambda *s: torch.randn(*s, dtype=torch.complex128, generator=g, device=device)  # noqa: E731
    z, s, t, sig = cn(batch), cn(nnz), cn(nnz), cn(batch, nnz + 2)
    want = z[:, None] * s + t
    out = sig.clone()
    size = (z[:, None] * s).abs() + t.abs()
    if with_sigma:
        want, size = want - sig[:, :nnz], size + sig[:, :nnz].abs()
    h = _lib.handle(device)
    rc = _lib.load().qx_assemble_system_matrix(
        h, _lib.stream_ptr(device), batch, nnz, z.data_ptr(), s.data_ptr(), t.data_ptr(),
        out.data_ptr() if with_sigma else None, nnz + 2, out.data_ptr(), nnz + 2)
    _lib.check(rc, h, "assemble")
    assert bool(((out[:, :nnz] - want).abs() <= 4 * np.finfo(float).eps * size).all())
    assert torch.equal(torch.view_as_real(out[:, nnz:]), torch.view_as_real(sig[:, nnz:]))


@pytest.mark.parametrize("with_sigma", [True, False])
@pytest.mark.parametrize("shape", ["energies", "rows", "entries"])
def test_assembly_of_more_than_one_launch(device, shape, with_sigma):
    """A launch takes 2^28 threads and a grid 65535 rows: stacks and patterns beyond one, the second
    launch's first and last elements among those looked at."""
    from quatrex_amd import _lib

    line = 1 << 28
    if shape == "energies":
        batch, nnz = (4 if with_sigma else 8) * line + 9, 1
    elif shape == "rows":  # of a grid, 65535 at most
        batch, nnz = (4 if with_sigma else 8) * 65535 + 9, 2048
    else:
        batch, nnz = 2, line + 9
    n = batch * nnz
    z = torch.arange(batch, dtype=torch.float64, device=device) + 0j
    s = torch.ones(nnz, dtype=torch.complex128, device=device)
    t = torch.arange(nnz, dtype=torch.float64, device=device) * 1j
    out = torch.full((n,), 0.5, dtype=torch.complex128, device=device)
    h = _lib.handle(device)
    rc = _lib.load().qx_assemble_system_matrix(
        h, _lib.stream_ptr(device), batch, nnz, z.data_ptr(), s.data_ptr(), t.data_ptr(),
        out.data_ptr() if with_sigma else None, nnz, out.data_ptr(), nnz)
    _lib.check(rc, h, "assemble")
    less = 0.5 if with_sigma else 0.0
    for lo in range(0, n, line):
        i = torch.arange(lo, min(lo + line, n), device=device)
        want = torch.complex((i // nnz).double() - less, (i % nnz).double())
        assert torch.equal(torch.view_as_real(out[lo:lo + line]), torch.view_as_real(want))
