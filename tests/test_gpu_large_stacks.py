"""Stacks of very many small matrices: more workgroups times threads than one
launch takes (2^32 threads).  Energies repeat in a short cycle, so every
result has to be that of the same call on one cycle."""

import numpy as np
import pytest
import torch

from quatrex_amd import _lib
from quatrex_amd.boundary_conditions import SanchoRubio
from quatrex_amd.datastructures import DSDBCOO, btd_pattern, empty_btd
from quatrex_amd.greens_function_solver import RGF
from quatrex_amd.ops import inv

pytestmark = pytest.mark.gpu

CYCLE = 7


def _tiled(block, n):
    return block.repeat((n + len(block) - 1) // len(block), 1)[:n].contiguous()


def _chain(device, n_blocks, n_e):
    """A and Sigma^<, Sigma^> of a chain of single orbitals, the energies in a
    cycle of CYCLE."""
    sizes = [1] * n_blocks
    rng = np.random.default_rng(n_blocks)
    containers = []
    for skew in (False, True, True):
        rows, cols, _ = btd_pattern(sizes, offdiag=not skew)
        x = rng.standard_normal((CYCLE, len(rows))) + 1j * rng.standard_normal((CYCLE, len(rows)))
        x = 1j * x.imag if skew else 0.4 * x + 4.0 * (rows == cols)
        containers.append(DSDBCOO(_tiled(torch.as_tensor(x, device=device), n_e), rows, cols,
                                  sizes, (n_e,)))
    return sizes, containers


def _equal_cycles(x, ref):
    """x (n, ...) repeats ref (CYCLE, ...), bitwise."""
    n = len(x) // CYCLE * CYCLE
    whole = x[:n].reshape(-1, CYCLE, *x.shape[1:])
    return bool((whole == ref).all()) and bool((x[n:] == ref[:len(x) - n]).all())


@pytest.mark.parametrize("last_skew", [True, False])
def test_skew_check_of_many_energies(device, monkeypatch, last_skew):
    """33 blocks take one launch per product; the skew-Hermitian check of 262151
    energies, 64 blocks at a time, is of more threads than one launch takes, and
    finds an energy at the very end that is not skew-Hermitian."""
    n_e = (1 << 18) + CYCLE
    sizes, (a, sl, sg) = _chain(device, 33, n_e)
    if not last_skew:
        sg.data[n_e - 1, 5] += 0.25
    h = _lib.new_handle(device)
    _lib.set_tuning(h, streams=1)
    outs = {}
    with _lib.use_handle(h):
        for check in (_lib.SOLVE_SKEW_CHECK, 0):
            monkeypatch.setattr(_lib, "SOLVE_SKEW_CHECK", check)
            outs[check] = [empty_btd(sizes, (n_e,), device=device)[0] for _ in range(2)]
            RGF(n_e).selected_solve(a, sl, sg, out=tuple(outs[check]))
    _lib.load().qx_destroy(h)
    x, y = ([m.data for m in outs[check]] for check in (32, 0))
    equal = all(torch.equal(torch.view_as_real(p), torch.view_as_real(q)) for p, q in zip(x, y))
    assert equal == (not last_skew)  # the general sweep exactly when one is not skew
    for p, q in zip(x, y):
        assert float((p - q).abs().max()) <= 1e-12 * float(q.abs().max())


def test_fused_inverse_of_many_energies(device):
    """The fused kernel runs 512 threads an energy: 2^23 of them fill a launch."""
    n_e = (1 << 23) + 5
    sizes, (a, _, _) = _chain(device, 17, n_e)
    x = empty_btd(sizes, (n_e,), device=device, zero=False)[0]
    RGF(n_e).selected_inv(a, out=x)
    _, (a, _, _) = _chain(device, 17, CYCLE)
    ref = empty_btd(sizes, (CYCLE,), device=device)[0]
    RGF(CYCLE).selected_inv(a, out=ref)
    assert _equal_cycles(x.data, ref.data)


def test_sancho_rubio_of_many_leads(device):
    """The norms of the stop rule take a workgroup of 1024 threads a lead: 2^22
    of them fill a launch.  The last lead converges last."""
    n_e = (1 << 22) + 3
    e = torch.linspace(2.0, 2.5, CYCLE, dtype=torch.float64, device=device) + 0.2j
    slow = torch.tensor([0.1 + 1e-3j], device=device, dtype=torch.complex128)

    def solve(n):
        a_ii = torch.cat([_tiled(e.reshape(CYCLE, 1), n - 1), slow.reshape(1, 1)])
        a_ij, a_ji = torch.full_like(a_ii, -0.3 + 0.1j), torch.full_like(a_ii, -0.3 - 0.1j)
        s = SanchoRubio(max_iterations=100, convergence_tol=1e-10)
        return s(*(x.reshape(n, 1, 1) for x in (a_ii, a_ij, a_ji))), s.iterations

    ref, iterations = solve(CYCLE + 1)
    got, n = solve(n_e)
    assert n == iterations
    assert _equal_cycles(got[:-1], ref[:-1])
    assert torch.equal(torch.view_as_real(got[-1]), torch.view_as_real(ref[-1]))


def test_inverse_of_many_matrices(device):
    """Workgroups of 128 threads: 33554431 matrices fill a launch."""
    x = torch.arange(1, 33554431 + 4, dtype=torch.float64, device=device)
    got = inv((x + 0j).reshape(-1, 1, 1)).reshape(-1)
    assert float((got * x - 1).abs().max()) < 1e-15 * 4
