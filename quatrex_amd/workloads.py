"""Synthetic, seeded inputs of the benchmark configurations.

Distributions (all seeded through ``numpy.random.default_rng(seed)``):

- complex normal CN := (x + i y) / sqrt(2), x, y ~ N(0, 1);
- block-tridiagonal Hamiltonian, N blocks of b: H_ii = (X + X^H)/2 with
  X ~ CN / sqrt(b); H_{i,i+1} ~ CN / sqrt(b), H_{i+1,i} = H_{i,i+1}^H;
- energies E ~ U[-1, 1] plus i * eta (eta = 1e-3);
- boundary self-energies Sigma_B = -i B B^H / b on the first and last
  diagonal block (independent B_L, B_R ~ CN);
- system matrix A = E I - H - Sigma_B;
- Sigma^< block-diagonal, i C_i C_i^H / b per block;
  Sigma^> block-diagonal, -i D_i D_i^H / b per block (independent D_i).

``Workload.assemble`` writes the dense-block DSDBCOO stacks straight into
device memory, one block slice at a time.
"""

from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import torch

from quatrex_amd.datastructures import DSDBCOO, empty_btd


def cn(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / np.sqrt(2.0)


@dataclass
class Workload:
    energies: np.ndarray        # (n_e,) complex
    h_diag: list                # N x (b, b)
    h_upper: list               # N-1 x (b, b)
    sigma_b_left: np.ndarray    # (b, b)
    sigma_b_right: np.ndarray   # (b, b)
    sl_diag: list               # N x (b, b)
    sg_diag: list               # N x (b, b)

    @property
    def block_sizes(self):
        return [d.shape[0] for d in self.h_diag]

    @property
    def n_blocks(self):
        return len(self.h_diag)

    def a_blocks(self, energies=None):
        """Dense numpy blocks of A for the given energies (host; small sizes)."""
        e = self.energies if energies is None else energies
        n = self.n_blocks
        diag = []
        for i, h in enumerate(self.h_diag):
            eye = np.eye(h.shape[0])
            d = e[:, None, None] * eye - h[None]
            if i == 0:
                d = d - self.sigma_b_left
            if i == n - 1:
                d = d - self.sigma_b_right
            diag.append(d)
        upper = [np.broadcast_to(-u, (len(e),) + u.shape).copy() for u in self.h_upper]
        lower = [np.broadcast_to(-u.conj().T, (len(e),) + u.shape[::-1]).copy() for u in self.h_upper]
        return diag, upper, lower

    def assemble(self, device, energy_slice=slice(None)) -> tuple[DSDBCOO, DSDBCOO, DSDBCOO]:
        """(A, Sigma^<, Sigma^>) as dense-block DSDBCOO stacks on ``device``.

        A has the full BTD pattern; the self-energies are block-diagonal.
        """
        e = torch.as_tensor(self.energies[energy_slice], device=device)
        ne = e.shape[0]
        bs = self.block_sizes
        n = len(bs)
        a, aoff = empty_btd(bs, (ne,), offdiag=True, device=device, zero=False)
        sl, loff = empty_btd(bs, (ne,), offdiag=False, device=device, zero=False)
        sg, goff = empty_btd(bs, (ne,), offdiag=False, device=device, zero=False)
        for i in range(n):
            b = bs[i]
            h = torch.as_tensor(self.h_diag[i], device=device)
            if i == 0:
                h = h + torch.as_tensor(self.sigma_b_left, device=device)
            if i == n - 1:
                h = h + torch.as_tensor(self.sigma_b_right, device=device)
            eye = torch.eye(b, dtype=torch.complex128, device=device)
            blk = e[:, None, None] * eye - h[None]
            o = aoff[(i, i)]
            a.data[:, o:o + b * b] = blk.reshape(ne, b * b)
            o = loff[(i, i)]
            sl.data[:, o:o + b * b] = torch.as_tensor(self.sl_diag[i], device=device).reshape(1, -1)
            o = goff[(i, i)]
            sg.data[:, o:o + b * b] = torch.as_tensor(self.sg_diag[i], device=device).reshape(1, -1)
            if i + 1 < n:
                u = torch.as_tensor(self.h_upper[i], device=device)
                o = aoff[(i, i + 1)]
                a.data[:, o:o + u.numel()] = (-u).reshape(1, -1)
                o = aoff[(i + 1, i)]
                a.data[:, o:o + u.numel()] = (-u.conj().T).reshape(1, -1)
        return a, sl, sg


def make_workload(seed: int = 0, n_energies: int = 16, n_blocks: int = 8, block_size: int = 32,
                  eta: float = 1e-3) -> Workload:
    """Seeded instance of the BTD configuration (defaults: 16 E, 8 blocks of 32)."""
    rng = np.random.default_rng(seed)
    b = block_size
    energies = rng.uniform(-1.0, 1.0, n_energies) + 1j * eta
    h_diag, h_upper = [], []
    for i in range(n_blocks):
        x = cn(rng, (b, b)) / np.sqrt(b)
        h_diag.append((x + x.conj().T) / 2)
    for i in range(n_blocks - 1):
        h_upper.append(cn(rng, (b, b)) / np.sqrt(b))
    bl = cn(rng, (b, b))
    br = cn(rng, (b, b))
    sbl = -1j * (bl @ bl.conj().T) / b
    sbr = -1j * (br @ br.conj().T) / b
    sl, sg = [], []
    for i in range(n_blocks):
        c = cn(rng, (b, b))
        sl.append(1j * (c @ c.conj().T) / b)
    for i in range(n_blocks):
        d = cn(rng, (b, b))
        sg.append(-1j * (d @ d.conj().T) / b)
    return Workload(energies, h_diag, h_upper, sbl, sbr, sl, sg)


def lead_blocks(seed: int = 0, n_energies: int = 1024, block_size: int = 256, eta: float = 1e-3,
                onsite_scale: float = 1.0):
    """Semi-infinite lead of one principal layer: (m_ji, m_ii, m_ij) stacks.

    H00 Hermitian (its spread multiplied by ``onsite_scale``),
    H01 ~ CN / sqrt(b), H10 = H01^H; M = (E + i eta) I - H, E ~ U[-1, 1].
    Returned as numpy arrays (n_e, b, b).  At layer 256 about 280 of the 512
    eigenvalues of the lead's quadratic eigenproblem lie in the annulus
    2/3 < |w| < 3/2 at onsite_scale 1, about 30 at onsite_scale 8.
    """
    rng = np.random.default_rng(seed)
    b = block_size
    e = rng.uniform(-1.0, 1.0, n_energies) + 1j * eta
    x = cn(rng, (b, b)) / np.sqrt(b)
    h00 = onsite_scale * (x + x.conj().T) / 2
    h01 = cn(rng, (b, b)) / np.sqrt(b)
    m_ii = e[:, None, None] * np.eye(b) - h00[None]
    m_ij = np.broadcast_to(-h01, (n_energies, b, b)).copy()
    m_ji = np.broadcast_to(-h01.conj().T, (n_energies, b, b)).copy()
    return m_ji, m_ii, m_ij, e


def solve_flops(n_blocks: int, b: int) -> float:
    """Flops of one selected_solve energy (G^R, G^<, G^>) as the reference
    algorithm (rgf.py:115-414) issues them: 4 + 33 (N - 1) block products and
    N block inverses per energy, each 8 b^3 real flops.  With the
    block-diagonal Sigma^<> of these workloads 10 of the 33 products per
    block step multiply a zero block; see ``required_flops``.
    """
    return 8.0 * b ** 3 * ((4 + 33 * (n_blocks - 1)) + n_blocks)


def required_flops(n_blocks: int, b: int) -> float:
    """Flops one selected_solve energy (G^R diagonal, G^<, G^>) requires
    when Sigma^< and Sigma^> are block-diagonal and skew-Hermitian, as in these
    workloads: the reference's products with Sigma_{i,i+1} (rgf.py:270, 283,
    336-346, 358-368) are products with a zero block, and for skew-Hermitian
    x the backward sweep needs three products per quantity instead of four.
    Per block step 10 products and one inverse in the forward sweep
    (a_ji x^R_ii, a_jj - t a_ij, and per lesser / greater quantity a_ji x_ii,
    (.) a_ji^H + Sigma_jj, x^R_jj (.), (.) x^R_jj^H) and 10 products in the
    backward sweep (B1 = x^R_ii a_ij, B2 = x^R_jj a_ji, B1 B2, the G^R_ii
    update, and per quantity B2 x_ii, x_jj B1^H and the product of B1 with
    their sum); block 0 has 4 products and one inverse.  Each product and each
    inverse is 8 b^3 real flops.  (The reduced-precision arithmetics run 22.)
    """
    return 8.0 * b ** 3 * ((4 + 20 * (n_blocks - 1)) + n_blocks)
