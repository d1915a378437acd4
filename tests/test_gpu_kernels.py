"""HIP kernels through the C ABI: batched complex GEMM and batched inverse.

Checked against NumPy float64/complex128 on the CPU (the plain fp64
reference of the same op).  Tolerances: complex128 arithmetic 1e-12
relative Frobenius per matrix; complex64 arithmetic 2e-5.
"""

import ctypes

import numpy as np
import pytest
import torch

from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


def _lib():
    from quatrex_amd import _lib

    return _lib


def _cplx(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _zgemm(dev, A, B, C, opa, opb, alpha, beta, prec, lda=None, ldb=None, ldc=None):
    L = _lib()
    lib = L.load()
    h, st = L.handle(dev), L.stream_ptr(dev)
    batch = C.shape[0]
    m, n = C.shape[1], C.shape[2]
    k = A.shape[2] if opa == L.OP_N else A.shape[1]
    al = (ctypes.c_double * 2)(alpha.real, alpha.imag)
    be = (ctypes.c_double * 2)(beta.real, beta.imag)
    rc = lib.qx_zgemm_batched(h, st, batch, m, n, k, opa, opb, al, A.data_ptr(), A.stride(1),
                              A.stride(0), B.data_ptr(), B.stride(1), B.stride(0), be,
                              C.data_ptr(), C.stride(1), C.stride(0), prec)
    L.check(rc, h, "zgemm")
    L.sync_check(dev, "zgemm")


SHAPES = [(1, 1, 1), (5, 7, 3), (16, 16, 16), (64, 64, 64), (100, 37, 129), (130, 66, 70),
          (256, 256, 256)]


@pytest.mark.parametrize("mnk", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("ops", [(0, 0), (0, 2), (2, 0), (2, 2)], ids=["NN", "NC", "CN", "CC"])
@pytest.mark.parametrize("prec", [0, 1, 3], ids=["c128", "c64", "c128_3m"])
def test_zgemm(device, mnk, ops, prec):
    m, n, k = mnk
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    batch = 3
    opa, opb = ops
    a_shape = (batch, m, k) if opa == 0 else (batch, k, m)
    b_shape = (batch, k, n) if opb == 0 else (batch, n, k)
    a, b, c = _cplx(rng, a_shape), _cplx(rng, b_shape), _cplx(rng, (batch, m, n))
    alpha, beta = 0.7 - 0.3j, (0.0 if (m + n) % 2 else -1.2 + 0.5j)
    # padded leading dimensions: operate on a column slice of a wider buffer
    A = torch.zeros(a_shape[:2] + (a_shape[2] + 3,), dtype=torch.complex128, device=device)
    A[..., :a_shape[2]] = torch.as_tensor(a, device=device)
    B = torch.as_tensor(b, device=device)
    C = torch.as_tensor(c, device=device)
    if beta == 0.0:
        C[:] = float("nan")  # beta == 0 must not read C
    _zgemm(device, A[..., :a_shape[2]], B, C, opa, opb, alpha, beta, prec)
    opA = a if opa == 0 else np.conj(np.swapaxes(a, 1, 2))
    opB = b if opb == 0 else np.conj(np.swapaxes(b, 1, 2))
    ref = alpha * opA @ opB + (beta * c if beta != 0.0 else 0)
    tol = {0: 1e-12, 1: 2e-5, 3: 1e-12}[prec]
    got = C.cpu().numpy()
    for e in range(batch):
        assert rel_err(got[e], ref[e]) < tol
    # the padding columns of A are untouched
    assert torch.all(A[..., a_shape[2]:] == 0)


BIG = [(256, 256, 256, 64), (200, 136, 72, 130), (384, 130, 33, 100)]


@pytest.mark.parametrize("mnkb", BIG, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("ops", [(0, 0), (0, 2), (2, 0), (2, 2)], ids=["NN", "NC", "CN", "CC"])
@pytest.mark.parametrize("prec", [0, 1, 3], ids=["c128", "c64", "c128_3m"])
def test_zgemm_large_stack(device, mnkb, ops, prec):
    """Stacks with >= 256 tiles of 128 x 128 (the large-tile kernel shape)."""
    m, n, k, batch = mnkb
    rng = np.random.default_rng(m + n + k + batch)
    opa, opb = ops
    a_shape = (batch, m, k) if opa == 0 else (batch, k, m)
    b_shape = (batch, k, n) if opb == 0 else (batch, n, k)
    a, b, c = _cplx(rng, a_shape), _cplx(rng, b_shape), _cplx(rng, (batch, m, n))
    alpha, beta = 1.1 + 0.2j, -0.5 + 0.25j
    A, B = torch.as_tensor(a, device=device), torch.as_tensor(b, device=device)
    C = torch.as_tensor(c, device=device)
    _zgemm(device, A, B, C, opa, opb, alpha, beta, prec)
    got = C.cpu().numpy()
    tol = {0: 1e-12, 1: 2e-5, 3: 1e-12}[prec]
    for e in (0, batch // 2, batch - 1):
        opA = a[e] if opa == 0 else np.conj(a[e].T)
        opB = b[e] if opb == 0 else np.conj(b[e].T)
        assert rel_err(got[e], alpha * opA @ opB + beta * c[e]) < tol


REG_CASES = [(256, 256, 256, 8), (128, 128, 64, 4), (200, 136, 72, 3), (5, 7, 3, 2),
             (416, 416, 416, 2)]


@pytest.mark.parametrize("mnkb", REG_CASES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("ops", [(0, 0), (0, 2), (2, 0), (2, 2)], ids=["NN", "NC", "CN", "CC"])
@pytest.mark.parametrize("prec", [0, 3, 1], ids=["c128", "c128_3m", "c64"])
def test_zgemm_register_kernels_match_lds(device, monkeypatch, mnkb, ops, prec):
    """Every register-direct GEMM shape gives the bits of the LDS-staged
    kernel: both sum k in the same order with the same 4M / 3M split (full
    tiles, ragged tiles and k not a multiple of 4).  complex64 arithmetic
    (3M, register-direct on request: QX_ZGEMM_F32=reg): both round the
    operands to float and form the 3M sums in float."""
    monkeypatch.setenv("QX_ZGEMM_F32", "reg")
    L = _lib()
    m, n, k, batch = mnkb
    rng = np.random.default_rng(m + 2 * n + 3 * k)
    opa, opb = ops
    a_shape = (batch, m, k) if opa == 0 else (batch, k, m)
    b_shape = (batch, k, n) if opb == 0 else (batch, n, k)
    A = torch.as_tensor(_cplx(rng, a_shape), device=device)
    B = torch.as_tensor(_cplx(rng, b_shape), device=device)
    C0 = torch.as_tensor(_cplx(rng, (batch, m, n)), device=device)
    alpha, beta = 0.9 + 0.4j, 0.3 - 0.7j
    h = L.handle(device)
    outs = {}
    try:
        for code in (L.GEMM_LDS_64, L.GEMM_REG_64x64, L.GEMM_REG_64x128, L.GEMM_REG_128x64):
            L.set_tuning(h, 4, code)
            C = C0.clone()
            _zgemm(device, A, B, C, opa, opb, alpha, beta, prec)
            outs[code] = C
    finally:
        L.set_tuning(h, 4, L.GEMM_AUTO)
    for code in (L.GEMM_REG_64x64, L.GEMM_REG_64x128, L.GEMM_REG_128x64):
        assert torch.equal(outs[code], outs[L.GEMM_LDS_64]), code


def _inv(dev, A, X, prec, S=None):
    L = _lib()
    lib = L.load()
    h, st = L.handle(dev), L.stream_ptr(dev)
    n = A.shape[-1]
    sp = S.data_ptr() if S is not None else None
    rc = lib.qx_inv_batched(h, st, A.shape[0], n, A.data_ptr(), A.stride(1), A.stride(0), sp,
                            n, n * n, X.data_ptr(), X.stride(1), X.stride(0), prec)
    L.check(rc, h, "inv")
    L.sync_check(dev, "inv")


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 64, 100, 256, 416, 512])
@pytest.mark.parametrize("prec", [0, 1], ids=["c128", "c64"])
def test_inverse(device, n, prec):
    rng = np.random.default_rng(n)
    batch = 4
    a = _cplx(rng, (batch, n, n))
    if n > 1:
        a[:, 0, 0] = 0.0  # forces a row interchange at the first pivot
    s = 0.1 * _cplx(rng, (batch, n, n))
    A = torch.as_tensor(a, device=device)
    S = torch.as_tensor(s, device=device)
    X = torch.empty_like(A)
    _inv(device, A, X, prec, S)
    ref = np.linalg.inv(a - s)
    got = X.cpu().numpy()
    cond = max(np.linalg.cond(a[e] - s[e]) for e in range(batch))
    tol = (1e-15 if prec == 0 else 1e-7) * cond * max(n, 4)
    for e in range(batch):
        assert rel_err(got[e], ref[e]) < tol, (e, rel_err(got[e], ref[e]), tol)


@pytest.mark.parametrize("n", [1, 3, 20, 32])
@pytest.mark.parametrize("batch", [1, 5, 9])
def test_small_inverse_matches_split_kernels(device, monkeypatch, n, batch):
    """n <= 32 (complex128): one launch, one matrix per wave or per
    workgroup; same pivot rule as the panel kernels, so the same permutation
    and results to rounding (batch not a multiple of the four matrices per
    workgroup of the per-wave kernel)."""
    rng = np.random.default_rng(10 * n + batch)
    a = _cplx(rng, (batch, n, n))
    s = 0.1 * _cplx(rng, (batch, n, n))
    A, S = torch.as_tensor(a, device=device), torch.as_tensor(s, device=device)
    outs = []
    for small in ("1", "2", "0"):  # per wave, per workgroup, split panel kernels
        monkeypatch.setenv("QX_INV_SMALL", small)
        X = torch.empty_like(A)
        _inv(device, A, X, 0, S)
        outs.append(X.cpu().numpy())
    cond = max(np.linalg.cond(a[e] - s[e]) for e in range(batch))
    for e in range(batch):
        for o in outs[:2]:
            assert rel_err(o[e], outs[2][e]) < 1e-15 * cond * max(n, 4)
            assert rel_err(o[e], np.linalg.inv(a[e] - s[e])) < 1e-15 * cond * max(n, 4)


@pytest.mark.parametrize("n", [12, 32, 100, 300])
@pytest.mark.parametrize("scale", [2.0 ** -1000, 1e-150, 1e150, 2.0 ** 1000])
def test_inverse_extreme_scales(device, n, scale):
    """Pivot reciprocals are formed from parts scaled by a power of two:
    matrices whose entries are near the ends of the double range invert as
    accurately as unit-scale ones (inv(s A) = inv(A) / s), on the per-workgroup
    small path (n <= 32) and both panel kernels (n <= 256, n > 256)."""
    rng = np.random.default_rng(n)
    a = _cplx(rng, (2, n, n))
    a[:, 0, 0] = 0.0
    A = torch.as_tensor(a * scale, device=device)
    X = torch.empty_like(A)
    _inv(device, A, X, 0)
    got = X.cpu().numpy() * scale
    for e in range(2):
        ref = np.linalg.inv(a[e])
        assert np.isfinite(got[e]).all()
        assert rel_err(got[e], ref) < 1e-15 * np.linalg.cond(a[e]) * n, (e, rel_err(got[e], ref))


@pytest.mark.parametrize("n", [33, 64, 100, 256, 300, 416, 512])
@pytest.mark.parametrize("prec", [0, 1], ids=["c128", "c64"])
def test_panel_kernels_agree(device, monkeypatch, n, prec):
    """The column-group panel kernel (default; 4 or 8 columns per wave)
    against the four-threads-per-row kernel (n <= 256) and the
    one-thread-per-row kernel (all n): the same Gauss-Jordan elimination with
    partial pivoting, so equal to rounding (near-ties between pivot
    candidates may be broken differently)."""
    rng = np.random.default_rng(3 * n + prec)
    batch = 3
    a = _cplx(rng, (batch, n, n))
    a[:, 0, 0] = 0.0
    A = torch.as_tensor(a, device=device)
    variants = [("0", "4"), ("0", "8"), ("1", "8")] + ([("4", "8")] if n <= 256 else [])
    outs = {}
    for kind, cw in variants:
        monkeypatch.setenv("QX_INV_PANEL", kind)
        monkeypatch.setenv("QX_INV_CW", cw)
        X = torch.empty_like(A)
        _inv(device, A, X, prec)
        outs[(kind, cw)] = X.cpu().numpy()
    cond = max(np.linalg.cond(a[e]) for e in range(batch))
    tol = (1e-15 if prec == 0 else 1e-7) * cond * n
    for e in range(batch):
        ref = np.linalg.inv(a[e])
        for v, o in outs.items():
            assert rel_err(o[e], ref) < tol, (v, e, rel_err(o[e], ref))
            assert rel_err(o[e], outs[("1", "8")][e]) < tol, (v, e)


@pytest.mark.parametrize("n", [33, 64, 65, 100, 128, 200, 256])
@pytest.mark.parametrize("prec", [0, 1], ids=["c128", "c64"])
@pytest.mark.parametrize("in_place", [False, True])
def test_panel_width_64(device, monkeypatch, n, prec, in_place):
    """64-column panels (eight waves of eight columns) with rank-64 updates in
    two k-chunks, against the 32-column panels and NumPy: the same
    elimination blocked differently, so equal to rounding; in place and with
    a separate output (the panel count's parity picks the start buffer)."""
    rng = np.random.default_rng(7 * n + prec)
    batch = 3
    a = _cplx(rng, (batch, n, n))
    a[:, 0, 0] = 0.0  # a row interchange at the first pivot
    a[:, n - 1, n - 1] = 0.0
    outs = {}
    for nb in ("64", "32"):
        monkeypatch.setenv("QX_INV_NB", nb)
        A = torch.as_tensor(a, device=device)
        X = A if in_place else torch.empty_like(A)
        _inv(device, A, X, prec)
        outs[nb] = X.cpu().numpy()
    cond = max(np.linalg.cond(a[e]) for e in range(batch))
    tol = (1e-15 if prec == 0 else 1e-7) * cond * n
    for e in range(batch):
        ref = np.linalg.inv(a[e])
        assert rel_err(outs["64"][e], ref) < tol, (e, rel_err(outs["64"][e], ref), tol)
        assert rel_err(outs["64"][e], outs["32"][e]) < tol


@pytest.mark.parametrize("n", [40, 100, 256])
@pytest.mark.parametrize("prec", [0, 1], ids=["c128", "c64"])
def test_update_chunk_depth_bitwise(device, monkeypatch, n, prec):
    """The trailing update staged in 16-deep k-chunks (four workgroups per
    CU, the default from 256 matrices per call) or 32-deep ones (two): the
    same products summed in the same k order, so the same bits."""
    rng = np.random.default_rng(11 * n + prec)
    a = _cplx(rng, (5, n, n))
    a[:, 0, 0] = 0.0
    outs = {}
    for depth in ("16", "32"):
        monkeypatch.setenv("QX_INV_UPDATE", depth)
        A = torch.as_tensor(a, device=device)
        X = torch.empty_like(A)
        _inv(device, A, X, prec)
        outs[depth] = X.cpu().numpy()
    assert np.array_equal(outs["16"].view(np.uint64), outs["32"].view(np.uint64))
    cond = max(np.linalg.cond(a[e]) for e in range(5))
    tol = (1e-15 if prec == 0 else 1e-7) * cond * n
    for e in range(5):
        assert rel_err(outs["16"][e], np.linalg.inv(a[e])) < tol


@pytest.mark.parametrize("n,batch", [(40, 5), (64, 3), (100, 5), (256, 6), (256, 300),
                                     (300, 4), (512, 2), (130, 260)])
@pytest.mark.parametrize("prec", [0, 1], ids=["c128", "c64"])
def test_lookahead_bitwise(device, monkeypatch, n, batch, prec):
    """Look-ahead (the next panel launched beside the rest of the current
    update) against the panel / update sequence: the same kernels' arithmetic
    on the same data, so the same bits, for one and several column tiles and
    both panel row counts (n > 256).  From 256 matrices on (300, 260) both
    settings run the sequence."""
    rng = np.random.default_rng(7 * n + batch + prec)
    a = _cplx(rng, (batch, n, n))
    a[:, 0, 0] = 0.0  # the first pivot needs a row interchange
    outs = {}
    for la in ("1", "0"):
        monkeypatch.setenv("QX_INV_LOOKAHEAD", la)
        A = torch.as_tensor(a, device=device)
        X = torch.empty_like(A)
        _inv(device, A, X, prec)
        outs[la] = X.cpu().numpy()
    assert np.array_equal(outs["1"].view(np.uint64), outs["0"].view(np.uint64))
    for e in range(2):
        cond = np.linalg.cond(a[e])
        tol = (1e-15 if prec == 0 else 1e-7) * cond * n
        assert rel_err(outs["1"][e], np.linalg.inv(a[e])) < tol


@pytest.mark.parametrize("nb", ["32", "64"])
@pytest.mark.parametrize("n", [64, 300])
def test_singular_panel_raises(device, monkeypatch, nb, n):
    monkeypatch.setenv("QX_INV_NB", nb)
    a = np.zeros((2, n, n), complex)
    a[0] = np.eye(n)
    a[1, :, : n // 2] = 1.0  # rank 1
    A = torch.as_tensor(a, device=device)
    X = torch.empty_like(A)
    with pytest.raises(np.linalg.LinAlgError):
        _inv(device, A, X, 0)


def test_inverse_in_place(device):
    rng = np.random.default_rng(5)
    a = _cplx(rng, (3, 40, 40))
    A = torch.as_tensor(a, device=device)
    _inv(device, A, A, 0)
    got = A.cpu().numpy()
    for e in range(3):
        assert rel_err(got[e], np.linalg.inv(a[e])) < 1e-12
    # the one-wave path (n <= 16) in place
    b = _cplx(rng, (5, 12, 12))
    B = torch.as_tensor(b, device=device)
    _inv(device, B, B, 0)
    for e in range(5):
        assert rel_err(B[e].cpu().numpy(), np.linalg.inv(b[e])) < 1e-12


def test_singular_block_raises(device):
    a = np.zeros((2, 8, 8), complex)
    a[0] = np.eye(8)
    A = torch.as_tensor(a, device=device)
    X = torch.empty_like(A)
    with pytest.raises(np.linalg.LinAlgError):
        _inv(device, A, X, 0)
    # the error flag is cleared after it was reported
    A[1] = torch.eye(8, dtype=A.dtype, device=device)
    _inv(device, A, X, 0)


@pytest.mark.parametrize("batch,n", [(159, 192), (160, 192), (161, 191), (160, 208), (256, 207),
                                     (300, 255), (160, 256), (512, 193)])
def test_wide_panel_rule(device, batch, n):
    """Both sides of the line between 32- and 64-column panels (matrices per
    call, size, filling of the last panel): residual of elimination with
    partial pivoting, 16 n eps |A| |X|, and the 32-column panels to the
    conditioning of the matrices times eps."""
    g = torch.Generator(device=device).manual_seed(batch + n)
    A = torch.randn((batch, n, n), dtype=torch.complex128, device=device, generator=g)
    A[:, 0, 0] = 0.0
    outs = []
    for nb in (None, "32"):
        with pytest.MonkeyPatch.context() as mp:
            if nb:
                mp.setenv("QX_INV_NB", nb)
            X = torch.empty_like(A)
            _inv(device, A, X, 0)
            outs.append(X)
    eps = np.finfo(float).eps
    for e in (0, batch // 2, batch - 1):
        a, x = A[e].cpu().numpy(), outs[0][e].cpu().numpy()
        kappa = np.linalg.norm(a) * np.linalg.norm(x)
        assert np.linalg.norm(x @ a - np.eye(n)) <= 16 * n * eps * kappa
        assert rel_err(x, outs[1][e].cpu().numpy()) <= 32 * n * eps * kappa


@pytest.mark.parametrize("m,n,k", [(32, 32, 16), (96, 32, 16), (32, 160, 48), (96, 96, 96),
                                   (97, 65, 33), (33, 161, 20), (160, 224, 64), (288, 320, 32),
                                   (320, 257, 17)])
@pytest.mark.parametrize("opb", [0, 2])
def test_zgemm_wave_tiles(device, m, n, k, opb):
    """Waves as the unit of the split: odd counts of 32-wide tiles (workgroups
    that hold tiles of two matrices, a last band of one tile row, a last odd
    tile column) with and without a partial tile, for an odd number of
    matrices.  Bound: the k-term dot products, 4 k eps |A| |B|."""
    rng = np.random.default_rng(m * 1000 + n)
    a = _cplx(rng, (5, m, k))
    b = _cplx(rng, (5, k, n) if opb == 0 else (5, n, k))
    c = _cplx(rng, (5, m, n))
    C = torch.as_tensor(c, device=device).clone()
    _zgemm(device, torch.as_tensor(a, device=device), torch.as_tensor(b, device=device), C, 0, opb,
           -1.0 + 0j, 1.0 + 0j, 0)
    bo = b if opb == 0 else b.conj().transpose(0, 2, 1)
    bound = 4 * (k + 2) * np.finfo(float).eps * (np.abs(a) @ np.abs(bo) + np.abs(c))
    assert (np.abs(C.cpu().numpy() - (c - a @ bo)) <= bound).all()


@pytest.mark.parametrize("n", [129, 160, 161, 191, 192, 193, 255, 257, 320, 321, 384, 385, 448, 449,
                               511, 512])
def test_column_panel_edges(device, n):
    """n > 128: panels of eight waves, at the edges of the rows a lane holds (64)
    and with full and nearly empty last panels (32).  Residual of elimination
    with partial pivoting, 16 n eps |A| |X| (growth of a random matrix well
    below n); the same bits with and without look-ahead; row permuted input
    with a zero first pivot candidate; a singular matrix is reported."""
    rng = np.random.default_rng(n)
    a = _cplx(rng, (3, n, n))
    a[0] = a[0][rng.permutation(n)]
    a[:, 0, 0] = 0.0
    A = torch.as_tensor(a, device=device)
    outs = []
    for look in ("1", "0"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("QX_INV_LOOKAHEAD", look)
            X = torch.empty_like(A)
            _inv(device, A, X, 0)
            outs.append(X.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    for e in range(3):
        x = outs[0][e]
        res = np.linalg.norm(x @ a[e] - np.eye(n))
        assert res <= 16 * n * np.finfo(float).eps * np.linalg.norm(x) * np.linalg.norm(a[e])
    A[1, :, n - 1] = 0.0
    with pytest.raises(np.linalg.LinAlgError):
        _inv(device, A, X, 0)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 17, 31, 32, 33, 40, 63, 64, 65, 95, 96, 97, 127, 128])
@pytest.mark.parametrize("in_place", [False, True])
def test_whole_inverse_edges(device, n, in_place):
    """n <= 128: one workgroup per matrix with the matrix in registers, at the
    edges of its shapes (32, 64, 96, 128), tiles (16) and sub-panels (8), with
    a subtracted matrix and leading dimensions above n, against NumPy and (to
    rounding, same pivot rule) against the split panel kernels.  Columns past
    n are left alone."""
    rng = np.random.default_rng(13 * n)
    batch, ld = 3, n + 3
    a = _cplx(rng, (batch, n, ld))
    s = 0.1 * _cplx(rng, (batch, n, n))
    a[:, 0, 0] = s[:, 0, 0] if n > 1 else a[:, 0, 0]  # a zero first pivot candidate
    from quatrex_amd import _lib as ql

    lib, h = ql.load(), ql.handle(device)
    S = torch.as_tensor(s, device=device)
    outs = {}
    for whole in ("128", "0"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("QX_INV_WHOLE", whole)
            A = torch.as_tensor(a, device=device).clone()
            X = A if in_place else torch.full_like(A, 7.0)
            rc = lib.qx_inv_batched(h, ql.stream_ptr(device), batch, n, A.data_ptr(), ld, n * ld,
                                    S.data_ptr(), n, n * n, X.data_ptr(), ld, n * ld, 0)
            ql.check(rc, h, "inv")
            ql.sync_check(device, "inv")
            outs[whole] = X.cpu().numpy()
    pad = a[:, :, n:] if in_place else 7.0
    for e in range(batch):
        m = a[e, :, :n] - s[e]
        tol = 1e-15 * np.linalg.cond(m) * max(n, 4)
        assert rel_err(outs["128"][e, :, :n], np.linalg.inv(m)) < tol
        assert rel_err(outs["128"][e, :, :n], outs["0"][e, :, :n]) < 2 * tol
    assert np.array_equal(outs["128"][:, :, n:], np.broadcast_to(pad, outs["128"][:, :, n:].shape))


@pytest.mark.parametrize("n", [20, 48, 80, 128])
def test_whole_inverse_singular_raises(device, n):
    a = np.zeros((2, n, n), complex)
    a[0] = np.eye(n)
    a[1, :, : n // 2] = 1.0  # rank 1
    A = torch.as_tensor(a, device=device)
    X = torch.empty_like(A)
    with pytest.raises(np.linalg.LinAlgError):
        _inv(device, A, X, 0)
    assert np.array_equal(X[0].cpu().numpy(), np.eye(n))


@pytest.mark.parametrize("batch,n,wide", [(159, 240, False), (160, 240, True), (160, 208, False),
                                          (223, 224, False), (224, 224, True), (224, 208, True),
                                          (256, 207, False), (257, 256, False), (256, 191, False)])
def test_wide_panel_lines(device, monkeypatch, batch, n, wide):
    """Which calls take 64-column panels: the bits are those of the width forced,
    and the two widths differ."""
    g = torch.Generator(device=device).manual_seed(n)
    A = torch.randn((batch, n, n), dtype=torch.complex128, device=device, generator=g)
    outs = []
    for nb in (None, "32", "64"):
        if nb:
            monkeypatch.setenv("QX_INV_NB", nb)
        X = torch.empty_like(A)
        _inv(device, A, X, 0)
        outs.append(torch.view_as_real(X))
    assert torch.equal(outs[0], outs[2 if wide else 1])
    assert not torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("n", [2, 3, 4, 5])
@pytest.mark.parametrize("in_place", [False, True])
def test_whole_inverse_smallest(device, n, in_place):
    """Both sides of the shape for n <= 4, as test_whole_inverse_edges."""
    test_whole_inverse_edges(device, n, in_place)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
def test_whole_inverse_smallest_bits(device, n):
    """The shape for n <= 4 gives the bits of the one for n <= 32, which the fused
    small-block inversion of a single block runs; a singular matrix raises."""
    from quatrex_amd.datastructures import DSDBCOO
    from quatrex_amd.greens_function_solver import RGF

    rng = np.random.default_rng(n)
    A = torch.as_tensor(_cplx(rng, (70, n, n)), device=device)
    if n > 1:
        A[:, 0, 0] = 0.0  # a row interchange at the first pivot
    X = torch.empty_like(A)
    _inv(device, A, X, 0)
    a = DSDBCOO(A.reshape(70, -1), np.repeat(np.arange(n), n), np.tile(np.arange(n), n), [n], (70,))
    ref = RGF(70).selected_inv(a).data.reshape(X.shape)
    assert torch.equal(torch.view_as_real(X), torch.view_as_real(ref))
    A[3, :, 0] = 0.0
    with pytest.raises(np.linalg.LinAlgError):
        _inv(device, A, X, 0)


@pytest.mark.parametrize("n", [40, 64, 65, 100, 128])
@pytest.mark.parametrize("batch", [5, 260])
def test_split_inverse_variants_up_to_128(device, monkeypatch, n, batch):
    """complex128 matrices up to 128 on the split kernels, which their whole
    inverse leaves unused by default: 16- and 32-deep chunks of the update, and
    the look-ahead or not, sum the same products in the same order."""
    rng = np.random.default_rng(11 * n + batch)
    a = _cplx(rng, (batch, n, n))
    a[:, 0, 0] = 0.0  # a row interchange at the first pivot
    A = torch.as_tensor(a, device=device)
    monkeypatch.setenv("QX_INV_WHOLE", "0")

    def run():
        X = torch.empty_like(A)
        _inv(device, A, X, 0)
        return X.cpu().numpy()

    outs = []
    for depth in ("16", "32"):
        monkeypatch.setenv("QX_INV_UPDATE", depth)
        for look in ("1", "0"):
            monkeypatch.setenv("QX_INV_LOOKAHEAD", look)
            outs.append(run())
    monkeypatch.delenv("QX_INV_UPDATE")
    monkeypatch.delenv("QX_INV_LOOKAHEAD")
    monkeypatch.delenv("QX_INV_WHOLE")
    whole = run()
    for x in outs[1:]:
        assert np.array_equal(outs[0].view(np.uint64), x.view(np.uint64))
    assert not np.array_equal(whole, outs[0])  # other kernels indeed
    for e in range(2):
        tol = 1e-15 * np.linalg.cond(a[e]) * n
        assert rel_err(outs[0][e], np.linalg.inv(a[e])) < tol
        assert rel_err(whole[e], outs[0][e]) < 2 * tol


@pytest.mark.parametrize("n", [3, 20, 32])
@pytest.mark.parametrize("batch", [1, 5, 9])
def test_smallest_whole_inverse_against_split_kernels(device, monkeypatch, n, batch):
    """n <= 32 with a subtracted matrix: the whole inverse against the split
    panels, same pivot rule, results to rounding."""
    rng = np.random.default_rng(10 * n + batch)
    a, s = _cplx(rng, (batch, n, n)), 0.1 * _cplx(rng, (batch, n, n))
    A, S = torch.as_tensor(a, device=device), torch.as_tensor(s, device=device)
    outs = []
    for whole in ("32", "0"):
        monkeypatch.setenv("QX_INV_WHOLE", whole)
        X = torch.empty_like(A)
        _inv(device, A, X, 0, S)
        outs.append(X.cpu().numpy())
    assert not np.array_equal(outs[0], outs[1])
    for e in range(batch):
        tol = 1e-15 * np.linalg.cond(a[e] - s[e]) * max(n, 4)
        assert rel_err(outs[0][e], outs[1][e]) < tol
        assert rel_err(outs[0][e], np.linalg.inv(a[e] - s[e])) < tol


def _inverse_error(A, X):
    """Log of the relative error of X as the inverse of A, per matrix: |X R| / |X|
    with the residual R = I - A X from products of 22-bit slices, whose sums over
    up to 256 terms are exact in double precision."""
    def slices(m, dim):
        scale = torch.exp2(torch.ceil(torch.log2(m.abs().amax(dim, keepdim=True))))
        out, rest = [], m / scale
        for k in (1, 2, 3):
            s = torch.round(rest * 2.0 ** (22 * k)) / 2.0 ** (22 * k)
            out.append(s * scale)
            rest = rest - s
        return out

    def products(a, b):
        sa, sb = slices(a.contiguous(), -1), slices(b.contiguous(), -2)
        return [(i + j, sa[i] @ sb[j]) for i in range(3) for j in range(3) if i + j < 4]

    re = products(A.real, X.real) + [(k, -p) for k, p in products(A.imag, X.imag)]
    im = products(A.real, X.imag) + products(A.imag, X.real)
    r = torch.eye(A.shape[-1], dtype=torch.float64, device=A.device).expand(A.shape)
    i = torch.zeros_like(r)
    for _, p in sorted(re, key=lambda t: t[0]):
        r = r - p
    for _, p in sorted(im, key=lambda t: t[0]):
        i = i - p
    e = X @ torch.complex(r, i)
    return (torch.linalg.norm(e, dim=(-2, -1)) / torch.linalg.norm(X, dim=(-2, -1))).log()


@pytest.mark.parametrize("n,batch,knob,values,most", [
    (24, 1000, "QX_INV_WHOLE", ("32", "0"), -0.05), (32, 1000, "QX_INV_WHOLE", ("32", "0"), -0.05),
    (208, 250, "QX_INV_NB", ("64", "32"), 0.07), (256, 250, "QX_INV_NB", ("64", "32"), 0.07)])
def test_inverse_rounding(device, monkeypatch, n, batch, knob, values, most):
    """Where products are summed before they are subtracted (whole inverses up to
    32 rows, 64-column panels) the error is not above that of the 32-column panels
    beside them, which choose the same pivots and fuse product by product: mean of
    the logarithm over matrices E + i eta - H, H Hermitian, standard error 0.01 and
    0.03.  Fused they were 0.03 to 0.06 and 0.10 to 0.17 above."""
    g = torch.Generator(device=device).manual_seed(n)
    x = torch.randn((batch, n, n), dtype=torch.complex128, device=device, generator=g)
    h = (x + x.conj().transpose(1, 2)) / (2 * n) ** 0.5
    e = 2 * torch.rand((batch, 1, 1), dtype=torch.float64, device=device, generator=g) - 1
    A = (e + 1e-3j) * torch.eye(n, device=device) - h
    log = []
    for v in values:
        monkeypatch.setenv(knob, v)
        X = torch.empty_like(A)
        _inv(device, A, X, 0)
        log.append(_inverse_error(A, X))
    assert float((log[0] - log[1]).mean()) <= most
