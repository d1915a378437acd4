"""The sub-batches of one RGF call (streams of a handle) change only timing.

A call's energies run in up to four contiguous ranges on streams of their own.
The energies are independent, so every output is bitwise that of the call run
in one range, whatever the number of ranges and however the energies divide
between them.  The launch counts show how many ranges a call really took, so
the comparison cannot become one of a path with itself.
"""

import pytest
import torch

from quatrex_amd import _lib
from quatrex_amd.datastructures import empty_btd
from quatrex_amd.greens_function_solver import RGF, OBCBlocks

pytestmark = pytest.mark.gpu


def _h(x):
    return x.transpose(-1, -2).conj()


def _stack(device, sizes, n_e, seed, skew):
    """Random block-tridiagonal stack, every energy another one: diagonally
    dominant, or block-diagonal and skew-Hermitian."""
    g = torch.Generator(device=device).manual_seed(seed)
    m, off = empty_btd(sizes, (n_e,), offdiag=not skew, device=device, zero=False)

    def cn(*shape):
        return torch.randn(*shape, dtype=torch.complex128, generator=g, device=device)

    def put(i, j, x):
        o = off[i, j]
        m.data[:, o:o + x[0].numel()] = x.reshape(n_e, -1)

    for i, b in enumerate(sizes):
        x = cn(n_e, b, b) / b ** 0.5
        put(i, i, x - _h(x) if skew else x + 4 * torch.eye(b, device=device))
        if not skew and i + 1 < len(sizes):
            c = sizes[i + 1]
            put(i, i + 1, 0.5 * cn(n_e, b, c) / b ** 0.5)
            put(i + 1, i, 0.5 * cn(n_e, c, b) / b ** 0.5)
    return m


def _boundary(device, sizes, n_e):
    obc = OBCBlocks(len(sizes))
    g = torch.Generator(device=device).manual_seed(7)
    for i in (0, len(sizes) - 1):
        b = sizes[i]
        x = torch.randn(n_e, b, b, dtype=torch.complex128, generator=g, device=device) / b
        obc.retarded[i], obc.lesser[i], obc.greater[i] = x, x - _h(x), 0.5 * (_h(x) - x)
    return obc


def _on_streams(device, streams, call):
    """(outputs of call(), product launches) with at most `streams` ranges."""
    h = _lib.new_handle(device)
    _lib.set_tuning(h, streams=streams)
    with _lib.use_handle(h):
        with _lib.KernelTimer(device) as timer:
            out = call()
    _lib.load().qx_destroy(h)
    return out, timer.stats["gemm"]["launches"]


def _same_bits(device, call, counts):
    ref, launches = _on_streams(device, 1, call)
    for streams in counts:
        got, n = _on_streams(device, streams, call)
        assert n == streams * launches, "the call did not run in that many ranges"
        for name in ref:
            x, y = (torch.view_as_real(t) if t.is_complex() else t for t in (got[name], ref[name]))
            assert torch.equal(x, y), (streams, name)


# (energies, block sizes): ranges of unequal lengths; whole inverses, and panels
# on a stack that a call in one range passes to the inverse as 250 matrices
STACKS = [(518, [64, 48, 64]), (250, [208, 256, 200])]


@pytest.mark.parametrize("n_e,sizes", STACKS, ids=["518x64", "250x256"])
@pytest.mark.parametrize("precision", ["c128", "c128-3m", "mixed"])
@pytest.mark.parametrize("sigma", ["skew", "one-not-skew"])
def test_solve_bits(device, n_e, sizes, precision, sigma):
    """selected_solve with boundary blocks and every optional output; with one
    energy whose Sigma is not skew-Hermitian, in the last range only."""
    a = _stack(device, sizes, n_e, 1, False)
    sl, sg = _stack(device, sizes, n_e, 2, True), _stack(device, sizes, n_e, 3, True)
    if sigma != "skew":
        sg.data[n_e - 2, 5] += 0.25
    obc = _boundary(device, sizes, n_e)

    def call():
        out = [empty_btd(sizes, (n_e,), device=device)[0] for _ in range(2)]
        out.append(empty_btd(sizes, (n_e,), offdiag=False, device=device)[0])
        density = torch.zeros(n_e, sum(sizes), dtype=torch.float64, device=device)
        corner = torch.zeros(n_e, sizes[0], sizes[-1], dtype=torch.complex128, device=device)
        current = RGF(n_e, precision=precision).selected_solve(
            a, sl, sg, obc_blocks=obc, out=tuple(out), return_retarded=True, return_current=True,
            density=density, corner=corner)
        return {"lesser": out[0].data, "greater": out[1].data, "retarded": out[2].data,
                "current": current, "density": density, "corner": corner}

    _same_bits(device, call, (2, 3, 4))


@pytest.mark.parametrize("n_e,sizes", STACKS, ids=["518x64", "250x256"])
@pytest.mark.parametrize("precision", ["c128", "c128-3m", "mixed"])
def test_inverse_bits(device, n_e, sizes, precision):
    """selected_inv with boundary blocks, new output and output over A."""
    a = _stack(device, sizes, n_e, 1, False)
    obc = _boundary(device, sizes, n_e)

    def call():
        x = empty_btd(sizes, (n_e,), device=device)[0]
        RGF(n_e, precision=precision).selected_inv(a, obc_blocks=obc, out=x)
        y = empty_btd(sizes, (n_e,), device=device)[0]
        y.data.copy_(a.data)
        RGF(n_e, precision=precision).selected_inv(y, obc_blocks=obc, out=y)
        return {"x": x.data, "in place": y.data}

    _same_bits(device, call, (2, 3, 4))


@pytest.mark.parametrize("n_e,sizes", STACKS, ids=["518x64", "250x256"])
def test_offset_of_the_ranges_bits(device, monkeypatch, n_e, sizes):
    """The odd ranges start after the first one's first block inverse
    (QX_RGF_STAGGER): the bits of ranges started together, over several calls on
    one handle."""
    a = _stack(device, sizes, n_e, 1, False)
    sl, sg = _stack(device, sizes, n_e, 2, True), _stack(device, sizes, n_e, 3, True)

    def call():
        out = [empty_btd(sizes, (n_e,), device=device)[0] for _ in range(3)]
        for _ in range(3):
            RGF(n_e).selected_solve(a, sl, sg, out=tuple(out), return_retarded=True)
        return {k: m.data for k, m in enumerate(out)}

    outs = []
    for stagger in ("1", "0"):
        monkeypatch.setenv("QX_RGF_STAGGER", stagger)
        outs.append(_on_streams(device, 4, call))
    (ref, launches), (got, n) = outs
    assert n == launches == 4 * _on_streams(device, 1, call)[1]
    for k in ref:
        assert torch.equal(torch.view_as_real(got[k]), torch.view_as_real(ref[k]))
