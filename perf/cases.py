"""Performance cases: the work a user of this framework has it do, each through a public entry point.

``listed()`` holds the named cases, ``draw(rng)`` one more case of the same ranges,
``prepare(case, seed)`` what a program has in hand before the call, ``run(state)`` one pass,
``work(case)`` the bytes and flops a pass cannot do without, and ``exact(case, seed)`` the same
outputs from plain torch operations in 64 bits.

Kinds of cases and where their sizes come from:

- ``solve``: ``RGF.selected_solve``, the product's main call (G^<, G^>, and on request the diagonal
  of G^R, the layer current, the density, boundary blocks).  Block sizes 16 to 416, 4 to 64 blocks,
  16 to 512 energies: the range between the 16 x 8 x 32 configuration and the 512 x 64 x 256 one.
- ``inverse``: ``RGF.selected_inv`` (G^R alone: transmission, LDOS), same range.
- ``lead``: ``SanchoRubio``, the surface Green's function of a lead over an energy grid (the
  1024-energy, 256-orbital lead configuration and below).
- ``contacts``: ``contact_obc_blocks``, both contacts of a device from its system matrix to the
  boundary self-energies, as a transport iteration runs it before every solve.
- ``contour``: ``operator_inverse``, the contour-node inverses of the Beyn eigenvalue solver (many
  independent dense inverses in one call).
- ``assemble``: ``SystemMatrixAssembler``, A = (E + i eta) - H - Sigma^R over an energy grid.
- ``mix``: ``UnevenBatch``, devices of different block sizes side by side on lanes.

All data is complex128, the only storage type of the framework; the arithmetic option that keeps its
accuracy ("c128-3m") has a case of its own.
"""

import math

import numpy as np
import torch

from quatrex_amd.boundary_conditions import OBCSystem, SanchoRubio
from quatrex_amd.datastructures import empty_btd
from quatrex_amd.engine import UnevenBatch, Device
from quatrex_amd.greens_function_solver import RGF, OBCBlocks
from quatrex_amd.leads import contact_obc_blocks
from quatrex_amd.nevp import operator_inverse
from quatrex_amd.observables import SystemMatrixAssembler
from quatrex_amd.workloads import make_workload

ETA = 1e-3
DEV = "cuda"
C128 = torch.complex128


def _solve(name, energies, blocks, size, ragged=0, precision="c128", retarded=True, current=False,
           contacts=False, density=False):
    return {"name": name, "kind": "solve", "energies": energies, "blocks": blocks, "size": size,
            "ragged": ragged, "precision": precision, "retarded": retarded, "current": current,
            "contacts": contacts, "density": density}


def listed():
    return [
        # a short device in a small basis, with its layer current: the smallest call, all latency
        _solve("solve_16x8x32", 16, 8, 32, current=True),
        # a whole energy grid of a narrow device, odd block size: small blocks, many energies
        _solve("solve_300x11x20", 300, 11, 20),
        # a nanowire in a minimal basis over an energy grid: small blocks, a longer chain
        _solve("solve_256x32x64", 256, 32, 64),
        # a device with layers of different widths and its boundary self-energies, current and
        # density: every optional part of the call, no size a multiple of a tile
        _solve("solve_48x10_ragged", 48, 10, 176, ragged=1, current=True, contacts=True,
               density=True),
        # one energy batch of the large production shape
        _solve("solve_64x64x256", 64, 64, 256),
        # the three-multiplication complex product at the same block size
        _solve("solve_3m_32x16x256", 32, 16, 256, precision="c128-3m"),
        # retarded Green's function only
        {"name": "inverse_128x24x128", "kind": "inverse", "energies": 128, "blocks": 24,
         "size": 128, "ragged": 0},
        # the large lead layer
        {"name": "lead_512x256", "kind": "lead", "energies": 512, "size": 256},
        # both contacts of a mid-sized device, few energies
        {"name": "contacts_32x96", "kind": "contacts", "energies": 32, "size": 96},
        # contour nodes of a lead's eigenvalue problem
        {"name": "contour_4x64x256", "kind": "contour", "energies": 4, "nodes": 64, "size": 256},
        # system matrix of a whole energy grid, with a scattering self-energy
        {"name": "assemble_256x32x96", "kind": "assemble", "energies": 256, "blocks": 32,
         "size": 96},
        # four devices, one of each block size of the uneven configuration
        {"name": "mix_4", "kind": "mix", "energies": 48, "blocks": 16, "size": 416},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# A drawn case does no more than this (flops, bytes), below the largest listed case.
_MOST_FLOPS, _MOST_BYTES = 6e12, 1.2e10


def draw(rng):
    kind = rng.choice(["solve"] * 6 + ["inverse"] * 2 + ["lead", "contacts", "contour", "assemble"])
    while True:
        energies = _log_int(rng, 16, 512)
        if kind in ("solve", "inverse"):
            size, blocks = _log_int(rng, 16, 320), rng.randint(4, 40)
            case = {"kind": kind, "energies": energies, "blocks": blocks, "size": size,
                    "ragged": rng.choice([0, 0, 1])}
            if kind == "solve":
                option = rng.choice(["", "", "current", "contacts"])
                case = dict(_solve("", energies, blocks, size, ragged=case["ragged"],
                                   precision=rng.choice(["c128", "c128", "c128", "c128-3m"]),
                                   retarded=rng.choice([True, True, False]),
                                   current=option == "current", contacts=option == "contacts",
                                   density=option == "contacts"))
                del case["name"]
        elif kind in ("lead", "contacts"):
            case = {"kind": kind, "energies": energies, "size": _log_int(rng, 32, 288)}
        elif kind == "contour":
            case = {"kind": kind, "energies": rng.randint(1, 8), "nodes": rng.choice([16, 32, 64]),
                    "size": _log_int(rng, 32, 288)}
        else:
            case = {"kind": kind, "energies": energies, "blocks": rng.randint(8, 40),
                    "size": _log_int(rng, 32, 160)}
        w = work(case)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return case


# ---- inputs ------------------------------------------------------------------------------------


def _sizes(case):
    """Block sizes: all equal, or spread by up to a quarter around the size."""
    n, b = case["blocks"], case["size"]
    if not case.get("ragged"):
        return [b] * n
    return [max(2, b + (b * ((5 * i) % 7 - 3)) // 12) for i in range(n)]


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _cn(g, *shape):
    return torch.randn(*shape, dtype=C128, generator=g, device=DEV)


def _h(x):
    return x.transpose(-1, -2).conj()


def _broadening(g, b):
    x = _cn(g, b, b)
    return (x @ _h(x)) / b


class _System:
    """Blocks of A = E - H - Sigma_B per energy and of Sigma^< and Sigma^>, as a transport problem
    has them: Hermitian H with unit-spread blocks, energies in its band, i Gamma f and
    -i Gamma (1 - f) self-energies on every block."""

    def __init__(self, seed, n_e, sizes, contacts=False):
        g = _generator(seed)
        n = len(sizes)
        self.sizes, self.n_e = sizes, n_e
        self.energies = (2 * torch.rand(n_e, dtype=torch.float64, generator=g, device=DEV) - 1) + 0j
        self.energies = self.energies + 1j * ETA
        self.h, self.u, self.sl, self.sg = [], [], [], []
        for i, b in enumerate(sizes):
            x = _cn(g, b, b) / math.sqrt(b)
            self.h.append((x + _h(x)) / 2)
            self.sl.append(1j * _broadening(g, b))
            self.sg.append(-1j * _broadening(g, b))
            if i + 1 < n:
                self.u.append(_cn(g, b, sizes[i + 1]) / math.sqrt(b))
        self.lead = {}
        for i in {0, n - 1}:
            gamma = _broadening(g, sizes[i])
            if contacts:  # boundary blocks handed to the solver, one stack per quantity
                f = torch.rand(n_e, 1, 1, dtype=torch.float64, generator=g, device=DEV)
                self.lead[i] = ((-1j * gamma).expand(n_e, -1, -1).contiguous(),
                                1j * f * gamma, -1j * (1 - f) * gamma)
            else:  # folded into the system matrix
                self.h[i] = self.h[i] - 1j * gamma

    def a_diag(self, i):
        b = self.sizes[i]
        eye = torch.eye(b, dtype=C128, device=DEV)
        return self.energies[:, None, None] * eye - self.h[i]


def _fill(container, offsets, blocks):
    for (i, j), block in blocks:
        o = offsets[i, j]
        n = block.shape[-2] * block.shape[-1]
        container.data[:, o:o + n] = block.reshape(-1, n)


def _matrix(system):
    n = len(system.sizes)
    a, off = empty_btd(system.sizes, (system.n_e,), device=DEV, zero=False)
    _fill(a, off, (((i, i), system.a_diag(i)) for i in range(n)))
    _fill(a, off, (((i, i + 1), -u) for i, u in enumerate(system.u)))
    _fill(a, off, (((i + 1, i), -_h(u)) for i, u in enumerate(system.u)))
    return a


def _block_diagonal(system, blocks):
    x, off = empty_btd(system.sizes, (system.n_e,), offdiag=False, device=DEV, zero=False)
    _fill(x, off, (((i, i), b) for i, b in enumerate(blocks)))
    return x


def _lead(case, seed):
    """(a_ii, a_ij, a_ji) of a semi-infinite lead of one principal layer."""
    g, b = _generator(seed), case["size"]
    e = 2 * torch.rand(case["energies"], dtype=torch.float64, generator=g, device=DEV) - 1
    x = _cn(g, b, b) / math.sqrt(b)
    h01 = _cn(g, b, b) / math.sqrt(b)
    eye = torch.eye(b, dtype=C128, device=DEV)
    a_ii = (e + 1j * ETA)[:, None, None] * eye - (x + _h(x)) / 2
    n = case["energies"]
    return (a_ii, (-h01).expand(n, b, b).contiguous(), (-_h(h01)).expand(n, b, b).contiguous())


def _contacts_system(case, seed):
    """A device whose first and last layers repeat into its leads."""
    return _System(seed, case["energies"], [case["size"]] * 4)


def _occupations(case, seed):
    g = _generator(seed + 1)
    e = torch.rand(2, case["energies"], dtype=torch.float64, generator=g, device=DEV)
    return e[0], e[1]


def _nodes(case):
    """Quadrature nodes on the outer contour, |z| = 1.5."""
    k = np.arange(case["nodes"]) + 1.5
    return (1.5 * np.exp(2j * np.pi * k / case["nodes"])).reshape(1, -1, 1, 1)


def _mix_shapes(case):
    """(energies, blocks, block size) of the devices: small blocks come with more energies."""
    top = case["size"]
    return [(case["energies"], case["blocks"] + 8, max(8, 64 * top // 416)),
            (case["energies"] // 2, case["blocks"] + 4, max(8, 128 * top // 416)),
            (case["energies"] // 3, case["blocks"], max(8, 256 * top // 416)),
            (case["energies"] // 6, case["blocks"], top)]


def _mix_workloads(case, seed):
    return [make_workload(seed=seed + 17 * k, n_energies=e, n_blocks=n, block_size=b)
            for k, (e, n, b) in enumerate(_mix_shapes(case))]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        s = _System(seed, case["energies"], _sizes(case), case["contacts"])
        a, sl, sg = _matrix(s), _block_diagonal(s, s.sl), _block_diagonal(s, s.sg)
        out = [empty_btd(s.sizes, (s.n_e,), device=DEV)[0] for _ in range(2)]
        if case["retarded"]:
            out.append(empty_btd(s.sizes, (s.n_e,), offdiag=False, device=DEV)[0])
        obc = None
        if case["contacts"]:
            obc = OBCBlocks(len(s.sizes))
            for i, (r, lo, gr) in s.lead.items():
                obc.retarded[i], obc.lesser[i], obc.greater[i] = r, lo, gr
        density = None
        if case["density"]:
            density = torch.zeros(s.n_e, sum(s.sizes), dtype=torch.float64, device=DEV)
        return {"kind": kind, "case": case, "a": a, "sl": sl, "sg": sg, "out": tuple(out),
                "obc": obc, "density": density,
                "solver": RGF(max_batch_size=s.n_e, precision=case["precision"])}
    if kind == "inverse":
        s = _System(seed, case["energies"], _sizes(case))
        return {"kind": kind, "a": _matrix(s), "out": empty_btd(s.sizes, (s.n_e,), device=DEV)[0],
                "solver": RGF(max_batch_size=s.n_e)}
    if kind == "lead":
        return {"kind": kind, "blocks": _lead(case, seed),
                "solver": SanchoRubio(max_iterations=100, convergence_tol=1e-6)}
    if kind == "contacts":
        left, right = _occupations(case, seed)
        return {"kind": kind, "a": _matrix(_contacts_system(case, seed)), "left": left,
                "right": right,
                "system": OBCSystem(SanchoRubio(max_iterations=100, convergence_tol=1e-6),
                                    memoization_mode="off")}
    if kind == "contour":
        a_ii, a_ij, a_ji = _lead(case, seed)
        return {"kind": kind, "a_xx": tuple(x[:, None] for x in (a_ji, a_ii, a_ij)),
                "z": _nodes(case)}
    if kind == "assemble":
        sizes = [case["size"]] * case["blocks"]
        g = _generator(seed)
        pattern, _ = empty_btd(sizes, (case["energies"],), device=DEV)
        sigma, _ = empty_btd(sizes, (case["energies"],), device=DEV, zero=False)
        for row in sigma.data:
            row.copy_(_cn(g, row.shape[0]))
        return {"kind": kind, "sigma": sigma, "out": pattern,
                "energies": _grid(case, seed),
                "assembler": SystemMatrixAssembler(pattern, _hamiltonian(case, seed))}
    devices = [Device(w, DEV) for w in _mix_workloads(case, seed)]
    return {"kind": kind, "batch": UnevenBatch(devices, n_lanes=4, default_chunk=16)}


def _grid(case, seed):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, case["energies"])


def _hamiltonian(case, seed):
    """Sparse block-tridiagonal Hamiltonian of the device (host, as a program reads it)."""
    import scipy.sparse as sps

    n, b = case["blocks"], case["size"]
    rng = np.random.default_rng(seed + 1)
    grid = [[None] * n for _ in range(n)]
    for i in range(n):
        x = rng.standard_normal((b, b)) + 1j * rng.standard_normal((b, b))
        grid[i][i] = sps.coo_matrix((x + x.conj().T) / (2 * math.sqrt(2 * b)))
        if i + 1 < n:
            u = (rng.standard_normal((b, b)) + 1j * rng.standard_normal((b, b))) / math.sqrt(2 * b)
            grid[i][i + 1], grid[i + 1][i] = sps.coo_matrix(u), sps.coo_matrix(u.conj().T)
    return sps.bmat(grid, format="csr")


# ---- one pass ----------------------------------------------------------------------------------


def run(state):
    kind = state["kind"]
    if kind == "solve":
        case = state["case"]
        more = {"density": state["density"]} if case["density"] else {}
        current = state["solver"].selected_solve(
            state["a"], state["sl"], state["sg"], obc_blocks=state["obc"], out=state["out"],
            return_retarded=case["retarded"], return_current=case["current"], **more)
        result = {"lesser": state["out"][0].data, "greater": state["out"][1].data, **more}
        if case["retarded"]:
            result["retarded"] = state["out"][2].data
        if case["current"]:
            result["current"] = current
        return result
    if kind == "inverse":
        state["solver"].selected_inv(state["a"], out=state["out"])
        return state["out"].data
    if kind == "lead":
        return state["solver"](*state["blocks"], contact="left")
    if kind == "contacts":
        obc = contact_obc_blocks(state["a"], state["system"], state["left"], state["right"])
        return {name: [blocks[0], blocks[-1]] for name, blocks in
                (("retarded", obc.retarded), ("lesser", obc.lesser), ("greater", obc.greater))}
    if kind == "contour":
        return operator_inverse(state["a_xx"], state["z"])
    if kind == "assemble":
        return state["assembler"](state["energies"], ETA, sse_retarded=state["sigma"],
                                  out=state["out"]).data
    state["batch"].run_eager()
    return [{"density": d.density, "transmission": d.transmission}
            for d in state["batch"].devices]


# ---- what a pass cannot do without -------------------------------------------------------------


def _chain(sizes, n_e, products_first, products_step):
    """Flops of a block recursion: an inverse per block, products of 8 b^3 per block and step."""
    f = [8.0 * b ** 3 for b in sizes]
    return n_e * (sum(f) + products_first * f[0]
                  + products_step * sum((x + y) / 2 for x, y in zip(f, f[1:])))


def _btd_bytes(sizes, n_e, offdiag=True):
    n = sum(b * b for b in sizes)
    if offdiag:
        n += 2 * sum(x * y for x, y in zip(sizes, sizes[1:]))
    return 16.0 * n * n_e


def work(case):
    kind, n_e = case["kind"], case.get("energies", 0)
    if kind == "solve":
        # forward: two products per step for G^R, four each for G^< and G^>; backward: four for
        # G^R, three each for the skew-Hermitian G^< and G^>
        sizes = _sizes(case)
        read = _btd_bytes(sizes, n_e) + 2 * _btd_bytes(sizes, n_e, False)
        written = 2 * _btd_bytes(sizes, n_e)
        if case["retarded"]:
            written += _btd_bytes(sizes, n_e, False)
        return {"bytes": read + written, "flops": _chain(sizes, n_e, 4, 20)}
    if kind == "inverse":
        sizes = _sizes(case)
        return {"bytes": 2 * _btd_bytes(sizes, n_e), "flops": _chain(sizes, n_e, 0, 6)}
    b = case["size"]
    bb = 16.0 * b * b
    if kind == "lead":  # about 14 iterations of an inverse and six products, and a last inverse
        return {"bytes": 4 * bb * n_e, "flops": 8.0 * b ** 3 * n_e * (14 * 7 + 1)}
    if kind == "contacts":  # two leads; refinement step and residual; Sigma^R, Sigma^<, Sigma^>
        return {"bytes": 12 * bb * n_e, "flops": 2 * 8.0 * b ** 3 * n_e * (14 * 7 + 1 + 3 + 2)}
    if kind == "contour":
        nodes = n_e * case["nodes"]
        return {"bytes": bb * (3 * n_e + nodes), "flops": 8.0 * b ** 3 * nodes}
    if kind == "assemble":
        one = _btd_bytes([b] * case["blocks"], 1)
        return {"bytes": one * (2 * n_e + 2), "flops": one / 16 * n_e * 12}
    flops, read = 0.0, 0.0
    for e, n, size in _mix_shapes(case):
        # the recursion, the corner block (two products per step) and the transmission (three)
        flops += _chain([size] * n, e, 4 + 3, 20 + 2)
        read += _btd_bytes([size] * n, 1) + 2 * _btd_bytes([size] * n, 1, False) + 8.0 * e * n * size
    return {"bytes": read, "flops": flops}


# ---- the same outputs in plain torch -----------------------------------------------------------


def _inv(x):
    flat = x.reshape(-1, *x.shape[-2:])
    return torch.cat([torch.linalg.inv(part) for part in flat.split(64)]).reshape(x.shape)


def _recursion(a_diag, upper, lower, sl, sg):
    """Selected blocks of G^R = A^-1 and G^<> = G^R Sigma^<> G^R^H for block-diagonal Sigma^<>:
    the standard forward and backward recursion, every block product a plain torch product."""
    n = len(a_diag)
    g, x = [_inv(a_diag[0])], [[], []]
    for q, s in enumerate((sl, sg)):
        x[q].append(g[0] @ s[0] @ _h(g[0]))
    for i in range(n - 1):
        g.append(_inv(a_diag[i + 1] - lower[i] @ g[i] @ upper[i]))
        for q, s in enumerate((sl, sg)):
            x[q].append(g[-1] @ (s[i + 1] + lower[i] @ x[q][i] @ _h(lower[i])) @ _h(g[-1]))
    left = list(g)
    up, down = [None] * (n - 1), [None] * (n - 1)
    ups = [[None] * (n - 1), [None] * (n - 1)]
    for i in range(n - 2, -1, -1):
        down[i] = -g[i + 1] @ lower[i] @ g[i]
        b1, t = g[i] @ upper[i], g[i + 1] @ lower[i]
        for q in range(2):
            ups[q][i] = -b1 @ x[q][i + 1] - x[q][i] @ _h(t)
            cross = b1 @ t @ x[q][i]
            x[q][i] = x[q][i] + (cross - _h(cross)) + b1 @ x[q][i + 1] @ _h(b1)
        up[i] = -b1 @ g[i + 1]
        g[i] = g[i] - b1 @ down[i]
    return {"g": g, "up": up, "down": down, "x": x, "ups": ups, "left": left}


def _btd(diag, up, down):
    """Blocks in the container's order: (i, i-1), (i, i), (i, i+1) of each block row."""
    parts, n = [], len(diag)
    for i in range(n):
        if i > 0 and down is not None:
            parts.append(down[i - 1])
        parts.append(diag[i])
        if i + 1 < n and up is not None:
            parts.append(up[i])
    n_e = diag[0].shape[0]
    return torch.cat([p.reshape(n_e, -1) for p in parts], dim=-1)


def _skew(x):
    return (x - _h(x)) / 2


def _exact_solve(case, seed):
    s = _System(seed, case["energies"], _sizes(case), case["contacts"])
    n = len(s.sizes)
    diag = [s.a_diag(i) for i in range(n)]
    sl, sg = list(s.sl), list(s.sg)
    for i, (r, lo, gr) in s.lead.items():
        diag[i], sl[i], sg[i] = diag[i] - r, sl[i] + lo, sg[i] + gr
    upper, lower = [-u for u in s.u], [-_h(u) for u in s.u]
    r = _recursion(diag, upper, lower, sl, sg)
    result = {}
    for q, name in enumerate(("lesser", "greater")):
        result[name] = _btd([_skew(x) for x in r["x"][q]], r["ups"][q],
                            [-_h(x) for x in r["ups"][q]])
    if case["density"]:
        result["density"] = torch.cat([torch.diagonal(x, dim1=-2, dim2=-1).imag
                                       for x in r["x"][0]], dim=-1)
    if case["retarded"]:
        result["retarded"] = _btd(r["g"], None, None)
    if case["current"]:
        # layer currents Tr[Sigma~^> G^< - G^> Sigma~^<] from the left-connected blocks
        left = _recursion_left(r["left"], lower, sl, sg)
        cur = []
        for i in range(n - 1):
            t = [lower[i] @ left[q][i] @ _h(lower[i]) for q in range(2)]
            m = t[1] @ r["x"][0][i + 1] - r["x"][1][i + 1] @ t[0]
            cur.append(torch.diagonal(m, dim1=-2, dim2=-1).sum(-1))
        result["current"] = torch.stack(cur, dim=-1)
    return result


def _recursion_left(g, lower, sl, sg):
    """Left-connected G^<> blocks."""
    x = [[], []]
    for q, s in enumerate((sl, sg)):
        x[q].append(g[0] @ s[0] @ _h(g[0]))
        for i in range(len(g) - 1):
            inner = s[i + 1] + lower[i] @ x[q][i] @ _h(lower[i])
            x[q].append(g[i + 1] @ inner @ _h(g[i + 1]))
    return x


def _surface(a_ii, a_ij, a_ji):
    """Surface Green's function of a lead by decimation until the couplings vanish."""
    eps, surface, alpha, beta = a_ii, a_ii, a_ji, a_ij
    for _ in range(60):
        g = _inv(eps)
        step = alpha @ g @ beta
        eps, surface = eps - step - beta @ g @ alpha, surface - step
        alpha, beta = alpha @ g @ alpha, beta @ g @ beta
        if float((alpha.abs() + beta.abs()).amax()) < 1e-13:
            break
    return _inv(surface)


def _flip(x):
    return torch.flip(x, dims=(-2, -1))


def _exact_contacts(case, seed):
    s = _contacts_system(case, seed)
    left, right = _occupations(case, seed)
    n_e = case["energies"]
    last = len(s.sizes) - 1
    result = {"retarded": [], "lesser": [], "greater": []}
    first = (s.a_diag(0), (-s.u[0]).expand(n_e, -1, -1), (-_h(s.u[0])).expand(n_e, -1, -1))
    end = (s.a_diag(last), (-_h(s.u[-1])).expand(n_e, -1, -1), (-s.u[-1]).expand(n_e, -1, -1))
    for (a_ii, a_ij, a_ji), f, flip in ((first, left, lambda x: x), (end, right, _flip)):
        g = flip(_surface(flip(a_ii), flip(a_ij), flip(a_ji)))
        sigma = a_ji @ g @ a_ij
        gamma = sigma - _h(sigma)
        f = f[:, None, None]
        result["retarded"].append(sigma)
        result["lesser"].append(-f * gamma)
        result["greater"].append((1 - f) * gamma)
    return result


def _exact_mix(case, seed):
    result = []
    for w in _mix_workloads(case, seed):
        n, e = w.n_blocks, len(w.energies)

        def dev(x):
            return torch.as_tensor(np.ascontiguousarray(x), device=DEV)

        diag, upper, lower = w.a_blocks()
        diag, upper, lower = ([dev(x) for x in v] for v in (diag, upper, lower))
        sl, sg = [dev(x) for x in w.sl_diag], [dev(x) for x in w.sg_diag]
        r = _recursion(diag, upper, lower, sl, sg)
        density = torch.cat([torch.diagonal(x, dim1=-2, dim2=-1).imag for x in r["x"][0]], dim=-1)
        corner = r["left"][0]
        for i in range(n - 1):
            corner = -corner @ upper[i] @ r["left"][i + 1]
        gl, gr = (dev(1j * (x - x.conj().T)) for x in (w.sigma_b_left, w.sigma_b_right))
        t = gl @ corner @ gr @ _h(corner)
        result.append({"density": density,
                       "transmission": torch.diagonal(t, dim1=-2, dim2=-1).sum(-1).real})
    return result


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        return _exact_solve(case, seed)
    if kind == "inverse":
        s = _System(seed, case["energies"], _sizes(case))
        n = len(s.sizes)
        zero = [torch.zeros_like(x) for x in s.sl]
        r = _recursion([s.a_diag(i) for i in range(n)], [-u for u in s.u], [-_h(u) for u in s.u],
                       zero, zero)
        return _btd(r["g"], r["up"], r["down"])
    if kind == "lead":
        return _surface(*_lead(case, seed))
    if kind == "contacts":
        return _exact_contacts(case, seed)
    if kind == "contour":
        a_ii, a_ij, a_ji = (x[:, None] for x in _lead(case, seed))
        z = torch.as_tensor(_nodes(case), device=DEV)
        m = a_ji / z + a_ii + a_ij * z
        return _inv(m.reshape(-1, *m.shape[-2:])).reshape(m.shape)
    if kind == "assemble":
        rows_cols = empty_btd([case["size"]] * case["blocks"], (1,), device="cpu")[0]
        rows, cols = rows_cols.rows, rows_cols.cols
        h = np.asarray(_hamiltonian(case, seed)[rows, cols]).ravel()
        g = _generator(seed)
        e = torch.as_tensor(_grid(case, seed) + 1j * ETA, device=DEV)
        unit = torch.as_tensor((rows == cols).astype(np.complex128), device=DEV)
        base = torch.as_tensor(h, device=DEV)
        return torch.stack([z * unit - base - _cn(g, len(rows)) for z in e])
    return _exact_mix(case, seed)
