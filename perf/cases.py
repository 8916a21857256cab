"""Performance cases of the CheFSI + AAR hot path through sparc_amd's public
entry points: the Chebyshev filter, single Hamiltonian applications, the
subspace projection, rotation and eigensolve, the AAR Poisson solve with the
Jacobi and the learned preconditioner, the training of the latter, and whole
SCF iterations.

Sizes are those of the framework's own workloads (diamond-cubic Si with 8, 64
and 216 atoms on 26^3, 52^3 and 78^3 grids with 24, 160 and 480 states, the
96^3 x 512 degree-24 operator filter, the 128^3 Poisson problem) and odd or
ragged ones around them.

A case is a dict of plain values.  prepare() makes the inputs from the seed
and the context, blocks and operator data a program keeps; run() is one pass;
exact() is the same in 64 bits with plain torch.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from sparc_amd import gpu
from sparc_amd.model import diamond_cubic
from sparc_amd.systems import silicon
from sparc_amd.workloads import Grid, gaussian_projectors

ORDER = 12
CELL = 10.26  # Bohr, the 8-atom diamond-cubic cell


def listed():
    return [
        # one filter of the 8-atom cell: 421k values per block, launch and latency bound
        dict(name="filter_8atoms_f32", kind="filter", nx=26, ny=26, nz=26, h=0.3946, dirichlet_z=False,
             ncol=24, degree=20, dtype="f32", rc=2.0, sites=8),
        # the all-FP64 filter of the 64-atom cell (reference precision)
        dict(name="filter_64atoms_f64", kind="filter", nx=52, ny=52, nz=52, h=0.3946, dirichlet_z=False,
             ncol=160, degree=20, dtype="f64", rc=2.0, sites=64),
        # the filter of the largest SCF system, in the mixed-precision mode it runs in
        dict(name="filter_216atoms_f32", kind="filter", nx=78, ny=78, nz=78, h=0.3946, dirichlet_z=False,
             ncol=480, degree=20, dtype="f32", rc=2.0, sites=216),
        # the operator-level benchmark: large projector spheres that overlap
        dict(name="filter_96cubed_f32", kind="filter", nx=96, ny=96, nz=96, h=0.3, dirichlet_z=False,
             ncol=512, degree=24, dtype="f32", rc=6.0, sites=64),
        # one Hamiltonian application on a slab (Dirichlet along z) with odd
        # dimensions and an odd column count, as a residual check makes it
        dict(name="hamiltonian_slab_f64", kind="hamiltonian", nx=45, ny=51, nz=73, h=0.38, dirichlet_z=True,
             ncol=37, dtype="f64", rc=2.0, sites=40),
        # H Y, Mp = Y'Y and Hp = Y'HY of the 216-atom cell (mixed precision)
        dict(name="project_216atoms_f32", kind="project", nx=78, ny=78, nz=78, h=0.3946, dirichlet_z=False,
             ncol=480, dtype="f32", rc=2.0, sites=216),
        # Psi = Y Q of the 216-atom cell (mixed precision)
        dict(name="rotate_216atoms_f32", kind="rotate", nx=78, ny=78, nz=78, h=0.3946, dirichlet_z=False,
             ncol=480, dtype="f32"),
        # the FP64 subspace eigensolve of the 216-atom cell
        dict(name="eigensolve_480", kind="eigensolve", n=480),
        # the Poisson problem of 216 Gaussian charges, Jacobi-AAR
        dict(name="poisson_128cubed", kind="poisson", nx=128, ny=128, nz=128, h=0.35, charges=216,
             learned=False),
        # a Poisson solve with the U-Net inside AAR (inference at every step)
        dict(name="poisson_unet_52cubed", kind="poisson", nx=52, ny=52, nz=52, h=0.3946, charges=64,
             learned=True),
        # Adam steps of the U-Net on harvested pairs: forward and backward
        dict(name="unet_train_52cubed", kind="train", nx=52, ny=52, nz=52, h=0.3946, charges=64, steps=8),
        # the first SCF iterations of the 64-atom cell, mixed precision
        dict(name="scf_64atoms_f32", kind="scf", ncell=2, n=52, nstates=160, iterations=3, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# values of one block of the largest listed filter, in FP32 words
_MOST = 96 ** 3 * 512


def draw(rng):
    kind = rng.choice(["filter", "filter", "filter", "filter", "hamiltonian", "hamiltonian", "project",
                       "project", "rotate", "eigensolve", "poisson", "train", "scf"])
    if kind == "eigensolve":
        return dict(kind=kind, n=_log_int(rng, 24, 480))
    if kind == "scf":
        if rng.random() < 0.5:
            return dict(kind=kind, ncell=1, n=rng.randint(24, 32), nstates=rng.randint(20, 32),
                        iterations=rng.randint(2, 5), dtype="f32")
        return dict(kind=kind, ncell=2, n=rng.randint(48, 56), nstates=rng.randint(150, 180),
                    iterations=rng.randint(2, 3), dtype="f32")
    h = round(rng.uniform(0.3, 0.42), 4)
    if kind == "poisson" or kind == "train":
        learned = kind == "poisson" and rng.random() < 0.4
        n = _log_int(rng, 26, 52 if kind == "train" or learned else 128)
        dims = [max(24, min(128, n + rng.randint(-2, 2))) for _ in range(3)]
        c = dict(kind=kind, nx=dims[0], ny=dims[1], nz=dims[2], h=h,
                 charges=max(4, int(dims[0] * dims[1] * dims[2] * h ** 3 / 135.0)))
        c.update(steps=rng.randint(2, 8)) if kind == "train" else c.update(learned=learned)
        return c
    dtype = rng.choice(["f32", "f32", "f64"])
    words = 1 if dtype == "f32" else 3  # FP64 moves twice the bytes at a lower product rate
    n = _log_int(rng, 22, 96 if kind in ("filter", "hamiltonian") else 78)
    dims = [max(20, min(100, n + rng.randint(-4, 4))) for _ in range(3)]
    nd = dims[0] * dims[1] * dims[2]
    most = (_MOST if kind in ("filter", "hamiltonian") else 78 ** 3 * 480) // words
    ncol = max(4, min(_log_int(rng, 8, 512 if kind in ("filter", "hamiltonian") else 480), most // nd))
    c = dict(kind=kind, nx=dims[0], ny=dims[1], nz=dims[2], h=h, dirichlet_z=rng.random() < 0.25, ncol=ncol,
             dtype=dtype)
    if kind == "rotate":
        return c
    vol = nd * h ** 3
    if rng.random() < 0.25:  # large, overlapping spheres
        c.update(rc=round(min(6.0, 0.4 * min(dims) * h), 3), sites=max(1, int(vol / 373.0)))
    else:
        c.update(rc=round(min(rng.uniform(1.6, 2.4), 0.4 * min(dims) * h), 3), sites=max(2, int(vol / 135.0)))
    if kind == "filter":
        c.update(degree=rng.randint(14, 24))
    return c


# ---------------------------------------------------------------- inputs


def _grid(c):
    return Grid(c["nx"], c["ny"], c["nz"], c["h"], c["h"], c["h"], bcz=1 if c.get("dirichlet_z") else 0,
                order=ORDER)


def _axis_gaussians(n, h, length, periodic, centre, width):
    d = np.arange(n)[None, :] * h - centre[:, None]
    if periodic:
        d -= length * np.round(d / length)
    return np.exp(-d * d / (2.0 * width[:, None] ** 2))


def _gaussians(g, amp, centre, width):
    """sum_i amp_i exp(-|r - c_i|^2 / 2 w_i^2) on the grid (x fastest, flat)."""
    ax = [_axis_gaussians(n, h, length, not bc, centre[:, k], width)
          for k, (n, h, length, bc) in enumerate(((g.nx, g.hx, g.lengths[0], g.bcx),
                                                  (g.ny, g.hy, g.lengths[1], g.bcy),
                                                  (g.nz, g.hz, g.lengths[2], g.bcz)))]
    zy = (amp[:, None] * ax[2])[:, :, None] * ax[1][:, None, :]
    return (zy.reshape(len(amp), -1).T @ ax[0]).ravel()


def _operator(c, seed):
    """Veff (attractive Gaussians, -2..0 Ha) and the projectors: atoms on
    displaced diamond sites where their number is a whole supercell's, else
    uniformly placed; 2 radial functions x l <= 1, 8 per atom."""
    g = _grid(c)
    rng = np.random.default_rng(seed)
    length = np.asarray(g.lengths)
    veff = _gaussians(g, rng.uniform(-2.0, 0.0, 16), rng.uniform(0, 1, (16, 3)) * length,
                      rng.uniform(1.0, 3.0, 16))
    ncell = round((c["sites"] / 8) ** (1 / 3))
    if 8 * ncell ** 3 == c["sites"] and c["rc"] <= 3.0:
        sites = diamond_cubic(ncell, CELL, 0.02, seed) / (CELL * ncell) % 1.0 * length
    else:
        sites = rng.uniform(0, 1, (c["sites"], 3)) * length
    s = c["rc"] / 4.0
    nl = gaussian_projectors(g, sites, c["rc"], sigmas=(s, s / 1.5), gammas=(1.0, -1.0), lmax=1)
    # bounds: kinetic maximum (all axes at the Nyquist wave number) with a
    # margin for the projectors; the lowest wanted level below Veff's depth
    top = 0.5 * sum(sum(abs(w) * (2 if k else 1) for k, w in enumerate(_weights(g.hx))) for _ in range(3))
    return g, veff, nl, float(veff.min()) - 2.0, top + 12.0


def _weights(h):
    """Second-derivative weights of order 12 at offsets 0..6."""
    n = ORDER // 2
    w = [0.0] * (n + 1)
    for p in range(1, n + 1):
        r = 1.0
        for k in range(1, p + 1):
            r *= (n - k + 1) / (n + k)
        w[p] = 2.0 * (-1) ** (p + 1) * r / p ** 2 / h ** 2
        w[0] -= 2.0 / p ** 2 / h ** 2
    return w


def _charges(c, seed):
    """4 pi (rho - mean) of normalised Gaussian charges of +4 (width 0.8-1.5 Bohr)."""
    g = _grid(c)
    rng = np.random.default_rng(seed)
    w = rng.uniform(0.8, 1.5, c["charges"])
    rho = _gaussians(g, 4.0 / ((2 * np.pi) ** 1.5 * w ** 3), rng.uniform(0, 1, (c["charges"], 3))
                     * np.asarray(g.lengths), w)
    return g, 4.0 * np.pi * (rho - rho.mean())


def _subspace(n, seed):
    """Hp, Mp of a filtered block: a well conditioned overlap and levels from
    the valence bottom to above the Fermi level."""
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    lam = np.sort(rng.uniform(-0.5, 1.0, n))
    t = q * np.exp(rng.uniform(-1.0, 1.0, n))  # Y = Psi t
    Mp, Hp = t.T @ t, (t.T * lam) @ t
    return 0.5 * (Hp + Hp.T), 0.5 * (Mp + Mp.T)


def _rotation(n, seed):
    q, r = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))
    return np.asfortranarray(q * np.sign(np.diag(r)))


# ---------------------------------------------------------------- state


class _Storage:
    """The storage of a device block for torch.as_tensor: the block's address
    is the last word of its handle, its columns are ld apart."""

    def __init__(self, block):
        self.block = block  # keeps the block and its context
        ptr = ctypes.c_uint64.from_address(block.h.value + 24).value
        size, kind = (4, "<f4") if block.dtype == gpu.F32 else (8, "<f8")
        ld = block.ctx.lib.sgpu_block_ld(block.h)
        self.__cuda_array_interface__ = {"shape": (block.ncol, block.ctx.nd), "typestr": kind,
                                         "data": (ptr, False), "strides": (ld * size, size), "version": 3}


def _tensor(block):
    """A block as an ncol x Nd tensor on the device, without a copy."""
    return torch.as_tensor(_Storage(block), device="cuda")


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind == "eigensolve":
        s["ctx"] = gpu.Context(Grid(24, 24, 24, 0.4, 0.4, 0.4))
        s["Hp"], s["Mp"] = _subspace(c["n"], seed)
        return s
    if kind == "scf":
        st, p = silicon(c["ncell"], c["n"], c["nstates"], seed=seed % (1 << 31))
        s["ctx"] = gpu.Context(st.grid)
        s["ctx"].set_nonlocal(st.nloc)
        s["system"] = st
        s["params"] = dict(p, max_scf=c["iterations"], min_scf=c["iterations"], dtype=_dtype(c))
        return s
    if kind in ("poisson", "train"):
        g, s["b"] = _charges(c, seed)
        s["ctx"] = gpu.Context(g)
        s["x0"] = np.zeros(g.nd)
        if kind == "train" or c["learned"]:
            s["net"] = s["ctx"].unet(seed=1)
            # a network near its initial state (the Jacobi preconditioner)
            w = s["net"].get_weights()
            rng = np.random.default_rng(seed + 1)
            s["weights"] = (w + 2e-4 * rng.standard_normal(w.size)).astype(np.float32)
            s["net"].set_weights(s["weights"])
        if kind == "train":
            s["net"].harvest(s["b"], s["x0"], tol=1e-8, max_iter=3000, stride=2, max_pairs=64)
        return s
    dt = _dtype(c)
    if kind == "rotate":
        s["ctx"] = gpu.Context(_grid(c))
        s["Q"] = _rotation(c["ncol"], seed)
    else:
        g, veff, nl, s["a0"], s["b"] = _operator(c, seed)
        s["a"] = s["a0"] + 0.08 * (s["b"] - s["a0"])
        s["ctx"] = gpu.Context(g)
        s["ctx"].set_veff(veff)
        s["ctx"].set_nonlocal(nl)
    s["X"] = s["ctx"].block(c["ncol"], dt).fill_uniform(seed + 1, -0.5, 0.5)
    s["Y"] = s["ctx"].block(c["ncol"], dt)
    if kind == "filter":
        s["psi"] = s["ctx"].block(c["ncol"], dt).copy_from(s["X"])
    return s


def _dtype(c):
    return gpu.F32 if c["dtype"] == "f32" else gpu.F64


def run(state):
    s, c = state, state["case"]
    ctx, kind = s["ctx"], c["kind"]
    if kind == "filter":
        # the filter overwrites its input, so the orbitals are copied in first
        s["X"].copy_from(s["psi"])
        ctx.chebyshev_filter_dev(s["X"], s["Y"], c["degree"], s["a"], s["b"], s["a0"])
        return {"filtered": _tensor(s["Y"]), "previous": _tensor(s["X"])}
    if kind == "hamiltonian":
        ctx.hamiltonian_dev(-0.2, s["X"], s["Y"])
        return _tensor(s["Y"])
    if kind == "project":
        Hp, Mp = ctx.project_dev(s["X"], s["Y"])
        return {"Hp": Hp, "Mp": Mp, "HY": _tensor(s["Y"])}
    if kind == "rotate":
        ctx.rotate_dev(s["X"], s["Q"], s["Y"])
        return _tensor(s["Y"])
    if kind == "eigensolve":
        lam, Q = ctx.DP_Solve_Generalized_EigenProblem(s["Hp"], s["Mp"])
        # an eigenvector's sign is arbitrary: the first component positive
        return {"lambda": lam, "Q": Q * np.where(Q[0] < 0, -1.0, 1.0)}
    if kind == "poisson":
        # taken far enough that the potential itself is settled to nine digits;
        # a periodic potential is fixed up to a constant: zero mean
        if c["learned"]:
            x = ctx.AAR_unet(s["net"], s["x0"], s["b"], tol=1e-11, max_iter=3000)[0]
        else:
            x = ctx.AAR(s["x0"], s["b"], tol=1e-11, max_iter=3000)[0]
        return x - x.mean()
    if kind == "train":
        s["net"].set_weights(s["weights"])
        loss = s["net"].train(c["steps"], batch=4, lr=2e-3, seed=7)
        # the losses are FP32 sums in FP64 words
        return {"weights": s["net"].get_weights(), "loss": loss.astype(np.float32)}
    r = ctx.scf_run(s["system"].b, s["system"].rho_at, s["params"], rho_core=s["system"].rho_core)
    # mixed precision: the orbitals, and what comes from them, hold 24 bits
    t = np.float32 if c["dtype"] == "f32" else np.float64
    return {k: np.asarray(r[k], t) for k in ("lambda_", "rho", "phi", "Etot")}


# ---------------------------------------------------------------- work


def work(case):
    """Bytes and operations of one pass.  An application reads its input (and
    the recurrence's second term) and writes its output once, with Veff and
    the projector values once; a filter is `degree` of them, its blocks being
    far larger than what the chip holds."""
    c, kind = case, case["kind"]
    if kind == "eigensolve":
        # Cholesky, reduction, tridiagonalisation, back-transformations
        return {"bytes": 8.0 * 3 * c["n"] ** 2, "flops": (1 / 3 + 2 + 4 / 3 + 2 + 1 + 2) * c["n"] ** 3}
    if kind == "scf":
        nd, ns, atoms = c["n"] ** 3, c["nstates"], 8 * c["ncell"] ** 3
        chi = atoms * 8 * 4.19 * 1.9 ** 3 / (CELL * c["ncell"] / c["n"]) ** 3
        passes, size = c["iterations"] + 3, 4 if c["dtype"] == "f32" else 8
        b = passes * (size * nd * ns * (2 + 3 * 19 + 6) + 20 * size * (nd + 2 * chi))
        return {"bytes": b, "flops": passes * ns * (21 * (75.0 * nd + 4 * chi) + 6.0 * nd * ns)}
    nd = c["nx"] * c["ny"] * c["nz"]
    if kind == "poisson":
        # a 1e-11 solve takes some hundred iterations; per iteration the
        # residual and the update: x, b, r and the history once each
        it = 500
        net = 16 * (nd / 8) * (2 * 27 * 16 * 2) * 1.6 if c["learned"] else 0.0
        return {"bytes": it * 8.0 * nd * 6, "flops": it * (75.0 * nd + net)}
    if kind == "train":
        fwd = 27 * 2.0 * 16 * (nd / 8) * (1 + 16 * 3 + 16 * 3 / 8 + 8)
        return {"bytes": c["steps"] * 4 * 2 * 4.0 * nd, "flops": c["steps"] * 4 * 3 * fwd}
    ns, size = c["ncol"], 4 if c["dtype"] == "f32" else 8
    if kind == "rotate":
        return {"bytes": 2.0 * size * nd * ns, "flops": 2.0 * nd * ns * ns}
    chi = 8.0 * c["sites"] * 4.18879 * c["rc"] ** 3 / c["h"] ** 3
    m = c["degree"] if kind == "filter" else 1
    w = {"bytes": size * (nd * ns * (2.0 + 3 * (m - 1)) + m * (nd + chi)),
         "flops": m * ns * (75.0 * nd + 4 * chi)}
    if kind == "project":
        w["flops"] += 4.0 * nd * ns * ns
    return w


# ---------------------------------------------------------------- 64 bits


def _uniform(nd, ncol, seed, lo, hi):
    """The counter-based uniform values of a block fill, ncol x nd."""
    def mix(z):
        shr = lambda v, k: (v >> k) & ((1 << (64 - k)) - 1)  # noqa: E731
        z = z + torch.tensor(0x9E3779B97F4A7C15 - (1 << 64), device="cuda")
        z = (z ^ shr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
        z = (z ^ shr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
        return z ^ shr(z, 31)

    out = torch.empty(ncol, nd, dtype=torch.float64, device="cuda")
    for c0 in range(0, ncol, 64):
        c1 = min(ncol, c0 + 64)
        r = mix(mix(torch.arange(c0 * nd, c1 * nd, device="cuda")) ^ int(seed))
        out[c0:c1] = (((r >> 11) & ((1 << 53) - 1)).double() / 9007199254740992.0).view(c1 - c0, nd)
    return lo + (hi - lo) * out


def _second_derivative(n, h, periodic):
    w, d = _weights(h), torch.zeros(n, n, dtype=torch.float64)
    for i in range(n):
        for k in range(-(ORDER // 2), ORDER // 2 + 1):
            if periodic:
                d[i, (i + k) % n] += w[abs(k)]
            elif 0 <= i + k < n:
                d[i, i + k] += w[abs(k)]
    return d.cuda()


class _Hamiltonian:
    """-1/2 Lap + Veff + sum Chi Gamma Chi' dV on ncol x nd blocks."""

    def __init__(self, g, veff, nl):
        self.shape = (g.nz, g.ny, g.nx)
        self.d = [_second_derivative(n, h, not bc) for n, h, bc in
                  ((g.nx, g.hx, g.bcx), (g.ny, g.hy, g.bcy), (g.nz, g.hz, g.bcz))]
        self.v = torch.from_numpy(np.ascontiguousarray(veff)).cuda()
        p = torch.zeros(g.nd, nl.n_alpha, dtype=torch.float64, device="cuda")
        for k in range(nl.n_influence):
            n, q = int(nl.ndc[k]), int(nl.nproj[k])
            at = torch.from_numpy(nl.grid_pos[nl.pos_off[k]:nl.pos_off[k] + n].astype(np.int64)).cuda()
            chi = torch.from_numpy(nl.chi[nl.chi_off[k]:nl.chi_off[k] + n * q].reshape(q, n).T.copy()).cuda()
            a0 = int(nl.alpha_off[k])
            p[at, a0:a0 + q] += chi
        self.p, self.pt = p, p.t().contiguous()
        self.gamma = torch.from_numpy(nl.gamma).cuda() * nl.dV

    def __call__(self, x):
        nz, ny, nx = self.shape
        n = x.shape[0]
        y = ((x @ self.p) * self.gamma) @ self.pt + self.v * x
        lap = (x.view(-1, nx) @ self.d[0]).view(n, nz, ny, nx)
        xz = x.view(n, nz, ny * nx)
        for k in range(n):
            lap[k] += (self.d[2] @ xz[k]).view(nz, ny, nx)
        lap += torch.matmul(self.d[1], x.view(n, nz, ny, nx))
        return y - 0.5 * lap.view(n, -1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("scf", "train"):
        return None
    if kind == "eigensolve":
        Hp, Mp = (torch.from_numpy(a) for a in _subspace(c["n"], seed))
        low = torch.linalg.cholesky(Mp)
        inv = torch.linalg.solve_triangular(low, torch.eye(c["n"], dtype=torch.float64), upper=False)
        m = inv @ Hp @ inv.T
        lam, z = torch.linalg.eigh(0.5 * (m + m.T))
        q = inv.T @ z
        return {"lambda": lam, "Q": q * torch.where(q[0] < 0, -1.0, 1.0)}
    if kind == "poisson":
        g, b = _charges(c, seed)
        sym = 0.0
        for k, (n, h) in enumerate(((g.nz, g.hz), (g.ny, g.hy), (g.nx, g.hx))):
            t = 2 * np.pi * np.arange(n) / n
            w = _weights(h)
            line = w[0] + 2 * sum(w[p] * np.cos(p * t) for p in range(1, ORDER // 2 + 1))
            sym = sym + line.reshape([-1 if j == k else 1 for j in range(3)])
        sym[0, 0, 0] = 1.0
        f = np.fft.fftn(b.reshape(g.nz, g.ny, g.nx)) / -sym
        f[0, 0, 0] = 0.0
        return np.ascontiguousarray(np.fft.ifftn(f).real.ravel())
    nd = c["nx"] * c["ny"] * c["nz"]
    x = _uniform(nd, c["ncol"], seed + 1, -0.5, 0.5)
    if c["dtype"] == "f32":
        x = x.float().double()
    if kind == "rotate":
        q = torch.from_numpy(_rotation(c["ncol"], seed)).cuda()
        return q.t().contiguous() @ x
    g, veff, nl, a0, b = _operator(c, seed)
    ham = _Hamiltonian(g, veff, nl)
    if kind == "hamiltonian":
        return ham(x) - 0.2 * x
    if kind == "project":
        hy = ham(x)
        xt = x.t().contiguous()
        hp = x @ hy.t().contiguous()
        return {"Hp": (0.5 * (hp + hp.t())).cpu(), "Mp": (x @ xt).cpu(), "HY": hy}
    a = a0 + 0.08 * (b - a0)
    e, mid = 0.5 * (b - a), 0.5 * (b + a)
    sigma = e / (a0 - mid)
    gamma = 2.0 / sigma
    y = (ham(x) - mid * x) * (sigma / e)
    for _ in range(1, c["degree"]):
        sigma2 = 1.0 / (gamma - sigma)
        x, y = y, (ham(y) - mid * y) * (2.0 * sigma2 / e) - (sigma * sigma2) * x
        sigma = sigma2
    return {"filtered": y, "previous": x}
