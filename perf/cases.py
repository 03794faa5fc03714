"""Cases for measuring the Kohn-Sham path on one GPU through the package's public entry points.

A case names a crystal, a cutoff, a grid, a number of bands, a precision and what is done with
them: op_H on one k-point, op_H on every k-point at once, calc_rhoe, a block of LOBPCG
iterations followed by the density (one SCF step on one k-point or on all of them), the
pseudopotential forces, or whole SCF iterations.  The crystals are the ones of the benchmark
and the tests (diamond Si cells and supercells, fcc Al), with non-cubic supercells, odd band
counts and other cutoffs drawn beside them.

The Hamiltonian (grid, projectors, potential) is what a program keeps over many calls, so it is
made once per system here; the wave functions and densities come from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pwdft.jl_amd"))

import pwdft_hip as ph  # noqa: E402

A_SI, A_AL = 10.2631, 7.6  # bohr, conventional cells
Z_VAL = {"Si": 4, "Al": 3}
PSP = {"Si": "Si-q4.lda.gth", "Al": "Al-q3.lda.gth"}

BASE = {"cell": "sc", "atom": "Si", "r1": 1, "r2": 1, "r3": 1, "ecut": 15.0, "grid": 0, "mesh": 1, "shift": 0,
        "symmetry": False, "mixed": False, "iters": 0}


def _case(**kw):
    return dict(BASE, **kw)


def listed():
    return [
        # one k-point of the two-atom Si cell: the smallest op_H a solver calls, all latency
        _case(name="op_H Si2 fp64", do="op_H", cell="fcc", mesh=3, symmetry=True, nb=8),
        # an ordinary cell at a denser cutoff, mixed precision
        _case(name="op_H Si8 mixed", do="op_H", ecut=20.0, nb=20, mixed=True),
        # the benchmark's supercell: 64 atoms, 72^3 grid, 160 bands, both precisions
        _case(name="op_H Si64 fp64", do="op_H", r1=2, r2=2, r3=2, grid=72, nb=160),
        _case(name="op_H Si64 mixed", do="op_H", r1=2, r2=2, r3=2, grid=72, nb=160, mixed=True),
        # the largest op_H: twice the cutoff (108^3 grid) and an odd number of bands
        _case(name="op_H Si64 30Ha mixed", do="op_H", r1=2, r2=2, r3=2, ecut=30.0, nb=243, mixed=True),
        # metals: many small k-points, every band of every k-point in one call
        _case(name="op_H Al 182k mixed", do="op_H_batch", cell="fcc", atom="Al", mesh=12, shift=1, symmetry=True, nb=8,
              mixed=True),
        # density of the benchmark's supercell
        _case(name="rhoe Si64 fp64", do="rhoe", r1=2, r2=2, r3=2, grid=72, nb=160),
        # density over the k-points of a non-cubic supercell (another length per axis), odd bands
        _case(name="rhoe Si16 8k mixed", do="rhoe", r1=2, mesh=2, nb=37, mixed=True),
        # one SCF step on a large cell: block eigensolver iterations, then the density
        _case(name="lobpcg Si64 fp64", do="lobpcg", r1=2, r2=2, r3=2, grid=72, nb=160, iters=3),
        # one SCF step on a metal: every k-point's eigensolver together, then the density
        _case(name="lobpcg Al 182k fp64", do="lobpcg_batch", cell="fcc", atom="Al", mesh=12, shift=1, symmetry=True,
              nb=8, iters=4),
        # forces of the displaced eight-atom cell, as after each geometry step
        _case(name="forces Si8 8k fp64", do="forces", ecut=20.0, mesh=2, nb=20),
        # whole SCF iterations on the two-atom cell: solver, density, mixing, potential, energies
        _case(name="scf Si2 fp64", do="scf", cell="fcc", mesh=3, symmetry=True, nb=8, iters=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["op_H", "op_H", "op_H", "op_H", "op_H_batch", "rhoe", "rhoe", "lobpcg", "lobpcg_batch", "forces", "scf"])
    c = _case(do=do, ecut=round(math.exp(rng.uniform(math.log(8.0), math.log(30.0))), 2))
    if do in ("op_H_batch", "lobpcg_batch"):
        c.update(cell="fcc", atom=rng.choice(["Al", "Si"]), mesh=rng.randint(4, 12), shift=1, symmetry=True,
                 ecut=round(rng.uniform(10.0, 18.0), 2))
        c.update(nb=rng.randint(4, 12), mixed=do == "op_H_batch" and rng.random() < 0.5)
        c.update(iters=rng.randint(2, 4) if do == "lobpcg_batch" else 0)
        return c
    if do == "scf":
        c.update(cell="fcc", mesh=rng.randint(2, 4), symmetry=True, nb=rng.randint(5, 10), iters=3)
        return c
    if do == "forces":
        c.update(r1=rng.randint(1, 2), mesh=rng.randint(1, 2))
    else:
        c.update(r1=rng.randint(1, 2), r2=rng.randint(1, 2), r3=rng.randint(1, 2))
        if do == "rhoe" and c["r2"] * c["r3"] == 1:
            c.update(mesh=rng.randint(1, 2))
    occupied = 16 * c["r1"] * c["r2"] * c["r3"]
    if do == "op_H":
        c.update(nb=_log_int(rng, 3, 243))
    elif do == "lobpcg":
        c.update(ecut=round(rng.uniform(8.0, 15.0), 2), nb=occupied + rng.randint(1, 25), iters=rng.randint(2, 3))
    else:
        c.update(nb=occupied + rng.randint(0, 25))
    # LOBPCG, forces and SCF return what FP64 fixes; the products run in either precision
    c.update(mixed=do in ("op_H", "rhoe") and rng.random() < 0.5)
    return c


# ------------------------------------------------------------------------------- the systems

_KEPT = {}


def _system(case):
    """The Hamiltonian of a case: kept for the next call on the same system (the two last used)."""
    key = tuple(case[k] for k in ("cell", "atom", "r1", "r2", "r3", "ecut", "grid", "mesh", "shift", "symmetry",
                                  "mixed")) + (case["nb"] if case["do"] != "op_H" else 0,)
    if key in _KEPT:
        _KEPT[key] = _KEPT.pop(key)
        return _KEPT[key]
    while len(_KEPT) >= 2:
        _KEPT.pop(next(iter(_KEPT)))
    reps = np.array([case["r1"], case["r2"], case["r3"]])
    if case["cell"] == "fcc":
        L = ph.gen_lattice_fcc(A_SI if case["atom"] == "Si" else A_AL)
        frac = [[0.0, 0.0, 0.0], [0.25, 0.25, 0.25]] if case["atom"] == "Si" else [[0.0, 0.0, 0.0]]
    else:
        L = A_SI * np.diag(reps.astype(float))
        base = ph.diamond_supercell(1.0, 1)
        cells = [(i, j, k) for i in range(reps[0]) for j in range(reps[1]) for k in range(reps[2])]
        frac = np.array([(b + np.array(s)) / reps for s in cells for b in base])
        # atoms off their ideal places, as in a relaxation (fixed for the system)
        frac = frac + np.linalg.solve(L, np.random.default_rng(64).uniform(-0.05, 0.05, (3, len(frac)))).T
    atoms = ph.Atoms([case["atom"]] * len(frac), frac, L)
    n = case["grid"]
    H = ph.Hamiltonian(atoms, [PSP[case["atom"]]], case["ecut"], meshk=(case["mesh"],) * 3,
                       shiftk=(case["shift"],) * 3, Ns_=(n, n, n) if n else None,
                       Nstates=case["nb"] if case["do"] != "op_H" else None,
                       use_symmetry=case["symmetry"], mixed=case["mixed"], band_batch=256)
    H.update(_density(H, 1.0))
    _KEPT[key] = H
    return H


def _density(H, depth):
    """A smooth positive density of the right charge: a constant and a few long waves."""
    n1, n2, n3 = H.pw.Ns
    x = [np.cos(2 * math.pi * np.arange(n) / n) for n in (n1, n2, n3)]
    w = x[2][:, None, None] + 0.7 * x[1][None, :, None] + 0.4 * x[0][None, None, :]
    w = 1.0 + 0.3 * depth * w / 2.1
    return (H.electrons.Nelectrons / H.pw.CellVolume * w / w.mean()).reshape(-1)


class _Block(ph.DeviceMatrix):
    """A column-major block in memory that a torch tensor owns (cols x rows, row-major)."""

    def __init__(self, ctx, t):
        import ctypes
        self.ctx, self.t = ctx, t
        self.cols, self.rows = t.shape
        self.p = ctypes.c_void_p(t.data_ptr())

    def free(self):
        self.t = self.p = None


class _Field(ph.DeviceVector):
    """A grid field in memory that a torch tensor owns."""

    def __init__(self, ctx, t):
        import ctypes
        self.ctx, self.t, self.n = ctx, t, t.numel()
        self.p = ctypes.c_void_p(t.data_ptr())

    def free(self):
        self.t = self.p = None


def _ks(case, H):
    """The k-points a case works on (op_H: one that is not Gamma where there is one)."""
    return [min(1, H.pw.Nkpt - 1)] if case["do"] in ("op_H", "lobpcg") else list(range(H.pw.Nkpt))


def _psi(H, ks, nb, seed):
    """Orthonormal random blocks of the k-points, one tensor of nb x Ngw each, in one buffer."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    sizes = [nb * int(H.pw.Ngw[ik]) for ik in ks]
    flat = torch.empty(sum(sizes), dtype=torch.complex128, device="cuda")
    out, at = [], 0
    for ik, n in zip(ks, sizes):
        a = torch.randn(nb, n // nb, 2, dtype=torch.float64, device="cuda", generator=g)
        a = torch.view_as_complex(a)
        S = (a.conj() @ a.T).cpu().numpy()            # S[i, j] = <a_i, a_j>
        w, U = np.linalg.eigh(S)
        M = torch.from_numpy((U / np.sqrt(w)) @ U.conj().T).to("cuda")
        t = flat[at:at + n].view(nb, n // nb)
        t.copy_(M.T @ a)
        out.append(t)
        at += n
    return flat, out


def prepare(case, seed):
    H = _system(case)
    ks = _ks(case, H)
    flat, psi = _psi(H, ks, case["nb"], seed)
    s = {"case": case, "H": H, "ks": ks, "flat": flat, "psi_t": psi, "psi": [_Block(H.ctx, t) for t in psi]}
    if case["do"] in ("op_H", "op_H_batch"):
        s["out_flat"] = torch.zeros_like(flat)
        at, s["out"] = 0, []
        for t in psi:
            s["out"].append(_Block(H.ctx, s["out_flat"][at:at + t.numel()].view(t.shape)))
            at += t.numel()
    if case["do"] in ("lobpcg", "lobpcg_batch", "scf"):
        s["work"] = _Block(H.ctx, torch.zeros(1, flat.numel(), dtype=torch.complex128, device="cuda"))
        s["start"] = _Block(H.ctx, flat.view(1, -1))
        at, s["X"] = 0, []
        for t in psi:
            s["X"].append(_Block(H.ctx, s["work"].t.view(-1)[at:at + t.numel()].view(t.shape)))
            at += t.numel()
    if case["do"] in ("rhoe", "lobpcg", "lobpcg_batch"):
        s["rho"] = _Field(H.ctx, torch.zeros(H.pw.Npoints, dtype=torch.float64, device="cuda"))
    if case["do"] == "forces":
        s["rho_host"] = _density(H, 0.5 + (seed % 97) / 97.0)
    torch.cuda.synchronize()
    return s


def _restart(s):
    """The solver overwrites its block: start from the prepared one."""
    s["H"].ctx.call("pw_memcpy_d2d", s["work"].p, s["start"].p, 16 * s["flat"].numel())


def run(s):
    case, H = s["case"], s["H"]
    do = case["do"]
    if do == "op_H":
        H.ik = s["ks"][0]
        ph.op_H_(H, s["psi"][0], s["out"][0])
        return s["out_flat"]
    if do == "op_H_batch":
        ph.op_H_batch(H, s["psi"], out=s["out"])
        return s["out_flat"]
    if do == "rhoe":
        ph.calc_rhoe_(H, s["psi"], s["rho"])
        return s["rho"].t
    if do == "lobpcg":
        _restart(s)
        H.ik = s["ks"][0]
        ev, _ = ph.diag_LOBPCG_(H, s["X"][0], tol=0.0, NiterMax=case["iters"])
        ph.calc_rhoe_(H, s["X"], s["rho"])
        return {"evals": ev, "rho": s["rho"].t}
    if do == "lobpcg_batch":
        _restart(s)
        ev, _ = ph.diag_LOBPCG_batch(H, s["X"], tol=0.0, NiterMax=case["iters"])
        ph.calc_rhoe_(H, s["X"], s["rho"])
        return {"evals": ev, "rho": s["rho"].t}
    if do == "forces":
        return {"loc": ph.calc_forces_Ps_loc(H, s["rho_host"]), "nloc": ph.calc_forces_Ps_nloc(H, s["psi"])}
    _restart(s)
    r = ph.KS_solve_SCF_(H, psiks=s["X"], NiterMax=case["iters"], etot_conv_thr=0.0)
    return {"energies": r["energies"], "evals": r["evals"], "rho": r["rho"]}


# ------------------------------------------------------------------------------- what it costs

def _op_cost(N, ngw, nbeta, nb):
    """One op_H: every coefficient in and out, the projectors and the potential once; the two
    projector products and the two transforms, of which a sphere of half the grid's radius
    needs pi/16 of the z lines, half of the y lines and every x line."""
    fft = 2 * nb * 5 * N * math.log2(max(N, 2)) / 3 * (math.pi / 16 + 0.5 + 1.0)
    return 32.0 * ngw * nb + 16.0 * ngw * nbeta + 8.0 * N, 16.0 * nbeta * ngw * nb + fft + 2.0 * N * nb


def work(case):
    # sizes from the cutoff alone: sphere and grid of a cell of volume V
    reps = case["r1"] * case["r2"] * case["r3"]
    V = (A_SI if case["atom"] == "Si" else A_AL) ** 3 * (0.25 if case["cell"] == "fcc" else reps)
    atoms = {"fcc": 2 if case["atom"] == "Si" else 1, "sc": 8 * reps}[case["cell"]]
    kmax = math.sqrt(2 * case["ecut"])
    ngw = V * kmax ** 3 / (6 * math.pi ** 2)
    N = float(case["grid"] ** 3) if case["grid"] else V * (2 * kmax / math.pi) ** 3
    nb, nbeta, it = case["nb"], 5 * atoms, case["iters"]
    nk = {1: 1}.get(case["mesh"], max(1.0, case["mesh"] ** 3 / (9.5 if case["symmetry"] else 1)))
    if case["do"] in ("op_H", "lobpcg"):
        nk = 1
    b, f = _op_cost(N, ngw, nbeta, nb)
    rho_b, rho_f = 16.0 * ngw * nb + 8.0 * N, nb * 5 * N * math.log2(max(N, 2)) / 3 * (math.pi / 16 + 0.5 + 1) + 3 * N * nb
    # one LOBPCG iteration: op_H, the Gram products (7 blocks of W'W, P'P, Q'Q, Q'HQ beyond the
    # known ones) and the updates of X, HX, P, HP, and the eigenproblem of order 3 nb
    lob_f = f + 8.0 * ngw * nb * nb * (14 + 10) + 4 * 9.0 * (3 * nb) ** 3
    lob_b = b + 16.0 * ngw * nb * 12
    if case["do"] in ("op_H", "op_H_batch"):
        return {"bytes": nk * b, "flops": nk * f}
    if case["do"] == "rhoe":
        return {"bytes": nk * rho_b, "flops": nk * rho_f}
    if case["do"] == "forces":
        return {"bytes": nk * (16.0 * ngw * (nb + nbeta)) + 16.0 * N, "flops": nk * 32.0 * nbeta * ngw * nb + 40.0 * N}
    if case["do"] == "scf":
        return {"bytes": it * nk * (4 * lob_b + rho_b), "flops": it * nk * (4 * lob_f + rho_f)}
    return {"bytes": nk * (it * lob_b + rho_b), "flops": nk * (it * lob_f + rho_f)}


# ------------------------------------------------------------------------------- in 64 bits

def _gth(H, ik):
    """beta (Ngw x Nproj) and D of the GTH projectors s1, s2 and p1 of every atom, from the
    parameters of the pseudopotential file (Goedecker, Teter, Hutter 1996)."""
    psp, at = H.pspots[0], H.atoms
    g = torch.from_numpy(np.ascontiguousarray(H.pw.gk(ik))).to("cuda")
    tau = torch.from_numpy(np.ascontiguousarray(at.positions)).to("cuda")
    q = g.pow(2).sum(0).sqrt()
    ph_ = torch.polar(torch.ones(1, dtype=torch.float64, device="cuda"), -(g.T @ tau))    # Ngw x Natoms
    r0, r1, vol = float(psp.rc[0]), float(psp.rc[1]), H.pw.CellVolume
    x0, x1 = (q * r0) ** 2, (q * r1) ** 2
    y00, y1 = 0.5 / math.sqrt(math.pi), 0.5 * math.sqrt(3.0 / math.pi)
    s = 4 * math.pi ** 1.25 * math.sqrt(2.0 * r0 ** 3 / vol) * torch.exp(-0.5 * x0) * y00
    p = 4 * math.pi ** 1.25 * math.sqrt(4.0 * r1 ** 5 / vol) * torch.exp(-0.5 * x1) * y1 / math.sqrt(3.0)
    radial = torch.stack([s, s * 2.0 / math.sqrt(15.0) * (3.0 - x0), p * g[0], p * g[1], p * g[2]])
    beta = (radial.T[:, None, :] * ph_[:, :, None]).reshape(len(q), -1)
    D = np.zeros((5, 5))
    D[:2, :2] = psp.h[0][:2, :2]
    D[2, 2] = D[3, 3] = D[4, 4] = psp.h[1][0, 0]
    return g, beta, torch.from_numpy(np.kron(np.eye(at.Natoms), D)).to("cuda").to(torch.complex128)


def _to_grid(H, ik, psi):
    n1, n2, n3 = H.pw.Ns
    idx = torch.from_numpy(np.ascontiguousarray(H.pw.idx_gw2r[ik])).to("cuda")
    f = torch.zeros(psi.shape[0], n1 * n2 * n3, dtype=torch.complex128, device="cuda")
    f[:, idx] = psi
    return idx, torch.fft.ifftn(f.view(-1, n3, n2, n1), dim=(1, 2, 3))


def _exact_op_H(H, ik, psi):
    n1, n2, n3 = H.pw.Ns
    V = torch.from_numpy(np.ascontiguousarray(H.potentials.Total[:, 0])).to("cuda").view(n3, n2, n1)
    g, beta, D = _gth(H, ik)
    out = 0.5 * g.pow(2).sum(0) * psi + ((psi @ beta.conj()) @ D) @ beta.T
    for b in range(0, psi.shape[0], 16):
        idx, f = _to_grid(H, ik, psi[b:b + 16])
        out[b:b + 16] += torch.fft.fftn(f * V, dim=(1, 2, 3)).reshape(f.shape[0], -1)[:, idx]
    return out


def exact(case, seed):
    if case["do"] in ("lobpcg", "lobpcg_batch", "scf"):
        return None
    s = prepare(case, seed)
    H = s["H"]
    if case["do"] in ("op_H", "op_H_batch"):
        return torch.cat([_exact_op_H(H, ik, t).reshape(-1) for ik, t in zip(s["ks"], s["psi_t"])])
    if case["do"] == "rhoe":
        N = H.pw.Npoints
        rho = torch.zeros(N, dtype=torch.float64, device="cuda")
        for ik, t in zip(s["ks"], s["psi_t"]):
            w = torch.from_numpy(H.pw.wk[ik] * H.electrons.Focc[:, ik]).to("cuda")
            for b in range(0, t.shape[0], 16):
                f = _to_grid(H, ik, t[b:b + 16])[1].reshape(-1, N)
                rho += (w[b:b + 16, None] * (f.real ** 2 + f.imag ** 2)).sum(0)
        return rho * (float(N) ** 2 / H.pw.CellVolume)
    # forces: the gradients of the local energy by the structure factor and of the nonlocal one
    n1, n2, n3 = H.pw.Ns
    psp, at = H.pspots[0], H.atoms
    rho = torch.from_numpy(s["rho_host"]).to("cuda").view(n3, n2, n1).to(torch.complex128)
    rg = torch.fft.fftn(rho).reshape(-1)[torch.from_numpy(np.ascontiguousarray(H.pw.idx_g2r)).to("cuda")] / H.pw.Npoints
    G = torch.from_numpy(np.ascontiguousarray(H.pw.G)).to("cuda")[:, 1:]
    tau = torch.from_numpy(np.ascontiguousarray(at.positions)).to("cuda")
    G2 = G.pow(2).sum(0)
    rl, c = psp.rlocal, psp.c
    x = G2 * rl * rl
    v = torch.exp(-0.5 * x) * (-4 * math.pi * psp.zval / G2 + math.sqrt(8 * math.pi ** 3) * rl ** 3 * (
        c[0] + c[1] * (3 - x) + c[2] * (15 - 10 * x + x ** 2) + c[3] * (105 - 105 * x + 21 * x ** 2 - x ** 3)))
    S = torch.polar(torch.ones(1, dtype=torch.float64, device="cuda"), -(G.T @ tau))
    loc = (G.to(torch.complex128) @ ((1j * v * rg[1:].conj())[:, None] * S)).real
    nloc = torch.zeros(3, at.Natoms, dtype=torch.float64, device="cuda")
    for ik, t in zip(s["ks"], s["psi_t"]):
        g, beta, D = _gth(H, ik)
        w = torch.from_numpy(2.0 * H.pw.wk[ik] * H.electrons.Focc[:, ik]).to("cuda")
        bp = (t @ beta.conj()) @ D                                    # nb x Nproj
        for d in range(3):
            db = t @ (1j * g[d][:, None] * beta).conj()
            nloc[d] += (w[:, None] * (bp.conj() * db).real).view(-1, at.Natoms, 5).sum((0, 2))
    return {"loc": loc, "nloc": nloc}
