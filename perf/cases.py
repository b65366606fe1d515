"""Performance cases: the work a plane-wave code hands to this library, through its public entry points.

Kinds of case (the "kind" entry):
  apply   H.psi of a block resident in device memory (Hamiltonian.apply_dev): what an eigensolver
          calls once per iteration and k-point, from one vector to a full block of bands
  host    H.psi of a block in host memory (Hamiltonian.apply): the operator callback of a solver that
          keeps its vectors on the host
  set     H.psi of all k-points of a small metallic cell in one call (HamSet.apply_dev)
  heev    the dense subspace eigenproblem of a block Davidson step (Context.heev_dev)
  solve   lowest bands of one k-point, then their density (eig_solve, density_solution): one k-point
          of one SCF iteration (the density only of tightly converged bands: at a loose tolerance it
          holds the tolerance's own error)
  xc      V_Hartree + V_xc of a density (ScfGrid.init_rho, read): the grid part of an SCF iteration

Cells are orthorhombic, atoms displaced at random from a lattice, with the s and p Gaussian projectors
and the Gaussian-screened ionic potential of the SCF systems in dzhip/scf.py.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dft-zig_amd"))

import dzhip  # noqa: E402
from dzhip import tables  # noqa: E402

SI_A = 5.431 * tables.ANGSTROM_TO_BOHR
GAAS_A = 5.653 * tables.ANGSTROM_TO_BOHR
AL_A = 4.05 * tables.ANGSTROM_TO_BOHR

# Projector radii (bohr) and strengths (Ry), valence charge and local radius of the pseudo-atom.
R_S, R_P, D_S, D_P = 0.422738, 0.484278, 11.853856, -0.6
Z_ION, R_LOC, C1 = 4.0, 0.44, -7.336103
DIAMOND = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0],
                    [.25, .25, .25], [.25, .75, .75], [.75, .25, .75], [.75, .75, .25]])


def listed():
    return [
        # One band at a time, as a conjugate-gradient solver applies H: launches and latency only.
        _hpsi("apply", "apply_si8_vector", (SI_A,) * 3, 8, 20.0, (0.25, 0.25, 0.25), 1, "fp64"),
        # The 8-atom cell's block through the host callback.
        _hpsi("host", "host_si8", (SI_A,) * 3, 8, 20.0, (0.25, 0.25, 0.25), 20, "fp64"),
        # A ragged cell: three different grid lengths, an odd number of bands.
        _hpsi("apply", "apply_slab", (11.3, 17.1, 20.5), 28, 25.0, (0.0, 0.5, 0.25), 37, "fp64"),
        # One k-point of the 64-atom Si supercell in both precisions of the SCF (FP32 in the early
        # iterations of a mixed-precision solve).
        _hpsi("apply", "apply_si64", (2 * SI_A,) * 3, 64, 30.0, (0.5, 0.5, 0.5), 160, "fp64"),
        _hpsi("apply", "apply_si64_fp32", (2 * SI_A,) * 3, 64, 30.0, (0.5, 0.5, 0.5), 160, "fp32"),
        # The 64-atom GaAs supercell at Gamma, the largest grid.
        _hpsi("apply", "apply_gaas64", (2 * GAAS_A,) * 3, 64, 35.0, (0.0, 0.0, 0.0), 160, "fp64"),
        # fcc Al: many k-points of a small cell.
        {"name": "set_al4", "kind": "set", "lx": AL_A, "ly": AL_A, "lz": AL_A, "atoms": 4, "ecut": 30.0, "mesh": 4,
         "bands": 12, "precision": "fp64"},
        # The first Rayleigh-Ritz problem of a 160-band solve, and one on its full subspace.
        {"name": "heev_164", "kind": "heev", "m": 164, "nev": 160},
        {"name": "heev_648", "kind": "heev", "m": 648, "nev": 160},
        # Whole solves: tightly converged bands of the small cell from a random start, with their
        # density; the bands of the large one from plane waves, as its first SCF step asks for them.
        {**_hpsi("solve", "solve_si8", (SI_A,) * 3, 8, 20.0, (0.25, 0.25, 0.25), 20, "fp64"), "tol": 1e-10, "plane_waves": False,
         "density": True},
        {**_hpsi("solve", "solve_si64", (2 * SI_A,) * 3, 64, 30.0, (0.5, 0.5, 0.5), 160, "fp64"), "tol": 1e-5, "plane_waves": True,
         "density": False},
        # The gradient-corrected potential of the Al cell's grid.
        {"name": "xc_al4_pbe", "kind": "xc", "nx": 30, "ny": 30, "nz": 30, "xc": "pbe"},
    ]


def _hpsi(kind, name, cell, atoms, ecut, k, bands, precision):
    return {"name": name, "kind": kind, "lx": cell[0], "ly": cell[1], "lz": cell[2], "atoms": atoms, "ecut": ecut,
            "kx": k[0], "ky": k[1], "kz": k[2], "bands": bands, "precision": precision}


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "host", "set", "heev", "heev", "solve", "xc"])
    if kind == "heev":
        m = round(_log(rng, 24, 760))
        return {"kind": kind, "m": m, "nev": max(1, min(m, round(m * rng.uniform(0.2, 1.0)), 200))}
    if kind == "xc":
        n = [rng.choice([24, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75]) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "xc": rng.choice(["pbe", "lda_pz"])}
    if kind == "set":
        a = rng.uniform(7.0, 8.5)
        return {"kind": kind, "lx": a, "ly": a * rng.uniform(0.95, 1.1), "lz": a * rng.uniform(0.95, 1.1), "atoms": 4,
                "ecut": rng.uniform(18.0, 32.0), "mesh": rng.choice([2, 3, 4]), "bands": rng.randint(6, 24),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "solve":  # the small cell under strain: an insulator, so that its density is defined
        cell = [SI_A * rng.uniform(0.96, 1.04) for _ in range(3)]
    else:
        cell = [_log(rng, 7.5, 16.0 if kind == "host" else 21.0) for _ in range(3)]
    volume = cell[0] * cell[1] * cell[2]
    atoms = 8 if kind == "solve" else max(2, min(64, round(volume / 135.0)))
    k = [rng.choice([0.0, 0.25, 0.5, round(rng.uniform(-0.5, 0.5), 3)]) for _ in range(3)]
    ecut = rng.uniform(12.0, 20.0) if kind == "solve" else rng.uniform(18.0, 34.0)
    bands = 16 + rng.randint(4, 8) if kind == "solve" else round(_log(rng, 1, 160))
    precision = "fp64" if kind == "solve" else rng.choice(["fp64", "fp64", "fp32"])
    case = {key: v for key, v in _hpsi(kind, "", cell, atoms, ecut, k, bands, precision).items() if key != "name"}
    if kind == "solve":
        case |= {"tol": 1e-9, "plane_waves": False, "density": False}
    return case


# ------------------------------------------------------------------ inputs
def _stream():
    """The stream of every case: one program, one stream."""
    global _THE_STREAM
    if _THE_STREAM is None:
        _THE_STREAM = torch.cuda.Stream()
    return _THE_STREAM


_THE_STREAM = None


def _cell(case):
    return np.diag([case["lx"], case["ly"], case["lz"]])


def _positions(case, rng):
    """Atoms on their lattice (4: fcc, 8 and 64: diamond in one or 2 x 2 x 2 cells, else sites of a
    grid that has room for them), displaced by N(0, 0.04 bohr)."""
    lengths = np.array([case["lx"], case["ly"], case["lz"]])
    n = case["atoms"]
    if n in (4, 8, 64):
        rep = 2 if n == 64 else 1
        sites = np.array([c + f for c in np.ndindex(rep, rep, rep) for f in DIAMOND[:4 if n == 4 else 8]]) / rep
    else:
        step = (float(np.prod(lengths)) / n) ** (1.0 / 3.0)
        cells = np.maximum(1, np.round(lengths / step)).astype(int)
        while np.prod(cells) < n:
            cells[int(np.argmax(lengths / cells))] += 1
        sites = np.array(list(np.ndindex(*cells)))
        sites = sites[np.linspace(0, len(sites) - 1, n).round().astype(int)] / cells
    return sites * lengths + rng.normal(0.0, 0.04, size=(n, 3))


def _freqs(n):
    i = np.arange(n)
    return np.where(i <= (n - 1) // 2, i, i - n)


def _potential(case, grid, pos):
    """Start potential of an SCF (Ry, FFT order): the local part of the pseudo-atoms, the Hartree
    potential of a Gaussian valence density of 1.2 bohr on each, and that density's Slater exchange."""
    lengths = [case["lx"], case["ly"], case["lz"]]
    g = [2.0 * math.pi / lengths[i] * _freqs(grid[i]) for i in range(3)]
    ph = [np.exp(-1j * np.outer(pos[:, i], g[i])) for i in range(3)]
    sf = np.einsum("az,ay->azy", ph[2], ph[1]).reshape(len(pos), -1).T @ ph[0]
    q2 = ((g[2] ** 2)[:, None, None] + (g[1] ** 2)[None, :, None] + (g[0] ** 2)[None, None, :]).reshape(-1, grid[0])
    safe = np.where(q2 > 1e-12, q2, 1.0)
    bare = (-4.0 * math.pi * Z_ION / safe + C1 * (2.0 * math.pi) ** 1.5 * R_LOC ** 3) * np.exp(-0.5 * q2 * R_LOC ** 2)
    vq = 2.0 * np.where(q2 > 1e-12, bare + 4.0 * math.pi * Z_ION / safe * np.exp(-0.5 * q2 * 1.44), 0.0)
    shape, per_cell = (grid[2], grid[1], grid[0]), q2.size / np.prod(lengths)
    v = np.fft.ifftn((sf * vq).reshape(shape)).real * per_cell
    rho = np.fft.ifftn((sf * Z_ION * np.exp(-0.5 * q2 * 1.44)).reshape(shape)).real * per_cell
    return (v - 2.0 * np.cbrt(3.0 / math.pi * np.maximum(rho, 0.0))).reshape(-1)


def _system(case, seed):
    """Grid, potential, species and atoms shared by the k-points of a case."""
    rng = np.random.Generator(np.random.PCG64(seed))
    recip = tables.reciprocal(_cell(case))
    grid = tables.auto_grid(case["ecut"], recip)
    pos = _positions(case, rng)
    return {"recip": recip, "grid": grid, "pos": pos, "v": _potential(case, grid, pos), "dij": np.diag([D_S, D_P]),
            "omega": case["lx"] * case["ly"] * case["lz"]}


def _kpoint(case, s, k):
    basis = tables.generate_basis(s["recip"], case["ecut"], np.asarray(k) @ s["recip"])
    phi = tables.build_phi(basis.kpg, [0, 1], [tables.gaussian_radial(0, R_S), tables.gaussian_radial(1, R_P)])
    return basis, phi


def _hamiltonian(ctx, s, basis, phi):
    species = [{"l_list": [0, 1], "dij": s["dij"], "phi": phi}]
    return dzhip.Hamiltonian(ctx, s["grid"], tables.fft_indices(basis, s["grid"]), basis.kinetic, basis.cart, s["v"],
                             1.0 / s["omega"], species, s["pos"], np.zeros(len(s["pos"]), dtype=np.int32))


def _block(case, kinetic, bands, seed):
    """Random wave functions damped at large |k+G|^2, unit-normalised (device, complex)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((bands, kinetic.shape[0], 2), generator=gen, dtype=torch.float64, device="cuda")
    x = torch.view_as_complex(x) / (1.0 + torch.from_numpy(kinetic).cuda())
    x = x / torch.linalg.vector_norm(x, dim=1, keepdim=True)
    return x.to(torch.complex64) if case["precision"] == "fp32" else x


def _mesh(n):
    """Unshifted n x n x n mesh with k and -k merged, in units of the reciprocal vectors."""
    seen, pts = set(), []
    for i in range(n):
        for j in range(n):
            for k in range(n):
                if (i, j, k) not in seen:
                    seen.update({(i, j, k), (-i % n, -j % n, -k % n)})
                    pts.append((i / n, j / n, k / n))
    return pts


def _subspace_matrix(case, seed):
    """A Rayleigh-Ritz matrix: the Ritz values of the wanted bands on the diagonal, weakly coupled to
    directions of higher energy."""
    m, nev = case["m"], case["nev"]
    rng = np.random.Generator(np.random.PCG64(seed))
    d = np.concatenate([-0.6 + 1.2 * (np.arange(nev) + 0.6 * rng.random(nev)) / nev,
                        1.0 + 12.0 * (np.arange(m - nev) + 0.6 * rng.random(m - nev)) / max(1, m - nev)])
    g = (rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))) * (0.3 / math.sqrt(m))
    g[:nev, :nev] *= 0.01
    a = np.tril(g, -1)
    return a + a.conj().T + np.diag(d)


def _probe(m):
    rng = np.random.Generator(np.random.PCG64(m))
    return rng.standard_normal(m) + 1j * rng.standard_normal(m)


def _fix_phase(z, probe):
    """Rows of z, each times the phase that makes its product with probe real and positive."""
    return z * torch.sgn(z @ probe).conj()[:, None]


def _density(case, seed):
    """A positive, smooth random density of about 0.03 electrons per cubic bohr on a cell with
    0.255 bohr between grid points, as the Al cell has."""
    grid = (case["nx"], case["ny"], case["nz"])
    rng = np.random.Generator(np.random.PCG64(seed))
    g = [2.0 * math.pi / (0.255 * n) * _freqs(n) for n in grid]
    q2 = (g[2] ** 2)[:, None, None] + (g[1] ** 2)[None, :, None] + (g[0] ** 2)[None, None, :]
    noise = np.fft.fftn(rng.standard_normal(q2.shape)) * np.exp(-0.25 * q2)
    f = np.fft.ifftn(noise).real
    return (0.03 * np.exp(0.5 * f / max(float(np.std(f)), 1e-300))).reshape(-1)


def _xc_cell(case):
    return np.diag([0.255 * case["nx"], 0.255 * case["ny"], 0.255 * case["nz"]])


def prepare(case, seed):
    kind = case["kind"]
    ctx = dzhip.Context(0)
    if kind == "heev":
        m, nev = case["m"], case["nev"]
        a = torch.from_numpy(np.ascontiguousarray(_subspace_matrix(case, seed).T)).cuda()
        return {"kind": kind, "ctx": ctx, "m": m, "nev": nev, "a": a, "w": torch.empty(nev, dtype=torch.float64, device="cuda"),
                "z": torch.empty((nev, m), dtype=torch.complex128, device="cuda"),
                "probe": torch.from_numpy(_probe(m)).cuda(), "stream": _stream()}
    if kind == "xc":
        cell = _xc_cell(case)
        grid = dzhip.ScfGrid(ctx, (case["nx"], case["ny"], case["nz"]), tables.reciprocal(cell), float(np.prod(np.diag(cell))))
        grid.set_ion(np.zeros(case["nx"] * case["ny"] * case["nz"]))
        grid.set_xc(case["xc"])
        return {"kind": kind, "ctx": ctx, "grid": grid, "rho": _density(case, seed)}
    s = _system(case, seed)
    if kind == "set":
        hams = [_hamiltonian(ctx, s, *_kpoint(case, s, k)) for k in _mesh(case["mesh"])]
        group = dzhip.HamSet(hams)
        group.set_stream(_stream().cuda_stream)
        kinetic = np.concatenate([h._kinetic for h in hams])
        x = _block(case, kinetic, case["bands"], seed)
        return {"kind": kind, "ctx": ctx, "hams": hams, "set": group, "x": x, "y": torch.empty_like(x),
                "bands": case["bands"], "precision": dzhip.FP32 if case["precision"] == "fp32" else dzhip.FP64}
    basis, phi = _kpoint(case, s, (case["kx"], case["ky"], case["kz"]))
    ham = _hamiltonian(ctx, s, basis, phi)
    state = {"kind": kind, "ctx": ctx, "ham": ham, "bands": case["bands"],
             "precision": dzhip.FP32 if case["precision"] == "fp32" else dzhip.FP64}
    if kind == "solve":
        occupied = 2 * case["atoms"]
        state |= {"weights": np.full(occupied, 2.0), "tol": case["tol"], "nconv": occupied,
                  "plane_waves": case["plane_waves"], "density": case["density"]}
    elif kind == "host":
        state["x"] = _block(case, basis.kinetic, case["bands"], seed).to(torch.complex128).cpu().numpy()
    else:
        x = _block(case, basis.kinetic, case["bands"], seed)
        ham.set_stream(_stream().cuda_stream)
        state |= {"x": x, "y": torch.empty_like(x)}
    return state


def run(state):
    kind = state["kind"]
    if kind == "apply":
        state["ham"].apply_dev(state["x"].data_ptr(), state["y"].data_ptr(), state["bands"], state["precision"])
        return state["y"]
    if kind == "host":
        return state["ham"].apply(state["x"], state["precision"])
    if kind == "set":
        state["set"].apply_dev(state["x"].data_ptr(), state["y"].data_ptr(), state["bands"], state["precision"])
        return state["y"]
    if kind == "heev":
        state["ctx"].heev_dev(state["a"].data_ptr(), state["m"], state["m"], state["nev"], state["w"].data_ptr(),
                              state["z"].data_ptr(), state["m"], state["stream"].cuda_stream)
        # An eigenvector has no phase of its own: each is given a real positive overlap with a
        # fixed vector, the convention that makes bands of different calls comparable.
        with torch.cuda.stream(state["stream"]):
            return {"values": state["w"], "vectors": _fix_phase(state["z"], state["probe"])}
    if kind == "xc":
        state["grid"].init_rho(state["rho"])
        return state["grid"].read(dzhip.GRID_VIN)
    # The occupied bands are converged, the others are a buffer, as the SCF asks for them.
    values, _, _ = state["ham"].eig_solve(state["bands"], tol=state["tol"], max_iter=200, want_vectors=False,
                                          init_diagonal=state["plane_waves"], nconv=state["nconv"])
    out = {"values": values[:state["nconv"]]}
    if state["density"]:
        out["rho"] = state["ham"].density_solution(state["weights"])
    return out


# ------------------------------------------------------------------ accounting
def _sphere(case):
    """Plane waves and grid points, from the sphere's volume."""
    omega = case["lx"] * case["ly"] * case["lz"]
    n_pw = omega * case["ecut"] ** 1.5 / (6.0 * math.pi ** 2)
    grid = tables.auto_grid(case["ecut"], tables.reciprocal(_cell(case)))
    return n_pw, float(np.prod(grid))


def _apply_work(n_pw, points, projectors, bands, size):
    """Block in and out, potential and kinetic energies; two transforms of which the sphere's zeros
    save about 40 %, and the two projector products."""
    fft = 0.6 * 2.0 * 5.0 * points * math.log2(points)
    return {"bytes": bands * 2.0 * n_pw * size + (points + n_pw + 4.0 * n_pw) * size / 2.0 + 4.0 * n_pw,
            "flops": bands * (fft + 16.0 * projectors * n_pw)}


def work(case):
    kind = case["kind"]
    if kind == "heev":
        m, nev = case["m"], case["nev"]
        return {"bytes": 16.0 * m * m / 2 + 16.0 * m * nev + 8.0 * nev, "flops": 16.0 / 3.0 * m ** 3 + 8.0 * m * m * nev}
    if kind == "xc":
        n = float(case["nx"] * case["ny"] * case["nz"])
        ffts = 10 if case["xc"] == "pbe" else 2
        return {"bytes": 16.0 * n, "flops": n * (ffts * 5.0 * math.log2(n) + (300.0 if case["xc"] == "pbe" else 60.0))}
    n_pw, points = _sphere(case)
    size = 8.0 if case["precision"] == "fp32" else 16.0
    if kind == "set":
        n_k = len(_mesh(case["mesh"]))
        one = _apply_work(n_pw, points, 4 * case["atoms"], case["bands"], size)
        return {"bytes": n_k * one["bytes"], "flops": n_k * one["flops"]}
    one = _apply_work(n_pw, points, 4 * case["atoms"], case["bands"], size)
    if kind == "solve":
        # A residual falls by about a factor 2.5 per step of the block; each step applies H once and
        # makes the products with a basis of about twice the bands.
        steps = math.log(1.0 / case["tol"]) / math.log(2.5)
        b = case["bands"]
        return {"bytes": steps * (one["bytes"] + 16.0 * n_pw * 4 * b), "flops": steps * (one["flops"] + 8.0 * n_pw * 8.0 * b * b)}
    return one


# ------------------------------------------------------------------ the same in 64 bits, plain torch
def _projectors(s, basis, phi):
    """[atoms * 4, n_pw] complex: phi e^{iG.tau}."""
    ph = np.exp(1j * (s["pos"] @ basis.cart.T))
    return torch.from_numpy((ph[:, None, :] * phi[None]).reshape(-1, basis.n)).cuda()


def _exact_apply(s, basis, phi, x):
    nx, ny, nz = s["grid"]
    idx = torch.from_numpy(tables.fft_indices(basis, s["grid"]).astype(np.int64)).cuda()
    v = torch.from_numpy(s["v"]).cuda().reshape(nz, ny, nx)
    a = _projectors(s, basis, phi)
    d = torch.from_numpy(np.tile(np.repeat(np.diag(s["dij"]), [1, 3]), len(s["pos"]))).cuda() / s["omega"]
    kinetic = torch.from_numpy(basis.kinetic).cuda()
    x = x.to(torch.complex128)
    y = x * kinetic + ((x @ a.T) * d) @ a.conj()
    for b in range(0, x.shape[0], 16):
        part = x[b:b + 16]
        f = torch.zeros((part.shape[0], nz * ny * nx), dtype=torch.complex128, device="cuda")
        f[:, idx] = part
        f = torch.fft.ifftn(f.reshape(-1, nz, ny, nx), dim=(1, 2, 3)) * v
        y[b:b + 16] += torch.fft.fftn(f, dim=(1, 2, 3)).reshape(part.shape[0], -1)[:, idx]
    return y


def _exact_solve(case, s, basis, phi):
    """Dense diagonalisation of H; None above 2,100 plane waves."""
    if basis.n > 2100:
        return None
    nx, ny, nz = s["grid"]
    vg = np.fft.fftn(s["v"].reshape(nz, ny, nx)) / s["v"].size
    dx, dy, dz = (q[:, None] - q[None, :] for q in (basis.h, basis.k, basis.l))
    a = _projectors(s, basis, phi).cpu().numpy()
    d = np.tile(np.repeat(np.diag(s["dij"]), [1, 3]), len(s["pos"])) / s["omega"]
    h = vg[dz % nz, dy % ny, dx % nx] + (a.conj().T * d) @ a
    h[np.diag_indices(basis.n)] += basis.kinetic
    occupied = 2 * case["atoms"]
    w, z = np.linalg.eigh(h)
    if not case["density"]:
        return {"values": w[:occupied]}
    idx = tables.fft_indices(basis, s["grid"])
    rho = np.zeros(nx * ny * nz)
    for b in range(occupied):
        f = np.zeros(nx * ny * nz, dtype=np.complex128)
        f[idx] = z[:, b]
        psi = np.fft.ifftn(f.reshape(nz, ny, nx)).reshape(-1) * f.size
        rho += 2.0 * (psi.real ** 2 + psi.imag ** 2) / s["omega"]
    return {"values": w[:occupied], "rho": rho}


def _exact_xc(case, rho):
    """V_H + V_xc (Ry): the published energy of each functional, its potential by differentiating the
    energy of the grid density."""
    n = (case["nz"], case["ny"], case["nx"])
    g = [2.0 * math.pi / (0.255 * k) * torch.from_numpy(_freqs(k).astype(np.float64)) for k in n]
    g = [g[2][None, None, :], g[1][None, :, None], g[0][:, None, None]]
    q2 = g[0] ** 2 + g[1] ** 2 + g[2] ** 2
    r = torch.from_numpy(rho).reshape(n).requires_grad_(True)
    rg = torch.fft.fftn(r)
    kernel = torch.where(q2 > 1e-12, 8.0 * math.pi / torch.where(q2 > 1e-12, q2, 1.0), 0.0)
    vh = torch.fft.ifftn(kernel * rg.detach()).real
    rs = (3.0 / (4.0 * math.pi * r)) ** (1.0 / 3.0)
    ex = -0.75 * (3.0 / math.pi) ** (1.0 / 3.0) * r ** (1.0 / 3.0)
    ln, sq = torch.log(rs), torch.sqrt(rs)
    if case["xc"] == "lda_pz":
        ec = torch.where(rs < 1.0, 0.0311 * ln - 0.048 + 0.0020 * rs * ln - 0.0116 * rs,
                         -0.1423 / (1.0 + 1.0529 * sq + 0.3334 * rs))
    else:
        mu, kappa, beta, gamma = 0.2195149727645171, 0.804, 0.06672455060314922, 0.031090690869654895
        grad2 = sum(torch.fft.ifftn(1j * k * rg).real ** 2 for k in g)
        kf = (3.0 * math.pi ** 2 * r) ** (1.0 / 3.0)
        ex = ex * (1.0 + kappa - kappa / (1.0 + mu / kappa * grad2 / (4.0 * kf ** 2 * r ** 2)))
        f = 7.5957 * sq + 3.5876 * rs + 1.6382 * rs * sq + 0.49294 * rs ** 2
        ec = -0.062182 * (1.0 + 0.21370 * rs) * torch.log(1.0 + 1.0 / (0.062182 * f))
        t2 = grad2 / (16.0 * kf / math.pi * r ** 2)
        at2 = beta / gamma / (torch.exp(-ec / gamma) - 1.0) * t2
        ec = ec + gamma * torch.log(1.0 + beta / gamma * t2 * (1.0 + at2) / (1.0 + at2 + at2 ** 2))
    vxc, = torch.autograd.grad((2.0 * r * (ex + ec)).sum(), r)
    return (vh + vxc).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "heev":
        w, z = np.linalg.eigh(_subspace_matrix(case, seed))
        z = torch.from_numpy(np.ascontiguousarray(z[:, :case["nev"]].T))
        return {"values": w[:case["nev"]], "vectors": _fix_phase(z, torch.from_numpy(_probe(case["m"])))}
    if kind == "xc":
        return _exact_xc(case, _density(case, seed))
    s = _system(case, seed)
    if kind == "set":
        parts = [_kpoint(case, s, k) for k in _mesh(case["mesh"])]
        kinetic = np.concatenate([b.kinetic for b, _ in parts])
        x = _block(case, kinetic, case["bands"], seed)
        y = torch.empty_like(x, dtype=torch.complex128)
        at = 0
        for basis, phi in parts:
            y[:, at:at + basis.n] = _exact_apply(s, basis, phi, x[:, at:at + basis.n].contiguous())
            at += basis.n
        return y
    basis, phi = _kpoint(case, s, (case["kx"], case["ky"], case["kz"]))
    if kind == "solve":
        return _exact_solve(case, s, basis, phi)
    y = _exact_apply(s, basis, phi, _block(case, basis.kinetic, case["bands"], seed))
    return y.cpu().numpy() if kind == "host" else y
