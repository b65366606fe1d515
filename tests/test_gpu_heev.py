"""The device Hermitian eigensolver (dzhip_heev: Householder tridiagonalisation in one
grid-synchronised launch, multisection, inverse iteration, back-transformation) against numpy.linalg.eigh, which is
LAPACK zheevd: the reference's subspace eigenproblems call LAPACK zheev
(src/features/linalg/lobpcg/common.zig:440-537).

Bars: eigenvalues within 1e-12 of the spectral radius; Z^H Z = I within 1e-12; residuals
|A z - lambda z| within 1e-11 of the spectral radius.  Sizes 1, 2, 20, 164 and 648 (the block
Davidson's first and largest subspaces at 160 bands), exact and near degeneracies, and a
Rayleigh-Ritz matrix of the Si-8 Hamiltonian."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_hermitian(m, rng, spectrum=None):
    q, _ = np.linalg.qr(rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m)))
    lam = np.sort(rng.uniform(-2.0, 30.0, m)) if spectrum is None else np.asarray(spectrum, dtype=float)
    a = (q * lam) @ q.conj().T
    return 0.5 * (a + a.conj().T), lam


def check(ctx, a, nev, tol_val=1e-12, tol_res=1e-11):
    w, z = ctx.heev(a, nev)
    ref = np.linalg.eigvalsh(a)[:nev]
    scale = max(1.0, float(np.max(np.abs(ref))), float(np.linalg.norm(a, 2)))
    dval = float(np.max(np.abs(w - ref)))
    orth = float(np.max(np.abs(z.conj().T @ z - np.eye(nev))))
    res = float(np.max(np.linalg.norm(a @ z - z * w, axis=0)))
    print(f"m={a.shape[0]} nev={nev} |dw|={dval:.2e} orth={orth:.2e} res={res:.2e} scale={scale:.1f}")
    assert dval <= tol_val * scale
    assert orth <= 1e-12
    assert res <= tol_res * scale
    return w, z


@pytest.mark.parametrize("m,nev", [(1, 1), (2, 2), (20, 20), (20, 7), (164, 160), (648, 160), (648, 648)])
def test_heev_random(ctx, m, nev):
    rng = np.random.default_rng(1000 + m + nev)
    a, _ = random_hermitian(m, rng)
    check(ctx, a, nev)


@pytest.mark.parametrize("m", [3, 4, 5, 63, 64, 65, 66, 127, 129, 193, 257, 385, 513, 705, 833, 1023, 1024])
def test_heev_register_chunks(ctx, m):
    """Sizes at the edges of the tridiagonalisation's 64-row register chunks and of its four columns
    per workgroup, one more row than each instance holds, and the largest; bars as above."""
    rng = np.random.default_rng(2000 + m)
    g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    check(ctx, 0.5 * (g + g.conj().T) + np.diag(np.linspace(0.0, 20.0, m)), min(m, 24))


@pytest.mark.parametrize("m", [7, 8, 9, 10, 16, 17, 18, 25, 256, 258, 272, 273, 274, 521, 769])
def test_heev_reflector_blocks(ctx, m):
    """Sizes at the edges of the back-transformation's blocks of eight reflectors, of its pairs of
    blocks and of its 256-row groups; bars as above."""
    rng = np.random.default_rng(3000 + m)
    g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    check(ctx, 0.5 * (g + g.conj().T), min(m, 20))


@pytest.mark.parametrize("m,nev", [(5, 3), (15, 15), (16, 16), (17, 17), (65, 33), (79, 64), (80, 65), (200, 161)])
def test_heev_orthonormalisation_tiles(ctx, m, nev):
    """Sizes at the edges of the Newton-Schulz products' 16 x 16 tiles and of the chunks that their four
    wavefronts share; bars as above."""
    rng = np.random.default_rng(4000 + m)
    g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    check(ctx, 0.5 * (g + g.conj().T), nev)


def test_heev_degenerate_and_clustered(ctx):
    """Exactly degenerate triplets and pairs (symmetry-degenerate bands), a cluster split by
    1e-13, and a zero off-diagonal block (a reducible tridiagonal)."""
    rng = np.random.default_rng(7)
    lam = np.sort(np.concatenate([np.repeat(rng.uniform(-1, 1, 20), 3), np.repeat(rng.uniform(1, 5, 30), 2),
                                  1.5 + 1e-13 * np.arange(6), rng.uniform(5, 20, 100)]))
    a, _ = random_hermitian(lam.size, rng, lam)
    check(ctx, a, 160)
    # Block diagonal: the reduction meets zero columns (tau = 0 reflectors).
    b1, _ = random_hermitian(40, rng)
    b = np.zeros((80, 80), dtype=complex)
    b[:40, :40] = b1
    b[40:, 40:] = b1
    check(ctx, b, 80)
    # Real diagonal matrix: every reflector is the identity.
    check(ctx, np.diag(np.linspace(-3, 3, 50)).astype(complex), 50)


def test_heev_errors(dz, ctx):
    with pytest.raises(dz.BadArgument):
        ctx.heev(np.eye(4, dtype=complex), 5)
    with pytest.raises(dz.BadArgument):
        ctx.heev(np.eye(1025, dtype=complex), 4)


def test_heev_rayleigh_ritz_matrix(dz, ctx):
    """T = V^H H V of the Si-8 Hamiltonian over an orthonormalised random block (the subspace
    matrix the Davidson solver diagonalises)."""
    from dzhip import workloads
    from oracle import adapters, hamiltonian

    w = workloads.si8(nbands=8)
    rng = np.random.default_rng(3)
    v = rng.standard_normal((w.npw, 200)) + 1j * rng.standard_normal((w.npw, 200))
    v, _ = np.linalg.qr(v)
    hv = hamiltonian.apply_hamiltonian_batched(adapters.context_from_workload(w), v.T).T
    t = v.conj().T @ hv
    t = 0.5 * (t + t.conj().T)
    check(ctx, t, 160)


def test_heev_concurrent_threads(dz, ctx):
    """Six host threads, each with its own context (own stream), solving at the same time.  The
    blocking eigensolver launches its tridiagonalisation as an ordinary dispatch admitted by the
    device's gate: at m = 648 a grid takes 14 CUs of each XCD, so at most two of these grids run
    at once and the rest wait for their share.  Every result must equal the one-thread result."""
    import threading

    rng = np.random.default_rng(11)
    sizes = (648, 492, 328, 648, 164, 492)
    mats = [random_hermitian(m, rng)[0] for m in sizes]
    ctxs = [dz.Context(0) for _ in sizes]
    alone = [ctxs[0].heev(a, 160) for a in mats]
    out, errs = [None] * len(sizes), []

    def work(i):
        try:
            res = []
            for _ in range(3):
                res.append(ctxs[i].heev(mats[i], 160))
            out[i] = res
        except Exception as e:  # reported on the main thread
            errs.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for c in ctxs:
        c.close()
    assert not errs, errs
    for i, a in enumerate(mats):
        ref = np.linalg.eigvalsh(a)[:160]
        for w, z in out[i]:
            assert np.array_equal(w, alone[i][0]) and np.array_equal(z, alone[i][1])
        assert np.max(np.abs(alone[i][0] - ref)) <= 1e-12 * max(1.0, float(np.max(np.abs(ref))))


def test_heev_shared_launch_falls_back_to_cooperative():
    """The blocking eigensolver's admitted launch gives up when its barrier waits longer than its
    spin limit and the call is repeated cooperatively.  Forced from the host: a child process with
    the admitted launch's spin limit at one poll (its barrier gives up at once; every workgroup
    exits normally) must still return the exact spectrum."""
    import os
    import subprocess
    import sys
    from pathlib import Path

    root = Path(__file__).resolve().parents[1]
    script = (
        "import sys, numpy as np; sys.path.insert(0, %r); import dzhip\n"
        "rng = np.random.default_rng(5); m = 648\n"
        "q, _ = np.linalg.qr(rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m)))\n"
        "lam = np.sort(rng.uniform(-2.0, 30.0, m)); a = (q * lam) @ q.conj().T; a = 0.5 * (a + a.conj().T)\n"
        "ctx = dzhip.Context(0); w, z = ctx.heev(a, 160)\n"
        "print(float(np.max(np.abs(w - lam[:160]))), float(np.max(np.abs(z.conj().T @ z - np.eye(160)))))\n"
    ) % str(root / "dft-zig_amd")
    env = dict(os.environ, DZHIP_HEEV_SHARED_SPIN="1")
    print("child: heev m=648 nev=160 with DZHIP_HEEV_SHARED_SPIN=1", flush=True)
    out = subprocess.run([sys.executable, "-c", script], env=env, capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr[-2000:]
    dval, orth = map(float, out.stdout.split()[-2:])
    assert dval < 1e-12 * 30.0 and orth < 1e-12


@pytest.mark.parametrize("tiny,bar", [(1e-150, 1e-12), (3e-155, 1e-12), (1e-158, 1e-6), (1e-170, 1e-12), (1e-310, 1e-12)])
@pytest.mark.parametrize("m", [3, 70])
def test_heev_tiny_columns(ctx, m, tiny, bar):
    """One row coupled to the rest by a tiny fraction of its size.  Bars as above, but for 1e-158, whose
    squares are subnormal numbers of about 1e-317: a norm from them, and with it the reflector, is good to
    5e-324 / 1e-317 = 5e-7.  Below 1e-162 they are zero and the row is taken as decoupled."""
    rng = np.random.default_rng(5000 + m)
    g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    a = 0.5 * (g + g.conj().T)
    a[0, 1:] *= tiny
    a[1:, 0] *= tiny

    def bars(b):
        w, z = ctx.heev(b, m)
        err = (np.max(np.abs(w - np.linalg.eigvalsh(b))), np.max(np.abs(z.conj().T @ z - np.eye(m))),
               np.max(np.linalg.norm(b @ z - z * w, axis=0)))
        scale = max(1.0, float(np.linalg.norm(b, 2)))
        print(f"m={m} {tiny}: values {err[0]:.1e} orthonormality {err[1]:.1e} residual {err[2]:.1e}", flush=True)
        assert err[0] <= bar * scale and err[1] <= bar and err[2] <= 10 * bar * scale

    bars(a)
    # The same in the last columns, and real (alpha has no imaginary part).
    bars(np.ascontiguousarray(a[::-1, ::-1]))
    bars(a.real.astype(complex))
    # Tiny below an ordinary complex or real coupling of the first two rows.
    a[1, 0] = 0.7 + 0.2j
    a[0, 1] = a[1, 0].conj()
    bars(a)
    bars(a.real.astype(complex))


@pytest.mark.parametrize("cols,sizes", [(8, (1, 8, 9, 129, 193, 257, 385, 513, 705, 833, 1024)),
                                        (16, (1, 16, 17, 257, 384, 385, 513, 704))])
def test_heev_columns_per_workgroup(cols, sizes):
    """The tridiagonalisation's instances of two and four columns a wavefront, which a device of fewer CUs
    takes, selected from the host in a child process (DZHIP_HEEV_COLS), at the edges of their sizes;
    bars as above, against LAPACK's eigenvalues."""
    import os
    import subprocess
    import sys
    from pathlib import Path

    root = Path(__file__).resolve().parents[1]
    script = (
        "import sys, numpy as np; sys.path.insert(0, %r); import dzhip\n"
        "ctx = dzhip.Context(0)\n"
        "for m in %r:\n"
        "    rng = np.random.default_rng(6000 + m); g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))\n"
        "    a = 0.5 * (g + g.conj().T); nev = min(m, 24); print('m', m, file=sys.stderr, flush=True)\n"
        "    w, z = ctx.heev(a, nev); s = max(1.0, float(np.linalg.norm(a, 2)))\n"
        "    print(m, np.max(np.abs(w - np.linalg.eigvalsh(a)[:nev])) / s, np.max(np.abs(z.conj().T @ z - np.eye(nev))),\n"
        "          np.max(np.linalg.norm(a @ z - z * w, axis=0)) / s, flush=True)\n"
    ) % (str(root / "dft-zig_amd"), sizes)
    print(f"child: heev of {sizes} with DZHIP_HEEV_COLS={cols}", flush=True)
    out = subprocess.run([sys.executable, "-c", script], env=dict(os.environ, DZHIP_HEEV_COLS=str(cols)),
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    lines = [l.split() for l in out.stdout.splitlines()]
    assert [int(l[0]) for l in lines] == list(sizes)
    for l in lines:
        print(*l, flush=True)
        dval, orth, res = map(float, l[1:])
        assert dval <= 1e-12 and orth <= 1e-12 and res <= 1e-11


def test_heev_shared_launch_repeats_are_counted():
    """With the admitted launch's spin limit at one poll the exchange gives up (every workgroup exits
    normally, whichever of its wavefronts gives up first) and the call is repeated cooperatively: sizes of
    two to 162 workgroups, each call counted as a repeat and its spectrum LAPACK's (1e-12 of the largest
    eigenvalue)."""
    import os
    import subprocess
    import sys
    from pathlib import Path

    root = Path(__file__).resolve().parents[1]
    sizes = (40, 164, 328, 648)
    script = (
        "import sys, numpy as np; sys.path.insert(0, %r); import dzhip\n"
        "ctx = dzhip.Context(0)\n"
        "for m in %r:\n"
        "    rng = np.random.default_rng(7000 + m); g = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))\n"
        "    a = 0.5 * (g + g.conj().T); ref = np.linalg.eigvalsh(a)[:20]; before = dzhip.heev_retries()\n"
        "    w, _ = ctx.heev(a, 20)\n"
        "    print(m, np.max(np.abs(w - ref)) / np.max(np.abs(ref)), dzhip.heev_retries() - before, flush=True)\n"
    ) % (str(root / "dft-zig_amd"), sizes)
    print(f"child: heev of {sizes} with DZHIP_HEEV_SHARED_SPIN=1", flush=True)
    out = subprocess.run([sys.executable, "-c", script], env=dict(os.environ, DZHIP_HEEV_SHARED_SPIN="1"),
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    lines = [l.split() for l in out.stdout.splitlines()]
    assert [int(l[0]) for l in lines] == list(sizes)
    for l in lines:
        print(*l, flush=True)
        assert float(l[1]) < 1e-12 and int(l[2]) == 1


@pytest.mark.parametrize("copies,h", [(2, 20), (2, 65), (2, 130), (3, 20), (3, 65), (3, 130), (3, 200)])
def test_heev_equal_blocks(ctx, copies, h):
    """Equal diagonal blocks: T splits, and inverse iteration gives the members of a cluster nearly
    parallel vectors for some of the pairs; bars as above."""
    for seed in range(6):
        rng = np.random.default_rng(8000 + seed)
        g = rng.standard_normal((h, h)) + 1j * rng.standard_normal((h, h))
        check(ctx, np.kron(np.eye(copies), 0.5 * (g + g.conj().T)), 3 * copies * h // 4)
