"""Kernels of the short axes (two-factor plans) against the oracle: the column z solve at every
nz it takes, at the smallest and largest Lmax, with ragged column groups, both storage types of
the spectrum, and as batched jobs; the two-pass plane kernels at every edge along x and along y,
and fused against unfused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the repository's parity bound (FP64 path) and its FP32-spectrum bound on short chains
TOL, TOL32 = 1e-10, 2e-6

SHORT = (8, 12, 16, 18, 24, 32, 36, 48, 54)


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def _case(shape, Nblk, L, seed):
    box = tuple(0.12 * e + 0.5 for e in shape[::-1])
    lam = (1.0, 0.5, 2.0)[:len(Nblk)]
    w = 1.5 * np.random.default_rng(seed).standard_normal((len(Nblk),) + shape)
    return box, lam, w


def _check(wlc, oracle, shape, Nblk, L, spec32=False):
    box, lam, w = _case(shape, Nblk, L, sum(shape))
    orc = oracle.Oracle(shape, box, Nblk, L, lam)
    q, qs = orc.forward(w), orc.backward(w)
    phi, Q, td = orc.density(q, qs)
    g = wlc.WormlikeMDE(shape, box, Nblk, L, lam, keep_qstar=True, spectrum_fp32=spec32)
    g.set_w(w)
    g.MDE_q()
    g.MDE_qstar()
    gphi, gQ, gtd = g.density()
    tol = TOL32 if spec32 else TOL
    for s in range(sum(Nblk) + 1):
        assert _rel(g.get_q(+1, s), orc.slice(q, s)) < tol, f"forward slice {s}"
        assert _rel(g.get_q(-1, s), orc.slice(qs, s)) < tol, f"backward slice {s}"
    assert _rel(gphi, phi) < tol and abs(gQ - Q) / Q < tol and abs(gtd - td) / td < tol
    g.close()
    orc.close()


# nx = 6: one column beyond a full tile; nx = 12: three columns beyond one; nx = 8: one group of
# two columns half padding
@pytest.mark.parametrize("nx,L", [(6, (1, 4)), (12, (6, 3)), (8, (8, 7))])
@pytest.mark.parametrize("nz", SHORT)
def test_z_columns(wlc, oracle, nz, nx, L):
    _check(wlc, oracle, (nz, 4, nx), (2, 3), L)


@pytest.mark.parametrize("nz", (16, 18, 36, 54))
def test_z_columns_fp32_spectrum(wlc, oracle, nz):
    _check(wlc, oracle, (nz, 6, 8), (3, 3), (2, 5), spec32=True)


def test_z_columns_full_blocks_and_l0(wlc, oracle):
    # 8 column groups per row and a multiple of 8 of them in all (the XCD order); Lmax 0
    _check(wlc, oracle, (24, 16, 30 + 2), (2, 2, 2), (0, 2, 1))


def test_z_columns_batched(wlc):
    cases = []
    for nz, L in ((18, 4), (18, 4), (36, 6), (54, 5), (12, 8)):
        shape = (nz, 4, 6)
        box, lam, w = _case(shape, (3, 4), (L, L), nz + len(cases))
        cases.append(dict(shape=shape, box=box, Nblk=(3, 4), L=(L, L), lam=lam, w=w,
                          chi=np.array([[0, 15, 0], [15, 0, 0], [0, 0, 0]], float)))
    b = wlc.Batch(cases)
    for i, c in enumerate(cases):
        b.set_w(i, c["w"])
    b.sweep()
    for i, c in enumerate(cases):
        g = wlc.WormlikeMDE(c["shape"], c["box"], c["Nblk"], c["L"], c["lam"])
        g.set_w(c["w"])
        g.MDE_q()
        g.MDE_qstar()
        phi, Q, td = g.density()
        bphi, bQ, btd = b.density(i)
        # the twins run the same operations; contraction may differ
        assert _rel(bphi, phi) < 1e-13 and abs(bQ - Q) / Q < 1e-13 and abs(btd - td) / td < 1e-13
        g.close()
    b.close()


# every edge as nx and as ny, short with long (idle lanes in one role), compile-time squares
PLANES = [(8, 72), (72, 8), (12, 54), (54, 12), (16, 36), (36, 16), (18, 48), (48, 18), (24, 32),
          (32, 24), (64, 18), (12, 64), (24, 24), (32, 32), (48, 48), (72, 72), (36, 54)]


@pytest.mark.parametrize("ny,nx", PLANES)
def test_two_pass_planes(wlc, oracle, ny, nx):
    # the basis shrinks, then grows; nz = 2 walks contiguous (harmonic, z)
    _check(wlc, oracle, (2, ny, nx), (3, 2, 3), (2, 1, 3))


@pytest.mark.parametrize("shape,spec32", [((8, 18, 24), False), ((6, 54, 36), False), ((4, 32, 32), True),
                                          ((4, 16, 72), True)])
def test_two_pass_planes_fused_equals_unfused(wlc, monkeypatch, shape, spec32):
    Nblk, L = (3, 3, 2), (3, 1, 2)
    box, lam, w = _case(shape, Nblk, L, 9)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("WLC_FUSE", fuse)
        g = wlc.WormlikeMDE(shape, box, Nblk, L, lam, keep_qstar=True, spectrum_fp32=spec32)
        g.set_w(w)
        g.MDE_q()
        g.MDE_qstar()
        out.append([g.get_q(d, s) for d in (1, -1) for s in range(sum(Nblk) + 1)])
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_two_pass_planes_batched(wlc):
    cases = []
    for shape, L in (((4, 24, 18), 2), ((4, 24, 18), 2), ((8, 36, 54), 1), ((4, 48, 48), 3)):
        box, lam, w = _case(shape, (3, 4), (L, L), sum(shape) + len(cases))
        cases.append(dict(shape=shape, box=box, Nblk=(3, 4), L=(L, L), lam=lam, w=w,
                          chi=np.array([[0, 15, 0], [15, 0, 0], [0, 0, 0]], float)))
    b = wlc.Batch(cases)
    for i, c in enumerate(cases):
        b.set_w(i, c["w"])
    b.sweep()
    for i, c in enumerate(cases):
        g = wlc.WormlikeMDE(c["shape"], c["box"], c["Nblk"], c["L"], c["lam"])
        g.set_w(c["w"])
        g.MDE_q()
        g.MDE_qstar()
        phi, Q, td = g.density()
        bphi, bQ, btd = b.density(i)
        assert _rel(bphi, phi) < 1e-13 and abs(bQ - Q) / Q < 1e-13 and abs(btd - td) / td < 1e-13
        g.close()
    b.close()
