"""The three-part z solve at nz = 128 (Lmax 5-8): against the oracle on ragged column pairs (a pair
with one real column, a padding pair, a whole tile), with the FP32 spectrum, with Lmax changing at
a junction, against the whole-column kernel where a workgroup takes more than one pair, and as
batched jobs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the repository's parity bound (FP64 path) and its FP32-spectrum bound on short chains
TOL, TOL32 = 1e-10, 2e-6


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def _case(shape, nblk, seed):
    box = tuple(0.12 * e + 0.5 for e in shape[::-1])
    return box, (1.0, 0.5)[:nblk], 1.5 * np.random.default_rng(seed).standard_normal((nblk,) + shape)


# nx / 2 + 1 = 4 (a full tile), 5 (half a pair, then a padding pair), 7 (half a pair)
@pytest.mark.parametrize("nx,L,spec32", [(6, (5, 8), False), (8, (6, 7), False), (12, (8, 6), False),
                                         (8, (7, 8), True), (12, (5, 6), True)])
def test_matches_oracle(wlc, oracle, nx, L, spec32):
    shape, Nblk = (128, 2, nx), (2, 3)
    box, lam, w = _case(shape, 2, nx)
    orc = oracle.Oracle(shape, box, Nblk, L, lam)
    q, qs = orc.forward(w), orc.backward(w)
    g = wlc.WormlikeMDE(shape, box, Nblk, L, lam, keep_qstar=True, spectrum_fp32=spec32)
    g.set_w(w)
    g.MDE_q()
    g.MDE_qstar()
    tol = TOL32 if spec32 else TOL
    for s in range(sum(Nblk) + 1):
        assert _rel(g.get_q(+1, s), orc.slice(q, s)) < tol, f"forward slice {s}"
        assert _rel(g.get_q(-1, s), orc.slice(qs, s)) < tol, f"backward slice {s}"
    g.close()
    orc.close()


@pytest.mark.parametrize("L", [5, 8])
def test_many_pairs_match_whole_columns(wlc, monkeypatch, L):
    # 6 pairs and a half real one a row, 48 rows: 42 an XCD, more than its 32 workgroups
    shape, Nblk = (128, 48, 24), (4,)
    box, lam, w = _case(shape, 1, L)
    out = []
    for split in ("0", "1"):
        monkeypatch.setenv("WLC_ZSOLVE_SPLIT", split)
        g = wlc.WormlikeMDE(shape, box, Nblk, (L,), lam, keep_qstar=True)
        g.set_w(w)
        g.MDE_q()
        g.MDE_qstar()
        out.append([g.get_q(d, s) for d in (1, -1) for s in range(5)])
        g.close()
    # the same transforms and rotations, contracted differently: a few roundings per step
    for a, b in zip(*out):
        assert _rel(b, a) < 1e-13


def test_batched(wlc):
    cases = []
    for L in (6, 6, 8):
        shape = (128, 2, 12)
        box, lam, w = _case(shape, 2, L + len(cases))
        cases.append(dict(shape=shape, box=box, Nblk=(2, 3), L=(L, L), lam=lam, w=w,
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
