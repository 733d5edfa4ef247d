"""Where the library changes from one kernel to another by the size of a launch: which kernel runs on
either side of the line (on the host, launches recorded), and both sides against the oracle."""
import numpy as np
import pytest

import host_hip

# the repository's parity bound (FP64 path) and its FP32-spectrum bound on short chains
TOL, TOL32 = 1e-10, 2e-6

SWEEP = """
    shape, Nblk, L, sp = {shape}, {Nblk}, {L}, {sp}
    g = W.WormlikeMDE(shape, (3.0, 3.5, 4.0), Nblk, L, (1.0,) * len(L), spectrum_fp32=sp)
    g.set_w(np.zeros((len(L),) + shape))
    H.host_hip_forget()
    g.MDE_q()
    print("\\n".join(launches()))
"""


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


def _launches(so, shape, Nblk, L, sp=False):
    return host_hip.run(so, SWEEP.format(shape=shape, Nblk=Nblk, L=L, sp=sp))


def _matches_oracle(wlc, oracle, shape, Nblk, L, spec32=False):
    box, lam = tuple(0.12 * e + 0.5 for e in shape[::-1]), (1.0, 0.5, 2.0)[:len(L)]
    w = 1.5 * np.random.default_rng(sum(shape)).standard_normal((len(L),) + shape)
    orc = oracle.Oracle(shape, box, Nblk, L, lam)
    g = wlc.WormlikeMDE(shape, box, Nblk, L, lam, keep_qstar=True, spectrum_fp32=spec32)
    g.set_w(w)
    g.MDE_q()
    g.MDE_qstar()
    for d, ref in ((1, orc.forward(w)), (-1, orc.backward(w))):
        for s in range(sum(Nblk) + 1):
            a, b = g.get_q(d, s), orc.slice(ref, s)
            assert np.abs(a - b).max() < (TOL32 if spec32 else TOL) * np.abs(b).max(), (d, s)
    g.close()
    orc.close()


def _batch_matches_handles(wlc, instances):
    cases = []
    for shape, L in instances:
        w = 1.5 * np.random.default_rng(len(cases)).standard_normal((1,) + shape)
        cases.append(dict(shape=shape, box=(4.0, 3.5, 3.0), Nblk=(3,), L=(L,), lam=(1.0,), w=w,
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
        assert np.abs(bphi - phi).max() < 1e-13 * np.abs(phi).max()
        assert abs(bQ - Q) / Q < 1e-13 and abs(btd - td) / td < 1e-13
        g.close()
    b.close()


# 48 x 72 planes: two-pass kernels up to 512 planes of the largest block's launches, the run-time kernels
# above; all launches of a chain alike
def test_planes_of_five_waves(so):
    for ny, nx in ((48, 72), (72, 48)):
        for nz, L, two in ((32, (3,), True), (36, (3,), False), (18, (4,), True), (24, (4,), False)):
            k = [x for x in _launches(so, (nz, ny, nx), (4,), L) if "k2_" in x or "rhs" in x or "ifft" in x]
            assert len(k) == 5 and all(("k2_" in x) == two for x in k), (ny, nx, nz, L)
    for L in ((2, 3), (3, 2)):
        k = [x for x in _launches(so, (36, 48, 72), (3, 3), L) if "k2_" in x or "rhs" in x or "ifft" in x]
        assert len(k) == 7 and not any("k2_" in x for x in k), L
    # other planes keep the two-pass kernels at any number
    for nz, ny, nx in ((72, 54, 72), (64, 64, 72), (64, 72, 72), (72, 36, 72)):
        k = _launches(so, (nz, ny, nx), (4,), (4,))
        assert sum("k2_" in x for x in k) == 5, (nz, ny, nx)


# 72 x 64, 64 x 72 and 72 x 72 planes on a z axis longer than 64: run-time kernels between 600 and 3300
# planes
def test_planes_of_more_waves(so):
    for ny, nx in ((72, 64), (64, 72), (72, 72)):
        for nz, L, two in ((72, 1, True), (72, 2, False), (64, 3, True), (96, 3, False), (72, 5, False), (72, 6, True)):
            k = [x for x in _launches(so, (nz, ny, nx), (4,), (L,)) if "k2_" in x or "rhs" in x or "ifft" in x]
            assert len(k) == 5 and all(("k2_" in x) == two for x in k), (ny, nx, nz, L)


@pytest.mark.gpu
@pytest.mark.parametrize("ny,nx", [(72, 64), (64, 72)])
def test_planes_of_more_waves_match_oracle(wlc, oracle, ny, nx):
    # 648 planes and, after the junction, 288
    _matches_oracle(wlc, oracle, (72, ny, nx), (2, 2), (2, 1))


# 72 x 12, 16 and 24 planes: run-time kernels above 1280 planes
def test_thin_planes(so):
    for ny, nx, thin in ((72, 12, True), (12, 72, True), (72, 16, True), (16, 72, True), (72, 24, True),
                         (24, 72, True), (72, 18, False), (18, 72, False), (72, 32, False), (54, 12, False)):
        for nz, L in ((48, 4), (54, 4)):
            k = [x for x in _launches(so, (nz, ny, nx), (4,), (L,)) if "k2_" in x or "rhs" in x or "ifft" in x]
            assert len(k) == 5 and all(("k2_" in x) != (thin and nz == 54) for x in k), (ny, nx, nz)


@pytest.mark.gpu
@pytest.mark.parametrize("ny,nx", [(72, 12), (12, 72), (72, 16), (24, 72)])
def test_thin_planes_match_oracle(wlc, oracle, ny, nx):
    # 1350 planes and, after the junction, 486
    _matches_oracle(wlc, oracle, (54, ny, nx), (3, 3), (4, 2))


# a checkpointed sweep restarts with the kernel that only forms the right-hand side, and ends a segment
# with the one that only transforms back, where the first sweep ran the fused kernel: the recomputed slices
# and all that comes of them keep their bits, at a junction too
@pytest.mark.gpu
@pytest.mark.parametrize("shape,L", [((54, 72, 12), (4, 2)), ((54, 24, 72), (2, 4)), ((72, 64, 72), (2, 1)),
                                     ((36, 48, 72), (3, 2)), ((24, 36, 54), (3, 1))])
def test_recomputed_slices_keep_their_bits(wlc, monkeypatch, shape, L):
    monkeypatch.setenv("WLC_CONCURRENT", "0")
    w = 1.5 * np.random.default_rng(5).standard_normal((2,) + shape)
    res = []
    for k in (0, 3):
        g = wlc.WormlikeMDE(shape, (4.0, 3.5, 3.0), (6, 7), L, (1.0, 0.5), ckpt_every=k)
        g.set_w(w)
        g.MDE_q()
        g.MDE_qstar()
        res.append((*g.density(), g.get_q(+1, 13), g.get_q(-1, 0)))
        g.close()
    assert all(np.array_equal(a, b) for a, b in zip(*res))


@pytest.mark.gpu
@pytest.mark.parametrize("ny,nx", [(48, 72), (72, 48)])
def test_planes_of_five_waves_match_oracle(wlc, oracle, ny, nx):
    # 324 planes and, after the junction, 576
    _matches_oracle(wlc, oracle, (36, ny, nx), (3, 3), (2, 3))


# short z axes at Lmax 0, 1 (and 2 at nz = 8): the column kernel up to a number of column groups (four
# columns to nz = 16, else two), the generic kernel above
@pytest.mark.parametrize("nz,L,line,few,many", [
    (8, 0, 1024, (72, 108), (108, 72)), (12, 0, 1024, (72, 108), (108, 72)), (16, 1, 1024, (72, 108), (108, 72)),
    (24, 0, 1024, (72, 54), (64, 64)), (32, 1, 1024, (72, 54), (64, 64)), (48, 0, 640, (48, 48), (54, 48)),
    (36, 0, 640, (48, 48), (54, 48)), (48, 1, 1024, (72, 54), (64, 64)), (18, 1, 3072, (108, 108), (128, 96)),
    (54, 1, 1536, (72, 72), (108, 64)), (8, 2, 2048, (144, 108), (128, 128)), (36, 2, 4096, (128, 96), (128, 128)),
    (48, 2, 2048, (72, 72), (96, 96)),
])
def test_few_harmonics_many_columns(so, nz, L, line, few, many):
    cols = 4 if nz <= 16 else 2
    for (ny, nx), col in ((few, True), (many, False)):
        assert (-(-(nx // 2 + 1) // cols) * ny <= line) == col
        k = [x for x in _launches(so, (nz, ny, nx), (4,), (L,)) if "zcol" in x or "zsolve" in x]
        assert len(k) == 4 and all(("zcol" in x) == col for x in k), (ny, nx)
    # more harmonics: the column kernel at any number of columns
    k = [x for x in _launches(so, (nz, *many), (4,), (3,)) if "zcol" in x or "zsolve" in x]
    assert len(k) == 4 and all("zcol" in x for x in k)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,L", [((24, 64, 64), (0, 1)), ((8, 108, 72), (1, 0)), ((18, 128, 96), (1, 2)),
                                     ((8, 128, 128), (2, 3))])
def test_few_harmonics_many_columns_match_oracle(wlc, oracle, shape, L):
    _matches_oracle(wlc, oracle, shape, (3, 2), L)


# nz = 48, Lmax 7: the column kernel up to 960 column groups, a half-tile kernel above
def test_nz48_lmax7(so):
    for (ny, nx), col in (((54, 54), True), ((48, 72), True), ((72, 54), False), ((64, 64), False)):
        k = [x for x in _launches(so, (48, ny, nx), (4,), (7,)) if "zcol" in x or "zsolve" in x]
        assert len(k) == 4 and all(("zcol" in x) == col and ("zsolve48" in x) != col for x in k), (ny, nx)
    # other Lmax, and the FP32 spectrum: as at any number of columns
    for L, sp in ((6, False), (8, False), (7, True)):
        k = [x for x in _launches(so, (48, 64, 64), (4,), (L,), sp) if "zcol" in x or "zsolve" in x]
        assert len(k) == 4 and all("zsolve48" not in x and ("zcol" in x) != sp for x in k), (L, sp)


@pytest.mark.gpu
def test_nz48_lmax7_matches_oracle(wlc, oracle):
    # nxh = 33 and 37: a tile of one real column; blocks of the other Lmax take the column kernel
    for shape, L in (((48, 64, 64), (7,)), ((48, 64, 72), (7, 2))):
        _matches_oracle(wlc, oracle, shape, (3, 2)[:len(L)], L)


@pytest.mark.gpu
def test_nz48_lmax7_batched(wlc):
    # rows of half tiles in and out of the XCD order (2 nt ny a multiple of 16 or not)
    _batch_matches_handles(wlc, [((48, 64, 64), 7), ((48, 64, 64), 7), ((48, 54, 72), 7)])


# nz = 128: a column to each CU (Lmax 5, 6, with the FP32 spectrum to 8) up to 256 columns, with the
# FP32 spectrum at Lmax 5 and 6 beyond them too; the three-part kernel for the rest
@pytest.mark.parametrize("L,sp,few_cols,many_cols", [
    (5, False, True, False), (6, False, True, False), (7, False, False, False), (8, False, False, False),
    (5, True, True, True), (6, True, True, True), (7, True, True, False), (8, True, True, False)])
def test_nz128_two_parts(so, L, sp, few_cols, many_cols):
    for (ny, nx), few in (((64, 6), True), ((16, 24), True), ((72, 6), False), ((24, 24), False)):
        assert (ny * (nx // 2 + 1) <= 256) == few
        k = [x for x in _launches(so, (128, ny, nx), (4,), (L,), sp) if "z128" in x or "zsolve" in x]
        one = few_cols if few else many_cols
        assert len(k) == 4 and all(("k_zsolve128s" in x) == one and ("k_z128" in x) != one for x in k), (ny, nx)


# beyond 256 columns: a pair with one real column, a padding pair, whole tiles; Lmax changing at a
# junction; the FP32 spectrum at the bound of the short chains' tests
@pytest.mark.gpu
@pytest.mark.parametrize("ny,nx,L,spec32", [(72, 6, (5, 8), False), (54, 8, (6, 7), False), (48, 12, (8, 6), False),
                                            (54, 8, (7, 8), True), (48, 12, (7, 7), True)])
def test_nz128_three_parts_match_oracle(wlc, oracle, ny, nx, L, spec32):
    _matches_oracle(wlc, oracle, (128, ny, nx), (2, 3), L, spec32)


@pytest.mark.gpu
def test_nz128_two_parts_match_oracle(wlc, oracle):
    # more columns than CUs, rows of four-column tiles in the XCD order and not
    _matches_oracle(wlc, oracle, (128, 48, 12), (2, 3), (5, 6), spec32=True)
    _matches_oracle(wlc, oracle, (128, 54, 8), (2, 3), (6, 5), spec32=True)


@pytest.mark.gpu
def test_nz128_batched(wlc):
    _batch_matches_handles(wlc, [((128, 48, 12), 6), ((128, 48, 12), 6), ((128, 4, 12), 6), ((128, 4, 12), 5)])


# density runs of concurrent sweeps: two fifths of the terms left, of slices whose q fit in 64 MB
@pytest.mark.parametrize("nz,L,runs", [(48, 6, [1] * 13), (48, 5, [2, 2, 2, 1, 2, 2, 2]), (16, 3, [3, 2, 2, 3, 2, 1])])
def test_density_runs(so, nz, L, runs):
    out = host_hip.run(so, f"""
        g = W.WormlikeMDE(({nz}, 48, 48), (4.0, 4.0, 4.0), (12,), ({L},), (1.0,))
        g.set_w(np.zeros((1, {nz}, 48, 48)))
        g.MDE_q()
        H.host_hip_forget()
        g.MDE_qstar()
        print(sum("density_run" in k for k in launches()))
    """)
    assert int(out[0]) == len(runs)
