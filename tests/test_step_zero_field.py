"""The zero field of wlc_mde_step_noalloc after calls that have written over its place: the array
holds one zero field and then the half spectrum of the step at hand, so a step on a smaller grid with
many harmonics leaves its spectrum where a larger grid's zero field comes to lie.  Steps that miss
history read zeros there all the same, through every family of plane kernel."""
import numpy as np
import pytest

import host_hip

BOX, NBLK, L, LAM = (3.0, 2.5, 4.0), (4, 5), (2, 4), (1.0, 0.5)
# order 1, order 2, the junction 9 -> 25 harmonics with one, two and three short slices, backward order 2
STEPS = ((1, 1), (1, 2), (1, 5), (1, 6), (1, 7), (-1, 7))
# run-time passes, two passes with run-time and compile-time edges, 24^2, 32^2, 64^2, 128^2
SHAPES = [(6, 12, 6), (8, 16, 24), (2, 48, 48), (4, 24, 24), (4, 32, 32), (4, 64, 64), (4, 128, 128)]
DIRT = ((8, 16, 16), (2, 8, 8))  # the larger first: together they cover a tested field but 1 KB


def _zero_bytes(shape):
    return (8 * int(np.prod(shape)) + 255) // 256 * 256


def _spectrum_bytes(shape, lmax):
    nz, ny, nx = shape
    return 16 * (lmax + 1) ** 2 * ny * ((nx // 2 + 4) // 4) * 4 * nz


def _block(s):
    return 0 if s <= NBLK[0] else 1


@pytest.mark.parametrize("shape", SHAPES)
def test_calls_before_have_written_there(shape):
    end = _zero_bytes(shape)
    done = _zero_bytes(DIRT[1])
    assert done <= 1024 < end
    for d in reversed(DIRT):
        if _zero_bytes(d) <= done:
            done = max(done, _zero_bytes(d) + _spectrum_bytes(d, 8))
    assert done >= end


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_missing_history_reads_zeros(wlc, shape):
    from hipmem import DeviceArray, Stream
    rng = np.random.default_rng(sum(shape))
    M = [(l + 1) ** 2 for l in L]
    st = Stream()
    dirt = []
    for big in DIRT:
        dirt.append((wlc.make_params(big, BOX, (9,), (8,), (1.0,)),
                     [DeviceArray(rng.standard_normal((81,) + big)) for _ in range(3)],
                     DeviceArray(rng.standard_normal((1,) + big)), DeviceArray(shape=(81,) + big)))
    p = wlc.make_params(shape, BOX, NBLK, L, LAM)
    w = DeviceArray(rng.standard_normal((2,) + shape))
    g = wlc.WormlikeMDE(shape, BOX, NBLK, L, LAM)
    for d, s in STEPS:
        order = min(s, 3) if d > 0 else min(sum(NBLK) - s, 3)
        for q, h, wq, out in dirt:
            wlc.step_noalloc(q, 1, 5, [x.ptr for x in h], wq.ptr, out.ptr, st.ptr)
        hist = [DeviceArray(rng.standard_normal((M[_block(s - d * (j + 1))],) + shape)) for j in range(order)]
        ptrs = [x.ptr for x in hist] + [None] * (3 - order)
        a, b = (DeviceArray(shape=(M[_block(s)],) + shape) for _ in range(2))
        wlc.step_noalloc(p, d, s, ptrs, w.ptr, a.ptr, st.ptr)
        st.sync()
        g.step_device(d, s, ptrs, w.ptr, b.ptr)
        g.sync()
        assert np.array_equal(a.get(), b.get()), (d, s)
    g.close()
    st.close()


def test_cleared_for_the_steps_that_read_it(tmp_path):
    """On the host: the clear goes before the three kernels of exactly the steps that miss history."""
    out = host_hip.run(host_hip.build(tmp_path), """
        for L in ((2, 4), (4, 2)):
            p = W.make_params((8, 16, 24), (3.0, 2.5, 4.0), (4, 5), L, (1.0, 0.5))
            for d, s in [(1, s) for s in range(1, 10)] + [(-1, s) for s in range(8, -1, -1)]:
                H.host_hip_forget()
                W.step_noalloc(p, d, s, [64, 64, 64], 64, 64, None)
                k = launches()
                print(len(k) - 3, int("k_fill" in k[0]), sum("k_fill" in x for x in k))
    """)
    got = [int(l.split()[0]) for l in out]
    assert all(l.split() == [l.split()[0]] * 3 for l in out)
    # forward s = 1 .. 9, backward s = 8 .. 0; block 0 holds s <= 4
    grow = [1, 1, 0, 0, 1, 1, 1, 0, 0] + [1, 1, 0, 0, 0, 0, 0, 0, 0]
    back = [1, 1, 0, 0, 0, 0, 0, 0, 0] + [1, 1, 0, 0, 1, 1, 1, 0, 0]
    assert got == grow + back
