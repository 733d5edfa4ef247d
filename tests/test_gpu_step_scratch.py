"""wlc_mde_step_noalloc clears its zero field only for the steps that read it: steps that miss
history (BDF order below 3, a junction that grows the basis) after a call that left other data
there, through every family of plane kernel, equal the handle's step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(8, 16, 24), (6, 12, 6), (4, 64, 64), (4, 32, 32)]


@pytest.mark.parametrize("shape", SHAPES)
def test_missing_history_reads_zeros(wlc, shape):
    from hipmem import DeviceArray, Stream
    box, Nblk, L, lam = (3.0, 2.5, 4.0), (4, 5), (2, 4), (1.0, 0.5)
    rng = np.random.default_rng(sum(shape))
    M = [(l + 1) ** 2 for l in L]
    block = lambda s: 0 if s <= Nblk[0] else 1
    st = Stream()
    # a full step of another size fills the scratch
    big = (16, 48, 48)
    p = wlc.make_params(big, box, Nblk, (4, 4), lam)
    h = [DeviceArray(rng.standard_normal((25,) + big)) for _ in range(3)]
    w = DeviceArray(rng.standard_normal((2,) + big))
    out = DeviceArray(shape=(25,) + big)
    p1 = wlc.make_params(shape, box, Nblk, L, lam)
    w1 = DeviceArray(rng.standard_normal((2,) + shape))
    # order 1, order 2, the junction 9 -> 25 harmonics with one and two short slices, backward order 2
    for d, s in ((1, 1), (1, 2), (1, 5), (1, 6), (-1, 7)):
        order = min(s, 3) if d > 0 else min(sum(Nblk) - s, 3)
        wlc.step_noalloc(p, 1, 8, [x.ptr for x in h], w.ptr, out.ptr, st.ptr)
        hist = [DeviceArray(rng.standard_normal((M[block(s - d * (j + 1))],) + shape)) for j in range(order)]
        ptrs = [x.ptr for x in hist] + [None] * (3 - order)
        a, b = (DeviceArray(shape=(M[block(s)],) + shape) for _ in range(2))
        wlc.step_noalloc(p1, d, s, ptrs, w1.ptr, a.ptr, st.ptr)
        st.sync()
        g = wlc.WormlikeMDE(shape, box, Nblk, L, lam)
        g.step_device(d, s, ptrs, w1.ptr, b.ptr)
        g.sync()
        g.close()
        assert np.array_equal(a.get(), b.get()), (d, s)
    st.close()
