"""Device memory of a checkpointed handle: the two segment buffers hold the slices a segment computes,
its restart history being read where it is kept (on the host, allocations recorded)."""
import pytest

import host_hip


@pytest.mark.parametrize("K,Ns,stored", [(8, 24, 0), (3, 20, 0), (5, 23, 2), (16, 12, 0)])
def test_segment_buffers_hold_a_segment(tmp_path, K, Ns, stored):
    nz, ny, nx, L = 12, 8, 16, 3
    out = host_hip.run(host_hip.build(tmp_path), f"""
        g = W.WormlikeMDE(({nz}, {ny}, {nx}), (4., 4., 4.), ({Ns},), ({L},), (1.,), ckpt_every={K})
        g.set_w(np.zeros((1, {nz}, {ny}, {nx})))
        g.MDE_q(); g.MDE_qstar()
        print(*[H.host_hip_alloc_bytes(i) for i in range(H.host_hip_allocs())])
    """, env={"WLC_STORED_SEGMENTS": str(stored)})
    # a slice: (L + 1)^2 harmonics of nz padded planes
    slot = 8 * (L + 1) ** 2 * (nz * (nx * ny + 16) + 32)
    slots = [b // slot for b in map(int, out[0].split()) if b % slot == 0]
    nseg = -(-Ns // K)
    nck = nseg - (stored + 1 if stored else 1)
    want = [4, 4, 1, K + 1, K + 1]  # the two rings, q(Ns), the segment buffers
    want += [stored * K + 1] if stored else []
    want += [3 * nck] if nck > 0 else []
    assert sorted(slots) == sorted(want)
