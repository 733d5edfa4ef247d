"""A handle creates the streams it works on and no other: each further one can make two of them share a
hardware queue, of which a process has four (on the host, calls recorded)."""
import pytest

import host_hip


@pytest.mark.parametrize("kw,concurrent", [("", "1"), ("ckpt_every=8", "1"), ("ckpt_every=8", "0")])
def test_three_streams(tmp_path, kw, concurrent):
    out = host_hip.run(host_hip.build(tmp_path), f"""
        before = H.host_hip_streams()
        g = W.WormlikeMDE((8, 12, 16), (4., 4., 4.), (24,), (2,), (1.,), {kw})
        g.set_w(np.zeros((1, 8, 12, 16)))
        g.MDE_q()
        g.MDE_qstar()
        print(H.host_hip_streams() - before)
    """, env={"WLC_CONCURRENT": concurrent})
    assert out == ["3"]
