"""A resize of the warm-start network that runs out of memory leaves a network that refuses to run
until a resize succeeds, and touches no memory that is not its own (on the host, with the HIP
runtime replaced by a recording one)."""
import pytest

import host_hip


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


def test_failed_resize_refuses_until_the_next_one(so):
    out = host_hip.run(so, """
        net = W.UNet(16, 1, seed=3)
        x = np.zeros((1, 16, 16, 16, 11), np.float32)
        t = np.zeros((1, 16, 16, 16, 3), np.float32)
        net.forward(x)
        p = net.params()
        H.host_hip_fail(1)
        def code(f):
            try:
                f()
            except W.WlcError as e:
                return e.code
            return 0
        print(code(lambda: net.resize(24, 2)))
        H.host_hip_forget()
        print(code(lambda: net.forward(x)), code(lambda: net.gradients(x, t)),
              code(lambda: net.train_step(x, t, 1e-3)))
        print(len(launches()), H.host_hip_bad())
        # parameters are kept, and the next resize brings the network back
        print(np.array_equal(net.params(), p))
        print(code(lambda: net.resize(16, 1)), code(lambda: net.forward(x)), code(lambda: net.gradients(x, t)))
        net.close()
        print(H.host_hip_bad(), sum(H.host_hip_alloc_live(i) for i in range(H.host_hip_allocs())))
    """)
    assert out == ["-2", "-4 -4 -4", "0 0", "True", "0 0 0", "0 0"]
