"""Fields that are on the GPU already go into the handle's layout by one strided copy each, with no
second pass over them (on the host, calls recorded)."""
import host_hip


def test_fields_from_device_memory(tmp_path):
    out = host_hip.run(host_hip.build(tmp_path), """
        g = W.WormlikeMDE((8, 12, 16), (4., 4., 4.), (4, 5), (2, 3), (1., 1.))
        w = ctypes.c_void_p()
        n = 2 * 8 * 12 * 16
        H.hipMalloc(ctypes.byref(w), ctypes.c_size_t(8 * n))
        H.host_hip_forget()
        g.set_w_device(w.value)
        print(H.host_hip_copies(0), H.host_hip_copies(1), len(launches()), H.host_hip_bad())
        # memory that ends before the last field does is refused
        try:
            g.set_w_device(w.value + 8)
        except W.WlcError as e:
            print(e.code)
    """)
    assert out == ["0 2 0 0", "-3"]
