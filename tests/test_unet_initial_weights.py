"""The warm-start network's initial parameters: the normal deviates of the C++ library on a 64-bit
Mersenne twister, scaled by the real fan-in (on the host, with the HIP runtime replaced by a
recording one)."""
import os
import subprocess

import numpy as np
import pytest

import host_hip

DRAWS = """
#include <cstdio>
#include <cstdlib>
#include <random>
int main(int, char** a) {
  std::mt19937_64 rng(std::strtoull(a[1], nullptr, 10));
  std::normal_distribution<float> nd(0.f, 1.f);
  for (long i = std::atol(a[2]); i > 0; --i) {
    const float w = nd(rng);
    std::fwrite(&w, 4, 1, stdout);
  }
}
"""


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.fixture(scope="module")
def draws(tmp_path_factory):
    d = tmp_path_factory.mktemp("draws")
    src, exe = os.path.join(str(d), "draws.cpp"), os.path.join(str(d), "draws")
    with open(src, "w") as f:
        f.write(DRAWS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, src], check=True)
    return exe


@pytest.mark.parametrize("seed", [0, 3, 2**64 - 1])
def test_initial_parameters(so, draws, tmp_path, seed):
    out = os.path.join(str(tmp_path), "p.npy")
    lines = host_hip.run(so, f"""
        net = W.UNet(8, 1, seed={seed})
        np.save({out!r}, net.params())
        for l in net.layers():
            print(l["cin"], l["cout"], l["cin_real"], l["cout_real"], l["woff"], l["boff"])
        net.close()
    """)
    p = np.load(out)
    layers = [tuple(map(int, s.split())) for s in lines]
    n = sum(27 * ci * co for ci, co, *_ in layers)
    raw = np.frombuffer(subprocess.run([draws, str(seed), str(n)], capture_output=True, check=True).stdout, np.float32)
    want = np.zeros_like(p)
    at = 0
    for k, (ci, co, cir, cor, woff, boff) in enumerate(layers):
        # the scale is a C++ float expression: sqrt of the float quotient, the output layer's times 0.1
        sd = np.sqrt(np.float32(2) / np.float32(27 * cir)) * np.float32(0.1 if k == len(layers) - 1 else 1)
        w = (raw[at:at + 27 * ci * co].reshape(co, 27, ci) * np.float32(sd)).astype(np.float32)
        w[cor:] = 0
        w[:, :, cir:] = 0
        want[woff:woff + w.size] = w.reshape(-1)
        at += w.size
    assert np.array_equal(p, want)
