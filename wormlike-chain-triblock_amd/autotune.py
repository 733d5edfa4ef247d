"""Autotuner of kernel B (z FFT + k-aligned solve + inverse z FFT) variants.

For each (nz, Lmax, spectrum precision) every admissible variant of kernel B is timed on
the device inside a short forward + backward sweep (per-launch HIP events, timing mode 2:
each step kernel with the GPU to itself) on a cubic grid of edge nz, and the fastest is
written to csrc/wlc_tune.inc, the table the library compiles in (wlc_tune.cpp).  Variants:
the one-wave nz = 64 kernel at one or two waves per SIMD, the degree-split two-column and
whole-tile nz = 64 kernels (Lmax 5-7), the column kernel of the short axes (nz = 24, 32, 48),
the nz = 128 kernels (whole columns; three degree parts at Lmax 5-8), and the generic kernel with
every admissible number of kx columns per workgroup, with and without the degree split
(Lmax 4-7).  Candidates are selected through the library's measurement switches
(WLC_GENERIC_ZSOLVE, WLC_ZSOLVE_SPLIT, WLC_ZSOLVE_OCC, WLC_ZSOLVE_TX).

usage: python autotune.py [out.inc] [nz,nz,...]   (needs a GPU; prints one line per timed
variant; with a list of nz only those edges are tuned)
"""
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

# (nz, Lmax values, spectrum precisions): the grids and Lmax of the batched instances, the
# 64^3 benchmark, the 128^3 precision workload
SPACE = [
    (24, (4, 6), (0,)),
    (32, (4, 6), (0,)),
    (48, (4, 6), (0,)),
    (64, (4, 5, 6, 7, 8), (0,)),
    (64, (6,), (1,)),
    (128, (6, 7, 8), (0,)),
    (128, (8,), (1,)),
]
SWITCHES = ("WLC_GENERIC_ZSOLVE", "WLC_ZSOLVE_SPLIT", "WLC_ZSOLVE_OCC", "WLC_ZSOLVE_TX")


def candidates(nz, L):
    """(generic, split, occ, tx) variants the library accepts for this nz and Lmax."""
    out = []
    split_ok = 4 <= L <= 7
    if nz == 64:
        out += [(0, 0, 1, 1), (0, 0, 2, 1)]
        if 5 <= L <= 7:
            out += [(0, 1, 1, 1), (0, 2, 1, 1), (0, 3, 1, 1)]
    if nz in (24, 32, 48) and 4 <= L <= 7:
        out += [(0, 3, 1, 1)]
    if nz == 128:
        out += [(0, 0, 1, 1)]
        if 5 <= L <= 8:
            out += [(0, 1, 1, 1)]
    # kx columns per workgroup: at least one wave, at most 256 threads per part; the smallest,
    # the library's built-in choice min(4, 256 / nz) (at least one wave), and the doublings
    tmin = max(1, -(-64 // nz))
    txs = {tmin, max(min(4, 256 // nz), tmin)}
    tx = tmin
    while tx * nz <= 256:
        txs.add(tx)
        tx *= 2
    for tx in sorted(t for t in txs if t * nz <= 256):
        out.append((1, 0, 1, tx))
        if split_ok and 2 * tx * nz <= 512:
            out.append((1, 1, 1, tx))
    return out


def time_variant(W, nz, L, spec32, var, Nblk=(4, 4, 4)):
    gen, split, occ, tx = var
    env = dict(zip(SWITCHES, (str(gen), str(split), str(occ), str(tx))))
    old = {k: os.environ.get(k) for k in SWITCHES}
    os.environ.update(env)
    try:
        rng = np.random.default_rng(3)
        w = rng.standard_normal((3, nz, nz, nz))
        g = W.WormlikeMDE((nz,) * 3, (4.0,) * 3, Nblk, (L,) * 3, (1.0,) * 3,
                          spectrum_fp32=bool(spec32))
        g.set_w(w)
        g.MDE_q()
        g.MDE_qstar()
        g.density_device()
        g.set_timing(2)
        for _ in range(2):
            g.MDE_q()
            g.MDE_qstar()
            g.density_device()
        ms, cnt = g.get_timing()
        g.set_timing(0)
        g.close()
        return 1e3 * ms[1] / cnt[1]
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def main():
    import wlc_mde as W
    out = sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "csrc", "wlc_tune.inc")
    only = {int(x) for x in sys.argv[2].split(",")} if len(sys.argv) > 2 else None
    rows = []
    for nz, Ls, precs in SPACE:
        if only and nz not in only:
            continue
        for L in Ls:
            for sp in precs:
                best = None
                for var in candidates(nz, L):
                    try:
                        us = time_variant(W, nz, L, sp, var)
                    except W.WlcError as e:
                        print(f"nz {nz} L {L} fp32 {sp} {var}: rejected ({e})", flush=True)
                        continue
                    print(f"nz {nz} L {L} fp32 {sp} generic {var[0]} split {var[1]} occ {var[2]} "
                          f"tx {var[3]}: {us:.1f} us", flush=True)
                    if best is None or us < best[1]:
                        best = (var, us)
                if best:
                    rows.append((nz, L, sp) + best[0] + (best[1],))
    with open(out, "w") as f:
        f.write("// generated by autotune.py: nz, L, spec32, generic, split, occ, tx, measured us\n")
        for r in rows:
            f.write("    {%d, %d, %d, %d, %d, %d, %d, %.1f},\n" % r)
    print(f"wrote {len(rows)} rows to {out}", flush=True)


if __name__ == "__main__":
    main()
