"""The mixed path rounds alike in every launch structure, and as it always has.

Its FP32 Riemann solves divide by differences that can cancel down to their
rounding, so that a multiply-add fused in one kernel and not in another can
change a cell by as much as it holds; a norm over the block cannot see that.
The states here take neighbouring cells independently, which puts such faces
into every block.  Every structure's result is compared bit for bit, cell by
cell, and the results' digests with those of the separate launches from before
the solves' multiply-adds were written out (three steps, every field and dt).
"""
import hashlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

G = 3
SOLVERS = [("hlld", "nn"), ("hlld", "plm"), ("hlld", "plm_athena"),
           ("hlle", "nn"), ("hlle", "plm"), ("hlle", "plm_athena"),
           ("hllc", "nn"), ("hllc", "plm"), ("hllc", "plm_athena")]
# (block, count): one small block, one and several above the marched stages'
# size (2^18 active cells), with partial tiles on every axis
SHAPES = [((19, 17, 23), 1), ((70, 66, 58), 1), ((33, 40, 30), 7)]


def _ev():
    import enzoe_vlct as ev
    return ev


def _state(n, seed, mhd):
    """Independent values in neighbouring cells, from the generator's uniform
    numbers by sums, products and quotients only (the same on every host)."""
    rng = np.random.default_rng(seed)
    m = [x + 2 * G for x in n[::-1]]

    def flat(shape, lo, hi):
        return lo + (hi - lo) * rng.random(shape)

    a = {"density": flat(m, 0.3, 2.5)}
    for c in "xyz":
        a["velocity_" + c] = flat(m, -1.4, 1.4)
    b2 = 0.0
    for ax, c in zip((2, 1, 0), "xyz") if mhd else ():
        shape = list(m)
        shape[ax] += 1
        f = a["bfieldi_" + c] = flat(shape, -1.0, 1.0) + (0.4 if c == "x" else 0.0)
        b = a["bfield_" + c] = 0.5 * (np.take(f, range(1, shape[ax]), ax)
                                      + np.take(f, range(shape[ax] - 1), ax))
        b2 = b2 + b * b
    a["total_energy"] = flat(m, 0.9, 2.4) / a["density"] + 0.5 * (
        a["velocity_x"] * a["velocity_x"] + a["velocity_y"] * a["velocity_y"]
        + a["velocity_z"] * a["velocity_z"]) + 0.5 * b2 / a["density"]
    return a


def _run(n, count, riemann, recon, pressure_floor=1e-10, structure=None, shape=None):
    """Three cycles (refresh, step, next dt): the fields of every block and
    the dts."""
    ev = _ev()
    mhd = riemann != "hllc"
    states = [_state(n, 31 + s, mhd) for s in range(min(3, count))]
    m = ev.VlctMethod(mhd=mhd, riemann=riemann, reconstruct=recon, theta=1.7, courant=0.3,
                      precision=ev.ENZOE_PREC_MIXED, pressure_floor=pressure_floor)
    if structure is not None:
        m.set_fused_ct(structure)
    if shape is not None:
        m.set_flux_shape(shape)
    blocks = []
    for i in range(count):
        b = ev.DeviceBlock(n[0] + 2 * G, n[1] + 2 * G, n[2] + 2 * G, G,
                           (1.0 / n[0], 1.1 / n[1], 0.9 / n[2]), mhd=mhd)
        b.upload(states[i % len(states)])
        blocks.append(b)
    ev.profiling(True)
    dt = m.timestep(blocks)
    dts = [dt]
    for _ in range(3):
        m.refresh(blocks, (count, 1, 1), ("periodic",) * 3)
        dt = m.compute_timestep(blocks, min(dt, 2e-3))
        dts.append(dt)
    names = ev.profile_report()
    ev.profiling(False)
    return [b.download() for b in blocks], dts, names


def _equal(xs, ys):
    for i, (x, y) in enumerate(zip(xs, ys)):
        for k in x:
            assert np.array_equal(x[k], y[k], equal_nan=True), (i, k)


@pytest.mark.parametrize("n,count", SHAPES)
@pytest.mark.parametrize("riemann,recon", SOLVERS)
def test_mixed_default_launches_equal_the_separate_ones(riemann, recon, n, count):
    """The default (marched, or for a small block tiled, face-split and fused
    launches) against one thread a cell and separate launches."""
    got, dts, names = _run(n, count, riemann, recon)
    want, dts0, names0 = _run(n, count, riemann, recon, structure=0, shape=0)
    if count > 1 or n[0] > 32:
        assert "k_march_nn" in names
    assert "k_flux_nn" in names0 and "k_march_nn" not in names0
    assert dts == dts0
    _equal(got, want)


@pytest.mark.parametrize("riemann,recon", SOLVERS)
def test_mixed_z_pencils_and_fused_updates_equal_the_separate_launches(riemann, recon):
    n = (26, 19, 21)
    want, dts0, _ = _run(n, 2, riemann, recon, structure=0, shape=0)
    for structure in (0, 1, 2, 3, 4, 5) if riemann != "hllc" else (0, 5):
        for shape in (1, 2):
            got, dts, _ = _run(n, 2, riemann, recon, structure=structure, shape=shape)
            assert dts == dts0
            _equal(got, want)


# sha256 (first 16 digits) over the fields in name order, block by block, and
# the dts; the second of each pair with a pressure floor that many cells meet
DIGESTS = {
    ("hlld", "nn", (19, 17, 23)): ("5a2dd3c9d65686bf", "8853c08dd2bf0786"),
    ("hlld", "nn", (70, 66, 58)): ("3e75bbc7e2b41ca3", "b8a285662f793fda"),
    ("hlld", "nn", (33, 40, 30)): ("e00e3489f5b5494d", "f54e052c7ddfac3c"),
    ("hlld", "plm", (19, 17, 23)): ("e7832af8061a1f59", "27a7c7c0ab85d8b3"),
    ("hlld", "plm", (70, 66, 58)): ("47b9c4f4dc5ef72d", "7ac0146ab2926cd0"),
    ("hlld", "plm", (33, 40, 30)): ("e2756a3e500b82cc", "4df993e3cd4e8547"),
    ("hlld", "plm_athena", (19, 17, 23)): ("255056c508f0cb0b", "7ac7fc04656c52cc"),
    ("hlld", "plm_athena", (70, 66, 58)): ("c159d71235af70d9", "f836276953b6bd8f"),
    ("hlld", "plm_athena", (33, 40, 30)): ("0262cd6d3aeb15ff", "36396d4d9d26ff50"),
    ("hlle", "nn", (19, 17, 23)): ("2d96a1dfb1b64195", "57ef70d9ba484cb6"),
    ("hlle", "nn", (70, 66, 58)): ("4392778c5d65af0a", "467a66b47a32cc5f"),
    ("hlle", "nn", (33, 40, 30)): ("29544bb2348f69c0", "5ea88460bcf98ab2"),
    ("hlle", "plm", (19, 17, 23)): ("9e39a6044b9ef9bf", "69745e7539a81343"),
    ("hlle", "plm", (70, 66, 58)): ("bb7f210aa6091234", "c89876a0643280dc"),
    ("hlle", "plm", (33, 40, 30)): ("11db75e08740570e", "90502497c2185fe7"),
    ("hlle", "plm_athena", (19, 17, 23)): ("af11ae33805642ce", "ea1eac069aaee161"),
    ("hlle", "plm_athena", (70, 66, 58)): ("a3c4b86b8b0a6fbc", "15ffa57eff3d7466"),
    ("hlle", "plm_athena", (33, 40, 30)): ("ac16ed605bdcc316", "522513be2e9805c5"),
    ("hllc", "nn", (19, 17, 23)): ("443d2886a80f3505", "72b8de89fd1ac5e9"),
    ("hllc", "nn", (70, 66, 58)): ("8ea80cc90be6348f", "b2d6ba6412840826"),
    ("hllc", "nn", (33, 40, 30)): ("85317cf46aa4f5e5", "18f2f395e0ea6ff9"),
    ("hllc", "plm", (19, 17, 23)): ("071fdd9f40b22d99", "35c7d23f7deb9c85"),
    ("hllc", "plm", (70, 66, 58)): ("a2d9e4a512fbe7cd", "cc53b163d45b9500"),
    ("hllc", "plm", (33, 40, 30)): ("baad021f1b8fe7da", "deb66cf780cb7864"),
    ("hllc", "plm_athena", (19, 17, 23)): ("09628225adcc029f", "de24abea6763dc41"),
    ("hllc", "plm_athena", (70, 66, 58)): ("b324a9d37f0d8b1d", "5872dc011c9247aa"),
    ("hllc", "plm_athena", (33, 40, 30)): ("07689eb4390c8041", "d8e3c37e92c3073f"),
}


def _digest(fields, dts):
    h = hashlib.sha256()
    for block in fields:
        for k in sorted(block):
            h.update(np.ascontiguousarray(block[k]).tobytes())
    h.update(np.array(dts).tobytes())
    return h.hexdigest()[:16]


@pytest.mark.parametrize("n,count", SHAPES)
@pytest.mark.parametrize("riemann,recon", SOLVERS)
def test_mixed_results_keep_their_bits(riemann, recon, n, count):
    got = tuple(_digest(*_run(n, count, riemann, recon, floor)[:2]) for floor in (1e-10, 0.8))
    assert got == DIGESTS[riemann, recon, n]
