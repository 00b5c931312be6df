"""The marched stages (k_march, k_march_hd) against the separate launches: the same bits
in FP64 for every solver, limiter and precision mode, over block shapes at
the edges of the marched tiles, with per-block time steps, device-driven and
captured cycles, and states that hold NaN and huge values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

G = 3


def _ev():
    import enzoe_vlct as ev
    return ev


def _state(n, seed, dual=False, mhd=True):
    """A rough random state of one block (independent values in neighbouring
    cells: every branch of the solvers is taken somewhere)."""
    rng = np.random.default_rng(seed)
    m = [x + 2 * G for x in n[::-1]]
    a = {"density": np.exp(0.4 * rng.standard_normal(m))}
    for c in "xyz":
        a["velocity_" + c] = 0.7 * rng.standard_normal(m)
    for ax, c in zip((2, 1, 0), "xyz") if mhd else ():
        shp = list(m)
        shp[ax] += 1
        f = 0.5 * rng.standard_normal(shp) + (0.4 if c == "x" else 0.0)
        a["bfieldi_" + c] = f
        a["bfield_" + c] = 0.5 * (np.take(f, range(1, shp[ax]), ax)
                                  + np.take(f, range(shp[ax] - 1), ax))
    e = 1.5 * np.exp(0.3 * rng.standard_normal(m)) / a["density"]
    a["total_energy"] = e + 0.5 * sum(a["velocity_" + c] ** 2 for c in "xyz") \
        + 0.5 * sum(a["bfield_" + c] ** 2 for c in "xyz" if mhd) / a["density"]
    if dual:
        a["internal_energy"] = e
    return a


def _blocks(ev, n, states, count, dual=False, mhd=True):
    out = []
    for i in range(count):
        b = ev.DeviceBlock(n[0] + 2 * G, n[1] + 2 * G, n[2] + 2 * G, G,
                           (1.0 / n[0], 1.1 / n[1], 0.9 / n[2]), mhd=mhd, dual_energy=dual)
        b.upload(states[i % len(states)])
        out.append(b)
    return out


def _equal(xs, ys):
    for i, (x, y) in enumerate(zip(xs, ys)):
        a, b = x.download(), y.download()
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), (i, k)


# (block, count): from 2^18 active cells on (FP64 hydro: 3 2^17) the default is
# the marched launch; sides from one partial tile to several, of every tile
# size
SHAPES = [((32, 32, 32), 12), ((9, 8, 7), 781), ((13, 41, 29), 26), ((130, 57, 57), 1),
          ((70, 12, 50), 10), ((16, 16, 16), 96)]


@pytest.mark.parametrize("riemann,recon,dual", [("hlld", "plm", False), ("hlld", "nn", False),
                                                ("hlle", "plm_athena", False),
                                                ("hlld", "plm", True), ("hlle", "nn", True),
                                                ("hllc", "plm", False), ("hllc", "nn", False),
                                                ("hllc", "plm_athena", True)])
@pytest.mark.parametrize("n,count", SHAPES)
def test_marched_stages_equal_the_separate_launches(n, count, riemann, recon, dual):
    """Two steps with per-block dt (one block's step zero), the second with
    the CFL minimum fused: every field, ghost zones included, and the next
    dt equal bit for bit."""
    ev = _ev()
    mhd = riemann != "hllc"
    states = [_state(n, 100 + s, dual, mhd) for s in range(min(3, count))]
    dts = [2e-4 * (1 + (i % 4)) for i in range(count)]
    if count > 1:
        dts[1] = 0.0
    out, nxt = [], []
    for structure in (-1, 0):
        m = ev.VlctMethod(mhd=mhd, riemann=riemann, reconstruct=recon, theta=2.0, courant=0.4,
                          dual_energy_eta=0.001 if dual else None)
        m.set_fused_ct(structure)
        blocks = _blocks(ev, n, states, count, dual, mhd)
        ev.profiling(True)
        m.compute_dt(blocks, dts)
        nxt.append(m.compute_timestep(blocks, 1e-4))
        names = ev.profile_report()
        ev.profiling(False)
        assert ("k_march_nn" in names) == (structure == -1)
        out.append(blocks)
    assert nxt[0] == nxt[1]
    _equal(out[0], out[1])


@pytest.mark.parametrize("recon,dual,precision", [
    ("plm", False, "double"), ("nn", False, "double"), ("plm_athena", False, "double"),
    ("plm", True, "double"), ("nn", True, "double"), ("plm", False, "mixed"),
    ("plm", False, "fma")])
@pytest.mark.parametrize("n,count", [((1, 1, 1), 1), ((16, 16, 16), 1), ((9, 5, 3), 3),
                                     ((23, 7, 10), 2), ((2, 18, 33), 1)])
def test_tiled_stages_equal_the_separate_launches(n, count, recon, dual, precision):
    """Small hydrodynamic blocks, one launch a stage: per-block dt, the fused
    CFL, cells with NaN and huge values.  The same bits in FP64; the mixed
    and contracted builds within a few of their own roundings."""
    ev = _ev()
    states = [_state(n, 70 + s, dual, mhd=False) for s in range(count)]
    if precision == "double":
        states[0]["velocity_x"][-4, 3, 3] = np.nan
        states[-1]["velocity_z"][3, -5, 4] = 1.5e308
    prec = {"double": ev.ENZOE_PREC_DOUBLE, "mixed": ev.ENZOE_PREC_MIXED,
            "fma": ev.ENZOE_PREC_DOUBLE_FMA}[precision]
    dts = [2e-4 * (1 + i) for i in range(count)]
    if count > 2:
        dts[1] = 0.0
    out, nxt = [], []
    for structure in (-1, 0):
        m = ev.VlctMethod(mhd=False, riemann="hllc", reconstruct=recon, theta=2.0, courant=0.4,
                          precision=prec, dual_energy_eta=0.001 if dual else None)
        m.set_fused_ct(structure)
        blocks = _blocks(ev, n, states, count, dual, mhd=False)
        ev.profiling(True)
        m.compute_dt(blocks, dts)
        nxt.append(m.compute_timestep(blocks, 1e-4))
        names = ev.profile_report()
        ev.profiling(False)
        assert ("k_tile_nn" in names) == (structure == -1)
        out.append(blocks)
    if precision == "double":
        assert np.array_equal(*nxt, equal_nan=True)
        _equal(out[0], out[1])
        return
    # two steps, each two sums of some 30 rounded terms of the size of
    # the largest state value (about 10): 120 roundings
    tol = 120 * 10 * {"mixed": 2.0 ** -24, "fma": 2.0 ** -53}[precision]
    for x, y in zip(out[0], out[1]):
        a, b = x.download(), y.download()
        for k in a:
            assert np.abs(a[k] - b[k]).max() <= tol, k


@pytest.mark.parametrize("mhd", [True, False])
def test_marched_stages_spread_nan_and_huge_values_as_the_separate_launches(mhd):
    """Cells with NaN, infinities and magnitudes whose differences overflow
    take the limiter's general form: the same cells end non-finite, the
    others keep the same bits."""
    ev = _ev()
    n = (40, 36, 48)
    count = 4 if mhd else 6
    states = [_state(n, 7 + s, mhd=mhd) for s in range(4)]
    for s, (k, j, i) in enumerate([(9, 8, 7), (G, G, G), (30, 20, 44), (50, 41, 3)]):
        f = states[s]
        f["velocity_x"][k, j, i] = np.nan
        f["bfield_y" if mhd else "density"][k - 2, j, i] = np.inf
        f["velocity_z"][(k + 9) % 54, j, i] = 1.5e308
        f["velocity_z"][(k + 10) % 54, j, i] = -1.5e308
    out = []
    for structure in (-1, 0):
        m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                          theta=2.0, courant=0.4)
        m.set_fused_ct(structure)
        blocks = _blocks(ev, n, states, count, mhd=mhd)
        m.compute(blocks, 1e-4)
        m.compute_timestep(blocks, 1e-4)
        out.append(blocks)
    _equal(out[0], out[1])


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("precision", ["mixed", "fma"])
def test_marched_stages_of_the_contracted_builds_are_as_close_to_fp64(precision, mhd):
    """The mixed and contracted builds may fuse their flux arithmetic
    otherwise in another kernel: per field the marched result's L1 distance
    to the FP64 one is at most twice the separate launches' (both are sums
    of independent roundings of the same size)."""
    ev = _ev()
    n, count = (45, 33, 30), 9
    states = [_state(n, 50 + s, mhd=mhd) for s in range(3)]
    prec = {"mixed": ev.ENZOE_PREC_MIXED, "fma": ev.ENZOE_PREC_DOUBLE_FMA}[precision]
    res = []
    for p, structure in ((ev.ENZOE_PREC_DOUBLE, 0), (prec, 0), (prec, -1)):
        m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                          theta=1.5, courant=0.4, precision=p)
        m.set_fused_ct(structure)
        blocks = _blocks(ev, n, states, count, mhd=mhd)
        for _ in range(2):
            m.compute(blocks, 2e-4)
        res.append([b.download() for b in blocks])
    for k in ("density", "velocity_x", "velocity_y", "velocity_z", "total_energy",
              "bfieldi_x", "bfieldi_y", "bfieldi_z"):
        if k not in res[0][0]:
            continue
        ref = sum(np.abs(b[k]).sum() for b in res[0])
        d = [sum(np.abs(a[k] - b[k]).sum() for a, b in zip(r, res[0])) / ref for r in res[1:]]
        assert d[1] <= 2.0 * d[0] + 1e-17, (k, d)


def test_marched_cycles_on_the_device_and_from_a_graph_equal_host_driven_ones():
    """A 64^3 block: cycles enqueued without a graph, and graph replays with
    eager work of the same method between them, equal host-driven cycles."""
    ev = _ev()
    n = (64, 64, 64)
    state = _state(n, 3)
    grids = []
    for _ in range(3):
        m = ev.VlctMethod(mhd=True, riemann="hlld", reconstruct="plm", theta=2.0, courant=0.3)
        g = ev.DeviceGrid(m, (1, 1, 1), n, [(1.0 / 64,) * 3])
        g.upload_from([state])
        grids.append(g)
    host, dev, graph = grids
    t_stop, t = 1.0, 0.0
    for _ in range(6):
        t += host.cycle(t, t_stop)
    dev.evolve_device(0.0, t_stop, ncycles=6, max_calls=1)
    cg = graph.graph(0.0, t_stop, 2)
    scratch = _blocks(ev, (40, 40, 40), [_state((40, 40, 40), 5)], 5)
    for _ in range(3):
        cg.launch()
        graph.method.compute(scratch, 1e-4)
        ev.synchronize()
    assert cg.time() == t
    cg.destroy()
    s = (slice(G, -G),) * 3
    for other in (dev, graph):
        a, b = host.blocks[0].download(), other.blocks[0].download()
        for k in a:
            if k != "pressure":
                assert np.array_equal(a[k][s], b[k][s]), k


@pytest.mark.parametrize("mhd,dual", [(True, False), (True, True), (False, False), (False, True)])
@pytest.mark.parametrize("n,nblocks,bc", [
    ((5, 4, 3), (2, 1, 3), "periodic"), ((2, 7, 1), (3, 2, 1), "periodic"),
    ((33, 18, 9), (1, 2, 2), "periodic"), ((6, 5, 7), (1, 1, 1), "outflow")])
def test_refresh_copies_every_field(n, nblocks, bc, mhd, dual):
    """The refresh, two fields to a thread: every ghost element of every
    field against the index arithmetic in numpy, also for blocks thinner
    than the ghost zone, with an odd number of fields."""
    ev = _ev()
    count = nblocks[0] * nblocks[1] * nblocks[2]
    states = [_state(n, 40 + i, dual, mhd) for i in range(count)]
    blocks = _blocks(ev, n, states, count, dual, mhd)
    m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc",
                      dual_energy_eta=0.001 if dual else None)
    m.refresh(blocks, nblocks, (bc,) * 3)
    got = [b.download() for b in blocks]
    for i in range(count):
        at = (i % nblocks[0], i // nblocks[0] % nblocks[1], i // nblocks[0] // nblocks[1])
        for name, x in got[i].items():
            if name == "pressure":  # derived, not refreshed
                continue
            src, idx = [], []
            for a in range(3):      # x, y, z
                face = name == "bfieldi_" + "xyz"[a]
                N = n[a] * nblocks[a]
                e = np.arange(n[a] + 2 * G + face)
                p = at[a] * n[a] + e - G
                inside = (e >= G) & (e < G + n[a] + face)
                q = p % N if bc == "periodic" else np.clip(p, 0, N - 1 + face)
                last = face & (q == N)
                src.append(np.where(inside, at[a], np.where(last, nblocks[a] - 1, q // n[a])))
                idx.append(np.where(inside, e, np.where(last, G + n[a], q % n[a] + G)))
            b = (src[2][:, None, None] * nblocks[1] + src[1][:, None]) * nblocks[0] + src[0]
            want = np.stack([s[name] for s in states])[
                b, idx[2][:, None, None], idx[1][:, None], idx[0]]
            assert np.array_equal(x, want), (i, name)


@pytest.mark.parametrize("n", [(10, 9, 8), (25, 18, 21), (72, 70, 68)])
@pytest.mark.parametrize("recon,dual", [("nn", False), ("plm", False), ("plm_athena", False),
                                        ("plm", True)])
def test_one_stage_scheme_equals_the_oracle(recon, dual, n):
    """The one-stage ("euler") scheme updates the state in place, so its stage
    may not be one launch that solves the faces around the cells it updates:
    small and large hydrodynamic blocks against the oracle, and no tiled or
    marched launch."""
    from _states import random_periodic_grid
    from test_gpu_parity import device_copy
    ev = _ev()
    grid = random_periodic_grid(mhd=False, seed=3, n=n, riemann="hllc", recon=(recon,),
                                theta=1.6, vamp=0.6)
    assert grid.cfg.nstages == 1
    if dual:
        grid.cfg.dual_energy = 1
        grid.cfg.eta = 0.001
        arr = grid.block_arrays(0)
        arr["internal_energy"][...] = arr["total_energy"] - 0.5 * sum(
            np.square(arr["velocity_" + c]) for c in "xyz")
    c = grid.cfg
    m = ev.VlctMethod(mhd=False, riemann="hllc", reconstruct=recon, time_scheme="euler",
                      theta=c.theta_limiter, courant=c.courant, gamma=c.gamma,
                      density_floor=c.density_floor, pressure_floor=c.pressure_floor,
                      dual_energy_eta=c.eta if dual else None)
    dg = device_copy(grid, m)
    ev.profiling(True)
    t = 0.0
    for _ in range(3):
        dt = grid.cycle(t, 10.0)
        assert dg.cycle(t, 10.0) == dt
        t += dt
    names = ev.profile_report()
    ev.profiling(False)
    assert not any(k.startswith(("k_tile", "k_march")) for k in names)
    got, want = dg.blocks[0].download(), grid.block_arrays(0)
    for k in got:
        if k in want:
            assert np.array_equal(got[k], want[k]), k


def _names_of_a_step(ev, m, blocks, dt):
    ev.profiling(True)
    nxt = m.compute_timestep(blocks, dt)
    names = set(ev.profile_report())
    ev.profiling(False)
    return names, nxt


@pytest.mark.parametrize("mhd,n,tuned,called,kernel", [
    # one block tuned, a batch above the marched stages' size called, and the
    # other way round
    (True, (32, 32, 32), 1, 12, "k_march_nn"), (True, (20, 18, 16), 48, 1, "k_flux_nn"),
    (False, (32, 32, 32), 1, 14, "k_march_nn"), (False, (16, 16, 16), 60, 1, "k_tile_nn")])
def test_a_tuned_shape_keeps_the_choice_by_size_for_other_batches(mhd, n, tuned, called, kernel):
    """The autotuner's choice between separate launches and a whole stage as
    one holds for launches of the sample's size; a batch of another size
    of the same shape takes the one that its size asks for, with the same
    bits."""
    ev = _ev()
    states = [_state(n, 90 + s, mhd=mhd) for s in range(2)]
    out, nxt = [], []
    for tune in (True, False):
        m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                          theta=2.0, courant=0.4)
        if tune:
            m.autotune(_blocks(ev, n, states, tuned, mhd=mhd), 1e-4)
        else:
            m.set_fused_ct(0)
        blocks = _blocks(ev, n, states, called, mhd=mhd)
        names, dt = _names_of_a_step(ev, m, blocks, 1e-4)
        if tune:
            assert kernel in names, names
        nxt.append(dt)
        out.append(blocks)
    assert nxt[0] == nxt[1]
    _equal(out[0], out[1])


@pytest.mark.parametrize("mhd,dual,n,count", [(True, False, (32, 32, 32), 12),
                                              (False, False, (12, 12, 12), 1),
                                              (False, True, (24, 20, 16), 1)])
def test_tuned_batches_keep_their_results(mhd, dual, n, count):
    """At the sample's own size, whatever the autotuner chose: the same bits,
    and calls with debug counts still take the separate launches."""
    ev = _ev()
    states = [_state(n, 95 + s, dual, mhd) for s in range(2)]
    out = []
    for tune in (True, False):
        m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                          theta=2.0, courant=0.4, dual_energy_eta=0.001 if dual else None)
        blocks = _blocks(ev, n, states, count, dual, mhd)
        if tune:
            mask = m.autotune(blocks, 1e-4)
            assert m.launch_choice(tuple(x + 2 * G for x in n))[0] == mask
        else:
            m.set_fused_ct(0)
        m.compute(blocks, 1e-4)
        m.compute_timestep(blocks, 1e-4)
        if tune:
            m.set_debug_checks(True)
        names, _ = _names_of_a_step(ev, m, blocks, 1e-4)
        if tune:
            assert not any(k.startswith(("k_march", "k_tile")) for k in names)
        out.append(blocks)
    _equal(out[0], out[1])


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("mhd,n,count,kernel", [(True, (32, 32, 32), 12, "k_march_nn"),
                                                (False, (32, 32, 32), 14, "k_march_nn"),
                                                (False, (16, 14, 12), 2, "k_tile_nn")])
def test_gravity_in_whole_stage_launches(mhd, n, count, kernel, precision):
    """The acceleration of every cell added in the marched and tiled second
    stage, as in the separate one: the same bits."""
    ev = _ev()
    states = [_state(n, 60 + s, mhd=mhd) for s in range(2)]
    rng = np.random.default_rng(8)
    m3 = tuple(x + 2 * G for x in n[::-1])
    out = []
    acc = []
    for _ in range(count):
        buf = ev.DeviceBuffer(3 * 8 * int(np.prod(m3)))
        ev.to_device(buf.ptr.value, rng.standard_normal((3,) + m3))
        acc.append(buf)
    ptrs = [tuple(b.ptr.value + 8 * a * int(np.prod(m3)) for a in range(3)) for b in acc]
    for structure in (-1, 0):
        m = ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                          theta=1.5, courant=0.4,
                          precision=ev.ENZOE_PREC_MIXED if precision == "mixed"
                          else ev.ENZOE_PREC_DOUBLE)
        m.set_fused_ct(structure)
        blocks = _blocks(ev, n, states, count, mhd=mhd)
        ev.profiling(True)
        ev.compute_gravity(m, blocks, 2e-4, ptrs)
        names = ev.profile_report()
        ev.profiling(False)
        assert (kernel in names) == (structure == -1)
        out.append(blocks)
    _equal(out[0], out[1])
    plain = _blocks(ev, n, states, count, mhd=mhd)
    m.compute(plain, 2e-4)
    assert not np.array_equal(plain[0].download()["velocity_x"],
                              out[1][0].download()["velocity_x"])
