"""FP32 cell-relative form against the FP64 oracle.

The FP32 form stores an integer cell plus FP32 offsets and u = gamma v, and
evaluates push and deposit in FP32 (FP64 grid sums, axis cell, fields).  It
cannot be bit-compatible with the reference; its contract is accuracy:
  * packing an FP64 state and unpacking it again loses only FP32 rounding of
    the in-cell offset and of u;
  * one step from identical state agrees with FP64 to FP32 round-off;
  * after 100 steps of the 64x256 configuration, E_z has a relative RMS error
    of at most 1e-4 against the oracle (the precision target), E_r and H_phi
    at most 1e-3, and J_z, J_r (which carry the particles' individual rounding
    rather than a field's average) at most 1e-2.
The reduced copies of cfg2, cfg3 and cfg4 are compared with the oracle in
test_gpu_configs.py; bench.py reports cfg3's E_z error after its 1000 steps
on the full grid against the GPU's FP64 form with the strict-radial
precedence fix, and against the plain FP64 form beside it.
"""
import numpy as np
import pytest

from helpers import normwise, oracle_from_workload

pytestmark = pytest.mark.gpu


def rel_rms(a, ref):
    den = np.sqrt(np.mean(ref ** 2))
    return float(np.sqrt(np.mean((a - ref) ** 2)) / den) if den > 0 else float(np.sqrt(np.mean(a ** 2)))


def test_pack_unpack_roundtrip():
    from pdp3_amd import capi

    rng = np.random.default_rng(21)
    nr, nz, dr = 33, 129, 5e-4
    sim = capi.Simulation(nr, nz, 32 * dr, 128 * dr, 0.5 * dr / 3e8, precision=capi.PREC_FP32)
    n = 5000
    r = rng.uniform(dr / 2, 31.5 * dr, n)
    z = rng.uniform(dr / 2, 127.5 * dr, n)
    v = rng.standard_normal((3, n)) * 2e7
    w = rng.uniform(1e3, 1e6, n)
    idx = sim.add_plasma(-1, 1.0, r, z, v[0], v[1], v[2], w)
    out = sim.download(idx)
    assert np.all(np.abs(out["r"] - r) <= dr * 2.0 ** -23)
    assert np.all(np.abs(out["z"] - z) <= dr * 2.0 ** -23)
    for j, k in enumerate(("vr", "vphi", "vz")):
        assert normwise(out[k], v[j]) <= 3e-7
    assert normwise(out["w"], w) <= 1e-7
    assert np.all(out["alive"] == 1)


@pytest.mark.parametrize("pusher", [0, 1])
def test_one_step_against_fp64(pusher, orc):
    """One full step of plasma in random fields: FP32 and FP64 particle
    states agree to FP32 round-off (relative ~1e-6)."""
    from pdp3_amd import capi

    rng = np.random.default_rng(22 + pusher)
    nr, nz, dr = 33, 129, 5e-4
    dt = 0.5 * dr / 3e8
    sims = [capi.Simulation(nr, nz, 32 * dr, 128 * dr, dt, pusher=pusher, precision=p)
            for p in (capi.PREC_FP64, capi.PREC_FP32)]
    fields = {name: rng.standard_normal((nr, nz)) * (3e4 if name[0] == "E" else 30.0)
              for name in ("E_r", "E_phi", "E_z", "H_r", "H_phi", "H_z")}
    n = 20000
    r = rng.uniform(dr / 2, 31.5 * dr, n)
    z = rng.uniform(dr / 2, 127.5 * dr, n)
    v = rng.standard_normal((3, n)) * 3e7
    w = rng.uniform(1e3, 1e6, n)
    for s in sims:
        for name, a in fields.items():
            s.set_field(name, a)
        s.add_plasma(-1, 1.0, r, z, v[0], v[1], v[2], w)
        s.step(1)
    a, b = sims[0].download(0), sims[1].download(0)
    errs = {k: normwise(b[k], a[k]) for k in ("r", "z", "vr", "vphi", "vz")}
    jerr = {k: normwise(sims[1].field(k), sims[0].field(k)) for k in ("J_r", "J_phi", "J_z")}
    print("particles", errs, "currents", jerr)
    assert np.array_equal(a["alive"], b["alive"])
    for k, e in errs.items():
        assert e <= 2e-6, (k, e)
    for k, e in jerr.items():
        assert e <= 1e-4, (k, e)


@pytest.mark.parametrize("axis", ["z", "r"])
def test_face_crossing_below_fp32_resolution(axis):
    """Particles 4.2e-9 cells above a cell face move 5e-9 cells across it
    (and 0.01 cells along the other axis): the new offset, 1 - 8e-10 in the
    cell below, is 1.0f, so the displacement in cell units rounds to 0 while
    the cell index changes.  The deposit must stay finite (it once divided by
    that zero) and carry the current of the move that FP32 keeps (the 4.2e-9
    cells up to the face); the run stays finite.  Against the FP64 form:
      * the 0.01-cell component (J_r for the z crossing, J_z for the r
        crossing) to 1e-4 normwise;
      * the crossing component for the z crossing to 0.3 (FP64 puts 16% of it,
        the 0.8e-9 cells past the face, in the cell below);
      * the crossing component for the r crossing only in size (at most 1e-3
        of the other component): the reference's J_r formula takes it as the
        difference of O(r dz) terms and log((r + dr) / r) of a ratio within
        1e-10 of 1, so the FP64 form's value is round-off at this step
        (src/particles.cpp simple_current_distribution)."""
    from pdp3_amd import capi

    rng = np.random.default_rng(31)
    nr, nz, dr = 33, 129, 5e-4
    dt = 0.5 * dr / 3e8
    n = 4096
    i = rng.integers(3, 29, n)
    k = rng.integers(3, 125, n)
    r = (i + rng.uniform(0.1, 0.9, n)) * dr
    z = (k + rng.uniform(0.1, 0.9, n)) * dr
    v = np.zeros((3, n))
    speed = 5e-9 * dr / dt  # 5e-9 cells per step
    if axis == "z":
        z = (k + 4.2e-9) * dr
        v[2] = -speed
        v[0] = 2e6 * speed  # 0.01 cells per step
        cross, other = "J_z", "J_r"
    else:
        r = (i + 4.2e-9) * dr
        v[0] = -speed
        v[2] = 2e6 * speed
        cross, other = "J_r", "J_z"
    w = np.full(n, 1e6)
    sims = [capi.Simulation(nr, nz, 32 * dr, 128 * dr, dt, precision=p) for p in (capi.PREC_FP64, capi.PREC_FP32)]
    for s in sims:
        s.add_plasma(-1, 1.0, r, z, v[0], v[1], v[2], w)
        s.step(1)
    for name in ("J_r", "J_phi", "J_z"):
        assert np.all(np.isfinite(sims[1].field(name))), name
    e_other = normwise(sims[1].field(other), sims[0].field(other))
    print(axis, other, "FP32 vs FP64", e_other)
    assert e_other <= 1e-4, e_other
    if axis == "z":
        e = normwise(sims[1].field(cross), sims[0].field(cross))
        print(axis, cross, "FP32 vs FP64", e)
        assert e <= 0.3, e
    else:
        ratio = np.max(np.abs(sims[1].field(cross))) / np.max(np.abs(sims[1].field(other)))
        print(axis, cross, "max relative to", other, ratio)
        assert ratio <= 1e-3, ratio
    sims[1].step(3)
    for name in ("E_r", "E_phi", "E_z", "H_r", "H_phi", "H_z", "J_r", "J_phi", "J_z"):
        assert np.all(np.isfinite(sims[1].field(name))), name
    out = sims[1].download(0)
    for key in ("r", "z", "vr", "vphi", "vz"):
        assert np.all(np.isfinite(out[key])), key
    for s in sims:
        s.close()


@pytest.mark.parametrize("direction", [-1, 1])
def test_strict_radial_crossing_precedence(direction):
    """Purely radial moves (v_z = 0) of 0.01 cells across a radial face take
    the reference's strict_motion_weighting, whose crossing branch parses
    `r0 * r0 / i_n * dr` as ((r0^2)/i_n) dr (src/particles.cpp:941, :976).
    With pdp3_set_strict_radial_fix the FP64 form evaluates r0^2/(i_n dr) and
    its J_r matches the FP32 form's closed forms to 1e-5 normwise; without it
    (the reference's arithmetic) J_r is larger by orders of magnitude."""
    from pdp3_amd import capi

    rng = np.random.default_rng(33)
    nr, nz, dr = 33, 129, 5e-4
    dt = 0.5 * dr / 3e8
    n = 512
    i = rng.integers(3, 29, n)
    k = rng.integers(3, 125, n)
    off = 0.005 if direction < 0 else 0.995
    r = (i + off) * dr
    z = (k + 0.5) * dr
    v = np.zeros((3, n))
    v[0] = direction * 0.01 * dr / dt
    w = np.full(n, 1e6)
    plain = capi.Simulation(nr, nz, 32 * dr, 128 * dr, dt, precision=capi.PREC_FP64)
    fixed = capi.Simulation(nr, nz, 32 * dr, 128 * dr, dt, precision=capi.PREC_FP64)
    fixed.set_strict_radial_fix(True)
    fp32 = capi.Simulation(nr, nz, 32 * dr, 128 * dr, dt, precision=capi.PREC_FP32)
    for s in (plain, fixed, fp32):
        s.add_plasma(-1, 1.0, r, z, v[0], v[1], v[2], w)
        s.step(1)
    jp, jf, j32 = (s.field("J_r") for s in (plain, fixed, fp32))
    e_fix = normwise(j32, jf)
    ratio = np.abs(jp).max() / np.abs(jf).max()
    print("direction", direction, "FP32 vs FP64 (fixed)", e_fix, "plain / fixed max", ratio)
    assert e_fix <= 1e-5, e_fix
    assert ratio >= 10, ratio
    for s in (plain, fixed, fp32):
        s.close()


@pytest.mark.parametrize("pusher", [0, 1])
def test_cfg1_100_steps_error(pusher, orc):
    from pdp3_amd import capi
    from pdp3_amd import workloads as wl

    w = wl.config("cfg1", pusher=pusher)
    g64 = wl.build_simulation(w, precision=capi.PREC_FP64)
    states = [g64.download(j) for j in range(len(w.plasma))]
    g64.close()
    ora = oracle_from_workload(orc, w, None, states)
    g32 = wl.build_simulation(w, precision=capi.PREC_FP32)
    ora.step(100)
    g32.step(100)
    errs = {name: rel_rms(g32.field(name), ora.field(name)) for name in ("E_r", "E_z", "H_phi", "J_z", "J_r")}
    print("relative RMS errors after 100 steps", errs)
    assert errs["E_z"] <= 1e-4, errs
    for name in ("E_r", "H_phi"):
        assert errs[name] <= 1e-3, (name, errs[name])
    for name in ("J_z", "J_r"):
        assert errs[name] <= 1e-2, (name, errs[name])


def test_tile_shapes_agree_and_autotune():
    """Every tile shape of the FP32 plasma kernel computes the same step (the
    per-particle FP32 arithmetic is identical; only the order of the FP64 grid
    sums differs); the autotuner returns one of them."""
    from pdp3_amd import capi
    from pdp3_amd import workloads as wl

    w = wl.config("cfg1", pml_cells=8)
    w.bunches = []
    shapes = [(16, 4), (16, 2), (16, 1), (8, 4), (8, 2), (4, 4)]
    ref = None
    for ppt, waves in shapes:
        print("tile", ppt, waves, flush=True)
        sim = wl.build_simulation(w, precision=capi.PREC_FP32)
        sim.set_tile(ppt, waves)
        assert sim.tile() == (ppt, waves)
        sim.step(10)
        f = {n: sim.field(n) for n in ("E_r", "E_z", "H_phi", "J_z")}
        st = sim.download(0)
        sim.close()
        if ref is None:
            ref = (f, st)
            continue
        for n in f:
            assert normwise(f[n], ref[0][n]) <= 1e-10, (ppt, waves, n, normwise(f[n], ref[0][n]))
        for k in ("r", "z", "vr", "vz"):
            assert normwise(st[k], ref[1][k]) <= 1e-10, (ppt, waves, k)
    sim = wl.build_simulation(w, precision=capi.PREC_FP32)
    best = sim.autotune(1)
    assert best in shapes
    assert sim.time > 0
    sim.close()
    with pytest.raises(capi.Pdp3Error):
        sim2 = wl.build_simulation(w, precision=capi.PREC_FP32)
        try:
            sim2.set_tile(3, 3)
        finally:
            sim2.close()


@pytest.mark.parametrize("cells_r,cells_z,ppc", [
    (21, 43, 3),      # 256-particle tiles, the last chunk mostly padding
    (9, 1000, 1),     # the same, tiles that overrun the field box
    (64, 256, 16),    # 256-particle tiles, whole chunks
    (128, 512, 15),   # 512-particle tiles
    (128, 1024, 13),  # one chunk per tile
    (256, 1024, 33),  # 2048-particle tiles, half the field box's width
    (512, 2048, 17),  # the same, its whole width
])
def test_tile_chosen_by_size(cells_r, cells_z, ppc):
    """Without a set or autotuned shape a species runs on the tile that suits
    its size; the step is that of the 16 x 4 shape up to the order of the FP64
    sums (per-particle arithmetic is identical: a deposit of n FP64 terms
    reordered moves by at most n ulps, far below 1e-11 of the maximum)."""
    from pdp3_amd import capi

    d = 5e-4
    out = []
    for shape in (None, (16, 4)):
        sim = capi.Simulation(cells_r + 1, cells_z + 1, cells_r * d, cells_z * d, 0.5 * d / 3e8,
                              precision=capi.PREC_FP32)
        sim.boundary_conditions()
        idx = sim.add_species(-1, 1.0, ppc * cells_r * cells_z)
        sim.init_uniform(idx, 11, ppc, 1e17, 0, 50.0)
        if shape:
            sim.set_tile(*shape)
        assert sim.tile() == (16, 4)
        sim.step(4)
        out.append({n: sim.field(n) for n in ("E_r", "E_phi", "E_z", "H_phi", "J_r", "J_phi", "J_z")})
        out[-1].update({k: v for k, v in sim.download(idx).items() if k in ("r", "z", "vr", "vphi", "vz")}
                       if cells_r < 200 else {})
        sim.close()
    for n in out[0]:
        assert normwise(out[0][n], out[1][n]) <= 1e-11, (n, normwise(out[0][n], out[1][n]))


@pytest.mark.parametrize("precision,cells_r,cells_z,n", [
    (1, 33, 131, 20000),    # 256-particle tiles, 4 per cell: the box's whole width
    (1, 16, 64, 30011),     # the same, half its width
    (1, 64, 256, 393216),   # 512-particle tiles
    (1, 200, 801, 400001),  # the same, the whole width
    (0, 33, 131, 20000),
    (0, 16, 64, 30011),
])
def test_small_tiles_of_particles_in_no_order(precision, cells_r, cells_z, n):
    """Tiles whose particles lie anywhere on the grid (most deposits miss the
    box), some of them dead: fields and states as with the particles in cell
    order, up to the order of the FP64 sums (see above; states are compared
    particle by particle after one step, whose inputs are the same)."""
    from pdp3_amd import capi

    d = 5e-4
    rng = np.random.default_rng(n)
    r, z = rng.uniform(d / 2, (cells_r - 0.5) * d, n), rng.uniform(d / 2, (cells_z - 0.5) * d, n)
    v = 1e7 * rng.standard_normal((3, n))
    w = rng.uniform(1, 2, n)
    alive = (rng.random(n) > 0.03).astype(np.uint8)
    out = []
    for order in (np.arange(n), np.lexsort((np.ceil(z / d), np.ceil(r / d)))):
        sim = capi.Simulation(cells_r + 1, cells_z + 1, cells_r * d, cells_z * d, 0.5 * d / 3e8, precision=precision)
        sim.boundary_conditions()
        for name in ("E_r", "E_phi", "E_z", "H_r", "H_phi", "H_z"):
            g = np.random.default_rng(len(name)).standard_normal((cells_r + 1, cells_z + 1))
            sim.set_field(name, (1e6 if name[0] == "E" else 2e3) * g)
        idx = sim.add_plasma(-1, 1.0, r[order], z[order], v[0][order], v[1][order], v[2][order], w[order], alive[order])
        sim.step(1)
        st = sim.download(idx)
        back = np.argsort(order)
        out.append({k: st[k][back] for k in ("r", "z", "vr", "vphi", "vz", "alive")})
        out[-1].update({k: sim.field(k) for k in ("J_r", "J_phi", "J_z", "E_z")})
        sim.close()
    for k in ("r", "z", "vr", "vphi", "vz", "alive"):
        assert np.array_equal(out[0][k], out[1][k]), k
    for k in ("J_r", "J_phi", "J_z", "E_z"):
        assert normwise(out[0][k], out[1][k]) <= 1e-11, (k, normwise(out[0][k], out[1][k]))


def test_tile_of_a_species_long_unsorted():
    """After 500 steps without a sort a species of any size runs on the small
    tiles.  The plasma is thin enough for its fields not to feed back: J is that
    of the 16 x 4 shape up to the order of the FP64 sums."""
    from pdp3_amd import capi

    d, cells_r, cells_z, ppc = 5e-4, 128, 1024, 13
    out = []
    for shape in (None, (16, 4)):
        sim = capi.Simulation(cells_r + 1, cells_z + 1, cells_r * d, cells_z * d, 0.5 * d / 3e8,
                              precision=capi.PREC_FP32)
        sim.boundary_conditions()
        idx = sim.add_species(-1, 1.0, ppc * cells_r * cells_z)
        sim.init_uniform(idx, 11, ppc, 1e2, 0, 1.0)
        if shape:
            sim.set_tile(*shape)
        for steps in (499, 3):
            sim.step(steps)
            out.append({n: sim.field(n) for n in ("J_r", "J_phi", "J_z")})
        sim.close()
    for a, b in ((out[0], out[2]), (out[1], out[3])):
        for n in a:
            assert normwise(a[n], b[n]) <= 1e-11, (n, normwise(a[n], b[n]))


def test_autotune_keeps_the_automatic_choice():
    """Where the automatic choice is the fastest candidate (1.6e5 particles take
    11 us on one particle per lane, 23 us on the fastest shape that can be set)
    the autotuner keeps it; it advances the simulation by six times the steps,
    whatever it chooses, and returns a shape that can be set."""
    from pdp3_amd import capi

    d = 5e-4
    sim = capi.Simulation(65, 257, 64 * d, 256 * d, 0.5 * d / 3e8, precision=capi.PREC_FP32)
    sim.boundary_conditions()
    idx = sim.add_species(-1, 1.0, 10 * 64 * 256)
    sim.init_uniform(idx, 11, 10, 1e17, 0, 1.0)
    assert sim.species_tile(idx) == (1, 4)
    best = sim.autotune(8)
    assert abs(sim.time - 48 * sim.dt) <= 1e-6 * sim.dt
    assert best in [(16, 4), (16, 1), (8, 4), (8, 2), (4, 4)] and sim.tile() == best
    assert sim.species_tile(idx) == (1, 4)
    sim.set_tile(8, 4)
    assert sim.tile() == (8, 4) and sim.species_tile(idx) == (8, 4)
    with pytest.raises(capi.Pdp3Error):
        sim.species_tile(1)
    sim.close()


def test_autotune_failure_leaves_the_shape():
    """Steps that fail (a particle past the outer wall, reported by the gather's
    bounds check) leave the shape as it was."""
    from pdp3_amd import capi

    d = 5e-4
    for shape in (None, (8, 2)):
        sim = capi.Simulation(9, 33, 8 * d, 32 * d, 0.5 * d / 3e8, precision=capi.PREC_FP32)
        n = 2000
        r = np.full(n, 3.3 * d)
        r[7] = 8.3 * d
        sim.add_plasma(-1, 1.0, r, np.full(n, 7.3 * d), np.zeros(n), np.zeros(n), np.zeros(n), np.ones(n))
        if shape:
            sim.set_tile(*shape)
        before = sim.tile(), sim.species_tile(0)
        with pytest.raises(capi.Pdp3Error):
            sim.autotune(1)
        assert (sim.tile(), sim.species_tile(0)) == before
        sim.close()
