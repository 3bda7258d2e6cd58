"""Kernel variants at the sizes where they can go wrong, against the CPU oracle:
row and wavefront edges of the geometry EHSS kernel, and the field-array
kernels' kept cell under ions that change cells in nearly every stage.

FP64 runs draw the same random numbers on both sides and differ by rounding
only: 1e-9 relative, as the parity tests; a contact or collision decided within
rounding of its threshold (some 1e-15 of the tests) does not occur at these
sizes, so every ion has to match.
"""
import os

import numpy as np
import pytest

from icarion_amd import _abi
from icarion_amd import workloads as W
from test_gpu_parity import compare_ions, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


def cluster_table(counts, spread, seed):
    """Species of counts[s] atoms (1.7 A) spread over a cube of half edge spread[s]."""
    rng = np.random.default_rng(seed)
    atoms, species, off = [], [], 0
    for c, h in zip(counts, spread):
        a = np.zeros((c, 4), np.float32)
        a[:, :3] = rng.uniform(-h, h, (c, 3))
        a[:, 3] = 1.7e-10
        atoms.append(a)
        species.append(W.species(sigma_ehss=3e-18, atom_offset=off, atom_count=c))
        off += c
    return np.concatenate(atoms), species


# atoms per cluster about the 64-atom rows and the 512 staged ones; the sparse
# pair (atoms several nm apart) is missed by most impact parameters, so that the
# draws go past the ones made ahead, past the expansion and past the last attempt
COUNTS = (1, 2, 63, 64, 65, 128, 449, 511, 512, 513, 700)
SPREAD = (0.0, 4e-9, 8e-10, 8e-10, 8e-10, 8e-10, 1.2e-9, 1.2e-9, 1.2e-9, 1.2e-9, 1.2e-9)


@pytest.mark.parametrize("n,steps", [(1, 25), (63, 25), (2047, 25), (2049, 25), (5000, 25),
                                     # two and three passes of draws ahead (22 and 35 ions per
                                     # wavefront), and a second round of wavefronts
                                     (45001, 5), (70001, 4), (131073, 3)])
def test_geometry_ehss_rows_and_wavefronts(oracle, n, steps):
    atoms, species = cluster_table(COUNTS, SPREAD, seed=5)
    w = W.ehss_surrogate_workload(n=1, seed=17, precision=_abi.PRECISION_FP64, ehss_mode=_abi.EHSS_GEOMETRY)
    rng = np.random.default_rng(n)
    which = rng.integers(0, len(species), n).astype(np.uint32)
    which[:min(n, len(species))] = np.arange(min(n, len(species)))
    ens = W.gaussian_cloud(n, 1200.0, 0.5e-3, seed=n)
    ens.species[:] = which
    w.update(species=species, atoms=atoms, ensemble=ens)
    g, o = ens.copy(), ens.copy()
    sg = gpu_run(w, g, steps)
    so = oracle_run(oracle, w, o, steps)
    assert so.collisions > 0 or n < 63
    assert sg.collisions == so.collisions
    assert compare_ions(g, o, rtol=1e-9).all()


@pytest.mark.parametrize("integrator", [_abi.INTEGRATOR_RK4, _abi.INTEGRATOR_BORIS])
@pytest.mark.parametrize("precision", [_abi.PRECISION_FP64, _abi.PRECISION_FP32_KAHAN])
@pytest.mark.parametrize("n,grid", [(1, (2, 2, 2)), (257, (2, 3, 65)), (3001, (64, 63, 2)), (70001, (40, 41, 200))])
def test_field_array_cell_changes(oracle, n, grid, precision, integrator):
    """Ions at 10 km/s with steps of a good part of a cell: most stages find the
    ion in another cell than the last one.  FP32 against the FP64 oracle: cell
    coordinates of up to 200 in FP32 place an ion to 200 * 2^-24 of a cell, and
    the field is continuous across cells, so 2e-5 as for the other collisionless
    FP32 runs.  Potentials of a few volts: the field gradient of 5 V / mm^2 then
    multiplies a deviation by less than exp(omega t) = 5 over the run (omega^2 =
    q E' / m = 1.6e12 s^-2, t = 1.2 us); kilovolts would multiply it by exp(48)."""
    E, origin, spacing = W.gaussian_potential_field(grid, n_gauss=4, seed=2)
    E *= np.float32(1e-3)
    w = W.field_array_workload(n=1, grid=(2, 2, 2), seed=2, precision=precision)
    w["physics"] = W.physics(integrator, _abi.COLLISION_NONE, precision=precision, seed=2)
    ens = W.gaussian_cloud(n, 300.0, (1e-3, 1e-3, 4e-3), center=(0.0, 0.0, 20e-3), seed=n)
    ens.vx += 2e3
    ens.vz += 1e4
    w.update(ensemble=ens, field=(E, origin, spacing), dt=2e-8)
    g, o = ens.copy(), ens.copy()
    gpu_run(w, g, 60)
    oracle_run(oracle, w, o, 60)
    assert (g.active == o.active).mean() >= 0.999
    both = (g.active != 0) & (o.active != 0)
    tol = 1e-9 if precision == _abi.PRECISION_FP64 else 2e-5
    for f, scale in (("x", 1e-3), ("y", 1e-3), ("z", 1e-2), ("vx", 1e3), ("vy", 1e3), ("vz", 1e4)):
        d = np.abs(getattr(g, f) - getattr(o, f))[both]
        assert d.size == 0 or d.max() <= tol * np.maximum(scale, np.abs(getattr(o, f))[both].max()), f


@pytest.mark.parametrize("kind", ["drift", "trap_ou", "trap_quiet", "none", "friction"])
@pytest.mark.parametrize("integrator", [_abi.INTEGRATOR_RK4, _abi.INTEGRATOR_BORIS])
@pytest.mark.parametrize("n", [1, 15, 1025, 49152, 49153])
def test_fp64_lanes_per_ion(oracle, n, integrator, kind):
    """Both sides of the four-lanes-per-ion bound, partial quads and wavefronts,
    births during the run, arrivals and losses, a rotated domain."""
    if kind == "drift":
        w = W.ims_hss_workload(n=n, seed=n)
        w["domain"].detector_z_m = 2e-4
        c, s = np.cos(0.3), np.sin(0.3)
        w["domain"].rot_g2l = (1.0, 0.0, 0.0, 0.0, c, s, 0.0, -s, c)
        w["domain"].rot_l2g = (1.0, 0.0, 0.0, 0.0, c, -s, 0.0, s, c)
        w["domain"].radius_m = 2.5e-3
        coll, ou, steps = _abi.COLLISION_HSS, 0, 40
    else:
        w = W.quadrupole_workload(n=n, seed=n, U=20.0)
        coll = {"none": _abi.COLLISION_NONE, "friction": _abi.COLLISION_FRICTION}.get(kind, _abi.COLLISION_LANGEVIN)
        ou, steps = int(kind == "trap_ou"), 40
        w["domain"].radius_m = 0.5e-3   # ions lost during the run
        w["species"] = [W.species(K0=2.1, ccs=100e-20)]
    w["physics"] = W.physics(integrator, coll, ou=ou, seed=n)
    ens = w["ensemble"]
    rng = np.random.default_rng(n)
    ens.birth_time_s = np.where(rng.random(n) < 0.3, rng.uniform(0.0, 50.0, n) * w["dt"], 0.0)
    ens.born[:] = ens.birth_time_s == 0.0
    ens.active[:] = ens.born
    g, o = ens.copy(), ens.copy()
    sg = gpu_run(w, g, steps)
    so = oracle_run(oracle, w, o, steps)
    assert (sg.ion_steps, sg.collisions, sg.alive, sg.arrived) == (so.ion_steps, so.collisions, so.alive, so.arrived)
    assert compare_ions(g, o, rtol=1e-9).all()
    assert np.array_equal(g.born, o.born) and np.array_equal(g.n_collisions, o.n_collisions)
    np.testing.assert_allclose(g.death_time_s, o.death_time_s, rtol=1e-12)
    np.testing.assert_allclose(g.arrival_time_s, o.arrival_time_s, rtol=1e-9)


@pytest.mark.parametrize("integrator", [_abi.INTEGRATOR_RK4, _abi.INTEGRATOR_BORIS])
@pytest.mark.parametrize("n", [1, 5, 4097, 65536, 65537, 131072, 131073])
def test_surrogate_launch_shapes(n, integrator):
    """An ion's run depends on its index and the seed alone: the first ions of a
    cloud, stepped in clouds of other sizes (other ions per wavefront, the other
    instantiation), take the same course bit for bit."""
    from icarion_amd import gpu
    import icarion_amd
    m = min(n, 1000)
    w = W.ehss_surrogate_workload(n=1, seed=3)
    w["physics"].integrator = integrator
    w["domain"].detector_z_m = 1e-5
    params = np.load(icarion_amd.__path__[0] + "/data/surrogate_he_20td_clusters.npy")
    counts = W.ehss_cluster_counts(40, 3)
    rng = np.random.default_rng(9)
    full = W.gaussian_cloud(131073, 1500.0, 0.5e-3, seed=3)
    full.species[:] = rng.integers(0, 40, full.n)
    full.birth_time_s = np.where(rng.random(full.n) < 0.3, rng.uniform(0.0, 60.0, full.n) * w["dt"], 0.0)
    full.born[:] = full.active[:] = full.birth_time_s == 0.0
    out = []
    for size in (n, 2001):
        e = full.subset(np.arange(size))
        with gpu.Handle(device=0) as h:
            h.set_domain(w["domain"], w["physics"])
            h.synth_clusters(counts, seed=3)
            h.surrogate_set_params(params)
            h.upload_state(e)
            st = h.step(0.0, w["dt"], 50)
            h.download_state(e)
        born = e.born != 0
        assert st.ion_steps == np.where(e.birth_time_s == 0.0, 50, 50 - np.ceil(e.birth_time_s / w["dt"]))[born].sum()
        assert st.collisions == e.n_collisions.sum()
        out.append(e.subset(np.arange(m)))
    a, b = out
    for f in ("x", "y", "z", "vx", "vy", "vz", "death_time_s", "arrival_time_s", "active", "born", "n_collisions"):
        np.testing.assert_array_equal(getattr(a, f), getattr(b, f), err_msg=f)


@pytest.mark.parametrize("precision", [_abi.PRECISION_FP64, _abi.PRECISION_FP32_KAHAN])
def test_lost_ions_leave_the_launches(precision):
    """A large trap that loses ions in every launch, among them all but a few at
    last: the ions run alone after the first launches are the same, bit for bit,
    as with one launch for the whole run, where no lane is dropped."""
    w = W.quadrupole_workload(n=262144 + 77, seed=8, precision=precision)
    w["domain"].radius_m = 0.6e-3
    a, b = w["ensemble"].copy(), w["ensemble"].copy()
    for e in (a, b):
        e.active[::1001] = 0     # dead on arrival
    sa = gpu_run(w, a, 3000, steps_per_launch=150)
    sb = gpu_run(w, b, 3000, steps_per_launch=3000)
    assert 0 < sa.alive < 0.7 * a.n
    assert (sa.ion_steps, sa.collisions, sa.alive) == (sb.ion_steps, sb.collisions, sb.alive)
    for f in ("x", "y", "z", "vx", "vy", "vz", "death_time_s", "active", "born"):
        assert np.array_equal(getattr(a, f), getattr(b, f)), f


@pytest.mark.parametrize("kind", ["hss", "mixture", "snapshots"])
@pytest.mark.parametrize("precision", [_abi.PRECISION_FP64, _abi.PRECISION_FP32_KAHAN])
def test_dropped_lanes_leave_no_trace(precision, kind):
    """Half of the ions are outside the domain at the start, so that the first
    count drops their lanes, and others arrive and leave later.  The same ions in
    a cloud of one less than the rule's size run with every lane in place, in the
    same launches: bit for bit the same, the snapshots during the run too."""
    from icarion_amd import gpu
    n = 262144
    if kind == "mixture":
        w = W.ims_mixture_workload(n=n, seed=12, precision=precision)
    else:
        w = W.ims_hss_workload(n=n, seed=12, precision=precision)
    ens = w["ensemble"]
    r = np.hypot(ens.x, ens.y)
    w["domain"].radius_m = float(np.median(r))
    w["domain"].detector_z_m = float(np.quantile(ens.z, 0.5)) + 1e-9    # crossed by some hundred ions
    out = []
    for size in (n, n - 1):
        e = ens.subset(np.arange(size))
        with gpu.Handle(steps_per_launch=40) as h:
            h.set_domain(w["domain"], w["physics"])
            h.set_species(w["species"])
            if kind == "mixture":
                h.set_gas_mixture(*w["mixture"])
            h.upload_state(e)
            if kind == "snapshots":
                snaps, _, st = h.step_snapshots(0.0, w["dt"], 400, 70 * w["dt"])
                assert len(snaps) >= 5
            else:
                snaps, st = [], h.step(0.0, w["dt"], 400)
            h.download_state(e)
        m = n - 1
        assert st.alive == (e.active != 0).sum() < 0.55 * size and st.collisions == e.n_collisions.sum()
        out.append((e.subset(np.arange(m)), [(x["step"], x["positions"][:m], x["velocities"][:m], x["flags"][:m])
                                              for x in snaps]))
    (a, sa), (b, sb) = out
    assert np.isfinite(a.arrival_time_s).sum() > 100 and a.n_collisions.max() > 0
    for f in ("x", "y", "z", "vx", "vy", "vz", "death_time_s", "arrival_time_s", "active", "born", "n_collisions"):
        np.testing.assert_array_equal(getattr(a, f), getattr(b, f), err_msg=f)
    assert len(sa) == len(sb)
    for x, y in zip(sa, sb):
        assert x[0] == y[0] and all(np.array_equal(p, q) for p, q in zip(x[1:], y[1:]))


def test_all_ions_lost(precision=_abi.PRECISION_FP32_KAHAN):
    """Launches after the last ion is gone have nothing to run."""
    w = W.quadrupole_workload(n=262144, seed=8, precision=precision)
    w["domain"].length_m = 1e-9
    g = w["ensemble"].copy()
    st = gpu_run(w, g, 400, steps_per_launch=100)
    assert st.alive == 0 and not g.active.any()


@pytest.mark.parametrize("integrator", [_abi.INTEGRATOR_RK4, _abi.INTEGRATOR_BORIS])
@pytest.mark.parametrize("n", [1, 1023])
def test_fp32_push_rounds_alike_in_every_kernel(n, integrator):
    """A rising axial field, with and without an RF term of zero, and an RF field,
    each with and without the HSS stage for ions of no cross section, over one and
    several domains; free flight with a damping force without mobility and in a
    field array of zeros: the forces are the same, so that the same products and
    sums have to give the same bits, whatever else the kernel around them holds."""
    from icarion_amd import gpu
    masses = np.random.default_rng(n).uniform(100.0, 900.0, n)
    ens = W.gaussian_cloud(n, masses, 1e-3, center=(0.0, 0.0, 25e-3), seed=n)
    zero = _abi.waveform(_abi.WAVEFORM_LINEAR, (0.0, 0.0, 0.0, 1e-3))

    def run(collision, kind, axial_V, rf_V):
        ph = W.physics(integrator, collision, precision=_abi.PRECISION_FP32_KAHAN, seed=1)
        d = W.ims_domain(origin_z=0.0, length=50e-3, radius=5e-3, axial_V=axial_V, pressure_Pa=300.0)
        d.rf_voltage_V, d.rf_frequency_Hz = rf_V, 3e6
        d.use_field_array = int(kind == "array")
        e = ens.copy()
        with gpu.Handle() as h:
            if kind == "domains":
                far = W.ims_domain(origin_z=50e-3, length=5e-3, radius=5e-3, axial_V=0.0, pressure_Pa=300.0)
                h.set_domains([d, far], ph, [0.0, 0.0])
            else:
                h.set_domain(d, ph)
            h.set_species([W.species()])
            if kind == "array":
                h.upload_field_array(np.zeros((9, 5, 5, 3), np.float32), (-5e-3, -5e-3, 0.0), (2.5e-3, 2.5e-3, 6.25e-3))
            if axial_V:   # rising by half during the run
                slots = {_abi.SLOT_DC_AXIAL: _abi.waveform(_abi.WAVEFORM_LINEAR, (axial_V, 1.5 * axial_V, 0.0, 5e-7))}
                if kind == "rf":
                    slots[_abi.SLOT_RF_VOLTAGE] = zero
                if kind == "domains":
                    h.set_domain_waveforms(0, slots)
                else:
                    h.set_waveforms(slots)
            h.upload_state(e)
            h.step(0.0, 1e-9, 500)
            h.download_state(e)
        assert e.active.all()
        return e

    none, hss, friction = _abi.COLLISION_NONE, _abi.COLLISION_HSS, _abi.COLLISION_FRICTION
    for fields, others in (
            ((20.0, 0.0), [(none, "rf"), (hss, "uniform"), (hss, "rf"), (none, "domains"), (hss, "domains")]),
            ((20.0, 300.0), [(hss, "uniform"), (none, "domains"), (hss, "domains")]),
            ((0.0, 0.0), [(friction, "uniform"), (none, "array"), (hss, "array"), (friction, "array")])):
        a = run(none, "uniform", *fields)
        assert not np.array_equal(a.x, ens.x)
        for collision, kind in others:
            b = run(collision, kind, *fields)
            for f in ("x", "y", "z", "vx", "vy", "vz"):
                assert np.array_equal(getattr(a, f), getattr(b, f)), (fields, collision, kind, f)


def pinned_runs(kind):
    """Short FP32 runs with collisions, by name: the final states of 64 ions."""
    from icarion_amd import gpu
    import icarion_amd
    out = {}
    for name, integrator in (("rk4", _abi.INTEGRATOR_RK4), ("boris", _abi.INTEGRATOR_BORIS)):
        if kind == "surrogate":
            w = W.ehss_surrogate_workload(n=64, seed=3)
            w["physics"].integrator = integrator
            e = w["ensemble"].copy()
            with gpu.Handle(device=0) as h:
                h.set_domain(w["domain"], w["physics"])
                h.synth_clusters(w["counts"], seed=3)
                h.surrogate_set_params(np.load(icarion_amd.__path__[0] + "/data/surrogate_he_20td_clusters.npy"))
                h.upload_state(e)
                h.step(0.0, w["dt"], 2000)
                h.download_state(e)
        else:
            w = W.field_array_workload(n=64, grid=(24, 20, 40), seed=2, precision=_abi.PRECISION_FP32_KAHAN)
            w["physics"] = W.physics(integrator, _abi.COLLISION_HSS, precision=_abi.PRECISION_FP32_KAHAN, seed=5)
            e = w["ensemble"].copy()
            gpu_run(w, e, 4000)
        assert e.n_collisions.min() > 0
        out[name] = np.stack([e.x, e.y, e.z, e.vx, e.vy, e.vz])
    return out


@pytest.mark.parametrize("kind", ["surrogate", "field_array"])
def test_fp32_results_stay_the_same(kind):
    """The rounding of these kernels is written out, so that a change around it
    leaves the results as they were, bit for bit (tests/golden, made on an MI355X;
    an ulp would flip a collision test in some 1e7)."""
    with np.load(os.path.join(os.path.dirname(__file__), "golden", f"fp32_{kind}.npz"), allow_pickle=False) as want:
        for name, got in pinned_runs(kind).items():
            np.testing.assert_array_equal(got, want[name], err_msg=name)


def test_field_array_cell_follows_from_the_position():
    """Positions within rounding below a cell's face, whose cell coordinate as a
    rounded product lies on the face: the next cell's, whether an ion is there
    from the start or comes there from the cell before, which it has kept.  The
    field is zero on the kept cell's nodes and 1 MV/m on the next one along x, so
    that an ion with the wrong cell feels no force at all.  Boris in powers of two:
    the second step begins exactly at the position."""
    nx, spacing, first = 96, 1e-2 / 95, -5e-3
    f32 = np.float32
    x0, inv = f32(first), f32(1.0 / spacing)
    p2 = []
    for i in range(2, nx - 2, 3):   # faces between a zero cell and one that ends at a charged node
        p = f32(first + i * spacing)
        for _ in range(8):
            p = np.nextafter(p, f32(-1.0))
        for _ in range(16):
            p = np.nextafter(p, f32(1.0))
            d = f32(p - x0)
            if f32(d * inv) >= i and float(d) * float(inv) < i and float(p) - 2.0**-14 == f32(p - f32(2.0**-14)):
                p2.append(p)
    assert len(p2) >= 8
    E = np.zeros((5, 5, nx, 3), np.float32)
    E[:, :, 3::3, 0] = 1e6
    n = len(p2)
    w = W.field_array_workload(n=1, grid=(2, 2, 2), seed=2)
    w["physics"] = W.physics(_abi.INTEGRATOR_BORIS, _abi.COLLISION_NONE, precision=_abi.PRECISION_FP32_KAHAN, seed=2)
    ens = W.gaussian_cloud(2 * n, 100.0, 1e-6, center=(0.0, 0.0, 20e-3), seed=6)
    ens.vx[:] = ens.vy[:] = ens.vz[:] = 0.0
    ens.x[:n] = ens.x[n:] = np.array(p2, np.float64)
    ens.x[n:] -= 2.0**-14
    ens.vx[n:] = 2.0**16
    w.update(ensemble=ens, field=(E, (first, -5e-3, 0.0), (spacing, 2.5e-3, 1.25e-2)), dt=2.0**-30)
    gpu_run(w, ens, 2)
    there, coming = ens.vx[:n] / 2.0, ens.vx[n:] - 2.0**16   # two steps at the position, and one
    assert (np.abs(there) > 1e-5).all()
    np.testing.assert_allclose(coming, there, rtol=1e-4)
