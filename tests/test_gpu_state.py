"""States set from fields, planes and noise on the device have the bits of the
host expressions (the reference forms them on the host in FP32, one rounding
per product and sum, lattice_grid_3d.cpp:95-131), and read-back returns them
whole: reads that fit one pinned chunk, ragged ones, and ones that several
workers share."""
import numpy as np
import pytest

import oracle_bind as ob

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def wa():
    import wake_amd

    if wake_amd._lib.lib().wake_hip_device_count() <= 0:
        pytest.fail("no GPU visible to the HIP runtime")
    return wake_amd


def _grid(wa, lattice, shape, storage):
    nx, ny, nz = shape
    if lattice == 9:
        return wa.LatticeGrid2D(nx, ny, 0.7, storage=storage)
    return wa.LatticeGrid3D(nx, ny, nz, 0.7, lattice=lattice, storage=storage)


def _fields(shape, lattice):
    n = int(np.prod(shape))
    r = np.random.default_rng(n)
    f = [r.uniform(0.9, 1.1, n)] + [r.uniform(-0.1, 0.1, n) for _ in range(2 if lattice == 9 else 3)]
    return [v.astype(np.float32) for v in f]


def _splitmix(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _stored(f, w, storage):
    """FP32 planes after the round trip through the population storage."""
    if storage == 0:
        return f
    d = f - w[:, None]
    if storage == 1:
        return (w[:, None] + d.astype(np.float16).astype(np.float32)).astype(np.float32)
    b = d.view(np.uint32)
    b = (b + np.uint32(0x7FFF) + ((b >> np.uint32(16)) & np.uint32(1))) & np.uint32(0xFFFF0000)
    return (w[:, None] + b.view(np.float32)).astype(np.float32)


CASES = [(9, (53, 37, 1)), (19, (31, 17, 9)), (27, (16, 8, 5)), (19, (160, 96, 80))]


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("lattice,shape", CASES)
def test_state_from_fields_and_noise_bits(wa, lattice, shape, storage):
    g = _grid(wa, lattice, shape, storage)
    F = _fields(shape, lattice)
    g.initialize_fields(*F)
    o = ob.OracleGrid(2 if lattice == 9 else 3, *shape, tau=0.7, lattice=lattice)
    o.initialize_fields(*F)
    f0 = np.array(o.f_src(), np.float32).reshape(lattice, -1)
    one = _grid(wa, lattice, (8, 4, 2), 0)
    one.initialize(1.0)
    w = one.f_src_data()[:, 0].copy()  # feq at rest: the weights
    assert np.array_equal(g.f_src_data(), _stored(f0, w, storage))
    # the fields read back are the ones given, before and after the populations were read
    reads = [g.rho_data(), g.ux_data(), g.uy_data()] + ([] if lattice == 9 else [g.uz_data()])
    for a, b in zip(reads, F):
        assert np.array_equal(a, b)
    assert np.array_equal(g.f_dst_data() if lattice == 9 else g.f_src_data(), _stored(f0, w, storage))
    s0 = g.f_src_data().copy()
    g.add_noise(1e-3, 42)
    n = s0.shape[1]
    ctr = np.arange(n, dtype=np.uint64)[None, :] * np.uint64(lattice) + np.arange(lattice, dtype=np.uint64)[:, None]
    u = (_splitmix(np.uint64(42) ^ ctr) >> np.uint64(40)).astype(np.float64) / 16777216.0
    f1 = s0 + np.float32(1e-3) * (2.0 * u - 1.0).astype(np.float32)
    assert np.array_equal(g.f_src_data(), _stored(f1, w, storage))
    # planes set and read back
    g.set_populations(f0)
    assert np.array_equal(g.f_src_data(), _stored(f0, w, storage))


def test_convective_store_from_fields(wa):
    """The outlet store starts from the state set: a run from fields given
    before and after the outlet was switched on is the same."""
    out = []
    for first in (True, False):
        g = wa.LatticeGrid3D(24, 12, 10, 0.6)
        g.set_periodic_axes(True, True)
        F = _fields((24, 12, 10), 19)
        if first:
            g.initialize_fields(*F)
        g.set_inflow_west(0.05, 0.0)
        g.set_convective_outflow_east(0.05)
        if not first:
            g.initialize_fields(*F)
        g.run(7, "MRT")
        out.append(g.f_src_data().copy())
    assert np.array_equal(*out)


def test_diagnostics_and_analytics_without_host_fields(wa):
    g = _grid(wa, 19, (61, 33, 20), 0)
    g.initialize_fields(*_fields((61, 33, 20), 19))
    g.run(3, "BGK")
    mass, energy, speed = g.compute_total_mass(), g.compute_total_kinetic_energy(), g.compute_max_speed()
    w = [v.copy() for v in g.vorticity_q_data()]
    rho, u = g.rho_data(), [g.ux_data(), g.uy_data(), g.uz_data()]
    sp = g.speed_data()
    assert mass == pytest.approx(rho.astype(np.float64).sum(), rel=1e-12)
    assert energy == pytest.approx((np.float32(0.5) * rho * sp * sp).astype(np.float64).sum(), rel=1e-12)
    assert speed == sp.max()
    oz, oy = np.zeros_like(rho), np.zeros_like(rho)
    ox, qc = np.zeros_like(rho), np.zeros_like(rho)
    wa.kernels.kernel("compute_vorticity_and_q_criterion_3d", *u, ox, oy, oz, qc, 61, 33, 20)
    for a, b in zip(w, (ox, oy, oz, qc)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("steps", [0, 1, 2, 3, 8, 9, 16, 21])
@pytest.mark.parametrize("op", ["populations", "noise", "fields", "uniform"])
def test_temperature_goes_on_from_a_new_flow_state(wa, op, steps, storage):
    """Setting the flow leaves the temperature where it is, whichever buffer
    the steps before ended in, one launch per step or several."""
    ends = []
    nx, ny = 40, 27
    for multi in (True, False):
        g = wa.LatticeGrid2D(nx, ny, 0.6, storage=storage)
        g.initialize(1.0)
        g.set_solid_box(0, 0, nx - 1, 0)
        g.set_solid_box(0, ny - 1, nx - 1, ny - 1)
        g.enable_thermal(0.62, 1e-3, 0.5, 0.5)
        g.set_temperature_field(np.random.default_rng(2).uniform(0, 1, nx * ny).astype(np.float32))
        g.set_wall_temperature(0, 0, nx - 1, 0, 0.87)
        g.set_multistep(multi)
        g.run(steps, "MRT")
        t0 = g.temperature_data().copy()
        if op == "populations":
            g.set_populations(g.f_src_data().copy())
        elif op == "noise":
            g.add_noise(1e-4, 5)
        elif op == "fields":
            g.initialize_fields(*_fields((nx, ny, 1), 9))
        else:
            g.initialize(1.0, 0.01, 0.0)
        g.update_macroscopic()
        assert np.array_equal(g.temperature_data(), t0)
        g.run(3, "MRT")
        ends.append([g.temperature_data().copy(), g.f_src_data().copy()])
    for a, b in zip(*ends):
        assert np.array_equal(a, b)


def _vorticity(wa, g, shape):
    nx, ny, nz = shape
    if nz == 1:
        w = np.zeros(nx * ny, np.float32)
        wa.kernels.kernel("compute_vorticity_2d", g.ux_data(), g.uy_data(), w, nx, ny)
        return [w]
    out = [np.zeros(nx * ny * nz, np.float32) for _ in range(4)]
    wa.kernels.kernel("compute_vorticity_and_q_criterion_3d", g.ux_data(), g.uy_data(), g.uz_data(), *out, nx, ny, nz)
    return out


@pytest.mark.parametrize("lattice,shape", [(9, (53, 37, 1)), (19, (21, 17, 9))])
def test_analytics_follow_a_new_state(wa, lattice, shape):
    """Vorticity and Q read before a state was set are not given for it."""
    g = _grid(wa, lattice, shape, 0)
    read = (lambda: [g.vorticity_data()]) if lattice == 9 else g.vorticity_q_data
    F = _fields(shape, lattice)

    def check():
        for a, b in zip(read(), _vorticity(wa, g, shape)):
            assert np.array_equal(a, b)

    def with_temperature():
        g.enable_thermal(0.62, 1e-2, 0.5, 0.5)
        g.run(2, "BGK", gx=1e-4, gy=2e-4)
        read()
        g.set_temperature_field(np.random.default_rng(4).uniform(0, 1, g.total_nodes()).astype(np.float32))

    ops = [lambda: g.initialize_fields(*F), lambda: g.initialize(1.0, 0.02, 0.0),
           lambda: g.initialize_fields(*[F[0]] + [np.float32(0.5) * u for u in F[1:]]),
           lambda: g.run(3, "BGK", gx=1e-4, gy=2e-4), g.update_macroscopic, lambda: g.set_populations(g.f_src_data()),
           lambda: g.add_noise(1e-3, 1)] + ([with_temperature] if lattice == 9 else [])
    check()
    for op in ops:
        op()
        check()


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("lattice,shape", [(9, (53, 37, 1)), (19, (21, 17, 9))])
def test_fields_after_noise(wa, lattice, shape, storage):
    """They are those of the state without the noise until the next step,
    whether or not a field was read before; FP32 planes just set have none."""
    read = lambda g: [v.copy() for v in (g.rho_data(), g.ux_data(), g.uy_data(), g.speed_data())]

    def stepped():
        g = _grid(wa, lattice, shape, storage)
        g.initialize_fields(*_fields(shape, lattice))
        g.run(3, "BGK", gx=1e-4, gy=2e-4)
        return g

    clean = read(stepped())
    for before in (lambda g: None, lambda g: g.rho_data(), lambda g: g.f_src_data(), lambda g: g.compute_max_speed()):
        g = stepped()
        before(g)
        g.add_noise(1e-3, 8)
        assert all(np.array_equal(a, b) for a, b in zip(read(g), clean))
        g.add_noise(1e-3, 9)
        assert all(np.array_equal(a, b) for a, b in zip(read(g), clean))
        g.update_macroscopic()
        assert not np.array_equal(g.rho_data(), clean[0])
    g, h = stepped(), stepped()
    f = g.f_src_data().copy()
    for d in (g, h):
        d.set_populations(f)
    g.add_noise(1e-3, 8)
    if storage:
        want = read(h)
    else:
        h.set_populations(g.f_src_data().copy())
        want = read(h)
    assert all(np.array_equal(a, b) for a, b in zip(read(g), want))


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("lattice,shape", CASES)
def test_setting_populations_takes_no_device_memory(wa, lattice, shape, storage):
    """A domain admitted by its size can take its state: no scratch is kept."""
    g = _grid(wa, lattice, shape, storage)
    before = g.device_bytes()
    f = np.random.default_rng(1).uniform(0.01, 0.4, (lattice, g.total_nodes())).astype(np.float32)
    g.run(2, "BGK")
    g.set_populations(f)
    assert g.device_bytes() == before
    one = _grid(wa, lattice, (8, 4, 2), 0)
    one.initialize(1.0)
    assert np.array_equal(g.f_src_data(), _stored(f, one.f_src_data()[:, 0].copy(), storage))


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("lattice,shape", [(9, (53, 37, 1)), (19, (21, 17, 9)), (27, (16, 8, 5))])
def test_fields_go_with_the_populations_read(wa, lattice, shape, storage):
    """The fields read after the populations are theirs, also when a change of
    the geometry has rounded the state to its storage in between."""
    ends = []
    for read in (lambda g: g.rho_data(), lambda g: g.f_src_data()):
        g = _grid(wa, lattice, shape, storage)
        g.initialize_fields(*_fields(shape, lattice))
        g.set_inflow_west(0.04, 0.0)  # its nodes form values the storage does not hold
        g.run(3, "BGK", gx=1e-4, gy=2e-4)
        read(g)
        f = g.f_src_data().copy()
        g.set_cell_type(*(3, 3, 3)[:2 if lattice == 9 else 3], 1)
        assert np.array_equal(g.f_src_data(), f)  # as read before
        ends.append([g.rho_data(), g.ux_data(), g.uy_data(), g.speed_data()])
    for a, b in zip(*ends):
        assert np.array_equal(a, b)
