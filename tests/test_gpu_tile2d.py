"""Bounded 2D domains run up to 8 steps per launch from LDS tiles
(tile2d.hpp).  Every node update is the single-step kernel's, so a run must
give the same bits as the same number of single steps: walls, obstacles, a
moving wall, parabolic and noisy inlets, the pressure outlet, solid nodes in
periodic streaming, the temperature coupling and the force history, at sizes
around the tiles' own extent and their halo, and when runs of every length
alternate with single steps, force reads and geometry changes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(240, 80), (64, 33), (33, 17), (16, 16), (17, 48), (9, 5), (131, 8)]


@pytest.fixture(scope="module")
def wa():
    import wake_amd

    if wake_amd._lib.lib().wake_hip_device_count() <= 0:
        pytest.fail("no GPU visible to the HIP runtime")
    return wake_amd


def _start(g, nx, ny, seed=3):
    r = np.random.default_rng(seed)
    u = r.uniform(-0.02, 0.02, (2, nx * ny)).astype(np.float32)
    g.initialize_fields(np.ones(nx * ny, np.float32), u[0] + np.float32(0.03), u[1])


def _channel(wa, nx, ny, storage, turb=False):
    g = wa.LatticeGrid2D(nx, ny, 0.6, storage=storage)
    _start(g, nx, ny)
    g.set_les_coupled(True)
    g.set_inflow_parabolic(0.05)
    if turb:
        g.set_inflow_turbulence(0.05, 11)
    g.set_outflow_east(1.0)
    g.set_solid_box(0, 0, nx - 1, 0)
    g.set_solid_box(0, ny - 1, nx - 1, ny - 1)
    g.set_solid_circle(nx / 3.0, ny / 2.0, max(1.0, ny / 8.0))
    return g


def _lid(wa, nx, ny, storage, periodic_y=False):
    g = wa.LatticeGrid2D(nx, ny, 0.58, storage=storage)
    _start(g, nx, ny, 5)
    g.set_solid_box(0, 0, 0, ny - 1)
    g.set_solid_box(nx // 2, ny // 3, nx // 2 + 1, ny // 2)
    g.set_moving_wall_north(0.06)
    if periodic_y:
        g.set_periodic_axes(True, False)
    return g


def _solid_in_periodic(wa, nx, ny, storage):
    g = wa.LatticeGrid2D(nx, ny, 0.7, storage=storage)
    _start(g, nx, ny, 9)
    g.set_solid_box(1, 1, 2, 2)
    g.set_periodic(True)
    return g


def _cavity(wa, nx, ny, storage):
    g = wa.LatticeGrid2D(nx, ny, 0.58, storage=storage)
    g.initialize(1.0, 0.0, 0.0)
    for box in ((0, 0, nx - 1, 0), (0, ny - 1, nx - 1, ny - 1), (0, 0, 0, ny - 1), (nx - 1, 0, nx - 1, ny - 1)):
        g.set_solid_box(*box)
    g.enable_thermal(0.62, 1e-3, 0.5, 0.5)
    g.set_temperature_field(np.random.default_rng(1).uniform(0, 1, nx * ny).astype(np.float32))
    g.set_wall_temperature(0, 0, 0, ny - 1, 1.0)
    return g


SCENES = {
    "channel": (_channel, [("TRT", False), ("MRT", True), ("BGK", False), ("TRT", True)], True),
    "noisy": (lambda *a: _channel(*a, turb=True), [("BGK", True)], True),
    "lid": (_lid, [("BGK", False), ("TRT", True)], True),
    "lid_periodic_y": (lambda *a: _lid(*a, periodic_y=True), [("MRT", False)], True),
    "solid_periodic": (_solid_in_periodic, [("MRT", False)], False),
    "cavity": (_cavity, [("MRT", False), ("BGK", False)], None),
}


def _state(g, thermal):
    out = [g.f_src_data().copy(), g.rho_data(), g.ux_data(), g.uy_data()]
    return out + ([g.temperature_data()] if thermal else [])


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("scene", list(SCENES))
@pytest.mark.parametrize("nx,ny", SIZES)
def test_tile_run_equals_single_steps(wa, nx, ny, scene, storage):
    make, kinds, forces = SCENES[scene]
    for coll, les, gx, gy in [k + g for k in kinds for g in ((1e-6, -2e-6), (0.0, 0.0))]:
        ends = []
        for multi in (True, False):
            g = make(wa, nx, ny, storage)
            g.set_multistep(multi)
            if forces:
                g.set_force_probe(nx / 3.0, ny / 2.0, 0.0, 0.0)
            for steps in (1, 3, 8, 2, 21):  # from a materialised state, remainders, several launches
                g.run(steps, coll, gx=gx, gy=gy, use_les=les, smag=0.17)
            end = _state(g, forces is None)
            if forces:
                end.append(g.force_history()[1])
                assert end[-1].shape == (36, 3)
            ends.append(end)
        for a, b in zip(*ends):
            assert np.array_equal(a, b, equal_nan=True), (coll, les, gx)


def test_force_history_over_mixed_steps(wa):
    """Tile launches, single steps, reads, a ring's worth of steps and a
    geometry change between them leave the history of single steps."""
    hist = []
    for multi in (True, False):
        g = _channel(wa, 150, 50, 0)
        g.set_multistep(multi)
        g.set_force_probe(50.0, 25.0, 0.0, 20.0)
        g.run(70, "MRT", use_les=True, smag=0.17)
        g.step("MRT", use_les=True, smag_const=0.17)
        g.run(9, "MRT", use_les=True, smag=0.17)
        mid = g.force_history()[1].copy()
        g.run(5, "MRT", use_les=True, smag=0.17)
        g.set_solid_box(90, 20, 92, 24)
        g.run(130, "MRT", use_les=True, smag=0.17)
        first, f = g.force_history()
        assert first == 0 and f.shape == (216, 3) and np.array_equal(f[:81], mid)
        hist.append(f)
    assert np.array_equal(*hist)


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("scene,chunk,graph", [("channel", 7, True), ("noisy", 16, False), ("lid", 100, True),
                                               ("cavity", 6, True)])
def test_batch_tiles_equal_single_steps(wa, scene, chunk, graph, storage):
    """A batch takes tile launches where all its members may: members of
    several sizes with their own step counts (ends inside a launch, chunks
    that are no multiple of a launch, a graph that is replayed) keep the bits
    and the forces of single-step launches, and can be stepped on alone."""
    make, kinds, forces = SCENES[scene]
    coll, les = kinds[0]
    sizes, steps = [(240, 80), (33, 17), (16, 16), (64, 33)], [5, 12, 43, 8]
    ends = []
    for multi in (True, False):
        grids = [make(wa, nx, ny, storage) for nx, ny in sizes]
        for g in grids:
            g.set_multistep(multi)
            if les or scene in ("channel", "noisy"):
                g.set_les_coupled(les)
        b = wa.Batch(lattice=9, storage=storage, collision=coll, use_les=les, chunk=chunk, thermal=forces is None)
        ids = [b.add(g, k, g=(1e-6, -1e-6, 0.0), smag=0.17,
                     forces=(nx / 3.0, ny / 2.0, 0.0, 0.0) if forces else None)
               for g, k, (nx, ny) in zip(grids, steps, sizes)]
        b.run(20, use_graph=graph)
        b.run(30, use_graph=graph)
        end = [b.forces(i) for i in ids]
        assert not forces or [len(f) for f in end] == steps
        for i, g in zip(ids, grids):
            b.remove(i)
            g.run(3, coll, use_les=les, smag=0.17)
            end += _state(g, forces is None)
        ends.append(end)
    for a, c in zip(*ends):
        assert np.array_equal(a, c, equal_nan=True)


def _warm_cavity(wa, nx, ny, storage):
    """Side walls at temperatures whose product with 2 w rounds."""
    g = _cavity(wa, nx, ny, storage)
    g.set_wall_temperature(0, 0, 0, ny - 1, 0.87)
    g.set_wall_temperature(nx - 1, 0, nx - 1, ny - 1, 0.21)
    return g


def _same_as_single_steps(wa, make, nx, ny, storage, coll, les=False, gx=0.0, gy=0.0, thermal=False, probe=False,
                          runs=(1, 3, 8, 2, 21)):
    ends = []
    for multi in (True, False):
        g = make(wa, nx, ny, storage)
        g.set_multistep(multi)
        if probe:
            # the node lists are built, then the history and the state set anew
            g.set_force_probe(nx / 3.0, ny / 2.0, 0.0, 0.0)
            g.run(24, coll, gx=gx, gy=gy, use_les=les, smag=0.17)
            g.add_noise(1e-4, 3)
        for steps in runs:
            g.run(steps, coll, gx=gx, gy=gy, use_les=les, smag=0.17)
        end = _state(g, thermal) + [g.f_dst_data().copy()]
        if probe:
            end.append(g.force_history()[1])
        ends.append(end)
    for k, (a, b) in enumerate(zip(*ends)):
        assert np.array_equal(a, b, equal_nan=True), k


@pytest.mark.parametrize("coll", ["BGK", "TRT", "MRT"])
@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("nx,ny", [(33, 17), (131, 8), (240, 80), (256, 256)])
def test_wall_temperatures_in_tiles(wa, nx, ny, storage, coll):
    """The anti-bounce-back term 2 w T_wall keeps the single step's rounding."""
    _same_as_single_steps(wa, _warm_cavity, nx, ny, storage, coll, gx=1e-6, gy=-2e-6, thermal=True)


def _thick_channel(wa, nx, ny, storage, turb=False):
    """Solid nodes inside the inlet and outlet rows: walls two nodes thick, a
    step at the inlet and a sill at the outlet."""
    g = _channel(wa, nx, ny, storage, turb)
    g.set_solid_box(0, 1, nx - 1, 1)
    g.set_solid_box(0, ny - 3, min(4, nx // 3), ny - 2)
    g.set_solid_box(nx - 2, ny // 2, nx - 1, ny // 2)
    return g


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("coll,les,turb", [("MRT", True, False), ("TRT", False, True)])
@pytest.mark.parametrize("nx,ny", [(240, 80), (33, 17), (17, 48), (9, 8)])
def test_solid_nodes_on_open_boundaries(wa, nx, ny, coll, les, turb, storage):
    """Their post-collision populations take the closures as in a single step."""
    _same_as_single_steps(wa, lambda *a: _thick_channel(*a, turb=turb), nx, ny, storage, coll, les, probe=True)


def test_solid_nodes_on_open_boundaries_of_a_cavity(wa):
    def make(wa, nx, ny, storage):
        g = _thick_channel(wa, nx, ny, storage)
        g.set_les_coupled(False)
        g.enable_thermal(0.62, 1e-3, 0.5, 0.5)
        g.set_temperature_field(np.random.default_rng(1).uniform(0, 1, nx * ny).astype(np.float32))
        g.set_wall_temperature(0, 0, nx - 1, 1, 0.87)
        return g

    _same_as_single_steps(wa, make, 64, 33, 0, "MRT", thermal=True)


@pytest.mark.parametrize("read", [False, True])
@pytest.mark.parametrize("gap", [1, 10, 100])
def test_force_history_around_batch_steps(wa, gap, read):
    """A batch takes no probe samples: the history ends where it stood, and
    later runs add none of steps that were not sampled."""
    hist = []
    for multi in (True, False):
        g = _channel(wa, 150, 50, 0)
        g.set_multistep(multi)
        g.set_force_probe(50.0, 25.0, 0.0, 20.0)
        g.run(20, "MRT", use_les=True, smag=0.17)
        before = g.force_history()[1].copy() if read else None
        b = wa.Batch(lattice=9, collision="MRT", use_les=True)
        slot = b.add(g, gap, smag=0.17)
        b.run(gap)
        b.remove(slot)
        g.run(30, "MRT", use_les=True, smag=0.17)
        first, f = g.force_history()
        assert first == 0 and (before is None or np.array_equal(f[:len(before)], before))
        # read at step 20, sample 20 is there, and a batch of one step leaves no gap
        assert len(f) == (20 + 1 + 30 + 1 if read and gap == 1 else 21 if read else 20)
        g.set_force_probe(50.0, 25.0, 0.0, 20.0)
        g.run(9, "MRT", use_les=True, smag=0.17)
        hist.append((f, g.force_history()[1]))
        assert len(hist[-1][1]) == 10
    for a, b in zip(*hist):
        assert np.array_equal(a, b)


def _porous(wa, nx, ny, storage):
    g = _channel(wa, nx, ny, storage)
    x, y = np.meshgrid(np.arange(nx), np.arange(ny))
    for i, j in zip(x[(x + y) % 3 == 0], y[(x + y) % 3 == 0]):
        if 4 < i < nx - 4:
            g.set_cell_type(int(i), int(j), 1)
    return g


def test_force_history_of_short_runs(wa):
    """Runs too short to pay for the node lists, geometries and probes that
    change between them, and runs after the lists were built."""
    hist = []
    for multi in (True, False):
        g = _channel(wa, 150, 50, 0)
        g.set_multistep(multi)
        g.set_force_probe(50.0, 25.0, 0.0, 20.0)
        out = []
        for k, steps in enumerate((7, 8, 8, 7, 9, 2, 40, 3, 8, 30, 1, 25)):
            if k in (3, 7):
                g.set_solid_box(90 + k, 20, 91 + k, 24)
            if k == 9:
                out.append(g.force_history()[1].copy())
                g.set_force_probe(60.0, 25.0, 0.0, 30.0)
            g.run(steps, "MRT", use_les=True, smag=0.17)
        out.append(g.force_history()[1].copy())
        assert [len(f) for f in out] == [93, 57]
        hist.append(out)
    for a, b in zip(*hist):
        assert np.array_equal(a, b)


def test_force_samples_of_a_porous_body(wa):
    """The lists of a tile launch's samples are bounded by the state's size:
    a body with a link in most nodes is sampled by single steps."""
    nx, ny = 512, 300
    hist = []
    for multi in (True, False):
        g = _porous(wa, nx, ny, 0)
        g.set_multistep(multi)
        g.run(2, "TRT")
        before = g.device_bytes()
        g.set_force_probe(nx / 2.0, ny / 2.0, 0.0, 0.0)
        g.run(3, "TRT")
        g.run(60, "TRT")
        assert g.device_bytes() - before < 64 << 20
        hist.append(g.force_history()[1])
    assert np.array_equal(*hist)


# One size for each instance of the tile kernels besides the 32 x 24 tile of
# the sizes above: 32 x 32 tiles of 8 steps (more than 256 low tiles, at most
# 512 high ones; 256 with FP32 temperature), and of 4 steps beyond.
EIGHT, FOUR = (259, 250), (530, 263)


def _tiles(nx, ny, w, h):
    return -(-nx // w) * -(-ny // h)


def test_sizes_reach_their_instances():
    assert _tiles(*EIGHT, 16, 8) > 256 and _tiles(*EIGHT, 16, 16) <= 512
    assert _tiles(*FOUR, 16, 16) > 512
    assert _tiles(240, 250, 16, 8) > 256 and _tiles(240, 250, 16, 16) <= 256
    assert _tiles(*EIGHT, 16, 16) > 256  # FP32 temperature: 4 steps from here


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("coll,les", [("BGK", False), ("BGK", True), ("TRT", False), ("TRT", True), ("MRT", False),
                                      ("MRT", True)])
@pytest.mark.parametrize("nx,ny", [EIGHT, FOUR])
def test_larger_tiles_with_edges(wa, nx, ny, coll, les, storage, force):
    gx, gy = (1e-6, -2e-6) if force else (0.0, 0.0)
    _same_as_single_steps(wa, _thick_channel, nx, ny, storage, coll, les, gx, gy, probe=True, runs=(1, 3, 8, 13))
    _same_as_single_steps(wa, _lid, nx, ny, storage, coll, False, gx, gy, runs=(5, 8))


def _vortex(wa, nx, ny, storage):
    g = wa.LatticeGrid2D(nx, ny, 0.7, storage=storage)
    _start(g, nx, ny, 4)
    g.set_les_coupled(True)
    g.set_periodic(True)
    return g


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("coll,les", [("BGK", False), ("BGK", True), ("TRT", False), ("TRT", True), ("MRT", False),
                                      ("MRT", True)])
@pytest.mark.parametrize("nx,ny", [(240, 80), EIGHT, FOUR])
def test_larger_tiles_of_periodic_domains(wa, nx, ny, coll, les, storage, force):
    gx, gy = (1e-6, -2e-6) if force else (0.0, 0.0)
    _same_as_single_steps(wa, _vortex, nx, ny, storage, coll, les, gx, gy, runs=(1, 3, 8, 13))


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("coll", ["BGK", "TRT", "MRT"])
@pytest.mark.parametrize("nx,ny", [(240, 250), EIGHT, FOUR])
def test_larger_tiles_with_temperature(wa, nx, ny, coll, storage):
    _same_as_single_steps(wa, _warm_cavity, nx, ny, storage, coll, gx=1e-6, gy=-2e-6, thermal=True,
                          runs=(1, 3, 8, 13))


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("coll,les", [("BGK", False), ("BGK", True), ("TRT", False), ("TRT", True), ("MRT", False),
                                      ("MRT", True)])
@pytest.mark.parametrize("sizes", [[(96, 40), (33, 17)], [FOUR, (96, 40)]])
def test_batch_tiles_of_both_spans(wa, sizes, coll, les, storage, force):
    """Eight steps per launch, and four once the batch has more than 512 tiles."""
    few = sum(_tiles(nx, ny, 16, 16) for nx, ny in sizes) <= 512
    assert few == (sizes[0] != FOUR)
    ends = []
    for multi in (True, False):
        grids = [_thick_channel(wa, nx, ny, storage) for nx, ny in sizes]
        for g in grids:
            g.set_les_coupled(les)
            g.set_multistep(multi)
        b = wa.Batch(lattice=9, storage=storage, collision=coll, use_les=les, chunk=11)
        ids = [b.add(g, k, g=(1e-6, -1e-6, 0.0) if force else (0.0, 0.0, 0.0), smag=0.17,
                     forces=(nx / 3.0, ny / 2.0, 0.0, 0.0))
               for g, k, (nx, ny) in zip(grids, (23, 14), sizes)]
        b.run(23)
        end = [b.forces(i) for i in ids]
        for g in grids:
            end += _state(g, False) + [g.f_dst_data().copy()]
        ends.append(end)
    for a, c in zip(*ends):
        assert np.array_equal(a, c, equal_nan=True)


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("coll", ["BGK", "TRT", "MRT"])
@pytest.mark.parametrize("sizes", [[(96, 40), (33, 17)], [FOUR, (96, 40)]])
def test_batch_tiles_of_cavities(wa, sizes, coll, storage):
    """The members end as when stepped alone, one launch per step."""
    ends = []
    for batched in (True, False):
        grids = [_warm_cavity(wa, nx, ny, storage) for nx, ny in sizes]
        if batched:
            b = wa.Batch(lattice=9, storage=storage, collision=coll, chunk=11, thermal=True)
            for g, k in zip(grids, (23, 14)):
                b.add(g, k)
            b.run(23)
        else:
            for g, k in zip(grids, (23, 14)):
                g.set_multistep(False)
                g.run(k, coll)
        ends.append([v for g in grids for v in _state(g, True)])
    for a, c in zip(*ends):
        assert np.array_equal(a, c, equal_nan=True)


@pytest.mark.parametrize("storage", [0, 1, 2])
def test_solid_nodes_on_open_boundaries_between_calls(wa, storage):
    """f_dst after a change of the geometry, after one step from a given state
    (which closes nothing) and after a batch."""
    ends = []
    for multi in (True, False):
        g = _thick_channel(wa, 64, 33, storage, turb=True)
        g.set_multistep(multi)
        out = []
        for steps in (9, 2, 16):
            g.run(steps, "TRT")
            g.set_cell_type(0, 30, 0)
            g.set_cell_type(0, 29, 1)
            out.append(g.f_dst_data().copy())
            g.run(1, "TRT")
            out.append(g.f_dst_data().copy())
            g.set_populations(1.01 * g.f_src_data())
            g.run(1, "TRT")
            out.append(g.f_dst_data().copy())
            g.run(2, "TRT")
            out.append(g.f_dst_data().copy())
            b = wa.Batch(lattice=9, storage=storage, collision="TRT", use_les=True, chunk=5)
            slot = b.add(g, steps, smag=0.17)
            b.run(steps)
            b.remove(slot)
            out.append(g.f_dst_data().copy())
            out.append(g.f_src_data().copy())
        ends.append(out)
    for k, (a, b) in enumerate(zip(*ends)):
        assert np.array_equal(a, b), k
