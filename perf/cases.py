"""The work that programs on this package spend their time in, as cases.

A case is one call sequence that a user's program repeats: advance a grid by
some steps and read back what the program looks at (force histories, fields,
flow features, checkpoints), run a batch of domains, or call the kernel
exports on host arrays.  `prepare` makes what the program holds before the
call (grids with their geometry, boundary conditions and initial state),
`run` is the call, `exact` the same result from plain torch in 64 bits.

Kinds of cases and where they stand for real use:
  * "flow": one grid advanced by `steps` steps through run(), then read back.
    Scenes: "vortex" (periodic, no walls: validation runs), "cylinder" (2D
    channel with a circle, the wake scenario), "lid" (box with a moving lid
    and an obstacle), "cavity" (2D flow coupled to a temperature), "sphere"
    (3D with curved-wall links, turbulent inlet, convective outlet),
    "ellipsoid" (the same outer flow around a voxelized body) and "wing" (a
    NACA section between side walls).
  * "batch": many 2D wakes of uneven size advanced together, with the force
    of every step, as a parameter sweep does.
  * "fields": a few steps, then the observables of a monitored run:
    vorticity, Q-criterion, total mass, kinetic energy, largest speed.
  * "restart": a grid set from fields, advanced, and its populations and
    moments read back, as a checkpointing program does.
  * "kernels": one step of a program that calls the exported kernels on its
    own host arrays (collide, stream, moments, speed).
"""
import math

import numpy as np
import torch

F32, F16, BF16 = 0, 1, 2
CS = 0.17


def listed():
    return [
        # the plain periodic validation run, 256 x 256
        dict(name="vortex_2d_256", kind="flow", scene="vortex", lattice=9, nx=256, ny=256, nz=1, storage=F32,
             collision="BGK", les=False, tau=0.8, steps=100, forces=False),
        # the wake scenario at the size of the integration test, force of every step
        dict(name="cylinder_2d_240", kind="flow", scene="cylinder", lattice=9, nx=240, ny=80, nz=1, storage=F32,
             collision="TRT", les=False, tau=0.56, steps=100, forces=True),
        # a well resolved 2D wake, ragged rows
        dict(name="cylinder_2d_1500", kind="flow", scene="cylinder", lattice=9, nx=1500, ny=403, nz=1, storage=F32,
             collision="MRT", les=True, tau=0.51, steps=200, forces=True),
        # a heated cavity of the request mix
        dict(name="cavity_2d_256", kind="flow", scene="cavity", lattice=9, nx=256, ny=256, nz=1, storage=F32,
             collision="MRT", les=False, tau=0.55, steps=200, forces=False),
        # a small closed 3D box, odd sizes: launches and latency count
        dict(name="lid_3d_61", kind="flow", scene="lid", lattice=19, nx=61, ny=45, nz=37, storage=F32,
             collision="TRT", les=False, tau=0.6, steps=50, forces=False),
        # the headline configuration: its result is the force history
        dict(name="sphere_3d_256", kind="flow", scene="sphere", lattice=19, nx=256, ny=256, nz=256, storage=F32,
             collision="MRT", les=True, tau=0.505, steps=100, forces=True),
        # a bluff body of the request mix with 16-bit storage, fields read at the end
        dict(name="ellipsoid_3d_128_f16", kind="flow", scene="ellipsoid", lattice=19, nx=128, ny=128, nz=128,
             storage=F16, collision="MRT", les=True, tau=0.52, steps=100, forces=False),
        # the wing channel at half size
        dict(name="wing_3d_192_bf16", kind="flow", scene="wing", lattice=27, nx=192, ny=96, nz=96, storage=BF16,
             collision="TRT", les=True, tau=0.52, steps=100, forces=True),
        # a sweep of wakes in one batch
        dict(name="batch_2d_32", kind="batch", members=32, lattice=9, nx=448, steps=200),
        # observables of a monitored 3D run
        dict(name="fields_3d_144", kind="fields", lattice=19, nx=144, ny=120, nz=97, storage=F32, collision="MRT",
             les=True, tau=0.55, steps=10),
        # set from fields, advanced, checkpointed
        dict(name="restart_3d_96", kind="restart", lattice=19, nx=96, ny=80, nz=64, storage=F32, collision="BGK",
             les=False, tau=0.7, steps=10),
        # the exported kernels on host arrays, as a program linked against them calls them
        dict(name="kernels_3d_40", kind="kernels", lattice=19, nx=40, ny=36, nz=33, collision="MRT", tau=0.6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["flow2", "flow2", "cavity", "flow3", "flow3", "batch", "fields", "restart", "kernels"])
    coll, les = rng.choice([("BGK", False), ("TRT", False), ("MRT", False), ("MRT", True), ("TRT", True)])
    storage = rng.choice([F32, F32, F16, BF16])
    steps = rng.randint(40, 120)
    tau = round(rng.uniform(0.52, 0.8), 4)
    if kind == "flow2":
        scene = rng.choice(["vortex", "cylinder", "lid"])
        nx = _log(rng, 96, 1600)
        ny = max(40, int(nx * rng.uniform(0.25, 0.6)))
        return dict(kind="flow", scene=scene, lattice=9, nx=nx, ny=ny, nz=1, storage=storage, collision=coll,
                    les=les, tau=tau, steps=steps, forces=scene == "cylinder")
    if kind == "cavity":
        n = _log(rng, 96, 512)
        return dict(kind="flow", scene="cavity", lattice=9, nx=n, ny=n, nz=1, storage=storage, collision="MRT",
                    les=False, tau=tau, steps=steps, forces=False)
    if kind == "flow3":
        scene = rng.choice(["vortex", "lid", "sphere", "ellipsoid", "wing"])
        n = _log(rng, 40, 200)
        lat = 27 if scene == "wing" else 19
        if lat == 27 and coll == "MRT":
            coll = "TRT"
        return dict(kind="flow", scene=scene, lattice=lat, nx=n, ny=max(32, int(n * rng.uniform(0.5, 1.0))),
                    nz=max(32, int(n * rng.uniform(0.4, 0.9))), storage=storage, collision=coll, les=les, tau=tau,
                    steps=rng.randint(20, 60), forces=scene in ("sphere", "wing") and rng.random() < 0.7)
    if kind == "batch":
        return dict(kind="batch", members=rng.randint(8, 32), lattice=9, nx=32 * rng.randint(4, 18),
                    steps=rng.randint(100, 200))
    if kind == "fields":
        n = _log(rng, 48, 160)
        return dict(kind="fields", lattice=19, nx=n, ny=max(32, int(n * rng.uniform(0.5, 1.0))),
                    nz=max(32, int(n * rng.uniform(0.5, 1.0))), storage=rng.choice([F32, F16]), collision=coll,
                    les=les, tau=tau, steps=rng.randint(5, 20))
    if kind == "restart":
        n = _log(rng, 40, 112)
        return dict(kind="restart", lattice=rng.choice([19, 27]), nx=n, ny=max(32, int(n * rng.uniform(0.5, 1.0))),
                    nz=max(32, int(n * rng.uniform(0.5, 1.0))), storage=F32, collision="BGK", les=False, tau=tau,
                    steps=rng.randint(5, 20))
    return dict(kind="kernels", lattice=19, nx=rng.randint(24, 72), ny=rng.randint(24, 64), nz=rng.randint(16, 48),
                collision=rng.choice(["BGK", "TRT", "MRT"]), tau=tau)


def work(case):
    """Bytes and operations that a pass cannot do without: the state read and
    written once a step where it is larger than what the chip's local memories
    hold (40 MB), once a pass where it fits, and the results once; operations
    as a plain collision of the lattice counts them."""
    flops_node = {9: 250.0, 19: 700.0, 27: 1000.0}
    if case["kind"] == "batch":
        n = sum(nx * ny for nx, ny, *_ in _wakes(case, 1))
        q, elem, fields, steps = 9, 4, 3, case["steps"]
    else:
        n = case["nx"] * case["ny"] * case["nz"]
        q = case["lattice"] + (5 if case.get("scene") == "cavity" else 0)
        elem = 4 if case.get("storage", F32) == F32 else 2
        steps = case.get("steps", 1)
        fields = {"flow": 1 if case.get("nz") == 256 else 4, "fields": 4 + 4, "restart": 8 + q, "kernels": q + 4}[
            case["kind"]]
    state = 2.0 * q * elem * n
    times = steps if state / 2 > 40e6 else 1
    return {"bytes": state * times + 4.0 * fields * n, "flops": flops_node[case["lattice"]] * n * steps}


# ------------------------------------------------------------ scene geometry
def _f(v):
    """The value a float argument of the library takes."""
    return float(np.float32(v))


def _scene(case, seed):
    """Parameters of a scene, drawn from the seed."""
    r = np.random.default_rng(1000 + seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    s = dict(tau=_f(case["tau"]), u=_f(0.05 * r.uniform(0.8, 1.1)), seed=int(r.integers(1, 1 << 30)))
    scene = case["scene"]
    if scene == "cylinder":
        D = ny / 8.0
        s.update(D=D, cx=_f(nx / 5.0 + r.uniform(-1, 1)), cy=_f(ny / 2.0 + r.uniform(-2, 2)))
    elif scene == "lid":
        s.update(uw=_f(0.06 * r.uniform(0.8, 1.1)), box=int(r.integers(nx // 4, nx // 2)))
    elif scene == "cavity":
        s.update(t0=r.uniform(0.4, 0.5), dt=_f(r.uniform(0.8, 1.0)))
    elif scene in ("sphere", "ellipsoid"):
        m = min(nx, ny, nz)
        s.update(R=_f(m * 0.094), cx=_f(nx / 4.0 + r.uniform(-1, 1)), cy=_f(ny / 2.0 + r.uniform(-1, 1)),
                 cz=_f(nz / 2.0 + r.uniform(-1, 1)), axes=[_f(m * v) for v in r.uniform(0.08, 0.16, 3)])
    elif scene == "wing":
        s.update(chord=_f(nx / 4.0), aoa=_f(r.uniform(5.0, 9.0)), lx=_f(nx / 4.0), ly=_f(ny / 2.0 + r.uniform(-1, 1)))
    return s


def _modes(case, seed):
    """A smooth periodic start of the flow: density and velocity fields, float32."""
    r = np.random.default_rng(2000 + seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    x = 2 * np.pi * np.arange(nx) / nx
    y = 2 * np.pi * np.arange(ny) / ny
    z = 2 * np.pi * np.arange(nz) / nz
    Z, Y, X = np.meshgrid(z, y, x, indexing="ij", sparse=True)
    a = 0.04 * r.uniform(0.8, 1.1)
    px, py, pz = r.uniform(0, 2 * np.pi, 3)
    one = np.ones((nz, ny, nx))
    if nz == 1:
        ux = a * np.sin(X + px) * np.cos(Y + py) * one
        uy = -a * np.cos(X + px) * np.sin(Y + py) * one
        uz = 0 * one
    else:
        ux = a * np.cos(X + px) * np.sin(Y + py) * np.sin(Z + pz) * one
        uy = -0.5 * a * np.sin(X + px) * np.cos(Y + py) * np.sin(Z + pz) * one
        uz = -0.5 * a * np.sin(X + px) * np.sin(Y + py) * np.cos(Z + pz) * one
    rho = 1.0 + 0.02 * a * np.cos(X + px) * np.cos(Y + py) * one
    return tuple(np.ascontiguousarray(v, dtype=np.float32) for v in (rho, ux, uy, uz))


def _disturbed(case, seed, u):
    """A stream along x with smooth disturbances, float32 fields."""
    rho, ux, uy, uz = _modes(case, seed)
    k = np.float32(0.25)
    return rho, np.float32(u) + k * ux, k * uy, k * uz


def _profile(ny, umax):
    s = np.arange(ny, dtype=np.float64) - 0.5
    H = ny - 2
    return np.clip(4.0 * umax * s * (H - s) / (H * H), 0.0, None)


def _wakes(case, seed):
    """(nx, ny, tau, cx, cy, D) of the members of a batch of wakes."""
    r = np.random.default_rng(3000 + seed)
    out = []
    for i in range(case["members"]):
        # sizes are the case's own, flows the seed's: NX uneven around the case's
        nx = max(128, case["nx"] + 32 * ((i * 7) % 9 - 4))
        ny = nx // 4
        D = ny / 8.0
        re = math.exp(r.uniform(math.log(50.0), math.log(300.0)))
        out.append((nx, ny, _f(3.0 * (2.0 / 3.0 * 0.05) * D / re + 0.5), _f(nx / 5.0),
                    _f(ny / 2.0 + float(r.integers(-2, 3))), D))
    return out


def _wake_grid(wake_amd, nx, ny, tau, cx, cy, D, umax=0.05):
    g = wake_amd.LatticeGrid2D(nx, ny, tau)
    prof = np.repeat(_profile(ny, umax), nx).astype(np.float32)
    g.initialize_fields(np.ones(nx * ny, np.float32), prof, np.zeros(nx * ny, np.float32))
    g.set_les_coupled(True)
    g.set_inflow_parabolic(umax)
    g.set_outflow_east(1.0)
    g.set_solid_box(0, 0, nx - 1, 0)
    g.set_solid_box(0, ny - 1, nx - 1, ny - 1)
    g.set_solid_circle(cx, cy, D / 2)
    return g


def _grid(case, seed):
    """The grid of a "flow" case with its geometry, boundaries and state."""
    import wake_amd

    nx, ny, nz, scene = case["nx"], case["ny"], case["nz"], case["scene"]
    s = _scene(case, seed)
    two = case["lattice"] == 9
    if two:
        g = wake_amd.LatticeGrid2D(nx, ny, s["tau"], storage=case["storage"])
    else:
        g = wake_amd.LatticeGrid3D(nx, ny, nz, s["tau"], lattice=case["lattice"], storage=case["storage"])
    if case["les"]:
        g.set_les_coupled(True)
    if scene == "vortex":
        if two:
            g.set_periodic(True)
            g.initialize_fields(*_modes(case, seed)[:3])
        else:
            g.initialize_fields(*_modes(case, seed))
    elif scene == "cylinder":
        prof = np.repeat(_profile(ny, s["u"]), nx).astype(np.float32)
        g.initialize_fields(np.ones(nx * ny, np.float32), prof, np.zeros(nx * ny, np.float32))
        g.set_inflow_parabolic(s["u"])
        g.set_outflow_east(1.0)
        g.set_solid_box(0, 0, nx - 1, 0)
        g.set_solid_box(0, ny - 1, nx - 1, ny - 1)
        g.set_solid_circle(s["cx"], s["cy"], s["D"] / 2)
    elif scene == "lid":
        b = s["box"]
        if two:
            g.initialize(1.0, 0.0, 0.0)
            g.set_solid_box(0, 0, 0, ny - 1)
            g.set_solid_box(nx - 1, 0, nx - 1, ny - 1)
            g.set_solid_box(b, ny // 3, b + nx // 8, ny // 3 + ny // 8)
            g.set_moving_wall_north(s["uw"])
        else:
            g.initialize(1.0, 0.0, 0.0, 0.0)
            g.set_solid_box(0, 0, 0, 0, ny - 1, nz - 1)
            g.set_solid_box(nx - 1, 0, 0, nx - 1, ny - 1, nz - 1)
            g.set_solid_box(b, ny // 3, nz // 3, b + nx // 8, ny // 3 + ny // 8, nz // 3 + nz // 8)
            g.set_moving_wall_top(s["uw"], 0.0)
    elif scene == "cavity":
        n, H = nx, nx - 2
        g.initialize(1.0, 0.0, 0.0)
        for box in ((0, 0, n - 1, 0), (0, n - 1, n - 1, n - 1), (0, 0, 0, n - 1), (n - 1, 0, n - 1, n - 1)):
            g.set_solid_box(*box)
        g.enable_thermal(s["tau"] + 0.1, 0.01 / H, 0.5, 0.5)
        g.set_temperature_field(_temperature(case, s))
        g.set_wall_temperature(0, 0, 0, n - 1, s["dt"])
        g.set_wall_temperature(n - 1, 0, n - 1, n - 1, 0.0)
    else:
        g.set_periodic_axes(scene != "wing", True)
        if scene == "wing":
            g.initialize_fields(*_disturbed(case, seed, s["u"]))
        else:
            g.initialize(1.0, s["u"], 0.0, 0.0)
        g.set_inflow_west(s["u"], 0.0)
        g.set_convective_outflow_east(s["u"])
        if scene != "ellipsoid":
            g.set_inflow_turbulence(0.01, s["seed"])
        if scene == "sphere":
            g.set_solid_sphere(s["cx"], s["cy"], s["cz"], s["R"])
            g.build_curved_sphere_links(s["cx"], s["cy"], s["cz"], s["R"])
        elif scene == "ellipsoid":
            g.set_solid_ellipsoid(s["cx"], s["cy"], s["cz"], *s["axes"])
        else:
            g.set_solid_naca("0012", s["chord"], s["aoa"], s["lx"], s["ly"])
    return g, s


def _temperature(case, s):
    n = case["nx"]
    x = np.linspace(0.0, 1.0, n)
    return np.ascontiguousarray(np.broadcast_to(s["t0"] + 0.4 * np.cos(np.pi * x), (n, n)), dtype=np.float32)


def _probe(case, s):
    """Centre and radius of the force sums of a scene."""
    if case["scene"] == "cylinder":
        return (s["cx"], s["cy"], 0.0, _f(1.5 * s["D"]))
    if case["scene"] == "wing":
        return (0.0, 0.0, 0.0, 0.0)
    return (s["cx"], s["cy"], s["cz"], _f(2.0 * s["R"]))


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    import wake_amd

    kind = case["kind"]
    if kind == "flow":
        g, s = _grid(case, seed)
        g.synchronize()
        if case["scene"] == "cavity":
            reads = [g.rho_data, g.ux_data, g.uy_data, g.temperature_data]
        elif case["lattice"] == 9:
            reads = [g.rho_data, g.ux_data, g.uy_data]
        elif case["nz"] == 256:
            reads = []
        else:
            reads = [g.rho_data, g.ux_data, g.uy_data, g.uz_data]
        return dict(case=case, g=g, probe=_probe(case, s) if case["forces"] else None, reads=reads)
    if kind == "batch":
        members = _wakes(case, seed)
        return dict(case=case, members=members, grids=[_wake_grid(wake_amd, *m) for m in members])
    if kind in ("fields", "restart"):
        g = wake_amd.LatticeGrid3D(case["nx"], case["ny"], case["nz"], _f(case["tau"]), lattice=case["lattice"],
                                   storage=case["storage"])
        if case["les"]:
            g.set_les_coupled(True)
        start = _modes(case, seed)
        if kind == "fields":
            g.initialize_fields(*start)
        g.synchronize()
        return dict(case=case, g=g, start=start)
    f, cells = _host_arrays(case, seed)
    n = cells.size
    out = dict(case=case, f=f, cells=cells, a=np.empty_like(f), s=np.empty_like(f))
    for k in ("rho", "ux", "uy", "uz", "speed"):
        out[k] = np.zeros(n, np.float32)
    return out


def _host_arrays(case, seed):
    """Populations near an equilibrium and cell types with a solid block."""
    rho, ux, uy, uz = (torch.from_numpy(v).double() for v in _modes(case, seed))
    L = _Lat(19, "cpu")
    f = torch.stack([_feq(L, q, rho, ux, uy, uz) for q in range(19)])
    noise = torch.from_numpy(np.random.default_rng(4000 + seed).uniform(-1e-3, 1e-3, tuple(f.shape)))
    w = torch.tensor(L.w).view(19, 1, 1, 1)
    f = np.ascontiguousarray((f + w * noise).numpy().astype(np.float32).reshape(19, -1))
    cells = np.zeros((case["nz"], case["ny"], case["nx"]), np.uint8)
    b = case["nx"] // 3
    cells[case["nz"] // 3: case["nz"] // 2, case["ny"] // 3: case["ny"] // 2, b:b + 6] = 1
    return f, cells.reshape(-1)


# ----------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "flow":
        g, out = state["g"], {}
        if state["probe"]:
            g.set_force_probe(*state["probe"])
        g.run(case["steps"], case["collision"], use_les=case["les"], smag=CS)
        if state["probe"]:
            out["forces"] = g.force_history()[1]
        out["fields"] = [read() for read in state["reads"]]
        return out
    if kind == "batch":
        return _run_batch(state)
    if kind == "fields":
        g = state["g"]
        g.run(case["steps"], case["collision"], use_les=case["les"], smag=CS)
        return {"features": list(g.vorticity_q_data()), "mass": g.compute_total_mass(),
                "energy": g.compute_total_kinetic_energy(), "speed": g.compute_max_speed()}
    if kind == "restart":
        g = state["g"]
        g.initialize_fields(*state["start"])
        g.run(case["steps"], case["collision"], use_les=case["les"], smag=CS)
        return {"populations": g.f_src_data(), "fields": [g.rho_data(), g.ux_data(), g.uy_data(), g.uz_data()]}
    return _run_kernels(state)


def _run_batch(state):
    import wake_amd

    case = state["case"]
    b = wake_amd.Batch(lattice=9, collision="MRT", use_les=True, chunk=100)
    ids = [b.add(g, case["steps"], smag=CS, forces=(cx, cy, 0.0, _f(1.5 * D)))
           for g, (nx, ny, tau, cx, cy, D) in zip(state["grids"], state["members"])]
    b.run(case["steps"])
    out = {"forces": np.stack([b.forces(i) for i in ids])}
    for i in ids:
        b.remove(i)
    out["ux"] = np.concatenate([g.ux_data() for g in state["grids"]])
    out["uy"] = np.concatenate([g.uy_data() for g in state["grids"]])
    return out


def _run_kernels(state):
    from wake_amd import kernels

    case, k = state["case"], kernels.kernel
    f, a, s, cells = state["f"], state["a"], state["s"], state["cells"]
    rho, ux, uy, uz = state["rho"], state["ux"], state["uy"], state["uz"]
    n, tau = cells.size, _f(case["tau"])
    if case["collision"] == "BGK":
        k("d3q19_collide_bgk", f, a, cells, rho, ux, uy, uz, tau, 0.0, 0.0, 0.0, n)
    elif case["collision"] == "TRT":
        k("d3q19_collide_trt", f, a, cells, rho, ux, uy, uz, tau, _f(_tau_a(tau)), 0.0, 0.0, 0.0, n)
    else:
        k("d3q19_collide_mrt", f, a, cells, rho, ux, uy, uz, tau, _f(1.19), 0.0, 0.0, 0.0, n)
    k("d3q19_stream_with_boundaries", a, s, cells, case["nx"], case["ny"], case["nz"], 0.0, 0.0, 0.0)
    k("d3q19_compute_macroscopic_moments_forced", s, rho, ux, uy, uz, 0.0, 0.0, 0.0, n)
    k("d3q19_compute_velocity_magnitude", ux, uy, uz, state["speed"], n)
    return {"populations": s, "fields": [rho, ux, uy, uz, state["speed"]]}


# ------------------------------------------------------- the same in 64 bits
class _Lat:
    """A velocity set: directions, weights, opposites."""

    def __init__(self, q, dev):
        if q == 9:
            c = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (1, 1, 0), (-1, 1, 0), (-1, -1, 0),
                 (1, -1, 0)]
            wt = {0: 4 / 9, 1: 1 / 9, 2: 1 / 36}
        else:
            c = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
            c += [(a, b, 0) for b in (1, -1) for a in (1, -1)]
            c += [(a, 0, b) for b in (1, -1) for a in (1, -1)]
            c += [(0, a, b) for b in (1, -1) for a in (1, -1)]
            if q == 27:
                c += [(a, b, d) for d in (1, -1) for b in (1, -1) for a in (1, -1)]
            wt = ({0: 1 / 3, 1: 1 / 18, 2: 1 / 36} if q == 19 else {0: 8 / 27, 1: 2 / 27, 2: 1 / 54, 3: 1 / 216})
        self.Q, self.c, self.dev = q, c, dev
        self.w = [wt[sum(v * v for v in d)] for d in c]
        self.opp = [c.index(tuple(-v for v in d)) for d in c]


def _feq(L, q, rho, ux, uy, uz):
    cu = L.c[q][0] * ux + L.c[q][1] * uy + L.c[q][2] * uz
    return L.w[q] * rho * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * (ux * ux + uy * uy + uz * uz))


def _tau_a(tau):
    return 0.5 + 0.25 / max(1e-4, tau - 0.5)


def _signed(L, f, weight):
    """Sum over q of an integer weight times f_q."""
    s = None
    for q in range(L.Q):
        k = weight(*L.c[q])
        if k:
            t = f[q] if k == 1 else -f[q] if k == -1 else k * f[q]
            s = t.clone() if s is None else s.add_(t)
    return s


def _basis(L):
    """Moment basis as rows of values at the velocities, and its rates by name."""
    rows = []
    for x, y, z in L.c:
        r2 = x * x + y * y + z * z
        if L.Q == 9:
            rows.append([1, 3 * r2 - 4, (9 * r2 * r2 - 21 * r2 + 8) / 2, x, (3 * r2 - 5) * x, y, (3 * r2 - 5) * y,
                         x * x - y * y, x * y])
        else:
            rows.append([1, 19 * r2 - 30, (21 * r2 * r2 - 53 * r2 + 24) / 2, x, (5 * r2 - 9) * x, y,
                         (5 * r2 - 9) * y, z, (5 * r2 - 9) * z, 3 * x * x - r2, (3 * r2 - 5) * (3 * x * x - r2),
                         y * y - z * z, (3 * r2 - 5) * (y * y - z * z), x * y, y * z, x * z, (y * y - z * z) * x,
                         (z * z - x * x) * y, (x * x - y * y) * z])
    return np.array(rows, dtype=np.float64).T


def _collide(L, f, coll, tau, les, gy=None):
    """Collided populations of every node (gy: an acceleration per node, 2D)."""
    dim2 = L.Q == 9
    rho = f.sum(0)
    jx, jy = _signed(L, f, lambda x, y, z: x), _signed(L, f, lambda x, y, z: y)
    jz = None if dim2 else _signed(L, f, lambda x, y, z: z)
    ux, uy = jx / rho, jy / rho
    if gy is not None:
        uy = uy + 0.5 * gy
    uz = torch.zeros((), dtype=torch.float64, device=f.device) if dim2 else jz / rho
    if les:
        t = 0
        pairs = [(0, 0), (1, 1), (0, 1)] + ([] if dim2 else [(2, 2), (1, 2), (0, 2)])
        u = (ux, uy, uz)
        for a, b in pairs:
            p = _signed(L, f, lambda *c: c[a] * c[b]) - rho * u[a] * u[b]
            if a == b:
                p = p - rho / 3
            t = t + (p * p if a == b else 2 * p * p)
        tau_e = 0.5 * (tau + torch.sqrt(tau * tau + 18 * math.sqrt(2.0) * _f(CS) ** 2 / rho * torch.sqrt(2 * t)))
    else:
        tau_e = tau
    if coll == "MRT" and L.Q != 27:
        M = _basis(L)
        u2 = ux * ux + uy * uy + uz * uz
        n = f.shape[1:]
        m = (torch.from_numpy(M).to(f.device) @ f.reshape(L.Q, -1)).reshape(L.Q, *n)
        s = 1.0 / tau_e
        if dim2:
            eq = {1: rho * (-2 + 3 * u2), 2: rho * (1 - 3 * u2), 4: -rho * ux, 6: -rho * uy,
                  7: rho * (ux * ux - uy * uy), 8: rho * ux * uy}
            rate = {1: 1 / 1.63, 2: 1.4, 4: 1.6, 6: 1.6, 7: s, 8: s}
            inv = np.linalg.inv(M)
        else:
            d = rho * (2 * ux * ux - uy * uy - uz * uz)
            e = rho * (uy * uy - uz * uz)
            eq = {1: rho * (-11 + 19 * u2), 2: rho * (3 - 5.5 * u2), 4: -2 / 3 * rho * ux, 6: -2 / 3 * rho * uy,
                  8: -2 / 3 * rho * uz, 9: d, 10: -0.5 * d, 11: e, 12: -0.5 * e, 13: rho * ux * uy, 14: rho * uy * uz,
                  15: rho * ux * uz, 16: 0.0, 17: 0.0, 18: 0.0}
            rate = {1: 1 / 1.19, 2: 1.4, 4: 1.2, 6: 1.2, 8: 1.2, 9: s, 10: 1.4, 11: s, 12: 1.4, 13: s, 14: s, 15: s,
                    16: 1.98, 17: 1.98, 18: 1.98}
            inv = np.round(np.linalg.inv(M), 7)  # the scheme's inverse has seven decimals
        for k, v in eq.items():
            m[k] -= rate[k] * (m[k] - v)
        if gy is not None:
            F, h = rho * gy, 1 - 0.5 * s
            m[1] += h * 6 * uy * F
            m[2] -= h * 6 * uy * F
            m[5] += F
            m[6] -= h * F
            m[7] -= h * 2 * uy * F
            m[8] += h * ux * F
        return (torch.from_numpy(inv).to(f.device) @ m.reshape(L.Q, -1)).reshape(L.Q, *n)
    out = torch.empty_like(f)
    if coll == "BGK":
        for q in range(L.Q):
            out[q] = f[q] - (f[q] - _feq(L, q, rho, ux, uy, uz)) / tau_e
        return out
    # TRT, magic parameter 1/4
    ws = 1.0 / tau_e
    wa = 1.0 / (0.5 + 0.25 / torch.clamp(tau_e - 0.5, min=1e-4)) if les else 1.0 / _tau_a(tau)
    for q in range(L.Q):
        o = L.opp[q]
        d, e = f[q] - _feq(L, q, rho, ux, uy, uz), f[o] - _feq(L, o, rho, ux, uy, uz)
        out[q] = f[q] - ws * 0.5 * (d + e) - wa * 0.5 * (d - e)
    return out


class _Plain:
    """A flow in 64 bits: collide, stream, curved links, open boundaries."""

    def __init__(self, L, shape, tau, coll, les, per_y=True, per_z=True, periodic=False):
        self.L, self.shape, self.tau, self.coll, self.les = L, shape, tau, coll, les
        self.per_y, self.per_z, self.periodic = per_y, per_z, periodic
        self.cells = torch.zeros(shape, dtype=torch.uint8, device=L.dev)
        self.uw = (0.0, 0.0)
        self.inlet = self.outlet = self.thermal = None
        self.turb = None
        self.links = None
        self.n = 0

    def start(self, rho, ux, uy, uz):
        L, sh, dev = self.L, self.shape, self.L.dev
        v = [torch.as_tensor(a, dtype=torch.float64, device=dev).expand(sh) if np.isscalar(a) else
             torch.as_tensor(np.asarray(a), device=dev).double().reshape(sh) for a in (rho, ux, uy, uz)]
        self.f = torch.stack([_feq(L, q, *v) for q in range(L.Q)])

    def walls(self):
        """Masks of the pull sources that reflect, from the cell types."""
        L, c = self.L, self.cells
        nz, ny, nx = self.shape
        self.solid = c == 1
        self.bounce, self.moving = [], []
        for q in range(L.Q):
            cx, cy, cz = L.c[q]
            t = torch.roll(c, (cz, cy, cx), (0, 1, 2))
            b, m = (t == 1) | (t == 6), t == 6
            if cy and not self.per_y:
                b[:, 0 if cy > 0 else ny - 1] = True
                m[:, 0 if cy > 0 else ny - 1] = False
            if cz and not self.per_z:
                b[0 if cz > 0 else nz - 1] = True
                m[0 if cz > 0 else nz - 1] = False
            self.bounce.append(b)
            self.moving.append(m if bool(m.any()) else None)
        y0, y1 = (0, ny) if self.per_y else (1, ny - 1)
        z0, z1 = (0, nz) if (self.per_z or nz == 1) else (1, nz - 1)
        self.rows = (slice(z0, z1), slice(y0, y1))
        self.prev = self.f[:, :, :, -1].clone()

    def curved(self, cx, cy, cz, R):
        """Curved-wall links to a sphere: node, direction and wall fraction."""
        L = self.L
        nz, ny, nx = self.shape
        fluid = self.cells == 0
        n_, q_, d_, u_ = [], [], [], []
        for q in range(1, L.Q):
            c = L.c[q]
            hit = fluid & (torch.roll(self.cells, (-c[2], -c[1], -c[0]), (0, 1, 2)) == 1)
            z, y, x = torch.nonzero(hit, as_tuple=True)
            p = (x.double() - cx, y.double() - cy, z.double() - cz)
            a = float(sum(v * v for v in c))
            b = 2 * sum(pi * ci for pi, ci in zip(p, c))
            k = sum(pi * pi for pi in p) - R * R
            disc = b * b - 4 * a * k
            r = torch.sqrt(torch.clamp(disc, min=0))
            t1, t2 = (-b - r) / (2 * a), (-b + r) / (2 * a)
            d = torch.where((t2 >= 0) & (t2 <= 1), t2, torch.full_like(t2, 0.5))
            d = torch.where((t1 >= 0) & (t1 <= 1), t1, d)
            d = torch.where(disc >= 0, d, torch.full_like(d, 0.5)).clamp(0.01, 0.99)
            n_.append((z * ny + y) * nx + x)
            u_.append((((z - c[2]) % nz) * ny + (y - c[1]) % ny) * nx + (x - c[0]) % nx)
            q_.append(torch.full_like(x, q))
            d_.append(d)
        node, q, up, self.delta = torch.cat(n_), torch.cat(q_), torch.cat(u_), torch.cat(d_)
        N = nx * ny * nz
        opp = torch.tensor(L.opp, device=node.device)[q]
        self.links = (q * N + node, q * N + up, opp * N + node)

    def _inlet(self, S):
        L = self.L
        zs, ys = self.rows
        nz, ny, nx = self.shape
        f = S[:, zs, ys, 0]
        u = self.inlet
        if u == "profile":
            y = torch.arange(ny, dtype=torch.float64, device=L.dev)[ys] - 0.5
            H = ny - 2
            u = 4 * self.umax * y * (H - y) / (H * H)
        if self.turb:
            z, y = np.meshgrid(np.arange(nz)[zs], np.arange(ny)[ys], indexing="ij")
            node = ((z * ny + y) * nx).astype(np.uint64)
            noise = _uniform(self.turb[1], node + np.uint64(self.n * nx * ny * nz))
            u = u * (1 + self.turb[0] * torch.from_numpy(noise).to(L.dev))
        if L.Q == 9:
            rho = (f[0] + f[2] + f[4] + 2 * (f[3] + f[6] + f[7])) / (1 - u)
            a, b, d = (f[3] + 2 / 3 * rho * u, f[7] - 0.5 * (f[2] - f[4]) + rho * u / 6,
                       f[6] + 0.5 * (f[2] - f[4]) + rho * u / 6)
            f[1], f[5], f[8] = a, b, d
            return
        c = L.c
        s0 = sum(f[q] for q in range(L.Q) if c[q][0] == 0)
        sm = sum(f[q] for q in range(L.Q) if c[q][0] < 0)
        rho = (s0 + 2 * sm) / (1 - u)
        plus = [q for q in range(L.Q) if c[q][0] > 0]
        N = [sum(c[q][k] * f[q] for q in range(L.Q) if c[q][0] == 0) / sum(c[q][k] ** 2 for q in plus) for k in (1, 2)]
        h = [f[q] for q in range(L.Q)]
        for q in plus:
            h[q] = f[L.opp[q]] + 6 * L.w[q] * rho * u - (c[q][1] * N[0] + c[q][2] * N[1])
        zero = torch.zeros_like(rho)
        u = zero + u
        eq = [_feq(L, q, rho, u, zero, zero) for q in range(L.Q)]
        P = {}
        for a in range(3):
            for b in range(a, 3):
                P[a, b] = sum(c[q][a] * c[q][b] * (h[q] - eq[q]) for q in range(L.Q))
        tr = (P[0, 0] + P[1, 1] + P[2, 2]) / 3
        for q in range(L.Q):
            t = -tr
            for (a, b), p in P.items():
                k = c[q][a] * c[q][b] * (1 if a == b else 2)
                if k:
                    t = t + k * p
            f[q] = eq[q] + 4.5 * L.w[q] * t

    def _outlet(self, S):
        zs, ys = self.rows
        kind, v = self.outlet
        if kind == "pressure":
            f = S[:, zs, ys, -1]
            u = -1 + (f[0] + f[2] + f[4] + 2 * (f[1] + f[5] + f[8])) / v
            a, b, d = (f[1] - 2 / 3 * v * u, f[8] - 0.5 * (f[2] - f[4]) - v * u / 6,
                       f[5] + 0.5 * (f[2] - f[4]) - v * u / 6)
            f[3], f[6], f[7] = a, b, d
            return
        new = (self.prev[:, zs, ys] + v * S[:, zs, ys, -2]) / (1 + v)
        S[:, zs, ys, -1] = new
        self.prev[:, zs, ys] = new

    def step(self):
        L = self.L
        self.n += 1
        gy = None
        if self.thermal:
            gy = self.thermal["gb"] * (self.g.sum(0) - 0.5)
        A = _collide(L, self.f, self.coll, self.tau, self.les, gy)
        if not self.periodic:
            A = torch.where(self.solid, self.f, A)
        S = torch.empty_like(A)
        for q in range(L.Q):
            cx, cy, cz = L.c[q]
            r = torch.roll(A[q], (cz, cy, cx), (0, 1, 2))
            if not self.periodic:
                back = A[L.opp[q]]
                if self.moving[q] is not None:
                    back = back + self.moving[q] * (6 * L.w[q] * (cx * self.uw[0] + cz * self.uw[1]))
                r = torch.where(self.solid, A[q], torch.where(self.bounce[q], back, r))
            S[q] = r
        if self.links is not None:
            here, up, opp = self.links
            fa, d = A.view(-1), self.delta
            near = 2 * d * fa[here] + (1 - 2 * d) * fa[up]
            far = fa[here] / (2 * d) + (1 - 1 / (2 * d)) * fa[opp]
            S.view(-1)[opp] = torch.where(d < 0.5, near, far)
        if self.inlet is not None:
            self._inlet(S)
        if self.outlet is not None:
            self._outlet(S)
        if self.thermal:
            self._step_g(A, gy)
        self.f = S

    def _step_g(self, A, gy):
        t, f, g = self.thermal, self.f, self.g
        T, rho = g.sum(0), f.sum(0)
        ux = _signed(self.L, f, lambda x, y, z: x) / rho
        uy = _signed(self.L, f, lambda x, y, z: y) / rho + 0.5 * gy
        c5, o5, w5 = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1)], [0, 3, 4, 1, 2], [1 / 3] + [1 / 6] * 4
        G = torch.stack([g[q] - (g[q] - w5[q] * T * (1 + 3 * (c5[q][0] * ux + c5[q][1] * uy))) / t["tau"]
                         for q in range(5)])
        G = torch.where(self.solid, g, G)
        new = torch.empty_like(G)
        for q in range(5):
            sh = (c5[q][1], c5[q][0])
            tw = torch.roll(t["wall"], sh, (1, 2))
            back = torch.where(torch.isnan(tw), G[o5[q]], 2 * w5[q] * torch.nan_to_num(tw) - G[o5[q]])
            r = torch.where(torch.roll(self.solid, sh, (1, 2)), back, torch.roll(G[q], sh, (1, 2)))
            new[q] = torch.where(self.solid, G[q], r)
        self.g = new

    def probe(self, cx, cy, cz, rmax):
        """Links of the force sums: per direction the nodes and midpoint offsets."""
        nz, ny, nx = self.shape
        out = []
        for q in range(1, self.L.Q):
            c = self.L.c[q]
            t = torch.roll(self.cells, (-c[2], -c[1], -c[0]), (0, 1, 2))
            hit = (self.cells == 0) & ((t == 1) | (t == 6))
            if c[1] and not self.per_y:
                hit[:, ny - 1 if c[1] > 0 else 0] = False
            if c[2] and not self.per_z and nz > 1:
                hit[nz - 1 if c[2] > 0 else 0] = False
            z, y, x = torch.nonzero(hit, as_tuple=True)
            r = [v.double() + 0.5 * k - m for v, k, m in zip((x, y, z), c, (cx, cy, cz))]
            if rmax > 0:
                far = r[0] ** 2 + r[1] ** 2 + (r[2] ** 2 if self.L.Q > 9 else 0)
                keep = far <= rmax * rmax
                z, y, x, r = z[keep], y[keep], x[keep], [v[keep] for v in r]
            out.append((q, c, (z * ny + y) * nx + x, r))
        self.sums = out

    def force(self):
        F = torch.zeros(3, dtype=torch.float64, device=self.f.device)
        for q, c, n, r in self.sums:
            v = 2 * self.f[q].reshape(-1)[n]
            s = v.sum()
            if c[0]:
                F[0] += c[0] * s
            if c[1]:
                F[1] += c[1] * s
            if self.L.Q == 9:
                F[2] += (v * (r[0] * c[1] - r[1] * c[0])).sum()
            elif c[2]:
                F[2] += c[2] * s
        return F

    def moments(self):
        L, f = self.L, self.f
        rho = f.sum(0)
        u = [_signed(L, f, lambda *c: c[k]) / rho for k in range(2 if L.Q == 9 else 3)]
        if self.thermal:
            u[1] = u[1] + 0.5 * self.thermal["gb"] * (self.g.sum(0) - 0.5)
        return [rho] + u


def _uniform(seed, counter):
    """Seeded uniform numbers in [-1, 1): splitmix64 of seed ^ counter, 24 bits."""
    with np.errstate(over="ignore"):
        x = (np.uint64(seed) ^ counter) + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        x = x ^ (x >> np.uint64(31))
    return 2.0 * ((x >> np.uint64(40)).astype(np.float64) / (1 << 24)) - 1.0


def _ball(shape, centre, radii=None, R=None):
    """Cells inside a ball or ellipsoid, by the float32 test of the setters."""
    nz, ny, nx = shape
    f = np.float32
    dz, dy, dx = np.meshgrid(np.arange(nz, dtype=f) - f(centre[2]), np.arange(ny, dtype=f) - f(centre[1]),
                             np.arange(nx, dtype=f) - f(centre[0]), indexing="ij", sparse=True)
    if radii is None:
        return (dx * dx + dy * dy) + dz * dz <= f(R) * f(R)
    i = [f(1) / (f(r) * f(r)) for r in radii]
    return (dx * dx * i[0] + dy * dy * i[1]) + dz * dz * i[2] <= f(1)


def _section(shape, s):
    """Cells of the NACA 0012 section, by the float32 test of the setter."""
    nz, ny, nx = shape
    f = np.float32
    a = -f(s["aoa"]) * (f(math.pi) / f(180))
    ca, sa = np.cos(f(-a)), np.sin(f(-a))
    dx = (np.arange(nx, dtype=f) - f(s["lx"]))[None, :]
    dy = (np.arange(ny, dtype=f) - f(s["ly"]))[:, None]
    xc, yc = dx * ca - dy * sa, dx * sa + dy * ca
    inside = (xc >= 0) & (xc <= f(s["chord"]))
    x = np.where(inside, xc, f(0)) / f(s["chord"])
    yt = f(5) * f(0.12) * (f(0.2969) * np.sqrt(x) - f(0.1260) * x - f(0.3516) * x * x + f(0.2843) * x * x * x
                           - f(0.1036) * x * x * x * x) * f(s["chord"])
    return np.broadcast_to(inside & (np.abs(yc) <= yt), shape)


def _plain_flow(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    L = _Lat(case["lattice"], dev)
    nx, ny, nz, scene = case["nx"], case["ny"], case["nz"], case["scene"]
    shape = (nz, ny, nx)
    s = _scene(case, seed)
    open3 = scene in ("sphere", "ellipsoid", "wing")
    P = _Plain(L, shape, s["tau"], case["collision"], case["les"], per_y=open3 and scene != "wing", per_z=open3,
               periodic=scene == "vortex")
    mark = np.zeros(shape, np.uint8)
    if scene == "vortex":
        P.start(*_modes(case, seed))
        return P, s
    if scene == "cylinder":
        P.start(1.0, np.broadcast_to(_profile(ny, s["u"]).astype(np.float32)[None, :, None], shape).copy(), 0.0, 0.0)
        mark[:, 0] = mark[:, -1] = 1
        mark[_ball(shape, (s["cx"], s["cy"], 0.0), R=s["D"] / 2)] = 1
        P.inlet, P.umax, P.outlet = "profile", s["u"], ("pressure", 1.0)
    elif scene == "lid":
        b = s["box"]
        P.start(1.0, 0.0, 0.0, 0.0)
        mark[:, :, 0] = mark[:, :, -1] = 1
        if nz == 1:
            mark[:, ny // 3:ny // 3 + ny // 8 + 1, b:b + nx // 8 + 1] = 1
            mark[:, -1] = 6
        else:
            mark[nz // 3:nz // 3 + nz // 8 + 1, ny // 3:ny // 3 + ny // 8 + 1, b:b + nx // 8 + 1] = 1
            mark[:, -1] = 6
        P.uw = (s["uw"], 0.0)
    elif scene == "cavity":
        P.start(1.0, 0.0, 0.0, 0.0)
        mark[:, 0] = mark[:, -1] = 1
        mark[:, :, 0] = mark[:, :, -1] = 1
        wall = torch.full(shape, float("nan"), dtype=torch.float64, device=dev)
        wall[:, :, 0], wall[:, :, -1] = s["dt"], 0.0
        P.thermal = dict(tau=_f(s["tau"] + 0.1), gb=_f(0.01 / (nx - 2)), wall=wall)
        T = torch.from_numpy(_temperature(case, s)).to(dev).double().reshape(shape)
        P.g = torch.stack([w * T for w in [1 / 3] + [1 / 6] * 4])
    else:
        if scene == "wing":
            P.start(*_disturbed(case, seed, s["u"]))
        else:
            P.start(1.0, s["u"], 0.0, 0.0)
        P.inlet, P.outlet = s["u"], ("convective", s["u"])
        if scene != "ellipsoid":
            P.turb = (_f(0.01), s["seed"])
        if scene == "sphere":
            mark[_ball(shape, (s["cx"], s["cy"], s["cz"]), R=s["R"])] = 1
        elif scene == "ellipsoid":
            mark[_ball(shape, (s["cx"], s["cy"], s["cz"]), radii=s["axes"])] = 1
        else:
            mark[_section(shape, s)] = 1
    P.cells = torch.from_numpy(mark).to(dev)
    P.walls()
    if scene == "sphere":
        P.curved(s["cx"], s["cy"], s["cz"], s["R"])
    return P, s


def _flat(v):
    return v.reshape(-1).cpu()


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        P, s = _plain_flow(case, seed)
        out, F = {}, []
        if case["forces"]:
            P.probe(*_probe(case, s))
            F.append(P.force())  # the state that the history starts from
        for _ in range(case["steps"]):
            P.step()
            if case["forces"]:
                F.append(P.force())
        if case["forces"]:
            out["forces"] = torch.stack(F).cpu()
        out["fields"] = [] if case["nz"] == 256 else [_flat(v) for v in P.moments()]
        if P.thermal:
            out["fields"].append(_flat(P.g.sum(0)))
        return out
    if kind == "batch":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        L, forces, ux, uy = _Lat(9, dev), [], [], []
        for nx, ny, tau, cx, cy, D in _wakes(case, seed):
            shape = (1, ny, nx)
            P = _Plain(L, shape, tau, "MRT", True, per_y=False, per_z=False)
            P.start(1.0, np.broadcast_to(_profile(ny, 0.05).astype(np.float32)[None, :, None], shape).copy(), 0.0, 0.0)
            mark = np.zeros(shape, np.uint8)
            mark[:, 0] = mark[:, -1] = 1
            mark[_ball(shape, (cx, cy, 0.0), R=D / 2)] = 1
            P.cells = torch.from_numpy(mark).to(dev)
            P.inlet, P.umax, P.outlet = "profile", _f(0.05), ("pressure", 1.0)
            P.walls()
            P.probe(cx, cy, 0.0, _f(1.5 * D))
            F = []
            for _ in range(case["steps"]):
                P.step()
                F.append(P.force())
            forces.append(torch.stack(F).cpu())
            m = P.moments()
            ux.append(_flat(m[1]))
            uy.append(_flat(m[2]))
        return {"forces": torch.stack(forces), "ux": torch.cat(ux), "uy": torch.cat(uy)}
    if kind in ("fields", "restart"):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        P = _Plain(_Lat(case["lattice"], dev), (case["nz"], case["ny"], case["nx"]), _f(case["tau"]),
                   case["collision"], case["les"], periodic=True)
        P.start(*_modes(case, seed))
        for _ in range(case["steps"]):
            P.step()
        rho, ux, uy, uz = P.moments()
        if kind == "restart":
            return {"populations": P.f.reshape(P.L.Q, -1).cpu(), "fields": [_flat(v) for v in (rho, ux, uy, uz)]}
        d = [[0.5 * (torch.roll(u, -1, k) - torch.roll(u, 1, k)) for k in (2, 1, 0)] for u in (ux, uy, uz)]
        wx, wy, wz = d[2][1] - d[1][2], d[0][2] - d[2][0], d[1][0] - d[0][1]
        strain = sum(d[k][k] ** 2 for k in range(3)) + 0.5 * (
            (d[0][1] + d[1][0]) ** 2 + (d[1][2] + d[2][1]) ** 2 + (d[0][2] + d[2][0]) ** 2)
        q = 0.5 * (0.5 * (wx * wx + wy * wy + wz * wz) - strain)
        sp = ux * ux + uy * uy + uz * uz
        return {"features": [_flat(v) for v in (wx, wy, wz, q)], "mass": float(rho.sum()),
                "energy": float((0.5 * rho * sp).sum()), "speed": float(sp.max().sqrt())}
    f, cells = _host_arrays(case, seed)
    shape = (case["nz"], case["ny"], case["nx"])
    P = _Plain(_Lat(19, "cpu"), shape, _f(case["tau"]), case["collision"], False, per_y=False, per_z=False)
    P.f = torch.from_numpy(f).double().reshape(19, *shape)
    P.cells = torch.from_numpy(cells).reshape(shape)
    P.walls()
    P.step()
    m = P.moments()
    speed = (m[1] ** 2 + m[2] ** 2 + m[3] ** 2).sqrt()
    return {"populations": P.f.reshape(19, -1), "fields": [_flat(v) for v in m + [speed]]}
