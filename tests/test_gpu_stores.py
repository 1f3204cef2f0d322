"""Population stores kept in the caches or past them (by the bytes that share
the last-level cache) give the same bits: a domain whose two buffers fit the
cache, stepped alone (kept) and in a batch with a member that makes the batch
too large for it (past)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,storage,shape", [(19, 0, (96, 80, 65)), (19, 1, (131, 80, 96)), (27, 2, (96, 96, 97)),
                                                   (27, 0, (64, 64, 64))])
def test_kept_and_passing_stores_agree(lattice, storage, shape):
    import wake_amd as wa

    if wa._lib.lib().wake_hip_device_count() <= 0:
        pytest.fail("no GPU visible to the HIP runtime")
    elem = 4 if storage == 0 else 2
    nx, ny, nz = shape
    both = 2 * lattice * elem * nx * ny * nz
    assert (48 << 20) <= both <= (240 << 20)

    def grid(n, pad=-1):
        g = wa.LatticeGrid3D(*n, 0.55, lattice=lattice, storage=storage, plane_pad=pad)
        g.set_periodic_axes(True, True)
        g.initialize(1.0, 0.05, 0.0, 0.0)
        g.set_les_coupled(True)
        g.set_inflow_west(0.05, 0.0)
        g.set_inflow_turbulence(0.02, 3)
        g.set_convective_outflow_east(0.05)
        g.set_solid_sphere(n[0] / 3.0, n[1] / 2.0, n[2] / 2.0, 9.0)
        g.build_curved_sphere_links(n[0] / 3.0, n[1] / 2.0, n[2] / 2.0, 9.0)
        return g

    pad = (260 << 20) // (2 * lattice * elem) // 256 * 256
    ends = []
    for g in (grid(shape), grid(shape, pad)):
        g.run(12, "TRT", use_les=True, smag=0.17)
        ends.append(g.f_src_data().copy())
    assert np.array_equal(*ends)
    ends = []
    for others in ([], [grid((256, 160, 128))]):
        b = wa.Batch(lattice=lattice, storage=storage, collision="TRT", use_les=True, chunk=12)
        g = grid(shape)
        for m in [g] + others:
            b.add(m, 12, smag=0.17)
        b.run(12)
        ends.append(g.f_src_data().copy())
    assert np.array_equal(*ends)
