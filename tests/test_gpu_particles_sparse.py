"""GPU: the nearest-particle search where its forms meet -- grids smaller than the search windows,
cubes wider than the or-ed rows (r > 4) and than a window (r > 15), cubes that wrap onto themselves,
crowded cells -- against the oracle's linked lists.  Cell counts are integers and match exactly; the
density matches to 1 ulp (the normalising sum's order)."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("ng,npart,clump", [(2, 1, 0), (3, 2, 0), (7, 3, 0), (9, 40, 0), (34, 2, 0), (33, 60, 0),
                                            (37, 5000, 1), (64, 30000, 1), (101, 20001, 0)])
def test_search_matches_oracle(ctx, ng, npart, clump):
    print("case particle search ng=%d np=%d" % (ng, npart), flush=True)
    rng = np.random.default_rng(ng + npart)
    x = rng.random((npart, 3))
    if clump:  # most particles in a corner, across the periodic edge
        m = (9 * npart) // 10
        x[:m] = (0.97 + 0.08 * x[:m]) % 1.0
    xp = (x * 2 * ng).astype(np.float32)
    den_o, wp_o = R.or_particle_density(xp, ng, 2.0 * ng)
    den = torch.zeros(ng ** 3, dtype=torch.float32, device="cuda")
    wp = torch.zeros(npart, dtype=torch.int32, device="cuda")
    for _ in range(2):
        ctx.particle_density(torch.from_numpy(xp).cuda(), ng, 2.0 * ng, den, wp)
        assert np.array_equal(wp.cpu().numpy(), wp_o)
        assert np.allclose(den.cpu().numpy(), den_o.ravel(), rtol=1.2e-7, atol=0)


@pytest.mark.parametrize("ng,npart", [(6, 3), (20, 60), (33, 900)])
def test_particles_without_a_position_attract_no_cell(ctx, ng, npart):
    """A particle of NaN coordinates lies in the first cell and is at no distance from any other: the empty
    cells around it find theirs in wider cubes, as without it."""
    print("case particle search with NaN ng=%d np=%d" % (ng, npart), flush=True)
    rng = np.random.default_rng(ng)
    x = (1.0 + rng.random((npart, 3)) * (ng - 1)).astype(np.float32)  # none in the first cell's planes
    _, wp_o = R.or_particle_density(x, ng, float(ng))
    # the first cell's own particle without the NaN one: nearest in the smallest cube that holds any
    cell = np.floor(x).astype(int)
    d = np.minimum(np.abs(x - np.float32(0.5)), ng - np.abs(x - np.float32(0.5)))
    cube = np.minimum(cell, ng - cell).max(1)
    first = cube == cube.min()
    p0 = np.flatnonzero(first)[np.argmin((d[first].astype(np.float64) ** 2).sum(1))]
    wp_o = wp_o.copy()
    wp_o[p0] -= 1
    xn = np.concatenate([x, np.full((1, 3), np.nan, np.float32)])
    den = torch.zeros(ng ** 3, dtype=torch.float32, device="cuda")
    wp = torch.zeros(npart + 1, dtype=torch.int32, device="cuda")
    ctx.particle_density(torch.from_numpy(xn).cuda(), ng, float(ng), den, wp)
    assert np.array_equal(wp.cpu().numpy(), np.append(wp_o, 1))


@pytest.mark.parametrize("ng,npart,boxes", [(12, 40, 2.0 ** 26), (33, 500, 2.0 ** 25), (33, 500, 2.0 ** 20)])
def test_coordinates_far_outside_the_box(ctx, ng, npart, boxes):
    """Coordinates millions of boxes out, whose modulo in FP32 leaves the box: distances to them are periodic
    all the same.  Counts match exactly."""
    print("case particle search far ng=%d boxes=%g" % (ng, boxes), flush=True)
    rng = np.random.default_rng(ng)
    nf = np.float32(3.7)
    x = rng.random((npart, 3)) * nf
    far = rng.random((npart, 3)) < 0.3
    x[far] += nf * np.round(boxes * rng.standard_normal(int(far.sum())))
    xp = x.astype(np.float32)
    den_o, wp_o = R.or_particle_density(xp, ng, float(nf))
    den = torch.zeros(ng ** 3, dtype=torch.float32, device="cuda")
    wp = torch.zeros(npart, dtype=torch.int32, device="cuda")
    ctx.particle_density(torch.from_numpy(xp).cuda(), ng, float(nf), den, wp)
    assert np.array_equal(wp.cpu().numpy(), wp_o)
    assert np.allclose(den.cpu().numpy(), den_o.ravel(), rtol=1.2e-7, atol=0)


@pytest.mark.parametrize("ng,npart,clump", [(103, 20001, 1), (103, 3000, 0), (130, 300000, 0), (207, 400000, 0)])
def test_workgroups_of_several_chunks(ctx, ng, npart, clump):
    """Grids whose workgroups of the first pass take 2, 4 and 16 chunks of cells (from 2^20 cells on), the last
    of them past the end, with a few cells for the second pass and with most.  As above."""
    print("case particle chunks ng=%d np=%d" % (ng, npart), flush=True)
    test_search_matches_oracle(ctx, ng, npart, clump)
