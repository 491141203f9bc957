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
