"""The x and y one-way faces in one launch, on the smallest grids they take,
bit for bit against the CPU oracle: the same operations, so no tolerance."""
import numpy as np
import pytest

from wavefield_imaging_amd import awefd, synth

pytestmark = pytest.mark.gpu


# padded axes of 2 nop + 4 nodes (the faces' shells meet, no line is left
# between the corner patches) and a few more, in x, in y and in both
@pytest.mark.parametrize("fdorder", [2, 4, 8, 12])
@pytest.mark.parametrize("n2,n3", [(4, 4), (4, 9), (11, 4), (5, 6), (40, 33)])
def test_smallest_grids(orc, fdorder, n2, n3):
    rng = np.random.default_rng(100 * fdorder + 10 * n2 + n3)
    n, nb = [17, n2, n3], fdorder // 2
    par = dict(n=n, o=[0.0] * 3, d=[5.0] * 3, nt=25, dt=synth.DT, nb=nb, dabc=True, fdorder=fdorder, expl=False)
    vel = rng.uniform(1.2e8, 3.0e8, n[::-1]).astype(np.float32)
    lo, hi = -5.0 * nb, np.array([n2, n3, n[0]]) * 5.0 + 5.0 * nb - 8.0
    pts = rng.uniform(lo, hi, (200, 3)).astype(np.float32)
    wav = rng.standard_normal((25, 200)).astype(np.float32)
    tr, _, f = awefd.run("cart3d", par, vel, pts, pts, wav)
    ref, uf, _ = orc.run("cart3d", par, vel, pts, pts, wav)
    assert np.any(f)
    np.testing.assert_array_equal(tr, ref)
    np.testing.assert_array_equal(f, uf)
