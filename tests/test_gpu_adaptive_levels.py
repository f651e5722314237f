"""GPU tests of the adaptive integrator's batched levels: every patch order, ragged numbers of
targets per patch, off-surface targets, deep trees, and pairs sent back to another pass,
against the CPU oracle (same weights to rounding, same refinement counts)."""
import numpy as np
import pytest

from fmm3dbie_amd.layer import SELF_NR, SELF_NT, SELF_TAU
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _targets(g, n, seed):
    """n targets off a surface: most within its near field, some on top of it (trees that go
    several levels below the batched ones), one patch's neighbourhood with none."""
    rng = np.random.default_rng(seed)
    x = g["srcvals"][rng.integers(0, len(g["srcvals"]), n)]
    dist = np.where(np.arange(n) % 4 == 0, 1e-3, rng.uniform(0.02, 0.5, n))
    return np.ascontiguousarray(x[:, :3] + (dist * rng.choice([-1.0, 1.0], n))[:, None] * x[:, 9:12])


# orders 1..9 in both kernels (order 9: the largest LDS of a tile); 1, 15, 16, 17 targets and
# enough for several tiles of a patch
CASES = [(True, 1, 40), (False, 2, 17), (True, 3, 16), (False, 4, 15), (True, 5, 33), (False, 6, 1), (True, 7, 40),
         (True, 8, 25), (False, 8, 40), (True, 9, 30), (False, 9, 5), (True, 4, 400)]


@pytest.mark.parametrize("helm,norder,nt", CASES)
def test_batched_levels_match_oracle(cuda, helm, norder, nt):
    from fmm3dbie_amd import geometry as G, layer, near
    g = G.get_sphere_npat(1.0, 1, (0, 0, 0), norder)
    pars = np.array([2.0, 2.0j, 1.0]) if helm else np.array([1.0, 0.5])
    targs = _targets(g, nt, 7 * norder + nt)
    cms, rads = near.get_centroid_rads(g)
    rfac, rfac0 = near.get_rfacs(norder)
    rp, ci = near.findnear(cms, rads * max(rfac, rfac0), targs)
    iq = near.get_iquad_rsc(g, rp, ci)
    pid = -np.ones(nt, np.int64)
    uvs = np.zeros((nt, 2))
    ref, cls, nref = O.getnearquad(g, targs, pid, uvs, 1e-6, O.HELM_COMB if helm else O.LAP_COMB, pars, rp, ci, iq,
                                   rfac0, O.SELF_POLAR, SELF_NR, SELF_NT, self_tau=SELF_TAU, want_class=True)
    nq = layer.NearQuadDevice(g, helm, pars, 1e-6, rp, ci, iq, rfac0, device=cuda, targets=targs, ipatch_id=pid,
                              uvs_targ=uvs)
    w = nq.run(want_detail=True).cpu().numpy()
    assert np.array_equal(nq.stats["cls"], cls)
    assert np.array_equal(nq.stats["nref"][cls == 1], nref[cls == 1])
    # rounding of sums of the children of children, as the parity tests hold the integrator to
    # (relative to the largest weight; targets 1e-3 off the surface have 10 times its terms)
    assert np.abs(w - ref).max() < 1e-11 * np.abs(ref).max()
    # another run: other places in the tiles, the same bits
    assert np.array_equal(nq.run().cpu().numpy(), w)
