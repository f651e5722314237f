"""GPU tests of the adaptive integrator's batched levels: every patch order, ragged numbers of
targets per patch, off-surface targets and deep trees against the CPU oracle (same weights to
rounding, same refinement counts), and pairs that take another pass because the slot pool is
used up or by a level cap against the run where none does (same bits)."""
import numpy as np
import pytest

from fmm3dbie_amd.layer import SELF_NR, SELF_NT, SELF_TAU
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _targets(g, n, seed):
    """n targets off a surface: most within its near field, some on top of it (trees that go
    several levels below the batched ones)."""
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


# Slots in all: those of one pair (one pair at a time in the last passes), part of the root level's, and
# all but a few of what the pairs need
@pytest.mark.parametrize("helm,norder,slots", [(True, 3, 21), (True, 4, 100), (False, 6, 700), (True, 6, 100),
                                               (False, 2, 450)])
def test_pairs_without_a_slot_take_another_pass(cuda, helm, norder, slots):
    import torch
    from fmm3dbie_amd import geometry as G, layer, problem, selector as S
    g = G.get_sphere_npat(1.0, 1, (0, 0, 0), norder)
    pars = np.array([2.0, 2.0j, 1.0]) if helm else np.array([1.0, 0.5])
    P = problem.setup(g, 1e-6, helm, pars)
    nq = layer.NearQuadDevice(g, helm, pars, 1e-6, P["row_ptr"], P["col_ind"], P["iquad"], P["rfac0"], device=cuda)
    w0 = nq.run(want_detail=True).cpu().numpy().copy()
    st0 = nq.stats
    assert st0["nnoslot"] == 0
    nref0, lev0, unc0 = st0["nref"].copy(), st0["lev"].copy(), st0["unc"].copy()

    def check(st):
        assert 0 < st["nnoslot"] + st["nfallback"] <= st0["nadap"]
        assert np.array_equal(st["nref"], nref0) and np.array_equal(st["lev"], lev0)
        assert np.array_equal(st["unc"], unc0)

    for rep in range(2):  # (which pairs find a slot differs from run to run)
        assert np.array_equal(nq.run(want_detail=True, max_slots=slots).cpu().numpy(), w0)
        check(nq.stats)
        assert nq.stats["nfallback"] == 0
    # with a selector: the plain class with a level cap (a list of its own for the pairs sent back),
    # and another class whose pairs all go back at a cap of 1 or for want of a slot, joined with
    # the plain class's
    plain = torch.as_tensor(S.forced(S.PLAIN_CLASS), device=cuda)
    w = nq.run(want_detail=True, selector=plain, route_lmax=[2] * 6, max_slots=slots).cpu().numpy()
    assert np.array_equal(w, w0)
    check(nq.stats)
    other = torch.as_tensor(S.forced(4), device=cuda)
    ad = st0["cls"] == 1
    for caps in ([1] * 6, [20] * 6, [20, 20, 20, 20, 1, 20]):
        w = nq.run(want_detail=True, selector=other, route_lmax=caps, max_slots=slots).cpu().numpy()
        assert caps[4] == 20 or nq.stats["nfallback"] > 0
        for j in np.nonzero(ad)[0]:
            a, b = P["iquad"][j] - 1, P["iquad"][j + 1] - 1
            # both rules are within the integrator's own tolerance of 1e-5
            assert np.abs(w[a:b] - w0[a:b]).max() < 2e-5 * np.abs(w0[a:b]).max()
