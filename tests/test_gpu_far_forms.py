"""GPU tests of the far sum's forms: every size of a block of right-hand sides (vector groups,
padded groups, matrix cores), kernel (Laplace, real and complex wavenumber, no double or no
single layer, alpha and beta of any size and phase), precision and near-correction mode,
against one 64-bit sum in plain torch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _over(g, P, sig):
    """sigma_over * w at the oversampled nodes, (nrhs, nptso)."""
    from fmm3dbie_amd import basis
    over = np.zeros((len(sig), len(P["whtsover"])), complex)
    for ip, nv in enumerate(P["novers"]):
        no = int(g["norders"][ip])
        uv, _ = basis.rv_nodes(int(nv))
        im = np.stack([basis.koorn_pols(u, v, no) for u, v in uv]) @ basis.rv_umat(no)
        a, b = P["ixyzso"][ip] - 1, P["ixyzso"][ip + 1] - 1
        over[:, a:b] = sig[:, g["ixyzs"][ip] - 1:g["ixyzs"][ip + 1] - 1] @ im.T
    return over * P["whtsover"]


def _kernel(g, P, helm, pars):
    """Kernel matrix (npts, nptso) over all oversampled sources, and with those of each
    target's near patches zeroed."""
    import torch
    t = torch.as_tensor
    d = t(g["srcvals"][:, None, :3] - P["srcover"][None, :, :3])
    r = d.square().sum(-1).sqrt()
    ri = torch.where(r > 1e-14, 1 / r, torch.zeros_like(r))
    dn = (d * t(P["srcover"][None, :, 9:12])).sum(-1) * ri * ri
    zk, a, b = (pars if helm else (0.0, pars[0], pars[1]))
    zk = complex(zk)
    ker = (a + b * dn * (1 - 1j * zk * r)) * torch.exp(1j * zk * r) * ri / (4 * np.pi)
    patch = np.repeat(np.arange(len(P["novers"])), np.diff(P["ixyzso"]))
    near = np.zeros((len(r), len(P["novers"])), bool)
    rows = np.repeat(np.arange(len(r)), np.diff(P["row_ptr"]))
    near[rows, P["col_ind"] - 1] = True
    return ker, torch.where(t(near[:, patch]), 0, ker)


def _sum64(g, P, helm, pars, sig):
    """All oversampled sources except those of near patches (near weights zero), (nrhs, npts)
    in 64 bits (the add/subtract form is the same sum), and the sums of |K| |s| over those
    sources and over all sources, which bound the rounding of either form."""
    import torch
    over = torch.as_tensor(_over(g, P, sig))
    ker, far = _kernel(g, P, helm, pars)
    size = [(over.abs() @ k.abs().T).numpy() for k in (far, ker)]
    return (over @ far.T).numpy(), size[0], size[1]


# helm, (k, alpha, beta); the sphere's points are ragged: 27 targets of the last wavefront at
# order 3 (12 patches of 10 points), 52 at order 4
CASES = [(False, (0.7, -1.3), 3), (False, (1.0, 0.0), 4), (False, (0.0, 2.0), 3),
         (True, (5.0, 5.0j, 1.0), 4), (True, (2.0, 0.0, 1.0), 3), (True, (3.0, 1.0 - 2.0j, 0.0), 4),
         (True, (1.5, 3e4 + 1e3j, -2e-3 + 1e-3j), 3), (True, (0.0, 1.0 + 0.5j, 1.0j), 3),
         (True, (2.0 + 0.7j, 1.0, 1.0), 4), (True, (-4.0, 1.0, 1.0), 3)]


@pytest.mark.parametrize("helm,pars,norder", CASES)
def test_far_sum_forms_match_a_64_bit_sum(cuda, helm, pars, norder):
    import torch
    from fmm3dbie_amd import geometry as G, layer, problem
    g = G.get_sphere_npat(1.0, 2 if norder == 3 else 1, (0, 0, 0), norder)
    pars = np.array(pars)
    P = problem.setup(g, 1e-6, helm, pars)
    w = np.zeros(P["nquad"], complex if helm else float)
    plan = layer.ApplyPlan(g, helm, pars, P["row_ptr"], P["col_ind"], P["iquad"], w, P["novers"], P["ixyzso"],
                           P["srcover"], P["whtsover"])
    rng = np.random.default_rng(3)
    N = len(g["srcvals"])
    S = rng.standard_normal((33, N)) + 1j * rng.standard_normal((33, N))
    ref, size_far, size_all = _sum64(g, P, helm, pars, S)
    # A kernel value has a relative error of a few roundings (1/r three, its powers, the dipole
    # factor, the phase k r <= 10), a sum of n terms up to sqrt(n) more (n <= 500 here): 30
    # roundings of the sum of |K| |s|, over all sources where the near part is added and
    # subtracted again
    for nrhs in (1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 33):
        s = torch.as_tensor(S[:nrhs], device=cuda)
        s = s[0] if nrhs == 1 else s
        for prec, mode, unit, size in ((64, 1, 2.0 ** -53, size_far), (64, 0, 2.0 ** -53, size_all),
                                       (32, 1, 2.0 ** -24, size_far)):
            sp = s if prec == 64 else s.to(torch.complex64)
            out = np.atleast_2d(plan.apply(sp.contiguous(), prec, mode).cpu().numpy())
            err = np.linalg.norm(out - ref[:nrhs]) / np.linalg.norm(size[:nrhs])
            assert err < 30 * unit, (nrhs, prec, mode, err / unit)
    plan.close()


def _mixed_sphere(na, orders):
    """A sphere whose patches alternate between the orders."""
    from fmm3dbie_amd import geometry as G
    gs = [G.get_sphere_npat(1.0, na, (0, 0, 0), n) for n in orders]
    npat = len(gs[0]["norders"])
    pick = [gs[ip % len(gs)] for ip in range(npat)]
    rows = [slice(q["ixyzs"][ip] - 1, q["ixyzs"][ip + 1] - 1) for ip, q in enumerate(pick)]
    g = dict(gs[0])
    g["norders"] = np.array([q["norders"][ip] for ip, q in enumerate(pick)])
    g["iptype"] = np.array([q["iptype"][ip] for ip, q in enumerate(pick)])
    g["ixyzs"] = np.cumsum([1] + [r.stop - r.start for r in rows])
    for key in ("srcvals", "srccoefs"):
        g[key] = np.concatenate([q[key][r] for q, r in zip(pick, rows)])
    return g


# patches of several orders: the general CSR kernel, the near subtraction as a kernel of its own, the
# reduction over source splits on its own, interpolation matrices by patch
@pytest.mark.parametrize("helm,pars,orders", [(True, (2.0, 2.0j, 1.0), (3, 4)), (False, (1.0, 0.5), (2, 5, 3)),
                                              (True, (2.0 + 0.5j, 1.0, 1.0j), (4, 3))])
def test_patches_of_several_orders(cuda, helm, pars, orders):
    import torch
    from fmm3dbie_amd import layer, problem
    g = _mixed_sphere(2, orders)
    pars = np.array(pars)
    P = problem.setup(g, 1e-6, helm, pars, nover_fixed=5)
    rng = np.random.default_rng(8)
    # (of the size of quadrature weights)
    w = 1e-3 * rng.standard_normal(P["nquad"])
    if helm:
        w = w + 1e-3j * rng.standard_normal(P["nquad"])
    plan = layer.ApplyPlan(g, helm, pars, P["row_ptr"], P["col_ind"], P["iquad"], w, P["novers"], P["ixyzso"],
                           P["srcover"], P["whtsover"])
    assert plan.info()[3] == 0  # no uniform patch size
    N = len(g["srcvals"])
    S = rng.standard_normal((17, N)) + 1j * rng.standard_normal((17, N))
    ref, size_far, size_all = _sum64(g, P, helm, pars, S)
    near, size_near = np.zeros_like(ref), np.zeros(ref.shape)
    for i in range(N):
        for j in range(P["row_ptr"][i] - 1, P["row_ptr"][i + 1] - 1):
            ip = P["col_ind"][j] - 1
            wj = w[P["iquad"][j] - 1:P["iquad"][j + 1] - 1]
            sj = S[:, g["ixyzs"][ip] - 1:g["ixyzs"][ip + 1] - 1]
            near[:, i] += sj @ wj
            size_near[:, i] += np.abs(sj) @ np.abs(wj)
    ref = ref + near
    for nrhs in (1, 3, 8, 17):
        s = torch.as_tensor(S[:nrhs], device=cuda)
        s = s[0] if nrhs == 1 else s
        for prec, mode, unit, size in ((64, 1, 2.0 ** -53, size_far), (64, 0, 2.0 ** -53, size_all),
                                       (32, 1, 2.0 ** -24, size_far)):
            sp = s if prec == 64 else s.to(torch.complex64)
            out = np.atleast_2d(plan.apply(sp.contiguous(), prec, mode).cpu().numpy())
            err = np.linalg.norm(out - ref[:nrhs]) / np.linalg.norm(size[:nrhs] + size_near[:nrhs])
            assert err < 30 * unit, (nrhs, prec, mode, err / unit)  # the bound above
    plan.close()


# densities far down FP32's range at a long wavelength: the unit in which a plan stores its coordinates
# must not enter the strengths or a product with them (k / (2 pi) is 1.6e-5 here, the strengths 2e-36), nor
# the smallest value of the terms of the split products (strengths of 2e-35 here); and far up
@pytest.mark.parametrize("nrhs,size", [(1, 1e-34), (3, 1e-34), (8, 1e-34), (9, 1e-33), (16, 1e-33), (17, 1e-33),
                                       (33, 1e-33), (64, 1e-33), (16, 1e36), (64, 1e36)])
def test_densities_of_extreme_size_at_a_long_wavelength(cuda, nrhs, size):
    import torch
    from fmm3dbie_amd import geometry as G, layer, problem
    g = G.get_sphere_npat(1.0, 1, (0, 0, 0), 4)
    pars = np.array([1e-4, 1.0, 1.0])
    P = problem.setup(g, 1e-6, True, pars)
    plan = layer.ApplyPlan(g, True, pars, P["row_ptr"], P["col_ind"], P["iquad"], np.zeros(P["nquad"], complex),
                           P["novers"], P["ixyzso"], P["srcover"], P["whtsover"])
    rng = np.random.default_rng(2)
    N = len(g["srcvals"])
    S = rng.standard_normal((nrhs, N)) + 1j * rng.standard_normal((nrhs, N))
    ref, bound, _ = _sum64(g, P, True, pars, S)
    s = torch.as_tensor(size * S, device=cuda).to(torch.complex64)
    out = plan.apply(s[0].contiguous() if nrhs == 1 else s.contiguous(), 32, 1).cpu().numpy()
    out = np.atleast_2d(out).astype(complex) / size
    err = np.linalg.norm(out - ref) / np.linalg.norm(bound)
    assert err < 30 * 2.0 ** -24, err * 2.0 ** 24  # the bound above
    plan.close()


# several groups of 16 in FP32 (split products), at the edges of the groups; the 10-point patches
# leave a ragged last tile of 32 sources
@pytest.mark.parametrize("helm,pars", [(False, (0.7, -1.3)), (True, (5.0, 5.0j, 1.0)), (True, (2.0 + 0.7j, 1.0, 1.0))])
def test_far_sum_split_products_match_a_64_bit_sum(cuda, helm, pars):
    import torch
    from fmm3dbie_amd import geometry as G, layer, problem
    g = G.get_sphere_npat(1.0, 2, (0, 0, 0), 3)
    pars = np.array(pars)
    P = problem.setup(g, 1e-6, helm, pars)
    plan = layer.ApplyPlan(g, helm, pars, P["row_ptr"], P["col_ind"], P["iquad"],
                           np.zeros(P["nquad"], complex if helm else float), P["novers"], P["ixyzso"], P["srcover"],
                           P["whtsover"])
    rng = np.random.default_rng(5)
    N = len(g["srcvals"])
    # (the size of a right-hand side is its own: each is checked by itself, from 1e-20 to 1e12)
    S = (rng.standard_normal((64, N)) + 1j * rng.standard_normal((64, N))) * 10.0 ** (np.arange(64) / 2 - 20)[:, None]
    ref, size, _ = _sum64(g, P, helm, pars, S)
    for nrhs in (18, 32, 34, 48, 50, 64):
        s = torch.as_tensor(S[:nrhs], device=cuda).to(torch.complex64).contiguous()
        out = plan.apply(s, 32, 1).cpu().numpy()
        err = np.linalg.norm(out - ref[:nrhs], axis=1) / np.linalg.norm(size[:nrhs], axis=1)
        assert err.max() < 30 * 2.0 ** -24, (nrhs, err.max() * 2.0 ** 24)  # the bound above
    plan.close()


# The imaginary part of the single layer of a real density is k times the real part's size: the error
# of each part is held to the sum of its own products, which a block's columns have to keep as a
# density on its own does (the complex product is not to be formed from three real ones)
@pytest.mark.parametrize("zk", [0.01, 1.0])
def test_block_of_real_densities_keeps_each_part(cuda, zk):
    import torch
    from fmm3dbie_amd import geometry as G, layer, problem
    g = G.get_sphere_npat(1.0, 1, (0, 0, 0), 4)
    pars = np.array([zk, 1.0, 0.0])
    P = problem.setup(g, 1e-6, True, pars)
    plan = layer.ApplyPlan(g, True, pars, P["row_ptr"], P["col_ind"], P["iquad"], np.zeros(P["nquad"], complex),
                           P["novers"], P["ixyzso"], P["srcover"], P["whtsover"])
    rng = np.random.default_rng(9)
    S = rng.standard_normal((64, len(g["srcvals"]))) + 0j
    over = torch.as_tensor(_over(g, P, S).real)
    ker, far = _kernel(g, P, True, pars)
    for nrhs in (1, 3, 8, 9, 15, 16, 17, 33, 48, 64):
        s = torch.as_tensor(S[:nrhs], device=cuda)
        s = s[0] if nrhs == 1 else s
        for prec, mode, unit, k in ((64, 1, 2.0 ** -53, far), (64, 0, 2.0 ** -53, ker), (32, 1, 2.0 ** -24, far)):
            sp = s if prec == 64 else s.to(torch.complex64)
            out = torch.as_tensor(np.atleast_2d(plan.apply(sp.contiguous(), prec, mode).cpu().numpy()))
            for part in ("real", "imag"):
                ref = over[:nrhs] @ getattr(far, part).T
                size = over[:nrhs].abs() @ getattr(k, part).abs().T
                err = float((getattr(out, part) - ref).norm() / size.norm())
                # 30 roundings, the bound above
                assert err < 30 * unit, (nrhs, prec, mode, part, err / unit)
    plan.close()
