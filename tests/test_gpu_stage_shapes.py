"""The T, S and final stage kernels at the shapes where a tile or a pipeline can go wrong: sectors
smaller and larger than a tile, odd sizes, chain ends, groups of one and of few key tiles, against
the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from mqdmrg import engine as E
from mqdmrg.workloads import SyntheticSite

pytestmark = pytest.mark.gpu

# FP64: sums of ~1e3 terms of either sign, each rounded to 2^-53.  FP32: each product and partial sum
# rounded to 2^-24.  BF16x3: operands kept to 2^-17 (x = hi + lo).  Errors of different terms add
# like random signs, so the norm of the difference stays near the rounding of one term; the
# factors below are ~100 of it.
RTOL = {E.PREC_F64: 1e-13, E.PREC_F32: 1e-5, E.PREC_BF16X3: 1e-3}

SHAPES = [
    ("heisenberg", 16, 7, 150),   # few keys (one or two key tiles), sectors of 1 to 60
    ("heisenberg", 12, 1, 64),    # left end
    ("hubbard", 12, 5, 301),
    ("hubbard", 10, 7, 90),       # right end
    ("qc", 8, 3, 77),
    ("qc", 10, 1, 60),
    ("qc_su2", 10, 4, 131),
    ("qc_su2", 12, 8, 57),
    ("qc_su2", 14, 6, 101),   # several 128-column panels, runs of odd and even numbers of key tiles
    ("heisenberg", 20, 9, 420),   # sectors of 65 to 144 and of more than 144
    ("heisenberg", 24, 11, 1100),   # and of more than 288
]


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("model,L,site,m", SHAPES)
def test_sigma_stages_match_oracle(eng, model, L, site, m):
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    Lc, Rc = ws.random_cohorts(ws.left_index), ws.random_cohorts(ws.right_index)
    host = [O.HostBoundary(i, [x if x is not None else np.zeros(0) for x in c])
            for i, c in ((ws.left_index, Lc), (ws.right_index, Rc))]
    psi_h = ws.random_psi()
    ref = O.SigmaOracle(ws.site_desc, ws.mpo_desc, *host).apply(psi_h)
    Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(psi_h).to("cuda:0")
    for prec, tol in RTOL.items():
        out = torch.full_like(psi, float("nan"))
        plan.apply(psi, out, precision=prec)
        eng.sync()
        err = np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)
        print("%s L=%d site=%d m=%d precision %d: %.2e" % (model, L, site, m, prec, err), flush=True)
        assert err <= tol
        first = out.clone()
        for _ in range(3):   # captured on the second application, replayed after it
            plan.apply(psi, out, precision=prec)
            eng.sync()
            assert torch.equal(first, out)


@pytest.mark.parametrize("kind", ["left", "right"])
@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 16, 7, 150), ("heisenberg", 12, 1, 64), ("hubbard", 12, 5, 301),
                                            ("qc", 8, 3, 77), ("qc_su2", 10, 4, 131), ("qc_su2", 12, 8, 57)])
def test_steps_match_oracle(eng, kind, model, L, site, m):
    """Boundary steps over one site: sectors below and above one 64-row / 64-column tile, odd sizes."""
    from mqdmrg.engine import MpoDesc, SiteDesc
    from mqdmrg import mps
    from mqdmrg.symmetry import SiteLayout
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    k = site if kind == "left" else site + 1
    index = ws.left_index if kind == "left" else ws.right_index
    lay = SiteLayout(ws.bonds[k], ws.basis.phys, ws.bonds[k + 1])
    sd, md = SiteDesc(ws.basis.sym, ws.bonds[k], ws.basis.phys, ws.bonds[k + 1]), MpoDesc(ws.mpo[k])
    coh = ws.random_cohorts(index)
    hb = O.HostBoundary(index, [x if x is not None else np.zeros(0) for x in coh])
    bra, ket = mps.random_site_vector(lay, ws.rng), mps.random_site_vector(lay, ws.rng)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")  # noqa: E731
    b = E.DeviceBoundary.upload(eng, index, coh)
    if kind == "left":
        ref = O.left_step(sd, md, mps.rp_to_lp(lay, bra), ket, hb, True)
        new = E.left_step(eng, sd, md, d(mps.rp_to_lp(lay, bra)), d(ket), b)
    else:
        ref = O.right_step(sd, md, bra, ket, hb, True)
        new = E.right_step(eng, sd, md, d(bra), d(ket), b)
    num = den = 0.0
    for x, y in zip(new.download(), ref.cohorts):
        if len(y):
            num += float(np.sum((x - y) ** 2))
            den += float(np.sum(y ** 2))
    print("%s %s L=%d site=%d m=%d: %.2e" % (kind, model, L, site, m, np.sqrt(num / den)), flush=True)
    assert np.sqrt(num / den) <= RTOL[E.PREC_F64]


@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 16, 7, 150), ("hubbard", 10, 7, 90), ("qc", 6, 2, 40),
                                            ("qc_su2", 6, 2, 60)])
def test_adjoint_matches_oracle(eng, model, L, site, m):
    """Gradients per MPO term: terms of one entry and of thousands (64 entries a turn), groups of very
    different sizes side by side, and a second gradient through the same plan."""
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    Lc, Rc = ws.random_cohorts(ws.left_index), ws.random_cohorts(ws.right_index)
    host = [O.HostBoundary(i, [x if x is not None else np.zeros(0) for x in c])
            for i, c in ((ws.left_index, Lc), (ws.right_index, Rc))]
    Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb, algorithm=E.SIGMA_GROUPED, adjoint=True)
    for _ in range(2):
        psi_h = ws.random_psi()
        ref = O.sigma_term_gradient(ws.site_desc, ws.mpo_desc, *host, psi_h)
        g = plan.adjoint(torch.from_numpy(psi_h).to("cuda:0"))
        err = np.linalg.norm(g - ref) / np.linalg.norm(ref)
        print("adjoint %s L=%d site=%d m=%d: %.2e" % (model, L, site, m, err), flush=True)
        assert err <= 10 * RTOL[E.PREC_F64]   # two products in a row and the sum over a term's entries
