"""Forms of the stage kernels and of the plans around them that the chains' ordinary sites do not
reach: boundaries with cohorts left out, sectors beyond one tile of the step kernel, the adjoint's
products side by side, wide groups, large stages."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import oracle as O
from mqdmrg import engine as E
from mqdmrg.capi import BIndex
from mqdmrg.workloads import SyntheticSite

pytestmark = pytest.mark.gpu

RTOL = {E.PREC_F64: 1e-13, E.PREC_F32: 1e-5, E.PREC_BF16X3: 1e-4}


@pytest.fixture(scope="module")
def eng():
    e = E.Engine(0)
    yield e
    e.close()


def host_boundary(index, cohorts):
    return O.HostBoundary(index, [x if x is not None else np.zeros(0) for x in cohorts])


def check_sigma(eng, ws, left_index, right_index, label):
    """sigma of a site with the given boundary indices against the oracle, in all three precisions."""
    Lc, Rc = ws.random_cohorts(left_index), ws.random_cohorts(right_index)
    psi_h = ws.random_psi()
    ref = O.SigmaOracle(ws.site_desc, ws.mpo_desc, host_boundary(left_index, Lc), host_boundary(right_index, Rc)).apply(psi_h)
    assert np.linalg.norm(ref) > 0
    Lb, Rb = E.DeviceBoundary.upload(eng, left_index, Lc), E.DeviceBoundary.upload(eng, right_index, Rc)
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(psi_h).to("cuda:0")
    for prec, tol in RTOL.items():
        print("%s precision %d" % (label, prec), flush=True)
        out = torch.full_like(psi, float("nan"))
        plan.apply(psi, out, precision=prec)
        eng.sync()
        err = np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)
        print("  relative error %.2e" % err, flush=True)
        assert err <= tol
    plan.close()


def subset(index, keep):
    """The boundary index with only the cohorts `keep`."""
    keep = np.asarray(keep)
    return BIndex(index.bra, index.ket, index.aux_dim, index.bra_pos[keep], index.ket_pos[keep], index.tr[keep],
                  index.n_blocks[keep], index.offsets[keep], index.conj_scales[keep], index.transposes[keep])


@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 26, 12, 8192), ("heisenberg", 20, 9, 420), ("hubbard", 12, 5, 301),
                                            ("qc", 10, 4, 150)])
def test_right_boundary_with_one_sector(model, L, site, m):
    """A right boundary that holds its smallest sector alone: most output columns then have no S_D block
    in most segments (units the kernels load masked).  What T_D and S_D need is far smaller than a left
    sector times a right one, the extent of such a unit's addresses: the workspace has to hold that
    too, or the plan's check of its tables, which leaves no unit out, refuses it."""
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    idx = ws.right_index
    diag = [c for c in range(idx.n_cohorts) if idx.bra_pos[c] == idx.ket_pos[c] and not idx.tr[c] and idx.cohort_size(c)]
    small = min(diag, key=lambda c: idx.bra.sizes[idx.bra_pos[c]])
    eng = E.Engine(0)   # no workspace of an earlier plan
    try:
        check_sigma(eng, ws, ws.left_index, subset(idx, [small]), "%s L=%d site=%d m=%d" % (model, L, site, m))
    finally:
        eng.close()


def test_workspace_bytes_are_the_plan_s_allocations():
    """What a second plan of a site takes from the device (the first one's lowering has left its entry
    staging in the pool) is what it reports, headroom of the pooled buffers included."""
    ws = SyntheticSite("qc_su2", 16, 7, 256, seed=2)
    eng = E.Engine(0)
    try:
        Lb = E.DeviceBoundary.upload(eng, ws.left_index, ws.random_cohorts(ws.left_index))
        Rb = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
        first = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
        free0 = torch.cuda.mem_get_info()[0]
        second = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
        taken = free0 - torch.cuda.mem_get_info()[0]
        print("taken %d reported %d" % (taken, second.workspace_bytes), flush=True)
        # four allocations (T and S, partial sums, tables, W tiles), each with up to a page of 2 MiB that the
        # device may have had in reserve
        assert abs(taken - second.workspace_bytes) <= 4 * (2 << 20)
        assert first.workspace_bytes == second.workspace_bytes
        second.close()
        first.close()
    finally:
        eng.close()


def test_adjoint_plan_takes_no_memory_it_does_not_use():
    """An adjoint plan of groups too small to run side by side takes no side streams (their library
    handles hold device memory), and no adjoint plan takes hipBLASLt workspaces (64 MiB a stream)."""
    ws = SyntheticSite("qc_su2", 10, 4, 67, seed=2)
    eng = E.Engine(0)
    try:
        Lb = E.DeviceBoundary.upload(eng, ws.left_index, ws.random_cohorts(ws.left_index))
        Rb = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
        psi = torch.from_numpy(ws.random_psi()).to("cuda:0")
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb, algorithm=E.SIGMA_GROUPED, adjoint=True)
        taken = free0 - torch.cuda.mem_get_info()[0]
        print("taken %d reported %d" % (taken, plan.workspace_bytes), flush=True)
        assert taken - plan.workspace_bytes < 64 << 20
        assert np.all(np.isfinite(plan.adjoint(psi)))
        plan.close()
    finally:
        eng.close()


def test_adjoint_without_room_for_side_streams():
    """Where the device has no room for the side streams' library handles, an adjoint plan is made all
    the same and its products run on one stream: the same gradient, bit for bit, as with room."""
    ws = SyntheticSite("qc_su2", 10, 4, 131, seed=2)
    Lc, Rc = ws.random_cohorts(ws.left_index), ws.random_cohorts(ws.right_index)
    psi = torch.from_numpy(ws.random_psi()).to("cuda:0")

    def gradient(room=None):
        eng = E.Engine(0)
        try:
            Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
            fill = None
            if room is not None:
                torch.cuda.synchronize()
                fill = torch.empty(torch.cuda.mem_get_info()[0] - room, dtype=torch.uint8, device="cuda:0")
            plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb, algorithm=E.SIGMA_GROUPED, adjoint=True)
            g = plan.adjoint(psi)
            print("room %s: %d bytes of the plan, %d left" % (room, plan.workspace_bytes, torch.cuda.mem_get_info()[0]),
                  flush=True)
            plan.close()
            del fill
            torch.cuda.empty_cache()
            return g
        finally:
            eng.close()

    want = gradient()
    # the plan and the adjoint's buffers take about 90 MiB, the four library handles about 150 MiB each
    assert np.array_equal(gradient(room=400 << 20), want)


AUTOTUNE = """
import numpy as np
from mqdmrg import engine as E
from mqdmrg.workloads import SyntheticSite
ws = SyntheticSite("heisenberg", 16, 7, 150, seed=3)
eng = E.Engine(0)
Lb = E.DeviceBoundary.upload(eng, ws.left_index, ws.random_cohorts(ws.left_index))
Rb = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
print("timed", plan.autotune(E.PREC_F64), plan.autotune(E.PREC_F32))
plan.close()
eng.close()
"""


def test_autotune_times_only_what_a_choice_changes():
    """A small stage's final tasks run in the wave kernel in FP64 whatever tile is chosen for them: their
    tiles are not timed there (and noise picks none, which FP32 applications of the plan would then use).
    MQ_F_GENERIC=1 sends them to the tile kernels, where every candidate is timed."""
    def timed(**env):
        r = subprocess.run([sys.executable, "-c", AUTOTUNE], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path), **env))
        assert r.returncode == 0, r.stderr[-2000:]
        return [int(x) for x in r.stdout.split("timed")[1].split()]

    wave, tiles = timed(), timed(MQ_F_GENERIC="1")
    print("timed FP64, FP32: wave kernel %s, tile kernels %s" % (wave, tiles), flush=True)
    assert 0 < wave[0] < tiles[0]


STEP = """
import hashlib
import sys
import numpy as np
import torch
from mqdmrg import engine as E, mps
from mqdmrg.symmetry import SiteLayout
from mqdmrg.workloads import SyntheticSite
ws = SyntheticSite("qc_su2", 10, 4, 131, seed=3)
k = ws.site + 1
lay = SiteLayout(ws.bonds[k], ws.basis.phys, ws.bonds[k + 1])
sd, md = E.SiteDesc(ws.basis.sym, ws.bonds[k], ws.basis.phys, ws.bonds[k + 1]), E.MpoDesc(ws.mpo[k])
eng = E.Engine(0)
b = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
bra, ket = (torch.from_numpy(mps.random_site_vector(lay, ws.rng)).to("cuda:0") for _ in range(2))
h = hashlib.sha256()
for x in E.right_step(eng, sd, md, bra, ket, b).download():
    h.update(np.ascontiguousarray(x).tobytes())
print("digest", h.hexdigest())
"""


def test_generic_switches_are_of_one_stage_each():
    """MQ_T_GENERIC is the T stage's switch and MQ_F_GENERIC the final stage's, of a boundary step too: the
    final stage's own kernel and the generic one sum in another order, so turning it off shows in the bits
    with either form of the T stage."""
    def digest(**env):
        r = subprocess.run([sys.executable, "-c", STEP], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path), **env))
        assert r.returncode == 0, r.stderr[-2000:]
        return r.stdout.split("digest")[1].strip()

    assert digest() != digest(MQ_F_GENERIC="1")
    assert digest(MQ_T_GENERIC="1") != digest(MQ_T_GENERIC="1", MQ_F_GENERIC="1")


@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 20, 9, 420), ("qc_su2", 10, 4, 131), ("qc", 10, 4, 150),
                                            ("heisenberg", 24, 11, 1100)])
def test_bf16x3_of_halfway_values(eng, model, L, site, m):
    """BF16x3 where every value of the right boundary is, rounded to FP32, halfway between two bf16 and in
    FP64 a little above or below: the case in which the T stage's split depends on what it rounds.  The
    split keeps 17 bits whichever way such a value goes."""
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    Lc = ws.random_cohorts(ws.left_index)

    def halfway(x):
        bits = (x.astype(np.float32).view(np.uint32) & 0xffff0000) | 0x8000
        return bits.view(np.float32).astype(np.float64) * (1 + 1e-9 * np.sign(ws.rng.standard_normal(len(x))))
    Rc = [halfway(x) if x is not None else None for x in ws.random_cohorts(ws.right_index)]
    psi_h = ws.random_psi()
    ref = O.SigmaOracle(ws.site_desc, ws.mpo_desc, host_boundary(ws.left_index, Lc), host_boundary(ws.right_index, Rc)).apply(psi_h)
    Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(psi_h).to("cuda:0")
    out = torch.full_like(psi, float("nan"))
    plan.apply(psi, out, precision=E.PREC_BF16X3)
    eng.sync()
    err = np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref)
    print("%s L=%d site=%d m=%d: %.2e" % (model, L, site, m, err), flush=True)
    assert err <= RTOL[E.PREC_BF16X3]
    plan.close()


SIGMA_SHAPES = [("heisenberg", 16, 7, 150), ("heisenberg", 12, 1, 64), ("hubbard", 12, 5, 301), ("hubbard", 10, 7, 90),
                ("qc", 8, 3, 77), ("qc", 10, 1, 60), ("qc_su2", 10, 4, 131), ("qc_su2", 12, 8, 57), ("qc_su2", 14, 6, 101),
                ("heisenberg", 20, 9, 420), ("heisenberg", 24, 11, 1100)]


@pytest.mark.parametrize("model,L,site,m", SIGMA_SHAPES)
def test_every_output_block_matches_oracle(eng, model, L, site, m):
    """sigma block by block and in strips of 64 columns: a wrong edge tile of a small block does not drown
    in the norm of the whole vector.  An element's error is measured against the larger of its strip's rms
    and the vector's.  BF16x3 keeps 17 bits of every operand (7.6e-6); a lost low part would be 1.5e-3 in
    the elements it concerns."""
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    Lc, Rc = ws.random_cohorts(ws.left_index), ws.random_cohorts(ws.right_index)
    psi_h = ws.random_psi()
    ref = O.SigmaOracle(ws.site_desc, ws.mpo_desc, host_boundary(ws.left_index, Lc), host_boundary(ws.right_index, Rc)).apply(psi_h)
    Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(psi_h).to("cuda:0")
    lay = ws.layout
    n = sum(ls * cols for ls, cols in zip(lay.left.sizes, lay.rp_cols))
    rms = np.linalg.norm(ref) / np.sqrt(n)
    for prec, tol in RTOL.items():
        out = torch.full_like(psi, float("nan"))
        plan.apply(psi, out, precision=prec)
        eng.sync()
        got, worst = out.cpu().numpy(), 0.0
        for ls, cols, o in zip(lay.left.sizes, lay.rp_cols, lay.rp_offset):
            for c in range(0, cols, 64):
                a, b = o + c * ls, o + min(c + 64, cols) * ls
                scale = max(np.linalg.norm(ref[a:b]), rms * np.sqrt(b - a))
                worst = max(worst, np.linalg.norm(got[a:b] - ref[a:b]) / scale)
        print("%s L=%d site=%d m=%d precision %d: worst strip %.2e" % (model, L, site, m, prec, worst), flush=True)
        assert worst <= tol
    plan.close()


def final_tiles(ws, cols, small_only):
    """Tiles of 32 rows x `cols` columns of the final stage's tasks (one per output block and part of its
    summation range, of about 2048 keys each), all of them or those of at most 32 rows."""
    idx, lay, n = ws.left_index, ws.layout, 0
    blocks = {(int(idx.bra_pos[c]), int(idx.ket_pos[c])): int((idx.offsets[c] > -1).sum()) for c in range(idx.n_cohorts)}
    for lo, (ls, N) in enumerate(zip(lay.left.sizes, lay.rp_cols)):
        segs = []
        for lb, s in enumerate(lay.left.sizes):
            per = max(1, 2048 // s)
            segs += [min(per, blocks.get((lo, lb), 0) - j) * s for j in range(0, blocks.get((lo, lb), 0), per)]
        if N and segs and (ls <= 32 or not small_only):
            n += min(len(segs), 64, -(-sum(segs) // 2048)) * (-(-ls // 32)) * (-(-N // cols))
    return n


@pytest.mark.parametrize("m", [500, 1200])
def test_wave_form_of_32_rows(eng, m):
    """Stages with at least 1024 tiles of the final stage's wave form, which then takes 32 rows per wave:
    in FP64 (m = 500, 1200) and in FP32 (m = 1200)."""
    ws = SyntheticSite("qc", 12 if m == 500 else 16, 5 if m == 500 else 7, m, seed=m)
    assert final_tiles(ws, 16, m == 1200) >= 1024
    assert m == 500 or final_tiles(ws, 64, True) >= 1024
    check_sigma(eng, ws, ws.left_index, ws.right_index, "qc m=%d" % m)


@pytest.mark.parametrize("kind", ["left", "right"])
@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 20, 9, 420), ("heisenberg", 24, 11, 1100), ("qc_su2", 14, 6, 1500)])
def test_steps_over_sectors_of_several_tiles(eng, kind, model, L, site, m):
    """Boundary steps whose tasks have several column tiles (a sector of the bra above 64, with a remainder)
    and several row tiles per block."""
    from mqdmrg import mps
    from mqdmrg.symmetry import SiteLayout
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    k = site if kind == "left" else site + 1
    index = ws.left_index if kind == "left" else ws.right_index
    lay = SiteLayout(ws.bonds[k], ws.basis.phys, ws.bonds[k + 1])
    # the new boundary's sectors: its tasks' columns
    sectors = (lay.right if kind == "left" else lay.left).sizes
    assert max(sectors) > 64 and any(s > 64 and s % 64 and s % 16 for s in sectors)
    sd, md = E.SiteDesc(ws.basis.sym, ws.bonds[k], ws.basis.phys, ws.bonds[k + 1]), E.MpoDesc(ws.mpo[k])
    coh = ws.random_cohorts(index)
    hb = host_boundary(index, coh)
    bra, ket = mps.random_site_vector(lay, ws.rng), mps.random_site_vector(lay, ws.rng)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")  # noqa: E731
    b = E.DeviceBoundary.upload(eng, index, coh)
    if kind == "left":
        ref = O.left_step(sd, md, mps.rp_to_lp(lay, bra), ket, hb, True)
        new = E.left_step(eng, sd, md, d(mps.rp_to_lp(lay, bra)), d(ket), b)
    else:
        ref = O.right_step(sd, md, bra, ket, hb, True)
        new = E.right_step(eng, sd, md, d(bra), d(ket), b)
    got = new.download()
    rms = np.sqrt(sum(float(np.sum(y ** 2)) for y in ref.cohorts) / max(1, sum(len(y) for y in ref.cohorts)))
    worst = 0.0
    for x, y in zip(got, ref.cohorts):
        if len(y):
            worst = max(worst, np.linalg.norm(x - y) / max(np.linalg.norm(y), rms * np.sqrt(len(y))))
    print("%s %s L=%d site=%d m=%d: worst cohort %.2e" % (kind, model, L, site, m, worst), flush=True)
    assert worst <= RTOL[E.PREC_F64]


@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 24, 11, 1100), ("qc_su2", 10, 4, 131)])
def test_adjoint_of_groups_side_by_side(model, L, site, m):
    """Gradients of plans whose groups' products run on the side streams (a context of its own shows them
    being made: four library handles of at least 32 MiB each beyond what the plan reports), three through
    one plan, against the oracle: all terms of the spin chain, a sample of the ab initio one."""
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    Lc, Rc = ws.random_cohorts(ws.left_index), ws.random_cohorts(ws.right_index)
    host = host_boundary(ws.left_index, Lc), host_boundary(ws.right_index, Rc)
    n = ws.mpo_desc.desc.n_terms
    terms = range(n) if n < 50 else sorted(set(ws.rng.integers(0, n, 40).tolist()))
    eng = E.Engine(0)
    try:
        Lb, Rb = E.DeviceBoundary.upload(eng, ws.left_index, Lc), E.DeviceBoundary.upload(eng, ws.right_index, Rc)
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb, algorithm=E.SIGMA_GROUPED, adjoint=True)
        assert free0 - torch.cuda.mem_get_info()[0] - plan.workspace_bytes >= 128 << 20
        psis = [ws.random_psi() for _ in range(2)]
        grads = [plan.adjoint(torch.from_numpy(x).to("cuda:0")) for x in psis + psis[:1]]
        assert np.array_equal(grads[0], grads[2])
        for x, g in zip(psis, grads):
            ref = np.array([float(np.dot(x, O.SigmaOracle(ws.site_desc, O._TermMpo(ws.mpo_desc, t), *host).apply(x)))
                            for t in terms])
            err = np.linalg.norm(g[list(terms)] - ref) / np.linalg.norm(ref)
            print("adjoint %s L=%d site=%d m=%d: %.2e" % (model, L, site, m, err), flush=True)
            assert err <= 10 * RTOL[E.PREC_F64]   # two products in a row and the sum over a term's entries
        plan.close()
    finally:
        eng.close()


WIDE = """
import hashlib
import torch
from mqdmrg import engine as E
from mqdmrg.workloads import SyntheticSite
eng = E.Engine(0)
for a in [("heisenberg", 16, 7, 150), ("qc", 8, 3, 77), ("qc_su2", 10, 4, 131), ("qc_su2", 14, 6, 101)]:
    ws = SyntheticSite(*a, seed=3)
    Lb = E.DeviceBoundary.upload(eng, ws.left_index, ws.random_cohorts(ws.left_index))
    Rb = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(ws.random_psi()).to("cuda:0")
    for prec in (E.PREC_F64, E.PREC_F32, E.PREC_BF16X3):
        out = torch.empty_like(psi)
        plan.apply(psi, out, precision=prec)
        eng.sync()
        print("digest", *a, prec, hashlib.sha256(out.cpu().numpy().tobytes()).hexdigest(), flush=True)
    plan.close()
eng.close()
"""


def test_wide_groups_have_the_same_bits():
    """Groups of 2^24 rows and more address T_D with 64-bit offsets and plain loads: MQ_S_WIDE=1 takes that
    form at any size, with every bit as with 32-bit offsets (which the oracle tests cover)."""
    def digests(**env):
        r = subprocess.run([sys.executable, "-c", WIDE], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path), **env))
        assert r.returncode == 0, r.stderr[-2000:]
        return [x for x in r.stdout.splitlines() if x.startswith("digest")]

    narrow = digests()
    assert len(narrow) == 12 and digests(MQ_S_WIDE="1") == narrow


def test_profile_counts_the_products_made(eng):
    """The S-stage flops that a profile reports are those of the blocks the kernel multiplies: their rate is
    below the chip's FP64 matrix peak (78.6 TFLOP/s), which the visited tiles counted whole exceed."""
    ws = SyntheticSite("qc_su2", 24, 11, 700, seed=2)
    Lb = E.DeviceBoundary.upload(eng, ws.left_index, ws.random_cohorts(ws.left_index))
    Rb = E.DeviceBoundary.upload(eng, ws.right_index, ws.random_cohorts(ws.right_index))
    plan = E.SigmaPlan(eng, ws.site_desc, ws.mpo_desc, Lb, Rb)
    psi = torch.from_numpy(ws.random_psi()).to("cuda:0")
    ms, flops, _ = plan.profile(psi, torch.empty_like(psi), reps=5)
    model = plan.flops - flops[0] - flops[2]   # one multiplication per nonzero coupling
    print("S stage %.3f ms, %.3e flops, %.1f TFLOP/s; couplings %.3e" % (ms[2], flops[1], flops[1] / ms[2] * 1e-9, model), flush=True)
    assert 0 < model < flops[1] < 78.6e9 * ms[2]
    plan.close()


@pytest.mark.parametrize("kind", ["left", "right"])
@pytest.mark.parametrize("model,L,site,m", [("heisenberg", 16, 7, 150), ("hubbard", 12, 5, 301)])
def test_step_keeps_infinities_of_the_bra(eng, kind, model, L, site, m):
    """An infinity in the bra reaches the elements of the new boundary that it contributes to as an infinity of
    the oracle's sign, also where it is the last key of a segment that is no multiple of 16 (a NaN if the
    padding multiplied it).  Elsewhere a zero of S_D may meet it, which the oracle's sum does not hold."""
    from mqdmrg import mps
    from mqdmrg.symmetry import SiteLayout
    ws = SyntheticSite(model, L, site, m, seed=L + m)
    k = site if kind == "left" else site + 1
    index = ws.left_index if kind == "left" else ws.right_index
    lay = SiteLayout(ws.bonds[k], ws.basis.phys, ws.bonds[k + 1])
    sd, md = E.SiteDesc(ws.basis.sym, ws.bonds[k], ws.basis.phys, ws.bonds[k + 1]), E.MpoDesc(ws.mpo[k])
    coh = ws.random_cohorts(index)
    hb = host_boundary(index, coh)
    bra, ket = mps.random_site_vector(lay, ws.rng), mps.random_site_vector(lay, ws.rng)
    # the last element of the largest block: last key of its row (left step) or column segment (right step)
    lb = max(range(len(lay.left.sizes)), key=lambda i: lay.left.sizes[i] * lay.rp_cols[i])
    bra[lay.rp_offset[lb] + lay.left.sizes[lb] * lay.rp_cols[lb] - 1] = np.inf
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")  # noqa: E731
    b = E.DeviceBoundary.upload(eng, index, coh)
    if kind == "left":
        ref = O.left_step(sd, md, mps.rp_to_lp(lay, bra), ket, hb, True)
        new = E.left_step(eng, sd, md, d(mps.rp_to_lp(lay, bra)), d(ket), b)
    else:
        ref = O.right_step(sd, md, bra, ket, hb, True)
        new = E.right_step(eng, sd, md, d(bra), d(ket), b)
    got, want = np.concatenate(new.download()), np.concatenate(ref.cohorts)
    print("%s %s: infinities %d of %d, NaN %d of %d" % (kind, model, np.isinf(got).sum(), np.isinf(want).sum(),
                                                       np.isnan(got).sum(), np.isnan(want).sum()), flush=True)
    assert np.isinf(want).any()
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
