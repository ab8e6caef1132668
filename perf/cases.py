"""Timed workloads of the engine: what a two-site DMRG program asks of it, through mqdmrg.engine.

A sweep spends its time in four calls, and these are the cases:

  sigma    one H_eff psi product with a plan that the site keeps (SigmaPlan.apply); a site makes
           about eight of them, in FP64, FP32 or BF16x3
  left     the left boundary moved over one site (engine.left_step)
  right    the right boundary moved over one site (engine.right_step)
  jd       the whole eigensolver of a site (SigmaPlan.jd), on a real canonical state
  adjoint  the derivative of psi.H_eff psi with respect to every MPO term, from which the reduced
           density matrices follow (SigmaPlan.adjoint)

Models: spin chains (U1, a handful of MPO terms), the Hubbard chain (TwoU1), and ab initio
Hamiltonians in TwoU1 ("qc") and spin-adapted SU2U1 ("qc_su2") symmetry, whose MPOs have hundreds
of bond states and tens of thousands of terms.  Bond dimension m counts states (multiplets for
qc_su2).  Shapes come from mqdmrg.workloads: site tensors and boundaries have the sector structure
of a chain's interior, with random contents (jd: a random state brought to canonical form)."""
import functools
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "maquis-dmrg_amd"))

from mqdmrg import engine as E  # noqa: E402
from mqdmrg import models  # noqa: E402
from mqdmrg.dmrg import TwoSiteDMRG  # noqa: E402
from mqdmrg.symmetry import SiteLayout  # noqa: E402
from mqdmrg.workloads import SyntheticSite  # noqa: E402


# ---------------------------------------------------------------------------- the cases
def _case(name, op, model, L, site, m, precision="f64"):
    return {"name": name, "op": op, "model": model, "L": L, "site": site, "m": m, "precision": precision}


def listed():
    return [
        # a spin chain at a small bond dimension: blocks of tens of rows, all latency
        _case("sigma heisenberg L32", "sigma", "heisenberg", 32, 15, 128),
        # the Hubbard chain at production size: many small blocks, a sparse MPO
        _case("sigma hubbard L64", "sigma", "hubbard", 64, 31, 1024),
        # ab initio, TwoU1, small active space off the middle of the chain, odd bond dimension
        _case("sigma qc L16 f32", "sigma", "qc", 16, 5, 301, "f32"),
        # the early sweeps of a spin-adapted calculation (small m, converged quickly)
        _case("sigma qc_su2 L16", "sigma", "qc_su2", 16, 7, 256, "bf16x3"),
        # production size of a 24-orbital active space, both precisions that are used for sweeps
        _case("sigma qc_su2 L24", "sigma", "qc_su2", 24, 11, 1000),
        _case("sigma qc_su2 L24 bf16x3", "sigma", "qc_su2", 24, 11, 1000, "bf16x3"),
        # 30 orbitals, the largest whose plan in both precisions fits the card three times
        _case("sigma qc_su2 L30", "sigma", "qc_su2", 30, 14, 1500),
        _case("sigma qc_su2 L30 bf16x3", "sigma", "qc_su2", 30, 14, 1500, "bf16x3"),
        # the boundary steps between two sites of those sweeps
        _case("left qc_su2 L24", "left", "qc_su2", 24, 11, 1000),
        _case("right qc_su2 L30", "right", "qc_su2", 30, 14, 1500),
        # a whole site optimisation of the early sweeps
        _case("jd qc_su2 L16", "jd", "qc_su2", 16, 7, 256),
        # one site of the derivative sweep (orbital gradients, density matrices)
        _case("adjoint qc_su2 L16", "adjoint", "qc_su2", 16, 7, 256),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    op = rng.choice(["sigma"] * 6 + ["left", "right", "left", "right", "jd", "adjoint"])
    if op == "jd":
        L = rng.randint(10, 16)
        return {"op": op, "model": "qc_su2", "L": L, "site": L // 2 - 1, "m": _log_int(rng, 40, 300), "precision": "f64"}
    if op == "adjoint":
        L = rng.randint(10, 16)
        return {"op": op, "model": "qc_su2", "L": L, "site": rng.randint(1, L - 4), "m": _log_int(rng, 40, 300),
                "precision": "f64"}
    model = rng.choice(["heisenberg", "hubbard", "qc", "qc_su2", "qc_su2", "qc_su2"])
    L, m = {"heisenberg": (rng.randint(12, 64), _log_int(rng, 32, 512)),
            "hubbard": (rng.randint(12, 64), _log_int(rng, 64, 1500)),
            "qc": (rng.randint(8, 16), _log_int(rng, 40, 400)),
            "qc_su2": (rng.randint(12, 30), _log_int(rng, 100, 1400))}[model]
    # mostly the interior of the chain; the ends have small bonds and few MPO states
    site = rng.randint(L // 2 - 2, L // 2) if rng.random() < 0.7 else rng.randint(1, L - 4)
    precision = rng.choice(["f64", "f64", "f32", "bf16x3", "bf16x3"]) if op == "sigma" else "f64"
    return {"op": op, "model": model, "L": L, "site": site, "m": m, "precision": precision}


# ---------------------------------------------------------------------------- shapes (host, no data)
@functools.lru_cache(maxsize=None)
def _chain(model, L):
    return models.chain(model, L)


@functools.lru_cache(maxsize=8)
def _site(model, L, site, m):
    return SyntheticSite(model, L, site, m, chain=_chain(model, L))


class _Shape:
    """The tensors of one case: site layout, MPO and boundary indices."""

    def __init__(self, c):
        ws = _site(c["model"], c["L"], c["site"], c["m"])
        k = c["site"]
        self.left = self.right = None
        if c["op"] in ("left", "right"):   # one-site tensors: site k (left step), site k + 1 (right step)
            k = k if c["op"] == "left" else k + 1
            self.W, phys = ws.mpo[k], ws.basis.phys
            self.mpo_desc = E.MpoDesc(self.W)
            self.layout = SiteLayout(ws.bonds[k], phys, ws.bonds[k + 1])
            self.site_desc = E.SiteDesc(ws.basis.sym, ws.bonds[k], phys, ws.bonds[k + 1])
            if c["op"] == "left":
                self.left = ws.left_index
            else:
                self.right = ws.right_index
        else:
            self.W, self.mpo_desc, self.layout, self.site_desc = ws.W12, ws.mpo_desc, ws.layout, ws.site_desc
            self.left, self.right = ws.left_index, ws.right_index
        self.sym = ws.basis.sym


@functools.lru_cache(maxsize=8)
def _shape(op, model, L, site, m):
    return _Shape({"op": op, "model": model, "L": L, "site": site, "m": m})


def _shape_of(c):
    return _shape("sigma" if c["op"] in ("jd", "adjoint") else c["op"], c["model"], c["L"], c["site"], c["m"])


# ---------------------------------------------------------------------------- inputs from a seed
_DEVICE = "cuda:0" if torch.cuda.is_available() else "cpu"


def _generator(seed):
    g = torch.Generator(device=_DEVICE)
    g.manual_seed(int(seed))
    return g


def _cohorts(index, gen):
    """Host data of a boundary: one array per stored cohort (N(0, 1) elements)."""
    sizes = [0 if index.tr[ci] else index.cohort_size(ci) for ci in range(index.n_cohorts)]
    flat = torch.randn(sum(sizes), dtype=torch.float64, device=_DEVICE, generator=gen).cpu().numpy()
    out, at = [], 0
    for n in sizes:
        out.append(flat[at:at + n] if n else None)
        at += n
    return out


def _vector(layout, gen):
    """A normalised site tensor in the padded right-paired layout (padding zero), on the device."""
    v = torch.zeros(layout.rp_total, dtype=torch.float64, device=_DEVICE)
    for lb, ls in enumerate(layout.left.sizes):
        n = ls * layout.rp_cols[lb]
        v[layout.rp_offset[lb]:layout.rp_offset[lb] + n] = torch.randn(n, dtype=torch.float64, device=_DEVICE, generator=gen)
    return v / torch.linalg.norm(v)


def _inputs(c, seed):
    """(left cohorts, right cohorts, psi) of a case, from its seed alone."""
    s, gen = _shape_of(c), _generator(seed)
    left = _cohorts(s.left, gen) if s.left is not None else None
    right = _cohorts(s.right, gen) if s.right is not None else None
    return left, right, _vector(s.layout, gen)


@functools.lru_cache(maxsize=1)
def _engine():
    return E.Engine(0)


@functools.lru_cache(maxsize=4)
def _two_site_mpo(model, L, site):
    return {}   # site -> two-site MPO, filled by TwoSiteDMRG and shared by later states


def _canonical(c, seed):
    """A random state of bond dimension m in mixed canonical form around the pair (site, site + 1),
    with both boundaries: what the driver has in hand when it optimises that pair."""
    eng, i = _engine(), c["site"]
    basis, mpo, target = _chain(c["model"], c["L"])
    d = TwoSiteDMRG(eng, c["model"], c["L"], m=c["m"], init_m=c["m"], init_bonds="total", seed=int(seed), mpo=mpo,
                    basis=basis, target=target)
    d.ts_mpo = _two_site_mpo(c["model"], c["L"], i)
    d.init_boundaries()
    for j in range(i):
        d.move_center_right(j)
        a = d.sites[j]
        d.Lb[j + 1] = E.left_step(eng, a.desc, d.mpo_desc[j], a.lp_data(), a.data, d.Lb[j])
    return d


def prepare(case, seed):
    c, eng = case, _engine()
    st = {"op": c["op"], "eng": eng, "precision": E.PRECISIONS[c["precision"]]}
    if c["op"] == "jd":
        d = _canonical(c, seed)
        theta = d.merge(c["site"])
        wdesc = d.twosite_mpo(c["site"])[1]
        st["psi"] = theta.data / torch.linalg.norm(theta.data)
        st["out"] = torch.zeros_like(st["psi"])
        st["plan"] = E.SigmaPlan(eng, theta.desc, wdesc, d.Lb[c["site"]], d.Rb[c["site"] + 2])
        return st
    s = _shape_of(c)
    left, right, psi = _inputs(c, seed)
    st["psi"] = psi
    lb = E.DeviceBoundary.upload(eng, s.left, left) if left is not None else None
    rb = E.DeviceBoundary.upload(eng, s.right, right) if right is not None else None
    st.update(shape=s, left=lb, right=rb)
    if c["op"] in ("sigma", "adjoint"):
        st["plan"] = E.SigmaPlan(eng, s.site_desc, s.mpo_desc, lb, rb, adjoint=c["op"] == "adjoint")
        st["sigma"] = torch.zeros_like(psi)
    elif c["op"] == "left":
        st["bra_lp"] = torch.zeros(s.layout.lp_total, dtype=torch.float64, device=_DEVICE)
        E.reshape_right_to_left(eng, s.site_desc, psi, st["bra_lp"])
    return st


class _Block:
    """Device memory as an array: a boundary's cohorts lie in one allocation.  A tensor made from it
    holds this object, and with it the boundary."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False), "version": 3}


def _boundary_data(b):
    """All cohorts of a device boundary, in place (no copy)."""
    from ctypes import byref, c_void_p
    p = c_void_p()
    E.check(E.lib().mq_boundary_cohort_ptr(b.h, 0, byref(p)))
    return torch.as_tensor(_Block(b, p.value, _offsets(b.index)[1]), device=_DEVICE)


def run(state):
    op, eng = state["op"], state["eng"]
    if op == "sigma":
        state["plan"].apply(state["psi"], state["sigma"], precision=state["precision"])
        return state["sigma"]
    if op == "adjoint":
        return state["plan"].adjoint(state["psi"])
    if op == "jd":
        e, n = state["plan"].jd(state["psi"], state["out"], tol=1e-8, max_iter=8)
        return {"energy": e, "iterations": n, "vector": state["out"]}
    s = state["shape"]
    if op == "left":
        new = E.left_step(eng, s.site_desc, s.mpo_desc, state["bra_lp"], state["psi"], state["left"])
    else:
        new = E.right_step(eng, s.site_desc, s.mpo_desc, state["psi"], state["psi"], state["right"])
    return _boundary_data(new)


# ---------------------------------------------------------------------------- what a pass cannot do without
def _offsets(index):
    """Element offset of every cohort in a boundary's allocation (each rounded up to 32), and its size."""
    off, at = [], 0
    for ci in range(index.n_cohorts):
        off.append(at)
        at += -(-index.cohort_size(ci) // 32) * 32
    return off, max(at, 32)


def _new_index(c):
    s = _shape_of(c)
    return E.step_index(c["op"], s.site_desc, s.mpo_desc, s.left if c["op"] == "left" else s.right)


def _entries(s):
    """The distinct nonzeros of the MPO tensor as (b1, b2, sector in, state in, sector out, state out)."""
    pos = {p: i for i, p in enumerate(s.layout.phys.charges)}
    seen = {}
    for (b1, b2), terms in _term_lists(s.W):
        for op, scale in terms:
            for (cin, cout), ents in op.blocks.items():
                for e in ents:
                    k = (b1, b2, pos[tuple(cin)], e[0], pos[tuple(cout)], e[1])
                    seen[k] = seen.get(k, 0.0) + scale * e[2]
    return seen


def _term_lists(W):
    if hasattr(W, "sorted_terms"):
        b1, b2, op, sc = W.sorted_terms()
        for x, y, o, z in zip(b1, b2, op, sc):
            yield (int(x), int(y)), [(W.ops[int(o)], float(z))]
    else:
        yield from sorted(W.terms.items())


def _has(index):
    """has[cohort][b] and a (bra sector, ket sector) -> cohort map of a boundary index."""
    return index.offsets >= 0, {(int(a), int(b)): ci for ci, (a, b) in enumerate(zip(index.bra_pos, index.ket_pos))}


@functools.lru_cache(maxsize=None)
def _flops(op, model, L, site, m):
    """2 flops per element of the three contractions in the reference's model: T = psi R (or L psi),
    one scaled add of a slab per MPO coupling, and the product with the other boundary (steps: the bra).
    Couplings that a spin recoupling factor happens to cancel are counted."""
    c = {"op": op, "model": model, "L": L, "site": site, "m": m}
    s = _shape_of(c)
    lay = s.layout
    ent = np.asarray(list(_entries(s)), np.int64).reshape(-1, 6)
    lsz, rsz, nph = lay.left.sizes, lay.right.sizes, len(lay.phys)
    new = _new_index(c) if op in ("left", "right") else None
    kin, nout = (s.left, new) if op == "left" else (s.right, s.left if op == "sigma" else new)
    hk, mk = _has(kin)
    hn, mn = _has(nout)
    at = lambda i, sign, s_, sec: sec.position((i[0] + sign * s_[0], i[1] + sign * s_[1]))  # noqa: E731
    npair = len(lsz) * len(rsz)
    slab = np.outer(lsz, rsz).ravel().astype(np.float64)
    K = np.zeros((nph, npair, kin.aux_dim), np.float32)    # keys of the first contraction per sector pair
    N = np.zeros((nph, npair, nout.aux_dim), np.float32)   # and of the last
    total = 0.0
    for lb, lc in enumerate(lay.left.charges):
        for rb, rc in enumerate(lay.right.charges):
            p = lb * len(rsz) + rb
            for q, pc in enumerate(lay.phys.charges):
                d = lay.phys.sizes[q]
                r, l = at(lc, 1, pc, lay.right), at(rc, -1, pc, lay.left)
                if op == "left":   # pair (bra left sector, ket right sector)
                    ck, cn, inner, outer = mk.get((lb, l)), mn.get((r, rb)), (lsz + [0])[l], (rsz + [0])[r]
                else:              # pair (ket left sector, bra right sector)
                    ck, inner, outer = mk.get((r, rb)), (rsz + [0])[r], (lsz + [0])[l]
                    cn = mn.get((l, lb) if op == "sigma" else (lb, l))
                if ck is not None:
                    K[q, p] = hk[ck]
                    total += 2 * slab[p] * inner * d * int(hk[ck].sum())
                if cn is not None and not (new is not None and new.tr[cn]):
                    N[q, p] = hn[cn]
                    total += 2 * slab[p] * outer * d * int(hn[cn].sum())
    bk, bn = (ent[:, 0], ent[:, 1]) if op == "left" else (ent[:, 1], ent[:, 0])
    for qi in range(nph):
        for qo in range(nph):
            pick = (ent[:, 2] == qi) & (ent[:, 4] == qo)
            if pick.any():
                count = np.zeros((kin.aux_dim, nout.aux_dim), np.float32)
                np.add.at(count, (bk[pick], bn[pick]), 1.0)
                total += 2 * float(np.einsum("p,pn,pn->", slab, K[qi] @ count, N[qo], optimize=True))
    return float(total), len(ent)


def work(case):
    c = case
    s = _shape_of(c)
    size = lambda index: 0 if index is None else sum(0 if index.tr[i] else index.cohort_size(i)  # noqa: E731
                                                     for i in range(index.n_cohorts))
    op = c["op"] if c["op"] in ("left", "right") else "sigma"
    fl, nw = _flops(op, c["model"], c["L"], c["site"], c["m"])
    reads = size(s.left) + size(s.right) + s.layout.rp_total + nw
    if op == "sigma":
        written = s.layout.rp_total
    else:
        new = _new_index(c)
        written = size(new)
        reads += s.layout.lp_total if c["op"] == "left" else 0
    times = 8 if c["op"] == "jd" else 1   # iterations, each one product
    return {"bytes": 8.0 * times * (reads + written), "flops": times * fl}


# ---------------------------------------------------------------------------- 64-bit results without the engine
def _dense_boundary(index, cohorts, bra_sizes, ket_sizes):
    """B[b, bra state, ket state] of block-sparse boundary data."""
    ob, ok = np.cumsum([0] + list(bra_sizes)), np.cumsum([0] + list(ket_sizes))
    out = torch.zeros(index.aux_dim, ob[-1], ok[-1], dtype=torch.float64)
    where = {(int(a), int(b)): ci for ci, (a, b) in enumerate(zip(index.bra_pos, index.ket_pos))}
    for ci in range(index.n_cohorts):
        i, j = int(index.bra_pos[ci]), int(index.ket_pos[ci])
        ls, rs = bra_sizes[i], ket_sizes[j]
        data = torch.from_numpy(cohorts[where[(j, i)]] if index.tr[ci] else cohorts[ci]) if ls * rs else None
        for b in range(index.aux_dim):
            o = int(index.offsets[ci, b])
            if o < 0 or data is None:
                continue
            blk = data[o:o + ls * rs]
            blk = blk.view(ls, rs) if index.tr[ci] else blk.view(rs, ls).t()
            out[b, ob[i]:ob[i + 1], ok[j]:ok[j + 1]] = float(index.conj_scales[ci, b]) * blk
    return out.to(_DEVICE)


def _dense_vector(layout, v):
    """psi[left state, physical state, right state]."""
    oL, oR = np.cumsum([0] + layout.left.sizes), np.cumsum([0] + layout.right.sizes)
    oP = np.cumsum([0] + layout.phys.sizes)
    out = torch.zeros(oL[-1], oP[-1], oR[-1], dtype=torch.float64, device=_DEVICE)
    for lb, q, ss, rb, at in _slabs(layout):
        ls, rs = layout.left.sizes[lb], layout.right.sizes[rb]
        out[oL[lb]:oL[lb + 1], oP[q] + ss, oR[rb]:oR[rb + 1]] = v[at:at + ls * rs].view(rs, ls).t()
    return out


def _slabs(layout):
    for lb, lc in enumerate(layout.left.charges):
        for q, pc in enumerate(layout.phys.charges):
            rc = (lc[0] + pc[0], lc[1] + pc[1])
            rb = layout.right.position(rc)
            if rb == len(layout.right):
                continue
            for ss in range(layout.phys.sizes[q]):
                col = layout.rpb(pc, rc) + ss * layout.right.sizes[rb]
                yield lb, q, ss, rb, layout.rp_offset[lb] + col * layout.left.sizes[lb]


def exact(case, seed):
    c = case
    if c["op"] in ("jd", "adjoint") or c["model"] == "qc_su2":
        return None   # spin-adapted contractions need 9j recoupling; an eigensolver has a path of its own
    s = _shape_of(c)
    lay = s.layout
    left, right, psi = _inputs(c, seed)
    oP = np.cumsum([0] + lay.phys.sizes)
    d = int(oP[-1])
    w1, w2 = s.W.row_dim, s.W.col_dim
    W = np.zeros((w1, d, w2, d))   # [b1, out, b2, in]
    for (b1, b2, qi, ri, qo, co), v in _entries(s).items():
        W[b1, oP[qo] + co, b2, oP[qi] + ri] += v
    W = torch.from_numpy(W).to(_DEVICE)
    x = _dense_vector(lay, psi)
    nl, nr = x.shape[0], x.shape[2]
    if c["op"] == "left":
        Ld = _dense_boundary(s.left, left, lay.left.sizes, lay.left.sizes)
        T = (Ld.reshape(w1 * nl, nl) @ x.reshape(nl, d * nr)).reshape(w1, nl, d, nr)          # b1, l', in, r
        T = T.permute(0, 2, 1, 3).reshape(w1 * d, nl * nr)
        S = (W.permute(2, 1, 0, 3).reshape(w2 * d, w1 * d) @ T).reshape(w2, d, nl, nr)        # b2, out, l', r
        S = S.reshape(w2, d * nl, nr)
        new = torch.matmul(x.permute(1, 0, 2).reshape(d * nl, nr).t().contiguous(), S)        # b2, r', r
        return _pack(_new_index(c), new, lay.right.sizes, lay.right.sizes)
    Rd = _dense_boundary(s.right, right, lay.right.sizes, lay.right.sizes)
    T = x.reshape(nl * d, nr) @ Rd.permute(1, 0, 2).reshape(nr, w2 * nr)                      # (l, in), (b2, r')
    T = T.reshape(nl, d, w2, nr).permute(2, 1, 0, 3).reshape(w2 * d, nl * nr)
    S = (W.reshape(w1 * d, w2 * d) @ T).reshape(w1, d, nl, nr)                                # b1, out, l, r'
    if c["op"] == "right":
        S = S.permute(0, 2, 1, 3).reshape(w1 * nl, d * nr)
        new = (S @ x.reshape(nl, d * nr).t()).reshape(w1, nl, nl)                             # b1, l, l'
        return _pack(_new_index(c), new, lay.left.sizes, lay.left.sizes)
    Ld = _dense_boundary(s.left, left, lay.left.sizes, lay.left.sizes)                        # b1, l', l
    y = Ld.permute(1, 0, 2).reshape(nl, w1 * nl) @ S.permute(0, 2, 1, 3).reshape(w1 * nl, d * nr)
    y = y.reshape(nl, d, nr)
    out = torch.zeros_like(psi)
    oL, oR = np.cumsum([0] + lay.left.sizes), np.cumsum([0] + lay.right.sizes)
    for lb, q, ss, rb, at in _slabs(lay):
        n = lay.left.sizes[lb] * lay.right.sizes[rb]
        out[at:at + n] = y[oL[lb]:oL[lb + 1], oP[q] + ss, oR[rb]:oR[rb + 1]].t().reshape(-1)
    return out


def _pack(index, dense, bra_sizes, ket_sizes):
    """Dense boundary -> the stored cohorts of `index`, laid out as the engine's allocation."""
    off, total = _offsets(index)
    out = torch.zeros(total, dtype=torch.float64, device=_DEVICE)
    ob, ok = np.cumsum([0] + list(bra_sizes)), np.cumsum([0] + list(ket_sizes))
    for ci in range(index.n_cohorts):
        if index.tr[ci]:
            continue
        i, j = int(index.bra_pos[ci]), int(index.ket_pos[ci])
        n = bra_sizes[i] * ket_sizes[j]
        for b in range(index.aux_dim):
            o = int(index.offsets[ci, b])
            if o >= 0 and n:
                out[off[ci] + o:off[ci] + o + n] = dense[b, ob[i]:ob[i + 1], ok[j]:ok[j + 1]].t().reshape(-1)
    return out
