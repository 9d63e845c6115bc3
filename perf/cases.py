"""The work this framework is measured on: two-site H*psi products, bond
truncations and whole DMRG runs, through the public entry points.

Kinds of case
  hpsi_dense  one H*psi of dense operands: the three-stage chain of
              LocalOp::product (psi*L, *W1W2, *R) on plans kept by the
              program, replayed as itx_chain_launch does in a Davidson call
  hpsi_qn     the same product of Sz-conserving block-sparse operands
  bond        svdBond of a two-site tensor (density-matrix or SVD route),
              then the two-site tensor of the truncated pair on every
              flux-allowed block
  dmrg        a whole dmrg() call on a Heisenberg chain
"""
import math

import numpy as np
import torch

from itensor_amd import host as H
from itensor_amd import workloads as W
from itensor_amd.itx import Context


def listed():
    return [
        # the first sweeps of a run and short chains: three launches of almost nothing
        {"name": "hpsi-dense-32", "kind": "hpsi_dense", "chi": 32, "d": 2, "k": 5, "prec": "f64"},
        # a bond dimension that a cutoff left odd
        {"name": "hpsi-dense-255", "kind": "hpsi_dense", "chi": 255, "d": 2, "k": 5, "prec": "f64"},
        # the benchmark's headline product
        {"name": "hpsi-dense-1024", "kind": "hpsi_dense", "chi": 1024, "d": 2, "k": 5, "prec": "f64"},
        # the mixed-precision forms at ordinary dense sizes
        {"name": "hpsi-dense-512-f32", "kind": "hpsi_dense", "chi": 512, "d": 2, "k": 5, "prec": "f32"},
        {"name": "hpsi-dense-768-bf16x3", "kind": "hpsi_dense", "chi": 768, "d": 2, "k": 5, "prec": "bf16x3"},
        # the bond dimension at which the N = 100 chain saturates at cutoff 1e-10
        {"name": "hpsi-qn-110", "kind": "hpsi_qn", "chi": 110, "prec": "f64"},
        # the block-sparse benchmark: 31 Sz sectors
        {"name": "hpsi-qn-1024", "kind": "hpsi_qn", "chi": 1024, "prec": "f64"},
        # truncation of a bond after Davidson: ordinary, large, without quantum numbers
        {"name": "bond-qn-250", "kind": "bond", "chi": 250, "qn": True, "svd": False},
        {"name": "bond-qn-1024", "kind": "bond", "chi": 1024, "qn": True, "svd": False},
        {"name": "bond-dense-150", "kind": "bond", "chi": 150, "qn": False, "svd": False},
        # the accurate route that svdBond takes below cutoff 1e-12 and on request
        {"name": "bond-svd-qn-160", "kind": "bond", "chi": 160, "qn": True, "svd": True},
        # a whole run: ramp, environments, Davidson, truncation, all small
        {"name": "dmrg-32", "kind": "dmrg", "sites": 32, "maxdim": 80, "sweeps": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["hpsi_dense", "hpsi_qn", "bond", "dmrg"], [4, 3, 4, 1])[0]
    if kind == "hpsi_dense":
        # spin-1/2 Heisenberg (d = 2, MPO bond 5) or electrons (d = 4, MPO bond 18)
        d, k = rng.choice([(2, 5), (2, 5), (2, 5), (4, 18)])
        top = 1024 if d == 2 else 330
        return {"kind": kind, "chi": _log_int(rng, 16, top), "d": d, "k": k,
                "prec": rng.choice(["f64", "f64", "f32", "bf16x3"])}
    if kind == "hpsi_qn":
        return {"kind": kind, "chi": _log_int(rng, 24, 1024), "prec": rng.choice(["f64", "f64", "f32", "bf16x3"])}
    if kind == "bond":
        qn, svd = rng.random() < 0.75, rng.random() < 0.25
        top = (200 if qn else 50) if svd else (1024 if qn else 200)
        return {"kind": kind, "chi": _log_int(rng, 16, top), "qn": qn, "svd": svd}
    return {"kind": kind, "sites": rng.randint(8, 32), "maxdim": _log_int(rng, 10, 80), "sweeps": rng.randint(2, 4)}


# ---- one context on torch's stream, kept by the program --------------------
_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(Context(0, torch.cuda.current_stream().cuda_stream))
    return _CTX[0]


class _OnDevice(dict):
    """Results that stay on the device; a tensor's values are copied out when they are looked at."""

    def __getitem__(self, key):
        v = dict.__getitem__(self, key)
        return v.store() if isinstance(v, H.ITensor) else v


# ---- Sz sectors and block layout --------------------------------------------
SITE = [(1, 1), (-1, 1)]           # (2 Sz, dimension)
MPO_LINK = [(0, 3), (-2, 1), (2, 1)]


def _bond_sectors(chi):
    """Sectors of a bond of the Heisenberg chain's middle, weighted as the 31 of the chi = 1024 bond; for a
    smaller bond those without a state are left out."""
    if chi == 1024:
        dims = W.SECTORS_1024
    else:
        dims = [int(round(x * chi / 1024)) for x in W.SECTORS_1024]
    return [(q, d) for q, d in zip(range(-30, 31, 2), dims) if d > 0]


def _layout(legs):
    """Blocks of flux 0 as (sector numbers, dimensions), the last index slowest. A leg is (sectors, sign)."""
    out = []

    def rec(at, num, charge):
        if at < 0:
            if charge == 0:
                out.append((tuple(num), tuple(legs[i][0][n][1] for i, n in enumerate(num))))
            return
        sec, sign = legs[at]
        for n, (q, _) in enumerate(sec):
            rec(at - 1, [n] + num, charge + sign * q)

    rec(len(legs) - 1, [], 0)
    return out


def _starts(sec):
    return np.concatenate([[0], np.cumsum([d for _, d in sec])])


def _to_dense(store, legs):
    """The dense array of a block store, its axes in reversed index order (a column-major tensor's view)."""
    st = [_starts(s) for s, _ in legs]
    full = torch.zeros([int(s[-1]) for s in st][::-1], dtype=torch.float64, device=store.device)
    at = 0
    for num, dims in _layout(legs):
        n = int(np.prod(dims))
        where = tuple(slice(int(st[i][b]), int(st[i][b + 1])) for i, b in reversed(list(enumerate(num))))
        full[where] = store[at:at + n].view(dims[::-1])
        at += n
    return full


def _from_dense(full, legs):
    st = [_starts(s) for s, _ in legs]
    parts = []
    for num, _ in _layout(legs):
        where = tuple(slice(int(st[i][b]), int(st[i][b + 1])) for i, b in reversed(list(enumerate(num))))
        parts.append(full[where].reshape(-1))
    return torch.cat(parts)


def _size(legs):
    return sum(int(np.prod(d)) for _, d in _layout(legs))


def _hpsi_legs(chi):
    b = _bond_sectors(chi)
    return {"phi": [(b, -1), (SITE, 1), (SITE, 1), (b, 1)],
            "L": [(b, 1), (MPO_LINK, 1), (b, -1)],
            "R": [(b, -1), (MPO_LINK, -1), (b, 1)]}


def _normal(n, gen):
    return torch.randn(n, dtype=torch.float64, device="cuda", generator=gen)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


# ---- hpsi_dense ---------------------------------------------------------------
def _dense_inputs(case, seed):
    chi, d, k = case["chi"], case["d"], case["k"]
    g = _generator(seed)
    psi, L, R = _normal(chi * d * d * chi, g), _normal(chi * k * chi, g), _normal(chi * k * chi, g)
    if (d, k) == (2, 5):
        w = torch.from_numpy(W.heisenberg_w()).cuda()  # (h_in, s, s', h_out)
    else:
        w = _normal(k * d * d * k, g).view(k, d, d, k)
    w12 = torch.einsum("hstm,mabk->hstabk", w, w)
    return psi, L, w12.permute(5, 4, 3, 2, 1, 0).contiguous().reshape(-1), R


def _prepare_dense(case, seed):
    chi, d, k = case["chi"], case["d"], case["k"]
    c = _ctx()
    psi, L, w12, R = _dense_inputs(case, seed)
    stages = W.fused_dims(chi, d, k)
    plans = [c.plan_dense(dm[0], lb[0], dm[1], lb[1], dm[2], lb[2], prec=case["prec"])
             for dm, lb in zip(stages, W.FUSED)]
    mid = [torch.empty(int(np.prod(dm[2])), dtype=torch.float64, device="cuda") for dm in stages]
    return {"chain": c.chain(plans), "A": [psi, mid[0], mid[1]], "B": [L, w12, R], "C": mid}


def _exact_dense(case, seed):
    chi, d, k = case["chi"], case["d"], case["k"]
    psi, L, w12, R = _dense_inputs(case, seed)
    return [_hpsi_exact(psi.view(chi, d, d, chi), L.view(chi, k, chi), w12.view(k, d, d, d, d, k), R.view(chi, k, chi))
            .reshape(-1)]


def _hpsi_exact(psi, L, w12, R):
    """All operands with reversed axes: psi[r,s2,s1,l], L[l',h,l], w12[k,s2',s2,s1',s1,h], R[r',k,r]."""
    t = torch.einsum("rbal,mhl->rbamh", psi, L)
    t = torch.einsum("rbamh,kybxah->rmyxk", t, w12)
    return torch.einsum("rmyxk,nkr->nyxm", t, R)


# ---- hpsi_qn --------------------------------------------------------------------
def _index(number, sec, tags):
    return H.Index(number, sum(d for _, d in sec), 1, 0, tags, [([("Sz", q)] if q else [], d) for q, d in sec])


def _hpsi_indices(chi):
    b = _bond_sectors(chi)
    return {"l": _index(7001, b, "Link,l=49"), "r": _index(7002, b, "Link,l=51"),
            "s1": _index(7003, SITE, "Site,n=50"), "s2": _index(7004, SITE, "Site,n=51"),
            "hl": _index(7005, MPO_LINK, "Link,h=49"), "hm": _index(7006, MPO_LINK, "Link,h=50"),
            "hr": _index(7007, MPO_LINK, "Link,h=51")}


def _qn_inputs(case, seed):
    legs = _hpsi_legs(case["chi"])
    g = _generator(seed)
    return legs, {n: _normal(_size(legs[n]), g) for n in ("phi", "L", "R")}


def _labels(Ai, Bi, Ci):
    """The labels of C = A*B: negative ones for the indices that A and B share."""
    la, lb = [0] * len(Ai), [0] * len(Bi)
    n = 0
    for i, a in enumerate(Ai):
        for j, b in enumerate(Bi):
            if a == b:
                n += 1
                la[i] = lb[j] = -n
    for i, c in enumerate(Ci):
        for lab, inds in ((la, Ai), (lb, Bi)):
            for j, x in enumerate(inds):
                if lab[j] >= 0 and x == c:
                    lab[j] = i + 1
    return la, lb, list(range(1, len(Ci) + 1))


def _prepare_qn(case, seed):
    c = _ctx()
    legs, x = _qn_inputs(case, seed)
    i = _hpsi_indices(case["chi"])
    w = np.ascontiguousarray(W.heisenberg_w().transpose(1, 2, 0, 3))
    w1 = H.from_dense([i["s1"].dag(), i["s1"].prime(), i["hl"].dag(), i["hm"]], w)
    w2 = H.from_dense([i["s2"].dag(), i["s2"].prime(), i["hm"].dag(), i["hr"]], w)
    w12 = w1 * w2
    phi = [i["l"].dag(), i["s1"], i["s2"], i["r"]]
    L = [i["l"], i["hl"], i["l"].dag().prime()]
    R = [i["r"].dag(), i["hr"].dag(), i["r"].prime()]
    cur, cur_off = phi, H.block_offsets(phi)[0]
    ops = [(L, H.block_offsets(L)[0]), (w12.inds, w12.offsets), (R, H.block_offsets(R)[0])]
    plans, mid = [], []
    for inds, off in ops:
        t = H.qn_task_list(cur, cur_off, inds, off)
        la, lb, lc = _labels(cur, inds, t["inds"])
        plans.append(c.plan_qn(la, lb, lc, t["offs"], t["bda"], t["bdb"], prec=case["prec"]))
        mid.append(torch.zeros(int(t["csize"]), dtype=torch.float64, device="cuda"))
        cur, cur_off = t["inds"], t["coffs"]
    w12 = torch.from_numpy(np.array(w12.store())).cuda()
    return {"chain": c.chain(plans), "A": [x["phi"], mid[0], mid[1]], "B": [x["L"], w12, x["R"]], "C": mid}


def _exact_qn(case, seed):
    legs, x = _qn_inputs(case, seed)
    w = torch.from_numpy(W.heisenberg_w()).cuda()
    w12 = torch.einsum("hstm,mabk->hstabk", w, w).permute(5, 4, 3, 2, 1, 0)
    full = _hpsi_exact(*(_to_dense(x[n], legs[n]) for n in ("phi", "L")), w12, _to_dense(x["R"], legs["R"]))
    return [_from_dense(full, legs["phi"])]


def _hpsi_qn_flops(chi):
    """Two flops for every product of the three block-sparse contractions."""
    bond = dict(_bond_sectors(chi))
    h = dict(MPO_LINK)
    f = 0
    for r, nr in bond.items():
        for s1 in (1, -1):
            for s2 in (1, -1):
                if r + s1 + s2 in bond:
                    l = r + s1 + s2
                    f += sum(bond[l] * nr * nh * bond[l + q] for q, nh in h.items() if l + q in bond)  # phi*L
        for l, nl in bond.items():  # *R, over the charge that each (l', s1', s2', k) block carries
            for s in (2, 0, 0, -2):
                for q, nh in h.items():
                    if l - s - q == r and l - s in bond:
                        f += nl * nh * nr * bond[l - s]
    return 2.0 * f


# ---- bond -----------------------------------------------------------------------
def _bond_legs(case):
    b = _bond_sectors(case["chi"]) if case["qn"] else [(0, case["chi"])]
    s = SITE if case["qn"] else [(0, 2)]
    return [(b, -1), (s, 1), (s, 1), (b, 1)]


def _bond_phi(case, seed):
    """A normalised two-site tensor whose Schmidt weights fall off over about five decades, as those of a bond
    that is worth truncating do."""
    legs = _bond_legs(case)
    rng = np.random.default_rng(seed)
    parts = []
    for _, dims in _layout(legs):
        x = rng.standard_normal(dims[::-1])  # (r, s2, s1, l)
        fall = [np.exp(-3.0 * (np.arange(n) + 1.0) / (n + 1.0)) for n in (dims[3], dims[0])]
        x = x * fall[0][:, None, None, None] * fall[1][None, None, None, :]
        parts.append(x.ravel())
    x = np.concatenate(parts)
    return legs, x / np.linalg.norm(x)


def _bond_args(case):
    args = {"MaxDim": case["chi"], "MinDim": 1, "Cutoff": 1e-10, "DoNormalize": True}
    if case["svd"]:
        args["UseSVD"] = True
    return args


def _prepare_bond(case, seed):
    legs, x = _bond_phi(case, seed)
    if case["qn"]:
        b = legs[0][0]
        l, r = _index(7101, b, "Link,l=1"), _index(7102, b, "Link,l=3")
        s1, s2 = _index(7103, SITE, "Site,n=2"), _index(7104, SITE, "Site,n=3")
        m = _index(7105, [(q + 1, 1) for q, _ in b], "Link,l=2")
        phi = [l.dag(), s1, s2, r]
        T = H.qdense(phi, H.block_offsets(phi)[0], x)
    else:
        chi = case["chi"]
        l, r = H.Index(7101, chi, 1, 0, "Link,l=1"), H.Index(7102, chi, 1, 0, "Link,l=3")
        s1, s2 = H.Index(7103, 2, 1, 0, "Site,n=2"), H.Index(7104, 2, 1, 0, "Site,n=3")
        m = H.Index(7105, 2, 1, 0, "Link,l=2")
        T = H.dense([l, s1, s2, r], x)
    pair = [H.random_itensor([l.dag(), s1, m], [], 1), H.random_itensor([m.dag(), s2, r], [], 2)]
    return {"pair": pair, "phi": T, "args": _bond_args(case), "wide": T * 0.0}


def _padded(eigs, n):
    out = np.zeros(max(n, len(eigs)))
    out[:len(eigs)] = eigs
    return out


def _run_bond(s):
    A, B, eigs, _ = H.svd_bond(s["pair"], 1, s["phi"], True, s["args"])
    # the pair's two-site tensor on every block of flux 0, as dmrg forms it for the next Davidson call
    return _OnDevice(eigs=_padded(eigs, s["args"]["MaxDim"]), phi=s["wide"] + A * B)


def _kept(P, maxdim, cutoff):
    """How many of the weights P (largest first) svdBond keeps, degenerate ones together; the bounds between."""
    P = np.maximum(P / P[0], 0.0)
    n, err = len(P) - 1, 0.0
    while n >= maxdim:
        err += P[n]
        n -= 1
    while err + P[n] <= cutoff * P.sum() and n >= 1:
        err += P[n]
        n -= 1
    near = 1e-3 * P[n]
    below = above = 0
    while n - below - 1 >= 0 and abs(P[n - below - 1] - P[n]) < near:
        below += 1
    while n + above + 1 < len(P) and abs(P[n + above + 1] - P[n]) < near:
        above += 1
    if below + above == 0:
        return n + 1
    return n - below if maxdim < n + 1 + above else n + 1 + above


def _exact_bond(case, seed):
    legs, x = _bond_phi(case, seed)
    full = _to_dense(torch.from_numpy(x), legs).numpy()  # (r, s2, s1, l)
    bond, site = legs[0][0], legs[1][0]
    ql = np.repeat([q for q, _ in bond], [d for _, d in bond])
    qs = np.repeat([q for q, _ in site], [d for _, d in site])
    nr, ns, _, nl = full.shape
    row = (ql[None, :] - qs[:, None]).reshape(-1)   # charge of (s1, l)
    col = (ql[:, None] + qs[None, :]).reshape(-1)   # charge of (r, s2)
    mat = full.reshape(nr * ns, ns * nl)
    found = []
    for q in sorted(set(row) & set(col)):
        i, j = np.flatnonzero(col == q), np.flatnonzero(row == q)
        u, sv, v = np.linalg.svd(mat[np.ix_(i, j)], full_matrices=False)
        found.append((q, i, j, u, sv, v))
    P = np.sort(np.concatenate([f[4] ** 2 for f in found]))[::-1]
    # the weights that svdBond ranks include the zeros of a side that is longer than the other
    keep = _kept(P, case["chi"], 1e-10)
    least = P[keep - 1]
    out = np.zeros_like(mat)
    for q, i, j, u, sv, v in found:
        n = int(np.sum(sv ** 2 >= least * (1 - 1e-12)))
        out[np.ix_(i, j)] = (u[:, :n] * sv[:n]) @ v[:n]
    out = torch.from_numpy((out / np.linalg.norm(out)).reshape(nr, ns, ns, nl))
    return {"eigs": _padded(P[:keep], case["chi"]), "phi": _from_dense(out, legs)}


# ---- dmrg -----------------------------------------------------------------------
def _prepare_dmrg(case, seed):
    """A Heisenberg chain with bond disorder and the Neel state."""
    n = case["sites"]
    rng = np.random.default_rng(seed)
    sites = H.spin_half_sites(n)
    ampo = H.AutoMPO(sites)
    for i in range(1, n):
        J = float(1.0 + 0.2 * rng.uniform(-1, 1))
        ampo.add(J, "Sz", i, "Sz", i + 1)
        ampo.add(0.5 * J, "S+", i, "S-", i + 1)
        ampo.add(0.5 * J, "S-", i, "S+", i + 1)
    psi, q, prev = [], 0, None
    for i in range(1, n + 1):
        up = i % 2 == 1
        q -= 1 if up else -1
        v = np.array([1.0, 0.0]) if up else np.array([0.0, 1.0])
        inds, shape = [sites(i)], [2]
        if prev is not None:
            inds, shape = [prev.dag()] + inds, [1] + shape
        prev = H.Index(9000 + i, 1, 1, 0, "Link,l=%d" % i, [([("Sz", q)] if q else [], 1)]) if i < n else None
        if prev is not None:
            inds, shape = inds + [prev], shape + [1]
        psi.append(H.from_dense(inds, v.reshape(shape)))
    dims = [max(4, case["maxdim"] >> (case["sweeps"] - 1 - k)) for k in range(case["sweeps"])]
    return {"H": ampo.to_mpo(), "psi": psi, "sweeps": [{"MaxDim": m, "Cutoff": 1e-10, "Niter": 2} for m in dims]}


def _run_dmrg(s):
    energy, steps, _, _ = H.dmrg(s["H"], s["psi"], s["sweeps"], {})
    return {"energy": energy, "steps": np.array([r["energy"] for r in steps])}


# ---- the five functions of a set of cases -----------------------------------------
_PREPARE = {"hpsi_dense": _prepare_dense, "hpsi_qn": _prepare_qn, "bond": _prepare_bond, "dmrg": _prepare_dmrg}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


def run(s):
    if s["kind"] == "bond":
        return _run_bond(s)
    if s["kind"] == "dmrg":
        return _run_dmrg(s)
    s["chain"].launch([t.data_ptr() for t in s["A"]], [t.data_ptr() for t in s["B"]], [t.data_ptr() for t in s["C"]])
    return [s["C"][2]]


def exact(case, seed):
    if case["kind"] == "dmrg":
        return None
    return {"hpsi_dense": _exact_dense, "hpsi_qn": _exact_qn, "bond": _exact_bond}[case["kind"]](case, seed)


def work(case):
    kind = case["kind"]
    if kind == "hpsi_dense":
        chi, d, k = case["chi"], case["d"], case["k"]
        return {"bytes": 8.0 * (2 * chi * chi * d * d + 2 * chi * chi * k + (d * d * k) ** 2),
                "flops": W.hpsi_flops(chi, d, k)}
    if kind == "hpsi_qn":
        legs = _hpsi_legs(case["chi"])
        return {"bytes": 8.0 * (2 * _size(legs["phi"]) + _size(legs["L"]) + _size(legs["R"])),
                "flops": _hpsi_qn_flops(case["chi"])}
    if kind == "bond":
        # density matrix, its tridiagonal form and eigenvectors, projection, product
        legs = _bond_legs(case)
        bond, site = legs[0][0], legs[1][0]
        rows, cols = {}, {}
        for q, d in bond:
            for s, e in site:
                rows[q - s] = rows.get(q - s, 0) + d * e
                cols[q + s] = cols.get(q + s, 0) + d * e
        f = 0.0
        for q in rows:
            m, n = rows[q], cols.get(q, 0)
            if n:
                f += m * m * n + 10.0 / 3.0 * m ** 3 + 4.0 * m * n * (m / 2)
        return {"bytes": 8.0 * 4 * _size(legs), "flops": f}
    # dmrg: three products a step on blocks of about a fifth of the bond dimension, five sectors of them
    n, f, b = case["sites"], 0.0, 0.0
    for k in range(case["sweeps"]):
        top = max(4, case["maxdim"] >> (case["sweeps"] - 1 - k))
        for i in range(1, n):
            chi = min(top, 2 ** min(i, n - i))
            f += 2 * 3 * 80.0 * (chi / 5.0) ** 3 * 5
            b += 2 * 8.0 * (3 * 8 * chi * chi + 10 * chi * chi) / 5.0
    return {"bytes": b, "flops": f}
