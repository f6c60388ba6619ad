"""The lane-group tables of the whole-cell kernel (Mech::G_* in pelec_amd/csrc/gen/mech_<name>.h),
evaluated in numpy as whole_cell.h evaluates them, against the CPU oracle: production rates from the
reaction records and the chunked species lists, and the species block of the rate Jacobian from the
schedule of terms (elements dealt to lanes, columns beyond n for the efficiency sets and dq/dT).
Bound: 1e-11 of a row's largest entry (sums of up to ~140 terms in another order than the oracle's,
each rounded to 1.1e-16, amplified by the cancellation within a rate)."""
import ast
import dataclasses
import re

import numpy as np
import pytest

from pelec_amd import inputs, mechanism as M
from pelec_amd import mechgen

MECHS = ("LiDryer", "drm19", "drm19_inert40", "gri30", "dodecane_lu")


def tables(mech):
    return decode(open(mechgen.generate(mech)).read())


def decode(txt):
    out = {"REFC": M.P_ATM / M.R_ERG}
    for m in re.finditer(r"static constexpr (\w+) G_(\w+)((?:\[\d+\])*) = ([^;]+);", txt):
        ctype, name, dims, val = m.groups()
        val = val.strip().replace("ull", "").replace("true", "1").replace("false", "0")
        if not dims:
            out[name] = int(val)
            continue
        a = np.array(ast.literal_eval(val.replace("{", "[").replace("}", "]")),
                     dtype=float if ctype == "double" else np.uint64 if ctype == "uint64_t"
                     else np.int64)
        assert a.shape == tuple(int(d) for d in re.findall(r"\[(\d+)\]", dims)), name
        out[name] = a
    return out


def sgn4(x):
    x = int(x) & 15
    return x - 16 if x > 7 else x


def coefs(tab, b, k):
    return tab[b, :, k, :].ravel()


def evaluate(t, N, C, T):
    """(wdot_k, J_km = dwdot_k/dC_m, dwdot_k/dT) of the species lanes."""
    G, RR = t["W"], t["RR"]
    P, n = G * RR, N + 1
    lnT, iT = np.log(T), 1.0 / T
    E, hR = np.ones(G), np.zeros(G)
    for k in range(N):
        b = 0 if T < t["TMID"][k] else 1
        c, h = coefs(t["G"], b, k), coefs(t["H"], b, k)
        E[k] = np.exp(np.polyval(c[4::-1], T) - c[5] * lnT + c[6] * iT)
        hR[k] = np.polyval(h[4::-1], T) + h[5] * iT
    Cx = np.ones(G)
    Cx[:N] = C
    ns = t["JC"] - n - 1
    Mset = [C.sum() + sum(t["MD"][e, s] * Cx[t["MI"][e, s]] for e in range(t["MN"]))
            for s in range(ns)]
    Q, JV = np.zeros(P + 1), np.zeros(t["NJ"] + 1)
    for p in range(P):
        pk = int(t["RP"][p])
        sl = [pk >> (8 * u) & 255 for u in range(6)]
        eff, kind, rev, dnu = pk >> 48 & 255, pk >> 56 & 3, pk >> 58 & 1, (pk >> 59 & 7) - 2
        A, b = t["RA"][p]
        kf = A * np.exp(b * lnT - t["RE"][p] * iT)
        dlnk, dkdM = (b + t["RE"][p] * iT) * iT, 0.0
        if kind == 1:
            dkdM, kf = kf, kf * Mset[eff]
        elif kind == 2:
            l0, l1, l2 = t["LOW"][:, p]
            k0 = np.exp(l0 + l1 * lnT - l2 * iT)
            Pr = max(k0 * Mset[eff], 1e-300)
            F, g, dF = 1.0, 0.0, 0.0
            if t["TROEK"][p]:
                tr = t["TROE"][:, p]
                dFc = 0.0
                if t["TCONST"]:
                    lF = tr[0]
                else:
                    e3, e1 = np.exp(tr[1] * T), np.exp(tr[3] * T)
                    e2 = np.exp(-tr[4] * iT) if tr[5] else 0.0
                    Fc = tr[0] * e3 + tr[2] * e1 + e2
                    lF = np.log10(Fc)
                    dFc = (tr[6] * e3 + tr[7] * e1 + tr[4] * iT * iT * e2) / Fc
                cc, nn = -0.4 - 0.67 * lF, 0.75 - 1.27 * lF
                xx = np.log10(Pr) + cc
                D = 1.0 / (nn - 0.14 * xx)
                f1 = xx * D
                i1 = 1.0 / (1.0 + f1 * f1)
                F = np.exp(np.log(10.0) * lF * i1)
                g = -lF * 2 * f1 * nn * D * D * i1 * i1
                dF = (i1 - lF * 2 * f1 * ((-0.67 * nn + 1.27 * xx) * D * D) * i1 * i1) * dFc
            dPr = (l1 + l2 * iT) * iT
            dkdM = kf * k0 * F * (1 / (1 + Pr) ** 2 + g / (1 + Pr))
            dlnk += dPr / (1 + Pr) + g * dPr + dF
            kf = kf * Pr / (1 + Pr) * F
        r, q = sl[:3], sl[3:]
        fac = (1.0 / (t["REFC"] * iT)) ** dnu
        iKc = np.prod(E[q]) / np.prod(E[r]) * fac if rev else 0.0
        Pf, Pb = np.prod(Cx[r]), np.prod(Cx[q])
        net = Pf - iKc * Pb
        Q[p] = kf * net
        o = int(t["JD"][p])
        for u in range(6):
            if sl[u] == N:
                continue
            side = r if u < 3 else q
            others = np.prod([Cx[x] for i, x in enumerate(side) if i != u % 3])
            JV[o] = kf * others if u < 3 else -kf * iKc * others
            o += 1
        dlnKc = (hR[q].sum() - hR[r].sum() - dnu) * iT
        JV[t["DT"] + p] = kf * (dlnk * net + iKc * Pb * dlnKc) if rev else kf * dlnk * net
        if kind:
            JV[t["DM"] + p] = dkdM * net
    part = np.zeros(G)
    for i in range(t["L8"]):
        for l in range(G):
            for w in t["GE"][i, l]:
                w = int(w)
                part[l] += sgn4(w >> 12) * Q[(w & 0xfff) // 8]
                part[l] += sgn4(w >> 28) * Q[(w >> 16 & 0xfff) // 8]
    wd = np.array([part[(cp & 255):(cp & 255) + (cp >> 8)].sum() for cp in t["CP"][:N]])
    ws = np.zeros(t["JC"] * G)
    stored = set()
    for l in range(G):
        acc = 0.0
        for i in range(t["JT4"]):
            for e in t["JE"][i, l]:
                e = int(e)
                acc += sgn4(e >> 12) * JV[e & 0xfff]
                if e & 0x10000:
                    assert e >> 17 not in stored  # one lane, once
                    stored.add(e >> 17)
                    ws[e >> 17] = acc
                    acc = 0.0
        assert acc == 0.0
    ws = ws.reshape(t["JC"], G)
    J = ws[:N, :N].T.copy()
    for s in range(ns):
        eff = np.ones(N)
        for e in range(t["MN"]):
            if t["MI"][e, s] < N:
                eff[t["MI"][e, s]] += t["MD"][e, s]
        J += ws[n + s, :N][:, None] * eff[None, :]
    return wd, J, ws[n + ns, :N]


@pytest.mark.parametrize("name", MECHS)
def test_group_tables_against_oracle(name, oracle_lib):
    check(M.load(name), tables(name), oracle_lib)


def check(mech, t, oracle_lib):
    name, om, N = mech.name, oracle_lib.OracleMech(mech), mech.nsp
    assert t["W"] >= N + 1 and t["NJ"] < 4096 and t["JC"] * t["W"] < 1 << 15
    rng = np.random.default_rng(3)
    nu = np.zeros((mech.nrxn, N))
    for j, r in enumerate(mech.reactions):
        for k, v in r.products.items():
            nu[j, k] += v
        for k, v in r.reactants.items():
            nu[j, k] -= v
    for T in (700.0, 999.9, 1650.0, 2600.0):
        C = rng.uniform(0.0, 1.0, N) ** 4 * 1e-6
        wd, J, dT = evaluate(t, N, C, T)
        q, dqdC, dqdT = om.progress(C, T, jac=True)
        ref, Jr, Tr = om.wdot(C, T), nu.T @ dqdC, nu.T @ dqdT
        mag = np.abs(nu.T) @ np.abs(q) + 1e-300
        assert (np.abs(wd - ref) <= 1e-11 * mag).all(), name
        magJ = (np.abs(nu.T) @ np.abs(dqdC)).max(1, keepdims=True) + 1e-300
        assert (np.abs(J - Jr) <= 1e-11 * magJ).all(), name
        assert (np.abs(dT - Tr) <= 1e-10 * (np.abs(nu.T) @ np.abs(dqdT) + 1e-300)).all(), name


def repeated(name, nrxn):
    """The mechanism with its elementary reactions repeated until it has nrxn reactions."""
    m = M.load(name)
    el = [r for r in m.reactions if r.kind == "elementary"]
    more = [el[i % len(el)] for i in range(nrxn - m.nrxn)]
    return dataclasses.replace(m, reactions=m.reactions + more)


def with_reaction(name, **kw):
    m = M.load(name)
    r = dataclasses.replace(next(r for r in m.reactions if r.kind == "elementary"), **kw)
    return dataclasses.replace(m, reactions=m.reactions + [r])


def with_sets(name, nsets):
    """The mechanism with nsets distinct efficiency sets."""
    m = M.load(name)
    r = next(r for r in m.reactions if r.kind == "three-body")
    have = len({tuple(x.efficiencies) for x in m.reactions if x.efficiencies})
    more = [dataclasses.replace(r, efficiencies=[2.0 + i] + r.efficiencies[1:])
            for i in range(nsets - have)]
    return dataclasses.replace(m, reactions=m.reactions + more)


#: on either side of each field's limit: 12-bit byte offsets of the reaction positions (448, 480 and
#: 496 reactions at 64, 32 and 16 lanes), 4-bit net coefficients (of irreversible reactions: the
#: reverse rate allows three species), one efficiency set per lane, three slots per side
LIMITS = {
    "gri30 448": (lambda: repeated("gri30", 448), True),
    "gri30 449": (lambda: repeated("gri30", 449), False),
    "gri30 512": (lambda: repeated("gri30", 512), False),
    "gri30 900": (lambda: repeated("gri30", 900), False),
    "drm19 480": (lambda: repeated("drm19", 480), True),
    "drm19 481": (lambda: repeated("drm19", 481), False),
    "LiDryer 496": (lambda: repeated("LiDryer", 496), True),
    "LiDryer 497": (lambda: repeated("LiDryer", 497), False),
    "LiDryer nu 7": (lambda: with_reaction("LiDryer", reactants={0: 1.0}, products={1: 7.0},
                                           reversible=False), True),
    "LiDryer nu 8": (lambda: with_reaction("LiDryer", reactants={0: 1.0}, products={1: 8.0},
                                           reversible=False), False),
    "LiDryer order 4": (lambda: with_reaction("LiDryer", reactants={0: 2.0, 1: 2.0},
                                              products={2: 2.0}, reversible=False), False),
    "LiDryer 16 sets": (lambda: with_sets("LiDryer", 16), True),
    "LiDryer 17 sets": (lambda: with_sets("LiDryer", 17), False),
}


@pytest.mark.parametrize("case", LIMITS)
def test_field_limits(case, oracle_lib):
    """Mechanisms at the limits of the packed fields get tables that hold, those above get none (and
    a header all the same)."""
    make, fits = LIMITS[case]
    mech = make()
    txt = mechgen.Gen(mech).generate()
    assert f"static constexpr bool G_OK = {'true' if fits else 'false'};" in txt
    if fits:
        check(mech, decode(txt), oracle_lib)
    else:
        assert "G_GE" not in txt and "static constexpr bool T_OK = true;" in txt
