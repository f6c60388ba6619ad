"""GPU: a mechanism that the lane-group tables cannot hold (mech/LiDryer_order4.yaml, n = 10) runs the
work queue with FP64 factors, ReactorRK64 and the adjoint with one cell per lane, and the cooperative
model with the data tables' kinetics, against the oracle. Gates as in the parity tests: 1e-3 K and
1e-8 in Y; gradients 1e-5 relative."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from pelec_amd import inputs, mechanism as M  # noqa: E402
from pelec_amd.reactor import Eos, Reactor  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
MECH = "LiDryer_order4"
GATE_T = 1e-3
GATE_Y = 1e-8
W = inputs.WORKLOADS["lidryer_32"]


def to_dev(a, dtype=torch.float64):
    return torch.tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


@pytest.fixture(scope="module")
def case(oracle_lib):
    """2000 cells, a fifth of them masked, with radicals enough for the order-four reaction to
    carry a share of the heat release; the oracle's end states with and without it."""
    n = 2000
    d = inputs.make_inputs(W.name, n)
    m = M.load(MECH)
    rY = d["rY"].copy()
    rho = rY.sum(0)
    for s, f in (("H", 1e-3), ("OH", 1e-2)):
        rY[m.species_index(s)] += f * rho
    om = oracle_lib.OracleMech(m)
    e = np.array([om.thermo(T)[1] - 1.0 for T in d["T"]]).T * 8.31446261815324e7 * d["T"]
    d = {"rY": rY, "T": d["T"], "rE": (rY * e / np.array(m.weights)[:, None]).sum(0),
         "mask": (inputs.uniform(17, 0, np.arange(n)) >= 0.2).astype(np.int32)}
    kw = dict(rtol=W.rtol, atol=W.atol, mask=d["mask"], nthreads=8)
    ref = om.react(d["rY"], d["T"], d["rE"], W.dt, **kw)
    other = oracle_lib.OracleMech(M.load("LiDryer")).react(d["rY"], d["T"], d["rE"], W.dt, **kw)
    assert np.abs(ref["T"] - other["T"]).max() > 1.0  # the reaction counts
    return om, d, ref


def check(out, ref, d):
    on = d["mask"] == 1
    assert np.abs(out["T"] - ref["T"])[on].max() <= GATE_T
    assert (np.abs(out["rY"] - ref["rY"]) / ref["rY"].sum(0))[:, on].max() <= GATE_Y
    for k in ("rY", "T", "rE"):
        np.testing.assert_array_equal(out[k][..., ~on], d[k][..., ~on])


def react(d, dt=W.dt, kind="ReactorCvode", noalloc=False, params=(), **cfg):
    r = Reactor(MECH, kind)
    r.configure(rtol=W.rtol, atol=W.atol, **cfg)
    for k, v in params:
        r.set_param(k, v)
    a = {k: to_dev(d[k]) for k in ("rY", "T", "rE")}
    call = r.react_flat_noalloc if noalloc else r.react_flat
    print(f"[gpu-test] {MECH} {kind} noalloc={noalloc} {cfg} {params}", flush=True)
    call(a["rY"], a["T"], a["rE"], dt, mask=to_dev(d["mask"], torch.int32))
    torch.cuda.synchronize()
    assert r.last_failures() == 0
    out = {k: v.cpu().numpy() for k, v in a.items()}
    if cfg.get("kernel_timing"):
        out["ms"], _ = r.kernel_times()
    r.close()
    return out


@pytest.mark.parametrize("kw", [{}, {"cooperative": 0}, {"cooperative": 3}, {"max_slots": 64},
                                {"noalloc": True}, {"lu_fp32": True}], ids=str)
def test_queue_with_fp64_factors(kw, case):
    om, d, ref = case
    check(react(d, form="batched", **dict(dict(lu_fp32=False), **kw)), ref, d)


def test_the_queue_is_what_ran(case):
    om, d, ref = case
    out = react(d, form="batched", lu_fp32=False, kernel_timing=True)
    assert all(v > 0.0 for v in out["ms"].values()), out["ms"]
    check(out, ref, d)


def test_compactions_do_not_change_a_cell(case):
    """6000 cells: the queue compacts only above 4096 slots in use."""
    om, d, ref = case
    d = {k: np.tile(v, 3) for k, v in d.items()}
    outs = [react(d, form="batched", lu_fp32=False, cooperative=0,
                  params=(("prc.compact_pct", 90), ("prc.compact_every", every)))
            for every in (0, 3)]
    for k in ("rY", "T", "rE"):
        np.testing.assert_array_equal(outs[1][k], outs[0][k])
    check(outs[1], {k: np.tile(ref[k], 3) for k in ("rY", "T")}, d)


def test_rk64(case):
    om, d, _ = case
    ref = om.react_rk64(d["rY"], d["T"], d["rE"], W.dt, rtol=W.rtol, atol=W.atol, mask=d["mask"],
                        nthreads=8)
    assert ref["nfail"] == 0
    check(react(d, kind="ReactorRK64"), ref, d)


@pytest.mark.parametrize("cooperative", [False, True])
def test_model(cooperative, case):
    om, d, _ = case
    nc = 65
    y = np.vstack([d["rY"][:, :nc], d["T"][None, :nc]])
    f, J = Eos(MECH).model(0.0, to_dev(y), to_dev(d["rE"][:nc]), cooperative=cooperative)
    f, J = f.cpu().numpy(), J.cpu().numpy()
    for c in range(nc):
        fr, _ = om.rhs(0.0, y[:, c], d["rE"][c])
        Jr = om.jac(0.0, y[:, c], d["rE"][c])
        assert np.abs(f[:-1, c] - fr[:-1]).max() <= 1e-9 * np.abs(fr[:-1]).max()
        rows = np.abs(Jr).max(1, keepdims=True)
        assert (np.abs(J[c] - Jr) <= 1e-8 * np.where(rows == 0.0, 1.0, rows)).all()


def test_adjoint(case):
    """Against the tangent-linear replay of the device's tape, along rho e0 and a few species and
    rate constants (the order-four reaction's among them)."""
    om, d, _ = case
    m, n = M.load(MECH), 3
    rng = np.random.default_rng(2)
    x = {k: d[k][..., :n] for k in ("rY", "T", "rE")}
    ct, cT = rng.normal(size=x["rY"].shape) / x["rY"].sum(0), rng.normal(size=n) / 1000.0
    r = Reactor(MECH)
    r.configure(rtol=1e-6, atol=W.atol)
    print(f"[gpu-test] {MECH} adjoint", flush=True)
    out = r.adjoint(*(to_dev(x[k]) for k in ("rY", "T", "rE")), W.dt, ct_rY=to_dev(ct),
                    ct_T=to_dev(cT), tape_cap=2048)
    torch.cuda.synchronize()
    out = {k: v.cpu().numpy() for k, v in out.items()}
    r.close()
    assert (out["status"] == 0).all()

    def along(c, dy, de, dla):
        tape = out["tape"][c, :out["tape_count"][c]]
        y0 = np.concatenate([x["rY"][:, c], [x["T"][c]]])
        _, _, dye, dTe = om.replay(tape, y0, x["rE"][c], W.dt, tangent=(dy, de, dla))
        return ct[:, c] @ dye[:-1] + cT[c] * dTe

    z, zl = np.zeros(m.nsp + 1), np.zeros(m.nrxn)
    for c in range(n):
        t = along(c, z, 1.0, zl)
        assert abs(out["g_rE0"][c] - t) <= 1e-5 * abs(t)
        for k in (0, 1, m.species_index("H"), m.species_index("OH")):
            t = along(c, np.eye(m.nsp + 1)[k], 0.0, zl)
            assert abs(out["g_rY0"][k, c] - t) <= 1e-5 * abs(t), (c, k)
        ts = np.array([along(c, z, 0.0, np.eye(m.nrxn)[j]) for j in range(m.nrxn)])
        assert (np.abs(out["g_logA"][:, c] - ts) <= 1e-5 * np.abs(ts) + 1e-9 * np.abs(ts).max()).all()
