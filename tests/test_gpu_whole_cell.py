"""GPU: the kernels that give a lane group a whole cell (batched FP64 form, ReactorRK64, adjoint),
and the launch shape that the FP32-factor queue takes by itself, at the sizes where they can go wrong.

A cell's arithmetic does not depend on its neighbours, on the group or wave that takes it or on how
many cells share the call, so a cell taken out of a larger call has to give the same bits: that is the
tolerance of the size tests (none). The larger calls themselves are held to the oracle here or in the
parity tests.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from pelec_amd import inputs, mechanism as M  # noqa: E402
from pelec_amd.reactor import Reactor  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GATE_T = 1e-3
GATE_Y = 1e-8
#: n = 10 (16 lanes), 22 (32 lanes), 54 (64 lanes) unknowns per cell
WORKLOADS = ["lidryer_32", "drm19_64", "gri30_flat", "dodecane_64"]
NBIG = 200


def to_dev(a, dtype=torch.float64):
    return torch.tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


def react(wl, d, idx, dt=None, rk64=False, noalloc=False, **opts):
    """The cells idx of d in one flat call -> dict of numpy arrays."""
    W = inputs.WORKLOADS[wl]
    r = Reactor(W.mech, chem_integrator="ReactorRK64" if rk64 else "ReactorCvode")
    if not rk64:
        opts = dict(dict(form="batched", lu_fp32=False), **opts)
    shape = {k: opts.pop(k) for k in list(opts) if k.startswith("prc.")}
    r.configure(rtol=W.rtol, atol=W.atol, **opts)
    for k, v in shape.items():
        r.set_param(k, v)
    a = {k: to_dev(d[k][..., idx]) for k in ("rY", "T", "rE")}
    n = len(idx)
    diag = torch.zeros((8, n), dtype=torch.int32, device=DEV)
    r.set_diagnostics(diag)
    src = {k: to_dev(d[k][..., idx]) for k in ("rYsrc", "rEsrc") if k in d}
    mask = to_dev(d["mask"][idx], torch.int32) if "mask" in d else None
    call = r.react_flat_noalloc if noalloc else r.react_flat
    call(a["rY"], a["T"], a["rE"], W.dt if dt is None else dt, mask=mask, **src)
    torch.cuda.synchronize()
    out = {k: v.cpu().numpy() for k, v in a.items()}
    out["diag"] = diag.cpu().numpy()
    out["nfail"] = r.last_failures()
    r.close()
    return out


def same(out, big, idx):
    for k in ("rY", "T", "rE", "diag"):
        np.testing.assert_array_equal(out[k], big[k][..., idx], err_msg=k)


@pytest.fixture(scope="module")
def big():
    """NBIG cells of each workload with sources and a mask (some waves of four, two and one cells
    lose part of their cells, one loses all), in one call."""
    cache = {}

    def get(wl):
        if wl not in cache:
            d = inputs.make_inputs(wl, NBIG)
            rng = np.random.default_rng(31)
            d = dict(d)
            d["rEsrc"] = rng.normal(0, 1e8, NBIG)
            d["rYsrc"] = rng.normal(0, 1e-4, d["rY"].shape) * d["rY"]
            d["mask"] = (rng.uniform(size=NBIG) > 0.2).astype(np.int32)
            d["mask"][64:72] = 0
            cache[wl] = d, react(wl, d, np.arange(NBIG))
        return cache[wl]
    return get


@pytest.mark.parametrize("wl", WORKLOADS)
@pytest.mark.parametrize("first,n", [(0, 1), (3, 2), (64, 8), (1, 63), (60, 65), (7, 193)])
def test_cells_do_not_depend_on_the_call(wl, first, n, big):
    d, ref = big(wl)
    idx = np.arange(first, first + n)
    out = react(wl, d, idx)
    assert out["nfail"] == ref["nfail"] == 0
    same(out, ref, idx)
    off = d["mask"][idx] == 0
    for k in ("rY", "T", "rE"):
        np.testing.assert_array_equal(out[k][..., off], d[k][..., idx[off]])


@pytest.mark.parametrize("wl", WORKLOADS)
@pytest.mark.parametrize("max_slots", [1, 5, 130])
def test_refilled_groups(wl, max_slots, big):
    """Fewer cells in flight than cells in the call: every group takes several cells in turn."""
    d, ref = big(wl)
    idx = np.arange(60 if max_slots == 1 else NBIG)
    same(react(wl, d, idx, max_slots=max_slots), ref, idx)


@pytest.mark.parametrize("wl,n", [("lidryer_32", 12300), ("drm19_64", 6200)])
@pytest.mark.parametrize("max_slots", [1, 2, 3, 0])
def test_max_slots_bounds_the_cells_in_flight(wl, n, max_slots):
    """In a call of more cells than the grid has groups (all but a few masked), where a wave would
    take several cells."""
    W = inputs.WORKLOADS[wl]
    d = inputs.make_inputs(wl, n)
    on = np.arange(0, n, n // 10)
    mask = np.zeros(n, np.int32)
    mask[on] = 1
    r = Reactor(W.mech)
    r.configure(rtol=W.rtol, atol=W.atol, form="batched", lu_fp32=False, max_slots=max_slots)
    a = {k: to_dev(d[k]) for k in ("rY", "T", "rE")}
    r.react_flat(a["rY"], a["T"], a["rE"], W.dt, mask=to_dev(mask, torch.int32))
    torch.cuda.synchronize()
    slots = r.get_param("prc.slots")
    assert r.last_failures() == 0 and 1 <= slots <= (max_slots or n)
    r.close()
    few = react(wl, {k: d[k] for k in a}, on)
    for k in a:
        np.testing.assert_array_equal(a[k].cpu().numpy()[..., on], few[k], err_msg=k)


@pytest.mark.parametrize("wl,sizes", [("lidryer_32", (12289, 1536, 1537, 4609)),
                                      ("drm19_64", (6145, 1025, 3072, 3073, 6144)),
                                      ("gri30_flat", (2049, 1024, 1025, 2048))])
def test_grid_rules(wl, sizes):
    """Calls on both sides of the grid's lines (256 CUs: 1024, 1536, 2048, 3072 waves; 6144 and 12,288
    groups) give the bits of the first, larger one."""
    d = inputs.make_inputs(wl, sizes[0])
    ref = react(wl, d, np.arange(sizes[0]))
    assert ref["nfail"] == 0
    for n in sizes[1:]:
        idx = np.arange(n)
        same(react(wl, d, idx), ref, idx)


@pytest.mark.parametrize("wl", WORKLOADS)
def test_workspace_as_the_memory_allows(wl, big):
    """Workspace refused for more groups than a few waves have: the grid is halved until it fits and
    the cells go in turn; refused for a single wave: PRC_ENOMEM, and the next call is served."""
    d, ref = big(wl)
    W = inputs.WORKLOADS[wl]
    per_wave = 1 if M.load(W.mech).nsp >= 32 else 2 if M.load(W.mech).nsp >= 16 else 4
    r = Reactor(W.mech)
    r.configure(rtol=W.rtol, atol=W.atol, form="batched", lu_fp32=False)
    a = {k: to_dev(d[k]) for k in ("rY", "T", "rE")}
    kw = dict(rYsrc=to_dev(d["rYsrc"]), rEsrc=to_dev(d["rEsrc"]), mask=to_dev(d["mask"], torch.int32))
    if per_wave > 1:
        r.set_param("prc.test_max_groups", per_wave - 1)
        with pytest.raises(Exception, match="ENOMEM"):
            r.react_flat(a["rY"], a["T"], a["rE"], W.dt, **kw)
    for groups in (per_wave, 9 * per_wave):
        r.set_param("prc.test_max_groups", groups)
        for k in a:
            a[k].copy_(to_dev(d[k]))
        r.react_flat(a["rY"], a["T"], a["rE"], W.dt, **kw)
        torch.cuda.synchronize()
        assert r.last_failures() == 0 and 1 <= r.get_param("prc.slots") <= groups
        for k in a:
            np.testing.assert_array_equal(a[k].cpu().numpy(), ref[k], err_msg=k)
    r.close()


@pytest.mark.parametrize("n", [1001, 4096, 4097])
def test_cells_in_order_of_their_rates(n):
    """More cells than groups (prc.max_slots), counted and placed by one and two blocks of the counting
    sort, masked and bad-input cells among them, against the call that has them all in flight."""
    wl = "drm19_64"
    d = dict(inputs.make_inputs(wl, n))
    d["mask"] = (np.random.default_rng(8).uniform(size=n) > 0.5).astype(np.int32)
    d["mask"][700] = 1
    d["T"] = d["T"].copy()
    d["T"][700] = -1.0
    idx = np.arange(n)
    ref = react(wl, d, idx)
    assert ref["nfail"] == 1 and ref["diag"][0][700] != 0
    for noalloc in (False, True):
        out = react(wl, d, idx, max_slots=1000, noalloc=noalloc)
        assert out["nfail"] == 1
        same(out, ref, idx)


def test_noalloc_gives_the_same_cells(big):
    for wl in WORKLOADS[:2]:
        d, ref = big(wl)
        idx = np.arange(NBIG)
        same(react(wl, d, idx, noalloc=True), ref, idx)


@pytest.mark.parametrize("wl", ["lidryer_32", "drm19_64"])
def test_big_call_vs_oracle(wl, big, oracle_lib):
    W = inputs.WORKLOADS[wl]
    d, out = big(wl)
    ref = oracle_lib.OracleMech(M.load(W.mech)).react(
        d["rY"], d["T"], d["rE"], W.dt, rYsrc=d["rYsrc"], rEsrc=d["rEsrc"], mask=d["mask"],
        rtol=W.rtol, atol=W.atol)
    on = d["mask"] == 1
    rho = ref["rY"].sum(0)
    assert np.abs(out["T"] - ref["T"])[on].max() <= GATE_T
    assert (np.abs(out["rY"] - ref["rY"]) / rho)[:, on].max() <= GATE_Y
    np.testing.assert_array_equal(out["rE"][on], (d["rE"] + W.dt * d["rEsrc"])[on])


@pytest.mark.parametrize("wl", WORKLOADS)
def test_singular_newton_matrix(wl):
    """Every inversion reports a singular matrix: ten convergence failures, the inputs kept."""
    n = 67
    d = inputs.make_inputs(wl, n)
    out = react(wl, d, np.arange(n), **{"prc.test_lu_fail": 1})
    assert out["nfail"] == n
    for row, v in ((0, 3), (1, 0), (4, 10), (7, 10)):  # status, steps, set-ups, failures
        np.testing.assert_array_equal(out["diag"][row], v)
    for k in ("rY", "T", "rE"):
        np.testing.assert_array_equal(out[k], d[k])


@pytest.mark.parametrize("wl,dt", [("lidryer_32", None), ("drm19_64", 1e-7), ("gri30_flat", 1e-8)])
def test_rk64_cells_do_not_depend_on_the_call(wl, dt, big):
    d, _ = big(wl)
    ref = react(wl, d, np.arange(NBIG), dt=dt, rk64=True)
    assert ref["nfail"] == 0 and (ref["diag"][1][d["mask"] == 1] > 0).all()
    for first, n in ((0, 1), (2, 3), (64, 8), (1, 63), (60, 65)):
        idx = np.arange(first, first + n)
        same(react(wl, d, idx, dt=dt, rk64=True), ref, idx)


@pytest.mark.parametrize("n", [20480, 20481])
def test_rk64_on_both_sides_of_the_lane_kernels_line(n, oracle_lib):
    """H2/air cells go one per group of lanes up to 20,480 of them, one per lane above."""
    wl = "lidryer_32"
    W = inputs.WORKLOADS[wl]
    d = dict(inputs.make_inputs(wl, n))
    d["mask"] = (np.random.default_rng(3).uniform(size=n) > 0.2).astype(np.int32)
    out = react(wl, d, np.arange(n), rk64=True)
    assert out["nfail"] == 0
    idx = np.r_[0:80, n - 80:n]
    ref = oracle_lib.OracleMech(M.load(W.mech)).react_rk64(
        d["rY"][:, idx], d["T"][idx], d["rE"][idx], W.dt, rtol=W.rtol, atol=W.atol,
        mask=d["mask"][idx], nthreads=8)
    assert np.abs(out["T"][idx] - ref["T"]).max() <= GATE_T
    assert (np.abs(out["rY"][:, idx] - ref["rY"]) / ref["rY"].sum(0)).max() <= GATE_Y
    np.testing.assert_array_equal(out["diag"][1][idx], ref["stats"][:, 0])


def test_rk64_more_lanes_than_a_launch_has(big):
    """2^27 + 5 drm19 cells of 32 lanes each are more than the 2^32 threads of a launch: all but a
    few are masked, at both ends, across the launches' seam and in between."""
    d, _ = big("drm19_64")
    n = 2 ** 27 + 5
    at = torch.tensor([0, 1, 2 ** 25 - 1, 2 ** 25, 2 ** 25 + 1, 2 ** 26 + 7, 2 ** 27 - 1, 2 ** 27,
                       n - 1], device=DEV)
    idx = np.arange(at.numel())
    d = {k: d[k][..., :idx.size] for k in ("rY", "T", "rE")}
    ref = react("drm19_64", d, idx, dt=1e-7, rk64=True)
    W = inputs.WORKLOADS["drm19_64"]
    a = {k: torch.zeros(*d[k].shape[:-1], n, dtype=torch.float64, device=DEV) for k in d}
    for k in a:
        a[k][..., at] = to_dev(d[k])
    mask = torch.zeros(n, dtype=torch.int32, device=DEV)
    mask[at] = 1
    r = Reactor(W.mech, chem_integrator="ReactorRK64")
    r.configure(rtol=W.rtol, atol=W.atol)
    print(f"[gpu-test] rk64 n={n}", flush=True)
    r.react_flat(a["rY"], a["T"], a["rE"], 1e-7, mask=mask)
    torch.cuda.synchronize()
    r.close()
    for k in a:
        np.testing.assert_array_equal(a[k][..., at].cpu().numpy(), ref[k], err_msg=k)
        a[k][..., at] = 0.0
        assert not a[k].any()


@pytest.mark.parametrize("mech,wl", [("LiDryer", "lidryer_32"), ("drm19", "drm19_adj")])
def test_adjoint_cells_do_not_depend_on_the_call(mech, wl):
    W = inputs.WORKLOADS[wl]
    d = inputs.make_inputs(wl, 130)
    rng = np.random.default_rng(5)
    rho = d["rY"].sum(0)
    d = dict(d, ct_rY=rng.normal(size=d["rY"].shape) / rho, ct_T=rng.normal(size=rho.size) / 1000.0,
             rYsrc=rng.normal(0, 1e-4, d["rY"].shape) * d["rY"], rEsrc=rng.normal(0, 1e8, rho.size))
    logA = rng.normal(0, 0.05, M.load(mech).nrxn)

    def go(idx):
        r = Reactor(mech)
        r.configure(rtol=W.rtol, atol=W.atol)
        x = {k: to_dev(d[k][..., idx]) for k in d if k in
             ("rY", "T", "rE", "ct_rY", "ct_T", "rYsrc", "rEsrc")}
        out = r.adjoint(x["rY"], x["T"], x["rE"], W.dt, logA=to_dev(logA), ct_rY=x["ct_rY"],
                        ct_T=x["ct_T"], rYsrc=x["rYsrc"], rEsrc=x["rEsrc"])
        torch.cuda.synchronize()
        res = {k: v.cpu().numpy() for k, v in out.items() if v is not None}
        r.close()
        return res

    ref = go(np.arange(130))
    assert (ref["status"] == 0).all()
    for first, n in ((0, 1), (5, 2), (1, 63), (63, 65)):
        idx = np.arange(first, first + n)
        for k, v in go(idx).items():
            np.testing.assert_array_equal(v, ref[k][..., idx], err_msg=f"{k} {first} {n}")


def test_adjoint_workspace_is_one_share_per_cell():
    """A single cell with many checkpoints (320 MB of them at n = 10) takes one group's share of
    workspace, not that of the four groups of its wave."""
    wl, n, ck = "lidryer_32", 10, 200000
    W = inputs.WORKLOADS[wl]
    d = inputs.make_inputs(wl, 1)
    a = [to_dev(d[k]) for k in ("rY", "T", "rE")]

    def go(r):
        out = r.adjoint(*a, W.dt, ct_rY=torch.ones_like(a[0]), ct_T=torch.ones_like(a[1]))
        torch.cuda.synchronize()
        assert int(out["status"][0]) == 0
        return {k: v.cpu().numpy() for k, v in out.items()}

    r = Reactor(W.mech)
    r.configure(rtol=W.rtol, atol=W.atol)
    ref = go(r)
    free0 = torch.cuda.mem_get_info()[0]
    r.set_param("adj.max_checkpoints", ck)
    out = go(r)
    used = free0 - torch.cuda.mem_get_info()[0]
    r.close()
    share = 8 * ck * ((6 + n) * n + 60)  # a checkpoint: z, the Jacobian, the integrator's scalars
    assert 0.5 * share <= used <= 2.0 * share, (used, share)
    for k in ref:
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


@pytest.mark.parametrize("n", [1, 12288, 12289])
def test_fp32_queue_shape_of_its_own(n, oracle_lib):
    """FP32 factors with neither prc.cooperative nor prc.coop_tail_slots set: H2/air cells run in
    groups from the start up to 12,288 slots, one per lane until that many are left above; both sides
    of the line meet the gate, and an explicit choice stands."""
    wl = "lidryer_32"
    W = inputs.WORKLOADS[wl]
    d = inputs.make_inputs(wl, n)
    ref = oracle_lib.OracleMech(M.load(W.mech)).react(d["rY"], d["T"], d["rE"], W.dt, rtol=W.rtol,
                                                      atol=W.atol)
    rho = ref["rY"].sum(0)
    for kw in ({}, {"cooperative": 0}):
        out = react(wl, d, np.arange(n), lu_fp32=True, **kw)
        assert out["nfail"] == 0
        assert np.abs(out["T"] - ref["T"]).max() <= GATE_T
        assert (np.abs(out["rY"] - ref["rY"]) / rho).max() <= GATE_Y
