"""GPU parity of the ladder from the resident virtual block (ab|cd)
(ladder_vv.hip) against the oracle, and against the Cholesky-direct ladder of
the same plan inputs.  TCI_LADDER_VV=1 forces the resident ladder whenever it
fits (with or without autotuning); TCI_LADDER_VV=0 switches it off."""
import contextlib
import os
import sys

import numpy as np
import pytest

import tigerci_amd as tci
from oracle.problem import make_problem, random_ci_vector
from oracle.sigma import Integrals, sigma as oracle_sigma

pytestmark = pytest.mark.gpu
TOL = 1e-10
SPLIT_TOL = {"bf16x3": 5e-5, "fp16x3": 2e-6}


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _sigma(plan, x, **kw):
    c = tci.DeviceArray.from_numpy(x)
    out = tci.DeviceArray(plan.n_csf)
    plan.sigma(c, out, **kw)
    return out.numpy()


@contextlib.contextmanager
def _env(**kv):
    old = {k: os.environ.get(k) for k in kv}
    os.environ.update({k: str(v) for k, v in kv.items()})
    try:
        yield
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


CASES = [
    dict(n_int=2, n_v=5, n_chol=7, seed=1),
    dict(n_int=4, n_v=37, n_chol=45, seed=2),
    dict(n_int=6, n_v=70, n_chol=50, seed=3, domain_range=(9, 70), weak_below=12),
    dict(n_int=5, n_v=64, n_chol=80, seed=6, domain_range=(20, 64), h_offdiag=0.2),
    dict(n_int=4, n_v=150, n_chol=300, seed=5),
]


@pytest.mark.parametrize("autotune", ["0", "1"])
@pytest.mark.parametrize("args", CASES)
def test_vv_sigma_fp64(args, autotune):
    _say("case: resident ladder fp64", args, "autotune", autotune)
    prob = make_problem(**args)
    ints = Integrals(prob)
    with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=autotune):
        plan = tci.Plan.from_problem(prob)
        assert "fp64 ladder (ab|cd) resident" in plan.tuning() and "-> resident" in plan.tuning()
        for k in range(2):
            x = random_ci_vector(prob, 80 + k)
            assert _rel(_sigma(plan, x), oracle_sigma(prob, x, ints)) < TOL


@pytest.mark.parametrize("precision", ["bf16x3", "fp16x3"])
@pytest.mark.parametrize("args", CASES)
def test_vv_sigma_split(args, precision):
    _say("case: resident ladder", precision, args)
    prob = make_problem(**args)
    ints = Integrals(prob)
    with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=0):
        plan = tci.Plan.from_problem(prob)
        for k in range(2):
            x = random_ci_vector(prob, 90 + k)
            got = _sigma(plan, x, precision=precision)
            assert _rel(got, oracle_sigma(prob, x, ints)) < SPLIT_TOL[precision]
        assert precision + " ladder (ab|cd) resident" in plan.tuning()


def test_vv_matches_cholesky_direct_and_graph_replays():
    """Same inputs, resident and Cholesky-direct ladders: FP64 sigma to 1e-12;
    the resident FP64 and bf16x3 builds replayed from HIP graphs match their
    eager builds over several replays with eager work between them."""
    args = dict(n_int=5, n_v=48, n_chol=70, seed=7, domain_range=(12, 48), weak_below=14)
    _say("case: resident vs Cholesky-direct", args)
    prob = make_problem(**args)
    with _env(TCI_LADDER_VV=0, TCI_AUTOTUNE=0):
        p0 = tci.Plan.from_problem(prob)
        assert "resident" not in p0.tuning()
    with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=0):
        p1 = tci.Plan.from_problem(prob)
        xs = [random_ci_vector(prob, 100 + k) for k in range(3)]
        for x in xs:
            assert _rel(_sigma(p1, x), _sigma(p0, x)) < 1e-12
        for prec in ("fp64", "bf16x3"):
            eager = [_sigma(p1, x, precision=prec) for x in xs]
            for rep in range(3):
                for x, e in zip(xs, eager):
                    g = _sigma(p1, x, precision=prec, graph=True)
                    assert np.array_equal(g, e), (prec, rep)
                _sigma(p1, xs[0], precision=prec)  # eager work between replays


def test_vv_davidson_roots():
    """Davidson roots with the resident ladder (FP64 and mixed) equal those of
    the Cholesky-direct ladder."""
    args = dict(n_int=5, n_v=30, n_chol=40, seed=3)
    _say("case: resident ladder Davidson", args)
    prob = make_problem(**args)
    with _env(TCI_LADDER_VV=0, TCI_AUTOTUNE=0):
        e0, _ = tci.Plan.from_problem(prob).davidson(roots=2, energy_tol=1e-11, norm_tol=1e-8)
    with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=0):
        plan = tci.Plan.from_problem(prob)
        e1, _ = plan.davidson(roots=2, energy_tol=1e-11, norm_tol=1e-8)
        e2, r2 = plan.davidson(roots=2, energy_tol=1e-11, norm_tol=1e-8, precision="bf16x3")
    _say("fp64", e0, "resident", e1, "resident mixed", e2, r2)
    assert r2["converged"]
    assert np.max(np.abs(np.asarray(e1) - np.asarray(e0))) < 1e-9
    assert np.max(np.abs(np.asarray(e2) - np.asarray(e0))) < 1e-6


@pytest.mark.parametrize("schedule", ["128/1", "128/2x", "192/4", "192/1x", "64/1", "32k4/4x", "256/6", "256/1x",
                                      "128x192/2"])
@pytest.mark.parametrize("args", CASES[2:])
def test_vv_product_on_every_tile(args, schedule):
    """The product S = X V on every tile of the NT GEMM, on several K-splits
    (the last one with the 4-internal range behind it) and both workgroup
    orders (TCI_VV_TILE), without and with the autotuner's route: against the
    oracle; the tile is the one that ran."""
    _say("case: resident ladder on", schedule, args)
    tile, ks = schedule.rstrip("x").split("/")
    shape = {"32k4": "32x32,k4"}.get(tile, tile if "x" in tile else f"{tile}x{tile}")
    prob = make_problem(**args)
    ints = Integrals(prob)
    x = random_ci_vector(prob, 110)
    ref = oracle_sigma(prob, x, ints)
    for autotune in "01":
        with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=autotune, TCI_VV_TILE=schedule, TCI_MERGE=0):
            plan = tci.Plan.from_problem(prob)
            plan.profile(True)
            for precision in ("bf16x3", "fp16x3") if tile in ("256", "128x192") else ("fp64", "bf16x3", "fp16x3"):
                y = _sigma(plan, x, precision=precision)
                names = [k["name"] for k in plan.profile_kernels(precision) if "(ab|cd) product" in k["name"]]
                _say(f"  {precision} rel err {_rel(y, ref):.2e} {names}")
                assert _rel(y, ref) < SPLIT_TOL.get(precision, TOL)
                assert len(names) == 1 and shape + ">" in names[0]
                most = min(int(ks), 4 if precision == "fp64" else 8)
                least = max(most, 4) if precision == "fp16x3" else most
                assert (f"K-split {least} " in names[0]) if least > 1 else "K-split" not in names[0]
                assert np.array_equal(_sigma(plan, x, precision=precision, graph=True), y)


@pytest.mark.parametrize("autotune", ["0", "1"])
@pytest.mark.parametrize("first", ["bf16x3", "fp16x3"])
def test_fp16x3_k_splits(first, autotune):
    """fp16x3 keeps its FP32 chains at a quarter of the contraction whichever
    split precision is prepared first and without autotuning: the product that
    ran names at least four K-splits."""
    _say("case: fp16x3 K-splits,", first, "first, autotune", autotune)
    prob = make_problem(4, 60, 70, 12)
    x = random_ci_vector(prob, 5)
    with _env(TCI_LADDER_VV=1, TCI_AUTOTUNE=autotune):
        plan = tci.Plan.from_problem(prob)
        _sigma(plan, x, precision=first)
        plan.profile(True)
        got = _sigma(plan, x, precision="fp16x3")
        names = [k["name"] for k in plan.profile_kernels("fp16x3") if "(ab|cd) product" in k["name"]]
        plan.profile(False)
    _say("  ", names)
    assert len(names) == 1 and any(f"K-split {k} " in names[0] for k in (4, 5, 6, 7, 8))
    assert _rel(got, oracle_sigma(prob, x, Integrals(prob))) < SPLIT_TOL["fp16x3"]
