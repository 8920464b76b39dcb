"""GPU parity of the HIP sigma path against the oracle (FP64: <= 1e-10 relative 2-norm)."""
import os
import sys

import numpy as np
import pytest

import tigerci_amd as tci
from oracle.problem import Problem, make_problem, random_ci_vector
from oracle.sigma import Integrals, sigma as oracle_sigma, diagonal as oracle_diagonal

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = 1e-10


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def _gpu_sigma(plan, x, **kw):
    c = tci.DeviceArray.from_numpy(x)
    out = tci.DeviceArray(plan.n_csf)
    plan.sigma(c, out, **kw)
    return out.numpy()


def test_mfma_lane_layouts():
    _say("case: mfma self-test")
    tci.selftest_mfma()


@pytest.mark.parametrize("name", ["full_n3_v12", "local_n4_v30"])
def test_sigma_golden(name):
    _say("case: golden", name)
    z = np.load(os.path.join(ROOT, "tests", "golden", f"{name}.npz"))
    prob = Problem(int(z["n_int"]), int(z["n_v"]), int(z["n_chol"]), z["eps"], z["L"], z["pairs"],
                   z["dom_off"], z["dom_idx"])
    plan = tci.Plan.from_problem(prob)
    for x, s in zip(z["x"], z["sigma"]):
        assert _rel(_gpu_sigma(plan, x), s) < TOL
    assert _rel(plan.diagonal(), z["diag"]) < 1e-12


@pytest.mark.parametrize("args", [
    dict(n_int=2, n_v=5, n_chol=7, seed=1),
    dict(n_int=5, n_v=40, n_chol=60, seed=2),
    dict(n_int=6, n_v=70, n_chol=50, seed=3, domain_range=(10, 70), weak_below=16),
    dict(n_int=3, n_v=300, n_chol=30, seed=4, domain_range=(200, 300)),
])
def test_sigma_random(args):
    _say("case: random", args)
    prob = make_problem(**args)
    ints = Integrals(prob)
    plan = tci.Plan.from_problem(prob)
    assert plan.n_csf == prob.layout().n_csf
    for k in range(2):
        x = random_ci_vector(prob, 50 + k)
        assert _rel(_gpu_sigma(plan, x), oracle_sigma(prob, x, ints)) < TOL


def test_sigma_unit_vectors_and_flags():
    _say("case: unit vectors / flags")
    prob = make_problem(3, 8, 9, 5, domain_range=(3, 8), weak_below=4)
    ints = Integrals(prob)
    plan = tci.Plan.from_problem(prob)
    n = plan.n_csf
    rng = np.random.default_rng(0)
    for k in rng.choice(n, 12, replace=False).tolist() + [0, 1, n - 1]:
        e = np.zeros(n)
        e[k] = 1.0
        ref = oracle_sigma(prob, e, ints)
        assert np.abs(_gpu_sigma(plan, e) - ref).max() < 1e-11 * max(1.0, np.abs(ref).max())
    x = random_ci_vector(prob, 9)
    c = tci.DeviceArray.from_numpy(x)
    base = rng.standard_normal(n)
    out = tci.DeviceArray.from_numpy(base)
    plan.sigma(c, out, accumulate=True, add_eref=True)
    expect = base + oracle_sigma(prob, x, ints) + plan.info.e_ref * x
    assert _rel(out.numpy(), expect) < TOL
    # host htimesc: sigmavec += H civec
    sv = np.ones(n)
    tci.htimesc(x, sv, plan)
    assert _rel(sv, 1.0 + oracle_sigma(prob, x, ints) + plan.info.e_ref * x) < TOL


def test_e_ref_matches_determinant_energy():
    _say("case: e_ref")
    from oracle.problem import reference_energy
    prob = make_problem(4, 6, 10, 8)
    plan = tci.Plan.from_problem(prob)
    assert abs(plan.info.e_ref - reference_energy(prob)) < 1e-10 * abs(reference_energy(prob))


def test_sigma_config1_size():
    """The 10/100/400 full-domain synthetic sigma (500k CSFs), one build."""
    _say("case: n_int=10 n_v=100 n_chol=400")
    prob = make_problem(10, 100, 400, 2024)
    plan = tci.Plan.from_problem(prob)
    x = random_ci_vector(prob, 1)
    ints = Integrals(prob)
    ref = oracle_sigma(prob, x, ints)
    got = _gpu_sigma(plan, x)
    assert _rel(got, ref) < TOL
    # the CPU baseline's sigma (the ladder in C with the reference's loop
    # structure) agrees with the GPU FP64 sigma as well
    from oracle.cpu_sigma import cpu_sigma
    cs = cpu_sigma(prob, x, ints)
    _say(f"  GPU vs oracle {_rel(got, ref):.2e}, GPU vs CPU baseline sigma {_rel(got, cs):.2e}")
    assert _rel(got, cs) < TOL


def test_dense_pair_path_matches_gather_path():
    """Full domains take the pair panels for the ring and 4-internal terms;
    TCI_DENSE_PAIRS=0 forces the per-walk gather GEMMs.
    Both must agree with the oracle (and so with each other)."""
    _say("case: dense pair products vs gather path")
    prob = make_problem(5, 37, 50, 21)
    ints = Integrals(prob)
    x = random_ci_vector(prob, 5)
    ref = oracle_sigma(prob, x, ints)
    dense = tci.Plan.from_problem(prob)
    os.environ["TCI_DENSE_PAIRS"] = "0"
    try:
        gather = tci.Plan.from_problem(prob)
    finally:
        del os.environ["TCI_DENSE_PAIRS"]
    a, b = _gpu_sigma(dense, x), _gpu_sigma(gather, x)
    assert _rel(a, ref) < TOL and _rel(b, ref) < TOL
    am, bm = _gpu_sigma(dense, x, precision="bf16x3"), _gpu_sigma(gather, x, precision="bf16x3")
    assert _rel(am, ref) < 5e-5 and _rel(bm, ref) < 5e-5


@pytest.mark.parametrize("env", [{}, {"TCI_LADDER_MERGED": "0"}, {"TCI_LADDER_MERGED": "0", "TCI_DENSE_PAIRS": "0"}])
def test_full_domain_variants(env):
    """Full domains run the Cholesky-direct split ladder as single products
    over all walks; the per-walk programs (TCI_LADDER_MERGED=0) must give the
    same sigma, including a domain size that is not a multiple of 4 or 8."""
    _say("case: full-domain variants", env)
    env = {"TCI_LADDER_VV": "0", **env}
    for args in [dict(n_int=4, n_v=37, n_chol=30, seed=31), dict(n_int=3, n_v=64, n_chol=20, seed=32)]:
        prob = make_problem(**args)
        ints = Integrals(prob)
        x = random_ci_vector(prob, 6)
        ref = oracle_sigma(prob, x, ints)
        os.environ.update(env)
        try:
            plan = tci.Plan.from_problem(prob)
            assert _rel(_gpu_sigma(plan, x), ref) < TOL
            assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5
        finally:
            for k in env:
                del os.environ[k]


@pytest.mark.parametrize("dense", ["0", "1"])
def test_local_domain_pair_paths(dense):
    """Local domains with weak pairs: the ring, 3-external and 4-internal terms
    as products over packed panels (TCI_DENSE_PAIRS=1) and as per-walk gathered
    programs (=0) both reproduce the oracle."""
    _say("case: local-domain pair paths, TCI_DENSE_PAIRS =", dense)
    prob = make_problem(6, 45, 40, 41, domain_range=(9, 45), weak_below=14)
    ints = Integrals(prob)
    os.environ["TCI_DENSE_PAIRS"] = dense
    try:
        plan = tci.Plan.from_problem(prob)
    finally:
        del os.environ["TCI_DENSE_PAIRS"]
    for k in range(2):
        x = random_ci_vector(prob, 60 + k)
        ref = oracle_sigma(prob, x, ints)
        assert _rel(_gpu_sigma(plan, x), ref) < TOL
        assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5


def test_pair_panels_across_precisions():
    """The panels of one plan through every precision and back, with local
    domains and weak pairs: each against the oracle."""
    _say("case: pair panels across precisions")
    prob = make_problem(6, 45, 40, 43, domain_range=(9, 45), weak_below=14)
    ints = Integrals(prob)
    os.environ["TCI_DENSE_PAIRS"] = "1"
    try:
        plan = tci.Plan.from_problem(prob)
    finally:
        del os.environ["TCI_DENSE_PAIRS"]
    for k in range(2):
        x = random_ci_vector(prob, 64 + k)
        ref = oracle_sigma(prob, x, ints)
        assert _rel(_gpu_sigma(plan, x), ref) < TOL
        assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5
        assert _rel(_gpu_sigma(plan, x, precision="fp16x3"), ref) < 2e-6
        assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5  # back after the switch


@pytest.mark.parametrize("args", [
    dict(n_int=34, n_v=6, n_chol=10, seed=81),
    dict(n_int=34, n_v=8, n_chol=12, seed=83, domain_range=(3, 8), weak_below=2),
    dict(n_int=2, n_v=150, n_chol=20, seed=82),
])
def test_sigma_pair_block_strips(args):
    """The (ia|jb) and (ki|bj) terms of the pair blocks run in 16-row strips
    over 128 columns and 32 internal orbitals at a time: n_int = 34 takes two
    passes over k (also with local domains and weak pairs), d = 150 two
    column passes.  FP64 and bf16x3 against the oracle."""
    _say("case: pair-block strips", args)
    prob = make_problem(**args)
    ints = Integrals(prob)
    plan = tci.Plan.from_problem(prob)
    x = random_ci_vector(prob, 90)
    ref = oracle_sigma(prob, x, ints)
    assert _rel(_gpu_sigma(plan, x), ref) < TOL
    assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5


TILES = {"128": "128x128", "192": "192x192", "64": "64x64", "32k4": "32x32,k4", "256": "256x256", "128x192": "128x192"}


@pytest.mark.parametrize("schedule", ["128/1", "128/4x", "192/2", "64/8", "64/1x", "32k4/4", "256/4", "256/8x",
                                      "128x192/5"])
@pytest.mark.parametrize("args", [
    dict(n_int=6, n_v=45, n_chol=40, seed=47, domain_range=(9, 45), weak_below=14),
    dict(n_int=3, n_v=200, n_chol=33, seed=48, domain_range=(60, 200)),
], ids=["6x45", "3x200"])
def test_pair_panels_on_every_tile(args, schedule):
    """W and the pair products on every tile of the NT GEMM, on several K-splits
    and both workgroup orders (TCI_PANEL_TILE): outputs of less than a tile and
    of a whole and a ragged one.  Every precision against the oracle; the tile
    is the one that ran."""
    _say("case: pair panels on", schedule, args)
    tile = schedule.split("/")[0]
    split_only = tile in ("256", "128x192")
    prob = make_problem(**args)
    ints = Integrals(prob)
    env = {"TCI_DENSE_PAIRS": "1", "TCI_PANEL_TILE": schedule, "TCI_LADDER_VV": "1", "TCI_AUTOTUNE": "0",
           "TCI_MERGE": "0"}
    os.environ.update(env)
    try:
        plan = tci.Plan.from_problem(prob)
        plan.profile(True)
        for precision, tol in (("bf16x3", 5e-5), ("fp16x3", 2e-6)) if split_only else \
                (("fp64", TOL), ("bf16x3", 5e-5), ("fp16x3", 2e-6)):
            x = random_ci_vector(prob, 66)
            err = _rel(_gpu_sigma(plan, x, precision=precision), oracle_sigma(prob, x, ints))
            names = [k["name"] for k in plan.profile_kernels(precision) if "pair product" in k["name"]]
            _say(f"  {precision} rel err {err:.2e} {names}")
            assert err < tol
            assert len(names) == 2 and all(TILES[tile] + ">" in n for n in names)
    finally:
        for k in env:
            del os.environ[k]


@pytest.mark.parametrize("merge", ["64/1", "64/3", "32k4/1", "32k4/8"])
@pytest.mark.parametrize("args", [
    dict(n_int=5, n_v=30, n_chol=40, seed=49),
    dict(n_int=5, n_v=33, n_chol=41, seed=50, domain_range=(5, 33), weak_below=9, h_offdiag=0.2),
    dict(n_int=3, n_v=70, n_chol=20, seed=51),
], ids=["5x30", "5x33", "3x70"])
def test_merged_launches(args, merge):
    """S, W and Y as one launch, the pair products and gW as another
    (TCI_MERGE), against the separate launches (summation order only) and the
    oracle, even and odd n_v; FP32 L^J keeps the singles products apart."""
    _say("case: merged launches", merge, args)
    prob = make_problem(**args)
    x = random_ci_vector(prob, 67)
    ref = oracle_sigma(prob, x, Integrals(prob))
    env = {"TCI_LADDER_VV": "1", "TCI_AUTOTUNE": "0"}
    os.environ.update(env, TCI_MERGE="0")
    try:
        apart = _gpu_sigma(tci.Plan.from_problem(prob), x)
        os.environ["TCI_MERGE"] = merge
        plan = tci.Plan.from_problem(prob)
        f32 = tci.Plan.from_problem(prob, ladder_dtype="f32")
    finally:
        for k in [*env, "TCI_MERGE"]:
            del os.environ[k]
    plan.profile(True)
    y = _gpu_sigma(plan, x)
    names = [k["name"] for k in plan.profile_kernels("fp64")]
    _say(f"  rel err {_rel(y, ref):.2e}, against separate launches {_rel(y, apart):.2e}")
    tile = TILES[merge.split("/")[0]] + ">"
    assert any(n.startswith("fp64 products S, W, Y") and tile in n for n in names)
    assert any("pair products, gW" in n and tile in n for n in names)
    assert _rel(y, ref) < TOL and _rel(y, apart) < 1e-12
    assert np.array_equal(_gpu_sigma(plan, x, graph=True), y)
    assert _rel(_gpu_sigma(f32, x), ref) < 1e-6  # L^J rounded to FP32
    assert _rel(_gpu_sigma(plan, x, precision="bf16x3"), ref) < 5e-5  # the separate programs
