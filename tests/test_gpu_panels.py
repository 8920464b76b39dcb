"""GPU parity of the pair-panel sigma (pair_panels.hip, ngemm_kernel.hpp) at the
sizes where its tiles and K-ranges end: against the oracle, and against the
gathered pair terms (TCI_DENSE_PAIRS=0) that accept every layout; with panels
over the domains and with wide ones (TCI_DENSE_PAIRS=2).  Odd and even virtual spaces, domains on both sides of 64, 128, 192 and 256, explicit
one-electron parts, FP32 L^J, both ladders, tuned and fixed schedules, graph
replays; the host-vector htimesc around its slot length.

Tolerances (relative 2-norm): FP64 1e-10, bf16x3 5e-5, fp16x3 2e-6 as in the
other sigma tests; two FP64 routes of one plan 1e-12 (summation order only)."""
import contextlib
import os
import sys
import threading

import numpy as np
import pytest

import tigerci_amd as tci
from oracle.problem import make_problem, random_ci_vector
from oracle.sigma import Integrals, sigma as oracle_sigma
from tigerci_amd.synthetic import make_synthetic, random_vector

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-10, "bf16x3": 5e-5, "fp16x3": 2e-6}


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
    os.environ.update(kv)
    try:
        yield
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


CASES = [
    dict(n_int=1, n_v=2, n_chol=3, seed=301),
    dict(n_int=2, n_v=1, n_chol=2, seed=302),
    dict(n_int=3, n_v=65, n_chol=37, seed=303),
    dict(n_int=5, n_v=33, n_chol=40, seed=304, domain_range=(2, 33), weak_below=9, h_offdiag=0.2),
    dict(n_int=17, n_v=9, n_chol=21, seed=305, domain_range=(1, 9), h_offdiag=0.1),
    dict(n_int=3, n_v=129, n_chol=24, seed=306, h_offdiag=0.1),
    dict(n_int=3, n_v=260, n_chol=13, seed=307, domain_range=(190, 260)),
    dict(n_int=4, n_v=200, n_chol=18, seed=308, domain_range=(60, 200), weak_below=70),
]
ENVS = [{}, {"TCI_AUTOTUNE": "0"}, {"TCI_LADDER_VV": "0"}, {"TCI_LADDER_VV": "1", "TCI_AUTOTUNE": "0"},
        {"TCI_DENSE_PAIRS": "2"}, {"TCI_DENSE_PAIRS": "2", "TCI_LADDER_VV": "0", "TCI_AUTOTUNE": "0"}]


@pytest.mark.parametrize("env", ENVS, ids=lambda e: ",".join(e) or "tuned")
@pytest.mark.parametrize("args", CASES, ids=lambda a: "{n_int}x{n_v}x{n_chol}".format(**a))
def test_panels_match_oracle_and_gathered_terms(args, env):
    _say("case: pair panels", args, env)
    prob = make_problem(**args)
    ints = Integrals(prob)
    x = random_ci_vector(prob, 21)
    ref = oracle_sigma(prob, x, ints)
    with _env(**{**env, "TCI_DENSE_PAIRS": "0"}):
        gathered = _sigma(tci.Plan.from_problem(prob), x)
    with _env(**env):
        plan = tci.Plan.from_problem(prob)
        for precision in ("fp64", "bf16x3", "fp16x3", "fp64"):
            y = _sigma(plan, x, precision=precision)
            _say(f"  {precision} rel err {_rel(y, ref):.2e}")
            assert _rel(y, ref) < TOL[precision]
            if precision == "fp64":
                assert _rel(y, gathered) < 1e-12
            # replays with eager builds between them
            for _ in range(3):
                assert np.array_equal(_sigma(plan, x, precision=precision, graph=True), y)
                assert np.array_equal(_sigma(plan, x, precision=precision), y)
        if args["n_v"] < 100:
            f32 = tci.Plan.from_problem(prob, ladder_dtype="f32")
            assert _rel(_sigma(f32, x), ref) < 1e-6  # L^J rounded to FP32: 24 bits
            assert _rel(_sigma(f32, x, precision="bf16x3"), ref) < TOL["bf16x3"]


def test_wide_panels_where_the_others_do_not_fit():
    """60 internal orbitals with 168 full virtuals: panels over the domains would
    take 75 GB, the plan takes the wide ones; against the gathered products."""
    _say("case: wide panels at 60x168x24")
    syn = make_synthetic(60, 168, 24, 309)
    with _env(TCI_DENSE_PAIRS="0", TCI_LADDER_VV="1"):
        plan = tci.Plan.from_problem(syn)
        x = random_vector(plan.n_csf, 7)
        ref = _sigma(plan, x)
        del plan
    with _env(TCI_LADDER_VV="1"):
        plan = tci.Plan.from_problem(syn)
        assert "wide pair panels" in plan.tuning()
        y = _sigma(plan, x)
        z = _sigma(plan, x, precision="bf16x3")
    _say(f"  fp64 {_rel(y, ref):.2e} bf16x3 {_rel(z, ref):.2e}")
    assert _rel(y, ref) < 1e-12 and _rel(z, ref) < TOL["bf16x3"]


@pytest.mark.parametrize("n_int,n_v", [(2, 5), (3, 174), (9, 81)])
def test_host_htimesc_pieces(n_int, n_v):
    """Vectors below one 65,536-element slot, just above one, and longer than
    the ring of four: sigmavec + H civec + E_ref civec as the device call forms
    it, bit for bit; then two threads on one plan."""
    prob = make_problem(n_int, n_v, 8, 310 + n_int)
    plan = tci.Plan.from_problem(prob)
    n = plan.n_csf
    _say("case: htimesc pieces", n_int, n_v, "CSFs", n)
    xs = [random_ci_vector(prob, 31 + k) for k in range(2)]
    base = np.random.default_rng(5).standard_normal(n)
    want = []
    for x in xs:
        c, out = tci.DeviceArray.from_numpy(x), tci.DeviceArray.from_numpy(base)
        plan.sigma(c, out, accumulate=True, add_eref=True)
        want.append(out.numpy())
        got = base.copy()
        tci.htimesc(x, got, plan)
        assert np.array_equal(got, want[-1])
    outs = [base.copy(), base.copy()]
    threads = [threading.Thread(target=tci.htimesc, args=(xs[k], outs[k], plan)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert np.array_equal(outs[k], want[k])
