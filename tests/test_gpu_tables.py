"""Window tables that a call fills for itself: their time is part of the call's B stage, and those of
pnfft_precompute_psi are kept and used (GPU)."""
import pytest

import pnfft_amd as PA
from pnfft_amd.device import DevicePlan
from pnfft_amd.workloads import SplitMix64

pytestmark = pytest.mark.gpu

F, G, H = PA.PNFFT_COMPUTE_F, PA.PNFFT_COMPUTE_GRAD_F, PA.PNFFT_COMPUTE_HESSIAN_F
LOOP_B, MATRIX_B = 2, 5  # PNFFT_TIMER_LOOP_B, PNFFT_TIMER_MATRIX_B


def plan(precision, m, flags=0, M=3000):
    rng = SplitMix64(9000 + m)
    dp = DevicePlan((16, 16, 16), (32, 32, 32), m, flags, M, precision=precision)
    dp.set_x(rng.uniform(3 * M).reshape(M, 3) - 0.5)
    dp.set_f_hat(rng.complex_normal(16 ** 3))
    dp.set_f(rng.complex_normal(M))
    dp.set_grad(rng.complex_normal(3 * M))
    return dp


def fills(dp):
    return dp.kernel_times()["tables"][1]


@pytest.mark.parametrize("precision,m", [("double", 4), ("double", 6), ("float", 8)])
def test_tables_are_timed_with_the_b_stage(gpu, precision, m):
    """Evaluating the windows is in PNFFT_TIMER_MATRIX_B and PNFFT_TIMER_LOOP_B, in a table kernel as in the gather:
    the slots hold the table kernel's time and that of the stage's other kernels (beside the gaps between them), up to the
    2^-23 of an event time (FP32) for each of at most four intervals."""
    print("case table timers", precision, m, flush=True)
    dp = plan(precision, m)
    for run, side, kernels in ((dp.trafo, 0, ("gather_tiled", "gather_direct")),
                               (dp.adj, 1, ("scatter_tiled", "scatter_fold", "scatter_direct"))):
        dp.reset_timers()
        run(F)
        kt = dp.kernel_times()
        assert kt["tables"][1] == 1 and kt["tables"][0] > 0
        total = 1e-3 * (kt["tables"][0] + sum(kt[k][0] for k in kernels))
        for slot in (MATRIX_B, LOOP_B):
            assert dp.timers()[side][slot] >= total * (1 - 4 * 2.0 ** -23)
    dp.close()


@pytest.mark.parametrize("precision,m", [("double", 5), ("float", 7)])
def test_derivative_tables_are_kept(gpu, precision, m):
    """After precompute_psi(PRE_PSI) the first gradient makes psi' once; set_x discards it."""
    print("case derivative tables", precision, m, flush=True)
    dp = plan(precision, m)
    dp.precompute(PA.PNFFT_PRE_PSI)
    dp.trafo(F)
    assert fills(dp) == 0
    dp.trafo(G)
    for run in (dp.trafo, dp.adj):
        run(G)
        run(F | G)
        run(F)
    assert fills(dp) == 1
    dp.set_x(dp.x.clone())
    dp.trafo(G)
    assert fills(dp) == 2 and dp.api.last_error() is None
    dp.close()


@pytest.mark.parametrize("precision,m", [("double", 5), ("float", 7)])
@pytest.mark.parametrize("other", ["gauss", "bessel"])
def test_another_plan_leaves_precomputed_tables(gpu, precision, m, other):
    """Two plans of one n and m on one node set: the second, whose window differs (or always comes from
    tables), fills tables for its own calls and leaves those of the first."""
    print("case two plans", precision, m, other, flush=True)
    flags = PA.PNFFT_WINDOW_GAUSSIAN if other == "gauss" else PA.PNFFT_WINDOW_BESSEL_I0
    a, b = plan(precision, m), plan(precision, m, flags)
    a.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
    a.trafo(F | G)
    f, g = a.f.cpu().numpy().copy(), a.grad.cpu().numpy().copy()
    for cf in (F, F | G):
        b.api.trafo(b.plan, a.nodes, cf)
        assert b.api.last_error() is None
    assert fills(b) == 2
    for _ in range(2):
        a.trafo(F | G)
        assert (a.f.cpu().numpy() == f).all() and (a.grad.cpu().numpy() == g).all()
    assert fills(a) == 0
    a.close()
    b.close()


@pytest.mark.parametrize("precision,m", [("double", 4), ("float", 8)])
def test_hessian_fills_no_gather_tables(gpu, precision, m):
    """A call for the Hessian alone evaluates psi, psi' and psi'' in its own kernel: no tables for a gather that
    does not run."""
    print("case hessian alone", precision, m, flush=True)
    dp = plan(precision, m)
    dp.alloc_hessian()
    dp.trafo(H)
    assert dp.api.last_error() is None and fills(dp) == 0
    h = dp.hess.cpu().numpy().copy()
    dp.trafo(F | H)
    assert fills(dp) == 1 and (dp.hess.cpu().numpy() == h).all()
    dp.close()
