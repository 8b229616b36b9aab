"""Routes of the matrix-core gather and scatter that small uniform node sets do not reach, against the oracle
(GPU): the FP64 gather at m = 3 (light tiles only), a tile cut into several work items and slots whose nodes start
in both halves of axis 2, nodes that moved in place since their windows were tabulated, and the vector and
LDS-atomic kernels that serve calls without the matrix cores.

Both sides sum the same O((2m+1)^3) products in another order.  FP64 rel-l2 stays below 1e-12 (about 1e-15 times
the growth of the window factors), FP32 below the 1e-5 of the other FP32 comparisons with the oracle.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

if __name__ == "__main__":
    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import pnfft_amd as PA
from pnfft_amd.device import DevicePlan
from pnfft_amd.workloads import SplitMix64

pytestmark = pytest.mark.gpu

TOL = {"double": 1e-12, "float": 1e-5}
WINDOWS = {"kb": PA.PNFFT_WINDOW_KAISER_BESSEL, "gauss": PA.PNFFT_WINDOW_GAUSSIAN,
           "bspline": PA.PNFFT_WINDOW_BSPLINE, "sinc": PA.PNFFT_WINDOW_SINC_POWER}
F, G = PA.PNFFT_COMPUTE_F, PA.PNFFT_COMPUTE_GRAD_F
TABLES = PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI


def rel(a, b):
    a, b = np.asarray(a).reshape(-1), np.asarray(b).reshape(-1)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def tile_size(m, precision):
    """Cells per axis of a tile: 8, or 4 where the padded subgrid of 8 would be too large."""
    return 8 if m <= 4 or (m <= 6 and precision == "double") else 4


def torus(x, precision):
    """x wrapped to [-1/2, 1/2) and rounded to the plan's precision."""
    x = x - np.floor(x + 0.5)
    if precision == "float":
        x = x.astype(np.float32).astype(np.float64)
    x[x >= 0.5] = -0.5
    return np.ascontiguousarray(x)


def tile_counts(dp):
    """Nodes per nonempty tile, from the bin keys (tile-major)."""
    keys = dp.node_bins()[1].cpu().numpy().view(np.uint32)
    return np.unique(keys // tile_size(dp.m, dp.precision) ** 3, return_counts=True)[1]


def cluster(n, m, ts, count, rng):
    """count nodes whose stencils start in the tile of the cells ts .. 2 ts - 1 on every axis."""
    start = ts + ts * rng.uniform(3 * count).reshape(count, 3)
    return (start + m) / np.array(n)


def coefficients(N, c2r, rng):
    if not c2r:
        return rng.complex_normal(int(np.prod(N))).reshape(N)
    fh = rng.complex_normal(N[0] * N[1] * (N[2] // 2 + 1)).reshape(N[0], N[1], -1)
    fh[0], fh[:, 0], fh[:, :, 0] = 0, 0, 0  # Nyquist planes
    return fh


def check_all(oracle, dp, P, x, fh, fv, gv, tol):
    """Every mode of trafo, x-VJP and adj at the positions x (already on the device)."""
    import torch
    f_o, g_o = (P.trafo_c2r if P.c2r else P.trafo)(x, fh, compute_grad=True)
    adj = P.adj_c2r if P.c2r else P.adj
    a_f, a_g = (np.asarray(adj(x, f=fv)).reshape(-1), np.asarray(adj(x, grad=gv)).reshape(-1))
    dp.set_f_hat(fh)
    for flags in (F, G, F | G):
        dp.trafo(flags)
        assert dp.api.last_error() is None
        if flags & F:
            assert rel(dp.f.cpu().numpy(), f_o) < tol, flags
        if flags & G:
            assert rel(dp.grad.cpu().numpy(), g_o) < tol, flags
    gx = dp.grad_x_vjp(torch.as_tensor(fv, device="cuda:0")).cpu().numpy()
    assert rel(gx, (np.conj(fv)[:, None] * np.asarray(g_o).reshape(len(x), 3)).real) < tol
    dp.set_f(fv)
    dp.set_grad(gv)
    for flags, ref in ((F, a_f), (G, a_g), (F | G, a_f + a_g)):
        dp.adj(flags)
        assert dp.api.last_error() is None
        assert rel(dp.f_hat.cpu().numpy(), ref) < tol, flags


def values(k, c2r, rng):
    return rng.normal(k) if c2r else rng.complex_normal(k)


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("heavy", [False, True])
def test_fp64_gather_m3_light_tiles(gpu, oracle, c2r, heavy):
    """FP64 at m = 3 takes the matrix cores where tiles are light: 70000 nodes over the 4096 tiles of n = 128^3,
    tiles of up to three nodes among them (a corner left nearly empty), with and without one of more than the 512
    nodes of a work item."""
    import torch
    print("case mm64 m3", c2r, heavy, flush=True)
    rng = SplitMix64(8100 + c2r)
    N, n, m = (64, 64, 64), (128, 128, 128), 3
    x = rng.uniform(3 * 80000).reshape(80000, 3) - 0.5
    inside = np.all((x > -0.4) & (x < -0.1), axis=1)
    x = np.concatenate([x[~inside], x[inside][:40], cluster(n, m, 8, 700 if heavy else 250, rng)])
    x = torus(x, "double")
    M = len(x)
    fh = coefficients(N, c2r, rng)
    w = values(M, c2r, rng)
    dp = DevicePlan(N, n, m, 0, M, c2r=c2r)
    dp.set_x(x)
    counts = tile_counts(dp)
    assert M >= 65536 and M / np.sum((counts + 511) // 512) < 150 and (counts.max() > 512) == heavy
    assert all(np.any(counts == k) for k in (1, 2, 3))
    # the nodes to compare: light and heavy regions
    some = np.concatenate([np.arange(0, 2000, 5), np.arange(M - (740 if heavy else 290), M)])
    f_o, g_o = (lambda P: (P.trafo_c2r if c2r else P.trafo)(x[some], fh, compute_grad=True))(
        oracle.Plan(N, n, m, 0, c2r=c2r))
    vjp = (np.conj(w[some])[:, None] * np.asarray(g_o).reshape(-1, 3)).real
    dp.set_f_hat(fh)
    for tables in (False, True):
        if tables:
            dp.precompute(TABLES)
        for flags in (F, G, F | G):
            dp.f.zero_()
            dp.grad.zero_()
            dp.trafo(flags)
            assert dp.api.last_error() is None
            if flags & F:
                assert rel(dp.f.cpu().numpy()[some], f_o) < 1e-12
            if flags & G:
                assert rel(dp.grad.cpu().numpy()[some], g_o) < 1e-12
        gx = dp.grad_x_vjp(torch.as_tensor(w, device="cuda:0")).cpu().numpy()
        assert rel(gx[some], vjp) < 1e-12
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("m", [5, 6])
def test_fp64_scatter_light_tiles(gpu, oracle, m, c2r):
    """More than 1024 tiles of a few nodes each, one of 200 beside them: the adjoint of f in FP64 at m = 5, 6 has a
    variant for one block per CU there."""
    print("case light scatter", m, c2r, flush=True)
    rng = SplitMix64(8500 + m)
    N, n = (64, 64, 64), (128, 128, 128)
    x = torus(np.concatenate([rng.uniform(3 * 4000).reshape(4000, 3) - 0.5, cluster(n, m, 8, 200, rng)]), "double")
    M = len(x)
    fv = values(M, c2r, rng)
    dp = DevicePlan(N, n, m, 0, M, c2r=c2r)
    dp.set_x(x)
    counts = tile_counts(dp)
    assert len(counts) >= 1024 and M < 64 * len(counts) and counts.max() >= 200
    dp.set_f(fv)
    P = oracle.Plan(N, n, m, 0, c2r=c2r)
    ref = (P.adj_c2r if c2r else P.adj)(x, f=fv)
    for tables in (False, True):
        if tables:
            dp.precompute(TABLES)
        dp.adj(F)
        assert dp.api.last_error() is None
        assert rel(dp.f_hat.cpu().numpy(), ref) < 1e-12
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("precision,m", [("double", m) for m in (2, 3, 4, 5, 6)] + [("float", m) for m in range(2, 9)])
def test_cut_tile(gpu, oracle, precision, m, c2r):
    """3001 nodes that start in one tile, all over its cells (both halves of axis 2 and nearly empty ends of its
    parts): its work items, order entries and slots."""
    print("case cut tile", precision, m, c2r, flush=True)
    rng = SplitMix64(8200 + m)
    N, n = (16, 16, 16), (32, 32, 32)
    x = np.concatenate([cluster(n, m, tile_size(m, precision), 3001, rng), rng.uniform(3 * 150).reshape(150, 3) - 0.5])
    x = torus(x, precision)
    M = len(x)
    flags = WINDOWS["kb" if m < 8 else "gauss"]
    dp = DevicePlan(N, n, m, flags, M, precision=precision, c2r=c2r)
    dp.set_x(x)
    assert tile_counts(dp).max() > 2900  # more than a part, a slot and a work item hold
    check_all(oracle, dp, oracle.Plan(N, n, m, flags, c2r=c2r), x, coefficients(N, c2r, rng), values(M, c2r, rng),
              values(3 * M, c2r, rng), TOL[precision])
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("wname", list(WINDOWS))
@pytest.mark.parametrize("precision,m", [("double", 2), ("double", 3), ("double", 5), ("double", 6), ("float", 7),
                                         ("float", 8)])
def test_moved_nodes(gpu, oracle, precision, m, wname, c2r):
    """Positions that changed in place since precompute_psi, in every window: by less than a cell, to the other half
    of the tile along axis 2, to another tile, and not at all; the kernels evaluate the windows of those that
    moved."""
    import torch
    print("case moved", precision, m, wname, c2r, flush=True)
    rng = SplitMix64(8300 + m)
    N, n = (16, 16, 16), (32, 32, 32)
    ts = tile_size(m, precision)
    x = torus(np.concatenate([cluster(n, m, ts, 400, rng), rng.uniform(3 * 403).reshape(403, 3) - 0.5]), precision)
    M = len(x)
    x2 = x.copy()
    x2[0::4] += (rng.uniform(3 * len(x2[0::4])).reshape(-1, 3) - 0.5) / np.array(n)
    x2[1::4, 2] += (ts / 2) / n[2]
    x2[2::4] = rng.uniform(3 * len(x2[2::4])).reshape(-1, 3) - 0.5
    x2 = torus(x2, precision)
    flags = WINDOWS[wname]
    dp = DevicePlan(N, n, m, flags, M, precision=precision, c2r=c2r)
    P = oracle.Plan(N, n, m, flags, c2r=c2r)
    dp.set_x(x)
    dp.precompute(TABLES)
    dp.x.copy_(torch.as_tensor(x2).to(dp.x.dtype))
    torch.cuda.synchronize()
    check_all(oracle, dp, P, x2, coefficients(N, c2r, rng), values(M, c2r, rng), values(3 * M, c2r, rng),
              TOL[precision])
    dp.close()


@pytest.mark.parametrize("m,n,per", [(3, 64, 3), (3, 64, 18), (3, 128, 16), (3, 64, 160), (5, 64, 160), (5, 64, 300), (5, 64, 600),
                                     (5, 32, 1562)])
def test_fp64_gather_route_by_density(gpu, oracle, m, n, per):
    """The FP64 gather at m = 3 and its gradients at m = 5 run on the matrix cores or on the vector kernel by nodes per
    tile: uniform sets of `per` on both sides of the bounds."""
    import torch
    print("case density", m, n, per, flush=True)
    rng = SplitMix64(8700 + m + per)
    N, nn = (n // 2,) * 3, (n,) * 3
    M = per * (n // 8) ** 3
    x = torus(rng.uniform(3 * M).reshape(M, 3) - 0.5, "double")
    fh, w = coefficients(N, False, rng), values(M, False, rng)
    some = np.arange(0, M, max(1, M // 1000))
    f_o, g_o = oracle.Plan(N, nn, m, 0).trafo(x[some], fh, compute_grad=True)
    vjp = (np.conj(w[some])[:, None] * np.asarray(g_o).reshape(-1, 3)).real
    dp = DevicePlan(N, nn, m, 0, M)
    dp.set_x(x)
    dp.set_f_hat(fh)
    for tables in (False, True):
        if tables:
            dp.precompute(TABLES)
        for flags in (F, G, F | G):
            dp.trafo(flags)
            assert dp.api.last_error() is None
            if flags & F:
                assert rel(dp.f.cpu().numpy()[some], f_o) < 1e-12
            if flags & G:
                assert rel(dp.grad.cpu().numpy()[some], g_o) < 1e-12
        gx = dp.grad_x_vjp(torch.as_tensor(w, device="cuda:0")).cpu().numpy()
        assert rel(gx[some], vjp) < 1e-12
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("kind", ["light", "dense", "cut"])
@pytest.mark.parametrize("m", [2, 3, 4])
def test_fp32_vjp_small_m(gpu, oracle, m, kind, c2r):
    """The x-VJP of FP32 plans at m = 2, 3, 4 runs on the matrix cores or on the vector kernel by nodes per tile: about
    one, eight and more, and a tile cut into parts."""
    import torch
    print("case vjp", m, kind, c2r, flush=True)
    rng = SplitMix64(8600 + m)
    N, n = (16, 16, 16), (32, 32, 32)
    x = {"light": lambda: rng.uniform(3 * 60).reshape(60, 3) - 0.5,
         "dense": lambda: rng.uniform(3 * 900).reshape(900, 3) - 0.5,
         "cut": lambda: cluster(n, m, 8, 1500, rng)}[kind]()
    x = torus(x, "float")
    M = len(x)
    fh, w = coefficients(N, c2r, rng), values(M, c2r, rng)
    dp = DevicePlan(N, n, m, 0, M, precision="float", c2r=c2r)
    dp.set_x(x)
    counts = tile_counts(dp)
    assert {"light": M < 3 * len(counts), "dense": M >= 6 * len(counts), "cut": counts.max() > 1024}[kind]
    dp.set_f_hat(fh)
    P = oracle.Plan(N, n, m, 0, c2r=c2r)
    g_o = np.asarray((P.trafo_c2r if c2r else P.trafo)(x, fh, compute_grad=True)[1]).reshape(M, 3)
    for tables in (False, True):
        if tables:
            dp.precompute(TABLES)
        gx = dp.grad_x_vjp(torch.as_tensor(w, device="cuda:0")).cpu().numpy()
        assert dp.api.last_error() is None
        assert rel(gx, (np.conj(w)[:, None] * g_o).real) < 1e-5
    dp.close()


def fallback_cases():
    """The kernels in use under the environment's switches, on a cut tile beside tiles of a few nodes."""
    from oracle import oracle
    oracle.lib()
    for precision, ms in (("double", range(2, 8)), ("float", range(2, 9))):
        for m in ms:
            for c2r in (False, True):
                if c2r and precision == "double" and m > 6:
                    continue  # rejected plans
                print("case fallback", precision, m, c2r, flush=True)
                rng = SplitMix64(8400 + m)
                N, n = (16, 16, 16), (32, 32, 32)
                x = torus(np.concatenate([cluster(n, m, tile_size(m, precision), 1301, rng),
                                          rng.uniform(3 * 90).reshape(90, 3) - 0.5]), precision)
                M = len(x)
                flags = WINDOWS["kb" if m < 8 else "gauss"]
                dp = DevicePlan(N, n, m, flags, M, precision=precision, c2r=c2r)
                dp.set_x(x)
                check_all(oracle, dp, oracle.Plan(N, n, m, flags, c2r=c2r), x, coefficients(N, c2r, rng),
                          values(M, c2r, rng), values(3 * M, c2r, rng), TOL[precision])
                dp.close()


@pytest.mark.parametrize("scatter", ["column", "atomic"])
def test_kernels_without_matrix_cores(gpu, oracle, scatter):
    """PNFFT_AMD_MFMA=0 (read once per process): the kernels that serve calls without memory for window tables, with
    the column scatter and with the LDS-atomic one."""
    env = dict(os.environ, PNFFT_AMD_MFMA="0", PNFFT_AMD_SCATTER=scatter)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], env=env, capture_output=True, text=True,
                       timeout=100)
    print(r.stdout[-2000:], flush=True)
    assert r.returncode == 0, r.stderr[-3000:]


if __name__ == "__main__":
    fallback_cases()
