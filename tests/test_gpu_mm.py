"""Matrix-core gather and scatter (FP64; FP32 at m = 7, 8; FP32 gather at m <= 6) against the oracle
at the sizes where their tiling can go wrong (GPU).

A tile holds 8^3 cells and its padded subgrid 8 + 2m per axis (12 to 20: below, at and past the sixteen
rows of a product, with 2 or 4 rows left over); nodes are taken in groups of 16, work items in chunks of
512 nodes, and items of at most three nodes take the per-node path.  Both sides sum the same
O((2m+1)^3) products in FP64 in different orders on coefficients of size 1, so the rel-l2 of f, grad_f
stays below 1e-12 (about 1e-15 times the growth of the window factors).
"""
import numpy as np
import pytest

import pnfft_amd as PA
from pnfft_amd.device import DevicePlan
from pnfft_amd.workloads import SplitMix64

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel(a, b):
    a, b = np.asarray(a).reshape(-1), np.asarray(b).reshape(-1)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def node_set(kind, rng, n):
    h = 1.0 / np.array(n)
    if kind == "few":  # tiles of one to four nodes, some alone
        x = rng.uniform(3 * 70).reshape(70, 3) - 0.5
    elif kind == "tile":  # one tile's worth of cells, 513 + 40 nodes: two items, ragged groups
        x = (np.array([8, 8, 8]) + 8 * rng.uniform(3 * 553).reshape(553, 3)) * h - 0.5
    elif kind == "corner":  # around the wrap of every axis, and exactly on cell borders
        x = (rng.uniform(3 * 300).reshape(300, 3) - 0.5) * 6 * h + 0.5
        x[:40] = np.round(x[:40] / h) * h
    else:  # one cell run along each axis: groups whose offsets reach a single row, plane or K-block
        x = np.concatenate([np.stack([np.where(t == k, 8 * u, 3.5) for k in range(3)], 1)
                            for t, u in ((t, rng.uniform(37)) for t in range(3))]) * h
    x = x - np.floor(x + 0.5)
    x[x >= 0.5] = -0.5
    return np.ascontiguousarray(x)


@pytest.mark.parametrize("kind", ["few", "tile", "corner", "lines"])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("tables", [False, True])
def test_gather_matches_oracle(gpu, oracle, kind, m, tables):
    print("case mm64 gather", kind, m, tables, flush=True)
    rng = SplitMix64(1000 + 10 * m + len(kind))
    N, n = (8, 16, 12), (16, 32, 32)
    x = node_set(kind, rng, n)
    M = len(x)
    fh = rng.complex_normal(int(np.prod(N)))
    w = rng.complex_normal(M)
    dp = DevicePlan(N, n, m, 0, M)
    dp.set_x(x)
    dp.set_f_hat(fh)
    if tables:
        dp.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
    dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
    both = dp.f.cpu().numpy().copy(), dp.grad.cpu().numpy().copy()
    dp.trafo(PA.PNFFT_COMPUTE_F)
    f = dp.f.cpu().numpy().copy()
    dp.trafo(PA.PNFFT_COMPUTE_GRAD_F)
    g = dp.grad.cpu().numpy().copy()
    import torch
    gx = dp.grad_x_vjp(torch.as_tensor(w, device="cuda:0")).cpu().numpy()
    assert dp.api.last_error() is None
    dp.close()
    f_o, g_o = oracle.Plan(N, n, m, 0).trafo(x, fh, compute_grad=True)
    assert rel(f, f_o) < TOL and rel(both[0], f_o) < TOL
    assert rel(g, g_o) < TOL and rel(both[1], g_o) < TOL
    assert rel(gx, (np.conj(w)[:, None] * np.asarray(g_o).reshape(M, 3)).real) < TOL


@pytest.mark.parametrize("kind", ["few", "tile", "corner"])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6])
def test_gather_real_grid_matches_oracle(gpu, oracle, kind, m):
    print("case mm64 gather c2r", kind, m, flush=True)
    rng = SplitMix64(2000 + 10 * m + len(kind))
    N, n = (8, 16, 12), (16, 32, 32)
    x = node_set(kind, rng, n)
    M = len(x)
    fh = rng.complex_normal(8 * 16 * 7).reshape(8, 16, 7)
    fh[0], fh[:, 0], fh[:, :, 0] = 0, 0, 0  # Nyquist planes
    dp = DevicePlan(N, n, m, 0, M, c2r=True)
    dp.set_x(x)
    dp.set_f_hat(fh)
    dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
    assert dp.api.last_error() is None
    f, g = dp.f.cpu().numpy().copy(), dp.grad.cpu().numpy().copy()
    dp.close()
    f_o, g_o = oracle.Plan(N, n, m, 0, c2r=True).trafo_c2r(x, fh, compute_grad=True)
    assert rel(f, f_o) < TOL and rel(g, g_o) < TOL


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("kind", ["few", "tile", "corner", "lines"])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6])
def test_scatter_matches_oracle(gpu, oracle, kind, m, c2r):
    """adj of f, of grad_f and of both, without tables and with them (the two phases of m = 5, 6 with
    one of them empty: "lines" along axes 0 and 1)."""
    print("case mm64 scatter", kind, m, c2r, flush=True)
    rng = SplitMix64(3000 + 10 * m + len(kind))
    N, n = (8, 16, 12), (16, 32, 32)
    x = node_set(kind, rng, n)
    if kind == "lines":
        x = x[:74]
    M = len(x)
    fv = rng.normal(M) if c2r else rng.complex_normal(M)
    gv = rng.normal(3 * M) if c2r else rng.complex_normal(3 * M)
    P = oracle.Plan(N, n, m, 0, c2r=c2r)
    adj = P.adj_c2r if c2r else P.adj
    refs = [np.asarray(adj(x, f=fv)).reshape(-1), np.asarray(adj(x, grad=gv)).reshape(-1)]
    refs.append(refs[0] + refs[1])
    dp = DevicePlan(N, n, m, 0, M, c2r=c2r)
    dp.set_x(x)
    dp.set_f(fv)
    dp.set_grad(gv)
    for tables in (False, True):
        if tables:
            dp.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
        for flags, ref in zip((PA.PNFFT_COMPUTE_F, PA.PNFFT_COMPUTE_GRAD_F,
                               PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F), refs):
            dp.adj(flags)
            assert dp.api.last_error() is None
            assert rel(dp.f_hat.cpu().numpy(), ref) < TOL, (flags, tables)
    dp.close()


@pytest.mark.parametrize("precision,tol", [("double", TOL), ("float", 1e-5)])
@pytest.mark.parametrize("m", [4, 6, 8])
def test_tile_of_several_slots(gpu, oracle, precision, tol, m):
    """More nodes in one tile than a block takes: it is scattered into several slots and gathered by several
    blocks (m = 8: tiles of 4 cells, the vector kernels); adj repeats bit for bit.  The oracle sums the
    same terms; FP32 at 1e-5 as for the other FP32 comparisons with it."""
    print("case several slots", precision, m, flush=True)
    rng = SplitMix64(4000 + m)
    N, n = (16, 16, 16), (32, 32, 32)
    x = (rng.uniform(3 * 7001).reshape(7001, 3) * 3.9 + 4.05) / 32 - 0.25  # 7001 nodes in one tile ...
    x = np.concatenate([x, rng.uniform(3 * 500).reshape(500, 3) - 0.5])     # ... and some everywhere
    if precision == "float":
        x = x.astype(np.float32).astype(np.float64)
    M = len(x)
    fh, fv = rng.complex_normal(16 ** 3), rng.complex_normal(M)
    dp = DevicePlan(N, n, m, PA.PNFFT_WINDOW_GAUSSIAN, M, precision=precision)
    dp.set_x(x)
    dp.set_f_hat(fh)
    dp.trafo(PA.PNFFT_COMPUTE_F)
    f = dp.f.cpu().numpy().copy()
    dp.set_f(fv)
    out = []
    for _ in range(2):
        dp.adj(PA.PNFFT_COMPUTE_F)
        out.append(dp.f_hat.cpu().numpy().copy())
    assert dp.api.last_error() is None
    dp.close()
    P = oracle.Plan(N, n, m, PA.PNFFT_WINDOW_GAUSSIAN)
    assert rel(f, P.trafo(x, fh)[0]) < tol
    assert rel(out[0], P.adj(x, f=fv)) < tol
    if precision == "float" or m <= 6:  # (FP64 m = 8 scatters by atomics)
        assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("kind", ["few", "tile", "corner", "lines"])
@pytest.mark.parametrize("m,wname", [(7, "bspline"), (8, "gauss"), (7, "kb")])
def test_fp32_wide_windows_match_oracle(gpu, oracle, kind, m, wname, c2r):
    """FP32 at m = 7, 8 (tiles of 4 cells, subgrids of 18 and 20 rows): trafo, gradient, x-VJP and adj of
    both, at the 1e-5 of the other FP32 comparisons with the oracle."""
    import torch
    print("case fp32 wide", kind, m, wname, c2r, flush=True)
    rng = SplitMix64(5000 + 10 * m + len(kind))
    flags = {"kb": 0, "gauss": PA.PNFFT_WINDOW_GAUSSIAN, "bspline": PA.PNFFT_WINDOW_BSPLINE}[wname]
    N, n = (8, 16, 12), (16, 32, 32) if m == 7 else (32, 32, 32)
    x = node_set(kind, rng, n).astype(np.float32).astype(np.float64)
    M = len(x)
    fh = rng.complex_normal(8 * 16 * (7 if c2r else 12)).reshape(8, 16, -1)
    if c2r:
        fh[0], fh[:, 0], fh[:, :, 0] = 0, 0, 0  # Nyquist planes
    fv = rng.normal(M) if c2r else rng.complex_normal(M)
    gv = rng.normal(3 * M) if c2r else rng.complex_normal(3 * M)
    P = oracle.Plan(N, n, m, flags, c2r=c2r)
    f_o, g_o = (P.trafo_c2r if c2r else P.trafo)(x, fh, compute_grad=True)
    adj = P.adj_c2r if c2r else P.adj
    a_o = np.asarray(adj(x, f=fv)).reshape(-1)
    ag_o = np.asarray(adj(x, grad=gv)).reshape(-1)
    dp = DevicePlan(N, n, m, flags, M, precision="float", c2r=c2r)
    dp.set_x(x)
    for tables in (False, True):
        if tables:
            dp.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
        dp.set_f_hat(fh)
        dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        assert rel(dp.f.cpu().numpy(), f_o) < 1e-5 and rel(dp.grad.cpu().numpy(), g_o) < 1e-5
        dp.trafo(PA.PNFFT_COMPUTE_F)
        assert rel(dp.f.cpu().numpy(), f_o) < 1e-5
        gx = dp.grad_x_vjp(torch.as_tensor(fv, device="cuda:0")).cpu().numpy()
        assert rel(gx, (np.conj(fv)[:, None] * np.asarray(g_o).reshape(M, 3)).real) < 1e-5
        dp.set_f(fv)
        dp.set_grad(gv)
        dp.adj(PA.PNFFT_COMPUTE_F)
        assert rel(dp.f_hat.cpu().numpy(), a_o) < 1e-5
        dp.adj(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        assert rel(dp.f_hat.cpu().numpy(), a_o + ag_o) < 1e-5
        assert dp.api.last_error() is None
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("kind", ["few", "tile", "corner", "lines"])
@pytest.mark.parametrize("m,wname", [(3, "kb"), (4, "gauss"), (5, "kb"), (5, "bspline"), (6, "gauss"), (6, "bspline")])
def test_fp32_gather_matches_oracle(gpu, oracle, kind, m, wname, c2r):
    """FP32 gather at m <= 6: f, gradient, both and x-VJP on tiles of one node, of two groups and of more,
    at the 1e-5 of the other FP32 comparisons with the oracle; the magnitude of the coefficients leaves
    the relative error alone."""
    import torch
    print("case fp32 gather", kind, m, wname, c2r, flush=True)
    rng = SplitMix64(6000 + 10 * m + len(kind))
    flags = {"kb": 0, "gauss": PA.PNFFT_WINDOW_GAUSSIAN, "bspline": PA.PNFFT_WINDOW_BSPLINE}[wname]
    N, n = (8, 16, 12), (16, 32, 32)
    x = node_set(kind, rng, n).astype(np.float32).astype(np.float64)
    x[x >= 0.5] = -0.5
    M = len(x)
    fh = rng.complex_normal(8 * 16 * (7 if c2r else 12)).reshape(8, 16, -1)
    if c2r:
        fh[0], fh[:, 0], fh[:, :, 0] = 0, 0, 0  # Nyquist planes
    fv = rng.normal(M) if c2r else rng.complex_normal(M)
    P = oracle.Plan(N, n, m, flags, c2r=c2r)
    f_o, g_o = (P.trafo_c2r if c2r else P.trafo)(x, fh, compute_grad=True)
    dp = DevicePlan(N, n, m, flags, M, precision="float", c2r=c2r)
    dp.set_x(x)
    for tables, scale in ((False, 1.0), (True, 1.0), (True, 2.0 ** -80), (True, 2.0 ** 80)):
        if tables:
            dp.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
        dp.set_f_hat(fh * scale)
        dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        f, g = dp.f.cpu().numpy() / scale, dp.grad.cpu().numpy() / scale
        assert rel(f, f_o) < 1e-5 and rel(g, g_o) < 1e-5
        dp.trafo(PA.PNFFT_COMPUTE_GRAD_F)
        assert np.array_equal(dp.grad.cpu().numpy() / scale, g)
        dp.trafo(PA.PNFFT_COMPUTE_F)
        assert rel(dp.f.cpu().numpy() / scale, f_o) < 1e-5
        gx = dp.grad_x_vjp(torch.as_tensor(fv, device="cuda:0")).cpu().numpy() / scale
        assert rel(gx, (np.conj(fv)[:, None] * np.asarray(g_o).reshape(M, 3)).real) < 1e-5
        assert dp.api.last_error() is None
    dp.close()


@pytest.mark.parametrize("c2r", [False, True])
@pytest.mark.parametrize("large", ["f", "gx"])
@pytest.mark.parametrize("m,wname", [(7, "kb"), (8, "gauss")])
def test_fp32_wide_scatter_keeps_small_terms(gpu, oracle, m, wname, large, c2r):
    """Pairs of nodes at one place whose large values cancel: what is left of the adjoint is the small ones'.
    The terms of a node (f; d/dx; d/dy and d/dz) are added in FP64, so each keeps its own FP32 accuracy, the 1e-5
    of the other FP32 comparisons; a sum of a large and a small one in FP32 loses 2^-24 of the large (here 2^18
    times the small, n times its derivative: 2^-24 2^18 / 32 = 5e-4 of the result)."""
    print("case small terms", m, wname, large, c2r, flush=True)
    rng = SplitMix64(7000 + m)
    flags = {"kb": 0, "gauss": PA.PNFFT_WINDOW_GAUSSIAN}[wname]
    N, n = (16, 16, 16), (32, 32, 32)
    x = (rng.uniform(3 * 301).reshape(301, 3) - 0.5).astype(np.float32).astype(np.float64)
    x[x >= 0.5] = -0.5
    x = np.repeat(x, 2, axis=0)
    M = len(x)

    def values(k):
        v = rng.normal(k) if c2r else rng.complex_normal(k)
        return v.astype(np.float32 if c2r else np.complex64).astype(v.dtype)

    big = np.repeat(values(M // 2), 2) * np.tile([1.0, -1.0], M // 2)
    f, g = np.zeros_like(big), values(3 * M).reshape(M, 3) * 2.0 ** -18
    if large == "f":
        f = big
    else:
        g[:, 0] = big
    small = g.copy()
    if large == "gx":
        small[:, 0] = 0
    P = oracle.Plan(N, n, m, flags, c2r=c2r)
    ref = np.asarray((P.adj_c2r if c2r else P.adj)(x, grad=small.reshape(-1))).reshape(-1)
    dp = DevicePlan(N, n, m, flags, M, precision="float", c2r=c2r)
    dp.set_x(x)
    dp.set_f(f)
    dp.set_grad(g)
    for cf in (PA.PNFFT_COMPUTE_GRAD_F,) * (large == "gx") + (PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F,):
        dp.adj(cf)
        assert dp.api.last_error() is None
        assert rel(dp.f_hat.cpu().numpy(), ref) < 1e-5, cf
    dp.close()
