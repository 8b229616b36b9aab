"""What the speed of this NFFT is judged by: calls of the public entry points at the sizes, node sets,
precisions and plan options that programs use it with.

Every case is one call sequence (`op`) on a plan and a node set that the program keeps:

  trafo       pnfft_trafo(F) on nodes whose bins and tables were precomputed (fixed sampling pattern)
  trafo_grad  pnfft_trafo(F | GRAD_F) on such nodes
  adj         pnfft_adj(F) on such nodes
  adj_dipole  pnfft_adj(F | GRAD_F) (charges and dipoles), nodes not precomputed
  step        trafo(F), adj(F) of the samples, trafo(GRAD_F): the iteration of an inverse problem and
              the benchmark's step
  particles   one time step of a particle-mesh program: new positions, adj(F) of the charges, the
              coefficients times an influence function, trafo(F | GRAD_F) for potentials and fields;
              with `tables` the program calls pnfft_precompute_psi for the new positions first
  autograd    forward and backward of pnfft_amd.autograd.nfft with new positions and coefficients

`listed()` gives the fixed cases, `draw(rng)` further ones of the same ranges.  `exact` evaluates the
same sums directly (the nonequispaced DFT by its definition) in FP64.
"""
import ctypes
import math

import torch

import pnfft_amd as PA
from pnfft_amd.autograd import nfft
from pnfft_amd.device import DevicePlan

WINDOWS = {"kb": PA.PNFFT_WINDOW_KAISER_BESSEL, "gauss": PA.PNFFT_WINDOW_GAUSSIAN,
           "bspline": PA.PNFFT_WINDOW_BSPLINE, "sinc": PA.PNFFT_WINDOW_SINC_POWER}


def _case(op, precision, N, m, M, nodes="uniform", window="kb", n=None, c2r=False, interlaced=False, ik=False,
          tables=True, name=None):
    n = n or [2 * v for v in N]
    c = dict(op=op, precision=precision, N0=N[0], N1=N[1], N2=N[2], n0=n[0], n1=n[1], n2=n[2], m=m, M=M, nodes=nodes,
             window=window, c2r=c2r, interlaced=interlaced, ik=ik, tables=tables)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest plan in use: one evaluation of a low-order field at a few thousand points (launches, waits)
        _case("trafo", "double", (16, 16, 16), 6, 4096, name="f64_small_trafo"),
        # a small molecular system, particle-mesh with interlacing and ik-differentiation, moving every call
        _case("particles", "double", (32, 32, 32), 4, 20001, c2r=True, interlaced=True, ik=True, tables=False,
              name="f64_small_particles_interlaced_ik"),
        # default accuracy of the interface (m = 6, double precision) on a fixed set of nodes, each direction
        _case("trafo", "double", (128, 128, 128), 6, 1 << 22, name="f64_trafo_128"),
        _case("adj", "double", (128, 128, 128), 6, 1 << 22, name="f64_adj_128"),
        # values and gradients on an anisotropic grid of odd sizes and a clustered, odd number of nodes
        _case("trafo_grad", "double", (101, 60, 90), 5, 1000003, nodes="gaussmix", n=[256, 128, 256],
              name="f64_trafo_grad_ragged"),
        # charges and dipoles onto the grid, once per node set
        _case("adj_dipole", "double", (64, 64, 64), 4, 1 << 19, tables=False, name="f64_adj_dipole_64"),
        # particle-mesh time step of a million charges with the real transforms
        _case("particles", "double", (64, 64, 64), 6, 1 << 20, window="gauss", c2r=True, tables=False,
              name="f64_particles_c2r_64"),
        # the same in single precision with the wide Gaussian window, tabulated once per step
        _case("particles", "float", (64, 64, 64), 8, 1 << 20, window="gauss", c2r=True, name="f32_particles_c2r_m8_64"),
        # small single-precision transform of a ragged number of clustered samples
        _case("adj", "float", (48, 48, 30), 4, 10007, nodes="gaussmix", n=[128, 128, 64], name="f32_small_adj_ragged"),
        # a differentiable NFFT layer: forward, d/dx and d/df_hat on positions that change every call
        _case("autograd", "float", (128, 128, 128), 4, 1 << 21, tables=False, name="f32_autograd_128"),
        # the benchmark's workload
        _case("step", "float", (256, 256, 256), 4, 1 << 24, nodes="gaussmix", name="f32_step_256"),
        # anisotropic grid, B-spline window, nodes crowded into a slab: the largest node set
        _case("step", "float", (256, 256, 64), 6, 1 << 25, nodes="slab", window="bspline", name="f32_step_bspline_slab"),
    ]


def draw(rng):
    def loguni(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["trafo", "trafo_grad", "adj", "adj_dipole", "step", "particles", "particles", "autograd"])
    precision = rng.choice(["double", "float"])
    c2r = op == "particles" and rng.random() < 0.7
    N = [loguni(12, 160) for _ in range(3)]
    if c2r:
        N[2] += N[2] % 2
    n = [1 << (2 * v - 1).bit_length() for v in N]
    window = rng.choice(["kb", "kb", "gauss", "bspline", "sinc"])
    m = rng.choice([3, 4, 4, 5, 6, 6])
    if precision == "float" and window == "gauss" and rng.random() < 0.3:
        m = 8
    interlaced = op == "particles" and rng.random() < 0.3
    ik = op == "particles" and rng.random() < 0.3
    M = loguni(4096, 1 << (21 if precision == "double" else 23))
    return _case(op, precision, N, m, M, nodes=rng.choice(["uniform", "gaussmix", "slab"]), window=window, n=n, c2r=c2r,
                 interlaced=interlaced, ik=ik, tables=op not in ("adj_dipole", "autograd") and rng.random() < 0.6)


# ---------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _shape(case):
    N = [case["N0"], case["N1"], case["N2"]]
    return (N[0], N[1], N[2] // 2 + 1) if case["c2r"] else tuple(N)


def _nodes(kind, M, gen, dev):
    def uni(*s):
        return torch.rand(*s, generator=gen, device=dev, dtype=torch.float64)

    if kind == "uniform":
        x = uni(M, 3) - 0.5
    elif kind == "gaussmix":  # eight Gaussian clusters, wrapped onto the torus
        centers = uni(8, 3) - 0.5
        which = torch.randint(8, (M,), generator=gen, device=dev)
        x = centers[which] + 0.05 * torch.randn(M, 3, generator=gen, device=dev, dtype=torch.float64)
    else:  # half uniform, half in a thin slab around z = 0
        x = uni(M, 3) - 0.5
        x[M // 2:, 2] *= 0.04
    x -= torch.floor(x + 0.5)
    return x


def _inputs(case, seed):
    """x, coefficients, samples, gradient samples and influence function, from the seed alone."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    real = torch.float64 if case["precision"] == "double" else torch.float32
    cplx = torch.complex128 if case["precision"] == "double" else torch.complex64
    M, shape = case["M"], _shape(case)
    x = _nodes(case["nodes"], M, gen, dev).to(real)
    x[x >= 0.5] = -0.5  # a coordinate that rounded up to 1/2

    def cnormal(*s):
        return torch.randn(*s, generator=gen, device=dev, dtype=cplx)

    out = {"x": x}
    op = case["op"]
    if op in ("trafo", "trafo_grad", "step", "autograd"):
        out["f_hat"] = cnormal(*shape)
    if op in ("adj", "adj_dipole", "autograd"):
        out["f"] = cnormal(M)
    if op == "adj_dipole":
        out["grad"] = cnormal(M, 3)
    if op == "particles":
        q = torch.randn(M, generator=gen, device=dev, dtype=real)
        out["f"] = q if case["c2r"] else q.to(cplx)
        # smoothed Coulomb influence function, zero at k = 0 and on the Nyquist planes
        k = _freqs(case, dev)
        k2 = k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2
        w = torch.where(k2 > 0, torch.exp(-k2 / (0.15 * min(case["N0"], case["N1"], case["N2"])) ** 2) / k2.clamp(min=1),
                        torch.zeros_like(k2))
        for t in range(3):
            nt = case["N%d" % t]
            if nt % 2 == 0:
                w[(slice(None),) * t + (k[t] == -(nt // 2),)] = 0
        out["w"] = w.to(real)
    return out


def prepare(case, seed):
    v = _inputs(case, seed)
    flags = WINDOWS[case["window"]]
    flags |= PA.PNFFT_INTERLACED if case["interlaced"] else 0
    flags |= PA.PNFFT_DIFF_IK if case["ik"] else 0
    op = case["op"]
    dp = DevicePlan((case["N0"], case["N1"], case["N2"]), (case["n0"], case["n1"], case["n2"]), case["m"], flags,
                    case["M"], precision=case["precision"], c2r=case["c2r"],
                    alloc_grad=op in ("trafo_grad", "adj_dipole", "step", "particles"))
    s = {"op": op, "plan": dp, "tables": case["tables"], **v}
    if op not in ("particles", "autograd"):
        dp.set_x(v["x"])
        if "f_hat" in v:
            dp.set_f_hat(v["f_hat"])
        if "f" in v:
            dp.set_f(v["f"])
        if "grad" in v:
            dp.set_grad(v["grad"])
        if case["tables"]:
            grad = op in ("trafo_grad", "step")
            dp.precompute(PA.PNFFT_PRE_PSI | (PA.PNFFT_PRE_GRAD_PSI if grad else 0))
    if op == "step":
        s["f_hat_out"] = torch.zeros_like(dp.f_hat)
    if op == "autograd":
        s["x"].requires_grad_(True)
        s["f_hat"].requires_grad_(True)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------
def run(s):
    dp, op = s["plan"], s["op"]
    if op == "trafo":
        dp.trafo(PA.PNFFT_COMPUTE_F)
        return {"f": dp.f}
    if op == "trafo_grad":
        dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        return {"f": dp.f, "grad": dp.grad}
    if op == "adj":
        dp.adj(PA.PNFFT_COMPUTE_F)
        return {"f_hat": dp.f_hat}
    if op == "adj_dipole":
        dp.adj(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        return {"f_hat": dp.f_hat}
    if op == "step":
        a, b = ctypes.c_void_p(dp.f_hat.data_ptr()), ctypes.c_void_p(s["f_hat_out"].data_ptr())
        dp.trafo(PA.PNFFT_COMPUTE_F)
        dp.api.set_f_hat(b, dp.plan)
        dp.adj(PA.PNFFT_COMPUTE_F)
        dp.api.set_f_hat(a, dp.plan)
        dp.trafo(PA.PNFFT_COMPUTE_GRAD_F)
        return {"f": dp.f, "f_hat": s["f_hat_out"], "grad": dp.grad}
    if op == "particles":
        dp.set_x(s["x"])
        if s["tables"]:
            dp.precompute(PA.PNFFT_PRE_PSI | PA.PNFFT_PRE_GRAD_PSI)
        dp.set_f(s["f"])
        dp.adj(PA.PNFFT_COMPUTE_F)
        dp.f_hat.mul_(s["w"])
        dp.trafo(PA.PNFFT_COMPUTE_F | PA.PNFFT_COMPUTE_GRAD_F)
        return {"f_hat": dp.f_hat, "f": dp.f, "grad": dp.grad}
    if op == "autograd":
        f = nfft(s["x"], s["f_hat"], dp)
        gx, gh = torch.autograd.grad(f, (s["x"], s["f_hat"]), s["f"])
        return {"f": f.detach(), "grad_x": gx, "grad_f_hat": gh}
    raise ValueError(op)


# ---------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------
def work(case):
    """Every input read once, every output written once; the oversampled FFT of each transform as
    5 n log2 n flops (half for the real transforms) and the separable stencil sums, 4 flops per stencil
    point for values and 8 for gradients (half for the real transforms)."""
    rs = 8 if case["precision"] == "double" else 4
    cs = 2 * rs
    M, n = case["M"], case["n0"] * case["n1"] * case["n2"]
    nfh = math.prod(_shape(case)) * cs
    half = 0.5 if case["c2r"] else 1.0
    vs = cs * half
    fft = 5.0 * n * math.log2(n) * half
    st = (2 * case["m"] + 1) ** 3 * M * 4.0 * half
    x = 3 * M * rs
    op = case["op"]
    if op in ("trafo", "adj"):
        return {"bytes": x + nfh + M * vs, "flops": fft + st}
    if op == "trafo_grad":
        return {"bytes": x + nfh + 4 * M * vs, "flops": fft + 3 * st}
    if op == "adj_dipole":
        return {"bytes": x + nfh + 4 * M * vs, "flops": fft + 3 * st}
    if op == "step":
        return {"bytes": x + 2 * nfh + 4 * M * vs, "flops": 3 * fft + 4 * st}
    if op == "particles":
        passes = 2 if case["interlaced"] else 1
        flops = passes * ((4 if case["ik"] else 1) * fft + (4 if case["ik"] else 3) * st + fft + st)
        return {"bytes": x + M * vs + nfh * 1.5 + 4 * M * vs, "flops": flops}
    # autograd: x, f_hat and the cotangent in; f and both gradients out
    return {"bytes": 2 * x + 2 * nfh + 2 * M * vs, "flops": 3 * fft + 4 * st}


# ---------------------------------------------------------------------------------------------------
# the sums by their definition, FP64
# ---------------------------------------------------------------------------------------------------
def _freqs(case, dev):
    N = [case["N0"], case["N1"], case["N2"]]
    k = [torch.arange(-(v // 2), v - v // 2, device=dev, dtype=torch.float64) for v in N]
    if case["c2r"]:
        k[2] = torch.arange(-(N[2] // 2), 1, device=dev, dtype=torch.float64)
    return k


def _phases(x, k, sign):
    return [torch.exp(torch.complex(torch.zeros((), dtype=torch.float64, device=x.device),
                                    torch.tensor(sign * 2 * math.pi, dtype=torch.float64, device=x.device))
                      * (x[:, t, None] * k[t][None, :])) for t in range(3)]


def _chunks(M, shape):
    step = max(1, min(M, int(1.5e8 / (shape[1] * shape[2]))))
    return [(a, min(M, a + step)) for a in range(0, M, step)]


def _direct_trafo(case, x, fh, want_grad):
    k, shape = _freqs(case, x.device), _shape(case)
    fh = fh.to(torch.complex128)
    if case["c2r"]:  # each stored coefficient and its conjugate partner, k2 = 0 once
        wt = torch.full((shape[2],), 2.0, dtype=torch.float64, device=x.device)
        wt[-1] = 1.0
        fh = fh * wt
    flat = fh.reshape(shape[0], -1)
    ik = [(-2j * math.pi) * kt for kt in k]
    f, g = [], []
    for a, b in _chunks(len(x), shape):
        E = _phases(x[a:b].double(), k, -1.0)
        T = (E[0] @ flat).reshape(b - a, shape[1], shape[2])
        Tz = (T * E[2][:, None, :]).sum(2)
        v = (Tz * E[1]).sum(1)
        f.append(v.real if case["c2r"] else v)
        if want_grad:
            g1 = (Tz * E[1] * ik[1]).sum(1)
            g2 = ((T * (E[2] * ik[2])[:, None, :]).sum(2) * E[1]).sum(1)
            del T
            T = ((E[0] * ik[0]) @ flat).reshape(b - a, shape[1], shape[2])
            g0 = ((T * E[2][:, None, :]).sum(2) * E[1]).sum(1)
            gg = torch.stack([g0, g1, g2], 1)
            g.append(gg.real if case["c2r"] else gg)
        del T
    return torch.cat(f), torch.cat(g) if want_grad else None


def _direct_adj(case, x, f, grad=None):
    k, shape = _freqs(case, x.device), _shape(case)
    out = torch.zeros((shape[0], shape[1] * shape[2]), dtype=torch.complex128, device=x.device)
    for a, b in _chunks(len(x), shape):
        E = _phases(x[a:b].double(), k, 1.0)
        v = f[a:b].to(torch.complex128)
        if grad is None:
            W = (v[:, None] * E[1])[:, :, None] * E[2][:, None, :]
        else:
            ik = [(2j * math.pi) * kt for kt in k]
            gv = grad[a:b].to(torch.complex128)
            yz = v[:, None] * E[1] + gv[:, 1, None] * (E[1] * ik[1])
            W = yz[:, :, None] * E[2][:, None, :] + (gv[:, 2, None] * E[1])[:, :, None] * (E[2] * ik[2])[:, None, :]
        out += E[0].transpose(0, 1).contiguous() @ W.reshape(b - a, -1)
        if grad is not None:
            W = (gv[:, 0, None] * E[1])[:, :, None] * E[2][:, None, :]
            out += (E[0] * ik[0]).transpose(0, 1).contiguous() @ W.reshape(b - a, -1)
        del W
    return out.reshape(shape)


def exact(case, seed):
    # one complex product of M x (N0 N1 N2) costs 8 flops per entry; the largest cases would take minutes
    passes = {"trafo": 1, "adj": 1, "trafo_grad": 2, "adj_dipole": 2, "step": 4, "particles": 3, "autograd": 4}[case["op"]]
    if 8.0 * case["M"] * math.prod(_shape(case)) * passes > 2.5e14:
        return None
    with torch.no_grad():
        v = _inputs(case, seed)
        op, x = case["op"], v["x"]
        if op == "trafo":
            return {"f": _direct_trafo(case, x, v["f_hat"], False)[0]}
        if op == "trafo_grad":
            f, g = _direct_trafo(case, x, v["f_hat"], True)
            return {"f": f, "grad": g}
        if op == "adj":
            return {"f_hat": _direct_adj(case, x, v["f"])}
        if op == "adj_dipole":
            return {"f_hat": _direct_adj(case, x, v["f"], v["grad"])}
        if op == "step":
            f, g = _direct_trafo(case, x, v["f_hat"], True)
            return {"f": f, "f_hat": _direct_adj(case, x, f), "grad": g}
        if op == "particles":
            fh = _direct_adj(case, x, v["f"]) * v["w"].double()
            f, g = _direct_trafo(case, x, fh, True)
            return {"f_hat": fh, "f": f, "grad": g}
        f, g = _direct_trafo(case, x, v["f_hat"], True)
        gx = (v["f"].to(torch.complex128).conj()[:, None] * g).real
        return {"f": f, "grad_x": gx, "grad_f_hat": _direct_adj(case, x, v["f"])}
