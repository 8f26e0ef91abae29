"""The work that programs have this library do, as timed cases.

A case is one operator on one set of points (or several merged ones) and one product with it,
through the package's classes: `init` belongs to what a program keeps (a solver applies one
operator some tens to thousands of times), `mult` is what it repeats.  `helmholtz_apply`, the
differentiable product, builds its operator on every call, so there the whole call is timed.

Points are uniform on the surfaces this library is used and tested on (unit sphere, spheroid
with semi-axes 1, 1, 0.5, torus with R = 1, r = 0.4, sphere with a smooth perturbation) or, for
field evaluation, in a cube around them; densities are complex with N(0, 1) parts.  Programs
that take the mixed form (FP32 arithmetic) hold their vectors in single precision, as
`helmholtz_apply` does for such densities; those of the FP64 form hold them in double.
"""
import math

import numpy as np
import torch

import ifgf_amd
from ifgf_amd.autograd import helmholtz_apply

DEV = "cuda"

# kernel: class of the operator.  k_re, k_im: the wavenumber (real kappa in k_im for the
# Helmholtz and combined-field kernels, which take one real number).  targets: 0 for the sources
# themselves, else that many points in a cube.  tol: -1 takes the orders as they are, else the
# library picks the orders.  io: "host" numpy arrays, "device" torch tensors.
_BASE = dict(kernel="helmholtz", surface="sphere", n=10000, targets=0, k_re=0.0, k_im=10.0, leaf=64,
             order=6, tol=-1.0, precision="mixed", columns=1, parts=1, io="device", graph=False,
             call="mult")


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest problems: a coarse mesh, arrays in and out of host memory; launches and
        # copies are most of the time
        _case("sphere_1k_host", n=1000, k_im=4.0, io="host"),
        # a small problem solved to a tolerance, the product replayed as a graph in an
        # iterative solver
        _case("sphere_10k_tol_graph", n=10000, k_im=10.0, tol=1e-6, graph=True),
        # the large scattering problem at an error below 1e-4
        _case("sphere_1m_tol", n=1048576, k_im=100.0, tol=1e-5),
        # an ordinary size at fixed orders (error about 1e-3): preconditioners, first passes
        _case("sphere_262k", n=262144, k_im=50.0),
        # the FP64 form, for reference solutions
        _case("sphere_100k_fp64_tol", n=99991, k_im=32.0, tol=1e-5, precision="fp64"),
        # many right-hand sides on one geometry: incident directions, block solvers
        _case("spheroid_262k_32col", surface="spheroid", n=262144, k_im=64.0, columns=32),
        # a few right-hand sides to a tolerance
        _case("spheroid_50k_5col_tol", surface="spheroid", n=49999, k_im=24.0, columns=5, tol=1e-4),
        # the combined-field equation on a torus, order 8 and a tolerance
        _case("torus_131k_combined_tol", kernel="combined", surface="torus", n=131072, k_im=40.0,
              order=8, tol=1e-5),
        # a boundary-element program's potential at field points off the surface, modified
        # Helmholtz with a complex wavenumber, host arrays
        _case("spheroid_40k_field_host", kernel="modhelmholtz", surface="spheroid", n=40000,
              targets=30001, k_re=0.5, k_im=-9.0, order=8, io="host"),
        # electrostatics: the Laplace kernel
        _case("sphere_200k_laplace", kernel="laplace", n=200003, k_im=0.0, order=8),
        # several scatterers of uneven sizes as one operator
        _case("spheres_8_merged", n=160000, k_im=24.0, parts=8),
        # shape and density optimisation: a forward and a backward pass
        _case("perturbed_32k_gradients", surface="perturbed", n=32768, k_im=20.0, call="gradients"),
    ]


def _log_size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n | 1 if rng.random() < 0.5 else n


def draw(rng):
    """One more case of the same kinds: sizes log-uniform over 1,000 to 400,000 points, up to 32
    columns, every kernel, surface, form and option above."""
    kind = rng.choice(["plain", "plain", "tol", "tol", "fp64", "columns", "combined", "field",
                       "laplace", "merged", "gradients", "double"])
    surface = rng.choice(["sphere", "spheroid", "torus", "perturbed"])
    io = rng.choice(["host", "device", "device"])
    graph = io == "device" and rng.random() < 0.3

    def kappa(n):  # a few to some tens of points per wavelength, as on the listed problems
        return round(math.sqrt(n) * rng.uniform(0.06, 0.14) + rng.uniform(0, 2), 2)

    tol = rng.choice([1e-3, 1e-4, 1e-5, 3e-5, 1e-6])
    if kind == "plain":
        n = _log_size(rng, 1000, 400000)
        return _case(surface=surface, n=n, k_im=kappa(n), io=io, graph=graph,
                     order=rng.choice([6, 6, 7, 8]), leaf=rng.choice([40, 64, 64, 100]))
    if kind == "tol":
        n = _log_size(rng, 2000, 300000)
        return _case(surface=surface, n=n, k_im=kappa(n), io=io, graph=graph, tol=tol)
    if kind == "fp64":
        n = _log_size(rng, 1000, 120000)
        return _case(surface=surface, n=n, k_im=kappa(n), io=io, precision="fp64",
                     tol=rng.choice([-1.0, tol]))
    if kind == "columns":
        n = _log_size(rng, 2000, 100000)
        return _case(surface=surface, n=n, k_im=kappa(n), io=io, columns=rng.randint(2, 32),
                     tol=rng.choice([-1.0, -1.0, 1e-4]))
    if kind == "combined":
        n = _log_size(rng, 4000, 130000)
        return _case(kernel="combined", surface="torus", n=n, k_im=kappa(n) * 0.9, order=8, io=io,
                     graph=graph, tol=rng.choice([-1.0, 1e-4, 1e-5]))
    if kind == "double":
        n = _log_size(rng, 2000, 100000)
        return _case(kernel="doublelayer", surface=rng.choice(["torus", "sphere"]), n=n, k_re=0.5,
                     k_im=-0.5 * kappa(n), order=rng.choice([7, 8]), leaf=40, io=io)
    if kind == "field":
        n = _log_size(rng, 1000, 100000)
        return _case(kernel=rng.choice(["modhelmholtz", "helmholtz"]), surface=surface, n=n,
                     targets=_log_size(rng, 500, 100000), k_re=0.5, k_im=-0.5 * kappa(n),
                     order=rng.choice([7, 8, 8]), io=io)
    if kind == "laplace":
        n = _log_size(rng, 1000, 300000)
        return _case(kernel="laplace", surface=surface, n=n, k_im=0.0, order=rng.choice([7, 8]),
                     io=io)
    if kind == "merged":
        n = _log_size(rng, 8000, 200000)
        return _case(n=n, k_im=round(rng.uniform(8, 32), 2), parts=rng.randint(2, 12))
    n = _log_size(rng, 2000, 40000)
    return _case(surface=rng.choice(["perturbed", "spheroid"]), n=n, k_im=kappa(n),
                 call="gradients")


# --- inputs ------------------------------------------------------------------------------
def _points(surface, n, g):
    """n points on the surface and the unit normals there (None where no kernel asks for them)."""
    if surface == "torus":
        big, small = 1.0, 0.4
        us, vs, have = [], [], 0
        while have < n:
            u, v, w = torch.rand((3, 2 * n + 64), generator=g, device=DEV, dtype=torch.float64)
            u, v = 2 * math.pi * u, 2 * math.pi * v
            keep = w < (big + small * torch.cos(v)) / (big + small)
            us.append(u[keep])
            vs.append(v[keep])
            have += us[-1].numel()
        u, v = torch.cat(us)[:n], torch.cat(vs)[:n]
        rho = big + small * torch.cos(v)
        x = torch.stack([rho * torch.cos(u), rho * torch.sin(u), small * torch.sin(v)], 1)
        nrm = torch.stack([torch.cos(v) * torch.cos(u), torch.cos(v) * torch.sin(u), torch.sin(v)],
                          1)
        return x, nrm

    def directions(k):
        p = torch.randn((k, 3), generator=g, device=DEV, dtype=torch.float64)
        return p / p.norm(dim=1, keepdim=True)

    if surface == "sphere":
        p = directions(n)
        return p, p.clone()
    if surface == "spheroid":
        xs, have = [], 0
        while have < n:
            p = directions(2 * n + 64)
            dens = torch.sqrt(0.25 * (p[:, 0] ** 2 + p[:, 1] ** 2) + p[:, 2] ** 2)
            w = torch.rand(p.shape[0], generator=g, device=DEV, dtype=torch.float64)
            xs.append((p * torch.tensor([1.0, 1.0, 0.5], device=DEV, dtype=torch.float64))[w < dens])
            have += xs[-1].shape[0]
        return torch.cat(xs)[:n], None
    # smooth bumps of the unit sphere, amplitude about 0.1
    p = directions(n)
    axes = torch.randn((6, 3), generator=g, device=DEV, dtype=torch.float64) * 2.0
    amps = torch.randn(6, generator=g, device=DEV, dtype=torch.float64)
    r = 1.0 + 0.1 * (torch.sin(p @ axes.t() + amps) * amps).sum(1) / 3.0
    return p * r[:, None].clamp(0.5, 1.5), None


def _part_sizes(case):
    """Uneven sizes of a merged operator's parts (about geometric, factor 16 from first to last),
    summing to n."""
    q = case["parts"]
    w = [16.0 ** (i / max(1, q - 1)) for i in range(q)]
    sizes = [max(256, int(case["n"] * x / sum(w))) for x in w]
    return sizes


def _inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)
    single = case["precision"] == "mixed"
    ctype = torch.complex64 if single else torch.complex128
    clouds = []
    for n in (_part_sizes(case) if case["parts"] > 1 else [case["n"]]):
        x, nrm = _points(case["surface"], n, g)
        y = x
        if case["targets"]:
            # field points in a cube around the surface, none of them on it
            y = (torch.rand((case["targets"], 3), generator=g, device=DEV, dtype=torch.float64) - 0.5) * 3.2
        clouds.append((x, y, nrm))
    if case["call"] == "gradients":  # mesh vertices in single precision, as they are optimised
        clouds = [(x.float().double(),) * 2 + (None,) for x, _, _ in clouds]
    total = sum(x.shape[0] for x, _, _ in clouds)
    shape = (total,) if case["columns"] == 1 else (total, case["columns"])
    if case["kernel"] == "laplace":
        w = torch.randn(shape, generator=g, device=DEV, dtype=torch.float64)
        w = w.float() if single else w
    else:
        w = torch.view_as_complex(torch.randn((*shape, 2), generator=g, device=DEV,
                                              dtype=torch.float64)).to(ctype)
    b = torch.view_as_complex(torch.randn((total, 2), generator=g, device=DEV,
                                          dtype=torch.float64)).to(ctype)
    return clouds, w, b


def _wavenumbers(case):
    return [case["k_im"] * (1.0 - 0.5 * i / case["parts"]) for i in range(case["parts"])]


def _operator(case, k_im):
    rest = (case["leaf"], case["order"], 1, case["tol"])
    prec = case["precision"]
    kind = case["kernel"]
    if kind == "helmholtz":
        return ifgf_amd.HelmholtzIfgfOperator(abs(k_im), *rest, precision=prec)
    if kind == "combined":
        return ifgf_amd.CombinedFieldHelmholtzIfgfOperator(k_im, *rest, precision=prec)
    if kind == "laplace":
        return ifgf_amd.LaplaceIfgfOperator(*rest, precision=prec)
    k = complex(case["k_re"], k_im)
    if kind == "doublelayer":
        return ifgf_amd.DoubleLayerHelmholtzIfgfOperator(k, *rest, precision=prec)
    return ifgf_amd.MofifiedHelmholtzIfgfOperator(k, *rest, precision=prec)


def prepare(case, seed):
    clouds, w, b = _inputs(case, seed)
    if case["call"] == "gradients":
        x = clouds[0][0].float().requires_grad_()
        return {"case": case, "x": x, "sigma": w.requires_grad_(), "b": b}
    ops = []
    for (x, y, nrm), k in zip(clouds, _wavenumbers(case)):
        op = _operator(case, k)
        xs, ys = x.cpu().numpy().T, y.cpu().numpy().T
        if case["kernel"] in ("combined", "doublelayer"):
            op.init(xs, ys, nrm.cpu().numpy().T)
        else:
            op.init(xs, ys)
        ops.append(op)
    op = ops[0] if len(ops) == 1 else ifgf_amd.merge(ops)
    op.use_graph = case["graph"]
    return {"case": case, "op": op, "w": w.cpu().numpy() if case["io"] == "host" else w}


def run(state):
    case = state["case"]
    if case["call"] == "gradients":
        x, sigma, b = state["x"], state["sigma"], state["b"]
        u = helmholtz_apply(sigma, x, kappa=case["k_im"], leaf=case["leaf"], order=case["order"],
                            tol=case["tol"], precision=case["precision"])
        r = u - b
        loss = (r.real.square() + r.imag.square()).sum()
        gs, gx = torch.autograd.grad(loss, [sigma, x])
        return {"u": u.detach(), "grad_density": gs, "grad_points": gx}
    w = state["w"]
    u = state["op"].mult(w)
    # the program's vectors keep the precision of its densities
    return u.astype(w.dtype) if case["io"] == "host" else u.to(w.dtype)


# --- the same products by direct summation in 64 bits -------------------------------------------
def _direct(case, k_im, x, y, nrm, w):
    """out[j, c] = sum_i G(x_i, y_j) w[i, c] (pairs at distance 0 left out), w (N, C) complex."""
    kind = case["kernel"]
    kre = case["k_re"] if kind in ("modhelmholtz", "doublelayer") else 0.0
    # e^{-k d}: k = -i kappa for the real-wavenumber kernels
    kim = -abs(k_im) if kind in ("helmholtz", "combined") else k_im
    wr, wi = w.real.contiguous(), w.imag.contiguous()
    out = torch.empty((y.shape[0], w.shape[1]), dtype=torch.complex128, device=DEV)
    step = max(1, int(6e7) // x.shape[0])
    for j in range(0, y.shape[0], step):
        yy = y[j:j + step]
        d2 = torch.zeros((yy.shape[0], x.shape[0]), dtype=torch.float64, device=DEV)
        for a in range(3):
            d2.addcmul_(t := yy[:, a, None] - x[None, :, a], t)
        far = d2 > 0
        d = torch.where(far, d2, 1.0).sqrt_()
        f = far / (4 * math.pi * d)
        if kind == "laplace":
            out[j:j + step] = torch.complex(f @ wr, f @ wi)
            continue
        if kre:
            f *= torch.exp(-kre * d)
        c, s = torch.cos(kim * d), -torch.sin(kim * d)
        if kind in ("combined", "doublelayer"):
            # n_x . (y - x), from the differences: about d^2 on a smooth surface
            nv = torch.zeros_like(d)
            for a in range(3):
                nv += (yy[:, a, None] - x[None, :, a]) * nrm[None, :, a]
            if kind == "combined":
                kap = abs(kim)
                pr, pi = nv / d2.clamp_min(1e-300), -kap * (nv + d) / d  # (nv (1 - i k d) - i k d^2)/d^2
                pr, pi = torch.where(far, pr, 0.0), torch.where(far, pi, 0.0)
            else:
                q = -nv / d  # (1/4pi d) e^{-kd} (k + 1/d) (n.(x-y)) / d
                pr, pi = (kre + 1 / d) * q, kim * q
            c, s = c * pr - s * pi, c * pi + s * pr
        c *= f
        s *= f
        out[j:j + step] = torch.complex(c @ wr - s @ wi, c @ wi + s @ wr)
    return out


def _direct_gradients(case, x, sigma, b):
    kap = case["k_im"]
    n = x.shape[0]
    step = max(1, int(5e7) // n)

    def sums(cols_g, cols_h):
        """G cols_g and H cols_h, H = G'(d) / d"""
        og = torch.empty((n, cols_g.shape[1]), dtype=torch.complex128, device=DEV)
        oh = torch.empty((n, cols_h.shape[1]), dtype=torch.complex128, device=DEV)
        for j in range(0, n, step):
            d2 = torch.zeros((min(step, n - j), n), dtype=torch.float64, device=DEV)
            for a in range(3):
                d2.addcmul_(t := x[j:j + step, a, None] - x[None, :, a], t)
            far = d2 > 0
            d = torch.where(far, d2, 1.0).sqrt_()
            f = far / (4 * math.pi * d)
            c, s = torch.cos(kap * d) * f, torch.sin(kap * d) * f
            for cols, to, cc, ss in (
                    (cols_g, og, c, s),
                    (cols_h, oh, (-c - kap * d * s) / (d * d), (kap * d * c - s) / (d * d))):
                if cols.shape[1]:
                    cr, ci = cols.real.contiguous(), cols.imag.contiguous()
                    to[j:j + step] = torch.complex(cc @ cr - ss @ ci, cc @ ci + ss @ cr)
        return og, oh

    none = torch.empty((n, 0), dtype=torch.complex128, device=DEV)
    u = sums(sigma[:, None], none)[0][:, 0]
    g = 2 * (u - b)
    gc = g.conj().resolve_conj()
    cols = torch.cat([torch.cat([v[:, None], v[:, None] * x], 1) for v in (sigma, gc)], 1)
    og, oh = sums(gc[:, None], cols)
    grad_density = og[:, 0].conj().resolve_conj()
    ds = x * oh[:, 0:1] - oh[:, 1:4]  # sum_j H_kj (x_k - x_j) sigma_j
    dg = x * oh[:, 4:5] - oh[:, 5:8]
    gx = (gc[:, None] * ds + sigma[:, None] * dg).real
    return {"u": u, "grad_density": grad_density, "grad_points": gx}


def exact(case, seed):
    m = case["targets"] or case["n"]
    if case["n"] * m > 8e10:
        return None
    clouds, w, b = _inputs(case, seed)
    if case["call"] == "gradients":
        return _direct_gradients(case, clouds[0][0], w.to(torch.complex128), b.to(torch.complex128))
    w2 = w.to(torch.complex128).reshape(w.shape[0], -1)
    outs, at = [], 0
    for (x, y, nrm), k in zip(clouds, _wavenumbers(case)):
        outs.append(_direct(case, k, x, y, nrm, w2[at:at + x.shape[0]]))
        at += x.shape[0]
    u = torch.cat(outs)
    if case["kernel"] == "laplace":
        u = u.real.contiguous()
    u = u[:, 0].contiguous() if case["columns"] == 1 else u
    return u.cpu().numpy() if case["io"] == "host" else u


def work(case):
    """Bytes: points, densities and results once.  Flops: an estimate of the factorization's own
    operations on a surface with leaves of this size: direct pairs with the neighbouring leaves
    (about nine), sampling of each leaf's cones, and on each of the levels above the transfer
    and the interpolation of a few cones' worth of nodes per point."""
    n, m, q = case["n"], case["targets"] or case["n"], case["columns"]
    small = case["precision"] == "mixed"
    cell = (4 if small else 8) * (1 if case["kernel"] == "laplace" else 2)
    nbytes = 24 * (n + m) + cell * q * (n + m)
    hi = (case["order"] - (3 if case["tol"] <= 0 else 0)) * case["order"] ** 2
    lo = max(2, case["order"] - 3) ** 2 * max(2, case["order"] - (6 if case["tol"] <= 0 else 3))
    levels = max(1.0, math.log2(max(2.0, n / case["leaf"])) / 2)
    per_point = 23 * 12 * case["leaf"] + 26 * 8 * hi + levels * 35 * (50 + 4 * lo) * 2
    flops = per_point * (n + m) / 2 * q
    if case["call"] == "gradients":
        flops, nbytes = 9 * flops, 3 * nbytes
    return {"bytes": float(nbytes), "flops": float(flops)}
