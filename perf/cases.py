"""The workloads this library is timed on, through its public entry points.

Four kinds of call, the ones a user of the Kress / Beyn path makes:
  window       one Beyn window: assembly and LU of every contour node, the moment
               solves and their QR on the device (Window + moments_qr), complex128 or
               mixed precision, of a plain or a symmetry-reduced geometry;
  matrices     construct_boundary_matrices into host buffers (host: true) or
               qb_assemble into device memory (QB_OUT_DEVICE);
  derivatives  T, dT/dk and d2T/dk2 (qb_assemble_deriv) into device memory, the
               input of an expanded-boundary-integral solver;
  residuals    the residual norms of candidate eigenpairs (residual_norms).

Sizes follow the library's rule of 10 points per wavelength, N = 10 k L / 2 pi, over
the wavenumbers of its serving stream (k0 from 50 on), its benchmark window (star,
N = 8192, 48 nodes, 768 probes), its assembly benchmark (ellipse, N = 4096) and its
uneven windows (disk with a hole).  The probe counts are probe_count's.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "quantumbilliards.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qbhip as q  # noqa: E402

SHAPES = {
    "star": lambda: q.make_star_polar_boundary(1.0, 0.2, 5),
    "ellipse": lambda: q.make_full_ellipse(1.0, 0.6),
    "circle_hole": lambda: q.CircularHoleBilliard(1.0, holes=[(0.3, 0.35, 0.0)]),
}
HOLE = (0.3, 0.35, 0.0)
SVD_TOL = 1e-10  # the serving loop's and the benchmark's rank threshold


def _k0(shape, N):
    """The wavenumber that 10 points per wavelength give for N nodes."""
    return round(2 * math.pi * N / (10.0 * SHAPES[shape]().length), 3)


def _window(shape, N, nq=32, R=0.5, op="cfie", precision="fp64", irreps=0):
    b, k0 = SHAPES[shape](), _k0(shape, N)
    r = q.probe_count(b, k0, R, nq, SVD_TOL, r0=32)
    if irreps:  # each irrep of the group holds its share of the levels
        r = 32 * (-(-r // (32 * irreps)) + 1)
    return {"kind": "window", "op": op, "shape": shape, "N": N, "k0": k0, "R": R, "nq": nq,
            "r": min(r, N // max(irreps, 1)), "precision": precision, "irreps": irreps}


def _matrices(shape, N, nz, op="cfie", host=False, kind="matrices"):
    return {"kind": kind, "op": op, "shape": shape, "N": N, "k0": _k0(shape, N), "nz": nz,
            "host": host}


def listed():
    named = [
        # the smallest call: one T(k) on the host, as an interactive check makes it
        ("matrix_star_128_host", _matrices("star", 128, 1, host=True)),
        # the assembly benchmark's operator and size (DLP, ellipse, N = 4096), 16 nodes
        ("matrices_dlp_ellipse_4096", _matrices("ellipse", 4096, 16, op="dlp")),
        # two components of ragged sizes, the contour of a small window
        ("matrices_cfie_hole_1562", _matrices("circle_hole", 1562, 24)),
        # the matrices of one expanded-boundary-integral step
        ("derivatives_star_1500", _matrices("star", 1500, 6, kind="derivatives")),
        # the spurious-root filter over a window's candidates
        ("residuals_star_2050", _matrices("star", 2050, 32, kind="residuals")),
        # the smallest windows of the serving stream (k0 about 50 to 60): many launches
        ("window_ellipse_530", _window("ellipse", 530, R=0.3)),
        # a small DLP window of odd size on the same shape
        ("window_dlp_ellipse_1141", _window("ellipse", 1141, op="dlp")),
        # a window of the uneven workload, two components
        ("window_hole_1792", _window("circle_hole", 1792)),
        # a medium window of the serving stream, an odd size
        ("window_star_4100", _window("star", 4100)),
        # complex64 LU with FP64 refinement, a precision the caller may ask for
        ("window_star_3072_mixed", _window("star", 3072, precision="mixed")),
        # the benchmark disk reduced by C_5: five irreps of 1640 unknowns, one batch
        ("window_c5_star_8200", _window("star", 8200, nq=48, irreps=5)),
        # the benchmark window: star, N = 8192, 48 nodes, 768 probes
        ("window_star_8192", dict(_window("star", 8192, nq=48), k0=800.0, r=768)),
    ]
    return [dict(c, name=n) for n, c in named]


def draw(rng):
    """A case of the ranges above: windows of the serving stream and the uneven workload
    up to N = 4800, assemblies up to 16 nodes of N = 4096."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    u = rng.random()
    if u < 0.64:
        shape = rng.choice(["star", "star", "ellipse", "circle_hole"])
        op = "dlp" if shape == "ellipse" and rng.random() < 0.4 else "cfie"
        nq, R = rng.choice([24, 32, 48]), round(rng.uniform(0.25, 0.5), 3)
        v = rng.random()
        if v < 0.15:
            return _window("star", 10 * size(100, 820), nq=32, R=R, irreps=5)
        if v < 0.3:
            return _window(shape, size(800, 3100), nq=nq, R=R, precision="mixed")
        return _window(shape, size(500, 4800), nq=nq, R=R, op=op)
    shape = rng.choice(["star", "ellipse", "circle_hole"])
    op = "dlp" if shape == "ellipse" and rng.random() < 0.5 else "cfie"
    if u < 0.72:
        return _matrices(shape, size(100, 700), rng.randint(1, 4), op=op, host=True)
    if u < 0.84:
        return _matrices(shape, size(500, 4096), rng.randint(2, 16), op=op)
    if u < 0.92:
        return _matrices(shape, size(300, 2000), rng.randint(1, 6), op=op, kind="derivatives")
    return _matrices(shape, size(400, 2600), rng.randint(4, 40), op=op, kind="residuals")


# -- inputs ------------------------------------------------------------------
def _counts(case):
    """Nodes per component: a disk with a hole splits them as the circumferences, 10 : 3."""
    N = case["N"]
    if case["shape"] != "circle_hole":
        return [N]
    n = int(round(N * 10.0 / 13.0))
    return [n, N - n]


def _inputs(case, seed):
    """The seed's wavenumbers and blocks: a disk or a contour whose centre lies within 1/4 of
    the case's k0, the probes N(0, 1/2) + i N(0, 1/2), candidate vectors of unit norm."""
    rng = np.random.default_rng(seed)
    k0 = case["k0"] + rng.uniform(-0.25, 0.25)
    if case["kind"] == "window":
        m = case["N"] // max(case["irreps"], 1)
        return {"k0": k0, "V": q.probe_block(rng, m, case["r"])}
    nz = case["nz"]
    if case["kind"] == "residuals":  # roots in the disk, real up to the solves' rounding
        phi = rng.standard_normal((case["N"], nz)) + 1j * rng.standard_normal((case["N"], nz))
        phi = np.asfortranarray(phi / np.linalg.norm(phi, axis=0))
        return {"z": k0 + rng.uniform(-0.5, 0.5, nz) + 1e-12j * rng.standard_normal(nz), "phi": phi}
    if nz == 1:
        return {"z": np.array([k0 + 0.1j])}
    return {"z": k0 + 0.5 * np.exp(2j * np.pi * np.arange(nz) / nz)}


def prepare(case, seed):
    inp = _inputs(case, seed)
    b = SHAPES[case["shape"]]()
    make = q.DLP_kress if case["op"] == "dlp" else q.CFIE_kress
    irreps = [q.CFIE_kress(10.0, b, symmetry=q.Rotation(5, m)) for m in range(case.get("irreps", 0))]
    solver = irreps[0] if irreps else make(10.0, b)
    pts = q.evaluate_points(solver, b, case["k0"], N=_counts(case))
    geom = q.Geometry(pts, solver=solver, irreps=irreps or None)
    s = {"case": case, "solver": solver, "pts": pts, "geom": geom}
    z = inp.get("z")
    if z is None:
        z = inp["k0"] + case["R"] * np.exp(2j * np.pi * np.arange(case["nq"]) / case["nq"])
    # table sizes as a user's program chooses them, once per geometry and wavenumber range
    nh, mh, nj, mj, _ = q.chebyshev_params(solver, pts, z, tol=1e-12, geom=geom)
    s.update(inp, cheb=dict(n_panels_h=nh, M_h=mh, n_panels_j=nj, M_j=mj))
    if case["kind"] == "window":
        s["V"] = q.pinned_array(inp["V"].shape)
        s["V"][...] = inp["V"]
        return s
    N, nz = case["N"], case["nz"]
    if case["kind"] == "residuals":
        return s
    if case["host"]:
        s["out"] = [np.empty((N, N), np.complex128, order="F") for _ in range(nz)]
    else:
        n = 3 if case["kind"] == "derivatives" else 1
        # [z][column][row]: each matrix column-major, the library's layout
        s["out"] = [torch.zeros(nz, N, N, dtype=torch.complex128, device="cuda") for _ in range(n)]
        s["params"] = q._lib.ChebParams(nh, mh, nj, mj)
    return s


def run(s):
    case, geom = s["case"], s["geom"]
    if case["kind"] == "window":
        tol = 1e-12 if case["precision"] == "mixed" else 1e-13
        w = q.Window(s["solver"], s["pts"], s["k0"], case["R"], case["nq"], geom=geom,
                     precision=case["precision"], **s["cheb"])
        R, C = w.moments_qr(s["V"], refine_tol=tol)
        w.close()
        return {"R": R, "C": C}
    if case["kind"] == "residuals":
        return list(q.residual_norms(s["solver"], s["pts"], s["z"], s["phi"], geom=geom, **s["cheb"]))
    if case["host"]:
        q.construct_boundary_matrices(s["out"], s["solver"], s["pts"], s["z"], geom=geom, **s["cheb"])
        return s["out"]
    ctx, z = geom.ctx, s["z"]
    fn = q.lib().qb_assemble_deriv if case["kind"] == "derivatives" else q.lib().qb_assemble
    rc = fn(ctx.ptr, geom.ptr, s["solver"].op, z.ctypes.data, len(z), ctypes.byref(s["params"]),
            *[o.data_ptr() for o in s["out"]], q._lib.QB_OUT_DEVICE, None)
    q._lib.check(ctx.ptr, rc)
    return s["out"]


def work(case):
    N = case["N"]
    # per entry the value's series and Kress terms (Clenshaw of degree 7 for the Hankel and
    # the Bessel pair): what the tables route of the reference evaluates
    entry = 64.0 if case["op"] == "dlp" else 134.0
    if case["kind"] == "window":
        n_mat, m = case["nq"] * max(case["irreps"], 1), N // max(case["irreps"], 1)
        r, blocks = case["r"], max(case["irreps"], 1)
        images = m * m * max(case["irreps"], 1) * case["nq"]  # evaluated once for all irreps
        flops = entry * images + n_mat * (8.0 / 3.0 * m ** 3 + 8.0 * m * m * r)
        flops += blocks * 16.0 * m * r * r  # QR of A0, its Q^H on A1
        return {"bytes": 16.0 * (m * r + 2 * blocks * r * r), "flops": flops}
    n2 = float(N) * N * case["nz"]
    if case["kind"] == "residuals":
        return {"bytes": 16.0 * N * case["nz"], "flops": (entry + 14.0) * n2}
    n_out = 3 if case["kind"] == "derivatives" else 1
    return {"bytes": 16.0 * n2 * n_out, "flops": (entry + 40.0 * (n_out - 1)) * n2}


# -- the same in 64 bits, from the formulas ------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _hankel(z):
    """H0, H1 of the first kind: the power series below |z| = 2, above it the integral
    H_n = (2 / pi z)^(1/2) e^(i(z - n pi/2 - pi/4)) / Gamma(n + 1/2)
          int_0^oo e^-u u^(n - 1/2) (1 + iu / 2z)^(n - 1/2) du
    with u = t^2 by the trapezoidal rule (step 0.2: exponentially accurate)."""
    zs = torch.where(z.abs() < 2.0, torch.full_like(z, 2.0), z)
    c = 0.5j / zs
    h = 0.2
    s0 = torch.ones_like(z)
    s1 = torch.zeros_like(z)
    for n in range(1, 33):
        t2 = (h * n) ** 2
        g = torch.sqrt(1.0 + c * t2)
        s0 += (2.0 * math.exp(-t2)) / g
        s1 += (2.0 * math.exp(-t2) * t2) * g
    pre = torch.sqrt(2.0 / (math.pi * zs)) * torch.exp(1j * zs) * complex(math.sqrt(0.5), -math.sqrt(0.5))
    h0 = pre * s0 * (h / math.sqrt(math.pi))
    h1 = pre * s1 * (-2j * h / math.sqrt(math.pi))
    small = z.abs() < 2.0
    if bool(small.any()):
        x = z[small]
        w = -0.25 * x * x
        a, lg = torch.ones_like(x), torch.log(0.5 * x) + 0.5772156649015328606
        j0, j1, y0, y1 = a.clone(), a.clone(), torch.zeros_like(x), torch.ones_like(x)
        a1, hk = a.clone(), 0.0
        for k in range(1, 26):
            hk += 1.0 / k
            a = a * w / (k * k)
            a1 = a1 * w / (k * (k + 1))
            j0 += a
            j1 += a1
            y0 -= hk * a
            y1 += (2 * hk + 1.0 / (k + 1)) * a1
        j1 = j1 * 0.5 * x
        h0[small] = j0 + 1j * ((2 / math.pi) * (lg * j0 + y0))
        h1[small] = j1 + 1j * ((2 / math.pi) * lg * j1 - 2 / (math.pi * x) - x / (2 * math.pi) * y1)
    return h0, h1


def _curve(kind, n):
    t = 2 * math.pi * (torch.arange(1, n + 1, dtype=torch.float64, device=_dev()) - 0.5) / n
    c, s = torch.cos(t), torch.sin(t)
    if kind == "ellipse":
        return t, c, 0.6 * s, -s, 0.6 * c, -c, -0.6 * s
    if kind == "star":
        r, r1, r2 = 1 + 0.2 * torch.cos(5 * t), -torch.sin(5 * t), -5 * torch.cos(5 * t)
        return (t, r * c, r * s, r1 * c - r * s, r1 * s + r * c,
                r2 * c - 2 * r1 * s - r * c, r2 * s + 2 * r1 * c - r * s)
    rad, cx, cy = (1.0, 0.0, 0.0) if kind == "circle" else HOLE
    v = (t, rad * c + cx, rad * s + cy, -rad * s, rad * c, -rad * c, -rad * s)
    if kind == "circle":
        return v
    t, x, y, dx, dy, ddx, ddy = (a.flip(0) for a in v)  # a hole runs the other way round
    return t, x, y, -dx, -dy, ddx, ddy


def _kress_column(n):
    d = torch.arange(n, device=_dev())
    m = torch.arange(1, (n - 1) // 2 + 1, device=_dev())
    acc = torch.zeros(n, dtype=torch.float64, device=_dev())
    for part in m.split(512):
        acc += (torch.cos(2 * math.pi * ((part[:, None] * d) % n).double() / n) / part[:, None]).sum(0)
    col = -(4 * math.pi / n) * acc
    if n % 2 == 0:
        col -= (4 * math.pi / n ** 2) * (1.0 - 2.0 * (d % 2).double())
    return col


class _Operator:
    """T(z) (and its first two z derivatives) of a case's operator; rows: only the first
    `rows` of them (one component)."""

    def __init__(self, case, rows=None):
        self.dlp = case["op"] == "dlp"
        kinds = ["circle", "hole"] if case["shape"] == "circle_hole" else [case["shape"]]
        self.comps = [_curve(k, n) for k, n in zip(kinds, _counts(case))]
        self.rows = rows
        self.blocks = {}
        for a, ca in enumerate(self.comps):
            for b, cb in enumerate(self.comps):
                self.blocks[a, b] = self._geometry(ca, cb, a == b)

    def _geometry(self, ca, cb, same):
        m = self.rows or len(ca[0])
        n = len(cb[0])
        dx, dy = ca[1][:m, None] - cb[1], ca[2][:m, None] - cb[2]
        r = torch.hypot(dx, dy)
        inn = cb[4] * dx - cb[3] * dy
        sp = torch.hypot(cb[3], cb[4])
        g = {"inn": inn, "s": sp, "w": 2 * math.pi / n, "same": same}
        if same:
            i = torch.arange(m, device=_dev())
            r[i, i] = 1.0
            d = (i[:, None] - torch.arange(n, device=_dev())) % n
            g["R"] = _kress_column(n)[d]
            lt = 2.0 * torch.log(2.0 * torch.sin(math.pi * d.double() / n).abs())
            lt[i, i] = 0.0
            g["lt"] = lt
            k = -(cb[3] * cb[6] - cb[4] * cb[5]) / (2 * math.pi * (cb[3] ** 2 + cb[4] ** 2))
            g.update(i=i, kap=k[:m], sd=sp[:m])
        g["r"] = r
        return g

    def hankels(self, z):
        return {ab: _hankel(z * g["r"]) for ab, g in self.blocks.items()}

    def values(self, z, H, Hc, deriv=False):
        """H, Hc: the Hankel values at z and at conj(z); J_n(z) = (H_n(z) + conj H_n(conj z)) / 2."""
        n = len(self.comps)
        rows = [[self._block(z, self.blocks[a, b], H[a, b], Hc[a, b], deriv) for b in range(n)]
                for a in range(n)]
        return [torch.cat([torch.cat([blk[d] for blk in row], 1) for row in rows], 0)
                for d in range(3 if deriv else 1)]

    def _block(self, k, g, H, Hc, deriv):
        (h0, h1), r, inn, w, s = H, g["r"], g["inn"], g["w"], g["s"]
        kr, ik, tp = k * r, 1j * k, 1 / (2 * math.pi)
        if g["same"]:
            j0, j1 = 0.5 * (h0 + Hc[0].conj()), 0.5 * (h1 + Hc[1].conj())
            R, lt = g["R"], g["lt"]

            def split(j, h):  # Kress's split of a kernel with the logarithm j and the rest h
                return R * j - w * (lt * j + 1j * math.pi * h)
            D = [-k * tp * inn / r * split(j1, h1)]
            S = [-tp * s * split(j0, h0)]
            if deriv:
                D += [-k * tp * inn * split(j0, h0), tp * inn * split(kr * j1 - j0, kr * h1 - h0)]
                S += [tp * r * s * split(j1, h1), tp * r * s / k * split(kr * j0 - j1, kr * h0 - h1)]
        else:
            # the derivatives' double-layer terms between components carry the reference's sign
            D = [w * inn / r * 0.5j * k * h1, -0.5j * w * inn * k * h0, -0.5j * w * inn * (h0 - kr * h1)]
            S = [0.5j * w * s * h0, -0.5j * w * s * r * h1, 0.5j * w * s * r * (h1 - kr * h0) / k]
        if self.dlp:
            out = [-d for d in D]
        else:
            out = [-(D[0] + ik * S[0])]
            if deriv:
                out += [-(D[1] + 1j * S[0] + ik * S[1]), -(D[2] + 2j * S[1] + ik * S[2])]
        if g["same"]:
            i, kap, sd = g["i"], g["kap"], g["sd"]
            d0 = 1.0 - w * kap + 0j
            sv = -tp * g["R"][0, 0] * sd + w * sd * (
                (0.5j - 0.5772156649015328606 / math.pi) - tp * torch.log((k * k / 4.0) * (sd * sd)))
            out[0][i, i] = d0 if self.dlp else d0 - ik * sv
            if deriv and self.dlp:
                out[1][i, i] = 0.0
                out[2][i, i] = 0.0
            elif deriv:
                s1, s2 = -w * sd / (math.pi * k), w * sd / (math.pi * k * k)
                out[1][i, i] = -(1j * sv + ik * s1)
                out[2][i, i] = -(2j * s1 + ik * s2)
        return out[: 3 if deriv else 1]


def _tensor(z):
    return torch.tensor(complex(z), dtype=torch.complex128, device=_dev())


def _exact_window(case, inp):
    nq, irr = case["nq"], max(case["irreps"], 1)
    m = case["N"] // irr
    op = _Operator(case, rows=m if irr > 1 else None)
    e = np.exp(2j * np.pi * np.arange(nq) / nq)
    z, w = inp["k0"] + case["R"] * e, case["R"] / nq * e
    V = torch.from_numpy(np.ascontiguousarray(inp["V"])).to(_dev())
    A = [[torch.zeros_like(V) for _ in range(2)] for _ in range(irr)]
    for j in range(nq // 2 + 1):  # the nodes j and nq - j are conjugates
        H = {}
        pair = [j] if (2 * j) % nq == 0 else [j, nq - j]
        zz = [_tensor(complex(z[j].real, 0.0 if len(pair) == 1 else z[j].imag))]
        zz.append(zz[0].conj().resolve_conj())
        H = [op.hankels(zz[0])]
        H.append(H[0] if len(pair) == 1 else op.hankels(zz[1]))
        for p, jj in enumerate(pair):
            T = op.values(zz[p], H[p], H[1 - p])[0]
            for b in range(irr):
                Tb = T
                if irr > 1:  # sum over the rotations of the star, weighted by the character
                    chi = torch.from_numpy(np.exp(2j * np.pi * b * np.arange(irr) / irr)).to(_dev())
                    Tb = (T.view(m, irr, m) * chi[None, :, None]).sum(1)
                X = torch.linalg.solve(Tb, V)
                A[b][0] += complex(w[jj]) * X
                A[b][1] += complex(w[jj] * z[jj]) * X
    R, C = [], []
    for a0, a1 in A:
        Q, r = np.linalg.qr(a0.cpu().numpy())
        R.append(r)
        C.append(Q.conj().T @ a1.cpu().numpy())
    return {"R": np.stack(R) if irr > 1 else R[0], "C": np.stack(C) if irr > 1 else C[0]}


def exact(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] == "window":
        m = case["N"] // max(case["irreps"], 1)
        if case["nq"] * max(case["irreps"], 1) * m ** 3 > 2.6e12:
            return None
        return _exact_window(case, inp)
    op = _Operator(case)
    deriv = case["kind"] == "derivatives"
    outs = []
    for i, zc in enumerate(inp["z"]):
        z = _tensor(zc)
        T = op.values(z, op.hankels(z), op.hankels(z.conj().resolve_conj()), deriv)
        if case["kind"] == "residuals":
            y = T[0] @ torch.from_numpy(inp["phi"][:, i].copy()).to(_dev())
            a = T[0].abs()
            outs.append([float(v) for v in (y.abs().square().sum().sqrt(), y.abs().sum(), y.abs().max(),
                                            a.sum(0).max(), a.sum(1).max())])
        elif case["host"]:
            outs.append(T[0].cpu().numpy())
        else:
            outs.append([t.T.contiguous() for t in T])
    if case["kind"] == "residuals":
        return [np.array(v) for v in zip(*outs)]
    return outs if case["host"] else [torch.stack(v) for v in zip(*outs)]
