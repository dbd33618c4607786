"""Performance cases of the library's main paths, through its C entry points.

Each case is one thing a program using this library does in earnest: a stencil
apply on one box, the face averages of a finite-volume step, a fused residual,
a ghost exchange, a multigrid solve, a batch operator over uneven patches, a
served stream of solves.  listed() are the representative sizes; draw() gives
others of the same ranges.  Arrays are torch tensors on the GPU (the library
takes their device pointers); everything runs on the null stream, which is
torch's default stream too.
"""
import ctypes
import math
import random

import numpy as np
import torch

import proto_amd as pa

_I = ctypes.POINTER(ctypes.c_int)
_D = ctypes.POINTER(ctypes.c_double)
_DT = {"f64": (pa.PM_F64, torch.float64, 8), "f32": (pa.PM_F32, torch.float32, 4)}


def listed():
    return [
        # the smallest call: a 2-D 5-point Laplacian on a 256 x 256 box followed by absMax (apply + norm test)
        {"name": "apply2d_256_f64", "kind": "apply2d", "nx": 256, "ny": 256, "dtype": "f64"},
        # one operator apply on a single odd-sized box in single precision (27-point Laplacian)
        {"name": "apply27_199x131x97_f32", "kind": "apply3d", "op": "L27", "nx": 199, "ny": 131, "nz": 97, "ncomp": 1,
         "dtype": "f32"},
        # the flux loop of a 4th-order finite-volume step: cell to face averages of 5 components in every direction
        {"name": "faces4_128_c5_f64", "kind": "faces", "nx": 128, "ny": 128, "nz": 128, "ncomp": 5, "dtype": "f64"},
        # the benchmark's step: both operators' residuals of 512^3 cells with absMax and sum
        {"name": "residual2_512_f64", "kind": "residual", "n": 512, "ghost": 2, "dtype": "f64"},
        # ghost fill between stages of a multi-component solver: 5 components, 4 ghost layers, 32^3 boxes
        {"name": "exchange_192_b32_c5_f64", "kind": "exchange", "box": 32, "kx": 6, "ky": 6, "kz": 6, "ghost": 4,
         "ncomp": 5, "dtype": "f64"},
        # a small Poisson solve, where launches and the per-cycle norm read-back count
        {"name": "mg_ir_64_b32", "kind": "mg", "box": 32, "k": 2, "precision": 1, "inner": 1},
        # a plain FP64 Poisson solve in the usual 32^3 boxes
        {"name": "mg_f64_256_b32", "kind": "mg", "box": 32, "k": 8, "precision": 0, "inner": 1},
        # the largest solve: 512^3 in 64^3 boxes, FP32 cycles inside FP64 refinement
        {"name": "mg_ir_512_b64", "kind": "mg", "box": 64, "k": 8, "precision": 1, "inner": 4},
        # the library (FAS, 4th-order operator) solver
        {"name": "fas_128_b32", "kind": "fas", "box": 32, "k": 4, "tol": 1e-8},
        # smoothing of a whole AMR level of uneven patches, double precision
        {"name": "batch_gsrb_2000_f64", "kind": "batch_gsrb", "boxes": 2000, "edges": "16,24,32,48,64", "ghost": 2,
         "dtype": "f64"},
        # the 27-point operator on a smaller set of uneven patches with odd sizes, single precision
        {"name": "batch_apply_300_f32", "kind": "batch_apply", "boxes": 300, "edges": "15,20,33,47,64", "ghost": 2,
         "dtype": "f32"},
        # a burst of solve requests of mixed sizes with their answers read back
        {"name": "serve_24", "kind": "serve", "requests": 24, "sizes": "32,48,64,96,128", "tol": 1e-8, "inner": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, sizes spread over the logarithm of its range."""
    kind = rng.choice(["apply2d", "apply3d", "faces", "residual", "exchange", "mg", "mg", "fas", "batch_gsrb",
                       "batch_apply", "serve"])
    dtype = rng.choice(["f64", "f32"])
    if kind == "apply2d":
        return {"kind": kind, "nx": _log(rng, 33, 2048), "ny": _log(rng, 33, 2048), "dtype": dtype}
    if kind == "apply3d":
        return {"kind": kind, "op": rng.choice(["L7", "L19", "L27"]), "nx": _log(rng, 24, 320), "ny": _log(rng, 24, 320),
                "nz": _log(rng, 24, 320), "ncomp": rng.choice([1, 1, 2, 3]), "dtype": dtype}
    if kind == "faces":
        return {"kind": kind, "nx": _log(rng, 24, 160), "ny": _log(rng, 24, 160), "nz": _log(rng, 24, 160),
                "ncomp": rng.choice([1, 3, 5]), "dtype": dtype}
    if kind == "residual":
        return {"kind": kind, "n": _log(rng, 40, 448), "ghost": rng.choice([1, 2]), "dtype": dtype}
    if kind == "exchange":
        box = rng.choice([16, 24, 32, 48, 64])
        most = 256 // box
        return {"kind": kind, "box": box, "kx": rng.randint(1, most), "ky": rng.randint(1, most),
                "kz": rng.randint(1, most), "ghost": rng.randint(1, 4), "ncomp": rng.choice([1, 2, 3, 5]),
                "dtype": dtype}
    if kind == "mg":
        box = rng.choice([16, 24, 32, 48, 64])
        precision = rng.choice([0, 1])
        most = (320 if precision == 0 else 400) // box
        # grids that halve down to a coarsest level of a few cells, as multigrid wants them
        ks = [k for k in range(1, most + 1) if (box * k) >> _coarsenings(box * k) <= 12]
        size = _log(rng, 1, most)
        return {"kind": kind, "box": box, "k": min(ks, key=lambda k: abs(math.log(k / size))),
                "precision": precision, "inner": rng.randint(1, 4) if precision else 1}
    if kind == "fas":
        box = rng.choice([16, 24, 32, 48, 64])
        ks = [k for k in range(1, 192 // box + 1) if box * k >= 32 and (box * k) >> _coarsenings(box * k) <= 12]
        return {"kind": kind, "box": box, "k": rng.choice(ks), "tol": rng.choice([1e-5, 1e-6, 1e-7, 1e-8])}
    if kind in ("batch_gsrb", "batch_apply"):
        edges = rng.sample([12, 15, 16, 20, 24, 32, 33, 40, 47, 48, 64], 4) if rng.random() < 0.5 else \
            rng.sample([16, 24, 32, 40, 48, 64], 3)
        return {"kind": kind, "boxes": _log(rng, 20, 2000), "edges": ",".join(str(e) for e in sorted(edges)),
                "ghost": rng.choice([1, 2]), "dtype": dtype}
    sizes = rng.sample([32, 48, 64, 96, 128, 192], 3)
    return {"kind": "serve", "requests": _log(rng, 4, 24), "sizes": ",".join(str(v) for v in sorted(sizes)),
            "tol": rng.choice([1e-8, 1e-10]), "inner": rng.choice([1, 4])}


# ---------------------------------------------------------------- stencils
def _laplacian(name, dim=3):
    """Coefficients and (x, y, z) offsets of the library's Laplacians."""
    if name == "L7":
        axes = [[1 if k == d else 0 for k in range(3)] for d in range(dim)]
        offs = [[0, 0, 0]] + [o for a in axes for o in (a, [-v for v in a])]
        return [-2.0 * dim] + [1.0] * (2 * dim), offs
    weights = {"L19": (-4.0, {1: 1.0 / 3.0, 2: 1.0 / 6.0}),
               "L27": (-64.0 / 15.0, {1: 7.0 / 15.0, 2: 1.0 / 10.0, 3: 1.0 / 30.0})}
    centre, by_distance = weights[name]
    coefs, offs = [centre], [[0, 0, 0]]
    for z in (-1, 0, 1):
        for y in (-1, 0, 1):
            for x in (-1, 0, 1):
                s = abs(x) + abs(y) + abs(z)
                if s in by_distance:
                    coefs.append(by_distance[s])
                    offs.append([x, y, z])
    return coefs, offs


def _to_face(axis):
    """CellToFace(axis, Low, 4): the 4th-order average on the low face of a cell."""
    coefs = [-1.0 / 12.0, -1.0 / 12.0, 7.0 / 12.0, 7.0 / 12.0]
    return coefs, [[o if k == axis else 0 for k in range(3)] for o in (-2, 1, -1, 0)]


def _apply64(coefs, offs, u, lo, shape, scale=1.0):
    """sum_j c_j u[p + o_j] over `shape` (z, y, x); u is (..., z, y, x) in 64 bits, lo the index of cell 0."""
    out = None
    for c, (ox, oy, oz) in zip(coefs, offs):
        v = u[..., lo[2] + oz:lo[2] + oz + shape[0], lo[1] + oy:lo[1] + oy + shape[1], lo[0] + ox:lo[0] + ox + shape[2]]
        out = v * (c * scale) if out is None else out.add_(v, alpha=c * scale)
    return out


# ---------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(shape, dtype, gen):
    """U[-1, 1)."""
    return torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen).mul_(2).sub_(1).to(dtype)


def _smooth_box(n, g, seed):
    """A smooth periodic field with 1e-3 of noise on [-g, n + g)^3, ghosts the periodic images (64 bits)."""
    gen = _generator(seed)
    x = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) / n
    ph = torch.rand(3, dtype=torch.float64, device="cuda", generator=gen)
    s = [torch.sin(2 * math.pi * (x + ph[d])) for d in range(3)]
    u = s[2][:, None, None] * s[1][None, :, None] * s[0][None, None, :]
    u += _uniform((n, n, n), torch.float64, gen).mul_(1e-3)
    at = torch.arange(-g, n + g, device="cuda") % n
    return u[at][:, at][:, :, at].contiguous()


def _gaussians(x, cen, amp, sigma=0.05):
    """sum_k amp_k exp(-|x - c_k|^2 / (2 sigma^2)) on the periodic unit cube, minus its mean; (z, y, x)."""
    n = x.numel()
    d = (x[None, None, :] - cen[:, :, None]).abs()
    d = torch.minimum(d, 1.0 - d)
    t = torch.exp(-(d * d) / (2 * sigma * sigma))  # (3, K, n)
    yx = (t[1][:, :, None] * t[0][:, None, :]).reshape(t.shape[1], n * n)
    f = torch.mm((t[2] * amp[:, None]).t().contiguous(), yx).reshape(n, n, n)
    return f - f.mean()


def _poisson_rhs(n, seed):
    gen = _generator(seed)
    k = 16
    cen = torch.rand((3, k), dtype=torch.float64, device="cuda", generator=gen)
    amp = torch.where(torch.rand(k, dtype=torch.float64, device="cuda", generator=gen) < 0.5, -1.0, 1.0).double()
    x = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) / n
    return _gaussians(x, cen, amp)


def _to_boxes(f, box, g):
    """A periodic (z, y, x) field as level storage: boxes x fastest, each with g ghost layers."""
    kz, ky, kx = (s // box for s in f.shape)
    out = torch.empty((kz, ky, kx, box + 2 * g, box + 2 * g, box + 2 * g), dtype=f.dtype, device=f.device)
    at = [[torch.arange(b * box - g, (b + 1) * box + g, device=f.device) % s for b in range(k)]
          for k, s in zip((kz, ky, kx), f.shape)]
    for z in range(kz):
        for y in range(ky):
            zy = f[at[0][z]][:, at[1][y]]
            for x in range(kx):
                out[z, y, x] = zy[:, :, at[2][x]]
    return out


def _from_gen(box, kx, ky, kz, ncomp, g, dtype, seed):
    """Level storage (box, comp, z, y, x) with random valid cells and stale ghosts."""
    gen = _generator(seed)
    b = box + 2 * g
    return _uniform((kx * ky * kz, ncomp, b, b, b), dtype, gen)


def _request_gaussians(count, seed):
    """Centres and amplitudes a served request's seed stands for (SplitMix64, stream 7)."""
    m = (1 << 64) - 1
    s0 = (seed + 7 * 0x632BE59BD9B4E019) & m
    u = []
    for i in range(4 * count):
        z = (s0 + (i + 1) * 0x9E3779B97F4A7C15) & m
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
        z ^= z >> 31
        u.append(((z >> 11) * 2.0 ** -53) * 2.0 - 1.0)
    u = torch.tensor(u, dtype=torch.float64, device="cuda")
    cen = (u[:3 * count].reshape(count, 3) + 1.0) * 0.5
    return cen.t().contiguous(), torch.where(u[3 * count:] >= 0, 1.0, -1.0).double()


def _requests(case, seed):
    rng = random.Random(seed)
    sizes = [int(v) for v in case["sizes"].split(",")]
    # every size in turn, so that a stream of a few requests has them all
    return [{"arrival_s": 0.0, "n": sizes[i % len(sizes)], "ngauss": rng.randint(4, 32), "seed": rng.randrange(1 << 31),
             "tol": case["tol"], "keep_result": 1} for i in range(case["requests"])]


def _sizes(case):
    """Extents (nx, ny, nz) of every patch; part of the case, the same for every seed."""
    rng = random.Random(case["boxes"])
    edges = [int(v) for v in case["edges"].split(",")]
    return [[rng.choice(edges) for _ in range(3)] for _ in range(case["boxes"])]


def _poisson64(rhs, fourth=False):
    """The zero-mean solution of the discrete periodic Poisson problem on the unit cube, by FFT in 64 bits."""
    n = rhs.shape[0]
    th = 2 * math.pi * torch.arange(n, dtype=torch.float64, device="cuda") / n
    if fourth:
        s = (-torch.cos(2 * th) + 16 * torch.cos(th) - 15) * (n * n / 6.0)
    else:
        s = (torch.cos(th) - 1) * (2.0 * n * n)
    r = torch.fft.rfftn(rhs)
    lam = s[:, None, None] + s[None, :, None] + s[None, None, :n // 2 + 1]
    lam[0, 0, 0] = 1.0
    r /= lam
    r[0, 0, 0] = 0
    return torch.fft.irfftn(r, s=(n, n, n))


# ---------------------------------------------------------------- handles
class _Handle:
    """A native handle with its destroy function."""

    def __init__(self, make, destroy, *args):
        self.h, self._destroy = ctypes.c_void_p(), destroy
        pa.call(make, ctypes.byref(self.h), *args)

    def __del__(self):
        if self.h and pa is not None:
            getattr(pa.lib(), self._destroy)(self.h)
            self.h = None


def _layout(box, kx, ky, kz):
    lows = np.array([(x * box, y * box, z * box) for z in range(kz) for y in range(ky) for x in range(kx)],
                    dtype=np.int32).reshape(-1)
    return _Handle("pm_layout_create", "pm_layout_destroy", 3, pa.i3([kx * box, ky * box, kz * box]), pa.i3([box] * 3),
                   pa.i3([1, 1, 1]), kx * ky * kz, lows.ctypes.data_as(_I))


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _coarsenings(n):
    """Halvings down to a coarsest level of at most 8 cells, or the last even one."""
    k = 0
    while n > 8 and n % 4 == 0:
        n //= 2
        k += 1
    return k


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("apply2d", "apply3d", "faces"):
        code, dtype, _ = _DT[case["dtype"]]
        nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
        s["scale"] = float(nx) ** 2
        gen = _generator(seed)
        if kind == "apply2d":
            coefs, offs = _laplacian("L7", 2)
            s["st"] = pa.Stencil(coefs, offs, code, 2)
            s["u"] = _uniform((ny + 2, nx + 2), dtype, gen)
            s["src_box"], s["box"] = pa.Box.of([-1, -1], [nx, ny]), pa.Box.of([0, 0], [nx - 1, ny - 1])
            s["out"] = torch.zeros((ny, nx), dtype=dtype, device="cuda")
            s["norm"] = torch.zeros(1, dtype=dtype, device="cuda")
        elif kind == "apply3d":
            coefs, offs = _laplacian(case["op"])
            s["st"] = pa.Stencil(coefs, offs, code, 3)
            s["u"] = _uniform((case["ncomp"], nz + 2, ny + 2, nx + 2), dtype, gen)
            s["src_box"] = pa.Box.of([-1] * 3, [nx, ny, nz])
            s["box"] = pa.Box.of([0] * 3, [nx - 1, ny - 1, nz - 1])
            s["out"] = torch.zeros((case["ncomp"], nz, ny, nx), dtype=dtype, device="cuda")
        else:
            s["u"] = _uniform((case["ncomp"], nz + 8, ny + 8, nx + 8), dtype, gen)
            s["src_box"] = pa.Box.of([-4] * 3, [nx + 3, ny + 3, nz + 3])
            s["st"], s["box"], s["out"] = [], [], []
            for d in range(3):
                n = [nx, ny, nz]
                n[d] += 1  # the faces along d
                s["st"].append(pa.Stencil(*_to_face(d), code, 3))
                s["box"].append(pa.Box.of([0] * 3, [v - 1 for v in n]))
                s["out"].append(torch.zeros((case["ncomp"], n[2], n[1], n[0]), dtype=dtype, device="cuda"))
    elif kind == "residual":
        code, dtype, _ = _DT[case["dtype"]]
        n, g = case["n"], case["ghost"]
        s["st"] = [pa.Stencil(*_laplacian(name), code, 3) for name in ("L7", "L27")]
        s["u"] = _smooth_box(n, g, seed).to(dtype)
        s["f"] = _uniform((n, n, n), dtype, _generator(seed + 1))
        s["r"] = [torch.zeros((n, n, n), dtype=dtype, device="cuda") for _ in range(2)]
        s["red"] = torch.zeros(4, dtype=dtype, device="cuda")
        s["src_box"], s["box"] = pa.Box.of([-g] * 3, [n - 1 + g] * 3), pa.Box.of([0] * 3, [n - 1] * 3)
    elif kind == "exchange":
        dtype = _DT[case["dtype"]][1]
        k = (case["kx"], case["ky"], case["kz"])
        s["layout"] = _layout(case["box"], *k)
        s["data"] = _from_gen(case["box"], *k, case["ncomp"], case["ghost"], dtype, seed)
        s["ghost"] = pa.i3([case["ghost"]] * 3)
    elif kind in ("mg", "fas"):
        box, k = case["box"], case["k"]
        n, g = box * k, 1 if kind == "mg" else 2
        s["layout"] = _layout(box, k, k, k)
        s["rhs"] = _to_boxes(_poisson_rhs(n, seed), box, 0)
        s["phi"] = torch.zeros((k, k, k) + (box + 2 * g,) * 3, dtype=torch.float64, device="cuda")
        s["hist"], s["iters"] = np.zeros(81), ctypes.c_int()
        if kind == "mg":
            opt = pa.MgOptions()
            pa.lib().pm_mg_default_options(ctypes.byref(opt))
            opt.precision, opt.inner, opt.max_iter, opt.tol = case["precision"], case["inner"], 80, 1e-10
            s["solver"] = _Handle("pm_mg_create", "pm_mg_destroy", s["layout"].h, _coarsenings(n), 1.0 / n,
                                  ctypes.byref(opt))
        else:
            s["solver"] = _Handle("pm_fas_create", "pm_fas_destroy", s["layout"].h, _coarsenings(n) + 1, 1.0 / n)
    elif kind in ("batch_gsrb", "batch_apply"):
        code, dtype, _ = _DT[case["dtype"]]
        s["batch"] = pa.Batch(_sizes(case), case["ghost"])
        gen = _generator(seed)
        s["u"] = _uniform((s["batch"].ghosted_elems,), dtype, gen)
        if kind == "batch_gsrb":
            s["rhs"] = _uniform((s["batch"].valid_elems,), dtype, gen)
            s["out"] = s["u"].clone()  # the ghosts of the output are the input's
        else:
            s["st"] = pa.Stencil(*_laplacian("L27"), code, 3)
            s["out"] = torch.zeros(s["batch"].valid_elems, dtype=dtype, device="cuda")
    else:
        s["server"] = pa.Server(mode=0, inner=case["inner"])
        s["requests"] = _requests(case, seed)
    return s


# ---------------------------------------------------------------- run
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "apply2d":
        box = ctypes.byref(s["box"])
        pa.call("pm_stencil_apply_reduce", s["st"].h, _p(s["u"]), ctypes.byref(s["src_box"]), _p(s["out"]), box, box, 1,
                s["scale"], pa.RED_ABS, _p(s["norm"]), 0, None)
        return {"out": s["out"], "norm": s["norm"]}
    if kind == "apply3d":
        box = ctypes.byref(s["box"])
        pa.call("pm_stencil_apply", s["st"].h, _p(s["u"]), ctypes.byref(s["src_box"]), _p(s["out"]), box, box,
                case["ncomp"], 1, s["scale"], None)
        return s["out"]
    if kind == "faces":
        for st, b, out in zip(s["st"], s["box"], s["out"]):
            box = ctypes.byref(b)
            pa.call("pm_stencil_apply", st.h, _p(s["u"]), ctypes.byref(s["src_box"]), _p(out), box, box, case["ncomp"],
                    1, 1.0, None)
        return s["out"]
    if kind == "residual":
        h2 = float(case["n"]) ** 2
        pa.call("pm_stencil_residual2", s["st"][0].h, s["st"][1].h, _p(s["u"]), ctypes.byref(s["src_box"]), _p(s["f"]),
                _p(s["r"][0]), _p(s["r"][1]), ctypes.byref(s["box"]), h2, h2, _p(s["red"]), None)
        return {"r7": s["r"][0], "r27": s["r"][1], "red": s["red"]}
    if kind == "exchange":
        pa.call("pm_level_exchange", s["layout"].h, _DT[case["dtype"]][0], _p(s["data"]), s["ghost"], case["ncomp"],
                None)
        return s["data"]
    if kind in ("mg", "fas"):
        phi = s["phi"]
        s["hist"].fill(0.0)
        pa.call("pm_memset_zero", _p(phi), phi.numel() * 8, None)  # the zero initial guess
        hist, iters = s["hist"].ctypes.data_as(_D), ctypes.byref(s["iters"])
        if kind == "mg":
            pa.call("pm_mg_solve", s["solver"].h, _p(phi), _p(s["rhs"]), hist, iters, None)
        else:
            pa.call("pm_fas_solve", s["solver"].h, _p(phi), _p(s["rhs"]), 80, case["tol"], hist, iters, None)
        return {"phi": phi, "hist": s["hist"].copy(), "iters": s["iters"].value}
    if kind == "batch_gsrb":
        s["batch"].gsrb(_DT[case["dtype"]][0], _p(s["u"]), _p(s["out"]), _p(s["rhs"]), 1.0 / 64)
        return s["out"]
    if kind == "batch_apply":
        s["batch"].apply(s["st"], _p(s["u"]), _p(s["out"]), 1.0)
        return s["out"]
    stats = s["server"].run(s["requests"])
    phi = [s["server"].result(i, q["n"]) for i, q in enumerate(s["requests"])]
    return {"phi": phi, "iters": [r["iters"] for r in stats]}


# ---------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    e = _DT[case["dtype"]][2] if "dtype" in case else 8
    if kind == "apply2d":
        nx, ny = case["nx"], case["ny"]
        return {"bytes": e * ((nx + 2) * (ny + 2) + nx * ny), "flops": 11 * nx * ny}
    if kind == "apply3d":
        nx, ny, nz, c = case["nx"], case["ny"], case["nz"], case["ncomp"]
        taps = int(case["op"][1:])
        return {"bytes": e * c * ((nx + 2) * (ny + 2) * (nz + 2) + nx * ny * nz), "flops": 2 * taps * c * nx * ny * nz}
    if kind == "faces":
        nx, ny, nz, c = case["nx"], case["ny"], case["nz"], case["ncomp"]
        faces = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
        cells = nx * ny * nz + 4 * (nx * ny + ny * nz + nx * nz)
        return {"bytes": e * c * (cells + faces), "flops": 8 * c * faces}
    if kind == "residual":
        n = case["n"]
        return {"bytes": e * ((n + 2) ** 3 + 3 * n ** 3), "flops": 74 * n ** 3}
    if kind == "exchange":
        b, g, boxes = case["box"], case["ghost"], case["kx"] * case["ky"] * case["kz"]
        return {"bytes": 2 * e * case["ncomp"] * boxes * ((b + 2 * g) ** 3 - b ** 3), "flops": 0}
    if kind in ("mg", "fas"):
        # the right-hand side read, the solution written; the smallest count of cycles that reaches the tolerance
        n = case["box"] * case["k"]
        return {"bytes": 16 * n ** 3, "flops": (10 * 100 if kind == "mg" else 20 * 400) * n ** 3}
    if kind in ("batch_gsrb", "batch_apply"):
        sizes = _sizes(case)
        valid = sum(x * y * z for x, y, z in sizes)
        foot = sum((x + 2) * (y + 2) * (z + 2) for x, y, z in sizes)
        if kind == "batch_gsrb":
            return {"bytes": e * (foot + 2 * valid), "flops": 17 * valid}
        return {"bytes": e * (foot + valid), "flops": 54 * valid}
    sizes = [int(v) for v in case["sizes"].split(",")]
    cells = sum(sizes[i % len(sizes)] ** 3 for i in range(case["requests"]))
    return {"bytes": 16 * cells, "flops": 8 * 100 * cells}


# ---------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind in ("apply2d", "apply3d", "faces"):
        s = prepare(case, seed)
        u = s["u"].double()
        nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
        if kind == "apply2d":
            coefs, offs = _laplacian("L7", 2)
            out = _apply64(coefs, offs, u[None], (1, 1, 0), (1, ny, nx), s["scale"])[0]
            return {"out": out, "norm": out.abs().max().reshape(1)}
        if kind == "apply3d":
            return _apply64(*_laplacian(case["op"]), u, (1, 1, 1), (nz, ny, nx), s["scale"])
        return [_apply64(*_to_face(d), u, (4, 4, 4), (nz + (d == 2), ny + (d == 1), nx + (d == 0))) for d in range(3)]
    if kind == "residual":
        s = prepare(case, seed)
        n, g = case["n"], case["ghost"]
        u, f = s["u"].double(), s["f"].double()
        r = [f - _apply64(*_laplacian(name), u, (g, g, g), (n, n, n), float(n) ** 2) for name in ("L7", "L27")]
        red = torch.stack([r[0].abs().max(), r[0].sum(), r[1].abs().max(), r[1].sum()])
        return {"r7": r[0], "r27": r[1], "red": red}
    if kind == "exchange":
        b, g, c = case["box"], case["ghost"], case["ncomp"]
        kx, ky, kz = case["kx"], case["ky"], case["kz"]
        d = _from_gen(b, kx, ky, kz, c, g, _DT[case["dtype"]][1], seed).double()
        valid = d[:, :, g:g + b, g:g + b, g:g + b].reshape(kz, ky, kx, c, b, b, b)
        out = torch.empty_like(d)
        for k in range(c):
            f = valid[:, :, :, k].permute(0, 3, 1, 4, 2, 5).reshape(kz * b, ky * b, kx * b)
            out[:, k] = _to_boxes(f, b, g).reshape(kx * ky * kz, b + 2 * g, b + 2 * g, b + 2 * g)
        return out
    if kind in ("mg", "fas"):
        n = case["box"] * case["k"]
        phi = _poisson64(_poisson_rhs(n, seed), kind == "fas")
        return {"phi": _to_boxes(phi, case["box"], 1 if kind == "mg" else 2), "hist": None, "iters": None}
    if kind in ("batch_gsrb", "batch_apply"):
        g, gen = case["ghost"], _generator(seed)
        sizes = _sizes(case)
        dtype = _DT[case["dtype"]][1]
        nvalid = sum(x * y * z for x, y, z in sizes)
        u = _uniform((sum((x + 2 * g) * (y + 2 * g) * (z + 2 * g) for x, y, z in sizes),), dtype, gen).double()
        rhs = _uniform((nvalid,), dtype, gen).double() if kind == "batch_gsrb" else None
        out = u.clone() if kind == "batch_gsrb" else torch.empty(nvalid, dtype=torch.float64, device="cuda")
        at, av = 0, 0
        for x, y, z in sizes:
            ng, nv = (x + 2 * g) * (y + 2 * g) * (z + 2 * g), x * y * z
            box = u[at:at + ng].view(z + 2 * g, y + 2 * g, x + 2 * g)
            if kind == "batch_apply":
                out[av:av + nv] = _apply64(*_laplacian("L27"), box, (g, g, g), (z, y, x)).reshape(-1)
            else:
                v = out[at:at + ng].view(z + 2 * g, y + 2 * g, x + 2 * g)
                f = rhs[av:av + nv].view(z, y, x) / 64.0 ** 2
                for colour in (0, 1):
                    for a in range(2):  # the parity of z and of y fix that of x
                        for b in range(2):
                            c = (colour + a + b) % 2
                            iz, iy, ix = slice(g + a, g + z, 2), slice(g + b, g + y, 2), slice(g + c, g + x, 2)

                            def nb(sl, o):
                                return slice(sl.start + o, sl.stop + o, 2)
                            t = (v[iz, iy, nb(ix, 1)] + v[iz, iy, nb(ix, -1)] + v[iz, nb(iy, 1), ix] +
                                 v[iz, nb(iy, -1), ix] + v[nb(iz, 1), iy, ix] + v[nb(iz, -1), iy, ix])
                            v[iz, iy, ix] = (t - f[a::2, b::2, c::2]) / 6.0
            at, av = at + ng, av + nv
        return out
    reqs = _requests(case, seed)
    phi = []
    for q in reqs:
        x = (torch.arange(q["n"], dtype=torch.float64, device="cuda") + 0.5) / q["n"]
        rhs = _gaussians(x, *_request_gaussians(q["ngauss"], q["seed"]))
        phi.append(_poisson64(rhs).reshape(-1).cpu().numpy())
    return {"phi": phi, "iters": None}
