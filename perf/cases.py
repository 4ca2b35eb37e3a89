"""The calls whose time is watched: what a program built on this package runs.

A case is one pass through the package's public surface -- ``opr * x``,
``egoOpr_``, ``mul_``, ``LippmannSchwinger.apply`` or one Arnoldi step of the
solver.  Green data is handed in as
``egoFur`` (point-collocated dyadic Green tensor of the geometry, the type the
operator holds), so that ``exact`` can form the same product in 64 bits with
plain FFTs; the cases marked ``green: geometry`` let the library compute it.

Fields of a case (plain values):
  what    matvec (opr * x, or egoOpr_ for several right-hand sides), mul
          (mul_), ls (Lippmann-Schwinger apply), arnoldi
  type    c64 or c128
  target  cells of the target volume, of side 1/32 wavelength
  source  cells of the source volume ("" for a self operator)
  ratio   source cells per target cell and axis (2: a finer source volume)
  inside  the source lies centred inside the target (else beside it, on z)
  rhs     right-hand sides
  green   given or geometry
"""
import importlib.util
import math
import os
import sys
from fractions import Fraction

import numpy as np
import torch

H = Fraction(1, 32)
BASIS = 16          # vectors of the Arnoldi step's basis (mid-cycle of GMRES(30))
NPC = {"c64": np.complex64, "c128": np.complex128}
TPC = {"c64": torch.complex64, "c128": torch.complex128}


def _gila():
    """The package, under the name its own documentation loads it by."""
    if "gila_amd" in sys.modules:
        return sys.modules["gila_amd"]
    d = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gilaelectromagnetics.jl_amd")
    spec = importlib.util.spec_from_file_location("gila_amd", os.path.join(d, "__init__.py"),
                                                  submodule_search_locations=[d])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["gila_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


def _case(name, what, typ, target, source="", ratio=1, inside=False, rhs=1, green="given"):
    return {"name": name, "what": what, "type": typ, "target": target, "source": source, "ratio": ratio,
            "inside": inside, "rhs": rhs, "green": green}


def listed():
    return [
        # a small scatterer: launches and latency are all there is
        _case("self 16^3 c64", "matvec", "c64", "16x16x16"),
        # cell counts as a geometry happens to give them, default precision
        _case("self 30x22x14 c128", "matvec", "c128", "30x22x14"),
        # four media on one grid, as a batched solver applies them
        _case("ls 4 rhs 32x48x64 c64", "ls", "c64", "32x48x64", rhs=4),
        # an ordinary volume in the default precision
        _case("self 64^3 c128", "matvec", "c128", "64x64x64"),
        # a larger volume whose cell counts are no transform-friendly lengths
        _case("self 100x60x44 c64", "matvec", "c64", "100x60x44"),
        # many sources on one volume
        _case("16 rhs 96^3 c64", "matvec", "c64", "96x96x96", rhs=16),
        # the benchmark's operator, in both precisions (the second through
        # mul_ into a kept vector, as an iterative solver calls it)
        _case("self 128^3 c64", "matvec", "c64", "128x128x128"),
        _case("mul 128^3 c128", "mul", "c128", "128x128x128"),
        # fields of one volume in another: a small uneven pair, and the
        # waveguide in its surroundings (the largest)
        _case("external 40x18x17 in 64x64x33 c128", "matvec", "c128", "64x64x33", "40x18x17"),
        _case("external 256x34x34 in 256x256x128 c64", "matvec", "c64", "256x256x128", "256x34x34", inside=True,
              green="geometry"),
        # a finely meshed source beside a coarse target (8 partitions)
        _case("fine source 48^3 to 24^3 c64", "matvec", "c64", "24x24x24", "48x48x48", ratio=2),
        # one step of the batched GMRES: operator, Gram-Schmidt, next vector
        _case("arnoldi 8 rhs 64x64x48 c64", "arnoldi", "c64", "64x64x48", rhs=8),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cells(rng, lo, hi):
    base = _logu(rng, lo, hi)
    return [min(hi, max(lo, int(round(base * rng.uniform(0.6, 1.4))))) for _ in range(3)]


def _txt(c):
    return "x".join(str(v) for v in c)


def draw(rng):
    """One more case: every kind, sizes over the whole range, odd ones among them."""
    while True:
        what = rng.choices(["self", "batch", "mul", "ls", "external", "inside", "fine", "arnoldi"],
                           [5, 1, 2, 1, 2, 1, 1, 1])[0]
        typ = rng.choice(["c64", "c128"])
        if what in ("self", "mul"):
            c = _case("", "matvec" if what == "self" else "mul", typ, _txt(_cells(rng, 12, 128)))
        elif what in ("batch", "ls"):
            c = _case("", "matvec" if what == "batch" else "ls", typ, _txt(_cells(rng, 12, 96)),
                      rhs=_logu(rng, 2, 16))
        elif what == "arnoldi":
            c = _case("", "arnoldi", typ, _txt(_cells(rng, 16, 64)), rhs=_logu(rng, 2, 8))
        elif what == "fine":
            # even counts: odd ones would have the constructor regenerate the volumes
            t, s = ([v + v % 2 for v in _cells(rng, 8, 32)] for _ in range(2))
            c = _case("", "matvec", typ, _txt(t), _txt([2 * v for v in s]), ratio=2)
        else:
            t = _cells(rng, 16, 128)
            s = [max(2, int(round(v * rng.uniform(0.2, 0.9)))) for v in t]
            s = [v + (v + w) % 2 for v, w in zip(s, t)]
            c = _case("", "matvec", typ, _txt(t), _txt(s), inside=what == "inside")
        del c["name"]
        if _moved(c) <= 2.6e9:
            return c


# --- geometry -----------------------------------------------------------

def _ints(t):
    return [int(v) for v in t.split("x")]


class _Geo:
    """Partition cells, branch lengths, stored extents and first-centre
    distances of a case (x, y, z order)."""

    def __init__(self, case):
        self.T = _ints(case["target"])
        self.self_ = not case["source"]
        self.r = int(case["ratio"])
        full = self.T if self.self_ else _ints(case["source"])
        self.S = [v // self.r for v in full]
        self.src_full = full
        self.hT, self.hS = float(H), float(H) / self.r
        self.L = [s + t for s, t in zip(self.S, self.T)]
        # source centre: beside the target on z, four cells away, or at its centre
        self.org = [0, 0, 0]
        if not self.self_ and not case["inside"]:
            self.org[2] = -(Fraction(self.T[2] + self.S[2], 2) + 4) * H
        first = lambda n, h, o: float(o) - h * (n - 1) / 2
        self.d0 = [first(t, self.hT, 0) - first(s, self.hS, o) for t, s, o in zip(self.T, full, self.org)]
        np_ = self.r ** 3
        self.offs = [(p % self.r, (p // self.r) % self.r, p // self.r ** 2) for p in range(np_)]
        sym = [s == t and o == 0 and np_ == 1 for s, t, o in zip(self.S, self.T, self.org)]
        self.U = [((t + 1) // 2 + (t % 2 == 0)) if y else l // 2 for t, y, l in zip(self.T, sym, self.L)]


def _spectrum(geo, off, dev, typ):
    """(6, L3, L2, L1) Fourier Green data of source partition `off`: the
    dyadic Green function at the cell-centre separations times the source
    cell's volume, embedded in the circulant, transformed in 64 bits and
    rounded to the operator's type (as complex128)."""
    k = 2 * math.pi
    sep = []
    for a in range(3):
        n = torch.arange(geo.L[a], dtype=torch.float64, device=dev)
        m = torch.where(n < geo.T[a], n, n - geo.L[a])
        sep.append((geo.d0[a] - off[a] * geo.hS + m * geo.hT))
    r = [sep[2][:, None, None], sep[1][None, :, None], sep[0][None, None, :]][::-1]
    r2 = r[0] ** 2 + r[1] ** 2 + r[2] ** 2
    zero = r2 < 1e-16
    r2 = torch.where(zero, torch.ones_like(r2), r2)
    rr = torch.sqrt(r2)
    vol = geo.hS ** 3
    e = torch.polar(k * k * vol / (4 * math.pi * rr), k * rr)
    kr = k * rr
    a = torch.complex(1 - 1 / kr ** 2, 1 / kr) * e
    b = torch.complex(3 / kr ** 2 - 1, -3 / kr) * e / r2
    rad = k * (3 * vol / (4 * math.pi)) ** (1 / 3)
    own = -1 / 3 + 2 / 3 * ((1 - 1j * rad) * complex(math.cos(rad), math.sin(rad)) - 1)
    keep = torch.ones_like(r2)
    for ax in range(3):          # the one separation between T - 1 and -(S - 1) is no pair of cells
        idx = [slice(None)] * 3
        idx[2 - ax] = geo.T[ax]
        keep[tuple(idx)] = 0
    out = torch.empty((6,) + tuple(r2.shape), dtype=torch.complex128, device=dev)
    for i, (p, q) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
        g = b * (r[p] * r[q])
        if p == q:
            g = g + a
        g = torch.where(zero, torch.full_like(g, own if p == q else 0), g) * keep
        out[i] = torch.fft.fftn(g)
    return out.to(TPC[typ]).to(torch.complex128) if typ == "c64" else out


def _branches(geo, typ, dev):
    """The eight egoFur branches, (U1,U2,U3,6) or (U1,U2,U3,6,Ps,1)."""
    U = geo.U
    per = [_spectrum(geo, o, dev, typ) for o in geo.offs]
    out = []
    for bits in range(8):
        p1, p2, p3 = bits >> 2, (bits >> 1) & 1, bits & 1
        br = torch.stack([f[:, p3::2, p2::2, p1::2][:, :U[2], :U[1], :U[0]] for f in per])
        br = br.to(TPC[typ]).cpu().numpy()
        br = br.transpose(4, 3, 2, 1, 0)
        out.append(br[..., 0] if len(per) == 1 else br[..., None])
    return out


def _operator(case, geo, frq=1.0 + 0.0j):
    g = _gila()
    trg = g.GlaVol(geo.T, (H,) * 3)
    src = trg if geo.self_ else g.GlaVol(geo.src_full, (H / geo.r,) * 3, geo.org)
    fur = None if case["green"] == "geometry" else _branches(geo, case["type"], torch.device("cuda"))
    return g.GlaOpr(g.GlaOprMem(g.GlaKerOpt(frq, devMod=True), trg, src, egoFur=fur, setTyp=NPC[case["type"]]))


def _randn(shape, seed, what, typ):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * (seed + 1) + what)
    return torch.randn(shape, generator=gen, dtype=TPC[typ], device="cuda")


def _rand(shape, seed, what):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * (seed + 1) + what)
    return torch.rand(shape, generator=gen, dtype=torch.float64, device="cuda")


def _field(cells, rhs, seed, what, typ):
    """A column-major field (c1,c2,c3,3), with a trailing rhs axis for several."""
    t = _randn((rhs, 3) + tuple(reversed(cells)), seed, what, typ)
    t = t.permute(4, 3, 2, 1, 0)
    return t[..., 0] if rhs == 1 else t


def _medium(cells, rhs, seed, typ):
    """A lossy dielectric ball per right-hand side (chi = 0 outside)."""
    ax = [torch.linspace(-1, 1, c, dtype=torch.float64, device="cuda") for c in cells]
    r2 = (ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2)
    u = _rand((rhs, 3), seed, 5)
    chi = [torch.where(r2 < (0.3 + 0.7 * u[i, 0]) ** 2, torch.complex(0.5 + 2.5 * u[i, 1], 0.1 * u[i, 2]),
                       torch.zeros((), dtype=torch.complex128, device="cuda")) for i in range(rhs)]
    return torch.stack([c.permute(2, 1, 0) for c in chi]).contiguous().permute(3, 2, 1, 0).to(TPC[typ])


def _basis(case, n, seed):
    v = _randn((case["rhs"], BASIS + 1, n), seed, 3, case["type"])
    for i in range(BASIS + 1):
        v[:, i] /= torch.linalg.vector_norm(v[:, i], dim=1, keepdim=True)
    return v


def prepare(case, seed):
    g = _gila()
    geo = _Geo(case)
    typ, rhs = case["type"], case["rhs"]
    st = {"what": case["what"], "opr": _operator(case, geo), "rhs": rhs}
    if case["what"] in ("matvec", "mul"):
        st["x"] = _field(geo.src_full, rhs, seed, 1, typ)
    if case["what"] == "mul":
        st["y"] = _field(geo.T, 1, seed, 2, typ)
    if case["what"] in ("ls", "arnoldi"):
        n = 3 * geo.T[0] * geo.T[1] * geo.T[2]
        st["A"] = g.solve.LippmannSchwinger(st["opr"], _medium(geo.T, rhs, seed, typ))
        st["x"] = _randn((rhs, n), seed, 1, typ)
        if case["what"] == "arnoldi":
            st["x"] /= torch.linalg.vector_norm(st["x"], dim=1, keepdim=True)
            st["V"] = _basis(case, n, seed)
            st["kry"] = g.solve.KrylovOps()
            st["w"] = torch.empty_like(st["x"])
            st["next"] = torch.empty_like(st["x"])
            st["at"] = torch.full((rhs,), BASIS, dtype=torch.int64, device="cuda")
    return st


def run(st):
    g = _gila()
    what = st["what"]
    if what == "matvec":
        return st["opr"] * st["x"] if st["rhs"] == 1 else g.egoOpr_(st["opr"].mem, st["x"])
    if what == "mul":
        return g.mul_(st["y"], st["opr"], st["x"])
    if what == "ls":
        return st["A"].apply(st["x"])
    # one Arnoldi step: w = A x, orthogonalized against the basis, and the
    # normalized next vector stored in the basis and staged
    k, w, V = st["rhs"], st["w"], st["V"]
    st["A"].apply(st["x"], w)
    s = torch.cuda.current_stream().cuda_stream
    h, n0, n1 = g.solve.gs_pass(st["kry"], V, k, BASIS, w, s)
    st["kry"].next(V, k, st["at"], w, n1, s, stage=st["next"])
    # coefficients and norms as precise as the vectors they are sums of
    real = torch.float32 if V.dtype == torch.complex64 else torch.float64
    return {"next": st["next"], "h": h.to(V.dtype), "before": n0.to(real), "after": n1.to(real)}


# --- work and exact results --------------------------------------------

def work(case):
    """Inputs, Green data and outputs once; the pruned transforms and the
    symmetric 3x3 product of one pass."""
    geo = _Geo(case)
    s = 8 if case["type"] == "c64" else 16
    S, T, L, rhs, P = geo.S, geo.T, geo.L, case["rhs"], len(geo.offs)
    nS, nT, nL = (v[0] * v[1] * v[2] for v in (S, T, L))
    fft = lambda n: 5 * n * math.log2(n)
    half = lambda c: 3 * (c[1] * c[2] * fft(L[0]) + L[0] * c[2] * fft(L[1]) + L[0] * L[1] * fft(L[2]))
    by = s * (8 * geo.U[0] * geo.U[1] * geo.U[2] * 6 * P + 3 * rhs * (nS * P + nT))
    fl = rhs * (P * half(S) + half(T) + P * nL * 66)
    n = 3 * nT * rhs
    if case["what"] in ("ls", "arnoldi"):
        by += s * n // 3
        fl += 8 * n
    if case["what"] == "arnoldi":
        by += s * n * (BASIS + 1)
        fl += n * (16 * BASIS + 8)
    return {"bytes": int(by), "flops": int(fl)}


def _moved(case):
    """Bytes of an axis-by-axis pass over a case (bounds what draw gives)."""
    geo = _Geo(case)
    s = 8 if case["type"] == "c64" else 16
    S, T, L = geo.S, geo.T, [1.2 * v for v in geo.L]
    f = 3 * case["rhs"] * len(geo.offs) * s
    rows = S[1] * S[2] + T[1] * T[2]
    return f * 2 * (L[0] * rows + L[0] * L[1] * (S[2] + T[2])) + 48 * s * L[0] * L[1] * L[2] / 8 * len(geo.offs)


def _apply64(case, geo, x):
    """G x in 64 bits by plain FFTs; x (rhs, 3, s3, s2, s1) on its device."""
    dev = x.device
    out = torch.zeros((x.shape[0], 3) + tuple(reversed(geo.T)), dtype=torch.complex128, device=dev)
    pick = ((0, 3, 4), (3, 1, 5), (4, 5, 2))
    r = geo.r
    for off in geo.offs:
        f = _spectrum(geo, off, dev, case["type"])
        for i in range(x.shape[0]):
            part = x[i, :, off[2]::r, off[1]::r, off[0]::r].to(torch.complex128)
            X = torch.fft.fftn(part, s=tuple(reversed(geo.L)), dim=(1, 2, 3))
            for c in range(3):
                y = f[pick[c][0]] * X[0] + f[pick[c][1]] * X[1] + f[pick[c][2]] * X[2]
                out[i, c] += torch.fft.ifftn(y)[:geo.T[2], :geo.T[1], :geo.T[0]]
    return out


def _back(t, rhs):
    t = t.permute(4, 3, 2, 1, 0)
    return t[..., 0] if rhs == 1 else t


def exact(case, seed):
    if case["green"] == "geometry":
        return None      # needs every face-pair integral of the geometry
    geo = _Geo(case)
    typ, rhs = case["type"], case["rhs"]
    if case["what"] in ("matvec", "mul"):
        x = _field(geo.src_full, rhs, seed, 1, typ)
        x = x.permute(*range(x.dim() - 1, -1, -1))
        y = _back(_apply64(case, geo, x[None] if rhs == 1 else x), rhs)
        return y
    n = 3 * geo.T[0] * geo.T[1] * geo.T[2]
    x = _randn((rhs, n), seed, 1, typ)
    if case["what"] == "arnoldi":
        x /= torch.linalg.vector_norm(x, dim=1, keepdim=True)
    chi = _medium(geo.T, rhs, seed, typ).permute(3, 2, 1, 0).to(torch.complex128)
    y = _apply64(case, geo, x.reshape((rhs, 3) + tuple(reversed(geo.T))))
    w = x.to(torch.complex128) - (chi[:, None] * y).reshape(rhs, n)
    if case["what"] == "ls":
        return w
    V = _basis(case, n, seed)[:, :BASIS].to(torch.complex128)
    before = torch.linalg.vector_norm(w, dim=1) ** 2
    h = torch.stack([(V[:, i].conj() * w).sum(1) for i in range(BASIS)], 1)
    for i in range(BASIS):
        w = w - h[:, i:i + 1] * V[:, i]
    after = torch.linalg.vector_norm(w, dim=1) ** 2
    return {"next": w / torch.sqrt(after)[:, None], "h": h, "before": before, "after": after}
