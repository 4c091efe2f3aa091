"""Performance cases of the hopping matrix, the solvers and the drop-in calls.

Each case is one call (or the fixed pair of calls) that a program makes again
and again with everything else in place: links uploaded, sources on the GPU,
or, for the drop-in calls, everything in host arrays.  The inputs are random
SU(3) links and Gaussian sources, the ones the repository's benchmark uses.

Keys of a case:
  path    hop     H on the whole lattice (both parities)
          halves  H_eo, then H_oe, as the reference's harness calls them
          schur   in - kappa^2 H H in on one parity
          m       M = 1 - kappa H, or its adjoint ("dagger")
          batch   H on several lattices in one call
          cg      conjugate gradient on M^+ M x = b
          dropin  the reference's own two calls, eo then oe, on host arrays
  L       extents "x,y,z,t" ("batch": several, separated by spaces)
  prec    storage of fields and links: f64, f32 or f16 ("cg": of the inner
          iteration; the outer one is f64)
  links   18 or 12 reals per link
  rhs     right-hand sides
  mode    wilson (the operator as written down) or compat (as the reference
          computes it), where the call takes a mode
"""
import math

import numpy as np
import torch

from plqcd_amd import hopping as hp
from plqcd_amd import solver

PREC = {"f64": hp.PREC_F64, "f32": hp.PREC_F32, "f16": hp.PREC_F16}
MODE = {"wilson": hp.HOP_WILSON, "compat": hp.HOP_COMPAT}
KAPPA = 0.124
TOL = 1e-10


def listed():
    return [
        # The smallest lattice the benchmark configurations name, applied as
        # the reference's harness does: two kernels of a few microseconds, so
        # the calls and the launches are what is paid for.
        _case("halves_f64_8c16", "halves", "8,8,8,16"),
        # The operator at the size the headline is quoted on.
        _case("hop_f64_32c64", "hop", "32,32,32,64"),
        # An ordinary lattice whose extents are no powers of two, in single
        # precision, one source.
        _case("hop_f32_24c48", "hop", "24,24,24,48", prec="f32"),
        # A propagator's twelve sources at once in double precision.
        _case("hop_f64_24c48_12rhs", "hop", "24,24,24,48", rhs=12),
        # The inner operator of the batched mixed-precision solve: half
        # precision, 12-real links, twelve sources, at the benchmark's size.
        _case("hop_f16_32c64_12rhs", "hop", "32,32,32,64", prec="f16", links=12, rhs=12),
        # The parity halves in turn, as the reference's harness applies them,
        # on extents that share no large power of two, the reference's output.
        _case("halves_f64_compat_ragged", "halves", "28,20,36,44", mode="compat"),
        # The even-odd operator that a preconditioned solver iterates.
        _case("schur_f64_32c64", "schur", "32,32,32,64"),
        # M^+ on a few sources in single precision with 12-real links on a
        # small ragged lattice.
        _case("mdag_f32_ragged_4rhs", "m", "12,20,18,30", prec="f32", links=12, rhs=4, dagger=True),
        # Independent ensembles of different volumes in one call.
        _case("batch_f32_4rhs", "batch", "8,8,8,16 16,16,16,32 20,20,20,40 24,24,24,48", prec="f32", links=12, rhs=4),
        # A whole double-precision solve on a small lattice, where latency
        # between the iteration's launches shows.
        _case("cg_f64_16c32", "cg", "16,16,16,32"),
        # A whole mixed-precision solve for twelve sources.
        _case("cg_f16_24c48_12rhs", "cg", "24,24,24,48", prec="f16", links=12, rhs=12),
        # A program of the reference that has only replaced its calls: host
        # arrays in and out, links not kept between calls.
        _case("dropin_24c48", "dropin", "24,24,24,48", mode="compat"),
    ]


def _case(name, path, L, prec="f64", links=18, rhs=1, mode="wilson", dagger=False):
    c = {"path": path, "L": L, "prec": prec, "links": links, "rhs": rhs, "mode": mode, "dagger": dagger}
    return dict(c, name=name) if name else c


def draw(rng):
    """Another call of the same kinds: any even extents, some ten thousand to two million sites."""
    path = rng.choice(["hop", "hop", "hop", "halves", "schur", "m", "batch", "cg", "dropin"])
    fmt = [("f64", 18), ("f64", 12), ("f32", 18), ("f32", 12), ("f16", 18), ("f16", 12)]
    prec, links = ("f64", 18) if path == "dropin" else rng.choice(fmt)
    rhs = 1 if path == "dropin" else rng.choice([1, 1, 1, 2, 3, 4, 6, 8, 12])
    # sites times sources
    most = {"cg": 24**3 * 48 * 8, "dropin": 24**3 * 40}.get(path, 32**3 * 64 * 4)
    least = {"batch": 8**3 * 16 * rhs}.get(path, 12**3 * 24)
    n = math.exp(rng.uniform(math.log(least), math.log(most)))
    if path == "batch":
        k = rng.randint(2, 6)
        L = " ".join(_extents(rng, n * f / rhs) for f in ([1 / k] * k if rng.random() < 0.3 else _shares(rng, k)))
    else:
        L = _extents(rng, min(n / rhs, 32**3 * 64))
    mode = rng.choice(["wilson", "wilson", "compat"]) if path in ("hop", "halves", "batch") else "wilson"
    if path == "dropin":
        mode = "compat"
    return _case(None, path, L, prec, links, rhs, mode, path == "m" and rng.random() < 0.5)


def _shares(rng, k):
    w = [math.exp(rng.uniform(0, 3)) for _ in range(k)]
    return [x / sum(w) for x in w]


def _extents(rng, sites):
    """Even extents of at least 4 whose volume is near `sites` and not above it (4^4 at least)."""
    sites = max(sites, 256.0)
    for _ in range(1000):
        side = (sites / 2) ** 0.25
        d = [max(4, 2 * round(side * math.exp(rng.uniform(-0.5, 0.5)) / 2)) for _ in range(3)]
        t = 2 * int(sites / (d[0] * d[1] * d[2]) / 2)
        if 4 <= t <= 128:
            return "%d,%d,%d,%d" % (d[0], d[1], d[2], t)
    return "4,4,4,4"


def _lattices(case):
    return [tuple(int(x) for x in L.split(",")) for L in case["L"].split()]


# ------------------------------------------------------------------ inputs
#
# Sites are in the repository's even-odd order: all even sites, then all odd
# ones, each in the order of the lexicographic index (x fastest).


def _links(V, gen):
    """Random SU(3) links (V, 4, 3, 3): two rows orthonormalised, the third their cross product."""
    a = torch.randn(V, 4, 3, dtype=torch.complex128, device="cuda", generator=gen)
    b = torch.randn(V, 4, 3, dtype=torch.complex128, device="cuda", generator=gen)
    a /= torch.linalg.vector_norm(a, dim=-1, keepdim=True)
    b -= (a.conj() * b).sum(-1, keepdim=True) * a
    b /= torch.linalg.vector_norm(b, dim=-1, keepdim=True)
    return torch.stack([a, b, torch.linalg.cross(a, b).conj()], dim=2).resolve_conj()


def _source(V, gen):
    return torch.randn(V, 4, 3, dtype=torch.complex128, device="cuda", generator=gen)


def _inputs(case, seed):
    """(extents, links, function giving the sources one by one) of each lattice of the case."""
    for k, L in enumerate(_lattices(case)):
        gen = torch.Generator(device="cuda").manual_seed(1000 * int(seed) + k)
        V = math.prod(L)
        u = _links(V, gen)
        yield L, u, lambda V=V, gen=gen: _source(V, gen)


def _kappas(case):
    """Sources of one call may belong to different quark masses."""
    return [KAPPA - 0.002 * (r % 3) for r in range(case["rhs"])]


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


# ---------------------------------------------------------------- the calls


class _OnDevice(list):
    """Device fields that a call wrote, as host arrays when they are looked at.

    The calls leave their results on the GPU, where a program goes on with
    them; a program that wants numbers downloads a field.  So does this list,
    when its elements are read: an array for each source of each field, in the
    type that the field is stored in, the parity half `half` of it only where
    the call writes no other."""

    def __init__(self, fields):
        super().__init__((f, r, half) for f, half in fields for r in range(f.nrhs))

    def __iter__(self):
        for f, r, half in super().__iter__():
            a = f.download(r)
            if half is not None:
                a = a[half * (len(a) // 2) : (half + 1) * (len(a) // 2)]
            if f.prec == hp.PREC_F64:
                yield a
            elif f.prec == hp.PREC_F32:
                yield a.astype(np.complex64)
            else:
                yield np.ascontiguousarray(a).view(np.float64).astype(np.float16)

    def __getitem__(self, i):
        return list(self)[i]


def prepare(case, seed):
    path, prec, rhs = case["path"], PREC[case["prec"]], case["rhs"]
    if path == "dropin":
        L, u, source = next(_inputs(case, seed))
        if hp.plqcd_g().init != 1 or tuple(hp.plqcd_g().latdims) != L:
            hp.init_dims(L)
        hp.set_mode(MODE[case["mode"]])
        return {"case": case, "u": _host(u), "in": _host(source()), "out": hp.spinor_field(math.prod(L))}
    state = {"case": case, "lat": [], "gauge": [], "sloppy": [], "in": [], "out": [], "tmp": []}
    field_prec = hp.PREC_F64 if path == "cg" else prec
    stream = None
    for L, u, source in _inputs(case, seed):
        lat = hp.Lattice(L)
        if path == "batch":  # the lattices of a batch share a stream
            stream = stream or hp.lib().plqcd_hip_lattice_stream(lat.h)
            lat.set_stream(stream)
        u = _host(u)
        state["lat"].append(lat)
        if path == "cg":
            state["gauge"].append(hp.Gauge(lat).upload(u))
            same = case["prec"] == "f64" and case["links"] == 18
            state["sloppy"].append(None if same else hp.Gauge(lat, prec, case["links"]).upload(u))
        else:
            state["gauge"].append(hp.Gauge(lat, prec, case["links"]).upload(u))
        f = hp.Field(lat, field_prec, rhs)
        for r in range(rhs):
            f.upload(_host(source()), r)
        state["in"].append(f)
        state["out"].append(hp.Field(lat, field_prec, rhs))
        if path == "schur":
            state["tmp"].append(hp.Field(lat, field_prec, rhs))
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "dropin":
        hp.hopping_matrix_eo(state["in"], state["out"], state["u"])
        hp.hopping_matrix_oe(state["in"], state["out"], state["u"])
        return state["out"]
    if path == "batch":
        hp.hop_batch(state["gauge"], state["in"], state["out"], MODE[case["mode"]])
        return _OnDevice([(f, None) for f in state["out"]])
    g, fin, fout = state["gauge"][0], state["in"][0], state["out"][0]
    if path == "hop":
        hp.hop(g, fin, fout, hp.PARITY_ALL, MODE[case["mode"]])
    elif path == "halves":
        hp.hop(g, fin, fout, hp.PARITY_EVEN, MODE[case["mode"]])
        hp.hop(g, fin, fout, hp.PARITY_ODD, MODE[case["mode"]])
    elif path == "m":
        solver.apply_m(g, fin, fout, _kappas(case), case["dagger"])
    elif path == "schur":
        tmp = state["tmp"][0]
        solver.apply_schur(g, fin, tmp, fout, _kappas(case), 0)
        return _OnDevice([(fout, 0), (tmp, 1)])
    else:
        stats = solver.cg_solve(g, fin, fout, _kappas(case), TOL, sloppy=state["sloppy"][0])
        return {"converged": [s["converged"] for s in stats], "x": _OnDevice([(fout, None)])}
    return _OnDevice([(fout, None)])


# ------------------------------------------------------------------- costs


def work(case):
    """Each link, source and result once; 1320 flop for H at a site."""
    flops = bytes_ = 0.0
    spinor = {"f64": 192, "f32": 96, "f16": 52}[case["prec"]]
    link = case["links"] * {"f64": 8, "f32": 4, "f16": 2}[case["prec"]]
    rhs = case["rhs"]
    for L in _lattices(case):
        V = math.prod(L)
        h = 1320.0 * V * rhs
        if case["path"] == "cg":
            # about 50 iterations of two applications of H, each of which
            # reads the links and a field and writes one, and 4 reads or
            # writes of a field more
            bytes_ += 50.0 * V * (2 * (4 * link + 2 * spinor * rhs) + 4 * spinor * rhs)
            flops += 100.0 * h
        elif case["path"] == "schur":
            # the links once (both hops use all of them), half a source, half
            # the result, and the other parity's half in between
            bytes_ += V * (4 * link + 1.5 * spinor * rhs)
            flops += h
        else:
            bytes_ += V * (4 * link + 2 * spinor * rhs)
            flops += h
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------- 64-bit results
#
# The operator from its definition with explicit gamma matrices, on the GPU
# through plain torch:
#   (H psi)(x) = sum_mu U_mu(x) (1 - gamma_mu) psi(x+mu)
#                     + U_mu(x-mu)^+ (1 + gamma_mu) psi(x-mu)

# gamma_mu psi: component s is GAMMA[mu][s][1] * psi[GAMMA[mu][s][0]]
GAMMA = (
    ((2, -1), (3, -1), (0, -1), (1, -1)),
    ((3, -1j), (2, -1j), (1, 1j), (0, 1j)),
    ((3, -1), (2, 1), (1, 1), (0, -1)),
    ((2, -1j), (3, 1j), (0, 1j), (1, -1j)),
)


def _neighbours(L):
    """Index in even-odd order of the site at +mu and at -mu, for each mu and site."""
    x = torch.meshgrid(*[torch.arange(L[m], device="cuda") for m in (3, 2, 1, 0)], indexing="ij")
    x = [c.reshape(-1) for c in reversed(x)]  # x, y, z, t of each site in lexicographic order

    def index(c):
        lex = c[0] + L[0] * (c[1] + L[1] * (c[2] + L[2] * c[3]))
        return lex // 2 + (sum(c) & 1) * (math.prod(L) // 2)

    me = index(x)
    out = []
    for mu in range(4):
        for step in (1, -1):
            c = list(x)
            c[mu] = (c[mu] + step) % L[mu]
            n = torch.empty_like(me)
            n[me] = index(c)
            out.append(n)
    return out


class _Operator:
    def __init__(self, L, u, compat=False):
        self.u, self.n, self.compat = u, _neighbours(L), compat
        self.half = math.prod(L) // 2

    def h(self, psi, dagger=False):
        out = torch.zeros_like(psi)
        for mu in range(4):
            u = self.u[:, mu]
            up, dn = self.n[2 * mu], self.n[2 * mu + 1]
            # forward: the reference takes the even site's links on odd sites,
            # and lets these terms reach the two upper components only
            uf = torch.cat([u[: self.half], u[: self.half]]) if self.compat else u
            f = self._project(psi[up], mu, 1 if dagger else -1)
            f = self._multiply(uf, f, False)
            if self.compat:
                f[:, 2:] = 0
            out += f
            out += self._multiply(u[dn], self._project(psi[dn], mu, -1 if dagger else 1), True)
        return out

    def m(self, psi, kappa, dagger=False):
        return psi - kappa * self.h(psi, dagger)

    @staticmethod
    def _project(f, mu, sign):
        g = torch.stack([f[:, s] * p for s, p in GAMMA[mu]], dim=1)
        return f + sign * g

    @staticmethod
    def _multiply(u, f, dagger):
        u = u.conj().transpose(1, 2) if dagger else u
        return sum(u[:, None, :, b] * f[:, :, b, None] for b in range(3))

    def solve(self, b, kappa):
        """x with M^+ M x = b, to the last digits that 64 bits give."""
        x, r = torch.zeros_like(b), b.clone()
        p, rr = r.clone(), float(torch.linalg.vector_norm(r)) ** 2
        stop = 1e-28 * rr
        for _ in range(500):
            q = self.m(self.m(p, kappa), kappa, True)
            alpha = rr / float((p.conj() * q).sum().real)
            x += alpha * p
            r -= alpha * q
            new = float(torch.linalg.vector_norm(r)) ** 2
            if new < stop:
                break
            p = r + (new / rr) * p
            rr = new
        return x


def exact(case, seed):
    path, kappas = case["path"], _kappas(case)
    sites = sum(math.prod(L) for L in _lattices(case)) * case["rhs"]
    if path == "cg" and sites > 24**3 * 48 * 12:
        return None
    per_rhs, second = [], []
    for L, u, source in _inputs(case, seed):
        op = _Operator(L, u, case["mode"] == "compat")
        half = op.half
        for r in range(case["rhs"]):
            psi = source()
            if path == "m":
                out = op.m(psi, kappas[r], case["dagger"])
            elif path == "schur":
                even = psi.clone()
                even[half:] = 0
                mid = op.h(even)  # lives on the odd sites
                second.append(mid[half:].cpu())
                out = (even - kappas[r] ** 2 * op.h(mid))[:half]
            elif path == "cg":
                out = op.solve(psi, kappas[r])
            else:
                out = op.h(psi)
            per_rhs.append(out.cpu())
    if path == "dropin":
        return per_rhs[0]
    if path == "cg":
        return {"converged": [None] * case["rhs"], "x": per_rhs}
    return per_rhs + second
