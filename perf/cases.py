"""The timed work of this package: operator applications, solves, a force step and served
batches, as a program that uses hila_amd.wilson makes them.

A case is a dict of plain values:
    kind   "op"     one application of the hopping term ("hop"), M ("M") or M^dag ("Mdag")
           "cg"     one solve of M^dag M x = b from x = 0, to `tol`
           "force"  one HMC fermion force step from psi = 0 (solve, force, momentum update)
           "serve"  one closed batch of requests through the solve server
    dims   the lattice "LxXLyXLzXLt" ("serve": several, one request each, with "/" between)
    prec   storage of the operator's fields (op), or the inner precision of the solve
    rhs    right-hand sides ("serve": per request, with "/" between)
    mh     Hasenbusch shift

Links are random special unitary matrices near 1, sources and momenta are Gaussian, as in the
package's tests and benchmark.  Fields stay on the device between the calls of a program, so
the outputs are the state's own device fields; `Fields` copies one to the host when its value
is asked for.
"""
import math

import numpy as np
import torch

from hila_amd import wilson as W

KAPPA = 0.125
TOL = 1e-10
PREC = {"f64": W.F64, "f32": W.F32, "f16": W.F16}
HOST = {"f64": np.float64, "f32": np.float32, "f16": np.float16}
SPINOR = {"f64": 192, "f32": 96, "f16": 52}   # bytes of a stored Wilson vector
LINK = {"f64": 144, "f32": 72, "f16": 36}     # bytes of a stored link
ITERATIONS = 60                               # a solve of these links to 1e-10 takes about this many


def listed():
    def case(name, kind, dims, prec, **more):
        return dict(dict(name=name, kind=kind, op="", dims=dims, prec=prec, rhs="1", mh=0.0), **more)

    return [
        # the smallest lattice of the tests: an operator call is launches and latency
        case("M 8^4 f64", "op", "8x8x8x8", "f64", op="M"),
        # a lattice whose time slices are no whole number of 64-site waves, the inner operator
        # of a mixed-precision solve
        case("Mdag 20^3x40 f32", "op", "20x20x20x40", "f32", op="Mdag"),
        # the benchmark's hopping term
        case("hop 32^4 f64", "op", "32x32x32x32", "f64", op="hop"),
        # the largest lattice of the benchmark
        case("M 48^3x96 f64", "op", "48x48x48x96", "f64", op="M"),
        # many sources at once: a propagator's twelve spin-colour columns, and a small group
        case("M 32^4 f16 12 rhs", "op", "32x32x32x32", "f16", op="M", rhs="12"),
        case("Mdag 24^3x48 f32 5 rhs", "op", "24x24x24x48", "f32", op="Mdag", rhs="5"),
        # solves: the smallest lattice, the benchmark's in FP64 and with FP32 inside, and a
        # propagator with FP16 inside
        case("cg 8^4 f64", "cg", "8x8x8x8", "f64"),
        case("cg 32^4 f64", "cg", "32x32x32x32", "f64"),
        case("cg 24^3x48 f32", "cg", "24x24x24x48", "f32"),
        case("cg 24^3x48 f16 12 rhs", "cg", "24x24x24x48", "f16", rhs="12"),
        # one force step of HMC, for the first of two Hasenbusch terms
        case("force 16^3x32 f64", "force", "16x16x16x32", "f64", mh=0.1),
        # requests of several sizes at once
        case("serve 8 requests f16", "serve",
             "16x16x16x16/24x24x24x48/16x16x16x16/16x16x16x32/24x24x24x24/16x16x16x32/16x16x16x16/24x24x24x48",
             "f16", rhs="4/1/6/12/5/2/1/4"),
    ]


def draw(rng):
    """A case of the same ranges: lattices of 8^4 to 2^20 sites with even, mostly unequal
    extents (an operator alone up to four times that), every precision and direction."""
    def lattice(lo, hi):
        while True:
            v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
            side = v ** 0.25
            d = [2 * max(2, round(side * math.exp(rng.uniform(-0.35, 0.35)) / 2)) for _ in range(4)]
            if lo <= math.prod(d) <= hi and max(d) <= 96:
                return "x".join(str(x) for x in d)

    kind = rng.choice(["op", "op", "op", "cg", "cg", "force", "serve"])
    prec = rng.choice(["f64", "f32", "f16"])
    case = dict(kind=kind, op="", dims="", prec=prec, rhs="1", mh=0.0)
    if kind == "op":
        rhs = rng.choice([1, 1, 1, 2, 3, 4, 6, 7, 12])
        case.update(op=rng.choice(["hop", "M", "Mdag"]), rhs=str(rhs), dims=lattice(4096, (1 << 22) // rhs))
    elif kind == "cg":
        rhs = rng.choice([1, 1, 2, 3, 6, 8])
        case.update(rhs=str(rhs), dims=lattice(4096, (1 << 20) // rhs), mh=rng.choice([0.0, 0.0, 0.1]))
    elif kind == "force":
        case.update(prec=rng.choice(["f64", "f32"]), dims=lattice(4096, 1 << 19), mh=rng.choice([0.0, 0.1]))
    else:
        n = rng.randint(3, 8)
        sizes = [lattice(8192, 1 << 18) for _ in range(3)]
        case.update(prec=rng.choice(["f32", "f16"]), dims="/".join(rng.choice(sizes) for _ in range(n)),
                    rhs="/".join(str(rng.choice([1, 2, 3, 4, 6])) for _ in range(n)))
    return case


# ------------------------------------------------------------------------- inputs ------

def _dims(text):
    return tuple(int(x) for x in text.split("x"))


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)


def _links(gen, V):
    """(4, V, 3, 3) special unitary matrices near 1: rows of 1 + 0.3 i H, H Hermitian with
    Gaussian entries, orthonormalised."""
    out = torch.empty((4, V, 3, 3), dtype=torch.complex128, device="cuda")
    for mu in range(4):
        a = torch.view_as_complex(_normal(gen, V, 3, 3, 2))
        h = (a + a.mH) * 0.5
        u = torch.eye(3, dtype=torch.complex128, device="cuda") + 0.3j * h
        r0 = u[:, 0] / torch.linalg.vector_norm(u[:, 0], dim=-1, keepdim=True)
        r1 = u[:, 1] - (r0.conj() * u[:, 1]).sum(-1, keepdim=True) * r0
        r1 = r1 / torch.linalg.vector_norm(r1, dim=-1, keepdim=True)
        out[mu, :, 0], out[mu, :, 1], out[mu, :, 2] = r0, r1, torch.linalg.cross(r0, r1).conj()
    return out


def _spinors(gen, n, Vh):
    """(n, Vh, 4, 3) Gaussian Wilson vectors on one parity."""
    return torch.view_as_complex(_normal(gen, n, Vh, 4, 3, 2))


def _inputs(case, seed):
    """[(dims, links, source vectors)] of the case, one entry per lattice (per request)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1 + 1000003 * seed)
    found = []
    for text, n in zip(case["dims"].split("/"), case["rhs"].split("/")):
        d = _dims(text)
        V = math.prod(d)
        found.append((d, _links(gen, V), _spinors(gen, int(n), V // 2)))
    return found


def _momentum(seed, V):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2 + 1000003 * seed)
    a = torch.view_as_complex(_normal(gen, 4, V, 3, 3, 2))
    return _antihermitian(a)


def _real(t):
    """Complex matrices or spinors as the host layout's rows of (re, im) pairs."""
    return torch.view_as_real(t).reshape(t.shape[:-2] + (-1,)).cpu().numpy()


# ---------------------------------------------------------------------------- run ------

class Fields(dict):
    """Outputs where the pass left them: a device field is copied to the host when its value
    is asked for."""

    def __getitem__(self, key):
        return dict.__getitem__(self, key)()


def _reader(field, j, prec):
    return lambda: field.download(j).astype(HOST[prec], copy=False)


def prepare(case, seed):
    found = _inputs(case, seed)
    if case["kind"] == "serve":
        return _prepare_serve(case, found)
    (d, links, source), = found
    prec, n, mh = case["prec"], source.shape[0], case["mh"]
    lat = W.Lattice(d)
    lat.upload_gauge(_real(links))
    D = W.Dirac_Wilson_evenodd(KAPPA, lat)
    A = W.Hasenbusch_operator(D, mh) if mh else D
    fprec = PREC[prec] if case["kind"] == "op" else W.F64
    fin = W.Field(lat, W.EVEN, fprec, n)
    fout = W.Field(lat, W.ODD if case["op"] == "hop" else W.EVEN, fprec, n)
    for j in range(n):
        fin.upload(_real(source[j]), j)
    s = dict(case=case, lat=lat, A=A, fin=fin, fout=fout)
    outs = Fields((f"x{j}", _reader(fout, j, prec if case["kind"] == "op" else "f64")) for j in range(n))
    if case["kind"] == "cg":
        s["cg"] = W.CG(A, TOL, 2000, precision=prec, delta=0.01 if prec == "f16" else 1e-3)
    elif case["kind"] == "force":
        lat.upload_momentum(_real(_momentum(seed, lat.V)))
        outs["momentum"] = lat.download_momentum
    s["outs"] = outs
    return s


def _prepare_serve(case, found):
    """A server with its slots in place, and the requests' page-locked arrays."""
    server = W.Server()
    largest = {}
    for d, _, source in found:
        n, count = largest.get(d, (0, 0))
        largest[d] = (max(n, source.shape[0]), min(count + 1, 6))
    for d, (n, count) in largest.items():
        server.provision(d, n, count, precision=case["prec"])
    requests = []
    for d, links, source in found:
        gauge = W.HostBuffer((4, math.prod(d), 18))
        src = W.HostBuffer((source.shape[0], math.prod(d) // 2, 24))
        sol = W.HostBuffer(src.shape)
        gauge.array[:] = _real(links)
        src.array[:] = _real(source)
        sol.array[:] = 0.0
        requests.append((d, gauge, src, sol))
    # a page-locked array is its buffer's memory: the outputs keep the buffers
    outs = Fields((f"x{i}", lambda sol=sol: sol.array) for i, (_, _, _, sol) in enumerate(requests))
    return dict(case=case, server=server, requests=requests, outs=outs)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "op":
        {"hop": s["A"].hop_set, "M": s["A"].apply, "Mdag": s["A"].dagger}[case["op"]](s["fin"], s["fout"])
        return s["outs"]
    if kind == "cg":
        s["fout"].zero()
        s["cg"].apply(s["fin"], s["fout"], raise_on_noconv=True)
        return s["outs"]
    if kind == "force":
        s["fout"].zero()
        W.force_step(s["A"], s["fin"], s["fout"], 0.05, accuracy=TOL, maxiters=2000, precision=case["prec"],
                     delta=1e-3)
        return s["outs"]
    server, prec = s["server"], case["prec"]
    tickets = [server.submit(d, gauge.array, src.array, sol.array, KAPPA, TOL, maxiters=2000, precision=prec,
                             delta=0.01 if prec == "f16" else 1e-3)
               for d, gauge, src, sol in s["requests"]]
    for t in tickets:
        result, _ = server.wait(t)
        if result["status"] != W.WL_OK:
            raise RuntimeError(result["message"])
    return s["outs"]


def work(case):
    """Bytes and operations that a pass cannot do without.  An operator: every link and the
    input once in, the output once out, 1320 operations a site for a half-lattice hop.  A
    solve: per iteration M and M^dag over links read once, and r, p, x read and written."""
    total = {"bytes": 0.0, "flops": 0.0}
    prec, kind = case["prec"], case["kind"]
    for text, n in zip(case["dims"].split("/"), case["rhs"].split("/")):
        vh, n = math.prod(_dims(text)) // 2, int(n)
        links = 8 * vh * LINK[prec]
        if kind == "op":
            total["bytes"] += links + 2 * n * vh * SPINOR[prec]
            total["flops"] += n * vh * (1320 if case["op"] == "hop" else 2 * 1320 + 48)
        else:
            its = ITERATIONS * (0.75 if case["mh"] else 1.0)
            total["bytes"] += its * (links + 6 * n * vh * SPINOR[prec])
            total["flops"] += its * n * vh * (4 * 1320 + 2 * 48 + 8 * 24)
        if kind == "force":
            total["bytes"] += 3 * 8 * vh * 144 + 4 * vh * 192
    return total


# -------------------------------------------------------------------------- exact ------
# The operator in plain torch, complex128, on checkerboarded arrays (..., T, Z, Y, X/2): a
# site's index within its parity is its lexicographic index (x fastest) halved.

def _antihermitian(m):
    a = (m - m.mH) * 0.5
    tr = torch.diagonal(a, dim1=-2, dim2=-1).sum(-1) / 3.0
    return a - tr[..., None, None] * torch.eye(3, dtype=m.dtype, device=m.device)


class Exact:
    # (1 + s g_mu) w: the two upper rows are w_a + s c w_b, the lower ones follow from them.
    # Per direction: for upper rows 0, 1 the row b and the factor c; for lower rows 2, 3 the
    # upper row and the factor.
    UP = (((3, 1j), (2, 1j)), ((3, -1.0), (2, 1.0)), ((2, 1j), (3, -1j)), ((2, 1.0), (3, 1.0)))
    LOW = (((1, -1j), (0, -1j)), ((1, 1.0), (0, -1.0)), ((0, -1j), (1, 1j)), ((0, 1.0), (1, 1.0)))

    def __init__(self, dims, links, kappa, mh=0.0):
        Lx, Ly, Lz, Lt = dims
        self.shape = (Lt, Lz, Ly, Lx // 2)
        self.kappa, self.mh = kappa, mh
        vh = math.prod(dims) // 2
        # colour and matrix indices first, sites last
        self.U = [[links[mu, p * vh:(p + 1) * vh].permute(1, 2, 0).reshape((3, 3) + self.shape).contiguous()
                   for mu in range(4)] for p in (0, 1)]
        t, z, y = (torch.arange(n, device=links.device) for n in (Lt, Lz, Ly))
        self.row = ((t[:, None, None] + z[None, :, None] + y[None, None, :]) & 1)[..., None].bool()

    def shift(self, a, mu, fwd, p):
        """a, on parity 1 - p, at x + mu (fwd) or x - mu of the sites x of parity p, with the
        antiperiodic sign of the time edge."""
        if mu == 0:
            # parity p has x = 2 i + (row + p) % 2
            high = self.row if p == 0 else ~self.row
            moved = torch.roll(a, -1 if fwd else 1, -1)
            return torch.where(high if fwd else ~high, moved, a)
        dim = {1: -2, 2: -3, 3: -4}[mu]
        a = torch.roll(a, -1 if fwd else 1, dim)
        if mu == 3:
            a = a.clone() if a._is_view() else a
            a.narrow(-4, self.shape[0] - 1 if fwd else 0, 1).neg_()
        return a

    def half(self, w, mu, s):
        return torch.stack([w[a] + (s * self.UP[mu][a][1]) * w[self.UP[mu][a][0]] for a in (0, 1)])

    def hop(self, w, p, s):
        """H_s w on parity p of w (4, 3, ...) on parity 1 - p."""
        out = torch.zeros_like(w)
        for mu in range(4):
            for fwd in (True, False):
                sg = s if fwd else -s
                if fwd:
                    h = self.shift(self.half(w, mu, sg), mu, True, p)
                    u = self.U[p][mu]
                    v = [u[:, 0] * h[a, 0] + u[:, 1] * h[a, 1] + u[:, 2] * h[a, 2] for a in (0, 1)]
                else:
                    h = self.half(w, mu, sg)
                    u = self.U[1 - p][mu].conj()
                    v = torch.stack([u[0] * h[a, 0] + u[1] * h[a, 1] + u[2] * h[a, 2] for a in (0, 1)])
                    v = self.shift(v, mu, False, p)
                for a in (0, 1):
                    out[a] += v[a]
                    b, c = self.LOW[mu][a]
                    out[2 + a] += (sg * c) * v[b]
        return out

    def M(self, w, s):
        return (1.0 + self.mh) * w - self.kappa ** 2 * self.hop(self.hop(w, 1, s), 0, s)

    def solve(self, b):
        """x with M^dag M x = b, to rounding."""
        x = torch.zeros_like(b)
        bb = b.abs().square().sum()
        for _ in range(2):  # once more from the true residual
            r = b - self.M(self.M(x, 1), -1)
            p, rr = r.clone(), r.abs().square().sum()
            for i in range(1000):
                q = self.M(p, 1)
                alpha = rr / q.abs().square().sum()
                x += alpha * p
                r -= alpha * self.M(q, -1)
                new = r.abs().square().sum()
                p = r + (new / rr) * p
                rr = new
                if i % 10 == 9 and float(rr / bb) < 1e-28:
                    break
        return x

    def into(self, w):
        """(Vh, 4, 3) -> (4, 3, T, Z, Y, X/2)"""
        return w.permute(1, 2, 0).reshape((4, 3) + self.shape).contiguous()

    def out(self, w):
        return _real(w.reshape(4, 3, -1).permute(2, 0, 1).contiguous())

    def force_step(self, chi, momentum, eps):
        """psi and the momentum after momentum += P(U F), F = -2 eps times the derivative of
        Re <M psi, M psi> / 2 by the links."""
        psi = self.solve(chi)
        even = (psi, self.M(psi, 1))
        odd = tuple(-self.kappa * self.hop(f, 1, s) for f, s in zip(even, (1, -1)))
        new = momentum.clone()
        vh = math.prod(self.shape)
        for p, mu in ((p, mu) for p in (0, 1) for mu in range(4)):
            # X of parity p: sum of (1 + s g)a(X + mu) (x) b(X)^dag
            (psi_e, mpsi_e), (t_psi, t_mpsi) = even, odd
            pairs = ((t_mpsi, psi_e, -1), (t_psi, mpsi_e, 1)) if p == 0 else ((psi_e, t_mpsi, 1), (mpsi_e, t_psi, -1))
            F = 0
            for a, b, s in pairs:
                ha = self.shift(self.half(a, mu, s), mu, True, p)
                hb = self.half(b, mu, s)
                F = F + (ha[:, :, None] * hb[:, None].conj()).sum(0)
            F = (-2.0 * eps * self.kappa) * F
            U = self.U[p][mu]
            G = (U[:, :, None] * F[None]).sum(1).reshape(3, 3, vh).permute(2, 0, 1)
            new[mu, p * vh:(p + 1) * vh] += _antihermitian(G)
        return psi, new


def exact(case, seed):
    kind = case["kind"]
    found = _inputs(case, seed)
    sites = sum(math.prod(d) * (1 if kind == "op" else 60 * s.shape[0]) for d, _, s in found)
    if sites > 6e8:  # over about 20 s
        return None
    answers = []
    for d, links, source in found:
        E = Exact(d, links, KAPPA, case["mh"])
        if kind == "force":
            psi, momentum = E.force_step(E.into(source[0]), _momentum(seed, math.prod(d)), 0.05)
            return {"x0": E.out(psi), "momentum": _real(momentum)}
        xs = []
        for w in source:
            w = E.into(w)
            if kind != "op":
                xs.append(E.out(E.solve(w)))
            elif case["op"] == "hop":
                xs.append(E.out(-KAPPA * E.hop(w, 1, 1)))
            else:
                xs.append(E.out(E.M(w, 1 if case["op"] == "M" else -1)))
        answers.append(xs)
    if kind == "serve":
        return {f"x{i}": np.stack(xs) for i, xs in enumerate(answers)}
    return {f"x{j}": x for j, x in enumerate(answers[0])}
