"""The measured cases: what users of the engine have it do, from the smallest
lattice of a spin-dynamics run to the largest one-GPU solves.

A case names a lattice kind, its shape, the number of Chebyshev moments M, the
probing periods (which give the S probe columns), the engine's element type
and vector precision, and what one pass does:

  step         set_H + moments + autodiff_matrix: energy and dE/dH of a new
               Hamiltonian, one time step of a spin- or molecular-dynamics
               loop (R stays, H changes every step)
  solve        moments + autodiff_matrix + stoch_matrix on a held H: energy,
               dE/dH and the density matrix, the full solve of one H
  density      set_H + moments + stoch_matrix: density of states and density
               matrix of a disorder realisation
  conductivity moments2_v1 of the x current on a held H
  serving      several energy-and-force requests of mixed shape through the
               batched engine, all in flight together

Lattices: "square" (one real orbital per site, Anderson disorder), "kondo"
(2 spin orbitals, complex 2x2 blocks, Kondo coupling to random classical
spins, optional Anderson disorder; 2-D or 3-D) and "orbital" (dense complex
blocks of b orbitals, 2-D or 3-D).  Single-precision storage is measured on
the single-precision engine type, double on the double one.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from fastkpm_amd import HipEngine
from fastkpm_amd.engine import EnergyScale, SpMatBsr
from fastkpm_amd.serving import BatchEngine


def _case(name, kind, shape, periods, M, op, dtype="cx_double", prec="fp64", b=2, J=0.0, W=0.0,
          tune=False):
    c = {"kind": kind, "dims": len(shape), "periods": "x".join(map(str, periods)), "M": M,
         "op": op, "dtype": dtype, "prec": prec, "b": b, "J": J, "W": W, "tune": tune}
    for d, n in enumerate(shape):
        c["n%d" % d] = n
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest dynamics run: a 16x16 Kondo lattice, one Langevin step
        # (launches and latency set its time)
        _case("kondo 16x16 step", "kondo", (16, 16), (4, 2), 128, "step", J=2.0),
        # the small scalar lattice at high order: 32x32 tight binding, the full solve
        _case("square 32x32 solve", "square", (32, 32), (4, 4), 500, "solve", b=1),
        # an ordinary dynamics step in single precision on an odd lattice
        _case("kondo 45x42 fp32 step", "kondo", (45, 42), (5, 3), 256, "step", "cx_float", "fp32",
              J=1.0, W=1.0),
        # an ordinary dynamics step in double precision, medium lattice
        _case("kondo 128x128 step", "kondo", (128, 128), (4, 4), 256, "step", J=2.0),
        # real engine, ragged cube, odd column count: density of states and
        # density matrix of an Anderson realisation
        _case("square 31x29x27 density", "square", (31, 29, 27), (3, 3, 3), 200, "density",
              "double", b=1, W=4.0),
        # the large 2-D Kondo lattice (N = 131072, S = 64), double and single
        _case("kondo 256x256 solve", "kondo", (256, 256), (4, 8), 200, "solve", J=2.0),
        _case("kondo 256x256 fp32 solve", "kondo", (256, 256), (4, 8), 200, "solve", "cx_float",
              "fp32", J=2.0),
        # the largest: cubic 64^3 with disorder (N = 524288, S = 128), at an
        # order whose forward vectors do not fit the device; tuned kernels, as
        # long solves on one shape use them
        _case("kondo 64^3 solve", "kondo", (64, 64, 64), (4, 4, 4), 160, "solve", J=1.0, W=4.0,
              tune=True),
        # dense 8x8 orbital blocks (N = 262144, S = 256), single precision
        _case("orbital 32^3 fp32 step", "orbital", (32, 32, 32), (4, 4, 2), 64, "step",
              "cx_float", "fp32", b=8),
        # dense 8x8 blocks on a ragged 3-D lattice, double precision
        _case("orbital 18x15x13 solve", "orbital", (18, 15, 13), (3, 3, 2), 128, "solve", b=8),
        # two-current moments for the conductivity of the 2-D Kondo lattice
        _case("conductivity 192x160", "kondo", (192, 160), (4, 8), 64, "conductivity", J=2.0),
        # a handful of queued requests of mixed shape on the batched engine
        _case("serving 8 requests", "kondo", (48, 48), (4, 4), 256, "serving", J=1.0, W=3.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case of the same ranges (sizes over their logarithm, odd ones among them)."""
    op = rng.choice(["step", "step", "solve", "solve", "density", "conductivity", "serving"])
    single = rng.random() < 0.4
    M = 2 * int(_log(rng, 32, 256))
    if op == "serving":
        L = rng.randint(32, 96)
        return _case(None, "kondo", (L, L), (4, 4), M, op, J=1.0, W=rng.uniform(0.0, 6.0))
    if op == "conductivity":
        shape = (rng.randint(24, 200), rng.randint(24, 160))
        return _case(None, "kondo", shape, (4, rng.choice([2, 4, 8])), rng.choice([24, 32, 48, 64]),
                     op, "cx_float" if single else "cx_double", "fp32" if single else "fp64",
                     J=rng.uniform(0.5, 2.0))
    kind = rng.choice(["square", "kondo", "kondo", "orbital"])
    dims = rng.choice([2, 3])
    b = {"square": 1, "kondo": 2, "orbital": rng.choice([4, 8, 8])}[kind]
    # orbital rows N = sites * b, within the listed largest solves' cost
    N = _log(rng, 512, 130000 if kind != "orbital" else 50000)
    side = max(5.0, (N / b) ** (1.0 / dims))
    shape = tuple(max(4, int(round(side * rng.uniform(0.8, 1.25)))) for _ in range(dims))
    periods = tuple(rng.choice([2, 3, 4] if dims == 3 else [2, 3, 4, 5]) for _ in range(dims))
    if kind == "orbital":
        periods = tuple(min(p, 3) for p in periods)
    real = kind == "square" and rng.random() < 0.5
    dtype = ("float" if single else "double") if real else ("cx_float" if single else "cx_double")
    return _case(None, kind, shape, periods, M, op, dtype, "fp32" if single else "fp64", b=b,
                 J=rng.uniform(0.5, 2.0) if kind == "kondo" else 0.0,
                 W=rng.uniform(0.0, 4.0) if kind != "orbital" else 0.0)


# --- inputs ------------------------------------------------------------------

_NP = {"float": np.float32, "double": np.float64, "cx_float": np.complex64,
       "cx_double": np.complex128}


def _shape(case):
    return tuple(case["n%d" % d] for d in range(case["dims"]))


@functools.lru_cache(maxsize=16)
def _pattern(shape):
    """Periodic nearest-neighbour pattern with the diagonal: columns (sites x
    degree, each row sorted), the direction of every block (0: on-site,
    +-(d + 1): the neighbour along axis d) and, per axis, the row of the +1
    block and of its partner."""
    idx = np.arange(int(np.prod(shape))).reshape(shape, order="F")
    cols = [idx.reshape(-1, order="F")]
    dirs = [0]
    for d in range(len(shape)):
        for s in (1, -1):
            cols.append(np.roll(idx, -s, axis=d).reshape(-1, order="F"))
            dirs.append(s * (d + 1))
    cols = np.stack(cols, axis=1)
    order = np.argsort(cols, axis=1, kind="stable")
    return np.take_along_axis(cols, order, axis=1).astype(np.int32), np.array(dirs)[order]


def _hamiltonian(case, shape, rng):
    """H of the case's kind and its spectral bounds."""
    b, kind = case["b"], case["kind"]
    cols, dirs = _pattern(shape)
    ns, deg = cols.shape
    val = np.zeros((ns, deg, b, b), dtype=np.complex128)  # [site, block, bj, bi]
    on = val[dirs == 0]
    eye = np.eye(b)
    eps = rng.uniform(-0.5, 0.5, ns) * case["W"]
    on += eps[:, None, None] * eye
    if kind == "orbital":
        X = rng.standard_normal((ns, b, b)) + 1j * rng.standard_normal((ns, b, b))
        on += (X + np.conj(X.transpose(0, 2, 1))) / 2
        val[dirs == 0] = on
        for d in range(len(shape)):
            T = (rng.standard_normal((ns, b, b)) + 1j * rng.standard_normal((ns, b, b))) \
                * math.sqrt(0.5)
            to = cols[dirs == d + 1]
            back = np.empty_like(T)
            back[to] = np.conj(T.transpose(0, 2, 1))
            val[dirs == d + 1] = T.transpose(0, 2, 1)
            val[dirs == -(d + 1)] = back.transpose(0, 2, 1)
        bound = 2.1 * math.sqrt(b * (2 * len(shape) + 1)) + 1.5
    else:
        if kind == "kondo":
            s = rng.standard_normal((ns, 3))
            s /= np.linalg.norm(s, axis=1, keepdims=True)
            J = case["J"]
            on[:, 0, 0] -= J * s[:, 2]
            on[:, 1, 1] += J * s[:, 2]
            on[:, 1, 0] -= J * (s[:, 0] - 1j * s[:, 1])
            on[:, 0, 1] -= J * (s[:, 0] + 1j * s[:, 1])
        val[dirs == 0] = on
        val[dirs != 0] = -1.0 * eye
        bound = 2 * len(shape) + case["J"] + case["W"] / 2 + 0.1
    dt = _NP[case["dtype"]]
    flat = val.reshape(-1)
    flat = flat.astype(dt) if np.issubdtype(dt, np.complexfloating) else flat.real.astype(dt)
    H = SpMatBsr(ns, ns, b, np.repeat(np.arange(ns, dtype=np.int32), deg),
                 np.ascontiguousarray(cols.reshape(-1)),
                 np.arange(0, ns * deg + 1, deg, dtype=np.int32), np.ascontiguousarray(flat))
    return H, EnergyScale(-bound, bound)


def _colours(case, shape):
    """Probing colour of every orbital row: orbital + b * (position modulo the periods)."""
    grids = np.meshgrid(*[np.arange(n) for n in shape], indexing="ij")
    col, mult = np.zeros(int(np.prod(shape)), dtype=np.int64), 1
    for g, p in zip(grids, map(int, case["periods"].split("x"))):
        col += (g.reshape(-1, order="F") % p) * mult
        mult *= p
    b = case["b"]
    return (np.arange(b)[None, :] + b * col[:, None]).reshape(-1)


def _columns(case):
    return case["b"] * math.prod(map(int, case["periods"].split("x")))


def _probes(case, shape, rng):
    """Random-phase probing vectors, one nonzero per orbital row (n x S, column-major)."""
    g = _colours(case, shape)
    dt = _NP[case["dtype"]]
    R = np.zeros((len(g), _columns(case)), dtype=dt, order="F")
    if np.issubdtype(dt, np.complexfloating):
        R[np.arange(len(g)), g] = np.array([1, 1j, -1, -1j])[rng.integers(0, 4, len(g))]
    else:
        R[np.arange(len(g)), g] = np.array([1.0, -1.0])[rng.integers(0, 2, len(g))]
    return R


def _coefficients(M, es, energy):
    """Jackson-damped Chebyshev coefficients of the Fermi function's energy or
    density at mu = 0, kT = 0.05."""
    Mq = 2 * M
    th = np.pi * (np.arange(Mq) + 0.5) / Mq
    x = np.cos(th) * es.mag() + es.avg()
    a = x / 0.05
    f = -0.05 * np.logaddexp(0.0, -a) if energy else 1.0 / (np.exp(np.minimum(a, 700.0)) + 1.0)
    m = np.arange(M)
    Mp = M + 1.0
    jackson = ((Mp - m) * np.cos(np.pi * m / Mp) + np.sin(np.pi * m / Mp) / np.tan(np.pi / Mp)) / Mp
    c = (np.cos(m[:, None] * th[None, :]) @ f) * (2.0 / Mq)
    c[0] *= 0.5
    return jackson * c


def _current(case, shape, H):
    """Current operator i [H, x]: the blocks along the first axis, times i times the step."""
    cols, dirs = _pattern(shape)
    b = case["b"]
    keep = np.abs(dirs) == 1
    blk = np.asarray(H.val).reshape(cols.shape + (b, b))[keep] * \
        (1j * np.sign(dirs[keep]))[:, None, None].astype(_NP[case["dtype"]])
    ns = H.n_rows
    return SpMatBsr(ns, ns, b, np.repeat(np.arange(ns, dtype=np.int32), 2),
                    np.ascontiguousarray(cols[keep].astype(np.int32)),
                    np.arange(0, 2 * ns + 1, 2, dtype=np.int32),
                    np.ascontiguousarray(blk.reshape(-1).astype(_NP[case["dtype"]])))


def _requests(case):
    """The requests of a serving case: lattices around the case's size, 2-D and
    3-D, spin and orbital blocks, of uneven order and column count."""
    L, M = case["n0"], case["M"]
    cube = max(6, int(round((L * L) ** (1.0 / 3.0))))
    out = []
    for k in range(8):
        r = dict(case)
        if k % 4 == 3:
            n = max(4, int(round((L * L / 6.0) ** (1.0 / 3.0))) + k // 4)
            r.update(kind="orbital", b=8, dims=3, n0=n, n1=n, n2=n, periods="2x2x2", J=0.0, W=0.0)
        elif k % 4 == 1:
            r.update(dims=3, n0=cube, n1=cube + 1, n2=cube + 2 + k // 4, periods="3x3x2")
        else:
            r.update(n0=L + 8 * (k // 2), n1=L + 5 * k, periods="4x4" if k % 4 else "3x5")
        r["M"] = 2 * (M // 4 + (M // 16) * k)
        out.append(r)
    return out


def _inputs(case, seed):
    shape = _shape(case)
    rng = np.random.default_rng([int(seed), 17])
    H, es = _hamiltonian(case, shape, rng)
    R = _probes(case, shape, rng)
    return H, es, R


def prepare(case, seed):
    """H, coefficients and an engine holding R (and H, where a pass keeps it)."""
    st = {"op": case["op"], "M": case["M"]}
    if case["op"] == "serving":
        reqs = []
        for k, r in enumerate(_requests(case)):
            H, es, R = _inputs(r, int(seed) * 8 + k)
            rcol = _colours(r, _shape(r)).astype(np.int32)
            rval = np.ascontiguousarray(R[np.arange(len(rcol)), rcol])
            reqs.append((H, es, _coefficients(r["M"], es, True), (rcol, rval, R.shape[1])))
        st["requests"] = reqs
        st["engine"] = BatchEngine(case["prec"], hbm_bytes=4 << 30, max_slots=16)
        return st
    H, es, R = _inputs(case, seed)
    eng = HipEngine(case["dtype"], case["prec"])
    eng.set_R(R)
    if case["op"] in ("solve", "conductivity") or case["tune"]:
        eng.set_H(H, es)
    if case["tune"]:
        eng.autotune()
    st.update(engine=eng, H=H, es=es, cE=_coefficients(case["M"], es, True),
              cF=_coefficients(case["M"], es, False), dE=H.like(), rho=H.like())
    if case["op"] == "conductivity":
        st["jx"] = _current(case, _shape(case), H)
    return st


def run(state):
    """One pass; results in host memory, as the engine returns them."""
    op, eng = state["op"], state["engine"]
    if op == "serving":
        ids = [eng.submit(H, es, c, probing=p) for H, es, c, p in state["requests"]]
        out = [eng.wait(i) for i in ids]
        return [{"mu": r.mu, "energy": r.energy, "dE": r.D} for r in out]
    if op == "conductivity":
        return {"mu2": eng.moments2_v1(state["M"], state["jx"], state["jx"])}
    if op in ("step", "density"):
        eng.set_H(state["H"], state["es"])
    out = {"mu": eng.moments(state["M"])}
    if op in ("step", "solve"):
        eng.autodiff_matrix(state["cE"], state["dE"])
        out["dE"] = state["dE"].val
    if op in ("solve", "density"):
        eng.stoch_matrix(state["cF"], state["rho"])
        out["rho"] = state["rho"].val
    return out


# --- what a pass cannot do without ---------------------------------------------

_LLC = 256 << 20  # last-level cache: a recursion whose vectors fit it need not read them from HBM


def _work_one(case, op):
    ns = math.prod(_shape(case))
    b, S, M = case["b"], _columns(case), case["M"]
    cx = case["dtype"].startswith("cx")
    single = case["prec"] == "fp32"
    v = (4 if single else 8) * (2 if cx else 1)
    deg = 2 * case["dims"] + 1
    vec, hb = ns * b * S * v, ns * deg * b * b * v
    spmm = ns * deg * b * b * S * (8 if cx else 2)  # also one outer product on H's pattern
    stream = 3 * vec > _LLC
    byts, flops = hb + vec + 8 * M, 0
    fwd, bwd = M // 2, M // 2 - 1
    if op == "conductivity":
        return {"bytes": hb + (3 * M * 3 * vec + 2 * M * vec if stream else vec),
                "flops": 3 * M * spmm + ns * b * S * M * M * (8 if cx else 2)}
    flops += fwd * spmm
    byts += fwd * (3 * vec + hb) if stream else 0
    if op in ("step", "solve"):
        flops += 2 * bwd * spmm
        byts += hb + (bwd * (6 * vec + hb) if stream else 0)
    if op in ("solve", "density"):
        flops += fwd * spmm
        byts += hb + (fwd * (3 * vec + hb) if stream else 0)
    return {"bytes": byts, "flops": flops}


def work(case):
    if case["op"] != "serving":
        return _work_one(case, case["op"])
    each = [_work_one(r, "step") for r in _requests(case)]
    return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}


# --- the same results in 64 bits, plain torch ------------------------------------

class _Exact:
    """The recursions on one H in 64 bits: vectors (sites, b, S)."""

    def __init__(self, case, H, es, R):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        cols, _ = _pattern(_shape(case))
        ns, deg = cols.shape
        b = case["b"]
        wide = torch.complex128 if case["dtype"].startswith("cx") else torch.float64
        self.b, self.deg = b, deg
        self.cols = torch.from_numpy(cols.astype(np.int64)).to(dev)
        blk = torch.from_numpy(np.asarray(H.val)).to(dev).to(wide).reshape(ns, deg, b, b)
        blk = blk.transpose(2, 3) / es.mag()  # [site, block, bi, bj]
        diag = (self.cols == torch.arange(ns, device=dev)[:, None])
        blk[diag] -= (es.avg() / es.mag()) * torch.eye(b, device=dev, dtype=wide)
        self.blk, self.mag = blk.contiguous(), es.mag()
        self.R = torch.from_numpy(np.ascontiguousarray(R)).to(dev).to(wide).reshape(ns, b, -1)
        self.partner = None

    def mul(self, x, blk=None, cols=None):
        blk = self.blk if blk is None else blk
        cols = self.cols if cols is None else cols
        y = torch.zeros_like(x)
        for d in range(blk.shape[1]):
            g = x[cols[:, d]]
            if self.b >= 4:
                y += torch.matmul(blk[:, d].contiguous(), g)
                continue
            for bi in range(self.b):
                for bj in range(self.b):
                    y[:, bi].addcmul_(blk[:, d, bi, bj, None], g[:, bj])
        return y

    def outer(self, a, c, f, D):
        """D[site, block, bj, bi] += f sum_s a_i conj(c_j)."""
        for d in range(self.deg):
            g = c[self.cols[:, d]].conj().resolve_conj()
            if self.b >= 4:
                D[:, d] += f * torch.matmul(a, g.transpose(1, 2).contiguous()).transpose(1, 2)
                continue
            for bi in range(self.b):
                for bj in range(self.b):
                    D[:, d, bj, bi] += f * (a[:, bi] * g[:, bj]).sum(-1)

    @staticmethod
    def dot(a, c):
        if a.is_complex():
            return (torch.view_as_real(a) * torch.view_as_real(c)).sum().item()
        return (a * c).sum().item()

    def moments(self, M):
        mu = np.zeros(M)
        a0, a1 = self.R, self.mul(self.R)
        mu[0], mu[1] = self.dot(a0, a0), self.dot(a1, a0)
        for m in range(1, M // 2):
            a0, a1 = a1, 2 * self.mul(a1) - a0
            mu[2 * m] = 2 * self.dot(a0, a0) - mu[0]
            mu[2 * m + 1] = 2 * self.dot(a1, a0) - mu[1]
        self.last = (a0, a1)
        return mu

    def autodiff(self, M, c):
        D = torch.zeros_like(self.blk)
        self.outer(self.R, self.R, c[1] - c[3::2].sum(), D)
        am, ap = self.last  # alpha_{M/2-1}, alpha_{M/2}
        if M > 2:
            b1, b2 = 2 * c[M - 1] * am, torch.zeros_like(am)
            for m in range(M // 2 - 1, 0, -1):
                self.outer(am, b1, 2.0, D)
                prev = 2 * self.mul(am) - ap
                new = 2 * self.mul(b1) - b2 + 4 * c[2 * m] * am + 2 * c[2 * m + 1] * ap
                if m > 1:
                    new += 2 * c[2 * m - 1] * prev
                am, ap, b1, b2 = prev, am, new, b1
            self.outer(am, b1, 1.0, D)
        return self.hermitian(D) / self.mag

    def hermitian(self, D):
        if self.partner is None:
            ns = self.cols.shape[0]
            key = self.cols * ns + torch.arange(ns, device=self.cols.device)[:, None]
            own = (torch.arange(ns, device=key.device)[:, None] * ns + self.cols).reshape(-1)
            order = torch.argsort(own)
            self.partner = order[torch.searchsorted(own[order], key.reshape(-1))]
        E = D.reshape(-1, self.b, self.b)
        return ((E + E[self.partner].transpose(1, 2).conj()) / 2).reshape(D.shape)

    def stoch(self, c):
        a0, a1 = self.R, self.mul(self.R)
        xi = c[0] * a0 + c[1] * a1
        for m in range(2, len(c)):
            a0, a1 = a1, 2 * self.mul(a1) - a0
            xi += c[m] * a1
        D = torch.zeros_like(self.blk)
        self.outer(self.R, xi, 0.5, D)
        self.outer(xi, self.R, 0.5, D)
        return D

    def moments2(self, M, jcols, jblk):
        def kept(x, f):
            a0, a1 = x, self.mul(x)
            out = [f(a0).reshape(-1), f(a1).reshape(-1)]
            for _ in range(2, M):
                a0, a1 = a1, 2 * self.mul(a1) - a0
                out.append(f(a1).reshape(-1))
            return torch.stack(out)
        A = kept(self.R, lambda x: x)
        B = kept(self.mul(self.R, jblk, jcols), lambda x: self.mul(x, jblk, jcols))
        return (A.conj().resolve_conj() @ B.transpose(0, 1).contiguous()).cpu().numpy()


def _flat(D):
    return D.reshape(-1).cpu().numpy()


def exact(case, seed):
    if case["op"] == "serving":
        out = []
        for k, r in enumerate(_requests(case)):
            H, es, R = _inputs(r, int(seed) * 8 + k)
            E = _Exact(r, H, es, R)
            c = _coefficients(r["M"], es, True)
            mu = E.moments(r["M"])
            out.append({"mu": mu, "energy": float(np.dot(c, mu)), "dE": _flat(E.autodiff(r["M"], c))})
        return out
    H, es, R = _inputs(case, seed)
    E = _Exact(case, H, es, R)
    del R
    if case["op"] == "conductivity":
        j = _current(case, _shape(case), H)
        cols = torch.from_numpy(j.col_idx.astype(np.int64)).to(E.cols.device).reshape(-1, 2)
        blk = torch.from_numpy(j.val).to(E.blk.device).to(E.blk.dtype)
        b = case["b"]
        return {"mu2": E.moments2(case["M"], cols,
                                  blk.reshape(-1, 2, b, b).transpose(2, 3).contiguous())}
    out = {"mu": E.moments(case["M"])}
    if case["op"] in ("step", "solve"):
        out["dE"] = _flat(E.autodiff(case["M"], _coefficients(case["M"], es, True)))
    if case["op"] in ("solve", "density"):
        out["rho"] = _flat(E.stoch(_coefficients(case["M"], es, False)))
    return out
