"""Performance cases: the calls a lattice-QCD program makes of this package.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs, lattices and networks that such a program holds
    run(state)           one pass through the public entry points, with its outputs
    work(case)           bytes and flops one pass cannot do without
    exact(case, seed)    the outputs in 64 bits from plain torch

Kinds of case:
  hop            Lattice.dslash, FP64, one parity: the operator alone, as analysis
                 code and other solvers call it
  legacy         pyqcu.dslashCloverQcu on both parities of one gauge field: the
                 reference's binding, which is handed the gauge with every call
  mat            Lattice.mat, the full operator (residual checks, other solvers)
  configuration  a new gauge field: Lattice.load_gauge, then the clover hop onto
                 both parities; paid once per configuration of an ensemble
  solve          Lattice.solve of one right-hand side
  propagator     propagator.invert: 12 spin-colour solves from a point source
  batch          Batch.solve over Wilson lattices of several shapes
  learned        Lattice.solve with a LearnedPreconditioner
  train          LearnedPreconditioner.loss_grad: one source's share of a training step

Gauge links scatter around the unit matrix by `eps`; the couplings are those of
the workloads of qcu_amd/configbench.py.  The network computes and stores its
weights in FP32, so its loss and gradient are handed on in FP32.
"""
import math

import numpy as np
import torch

from qcu_amd import propagator, pyqcu
from qcu_amd.lattice import FP16, FP32, FP64, Batch, Lattice, LearnedPreconditioner

PREC = {"fp64": FP64, "fp32": FP32, "fp16": FP16}
CHANNELS = (1, 8, 8, 8, 1)
C128 = torch.complex128
DEVICE = "cuda"


# --------------------------------------------------------------------------- the cases
def _case(name, kind, L, **kw):
    c = {"kind": kind, "L": "x".join(str(v) for v in L), **kw}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a single small hop: what the call itself costs
        _case("hop_wilson_8x8x8x8", "hop", (8, 8, 8, 8), eps=0.3, csw=0.0, parity=0),
        # the operator at the largest usual size of one GPU
        _case("hop_clover_32x32x32x64", "hop", (32, 32, 32, 64), eps=0.2, csw=1.0, parity=1),
        # an existing caller of the reference's binding
        _case("legacy_clover_16x16x16x32", "legacy", (16, 16, 16, 32), eps=0.05),
        # extents that fill neither a wavefront row nor a block
        _case("mat_clover_12x10x14x22", "mat", (12, 10, 14, 22), eps=0.3, csw=1.0),
        # the next configuration of an ensemble
        _case("configuration_24x24x24x48", "configuration", (24, 24, 24, 48), eps=0.25, csw=1.0),
        # many small solves in a row, as in tests and coarse ensembles
        _case("solve_wilson_8x8x8x8", "solve", (8, 8, 8, 8), eps=0.3, csw=0.0, kappa=0.124, prec="fp64", tol=1e-10),
        # the plain FP64 solve of a middle-sized clover lattice
        _case("solve_clover_16x16x16x32", "solve", (16, 16, 16, 32), eps=0.3, csw=1.0, kappa=0.124, prec="fp64",
              tol=1e-10),
        # mixed precision at the headline size, launch shapes tuned beforehand
        _case("solve_mixed_32x32x32x64", "solve", (32, 32, 32, 64), eps=0.2, csw=1.0, kappa=0.1248, prec="fp16",
              tol=1e-12),
        # a quark propagator: the standard measurement
        _case("propagator_24x24x24x48", "propagator", (24, 24, 24, 48), eps=0.25, csw=1.0, kappa=0.1245, prec="fp32",
              tol=1e-12),
        # several ensembles at once
        _case("batch_wilson_mixed_shapes", "batch", (16, 16, 16, 32), eps=0.3, csw=0.0, kappa=0.124, prec="fp32",
              tol=1e-12, each=2),
        # the learned preconditioner inside a mixed-precision solve
        _case("learned_24x24x24x48", "learned", (24, 24, 24, 48), eps=0.25, csw=1.0, kappa=0.1245, prec="fp16",
              tol=1e-12),
        # training the preconditioner: forward, operator, backward, weight gradient
        _case("train_16x16x16x32", "train", (16, 16, 16, 32), eps=0.3, csw=1.0, kappa=0.124),
    ]


def _extents(rng, lo, hi):
    """even extents with a volume spread over [lo, hi] in its logarithm, time the longest on average"""
    while True:
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        side = (v / 1.7) ** 0.25
        L = [max(4, 2 * round(side * math.exp(rng.uniform(-0.3, 0.3)) / 2)) for _ in range(3)]
        L.append(max(4, 2 * round(v / (L[0] * L[1] * L[2]) / 2)))
        if L[3] <= 6 * side and lo <= L[0] * L[1] * L[2] * L[3] <= hi:
            return tuple(L)


def draw(rng):
    kind = rng.choice(["hop", "legacy", "mat", "configuration", "solve", "propagator", "batch", "learned", "train"])
    small, c1, c2, c4 = 8 ** 4, 16 ** 3 * 32, 24 ** 3 * 48, 32 ** 3 * 64
    csw = rng.choice([0.0, 1.0])
    if kind == "hop":
        return _case(None, kind, _extents(rng, small, c4), eps=0.25, csw=csw, parity=rng.randrange(2))
    if kind == "legacy":
        return _case(None, kind, _extents(rng, small, c2), eps=0.05)
    if kind == "mat":
        return _case(None, kind, _extents(rng, small, c4), eps=0.25, csw=csw)
    if kind == "configuration":
        return _case(None, kind, _extents(rng, small, c2), eps=0.25, csw=csw)
    if kind == "solve":
        prec = rng.choice(["fp64", "fp32", "fp16"])
        return _case(None, kind, _extents(rng, small, c4), eps=0.25, csw=csw, kappa=0.124, prec=prec,
                     tol=1e-10 if prec == "fp64" else 1e-12)
    if kind == "propagator":
        return _case(None, kind, _extents(rng, small, c1), eps=0.25, csw=csw, kappa=0.124,
                     prec=rng.choice(["fp32", "fp16"]), tol=1e-12)
    if kind == "batch":
        return _case(None, kind, _extents(rng, 2 * small, c1), eps=0.3, csw=0.0, kappa=0.124,
                     prec=rng.choice(["fp64", "fp32"]), tol=1e-12, each=rng.randint(1, 4))
    if kind == "learned":
        return _case(None, kind, _extents(rng, small, c2), eps=0.25, csw=csw, kappa=0.124, prec="fp16", tol=1e-12)
    return _case(None, kind, _extents(rng, small, c1), eps=0.3, csw=csw, kappa=0.124)


def _lattice_size(case):
    return tuple(int(v) for v in case["L"].split("x"))


def _batch_sizes(case):
    """shapes of a batch: the largest, about a third and about an eighth of its volume"""
    L = _lattice_size(case)
    third = tuple(max(4, 2 * round(v * 0.76 / 2)) for v in L)
    eighth = tuple(max(4, 2 * round(v * 0.59 / 2)) for v in L)
    return [s for s in (eighth, third, L) for _ in range(case["each"])]


# --------------------------------------------------------------------------- inputs
def _half(L):
    return (L[3], L[2], L[1], L[0] // 2)


def _generator(seed, what):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 1000003 + what)
    return g


def _gauge(L, eps, seed, what=0):
    """SU(3) links around the unit matrix: 1 + i eps H with Gaussian Hermitian H,
    rows made orthonormal, the third the conjugate cross product of the others"""
    n = (4, 2) + _half(L)
    g = _generator(seed, what)
    U = torch.empty(n + (3, 3), dtype=C128, device=DEVICE)
    w = eps * torch.randn(n + (8,), generator=g, dtype=torch.float64, device=DEVICE)
    s = 3.0 ** -0.5
    zero = torch.zeros_like(w[..., 0])
    rows = []
    for r in (0, 1):
        re = [torch.ones_like(zero), w[..., 1], w[..., 4]] if r == 0 else [-w[..., 1], torch.ones_like(zero), w[..., 6]]
        im = [w[..., 2] + s * w[..., 7], w[..., 0], w[..., 3]] if r == 0 else [w[..., 0], s * w[..., 7] - w[..., 2], w[..., 5]]
        rows.append(torch.complex(torch.stack(re, -1), torch.stack(im, -1)))
    a, b = rows
    a = a / torch.sqrt((a.abs() ** 2).sum(-1, keepdim=True))
    b = b - (a.conj() * b).sum(-1, keepdim=True) * a
    b = b / torch.sqrt((b.abs() ** 2).sum(-1, keepdim=True))
    U[..., 0, :] = a
    U[..., 1, :] = b
    for k, (i, j) in enumerate(((1, 2), (2, 0), (0, 1))):
        U[..., 2, k] = (a[..., i] * b[..., j] - a[..., j] * b[..., i]).conj()
    return U


def _gaussian(L, seed, what, full=True):
    return torch.randn(((2,) if full else ()) + _half(L) + (4, 3), generator=_generator(seed, what), dtype=C128,
                       device=DEVICE) * 2 ** 0.5


_GAMMA = np.array([[[0, 0, 0, 1j], [0, 0, 1j, 0], [0, -1j, 0, 0], [-1j, 0, 0, 0]],
                   [[0, 0, 0, -1], [0, 0, 1, 0], [0, 1, 0, 0], [-1, 0, 0, 0]],
                   [[0, 0, 1j, 0], [0, 0, 0, -1j], [-1j, 0, 0, 0], [0, 1j, 0, 0]],
                   [[0, 0, 1, 0], [0, 0, 0, 1], [1, 0, 0, 0], [0, 1, 0, 0]]])


def _network_weights(kappa, seed):
    """weights as after training: one channel carries the four linear factors of
    1 + kD + ... + (kD)^4, the truncated hopping series of the inverse, the others noise"""
    rng = np.random.default_rng(int(seed))
    out = []
    for layer in range(len(CHANNELS) - 1):
        shape = (9, CHANNELS[layer + 1], CHANNELS[layer], 4, 4)
        w = 0.005 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
        root = np.exp(2j * np.pi * (layer + 1) / 5)
        for mu in range(4):
            w[2 * mu, 0, 0] -= kappa * root * (np.eye(4) - _GAMMA[mu])
            w[2 * mu + 1, 0, 0] -= kappa * root * (np.eye(4) + _GAMMA[mu])
        w[8, 0, 0] += np.eye(4)
        out.append(w.reshape(-1))
    return np.concatenate(out).astype(np.complex64).astype(np.complex128)


def _point(L, seed):
    """the origin of a propagator, moved from configuration to configuration"""
    rng = np.random.default_rng(int(seed))
    return [int(rng.integers(0, v)) for v in L]


class State:
    pass


def prepare(case, seed):
    s = State()
    s.kind, s.case, L = case["kind"], case, _lattice_size(case)
    s.L = L
    if s.kind == "legacy":
        s.U = _gauge(L, case["eps"], seed)
        s.inp = [_gaussian(L, seed, 1, full=False), _gaussian(L, seed, 2, full=False)]
        s.param = pyqcu.QcuParam()
        s.param.lattice_size = list(L)
        torch.cuda.synchronize()
        return s
    if s.kind == "batch":
        s.lats, s.bs = [], []
        for k, size in enumerate(_batch_sizes(case)):
            lat = Lattice(size, case["kappa"], 0.0, -1)
            U = _gauge(size, case["eps"], seed, 10 + k)
            torch.cuda.synchronize()
            lat.load_gauge(U)
            s.lats.append(lat)
            s.bs.append(_gaussian(size, seed, 100 + k))
        s.batch = Batch(s.lats, [1] * len(s.lats))
        torch.cuda.synchronize()
        return s
    s.lat = Lattice(L, case.get("kappa", 0.124), case["csw"], -1)
    s.U = _gauge(L, case["eps"], seed)
    torch.cuda.synchronize()
    s.lat.load_gauge(s.U)
    if s.kind == "hop":
        s.inp = _gaussian(L, seed, 1, full=False)
    elif s.kind == "configuration":
        s.inp = [_gaussian(L, seed, 1, full=False), _gaussian(L, seed, 2, full=False)]
    elif s.kind == "propagator":
        s.origin = _point(L, seed)
    elif s.kind == "train":
        s.inp = _gaussian(L, seed, 1, full=False)
    else:
        s.inp = _gaussian(L, seed, 1)
    if s.kind in ("learned", "train"):
        s.net = LearnedPreconditioner(s.lat, CHANNELS)
        s.net.set_weights(_network_weights(case["kappa"], seed))
    if case.get("prec") == "fp16":
        s.lat.tune(FP64)
        s.lat.tune(FP16)
    if s.kind != "configuration":
        s.U = None  # the lattice keeps its own links
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------------- one pass
def run(s):
    c, kind = s.case, s.kind
    if kind == "hop":
        return s.lat.dslash(s.inp, parity=c["parity"], clover=c["csw"] != 0, prec=FP64)
    if kind == "legacy":
        out = [torch.empty_like(v) for v in s.inp]
        for p in (0, 1):
            pyqcu.dslashCloverQcu(out[p], s.inp[p], s.U, s.param, p)
        return out
    if kind == "mat":
        return s.lat.mat(s.inp)
    if kind == "configuration":
        s.lat.load_gauge(s.U)
        return [s.lat.dslash(s.inp[p], parity=p, clover=c["csw"] != 0, prec=FP64) for p in (0, 1)]
    if kind == "solve":
        return s.lat.solve(s.inp, tol=c["tol"], prec=PREC[c["prec"]], reliable_delta=0.01)[0]
    if kind == "propagator":
        return propagator.invert(s.lat, "point", s.origin, tol=c["tol"], prec=PREC[c["prec"]])[0]
    if kind == "batch":
        return s.batch.solve(s.bs, tol=c["tol"], prec=PREC[c["prec"]], reliable_delta=0.01)[0]
    if kind == "learned":
        return s.lat.solve(s.inp, tol=c["tol"], prec=FP16, reliable_delta=0.01, precond=s.net)[0]
    loss, grad = s.net.loss_grad(s.inp)
    return {"loss": np.float32(loss), "gradient": grad.astype(np.complex64)}


# --------------------------------------------------------------------------- what a pass cannot do without
# iterations of the solves at these couplings and tolerances (BiCGSTAB, two
# applications of the Schur operator each)
ITERS = {"fp64": 20, "fp32": 24, "fp16": 24}


def _solve_work(L, clover, prec, rhs, iters):
    """FP64 set-up and check, then per iteration two Schur operators (each link and
    clover block once, each vector once) and the recurrence's vectors"""
    vh = L[0] * L[1] * L[2] * L[3] // 2
    real = {"fp64": 8, "fp32": 4, "fp16": 2}[prec]
    field = 24 * real
    operator = 2 * 8 * 12 * real + (2 * 72 * real if clover else 0) + rhs * 2 * field
    vectors = rhs * 9 * field
    setup = 4 * (8 * 12 * 8 + (72 * 8 if clover else 0)) + rhs * 4 * 192
    flops = rhs * (iters * (4 * 1320 + (4 * 504 if clover else 0) + 24 * 24) + 6 * 1320)
    return vh * (iters * (2 * operator + vectors) + setup), vh * flops


def work(case):
    L, kind = _lattice_size(case), case["kind"]
    vh = L[0] * L[1] * L[2] * L[3] // 2
    clover = case.get("csw", 1.0) != 0
    links, block, spinor = 8 * 96, 576 if clover else 0, 192  # bytes per site of one parity, FP64
    hop_flops = 1320 + (504 if clover else 0)
    if kind == "hop":
        return {"bytes": vh * (links + block + 2 * spinor), "flops": vh * hop_flops}
    if kind == "mat":
        return {"bytes": 2 * vh * (links // 2 + block + 2 * spinor), "flops": 2 * vh * (hop_flops + 48)}
    if kind in ("legacy", "configuration"):
        # the external links (3x3) are read; two hops with their clover terms
        build = 2 * (6 * 4 * 3 * 198 + 4000) if clover else 0
        return {"bytes": vh * (8 * 144 + 2 * 2 * spinor), "flops": vh * (2 * hop_flops + build)}
    if kind == "solve":
        b, f = _solve_work(L, clover, case["prec"], 1, ITERS[case["prec"]])
    elif kind == "propagator":
        b, f = _solve_work(L, clover, case["prec"], 12, ITERS[case["prec"]])
    elif kind == "batch":
        each = [_solve_work(size, False, case["prec"], 1, ITERS[case["prec"]]) for size in _batch_sizes(case)]
        b, f = sum(v[0] for v in each), sum(v[1] for v in each)
    else:
        # network: channels of every layer written and read once, links once per layer
        pairs = sum(CHANNELS[k] * CHANNELS[k + 1] for k in range(len(CHANNELS) - 1))
        act = sum(CHANNELS[1:-1])
        net_b = 2 * vh * (2 * act * 96 + 4 * 4 * 48 + 2 * 96)
        net_f = 2 * vh * (pairs * 9 * 4 * 4 * 3 * 8 + sum(CHANNELS[:-1]) * 8 * 4 * 66)
        if kind == "train":
            return {"bytes": 3 * net_b, "flops": 3 * net_f}
        b, f = _solve_work(L, clover, case["prec"], 1, 10)
        b, f = b + 20 * net_b, f + 20 * net_f / 2
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------------------- 64-bit values in plain torch
# fields keep the even-odd layout: [2][t][z][y][x/2][...]
def _shift(f, L, mu, d, p):
    """the value at x + d mu of a field of the other parity, as sites of parity p see it"""
    if mu:
        return torch.roll(f, -d, 3 - mu)
    t, z, y, _ = _half(L)
    i = lambda n, k: torch.arange(n, device=f.device).view([n if a == k else 1 for a in range(4)])  # noqa: E731
    odd = ((i(t, 0) + i(z, 1) + i(y, 2) + p) % 2 == 1).view((t, z, y, 1) + (1,) * (f.dim() - 4))
    moved = torch.roll(f, -d, 3)
    return torch.where(odd, moved, f) if d > 0 else torch.where(odd, f, moved)


def _colour(U, v):
    """U v on the last index of v, any indices between the site and the colour"""
    U = U.reshape(U.shape[:4] + (1,) * (v.dim() - 5) + (3, 3))
    return torch.stack([sum(U[..., a, b] * v[..., b] for b in range(3)) for a in range(3)], -1)


def _dagger(U):
    return U.conj().transpose(-1, -2)


def _sign(v, L, mu, edge, tb):
    if mu == 3 and tb < 0:
        s = torch.ones(L[3], dtype=torch.float64, device=v.device)
        s[edge] = -1
        v = v * s.view((-1,) + (1,) * (v.dim() - 1))
    return v


def _spin(m, v):
    m = np.asarray(m)
    rows = []
    for r in range(4):
        cols = [complex(m[r, k]) * v[..., k, :] for k in range(4) if m[r, k] != 0]
        rows.append(sum(cols[1:], cols[0]))
    return torch.stack(rows, -2)


def _hop(v, U, L, p, tb):
    """D v on the sites of parity p, v on the other parity"""
    out = 0
    for mu in range(4):
        f = _sign(_colour(U[mu, p], _shift(v, L, mu, 1, p)), L, mu, L[3] - 1, tb)
        out = out + _spin(np.eye(4) - _GAMMA[mu], f)
        b = _sign(_shift(_colour(_dagger(U[mu, 1 - p]), v), L, mu, -1, p), L, mu, 0, tb)
        out = out + _spin(np.eye(4) + _GAMMA[mu], b)
    return out


def _mul(a, b):
    return sum(a[..., :, k, None] * b[..., k, None, :] for k in range(3))


def _clover(U, L, coeff):
    """A = 1 - coeff sum sigma F per parity as two 6x6 chiral blocks [2][sites][2][6][6]"""
    def at(F, *moves):  # F at x + moves, on sites of both parities
        for mu, d in moves:
            F = torch.stack([_shift(F[1 - p], L, mu, d, p) for p in (0, 1)])
        return F

    A = torch.zeros((2,) + _half(L) + (2, 2, 3, 2, 3), dtype=C128, device=U.device)
    for mu in range(4):
        for nu in range(mu + 1, 4):
            M, N = U[mu], U[nu]
            Q = _mul(_mul(M, at(N, (mu, 1))), _mul(_dagger(at(M, (nu, 1))), _dagger(N)))
            Q = Q + _mul(_mul(N, _dagger(at(M, (mu, -1), (nu, 1)))), _mul(_dagger(at(N, (mu, -1))), at(M, (mu, -1))))
            Q = Q + _mul(_mul(_dagger(at(M, (mu, -1))), _dagger(at(N, (mu, -1), (nu, -1)))),
                         _mul(at(M, (mu, -1), (nu, -1)), at(N, (nu, -1))))
            Q = Q + _mul(_mul(_dagger(at(N, (nu, -1))), at(M, (nu, -1))), _mul(at(N, (mu, 1), (nu, -1)), _dagger(M)))
            F = (Q - _dagger(Q)) / 8j
            sig = 0.5j * (_GAMMA[mu] @ _GAMMA[nu] - _GAMMA[nu] @ _GAMMA[mu])
            for r in range(4):
                for s in range(4):
                    if sig[r, s] != 0:
                        A[..., r // 2, r % 2, :, s % 2, :] -= coeff * complex(sig[r, s]) * F
    A = A.reshape((2,) + _half(L) + (2, 6, 6))
    return A + torch.eye(6, dtype=C128, device=U.device)


def _inverse6(A):
    """Gauss-Jordan on Hermitian blocks near the unit matrix"""
    A, B = A.clone(), torch.zeros_like(A) + torch.eye(6, dtype=C128, device=A.device)
    for k in range(6):
        d = 1 / A[..., k, k]
        A[..., k, :] = A[..., k, :] * d[..., None]
        B[..., k, :] = B[..., k, :] * d[..., None]
        f = A[..., :, k].clone()
        f[..., k] = 0
        ra, rb = A[..., k, :].clone(), B[..., k, :].clone()
        A -= f[..., :, None] * ra[..., None, :]
        B -= f[..., :, None] * rb[..., None, :]
    return B


def _blocks(A, v):
    """two 6x6 blocks times a spinor"""
    if A is None:
        return v
    w = v.reshape(v.shape[:-2] + (2, 6))
    A = A.reshape(A.shape[:4] + (1,) * (w.dim() - 6) + A.shape[4:])
    return sum(A[..., :, k] * w[..., k, None] for k in range(6)).reshape(v.shape)


class _Operator:
    def __init__(self, U, L, kappa, csw, tb):
        self.U, self.L, self.kappa, self.tb = U, L, kappa, tb
        self.A = _clover(U, L, kappa * csw) if csw else [None, None]
        self.Ai = [_inverse6(a) for a in self.A] if csw else [None, None]

    def hop(self, v, p):
        return _hop(v, self.U, self.L, p, self.tb)

    def mat(self, x):
        return torch.stack([_blocks(self.A[p], x[p]) - self.kappa * self.hop(x[1 - p], p) for p in (0, 1)])

    def schur(self, v):
        k = self.kappa
        return v - k * k * _blocks(self.Ai[1], self.hop(_blocks(self.Ai[0], self.hop(v, 0)), 1))

    def solve(self, b):
        """M x = b, the odd-site system by BiCGSTAB restarted on its recomputed residual"""
        k = self.kappa
        rhs = _blocks(self.Ai[1], b[1] + k * self.hop(_blocks(self.Ai[0], b[0]), 1))
        xo = torch.zeros_like(rhs)
        dot = lambda a, c: complex(torch.vdot(a.reshape(-1), c.reshape(-1)))  # noqa: E731
        norm = math.sqrt(dot(rhs, rhs).real)
        for _ in range(4):
            r = rhs - self.schur(xo)
            start = math.sqrt(dot(r, r).real)
            if start <= 1e-14 * norm:
                break
            r0, p, rho = r.clone(), r.clone(), dot(r, r)
            for _ in range(200):
                v = self.schur(p)
                alpha = rho / dot(r0, v)
                s = r - alpha * v
                t = self.schur(s)
                omega = dot(t, s) / dot(t, t).real
                xo = xo + alpha * p + omega * s
                r = s - omega * t
                if math.sqrt(dot(r, r).real) <= max(1e-7 * start, 2e-15 * norm):
                    break
                new = dot(r0, r)
                p = r + (new / rho) * (alpha / omega) * (p - omega * v)
                rho = new
        xe = _blocks(self.Ai[0], b[0] + k * self.hop(xo, 0))
        return torch.stack([xe, xo])


def _network(x, weights, op):
    """K on [2][sites][channel][4][3]"""
    def mix(w, v):  # w [out][in][4][4]
        o, i = w.shape[:2]
        m = w.permute(0, 2, 1, 3).reshape(o * 4, i * 4)
        u = torch.matmul(m, v.reshape(-1, i * 4, 3).permute(1, 0, 2).reshape(i * 4, -1))
        return u.reshape(o * 4, -1, 3).permute(1, 0, 2).reshape(v.shape[:4] + (o, 4, 3))

    for w in weights:
        out = []
        for p in (0, 1):
            y = mix(w[8], x[p])
            for mu in range(4):
                f = _sign(_colour(op.U[mu, p], _shift(x[1 - p], op.L, mu, 1, p)), op.L, mu, op.L[3] - 1, op.tb)
                b = _sign(_shift(_colour(_dagger(op.U[mu, 1 - p]), x[1 - p]), op.L, mu, -1, p), op.L, mu, 0, op.tb)
                y = y + mix(w[2 * mu], f) + mix(w[2 * mu + 1], b)
            out.append(y)
        x = out
    return x


def exact(case, seed):
    kind, L = case["kind"], _lattice_size(case)
    if kind == "batch":
        out = []
        for k, size in enumerate(_batch_sizes(case)):
            op = _Operator(_gauge(size, case["eps"], seed, 10 + k), size, case["kappa"], 0.0, -1)
            out.append(op.solve(_gaussian(size, seed, 100 + k)))
        return out
    if kind == "propagator" and L[0] * L[1] * L[2] * L[3] > 16 ** 3 * 32:
        return None  # twelve solves take too long
    U = _gauge(L, case["eps"], seed)
    if kind == "legacy":
        op = _Operator(U, L, 1.0, 1.0, 1)
    else:
        op = _Operator(U, L, case.get("kappa", 0.124), case["csw"], -1)
    if kind == "hop":
        p = case["parity"]
        return _blocks(op.Ai[p], op.hop(_gaussian(L, seed, 1, full=False), p))
    if kind in ("legacy", "configuration"):
        return [_blocks(op.Ai[p], op.hop(_gaussian(L, seed, 1 + p, full=False), p)) for p in (0, 1)]
    if kind == "mat":
        return op.mat(_gaussian(L, seed, 1))
    if kind in ("solve", "learned"):
        return op.solve(_gaussian(L, seed, 1))
    if kind == "propagator":
        prop = torch.empty((2,) + _half(L) + (4, 4, 3, 3), dtype=C128, device=DEVICE)
        x, y, z, t = _point(L, seed)
        for s in range(4):
            for c in range(3):
                b = torch.zeros((2,) + _half(L) + (4, 3), dtype=C128, device=DEVICE)
                b[(x + y + z + t) % 2, t, z, y, x // 2, s, c] = 1
                prop[..., :, s, :, c] = 2 * case["kappa"] * op.solve(b)
        return prop
    w = torch.from_numpy(_network_weights(case["kappa"], seed)).to(DEVICE).requires_grad_()
    parts, at = [], 0
    for layer in range(len(CHANNELS) - 1):
        shape = (9, CHANNELS[layer + 1], CHANNELS[layer], 4, 4)
        n = int(np.prod(shape))
        parts.append(w[at:at + n].reshape(shape))
        at += n
    src = _gaussian(L, seed, 1, full=False)
    y = _network([torch.zeros_like(src).unsqueeze(4), src.unsqueeze(4)], parts, op)[1].squeeze(4)
    loss = ((op.schur(y) - src).abs() ** 2).sum() / (src.abs() ** 2).sum()
    loss.backward()
    return {"loss": float(loss), "gradient": w.grad}
