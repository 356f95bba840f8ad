"""Workloads of csipm that are timed: what its users have it do, by entry point.

A case is a dict of plain values: "kind" names the entry point, "dims" the
problem's sizes ("255x255"), "prec" the handle's precision (f64, f32 or
mixed).  Kinds:

  mtm      M_perpt_M_perp_vec, the operator of every solver
  forward  M_perp_beta: a spectrum to its observed samples
  adjoint  M_perpt_z: samples to the spectrum
  kkt      CondensedFFTKKTSystem.mul, one Krylov product of the KKT system
  maps     beta_to_DFT and DFT_to_beta, the packing maps on their own
  newton   FFTKKTSystem.build_kkt and solve_kkt: one Newton system
  solve    ipm_solve of one problem
  batch    solve_batch of a set of uneven problems
  realdata index_missing_from_mask and reconstruct, the ends of a real-data run

listed() and draw() give cases, prepare() what a program holds before the
call, run() one pass, work() the bytes and operations it cannot do without and
exact() the result in 64 bits by plain numpy / torch.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "compressedsensingipm.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)


def listed():
    return [
        # the smallest documented problem: a 1D signal of 1024 samples, one
        # operator product; latency
        {"name": "mtm_1d_1024_f64", "kind": "mtm", "dims": "1024", "prec": "f64"},
        # a long 1D line of odd, prime length, as the serving stream's 1D
        # requests (1024 to 65536 samples) bring, in the server's precision
        {"name": "mtm_1d_49999_f32", "kind": "mtm", "dims": "49999", "prec": "f32"},
        # one Krylov product of the 255 x 255 configuration, FP64
        {"name": "kkt_2d_255_f64", "kind": "kkt", "dims": "255x255", "prec": "f64"},
        # both directions of the operator at ragged 2D sizes of the stream
        {"name": "forward_2d_509x384_f64", "kind": "forward", "dims": "509x384", "prec": "f64"},
        {"name": "adjoint_3d_158_f32", "kind": "adjoint", "dims": "158x185x127", "prec": "f32"},
        # one Krylov product of the 3D size sweep, FP64: the largest operator
        {"name": "kkt_3d_256_f64", "kind": "kkt", "dims": "256x256x256", "prec": "f64"},
        # the packing maps of a 3D model (FFTNLPModel users, plots, real data)
        {"name": "maps_3d_255", "kind": "maps", "dims": "255x255x255", "prec": "f64"},
        # one Newton system of an interior-point loop that runs outside
        # (MadNLP's role in the reference)
        {"name": "newton_2d_255_f64", "kind": "newton", "dims": "255x255", "prec": "f64"},
        # a whole solve in the reference's arithmetic
        {"name": "solve_2d_255_f64", "kind": "solve", "dims": "255x255", "prec": "f64"},
        # a whole solve of a 3D request in mixed precision
        {"name": "solve_3d_127_mixed", "kind": "solve", "dims": "127x127x127", "prec": "mixed"},
        # a set of uneven requests in the serving stream's mix, mixed precision
        {"name": "batch_48_mixed", "kind": "batch", "count": 48, "mix": 1, "prec": "mixed"},
        # a measured 3D volume: its mask's missing samples, its reconstruction
        {"name": "realdata_3d_200", "kind": "realdata", "dims": "200x160x144", "prec": "f64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _text(dims):
    return "x".join(str(d) for d in dims)


def draw(rng):
    """One more case: 1D 1024-65536, 2D sides 63-511, 3D sides 63-256 for
    single products; 2D sides 63-255 and 3D sides 63-127 for whole solves."""
    kind = rng.choice(["mtm", "forward", "adjoint", "kkt", "kkt", "maps", "newton", "solve",
                       "batch", "realdata"])
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(16, 48), "mix": rng.randint(2, 10**6),
                "prec": "mixed"}
    if kind == "newton":
        s = rng.randint(63, 400)
        return {"kind": kind, "dims": _text((s, s + rng.randint(-20, 20))), "prec": "f64"}
    if kind == "solve":
        if rng.random() < 0.5:
            s = rng.randint(63, 255)
            return {"kind": kind, "dims": _text((s, s)), "prec": "f64"}
        s = rng.randint(63, 127)
        return {"kind": kind, "dims": _text((s, s, s)), "prec": "mixed"}
    if kind in ("maps", "realdata"):
        return {"kind": kind, "dims": _text(_log_int(rng, 63, 240) for _ in range(3)),
                "prec": "f64"}
    prec = rng.choice(["f64", "f32"])
    d = rng.choice([1, 2, 2, 3, 3])
    if d == 1:
        dims = (_log_int(rng, 1024, 65536),)
    elif d == 2:
        dims = (_log_int(rng, 63, 511), _log_int(rng, 63, 511))
    else:
        dims = tuple(_log_int(rng, 63, 250) for _ in range(3))
    return {"kind": kind, "dims": _text(dims), "prec": prec}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _dtype(case):
    return torch.float64 if case["prec"] == "f64" else torch.float32


def _inputs(case, seed):
    """Host inputs of the single-product kinds."""
    dims = _dims(case)
    n = int(np.prod(dims))
    rng = np.random.default_rng(seed)
    k = round(0.15 * n)   # 15% of the samples are missing
    miss = np.sort(np.argpartition(rng.random(n, dtype=np.float32), k)[:k])
    kind = case["kind"]
    if kind == "mtm" or kind == "forward":
        return dims, miss, rng.standard_normal(n)
    if kind == "adjoint":
        z = rng.standard_normal(n)
        z[miss] = 0.0
        return dims, miss, z
    if kind == "maps":
        return dims, miss, rng.standard_normal(n)
    if kind == "kkt":
        # the slack diagonals of an interior-point iterate: most entries off
        # the support (both slacks alike), some on it (one slack active)
        s1, s2 = _sigmas(rng, n)
        return dims, miss, rng.standard_normal(2 * n), s1 + s2, s1 - s2
    if kind == "newton":
        s1, s2 = _sigmas(rng, n)
        return dims, miss, s1, s2, rng.standard_normal(6 * n)
    w = rng.random(n)   # realdata: nonzero weights at the observed samples
    w[miss] = 0.0
    return dims, miss, w, rng.standard_normal(n)


def _sigmas(rng, n):
    s1 = np.exp(rng.standard_normal(n))
    s2 = np.exp(rng.standard_normal(n))
    on = rng.random(n) < 0.05
    s1[on] *= 1e3
    s2[on] *= 1e-3
    return s1, s2


def _problem(case, seed):
    from csipm import workloads
    return workloads.stream_problem(_dims(case), seed)


def _batch_shapes(case):
    """Shapes of the stream's mix: 70% 1D, 25% 2D, 5% 3D, at least one of each."""
    rng = np.random.default_rng(1000 + case["mix"])
    n = case["count"]
    n3 = max(1, round(0.05 * n))
    n2 = max(1, round(0.25 * n))
    shapes = []
    for k in range(n):
        if k < n3:
            shapes.append((int(rng.integers(31, 64) * 2 + 1),) * 3)
        elif k < n3 + n2:
            shapes.append((int(rng.integers(63, 256) * 2 + 1),) * 2)
        else:
            shapes.append((int(round(math.exp(rng.uniform(math.log(1024), math.log(65536))))),))
    return shapes


def prepare(case, seed):
    from csipm import batch, fft_operator, model, workloads
    kind, dev = case["kind"], torch.device("cuda:0")
    if kind == "batch":
        ops, z0s, lams = [], [], []
        for k, shape in enumerate(_batch_shapes(case)):
            p = workloads.stream_problem(shape, 1000 * seed + k)
            ops.append(fft_operator.FFTOperator(p.N, len(p.dims), p.dims, p.missing, device=dev,
                                                mixed=True))
            z0s.append(torch.from_numpy(p.z0).to(dev))
            lams.append(p.lam)
        return {"call": batch.solve_batch, "kind": kind, "ops": ops, "z0s": z0s, "lams": lams}
    if kind == "solve":
        p = _problem(case, seed)
        par = fft_operator.FFTParameters(len(p.dims), p.dims, torch.from_numpy(p.z0).to(dev),
                                         p.lam, p.missing)
        nlp = model.FFTNLPModel(par, rdft=True, device=dev, mixed=case["prec"] == "mixed")
        return {"call": model.ipm_solve, "kind": kind, "nlp": nlp}
    dims, miss, *arrays = _inputs(case, seed)
    n, dt = int(np.prod(dims)), _dtype(case)
    arrays = [torch.from_numpy(a).to(dev, torch.float64 if kind == "realdata" else dt)
              for a in arrays]
    if kind in ("kkt", "newton"):
        par = fft_operator.FFTParameters(len(dims), dims, torch.zeros(n, dtype=dt, device=dev),
                                         0.05, miss)
        nlp = model.FFTNLPModel(par, rdft=True, dtype=dt, device=dev)
        if kind == "kkt":
            K = model.CondensedFFTKKTSystem(nlp)
            K.L1.copy_(arrays[1])
            K.L2.copy_(arrays[2])
            return {"kind": kind, "K": K, "x": arrays[0],
                    "y": torch.empty(2 * n, dtype=dt, device=dev)}
        K = model.FFTKKTSystem(nlp)
        K.initialize()
        s1, s2 = K.sigmas()
        s1.copy_(arrays[0])
        s2.copy_(arrays[1])
        return {"kind": kind, "K": K, "rhs": arrays[2], "w": torch.empty_like(arrays[2])}
    if kind == "realdata":
        op = fft_operator.FFTOperator(n, len(dims), dims, np.zeros(0, np.int64), device=dev)
        return {"kind": kind, "op": op, "mask": arrays[0], "beta": arrays[1]}
    op = fft_operator.FFTOperator(n, len(dims), dims, miss, dtype=dt, device=dev)
    return {"kind": kind, "op": op, "x": arrays[0]}


def run(state):
    from csipm import fft_operator as fo
    from csipm import realdata
    kind = state["kind"]
    if kind == "mtm":
        return fo.M_perpt_M_perp_vec(state["op"], state["x"])
    if kind == "forward":
        return fo.M_perp_beta(state["op"], state["x"])
    if kind == "adjoint":
        return fo.M_perpt_z(state["op"], state["x"])
    if kind == "kkt":
        return state["K"].mul(state["y"], state["x"])
    if kind == "maps":
        v = fo.beta_to_DFT(state["op"], state["x"])
        return v, fo.DFT_to_beta(state["op"], v)
    if kind == "newton":
        K, w = state["K"], state["w"]
        w.copy_(state["rhs"])
        K.build_kkt()
        K.solve_kkt(w)
        return w
    if kind == "realdata":
        return (realdata.index_missing_from_mask(state["mask"]),
                realdata.reconstruct(state["op"], state["beta"]))
    if kind == "solve":
        st = state["call"](state["nlp"], tol=1e-8)
        return st.solution, st.objective, st.status == "solved"
    res = state["call"](state["ops"], state["z0s"], state["lams"], mixed=True, tol=1e-8)
    return (torch.cat([r.beta for r in res]), np.asarray([r.objective for r in res]),
            all(r.status == "solved" for r in res))


# ---------------------------------------------------------------------------
# work: each input read once, each output written once; the operations of
# real FFTs (2.5 N log2 N) and the elementwise work
# ---------------------------------------------------------------------------

def _mtm_flops(n):
    return 5.0 * n * math.log2(n)


def work(case):
    kind = case["kind"]
    s = 8 if case["prec"] == "f64" else 4
    if kind == "batch":
        total = [int(np.prod(d)) for d in _batch_shapes(case)]
        # 7 interior-point steps of 9 FP32 products and one FP64 one each
        return {"bytes": sum(7.0 * (9 * 14 * 4 + 60 * 8) * n for n in total),
                "flops": sum(7.0 * 10 * _mtm_flops(n) for n in total)}
    n = int(np.prod(_dims(case)))
    if kind == "mtm":
        return {"bytes": 2.0 * n * s + n / 8, "flops": _mtm_flops(n)}
    if kind in ("forward", "adjoint"):
        return {"bytes": 2.0 * n * s + n / 8, "flops": 0.5 * _mtm_flops(n)}
    if kind == "kkt":
        return {"bytes": 6.0 * n * s + n / 8, "flops": _mtm_flops(n) + 8.0 * n}
    if kind == "maps":
        return {"bytes": 4.0 * n * 8, "flops": 2.0 * n}
    if kind == "realdata":
        return {"bytes": (1 + 0.15 + 2) * 8.0 * n, "flops": 0.5 * _mtm_flops(n)}
    if kind == "newton":
        # 25 Krylov products with their vector updates
        return {"bytes": 25 * 20.0 * n * s, "flops": 25 * (_mtm_flops(n) + 30.0 * n)}
    steps, its = (8, 14) if case["prec"] == "f64" else (8, 11)
    return {"bytes": steps * its * (20 if s == 8 else 14) * float(n) * s,
            "flops": steps * its * (_mtm_flops(n) + 30.0 * n)}


# ---------------------------------------------------------------------------
# exact: the single products in 64 bits
# ---------------------------------------------------------------------------

def _elements(dims):
    """For every entry of beta: its element of the full spectrum (linear,
    dimension 1 fastest), whether it is the imaginary part, whether it is a
    self-conjugate vertex."""
    d = len(dims)
    S = [[0] if n % 2 else [0, n // 2] for n in dims]
    R = [list(range(1, (n - 1) // 2 + 1)) for n in dims]
    H = [list(range(n // 2 + 1, n // 2 + 1 + (n - 1) // 2)) for n in dims]
    if d == 1:
        vert, pairs = [[[a]] for a in S[0]], [[R[0]]]
    elif d == 2:
        vert = [[[a], [b]] for a in S[0] for b in S[1]]
        pairs = [[[a], R[1]] for a in S[0]] + [[R[0], [b]] for b in S[1]]
        pairs += [[R[0], R[1]], [R[0], H[1]]]
    else:
        vert = [[[a], [b], [c]] for a in S[0] for b in S[1] for c in S[2]]
        pairs = [[[a], [b], R[2]] for a in S[0] for b in S[1]]
        pairs += [[[a], R[1], [c]] for a in S[0] for c in S[2]]
        pairs += [[R[0], [b], [c]] for b in S[1] for c in S[2]]
        pairs += [[[a], y, R[2]] for a in S[0] for y in (R[1], H[1])]
        pairs += [[x, [b], R[2]] for b in S[1] for x in (R[0], H[0])]
        pairs += [[x, R[1], [c]] for c in S[2] for x in (R[0], H[0])]
        pairs += [[x, y, R[2]] for y in (R[1], H[1]) for x in (R[0], H[0])]
    stride = [int(np.prod(dims[:k])) for k in range(d)]

    def linear(axes):
        lin = np.zeros(1, np.int64)
        for a, st in reversed(list(zip(axes, stride))):   # dimension 1 fastest
            lin = (lin[:, None] + np.asarray(a, np.int64)[None, :] * st).reshape(-1)
        return lin

    lin = [linear(a) for a in vert]
    comp = [np.zeros(len(v), bool) for v in lin]
    nvert = len(lin)
    for a in pairs:
        g = linear(a)
        lin += [g, g]
        comp += [np.zeros(len(g), bool), np.ones(len(g), bool)]
    return np.concatenate(lin), np.concatenate(comp), nvert


class _Exact:
    def __init__(self, dims, miss):
        self.dims, self.miss = dims, torch.from_numpy(np.asarray(miss, np.int64))
        self.n = int(np.prod(dims))
        lin, comp, nv = _elements(dims)
        self.lin, self.comp, self.nv = torch.from_numpy(lin), torch.from_numpy(comp), nv

    def spectrum(self, beta):
        """The full Hermitian spectrum of beta, its reversed (C-order) shape."""
        part = beta / math.sqrt(2.0)
        part[:self.nv] = beta[:self.nv]
        f = torch.zeros(self.n, dtype=torch.complex128)
        v = torch.view_as_real(f)
        v[self.lin[~self.comp], 0] = part[~self.comp]
        v[self.lin[self.comp], 1] = part[self.comp]
        f = f.reshape(self.dims[::-1])
        # the conjugate partners of the stored elements, -k mod n per axis
        ax = tuple(range(len(self.dims)))
        g = torch.roll(torch.flip(f, ax), [1] * len(ax), ax).conj()
        have = torch.zeros(self.n, dtype=torch.bool)
        have[self.lin] = True
        return torch.where(have.reshape(f.shape), f, g)

    def beta(self, spec):
        v = torch.view_as_real(spec.reshape(-1).contiguous())
        out = torch.where(self.comp, v[self.lin, 1], v[self.lin, 0]) * math.sqrt(2.0)
        out[:self.nv] /= math.sqrt(2.0)
        return out

    def m(self, beta, mask=True):
        x = torch.fft.ifftn(self.spectrum(beta)).real.reshape(-1) * math.sqrt(self.n)
        if mask:
            x[self.miss] = 0.0
        return x

    def mt(self, z):
        return self.beta(torch.fft.fftn(z.reshape(self.dims[::-1]).to(torch.complex128))
                         / math.sqrt(self.n))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "solve"):
        return None   # iterates at a finite tolerance
    dims, miss, *arrays = _inputs(case, seed)
    # the inputs as the handle's precision holds them
    a = [torch.from_numpy(v).to(torch.float64 if kind == "realdata" else _dtype(case)).double()
         for v in arrays]
    E = _Exact(dims, miss)
    n = E.n
    if kind == "mtm":
        return E.mt(E.m(a[0]))
    if kind == "forward":
        return E.m(a[0])
    if kind == "adjoint":
        return E.mt(a[0])
    if kind == "kkt":
        x, l1, l2 = a
        return torch.cat([E.mt(E.m(x[:n])) + l1 * x[:n] + l2 * x[n:], l2 * x[:n] + l1 * x[n:]])
    if kind == "maps":
        half = E.spectrum(a[0])[..., :dims[0] // 2 + 1]
        return half.reshape(-1), a[0]
    if kind == "realdata":
        return torch.from_numpy(np.asarray(miss, np.int64)), E.m(a[1], mask=False)
    # newton: the condensed system by conjugate gradients, then the unpack
    s1, s2, w = a
    if n > 200000:
        return None
    w1, w2, w3, w4, w5, w6 = w.reshape(6, n)
    l1, l2 = s1 + s2, s1 - s2
    b = torch.cat([w1 - w3 + w4 - s1 * w5 + s2 * w6, w2 - w3 - w4 - s1 * w5 - s2 * w6])
    det = l1 + 4 * s1 * s2

    def K(x):
        return torch.cat([E.mt(E.m(x[:n].clone())) + l1 * x[:n] + l2 * x[n:],
                          l2 * x[:n] + l1 * x[n:]])

    def P(x):
        return torch.cat([(l1 * x[:n] - l2 * x[n:]) / det,
                          (-l2 * x[:n] + (1 + l1) * x[n:]) / det])

    x, r = torch.zeros_like(b), b.clone()
    z = P(r)
    p, g = z.clone(), torch.dot(r, z)
    for _ in range(400):
        q = K(p)
        al = g / torch.dot(p, q)
        x += al * p
        r -= al * q
        z = P(r)
        g, old = torch.dot(r, z), g
        if float(g) <= 1e-28:
            break
        p = z + (g / old) * p
    d1, d2 = x[:n], x[n:]
    v5 = -(w3 + s1 * (d1 + d2 + w5))
    v6 = -(w4 + s2 * (-d1 + d2 + w6))
    return torch.cat([d1, d2, (w3 + v5) / s1, (w4 + v6) / s2, v5, v6])
