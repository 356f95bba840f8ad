"""GPU parity of the fused FFT operator through the C ABI.

FP64: within 1e-12 relative (max-norm) of the FP64 CPU oracle; the
reference's identities (M^T M = I without mask, norm preservation,
test/unit_tests_ipm.jl:7-30) hold to the same tolerance.  FP32: 2e-6.
"""
import os

import numpy as np
import pytest
import torch

from oracle import kkt, maps
from oracle import operator as op

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")
TOL64 = 1e-12
TOL32 = 2e-6


def _rel(a, b):
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(np.asarray(b)).max(), 1e-300))


def _make(dims, missing=(), dtype=torch.float64):
    from csipm.fft_operator import FFTOperator
    return FFTOperator(int(np.prod(dims)), len(dims), dims, np.asarray(missing, np.int64),
                       rdft=True, dtype=dtype)


UNIT = [(100,), (200,), (500,), (16, 16), (12, 18), (16, 24), (32, 32), (8, 8, 8), (2, 4, 6),
        (6, 10, 12), (14, 8, 4), (8, 6, 4), (16, 16, 16)]


@pytest.mark.parametrize("dims", UNIT + [(255,), (1024,), (255, 255), (15, 17, 9)])
def test_identities_no_mask(cuda, dims):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("identities", dims, flush=True)
    rng = np.random.default_rng(1)
    z = rng.uniform(size=int(np.prod(dims)))
    o = _make(dims)
    zt = torch.from_numpy(z).to(cuda)
    assert _rel(M_perpt_M_perp_vec(o, zt).cpu().numpy(), z) <= TOL64
    r1 = M_perpt_z(o, zt).cpu().numpy()
    r2 = M_perp_beta(o, zt).cpu().numpy()
    assert abs(np.linalg.norm(r1) - np.linalg.norm(z)) <= TOL64 * np.linalg.norm(z)
    assert abs(np.linalg.norm(r2) - np.linalg.norm(z)) <= TOL64 * np.linalg.norm(z)
    assert _rel(r1, op.m_perpt_z(z, dims)) <= TOL64
    assert _rel(r2, op.m_perp_beta(z, dims)) <= TOL64


@pytest.mark.parametrize("fname", sorted(f for f in os.listdir(GOLD) if f.startswith("op_")))
def test_operator_golden(cuda, fname):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    d = np.load(os.path.join(GOLD, fname))
    dims = tuple(int(v) for v in d["dims"])
    print("operator", dims, flush=True)
    o = _make(dims, d["missing"])
    x = torch.from_numpy(d["x"]).to(cuda)
    z = torch.from_numpy(d["z"]).to(cuda)
    assert _rel(M_perpt_M_perp_vec(o, x).cpu().numpy(), d["mtm"]) <= TOL64
    assert _rel(M_perp_beta(o, x).cpu().numpy(), d["m_perp_beta"]) <= TOL64
    assert _rel(M_perpt_z(o, z).cpu().numpy(), d["m_perpt_z"]) <= TOL64


# lengths whose prime factors are at most 31 factor directly (radices 19..31)
LARGE_RADIX = [(19, 23), (23, 19, 29), (31, 62), (57, 87)]
# a prime length whose L - 1 factors runs Rader's form (including dimension 1
# of a 2D/3D problem and the long-line kernel of 1D N = 4001)
RADER = [(127,), (4001,), (191, 127), (127, 60), (12, 10, 37), (37, 41, 47), (53, 59, 61)]
# other lengths with a prime factor above 31 run Bluestein's chirp-z form with
# a factorable convolution length M >= 2L - 1 (4007: M = 8064 on the 1024-thread kernel)
BLUESTEIN = [(83,), (4007,), (111, 20), (20, 111), (9, 8, 83), (107, 13, 10)]
# 1D lines above 4096 run as four-step transforms: direct when N factors into
# the supported radices, else with an outer Bluestein convolution
FOURSTEP = [(8192,), (50000,), (65536,), (4097,), (12289,), (65521,)]


@pytest.mark.parametrize("dims", [(1024,), (255, 255), (64, 48, 30), (51, 45, 35)] + LARGE_RADIX +
                         RADER + BLUESTEIN + FOURSTEP)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_operator_masked_vs_oracle(cuda, dims, dtype):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("operator", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


# a tuned Bluestein convolution length (csipm_tune_bluestein) changes the
# plan, not the operator
@pytest.mark.parametrize("dims,L,M", [((83,), 83, 176), ((111, 20), 111, 240),
                                      ((9, 8, 83), 83, 171), ((37, 41, 47), 37, 80)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_operator_tuned_bluestein(cuda, dims, L, M, dtype):
    from csipm import _lib, tune
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("tuned Bluestein", dims, L, M, dtype, flush=True)
    lib = _lib.lib()
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + M)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    assert lib.csipm_tune_bluestein(L, M) == 0
    try:
        o = _make(dims, miss, dtype)
        axis = list(dims).index(L)
        if (L, dims) == (37, (37, 41, 47)):
            assert tune.fft_shape(o, axis)[2] == 2       # a Rader length keeps Rader's form
        else:
            assert tune.fft_shape(o, axis) == (M, M, 1)
        xt = torch.from_numpy(x).to(cuda, dtype)
        assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
        assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
        assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol
    finally:
        lib.csipm_tune_bluestein(L, 0)
        tune.load(lib)


@pytest.mark.parametrize("dims", [(1024,), (255, 255), (33, 30, 26)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_kkt_and_precond(cuda, dims, dtype):
    from csipm import _lib
    from csipm.fft_operator import _ptr
    print("kkt", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(3)
    miss = np.sort(rng.choice(n, size=n // 10, replace=False))
    o = _make(dims, miss, dtype)
    s1 = rng.uniform(0.05, 5.0, n)
    s2 = rng.uniform(0.05, 5.0, n)
    T = lambda a: torch.from_numpy(np.asarray(a)).to(cuda, dtype).contiguous()   # noqa: E731
    L1, L2, P11, P12, P22 = (torch.empty(n, device=cuda, dtype=dtype) for _ in range(5))
    s1t, s2t = T(s1), T(s2)       # keep the inputs alive while the kernels run
    _lib.call("csipm_precond_build", o.handle, _ptr(s1t), _ptr(s2t), _ptr(L1), _ptr(L2),
              _ptr(P11), _ptr(P12), _ptr(P22))
    ref = kkt.precond_build(s1, s2)
    tol = TOL64 if dtype == torch.float64 else TOL32
    for got, want in zip((L1, L2, P11, P12, P22), ref):
        assert _rel(got.double().cpu().numpy(), want) <= 10 * tol
    x = rng.standard_normal(2 * n)
    y0 = rng.standard_normal(2 * n)
    y = T(y0)
    xt = T(x)
    _lib.call("csipm_kkt_apply", o.handle, _ptr(xt), _ptr(y), _ptr(L1), _ptr(L2), 0.75, -0.5)
    want = kkt.kkt_mul(y0, x, ref[0], ref[1], lambda v: op.mtm(v, dims, miss), 0.75, -0.5)
    assert _rel(y.double().cpu().numpy(), want) <= 10 * tol
    y = T(y0)
    _lib.call("csipm_precond_apply", o.handle, _ptr(xt), _ptr(y), _ptr(P11), _ptr(P12),
              _ptr(P22), 2.0, 0.25)
    want = kkt.precond_mul(y0, x, ref[2], ref[3], ref[4], 2.0, 0.25)
    assert _rel(y.double().cpu().numpy(), want) <= 10 * tol


@pytest.mark.parametrize("dims", [(1024,), (255, 255), (33, 30, 26), (127, 60), (20000,),
                                  (12289,)])
def test_cg_solve(cuda, dims):
    import ctypes
    from csipm import _lib
    from csipm.fft_operator import _ptr
    print("cg", dims, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(4)
    miss = np.sort(rng.choice(n, size=n // 10, replace=False))
    o = _make(dims, miss)
    s1 = rng.uniform(0.05, 5.0, n)
    s2 = rng.uniform(0.05, 5.0, n)
    L1, L2, P11, P12, P22 = kkt.precond_build(s1, s2)
    b = rng.standard_normal(2 * n)
    mt = lambda v: op.mtm(v, dims, miss)      # noqa: E731
    xr, itr, resr, str_ = kkt.pcg(lambda v: kkt.kkt_mul(np.zeros(2 * n), v, L1, L2, mt),
                                  b, lambda r: kkt.precond_mul(np.zeros(2 * n), r, P11, P12, P22),
                                  atol=1e-12, rtol=0.0)
    T = lambda a: torch.from_numpy(np.asarray(a)).to(cuda).contiguous()   # noqa: E731
    x = torch.zeros(2 * n, device=cuda, dtype=torch.float64)
    it = ctypes.c_int64()
    res = ctypes.c_double()
    st = ctypes.c_int()
    keep = [T(a) for a in (b, L1, L2, P11, P12, P22)]   # alive during the solve
    bt, L1t, L2t, P11t, P12t, P22t = keep
    _lib.call("csipm_cg_solve", o.handle, _ptr(bt), _ptr(x), _ptr(L1t), _ptr(L2t),
              _ptr(P11t), _ptr(P12t), _ptr(P22t), 1e-12, 0.0, 0, ctypes.byref(it),
              ctypes.byref(res), ctypes.byref(st))
    assert st.value == 0 and str_ == "solved"
    assert abs(it.value - itr) <= 1
    assert res.value <= 1e-12
    assert _rel(x.cpu().numpy(), xr) <= 1e-10


@pytest.mark.parametrize("dims", [(1000,), (16, 12), (15, 17), (9, 10, 7), (20000,)])
def test_complex_path_operator(cuda, dims):
    """An rdft=False handle (the reference's default) against the oracle's
    complex path; its maps default to the full spectrum."""
    from csipm.fft_operator import (FFTOperator, M_perp_beta, M_perpt_M_perp_vec, M_perpt_z,
                                    beta_to_DFT, DFT_to_beta)
    print("complex path", dims, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 2)
    miss = np.sort(rng.choice(n, size=n // 8, replace=False))
    o = FFTOperator(n, len(dims), dims, miss, rdft=False)
    x = rng.standard_normal(n)
    xt = torch.from_numpy(x).to(cuda)
    assert _rel(M_perpt_M_perp_vec(o, xt).cpu().numpy(), op.mtm(x, dims, miss, rdft=False)) <= TOL64
    assert _rel(M_perp_beta(o, xt).cpu().numpy(), op.m_perp_beta(x, dims, miss, rdft=False)) <= TOL64
    assert _rel(M_perpt_z(o, xt).cpu().numpy(), op.m_perpt_z(x, dims, rdft=False)) <= TOL64
    v = beta_to_DFT(o, xt).cpu().numpy()
    assert v.size == n
    assert np.array_equal(v, maps.beta_to_dft(x, dims, rdft=False))
    assert np.array_equal(DFT_to_beta(o, torch.from_numpy(v).to(cuda)).cpu().numpy(),
                          maps.dft_to_beta(v, dims))


# the workgroup size follows from the tile: 256 threads up to 2048 elements,
# 512 to 4096, 1024 to 8192 and, 16 elements each, beyond (dimension 1);
# sizes on both sides of each line, in every pass kind (4091: Bluestein of
# about 8190; 65536 = 256 x 256 and 4608 = 64 x 72 four-step)
@pytest.mark.parametrize("dims", [(2048,), (2058,), (4096,), (4091,), (9000, 2), (4104, 3),
                                  (2, 2048), (6, 2058), (6, 4096), (4608,), (3, 5, 2058)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_workgroup_sizes(cuda, dims, dtype):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("workgroups", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 3)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


# axes of lengths the radices do not cover, as dense products on the matrix
# cores: one to four blocks of output rows a wave (up to 126, 127..254 and on),
# odd and even, primes and not, both sides of 256 (above it only where the
# other axes give 2048 lines), few lines and many, the longest, and the short
# ones with a factor 29 or 31
@pytest.mark.parametrize("dims", [(37, 3), (2, 41), (62, 74), (5, 126, 2), (127, 33), (128, 127),
                                  (3, 129, 2), (254, 74), (253, 2, 3), (2, 3, 251), (43, 47, 53),
                                  (257, 33), (4, 262, 1100), (383, 2300), (2100, 386),
                                  (509, 4000), (6, 800, 511), (58, 93), (124, 3, 87), (2, 116)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_dense_lengths(cuda, dims, dtype):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("dense", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 7)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


def test_infinite_entry(cuda):
    """An infinite spectrum entry gives infinite samples, not NaN, where the
    transform only adds it: beta of frequency 1 of four samples, cos(pi n / 2)."""
    from csipm.fft_operator import M_perp_beta
    print("infinite entry", flush=True)
    for dtype in (torch.float64, torch.float32):
        o = _make((4,), np.zeros(0, np.int64), dtype)
        beta = torch.tensor([0.0, 0.0, np.inf, 0.0], dtype=dtype, device=cuda)
        x = M_perp_beta(o, beta).cpu().numpy()
        assert x[0] == np.inf and x[2] == -np.inf


# stages of radix 29 and 31 (matrix products): alone, twice (twiddles between),
# with every kind of stage after them; column tiles full and not, one line and
# 16, 128 to 1024 threads, four-step (7192), Rader's inner transforms (59: 58;
# 311 on few lines: 310)
@pytest.mark.parametrize("dims", [(29,), (31,), (58,), (59,), (841,), (899,), (961,), (3596,), (7192,),
                                  (29791,), (155, 3), (3, 217), (145, 155, 7), (4, 6, 248), (3596, 2),
                                  (2, 3596), (8990, 2), (16, 217, 1030), (311, 5), (5, 311)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_matrix_stages(cuda, dims, dtype):
    from csipm import tune
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("matrix stages", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 11)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    for axis, length in enumerate(dims):
        if length % 29 == 0 or length % 31 == 0:
            assert tune.fft_shape(o, axis)[2] in (0, 3)   # a plan, four-step or not
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


# The form each axis is planned in (0 direct, 1 Bluestein, 2 Rader, 4 dense), on
# line passes as well as along dimension 1.  Axes up to 256 that do not factor
# are dense, those to 511 where 2048 lines share the launch (so the 2D / 3D sizes
# of RADER, BLUESTEIN and LARGE_RADIX above are); beyond, a prime whose
# predecessor factors is Rader's and the rest Bluestein's (433 - 1 and 1021 - 1
# factor, 509 - 1 and 262 do not).
FORMS = [((24, 257), (0, 2)), ((257, 24), (2, 0)), ((6, 5, 433), (0, 0, 2)), ((6, 433, 5), (0, 2, 0)),
         ((433, 6, 5), (2, 0, 0)), ((3, 1021), (0, 2)), ((1021, 3), (2, 0)),
         ((24, 262), (0, 1)), ((262, 24), (1, 0)), ((6, 5, 509), (0, 0, 1)), ((6, 509, 5), (0, 1, 0)),
         ((509, 6, 5), (1, 0, 0)), ((3, 514), (0, 1)), ((514, 3), (1, 0)), ((433, 262), (2, 1)),
         ((155, 217), (0, 0)), ((145, 186, 4), (0, 0, 0)),
         ((191, 127), (4, 4)), ((37, 41, 47), (4, 4, 4)), ((111, 20), (4, 0)), ((9, 8, 83), (0, 0, 4)),
         ((31, 62), (0, 4)), ((57, 87), (0, 4)), ((383, 2300), (4, 0)), ((2300, 383), (0, 4))]


@pytest.mark.parametrize("dims,forms", FORMS)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_forms(cuda, dims, forms, dtype):
    from csipm import tune
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("forms", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 13)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    assert tuple(tune.fft_shape(o, axis)[2] for axis in range(len(dims))) == forms
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


# dense tiles of 16 and 32 lines (32 or 64 real columns), which a launch takes
# when it has 1024 of them: 32 lines of 37 (18 of 32 valid), 16 of 185 (FP32; 8 in
# FP64) and of 126, along dimension 1 32 pairs of 37 and 16 of 131 (FP32)
@pytest.mark.parametrize("dims", [(34, 37, 1030), (18, 185, 1030), (17, 1030, 126), (37, 260, 256),
                                  (131, 182, 182)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_wide_dense_tiles(cuda, dims, dtype):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("wide dense tiles", dims, dtype, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 17)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    tol = TOL64 if dtype == torch.float64 else TOL32
    o = _make(dims, miss, dtype)
    xt = torch.from_numpy(x).to(cuda, dtype)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= tol
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= tol
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= tol


# FP32 tiles of 16 elements a thread: along dimension 1 (270, 8 pairs) and on the
# middle line passes (300, 8 lines; 16 of them, and 51, the last tile in part)
@pytest.mark.parametrize("dims", [(270, 128, 130), (30, 300, 512), (100, 300, 150)])
def test_sixteen_element_tiles(cuda, dims):
    from csipm.fft_operator import M_perp_beta, M_perpt_M_perp_vec, M_perpt_z
    print("sixteen elements", dims, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n + 19)
    miss = np.sort(rng.choice(n, size=n // 9, replace=False))
    x = rng.standard_normal(n)
    o = _make(dims, miss, torch.float32)
    xt = torch.from_numpy(x).to(cuda, torch.float32)
    assert _rel(M_perpt_M_perp_vec(o, xt).double().cpu().numpy(), op.mtm(x, dims, miss)) <= TOL32
    assert _rel(M_perp_beta(o, xt).double().cpu().numpy(), op.m_perp_beta(x, dims, miss)) <= TOL32
    assert _rel(M_perpt_z(o, xt).double().cpu().numpy(), op.m_perpt_z(x, dims)) <= TOL32
