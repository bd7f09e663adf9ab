"""The device layer called through its own C ABI (include/lmie_gpu.h), for the
jobs that the interface above it does not make."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from test_tangent_arith import build

pytestmark = pytest.mark.gpu

DP, IP = C.POINTER(C.c_double), C.POINTER(C.c_int)
FP64, MIXED = 0, 1


def say(*a):
    print(*a, flush=True)


class Job(C.Structure):
    _fields_ = [("n_size", C.c_int), ("x", DP), ("f", DP), ("n1", IP), ("n2", IP), ("sx", DP), ("cx", DP),
                ("mr", C.c_double), ("mi", C.c_double), ("n1_max", C.c_int), ("n_qang", C.c_int), ("n_coef", C.c_int),
                ("calc_gc", C.c_int), ("calc_lc", C.c_int), ("n_tan", C.c_int), ("dx", DP), ("dm", DP), ("df_tan", DP),
                ("n_wgt", C.c_int), ("df_wgt", DP), ("save_control", C.c_int), ("saved1", DP), ("saved2", DP),
                ("precision", C.c_int), ("device", C.c_int), ("keep", C.c_int)]


class Result(C.Structure):
    _fields_ = [("sums", C.c_double * 4), ("sums_ch", DP), ("gc_raw", DP), ("lc_raw", DP), ("save1", DP), ("save2", DP),
                ("state", C.c_void_p), ("precision", C.c_int)]


class AdjIn(C.Structure):
    _fields_ = [("sums_bar", DP), ("gc_bar", DP), ("lc_bar", DP)]


class AdjOut(C.Structure):
    _fields_ = [("f_bar", DP), ("m_bar", C.c_double * 2), ("x_bar", DP)]


def order_n1(x):
    return int(x + 4.05 * x ** (1.0 / 3.0) + 8)


def order_n2(n1, x, m):
    a = max(float(n1), abs(m) * x)
    return int(a + 6.40 * a ** (1.0 / 3.0) + 8)


@pytest.fixture(scope="module")
def dev(product):
    product.lmie_gpu_forward.argtypes = [C.POINTER(Job), C.POINTER(Result)]
    product.lmie_gpu_adjoint.argtypes = [C.c_void_p, C.POINTER(AdjIn), C.POINTER(AdjOut)]
    product.lmie_gpu_release.argtypes = [C.c_void_p]
    product.lmie_gpu_release.restype = None
    product.lmie_gpu_batch_open.restype = C.c_void_p
    product.lmie_gpu_batch_enter.argtypes = [C.c_void_p, C.c_int]
    product.lmie_gpu_batch_fused.argtypes = [C.c_void_p, C.c_int]
    product.lmie_gpu_batch_close.argtypes = [C.c_void_p]
    product.lmie_gpu_batch_close.restype = None
    product.lmie_gpu_last_error.restype = C.c_char_p
    return product


def arr(a, t=np.float64):
    return np.ascontiguousarray(a, dtype=t)


def ptr(a):
    return None if a is None else a.ctypes.data_as(IP if a.dtype == np.intc else DP)


def test_batched_reverse_pass_of_a_64_size_state(dev):
    """A state kept by a forward that a batch ran alone (weight-only channels are
    not fused) under LMIE_UGEMM_WAVES=2, whose reverse task list is of tiles of
    64 sizes: its reverse pass in the batch gives the single call's bits, and
    the default shape's cotangents to the mixed path's 1e-5."""
    say("case: reverse pass in a batch of a state with 64-size tiles (300 sizes to x 40)")
    N = 300
    x = arr(np.linspace(0.3, 40.0, N))
    f = arr(np.exp(-0.1 * x) / N)
    n1 = arr([order_n1(v) for v in x], np.intc)
    n2 = arr([order_n2(n, v, 1.5 - 0.01j) for n, v in zip(n1, x)], np.intc)
    nm = int(n1.max())
    wgt = arr(f * np.cos(x))
    rng = np.random.Generator(np.random.PCG64(5))
    gc_bar, sums_bar = arr(rng.standard_normal((6, 2 * nm))), arr([0.3, -0.2, 0.1, 0.4])

    def run(shape, batch):
        ch, gc = np.zeros((1, 4)), np.zeros((2, 6, 2 * nm))
        job = Job(n_size=N, x=ptr(x), f=ptr(f), n1=ptr(n1), n2=ptr(n2), mr=1.5, mi=0.01, n1_max=nm, n_qang=2 * nm,
                  n_coef=2 * nm, calc_gc=1, n_wgt=1, df_wgt=ptr(wgt), precision=MIXED, keep=1)
        res = Result(sums_ch=ptr(ch), gc_raw=ptr(gc))
        fb, xb = np.full(N, np.nan), np.full(N, np.nan)
        ain, aout = AdjIn(ptr(sums_bar), ptr(gc_bar), None), AdjOut(f_bar=ptr(fb), x_bar=ptr(xb))
        old = os.environ.get("LMIE_UGEMM_WAVES")
        b = dev.lmie_gpu_batch_open(1) if batch else None
        fused = None
        try:
            os.environ["LMIE_UGEMM_WAVES"] = shape
            if batch:
                assert dev.lmie_gpu_batch_enter(b, 0) == 0
            assert dev.lmie_gpu_forward(C.byref(job), C.byref(res)) == 0, dev.lmie_gpu_last_error()
            assert res.precision == MIXED
            assert dev.lmie_gpu_adjoint(res.state, C.byref(ain), C.byref(aout)) == 0, dev.lmie_gpu_last_error()
        finally:
            if old is None:
                del os.environ["LMIE_UGEMM_WAVES"]
            else:
                os.environ["LMIE_UGEMM_WAVES"] = old
            if batch:
                dev.lmie_gpu_batch_leave()
                fused = [dev.lmie_gpu_batch_fused(b, p) for p in (0, 1)]
                dev.lmie_gpu_batch_close(b)
            if res.state:
                dev.lmie_gpu_release(res.state)
        return fb, xb, np.array(aout.m_bar[:]), fused

    single, batched, ref = run("2", False), run("2", True), run("8", True)
    assert batched[3] == [0, 0] and ref[3] == [0, 1]
    for k in range(3):
        assert np.array_equal(batched[k], single[k]), k
        err = np.linalg.norm(batched[k] - ref[k]) / np.linalg.norm(ref[k])
        say("  against the 128-size shape", k, err)
        assert err <= 1e-5, (k, err)


@pytest.mark.parametrize("mr,mi", [(1.5, 0.01), (1.33, 0.3)])
def test_series_and_tangents_at_large_x(dev, tmp_path, mr, mi):
    """The series sums of 83 sizes of two waves and their derivatives along x, mr and
    mi against the recurrences in 113 bits (tests/c/tangent_quad.c): x = k pi + d for
    k = 285 .. 300 and d = 0.8, -0.3, 1e-2, -1e-4, k = 1, 30, 588 with d down to
    1e-6, small x, and cuts inside x (n1 < x, only reachable here).

    Each size by a bound: the chains' relative errors, 8 sqrt(n2) ulp (four
    standard deviations of their roundings), divided by |sin x| for psi and sin^2 x
    for psi' (psi starts at sin x), times 16 for three such chains in a handful of
    products, of the sum of the terms' magnitudes.

    And the 16 sizes of each d by the reference's own recurrences in double (ratios of
    psi, differentiated): the same accuracy by other roundings, so the root mean
    squares of the errors differ by what 64 samples scatter; four times is
    allowed (1/x rounded once in the chains was 20 times)."""
    say("case: series and tangents of 83 sizes, m = %g - %gi" % (mr, mi))
    m = mr - 1j * mi
    ds = (0.8, -0.3, 1e-2, -1e-4)
    sizes = [(k * np.pi + d, None) for d in ds for k in range(285, 301)]
    sizes += [(k * np.pi + d, None) for k in (1, 30, 588) for d in (0.8, -1e-2, 1e-4, 1e-6)]
    sizes += [(0.02, None), (0.05, None), (0.3, None), (0.7, None), (2.0, None), (99.2, 60), (33.3, 20)]
    x = arr([v for v, _ in sizes])
    N = len(x)
    n1 = arr([n or order_n1(v) for v, n in sizes], np.intc)
    n2 = arr([order_n2(n, v, m) for n, v in zip(n1, x)], np.intc)
    text = "".join("%.17g %.17g %.17g %d %d\n" % (x[i], mr, mi, n1[i], n2[i]) for i in range(N))
    r = subprocess.run([build(tmp_path)], input=text, capture_output=True, text=True, timeout=120)
    ref = np.array([[float(v) for v in line.split()] for line in r.stdout.splitlines()]).reshape(N, 3, 4, 4)
    eps = 128 * np.sqrt(n2) * 2.3e-16
    isin = np.where(x > 1.0, 1.0 / np.abs(np.sin(x)), 1.0)
    f = arr(1.0 / x ** 2)
    # the value of each size, its derivative along x, then mr and mi of all
    nt = 2 * N + 2
    dx, dft, dm = np.zeros((nt, N)), np.zeros((nt, N)), np.zeros((nt, 2))
    for i in range(N):
        dft[i, i] = 1.0
        dx[N + i, i] = 1.0 / f[i]
    dm[2 * N, 0], dm[2 * N + 1, 1] = 1.0, -1.0
    ch = np.full((nt, 4), np.nan)
    job = Job(n_size=N, x=ptr(x), f=ptr(f), n1=ptr(n1), n2=ptr(n2), mr=mr, mi=mi, n1_max=int(n1.max()), n_tan=nt,
              dx=ptr(dx), dm=ptr(dm), df_tan=ptr(dft), precision=FP64)
    res = Result(sums_ch=ptr(ch))
    assert dev.lmie_gpu_forward(C.byref(job), C.byref(res)) == 0, dev.lmie_gpu_last_error()
    bad = []
    w = eps * isin
    for name, got, val, mag in (("value", ch[:N], ref[:, 0, 0], ref[:, 1, 0] * w[:, None]),
                                ("x", ch[N:2 * N], ref[:, 0, 1], ref[:, 1, 1] * (w * isin)[:, None]),
                                ("mr", ch[2 * N], f @ ref[:, 0, 2], (f * w) @ ref[:, 1, 2]),
                                ("mi", ch[2 * N + 1], f @ ref[:, 0, 3], (f * w) @ ref[:, 1, 3]),
                                ("sum", np.array(res.sums[:]), f @ ref[:, 0, 0], (f * w) @ ref[:, 1, 0])):
        e = np.abs(got - val) / mag
        if e.ndim == 2:
            # b_n and a_2 at small x are differences that cancel in the formula itself
            # (psi_n (m D_n + n/x) - psi_{n-1}, as the reference forms it): asym, products of
            # them with a_1, is left out there
            e[x < 0.1, 3] = 0.0
        say("  %-5s largest error %.2e of its bound" % (name, e.max()))
        if not np.all(e <= 1.0):
            bad.append((name, np.argwhere(~(e <= 1.0)).tolist(), e.max()))
    for q, d in enumerate(ds):
        g = slice(16 * q, 16 * q + 16)
        for name, got, k in (("value", ch[:N], 0), ("x", ch[N:2 * N], 1)):
            rms = [np.sqrt(np.mean(((v[g] - ref[g, 0, k]) / ref[g, 1, k]) ** 2)) for v in (got, ref[:, 2, k])]
            say("  d %g %-5s root mean square error %.2e, ratio recurrences %.2e" % (d, name, *rms))
            if not rms[0] <= 4.0 * rms[1]:
                bad.append((name, d, rms))
    assert not bad, bad
