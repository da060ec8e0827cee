"""Products whose result goes through an elementwise operator before it leaves (gemm_tail of csrc/gemm_plan.h): the SwiGLU of
two products (gated), the rotation of q and k, and the SwiGLU's adjoint, at the sizes where the tiles, stages and pieces of
every kernel end.  Against float64 of the stored values: a product is off by half a unit of its type and the roundings of its
sum, n * 2^-24 * sum |a b| to first order, twice that allowed; the operator passes that on times its derivative, and rounds
its result once more (fp32: the hardware's exponential and reciprocal, a unit or two each, 2^-19 allowed)."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import dev, host

pytestmark = pytest.mark.gpu
GATED, ROTATED, ADJOINT = 2, 3, 4


class _Tail(ctypes.Structure):
    _fields_ = [("mode", ctypes.c_int), ("B", ctypes.c_void_p * 3), ("C", ctypes.c_void_p * 3), ("table", ctypes.c_void_p), ("seq", ctypes.c_int),
                ("head_dim", ctypes.c_int), ("rotated", ctypes.c_int), ("count", ctypes.c_int), ("h1", ctypes.c_void_p), ("h3", ctypes.c_void_p),
                ("A1", ctypes.c_void_p), ("B1", ctypes.c_void_p * 3)]


def _run(x, w, tail, M, N, K, tb, dt):
    from enzyme_ad.jax import _native
    f = _native.lib()._ZN3emi9gemm_tailEP12ihipStream_tPKvS3_RKNS_11ProductTailEllllii
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p] * 3 + [ctypes.POINTER(_Tail)] + [ctypes.c_int64] * 4 + [ctypes.c_int] * 2
    return f(torch.cuda.current_stream().cuda_stream, x.data_ptr(), w.data_ptr(), ctypes.byref(tail), M, N, K, K if tb else N, tb,
             16 if dt == "bf16" else 11)


def _product(xr, wr, tb, dt):
    w = wr.T if tb else wr
    p, mag, k = xr @ w, np.abs(xr) @ np.abs(w), xr.shape[1]
    return p, (2.0 ** -8 * np.abs(p) if dt == "bf16" else 0.0) + (k + 2) * 2.0 ** -23 * mag


def _close(got, want, bound, dt, what):
    err, room = np.abs(host(got) - want), bound + (2.0 ** -8 if dt == "bf16" else 2.0 ** -19) * np.abs(want)
    assert np.all(err <= room), "%s: worst error / bound %.2f" % (what, float(np.max(err / room)))


def _sigmoid(a):
    return 1.0 / (1.0 + np.exp(-a))


SIZES = {
    ("f32", GATED): [(9, 8, 8), (33, 44, 68), (200, 772, 292), (308, 1404, 516)],
    ("f32", ROTATED): [(9, 8, 8), (35, 72, 68), (235, 288, 292), (721, 288, 284)],
    ("f32", ADJOINT): [(9, 8, 8), (35, 76, 68), (198, 1412, 516), (817, 764, 284)],
    ("bf16", GATED): [(9, 8, 8), (33, 24, 264), (300, 2040, 776), (450, 2808, 1032), (1500, 768, 288), (1500, 1400, 520), (2181, 2040, 776)],
    ("bf16", ROTATED): [(9, 8, 8), (300, 1400, 520), (450, 520, 520), (600, 776, 776), (340, 2056, 2056), (1000, 776, 776), (4001, 1400, 520),
                        (5000, 24, 264)],
    ("bf16", ADJOINT): [(9, 8, 8), (33, 24, 264), (340, 520, 520), (1000, 776, 776), (777, 1400, 520), (1500, 776, 776), (2181, 1032, 1032),
                        (1500, 2040, 776), (5000, 776, 776)],
}
CASES = [(dt, mode) + size for (dt, mode), sizes in SIZES.items() for size in sizes]


@pytest.mark.parametrize("dt,mode,M,N,K", CASES)
def test_products_with_an_elementwise_tail(dt, mode, M, N, K):
    rng = np.random.default_rng(M + N + K + mode)
    x, xr = dev(rng.standard_normal((M, K)), dt)
    out = [torch.full((M, N), 7.0, device=x.device, dtype=x.dtype) for _ in range(3)]
    for tb in (1, 0) if mode == ADJOINT else (1,):
        ws = [dev(rng.standard_normal((N, K) if tb else (K, N)) / np.sqrt(K), dt) for _ in range(3)]
        tail = _Tail(mode=mode)
        for i in range(3):
            tail.C[i] = out[i].data_ptr()
        if mode == ADJOINT:
            (h1, a), (h3, b) = (dev(rng.standard_normal((M, N)), dt) for _ in range(2))
            tail.h1, tail.h3, tail.C[2] = h1.data_ptr(), h3.data_ptr(), None
        else:
            for i in range(3 if mode == ROTATED else 2):
                tail.B[i] = ws[i][0].data_ptr()
        if mode == ROTATED:
            d, seq = max(e for e in (8, 4, 2, 36, 48) if N % e == 0 and e < N or e == 2), (M + 1) // 2
            table, tr = dev(rng.standard_normal((seq, d // 2, 2)), "f32")
            tail.table, tail.seq, tail.head_dim, tail.rotated, tail.count = table.data_ptr(), seq, d, 2, 3
        assert _run(x, ws[0][0], tail, M, N, K, tb, dt) == 0
        prods = [_product(xr, w[1], tb, dt) for w in ws]
        if mode == GATED:
            for i in range(2):
                _close(out[i], prods[i][0], prods[i][1], dt, "h%d" % (1 + 2 * i))
            a, b = host(out[0]), host(out[1])
            _close(out[2], a * _sigmoid(a) * b, 0.0, dt, "g")
        elif mode == ADJOINT:
            (dg, e), s = prods[0], _sigmoid(a)
            slope = 1.0 + a * (1.0 - s)
            _close(out[0], dg * b * s * slope, np.abs(b * s) * (np.abs(slope) * e + 2.0 ** -19 * np.abs(dg) * (1.0 + np.abs(a))), dt, "dh1")
            _close(out[1], dg * a * s, np.abs(a * s) * e, dt, "dh3")
        else:
            at, pair = np.arange(M)[:, None] % seq, np.arange(N)[None, :] % d // 2
            c, s = tr[at, pair, 0], tr[at, pair, 1]
            for i in range(2):
                (p, e), other = prods[i], np.arange(N) ^ 1
                sign = np.where(np.arange(N) % 2 == 0, -1.0, 1.0)
                _close(out[i], c * p + sign * s * p[:, other], np.abs(c) * e + np.abs(s) * e[:, other] + 2.0 ** -22 * (np.abs(c * p) + np.abs(s * p[:, other])), dt, "result %d" % i)
            _close(out[2], prods[2][0], prods[2][1], dt, "result 2")


PAIRS = [("f32", 9, 8, 8, 2), ("f32", 35, 72, 68, 2), ("f32", 130, 1408, 516, 0), ("f32", 235, 288, 292, 2), ("bf16", 9, 8, 8, 2), ("bf16", 33, 24, 264, 2),
         ("bf16", 300, 1400, 520, 0), ("bf16", 450, 520, 520, 2), ("bf16", 777, 776, 776, 2), ("bf16", 1000, 2056, 2056, 0)]


@pytest.mark.parametrize("dt,M,N,K,rotated", PAIRS)
def test_results_of_two_products_each(dt, M, N, K, rotated):
    """A tangent's two products, of three results (two turned) or of two, in one launch."""
    rng = np.random.default_rng(M + N + K)
    (x, xr), (x1, x1r) = (dev(rng.standard_normal((M, K)), dt) for _ in range(2))
    count, d, seq = 3 if rotated else 2, 8, (M + 1) // 2
    ws, w1s = ([dev(rng.standard_normal((N, K)) / np.sqrt(K), dt) for _ in range(count)] for _ in range(2))
    out = [torch.full((M, N), 7.0, device=x.device, dtype=x.dtype) for _ in range(count)]
    table, tr = dev(rng.standard_normal((seq, d // 2, 2)), "f32")
    tail = _Tail(mode=ROTATED, table=table.data_ptr() if rotated else None, seq=seq, head_dim=d, rotated=rotated, count=count, A1=x1.data_ptr())
    for i in range(count):
        tail.B[i], tail.B1[i], tail.C[i] = ws[i][0].data_ptr(), w1s[i][0].data_ptr(), out[i].data_ptr()
    assert _run(x, ws[0][0], tail, M, N, K, 1, dt) == 0
    at, pair, other = np.arange(M)[:, None] % seq, np.arange(N)[None, :] % d // 2, np.arange(N) ^ 1
    c, s, sign = tr[at, pair, 0], tr[at, pair, 1], np.where(np.arange(N) % 2 == 0, -1.0, 1.0)
    for i in range(count):
        p = xr @ ws[i][1].T + x1r @ w1s[i][1].T
        mag = np.abs(xr) @ np.abs(ws[i][1]).T + np.abs(x1r) @ np.abs(w1s[i][1]).T
        e = (2.0 ** -8 * np.abs(p) if dt == "bf16" else 0.0) + (2 * K + 2) * 2.0 ** -23 * mag
        if i < rotated:
            e = np.abs(c) * e + np.abs(s) * e[:, other] + 2.0 ** -22 * (np.abs(c * p) + np.abs(s * p[:, other]))
            p = c * p + sign * s * p[:, other]
        _close(out[i], p, e, dt, "result %d" % i)


def test_what_the_kernels_do_not_take_is_left_to_the_separate_launches():
    """Rows of no whole pieces, operands off 16 bytes, few rows, a k-major weight where there is no kernel: -1 and nothing written."""
    x, w, h = (torch.ones(64 * 64 + 8, device="cuda") for _ in range(3))
    out = [torch.full((64, 64), 7.0, device="cuda") for _ in range(3)]

    def tail(mode, shift=0):
        t = _Tail(mode=mode, h1=h.data_ptr() + shift, h3=h.data_ptr())
        for i in range(3):
            t.B[i], t.C[i] = w.data_ptr(), out[i].data_ptr()
        return t

    for M, N, K, tb, t in ((64, 62, 64, 1, tail(GATED)), (64, 64, 62, 1, tail(ADJOINT)), (8, 64, 64, 1, tail(GATED)), (64, 64, 64, 0, tail(GATED)),
                           (64, 64, 64, 1, tail(ADJOINT, 4))):
        assert _run(x, w, t, M, N, K, tb, "f32") == -1
    assert all(bool((o == 7.0).all()) for o in out)


@pytest.mark.parametrize("dt,mode,M,N,K", CASES + [(dt, 5, M, N, K) for dt, M, N, K, _ in PAIRS])
def test_tails_write_nothing_outside_their_results(dt, mode, M, N, K):
    """Every size above (5: two products to each of three results), the results with room before and behind them."""
    pairs = mode == 5
    mode = ROTATED if pairs else mode
    x, x1, w = (torch.randn(n, K, device="cuda").to(torch.bfloat16 if dt == "bf16" else torch.float32) for n in (M, M, N))
    h = torch.randn(M, N, device="cuda").to(x.dtype)
    table = torch.randn(M, N // 2, 2, device="cuda")
    edge = 4096
    for tb in (1, 0) if mode == ADJOINT else (1,):
        room = [torch.full((M * N + 2 * edge,), 7.0, device="cuda", dtype=x.dtype) for _ in range(3)]
        tail = _Tail(mode=mode, table=table.data_ptr(), seq=M, head_dim=N, rotated=2, count=3, h1=h.data_ptr(), h3=h.data_ptr(),
                     A1=x1.data_ptr() if pairs else None)
        for i in range(3):
            tail.B[i], tail.B1[i], tail.C[i] = w.data_ptr(), w.data_ptr() if pairs else None, room[i].data_ptr() + edge * x.element_size()
        rc = _run(x, w, tail, M, N, K, tb, dt)
        written = {GATED: 3, ROTATED: 3, ADJOINT: 2}[mode] if rc == 0 else 0
        assert rc == 0 or (pairs and rc == -1)           # (three results where the test above has two)
        for i, r in enumerate(room):
            inside = r[edge:edge + M * N]
            assert bool((r[:edge] == 7.0).all()) and bool((r[edge + M * N:] == 7.0).all()), i
            assert bool((inside != 7.0).any()) == (i < written)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_what_either_type_leaves_to_the_separate_launches(dt):
    """As above in both types: rows and contractions of no whole pieces, few rows, operands and results off 16 bytes, a k-major weight
    of two or three results."""
    dtype, v = (torch.bfloat16, 8) if dt == "bf16" else (torch.float32, 4)
    x, w, h = (torch.ones(64 * 64 + 16, device="cuda", dtype=dtype) for _ in range(3))
    table = torch.ones(64 * 64 + 4, device="cuda")
    room = [torch.full((64 * 64 + 16,), 7.0, device="cuda", dtype=dtype) for _ in range(3)]

    def tail(mode, h1=0, c=0, b=0, angles=0):
        t = _Tail(mode=mode, h1=h.data_ptr() + h1, h3=h.data_ptr(), table=table.data_ptr() + angles, seq=64, head_dim=8, rotated=2, count=3)
        for i in range(3):
            t.B[i], t.C[i] = w.data_ptr() + b, room[i].data_ptr() + c
        return t

    for mode in (GATED, ROTATED, ADJOINT):
        for M, N, K in ((64, 64 - v // 2, 64), (64, 64, 64 - v // 2), (8, 64, 64)):
            assert _run(x, w, tail(mode), M, N, K, 1, dt) == -1
        assert _run(x, w, tail(mode, c=8), 64, 64, 64, 1, dt) == -1 and _run(x, w, tail(mode, b=8), 64, 64, 64, 1, dt) == -1
        assert mode == ADJOINT or _run(x, w, tail(mode), 64, 64, 64, 0, dt) == -1
    assert _run(x, w, tail(ADJOINT, h1=8), 64, 64, 64, 1, dt) == -1 and _run(x, w, tail(ROTATED, angles=8), 64, 64, 64, 1, dt) == -1
    assert all(bool((r == 7.0).all()) for r in room)


@pytest.mark.parametrize("dt,pairs", [(dt, pairs) for dt in ("f32", "bf16") for pairs in (0, 1)])
@pytest.mark.parametrize("M,N,K", [(35, 72, 72), (233, 288, 288)])
def test_a_result_that_is_not_turned_keeps_its_infinities(dt, pairs, M, N, K):
    """One infinity or NaN in a weight's row j: column j of that result, and of a turned one its pair's other column, nothing else."""
    for value in (float("inf"), float("nan")):
        x, x1 = (torch.rand(M, K, device="cuda").to(torch.bfloat16 if dt == "bf16" else torch.float32) + 0.5 for _ in range(2))
        ws, w1s = ([torch.randn(N, K, device="cuda").to(x.dtype) for _ in range(3)] for _ in range(2))
        for i, j in enumerate((4, 11, N - 1)):
            (w1s if pairs else ws)[i][j, 5] = value
        out = [torch.full((M, N), 7.0, device="cuda", dtype=x.dtype) for _ in range(3)]
        table = torch.rand(M, 4, 2, device="cuda") + 0.5
        tail = _Tail(mode=ROTATED, table=table.data_ptr(), seq=M, head_dim=8, rotated=2, count=3, A1=x1.data_ptr() if pairs else None)
        for i in range(3):
            tail.B[i], tail.B1[i], tail.C[i] = ws[i].data_ptr(), w1s[i].data_ptr() if pairs else None, out[i].data_ptr()
        assert _run(x, ws[0], tail, M, N, K, 1, dt) == 0
        for o, columns in zip(out, ((4, 5), (10, 11), (N - 1,))):
            wrong = torch.zeros(N, dtype=torch.bool, device="cuda")
            wrong[list(columns)] = True
            assert bool((o.isfinite() == ~wrong).all())
        assert bool((out[2][:, N - 1].isnan() if value != value else out[2][:, N - 1] == value).all())
