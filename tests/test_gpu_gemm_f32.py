"""The fp32 GEMM kernels at the sizes where their tiles, stages and splits end: every block shape, each layout, one
product, a group of independent ones and a group summed into one, against float64 products.  An fp32 sum of n products in
any order is within n * 2^-24 * sum |a b| of the exact one, to first order (its roundings, one per term and one per
product, are each at most half a unit in the last place of a partial sum); twice that is allowed."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host

pytestmark = pytest.mark.gpu


def _check(got, ref, bound, what):
    err = np.abs(host(got) - ref)
    assert np.all(err <= bound), "%s: worst error / bound %.2f" % (what, float(np.max(err / bound)))


# what each is there for; tests/test_host_boundary.py holds them to reaching every kernel
SIZES = [
    (4, 4, 4, 2),            # less than one piece of every stage
    (32, 32, 64, 3),         # exactly one 32-tile and one stage
    (36, 28, 68, 3),         # a ragged row of tiles, one piece past a stage
    (100, 512, 516, 3),      # 32-tiles, ragged rows
    (12, 20, 20004, 2),      # a single tile: splits of a long contraction, ragged last stage
    (260, 1028, 772, 2),     # 64-tiles of the fp32 instructions, splits
    (704, 2812, 1028, 2),    # ragged columns: 64-tiles of the bf16 instructions, summed too; a group: of the fp32 ones
    (708, 1540, 292, 2),     # 128 x 64, ragged both ways
    (1996, 772, 2052, 2),    # 128-tiles, splits; summed: splits that straddle the products
    (2052, 2044, 68, 2),     # 64-tiles of the fp32 instructions, ragged both ways; a group, summed: 128 x 64
    (772, 1412, 28, 6),      # a group: 128-tiles of the fp32 instructions, one stage
    (1412, 260, 772, 3),     # a group: 128 x 64; summed: its splits straddle the products
    (516, 1092, 516, 3),     # a group: 64-tiles of the bf16 instructions; summed: 128-tiles with splits
    (1004, 772, 516, 2),     # 64-tiles of the fp32 instructions; a group: 128 x 64; summed: 128-tiles with splits
]


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,count", SIZES)
def test_f32_tiles_stages_and_splits(ta, tb, M, N, K, count):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + 3 * N + 7 * K + 2 * ta + tb)
    As, Ars = zip(*[dev(rng.standard_normal((K, M) if ta else (M, K)), "f32") for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((N, K) if tb else (K, N)), "f32") for _ in range(count)])
    Rs, Rrs = zip(*[dev(rng.standard_normal((M, N)), "f32") for _ in range(count)])
    mm = lambda f: [f(a.T if ta else a) @ f(b.T if tb else b) for a, b in zip(Ars, Brs)]
    prods, mags = mm(lambda t: t), mm(np.abs)
    eps = 2.0 ** -23
    bounds = [(K + 2) * eps * (m + np.abs(r)) for m, r in zip(mags, Rrs)]
    _check(ops.gemm(As[0], Bs[0], bool(ta), bool(tb)), prods[0], bounds[0], "one product")
    _check(ops.gemm(As[0], Bs[0], bool(ta), bool(tb), Rs[0]), prods[0] + Rrs[0], bounds[0], "one product + residual")
    for o, p, r, b in zip(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), list(Rs)), prods, Rrs, bounds):
        _check(o, p + r, b, "group + residual")
    total = ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), [Rs[0]], sum_into_one=True)
    _check(total, sum(prods) + Rrs[0], (count * K + 2) * eps * (sum(mags) + np.abs(Rrs[0])), "summed + residual")
    again = ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), [Rs[0]], sum_into_one=True)
    assert torch.equal(total, again)          # fixed order of summation


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0)])
@pytest.mark.parametrize("M,N,K,count", [(2048, 2048, 4096, 1), (1996, 772, 2052, 3), (36, 768, 8192, 3), (256, 288, 4000, 12)])
def test_f32_sums_in_short_chains(ta, tb, M, N, K, count):
    """With terms of random sign the partial sum of j of them has variance j, and each addition is off by at most 2^-24 of
    it: chains of c of K terms, added up, are off by sqrt((c + K / c) / 2) 2^-24 of the result in the mean square, and one
    chain of all K terms by sqrt(K / 2) 2^-24 (and both in practice by about 0.45 of that).  Chains are of 32 to 64 terms."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    As, Ars = zip(*[dev(rng.standard_normal((K, M) if ta else (M, K)), "f32") for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((N, K) if tb else (K, N)), "f32") for _ in range(count)])
    prods = [(a.T if ta else a) @ (b.T if tb else b) for a, b in zip(Ars, Brs)]
    off = lambda got, ref: float(np.linalg.norm(host(got) - ref) / np.linalg.norm(ref))
    bound = lambda k: 2.0 ** -24 * np.sqrt((64 + k / 32) / 2)
    assert off(ops.gemm(As[0], Bs[0], bool(ta), bool(tb)), prods[0]) <= bound(K)
    if count > 1:
        for o, p in zip(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb)), prods):
            assert off(o, p) <= bound(K)
        assert off(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), sum_into_one=True), sum(prods)) <= bound(count * K)


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,count", [
    (9, 3, 4, 2), (31, 33, 256, 3), (65, 101, 260, 2), (33, 63, 384, 48), (129, 31, 388, 3), (63, 97, 768, 2), (97, 33, 772, 3),
    (33, 31, 4100, 2),       # splits one by one
    (321, 801, 520, 5),      # more than 1024 blocks
])
def test_f32_rows_that_are_no_whole_pieces(ta, tb, M, N, K, count):
    """k-major operands with odd rows, k-contiguous ones of whole 16-byte pieces: the contraction at the edges of the
    forms that take all of it at once, one product and a group with and without residuals."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + 3 * N + 7 * K + 2 * ta + tb)
    As, Ars = zip(*[dev(rng.standard_normal((K, M) if ta else (M, K)), "f32") for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((N, K) if tb else (K, N)), "f32") for _ in range(count)])
    Rs, Rrs = zip(*[dev(rng.standard_normal((M, N)), "f32") for _ in range(count)])
    mm = lambda f: [f(a.T if ta else a) @ f(b.T if tb else b) for a, b in zip(Ars, Brs)]
    prods, mags = mm(lambda t: t), mm(np.abs)
    bounds = [(K + 2) * 2.0 ** -23 * (m + np.abs(r)) for m, r in zip(mags, Rrs)]
    _check(ops.gemm(As[0], Bs[0], bool(ta), bool(tb), Rs[0]), prods[0] + Rrs[0], bounds[0], "one product + residual")
    for o, p, b in zip(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb)), prods, bounds):
        _check(o, p, b, "group")
    for o, p, r, b in zip(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), list(Rs)), prods, Rrs, bounds):
        _check(o, p + r, b, "group + residual")


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [
    (2050, 1538, 262),       # 128-tiles, every edge ragged
    (258, 290, 20010),       # 128-tiles in planes of K
    (130, 70, 258),          # 32-tiles
])
def test_f32_windows_of_odd_rows(ta, tb, M, N, K):
    """Aligned rows that are two elements short of whole 16-byte pieces, with NaN between them, and no memory behind the
    last row: nothing of either enters the product, nothing is written between the rows of the result."""
    from enzyme_ad.jax import _native as nat
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)

    def window(rows, cols):
        a = rng.standard_normal((rows, cols))
        ld = cols + 2
        room = torch.full((rows * ld - 2,), float("nan"), device="cuda")
        t = torch.as_strided(room, (rows, cols), (ld, 1))
        t.copy_(torch.from_numpy(a))
        return t, ld, host(t)

    A, lda, Ar = window(*((K, M) if ta else (M, K)))
    B, ldb, Br = window(*((N, K) if tb else (K, N)))
    R, ldr, Rr = window(M, N)
    C = torch.full((M, N + 2), 7.0, device="cuda")
    a, b = Ar.T if ta else Ar, Br.T if tb else Br
    lib = nat.lib()
    nbytes = lib.emi_gemm_workspace_bytes(M, N, K, ta, tb, nat.EMI_F32)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
    nat.check(lib.emi_gemm_ws(torch.cuda.current_stream().cuda_stream, A.data_ptr(), B.data_ptr(), R.data_ptr(), C.data_ptr(), ws.data_ptr(),
                              nbytes, M, N, K, lda, ldb, ldr, N + 2, ta, tb, nat.EMI_F32))
    _check(C[:, :N], a @ b + Rr, (K + 2) * 2.0 ** -23 * (np.abs(a) @ np.abs(b) + np.abs(Rr)), "windows")
    assert bool((C[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(1, 64, 4100), (4, 688, 5692), (8, 68, 20000), (5, 688, 5689)])
def test_f32_gradients_of_few_rows(M, N, K):
    """A handful of rows of a k-major A against a long contraction: split where rows are whole 16-byte pieces."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K)
    (A, Ar), (B, Br), (R, Rr) = (dev(rng.standard_normal(s), "f32") for s in ((K, M), (K, N), (M, N)))
    bound = (K + 2) * 2.0 ** -23 * (np.abs(Ar).T @ np.abs(Br) + np.abs(Rr))
    _check(ops.gemm(A, B, True, False), Ar.T @ Br, bound, "one product")
    _check(ops.gemm(A, B, True, False, R), Ar.T @ Br + Rr, bound, "one product + residual")


@pytest.mark.parametrize("dt,ta,tb,M,N,K,count", [("f32", 1, 0, 64, 64, 8192, 4), ("f32", 0, 0, 300, 64, 4096, 2), ("bf16", 0, 0, 16, 1032, 8200, 3),
                                                  ("bf16", 0, 1, 24, 72, 16400, 2)])
def test_groups_that_run_faster_one_by_one(dt, ta, tb, M, N, K, count):
    """Few tiles and a long contraction: each product of the group is split over K.  Their planes share the workspace, one
    after the other on the stream."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K + ta)
    As, Ars = zip(*[dev(rng.standard_normal((K, M) if ta else (M, K)), dt) for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((N, K) if tb else (K, N)), dt) for _ in range(count)])
    Rs, Rrs = zip(*[dev(rng.standard_normal((M, N)), dt) for _ in range(count)])
    unit = 2.0 ** -8 if dt == "bf16" else 0.0
    for rs, adds in ((None, [0.0] * count), (list(Rs), Rrs)):
        for o, a, b, r in zip(ops.gemm_grouped(list(As), list(Bs), bool(ta), bool(tb), rs), Ars, Brs, adds):
            x, y = a.T if ta else a, b.T if tb else b
            ref = x @ y + r
            _check(o, ref, unit * np.abs(ref) + (K + 2) * 2.0 ** -23 * (np.abs(x) @ np.abs(y) + np.abs(r)), "group")
