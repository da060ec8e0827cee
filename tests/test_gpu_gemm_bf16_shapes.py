"""The bf16 GEMM's block shapes for few tokens and narrow results, at the sizes where their tiles, stages and splits end:
one product, a group of independent ones and a group summed into one, B k-contiguous and k-major, against float64 products
of the stored values.  The result is an fp32 sum rounded once to bf16: half a unit in the last place of the result (2^-9
relative) plus the roundings of the sum, at most n * 2^-24 * sum |a b| to first order; twice that sum is allowed."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host

pytestmark = pytest.mark.gpu


def _check(got, ref, mag, n, what):
    bound = 2.0 ** -8 * np.abs(ref) + (n + 2) * 2.0 ** -23 * mag
    err = np.abs(host(got) - ref)
    assert np.all(err <= bound), "%s: worst error / bound %.2f" % (what, float(np.max(err / bound)))


# what each is there for; tests/test_host_boundary.py holds them to reaching every kernel
SIZES = [
    (9, 8, 8, 2),             # less than one piece of every stage
    (33, 24, 264, 3),         # 32-tiles whose wavefronts share k (k-contiguous B), one piece past a stage
    (64, 768, 768, 3),        # exact 32-tiles
    (40, 104, 8200, 2),       # few tiles, long contraction: splits, a ragged last stage
    (300, 1400, 520, 2),      # 64-tiles in a ring of three stages, ragged rows and columns
    (300, 2808, 1032, 2),     # a group: 64-tiles, two to a CU, in a ring of two
    (1500, 504, 512, 3),      # a group: 64-tiles of 64 k a stage, three to a CU (k-contiguous B)
    (30, 2800, 504, 12),      # the same, k-major B
    (777, 2040, 776, 2),      # 128 x 64 tiles of 128 k a stage, ragged
    (900, 520, 328, 2),       # a group: 128 x 64 tiles of 64 k a stage (k-major B)
    (1000, 4088, 520, 2),     # 128-tiles in a ring of three stages, eight wavefronts
    (3000, 1032, 328, 2),     # 128 x 64 tiles of 64 k a stage; a group: 128-tiles, two to a CU; summed: one pass over both
    (600, 2056, 4104, 2),     # 128-tiles, of sixteen wavefronts; with splits (k-contiguous B); summed: splits that straddle the products
    (777, 264, 2056, 2),      # summed: 128 x 64 tiles with splits (k-major B)
    (300, 1000, 16392, 2),    # 64-tiles with splits
    (1000, 2056, 8200, 1),    # 256-tiles with splits (k-contiguous B)
    (2056, 2048, 8200, 1),    # more than 4 M results: 256-tiles with splits all the same (k-contiguous B)
]


@pytest.mark.parametrize("tb", [1, 0])
@pytest.mark.parametrize("M,N,K,count", SIZES)
def test_bf16_tiles_stages_and_splits(tb, M, N, K, count):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + 3 * N + 7 * K + tb)
    As, Ars = zip(*[dev(rng.standard_normal((M, K)), "bf16") for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((N, K) if tb else (K, N)), "bf16") for _ in range(count)])
    Rs, Rrs = zip(*[dev(rng.standard_normal((M, N)), "bf16") for _ in range(count)])
    mm = lambda f: [f(a) @ f(b.T if tb else b) for a, b in zip(Ars, Brs)]
    prods, mags = mm(lambda t: t), mm(np.abs)
    _check(ops.gemm(As[0], Bs[0], False, bool(tb)), prods[0], mags[0], K, "one product")
    _check(ops.gemm(As[0], Bs[0], False, bool(tb), Rs[0]), prods[0] + Rrs[0], mags[0] + np.abs(Rrs[0]), K, "one product + residual")
    for o, p, r, m in zip(ops.gemm_grouped(list(As), list(Bs), False, bool(tb), list(Rs)), prods, Rrs, mags):
        _check(o, p + r, m + np.abs(r), K, "group + residual")
    total = ops.gemm_grouped(list(As), list(Bs), False, bool(tb), [Rs[0]], sum_into_one=True)
    _check(total, sum(prods) + Rrs[0], sum(mags) + np.abs(Rrs[0]), count * K, "summed + residual")
    again = ops.gemm_grouped(list(As), list(Bs), False, bool(tb), [Rs[0]], sum_into_one=True)
    assert torch.equal(total, again)          # fixed order of summation


@pytest.mark.parametrize("M,N,K,count", [
    (136, 72, 3, 2),          # fewer tokens than a k-row group
    (256, 264, 77, 3),        # 128-tiles, a ragged last stage
    (264, 136, 4099, 2),      # splits of a long odd contraction
    (4096, 3080, 301, 1),     # 256-tiles
    (256, 256, 301, 48),      # a group that fills the chip with 256-tiles
])
def test_bf16_weight_gradients_of_any_number_of_tokens(M, N, K, count):
    """dW = dY^T . X: both operands are k-major, K (the tokens) is a multiple of nothing."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K)
    As, Ars = zip(*[dev(rng.standard_normal((K, M)), "bf16") for _ in range(count)])
    Bs, Brs = zip(*[dev(rng.standard_normal((K, N)), "bf16") for _ in range(count)])
    r, rr = dev(rng.standard_normal((M, N)), "bf16")
    prods, mags = [a.T @ b for a, b in zip(Ars, Brs)], [np.abs(a).T @ np.abs(b) for a, b in zip(Ars, Brs)]
    _check(ops.gemm(As[0], Bs[0], True, False, r), prods[0] + rr, mags[0] + np.abs(rr), K, "one product + residual")
    if count > 1:
        for o, p, m in zip(ops.gemm_grouped(list(As), list(Bs), True, False), prods, mags):
            _check(o, p, m, K, "group")
