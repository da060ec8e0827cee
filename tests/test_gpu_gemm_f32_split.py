"""fp32 products on the bf16 matrix cores: the sizes at which each block shape is chosen and its tiles, stages in flight and
splits end, and operands that three bf16 numbers do not hold (infinite, NaN, beyond the largest bf16, below what the
third one reaches), which are multiplied as fp32 numbers.  Against float64 products."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host

pytestmark = pytest.mark.gpu

# what each is there for; tests/test_host_boundary.py holds them to reaching every kernel
SIZES = [
    (780, 2308, 772),        # blocks of 64 x 64, a last round of one stage
    (180, 2820, 1284),       # the same, three splits
    (4004, 2372, 28),        # 128 x 64, fewer stages than are in flight
    (900, 1284, 1036),       # the same, three splits
    (716, 2756, 100),        # 128 x 128, a last round of one stage
    (708, 1092, 2052),       # the same, four splits
]


def _operands(rng, M, N, K, ta, tb):
    return rng.standard_normal((K, M) if ta else (M, K)), rng.standard_normal((N, K) if tb else (K, N))


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", SIZES + [(1000, 1028, 1036), (1996, 772, 2052), (1060, 1092, 2052), (777, 4096, 772)])
def test_errors_of_an_fp32_product(ta, tb, M, N, K):
    """Within (K + 2) 2^-23 sum |a b|, as any order of fp32 sums is (three dropped products of 2^-25 each are less than what
    the roundings of a shorter chain leave of it), and in the mean square no further off than chains of 64 terms."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    a, b = _operands(rng, M, N, K, ta, tb)
    (A, Ar), (B, Br), (R, Rr) = dev(a, "f32"), dev(b, "f32"), dev(rng.standard_normal((M, N)), "f32")
    x, y = Ar.T if ta else Ar, Br.T if tb else Br
    ref = x @ y
    got = host(ops.gemm(A, B, bool(ta), bool(tb), R))
    bound = (K + 2) * 2.0 ** -23 * (np.abs(x) @ np.abs(y) + np.abs(Rr))
    assert np.all(np.abs(got - ref - Rr) <= bound)
    got = host(ops.gemm(A, B, bool(ta), bool(tb)))
    assert np.linalg.norm(got - ref) <= 2.0 ** -24 * np.sqrt((64 + K / 32) / 2) * np.linalg.norm(ref)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0)])
@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("what", ["infinite", "nan", "huge", "tiny", "tiny rows", "tiny products", "denormal", "zero"])
def test_numbers_that_do_not_split(what, ta, tb, M, N, K):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    a, b = _operands(rng, M, N, K, ta, tb)
    a, b = a.astype(np.float32), b.astype(np.float32)
    at = lambda m, k: (k, m) if ta else (m, k)                  # of row m of the result, term k
    if what == "infinite":
        a[at(3, 5)], a[at(M - 1, K - 1)] = np.inf, -np.inf
        b[(N - 2, 7) if tb else (7, N - 2)] = np.inf
    elif what == "nan":
        a[at(M // 2, K - 2)] = np.nan
    elif what == "huge":                                        # finite, but rounds to an infinite bf16
        a[at(3, 5)] = 3.4e38
        b *= np.float32(1e-3)
    elif what == "tiny":
        a *= np.float32(1e-36)
    elif what == "tiny rows":                                   # beside ordinary ones
        a[(slice(None), slice(5, 9)) if ta else slice(5, 9)] *= np.float32(1e-36)
    elif what == "tiny products":                               # of numbers that split
        a *= np.float32(1e-20)
        b *= np.float32(1e-21)
    elif what == "denormal":                                    # and exactly a bf16 number
        a = np.copysign(np.float32(2.0 ** -130), a)
        b *= np.float32(1e10)
    else:
        a[:] = 0
    A, B = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    got = host(ops.gemm(A, B, bool(ta), bool(tb)))
    x, y = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = x @ y
        mag = np.abs(x) @ np.abs(y)
    finite = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    bound = (K + 2) * 2.0 ** -23 * mag + 2.0 ** -149 * K         # denormal results
    assert np.all(np.abs(got[finite] - ref[finite]) <= bound[finite])


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [s for s in SIZES if s[2] > 32])
@pytest.mark.parametrize("scale", [1e-31, 1e-34, 1e-37, 1e-41])
def test_small_numbers_keep_their_bits(scale, ta, tb, M, N, K):
    """A row of A, a column of B and single terms far below their neighbours are as exact as any other: what a number loses
    is not measured by the largest one of its tile.  An fp32 sum of K terms, plus the step of denormal products."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    a0, b0 = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)

    def check(a, b, what):
        put = lambda t, turn: torch.from_numpy(np.ascontiguousarray(t.T if turn else t)).cuda()
        got = host(ops.gemm(put(a, ta), put(b, tb), bool(ta), bool(tb)))
        x, y = a.astype(np.float64), b.astype(np.float64)
        err, bound = np.abs(got - x @ y), (K + 2) * 2.0 ** -23 * (np.abs(x) @ np.abs(y)) + 2.0 ** -149 * K
        assert np.all(err <= bound), "%s: worst error / bound %.2f" % (what, float(np.max(err / bound)))

    a, b = a0.copy(), b0.copy()
    a[5:9] *= np.float32(scale)
    b[:, N - 3:] *= np.float32(scale)
    check(a, b0, "rows of A")
    check(a0, b, "columns of B")
    check(a, b0 * np.float32(1e20), "rows of A against large numbers")
    a, b = a0.copy(), b0.copy()
    a[:, K // 2:] *= np.float32(scale)
    b[:K // 2] = 0
    check(a, b, "terms whose neighbours meet zeros")


@pytest.mark.parametrize("M,N,K", [(2000, 768, 768), (776, 4096, 4096)])
def test_a_product_that_is_multiplied_again_takes_a_few_times_as_long(M, N, K):
    """Every tile of a product with numbers that do not split: once as bf16 numbers and once on the fp32 instructions, whose
    products take 1.2 to 1.4 times as long.  Twice that is allowed; loads without a stage in the LDS took 7 to 11 times."""
    from enzyme_ad.jax import ops
    a, b = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")

    def us(a):
        for _ in range(3):
            ops.gemm(a, b, False, True)
        times = []
        for _ in range(5):
            start, end = torch.cuda.Event(True), torch.cuda.Event(True)
            start.record()
            for _ in range(10):
                ops.gemm(a, b, False, True)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[2]

    assert us(a * 1e-36) <= 5 * us(a)
