"""fp32 attention at the sizes where its four wavefronts run out of 16-row tiles, a tile is cut by the end of the sequence,
and the blocks do not divide over the XCDs; forward, log-sum-exp and adjoint against float64.  A row's output is a
combination of S rows of v whose weights carry about (d + S) roundings each; with inputs of order one the differences stay
below (d + S) * 2^-23 of the largest entry, and an adjoint entry goes through two such sums.  With one key dS is the
difference of two sums of d products dO v that are equal but for their rounding, and dQ and dK are that times an entry of
k or q: zero up to the same bound on those sums."""
import numpy as np
import pytest
import torch

from gpu_util import dev, rel_err, host
from oracle import llama_ref as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,h,S,d", [(1, 1, 1, 16), (1, 3, 15, 32), (2, 5, 16, 48), (1, 3, 17, 64), (1, 2, 48, 80), (3, 3, 63, 48), (2, 7, 64, 64),
                                     (1, 9, 65, 96), (1, 2, 129, 112), (1, 3, 250, 128), (2, 3, 515, 64)])
def test_f32_attention_tiles(B, h, S, d, causal):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(1000 * S + d)
    (q, qr), (k, kr), (v, vr), (do, dor) = (dev(rng.standard_normal((B, h, S, d)), "f32") for _ in range(4))
    with ops.Tape() as tape:
        o = ops.attention(q, k, v, h, causal=causal, layout="bhsd")
    grads = tape.backward([o], [do], [q, k, v])
    _, lse, _ = ops.attention_raw(q, k, v, h, 1.0 / np.sqrt(d), causal, "bhsd")
    ro, rlse = L.attention_fwd(qr, kr, vr, causal=causal)
    bound = (d + S) * 2.0 ** -23
    assert rel_err(host(o), ro) <= bound
    assert rel_err(host(lse).reshape(rlse.shape), rlse) <= bound
    for got, want, other, name in zip(grads, L.attention_bwd(qr, kr, vr, dor, causal=causal), (kr, qr, qr), "qkv"):
        size = float(np.max(np.abs(want)))
        if S == 1 and name != "v":
            assert size < 1e-12
            size = float(np.max(np.abs(dor)) * np.max(np.abs(vr)) * np.max(np.abs(other)) * np.sqrt(d))
        assert float(np.max(np.abs(host(got) - want))) <= 2 * bound * size, name


def test_f32_attention_keeps_non_finite_values():
    """A NaN or an infinity in a row of v reaches the queries that see it.  Of the others it reaches at most those of the
    same 16-row tile, whose weight for that row is 0 and is multiplied by it."""
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(5)
    q, k, v = (dev(rng.standard_normal((1, 2, 100, 48)), "f32")[0] for _ in range(3))
    clean = ops.attention(q, k, v, 2, layout="bhsd")
    for at, value in ((37, float("nan")), (70, float("inf"))):
        bad = v.clone()
        bad[0, 1, at] = value
        o = ops.attention(q, k, bad, 2, layout="bhsd")
        assert torch.equal(o[0, 0], clean[0, 0]) and torch.equal(o[0, 1, :at - at % 16], clean[0, 1, :at - at % 16])
        assert not torch.isfinite(o[0, 1, at:]).any()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,h,S,d", [(1, 1, 1, 16), (1, 3, 17, 32), (2, 5, 63, 48), (1, 7, 64, 64), (1, 2, 130, 80), (1, 9, 250, 128), (1, 19, 513, 128),
                                     (2, 12, 545, 96), (3, 9, 700, 80), (5, 40, 31, 112), (2, 3, 515, 64)])
def test_f32_attention_tangent_tiles(B, h, S, d, causal):
    """One and two sets of 16 queries a block (head sizes from 80 on, rows and blocks enough: 513, 545, 700 causal; 200 pairs of
    tiles without the mask), the last set cut or empty.  A tangent entry is the sum of S products with weights of 2d products
    each, minus the mean weight times a sum of S: two such sums, each within the bound of the module, of terms as large as
    sqrt(2 d) scale = sqrt(2) times the entries' own size."""
    from enzyme_ad.jax import ops, jvp
    rng = np.random.default_rng(7 * S + d)
    (q, qr), (k, kr), (v, vr), (tq, tqr), (tk, tkr), (tv, tvr) = (dev(rng.standard_normal((B, h, S, d)), "f32") for _ in range(6))

    def fn(a, b, c):
        return ops.attention(a, b, c, h, causal=causal, layout="bhsd")

    bound = 4 * (d + S) * 2.0 ** -23
    for given in ((1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1)):
        _, to = jvp(fn, (q, k, v), tuple(t if g else None for t, g in zip((tq, tk, tv), given)))
        want = L.attention_jvp(qr, kr, vr, *(t * g for t, g in zip((tqr, tkr, tvr), given)), causal=causal)
        size = max(float(np.max(np.abs(want))), 1.0)      # one key: the tangent is tv, what q and k give is rounding
        assert float(np.max(np.abs(host(to) - want))) <= bound * size, given


def test_f32_attention_tangent_of_other_layouts():
    """Rows that do not start on 16-byte boundaries go to the kernel of one wavefront per query; both layouts agree with it."""
    from enzyme_ad.jax import ops, jvp
    rng = np.random.default_rng(11)
    B, h, S, d = 2, 4, 70, 80
    x = [dev(rng.standard_normal((B, S, h * d)), "f32") for _ in range(6)]
    heads = lambda a: np.ascontiguousarray(a.reshape(B, S, h, d).transpose(0, 2, 1, 3))
    want = L.attention_jvp(*(heads(r) for _, r in x), causal=True)
    bound = 4 * (d + S) * 2.0 ** -23 * float(np.max(np.abs(want)))
    for shift in (0, 1):
        args = []
        for t, _ in x:
            room = torch.empty(t.numel() + 4, device=t.device)
            moved = room[shift:shift + t.numel()].view(t.shape)
            moved.copy_(t)
            args.append(moved)
        _, to = jvp(lambda a, b, c: ops.attention(a, b, c, h), tuple(args[:3]), tuple(args[3:]))
        assert float(np.max(np.abs(heads(host(to)) - want))) <= bound, shift


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,h,S,d", [(1, 3, 96, 48), (1, 5, 257, 32), (1, 2, 385, 64), (2, 3, 390, 16), (1, 7, 520, 48), (1, 40, 96, 48)])
def test_f32_attention_eight_wavefronts(B, h, S, d, causal):
    """Few blocks of long rows have eight wavefronts, some of them without a tile of a short row; one launch and two of the
    adjoint beside each other.  Bounds as above."""
    test_f32_attention_tiles(B, h, S, d, causal)


@pytest.mark.parametrize("B,h,S,d", [(1, 8, 321, 48), (1, 9, 321, 48), (1, 6, 430, 64), (1, 5, 590, 64), (2, 2, 650, 48), (1, 3, 900, 32)])
def test_f32_attention_long_rows_of_several_heads(B, h, S, d):
    """More than 160 blocks: eight wavefronts where an XCD's rows begin with a head's or are part of one, else four.  Bounds as above."""
    test_f32_attention_tiles(B, h, S, d, True)


@pytest.mark.parametrize("h,S,d", [(3, 40, 48), (6, 256, 48), (5, 33, 80), (2, 70, 32), (40, 300, 64), (3, 50, 40)])
def test_f32_attention_adjoint_turns_its_operands_back(h, S, d):
    """The inverse rotation where dq and dk leave, with an odd and an even number of 16-column tiles a head (a pair's elements in
    two lanes or in one), against the adjoint and a pass over each: the same bits; head_dim 40 takes the passes."""
    from enzyme_ad.jax import ops, _native
    rng = np.random.default_rng(S + d)
    q, k, v, do = (dev(rng.standard_normal((2, S, h * d)), "f32")[0] for _ in range(4))
    table = ops.rope_table(S, d, device=q.device)
    o, lse, shape = ops.attention_raw(q, k, v, h, d ** -0.5, True, "bshd")
    B, S_, d_, sb, sh, ss = shape
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    ws = torch.empty(lib.emi_attn_bwd_workspace_bytes(B, h, S, d), dtype=torch.uint8, device=q.device)
    one, two = ([torch.empty_like(q) for _ in range(3)] for _ in range(2))
    head = [t.data_ptr() for t in (q, k, v, o, lse, do)]
    tail = [ws.data_ptr(), ws.numel(), B, h, S, d, sb, sh, ss, d ** -0.5, 1, 11]
    _native.check(lib.emi_attn_bwd_rope(st, *head, *(t.data_ptr() for t in one), table.data_ptr(), *tail))
    _native.check(lib.emi_attn_bwd(st, *head, *(t.data_ptr() for t in two), *tail))
    for t in two[:2]:
        _native.check(lib.emi_rope(st, t.data_ptr(), table.data_ptr(), t.data_ptr(), B, S, h, d, 1, 11))
    assert all(torch.equal(a, b) for a, b in zip(one, two))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("h,S,d", [(2, 100, 48), (3, 50, 40), (19, 530, 128)])
def test_f32_attention_tangent_keeps_non_finite_values(h, S, d, causal):
    """A NaN or an infinity in a row of v or of its tangent reaches the queries that see it and no other: one and two sets of 16
    queries a block (530 of 19 heads), head_dim 40 in the kernel of one wavefront per query.  The row of the last key also stands
    in for rows past the end; an infinity that every query sees stays one.  Bound of the finite entries as above."""
    from enzyme_ad.jax import ops, jvp
    rng = np.random.default_rng(S + d)
    raw = [rng.standard_normal((1, h, S, d)) for _ in range(6)]
    bound = 4 * (d + S) * 2.0 ** -23

    def run(arrays):
        a = [dev(x, "f32")[0] for x in arrays]
        return host(jvp(lambda q, k, v: ops.attention(q, k, v, h, causal=causal, layout="bhsd"), tuple(a[:3]), tuple(a[3:]))[1])

    clean = run(raw)
    for which in (2, 5):
        for at, value in ((S - 1, np.inf), (37, np.nan), (21, np.inf), (16, np.nan)):
            bad, without = list(raw), list(raw)
            bad[which], without[which] = raw[which].copy(), raw[which].copy()
            bad[which][0, 1, at] = value
            without[which][0, 1, at] = 0.0
            got = run(bad)
            seen = slice(at, S) if causal else slice(0, S)
            assert np.array_equal(got[0, 0], clean[0, 0]) and np.array_equal(got[0, 2:], clean[0, 2:])
            assert not np.isfinite(got[0, 1, seen]).any()
            if which == 5 and value == np.inf:
                assert np.isposinf(got[0, 1, seen]).all()
            if causal:
                want = L.attention_jvp(*(dev(x, "f32")[1][:, 1:2] for x in without), causal=True)
                size = max(float(np.max(np.abs(want))), 1.0)
                assert float(np.max(np.abs(got[0, 1, :at] - want[0, 0, :at]))) <= bound * size, (which, at, value)
