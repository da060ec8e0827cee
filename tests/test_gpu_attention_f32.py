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
