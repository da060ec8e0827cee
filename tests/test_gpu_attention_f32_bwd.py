"""The fp32 attention adjoint on both sides of the number of blocks up to which dQ and dK/dV are one launch (and dK/dV forms
rowsum(dO O) itself), against float64.  The bound is that of the tiles' test: two sums of up to d + S roundings each."""
import numpy as np
import pytest

from gpu_util import dev, host
from oracle import llama_ref as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("B,h,S,d", [(4, 16, 256, 64), (4, 16, 257, 64), (1, 7, 31, 48), (2, 32, 128, 128), (2, 32, 129, 128), (1, 3, 47, 112),
                                     # heads of 128: rows of middling length, few short ones, few long ones; long rows of 48; without the mask
                                     (2, 16, 255, 128), (2, 16, 257, 128), (1, 12, 128, 128), (1, 2, 1040, 128), (1, 8, 1030, 48), (1, 8, 1041, 48),
                                     (1, 28, 256, 96), (1, 32, 255, 96), (1, 20, 512, 48), (3, 11, 512, 48)])
def test_f32_attention_adjoint_as_one_launch_or_two(B, h, S, d, layout, causal):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(S * d + h)

    def put(a):
        if layout == "bshd":
            t, r = dev(a.transpose(0, 2, 1, 3).reshape(B, S, h * d), "f32")
            return t, r.reshape(B, S, h, d).transpose(0, 2, 1, 3)
        return dev(a, "f32")

    (q, qr), (k, kr), (v, vr), (do, dor) = (put(rng.standard_normal((B, h, S, d))) for _ in range(4))
    with ops.Tape() as tape:
        o = ops.attention(q, k, v, h, causal=causal, layout=layout)
    for got, want in zip(tape.backward([o], [do], [q, k, v]), L.attention_bwd(qr, kr, vr, dor, causal=causal)):
        got = host(got)
        if layout == "bshd":
            got = got.reshape(B, S, h, d).transpose(0, 2, 1, 3)
        assert float(np.max(np.abs(got - want))) <= 2 * (d + S) * 2.0 ** -23 * float(np.max(np.abs(want)))
