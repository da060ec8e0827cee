"""bf16 attention where the keys of 32 queries are dealt to four wavefronts, and on both sides of the sizes at which that is
chosen: shares cut by the end of the sequence, wavefronts that see no key at all, both head sizes, both layouts.  Against
float64 on the stored values; P and the outputs are rounded to 8 bits once each, dS once more."""
import numpy as np
import pytest

from gpu_util import check, dev, host
from oracle import llama_ref as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("B,h,S,d", [
    (1, 1, 65, 64), (2, 3, 97, 128), (1, 5, 128, 64), (1, 2, 129, 128), (3, 3, 161, 64), (1, 2, 511, 128), (1, 2, 640, 64),
    (1, 32, 512, 128),      # the second round that is still dealt
    (4, 24, 170, 64),       # more 32-query blocks than run at one time: 128-query blocks
    (4, 12, 190, 128),
    (4, 24, 520, 64),       # 128-query blocks above 512 keys: the last block of 256 would be nearly empty
    (3, 20, 530, 128),      # blocks of 256 all the same: they run at one time
])
def test_bf16_attention_key_shares(B, h, S, d, layout, causal):
    from enzyme_ad.jax import ops
    rng = np.random.default_rng(S * d + h)

    def put(a):
        if layout == "bshd":
            t, r = dev(a.transpose(0, 2, 1, 3).reshape(B, S, h * d), "bf16")
            return t, r.reshape(B, S, h, d).transpose(0, 2, 1, 3)
        return dev(a, "bf16")

    def get(t):
        a = host(t)
        return a.reshape(B, S, h, d).transpose(0, 2, 1, 3) if layout == "bshd" else a

    (q, qr), (k, kr), (v, vr), (do, dor) = (put(rng.standard_normal((B, h, S, d))) for _ in range(4))
    with ops.Tape() as tape:
        o = ops.attention(q, k, v, h, causal=causal, layout=layout)
    ro, rlse = L.attention_fwd(qr, kr, vr, causal=causal)
    check(get(o), ro, "bf16", "attention out")
    _, lse, _ = ops.attention_raw(q, k, v, h, 1.0 / np.sqrt(d), causal, layout)
    check(host(lse).reshape(rlse.shape), rlse, "f32", "log-sum-exp")
    for got, want, name in zip(tape.backward([o], [do], [q, k, v]), L.attention_bwd(qr, kr, vr, dor, causal=causal), "qkv"):
        check(get(got), want, "bf16", "attention d" + name)
