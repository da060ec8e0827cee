"""The adjoint of rope(rmsnorm(x)), whose rotation runs inside the RMSNorm adjoint where the normalised array has no other
reader, at the edges of its rows (one piece, ragged pieces of a wavefront and of a block, the longest row), and where it does
not apply: the array is read twice, asked for itself, or its heads are no whole pieces.  Against the two adjoints one by one,
whose roundings it keeps."""
import numpy as np
import pytest
import torch

from gpu_util import dev

pytestmark = pytest.mark.gpu


def _one_by_one(x, gamma, dy, heads):
    from enzyme_ad.jax import ops
    with ops.Tape() as tape:
        y = ops.rmsnorm(x, gamma)
    with ops.Tape() as rot:
        z = ops.rope(y, heads)
    return z, tape.backward([y], rot.backward([z], [dy], [y]), [x, gamma])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("B,S,heads,d", [(1, 1, 1, 8), (2, 3, 3, 8), (3, 5, 6, 48), (2, 700, 12, 64), (1, 33, 65, 16), (2, 9, 32, 128), (1, 4, 64, 128)])
def test_rotation_inside_the_norm_adjoint(B, S, heads, d, dtype, monkeypatch):
    from enzyme_ad.jax import _native, ops
    rng = np.random.default_rng(B + S + heads + d)
    D = heads * d
    x, dy = (dev(rng.standard_normal((B, S, D)), dtype)[0] for _ in range(2))
    gamma = dev(1 + 0.25 * rng.standard_normal(D), dtype)[0]
    rz, (rdx, rdg) = _one_by_one(x, gamma, dy, heads)
    calls = []
    real = _native.lib().emi_rmsnorm_bwd_rope
    monkeypatch.setattr(_native.lib(), "emi_rmsnorm_bwd_rope", lambda *a: calls.append(1) or real(*a))
    with ops.Tape() as tape:
        z = ops.rope(ops.rmsnorm(x, gamma), heads)
    dx, dg = tape.backward([z], [dy], [x, gamma])
    assert calls and torch.equal(z, rz)
    # the same operations on the same values: at most a contraction of the compiler's apart
    unit = 2.0 ** -7 if dtype == "bf16" else 2.0 ** -21
    for a, b in ((dx, rdx), (dg, rdg)):
        a, b = a.double(), b.double()
        assert float((a - b).abs().max()) <= unit * float(b.abs().max())


@pytest.mark.parametrize("why", ["read twice", "asked for", "odd heads", "two rotations"])
def test_rotation_that_stays_a_pass_of_its_own(why, monkeypatch):
    from enzyme_ad.jax import _native, ops
    rng = np.random.default_rng(7)
    heads, d = (4, 6) if why == "odd heads" else (3, 16)
    D = heads * d
    x, dy, dz = (dev(rng.standard_normal((2, 5, D)), "f32")[0] for _ in range(3))
    gamma = dev(1 + 0.25 * rng.standard_normal(D), "f32")[0]
    monkeypatch.setattr(_native.lib(), "emi_rmsnorm_bwd_rope", lambda *a: pytest.fail("fused"))
    with ops.Tape() as tape:
        y = ops.rmsnorm(x, gamma)
        z = ops.rope(y, heads)
        if why == "read twice":
            z = ops.add(z, y)
        if why == "two rotations":
            z = ops.add(z, ops.rope(y, heads))
    wrt = [x, gamma, y] if why == "asked for" else [x, gamma]
    got = tape.backward([z], [dy], wrt)
    with ops.Tape() as rot:
        r = ops.rope(y, heads)
    cy = rot.backward([r], [dy], [y])[0]
    total = {"read twice": cy + dy, "two rotations": cy + cy}.get(why, cy)
    with ops.Tape() as norm:
        y2 = ops.rmsnorm(x, gamma)
    for a, b in zip(got[:2], norm.backward([y2], [total], [x, gamma])):
        assert float((a - b).abs().max()) <= 2.0 ** -20 * float(b.abs().max())
