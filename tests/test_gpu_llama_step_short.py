"""The single-token step over a short cache, whose attention is worked out inside the product with wo: one and two rounds of
keys and of heads, the first cache and head count beyond them, heads that fill a row of 16 lanes, rows that are no whole
batch of loads, and keys without a finite score.  The reverse turns dq and dk back where a head's only block leaves them."""
import numpy as np
import pytest
import torch

from oracle import llama_ref as L
from gpu_util import check
from test_gpu_llama_step import _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,dim,heads,pos", [
    ("f32", 288, 6, 7), ("f32", 288, 6, 8), ("f32", 288, 6, 15), ("f32", 288, 6, 16),     # 8, 9, 16 | 17 keys
    ("f32", 64, 16, 15), ("f32", 68, 17, 7), ("f32", 68, 17, 8),                          # 16, 17 heads | 17 and 9 keys
    ("f32", 1024, 16, 3),                                                                 # head_dim 64: all 16 lanes
    ("f32", 516, 3, 2), ("bf16", 352, 2, 40),                                             # two pieces a lane: the general kernels
    ("bf16", 1024, 8, 11), ("bf16", 264, 33, 1), ("bf16", 256, 32, 7), ("bf16", 1056, 12, 9),
])
def test_short_cache_matches_oracle(dt, dim, heads, pos):
    from enzyme_ad.jax import llama, vjp
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), (dy, dyr)) = _inputs(dt, dim, 40, 2, heads, pos, dim + pos)
    y, pull = vjp(lambda x, w, k, v: llama.forward_step(x, cfg, w, k, v), x, wd, kc, vc)
    gx, _, gk, gv = pull(dy)                              # the reverse reads att and lse as this kernel left them
    ry, rdx, _, rdk, rdv = L.forward_step_vjp(xr, cfg, wr, kcr, vcr, dyr)
    check(y, ry, dt, "y")
    check(gx, rdx, dt, "dx")
    check(gk, rdk, dt, "dkey_cache")
    check(gv, rdv, dt, "dvalue_cache")


@pytest.mark.parametrize("dt,dim,heads", [("f32", 288, 6), ("bf16", 768, 12)])
def test_masked_keys_are_dropped(dt, dim, heads):
    """Keys whose scores are all -infinity weigh nothing: the whole first round of keys, and one of the second."""
    from enzyme_ad.jax import llama
    masked = [0, 1, 2, 3, 4, 5, 6, 7, 11]
    cfg, wd, _, ((x, _), (kc, _), (vc, _), _) = _inputs(dt, dim, 40, 1, heads, 13, 5)
    kc[0, masked] = -torch.sign(_query(cfg, wd, x, 13)) * torch.finfo(kc.dtype).max
    y = llama.forward_step(x, cfg, wd, kc, vc)
    vc[0, masked] = 1.0                                   # their values do not matter
    assert torch.isfinite(y).all()
    assert torch.equal(y, llama.forward_step(x, cfg, wd, kc, vc))


def _query(cfg, wd, x, pos):
    """The step's rotated query, in float64 on the host; only its signs are used."""
    dim, d = x.shape[0], x.shape[0] // cfg["n_heads"]
    h = x.double().cpu().numpy()
    n = wd["rms_att_weight"][0].double().cpu().numpy() * h / np.sqrt(np.mean(h * h) + 1e-5)
    q = wd["wq"][0].double().cpu().numpy() @ n
    cos, sin = (t[0] for t in L.rope_angles(1, d, pos0=pos))
    q = q.reshape(cfg["n_heads"], d // 2, 2)
    r = np.stack([q[..., 0] * cos - q[..., 1] * sin, q[..., 1] * cos + q[..., 0] * sin], -1)
    return torch.from_numpy(r.reshape(dim)).to(x.device, x.dtype)
