"""The single-token step as one operator (ops.llama_step): the value and all thirteen cotangents against the oracle's
forward_step / forward_step_vjp at the sizes where its kernels change - rows shorter and longer than a batch of loads, one
and several key blocks per head, one and two 16-byte pieces of a head per lane, one and several bands and column groups of
the adjoint products - and the operators it stands for, which forward mode and odd shapes still take."""
import numpy as np
import pytest
import torch

from oracle import llama_ref as L
from gpu_util import dev, check, rel_err, host

pytestmark = pytest.mark.gpu


def _inputs(dt, dim, hidden, layers, heads, pos, seed):
    cfg = dict(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=heads, vocab_size=8, seq_len=pos + 1)
    rng = np.random.Generator(np.random.PCG64(seed))
    w = L.make_weights(cfg, seed, std=1.0 / np.sqrt(dim), embedding=False, norm_gain="uniform")
    w.pop("wcls", None)
    wd, wr = {}, {}
    for k, a in w.items():
        wd[k], wr[k] = dev(a, dt)
    arrays = [rng.standard_normal(s) for s in ((dim,), (layers, pos, dim), (layers, pos, dim), (dim,))]
    return cfg, wd, wr, [dev(a, dt) for a in arrays]


@pytest.mark.parametrize("dt,dim,hidden,layers,heads,pos", [
    ("f32", 288, 768, 2, 6, 1),           # the reference's own sizes
    ("f32", 288, 768, 2, 6, 255),         # exactly one pass of keys
    ("f32", 288, 768, 1, 6, 256),         # one key more: the token's own row opens a second block
    ("f32", 512, 516, 1, 4, 700),         # two pieces of a head per lane, several key blocks
    ("f32", 516, 36, 2, 3, 40),           # rows just over two batches; short ffn
    ("bf16", 64, 40, 3, 2, 3),
    ("bf16", 1024, 2816, 2, 8, 300),      # head_dim 128
    ("bf16", 1056, 264, 1, 11, 129),      # rows just over two batches
    ("f32", 200, 40, 1, 4, 5),            # head_dim 50: operator by operator
    ("bf16", 2112, 5632, 1, 12, 520),     # head_dim 176: two pieces per lane; two column groups in the adjoint
    ("bf16", 4096, 1024, 1, 32, 1030),
])
def test_llama_step_matches_oracle(dt, dim, hidden, layers, heads, pos):
    from enzyme_ad.jax import llama, ops, vjp
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), (dy, dyr)) = _inputs(dt, dim, hidden, layers, heads, pos, dim + pos)
    applies = ops.llama_step_applies(x, [wd[k] for k in ops.STEP_WEIGHTS], kc, vc, heads)
    assert applies == (dim != 200)
    y, pull = vjp(lambda x, w, k, v: llama.forward_step(x, cfg, w, k, v), x, wd, kc, vc)
    gx, gw, gk, gv = pull(dy)
    ry, rdx, rgw, rdk, rdv = L.forward_step_vjp(xr, cfg, wr, kcr, vcr, dyr)
    check(y, ry, dt, "y")
    check(gx, rdx, dt, "dx")
    check(gk, rdk, dt, "dkey_cache")
    check(gv, rdv, dt, "dvalue_cache")
    for k in wd:
        # dwk is the outer product of one key's cotangent, per head p scale (dO . v - dO . o) q: the two products cancel.
        # Their operands are rounded to 2^-9, so with z = dO . (v - o) in units of |dO| |v - o| / sqrt(head_dim) a head's
        # row is off by about 2^-8 / |z|; twelve or more heads have one at |z| ~ 0.1, i.e. 4e-2
        # (measured here: 2.3e-2, and 4.6e-2 operator by operator).
        check(gw[k], rgw[k], dt, "d" + k, factor=2.0 if k == "wk" and dt == "bf16" else 1.0)


@pytest.mark.parametrize("dt,dim,hidden,heads,pos", [
    ("f32", 272, 520, 4, 70),             # blocks of 8 pieces, the last one cut; two blocks of keys
    ("f32", 16, 131080, 1, 3),            # half a block of pieces; more rows than the bands of at most 4096 take
    ("f32", 528, 1412, 6, 130),           # 16 pieces; bands that do not divide the rows
    ("f32", 1040, 300, 5, 4),             # 32
    ("f32", 2064, 36, 12, 64),            # 64; nine bands' worth of rows in a hidden layer shorter than a band
    ("bf16", 4160, 72, 20, 5),            # 64, and one row lane a wavefront
])
def test_llama_step_adjoint_blocks(dt, dim, hidden, heads, pos):
    """Block widths and bands of the reverse products, whose sums the next product adds up for its own rows."""
    from enzyme_ad.jax import llama, vjp
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), (dy, dyr)) = _inputs(dt, dim, hidden, 2 if dim < 1000 else 1, heads, pos, dim + pos)
    y, pull = vjp(lambda x, w, k, v: llama.forward_step(x, cfg, w, k, v), x, wd, kc, vc)
    gx, gw, gk, gv = pull(dy)
    ry, rdx, rgw, rdk, rdv = L.forward_step_vjp(xr, cfg, wr, kcr, vcr, dyr)
    for got, want, name in ((y, ry, "y"), (gx, rdx, "dx"), (gk, rdk, "dkey_cache"), (gv, rdv, "dvalue_cache")):
        check(got, want, dt, name)
    for k in wd:
        check(gw[k], rgw[k], dt, "d" + k, factor=2.0 if k == "wk" and dt == "bf16" else 1.0)      # see above


@pytest.mark.parametrize("dt,dim,heads,pos", [
    ("f32", 96, 2, 222), ("f32", 96, 2, 223),         # 224 keys: the first count in blocks of 64, here four of them
    ("f32", 288, 6, 511), ("bf16", 288, 6, 512),      # eight blocks are one round of loads; the ninth holds the token's own key alone
    ("f32", 256, 4, 1023), ("f32", 256, 4, 1024),     # sixteen are two rounds, with one more a launch adds them up
    ("f32", 384, 3, 94), ("f32", 384, 3, 95),         # two pieces of a head a lane: from 96 keys
    ("f32", 1040, 5, 127), ("bf16", 2064, 12, 300),   # more pieces of the vector than threads
    ("f32", 3120, 39, 230),                           # four rounds, the last with 12 of 256 threads
])
def test_llama_step_adds_up_blocks_of_keys(dt, dim, heads, pos):
    """The product with wo adds up the attention's key blocks: one and several rounds of shares, and the edges of the rule."""
    from enzyme_ad.jax import llama
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), _) = _inputs(dt, dim, 40, 1, heads, pos, dim + pos)
    check(llama.forward_step(x, cfg, wd, kc, vc), L.forward_step(xr, cfg, wr, kcr, vcr), dt, "y")


def test_llama_step_accumulates_and_repeats():
    """The step's cotangents add to what other uses of its operands contribute, and are the same bits run to run."""
    from enzyme_ad.jax import llama, ops, vjp
    cfg, wd, wr, ((x, _), (kc, _), (vc, _), (dy, _)) = _inputs("f32", 96, 64, 2, 2, 5, 3)

    def f(x, w, k, v):
        return ops.add(llama.forward_step(x, cfg, w, k, v), x)

    y, pull = vjp(f, x, wd, kc, vc)
    a, b = pull(dy), pull(dy)
    _, plain = vjp(lambda x, w, k, v: llama.forward_step(x, cfg, w, k, v), x, wd, kc, vc)
    c = plain(dy)
    assert torch.equal(a[0], b[0]) and all(torch.equal(a[1][k], b[1][k]) for k in wd)
    assert rel_err(host(a[0]), host(c[0]) + host(dy)) < 1e-6


def _own_key_out_of_reach(wd, wr, xr, pos, heads):
    """One infinite weight at the start of a row of wk that gives the token's own key a score of -infinity in one head."""
    dim = xr.shape[0]
    d = dim // heads
    cos, sin = (t[0] for t in L.rope_angles(1, d, pos0=pos))
    xb = L.rmsnorm(xr, wr["rms_att_weight"][0])
    q = (wr["wq"][0] @ xb).reshape(heads, d // 2, 2)
    rq = np.stack([cos * q[..., 0] - sin * q[..., 1], sin * q[..., 0] + cos * q[..., 1]], -1)
    # a key row whose element 2 i is infinite is turned into (cos, sin) times that: one sign in both products with rq
    side = np.sign(rq * np.stack([cos, sin], -1))
    h, i = np.argwhere((side[..., 0] == side[..., 1]) & (np.abs(rq).min(-1) > 0.1))[0]
    wr["wk"][0, h * d + 2 * i, 0] = -side[h, i, 0] * np.sign(xb[0]) * np.inf
    wd["wk"][0, h * d + 2 * i, 0] = float(wr["wk"][0, h * d + 2 * i, 0])


@pytest.mark.parametrize("dt,dim,heads", [("f32", 288, 6), ("f32", 516, 3), ("bf16", 768, 12)])
def test_llama_step_drops_what_lies_past_a_row(dt, dim, heads):
    """Rows that are no whole number of batches of loads: an infinite weight at a row's start counts once, where it stands.
    The key it makes infinite has a weight of exactly 0, so everything stays finite."""
    from enzyme_ad.jax import llama
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), _) = _inputs(dt, dim, 64, 1, heads, 5, 7)
    _own_key_out_of_reach(wd, wr, xr, 5, heads)
    check(llama.forward_step(x, cfg, wd, kc, vc), L.forward_step(xr, cfg, wr, kcr, vcr), dt, "y")


def test_llama_step_whose_last_block_holds_no_finite_score():
    """Two pieces of a head per lane, and the token's own key alone in the last block of keys with a score of -infinity."""
    from enzyme_ad.jax import llama
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), _) = _inputs("f32", 384, 64, 1, 3, 256, 7)
    _own_key_out_of_reach(wd, wr, xr, 256, 3)
    check(llama.forward_step(x, cfg, wd, kc, vc), L.forward_step(xr, cfg, wr, kcr, vcr), "f32", "y")


@pytest.mark.parametrize("n_layers", [0, 1, 2, 5])
def test_llama_step_runs_as_many_layers_as_the_config_says(n_layers):
    """Fewer layers than the stacks hold leave the rest alone; more go round them (`ops.select`), with and without a tape."""
    from enzyme_ad.jax import llama, vjp
    cfg, wd, wr, ((x, xr), (kc, kcr), (vc, vcr), (dy, dyr)) = _inputs("f32", 96, 64, 3, 2, 5, 3)
    cfg = dict(cfg, n_layers=n_layers)
    turn = [i % 3 for i in range(n_layers)]
    wt = {k: a if k == "rms_final_weight" else a[turn] for k, a in wr.items()}
    y, pull = vjp(lambda x, w, k, v: llama.forward_step(x, cfg, w, k, v), x, wd, kc, vc)
    check(llama.forward_step(x, cfg, wd, kc, vc), L.forward_step(xr, cfg, wt, kcr[turn], vcr[turn]), "f32", "y")
    if n_layers in (1, 2):
        gw = pull(dy)[1]
        ref = L.forward_step_vjp(xr, cfg, wt, kcr[turn], vcr[turn], dyr)[2]
        assert torch.equal(y, llama.forward_step(x, cfg, wd, kc, vc))
        for k in ("wq", "w2"):
            check(gw[k][:n_layers], ref[k], "f32", "d" + k)
            assert not gw[k][n_layers:].any()


def test_llama_step_refuses_what_it_does_not_serve():
    """Operands that the call would read out of range or mistake for something else raise on the host."""
    from enzyme_ad.jax import ops
    _, wd, _, ((x, _), (kc, _), (vc, _), _) = _inputs("f32", 96, 64, 2, 2, 5, 3)
    w, table = [wd[k] for k in ops.STEP_WEIGHTS], ops.rope_table(1, 48, pos0=5, device=x.device)
    ops.llama_step(x, w, kc, vc, 2, table)
    for bad in (table.double(), table.bfloat16(), table[:, :7].contiguous(), table[:, :0], table.reshape(-1, 1)):
        with pytest.raises(ValueError):
            ops.llama_step(x, w, kc, vc, 2, bad)
    for i, t in ((6, w[6][:, :-4].contiguous()), (7, w[6]), (1, w[1][:1].contiguous()), (9, w[9][:95].contiguous())):
        with pytest.raises(ValueError):
            ops.llama_step(x, w[:i] + [t] + w[i + 1:], kc, vc, 2, table)
    with pytest.raises(ValueError):
        ops.llama_step(x, w[:9], kc, vc, 2, table)
    with pytest.raises(ValueError):
        ops.llama_step(x, w, kc, vc[:, :-1].contiguous(), 2, table)
    with pytest.raises(TypeError):
        ops.llama_step(x.bfloat16(), w, kc, vc, 2, table)
    with ops.Forward(), pytest.raises(ValueError):
        ops.llama_step(x, w, kc, vc, 2, table)
