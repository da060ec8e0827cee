"""Decoder layers as one operator (ops.llama_layers): the value and every cotangent against the oracle's layers where its
launches change - one layer and several, weight gradients grouped over the layers or not, weights read in place and turned,
ragged token counts - from Python and from a program's text; and the operators it stands for, under forward mode."""
import numpy as np
import pytest
import torch

from oracle import llama_ref as L
from gpu_util import dev, check, rel_err, host

pytestmark = pytest.mark.gpu


def _inputs(dt, dim, hidden, layers, heads, batch, seq):
    cfg = dict(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=heads, n_kv_heads=heads, vocab_size=8, seq_len=seq)
    rng = np.random.Generator(np.random.PCG64(dim + seq))
    w = L.make_weights(cfg, dim + seq, std=1.0 / np.sqrt(dim), embedding=False, norm_gain="uniform")
    wd, wr = {}, {}
    for k, a in w.items():
        if k not in ("wcls", "rms_final_weight"):
            wd[k], wr[k] = dev(a, dt)
    x, xr = dev(rng.standard_normal((batch, seq, dim)), dt)
    dy, dyr = dev(rng.standard_normal((batch, seq, dim)), dt)
    return cfg, wd, wr, x, xr, dy, dyr


def _reference(xr, wr, dyr, layers, heads):
    caches, h = [], xr
    for i in range(layers):
        h, cache = L.layer_fwd(h, L._layer_weights(wr, i), heads)
        caches.append(cache)
    d, grads = dyr, {k: np.zeros(v.shape) for k, v in wr.items()}
    for i in reversed(range(layers)):
        d, g = L.layer_bwd(d, L._layer_weights(wr, i), caches[i], heads)
        for k in grads:
            grads[k][i] = g[k]
    return h, d, grads


# products split over K whose planes the next RMSNorm (or, in reverse, its adjoint) adds up; tests/test_host_boundary.py holds them to that
SPLIT_SIZES = [
    ("bf16", 1024, 2816, 2, 8, 1, 257, None),     # w2: a wavefront to a row
    ("bf16", 2048, 5632, 2, 16, 2, 65, None),     # w2: 256 threads to a row
    ("bf16", 4096, 264, 1, 32, 1, 77, None),      # wo, two pieces a thread
    ("bf16", 2048, 8200, 2, 16, 2, 515, None),    # w2 in 256-tiles
    ("f32", 1032, 2824, 2, 43, 1, 33, None),      # wo and w2, 256 threads to a row of 129 pairs of pieces
]


@pytest.mark.parametrize("dt,dim,hidden,layers,heads,batch,seq,pending", SPLIT_SIZES + [
    ("f32", 32, 24, 51, 2, 1, 9, None),       # more norms in a group than one launch sums
    ("f32", 64, 72, 5, 2, 1, 33, 2),          # groups of two: the second one's first dy lies in the last slot of the first
    ("f32", 288, 768, 3, 6, 1, 9, None),
    ("f32", 128, 264, 2, 2, 3, 77, 1),        # one layer's cotangents at a time
    ("bf16", 128, 256, 3, 2, 2, 131, None),   # all layers in one group
    ("bf16", 256, 264, 1, 2, 1, 640, None),
    ("bf16", 128, 136, 2, 1, 4, 801, None),   # more tokens than are worth reading a weight in place for
])
def test_llama_layers_match_oracle(dt, dim, hidden, layers, heads, batch, seq, pending, monkeypatch):
    from enzyme_ad.jax import llama, ops, vjp
    cfg, wd, wr, x, xr, dy, dyr = _inputs(dt, dim, hidden, layers, heads, batch, seq)
    if pending is not None:
        layer_bytes = ops.N.lib().emi_llama_layers_cotangent_bytes(batch, seq, dim, hidden, heads, ops._code(x))
        monkeypatch.setattr(ops, "_PENDING_DW_BYTES", pending * layer_bytes)
    table = ops.rope_table(seq, dim // heads, device=x.device)
    names = llama.LAYER_KEYS
    assert ops.llama_layers_apply(x, [wd[k] for k in names], heads)

    def f(x, w):
        return ops.add(ops.llama_layers(x, [w[k] for k in names], heads, table), x)      # a second cotangent of x

    y, pull = vjp(f, x, wd)
    gx, gw = pull(dy)
    ry, rdx, rgw = _reference(xr, wr, dyr, layers, heads)
    check(y, ry + xr, dt, "y")
    check(gx, rdx + dyr, dt, "dx")
    for k in names:
        check(gw[k], rgw[k], dt, "d" + k)
    assert torch.equal(f(x, wd), y)           # without a tape one buffer serves all layers: the same bits


def test_llama_layers_of_a_text():
    """A program's text runs its layers as this operator and gives the bits of the model built in Python; under forward
    mode it runs the operators the layers were made of."""
    from enzyme_ad.jax import hlo_call, jvp, llama, stablehlo, vjp
    from enzyme_ad.jax.llama_text import MODEL_ORDER, llama_model_text
    cfg, wd, wr, x, xr, dy, _ = _inputs("f32", 96, 160, 2, 2, 1, 33)
    cfg = dict(cfg, vocab_size=64)
    rng = np.random.Generator(np.random.PCG64(5))
    text, _ = llama_model_text(cfg, 1, 33, "f32", None)
    w = dict(wd, rms_final_weight=dev(rng.uniform(0.5, 1.5, 96), "f32")[0], wcls=dev(rng.standard_normal((64, 96)) * 0.1, "f32")[0],
             token_embedding_table=dev(rng.standard_normal((64, 96)), "f32")[0])
    tokens = torch.from_numpy(rng.integers(0, 64, (1, 33)).astype(np.int32)).cuda()
    exe = stablehlo.compile_text(text)
    assert [o.name for o in exe.funcs["main"].layer_ops].count("emi.llama_layers") == 1
    args = [w[k] for k in MODEL_ORDER]

    def fn(*a):
        return hlo_call(tokens, *a, source=text)[0]

    got, pull = vjp(fn, *args)
    c = dev(rng.standard_normal(tuple(got.shape)), "f32")[0]
    ref, ref_pull = vjp(lambda w: llama.forward(tokens, cfg, w, logits=True), w)
    assert rel_err(host(got), host(ref).reshape(got.shape)) < 1e-5      # the angles come from the text's constants
    grads, (ref_grads,) = pull(c), ref_pull(c.reshape(ref.shape))
    for k, g in zip(MODEL_ORDER, grads):
        assert rel_err(host(g), host(ref_grads[k])) < 1e-4, k
    tangents = [dev(rng.standard_normal(tuple(a.shape)) * 0.1, "f32")[0] for a in args]
    value, tangent = jvp(fn, tuple(args), tuple(tangents))
    assert rel_err(host(value), host(got)) < 1e-5
    # <c, J t> = <J^T c, t>
    a = float((c.double() * tangent.double()).sum())
    b = sum(float((g.double() * t.double()).sum()) for g, t in zip(grads, tangents))
    assert abs(a - b) <= 1e-4 * max(abs(a), float(c.double().norm() * tangent.double().norm()) * 1e-2)


def test_a_stack_is_no_layer_and_a_layer_no_stack():
    """`llama.layer` takes one layer's weights and `llama.forward` stacks of them; neither takes the other's."""
    from enzyme_ad.jax import llama
    cfg, wd, _, x, _, _, _ = _inputs("f32", 64, 72, 2, 2, 1, 33)
    with pytest.raises(ValueError):
        llama.layer(x, wd, 2)
    final = dict(rms_final_weight=torch.ones(64, device="cuda"))
    with pytest.raises(ValueError):
        llama.forward(x, dict(cfg, n_layers=72), dict({k: w[0] for k, w in wd.items()}, **final))
    assert torch.equal(llama.forward(x, dict(cfg, n_layers=0), final), llama.ops.rmsnorm(x, final["rms_final_weight"]))


def test_llama_layers_refuse_what_they_do_not_serve():
    """Operands that the call would read out of range or mistake for something else raise on the host."""
    from enzyme_ad.jax import llama, ops
    _, wd, _, x, _, _, _ = _inputs("f32", 64, 72, 2, 2, 1, 33)
    w, table = [wd[k] for k in llama.LAYER_KEYS], ops.rope_table(33, 32, device=x.device)
    ops.llama_layers(x, w, 2, table)
    for bad in (ops.rope_table(32, 32, device=x.device), ops.rope_table(33, 16, device=x.device), table.double(), table.bfloat16(), table.reshape(33, 32)):
        with pytest.raises(ValueError):
            ops.llama_layers(x, w, 2, bad)
    for i, t in ((6, w[6][:, :-8].contiguous()), (7, w[6]), (1, w[1][:1].contiguous()), (0, w[0][:, :60].contiguous())):
        with pytest.raises(ValueError):
            ops.llama_layers(x, w[:i] + [t] + w[i + 1:], 2, table)
    with pytest.raises(ValueError):
        ops.llama_layers(x, w[:8], 2, table)
    with pytest.raises(TypeError):
        ops.llama_layers(x.bfloat16(), w, 2, table)
    with ops.Forward(), pytest.raises(ValueError):
        ops.llama_layers(x, w, 2, table)


@pytest.mark.parametrize("dt,dim,hidden,layers,heads,batch,seq", [
    ("f32", 64, 72, 5, 2, 1, 33),             # tiles of 32: two products to a result in one launch; all layers in one set of buffers
    ("f32", 288, 768, 2, 6, 3, 100),
    ("f32", 512, 1408, 1, 8, 2, 701),         # on the bf16 instructions: a launch to a result, and a pass to turn q and k
    ("f32", 64, 304, 3, 2, 2, 45),            # a hidden layer longer than q, k, v and the attention together
    ("bf16", 128, 136, 3, 2, 2, 131),
    ("bf16", 64, 520, 2, 1, 1, 70),
    ("bf16", 768, 2048, 1, 12, 1, 777),
    ("bf16", 2048, 1024, 1, 16, 2, 512),      # wide enough for two products one after the other
])
def test_llama_layers_forward_mode(dt, dim, hidden, layers, heads, batch, seq):
    """Values and tangents of the layers as one operator against the oracle; the values are those without tangents, and a
    missing tangent takes the operators one by one to the same result as a zero one."""
    from enzyme_ad.jax import jvp, llama, ops
    cfg, wd, wr, x, xr, _, _ = _inputs(dt, dim, hidden, layers, heads, batch, seq)
    rng = np.random.Generator(np.random.PCG64(3))
    twd, twr = {}, {}
    for k in wd:
        twd[k], twr[k] = dev(rng.standard_normal(wr[k].shape) / np.sqrt(dim), dt)
    tx, txr = dev(rng.standard_normal(xr.shape), dt)
    names, table = list(llama.LAYER_KEYS), ops.rope_table(seq, dim // heads, device=x.device)

    def fn(x, w):
        return ops.llama_layers(x, [w[k] for k in names], heads, table)

    y, ty = jvp(fn, (x, wd), (tx, twd))
    h, t = xr, txr
    for i in range(layers):
        h, t = L.layer_jvp(h, L._layer_weights(wr, i), t, L._layer_weights(twr, i), heads)
    check(y, h, dt, "y")
    check(ty, t, dt, "ty")
    assert torch.equal(y, fn(x, wd))
    if layers == 1:
        one, zero = {k: w[0] for k, w in wd.items()}, dict({k: w[0] for k, w in twd.items()}, wq=torch.zeros_like(wd["wq"][0]))
        a = jvp(lambda x, w: llama.layer(x, w, heads), (x, one), (tx, zero))
        b = jvp(lambda x, w: llama.layer(x, w, heads), (x, one), (tx, dict(zero, wq=None)))
        tol = 1e-5 if dt == "f32" else 2e-2
        assert rel_err(host(a[0]), host(b[0])) < tol and rel_err(host(a[1]), host(b[1])) < tol


def test_llama_layer_tangent_in_the_operators_order():
    """Of so many tokens that each product is a launch, a tangent's two products run in the operators' order, each result's second
    behind its first: the operators' bits, where the values are (no rotation and no gate, which the layer's products apply)."""
    from enzyme_ad.jax import jvp, llama, ops
    dim, heads = 2048, 16
    _, wd, _, x, _, _, _ = _inputs("bf16", dim, 2304, 1, heads, 6, 1024)
    rng = np.random.Generator(np.random.PCG64(4))
    w = {k: torch.zeros_like(t[0]) if k in ("wq", "wk", "w1") else t[0].contiguous() for k, t in wd.items()}
    tw = {k: dev(rng.standard_normal(tuple(t.shape)) / np.sqrt(dim), "bf16")[0] for k, t in w.items()}
    tx = dev(rng.standard_normal(tuple(x.shape)), "bf16")[0]

    def run():
        return jvp(lambda x, w: llama.layer(x, w, heads), (x, w), (tx, tw))

    y, ty = run()
    with ops.Tape():                                     # under a tape the operators run one by one
        want, twant = run()
    assert torch.equal(y, want) and torch.equal(ty, twant)


def test_llama_layers_jvp_checks_its_arguments():
    """A short workspace, a null tangent, weight or operand, and shapes and types that are not served are errors before any launch."""
    import ctypes
    from enzyme_ad.jax import llama, ops
    from enzyme_ad.jax import _native as N
    lib, B, S, D, H, heads = N.lib(), 1, 33, 64, 72, 2
    _, wd, _, x, _, _, _ = _inputs("f32", D, H, 2, heads, B, S)
    w, table = [wd[k] for k in llama.LAYER_KEYS], ops.rope_table(S, D // heads, device=x.device)
    y, ty = torch.full_like(x, 7.0), torch.full_like(x, 7.0)
    need = lib.emi_llama_layers_jvp_workspace_bytes(B, S, D, H, heads, 11)
    ws = torch.empty(need, dtype=torch.uint8, device=x.device)
    ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*[None if t is None else t.data_ptr() for t in ts])

    def call(weights=w, tangents=w, tx=x, nws=need, dims=(2, B, S, D, H, heads), dt=11):
        return lib.emi_llama_layers_jvp(torch.cuda.current_stream().cuda_stream, ptrs(weights), ptrs(tangents), x.data_ptr(),
                                        None if tx is None else tx.data_ptr(), table.data_ptr(), y.data_ptr(), ty.data_ptr(), ws.data_ptr(), nws,
                                        *dims, 1e-5, 0.2, dt)

    for i in range(9):
        assert call(tangents=w[:i] + [None] + w[i + 1:]) == 3 and call(weights=w[:i] + [None] + w[i + 1:]) == 3
    assert call(tx=None) == 3 and call(nws=need - 1) == 3 and call(nws=0) == 3 and call(dt=7) == 3
    for dims in ((0, B, S, D, H, heads), (2, 0, S, D, H, heads), (2, B, S, D, H, 3), (2, B, S, 62, H, heads), (2, B, S, D, 70, heads)):
        assert call(dims=dims) == 3 and (dims[0] == 0 or lib.emi_llama_layers_jvp_workspace_bytes(*dims[1:], 11) == 0), dims
    assert bool((y == 7.0).all()) and bool((ty == 7.0).all())
    assert call() == 0 and bool((y != 7.0).any()) and bool((ty != 7.0).any())
