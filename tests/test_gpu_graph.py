"""HIP-graph capture of the reference's step (forward + reverse mode): every replay is checked
against the eager result on fresh inputs, with eager work and synchronisations between
replays."""
import numpy as np
import pytest
import torch

from oracle import llama_ref as L
from gpu_util import dev, host

pytestmark = pytest.mark.gpu

CFG = {"dim": 288, "hidden_dim": 768, "n_layers": 6, "n_heads": 6, "n_kv_heads": 6, "vocab_size": 32000, "seq_len": 256}


def _inputs(seed, pos):
    rng = np.random.Generator(np.random.PCG64(seed))
    w = L.make_weights(CFG, seed, std=0.05, embedding=False, norm_gain="uniform")
    wd = {k: dev(a, "f32")[0] for k, a in w.items()}
    x, dy = (dev(rng.standard_normal(CFG["dim"]), "f32")[0] for _ in range(2))
    kc, vc = (dev(rng.standard_normal((CFG["n_layers"], pos, CFG["dim"])), "f32")[0] for _ in range(2))
    return x, wd, kc, vc, dy


def _flat(out):
    y, (gx, gw, gkc, gvc) = out
    return [y, gx, gkc, gvc] + [gw[k] for k in sorted(gw)]


def test_captured_step_replays_match_eager():
    from enzyme_ad.jax import llama, vjp
    from enzyme_ad.jax.graph import capture

    def step(x, w, kc, vc, dy):
        y, f_vjp = vjp(lambda a, b, c, d: llama.forward_step(a, CFG, b, c, d), x, w, kc, vc)
        return y, f_vjp(dy)

    g = capture(step, *_inputs(1, 5))
    for seed in (2, 3, 4, 5):
        args = _inputs(seed, 5)
        eager = [t.clone() for t in _flat(step(*args))]
        torch.cuda.synchronize()
        junk = torch.randn(1 << 20, device="cuda").sin_()            # unrelated eager work between replays
        got = _flat(g(*args))
        torch.cuda.synchronize()
        for a, b in zip(got, eager):
            assert torch.equal(a, b)
        del junk
    assert g.replays == 4
    with pytest.raises(ValueError):
        g(*_inputs(6, 6))                                            # another cache length: shapes are fixed at capture


def test_captured_text_step_replays_match_eager():
    """The same through the StableHLO text front end (parsed-module constants are uploaded in
    the eager run before capture)."""
    from enzyme_ad.jax import hlo_call, vjp
    from enzyme_ad.jax.graph import capture
    from enzyme_ad.jax.llama_text import WEIGHT_ORDER, llama_step_text

    cfg = dict(CFG, n_layers=2)
    text, order = llama_step_text(cfg, 5)

    def step(dy, *args):
        y, f_vjp = vjp(lambda *a: hlo_call(*a, source=text)[0], *args)
        return (y,) + tuple(f_vjp(dy))

    def inputs(seed):
        x, wd, kc, vc, dy = _inputs(seed, 5)
        return [dy, x] + [wd[k][:2].contiguous() for k in WEIGHT_ORDER[:-1]] + [wd["rms_final_weight"], kc[:2].contiguous(), vc[:2].contiguous()]

    g = capture(step, *inputs(1))
    for seed in (7, 8, 9):
        args = inputs(seed)
        eager = [t.clone() for t in step(*args)]
        torch.cuda.synchronize()
        got = g(*args)
        torch.cuda.synchronize()
        for a, b in zip(got, eager):
            assert torch.equal(a, b)


def test_copy_many():
    """Arrays of no bytes, of fewer than a piece, off 16-byte boundaries on either side, of several blocks and of one block exactly,
    more arrays than one launch takes; nothing beyond an array is written."""
    from enzyme_ad.jax import _native
    import ctypes
    sizes = [0, 1, 15, 16, 17, 4095, 65535, 65536, 65537, 200003] + [33] * 60
    shifts = [(0, 0), (0, 1), (3, 0), (5, 5)]
    src, dst, want = [], [], []
    for i, n in enumerate(sizes):
        a, b = shifts[i % 4]
        room = torch.randint(0, 255, (n + 32,), dtype=torch.uint8, device="cuda")
        out = torch.full((n + 32,), 7, dtype=torch.uint8, device="cuda")
        ref = out.clone()
        ref[b:b + n] = room[a:a + n]
        src.append(room[a:])
        dst.append((out, b))
        want.append(ref)
    table = ctypes.c_void_p * len(sizes)
    _native.check(_native.lib().emi_copy_many(torch.cuda.current_stream().cuda_stream, len(sizes), table(*[s.data_ptr() for s in src]),
                                              table(*[o.data_ptr() + b for o, b in dst]), (ctypes.c_int64 * len(sizes))(*sizes)))
    assert all(torch.equal(o, w) for (o, _), w in zip(dst, want))
    assert _native.lib().emi_copy_many(None, 1, table(), table(), (ctypes.c_int64 * 1)(4)) == 3          # null array
    assert _native.lib().emi_copy_many(None, 1, table(*[16] * len(sizes)), table(*[16] * len(sizes)), (ctypes.c_int64 * 1)(-1)) == 3


def test_captured_takes_arguments_of_any_layout_and_its_own_buffers():
    """Strided, host and misaligned arguments; an output that is one of the graph's argument buffers, passed back as another one,
    is read before it is written, in the order of the arguments."""
    from enzyme_ad.jax import ops
    from enzyme_ad.jax.graph import capture
    a, b = (torch.randn(300, 8, device="cuda") for _ in range(2))
    g = capture(lambda a, b: (ops.add(a, b), a, b), a, b)
    strided = torch.randn(8, 300, device="cuda").t()
    off = torch.randn(300 * 8 + 1, device="cuda")[1:].view(300, 8)
    for x, y in ((strided, off), (torch.randn(300, 8), b), (a, a), (off, strided)):
        assert torch.equal(g(x, y)[0], x.cuda() + y.cuda())
    _, ga, gb = g(a, b)
    assert torch.equal(g(b, ga)[0], b + b)                # b into the first buffer, which is then the second argument
    _, ga, gb = g(a, b)
    assert torch.equal(g(gb, b)[0], b + b) and torch.equal(g(ga, gb)[0], b + b)


def test_copy_many_of_words():
    """Arrays whose two addresses are whole numbers of 4, of 2 and of no more than one byte: less than a word, less than a batch of a
    block's loads, one batch and a little more, one block and a little more."""
    from enzyme_ad.jax import _native
    import ctypes
    cases = [(n, a, b) for a, b in ((4, 0), (0, 12), (4, 8), (2, 0), (6, 12), (1, 3)) for n in (1, 5, 1023, 4095, 16384, 16391, 65536, 65543, 150001)]
    room = torch.randint(0, 255, (200000,), dtype=torch.uint8, device="cuda")
    out = [torch.full((n + 32,), 7, dtype=torch.uint8, device="cuda") for n, _, _ in cases]
    table = ctypes.c_void_p * len(cases)
    _native.check(_native.lib().emi_copy_many(torch.cuda.current_stream().cuda_stream, len(cases), table(*[room.data_ptr() + a for _, a, _ in cases]),
                                              table(*[o.data_ptr() + b for o, (_, _, b) in zip(out, cases)]), (ctypes.c_int64 * len(cases))(*[c[0] for c in cases])))
    for o, (n, a, b) in zip(out, cases):
        assert torch.equal(o[b:b + n], room[a:a + n]) and bool((o[:b] == 7).all()) and bool((o[b + n:] == 7).all()), (n, a, b)


def test_captured_takes_three_arguments_of_any_layout_and_its_own_buffers():
    """As above with arguments enough for the one launch: whole arrays beside strided, host and misaligned ones, and outputs that are
    the graph's argument buffers."""
    from enzyme_ad.jax import ops
    from enzyme_ad.jax.graph import capture
    a, b, c = (torch.randn(300, 8, device="cuda") for _ in range(3))
    g = capture(lambda a, b, c: (ops.add(ops.add(a, b), c), a, b, c), a, b, c)
    strided = torch.randn(8, 300, device="cuda").t()
    off = torch.randn(300 * 8 + 1, device="cuda")[1:].view(300, 8)
    for x, y, z in ((a, b, c), (strided, off, b), (torch.randn(300, 8), b, off), (a, a, a), (off, strided, a)):
        assert torch.equal(g(x, y, z)[0], (x.cuda() + y.cuda()) + z.cuda())
    _, ga, gb, gc = g(a, b, c)
    assert torch.equal(g(b, ga, c)[0], (b + b) + c)       # b into the first buffer, which is then the second argument
    _, ga, gb, gc = g(a, b, c)
    assert torch.equal(g(gc, a, gb)[0], (c + a) + a)      # (gb is read after a has gone into it)
