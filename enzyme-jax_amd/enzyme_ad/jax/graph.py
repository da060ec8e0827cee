"""HIP-graph capture of a whole program of operator calls.

The reference compiles a decorated function once (`jax.jit`) and replays the executable; its
own benchmark case (test/llama.py: one token, dim 288) is a few hundred small kernels, so on a
GPU the step is bound by launch and host overhead, not by the kernels.  Here the counterpart of
the compiled executable is a captured HIP graph: `capture(fn, *example_args)` runs `fn` once
eagerly (so that trace-time constants such as RoPE tables and parsed-module constants exist),
records a second run into a graph on private memory, and returns a callable that copies new
argument values into the graph's input buffers and replays it.  `fn` may be any composition of
this package's operators, `vjp` / `jvp` / `hlo_call` included (e.g. `lambda *a: vjp(f, *a)[1](dy)`).

The result tensors belong to the graph and are overwritten by the next replay; clone what must
outlive it.  Argument shapes and dtypes are fixed at capture.  Nothing here records a memset
node: buffers are cleared by fill kernels.
"""
import bisect
import ctypes

import torch

from . import _native as N
from .primitives import tree_flatten, tree_unflatten


class Captured:
    def __init__(self, fn, example_args):
        leaves, self._treedef = tree_flatten(tuple(example_args))
        for l in leaves:
            if isinstance(l, torch.Tensor) and not l.is_cuda:
                raise RuntimeError("argument is not in device memory: the HIP path has no CPU fallback")
        self._inputs = [l.clone() if isinstance(l, torch.Tensor) else l for l in leaves]
        spans = sorted((t.data_ptr(), t.data_ptr() + max(t.untyped_storage().nbytes(), 1)) for t in self._inputs if isinstance(t, torch.Tensor))
        self._starts, self._ends = [a for a, _ in spans], [b for _, b in spans]
        args = tree_unflatten(self._treedef, self._inputs)
        side = torch.cuda.Stream()                       # default priority
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            fn(*args)                                    # eager run: fills caches, surfaces errors outside capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self._outputs = fn(*args)
        self.replays = 0

    def __call__(self, *args):
        leaves, treedef = tree_flatten(tuple(args))
        if len(leaves) != len(self._inputs):
            raise ValueError("captured with %d argument leaves, called with %d" % (len(self._inputs), len(leaves)))
        pairs = []
        for s, a in zip(self._inputs, leaves):
            if isinstance(s, torch.Tensor):
                if not isinstance(a, torch.Tensor) or a.shape != s.shape or a.dtype != s.dtype:
                    raise ValueError("argument does not match the captured %s/%s" % (tuple(s.shape), s.dtype))
                pairs.append((s, a))
            elif a != s:
                raise ValueError("non-tensor argument %r differs from the captured %r" % (a, s))
        self._copy_in(pairs)
        self.graph.replay()
        self.replays += 1
        return self._outputs

    def _copy_in(self, pairs):
        """New argument values into the graph's buffers, on the current stream: whole arrays on its device by one launch.  One by
        one, in order, where an argument is itself one of those buffers (an output that is an argument passed through)."""
        # the tables and checks cost the host 7 us, a copy of its own 4.5 (replay, a copy each | one launch: of one argument 20 | 27 us, of
        # two 25 | 29, of four 38 | 35, of twelve 72 | 52)
        if len(pairs) < 3:
            for s, a in pairs:
                s.copy_(a)
            return
        here = torch.cuda.current_device()
        plain = [type(a) is torch.Tensor and a.device.type == "cuda" and a.device.index == here == s.device.index and a.is_contiguous()
                 and s.is_contiguous() and not (a.is_conj() or a.is_neg()) for s, a in pairs]
        for _, a in pairs:
            p = a.data_ptr() if a.device.type == "cuda" and a.layout == torch.strided else 0
            at = bisect.bisect_right(self._starts, p) - 1
            if at >= 0 and p < self._ends[at]:
                plain = [False] * len(pairs)
                break
        for (s, a), whole in zip(pairs, plain):
            if not whole:
                s.copy_(a)
        pairs = [pair for pair, whole in zip(pairs, plain) if whole]
        if pairs:
            table, sizes = ctypes.c_void_p * len(pairs), ctypes.c_int64 * len(pairs)
            N.check(N.lib().emi_copy_many(torch._C._cuda_getCurrentRawStream(here), len(pairs), table(*[a.data_ptr() for _, a in pairs]),
                                          table(*[s.data_ptr() for s, _ in pairs]), sizes(*[s.numel() * s.element_size() for s, _ in pairs])))


def capture(fn, *example_args):
    """Capture `fn(*example_args)` into a HIP graph; the returned callable takes arguments of
    the same structure, shapes and dtypes and returns the graph's (reused) result tensors."""
    return Captured(fn, example_args)
