"""The Python side of the operators on CPU tensors: the library's entry points are replaced by a stub that looks at every tensor
handed to it (its type against the I/O type named in the call, its alignment) and fills what the call would write.

New memory is NaN until a stub fills it, so that a result nobody wrote shows.  The values mean nothing; what is checked are the
routes, the operands' types and the graph."""
import torch

IO = {0: torch.float32, 1: torch.bfloat16}

#: floating-point arguments of another type than the call's I/O type, by position (statistics, residuals, states, parameter sums)
OTHER = {
    "hiprwkv_rwkv7_ln_shiftmix": {20}, "hiprwkv_rwkv7_ln_shiftmix_bwd": {7}, "hiprwkv_wkv7_fwd_parts": {13, 17, 18},
    "hiprwkv_wkv7_step": {13, 18}, "hiprwkv_wkv7_bwd": {13, 17, 18, 25}, "hiprwkv_rwkv7_postmix_bwd": {20, 21, 22},
    "hiprwkv_rwkv7_shiftmix_bwd": {15},
}

#: position of the shift row, whose batch stride follows it
SHIFT_ROW = {"hiprwkv_rwkv7_ln_shiftmix": 11, "hiprwkv_rwkv7_ln_shiftmix_bwd": 10, "hiprwkv_rwkv7_shiftmix": 7,
             "hiprwkv_rwkv7_shiftmix_bwd": 7}


def _tensors(args):
    for i, a in enumerate(args):
        if torch.is_tensor(a):
            yield i, a
        elif isinstance(a, list):
            yield from ((i, t) for t in a)


class Library:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name.endswith("fwd_workspace_bytes"):
            return lambda *a: 0
        if name.endswith("workspace_bytes"):
            return lambda *a: 64

        def call(stream, io, *args):
            self.calls.append(name)
            fill([t for _, t in _tensors(args)])
            if name in SHIFT_ROW:
                row, stride = args[SHIFT_ROW[name] - 2:][:2]
                assert row is None or len(row) == 1 or row.stride(0) == stride, (name, row.stride(), stride)
            for i, t in _tensors(args):
                assert t.data_ptr() % 16 == 0 or not t.is_floating_point(), (name, i + 2)
                if t.is_floating_point() and i + 2 not in OTHER.get(name, ()):
                    assert t.dtype == IO[io], (name, i + 2, t.dtype, IO[io])
            return 0
        return call


def fill(tensors):
    with torch.no_grad():
        for t in tensors:
            if t.is_floating_point() and not t.is_meta and t.isnan().any():
                t.data.masked_fill_(t.isnan(), 0.01)


def install(monkeypatch):
    """Puts the stub in the library's place and returns it; ``stub.calls`` lists the entry points called, in order."""
    from jaxrwkv_amd import _lib, blocks7, ops
    stub = Library()
    empty, empty_like = torch.empty, torch.empty_like

    def nan(t):
        return t.fill_(float("nan")) if t.is_floating_point() else t

    def gemm(jobs):
        stub.calls.append("hiprwkv_gemm")
        for out, x, w, km, kn, act, aux in jobs:
            ops._one_dtype(torch.bfloat16, out, x, w, aux)
            M, K = x.T.shape if km else x.shape
            assert (K, out.shape[1]) == tuple(w.shape if kn else w.T.shape) and out.shape[0] == M
        fill([j[0] for j in jobs])

    monkeypatch.setattr(torch, "empty", lambda *a, **k: nan(empty(*a, **k)))
    monkeypatch.setattr(torch, "empty_like", lambda *a, **k: nan(empty_like(*a, **k)))
    new_empty = torch.Tensor.new_empty
    monkeypatch.setattr(torch.Tensor, "new_empty", lambda *a, **k: nan(new_empty(*a, **k)))
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True))
    monkeypatch.setattr(_lib, "load", lambda: stub)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_p", lambda t: t)
    monkeypatch.setattr(ops, "_ptr_array", list)
    monkeypatch.setattr(blocks7, "_gemm", gemm)
    return stub
