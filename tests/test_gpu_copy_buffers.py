"""The one-launch copy of a captured block's inputs (dwm_copy_buffers): whole
16-byte, 4-byte and odd sizes, unaligned buffers, and MoeBlockGraph inputs
that are not plain copies."""
import ctypes

import numpy as np
import pytest
import torch

from dw_tpu_amd import _lib


def _copy(src, dst, nbytes, stream=None):
    n = len(src)
    return _lib.call("dwm_copy_buffers", (ctypes.c_void_p * max(n, 1))(*src), (ctypes.c_void_p * max(n, 1))(*dst),
                     (ctypes.c_int64 * max(n, 1))(*nbytes), n, stream)


def test_copy_buffers_rejects_bad_arguments():
    with pytest.raises(ValueError, match="0 .. 4 buffers"):
        _copy([16] * 5, [32] * 5, [4] * 5)
    with pytest.raises(ValueError, match="bad buffer 1"):
        _copy([16, 0], [32, 48], [0, 4])
    with pytest.raises(ValueError, match="bad buffer 0"):
        _copy([16], [32], [-1])
    _copy([], [], [])           # nothing to copy
    _copy([16], [16], [64])     # onto itself


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(1,), (14336, 32, 32), (4096, 4100, 4097, 0), (16, 3, 1 << 20, 10_000_004)])
@pytest.mark.parametrize("shift", [0, 4, 1])
def test_copy_buffers(dev, sizes, shift):
    g = torch.Generator(device=dev).manual_seed(3)
    src = [torch.randint(0, 256, (n + 32,), generator=g, dtype=torch.uint8, device=dev) for n in sizes]
    dst = [torch.full((n + 32,), 7, dtype=torch.uint8, device=dev) for n in sizes]
    _copy([t.data_ptr() + shift for t in src], [t.data_ptr() + 16 for t in dst], sizes, _lib.stream_handle(dev))
    torch.cuda.synchronize()
    for n, s, d in zip(sizes, src, dst):
        assert torch.equal(d[16:16 + n], s[shift:shift + n])
        assert (d[:16] == 7).all() and (d[16 + n:] == 7).all()


@pytest.mark.gpu
def test_graph_inputs_of_other_forms(dev, rng):
    from dw_tpu_amd import MoeBlockGraph, fp4_weight_to_codes, moe_block
    T, E, topk, H, I = 24, 8, 2, 256, 128
    fp4 = lambda *s: torch.from_numpy(rng.integers(0, 256, s, dtype=np.uint8)).to(dev)  # noqa: E731
    sc = lambda *s: torch.from_numpy(rng.integers(120, 126, s, dtype=np.uint8)).to(dev)  # noqa: E731
    w13 = fp4_weight_to_codes(fp4(E, H, I), sc(E, H // 32, 1, 2 * I), gate_up=True)
    w2 = fp4_weight_to_codes(fp4(E, I, H // 2), sc(E, I // 32, 1, H))
    new = lambda: (torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(dev).bfloat16(),  # noqa: E731
                   torch.from_numpy(rng.integers(0, E, (T, topk)).astype(np.int32)).to(dev),
                   torch.from_numpy(rng.random((T, topk)).astype(np.float32)).to(dev))
    graph = MoeBlockGraph(*new(), w13, w2, E)
    for form in ("plain", "strided", "int64 ids", "host weights", "own buffer"):
        h, ids, w = new()
        want = moe_block(h, ids, w, w13, w2, E)
        if form == "strided":
            got = graph(h.t().contiguous().t(), ids, w)
        elif form == "int64 ids":
            got = graph(h, ids.long(), w)
        elif form == "host weights":
            got = graph(h, ids, w.cpu())
        elif form == "own buffer":
            graph.hidden.copy_(h)
            got = graph(graph.hidden, ids, w)
        else:
            got = graph(h, ids, w)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), form
    with pytest.raises(ValueError, match="captured"):
        graph(h[:8], ids, w)


@pytest.mark.gpu
def test_graph_inputs_with_a_lazy_sign(dev, rng):
    """A negated view's bytes are those of its base: torch's copy resolves it."""
    from dw_tpu_amd import MoeBlockGraph, fp4_weight_to_codes, moe_block
    T, E, topk, H, I = 24, 8, 2, 256, 128
    fp4 = lambda *s: torch.from_numpy(rng.integers(0, 256, s, dtype=np.uint8)).to(dev)  # noqa: E731
    sc = lambda *s: torch.from_numpy(rng.integers(120, 126, s, dtype=np.uint8)).to(dev)  # noqa: E731
    w13 = fp4_weight_to_codes(fp4(E, H, I), sc(E, H // 32, 1, 2 * I), gate_up=True)
    w2 = fp4_weight_to_codes(fp4(E, I, H // 2), sc(E, I // 32, 1, H))
    h = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(dev)
    ids = torch.from_numpy(rng.integers(0, E, (T, topk)).astype(np.int32)).to(dev)
    w = torch.from_numpy(rng.random((T, topk)).astype(np.float32)).to(dev)
    graph = MoeBlockGraph(h.bfloat16(), ids, w, w13, w2, E)
    neg = torch._neg_view(w)
    assert neg.is_neg() and neg.is_contiguous()
    got = graph(h.bfloat16(), ids, neg)
    want = moe_block(h.bfloat16(), ids, -w, w13, w2, E)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
