"""The streaming kernel of the grouped matmul (csrc/gmm_stream.hip), which
takes launches with few rows per expert: against the float64 oracle under the
stated bound, and bit for bit against the 96-row tiles, which the same rows
take when every group is padded with further rows (a row's result depends on
its own lhs row and expert only)."""
import numpy as np
import pytest
import torch

from conftest import bf16_bits, bf16_tensor
from oracle import fp4 as ofp4
from oracle import gmm as ogmm
from oracle.numerics import bf16_bits as f32_to_bf16_bits
from oracle.numerics import bf16_to_f32

pytestmark = pytest.mark.gpu


def _sizes(E, pattern):
    return np.array([pattern[i % len(pattern)] for i in range(E)], np.int32)


# K: 1, 2, 3, 4, 5, 7, 8 and 11 K blocks around the register ring's depths (3
# and 4); N: ragged 64-column groups; groups past 64 and 256 (4 and 16 sizes
# per lane); one- and four-wave blocks (the 300 groups); rows 15 / 16 / 17 and
# 31 / 32 / 33 around the 16- and 32-row tiles; a few groups of many rows.
CASES = [
    (4, 128, 16, [1, 0, 2, 1], None, False, "none"),
    (8, 256, 80, [1, 3, 0, 4], None, False, "f32"),
    (12, 384, 272, [17, 0, 1, 0, 1, 2], None, False, "bias"),
    (12, 512, 128, [16, 0, 15, 0, 1, 2], None, True, "none"),
    (24, 640, 192, [31, 0, 0, 33, 0, 1, 0, 0, 0, 5, 0, 0], None, True, "bias"),
    (40, 896, 320, [32, 0, 0, 0, 0, 70, 0, 0, 0, 0, 0, 0, 0, 1, 2, 3, 0, 0, 0, 0], None, False, "gather"),
    (100, 1024, 64, [0, 1, 2, 0, 16, 0, 17, 3] + [0] * 12, (30, 40), False, "none"),
    (300, 1408, 1280, [1, 0, 0, 2], None, False, "gather"),
    (300, 128, 1040, [0, 1, 3, 0, 8], (7, 290), False, "f32"),
    (1024, 256, 128, [0, 0, 1], None, True, "gather"),
    # four-wave blocks that run one (4 experts of 32 rows, 12 of 96) or two waves (24 x 64 column groups), 18 experts
    # whose one-wave list would not fit the grid, and one large group among single rows (16-row tiles in two rounds)
    (64, 256, 4096, [32] + [0] * 15, None, False, "none"),
    (64, 128, 4096, [96] + [0] * 15, None, False, "gather"),
    (128, 128, 4096, [192] + [0] * 31, None, True, "none"),
    (64, 128, 4096, [7, 0, 0, 0, 0, 7, 0], None, False, "f32"),
    (64, 256, 4096, [64] + [1] * 63, None, False, "none"),
    # one-wave blocks with the choice of 16-row tiles (a group of 20 among single rows) and just too small for it
    (32, 256, 4096, [20] + [1] * 20 + [0] * 11, None, False, "none"),
    (32, 256, 4096, [16] + [1] * 16 + [0] * 15, None, True, "none"),
    # more rows per expert, in launches too small to fill the chip with tiles: 33 .. 64 rows of all, one and both
    # clauses' edges (12 and 64 rows per expert), a window
    (4, 384, 640, [50, 0, 64, 33], None, False, "none"),
    (8, 256, 2560, [12], None, True, "none"),
    (3, 640, 272, [64], None, False, "f32"),
    (40, 128, 80, [0, 70, 16, 31], (5, 30), False, "gather"),
    (2, 1408, 1040, [65, 63], None, False, "bias"),
]


@pytest.mark.parametrize("E,K,N,pattern,window,act,form", CASES)
def test_stream_kernel_against_oracle_and_tiles(dev, rng, E, K, N, pattern, window, act, form):
    from dw_tpu_amd import _lib, fp4_weight_to_codes, gmm_v2
    sizes = _sizes(E, pattern)
    go, e_local = window if window else (0, E)
    M = int(sizes.sum())
    assert 0 < M <= 64 * e_local
    rhs = rng.integers(0, 256, (e_local, K, N // 2), dtype=np.uint8)
    sc = rng.integers(123, 130, (e_local, K // 32, 1, N), dtype=np.uint8)
    pw = fp4_weight_to_codes(torch.from_numpy(rhs).to(dev), torch.from_numpy(sc).to(dev), gate_up=act)
    bits = f32_to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    bias = torch.from_numpy(rng.standard_normal((e_local, N)).astype(np.float32)).to(dev) if form == "bias" else None
    kw = dict(rhs_bias=bias, group_offset=go if window else None,
              preferred_element_type=torch.float32 if form == "f32" else None,
              fuse_act="silu_and_mul_with_clamp" if act else None)
    gs = torch.from_numpy(sizes).to(dev)
    lhs = bf16_tensor(bits, dev)
    if form == "gather":
        idx = rng.permutation(M).astype(np.int32)
        src = np.empty_like(bits)
        src[idx] = bits
        y = gmm_v2(bf16_tensor(src, dev), pw, gs, lhs_row_indices=torch.from_numpy(idx).to(dev), **kw)
    else:
        y = gmm_v2(lhs, pw, gs, **kw)
    assert _lib.last_kernel() == "gmm_stream"
    # The same rows at the head of groups padded to more than 72 rows each.
    pad = 80
    big = sizes + pad
    assert big.sum() > 64 * e_local
    starts = np.concatenate([[0], np.cumsum(big)[:-1]])
    at = np.concatenate([s + np.arange(n) for s, n in zip(starts, sizes)]).astype(np.int64)
    rows = np.zeros((int(big.sum()), K), np.uint16)
    rows[at] = bits
    at = torch.from_numpy(at).to(dev)
    yb = gmm_v2(bf16_tensor(rows, dev), pw, torch.from_numpy(big).to(dev), **kw)[at]
    assert _lib.last_kernel() == "gmm_ws"
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int32 if form == "f32" else torch.int16),
                       yb.view(torch.int32 if form == "f32" else torch.int16))
    lo, hi = int(sizes[:go].sum()), int(sizes[:go + e_local].sum())
    assert (y[:lo] == 0).all() and (y[hi:] == 0).all()
    if act or form == "bias":
        return  # the epilogue is the tiles' own, compared bit for bit above
    x = bf16_to_f32(bits)[lo:hi]
    loc = sizes[go:go + e_local]
    w = ogmm.dequant_rhs(ofp4.e2m1_to_codes(ofp4.unpack_nibbles(rhs)), ofp4.e8m0_decode(sc))
    y64, _ = ogmm.gmm(x, None, None, loc, out_dtype="float64", w=w)
    got = y[lo:hi].cpu().numpy() if form == "f32" else bf16_to_f32(bf16_bits(y[lo:hi]))
    err = np.abs(got.astype(np.float64) - y64)
    assert np.all(err <= ogmm.error_bound(y64, ogmm.abs_product(x, w, loc), K,
                                          "float32" if form == "f32" else "bfloat16")), ogmm.error_stats(got, y64)


@pytest.mark.parametrize("E,K,N,pattern,window,act,form", CASES)
@pytest.mark.parametrize("fmt", ["e4m3", "e2m1"])
def test_mx_stream_kernel_equals_tiles(dev, rng, E, K, N, pattern, window, act, form, fmt):
    """The MX form gives the bits of the MX tiles (both K step depths: K below
    and from 4096 on) for every group and epilogue form above."""
    from dw_tpu_amd import MxLhs, _lib, fp4_weight_to_codes, gmm_v2, mx_quantize
    if E == 4:
        K = 4224
    sizes = _sizes(E, pattern)
    go, e_local = window if window else (0, E)
    M = int(sizes.sum())
    assert 0 < M <= 64 * e_local
    pw = fp4_weight_to_codes(torch.from_numpy(rng.integers(0, 256, (e_local, K, N // 2), dtype=np.uint8)).to(dev),
                             torch.from_numpy(rng.integers(123, 130, (e_local, K // 32, 1, N), dtype=np.uint8)).to(dev),
                             gate_up=act)
    x = mx_quantize(bf16_tensor(f32_to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32)), dev), fmt)
    bias = torch.from_numpy(rng.standard_normal((e_local, N)).astype(np.float32)).to(dev) if form == "bias" else None
    kw = dict(rhs_bias=bias, group_offset=go if window else None,
              preferred_element_type=torch.float32 if form == "f32" else None,
              fuse_act="silu_and_mul_with_clamp" if act else None)
    if form == "gather":
        p = torch.from_numpy(rng.permutation(M).astype(np.int32)).to(dev)
        codes, scales = torch.empty_like(x.codes), torch.empty_like(x.scales)
        codes[p.long()], scales[p.long()] = x.codes, x.scales
        y = gmm_v2(MxLhs(codes, scales, fmt), pw, torch.from_numpy(sizes).to(dev), lhs_row_indices=p, **kw)
    else:
        y = gmm_v2(x, pw, torch.from_numpy(sizes).to(dev), **kw)
    assert _lib.last_kernel() == "gmm_mx_stream"
    big = sizes + 80
    assert big.sum() > 64 * e_local
    starts = np.concatenate([[0], np.cumsum(big)[:-1]])
    at = torch.from_numpy(np.concatenate([s + np.arange(n) for s, n in zip(starts, sizes)]).astype(np.int64)).to(dev)
    codes = torch.zeros((int(big.sum()), x.codes.shape[1]), dtype=torch.uint8, device=dev)
    scales = torch.full((int(big.sum()), x.scales.shape[1]), 127, dtype=torch.uint8, device=dev)
    codes[at], scales[at] = x.codes, x.scales
    yb = gmm_v2(MxLhs(codes, scales, fmt), pw, torch.from_numpy(big).to(dev), **kw)[at]
    assert _lib.last_kernel() == ("gmm_mx128" if K >= 4096 else "gmm_mx")
    torch.cuda.synchronize()
    v = torch.int32 if form == "f32" else torch.int16
    assert torch.equal(y.view(v), yb.view(v)) and bool((y != 0).any())


@pytest.mark.parametrize("E,M,N,mx,kernel", [
    (32, 192, 4096, False, "gmm_stream"),   # 6 rows per expert
    (32, 193, 8192, False, "gmm_ws"),       # 33 tiles x 32 column tiles: past half of the CUs
    (8, 512, 2304, True, "gmm_mx_stream"),  # 64 rows per expert, 13 x 9 tiles of 128 allowed
    (8, 513, 2304, True, "gmm_mx"),
    (8, 512, 2560, False, "gmm_ws"),        # 13 x 10
    (8, 300, 2816, False, "gmm_stream"),    # 11 x 11
])
def test_stream_rule(dev, rng, E, M, N, mx, kernel):
    from dw_tpu_amd import _lib, fp4_weight_to_codes, gmm_v2
    K = 128
    pw = fp4_weight_to_codes(torch.zeros((E, K, N // 2), dtype=torch.uint8, device=dev),
                             torch.full((E, K // 32, 1, N), 127, dtype=torch.uint8, device=dev))
    gs = torch.from_numpy(rng.multinomial(M, np.ones(E) / E).astype(np.int32)).to(dev)
    y = gmm_v2(torch.ones((M, K), dtype=torch.bfloat16, device=dev), pw, gs,
               lhs_quant_dtype=torch.float8_e4m3fn if mx else None)
    assert _lib.last_kernel() == kernel
    assert not y.any()


def test_stream_kernel_skips_rows_past_m(dev, rng):
    """Device group sizes whose sum passes M: no row past M is read or
    written (lhs and out are padded), and rows below M are those of sizes cut
    to fit."""
    import ctypes
    from dw_tpu_amd import _lib, fp4_weight_to_codes
    E, K, N, M, pad = 16, 256, 128, 60, 64
    sizes = _sizes(E, [5, 0, 40, 3])
    assert M <= 6 * E and sizes.sum() > M + 40
    pw = fp4_weight_to_codes(torch.from_numpy(rng.integers(0, 256, (E, K, N // 2), dtype=np.uint8)).to(dev),
                             torch.from_numpy(rng.integers(123, 130, (E, K // 32, 1, N), dtype=np.uint8)).to(dev))
    lhs = bf16_tensor(f32_to_bf16_bits(rng.standard_normal((M + pad, K)).astype(np.float32)), dev)
    fit = np.minimum(sizes, np.maximum(0, M - np.concatenate([[0], np.cumsum(sizes)[:-1]]))).astype(np.int32)
    outs = []
    for s in (sizes, fit):
        gs = torch.from_numpy(s).to(dev)
        out = torch.full((M + pad, N), 0x1234, dtype=torch.int16, device=dev)
        P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        _lib.call("dwm_gmm_fp4", P(lhs), M, K, P(pw.weight), P(pw.scale), P(gs), E, None, E, N, P(out), _lib.BF16, 0,
                  _lib.ACT_NONE, _lib.stream_handle(dev))
        torch.cuda.synchronize()
        assert (out[M:] == 0x1234).all()
        outs.append(out[:M])
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("mx", [False, True])
@pytest.mark.parametrize("E,sizes,M", [
    (8, {0: 10000}, 20),                         # the first group alone runs far past M
    (8, {0: 3, 2: 40, 5: 1 << 30, 6: 1 << 30}, 47),  # the sum leaves int32
    (300, {7: 5, 40: 33, 120: 2000, 280: 2000}, 60),  # several sizes per lane
])
def test_stream_kernel_covers_the_rows_below_m(dev, rng, mx, E, sizes, M):
    """Device group sizes that sum far past M, with many more tiles than the
    grid has blocks: every row below M is that of sizes cut to fit, and none
    past it is written."""
    import ctypes
    from dw_tpu_amd import _lib, fp4_weight_to_codes, mx_quantize
    K, N, pad = 256, 512, 64
    s = np.zeros(E, np.int64)
    s[list(sizes)] = list(sizes.values())
    fit = np.minimum(s, np.maximum(0, M - np.concatenate([[0], np.cumsum(s)[:-1]])))
    assert M <= 6 * E and fit.sum() == M
    pw = fp4_weight_to_codes(torch.from_numpy(rng.integers(0, 256, (E, K, N // 2), dtype=np.uint8)).to(dev),
                             torch.from_numpy(rng.integers(123, 130, (E, K // 32, 1, N), dtype=np.uint8)).to(dev))
    lhs = bf16_tensor(f32_to_bf16_bits(rng.standard_normal((M + pad, K)).astype(np.float32)), dev)
    q = mx_quantize(lhs)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    outs = []
    for v in (s, fit):
        gs = torch.from_numpy(v.astype(np.int32)).to(dev)
        out = torch.full((M + pad, N), 0x1234, dtype=torch.int16, device=dev)
        tail = (M, K, P(pw.weight), P(pw.scale), P(gs), E, None, E, N, P(out), _lib.BF16, 0, _lib.ACT_NONE,
                _lib.stream_handle(dev))
        if mx:
            _lib.call("dwm_gmm_fp4_mx", P(q.codes), P(q.scales), M, None, *tail)
        else:
            _lib.call("dwm_gmm_fp4", P(lhs), *tail)
        torch.cuda.synchronize()
        assert (out[M:] == 0x1234).all()
        outs.append(out[:M])
    assert (outs[1] != 0x1234).any(dim=1).all()
    assert torch.equal(outs[0], outs[1])
