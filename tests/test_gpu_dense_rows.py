"""The dense FP8 launches for few rows: the rows kernel (17 .. 32 rows, W8A8 .. 96)
and W8A16's 64-row MFMA tiles at the edges of its row tiles, K runs and column tiles, and the skinny
kernel's forms for shallow K (fewer waves) and wide N (four column groups per
block), against the float64 oracle under the stated bound, with the plan the
library launched."""
import numpy as np
import pytest
import torch

from conftest import bf16_bits, bf16_tensor
from oracle import dense_fp8 as odf
from oracle import gmm as ogmm
from oracle.numerics import bf16_to_f32

pytestmark = pytest.mark.gpu


def _check(out, y64, ap, K):
    y = bf16_to_f32(bf16_bits(out)).astype(np.float64)
    err = np.abs(y - y64)
    assert np.all(np.isfinite(y))
    assert np.all(err <= odf.error_bound(y64, ap, K)), ogmm.error_stats(y, y64)


@pytest.mark.parametrize("M,K,N,plan", [
    (17, 128, 128, (4, 32, 64, 1, 2)),     # one K block: seven of eight waves have none
    (32, 4224, 256, (4, 32, 64, 4, 2)),    # 33 K blocks: past the 32 of one run
    (33, 1152, 384, (4, 48, 32, 1, 2)),
    (48, 2048, 128, (4, 48, 32, 2, 2)),
    (49, 3072, 512, (4, 64, 32, 3, 2)),
    (64, 1408, 256, (4, 64, 32, 1, 2)),
    (65, 1024, 128, (4, 96, 32, 2, 2)),
    (95, 2176, 640, (4, 96, 32, 4, 2)),    # 17 K blocks in runs of 5, 5, 5, 2
    (96, 640, 8192, (4, 96, 32, 1, 2)),    # 256 column tiles
    (96, 640, 8320, (2, 128, 128, 3, 4)),  # 260: the MFMA tiles
    (97, 1024, 256, (2, 128, 128, 8, 4)),
    (32, 256, 16640, (4, 32, 64, 1, 2)),   # two rounds of column tiles
    (32, 256, 32768, (2, 128, 128, 1, 4)),  # under 4 K blocks: one round of MFMA tiles instead
    (80, 4224, 8192, (2, 128, 128, 4, 4)),  # past 64 rows, 33 K blocks in one run against one round of tiles
])
def test_w8a8_rows_plans_against_oracle(dev, M, K, N, plan):
    from dw_tpu_amd.dense_fp8 import last_plan, matmul_w8a8
    from dw_tpu_amd.dense_fp8_tiles import plan_to_tile
    from dw_tpu_amd.workloads import make_dense_workload
    wl = make_dense_workload(M, K, N, seed=M + K)
    args = [torch.from_numpy(v).to(dev) for v in (wl.xq, wl.sx, wl.wq, wl.sw)]
    out = matmul_w8a8(*args)
    torch.cuda.synchronize()
    p = last_plan()
    assert p.astuple() == plan
    y64 = odf.matmul_w8a8(wl.xq, wl.sx, wl.wq, wl.sw, out_dtype="float64")
    _check(out, y64, odf.abs_product_w8a8(wl.xq, wl.sx, wl.wq, wl.sw), K)
    again = matmul_w8a8(*args, tile=plan_to_tile(p, K))
    assert torch.equal(again.view(torch.int16), out.view(torch.int16)) and last_plan().astuple() == plan


@pytest.mark.parametrize("M,K,N,plan", [
    (17, 512, 128, (4, 32, 64, 1, 2)),
    (32, 4224, 256, (4, 32, 64, 4, 2)),
    (24, 1152, 384, (4, 32, 64, 1, 2)),
    (32, 1152, 16640, (4, 32, 64, 1, 2)),   # two rounds of column tiles
    # up to three K blocks, up to eight in a second round, narrow products: 64-row MFMA tiles
    (17, 128, 128, (2, 64, 128, 1, 4)),
    (32, 256, 16640, (2, 64, 128, 1, 4)),
    (31, 1152, 384, (2, 64, 128, 5, 4)),
    (24, 2176, 128, (2, 64, 128, 6, 4)),    # 17 K blocks in runs of 3, 3, 3, 3, 3, 2
    (33, 1024, 256, (2, 64, 128, 8, 4)),   # past 32 rows: 64-row MFMA tiles
    (64, 1152, 128, (2, 64, 128, 5, 4)),   # runs of 2, 2, 2, 2, 1 K blocks: two steps in a four-stage ring
    (48, 384, 33024, (2, 64, 128, 1, 4)),
    (65, 1024, 256, (2, 128, 128, 8, 3)),
    # widths off the 128 grid: rows kernel, general tiles (33 .. 64 rows), MFMA tiles with a part-filled last one
    (17, 256, 16, (4, 32, 64, 1, 2)),
    (17, 128, 16, (3, 64, 128, 1, 2)),      # one K block: general tiles
    (32, 256, 16400, (3, 64, 128, 2, 2)),   # two in a second round
    (32, 2048, 208, (4, 32, 64, 2, 2)),
    (29, 384, 4080, (4, 32, 64, 1, 2)),
    (64, 512, 144, (3, 64, 128, 4, 2)),
    (65, 512, 144, (5, 128, 128, 4, 3)),
    (128, 1152, 240, (5, 128, 128, 5, 3)),
    (300, 256, 1040, (5, 128, 128, 2, 3)),
    (200, 512, 112, (3, 128, 128, 4, 2)),   # a single part-filled tile stays on the general kernel
    (2049, 128, 3600, (5, 256, 128, 1, 3)),
])
def test_w8a16_rows_plans_against_oracle(dev, M, K, N, plan):
    from dw_tpu_amd.dense_fp8 import last_plan, matmul, prepack_fp8, try_dense_fp8
    from dw_tpu_amd.dense_fp8_tiles import plan_to_tile
    from dw_tpu_amd.workloads import make_dense_workload
    wl = make_dense_workload(M, K, N, seed=M + K + 2)
    x, pw = bf16_tensor(wl.x_bits, dev), prepack_fp8(torch.from_numpy(wl.wq).to(dev))
    s = torch.from_numpy(wl.s_w8a16).to(dev)
    out = try_dense_fp8(x, pw, s)
    torch.cuda.synchronize()
    p = last_plan()
    assert p.astuple() == plan
    xf = bf16_to_f32(wl.x_bits)
    _check(out, odf.matmul_w8a16(xf, wl.wq, wl.s_w8a16, out_dtype="float64"),
           odf.abs_product_w8a16(xf, wl.wq, wl.s_w8a16), K)
    t = plan_to_tile(p, K)
    again = matmul(x, pw, s, mode=t.mode, tm=t.tm, tk=t.tk, tn=t.tn, stages=t.stages)
    assert torch.equal(again.view(torch.int16), out.view(torch.int16)) and last_plan().astuple() == plan


@pytest.mark.parametrize("a8,M,K,N,plan", [
    (False, 17, 128, 128, (4, 32, 64, 1, 2)),   # one K block: seven of eight waves have none
    (False, 31, 1152, 384, (4, 32, 64, 1, 2)),
    (False, 24, 2176, 128, (4, 32, 64, 2, 2)),  # runs of 9 and 8 K blocks
    (False, 32, 256, 16640, (4, 32, 64, 1, 2)),
    (False, 20, 8192, 64, (4, 32, 64, 1, 2)),   # 64 K blocks in one run, the most
    (True, 20, 8192, 128, (4, 32, 64, 1, 2)),
    (True, 48, 8192, 128, (4, 48, 32, 1, 2)),
    (True, 64, 8320, 128, (4, 64, 32, 2, 2)),   # runs of 33 and 32
    (True, 96, 8192, 128, (4, 96, 32, 1, 2)),
])
def test_rows_kernel_by_plan(dev, a8, M, K, N, plan):
    """The rows kernel where the library's own rule takes other tiles."""
    from dw_tpu_amd import _lib
    from dw_tpu_amd.dense_fp8 import last_plan, matmul, matmul_w8a8
    from dw_tpu_amd.dense_fp8_tiles import plan_to_tile
    from dw_tpu_amd.workloads import make_dense_workload
    wl = make_dense_workload(M, K, N, seed=M + K + 3)
    t = plan_to_tile(_lib.DensePlan(*plan), K)
    if a8:
        out = matmul_w8a8(*(torch.from_numpy(v).to(dev) for v in (wl.xq, wl.sx, wl.wq, wl.sw)), tile=t)
        y64, ap = (f(wl.xq, wl.sx, wl.wq, wl.sw, **kw) for f, kw in (
            (odf.matmul_w8a8, {"out_dtype": "float64"}), (odf.abs_product_w8a8, {})))
    else:
        xf = bf16_to_f32(wl.x_bits)
        out = matmul(bf16_tensor(wl.x_bits, dev), torch.from_numpy(wl.wq).to(dev).view(torch.float8_e4m3fn),
                     torch.from_numpy(wl.s_w8a16).to(dev), mode=t.mode, tm=t.tm, tk=t.tk, tn=t.tn, stages=t.stages)
        y64 = odf.matmul_w8a16(xf, wl.wq, wl.s_w8a16, out_dtype="float64")
        ap = odf.abs_product_w8a16(xf, wl.wq, wl.s_w8a16)
    torch.cuda.synchronize()
    assert last_plan().astuple() == plan
    _check(out, y64, ap, K)


@pytest.mark.parametrize("a8", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 128, 48), (16, 512, 128), (5, 640, 256), (16, 1024, 80), (7, 1152, 128),
                                   (3, 256, 32768), (16, 512, 32832), (9, 896, 32768), (16, 1024, 33024)])
def test_skinny_forms_against_oracle(dev, a8, M, K, N):
    from dw_tpu_amd import _lib
    from dw_tpu_amd.dense_fp8 import last_plan, matmul, matmul_w8a8
    from dw_tpu_amd.workloads import make_dense_workload
    if a8:
        N = -(-N // 128) * 128
    wl = make_dense_workload(M, K, N, seed=M + K + 1)
    cols = np.unique(np.r_[0, 15, 16, 63, N - 17, N - 1, np.random.default_rng(1).integers(0, N, 200)] % N)
    if a8:
        out = matmul_w8a8(*(torch.from_numpy(v).to(dev) for v in (wl.xq, wl.sx, wl.wq, wl.sw)))
        sw = np.repeat(wl.sw, 128, axis=1)[:, cols]
        y64 = np.zeros((M, len(cols)))
        ap = np.zeros_like(y64)
        from oracle.numerics import E4M3_VALUES
        xv, wv = E4M3_VALUES[wl.xq].astype(np.float64), E4M3_VALUES[wl.wq[:, cols]].astype(np.float64)
        for kb in range(K // 128):
            sl = slice(kb * 128, kb * 128 + 128)
            f = wl.sx[:, kb][:, None].astype(np.float64) * sw[kb][None, :]
            y64 += (xv[:, sl] @ wv[sl]) * f
            ap += (np.abs(xv[:, sl]) @ np.abs(wv[sl])) * np.abs(f)
    else:
        out = matmul(bf16_tensor(wl.x_bits, dev), torch.from_numpy(wl.wq).to(dev).view(torch.float8_e4m3fn),
                     torch.from_numpy(wl.s_w8a16).to(dev))
        xf, wc, sc = bf16_to_f32(wl.x_bits), wl.wq[:, cols], wl.s_w8a16[:, :, cols]
        y64 = odf.matmul_w8a16(xf, wc, sc, out_dtype="float64")
        ap = odf.abs_product_w8a16(xf, wc, sc)
    torch.cuda.synchronize()
    assert last_plan().astuple() == (1, 16, 16, 16, 2)
    waves = 4 if K <= 512 else 8 if K <= 1024 else 16
    wide = K <= 1024 and N % 64 == 0 and N >= 128 * torch.cuda.get_device_properties(dev).multi_processor_count
    assert _lib.last_kernel() == f"dense_skinny/{waves}/{2 if waves == 16 else 1}/{4 if wide else 1}"
    _check(out[:, torch.from_numpy(cols).to(dev)], y64, ap, K)


def test_w8a8_rows_in_block_accumulation(dev):
    """The 16x16x128 fp8 MFMA of the rows kernel on rows that cancel inside
    one K block (448, -448 at some distance, then small values; weights and
    scales 1): it loses what the 32x32x64 MFMA of the tiles loses.  That is the
    alignment of small products to a large one, up to 2^-12 of it (the scaled
    MFMA's measured figure, see ``gmm.mx_error_bound``), here for two large
    ones, next to the bf16 output's half ulp."""
    from dw_tpu_amd import _lib
    from dw_tpu_amd.dense_fp8 import matmul_w8a8
    from dw_tpu_amd.dense_fp8_tiles import DenseTile
    K, N = 128, 128
    rows = []
    for v in (1.0, 0.375, 0.0625, 0.046875, 2.0 ** -5, 2.0 ** -6, 2.0 ** -7, 2.0 ** -9, 3 * 2.0 ** -9):
        for at in (1, 9, 17, 33, 40, 65, 100, 127):
            r = np.full(K, v, np.float32)
            r[0], r[at] = 448.0, -448.0
            rows.append(r)
    x = torch.from_numpy(np.stack(rows)).to(dev).to(torch.float8_e4m3fn)
    M = len(rows)
    assert 65 <= M <= 96
    args = (x, torch.ones((M, 1), device=dev), torch.ones((K, N), device=dev).to(torch.float8_e4m3fn),
            torch.ones((1, 1), device=dev))
    want = x.float().double().sum(1).cpu().numpy()
    err = {}
    for tile in (None, DenseTile("native", 128, 128, 128, 4)):
        y = matmul_w8a8(*args, **({} if tile is None else dict(tile=tile)))
        y = y[:, 0].float().cpu().numpy().astype(np.float64)
        err[_lib.last_kernel()] = np.maximum(0, np.abs(y - want) - 2.0 ** -9 * np.abs(want)) / 448.0
    print({k: float(e.max()) for k, e in err.items()})
    assert np.array_equal(err["dense_rows"], err["dense_mfma"])
    assert err["dense_rows"].max() <= 2 * 2.0 ** -12
