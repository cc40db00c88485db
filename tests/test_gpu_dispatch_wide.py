"""The one-launch dispatch over several blocks (dispatch_wide_kernel in
csrc/moe.hip) and its neighbours, bit for bit against a stable argsort:
portions of 1024 ids (one portion in a block of fewer waves), the rounds of
8192 ids each block counts, 1, 4 and 8 copies of the counters, the largest
batches of one launch (49152 ids under 128 experts, else 65536), the three
launches above them, and ids outside the experts."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,topk,E", [
    (1, 1, 64), (341, 3, 64), (512, 2, 256), (205, 5, 1024),    # 1, 1023, 1024 and 1025 ids
    (4096, 2, 63), (8193, 1, 63), (8193, 1, 64), (1365, 6, 256),  # 8192 ids over few experts, 8193, 8190
    (4096, 6, 256), (5461, 12, 8), (8192, 8, 1024),              # 24576, 65532 and 65536 ids
    (8192, 3, 1024), (8192, 3, 128), (24577, 1, 300), (200, 2, 70),  # 24576 and 24577 ids; 400
    (49152, 1, 64), (49153, 1, 64), (49153, 1, 128),             # both sides of the limit under 128 experts
    (65537, 1, 100), (65537, 1, 1024), (9000, 8, 32),            # past one launch
])
@pytest.mark.parametrize("skew", [False, True])
def test_dispatch_is_a_stable_argsort(dev, T, topk, E, skew):
    from dw_tpu_amd import moe_dispatch
    rng = np.random.default_rng(T + E)
    ids = rng.integers(0, E, (T, topk)).astype(np.int32)
    if skew:  # one expert takes most rows, some ids are outside [0, E)
        ids[rng.random((T, topk)) < 0.8] = E // 2
        ids[rng.random((T, topk)) < 0.01] = E + 5
        ids[rng.random((T, topk)) < 0.01] = -3
    d = moe_dispatch(torch.from_numpy(ids).to(dev), E)
    torch.cuda.synchronize()
    key = np.where((ids.ravel() >= 0) & (ids.ravel() < E), ids.ravel(), E)
    perm = np.argsort(key, kind="stable")
    assert np.array_equal(d.topk_argsort_indices.cpu().numpy(), perm)
    assert np.array_equal(d.token_indices_sorted.cpu().numpy(), perm // topk)
    rev = np.empty_like(perm)
    rev[perm] = np.arange(perm.size)
    assert np.array_equal(d.topk_argsort_revert_indices.cpu().numpy(), rev)
    gs = np.bincount(key, minlength=E + 1)[:E]
    assert np.array_equal(d.group_sizes.cpu().numpy(), gs)
    assert np.array_equal(d.group_offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(gs)]))
    bad = bool(((ids < 0) | (ids >= E)).any())
    if bad:
        with pytest.raises(ValueError, match="outside"):
            moe_dispatch(torch.from_numpy(ids).to(dev), E, check=True)
