"""Stage 1 of long streams (`dispatch_block_kernel`: four tokens per workgroup, keys counted by destination in bytes) against a
stable sort, at the numbers of tokens, entries and ranks where it begins and ends."""
import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, MoEConfig

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check(W, E, K, H, T, indices):
    cfg = MoEConfig(E, K, H, T, torch.bfloat16, torch.bfloat16)
    a = HIPAllToAll(cfg, W - 1, W, device=DEV)
    x = torch.randint(-30000, 30000, (T, H), dtype=torch.int16, generator=torch.Generator().manual_seed(T)).view(torch.bfloat16)
    counts, buf, meta = a.dispatch_send(x.to(DEV), torch.from_numpy(indices).to(DEV))
    e = indices.reshape(-1).astype(np.int64)
    dest = np.where((e >= 0) & (e < E), e // (E // W), W)  # (an id that names no expert comes last)
    order = np.argsort(dest, kind="stable")
    token = order // K
    want = np.stack([e[order], np.full_like(order, W - 1), token, order % K, np.zeros_like(order)], 1)
    assert np.array_equal(counts.cpu().numpy(), np.bincount(dest, minlength=W + 1)[:W])
    assert np.array_equal(meta[:T * K].cpu().numpy(), want)
    assert torch.equal(buf[:T * K].cpu().view(torch.int16), x.view(torch.int16)[torch.from_numpy(token)])


@pytest.mark.parametrize("W,E,K,H,T", [
    (8, 16, 1, 8, 1281), (1, 3, 3, 24, 427), (8, 64, 4, 64, 257), (3, 15, 5, 1032, 410), (2, 6, 16, 37, 66), (8, 256, 8, 520, 1023),
    (7, 21, 6, 4104, 345), (8, 88, 2, 2048, 1601), (5, 10, 7, 7168, 1799), (8, 8, 8, 16, 4096), (4, 32, 4, 8, 16320), (4, 32, 4, 8, 16321),
    (9, 18, 4, 8, 400), (8, 32, 17, 8, 70)])  # (the last three are other kernels')
@pytest.mark.parametrize("ids", ["any", "one", "stray"])
def test_against_a_stable_sort(W, E, K, H, T, ids):
    print(f"block {W} {E} {K} {H} {T} {ids}", flush=True)
    rng = np.random.default_rng(T)
    indices = rng.integers(0, E, (T, K), dtype=np.int32)
    if ids == "one":  # every key of a lane counts in the same byte
        indices[:] = E - 1
    if ids == "stray":
        indices[rng.random((T, K)) < 0.2] = E + 3
        indices[rng.random((T, K)) < 0.2] = -5
    check(W, E, K, H, T, indices)
