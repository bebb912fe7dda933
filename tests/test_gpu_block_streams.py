"""Stage 1 against a stable sort: `dispatch_block_kernel` (four tokens per workgroup, keys counted by destination in bytes) on every
cut of a row, and the numbers of tokens, entries, ranks and row lengths where it and the kernels of short streams begin and end."""
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


# ranks, experts, entries per token, hidden, tokens -> the kernel, and for dispatch_block_kernel vectors per lane and pieces of a
# row (csrc/stream_rules.h; test_stream_rules.py holds the cases to that)
CASES = {
    (8, 16, 1, 8, 1281): ("block", 1, 1), (1, 3, 3, 24, 427): ("block", 1, 1), (8, 64, 4, 64, 257): ("block", 1, 1),
    (2, 2, 1, 1000, 1282): ("block", 2, 1), (8, 256, 8, 520, 1023): ("block", 2, 1), (3, 15, 5, 1032, 410): ("block", 2, 2),
    (5, 10, 3, 4104, 700): ("block", 2, 5), (4, 4, 1, 1032, 1290): ("block", 4, 1), (8, 88, 2, 2048, 1601): ("block", 4, 1),
    (4, 8, 4, 4104, 1601): ("block", 4, 3), (8, 16, 2, 7168, 1605): ("block", 4, 4), (2, 4, 1, 2056, 3001): ("block", 6, 1),
    (8, 8, 1, 4096, 3007): ("block", 8, 1), (3, 3, 1, 6144, 1285): ("block", 12, 1), (2, 4, 1, 7168, 1301): ("block", 14, 1),
    (2, 2, 1, 8192, 1283): ("block", 16, 1), (2, 2, 1, 8200, 1282): ("block", 16, 2),
    (2, 6, 16, 37, 66): ("block", 16, 1), (4, 8, 5, 2051, 300): ("block", 16, 3), (2, 4, 1, 3001, 2710): ("block", 16, 3),  # single elements
    (8, 16, 2, 2560, 700): ("block", 6, 1), (4, 8, 2, 4096, 661): ("block", 8, 1), (2, 4, 2, 7168, 650): ("block", 4, 4),
    (8, 16, 3, 3072, 501): ("block", 6, 1), (8, 8, 8, 16, 4096): ("block", 1, 1), (4, 32, 4, 8, 16320): ("block", 1, 1),
    (4, 32, 4, 8, 16321): "fanout", (9, 18, 4, 8, 400): "fanout", (8, 32, 17, 8, 70): "fanout",
    (7, 21, 6, 4104, 345): "wide fanout", (5, 10, 7, 7168, 1799): "wide fanout", (9, 18, 2, 24, 700): "by entry",
    # two and eight entries ranked per pass, in one, two and nine passes, ids in registers and past them
    (9, 36, 11, 2056, 400): "wide fanout", (9, 36, 11, 4104, 130): "wide fanout", (9, 18, 6, 2056, 700): "wide fanout",
    (9, 90, 70, 4104, 60): "wide fanout", (9, 90, 70, 2056, 20): "wide fanout", (9, 36, 11, 520, 400): "fanout", (9, 90, 70, 24, 20): "fanout",
    (4, 8, 1, 7167, 100): "few", (4, 8, 1, 7167, 300): "by entry", (8, 16, 4, 4097, 60): "few", (8, 16, 4, 4097, 100): "by entry",
    (16, 32, 8, 2049, 120): "by entry", (8, 64, 1, 7168, 500): "few", (2, 4, 1, 2304, 728): "by entry",
    (8, 16, 4, 2304, 400): "wide fanout", (4, 16, 8, 4096, 520): "wide fanout", (8, 16, 8, 4096, 400): ("block", 2, 4),
    (8, 16, 1, 2304, 3000): "by entry", (2, 4, 1, 5120, 1281): "by entry", (8, 16, 1, 72, 2049): "by entry", (8, 16, 1, 517, 2700): "by entry"}


@pytest.mark.parametrize("W,E,K,H,T", CASES)
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
