"""Stage 4 of more tokens than units (`combine_recv_block_kernel`): tokens that share a workgroup, streams read in one batch and in several,
rows that end in a piece, and what a caller-made stream may hold: pairs that repeat, tokens and entries out of range, rows past the counts."""
import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll
from amd_distributed_2025_amd.task import MoEConfig
from oracle import moe_a2a_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
# (257 tokens in pairs; 767 / 768: fours for 256 workgroups, pairs for 512; 8193: 17 and a last one; more rows than a first batch of 4096)
@pytest.mark.parametrize("T,K,H,W", [(257, 8, 512, 3), (300, 3, 8, 1), (767, 2, 520, 2), (768, 1, 1032, 8), (769, 6, 2056, 4), (1700, 5, 16, 70),
                                     (8193, 1, 264, 2)])
def test_streams_of_every_kind(T, K, H, W, dtype):
    print(f"combine block T={T} K={K} H={H} W={W} {dtype}", flush=True)
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    cfg = MoEConfig(W * 8, K, H, T, dt, dt)
    a = HIPAllToAll(cfg, 0, W, device=DEV)
    rng = np.random.default_rng(T + K)
    S = T * K
    order = rng.permutation(S)
    whole = np.zeros((S, 5), np.int32)
    whole[:, 2], whole[:, 3] = order // K, order % K
    weights = torch.from_numpy(rng.random((T, K), dtype=np.float32))
    for kind in ("whole", "few", "repeats", "one token", "stray"):
        meta = whole.copy()
        R = S
        if kind == "few":  # (most tokens get nothing; what lies past the counts is not read as rows)
            R = S // 5
        elif kind == "repeats":
            meta[rng.integers(0, S, S // 3)] = meta[rng.integers(0, S, S // 3)]
        elif kind == "one token":
            meta[:40, 2], meta[:40, 3] = T - 1, 0
        elif kind == "stray":
            hit = rng.random(S) < 0.2
            meta[hit, 2] = rng.choice(np.array([-1, T, T + 5, 2**31 - 1, -2**31], np.int64), hit.sum()).astype(np.int32)
            meta[::7, 3] = rng.choice(np.array([-1, K, 9, 2**31 - 1]), len(meta[::7])).astype(np.int32)
        rows = torch.from_numpy(rng.standard_normal((S, H)).astype(np.float32)).to(dt)
        counts = np.diff(np.sort(np.concatenate([[0, R], rng.integers(0, R + 1, W - 1)]))).astype(np.int32)
        start = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(dt)
        args = (weights.to(DEV), torch.from_numpy(counts).to(DEV), rows.to(DEV), torch.from_numpy(meta).to(DEV))
        ok = np.arange(S) < R
        ok &= (meta[:, 2] >= 0) & (meta[:, 2] < T) & (meta[:, 3] >= 0) & (meta[:, 3] < K)
        for accumulate in (False, True):
            y = start.to(DEV) if accumulate else torch.empty(T, H, dtype=dt, device=DEV)
            a.combine_recv(y, *args, accumulate=accumulate, unique_pairs=False)
            want = orc.combine_recv(bits(rows)[ok], meta[ok], weights.numpy(), T, dtype, bits(start) if accumulate else None)
            assert np.array_equal(bits(y), want), (kind, accumulate)


def test_rows_beyond_the_caller_s_row_count():
    """The row count is a hint: a stream of more rows than it says is added up in full."""
    T, K, H, W = 600, 4, 136, 2
    rng = np.random.default_rng(3)
    S = T * K
    meta = np.zeros((S, 5), np.int32)
    order = rng.permutation(S)
    meta[:, 2], meta[:, 3] = order // K, order % K
    rows = torch.from_numpy(rng.standard_normal((S, H)).astype(np.float32)).bfloat16()
    weights = torch.from_numpy(rng.random((T, K), dtype=np.float32))
    want = orc.combine_recv(bits(rows), meta, weights.numpy(), T, "bf16")
    dev = [t.to(DEV) for t in (rows, torch.from_numpy(meta), torch.tensor([S - 100, 100], dtype=torch.int32), weights)]
    a = HIPAllToAll(MoEConfig(16, K, H, T, torch.bfloat16, torch.bfloat16), 0, W, device=DEV)
    for hint in (513, 700, S):
        y = torch.empty(T, H, dtype=torch.bfloat16, device=DEV)
        a.binding.combine_recv(a.shape, dev[0], dev[1], dev[2], hint, dev[3], T, y, False, torch.cuda.current_stream().cuda_stream, None)
        torch.cuda.synchronize()
        assert np.array_equal(bits(y), want), hint
