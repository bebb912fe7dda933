"""The way back of jobs whose ranks share the GPU, whose kernels are made for up to 2, 4, 6 and 8 entries per token, and for results that go
past the caches. Every bit has to be what the stages with an exchange between them give (which other files check against the oracle)."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, custom_kernel_job
from tests.test_gpu_local import DEV, config, rank_data

pytestmark = pytest.mark.gpu
STREAM_BYTES, RANKS_STREAM_BYTES = 80 << 20, 128 << 20  # of rows and results (JOB_STREAM_BYTES, JOB_RANKS_STREAM_BYTES)


def check_job(W, E, K, H, tokens, spoil, dtype):
    print(f"addends W={W} E={E} K={K} H={H} {tokens[:3]} {spoil} {dtype}", flush=True)
    cfg = config(E, K, H, max(tokens), dtype, dtype)
    data = [rank_data(cfg, t, 31 * r + K, spoil) for r, t in enumerate(tokens)]
    want = [y.clone() for y in LocalWorld(cfg, W, device=DEV).run(data)]
    ys = custom_kernel_job([(cfg, d, r, W) for r, d in enumerate(data)])
    for r in range(W):
        assert torch.equal(ys[r], want[r]), f"rank {r}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H", [512, 2568, 4104])  # less than a chunk, two vectors per lane, more chunks
@pytest.mark.parametrize("K", range(1, 10))
def test_every_number_of_entries(K, H, dtype):
    check_job(2, 18, K, H, [33, 7], "ids", dtype)       # (entries without a row)
    check_job(9, 18, K, H, [5, 0, 1, 9, 2, 3, 1, 1, 4], None, dtype)


@pytest.mark.parametrize("W,K,H", [(1, 1, 4096), (1, 3, 2568), (2, 6, 5128), (9, 8, 7168), (1, 9, 2048)])
def test_results_past_the_caches(W, K, H):
    tokens = -(-(STREAM_BYTES if W == 1 else RANKS_STREAM_BYTES) // ((K + 1) * H * 2 * W))
    check_job(W, 18, K, H, [tokens] * W, None, torch.bfloat16)


@pytest.mark.parametrize("K", [2, 4, 6, 8])
def test_results_past_the_caches_are_added(K):
    """`combine` adds to what is there; dispatch, expert and combine of one rank against the halves."""
    H = 3080
    cfg = config(12, K, H, -(-STREAM_BYTES // ((K + 1) * H * 2)))
    d = rank_data(cfg, cfg.max_num_tokens, K, "ids")
    got = []
    for reuse in (True, False):
        a = HIPAllToAll(cfg, 0, 1, device=DEV, reuse_placement=reuse)
        num, ex, em = a.dispatch(d.x, d.indices)
        y = torch.randn(cfg.max_num_tokens, H, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(cfg.out_dtype)
        a.combine(y, d.weights, em, a.expert_scale(ex, num), num)
        got.append(y)
    assert torch.equal(*got)
