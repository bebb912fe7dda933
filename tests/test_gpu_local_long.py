"""The way out of one-GPU jobs whose movers rank their own entries (`local_dispatch_long_kernel`): tokens that share a workgroup, the last one
with fewer, ranks that begin inside one, rows that end in a piece. Every bit has to be what the stages with an exchange between them give."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, custom_kernel_job
from tests.test_gpu_local import DEV, config, rank_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spoil", [None, "ids", "twins"])
@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("E,K,H,T", [
    (16, 8, 8, 257),          # 2056 entries: two tokens for each workgroup, one for the last
    (7, 3, 520, 1000),        # one vector past a piece
    (512, 8, 1032, 300), (513, 8, 1032, 300),  # the most experts, and one more (a plan)
    (5, 1, 2056, 2049), (64, 64, 136, 40),     # one entry and 64 per token
    (12, 8, 24, 4096), (12, 8, 24, 4097),      # the most entries, and more (a plan)
    (6, 5, 4104, 3300),       # 135 MB: four vectors per lane
])
def test_one_rank(E, K, H, T, layout, spoil):
    print(f"local long E={E} K={K} H={H} T={T} {layout} {spoil}", flush=True)
    if K > E and spoil is None:
        pytest.skip("distinct experts")
    cfg = config(E, K, H, T)
    d = rank_data(cfg, T, 5 + K, spoil)
    got = []
    for reuse in (True, False):
        a = HIPAllToAll(cfg, 0, 1, device=DEV, layout=layout, reuse_placement=reuse)
        rows = (a.compact_rows,) if layout == "compact" else (E, a.max_recv)
        a._buf("expert_x", rows + (H,), cfg.in_dtype).fill_(77)  # rows that nothing fills stay as they are
        a._buf("expert_meta", rows + (5,), torch.int32).fill_(77)
        num, ex, em = a.dispatch(d.x, d.indices)
        y = torch.ones(T, H, dtype=cfg.out_dtype, device=DEV)
        a.combine(y, d.weights, em, a.expert_scale(ex, num), num)
        torch.cuda.synchronize()
        got.append((num, ex, em, y, a.expert_offsets))
    for what, p, q in zip(("counts", "rows", "meta", "result", "offsets"), *got):
        assert (p is None and q is None) or torch.equal(p, q), what


@pytest.mark.parametrize("din,dout", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.float16, torch.bfloat16),
                                      (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("W,E,K,H,tokens", [(8, 64, 8, 264, [40, 1, 0, 77, 33, 60, 31, 90]), (3, 9, 3, 1032, [700, 5, 333]), (2, 2, 1, 64, [1500, 1200])])
def test_jobs(W, E, K, H, tokens, din, dout):
    print(f"local long job W={W} {din} {dout}", flush=True)
    cfg = config(E, K, H, max(tokens), din, dout)
    for spoil in (None, "ids"):
        data = [rank_data(cfg, t, 3 * r + K, spoil) for r, t in enumerate(tokens)]
        want = [y.clone() for y in LocalWorld(cfg, W, device=DEV).run(data)]
        ys = custom_kernel_job([(cfg, d, r, W) for r, d in enumerate(data)])
        for r in range(W):
            assert torch.equal(ys[r], want[r]), (spoil, r)
