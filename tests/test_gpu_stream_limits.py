"""Stages 1, 2 and 4 of long streams, and jobs on one GPU, at the limits of the kernels that run there by now (`csrc/stream_rules.h`;
test_long_stream_rules.py holds the sizes to the kernels that they are meant for)."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, _binding
from amd_distributed_2025_amd.task import MoEConfig
from tests import test_gpu_block_streams as block_streams
from tests import test_gpu_combine_block as combine_block
from tests import test_gpu_large_streams as large_streams
from tests import test_gpu_local_long as local_long
from tests.test_gpu_parity import DEV

pytestmark = pytest.mark.gpu

# ranks, experts, entries per token, hidden, tokens -> tokens of a workgroup of dispatch_long_kernel, or what else runs
SEND_CASES = {
    (8, 256, 8, 520, 1023): 4, (4, 8, 4, 4104, 1601): 4, (8, 8, 8, 16, 4096): 8, (4, 32, 4, 8, 16320): 16,
    (4, 32, 4, 8, 16321): 16, (4, 32, 4, 8, 65280): 16, (4, 32, 4, 8, 65281): "fanout",  # the most keys that 1024 lanes count in bytes, and more
    (4, 32, 4, 3, 16320): "block", (4, 32, 4, 3, 16321): "fanout",  # that 256 lanes count (rows of elements), and more
    (8, 256, 8, 520, 639): "block", (4, 8, 3, 6144, 1650): "block",
    (4, 256, 64, 16, 1021): 1, (8, 40, 20, 64, 3300): 3, (8, 16, 16, 1032, 4090): 4,  # many entries per token
    (4, 16, 8, 728, 2235): "block", (8, 64, 6, 1456, 2637): 10, (8, 8, 4, 4608, 3500): 4,
}
# the same, of skewed routing
LONG_CASES = {
    (8, 16, 1, 8, 5120): 20, (3, 15, 5, 520, 1024): 4, (2, 6, 6, 1032, 2561): 10, (8, 8, 7, 64, 2311): 9, (5, 20, 3, 3208, 1800): 4,
    (2, 4, 2, 8, 32641): 32, (1, 2, 1, 7168, 5121): 11,  # (these are test_gpu_large_streams.py's)
    (4, 256, 64, 16, 1021): 1, (4, 8, 4, 4104, 2000): 2,
}
# tokens, entries per token, hidden, ranks -> tokens of a workgroup of combine_recv_block_kernel
COMBINE_CASES = {(257, 8, 512, 3): 2, (300, 3, 8, 1): 2, (767, 2, 520, 2): 3, (768, 1, 1032, 8): 2, (769, 6, 2056, 4): 2, (1700, 5, 16, 70): 4,
                 (8193, 1, 264, 2): 17, (33000, 1, 16, 2): 64}
# experts, entries per token, hidden, tokens -> tokens of a workgroup of local_dispatch_long_kernel (0: a plan) and vectors per lane
LOCAL_CASES = {
    (16, 8, 8, 257): (2, 1), (7, 3, 520, 1000): (4, 2), (512, 8, 1032, 300): (2, 2), (513, 8, 1032, 300): (0, 2), (5, 1, 2056, 2049): (9, 2),
    (64, 64, 136, 40): (1, 1), (12, 8, 24, 4096): (16, 1), (12, 8, 24, 4097): (0, 1), (6, 5, 4104, 3300): (13, 4),
    (3, 2, 1032, 1200): (5, 2), (1, 1, 24, 32768): (128, 1), (64, 64, 24, 512): (2, 1),  # one vector past a piece; the most entries, of one a token and of 64
}


@pytest.mark.parametrize("W,E,K,H,T", SEND_CASES)
@pytest.mark.parametrize("ids", ["any", "one", "stray"])
def test_stage_1_against_a_stable_sort(W, E, K, H, T, ids):
    block_streams.test_against_a_stable_sort(W, E, K, H, T, ids)


@pytest.mark.parametrize("W,E,K,H,T", [(4, 256, 64, 16, 1021), (4, 8, 4, 4104, 2000)])
def test_stage_1_of_skewed_streams(W, E, K, H, T):
    large_streams.test_stage_one_of_long_streams(W, E, K, H, T)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_64_tokens_of_a_workgroup_of_stage_4(dtype):
    combine_block.test_streams_of_every_kind(33000, 1, 16, 2, dtype)


@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("E,K,H,T", [(3, 2, 1032, 1200), (1, 1, 24, 32768), (64, 64, 24, 512)])
def test_jobs_of_one_rank(E, K, H, T, layout):
    for spoil in (None, "ids", "twins"):
        local_long.test_one_rank(E, K, H, T, layout, spoil)


def test_planned_places_of_a_shape_that_could_hold_far_more():
    """128 experts that could each take 1.2 million rows, of which 4100 arrive: more than the experts' pieces could be numbered."""
    W, nle, H, R = 8, 128, 7168, 4100
    a = HIPAllToAll(MoEConfig(W * nle, 1, H, 150000, torch.bfloat16, torch.bfloat16), 3, W, device=DEV, layout="compact", compact_rows=4200)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1)
    recv = torch.randn(R, H, device=DEV, generator=gen).to(torch.bfloat16)
    meta = torch.randint(0, 1000, (R, 5), device=DEV, generator=gen, dtype=torch.int32)
    meta[:, 0] = 3 * nle + torch.randint(0, nle, (R,), device=DEV, generator=gen, dtype=torch.int32)
    counts = torch.tensor([R - 70] + [10] * 7, dtype=torch.int32, device=DEV)
    num, ex, em = a.dispatch_recv(counts, recv, meta, R)
    torch.cuda.synchronize()
    order = torch.argsort(meta[:, 0], stable=True)
    assert torch.equal(ex[:R], recv[order]) and torch.equal(em[:R], meta[order])
    want = torch.bincount(meta[:, 0] - 3 * nle, minlength=nle)
    assert torch.equal(num.long(), want) and torch.equal(a.expert_offsets[1:].long(), want.cumsum(0))


@pytest.mark.parametrize("rows", [40, 4096, 5000])
def test_a_binding_whose_compact_call_takes_no_places(rows):
    class Own(_binding.CtypesBinding):
        def dispatch_recv_compact(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens, expert_offsets, expert_x,
                                  expert_meta, send_back_plan, stream):
            calls.append(rows_hint)
            super().dispatch_recv_compact(shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens, expert_offsets, expert_x,
                                          expert_meta, send_back_plan, stream)

    calls, got = [], []
    for own in (True, False):
        a = HIPAllToAll(MoEConfig(6, 1, 64, 5000, torch.bfloat16, torch.bfloat16), 0, 2, device=DEV, layout="compact")
        if own:
            a.binding = Own()
        gen = torch.Generator(device=DEV)
        gen.manual_seed(rows)
        recv = torch.randn(rows, 64, device=DEV, generator=gen).to(torch.bfloat16)
        meta = torch.randint(0, 3, (rows, 5), device=DEV, generator=gen, dtype=torch.int32)
        counts = torch.tensor([rows - 9, 9], dtype=torch.int32, device=DEV)
        num, ex, em = a.dispatch_recv(counts, recv, meta, rows)
        got.append((num, a.expert_offsets, ex[:rows], em[:rows]))
    torch.cuda.synchronize()
    assert calls == [rows]
    assert all(torch.equal(p, q) for p, q in zip(*got))


# hidden, rows -> vectors per lane; more than the 40 MB from which stage 2 reads rows past the caches
RECV_PAST_CASES = {(1032, 20500): 1, (2048, 10300): 1, (2056, 10300): 2, (7168, 3000): 2, (7168, 21200): 1}


@pytest.mark.parametrize("hidden_dim,rows", RECV_PAST_CASES)
@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("plan", [True, False])
def test_stage_2_of_large_streams(hidden_dim, rows, layout, plan):
    print(f"stage 2, {rows} rows of {hidden_dim}, {layout}, plan {plan}", flush=True)
    W, nle = 2, 3
    a = HIPAllToAll(MoEConfig(W * nle, 1, hidden_dim, rows, torch.bfloat16, torch.bfloat16), 1, W, device=DEV, reuse_placement=plan,
                    layout=layout, compact_rows=rows + 5 if layout == "compact" else None)
    a.long_stream_rows = 0
    gen = torch.Generator(device=DEV)
    gen.manual_seed(rows)
    recv = torch.randint(-30000, 30000, (rows + 9, hidden_dim), device=DEV, generator=gen, dtype=torch.int16).view(torch.bfloat16)
    meta = torch.randint(0, 1000, (rows + 9, 5), device=DEV, generator=gen, dtype=torch.int32)
    meta[:, 0] = nle + torch.randint(0, nle, (rows + 9,), device=DEV, generator=gen, dtype=torch.int32)
    counts = torch.tensor([rows - 700, 700], dtype=torch.int32, device=DEV)  # (nine rows more than arrived lie in the buffers)
    num, ex, em = a.dispatch_recv(counts, recv, meta, rows)
    torch.cuda.synchronize()
    le = meta[:rows, 0] - nle
    assert torch.equal(num.long(), torch.bincount(le, minlength=nle))
    first = 0
    for e in range(nle):
        of, n = torch.nonzero(le == e).flatten(), int(num[e])
        got, got_meta = (ex[first:first + n], em[first:first + n]) if layout == "compact" else (ex[e, :n], em[e, :n])
        assert torch.equal(got.view(torch.int16), recv[of].view(torch.int16)) and torch.equal(got_meta, meta[of]), e
        first += n


# hidden, entries per token, tokens -> vectors per lane; rows and results of more than the 80 MB from which stage 4 reads past the caches
MAPPED_PAST_CASES = {(2048, 1, 10300): 2, (7168, 2, 2000): 2, (4104, 3, 2560): 2, (2056, 4, 4100): 2, (512, 4, 16500): 1, (3080, 6, 1950): 1,
                     (1032, 8, 4600): 1}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hidden_dim,K,tokens", MAPPED_PAST_CASES)
def test_stage_4_of_large_streams(hidden_dim, K, tokens, dtype):
    """With a table against the kernels that scan, which other files hold to the oracle. A third of the rows names other tokens' entries, and some lie past
    the counts."""
    print(f"stage 4, {tokens} tokens x {K} of {hidden_dim} {dtype}", flush=True)
    a = HIPAllToAll(MoEConfig(16, K, hidden_dim, tokens, dtype, dtype), 0, 2, device=DEV)
    a.long_stream_rows = 0
    gen = torch.Generator(device=DEV)
    gen.manual_seed(tokens)
    S = tokens * K
    order = torch.randperm(S, device=DEV, generator=gen)
    meta = torch.stack([order, order, order // K, order % K, order], 1).int()
    meta[::3, 2] += tokens
    rows = torch.randn(S, hidden_dim, device=DEV, generator=gen).to(dtype)
    weights = torch.rand(tokens, K, device=DEV, generator=gen)
    counts = torch.tensor([S - 900, 800], dtype=torch.int32, device=DEV)
    start = torch.randn(tokens, hidden_dim, device=DEV, generator=gen).to(dtype)
    for accumulate in (True, False):
        got = [start.clone() for _ in range(2)]
        for y, unique in zip(got, (True, False)):
            a.combine_recv(y, weights, counts, rows, meta, accumulate=accumulate, unique_pairs=unique)
        torch.cuda.synchronize()
        assert "entry_row" in a._ws and torch.equal(*[y.view(torch.int16) for y in got]), accumulate
