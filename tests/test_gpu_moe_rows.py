"""GPU parity of the row-block MoE GEMM (at most one routed row per expert on average) against the CPU oracle.

Bar: the oracle rounds the same weights and accumulates in fp32, so a result may differ where another
summation order flips a rounding to the output type: plain outputs pass one rounding, gated ones three
(gate, up, product; |d silu/dg| <= 1.1), each by at most one unit eps of the value: 4 eps * max|ref| in all.
"""

import pytest
import torch

from oracle import awq_oracle as oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
EPS = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}

CASES = [  # (T, E, k, K, N, G, block size, routing)
    (1, 8, 8, 256, 128, 128, 16, "spread"),     # one row per expert, as many blocks as experts
    (1, 6, 1, 128, 96, 128, 16, "spread"),      # one k-tile for four waves
    (3, 130, 4, 352, 96, 32, 16, "spread"),     # eight experts a lane, four groups a k-tile, K % 128 != 0
    (9, 70, 6, 640, 64, 64, 16, "dropped"),     # two groups a k-tile, two waves, ids of -1
    (5, 48, 2, 384, 160, -1, 16, "spread"),     # one group, K of three k-tiles
    (4, 12, 3, 256, 200, 128, 16, "spread"),    # n == E; N % 16 == 8 (plain only)
    (40, 40, 1, 256, 64, 128, 16, "one"),       # all rows on one expert: three blocks, the last of 8 rows
    (24, 26, 1, 256, 64, 128, 64, "two"),       # buckets of 64: blocks of padding alone
    (2, 512, 4, 256, 64, 128, 16, "last"),      # the last expert
    (1, 4, 1, 256, 64, 128, 1024, "spread"),    # 63 blocks of padding behind one row, one workgroup per column group
    (5, 130, 7, 256, 64, 128, 256, "spread"),   # padding blocks dealt to every workgroup
    (6, 136, 20, 256, 96, 64, 16, "last"),      # eight experts a lane as vectors, the last lanes without any
    (2, 128, 8, 256, 1024, 32, 16, "spread"),   # short K: below the row-block form's line, ...
    (8, 128, 8, 256, 1024, 32, 16, "spread"),   # ... and above it: the pipelined form
]


@pytest.mark.parametrize("T,E,k,K,N,G,bs,routing", CASES)
@pytest.mark.parametrize("activation,mul", [(None, True), (None, False), ("silu", False), ("gelu", True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_row_blocks_match_oracle(T, E, k, K, N, G, bs, routing, activation, mul, dtype):
    if activation and N % 32:
        pytest.skip("gate/up pairing needs I % 16 == 0")
    from sglite_amd import ops

    assert T * k <= E
    gen = torch.Generator().manual_seed(T * E + K)
    ids = torch.stack([torch.randperm(E, generator=gen)[:k] for _ in range(T)]).to(torch.int32)
    if routing == "dropped":
        ids[::3, 0] = -1
    elif routing == "one":
        ids[:] = E // 2
    elif routing == "two":
        ids[:] = torch.arange(T).remainder(2).mul(E - 1).view(T, 1).to(torch.int32)
    elif routing == "last":
        ids[:, 0] = E - 1
    tw = torch.rand((T, k), generator=gen)
    used = sorted(set(ids.reshape(-1).tolist()) - {-1})
    one = {e: oracle.make_awq_linear(K, N, G, seed=e, dtype=dtype) for e in used}
    blank = {key: torch.zeros_like(v) for key, v in one[used[0]].items()}
    W = {key: torch.stack([one.get(e, blank)[key] for e in range(E)]) for key in ("qweight", "qzeros", "scales")}
    x = oracle.make_activation(T, K, seed=T + K).to(dtype)
    ref = oracle.moe_grouped_gemm(x, W, tw, ids, k, G, activation, mul)
    ex = ops.repack_experts(*(W[key].to(DEV) for key in ("qweight", "qzeros", "scales")))
    align = ops.moe_align_block_size(ids.to(DEV), bs, E)
    out = ops.moe_gemm(x.to(DEV), ex, K, N, G, align, tw.to(DEV), T * k, k, activation, mul).cpu()
    valid = ids.reshape(-1) >= 0
    err = (out[valid].float() - ref[valid].float()).abs().max().item()
    assert err <= 4 * EPS[dtype] * ref[valid].float().abs().max().item()


@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (1, 64, 8), (15, 200, 6), (16, 65, 4), (16, 512, 64), (17, 128, 8),
                                   (200, 60, 4)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("renorm", [True, False])
def test_route_matches_its_two_stages(T, E, k, dtype, renorm):
    """One launch or two, 16-bit logits or fp32: the ids, weights and layout of the separate entry points."""
    from sglite_amd import ops

    logits = torch.randn((T, E), generator=torch.Generator().manual_seed(T * E + k)).to(dtype).to(DEV)
    w, ids, align = ops.moe_route(logits, k, renorm, 16)
    rw, rids = ops.moe_topk_softmax(logits.float(), k, renorm)
    ref = ops.moe_align_block_size(rids, 16, E)
    assert torch.equal(w, rw) and torch.equal(ids, rids)
    total = int(ref.num_tokens_post_pad.item())
    assert torch.equal(align.sorted_ids[:total], ref.sorted_ids[:total])
    for got, want in zip(align[1:], ref[1:]):
        assert torch.equal(got, want)
