"""The workgroup shapes of chunked prefill (chosen by the launch's size), each at its query and key tile
edges, and a mixed step's decode rows at the limits of their block-by-block form.  Against the oracle with
the tolerance of the prefill tests (2e-2 max-abs on bf16 outputs)."""

import pytest
import torch

from mini_infra_qwen3_amd import data_plane, workloads
from oracle import torch_ref

pytestmark = pytest.mark.gpu

TOL = 2e-2
SCALE = 128 ** -0.5


def _chunk_case(seed, starts, lens, kv_heads, group):
    gen = torch.Generator().manual_seed(seed)
    width, rows = max(lens), len(lens)
    totals = [s + n for s, n in zip(starts, lens)]
    num_blocks = 1 + sum(-(-t // 16) for t in totals)
    tables = workloads.permuted_tables(totals, num_blocks, gen)
    kp, vp = (torch.randn(num_blocks, 16, kv_heads, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(rows, group * kv_heads, width, 128, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn(rows, kv_heads, width, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
    hist = torch.zeros((rows, max(-(-s // 16) for s in starts)), dtype=torch.long)
    for b, s in enumerate(starts):
        hist[b, :-(-s // 16)] = torch.tensor(tables[b][:-(-s // 16)], dtype=torch.long)
    return q, k, v, kp, vp, hist


# The launch's size and the history's length decide (tests/test_prefill_routes.py holds the rule): narrow is 32
# queries with split keys, half split 64 with split keys, half 64, wide 128.
@pytest.mark.parametrize("starts,lens,kv_heads,group", [
    ([0], [1], 8, 2),                              # narrow: one query, one key, the second key half idle
    ([64, 0], [33, 32], 8, 2),                     # narrow: one past a 32-query tile
    ([129, 63, 1], [65, 64, 31], 8, 5),            # narrow: odd group, an odd number of key tiles
    ([0] * 15, [130 - i for i in range(15)], 4, 2),          # narrow, more workgroups than CUs
    ([0, 70] * 8, [129 + i for i in range(16)], 4, 2),       # half split
    ([17] * 31, [97 + i for i in range(31)], 8, 2),          # half
    ([0] * 11, [257 + i for i in range(11)], 8, 2),          # half
    ([0] * 64, [1 + i for i in range(64)], 8, 2),            # half
    ([0, 0], [600, 513], 8, 2),                              # narrow: eleven key tiles, the halves uneven
    ([600, 70], [513, 450], 8, 2),                           # half split: history as long as the chunk
    ([0, 65], [1100, 1025], 8, 2),                           # half split: long rows
    ([140] * 20, [128 - i for i in range(20)], 8, 2),        # wide: history as long as the chunk
    ([1] * 26, [256 - i for i in range(26)], 8, 2),          # wide
])
def test_shapes_match_oracle(native_lib, device, starts, lens, kv_heads, group):
    q, k, v, kp, vp, hist = _chunk_case(len(lens) + sum(lens), starts, lens, kv_heads, group)
    got = data_plane.chunked_prefill_attention(
        *(t.to(device) for t in (q, k, v, kp, vp, hist)), torch.tensor(starts, device=device),
        torch.tensor(lens, device=device), SCALE).float().cpu()
    ref = torch_ref.chunked_prefill_attention(q, k, v, (kp, vp), hist, starts, lens, SCALE).float()
    width = q.shape[2]
    for b, n in enumerate(lens):
        assert (got[b, width - n:] - ref[b, width - n:]).abs().max().item() <= TOL, f"row {b}"
        assert not got[b, :width - n].any(), f"row {b}: padding rows must be zero"


def _decode_rows(seed, contexts, max_blocks, group, kv_heads):
    gen = torch.Generator().manual_seed(seed)
    rows = len(contexts)
    num_blocks = 1 + rows * max(max_blocks, 1)
    kp, vp = (torch.randn(num_blocks, 16, kv_heads, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
    table = (torch.randperm(num_blocks - 1, generator=gen) + 1)[:rows * max_blocks].view(rows, max_blocks)
    q = torch.randn(rows, group * kv_heads, 128, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn(rows, kv_heads, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
    return q, k, v, kp, vp, table


# Tables of 511 blocks are the last attended block by block; contexts that end on a block, one past it, and
# past the table (the history is what the table holds, the token comes after it); no table at all.
@pytest.mark.parametrize("contexts,max_blocks", [
    ([1, 2, 16, 17, 128, 129, 0], 9),
    ([160, 161, 500], 10),
    ([8176, 8177, 9000, 8000], 511),
    ([8192, 8193, 100], 512),
    ([1, 0, 40], 0),
])
@pytest.mark.parametrize("group,kv_heads,exact", [(2, 8, False), (8, 4, False), (1, 2, False), (16, 1, False),
                                                  (2, 8, True), (8, 2, True), (5, 1, True)])
def test_decode_rows_of_a_mixed_step(native_lib, device, contexts, max_blocks, group, kv_heads, exact):
    q, k, v, kp, vp, table = _decode_rows(len(contexts) + max_blocks, contexts, max_blocks, group, kv_heads)
    rows = len(contexts)
    none = torch.zeros(0, dtype=torch.long, device=device)
    pools = kp.to(device), vp.to(device)
    out = data_plane.mixed_paged_attention(
        q.to(device), k.to(device), v.to(device), *pools, 0, 0, torch.zeros((0, 0), dtype=torch.long, device=device), none,
        none, table.to(device), torch.tensor(contexts).to(device), torch.full((rows,), -1).to(device), SCALE,
        exact=exact).float().cpu()
    assert torch.equal(pools[0].cpu(), kp) and torch.equal(pools[1].cpu(), vp)
    for b, n in enumerate(contexts):
        if n == 0:
            assert not out[b].any()
            continue
        nh = min(n - 1, 16 * max_blocks)
        keys = torch.cat((kp[table[b]].view(-1, kv_heads, 128)[:nh], k[b:b + 1]))
        values = torch.cat((vp[table[b]].view(-1, kv_heads, 128)[:nh], v[b:b + 1]))
        s = torch.einsum("hd,thd->ht", q[b].float(), keys.float().repeat_interleave(group, 1)).to(torch.bfloat16)
        p = (s * SCALE).to(torch.bfloat16).float().softmax(-1).to(torch.bfloat16)
        ref = torch.einsum("ht,thd->hd", p.float(), values.float().repeat_interleave(group, 1)).reshape(-1)
        assert (out[b] - ref).abs().max().item() <= TOL, f"row {b}"


def test_uncovered_tokens_of_many_rows(native_lib, device):
    """130 ragged rows (three reads of 64 by the zeroing workgroups) with a gap before each: zero rows there."""
    rows, kv_heads, heads = 130, 2, 4
    gen = torch.Generator().manual_seed(5)
    lens = torch.randint(0, 6, (rows,), generator=gen)
    gaps = torch.randint(0, 3, (rows,), generator=gen)
    first = torch.cumsum(lens + gaps, 0) - lens
    tokens = int(first[-1] + lens[-1]) + 3
    q = torch.randn(tokens, heads, 128, generator=gen).to(torch.bfloat16).to(device)
    k, v = (torch.randn(tokens, kv_heads, 128, generator=gen).to(torch.bfloat16).to(device) for _ in range(2))
    pool = torch.zeros(2, 16, kv_heads, 128, dtype=torch.bfloat16, device=device)
    none = torch.zeros(0, dtype=torch.long, device=device)
    covered = torch.zeros(tokens, dtype=torch.bool)
    for f, n in zip(first.tolist(), lens.tolist()):
        covered[f:f + n] = True
    for exact in (False, True):
        out = torch.full((tokens, heads * 128), float("nan"), dtype=torch.bfloat16, device=device)
        data_plane.mixed_paged_attention(
            q, k, v, pool.clone(), pool.clone(), rows, 6, torch.zeros((rows, 0), dtype=torch.long, device=device),
            torch.zeros(rows, dtype=torch.long, device=device), lens.to(device),
            torch.zeros((0, 1), dtype=torch.long, device=device), none, none, SCALE, out=out, exact=exact,
            chunk_first=first.to(device), chunk_tokens=tokens)
        out = out.cpu()
        assert (out[~covered] == 0).all()
        assert (out[covered].float().abs().sum(1) > 0).all() and torch.isfinite(out[covered].float()).all()


@pytest.mark.parametrize("starts,lens", [([0], [300]), ([700, 513], [513, 600]), ([0, 0], [1100, 1025])])
@pytest.mark.parametrize("max_blocks", [40, 8192, 8193])
def test_chunk_rows_of_a_mixed_step_have_the_bits_of_a_prefill(native_lib, device, starts, lens, max_blocks):
    """Whatever shape the chunk rows take, and however wide the decode rows' table is beside them (8193 blocks no
    longer fit the split shapes' LDS)."""
    q, k, v, kp, vp, hist = _chunk_case(sum(lens), starts, lens, 8, 2)
    rows, width = len(lens), max(lens)
    gen = torch.Generator().manual_seed(max_blocks)
    dec = 3
    dq, dk, dv = (torch.randn(dec, h, 128, generator=gen).to(torch.bfloat16) for h in (16, 8, 8))
    table = torch.randint(1, kp.shape[0], (dec, max_blocks), generator=gen)
    flat = [torch.cat((t.transpose(1, 2).reshape(rows * width, t.shape[1], 128), d)).to(device)
            for t, d in ((q, dq), (k, dk), (v, dv))]
    kp, vp, hist = kp.to(device), vp.to(device), hist.to(device)
    starts, lens = torch.tensor(starts, device=device), torch.tensor(lens, device=device)
    want = data_plane.chunked_prefill_attention(q.to(device), k.to(device), v.to(device), kp, vp, hist, starts, lens, SCALE)
    got = data_plane.mixed_paged_attention(
        *flat, kp, vp, rows, width, hist, starts, lens, table.to(device), torch.tensor([33, 1, 600]).to(device),
        torch.full((dec,), -1).to(device), SCALE)
    assert torch.equal(got[:rows * width].view(torch.int16), want.view(rows * width, -1).view(torch.int16))
    # The decode rows against the same rows beside a table that holds their contexts and no more.
    alone = data_plane.mixed_paged_attention(
        *(t[rows * width:] for t in flat), kp, vp, 0, 0, hist[:0], starts[:0], lens[:0], table[:, :40].to(device),
        torch.tensor([33, 1, 600]).to(device), torch.full((dec,), -1).to(device), SCALE)
    assert (got[rows * width:].float() - alone.float()).abs().max().item() <= TOL


@pytest.mark.parametrize("max_blocks", [5, 512])
@pytest.mark.parametrize("group,kv_heads,exact", [(2, 8, False), (8, 2, False), (2, 8, True), (5, 1, True)])
def test_decode_rows_of_a_mixed_step_do_not_see_what_lies_past_their_history(native_lib, device, max_blocks, group, kv_heads,
                                                                             exact):
    """NaN in every pool row that no history holds: the rest of a block just handed out (histories that end on a
    block), and the table's end (the token comes after the 80 positions it holds)."""
    contexts = [1, 17, 33, 65, 81, 100, 2, 48] if max_blocks == 5 else [1, 17, 4097, 8177]
    q, k, v, kp, vp, table = _decode_rows(7, contexts, max_blocks, group, kv_heads)
    rows = len(contexts)
    clean_k, clean_v = kp.clone(), vp.clone()
    kp.fill_(float("nan")), vp.fill_(float("nan"))
    for b, n in enumerate(contexts):
        nh = min(n - 1, 16 * max_blocks)
        for pool, clean in ((kp, clean_k), (vp, clean_v)):
            pool.view(-1, kv_heads, 128)[(table[b, :, None] * 16 + torch.arange(16)).view(-1)[:nh]] = \
                clean.view(-1, kv_heads, 128)[(table[b, :, None] * 16 + torch.arange(16)).view(-1)[:nh]]
    ends = [b for b, n in enumerate(contexts) if min(n - 1, 16 * max_blocks) % 16 == 0]
    none = torch.zeros(0, dtype=torch.long, device=device)
    outs = []
    for pools in ((kp, vp), (clean_k, clean_v)):
        outs.append(data_plane.mixed_paged_attention(
            q.to(device), k.to(device), v.to(device), pools[0].to(device), pools[1].to(device), 0, 0,
            torch.zeros((0, 0), dtype=torch.long, device=device), none, none, table.to(device),
            torch.tensor(contexts).to(device), torch.full((rows,), -1).to(device), SCALE, exact=exact).cpu())
    assert len(ends) >= 4 and torch.equal(outs[0][ends], outs[1][ends])
