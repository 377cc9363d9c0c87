"""The per-sequence decode kernels (stripes, spread stripes, parts): tables at the length where sequences start to be cut, contexts
that end inside, at and past part boundaries, and the fused prologue with the new token's slot in the
first, a middle and the last part.  Fused against the two entry points it stands for, bit for bit (the
new rows are put in place in registers, not read back from the pool), and against the oracle with the
tolerance of the decode tests (2e-2 max-abs on bf16 outputs)."""

import pytest
import torch

from mini_infra_qwen3_amd import data_plane
from oracle import torch_ref

pytestmark = pytest.mark.gpu

TOL = 2e-2
SCALE = 128 ** -0.5


def _case(seed, ctx, width, group, kv_heads=8):
    gen = torch.Generator().manual_seed(seed)
    num_blocks = 1 + sum(-(-max(n, 1) // 16) for n in ctx) + 4
    tables = torch.zeros(len(ctx), width, dtype=torch.long)
    perm = torch.randperm(num_blocks - 1, generator=gen) + 1
    at = 0
    for b, n in enumerate(ctx):
        need = -(-max(n, 1) // 16)
        tables[b, :need] = perm[at:at + need]
        at += need
    kp = torch.randn(num_blocks, 16, kv_heads, 128, generator=gen).to(torch.bfloat16)
    vp = torch.randn(num_blocks, 16, kv_heads, 128, generator=gen).to(torch.bfloat16)
    heads = group * kv_heads
    qkv = torch.randn(len(ctx), (heads + 2 * kv_heads) * 128, generator=gen).to(torch.bfloat16)
    w = [(1 + 0.1 * torch.randn(128, generator=gen)).to(torch.bfloat16) for _ in range(2)]
    angle = torch.randn(len(ctx), 128, generator=gen)
    return kp, vp, tables, qkv, w, angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16)


# Widths 32 and 63: stripes in one workgroup, 64 to 128 spread, 129 on parts (72 with 64 rows too); 520 is past the
# per-sequence kernel.  Contexts: empty, one token, the edges of a 16-token block and of 8-block parts.
@pytest.mark.parametrize("width,ctx", [
    (32, [512, 511, 1, 0, 497]),
    (63, [1000, 3, 0]),
    (64, [1024, 1009, 0, 15]),
    (128, [2048, 1]),
    (129, [2064, 129, 128, 127, 0]),
    (33, [528, 513, 512, 129, 128, 127, 1, 0]),
    (72, [1150, 1025, 1024, 255, 256, 257, 17, 16, 15]),
    (72, [1 + 29 * i % 1150 for i in range(64)]),
    (512, [8192, 4097, 300]),
    (520, [8300, 40]),
])
@pytest.mark.parametrize("group", [1, 2, 8])
def test_fused_equals_the_two_entry_points(native_lib, device, width, ctx, group):
    kp, vp, tables, qkv, (qw, kw), cos, sin = _case(width + group, ctx, width, group)
    heads, kv = group * 8, 8
    slots = torch.tensor([int(tables[b, (n - 1) // 16]) * 16 + (n - 1) % 16 if n else -1 for b, n in enumerate(ctx)])
    # Up to two rows put their token elsewhere in their own blocks: in the first block, and in a middle one.
    slots[0] = int(tables[0, 0]) * 16 + 3
    if len(ctx) > 2 and ctx[2] > 40:
        slots[2] = int(tables[2, (ctx[2] - 1) // 32]) * 16 + 15
    dev = [t.to(device) for t in (kp, vp, tables, qkv, qw, kw, cos, sin, slots)]
    kp_d, vp_d, tables_d, qkv_d, qw_d, kw_d, cos_d, sin_d, slots_d = dev
    ctx_d = torch.tensor(ctx).to(device)
    q, k, v = qkv_d.split((heads * 128, kv * 128, kv * 128), dim=1)
    kp2, vp2 = kp_d.clone(), vp_d.clone()
    out = data_plane.paged_decode_attention_fused(q, k, v, qw_d, kw_d, cos_d, sin_d, 1e-6, slots_d, kp_d, vp_d, tables_d,
                                                  ctx_d, SCALE)
    q_rot, _, _ = data_plane.qk_norm_rope(q, k, v, qw_d, kw_d, cos_d, sin_d, 1e-6, slot_mapping=slots_d, key_pool=kp2,
                                          value_pool=vp2)
    want = data_plane.paged_decode_attention(q_rot.view(len(ctx), heads, 128), kp2, vp2, tables_d, ctx_d, SCALE)
    assert torch.equal(kp_d.view(torch.int16), kp2.view(torch.int16))
    assert torch.equal(vp_d.view(torch.int16), vp2.view(torch.int16))
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    ref = torch_ref.paged_decode_attention(q_rot.view(len(ctx), heads, 128).cpu(), kp2.cpu(), vp2.cpu(), tables,
                                           torch.tensor(ctx), SCALE)
    live = torch.tensor(ctx) > 0
    assert (out.float().cpu()[live] - ref.float().view(len(ctx), -1)[live]).abs().max().item() <= TOL
    assert not out.cpu()[~live].any()


def test_fused_takes_rows_of_any_alignment(native_lib, device):
    """Projection rows that start on a 2-byte boundary: the append and rotation run on their own."""
    ctx = [300, 17]
    kp, vp, tables, qkv, (qw, kw), cos, sin = _case(3, ctx, 72, 2)
    slots = torch.tensor([int(tables[b, (n - 1) // 16]) * 16 + (n - 1) % 16 for b, n in enumerate(ctx)]).to(device)
    kp, vp, tables, qkv, qw, kw, cos, sin = [t.to(device) for t in (kp, vp, tables, qkv, qw, kw, cos, sin)]
    odd = torch.zeros(2, qkv.shape[1] + 1, dtype=torch.bfloat16, device=device)
    odd[:, 1:] = qkv
    outs = []
    for rows in (qkv, odd[:, 1:]):
        q, k, v = rows.split((2048, 1024, 1024), dim=1)
        pools = kp.clone(), vp.clone()
        outs.append((data_plane.paged_decode_attention_fused(q, k, v, qw, kw, cos, sin, 1e-6, slots, *pools, tables,
                                                             torch.tensor(ctx).to(device), SCALE), *pools))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("rows,lo,hi", [(20, 40, 1100), (66, 1, 500), (40, 1000, 2500)])
def test_rows_that_share_a_sequence_see_each_others_token(native_lib, device, rows, lo, hi):
    """Each sequence as two rows, one token apart (the second row's context holds the first one's token), in
    launches of more (row, KV head) pairs than CUs: the append comes before every row's attention."""
    gen = torch.Generator().manual_seed(rows)
    ctx = torch.randint(lo, hi, (rows,), generator=gen).tolist()
    ctx = [n for m in ctx for n in (m, m + 1)]
    kp, vp, tables, qkv, (qw, kw), cos, sin = _case(rows, ctx, max(-(-n // 16) for n in ctx), 2)
    tables[0::2] = tables[1::2]  # one table per sequence
    slots = torch.tensor([int(tables[b, (n - 1) // 16]) * 16 + (n - 1) % 16 for b, n in enumerate(ctx)])
    kp, vp, tables, qkv, qw, kw, cos, sin, slots = [t.to(device) for t in (kp, vp, tables, qkv, qw, kw, cos, sin, slots)]
    ctx_d = torch.tensor(ctx).to(device)
    q, k, v = qkv.split((2048, 1024, 1024), dim=1)
    kp2, vp2 = kp.clone(), vp.clone()
    q_rot, _, _ = data_plane.qk_norm_rope(q, k, v, qw, kw, cos, sin, 1e-6, slot_mapping=slots, key_pool=kp2, value_pool=vp2)
    want = data_plane.paged_decode_attention(q_rot.view(2 * rows, 16, 128), kp2, vp2, tables, ctx_d, SCALE)
    out = data_plane.paged_decode_attention_fused(q, k, v, qw, kw, cos, sin, 1e-6, slots, kp, vp, tables, ctx_d, SCALE)
    assert torch.equal(kp.view(torch.int16), kp2.view(torch.int16)) and torch.equal(vp.view(torch.int16), vp2.view(torch.int16))
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("width,ctx", [(30, [480, 3, 0]), (72, [1150, 17, 600, 1]), (200, [3200, 129]), (512, [8192, 1, 0, 700])])
def test_small_launches_leave_the_callers_workspace_untouched(native_lib, device, width, ctx):
    """Through the C ABI with a filled workspace, and through the Python layer with the same one; spread, tables
    of up to 128 blocks have the same bits, longer ones agree within the tolerance."""
    kp, vp, tables, qkv, _, _, _ = _case(width, ctx, width, 2)
    q = qkv[:, :2048].reshape(len(ctx), 16, 128).contiguous().to(device)
    kp, vp, tables, ctx_d = kp.to(device), vp.to(device), tables.to(device), torch.tensor(ctx).to(device)
    need = native_lib.mi_paged_decode_workspace_bytes(len(ctx), width, 16, 8, 128, 16)
    ws = torch.full((need,), 171, dtype=torch.uint8, device=device)
    out = torch.empty((len(ctx), 2048), dtype=torch.bfloat16, device=device)
    rc = native_lib.mi_paged_decode_attention(
        out.data_ptr(), 2048, q.data_ptr(), 2048, 128, kp.data_ptr(), vp.data_ptr(), kp.shape[0], tables.data_ptr(), width,
        width, ctx_d.data_ptr(), 1, len(ctx), 16, 8, 128, 16, SCALE, ws.data_ptr(), need,
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    spread = data_plane.paged_decode_attention(q, kp, vp, tables, ctx_d, SCALE, workspace=ws)
    assert (ws == 171).all()
    if width <= 128:
        assert torch.equal(out.view(torch.int16), spread.view(torch.int16))
    assert (out.float() - spread.float()).abs().max().item() <= TOL


@pytest.mark.parametrize("batch,kv_heads,group", [(129, 8, 1), (300, 8, 2), (200, 8, 8), (520, 2, 2), (1025, 1, 5)])
def test_merge_of_many_sequences(native_lib, device, monkeypatch, batch, kv_heads, group):
    """More sequences than half the block ranges (a merge workgroup per sequence): empty, one-token and
    two-block contexts among longer ones, one cut into many ranges.  Against the per-sequence kernels, which
    other tests hold against the oracle."""
    gen = torch.Generator(device=device).manual_seed(batch)
    ctx = torch.randint(0, 300, (batch,), generator=gen, device=device)
    ctx[::7] = torch.tensor([0, 1, 16, 17, 31, 32, 33], device=device).repeat(-(-len(ctx[::7]) // 7))[:len(ctx[::7])]
    ctx[batch // 2] = 8000
    width = 512
    num_blocks = 3000
    tables = torch.randint(1, num_blocks, (batch, width), generator=gen, device=device)
    kp, vp = (torch.randn(num_blocks, 16, kv_heads, 128, generator=gen, device=device).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(batch, group * kv_heads, 128, generator=gen, device=device).to(torch.bfloat16)
    outs = []
    for path in ("stream", "seq"):
        monkeypatch.setenv("MI_DECODE_PATH", path)
        out = torch.full((batch, group * kv_heads * 128), float("nan"), dtype=torch.bfloat16, device=device)
        outs.append(data_plane.paged_decode_attention(q, kp, vp, tables, ctx, SCALE, out=out).float())
    assert (outs[0] - outs[1]).abs().max().item() <= TOL  # NaN (a row not written) fails too
    assert not outs[0][ctx == 0].any()


@pytest.mark.parametrize("ctx", [[2577], [2064, 129], [8000, 300, 15]])
def test_an_infinite_value_stays_infinite(native_lib, device, monkeypatch, ctx):
    """Parts of an odd number of blocks attend the last one beside a masked copy of itself: an infinity in its values
    gives an infinite output, as in the stream kernel, not a NaN."""
    width = max(-(-n // 16) for n in ctx)
    kp, vp, tables, qkv, _, _, _ = _case(sum(ctx), ctx, max(width, 130), 2)
    for b, n in enumerate(ctx):
        vp[tables[b, (n - 1) // 16], (n - 1) % 16, :, ::3] = float("inf")
        vp[tables[b, 0], 0, :, 1::3] = -float("inf")
    q = qkv[:, :2048].reshape(len(ctx), 16, 128).contiguous().to(device)
    outs = []
    for path in ("stream", "seq"):
        monkeypatch.setenv("MI_DECODE_PATH", path)
        outs.append(data_plane.paged_decode_attention(q, kp.to(device), vp.to(device), tables.to(device),
                                                      torch.tensor(ctx).to(device), SCALE).float())
    inf = outs[0].isinf()
    assert inf.float().mean() > 0.6 and torch.equal(outs[0][inf], outs[1][inf])
    assert (outs[0][~inf] - outs[1][~inf]).abs().max().item() <= TOL
