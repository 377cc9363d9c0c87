"""Which kernels the decode entry points launch, on the CPU against a stand-in HIP runtime (no GPU): what the
entry points promise about ordering and about the caller's workspace is a matter of the route."""

import hip_standin

CALLS = """
P = 4096
def attention(entry, batch, mb, ws=P, nbytes=1 << 30, heads=16, kv=8):
    return getattr(lib, entry)(P, heads * 128, P, heads * 128, 128, P, P, 1000, P, max(mb, 1), mb, P, 1, batch, heads, kv, 128, 16,
                               0.1, *(() if entry.endswith("noalloc") else (ws, nbytes)), None)
def fused(entry, batch, mb, ws=P, nbytes=1 << 30, offset=0, heads=16, kv=8):
    return getattr(lib, entry)(P, heads * 128, P + offset, 4096, P, 4096, P, 4096, P, P, P, P, 1e-6, P, 1, P, P, 1000, P,
                               max(mb, 1), mb, P, 1, batch, heads, kv, 128, 16, 0.1, P, ws, nbytes, None)
"""


def test_a_fused_launch_of_more_pairs_than_cus_appends_before_it_attends():
    """Rows that read each other's new token (one sequence as two rows) are ordered after the append there."""
    routes = hip_standin.run(CALLS + """
result = []
for batch, kv in [(32, 8), (33, 8), (64, 8), (128, 8), (300, 8), (129, 2), (256, 1), (257, 1)]:
    for mb in (4, 30, 72, 200, 512):
        assert fused("mi_paged_decode_attention_fused", batch, mb, heads=2 * kv, kv=kv) == 0
        result.append((batch * kv, [(l["kernel"], l["args"]) for l in launches()]))
""")
    for pairs, calls in routes:
        names = [name for name, _ in calls]
        fused = [name for name, args in calls if name in ("paged_decode_stripe_kernel", "paged_decode_parts_kernel") and args[2]]
        if pairs <= 256:
            assert names[0] in fused
        else:
            assert names[0].startswith("qk_norm_rope") and not fused, (pairs, names)


def test_small_fused_launches_need_no_workspace_whatever_the_alignment_of_their_rows():
    """Up to one (sequence, KV head) pair per CU and 512 table blocks: the sequences stay whole without one."""
    routes = hip_standin.run(CALLS + """
result = []
for batch in (1, 8, 32):
    for mb in (1, 30, 72, 200, 512):
        for ws, nbytes in [(None, 0), (P, 16), (P + 8, 1 << 30)]:
            for offset in (0, 2):
                rc = fused("mi_paged_decode_attention_fused", batch, mb, ws, nbytes, offset)
                result.append((offset, rc, [(l["kernel"], l["args"]) for l in launches()]))
""")
    for offset, rc, calls in routes:
        assert rc == 0
        assert [name for name, _ in calls] == (["qk_norm_rope_kernel"] if offset else []) + ["paged_decode_stripe_kernel"]
        assert calls[-1][1] == [8, 2, 0 if offset else 1, 8]  # every stripe in one workgroup


def test_small_launches_leave_the_callers_workspace_untouched():
    """Calls that overlap on two streams may share one workspace while all of them are small: no partials, no
    merge.  The spread entry points cut the sequences (their workspace is the call's own), and
    mi_paged_decode_spread_bytes says where."""
    routes = hip_standin.run(CALLS + """
result = []
for batch, kv in [(1, 8), (8, 8), (32, 8), (128, 2), (256, 1), (33, 8), (96, 8)]:
    for mb in (1, 30, 64, 128, 129, 512, 513):
        for fn, entry in ((attention, "mi_paged_decode_attention"), (fused, "mi_paged_decode_attention_fused"),
                          (attention, "mi_paged_decode_attention_noalloc"), (attention, "mi_paged_decode_attention_spread"),
                          (fused, "mi_paged_decode_attention_fused_spread")):
            rc = fn(entry, batch, mb, heads=2 * kv, kv=kv)
            names = [l["kernel"] for l in launches()]
            result.append((entry, batch * kv, mb, rc, names, lib.mi_paged_decode_spread_bytes(batch, mb, 2 * kv, kv, 128, 16),
                           lib.mi_paged_decode_workspace_bytes(batch, mb, 2 * kv, kv, 128, 16)))
""")
    for entry, pairs, mb, rc, names, spread, need in routes:
        assert rc == 0 or (rc == -3 and entry.endswith("noalloc") and need > 8 << 20)
        small = pairs <= 256 and mb <= 512
        assert spread in ((0, need) if small else (0,))
        if small and entry.endswith("spread"):
            merged = ["paged_decode_stripe_merge_kernel"] if mb <= 128 else ["paged_decode_merge_kernel"]
            assert names[1:] == (merged if spread else [])
            assert (mb >= 129) <= (spread > 0)
        elif small:
            assert names == ["paged_decode_stripe_kernel"]


def test_many_sequences_are_merged_by_one_workgroup_each():
    """The stream form's merge: a workgroup per sequence where a sequence spans under two ranges, else one per
    (sequence, KV head)."""
    routes = hip_standin.run(CALLS + """
result = []
for batch, kv in [(64, 8), (128, 8), (129, 8), (512, 8), (4096, 8), (512, 2), (513, 2), (4500, 8)]:
    assert attention("mi_paged_decode_attention", batch, 600, heads=2 * kv, kv=kv) == 0
    result.append((batch, kv, [(l["kernel"], l["args"], l["grid"], l["block"]) for l in launches()]))
""")
    for batch, kv, calls in routes:
        for at, rows in enumerate([min(batch, 4096), batch - 4096] if batch > 4096 else [batch]):
            name, args, grid, block = calls[2 * at + 1]
            if (1024 if kv == 2 else 256) < 2 * rows:
                assert (name, args, grid, block) == ("paged_decode_merge_rows_kernel", [2 * kv], [rows, 1, 1], 256)
            else:
                assert (name, args, grid) == ("paged_decode_merge_kernel", [kv, 2, 0], [rows, kv, 1])


def test_sequences_of_large_launches_are_cut_or_streamed():
    """Past one pair per CU the per-sequence kernels take a launch only where they can cut its sequences in two;
    the workgroup of eight stripes per (sequence, KV head) does not serve thousands of short sequences."""
    routes = hip_standin.run(CALLS + """
result = []
for batch, kv in [(33, 8), (64, 8), (191, 8), (192, 8), (256, 8), (512, 8), (4096, 8), (767, 2), (768, 2), (1535, 1), (1536, 1)]:
    for mb in (1, 8, 19, 44, 72, 300):
        assert attention("mi_paged_decode_attention", batch, mb, heads=2 * kv, kv=kv) == 0
        result.append((batch * kv, mb, launches()[0]["kernel"]))
""")
    for pairs, mb, kernel in routes:
        per_sequence = pairs < 6 * 256 and pairs * mb <= 98304
        assert (kernel != "paged_decode_kernel") == per_sequence, (pairs, mb, kernel)


def test_refused_fused_launches_append_nothing():
    """A call that the attention's checks refuse launches nothing, the append included."""
    got = hip_standin.run(CALLS + """
result = []
for entry in ("mi_paged_decode_attention_fused", "mi_paged_decode_attention_fused_spread"):
    for batch, mb, ws, nbytes in [(64, 72, None, 0), (64, 72, P, 1 << 10), (64, 72, P + 8, 1 << 30), (8, 600, None, 0), (64, 1 << 20, P, 1 << 40)]:
        result.append((fused(entry, batch, mb, ws, nbytes), len(launches())))
    assert fused(entry, 64, 72) == 0 and len(launches()) == 3
""")
    for rc, count in got:
        assert rc < 0 and count == 0
