"""Which workgroup shapes the prefill and mixed entry points launch, on the CPU against a stand-in HIP runtime (no
GPU, 256 CUs)."""

import hip_standin

CALLS = """
P = 4096
def prefill(rows, width, hist, group=2, kv=8):
    heads = group * kv
    return lib.mi_chunked_prefill_attention(P, width * heads * 128, heads * 128, P, width * heads * 128, 128, heads * 128,
                                            P, width * kv * 128, 128, kv * 128, P, width * kv * 128, 128, kv * 128, P, P, 100, P,
                                            max(hist, 1), hist, P, P, 1, rows, width, heads, kv, 128, 16, 0.1, None)
def mixed(rows, width, hist, decode_rows, mb, group=2, kv=8, exact="", first=None, tokens=0):
    heads = group * kv
    return getattr(lib, "mi_mixed_paged_attention" + exact)(
        P, heads * 128, P, heads * 128, 128, P, kv * 128, 128, P, kv * 128, 128, P, P, 100, rows, width, tokens, first, P,
        max(hist, 1), hist, P, P, 1, decode_rows, P, max(mb, 1), mb, P, 1, P, 1, heads, kv, 128, 16, 0.1, None)
def shapes():
    return [(l["args"], l["grid"][0], l["block"], l["lds"]) for l in launches()]
"""
WIDE, HALF, HALF_SPLIT, NARROW = [2, 4, 1], [2, 2, 1], [2, 2, 2], [1, 2, 2]


def test_prefill_shapes_by_launch_size_and_history():
    cases = [
        # narrow: one round of its workgroups, or 11/8 of one without much history
        (1, 1, 0, 2, NARROW), (1, 1024, 0, 2, NARROW), (1, 60, 250, 2, NARROW), (8, 128, 8, 2, NARROW),
        (1, 1025, 33, 2, HALF_SPLIT), (1, 1025, 32, 2, NARROW), (2, 704, 0, 2, NARROW), (2, 705, 0, 2, HALF_SPLIT),
        # short rows without history: half
        (9, 128, 0, 2, NARROW), (12, 128, 0, 2, HALF), (16, 256, 0, 2, HALF), (64, 128, 0, 2, HALF), (100, 256, 0, 2, HALF),
        # up to half of the CUs in wide workgroups: half split
        (12, 128, 1, 2, HALF_SPLIT), (16, 128, 8, 2, HALF_SPLIT), (5, 257, 0, 2, HALF_SPLIT), (1, 2048, 0, 2, HALF_SPLIT),
        # up to all of them: wide with history, else half split for long rows
        (17, 128, 8, 2, WIDE), (17, 128, 7, 2, HALF), (2, 1152, 0, 2, HALF_SPLIT), (2, 1152, 72, 2, WIDE), (4, 640, 0, 2, HALF),
        (4, 641, 0, 2, HALF_SPLIT), (1, 4096, 0, 2, HALF_SPLIT), (32, 128, 8, 2, WIDE),
        # a second wide round up to 9/16 full: half; beyond: wide
        (33, 128, 300, 2, HALF), (50, 128, 300, 2, HALF), (51, 128, 300, 2, WIDE), (25, 257, 0, 2, WIDE), (64, 128, 1, 2, WIDE),
        # the table beside split tiles in LDS
        (1, 60, 8192, 2, NARROW), (1, 60, 8193, 2, HALF), (4, 2048, 640, 2, WIDE), (2, 700, 0, 5, HALF),
    ]
    got = hip_standin.run(CALLS + f"""
result = []
for rows, width, hist, group in {[c[:4] for c in cases]}:
    assert prefill(rows, width, hist, group) == 0
    result.append(shapes())
""")
    for (rows, width, hist, group, want), launches in zip(cases, got):
        (args, grid, block, lds), = launches
        assert args[1:] == want, (rows, width, hist, group, args)
        tile = 16 * args[1] * args[2]
        assert grid == 8 * ((group + 1) // 2) * rows * -(-width // tile) and lds <= 160 * 1024
        assert block == 64 * 2 * args[2] * args[3]


def test_mixed_chunk_rows_take_the_shape_of_a_prefill():
    """The same order of sums (the wide shape sums as the half one does), whatever the decode rows' table."""
    got = hip_standin.run(CALLS + """
result = []
for rows, width, hist in [(1, 300, 0), (1, 700, 40), (2, 700, 0), (2, 700, 50), (2, 1200, 0), (4, 640, 0), (33, 128, 0), (4, 2048, 640)]:
    assert prefill(rows, width, hist) == 0
    alone = shapes()
    for mb in (0, 72, 512, 8192, 8193, 16384):
        assert mixed(rows, width, hist, 7, mb) == 0
        result.append((mb, alone[0], shapes()))
    assert mixed(rows, width, hist, 7, 16385) == -2 and not launches()  # refused before any launch
""")
    for mb, (want, _, _, _), launches in got:
        split = want[3] == 2
        args = [l[0] for l in launches]
        assert args[0][3] == want[3] and (args[0] == want if split else args[0][1:] == WIDE)
        assert all(l[3] <= 160 * 1024 for l in launches)
        assert len(launches) == (2 if split and mb > 8192 else 1)
        if len(launches) == 2:
            assert args[1][1:] == WIDE


def test_refused_mixed_steps_launch_nothing():
    """The decode rows append to the pool: a step that a size check refuses must not have run them."""
    got = hip_standin.run(CALLS + """
result = []
for exact in ("", "_exact"):
    for rows, width, first, tokens in [(1, 64, P, 1 << 31), (65535, 1 << 20, None, 0), (65535, 1 << 20, P, 4096)]:
        result.append((exact, mixed(rows, width, 4, 3, 20, exact=exact, first=first, tokens=tokens), len(launches())))
    assert mixed(1, 64, 4, 3, 20, exact=exact, first=P, tokens=100) == 0 and launches()
""")
    for exact, rc, count in got:
        assert (rc, count) == (-2, 0), exact


def test_exact_decode_rows_go_beside_the_chunk_rows_where_they_are_few_and_short():
    """One launch where a decode row's table holds at most 128 keys more than a chunk row sees and the rows fill at most
    half the CUs; else the decode body in a launch of its own, first."""
    got = hip_standin.run(CALLS + """
result = []
for width, hist, decode_rows, mb in [(96, 19, 1, 13), (96, 19, 1, 33), (96, 19, 1, 34), (97, 0, 16, 14), (97, 0, 16, 15), (97, 0, 17, 6),
                                     (650, 0, 7, 72), (2048, 0, 8, 136), (2048, 0, 8, 137), (64, 4, 3, 0), (0, 0, 3, 20)]:
    assert mixed(1 if width else 0, width, hist, decode_rows, mb, exact="_exact") == 0
    result.append((16 * mb <= 16 * hist + width + 128 and decode_rows <= 16 or mb == 0, bool(width),
                   [(l["kernel"], l["args"]) for l in launches()]))
# Ragged rows: a launch wider than a row's share of the chunk tokens counts the share, without the history.
for rows, width, tokens, decode_rows, mb in [(1, 1023, 128, 8, 16), (1, 1023, 128, 8, 17), (1, 1023, 1024, 8, 135), (3, 1023, 1024, 8, 29),
                                             (3, 1023, 1024, 8, 30), (2, 512, 1024, 8, 104), (2, 512, 1023, 8, 104), (2, 513, 1024, 8, 41)]:
    assert mixed(rows, width, 64, decode_rows, mb, exact="_exact", first=P, tokens=tokens) == 0
    share = -(-tokens // rows)
    keys = share if share < width else width + 64 * 16
    result.append((16 * mb <= keys + 128, True, [(l["kernel"], l["args"]) for l in launches()]))
# A score cache that the decode rows' tables outgrow: the chunk rows keep theirs.
for mb in range(1, 400):
    assert mixed(1, 16 * mb, 0, 1, mb + 8, exact="_exact") == 0 and prefill_exact(1, 16 * mb) == 0
    calls = launches()
    result.append((None, True, [(l["kernel"], l["args"]) for l in calls]))
""".replace("result = []", """
def prefill_exact(rows, width, group=2, kv=8):
    heads = group * kv
    return lib.mi_chunked_prefill_attention_exact(P, width * heads * 128, heads * 128, P, width * heads * 128, 128, heads * 128,
                                                  P, width * kv * 128, 128, kv * 128, P, width * kv * 128, 128, kv * 128, P, P, 100,
                                                  P, 1, 0, P, P, 1, rows, width, heads, kv, 128, 16, 0.1, None)
result = []"""))
    for beside, chunks, calls in got:
        kernels = [name for name, _ in calls]
        if beside is None:
            assert calls[-2] == calls[-1]  # the chunk rows' kernel, cached or not, as without decode rows
        elif not chunks:
            assert kernels == ["exact_decode_kernel"]
        else:
            assert kernels == (["exact_prefill_kernel"] if beside else ["exact_decode_kernel", "exact_prefill_kernel"])
