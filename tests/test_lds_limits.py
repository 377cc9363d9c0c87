"""Kernels with more than 64 KiB of dynamic LDS have their limit raised on every device that launches them, on the
CPU against a stand-in HIP runtime with two devices (no GPU)."""

import hip_standin
from test_prefill_routes import CALLS


def test_the_limit_is_raised_on_each_device_before_its_first_launch():
    got = hip_standin.run(CALLS + """
def decode_exact(batch, mb, heads=16, kv=8):
    return lib.mi_paged_decode_attention_exact(P, heads * 128, P, heads * 128, 128, None, 0, None, 0, None, None, None, None, 0.0, None,
                                               0, P, P, 1000, P, mb, mb, P, 1, batch, heads, kv, 128, 16, 0.1, None, 0, None)
def prefill_exact(rows, width, group=2, kv=8):
    heads = group * kv
    return lib.mi_chunked_prefill_attention_exact(P, width * heads * 128, heads * 128, P, width * heads * 128, 128, heads * 128,
                                                  P, width * kv * 128, 128, kv * 128, P, width * kv * 128, 128, kv * 128, P, P, 100,
                                                  P, 1, 0, P, P, 1, rows, width, heads, kv, 128, 16, 0.1, None)
result = []
for device in (0, 1, 0):
    hip.standin_set_device(device)
    rcs = [decode_exact(40, 100), decode_exact(40, 1500), prefill_exact(2, 300), prefill_exact(1, 3000), prefill_exact(1, 4000),
           prefill_exact(1, 30000), mixed(1, 64, 4, 7, 1500, exact="_exact"),
           prefill(1, 100, 0), mixed(1, 100, 0, 3, 20)]
    raised = sorted({hip.standin_attr_name(i).decode() for i in range(hip.standin_attrs())
                     if hip.standin_attr_device(i) == device})
    result.append([rcs, raised, sorted({l["mangled"] for l in launches() if l["lds"] > 65536})])
""")
    (rc0, raised0, large0), (rc1, raised1, large1), (rc2, raised2, large2) = got
    assert not any(rc0 + rc1 + rc2) and large0 == large1 == large2 and len(large0) >= 3
    assert set(large0) <= set(raised0) and raised0 == raised1
    assert raised2 == []  # once per kernel and device
