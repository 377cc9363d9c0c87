"""The shape checks of the fused decode entry point in the Python layer, on the CPU with a stand-in library that
records the native calls (no GPU)."""

import types

import pytest
import torch

from mini_infra_qwen3_amd import _native, data_plane

B, HEADS, KV, D = 8, 16, 8, 128


class Recorder:
    """Stands in for the loaded library: every entry point succeeds and is noted by name."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def entry(*args):
            self.calls.append(name)
            return 4096 if name.endswith("workspace_bytes") else _native.MI_OK

        return entry


@pytest.fixture
def library(monkeypatch):
    lib = Recorder()
    monkeypatch.setattr(data_plane, "_native", types.SimpleNamespace(load=lambda: lib, check=_native.check))
    monkeypatch.setattr(data_plane, "_require_gpu", lambda *args, **kwargs: None)  # CPU tensors stand in
    monkeypatch.setattr(data_plane, "_stream", lambda device: 0)
    return lib


def bf16(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def call(q, k, v, exact=False):
    pool = bf16(64, 16, KV, D)
    return data_plane.paged_decode_attention_fused(
        q, k, v, bf16(D), bf16(D), bf16(B, D), bf16(B, D), 1e-6, torch.arange(B), pool, pool.clone(),
        torch.zeros((B, 4), dtype=torch.long), torch.ones(B, dtype=torch.long), 0.1, exact=exact)


def native_calls(lib):
    return [name for name in lib.calls if not name.endswith("_bytes")]


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("rows", [1, 2, 4, 7, 16])
def test_key_and_value_rows_of_another_token_count_are_refused(library, rows, exact):
    """Fewer rows than tokens: the kernel would read past the rows' end and append what it found there."""
    with pytest.raises(ValueError, match="inconsistent head sizes"):
        call(bf16(B, HEADS * D), bf16(rows, KV * D), bf16(rows, KV * D), exact)
    with pytest.raises(ValueError, match="inconsistent head sizes"):
        call(bf16(B, HEADS * D), bf16(B, KV * D), bf16(rows, KV * D), exact)
    with pytest.raises(ValueError, match="inconsistent head sizes"):
        call(bf16(B, HEADS * D), bf16(rows, KV * D), bf16(B, KV * D), exact)
    assert native_calls(library) == []


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("shape", [(B, KV * D), (B, 1, KV * D), (B, KV, D), (B * KV, D)])
def test_layouts_of_the_same_rows_are_accepted(library, shape, exact):
    out = call(bf16(B, HEADS * D), bf16(*shape), bf16(*shape), exact)
    assert out.shape == (B, HEADS * D) and len(native_calls(library)) == 1
    projection = bf16(B, (HEADS + 2 * KV) * D)  # one projection's rows, as views
    q, k, v = projection.split((HEADS * D, KV * D, KV * D), dim=1)
    call(q, k, v, exact)
    assert len(native_calls(library)) == 2
