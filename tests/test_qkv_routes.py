"""Where the QKV projection of a prompt may make queries, keys and values in one launch:
what that launch cannot read goes to the product and the pass behind it."""

from types import SimpleNamespace

import pytest
import torch

from sutro_amd import ops
from sutro_amd.models.qwen3 import Qwen3Attention

M, HQ, HK, K = 4096, 16, 8, 512


@pytest.fixture
def kernels(monkeypatch):
    """Stands in for the extension: counts the calls that reach it."""
    class Kernels:
        calls = 0

        def linear_heads(self, *args):
            self.calls += 1
            return args[0]

    k = Kernels()
    monkeypatch.setattr(ops, "_use_hip", lambda t: True)
    monkeypatch.setattr(ops, "_require_hip", lambda: k)
    return k


def _operands():
    bf = dict(dtype=torch.bfloat16)              # (never read)
    return dict(
        x=torch.empty(M, K, **bf), w=torch.empty((HQ + 2 * HK) * 128, K, **bf),
        num_heads=HQ, num_kv_heads=HK, head_dim=128,
        positions=torch.zeros(M, dtype=torch.int64),
        slot_mapping=torch.zeros(M, dtype=torch.int64),
        k_cache=torch.empty(4, HK, 32, 128, **bf),
        v_cache=torch.empty(4, HK, 32, 128, **bf),
        cos_sin=torch.empty(9, 128), q_norm_w=torch.empty(128, **bf),
        k_norm_w=torch.empty(128, **bf))


def _calls(kernels, **other):
    got = ops.linear_qkv_prep(**{**_operands(), **other})
    assert (got is not None) == kernels.calls
    return kernels.calls


@pytest.mark.parametrize("norm", [True, False])
def test_taken(kernels, norm):
    assert _calls(kernels, **({} if norm else dict(q_norm_w=None, k_norm_w=None))) == 1


@pytest.mark.parametrize("name", ["positions", "slot_mapping", "k_cache", "v_cache",
                                  "cos_sin", "q_norm_w", "k_norm_w"])
def test_operands_elsewhere(kernels, name):
    """On another device than the rows."""
    assert _calls(kernels, **{name: _operands()[name].to("meta")}) == 0


@pytest.mark.parametrize("name,make", [
    # as many positions and slots as the largest batch, of which the first are used
    ("positions", lambda t: torch.zeros(M + 64, dtype=torch.int64)),
    ("slot_mapping", lambda t: torch.zeros(M + 64, dtype=torch.int64)),
    ("q_norm_w", lambda t: torch.cat([t, t])), ("k_norm_w", lambda t: torch.cat([t, t])),
    # (the pass refuses these)
    ("num_heads", lambda n: n + 2), ("num_kv_heads", lambda n: n + 1),
    ("k_cache", lambda t: t[:, :4].contiguous()), ("k_cache", lambda t: t.flatten(2))])
def test_sizes_that_differ(kernels, name, make):
    other = {name: make(_operands()[name])}
    if name == "k_cache":
        other["v_cache"] = other[name]
    assert _calls(kernels, **other) == 0


@pytest.mark.parametrize("rows,k,wide,one", [
    # few places taken: a short k gains all the same
    (5045, 512, 4096, 1), (5045, 576, 4096, 0), (5045, 1024, 4096, 0),
    (3336, 1024, 6144, 0), (7138, 1024, 3072, 0), (6438, 768, 3072, 0),
    (6000, 1024, 4096, 1), (4096, 1024, 4096, 1), (24000, 1024, 4096, 1),
    (9130, 2048, 4096, 0), (6048, 2048, 6144, 0), (9400, 2048, 4096, 1),
    (32768, 2048, 3072, 1), (8192, 4096, 6144, 1), (7600, 4096, 6144, 0),
    (16384, 8192, 4096, 0)])
def test_sizes(kernels, rows, k, wide, one):
    bf = dict(dtype=torch.bfloat16, device="meta")
    heads = wide // 128 // 4
    i64 = torch.zeros(rows, dtype=torch.int64, device="meta")
    norm, pages = torch.empty(128, **bf), torch.empty(4, heads, 32, 128, **bf)
    assert _calls(kernels, x=torch.empty(rows, k, **bf), w=torch.empty(wide, k, **bf),
                  num_heads=2 * heads, num_kv_heads=heads, positions=i64,
                  slot_mapping=i64, k_cache=pages, v_cache=pages, q_norm_w=norm,
                  k_norm_w=norm, cos_sin=torch.empty(9, 128, device="meta")) == one


@pytest.mark.parametrize("rows,asked", [(1, 0), (21, 0), (1000, 0), (3840, 0), (3841, 1)])
def test_few_rows_are_not_asked(monkeypatch, rows, asked):
    """Eager steps of few rows are bound by what is asked on the host."""
    spec = SimpleNamespace(num_heads=30, num_kv_heads=1, head_dim=128, hidden_size=4,
                           qk_norm=True, rms_eps=1e-6)
    attn = Qwen3Attention(spec, torch.float32, 0)
    calls = []
    monkeypatch.setattr(ops, "linear_qkv_prep", lambda *a: calls.append(1))
    monkeypatch.setattr(ops, "fused_qkv_prep",
                        lambda qkv, *a: qkv[:, :3840].reshape(-1, 30, 128))
    monkeypatch.setattr(ops, "paged_attention", lambda q, *a: q)
    fb = SimpleNamespace(**dict.fromkeys((
        "positions", "slot_mapping", "block_tables", "seq_lens", "query_start_locs",
        "num_decodes_tail", "tile_seq", "tile_q0", "prefill_token_count")))
    kv = SimpleNamespace(k_cache=[None], v_cache=[None])
    assert attn(torch.zeros(rows, 4), fb, kv, None).shape == (rows, 4)
    assert len(calls) == asked
