"""The engine's batch tensors against a token-by-token build: whole prompts,
chunks, decode rows (one with its token still in flight), the token before
each row's token, state slots, pages in any order."""

import pytest
import torch

from sutro_amd.engine.batch import ScheduledBatch
from sutro_amd.engine.config import EngineConfig
from sutro_amd.engine.engine import LLMEngine
from sutro_amd.engine.request import Request, SamplingParams
from sutro_amd.models.registry import tiny_spec_for_tests


@pytest.fixture(scope="module")
def engine():
    return LLMEngine(EngineConfig(spec=tiny_spec_for_tests(), device="cpu",
                                  num_kv_blocks=64, max_num_seqs=8))


def _naive(eng, sb, prev):
    bs = eng.kv.block_size
    out = {k: [] for k in ("input_ids", "positions", "slot_mapping", "token_seq",
                           "prev_ids", "tile_seq", "tile_q0", "logits_idx")}
    qlocs, lens = [0], []
    for s, (r, c) in enumerate(zip(sb.reqs, sb.num_new_tokens)):
        table = eng.kv.block_tables[r.req_id]
        for j in range(c):
            p = r.num_computed_tokens + j
            out["input_ids"].append(r.token_at(p) if p < r.total_len else 0)
            out["positions"].append(p)
            out["slot_mapping"].append(table[p // bs] * bs + p % bs)
            out["token_seq"].append(s)
            out["prev_ids"].append(r.token_at(p - 1) if p else -1)
        qlocs.append(qlocs[-1] + c)
        lens.append(r.num_computed_tokens + c)
        if s < sb.num_prefills:
            for j in range(0, c, 32):
                out["tile_seq"].append(s)
                out["tile_q0"].append(j)
        if s >= sb.num_prefills or lens[-1] == r.num_prompt_tokens:
            out["logits_idx"].append(qlocs[-1] - 1)
    if not prev:
        out.pop("prev_ids")
    out["query_start_locs"], out["seq_lens"] = qlocs, lens
    return out


@pytest.mark.parametrize("prev", [False, True])
def test_batch_matches_a_token_by_token_build(engine, prev, monkeypatch):
    if prev:
        monkeypatch.setattr(engine.model, "uses_prev_ids", True, raising=False)
    rows = [(70, 0, 0, 70), (100, 33, 0, 40), (40, 39, 0, 1), (1, 0, 0, 1),
            (12, 14, 3, 1), (33, 36, 3, 1)]    # the last one is in flight
    reqs = []
    for i, (n, done, outs, _) in enumerate(rows):
        r = Request(req_id=1000 + i, prompt_token_ids=list(range(3, 3 + n)),
                    sampling=SamplingParams(max_tokens=8))
        r.output_token_ids = [200 + k for k in range(outs)]
        r.num_computed_tokens = done
        reqs.append(r)
    for step in range(3):      # pages of the rows interleaved
        for r, (n, done, _, c) in zip(reqs, rows):
            engine.kv.grow(r.req_id, max(1, (done + c) * (step + 1) // 3))
    sb = ScheduledBatch(reqs=reqs, num_new_tokens=[c for *_, c in rows],
                        num_prefills=4)
    fb = engine._build_forward_batch(sb)
    for name, want in _naive(engine, sb, prev).items():
        got = getattr(fb, name)
        assert got.tolist() == want, name
        assert got.is_contiguous()
    assert (fb.prev_ids is None) == (not prev)
    assert fb.prefill_token_count == 112 and fb.num_decodes_tail == 2
    assert fb.max_seq_len == 73 and fb.max_query_len == 70
    for s, r in enumerate(reqs):
        t = engine.kv.block_tables[r.req_id]
        assert fb.block_tables[s, :len(t)].tolist() == t
        engine.kv.release(r.req_id)


def test_equal_fields_are_not_the_same_request():
    a, b = (Request(req_id=1, prompt_token_ids=[1], sampling=SamplingParams())
            for _ in range(2))
    assert a in [a] and a not in [b]
