"""The uniforms of seeded rows, in native code and in numpy."""

import numpy as np
import pytest
import torch

from sutro_amd import ops
from sutro_amd.engine.request import Request, SamplingParams
from sutro_amd.engine.sampler import Sampler, seeded_uniform

pytestmark = pytest.mark.skipif(not ops.hip_available(),
                                reason="extension not built")


class Longer(Request):
    @property
    def total_len(self):
        return 1000


def _reqs(n):
    g = np.random.default_rng(n)
    kinds = (Request, Longer)
    return [kinds[i % 5 == 4](
        req_id=i, prompt_token_ids=[1] * int(g.integers(1, 9)),
        output_token_ids=[2] * int(g.integers(0, 9)),
        sampling=SamplingParams(seed=None if i % 7 == 3 else int(
            g.integers(0, 2 ** 63)) * 2 + i % 2)) for i in range(n)]


@pytest.mark.parametrize("n", [1, 4, 100])
@pytest.mark.parametrize("override", [False, True])
def test_as_in_numpy(n, override):
    reqs = _reqs(n)
    rows = np.array([i for i, r in enumerate(reqs) if r.sampling.seed is not None])
    seeds = np.array([reqs[i].sampling.seed for i in rows], dtype=np.uint64)
    steps = np.arange(7, 7 + n) if override else None
    used = steps[rows] if override else [reqs[i].total_len for i in rows]
    out = torch.full((n,), -1.0)
    assert ops.seeded_uniforms(out, reqs, rows, seeds, steps, Request)
    want = np.full(n, -1.0)
    want[rows] = seeded_uniform(seeds, np.array(used))
    assert np.array_equal(out.numpy(), want.astype(np.float32))


def test_without_native_code(monkeypatch):
    """`Sampler` gives the same uniforms either way, those of rows without a seed
    among them."""
    reqs = _reqs(30)
    got = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_C", None)
        s = Sampler("cpu", seed=5)
        dev = torch.device("cpu")
        p = s._param_tensors(reqs, dev)
        got.append(s._uniforms(reqs, *p[3:], None, dev, len(reqs)))
    assert torch.equal(*got)


def test_errors():
    out = torch.zeros(2)
    seeds = np.ones(1, np.uint64)
    for row in (2, -1):
        with pytest.raises(RuntimeError):
            ops.seeded_uniforms(out, _reqs(2), np.array([row]), seeds, None, Request)
    with pytest.raises(AttributeError):
        ops.seeded_uniforms(out, [1, 2], np.array([0]), seeds, None, Request)
    odd = _reqs(1)
    odd[0].prompt_token_ids = None
    with pytest.raises(TypeError):
        ops.seeded_uniforms(out, odd, np.array([0]), seeds, None, Request)
