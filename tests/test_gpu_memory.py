"""The fragment-ordered copies of the weights only make calls faster: an engine that
has just enough device memory without them answers every call with them allowed,
on the products over the stored rows where a copy found no room or was given up."""

import numpy as np
import pytest

from conftest import make_prompt
from oracle import oracle as O
from s2hip import synth

pytestmark = pytest.mark.gpu

SHAPE = synth.TINY.with_(name="memory", slow_layers=2, fast_layers=1, vocab=2304, semantic_begin=1024,
                         semantic_end=2047, im_end_id=1000)
TYPES = {"f16": synth.GGML_F16, "q8_0": synth.GGML_Q8_0, "q4_0": synth.GGML_Q4_0}
KV = 700
STEP = 256 * 1024  # resolution of the search; the copies are megabytes


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1e-30, float(np.max(np.abs(b)))))


def _calls(path):
    """Calls that each need more than the one before: a prompt, a step, codebooks, one
    request, then four, then a longer prompt."""
    from s2hip import Engine

    with Engine(path, KV, SHAPE.im_end_id) as e:
        out = [e.eval(make_prompt(SHAPE, 40, seed=1)), e.eval(make_prompt(SHAPE, 1, seed=2))]
        e.fast_codebooks(out[0][0], 5)
        e.generate_codes(make_prompt(SHAPE, 20, seed=3), 6, min_tokens_before_end=100)
        e.generate_codes_batch([make_prompt(SHAPE, 9 + b, seed=4 + b) for b in range(4)], 420, min_tokens_before_end=0)
        e.generate_codes(make_prompt(SHAPE, 20, seed=3), 6, min_tokens_before_end=100)
        e.reset()
        out.append(e.eval(make_prompt(SHAPE, 600, seed=9)))
    return out


@pytest.mark.parametrize("weights", sorted(TYPES))
def test_copies_never_take_the_memory_that_a_call_needs(model_dir, monkeypatch, weights):
    from s2hip import S2HipError

    path = synth.ensure_gguf(SHAPE.with_(linear_type=TYPES[weights]), model_dir)
    monkeypatch.setenv("S2HIP_BMM_MIN_COLS", "0")
    lo, hi = 0, 512 << 20  # MiB: too little, enough
    while hi - lo > STEP:
        mid = (lo + hi) // 2
        monkeypatch.setenv("S2HIP_DEVICE_BYTES", str(mid))
        try:
            _calls(path)
            hi = mid
        except S2HipError as e:
            assert "out of memory" in str(e), e
            lo = mid
    monkeypatch.delenv("S2HIP_BMM_MIN_COLS")
    o = O.OracleModel(path, KV, SHAPE.im_end_id)
    want = [o.eval(make_prompt(SHAPE, 40, seed=1)), o.eval(make_prompt(SHAPE, 1, seed=2))]
    o.reset()
    want.append(o.eval(make_prompt(SHAPE, 600, seed=9)))
    for budget in (hi, hi + (4 << 20), 512 << 20):  # no room for copies, for some, for all
        monkeypatch.setenv("S2HIP_DEVICE_BYTES", str(budget))
        for (hg, lg), (ho, lo_) in zip(_calls(path), want):
            assert _rel(hg, ho) < 1e-4 and _rel(lg, lo_) < 1e-4, budget
