"""Prompt lengths around the tile edges of the prefill products, on every weight
type: one token past and short of a 64- and 128-token tile, past the length
where the wide tile takes over, and past one prefill pass (2048 tokens).  The
second shape's FFN width is no multiple of a weight tile.  f32-level products:
hidden states and logits agree with the oracle to 1e-4 relative."""

import numpy as np
import pytest

from conftest import make_prompt
from oracle import oracle as O
from s2hip import synth

pytestmark = pytest.mark.gpu

BASE = synth.TINY.with_(name="tiles", slow_layers=2, fast_layers=1, vocab=2304, semantic_begin=1024, semantic_end=2047,
                        im_end_id=1000)
TYPES = {"f16": synth.GGML_F16, "q8_0": synth.GGML_Q8_0, "q4_0": synth.GGML_Q4_0}


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1e-30, float(np.max(np.abs(b)))))


@pytest.mark.parametrize("weights", sorted(TYPES))
@pytest.mark.parametrize("ffn,lengths", [(1536, (1, 2, 3, 4, 5, 17, 63, 65, 129, 257, 289, 321, 770, 2100)), (1504, (5, 33, 300))])
def test_prefill_lengths_match_oracle(model_dir, weights, ffn, lengths):
    from s2hip import Engine

    shape = BASE.with_(name=f"tiles{ffn}", linear_type=TYPES[weights], ffn=ffn)
    path = synth.ensure_gguf(shape, model_dir)
    o = O.OracleModel(path, 2200, shape.im_end_id)
    with Engine(path, 2200, shape.im_end_id) as e:
        for n in lengths:
            prompt = make_prompt(shape, n, seed=n)
            e.reset()
            o.reset()
            hg, lg = e.eval(prompt)
            ho, lo = o.eval(prompt)
            assert e.n_past == n
            assert _rel(hg, ho) < 1e-4 and _rel(lg, lo) < 1e-4, (n, _rel(hg, ho), _rel(lg, lo))


def test_short_eval_beyond_the_batched_range(model_dir, tmp_path):
    """Three tokens take the batched decode product; an FFN channel far above the
    first 256 of its row (past the product's per-wave headroom) makes the call
    run again on the prefill products, in KV slot 1 and at a later position."""
    import shutil

    import gguf_util
    from s2hip import Engine

    path = str(tmp_path / "outlier.gguf")
    shutil.copyfile(synth.ensure_gguf(synth.TINY, model_dir), path)
    for l in range(synth.TINY.slow_layers):
        for w in ("w1", "w3"):
            gguf_util.scale_rows(path, f"layers.{l}.feed_forward.{w}.weight", [300], 300.0)
    o = O.OracleModel(path, 64, synth.TINY.im_end_id)
    with Engine(path, 64, synth.TINY.im_end_id) as e:
        for n, seed in ((2, 1), (3, 2), (1, 3), (4, 4)):
            prompt = make_prompt(synth.TINY, n, seed=seed)
            hg, lg = e.eval_slot(1, prompt)
            ho, lo = o.eval(prompt)
            assert _rel(hg, ho) < 1e-4 and _rel(lg, lo) < 1e-4, n
        assert e.n_past_slot(1) == o.n_past == 10 and e.n_past == 0


@pytest.mark.parametrize("weights", sorted(TYPES))
@pytest.mark.parametrize("ffn", [1536, 1504])
def test_prefill_over_the_stored_rows_matches_oracle(model_dir, weights, ffn, monkeypatch):
    """Without fragment-ordered copies (S2HIP_BMM_MIN_COLS=0, or no memory for them)
    the products read the file's rows: lengths around their 128-token tile, with and
    without K splits."""
    from s2hip import Engine

    monkeypatch.setenv("S2HIP_BMM_MIN_COLS", "0")
    shape = BASE.with_(name=f"tiles{ffn}", linear_type=TYPES[weights], ffn=ffn)
    path = synth.ensure_gguf(shape, model_dir)
    o = O.OracleModel(path, 800, shape.im_end_id)
    with Engine(path, 800, shape.im_end_id) as e:
        for n in (3, 5, 33, 127, 129, 300, 770):
            prompt = make_prompt(shape, n, seed=n)
            e.reset()
            o.reset()
            hg, lg = e.eval(prompt)
            ho, lo = o.eval(prompt)
            assert _rel(hg, ho) < 1e-4 and _rel(lg, lo) < 1e-4, (n, _rel(hg, ho), _rel(lg, lo))


@pytest.mark.parametrize("head_dim", [64, 128])
def test_long_prefill_with_an_f16_cache_matches_oracle(model_dir, head_dim):
    """Two query groups per attention block (past 256 queries) over an f16 KV cache, at
    ragged lengths, then a second prompt that attends the first."""
    from s2hip import Engine

    shape = BASE.with_(name=f"tileskv{head_dim}", head_dim=head_dim)
    path = synth.ensure_gguf(shape, model_dir)
    for n, more in ((257, 300), (289, 33), (770, 271)):
        o = O.OracleModel(path, 1100, shape.im_end_id, flags=O.KV_F16)
        with Engine(path, 1100, shape.im_end_id, kv_f16=True) as e:
            for m in (n, more):
                prompt = make_prompt(shape, m, seed=m)
                (hg, lg), (ho, lo) = e.eval(prompt), o.eval(prompt)
                # a key or value on the other side of an f16 rounding: 5e-4 of it, among hundreds
                assert _rel(hg, ho) < 5e-4 and _rel(lg, lo) < 5e-4, (n, m, _rel(hg, ho), _rel(lg, lo))
